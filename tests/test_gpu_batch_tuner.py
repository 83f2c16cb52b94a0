"""The batch's tuner times, and reports, forms that differ: 4, 2 or 1 rows per
thread in the Y sweep.  Which of two equal forms is the faster is chance, so the
tuner is asked several times, on batches of two sizes."""
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"


@pytest.mark.parametrize("ov", ["Nx=768 Ny=192", "Nx=1024 Ny=320"])
def test_forms_reported(ov):
    import fargo3d_amd as fa
    b = fa.Batch([(C1, ov)] * 4)
    b.step(2)
    for _ in range(12):
        rows, tile = b.tune(reps=2)
        assert rows in (1, 2, 4) and tile in (64, 128, 256), (rows, tile)
    b.close()
