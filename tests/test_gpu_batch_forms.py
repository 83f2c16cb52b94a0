"""A batch whose instances take different source kernels (constant nu, alpha,
none), on rings and rows at the edges of the tiles of the one-pass sources (62
cells, 4 rows) and of the potential (256 cells): every instance bit for bit as in a
batch of its own, and close to the single disk's FP32 form over one step.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"
SPECS = [(C1, "Nx=61 Ny=33 Nu=1e-5"), (C1, "Nx=62 Ny=36 Nu=0.0 Alpha=1e-3"), (C1, "Nx=125 Ny=41 Nu=0.0"),
         (C1, "Nx=257 Ny=38 Nu=1e-4"), (C1, "Nx=63 Ny=39 Nu=0.0 PlanetMass=0.0")]


def state(s):
    return {f: np.array(s.field(f)) for f in ("Density", "Vx", "Vy")}


def test_mixed_instances():
    import fargo3d_amd as fa
    b = fa.Batch(SPECS)
    b.step(3)
    b.sync()
    together = [state(s) for s in b.instances]
    b.close()
    for k, spec in enumerate(SPECS):
        print(spec, flush=True)
        one = fa.Batch([spec])
        one.step(3)
        one.sync()
        alone = state(one.instances[0])
        one.close()
        for f in alone:
            assert np.array_equal(alone[f].view(np.int64), together[k][f].view(np.int64)), (spec, f)


@pytest.mark.parametrize("spec", SPECS, ids=[s[1].replace(" ", "_") for s in SPECS])
def test_one_step_of_a_single_disk(spec):
    import fargo3d_amd as fa
    one = fa.Batch([spec])
    one.step(1)
    one.sync()
    a = state(one.instances[0])
    one.close()
    s = fa.Simulation(spec[0], spec[1] + " Precision=32")
    s.step()
    # one step rounds each field's balancing terms, up to (r/h)^2 = 400 times the
    # field's scale, a few times in FP32
    for f, v in state(s).items():
        assert np.abs(a[f] - v).max() <= 4 * 400 * 2.0**-24 * np.abs(v).max(), (spec, f)
    s.close()
