"""The planes per thread that the Z sweep chooses by itself (1, 2 and 4, by the
mesh's waves), against the oracle bit for bit; the precision form, which chooses
alike, against its form of 4 rows and planes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C2 = "fargo3d_amd/setups/c2_p3d.par"
R = " Ymin=1.0 Ymax=2.0"  # every ghost row at a positive radius
AD3 = " Eos=adiabatic EnergyBoundary=symmetric Gamma=1.4"
MESHES = ["Nx=20 Ny=9 Nz=5" + R, "Nx=70 Ny=40 Nz=12" + R, "Nx=70 Ny=40 Nz=13" + R + AD3, "Nx=130 Ny=60 Nz=44" + R]


def fields(s, get):
    act = (slice(3, -3), slice(3, -3))
    return {f: np.ascontiguousarray(np.array(get(f))[act])
            for f in ["Density", "Vx", "Vy", "Vz"] + (["Energy"] if s.adiabatic else [])}


@pytest.mark.parametrize("ov", MESHES)
def test_chosen_planes(ov):
    import fargo3d_amd as fa
    import oracle
    print(ov, flush=True)
    assert fa.lib().f3d_fused_set_tiling(0, 0) == 0
    o, s = oracle.Oracle(C2, ov), fa.Simulation(C2, ov)
    assert [s.step() for _ in range(2)] == [o.step() for _ in range(2)]
    a, b = fields(s, s.field), fields(s, o.field)
    for f in a:
        assert np.array_equal(a[f].view(np.int64), b[f].view(np.int64)), f
    s.close()
    o.close()


@pytest.mark.parametrize("ov", MESHES)
def test_chosen_planes_of_the_precision_form(ov):
    import fargo3d_amd as fa
    L = fa.lib()
    out = []
    for rows in (4, 0):
        print(ov, rows, flush=True)
        assert L.f3d32_fused_set_tiling(rows, rows) == 0
        s = fa.Simulation(C2, ov + " Precision=32")
        for _ in range(2):
            s.step()
        out.append(fields(s, s.field))
        s.close()
    # one float32 rounding a step of the terms that balance in the disk, which are
    # up to (r/h)^2 = 400 times what is left of them
    for f in out[0]:
        assert np.abs(out[1][f] - out[0][f]).max() <= 2 * 400 * 2.0**-24 * np.abs(out[0][f]).max(), f
