"""The Y and Z sweeps' forms (4 or 2 rows per thread, one row by two threads) at
the edges of their row blocks, against the oracle bit for bit; the precision
form, whose forms do the same arithmetic, against its own first form.

Row counts one below, at and above a multiple of 4 and of 2, down to one row past the
ghosts' stencil; rings of one lane more and less than a wave; 2-D and 3-D,
isothermal and adiabatic, several fluids.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"
C2 = "fargo3d_amd/setups/c2_p3d.par"
C3 = "fargo3d_amd/setups/c3_adiabatic2d.par"
C4 = "fargo3d_amd/setups/c4_multifluid2d.par"
AD3 = " Eos=adiabatic EnergyBoundary=symmetric Gamma=1.4"
R = " Ymin=1.0 Ymax=2.0"  # every ghost row at a positive radius
FORMS = [(0, 4), (1, 1), (2, 2), (4, 4), (5, 3)]


@pytest.fixture(scope="module")
def fa():
    import fargo3d_amd
    return fargo3d_amd


def fields(s, get):
    act = (slice(3, -3) if s.dimz else slice(None), slice(3, -3))
    names = ["Density", "Vx", "Vy"] + (["Vz"] if s.dimz else []) + (["Energy"] if s.adiabatic else [])
    return {f: np.ascontiguousarray(np.array(get(f))[act]) for f in names}


@pytest.mark.parametrize("par,ov", [(C1, "Nx=63 Ny=7"), (C1, "Nx=65 Ny=12"), (C3, "Nx=130 Ny=13"), (C3, "Nx=40 Ny=15"),
                                    (C4, "Nx=66 Ny=10 NFluids=2"), (C2, "Nx=20 Ny=9 Nz=5"),
                                    (C2, "Nx=70 Ny=14 Nz=8" + AD3), (C2, "Nx=64 Ny=11 Nz=7")])
def test_forms(fa, par, ov):
    import oracle
    ov += R
    L = fa.lib()
    o = oracle.Oracle(par, ov)
    dts = [o.step() for _ in range(3)]
    try:
        for ry, rz in FORMS:
            print(par, ov, ry, rz, flush=True)
            assert L.f3d_fused_set_tiling(ry, rz) == 0
            s = fa.Simulation(par, ov)
            assert [s.step() for _ in range(3)] == dts
            for fluid in range(s.nfluids):
                o.select_fluid(fluid)
                s.select_fluid(fluid)
                a, b = fields(s, s.field), fields(s, o.field)
                for f in a:
                    assert np.array_equal(a[f].view(np.int64), b[f].view(np.int64)), (f, fluid, ry, rz)
            s.close()
    finally:
        L.f3d_fused_set_tiling(0, 4)
    o.close()


@pytest.mark.parametrize("par,ov", [(C1, "Nx=63 Ny=7"), (C3, "Nx=130 Ny=13"), (C2, "Nx=20 Ny=9 Nz=5"),
                                    (C2, "Nx=70 Ny=14 Nz=8" + AD3)])
def test_forms_of_the_precision_form(fa, par, ov):
    ov += R
    L = fa.lib()
    first = None
    try:
        for ry, rz in FORMS:
            print(par, ov, ry, rz, flush=True)
            assert L.f3d32_fused_set_tiling(ry, rz) == 0
            s = fa.Simulation(par, ov + " Precision=32")
            for _ in range(3):
                s.step()
            a = fields(s, s.field)
            s.close()
            first = first or a
            # one float32 rounding a step of the terms that balance in the
            # disk, which are up to (r/h)^2 = 400 times what is left of them
            for f in a:
                assert np.abs(a[f] - first[f]).max() <= 3 * 400 * 2.0**-24 * np.abs(first[f]).max(), (f, ry, rz)
    finally:
        L.f3d32_fused_set_tiling(0, 4)
