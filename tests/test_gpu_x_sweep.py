"""The X sweep's forms at the edges of their tiles, against the oracle bit for bit.

A wave holds 64, 128, 192 or 256 cells, of which 12 are halos (or a whole ring of
256), and one wave carries all quantities or two each.  Rings one cell
shorter and longer than one, two and more tiles, rings shorter than the halos,
2-D and 3-D, isothermal and adiabatic, several fluids, with and without FARGO's
shift of many cells a step (the inner rings of a wide disk).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"
C2 = "fargo3d_amd/setups/c2_p3d.par"
C3 = "fargo3d_amd/setups/c3_adiabatic2d.par"
C4 = "fargo3d_amd/setups/c4_multifluid2d.par"


@pytest.fixture(scope="module")
def fa():
    import fargo3d_amd
    return fargo3d_amd


def compare(fa, par, ov, steps, what):
    import oracle
    print(what, par, ov, flush=True)
    o, s = oracle.Oracle(par, ov), fa.Simulation(par, ov)
    for _ in range(steps):
        assert o.step() == s.step(), what
    for fluid in range(s.nfluids):
        o.select_fluid(fluid)
        s.select_fluid(fluid)
        act = (slice(3, -3) if s.dimz else slice(None), slice(3, -3))
        for f in ["Density", "Vx", "Vy"] + (["Vz"] if s.dimz else []) + (["Energy"] if s.adiabatic else []):
            a, b = s.field(f)[act], np.array(o.field(f))[act]
            bad = np.count_nonzero(np.ascontiguousarray(a).view(np.int64) != np.ascontiguousarray(b).view(np.int64))
            assert bad == 0, (what, f, fluid, bad)
    assert np.array_equal(s.nshift()[act], np.array(o.nshift())[act]), what
    s.close()
    o.close()


@pytest.mark.parametrize("nx", [8, 51, 52, 53, 64, 103, 105, 116, 117, 181, 244, 245, 256, 361, 489])
def test_ring_lengths(fa, nx):
    L = fa.lib()
    try:
        for mode, tile, split in [(0, 128, -1), (2, 64, 0), (2, 128, 1), (2, 256, 0), (4, 128, -1), (4, 128, 1)]:
            assert L.f3d_fused_set_xmode(mode) == 0 and L.f3d_fused_set_xtile(tile) == 0
            assert L.f3d_fused_set_xsplit(split) == 0
            what = "mode %d tile %d split %d" % (mode, tile, split)
            compare(fa, C1, "Nx=%d Ny=14" % nx, 3, what)
    finally:
        L.f3d_fused_set_xmode(0)
        L.f3d_fused_set_xtile(128)
        L.f3d_fused_set_xsplit(-1)


# the form chosen by the sizes: one cell per lane in groups, one, two, three and
# four cells per lane, whole rings
@pytest.mark.parametrize("par,ov", [(C3, "Nx=100 Ny=12"), (C3, "Nx=1040 Ny=110"), (C3, "Nx=540 Ny=200"),
                                    (C3, "Nx=976 Ny=512"), (C3, "Nx=256 Ny=2048"), (C4, "Nx=130 Ny=400 NFluids=3"),
                                    (C2, "Nx=50 Ny=12 Nz=8"), (C2, "Nx=500 Ny=20 Nz=12"),
                                    (C2, "Nx=232 Ny=40 Nz=22"), (C2, "Nx=256 Ny=64 Nz=32"),
                                    (C2, "Nx=104 Ny=50 Nz=24 Eos=adiabatic EnergyBoundary=symmetric Gamma=1.4")])
def test_chosen_form(fa, par, ov):
    compare(fa, par, ov, 2, "chosen form")
