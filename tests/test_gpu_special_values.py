"""Quotients of zero, infinite, NaN and tiny operands: IEEE results.

The kernels' short division has a range (fargo3d_amd/csrc/hip/f3d_device_body.h);
outside it the entry points still give what a / d gives.  Fields with such values
strewn in them go through the routines one by one and through the fused
sources, against the oracle bit for bit (any NaN equals any NaN).
The precision form's step is scale free in the density, so with densities
whose products with the zone sizes are subnormal it must stay finite and close
to the same step at the ordinary scale.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"
C2 = "fargo3d_amd/setups/c2_p3d.par"
C3 = "fargo3d_amd/setups/c3_adiabatic2d.par"
INF, NAN = np.inf, np.nan
SCALARS = [0.0, -0.0, INF, -INF, NAN, 1e-310, -3e-320, 1e-290, 1e300]


def pair(par, ov):
    import fargo3d_amd as fa
    import oracle
    print(par, ov, flush=True)
    o, s = oracle.Oracle(par, ov), fa.Simulation(par, ov)
    o.set_shape(s.nx, s.ny, s.nz, s.dimz)
    for _ in range(2):
        o.step()
    return o, s


def copy(o, s):
    names = ["Density", "Energy", "Vx", "Vy", "Vx_temp", "Vy_temp", "Mpx", "Mmx", "Mpy", "Mmy", "Pot", "Slope",
             "DivRho", "DensStar", "Qs", "Pressure", "QL", "QR"]
    names += ["Vz", "Vz_temp", "Mpz", "Mmz"] if s.dimz else []
    for n in names + ["VxMed"]:
        s.set_field(n, o.field(n))
    s.set_nshift(o.nshift())
    s.set_planets(o.planets())
    s.set_scalars(o.scalars())
    return names


def strew(o, names, values, seed):
    """A value of `values` in a few cells of every field, and a pair of
    neighbours without density."""
    rng = np.random.default_rng(seed)
    for n in names:
        f = o.field(n)
        v = values[n] if isinstance(values, dict) else values
        for x in v:
            f[tuple(rng.integers(0, k) for k in f.shape)] = x
    d = o.field("Density")
    d[d.shape[0] // 2, d.shape[1] // 2, 4:6] = 0.0


def differ(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return int(((a.view(np.int64) != b.view(np.int64)) & ~(np.isnan(a) & np.isnan(b))).sum())


COMMON = [("SubStep1_x", ("dt",)), ("SubStep1_y", ("dt",)), ("SubStep2_a", ("dt",)), ("SubStep2_b", ("dt",)),
          ("DivideByRho", ("Mpx",)), ("VanLeerY_a", ("DivRho",)), ("VanLeerY_b", ("dt", "DivRho", "Qs")),
          ("UpdateY", ("dt", "Mpx", "Qs")), ("UpdateDensityY", ("dt", "Density")), ("VanLeerX_a", ("Density",)),
          ("VanLeerX_b", ("dt", "Density", "DensStar", "Vx")), ("VanLeerX_PPA_d", ("dt", "DivRho", "Qs", "Vx_temp")),
          ("UpdateX", ("dt", "Mpx", "Qs", "Vx")), ("UpdateDensityX", ("dt", "Density", "Vx")), ("NewVelocity_x", ()),
          ("NewVelocity_y", ()), ("StockholmBoundary", ("dt",))]
CYL = [("visctensor_cyl", ()), ("addviscosity_cyl", ("dt",))]
SPH = [("visctensor_sph", ()), ("addviscosity_sph", ("dt",)), ("SubStep1_z", ("dt",)), ("VanLeerZ_a", ("Density",)),
       ("VanLeerZ_b", ("dt", "Density", "DensStar")), ("UpdateZ", ("dt", "Mpz", "Qs")),
       ("UpdateDensityZ", ("dt", "Density")), ("NewVelocity_z", ())]


@pytest.mark.parametrize("par,ov,routines", [(C1, "Nx=96 Ny=40", COMMON + CYL),
                                             (C2, "Nx=48 Ny=20 Nz=12", COMMON + SPH),
                                             (C3, "Nx=96 Ny=40", COMMON + CYL + [("SubStep3", ("dt",))])],
                         ids=["2d", "3d", "adiabatic"])
def test_routines(par, ov, routines):
    o, s = pair(par, ov)
    clean = {n: o.field(n).copy() for n in copy(o, s)}
    for k, (name, args) in enumerate(routines):
        for n in clean:
            o.field(n)[...] = clean[n]
        strew(o, clean, SCALARS, k)
        copy(o, s)
        a = [1e-3 if x == "dt" else x for x in args]
        o.call(name, *a)
        s.call(name, *a)
        bad = {n: differ(s.field(n), o.field(n)) for n in clean}
        assert not any(bad.values()), (name, {n: b for n, b in bad.items() if b})
    s.close()
    o.close()


@pytest.mark.parametrize("par,ov", [(C1, "Nx=130 Ny=41"), (C1, "Nx=20 Ny=14 ViscosityModel=alpha Alpha=1e-3"),
                                    (C1, "Nx=96 Ny=40 ViscosityModel=none"), (C3, "Nx=130 Ny=41"),
                                    (C3, "Nx=96 Ny=40 ViscosityModel=alpha Alpha=1e-3"), (C2, "Nx=48 Ny=20 Nz=12"),
                                    (C2, "Nx=48 Ny=20 Nz=12 Eos=adiabatic EnergyBoundary=symmetric Gamma=1.4")])
def test_fused_sources(par, ov):
    o, s = pair(par, ov)
    names = copy(o, s)
    ad, visc = s.adiabatic, "none" not in ov
    # a subnormal density leaves a stress of a few bits, so none in 3-D, whose stresses
    # go through arrays
    values = {n: [] for n in names}
    values["Density"] = [0.0, INF, NAN] + ([] if s.dimz else [1e-310])
    for v in ["Vx", "Vy"] + (["Vz"] if s.dimz else []):
        values[v] = [0.0, INF, -INF, NAN]
    values["Pot"] = [-INF]
    if ad:
        values["Energy"] = [0.0, INF, NAN]
    clean = {n: o.field(n).copy() for n in names}
    for seed in range(3):
        for n in clean:
            o.field(n)[...] = clean[n]
        strew(o, names, values, seed)
        copy(o, s)
        o.call("ComputePressureFieldAd" if ad else "ComputePressureFieldIso")
        for r in ["SubStep1_x", "SubStep1_y"] + (["SubStep1_z"] if s.dimz else []):
            o.call(r, 1e-3)
        if visc:
            o.call("visctensor_sph" if s.dimz else "visctensor_cyl")
            o.call("addviscosity_sph" if s.dimz else "addviscosity_cyl", 1e-3)
        o.call("SubStep2_a", 1e-3)
        o.call("SubStep2_b", 1e-3)
        if ad:
            o.call("SubStep3", 1e-3)
        s.call("fused_sources", 1e-3, 0.0)
        # the ghost fill that follows clears the velocities normal to the first faces
        act = (slice(4, -3) if s.dimz else slice(None), slice(4, -3))
        for n in ["Vx_temp", "Vy_temp"] + (["Vz_temp"] if s.dimz else []) + (["Energy"] if ad else []):
            assert differ(s.field(n)[act], o.field(n)[act]) == 0, (n, seed)
    s.close()
    o.close()


@pytest.mark.parametrize("par,ov", [(C1, "Nx=128 Ny=64"), (C1, "Nx=128 Ny=64 ViscosityModel=none"),
                                    (C2, "Nx=64 Ny=24 Nz=12")])
def test_tiny_densities_of_the_precision_form(par, ov):
    import fargo3d_amd as fa
    print(par, ov, flush=True)
    a = fa.Simulation(par, ov + " Precision=32")
    b = fa.Simulation(par, ov + " Precision=32")
    rho = a.field("Density")
    scale = 2.0 ** np.round(np.log2(2.0 ** -122 / rho.min()))
    for n in ("Density", "Density0"):
        b.set_field(n, a.field(n) * scale)
    assert a.step() == b.step()
    # a mass rho Vol keeps 2^-149 / (rho Vol) of its value, and a dozen roundings
    # of that size act on a velocity in one step
    vol = (2 * np.pi / a.nx) * (2.1 / a.ny) * 0.4 * (0.3 / a.nz if a.dimz else 1.0)
    tol = 12 * 2.0 ** -149 / (rho.min() * scale * vol)
    act = (slice(4, -4) if a.dimz else slice(None), slice(4, -4))
    for n in ["Vx", "Vy"] + (["Vz"] if a.dimz else []):
        u, v = a.field(n)[act], b.field(n)[act]
        assert np.isfinite(v).all(), n
        assert np.abs(u - v).max() <= tol * np.abs(a.field("Vx")[act]).max(), n
    a.close()
    b.close()
