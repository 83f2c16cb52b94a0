"""The ring sums equal the literal chain of additions bit for bit.

The device adds a ring's terms by runs that stay inside one binade of the
running sum (fargo3d_amd/csrc/hip/f3d_ringsum.h) instead of one after the
other.  Compared with numpy's sequential cumulative sum on rings at the edges of
the lanes' and chunks' sizes, with terms that keep the running sum in a binade,
hold halfway cases, cancel, change sign, cross zero, vanish or are not finite.
"""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"
NY = 26


def rings(n):
    """NY + 6 rings of n terms, each of its own kind."""
    rng = np.random.default_rng(n)
    x = 2 * np.pi * np.arange(n) / n
    out = np.zeros((NY + 6, n))
    for j in range(NY + 6):
        u = rng.uniform(-1, 1, n)
        k = j % 13
        out[j] = (1e-3 * (1 + 1e-4 * u), -(0.3 + 0.01 * np.cos(3 * x)), u, 1e-6 + 1e-3 * np.cos(2 * x + j),
                  np.ldexp(u, rng.integers(-40, 40, n)), rng.integers(-3, 4, n).astype(float),
                  np.ldexp(rng.integers(0, 1024, n) | 1, -10), (1 - 2 * (np.arange(n) % 2)) * (1 + 1e-3 * u),
                  np.where(u > 0, 0.0, -0.0), np.where(np.arange(n) == n // 2, 1e300, 1e284 * u), 1e-310 * u,
                  np.ldexp(np.sign(u), -rng.integers(0, 54, n)), 1.0 + 0.0 * u)[k]
    out[0, n // 3] = np.inf
    out[1, n // 2] = np.nan
    return out


def sequential(w):
    """((0 + w_0) + w_1) + ... along the last axis."""
    return np.cumsum(np.concatenate([np.zeros(w.shape[:-1] + (1,)), w], axis=-1), axis=-1)[..., -1]


def same_bits(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return (a.view(np.int64) == b.view(np.int64)) | (np.isnan(a) & np.isnan(b))


@pytest.fixture(scope="module")
def fa():
    import fargo3d_amd
    return fargo3d_amd


@pytest.mark.parametrize("n", [12, 63, 64, 65, 256, 257, 384, 511, 512, 513, 1024, 1025, 4096, 4099])
def test_ring_sums(fa, n):
    print("ring sums, %d terms" % n, flush=True)
    sim = fa.Simulation(C1, "Nx=%d Ny=%d CondInitOnDevice=yes" % (n, NY))
    f = rings(n)
    with np.errstate(all="ignore"):
        # reduction_SUM of a field, and of the whole active mesh
        sim.set_field("Slope", f)
        sim.call("reduction_SUM", "Slope", 0, NY + 6, 0, 1)
        want = sequential(f)
        assert same_bits(sim.field("Reduction2D")[0], want).all()
        total = ctypes.c_double()
        sim.call("reduction_full_SUM", "Slope", 3, NY + 3, 0, 1, ctypes.byref(total))
        assert same_bits(np.array([total.value]), sequential(want[3:-3][None])).all()
        # reduction_MIN: (acc < b) ? acc : b from 1e20
        sim.call("reduction_MIN", "Slope", 0, NY + 6, 0, 1)
        low = []
        for row in f:
            acc = 1e20
            for b in row:
                acc = acc if acc < b else b
            low.append(acc)
        assert same_bits(sim.field("Reduction2D")[0], np.array(low)).all()
        # VxMed of the fused CFL, from its own sums and from the pass of its own
        x = -3.14159265358979323844 + (2 * 3.14159265358979323844 / n) * np.arange(n + 1)
        sim.set_field("Vx", f)
        mean = sequential(f * np.diff(x)) / (2 * 3.14159265358979323844)
        try:
            for mode in (1, 3):
                sim.set_field("VxMed", np.zeros((1, NY + 6)))
                assert sim.L.f3d_fused_set_cflmode(mode) == 0
                sim.call("fused_cfl", ctypes.byref(ctypes.c_double()))
                assert same_bits(sim.field("VxMed")[0, 3:-3], mean[3:-3]).all(), mode
        finally:
            sim.L.f3d_fused_set_cflmode(-1)
    sim.close()
