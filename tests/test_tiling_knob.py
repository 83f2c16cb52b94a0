"""Both builds' sweeps can be set back to their automatic forms (no GPU needed:
the knobs only keep the numbers)."""
import fargo3d_amd as fa


def test_automatic_again():
    L = fa.lib()
    for set_tiling in (L.f3d_fused_set_tiling, L.f3d32_fused_set_tiling):
        assert set_tiling(4, 4) == 0
        assert set_tiling(0, 0) == 0
        assert set_tiling(-1, 0) == -2 and set_tiling(0, -1) == -2
