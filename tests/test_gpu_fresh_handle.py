"""A handle made right after another one was released takes its first time step
from its own fields, not from what the other left in the pinned result slots."""
import pytest

pytestmark = pytest.mark.gpu

C1 = "fargo3d_amd/setups/c1_fargo2d.par"


def test_first_step_after_another_handle():
    import fargo3d_amd as fa
    import oracle
    for ov in ["Nx=61 Ny=33", "Nx=125 Ny=41", "Nx=257 Ny=38", "Nx=63 Ny=39"] * 2:
        print(ov, flush=True)
        o, s = oracle.Oracle(C1, ov), fa.Simulation(C1, ov)
        assert s.step() == o.step(), ov
        s.close()
        o.close()
