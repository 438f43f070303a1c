"""The FEM tool's merged end of a step (friction sums, temperatures, wear, motion; heat exchange in the
near-tool pass) against the same step from the entry points, for record counts on both sides of a
workgroup and of the record buffer: on the first step every particle carries segment 0, so the
friction records number the particles.  The entry points order their sums with another workgroup size;
only above 4,096 records do both add the rest in an open order."""
import pytest

from helpers import assert_close, assert_equal
from sph_fem_2d_cutting_gpu_amd import cases
from sph_fem_2d_cutting_gpu_amd import solver as S
from test_gpu_step import Unfused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wear", [False, True])
@pytest.mark.parametrize("nx,ny", [(20, 14), (32, 16), (48, 16), (64, 32), (128, 32), (129, 32)])
def test_tool_end_equals_entry_points(nx, ny, wear):
    case = cases.perturbed(cases.small_cutting_case(nx=nx, ny=ny, wear=wear, tool_tris=500), vel_sd=1e-4, S_sd=1e-3)
    fused, ref = S.Simulation(case), S.Simulation(case)
    unf = Unfused(ref)
    exact = case.N <= 4096
    for k in range(3):
        print(f"N {case.N} wear {wear} step {k}", flush=True)
        fused.step(1)
        unf.step()
        fused.ctx.check_error()
        a, b = fused.tool_state(), ref.tool_state()
        for f in ("T", "k", "node_pos", "left", "right", "n", "K", "M", "heat_exchange", "fric_heat", "physical_para",
                  "sliding_force", "wear_nodes"):
            if exact:
                assert_equal(f"step {k} {f}", a[f], b[f])
            else:                       # sums of up to N terms in any order: N roundings of the sum
                assert_close(f"step {k} {f}", a[f], b[f], case.N * 2.3e-16)
        for f, v in b["scalars"].items():
            assert abs(a["scalars"][f] - v) <= (0.0 if exact else 1e-12 * max(abs(v), 1e-30)), f
    fused.close()
    ref.close()
