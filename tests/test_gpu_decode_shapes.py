"""Launch shapes the decode family takes for a short k (on plans for 16 compute units, where small matrices take them), for few rows
of whole lines and for 17 to 32 rows of 4-bit codes."""
import numpy as np
import pytest

from helpers import Problem, assert_close_ulp, run_gemm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,bits,group,want", [
    (1, 1040, 1000, 8, 0, (128, 8, 1)), (16, 2048, 1536, 8, 0, (128, 4, 1)), (17, 1808, 2048, 8, 64, (128, 8, 1)), (8, 1552, 2048, 4, 128, (128, 4, 1)),
    (32, 2048, 2048, 4, 0, (128, 8, 1))])
def test_launch_shapes_match_oracle(m, n, k, bits, group, want):
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 16)
        p = af.plan(m, n, k, bits, group)
        assert (p.tile_cols, p.waves, p.splits) == want, p.as_dict()
        problem = Problem(m, n, k, bits, group, seed=m + k)
        c = run_gemm(problem)
        assert_close_ulp(problem, c, f"{m}x{n}x{k} bits={bits} g={group}")
        assert np.array_equal(run_gemm(problem), c)
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("m,n,k,bits,group,want", [(3, 3072, 8192, 8, 0, (128, 4, 10)), (18, 22016, 2560, 4, 128, (128, 4, 4)), (32, 22016, 2176, 4, 0, (128, 4, 4))])
def test_launch_shapes_of_the_whole_machine_match_oracle(m, n, k, bits, group, want):
    import awesome_fusion_amd as af
    p = af.plan(m, n, k, bits, group)
    assert p.compute_units != 256 or (p.tile_cols, p.waves, p.splits) == want, p.as_dict()
    problem = Problem(m, n, k, bits, group, seed=m + k)
    c = run_gemm(problem)
    assert_close_ulp(problem, c, f"{m}x{n}x{k} bits={bits} g={group}")
    assert np.array_equal(run_gemm(problem), c)
