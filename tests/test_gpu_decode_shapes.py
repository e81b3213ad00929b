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
        p = af.plan(m, n, k, bits, group, which=af.DECODE)   # (by name: 17 to 32 rows run tiles by the library's own choice)
        assert (p.tile_cols, p.waves, p.splits) == want, p.as_dict()
        problem = Problem(m, n, k, bits, group, seed=m + k)
        c = run_gemm(problem, which=af.DECODE)
        assert_close_ulp(problem, c, f"{m}x{n}x{k} bits={bits} g={group}")
        assert np.array_equal(run_gemm(problem, which=af.DECODE), c)
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("m,n,k,bits,group,want", [(3, 3072, 8192, 8, 0, (128, 4, 10)), (18, 22016, 2560, 4, 128, (128, 4, 4)), (32, 22016, 2176, 4, 0, (128, 4, 4))])
def test_launch_shapes_of_the_whole_machine_match_oracle(m, n, k, bits, group, want):
    import awesome_fusion_amd as af
    p = af.plan(m, n, k, bits, group, which=af.DECODE)
    assert p.compute_units != 256 or (p.tile_cols, p.waves, p.splits) == want, p.as_dict()
    problem = Problem(m, n, k, bits, group, seed=m + k)
    c = run_gemm(problem, which=af.DECODE)
    assert_close_ulp(problem, c, f"{m}x{n}x{k} bits={bits} g={group}")
    assert np.array_equal(run_gemm(problem, which=af.DECODE), c)


# the family in rows and packed (one and two row blocks, 128 and 256 columns), the slab kernel with a scale for each column, chunk and block of
# rows, and the other tiled kernels
@pytest.mark.parametrize("which,m,n,k,bits,group,packed", [
    ("DECODE", 5, 144, 512, 4, 32, False), ("DECODE", 16, 272, 640, 4, 128, False), ("DECODE", 32, 272, 1024, 4, 128, False),
    ("DECODE", 2, 8192, 8192, 4, 128, False), ("DECODE", 40, 272, 640, 4, 0, False), ("DECODE", 9, 144, 512, 4, 64, True),
    ("DECODE", 2, 144, 512, 4, 128, True), ("DECODE", 5, 272, 640, 4, 0, True), ("DECODE", 16, 8192, 4096, 4, 128, True),
    ("DECODE", 5, 144, 512, 8, 64, False), ("DECODE", 3, 144, 512, 8, 0, True), ("DECODE", 40, 272, 640, 8, 32, True),
    ("PREFILL_256", 70, 272, 512, 8, 64, False), ("PREFILL_256", 70, 272, 512, 4, 128, True), ("PREFILL_256X128", 70, 272, 512, 8, 0, False),
    ("PREFILL_256X128", 70, 272, 512, 4, 64, True), ("PREFILL_128_LDS", 70, 272, 512, 8, 32, False), ("PREFILL_256_LDS", 70, 272, 512, 4, 64, False)])
def test_scales_of_any_sign_and_size(which, m, n, k, bits, group, packed):
    """A weight is q s, rounded once, whatever the scale: negative, zero, subnormal, and up to the format's limit of 2^120."""
    import torch
    import awesome_fusion_amd as af
    import helpers
    which = getattr(af, which)
    p = helpers.scales_of_any_sign_and_size(Problem(m, n, k, bits, group, seed=4))
    if packed:
        to_dev = helpers.to_dev
        w = torch.empty(af.prepack_bytes(n, k, bits), dtype=torch.uint8, device="cuda")
        af.prepack(w, to_dev(p.b_bytes), n, k, weight_bits=bits)
        c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
        ws = helpers._ws.get(af.prepacked_workspace_bytes(m, n, k, bits, group, which))
        af.gemm_prepacked(c, to_dev(p.a_bf), w, to_dev(p.s_bf), m, n, k, weight_bits=bits, group_size=group, workspace=ws, which=which)
        torch.cuda.synchronize()
        c = helpers.from_dev_u16(c)
    else:
        c = run_gemm(p, which=which)
    helpers.assert_close_at_any_scale(p, c, f"{m}x{n}x{k} bits={bits} g={group} packed={packed}")
