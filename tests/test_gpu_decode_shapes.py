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


@pytest.mark.parametrize("m,n,k,group,packed", [(5, 144, 512, 32, False), (16, 272, 640, 128, False), (9, 144, 512, 64, True), (32, 272, 1024, 128, False),
                                                  (2, 144, 512, 128, True), (5, 272, 640, 0, True)])
def test_scales_of_any_sign_and_size(m, n, k, group, packed):
    """4-bit codes by halves (the family with grouped scales, the slab kernel with a scale for each chunk): the conversion's two terms, (1024 + code) s and (1024 + 8) s, are exact whatever the scale:
    negative, zero, subnormal, large."""
    import torch
    import awesome_fusion_amd as af
    import helpers
    import oracle
    p = Problem(m, n, k, 4, group, seed=4)
    s = np.random.default_rng(6).uniform(-1.0, 1.0, size=p.s_bf.shape).astype(np.float32)
    s[:, 0::6] *= np.float32(2.0 ** -120)
    s[:, 1::6] *= np.float32(2.0 ** 90)
    s[:, 2::6] = 0.0
    p.s_bf, p._w = oracle.f32_to_bf16_rne(s), None
    if packed:
        to_dev = helpers.to_dev
        w = torch.empty(af.prepack_bytes(n, k, 4), dtype=torch.uint8, device="cuda")
        af.prepack(w, to_dev(p.b_bytes), n, k, weight_bits=4)
        c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
        ws = helpers._ws.get(af.prepacked_workspace_bytes(m, n, k, 4, group, af.DECODE))
        af.gemm_prepacked(c, to_dev(p.a_bf), w, to_dev(p.s_bf), m, n, k, weight_bits=4, group_size=group, workspace=ws, which=af.DECODE)
        torch.cuda.synchronize()
        c = helpers.from_dev_u16(c)
    else:
        c = run_gemm(p, which=af.DECODE)
    c = helpers.widen(c).astype(np.float64)
    w, a = helpers.widen(p.w_bf).astype(np.float64), helpers.widen(p.a_bf).astype(np.float64)
    exact, absum = a @ w, np.abs(a) @ np.abs(w)
    # (one rounding to bf16, 2^-8, and an fp32 sum of k terms, at most k x 2^-24 of the sum of their magnitudes)
    assert (np.abs(c - exact) <= 2.0 ** -8 * np.abs(exact) + k * 2.0 ** -24 * absum + 1e-38).all()
