"""A product in two launches by rows of A: the rows that fill their tiles, then the rest.  On plans for 16 compute units, where
small shapes show it (every plan is a correct launch on any device)."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, from_dev_u16, run_gemm, to_dev


@pytest.fixture
def few_units():
    import awesome_fusion_amd as af
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 16)
    yield af
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# one row past a tile; a row of tiles; tall, small and large tiles first; the rest with and without a split along k; odd k and
# columns past a tile
SHAPES = [(257, 1040, 1000, 8, 0), (272, 1024, 2048, 8, 64), (520, 784, 2048, 8, 0), (577, 1536, 1024, 4, 128), (777, 1040, 1000, 8, 0)]


@pytest.mark.parametrize("m,n,k,bits,group", SHAPES)
def test_the_plan_says_what_both_launches_are(few_units, m, n, k, bits, group):
    af = few_units
    one, two = af.plan(m, n, k, bits, group, which=af.PREFILL), af.plan(m, n, k, bits, group)
    assert two.launches == 2 and two.tail_workgroups > 0 and (two.workgroups, two.tile_rows) != (one.workgroups, one.tile_rows)
    assert two.splits == af.split_k(m, n, k, bits, group) and two.workspace_bytes == af.workspace_bytes(m, n, k, bits, group)
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 256)   # the same question for another machine is another question
    assert af.plan(m, n, k, bits, group).as_dict() != two.as_dict()
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 16)
    assert af.plan(m, n, k, bits, group).as_dict() == two.as_dict()


@pytest.mark.parametrize("m,n,k,bits,group,packed,rest", [
    (1568, 32144, 1664, 8, 128, False, 32), (2592, 24624, 2304, 8, 0, False, 32), (2075, 30496, 1280, 4, 64, True, 27), (2584, 29824, 3328, 8, 128, True, 24)])
def test_a_rest_of_17_to_32_rows_is_priced_as_the_tiles_it_runs_on(m, n, k, bits, group, packed, rest):
    """Whole large tiles, then 17 to 32 rows on tiles of 32, 4 to 11 % faster than the round of large tiles they would otherwise share."""
    import awesome_fusion_amd as af
    two, last = af.plan(m, n, k, bits, group, packed=packed), af.plan(rest, n, k, bits, group, packed=packed)
    if two.compute_units == 256:
        assert last.tiles_instead == last.workgroups == (n + 127) // 128
        assert (two.launches, two.workgroups, two.tail_workgroups) == (2, (m // 256) * ((n + 255) // 256), last.workgroups), two.as_dict()


# the same with a head of large or small tiles, on plans for 16 compute units
@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,bits,group,packed", [(529, 1296, 1152, 8, 128, False), (529, 1296, 1152, 8, 0, False), (273, 1152, 2176, 4, 128, False),
                                                     (273, 2064, 1152, 4, 0, True), (275, 1152, 3072, 8, 128, True)])
def test_rests_on_tiles_of_32_rows_match_oracle(few_units, m, n, k, bits, group, packed):
    import torch
    af = few_units
    pl = af.plan(m, n, k, bits, group, packed=packed)
    assert pl.launches == 2 and pl.tail_workgroups == (n + 127) // 128, pl.as_dict()
    p = Problem(m, n, k, bits, group, seed=m + n).with_bias().with_residual()
    if not packed:
        assert_close_ulp(p, run_gemm(p), f"{m}x{n}x{k}")
        return
    w = torch.empty(af.prepack_bytes(n, k, bits), dtype=torch.uint8, device="cuda")
    af.prepack(w, to_dev(p.b_bytes), n, k, weight_bits=bits)
    ws = helpers._ws.get(af.prepacked_workspace_bytes(m, n, k, bits, group))
    c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
    af.gemm_prepacked(c, to_dev(p.a_bf), w, to_dev(p.s_bf), m, n, k, weight_bits=bits, group_size=group, workspace=ws, bias=to_dev(p.bias_bf), residual=to_dev(p.residual_bf))
    torch.cuda.synchronize()
    assert_close_ulp(p, from_dev_u16(c), f"packed {m}x{n}x{k}")


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,bits,group", SHAPES)
def test_two_launches_match_oracle(few_units, m, n, k, bits, group):
    af = few_units
    p = Problem(m, n, k, bits, group, seed=m + n)
    c = run_gemm(p)
    assert_close_ulp(p, c, f"two launches: {m}x{n}x{k}")
    assert np.array_equal(run_gemm(p), c), "not reproducible"
    ldc = n + 24
    wide = run_gemm(p, ldc=ldc, c_fill=0x1234)
    assert np.array_equal(wide[:, :n], c) and (wide[:, n:] == 0x1234).all()
    p.with_bias().with_residual()
    assert_close_ulp(p, run_gemm(p), "bias and residual")
    g = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
    assert_close_gated(g, run_gemm(g, activation=af.ACT_SILU_GATE), "gated")


@pytest.mark.gpu
def test_two_launches_over_packed_weights(few_units):
    import torch
    af = few_units
    for (m, n, k, bits, group) in ((577, 1536, 1024, 4, 128), (272, 1024, 2048, 8, 64)):
        p = Problem(m, n, k, bits, group, seed=m)
        packed = torch.empty(af.prepack_bytes(n, k, bits), dtype=torch.uint8, device="cuda")
        af.prepack(packed, to_dev(p.b_bytes), n, k, weight_bits=bits)
        assert af.plan(m, n, k, bits, group, packed=True).tail_workgroups > 0
        ws = helpers._ws.get(af.prepacked_workspace_bytes(m, n, k, bits, group))
        c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
        af.gemm_prepacked(c, to_dev(p.a_bf), packed, to_dev(p.s_bf), m, n, k, weight_bits=bits, group_size=group, workspace=ws)
        torch.cuda.synchronize()
        assert_close_ulp(p, from_dev_u16(c), f"packed, two launches: {m}x{n}x{k}")


@pytest.mark.gpu
def test_without_the_scratch_for_two_launches_one_is_made(few_units):
    """A caller who brings no scratch (one launch over all rows needs none here) is served as ever; so is the entry point
    that brings its own."""
    import torch
    af = few_units
    m, n, k = 520, 784, 2048
    p = Problem(m, n, k, seed=8)
    assert af.workspace_bytes(m, n, k) > 0 == af.workspace_bytes(m, n, k, which=af.PREFILL)
    a, b, s = to_dev(p.a_bf), to_dev(p.b_bytes), to_dev(p.s_bf)
    c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
    af.gemm(c, a, b, s, m, n, k)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev_u16(c), run_gemm(p, which=af.PREFILL))
    af.gemm_static(c, a, b, s, m, n, k)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev_u16(c), run_gemm(p))
