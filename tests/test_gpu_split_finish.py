"""Small tiles with k split six ways and more: a second launch adds the splits' sums (bfaintb_split_finish_kernel)."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, run_gemm

pytestmark = pytest.mark.gpu


# (one row of tiles, a partial last tile of rows and of columns; 16 columns past a tile, a last step that is not whole; splits: 6, 7, 8, beyond one fetch of
# eight; 18 tiles x 12 splits, which are dealt out unevenly over the 8 dies if split by split; two rows of tiles)
@pytest.mark.parametrize("m,n,k,bits,group", [(33, 4512, 9600, 8, 0), (96, 4096, 11008, 8, 0), (65, 1040, 4104, 8, 0), (139, 1072, 15488, 8, 0),
                                              (64, 1024, 14336, 4, 128), (128, 5120, 5120, 4, 128), (255, 1200, 9728, 8, 64),
                                              (100, 528, 4096, 4, 0)])
def test_second_launch_matches_oracle_and_the_one_launch_form(m, n, k, bits, group):
    import awesome_fusion_amd as af
    pl = af.plan(m, n, k, bits, group, which=af.PREFILL_128)
    assert pl.splits >= 6 and pl.launches == 2 and pl.workspace_bytes == af.workspace_bytes(m, n, k, bits, group, af.PREFILL_128)
    assert pl.workspace_bytes == 256 + ((pl.splits * m * n * 4 + 255) & ~255) <= af.lib().bfaintb_gemm_static_scratch_bytes()
    p = Problem(m, n, k, bits, group, seed=m + n + k)
    c = run_gemm(p, which=af.PREFILL_128)
    assert_close_ulp(p, c, f"second launch: {m}x{n}x{k} bits={bits} g={group}")
    assert bool((helpers._ws.t[256:] == 0xFF).all()) and af.workspace_status(helpers._ws.t) == 0
    assert np.array_equal(run_gemm(p, which=af.PREFILL_128), c)
    # the caller's own factor keeps the one launch: the same sums in the same order
    assert np.array_equal(run_gemm(p, which=af.PREFILL_128, force_split_k=pl.splits), c)
    if af.plan(m, n, k, bits, group).launches != 2:
        return  # (the epilogues come with the library's own choice only, which is another kernel here)
    p.with_bias().with_residual()
    assert_close_ulp(p, run_gemm(p), "bias and residual")
    g = Problem(m, n, k, bits, group, seed=5, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
    assert_close_gated(g, run_gemm(g, activation=af.ACT_SILU_GATE), "gated")


@pytest.mark.parametrize("m,n,k,bits,packed", [(124, 2800, 1664, 8, False), (105, 4560, 3200, 8, True), (474, 1136, 1920, 8, False)])
def test_without_scratch_no_second_launch_is_made(m, n, k, bits, packed):
    """Calls that need scratch for the second launch only are served without any, by one launch."""
    import torch
    import awesome_fusion_amd as af
    from helpers import from_dev_u16, to_dev
    assert af.plan(m, n, k, bits, packed=packed).launches >= 2
    p = Problem(m, n, k, bits, seed=m)
    c = torch.zeros((m, n), dtype=torch.int16, device="cuda")
    a, b, s = to_dev(p.a_bf), to_dev(p.b_bytes), to_dev(p.s_bf)
    if packed:
        w = torch.empty(af.prepack_bytes(n, k, bits), dtype=torch.uint8, device="cuda")
        af.prepack(w, b, n, k, weight_bits=bits)
        af.gemm_prepacked(c, a, w, s, m, n, k, weight_bits=bits)
    else:
        af.gemm(c, a, b, s, m, n, k, weight_bits=bits)
    torch.cuda.synchronize()
    assert_close_ulp(p, from_dev_u16(c), f"no scratch: {m}x{n}x{k} bits={bits} packed={packed}")


def test_second_launch_reports_sums_that_never_came():
    """As in the one launch: NaNs, a poisoned header, and all well after initialisation."""
    import torch
    import awesome_fusion_amd as af
    from helpers import from_dev_u16, to_dev
    p = Problem(64, 1024, 4096, seed=9)
    ws = torch.empty(af.workspace_bytes(p.m, p.n, p.k, which=af.PREFILL_128), dtype=torch.uint8, device="cuda")
    af.workspace_init(ws)
    a, b, s = to_dev(p.a_bf), to_dev(p.b_bytes), to_dev(p.s_bf)
    c = torch.zeros((p.m, p.n), dtype=torch.int16, device="cuda")
    run = lambda: (af.gemm(c, a, b, s, p.m, p.n, p.k, workspace=ws, which=af.PREFILL_128), torch.cuda.synchronize())
    try:
        af.debug_control(af.DEBUG_WITHHOLD_PARTIALS, 1)
        run()
    finally:
        af.debug_control(af.DEBUG_WITHHOLD_PARTIALS, 0)
    assert bool(torch.isnan(c.view(torch.bfloat16)).all()) and af.workspace_status(ws) == af.ERR_WORKSPACE_POISONED
    af.workspace_init(ws)
    run()
    assert_close_ulp(p, from_dev_u16(c), "after initialisation")
    assert af.workspace_status(ws) == 0


def test_second_launch_replays_from_a_graph():
    import torch
    import awesome_fusion_amd as af
    from helpers import from_dev_u16, to_dev
    p = Problem(96, 4096, 11008, seed=10)
    assert af.plan(p.m, p.n, p.k).launches == 2
    ws = torch.empty(af.workspace_bytes(p.m, p.n, p.k), dtype=torch.uint8, device="cuda")
    af.workspace_init(ws)
    a, b, s = to_dev(p.a_bf), to_dev(p.b_bytes), to_dev(p.s_bf)
    c = torch.zeros((p.m, p.n), dtype=torch.int16, device="cuda")
    call = lambda: af.gemm(c, a, b, s, p.m, p.n, p.k, workspace=ws)
    call()
    torch.cuda.synchronize()
    want = from_dev_u16(c).copy()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(4):
        c.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(from_dev_u16(c), want)
        call()
        torch.cuda.synchronize()
    assert af.workspace_status(ws) == 0
