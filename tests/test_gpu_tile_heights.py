"""Tiles of 128 columns and 32 to 256 rows (bfaintb_prefill128_wreg_kernel): every height, stage count, weight order and scale grouping, at
the steps, rows and columns where they can go wrong.  The oracle is the repository's: 2 bf16 units of the fp32 sum."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, from_dev_u16, run_gemm, to_dev

pytestmark = pytest.mark.gpu

FORMATS = [(8, 0), (8, 64), (8, 32), (4, 0), (4, 128), (4, 32)]


def run_padded(p, pad_a, ldb, which=0, split=0):
    """run_gemm with rows of A pad_a elements longer (NaNs there) and rows of B ldb codes apart (codes there that must not count)."""
    a = np.full((p.m, p.k + pad_a), 0x7FC0, np.uint16)
    a[:, :p.k] = p.a_bf
    b = np.random.default_rng(9).integers(0, 256, size=(p.k, ldb * p.bits // 8), dtype=np.uint8)
    b[:, :p.n * p.bits // 8] = np.asarray(p.b_bytes).reshape(p.k, -1)
    return run_gemm(p, which=which, force_split_k=split, lda=p.k + pad_a, ldb=ldb, a_dev=to_dev(a), b_dev=to_dev(b))


def run(af, p, packed, which):
    import torch
    if not packed:
        return run_gemm(p, which=which)
    w = torch.empty(af.prepack_bytes(p.n, p.k, p.bits), dtype=torch.uint8, device="cuda")
    af.prepack(w, to_dev(p.b_bytes), p.n, p.k, weight_bits=p.bits)
    c = torch.zeros((p.m, p.n), dtype=torch.int16, device="cuda")
    ws = helpers._ws.get(af.prepacked_workspace_bytes(p.m, p.n, p.k, p.bits, p.group_size, which))
    af.gemm_prepacked(c, to_dev(p.a_bf), w, to_dev(p.s_bf), p.m, p.n, p.k, weight_bits=p.bits, group_size=p.group_size, workspace=ws, which=which)
    torch.cuda.synchronize()
    return from_dev_u16(c)


# 4, 6 and 8 blocks of 16 rows (33 .. 64, .. 96, .. 128 rows a tile), one tile and several, the last one of one row; one K-step, fewer than the
# stages, as many, one more, and several rounds of them
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits,group", FORMATS)
@pytest.mark.parametrize("m,n,k", [(33, 128, 128), (64, 272, 384), (65, 144, 512), (96, 128, 640), (97, 400, 256), (128, 272, 1408), (129, 128, 384), (257, 144, 1152)])
def test_small_tiles(m, n, k, bits, group, packed):
    import awesome_fusion_amd as af
    p = Problem(m, n, k, bits, group, seed=m + n + k + bits)
    c = run(af, p, packed, af.PREFILL_128)
    assert_close_ulp(p, c, f"{m}x{n}x{k} bits={bits} g={group} packed={packed}")
    assert np.array_equal(run(af, p, packed, af.PREFILL_128), c), "not reproducible"


# 10, 12 and 16 blocks: the tall tiles of the library's own choice, planned for few compute units
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits,group", FORMATS)
@pytest.mark.parametrize("m,n,k,blocks", [(320, 640, 2176, 10), (305, 528, 2304, 10), (384, 640, 1152, 12), (353, 528, 1280, 12), (512, 640, 1152, 16), (391, 656, 1408, 16)])
def test_tall_tiles(m, n, k, blocks, bits, group, packed):
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 14)
        pl = af.plan(m, n, k, bits, group, packed=packed, which=af.PREFILL)
        assert (pl.kernel, pl.tile_rows, pl.tile_cols, pl.waves, pl.splits) == (af.KERNEL_TILES_128, 16 * blocks, 128, 8, 1), pl.as_dict()
        p = Problem(m, n, k, bits, group, seed=m + k + bits)
        c = run(af, p, packed, af.PREFILL)
        assert_close_ulp(p, c, f"{blocks} blocks: {m}x{n}x{k} bits={bits} g={group} packed={packed}")
        assert np.array_equal(run(af, p, packed, af.PREFILL), c), "not reproducible"
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# the same over rows of A and B that are longer than they need be, for columns of which the last 16 are half (8-bit codes), a k that is no multiple
# of a K-step, and the small tiles beside them
@pytest.mark.parametrize("m,n,k,rows", [(305, 648, 2184, 160), (384, 648, 1160, 192), (391, 648, 1416, 256), (512, 648, 1160, 256), (300, 264, 1160, 128), (70, 136, 520, 96), (40, 136, 520, 64)])
@pytest.mark.parametrize("bits,group", [(8, 0), (4, 0)])
def test_longer_rows_and_ragged_columns(m, n, k, rows, bits, group):
    import awesome_fusion_amd as af
    n += 8 if bits == 4 else 0
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 14)
        pl = af.plan(m, n, k, bits, group, which=af.PREFILL)
        assert (pl.kernel, pl.tile_rows, n % 16) == (af.KERNEL_TILES_128, rows, 8 if bits == 8 else 0), pl.as_dict()
        p = Problem(m, n, k, bits, group, seed=m + k + bits)
        c = run_padded(p, 24, (n + 40) // 16 * 16, af.PREFILL)
        assert_close_ulp(p, c, f"{rows} rows: {m}x{n}x{k} bits={bits}")
        assert np.array_equal(run_padded(p, 0, (n + 15) // 16 * 16, af.PREFILL), c)
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


def test_tall_tiles_take_the_epilogues_and_strides():
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 14)
        for (m, n, k, bits, group) in ((500, 656, 1064, 8, 0), (300, 640, 2304, 4, 128)):   # (a last K-step that is not whole)
            assert af.variant(m, n, k, bits, group) == af.PREFILL and af.plan(m, n, k, bits, group).kernel == af.KERNEL_TILES_128
            p = Problem(m, n, k, bits, group, seed=m)
            c = run_gemm(p)
            wide = run_gemm(p, ldc=n + 24, c_fill=0x1234)
            assert np.array_equal(wide[:, :n], c) and (wide[:, n:] == 0x1234).all()
            p.with_bias().with_residual()
            assert_close_ulp(p, run_gemm(p), "bias and residual")
            g = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
            assert_close_gated(g, run_gemm(g, activation=af.ACT_SILU_GATE), "gated")
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# every height with (by 14 compute units, the tall ones) and without the copying wave
@pytest.mark.parametrize("bits,group,packed", [(8, 0, False), (8, 0, True), (8, 64, False), (8, 64, True), (4, 0, False), (4, 32, False), (4, 0, True), (4, 128, True)])
@pytest.mark.parametrize("m,n,k", [(20, 144, 512), (40, 144, 640), (70, 144, 512), (128, 272, 512), (320, 640, 2176), (384, 640, 1152), (512, 640, 1152)])
def test_scales_of_any_sign_and_size(m, n, k, bits, group, packed):
    """The conversion by halves gives q s whatever the scale, up to the format's limit: beyond 2^117 its second product is not finite for 8-bit
    codes, which then go another way."""
    import awesome_fusion_amd as af
    try:
        which = af.PREFILL_128
        if m > 128:
            af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 14)
            which = af.PREFILL
            assert af.plan(m, n, k, bits, group, packed=packed, which=which).kernel == af.KERNEL_TILES_128
        p = helpers.scales_of_any_sign_and_size(Problem(m, n, k, bits, group, seed=4))
        helpers.assert_close_at_any_scale(p, run(af, p, packed, which), f"{m}x{n}x{k} bits={bits} g={group} packed={packed}")
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# 2 blocks: fewer rows than a tile, one K-step, fewer than the stages, as many, one more, several rounds and an odd rest; a ragged last tile
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("bits,group", FORMATS)
@pytest.mark.parametrize("m,n,k", [(1, 128, 128), (16, 144, 384), (17, 272, 512), (32, 128, 640), (31, 400, 1408)])
def test_tiles_of_32_rows(m, n, k, bits, group, packed):
    import awesome_fusion_amd as af
    p = Problem(m, n, k, bits, group, seed=m + n + k + bits)
    c = run(af, p, packed, af.PREFILL_128)
    assert_close_ulp(p, c, f"{m}x{n}x{k} bits={bits} g={group} packed={packed}")
    assert np.array_equal(run(af, p, packed, af.PREFILL_128), c), "not reproducible"


# ... and as the library's own choice for 17 to 32 rows, planned for 8 compute units: 5 tiles (nine sixteenths of a round) to 8 and, of packed
# codes, more; k that is no multiple of a K-step; the family beside it agrees with the same oracle
@pytest.mark.parametrize("m,n,k,bits,group,packed", [(17, 656, 1032, 8, 0, False), (32, 1008, 1088, 8, 64, False), (21, 592, 1032, 4, 0, False),
                                                     (32, 1008, 1664, 4, 128, False), (24, 656, 3136, 8, 0, True), (32, 1552, 3072, 8, 64, True),
                                                     (17, 592, 1152, 4, 128, True), (32, 1552, 1280, 4, 0, True)])
def test_few_rows_choose_tiles(m, n, k, bits, group, packed):
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 8)
        pl = af.plan(m, n, k, bits, group, packed=packed)
        assert pl.variant == af.DECODE and pl.tiles_instead == pl.workgroups == (n + 127) // 128, pl.as_dict()
        assert (pl.kernel, pl.tile_rows, pl.tile_cols, pl.splits) == (af.KERNEL_TILES_128, 32, 128, 1), pl.as_dict()
        by_name = af.plan(m, n, k, bits, group, packed=packed, which=af.DECODE)
        assert by_name.tiles_instead == 0 and by_name.kernel == af.KERNEL_DECODE_FAMILY and by_name.workspace_bytes == pl.workspace_bytes
        p = Problem(m, n, k, bits, group, seed=m + n + k)
        c = run(af, p, packed, af.AUTO)
        assert_close_ulp(p, c, "tiles")
        assert_close_ulp(p, run(af, p, packed, af.DECODE), "family")
        if not packed:
            wide = run_gemm(p, ldc=n + 24, c_fill=0x1234)
            assert np.array_equal(wide[:, :n], c) and (wide[:, n:] == 0x1234).all()
            p.with_bias().with_residual()
            assert_close_ulp(p, run_gemm(p), "bias and residual")
            g = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
            assert_close_gated(g, run_gemm(g, activation=af.ACT_SILU_GATE), "gated")
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# ... over longer rows of A and B: the choice goes by the call's own distance of rows, a multiple of 1024 codes gets the family, any other the tiles
# (test_launches.py); a k that is no multiple of a K-step, columns of which the last 16 are half
@pytest.mark.parametrize("m,n,k,bits,group", [(17, 648, 1032, 8, 0), (32, 1000, 1088, 8, 64), (21, 592, 1032, 4, 0), (32, 1008, 1664, 4, 128)])
def test_few_rows_over_longer_rows(m, n, k, bits, group):
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 8)
        p = Problem(m, n, k, bits, group, seed=m + n + k)
        tiles, family = run_padded(p, 40, 2048 + 16), run_padded(p, 40, 2048)
        assert_close_ulp(p, tiles, "tiles")
        assert_close_ulp(p, family, "family")
        assert np.array_equal(run_padded(p, 0, (n + 15) // 16 * 16, af.PREFILL_128, 1), tiles) and np.array_equal(run_padded(p, 0, 1024, af.DECODE), family)
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("m,n,k,bits,group,packed", [(17, 656, 1032, 8, 0, False), (32, 1552, 3072, 8, 64, True), (24, 592, 1152, 4, 128, True)])
def test_few_rows_on_tiles_under_capture(m, n, k, bits, group, packed):
    """Recorded into a graph and replayed over new activations, other work on the same scratch between the replays."""
    import torch
    import awesome_fusion_amd as af
    try:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 8)
        assert af.plan(m, n, k, bits, group, packed=packed).tiles_instead
        problems = [Problem(m, n, k, bits, group, seed=s) for s in (1, 2, 3)]
        b, s = to_dev(problems[0].b_bytes), to_dev(problems[0].s_bf)
        if packed:
            w = torch.empty(af.prepack_bytes(n, k, bits), dtype=torch.uint8, device="cuda")
            af.prepack(w, b, n, k, weight_bits=bits)
            b = w
        a, c = to_dev(problems[0].a_bf), torch.zeros((m, n), dtype=torch.int16, device="cuda")
        ws = helpers._ws.get(max(af.workspace_bytes(m, n, k, bits, group), af.prepacked_workspace_bytes(m, n, k, bits, group) if packed else 0, af.workspace_bytes(4, n, 4096)))
        call = af.gemm_prepacked if packed else af.gemm
        af.init()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call(c, a, b, s, m, n, k, weight_bits=bits, group_size=group, workspace=ws)
        for i, q in enumerate(problems):
            a.copy_(to_dev(q.a_bf))
            c.fill_(0x7FC0)
            graph.replay()
            torch.cuda.synchronize()
            got = from_dev_u16(c)
            q.q, q.b_bytes, q.s_bf, q._w = problems[0].q, problems[0].b_bytes, problems[0].s_bf, None
            assert_close_ulp(q, got, f"replay {i}")
            call(c, a, b, s, m, n, k, weight_bits=bits, group_size=group, workspace=ws)
            torch.cuda.synchronize()
            assert np.array_equal(from_dev_u16(c), got)
            run_gemm(Problem(4, n, 4096, 8, 0, seed=5))   # a split call on the same scratch
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("m,n,k,group", [(18, 22016, 2560, 128), (32, 22016, 2176, 0)])
def test_the_familys_four_splits_by_name(m, n, k, group):
    """4-bit codes, 17 to 32 rows: the launch that the plan describes is what a call that names the family runs."""
    import awesome_fusion_amd as af
    p = Problem(m, n, k, 4, group, seed=m + k)
    assert_close_ulp(p, run_gemm(p, which=af.DECODE), f"{m}x{n}x{k} g={group}")


# more than two rows of tiles with grouped scales over codes in rows, k split: the copying wave there too (up to 64 steps a share)
@pytest.mark.parametrize("bits,group", [(8, 64), (8, 32), (4, 128), (4, 32)])
@pytest.mark.parametrize("m,n,k,splits", [(257, 272, 1152, 2), (300, 144, 640, 3), (520, 128, 8448, 2)])
def test_split_tiles_of_several_rows(m, n, k, splits, bits, group):
    p = Problem(m, n, k, bits, group, seed=m + n + bits)
    import awesome_fusion_amd as af
    c = run_gemm(p, which=af.PREFILL_128, force_split_k=splits)
    assert_close_ulp(p, c, f"{m}x{n}x{k} bits={bits} g={group} splits={splits}")
    assert np.array_equal(run_gemm(p, which=af.PREFILL_128, force_split_k=splits), c), "not reproducible"
