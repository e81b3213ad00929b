"""Tiles of 256 columns and 128 to 256 rows (bfaintb_prefill_wreg_kernel), every height: at the K-steps where the stages of LDS, the operand sets and
the fragments' rotation come round or do not, and at partial steps, rows and columns.  On plans for 64 compute units, where small products make
enough of them.  An output is one chain of products in ascending k, whatever the tile: the form that stages both operands in LDS has its bits."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, from_dev_u16, run_gemm, to_dev

pytestmark = pytest.mark.gpu

# rows of A one past a row of tiles, so that the last row of tiles holds one (or few) rows; columns half a column block past a tile
HEIGHTS = [(128, 257, 8208), (160, 385, 8208), (192, 481, 8208), (224, 577, 8208), (256, 673, 12304)]
# one step, two, three and a partial one, four, five, six, seven and a partial one, thirteen, seven
STEPS = [(8, 0, 64), (8, 64, 128), (8, 0, 200), (8, 32, 256), (4, 0, 320), (4, 128, 384), (8, 0, 456), (4, 64, 832), (4, 32, 448)]


@pytest.fixture
def units64():
    import awesome_fusion_amd as af
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 64)
    yield af
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


def run_packed(af, p, which=0, **kw):
    import torch
    w = torch.empty(af.prepack_bytes(p.n, p.k, p.bits), dtype=torch.uint8, device="cuda")
    af.prepack(w, to_dev(p.b_bytes), p.n, p.k, weight_bits=p.bits)
    c = torch.zeros((p.m, p.n), dtype=torch.int16, device="cuda")
    af.gemm_prepacked(c, to_dev(p.a_bf), w, to_dev(p.s_bf), p.m, p.n, p.k, weight_bits=p.bits, group_size=p.group_size, which=which, **kw)
    torch.cuda.synchronize()
    return from_dev_u16(c)


def is_wide(af, rows, p, packed=False):
    pl = af.plan(p.m, p.n, p.k, p.bits, p.group_size, packed=packed, which=af.PREFILL)
    assert (pl.kernel, pl.variant, pl.tile_rows, pl.tile_cols, pl.launches, pl.workspace_bytes) == (af.KERNEL_TILES_256, af.PREFILL, rows, 256, 1, 0), pl.as_dict()


@pytest.mark.parametrize("rows,m,n", HEIGHTS)
@pytest.mark.parametrize("bits,group,k", STEPS)
def test_every_height_has_the_bits_of_the_form_through_lds(units64, rows, m, n, bits, group, k):
    af = units64
    p = Problem(m, n, k, bits, group, seed=m + k)
    is_wide(af, rows, p)
    c = run_gemm(p, which=af.PREFILL)
    assert np.array_equal(c, run_gemm(p, which=af.PREFILL_256_LDS))
    if rows == 160 or k == 200:
        assert_close_ulp(p, c, f"{rows} rows: {m}x{n}x{k} bits={bits} g={group}")
    if k % (64 if bits == 8 else 128) == 0:
        is_wide(af, rows, p, True)
        assert np.array_equal(run_packed(af, p, af.PREFILL), c), "packed"


@pytest.mark.parametrize("rows,m,n", HEIGHTS)
@pytest.mark.parametrize("bits,group", [(8, 0), (4, 128)])
def test_epilogues_and_strides(units64, rows, m, n, bits, group):
    """Bias and residual, the gate, rows of C, A and B that are longer than they need be."""
    af, k = units64, 384
    p = Problem(m, n, k, bits, group, seed=rows)
    is_wide(af, rows, p)
    assert af.plan(m, n, k, bits, group).as_dict() == af.plan(m, n, k, bits, group, which=af.PREFILL).as_dict()  # (the fused calls name no variant)
    c = run_gemm(p, which=af.PREFILL)
    wide = run_gemm(p, which=af.PREFILL, ldc=n + 24, c_fill=0x1234)
    assert np.array_equal(wide[:, :n], c) and (wide[:, n:] == 0x1234).all()
    a = np.full((m, k + 24), 0x7FC0, np.uint16)
    a[:, :k] = p.a_bf
    b = np.random.default_rng(9).integers(0, 256, size=(k, (n + 32) * bits // 8), dtype=np.uint8)
    b[:, :n * bits // 8] = np.asarray(p.b_bytes).reshape(k, -1)
    assert np.array_equal(run_gemm(p, which=af.PREFILL, lda=k + 24, ldb=n + 32, a_dev=to_dev(a), b_dev=to_dev(b)), c)
    p.with_bias()
    assert_close_ulp(p, run_gemm(p), "bias", threads=16)
    p.with_residual()
    assert_close_ulp(p, run_gemm(p), "bias and residual", threads=16)
    g = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
    assert_close_gated(g, run_gemm(g, activation=af.ACT_SILU_GATE), "gated")


@pytest.mark.parametrize("rows,m,n", HEIGHTS)
@pytest.mark.parametrize("bits,group", [(8, 0), (4, 128)])
def test_the_gate_alone_and_with_a_residual(units64, rows, m, n, bits, group):
    """A gate alone is finished in a loop, one with a residual written out: the same sums (a residual of zeros changes no bit but a zero's sign), rows of
    the residual longer than they need be and NaN behind, in place."""
    from test_gpu_residual_rows import run
    af, k = units64, 384
    g = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
    is_wide(af, rows, g)
    alone = run(af, g, False, None, None, activation=af.ACT_SILU_GATE)
    assert_close_gated(g, alone, "gate")
    longer = np.full((m, n // 2 + 8), 0x7FC0, np.uint16)
    longer[:, :n // 2] = 0
    zeros = run(af, g, False, to_dev(longer), n // 2 + 8, activation=af.ACT_SILU_GATE)
    assert np.array_equal(zeros, np.where(alone == 0x8000, 0, alone))
    g.with_residual()
    g.residual_bf = np.ascontiguousarray(g.residual_bf[:, :n // 2])
    longer[:, :n // 2] = g.residual_bf
    c = run(af, g, False, to_dev(longer), n // 2 + 8, activation=af.ACT_SILU_GATE)
    assert_close_gated(g, c, "gate and residual")
    own = to_dev(g.residual_bf).clone()
    assert np.array_equal(run(af, g, True, own, n // 2, own, activation=af.ACT_SILU_GATE), c), "in place, packed"


# beyond 2^117 8-bit codes go a second way along k
@pytest.mark.parametrize("rows,m,n", HEIGHTS)
@pytest.mark.parametrize("bits,group,k", [(8, 0, 200), (8, 64, 384), (4, 0, 320), (4, 128, 384)])
def test_scales_of_any_sign_and_size(units64, rows, m, n, bits, group, k):
    af = units64
    p = helpers.scales_of_any_sign_and_size(Problem(m, n, k, bits, group, seed=4))
    is_wide(af, rows, p)
    c = run_gemm(p, which=af.PREFILL)
    helpers.assert_close_at_any_scale(p, c, f"{rows} rows: {m}x{n}x{k} bits={bits} g={group}")
    if k % 128 == 0:
        helpers.assert_close_at_any_scale(p, run_packed(af, p, af.PREFILL), f"{rows} rows, packed: {m}x{n}x{k} bits={bits} g={group}")


# 97 to 128 rows that make more small tiles than units: partial blocks of rows and columns, a partial step
@pytest.mark.parametrize("m", [97, 100, 128])
@pytest.mark.parametrize("bits,group,k", [(8, 0, 1024), (8, 0, 1032), (8, 64, 1088), (4, 128, 1024), (4, 0, 1280)])
def test_few_rows_against_many_columns(units64, m, bits, group, k):
    af, n = units64, 8208
    p = Problem(m, n, k, bits, group, seed=m)
    is_wide(af, 128, p)
    c = run_gemm(p, which=af.PREFILL)
    assert np.array_equal(c, run_gemm(p, which=af.PREFILL_256_LDS))
    if k % 128 == 0:
        is_wide(af, 128, p, True)
        assert np.array_equal(run_packed(af, p, af.PREFILL), c), "packed"
    # a call that names a split of k runs the small tiles, which have it
    assert af.plan(m, n, k, bits, group, which=af.PREFILL, force_split_k=2).splits == 2
    assert_close_ulp(p, run_gemm(p, which=af.PREFILL, force_split_k=2), "split")


# whole rounds of 256x256 tiles and a thin last one as halves of 128 rows, or the thin round alone, planned for 8 units: a last row of tiles of one row, of 128,
# of one more and of 256, columns a block past a tile; one step, a partial last one, six, seven
@pytest.mark.parametrize("m,n", [(257, 1296), (384, 1296), (385, 1296), (512, 1536), (300, 272), (641, 784)])
@pytest.mark.parametrize("bits,group,k", [(8, 0, 64), (8, 0, 200), (4, 128, 384), (8, 64, 448)])
def test_the_thin_last_round(m, n, bits, group, k):
    import awesome_fusion_amd as af
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 8)
    try:
        pl = af.plan(m, n, k, bits, group, which=af.PREFILL_256)
        tiles = -(-m // 256) * -(-n // 256)
        rest = tiles % 8
        assert 0 < rest <= 4 and (pl.workgroups, pl.tail_workgroups, pl.launches) == (tiles - rest, 2 * rest, (tiles > rest) + (rest > 0)), pl.as_dict()
        p = Problem(m, n, k, bits, group, seed=m + k)
        c = run_gemm(p, which=af.PREFILL_256)
        assert_close_ulp(p, c, f"{m}x{n}x{k} bits={bits} g={group}")
        assert np.array_equal(c, run_gemm(p, which=af.PREFILL_256_LDS))
        wide = run_gemm(p, which=af.PREFILL_256, ldc=n + 24, c_fill=0x1234)
        assert np.array_equal(wide[:, :n], c) and (wide[:, n:] == 0x1234).all()
        if k % (64 if bits == 8 else 128) == 0:
            assert np.array_equal(run_packed(af, p, af.PREFILL_256), c), "packed"
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


# the same with bias, residual (rows longer than they need be and NaN behind; in place) and the gate, by the library's own choice: last rows of tiles whose lower
# half is empty, one row, whole, and a row of tiles of 129 rows behind two whole ones
@pytest.mark.parametrize("m,n", [(383, 1296), (384, 1040), (385, 1296), (512, 1536), (641, 1296)])
@pytest.mark.parametrize("bits,group,k", [(8, 0, 256), (4, 128, 384), (8, 64, 448)])
def test_epilogues_of_the_thin_last_round(m, n, bits, group, k):
    import awesome_fusion_amd as af
    from test_gpu_residual_rows import run
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 8)
    try:
        tiles = -(-m // 256) * -(-n // 256)
        rest = tiles % 8
        for packed in (False, True):
            pl = af.plan(m, n, k, bits, group, packed=packed)
            assert (pl.kernel, pl.tile_rows, pl.workgroups, pl.tail_workgroups) == (af.KERNEL_TILES_256, 256, tiles - rest, 2 * rest), pl.as_dict()
            p = Problem(m, n, k, bits, group, seed=m + n).with_residual()
            longer = np.full((m, n + 8), 0x7FC0, np.uint16)
            longer[:, :n] = p.residual_bf
            c = run(af, p, packed, to_dev(longer), n + 8)
            assert_close_ulp(p, c, "residual", threads=16)
            own = to_dev(p.residual_bf).clone()
            assert np.array_equal(run(af, p, packed, own, n, own), c), "in place"
            p.with_bias()
            assert_close_ulp(p, run(af, p, packed, to_dev(longer), n + 8), "bias and residual", threads=16)
            p.residual_bf = None
            assert_close_ulp(p, run(af, p, packed, None, None), "bias", threads=16)
            g = Problem(m, n, k, bits, group, seed=5, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
            assert_close_gated(g, run(af, g, packed, None, None, activation=af.ACT_SILU_GATE), "gate", threads=16)
            g.with_residual()
            g.residual_bf = np.ascontiguousarray(g.residual_bf[:, :n // 2])
            own = to_dev(g.residual_bf).clone()
            assert_close_gated(g, run(af, g, packed, own, n // 2, own, activation=af.ACT_SILU_GATE), "gate and residual, in place", threads=16)
    finally:
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)
