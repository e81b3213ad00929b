"""The residual where a kernel requests all of a thread's rows at once: rows of it that are longer than they need be (the rest NaN: what belongs to
no output must not show), partial rows and columns of tiles, with the bias and without, plain, in place and behind the gate."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, from_dev_u16, to_dev

pytestmark = pytest.mark.gpu

FAMILY, SLAB, SMALL, TALL, WIDE = 1, 2, 3, 5, 6  # af.KERNEL_DECODE_FAMILY, _DECODE_SLAB, _TILES_128, _TILES_256X128, _TILES_256

# m, n, k, bits, group, compute units planned for (0: all), and what runs, row-major and packed: kernel, rows and columns of a tile, waves, splits, launches,
# workgroups of the thin last round
CALLS = [
    # the row-blocked family: unsplit; the sums of 2, 4, 6 and 8 splits fetched by two attempts in flight; by one (nine splits; tiles of 256 columns; two rows
    # a thread); a packed call of one row block on the slab kernel
    (5, 208, 96, 8, 0, 0, (FAMILY, 16, 128, 8, 1, 1, 0), None),
    (13, 208, 320, 8, 0, 0, (FAMILY, 16, 128, 8, 2, 1, 0), (SLAB, 16, 16, 8, 1, 1, 0)),
    (5, 208, 1024, 8, 0, 0, (FAMILY, 16, 128, 8, 4, 1, 0), (SLAB, 16, 16, 8, 1, 1, 0)),
    (16, 1040, 4096, 8, 0, 0, (FAMILY, 16, 128, 8, 8, 1, 0), (SLAB, 16, 16, 8, 1, 1, 0)),
    (3, 208, 2112, 8, 0, 0, (FAMILY, 16, 128, 8, 9, 1, 0), (SLAB, 16, 16, 8, 1, 1, 0)),
    (29, 2064, 4096, 8, 0, 0, (FAMILY, 16, 128, 8, 6, 1, 0), (FAMILY, 16, 80, 8, 4, 1, 0)),
    (13, 16400, 2048, 8, 0, 0, (FAMILY, 16, 256, 4, 3, 1, 0), (FAMILY, 16, 80, 8, 1, 1, 0)),
    (29, 16400, 2112, 8, 64, 0, (FAMILY, 32, 256, 4, 2, 1, 0), (FAMILY, 32, 80, 8, 1, 1, 0)),
    (33, 208, 512, 8, 0, 16, (FAMILY, 32, 128, 8, 2, 1, 0), (FAMILY, 16, 128, 8, 1, 1, 0)),
    (61, 208, 4096, 8, 64, 32, (FAMILY, 32, 128, 8, 8, 1, 0), (FAMILY, 32, 128, 8, 8, 1, 0)),
    (33, 1040, 96, 8, 0, 8, (FAMILY, 64, 128, 4, 1, 1, 0), None),
    (13, 12304, 4096, 4, 128, 0, (FAMILY, 16, 256, 8, 4, 1, 0), (FAMILY, 16, 128, 8, 2, 1, 0)),
    # tiles of 128 columns: unsplit and split in one launch, with the copying wave and without, 32 to 128 rows; with a second launch; 160 to 256 rows
    (17, 528, 1280, 8, 0, 8, (SMALL, 32, 128, 9, 1, 1, 0), (FAMILY, 16, 80, 8, 1, 1, 0)),
    (17, 528, 1280, 4, 128, 8, (SMALL, 32, 128, 9, 1, 1, 0), (SMALL, 32, 128, 9, 1, 1, 0)),
    (33, 208, 96, 8, 0, 0, (SMALL, 64, 128, 8, 1, 1, 0), None),
    (64, 6160, 256, 4, 128, 0, (SMALL, 64, 128, 8, 1, 1, 0), (SMALL, 64, 128, 9, 1, 1, 0)),
    (33, 1072, 1280, 8, 64, 16, (SMALL, 64, 128, 8, 1, 1, 0), (SMALL, 64, 128, 9, 1, 1, 0)),
    (33, 6160, 2048, 8, 0, 0, (SMALL, 64, 128, 8, 2, 1, 0), (FAMILY, 32, 128, 8, 2, 1, 0)),
    (33, 8240, 2048, 8, 64, 0, (SMALL, 64, 128, 8, 2, 1, 0), (SMALL, 64, 128, 9, 2, 1, 0)),
    (33, 4112, 4096, 8, 64, 128, (SMALL, 64, 128, 8, 3, 1, 0), (FAMILY, 16, 128, 8, 1, 1, 0)),
    (33, 6160, 4096, 8, 0, 0, (SMALL, 64, 128, 8, 4, 1, 0), (FAMILY, 64, 128, 4, 4, 1, 0)),
    (257, 208, 2048, 8, 64, 16, (SMALL, 96, 128, 9, 2, 1, 0), (SMALL, 96, 128, 9, 2, 1, 0)),
    (257, 208, 2048, 8, 0, 16, (SMALL, 96, 128, 8, 2, 1, 0), (SMALL, 96, 128, 8, 2, 1, 0)),
    (257, 528, 4096, 4, 64, 64, (SMALL, 96, 128, 9, 3, 1, 0), (FAMILY, 32, 128, 8, 1, 1, 0)),
    (385, 208, 2048, 8, 0, 16, (SMALL, 128, 128, 8, 2, 1, 0), (SMALL, 128, 128, 8, 2, 1, 0)),
    (300, 208, 4096, 4, 64, 32, (SMALL, 128, 128, 9, 4, 1, 0), (FAMILY, 32, 128, 8, 1, 1, 0)),
    (300, 208, 2048, 8, 64, 16, (SMALL, 128, 128, 9, 2, 1, 0), (FAMILY, 64, 128, 4, 1, 1, 0)),
    (97, 528, 4096, 4, 64, 16, (SMALL, 128, 128, 8, 2, 1, 0), (SMALL, 128, 128, 9, 2, 1, 0)),
    (97, 208, 1280, 4, 128, 0, (SMALL, 128, 128, 8, 7, 2, 0), (SMALL, 128, 128, 9, 7, 2, 0)),
    (300, 1040, 2048, 8, 64, 0, (SMALL, 128, 128, 9, 6, 2, 0), (FAMILY, 16, 128, 8, 1, 1, 0)),
    (300, 208, 256, 8, 64, 8, (SMALL, 128, 128, 8, 1, 1, 0), (SMALL, 128, 128, 9, 1, 1, 0)),
    (130, 528, 2112, 8, 0, 8, (SMALL, 160, 128, 8, 1, 1, 0), (SMALL, 160, 128, 8, 1, 1, 0)),
    (161, 528, 1280, 8, 64, 8, (SMALL, 192, 128, 8, 1, 1, 0), (FAMILY, 64, 128, 4, 1, 1, 0)),
    (200, 528, 1280, 4, 128, 8, (SMALL, 256, 128, 8, 1, 1, 0), (FAMILY, 64, 128, 4, 1, 1, 0)),
    (200, 528, 1280, 8, 64, 8, (SMALL, 256, 128, 8, 1, 1, 0), (SMALL, 256, 128, 8, 1, 1, 0)),
    # 256 x 128, in one chain
    (641, 208, 256, 4, 64, 8, (TALL, 256, 128, 4, 1, 1, 0), (TALL, 256, 128, 4, 1, 1, 0)),
    (200, 528, 256, 8, 0, 8, (TALL, 256, 128, 4, 1, 1, 0), (TALL, 256, 128, 4, 1, 1, 0)),
    # tiles of 256 columns, 128 to 256 rows; the thin last round of the 256-row ones as halves
    (97, 1040, 1024, 8, 64, 8, (WIDE, 128, 256, 4, 1, 1, 0), (WIDE, 128, 256, 4, 1, 1, 0)),
    (97, 1040, 1024, 4, 64, 8, (WIDE, 128, 256, 4, 1, 1, 0), (WIDE, 128, 256, 4, 1, 1, 0)),
    (385, 8208, 256, 8, 64, 64, (WIDE, 160, 256, 4, 1, 1, 0), (WIDE, 160, 256, 4, 1, 1, 0)),
    (500, 8208, 256, 8, 0, 64, (WIDE, 192, 256, 4, 1, 1, 0), (WIDE, 192, 256, 4, 1, 1, 0)),
    (385, 12304, 256, 4, 64, 8, (WIDE, 224, 256, 4, 1, 1, 0), (WIDE, 224, 256, 4, 1, 1, 0)),
    (130, 1040, 256, 8, 64, 8, (WIDE, 256, 256, 4, 1, 1, 0), (WIDE, 256, 256, 4, 1, 1, 0)),
    (385, 1296, 256, 8, 0, 8, (WIDE, 256, 256, 4, 1, 2, 8), (WIDE, 256, 256, 4, 1, 2, 8)),
    (512, 1552, 384, 4, 128, 8, (WIDE, 256, 256, 4, 1, 1, 0), (WIDE, 256, 256, 4, 1, 1, 0)),
    # larger ones
    (3, 4112, 2048, 8, 0, 0, (FAMILY, 16, 128, 8, 4, 1, 0), (SLAB, 16, 16, 8, 1, 1, 0)),
    (17, 22032, 256, 4, 128, 0, (FAMILY, 32, 128, 8, 1, 1, 0), (FAMILY, 16, 128, 8, 1, 1, 0)),
    (61, 16400, 256, 8, 0, 0, (SMALL, 64, 128, 8, 1, 1, 0), (FAMILY, 64, 128, 4, 1, 1, 0)),
    (97, 2064, 2048, 8, 0, 0, (SMALL, 128, 128, 8, 8, 2, 0), (FAMILY, 16, 128, 8, 2, 1, 0)),
    (33, 1040, 4096, 8, 0, 0, (FAMILY, 16, 128, 8, 8, 1, 0), (FAMILY, 16, 128, 8, 8, 1, 0)),
    (500, 12304, 320, 4, 64, 0, (TALL, 256, 128, 4, 1, 1, 0), None),
    (600, 12304, 2112, 8, 0, 0, (SMALL, 128, 128, 8, 1, 1, 0), (SMALL, 128, 128, 8, 1, 1, 0)),
    (1100, 4112, 512, 8, 0, 0, (TALL, 256, 128, 4, 1, 1, 0), (TALL, 256, 128, 4, 1, 1, 0)),
    (130, 33040, 576, 8, 0, 0, (WIDE, 160, 256, 4, 1, 1, 0), (WIDE, 160, 256, 4, 1, 1, 0)),
    (2100, 8208, 128, 4, 128, 0, (WIDE, 160, 256, 4, 1, 1, 0), (WIDE, 160, 256, 4, 1, 1, 0)),
]


def run(af, p, packed, residual, ldr, c=None, activation=0):
    import torch
    out_n = p.n // 2 if activation else p.n
    inputs = [to_dev(p.a_bf), to_dev(p.b_bytes), to_dev(p.s_bf)]
    call, need = af.gemm, af.workspace_bytes(p.m, p.n, p.k, p.bits, p.group_size)
    if packed:
        w = torch.empty(af.prepack_bytes(p.n, p.k, p.bits), dtype=torch.uint8, device="cuda")
        af.prepack(w, inputs[1], p.n, p.k, weight_bits=p.bits)
        inputs[1], call, need = w, af.gemm_prepacked, af.prepacked_workspace_bytes(p.m, p.n, p.k, p.bits, p.group_size)
    c = torch.zeros((p.m, out_n), dtype=torch.int16, device="cuda") if c is None else c
    call(c, *inputs, p.m, p.n, p.k, weight_bits=p.bits, group_size=p.group_size, workspace=helpers._ws.get(need), ldr=ldr, activation=activation,
         bias=None if p.bias_bf is None else to_dev(p.bias_bf), residual=residual)
    torch.cuda.synchronize()
    return from_dev_u16(c)


def what_runs(af, m, n, k, bits, group, packed):
    pl = af.plan(m, n, k, bits, group, packed=packed)
    return pl.kernel, pl.tile_rows, pl.tile_cols, pl.waves, pl.splits, pl.launches, pl.tail_workgroups


@pytest.fixture
def planned_for():
    import awesome_fusion_amd as af
    yield lambda units: af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, units)
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("m,n,k,bits,group,units,rows_form,packed_form", CALLS)
def test_residual_of_longer_rows(planned_for, m, n, k, bits, group, units, rows_form, packed_form):
    import awesome_fusion_amd as af
    planned_for(units)
    for packed, form in ((False, rows_form), (True, packed_form)):
        if form is None:  # (no packed order for such a k)
            continue
        assert what_runs(af, m, n, k, bits, group, packed) == form
        p = Problem(m, n, k, bits, group, seed=m + n).with_residual()
        longer = np.full((m, n + 40), 0x7FC0, np.uint16)
        longer[:, :n] = p.residual_bf
        c = run(af, p, packed, to_dev(longer), n + 40)
        assert_close_ulp(p, c, f"residual {m}x{n}x{k} packed={packed}", threads=16)
        own = to_dev(p.residual_bf).clone()
        assert np.array_equal(run(af, p, packed, own, n, own), c), "in place"
        p.with_bias()
        assert_close_ulp(p, run(af, p, packed, to_dev(longer), n + 40), "bias and residual", threads=16)
        g = Problem(m, n, k, bits, group, seed=5, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias().with_residual()
        g.residual_bf = np.ascontiguousarray(g.residual_bf[:, :n // 2])
        longer = np.full((m, n // 2 + 40), 0x7FC0, np.uint16)
        longer[:, :n // 2] = g.residual_bf
        c = run(af, g, packed, to_dev(longer), n // 2 + 40, activation=af.ACT_SILU_GATE)
        assert_close_gated(g, c, "gated", threads=16)
        own = to_dev(g.residual_bf).clone()
        assert np.array_equal(run(af, g, packed, own, n // 2, own, activation=af.ACT_SILU_GATE), c), "gated, in place"


# k in 2, 3, 4, 5 and 8 splits (the others' sums fetched by two attempts in flight), launch after launch over one workspace, with something added and without
@pytest.mark.parametrize("k,split", [(320, 2), (768, 3), (1024, 4), (1280, 5), (2048, 8)])
@pytest.mark.parametrize("m,n", [(16, 2064), (5, 656)])
def test_the_workspace_is_at_rest_behind_an_epilogue(m, n, k, split):
    import torch
    import awesome_fusion_amd as af
    p = Problem(m, n, k, seed=m + split).with_bias().with_residual()
    assert what_runs(af, m, n, k, 8, 0, False) == (FAMILY, 16, 128, 8, split, 1, 0)
    a, b, s, bias, residual = (to_dev(x) for x in (p.a_bf, p.b_bytes, p.s_bf, p.bias_bf, p.residual_bf))
    ws = torch.empty(af.workspace_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    af.workspace_init(ws)
    c, seen = torch.zeros((m, n), dtype=torch.int16, device="cuda"), {}
    for launch in range(24):
        added = launch % 3 != 2
        af.gemm(c, a, b, s, m, n, k, workspace=ws, bias=bias if added else None, residual=residual if added else None)
        torch.cuda.synchronize()
        assert bool((ws[256:] == 0xFF).all()), f"split {split}, launch {launch}: not at rest"
        got = from_dev_u16(c).copy()
        assert np.array_equal(seen.setdefault(added, got), got), f"split {split}, launch {launch}"
    assert_close_ulp(p, seen[True], f"split {split}, bias and residual", threads=16)
    p.bias_bf = p.residual_bf = None
    assert_close_ulp(p, seen[False], f"split {split}", threads=16)
    assert af.workspace_status(ws) == 0
