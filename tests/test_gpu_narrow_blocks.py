"""The decode family over packed weights with five, six and seven column blocks of 16 a workgroup: the last workgroup's blocks past n, every count of
rows at which the reduction deals them out differently, unsplit and split, on plans for few compute units, where small products take them."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp
from test_gpu_prepacked import packed_on_device, run_prepacked

pytestmark = pytest.mark.gpu

# columns of a workgroup, compute units planned for, n (past a whole number of workgroups), k, split
SHAPES = [(80, 8, 528, 1152, False), (80, 32, 528, 2048, True), (96, 8, 656, 1152, False), (96, 32, 416, 3072, True), (112, 8, 800, 1152, False)]
ROWS = {(80, 8): (1, 9, 16, 17, 32), (80, 32): (17, 19, 32), (96, 8): (1, 11, 16, 17, 32), (96, 32): (17, 22, 32), (112, 8): (13, 16)}
CASES = [(*s, m) for s in SHAPES for m in ROWS[s[:2]]] + [(80, 16, 528, 2048, True, 1), (80, 16, 528, 2048, True, 16), (96, 16, 416, 3072, True, 5),
                                                             (96, 16, 416, 3072, True, 16), (112, 8, 400, 1152, False, 17), (112, 8, 400, 1152, False, 32)]


@pytest.fixture
def planned():
    import awesome_fusion_amd as af

    def check(cols, units, split, p):
        af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, units)
        pl = af.plan(p.m, p.n, p.k, p.bits, p.group_size, packed=True, which=af.DECODE)  # (by name: 17 to 32 rows may run tiles)
        assert (pl.kernel, pl.tile_cols, pl.waves, pl.splits > 1) == (af.KERNEL_DECODE_FAMILY, cols, 8, split), pl.as_dict()
        assert pl.workgroups == -(-p.n // cols) * pl.splits * -(-p.m // pl.tile_rows), pl.as_dict()
        return af

    yield check
    af.debug_control(af.DEBUG_PLAN_COMPUTE_UNITS, 0)


@pytest.mark.parametrize("cols,units,n,k,split,m", CASES)
@pytest.mark.parametrize("bits,group", [(4, 128), (4, 32), (4, 0), (8, 0), (8, 64)])
def test_match_oracle(planned, cols, units, n, k, split, m, bits, group):
    p = Problem(m, n, k, bits, group, seed=m + n)
    af = planned(cols, units, split, p)
    pk = packed_on_device(af, p)
    c = run_prepacked(af, p, af.DECODE, pk=pk, ldc=n + 8)
    assert (c[:, n:] == 0x7FC0).all()
    assert_close_ulp(p, np.ascontiguousarray(c[:, :n]), f"{m}x{n}x{k} bits={bits} g={group}")
    assert np.array_equal(run_prepacked(af, p, af.DECODE, pk=pk), c[:, :n])
    p.with_bias().with_residual()
    assert_close_ulp(p, run_prepacked(af, p, pk=pk), "bias and residual")


@pytest.mark.parametrize("cols,units,n,k,split,m", [(80, 8, 528, 1152, False, 16), (96, 32, 416, 3072, True, 17), (112, 8, 800, 1152, False, 13)])
@pytest.mark.parametrize("bits,group", [(4, 128), (4, 0), (8, 64)])
def test_gate_and_scales_of_any_size(planned, cols, units, n, k, split, m, bits, group):
    p = Problem(m, n, k, bits, group, seed=3, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias()
    af = planned(cols, units, split, p)
    assert_close_gated(p, run_prepacked(af, p, activation=af.ACT_SILU_GATE), "gated")
    p = helpers.scales_of_any_sign_and_size(Problem(m, n, k, bits, group, seed=4))
    helpers.assert_close_at_any_scale(p, run_prepacked(af, p, af.DECODE), f"{m}x{n}x{k} bits={bits} g={group}")
