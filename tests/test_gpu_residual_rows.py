"""The residual where a kernel requests all of a thread's rows at once: rows of it that are longer than they need be (the rest NaN: what belongs to
no output must not show), partial rows and columns of tiles, with the bias and without, plain, in place and behind the gate."""
import numpy as np
import pytest

import helpers
from helpers import Problem, assert_close_gated, assert_close_ulp, from_dev_u16, to_dev

pytestmark = pytest.mark.gpu

# decode with two fetch attempts in flight (two splits; eight), with one (rows beyond a thread's), unsplit; small tiles unsplit, split, with a second
# launch, with the copying wave; tall tiles; 256 x 128; 256 columns (eight blocks; sixteen)
CALLS = [(3, 4112, 2048, 8, 0), (16, 1040, 4096, 8, 0), (29, 2064, 4096, 8, 0), (5, 208, 96, 8, 0), (17, 22032, 256, 4, 128), (61, 16400, 256, 8, 0), (97, 2064, 2048, 8, 0),
         (33, 1040, 4096, 8, 0), (300, 1040, 2048, 8, 64), (500, 12304, 320, 4, 64), (600, 12304, 2112, 8, 0), (1100, 4112, 512, 8, 0), (130, 33040, 576, 8, 0), (2100, 8208, 128, 4, 128)]


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


@pytest.mark.parametrize("m,n,k,bits,group", CALLS)
def test_residual_of_longer_rows(m, n, k, bits, group):
    import awesome_fusion_amd as af
    for packed in (False, True):
        if packed and k % (64 if bits == 8 else 128):
            continue
        p = Problem(m, n, k, bits, group, seed=m + n).with_residual()
        longer = np.full((m, n + 40), 0x7FC0, np.uint16)
        longer[:, :n] = p.residual_bf
        c = run(af, p, packed, to_dev(longer), n + 40)
        assert_close_ulp(p, c, f"residual {m}x{n}x{k} packed={packed}", threads=16)
        own = to_dev(p.residual_bf).clone()
        assert np.array_equal(run(af, p, packed, own, n, own), c), "in place"
        p.with_bias()
        assert_close_ulp(p, run(af, p, packed, to_dev(longer), n + 40), "bias and residual", threads=16)
        if n % 16 == 0:
            g = Problem(m, n, k, bits, group, seed=5, scale_lo=0.002, scale_hi=0.02 if bits == 8 else 0.2).with_bias().with_residual()
            g.residual_bf = np.ascontiguousarray(g.residual_bf[:, :n // 2])
            longer = np.full((m, n // 2 + 40), 0x7FC0, np.uint16)
            longer[:, :n // 2] = g.residual_bf
            assert_close_gated(g, run(af, g, packed, to_dev(longer), n // 2 + 40, activation=af.ACT_SILU_GATE), "gated", threads=16)
