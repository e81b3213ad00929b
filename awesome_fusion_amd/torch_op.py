"""PyTorch binding of the bfAintBGemm C ABI: a custom operator and a linear layer built on it.

The reference is a stand-alone harness with no framework side; its README names the intended use
("gemm fusion for llm", /root/reference/README.md:2) and its argument block is that of a linear layer's
forward pass: activations A [m, k], weights B [k, n], per-output-channel scale, output C [m, n]
(/root/reference/bfAintBGemm/bfAintBGemm.cc:17-28,119-133).  This module lets such a layer call the
library:

    torch.ops.awesome_fusion.bfaintb_gemm(a, b, scale, weight_bits, group_size, bias=None, residual=None, activation=0) -> c
    torch.ops.awesome_fusion.bfaintb_gemm_prepacked(a, packed, scale, weight_bits, group_size, bias=None, residual=None, activation=0) -> c

``a`` bf16 [m, k] (row stride a multiple of 8 elements), ``b`` uint8 [k, n] (8-bit, excess-128) or
[k, n/2] (4-bit, excess-8, even column in the low nibble), ``scale`` bf16 [groups, n], ``bias`` bf16 [n] and
``residual`` bf16 [m, n] (added to the fp32 sums before the one rounding, inside the kernel); returns bf16 [m, n].  The
operators are native code (``csrc/torch_binding.cpp``: the same path written in Python took 21 - 26 us of host time per
call); this module gives them their shape inference, and their Python form where the native one does not load (with a
warning).  torch supplies the output tensor, the current stream and a per-(device, stream) split-K workspace; all
arithmetic happens in ``libbfaintb_gemm.so``.  There is no CPU implementation: on a CPU tensor the operator raises.

``quantize_weight`` (host-side helper, symmetric round-to-nearest) and ``QuantLinear`` are conveniences
for trying the kernel on a float model; the quantiser is not part of the reference either.
"""
from typing import Optional

import torch

from .gemm import (binding as _binding, gemm as _gemm, gemm_prepacked as _gemm_prepacked, prepack as _prepack, prepack_bytes as _prepack_bytes,
                   prepack_colmajor as _prepack_colmajor, prepacked_workspace_bytes as _prepacked_workspace_bytes, quantize as _quantize,
                   workspace_bytes as _workspace_bytes, workspace_init as _workspace_init)

_native = _binding()  # registers the operators (csrc/torch_binding.cpp)
_OP = "awesome_fusion::bfaintb_gemm"


def release_workspaces():
    """Gives the operators' split-K workspaces (one per device and stream) back to torch's allocator."""
    if _native is not None:
        _native.release_workspaces()


def _check(a, b, scale, weight_bits, group_size, bias=None):
    if a.dim() != 2 or b.dim() != 2 or scale.dim() != 2:
        raise ValueError("bfaintb_gemm: a [m, k], b [k, n*bits/8], scale [groups, n] must be 2-D")
    if a.dtype != torch.bfloat16 or scale.dtype != torch.bfloat16 or b.dtype != torch.uint8:
        raise TypeError("bfaintb_gemm: a and scale must be bfloat16, b uint8")
    if weight_bits not in (8, 4):
        raise ValueError("bfaintb_gemm: weight_bits must be 8 or 4")
    k = a.shape[1]
    n = b.shape[1] * (8 // weight_bits)
    groups = k // group_size if group_size else 1
    if b.shape[0] != k or tuple(scale.shape) != (groups, n):
        raise ValueError(f"bfaintb_gemm: shapes do not agree: a {tuple(a.shape)}, b {tuple(b.shape)}, scale {tuple(scale.shape)}")
    if bias is not None and (bias.dtype != torch.bfloat16 or tuple(bias.shape) != (n,)):
        raise ValueError("bfaintb_gemm: bias must be bfloat16 [n]")
    return a.shape[0], n, k


def _out_cols(n, activation):
    """Columns of the output: n, or n / 2 for the SiLU-gate epilogue (activation = 1: columns 2j and 2j+1 of the weights
    are the gate and up projections of output column j)."""
    if activation not in (0, 1):
        raise ValueError("bfaintb_gemm: activation must be 0 (none) or 1 (SiLU gate)")
    return n // 2 if activation == 1 else n


def _check_residual(residual, m, n):
    if residual is None:
        return None
    if residual.dtype != torch.bfloat16 or tuple(residual.shape) != (m, n):
        raise ValueError("bfaintb_gemm: residual must be bfloat16 [m, n]")
    return residual


def _check_prepacked(a, packed, scale, weight_bits, group_size, bias=None):
    if a.dim() != 2 or scale.dim() != 2 or packed.dim() != 1:
        raise ValueError("bfaintb_gemm_prepacked: a [m, k], packed [k*n*bits/8], scale [groups, n]")
    if a.dtype != torch.bfloat16 or scale.dtype != torch.bfloat16 or packed.dtype != torch.uint8:
        raise TypeError("bfaintb_gemm_prepacked: a and scale must be bfloat16, packed uint8")
    if weight_bits not in (8, 4):
        raise ValueError("bfaintb_gemm_prepacked: weight_bits must be 8 or 4")
    k, n = a.shape[1], scale.shape[1]
    groups = k // group_size if group_size else 1
    if scale.shape[0] != groups or packed.numel() != k * n * weight_bits // 8:
        raise ValueError(f"bfaintb_gemm_prepacked: shapes do not agree: a {tuple(a.shape)}, packed {packed.numel()} bytes, scale {tuple(scale.shape)}")
    if bias is not None and (bias.dtype != torch.bfloat16 or tuple(bias.shape) != (n,)):
        raise ValueError("bfaintb_gemm_prepacked: bias must be bfloat16 [n]")
    return a.shape[0], n, k


def _in_python(packed, a, w, scale, weight_bits, group_size, bias, residual, activation):
    """An operator where the native binding does not load: the same call through ctypes, on a workspace of its own (from the
    current stream's memory, the graph's under capture)."""
    m, n, k = (_check_prepacked if packed else _check)(a, w, scale, weight_bits, group_size, bias)
    n_out = _out_cols(n, activation)
    _check_residual(residual, m, n_out)
    if not a.is_cuda:
        raise RuntimeError(f"bfaintb_gemm{'_prepacked' * packed} runs on the GPU only (no CPU implementation)")
    if a.stride(1) != 1 or a.stride(0) % 8 or a.data_ptr() % 16:
        a = a.contiguous()
    w, scale = w.contiguous(), scale.contiguous()
    bias, residual = (None if t is None else t.contiguous() for t in (bias, residual))
    c = torch.empty((m, n_out), dtype=torch.bfloat16, device=a.device)
    if m == 0 or n == 0:
        return c
    with torch.cuda.device(a.device):
        need = (_prepacked_workspace_bytes if packed else _workspace_bytes)(m, n, k, weight_bits, group_size)
        ws = torch.empty(need, dtype=torch.uint8, device=a.device) if need else None
        if need:
            _workspace_init(ws)
        (_gemm_prepacked if packed else _gemm)(c, a, w, scale, m, n, k, lda=a.stride(0), weight_bits=weight_bits, group_size=group_size, workspace=ws,
                                               bias=bias, residual=residual, activation=activation)
    return c


if _native is None:
    @torch.library.custom_op(_OP, mutates_args=())
    def _rows(a: torch.Tensor, b: torch.Tensor, scale: torch.Tensor, weight_bits: int, group_size: int, bias: Optional[torch.Tensor] = None,
              residual: Optional[torch.Tensor] = None, activation: int = 0) -> torch.Tensor:
        return _in_python(False, a, b, scale, weight_bits, group_size, bias, residual, activation)

    @torch.library.custom_op(_OP + "_prepacked", mutates_args=())
    def _packed(a: torch.Tensor, packed: torch.Tensor, scale: torch.Tensor, weight_bits: int, group_size: int, bias: Optional[torch.Tensor] = None,
                residual: Optional[torch.Tensor] = None, activation: int = 0) -> torch.Tensor:
        return _in_python(True, a, packed, scale, weight_bits, group_size, bias, residual, activation)


bfaintb_gemm = torch.ops.awesome_fusion.bfaintb_gemm
bfaintb_gemm_prepacked = torch.ops.awesome_fusion.bfaintb_gemm_prepacked


@torch.library.register_fake(_OP)
def _(a, b, scale, weight_bits, group_size, bias=None, residual=None, activation=0):
    m, n, _k = _check(a, b, scale, weight_bits, group_size, bias)
    _check_residual(residual, m, _out_cols(n, activation))
    return a.new_empty((m, _out_cols(n, activation)))


@torch.library.register_fake(_OP + "_prepacked")
def _(a, packed, scale, weight_bits, group_size, bias=None, residual=None, activation=0):
    m, n, _k = _check_prepacked(a, packed, scale, weight_bits, group_size, bias)
    _check_residual(residual, m, _out_cols(n, activation))
    return a.new_empty((m, _out_cols(n, activation)))


def prepack_weight(b, weight_bits=8, column_major=False):
    """Codes ``b`` on the GPU -> flat packed tensor for ``bfaintb_gemm_prepacked``.  Row-major: uint8 [k, n*bits/8];
    ``column_major``: uint8 [n, k*bits/8] — one row per output feature, the way a Linear keeps its weight (4-bit: two
    consecutive k per byte, low nibble first)."""
    per_byte = 8 // weight_bits
    if column_major:
        n, k = b.shape[0], b.shape[1] * per_byte
    else:
        k, n = b.shape[0], b.shape[1] * per_byte
    nbytes = _prepack_bytes(n, k, weight_bits)
    if nbytes == 0:
        raise ValueError("prepack_weight: the packed order needs n % 16 == 0 and k % 64 == 0 (k % 128 == 0 for 4-bit codes)")
    packed = torch.empty(nbytes, dtype=torch.uint8, device=b.device)
    with torch.cuda.device(b.device):
        if column_major:
            _prepack_colmajor(packed, b.contiguous(), n, k, weight_bits=weight_bits)
        else:
            _prepack(packed, b.contiguous(), n, k, weight_bits=weight_bits)
    return packed


_WEIGHT_TYPES = {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def _quantizes_on_device(weight, weight_bits, group_size):
    """Whether bfaintb_quantize serves this weight: on the GPU, of a type and shape the GEMM kernels can go on to read
    (anything else, and the CPU, takes the torch form, which gives the same codes)."""
    n, k = weight.shape
    return (weight.is_cuda and weight.dtype in _WEIGHT_TYPES and weight_bits in (8, 4) and n % 16 == 0 and k % 8 == 0 and 0 < n and 0 < k <= 1 << 21
            and (group_size == 0 or (group_size % 32 == 0 and k % group_size == 0)))


def _quantize_on_device(w, weight_bits, group_size):
    n, k = w.shape
    if w.stride(1) != 1 or w.stride(0) < k or w.stride(0) % 8 or w.data_ptr() % 16:
        w = w.contiguous()
    b = torch.empty((k, n * weight_bits // 8), dtype=torch.uint8, device=w.device)
    scale = torch.empty((k // group_size if group_size else 1, n), dtype=torch.bfloat16, device=w.device)
    with torch.cuda.device(w.device):
        _quantize(b, scale, w, n, k, ldw=w.stride(0), weight_type=_WEIGHT_TYPES[w.dtype], weight_bits=weight_bits, group_size=group_size)
    return b, scale


def quantize_weight(weight, weight_bits=8, group_size=0):
    """float weight [n_out, k_in] (a torch Linear's layout) -> (b uint8 [k, n*bits/8], scale bf16 [groups, n]).

    Symmetric: scale = max|w| over the group / qmax, rounded to bf16 first, q = round(w / scale) clamped to the
    code range, stored in the library's wire format (excess-128 bytes; excess-8 nibbles, even column low)."""
    if _quantizes_on_device(weight, weight_bits, group_size):
        return _quantize_on_device(weight.detach(), weight_bits, group_size)
    w = weight.detach().float().t().contiguous()  # [k, n]
    k, n = w.shape
    g = group_size if group_size else k
    if k % g or (weight_bits == 4 and n % 2):
        raise ValueError("quantize_weight: group_size must divide k; 4-bit needs an even n")
    qmax = 127 if weight_bits == 8 else 7
    wg = w.view(k // g, g, n)
    scale = (wg.abs().amax(dim=1) / qmax).clamp_min(1e-12).to(torch.bfloat16)  # [groups, n]
    q = torch.round(wg / scale.float()[:, None, :]).clamp_(-qmax - 1, qmax).view(k, n).to(torch.int16)
    if weight_bits == 8:
        b = (q + 128).to(torch.uint8)
    else:
        u = (q + 8).to(torch.uint8)
        b = (u[:, 0::2] | (u[:, 1::2] << 4)).contiguous()
    return b, scale


def _check_features(in_features, out_features):
    if out_features % 16 or in_features % 8:
        raise ValueError("QuantLinear: the kernels need out_features % 16 == 0 (rows of B stay 16-byte aligned) and in_features % 8 == 0")


class QuantLinear(torch.nn.Module):
    """y = x @ dequant(B, scale) (+ bias): a Linear whose weight lives as int8/int4 codes and bf16 scales.

    The bias, if any, is added inside the kernel, to the fp32 sums."""

    def __init__(self, in_features, out_features, weight_bits=8, group_size=0, bias=False, device=None):
        _check_features(in_features, out_features)
        groups = in_features // group_size if group_size else 1
        self._set_up(in_features, out_features, weight_bits, group_size,
                     torch.zeros((in_features, out_features * weight_bits // 8), dtype=torch.uint8, device=device),
                     torch.zeros((groups, out_features), dtype=torch.bfloat16, device=device),
                     torch.zeros(out_features, dtype=torch.bfloat16, device=device) if bias else None)

    def _set_up(self, in_features, out_features, weight_bits, group_size, qweight, scales, bias):
        super().__init__()
        self.in_features, self.out_features = in_features, out_features
        self.weight_bits, self.group_size = weight_bits, group_size
        self.prepacked = False
        self.register_buffer("qweight", qweight)
        self.register_buffer("scales", scales)
        self.bias = None if bias is None else torch.nn.Parameter(bias)

    @classmethod
    def from_float(cls, linear, weight_bits=8, group_size=0):
        if cls is QuantLinear:  # the quantiser's own tensors become the buffers: nothing is zeroed first and copied over
            _check_features(linear.in_features, linear.out_features)
            b, s = quantize_weight(linear.weight, weight_bits, group_size)
            q = cls.__new__(cls)
            q._set_up(linear.in_features, linear.out_features, weight_bits, group_size, b, s,
                      None if linear.bias is None else linear.bias.detach().to(torch.bfloat16, copy=True))
            return q
        q = cls(linear.in_features, linear.out_features, weight_bits, group_size, linear.bias is not None, linear.weight.device)
        b, s = quantize_weight(linear.weight, weight_bits, group_size)
        q.qweight.copy_(b)
        q.scales.copy_(s)
        if linear.bias is not None:
            q.bias.data.copy_(linear.bias.detach().to(torch.bfloat16))
        return q

    def prepack(self):
        """Switches the layer to the pre-packed weight order (on the GPU, once): the row-major codes are replaced."""
        if not self.prepacked:
            self.qweight = prepack_weight(self.qweight, self.weight_bits)
            self.prepacked = True
        return self

    def forward(self, x, residual=None):
        """``residual`` (same shape as the output, bf16) is added inside the kernel, before the rounding."""
        if _native is not None and not torch.compiler.is_compiling():
            y = _native.linear_forward(self.__dict__, x, residual)
            if y is not NotImplemented:
                return y
        # traced, or something the native form does not know (a tensor subclass, an attribute of another kind)
        lead = x.shape[:-1]
        op = torch.ops.awesome_fusion.bfaintb_gemm_prepacked if self.prepacked else torch.ops.awesome_fusion.bfaintb_gemm
        if residual is not None:
            residual = residual.reshape(-1, self.out_features).to(torch.bfloat16)
        y = op(x.reshape(-1, self.in_features).to(torch.bfloat16), self.qweight, self.scales, self.weight_bits, self.group_size,
               self.bias, residual)
        return y.reshape(*lead, self.out_features)
