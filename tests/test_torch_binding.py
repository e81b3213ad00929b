"""The native side of the PyTorch binding (awesome_fusion_amd/csrc/torch_binding.cpp): the linear layer's short way against
the operator it calls, what it hands on to the long way, its errors, and the operators' workspaces."""
import time

import pytest
import torch

import awesome_fusion_amd as af
import awesome_fusion_amd.torch_op as top


def test_layers_and_tensors_the_short_way_does_not_know_take_the_long_one():
    class Other(torch.Tensor):
        pass

    layer = top.QuantLinear(64, 32)
    short = top._native.linear_forward
    x = torch.zeros((2, 64), dtype=torch.bfloat16)
    assert short(layer.__dict__, x.as_subclass(Other), None) is NotImplemented
    assert short(layer.__dict__, None, None) is NotImplemented
    assert short({}, x, None) is NotImplemented
    with pytest.raises(RuntimeError, match="GPU only"):
        layer(x)
    with pytest.raises(ValueError, match="activation"):
        torch.ops.awesome_fusion.bfaintb_gemm(x, layer.qweight, layer.scales, 8, 0, None, None, 2)
    with pytest.raises(TypeError):
        torch.ops.awesome_fusion.bfaintb_gemm(x.float(), layer.qweight, layer.scales, 8, 0)


@pytest.fixture
def stand_in():
    """The row-major operator on CPU tensors: every output is the sum of its row of ``a``."""
    lib = torch.library.Library("awesome_fusion", "IMPL")
    lib.impl("bfaintb_gemm", lambda a, b, scale, bits, group, bias=None, residual=None, activation=0:
             a.float().sum(1, keepdim=True).expand(-1, scale.shape[1]).to(torch.bfloat16).contiguous(), "CPU", allow_override=True)
    yield
    lib._destroy()


@pytest.mark.filterwarnings("ignore:Warning only once for all operators")
@pytest.mark.parametrize("shape", [(2, 64), (64,), (0, 64), (0, 32), (2, 3, 64), (1, 1, 1, 64), (0, 2, 64),
                                   (4, 32), (2, 128), (64, 1), (128,), (2, 3, 32), (4, 16, 4)])
def test_inputs_of_another_width_are_refused(stand_in, shape):
    """Both ways through the layer take the same inputs: [..., in_features] (and nothing of another width whose number of
    elements happens to be a multiple of it)."""
    layer = top.QuantLinear(64, 32)
    x = torch.ones(shape, dtype=torch.bfloat16)
    want = x.reshape(-1, 64).float().sum(1, keepdim=True).expand(-1, 32).to(torch.bfloat16)
    if shape[-1] == 64 or x.numel() == 0:
        y = layer(x)
        assert y.shape == shape[:-1] + (32,) and torch.equal(y.reshape(-1, 32), want)
    else:
        with pytest.raises(RuntimeError, match="invalid for input of size"):
            layer(x)


@pytest.mark.filterwarnings("ignore:Warning only once for all operators", "ignore:.*torch.jit.trace:DeprecationWarning")
@pytest.mark.parametrize("lead,others", [((2, 3), [(5, 3), (2, 7), (4, 1)]), ((2,), [(7,), (1,)]), ((), [()])])
def test_traces_follow_the_leading_sizes(stand_in, lead, others):
    """torch.jit.trace of the layer, with and without a residual in the call, at other leading sizes than the traced ones."""
    layer = top.QuantLinear(64, 32)
    ones = lambda sizes, width: torch.ones(sizes + (width,), dtype=torch.bfloat16)
    for extra in (False, True):
        inputs = lambda sizes: (ones(sizes, 64), ones(sizes, 32)) if extra else (ones(sizes, 64),)
        traced = torch.jit.trace(layer, inputs(lead), check_trace=False)
        for sizes in [lead] + others:
            assert torch.equal(traced(*inputs(sizes)), layer(*inputs(sizes))), (lead, sizes, extra)


@pytest.mark.parametrize("packed", [False, True])
def test_what_a_call_writes_is_no_lazy_copy(packed):
    """The output and the workspace of a call have memory of their own before the call gets their addresses; what it only
    reads stays shared.  (The call itself is one that the library refuses before any launch.)"""
    call = af.gemm_prepacked if packed else af.gemm
    shared = [torch.zeros(4096, dtype=torch.uint8) for _ in range(7)]
    c, a, b, scale, bias, residual, workspace = copies = [torch._lazy_clone(t) for t in shared]
    assert all(torch._C._is_cow_tensor(t) for t in copies)
    rc = call(c, a, b, scale, 1, 16, 128, lda=8, bias=bias, residual=residual, workspace=workspace, stream=0, check=False)
    assert rc == -3
    assert [torch._C._is_cow_tensor(t) for t in copies] == [False, True, True, True, True, True, False]
    assert c.data_ptr() != shared[0].data_ptr() and workspace.data_ptr() != shared[6].data_ptr()


def test_a_workspace_of_another_kind_brings_its_own_size():
    """Whatever has data_ptr, numel and element_size serves as a workspace, as it does as an operand: large enough (refused for
    its alignment, the check after the size's), too small, without a size."""
    class Memory:
        def __init__(self, words):
            self.words = words

        def data_ptr(self):
            return 0x10008

        def numel(self):
            return self.words

        def element_size(self):
            return 4

    call = lambda ws: af.gemm(*[0x10000] * 4, 1, 4096, 4096, workspace=ws, stream=0, check=False)
    need = af.workspace_bytes(1, 4096, 4096)
    assert need > 0 and call(Memory(need // 4)) == -4 and call(Memory(need // 4 - 1)) == -6 and call(Memory(0)) == -6
    Memory.numel = None
    with pytest.raises(TypeError):
        call(Memory(need))


def _layer(n, k, bits, bias):
    lin = torch.nn.Linear(k, n, bias=bias).cuda()
    return top.QuantLinear.from_float(lin, bits, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("lead", [(512,), (1, 512), (3, 512), (0, 512), (2, 3, 512)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_short_and_long_way_agree(lead, dtype):
    torch.manual_seed(4)
    layer = _layer(272, 512, 8, True)
    x = torch.randn(lead, device="cuda", dtype=dtype)
    r = torch.randn(lead[:-1] + (272,), device="cuda", dtype=dtype)
    y = layer(x, residual=r)
    assert y.shape == r.shape and y.dtype == torch.bfloat16
    want = torch.ops.awesome_fusion.bfaintb_gemm(x.reshape(-1, 512).to(torch.bfloat16), layer.qweight, layer.scales, 8, 0, layer.bias,
                                                 r.reshape(-1, 272).to(torch.bfloat16))
    assert torch.equal(y.reshape(-1, 272), want)


@pytest.mark.gpu
def test_gradients_are_refused_and_library_errors_keep_their_code():
    layer = _layer(64, 128, 8, True)
    x = torch.randn((2, 128), device="cuda", dtype=torch.bfloat16)
    y = layer(x)
    assert y.requires_grad  # the bias is a parameter
    with pytest.raises(RuntimeError, match="autograd"):
        y.sum().backward()
    with torch.no_grad():
        assert not layer(x).requires_grad
    with pytest.raises(af.BfaintbError) as e:
        torch.ops.awesome_fusion.bfaintb_gemm(x, layer.qweight, layer.scales.repeat(3, 1)[:2].contiguous(), 8, 48 + 16 - 1)
    assert e.value.code == -5


@pytest.mark.gpu
def test_workspaces_by_stream_growth_and_capture():
    """Calls that split k: on several streams at once, growing, given back in between, and captured (the graph's workspace
    is not the one later calls outgrow or give back)."""
    torch.manual_seed(5)
    small, large = _layer(1024, 4096, 8, False), _layer(4096, 8192, 8, False)
    xs, xl = torch.randn((4, 4096), device="cuda", dtype=torch.bfloat16), torch.randn((32, 8192), device="cuda", dtype=torch.bfloat16)
    assert af.split_k(4, 1024, 4096) > 1 and af.split_k(32, 4096, 8192) > 1
    want_s, want_l = small(xs), large(xl)
    streams = [torch.cuda.Stream() for _ in range(3)]
    torch.cuda.synchronize()
    outs = []
    for i in range(6):
        with torch.cuda.stream(streams[i % 3]):
            outs.append((small(xs), large(xl)))
    torch.cuda.synchronize()
    assert all(torch.equal(a, want_s) and torch.equal(b, want_l) for a, b in outs)
    for warm in (True, False):  # with and without a workspace made before the capture
        top.release_workspaces()
        stream = torch.cuda.Stream()
        if warm:
            with torch.cuda.stream(stream):
                small(xs)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            c = small(xs)
        for _ in range(3):
            c.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, want_s)
            with torch.cuda.stream(stream):
                big = large(xl)
            top.release_workspaces()
            torch.full((64 << 20,), 7, dtype=torch.uint8, device="cuda")
            torch.cuda.synchronize()
            assert torch.equal(big, want_l)


@pytest.mark.gpu
def test_workspaces_of_graphs_are_given_back_with_them():
    """A program that captures, drops the graph, releases and captures again holds no more memory than after the first round;
    while a graph is there its workspace is, released, outgrown or not."""
    torch.manual_seed(6)
    small, large = _layer(1024, 4096, 8, False), _layer(4096, 8192, 8, False)
    xs, xl = torch.randn((4, 4096), device="cuda", dtype=torch.bfloat16), torch.randn((256, 8192), device="cuda", dtype=torch.bfloat16)
    assert 0 < af.workspace_bytes(4, 1024, 4096) <= 4 << 20 < af.workspace_bytes(256, 4096, 8192)
    want = small(xs)
    stream = torch.cuda.Stream()

    def held():
        torch.cuda.synchronize()
        return torch.cuda.memory_allocated()

    top.release_workspaces()
    before = held()
    for rep in range(4):
        with torch.cuda.stream(stream):
            small(xs)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            c, d = small(xs), small(xs)
        if rep % 2:
            with torch.cuda.stream(stream):
                large(xl)  # the stream's workspace is replaced by a larger one
        top.release_workspaces()
        assert held() - before >= 4 << 20, "the graph's workspace went before the graph"
        filler = torch.full((8 << 20,), 7, dtype=torch.uint8, device="cuda")
        for _ in range(2):
            c.zero_(), d.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(c, want) and torch.equal(d, want)
        del graph, c, d, filler
        for _ in range(100):  # (the runtime's own thread says that the graph is gone, a little after its end)
            top.release_workspaces()
            if held() - before < 1 << 20:
                break
            time.sleep(0.05)
        assert held() - before < 1 << 20, f"round {rep} left memory behind"


@pytest.mark.gpu
def test_a_stream_in_use_keeps_its_workspace():
    """More streams than workspaces are kept for, and one that is used all along: its workspace is never the one to go."""
    import ctypes
    torch.manual_seed(7)
    layer = _layer(1024, 4096, 8, False)
    x = torch.randn((4, 4096), device="cuda", dtype=torch.bfloat16)
    assert af.workspace_bytes(4, 1024, 4096) > 0
    want = layer(x)
    torch.cuda.synchronize()
    hip = ctypes.CDLL("libamdhip64.so.7")
    handles = [ctypes.c_void_p() for _ in range(72)]
    assert all(hip.hipStreamCreateWithFlags(ctypes.byref(h), 1) == 0 for h in handles)  # (non-blocking)
    made = lambda: torch.cuda.memory_stats()["allocation.all.allocated"]
    top.release_workspaces()
    layer(x)
    outs = []
    for h in handles:
        with torch.cuda.stream(torch.cuda.ExternalStream(h.value)):
            outs.append(layer(x))
        before = made()
        outs.append(layer(x))
        assert made() == before + 1, "more was allocated than the output"
    torch.cuda.synchronize()
    assert all(torch.equal(y, want) for y in outs)
    top.release_workspaces()
    del outs
    torch.cuda.synchronize()
    assert all(hip.hipStreamDestroy(h) == 0 for h in handles)
