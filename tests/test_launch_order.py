"""Two host threads on one stream and one workspace: a call whose launches meet in the workspace is not parted by another."""
import os
import subprocess
import threading

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_launches_of_one_call_follow_one_another(tmp_path):
    """On a stand-in runtime that records launches (tests/cpp/test_launch_order.cc): no GPU needed, none used."""
    import awesome_fusion_amd as af
    lib = os.path.dirname(af.library_path())
    exe = str(tmp_path / "test_launch_order")
    subprocess.run(["g++", "-std=c++17", "-O1", "-w", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "cpp", "test_launch_order.cc"), "-o", exe, "-L" + lib, "-l:libbfaintb_gemm.so",
                    "-Wl,-rpath," + lib, "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,/opt/rocm/lib", "-lpthread"], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "all checks passed" in r.stdout, r.stdout[-3000:]


@pytest.mark.gpu
def test_two_threads_share_a_stream():
    """The operators' workspace is one per stream: products in two launches and split decode calls from two threads."""
    import torch
    import awesome_fusion_amd as af
    import awesome_fusion_amd.torch_op as top
    torch.manual_seed(11)
    shapes = [(96, 4096, 11008), (1, 4096, 4096)]
    assert af.plan(*shapes[0]).launches == 2 and af.plan(*shapes[1]).splits > 1
    layers = [top.QuantLinear.from_float(torch.nn.Linear(k, n, bias=False).cuda(), 8, 0) for _, n, k in shapes]
    xs = [torch.randn((m, k), device="cuda", dtype=torch.bfloat16) for m, _, k in shapes]
    want = [layer(x) for layer, x in zip(layers, xs)]
    torch.cuda.synchronize()
    outs = [[], []]

    def work(i):
        for rep in range(40):
            j = (rep + i) % 2
            outs[i].append((j, layers[j](xs[j])))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert all(len(o) == 40 for o in outs)
    assert all(torch.equal(c, want[j]) for o in outs for j, c in o)
