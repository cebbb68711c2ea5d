"""Host threads that share one stream, as torch's default stream is shared:
every call of every thread gives its own result, also where a call hands
partial sums or padded copies from one launch to the next through the stream's
workspace (needs a gfx950 GPU; the order of the launches is checked on the CPU
in test_workspaces_host.py)."""
import threading

import pytest

torch = pytest.importorskip("torch")

from veritac_amd import _lib
from veritac_amd.specializations.hip_gemm import backend as hg

pytestmark = pytest.mark.gpu

CALLS = 12


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    assert _lib.load_library().vt_device_count() >= 1, "GPU visible but not gfx950"
    return torch.device("cuda", 0)


# (m, n, k, variant): unequal and equal K slices, copies for the persistent
# kernel, K slices in place, row-major and packed decode, finishing words
@pytest.mark.parametrize("m,n,k,variant", [
    (84, 1040, 14832, "auto"), (128, 4096, 8192, "auto"), (3000, 3008, 3024, "auto"),
    (70, 80, 4111, "generic"), (48, 4096, 14336, "auto"), (48, 4096, 14336, "skinny_packed"),
    (16, 4096, 8192, "auto"), (8, 4096, 14336, "skinny_packed")])
def test_two_threads_on_one_stream(dev, m, n, k, variant):
    print("shared stream", m, n, k, variant, flush=True)
    plan = hg.make_plan(m, n, k, variant=variant)
    work = []
    for seed in (1, 2):
        g = torch.Generator(device=dev)
        g.manual_seed(seed)
        A = torch.randint(-128, 128, (m, k), generator=g, device=dev, dtype=torch.int8)
        B = torch.randint(-128, 128, (k, n), generator=g, device=dev, dtype=torch.int8)
        want = torch.matmul(A.double(), B.double()).to(torch.int64).to(torch.int32)
        outs = [torch.full((m, n), -2**31, dtype=torch.int32, device=dev) for _ in range(CALLS)]
        work.append((A, hg.pack_b(B) if variant == "skinny_packed" else B, want, outs))
    torch.cuda.synchronize()
    start, failed = threading.Barrier(2), []

    def calls(A, B, want, outs):
        try:
            start.wait(30)
            for out in outs:
                hg.run(plan, A, B, out=out)
        except Exception as exc:
            failed.append(exc)

    threads = [threading.Thread(target=calls, args=w) for w in work]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not failed, failed
    for _, _, want, outs in work:
        for i, out in enumerate(outs):
            assert torch.equal(out, want), i


@pytest.mark.parametrize("m,n,k", [(84, 1040, 14832), (16, 4096, 8192)])
def test_workspace_growth_while_another_thread_captures(dev, m, n, k):
    """A call on a fresh stream allocates its workspace while another thread
    captures its own stream; both results are right."""
    print("growth beside a capture", m, n, k, flush=True)
    plan, small = hg.make_plan(m, n, k), hg.make_plan(256, 256, 256)
    A = torch.randint(-128, 128, (m, k), device=dev, dtype=torch.int8)
    B = torch.randint(-128, 128, (k, n), device=dev, dtype=torch.int8)
    a = torch.randint(-128, 128, (256, 256), device=dev, dtype=torch.int8)
    out = torch.full((m, n), -2**31, dtype=torch.int32, device=dev)
    c = torch.empty((256, 256), dtype=torch.int32, device=dev)
    captured, other, failed = torch.cuda.Stream(), torch.cuda.Stream(), []
    torch.cuda.synchronize()

    def call():
        try:
            hg.run(plan, A, B, out=out, stream=other.cuda_stream)
        except Exception as exc:
            failed.append(exc)

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=captured):
        hg.run(small, a, a, out=c)
        t = threading.Thread(target=call)
        t.start()
        t.join()
    assert not failed, failed
    for _ in range(3):
        c.fill_(-2**31)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(c, torch.matmul(a.double(), a.double()).to(torch.int32))
    assert torch.equal(out, torch.matmul(A.double(), B.double()).to(torch.int32))
