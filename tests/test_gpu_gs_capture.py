"""Captured gathers of tables that an eager call would reorder by windows.

A graph keeps its pointers, so a captured gather must hold nothing of the context's workspace: it has to stay right after
a later call has replaced the workspace by a larger one, beside eager calls between the replays, and without the context.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide,n", [(True, (1 << 26) + 5), (False, (1 << 27) + 4097)])
def test_captured_gather_outlives_the_workspace(torch_gpu, edpp, wide, n):
    torch = torch_gpu
    dt = torch.int64 if wide else torch.int32
    s = torch.cuda.Stream()
    g = torch.Generator(device="cuda")
    g.manual_seed(n % 1000)
    with torch.cuda.stream(s):
        src = torch.randint(-2**31, 2**31, (n,), device="cuda", generator=g).to(dt)
        idx = torch.randperm(n, device="cuda", dtype=torch.int32, generator=g)
        out, other = torch.empty_like(src), torch.empty_like(src)
        c = edpp.Context(0, stream=s.cuda_stream)
        c.gather(src, out, idx, wide=wide)  # the workspace is large enough for the call that is captured
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            c.gather(src, out, idx, wide=wide)

        def replay():
            idx.copy_(torch.randperm(n, device="cuda", dtype=torch.int32, generator=g))
            out.zero_()
            graph.replay()
            s.synchronize()
            assert torch.equal(out, src[idx.long()])

        replay()
        c.scatter(src, other, idx, wide=wide)  # needs a larger workspace than the gather
        replay()
        c.gather(src, other, idx, wide=wide)
        replay()
        c.close()
        replay()
        del graph
