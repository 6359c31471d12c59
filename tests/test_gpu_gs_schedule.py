"""What the library reports and does about gathers and scatters that may go by windows of the random side."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [False, True])
def test_default_candidate_of_large_calls_is_none(torch_gpu, ctx, edpp, wide):
    torch = torch_gpu
    n = (1 << 29) // (8 if wide else 4)
    buf = torch.empty(n + 16, dtype=torch.int64 if wide else torch.int32, device="cuda")
    out, idx = torch.empty_like(buf), torch.empty(n + 16, dtype=torch.int32, device="cuda")
    for op in (edpp.OP_GATHER, edpp.OP_SCATTER):
        def cand(m, shift=0):
            return ctx.default_candidate(edpp.make_call(op, m, buf, out, 8 if wide else 4, idx=idx[shift:]))
        assert cand(n) == -1
        assert cand(n - 1) >= 0  # below 512 MiB the pass loop runs
        assert cand(n, 1) >= 0   # and with indices off 16 bytes


def test_calls_without_room_for_the_workspace(torch_gpu, edpp):
    """With no memory left for the window order's copies the pass loop runs, the context keeps the workspace it has, and
    no error is left behind by a call that succeeded."""
    torch = torch_gpu
    n = (1 << 27) + 3
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    src = torch.randint(-2**31, 2**31, (n,), device="cuda", dtype=torch.int32, generator=g)
    idx = torch.randperm(n, device="cuda", dtype=torch.int32, generator=g)
    gathered, scattered = torch.empty_like(src), torch.empty_like(src)
    want = src[idx.long()]
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    with edpp.Context(0, stream=torch.cuda.current_stream().cuda_stream) as c:
        c.scatter(src, scattered, idx, passes=2)  # a small workspace: one flag per chunk
        hold = []
        for _ in range(64):
            free = torch.cuda.mem_get_info()[0]
            if free <= 1 << 29:  # the gather alone needs 6 bytes per element
                break
            hold.append(torch.empty(min(16 << 30, free - (1 << 28)), dtype=torch.uint8, device="cuda"))
        for _ in range(2):
            gathered.fill_(-1)
            scattered.fill_(-1)
            c.gather(src, gathered, idx)
            c.scatter(src, scattered, idx)
            c.sync()
            assert torch.cuda.mem_get_info()[0] == free
            assert c._L.edpp_last_error(c.h) == b""
        hold.clear()
        torch.cuda.empty_cache()
        assert torch.equal(gathered, want)
        want[idx.long()] = src
        assert torch.equal(scattered, want)
        free = torch.cuda.mem_get_info()[0]
        scattered.fill_(-1)
        c.scatter(src, scattered, idx)  # there is room again
        c.sync()
        assert torch.cuda.mem_get_info()[0] < free - 16 * n
        assert torch.equal(scattered, want)
