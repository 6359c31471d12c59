"""Gathers and scatters large enough for the window-ordered path (512 MiB; gathers of 8-byte elements 64 MiB), against
indexing by torch.

Lengths sit around the smallest calls that take the path; ragged ends leave a part of a 4096-element chunk, of a tile
and of a scatter's 64 KiB bin.
"""
import pytest

pytestmark = pytest.mark.gpu

WIDE = [(1 << 23) - 1, 1 << 23, (1 << 23) + 5, (1 << 23) + 4096 + 3, (1 << 24) + 8191, 1 << 26, (1 << 26) + 8191]
NARROW = [(1 << 27) - 1, 1 << 27, (1 << 27) + 4097]


def make_index(torch, n, kind, g):
    if kind == "random":
        return torch.randperm(n, device="cuda", dtype=torch.int32, generator=g)
    if kind == "reversed":  # every chunk local
        return torch.arange(n - 1, -1, -1, device="cuda", dtype=torch.int32)
    if kind == "outside":  # some indices are none
        idx = torch.randperm(n, device="cuda", dtype=torch.int32, generator=g)
        idx[::7] = -5
        idx[3::11] = n
        idx[5::13] = 2**31 - 1
        return idx
    # chunks of 4096 in random order, every other one reversed in itself (local), the others exchanged among themselves
    h = n // 8192 * 4096
    near = torch.arange(h, device="cuda", dtype=torch.int32).view(-1, 4096).flip(1)
    far = (torch.randperm(n - h, device="cuda", dtype=torch.int32, generator=g) + h)
    both = torch.stack([near, far[:h].view(-1, 4096)], 1).reshape(-1)
    return torch.cat([both, far[h:]])


@pytest.mark.parametrize("kind", ["random", "reversed", "outside", "mixed"])
@pytest.mark.parametrize("n,wide", [(n, True) for n in WIDE] + [(n, False) for n in NARROW])
def test_staged_gather_and_scatter(torch_gpu, ctx, n, wide, kind):
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(n % 1000 + 7)
    dt = torch.int64 if wide else torch.int32
    src = torch.randint(-2**31, 2**31, (n,), device="cuda", generator=g).to(dt)
    idx = make_index(torch, n, kind, g)
    ok = (idx >= 0) & (idx < n)
    at = idx.long().clamp(0, n - 1)

    out = torch.full((n,), -1, device="cuda", dtype=dt)
    ctx.gather(src, out, idx, wide=wide)
    assert torch.equal(out, torch.where(ok, src[at], torch.full_like(src, -1)))

    out.fill_(-1)
    ctx.scatter(src, out, idx, wide=wide)
    want = torch.full_like(src, -1)
    want[at[ok]] = src[ok]
    assert torch.equal(out, want)


def test_staged_gather_of_repeated_indices(torch_gpu, ctx):
    """A gather's indices may repeat: most of them in one window, one value for a third of them."""
    torch = torch_gpu
    n = (1 << 23) + 77
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    src = torch.randint(-2**62, 2**62, (n,), device="cuda", generator=g)
    idx = torch.randint(0, 300_000, (n,), device="cuda", dtype=torch.int32, generator=g)
    idx[::3] = 123_456
    idx[::4099] = torch.randint(0, n, (idx[::4099].numel(),), device="cuda", dtype=torch.int32, generator=g)
    out = torch.empty_like(src)
    ctx.gather(src, out, idx, wide=True)
    assert torch.equal(out, src[idx.long()])


@pytest.mark.parametrize("warm", [False, True])
def test_staged_under_capture(torch_gpu, edpp, warm):
    """Captured once and replayed with random, local and random indices in the same buffer; a fresh context, whose
    workspace must not grow under capture, takes the passes instead."""
    torch = torch_gpu
    n = (1 << 23) + 5
    s = torch.cuda.Stream()
    with torch.cuda.stream(s), edpp.Context(0, stream=s.cuda_stream) as c:
        src = torch.arange(n, device="cuda", dtype=torch.int64) * 3
        idx = torch.randperm(n, device="cuda", dtype=torch.int32)
        a, b = torch.empty_like(src), torch.empty_like(src)
        c.gather(src, a, idx, passes=2, wide=True)  # the passes' flags are all that a cold workspace holds
        if warm:
            c.gather(src, a, idx, wide=True)
            c.scatter(src, b, idx, wide=True)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            c.gather(src, a, idx, wide=True)
            c.scatter(src, b, idx, wide=True)
        for make in (lambda: torch.randperm(n, device="cuda", dtype=torch.int32),
                     lambda: torch.arange(n - 1, -1, -1, device="cuda", dtype=torch.int32),
                     lambda: torch.randperm(n, device="cuda", dtype=torch.int32)):
            idx.copy_(make())
            a.zero_()
            b.zero_()
            graph.replay()
            s.synchronize()
            at = idx.long()
            want = torch.empty_like(src)
            want[at] = src
            assert torch.equal(a, src[at]) and torch.equal(b, want)
        del graph
