"""Gathers and scatters of large tables whose indices are neither random nor local in blocks of 4096.

Interleaved streams, shuffled rows, columns of a table, few distinct indices: a direct pass moves these at close to copy
rate or from L2, so the default call must not be slower than the pass loop it stands for, beyond the launches that its
choice costs (up to 1.14 times the single pass where that is fastest), and it must be right whichever path its chunks take.
"""
import pytest

pytestmark = pytest.mark.gpu


def _index(torch, n, kind, g):
    i = torch.arange(n, device="cuda", dtype=torch.int64)
    if kind == "interleaved":  # two halves, element by element
        return ((i % 2) * (n // 2) + i // 2).to(torch.int32)
    if kind == "streams":  # 64 sorted runs, merged at random
        label = torch.randint(0, 64, (n,), device="cuda", generator=g, dtype=torch.int16)
        idx = torch.empty(n, device="cuda", dtype=torch.int32)
        idx[torch.sort(label, stable=True).indices] = i.to(torch.int32)
        return idx
    if kind.startswith("rows"):
        r = int(kind[4:])
        return (torch.randperm(n // r, device="cuda", generator=g)[:, None] * r + torch.arange(r, device="cuda")).reshape(
            -1).to(torch.int32)
    if kind == "columns":  # a table of 8 columns, column by column
        return ((i % (n // 8)) * 8 + i // (n // 8)).to(torch.int32)
    if kind == "transposed":
        return ((i % 16384) * (n // 16384) + i // 16384).to(torch.int32)
    if kind == "few":
        some = torch.randint(0, n, (1000,), device="cuda", generator=g, dtype=torch.int32)
        return some[torch.randint(0, 1000, (n,), device="cuda", generator=g)]
    if kind == "window":  # random inside a window of 2^20 elements
        return torch.argsort(((i >> 20) << 31) | torch.randint(0, 1 << 31, (n,), device="cuda", generator=g)).to(torch.int32)
    assert kind == "half"  # half of them random, half interleaved
    h = n // 2
    return torch.cat([torch.randperm(h, device="cuda", generator=g),
                      h + (i[:h] % 2) * (h // 2) + i[:h] // 2]).to(torch.int32)


def _fastest(f):
    f()
    return min(f() for _ in range(5))


KINDS = ["interleaved", "streams", "rows8", "rows32", "rows512", "columns", "transposed", "window", "half"]


@pytest.mark.parametrize("wide,n", [(False, (1 << 27) + (1 << 15)), (True, (1 << 26) + (1 << 15))])
@pytest.mark.parametrize("kind", KINDS + ["few"])
def test_patterns(torch_gpu, ctx, wide, n, kind):
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    dt = torch.int64 if wide else torch.int32
    src = torch.randint(-2**31, 2**31, (n,), device="cuda", generator=g).to(dt)
    idx = _index(torch, n, kind, g)
    at = idx.long()
    out = torch.full_like(src, -1)
    ctx.gather(src, out, idx, wide=wide)
    assert torch.equal(out, src[at])
    default = _fastest(lambda: ctx.gather(src, out, idx, wide=wide, timed=True))
    single = _fastest(lambda: ctx.gather(src, out, idx, wide=wide, passes=1, timed=True))
    assert default < 1.3 * single, f"gather {default:.3f} ms, in one pass {single:.3f} ms"
    if kind == "few":
        return
    out.fill_(-1)
    ctx.scatter(src, out, idx, wide=wide)
    want = torch.full_like(src, -2)
    want[at] = src
    assert torch.equal(out, want)
    passes = ctx.schedule_passes(n, scatter=True, wide=wide)
    default = _fastest(lambda: ctx.scatter(src, out, idx, wide=wide, timed=True))
    direct = _fastest(lambda: ctx.scatter(src, out, idx, wide=wide, passes=passes, timed=True))
    assert default < 1.3 * direct, f"scatter {default:.3f} ms, in {passes} passes {direct:.3f} ms"


@pytest.mark.parametrize("wide,n", [(False, (1 << 27) + 4097), (True, (1 << 26) + 4097)])
def test_mostly_invalid_indices(torch_gpu, ctx, wide, n):
    """Chunks with few or no valid indices among random and dense ones, and a ragged last chunk of each."""
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    dt = torch.int64 if wide else torch.int32
    src = torch.randint(-2**31, 2**31, (n,), device="cuda", generator=g).to(dt)
    for scale in (1.0, 0.02):
        idx = torch.randperm(n, device="cuda", generator=g, dtype=torch.int32)
        keep = torch.rand(n, device="cuda", generator=g) < scale * torch.rand(n // 4096 + 1, device="cuda",
                                                                              generator=g).repeat_interleave(4096)[:n]
        idx = torch.where(keep, idx, torch.full_like(idx, -7))
        ok, at = idx >= 0, idx.long().clamp(0, n - 1)
        out = torch.full_like(src, -1)
        ctx.gather(src, out, idx, wide=wide)
        assert torch.equal(out, torch.where(ok, src[at], torch.full_like(src, -1)))
        out.fill_(-1)
        ctx.scatter(src, out, idx, wide=wide)
        want = torch.full_like(src, -1)
        want[at[ok]] = src[ok]
        assert torch.equal(out, want)
