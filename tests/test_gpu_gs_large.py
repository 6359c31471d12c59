"""Default gathers and scatters of the largest tables that go by windows, and of the first ones past them.

2 GiB less one element is the upper end (1024 windows of a gather, 256 of a scatter, byte offsets just below 2^31); at
2 GiB the pass loop takes over.
"""
import pytest

pytestmark = pytest.mark.gpu

CASES = [(False, 1 << 28), (False, (1 << 29) - 1), (False, 1 << 29), (True, (1 << 28) - 1), (True, 1 << 28)]


@pytest.mark.parametrize("outside", [False, True])
@pytest.mark.parametrize("wide,n", CASES)
def test_largest_tables(torch_gpu, ctx, wide, n, outside):
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(n % 997 + outside)
    dt = torch.int64 if wide else torch.int32
    src = torch.randint(-2**31, 2**31 - 1, (n,), device="cuda", dtype=dt, generator=g)
    idx = torch.randperm(n, device="cuda", dtype=torch.int32, generator=g)
    if outside:
        idx[::7] = -1
        idx[3::11] = n
        idx[5::13] = -2**31
    ok = (idx >= 0) & (idx < n)
    at = idx.long().clamp_(0, n - 1)
    want = torch.where(ok, src[at], torch.full_like(src, -1))
    out = torch.full_like(src, -1)
    ctx.gather(src, out, idx, wide=wide)
    assert torch.equal(out, want)
    want.fill_(-1)
    want[at[ok]] = src[ok]
    out.fill_(-1)
    ctx.scatter(src, out, idx, wide=wide)
    assert torch.equal(out, want)
