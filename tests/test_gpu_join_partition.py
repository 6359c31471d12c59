"""Joins whose partition pass takes the 64-bucket, 512-lane, 8-keys-per-lane shape, against the oracle.

A relation of 2^17 to 2^18 keys asks for 64 partitions; the longer relation (2^22 keys or more) is then split into 64
buckets at the large-input shape, whose histogram must fit the workspace sized for it.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("big,small", [((1 << 22) - 1, 1 << 18), (1 << 22, (1 << 17) + 33), ((1 << 22) + 4097, 1 << 18)])
@pytest.mark.parametrize("swap", [False, True])
def test_join_of_64_partitions_with_a_long_relation(torch_gpu, ctx, orc, big, small, swap):
    torch = torch_gpu
    r, s = orc.gen_i32(big, 11, 0xFFFFF), orc.gen_i32(small, 12, 0xFFFFF)
    if swap:
        r, s = s, r
    cnt = torch.zeros(1, dtype=torch.int64, device="cuda")
    ctx.join_count(torch.from_numpy(r).cuda(), torch.from_numpy(s).cuda(), cnt)
    ctx.sync()
    assert int(cnt.item()) == orc.join_count(r, s)


# around the lengths at which the one-pass partition changes its slots (2^22), gives way to the two-pass split (2^24),
# or has a last chunk, tile or group that is nearly empty
@pytest.mark.parametrize("small,large", [(1, 1), (1, 70_001), (4095, 16_385), (65_536, 65_537), ((1 << 20) + 3, 3 << 20),
                                         ((1 << 22) - 1, 1 << 22), (1 << 22, (1 << 22) + 4097), (1 << 22, 1 << 25),
                                         (1 << 24, 1 << 24), ((1 << 24) + 1, 1 << 24)])
def test_one_pass_partition_counts(torch_gpu, ctx, small, large):
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(small % 997)
    r = torch.randint(-2**31, 2**31, (small,), device="cuda", dtype=torch.int32, generator=g)
    s = r[torch.randint(0, small, (large,), device="cuda", generator=g)]
    s[::5] = torch.randint(-2**31, 2**31, (s[::5].numel(),), device="cuda", dtype=torch.int32, generator=g)
    keys, count = torch.unique(r, return_counts=True)
    at = torch.searchsorted(keys, s).clamp_(max=keys.numel() - 1)
    want = int(torch.where(keys[at] == s, count[at], 0).sum())
    cnt = torch.full((1,), -1, dtype=torch.int64, device="cuda")
    for a, b in ((r, s), (s, r)):
        ctx.join_count(a, b, cnt)
        ctx.sync()
        assert int(cnt.item()) == want
    # keys that do not start on a 16-byte boundary take the two-pass split
    ctx.join_count(torch.cat([r[:1], r])[1:], s, cnt, small, large)
    assert int(cnt.item()) == want


@pytest.mark.parametrize("repeats", [254, 255, 256, 40_000])
def test_join_of_keys_repeated_past_a_slots_count(torch_gpu, ctx, repeats):
    """32-bit slots count to 255 with 8 partition bits: some keys reach that, or stop just short of it, on both sides."""
    torch = torch_gpu
    n = 1 << 22
    r = torch.arange(n, device="cuda", dtype=torch.int32)
    s = torch.arange(n, device="cuda", dtype=torch.int32) + 7
    for i, key in enumerate((-1, 0, -2**31)):
        r[i * 50_000:i * 50_000 + repeats] = key
        s[i * 50_000 + 1000:i * 50_000 + 1000 + repeats] = key
    rk, rc = torch.unique(r, return_counts=True)
    sk, sc = torch.unique(s, return_counts=True)
    at = torch.searchsorted(rk, sk).clamp_(max=rk.numel() - 1)
    want = int(torch.where(rk[at] == sk, rc[at] * sc, 0).sum())
    cnt = torch.zeros(1, dtype=torch.int64, device="cuda")
    ctx.join_count(r, s, cnt)
    ctx.sync()
    assert int(cnt.item()) == want


@pytest.mark.parametrize("repeats", [2, 4, 8, 12, 30])
@pytest.mark.parametrize("n", [(1 << 22) + 5, (1 << 23) - 1])
def test_join_of_keys_repeated_a_few_times(torch_gpu, ctx, repeats, n):
    """Partitions on both sides of the bucket lengths at which a pair goes over to slots with counts."""
    torch = torch_gpu
    g = torch.Generator(device="cuda").manual_seed(repeats)
    r = torch.randint(-2**31, 2**31, (n // repeats,), device="cuda", dtype=torch.int32, generator=g).repeat(repeats)
    s = torch.randint(-2**31, 2**31, (2 * n,), device="cuda", dtype=torch.int32, generator=g)
    s[:r.numel()] = r.flip(0)
    r = torch.cat([r, s[-(n - r.numel()):]]) if r.numel() < n else r
    r = r[torch.randperm(r.numel(), device="cuda", generator=g)].contiguous()
    keys, count = torch.unique(r, return_counts=True)
    at = torch.searchsorted(keys, s).clamp_(max=keys.numel() - 1)
    want = int(torch.where(keys[at] == s, count[at], 0).sum())
    cnt = torch.full((1,), -1, dtype=torch.int64, device="cuda")
    for a, b in ((r, s), (s, r)):
        ctx.join_count(a, b, cnt)
        ctx.sync()
        assert int(cnt.item()) == want
