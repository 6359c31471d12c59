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
