"""Joins by the two-pass split with 64 partitions and a long relation, on keys that do not start on 16 bytes.

Keys on 16 bytes take the one-pass partition at these sizes, so only a shifted relation reaches the 64-bucket split of 512
lanes and 8 keys per lane, whose tiles its histogram has to be sized for.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("big,small", [((1 << 22) - 1, 1 << 18), (1 << 22, (1 << 17) + 33), ((1 << 22) + 4097, 1 << 18),
                                       (1 << 24, (1 << 17) + 1)])
@pytest.mark.parametrize("shift_big", [False, True])
def test_unaligned_join_of_64_partitions(torch_gpu, ctx, orc, big, small, shift_big):
    torch = torch_gpu
    r, s = orc.gen_i32(big, 11, 0xFFFFF), orc.gen_i32(small, 12, 0xFFFFF)
    want = orc.join_count(r, s)
    dr, ds = torch.from_numpy(r).cuda(), torch.from_numpy(s).cuda()
    if shift_big:
        dr = torch.cat([dr[:1], dr])[1:]
    else:
        ds = torch.cat([ds[:1], ds])[1:]
    cnt = torch.zeros(1, dtype=torch.int64, device="cuda")
    for a, b in ((dr, ds), (ds, dr)):
        ctx.join_count(a, b, cnt)
        ctx.sync()
        assert int(cnt.item()) == want
