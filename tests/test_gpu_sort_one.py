"""Sorts by one workgroup (up to 12,288 keys) and just past it, against the oracle: lengths around a row of 64, a row per
wave and the two limits; bit ranges of one to four passes; keys in place; few distinct keys."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 65, 1000, 1024, 1025, 2113, 4096, 8191, 8192, 8193, 12_287, 12_288, 12_289])
@pytest.mark.parametrize("bits", [(0, 32), (0, 1), (3, 12), (5, 32), (31, 32), (8, 24)])
@pytest.mark.parametrize("signed", [False, True])
def test_one_workgroup_sort(torch_gpu, ctx, orc, n, bits, signed):
    torch = torch_gpu
    for few in (False, True):
        keys = orc.gen_i32(n, n + bits[0])
        if few:
            keys = (keys & 0x3).astype(np.int32) - 2
        vals = np.arange(n, dtype=np.int32)[::-1].copy()
        ko, vo = orc.sort(keys, vals, bits[0], bits[1], signed)
        dk, dv = torch.from_numpy(keys).cuda(), torch.from_numpy(vals).cuda()
        out, vout = torch.full_like(dk, 3), torch.full_like(dv, 3)
        ctx.sort(dk, out, dv, vout, begin_bit=bits[0], end_bit=bits[1], signed=signed)
        assert np.array_equal(out.cpu().numpy(), ko) and np.array_equal(vout.cpu().numpy(), vo)
        only = torch.full_like(dk, 3)
        ctx.sort(dk, only, begin_bit=bits[0], end_bit=bits[1], signed=signed)
        assert np.array_equal(only.cpu().numpy(), ko)
        ctx.sort(dk, dk, dv, dv, begin_bit=bits[0], end_bit=bits[1], signed=signed)
        assert np.array_equal(dk.cpu().numpy(), ko) and np.array_equal(dv.cpu().numpy(), vo)
