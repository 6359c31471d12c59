"""Splits and sorts of few tiles, whose scatter adds up the tiles' counts itself, against the oracle.

Lengths around one tile of 2048 keys and the bounds of the short form: 1024 tiles, 16,384 counts that the lanes read at
once (64 tiles at 256 buckets), 65,536 counts (256 tiles at 256 buckets).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("buckets,n", [(b, n) for b, ns in (
    (2, (1, 2047, 2049, 2048 * 1024, 2048 * 1024 + 1)),
    (8, (2048, 4097, 2048 * 1024 - 3)),
    (16, (1, 2048 * 32 + 5, 2048 * 1024, 2048 * 1024 + 1)),
    (32, (2048 * 257, 2048 * 512, 2048 * 512 + 9)),
    (256, (1, 2047, 2048 * 64, 2048 * 65 + 1, 2048 * 256, 2048 * 256 + 1)),
    (1024, (3000, 2048 * 128 + 1, 2048 * 513)),
) for n in ns])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("values", [False, True])
def test_short_split(torch_gpu, ctx, orc, buckets, n, wide, values):
    torch = torch_gpu
    keys, vals = orc.gen_split_keys(n, buckets, n % 2, n % 1000 + buckets)
    if wide:
        keys = keys.astype(np.int64) | (np.arange(n, dtype=np.int64) << 32)
    ko, vo, start = orc.split(keys, buckets, vals)
    dk = torch.from_numpy(keys).cuda()
    out = torch.full_like(dk, -1)
    dv = torch.from_numpy(vals).cuda() if values else None
    vout = torch.full_like(dv, -1) if values else None
    st = torch.full((buckets,), -1, dtype=torch.int32, device="cuda")
    ctx.split(dk, out, buckets, dv, vout, st, wide=wide)
    assert np.array_equal(out.cpu().numpy(), ko) and np.array_equal(st.cpu().numpy(), start)
    if values:
        assert np.array_equal(vout.cpu().numpy(), vo)


def test_short_split_with_a_long_tile_asked(torch_gpu, ctx, orc):
    """A tile of 1024 keys per bucket asks for a matrix of one column: the counts must not need its room."""
    torch = torch_gpu
    n, B = 2048 * 200 + 17, 256
    keys, vals = orc.gen_split_keys(n, B, 0, 9)
    ko, vo, _ = orc.split(keys, B, vals)
    dk, dv = torch.from_numpy(keys).cuda(), torch.from_numpy(vals).cuda()
    out, vout = torch.empty_like(dk), torch.empty_like(dv)
    ctx.set_tuning(split_ipt=8, split_tile_mult=1024)
    try:
        ctx.split(dk, out, B, dv, vout, strategy=1)
    finally:
        ctx.set_tuning()
    assert np.array_equal(out.cpu().numpy(), ko) and np.array_equal(vout.cpu().numpy(), vo)


@pytest.mark.parametrize("n", [1, 2048, 4097, 131_072, 2048 * 256, 2048 * 256 + 1])
@pytest.mark.parametrize("signed", [False, True])
def test_short_sort(torch_gpu, ctx, orc, n, signed):
    torch = torch_gpu
    keys = orc.gen_i32(n, 77 + n % 13)
    vals = np.arange(n, dtype=np.int32)
    ko, vo = orc.sort(keys, vals, 0, 32, signed)
    dk, dv = torch.from_numpy(keys).cuda(), torch.from_numpy(vals).cuda()
    out, vout = torch.empty_like(dk), torch.empty_like(dv)
    ctx.sort(dk, out, dv, vout, signed=signed)
    assert np.array_equal(out.cpu().numpy(), ko) and np.array_equal(vout.cpu().numpy(), vo)
    ctx.sort(dk, dk, signed=signed)
    assert np.array_equal(dk.cpu().numpy(), ko)
