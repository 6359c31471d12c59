"""Batched splits of one to many tiles, on both sides of the 256 tiles whose counts one workgroup scans, against the oracle.

Every shape (tiles of 1024, 2048 and 4096 keys), 1 to 256 buckets, both widths, with and without values and starts.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", range(6))
def test_split_jobs(torch_gpu, ctx, edpp, orc, shape):
    torch = torch_gpu
    jobs, checks = [], []
    lengths = (1, 1023, 2049, 40_000, 1024 * 256, 1024 * 256 + 1, 2048 * 256, 2048 * 256 + 1, 4096 * 256, 4096 * 256 + 1)
    for i, n in enumerate(lengths):
        for buckets in (256, (1, 2, 16, 64)[i % 4]):
            keys, vals = orc.gen_split_keys(n, buckets, i % 2, i)
            wide, kv = (i + buckets // 256) % 2 == 0, i % 3 != 0
            if wide:
                keys = keys.astype(np.int64) | (np.arange(n, dtype=np.int64) << 32)
            dk, dv = torch.from_numpy(keys).cuda(), torch.from_numpy(vals).cuda()
            out, vout = torch.full_like(dk, -1), torch.full_like(dv, -1)
            start = torch.full((buckets,), -1, dtype=torch.int32, device="cuda")
            jobs.append(edpp.make_job(edpp.JOB_SPLIT, n, dk, out, 8 if wide else 4, buckets=buckets,
                                      vals_in=dv if kv else None, vals_out=vout if kv else None, aux=start))
            checks.append((keys, vals, buckets, kv, dk, dv, out, vout, start))
    batch = edpp.Batch(ctx, jobs)
    batch.set_shape(shape)
    for _ in range(2):
        for c in checks:
            c[6].fill_(-1)
        batch.run()
        ctx.sync()
        for keys, vals, buckets, kv, _, _, out, vout, start in checks:
            ko, vo, so = orc.split(keys, buckets, vals)
            assert np.array_equal(out.cpu().numpy(), ko) and np.array_equal(start.cpu().numpy(), so)
            if kv:
                assert np.array_equal(vout.cpu().numpy(), vo)


@pytest.mark.parametrize("n", [1, 2, 8191, 8193, 65_536 + 2])
def test_wide_gather_jobs(torch_gpu, ctx, edpp, n):
    """Whole and ragged tiles of 8-byte values, some indices out of range."""
    torch = torch_gpu
    rng = np.random.default_rng(n)
    src, at = rng.integers(-2**62, 2**62, n), rng.integers(-2, n + 2, n).astype(np.int32)
    ds, da = torch.from_numpy(src).cuda(), torch.from_numpy(at).cuda()
    out = torch.full_like(ds, 5)
    for shape in range(6):
        out.fill_(5)
        batch = edpp.Batch(ctx, [edpp.make_job(edpp.JOB_GATHER, n, ds, out, 8, idx=da)])
        batch.set_shape(shape)
        batch.run()
        ctx.sync()
        ok = (at >= 0) & (at < n)
        assert np.array_equal(out.cpu().numpy(), np.where(ok, src[np.where(ok, at, 0)], 5))
