"""Which histogram scan a batch's split jobs get: one workgroup only where its chain of readings is short or hidden."""
import pytest

pytestmark = pytest.mark.gpu


def _splits(torch, edpp, n, count, buckets, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    step = -(-n // 64) * 64
    keys = torch.randint(-2**31, 2**31, (step * count,), device="cuda", dtype=torch.int32, generator=g)
    vals = torch.arange(step * count, device="cuda", dtype=torch.int32)
    out, vout = torch.full_like(keys, -1), torch.full_like(vals, -1)
    jobs = [edpp.make_job(edpp.JOB_SPLIT, n, keys[j * step:j * step + n], out[j * step:j * step + n], 4, buckets=buckets,
                          vals_in=vals[j * step:j * step + n], vals_out=vout[j * step:j * step + n])
            for j in range(count)]
    return jobs, step, keys, vals, out, vout


# tiles of 2048 keys: 256 lanes read 16 words each of 16 tiles of 256 buckets, or of 128 tiles of 32
@pytest.mark.parametrize("n,buckets,one", [(16 * 2048, 256, True), (16 * 2048 + 1, 256, False), (128 * 2048, 32, True),
                                           (128 * 2048 + 1, 32, False), (256 * 2048, 16, True), (256 * 2048, 256, False),
                                           (256 * 2048, 2, True), (256 * 2048 + 1, 2, False)])
def test_jobs_by_themselves(torch_gpu, ctx, edpp, n, buckets, one):
    torch = torch_gpu
    jobs, _, keys, vals, out, vout = _splits(torch, edpp, n, 1, buckets)
    batch = edpp.Batch(ctx, jobs)
    scans = batch.info()["hscan_tiles"]
    assert (scans == 1) if one else (scans == -(-(buckets * -(-n // 2048)) // 4096))
    batch.run()
    ctx.sync()
    order = torch.sort(keys[:n] & (buckets - 1), stable=True).indices
    assert torch.equal(out[:n], keys[:n][order]) and torch.equal(vout[:n], vals[:n][order])


def test_long_batches_take_one_workgroup_per_job(torch_gpu, ctx, edpp):
    torch = torch_gpu
    n, count = 100_000, 128
    jobs, step, keys, vals, out, vout = _splits(torch, edpp, n, count, 256)
    batch = edpp.Batch(ctx, jobs)
    assert batch.info()["hscan_tiles"] == count
    batch.run()
    ctx.sync()
    for j in (0, 63, 127):
        s = slice(j * step, j * step + n)
        order = torch.sort(keys[s] & 255, stable=True).indices
        assert torch.equal(out[s], keys[s][order]) and torch.equal(vout[s], vals[s][order])


def test_a_job_of_256_tiles_is_no_slower_than_a_longer_one(torch_gpu, ctx, edpp):
    torch = torch_gpu

    def fastest(n):
        batch = edpp.Batch(ctx, _splits(torch, edpp, n, 1, 256)[0])
        batch.run()
        return min(batch.run(timed=True) for _ in range(10))

    assert fastest(256 * 2048) < 1.5 * fastest(260 * 2048)
