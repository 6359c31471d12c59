"""Direct gathers of 8-byte values, two per lane and step: lengths around a step and a chunk, whole and several passes,
local and random indices, some out of range, against numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unroll", [1, 2, 4, 8])
@pytest.mark.parametrize("passes", [1, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 1023, 1025, 4096, 4098, 8193, 100_003])
def test_wide_gather(torch_gpu, ctx, unroll, passes, n):
    torch = torch_gpu
    rng = np.random.default_rng(n + unroll)
    src = torch.from_numpy(rng.integers(-2**62, 2**62, n)).cuda()
    local = (np.arange(n) // 1000 * 1000 + rng.integers(0, 1000, n)).clip(0, n - 1)
    wild = rng.integers(-3, n + 3, n)
    ctx.set_tuning(gs_unroll=unroll)
    try:
        for at in (local, wild):
            at = at.astype(np.int32)
            out = torch.full_like(src, 7)
            ctx.gather(src, out, torch.from_numpy(at).cuda(), passes=passes, wide=True)
            ok = (at >= 0) & (at < n)
            want = np.where(ok, src.cpu().numpy()[np.where(ok, at, 0)], 7)
            assert np.array_equal(out.cpu().numpy(), want)
    finally:
        ctx.set_tuning()
