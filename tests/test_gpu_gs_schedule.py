"""What the library reports and does about gathers and scatters that may go by windows of the random side."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wide", [False, True])
def test_default_candidate_of_large_calls_is_none(torch_gpu, ctx, edpp, wide):
    torch = torch_gpu
    n = (1 << 29) // (8 if wide else 4)
    buf = torch.empty(n + 16, dtype=torch.int64 if wide else torch.int32, device="cuda")
    out, idx = torch.empty_like(buf), torch.empty(n + 16, dtype=torch.int32, device="cuda")
    for op in (edpp.OP_GATHER, edpp.OP_SCATTER):
        def cand(m, shift=0):
            return ctx.default_candidate(edpp.make_call(op, m, buf, out, 8 if wide else 4, idx=idx[shift:]))
        assert cand(n) == -1
        assert cand(n - 1) >= 0  # below 512 MiB the pass loop runs
        assert cand(n, 1) >= 0   # and with indices off 16 bytes
