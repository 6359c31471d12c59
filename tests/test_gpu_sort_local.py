"""Sorts of 2^26 keys and more, which end segment by segment in LDS, against a stable sort in 64 bits.

Lengths on both sides of the threshold and of a change of the segment count; keys that are spread evenly, over 9/10 or
half of the range, with two long segments that 2^14 samples do not show, with segments just past what fits, all equal,
and already sorted.
"""
import pytest

pytestmark = pytest.mark.gpu

MIN = 1 << 26
FIT = 69 * 64  # keys of a segment that one workgroup orders in LDS
STEP = (FIT - FIT // 16 + 1) << 14  # from here on 2^15 segments


def _keys(torch, kind, n, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.randint(-(1 << 31), 1 << 31, (n,), generator=g, device="cuda", dtype=torch.int32)
    if kind == "half":
        k &= 0x7FFFFFFF
    elif kind == "most":  # segments a ninth longer
        k = (k.to(torch.int64) * 9 // 10).to(torch.int32)
    elif kind == "hot":  # 0.03% of the keys in two segments: about five samples
        m = n // 6000
        k[100_001:100_001 + m] = (k[100_001:100_001 + m] & 0x3FFF) | 0x12340000
        k[-m:] = (k[-m:] & 0x1) | 0x7A5B0000
    elif kind == "full":  # segments of exactly what fits, one key less and one key more
        low = k[:3 * FIT] & 0x3FFF
        k = torch.where((k >> 18) == (0x20000000 >> 18), k ^ 0x40000000, k)
        k = torch.where((k >> 18) == (0x30000000 >> 18), k ^ 0x40000000, k)
        k[::n // FIT][:FIT] = 0x20000000 | low[:FIT]
        k[1::n // (FIT + 1)][:FIT + 1] = 0x30000000 | low[FIT:2 * FIT + 1]
    elif kind == "equal":
        k.fill_(-7)
    elif kind == "sorted":
        k = torch.sort(k).values
    elif kind == "low":  # few low bits: many equal keys in a segment
        k &= ~0xFF00FF
    return k


def _check(torch, ctx, keys, signed, values, in_place):
    n = keys.numel()
    u = keys.to(torch.int64) if signed else keys.to(torch.int64) & 0xFFFFFFFF
    want, order = torch.sort(u, stable=True)
    vals = torch.arange(n, dtype=torch.int32, device="cuda").flip(0).contiguous() if values else None
    out = keys if in_place else torch.full_like(keys, 3)
    vout = (vals if in_place else torch.full_like(vals, 3)) if values else None
    expect = vals[order] if values else None
    ctx.sort(keys, out, vals, vout, signed=signed)
    got = out.to(torch.int64) if signed else out.to(torch.int64) & 0xFFFFFFFF
    assert torch.equal(got, want)
    if values:
        assert torch.equal(vout, expect)


@pytest.mark.parametrize("n", [MIN - 1, MIN, STEP - 1, STEP, 2 * STEP + 5])
@pytest.mark.parametrize("signed,values", [(False, True), (True, False)])
def test_lengths(torch_gpu, ctx, n, signed, values):
    _check(torch_gpu, ctx, _keys(torch_gpu, "even", n, n % 1000), signed, values, False)


@pytest.mark.parametrize("kind", ["half", "most", "hot", "full", "equal", "sorted", "low"])
@pytest.mark.parametrize("values", [True, False])
def test_distributions(torch_gpu, ctx, kind, values):
    for signed, in_place in ((False, False), (True, True)):
        _check(torch_gpu, ctx, _keys(torch_gpu, kind, MIN + 4099, 5), signed, values, in_place)


def test_replayed(torch_gpu, edpp):
    """A captured sort replayed on keys of both kinds, with eager sorts between."""
    torch = torch_gpu
    n = MIN + 99
    s = torch.cuda.Stream()
    with torch.cuda.stream(s), edpp.Context(0, stream=s.cuda_stream) as c:
        even, equal = _keys(torch, "even", n, 1), _keys(torch, "equal", n, 2)
        buf, out, again = even.clone(), torch.empty_like(even), torch.empty_like(even)
        c.sort(buf, out)
        s.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            c.sort(buf, out)
        for src in (even, equal, even):
            buf.copy_(src)
            out.fill_(1)
            graph.replay()
            s.synchronize()
            assert torch.equal(out.to(torch.int64) & 0xFFFFFFFF, torch.sort(src.to(torch.int64) & 0xFFFFFFFF).values)
            c.sort(src, again)
            s.synchronize()
            assert torch.equal(out, again)
        del graph
