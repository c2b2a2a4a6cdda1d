"""The causal attention kernel of prompt chunks (janus_amd/csrc/prefill.hip),
called by itself through its internal entry, against 64 bits: what a layer's
norm would spread over a whole row (a NaN in one head dim) or hide behind a
binary16 rounding is seen here where it arises.
"""
import ctypes as C
import math

import pytest
import torch

from janus_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# heads, KV heads, head size: four and one heads per KV head, and both head sizes
LAYOUTS = [(8, 2, 128), (4, 4, 128), (4, 1, 64), (4, 2, 64)]


def _prompt_attention(engine, q, k, v, p0):
    """Rows p0 .. p0 + n - 1 of one sequence (q [n][heads][hd]) over its cache k, v."""
    f = getattr(engine.lib, "_ZN5janus24prefill_attention_launchEP9janus_ctxPKfPKvS5_iPvjjjjjfi")
    f.argtypes = [C.c_void_p] * 4 + [C.c_int, C.c_void_p] + [C.c_uint] * 5 + [C.c_float, C.c_int]
    f.restype = C.c_int
    n, heads, hd = q.shape
    assert k.shape == v.shape == (p0 + n, k.shape[1], hd)
    out = torch.full_like(q, 7.0)
    dt = ops.DT_F16 if k.dtype == torch.float16 else ops.DT_F32
    engine._check(f(engine.ctx, q.data_ptr(), k.data_ptr(), v.data_ptr(), dt, out.data_ptr(), n, p0, heads, k.shape[1],
                    hd, 1.0 / math.sqrt(hd), 0))
    return out


def _decode_attention(engine, q, k, v, p0):
    """The same rows through the decode kernels, one call each."""
    out = torch.empty_like(q)
    base = torch.zeros(1, dtype=torch.int32, device=DEV)
    lens = torch.arange(p0 + 1, p0 + q.shape[0] + 1, dtype=torch.int32, device=DEV)
    for r in range(q.shape[0]):
        ops.compute_attention(engine, q[r:r + 1], k, v, out[r:r + 1], 1, 0, p0 + r + 1, q.shape[1], k.shape[1],
                              q.shape[2], base, lens[r:r + 1], p0 + r + 1)
    return out


def _exact(q, k, v, p0):
    """In 64 bits; positions a row does not see take no part, whatever they hold."""
    q, k, v = q.double().cpu(), k.double().cpu(), v.double().cpu()
    n, heads, hd = q.shape
    rep = heads // k.shape[1]
    out = torch.empty_like(q)
    for r in range(n):
        kk, vv = (t[:p0 + r + 1].repeat_interleave(rep, 1) for t in (k, v))
        p = torch.softmax((q[r] * kk).sum(-1) / math.sqrt(hd), 0)
        out[r] = (p[..., None] * vv).sum(0)
    return out


def _inputs(seed, n, p0, heads, kv_heads, hd, kv):
    g = torch.Generator().manual_seed(seed)
    q = torch.randn(n, heads, hd, generator=g)
    k, v = (torch.randn(p0 + n, kv_heads, hd, generator=g).to(kv) for _ in range(2))
    return q.to(DEV), k.to(DEV), v.to(DEV)


def _same_where_finite(got, want):
    """The same infinities and NaN, and 1e-5 of the largest value elsewhere
    (binary32 sums of 120 terms)."""
    got = got.double().cpu()
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    ok = want.isfinite()
    assert float((got[ok] - want[ok]).abs().max() / want[ok].abs().max()) <= 1e-5


@pytest.mark.parametrize("kv", [torch.float16, torch.float32])
@pytest.mark.parametrize("heads,kv_heads,hd", LAYOUTS)
def test_nonfinite_values_reach_their_dim_of_the_rows_that_see_them(engine, heads, kv_heads, hd, kv):
    """Infinities and NaN in single dims of V, in tiles that all rows of a
    wavefront see and in the last ones, with positions before the chunk and
    without: an infinity stays one (of its sign), in its dim, from its position on."""
    for n, p0 in ((70, 0), (40, 50)):
        q, k, v = _inputs(n, n, p0, heads, kv_heads, hd, kv)
        v[5, 0, 3] = float("inf")
        v[p0 + 20, 0, 40] = float("-inf")
        v[p0 + 37, kv_heads - 1, hd - 1] = float("nan")
        v[p0 + n - 1, 0, 9] = float("inf")
        _same_where_finite(_prompt_attention(engine, q, k, v, p0), _exact(q, k, v, p0))


@pytest.mark.parametrize("kv", [torch.float16, torch.float32])
@pytest.mark.parametrize("heads,kv_heads,hd", LAYOUTS)
def test_nan_scores_are_not_passed_over(engine, heads, kv_heads, hd, kv):
    """NaN in K rows with V finite. One such row: NaN from its position on.
    The whole first tile: NaN for every later row, whose other scores are
    finite. Rows without any other score (also a NaN q) are what the decode
    kernels make of them."""
    n, rep = 75, heads // kv_heads
    q, k, v = _inputs(1, n, 0, heads, kv_heads, hd, kv)
    k[2, 0, 1] = float("nan")
    _same_where_finite(_prompt_attention(engine, q, k, v, 0), _exact(q, k, v, 0))
    k[:32, 0] = float("nan")
    got, one = _prompt_attention(engine, q, k, v, 0), _decode_attention(engine, q, k, v, 0)
    assert bool(got[32:, :rep].isnan().all()) and bool(got[:, rep:].isfinite().all())
    assert torch.equal(got[:32, :rep], one[:32, :rep])
    q, k, v = _inputs(1, n, 0, heads, kv_heads, hd, kv)
    want = _prompt_attention(engine, q, k, v, 0)
    q[70, heads - 1] = float("nan")
    want[70, heads - 1] = _decode_attention(engine, q, k, v, 0)[70, heads - 1]
    assert torch.equal(_prompt_attention(engine, q, k, v, 0), want)


@pytest.mark.parametrize("heads,kv_heads,hd", LAYOUTS)
def test_infinite_keys_and_queries(engine, heads, kv_heads, hd):
    """Infinities in K of a binary16 cache (overflowed) and in q, where q runs
    in parts: a score of minus infinity takes its position out, one of plus
    infinity makes the row NaN, as q in one piece has it."""
    n = 75
    q, k, v = _inputs(2, n, 0, heads, kv_heads, hd, torch.float16)
    k[2, 0, 1] = float("-inf")
    k[40, 0, 7] = float("inf")
    q[:, 0, 1], q[:, 0, 7] = q[:, 0, 1].abs(), -q[:, 0, 7].abs()      # head 0: minus infinity both times
    want = _exact(q, k, v, 0)
    assert bool(want[:, 0].isfinite().all()) and (heads == kv_heads or bool(want.isnan().any()))
    _same_where_finite(_prompt_attention(engine, q, k, v, 0), want)
    q, k, v = _inputs(3, n, 0, heads, kv_heads, hd, torch.float16)
    k[:, 0, 5] = -k[:, 0, 5].abs()
    k[9, 0, 5] = 1.0
    q[4, 0, 5], q[50, 0, 5] = float("inf"), float("-inf")
    want = _exact(q, k, v, 0)
    want[4, 0] = _decode_attention(engine, q, k, v, 0)[4, 0].double().cpu()   # no score but minus infinity
    _same_where_finite(_prompt_attention(engine, q, k, v, 0), want)


@pytest.mark.parametrize("kv", [torch.float16, torch.float32])
@pytest.mark.parametrize("heads,kv_heads,hd", LAYOUTS)
@pytest.mark.parametrize("q_scale,k_scale", [(2.0, 1.0), (2.0 ** -10, 2.0 ** 10), (2.0 ** -14, 2.0 ** 12), (2.0 ** 40, 2.0 ** -12)])
def test_as_close_to_64_bits_as_the_decode_kernels(engine, heads, kv_heads, hd, kv, q_scale, k_scale):
    """The root-mean-square error over a prompt's rows is that of the decode
    kernels on the same rows, which hold q and the probabilities in binary32
    (1.25 of it: the ratio of two samples of rounding errors), whatever the
    sizes of q and K. A huge q leaves one position per row: its V exactly."""
    ours = theirs = 0.0
    for n, p0 in ((130, 0), (60, 100)):
        q, k, v = _inputs(n + hd, n, p0, heads, kv_heads, hd, torch.float32)
        q, k, v = q * q_scale, (k * k_scale).to(kv), v.to(kv)
        want = _exact(q, k, v, p0)
        got, one = (f(engine, q, k, v, p0).double().cpu() for f in (_prompt_attention, _decode_attention))
        ours += float((got - want).square().sum())
        theirs += float((one - want).square().sum())
    assert ours <= 1.25 ** 2 * theirs, math.sqrt(ours / theirs)
