"""GPU parity of the small-M MFMA GEMM (janus_gemm_auto with 2..64 rows of
binary16 activations).

The reference has no correct quantised product for M > 1 (it hands quantised
bytes to its f16 GEMM, crates/janus-engine/src/compute/ops/quantized.rs:77-90),
so parity is the invariant "GEMM(M) == M stacked GEMV(1)": every row must
match the M=1 kernel on the same binary16 row, and both must match an f64
product of the bit-exact dequantised weights within
|y - y64| <= 2e-5 * sum_i |w_i x_i|   (exact products, fp32 accumulation).
"""
import threading

import numpy as np
import pytest
import torch

from janus_amd import ops, synth
from oracle import oracle as O

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
GEN = {2: synth.random_q4_0, 8: synth.random_q8_0, 12: synth.random_q4_k, 13: synth.random_q5_k}


def _weight(engine, ggml_type, n, k, seed):
    rng = np.random.default_rng(seed)
    if ggml_type in GEN:
        raw = GEN[ggml_type](rng, n, k)
    else:
        raw = synth.f16_bits(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02))
    return raw, ops.GpuTensor(engine, ggml_type, n, k, raw)


def _acts(rows, k, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(rows, k, generator=g).to(torch.float16)


def _check_against_f64(y, wf, a16):
    x = a16.float().numpy().astype(np.float64)
    w = wf.astype(np.float64)
    ref = x @ w.T
    bound = 2e-5 * (np.abs(x) @ np.abs(w).T) + 1e-30
    err = np.abs(y.astype(np.float64) - ref)
    assert np.all(err <= bound), float(np.max(err / bound))


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13, 1])
@pytest.mark.parametrize("rows", [2, 7, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(96, 256), (200, 512), (4096, 4096), (1024, 14336)])
def test_mfma_gemm_matches_stacked_gemv_and_f64(engine, ggml_type, rows, n, k):
    raw, w = _weight(engine, ggml_type, n, k, 100 + ggml_type + n)
    a16 = _acts(rows, k, rows + n)
    a = a16.to(DEV)
    c = torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    stacked = torch.empty(rows, n, device=DEV)
    for r in range(rows):
        ops.gemm_auto(engine, a[r].contiguous(), w, stacked[r], 1, 1, k, n)
    torch.cuda.synchronize()
    got = c.cpu().numpy()
    wf = w.dequant().cpu().numpy()
    _check_against_f64(got, wf, a16)
    _check_against_f64(stacked.cpu().numpy(), wf, a16)


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13])
@pytest.mark.parametrize("rows", [32, 48, 64])
@pytest.mark.parametrize("n,k", [(6144, 4096), (4096, 14336)])
def test_pipelined_gemm_shapes_match_f64(engine, ggml_type, rows, n, k):
    """Shapes whose workgroups run several K passes take the cross-pass
    pipelined kernel (A double-buffered in LDS, next-pass weights in flight):
    one and two 32-row M tiles, every quantised format, K split over
    workgroups. Repeated calls are bitwise equal."""
    raw, w = _weight(engine, ggml_type, n, k, 300 + ggml_type + rows)
    a16 = _acts(rows, k, 7 * rows + n)
    a = a16.to(DEV)
    outs = []
    for _ in range(2):
        c = torch.empty(rows, n, device=DEV)
        ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
        outs.append(c.cpu())
    assert torch.equal(outs[0], outs[1])
    _check_against_f64(outs[0].numpy(), w.dequant().cpu().numpy(), a16)


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13])
@pytest.mark.parametrize("rows", [2, 8, 9, 16, 17])
@pytest.mark.parametrize("n,k", [(6144, 4096), (6176, 4352)])
def test_pipelined_gemm_row_trimmed_forms(engine, ggml_type, rows, n, k):
    """The pipelined kernel's forms for at most 8 and 16 rows (the scale FMAs,
    the stage and the stores stop at the row count), at their edges, with a
    partial row-group tile and a K split."""
    raw, w = _weight(engine, ggml_type, n, k, 600 + ggml_type + rows)
    a16 = _acts(rows, k, 13 * rows + n)
    c = torch.full((rows + 1, n), 7.0, device=DEV)
    ops.gemm_auto(engine, a16.to(DEV), w, c, rows, 1, k, n)
    torch.cuda.synchronize()
    assert bool((c[rows] == 7.0).all())
    _check_against_f64(c[:rows].cpu().numpy(), w.dequant().cpu().numpy(), a16)


@pytest.mark.parametrize("ggml_type", [2, 8])
@pytest.mark.parametrize("rows", [32, 40])
def test_pipelined_gemm_ragged_k_and_partial_tile(engine, ggml_type, rows):
    """k = 4160 leaves a 64-wide last pass (K-tail chunks clamped, not computed)
    and n = 6176 leaves a last tile with one active row group of four (the
    others stream a real group and discard it)."""
    n, k = 6176, 4160
    raw, w = _weight(engine, ggml_type, n, k, 500 + ggml_type + rows)
    a16 = _acts(rows, k, 11 * rows)
    a = a16.to(DEV)
    c = torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    torch.cuda.synchronize()
    _check_against_f64(c.cpu().numpy(), w.dequant().cpu().numpy(), a16)


@pytest.mark.parametrize("ggml_type", [2, 12])
def test_mfma_gemm_is_deterministic_under_split_k(engine, ggml_type):
    n, k, rows = 4096, 4096, 32          # few row tiles: the product is split over K
    _, w = _weight(engine, ggml_type, n, k, 7)
    a = _acts(rows, k, 3).to(DEV)
    outs = []
    for _ in range(3):
        c = torch.empty(rows, n, device=DEV)
        ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
        outs.append(c.cpu())
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[1], outs[2])


def test_mfma_gemm_residual_and_f16_output(engine):
    n, k, rows = 640, 1024, 5
    _, w = _weight(engine, 2, n, k, 21)
    a16 = _acts(rows, k, 4)
    a = a16.to(DEV)
    base = torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, base, rows, 1, k, n)
    resid = torch.randn(rows, n, device=DEV)
    out = torch.empty(rows, n, device=DEV)
    ops.gemm_residual(engine, a, w, resid, out, rows)
    torch.cuda.synchronize()
    assert torch.equal(out, base + resid)
    inplace = resid.clone()
    ops.gemm_residual(engine, a, w, inplace, inplace, rows)
    assert torch.equal(inplace, base + resid)
    h = torch.empty(rows, n, device=DEV, dtype=torch.float16)
    ops.gemm_auto(engine, a, w, h, rows, 1, k, n)
    assert torch.equal(h, base.to(torch.float16))


def test_mfma_gemm_q4_0_odd_block_count(engine):
    # k / 32 odd: the last 64-wide tile chunk carries one zero block
    n, k, rows = 70, 96, 3
    raw, w = _weight(engine, 2, n, k, 5)
    a16 = _acts(rows, k, 6)
    c = torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a16.to(DEV), w, c, rows, 1, k, n)
    torch.cuda.synchronize()
    _check_against_f64(c.cpu().numpy(), O.dequant(2, raw, n, k), a16)


def test_f32_activations_keep_the_reference_dtype(engine):
    # f32 rows go through the M=1 kernels row by row: bit-identical to single calls
    n, k, rows = 128, 512, 3
    _, w = _weight(engine, 8, n, k, 8)
    a = torch.randn(rows, k, device=DEV)
    c = torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    for r in range(rows):
        y = torch.empty(n, device=DEV)
        ops.gemm_auto(engine, a[r].contiguous(), w, y, 1, 1, k, n)
        assert torch.equal(y, c[r])


def _check_f32_against_f64(y, wf, x, bound=1e-5):
    x, w = x.double().cpu(), torch.from_numpy(wf).double()
    err = (y.double().cpu() - x @ w.T).abs()
    assert bool((err <= bound * (x.abs() @ w.abs().T) + 1e-30).all()), float((err / (x.abs() @ w.abs().T)).max())


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13, 1])
@pytest.mark.parametrize("rows", [3, 4, 8, 9, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,k", [(33, 256), (200, 512), (4096, 1280), (1000, 4352)])
def test_f32_rows_on_mfma_match_f64(engine, ggml_type, rows, n, k):
    """binary32 activations as three exact bfloat16 parts: at most 8, 16 and 32
    rows of an M tile, two M tiles, partial row groups and K passes, K split over workgroups. The
    parts and products are exact, so the M = 1 kernels' bound for binary32
    sums holds (1e-5 of sum |w x|); values from 2^-40 to 2^20 keep their
    digits, and a repeated call gives the same bits."""
    _, w = _weight(engine, ggml_type, n, k, 700 + ggml_type + n)
    g = torch.Generator().manual_seed(rows + n)
    x = torch.randn(rows, k, generator=g) * torch.exp2(torch.randint(-40, 21, (rows, 1), generator=g).float())
    x[:, ::7] *= 2.0 ** -12
    a, c, again = x.to(DEV), torch.empty(rows, n, device=DEV), torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    ops.gemm_auto(engine, a, w, again, rows, 1, k, n)
    assert torch.equal(c, again)
    _check_f32_against_f64(c, w.dequant().cpu().numpy(), x)


@pytest.mark.parametrize("ggml_type,n,k", [(2, 70, 96), (8, 70, 96), (8, 96, 160), (2, 6176, 4160), (1, 70, 1032)])
def test_f32_rows_on_mfma_ragged_k(engine, ggml_type, n, k):
    """K that ends inside a pass, a 64-wide chunk, or (F16) a 16-wide one."""
    _, w = _weight(engine, ggml_type, n, k, 900 + n + k)
    x = torch.randn(5, k, generator=torch.Generator().manual_seed(k))
    resid = torch.randn(5, n, device=DEV)
    base, out = torch.empty(5, n, device=DEV), resid.clone()
    ops.gemm_auto(engine, x.to(DEV), w, base, 5, 1, k, n)
    ops.gemm_residual(engine, x.to(DEV), w, out, out, 5)
    assert torch.equal(out, base + resid)
    h = torch.empty(5, n, device=DEV, dtype=torch.float16)
    ops.gemm_auto(engine, x.to(DEV), w, h, 5, 1, k, n)
    assert torch.equal(h, base.to(torch.float16))
    _check_f32_against_f64(base, w.dequant().cpu().numpy(), x)


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13, 1])
def test_f32_rows_with_infinities_and_nan_match_single_rows(engine, ggml_type):
    """Rows holding an infinity or a NaN: no finite value where a single call
    gives none, the same infinity where it gives one (Q8_0's row kernel turns
    infinities into NaN through its offset; here they stay), a NaN row all
    NaN, and the other rows are left alone."""
    n, k = 256, 512
    _, w = _weight(engine, ggml_type, n, k, 31)
    x = torch.randn(6, k, generator=torch.Generator().manual_seed(2))
    x[1, 77] = float("inf")
    x[2, 300] = float("-inf")
    x[4, 5] = float("nan")
    a, c = x.to(DEV), torch.empty(6, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, 6, 1, k, n)
    for r in (1, 2, 4):
        y = torch.empty(n, device=DEV)
        ops.gemm_auto(engine, a[r].contiguous(), w, y, 1, 1, k, n)
        assert torch.equal(y.isfinite(), c[r].isfinite())
        assert torch.equal(y[y.isinf()], c[r][y.isinf()])
        assert r != 4 or bool(c[r].isnan().all())
    keep = [0, 3, 5]
    _check_f32_against_f64(c[keep], w.dequant().cpu().numpy(), x[keep])


def test_f32_rows_with_nonfinite_f16_weights_match_single_rows(engine):
    """A binary16 weight with an infinity has no exact parts: such a weight
    keeps the row kernels, bit for bit."""
    n, k, rows = 128, 512, 7
    rng = np.random.default_rng(6)
    bits = synth.f16_bits(rng.standard_normal((n, k), dtype=np.float32) * np.float32(0.02)).copy()
    bits.reshape(n, k)[17, 3], bits.reshape(n, k)[40, 500] = 0x7C00, 0x7E00
    w = ops.GpuTensor(engine, 1, n, k, bits)
    a, c = torch.randn(rows, k, device=DEV), torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    for r in range(rows):
        y = torch.empty(n, device=DEV)
        ops.gemm_auto(engine, a[r].contiguous(), w, y, 1, 1, k, n)
        assert torch.equal(y.view(torch.int32), c[r].view(torch.int32))


def test_f32_rows_first_used_inside_a_capture(engine):
    """The first call on a weight may come inside a stream capture: nothing
    can be allocated there, so the row kernels run; a later eager call builds
    the tile copy. Both match f64, and every replay repeats its result."""
    n, k, rows = 1000, 1024, 9
    eng = ops.ComputeEngine(0)
    _, w = _weight(eng, 2, n, k, 77)
    a, c = torch.randn(rows, k, device=DEV), torch.empty(rows, n, device=DEV)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        eng.bind_stream(s)
        ops.gemm_auto(eng, a, w, c, rows, 1, k, n)
    eng.bind_stream(torch.cuda.current_stream())
    eager = torch.empty(rows, n, device=DEV)
    wf = w.dequant().cpu().numpy()
    for _ in range(3):
        c.zero_()
        g.replay()
        torch.cuda.synchronize()
        _check_f32_against_f64(c, wf, a)
        ops.gemm_auto(eng, a, w, eager, rows, 1, k, n)
        torch.cuda.synchronize()
        _check_f32_against_f64(eager, wf, a)
    del w, g
    eng.sync()
    eng.close()


@pytest.mark.parametrize("ggml_type", [2, 8, 12, 13, 1])
@pytest.mark.parametrize("rows,n,k", [(5, 1000, 4096), (20, 4096, 4096), (40, 32000, 4096), (64, 2048, 4096)])
def test_f32_rows_on_mfma_are_as_close_as_single_rows(engine, ggml_type, rows, n, k):
    """Several binary32 rows at once: the root-mean-square error against 64
    bits is no larger than that of the row kernels (within 1 %, more than two
    samples of 5000 rounding errors and more differ by): one M tile and two, K
    split 16 ways and not at all. A product that lost a part of x is outside."""
    _, w = _weight(engine, ggml_type, n, k, 40 + ggml_type)
    x = torch.randn(rows, k, generator=torch.Generator().manual_seed(rows)).to(DEV)
    c, one = torch.empty(rows, n, device=DEV), torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, x, w, c, rows, 1, k, n)
    for r in range(rows):
        ops.gemm_auto(engine, x[r], w, one[r], 1, 1, k, n)
    want = x.double() @ w.dequant().double().T.contiguous()
    err, single = (float((y.double() - want).norm()) for y in (c, one))
    assert err <= 1.01 * single, err / single
    # the bound tells a lost third part of x from rounding (x1 + x2 alone, in 64 bits)
    upper = lambda t: (t.view(torch.int32) & -65536).view(torch.float32)
    x12 = upper(x).double() + upper(x - upper(x)).double()
    assert float((x12 @ w.dequant().double().T.contiguous() - want).norm()) > 1.5 * single


@pytest.mark.parametrize("ggml_type", [12, 13])
@pytest.mark.parametrize("rows", [5, 40])
def test_f32_rows_on_mfma_at_the_top_of_the_range(engine, ggml_type, rows):
    """K-quant blocks whose six-bit scales and mins are 1 and x near the top of
    binary32: a block's sum of x times 8 or 16 exceeds it, the row kernel's sums
    do not, and neither do these. A row of 2^-124: each x keeps what is not
    below 2^-133, the last place of a bfloat16 (Q5_K: of x / 32)."""
    n, k = 64, 512
    rng = np.random.default_rng(3)
    blocks = np.zeros((n * k // 256, 144 if ggml_type == 12 else 176), np.uint8)
    blocks[:, 0:4] = np.array([2.0 ** -14, 2.0 ** -12], np.float16).view(np.uint8)   # d, dmin
    blocks[:, 4:12], blocks[:, 12:16] = 1, 0x11
    blocks[:, -128:] = rng.integers(0, 256, (len(blocks), 128)) & 0x11               # q of 0 or 1
    w = ops.GpuTensor(engine, ggml_type, n, k, blocks)
    x = torch.full((rows, k), 2.0 ** 122)
    x[1] = torch.randn(k, generator=torch.Generator().manual_seed(4)) * 2.0 ** -124
    x[:, 300:] *= -0.75
    a, c = x.to(DEV), torch.empty(rows, n, device=DEV)
    ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
    y = torch.empty(n, device=DEV)
    ops.gemm_auto(engine, a[0], w, y, 1, 1, k, n)
    assert bool(y.isfinite().all()) and bool(c.isfinite().all())
    keep = [0] + list(range(2, rows))
    _check_f32_against_f64(c[keep], w.dequant().cpu().numpy(), x[keep])
    wf = w.dequant().cpu().double()
    err = (c[1].double().cpu() - x[1].double() @ wf.T).abs()
    last = 2.0 ** (-133 if ggml_type == 12 else -128)
    assert bool((err <= 1.01 * last * wf.abs().sum(1)).all())


def test_f32_rows_keep_no_copy_of_a_weight_without_exact_parts(engine):
    """The tile copy of a binary16 weight (its size again) stays with the
    weight where binary32 rows run on it, and not where an infinity keeps them
    on the row kernels; binary16 rows may still build it."""
    n, k, rows = 8192, 4096, 5   # 64 MiB
    bits = synth.f16_bits(np.full((n, k), 0.02, np.float32)).reshape(n, k).copy()
    a, c = torch.randn(rows, k, device=DEV), torch.empty(rows, n, device=DEV)
    for kept, value in ((True, bits[3, 3]), (False, 0x7C00)):
        bits[3, 3] = value
        w = ops.GpuTensor(engine, 1, n, k, bits)
        ops.gemm_auto(engine, a[:1], w, c[:1], 1, 1, k, n)
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        for _ in range(2):
            ops.gemm_auto(engine, a, w, c, rows, 1, k, n)
        torch.cuda.synchronize()
        assert (free - torch.cuda.mem_get_info()[0] > 32 << 20) == kept
        h = torch.empty(rows, n, device=DEV)
        ops.gemm_auto(engine, a.half(), w, h, rows, 1, k, n)
        torch.cuda.synchronize()
        assert free - torch.cuda.mem_get_info()[0] > 32 << 20
        assert bool(h.isfinite().all(0)[3]) == kept and bool(h[:, 4:].isfinite().all())
        w.free()


def test_f32_rows_of_several_threads_on_one_weight():
    """Threads with a context and a stream each make the first call with
    several binary32 rows on a weight at the same time: the tile copy is built
    once, and all get the result of a call alone."""
    n, k, rows, count = 4096, 2048, 9, 6
    engines = [ops.ComputeEngine(0) for _ in range(count)]
    streams = [torch.cuda.Stream() for _ in range(count)]
    a = torch.randn(rows, k, device=DEV)
    outs = [torch.zeros(rows, n, device=DEV) for _ in range(count)]
    for e, s in zip(engines, streams):
        e.bind_stream(s)
    for turn in range(4):
        _, w = _weight(engines[0], 2, n, k, turn)
        torch.cuda.synchronize()
        start = threading.Barrier(count)

        def call(i):
            start.wait()
            ops.gemm_auto(engines[i], a, w, outs[i], rows, 1, k, n)
            engines[i].sync()

        threads = [threading.Thread(target=call, args=(i,)) for i in range(count)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        want = torch.empty(rows, n, device=DEV)
        torch.cuda.synchronize()
        ops.gemm_auto(engines[0], a, w, want, rows, 1, k, n)
        engines[0].sync()
        assert all(torch.equal(o, want) for o in outs)
        w.free()
    for e in engines:
        e.close()
