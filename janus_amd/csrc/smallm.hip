// smallm.hip -- products with 2..64 activation rows (ragged decode batches)
// and with any number of them (prompt chunks): the dequant-fused MFMA GEMM, on binary16 activations or on binary32 ones
// split into three bfloat16 parts.
//
// Replaces the reference's M>1 quantised path, which hands quantised bytes
// to the f16 GEMM (crates/janus-engine/src/compute/ops/quantized.rs:77-90,
// 104-117, 131-144; shaders/gemm.wgsl) and so has no correct result to match;
// parity is "equal to M stacked GEMVs" within fp32 accumulation tolerance.
//
// Weight tiles ("T32", built once per weight on first use from the GEMV
// layout): rows are grouped by 32 and K by chunks; for row group g and chunk c
// the 64 lanes of a wavefront each load 16 contiguous bytes (1 KiB per
// wavefront load) that are already the lane's B operand of
// v_mfma_f32_32x32x16_f16: lane l holds weight row 32g + (l % 32) and the
// K-half h = l / 32 of each 16-wide MFMA step.
//   Q4_0 / Q4_K: chunk = 64 K (two 32-element blocks). Per block two words:
//     elements 8h..8h+7 and 16+8h..16+8h+7, nibbles stored in the order
//     e0,e2,e4,e6,e1,e3,e5,e7 so that (w >> 4t) & 0x000f000f yields the
//     natural pair (e_2t, e_2t+1) as binary16 1024 + q.
//     Q4_0 side data: [g][c][32] u32 = the two blocks' binary16 scales.
//     Q4_K side data: [g][super-block][32] 16-byte headers as uploaded (d,
//     dmin, scale fields of kq_group).
//   Q5_K: as Q4_K (nibbles and headers), plus the fifth bits: one word per
//     lane and chunk [g][c][64], bit 4 * slot + i for the element in nibble
//     slot `slot` of the lane's word i (176 bytes per 256 weights, the GGUF
//     size).
//   Q8_0: chunk = 32 K (one block): bytes of elements 8h..8h+7 then
//     16+8h..16+8h+7; side data [g][c][32] binary16 scales.
//   F16: chunk = 16 K: the eight binary16 weights 8h..8h+7 of the chunk.
// Padding rows and K are zero (zero scale), so they add nothing.
//
// Kernel: a workgroup is 16 wavefronts, 4 K slices of 4 consecutive row groups
// (128 weight rows), over a range of K "passes". Per pass the activations
// A[rows][kr] (binary16) are staged in LDS once and shared by all wavefronts;
// each wavefront streams the weight chunks of its row group and K slice with 128-bit non-temporal loads,
// unpacks them in registers into exact binary16 integers, runs
// 32x32x16 MFMAs with fp32 accumulation per quantisation block, and applies
// the block scale to the fp32 block result (so products and scales round
// exactly as the M=1 kernels do). The K slices of a row group are added in
// slice order through LDS at the end. When there are too few row tiles to fill
// the GPU, K is split over workgroups; the partial tiles go to a workspace
// and a second kernel adds them in fixed split order, so results do not
// depend on scheduling.
#include "internal.h"

namespace janus {
namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef __bf16 b8 __attribute__((ext_vector_type(8)));
typedef __bf16 b2 __attribute__((ext_vector_type(2)));
typedef float f16x __attribute__((ext_vector_type(16)));

constexpr int WAVES = 4;   // row groups per workgroup

__device__ __forceinline__ jh2 as_h2(uint32_t u) { return __builtin_bit_cast(jh2, u); }

// 8 permuted nibbles -> 8 binary16 (1024 + q) - off, natural element order.
// Slots 0/4 and 2/6 (mask 0x000f000f) become 1024 + q; slots 1/5 and 3/7
// (mask 0x00f000f0) become 1024 + 16 q, scaled back exactly by one FMA
// ((1024 + 16 q) / 16 - 64 - (off - 1024) = q - (off - 1024)). The magic
// exponent sits in a VGPR so each mask-and-merge is one v_and_or_b32.
__device__ __forceinline__ h8 unpack_nib8(uint32_t u, _Float16 off) {
    const jh2 o = {off, off};
    const jh2 s16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    const _Float16 cb = (_Float16)(960.0f - (float)off);
    const jh2 c = {cb, cb};
    const uint32_t m = vgpr_const_6400();
    const uint32_t u8 = u >> 8;
    const jh2 p0 = as_h2((u & 0x000f000fu) | m) - o;
    const jh2 p1 = __builtin_elementwise_fma(as_h2((u & 0x00f000f0u) | m), s16, c);
    const jh2 p2 = as_h2((u8 & 0x000f000fu) | m) - o;
    const jh2 p3 = __builtin_elementwise_fma(as_h2((u8 & 0x00f000f0u) | m), s16, c);
    return (h8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

// unpack_nib8 with off = 1024 for 5-bit values: the fifth bits of the word's
// 8 elements (Q5_K layout above, word I of the lane) are OR-ed into the
// binary16 mantissas: bit 4 of 1024 + q (slots 0/4, 2/6) or bit 8 of
// 1024 + 16 q (slots 1/5, 3/7), so the values are q in 0..31, exact.
template <int I>
__device__ __forceinline__ h8 unpack_nib8_q5(uint32_t u, uint32_t fifth) {
    const jh2 o = {(_Float16)1024.0f, (_Float16)1024.0f};
    const jh2 s16 = {(_Float16)0.0625f, (_Float16)0.0625f};
    const jh2 c = {(_Float16)-64.0f, (_Float16)-64.0f};
    const uint32_t m = vgpr_const_6400();
    const uint32_t u8 = u >> 8;
    const uint32_t ta = fifth << (4 - I), tb = fifth >> (4 + I);   // slot s of word I -> bit 4 s + 4, 4 s - 4
    const jh2 p0 = as_h2((u & 0x000f000fu) | m | (ta & 0x00100010u)) - o;
    const jh2 p1 = __builtin_elementwise_fma(as_h2((u & 0x00f000f0u) | m | (ta & 0x01000100u)), s16, c);
    const jh2 p2 = as_h2((u8 & 0x000f000fu) | m | (tb & 0x00100010u)) - o;
    const jh2 p3 = __builtin_elementwise_fma(as_h2((u8 & 0x00f000f0u) | m | (tb & 0x01000100u)), s16, c);
    return (h8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

// 8 int8 (two words) -> 8 binary16 integers, natural order.
__device__ __forceinline__ h8 unpack_i8x8(uint32_t lo, uint32_t hi) {
    const jh2 o = {(_Float16)1152.0f, (_Float16)1152.0f};
    const uint32_t c64 = 0x64646464u;
    lo ^= 0x80808080u;
    hi ^= 0x80808080u;
    jh2 p0 = as_h2(__builtin_amdgcn_perm(lo, c64, 0x00050004u)) - o;
    jh2 p1 = as_h2(__builtin_amdgcn_perm(lo, c64, 0x00070006u)) - o;
    jh2 p2 = as_h2(__builtin_amdgcn_perm(hi, c64, 0x00050004u)) - o;
    jh2 p3 = as_h2(__builtin_amdgcn_perm(hi, c64, 0x00070006u)) - o;
    return (h8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

// ---- binary32 activations: three bfloat16 parts ---------------------------------
// A finite binary32 x of at least 2^-110 (Q5_K 2^-105) is exactly x1 + x2 + x3
// with bfloat16 parts of 8 significant bits each (x1 = the upper 16 bits of x,
// x2 those of x - x1, x3 the rest; what lies below 2^-133, Q5_K 2^-128, is cut
// off), and the quantised weights are exact bfloat16 integers. So a product of binary32 activations is three
// v_mfma_f32_32x32x16_bf16 per operand pair, every partial product exact and
// every sum binary32, with nothing rounded on the way in: the weights are read
// once for all rows instead of once per row by the M = 1 kernel.

// Bytes (b0, b1) / (b2, b3) of v (each below 16) times `unit`, a power of two, as
// exact bfloat16 (OCP e4m3 byte b < 16 is b * 2^-9; the conversion scales it).
template <bool HI> __device__ __forceinline__ b2 nib8_bf16(uint32_t v, float unit) {
    return __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.0f * unit, HI);
}

// The upper halves of two floats as a bfloat16 pair (exact for integers below 256).
__device__ __forceinline__ uint32_t pack_hi16(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// A T32 word of 8 nibbles -> 8 bfloat16 integers (times `unit`) in the order e0 e4 e1 e5 e2
// e6 e3 e7 (the byte order of the word's low and high nibbles); the
// activations are staged in the same order (SplitOrder).
__device__ __forceinline__ b8 unpack_nib8_b(uint32_t u, float unit = 1.0f) {
    const uint32_t lo = u & 0x0f0f0f0fu, hi = (u >> 4) & 0x0f0f0f0fu;
    const b2 p0 = nib8_bf16<false>(lo, unit), p1 = nib8_bf16<true>(lo, unit), p2 = nib8_bf16<false>(hi, unit),
             p3 = nib8_bf16<true>(hi, unit);
    return (b8){p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
}

__device__ __forceinline__ b8 as_b8(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    return __builtin_bit_cast(b8, make_uint4(a, b, c, d));
}

// Q5_K word I: the fifth bits join the nibble bytes (bit 4), then bytes -> bfloat16.
template <int I>
__device__ __forceinline__ b8 unpack_nib8_q5_b(uint32_t u, uint32_t fifth) {
    const uint32_t f = fifth >> I;
    const uint32_t lo = (u & 0x0f0f0f0fu) | ((f << 4) & 0x10101010u);
    const uint32_t hi = ((u >> 4) & 0x0f0f0f0fu) | (f & 0x10101010u);
    auto pair = [](uint32_t v, int s) { return pack_hi16((float)((v >> s) & 255u), (float)((v >> (s + 8)) & 255u)); };
    return as_b8(pair(lo, 0), pair(lo, 16), pair(hi, 0), pair(hi, 16));
}

// 8 int8 (two words) -> 8 bfloat16 integers, natural order.
__device__ __forceinline__ b8 unpack_i8x8_b(uint32_t lo, uint32_t hi) {
    auto pair = [](uint32_t v, int s) {
        return pack_hi16((float)(int)(int8_t)(v >> s), (float)(int)(int8_t)(v >> (s + 8)));
    };
    return as_b8(pair(lo, 0), pair(lo, 16), pair(hi, 0), pair(hi, 16));
}

// 8 finite binary16 weights -> their upper 8 bits and the remaining 3, both
// exact bfloat16 (natural order).
__device__ __forceinline__ void split_f16x8(const uint4 &q, b8 &hi, b8 &lo) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
    uint32_t a[4], b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float e = h2f((uint16_t)(w[i] & 0xffffu)), o = h2f((uint16_t)(w[i] >> 16));
        a[i] = pack_hi16(e, o);
        b[i] = pack_hi16(e - __uint_as_float(__float_as_uint(e) & 0xffff0000u),
                         o - __uint_as_float(__float_as_uint(o) & 0xffff0000u));
    }
    hi = as_b8(a[0], a[1], a[2], a[3]);
    lo = as_b8(b[0], b[1], b[2], b[3]);
}

// x[0..8) -> its three bfloat16 parts, 8 values each in one 16-byte word.
// ORDER4: in the order of unpack_nib8_b, else natural. An infinite x is all in
// the first part; a NaN stays a NaN in the second. Returns whether an x is
// infinite.
template <bool ORDER4>
__device__ __forceinline__ bool split_x8(const float (&x)[8], uint4 (&part)[3]) {
    float r[8];
    float top = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        r[i] = x[i] - __uint_as_float(__float_as_uint(x[i]) & 0xffff0000u);
        top = fmaxf(top, fabsf(x[i]));
    }
    if (top == INFINITY) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (fabsf(x[i]) == INFINITY) r[i] = 0.0f;
    }
    float s[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) s[i] = r[i] - __uint_as_float(__float_as_uint(r[i]) & 0xffff0000u);
    auto pack = [](const float (&v)[8]) {
        return ORDER4 ? make_uint4(pack_hi16(v[0], v[4]), pack_hi16(v[1], v[5]), pack_hi16(v[2], v[6]), pack_hi16(v[3], v[7]))
                      : make_uint4(pack_hi16(v[0], v[1]), pack_hi16(v[2], v[3]), pack_hi16(v[4], v[5]), pack_hi16(v[6], v[7]));
    };
    part[0] = pack(x);
    part[1] = pack(r);
    part[2] = pack(s);
    return top == INFINITY;
}

// The finite values of 8 bfloat16, infinities as 0.
__device__ __forceinline__ b8 strip_inf(b8 x) {
    uint4 v = __builtin_bit_cast(uint4, x);
    uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if ((u[i] & 0x7fffu) == 0x7f80u) u[i] &= 0xffff0000u;
        if ((u[i] & 0x7fff0000u) == 0x7f800000u) u[i] &= 0xffffu;
    }
    return as_b8(u[0], u[1], u[2], u[3]);
}

__device__ __forceinline__ f16x mfma_b(b8 a, b8 b, f16x c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// One 32-element block of one M-tile: t + (the three parts of A, rows at ap,
// `plane` halves apart) x (b0: elements 0-15, b1: 16-31). From t = 0 the
// smallest part goes first (only the leading part's two sums round at full
// size). FROM_OFFSET: t is the block's offset term, as large as the sums
// themselves; the leading part cancels most of it first.
template <bool FROM_OFFSET>
__device__ __forceinline__ f16x block_b(const _Float16 *ap, uint32_t plane, b8 b0, b8 b1, f16x t) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const int part = FROM_OFFSET ? i : 2 - i;
        t = mfma_b(*(const b8 *)(ap + part * plane), b0, t);
        t = mfma_b(*(const b8 *)(ap + part * plane + 16), b1, t);
    }
    return t;
}

// The per-row values of a lane's tile rows from s (one float per row): rows
// 8 j + 4 h + 0..3 (the MFMA C layout), the first VN of them.
template <int VN>
__device__ __forceinline__ f16x tile_rows(const float *s, int h) {
    f16x t = (f16x){};
#pragma unroll
    for (int j = 0; j < VN / 4; ++j) {
        const jf4 v = *(const jf4 *)(s + 8 * j + 4 * h);
        t[4 * j] = v.x;
        t[4 * j + 1] = v.y;
        t[4 * j + 2] = v.z;
        t[4 * j + 3] = v.w;
    }
    return t;
}

__device__ __forceinline__ f16x mfma(h8 a, h8 b, f16x c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ h8 lds_h8(const _Float16 *p) { return *(const h8 *)p; }

struct GemmArgs {
    const uint8_t *qs;     // T32 quant chunks [G][C][64][16 B]
    const uint8_t *side;   // T32 side data (scales / headers)
    const uint32_t *q5h;   // Q5_K fifth bits [G][C][64]
    const _Float16 *a;     // activations [rows][k]
    const float *a32;      // binary32 activations (X32 kernels; a is null then)
    void *c;               // output [rows][n]
    const float *resid;    // [rows][n] or null (may alias c)
    float *ws;             // split-K partials [ksplit][Mpad][Npad]
    uint32_t rows, n, k;
    uint32_t chunks;       // C: chunks per row group
    uint32_t pass_chunks;  // chunks per LDS pass
    uint32_t passes_per_wg;
    uint32_t total_passes;
    uint32_t ksplit;
    uint32_t tiles, mtiles;   // gemm_pipe_kernel: weight tiles of 32 NW rows, M tiles of 32 MT rows
    uint32_t pitch;        // LDS row pitch of A, in halves
    int c_f16;
    int to_ws;             // write partials to ws even when ksplit == 1 (epilogue kernels read them)
    uint32_t seg_shift;    // log2 of the 8-half A segments per row of a pass (pass length / 8)
    int swiglu;            // ksplit == 1 only: rows (2j, 2j+1) are (gate_j, up_j); c = silu(gate)*up [rows][n/2]
};

// ---- formats ------------------------------------------------------------------
// W: one chunk of one lane. load() reads it; mma() adds its contribution for
// MT M-tiles given the LDS A slice (row stride pitch) at chunk offset kl.

// Block results whose scale is applied one block later: the scale FMAs of a
// block then run while the next block's MFMAs are in flight instead of
// waiting for their own (the same FMAs in the same order).
template <int MT> struct Deferred {
    f16x t[MT];   // the last block's MFMA results
    float d;      // and its scale (0 before the first block)
};

// PIN keeps the arithmetic on a result tile where it is written. In the
// branch-free passes of the wide kernel the compiler otherwise sinks the scale
// FMAs of a whole pass behind its MFMAs and spills the block results held for
// them (28672x4096 at 512 rows: 1.8 ms against 0.17).
template <int MT, bool PIN>
__device__ __forceinline__ void pin(f16x (&acc)[MT]) {
    if constexpr (PIN)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(acc[mt]));
}

// Products with at most 8 or 16 rows use the first VN = 4 or 8 values of a
// lane's result tile (rows 8 (v / 4) + 4 (lane / 32) + v % 4): the scale FMAs,
// the K-slice sums and the stores stop there, and 8 or 16 rows of activations
// are staged, read by the lanes of rows that have none modulo that many.
template <int MT, int VN> constexpr int rows_staged() { return VN == 16 ? MT * 32 : 2 * VN; }
template <int VN> constexpr int row_mask() { return VN == 16 ? 31 : 2 * VN - 1; }

// acc += the pending block's scaled results; t with scale d becomes pending
// (from three M tiles on t is applied at once: the tiles' MFMAs cover each
// other's latency, and a second set of results does not fit the registers).
template <int MT, bool PIN = false, int VN = 16>
__device__ __forceinline__ void apply_deferred(f16x (&acc)[MT], Deferred<MT> &pend, const f16x (&t)[MT], float d) {
    if constexpr (MT >= 3) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(d, t[mt][v], acc[mt][v]);
        pin<MT, PIN>(acc);
        return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(pend.d, pend.t[mt][v], acc[mt][v]);
    pin<MT, PIN>(acc);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) pend.t[mt] = t[mt];
    pend.d = d;
}

struct GQ4_0 {
    static constexpr int CK = 64;
    static constexpr bool DEFER = true;
    static constexpr bool ORDER4 = true;
    static constexpr float XSUM = -8.0f;   // X32: per-block sums are staged times this
    static constexpr float XMUL = 1.0f;    // X32: x is staged times this
    static constexpr float WMUL = 1.0f;    // X32: and the weights' integers are times this, and the sums too
    struct W { uint4 q; uint32_t s; };
    // One chunk on binary32 activations: As holds their three bfloat16 parts
    // (`plane` halves apart). The offset -8 enters as the first accumulator,
    // -8 * sum(x) of the block, so the weights stay the integers 0..15.
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma_x32(const W &w, const _Float16 *As, uint32_t plane, uint32_t pitch, uint32_t kl,
                                   uint32_t, int lane, const float *Ss, f16x (&acc)[MT], Deferred<MT> &pend) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const uint32_t q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const b8 b0 = unpack_nib8_b(q[2 * b]), b1 = unpack_nib8_b(q[2 * b + 1]);
            f16x t[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt)
                t[mt] = block_b<true>(As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h, plane, b0, b1,
                                tile_rows<VN>(Ss + (size_t)(kl / 32 + b) * rows_staged<MT, VN>() + mt * 32, h));
            apply_deferred<MT, PIN, VN>(acc, pend, t, h2f((uint16_t)(b ? (w.s >> 16) : (w.s & 0xffffu))));
        }
    }
    // g and c are wavefront-uniform: the chunk base is scalar, the lane adds
    // a 32-bit offset
    __device__ static W load(const GemmArgs &a, uint32_t g, uint32_t c, int lane) {
        const size_t ch = (size_t)g * a.chunks + c;
        W w;
        w.q = ld_stream(a.qs + ch * 1024 + (uint32_t)lane * 16u);
        w.s = *(const uint32_t *)(a.side + ch * 128 + (uint32_t)(lane & 31) * 4u);
        return w;
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma_deferred(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                                        f16x (&acc)[MT], Deferred<MT> &pend) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const uint32_t q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const h8 b0 = unpack_nib8(q[2 * b], (_Float16)1032.0f);
            const h8 b1 = unpack_nib8(q[2 * b + 1], (_Float16)1032.0f);
            const float d = h2f((uint16_t)(b ? (w.s >> 16) : (w.s & 0xffffu)));
            f16x t[MT];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h;
                t[mt] = mfma(lds_h8(ap), b0, (f16x){});
                t[mt] = mfma(lds_h8(ap + 16), b1, t[mt]);
            }
            apply_deferred<MT, PIN, VN>(acc, pend, t, d);
        }
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                               const float *, uint32_t, f16x (&acc)[MT]) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const uint32_t q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const h8 b0 = unpack_nib8(q[2 * b], (_Float16)1032.0f);
            const h8 b1 = unpack_nib8(q[2 * b + 1], (_Float16)1032.0f);
            const float d = h2f((uint16_t)(b ? (w.s >> 16) : (w.s & 0xffffu)));
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h;
                f16x t = mfma(lds_h8(ap), b0, (f16x){});
                t = mfma(lds_h8(ap + 16), b1, t);
#pragma unroll
                for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(d, t[v], acc[mt][v]);
            }
        }
    }
};

struct GQ8_0 {
    static constexpr int CK = 32;
    static constexpr bool ORDER4 = false;
    static constexpr float XSUM = 0.0f;   // no sums
    static constexpr float XMUL = 1.0f, WMUL = 1.0f;
    struct W { uint4 q; uint16_t s; };
    // see GQ4_0::mma_x32
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma_x32(const W &w, const _Float16 *As, uint32_t plane, uint32_t pitch, uint32_t kl,
                                   uint32_t, int lane, const float *, f16x (&acc)[MT], Deferred<MT> &pend) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const b8 b0 = unpack_i8x8_b(w.q.x, w.q.y), b1 = unpack_i8x8_b(w.q.z, w.q.w);
        f16x t[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
            t[mt] = block_b<false>(As + (size_t)(mt * 32 + r) * pitch + kl + 8 * h, plane, b0, b1, (f16x){});
        apply_deferred<MT, PIN, VN>(acc, pend, t, h2f_q8(w.s));
    }
    __device__ static W load(const GemmArgs &a, uint32_t g, uint32_t c, int lane) {
        const size_t ch = (size_t)g * a.chunks + c;
        W w;
        w.q = ld_stream(a.qs + (ch * 64 + lane) * 16);
        w.s = ((const uint16_t *)a.side)[ch * 32 + (lane & 31)];
        return w;
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                               const float *, uint32_t, f16x (&acc)[MT]) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const h8 b0 = unpack_i8x8(w.q.x, w.q.y);
        const h8 b1 = unpack_i8x8(w.q.z, w.q.w);
        const float d = h2f_q8(w.s);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + 8 * h;
            f16x t = mfma(lds_h8(ap), b0, (f16x){});
            t = mfma(lds_h8(ap + 16), b1, t);
#pragma unroll
            for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(d, t[v], acc[mt][v]);
        }
        pin<MT, PIN>(acc);
    }
};

// Q4_K: w = (d*sc)*q - dmin*m per 32-element sub-block (shaders/gemm_q4_k.wgsl:82-113);
// the m term uses the per-(row, sub-block) activation sums staged in LDS.
struct GQ4_K {
    static constexpr int CK = 64;
    static constexpr bool ORDER4 = true;
    static constexpr float XSUM = -8.0f, XMUL = 1.0f, WMUL = 1.0f / 16.0f;
    struct W { uint4 q; uint4 hdr; };
    // binary32 activations (three bfloat16 parts, GQ4_0::mma_x32). The staged
    // sums are -8 sum(x) (Q5_K: -16), so the MFMA result is that of the centred
    // values q - 8 and ds * (q . x) - dm * sum(x) = ds * t + (dm - 8 ds) / 8 * staged:
    // the two large terms of a block mostly cancel before they are rounded.
    // Products and sums are made 16 times smaller (Q5_K: 32), so that the sums
    // stay finite wherever the row kernel's over 16 elements do: by the
    // conversion of the nibbles, in Q5_K, whose five bits have none, by x as it
    // is staged (either is within the spread of 63 us, 11008x4096 and back at 16
    // rows). c: chunk of the row group.
    template <int MT, bool PIN = false, int VN = 16, class G = GQ4_K>
    __device__ static void mma_x32(const typename G::W &w, const _Float16 *As, uint32_t plane, uint32_t pitch,
                                   uint32_t kl, uint32_t c, int lane, const float *Ss, f16x (&acc)[MT],
                                   Deferred<MT> &) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const float d = h2f((uint16_t)(w.hdr.x & 0xffffu)), dmin = h2f((uint16_t)(w.hdr.x >> 16));
        const int j = (int)(c & 3);   // chunk index within the super-block
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float sc, mn;
            scale_min(w.hdr, 2 * j + b, sc, mn);
            // powers of two are exact
            constexpr float up = 1.0f / (G::XMUL * G::WMUL);
            const float ds = d * sc * up, dm = dmin * mn * up;
            const float cs = fmaf(G::XSUM, ds, dm) * (-1.0f / G::XSUM);
            b8 b0, b1;
            G::unpack_b(w, b, b0, b1);
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const f16x s = tile_rows<VN>(Ss + (size_t)(kl / 32 + b) * rows_staged<MT, VN>() + mt * 32, h);
                const f16x t =
                    block_b<true>(As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h, plane, b0, b1, s);
#pragma unroll
                for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(cs, s[v], fmaf(ds, t[v], acc[mt][v]));
            }
            pin<MT, PIN>(acc);
        }
    }
    __device__ static void unpack_b(const W &w, int b, b8 &b0, b8 &b1) {
        b0 = unpack_nib8_b(b ? w.q.z : w.q.x, WMUL);
        b1 = unpack_nib8_b(b ? w.q.w : w.q.y, WMUL);
    }
    __device__ static W load(const GemmArgs &a, uint32_t g, uint32_t c, int lane) {
        const size_t ch = (size_t)g * a.chunks + c;
        W w;
        w.q = ld_stream(a.qs + (ch * 64 + lane) * 16);
        const size_t sb = (size_t)g * (a.chunks / 4) + c / 4;
        w.hdr = *(const uint4 *)(a.side + (sb * 32 + (lane & 31)) * 16);
        return w;
    }
    // (sc, m) of sub-block `sub` (uniform) from the packed scale words hdr.y..w
    __device__ static void scale_min(const uint4 &hdr, int sub, float &sc, float &mn) {
        const uint32_t g = kq_group(hdr.y, hdr.z, hdr.w, (uint32_t)sub >> 1), o = 6u * (uint32_t)(sub & 1);
        sc = (float)((g >> o) & 63u);
        mn = (float)((g >> (12u + o)) & 63u);
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                               const float *Ss, uint32_t chunk0, f16x (&acc)[MT]) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const uint32_t q[4] = {w.q.x, w.q.y, w.q.z, w.q.w};
        const float d = h2f((uint16_t)(w.hdr.x & 0xffffu)), dmin = h2f((uint16_t)(w.hdr.x >> 16));
        const int j = (int)((kl / 64 + chunk0) & 3);   // chunk index within the super-block (chunk0: the pass's first)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float sc, mn;
            scale_min(w.hdr, 2 * j + b, sc, mn);
            const float ds = d * sc, dm = dmin * mn;
            const h8 b0 = unpack_nib8(q[2 * b], (_Float16)1024.0f);
            const h8 b1 = unpack_nib8(q[2 * b + 1], (_Float16)1024.0f);
            const uint32_t sub = kl / 32 + b;   // sub-block index within the pass
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h;
                f16x t = mfma(lds_h8(ap), b0, (f16x){});
                t = mfma(lds_h8(ap + 16), b1, t);
                const float *sx = Ss + (size_t)sub * rows_staged<MT, VN>() + mt * 32 + 4 * h;
#pragma unroll
                for (int jj = 0; jj < VN / 4; ++jj) {
                    const jf4 s4 = *(const jf4 *)(sx + 8 * jj);
                    acc[mt][4 * jj + 0] = fmaf(-dm, s4.x, fmaf(ds, t[4 * jj + 0], acc[mt][4 * jj + 0]));
                    acc[mt][4 * jj + 1] = fmaf(-dm, s4.y, fmaf(ds, t[4 * jj + 1], acc[mt][4 * jj + 1]));
                    acc[mt][4 * jj + 2] = fmaf(-dm, s4.z, fmaf(ds, t[4 * jj + 2], acc[mt][4 * jj + 2]));
                    acc[mt][4 * jj + 3] = fmaf(-dm, s4.w, fmaf(ds, t[4 * jj + 3], acc[mt][4 * jj + 3]));
                }
            }
            pin<MT, PIN>(acc);
        }
    }
};

// Q5_K (GGML block_q5_K): the Q4_K tiles (nibbles, 16-byte headers) plus the
// fifth bits of the lane's 32 elements in one word per chunk; w = (d*sc)*q -
// dmin*m with q in 0..31, the m term from the staged activation sums.
struct GQ5_K {
    static constexpr int CK = 64;
    static constexpr bool ORDER4 = true;
    static constexpr float XSUM = -16.0f, XMUL = 1.0f / 32.0f, WMUL = 1.0f;
    struct W { uint4 q; uint4 hdr; uint32_t fifth; };
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma_x32(const W &w, const _Float16 *As, uint32_t plane, uint32_t pitch, uint32_t kl,
                                   uint32_t c, int lane, const float *Ss, f16x (&acc)[MT], Deferred<MT> &pend) {
        GQ4_K::mma_x32<MT, PIN, VN, GQ5_K>(w, As, plane, pitch, kl, c, lane, Ss, acc, pend);
    }
    __device__ static void unpack_b(const W &w, int b, b8 &b0, b8 &b1) {
        b0 = b ? unpack_nib8_q5_b<2>(w.q.z, w.fifth) : unpack_nib8_q5_b<0>(w.q.x, w.fifth);
        b1 = b ? unpack_nib8_q5_b<3>(w.q.w, w.fifth) : unpack_nib8_q5_b<1>(w.q.y, w.fifth);
    }
    __device__ static W load(const GemmArgs &a, uint32_t g, uint32_t c, int lane) {
        const size_t ch = (size_t)g * a.chunks + c;
        W w;
        w.q = ld_stream(a.qs + (ch * 64 + lane) * 16);
        w.fifth = __builtin_nontemporal_load(a.q5h + ch * 64 + lane);
        const size_t sb = (size_t)g * (a.chunks / 4) + c / 4;
        w.hdr = *(const uint4 *)(a.side + (sb * 32 + (lane & 31)) * 16);
        return w;
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                               const float *Ss, uint32_t chunk0, f16x (&acc)[MT]) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const float d = h2f((uint16_t)(w.hdr.x & 0xffffu)), dmin = h2f((uint16_t)(w.hdr.x >> 16));
        const int j = (int)((kl / 64 + chunk0) & 3);   // chunk index within the super-block (chunk0: the pass's first)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float sc, mn;
            GQ4_K::scale_min(w.hdr, 2 * j + b, sc, mn);
            const float ds = d * sc, dm = dmin * mn;
            const h8 b0 = b == 0 ? unpack_nib8_q5<0>(w.q.x, w.fifth) : unpack_nib8_q5<2>(w.q.z, w.fifth);
            const h8 b1 = b == 0 ? unpack_nib8_q5<1>(w.q.y, w.fifth) : unpack_nib8_q5<3>(w.q.w, w.fifth);
            const uint32_t sub = kl / 32 + b;   // sub-block index within the pass
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + b * 32 + 8 * h;
                f16x t = mfma(lds_h8(ap), b0, (f16x){});
                t = mfma(lds_h8(ap + 16), b1, t);
                const float *sx = Ss + (size_t)sub * rows_staged<MT, VN>() + mt * 32 + 4 * h;
#pragma unroll
                for (int jj = 0; jj < VN / 4; ++jj) {
                    const jf4 s4 = *(const jf4 *)(sx + 8 * jj);
                    acc[mt][4 * jj + 0] = fmaf(-dm, s4.x, fmaf(ds, t[4 * jj + 0], acc[mt][4 * jj + 0]));
                    acc[mt][4 * jj + 1] = fmaf(-dm, s4.y, fmaf(ds, t[4 * jj + 1], acc[mt][4 * jj + 1]));
                    acc[mt][4 * jj + 2] = fmaf(-dm, s4.z, fmaf(ds, t[4 * jj + 2], acc[mt][4 * jj + 2]));
                    acc[mt][4 * jj + 3] = fmaf(-dm, s4.w, fmaf(ds, t[4 * jj + 3], acc[mt][4 * jj + 3]));
                }
            }
            pin<MT, PIN>(acc);
        }
    }
};

// formats whose block scales are applied one block late (mma_deferred)
template <class F, class = void> struct Defers { static constexpr bool value = false; };
template <class F> struct Defers<F, std::void_t<decltype(F::DEFER)>> { static constexpr bool value = F::DEFER; };

template <int MT, int VN = 16>
__device__ __forceinline__ void flush_deferred(f16x (&acc)[MT], const Deferred<MT> &pend) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < VN; ++v) acc[mt][v] = fmaf(pend.d, pend.t[mt][v], acc[mt][v]);
}

// formats whose mins need the per-(row, sub-block) activation sums in LDS
template <class F> struct NeedsSums { static constexpr bool value = false; };
template <> struct NeedsSums<GQ4_K> { static constexpr bool value = true; };
template <> struct NeedsSums<GQ5_K> { static constexpr bool value = true; };

struct GF16 {
    static constexpr int CK = 16;
    static constexpr bool ORDER4 = false;
    static constexpr float XSUM = 0.0f, XMUL = 1.0f, WMUL = 1.0f;
    struct W { uint4 q; };
    // binary32 activations: the weight is two bfloat16 parts, so a 16-wide
    // chunk is six MFMAs. The product of the two leading parts goes to acc,
    // the five small ones (below 2^-7 of it) to pend.t, added at the end, so
    // their roundings stay at their own size. inf: an activation may be
    // infinite; it then meets only the leading weight part (the other may be 0).
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma_x32(const W &w, const _Float16 *As, uint32_t plane, uint32_t pitch, uint32_t kl,
                                   uint32_t inf, int lane, const float *, f16x (&acc)[MT], Deferred<MT> &pend) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        b8 hi, lo;
        split_f16x8(w.q, hi, lo);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            const _Float16 *ap = As + (size_t)(mt * 32 + r) * pitch + kl + 8 * h;
            const b8 x1 = *(const b8 *)ap, x2 = *(const b8 *)(ap + plane), x3 = *(const b8 *)(ap + 2 * plane);
            acc[mt] = mfma_b(x1, hi, acc[mt]);
            pend.t[mt] = mfma_b(x3, lo, pend.t[mt]);
            pend.t[mt] = mfma_b(x3, hi, pend.t[mt]);
            pend.t[mt] = mfma_b(x2, lo, pend.t[mt]);
            pend.t[mt] = mfma_b(x2, hi, pend.t[mt]);
            pend.t[mt] = mfma_b(inf ? strip_inf(x1) : x1, lo, pend.t[mt]);
        }
    }
    __device__ static W load(const GemmArgs &a, uint32_t g, uint32_t c, int lane) {
        const size_t ch = (size_t)g * a.chunks + c;
        W w;
        w.q = ld_stream(a.qs + (ch * 64 + lane) * 16);
        return w;
    }
    template <int MT, bool PIN = false, int VN = 16>
    __device__ static void mma(const W &w, const _Float16 *As, uint32_t pitch, uint32_t kl, int lane,
                               const float *, uint32_t, f16x (&acc)[MT]) {
        const int h = lane >> 5, r = lane & row_mask<VN>();
        const h8 b = __builtin_bit_cast(h8, w.q);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = mfma(lds_h8(As + (size_t)(mt * 32 + r) * pitch + kl + 8 * h), b, acc[mt]);
    }
};

// chunks per weight batch (two batches in flight per wavefront)
template <class F> struct Stage { static constexpr int PD = std::is_same<F, GQ4_0>::value ? 2 : (F::CK == 64 ? 4 : 8); };

// Output element (m, n) of wave-tile value v for lane (32x32 MFMA C layout):
// n = lane % 32, m = 8 * (v / 4) + 4 * (lane / 32) + v % 4.
__device__ __forceinline__ uint32_t out_row(int mt, int v, int lane) {
    return (uint32_t)(mt * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3));
}

template <int MT>
__device__ __forceinline__ void store_tile(const GemmArgs &a, uint32_t g, uint32_t m0, int lane, const f16x (&acc)[MT]) {
    const uint32_t n = g * 32 + (lane & 31);
    if (n >= a.n) return;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const uint32_t m = m0 + out_row(mt, v, lane);
            if (m < a.rows) {
                float val = acc[mt][v];
                const size_t at = (size_t)m * a.n + n;
                if (a.resid) val += a.resid[at];
                if (a.c_f16) ((uint16_t *)a.c)[at] = f2h_bits(val);
                else ((float *)a.c)[at] = val;
            }
        }
}

// SwiGLU store of a finished tile: columns 2j, 2j+1 (lanes l, l^1) hold gate_j
// and up_j of the same rows; the even lane writes silu(gate) * up (the
// arithmetic of elementwise_kernel's SwiGLU).
template <int MT, bool F32OUT>
__device__ __forceinline__ void store_swiglu(const GemmArgs &a, uint32_t g, uint32_t m0, int lane,
                                             const f16x (&acc)[MT]) {
    const uint32_t n = g * 32 + (lane & 31);
    const uint32_t half = a.n / 2;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float mine = acc[mt][v];
            const float other = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(mine), 0xb1, 0xf, 0xf, false));
            const uint32_t m = m0 + out_row(mt, v, lane);
            if (!(lane & 1) && m < a.rows && n + 1 < a.n) {
                const float act = mine * (1.0f / (1.0f + expf(-mine))) * other;
                if constexpr (F32OUT) ((float *)a.c)[(size_t)m * half + n / 2] = act;
                else ((uint16_t *)a.c)[(size_t)m * half + n / 2] = f2h_bits(act);
            }
        }
}

// KW wavefronts per row group, each on a K slice of the pass (4 where the
// format's registers fit 4 wavefronts per SIMD, else 2).
// SPT: 16-byte A segments per thread per pass, Mpad * kr / 8 / (256 * KW).
template <class F, int MT, int KW, int SPT, int PD = Stage<F>::PD>
__global__ __launch_bounds__(64 * WAVES * KW) void gemm_mfma_kernel(GemmArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr bool SUMS = NeedsSums<F>::value;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: scalar chunk bases
    const int rgw = wave % WAVES, kw = wave / WAVES;   // row group in the tile, K slice of the pass
    const uint32_t G = (a.n + 31) / 32;
    const uint32_t tile = blockIdx.x, ks = blockIdx.y;
    const uint32_t g = tile * WAVES + rgw;
    const bool active = g < G;
    const uint32_t Mpad = MT * 32;
    _Float16 *As = (_Float16 *)smem;
    float *Ss = (float *)(smem + (size_t)Mpad * a.pitch * 2);

    f16x acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = (f16x){};
    Deferred<MT> pend;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) pend.t[mt] = (f16x){};
    pend.d = 0.0f;

    const uint32_t cpk = a.pass_chunks / KW;   // chunks per K slice
    const uint32_t p_begin = ks * a.passes_per_wg;
    const uint32_t p_end = min(a.total_passes, p_begin + a.passes_per_wg);
    for (uint32_t p = p_begin; p < p_end; ++p) {
        const uint32_t c0 = p * a.pass_chunks, c1 = min(a.chunks, c0 + a.pass_chunks);
        const uint32_t m0 = min(c1, c0 + kw * cpk), m1 = min(c1, m0 + cpk);   // this wave's chunks
        typename F::W wa[PD], wb[PD];
        auto load = [&](typename F::W (&w)[PD], uint32_t cs) {
#pragma unroll
            for (int i = 0; i < PD; ++i)
                if (cs + i < m1) w[i] = F::load(a, g, cs + i, lane);
        };
        if (active) load(wa, m0);   // in flight while A is staged

        // stage A[0..Mpad)[c0*CK .. c0*CK + kr) as binary16, zero outside rows / k:
        // segment s (8 halves) is row s >> seg_shift, column (s & mask) * 8 of the
        // full pass width (a power of two), so no division; every thread issues
        // all of its 16-byte loads before its LDS stores
        const uint32_t kbase = c0 * F::CK;
        const uint32_t smask = (1u << a.seg_shift) - 1u;
        uint4 sv[SPT];
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            const uint32_t s = threadIdx.x + 64u * WAVES * KW * i;
            const uint32_t m = s >> a.seg_shift, col = kbase + (s & smask) * 8;
            sv[i] = make_uint4(0u, 0u, 0u, 0u);
            if (m < a.rows && col < a.k) sv[i] = *(const uint4 *)(a.a + (size_t)m * a.k + col);
        }
        __syncthreads();   // the previous pass is done with LDS
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            const uint32_t s = threadIdx.x + 64u * WAVES * KW * i;
            if ((s >> a.seg_shift) < Mpad) *(uint4 *)(As + (size_t)(s >> a.seg_shift) * a.pitch + (s & smask) * 8) = sv[i];
        }
        if (SUMS) {
            __syncthreads();
            const uint32_t nsub = (c1 - c0) * F::CK / 32;
            for (uint32_t i = threadIdx.x; i < nsub * Mpad; i += 64u * WAVES * KW) {
                const uint32_t sub = i / Mpad, m = i % Mpad;
                const _Float16 *p8 = As + (size_t)m * a.pitch + sub * 32;
                float s = 0.0f;
#pragma unroll
                for (int t = 0; t < 32; ++t) s += (float)p8[t];
                Ss[i] = s;
            }
        }
        __syncthreads();
        if (!active) continue;

        auto compute = [&](typename F::W (&w)[PD], uint32_t cs) {
#pragma unroll
            for (int i = 0; i < PD; ++i)
                if (cs + i < m1) {
                    if constexpr (Defers<F>::value)
                        F::template mma_deferred<MT>(w[i], As, a.pitch, (cs + i - c0) * F::CK, lane, acc, pend);
                    else
                        F::template mma<MT>(w[i], As, a.pitch, (cs + i - c0) * F::CK, lane, Ss, 0, acc);
                }
        };
        uint32_t cs = m0;
        for (; cs + PD < m1; cs += 2 * PD) {
            load(wb, cs + PD);
            compute(wa, cs);
            if (cs + 2 * PD < m1) load(wa, cs + 2 * PD);
            compute(wb, cs + PD);
        }
        if (cs < m1) compute(wa, cs);
    }
    if constexpr (Defers<F>::value) flush_deferred<MT>(acc, pend);

    // add the K slices of each row group in slice order (LDS, reusing the A area)
    if (KW > 1) {
        float *red = (float *)smem;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __syncthreads();
#pragma unroll
            for (int v = 0; v < 16; ++v) red[((size_t)wave * 16 + v) * 64 + lane] = acc[mt][v];
            __syncthreads();
            if (kw == 0) {
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    float sum = red[((size_t)rgw * 16 + v) * 64 + lane];
                    for (int j = 1; j < KW; ++j) sum += red[((size_t)(j * WAVES + rgw) * 16 + v) * 64 + lane];
                    acc[mt][v] = sum;
                }
            }
        }
    }
    if (kw != 0 || !active) return;
    if (a.ksplit == 1 && !a.to_ws) {
        if (a.swiglu) store_swiglu<MT, false>(a, g, 0, lane, acc);
        else store_tile<MT>(a, g, 0, lane, acc);
        return;
    }
    // split-K: this split's tile goes to the workspace; gemm_reduce_kernel adds
    // the splits in order (the kernel boundary makes the partials visible)
    const uint32_t Npad = G * 32, n = g * 32 + (lane & 31);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < 16; ++v)
            __builtin_nontemporal_store(acc[mt][v], a.ws + ((size_t)ks * Mpad + out_row(mt, v, lane)) * Npad + n);
}

constexpr int kWideKR = 128;   // pass length of the forms that take several M tiles

// Bytes of one staging buffer of gemm_pipe_kernel: the activations (three
// bfloat16 planes with X32) and, where the format needs them, the per-block sums.
template <class F, int MT, int KR, bool X32, int VN>
constexpr uint32_t pipe_buf() {
    constexpr uint32_t rows = rows_staged<MT, VN>();
    constexpr uint32_t abytes = rows * (KR + 8) * 2 * (X32 ? 3 : 1);
    constexpr bool sums = X32 ? F::XSUM != 0.0f : NeedsSums<F>::value;
    constexpr bool flag = X32 && std::is_same<F, GF16>::value;   // an infinite activation was staged
    return (abytes + (sums ? (uint32_t)(KR / 32) * rows * 4 : flag ? 4u : 0u) + 15u) / 16u * 16u;
}

// Cross-pass pipelined form of gemm_mfma_kernel (quantised and F16 weights),
// with the pass length KR fixed at compile time. A is double-buffered in LDS:
// the activations of pass p + 1 are requested while pass p computes and are
// stored at its end; each wavefront keeps one pass of weight chunks in
// registers and requests chunk i of the next pass as soon as chunk i of the
// current one is consumed, so a pass's weights are in flight during the
// previous pass and the barrier between them. One barrier per pass (two for
// the K-quants at most 64 binary16 rows, whose activation sums are built from
// the staged pass; elsewhere they come from the lanes that stage a block).
// Workgroup: NW row groups x KW K slices of a pass. Products,
// scale rounding, slice order and outputs are those of gemm_mfma_kernel.
// X32: binary32 activations, split into three bfloat16 parts as they are
// stored to LDS (three planes per buffer).
template <class F, int MT, int KW, int KR, bool X32, int NW = WAVES, int VN = 16>
__global__ __launch_bounds__(64 * NW * KW) void gemm_pipe_kernel(GemmArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr bool WIDE = KW == 1;   // the form for more than 64 rows
    constexpr bool SUMS = NeedsSums<F>::value && !X32;
    constexpr int NT = 64 * NW * KW;   // threads
    constexpr int PC = KR / F::CK;        // chunks per pass
    constexpr int CPW = PC / KW;          // chunks per wavefront per pass
    constexpr int MP = rows_staged<MT, VN>();   // padded rows
    constexpr int PITCH = KR + 8;         // LDS row pitch in halves
    constexpr int SEGS = KR / 8;          // 16-byte segments per row of a pass
    constexpr int SPT = (MP * SEGS + NT - 1) / NT;   // segments per thread
    constexpr bool PART = SPT * NT != MP * SEGS;     // the last wavefronts stage nothing
    static_assert(CPW >= 1 && CPW * KW == PC && (!PART || SPT == 1) && MP * SEGS % 64 == 0, "pass shape");
    static_assert(!X32 || !std::is_same<F, GF16>::value || CPW % 4 == 0, "parts of 64 of K");
    constexpr uint32_t PLANE = (uint32_t)MP * PITCH;   // halves of one staged part
    constexpr uint32_t ABYTES = PLANE * 2 * (X32 ? 3 : 1);
    constexpr uint32_t BUF = pipe_buf<F, MT, KR, X32, VN>();
    constexpr bool FLAG = X32 && std::is_same<F, GF16>::value;   // one word per buffer after the activations
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: scalar chunk bases
    const int rgw = wave % NW, kw = wave / NW;
    const uint32_t G = (a.n + 31) / 32;
    // Workgroup -> (weight tile, M tile). With several M tiles, those of one
    // weight tile are consecutive on one XCD (workgroup ids go round the 8
    // XCDs), so they share the tile's weights in that XCD's L2.
    uint32_t tile = blockIdx.x, mtile = 0;
    if (KR == kWideKR && a.mtiles > 1) {
        const uint32_t local = blockIdx.x >> 3;
        tile = (local / a.mtiles) * 8 + (blockIdx.x & 7u);
        mtile = local % a.mtiles;
        if (tile >= a.tiles) return;
    }
    const uint32_t g = tile * NW + rgw, ks = blockIdx.y, m0 = KR == kWideKR ? mtile * MP : 0;
    const bool active = g < G;
    const uint32_t p_begin = ks * a.passes_per_wg;
    const uint32_t p_end = min(a.total_passes, p_begin + a.passes_per_wg);

    f16x acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = (f16x){};
    Deferred<MT> pend;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) pend.t[mt] = (f16x){};
    pend.d = 0.0f;
    // X32: 256 of K are summed on their own (part) and then added to acc, so
    // the sum over K takes one long rounding per 256 and not one per block.
    f16x part[MT];
    if constexpr (X32)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) part[mt] = (f16x){};
    // F16 weights: part holds 64 of K and mid up to 8 of those, as the products
    // themselves leave less room there (rms error 1.04 of the row kernels' over
    // 32000x4096 at 40 rows without mid, 0.92 with it).
    constexpr bool FINE = X32 && std::is_same<F, GF16>::value;
    f16x mid[FINE ? MT : 1];
    if constexpr (FINE)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) mid[mt] = (f16x){};
    auto join = [&](f16x (&to)[MT], f16x (&from)[MT]) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
            for (int v = 0; v < VN; ++v) to[mt][v] += from[mt][v];
            from[mt] = (f16x){};
        }
    };
    typename F::W w[CPW];
    uint4 sv[SPT * (X32 ? 2 : 1)];

    // Every wavefront issues the same sequence of loads whatever the shape
    // (addresses clamped into range, out-of-range A zeroed when stored,
    // inactive wavefronts stream a real row group and discard it), so the
    // compiler's load counters stay exact and no wait covers a later load.
    const uint32_t gl = active ? g : G - 1;
    auto load_a = [&](uint32_t p) {
        const uint32_t kbase = p * KR;
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            const uint32_t s = threadIdx.x + NT * i;
            const uint32_t m = min(m0 + s / SEGS, a.rows - 1), col = min(kbase + (s % SEGS) * 8, a.k - 8);
            if constexpr (X32) {
                const uint4 *p = (const uint4 *)(a.a32 + (size_t)m * a.k + col);
                sv[2 * i] = p[0];
                sv[2 * i + 1] = p[1];
            } else {
                sv[i] = *(const uint4 *)(a.a + (size_t)m * a.k + col);
            }
        }
    };
    // the sum t of segment s joins those of its 32-element block (the four
    // lanes of a quad) in the stage's [sub-block][row] sums
    auto put_sum = [&](uint32_t p, uint32_t s, float t) {
        t += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0xb1, 0xf, 0xf, false));
        t += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x4e, 0xf, 0xf, false));
        float *Ss = (float *)(smem + (p & 1) * BUF + ABYTES);
        if (!(threadIdx.x & 3)) Ss[(s % SEGS) / 4 * MP + s / SEGS] = t;
    };
    auto store_a = [&](uint32_t p) {
        _Float16 *As = (_Float16 *)(smem + (p & 1) * BUF);
        const uint32_t kbase = p * KR;
        if (PART && threadIdx.x >= MP * SEGS) return;
#pragma unroll
        for (int i = 0; i < SPT; ++i) {
            const uint32_t s = threadIdx.x + NT * i;
            const bool ok = m0 + s / SEGS < a.rows && kbase + (s % SEGS) * 8 < a.k;
            if constexpr (X32) {
                const uint4 lo = sv[2 * i], hi = sv[2 * i + 1];
                const uint32_t u[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = ok ? __uint_as_float(u[e]) * F::XMUL : 0.0f;
                uint4 part[3];
                const bool inf = split_x8<F::ORDER4>(x, part);
                if (FLAG && inf) *(uint32_t *)(smem + (p & 1) * BUF + ABYTES) = 1u;
                _Float16 *at = As + (s / SEGS) * PITCH + (s % SEGS) * 8;
#pragma unroll
                for (int j = 0; j < 3; ++j) *(uint4 *)(at + j * PLANE) = part[j];
                if constexpr (F::XSUM != 0.0f)
                    put_sum(p, s, F::XSUM * F::WMUL * (((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]))));
                continue;
            }
            const uint4 v = ok ? sv[i] : make_uint4(0u, 0u, 0u, 0u);
            *(uint4 *)(As + (s / SEGS) * PITCH + (s % SEGS) * 8) = v;
            if constexpr (SUMS && WIDE) {
                const h8 x = __builtin_bit_cast(h8, v);
                const float t = (((float)x[0] + (float)x[1]) + ((float)x[2] + (float)x[3])) +
                                (((float)x[4] + (float)x[5]) + ((float)x[6] + (float)x[7]));
                put_sum(p, s, t);
            }
        }
    };
    // the sums of a staged pass, by a pass over it (with two M tiles the lanes'
    // own sums cost the registers that let two workgroups share a CU)
    auto sums = [&](uint32_t p) {
        const _Float16 *As = (const _Float16 *)(smem + (p & 1) * BUF);
        float *Ss = (float *)(smem + (p & 1) * BUF + ABYTES);
        const uint32_t c0 = p * PC, c1 = min(a.chunks, c0 + PC);
        const uint32_t n = (c1 - c0) * F::CK / 32 * MP;
        for (uint32_t i = threadIdx.x; i < n; i += NT) {
            const _Float16 *p8 = As + (i % MP) * PITCH + (i / MP) * 32;
            float t = 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) t += (float)p8[j];
            Ss[i] = t;
        }
        __syncthreads();
    };
    // chunk i of this wavefront's slice of pass p (K-tail slots repeat the
    // pass's last chunk and are not computed)
    auto chunk_of = [&](uint32_t p, int i) {
        return min(p * PC + kw * CPW + i, min(a.chunks, (p + 1) * PC) - 1);
    };
    // compute pass p from LDS buffer p & 1; with LOAD, request chunk i of pass
    // p + 1 into slot i as soon as slot i is consumed
    auto pass = [&](uint32_t p, auto load_next) {
        const _Float16 *As = (const _Float16 *)(smem + (p & 1) * BUF);
        const float *Ss = (const float *)(smem + (p & 1) * BUF + ABYTES);
        const uint32_t c1 = min(a.chunks, (p + 1) * PC), cw = p * PC + kw * CPW;
        // F16: Ss is the flag of an infinite activation in the staged passes
        const uint32_t inf = X32 && FLAG ? __builtin_amdgcn_readfirstlane(*(const uint32_t *)Ss) : 0u;
#pragma unroll
        for (int i = 0; i < CPW; ++i) {
            // Only the last pass can end before its last chunk. The wide form
            // takes the others without a branch (a branch per chunk costs it a
            // register copy of every result tile where the paths meet); with
            // one or two M tiles the branches keep the chunks' order for less.
            if ((WIDE && decltype(load_next)::value) || cw + i < c1) {
                if constexpr (X32)
                    F::template mma_x32<MT, true, VN>(w[i], As, PLANE, PITCH, (uint32_t)(kw * CPW + i) * F::CK,
                                            FLAG ? inf : cw + i, lane, Ss, part, pend);
                else if constexpr (Defers<F>::value)
                    F::template mma_deferred<MT, WIDE, VN>(w[i], As, PITCH, (uint32_t)(kw * CPW + i) * F::CK, lane, acc, pend);
                else
                    F::template mma<MT, WIDE, VN>(w[i], As, PITCH, (uint32_t)(kw * CPW + i) * F::CK, lane, Ss, p * PC, acc);
            }
            if constexpr (FINE)
                if (i % 4 == 3) join(mid, part);
            if (decltype(load_next)::value) w[i] = F::load(a, gl, chunk_of(p + 1, i), lane);
            if constexpr (WIDE) __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (FINE) {
            constexpr uint32_t N = 32 / CPW;   // passes to 8 parts
            if ((p - p_begin) % N == N - 1 || !decltype(load_next)::value) join(acc, mid);
        } else if constexpr (X32) {
            if (KR >= 256 || ((p - p_begin) & 1u) || !decltype(load_next)::value) join(acc, part);
        }
    };

    if (p_begin < p_end) {
        const uint32_t last = p_end - 1;
        load_a(p_begin);
        if constexpr (FLAG) {   // never cleared again: a set flag costs later passes time, not results
            if (threadIdx.x < 2) *(uint32_t *)(smem + threadIdx.x * BUF + ABYTES) = 0u;
            __syncthreads();
        }
#pragma unroll
        for (int i = 0; i < CPW; ++i) w[i] = F::load(a, gl, chunk_of(p_begin, i), lane);
        store_a(p_begin);
        load_a(min(p_begin + 1, last));
        __syncthreads();
        if constexpr (SUMS && !WIDE) sums(p_begin);
        for (uint32_t p = p_begin; p < last; ++p) {
            pass(p, std::true_type{});
            store_a(p + 1);   // that buffer was last read in pass p - 1
            load_a(min(p + 2, last));
            __syncthreads();
            if constexpr (SUMS && !WIDE) sums(p + 1);
        }
        pass(last, std::false_type{});
    }
    if constexpr (X32 && std::is_same<F, GF16>::value) pend.d = 1.0f;   // the small parts
    if constexpr (X32 ? !NeedsSums<F>::value : Defers<F>::value) flush_deferred<MT, VN>(acc, pend);

    if (KW > 1) {
        float *red = (float *)smem;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            __syncthreads();
#pragma unroll
            for (int v = 0; v < VN; ++v) red[((size_t)wave * 16 + v) * 64 + lane] = acc[mt][v];
            __syncthreads();
            if (kw == 0) {
#pragma unroll
                for (int v = 0; v < VN; ++v) {
                    float sum = red[((size_t)rgw * 16 + v) * 64 + lane];
                    for (int j = 1; j < KW; ++j) sum += red[((size_t)(j * NW + rgw) * 16 + v) * 64 + lane];
                    acc[mt][v] = sum;
                }
            }
        }
    }
    if (kw != 0 || !active) return;
    if (a.ksplit == 1 && !a.to_ws) {
        if (a.swiglu) store_swiglu<MT, X32>(a, g, m0, lane, acc);
        else store_tile<MT>(a, g, m0, lane, acc);
        return;
    }
    const uint32_t Npad = G * 32, n = g * 32 + (lane & 31);
    const uint32_t mpad = MT * 32 * (KR == kWideKR ? a.mtiles : 1);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int v = 0; v < VN; ++v)
            __builtin_nontemporal_store(acc[mt][v], a.ws + ((size_t)ks * mpad + m0 + out_row(mt, v, lane)) * Npad + n);
}

// LDS bytes of gemm_pipe_kernel: two staging buffers, at least the K-slice
// reduction area.
template <class F, int MT, int KW, int KR, bool X32, int NW, int VN>
constexpr size_t pipe_lds() {
    constexpr size_t buf = pipe_buf<F, MT, KR, X32, VN>();
    constexpr size_t red = (size_t)NW * KW * 16 * 64 * 4;
    static_assert(2 * buf <= 160 * 1024 && red <= 160 * 1024, "LDS");
    return 2 * buf > red ? 2 * buf : red;
}

constexpr size_t kHalfLds = 81 * 1024;   // more than half of a CU's 160 KB
template <class F, int MT, int KW, int KR, bool X32 = false, int NW = WAVES, int VN = 16>
void launch_pipe(janus_ctx *ctx, dim3 grid, const GemmArgs &a) {
    // thread-safe one-time set-up (a function-local static's initialiser)
    static const bool attr_set = [] {
        (void)hipFuncSetAttribute((const void *)gemm_pipe_kernel<F, MT, KW, KR, X32, NW, VN>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        return true;
    }();
    (void)attr_set;
    // Where the workgroups do not outnumber the CUs, each asks for more than
    // half of a CU's LDS: the dispatcher otherwise puts two on one CU and
    // leaves another idle.
    size_t lds = pipe_lds<F, MT, KW, KR, X32, NW, VN>();
    if (grid.x * grid.y <= (uint32_t)ctx->num_cus && lds < kHalfLds) lds = kHalfLds;
    hipLaunchKernelGGL((gemm_pipe_kernel<F, MT, KW, KR, X32, NW, VN>), grid, dim3(64 * NW * KW), lds, ctx->stream, a);
}

// Whether gemm_pipe_kernel has a form for at most 8 and 16 rows: one M tile of a
// quantised weight (14336x4096 at 8 binary16 rows: Q4_0 15.7 -> 13.4 us, Q5_K
// 21.8 -> 17.8; 11008x4096 Q4_K at 16 binary32 rows 25.7 -> 18.4). F16 weights
// have no scales to save and measured slower (32000x4096: 54 -> 66 us).
template <class F, int MT> constexpr bool trims_rows() { return MT == 1 && !std::is_same<F, GF16>::value; }

// gemm_pipe_kernel for the row count: at most 8, 16 or 32 rows of one M tile.
template <class F, int MT, int KW, int KR, bool X32>
void launch_pipe_rows(janus_ctx *ctx, dim3 grid, const GemmArgs &a) {
    if constexpr (trims_rows<F, MT>()) {
        if (a.rows <= 8) return launch_pipe<F, MT, KW, KR, X32, WAVES, 4>(ctx, grid, a);
        if (a.rows <= 16) return launch_pipe<F, MT, KW, KR, X32, WAVES, 8>(ctx, grid, a);
    }
    launch_pipe<F, MT, KW, KR, X32>(ctx, grid, a);
}

// Sums the split-K partials in split order and applies the epilogue. X32
// (binary32 activations): eight at a time as equals before they join the rest.
template <bool X32>
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs a, uint32_t Mpad) {
    const uint32_t Npad = (a.n + 31) / 32 * 32;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)a.rows * a.n) return;
    const uint32_t m = (uint32_t)(idx / a.n), n = (uint32_t)(idx % a.n);
    const float *p = a.ws + (size_t)m * Npad + n;
    const size_t stride = (size_t)Mpad * Npad;
    // split order; the loads of 8 splits are issued together
    float s = 0.0f;
    for (uint32_t j0 = 0; j0 < a.ksplit; j0 += 8) {
        float u[8];
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) u[jj] = j0 + jj < a.ksplit ? p[(j0 + jj) * stride] : 0.0f;
        if constexpr (X32) {
            s += ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
            continue;
        }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
            if (j0 + jj < a.ksplit) s += u[jj];
    }
    if (a.resid) s += a.resid[idx];
    if (a.c_f16) ((uint16_t *)a.c)[idx] = f2h_bits(s);
    else ((float *)a.c)[idx] = s;
}

// ---- T32 repack (one thread per lane of a chunk) -----------------------------

// Nibble slot of element j (0..7) within a T32 word.
__device__ __forceinline__ uint32_t nib_slot(int j) { return (uint32_t)((j >> 1) + 4 * (j & 1)); }

// Q4_0 / Q4_K word: nibbles nib(j), j = 0..7, in T32 slot order.
template <class GetNib>
__device__ __forceinline__ uint32_t pack_word(GetNib nib) {
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) w |= (nib(j) & 15u) << (4 * nib_slot(j));
    return w;
}

__global__ void t32_q4_0_kernel(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ sc, uint8_t *dq,
                                uint32_t *dside, uint32_t n, uint32_t k, uint32_t G, uint32_t C) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)G * C * 64) return;
    const int lane = (int)(t & 63), h = lane >> 5;
    const size_t ch = t >> 6;
    const uint32_t g = (uint32_t)(ch / C), c = (uint32_t)(ch % C);
    const uint32_t r = g * 32 + (lane & 31), nb = k / 32;
    uint32_t words[4] = {0u, 0u, 0u, 0u};
    uint16_t s[2] = {0, 0};
    for (int b = 0; b < 2; ++b) {
        const uint32_t blk = 2 * c + b;
        if (r >= n || blk >= nb) continue;
        const uint8_t *q = qs + ((size_t)r * nb + blk) * 16;
        words[2 * b] = pack_word([&](int j) { return (uint32_t)(q[8 * h + j] & 15); });
        words[2 * b + 1] = pack_word([&](int j) { return (uint32_t)(q[8 * h + j] >> 4); });
        s[b] = sc[(size_t)r * nb + blk];
    }
    *(uint4 *)(dq + t * 16) = make_uint4(words[0], words[1], words[2], words[3]);
    if (lane < 32) dside[ch * 32 + lane] = (uint32_t)s[0] | ((uint32_t)s[1] << 16);
}

__global__ void t32_q4_k_kernel(const uint8_t *__restrict__ blocks, uint8_t *dq, uint8_t *dside, uint32_t n,
                                uint32_t k, uint32_t G, uint32_t C) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)G * C * 64) return;
    const int lane = (int)(t & 63), h = lane >> 5;
    const size_t ch = t >> 6;
    const uint32_t g = (uint32_t)(ch / C), c = (uint32_t)(ch % C);
    const uint32_t r = g * 32 + (lane & 31), nsb = k / 256, sb = c / 4, j = c % 4;
    uint32_t words[4] = {0u, 0u, 0u, 0u};
    uint4 hdr = {0u, 0u, 0u, 0u};
    if (r < n) {
        const uint8_t *blk = blocks + ((size_t)r * nsb + sb) * 144;
        const uint8_t *q = blk + 16 + 32 * j;
        for (int b = 0; b < 2; ++b) {   // sub-block 2j + b: nibble b of bytes 32j + i
            const int sh = 4 * b;
            words[2 * b] = pack_word([&](int e) { return (uint32_t)(q[8 * h + e] >> sh); });
            words[2 * b + 1] = pack_word([&](int e) { return (uint32_t)(q[16 + 8 * h + e] >> sh); });
        }
        hdr = *(const uint4 *)blk;
    }
    *(uint4 *)(dq + t * 16) = make_uint4(words[0], words[1], words[2], words[3]);
    if (lane < 32 && j == 0) *(uint4 *)(dside + (((size_t)g * (C / 4) + sb) * 32 + lane) * 16) = hdr;
}

__global__ void t32_q5_k_kernel(const uint8_t *__restrict__ blocks, uint8_t *dq, uint8_t *dside, uint32_t *dfifth,
                                uint32_t n, uint32_t k, uint32_t G, uint32_t C) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)G * C * 64) return;
    const int lane = (int)(t & 63), h = lane >> 5;
    const size_t ch = t >> 6;
    const uint32_t g = (uint32_t)(ch / C), c = (uint32_t)(ch % C);
    const uint32_t r = g * 32 + (lane & 31), nsb = k / 256, sb = c / 4, j = c % 4;
    uint32_t words[4] = {0u, 0u, 0u, 0u}, fifth = 0u;
    uint4 hdr = {0u, 0u, 0u, 0u};
    if (r < n) {
        const uint8_t *blk = blocks + ((size_t)r * nsb + sb) * 176, *qs = blk + 48;
        // the upload's fifth-bit words: one per 16-byte quant chunk, bit
        // 8 (t % 4) + t / 4 (+ 4 for the high nibble) for quant byte t
        const uint32_t *qh = (const uint32_t *)(blk + 16);
        for (int b = 0; b < 2; ++b) {   // sub-block 2j + b: nibble b of bytes 32j + E
            for (int w = 0; w < 2; ++w) {
                const int i = 2 * b + w;
                words[i] = pack_word([&](int e) { return (uint32_t)(qs[32 * j + 16 * w + 8 * h + e] >> (4 * b)); });
                for (int e = 0; e < 8; ++e) {
                    const uint32_t tq = (uint32_t)(8 * h + e), pos = 8 * (tq % 4) + tq / 4 + 4 * (uint32_t)b;
                    const uint32_t bit = (qh[2 * j + w] >> pos) & 1u;
                    fifth |= bit << (4 * nib_slot(e) + (uint32_t)i);
                }
            }
        }
        hdr = *(const uint4 *)blk;
    }
    *(uint4 *)(dq + t * 16) = make_uint4(words[0], words[1], words[2], words[3]);
    dfifth[t] = fifth;
    if (lane < 32 && j == 0) *(uint4 *)(dside + (((size_t)g * (C / 4) + sb) * 32 + lane) * 16) = hdr;
}

__global__ void t32_q8_0_kernel(const uint8_t *__restrict__ qs, const uint16_t *__restrict__ sc, uint8_t *dq,
                                uint16_t *dside, uint32_t n, uint32_t k, uint32_t G, uint32_t C) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)G * C * 64) return;
    const int lane = (int)(t & 63), h = lane >> 5;
    const size_t ch = t >> 6;
    const uint32_t g = (uint32_t)(ch / C), c = (uint32_t)(ch % C);
    const uint32_t r = g * 32 + (lane & 31), nb = k / 32;
    uint8_t out[16] = {0};
    uint16_t s = 0;
    if (r < n) {
        const uint8_t *q = qs + ((size_t)r * nb + c) * 32;
        for (int e = 0; e < 8; ++e) {
            out[e] = q[8 * h + e];
            out[8 + e] = q[16 + 8 * h + e];
        }
        s = sc[(size_t)r * nb + c];
    }
    uint4 v;
    std::memcpy(&v, out, 16);
    *(uint4 *)(dq + t * 16) = v;
    if (lane < 32) dside[ch * 32 + lane] = s;
}

// nonfinite is set when any weight is infinite or NaN (cleared by the caller).
__global__ void t32_f16_kernel(const uint16_t *__restrict__ src, uint8_t *dq, uint32_t n, uint32_t k, uint32_t G,
                               uint32_t C, uint32_t *nonfinite) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)G * C * 64) return;
    const int lane = (int)(t & 63), h = lane >> 5;
    const size_t ch = t >> 6;
    const uint32_t g = (uint32_t)(ch / C), c = (uint32_t)(ch % C);
    const uint32_t r = g * 32 + (lane & 31);
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    const uint32_t k0 = c * 16 + 8 * h;
    if (r < n && k0 < k) {   // k % 8 == 0 (mfma_gemm_supported): whole 16-byte groups
        v = *(const uint4 *)(src + (size_t)r * k + k0);
        const uint32_t u[4] = {v.x, v.y, v.z, v.w};
        bool bad = false;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            bad |= (u[i] & 0x7c00u) == 0x7c00u || (u[i] & 0x7c000000u) == 0x7c000000u;
        if (bad) *nonfinite = 1u;
    }
    *(uint4 *)(dq + t * 16) = v;
}

uint32_t chunk_k(int type) {
    switch (type) {
    case JANUS_DT_Q4_0: case JANUS_DT_Q4_K: case JANUS_DT_Q5_K: return 64;
    case JANUS_DT_Q8_0: return 32;
    default: return 16;
    }
}

// Builds the weight's T32 copy (device memory, kept with the weight). Several
// threads, each with its context, may come here with one weight. exact: only a
// copy with exact parts is of use; for a weight that has none, t32_nonfinite is
// set and nothing kept.
int t32_ensure(janus_ctx *ctx, janus_weight *w, bool exact = false) {
    if (w->t32) return JANUS_OK;
    std::lock_guard<std::mutex> lock(w->t32_mu);
    if (w->t32 || (exact && w->t32_nonfinite)) return JANUS_OK;
    const uint32_t G = (w->n + 31) / 32, ck = chunk_k(w->type);
    const uint32_t C = (w->k + ck - 1) / ck;
    const size_t qbytes = (size_t)G * C * 64 * 16;
    size_t side = 0;
    if (w->type == JANUS_DT_Q4_0) side = (size_t)G * C * 32 * 4;
    else if (w->type == JANUS_DT_Q8_0) side = (size_t)G * C * 32 * 2;
    else if (w->type == JANUS_DT_Q4_K || w->type == JANUS_DT_Q5_K) side = (size_t)G * (C / 4) * 32 * 16;
    const size_t fifth = w->type == JANUS_DT_Q5_K ? (size_t)G * C * 64 * 4 : 0;
    void *mem = nullptr;
    JANUS_HIP_CHECK(ctx, hipMalloc(&mem, qbytes + side + fifth + 256));
    uint32_t *nonfinite = (uint32_t *)((uint8_t *)mem + qbytes + side + fifth);   // all multiples of 64 bytes
    uint32_t bad = 0;
    uint8_t *dq = (uint8_t *)mem, *ds = (uint8_t *)mem + qbytes;
    uint32_t *df = (uint32_t *)((uint8_t *)mem + qbytes + side);
    const size_t threads = (size_t)G * C * 64;
    const dim3 grid((unsigned)((threads + 255) / 256)), block(256);
    switch (w->type) {
    case JANUS_DT_Q4_0:
        hipLaunchKernelGGL(t32_q4_0_kernel, grid, block, 0, ctx->stream, w->qs, w->sc, dq, (uint32_t *)ds, w->n,
                           w->k, G, C);
        break;
    case JANUS_DT_Q4_K:
        hipLaunchKernelGGL(t32_q4_k_kernel, grid, block, 0, ctx->stream, w->qs, dq, ds, w->n, w->k, G, C);
        break;
    case JANUS_DT_Q5_K:
        hipLaunchKernelGGL(t32_q5_k_kernel, grid, block, 0, ctx->stream, w->qs, dq, ds, df, w->n, w->k, G, C);
        break;
    case JANUS_DT_Q8_0:
        hipLaunchKernelGGL(t32_q8_0_kernel, grid, block, 0, ctx->stream, w->qs, w->sc, dq, (uint16_t *)ds, w->n,
                           w->k, G, C);
        break;
    default:
        (void)hipMemsetAsync(nonfinite, 0, 4, ctx->stream);
        hipLaunchKernelGGL(t32_f16_kernel, grid, block, 0, ctx->stream, (const uint16_t *)w->qs, dq, w->n, w->k, G,
                           C, nonfinite);
        (void)hipMemcpyAsync(&bad, nonfinite, 4, hipMemcpyDeviceToHost, ctx->stream);
        break;
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e != hipSuccess) {
        (void)hipFree(mem);   // already failing: the repack error is the one reported
        return hip_fail(ctx, e, "t32 repack");
    }
    w->t32_nonfinite = bad != 0;
    if (exact && bad) {
        (void)hipFree(mem);
        return JANUS_OK;
    }
    w->t32_qs = dq;
    w->t32_side = ds;
    w->t32_q5h = fifth ? df : nullptr;
    w->t32_chunks = C;
    w->t32 = mem;
    return JANUS_OK;
}

template <class F, int MT>
constexpr int gemm_kw() {
    return (MT == 1 && std::is_same<F, GF16>::value) ? 4 : 2;
}

int launch_reduce(janus_ctx *ctx, const GemmArgs &a, uint32_t mpad) {
    const size_t total = (size_t)a.rows * a.n;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (a.a32) hipLaunchKernelGGL(gemm_reduce_kernel<true>, grid, dim3(256), 0, ctx->stream, a, mpad);
    else hipLaunchKernelGGL(gemm_reduce_kernel<false>, grid, dim3(256), 0, ctx->stream, a, mpad);
    JANUS_LAUNCH_CHECK(ctx);
    return JANUS_OK;
}

// kr_force / ks_force (0 = automatic) fix the pass length and the K split.
template <class F, int MT, int KW = gemm_kw<F, MT>(), int PD = Stage<F>::PD>
int launch_mfma(janus_ctx *ctx, GemmArgs a, const janus_weight *w, GemmPartials *parts, uint32_t kr_force = 0,
                uint32_t ks_force = 0) {
    constexpr int SPT1 = 16 / KW;   // kr = 1024 / MT
    if (!kr_force && !ks_force) {   // context-wide overrides (measurement)
        kr_force = ctx->gemm_kr;
        ks_force = ctx->gemm_ks;
    }
    const uint32_t G = (w->n + 31) / 32;
    const uint32_t tiles = (G + WAVES - 1) / WAVES;
    // K per LDS pass: 1024 (M <= 32) or 512 (M <= 64); products with too few
    // (tile, pass) pairs for two workgroups per CU use half-size passes
    const uint32_t want = 2u * (uint32_t)ctx->num_cus;
    uint32_t kr = MT == 1 ? 1024 : 512;
    if (tiles * ((w->t32_chunks * F::CK + kr - 1) / kr) < want && kr / F::CK >= 2 * KW) kr /= 2;
    uint32_t ks = 0;
    bool pipe = false;
    {
        // pipelined kernel (F16 LM head 128256x4096 at M = 32: 181.5 us
        // against 209.3 single-buffered; 512- / 1024-long passes 182.8 /
        // 188.4 us): 256-long passes, K split until
        // about 1.1 workgroups per CU, used when every workgroup then runs at
        // least 3 passes (fewer leave nothing to overlap)
        if (ctx->gemm_pipe && !kr_force && !ks_force) {
            const uint32_t pp = (w->t32_chunks * F::CK + 255) / 256;
            uint32_t pks = ((uint32_t)ctx->num_cus * 11 + 10 * tiles - 1) / (10 * tiles);
            // two M tiles: as many workgroups as run at once, one per CU for
            // Q4_0 (158 registers), two for the other formats (14336x4096 at 33
            // rows: Q4_0 26.4 -> 21.2 us with 224 workgroups instead of 336,
            // Q5_K 31.2 -> 28.5 with 448)
            if (MT == 2) pks = (uint32_t)ctx->num_cus * (std::is_same<F, GQ4_0>::value ? 1u : 2u) / tiles;
            if (pks > pp) pks = pp;
            if (pks < 1) pks = 1;
            if ((pp + pks - 1) / pks >= 3) {
                kr = 256;
                ks = pks;
                pipe = true;
            }
        } else if (ctx->gemm_pipe) {
            pipe = true;   // forced shapes use it wherever there are several passes per workgroup
        }
    }
    if (kr_force) kr = kr_force;
    if (kr % (F::CK * KW) || kr * MT > 2048) return fail(ctx, JANUS_E_INVALID_DIM, "gemm: bad pass length");
    a.pass_chunks = kr / F::CK;
    a.seg_shift = 0;
    while ((8u << a.seg_shift) < kr) ++a.seg_shift;
    if ((8u << a.seg_shift) != kr) return fail(ctx, JANUS_E_INVALID_DIM, "gemm: pass length must be a power of two");
    a.chunks = w->t32_chunks;
    a.total_passes = (a.chunks + a.pass_chunks - 1) / a.pass_chunks;
    // split K over workgroups until there are about two workgroups per CU
    if (!ks) ks = (want + tiles - 1) / tiles;
    if (ks_force) ks = ks_force;
    if (ks > a.total_passes) ks = a.total_passes;
    if (ks < 1) ks = 1;
    a.passes_per_wg = (a.total_passes + ks - 1) / ks;
    a.ksplit = (a.total_passes + a.passes_per_wg - 1) / a.passes_per_wg;
    a.pitch = a.pass_chunks * F::CK + 8;
    const bool sums = NeedsSums<F>::value;
    size_t lds = (size_t)MT * 32 * a.pitch * 2 + (sums ? (size_t)(kr / 32) * MT * 32 * 4 : 0);
    const size_t red = (size_t)WAVES * KW * 16 * 64 * 4;   // K-slice reduction, one M-tile at a time
    if (lds < red) lds = red;
    a.to_ws = parts != nullptr;
    size_t need = 0;
    if (a.ksplit > 1 || parts) {
        need = (size_t)a.ksplit * MT * 32 * G * 32 * 4;
        const size_t epi = parts ? (size_t)MT * 32 * kEpiSlices * 4 : 0;   // the epilogues' per-row area
        if (int e = ensure_gemm_ws(ctx, need + epi)) return e;
        a.ws = (float *)ctx->gemm_ws;
    }
    static const bool attr_set = [] {   // thread-safe one-time set-up
        (void)hipFuncSetAttribute((const void *)gemm_mfma_kernel<F, MT, KW, SPT1, PD>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        (void)hipFuncSetAttribute((const void *)gemm_mfma_kernel<F, MT, KW, 2 * SPT1, PD>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        return true;
    }();
    (void)attr_set;
    const dim3 grid(tiles, a.ksplit), block(64 * WAVES * KW);
    // the cross-pass pipelined kernel for the usual pass lengths
    bool piped = false;
    {
        if (pipe && a.passes_per_wg > 1) {
            piped = true;
            if (kr == 256) launch_pipe_rows<F, MT, KW, 256, false>(ctx, grid, a);
            else if (kr == 512) launch_pipe<F, MT, KW, 512>(ctx, grid, a);
            else if (MT == 1 && kr == 1024) launch_pipe<F, MT, KW, 1024 / MT>(ctx, grid, a);
            else piped = false;
        }
    }
    if (!piped && kr * MT <= 1024) hipLaunchKernelGGL((gemm_mfma_kernel<F, MT, KW, SPT1, PD>), grid, block, lds, ctx->stream, a);
    else if (!piped) hipLaunchKernelGGL((gemm_mfma_kernel<F, MT, KW, 2 * SPT1, PD>), grid, block, lds, ctx->stream, a);
    JANUS_LAUNCH_CHECK(ctx);
    if (parts) {
        parts->ws = a.ws;
        parts->ksplit = a.ksplit;
        parts->mpad = MT * 32;
        parts->npad = G * 32;
        parts->ss = a.ws + need / 4;
        return JANUS_OK;
    }
    if (a.ksplit > 1) return launch_reduce(ctx, a, MT * 32);
    return JANUS_OK;
}

template <int MT>
int launch_mt(janus_ctx *ctx, const GemmArgs &a, const janus_weight *w, GemmPartials *parts) {
    switch (w->type) {
    case JANUS_DT_Q4_0: return launch_mfma<GQ4_0, MT>(ctx, a, w, parts);
    case JANUS_DT_Q8_0: return launch_mfma<GQ8_0, MT>(ctx, a, w, parts);
    case JANUS_DT_Q4_K: return launch_mfma<GQ4_K, MT>(ctx, a, w, parts);
    case JANUS_DT_Q5_K: return launch_mfma<GQ5_K, MT>(ctx, a, w, parts);
    default: return launch_mfma<GF16, MT>(ctx, a, w, parts);
    }
}

// Splits the product for gemm_pipe_kernel on binary32 activations: fills the
// plan fields of a and returns the workspace bytes (0: no K split). MT M-tiles
// of 32 rows, KR-long passes. The staged parts of 32 and more rows fill most of
// a CU's LDS, so one workgroup runs per CU and K is split as far as the
// workgroups still fit in one round; with at most 16 rows two run, and K is
// split until there are two per CU (11008x4096 at 16 rows: 18.4 us against
// 20.4 with 344 workgroups and 23.0 with 172).
template <class F, int MT, int KR>
size_t plan_x32(const janus_ctx *ctx, GemmArgs &a, const janus_weight *w, dim3 &grid) {
    const uint32_t G = (w->n + 31) / 32, tiles = (G + WAVES - 1) / WAVES;
    a.chunks = w->t32_chunks;
    a.pass_chunks = KR / F::CK;
    a.total_passes = (a.chunks + a.pass_chunks - 1) / a.pass_chunks;
    uint32_t ks = (uint32_t)ctx->num_cus / tiles;
    if (trims_rows<F, MT>() && a.rows <= 16) ks = (2 * (uint32_t)ctx->num_cus + tiles - 1) / tiles;
    if (ks > a.total_passes) ks = a.total_passes;
    if (ks < 1) ks = 1;
    a.passes_per_wg = (a.total_passes + ks - 1) / ks;
    a.ksplit = (a.total_passes + a.passes_per_wg - 1) / a.passes_per_wg;
    grid = dim3(tiles, a.ksplit);
    return a.ksplit > 1 ? (size_t)a.ksplit * MT * 32 * G * 32 * 4 : 0;
}

// Binary32 rows take the MFMA kernel where it beats a GEMV per row. Per call,
// two rows: 19-32 us per-row against 19-29 us at 14336x4096 and 4096x14336 (no
// clear winner); three rows: 29 / 26 / 34 / 60 us per-row (Q4_0, Q8_0 4096x14336,
// Q4_K, F16 14336x4096) against 23 / 24 / 26 / 31; 16 rows 144 / 229 / 172 / 315
// against 23 / 25 / 25 / 31; 64 rows 565-1248 against 40-58. Launch-bound sizes
// (256 to 1024 square) cost 4-8 us against 2.4-3.5 us a row, so they gain from
// three rows too, but three rows below 2^20 weights stay with the row kernels:
// their results equal single calls bit for bit, and the time at stake is 3 us.
// Rows longer than the row kernels take (2048 units) stay with them, refused.
bool x32_pays(const janus_weight *w, uint32_t rows) {
    if (w->k / (w->type == JANUS_DT_F16 ? 8u : 32u) > 2048u) return false;
    return rows > 3 || (rows == 3 && (uint64_t)w->n * w->k >= (1u << 20));
}

bool capturing(const janus_ctx *ctx) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(ctx->stream, &cs) != hipSuccess || cs != hipStreamCaptureStatusNone;
}

// Binary32 rows (at most 64) on the MFMA kernel. *ran stays false, with nothing
// launched and no error, when the workspace cannot grow (out of memory, or
// inside a capture): the caller then runs one GEMV per row, which needs none.
template <class F, int MT, int KW = gemm_kw<F, MT>()>
int launch_x32(janus_ctx *ctx, GemmArgs a, const janus_weight *w, GemmPartials *parts, bool *ran) {
    constexpr int KR = MT == 1 ? 256 : 128;
    dim3 grid;
    size_t need = plan_x32<F, MT, KR>(ctx, a, w, grid);
    const uint32_t npad = (w->n + 31) / 32 * 32;
    if (parts) need = (size_t)a.ksplit * MT * 32 * npad * 4;
    if (need > ctx->gemm_ws_bytes) {
        if (capturing(ctx)) return JANUS_OK;
        if (ensure_gemm_ws(ctx, need)) {
            (void)hipGetLastError();
            ctx->last_error.clear();
            return JANUS_OK;
        }
    }
    a.ws = (float *)ctx->gemm_ws;
    a.to_ws = parts != nullptr;
    *ran = true;
    launch_pipe_rows<F, MT, KW, KR, true>(ctx, grid, a);
    JANUS_LAUNCH_CHECK(ctx);
    if (parts) {
        *parts = GemmPartials{a.ws, a.ksplit, MT * 32, npad, nullptr};
        return JANUS_OK;
    }
    if (a.ksplit > 1) return launch_reduce(ctx, a, MT * 32);
    return JANUS_OK;
}

template <int MT>
int launch_x32_mt(janus_ctx *ctx, const GemmArgs &a, const janus_weight *w, GemmPartials *parts, bool *ran) {
    switch (w->type) {
    case JANUS_DT_Q4_0: return launch_x32<GQ4_0, MT>(ctx, a, w, parts, ran);
    case JANUS_DT_Q8_0: return launch_x32<GQ8_0, MT>(ctx, a, w, parts, ran);
    case JANUS_DT_Q4_K: return launch_x32<GQ4_K, MT>(ctx, a, w, parts, ran);
    case JANUS_DT_Q5_K: return launch_x32<GQ5_K, MT>(ctx, a, w, parts, ran);
    default: return launch_x32<GF16, MT>(ctx, a, w, parts, ran);
    }
}

// ---- more than 64 rows (prompts) -----------------------------------------------
// gemm_pipe_kernel over M tiles of 32 MT rows with 8 row groups per workgroup
// (256 weight rows) and no K slices: a staged activation tile serves all 8
// wavefronts, and a weight chunk is unpacked once for MT MFMA pairs. MT = 4 or 3
// for binary16 rows (2 x 35 KB of LDS at 4); three bfloat16 parts take 64 rows
// (MT = 2, 2 x 52 KB), 96 (MT = 3, not for F16 weights) or 64 with 4 row groups
// and two K slices, whichever launch_wide reckons the fastest. Bound by the
// VALU (one scale FMA per weight and 32 rows, 0.4 more to unpack) on binary16
// rows and by LDS reads of the parts on binary32 rows. Q4_0 28672x4096 at 512
// rows: 167 us when the forms were compared (178 in a traced prompt) against
// 229 with 4 row groups x 2 K slices and 186 with MT = 2; binary32 rows 411 us
// with MT = 2, 464 with 4 row groups, and 556 with MT = 3, which pays only where
// it saves a round of workgroups. A product with too few tiles for the CUs
// splits K over workgroups.
constexpr int kWideNW = 8;

template <class F, int MT, bool X32, int NW = kWideNW, int KW = 1>
int launch_wide_mt(janus_ctx *ctx, GemmArgs a, const janus_weight *w, GemmPartials *parts) {
    const uint32_t G = (w->n + 31) / 32;
    a.tiles = (G + NW - 1) / NW;
    a.mtiles = (a.rows + 32 * MT - 1) / (32 * MT);
    a.chunks = w->t32_chunks;
    a.pass_chunks = kWideKR / F::CK;
    a.total_passes = (a.chunks + a.pass_chunks - 1) / a.pass_chunks;
    const uint64_t wgs = (uint64_t)a.tiles * a.mtiles;
    uint64_t ks = a.swiglu ? 1 : (uint64_t)ctx->num_cus / wgs;
    if (ks > a.total_passes / 4) ks = a.total_passes / 4;
    if (ks < 1) ks = 1;
    a.passes_per_wg = (a.total_passes + (uint32_t)ks - 1) / (uint32_t)ks;
    a.ksplit = (a.total_passes + a.passes_per_wg - 1) / a.passes_per_wg;
    const uint32_t mpad = a.mtiles * MT * 32;
    a.to_ws = parts != nullptr;
    if (a.ksplit > 1 || parts) {
        if (int e = ensure_gemm_ws(ctx, (size_t)a.ksplit * mpad * G * 32 * 4)) return e;
        a.ws = (float *)ctx->gemm_ws;
    }
    const uint32_t gx = a.mtiles > 1 ? (a.tiles + 7) / 8 * 8 * a.mtiles : a.tiles;
    launch_pipe<F, MT, KW, kWideKR, X32, NW>(ctx, dim3(gx, a.ksplit), a);
    JANUS_LAUNCH_CHECK(ctx);
    if (parts) {
        *parts = GemmPartials{a.ws, a.ksplit, mpad, G * 32, nullptr};
        return JANUS_OK;
    }
    if (a.ksplit > 1) return launch_reduce(ctx, a, mpad);
    return JANUS_OK;
}

template <class F>
int launch_wide(janus_ctx *ctx, const GemmArgs &a, const janus_weight *w, GemmPartials *parts) {
    if (a.a32) {
        // the form with the fewest rounds of workgroups over the CUs, weighed by
        // what one takes: 64 rows x 8 row groups, 96 rows x 8, or 64 x 4 with
        // two K slices (Q4_K 22016x4096 at 133 rows: 258 workgroups of the
        // first kind need a second round for the last two)
        const uint64_t cus = (uint64_t)ctx->num_cus;
        auto time = [&](uint32_t rows, uint32_t nw, float unit) {
            const uint64_t wgs = ((w->n + 31) / 32 + nw - 1) / nw * (uint64_t)((a.rows + rows - 1) / rows);
            const uint64_t ks = a.swiglu || wgs > cus ? 1 : cus / wgs;
            return unit * (float)((wgs * ks + cus - 1) / cus) / (float)ks;
        };
        const float t2 = time(64, 8, 1.0f), t4 = time(64, 4, 0.57f);
        if constexpr (!std::is_same<F, GF16>::value) {   // F16's sums of 96 rows do not fit the registers
            const float t3 = time(96, 8, 1.45f);
            if (t3 < t2 && t3 <= t4) return launch_wide_mt<F, 3, true>(ctx, a, w, parts);
        }
        return t2 <= t4 ? launch_wide_mt<F, 2, true>(ctx, a, w, parts) : launch_wide_mt<F, 2, true, 4, 2>(ctx, a, w, parts);
    }
    // the M tile with the least padded work (per workgroup, unpacking and
    // staging cost about what 0.7 of an M subtile does)
    auto cost = [&](uint32_t mt) { return (float)((a.rows + 32 * mt - 1) / (32 * mt)) * ((float)mt + 0.7f); };
    return cost(4) <= cost(3) ? launch_wide_mt<F, 4, false>(ctx, a, w, parts) : launch_wide_mt<F, 3, false>(ctx, a, w, parts);
}

int launch_wide_any(janus_ctx *ctx, const GemmArgs &a, const janus_weight *w, GemmPartials *parts) {
    switch (w->type) {
    case JANUS_DT_Q4_0: return launch_wide<GQ4_0>(ctx, a, w, parts);
    case JANUS_DT_Q8_0: return launch_wide<GQ8_0>(ctx, a, w, parts);
    case JANUS_DT_Q4_K: return launch_wide<GQ4_K>(ctx, a, w, parts);
    case JANUS_DT_Q5_K: return launch_wide<GQ5_K>(ctx, a, w, parts);
    default: return launch_wide<GF16>(ctx, a, w, parts);
    }
}

GemmArgs make_args(const janus_weight *w, const void *a, void *c, int c_f16, uint32_t rows, const float *residual) {
    GemmArgs g;
    std::memset(&g, 0, sizeof(g));
    g.qs = w->t32_qs;
    g.side = w->t32_side;
    g.q5h = w->t32_q5h;
    g.a = (const _Float16 *)a;
    g.c = c;
    g.resid = residual;
    g.rows = rows;
    g.n = w->n;
    g.k = w->k;
    g.c_f16 = c_f16;
    g.mtiles = 1;
    return g;
}

// ---- batched epilogues over the split-K partials ------------------------------
// Each sums the splits of an element in split order, like gemm_reduce_kernel;
// the loads of up to 8 splits are issued together.

template <typename V>
__device__ __forceinline__ V sum_splits(const float *q, size_t stride, uint32_t ksplit) {
    V s = {};
    for (uint32_t k0 = 0; k0 < ksplit; k0 += 8) {
        V u[8];
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
            if (k0 + kk < ksplit) u[kk] = *(const V *)(q + (k0 + kk) * stride);
#pragma unroll
        for (int kk = 0; kk < 8; ++kk)
            if (k0 + kk < ksplit) s += u[kk];
    }
    return s;
}

__device__ __forceinline__ jf2 sum_pair(const GemmPartials &p, uint32_t m, uint32_t col) {
    return sum_splits<jf2>(p.ws + (size_t)m * p.npad + col, (size_t)p.mpad * p.npad, p.ksplit);
}

// Fused-QKV rows (RoPE pairs of q heads, of k heads, then v in order): rotate
// q into q_out [rows][heads * hd] (f32) and k, append k and v to the cache row
// rowbase[m] + pos[m] (m * max_seq + pos[m] without a table; the rotation of
// rope.wgsl:71-72, the row layout of kv_update_kernel).
template <typename KV>
__global__ __launch_bounds__(256) void epi_qkv_rope_kernel(GemmPartials p, QkvEpilogue e, uint32_t rows) {
    const uint32_t pairs = e.q_pairs + e.k_pairs + e.kv_row / 2;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)rows * pairs) return;
    const uint32_t m = (uint32_t)(idx / pairs), g = (uint32_t)(idx % pairs);
    const uint32_t pos = (uint32_t)e.pos[m];
    if (pos >= e.max_seq) return;   // host checks keep positions in range; never index past the tables
    const jf2 r = sum_pair(p, m, 2 * g);
    const size_t row = (e.rowbase ? (size_t)(uint32_t)e.rowbase[m] : (size_t)m * e.max_seq) + pos;
    if (g < e.q_pairs + e.k_pairs) {
        const bool isq = g < e.q_pairs;
        const uint32_t gg = isq ? g : g - e.q_pairs, h = gg / e.half_hd, i = gg % e.half_hd;
        const float2 cs = *(const float2 *)(e.rope + 2 * ((size_t)pos * e.half_hd + i));
        const float y0 = r.x * cs.x - r.y * cs.y;
        const float y1 = r.x * cs.y + r.y * cs.x;
        if (isq) {
            float *q = e.q + (size_t)m * e.q_pairs * 2 + (size_t)h * 2 * e.half_hd + i;
            q[0] = y0;
            q[e.half_hd] = y1;
        } else {
            KV *k = (KV *)e.kc + row * e.kv_row + (size_t)h * 2 * e.half_hd + i;
            k[0] = (KV)y0;
            k[e.half_hd] = (KV)y1;
        }
    } else {
        KV *v = (KV *)e.vc + row * e.kv_row + 2 * (size_t)(g - e.q_pairs - e.k_pairs);
        v[0] = (KV)r.x;
        v[1] = (KV)r.y;
    }
}

// Gate/up rows interleaved (gate_j, up_j): act[m][j] = silu(gate) * up (the
// SwiGLU of elementwise_kernel).
template <typename T>
__global__ __launch_bounds__(256) void epi_swiglu_kernel(GemmPartials p, T *act, uint32_t rows, uint32_t ffn) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)rows * ffn) return;
    const uint32_t m = (uint32_t)(idx / ffn), j = (uint32_t)(idx % ffn);
    const jf2 r = sum_pair(p, m, 2 * j);
    const float v = r.x * (1.0f / (1.0f + expf(-r.x))) * r.y;
    act[idx] = (T)v;
}

// One 1024-thread workgroup per row: out[m] = resid[m] + product (f32, may
// alias resid), then xn[m] = (out[m] / rms) * gamma as binary16 with
// rms = sqrt(mean(out^2) + eps) (the arithmetic of rmsnorm_kernel).
template <int NV>
__global__ __launch_bounds__(1024) void epi_resnorm_kernel(GemmPartials p, const float *resid, float *out,
                                                           const float *__restrict__ gamma, float eps, _Float16 *xn,
                                                           uint32_t hidden) {
    __shared__ float red[16];
    const uint32_t m = blockIdx.x;
    const float *q = p.ws + (size_t)m * p.npad;
    const size_t stride = (size_t)p.mpad * p.npad;
    jf4 v[NV], g[NV];
    float s = 0.0f;
    // gamma is requested with the partials: one memory round trip before the reduction
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const uint32_t i = 4 * (threadIdx.x + 1024u * j);
        g[j] = i < hidden ? *(const jf4 *)(gamma + i) : jf4{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const uint32_t i = 4 * (threadIdx.x + 1024u * j);
        v[j] = jf4{0.0f, 0.0f, 0.0f, 0.0f};
        if (i < hidden) v[j] = sum_splits<jf4>(q + i, stride, p.ksplit) + *(const jf4 *)(resid + (size_t)m * hidden + i);
        s = fmaf(v[j].x, v[j].x, s);
        s = fmaf(v[j].y, v[j].y, s);
        s = fmaf(v[j].z, v[j].z, s);
        s = fmaf(v[j].w, v[j].w, s);
    }
    s = wave_sum_dpp(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; ++w) tot += red[w];
    // (x / rms) * gamma, the reference's formula (activations.wgsl:128), as in
    // the M = 1 kernels' fused norm
    const float rms = sqrtf(tot / (float)hidden + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const uint32_t i = 4 * (threadIdx.x + 1024u * j);
        if (i < hidden) {
            *(jf4 *)(out + (size_t)m * hidden + i) = v[j];
            const uint32_t lo = (uint32_t)f2h_bits((v[j].x / rms) * g[j].x) | ((uint32_t)f2h_bits((v[j].y / rms) * g[j].y) << 16);
            const uint32_t hi = (uint32_t)f2h_bits((v[j].z / rms) * g[j].z) | ((uint32_t)f2h_bits((v[j].w / rms) * g[j].w) << 16);
            *(uint2 *)((uint16_t *)xn + (size_t)m * hidden + i) = make_uint2(lo, hi);
        }
    }
}

// Residual + RMSNorm spread over the GPU in two launches (a row's sum of
// squares spans workgroups): epi_ressum_kernel, one 128-thread workgroup per
// (512-column slice, row), writes out = resid + the summed partials and the
// slice's sum of squares (threads, then the wavefront by DPP, then the two
// wavefronts in order) to p.ss[row][slice]; epi_norm_kernel, the same grid,
// adds the row's slice sums in slice order and writes (x / rms) * gamma as
// binary16 (activations.wgsl:128, as the M = 1 kernels' fused norm).
constexpr uint32_t kEpiCols = 512;
__global__ __launch_bounds__(128) void epi_ressum_kernel(GemmPartials p, const float *resid, float *out,
                                                         uint32_t hidden) {
    __shared__ float red[2];
    const uint32_t m = blockIdx.y, slice = blockIdx.x;
    const uint32_t i = slice * kEpiCols + 4 * threadIdx.x;
    const float *q = p.ws + (size_t)m * p.npad;
    jf4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i < hidden) {
        v = sum_splits<jf4>(q + i, (size_t)p.mpad * p.npad, p.ksplit) + *(const jf4 *)(resid + (size_t)m * hidden + i);
        *(jf4 *)(out + (size_t)m * hidden + i) = v;
    }
    float s = fmaf(v.x, v.x, 0.0f);
    s = fmaf(v.y, v.y, s);
    s = fmaf(v.z, v.z, s);
    s = fmaf(v.w, v.w, s);
    s = wave_sum_dpp(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) p.ss[(size_t)m * kEpiSlices + slice] = red[0] + red[1];
}

__global__ __launch_bounds__(128) void epi_norm_kernel(GemmPartials p, const float *out,
                                                       const float *__restrict__ gamma, float eps, _Float16 *xn,
                                                       uint32_t hidden) {
    const uint32_t m = blockIdx.y, slice = blockIdx.x;
    const uint32_t i = slice * kEpiCols + 4 * threadIdx.x;
    const uint32_t slices = (hidden + kEpiCols - 1) / kEpiCols;
    // the row and gamma are requested with the slice sums: one round trip
    jf4 v = {0.0f, 0.0f, 0.0f, 0.0f}, g = {0.0f, 0.0f, 0.0f, 0.0f};
    if (i < hidden) {
        v = *(const jf4 *)(out + (size_t)m * hidden + i);
        g = *(const jf4 *)(gamma + i);
    }
    float tot = 0.0f;
    for (uint32_t t = 0; t < slices; ++t) tot += p.ss[(size_t)m * kEpiSlices + t];
    const float rms = sqrtf(tot / (float)hidden + eps);
    if (i < hidden) {
        const uint32_t lo = (uint32_t)f2h_bits((v.x / rms) * g.x) | ((uint32_t)f2h_bits((v.y / rms) * g.y) << 16);
        const uint32_t hi = (uint32_t)f2h_bits((v.z / rms) * g.z) | ((uint32_t)f2h_bits((v.w / rms) * g.w) << 16);
        *(uint2 *)((uint16_t *)xn + (size_t)m * hidden + i) = make_uint2(lo, hi);
    }
}

int run_partials(janus_ctx *ctx, const void *a, int a_dt, const janus_weight *w, uint32_t rows, GemmPartials *parts) {
    if (!mfma_gemm_supported(JANUS_DT_F16, w))
        return fail(ctx, JANUS_E_UNSUPPORTED_DTYPE, "batched epilogue: weight has no MFMA path");
    if (rows == 0) return fail(ctx, JANUS_E_INVALID_DIM, "batched epilogue: no rows");
    if (int e = mfma_gemm_prepare(ctx, w)) return e;
    GemmArgs g = make_args(w, a_dt == JANUS_DT_F16 ? a : nullptr, nullptr, 0, rows, nullptr);
    if (a_dt == JANUS_DT_F16)
        return rows <= 32 ? launch_mt<1>(ctx, g, w, parts)
               : rows <= 64 ? launch_mt<2>(ctx, g, w, parts) : launch_wide_any(ctx, g, w, parts);
    if (w->t32_nonfinite) return fail(ctx, JANUS_E_UNSUPPORTED_DTYPE, "batched epilogue: weight has no exact parts");
    g.a32 = (const float *)a;
    if (rows > 64) return launch_wide_any(ctx, g, w, parts);
    bool ran = false;
    const int e = rows <= 32 ? launch_x32_mt<1>(ctx, g, w, parts, &ran) : launch_x32_mt<2>(ctx, g, w, parts, &ran);
    return e || ran ? e : fail(ctx, JANUS_E_OOM, "batched epilogue: workspace");
}

}  // namespace

bool mfma_gemm_supported(int a_dt, const janus_weight *w) {
    if (a_dt != JANUS_DT_F16 || w->k % 8) return false;
    return w->type == JANUS_DT_Q4_0 || w->type == JANUS_DT_Q8_0 || w->type == JANUS_DT_Q4_K ||
           w->type == JANUS_DT_Q5_K || w->type == JANUS_DT_F16;
}

int mfma_gemm_prepare(janus_ctx *ctx, const janus_weight *w) {
    return t32_ensure(ctx, const_cast<janus_weight *>(w));
}

void mfma_gemm_release(const janus_weight *cw) {
    janus_weight *w = const_cast<janus_weight *>(cw);
    if (w->t32) (void)hipFree(w->t32);
    w->t32 = nullptr;
    w->t32_qs = w->t32_side = nullptr;
    w->t32_q5h = nullptr;
    w->t32_chunks = 0;
}

int smallm_gemm_launch(janus_ctx *ctx, const void *a, int a_dt, const janus_weight *w, void *c, int c_dt,
                       uint32_t rows, const float *residual) {
    if (mfma_gemm_supported(a_dt, w)) {
        if (int e = mfma_gemm_prepare(ctx, w)) return e;
        const GemmArgs g = make_args(w, a, c, c_dt == JANUS_DT_F16, rows, residual);
        return rows <= 32 ? launch_mt<1>(ctx, g, w, nullptr) : launch_mt<2>(ctx, g, w, nullptr);
    }
    // f32 activations keep the reference's precision: three bfloat16 parts on
    // the MFMA kernel where the weight's tile copy can be had (built outside any
    // capture; a binary16 weight with an infinity or NaN has no exact parts),
    // else one GEMV launch per row
    if (a_dt == JANUS_DT_F32 && mfma_gemm_supported(JANUS_DT_F16, w) && x32_pays(w, rows)) {
        janus_weight *mw = const_cast<janus_weight *>(w);
        if (!w->t32 && !w->t32_nonfinite && !w->t32_denied && !capturing(ctx) && t32_ensure(ctx, mw, true)) {
            mw->t32_denied = true;
            (void)hipGetLastError();
            ctx->last_error.clear();
        }
        if (w->t32 && !w->t32_nonfinite) {
            GemmArgs g = make_args(w, nullptr, c, c_dt == JANUS_DT_F16, rows, residual);
            g.a32 = (const float *)a;
            bool ran = false;
            const int e = rows <= 32 ? launch_x32_mt<1>(ctx, g, w, nullptr, &ran)
                                     : launch_x32_mt<2>(ctx, g, w, nullptr, &ran);
            if (e || ran) return e;
        }
    }
    const size_t as = act_bytes(a_dt) * w->k, cs = act_bytes(c_dt) * w->n;
    for (uint32_t r = 0; r < rows; ++r) {
        int e = gemv_dispatch(ctx, (const uint8_t *)a + r * as, a_dt, w, (uint8_t *)c + r * cs, c_dt,
                              residual ? residual + (size_t)r * w->n : nullptr);
        if (e) return e;
    }
    return JANUS_OK;
}

int gemm_rows(janus_ctx *ctx, const void *a, int a_dt, const janus_weight *w, float *c, uint32_t rows,
              const float *residual) {
    if (rows <= 64) return gemm_dispatch(ctx, a, a_dt, w, c, JANUS_DT_F32, rows, residual);
    if (!mfma_rows_supported(a_dt, w)) return fail(ctx, JANUS_E_UNSUPPORTED_DTYPE, "gemm: weight has no MFMA path");
    if (int e = mfma_gemm_prepare(ctx, w)) return e;
    GemmArgs g = make_args(w, a_dt == JANUS_DT_F16 ? a : nullptr, c, 0, rows, residual);
    if (a_dt == JANUS_DT_F32) g.a32 = (const float *)a;
    return launch_wide_any(ctx, g, w, nullptr);
}

bool mfma_rows_supported(int a_dt, const janus_weight *w) {
    return mfma_gemm_supported(JANUS_DT_F16, w) && !(a_dt == JANUS_DT_F32 && w->t32_nonfinite);
}

int gemm_qkv_rope(janus_ctx *ctx, const void *a, int a_dt, const janus_weight *w, uint32_t rows, const QkvEpilogue &e,
                  int kv_f16) {
    if (w->n != 2 * (e.q_pairs + e.k_pairs) + e.kv_row || e.kv_row % 2)
        return fail(ctx, JANUS_E_INVALID_DIM, "qkv epilogue: row count does not match the head layout");
    GemmPartials p{};
    if (int r = run_partials(ctx, a, a_dt, w, rows, &p)) return r;
    const size_t total = (size_t)rows * (w->n / 2);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (kv_f16) hipLaunchKernelGGL(epi_qkv_rope_kernel<_Float16>, grid, dim3(256), 0, ctx->stream, p, e, rows);
    else hipLaunchKernelGGL(epi_qkv_rope_kernel<float>, grid, dim3(256), 0, ctx->stream, p, e, rows);
    JANUS_LAUNCH_CHECK(ctx);
    return JANUS_OK;
}

int gemm_swiglu(janus_ctx *ctx, const void *a, int a_dt, const janus_weight *w, uint32_t rows, void *act) {
    if (w->n % 2) return fail(ctx, JANUS_E_INVALID_DIM, "swiglu epilogue: odd row count");
    const uint32_t tiles = (w->n + 32 * WAVES - 1) / (32 * WAVES);
    const bool f16 = a_dt == JANUS_DT_F16;
    if (rows > 64 && mfma_rows_supported(a_dt, w)) {
        // K unsplit: SwiGLU is applied to the finished tile
        if (int e = mfma_gemm_prepare(ctx, w)) return e;
        GemmArgs g = make_args(w, f16 ? a : nullptr, act, f16, rows, nullptr);
        if (!f16) g.a32 = (const float *)a;
        g.swiglu = 1;
        return launch_wide_any(ctx, g, w, nullptr);
    }
    if (f16 && w->type == JANUS_DT_Q4_0 && rows <= 32 && 4 * tiles >= 3 * (uint32_t)ctx->num_cus) {
        // enough row tiles for every CU without splitting K: 16-wavefront
        // workgroups over the whole K, SwiGLU applied to the finished tile
        if (int e = mfma_gemm_prepare(ctx, w)) return e;
        GemmArgs g = make_args(w, a, act, 1, rows, nullptr);
        g.swiglu = 1;
        return launch_mfma<GQ4_0, 1, 4, 2>(ctx, g, w, nullptr, ctx->gemm_pipe ? 512 : 1024, 1);
    }
    GemmPartials p{};
    if (int r = run_partials(ctx, a, a_dt, w, rows, &p)) return r;
    const size_t total = (size_t)rows * (w->n / 2);
    const dim3 grid((unsigned)((total + 255) / 256));
    if (f16) hipLaunchKernelGGL(epi_swiglu_kernel<_Float16>, grid, dim3(256), 0, ctx->stream, p, (_Float16 *)act, rows, w->n / 2);
    else hipLaunchKernelGGL(epi_swiglu_kernel<float>, grid, dim3(256), 0, ctx->stream, p, (float *)act, rows, w->n / 2);
    JANUS_LAUNCH_CHECK(ctx);
    return JANUS_OK;
}

bool resnorm_supported(uint32_t hidden) { return hidden % 4 == 0 && hidden <= 8192; }

int gemm_residual_norm(janus_ctx *ctx, const void *a16, const janus_weight *w, uint32_t rows, const float *resid,
                       float *out, const float *gamma, float eps, void *xn16) {
    const uint32_t hidden = w->n;
    if (!resnorm_supported(hidden))
        return fail(ctx, JANUS_E_INVALID_DIM, "residual-norm epilogue: rows must be a multiple of 4, at most 8192");
    GemmPartials p{};
    if (rows > 64) return fail(ctx, JANUS_E_INVALID_DIM, "residual-norm epilogue: at most 64 rows");
    if (int r = run_partials(ctx, a16, JANUS_DT_F16, w, rows, &p)) return r;
    _Float16 *xn = (_Float16 *)xn16;
    if (ctx->epi_split) {
        const dim3 sgrid((hidden + kEpiCols - 1) / kEpiCols, rows), sblock(kEpiCols / 4);
        hipLaunchKernelGGL(epi_ressum_kernel, sgrid, sblock, 0, ctx->stream, p, resid, out, hidden);
        JANUS_LAUNCH_CHECK(ctx);
        hipLaunchKernelGGL(epi_norm_kernel, sgrid, sblock, 0, ctx->stream, p, out, gamma, eps, xn, hidden);
        JANUS_LAUNCH_CHECK(ctx);
        return JANUS_OK;
    }
    const dim3 grid(rows), block(1024);
    if (hidden <= 4096) hipLaunchKernelGGL(epi_resnorm_kernel<1>, grid, block, 0, ctx->stream, p, resid, out, gamma, eps, xn, hidden);
    else hipLaunchKernelGGL(epi_resnorm_kernel<2>, grid, block, 0, ctx->stream, p, resid, out, gamma, eps, xn, hidden);
    JANUS_LAUNCH_CHECK(ctx);
    return JANUS_OK;
}

}  // namespace janus
