// prefill.hip -- causal attention of a prompt chunk.
//
// The rows of a chunk are consecutive positions p0 .. p0 + n - 1 of one
// sequence whose K/V rows 0 .. p0 + n - 1 are in the cache; row i attends
// positions 0 .. p0 + i (shaders/attention.wgsl:62-186 for each row). The
// decode kernels would read the whole prefix once per row; here a wavefront
// holds 32 query rows of one head, and K and V tiles of 32 positions pass
// through LDS once for the four wavefronts of a workgroup: four heads of a KV
// head where it has that many, else two heads x two row tiles or four row tiles.
//
// Scores are S^T = K Q^T (positions x queries), so a lane's column is one
// query and the running maximum and sum, the rescale and the output scale
// are per lane; the probabilities are P.V's B operand as they lie, with the
// position order of V's operand chosen to match.
//  * binary16 caches: v_mfma_f32_32x32x16_f16. q is split into binary16
//    hi + mid + lo parts after a power-of-two prescale of its largest element
//    to 2^14 .. 2^15 (33 bits of that element, a fixed 2^-39 of it for the
//    others), P into three parts of 2^14 p (every bit down to 2^-38); V is
//    transposed on its way into LDS.
//  * binary32 caches: v_mfma_f32_32x32x2_f32 (a chain of two FMAs), nothing
//    split or rounded.
// Sums run as short chains joined as equals (four dims of a score, eight
// positions of P.V; four tiles of output before they join the running one), a
// score is scaled after the maximum is taken off and l is a double: against 64
// bits the output is as close as the decode kernels' (rms 0.8 to 1.02 of their
// error over up to 512 positions; with one chain per score and output, two parts
// of P and q scaled down only, it was 1.1 to 2.2, and 120 where q was small).
//
// Bound by the longest row tile's chain of K/V tiles (a 512-row chunk is 128
// workgroups of four heads, so CUs are idle). Per call, back to back: 50 us for
// 512 binary16 rows at 32/8/128 heads against 160 through the decode kernels,
// 38 us for 133 binary32 rows at 32/32/128 (38 and 33 with the longer chains).
// Built with MFMA results in vector registers: the compiler's choice for
// wavefronts of 512 registers, accumulation registers, takes a move per add
// (45 us for the binary32 rows).
#include <type_traits>

#include "internal.h"

namespace janus {
namespace {

typedef _Float16 ph8 __attribute__((ext_vector_type(8)));
typedef float pf16 __attribute__((ext_vector_type(16)));

constexpr int QT = 32, PT = 32;   // queries per wavefront, positions per tile

struct PrefillArgs {
    const float *q;        // [n][heads][D]
    const void *kc, *vc;   // the sequence's cache rows of one layer: [pos][kv_heads][D]
    void *out;             // [n][heads][D], f32 or binary16
    uint32_t n, p0, heads, kv_heads;
    float scale2;          // scale * log2(e)
    int out_f16;
};

__device__ __forceinline__ float swap32(float v) {   // value of lane ^ 32
    const uint32_t u = __float_as_uint(v);
    auto p = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return __uint_as_float((__lane_id() & 32) ? p[0] : p[1]);
}

// LDS of one K/V tile. binary16: K rows padded to D + 8 halves; V transposed,
// [dim][position] rows padded to PT + 4 halves (8-byte reads of 4 positions).
// binary32: K rows padded to D + 4 floats, V rows as they are. Behind them one
// word per wavefront: whether it stored an infinity or NaN of V (bit 0) and of
// K (bit 1).
template <typename KV, int D> struct Tile;
template <int D> struct Tile<_Float16, D> {
    static constexpr int KP = D + 8, VP = PT + 4;
    static constexpr uint32_t K = PT * KP * 2, FLAGS = K + D * VP * 2, BYTES = FLAGS + 16;
    static constexpr int SEG = 8;   // elements of a 16-byte segment
};
template <int D> struct Tile<float, D> {
    static constexpr int KP = D + 4, VP = D;
    static constexpr uint32_t K = PT * KP * 4, FLAGS = K + PT * VP * 4, BYTES = FLAGS + 16;
    static constexpr int SEG = 4;
};

// Whether the 16 bytes hold an infinity or NaN.
template <typename KV> __device__ __forceinline__ bool nonfinite(const ju4 &v) {
    uint32_t b = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        // adding one to an exponent of all ones carries into the sign's place
        b |= std::is_same<KV, _Float16>::value ? (v[i] & 0x7c007c00u) + 0x04000400u : (v[i] & 0x7f800000u) + 0x00800000u;
    return (b & (std::is_same<KV, _Float16>::value ? 0x80008000u : 0x80000000u)) != 0;
}

// The finite values of the 16 bytes, others as 0.
template <typename KV> __device__ __forceinline__ ju4 finite_only(ju4 v) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (std::is_same<KV, _Float16>::value) {
            if ((v[i] & 0x7c00u) == 0x7c00u) v[i] &= 0xffff0000u;
            if ((v[i] & 0x7c000000u) == 0x7c000000u) v[i] &= 0xffffu;
        } else if ((v[i] & 0x7f800000u) == 0x7f800000u) {
            v[i] = 0u;
        }
    }
    return v;
}

// o[d] += p * V over the infinities and NaN of a tile of V (rows of kvrow
// elements from `v` on, `rows` of them in the cache; LDS has zeros in their
// place): position j of the tile for the queries that see it (j < seen), so
// they reach the dims that hold them and no other row or dim. s: probabilities
// of the lane's positions. A tile that holds none does not come here.
template <typename KV, int D>
__device__ __forceinline__ void add_nonfinite(const KV *v, uint32_t kvrow, uint32_t rows, const pf16 &s, uint32_t seen,
                                              int h, pf16 (&o)[D / 32]) {
#pragma unroll 1
    for (uint32_t j = 0; j < PT; ++j) {
        const int at = (int)(j >> 3) * 4 + (int)(j & 3);   // position j is s[at] of half (j / 4) % 2
        float mine = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) mine = i == at ? s[i] : mine;
        const float other = swap32(mine), p = (int)((j >> 2) & 1) == h ? mine : other;
        const KV *row = v + (size_t)min(j, rows - 1) * kvrow;
#pragma unroll
        for (int d = 0; d < D / 32; ++d)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float x = (float)row[32 * d + 8 * (i >> 2) + 4 * h + (i & 3)];
                if (j < seen && (__float_as_uint(x) & 0x7f800000u) == 0x7f800000u) o[d][i] = fmaf(p, x, o[d][i]);
            }
    }
}

// The scores of a tile with q in one piece: s[v] = qs * (q . K row of the
// lane's position v), 8 (v / 4) + 4 h + v % 4.
template <int D>
__device__ __forceinline__ void whole_scores(const unsigned char *kt, const float *q, float qs, int h, pf16 &s) {
    s = (pf16){};
#pragma unroll 1
    for (int d = 0; d < D; ++d) {
        const float x = q[d];
#pragma unroll
        for (int v = 0; v < 16; ++v)
            s[v] = fmaf(x, (float)((const _Float16 *)kt)[(8 * (v >> 2) + 4 * h + (v & 3)) * Tile<_Float16, D>::KP + d], s[v]);
    }
#pragma unroll
    for (int v = 0; v < 16; ++v) s[v] *= qs;
}

// HW: heads of a KV head that a workgroup's wavefronts take (1, 2 or 4); the
// other factor of 4 is row tiles. A chunk seldom has more workgroups than there
// are CUs (4 per query head at most), so a wavefront may take a SIMD's registers.
template <typename KV, int D, int HW>
__global__ __launch_bounds__(256, 1) void prefill_attn_kernel(PrefillArgs a) {
    constexpr bool F16 = std::is_same<KV, _Float16>::value;
    typedef Tile<KV, D> T;
    constexpr int SEG = T::SEG, SROW = D / SEG;       // 16-byte segments per row
    constexpr int LD = PT * SROW / 256;               // K (and V) segments per thread
    static_assert(LD >= 1 && LD * 256 == PT * SROW, "tile load");
    constexpr int ND = D / 32;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, h = lane >> 5;
    const uint32_t G = a.heads / a.kv_heads;
    const uint32_t parts = G / HW, kvh = blockIdx.y / parts;
    const uint32_t head = kvh * G + (blockIdx.y % parts) * HW + wave % HW;
    // row tiles from the last (longest) to the first
    const uint32_t groups = gridDim.x, grp = groups - 1 - blockIdx.x;
    constexpr uint32_t TW = 4 / HW;   // row tiles per workgroup
    const uint32_t q0 = (grp * TW + wave / HW) * QT;   // may lie beyond n: such a wavefront only helps to load
    const uint32_t last_row = min(a.n, (grp + 1) * TW * QT) - 1;
    const uint32_t end_all = a.p0 + last_row + 1;      // positions the workgroup passes over
    const uint32_t kvrow = a.kv_heads * D;
    const KV *kc = (const KV *)a.kc + (size_t)kvh * D, *vc = (const KV *)a.vc + (size_t)kvh * D;

    ju4 kr[LD], vr[LD];
    // segment j of this thread: binary16 V goes to LDS transposed in pairs of
    // positions, so a thread takes two rows of the same dims
    auto row_of = [&](int j, bool v) -> uint32_t {
        const uint32_t s = threadIdx.x + 256u * j;
        if (F16 && v) return LD >= 2 ? (threadIdx.x / SROW) * 2 + j : threadIdx.x / SROW;
        return s / SROW;
    };
    auto seg_of = [&](int j, bool v) -> uint32_t {
        const uint32_t s = threadIdx.x + 256u * j;
        if (F16 && v) return threadIdx.x % SROW;
        return s % SROW;
    };
    auto load = [&](uint32_t p) {
#pragma unroll
        for (int j = 0; j < LD; ++j) {
            const uint32_t kp = min(p + row_of(j, false), end_all - 1), vp = min(p + row_of(j, true), end_all - 1);
            kr[j] = *(const ju4 *)(kc + (size_t)kp * kvrow + seg_of(j, false) * SEG);
            vr[j] = *(const ju4 *)(vc + (size_t)vp * kvrow + seg_of(j, true) * SEG);
        }
    };
    auto store = [&](unsigned char *t) {
        bool oddv = false, oddk = false;
#pragma unroll
        for (int j = 0; j < LD; ++j) {
            oddv = oddv || nonfinite<KV>(vr[j]);
            if (F16) oddk = oddk || nonfinite<KV>(kr[j]);
        }
        const uint32_t any = (uint32_t)(__any(oddv) != 0) | (uint32_t)(__any(oddk) != 0) << 1;
        if (lane == 0) *(uint32_t *)(t + T::FLAGS + 4 * wave) = any;
        // A probability of 0 does not mask an infinity or NaN of V, and one
        // split into parts turns an infinity into a NaN: such values stay out of
        // the MFMAs and are added on their own (the look at a tile takes about
        // a dozen instructions per 16 bytes).
        if (any & 1u)
#pragma unroll
            for (int j = 0; j < LD; ++j) vr[j] = finite_only<KV>(vr[j]);
#pragma unroll
        for (int j = 0; j < LD; ++j)
            *(ju4 *)(t + ((size_t)row_of(j, false) * T::KP + seg_of(j, false) * SEG) * sizeof(KV)) = kr[j];
        if constexpr (!F16) {
#pragma unroll
            for (int j = 0; j < LD; ++j)
                *(ju4 *)(t + T::K + ((size_t)row_of(j, true) * T::VP + seg_of(j, true) * SEG) * 4) = vr[j];
        } else if constexpr (LD == 2) {
            // rows r, r + 1 of dims 8 s .. 8 s + 7: one word per dim
            uint32_t *vt = (uint32_t *)(t + T::K);
            const ju4 a0 = vr[0], a1 = vr[LD - 1];
            const uint32_t d0 = seg_of(0, true) * 8, r2 = row_of(0, true) / 2;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vt[(d0 + 2 * i) * (T::VP / 2) + r2] = __builtin_amdgcn_perm(a1[i], a0[i], 0x05040100u);
                vt[(d0 + 2 * i + 1) * (T::VP / 2) + r2] = __builtin_amdgcn_perm(a1[i], a0[i], 0x07060302u);
            }
        } else {   // D = 64: one row per thread
            uint16_t *vt = (uint16_t *)(t + T::K);
            const ju4 a0 = vr[0];
            const uint32_t d0 = seg_of(0, true) * 8, r = row_of(0, true);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                vt[(d0 + 2 * i) * T::VP + r] = (uint16_t)(a0[i] & 0xffffu);
                vt[(d0 + 2 * i + 1) * T::VP + r] = (uint16_t)(a0[i] >> 16);
            }
        }
    };
    load(0);

    // q of this lane's query: binary16 caches: dims 16 s + 8 h + 0..7 of each
    // 16-wide step as three parts; binary32: dims 8 s + 4 h + 0..3
    const uint32_t qi = min(q0 + col, a.n - 1);
    const float *qp = a.q + ((size_t)qi * a.heads + head) * D;
    float sc2 = a.scale2, qs = 1.0f;   // q's parts are those of q * qs
    bool q_inf = false;
    ph8 qh[F16 ? D / 16 : 1], qm[F16 ? D / 16 : 1], ql[F16 ? D / 16 : 1];
    jf4 qf[F16 ? 1 : D / 8];
    if constexpr (F16) {
        float qmax = 0.0f;
#pragma unroll
        for (int s = 0; s < D / 16; ++s) {
            const jf4 x0 = *(const jf4 *)(qp + 16 * s + 8 * h), x1 = *(const jf4 *)(qp + 16 * s + 8 * h + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) qmax = fmaxf(qmax, fmaxf(fabsf(x0[i]), fabsf(x1[i])));
        }
        qmax = fmaxf(qmax, swap32(qmax));
        int qe = 0;
        (void)frexpf(qmax, &qe);                  // qmax < 2^qe
        const int sh = max(qe - 15, -100);        // 2^14 <= |qmax| 2^-sh < 2^15 (below 2^-85 no score counts)
        qs = ldexpf(1.0f, -sh);
        q_inf = __any(qmax == INFINITY);
        sc2 *= ldexpf(1.0f, sh);
        asm volatile("" : "+v"(qp));   // q is read again (from cache) rather than held beside its parts
#pragma unroll
        for (int s = 0; s < D / 16; ++s) {
            const jf4 x0 = *(const jf4 *)(qp + 16 * s + 8 * h), x1 = *(const jf4 *)(qp + 16 * s + 8 * h + 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float x = (i < 4 ? x0[i & 3] : x1[i & 3]) * qs;
                const _Float16 hi = (_Float16)x;
                const float r = x - (float)hi;
                const _Float16 mid = (_Float16)r;
                qh[s][i] = hi;
                qm[s][i] = mid;
                ql[s][i] = (_Float16)(r - (float)mid);
            }
        }
    } else {
#pragma unroll
        for (int s = 0; s < D / 8; ++s) qf[s] = *(const jf4 *)(qp + 8 * s + 4 * h);
    }

    // O^T: dims 32 d + 8 j + 4 h + i of query col (binary16 caches: times 2^14).
    // o4 is the sum over the last tiles (up to four), which then joins o.
    pf16 o[ND], o4[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = o4[d] = (pf16){};
    float m = -INFINITY;
    double l = 0.0;
    bool lost = false;
    const uint32_t my_end = a.p0 + q0 + col + 1;                         // this lane's query sees [0, my_end)
    const uint32_t wave_end = q0 < a.n ? a.p0 + min(q0 + QT, a.n) : 0;   // uniform

    store(smem);
    uint32_t buf = 0;
    for (uint32_t p = 0; p < end_all; p += PT) {
        load(min(p + PT, end_all - 1));   // the last tile's request repeats a row and is not used
        __syncthreads();
        const unsigned char *kt = smem + buf * T::BYTES, *vt = kt + T::K;
        if (p < wave_end) {
            const uint4 f = *(const uint4 *)(kt + T::FLAGS);
            const uint32_t flags = __builtin_amdgcn_readfirstlane(f.x | f.y | f.z | f.w);
            // Short chains, then sums of equals: a chain over all dims would round
            // every term at the size of the whole score.
            pf16 s = (pf16){}, s2 = (pf16){};
            if constexpr (F16) {
                pf16 sm = (pf16){};   // the small parts
#pragma unroll
                for (int t = 0; t < D / 16; ++t) {
                    const ph8 k = *(const ph8 *)(kt + ((size_t)col * T::KP + 16 * t + 8 * h) * 2);
                    sm = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, ql[t], sm, 0, 0, 0);
                    if (t & 1) s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qh[t], s2, 0, 0, 0);
                    else s = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qh[t], s, 0, 0, 0);
                    sm = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qm[t], sm, 0, 0, 0);
                }
#pragma unroll
                for (int v = 0; v < 16; ++v) s2[v] += sm[v];
            } else {
#pragma unroll
                for (int t = 0; t < D / 8; t += 2) {   // 16 dims as a tree over chains of four
                    pf16 c[4];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const jf4 k = *(const jf4 *)(kt + ((size_t)col * T::KP + 8 * (t + u) + 4 * h) * 4);
                        c[2 * u] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[0], qf[t + u][0], (pf16){}, 0, 0, 0);
                        c[2 * u + 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[2], qf[t + u][2], (pf16){}, 0, 0, 0);
                        c[2 * u] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[1], qf[t + u][1], c[2 * u], 0, 0, 0);
                        c[2 * u + 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(k[3], qf[t + u][3], c[2 * u + 1], 0, 0, 0);
                    }
                    pf16 &to = t & 2 ? s2 : s;
#pragma unroll
                    for (int v = 0; v < 16; ++v) to[v] += (c[0][v] + c[1][v]) + (c[2][v] + c[3][v]);
                }
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] += s2[v];
            // An infinity times a part of q that is 0 or of the other sign would
            // make a NaN of an infinite score: such tiles take q whole.
            if (F16 && (q_inf || (flags & 2u))) whole_scores<D>(kt, qp, qs, h, s);
            // s[4 j + i]: position p + 8 j + 4 h + i
            float bm = -INFINITY;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const bool live = p + 8 * (v >> 2) + 4 * h + (v & 3) < my_end;
                s[v] = live ? s[v] : -INFINITY;
                bm = fmaxf(bm, s[v]);
            }
            bm = fmaxf(bm, swap32(bm));
            // m is in the scores' unit: their differences are exact near the
            // maximum and are scaled after
            const float mn = fmaxf(m, bm);
            const float alpha = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f((m - mn) * sc2);
            // the maxima pass over a NaN: while there is no other score, it is kept here
            if (__any(mn == -INFINITY) && mn == -INFINITY)
#pragma unroll
                for (int v = 0; v < 16; ++v) lost = lost || s[v] != s[v];
#pragma unroll
            for (int v = 0; v < 16; ++v) s[v] = mn == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((s[v] - mn) * sc2);
            float sum[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) sum[v] = (s[4 * v] + s[4 * v + 1]) + (s[4 * v + 2] + s[4 * v + 3]);
            l = fma(l, (double)alpha, (double)((sum[0] + sum[1]) + (sum[2] + sum[3])));
            m = mn;
            if (__any(alpha != 1.0f))   // after the first tiles the maximum rarely moves
#pragma unroll
                for (int d = 0; d < ND; ++d)
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        o[d][v] *= alpha;
                        o4[d][v] *= alpha;
                    }
            // the tile's sums are made on their own and then added to o4
            if constexpr (F16) {
                // 16 positions per step: half h holds 4 h + 0..3 and 8 + 4 h + 0..3 of them
                ph8 pp[2][3];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float x = s[8 * t + e] * 16384.0f;
                        const _Float16 hi = (_Float16)x;
                        const float r = x - (float)hi;
                        const _Float16 mid = (_Float16)r;
                        pp[t][0][e] = hi;
                        pp[t][1][e] = mid;
                        pp[t][2][e] = (_Float16)(r - (float)mid);
                    }
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    ph8 v[2];
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        const unsigned char *vp = vt + ((size_t)(32 * d + col) * T::VP + 16 * t + 4 * h) * 2;
                        const uint2 v0 = *(const uint2 *)vp, v1 = *(const uint2 *)(vp + 16);
                        v[t] = __builtin_bit_cast(ph8, make_uint4(v0.x, v0.y, v1.x, v1.y));
                    }
                    pf16 c = (pf16){};
#pragma unroll
                    for (int i = 2; i >= 0; --i) {
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[0], pp[0][i], c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x16_f16(v[1], pp[1][i], c, 0, 0, 0);
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) o4[d][i] += c[i];
                }
            } else {
                // step v: positions 8 (v / 4) + v % 4 (half 0) and that plus 4 (half 1)
#pragma unroll
                for (int d = 0; d < ND; ++d) {
                    pf16 c[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        c[j] = (pf16){};
#pragma unroll
                        for (int v = 4 * j; v < 4 * j + 4; ++v) {
                            const float x = *(const float *)(vt + ((size_t)(8 * j + 4 * h + (v & 3)) * T::VP + 32 * d + col) * 4);
                            c[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, s[v], c[j], 0, 0, 0);
                        }
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) o4[d][i] += (c[0][i] + c[1][i]) + (c[2][i] + c[3][i]);
                }
            }
            if (flags & 1u) add_nonfinite<KV, D>(vc + (size_t)p * kvrow, kvrow, end_all - p, s, my_end - min(my_end, p), h, o4);
            if ((p / PT) % 4 == 3 || p + PT >= wave_end)
#pragma unroll
                for (int d = 0; d < ND; ++d) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) o[d][v] += o4[d][v];
                    o4[d] = (pf16){};
                }
        }
        buf ^= 1u;
        store(smem + buf * T::BYTES);   // last read before the barrier above
    }
    if (q0 + col >= a.n) return;
    // a row whose scores are all NaN stays 0, as in the decode kernels
    const float other = swap32(lost ? 1.0f : 0.0f);
    if ((lost || other != 0.0f) && m != -INFINITY) l = NAN;
    float lt = (float)l + swap32((float)l);
    lt = lt < 1e-20f ? 1e-20f : lt;   // a NaN stays
    const float inv = 1.0f / lt;
    auto divide = [&](float x) {   // x / lt: the remainder corrects the last bit
        if (F16) x *= 1.0f / 16384.0f;
        const float r = x * inv, rest = fmaf(-r, lt, x);
        return rest == rest ? fmaf(rest, inv, r) : r;
    };
    const size_t at = ((size_t)(q0 + col) * a.heads + head) * D + 4 * h;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float x0 = divide(o[d][4 * j]), x1 = divide(o[d][4 * j + 1]), x2 = divide(o[d][4 * j + 2]),
                        x3 = divide(o[d][4 * j + 3]);
            const size_t i = at + 32 * d + 8 * j;
            if (a.out_f16)
                *(uint2 *)((uint16_t *)a.out + i) = make_uint2((uint32_t)f2h_bits(x0) | ((uint32_t)f2h_bits(x1) << 16),
                                                               (uint32_t)f2h_bits(x2) | ((uint32_t)f2h_bits(x3) << 16));
            else *(jf4 *)((float *)a.out + i) = jf4{x0, x1, x2, x3};
        }
}

template <typename KV, int D, int HW>
void launch(janus_ctx *ctx, const PrefillArgs &a) {
    static const bool attr_set = [] {   // thread-safe one-time set-up
        (void)hipFuncSetAttribute((const void *)prefill_attn_kernel<KV, D, HW>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        return true;
    }();
    (void)attr_set;
    const uint32_t rows = 4 / HW * QT, G = a.heads / a.kv_heads;
    const dim3 grid((a.n + rows - 1) / rows, a.kv_heads * (G / HW));
    constexpr size_t lds = 2 * Tile<KV, D>::BYTES;
    hipLaunchKernelGGL((prefill_attn_kernel<KV, D, HW>), grid, dim3(256), lds, ctx->stream, a);
}

template <typename KV, int D>
void launch_heads(janus_ctx *ctx, const PrefillArgs &a) {
    const uint32_t G = a.heads / a.kv_heads;
    if (G % 4 == 0) launch<KV, D, 4>(ctx, a);
    else if (G % 2 == 0) launch<KV, D, 2>(ctx, a);
    else launch<KV, D, 1>(ctx, a);
}

}  // namespace

bool prefill_attention_supported(uint32_t hd) { return hd == 64 || hd == 128; }

int prefill_attention_launch(janus_ctx *ctx, const float *q, const void *kc, const void *vc, int kv_dt, void *out,
                             uint32_t n, uint32_t p0, uint32_t heads, uint32_t kv_heads, uint32_t hd, float scale,
                             int out_f16) {
    if (!prefill_attention_supported(hd)) return fail(ctx, JANUS_E_INVALID_DIM, "attention: head_dim must be 64 or 128");
    if (n == 0) return JANUS_OK;
    const PrefillArgs a{q, kc, vc, out, n, p0, heads, kv_heads, scale * 1.4426950408889634f, out_f16};
    if (kv_dt == JANUS_DT_F16) {
        if (hd == 64) launch_heads<_Float16, 64>(ctx, a);
        else launch_heads<_Float16, 128>(ctx, a);
    } else {
        if (hd == 64) launch_heads<float, 64>(ctx, a);
        else launch_heads<float, 128>(ctx, a);
    }
    JANUS_LAUNCH_CHECK(ctx);
    return JANUS_OK;
}

}  // namespace janus
