// prefill_attention.hip -- causal attention of several query tokens per
// sequence over the FP16 or the TurboQuant cache (fused_sdpa.metal:52-251 and
// turboquant.metal:202-462 with token_count > 1).
//
// A query row is a (token, head of the kv head's group) pair; a workgroup
// takes 32 rows per wave of one kv head, so each cache row is staged (and, for
// TurboQuant, looked up) once for all of them, where the decode kernels
// scan the cache once per token (FP16: per 4 rows) or per 16 rows.
//
// What bounds it: the matrix cores (v_mfma_f32_32x32x16_f16) with the vector
// softmax beside them at two waves per SIMD.  Both products are computed
// transposed -- S^T = K Q^T, O^T = V^T P^T -- so a query row is one column of
// every result, i.e. one lane pair (l, l + 32): the row maximum, sum and
// rescale are per lane (one exchange between the pair), and the weights leave
// the first product in exactly the registers that the second one reads (the
// contraction takes the positions in the order the result has them; V is
// staged in that order).  Nothing goes through LDS between the products.
//  * K rows are staged as they are ([position][dim], padded rows), V
//    transposed ([dim][position]) from four rows per thread.
//  * FP16: q, k, v are exact f16; the weights (scaled by 2^10, so that small
//    ones stay normal) enter as f16 hi + lo (~22 bits).
//  * TurboQuant: q and its QJL projection as f16 hi + lo planes, codebook
//    entries as hi + lo from bank-spread tables, the QJL signs as +-1: five
//    products per score (s_hi sgn + s_lo sgn first, scaled by the position's
//    residual norm in f32, then q_hi K_hi + q_hi K_lo + q_lo K_hi onto it), and
//    f16 weights (times the V scale) against V's hi and lo.
//
// Measured (us, write + attention, before -> after): FP16, two sequences of up
// to 2500 positions, T = 301, 16 / 8 heads 242 -> 46; one of 8192, T = 512, 32
// / 8 heads 1354 -> 126; TurboQuant at the latter sizes 403 -> 264.  The
// TurboQuant kernel keeps the matrix cores busy 53 % of the time: its score
// sums are one chain of 40 dependent products per 32 positions, and the
// registers (128 for the query planes, 64 for the result) leave no room for a
// second chain.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>

#include "hadamard.h"
#include "imh_internal.h"
#include "prefill_attention.h"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kD = 128;
constexpr int kKRow = 272;           // LDS bytes of a K row (16-byte pad)
constexpr int kTabBytes = 256 * 256; // bank-spread codebooks: row c = 32 copies of K entry c, 32 of V entry c
constexpr uint32_t kRsrcWord3 = 0x00020000u;

__device__ __forceinline__ uint32_t tab_entry(float v) {
    const _Float16 hi = (_Float16)v;
    const _Float16 lo = (_Float16)(v - (float)hi);
    return (uint32_t)__builtin_bit_cast(uint16_t, hi) | ((uint32_t)__builtin_bit_cast(uint16_t, lo) << 16);
}
// entry of code byte k of w; lane_off: 4 (l & 31), + 128 for V
__device__ __forceinline__ uint32_t tab_read(const uint8_t *tabs, uint32_t w, int k, uint32_t lane_off) {
    const uint32_t off = __builtin_amdgcn_perm(w, lane_off, 0x0C0C0000u | ((4u + (uint32_t)k) << 8));
    return *reinterpret_cast<const uint32_t *>(tabs + off);
}

// One row of the FP16 kernel by a wave, in f32 over the row's own positions
// [p_begin, lim) only (lane = position for the scores, two dims for the values):
// what a row is given whose matrix-core result is not finite.  There a weight of
// 0 (a position that the row does not see, or the low half of a weight) times an
// infinite value of another row's position is NaN.  Bound by the latency of its
// loads, which is why they are issued in batches: with an infinite value in
// position 0, so that every row comes here, T = 512 over 8192 positions at 32 / 8
// heads takes 5.6 ms (one load at a time 14.8; the kernel of few rows, for all, 1.5).
__device__ __forceinline__ void exact_row(const imh::PrefillAttention &a, size_t head_base, size_t qrow,
                                          int p_begin, int lim, int S, int split) {
    const int lane = threadIdx.x & 63;
    const _Float16 *q = a.q + qrow * kD;
    const _Float16 *k = reinterpret_cast<const _Float16 *>(a.k) + head_base * kD;
    const _Float16 *v = reinterpret_cast<const _Float16 *>(a.v) + head_base * kD;
    const float sl2 = a.attn_scale * 1.44269504f;
    float m = -INFINITY, l = 0.0f, o0 = 0.0f, o1 = 0.0f;
    for (int p0 = p_begin; p0 < lim; p0 += 64) {
        float s = -INFINITY;
        if (p0 + lane < lim) {
            s = 0.0f;
#pragma unroll 8
            for (int d = 0; d < kD; d += 8) {
                const half8_t kv = *reinterpret_cast<const half8_t *>(k + (size_t)(p0 + lane) * kD + d);
                for (int e = 0; e < 8; e++) s = __builtin_fmaf((float)q[d + e], (float)kv[e], s);
            }
            s *= sl2;
        }
        float nm = s;
        for (int st = 32; st >= 1; st >>= 1) nm = fmaxf(nm, __shfl_xor(nm, st));
        nm = fmaxf(nm, m);
        // scores that are all -inf weigh 0, scores that are no numbers stay so
        const float corr = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - nm);
        const float w = __builtin_amdgcn_exp2f(s - (nm == -INFINITY ? 0.0f : nm));
        m = nm;
        l = __builtin_fmaf(l, corr, w);
        o0 *= corr;
        o1 *= corr;
        const int n = min(64, lim - p0);
        auto add = [&](int j, half2_t vv) __attribute__((always_inline)) {
            const float wj = __shfl(w, j);
            o0 = __builtin_fmaf(wj, (float)vv[0], o0);
            o1 = __builtin_fmaf(wj, (float)vv[1], o1);
        };
        const half2_t *vp = reinterpret_cast<const half2_t *>(v + (size_t)p0 * kD) + lane;
        int j = 0;
        for (; j + 16 <= n; j += 16) {   // sixteen loads in flight
            half2_t vv[16];
#pragma unroll
            for (int i = 0; i < 16; i++) vv[i] = vp[(size_t)(j + i) * (kD / 2)];
#pragma unroll
            for (int i = 0; i < 16; i++) add(j + i, vv[i]);
        }
        for (; j < n; j++) add(j, vp[(size_t)j * (kD / 2)]);
    }
    for (int st = 32; st >= 1; st >>= 1) l += __shfl_xor(l, st);
    if (m == -INFINITY) {   // no position, or no score that is a number
        if (l == 0.0f) o0 = o1 = 0.0f;
        else m = 0.0f;
    }
    if (S > 1) {
        const size_t pi = qrow * S + split;
        a.part_o[pi * kD + 2 * lane] = o0;
        a.part_o[pi * kD + 2 * lane + 1] = o1;
        if (lane == 0) {
            a.part_m[pi] = m;
            a.part_l[pi] = l;
        }
    } else {
        const float inv = 1.0f / fmaxf(l, 1e-10f);
        a.out[qrow * kD + 2 * lane] = __float2half(o0 * inv);
        a.out[qrow * kD + 2 * lane + 1] = __float2half(o1 * inv);
    }
}

// grid (splits, kv heads, batch x row tiles), block 256 (TurboQuant 512).
template <bool TQ>
__global__ void __launch_bounds__(TQ ? 512 : 256) __attribute__((amdgpu_waves_per_eu(2, 2))) prefill_attention_kernel(
    const imh::PrefillAttention a) {
    constexpr int WAVES = TQ ? 8 : 4;
    constexpr int kTile = TQ ? 32 : 64;  // positions staged at a time, and per softmax step
    constexpr int NB = kTile / 32;
    constexpr int NK = TQ ? 3 : 1;       // K arrays: rows, or codebook hi, lo and signs
    constexpr int NV = TQ ? 2 : 1;       // V arrays
    constexpr int NP = TQ ? 4 : 1;       // query planes
    constexpr int kVRow = kTile * 2 + 16;   // LDS bytes of a V^T row
    constexpr int kKBytes = kTile * kKRow;
    constexpr int kVBytes = kD * kVRow;
    __shared__ __attribute__((aligned(16))) uint8_t Ks[2][NK][kKBytes];
    __shared__ __attribute__((aligned(16))) uint8_t Vs[2][NV][kVBytes];
    __shared__ __attribute__((aligned(16))) float scl[TQ ? 2 : 1][3][kTile];   // K scale, residual norm, V scale
    __shared__ __attribute__((aligned(16))) uint8_t tabs[TQ ? kTabBytes : 16];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, h = lane >> 5;
    const int S = gridDim.x, split = blockIdx.x, kvh = blockIdx.y;
    const int rows = a.T * a.gqa;
    const int ntile = (rows + 32 * WAVES - 1) / (32 * WAVES);
    const int b = blockIdx.z / ntile;
    const int r0 = (blockIdx.z - b * ntile) * 32 * WAVES;

    int L = a.seq_lens ? min(a.seq_lens[b], a.seq_len) : a.seq_len;
    L = L < 0 ? 0 : (L > a.max_seq ? a.max_seq : L);
    // token t sees positions < L - T + t + 1
    const int t_last = (min(r0 + 32 * WAVES, rows) - 1) / a.gqa;
    const int p_begin = split * a.split_len;
    const int p_end = min(p_begin + a.split_len, L - a.T + t_last + 1);
    const int r = r0 + 32 * wave + c;
    const bool row_ok = r < rows;
    const int t = min(r, rows - 1) / a.gqa;
    const int hd = kvh * a.gqa + min(r, rows - 1) - t * a.gqa;
    const size_t qrow = ((size_t)b * a.T + t) * a.nh + hd;
    const int lim = row_ok ? min(L - a.T + t + 1, p_end) : 0;
    // the wave's rows grow with c: its first row has the smallest limit, its last valid one the largest
    const int w_first = r0 + 32 * wave;
    const bool wave_ok = w_first < rows;
    const int lim_lo = L - a.T + w_first / a.gqa + 1;
    const int lim_hi = min(L - a.T + (min(w_first + 32, rows) - 1) / a.gqa + 1, p_end);

    // staging.  TurboQuant: K unit (position, eighth of its dims), V unit (four
    // positions, four dims); FP16: 16-byte chunks of K, V unit (four positions,
    // eight dims).  Rows at or past p_end read as zeros.
    const size_t head_base = ((size_t)b * a.nkv + kvh) * (size_t)a.max_seq;
    const int nrows = max(p_end, 0);
    constexpr int EB = TQ ? 1 : 2;
    const __amdgpu_buffer_rsrc_t k_r = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.k + head_base * kD * EB), 0, nrows * kD * EB, kRsrcWord3);
    const __amdgpu_buffer_rsrc_t v_r = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(a.v + head_base * kD * EB), 0, nrows * kD * EB, kRsrcWord3);
    const int unit = tid & 255;
    const bool do_k = WAVES == 4 || wave < 4, do_v = WAVES == 4 || wave >= 4;
    constexpr int kQuads = kTile / 4;
    const int quad = unit & (kQuads - 1), dg = unit / kQuads;
    const int vslot = 16 * (quad >> 2) + 8 * (quad & 1) + 4 * ((quad >> 1) & 1);
    u32x4_t kreg[TQ ? 1 : 4], vreg[4];
    float sreg = 0.0f;
    auto load_k = [&](int p0) __attribute__((always_inline)) {
        if constexpr (TQ) {
            kreg[0] = __builtin_bit_cast(
                u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(k_r, (p0 + (unit >> 3)) * kD + (unit & 7) * 16, 0, 0));
            if (wave < 3) {   // wave 0 the K scales, 1 the residual norms, 2 the V scales
                const float *src = wave == 0 ? a.k_scales : wave == 1 ? a.k_rnorm : a.v_scales;
                sreg = src[head_base + min(p0 + c, nrows - 1)];
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                kreg[i] = __builtin_bit_cast(
                    u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(k_r, (p0 * 16 + i * 256 + tid) * 16, 0, 0));
        }
    };
    auto load_v = [&](int p0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int p = p0 + 4 * quad + i;
            if constexpr (TQ)
                vreg[i][0] = __builtin_amdgcn_raw_buffer_load_b32(v_r, p * kD + dg * 4, 0, 0);
            else
                vreg[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(v_r, (p * kD + dg * 8) * 2, 0, 0));
        }
    };
    const uint32_t lk = 4u * (uint32_t)c, lv = lk + 128u;
    auto store_k = [&](int buf) __attribute__((always_inline)) {
        if constexpr (TQ) {
            uint8_t *kd = &Ks[buf][0][(unit >> 3) * kKRow + (unit & 7) * 32];
#pragma unroll
            for (int e = 0; e < 2; e++) {   // 8 codes -> 16 bytes of each array, slots {0, 2, 1, 3} of a word
                u32x4_t hi, lo, sg;
#pragma unroll
                for (int hw = 0; hw < 2; hw++) {
                    const uint32_t w = kreg[0][2 * e + hw];
                    const uint32_t t0 = tab_read(tabs, w, 0, lk), t1 = tab_read(tabs, w, 1, lk);
                    const uint32_t t2 = tab_read(tabs, w, 2, lk), t3 = tab_read(tabs, w, 3, lk);
                    hi[2 * hw] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
                    lo[2 * hw] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
                    hi[2 * hw + 1] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
                    lo[2 * hw + 1] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
                    // +1 (0x3C00) where bit 7 of the code is set, -1 (0xBC00) where not
                    sg[2 * hw] = ((w << 8) & 0x80008000u) ^ 0xBC00BC00u;
                    sg[2 * hw + 1] = (w & 0x80008000u) ^ 0xBC00BC00u;
                }
                *reinterpret_cast<u32x4_t *>(kd + e * 16) = hi;
                *reinterpret_cast<u32x4_t *>(kd + kKBytes + e * 16) = lo;
                *reinterpret_cast<u32x4_t *>(kd + 2 * kKBytes + e * 16) = sg;
            }
            if (wave < 3) scl[TQ ? buf : 0][wave][c] = sreg;   // the same value from both halves
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int ck = i * 256 + tid;
                *reinterpret_cast<u32x4_t *>(&Ks[buf][0][(ck >> 4) * kKRow + (ck & 15) * 16]) = kreg[i];
            }
        }
    };
    auto store_v = [&](int buf) __attribute__((always_inline)) {
        if constexpr (TQ) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint32_t e[4];
#pragma unroll
                for (int i = 0; i < 4; i++) e[i] = tab_read(tabs, vreg[i][0], j, lv);
                uint8_t *vd = &Vs[buf][0][(dg * 4 + j) * kVRow + vslot * 2];
                *reinterpret_cast<u32x2_t *>(vd) = (u32x2_t){__builtin_amdgcn_perm(e[1], e[0], 0x05040100u),
                                                             __builtin_amdgcn_perm(e[3], e[2], 0x05040100u)};
                *reinterpret_cast<u32x2_t *>(vd + kVBytes) = (u32x2_t){
                    __builtin_amdgcn_perm(e[1], e[0], 0x07060302u), __builtin_amdgcn_perm(e[3], e[2], 0x07060302u)};
            }
        } else {
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
                *reinterpret_cast<u32x2_t *>(&Vs[buf][0][(dg * 8 + j) * kVRow + vslot * 2]) =
                    (u32x2_t){__builtin_amdgcn_perm(vreg[1][j >> 1], vreg[0][j >> 1], sel),
                              __builtin_amdgcn_perm(vreg[3][j >> 1], vreg[2][j >> 1], sel)};
            }
        }
    };

    if (p_begin < p_end) {
        if (do_k) load_k(p_begin);
        if (do_v) load_v(p_begin);
    }
    // the query operands: lane (row c, half h), step s: elements [16 s + 8 h, +8)
    half8_t qf[NP][8];
    if (TQ || (reinterpret_cast<uintptr_t>(a.q) & 15) == 0) {
#pragma unroll
        for (int p = 0; p < NP; p++)
#pragma unroll
            for (int s = 0; s < 8; s++)
                qf[p][s] = *reinterpret_cast<const half8_t *>(a.q + (qrow * NP + p) * kD + 16 * s + 8 * h);
    } else {   // a caller's rows may be aligned to their elements only
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int e = 0; e < 8; e++) qf[0][s][e] = a.q[qrow * kD + 16 * s + 8 * h + e];
    }
    if constexpr (TQ) {   // the spread codebooks: entry e's copies, 16 bytes per thread and turn
#pragma unroll 4
        for (int i = 0; i < 4096 / (64 * WAVES); i++) {
            const int ck = i * 64 * WAVES + tid;
            const int e = ck >> 4;
            const uint32_t v = tab_entry((ck & 15) < 8 ? a.k_codebook[e & 127] : a.v_codebook[e]);
            *reinterpret_cast<u32x4_t *>(&tabs[e * 256 + (ck & 15) * 16]) = (u32x4_t){v, v, v, v};
        }
        __syncthreads();
    }

    const float sl2 = a.attn_scale * 1.44269504f;   // scores in log2 units
    constexpr float kQjl = 0.79788456080286536f / (float)kD;   // sqrt(2 / pi) / d
    constexpr float kShift = TQ ? 0.0f : 10.0f;     // weights are 2^kShift exp2(score - max)
    float m_run = -INFINITY, l_run = 0.0f;          // l_run: this lane's share
    float16_t o[4];
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] = 0.0f;

    auto compute = [&](int p0, int buf) __attribute__((always_inline)) {
        if (!wave_ok || p0 >= lim_hi) return;
        // LDS reads are issued three operands ahead of their products and held
        // there (left alone, the scheduler puts each next to its use)
        float16_t s[NB];
        const uint8_t *ka = &Ks[buf][0][c * kKRow + 16 * h];
        if constexpr (TQ) {
            // operand i < 8: the signs of step i; then K hi and lo of each step
            auto read_k = [&](int i) __attribute__((always_inline)) {
                const int st = i < 8 ? i : (i - 8) >> 1;
                const int arr = i < 8 ? 2 : (i & 1);
                return *reinterpret_cast<const half8_t *>(ka + (NK > 1 ? arr : 0) * kKBytes + 32 * st);
            };
            half8_t kr_[4];
#pragma unroll
            for (int i = 0; i < 3; i++) kr_[i] = read_k(i);
#pragma unroll
            for (int i = 0; i < 24; i++) {
                if (i + 3 < 24) kr_[(i + 3) & 3] = read_k(i + 3);
                const half8_t k = kr_[i & 3];
                if (i < 8) {
                    s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qf[NP - 2][i], i ? s[0] : float16_t{}, 0, 0, 0);
                    s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qf[NP - 1][i], s[0], 0, 0, 0);
                } else {
                    const int st = (i - 8) >> 1;
                    s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qf[0][st], s[0], 0, 0, 0);
                    if (!(i & 1)) s[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k, qf[NP > 1 ? 1 : 0][st], s[0], 0, 0, 0);
                }
                if (i == 7) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const float4_t kr = *reinterpret_cast<const float4_t *>(&scl[TQ ? buf : 0][1][8 * q + 4 * h]);
#pragma unroll
                        for (int j = 0; j < 4; j++) s[0][4 * q + j] *= kr[j] * kQjl;
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4_t ks = *reinterpret_cast<const float4_t *>(&scl[TQ ? buf : 0][0][8 * q + 4 * h]);
#pragma unroll
                for (int j = 0; j < 4; j++) s[0][4 * q + j] *= ks[j] * sl2;
            }
        } else {
            half8_t kf[3][NB];
            auto read_k = [&](int st) __attribute__((always_inline)) {
#pragma unroll
                for (int n = 0; n < NB; n++)
                    kf[st % 3][n] = *reinterpret_cast<const half8_t *>(ka + 32 * n * kKRow + 32 * st);
            };
            read_k(0);
            read_k(1);
#pragma unroll
            for (int st = 0; st < 8; st++) {
                if (st + 2 < 8) read_k(st + 2);
#pragma unroll
                for (int n = 0; n < NB; n++)
                    s[n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[st % 3][n], qf[0][st], st ? s[n] : float16_t{}, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int n = 0; n < NB; n++)
#pragma unroll
                for (int i = 0; i < 16; i++) s[n][i] *= sl2;
        }
        // result i of block n is position p0 + 32 n + 8 (i >> 2) + 4 h + (i & 3)
        const bool edge = p0 + kTile > lim_lo || p0 + kTile > p_end;   // of the positions some row sees
        if (edge) {
#pragma unroll
            for (int n = 0; n < NB; n++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (p0 + 32 * n + 8 * (i >> 2) + 4 * h + (i & 3) >= lim) s[n][i] = -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int i = 0; i < 16; i++) mx = fmaxf(mx, s[n][i]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float nm = fmaxf(m_run, mx);
        // a row with no position yet keeps weight 0
        const float base = nm == -INFINITY ? 0.0f : nm - kShift;
        if (__builtin_amdgcn_ballot_w64(nm > m_run)) {   // some row's maximum grew
            const float corr = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - nm);
            l_run *= corr;
#pragma unroll
            for (int db = 0; db < 4; db++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[db][i] *= corr;
            m_run = nm;
        }
#pragma unroll
        for (int n = 0; n < NB; n++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                s[n][i] = __builtin_amdgcn_exp2f(s[n][i] - base);
                l_run += s[n][i];
            }
        // O^T += V^T P^T, 16 positions a step
        const uint8_t *va = &Vs[buf][0][c * kVRow + 16 * h];
        if constexpr (TQ) {
            half8_t ph[2];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const float4_t vs = *reinterpret_cast<const float4_t *>(&scl[TQ ? buf : 0][2][8 * q + 4 * h]);
#pragma unroll
                for (int j = 0; j < 4; j++) ph[q >> 1][4 * (q & 1) + j] = (_Float16)(s[0][4 * q + j] * vs[j]);
            }
            if (edge) {   // no weight where the row does not see the position, whatever its V scale
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (p0 + 8 * (i >> 2) + 4 * h + (i & 3) >= lim) ph[i >> 3][i & 7] = (_Float16)0.0f;
            }
            // operand i: step i / 8, V hi (i & 4 == 0) or lo, dim block i & 3
            auto read_v = [&](int i) __attribute__((always_inline)) {
                return *reinterpret_cast<const half8_t *>(va + (NV > 1 && (i & 4) ? kVBytes : 0) + (i & 3) * 32 * kVRow +
                                                          (i >> 3) * 32);
            };
            half8_t vr[4];
#pragma unroll
            for (int i = 0; i < 3; i++) vr[i] = read_v(i);
#pragma unroll
            for (int i = 0; i < 16; i++) {
                if (i + 3 < 16) vr[(i + 3) & 3] = read_v(i + 3);
                o[i & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vr[i & 3], ph[i >> 3], o[i & 3], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            half8_t vf[2][4], ph[2], pl[2];
            auto read_v = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int db = 0; db < 4; db++)
                    vf[i & 1][db] = *reinterpret_cast<const half8_t *>(va + db * 32 * kVRow + i * 32);
            };
            auto weights = [&](int i) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const float x = s[(i >> 1) % NB][8 * (i & 1) + e], y = s[(i >> 1) % NB][8 * (i & 1) + e + 1];
                    const half2_t hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(x, y));
                    const half2_t lo =
                        __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(x - (float)hi[0], y - (float)hi[1]));
                    ph[i & 1][e] = hi[0];
                    ph[i & 1][e + 1] = hi[1];
                    pl[i & 1][e] = lo[0];
                    pl[i & 1][e + 1] = lo[1];
                }
            };
            read_v(0);
            weights(0);
#pragma unroll
            for (int i = 0; i < 2 * NB; i++) {
                if (i + 1 < 2 * NB) {
                    read_v(i + 1);
                    weights(i + 1);
                }
#pragma unroll
                for (int db = 0; db < 4; db++) {
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i & 1][db], ph[i & 1], o[db], 0, 0, 0);
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i & 1][db], pl[i & 1], o[db], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    // Double-buffered, one barrier a tile.  Of TurboQuant's eight waves the two
    // that share a SIMD are w and w + 4: the first stages K before it computes,
    // the other V after, so that one's lookups run beside the other's products.
    if (p_begin < p_end) {
        if (do_k) store_k(0);
        if (do_v) store_v(0);
        if (p_begin + kTile < p_end) {
            if (do_k) load_k(p_begin + kTile);
            if (do_v) load_v(p_begin + kTile);
        }
        __syncthreads();
    }
    int buf = 0;
    for (int p0 = p_begin; p0 < p_end; p0 += kTile, buf ^= 1) {
        const bool more = p0 + kTile < p_end, more2 = p0 + 2 * kTile < p_end;
        if (do_k && more) {
            store_k(buf ^ 1);
            if (more2) load_k(p0 + 2 * kTile);
        }
        if (WAVES == 4 && more) {
            store_v(buf ^ 1);
            if (more2) load_v(p0 + 2 * kTile);
        }
        compute(p0, buf);
        if (WAVES == 8 && do_v && more) {
            store_v(buf ^ 1);
            if (more2) load_v(p0 + 2 * kTile);
        }
        __syncthreads();
    }
    l_run += __shfl_xor(l_run, 32);
    bool done = !row_ok;
    if constexpr (!TQ) {
        float any = 0.0f;   // NaN if a result is not finite
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) any = __builtin_fmaf(o[db][i], 0.0f, any);
        const uint64_t lanes = __builtin_amdgcn_ballot_w64(row_ok && any != any);
        const uint32_t again = (uint32_t)lanes | (uint32_t)(lanes >> 32);
        for (uint32_t rest = again; rest; rest &= rest - 1) {
            const int i = __builtin_ctz(rest), ri = w_first + i, ti = ri / a.gqa;
            exact_row(a, head_base, ((size_t)b * a.T + ti) * a.nh + kvh * a.gqa + ri - ti * a.gqa, p_begin,
                      min(L - a.T + ti + 1, p_end), S, split);
        }
        done = done || (again >> c & 1);
    }
    if (done) return;   // both lanes of a pair; no barrier follows

    // o[db][4 q + j]: dim 32 db + 8 q + 4 h + j of the lane's row
    if (S > 1) {   // the split's partial, maximum in log2 units (of the scale the weights have)
        const size_t pi = qrow * S + split;
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                *reinterpret_cast<float4_t *>(a.part_o + pi * kD + 32 * db + 8 * q + 4 * h) =
                    (float4_t){o[db][4 * q], o[db][4 * q + 1], o[db][4 * q + 2], o[db][4 * q + 3]};
        if (h == 0) {
            a.part_m[pi] = m_run - kShift;
            a.part_l[pi] = l_run;
        }
        return;
    }
    const float inv = 1.0f / fmaxf(l_run, 1e-10f);
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[db][i] *= inv;
    if constexpr (TQ) {
        // rotate back: D H D / sqrt(d), the butterflies of strides 1, 2 (j), 4
        // (the lane pair), 8, 16 (q), 32, 64 (db)
        float4_t sg[4][4];
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                sg[db][q] = *reinterpret_cast<const float4_t *>(a.signs + 32 * db + 8 * q + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; j++) o[db][4 * q + j] *= sg[db][q][j];
            }
#pragma unroll
        for (int st = 1; st < 16; st *= 2) {   // strides 1, 2, then 8, 16 as register strides 4, 8
#pragma unroll
            for (int db = 0; db < 4; db++)
#pragma unroll
                for (int i = 0; i < 16; i++)
                    if (!(i & st)) {
                        const float x = o[db][i], y = o[db][i + st];
                        o[db][i] = x + y;
                        o[db][i + st] = x - y;
                    }
            if (st == 2) {
#pragma unroll
                for (int db = 0; db < 4; db++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const float y = __shfl_xor(o[db][i], 32);
                        o[db][i] = h ? y - o[db][i] : o[db][i] + y;
                    }
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float x = o[0][i] + o[1][i], y = o[0][i] - o[1][i], z = o[2][i] + o[3][i], w = o[2][i] - o[3][i];
            o[0][i] = x + z;
            o[1][i] = y + w;
            o[2][i] = x - z;
            o[3][i] = y - w;
        }
        const float rscale = 1.0f / sqrtf((float)kD);
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) o[db][i] *= sg[db][i >> 2][i & 3] * rscale;
    }
    __half *out = a.out + qrow * kD + 4 * h;
    if (reinterpret_cast<uintptr_t>(a.out) & 7) {
#pragma unroll
        for (int db = 0; db < 4; db++)
#pragma unroll
            for (int i = 0; i < 16; i++) out[32 * db + 8 * (i >> 2) + (i & 3)] = __float2half(o[db][i]);
        return;
    }
#pragma unroll
    for (int db = 0; db < 4; db++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            half2_t lo = {(_Float16)o[db][4 * q], (_Float16)o[db][4 * q + 1]};
            half2_t hi = {(_Float16)o[db][4 * q + 2], (_Float16)o[db][4 * q + 3]};
            *reinterpret_cast<u32x2_t *>(out + 32 * db + 8 * q) =
                (u32x2_t){__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
        }
}

// grid ceil(rows / 32), block 256.  Each wave rotates 8 of the workgroup's 32
// rows, then projects all 32 onto 32 columns of S^T with f32 matrix-core
// products (exact products, f32 sums: 64 v_mfma_f32_32x32x2 per wave).  The
// matrix is read once per 32 rows; at once per 4 rows, from vector FMAs, the
// prep of 16384 rows took 20 us.
constexpr int kPrepRows = 32;
constexpr int kPrepStride = kD + 1;
__device__ __forceinline__ int plane_dim(int p) { return (p & ~7) | ((p & 1) << 1) | ((p >> 1) & 1) | (p & 4); }
__global__ void __launch_bounds__(256) tq_query_prep_kernel(const __half *__restrict__ q, int rows,
                                                            const float *__restrict__ signs,
                                                            const float *__restrict__ qjl_t,
                                                            _Float16 *__restrict__ planes) {
    __shared__ float qs[2][kPrepRows * kPrepStride];   // rotated rows, their projections
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row0 = blockIdx.x * kPrepRows;
    const float rscale = 1.0f / sqrtf((float)kD);
    const float sg0 = signs[lane], sg1 = signs[lane + 64];
    // the wave's part of the matrix, in flight while it rotates
    const int n = lane & 31, h = lane >> 5;
    float bv[kD / 2];
#pragma unroll
    for (int s = 0; s < kD / 2; s++) bv[s] = qjl_t[(2 * s + h) * kD + 32 * wave + n];
    float x0[8], x1[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const __half *qh = q + (size_t)min(row0 + 8 * wave + i, rows - 1) * kD;
        x0[i] = __half2float(qh[lane]) * sg0;
        x1[i] = __half2float(qh[lane + 64]) * sg1;
    }
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float u = imh_tq::hadamard64(x0[i], lane), v = imh_tq::hadamard64(x1[i], lane);
        float *dst = &qs[0][(8 * wave + i) * kPrepStride];
        dst[lane] = (u + v) * (sg0 * rscale);
        dst[lane + 64] = (u - v) * (sg1 * rscale);
    }
    __syncthreads();
    float16_t acc = {};
    const float *ap = &qs[0][n * kPrepStride + h];
#pragma unroll
    for (int s = 0; s < kD / 2; s++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ap[2 * s], bv[s], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 16; i++) qs[1][(8 * (i >> 2) + 4 * h + (i & 3)) * kPrepStride + 32 * wave + n] = acc[i];
    __syncthreads();
    // chunk e of 8 plane elements: row e / 64, plane (e / 16) & 3
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int e = i * 256 + tid;
        const int row = e >> 6, p = (e >> 4) & 3, ck = e & 15;
        if (row0 + row >= rows) continue;
        const float *src = &qs[p >> 1][row * kPrepStride];
        half8_t v;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const float x = src[ck * 8 + plane_dim(j)];
            const _Float16 hi = (_Float16)x;
            v[j] = (p & 1) ? (_Float16)(x - (float)hi) : hi;
        }
        *reinterpret_cast<half8_t *>(planes + ((size_t)(row0 + row) * 4 + p) * kD + ck * 8) = v;
    }
}

// grid ceil(rows / 4), block 256, one wave per row: split s weighs exp2(m_s -
// M); lane l sums dims l and l + 64 over the splits in order.
template <bool TQ>
__global__ void __launch_bounds__(256) prefill_combine_kernel(const float *__restrict__ part_o,
                                                              const float *__restrict__ part_m,
                                                              const float *__restrict__ part_l, int rows, int S,
                                                              const float *__restrict__ signs,
                                                              __half *__restrict__ out) {
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float *pm = part_m + (size_t)row * S, *pl = part_l + (size_t)row * S;
    const float *po = part_o + (size_t)row * S * kD;
    float M = -INFINITY;
    for (int s = lane; s < S; s += 64) M = fmaxf(M, pm[s]);
#pragma unroll
    for (int st = 32; st >= 1; st >>= 1) M = fmaxf(M, __shfl_xor(M, st));
    float o0 = 0.0f, o1 = 0.0f, ls = 0.0f;
    for (int s0 = 0; s0 < S; s0 += 64) {
        float f = 0.0f;
        if (s0 + lane < S) {
            const float m = pm[s0 + lane];
            if (m != -INFINITY) f = __builtin_amdgcn_exp2f(m - M);
            ls = __builtin_fmaf(f, pl[s0 + lane], ls);
        }
        const int n = min(64, S - s0);
        for (int i = 0; i < n; i++) {
            const float w = __shfl(f, i);
            o0 = __builtin_fmaf(w, po[(size_t)(s0 + i) * kD + lane], o0);
            o1 = __builtin_fmaf(w, po[(size_t)(s0 + i) * kD + lane + 64], o1);
        }
    }
#pragma unroll
    for (int st = 32; st >= 1; st >>= 1) ls += __shfl_xor(ls, st);
    const float inv = 1.0f / fmaxf(ls, 1e-10f);
    o0 *= inv;
    o1 *= inv;
    if constexpr (TQ) {
        const float sg0 = signs[lane], sg1 = signs[lane + 64];
        const float rscale = 1.0f / sqrtf((float)kD);
        const float u = imh_tq::hadamard64(o0 * sg0, lane), v = imh_tq::hadamard64(o1 * sg1, lane);
        o0 = (u + v) * (sg0 * rscale);
        o1 = (u - v) * (sg1 * rscale);
    }
    out[(size_t)row * kD + lane] = __float2half(o0);
    out[(size_t)row * kD + lane + 64] = __float2half(o1);
}

}  // namespace

namespace imh {

int launch_tq_query_prep(imh_stream *s, const __half *q, size_t rows, const float *signs, const float *qjl_t,
                         _Float16 *planes) {
    hipLaunchKernelGGL(tq_query_prep_kernel, dim3((unsigned)((rows + kPrepRows - 1) / kPrepRows)), dim3(256), 0,
                       s->stream, q, (int)rows, signs, qjl_t, planes);
    IMH_HIP(hipGetLastError());
    return IMH_OK;
}

int launch_prefill_combine(imh_stream *s, bool tq, size_t rows, uint32_t splits, const float *part_o,
                           const float *part_m, const float *part_l, const float *signs, __half *out) {
    const dim3 grid((unsigned)((rows + 3) / 4));
    if (tq)
        hipLaunchKernelGGL(prefill_combine_kernel<true>, grid, dim3(256), 0, s->stream, part_o, part_m, part_l,
                           (int)rows, (int)splits, signs, out);
    else
        hipLaunchKernelGGL(prefill_combine_kernel<false>, grid, dim3(256), 0, s->stream, part_o, part_m, part_l,
                           (int)rows, (int)splits, signs, out);
    IMH_HIP(hipGetLastError());
    return IMH_OK;
}

// KV splits: the count (each at least 256 positions) that gives the fewest
// rounds of workgroup slots -- two workgroups per CU for the FP16 kernel, one
// for the TurboQuant kernel (LDS) -- per split, a split costing a flat 0.5 % of
// the unsplit round, whatever the bytes of its partials (520 per row, written
// and read: 2 x 31 MB for the six splits of 9632 rows).
uint32_t prefill_splits(bool tq, uint32_t groups, uint32_t L, int cus) {
    const uint32_t slots = (uint32_t)cus * (tq ? 1 : 2);
    uint32_t best = 1;
    double best_cost = 1e30;
    for (uint32_t n = 1; n <= 64 && n <= std::max<uint32_t>(1, L / 256); n++) {
        const double cost = (double)((groups * n + slots - 1) / slots) / n + 0.005 * (n - 1);
        if (cost < best_cost) {
            best_cost = cost;
            best = n;
        }
    }
    return best;
}

int prefill_row_tile(bool tq) { return tq ? 256 : 128; }

int launch_prefill_attention(imh_stream *s, bool tq, uint32_t batch, uint32_t splits, const PrefillAttention &a) {
    const uint32_t rows = (uint32_t)a.T * a.gqa;
    const uint32_t tile = (uint32_t)prefill_row_tile(tq);
    const dim3 grid(splits, a.nkv, batch * ((rows + tile - 1) / tile));
    if (tq) hipLaunchKernelGGL(prefill_attention_kernel<true>, grid, dim3(512), 0, s->stream, a);
    else hipLaunchKernelGGL(prefill_attention_kernel<false>, grid, dim3(256), 0, s->stream, a);
    IMH_HIP(hipGetLastError());
    return IMH_OK;
}

}  // namespace imh
