// wq_gemm.h -- the matrix-core GEMM of a prefill-sized activation with
// group-128 affine weights kept at 4 or 8 bits, f16 operands:
//
//     C[m][n] = f16( sum_g s[n][g] * sum_{k in g} a[m][k] * (q[n][k] - z[n][g]) ),  f32 accumulate
//
// a = x, or x / awq carried as f16 hi + lo planes (~22 bits, two products).
// The weights are never rounded: INT4 codes enter as q - zi, zi the whole number
// next to the zero-point (exact in f16), with what is left of a fractional or
// very large zero-point applied in f32 to the group's sums; INT8 codes as f16 denormals
// (q * 2^-24, exact) with the zero-point applied in f32 to the group's sums.
//
// What bounds it: the matrix cores (32 x 32 x 16: 32 cycles) against the
// vector instructions that expand the codes and fold the group sums -- with
// two waves per SIMD both streams overlap completely as long as there are at
// most ~7 vector instructions per MFMA (measured: 4 and 6 per MFMA are free,
// 8 cost 1.4x; one wave per SIMD issues vector instructions at half that
// rate).  So everything but the expansion and the fold is kept off the vector
// unit: global addresses are buffer resources per workgroup (one per 16 rows of
// the activation), one offset register per thread and a scalar offset along
// the row; LDS addresses are immediates.
//  * The weights go from memory straight into registers in the operand layout
//    (lane = column + 32 x K half) and are expanded there: and-or places two
//    codes beside the f16 exponent of 1024 (the upper nibble of a byte as 16 q,
//    undone by the packed multiply-add that subtracts the zero-point), nine
//    instructions per 8 codes where a byte unpack takes eleven.
//  * The activation goes through LDS in operand order (blocks of 64 lanes x 16
//    bytes, padded by 16 bytes so that neither the 16-byte stores of a row's
//    chunks nor the reads conflict on banks), double-buffered by group, one
//    barrier per group; the next group's loads are issued between the MFMAs.
//  * A wave owns 32 MI rows x 64 columns (two column fragments; for a gate/up
//    pair one of each matrix, so the activation is applied in registers); a
//    workgroup's four waves share the rows.
//  * SZT: scales and zero-points come from a transposed copy ([group][column])
//    that the prep launch writes.  Read in place, a group's two bytes per row
//    pull a cache line each, four times the traffic of the codes themselves
//    (the fp8 GEMM at M = 509, K 9728 -> N 2560: 49.6 us, 40.1 without those
//    reads).
//
// Measured (us, before -> after; before: 128 x 128 tiles of 16 x 16 MFMAs with
// both operands through LDS, and for INT8 the 8-row matvec once per 8 rows):
// FFN block 2560 / 9728 with AWQ at 777 rows 466 -> 245 (of it gate + up 320 ->
// ~155, ~1000 TFLOP/s counting both planes), INT8 9728 -> 2560 at 200 rows 1180
// -> 43.  The matrix cores are busy 71 % of the time that a SIMD has waves (gate +
// up; no LDS bank conflicts); freezing the addresses of the activation and
// weight loads changes nothing, a quarter of the fold saves 6 %.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include "dpp_reduce.h"
#include "imh_internal.h"

namespace imh_wq {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kGS = 128;
constexpr int kThreads = 256;
constexpr int kBlk = 1040;          // LDS bytes of one 32-row x 16-k operand block, padded
constexpr uint32_t kRsrcWord3 = 0x00020000u;
constexpr float kTwoM24 = 5.9604644775390625e-08f;
constexpr float kTwo24 = 16777216.0f;

enum GemmEpi : int { GE_STORE, GE_SILU, GE_GELU };

struct Mats {
    const uint8_t *data[2];
    const __half *scales[2];
    const __half *zeros[2];
    __half *out[2];
};

// Tile order.  Workgroup ids go round-robin over the 8 XCDs, each with its
// own L2, so the linear id is first turned into an index that is contiguous
// per XCD; that index then walks bands of `band` row tiles (M) with the row
// tile fastest, so the workgroups resident on one XCD share both their A rows
// (one band) and their B columns (neighbouring column tiles) in its L2.
struct TileOrder {
    int tiles_m, tiles_n, band, splits;
};
__device__ __forceinline__ void tile_of(const TileOrder &o, int &mt, int &nt, int &split) {
    const int T = o.tiles_m * o.tiles_n * o.splits;
    const int L = blockIdx.x;
    const int x = L & 7, j = L >> 3;
    const int q = T >> 3, r = T & 7;
    const int t = x * q + min(x, r) + j;             // contiguous per XCD
    const int per_split = o.tiles_m * o.tiles_n;
    split = t / per_split;
    const int u = t - split * per_split;
    const int per_band = o.band * o.tiles_n;
    const int b = u / per_band, v = u - b * per_band;
    mt = b * o.band + v % o.band;
    nt = v / o.band;
}

// Rows [r0, r0 + n) of a row-major array of `rows` rows of `pitch` bytes as a
// buffer of their own, the rows past the array left out of its size.  An access
// whose vector offset holds row and column within the slab, and whose scalar
// offset stays within a row, is in or out of bounds by its row alone -- also
// where the bounds check leaves the scalar offset out, as it is specified to:
// a row selected by the scalar offset would not be checked at all.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_slab(const void *base, int r0, int n, int rows, int pitch) {
    const int first = min(r0, rows);
    return __builtin_amdgcn_make_buffer_rsrc((void *)((const uint8_t *)base + (size_t)first * pitch), 0,
                                             min(rows - first, n) * pitch, kRsrcWord3);
}

__device__ __forceinline__ uint32_t as_u32(half2_t h) { return __builtin_bit_cast(uint32_t, h); }
__device__ __forceinline__ half2_t as_h2(uint32_t u) { return __builtin_bit_cast(half2_t, u); }

__device__ __forceinline__ float gate_act(float g, float u, int epi) {
    float act;
    if (epi == GE_GELU) {
        float inner = 0.7978845608f * (g + 0.044715f * g * g * g);
        inner = fminf(fmaxf(inner, -10.0f), 10.0f);
        act = 0.5f * g * (1.0f + tanhf(inner));
    } else {
        act = g / (1.0f + __expf(-g));
    }
    return act * u;
}

// The column constants of a group.  INT8: (scale * 2^24, -zero) as f32.  INT4:
// the scale as f32, and the zero-point z split into the whole number zi within
// +-1024 next to it, which the code expansion subtracts (q - zi is exact in
// f16), and the rest z - zi (exact in f16 for every z), which is 0 for the
// quantizer's ordinary zero-points and otherwise folded in f32 against the rows'
// sums: halves {-(1024 + zi), z - zi}.
template <int BITS>
__device__ __forceinline__ u32x2_t column_consts(uint16_t s, uint16_t zbits) {
    const _Float16 z = __builtin_bit_cast(_Float16, zbits);
    const float sf = (float)__builtin_bit_cast(_Float16, s);
    if (BITS == 4) {
        const _Float16 zi = __builtin_elementwise_roundeven(
            __builtin_amdgcn_fmed3h(z, (_Float16)-1024.0f, (_Float16)1024.0f));
        return (u32x2_t){__builtin_bit_cast(uint32_t, sf), as_u32((half2_t){(_Float16)-1024.0f - zi, z - zi})};
    }
    return (u32x2_t){__builtin_bit_cast(uint32_t, sf * kTwo24), __builtin_bit_cast(uint32_t, -(float)z)};
}

// INT4: the second word's bias against 1024 + q, and -(64 + zi) against (1024 + 16 q) / 16
__device__ __forceinline__ uint32_t code_bias(uint32_t cz) { return __builtin_amdgcn_perm(cz, cz, 0x01000100u); }
__device__ __forceinline__ uint32_t code_bias16(uint32_t b1) {
    return as_u32(as_h2(b1) + (half2_t){(_Float16)960.0f, (_Float16)960.0f});
}

// Some column of the wave has a zero-point with a rest (c0, c1: second words).
__device__ __forceinline__ bool any_zero_rest(uint32_t c0, uint32_t c1) {
    return __builtin_amdgcn_ballot_w64((c0 | c1) >> 16) != 0;
}

// The sums of 32 rows of a group over its operand (NPL planes, `plane` bytes
// apart), as the products see it, laid out as a result: products with ones.
template <int NPL, int UNROLL>
__device__ __forceinline__ float16_t row_sums(const uint8_t *ab, int plane) {
    const uint32_t one = 0x3C003C00u;
    const half8_t ones = __builtin_bit_cast(half8_t, (u32x4_t){one, one, one, one});
    float16_t r = {};
#pragma unroll UNROLL
    for (int st = 0; st < 8; st++)
#pragma unroll
        for (int p = 0; p < NPL; p++)
            r = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const half8_t *>(ab + p * plane + st * kBlk),
                                                       ones, r, 0, 0, 0);
    return r;
}

// One prep launch.  Workgroups below `ablocks`: the activation planes -- hi =
// f16(x / awq), lo = f16(x / awq - hi) (lo only with awq; without it hi = x) --
// a chunk of 8 elements per thread in the order the code expansion yields
// (INT4 {0, 4, 1, 5, 2, 6, 3, 7}, INT8 as it is), and for INT8 the rows' group
// sums * 2^-24.  The others transpose 64 columns x 16 groups of the scales
// and zero-points of matrix blockIdx / per into szt[mat][group][column].
template <int BITS>
__global__ void __launch_bounds__(256) prep_kernel(const __half *__restrict__ x, const __half *__restrict__ awq,
                                                   __half *__restrict__ hi_out, __half *__restrict__ lo_out,
                                                   float *__restrict__ gsum, size_t chunks, int K, int ablocks,
                                                   Mats mats, u32x2_t *__restrict__ szt, int N, int sz_per_mat) {
    const int G = K / kGS;
    if ((int)blockIdx.x >= ablocks) {
        int blk = (int)blockIdx.x - ablocks;
        const int mat = blk >= sz_per_mat ? 1 : 0;
        blk -= mat * sz_per_mat;
        const int gblk = (G + 15) / 16;
        const int n = (blk / gblk) * 64 + (int)(threadIdx.x & 63);
        const int g0 = (blk % gblk) * 16 + (int)(threadIdx.x >> 6) * 4;
        if (n >= N) return;
        const uint16_t *s = reinterpret_cast<const uint16_t *>(mat ? mats.scales[1] : mats.scales[0]) + (size_t)n * G;
        const uint16_t *z = reinterpret_cast<const uint16_t *>(mat ? mats.zeros[1] : mats.zeros[0]) + (size_t)n * G;
        uint16_t sv[4], zv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int g = min(g0 + i, G - 1);
            sv[i] = s[g];
            zv[i] = z[g];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (g0 + i < G) szt[((size_t)mat * G + g0 + i) * N + n] = column_consts<BITS>(sv[i], zv[i]);
        return;
    }
    const size_t c_raw = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool live = c_raw < chunks;
    const size_t c = live ? c_raw : 0;
    const int cpr = K / 8;
    const size_t m = c / cpr;
    const int ck = (int)(c - m * cpr);
    const u32x4_t xv = *reinterpret_cast<const u32x4_t *>(x + c * 8);
    const _Float16 *xh = reinterpret_cast<const _Float16 *>(&xv);
    half8_t hi, lo;
    float sum = 0.0f;
    u32x4_t wv = {};
    if (awq) wv = *reinterpret_cast<const u32x4_t *>(awq + (size_t)ck * 8);
    const _Float16 *wh = reinterpret_cast<const _Float16 *>(&wv);
    constexpr int kSlot4[8] = {0, 4, 1, 5, 2, 6, 3, 7};
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int e = BITS == 4 ? kSlot4[j] : j;
        const float v = awq ? (float)xh[e] * __builtin_amdgcn_rcpf((float)wh[e]) : (float)xh[e];
        hi[j] = (_Float16)v;
        lo[j] = (_Float16)(v - (float)hi[j]);
        if (BITS == 8) sum += (float)hi[j] + (awq ? (float)lo[j] : 0.0f);
    }
    if (live) {
        *reinterpret_cast<half8_t *>(hi_out + c * 8) = hi;
        if (awq) *reinterpret_cast<half8_t *>(lo_out + c * 8) = lo;
    }
    if (BITS == 8) {   // a group's 16 chunks are 16 consecutive lanes
        sum += __shfl_xor(sum, 1);
        sum += __shfl_xor(sum, 2);
        sum += __shfl_xor(sum, 4);
        sum += __shfl_xor(sum, 8);
        if (live && (threadIdx.x & 15) == 0) gsum[m * G + ck / 16] = sum * kTwoM24;
    }
}

// grid tiles_m * tiles_n * splits, block 256.  Split z covers groups [z * per,
// min((z + 1) * per, G)); with part the f32 partials go to part[z][M][mats *
// N], else the results (PAIR: both, or act(gate) * up) are stored.
//
// Operand layouts of v_mfma_f32_32x32x16_f16, k step s (0..7) of a group: lane
// (n or m = l & 31, h = l >> 5) holds the 8 elements [64 h + 8 s, +8) of its
// column or row; D: lane l, value i: row 8 (i >> 2) + 4 h + (i & 3), column l & 31.
// INT4: the lane's 32 code bytes of a group; INT8: its 64, half a group
// (steps 0-3, 4-7) at a time.
//
// DIRECT: the activation is x itself (row-major, natural order; reordered on
// the way to LDS), one plane.
template <int BITS, int NPL, int MI, bool PAIR, bool DIRECT, bool SZT>
__global__ void __launch_bounds__(kThreads, 2) wq_gemm_kernel(const __half *__restrict__ a_hi,
                                                              const __half *__restrict__ a_lo,
                                                              const float *__restrict__ gsum, Mats mats,
                                                              const u32x2_t *__restrict__ szt, float *__restrict__ part,
                                                              int M, int N, int K, int per, int epi, TileOrder order) {
    constexpr int BM = 32 * MI;
    constexpr int TN = PAIR ? 128 : 256;             // columns (of each matrix) per workgroup
    constexpr int PLANE = MI * 8 * kBlk;
    constexpr int ACH = MI * 2;                      // 16-byte chunks per thread, plane and group
    constexpr int HALVES = BITS == 8 ? 2 : 1;        // B register sets per group
    constexpr int SPB = 8 / HALVES;                  // k steps per B register set
    __shared__ __attribute__((aligned(16))) uint8_t As[2][NPL][PLANE];
    __shared__ __attribute__((aligned(16))) float Rs[2][BITS == 8 ? BM : 4];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int nl = lane & 31, h = lane >> 5;
    int mt, nt, split;
    tile_of(order, mt, nt, split);
    const int m0 = mt * BM;
    const int nb = nt * TN;                          // the workgroup's first column
    const int n0 = nb + wave * (TN / 4);
    const int G = K / kGS;
    const int g_begin = split * per;
    const int g_end = min(g_begin + per, G);

    // B: fragment j is columns n0 + 32 j of the one matrix, or columns n0 of matrix j
    const int row_bytes = K * BITS / 8;
    const int cols = min(TN, N - nb);
    __amdgpu_buffer_rsrc_t w_r[2], s_r[2], z_r[2];
    int bvo[2], svo[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int t = PAIR ? j : 0;
        w_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.data[t] + (size_t)nb * row_bytes), 0,
                                                   cols * row_bytes, kRsrcWord3);
        const int n = min(n0 + (PAIR ? 0 : 32 * j) + nl, N - 1) - nb;
        bvo[j] = n * row_bytes + (BITS == 4 ? 32 : 64) * h;
        if (SZT) {
            s_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(szt + (size_t)t * G * N + nb), 0,
                                                       (int)(((size_t)G * N - nb) * sizeof(u32x2_t)), kRsrcWord3);
            svo[j] = n * (int)sizeof(u32x2_t);
        } else {
            s_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.scales[t] + (size_t)nb * G), 0, cols * G * 2,
                                                       kRsrcWord3);
            z_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.zeros[t] + (size_t)nb * G), 0, cols * G * 2,
                                                       kRsrcWord3);
            svo[j] = n * G * 2;
        }
    }
    struct BRegs {
        u32x4_t w[2][2];
        u32x2_t c[2];      // column constants (!SZT: the scale's and zero's bits until used)
    };
    auto load_b = [&](int g, int half, BRegs &b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int so = g * (kGS * BITS / 8) + half * 32;
            b.w[j][0] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_r[j], bvo[j], so, 0));
            b.w[j][1] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_r[j], bvo[j] + 16, so, 0));
        }
    };
    auto load_c = [&](int g, u32x2_t *c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (SZT) {
                c[j] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                                       s_r[j], svo[j], g * N * (int)sizeof(u32x2_t), 0));
            } else {
                c[j][0] = __builtin_amdgcn_raw_buffer_load_b16(s_r[j], svo[j], g * 2, 0);
                c[j][1] = __builtin_amdgcn_raw_buffer_load_b16(z_r[j], svo[j], g * 2, 0);
            }
        }
    };

    // A: chunk i of a thread is row tid / 16, chunk tid % 16 of the group's i-th
    // slab of 16 rows (rows past M read as zeros); it lands in block (row / 32, k
    // step cc & 7)
    const int arows = min(BM, M - m0);
    const __half *planes[2] = {a_hi, a_lo};
    __amdgpu_buffer_rsrc_t a_r[NPL][ACH];
#pragma unroll
    for (int p = 0; p < NPL; p++)
#pragma unroll
        for (int i = 0; i < ACH; i++) a_r[p][i] = row_slab(planes[p], m0 + 16 * i, 16, M, K * 2);
    const int ar0 = tid >> 4, acc0 = tid & 15;
    const int avo = (ar0 * K + acc0 * 8) * 2;
    const int a_lds = (acc0 & 7) * kBlk + (ar0 + 32 * (acc0 >> 3)) * 16;
    auto load_a = [&](int g, int p, u32x4_t *ar) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ACH; i++)
            ar[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_r[p][i], avo, g * kGS * 2, 0));
    };
    auto store_a = [&](int buf, int p, const u32x4_t *ar) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ACH; i++) {
            u32x4_t v = ar[i];
            if (DIRECT && BITS == 4)   // natural order -> {0, 4, 1, 5, 2, 6, 3, 7}
                v = (u32x4_t){__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                              __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
            *reinterpret_cast<u32x4_t *>(&As[buf][p][a_lds + (i >> 1) * 8 * kBlk + (i & 1) * 256]) = v;
        }
    };
    float rsv = 0.0f;
    const __amdgpu_buffer_rsrc_t r_r =
        __builtin_amdgcn_make_buffer_rsrc((void *)(gsum + (size_t)m0 * G), 0, arows * G * 4, kRsrcWord3);
    const int rvo = (tid & (BM - 1)) * G * 4;
    auto load_rs = [&](int g) __attribute__((always_inline)) {
        if (BITS == 8) rsv = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_r, rvo, g * 4, 0));
    };
    auto store_rs = [&](int buf) __attribute__((always_inline)) {
        if (BITS == 8) Rs[buf][tid & (BM - 1)] = rsv;   // the same value from each wave
    };

    float16_t acc[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mi][j][i] = 0.0f;

    // in registers, so that each and-or is one instruction (a literal operand
    // would make it two)
    uint32_t m_lo, m_hi, exp1k;
    asm("s_mov_b32 %0, 0x000f000f" : "=s"(m_lo));
    asm("s_mov_b32 %0, 0x00f000f0" : "=s"(m_hi));
    asm("v_mov_b32 %0, 0x64006400" : "=v"(exp1k));
    // 8 codes of fragment j at step s of the register set, as MFMA operand
    auto expand = [&](const BRegs &b, int j, int s, uint32_t b1, uint32_t b16) __attribute__((always_inline)) {
        u32x4_t o;
        if (BITS == 4) {
            const uint32_t w = b.w[j][s >> 2][s & 3], w8 = w >> 8;
            const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
            o[0] = as_u32(as_h2((w & m_lo) | exp1k) + as_h2(b1));
            o[1] = as_u32(__builtin_elementwise_fma(as_h2((w & m_hi) | exp1k), sixteenth, as_h2(b16)));
            o[2] = as_u32(as_h2((w8 & m_lo) | exp1k) + as_h2(b1));
            o[3] = as_u32(__builtin_elementwise_fma(as_h2((w8 & m_hi) | exp1k), sixteenth, as_h2(b16)));
        } else {
            const uint32_t w0 = b.w[j][s >> 1][2 * (s & 1)], w1 = b.w[j][s >> 1][2 * (s & 1) + 1];
            o[0] = __builtin_amdgcn_perm(0u, w0, 0x0C010C00u);
            o[1] = __builtin_amdgcn_perm(0u, w0, 0x0C030C02u);
            o[2] = __builtin_amdgcn_perm(0u, w1, 0x0C010C00u);
            o[3] = __builtin_amdgcn_perm(0u, w1, 0x0C030C02u);
        }
        return __builtin_bit_cast(half8_t, o);
    };

    // One group from LDS buffer buf: the MFMAs of its eight k steps, the next
    // group's loads issued and its activation stored between them (hook), then
    // the fold.  cur[half] holds the group's codes, cc its column constants.
    auto compute = [&](int buf, BRegs *cur, const u32x2_t *cc, auto &&hook) __attribute__((always_inline)) {
        float sc[2], nz[2] = {};
        uint32_t cz[2], b1[2] = {}, b16[2] = {};
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const u32x2_t c = SZT ? cc[j] : column_consts<BITS>((uint16_t)cc[j][0], (uint16_t)cc[j][1]);
            const uint32_t cs = c[0];   // scalars: a bit cast of a vector element takes element 0
            cz[j] = c[1];
            sc[j] = __builtin_bit_cast(float, cs);
            if (BITS == 4) {
                b1[j] = code_bias(cz[j]);
                b16[j] = code_bias16(b1[j]);
            } else {
                nz[j] = __builtin_bit_cast(float, cz[j]);
            }
        }
        const uint8_t *ab = &As[buf][0][lane * 16];
        half8_t af[2][NPL][MI];
        auto read_a = [&](int st) __attribute__((always_inline)) {
#pragma unroll
            for (int p = 0; p < NPL; p++)
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
                    af[st & 1][p][mi] = *reinterpret_cast<const half8_t *>(ab + p * PLANE + (mi * 8 + st) * kBlk);
        };
        const float16_t zero16 = {};
        float16_t gg[MI][2];
        // the operands of step st + 1 are read and expanded while step st's
        // MFMAs run; nothing moves across the steps (left alone, the scheduler
        // sinks the next group's loads to their uses and waits for them there)
        half8_t bf[2][2];
        auto expand_step = [&](int st) __attribute__((always_inline)) {
#pragma unroll
            for (int j = 0; j < 2; j++) bf[st & 1][j] = expand(cur[st / SPB], j, st % SPB, b1[j], b16[j]);
        };
        read_a(0);
        expand_step(0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int st = 0; st < 8; st++) {
            if (st < 7) read_a(st + 1);
            hook(st);
            if (st < 7) expand_step(st + 1);
#pragma unroll
            for (int p = 0; p < NPL; p++)
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        gg[mi][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[st & 1][p][mi], bf[st & 1][j],
                                                                           st == 0 && p == 0 ? zero16 : gg[mi][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (BITS == 4 && any_zero_rest(cz[0], cz[1])) {
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
                const float16_t rs = row_sums<NPL, 8>(ab + mi * 8 * kBlk, PLANE);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const float rest = (float)as_h2(cz[j])[1];
#pragma unroll
                    for (int i = 0; i < 16; i++) gg[mi][j][i] = __builtin_fmaf(-rest, rs[i], gg[mi][j][i]);
                }
            }
        }
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
            float4_t rs[4];
            if (BITS == 8) {
#pragma unroll
                for (int q = 0; q < 4; q++) rs[q] = *reinterpret_cast<const float4_t *>(&Rs[buf][32 * mi + 8 * q + 4 * h]);
            }
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    float v = gg[mi][j][i];
                    if (BITS == 8) v = __builtin_fmaf(nz[j], rs[i >> 2][i & 3], v);
                    acc[mi][j][i] = __builtin_fmaf(sc[j], v, acc[mi][j][i]);
                }
        }
    };

    u32x4_t ar[ACH];
    BRegs b0[HALVES], b1r[HALVES];
    u32x2_t c0[2], c1[2];
    if (g_begin < g_end) {
        load_b(g_begin, 0, b0[0]);
        load_c(g_begin, c0);
        load_rs(g_begin);
#pragma unroll
        for (int p = 0; p < NPL; p++) {
            load_a(g_begin, p, ar);
            store_a(0, p, ar);
        }
        store_rs(0);
        __syncthreads();
    }
    // group g from buffer buf, its codes in cur; the next group's loads are
    // unconditional (past the last group the last one is loaded again), so no
    // wait for the current set has to cover them
    auto step = [&](int g, int buf, BRegs *cur, u32x2_t *cc, BRegs *nxt, u32x2_t *nc) __attribute__((always_inline)) {
        const int gn = min(g + 1, g_end - 1);
        compute(buf, cur, cc, [&](int st) __attribute__((always_inline)) {
            if (st == 0) {
                load_a(gn, 0, ar);
                if (HALVES == 2) load_b(g, 1, cur[1]);
            }
            if (st == 1) {
                if (HALVES == 1) load_b(gn, 0, nxt[0]);
                load_c(gn, nc);
                load_rs(gn);
            }
            if (NPL == 2 && st == 4) {
                store_a(buf ^ 1, 0, ar);
                load_a(gn, 1, ar);
            }
            if (HALVES == 2 && st == 4) load_b(gn, 0, nxt[0]);
        });
        store_a(buf ^ 1, NPL - 1, ar);
        store_rs(buf ^ 1);
        __syncthreads();
    };
    for (int g = g_begin; g < g_end; g += 2) {
        step(g, 0, b0, c0, b1r, c1);
        if (g + 1 >= g_end) break;
        step(g + 1, 1, b1r, c1, b0, c0);
    }

#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int m = m0 + 32 * mi + 8 * (i >> 2) + 4 * h + (i & 3);
            if (m >= M) continue;
            if (PAIR) {
                const int n = n0 + nl;
                if (n >= N) continue;
                const float g = acc[mi][0][i], u = acc[mi][1][i];
                if (part) {
                    float *p = part + ((size_t)split * M + m) * 2 * N + n;
                    p[0] = g;
                    p[N] = u;
                } else if (epi == GE_STORE) {
                    mats.out[0][(size_t)m * N + n] = __float2half(g);
                    mats.out[1][(size_t)m * N + n] = __float2half(u);
                } else {
                    mats.out[0][(size_t)m * N + n] = __float2half(gate_act(g, u, epi));
                }
            } else {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int n = n0 + 32 * j + nl;
                    if (n >= N) continue;
                    if (part) part[((size_t)split * M + m) * N + n] = acc[mi][j][i];
                    else mats.out[0][(size_t)m * N + n] = __float2half(acc[mi][j][i]);
                }
            }
        }
}

// Up to 32 rows in one launch: bound by memory latency and launches, not by
// any rate, so the activation's division and hi / lo split, the group sums and
// the scale reads are part of the launch, and a workgroup has the loads of a
// whole block of groups in flight before its first product (each wave 64
// columns, as above; one 32-row tile).  A group's registers are loaded again, a
// block on, as soon as it is done.  AWQ: x / awq in two planes; without, x in
// one (INT8's second plane would be zero).  A group costs a workgroup about
// 1.05 us on top of ~4 (one wave per SIMD issues the expansion at half rate);
// 16 x 16 products, and eight waves with the groups halved between them, came
// to the same or more (33 and 43 us for the FFN at 12 rows against 33).
constexpr int kRowsBlock = 4;   // groups per block (INT8: half, for its code bytes)
template <int BITS, bool AWQ, bool PAIR>
__global__ void __launch_bounds__(kThreads, 2) wq_rows_kernel(const __half *__restrict__ x,
                                                              const __half *__restrict__ awq, Mats mats,
                                                              float *__restrict__ part, int M, int N, int K, int per,
                                                              int epi, int tiles_n) {
    constexpr int NPL = AWQ ? 2 : 1;
    constexpr int TN = PAIR ? 128 : 256;
    constexpr int PB = BITS == 8 ? kRowsBlock / 2 : kRowsBlock;
    constexpr int WQ = BITS / 2;                     // code quads (16 bytes) per fragment and group
    constexpr int PLANE = 8 * kBlk;
    __shared__ __attribute__((aligned(16))) uint8_t As[PB][NPL][PLANE];
    __shared__ __attribute__((aligned(16))) float Rs[PB][BITS == 8 ? 32 : 4];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int nl = lane & 31, h = lane >> 5;
    const int nt = blockIdx.x % tiles_n, split = blockIdx.x / tiles_n;
    const int nb = nt * TN;
    const int n0 = nb + wave * (TN / 4);
    const int G = K / kGS;
    const int g_begin = split * per;
    const int g_end = min(g_begin + per, G);

    const int row_bytes = K * BITS / 8;
    const int cols = min(TN, N - nb);
    __amdgpu_buffer_rsrc_t w_r[2], s_r[2], z_r[2];
    int bvo[2], svo[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int t = PAIR ? j : 0;
        w_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.data[t] + (size_t)nb * row_bytes), 0,
                                                   cols * row_bytes, kRsrcWord3);
        s_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.scales[t] + (size_t)nb * G), 0, cols * G * 2, kRsrcWord3);
        z_r[j] = __builtin_amdgcn_make_buffer_rsrc((void *)(mats.zeros[t] + (size_t)nb * G), 0, cols * G * 2, kRsrcWord3);
        const int n = min(n0 + (PAIR ? 0 : 32 * j) + nl, N - 1) - nb;
        bvo[j] = n * row_bytes + (BITS == 4 ? 32 : 64) * h;
        svo[j] = n * G * 2;
    }
    u32x4_t bw[PB][2][WQ];
    uint16_t bs[PB][2], bz[PB][2];
    auto load_b = [&](int i, int g) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
#pragma unroll
            for (int q = 0; q < WQ; q++)
                bw[i][j][q] = __builtin_bit_cast(
                    u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_r[j], bvo[j] + 16 * q, g * (kGS * BITS / 8), 0));
            bs[i][j] = __builtin_amdgcn_raw_buffer_load_b16(s_r[j], svo[j], g * 2, 0);
            bz[i][j] = __builtin_amdgcn_raw_buffer_load_b16(z_r[j], svo[j], g * 2, 0);
        }
    };
    // the activation: rows tid / 16 and + 16, chunk tid % 16 of each group (rows past M read as zeros)
    const __amdgpu_buffer_rsrc_t x_r[2] = {row_slab(x, 0, 16, M, K * 2), row_slab(x, 16, 16, M, K * 2)};
    const __amdgpu_buffer_rsrc_t q_r =
        __builtin_amdgcn_make_buffer_rsrc((void *)(AWQ ? awq : x), 0, K * 2, kRsrcWord3);
    const int ar0 = tid >> 4, ac = tid & 15;
    const int xvo = (ar0 * K + ac * 8) * 2;
    const bool two = M > 16;
    const int a_lds = (ac & 7) * kBlk + (ar0 + 32 * (ac >> 3)) * 16;
    u32x4_t xr[PB][2], qr[PB];
    auto load_x = [&](int g0) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const int g = min(g0 + i, g_end - 1);
            if (AWQ) qr[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(q_r, ac * 16, g * 256, 0));
            xr[i][0] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_r[0], xvo, g * 256, 0));
            if (two) xr[i][1] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(x_r[1], xvo, g * 256, 0));
        }
    };
    constexpr int kSlot4[8] = {0, 4, 1, 5, 2, 6, 3, 7};
    auto store_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PB; i++) {
            const _Float16 *qh = reinterpret_cast<const _Float16 *>(&qr[i]);
            float inv[8];
            if (AWQ) {
#pragma unroll
                for (int e = 0; e < 8; e++) inv[e] = __builtin_amdgcn_rcpf((float)qh[e]);
            }
#pragma unroll
            for (int p = 0; p < 2; p++) {
                half8_t hi = {}, lo = {};   // rows 16-31 of a call with fewer: zeros
                float sum = 0.0f;
                if (p == 0 || two) {
                    const _Float16 *xh = reinterpret_cast<const _Float16 *>(&xr[i][p]);
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const int e = BITS == 4 ? kSlot4[k] : k;
                        const float v = AWQ ? (float)xh[e] * inv[e] : (float)xh[e];
                        hi[k] = (_Float16)v;
                        lo[k] = (_Float16)(v - (float)hi[k]);
                        if (BITS == 8) sum += (float)hi[k] + (AWQ ? (float)lo[k] : 0.0f);
                    }
                }
                *reinterpret_cast<half8_t *>(&As[i][0][a_lds + p * 256]) = hi;
                if (AWQ) *reinterpret_cast<half8_t *>(&As[i][NPL - 1][a_lds + p * 256]) = lo;
                if (BITS == 8) {   // a row's 16 chunks are 16 consecutive lanes
                    sum = imh_dpp::row16_sum(sum);
                    if (ac == 0) Rs[i][ar0 + 16 * p] = sum * kTwoM24;
                }
            }
        }
    };

    uint32_t m_lo, m_hi, exp1k;
    asm("s_mov_b32 %0, 0x000f000f" : "=s"(m_lo));
    asm("s_mov_b32 %0, 0x00f000f0" : "=s"(m_hi));
    asm("v_mov_b32 %0, 0x64006400" : "=v"(exp1k));
    float16_t acc[2];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[j][i] = 0.0f;
    uint32_t rests = 0;   // INT4: the high halves tell whether a column of the block has a zero-point with a rest
    auto compute = [&](int i) __attribute__((always_inline)) {
        float sc[2], nz[2];
        uint32_t cz[2], b1[2], b16[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const u32x2_t c = column_consts<BITS>(bs[i][j], bz[i][j]);
            const uint32_t cs = c[0];   // scalars: a bit cast of a vector element takes element 0
            cz[j] = c[1];
            sc[j] = __builtin_bit_cast(float, cs);
            nz[j] = __builtin_bit_cast(float, cz[j]);
            b1[j] = code_bias(cz[j]);
            b16[j] = code_bias16(b1[j]);
        }
        const float16_t zero16 = {};
        float16_t gg[2];
        const uint8_t *ab = &As[i][0][lane * 16];
#pragma unroll
        for (int st = 0; st < 8; st++) {
            half8_t af[NPL], bf[2];
#pragma unroll
            for (int p = 0; p < NPL; p++) af[p] = *reinterpret_cast<const half8_t *>(ab + p * PLANE + st * kBlk);
#pragma unroll
            for (int j = 0; j < 2; j++) {
                u32x4_t o;
                if (BITS == 4) {
                    const uint32_t w = bw[i][j][(st >> 2) % WQ][st & 3], w8 = w >> 8;
                    const half2_t sixteenth = {(_Float16)0.0625f, (_Float16)0.0625f};
                    o[0] = as_u32(as_h2((w & m_lo) | exp1k) + as_h2(b1[j]));
                    o[1] = as_u32(__builtin_elementwise_fma(as_h2((w & m_hi) | exp1k), sixteenth, as_h2(b16[j])));
                    o[2] = as_u32(as_h2((w8 & m_lo) | exp1k) + as_h2(b1[j]));
                    o[3] = as_u32(__builtin_elementwise_fma(as_h2((w8 & m_hi) | exp1k), sixteenth, as_h2(b16[j])));
                } else {
                    const uint32_t w0 = bw[i][j][(st >> 1) % WQ][2 * (st & 1)], w1 = bw[i][j][(st >> 1) % WQ][2 * (st & 1) + 1];
                    o[0] = __builtin_amdgcn_perm(0u, w0, 0x0C010C00u);
                    o[1] = __builtin_amdgcn_perm(0u, w0, 0x0C030C02u);
                    o[2] = __builtin_amdgcn_perm(0u, w1, 0x0C010C00u);
                    o[3] = __builtin_amdgcn_perm(0u, w1, 0x0C030C02u);
                }
                bf[j] = __builtin_bit_cast(half8_t, o);
            }
#pragma unroll
            for (int p = 0; p < NPL; p++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    gg[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[p], bf[j], st == 0 && p == 0 ? zero16 : gg[j], 0, 0, 0);
        }
        if (BITS == 4) rests |= cz[0] | cz[1];
        float4_t rs[4];
        if (BITS == 8) {
#pragma unroll
            for (int q = 0; q < 4; q++) rs[q] = *reinterpret_cast<const float4_t *>(&Rs[i][8 * q + 4 * h]);
        }
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int k = 0; k < 16; k++) {
                float v = gg[j][k];
                if (BITS == 8) v = __builtin_fmaf(nz[j], rs[k >> 2][k & 3], v);
                acc[j][k] = __builtin_fmaf(sc[j], v, acc[j][k]);
            }
    };

    if (g_begin < g_end) {
        load_x(g_begin);
#pragma unroll
        for (int i = 0; i < PB; i++) load_b(i, min(g_begin + i, g_end - 1));
        __builtin_amdgcn_sched_barrier(0);   // every load above issues before the first wait
    }
    for (int g0 = g_begin; g0 < g_end; g0 += PB) {
        store_x();
        __syncthreads();
        const bool more = g0 + PB < g_end;
        if (more) load_x(g0 + PB);
#pragma unroll
        for (int i = 0; i < PB; i++) {
            if (g0 + i < g_end) compute(i);
            if (more) load_b(i, min(g0 + PB + i, g_end - 1));
        }
        // one branch per block (one per group: 2 % of the launch), the constants read once more
        if (BITS == 4 && any_zero_rest(rests, 0)) {
#pragma unroll 1
            for (int i = 0; i < min(PB, g_end - g0); i++) {
                const float16_t rs = row_sums<NPL, 1>(&As[i][0][lane * 16], PLANE);
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const int so = (g0 + i) * 2;
                    const u32x2_t c = column_consts<BITS>(__builtin_amdgcn_raw_buffer_load_b16(s_r[j], svo[j], so, 0),
                                                          __builtin_amdgcn_raw_buffer_load_b16(z_r[j], svo[j], so, 0));
                    const uint32_t cs = c[0], cz = c[1];
                    const float f = __builtin_bit_cast(float, cs) * (float)as_h2(cz)[1];
#pragma unroll
                    for (int k = 0; k < 16; k++) acc[j][k] = __builtin_fmaf(-f, rs[k], acc[j][k]);
                }
            }
            rests = 0;
        }
        if (more) __syncthreads();   // the planes are rewritten next
    }

#pragma unroll
    for (int i = 0; i < 16; i++) {
        const int m = 8 * (i >> 2) + 4 * h + (i & 3);
        if (m >= M) continue;
        if (PAIR) {
            const int n = n0 + nl;
            if (n >= N) continue;
            const float g = acc[0][i], u = acc[1][i];
            if (part) {
                float *p = part + ((size_t)split * M + m) * 2 * N + n;
                p[0] = g;
                p[N] = u;
            } else if (epi == GE_STORE) {
                mats.out[0][(size_t)m * N + n] = __float2half(g);
                mats.out[1][(size_t)m * N + n] = __float2half(u);
            } else {
                mats.out[0][(size_t)m * N + n] = __float2half(gate_act(g, u, epi));
            }
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const int n = n0 + 32 * j + nl;
                if (n >= N) continue;
                if (part) part[((size_t)split * M + m) * N + n] = acc[j][i];
                else mats.out[0][(size_t)m * N + n] = __float2half(acc[j][i]);
            }
        }
    }
}

}  // namespace imh_wq
