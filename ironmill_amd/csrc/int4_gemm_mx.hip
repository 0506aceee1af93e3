// int4_gemm_mx.hip -- the INT4-affine (group 128) prefill GEMM with bf16 or
// fp8-e4m3 matrix-core operands (superblock_matmul_int4, affine_matmul.metal:
// 10-152, at the bf16 / fp8 precisions of the prefill workload):
//
//     C[m][n] = out( sum_g s[n][g] * sum_{k in g} a[m][k] * (q[n][k] - z[n][g]) ),  f32 accumulate
//
// with a = x / awq rounded once to the operand type (bf16, or e4m3 for the
// fp8 variant) and C rounded to bf16.  The weights are never rounded: the
// codes enter the matrix cores as exact small integers and the group's
// zero-point and scale are applied in f32 to the group's partial sums.
//
// MI355X design (not the Metal kernel's structure):
//  * A -- the activation -- goes through LDS; B -- the INT4 weights -- goes
//    straight from memory into registers in the MFMA operand layout (lane =
//    weight column + 32 x K half, two 16-byte loads per lane per group and
//    32-column fragment) and is expanded there, so a workgroup's weights
//    never touch LDS and each is read once per workgroup.
//  * bf16: a code q beside the bf16 exponent byte 0x43 is the bf16 value 128 + q
//    exactly (a shift and one and-or per two codes); the MFMA gives sum a (128 + q) and the group's correction subtracts (128 + z) sum a,
//    with sum a the row's group sum of the rounded operand (exact products,
//    f32 sums).  fp8: the code byte itself, read as e4m3, is q * 2^-9 exactly
//    (subnormals and the first binade), the matrix core's block scale 2^9
//    restores q, and the correction subtracts z sum a.  The correction is one more
//    matrix-core product per tile and group (the row sum split into three
//    exact bf16 pieces, against -128 and -z as two; the last of the group's bf16
//    products), so the fold of a group is one multiply-add.
//  * a prep kernel writes the operand rows (x / awq rounded, each 8-element
//    chunk in the slot order the code unpack produces) and their group sums.
//  * the 32 x 32 matrix-core shapes (v_mfma_f32_32x32x16_bf16,
//    v_mfma_scale_f32_32x32x64_f8f6f4): measured on the MI355X they sustain
//    ~2.3 / ~4.9 PFLOP/s where the 16 x 16 bf16 shape stops at ~1.7.
//  * the frame of wq_gemm.h, which says why: four waves of 64 rows x 64
//    columns, A in LDS in operand order, double-buffered by group with one
//    barrier per group; buffer resources with scalar group offsets and LDS
//    immediates, so that the vector unit does little but expand codes and fold
//    sums; loads held at their k step by scheduling barriers; scales and
//    zero-points from a transposed copy that the prep launch writes.  The row
//    sums' three pieces are formed once per group and row by the thread that
//    stages them, not by every wave.
//  * K is split over workgroups when the tile grid leaves workgroup slots (two
//    per CU) idle and a model of the dispatch says the split pays for its
//    partials; the f32 partials are summed in split order by a second kernel
//    (deterministic).
// Measured (us, AWQ, with the prep launch; before: row-major LDS rows, 64-bit
// addresses and in-place scale reads): bf16 M = 2048 K 2560 -> N 9728 126 -> 122,
// M = 1024 K 9728 -> N 2560 88 -> 79, M = 9 19.9 -> 16.9; fp8 M = 509 K 9728 ->
// N 2560 49.5 -> 43.1, M = 1024 77.7 -> 64.3.  At M = 2048 what is left is the
// matrix cores at their sustained clock (104 us with expansion and fold taken
// out) and the 2.4 rounds of tiles.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <string>

#include "dpp_reduce.h"
#include "imh_internal.h"
#include "wq_gemm.h"

namespace {

typedef int i32x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

using namespace imh_wq;

constexpr int kCols = 256;       // columns per workgroup, 64 per wave
constexpr float kE4M3Max = 448.0f;

enum Prec : int { PREC_BF16 = 1, PREC_FP8 = 2 };

// fp8 B operand: a code byte q (0..15) read as OCP E4M3 is q * 2^-9 exactly
// (0..7 are the subnormals m * 2^-9, 8..15 the first binade 2^-6 (1 + m / 8));
// the matrix core's E8M0 block scale 2^9 (exponent 127 + 9) restores q.
constexpr uint32_t kScaleCodesE8m0 = 0x88888888u;
constexpr uint32_t kScaleOneE8m0 = 0x7F7F7F7Fu;

// the column constants of a group: scale f32, and -z as two bf16 halves whose
// sum it is exactly (an f16 has 11 significant bits, a bf16 8)
__device__ __forceinline__ u32x2_t mx_consts(uint16_t s, uint16_t z) {
    const float nz = -(float)__builtin_bit_cast(_Float16, z);
    const __bf16 c0 = (__bf16)nz;
    const __bf16 c1 = (__bf16)(nz - (float)c0);
    return (u32x2_t){__builtin_bit_cast(uint32_t, (float)__builtin_bit_cast(_Float16, s)),
                     (uint32_t)__builtin_bit_cast(uint16_t, c0) | (uint32_t)__builtin_bit_cast(uint16_t, c1) << 16};
}

// Workgroups below ablocks: chunk c (8 elements) of the rows: a = x / awq (no
// awq: x) rounded to the operand type, stored in the order the code expansion
// yields (bf16 {0, 4, 1, 5, 2, 6, 3, 7}, fp8 {0, 2, 4, 6, 1, 3, 5, 7}); the 16
// chunks of a group (16 consecutive lanes) sum their rounded values into
// gsum[m][g].  The others transpose 64 columns x 16 groups of the scales and
// zero-points into szt[group][column].
template <int P>
__global__ void __launch_bounds__(256) gemm_mx_prep_kernel(const __bf16 *__restrict__ x,
                                                           const __half *__restrict__ awq,
                                                           uint8_t *__restrict__ aop, float *__restrict__ gsum,
                                                           size_t chunks, int K, int ablocks,
                                                           const uint16_t *__restrict__ scales,
                                                           const uint16_t *__restrict__ zeros,
                                                           u32x2_t *__restrict__ szt, int N) {
    if ((int)blockIdx.x >= ablocks) {
        const int G = K / kGS, gblk = (G + 15) / 16, blk = (int)blockIdx.x - ablocks;
        const int n = (blk / gblk) * 64 + (int)(threadIdx.x & 63);
        const int g0 = (blk % gblk) * 16 + (int)(threadIdx.x >> 6) * 4;
        if (n >= N) return;
        uint16_t sv[4], zv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const size_t at = (size_t)n * G + min(g0 + i, G - 1);
            sv[i] = scales[at];
            zv[i] = zeros[at];
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (g0 + i < G) szt[(size_t)(g0 + i) * N + n] = mx_consts(sv[i], zv[i]);
        return;
    }
    const size_t cr = (size_t)blockIdx.x * 256 + threadIdx.x;
    const bool live = cr < chunks;
    const size_t ca = live ? cr : 0;
    const int cpr = K / 8;
    const size_t m = ca / cpr;
    const int c = (int)(ca - m * cpr);
    const size_t off = ca * 8;
    const u32x4_t xv = *reinterpret_cast<const u32x4_t *>(x + off);
    const __bf16 *xb = reinterpret_cast<const __bf16 *>(&xv);
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = (float)xb[i];
    if (awq) {
        const u32x4_t wv = *reinterpret_cast<const u32x4_t *>(awq + (size_t)c * 8);
        const _Float16 *wh = reinterpret_cast<const _Float16 *>(&wv);
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = v[i] / (float)wh[i];
    }
    constexpr int kSlot4[8] = {0, 4, 1, 5, 2, 6, 3, 7}, kSlot8[8] = {0, 2, 4, 6, 1, 3, 5, 7};
    float sum = 0.0f;
    if (P == PREC_BF16) {
        bf16x8_t o;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            o[i] = (__bf16)v[kSlot4[i]];
            sum += (float)o[i];
        }
        if (live) *reinterpret_cast<bf16x8_t *>(aop + off * 2) = o;
    } else {
        uint32_t w[2];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float e[4];
#pragma unroll
            for (int i = 0; i < 4; i++) e[i] = fminf(fmaxf(v[kSlot8[4 * h + i]], -kE4M3Max), kE4M3Max);
            uint32_t p = __builtin_amdgcn_cvt_pk_fp8_f32(e[0], e[1], 0, false);
            p = __builtin_amdgcn_cvt_pk_fp8_f32(e[2], e[3], p, true);
            w[h] = p;
            // the rounded values, back from the encoding
            const float2_t r0 = __builtin_amdgcn_cvt_pk_f32_fp8(p, false);
            const float2_t r1 = __builtin_amdgcn_cvt_pk_f32_fp8(p, true);
            sum += r0[0];
            sum += r0[1];
            sum += r1[0];
            sum += r1[1];
        }
        if (live) *reinterpret_cast<uint2 *>(aop + off) = make_uint2(w[0], w[1]);
    }
    sum = imh_dpp::row16_sum(sum);
    if (live && (threadIdx.x & 15) == 0) gsum[(size_t)m * (K / kGS) + (size_t)c / 16] = sum;
}

// grid (tiles_m * tiles_n * splits), block 256; tile (mt, nt, split) from
// tile_of.  Split z covers groups [z * per, min((z + 1) * per, G)).  Without a
// split C is stored as bf16; with one the f32 partials go to part[z][M][N].
//
// Operand layouts of the 32 x 32 MFMAs (lane l: n or m = l & 31, h = l >> 5):
//   bf16 32x32x16, k step s (0..7) of a group: lane (n, h) holds the 8 codes
//     [64 h + 8 s, +8) of column n -- dword s of the 32 code bytes
//     [32 h, 32 h + 32) of the group row -- and A lane (m, h) the operand
//     chunk 8 h + s of row m;
//   fp8 32x32x64, k step t (0..1): lane (n, h) the 32 codes [64 t + 32 h, +32)
//     (code bytes [32 t + 16 h, +16)), A lane (m, h) the 32 operand bytes at
//     64 t + 32 h of row m (chunks 4 t + 2 h, + 1);
//   D: lane l, value i: row 8 (i >> 2) + 4 h + (i & 3), column l & 31.
// LDS: block (row / 32, k step) of 64 lanes x 16 bytes -- fp8: (row / 32, k
// step, half of the 32 bytes) -- padded by 16 bytes.
template <int P, int MI, bool SZT>
__global__ void __launch_bounds__(kThreads, 2) gemm_mx_kernel(
    const uint8_t *__restrict__ aop, const float *__restrict__ gsum, const uint8_t *__restrict__ wdata,
    const uint16_t *__restrict__ scales, const uint16_t *__restrict__ zeros, const u32x2_t *__restrict__ szt,
    __bf16 *__restrict__ out, float *__restrict__ part, int M, int N, int K, int per, TileOrder order) {
    constexpr int BM = 32 * MI;
    constexpr int EB = P == PREC_BF16 ? 2 : 1;     // operand bytes per element
    constexpr int CPR = kGS * EB / 16;             // 16-byte chunks of a row's group
    constexpr int NBLK = CPR / 2;                  // LDS blocks per 32 rows
    constexpr int RPP = kThreads / CPR;            // rows staged per pass
    constexpr int ACH = BM / RPP;                  // chunks per thread and group
    __shared__ __attribute__((aligned(16))) uint8_t As[2][MI * NBLK * kBlk];
    __shared__ __attribute__((aligned(16))) u32x4_t Cs[2][BM];   // row sums in three bf16 pieces

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int nl = lane & 31, h = lane >> 5;
    int mt, nt, split;
    tile_of(order, mt, nt, split);
    const int m0 = mt * BM;
    const int nb = nt * kCols;
    const int n0 = nb + wave * 64;
    const int G = K / kGS;
    const int g_begin = split * per;
    const int g_end = min(g_begin + per, G);

    const int row_bytes = K / 2;
    const int cols = min(kCols, N - nb);
    const __amdgpu_buffer_rsrc_t w_r = __builtin_amdgcn_make_buffer_rsrc((void *)(wdata + (size_t)nb * row_bytes), 0,
                                                                         cols * row_bytes, kRsrcWord3);
    __amdgpu_buffer_rsrc_t s_r, z_r;
    if (SZT) {
        s_r = z_r = __builtin_amdgcn_make_buffer_rsrc((void *)(szt + nb), 0,
                                                      (int)(((size_t)G * N - nb) * sizeof(u32x2_t)), kRsrcWord3);
    } else {
        s_r = __builtin_amdgcn_make_buffer_rsrc((void *)(scales + (size_t)nb * G), 0, cols * G * 2, kRsrcWord3);
        z_r = __builtin_amdgcn_make_buffer_rsrc((void *)(zeros + (size_t)nb * G), 0, cols * G * 2, kRsrcWord3);
    }
    int bvo[2], svo[2];
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = min(n0 + 32 * j + nl, N - 1) - nb;
        bvo[j] = n * row_bytes + (P == PREC_BF16 ? 32 : 16) * h;
        svo[j] = SZT ? n * (int)sizeof(u32x2_t) : n * G * 2;
    }
    struct BRegs {
        u32x4_t w[2][2];
    };
    auto load_b = [&](int g, BRegs &b) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i = 0; i < 2; i++)
                b.w[j][i] = __builtin_bit_cast(
                    u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(w_r, bvo[j] + i * (P == PREC_BF16 ? 16 : 32), g * 64, 0));
    };
    auto load_c = [&](int g, u32x2_t *c) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; j++) {
            if (SZT) {
                c[j] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(
                                                       s_r, svo[j], g * N * (int)sizeof(u32x2_t), 0));
            } else {
                c[j][0] = __builtin_amdgcn_raw_buffer_load_b16(s_r, svo[j], g * 2, 0);
                c[j][1] = __builtin_amdgcn_raw_buffer_load_b16(z_r, svo[j], g * 2, 0);
            }
        }
    };
    // A: pass i of a thread is row tid / CPR, chunk tid % CPR of the i-th slab of
    // RPP rows; rows past M read as zeros
    const int arows = min(BM, M - m0);
    __amdgpu_buffer_rsrc_t a_r[ACH];
#pragma unroll
    for (int i = 0; i < ACH; i++) a_r[i] = row_slab(aop, m0 + RPP * i, RPP, M, K * EB);
    const __amdgpu_buffer_rsrc_t r_r =
        __builtin_amdgcn_make_buffer_rsrc((void *)(gsum + (size_t)m0 * G), 0, arows * G * 4, kRsrcWord3);
    const int ar0 = tid / CPR, ac = tid % CPR;
    const int avo = ar0 * K * EB + ac * 16;
    const int ablk = P == PREC_BF16 ? (ac & 7) : 2 * (ac >> 2) + (ac & 1);
    const int ah = P == PREC_BF16 ? ac >> 3 : (ac >> 1) & 1;
    const int a_lds = ablk * kBlk + (ar0 + 32 * ah) * 16;
    const int rvo = (tid & (BM - 1)) * G * 4;
    auto load_a = [&](int g, u32x4_t *ar, float &rs) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ACH; i++)
            ar[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_r[i], avo, g * kGS * EB, 0));
        rs = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_r, rvo, g * 4, 0));
    };
    auto store_a = [&](int buf, const u32x4_t *ar, float rs) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < ACH; i++) {
            const int r = RPP * i;   // of the thread's rows, the part that is the same for all
            *reinterpret_cast<u32x4_t *>(&As[buf][a_lds + (r >> 5) * NBLK * kBlk + (r & 31) * 16]) = ar[i];
        }
        // rs = r0 + r1 + r2 exactly, in bf16 (the same value from each wave)
        const __bf16 r0 = (__bf16)rs;
        const float e1 = rs - (float)r0;
        const __bf16 r1 = (__bf16)e1;
        const __bf16 r2 = (__bf16)(e1 - (float)r1);
        auto bits = [](__bf16 v) { return (uint32_t)__builtin_bit_cast(uint16_t, v); };
        Cs[buf][tid & (BM - 1)] =
            (u32x4_t){bits(r0) | bits(r1) << 16, bits(r2) | bits(r0) << 16, bits(r1) | bits(r2) << 16, 0u};
    };

    float16_t acc[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[mi][j][i] = 0.0f;

    // in registers, so that each and-or is one instruction
    uint32_t m_lo, exp128;
    asm("s_mov_b32 %0, 0x000f000f" : "=s"(m_lo));
    asm("v_mov_b32 %0, 0x43004300" : "=v"(exp128));

    // One group from LDS buffer buf: the MFMAs of the tiles over the group's k
    // steps (hook(st): the next group's loads at k step st), the correction -(128
    // + z) rowsum (fp8: -z rowsum) as one more product of exact bf16 pieces (A lane
    // (m, h): the row sum's three pieces twice, B lane (n, 0): -128 (fp8: 0) three
    // times, then the first half of -z, lane (n, 1): its second half three times,
    // then zeros), then the fold with the scale of the lane's column.
    constexpr uint32_t kOffset = P == PREC_BF16 ? 0xC300C300u : 0u;   // -128 twice
    // byte selectors of B's words from the halves of -z (bytes 4-7) and kOffset (0-3)
    const uint32_t cs0 = h ? 0x07060706u : 0x03020100u, cs1 = h ? 0x0C0C0706u : 0x05040100u,
                   cs2 = h ? 0x0C0C0C0Cu : 0x05040504u;
    auto compute = [&](int buf, const BRegs &b, const u32x2_t *cc, auto &&hook) __attribute__((always_inline)) {
        float sc[2];
        bf16x8_t cb[2];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const u32x2_t c = SZT ? cc[j] : mx_consts((uint16_t)cc[j][0], (uint16_t)cc[j][1]);
            const uint32_t cs = c[0], cz = c[1];   // scalars: a bit cast of a vector element takes element 0
            sc[j] = __builtin_bit_cast(float, cs);
            cb[j] = __builtin_bit_cast(bf16x8_t, (u32x4_t){__builtin_amdgcn_perm(cz, kOffset, cs0),
                                                           __builtin_amdgcn_perm(cz, kOffset, cs1),
                                                           __builtin_amdgcn_perm(cz, kOffset, cs2), 0u});
        }
        const uint8_t *ab = &As[buf][lane * 16];
        bf16x8_t ca[MI];
        auto read_c = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int mi = 0; mi < MI; mi++) ca[mi] = __builtin_bit_cast(bf16x8_t, Cs[buf][32 * mi + nl]);
        };
        const float16_t zero16 = {};
        if constexpr (P == PREC_BF16) {
            bf16x8_t af[2][MI], bf[2][2];
            auto read_a = [&](int st) __attribute__((always_inline)) {
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
                    af[st & 1][mi] = *reinterpret_cast<const bf16x8_t *>(ab + (mi * NBLK + st) * kBlk);
            };
            // 8 codes -> bf16 128 + q in slot order {0, 4, 1, 5, 2, 6, 3, 7}
            auto expand = [&](int st) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    const uint32_t w = b.w[j][st >> 2][st & 3];
                    bf[st & 1][j] = __builtin_bit_cast(
                        bf16x8_t, (u32x4_t){(w & m_lo) | exp128, ((w >> 4) & m_lo) | exp128, ((w >> 8) & m_lo) | exp128,
                                            ((w >> 12) & m_lo) | exp128});
                }
            };
            float16_t gg[MI][2];
            read_a(0);
            expand(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int st = 0; st < 8; st++) {
                if (st < 7) read_a(st + 1);
                else read_c();
                hook(st);
                if (st < 7) expand(st + 1);
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        gg[mi][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[st & 1][mi], bf[st & 1][j],
                                                                            st == 0 ? zero16 : gg[mi][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    gg[mi][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca[mi], cb[j], gg[mi][j], 0, 0, 0);
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[mi][j][i] = __builtin_fmaf(sc[j], gg[mi][j][i], acc[mi][j][i]);
        } else {
            i32x8_t af[2][MI], bf[2][2];
            auto read_a = [&](int t) __attribute__((always_inline)) {
#pragma unroll
                for (int mi = 0; mi < MI; mi++) {
                    const u32x4_t a0 = *reinterpret_cast<const u32x4_t *>(ab + (mi * NBLK + 2 * t) * kBlk);
                    const u32x4_t a1 = *reinterpret_cast<const u32x4_t *>(ab + (mi * NBLK + 2 * t + 1) * kBlk);
                    af[t][mi] = (i32x8_t){(int)a0[0], (int)a0[1], (int)a0[2], (int)a0[3],
                                          (int)a1[0], (int)a1[1], (int)a1[2], (int)a1[3]};
                }
            };
            // code dword d = codes 8 d .. 8 d + 7 -> the even codes' bytes, then the odd
            auto expand = [&](int t) __attribute__((always_inline)) {
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int d = 0; d < 4; d++) {
                        const uint32_t w = b.w[j][t][d];
                        bf[t][j][2 * d] = (int)(w & 0x0F0F0F0Fu);
                        bf[t][j][2 * d + 1] = (int)((w >> 4) & 0x0F0F0F0Fu);
                    }
            };
            float16_t gg[MI][2];
            read_c();
            read_a(0);
            expand(0);
            __builtin_amdgcn_sched_barrier(0);
            hook(0);
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int j = 0; j < 2; j++)
                    gg[mi][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ca[mi], cb[j], zero16, 0, 0, 0);
            read_a(1);
            expand(1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2; t++) {
                hook(t + 1);
                // formats 0 / 0: e4m3 x e4m3; A scale x1, B scale x 2^9
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
#pragma unroll
                    for (int j = 0; j < 2; j++)
                        gg[mi][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
                            af[t][mi], bf[t][j], gg[mi][j], 0, 0, 0, kScaleOneE8m0, 0, kScaleCodesE8m0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int i = 0; i < 16; i++) acc[mi][j][i] = __builtin_fmaf(sc[j], gg[mi][j][i], acc[mi][j][i]);
        }
    };

    u32x4_t ar[ACH];
    float rs = 0.0f;
    BRegs b0, b1;
    u32x2_t c0[2], c1[2];
    if (g_begin < g_end) {
        load_b(g_begin, b0);
        load_c(g_begin, c0);
        load_a(g_begin, ar, rs);
        store_a(0, ar, rs);
        __syncthreads();
    }
    // the next group's loads are unconditional (past the last group the last
    // one is loaded again), so no wait for the current set has to cover them
    auto step = [&](int g, int buf, const BRegs &cur, const u32x2_t *cc, BRegs &nxt,
                    u32x2_t *nc) __attribute__((always_inline)) {
        const int gn = min(g + 1, g_end - 1);
        compute(buf, cur, cc, [&](int st) __attribute__((always_inline)) {
            if (st == 0) load_a(gn, ar, rs);
            if (st == 1) {
                load_b(gn, nxt);
                load_c(gn, nc);
            }
        });
        store_a(buf ^ 1, ar, rs);
        __syncthreads();
    };
    for (int g = g_begin; g < g_end; g += 2) {
        step(g, 0, b0, c0, b1, c1);
        if (g + 1 >= g_end) break;
        step(g + 1, 1, b1, c1, b0, c0);
    }

    // D of tile (mi, j): lane holds rows 32 mi + 8 (i >> 2) + 4 h + (i & 3), column 32 j + nl
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int n = n0 + 32 * j + nl;
        if (n >= N) continue;
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = m0 + 32 * mi + 8 * (i >> 2) + 4 * h + (i & 3);
                if (m >= M) continue;
                if (part) part[((size_t)split * M + m) * N + n] = acc[mi][j][i];
                else out[(size_t)m * N + n] = (__bf16)acc[mi][j][i];
            }
    }
}

// Sums the split partials in split order: grid ceil(M * N / 256), block 256.
__global__ void __launch_bounds__(256) gemm_mx_reduce_kernel(const float *__restrict__ part, int splits, size_t count,
                                                             __bf16 *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    float s = part[i];
    for (int z = 1; z < splits; z++) s += part[(size_t)z * count + i];
    out[i] = (__bf16)s;
}

int check_gemm_weight(const imh_affine_int4_weight *w, const char *who) {
    if (!w || !w->data || !w->scales || !w->zeros)
        return imh::fail(IMH_EINVAL, std::string(who) + ": weight or one of its arrays is NULL");
    if (w->group_size != kGS)
        return imh::fail(IMH_EUNSUPPORTED, std::string(who) + ": group_size " + std::to_string(w->group_size) +
                                               " not supported (built for 128)");
    if (w->n == 0 || w->k == 0 || w->k % kGS)
        return imh::fail(IMH_EUNSUPPORTED, std::string(who) + ": k must be a non-zero multiple of 128, n non-zero");
    if ((reinterpret_cast<uintptr_t>(w->data) & 15) != 0)
        return imh::fail(IMH_EINVAL, std::string(who) + ": weight data must be 16-byte aligned");
    return IMH_OK;
}

// K splits for a grid of `tiles` output tiles (fewer than the slots, two
// per CU).  Workgroups of a launch are dispatched as slots free up, and each
// is taken to cost the same per group: 2.4 us bf16 / 1.9 us fp8 with two per
// CU, 0.9 of that alone on its CU, and the same for 32-row tiles.  These were
// fitted to the tiling before this one (traced now: 2.7 bf16, 2.5 fp8 for 64
// rows), and not to the 32-row tiles.  So a grid of W workgroups runs full
// rounds of two per CU, then its remainder (one per CU where it fits); a
// split adds the partials' round trip (written during the GEMM, read back by
// the reduce launch at ~4.5 TB/s plus ~2 us).  Measured against the earlier
// rule (as many splits as fill two per CU, rounded up): K 2560 -> N 9728 at
// M = 512 (304 tiles) 1 split instead of 2, 65 -> 57 us (bf16); K 9728 ->
// N 2560 at M = 512 (80 tiles) 6 instead of 7, 72 -> 60 us; at M = 2048
// (320 tiles) 1 split took 200 us against 186 with 2 and 185-191 with 3.
// At least 4 groups per split.
double grid_us(long long W, int per, int cus, double g2) {
    double us = 0.0;
    for (; W > 2 * cus; W -= 2 * cus) us += per * g2;
    return us + per * (W > cus ? g2 : 0.9 * g2);
}
int gemm_splits(int tiles, int G, int M, int N, int cus, int P) {
    const double g2 = P == PREC_BF16 ? 2.4 : 1.9;
    int best = 1;
    double best_us = grid_us(tiles, G, cus, g2);
    for (int s = 2; s <= G / 4; s++) {
        const int per = (G + s - 1) / s;
        if ((G + per - 1) / per != s) continue;
        const double us = grid_us((long long)tiles * s, per, cus, g2) +
                          ((double)s * M * N * 4 + (double)M * N * 2) / 4.5e6 + 2.0;
        if (us < best_us * 0.98) {   // a split must win clearly
            best_us = us;
            best = s;
        }
    }
    return best;
}

}  // namespace

extern "C" {

int imh_affine_gemm_int4(imh_stream *stream, const void *x, uint32_t M, const imh_affine_int4_weight *w, void *y,
                         int precision) {
    const char *who = "imh_affine_gemm_int4";
    if (!stream || !x || !y) return imh::fail(IMH_EINVAL, std::string(who) + ": NULL argument");
    int rc = check_gemm_weight(w, who);
    if (rc) return rc;
    if (precision == IMH_GEMM_F16) {
        // the f16 path is the projection op (matvec or f16 GEMM)
        return imh_encode_affine_projection_int4(stream, static_cast<const uint16_t *>(x), M, w,
                                                 static_cast<uint16_t *>(y));
    }
    if (precision != IMH_GEMM_BF16 && precision != IMH_GEMM_FP8_E4M3)
        return imh::fail(IMH_EINVAL, std::string(who) + ": unknown precision " + std::to_string(precision));
    if ((reinterpret_cast<uintptr_t>(x) & 15) || (w->awq_scales && (reinterpret_cast<uintptr_t>(w->awq_scales) & 15)))
        return imh::fail(IMH_EINVAL, std::string(who) + ": x and awq_scales must be 16-byte aligned");
    if (M == 0) return IMH_OK;
    if (M > 65535u) return imh::fail(IMH_EINVAL, std::string(who) + ": M above 65535");
    rc = imh::use_device(stream->dev);
    if (rc) return rc;
    const int N = (int)w->n, K = (int)w->k, G = K / kGS;
    const int P = precision == IMH_GEMM_BF16 ? PREC_BF16 : PREC_FP8;
    const int eb = P == PREC_BF16 ? 2 : 1;
    const int cus = stream->dev->props.multiProcessorCount;
    const int bm = M <= 32 ? 32 : 64;
    TileOrder order;
    order.tiles_m = ((int)M + bm - 1) / bm;
    order.tiles_n = (N + kCols - 1) / kCols;
    const int tiles = order.tiles_m * order.tiles_n;
    int splits = tiles < 2 * cus ? gemm_splits(tiles, G, (int)M, N, cus, P) : 1;
    int per = (G + splits - 1) / splits;
    splits = (G + per - 1) / per;
    // scratch slot 2: split partials; without room for them (a capture, or no
    // memory) K is not split
    void *part_scr = nullptr;
    if (splits > 1 &&
        !imh::stream_scratch_optional(stream, 2, (size_t)splits * M * N * sizeof(float), &part_scr)) {
        splits = 1;
        per = G;
    }
    float *part = splits > 1 ? static_cast<float *>(part_scr) : nullptr;
    order.splits = splits;
    // band: the largest divisor of tiles_m that is at most tiles_m / 8 (so
    // each XCD gets about one band), at least 1
    order.band = 1;
    for (int b = std::max(1, order.tiles_m / 8); b >= 1; b--)
        if (order.tiles_m % b == 0) {
            order.band = b;
            break;
        }
    // scratch slot 0: operand rows, group sums and, where it has room, the
    // transposed column constants (a stream capturing with the scratch of the
    // first two reads scales and zero-points in place)
    const size_t a_bytes = ((size_t)M * K * eb + 255) / 256 * 256;
    const size_t gsum_bytes = ((size_t)M * G * sizeof(float) + 255) / 256 * 256;
    const size_t szt_bytes = (size_t)G * N * sizeof(u32x2_t);
    void *scr = nullptr;
    const bool has_szt = szt_bytes < (size_t)INT32_MAX &&
                         imh::stream_scratch_optional(stream, 0, a_bytes + gsum_bytes + szt_bytes, &scr);
    if (!has_szt) {
        rc = imh::stream_scratch(stream, 0, a_bytes + (size_t)M * G * sizeof(float), &scr);
        if (rc) return rc;
    }
    uint8_t *aop = static_cast<uint8_t *>(scr);
    float *gsum = reinterpret_cast<float *>(aop + a_bytes);
    u32x2_t *szt = reinterpret_cast<u32x2_t *>(aop + a_bytes + gsum_bytes);
    const __bf16 *xb = static_cast<const __bf16 *>(x);
    const __half *awq = reinterpret_cast<const __half *>(w->awq_scales);
    const size_t chunks = (size_t)M * K / 8;
    const int ablocks = (int)((chunks + 255) / 256);
    const dim3 pgrid((unsigned)(ablocks + (has_szt ? ((N + 63) / 64) * ((G + 15) / 16) : 0)));
    const dim3 grid((unsigned)(tiles * splits));
    __bf16 *out = static_cast<__bf16 *>(y);
#define IMH_MX(PR, MI, SZ)                                                                                              \
    hipLaunchKernelGGL((gemm_mx_kernel<PR, MI, SZ>), grid, dim3(kThreads), 0, stream->stream, aop, gsum, w->data, w->scales, \
                       w->zeros, szt, out, part, (int)M, N, K, per, order)
#define IMH_MX_ALL(PR)                                                                                               \
    hipLaunchKernelGGL(gemm_mx_prep_kernel<PR>, pgrid, dim3(256), 0, stream->stream, xb, awq, aop, gsum, chunks, K,   \
                       ablocks, w->scales, w->zeros, szt, N);                                                        \
    IMH_HIP(hipGetLastError());                                                                                      \
    if (has_szt) {                                                                                                   \
        if (bm == 32) IMH_MX(PR, 1, true);                                                                           \
        else IMH_MX(PR, 2, true);                                                                                    \
    } else {                                                                                                         \
        if (bm == 32) IMH_MX(PR, 1, false);                                                                          \
        else IMH_MX(PR, 2, false);                                                                                   \
    }
    if (P == PREC_BF16) {
        IMH_MX_ALL(PREC_BF16)
    } else {
        IMH_MX_ALL(PREC_FP8)
    }
#undef IMH_MX_ALL
#undef IMH_MX
    IMH_HIP(hipGetLastError());
    if (splits > 1) {
        const size_t count = (size_t)M * N;
        hipLaunchKernelGGL(gemm_mx_reduce_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream->stream,
                           part, splits, count, out);
        IMH_HIP(hipGetLastError());
    }
    return IMH_OK;
}

}  // extern "C"
