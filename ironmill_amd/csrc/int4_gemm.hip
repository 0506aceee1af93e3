// int4_gemm.hip -- the f16 prefill GEMMs over INT4 and INT8 weights (group 128)
// and the residual-norm rows kernel
// (superblock_matmul_int4, affine_matmul.metal:10-152, reached from
// encode_projection at token_count > 1, projection.rs:227-312; the INT8 weights
// of superblock_matvec_int8, affine_matvec.metal:123-189, at prefill sizes).
//
//     C[m][n] = f16( sum_g s[n][g] * sum_{k in g} (x[m][k] / awq[k]) * (q[n][k] - z[n][g]) ),  f32 accumulate
//
// No weight is rounded and x / awq keeps ~22 bits (f16 hi + lo).  The
// reference's prefill kernel instead rounds both the dequantized weight and a /
// awq to f16 (affine_matmul B dequant -> half, A rows = half(a / awq)), which
// costs several fp16 steps against the CPU path where terms cancel.  The
// kernel and its design are in wq_gemm.h; this file holds the launches, the K
// split and the split's reduction (f32 partials summed in split order by a
// second kernel: deterministic).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <string>

#include "imh_internal.h"
#include "int4_gemm.h"
#include "wq_gemm.h"

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

using namespace imh_wq;

constexpr int kRowsMax = 32;   // rows up to which the one-launch kernel runs

// Sum the split partials in split order, then store (or, for a gate/up pair,
// apply the activation): grid ceil(M*N / 256), block 256.
__global__ void __launch_bounds__(256) int4_gemm_reduce_kernel(const float *__restrict__ part, int splits,
                                                               int M, int N, int nmat, int epi,
                                                               __half *__restrict__ out0,
                                                               __half *__restrict__ out1) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t count = (size_t)M * N;
    if (i >= count) return;
    const size_t m = i / N, n = i - m * N;
    const size_t stride = (size_t)M * nmat * N;
    float v[2] = {0.0f, 0.0f};
    for (int t = 0; t < nmat; t++) {
        const size_t at = m * nmat * N + (size_t)t * N + n;
        float s = part[at];
        for (int z = 1; z < splits; z++) s += part[(size_t)z * stride + at];
        v[t] = s;
    }
    if (nmat == 2 && epi != GE_STORE) {
        out0[i] = __float2half(gate_act(v[0], v[1], epi));
    } else {
        out0[i] = __float2half(v[0]);
        if (nmat == 2) out1[i] = __float2half(v[1]);
    }
}

// Residual + RMSNorm rows (the prefill path and the 3-8-row decode FFN):
// grid (B), block 256.  residual_out = f16(a + b), normed_out = f16((a + b) *
// rms_inv * gamma).  Thread t takes chunks t, t + 256, ..: the first CPT of
// them are loaded before the reduction and stay in registers (all of them for
// K <= 2048 CPT); chunks past those are read again after it.
template <int CPT>
__global__ void __launch_bounds__(256) resnorm_rows_kernel(const __half *__restrict__ a,
                                                           const __half *__restrict__ b,
                                                           const __half *__restrict__ gamma, float eps,
                                                           __half *__restrict__ residual_out,
                                                           __half *__restrict__ normed_out, int K) {
    __shared__ float red[256];
    __shared__ float rms_s;
    const size_t row = (size_t)blockIdx.x * K;
    const int nchunk = K / 8;
    const int iters = (nchunk + 255) / 256;
    uint4 av[CPT], bv[CPT], gv[CPT];
#pragma unroll
    for (int it = 0; it < CPT; it++) {
        const int c_raw = it * 256 + (int)threadIdx.x;
        const int c = c_raw < nchunk ? c_raw : 0;
        av[it] = *reinterpret_cast<const uint4 *>(a + row + (size_t)c * 8);
        bv[it] = *reinterpret_cast<const uint4 *>(b + row + (size_t)c * 8);
        gv[it] = *reinterpret_cast<const uint4 *>(gamma + (size_t)c * 8);
    }
    float sq = 0.0f;
    auto add_sq = [&](const uint4 &x, const uint4 &y) __attribute__((always_inline)) {
        const _Float16 *ah = reinterpret_cast<const _Float16 *>(&x);
        const _Float16 *bh = reinterpret_cast<const _Float16 *>(&y);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float r = (float)ah[i] + (float)bh[i];
            sq = __builtin_fmaf(r, r, sq);
        }
    };
#pragma unroll
    for (int it = 0; it < CPT; it++)
        if (it * 256 + (int)threadIdx.x < nchunk) add_sq(av[it], bv[it]);
    for (int it = CPT; it < iters; it++) {
        const int c = it * 256 + (int)threadIdx.x;
        if (c < nchunk)
            add_sq(*reinterpret_cast<const uint4 *>(a + row + (size_t)c * 8),
                   *reinterpret_cast<const uint4 *>(b + row + (size_t)c * 8));
    }
    const float rms_inv = imh_int4::block_rms_inv(sq, red, &rms_s, K, eps);
    auto emit = [&](int c, const uint4 &x, const uint4 &y, const uint4 &gw) __attribute__((always_inline)) {
        const size_t off = row + (size_t)c * 8;
        const _Float16 *ah = reinterpret_cast<const _Float16 *>(&x);
        const _Float16 *bh = reinterpret_cast<const _Float16 *>(&y);
        const _Float16 *gh = reinterpret_cast<const _Float16 *>(&gw);
        half8_t res, nrm;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float r = (float)ah[i] + (float)bh[i];
            res[i] = (_Float16)r;
            nrm[i] = (_Float16)(r * rms_inv * (float)gh[i]);
        }
        *reinterpret_cast<half8_t *>(residual_out + off) = res;
        *reinterpret_cast<half8_t *>(normed_out + off) = nrm;
    };
#pragma unroll
    for (int it = 0; it < CPT; it++) {
        const int c = it * 256 + (int)threadIdx.x;
        if (c < nchunk) emit(c, av[it], bv[it], gv[it]);
    }
    for (int it = CPT; it < iters; it++) {
        const int c = it * 256 + (int)threadIdx.x;
        if (c < nchunk)
            emit(c, *reinterpret_cast<const uint4 *>(a + row + (size_t)c * 8),
                 *reinterpret_cast<const uint4 *>(b + row + (size_t)c * 8),
                 *reinterpret_cast<const uint4 *>(gamma + (size_t)c * 8));
    }
}

}  // namespace

namespace imh_int4 {

// K splits of the one-launch kernel, counted in whole blocks of groups (the
// launch then balances the splits by groups: G = 9 at 3 splits gives 3 each, not
// 4, 4 and 1); a round of workgroups (two per CU) costs ~4 us and ~1.05 per
// group, a split ~3 us of reduction and its partials' round trip.  Measured at 12 rows, AWQ,
// 9728 -> 2560: 1 / 2 / 3 / 5 blocks per split 16.1 / 18.9 / 20 / 33 us.
int rows_splits(int M, int N, int K, int nmat, int cus) {
    const int tiles = (N + 256 / nmat - 1) / (256 / nmat), G = K / kGS;
    int best = 1;
    double best_us = 1e30;
    for (int per = kRowsBlock;; per += kRowsBlock) {
        const int sp = (G + per - 1) / per;
        const double us = (double)(((long long)tiles * sp + 2 * cus - 1) / (2 * cus)) * (4.0 + 1.05 * std::min(per, G)) +
                          (sp > 1 ? 3.0 + (double)sp * M * nmat * N * 8 / 4.5e6 : 0.0);
        if (us < best_us) {
            best_us = us;
            best = sp;
        }
        if (sp == 1) break;
    }
    return best;
}

// K splits (whole groups each, at least 4 per split), only as many as keep
// the grid within one round of workgroup slots (two per CU).  Each
// workgroup is taken to cost the same per group (g2 = 2.2 us at two per CU, 0.6
// of that alone on a CU; one value for one plane, two planes and INT8 -- traced,
// two planes take 3.8-4.2 at two per CU, INT8 2.9 alone on its CU), and a split
// adds its partials' round trip (read back by the reduce launch at ~4.5 TB/s plus
// ~2 us).
int gemm_splits(int M, int N, int K, int nmat, int cus) {
    if (M <= kRowsMax) return rows_splits(M, N, K, nmat, cus);
    const int bm = 64;
    const int tiles = ((M + bm - 1) / bm) * ((N + 256 / nmat - 1) / (256 / nmat));
    const int G = K / kGS;
    if (tiles >= 2 * cus || G < 8) return 1;
    constexpr double g2 = 2.2;
    auto grid_us = [&](long long W, int per) {
        double us = 0.0;
        for (; W > 2 * cus; W -= 2 * cus) us += per * g2;
        return us + per * (W > cus ? g2 : 0.6 * g2);
    };
    int best = 1;
    double best_us = grid_us(tiles, G);
    for (int sp = 2; sp <= G / 4 && (long long)tiles * sp <= 2 * cus; sp++) {
        const int per = (G + sp - 1) / sp;
        if ((G + per - 1) / per != sp) continue;
        const double us = grid_us((long long)tiles * sp, per) +
                          ((double)sp * M * nmat * N * 4 + (double)M * nmat * N * 2) / 4.5e6 + 2.0;
        if (us < best_us * 0.98) {
            best_us = us;
            best = sp;
        }
    }
    return best;
}

size_t gemm_workspace_bytes(int M, int N, int K, int nmat, int cus) {
    const int splits = gemm_splits(M, N, K, nmat, cus);
    return splits > 1 ? (size_t)splits * M * nmat * N * sizeof(float) : 0;
}

namespace {

struct Launch {
    const __half *hi, *lo;
    const float *gsum;
    Mats mats;
    const u32x2_t *szt;
    float *part;
    int M, N, K, per, epi;
    TileOrder order;
};

template <int BITS, int NPL, bool DIRECT, bool SZT>
void launch_tile(hipStream_t st, const Launch &L, bool pair) {
    const dim3 grid((unsigned)(L.order.tiles_m * L.order.tiles_n * L.order.splits));
#define IMH_WQ(MI, PAIR)                                                                                          \
    hipLaunchKernelGGL((wq_gemm_kernel<BITS, NPL, MI, PAIR, DIRECT, SZT>), grid, dim3(kThreads), 0, st, L.hi, L.lo, \
                       L.gsum, L.mats, L.szt, L.part, L.M, L.N, L.K, L.per, L.epi, L.order)
    if constexpr (BITS == 4) {
        if (pair) {
            IMH_WQ(2, true);
            return;
        }
    }
    IMH_WQ(2, false);
#undef IMH_WQ
}

// Up to kRowsMax rows: one launch (and the reduction of a split).
template <int BITS>
void launch_rows(hipStream_t st, const Launch &L, const __half *awq, bool pair) {
    const dim3 grid((unsigned)(L.order.tiles_n * L.order.splits));
#define IMH_ROWS(AWQ, PAIR)                                                                                       \
    hipLaunchKernelGGL((wq_rows_kernel<BITS, AWQ, PAIR>), grid, dim3(kThreads), 0, st, L.hi, awq, L.mats, L.part, L.M, \
                       L.N, L.K, L.per, L.epi, L.order.tiles_n)
    if constexpr (BITS == 4) {
        if (pair) {
            if (awq) IMH_ROWS(true, true);
            else IMH_ROWS(false, true);
            return;
        }
    }
    if (awq) IMH_ROWS(true, false);
    else IMH_ROWS(false, false);
#undef IMH_ROWS
}

// The activation planes (with awq or INT8), transposed column constants where
// the scratch has room, the GEMM and, with a split, the reduction.
template <int BITS>
int encode_wq_gemm(imh_stream *s, const __half *x, int M, const Mats &mats, const __half *awq, int N, int K, int nmat,
                   int epi, void *workspace, bool *used) {
    const int cus = s->dev->props.multiProcessorCount;
    const int G = K / kGS;
    int splits = workspace ? gemm_splits(M, N, K, nmat, cus) : 1;
    const int per = (G + splits - 1) / splits;
    splits = (G + per - 1) / per;
    Launch L = {};
    L.hi = x;
    L.mats = mats;
    L.M = M;
    L.N = N;
    L.K = K;
    L.per = per;
    L.epi = epi;
    L.part = splits == 1 ? nullptr : static_cast<float *>(workspace);
    const int bm = 64, tn = 256 / nmat;
    L.order.tiles_m = (M + bm - 1) / bm;
    L.order.tiles_n = (N + tn - 1) / tn;
    L.order.splits = splits;
    // band: the largest divisor of tiles_m that is at most tiles_m / 8 (so
    // each XCD gets about one band), at least 1
    L.order.band = 1;
    for (int b = std::max(1, L.order.tiles_m / 8); b >= 1; b--)
        if (L.order.tiles_m % b == 0) {
            L.order.band = b;
            break;
        }
    const bool pair = nmat == 2;
    if (M <= kRowsMax) {
        launch_rows<BITS>(s->stream, L, awq, pair);
    } else if (BITS == 4 && !awq) {
        launch_tile<4, 1, true, false>(s->stream, L, pair);
    } else {
        const size_t mk = (size_t)M * K;
        const size_t plane_bytes = (mk * 2 * (awq ? 2 : 1) + 255) & ~(size_t)255;
        const size_t gsum_bytes = BITS == 8 ? ((size_t)M * G * sizeof(float) + 255) & ~(size_t)255 : 0;
        const size_t szt_bytes = (size_t)nmat * G * N * sizeof(u32x2_t);
        // the constants' copy is optional for INT4 (a stream capturing with
        // only the planes' scratch, or an index past 32 bits, reads them in place)
        bool szt = szt_bytes < (size_t)INT32_MAX;
        void *scr = nullptr;
        if (BITS == 8 && !szt) return IMH_OK;
        if (szt && !imh::stream_scratch_optional(s, 0, plane_bytes + gsum_bytes + szt_bytes, &scr)) {
            if (BITS == 8) return IMH_OK;
            szt = false;
        }
        if (!szt) {
            const int rc = imh::stream_scratch(s, 0, mk * 2 * sizeof(__half), &scr);
            if (rc) return rc;
        }
        uint8_t *p = static_cast<uint8_t *>(scr);
        __half *hi = reinterpret_cast<__half *>(p), *lo = hi + mk;
        float *gsum = reinterpret_cast<float *>(p + plane_bytes);
        u32x2_t *sz = reinterpret_cast<u32x2_t *>(p + plane_bytes + gsum_bytes);
        const size_t chunks = mk / 8;
        const int ablocks = (int)((chunks + 255) / 256);
        const int sz_per_mat = ((N + 63) / 64) * ((G + 15) / 16);
        hipLaunchKernelGGL(prep_kernel<BITS>, dim3((unsigned)(ablocks + (szt ? nmat * sz_per_mat : 0))), dim3(256), 0,
                           s->stream, x, awq, hi, lo, gsum, chunks, K, ablocks, mats, sz, N, sz_per_mat);
        IMH_HIP(hipGetLastError());
        L.hi = hi;
        L.lo = lo;
        L.gsum = gsum;
        L.szt = sz;
        if constexpr (BITS == 4) {
            if (szt) launch_tile<4, 2, false, true>(s->stream, L, pair);
            else launch_tile<4, 2, false, false>(s->stream, L, pair);
        } else {
            if (awq) launch_tile<8, 2, false, true>(s->stream, L, false);
            else launch_tile<8, 1, false, true>(s->stream, L, false);
        }
    }
    IMH_HIP(hipGetLastError());
    if (splits > 1) {
        const size_t count = (size_t)M * N;
        hipLaunchKernelGGL(int4_gemm_reduce_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, s->stream,
                           L.part, splits, M, N, nmat, epi, mats.out[0], mats.out[1]);
        IMH_HIP(hipGetLastError());
    }
    *used = true;
    return IMH_OK;
}

}  // namespace

int encode_gemm(imh_stream *s, const __half *x, int M, const imh_affine_int4_weight *w0,
                const imh_affine_int4_weight *w1, int epi, __half *y0, __half *y1, void *workspace) {
    Mats mats = {};
    const imh_affine_int4_weight *ws[2] = {w0, w1 ? w1 : w0};
    for (int i = 0; i < 2; i++) {
        mats.data[i] = ws[i]->data;
        mats.scales[i] = reinterpret_cast<const __half *>(ws[i]->scales);
        mats.zeros[i] = reinterpret_cast<const __half *>(ws[i]->zeros);
    }
    mats.out[0] = y0;
    mats.out[1] = y1;
    const int ge = epi == 2 ? GE_SILU : epi == 3 ? GE_GELU : GE_STORE;
    // both matrices of a pair divide x by the first one's awq scales
    bool used = false;
    return encode_wq_gemm<4>(s, x, M, mats, reinterpret_cast<const __half *>(w0->awq_scales), (int)w0->n, (int)w0->k,
                             w1 ? 2 : 1, ge, workspace, &used);
}

int encode_gemm_int8(imh_stream *s, const __half *x, int M, const imh_affine_int8_weight *w, __half *y, bool *used) {
    *used = false;
    const int N = (int)w->n, K = (int)w->k;
    const size_t ws_bytes = gemm_workspace_bytes(M, N, K, 1, s->dev->props.multiProcessorCount);
    void *ws = nullptr;
    if (ws_bytes && !imh::stream_scratch_optional(s, 2, ws_bytes, &ws)) return IMH_OK;
    Mats mats = {};
    mats.data[0] = mats.data[1] = w->data;
    mats.scales[0] = mats.scales[1] = reinterpret_cast<const __half *>(w->scales);
    mats.zeros[0] = mats.zeros[1] = reinterpret_cast<const __half *>(w->zeros);
    mats.out[0] = y;
    return encode_wq_gemm<8>(s, x, M, mats, reinterpret_cast<const __half *>(w->awq_scales), N, K, 1, GE_STORE, ws, used);
}

int encode_resnorm_rows(imh_stream *s, const __half *a, const __half *b, const __half *gamma, float eps,
                        __half *residual_out, __half *normed_out, int B, int K) {
    const int cpt = resnorm_cpt(K);
    auto kern = cpt == 1 ? resnorm_rows_kernel<1>
                : cpt == 2 ? resnorm_rows_kernel<2>
                : cpt == 4 ? resnorm_rows_kernel<4>
                           : resnorm_rows_kernel<8>;
    hipLaunchKernelGGL(kern, dim3(B), dim3(256), 0, s->stream, a, b, gamma, eps, residual_out, normed_out, K);
    IMH_HIP(hipGetLastError());
    return IMH_OK;
}

}  // namespace imh_int4
