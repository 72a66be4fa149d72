// lut_fc.hip -- fully connected LUT layer kernels for gfx950 (CDNA4, wave64).
//
// Data layout in HBM (all row-major, caller-owned):
//   W        fp32 [n_detectors * E][O]      row r = t*E + lookup_index
//   x        fp32 [B][I]
//   anchors  int32 pairs [n_detectors][n_anchors]
//   idx/md/mi [B][n_detectors]
//   out      fp32 [B][O];  x_grad fp32 [B][I];  w_grad like W
//
// Kernels and their schedules:
//   k_check_detectors   one thread per table over the x rows of a few samples
//                       staged in LDS (one thread per (b, t) for very wide x).
//   k_fill_blocks       one workgroup per (sample, column slice): a thread sums
//                       a block of `dgs` tables of a few columns in fp64, and
//                       the blocks' fp32 (or int32) commit values are added in
//                       ascending order through LDS -- the exact commit order
//                       of the reference CPU path, so the output is
//                       bit-identical to it.
//   k_fill_walk         the same order with one wavefront per (few samples,
//                       column slice), for a lone block or many outputs.
//   k_propagate_rows    one wavefront per (few samples, run of tables); a lane
//                       owns a 32-output block of a (sample, table) item, fed
//                       from coalesced row reads through LDS, and sums it in
//                       fp64 in output order (both summations).
//   k_propagate_fc_exact one thread per (b, t, output block): the reference's
//                       own decomposition, for int32 payloads of other block
//                       sizes, for few items of narrow rows and for rows of a
//                       few outputs (see rows_launch).
//   k_bucket_samples +  table-major weight gradient: a stable counting sort of
//   k_wgrad_slices      the samples of every table by lookup index, then a
//                       wavefront a few table rows, summing g over a row's bucket
//                       in ascending sample order (bit-identical to the reference
//                       CPU path) and writing the row once.  No HBM atomics, and
//                       the caller's zero-fill of w_grad can be fused away.
#include "lut_kernels.h"

#include <algorithm>
#include <type_traits>

namespace spiky {
namespace {

constexpr int kWave = 64;
constexpr int kBlock = 256;

__device__ __forceinline__ uint32_t uniform(uint32_t v) {
    return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ int32_t wrap_add(int32_t a, int32_t b) {
    return (int32_t)((uint32_t)a + (uint32_t)b);
}

// ROUNDED_COMPARISON_GREATER(d, 0.0, cmp_eps), spiky_cuda/misc/misc.h:16
__device__ __forceinline__ bool rounded_greater0(float d, float cmp_eps) {
    if (cmp_eps == 0.0f) return d > 0.0f;
    return (fabsf(d) < cmp_eps) ? false : (d > 0.0f);
}

// du = sign(u) * 0.5 / (1+|u|)^2, sign(u <= 0) = -1, evaluated in the
// reference's order (lut_runtime_kernels_logic.proto:1458-1465).
__device__ __forceinline__ double du_of_margin(float md) {
    double du = (double)md;
    double r = 1.0 / (1.0 + fabs(du));
    return (du > 0) ? r * (0.5 * r) : r * (-0.5 * r);
}

// ---------------------------------------------------------------------------
// check_detectors_logic / check_detectors_eval_logic
// (lut_runtime_kernels_logic.proto:1050-1158).  An anchor id outside
// [0, n_inputs) (including the unused-pair marker -1) is skipped, which is the
// reference's behaviour for the marker and keeps every read in bounds.
// ---------------------------------------------------------------------------
template <bool TRAIN>
__global__ __launch_bounds__(kBlock) void k_check_detectors(
    const float *__restrict__ x, const int2 *__restrict__ anchors, uint32_t n_inputs,
    uint32_t n_detectors, uint32_t n_anchors, uint32_t blocks_per_row, float cmp_eps,
    int32_t *__restrict__ idx, float *__restrict__ md, int32_t *__restrict__ mi) {
    const uint32_t b = blockIdx.x / blocks_per_row;
    const uint32_t t = (blockIdx.x % blocks_per_row) * kBlock + threadIdx.x;
    if (t >= n_detectors) return;
    const float *xb = x + (size_t)b * n_inputs;
    const int2 *ap = anchors + (size_t)t * n_anchors;
    int32_t li = 0;
    float mind = 0.0f;
    int32_t mink = -1;
    for (uint32_t k = 0; k < n_anchors; k++) {
        const int2 a = ap[k];
        if ((uint32_t)a.x >= n_inputs || (uint32_t)a.y >= n_inputs) continue;
        const float d = xb[a.x] - xb[a.y];
        if (rounded_greater0(d, cmp_eps)) li |= (1 << k);
        if (TRAIN) {
            if (mink == -1 || fabsf(d) < fabsf(mind)) {
                mind = d;
                mink = (int32_t)k;
            }
        }
    }
    const size_t o = (size_t)b * n_detectors + t;
    idx[o] = li;
    if (TRAIN) {
        md[o] = mind;
        mi[o] = mink;
    }
}

// The same logic with the x rows of `spb` consecutive samples staged in LDS.
// A thread owns one table: it loads the table's anchor pairs once and
// evaluates them for every staged sample, so the anchor reads are shared by
// spb samples and the 2 * n_anchors input reads per (sample, table) are LDS
// reads instead of dependent global loads.  A workgroup walks `rounds`
// consecutive sample groups with the same anchors in registers, staging each
// group's rows in turn.
constexpr int kCheckMaxAnchors = 16;
constexpr uint32_t kCheckLdsBytes = 64 * 1024;

template <bool TRAIN, int NA>
__global__ __launch_bounds__(1024) void k_check_detectors_lds(
    const float *__restrict__ x, const int2 *__restrict__ anchors, uint32_t batch,
    uint32_t n_inputs, uint32_t n_detectors, uint32_t n_anchors, uint32_t spb, float cmp_eps,
    int32_t *__restrict__ idx, float *__restrict__ md, int32_t *__restrict__ mi, uint32_t gx,
    uint32_t gy, uint32_t rounds) {
    extern __shared__ float xs[];
    // the gx table blocks of one run of sample groups run on one XCD
    // (workgroup i runs on XCD i % 8, consecutively there), so each group's x
    // rows are fetched from HBM once and then served by that XCD's L2
    const uint32_t wl = blockIdx.x;
    const uint32_t run = (wl % 8u) + 8u * (wl / (8u * gx));
    const uint32_t gxb = (wl / 8u) % gx;
    const uint32_t g0 = run * rounds;
    if (g0 >= gy) return;  // uniform over the workgroup
    const uint32_t t = gxb * blockDim.x + threadIdx.x;
    const bool active = t < n_detectors;
    // the table's pairs in registers (fully unrolled, compile-time indices);
    // pairs past n_anchors or with an input id outside [0, n_inputs) are
    // skipped, marked by x = -1
    int2 a[NA];
    const int2 *ap = anchors + (size_t)(active ? t : 0) * n_anchors;
#pragma unroll
    for (int k = 0; k < NA; k++) {
        int2 v = make_int2(-1, -1);
        if ((uint32_t)k < n_anchors) v = ap[k];
        if ((uint32_t)v.x >= n_inputs || (uint32_t)v.y >= n_inputs) v = make_int2(-1, -1);
        a[k] = v;
    }
    const uint32_t g1 = min(g0 + rounds, gy);
    for (uint32_t gyb = g0; gyb < g1; gyb++) {
        const uint32_t b0 = gyb * spb;
        const uint32_t nb = min(spb, batch - b0);
        const uint32_t n_el = nb * n_inputs;
        const float *src = x + (size_t)b0 * n_inputs;
        // every thread is done with the previous group's rows
        if (gyb != g0) __syncthreads();
        if ((n_el & 3u) == 0 && (reinterpret_cast<uintptr_t>(src) & 15u) == 0) {
            const float4 *s4 = reinterpret_cast<const float4 *>(src);
            float4 *d4 = reinterpret_cast<float4 *>(xs);
            for (uint32_t i = threadIdx.x; i < n_el / 4; i += blockDim.x) d4[i] = s4[i];
        } else {
            for (uint32_t i = threadIdx.x; i < n_el; i += blockDim.x) xs[i] = src[i];
        }
        __syncthreads();
        if (!active) continue;
        for (uint32_t sl = 0; sl < nb; sl++) {
            const float *xr = xs + sl * n_inputs;
            int32_t li = 0;
            float mind = 0.0f;
            int32_t mink = -1;
#pragma unroll
            for (int k = 0; k < NA; k++) {
                if (a[k].x >= 0) {
                    const float d = xr[a[k].x] - xr[a[k].y];
                    if (rounded_greater0(d, cmp_eps)) li |= (1 << k);
                    if (TRAIN) {
                        if (mink == -1 || fabsf(d) < fabsf(mind)) {
                            mind = d;
                            mink = (int32_t)k;
                        }
                    }
                }
            }
            const size_t o = (size_t)(b0 + sl) * n_detectors + t;
            idx[o] = li;
            if (TRAIN) {
                md[o] = mind;
                mi[o] = mink;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// fill_outputs_non_seq_fc_logic (proto:1214-1299), re-scheduled.
// ---------------------------------------------------------------------------
constexpr int kWPB = kBlock / kWave;  // wavefronts per workgroup

// Forward gather-sum.  A workgroup owns a sample's column slice, a thread VEC
// columns of one block of dgs tables at a time (16 rows in flight, fp64,
// ascending tables); the blocks' commit values meet in LDS and are added in
// ascending block order: the reference CPU path's arithmetic and commit order, so
// the output is bit-identical to it, and no scratch.  What bounds it is the gather
// (B = 128, T = 2048, E = 256, O = 1024: 166 us, 1.1 GB of rows at 6.5 TB/s) and, for
// a lone sample, its few dependent loads.  Against one wavefront a column slice
// walking all tables in order, with 16 rows in flight a slice (k_fill_walk):
//   fp32  B = 1,    T = 8192, E = 256,  O = 1024:  532 -> 26 us
//         B = 16,   T = 4096, E = 256,  O = 256:   255 -> 18 us
//         B = 100,  T = 1000, E = 128,  O = 301:    72 -> 24 us
//   int8  B = 32,   T = 4096, E = 256,  O = 1024:  399 -> 43 us
//
// Blocks smaller than the rows in flight are taken several at a time (RAGGED, up to
// 16 tables, each block committed where it ends), and a unit's last rows four at a
// time, so that few rows are loaded in vain: blocks of one table, B = 300, T = 512,
// O = 256: 65 us, 240 with a block at a time, 185 walked; B = 1, T = 8192, O = 1024:
// 152 and 214; blocks of 15 tables give up 10 % for it (B = 512, T = 256, O = 301:
// 26.4 and 23.5).
//
// A quad that would cross the row's end starts at n_outputs - 4 instead: its
// first columns repeat the quad before it, value for value.
constexpr int kBlocksThreads = 1024;
constexpr int kBlocksTables = 16;      // rows in flight a thread
constexpr uint32_t kBlocksLds = 8448;  // most commit values in LDS (33 KiB): 32 blocks of 256 columns + 4

typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

typedef int8_t i8x4u __attribute__((ext_vector_type(4), aligned(1)));

template <typename WT, int VEC>
__device__ __forceinline__ void load_columns(const WT *p, float *v) {
    if constexpr (VEC == 4) {
        typedef typename std::conditional<sizeof(WT) == 1, i8x4u, f32x4u>::type Quad;
        const Quad q = *reinterpret_cast<const Quad *>(p);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = (float)q[i];
    } else {
#pragma unroll
        for (int i = 0; i < VEC; i++) v[i] = (float)p[i];
    }
}

template <typename WT, int VEC, bool INT_MODE, bool SCALED, bool RAGGED>
__global__ __launch_bounds__(kBlocksThreads) void k_fill_blocks(
    const WT *__restrict__ w, const float *__restrict__ scales, const int32_t *__restrict__ idx,
    float *__restrict__ out, uint32_t n_outputs, uint32_t n_detectors, uint32_t n_entries,
    uint32_t dgs, uint32_t bpu, uint32_t nq, uint32_t n_slices, uint32_t n_blocks, uint32_t cap,
    double int_rescaler) {
    extern __shared__ uint32_t part[];  // a row of commit values for each block of a chunk
    constexpr int U = kBlocksTables;
    const uint32_t tid = threadIdx.x;
    const uint32_t slice = blockIdx.x % n_slices;
    const uint32_t b = blockIdx.x / n_slices;
    const uint32_t c0 = slice * nq * VEC;
    const uint32_t nc = min(nq * VEC, n_outputs - c0);
    const uint32_t q = tid % nq, g = tid / nq, groups = blockDim.x / nq;
    const uint32_t c = c0 + q * VEC;
    const bool on = g < groups && c < n_outputs;
    const uint32_t cs = min(c, n_outputs - VEC);  // n_outputs >= VEC
    const uint32_t width = nq * VEC + VEC;         // of a block's row in LDS, VEC spare columns first
    const uint32_t emask = n_entries - 1;
    const int32_t *ib = idx + (size_t)b * n_detectors;
    const WT *wc = w + cs;
    const size_t table = (size_t)n_entries * n_outputs;

    // the lookups of tables t .. t + U - 1 (past the last table: its lookup)
    auto lookups = [&](uint32_t (&r)[U], uint32_t t) {
        if (t + U <= n_detectors) {
#pragma unroll
            for (int u = 0; u < U; u += 4) {
                const i32x4u iv = *reinterpret_cast<const i32x4u *>(ib + t + u);
#pragma unroll
                for (int i = 0; i < 4; i++) r[u + i] = (uint32_t)iv[i] & emask;
            }
        } else {
#pragma unroll
            for (int u = 0; u < U; u++) r[u] = (uint32_t)ib[min(t + u, n_detectors - 1)] & emask;
        }
    };

    // the summing threads carry the running output over the chunks of blocks
    float run = 0.0f;
    int32_t irun = 0;
    float *op = out + (size_t)b * n_outputs + c0 + tid;
    if (tid < nc) {
        run = *op;
        irun = __float_as_int(run);
    }
    for (uint32_t k0 = 0; k0 < n_blocks; k0 += cap) {
        const uint32_t nk = min(cap, n_blocks - k0);
        for (uint32_t k = g * bpu; on && k < nk; k += groups * bpu) {
            uint32_t *row = part + k * width + VEC + cs - c0;
            double acc[VEC];
            auto commit = [&]() {
#pragma unroll
                for (int v = 0; v < VEC; v++) {
                    row[v] = INT_MODE ? (uint32_t)(int32_t)(acc[v] * kDenom32 * int_rescaler)
                                      : __float_as_uint((float)acc[v]);
                    acc[v] = 0.0;
                }
                row += width;
            };
            const uint32_t t0 = (k0 + k) * dgs;
            const uint32_t t1 = min(t0 + min(bpu, nk - k) * dgs, n_detectors);
            uint32_t last = t0 + dgs - 1;  // table of the block at hand
#pragma unroll
            for (int v = 0; v < VEC; v++) acc[v] = 0.0;
            for (uint32_t t = t0; t < t1; t += U) {
                uint32_t r[U];
                lookups(r, t);
                float vals[U][VEC];
                auto load = [&](int u) {
                    const uint32_t tt = min(t + u, n_detectors - 1);
                    load_columns<WT, VEC>(wc + tt * table + (size_t)r[u] * n_outputs, vals[u]);
                };
                if (RAGGED) {
                    // four rows at a time up to the unit's end
#pragma unroll
                    for (int u = 0; u < U; u += 4)
                        if (t + u < t1) {
#pragma unroll
                            for (int i = 0; i < 4; i++) load(u + i);
                        }
                } else {
#pragma unroll
                    for (int u = 0; u < U; u++) load(u);
                }
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (RAGGED && t + u >= t1) break;
                    const float sc = SCALED ? scales[min(t + u, n_detectors - 1)] : 1.0f;
#pragma unroll
                    for (int v = 0; v < VEC; v++) {
                        const float x = SCALED ? sc * vals[u][v] : vals[u][v];
                        acc[v] += (double)(t + u < t1 ? x : 0.0f);
                    }
                    if (RAGGED && (t + u == last || t + u + 1 == t1)) {
                        commit();
                        last += dgs;
                    }
                }
            }
            if (!RAGGED) commit();
        }
        __syncthreads();
        if (tid < nc) {
            const uint32_t *col = part + VEC + tid;
            uint32_t k = 0;
            for (; k + U <= nk; k += U) {
                uint32_t v[U];
#pragma unroll
                for (int u = 0; u < U; u++) v[u] = col[(k + u) * width];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    if (INT_MODE)
                        irun = wrap_add(irun, (int32_t)v[u]);
                    else
                        run += __uint_as_float(v[u]);
                }
            }
            for (; k < nk; k++) {
                if (INT_MODE)
                    irun = wrap_add(irun, (int32_t)col[k * width]);
                else
                    run += __uint_as_float(col[k * width]);
            }
        }
        __syncthreads();
    }
    if (tid < nc)
        // convert_integers_to_floats_logic, proto:200-213
        *op = INT_MODE ? (float)(((double)irun * kDenom32Reciproc) / int_rescaler) : run;
}

// The same sums in order, a wavefront SPW samples' column slice: a lane walks all the
// tables of its VEC columns, 16 rows in flight (32 with four samples), and adds a
// block's commit value to the running output where the block ends: no LDS and no
// barrier, but one chain of steps a wavefront.  It is for a lone block of tables, and
// for as many outputs as fill the chip by themselves, where the gather bounds it
// (B = 2048, T = 256, E = 512, O = 1024: 212 us, 289 with k_fill_blocks) and where
// consecutive workgroups take consecutive column slices, so that up to eight of them
// each keep to an XCD's L2 (O = 512, T = 64: 25 and 42 us).
template <typename WT, int VEC, int SPW, bool INT_MODE, bool SCALED>
__global__ __launch_bounds__(kBlock) void k_fill_walk(
    const WT *__restrict__ w, const float *__restrict__ scales, const int32_t *__restrict__ idx,
    float *__restrict__ out, uint32_t batch, uint32_t n_outputs, uint32_t n_detectors,
    uint32_t n_entries, uint32_t dgs, uint32_t n_slices, double int_rescaler) {
    constexpr uint32_t U = SPW == 1 ? 16 : 8;
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = uniform(threadIdx.x / kWave);
    const uint32_t slice = blockIdx.x % n_slices;
    const uint32_t b0 = (blockIdx.x / n_slices * kWPB + wave) * SPW;
    if (b0 >= batch) return;
    const uint32_t c = (slice * kWave + lane) * VEC;
    const bool on = c < n_outputs;
    const uint32_t cs = min(c, n_outputs - VEC);  // n_outputs >= VEC
    const WT *wc = w + cs;
    const size_t table = (size_t)n_entries * n_outputs;
    // samples past the batch repeat the last one and are not stored
    const int32_t *ib[SPW];
#pragma unroll
    for (int s = 0; s < SPW; s++) ib[s] = idx + (size_t)min(b0 + s, batch - 1) * n_detectors;

    float run[SPW][VEC];
    double acc[SPW][VEC];
#pragma unroll
    for (int s = 0; s < SPW; s++)
#pragma unroll
        for (int v = 0; v < VEC; v++) {
            run[s][v] = out[(size_t)min(b0 + s, batch - 1) * n_outputs + cs + v];
            acc[s][v] = 0.0;
        }
    uint32_t last = min(dgs, n_detectors) - 1;  // table of the block at hand
    // N tables from t
    auto step = [&](uint32_t t, auto n) {
        constexpr uint32_t N = decltype(n)::value;
        float vals[N][SPW][VEC];
#pragma unroll
        for (uint32_t u = 0; u < N; u++)
#pragma unroll
            for (int s = 0; s < SPW; s++) {
                const uint32_t r = (uint32_t)ib[s][t + u] & (n_entries - 1);
                load_columns<WT, VEC>(wc + (t + u) * table + (size_t)r * n_outputs, vals[u][s]);
            }
#pragma unroll
        for (uint32_t u = 0; u < N; u++) {
            const float sc = SCALED ? scales[t + u] : 1.0f;
            const bool ends = t + u == last;
#pragma unroll
            for (int s = 0; s < SPW; s++)
#pragma unroll
                for (int v = 0; v < VEC; v++) acc[s][v] += (double)(SCALED ? sc * vals[u][s][v] : vals[u][s][v]);
            if (!ends) continue;
#pragma unroll
            for (int s = 0; s < SPW; s++)
#pragma unroll
                for (int v = 0; v < VEC; v++) {
                    if (INT_MODE)
                        run[s][v] = __int_as_float(wrap_add(__float_as_int(run[s][v]),
                                                            (int32_t)(acc[s][v] * kDenom32 * int_rescaler)));
                    else
                        run[s][v] += (float)acc[s][v];
                    acc[s][v] = 0.0;
                }
            last = min(last + dgs, n_detectors - 1);
        }
    };
    uint32_t t = 0;
    for (; t + U <= n_detectors; t += U) step(t, std::integral_constant<uint32_t, U>());
    for (; t + 4 <= n_detectors; t += 4) step(t, std::integral_constant<uint32_t, 4>());
    for (; t < n_detectors; t++) step(t, std::integral_constant<uint32_t, 1>());
    if (!on) return;
#pragma unroll
    for (int s = 0; s < SPW; s++) {
        if (b0 + s >= batch) break;
        float *ob = out + (size_t)(b0 + s) * n_outputs + cs;
#pragma unroll
        for (int v = 0; v < VEC; v++)
            if (cs + v >= c)  // the columns before c are another lane's
                ob[v] = INT_MODE ? (float)(((double)__float_as_int(run[s][v]) * kDenom32Reciproc) / int_rescaler)
                                 : run[s][v];
    }
}

template <typename WT, int VEC, int SPW, bool INT_MODE, bool SCALED>
hipError_t launch_fill_walk(const FcShape &s, const WT *w, const float *scales, const int32_t *idx,
                            float *out, double int_rescaler, hipStream_t st) {
    const uint32_t n_slices = (s.n_outputs + kWave * VEC - 1) / (kWave * VEC);
    // as many samples a launch as it can hold threads of
    const uint64_t per_wg = kWPB * SPW;
    const uint32_t most = (uint32_t)std::min<uint64_t>(s.batch, kMaxLaunchThreads / ((uint64_t)n_slices * kBlock) * per_wg);
    for (uint32_t b0 = 0; b0 < s.batch;) {
        const uint32_t nb = std::min(most, s.batch - b0);
        const uint32_t grid = n_slices * (uint32_t)((nb + per_wg - 1) / per_wg);
        hipLaunchKernelGGL((k_fill_walk<WT, VEC, SPW, INT_MODE, SCALED>), dim3(grid), dim3(kBlock), 0, st, w,
                           scales, idx + (size_t)b0 * s.n_detectors, out + (size_t)b0 * s.n_outputs, nb,
                           s.n_outputs, s.n_detectors, s.n_entries, s.dgs, n_slices, int_rescaler);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        b0 += nb;
    }
    return hipSuccess;
}

template <typename WT, int VEC, bool INT_MODE, bool SCALED>
hipError_t launch_fill_blocks(const FcShape &s, const WT *w, const float *scales, const int32_t *idx,
                              float *out, double int_rescaler, hipStream_t st) {
    // slices of up to 64 quads, fewer where the batch alone leaves the 256 CUs
    // idle, down to 8 (128 bytes of a row; a lone sample's 4): B = 1, O = 1024:
    // 27 us at 4 quads, 29 at 8, 121 at 64; B = 16: 102 at 16, 188 at 64;
    // B = 255, O = 1000: 510 at 8, 341 at 64
    const uint32_t quads = (s.n_outputs + VEC - 1) / VEC;
    uint32_t n_slices = std::min<uint32_t>((quads + 7) / 8, 256 / s.batch);
    if ((uint64_t)s.batch * n_slices < 64) n_slices = std::min<uint32_t>((quads + 3) / 4, 256 / s.batch);
    n_slices = std::max<uint32_t>(n_slices, (quads + 63) / 64);
    const uint32_t nq = (quads + n_slices - 1) / n_slices;
    n_slices = (quads + nq - 1) / nq;  // every slice starts inside the row
    const uint32_t n_blocks = (s.n_detectors + s.dgs - 1) / s.dgs;
    // blocks a thread takes at a time; threads for those of a chunk
    const uint32_t bpu = std::max<uint32_t>(1, kBlocksTables / s.dgs);
    const bool ragged = s.dgs % kBlocksTables != 0;
    const uint32_t width = nq * VEC + VEC;
    const uint32_t cap = std::min<uint32_t>(n_blocks, kBlocksLds / width / bpu * bpu);  // blocks of a chunk
    const uint32_t units = (cap + bpu - 1) / bpu;
    const uint32_t want = std::max(nq * units, nq * VEC);
    const uint32_t threads = std::min<uint32_t>(kBlocksThreads, (want + kWave - 1) / kWave * kWave);
    // a launch holds fewer than 2^32 threads: more samples than that (4 M of 256
    // columns with 1024 threads) take several
    const uint32_t most = (uint32_t)std::max<uint64_t>(1, kMaxLaunchThreads / ((uint64_t)n_slices * threads));
    for (uint32_t b0 = 0; b0 < s.batch;) {
        const uint32_t nb = std::min(most, s.batch - b0);
#define SPIKY_FB(RG)                                                                              \
    hipLaunchKernelGGL((k_fill_blocks<WT, VEC, INT_MODE, SCALED, RG>), dim3(n_slices * nb), dim3(threads), \
                       cap * width * 4, st, w, scales, idx + (size_t)b0 * s.n_detectors,           \
                       out + (size_t)b0 * s.n_outputs, s.n_outputs, s.n_detectors, s.n_entries, s.dgs, \
                       bpu, nq, n_slices, n_blocks, cap, int_rescaler)
        if (ragged) SPIKY_FB(true); else SPIKY_FB(false);
#undef SPIKY_FB
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        b0 += nb;
    }
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// propagate_through_detectors_non_seq_fc_logic (proto:1421-1499), exact form:
// one thread per (b, t, output block), fp64 dots in ascending output order.
// ---------------------------------------------------------------------------
template <bool INT_MODE>
__global__ __launch_bounds__(kBlock) void k_propagate_fc_exact(
    const float *__restrict__ w, const float *__restrict__ g, const int32_t *__restrict__ idx,
    const float *__restrict__ md, const int32_t *__restrict__ mi, const int2 *__restrict__ anchors,
    float *__restrict__ x_grad, uint32_t n_inputs, uint32_t n_outputs, uint32_t n_detectors,
    uint32_t n_anchors, uint32_t n_entries, uint32_t ogs, uint32_t n_ob, uint64_t n_items,
    double int_rescaler) {
    const uint64_t item = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (item >= n_items) return;
    const uint64_t per_b = (uint64_t)n_detectors * n_ob;
    const uint32_t b = (uint32_t)(item / per_b);
    const uint32_t rem = (uint32_t)(item % per_b);
    const uint32_t t = rem / n_ob;
    const uint32_t ob = rem % n_ob;
    const size_t bt = (size_t)b * n_detectors + t;
    const int32_t m = mi[bt];
    if (m < 0 || (uint32_t)m >= n_anchors) return;
    const uint32_t r = (uint32_t)idx[bt] & (n_entries - 1);
    const uint32_t ra = r ^ (1u << m);
    double du = du_of_margin(md[bt]);
    const uint32_t o0 = ob * ogs;
    const uint32_t o1 = min(o0 + ogs, n_outputs);
    const float *wm = w + ((size_t)t * n_entries + r) * n_outputs;
    const float *wa = w + ((size_t)t * n_entries + ra) * n_outputs;
    const float *gb = g + (size_t)b * n_outputs;
    double ms = 0.0, as = 0.0;
    for (uint32_t o = o0; o < o1; o++) {
        const double gg = (double)gb[o];
        ms += (double)wm[o] * gg;
        as += (double)wa[o] * gg;
    }
    du *= ms - as;
    if (!(fabs(du) > kEps)) return;
    const int2 a = anchors[(size_t)t * n_anchors + m];
    if ((uint32_t)a.x >= n_inputs || (uint32_t)a.y >= n_inputs) return;
    float *xg = x_grad + (size_t)b * n_inputs;
    if (INT_MODE) {
        const int32_t d = (int32_t)(du * kDenom32 * int_rescaler);
        atomicAdd(reinterpret_cast<int32_t *>(xg + a.x), d);
        atomicAdd(reinterpret_cast<int32_t *>(xg + a.y), (int32_t)(0u - (uint32_t)d));
    } else {
        unsafeAtomicAdd(xg + a.x, (float)du);
        unsafeAtomicAdd(xg + a.y, (float)(-du));
    }
}

// ---------------------------------------------------------------------------
// The same gradient over gathered rows (both summations).  A unit is one
// 32-output block of one (sample, table) item, and a lane owns a unit: it sums
// its block of the main and the flipped row against g in fp64 in ascending
// output order -- the reference's own order, so an int32 payload is the
// oracle's -- and the item's units are summed over its lanes before one pair of
// atomics commits the item.  A wave takes `ib` samples and a run of tables, `it`
// tables a step (ib * it items of `nob` units), with g's block of every lane in
// registers as fp64 for the whole run.
//
// Rows are read coalesced, 8 lanes a 128-byte block, into registers while the
// step before is computed, and reach the owning lanes through the wave's 16 KiB
// of LDS (slots swizzled so that neither side meets a bank twice).  What bounds
// it is the gather where rows are many: the samples of a run of tables share an
// XCD's L2 (block order) and a step spans few tables, so a selected row crosses
// HBM once (B = 512, T = 1024, E = 256, O = 256: 298 MB fetched for tables of
// 268 MB).  With the rows in L2 the two wavefronts a SIMD (228 registers) leave
// a step's latencies half exposed: 90 us for those 524 k items.  Measured
// against one wavefront walking all tables of a sample (fp32) and one thread a
// unit (int32):
//   fp32   B = 1,   T = 8192, E = 64,  O = 256:   2000 -> 14 us
//          B = 16,  T = 4096, E = 256, O = 256:   1201 -> 33 us
//          B = 128, T = 2048, E = 256, O = 1024:   800 -> 295 us (distinct rows: 1.4 GB)
//   int32  B = 512, T = 1024, E = 256, O = 256:   2975 -> 113 us
// ---------------------------------------------------------------------------
constexpr int kRowBlock = 32;                       // outputs of a unit
constexpr int kRowPieces = kRowBlock / 4;           // its 16-byte pieces
constexpr uint32_t kRowSkip = 0x80000000u;          // an offset past every buffer: loads give 0

__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <bool INT_MODE, bool SCATTER, bool ODD, bool BIG>
__global__ __launch_bounds__(kWave) void k_propagate_rows(
    const float *__restrict__ w, const float *__restrict__ g, const int32_t *__restrict__ idx,
    const float *__restrict__ md, const int32_t *__restrict__ mi, const int2 *__restrict__ anchors,
    float *__restrict__ x_grad, uint32_t *__restrict__ du_out, uint32_t batch, uint32_t n_inputs,
    uint32_t n_outputs, uint32_t n_detectors, uint32_t n_anchors, uint32_t n_entries, uint32_t run, uint32_t n_runs,
    uint32_t n_obc, uint32_t nob, uint32_t ib, uint32_t it, bool cut_units, double int_rescaler) {
    __shared__ __attribute__((aligned(16))) u32x4 rows[2][kWave * kRowPieces];
    const uint32_t lane = threadIdx.x;
    // all samples of a run of tables and a chunk of outputs on one XCD (workgroup i
    // runs on XCD i % 8)
    const uint32_t groups = (batch + ib - 1) / ib, n_units = n_runs * n_obc;
    uint32_t job, b0;
    if (n_units >= 8) {
        const uint32_t local = blockIdx.x / 8u;
        job = (local / groups) * 8u + blockIdx.x % 8u;
        b0 = local % groups * ib;
    } else {
        job = blockIdx.x % n_units;
        b0 = blockIdx.x / n_units * ib;
    }
    if (job >= n_units) return;
    const uint32_t r = job / n_obc, obc = job % n_obc;
    const uint32_t t0 = r * run, t1 = min(t0 + run, n_detectors);
    // item i is sample b0 + i % ib of the step's table i / ib
    const uint32_t item = lane / nob, ol = lane % nob;
    const uint32_t bi = item % ib, ti = item / ib;
    const uint32_t b = b0 + bi;
    const uint32_t c0 = (obc * nob + ol) * kRowBlock;
    const bool unit = ti < it && b < batch && c0 < n_outputs;
    const uint32_t row_bytes = n_outputs * 4u;

    // lane l moves piece l % 8 of unit 8 i + l / 8; pieces of a row's last block
    // that lie past the row (they belong to the next one) are skipped by an
    // offset past the buffer: no branch, so that all loads of a step are in flight
    const uint32_t piece = lane & 7;
    uint32_t col[kRowPieces], past[kRowPieces];  // first output of the lane's piece i
#pragma unroll
    for (int i = 0; i < kRowPieces; i++) {
        col[i] = (obc * nob + (8u * i + (lane >> 3)) % nob) * kRowBlock + piece * 4u;
        past[i] = col[i] < n_outputs ? 0u : kRowSkip;
    }
    // ODD (n_outputs % 4 != 0): the piece that crosses the row's end holds
    // values of the next row
    auto clip = [&](u32x4 v, int i) {
        if (ODD) {
#pragma unroll
            for (int q = 1; q < 4; q++) v[q] = col[i] + q < n_outputs ? v[q] : 0u;
        }
        return v;
    };
    auto slot_in = [&](int i) {
        const uint32_t u = 8u * i + (lane >> 3);
        return u * kRowPieces + (piece ^ ((u >> 1) & 7));
    };
    auto slot_out = [&](int k) { return lane * kRowPieces + ((uint32_t)k ^ ((lane >> 1) & 7)); };

    // g's block of this lane; outputs past the row count as 0
    double gd[kRowBlock];
    {
        const float *gb = g + (size_t)b0 * n_outputs;
        const uint32_t nb = min(ib, batch - b0);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)gb, (short)0, (int)(nb * row_bytes), 0x00020000);
#pragma unroll
        for (int i = 0; i < kRowPieces; i++) {
            const uint32_t bu = (8u * i + (lane >> 3)) / nob % ib;
            rows[0][slot_in(i)] = clip(
                __builtin_amdgcn_raw_buffer_load_b128(rsrc, (bu * row_bytes + col[i] * 4u) | past[i], 0, 0), i);
        }
        wave_lds_fence();
#pragma unroll
        for (int k = 0; k < kRowPieces; k++) {
            const u32x4 v = rows[0][slot_out(k)];
#pragma unroll
            for (int q = 0; q < 4; q++) gd[4 * k + q] = (double)__uint_as_float(v[q]);
        }
        wave_lds_fence();
    }

    // an item's lookup, kept by all of its unit lanes
    struct Key {
        int32_t row, flip;
        float margin;
    };
    auto load_key = [&](uint32_t tb) {
        const uint32_t t = tb + ti;
        Key k{0, -1, 0.0f};
        if (unit && t < t1) {
            const size_t bt = (size_t)b * n_detectors + t;
            k.row = idx[bt];
            k.flip = mi[bt];
            k.margin = md[bt];
        }
        return k;
    };
    u32x4 stage[2][kRowPieces];
    // BIG: rows by their place in w instead, loads that the row ends cut short
    auto load_rows_far = [&](uint32_t tb, const Key &k) {
        constexpr uint64_t kNone = ~0ull;
        const bool used = k.flip >= 0 && (uint32_t)k.flip < n_anchors;
        const uint32_t rm = (uint32_t)k.row & (n_entries - 1);
        const uint64_t t_row = (uint64_t)(tb + ti) * n_entries;
        const uint64_t om = used ? (t_row + rm) * n_outputs + c0 : kNone;
        const uint64_t oa = used ? (t_row + (rm ^ (1u << k.flip))) * n_outputs + c0 : kNone;
        auto piece_of = [&](uint64_t o, int i) {
            u32x4 v = u32x4{0u, 0u, 0u, 0u};
            if (o == kNone || past[i]) return v;
            const uint32_t *p = reinterpret_cast<const uint32_t *>(w) + o + piece * 4u;
            if (col[i] + 4u <= n_outputs) {
                const i32x4u x = *reinterpret_cast<const i32x4u *>(p);
#pragma unroll
                for (int q = 0; q < 4; q++) v[q] = (uint32_t)x[q];
            } else {
#pragma unroll
                for (int q = 0; q < 3; q++)
                    if (col[i] + q < n_outputs) v[q] = p[q];
            }
            return v;
        };
#pragma unroll
        for (int i = 0; i < kRowPieces; i++) {
            const int u = 8 * i + (int)(lane >> 3);
            stage[0][i] = piece_of(__shfl((unsigned long long)om, u, kWave), i);
            stage[1][i] = piece_of(__shfl((unsigned long long)oa, u, kWave), i);
        }
    };
    auto load_rows = [&](uint32_t tb, const Key &k) {
        if constexpr (BIG) return load_rows_far(tb, k);
        const float *wb = w + (size_t)tb * n_entries * n_outputs;
        const uint64_t left = (uint64_t)(n_detectors - tb) * n_entries * row_bytes;
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void *)wb, (short)0, (int)min(left, (uint64_t)0x7fffffffu), 0x00020000);
        const bool used = k.flip >= 0 && (uint32_t)k.flip < n_anchors;
        const uint32_t rm = (uint32_t)k.row & (n_entries - 1);
        const uint32_t first = ti * n_entries * row_bytes + c0 * 4u;
        const uint32_t om = used ? first + rm * row_bytes : kRowSkip;
        const uint32_t oa = used ? first + (rm ^ (1u << k.flip)) * row_bytes : kRowSkip;
#pragma unroll
        for (int i = 0; i < kRowPieces; i++) {
            const int u = 8 * i + (int)(lane >> 3);
            const uint32_t vm = (uint32_t)__shfl((int)om, u, kWave);
            const uint32_t va = (uint32_t)__shfl((int)oa, u, kWave);
            stage[0][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (vm + piece * 16u) | past[i], 0, 0);
            stage[1][i] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (va + piece * 16u) | past[i], 0, 0);
        }
    };
    auto store_rows = [&]() {
#pragma unroll
        for (int i = 0; i < kRowPieces; i++) {
            rows[0][slot_in(i)] = clip(stage[0][i], i);
            rows[1][slot_in(i)] = clip(stage[1][i], i);
        }
    };

    Key key = load_key(t0);
    load_rows(t0, key);
    Key next = load_key(t0 + it);
    for (uint32_t tb = t0; tb < t1; tb += it) {
        store_rows();
        wave_lds_fence();
        const Key cur = key;
        key = next;
        if (tb + it < t1) {
            load_rows(tb + it, key);
            next = load_key(tb + 2 * it);
        }
        double ms = 0.0, as = 0.0;
#pragma unroll
        for (int h = 0; h < kRowPieces; h += 4) {
            u32x4 m[4], a[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                m[k] = rows[0][slot_out(h + k)];
                a[k] = rows[1][slot_out(h + k)];
            }
            __builtin_amdgcn_sched_barrier(0);  // all eight LDS reads in flight
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    ms += (double)__uint_as_float(m[k][q]) * gd[4 * (h + k) + q];
                    as += (double)__uint_as_float(a[k][q]) * gd[4 * (h + k) + q];
                }
        }
        wave_lds_fence();
        const bool used = cur.flip >= 0 && (uint32_t)cur.flip < n_anchors;
        double du = du_of_margin(cur.margin) * (ms - as);
        if (cut_units && !(fabs(du) > kEps)) du = 0.0;
        int32_t pay = 0;
        if (INT_MODE) pay = (int32_t)(du * kDenom32 * int_rescaler);
        for (uint32_t d = 1; d < nob; d <<= 1) {
            if (INT_MODE) {
                const int32_t o = __shfl_down(pay, d, kWave);
                if (ol + d < nob) pay = wrap_add(pay, o);
            } else {
                const double o = __shfl_down(du, d, kWave);
                if (ol + d < nob) du += o;
            }
        }
        if (SCATTER) {
            // one word an item; an item outside the run is another wave's
            if (unit && ol == 0 && tb + ti < t1) {
                const bool on = used && (INT_MODE || fabs(du) > kEps);
                du_out[(size_t)b * n_detectors + tb + ti] =
                    !on ? 0u : INT_MODE ? (uint32_t)pay : __float_as_uint((float)du);
            }
        } else if (unit && ol == 0 && used && (INT_MODE ? pay != 0 : fabs(du) > kEps)) {
            const int2 a = anchors[(size_t)(tb + ti) * n_anchors + cur.flip];
            if ((uint32_t)a.x < n_inputs && (uint32_t)a.y < n_inputs) {
                float *xg = x_grad + (size_t)b * n_inputs;
                if (INT_MODE) {
                    atomicAdd(reinterpret_cast<int32_t *>(xg + a.x), pay);
                    atomicAdd(reinterpret_cast<int32_t *>(xg + a.y), (int32_t)(0u - (uint32_t)pay));
                } else {
                    unsafeAtomicAdd(xg + a.x, (float)du);
                    unsafeAtomicAdd(xg + a.y, (float)(-du));
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// gather_w_gradients_non_seq_fc_logic (proto:1547-1585), generic atomic form:
// one thread per (b, t, o).
// ---------------------------------------------------------------------------
template <bool INT_MODE>
__global__ __launch_bounds__(kBlock) void k_wgrad_fc_atomic(
    const float *__restrict__ g, const int32_t *__restrict__ idx, float *__restrict__ target,
    uint32_t n_outputs, uint32_t n_detectors, uint32_t n_entries, uint64_t n_items, double lr,
    double int_rescaler) {
    const uint64_t item = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (item >= n_items) return;
    const uint32_t o = (uint32_t)(item % n_outputs);
    const uint64_t bt = item / n_outputs;
    const uint32_t t = (uint32_t)(bt % n_detectors);
    const uint32_t b = (uint32_t)(bt / n_detectors);
    const double gg = (double)g[(size_t)b * n_outputs + o];
    if (!(fabs(gg) > kEps)) return;
    const uint32_t r = (uint32_t)idx[bt] & (n_entries - 1);
    float *p = target + ((size_t)t * n_entries + r) * n_outputs + o;
    if (INT_MODE)
        atomicAdd(reinterpret_cast<int32_t *>(p), (int32_t)(gg * lr * kDenom32 * int_rescaler));
    else
        unsafeAtomicAdd(p, (float)(gg * lr));
}

// ---------------------------------------------------------------------------
// Stable counting sort of samples by lookup index, one wavefront per table.
// offsets[t][e] .. offsets[t][e+1] delimit bucket e in samples[t][*], and the
// samples of a bucket are in ascending order.
// ---------------------------------------------------------------------------
// The lookup indices come from idx [B][T] (a strided column per table) or, when
// key_t is given, from the transposed keys [T][key_pitch] that the table-major
// propagate writes (main << key_shift | (alternative << key_shift) << 16): one
// contiguous row per table.
__global__ __launch_bounds__(kWave) void k_bucket_samples(
    const int32_t *__restrict__ idx, const uint32_t *__restrict__ key_t, uint32_t key_pitch,
    uint32_t key_shift, uint32_t batch, uint32_t n_detectors, uint32_t n_entries, uint32_t n_bits,
    int32_t *__restrict__ offsets, int32_t *__restrict__ samples) {
    extern __shared__ int32_t cnt[];
    const uint32_t t = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const uint32_t emask = n_entries - 1;
    const uint32_t *kt = key_t ? key_t + (size_t)t * key_pitch : nullptr;
    auto key_of = [&](uint32_t b) -> uint32_t {
        return kt ? (((kt[b] & 0xFFFFu) >> key_shift) & emask) : ((uint32_t)idx[(size_t)b * n_detectors + t] & emask);
    };
    // up to kBsCache keys a lane stay in registers for both passes, all loaded
    // up front (a batch of at most 64 * kBsCache samples)
    constexpr int kBsCache = 16;
    const bool cached = batch <= (uint32_t)(kWave * kBsCache);
    uint32_t kc[kBsCache];
    if (cached) {
#pragma unroll
        for (int u = 0; u < kBsCache; u++) {
            const uint32_t b = u * kWave + lane;
            kc[u] = b < batch ? key_of(b) : 0u;
        }
    }
    for (uint32_t e = lane; e < n_entries; e += kWave) cnt[e] = 0;
    __syncthreads();
    if (cached) {
#pragma unroll
        for (int u = 0; u < kBsCache; u++)
            if (u * kWave + lane < batch) atomicAdd(&cnt[kc[u]], 1);
    } else {
        for (uint32_t base = 0; base < batch; base += kWave) {
            const uint32_t b = base + lane;
            if (b < batch) atomicAdd(&cnt[key_of(b)], 1);
        }
    }
    __syncthreads();
    // exclusive scan of cnt[0..E) by one wavefront: each lane sums a contiguous run
    const uint32_t per_lane = (n_entries + kWave - 1) / kWave;
    const uint32_t e0 = min(lane * per_lane, n_entries);
    const uint32_t e1 = min(e0 + per_lane, n_entries);
    int32_t local = 0;
    for (uint32_t e = e0; e < e1; e++) local += cnt[e];
    int32_t incl = local;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t y = __shfl_up(incl, off, kWave);
        if ((int)lane >= off) incl += y;
    }
    int32_t run = incl - local;
    __syncthreads();
    int32_t *off_t = offsets + (size_t)t * (n_entries + 1);
    for (uint32_t e = e0; e < e1; e++) {
        const int32_t c = cnt[e];
        cnt[e] = run;
        off_t[e] = run;
        run += c;
    }
    if (lane == kWave - 1) off_t[n_entries] = incl;
    __syncthreads();
    int32_t *smp_t = samples + (size_t)t * batch;
    // samples base .. base + 63 in order: ballot-ranked among equal keys
    auto scatter = [&](uint32_t base, uint32_t key) {
        const uint32_t b = base + lane;
        const bool valid = b < batch;
        uint64_t peers = __ballot(valid);
        for (uint32_t bit = 0; bit < n_bits; bit++) {
            const bool kb = (key >> bit) & 1u;
            const uint64_t bm = __ballot(kb);
            peers &= kb ? bm : ~bm;
        }
        const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
        const int32_t rank = __popcll(peers & lt);
        int32_t pos = 0;
        if (valid) pos = cnt[key] + rank;
        __syncthreads();
        if (valid) {
            smp_t[pos] = (int32_t)b;
            const uint32_t leader = 63u - (uint32_t)__clzll(peers);
            if (lane == leader) cnt[key] = pos + 1;
        }
        __syncthreads();
    };
    if (cached) {
#pragma unroll
        for (int u = 0; u < kBsCache; u++) {
            if ((uint32_t)u * kWave >= batch) break;  // uniform
            scatter((uint32_t)u * kWave, kc[u]);
        }
    } else {
        for (uint32_t base = 0; base < batch; base += kWave)
            scatter(base, base + lane < batch ? key_of(base + lane) : 0u);
    }
}

// The same sort with a 1024-thread workgroup per table, for few tables over
// many samples (the sequence layers: 16-64 tables of 8192 (b, s) rows).  Wave w
// takes a contiguous run of the samples; per-wave bucket counts (LDS) are
// scanned in (bucket, wave) order, so every wave knows where its run of each
// bucket starts, and the waves scatter their runs in sample order: the result
// equals the one-wavefront sort's.
constexpr int kBsThreads = 1024;
constexpr int kBsWaves = kBsThreads / kWave;
constexpr uint32_t kBsMaxEntries = 1024;

__global__ __launch_bounds__(kBsThreads) void k_bucket_samples_wg(
    const int32_t *__restrict__ idx, const uint32_t *__restrict__ key_t, uint32_t key_pitch,
    uint32_t key_shift, uint32_t batch, uint32_t n_detectors, uint32_t n_entries, uint32_t n_bits,
    int32_t *__restrict__ offsets, int32_t *__restrict__ samples) {
    extern __shared__ int32_t hist[];  // [kBsWaves][n_entries]
    __shared__ int32_t wsum[kBsWaves];
    const uint32_t t = blockIdx.x;
    const uint32_t tid = threadIdx.x, lane = tid & (kWave - 1), wave = tid / kWave;
    const uint32_t emask = n_entries - 1;
    const uint32_t *kt = key_t ? key_t + (size_t)t * key_pitch : nullptr;
    auto key_of = [&](uint32_t b) -> uint32_t {
        return kt ? (((kt[b] & 0xFFFFu) >> key_shift) & emask) : ((uint32_t)idx[(size_t)b * n_detectors + t] & emask);
    };
    // this wave's run of samples: whole 64-sample groups
    const uint32_t groups = (batch + kWave - 1) / kWave;
    const uint32_t per = (groups + kBsWaves - 1) / kBsWaves;
    const uint32_t r0 = min(wave * per * kWave, batch), r1 = min(r0 + per * kWave, batch);
    int32_t *h = hist + wave * n_entries;
    for (uint32_t e = lane; e < n_entries; e += kWave) h[e] = 0;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (kWave - lane));
    // lanes with the same key in a group of 64 samples, and this lane's rank among them
    auto peers_of = [&](uint32_t key, bool valid) -> uint64_t {
        uint64_t peers = __ballot(valid);
        for (uint32_t bit = 0; bit < n_bits; bit++) {
            const bool kb = (key >> bit) & 1u;
            const uint64_t bm = __ballot(kb);
            peers &= kb ? bm : ~bm;
        }
        return peers;
    };
    for (uint32_t base = r0; base < r1; base += kWave) {
        const uint32_t b = base + lane;
        const bool valid = b < r1;
        const uint32_t key = valid ? key_of(b) : 0u;
        const uint64_t peers = peers_of(key, valid);
        if (valid && lane == 63u - (uint32_t)__clzll(peers)) h[key] += __popcll(peers);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
    // bucket e's runs: exclusive prefix over the waves, then over the buckets
    int32_t tot = 0;
    if (tid < n_entries) {
        for (uint32_t w = 0; w < (uint32_t)kBsWaves; w++) {
            const int32_t c = hist[w * n_entries + tid];
            hist[w * n_entries + tid] = tot;
            tot += c;
        }
    }
    int32_t incl = tot;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int32_t y = __shfl_up(incl, off, kWave);
        if ((int)lane >= off) incl += y;
    }
    if (lane == kWave - 1) wsum[wave] = incl;
    __syncthreads();
    int32_t before = 0;
    for (uint32_t w = 0; w < wave; w++) before += wsum[w];
    int32_t *off_t = offsets + (size_t)t * (n_entries + 1);
    if (tid < n_entries) {
        const int32_t start = before + incl - tot;
        off_t[tid] = start;
        for (uint32_t w = 0; w < (uint32_t)kBsWaves; w++) hist[w * n_entries + tid] += start;
    }
    if (tid == 0) off_t[n_entries] = (int32_t)batch;
    __syncthreads();
    int32_t *smp_t = samples + (size_t)t * batch;
    for (uint32_t base = r0; base < r1; base += kWave) {
        const uint32_t b = base + lane;
        const bool valid = b < r1;
        const uint32_t key = valid ? key_of(b) : 0u;
        const uint64_t peers = peers_of(key, valid);
        if (valid) {
            smp_t[h[key] + __popcll(peers & lt)] = (int32_t)b;
            if (lane == 63u - (uint32_t)__clzll(peers)) h[key] += __popcll(peers);
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// Commit values of the weight gradient, one per (sample, output): what the
// reference adds to a table row for that sample (gather_weight_gradients_fc,
// proto:731-790): (float)((double)g * lr) if |(double)g| > EPS, or the int32
// payload (int32)(g * lr * DENOM32 * int_rescaler) for int32 summation.  A
// skipped term becomes -0.0f (float) or 0 (int), which leaves any sum
// unchanged bit for bit (x + -0.0f == x for every x, including +-0.0).
template <bool INT_MODE>
__global__ __launch_bounds__(kBlock) void k_wgrad_commit_values(
    const float *__restrict__ g, uint32_t *__restrict__ cv, uint64_t n, double lr,
    double int_rescaler) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double gg = (double)g[i];
    uint32_t v;
    if (INT_MODE)
        v = fabs(gg) > kEps ? (uint32_t)(int32_t)(gg * lr * kDenom32 * int_rescaler) : 0u;
    else
        v = fabs(gg) > kEps ? __float_as_uint((float)(gg * lr)) : 0x80000000u;
    cv[i] = v;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int VEC>
struct CvLoad;
template <>
struct CvLoad<1> {
    __device__ static void load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t *v) {
        v[0] = __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
    }
};
template <>
struct CvLoad<2> {
    __device__ static void load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t *v) {
        const u32x2 q = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
        v[0] = q.x;
        v[1] = q.y;
    }
};
template <>
struct CvLoad<4> {
    __device__ static void load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff, uint32_t *v) {
        const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
        v[0] = q.x;
        v[1] = q.y;
        v[2] = q.z;
        v[3] = q.w;
    }
};

typedef float f32x2u __attribute__((ext_vector_type(2), aligned(4)));

// Non-temporal store of VEC floats (one instruction, 4-byte aligned).
template <int VEC>
struct NtStore;
template <>
struct NtStore<1> {
    __device__ static void store(float *p, const float *v) { __builtin_nontemporal_store(v[0], p); }
};
template <>
struct NtStore<2> {
    __device__ static void store(float *p, const float *v) {
        __builtin_nontemporal_store(f32x2u{v[0], v[1]}, reinterpret_cast<f32x2u *>(p));
    }
};
template <>
struct NtStore<4> {
    __device__ static void store(float *p, const float *v) {
        __builtin_nontemporal_store(f32x4u{v[0], v[1], v[2], v[3]}, reinterpret_cast<f32x4u *>(p));
    }
};

// Table-major weight gradient over column slices.  Wavefront = `rpw` (<= 63)
// consecutive rows of one table x one column slice; workgroup i works on slice
// i % n_slices, so that an XCD's L2 holds only the slices' commit values that it
// re-reads.  The rows' buckets are contiguous in the table's sorted sample list:
// the wavefront walks that list in batches of KB samples (the next batch loading
// while the current one is added, ping-pong) and closes a row whenever the walk
// crosses its bucket end.  Within a row the commit values are added in ascending
// sample order into an fp32 (or int32) sum starting from the target value (or
// zero when overwriting): the reference CPU path's order, so the result is
// bit-identical to it, and each target element is written exactly once with no
// atomics.  Rows without samples are left alone when accumulating fp32.
// Commit-value rows are read with buffer loads whose row offset is a scalar
// register, so a sample costs VEC adds and one lane read.
//
// A lane whose columns would cross the row's end reads the row's last VEC
// columns instead and stores those that are its own.
template <int VEC, int KB, bool INT_MODE, bool OVERWRITE>
__global__ __launch_bounds__(kBlock) void k_wgrad_slices(
    const uint32_t *__restrict__ cv, const int32_t *__restrict__ offsets,
    const int32_t *__restrict__ samples, float *__restrict__ target, uint32_t batch,
    uint32_t n_outputs, uint32_t n_entries, uint32_t n_detectors, uint32_t n_slices, uint32_t lanes,
    uint32_t rpw, double int_rescaler) {
    const uint32_t lane = threadIdx.x & (kWave - 1);
    const uint32_t wave = uniform(threadIdx.x / kWave);
    const uint32_t slice = blockIdx.x % n_slices;
    const uint64_t unit = (uint64_t)(blockIdx.x / n_slices) * kWPB + wave;
    const uint32_t groups = n_entries / rpw;
    const uint64_t t64 = unit / groups;
    if (t64 >= n_detectors) return;
    const uint32_t t = (uint32_t)t64;
    const uint32_t e0 = (uint32_t)(unit % groups) * rpw;
    const uint32_t c = (slice * lanes + lane) * VEC;
    const bool active = lane < lanes && c < n_outputs;
    const uint32_t cc = active ? min(c, n_outputs - VEC) : 0u;
    const uint32_t own = active ? c - cc : (uint32_t)VEC;  // first of the VEC columns to store
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)cv, (short)0, (int)(batch * n_outputs * 4u), 0x00020000);
    const uint32_t voff = cc * 4u;
    const uint32_t row_bytes = n_outputs * 4u;

    // lane i <= rpw holds the start of bucket e0 + i
    const int32_t *off_t = offsets + (size_t)t * (n_entries + 1) + e0;
    const int32_t offv = lane <= rpw ? off_t[lane] : 0;
    const int32_t *smp = samples + (size_t)t * batch;
    float *tb = target + ((size_t)t * n_entries + e0) * n_outputs + cc;
    const int32_t kbeg = __builtin_amdgcn_readfirstlane(offv);
    const int32_t kend = __builtin_amdgcn_readlane(offv, rpw);
    // a row is opened where it starts, or, accumulating fp32, at its first sample
    constexpr bool kAll = OVERWRITE || INT_MODE;
    if (!kAll && kbeg == kend) return;

    uint32_t acc[VEC];
    auto init = [&](uint32_t e) {
#pragma unroll
        for (int q = 0; q < VEC; q++) acc[q] = 0u;  // +0.0f / int 0
        if (!OVERWRITE) {
            float v[VEC];
            load_columns<float, VEC>(tb + (size_t)e * n_outputs, v);
#pragma unroll
            for (int q = 0; q < VEC; q++) acc[q] = __float_as_uint(v[q]);
        }
    };
    // the rows are written once and not re-read here: non-temporal stores keep
    // them from evicting the commit values this XCD re-reads from its L2
    auto store = [&](uint32_t e) {
        float *p = tb + (size_t)e * n_outputs;
        float v[VEC];
#pragma unroll
        for (int q = 0; q < VEC; q++)
            v[q] = INT_MODE ? (float)(((double)(int32_t)acc[q] * kDenom32Reciproc) / int_rescaler)
                            : __uint_as_float(acc[q]);
        if (own == 0)
            NtStore<VEC>::store(p, v);
        else
#pragma unroll
            for (int q = 1; q < VEC; q++)
                if (q >= (int)own) NtStore<1>::store(p + q, v + q);
    };

    uint32_t e = 0;
    int32_t row_end = __builtin_amdgcn_readlane(offv, 1);
    bool open = kAll;
    if (kAll) init(0);
    for (int32_t k = kbeg; k < kend; k += kWave) {
        const int32_t n = min((int32_t)kWave, kend - k);
        const int32_t idv = smp[k + min((int32_t)lane, n - 1)];
        uint32_t va[KB][VEC], vb[KB][VEC];
        auto load = [&](uint32_t (&v)[KB][VEC], int32_t j0) {
#pragma unroll
            for (int j = 0; j < KB; j++) {
                const uint32_t b = (uint32_t)__builtin_amdgcn_readlane(idv, min(j0 + j, n - 1));
                CvLoad<VEC>::load(rsrc, voff, b * row_bytes, v[j]);
            }
        };
        auto add = [&](const uint32_t (&v)[KB][VEC], int32_t j0) {
#pragma unroll
            for (int j = 0; j < KB; j++) {
                if (j0 + j >= n) break;
                const int32_t kk = k + j0 + j;
                while (kk >= row_end) {
                    if (kAll || open) store(e);
                    e++;
                    row_end = __builtin_amdgcn_readlane(offv, e + 1);
                    if (kAll) init(e);
                    open = false;
                }
                if (!kAll && !open) {
                    init(e);
                    open = true;
                }
#pragma unroll
                for (int q = 0; q < VEC; q++) {
                    if (INT_MODE)
                        acc[q] = acc[q] + v[j][q];
                    else
                        acc[q] = __float_as_uint(__uint_as_float(acc[q]) + __uint_as_float(v[j][q]));
                }
            }
        };
        int32_t j0 = 0;
        load(va, 0);
        for (;;) {
            const bool more_b = j0 + KB < n;
            if (more_b) load(vb, j0 + KB);
            add(va, j0);
            j0 += KB;
            if (!more_b) break;
            const bool more_a = j0 + KB < n;
            if (more_a) load(va, j0 + KB);
            add(vb, j0);
            j0 += KB;
            if (!more_a) break;
        }
    }
    if (!kAll) {
        store(e);  // the row of the last sample
        return;
    }
    for (;;) {
        store(e);
        e++;
        if (e >= rpw) break;
        init(e);
    }
}

__global__ __launch_bounds__(kBlock) void k_zero(float *__restrict__ buf, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) buf[i] = 0.0f;
}

__global__ __launch_bounds__(kBlock) void k_convert_i2f(float *__restrict__ buf, uint64_t n,
                                                        double int_rescaler) {
    const uint64_t i = (uint64_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const double y = (double)__float_as_int(buf[i]) * kDenom32Reciproc;
    buf[i] = (float)(y / int_rescaler);
}

uint32_t blocks_for(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

// The bucketed weight gradient needs the per-table bucket counters in LDS and
// byte offsets of the commit values within 32 bits (buffer loads).
bool rowsum_applies(const FcShape &s) {
    return s.n_entries <= 4096 && (uint64_t)s.batch * s.n_outputs * 4 < 0x7fffffffull;
}

// Most samples of a step of k_propagate_rows: with more, a step's lookups come
// from as many lines of the [B][T] index arrays.
constexpr uint32_t kRowSamples = 8;

// The launch of k_propagate_rows: its split of the work, or that it has none.
struct RowsLaunch {
    bool applies = false;
    bool scatter = false;  // through du and the LDS scatter
    bool big = false;      // tables past 31-bit byte offsets
    uint32_t nob, n_obc, ib, it, run, n_runs, grid;
};

RowsLaunch rows_launch(const FcShape &s, bool int_mode) {
    RowsLaunch r;
    const uint64_t n_items = (uint64_t)s.batch * s.n_detectors;
    if (int_mode && s.ogs != (uint32_t)kRowBlock) return r;  // payloads are formed per 32 outputs
    // A few thousand items of a block or less are one wave's work of
    // k_propagate_fc_exact on every CU, without the staging (B = 64, T = 256,
    // O = 10: 7.9 against 8.8 us).
    if (s.n_outputs <= (uint32_t)kRowBlock && n_items <= (1u << 14)) return r;
    if (s.n_outputs >= (1u << 28)) return r;  // g's rows by 31-bit byte offsets
    const uint32_t blocks = (s.n_outputs + kRowBlock - 1) / kRowBlock;
    r.n_obc = (blocks + kWave - 1) / kWave;
    // Wide rows of many samples in up to eight chunks of 256 outputs or more, each an
    // XCD's: its L2 then holds a chunk of the table that the samples are at, and the
    // lanes of odd widths are filled (B = 1500, T = 64, E = 512: O = 1024 130 -> 77 us, O =
    // 2048 235 -> 146; B = 150, T = 64, O = 1500 29 -> 15; at B = 64 the pushes of the
    // parts cost more: int32, T = 64, E = 512, O = 1024 9 -> 12).
    if (s.n_outputs >= 768 && s.batch >= 128)
        r.n_obc = std::max<uint32_t>(r.n_obc, std::min<uint32_t>(8, (s.n_outputs + 255) / 256));
    r.nob = (blocks + r.n_obc - 1) / r.n_obc;
    const uint32_t items = kWave / r.nob;
    r.ib = std::min<uint32_t>({items, s.batch, kRowSamples});
    // a step's tables are read by 31-bit byte offsets, by 64-bit ones from 2 GiB a table
    const uint64_t table = (uint64_t)s.n_entries * std::max<uint32_t>(s.n_outputs, kRowBlock) * 4;
    r.big = table > 0x7fffffffull;
    r.it = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(items / r.ib, 0x7fffffffull / table));
    // steps a wave: one until ~6144 waves (three rounds of 8 a CU) are in the grid,
    // a row in chunks up to eight, for which g is loaded once, from ~1536; more where a
    // launch could not hold the waves
    const uint64_t groups = (s.batch + r.ib - 1) / r.ib;
    const uint64_t steps = (s.n_detectors + r.it - 1) / r.it;
    const uint64_t total = steps * groups * r.n_obc;
    uint64_t per_wave = std::max<uint64_t>(1, std::min<uint64_t>(32, total / 6144));
    if (r.n_obc > 1) per_wave = std::max(per_wave, std::min<uint64_t>(8, total / 1536));
    for (;; per_wave *= 2) {
        r.run = r.it * (uint32_t)std::min(per_wave, steps);
        r.n_runs = (s.n_detectors + r.run - 1) / r.run;
        const uint64_t units = (uint64_t)r.n_runs * r.n_obc;
        const uint64_t grid = (units >= 8 ? (units + 7) / 8 * 8 : units) * groups;
        r.grid = (uint32_t)grid;
        if (grid * kWave <= kMaxLaunchThreads) break;
        if (r.n_runs == 1) return r;
    }
    // Past 2^14 items the pushes go through du and the LDS scatter where that costs
    // less than a pair of global atomics an item: about 0.1 us a thousand items, or
    // 0.3 us an atomic on one input where few inputs take many (us, pushes / scatter;
    // O = 64 unless said): B = 200, T = 2048: 48 / 28 with 512 inputs; B = 200, T = 512:
    // 16 / 14; B = 16, T = 2048: 30 / 9 with 32 inputs; but B = 1200, T = 32, O = 12,
    // 4096 inputs: 8 / 21; B = 2048, T = 128, O = 33, 12000 inputs: 32 / 69.
    // Only while one wavefront holds a whole item: du has one word an item, and the
    // wavefronts of a row in chunks each have a part of its term, which they add with
    // atomics.  At most 4 GiB of du.
    const double crowd_us = 0.6 * s.n_detectors / s.n_inputs;
    const double scatter_us = input_grad_scatter_applies(s) ? input_grad_scatter_us(s, int_mode) : 1e30;
    r.scatter = r.n_obc == 1 && n_items > (1u << 14) && n_items <= (1u << 30) &&
                std::max(n_items * 95e-6, crowd_us) > scatter_us + 1.5;
    // Rows of a few outputs are one thread's work an item: k_propagate_fc_exact, whose
    // pushes take about 0.055 us a thousand, until the scatter saves more than the
    // staging costs (O = 4, 512 inputs, exact / rows: B = 500, T = 128: 7 / 8 us; B =
    // 64, T = 2048: 12 / 9; B = 200, T = 2048: 29 / 18).
    r.applies = s.n_outputs > 8 || s.ogs < s.n_outputs ||
                (r.scatter && std::max(n_items * 55e-6, crowd_us) > scatter_us + 4.0);
    return r;
}

}  // namespace

// ---------------------------------------------------------------------------
hipError_t launch_check_detectors(const FcShape &s, const float *x, const int32_t *anchors,
                                  float cmp_eps, int32_t *idx, float *min_deltas,
                                  int32_t *min_idx, hipStream_t st) {
    if ((uint64_t)s.batch * s.n_detectors == 0) return hipSuccess;
    const int2 *ap = reinterpret_cast<const int2 *>(anchors);
    const uint32_t spb_lds = kCheckLdsBytes / 4 / std::max<uint32_t>(s.n_inputs, 1);
    if (s.n_anchors <= (uint32_t)kCheckMaxAnchors && spb_lds >= 1 &&
        (uint64_t)(s.batch + 7) * ((s.n_detectors + 63) / 64) <= 0x7fffffffull) {
        // one thread per table, x rows of spb samples in LDS; spb is lowered so
        // that the grid still holds ~512 workgroups where the batch allows it
        const uint32_t threads = std::min<uint32_t>(1024, (s.n_detectors + 63) / 64 * 64);
        const uint32_t gx = (s.n_detectors + threads - 1) / threads;
        const uint64_t want = std::max<uint64_t>(1, (uint64_t)s.batch * gx / 512);
        const uint32_t spb = (uint32_t)std::min<uint64_t>({(uint64_t)spb_lds, want, 16});
        const uint32_t gy = (s.batch + spb - 1) / spb;
        // sample groups a workgroup walks: enough to leave ~512 workgroups
        const uint32_t rounds = (uint32_t)std::max<uint64_t>(1, (uint64_t)gy * gx / 512);
        const uint32_t runs = (gy + rounds - 1) / rounds;
        const uint64_t grid = 8ull * gx * ((runs + 7) / 8);
        if (grid > 0x7fffffffull) return hipErrorInvalidConfiguration;
        const size_t lds = (size_t)spb * s.n_inputs * sizeof(float);
#define SPIKY_CHK(TR, NA)                                                                       \
    hipLaunchKernelGGL((k_check_detectors_lds<TR, NA>), dim3((uint32_t)grid), dim3(threads), lds, st, x, \
                       ap, s.batch, s.n_inputs, s.n_detectors, s.n_anchors, spb, cmp_eps, idx,   \
                       min_deltas, min_idx, gx, gy, rounds)
        if (min_deltas) {
            if (s.n_anchors <= 8) SPIKY_CHK(true, 8); else SPIKY_CHK(true, 16);
        } else {
            if (s.n_anchors <= 8) SPIKY_CHK(false, 8); else SPIKY_CHK(false, 16);
        }
#undef SPIKY_CHK
        return hipGetLastError();
    }
    const uint32_t bpr = (s.n_detectors + kBlock - 1) / kBlock;
    const uint64_t grid = (uint64_t)bpr * s.batch;
    if (min_deltas)
        hipLaunchKernelGGL(k_check_detectors<true>, dim3((uint32_t)grid), dim3(kBlock), 0, st, x,
                           ap, s.n_inputs, s.n_detectors, s.n_anchors, bpr, cmp_eps, idx,
                           min_deltas, min_idx);
    else
        hipLaunchKernelGGL(k_check_detectors<false>, dim3((uint32_t)grid), dim3(kBlock), 0, st, x,
                           ap, s.n_inputs, s.n_detectors, s.n_anchors, bpr, cmp_eps, idx,
                           (float *)nullptr, (int32_t *)nullptr);
    return hipGetLastError();
}

template <typename WT, bool INT_MODE, bool SCALED>
static hipError_t launch_fill_fc(const FcShape &s, const WT *w, const float *scales, const int32_t *idx,
                                 float *out, double int_rescaler, hipStream_t st) {
    if ((uint64_t)s.batch * s.n_detectors * s.n_outputs == 0) return hipSuccess;
    const uint64_t n_blocks = (s.n_detectors + s.dgs - 1) / s.dgs;
    const uint64_t outputs = (uint64_t)s.batch * s.n_outputs;
#define SPIKY_FW(V, S) return launch_fill_walk<WT, V, S, INT_MODE, SCALED>(s, w, scales, idx, out, int_rescaler, st)
    // Walked in order (us, E = 512, blocks of 32 tables, blocks / walked): one block
    // (B = 255, O = 250, T = 19: 7.9 / 6.7), or enough outputs to fill the chip (O =
    // 256, T = 128: B = 300 11 / 15, B = 600 18 / 18, B = 2048 45 / 31; O = 1024, T = 200,
    // E = 64: B = 128 16 / 21, B = 255 33 / 29), if they are not so narrow that a wavefront is
    // mostly idle (O = 33, B = 10000: T = 64 34 / 26, T = 200 39 / 56).  int8 rows are a
    // quarter as long (B = 600, O = 512, T = 200: 26 / 33; B = 2500: 85 / 61).
    // Tables that an L2 holds need more wavefronts (B = 1692, T = 1689, E = 4, O = 126: 104 / 146).
    const uint64_t bytes = (uint64_t)s.n_detectors * s.n_entries * s.n_outputs * sizeof(WT);
    const bool fills = sizeof(WT) == 1 ? outputs >= (1u << 19) && s.n_outputs >= 192
                       : s.n_outputs >= 96 ? outputs >= (bytes <= (8u << 20) ? 6u << 16 : 3u << 16)
                                           : outputs >= (1u << 18) && s.n_detectors <= 64;
    if (n_blocks == 1 || fills) {
        if (outputs <= (1u << 17) || s.n_outputs < 4) SPIKY_FW(1, 1);
        if constexpr (sizeof(WT) == 4) {
            // Four samples a wavefront, one column a lane while the tables are not much
            // past the caches (B = 2048, O = 512: T = 64 25 us, 33 with four columns and
            // 41 with one sample; T = 512 231, 222 and 283), else four columns (O = 2048, T = 256:
            // 434, 599 with one column); a short walk of large tables has too few steps
            // for it (B = 8192, O = 1024, E = 2048, T = 16: 96, 98 with one sample).
            if (outputs < (1u << 20) && !(s.n_outputs < 96 && s.batch >= 4096)) SPIKY_FW(4, 1);
            if (s.n_outputs <= 768 ? bytes <= (192ull << 20) : s.n_detectors < 32 && bytes <= (48ull << 20)) SPIKY_FW(1, 4);
            if (s.n_detectors >= 32) SPIKY_FW(4, 4);
        }
        SPIKY_FW(4, 1);
    }
#undef SPIKY_FW
    // four columns a thread once there is work for the chip (B = 16, O = 1024, T = 64: 7.5
    // us, 6.5 with one; B = 200, O = 256, T = 300: 12.7 and 20.7)
    return s.n_outputs >= 4 && outputs * n_blocks > (1u << 15)
               ? launch_fill_blocks<WT, 4, INT_MODE, SCALED>(s, w, scales, idx, out, int_rescaler, st)
               : launch_fill_blocks<WT, 1, INT_MODE, SCALED>(s, w, scales, idx, out, int_rescaler, st);
}

hipError_t launch_fill_fc_f32(const FcShape &s, const float *w, const int32_t *idx, float *out,
                              bool int_mode, double int_rescaler, hipStream_t st) {
    return int_mode ? launch_fill_fc<float, true, false>(s, w, nullptr, idx, out, int_rescaler, st)
                    : launch_fill_fc<float, false, false>(s, w, nullptr, idx, out, int_rescaler, st);
}

hipError_t launch_fill_fc_i8(const FcShape &s, const int8_t *q8, const float *scales,
                             const int32_t *idx, float *out, bool int_mode, double int_rescaler,
                             hipStream_t st) {
    return int_mode ? launch_fill_fc<int8_t, true, true>(s, q8, scales, idx, out, int_rescaler, st)
                    : launch_fill_fc<int8_t, false, true>(s, q8, scales, idx, out, int_rescaler, st);
}

// scratch: du [B][T] u32 for the scattered input gradient, else none; without a
// buffer the pushes are direct
hipError_t launch_propagate_fc(const FcShape &s, const float *w, const float *g,
                               const int32_t *idx, const float *min_deltas,
                               const int32_t *min_idx, const int32_t *anchors, float *x_grad,
                               bool int_mode, double int_rescaler, Scratch &scratch, hipStream_t st) {
    RowsLaunch r = rows_launch(s, int_mode);
    if (scratch.mode == Scratch::Run && scratch.ptr == nullptr) r.scatter = false;
    ScratchLayout lay(scratch);
    uint32_t *du = r.scatter ? lay.take<uint32_t>((size_t)s.batch * s.n_detectors * 4) : nullptr;
    hipError_t e;
    if (lay.stop(&e, "propagate_through_detectors_fc")) return e;
    const int2 *ap = reinterpret_cast<const int2 *>(anchors);
    if (r.applies) {
#define SPIKY_PR(IM, SC, ODD, BIG)                                                                 \
    hipLaunchKernelGGL((k_propagate_rows<IM, SC, ODD, BIG>), dim3(r.grid), dim3(kWave), 0, st, w,    \
                       g, idx, min_deltas, min_idx, ap, x_grad, du, s.batch, s.n_inputs, s.n_outputs, \
                       s.n_detectors, s.n_anchors, s.n_entries, r.run, r.n_runs, r.n_obc, r.nob, r.ib, \
                       r.it, s.ogs == (uint32_t)kRowBlock, int_rescaler)
#define SPIKY_PR_O(IM, SC)                                                                         \
    if (r.big) SPIKY_PR(IM, SC, true, true);                                                       \
    else if (s.n_outputs % 4 != 0) SPIKY_PR(IM, SC, true, false);                                  \
    else SPIKY_PR(IM, SC, false, false)
        if (r.scatter) {
            if (int_mode) { SPIKY_PR_O(true, true); } else { SPIKY_PR_O(false, true); }
        } else {
            if (int_mode) { SPIKY_PR_O(true, false); } else { SPIKY_PR_O(false, false); }
        }
#undef SPIKY_PR_O
#undef SPIKY_PR
        e = hipGetLastError();
        if (e != hipSuccess) return e;
        if (r.scatter) return launch_input_grad_scatter(s, du, min_idx, anchors, x_grad, int_mode, int_rescaler, st);
    } else {
        const uint32_t n_ob = (s.n_outputs + s.ogs - 1) / s.ogs;
        const uint64_t n_items = (uint64_t)s.batch * s.n_detectors * n_ob;
        if (n_items == 0) return hipSuccess;
#define SPIKY_PE(IM)                                                                               \
    hipLaunchKernelGGL(k_propagate_fc_exact<IM>, dim3(blocks_for(n_items)), dim3(kBlock), 0, st, w, \
                       g, idx, min_deltas, min_idx, ap, x_grad, s.n_inputs, s.n_outputs,            \
                       s.n_detectors, s.n_anchors, s.n_entries, s.ogs, n_ob, n_items, int_rescaler)
        if (int_mode) SPIKY_PE(true); else SPIKY_PE(false);
#undef SPIKY_PE
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return int_mode ? launch_convert_i2f(x_grad, (uint64_t)s.batch * s.n_inputs, int_rescaler, st) : hipSuccess;
}

// scratch (bucketed path): bucket offsets [T][E+1] | sorted samples [T][B] |
// commit values [B][O]; the atomic fallback takes none
hipError_t launch_wgrad_fc(const FcShape &s, const float *g, const int32_t *idx, float *target,
                           double lr, bool int_mode, double int_rescaler, bool overwrite,
                           Scratch &scratch, hipStream_t st, const uint32_t *key_t,
                           uint32_t key_pitch, uint32_t key_shift) {
    const bool rowsum = rowsum_applies(s);
    ScratchLayout lay(scratch);
    int32_t *offsets = rowsum ? lay.take<int32_t>((size_t)s.n_detectors * (s.n_entries + 1) * 4) : nullptr;
    int32_t *samples = rowsum ? lay.take<int32_t>((size_t)s.n_detectors * s.batch * 4) : nullptr;
    uint32_t *cv = rowsum ? lay.take<uint32_t>((size_t)s.batch * s.n_outputs * 4) : nullptr;
    hipError_t e;
    if (lay.stop(&e, "gather_w_gradients_fc")) return e;
    if (rowsum) {
        e = launch_bucket_samples(s, idx, offsets, samples, st,
                                             s.n_entries <= 256 ? key_t : nullptr, key_pitch,
                                             key_shift);
        if (e != hipSuccess) return e;
        // 16 bytes a lane once a row fills the wavefront; an odd width's rows too
        // (B = 255, T = 2048, O = 1000: 600 us, 870 with 4 bytes a lane)
        const uint32_t vec = s.n_outputs > 128 ? 4 : s.n_outputs > 64 ? 2 : 1;
        const uint32_t pieces = (s.n_outputs + vec - 1) / vec;
        const uint32_t n_slices = (pieces + kWave - 1) / kWave;
        const uint32_t lanes = (pieces + n_slices - 1) / n_slices;
        // Rows a wavefront.  With few samples a row the writes bound the kernel, and
        // they run fastest when the grid writes the gradient in order, few rows a
        // workgroup (B = 256, T = 4096, E = 256, O = 256: 168 us at 4 rows, 213 at 32;
        // B = 128, O = 1024: 343 against 445).  From four samples a row the walk
        // bounds it, which a longer list amortises (B = 1024, T = 8192, O = 1024: 1698
        // us at 32, 1924 at 4); so do lists of a few samples among untouched rows.
        const bool walk = s.batch >= 4 * s.n_entries || (!overwrite && !int_mode);
        // int32 rows cost a conversion each: 8 (B = 256, T = 1024, O = 256: 57 us, 66 at 4).
        // Narrow rows are little to write, and a wavefront's start and its list cost
        // more: 32 rows up to 32 outputs (B = 3, T = 7000, E = 128, O = 16: 71 us at 4,
        // 39 at 32; B = 2, T = 2048, E = 1024: 145 and 70), 16 up to 64 (O = 64: 72 at 4,
        // 61 at 16, 62 at 32; B = 64, T = 1000, E = 256: 38, 29 and 30).
        const uint32_t most = s.n_outputs <= 32 || walk ? 32 : s.n_outputs <= 64 ? 16 : int_mode ? 8 : 4;
        uint32_t rpw = std::min<uint32_t>(s.n_entries, most);
        // Fewer again where few tables would leave the grid short of 32 wavefronts a
        // CU (narrow rows: 16), more where a launch could not hold the wavefronts.
        auto waves = [&](uint32_t r) { return (uint64_t)n_slices * s.n_detectors * (s.n_entries / r); };
        while (rpw > 4 && waves(rpw) < (s.n_outputs <= 64 ? 4096 : 8192)) rpw /= 2;
        while (rpw < std::min<uint32_t>(s.n_entries, 32) && (waves(rpw) + kWPB * n_slices) * kWave > kMaxLaunchThreads)
            rpw *= 2;
        const uint64_t units = (uint64_t)s.n_detectors * (s.n_entries / rpw);
        const uint64_t grid = (uint64_t)n_slices * ((units + kWPB - 1) / kWPB);
        if (grid > 0x7fffffffu) return hipErrorInvalidConfiguration;
        const uint64_t n_cv = (uint64_t)s.batch * s.n_outputs;
        if (int_mode)
            hipLaunchKernelGGL(k_wgrad_commit_values<true>, dim3(blocks_for(n_cv)), dim3(kBlock), 0,
                               st, g, cv, n_cv, lr, int_rescaler);
        else
            hipLaunchKernelGGL(k_wgrad_commit_values<false>, dim3(blocks_for(n_cv)), dim3(kBlock), 0,
                               st, g, cv, n_cv, lr, int_rescaler);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
#define SPIKY_WG(V, IM, OW)                                                                       \
    hipLaunchKernelGGL((k_wgrad_slices<V, 8, IM, OW>), dim3((uint32_t)grid), dim3(kBlock), 0, st, \
                       cv, offsets, samples, target, s.batch, s.n_outputs, s.n_entries,           \
                       s.n_detectors, n_slices, lanes, rpw, int_rescaler)
#define SPIKY_WG_V(IM, OW)                     \
    switch (vec) {                             \
        case 4: SPIKY_WG(4, IM, OW); break;    \
        case 2: SPIKY_WG(2, IM, OW); break;    \
        default: SPIKY_WG(1, IM, OW); break;   \
    }
        if (int_mode) {
            if (overwrite) { SPIKY_WG_V(true, true) } else { SPIKY_WG_V(true, false) }
        } else {
            if (overwrite) { SPIKY_WG_V(false, true) } else { SPIKY_WG_V(false, false) }
        }
#undef SPIKY_WG_V
#undef SPIKY_WG
        return hipGetLastError();
    }
    // generic atomic fallback: the caller must have zeroed target when overwrite was asked for
    const uint64_t n_items = (uint64_t)s.batch * s.n_detectors * s.n_outputs;
    if (n_items == 0) return hipSuccess;
    if (overwrite) {
        e = launch_zero(target, (uint64_t)s.n_detectors * s.n_entries * s.n_outputs, st);
        if (e != hipSuccess) return e;
    }
    if (int_mode)
        hipLaunchKernelGGL(k_wgrad_fc_atomic<true>, dim3(blocks_for(n_items)), dim3(kBlock), 0, st,
                           g, idx, target, s.n_outputs, s.n_detectors, s.n_entries, n_items, lr,
                           int_rescaler);
    else
        hipLaunchKernelGGL(k_wgrad_fc_atomic<false>, dim3(blocks_for(n_items)), dim3(kBlock), 0,
                           st, g, idx, target, s.n_outputs, s.n_detectors, s.n_entries, n_items,
                           lr, int_rescaler);
    e = hipGetLastError();
    if (e != hipSuccess || !int_mode) return e;
    return launch_convert_i2f(target, (uint64_t)s.n_detectors * s.n_entries * s.n_outputs,
                              int_rescaler, st);
}

hipError_t launch_wgrad_commit_values(const float *g, uint32_t *cv, uint64_t n, double lr,
                                      bool int_mode, double int_rescaler, hipStream_t st) {
    if (n == 0) return hipSuccess;
    if (int_mode)
        hipLaunchKernelGGL(k_wgrad_commit_values<true>, dim3(blocks_for(n)), dim3(kBlock), 0, st, g,
                           cv, n, lr, int_rescaler);
    else
        hipLaunchKernelGGL(k_wgrad_commit_values<false>, dim3(blocks_for(n)), dim3(kBlock), 0, st, g,
                           cv, n, lr, int_rescaler);
    return hipGetLastError();
}

hipError_t launch_bucket_samples(const FcShape &s, const int32_t *idx, int32_t *offsets,
                                 int32_t *samples, hipStream_t st, const uint32_t *key_t,
                                 uint32_t key_pitch, uint32_t key_shift) {
    if (s.n_detectors == 0) return hipSuccess;
    uint32_t n_bits = 0;
    while ((1u << n_bits) < s.n_entries) n_bits++;
    if (s.n_detectors < 1024 && s.batch >= 2048 && s.n_entries <= kBsMaxEntries) {
        // few tables over many samples: a workgroup per table
        hipLaunchKernelGGL(k_bucket_samples_wg, dim3(s.n_detectors), dim3(kBsThreads),
                           (size_t)kBsWaves * s.n_entries * sizeof(int32_t), st, idx, key_t, key_pitch,
                           key_shift, s.batch, s.n_detectors, s.n_entries, n_bits, offsets, samples);
        return hipGetLastError();
    }
    hipLaunchKernelGGL(k_bucket_samples, dim3(s.n_detectors), dim3(kWave),
                       s.n_entries * sizeof(int32_t), st, idx, key_t, key_pitch, key_shift,
                       s.batch, s.n_detectors, s.n_entries, n_bits, offsets, samples);
    return hipGetLastError();
}

hipError_t launch_zero(float *buf, uint64_t n, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_zero, dim3(blocks_for(n)), dim3(kBlock), 0, st, buf, n);
    return hipGetLastError();
}

hipError_t launch_convert_i2f(float *buf, uint64_t n, double int_rescaler, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_convert_i2f, dim3(blocks_for(n)), dim3(kBlock), 0, st, buf, n,
                       int_rescaler);
    return hipGetLastError();
}

}  // namespace spiky
