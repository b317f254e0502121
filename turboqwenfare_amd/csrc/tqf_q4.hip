// tqf_q4.hip -- Q4_0 row-lane layout, activation prep, GEMV and the three MoE
// layer kernels (route, gate/up + SwiGLU, down + weighted combine) for gfx950.
//
// The matrix layout and the integer-dot activation format are described in
// tqf_internal.h.  The matvecs read the weight bytes exactly once with 128-bit
// loads (a row's blocks spread over the lanes, 1 KiB per wavefront load) and
// combine partial sums in a fixed order (DPP / permlane transposes, then LDS),
// so results are deterministic run to run.  A pool of matrices is bound by
// HBM; one matrix, or one layer of a few tokens, by the latencies of its
// dependent loads (what each kernel says).
#include <hip/hip_runtime.h>

#include "tqf_device.h"
#include "tqf_internal.h"
#include "tqf_route.h"

namespace tqf {

// ---------------------------------------------------------------------------
// Repack: GGML Q4_0 (rows x B x 18 bytes) -> row-lane layout.  One thread per
// block; the destination was zero-filled (padding rows/blocks keep scale 0).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void repack_kernel(const uint8_t *__restrict__ aos,
                                                     MatrixDims d, uint8_t *__restrict__ dst) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (uint64_t)d.rows * d.blocks) return;
    const uint32_t r = (uint32_t)(idx / d.blocks), b = (uint32_t)(idx % d.blocks);
    const uint8_t *src = aos + idx * kQ4Block;
    uint8_t *nib = dst + nibble_offset(d, r, b);
#pragma unroll
    for (int i = 0; i < 16; ++i) nib[i] = src[2 + i];
    uint8_t *sc = dst + scale_offset(d, r, b);
    sc[0] = src[0];
    sc[1] = src[1];
}

hipError_t launch_repack(hipStream_t s, const uint8_t *d_aos, const MatrixDims &d,
                         uint8_t *dst) {
    const uint64_t n = (uint64_t)d.rows * d.blocks;
    if (n == 0) return hipSuccess;
    const uint32_t grid = (uint32_t)((n + 255) / 256);
    hipLaunchKernelGGL(repack_kernel, dim3(grid), dim3(256), 0, s, d_aos, d, dst);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Activation prep: x [m x cols] f32 -> xprep [m x blocks_padded x 32 dwords].
// One wavefront handles two blocks (32 lanes each).  Blocks past `cols` are
// written as zero records.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void prep_kernel(const float *__restrict__ x, uint32_t cols,
                                                   uint32_t blocks_padded,
                                                   uint32_t *__restrict__ xprep) {
    const uint32_t t = blockIdx.y;
    const uint32_t kb = (blockIdx.x * blockDim.x + threadIdx.x) / 32;
    if (kb >= blocks_padded) return;
    const uint32_t j = threadIdx.x & 31;
    const uint32_t col = kb * 32 + j;
    float v[1] = {col < cols ? x[(size_t)t * cols + col] : 0.0f};
    prep_block<1>(v, (int)j, xprep + (size_t)t * blocks_padded * kXprepDwords, blocks_padded, kb);
}

hipError_t launch_prep(hipStream_t s, const float *x, uint32_t m, uint32_t cols,
                       uint32_t blocks_padded, uint32_t *xprep) {
    const uint32_t threads = blocks_padded * 32;
    const uint32_t grid = (threads + 255) / 256;
    hipLaunchKernelGGL(prep_kernel, dim3(grid, m), dim3(256), 0, s, x, cols, blocks_padded,
                       xprep);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Standalone GEMV / small-M GEMM: y[mat][t][row] for `count` matrices of one
// shape.  Grid (row groups, count), eight wavefronts per workgroup.  Lane
// group j (LPR lanes) of a wavefront owns 8 consecutive rows (one octet);
// lane b reads block b (+ LPR, + 2 LPR, ... for long rows) of each of them.
// Per chunk of LPR blocks, every load (8 nibble vectors, the octet's scales
// and the activation records of up to four tokens) is issued before any
// arithmetic; the row sums come out of transpose_reduce, one row per lane.
// Tokens beyond four reuse the weights held in registers.
// ---------------------------------------------------------------------------
constexpr int kGemvWaves = 8;
constexpr int kGemvRows = 8;  // rows per lane group

template <int LPR, int TG>
__global__ __launch_bounds__(kGemvWaves * kWave) void gemv_kernel(
    const uint8_t *const *__restrict__ tables, MatrixDims d, const uint32_t *__restrict__ xprep,
    uint32_t m, float *__restrict__ y) {
    constexpr int G = kWave / LPR;
    constexpr int RW = kGemvRows * G;  // rows per wavefront
    constexpr int NL = kGemvRows;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const uint32_t j = (uint32_t)lane / LPR, b = (uint32_t)lane % LPR;
    const uint32_t mat = blockIdx.y;
    const uint32_t r0 = (blockIdx.x * kGemvWaves + wave) * RW;
    if (r0 >= d.rows_padded) return;
    const RowLane W = row_lane(tables[mat], d.blocks_padded);
    const uint32_t rl = r0 + j * NL;
    const uint32_t row = rl + reduced_index<LPR, NL>(lane);
    const bool writer = reduced_first_copy<LPR, NL>(lane) && row < d.rows;
    const uint32_t chunks = d.blocks_padded / LPR;
    const size_t xstride = (size_t)d.blocks_padded * kXprepDwords;
    for (uint32_t t0 = 0; t0 < m; t0 += TG) {
        float acc[TG][NL];
#pragma unroll
        for (int t = 0; t < TG; ++t)
#pragma unroll
            for (int n = 0; n < NL; ++n) acc[t][n] = 0.0f;
        for (uint32_t c = 0; c < chunks; ++c) {
            const uint32_t blk = c * LPR + b;
            uint4 nib[NL];
#pragma unroll
            for (int n = 0; n < NL; ++n) nib[n] = q4_signed(load_nibbles(W, rl + n, blk));
            const uint4 sc = load_scales(W, rl / 8, blk);
            uint32_t x[TG][28];
#pragma unroll
            for (int t = 0; t < TG; ++t) {
                const uint32_t tt = t0 + t < m ? t0 + t : 0;  // loads stay unconditional
                load_xrec(xprep + tt * xstride, d.blocks_padded, blk, x[t]);
                if (blk >= d.blocks) x[t][24] = 0;  // padding: exactly 0 whatever it holds
            }
            __builtin_amdgcn_sched_barrier(0);  // every load in flight before any math
#pragma unroll
            for (int t = 0; t < TG; ++t)
#pragma unroll
                for (int n = 0; n < NL; ++n)
                    acc[t][n] = fmaf(octet_scale(sc, n), q4_block_dot(nib[n], x[t]), acc[t][n]);
        }
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const float s = transpose_reduce<LPR, NL>(acc[t]);
            if (writer && t0 + t < m) y[((size_t)mat * m + t0 + t) * d.rows + row] = s;
        }
    }
}

template <int LPR>
hipError_t launch_gemv_lpr(hipStream_t s, const uint8_t *const *d_tables, uint32_t count,
                           const MatrixDims &d, const uint32_t *xprep, uint32_t m, float *y) {
    constexpr uint32_t rows_per_group = kGemvWaves * kGemvRows * (kWave / LPR);
    const dim3 grid((d.rows_padded + rows_per_group - 1) / rows_per_group, count);
    const dim3 block(kGemvWaves * kWave);
    if (m <= 1) hipLaunchKernelGGL((gemv_kernel<LPR, 1>), grid, block, 0, s, d_tables, d, xprep, m, y);
    else if (m <= 2) hipLaunchKernelGGL((gemv_kernel<LPR, 2>), grid, block, 0, s, d_tables, d, xprep, m, y);
    else hipLaunchKernelGGL((gemv_kernel<LPR, 4>), grid, block, 0, s, d_tables, d, xprep, m, y);
    return hipGetLastError();
}

hipError_t launch_gemv(hipStream_t s, const uint8_t *const *d_tables, uint32_t count,
                       const MatrixDims &d, const uint32_t *xprep, uint32_t m, float *y) {
    if (d.lpr == 16) return launch_gemv_lpr<16>(s, d_tables, count, d, xprep, m, y);
    if (d.lpr == 32) return launch_gemv_lpr<32>(s, d_tables, count, d, xprep, m, y);
    return launch_gemv_lpr<64>(s, d_tables, count, d, xprep, m, y);
}

// ---------------------------------------------------------------------------
// Route kernel.  One workgroup per two router rows (row n_experts is the
// shared-expert input gate, experts/mod.rs:1614).  Each workgroup
//   1. loads h [m x hidden], applies RMSNorm when `norm` is given
//      (weights.rs:216-239: x * (1/sqrt(mean(x^2) + 1e-6)) * w),
//   2. computes its router logits (experts/mod.rs:1491 router matvec),
//   3. writes the xprep / Q8_K records of the blocks assigned to it.
// The routes themselves are made from the logits by the gate/up kernels
// (tqf_route.h).  Bound by its latencies (loads, two block sums), not by its
// 2.1 MB: 4.4 / 6.1 / 8.3 us with the norm at 1 / 4 / 8 tokens (with the routing
// behind a poll of every workgroup's logits 7.7 / 10.4 / 14.0).
// ---------------------------------------------------------------------------
constexpr int kRouteRows = 2;
constexpr int kRouteThreads = 256;

template <int MT>
__global__ __launch_bounds__(kRouteThreads) void route_kernel(LayerDev L, const float *__restrict__ h,
                                                              const float *__restrict__ norm, uint32_t m,
                                                              uint32_t bp, uint32_t *__restrict__ xprep,
                                                              float *__restrict__ logits,
                                                              uint32_t *__restrict__ q8, uint32_t bp8) {
    __shared__ double s_dot[MT * kRouteRows][32];  // per value the partial sums of 32 groups of eight threads
    __shared__ float lds_red[4][MT * kRouteRows];
    __shared__ float lds_norm[4][MT];
    __shared__ float s_blk[MT][32];

    const int tid = threadIdx.x;
    const uint32_t H = L.hidden, E = L.n_experts;
    const int vpt = (int)(H / 256);  // 1..8 elements per thread
    const uint32_t col0 = (uint32_t)tid * vpt;

    // this workgroup's router rows, loaded first so that their latency
    // overlaps the activation loads and the records below
    // (the model geometry, hidden 2048, loads 8 contiguous floats per thread
    // as two 16-byte loads; other widths element by element)
    float wv[kRouteRows][8] = {};
    float x[MT][8] = {};
    float nw[8] = {};  // the norm's weights: loaded here, not behind the sum of squares
    if (vpt == 8) {
#pragma unroll
        for (int rr = 0; rr < kRouteRows; ++rr) {
            const uint32_t r = blockIdx.x * kRouteRows + rr;
            const float *wrow = (r < E) ? L.router + (size_t)r * H : L.shared_input_gate;
            const float4 a = r <= E ? *reinterpret_cast<const float4 *>(wrow + col0) : make_float4(0, 0, 0, 0);
            const float4 b = r <= E ? *reinterpret_cast<const float4 *>(wrow + col0 + 4) : make_float4(0, 0, 0, 0);
            wv[rr][0] = a.x; wv[rr][1] = a.y; wv[rr][2] = a.z; wv[rr][3] = a.w;
            wv[rr][4] = b.x; wv[rr][5] = b.y; wv[rr][6] = b.z; wv[rr][7] = b.w;
        }
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const float *xr = h + (size_t)t * H + col0;
            const float4 a = t < (int)m ? *reinterpret_cast<const float4 *>(xr) : make_float4(0, 0, 0, 0);
            const float4 b = t < (int)m ? *reinterpret_cast<const float4 *>(xr + 4) : make_float4(0, 0, 0, 0);
            x[t][0] = a.x; x[t][1] = a.y; x[t][2] = a.z; x[t][3] = a.w;
            x[t][4] = b.x; x[t][5] = b.y; x[t][6] = b.z; x[t][7] = b.w;
        }
        if (norm != nullptr) {
            const float4 a = *reinterpret_cast<const float4 *>(norm + col0), b = *reinterpret_cast<const float4 *>(norm + col0 + 4);
            nw[0] = a.x; nw[1] = a.y; nw[2] = a.z; nw[3] = a.w;
            nw[4] = b.x; nw[5] = b.y; nw[6] = b.z; nw[7] = b.w;
        }
    } else {
#pragma unroll
        for (int rr = 0; rr < kRouteRows; ++rr) {
            const uint32_t r = blockIdx.x * kRouteRows + rr;
            const float *wrow = (r < E) ? L.router + (size_t)r * H : L.shared_input_gate;
#pragma unroll
            for (int v = 0; v < 8; ++v) wv[rr][v] = (r <= E && v < vpt) ? wrow[col0 + v] : 0.0f;
        }
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int v = 0; v < 8; ++v)
                x[t][v] = (t < (int)m && v < vpt) ? h[(size_t)t * H + col0 + v] : 0.0f;
        if (norm != nullptr)
#pragma unroll
            for (int v = 0; v < 8; ++v) nw[v] = v < vpt ? norm[col0 + v] : 0.0f;
    }

    if (norm != nullptr) {
        float ss[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            ss[t] = 0.0f;
#pragma unroll
            for (int v = 0; v < 8; ++v) ss[t] += x[t][v] * x[t][v];
        }
        block_sum_256<MT>(ss, lds_norm);
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const float inv = 1.0f / sqrtf(ss[t] / (float)H + 1e-6f);
#pragma unroll
            for (int v = 0; v < 8; ++v) x[t][v] = x[t][v] * inv * nw[v];
        }
    }

    // 2. logits of this workgroup's rows.  For Q4_0 layers the products and
    //    sums are in 64 bits: the persistent stack kernel adds its partial
    //    logits in 64 bits, and what runs in its place holds them in no fewer
    //    (route weights of one and four normalised rows against 64 bits,
    //    relative: 0.88e-7 and 0.90e-7; f32 sums 1.45e-7 and 1.42e-7, the
    //    persistent kernel 1.07e-7 and 1.11e-7; 4.3 / 6.4 / 8.5 -> 4.4 / 6.1 /
    //    8.3 us at 1 / 4 / 8 tokens).  For Q4_K layers, which the persistent
    //    kernel does not run, they stay in f32: the 8-bit activations turn a
    //    changed last bit into another answer.
    if (q8 == nullptr) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            double s[kRouteRows] = {};
#pragma unroll
            for (int v = 0; v < 8; ++v)
#pragma unroll
                for (int rr = 0; rr < kRouteRows; ++rr) s[rr] = fma((double)x[t][v], (double)wv[rr][v], s[rr]);
#pragma unroll
            for (int rr = 0; rr < kRouteRows; ++rr) {
                s[rr] += dpp_d<kDppXor1>(s[rr]);
                s[rr] += dpp_d<kDppXor2>(s[rr]);
                s[rr] += dpp_d<kDppHalfMirror>(s[rr]);
                if ((tid & 7) == 0) s_dot[rr * MT + t][tid >> 3] = s[rr];
            }
        }
        __syncthreads();
        if (tid < 8 * MT * kRouteRows) {  // eight threads a value, four groups of eight threads each
            const int i = tid >> 3, t = i % MT, g = 4 * (tid & 7);
            double s = (s_dot[i][g] + s_dot[i][g + 1]) + (s_dot[i][g + 2] + s_dot[i][g + 3]);
            s += dpp_d<kDppXor1>(s);
            s += dpp_d<kDppXor2>(s);
            s += dpp_d<kDppHalfMirror>(s);
            const uint32_t r = blockIdx.x * kRouteRows + i / MT;
            if ((tid & 7) == 0 && r <= E && t < (int)m) logits[(size_t)t * (E + 1) + r] = (float)s;
        }
    } else {
        float dots[MT * kRouteRows];
#pragma unroll
        for (int rr = 0; rr < kRouteRows; ++rr) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                float s = 0.0f;
#pragma unroll
                for (int v = 0; v < 8; ++v) s = fmaf(x[t][v], wv[rr][v], s);
                dots[rr * MT + t] = s;
            }
        }
        block_sum_256<MT * kRouteRows>(dots, lds_red);
        if (tid == 0) {
#pragma unroll
            for (int rr = 0; rr < kRouteRows; ++rr) {
                const uint32_t r = blockIdx.x * kRouteRows + rr;
                if (r <= E)
                    for (int t = 0; t < (int)m; ++t) logits[(size_t)t * (E + 1) + r] = dots[rr * MT + t];
            }
        }
    }
    // 3. xprep (when asked for) of block kb is written by workgroup kb, one
    //    half-wavefront per token: the threads that hold the block's elements
    //    leave them in LDS.  (Made by those threads themselves, eight elements
    //    each and token after token, the records of eight tokens took longer
    //    than the rest.)  Records are strided by the gate/up matrices' padded
    //    block count bp.
    const uint32_t KB = xprep ? H / 32 : 0;
    for (uint32_t kb = blockIdx.x; kb < KB; kb += gridDim.x) {
        const int at = (int)col0 - (int)kb * 32;  // vpt need not divide 32
        __syncthreads();
        if (at > -vpt && at < 32) {
#pragma unroll
            for (int t = 0; t < MT; ++t)
#pragma unroll
                for (int v = 0; v < 8; ++v)
                    if (v < vpt && (uint32_t)(at + v) < 32u) s_blk[t][at + v] = x[t][v];
        }
        __syncthreads();
        const int t = tid >> 5, j = tid & 31;
        prep_block32(s_blk[t < MT ? t : 0][j], j, t < (int)m, xprep + (size_t)(t < MT ? t : 0) * bp * kXprepDwords, bp, kb,
                     PlainStore());
    }

    // 4. Q8_K records (when asked for): chunk j < m * H / 256 (chunk c = j %
    //    (H / 256) of row t = j / (H / 256)) by workgroup j; staged in LDS in
    //    the quantizer's lane order.
    const uint32_t cpr = H / 256;
    const uint32_t jq = blockIdx.x;
    if (q8 != nullptr && jq < m * cpr) {
        __shared__ float s_chunk[256];
        const uint32_t t = jq / cpr, c = jq % cpr;
#pragma unroll
        for (int tt = 0; tt < MT; ++tt)
            if (tt == (int)t)
#pragma unroll
                for (int v = 0; v < 8; ++v) {
                    const uint32_t e = col0 + (uint32_t)v;
                    if (v < vpt && e >= 256 * c && e < 256 * c + 256) s_chunk[e - 256 * c] = x[tt][v];
                }
        __syncthreads();
        if (tid < kWave) {
            const int k = tid >> 3, cc = tid & 7;
            float v4[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v4[i] = s_chunk[32 * k + cc + 8 * i];
            q8k_quantize_values(v4, q8 + (size_t)t * bp8 * kQ8KRecDwords, bp8, c);
        }
    }
}

hipError_t launch_route(hipStream_t s, const LayerDev &L, const float *h, const float *norm,
                        uint32_t m, float *logits, uint32_t *xprep, uint32_t *q8, uint32_t bp8) {
    if (q8 && (m * (L.hidden / 256) > (L.n_experts + 1 + kRouteRows - 1) / kRouteRows || bp8 < L.hidden / 32))
        return hipErrorInvalidValue;
    const uint32_t grid = (L.n_experts + 1 + kRouteRows - 1) / kRouteRows;
    const uint32_t bp = padded_blocks(L.hidden / 32);
#define TQF_ROUTE(MT) \
    hipLaunchKernelGGL(route_kernel<MT>, dim3(grid), dim3(kRouteThreads), 0, s, L, h, norm, m, bp, xprep, logits, q8, bp8)
    if (m <= 1) TQF_ROUTE(1);
    else if (m <= 2) TQF_ROUTE(2);
    else if (m <= 4) TQF_ROUTE(4);
    else TQF_ROUTE(8);
#undef TQF_ROUTE
    return hipGetLastError();
}

// The distinct down matrices among the tokens' routes: a lane counts when no
// lower one holds its matrix.
__global__ __launch_bounds__(kWave) void count_union_kernel(Plan *plan, uint32_t m) {
    const uint32_t n = m * kTopK, i = threadIdx.x;
    bool first = i < n;
    if (first) {
        const DownRec mine = plan->down[i / kTopK][1 + i % kTopK];
        if (mine.slot < 0) first = false;
        for (uint32_t j = 0; j < i; ++j)
            if (plan->down[j / kTopK][1 + j % kTopK].mat == mine.mat) first = false;
    }
    const uint64_t held = __ballot(first);
    if (i == 0) plan->n_union = __builtin_popcountll(held);
}

hipError_t launch_count_union(hipStream_t s, Plan *plan, uint32_t m) {
    hipLaunchKernelGGL(count_union_kernel, dim3(1), dim3(kWave), 0, s, plan, m);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Gate/up kernel.  Grid (width / (32 G) row groups, pair slots), four
// wavefronts per workgroup (with eight, one token's 9 slots made 72 workgroups
// for 256 CUs, and at 8 tokens one workgroup was resident per CU: 8.6 and 22.2
// us, 6.7 and 16.7 with four; 7.7 and 19.8 since the workgroups make their own
// routes, for which the route kernel takes 3.3 and 5.7 less); G = 64 / LPR lane groups per wavefront, LPR =
// the gate/up matrices' padded block count (hidden / 32 <= 64).  Lane group
// j of a wavefront owns 8 rows of both matrices: lane b loads block b of each
// row (16 nibble loads), the scales of its block for the 8 rows (one 16-byte
// load per matrix) and the activation record of block b of the slot's token,
// then reduces the 16 block products across the group (value 2n + u: row n,
// u = 0 gate, 1 up).  h = silu(gate) * up (weights.rs:241-259) meets in LDS
// and a half-wavefront per block writes it as xprep records for the down kernel.
// Held to 128 registers at LPR = 64 (136 without the bound), so that four
// workgroups are resident per CU instead of three: the 1152 of eight tokens take
// 1.1 rounds instead of 1.5; 40-layer verify step 1587 -> 1560 us there, 1045 ->
// 1027 at four tokens.  At LPR = 16 and 32 the bound would spill.
// ---------------------------------------------------------------------------
constexpr int kGateUpWaves = 4;
static_assert(kGateUpWaves == kRouteRecordWaves, "its workgroups also run route_record");
constexpr int kGateUpRows = 8;  // rows per lane group per matrix

template <int LPR, bool ROUTED>
__global__ __launch_bounds__(kGateUpWaves * kWave, LPR == 64 ? 4 : 1) void gate_up_kernel(
    LayerDev L, Plan *__restrict__ plan, const uint32_t *__restrict__ xprep, uint32_t *__restrict__ hprep,
    uint32_t rows_padded, uint32_t bp_down, RouteArgs rt) {
    constexpr int G = kWave / LPR;
    constexpr int RW = kGateUpRows * G;  // rows per wavefront per matrix
    constexpr int R = LPR / 16;          // copies of each reduced value
    __shared__ float s_h[kGateUpWaves * RW];
    const int slot = blockIdx.y;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const uint32_t j = (uint32_t)lane / LPR, b = (uint32_t)lane % LPR;
    const uint32_t r0 = (blockIdx.x * kGateUpWaves + wave) * RW;
    const uint8_t *mat_gate, *mat_up;
    uint32_t x[28];
    if constexpr (ROUTED) {
        __shared__ const uint8_t *s_mat[2];
        if (slot >= (int)rt.m * (kTopK + 1)) {  // below the matvecs: the routes' record
            const uint32_t t = (slot - rt.m * (kTopK + 1)) * gridDim.x + blockIdx.x;
            if (t < rt.m) route_record(L, rt.logits, rt.m, (int)t, wave, lane, plan, rt.ids, rt.w, rt.status);
            return;
        }
        const int tok = slot / (kTopK + 1), k = slot % (kTopK + 1);
        load_xrec(xprep + (size_t)tok * LPR * kXprepDwords, LPR, b, x);
        if (wave == 0) route_slot(L, rt.logits + (size_t)tok * (L.n_experts + 1), k, lane, s_mat);
        __syncthreads();
        mat_gate = uniform_ptr(s_mat[0]);
        mat_up = uniform_ptr(s_mat[1]);
    } else {
        load_xrec(xprep + (size_t)slot * LPR * kXprepDwords, LPR, b, x);
        mat_gate = L.mats[0];
        mat_up = L.mats[1];
    }
    if (r0 < rows_padded) {
        const RowLane Wg = row_lane(mat_gate, LPR);
        const RowLane Wu = row_lane(mat_up, LPR);
        const uint32_t rl = r0 + j * kGateUpRows;
        uint4 ng[kGateUpRows], nu[kGateUpRows];
#pragma unroll
        for (int n = 0; n < kGateUpRows; ++n) {
            ng[n] = q4_signed(load_nibbles(Wg, rl + n, b));
            nu[n] = q4_signed(load_nibbles(Wu, rl + n, b));
        }
        const uint4 sg = load_scales(Wg, rl / 8, b), su = load_scales(Wu, rl / 8, b);
        if (b >= L.hidden / 32) x[24] = 0;  // padding block: contributes exactly 0
        __builtin_amdgcn_sched_barrier(0);  // every load in flight before any math
        float v[2 * kGateUpRows];
#pragma unroll
        for (int n = 0; n < kGateUpRows; ++n) {
            v[2 * n] = octet_scale(sg, n) * q4_block_dot(ng[n], x);
            v[2 * n + 1] = octet_scale(su, n) * q4_block_dot(nu[n], x);
        }
        const float gate = transpose_reduce<LPR, 2 * kGateUpRows>(v);
        const float up = dpp_f<0x100 + R>(gate);  // row_shl:R -> the up value
        const uint32_t q = (uint32_t)lane % LPR;
        if (q % (2 * R) == 0)
            s_h[wave * RW + j * kGateUpRows + q / (2 * R)] = (gate / (1.0f + expf(-gate))) * up;
    }
    __syncthreads();
    constexpr int kBlocks = kGateUpWaves * RW / 32;  // blocks of h per workgroup, one per half-wavefront
    if (2 * wave < kBlocks) {
        const int q = 2 * wave + (lane >> 5);
        const uint32_t blk = blockIdx.x * kBlocks + (uint32_t)q;
        prep_block32(s_h[(q < kBlocks ? q : 0) * 32 + (lane & 31)], lane & 31, q < kBlocks && blk < L.width / 32,
                     hprep + (size_t)slot * bp_down * kXprepDwords, bp_down, blk, PlainStore());
    }
}

hipError_t launch_gate_up(hipStream_t s, const LayerDev &L, uint32_t slots, Plan *plan,
                          const uint32_t *xprep, uint32_t *hprep, const RouteArgs &rt) {
    const MatrixDims g = matrix_dims(L.width, L.hidden);
    const MatrixDims dn = matrix_dims(L.hidden, L.width);
    const uint32_t G = kWave / g.lpr;
    const uint32_t rows_per_group = kGateUpWaves * kGateUpRows * G;
    dim3 grid((g.rows_padded + rows_per_group - 1) / rows_per_group, slots);
    grid.y += route_record_rows(rt.m, grid.x);
    dim3 block(kGateUpWaves * kWave);
#define TQF_GU(LPR)                                                                                              \
    {                                                                                                            \
        if (rt.m)                                                                                                \
            hipLaunchKernelGGL((gate_up_kernel<LPR, true>), grid, block, 0, s, L, plan, xprep, hprep, g.rows_padded, \
                               dn.blocks_padded, rt);                                                            \
        else                                                                                                     \
            hipLaunchKernelGGL((gate_up_kernel<LPR, false>), grid, block, 0, s, L, plan, xprep, hprep, g.rows_padded, \
                               dn.blocks_padded, rt);                                                            \
    }
    if (g.blocks_padded == 16) TQF_GU(16)
    else if (g.blocks_padded == 32) TQF_GU(32)
    else if (g.blocks_padded == 64) TQF_GU(64)
    else return hipErrorInvalidValue;
#undef TQF_GU
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Down kernel.  Grid (hidden / (8 G) row groups, tokens), one wavefront per
// down record of the token (nine in a layer).  Lane group j owns 8 consecutive
// rows of the record's matrix; lane b reads block b of each (LPR = the padded
// block count of the width, <= 64) against block b of the slot's h records.
// The workgroup weights each by its coefficient (shared: sigmoid gate; routed:
// route weight) and adds them in the reference's order, shared expert first
// (experts/mod.rs:1609-1630), then the residual (runtime.rs:802) when given.
// Bound by its latencies (records, weights, records of h, dot, sum).  All of a
// token's records in one workgroup need no hand-off between workgroups: with
// four slots a workgroup, whose partials the last one of a row group added up,
// it took 6.1 / 14.1 us at 1 / 8 tokens, with all of them in one 5.5 / 10.6,
// and 1.3 us less at one token with the parts of octets that launch_down takes.
// ---------------------------------------------------------------------------
// ROWS: rows per lane group, an octet or a part of one (see launch_down).
template <int LPR, int ROWS>
__global__ __launch_bounds__((kTopK + 1) * kWave) void down_kernel(LayerDev L, const Plan *__restrict__ plan,
                                                                   const uint32_t *__restrict__ hprep,
                                                                   const float *resid, float *out) {
    constexpr int RW = ROWS * (kWave / LPR);  // rows per workgroup
    __shared__ float red[kTopK + 1][RW];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int lane = threadIdx.x % kWave;
    const uint32_t j = (uint32_t)lane / LPR, b = (uint32_t)lane % LPR;
    const uint32_t t = blockIdx.y, r0 = blockIdx.x * RW, H = L.hidden;
    const DownRec rec = load_down(&plan->down[t][wave]);
    const uint32_t r = threadIdx.x;
    if (rec.slot < 0) {  // routing failed: every wavefront leaves, the residual goes on unchanged
        if (resid && r < RW && r0 + r < H) out[(size_t)t * H + r0 + r] = resid[(size_t)t * H + r0 + r];
        return;
    }
    const float res = resid && r < RW && r0 + r < H ? resid[(size_t)t * H + r0 + r] : 0.0f;
    const RowLane W = row_lane(rec.mat, LPR);
    const uint32_t rl = r0 + j * ROWS;
    uint4 nib[ROWS];
#pragma unroll
    for (int n = 0; n < ROWS; ++n) nib[n] = q4_signed(load_nibbles(W, rl + n, b));
    uint4 sc = {};  // the scales of rows rl .. rl + ROWS - 1
    if constexpr (ROWS == 8) {
        sc = load_scales(W, rl / 8, b);
    } else {
        const auto *p = (const __attribute__((address_space(1))) uint32_t *)(W.base + (((size_t)(rl / 8) * 9 + 8) * LPR + b) * 16) + (rl & 7) / 2;
        sc.x = p[0];
        if constexpr (ROWS == 4) sc.y = p[1];
    }
    uint32_t x[28];
    load_xrec(hprep + (size_t)rec.slot * LPR * kXprepDwords, LPR, b, x);
    if (b >= L.width / 32) x[24] = 0;  // padding block: contributes exactly 0
    __builtin_amdgcn_sched_barrier(0);  // every load in flight before any math
    float a[ROWS];
#pragma unroll
    for (int n = 0; n < ROWS; ++n) a[n] = octet_scale(sc, n) * q4_block_dot(nib[n], x);
    const float v = rec.coef * transpose_reduce<LPR, ROWS>(a);
    if (reduced_first_copy<LPR, ROWS>(lane)) red[wave][j * ROWS + reduced_index<LPR, ROWS>(lane)] = v;
    __syncthreads();
    if (r < RW && r0 + r < H) {
        float sum = red[0][r];
        for (uint32_t w = 1; w < blockDim.x / kWave; ++w) sum += red[w][r];
        out[(size_t)t * H + r0 + r] = resid ? res + sum : sum;
    }
}

hipError_t launch_down(hipStream_t s, const LayerDev &L, uint32_t m, uint32_t per_token, const Plan *plan,
                       const uint32_t *hprep, const float *resid, float *out) {
    const MatrixDims dn = matrix_dims(L.hidden, L.width);
    // The fewest rows a workgroup that still make at most one workgroup per CU
    // (256): 2048 rows of width 512 at one token are 64 workgroups of whole
    // octets, whose nine wavefronts then share four SIMDs for 72 block products
    // a lane.  40-layer stack at one token 681 -> 627 us with two rows a lane
    // group, 16 layer calls 263 -> 243; whole octets from three tokens on.
    const uint32_t groups = kWave / dn.lpr;
    uint32_t rows = 2;
    while (rows < 8 && dn.rows_padded / (rows * groups) * m > 256) rows *= 2;
    const dim3 grid((dn.rows_padded + rows * groups - 1) / (rows * groups), m), block(per_token * kWave);
#define TQF_DOWN(LPR)                                                                                             \
    {                                                                                                            \
        if (rows == 2)                                                                                           \
            hipLaunchKernelGGL((down_kernel<LPR, 2>), grid, block, 0, s, L, plan, hprep, resid, out);            \
        else if (rows == 4)                                                                                      \
            hipLaunchKernelGGL((down_kernel<LPR, 4>), grid, block, 0, s, L, plan, hprep, resid, out);            \
        else                                                                                                     \
            hipLaunchKernelGGL((down_kernel<LPR, 8>), grid, block, 0, s, L, plan, hprep, resid, out);            \
    }
    if (dn.blocks_padded == 16) TQF_DOWN(16)
    else if (dn.blocks_padded == 32) TQF_DOWN(32)
    else if (dn.blocks_padded == 64) TQF_DOWN(64)
    else return hipErrorInvalidValue;
#undef TQF_DOWN
    return hipGetLastError();
}

}  // namespace tqf
