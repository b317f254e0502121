// tqf_grouped.hip -- prefill-shaped grouped expert GEMM on the matrix cores.
//
// T tokens, each routed to 8 experts with weights (ids/w given), through one
// prepared MoE layer's routed experts:
//   y[t] = sum_k w[t,k] * down_e(silu(gate_e x_t) * up_e x_t),  e = ids[t,k]
// which is the routed part of Qwen36ResidentMoe::forward
// (experts/mod.rs:1617-1630) over LoadedQwen36Expert::forward
// (model/qwen36/weights.rs:566-610), batched over tokens the way
// Qwen36StreamingMoe::forward_batch (experts/mod.rs:1540-1577) serves a
// prefill chunk.
//
// Kernels (stream-ordered, no host round trip):
//   plan     counting sort of the T*8 (token, k) pairs by expert (stable in
//            pair order), the tile list; x put in MFMA operand order;
//   gate_up  grid (F / 64 column blocks, tiles): gate and up on bf16 MFMA,
//            SwiGLU, h stored as bf16 hi + lo in operand order;
//   down     grid (H / 128 column blocks, tiles): down on bf16 MFMA;
//   combine  y[t] = sum_k w[t,k] * out[pos(t,k)] in route order.
// (Dealing a tile's column blocks to one XCD, so that they share its
// activation rows in one L2, measured no faster.)
//
// Exactness of the weights.  A Q4_0 block is (q - 8) * d with a per-row,
// per-32-column f16 scale d.  Rounding (q - 8) * d to bf16 would cost 8 bits,
// so the MFMA B operand is the exact bf16 value 16 + q, the bias is removed by
// starting each block's accumulation from sum_k x_k * (-24), and the block's
// fp32 result is scaled by d and accumulated in fp32.  Every product is exact
// (bf16 x bf16 fits fp32); rounding happens only in the fp32 sums.  (128 + q
// needs one shift less per operand, but starts the sums from -136 times the
// activations: 3.3e-6 of y against 64 bits, 2.5e-6 with 16 + q.)
// Activations: x is bf16 on entry (exact); h is split into bf16 hi + lo
// (16 significant bits), so down runs two MFMAs per block.
//
// v_mfma_f32_16x16x32_bf16 lane layout (l = lane, g = l / 16): A holds row l %
// 16, k = 8g .. 8g + 7; B holds column l % 16, the same k; D holds column l %
// 16, rows 4g + v for v = 0..3.  Both operands take the block's elements in the
// order of the nibbles: k = 8g + i is element 4g + i for i < 4 (low nibbles of
// qs dword g), 16 + 4g + i - 4 for i >= 4 (its high nibbles).
#include <hip/hip_runtime.h>

#include "tqf_device.h"
#include "tqf_internal.h"

namespace tqf {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / kWave;

__device__ __forceinline__ f32x4 mfma(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Four qs bytes of a block -> the B operand 16 + q of their eight elements:
// the low nibbles (elements 4g .. 4g + 3 for dword g), then the high nibbles
// (elements 16 + 4g ..).  16 + q is bf16 0x4180 | q << 3.
// `bit7` is 0x80808080 from a register (a shift and one v_and_or_b32 for four
// nibbles: two literals do not fit one instruction).
__device__ __forceinline__ bf16x8 biased_operand(uint32_t c, uint32_t bit7) {
    constexpr uint32_t kHi = 0x41414141u, kSel01 = 0x04010400u, kSel23 = 0x04030402u;
    const uint32_t l = ((c << 3) & 0x78787878u) | bit7, h = ((c >> 1) & 0x78787878u) | bit7;
    const u32x4 v = {__builtin_amdgcn_perm(kHi, l, kSel01), __builtin_amdgcn_perm(kHi, l, kSel23),
                     __builtin_amdgcn_perm(kHi, h, kSel01), __builtin_amdgcn_perm(kHi, h, kSel23)};
    return __builtin_bit_cast(bf16x8, v);
}

}  // namespace

// Activations in the order of the MFMA operands.  The MFMA of a Q4 block reads
// the block's 32 activations as four 16-byte pieces, piece g (for lane group
// g) holding elements 4g .. 4g + 3 and 16 + 4g .. 16 + 4g + 3, which is the
// order the nibbles of dword g come in.  A permuted row is [block][set][4
// pieces]: one set for x, two (bf16 hi, lo) for h.  Beside it -24 times each
// block's sum, [block][row], for the bias correction.  x is permuted by extra
// workgroups of the plan launch, which end before the plan's own; h is written
// this way by gate/up.
constexpr float kBias = -24.0f;
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xFFFF0000u); }
__device__ __forceinline__ uint32_t bf16_bits(float v) { return __builtin_bit_cast(uint16_t, (__bf16)v); }
// Piece i of x [T x 32 blocks]: i = 4 (blocks t + block) + piece.
__device__ __forceinline__ void permute_piece(const uint16_t *x, uint32_t i, uint32_t blocks, uint32_t T, uint4 *xp,
                                              float *x_sums) {
    const uint16_t *src = x + (size_t)(i >> 2) * 32 + (i & 3) * 4;  // x is 2-byte aligned only
    uint32_t v[4];
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const uint16_t *p = src + (d >> 1) * 16 + (d & 1) * 2;
        v[d] = (uint32_t)p[0] | ((uint32_t)p[1] << 16);
    }
    xp[i] = make_uint4(v[0], v[1], v[2], v[3]);
    float s = ((bf16_lo(v[0]) + bf16_hi(v[0])) + (bf16_lo(v[1]) + bf16_hi(v[1]))) +
              ((bf16_lo(v[2]) + bf16_hi(v[2])) + (bf16_lo(v[3]) + bf16_hi(v[3])));
    s += dpp_f<kDppXor1>(s);  // the block's four pieces are adjacent lanes
    s += dpp_f<kDppXor2>(s);
    const uint32_t q = i >> 2, t = q / blocks;
    if ((i & 3) == 0) x_sums[(size_t)(q - t * blocks) * T + t] = kBias * s;
}

// ---- plan: counting sort of the (token, k) pairs by expert ------------------
// Positions are stable in pair order (p = 8 t + k).  Workgroup b places the
// 1024 pairs p = 1024 b .. and needs nothing from the others: it counts all
// ids itself (LDS atomics, pairs before and after its own batch apart), its
// wavefronts rank equal experts of the batch with ballots, and the first lane
// of each peer group writes the group's size to the count slot of its
// wavefront, which one thread per expert turns into exclusive prefixes.  A
// pair's position is base[e] (the exclusive scan of all counts) + the pairs
// of e before the batch + its slot's prefix + its rank.  Workgroup 0 writes
// the tile list.  An expert's c pairs make ceil(c / tile_m) tiles of equal size,
// rounded up to 16 rows (the MFMA's); an entry is {first position, e | rows
// << 16}.  The tiles of experts with more than 16 pairs come first: they take
// longest.
// Bound by its serial steps, not by bytes.  One workgroup that walked the
// batches took 8.4-10.8 us at 4096 pairs and 74-88 us at 32768; this takes
// 5.0-6.1 and 8.9-11.0 us.
__device__ __forceinline__ int tile_rows(int c, int tile_m) {
    const int n = (c + tile_m - 1) / tile_m;
    return n ? ((c + n - 1) / n + 15) / 16 * 16 : 16;
}
__global__ __launch_bounds__(kPlanThreads) void gg_plan_kernel(
    const uint16_t *__restrict__ ids, uint32_t pairs, uint32_t E, int tile_m, int32_t *__restrict__ pos_of_pair,
    int32_t *__restrict__ pair_of_pos, uint2 *__restrict__ tiles, int32_t *__restrict__ n_tiles,
    int32_t *__restrict__ status, const uint16_t *__restrict__ x, uint32_t x_blocks, uint4 *__restrict__ xp,
    float *__restrict__ x_sums) {
    const uint32_t plan_blocks = (pairs + kPlanThreads - 1) / kPlanThreads;
    if (blockIdx.x >= plan_blocks) {
        const uint32_t i = (blockIdx.x - plan_blocks) * kPlanThreads + threadIdx.x;
        const uint32_t T = pairs / kTopK;
        if (i < 4 * x_blocks * T) permute_piece(x, i, x_blocks, T, xp, x_sums);
        return;
    }
    __shared__ uint16_t cnt[kPlanWaves][256];  // this batch, per wavefront: count of expert e, then its prefix
    __shared__ int32_t before[256], after[256], total[256], base[256], tbase[256];
    __shared__ int32_t s_bad;
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const uint64_t below = (1ull << lane) - 1;
    const uint32_t b0 = blockIdx.x * kPlanThreads;
    if (tid < 256) {
        before[tid] = 0;
        after[tid] = 0;
    }
    for (int i = tid; i < kPlanWaves * 256 / 8; i += kPlanThreads)
        reinterpret_cast<uint4 *>(&cnt[0][0])[i] = make_uint4(0, 0, 0, 0);
    if (tid == 0) s_bad = 0;
    __syncthreads();
    const uint32_t p = b0 + tid;
    uint32_t key = 256u;  // no expert
    if (p < pairs) {
        const uint32_t e = ids[p];
        if (e < E) key = e;
        else s_bad = 1;
    }
    if (plan_blocks > 1) {  // the other batches' ids, eight loads in flight per thread
        for (uint32_t r = tid; r < pairs; r += 8 * kPlanThreads) {
            uint32_t e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t q = r + (uint32_t)i * kPlanThreads;
                e[i] = q < pairs ? ids[q] : 0xFFFFu;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const uint32_t q = r + (uint32_t)i * kPlanThreads;
                if (q >= pairs) continue;
                if (e[i] >= E) s_bad = 1;
                else if (q - b0 >= (uint32_t)kPlanThreads) atomicAdd(q < b0 ? &before[e[i]] : &after[e[i]], 1);
            }
        }
    }
    const uint64_t peers = match_peers(key);
    const int rank = __popcll(peers & below);
    if (key < 256u && rank == 0) cnt[wave][key] = (uint16_t)__popcll(peers);
    __syncthreads();
    if (s_bad) {
        if (blockIdx.x == 0 && tid == 0) {
            *n_tiles = 0;
            if (status) *status = TQF_HIP_ERR_INVALID;
        }
        return;
    }
    if (tid < 256) {
        int s = 0;
#pragma unroll
        for (int v = 0; v < kPlanWaves; ++v) {
            const int c = cnt[v][tid];
            cnt[v][tid] = (uint16_t)s;
            s += c;
        }
        total[tid] = before[tid] + s + after[tid];
    }
    __syncthreads();
    if (wave == 0) {  // exclusive scans of pair and tile counts, 4 experts per lane
        int c[4], tc[4], s = 0, ts = 0;  // tile counts: over 16 pairs in the low half, others in the high half
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c[j] = total[4 * lane + j];
            tc[j] = (c[j] + tile_m - 1) / tile_m;
            if (c[j] <= 16) tc[j] <<= 16;
            s += c[j];
            ts += tc[j];
        }
        int is = s, its = ts;
#pragma unroll
        for (int d = 1; d < kWave; d *= 2) {
            const int x = __shfl_up(is, d), y = __shfl_up(its, d);
            if (lane >= d) {
                is += x;
                its += y;
            }
        }
        const int all = __shfl(its, kWave - 1), large = all & 0xFFFF;
        int o = is - s, to = its - ts;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            base[4 * lane + j] = o;
            tbase[4 * lane + j] = tc[j] >> 16 ? large + (to >> 16) : to & 0xFFFF;
            o += c[j];
            to += tc[j];
        }
        if (blockIdx.x == 0 && lane == 0) *n_tiles = large + (all >> 16);
    }
    __syncthreads();
    if (key < 256u) {
        const int pos = base[key] + before[key] + cnt[wave][key] + rank;
        pos_of_pair[p] = pos;
        pair_of_pos[pos] = (int32_t)p;
    }
    if (blockIdx.x == 0 && tid < (int)E) {
        const int c = total[tid], step = tile_rows(c, tile_m);
        for (int i = 0; i * step < c; ++i) {
            const int rows = c - i * step < step ? c - i * step : step;
            tiles[tbase[tid] + i] = make_uint2((uint32_t)(base[tid] + i * step), (uint32_t)tid | ((uint32_t)rows << 16));
        }
    }
}

// ---- the tiled GEMMs -----------------------------------------------------------
// A workgroup of 4 wavefronts owns one tile (<= 32 pairs of one expert), a
// wavefront two 16-row MFMA subtiles of weights (in gate/up the same 16 rows of
// gate and up, so SwiGLU stays in registers) for the full K.
//
// B operands are 16 + q in bf16.  The zero point and that bias (24 together)
// are cancelled by starting each block's MFMA from -24 times the block's
// activation sum; the result is scaled by the block's f16 scale in fp32.
//
// Everything comes through LDS with direct copies (buffer_load ... lds), so no
// register holds a byte on its way and every weight request is a whole 128-byte
// line: K advances in steps of 8 Q4 blocks, in which a row's nibbles are 128
// contiguous bytes.  (Loading 4 blocks of 16 rows per instruction straight to
// registers took 64-byte requests; their second halves came after the line had
// left the L1, and issuing one group's loads took 1,600-23,000 clocks against
// 2,500-3,500 for its arithmetic.)  Each wavefront copies its own weights, one
// step ahead of its arithmetic where its stage is free; the activations and
// their sums are copied by all of them, one stage per step (two with h's two
// sets), between two barriers.  Stages are single: three or four workgroups per
// CU run through each other's waits, and hide them better than two with
// double-buffered stages do.
//
// Per 16 x 16 x 32 unit the vector ALU has 4 fmas (16 clocks) and 9 / MS
// instructions for the B operand and the scale (MS: 16-row subtiles of the
// tile); an MFMA is 16 clocks of the matrix cores and takes 8 of vector issue
// (measured; v_permlane*_swap takes 8 as well); the LDS reads are about 11
// clocks of the CU's LDS.  So tiles of 16 rows are bound by the weight stream,
// long lists of full tiles by vector issue and LDS together.
// Tiles have up to 32 rows, up to 64 where experts average 32 pairs or more
// (half the operand work and weight traffic per row, against more workgroups in
// flight: 1024 even tokens 232 us, 512 Zipf tokens 152 us a layer).
// Measured, gate/up and down kernels in one run each (rocprof, medians): 37
// Zipf tokens 40.9 + 28.2 -> 32.4 + 20.5 us, 512 116 + 80 -> 89 + 56 us, 4096
// even tokens 411 + 286 -> 374 + 274 us against 32-row tiles of 8 wavefronts
// that staged weights through registers.  At 4096 tokens the clock falls under
// sustained load: the same kernels take 304-374 and 229-274 us, so figures of
// one run each do not rank what lies closer.  Tried on the way there and not
// kept: double-buffered stages at two workgroups per CU (439 + 305), K started
// at a step of the workgroup's own (no change).  Open: 64-row tiles of 8
// wavefronts with 4 subtiles each and the next step's weights in flight took 334
// + 265 us in a run of their own, not in turn with these (and 38 us for a lone
// tile, which a short prompt would wait for).
constexpr int kStepBlocks = 8;
constexpr int kGemmWaves = 4;
constexpr int kSub = 2;  // weight subtiles per wavefront

typedef __amdgpu_buffer_rsrc_t Desc;  // loads past `bytes` return zero
__device__ __forceinline__ Desc make_desc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}
// 16 (4) bytes per lane from descriptor + voff + soff to LDS byte lds + 16 (4) x
// lane.  Builtins: the wait states between a write of m0 or of a descriptor's
// register and the load are the compiler's to count, which it cannot inside an
// assembly string (there, one kernel had three where five are needed).
typedef __attribute__((address_space(3))) void lds_void;
__device__ __forceinline__ void copy16(Desc d, uint32_t voff, uint32_t soff, uint32_t lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (lds_void *)lds, 16, voff, soff, 0, 0);
}
__device__ __forceinline__ void copy4(Desc d, uint32_t voff, uint32_t soff, uint32_t lds) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(d, (lds_void *)lds, 4, voff, soff, 0, 0);
}
// This wavefront's LDS reads and writes are done, then the workgroup's; publish:
// its copies too.
__device__ __forceinline__ void rendezvous() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void publish() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
typedef __attribute__((address_space(3))) uint8_t lds_byte;
template <typename T>
__device__ __forceinline__ T lds_load(uint32_t at) {
    return *(const __attribute__((address_space(3))) T *)(at);
}

struct GroupedArgs {
    const uint8_t *const *mats;
    MatrixDims dims;        // of this GEMM's matrices
    uint32_t mat_bytes;
    uint32_t K, N;          // dims.cols, and the output's columns
    const uint8_t *act;     // permuted activations [act_rows][K]
    const float *sums;      // [K / 32][act_rows]
    uint32_t act_rows;
    const int32_t *pair_of_pos;
    const uint2 *tiles;
    const int32_t *n_tiles;
    uint8_t *h;             // gate/up: permuted h, its sums [N / 32][h_rows]
    float *h_sums;
    uint32_t h_rows;
    float *out;             // down
};

// GATE_UP: matrices 0 and 1 of the expert against x rows (the pair's token);
// else matrix 2 against h rows (the position).
//
// LDS.  Per wavefront a weight stage: 4 octets x [8 rows][8 blocks][16 B], where
// slot c of row r of octet o holds block c ^ r ^ (o & 1) (fragment reads free of
// bank conflicts), then 4 octets x [8 blocks][8 rows] f16 scales.  Then the
// activation stage, [block pair (one set) or block][row octet] x 1 KiB of
// [block of pair or set][4 pieces][8 rows][16 B], and the sums, [block][rows].
template <bool GATE_UP, int MS>
struct TileGemm {
    static constexpr int NW = kGemmWaves, NS = kSub;
    static constexpr int kMats = GATE_UP ? 2 : 1, kSets = GATE_UP ? 1 : 2;  // matrices; activation sets
    static constexpr int kPerMat = NS / kMats;                              // subtiles per matrix
    static constexpr int kCols = 16 * kPerMat;                              // output columns per wavefront
    static constexpr int kParts = kSets;              // activation stages per step: 8 blocks of one set, 4 of two
    static constexpr int kBlocks = kStepBlocks / kParts;
    static constexpr int kOctets = 2 * MS;            // row octets
    static constexpr int kRowSets = (kOctets + NW - 1) / NW;  // octets a wavefront copies
    static constexpr int kFence = kSets == 1 ? 8 : 2;
    static constexpr int kCopies = 4;                 // 1 KiB activation copies per octet and stage
    static constexpr uint32_t kWStage = NS * (2048 + 256), kAStage = kCopies * kOctets * 1024, kSumStage = kBlocks * MS * 64;
    static constexpr uint32_t kLds = NW * kWStage + kAStage + kSumStage;

    uint32_t w_lds, a_lds, sum_lds;  // this wavefront's weights; the workgroup's activations and sums
    Desc ws[kMats], as, cs;
    uint32_t wv[2], sv, row16;       // weight offsets by octet parity, scale offset; bytes of a row's nibbles
    uint32_t av[kRowSets], cv, act_rows;
    int wave, lane;

    __device__ __forceinline__ TileGemm(const GroupedArgs &p, uint32_t lds, uint32_t pos0, uint32_t e, uint32_t rows,
                                        uint32_t col0, int wave_, int lane_)
        : wave(wave_), lane(lane_) {
        w_lds = lds + wave * kWStage;
        a_lds = lds + NW * kWStage;
        sum_lds = a_lds + kAStage;
#pragma unroll
        for (int k = 0; k < kMats; ++k) ws[k] = make_desc(load_global_ptr(p.mats + e * 3 + (GATE_UP ? k : 2)), p.mat_bytes);
        act_rows = p.act_rows;
        as = make_desc(p.act, act_rows * p.K * 2 * kSets);
        cs = make_desc(p.sums, act_rows * (p.K / 32) * 4);
        row16 = p.dims.blocks_padded * 16;
        const uint32_t r = lane >> 3, c = lane & 7, oct0 = col0 >> 3;
#pragma unroll
        for (uint32_t o = 0; o < 2; ++o) wv[o] = (oct0 * 9 + r) * row16 + ((c ^ r ^ o) & 7) * 16;
        sv = ((oct0 + r) * 9 + 8) * row16 + c * 16;
        // tile rows past the last take the first: read, not used
        auto act_row = [&](uint32_t m) {
            const uint32_t pos = pos0 + (m < rows ? m : 0u);
            return GATE_UP ? (uint32_t)p.pair_of_pos[pos] / kTopK : pos;
        };
#pragma unroll
        for (int i = 0; i < kRowSets; ++i)
            av[i] = act_row(((wave + i * NW) % kOctets) * 8 + (lane & 7)) * (p.K * 2 * kSets) + (lane >> 3) * 16;
        cv = act_row(lane) * 4;
    }

    __device__ __forceinline__ void copy_weights(uint32_t step) const {
        const uint32_t at = step * (kStepBlocks * 16);
#pragma unroll
        for (int o = 0; o < 2 * NS; ++o)
            copy16(ws[o / (2 * kPerMat)], wv[o & 1], at + (o % (2 * kPerMat)) * 9 * row16, w_lds + o * 1024);
#pragma unroll
        for (int m = 0; m < kMats; ++m)
            if (lane < 16 * kPerMat) copy16(ws[m], sv, at, w_lds + NS * 2048 + m * (kPerMat * 256));
    }
    // Activation stage `at` of K (kBlocks blocks): [block pair (one set) or
    // block][row octet] x 1 KiB, and the blocks' sums.
    __device__ __forceinline__ void copy_act(uint32_t at) const {
        constexpr int kShare = NW / kOctets > 1 ? NW / kOctets : 1;  // wavefronts that share an octet
#pragma unroll
        for (int i = 0; i < kRowSets; ++i) {
            const int octet = kShare == 1 ? wave + i * NW : wave % kOctets;
            if (kShare == 1 && octet >= kOctets) break;
#pragma unroll
            for (int c = 0; c < kCopies; ++c)
                if (kShare == 1 || c % kShare == wave / kOctets)
                    copy16(as, av[i], at * (kCopies * 128) + c * 128, a_lds + (c * kOctets + octet) * 1024);
        }
#pragma unroll
        for (int b = 0; b < kBlocks; b += NW)
            if (lane < 16 * MS) copy4(cs, cv, (at * kBlocks + b + wave) * act_rows * 4, sum_lds + (b + wave) * (MS * 64));
    }
    // This lane's dword and scale of block b and subtile k in a weight stage:
    // row n = lane % 16 of the subtile, dword lane / 16.
    __device__ __forceinline__ uint32_t weight(int b, int k) const {
        const uint32_t o = (lane >> 3) & 1, r = lane & 7;
        return lds_load<uint32_t>(((w_lds + o * 1024 + r * 128 + ((r ^ o) << 4) + (lane >> 4) * 4) ^ (b << 4)) + k * 2048);
    }
    __device__ __forceinline__ uint16_t scale(int b, int k) const {
        return lds_load<uint16_t>(w_lds + NS * 2048 + ((lane >> 3) & 1) * 128 + (lane & 7) * 2 + b * 16 + k * 256);
    }
    // The blocks of activation stage `part` of a step.
    __device__ __forceinline__ void compute(int part, uint32_t bit7, f32x4 (&acc)[MS][NS]) const {
        const uint32_t grp = lane >> 4, o = (lane >> 3) & 1, r = lane & 7;
        const uint32_t al = a_lds + o * 1024 + grp * 128 + r * 16, cl = sum_lds + grp * 16;
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) {
            const int b = kBlocks * part + j;
            bf16x8 af[kSets][MS];
            f32x4 t0[MS];
#pragma unroll
            for (int i = 0; i < MS; ++i) {
                t0[i] = lds_load<f32x4>(cl + j * (MS * 64) + i * 64);
#pragma unroll
                for (int a = 0; a < kSets; ++a) {
                    const int at = kSets == 1 ? (j >> 1) * kOctets * 1024 + (j & 1) * 512 : j * kOctets * 1024 + a * 512;
                    af[a][i] = __builtin_bit_cast(bf16x8, lds_load<u32x4>(al + at + i * 2048));
                }
            }
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                const bf16x8 bw = biased_operand(weight(b, k), bit7);
                const float s = f16_to_f32(scale(b, k));
                f32x4 t[MS];
#pragma unroll
                for (int i = 0; i < MS; ++i) t[i] = mfma(af[0][i], bw, t0[i]);
                if (kSets == 2) {
#pragma unroll
                    for (int i = 0; i < MS; ++i) t[i] = mfma(af[kSets - 1][i], bw, t[i]);
                }
#pragma unroll
                for (int i = 0; i < MS; ++i)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[i][k][v] = fmaf(s, t[i][v], acc[i][k][v]);
            }
            if (j % kFence == kFence - 1) __builtin_amdgcn_sched_barrier(0);  // bounds the reads the compiler moves up
        }
        // the sums are values here: moved past the next branch, they would keep
        // every MFMA result of the stage live
#pragma unroll
        for (int i = 0; i < MS; ++i)
#pragma unroll
            for (int k = 0; k < NS; ++k) asm volatile("" : "+v"(acc[i][k]));
    }

    __device__ __forceinline__ void run(uint32_t steps, f32x4 (&acc)[MS][NS]) const {
        uint32_t bit7;
        asm("v_mov_b32 %0, 0x80808080" : "=v"(bit7));
#pragma unroll
        for (int i = 0; i < MS; ++i)
#pragma unroll
            for (int k = 0; k < NS; ++k) acc[i][k] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        copy_weights(0);
        for (uint32_t s = 0; s < steps; ++s) {
#pragma unroll
            for (int part = 0; part < kParts; ++part) {
                if (part > 0 || s > 0) rendezvous();  // every wavefront has read the last stage
                copy_act(kParts * s + part);
                publish();
                compute(part, bit7, acc);
            }
            if (s + 1 < steps) {
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the weights are read before they are overwritten
                copy_weights(s + 1);
            }
        }
    }
};

// SwiGLU of column col0 + n of rows 16 i + 4 grp + v (n = lane % 16, grp = lane
// / 16) into the permuted h; even lanes store the hi parts of columns n, n + 1,
// odd lanes the lo parts of n - 1, n.  A 32-column block spans two wavefronts,
// whose halves of its sum meet in LDS (at ps, 64 floats per wavefront).
template <int MS>
__device__ __forceinline__ void store_h(const GroupedArgs &p, const f32x4 (&acc)[MS][kSub], uint32_t ps, uint32_t pos0,
                                        uint32_t rows, uint32_t col0, int wave, int lane) {
    const uint32_t n = lane & 15, grp = lane >> 4, blk = col0 >> 5;
    const uint32_t in_block = (n & 1) * 64 + (n >> 2) * 16 + (wave & 1) * 8 + (n & 2) * 2;
    rendezvous();  // every wavefront is done with the stages
#pragma unroll
    for (int i = 0; i < MS; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float g = acc[i][0][v], u = acc[i][1][v];
            const float hv = (g / (1.0f + expf(-g))) * u;
            const uint32_t hi = bf16_bits(hv), lo = bf16_bits(hv - bf16_lo(hi));
            float sum = bf16_lo(hi) + bf16_lo(lo);
            sum += dpp_f<kDppXor1>(sum);
            sum += dpp_f<kDppXor2>(sum);
            sum += dpp_f<kDppHalfMirror>(sum);
            sum += dpp_f<kDppMirror>(sum);
            const uint32_t hi1 = (uint32_t)dpp_i<kDppXor1>((int)hi), lo1 = (uint32_t)dpp_i<kDppXor1>((int)lo);
            const uint32_t r = 16 * i + 4 * grp + v;
            if (n == 0) *(__attribute__((address_space(3))) float *)(ps + (wave * 64 + r) * 4) = sum;
            if (r < rows)
                *reinterpret_cast<uint32_t *>(p.h + ((size_t)(pos0 + r) * (p.N >> 5) + blk) * 128 + in_block) =
                    n & 1 ? lo1 | (lo << 16) : hi | (hi1 << 16);
        }
    rendezvous();
    const uint32_t q = wave, r = lane;  // the workgroup's block q, row r
    if (q < kGemmWaves / 2 && r < rows) {
        const float s = lds_load<float>(ps + (2 * q * 64 + r) * 4) + lds_load<float>(ps + ((2 * q + 1) * 64 + r) * 4);
        p.h_sums[(size_t)(blk - (wave >> 1) + q) * p.h_rows + pos0 + r] = kBias * s;
    }
}
// Even lanes store subtile 0's columns n, n + 1, odd lanes subtile 1's n - 1, n.
template <int MS>
__device__ __forceinline__ void store_out(const GroupedArgs &p, const f32x4 (&acc)[MS][kSub], uint32_t pos0, uint32_t rows,
                                          uint32_t col0, int lane) {
    const uint32_t n = lane & 15, odd = n & 1;
#pragma unroll
    for (int i = 0; i < MS; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float got = dpp_f<kDppXor1>(odd ? acc[i][0][v] : acc[i][1][v]);
            const uint32_t r = 16 * i + 4 * (lane >> 4) + v;
            if (r < rows)
                *reinterpret_cast<float2 *>(p.out + (size_t)(pos0 + r) * p.N + col0 + odd * 16 + (n & 14)) =
                    odd ? make_float2(got, acc[i][1][v]) : make_float2(acc[i][0][v], got);
        }
}

template <bool GATE_UP, int MS>
__device__ __forceinline__ void tile_pass(const GroupedArgs &p, uint32_t lds, uint32_t pos0, uint32_t e, uint32_t rows,
                                          int wave, int lane) {
    using G = TileGemm<GATE_UP, MS>;
    const uint32_t col0 = (blockIdx.x * kGemmWaves + wave) * G::kCols;
    const G g(p, lds, pos0, e, rows, col0, wave, lane);
    f32x4 acc[MS][kSub];
    g.run(p.K / (32 * kStepBlocks), acc);
    if constexpr (GATE_UP) store_h<MS>(p, acc, g.a_lds, pos0, rows, col0, wave, lane);
    else store_out<MS>(p, acc, pos0, rows, col0, lane);
}

template <bool GATE_UP, int MAX_MS>
__global__ __launch_bounds__(kGemmWaves * kWave) __attribute__((amdgpu_waves_per_eu(MAX_MS == 2 ? 4 : 3,
                                                                                  MAX_MS == 2 ? 4 : 3))) void
gg_gemm_kernel(GroupedArgs p) {
    extern __shared__ uint4 gg_smem[];
    const uint32_t lds = (uint32_t)(uintptr_t)(lds_byte *)(uint8_t *)gg_smem;
    if ((int)blockIdx.y >= *p.n_tiles) return;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint2 tl = p.tiles[blockIdx.y];
    const uint32_t pos0 = __builtin_amdgcn_readfirstlane(tl.x), er = __builtin_amdgcn_readfirstlane(tl.y);
    const uint32_t e = er & 0xFFFFu, rows = er >> 16;
    if (MAX_MS == 4 && rows > 48) tile_pass<GATE_UP, MAX_MS>(p, lds, pos0, e, rows, wave, lane);
    else if (MAX_MS == 4 && rows > 32) tile_pass<GATE_UP, MAX_MS - 1>(p, lds, pos0, e, rows, wave, lane);
    else if (rows > 16) tile_pass<GATE_UP, 2>(p, lds, pos0, e, rows, wave, lane);
    else tile_pass<GATE_UP, 1>(p, lds, pos0, e, rows, wave, lane);
}

// ---- combine: y[t] = sum_k w[t,k] * out[pos(t,k)], k in route order ----------
__global__ __launch_bounds__(256) void gg_combine_kernel(const float *__restrict__ out,
                                                         const int32_t *__restrict__ pos_of_pair,
                                                         const int32_t *__restrict__ n_tiles,
                                                         const float *__restrict__ w, uint32_t T,
                                                         uint32_t H, float *__restrict__ y) {
    if (*n_tiles == 0) return;  // the plan rejected the routes (status is set)
    const uint32_t per_row = H / 4;
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (uint64_t)T * per_row) return;
    const uint32_t t = (uint32_t)(idx / per_row), c = (uint32_t)(idx % per_row) * 4;
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < kTopK; ++k) {
        const int pos = pos_of_pair[t * kTopK + k];
        const float wk = w[t * kTopK + k];
        const float4 v = load_global_f4(out + (size_t)pos * H + c);
        acc.x = acc.x + wk * v.x;
        acc.y = acc.y + wk * v.y;
        acc.z = acc.z + wk * v.z;
        acc.w = acc.w + wk * v.w;
    }
    *reinterpret_cast<float4 *>(y + (size_t)t * H + c) = acc;
}

// ---- host side ----------------------------------------------------------------
namespace {
size_t round256(size_t v) { return (v + 255) / 256 * 256; }
// Most rows of a tile: 64 where experts average at least 32 pairs.
int tile_m_for(uint32_t T, uint32_t E) { return T * kTopK >= 32 * E ? 64 : 32; }
uint32_t max_tiles_for(uint32_t T, uint32_t E) {
    const uint32_t P = T * kTopK;
    return P / tile_m_for(T, E) + (E < P ? E : P);
}

template <bool GATE_UP, int MAX_MS>
hipError_t launch_tiles(hipStream_t s, const GroupedArgs &p, uint32_t tiles) {
    using G = TileGemm<GATE_UP, MAX_MS>;
    static const hipError_t attr = hipFuncSetAttribute((const void *)gg_gemm_kernel<GATE_UP, MAX_MS>,
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::kLds);
    if (attr != hipSuccess) return attr;
    hipLaunchKernelGGL((gg_gemm_kernel<GATE_UP, MAX_MS>), dim3(p.N / (kGemmWaves * G::kCols), tiles), dim3(kGemmWaves * kWave),
                       G::kLds, s, p);
    return hipGetLastError();
}

template <bool GATE_UP>
hipError_t launch_grouped_gemm(hipStream_t s, const LayerDev &L, const GroupedBuffers &g) {
    const uint32_t P = g.tokens * kTopK;
    GroupedArgs p;
    p.mats = L.mats;
    p.dims = GATE_UP ? matrix_dims(L.width, L.hidden) : matrix_dims(L.hidden, L.width);
    p.mat_bytes = (uint32_t)layout_bytes(p.dims);
    p.K = GATE_UP ? L.hidden : L.width;
    p.N = GATE_UP ? L.width : L.hidden;
    p.act = GATE_UP ? g.x : g.h;
    p.act_rows = GATE_UP ? g.tokens : P;
    p.sums = GATE_UP ? g.x_sums : g.h_sums;
    p.pair_of_pos = g.pair_of_pos;
    p.tiles = g.tiles;
    p.n_tiles = g.n_tiles;
    p.h = g.h;
    p.h_sums = g.h_sums;
    p.h_rows = P;
    p.out = g.out;
    return tile_m_for(g.tokens, L.n_experts) == 64 ? launch_tiles<GATE_UP, 4>(s, p, g.max_tiles)
                                                   : launch_tiles<GATE_UP, 2>(s, p, g.max_tiles);
}

template <typename F>
void carve(uint32_t T, uint32_t E, uint32_t H, uint32_t W, F take) {
    const size_t P = (size_t)T * kTopK;
    take(P * 4);                                                // pos_of_pair
    take(P * 4);                                                // pair_of_pos
    take((size_t)max_tiles_for(T, E) * 8);                      // tiles
    take(256);                                                  // n_tiles
    take((size_t)T * H * 2);                                    // x, permuted
    take((size_t)T * H / 8);                                    // x_sums
    take(P * W * 4);                                            // h, permuted
    take(P * W / 8);                                            // h_sums
    take(P * H * 4);                                            // out
}
}  // namespace

size_t grouped_scratch_bytes(uint32_t T, uint32_t E, uint32_t H, uint32_t F) {
    size_t sum = 0;
    carve(T, E, H, F, [&](size_t bytes) { sum += round256(bytes); });
    return sum;
}

GroupedBuffers grouped_buffers(void *scratch, uint32_t T, uint32_t E, uint32_t H, uint32_t F) {
    uint8_t *part[9], *p = static_cast<uint8_t *>(scratch);
    int n = 0;
    carve(T, E, H, F, [&](size_t bytes) {
        part[n++] = p;
        p += round256(bytes);
    });
    GroupedBuffers g;
    g.tokens = T;
    g.max_tiles = max_tiles_for(T, E);
    g.pos_of_pair = reinterpret_cast<int32_t *>(part[0]);
    g.pair_of_pos = reinterpret_cast<int32_t *>(part[1]);
    g.tiles = reinterpret_cast<uint2 *>(part[2]);
    g.n_tiles = reinterpret_cast<int32_t *>(part[3]);
    g.x = part[4];
    g.x_sums = reinterpret_cast<float *>(part[5]);
    g.h = part[6];
    g.h_sums = reinterpret_cast<float *>(part[7]);
    g.out = reinterpret_cast<float *>(part[8]);
    return g;
}

hipError_t launch_grouped_plan(hipStream_t s, const uint16_t *ids, const uint16_t *x, uint32_t T, uint32_t E, uint32_t H,
                               const GroupedBuffers &g, int32_t *status) {
    const uint32_t pairs = T * kTopK, pieces = T * H / 8;
    const uint32_t blocks = (pairs + kPlanThreads - 1) / kPlanThreads + (pieces + kPlanThreads - 1) / kPlanThreads;
    hipLaunchKernelGGL(gg_plan_kernel, dim3(blocks), dim3(kPlanThreads), 0, s, ids, pairs, E, tile_m_for(T, E), g.pos_of_pair, g.pair_of_pos,
                       g.tiles, g.n_tiles, status, x, H / 32, reinterpret_cast<uint4 *>(g.x), g.x_sums);
    return hipGetLastError();
}

hipError_t launch_grouped_gate_up(hipStream_t s, const LayerDev &L, const GroupedBuffers &g) {
    return launch_grouped_gemm<true>(s, L, g);
}

hipError_t launch_grouped_down(hipStream_t s, const LayerDev &L, const GroupedBuffers &g) {
    return launch_grouped_gemm<false>(s, L, g);
}

hipError_t launch_grouped_combine(hipStream_t s, const GroupedBuffers &g, const float *w,
                                  uint32_t T, uint32_t H, float *y) {
    const uint64_t threads = (uint64_t)T * (H / 4);
    hipLaunchKernelGGL(gg_combine_kernel, dim3((uint32_t)((threads + 255) / 256)), dim3(256), 0, s,
                       g.out, g.pos_of_pair, g.n_tiles, w, T, H, y);
    return hipGetLastError();
}

}  // namespace tqf
