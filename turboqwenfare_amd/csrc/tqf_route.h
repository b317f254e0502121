// tqf_route.h -- routing inside the gate/up kernels (gfx950).
//
// The route kernel leaves every token's router logits (and the shared expert's
// gate logit) in memory; the kernels after it make the routes from them, each
// workgroup the one that it needs.  Its first load is then the logits instead
// of a plan, and no workgroup waits for another.  While the route kernel's
// first workgroup polled the others' logits, made the routes and wrote a plan,
// that kernel took 7.7 / 10.4 / 14.0 us at 1 / 4 / 8 tokens, now 4.4 / 6.1 /
// 8.3; the routing costs the gate/up kernels 1.0 (Q4_0: 6.7 -> 7.7 us) at one
// token, 1.7 (Q4_K: 12.2 -> 13.9) at four and 3.1 (Q4_0: 16.7 -> 19.8) at
// eight.  Only one wavefront a workgroup routes, up to its own expert, and
// what the other kernels read is recorded by workgroups of their own: with
// every matvec's first workgroup recording and checking it took 27 us at
// eight tokens.
#pragma once

#include "tqf_device.h"
#include "tqf_internal.h"

namespace tqf {

// The softmax probabilities of one token's router logits, lane l holding
// experts l + 64 i (RouterResult::from_logits, experts/mod.rs:134-167).
__device__ __forceinline__ void route_probabilities(const float (&lv)[4], int lane, uint32_t E, float (&p)[4]) {
    const float mx = wave_max4(lv);
    float ssum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t e = (uint32_t)lane + 64u * i;
        p[i] = e < E ? expf(lv[i] - mx) : 0.0f;
        ssum += p[i];
    }
    ssum = group_reduce<64>(ssum, AddOp());
#pragma unroll
    for (int i = 0; i < 4; ++i) p[i] = ((uint32_t)lane + 64u * i < E) ? p[i] / ssum : -1.0f;
}

__device__ __forceinline__ const uint8_t *uniform_ptr(const uint8_t *p) {
    const uint64_t v = (uint64_t)(uintptr_t)p;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v), hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
    return (const uint8_t *)(uintptr_t)(((uint64_t)hi << 32) | lo);
}

// A token's logits as the routing wavefronts hold them.
__device__ __forceinline__ void load_logits(const float *lt, int lane, uint32_t E, float (&lv)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) lv[i] = (uint32_t)lane + 64u * i < E ? lt[lane + 64 * i] : -INFINITY;
}

// The gate/up workgroup's own routing: matvec k of a token with logits lt (0:
// the shared expert, 1 + i: the route's i-th expert in stable descending
// order, ties to the lower id).  Wavefront 0 leaves the matvec's two matrices
// in s_mat.  Logits that are not finite select some expert of the layer; the
// down records then say that the call failed, and its work goes unread.
__device__ __forceinline__ void route_slot(const LayerDev &L, const float *lt, int k, int lane, const uint8_t **s_mat) {
    const uint32_t E = L.n_experts;
    float lv[4];
    const uint8_t *mg[4], *mu[4];
    load_logits(lt, lane, E, lv);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t e = (uint32_t)lane + 64u * i;
        const uint32_t ec = k == 0 ? E : (e < E ? e : 0);
        mg[i] = L.mats[ec * 3];
        mu[i] = L.mats[ec * 3 + 1];
    }
    int id = 0;
    if (k > 0) {
        float p[4], psel[kTopK];
        int ids[kTopK] = {};
        route_probabilities(lv, lane, E, p);
        top8_by_probability(p, lane, E, psel, ids, k);
#pragma unroll
        for (int i = 0; i < kTopK; ++i)
            if (i == k - 1) id = ids[i];
        id = id < (int)E ? id : 0;
    }
    const int sel = id >> 6;
    if (lane == (id & 63)) {
        s_mat[0] = sel == 0 ? mg[0] : sel == 1 ? mg[1] : sel == 2 ? mg[2] : mg[3];
        s_mat[1] = sel == 0 ? mu[0] : sel == 1 ? mu[1] : sel == 2 ? mu[2] : mu[3];
    }
}

// One workgroup of kRouteRecordWaves wavefronts per token: its down records and route outputs.  All but the
// first wavefront see whether the logits of all tokens are finite; one that
// is not fails the call, every down record says so, and token 0's workgroup
// reports it.
constexpr int kRouteRecordWaves = 4;
__device__ __forceinline__ void route_record(const LayerDev &L, const float *logits, uint32_t m, int tok, int wave, int lane,
                                             Plan *plan, uint16_t *ids_out, float *w_out, int32_t *status_out) {
    const uint32_t E = L.n_experts;
    const float *lt = logits + (size_t)tok * (E + 1);
    bool fin = true;
    float psel[kTopK] = {}, gate = 0.0f;
    int ids[kTopK] = {};
    if (wave == 0) {
        float lv[4], p[4];
        load_logits(lt, lane, E, lv);
        gate = lt[E];
        route_probabilities(lv, lane, E, p);
        top8_by_probability(p, lane, E, psel, ids);
    } else {
        constexpr int kCheckers = kRouteRecordWaves - 1, kEach = (kMaxTokens + kCheckers - 1) / kCheckers;
        float lv[kEach][4];
#pragma unroll
        for (int i = 0; i < kEach; ++i) {
            const uint32_t t = (uint32_t)(wave - 1 + kCheckers * i);
            load_logits(logits + (size_t)(t < m ? t : 0) * (E + 1), lane, E, lv[i]);
        }
#pragma unroll
        for (int i = 0; i < kEach; ++i)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if ((uint32_t)lane + 64u * c < E && !(fabsf(lv[i][c]) <= 3.402823466e38f)) fin = false;
    }
    const bool bad = __syncthreads_or(!fin);
    if (wave != 0 || lane > kTopK) return;
    // lane k: matvec k
    float total = -0.0f, pk = 0.0f;
    int id = (int)E;
#pragma unroll
    for (int i = 0; i < kTopK; ++i) {
        total += psel[i];
        if (i == lane - 1) {
            pk = psel[i];
            id = ids[i];
        }
    }
    if (bad) {
        plan->down[tok][lane].slot = -1;
        if (tok == 0 && lane == 0 && status_out) *status_out = TQF_HIP_ERR_ROUTER;
        return;
    }
    const float coef = lane > 0 ? pk / total : 1.0f / (1.0f + expf(-gate));
    plan->down[tok][lane] = DownRec{L.mats[id * 3 + 2], tok * (kTopK + 1) + lane, coef};
    if (lane > 0) {
        if (ids_out) ids_out[tok * kTopK + lane - 1] = (uint16_t)id;
        if (w_out) w_out[tok * kTopK + lane - 1] = coef;
    }
}

// The workgroups of a gate/up grid of `x` columns that record the routes: so
// many rows below its matvecs'.
inline uint32_t route_record_rows(uint32_t m, uint32_t x) { return (m + x - 1) / x; }

}  // namespace tqf
