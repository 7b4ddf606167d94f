// Routing pieces shared by the MoE kernels and by the one-row grouped GEMV, whose workgroups
// redo the last, cheap part of the one-token routing themselves (ordered sum of the segment
// sums, top-k, sorted positions) instead of waiting for a launch that does it once.
//
// Arithmetic contract of the routing (the reference has no MoE arithmetic; the shapes follow
// crates/berth-plan/src/shape.rs:64-69 and plan.rs:24-59):
//   logits[e] = sum over 64-row segments of (sum_h x[h] * wr[h][e], fp32 fma in row order),
//               segments added in order, then + bias[e];
//   top-k on the logits, largest first, ties to the lowest expert index;
//   weights = exp(logit - max) normalised over the selected k (renorm) or over all experts.
#pragma once

#include "exl3_decode.cuh"
#include "hadamard.cuh"

namespace berth {

// one unit of grouped work: rows [row0, row0 + nrows) of the expert-sorted order
struct GroupProblem {
    int expert;
    int row0;
    int nrows;
    int lone;           // 1: all rows of the expert, at most sixteen (whichever list it is in)
};
constexpr int kLoneRows = 16;

constexpr int kRouteSeg = 64;       // rows of the router weight per partial sum
constexpr int kRouteTT = 4;         // tokens per route workgroup
constexpr int kRouteCounterStride = 32;   // words between the arrival counters of neighbouring token groups
constexpr int kMaxExperts = 1024;
constexpr int kMaxTopK = 32;

struct PermuteParams {
    const int32_t* idx;     // [P] expert of each (token, slot) pair, P = T * k; distinct within a token
    int32_t* offsets;       // [E + 1]
    int32_t* perm;          // [R] sorted position -> pair (pair / k = token)
    int32_t* inv;           // [P] pair -> sorted position
    int32_t* row_expert;    // [R] sorted position -> expert
    int32_t* counts;        // [3] number of VALU problems, small MFMA problems, big MFMA problems
    GroupProblem* vprob;
    GroupProblem* mprob;    // <= small_rows rows each
    GroupProblem* bprob;    // <= 128 rows each
    int T, k, E;
    int use_valu;           // 1: every expert is one VALU problem (<= 8 rows each); 0: MFMA problems: an
                            // expert's rows go to big problems of 128 and the rest to small ones of <= 32
    int shared_rows;        // 1: rows P .. P + T - 1 belong to an always-on expert with index E (token order)
    int small_rows;         // rows of a small problem: 32, or 16
    int big_min;            // a remainder of at least this many rows becomes a (partial) big problem
};

struct RouteParams {
    const _Float16* x;      // [T][H]
    const _Float16* wr;     // [H][E]
    const float* bias;      // [E] or null
    float* parts;           // [T][nseg][E]
    unsigned* counters;     // [ceil(T / kRouteTT)]
    int32_t* idx;           // [T][k]
    float* w;               // [T][k]
    float* logits;          // [T][E] or null
    int32_t* idx_out;       // [T][k], [T][k] or null: the caller's own copies of idx and w, written with them (two
    float* w_out;           // copy launches behind the layer cost 4 us of a one-token layer's 30, 8 under a profiler)
    int T, H, E, k, nseg, renorm;
    // one token only: the wave that selected the experts also sorts them and writes
    // what the permute kernel would (sort.perm != nullptr), saving its launch
    PermuteParams sort;
};

// Top-k of one token by one wave: lane holds the logits of experts lane + 64 i.
// Largest first, ties to the lowest expert index; weights exp(l - max) normalised
// over the selected k (renorm) or over all experts.
constexpr int kRoutePer = kMaxExperts / 64;

__device__ __forceinline__ float lane_value(float v, int lane_index)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane_index));
}

// the largest value of the wave (no NaN among them): one v_max_f32 with a DPP operand per distance, row
// sums handed on to the next row, the result read from the last lane.  (A DPP operand may be read two
// instructions after it was written at the earliest: the s_nop.)
__device__ __forceinline__ float wave_max(float v)
{
#define BERTH_MAX_STEP(ctrl) "s_nop 1\n\tv_max_f32_dpp %0, %0, %0 " ctrl "\n\t"
    asm volatile(BERTH_MAX_STEP("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf")
                 BERTH_MAX_STEP("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf")
                 BERTH_MAX_STEP("row_half_mirror row_mask:0xf bank_mask:0xf")
                 BERTH_MAX_STEP("row_mirror row_mask:0xf bank_mask:0xf")
                 BERTH_MAX_STEP("row_bcast:15 row_mask:0xa bank_mask:0xf")
                 BERTH_MAX_STEP("row_bcast:31 row_mask:0xc bank_mask:0xf")
                 "s_nop 1"
                 : "+v"(v));
#undef BERTH_MAX_STEP
    return lane_value(v, 63);
}
// PER: how many of the lane's registers can hold experts (ceil(E / 64) rounded up to 2, 8 or 16).
// A lane sorts its own experts once (largest first, ties in order of their index); a round is then the
// maximum of the lanes' heads, a ballot and one step of the winner's list.  What bounds it is one
// wave's chain of dependent instructions: looking through all registers for the maximum and again for
// its holder in every round, the top 8 of 128 took 2.0 us of a routing launch and the top 10 of 512 4.8;
// 1.4 and 3.3 now.
template <int PER>
__device__ __forceinline__ int route_topk_n(const float (&lg)[kRoutePer], int lane, const RouteParams& p, int t,
                                            bool store = true)
{
    float val[PER];
    int who[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        // registers past the last expert sort behind the lane's real ones and, with a higher index, lose
        // every tie; a logit that is no number ranks with minus infinity
        val[i] = lane + 64 * i < p.E && lg[i] == lg[i] ? lg[i] : -INFINITY;
        who[i] = lane + 64 * i;
    }
    // odd-even transposition: swaps neighbours only, so equal values keep their order
#pragma unroll
    for (int r = 0; r < PER; ++r) {
#pragma unroll
        for (int i = r & 1; i + 1 < PER; i += 2) {
            // (values, not elements, to choose from: a choice of elements becomes an indexed read of the array)
            const float a = val[i], b = val[i + 1];
            const int wa = who[i], wb = who[i + 1];
            const bool swap = b > a;
            val[i] = swap ? b : a;
            val[i + 1] = swap ? a : b;
            who[i] = swap ? wb : wa;
            who[i + 1] = swap ? wa : wb;
        }
    }
    float sel_logit = 0.0f;         // lane j keeps the logit of slot j
    int sel_idx = 0;
#pragma unroll 1
    for (int j = 0; j < p.k; ++j) {
        const float bv = wave_max(val[0]);
        // the lowest expert index among the lanes that hold it (nearly always one)
        unsigned long long holders = __builtin_amdgcn_ballot_w64(val[0] == bv);
        int bi = 0x7fffffff;
        do {
            bi = min(bi, __builtin_amdgcn_readlane(who[0], (int)__builtin_ctzll(holders)));
            holders &= holders - 1;
        } while (holders);
        const bool mine = who[0] == bi;
#pragma unroll
        for (int i = 0; i + 1 < PER; ++i) {
            const float a = val[i], b = val[i + 1];
            const int wa = who[i], wb = who[i + 1];
            val[i] = mine ? b : a;
            who[i] = mine ? wb : wa;
        }
        val[PER - 1] = mine ? -INFINITY : val[PER - 1];     // (an empty list loses every tie)
        who[PER - 1] = mine ? 0x7fffffff : who[PER - 1];
        if (lane == j) { sel_logit = bv; sel_idx = bi; }
    }
    // lane j is wave-uniform here: v_readlane instead of a round trip through the LDS crossbar
    const float mx = lane_value(sel_logit, 0);
    float ev = (lane < p.k) ? expf(sel_logit - mx) : 0.0f;
    float denom = 0.0f;
    if (p.renorm) {
        for (int j = 0; j < p.k; ++j) denom += lane_value(ev, j);       // slot order
    } else {
        float loc = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + 64 * i < p.E) loc += expf(lg[i] - mx);
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) loc += __shfl_xor(loc, d, 64);
        denom = loc;
    }
    if (store && lane < p.k) {
        const size_t at = (size_t)t * p.k + lane;
        const float weight = ev / denom;
        p.idx[at] = sel_idx;
        p.w[at] = weight;
        if (p.idx_out) p.idx_out[at] = sel_idx;
        if (p.w_out) p.w_out[at] = weight;
    }
    return sel_idx;     // lane j < k: expert of slot j
}

__device__ __forceinline__ int route_topk(const float (&lg)[kRoutePer], int lane, const RouteParams& p, int t)
{
    if (p.E <= 128) return route_topk_n<2>(lg, lane, p, t);         // workgroup-uniform
    if (p.E <= 512) return route_topk_n<8>(lg, lane, p, t);
    return route_topk_n<kRoutePer>(lg, lane, p, t);
}

// One token: what moe_permute_kernel writes, by the wave that holds the selection
// (lane j < k has the expert of slot j; the k experts are distinct).  Sorted position
// of slot j = number of selected experts with a smaller index; every expert is one
// single-row VALU problem; an always-on expert (shared_rows) takes row k.
__device__ __forceinline__ void route_sort_one_token(const PermuteParams& q, int lane, int sel_idx)
{
    const int k = q.k;
    int rank = 0;
    for (int j = 0; j < k; ++j) {
        const int other = __builtin_amdgcn_readlane(sel_idx, j);
        rank += (lane < k && other < sel_idx) ? 1 : 0;
    }
    if (lane < k) {
        q.perm[rank] = lane;
        q.inv[lane] = rank;
        q.row_expert[rank] = sel_idx;
        q.vprob[rank] = GroupProblem{sel_idx, rank, 1, 0};
    }
    // offsets[e] = number of selected experts below e
    for (int e0 = 0; e0 <= q.E; e0 += 64) {         // wave-uniform loop: every lane takes part in the exchanges
        const int e = e0 + lane;
        int below = 0;
        for (int j = 0; j < k; ++j) below += (__builtin_amdgcn_readlane(sel_idx, j) < e) ? 1 : 0;
        if (e <= q.E) q.offsets[e] = below;
    }
    if (lane == 0) {
        if (q.shared_rows) {
            q.perm[k] = 0;
            q.row_expert[k] = q.E;
            q.vprob[k] = GroupProblem{q.E, k, 1, 0};
        }
        q.counts[0] = k + (q.shared_rows ? 1 : 0);
        q.counts[1] = 0;
        q.counts[2] = 0;
    }
}


// One token, at most 128 experts: the routing's last part by one wave, from the segment sums
// parts[seg][e] that moe_route_segments_kernel left in memory: logits (segments added in
// order, bias), top-k, and the sorted position of every selected expert (lane j < k: expert of
// slot j and its sorted position).  Every wave that calls this gets the same bits; the wave
// with `writer` set also stores the routing results (logits, idx, w, and what the sort of the
// one token writes).  `summed` is called ahead of the selection.
struct RouteOneToken {
    int sel;
    int rank;
};

template <typename F>
__device__ __forceinline__ RouteOneToken route_one_token(const RouteParams& p, int lane, bool writer, F summed)
{
    float lg[kRoutePer];
#pragma unroll
    for (int i = 0; i < kRoutePer; ++i) lg[i] = -INFINITY;
    // Both of a lane's experts and their biases at once, 32 segments at a time (segments past the end re-read the last
    // one, experts past the end the last one, and are ignored); the adds stay in segment order.  One after the other,
    // the biases last, they were up to four round trips to memory instead of one.
    const uint32_t at[2] = {(uint32_t)min(lane, p.E - 1), (uint32_t)min(lane + 64, p.E - 1)};
    float v[2] = {0.0f, 0.0f}, bias[2] = {0.0f, 0.0f};
    for (int s0 = 0; s0 < p.nseg; s0 += 32) {
        float part[2][32];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (i == 1 && p.E <= 64) break;
#pragma unroll
            for (int j = 0; j < 32; ++j) part[i][j] = as_global(p.parts + (size_t)min(s0 + j, p.nseg - 1) * p.E)[at[i]];
        }
        if (s0 == 0 && p.bias) {
#pragma unroll
            for (int i = 0; i < 2; ++i) bias[i] = as_global(p.bias)[at[i]];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (i == 1 && p.E <= 64) break;
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const float nv = v[i] + part[i][j];
                v[i] = s0 + j < p.nseg ? nv : v[i];
            }
        }
    }
    summed();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int e = lane + 64 * i;
        if (e < p.E) {
            lg[i] = p.bias ? v[i] + bias[i] : v[i];
            if (writer && p.logits) p.logits[e] = lg[i];
        }
    }
    RouteOneToken r;
    r.sel = route_topk_n<2>(lg, lane, p, 0, writer);
    if (writer && p.sort.perm) route_sort_one_token(p.sort, lane, r.sel);
    r.rank = 0;
    for (int j = 0; j < p.k; ++j) {
        const int other = __builtin_amdgcn_readlane(r.sel, j);
        r.rank += other < r.sel ? 1 : 0;
    }
    return r;
}

// the expert whose sorted position is `want_rank` (the always-on expert E for want_rank == k)
__device__ __forceinline__ int route_expert_at(const RouteParams& p, const RouteOneToken& r, int lane, int want_rank)
{
    if (want_rank >= p.k) return p.E;
    const unsigned long long holder = __builtin_amdgcn_ballot_w64(lane < p.k && r.rank == want_rank);
    return __builtin_amdgcn_readlane(r.sel, (int)__builtin_ctzll(holder));
}

}  // namespace berth
