// Routing kernels: the MoE gate (fused2.gate_topk, fused2.py:418-471; model.MoE.gate, model.py:391-404) and the
// expert bucketing of (token, expert) pairs (cukern.moe_dispatch -> p2p.cu:90-132).
//
// gate_topk_kernel: one workgroup per token row. Scores -> softmax / sigmoid / sqrt(softplus), + bias for the
// selection only, TOPK rounds of a block-wide arg-max (lowest index wins ties, fused2.py:441), weights
// renormalised (+1e-20) and scaled.
// moe_dispatch_kernel: one workgroup per 1024 pairs. Histogram (LDS atomics), exclusive scan over experts, then a
// STABLE scatter: pairs keep ascending pair order within an expert (the reference's order is arbitrary,
// p2p.cu:91-93; a stable order makes the tables reproducible); within a wave the rank among same-expert lanes
// comes from ballots, across waves from per-wave counts in LDS.
#include "common.h"
#include "gate.h"

#define GATE_MAX_PER_LANE 32   // E <= 2048 scores per row, held in registers (32 per lane)

template <int PER>
__global__ void __launch_bounds__(64) gate_topk_kernel(const float* __restrict__ scores, long long lds, int nparts, long long pstride,
                                                       const float* __restrict__ bias, int E, float temp, int topk, float route_scale,
                                                       int mode, int norm, int* __restrict__ eid, float* __restrict__ wt) {
    int ki;
    float kw;
    gate_row_wave<PER>(scores + (long long)blockIdx.x * lds, nparts, pstride, bias, E, temp, topk, route_scale, mode, norm, &ki, &kw);
    if (threadIdx.x < topk) {
        eid[(long long)blockIdx.x * topk + threadIdx.x] = ki;
        wt[(long long)blockIdx.x * topk + threadIdx.x] = kw;
    }
}

extern "C" int dsv41_gate_topk(const float* scores, long long lds, const float* bias, int B, int E, float temp, int topk, float route_scale,
                               int score_func, int norm, int* eid, float* wt, int nparts, long long part_stride, void* stream) {
    if (!scores || !eid || !wt || B < 0 || E < 1 || E > 64 * GATE_MAX_PER_LANE || topk < 1 || topk > 64 || topk > E || score_func < 0 ||
        score_func > 2 || lds < E || nparts < 1 || (nparts > 1 && part_stride < (long long)B * lds))
        return DSV41_EINVAL;
    if (B == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
#define GATE_LAUNCH(PER) \
    gate_topk_kernel<PER><<<B, 64, 0, st>>>(scores, lds, nparts, part_stride, bias, E, temp, topk, route_scale, score_func, norm, eid, wt)
    if (E <= 64 * 4) GATE_LAUNCH(4);
    else if (E <= 64 * 6) GATE_LAUNCH(6);
    else if (E <= 64 * 8) GATE_LAUNCH(8);
    else GATE_LAUNCH(GATE_MAX_PER_LANE);
#undef GATE_LAUNCH
    return (int)hipGetLastError();
}

// ------------------------------------------------------------------------------------------ dispatch
#define DISP_THREADS 1024
#define DISP_WAVES (DISP_THREADS / WAVE)
#define DISP_MAX_E 512

// exclusive scans of v and w over the block's threads; the block totals land in *tv, *tw. One barrier: the scans of a wave run
// in registers, and every thread adds the earlier waves' totals itself.
__device__ __forceinline__ void block_exclusive_scan2(int& v, int& w, int2* s_tot, int* tv, int* tw) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int iv = v, iw = w;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int a = __shfl_up(iv, o), b = __shfl_up(iw, o);
        iv += lane >= o ? a : 0;
        iw += lane >= o ? b : 0;
    }
    if (lane == 63) s_tot[wave] = make_int2(iv, iw);
    __syncthreads();
    int sv = 0, sw = 0, pv = 0, pw = 0;
#pragma unroll
    for (int i = 0; i < DISP_WAVES; ++i) {
        const int2 t = s_tot[i];
        pv += i < wave ? t.x : 0;
        pw += i < wave ? t.y : 0;
        sv += t.x;
        sw += t.y;
    }
    *tv = sv;
    *tw = sw;
    v = pv + iv - v;
    w = pw + iw - w;
}

// Workgroup b places the pairs of chunk b = [b * 1024, b * 1024 + 1024). It reads every expert id (a few tens of
// KB, L2-resident) to histogram both all pairs and the pairs before its chunk, so each workgroup knows where its
// pairs go without a second launch or scratch memory: pos = start[e] + (pairs of e before the chunk) + (rank of
// the pair among the chunk's pairs of e), ranks from ballots within a wave and per-wave counts across waves.
// Workgroup 0 also writes the groups; the padding of the tables is shared out by chunk. Bound by chains, not bytes: the ids are
// read four at a time, a pair counts in one of two histograms (before the chunk, or not), and the scans take one barrier. The rank loop (up
// to 64 experts in a wave) reads its leader's id by readlane and the earlier waves' counts all at once: 288 pairs 12.6 -> 9.4 us,
// 16,384 pairs 17.4 -> 15.7.
__global__ void __launch_bounds__(DISP_THREADS) moe_dispatch_kernel(const int* __restrict__ eid, const float* __restrict__ wt, int n, int topk,
                                                                    int E, int gmax, int* __restrict__ tok_sorted, float* __restrict__ wt_sorted,
                                                                    int* __restrict__ inv, int* __restrict__ grp_expert, int* __restrict__ grp_start,
                                                                    int* __restrict__ n_groups) {
    __shared__ int s_count[DISP_MAX_E], s_before[DISP_MAX_E], s_start[DISP_MAX_E];
    __shared__ __align__(4) unsigned short s_wcnt[DISP_WAVES][DISP_MAX_E];
    __shared__ int2 s_tot[DISP_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int c0 = blockIdx.x * DISP_THREADS;
    for (int e = tid; e < E; e += DISP_THREADS) { s_count[e] = 0; s_before[e] = 0; }
#pragma unroll
    for (int i = 0; i < DISP_WAVES * DISP_MAX_E / 2; i += DISP_THREADS) ((uint32_t*)&s_wcnt[0][0])[i + tid] = 0u;
    __syncthreads();
    for (int p = tid; p < n; p += 4 * DISP_THREADS) {
        int e[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = p + i * DISP_THREADS < n ? eid[p + i * DISP_THREADS] : -1;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (e[i] >= 0 && e[i] < E) atomicAdd(p + i * DISP_THREADS < c0 ? &s_before[e[i]] : &s_count[e[i]], 1);
    }
    __syncthreads();
    // exclusive scans of the counts and of the group counts over experts (one expert per thread: E <= 512)
    const int cnt_e = tid < E ? s_count[tid] + s_before[tid] : 0;
    int start_e = cnt_e, gbase_e = (cnt_e + gmax - 1) / gmax, total_pairs, total_groups;
    block_exclusive_scan2(start_e, gbase_e, s_tot, &total_pairs, &total_groups);
    if (tid < E) s_start[tid] = start_e;
    __syncthreads();
    // stable scatter of this chunk
    const unsigned long long below = (lane == 63) ? ~0ull >> 1 : ((1ull << lane) - 1ull);
    const int p = c0 + tid;
    const bool valid = p < n;
    const int e = valid ? eid[p] : -1;
    const bool real = valid && e >= 0 && e < E;
    int rank = 0, cnt = 0;
    unsigned long long todo = __ballot(real);
    while (todo) {
        const int leader = __ffsll((long long)todo) - 1;
        const int le = __builtin_amdgcn_readlane(e, leader);   // the leader is the same for the whole wave: no trip through LDS
        const unsigned long long m = __ballot(real && e == le);
        if (real && e == le) { rank = __popcll(m & below); cnt = __popcll(m); }
        todo &= ~m;
    }
    if (real && rank == 0) s_wcnt[wave][e] = (unsigned short)cnt;
    __syncthreads();
    if (real) {
        int before = 0;
#pragma unroll
        for (int w = 0; w < DISP_WAVES; ++w) before += w < wave ? (int)s_wcnt[w][e] : 0;   // all reads in flight at once
        const int pos = s_start[e] + s_before[e] + before + rank;
        tok_sorted[pos] = p / topk;
        wt_sorted[pos] = wt ? wt[p] : 1.f;
        inv[p] = pos;
    }
    if (valid && !real) inv[p] = -1;   // a dropped pair (id outside [0, E)) has no sorted slot
    // groups of <= gmax pairs per expert, then padding (p2p.cu:124-131). The padding starts at the number of
    // placed pairs (n when every id is valid, as in the reference), so the last group ends there; the sorted slots
    // past it (left by dropped pairs) hold token 0 with weight 0.
    if (valid && p >= total_groups) {
        grp_expert[p] = -1;
        grp_start[p] = total_pairs;
    }
    if (valid && p >= total_pairs) {
        tok_sorted[p] = 0;
        wt_sorted[p] = 0.f;
    }
    if (blockIdx.x != 0) return;
    for (int g = 0; g * gmax < cnt_e; ++g) {   // tid < E
        grp_expert[gbase_e + g] = tid;
        grp_start[gbase_e + g] = start_e + g * gmax;
    }
    if (tid == 0) {
        grp_start[total_groups] = total_pairs;
        grp_start[n] = total_pairs;
        if (n_groups) *n_groups = total_groups;
    }
}

extern "C" int dsv41_moe_dispatch(const int* eid, const float* wt, int n, int topk, int E, int gmax, int* tok_sorted, float* wt_sorted,
                                  int* inv, int* grp_expert, int* grp_start, int* n_groups, void* stream) {
    if (!eid || !tok_sorted || !wt_sorted || !inv || !grp_expert || !grp_start || n < 0 || topk < 1 || E < 1 || E > 512 || gmax < 1)
        return DSV41_EINVAL;
    const int blocks = n > 0 ? (n + DISP_THREADS - 1) / DISP_THREADS : 1;   // one workgroup writes the (empty) tables when n == 0
    moe_dispatch_kernel<<<blocks, DISP_THREADS, 0, (hipStream_t)stream>>>(eid, wt, n, topk, E, gmax, tok_sorted, wt_sorted, inv, grp_expert, grp_start,
                                                                          n_groups);
    return (int)hipGetLastError();
}
