// Dense FP8 weights times bf16 activations: the reference's W8 / linear_w / oproj_a family
// (w8.py:57-124) behind cukern.fp8_gemm_tc and cukern.fp8_gemv (cukern.py:78-218).
//   out[t, n] = sum_k x[t, k] * w[n, k] * 2^(s[n / 32][k / 32] - 127)          fp32 accumulation
// w: float8_e4m3fn bytes [N][K]; s: E8M0 bytes [ceil(N/32)][K/32]. A bf16 activation times an E4M3 weight with a
// power-of-two scale is exact in fp32, as in the reference (exact decode to bf16, fp32 accumulation), so results
// differ from it only in the order of the fp32 additions.
//
// MFMA mapping (v_mfma_f32_16x16x32_bf16): the weights are the A operand (16 rows n), the activations the B
// operand (16 tokens). Lane l = 16 j + r holds 16 consecutive weight bytes of row r, k = 16 j .. 16 j + 15 of a
// 64-k chunk, decodes them with their block scale in the converter (v_cvt_scalef32_pk_bf16_fp8; e4m3 x 2^e is
// exact in bf16 over the normal range) and issues two MFMAs, one over the lower 8 k of every lane and one over
// the upper 8. Any fixed assignment of k to MFMA positions is valid while the activation lane holds the same k,
// so the weights need no k permutation (the reference stores a k-permuted order for its mma fragments,
// w8.py:21-37).
// Tiled layout [N/16][K/64][4][16][16 B]: the 16 bytes of lane l sit at byte 16 l of a 1 KiB tile, so a
// wave-load is one contiguous 1 KiB block. Natural layout: row-major with row stride ldw.
// One workgroup per 16-row block; its waves split K and add their partial tiles through LDS in wave order, so the
// result is deterministic and no workgroup waits for another. Every workgroup of a launch is meant to be resident at
// once (<= 128 VGPRs: two 512-thread workgroups per CU), which balances a grid of more row blocks than CUs. A K split
// across workgroups was measured and dropped: publishing partials needs a device-scope release, and its L2 write-back
// made each such workgroup cost microseconds.
#include "common.h"

struct Fp8Args {
    const uint8_t* W; long long ldw;     // bytes per row (natural layout); tiled: ldw == K
    const uint8_t* S; long long lds;     // E8M0 row stride in bytes (one row per 32 weight rows)
    int N, K, nk;                        // nk = K / 64 chunks
    const uint16_t* x; long long ldx;    // bf16 activations
    long long ldt;                       // element stride between the tokens of one output row set
    int M, gc;                           // output rows; gc > 0: row block nb reads x rows offset by (16 nb / gc)
    float* out; long long ldo;           // optional fp32 [M][ldo]
    uint16_t* outb; long long ldob;      // optional bf16 [M][ldob]
};

// bytes from x to the end of the last activation row a launch reads
static long long fp8_x_bytes(const Fp8Args& a) {
    const long long G = a.gc ? a.N / a.gc : 1;
    return ((a.M - 1) * a.ldt + (G - 1) * a.ldx + a.K) * 2;
}

template <int N>
struct Fp8Int {
    static constexpr int value = N;
};

template <int MT>
__device__ __forceinline__ void fp8_store(const Fp8Args& a, const v4f (&sum)[MT], int n0, int r, int t0 = 0) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int t = t0 + mt * 16 + r;
        if (t >= a.M) continue;
        const float v[4] = {sum[mt].x, sum[mt].y, sum[mt].z, sum[mt].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + i;
            if (n >= a.N) continue;
            if (a.out) a.out[(long long)t * a.ldo + n] = v[i];
            if (a.outb) a.outb[(long long)t * a.ldob + n] = (uint16_t)f32_to_bf16_bits(v[i]);
        }
    }
}

// WPG waves split the workgroup's chunk range; MT 16-token tiles share every weight tile (M <= 16 MT). RB row blocks
// per workgroup (16 RB rows): every activation load a wave makes then feeds RB weight tiles instead of one, so the
// vector memory pipe carries 2 / RB KiB of activations per KiB of weights instead of 2 KiB. Row blocks 2q and 2q + 1
// of a workgroup share their 32-row scale row (the first is even), and a row block past the last one reads the last
// one again and stores nothing. RB > 1 needs gc == 0 or gc % (16 RB) == 0 (one x offset for all the blocks).
template <int WPG, int PF, int MT, int TILED, int RB>
__global__ void __launch_bounds__(WPG * 64) fp8_gemm_kernel(const Fp8Args a) {
    __shared__ v4f s_red[WPG][RB * MT][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 15, j = lane >> 4;
    const int nbt = (a.N + 15) / 16;
    const int nb = blockIdx.x * RB;
    const int c0 = a.nk * wave / WPG, c1 = a.nk * (wave + 1) / WPG;
    const uint8_t* wp[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        const int nbr = min(nb + b, nbt - 1);
        const int row = min(nbr * 16 + r, a.N - 1);   // rows past N (natural layout) read row N-1, never stored
        wp[b] = TILED ? a.W + ((long long)nbr * a.nk + c0) * 1024 + lane * 16 : a.W + (long long)row * a.ldw + (long long)c0 * 64 + j * 16;
    }
    constexpr long long wstep = TILED ? 1024 : 64;
    constexpr int NS = (RB + 1) / 2;   // 32-row scale rows: row blocks 2q and 2q + 1 of the workgroup share one
    const uint8_t* sp8[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) sp8[q] = a.S + (long long)(min(nb + 2 * q, nbt - 1) >> 1) * a.lds + 2 * c0 + (j >> 1);
    const long long goff = a.gc ? (long long)((nb * 16) / a.gc) * a.ldx : 0;
    const uint16_t* xp[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
        const int t = min(mt * 16 + r, a.M - 1);   // token columns past M read row M-1, never stored
        xp[mt] = a.x + goff + (long long)t * a.ldt + (long long)c0 * 64 + j * 16;
    }
    v4f acc[RB][MT];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[b][mt] = v4f{0.f, 0.f, 0.f, 0.f};
    v4i A[PF][RB], X[PF][MT][2];
    int SB[PF][NS];
    pipelined<PF>(c1 - c0,
        [&](int s, int c) {
#pragma unroll
            for (int b = 0; b < RB; ++b) A[s][b] = __builtin_nontemporal_load((const v4i*)(wp[b] + (long long)c * wstep));
#pragma unroll
            for (int q = 0; q < NS; ++q) SB[s][q] = sp8[q][2 * c];
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                X[s][mt][0] = *(const v4i*)(xp[mt] + (long long)c * 64);
                X[s][mt][1] = *(const v4i*)(xp[mt] + (long long)c * 64 + 8);
            }
        },
        [&](int s) {
#pragma unroll
            for (int b = 0; b < RB; ++b) {
                v8bf16_t lo, hi;
                decode16(A[s][b], e8m0_to_f32((uint32_t)SB[s][b >> 1]), lo, hi);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    acc[b][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(v8bf16_t, X[s][mt][0]), acc[b][mt], 0, 0, 0);
                    acc[b][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(v8bf16_t, X[s][mt][1]), acc[b][mt], 0, 0, 0);
                }
            }
        });
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) s_red[wave][b * MT + mt][lane] = acc[b][mt];
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
        if (nb + b >= nbt) break;
        v4f sum[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
            sum[mt] = s_red[0][b * MT + mt][lane];
#pragma unroll
            for (int w = 1; w < WPG; ++w) sum[mt] += s_red[w][b * MT + mt][lane];
        }
        const int n0 = (nb + b) * 16 + 4 * j;   // the accumulator of lane l holds rows 4 (l / 16) .. +3, token l % 16
        fp8_store<MT>(a, sum, n0, r);
    }
}

// M <= 4 tokens (every wave owning at least one chunk): each wave first copies its own k range of the activations and of its row block's scale bytes into a
// private LDS region (no barrier: only the wave itself reads it), so the memory pipe carries nothing but the weight
// tiles while it streams them, and the prefetch slots hold weights only (deeper prefetch in fewer registers).
// LDS per wave: M x cpw x 128 B of activations + 2 cpw scale bytes + a 16-byte sink (cpw = chunks per wave, rounded up).
constexpr int FP8_XL_PIECES = 8;   // 16-byte activation pieces per lane: M x chunks per wave <= 64
__host__ __device__ constexpr int fp8_lds_region(int M, int cpw) { return M * cpw * 128 + ((2 * cpw + 15) & ~15) + 16; }

// One wave's part of the LDS-staged GEMV, with exactly P weight tiles in flight: the caller guarantees n >= P, so the
// prologue below is straight-line code and the wait counters track the activation loads exactly (a prologue behind
// a branch makes them wait for every load issued before the merge, draining the weight prefetch).
template <int P, int TILED>
__device__ __forceinline__ v4f fp8_lds_wave(const Fp8Args& a, int cpw, uint8_t* s_dyn, int wave, int lane, int c0, int n) {
    const int r = lane & 15, j = lane >> 4;
    const int nb = blockIdx.x;
    const int xrow = cpw * 64;                                          // bf16 elements per token row in LDS
    const int region = fp8_lds_region(a.M, cpw);
    uint16_t* xl = (uint16_t*)(s_dyn + (size_t)wave * region);
    uint8_t* sl = s_dyn + (size_t)wave * region + a.M * cpw * 128;
    uint8_t* sink = s_dyn + (size_t)wave * region + region - 16;       // target of the writes that carry nothing
    const long long goff = a.gc ? (long long)((nb * 16) / a.gc) * a.ldx : 0;
    // activations -> LDS: piece p of token t covers k = c0 * 64 + 8 q .. + 7 (q = p % (8 n)); every lane loads its
    // pieces first (clamped to a valid address), then stores them; pieces past the end go to the sink (a conditional
    // store would put a branch between the loads and their waits)
    const int per_tok = 8 * n, total = a.M * per_tok;
    v4i xr[FP8_XL_PIECES];
#pragma unroll
    for (int i = 0; i < FP8_XL_PIECES; ++i) {
        const int p = min(lane + 64 * i, total - 1);
        const int t = p / per_tok, q = p - t * per_tok;
        xr[i] = *(const v4i*)(a.x + goff + (long long)t * a.ldt + (long long)c0 * 64 + 8 * q);
    }
    const uint8_t* srow = a.S + (long long)(nb >> 1) * a.lds + 2 * c0;
    const int sb0 = srow[min(lane, 2 * n - 1)], sb1 = srow[min(lane + 64, 2 * n - 1)];
    const uint8_t* wp = TILED ? a.W + ((long long)nb * a.nk + c0) * 1024 + lane * 16
                              : a.W + (long long)min(nb * 16 + r, a.N - 1) * a.ldw + (long long)c0 * 64 + j * 16;
    constexpr long long wstep = TILED ? 1024 : 64;
    v4i A[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
        A[i] = __builtin_nontemporal_load((const v4i*)(wp + (long long)i * wstep));
        __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < FP8_XL_PIECES; ++i) {
        const int p = lane + 64 * i;
        const int t = p / per_tok, q = p - t * per_tok;
        *(v4i*)(p < total ? (uint8_t*)(xl + t * xrow + 8 * q) : sink) = xr[i];
    }
    *(lane < 2 * n ? sl + lane : sink) = (uint8_t)sb0;
    *(lane + 64 < 2 * n ? sl + lane + 64 : sink + 1) = (uint8_t)sb1;
    // other lanes of this wave read what these lanes wrote: keep the LDS reads after the writes
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const uint16_t* xt = xl + min(r, a.M - 1) * xrow + j * 16;         // token columns past M repeat row M-1
    const uint8_t* st = sl + (j >> 1);
    v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
    int ci = 0;
    pipeline_finish<P>(n,
        [&](int s, int c) { A[s] = __builtin_nontemporal_load((const v4i*)(wp + (long long)c * wstep)); },
        [&](int s) {
            v8bf16_t lo, hi;
            decode16(A[s], e8m0_to_f32((uint32_t)st[2 * ci]), lo, hi);
            const v4i X0 = *(const v4i*)(xt + ci * 64), X1 = *(const v4i*)(xt + ci * 64 + 8);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(v8bf16_t, X0), acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(v8bf16_t, X1), acc, 0, 0, 0);
            ++ci;
        });
    return acc;
}

template <int WPG, int PF, int TILED>
__global__ void __launch_bounds__(WPG * 64) fp8_gemv_lds_kernel(const Fp8Args a, int cpw) {
    extern __shared__ __align__(16) uint8_t s_dyn[];
    __shared__ v4f s_red[WPG][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = a.nk * wave / WPG, c1 = a.nk * (wave + 1) / WPG, n = c1 - c0;
    const v4f acc = n >= PF ? fp8_lds_wave<PF, TILED>(a, cpw, s_dyn, wave, lane, c0, n)
                  : n >= 4 ? fp8_lds_wave<4, TILED>(a, cpw, s_dyn, wave, lane, c0, n)
                           : fp8_lds_wave<1, TILED>(a, cpw, s_dyn, wave, lane, c0, n);
    s_red[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
    v4f sum[1] = {s_red[0][lane]};
#pragma unroll
    for (int w = 1; w < WPG; ++w) sum[0] += s_red[w][lane];
    fp8_store<1>(a, sum, blockIdx.x * 16 + 4 * (lane >> 4), lane & 15);
}

// ------------------------------------------------------------------------------------------ up to 64 rows: loader waves
// RB 16-row blocks x 16 MT tokens per workgroup. Waves 0 .. SW - 1 split K: each streams the weight tiles of its own range into
// registers, PW chunks ahead, and takes the activations of its chunk from LDS; waves SW .. SW + LW - 1 only load: they bring
// the SW chunks' activation rows of the next steps into LDS. A wave's loads complete in order, so in one wave the
// activations (from L2) would wait behind the weights (from HBM) issued before them, and the weights could be no further
// ahead than the activations, whose rows fill LDS; with waves of their own each side runs at its own depth.
// The activations are more bytes through a CU's load path than the weights (16 MT rows x 2 K against 16 RB x K), so they
// come as whole cache lines: one load takes 8 rows x 128 bytes (a 64-k chunk). LDS position s of row R holds the row's
// 16-byte piece s ^ (R >> 1), so the operand reads of 16 rows meet all banks once.
// Step s: chunk w * T + s of every stream wave w (T = ceil(nk / SW); chunks past the last one are skipped). Up to 48 tokens
// three or four steps' rows fit LDS and a step takes one barrier, for 64 two and two.
// Measured against fp8_gemm_kernel (median of 20 graph replays over copies larger than the last-level cache): 48 / 64 rows
// 5120 x 8192 30.6 -> 17.4 / 36.7 -> 21.5 us, 4608 x 5120 21.5 -> 13.0 / 25.8 -> 16.1, 1280 x 5120 19.0 -> 9.8 / 22.7 -> 13.1,
// 5120 x 2304 12.5 -> 8.1 / 14.5 -> 10.1. Eight chunks of weights in flight per wave instead of four changed nothing.
typedef __attribute__((address_space(3))) void fp8_lds_void;

template <int N>
__device__ __forceinline__ void fp8_wait_vm() {   // s_waitcnt vmcnt(N)
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}
__device__ __forceinline__ void fp8_wait_lds() { __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14)); }   // lgkmcnt(0)
__device__ __forceinline__ void fp8_barrier() {
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

constexpr int FS_SW = 8, FS_LW = 4, FS_THREADS = 64 * (FS_SW + FS_LW);

template <int PW, int NS, int MT, int RB, int TILED>
__device__ __forceinline__ void fp8_stream_block(const Fp8Args& a, const uint32_t x_bytes) {
    constexpr int SW = FS_SW, LW = FS_LW;
    constexpr int CH = 2 * MT * 1024, STAGE = SW * CH;   // a chunk's activations, a step's
    constexpr int PL = SW * 2 * MT / LW;                  // loads per loader wave and step
    constexpr bool ONE = NS >= 3;                         // one barrier per step: the stage of step s - 1 is refilled in step s
    static_assert(PL * (NS - 1) < 64 && PL * LW == SW * 2 * MT, "the loads in flight are counted in vmcnt");
    static_assert(SW * RB * MT * 1024 <= NS * STAGE, "the partial tiles fit the stages");
    extern __shared__ __align__(16) uint8_t s_dyn[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, j = lane >> 4;
    const int nbt = (a.N + 15) / 16, nb = blockIdx.x * RB;
    const int T = (a.nk + SW - 1) / SW;
    const long long goff = a.gc ? (long long)((nb * 16) / a.gc) * a.ldx : 0;
    v4f acc[RB][MT];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[b][mt] = v4f{0.f, 0.f, 0.f, 0.f};
    if (wave >= SW) {
        // loader wave: rows 8 q .. 8 q + 7 (q = 0 .. 2 MT - 1) of the chunks of stream waves l0 .. l0 + SW / LW - 1; rows past M
        // read row M - 1, chunks past the last one the last one (never used)
        const int l0 = (wave - SW) * (SW / LW);
        const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(a.x, x_bytes);
        uint32_t xoff[2 * MT];
#pragma unroll
        for (int q = 0; q < 2 * MT; ++q)
            xoff[q] = (uint32_t)((goff + (long long)min(8 * q + (lane >> 3), a.M - 1) * a.ldt) * 2 + 16 * ((lane & 7) ^ (4 * (q & 1) + (lane >> 4))));
        auto issue = [&](int s, int st) {
#pragma unroll
            for (int i = 0; i < SW / LW; ++i) {
                const uint32_t c = (uint32_t)min((l0 + i) * T + s, a.nk - 1) * 128;
                uint8_t* so = s_dyn + st * STAGE + (l0 + i) * CH;
#pragma unroll
                for (int q = 0; q < 2 * MT; ++q)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (fp8_lds_void*)(so + q * 1024), 16, xoff[q], c, 0, 0);
            }
        };
        constexpr int AHEAD = ONE ? NS - 1 : NS;          // steps issued before step 0
        static_assert(AHEAD == 2 || AHEAD == 3, "the waits below");
#pragma unroll
        for (int i = 0; i < AHEAD; ++i)
            if (i < T) issue(i, i);
        int st = 0;
        for (int s = 0; s < T; ++s) {
            const int later = T - 1 - s;                  // steps of this wave in flight behind step s: at most AHEAD - 1
            if (later >= AHEAD - 1) fp8_wait_vm<PL * (AHEAD - 1)>();   // own part of step s landed
            else if (AHEAD == 3 && later == 1) fp8_wait_vm<PL>();
            else fp8_wait_vm<0>();
            fp8_barrier();
            if constexpr (!ONE) fp8_barrier();            // the stream waves have read step s
            if (s + AHEAD < T) issue(s + AHEAD, ONE ? (st == 0 ? NS - 1 : st - 1) : st);
            st = st == NS - 1 ? 0 : st + 1;
        }
    } else {
        const int c0 = wave * T, n = min(T, a.nk - c0);   // this wave's chunks (n <= 0: none)
        // this wave's scale bytes in LDS (checked on the host: T <= 64), read by this wave only
        constexpr int NSC = (RB + 1) / 2;
        __shared__ uint8_t s_sc[SW][NSC][128];
#pragma unroll
        for (int q = 0; q < NSC; ++q) {
            const uint8_t* sp = a.S + (long long)(min(nb + 2 * q, nbt - 1) >> 1) * a.lds + 2 * min(c0 + lane, a.nk - 1);
            const uint8_t v0 = sp[0], v1 = sp[1];
            s_sc[wave][q][2 * lane] = v0;
            s_sc[wave][q][2 * lane + 1] = v1;
        }
        // weights: row blocks past the last one read the last one again; rows past N (natural layout) read row N - 1; chunks past
        // this wave's last read nothing (an offset past the descriptor)
        const uint8_t* wbase = TILED ? a.W + (long long)nb * a.nk * 1024 : a.W + (long long)nb * 16 * a.ldw;
        const uint32_t w_bytes = TILED ? (uint32_t)(min(RB, nbt - nb) * a.nk * 1024) : (uint32_t)((min(16 * RB, a.N - nb * 16) - 1) * a.ldw + a.K);
        const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(wbase, w_bytes);
        uint32_t woff[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int bb = min(b, nbt - 1 - nb);
            woff[b] = TILED ? (uint32_t)((bb * a.nk + c0) * 1024 + lane * 16) : (uint32_t)(min(bb * 16 + r, a.N - 1 - nb * 16) * a.ldw + c0 * 64 + j * 16);
        }
        constexpr uint32_t wstep = TILED ? 1024 : 64;
        v4i A[PW][RB];
        auto load = [&](int i, int s) {
            const uint32_t o = s < n ? (uint32_t)s * wstep : 0x80000000u;
#pragma unroll
            for (int b = 0; b < RB; ++b) A[i][b] = buffer_load_tile(wr, s < n ? woff[b] + o : o, 0);
        };
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            load(i, i);
            __builtin_amdgcn_sched_barrier(0);
        }
        const int x0 = wave * CH + r * 128 + (((2 * j) ^ (r >> 1)) * 16), x1 = wave * CH + r * 128 + (((2 * j + 1) ^ (r >> 1)) * 16);
        int st = 0;
        auto step = [&](int i, int s) {
            fp8_wait_lds();                               // own reads of step s - 1 done
            fp8_barrier();                                // step s landed
            const uint8_t* so = s_dyn + st * STAGE;
            st = st == NS - 1 ? 0 : st + 1;
            v4i X[MT][2];
            uint32_t sb[NSC];
#pragma unroll
            for (int q = 0; q < NSC; ++q) sb[q] = s_sc[wave][q][2 * s + (j >> 1)];
            if (ONE ? s < n : true) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) {
                    X[mt][0] = *(const v4i*)(so + x0 + mt * 2048);
                    X[mt][1] = *(const v4i*)(so + x1 + mt * 2048);
                }
            }
            if constexpr (!ONE) {
                fp8_wait_lds();
                fp8_barrier();                            // step s read
            }
            if (s < n) {
#pragma unroll
                for (int b = 0; b < RB; ++b) {
                    v8bf16_t lo, hi;
                    decode16(A[i][b], e8m0_to_f32(sb[b >> 1]), lo, hi);
#pragma unroll
                    for (int mt = 0; mt < MT; ++mt) {
                        acc[b][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(v8bf16_t, X[mt][0]), acc[b][mt], 0, 0, 0);
                        acc[b][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(v8bf16_t, X[mt][1]), acc[b][mt], 0, 0, 0);
                    }
                }
            }
        };
        for (int s = 0; s < T; s += PW) {
#pragma unroll
            for (int i = 0; i < PW; ++i) {
                if (s + i >= T) break;
                step(i, s + i);
                load(i, s + i + PW);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    // the stream waves' partial tiles through LDS, added in wave order; tile q by wave q % (SW + LW)
    __syncthreads();
    if (wave < SW) {
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) *(v4f*)(s_dyn + ((wave * RB * MT + b * MT + mt) * 64 + lane) * 16) = acc[b][mt];
    }
    __syncthreads();
    for (int q = wave; q < RB * MT; q += SW + LW) {
        const int b = q / MT, mt = q - b * MT;
        if (nb + b >= nbt) break;
        v4f sum[1] = {*(const v4f*)(s_dyn + (q * 64 + lane) * 16)};
#pragma unroll
        for (int w = 1; w < SW; ++w) sum[0] += *(const v4f*)(s_dyn + ((w * RB * MT + q) * 64 + lane) * 16);
        fp8_store<1>(a, sum, (nb + b) * 16 + 4 * j, r, mt * 16);
    }
}

template <int PW, int NS, int MT, int RB, int TILED>
__global__ void __launch_bounds__(FS_THREADS) fp8_stream_kernel(const Fp8Args a, uint32_t x_bytes) {
    fp8_stream_block<PW, NS, MT, RB, TILED>(a, x_bytes);
}

// ------------------------------------------------------------------------------------------ tiles with shared activations
// 128 weight rows x 16 MT tokens per workgroup over one of S ranges of K. Every operand goes through LDS by the load unit, NS
// stages of CS 64-k chunks, and is read from there by all the waves that need it, so a workgroup moves 128 weight
// rows against 16 MT token rows (the kernels above: 16 or 32 weight rows against all the tokens, which at 64 tokens is five
// activation bytes per weight byte through a CU's load path).
// KH (up to 64 tokens in all, two chunks per stage): wave w takes 32 rows (w & 3) x all tokens of chunk w >> 2 of a stage; the
// two k halves are added through LDS at the end. Otherwise (CS chunks per stage) 32 rows x half w >> 2 of the tokens.
// Bound by the chain of a k-step (barrier, operand reads, decoding, MFMAs), several times its MFMAs' time: about 0.35 us a
// chunk with one workgroup on a CU. One chunk per stage leaves room for two, whose chains overlap and then take 0.57 us each; so
// a K range of its own CU is worth more than sharing one, and sharing pays where ranges are long (hipkern.fp8_rows_plan).
// With S > 1 the fp32 tiles of the ranges go to `part` and a second launch adds them in range order (few weight rows would
// otherwise leave most CUs without a workgroup).
// LDS: weights per chunk and 16-row block 1 KB (tiled: as stored, lane l's operand at 16 l; row-major: 16 rows x 64 B, row
// R's piece c at c ^ (R >> 2)); activations per chunk and 8 rows 1 KB, row R's (of 16) piece c at c ^ (R >> 1).
#define FT_ROWS 128
#define FT_SC 512   // scale bytes of a range (two per chunk)

template <int MT, int NS, int CS, bool KH, int TILED>
__device__ __forceinline__ void fp8_tile_block(const Fp8Args& a, const uint32_t x_bytes, const int tm, const int S) {
    constexpr int TB = KH ? MT : MT / 2;                 // token blocks per wave
    constexpr int XQ = 2 * MT * CS, XW = (XQ + 7) / 8;         // activation loads per stage: all waves, at most per wave
    constexpr int STAGE = (8 * CS + XQ) * 1024;
    static_assert(!KH || CS == 2, "a k half is a chunk of the stage");
    extern __shared__ __align__(16) uint8_t s_dyn[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, j = lane >> 4;
    const int rg = wave & 3, hf = wave >> 2;
    const int L = (int)blockIdx.x, z = (int)blockIdx.y;
    const int nt = (L >> 3) / tm * 8 + (L & 7), t0 = (L >> 3) % tm * (16 * MT);
    if (nt * FT_ROWS >= a.N) return;
    const int nbt = (a.N + 15) / 16, nb0 = nt * (FT_ROWS / 16);
    const int nst = (a.nk + CS - 1) / CS;                      // stages of the whole K
    const int s0 = (int)((long long)nst * z / S), n = (int)((long long)nst * (z + 1) / S) - s0;   // this range: n >= 1
    // the scale bytes of the four 32-row blocks over this range
    __shared__ uint8_t s_sc[4][FT_SC];
    const int nsb = 2 * min(CS * n, a.nk - CS * s0);
    for (int i = (int)threadIdx.x & 127; i < nsb; i += 128) {
        const int q = (int)threadIdx.x >> 7;
        s_sc[q][i] = a.S[(long long)(min(nb0 + 2 * q, nbt - 1) >> 1) * a.lds + 2 * CS * s0 + i];
    }
    // weights: wave w loads row block w, both chunks. Row blocks past the last one read the last one again, rows past N row N - 1
    const int nbw = min(nb0 + wave, nbt - 1);
    const int wr_row = lane >> 2, wr_pc = (lane & 3) ^ (lane >> 4);
    const uint8_t* wbase = TILED ? a.W + (long long)nbw * a.nk * 1024 : a.W + (long long)nbw * 16 * a.ldw;
    const uint32_t w_bytes = TILED ? (uint32_t)(a.nk * 1024) : (uint32_t)(min(15, a.N - 1 - nbw * 16) * a.ldw + a.K);
    const uint32_t woff = TILED ? (uint32_t)(lane * 16) : (uint32_t)(min(wr_row, a.N - 1 - nbw * 16) * a.ldw + wr_pc * 16);
    constexpr uint32_t wstep = TILED ? 1024 : 64;
    const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(wbase, w_bytes), xr = buffer_rsrc(a.x, x_bytes);
    // activations: load q of a stage takes chunk q / (2 MT), rows 8 (q % (2 MT)) ..; wave w takes q = w, w + 8, ..
    const long long goff = a.gc ? (long long)((nb0 * 16) / a.gc) * a.ldx : 0;
    uint32_t xoff[XW];
#pragma unroll
    for (int i = 0; i < XW; ++i) {
        const int q = wave + 8 * i, rb = q < 2 * MT ? q : q - 2 * MT, row = 8 * rb + (lane >> 3);
        xoff[i] = (uint32_t)((goff + (long long)min(t0 + row, a.M - 1) * a.ldt) * 2 + 16 * ((lane & 7) ^ ((row & 15) >> 1)));
    }
    const int xw = (XQ - wave + 7) / 8;                   // activation loads of this wave: XW or XW - 1
    auto issue = [&](int s, int st, auto x_c) {
        uint8_t* so = s_dyn + st * STAGE;
        // an odd last chunk's second half: the first half again, never used
        const uint32_t c = CS * (uint32_t)(s0 + s), c1 = min(c + 1, (uint32_t)a.nk - 1);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (fp8_lds_void*)(so + wave * 1024), 16, woff, c * wstep, 0, 0);
        if constexpr (CS == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (fp8_lds_void*)(so + (8 + wave) * 1024), 16, woff, c1 * wstep, 0, 0);
#pragma unroll
        for (int i = 0; i < decltype(x_c)::value; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, (fp8_lds_void*)(so + (8 * CS + wave + 8 * i) * 1024), 16, xoff[i], (wave + 8 * i < 2 * MT ? c : c1) * 128, 0, 0);
    };
    v4f acc[2][TB];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int t = 0; t < TB; ++t) acc[b][t] = v4f{0.f, 0.f, 0.f, 0.f};
    const int wofs = TILED ? lane * 16 : r * 64 + ((j ^ (r >> 2)) * 16);
    const int x0 = r * 128 + (((2 * j) ^ (r >> 1)) * 16), x1 = r * 128 + (((2 * j + 1) ^ (r >> 1)) * 16);
    auto chunk = [&](const uint8_t* so, int ch, int s) {
        const uint8_t* xs = so + (8 * CS + ch * 2 * MT + (KH ? 0 : hf * MT)) * 1024;
        v4i W[2], X[TB][2];
#pragma unroll
        for (int b = 0; b < 2; ++b) W[b] = *(const v4i*)(so + (ch * 8 + 2 * rg + b) * 1024 + wofs);
#pragma unroll
        for (int t = 0; t < TB; ++t) {
            X[t][0] = *(const v4i*)(xs + t * 2048 + x0);
            X[t][1] = *(const v4i*)(xs + t * 2048 + x1);
        }
        const float sc = e8m0_to_f32((uint32_t)s_sc[rg][2 * (CS * s + ch) + (j >> 1)]);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            v8bf16_t lo, hi;
            decode16(W[b], sc, lo, hi);
#pragma unroll
            for (int t = 0; t < TB; ++t)
                acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(v8bf16_t, X[t][0]), acc[b][t], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < TB; ++t)
                acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(v8bf16_t, X[t][1]), acc[b][t], 0, 0, 0);
        }
    };
    auto kloop = [&](auto x_c) __attribute__((always_inline)) {
        constexpr int PS = CS + decltype(x_c)::value;
        static_assert(PS * (NS - 2) < 64, "the stages in flight are counted in vmcnt");
        // stage s: W later stages of this wave in flight once its own loads of stage s have landed; the barrier says so for
        // every wave, and that stage s - 1 is read, whose place takes stage s + NS - 1
        auto step = [&](int s, int st, auto iss_c, auto w_c) __attribute__((always_inline)) {
            fp8_wait_vm<PS * decltype(w_c)::value>();
            __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));   // lgkmcnt(0): own LDS reads done
            __builtin_amdgcn_s_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
            if constexpr (decltype(iss_c)::value != 0) issue(s + NS - 1, st == 0 ? NS - 1 : st - 1, x_c);
            const uint8_t* so = s_dyn + st * STAGE;
            if constexpr (KH) {
                if (2 * (s0 + s) + hf < a.nk) chunk(so, hf, s);      // an odd last chunk has no second half
            } else {
                chunk(so, 0, s);
                if (CS == 2 && 2 * (s0 + s) + 1 < a.nk) chunk(so, 1, s);
            }
        };
#pragma unroll
        for (int i = 0; i < NS - 1; ++i)
            if (i < n) issue(i, i, x_c);
        int st = 0, s = 0;
        for (; s < n - (NS - 1); ++s) {
            step(s, st, Fp8Int<1>{}, Fp8Int<NS - 2>{});
            st = st == NS - 1 ? 0 : st + 1;
        }
        for (; s < n; ++s) {   // nothing left to issue: n - 1 - s later stages in flight
            if (NS > 3 && n - 1 - s >= 2) step(s, st, Fp8Int<0>{}, Fp8Int<2>{});
            else if (n - 1 - s >= 1) step(s, st, Fp8Int<0>{}, Fp8Int<1>{});
            else step(s, st, Fp8Int<0>{}, Fp8Int<0>{});
            st = st == NS - 1 ? 0 : st + 1;
        }
    };
    static_assert(NS == 3 || NS == 4, "the drain counts up to two later stages");
    if (xw == XW) kloop(Fp8Int<XW>{});
    else kloop(Fp8Int<XW - 1>{});
    if constexpr (KH) {
        // the two k halves: each wave of a pair finishes one row block (half 0 + half 1)
        __syncthreads();
        v4f* red = (v4f*)s_dyn + (size_t)wave * TB * 64 + lane;
#pragma unroll
        for (int t = 0; t < TB; ++t) red[t * 64] = hf ? acc[0][t] : acc[1][t];
        __syncthreads();
        const v4f* other = (const v4f*)s_dyn + (size_t)(wave ^ 4) * TB * 64 + lane;
        if (nb0 + 2 * rg + hf >= nbt) return;
        v4f sum[TB];
#pragma unroll
        for (int t = 0; t < TB; ++t) sum[t] = hf ? other[t * 64] + acc[1][t] : acc[0][t] + other[t * 64];
        fp8_store<TB>(a, sum, (nb0 + 2 * rg + hf) * 16 + 4 * j, r, t0);
    } else {
#pragma unroll
        for (int b = 0; b < 2; ++b)
            if (nb0 + 2 * rg + b < nbt) fp8_store<TB>(a, acc[b], (nb0 + 2 * rg + b) * 16 + 4 * j, r, t0 + hf * (8 * MT));
    }
}

template <int MT, int NS, int CS, bool KH, int TILED>
__global__ void __launch_bounds__(512, CS == 1 ? 4 : 2) fp8_tile_kernel(const Fp8Args a, uint32_t x_bytes, int tm, int S) {
    Fp8Args b = a;
    if (S > 1) b.out = a.out + (long long)blockIdx.y * a.M * a.N;   // range z's partial tile rows
    fp8_tile_block<MT, NS, CS, KH, TILED>(b, x_bytes, tm, S);
}

// out[t][n] = sum over the S ranges' partial sums in range order; one thread per 4 consecutive n
__global__ void __launch_bounds__(256) fp8_reduce_kernel(const float* __restrict__ part, int S, int M, int N, float* __restrict__ out, long long ldo,
                                                         uint16_t* __restrict__ outb, long long ldob) {
    const int nq = N >> 2;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= (long long)M * nq) return;
    const int t = (int)(i / nq), n = (int)(i - (long long)t * nq) * 4;
    const float* p = part + (long long)t * N + n;
    v4f s = *(const v4f*)p;
    for (int z = 1; z < S; ++z) s += *(const v4f*)(p + (long long)z * M * N);
    const float v[4] = {s.x, s.y, s.z, s.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (out) out[(long long)t * ldo + n + q] = v[q];
        if (outb) outb[(long long)t * ldob + n + q] = (uint16_t)f32_to_bf16_bits(v[q]);
    }
}

// ------------------------------------------------------------------------------------------ dequantisation
// Exact fp32 bit pattern of E4M3 code c times 2^(b-127), as quant.dequant_fp8_block computes it in fp32
// (quant.py:90-95): w.float() * 2^(b-127) with IEEE rounding where the product is subnormal. Byte 255 is +inf.
__device__ __forceinline__ uint32_t e4m3_e8m0_f32_bits(uint32_t c, uint32_t b) {
    const uint32_t sign = (c & 0x80u) << 24;
    const uint32_t e = (c >> 3) & 15u, m = c & 7u;
    if (e == 15u && m == 7u) return sign | 0x7FC00000u;            // NaN code
    const uint32_t M = e ? (8u | m) : m;                            // value = M * 2^(E + b - 127)
    const int E = (int)(e ? e : 1u) - 10;
    if (b == 255u) return M ? (sign | 0x7F800000u) : 0xFFC00000u;   // x inf (0 x inf = NaN)
    if (M == 0u) return sign;
    const int h = 31 - __builtin_clz(M);                            // 0..3
    const int biased = h + E + (int)b;                              // biased fp32 exponent of the product
    if (biased >= 255) return sign | 0x7F800000u;
    if (biased >= 1) return sign | ((uint32_t)biased << 23) | ((M << (23 - h)) & 0x7FFFFFu);
    const int sh = E + (int)b + 22;                                 // subnormal: M * 2^sh units of 2^-149
    if (sh >= 0) return sign | (M << sh);
    if (sh < -5) return sign;                                       // below half the smallest subnormal
    const uint32_t q = M >> (-sh), rem = M & ((1u << (-sh)) - 1u), half = 1u << (-sh - 1);
    return sign | (q + ((rem > half || (rem == half && (q & 1u))) ? 1u : 0u));
}

// One thread per 16 weights of a row: 16 B in, 32 B out (natural row-major bf16). A wave takes 16 rows x 64 k, a stored tile
// when tiled: four consecutive lanes hold a row's 64 k, so the wave reads whole lines of the tile and writes whole lines of
// 16 output rows. Bound by the 3 bytes a weight moved; so the codes are decoded by instruction where the product is a normal
// number (then exact, and its upper half the bf16 value): scale bytes 10 (2^-9 x 2^-117 = 2^-126) to 246 (448 x 2^119 <
// 2^128), no NaN code. The rest takes the bit arithmetic. 32768 x 1280: 48.3 -> 25.9 us (2.6 -> 4.9 TB/s, a copy's rate; before: 16-byte
// reads 256 bytes apart and the bit arithmetic for every code).
__device__ __forceinline__ uint32_t dequant_pair_bits(uint32_t c0, uint32_t c1, uint32_t b) {
    return f32_to_bf16_bits(__uint_as_float(e4m3_e8m0_f32_bits(c0, b))) | (f32_to_bf16_bits(__uint_as_float(e4m3_e8m0_f32_bits(c1, b))) << 16);
}

__global__ void __launch_bounds__(256) dequant_fp8_kernel(const uint8_t* __restrict__ W, long long ldw, int tiled, const uint8_t* __restrict__ S,
                                                          long long lds, int N, int K, uint16_t* __restrict__ out, long long ldo) {
    const int lane = threadIdx.x & 63;
    const uint32_t ncb = ((uint32_t)K + 255u) >> 8, rb = blockIdx.x / ncb;   // workgroup: 16 rows x 256 k
    const int n = (int)rb * 16 + (lane >> 2);
    const int c = (int)(blockIdx.x - rb * ncb) * 4 + (int)(threadIdx.x >> 6), k16 = c * 4 + (lane & 3);
    if (n >= N || k16 >= (K >> 4)) return;
    const uint8_t* src;
    if (tiled) src = W + (((long long)rb * (K >> 6) + c) * 64 + (lane & 3) * 16 + (lane >> 2)) * 16;
    else src = W + (long long)n * ldw + (long long)k16 * 16;
    const v4i w = *(const v4i*)src;
    const uint32_t b = S[(long long)(n >> 5) * lds + (k16 >> 1)];
    uint32_t o[8];
    const uint32_t words[4] = {(uint32_t)w.x, (uint32_t)w.y, (uint32_t)w.z, (uint32_t)w.w};
    uint32_t nan = 0;   // bit 7 of a byte: its code is a NaN (0x7F or 0xFF)
#pragma unroll
    for (int i = 0; i < 4; ++i) nan |= (words[i] & 0x7F7F7F7Fu) + 0x01010101u;
    if (b >= 10u && b <= 246u && !(nan & 0x80808080u)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float v[4];
            fq8_values4_hw(words[i], (int)b - 127, v);
            o[2 * i] = (__float_as_uint(v[0]) >> 16) | (__float_as_uint(v[1]) & 0xFFFF0000u);
            o[2 * i + 1] = (__float_as_uint(v[2]) >> 16) | (__float_as_uint(v[3]) & 0xFFFF0000u);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t p = words[i >> 1] >> (16 * (i & 1));
            o[i] = dequant_pair_bits(p & 0xFFu, (p >> 8) & 0xFFu, b);
        }
    }
    v4i* dst = (v4i*)(out + (long long)n * ldo + (long long)k16 * 16);
    dst[0] = v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
    dst[1] = v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
}

// ------------------------------------------------------------------------------------------ entry points
template <int MT, int PF, int RB = 1>
static void fp8_launch_pf(const Fp8Args& a, int tiled, bool wide, hipStream_t st) {
    const dim3 grid(((a.N + 15) / 16 + RB - 1) / RB);
    if (wide) {
        if (tiled) fp8_gemm_kernel<16, PF, MT, 1, RB><<<grid, 1024, 0, st>>>(a);
        else fp8_gemm_kernel<16, PF, MT, 0, RB><<<grid, 1024, 0, st>>>(a);
    } else {
        if (tiled) fp8_gemm_kernel<8, PF, MT, 1, RB><<<grid, 512, 0, st>>>(a);
        else fp8_gemm_kernel<8, PF, MT, 0, RB><<<grid, 512, 0, st>>>(a);
    }
}

template <int MT>
static void fp8_launch(const Fp8Args& a, int tiled, hipStream_t st) {
    const int nb = (a.N + 15) / 16;
    // few row blocks: 16 waves per workgroup so the K split still fills the CUs (not for 4 token tiles, whose
    // registers do not fit 16 waves per CU)
    const bool wide = MT <= 2 && nb < 256 && a.nk >= 64;
    // (Figures of this kernel: fp8_stream_blocks gives most sizes past 8 tokens to the loader waves, which are faster there.)
    // >= 256 row blocks: two row blocks per 8-wave workgroup (every activation load feeds two weight tiles); one token
    // tile: 4 tiles in flight per wave, 3 when a wave has fewer than 4 chunks; two: 3; four: 2. Measured (median of 50
    // graph replays, against one row block per workgroup): 16 / 8 rows 5120 x 8192 20.4 -> 14.4 / 14.9 -> 12.0 us,
    // 4608 x 5120 14.3 -> 10.6 / 10.7 -> 9.0, 32768 x 1280 15.6 -> 12.1 / 11.4 -> 10.5, 5120 x 2304 7.6 -> 6.5 / 6.1 ->
    // 6.0; 32 / 64 rows 5120 x 8192 33.9 -> 21.0 / 63.7 -> 36.4, 32768 x 1280 27.8 -> 20.1 / 52.3 -> 38.4. 16-wave
    // workgroups were level or slower, four row blocks per workgroup slower (5120 x 8192 at 16 rows: 19.8), and fewer
    // row blocks (1280 x 5120: 40 workgroups) slower (8.2 -> 9.9 at 16 rows), so they keep one block each
    if (nb >= 256 && (a.gc == 0 || a.gc % 32 == 0)) {
        if (MT == 1 && a.nk < 32) fp8_launch_pf<1, 3, 2>(a, tiled, false, st);
        else fp8_launch_pf<MT, MT == 1 ? 4 : MT == 2 ? 3 : 2, 2>(a, tiled, false, st);
        return;
    }
    // one row block per workgroup, <= 128 VGPRs: two 8-wave workgroups per CU. One token tile: 6 tiles in flight per
    // wave, 3 when a wave has fewer than 6 chunks (measured at 16 / 8 rows: 32768 x 1280 17.9 -> 15.1 / 14.8 -> 11.0 us;
    // the other reference shapes within 1 %, and 2 / 4 / 8 in flight no better)
    if (MT == 1 && a.nk < 6 * (wide ? 16 : 8)) fp8_launch_pf<MT, 3>(a, tiled, wide, st);
    else fp8_launch_pf<MT, MT == 1 ? 6 : MT == 2 ? 4 : 2>(a, tiled, wide, st);
}

// Operands of the kernels that go through LDS: 16-byte pieces, 32-bit offsets, all the rows of a workgroup in one column group.
static bool fp8_lds_operands_ok(const Fp8Args& a, int tiled, int rows) {
    return !(((uintptr_t)a.x) & 15) && !(a.ldx & 7) && !(((uintptr_t)a.W) & 15) && (tiled || !(a.ldw & 15)) && (a.gc == 0 || a.gc % rows == 0) &&
           fp8_x_bytes(a) < 0x80000000ll && (long long)rows * a.ldw < 0x80000000ll;
}

// Row blocks per workgroup of the loader-wave kernel for this call (8: the 128-row tiles; 0: fp8_gemm_kernel). Both sides in us,
// fp8_gemm_kernel first unless said otherwise; medians of graph replays over weights larger than the last-level cache.
//  * fewer than 256 row blocks (one per workgroup): long rows only. 1280 x 5120 at 48 18.9 -> 9.8, 3328 x 7168 at 16 10.8 -> 9.2;
//    2048 x 512 at 32 4.1 / 4.2, so short rows (K < 1024; up to 16 tokens K < 2048) stay. A few tokens load too little for the
//    loader waves to pay: 3328 x 7168 at 5 7.9 / 8.4, 2992 x 5376 at 5 6.7 / 7.3, 1080 x 3008 at 7 5.65 / 5.94, 4000 x 3520 at 8 5.72 /
//    5.96, against 1600 x 7168 at 8 8.16 / 7.87, 4000 x 5120 at 12 8.07 / 7.82. Token rows a multiple of 8 KB apart (K % 4096 == 0)
//    collide in fp8_gemm_kernel's loads, so up to 192 blocks it loses from 5 on (1280 x 8192 at 5 / 8 7.99 -> 7.80 / 8.82 -> 7.85).
//  * up to 512: two. 5120 x 8192 at 32 21.4 -> 15.1 (one: 21.2, four: 19.9). Up to 16 tokens the gain is small (5120 x 8192 14.6 ->
//    13.1) and ends before 512 blocks (8192 x 2048 6.5 / 6.6).
//  * more: four. 16384 x 5120 at 48 43.2 -> 22.1 (two: 27.6), 16384 x 2048 21.9 -> 13.5. Up to 16 tokens long rows only
//    (16384 x 5120 22.8 -> 17.7, 16384 x 2048 10.3 / 10.3). With K % 4096 == 0 the weight streams of many blocks collide, so few
//    tokens take them up to 640 blocks (9600 x 4096 at 16 15.9 -> 14.4; 16384 x 4096 at 16 16.7 / 19.2, 16384 x 8192 29.8 / 36.9, 64000 x
//    4096 54.2 / 62.1), and past 896 blocks some more tokens are needed (14000 x 8192 at 17 31.7 ->
//    29.8, 16384 x 8192 33.0 / 38.0, at 24 36.9 / 37.4).
//    Beyond 1024 blocks they are more workgroups than CUs, one to a CU, and the last of them leave most of the chip idle; so up to
//    16 tokens only from 1536 blocks and 11 tokens on (24592 x 5120 at 9 / 16 27.9 / 31.0 and 34.1 / 32.4, 28800 x 5120 at 16 38.2 ->
//    32.4). Below 1536 blocks not with few tokens and short rows either: 20800 x 768 at 32 12.8 / 13.6, 20800 x 1280 at 24 / 32 14.8 /
//    15.3 and 16.5 / 16.3, 24000 x 2048 at 20 / 28 18.1 / 19.3 and 20.0 / 20.0, 24000 x 4096 at 18 28.0 / 30.3, 16640 x 2560 at 20
//    21.3 -> 19.9; 24000 x 1472 at 40 25.3 -> 17.7.
//  * 192 and more 128-row tiles with short rows: the tiles, whose activations are read once per 128 weight rows. 32768 x 1280 at
//    48 / 64 33.3 -> 15.2 / 38.6 -> 17.2 (four blocks: 18.5 / 22.2), 24576 x 1280 at 48 25.4 -> 15.1 (17.4).
static int fp8_stream_blocks(const Fp8Args& a, int nb) {
    if (a.M <= 4 || a.nk > 64 * FS_SW) return 0;
    const bool few = a.M <= 16, collide = a.nk % 64 == 0;
    if (nb < 256) {
        const int least = nb <= 192 ? (collide ? 5 : 8) : a.nk >= 64 ? 8 : 12;
        return few ? (a.nk >= 32 && a.M >= least ? 1 : 0) : a.nk >= 16 ? 1 : 0;
    }
    if (few && a.M <= 8) return 0;
    if (nb <= 512) return !few || (nb <= 448 && a.nk >= 24) ? 2 : 0;
    if (few) return a.nk >= 64 && (collide ? nb <= 640 : nb <= 1024 || (nb >= 1536 && a.M >= 11)) ? 4 : 0;
    if (nb >= 192 * 8) return a.nk <= 40 ? 8 : 4;
    const int most = nb <= 1024 ? (collide && nb > 896 ? 20 : 16) : a.nk >= 40 ? (collide ? 24 : 16) : a.nk >= 32 ? 24 : a.nk >= 16 ? 28 : 32;
    return a.M > most ? 4 : 0;   // up to `most` tokens fp8_gemm_kernel
}

template <int NS, int MT, int RB, int TILED>
static int fp8_stream_launch_t(const Fp8Args& a, hipStream_t st) {
    const size_t lds = (size_t)NS * FS_SW * 2 * MT * 1024;
    const hipError_t err = hipFuncSetAttribute((const void*)fp8_stream_kernel<4, NS, MT, RB, TILED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return (int)err;
    const dim3 grid(((a.N + 15) / 16 + RB - 1) / RB);
    fp8_stream_kernel<4, NS, MT, RB, TILED><<<grid, FS_THREADS, lds, st>>>(a, (uint32_t)fp8_x_bytes(a));
    return (int)hipGetLastError();
}

template <int RB, int TILED>
static int fp8_stream_launch_m(const Fp8Args& a, hipStream_t st) {
    switch ((a.M + 15) / 16) {
        case 1: return fp8_stream_launch_t<4, 1, RB, TILED>(a, st);
        case 2: return fp8_stream_launch_t<4, 2, RB, TILED>(a, st);
        case 3: return fp8_stream_launch_t<3, 3, RB, TILED>(a, st);
        default: return fp8_stream_launch_t<2, 4, RB, TILED>(a, st);
    }
}

static int fp8_stream_launch(const Fp8Args& a, int tiled, int rb, hipStream_t st) {
    if (rb == 1) return tiled ? fp8_stream_launch_m<1, 1>(a, st) : fp8_stream_launch_m<1, 0>(a, st);
    if (rb == 2) return tiled ? fp8_stream_launch_m<2, 1>(a, st) : fp8_stream_launch_m<2, 0>(a, st);
    return tiled ? fp8_stream_launch_m<4, 1>(a, st) : fp8_stream_launch_m<4, 0>(a, st);
}

// tiles of 128 rows x 16 MT tokens over S ranges of K; the caller has checked that a range's scale bytes fit FT_SC
template <int MT, int NS, int CS, bool KH, int TILED>
static int fp8_tile_launch_t(const Fp8Args& a, int S, hipStream_t st) {
    const size_t lds = (size_t)NS * (8 + 2 * MT) * CS * 1024;
    const hipError_t err = hipFuncSetAttribute((const void*)fp8_tile_kernel<MT, NS, CS, KH, TILED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (err != hipSuccess) return (int)err;
    const int tm = (a.M + 16 * MT - 1) / (16 * MT);
    const long long grid = (((long long)a.N + FT_ROWS - 1) / FT_ROWS + 7) / 8 * 8 * tm;
    if (grid > 0x7FFFFFFFll) return DSV41_EINVAL;
    fp8_tile_kernel<MT, NS, CS, KH, TILED><<<dim3((unsigned)grid, (unsigned)S), 512, lds, st>>>(a, (uint32_t)fp8_x_bytes(a), tm, S);
    return (int)hipGetLastError();
}

static int fp8_tile_launch_kh(const Fp8Args& a, int tiled, hipStream_t st) {
    switch ((a.M + 15) / 16) {
        case 1:
        case 2: return tiled ? fp8_tile_launch_t<2, 4, 2, true, 1>(a, 1, st) : fp8_tile_launch_t<2, 4, 2, true, 0>(a, 1, st);
        case 3: return tiled ? fp8_tile_launch_t<3, 4, 2, true, 1>(a, 1, st) : fp8_tile_launch_t<3, 4, 2, true, 0>(a, 1, st);
        default: return tiled ? fp8_tile_launch_t<4, 4, 2, true, 1>(a, 1, st) : fp8_tile_launch_t<4, 4, 2, true, 0>(a, 1, st);
    }
}

extern "C" int dsv41_fp8_gemm(const uint8_t* W, long long ldw, int tiled, const uint8_t* S, long long lds, int N, int K,
                              const uint16_t* x, long long ldx, int M, int group_cols, float* out, long long ldo,
                              uint16_t* outb, long long ldob, void* stream) {
    if (!W || !S || !x || (!out && !outb) || N <= 0 || K <= 0 || (K & 63) || M < 1 || M > 64) return DSV41_EINVAL;
    if (tiled ? ((N & 15) || ldw != K) : ldw < K) return DSV41_EINVAL;
    if (lds < K / 32 || ldx < K || (out && ldo < N) || (outb && ldob < N)) return DSV41_EINVAL;
    if (group_cols < 0 || (group_cols && ((group_cols & 15) || N % group_cols))) return DSV41_EINVAL;
    const long long G = group_cols ? N / group_cols : 1;
    Fp8Args a{W, ldw, S, lds, N, K, K / 64, x, ldx, ldx * G, M, group_cols, out, ldo, outb, ldob};
    hipStream_t st = (hipStream_t)stream;
    // up to 4 tokens whose activations fit 64 KiB of LDS per workgroup: the LDS-staged kernel. Launch shapes, measured
    // at one token over resident copies larger than the 256 MB last-level cache (median of 50 graph replays):
    //  * >= 256 row blocks: 4 waves per workgroup, 4 weight tiles in flight per wave (5120 x 8192: 9.5 us; 12 in flight
    //    10.9, 24 12.1, 8 waves 10.7-11.0, 16 waves 12.2-13.1); rows of <= 24 chunks (K <= 1536) 2 waves, each with
    //    more of the row (32768 x 1280: 9.2 us against 10.1 with 4 waves);
    //  * fewer row blocks: 4 waves with 10 tiles in flight (1280 x 5120: 5.0 us against 5.9 with 16 waves).
    // Deeper prefetch was slower for every shape with more row blocks than CUs.
    const int nb = (N + 15) / 16;
    const int wpg = nb >= 256 && a.nk <= 24 ? 2 : 4;
    const int cpw = (a.nk + wpg - 1) / wpg;
    const long long lds_bytes = (long long)wpg * fp8_lds_region(M, cpw);
    // every wave owns >= 1 chunk; activation pieces and scale bytes fit the per-lane staging registers
    if (M <= 4 && a.nk >= wpg && M * cpw <= 64 && 2 * cpw <= 128 && lds_bytes <= 65536) {
        const dim3 grid(nb);
        if (wpg == 2) {
            if (tiled) fp8_gemv_lds_kernel<2, 4, 1><<<grid, 128, lds_bytes, st>>>(a, cpw);
            else fp8_gemv_lds_kernel<2, 4, 0><<<grid, 128, lds_bytes, st>>>(a, cpw);
        } else if (nb >= 256) {
            if (tiled) fp8_gemv_lds_kernel<4, 4, 1><<<grid, 256, lds_bytes, st>>>(a, cpw);
            else fp8_gemv_lds_kernel<4, 4, 0><<<grid, 256, lds_bytes, st>>>(a, cpw);
        } else {
            if (tiled) fp8_gemv_lds_kernel<4, 10, 1><<<grid, 256, lds_bytes, st>>>(a, cpw);
            else fp8_gemv_lds_kernel<4, 10, 0><<<grid, 256, lds_bytes, st>>>(a, cpw);
        }
        return (int)hipGetLastError();
    }
    // more tokens x chunks than 4 waves can stage: 8 waves (16 for few row blocks with long rows), 12 tiles in flight
    const int wpg2 = nb < 256 && a.nk >= 64 ? 16 : 8, cpw2 = (a.nk + wpg2 - 1) / wpg2;
    const long long lds2 = (long long)wpg2 * fp8_lds_region(M, cpw2);
    if (M <= 4 && a.nk >= wpg2 && M * cpw2 <= 64 && 2 * cpw2 <= 128 && lds2 <= 65536) {
        const dim3 grid(nb);
        if (wpg2 == 16) {
            if (tiled) fp8_gemv_lds_kernel<16, 12, 1><<<grid, 1024, lds2, st>>>(a, cpw2);
            else fp8_gemv_lds_kernel<16, 12, 0><<<grid, 1024, lds2, st>>>(a, cpw2);
        } else {
            if (tiled) fp8_gemv_lds_kernel<8, 12, 1><<<grid, 512, lds2, st>>>(a, cpw2);
            else fp8_gemv_lds_kernel<8, 12, 0><<<grid, 512, lds2, st>>>(a, cpw2);
        }
        return (int)hipGetLastError();
    }
    const int rb = fp8_stream_blocks(a, nb);
    if (rb && fp8_lds_operands_ok(a, tiled, 16 * rb)) return rb == 8 ? fp8_tile_launch_kh(a, tiled, st) : fp8_stream_launch(a, tiled, rb, st);
    if (M <= 16) fp8_launch<1>(a, tiled, st);
    else if (M <= 32) fp8_launch<2>(a, tiled, st);
    else fp8_launch<4>(a, tiled, st);
    return (int)hipGetLastError();
}

// More than 64 rows: 128 weight rows x `tile` (64 or 128) activation rows per workgroup, K in `splits` ranges whose fp32 sums go
// through `part`.
extern "C" int dsv41_fp8_gemm_rows(const uint8_t* W, long long ldw, int tiled, const uint8_t* S, long long lds, int N, int K,
                                   const uint16_t* x, long long ldx, int M, float* out, long long ldo, uint16_t* outb, long long ldob,
                                   int tile, int splits, float* part, long long part_floats, void* stream) {
    if (!W || !S || !x || (!out && !outb) || N <= 0 || K <= 0 || (K & 63) || M < 1) return DSV41_EINVAL;
    if (tiled ? ((N & 15) || ldw != K) : ldw < K) return DSV41_EINVAL;
    if (lds < K / 32 || ldx < K || (out && ldo < N) || (outb && ldob < N)) return DSV41_EINVAL;
    if ((tile != 64 && tile != 128) || splits < 1 || splits > K / 64) return DSV41_EINVAL;
    if (splits > 1 && (!part || (N & 3) || (((uintptr_t)part) & 15) || part_floats < (long long)splits * M * N)) return DSV41_EINVAL;
    const Fp8Args a{W, ldw, S, lds, N, K, K / 64, x, ldx, ldx, M, 0, out, ldo, outb, ldob};
    if (!fp8_lds_operands_ok(a, tiled, FT_ROWS) || 2 * ((a.nk + splits - 1) / splits) > FT_SC) return DSV41_EINVAL;
    hipStream_t st = (hipStream_t)stream;
    Fp8Args b = a;
    if (splits > 1) {
        b.out = part;
        b.ldo = N;
        b.outb = nullptr;
    }
    const int rc = tile == 64 ? (tiled ? fp8_tile_launch_t<4, 4, 1, false, 1>(b, splits, st) : fp8_tile_launch_t<4, 4, 1, false, 0>(b, splits, st))
                              : (tiled ? fp8_tile_launch_t<8, 3, 1, false, 1>(b, splits, st) : fp8_tile_launch_t<8, 3, 1, false, 0>(b, splits, st));
    if (rc || splits == 1) return rc;
    const long long q = (long long)M * (N / 4);
    fp8_reduce_kernel<<<(unsigned)((q + 255) / 256), 256, 0, st>>>(part, splits, M, N, out, ldo, outb, ldob);
    return (int)hipGetLastError();
}

extern "C" int dsv41_dequant_fp8(const uint8_t* W, long long ldw, int tiled, const uint8_t* S, long long lds, int N, int K,
                                 uint16_t* out, long long ldo, void* stream) {
    if (!W || !S || !out || N <= 0 || K <= 0 || (K & 15) || ldo < K || lds < (K + 31) / 32) return DSV41_EINVAL;
    if (tiled ? ((N & 15) || (K & 63) || ldw != K) : ldw < K) return DSV41_EINVAL;
    // a launch takes fewer than 2^32 threads: rows beyond that go to launches of their own
    const long long ncb = ((long long)K + 255) / 256, step = max((1ll << 23) / ncb * 16 & ~31ll, 32ll);
    for (long long n0 = 0; n0 < N; n0 += step) {
        const long long rows = min(step, N - n0);
        dequant_fp8_kernel<<<(unsigned)((rows + 15) / 16 * ncb), 256, 0, (hipStream_t)stream>>>(W + n0 * (tiled ? K : ldw), ldw, tiled, S + n0 / 32 * lds, lds,
                                                                                          (int)rows, K, out + n0 * ldo, ldo);
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return (int)err;
    }
    return 0;
}
