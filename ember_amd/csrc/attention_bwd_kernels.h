// attention_bwd_kernels.h -- what the attention backward's kernels for longer
// sequences share (attention_bwd_tiles.hip, attention_bwd_w16.hip,
// attention_bwd_s128.hip): arguments, row statistics, ordered dQ.
//
// No reference counterpart (pawel002/ember has no attention); semantics are
// those of oracle/ember_oracle.c (oracle_attention_bwd): P is recomputed from
// the forward's LSE, never stored.
//
// Two launches on the null stream:
//  1. attn_bwd_pre (HBM-bound, one pass over O and dO): per query row
//     lse2 = lse * log2(e) and delta = <dO, O> into a row-statistics scratch
//     whose rows are padded per (b, h) to a multiple of 32 (padding rows get
//     lse2 = +inf, delta = 0, so every P they enter is exactly 0); and
//     dQ := 0 (dQ is accumulated with atomics).
//  2. a K/V-stationary kernel: a workgroup keeps its keys' K and V and their
//     dK and dV accumulators, and walks the query blocks (causal: only those
//     at or below its keys):
//        S  = Q K^T, dP = dO V^T
//        P  = exp2(S*c - lse2[m]), dS = P * (dP - delta[m])
//        dV += P^T dO,  dK += dS^T Q
//     and dS . K over the workgroup's keys is added to the global dQ with
//     hardware fp32 atomics (dq must be device memory).  Deterministic mode
//     (ember_set_deterministic) adds the same values with the same atomics,
//     but in a fixed order ("Ordered dQ" below).
#pragma once

#include <math.h>

#include <type_traits>

#include "common.h"
#include "lds_dma.h"
#include "mfma.h"

namespace ember {

int check_attention_args(const void *const *ptrs, int nptrs, int64_t B, int64_t H, int64_t S,
                         int64_t D, float scale, const int64_t *strides, int nstrides,
                         const char *who);

struct BwdArgs {
    const float *q, *k, *v, *o, *lse, *dout;
    float *dq, *dk, *dv;
    float *lse2, *delta;  // row statistics, (B*H, S_pad) each
    // Deterministic mode (ember_set_deterministic), null otherwise:
    // order[bh * (S_pad / 16) + m / 16] counts the contributions added so
    // far to the dQ rows of head bh from row m (16-row granularity);
    // attn_bwd_pre zeroes them.  order_timeouts counts waits that gave up (a
    // device counter that is never reset).
    int *order;
    int *order_timeouts;
    int order_group;  // key blocks per group of the order (see "Ordered dQ")
    int H, S, S_pad, nkb;
    float c;      // scale * log2(e)
    float scale;
    int64_t in_sb, in_sh, in_ss, out_sb, out_sh, out_ss;
};

// attention_bwd_tiles.hip: attn_bwd_pre, then the key-block workgroup kernel,
// whose dQ is added with atomics in arrival order or (args.order set) in
// key-block order.
int launch_bwd_tiles(const BwdArgs &args, int D, bool causal, int64_t rows_pad, int nblocks);

// attention_bwd_s128.hip: 64 < S <= 128 at D = 64 or 128, one workgroup
// per head (no row statistics and no atomics: args.lse2, delta, order
// unused).
int launch_bwd_s128(const BwdArgs &args, int D, bool causal, int nbh);
// attention_bwd_w16.hip: D = 64 at S > 128 (attn_bwd_pre, then attn_bwd_w16,
// ordered when args.order is set).
int launch_bwd_w16(const BwdArgs &args, int64_t rows_pad, bool causal, int nbh);

namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kBkw = 32;            // keys per wave
constexpr int kBk = kBkw * kWaves;  // keys per workgroup
constexpr int kBq = 32;             // queries per step
constexpr float kLog2e = 1.4426950408889634f;

// Row statistics and dQ := 0 (and, in deterministic mode, the tile
// counters := 0).  D/4 threads per (padded) row.
template <int D>
__global__ __launch_bounds__(256) void attn_bwd_pre(BwdArgs a, int64_t rows_pad)
{
    constexpr int TPR = D / 4;
    constexpr int RPB = 256 / TPR;
    const int sub = threadIdx.x % TPR;
    const int64_t row = (int64_t)blockIdx.x * RPB + threadIdx.x / TPR;
    if (row >= rows_pad) return;  // whole TPR-lane groups retire together
    if (a.order && sub == 0 && (row & 15) == 0) a.order[row >> 4] = 0;
    const int64_t bh = row / a.S_pad;
    const int m = (int)(row - bh * a.S_pad);
    if (m >= a.S) {
        if (sub == 0) {
            a.lse2[row] = INFINITY;
            a.delta[row] = 0.0f;
        }
        return;
    }
    const int b = (int)(bh / a.H);
    const int hh = (int)(bh - (int64_t)b * a.H);
    const int64_t ooff = (int64_t)b * a.out_sb + (int64_t)hh * a.out_sh + (int64_t)m * a.out_ss + 4 * sub;
    const f32x4 ov = *(const f32x4 *)(a.o + ooff);
    const f32x4 gv = *(const f32x4 *)(a.dout + ooff);
    float s = ov[0] * gv[0] + ov[1] * gv[1] + ov[2] * gv[2] + ov[3] * gv[3];
#pragma unroll
    for (int off = TPR / 2; off > 0; off >>= 1) s += __shfl_xor(s, off);
    if (sub == 0) {
        a.delta[row] = s;
        a.lse2[row] = a.lse[bh * a.S + m] * kLog2e;
    }
    const int64_t qoff = (int64_t)b * a.in_sb + (int64_t)hh * a.in_sh + (int64_t)m * a.in_ss + 4 * sub;
    *(f32x4 *)(a.dq + qoff) = f32x4{0.f, 0.f, 0.f, 0.f};
}

// ---- Ordered dQ (deterministic mode) ----
// fp32 addition is not associative, so dQ added with atomics in arrival
// order differs in its last bits from run to run.  In deterministic mode each
// dQ tile receives its key blocks' contributions in a fixed order: the wave
// that adds key block kb's share of a tile first waits until the tile's
// counter shows that every key block before kb in that order has added
// its share, then adds its own with the same atomics, waits for their
// acknowledgement and increments the counter.
// The order follows the hardware's schedule.  Work items keep the default
// mode's numbering (key block major, heaviest causal walks first, each
// head's workgroups on one XCD), and the workgroups of each XCD start in
// index order.  Key blocks come in groups of R (args.order_group): the
// groups in ascending order, and within a group descending, because the R
// key blocks of a group run at the same time and, causally, key block kb + 1
// starts its walk at the tile key block kb reaches four steps later, so
// that it is ahead at every tile they share.  A workgroup waits only for
// lower groups, which started earlier, and for higher key blocks of its own
// group; the host picks R so that the groups below the top key block of a
// group fit in the device at once, R <= 1 + (slots - 1) / (B * H) (slots:
// workgroups resident at once, an eighth kept spare), so the top key blocks,
// which wait on lower groups only, always start, and no wait can deadlock.
// The counter is polled a step ahead of its use.  A workgroup first reads
// the counter of the last tile it adds to: if every key block before it has
// added its share there, it has added all its tiles (each walks its tiles
// upward, and a key block that sees one of this workgroup's tiles sees its
// last one), and the workgroup walks without polls or waits
// (kDqOrderedFree), only counting its own adds.
// The adds are released by waiting for their acknowledgement (vmcnt), not by
// an agent-scope release fence: these atomics are performed where every XCD's
// atomics on the address meet (adds into one tile from several XCDs are
// exact), and an acknowledged atomic has been performed there; the fence
// would add an L2 write-back per wave and step (3.8x the time at B4 H32
// S4096 D128), and with it and without it dQ came out the same bits in
// every case measured (causal and not, D = 32, 64, 128).
// Each wait is still bounded, should those start-order assumptions ever not
// hold: after ~2 s (s_memrealtime runs at 100 MHz) it gives up, counts
// itself in order_timeouts, and from then on no wait blocks; the sum stays
// correct, only its order is lost, which ember_deterministic_timeouts()
// reports.
constexpr int kDqAtomic = 0, kDqOrdered = 1, kDqOrderedFree = 2;
constexpr uint64_t kOrderTimeoutTicks = 200000000ull;

// A tile counter (relaxed, device scope: the load bypasses this XCD's L2,
// so it sees increments made on other XCDs).
__device__ __forceinline__ int order_poll(const int *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until *turn >= expect (polled: an earlier read of *turn).
__device__ __forceinline__ void order_wait(const int *turn, int expect, int polled, int *timeouts)
{
    if (__builtin_amdgcn_readfirstlane(polled) < expect) {
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        for (;;) {
            __builtin_amdgcn_s_sleep(2);
            if (__builtin_amdgcn_readfirstlane(order_poll(turn)) >= expect) break;
            if (__builtin_amdgcn_readfirstlane(order_poll(timeouts)) != 0) break;
            if (__builtin_amdgcn_s_memrealtime() - t0 > kOrderTimeoutTicks) {
                if ((threadIdx.x & 63) == 0)
                    __hip_atomic_fetch_add(timeouts, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                break;
            }
        }
    }
    asm volatile("" ::: "memory");  // the adds that follow stay after the wait
}

// This wave's adds into the tile have been acknowledged (vmcnt 0: every
// vector memory operation of the wave has completed); count them.
__device__ __forceinline__ void order_done(int *turn)
{
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
    asm volatile("" ::: "memory");
    if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(turn, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int D>
struct BwdLayout {
    static constexpr int DB = D / 32;
    static constexpr int NSPLIT = 4 / DB;  // waves sharing a 32-wide d block of dQ
    static constexpr int NK = kBk / NSPLIT;  // keys each wave contracts for dQ
};

// A workgroup's part in dQ.
struct BwdBlock {
    float *dqp;  // dq at (b, h)
    int *turns;  // deterministic mode: tile counters of (b, h)
    int S, nq, w, kb, in_ss;
};

// Deterministic mode: the contributions that come before key block kb's at
// a tile whose last contributing key block is `last` (ordered dQ above):
// every key block of the lower groups, and those after kb in its own group.
__device__ __forceinline__ int order_before(int kb, int last, int R)
{
    const int g0 = kb - kb % R;
    return g0 + min(g0 + R - 1, last) - kb;
}

// How many increments this wave must see on the counter of the tile of rows
// m0.. before adding: four per key block before kb in the order (one per
// wave), and, where waves share dQ columns (D < 128), those of the lower
// waves of its own key block.
template <int D, bool CAUSAL>
__device__ __forceinline__ int dq_turn_expect(const BwdArgs &a, const BwdBlock &k, int m0)
{
    constexpr int DB = BwdLayout<D>::DB;
    const int last = CAUSAL ? min(a.nkb - 1, (m0 / kBq) >> 2) : a.nkb - 1;  // key blocks of 128 = 4 tiles
    return 4 * order_before(k.kb, last, a.order_group) + (k.w / DB) * DB;
}

// Deterministic mode: whether a wave counts its adds into a tile at once
// (waves that share dQ columns wait for each other within the step) or
// after the step's wait for its copies, which then costs no extra wait.
template <int D>
constexpr bool kDoneAtOnce = BwdLayout<D>::DB < 4;

// The finished dQ block (rows m0..m0+31) times scale, added into dq with atomics;
// deterministic mode (kDqOrdered) first waits for its turn (polled: an
// earlier read of the tile counter) and counts its adds (kDoneAtOnce) or
// leaves that to the caller.
template <int D, bool CAUSAL, int DQ>
__device__ __forceinline__ void dq_store(const BwdArgs &a, const BwdBlock &k, int m0, const f32x16 &qacc,
                                         float scale, int polled)
{
    constexpr int DB = BwdLayout<D>::DB;
    const int lane = threadIdx.x & 63;
    const int h32 = lane >> 5;
    const int l32 = lane & 31;
    const int dblk = k.w % DB;
    if constexpr (DQ == kDqOrdered)
        order_wait(k.turns + (m0 >> 4), dq_turn_expect<D, CAUSAL>(a, k, m0), polled, a.order_timeouts);
    else if constexpr (DQ == kDqOrderedFree)
        asm volatile("" ::: "memory");
    // Row i of the block: wave-uniform row base + unsigned lane offset.
    float *dqb = k.dqp + (int64_t)m0 * k.in_ss + 32 * dblk;
    const unsigned qoff = (unsigned)(4 * h32 * k.in_ss + l32);
    if (m0 + kBq <= k.S) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float *rowp = dqb + (int64_t)(((i >> 2) * 8 + (i & 3)) * k.in_ss);
            unsafeAtomicAdd(rowp + qoff, qacc[i] * scale);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float *rowp = dqb + (int64_t)(((i >> 2) * 8 + (i & 3)) * k.in_ss);
            if (m0 + acc_row(i, h32) < k.S) unsafeAtomicAdd(rowp + qoff, qacc[i] * scale);
        }
    }
    if constexpr (DQ != kDqAtomic && kDoneAtOnce<D>) order_done(k.turns + (m0 >> 4));
}

}  // namespace
}  // namespace ember

