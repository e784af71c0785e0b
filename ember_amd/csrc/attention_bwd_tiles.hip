// attention_bwd_tiles.hip -- the key-block attention backward on the bf16
// matrix cores at fp32 precision (split_bf16.h): S > 128 at D = 128, S > 64
// at D = 32, and longer walks in larger launches at D = 64.
//
// Launched after attn_bwd_pre (attention_bwd_kernels.h: row statistics, dQ :=
// 0).  One workgroup = 4 waves = 128 keys of one (b, h); it walks the query
// rows in blocks of 32 (causal: those at or below its keys).  LDS holds three
// bf16 planes (hi, mid, lo) of the workgroup's K rows for the whole walk and
// of the block's Q and dO rows; a wave keeps V of its 32 keys in registers and
// accumulates their dK and dV there.  Rows serve both kinds of operand: with
// the contraction along d they are read as they lie, with the contraction
// along the rows by the transposing LDS read (ds_read_b64_tr_b16), which hands
// each lane one column of four rows.  Per block and wave:
//   S   = Q K^T             beside it: this block's dO split and stored
//   dP  = dO V^T            beside it: P = exp2(S c - lse2), split
//   dV += P^T dO            beside it: dS = P (dP - delta), split (P and dS
//                           stand in the accumulators as the operand needs)
//   dK += dS^T Q            beside it: dS to LDS
//   dQ  = dS K over the workgroup's keys, added to the global dQ with
//                           atomics; beside it: next block's Q split and stored
// At D = 128 dS takes the place of the block's dO (LDS: 148 KB, one workgroup
// per CU).
//
// Signs (split_bf16.h).  K and V rows carry sign_of(key), so that S and dP
// have it too; P and dS carry it times the key block's parity, so that dK and
// dV rows get theirs, and dQ, where the keys' signs cancel, one that
// alternates from key block to key block.  All come off where a value is
// scaled anyway, and 2^32 of scale with them.
//
// What the scaled split cannot carry (Q or K from 2^44, V or dO from 2^111
// on, dS so large that dQ might pass 2^96, infinities, NaN) ends a workgroup's walk before that step
// adds its dQ; the waves then form their dK and dV, and the dQ of the rest of
// the walk, with the fp32 instruction straight from global memory, at the end
// of the kernel, where that code takes no registers from the walk.  (Done
// within the step, S and dP alone, 32 vector operations per step to look for
// it instead of 16: 4 heads of 300 at D = 128 72.8 us, now 70.4.)
//
// What bounds it: at D = 128 one workgroup per CU is one wave per SIMD, so a
// wave's own waits (four barriers and the LDS reads of each block's first
// operands) leave the matrix cores idle: B4 H32 S4096 D128 causal busy 52 % of
// cycles at 1.86 GHz (power limit), with 4.8 vector instructions to a matrix
// one, and bank conflicts of the transposing reads in 12 %.  Hence the vector work laid beside the
// products, and operands read a chunk ahead.  Against the kernel on the fp32
// instruction that it replaced: B4 H32 S4096 D128 causal 10740 -> 8090 us
// (128 -> 170 TFLOP/s; in deterministic order 4 % longer), 30 heads of 777 at
// D = 128 265 -> 172, 32 heads of 1024 causal 336 -> 212, 4 heads of 300 109 ->
// 70; D = 32, 64 heads of 1000 causal 166 -> 154.  Error against
// float64 (relative 2-norm, the first, dQ, dK, dV): 6.0e-7, 1.6e-6, 1.6e-6 ->
// 5.2e-7, 1.2e-6, 1.2e-6.
#include "attention_bwd_kernels.h"
#include "split_bf16.h"

namespace ember {
namespace {

template <int D>
struct BwdTiles {
    static constexpr int U = D / 8;            // 16-byte units per row and plane
    static constexpr int KPL = kBk * U;        // units per K plane
    static constexpr int QPL = kBq * U;        // units per Q or dO plane
    static constexpr int SPL = kBk * kBq / 8;  // units per dS plane, rows = keys
    static constexpr bool kShared = D == 128;  // dS in dO's place
    static constexpr int G = (QPL + kThreads - 1) / kThreads;  // Q (or dO) groups of 8 per thread
    static constexpr int KS = D / 16, DB = D / 32;
    static constexpr int NK = BwdLayout<D>::NK;  // keys a wave contracts for dQ
    static_assert(!kShared || 3 * SPL == 3 * QPL, "dS fills dO's place");

    // Unit u of row r of a plane with V units per row: 16 neighbouring rows
    // of one u fall on different banks, and so do 4 neighbouring rows of two
    // units 2m, 2m + 1 (read_columns).
    template <int V>
    static __device__ __forceinline__ int unit(int r, int u)
    {
        const int f = V == 16 ? (r & 7) << 1 | (r >> 3 & 1) : V == 8 ? (r & 6) | (r >> 3 & 1) : r >> 2 & 3;
        return r * V + (u ^ f);
    }
};

// Eight contraction rows of one column: rows r0 + 0..3 and r1 + 0..3 of a
// plane with V units per row, 16 columns from col per 16-lane group (the
// lane's own column is col + lane % 16).  The read takes a row from four
// lanes, 4 elements each.
template <int D, int V>
__device__ __forceinline__ u32x4 read_columns(const u32x4 *plane, int r0, int r1, int col, int lane)
{
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    const int li = lane & 15, c = col + 4 * (li & 3);
    const char *base = (const char *)plane + (c & 4) * 2;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4 *)(base + 16 * BwdTiles<D>::template unit<V>(r0 + (li >> 2), c >> 3)));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_s16x4 *)(base + 16 * BwdTiles<D>::template unit<V>(r1 + (li >> 2), c >> 3)));
    struct Pair {
        s16x4 a, b;
    };
    return __builtin_bit_cast(u32x4, Pair{lo, hi});
}

// P and dP of 32 query rows from m0 and 32 keys from n0 on the fp32 matrix
// instruction, straight from global memory, for what the split cannot carry;
// 0 where masked.  Register i holds row acc_row(i, h32), a lane
// column l32: rows are queries and columns keys, or (KEY_ROWS) the other way.
template <int D, bool CAUSAL, bool KEY_ROWS>
__device__ __forceinline__ void block_f32(const BwdArgs &a, int64_t in_base, int64_t out_base, const float *l2p,
                                          int m0, int n0, f32x16 &p, f32x16 &dp)
{
    const int lane = threadIdx.x & 63, h32 = lane >> 5, l32 = lane & 31;
    const int64_t mr = min(m0 + l32, a.S - 1), nr = min(n0 + l32, a.S - 1);
    const float *const qr = a.q + in_base + mr * a.in_ss + h32 * (D / 2), *const kr = a.k + in_base + nr * a.in_ss + h32 * (D / 2);
    const float *const gr = a.dout + out_base + mr * a.out_ss + h32 * (D / 2), *const vr = a.v + in_base + nr * a.in_ss + h32 * (D / 2);
    f32x16 s = zero16();
    dp = zero16();
#pragma unroll 2
    for (int kk = 0; kk < D / 2; kk += 4) {
        const f32x4 qv = *(const f32x4 *)(qr + kk), kv = *(const f32x4 *)(kr + kk);
        const f32x4 gv = *(const f32x4 *)(gr + kk), vv = *(const f32x4 *)(vr + kk);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s = KEY_ROWS ? mfma_32x32x2(kv[j], qv[j], s) : mfma_32x32x2(qv[j], kv[j], s);
            dp = KEY_ROWS ? mfma_32x32x2(vv[j], gv[j], dp) : mfma_32x32x2(gv[j], vv[j], dp);
        }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int m = m0 + (KEY_ROWS ? l32 : acc_row(i, h32)), n = n0 + (KEY_ROWS ? acc_row(i, h32) : l32);
        const bool seen = m < a.S && n < a.S && (!CAUSAL || n <= m);
        p[i] = seen ? __builtin_amdgcn_exp2f(fmaf(s[i], a.c, -l2p[m])) : 0.0f;
        dp[i] = seen ? dp[i] : 0.0f;
    }
}

__device__ __forceinline__ float not_finite(const f32x16 &v, float probe)
{
#pragma unroll
    for (int i = 0; i < 16; ++i) probe = fmaf(v[i], 0.0f, probe);
    return probe;
}

template <int D, bool CAUSAL, int DQ>
__global__ __launch_bounds__(kThreads, D == 32 ? 2 : 1) void attn_bwd_kernel(BwdArgs a)
{
    typedef BwdTiles<D> T;
    constexpr int U = T::U, KS = T::KS, DB = T::DB, G = T::G;
    __shared__ u32x4 Kp[3 * T::KPL], Qp[3 * T::QPL], Gp[3 * T::QPL];
    __shared__ u32x4 Sp_own[T::kShared ? 1 : 3 * T::SPL];
    __shared__ float St[2][2 * kBq];  // lse2 and delta of a block, two blocks
    __shared__ int lost_at;  // the step that met what the split cannot carry
    __shared__ float kmax_in[kWaves];
    u32x4 *const Sp = T::kShared ? Gp : Sp_own;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h32 = lane >> 5;
    const int l32 = lane & 31;

    const int BH = (int)(gridDim.x / a.nkb);
    const int kb = blockIdx.x / BH;  // ascending: the longest causal rows first
    const int bh = blockIdx.x - kb * BH;
    const int b = bh / a.H;
    const int hh = bh - b * a.H;
    const int S = a.S;
    const int n0 = kb * kBk, n0w = n0 + kBkw * w;
    const int64_t in_base = (int64_t)b * a.in_sb + (int64_t)hh * a.in_sh;
    const int64_t out_base = (int64_t)b * a.out_sb + (int64_t)hh * a.out_sh;
    const float *const qbase = a.q + in_base, *const gbase = a.dout + out_base;
    const float *const l2p = a.lse2 + (int64_t)bh * a.S_pad, *const dlp = a.delta + (int64_t)bh * a.S_pad;

    const unsigned parity = (unsigned)(kb & 1) << 31;
    const unsigned ksgn = sign_of(n0w + l32);   // on this lane's key of K and V, so on S and dP
    const unsigned psgn = ksgn ^ parity;        // on P and dS
    // Operands are scaled as split_bf16.h says: S, dP, dK, dV and dQ carry
    // 2^32, P and dS 2^16.  Q and K are multiplied in two steps, so that
    // elements from 2^44 on become infinite and S NaN: below that no sum in S
    // passes 2^95 (one of minus infinity would hide in a weight of 0).
    constexpr float kLift = 0x1p84f, kDrop = 0x1p-68f, kUnscale = 1.0f / (kSplitScale * kSplitScale);
    static_assert(kLift * kDrop == kSplitScale, "in all");
    // A scale that would become denormal is lost too.
    const float cs = a.scale > 0.0f && a.scale < 0x1p-94f ? NAN : flip(a.c * kUnscale, ksgn);
    const float pscale = flip(kSplitScale, psgn);
    const float dqscale = flip(a.scale * kUnscale, parity);

    BwdBlock k;
    k.dqp = a.dq + in_base;
    k.turns = DQ == kDqOrdered ? a.order + (int64_t)bh * (a.S_pad / 16) : nullptr;
    k.S = S;
    k.nq = (S + kBq - 1) / kBq;
    k.w = w;
    k.kb = kb;
    k.in_ss = (int)a.in_ss;  // row strides < 2^24, checked on the host

    const int qstart = CAUSAL ? n0 / kBq : 0;

    // ---- staging of the Q and dO rows ----
    // Addresses derive from copies of the lane and thread index that each
    // block makes opaque, so that the compiler keeps none live across the loop.
    int ln = lane, ti = tid;
    float qreg[G][8], greg[G][8], streg = 0.0f;
    auto load_rows = [&](const float *base, int64_t ss, int m0, float (&reg)[G][8]) {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int i = ti + kThreads * g, r = i / U, u = i % U;
            if (T::QPL < kThreads && i >= T::QPL) continue;
            const float *src = base + (int64_t)min(m0 + r, S - 1) * ss + 8 * u;
            const f32x4 x = *(const f32x4 *)src, y = *(const f32x4 *)(src + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) reg[g][j] = x[j], reg[g][4 + j] = y[j];
        }
    };
    unsigned part[3][2];
    // Pair i (of 4) of group g of Q or dO; every second one stores half a unit
    // of each plane.
    auto split_store = [&](bool q, int g, int i, u32x4 *to) {
        const float x = q ? qreg[g][2 * i] * kLift * kDrop : greg[g][2 * i] * kSplitScale;
        const float y = q ? qreg[g][2 * i + 1] * kLift * kDrop : greg[g][2 * i + 1] * kSplitScale;
        split_pair(x, y, part[0][i & 1], part[1][i & 1], part[2][i & 1]);
        if (i & 1) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            const int e = ti + kThreads * g;
            if (T::QPL < kThreads && e >= T::QPL) return;
            u32x2 *p = (u32x2 *)(to + T::template unit<U>(e / U, e % U)) + i / 2;
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) p[2 * pl * T::QPL] = u32x2{part[pl][0], part[pl][1]};
        }
    };
    auto m_of = [&](int qb) { return min(qb, k.nq - 1) * kBq; };  // past the end: the last again
    auto load_stats = [&](int m0) {  // padded rows: +inf and 0
        if (tid < 2 * kBq) streg = tid < kBq ? l2p[m0 + tid] : dlp[m0 + tid - kBq];
    };

    // First block: Q and the statistics here, dO in its step.
    load_rows(qbase, a.in_ss, qstart * kBq, qreg);
    load_rows(gbase, a.out_ss, qstart * kBq, greg);
    load_stats(qstart * kBq);

    // K of the workgroup's keys to LDS, V of this lane's key to registers
    // (rows past S re-read row S - 1; their P is 0).
    Split8 vf[KS];
    bool klost;    // K cannot be carried: not even a dS of 0 may meet it
    float dslimit;  // dS times this overflows before dQ, its sum over 128 keys
    {
        constexpr int N = T::KPL / kThreads;
        f32x4 kr[N][2], vr[KS][2];
#pragma unroll
        for (int it = 0; it < N; ++it) {
            const int i = it * kThreads + tid, r = i / U, u = i % U;
            const float *src = a.k + in_base + (int64_t)min(n0 + r, S - 1) * a.in_ss + 8 * u;
            kr[it][0] = *(const f32x4 *)src, kr[it][1] = *(const f32x4 *)(src + 4);
        }
        const float *vsrc = a.v + in_base + (int64_t)min(n0w + l32, S - 1) * a.in_ss + 8 * h32;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
            vr[ks][0] = *(const f32x4 *)(vsrc + 16 * ks), vr[ks][1] = *(const f32x4 *)(vsrc + 16 * ks + 4);

        float probe = 0.0f, kmax = 0.0f;
#pragma unroll
        for (int it = 0; it < N; ++it) {
            const int i = it * kThreads + tid, r = i / U, u = i % U;
            const float f = flip(kDrop, sign_of(n0 + r));
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                v[j] = kr[it][j / 4][j % 4] * kLift * f;
                probe = fmaf(v[j], 0.0f, probe);
                kmax = fmaxf(kmax, fabsf(v[j]));
            }
            const Split8 sp = split8(v);
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) Kp[pl * T::KPL + T::template unit<U>(r, u)] = sp.part[pl];
        }
        klost = __ballot(probe != 0.0f) != 0;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) kmax = fmaxf(kmax, __shfl_xor(kmax, o));
        if (lane == 0) kmax_in[w] = kmax;
        __syncthreads();
        kmax = fmaxf(fmaxf(kmax_in[0], kmax_in[1]), fmaxf(kmax_in[2], kmax_in[3]));
        // The sum over dS below may cancel once: a factor 2 beside the 2^7.
        dslimit = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(float_bits(kmax * 0x1p9f)));
        const float f = flip(kSplitScale, ksgn);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = vr[ks][j / 4][j % 4] * f;
            vf[ks] = split8(v);
        }
    }

    f32x16 dvacc[DB], dkacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) {
        dvacc[db] = zero16();
        dkacc[db] = zero16();
    }

    const int key = n0w + l32;
    // P[m][n] = 0 where mask_t - m0 > 8(i/4) + i%4: keys past the sequence
    // end, and causally keys past the row.
    const int mask_t = key >= S ? 1 << 30 : CAUSAL ? key - 4 * h32 : -(1 << 30);  // m0 < 2^28

    auto step = [&](auto mask, auto mode, int qb) {
        constexpr bool MASK = decltype(mask)::value;
        constexpr int Q = decltype(mode)::value;
        asm volatile("" : "+v"(ln), "+v"(ti));
        const int m0 = qb * kBq;
        const float *const st = St[(qb - qstart) & 1];
        const int lq = ln & 31, lh = ln >> 5, gl = (ln >> 4) & 1;  // column half of a 16-lane group
        int polled = 0;
        if (Q == kDqOrdered) polled = order_poll(k.turns + (m0 >> 4));

        // Each phase reads a chunk's operands while the one before is
        // multiplied (x, y: two sets in turn).
        Split8 x[2], y[2];

        // ---- S; beside it this block's dO is split and stored ----
        f32x16 sacc, pacc;
        auto read_qk = [&](int c) {
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) {
                x[c & 1].part[pl] = Qp[pl * T::QPL + T::template unit<U>(lq, 2 * c + lh)];
                y[c & 1].part[pl] = Kp[pl * T::KPL + kBkw * U * w + T::template unit<U>(lq, 2 * c + lh)];
            }
        };
        read_qk(0);
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            if (c + 1 < KS) read_qk(c + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (c == 0) sacc = zero16();
#pragma unroll
            for (int t = 0; t < 6; ++t) mfma_split_term(t, x[c & 1], y[c & 1], sacc);
#pragma unroll
            for (int u = 0; u < 4 * G; ++u)
                if (u * KS / (4 * G) == c) split_store(false, u / 4, u % 4, Gp);
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();  // dO complete
        __builtin_amdgcn_sched_barrier(0);
        load_rows(gbase, a.out_ss, m_of(qb + 1), greg);

        // ---- dP; beside it P ----
        f32x4 l2v[4], dlv[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            l2v[g] = *(const f32x4 *)&st[8 * g + 4 * lh];
            dlv[g] = *(const f32x4 *)&st[kBq + 8 * g + 4 * lh];
        }
        Split8 pf[2], sf[2];  // P^T, dS^T of the block's first and second 16 rows
        auto p_pair = [&](int i) {
            float p[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int r = i + j;
                p[j] = __builtin_amdgcn_exp2f(fmaf(sacc[r], cs, -l2v[r >> 2][r & 3]));
                if (MASK) p[j] = mask_t - m0 > 8 * (r >> 2) + (r & 3) ? 0.0f : p[j];
                p[j] *= pscale;
                sacc[r] = p[j];
            }
            unsigned h, m, l;
            split_pair(p[0], p[1], h, m, l);
            Split8 &f = pf[i / 8];
            f.part[0][i / 2 % 4] = h, f.part[1][i / 2 % 4] = m, f.part[2][i / 2 % 4] = l;
        };
        auto read_g = [&](int c) {
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) x[c & 1].part[pl] = Gp[pl * T::QPL + T::template unit<U>(lq, 2 * c + lh)];
        };
        // Columns of dO or Q: 16 rows from 16 s, column block db.
        auto read_t = [&](const u32x4 *rows, int c, Split8 &f) {
            const int s = c / DB, db = c % DB;
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                f.part[pl] = read_columns<D, U>(rows + pl * T::QPL, 16 * s + 4 * lh, 16 * s + 8 + 4 * lh,
                                                32 * db + 16 * gl, ln);
        };
        read_g(0);
#pragma unroll
        for (int c = 0; c < KS; ++c) {
            if (c + 1 < KS)
                read_g(c + 1);
            else
                read_t(Gp, 0, y[0]);
            __builtin_amdgcn_sched_barrier(0);
            if (c == 0) pacc = zero16();
#pragma unroll
            for (int t = 0; t < 6; ++t) mfma_split_term(t, x[c & 1], vf[c], pacc);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (u * KS / 8 == c) p_pair(2 * u);
            __builtin_amdgcn_sched_barrier(0);
        }

        // ---- dV; beside it dS ----
        float probe = 0.0f;  // not finite if some dS is not or dQ might not be
        auto ds_pair = [&](int i) {
            float d[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int r = i + j;
                d[j] = sacc[r] * fmaf(pacc[r], flip(kUnscale, ksgn), -dlv[r >> 2][r & 3]);
                probe = fmaf(d[j], dslimit, probe);
            }
            unsigned h, m, l;
            split_pair(d[0], d[1], h, m, l);
            Split8 &f = sf[i / 8];
            f.part[0][i / 2 % 4] = h, f.part[1][i / 2 % 4] = m, f.part[2][i / 2 % 4] = l;
        };
#pragma unroll
        for (int c = 0; c < 2 * DB; ++c) {
            if (c + 1 < 2 * DB)
                read_t(Gp, c + 1, y[(c + 1) & 1]);
            else
                read_t(Qp, 0, x[0]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 6; ++t) mfma_split_term(t, pf[c / DB], y[c & 1], dvacc[c % DB]);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (u * 2 * DB / 8 == c) ds_pair(2 * u);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (T::kShared) __syncthreads();  // every wave is done with dO

        // ---- dK; beside it dS to LDS, rows = keys ----
        const int dblk = w % DB, nb = (w / DB) * T::NK;  // this wave's part of dQ
        auto read_kt = [&](int c) {
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                y[c & 1].part[pl] = read_columns<D, U>(Kp + pl * T::KPL, nb + 16 * c + 8 * lh, nb + 16 * c + 8 * lh + 4,
                                                       32 * dblk + 16 * gl, ln);
        };
        auto read_s = [&](int c) {
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                x[c & 1].part[pl] = read_columns<D, 4>(Sp + pl * T::SPL, nb + 16 * c + 8 * lh, nb + 16 * c + 8 * lh + 4,
                                                       16 * gl, ln);
        };
        auto ds_store = [&](int g) {  // rows 8 g + 4 h32 + 0..3 of the block
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            u32x2 *p = (u32x2 *)(Sp + T::template unit<4>(kBkw * w + lq, g)) + lh;
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                p[2 * pl * T::SPL] = u32x2{sf[g / 2].part[pl][2 * (g % 2)], sf[g / 2].part[pl][2 * (g % 2) + 1]};
        };
#pragma unroll
        for (int c = 0; c < 2 * DB; ++c) {
            if (c + 1 < 2 * DB)
                read_t(Qp, c + 1, x[(c + 1) & 1]);
            else
                read_kt(0);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 6; ++t) mfma_split_term(t, sf[c / DB], x[c & 1], dkacc[c % DB]);
#pragma unroll
            for (int g = 0; g < 4; ++g)
                if (g * 2 * DB / 4 == c) ds_store(g);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (tid < 2 * kBq) St[(qb + 1 - qstart) & 1][tid] = streg;
        if ((klost || __ballot(!(fabsf(probe) < INFINITY)) != 0) && lane == 0) lost_at = qb;
        __syncthreads();  // dS complete, every wave done with Q
        const int lost = lost_at;

        // ---- dQ over this wave's share of the keys; beside it the next
        // block's Q is split and stored ----
        f32x16 qacc;
        constexpr int NC = T::NK / 16;
        read_s(0);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (c + 1 < NC) read_s(c + 1), read_kt(c + 1);
            __builtin_amdgcn_sched_barrier(0);
            if (c == 0) qacc = zero16();
#pragma unroll
            for (int t = 0; t < 6; ++t) mfma_split_term(t, x[c & 1], y[c & 1], qacc);
#pragma unroll
            for (int u = 0; u < 4 * G; ++u)
                if (u * NC / (4 * G) == c) split_store(true, u / 4, u % 4, Qp);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_rows(qbase, a.in_ss, m_of(qb + 2), qreg);
        load_stats(m_of(qb + 2));
        if (__builtin_amdgcn_readfirstlane(lost) >= 0) return false;
        dq_store<D, CAUSAL, Q>(a, k, m0, qacc, dqscale, polled);
        if (Q != kDqAtomic && !kDoneAtOnce<D>) order_done(k.turns + (m0 >> 4));
        __syncthreads();  // the next Q complete, every wave done with dS
        return true;
    };

#pragma unroll
    for (int u = 0; u < 4 * G; ++u) split_store(true, u / 4, u % 4, Qp);
    if (tid < 2 * kBq) St[0][tid] = streg;
    if (tid == 0) lost_at = -1;
    load_rows(qbase, a.in_ss, m_of(qstart + 1), qreg);
    load_stats(m_of(qstart + 1));
    __syncthreads();

    auto walk = [&](auto mode) {
        // The blocks that cross the diagonal need the mask; with a partial
        // last key block all do.  (At D = 32 all blocks take the masked copy:
        // a second one made the compiler spill.)
        const int masked = D == 32 ? k.nq : n0w + kBkw > S ? k.nq : CAUSAL ? min(k.nq, qstart + kBk / kBq) : qstart;
        int qb = qstart;
        for (; qb < masked; ++qb)
            if (!step(std::true_type{}, mode, qb)) return;
        if constexpr (D > 32)
            for (; qb < k.nq; ++qb)
                if (!step(std::false_type{}, mode, qb)) return;
    };
    if constexpr (DQ == kDqAtomic) {
        walk(std::integral_constant<int, kDqAtomic>{});
    } else {
        // Deterministic mode: whether the key blocks before this one have
        // added their share of its last tile, and so of all its tiles
        // (ordered dQ, attention_bwd_kernels.h); waves that share dQ columns
        // (D < 128) always wait for each other.
        const int m_last = (k.nq - 1) * kBq;
        const int seen = order_poll(k.turns + (m_last >> 4));
        if (!kDoneAtOnce<D> && __builtin_amdgcn_readfirstlane(seen) >= dq_turn_expect<D, CAUSAL>(a, k, m_last))
            walk(std::integral_constant<int, kDqOrderedFree>{});
        else
            walk(std::integral_constant<int, kDqOrdered>{});
    }

    // What the split cannot carry: the walk ended before dQ of the step
    // lost_at was added, or dK or dV is not finite.  The wave's dK and dV with
    // the fp32 instruction, and below dQ's rest.
    const int lost = __builtin_amdgcn_readfirstlane(lost_at);
    float probe = 0.0f, dkscale = a.scale * kUnscale, dvscale = kUnscale;
    unsigned signs = 0x80000000u;
#pragma unroll
    for (int db = 0; db < DB; ++db) probe = not_finite(dkacc[db], not_finite(dvacc[db], probe));
    if (__ballot(probe != 0.0f) != 0 || lost >= 0) {
        dkscale = a.scale, dvscale = 1.0f, signs = 0;
#pragma unroll
        for (int db = 0; db < DB; ++db) dvacc[db] = zero16(), dkacc[db] = zero16();
        for (int m0 = qstart * kBq; m0 < S; m0 += kBq) {
            f32x16 p, dp;
            block_f32<D, CAUSAL, false>(a, in_base, out_base, l2p, m0, n0w, p, dp);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = m0 + acc_row(i, h32);  // below S_pad
                const int64_t mr = min(m, S - 1);
                const float ds = p[i] * (dp[i] - dlp[m]);
                const float *const gr = gbase + mr * a.out_ss + l32, *const qr = qbase + mr * a.in_ss + l32;
#pragma unroll
                for (int db = 0; db < DB; ++db) {
                    dvacc[db] = mfma_32x32x2(p[i], gr[32 * db], dvacc[db]);
                    dkacc[db] = mfma_32x32x2(ds, qr[32 * db], dkacc[db]);
                }
            }
        }
    }

    // dK (scaled) and dV rows of this wave's keys: register i -> key
    // n0w + acc_row(i, h32), lane -> d = 32 db + l32.
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int n = n0w + acc_row(i, h32);
        if (n >= S) continue;
        const unsigned sg = (sign_of(n) ^ parity) & signs;
        const int64_t off = in_base + (int64_t)n * a.in_ss + l32;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            a.dk[off + 32 * db] = fmaf(dkacc[db][i], flip(dkscale, sg), 0.0f);
            a.dv[off + 32 * db] = fmaf(dvacc[db][i], flip(dvscale, sg), 0.0f);
        }
    }
    if (lost < 0) return;
    const int dblk = w % DB, nb = n0 + (w / DB) * T::NK;
    for (int m0 = lost * kBq; m0 < S; m0 += kBq) {
        int polled = 0;
        if (DQ != kDqAtomic) polled = order_poll(k.turns + (m0 >> 4));
        const float delta = dlp[m0 + l32];
        f32x16 qacc = zero16();
        for (int n = nb; n < nb + T::NK; n += 32) {
            f32x16 p, dp;
            block_f32<D, CAUSAL, true>(a, in_base, out_base, l2p, m0, n, p, dp);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int64_t nr = min(n + acc_row(i, h32), S - 1);
                qacc = mfma_32x32x2(p[i] * (dp[i] - delta), a.k[in_base + nr * a.in_ss + 32 * dblk + l32], qacc);
            }
        }
        dq_store<D, CAUSAL, DQ>(a, k, m0, qacc, a.scale, polled);
        if (DQ != kDqAtomic && !kDoneAtOnce<D>) order_done(k.turns + (m0 >> 4));
    }
}

template <int D, bool CAUSAL>
int launch(const BwdArgs &args, int64_t rows_pad, int nblocks)
{
    constexpr int RPB = 256 / (D / 4);
    hipLaunchKernelGGL((attn_bwd_pre<D>), dim3((unsigned)((rows_pad + RPB - 1) / RPB)), dim3(256), 0, 0, args, rows_pad);
    if (!launch_ok("attn_bwd_pre")) return EMBER_ERR_DEVICE;
    if (args.order)
        hipLaunchKernelGGL((attn_bwd_kernel<D, CAUSAL, kDqOrdered>), dim3(nblocks), dim3(kThreads), 0, 0, args);
    else
        hipLaunchKernelGGL((attn_bwd_kernel<D, CAUSAL, kDqAtomic>), dim3(nblocks), dim3(kThreads), 0, 0, args);
    return launch_ok("attn_bwd_kernel") ? EMBER_OK : EMBER_ERR_DEVICE;
}

}  // namespace

int launch_bwd_tiles(const BwdArgs &args, int D, bool causal, int64_t rows_pad, int nblocks)
{
    switch (D * 2 + (causal ? 1 : 0)) {
        case 64: return launch<32, false>(args, rows_pad, nblocks);
        case 65: return launch<32, true>(args, rows_pad, nblocks);
        case 128: return launch<64, false>(args, rows_pad, nblocks);
        case 129: return launch<64, true>(args, rows_pad, nblocks);
        case 256: return launch<128, false>(args, rows_pad, nblocks);
        default: return launch<128, true>(args, rows_pad, nblocks);
    }
}

}  // namespace ember
