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
//   S   = Q K^T             beside it: next block's dO split and stored
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
// scaled anyway.
//
// What bounds it: at D = 128 one workgroup per CU is one wave per SIMD, so a
// wave's own waits (four barriers and the LDS reads of each block's first
// operands) leave the matrix cores idle: B4 H32 S4096 D128 causal busy 52 % of
// cycles at 1.93 GHz (power limit), LDS busy 35 %, a third of that in bank
// conflicts of the transposing reads.  Hence the vector work laid beside the
// products, and operands read a chunk ahead.  Against the kernel on the fp32
// instruction that it replaced: B4 H32 S4096 D128 causal 10711 -> 8112 us
// (128 -> 169 TFLOP/s), 30 heads of 777 at D = 128 264 -> 170, 32 heads of 1024
// causal 335 -> 211, 4 heads of 300 110 -> 70; D = 32, 64 heads of 1000 causal
// 164 -> 148; in deterministic order 11028 -> 8281 at the first.  Error against
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

template <int D, bool CAUSAL, int DQ>
__global__ __launch_bounds__(kThreads, D == 32 ? 2 : 1) void attn_bwd_kernel(BwdArgs a)
{
    typedef BwdTiles<D> T;
    constexpr int U = T::U, KS = T::KS, DB = T::DB, G = T::G;
    __shared__ u32x4 Kp[3 * T::KPL], Qp[3 * T::QPL], Gp[3 * T::QPL];
    __shared__ u32x4 Sp_own[T::kShared ? 1 : 3 * T::SPL];
    __shared__ unsigned found_in[kWaves];
    __shared__ float St[2][2 * kBq];  // lse2 and delta of a block, two blocks
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
    // Pair i (of 4) of group g; every second one stores half a unit of each plane.
    auto split_store = [&](const float (&reg)[G][8], float f, int g, int i, u32x4 *to) {
        split_pair_full(reg[g][2 * i] * f, reg[g][2 * i + 1] * f, part[0][i & 1], part[1][i & 1], part[2][i & 1]);
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
    // (rows past S re-read row S - 1; their P is 0).  The split of very small
    // numbers, dS = P (dP - delta) among them, would lose bits
    // (split_bf16.h), so an input that is below 2^-63 throughout is scaled by
    // 2^32 as it is split, dS with dO and V, and the results are scaled back,
    // all of it exact.  For K and V the workgroup's keys decide, for Q and dO
    // their first block (with a scale from there, rows below 2^95 are right).
    Split8 vf[KS];
    float kscale, vscale, qscale, gscale;
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

        unsigned kbits = 0, vbits = 0, qbits = 0, gbits = 0;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int it = 0; it < N; ++it) kbits |= float_bits(kr[it][j / 4][j % 4]);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) vbits |= float_bits(vr[ks][j / 4][j % 4]);
            if (T::QPL >= kThreads || tid < T::QPL)
#pragma unroll
                for (int g = 0; g < G; ++g) qbits |= float_bits(qreg[g][j]), gbits |= float_bits(greg[g][j]);
        }
        // 1: some value is at least 2^-63; 2: some value is not zero.
        auto found = [](unsigned bits) {
            return (__ballot((bits & 0x60000000u) != 0) != 0 ? 1u : 0u) | (__ballot((bits & 0x7fffffffu) != 0) != 0 ? 2u : 0u);
        };
        auto scale_of = [](unsigned f) { return (f & 3) == 2 ? 0x1p32f : 1.0f; };
        const unsigned mine = found(kbits) | found(qbits) << 2 | found(gbits) << 4 | found(vbits) << 6;
        if (lane == 0) found_in[w] = mine;
        __syncthreads();
        const unsigned all = __builtin_amdgcn_readfirstlane(found_in[0] | found_in[1] | found_in[2] | found_in[3]);
        kscale = scale_of(all), qscale = scale_of(all >> 2), gscale = scale_of(all >> 4), vscale = scale_of(all >> 6);

#pragma unroll
        for (int it = 0; it < N; ++it) {
            const int i = it * kThreads + tid, r = i / U, u = i % U;
            const float f = flip(kscale, sign_of(n0 + r));
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = kr[it][j / 4][j % 4] * f;
            Split8 sp;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                {
                unsigned h, m, l;
                split_pair_full(v[2 * j], v[2 * j + 1], h, m, l);
                sp.part[0][j] = h, sp.part[1][j] = m, sp.part[2][j] = l;
            }
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) Kp[pl * T::KPL + T::template unit<U>(r, u)] = sp.part[pl];
        }
        const float f = flip(vscale, ksgn);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = vr[ks][j / 4][j % 4] * f;
            vf[ks] = split8(v);
        }
    }
    // S c = sacc * cs; dP and dS carry gscale * vscale, and so delta does.
    const float cs = flip(a.c, ksgn) / (qscale * kscale), dscale = gscale * vscale;
    BwdArgs aq = a;  // what dq_store reads
    aq.scale = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(
                                             float_bits(flip(a.scale / (dscale * kscale), parity))));

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
                if (u * KS / (4 * G) == c) split_store(greg, gscale, u / 4, u % 4, Gp);
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
                p[j] = flip(p[j], psgn);
                sacc[r] = p[j];
            }
            unsigned h, m, l;
            split_pair(p[0], p[1], h, m, l);
            Split8 &f = pf[i / 8];
            asm volatile("" : "+v"(h), "+v"(m), "+v"(l));  // here, not behind the branch below
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

        // What the split cannot carry (split_bf16.h): S and dP again with the
        // fp32 instruction, straight from global memory, so that an infinite
        // key that gets no weight stays without.  (dV, dK and dQ of what an
        // infinity does reach are not finite, and may be NaN.)
        float probe = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; ++i) probe = fmaf(pacc[i], 0.0f, fmaf(sacc[i], 0.0f, probe));
        if (__ballot(probe != 0.0f) != 0) {
            const int64_t mr = min(m0 + lq, S - 1), nr = min(key, S - 1);
            const float *qr = qbase + mr * a.in_ss + lh * (D / 2), *gr = gbase + mr * a.out_ss + lh * (D / 2);
            const float *kr = a.k + in_base + nr * a.in_ss + lh * (D / 2), *vr = a.v + in_base + nr * a.in_ss + lh * (D / 2);
            sacc = zero16();
            pacc = zero16();
            for (int kk = 0; kk < D / 2; ++kk) {
                sacc = mfma_32x32x2(qr[kk], kr[kk], sacc);
                pacc = mfma_32x32x2(gr[kk], vr[kk], pacc);
            }
            sacc *= flip(qscale * kscale, ksgn);
            pacc *= flip(gscale * vscale, ksgn);
#pragma unroll
            for (int u = 0; u < 8; ++u) p_pair(2 * u);
        }

        // ---- dV; beside it dS ----
        auto ds_pair = [&](int i) {
            float d[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int r = i + j;
                d[j] = sacc[r] * fmaf(pacc[r], flip(1.0f, ksgn), -dlv[r >> 2][r & 3]);
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
        if (tid < 2 * kBq) St[(qb + 1 - qstart) & 1][tid] = tid < kBq ? streg : streg * dscale;
        __syncthreads();  // dS complete, every wave done with Q

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
                if (u * NC / (4 * G) == c) split_store(qreg, qscale, u / 4, u % 4, Qp);
            __builtin_amdgcn_sched_barrier(0);
        }
        load_rows(qbase, a.in_ss, m_of(qb + 2), qreg);
        load_stats(m_of(qb + 2));
        dq_store<D, CAUSAL, Q>(aq, k, m0, qacc, polled);
        if (Q != kDqAtomic && !kDoneAtOnce<D>) order_done(k.turns + (m0 >> 4));
        __syncthreads();  // the next Q complete, every wave done with dS
    };

#pragma unroll
    for (int u = 0; u < 4 * G; ++u) split_store(qreg, qscale, u / 4, u % 4, Qp);
    if (tid < 2 * kBq) St[0][tid] = tid < kBq ? streg : streg * dscale;
    load_rows(qbase, a.in_ss, m_of(qstart + 1), qreg);
    load_stats(m_of(qstart + 1));
    __syncthreads();

    auto walk = [&](auto mode) {
        // The blocks that cross the diagonal need the mask; with a partial
        // last key block all do.  (At D = 32 all blocks take the masked copy:
        // a second one made the compiler spill.)
        const int masked = D == 32 ? k.nq : n0w + kBkw > S ? k.nq : CAUSAL ? min(k.nq, qstart + kBk / kBq) : qstart;
        int qb = qstart;
        for (; qb < masked; ++qb) step(std::true_type{}, mode, qb);
        if constexpr (D > 32)
            for (; qb < k.nq; ++qb) step(std::false_type{}, mode, qb);
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

    // dK (scaled) and dV rows of this wave's keys: register i -> key
    // n0w + acc_row(i, h32), lane -> d = 32 db + l32.
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int n = n0w + acc_row(i, h32);
        if (n >= S) continue;
        const unsigned sg = sign_of(n) ^ parity;
        const int64_t off = in_base + (int64_t)n * a.in_ss + l32;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            a.dk[off + 32 * db] = fmaf(dkacc[db][i], flip(a.scale / (dscale * qscale), sg), 0.0f);
            a.dv[off + 32 * db] = fmaf(dvacc[db][i], flip(1.0f / gscale, sg), 0.0f);
        }
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
