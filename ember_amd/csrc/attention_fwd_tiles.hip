// attention_fwd_tiles.hip -- the fused attention forward for S > 64 on the
// bf16 matrix cores at fp32 precision (split_bf16.h).
//
// One workgroup = 8 waves (or 4, where that many fill the chip) of 32 queries
// of one head.  The keys are walked in tiles (32 keys at D = 128, 64 at 64,
// 128 at 32: 4096 elements).  A tile's K and V are loaded once per workgroup
// into registers, split into three bf16 parts on the way into LDS, and read
// from there by every wave:
//   S^T (keys x 32 queries) = K . Q^T     -- Q^T's parts resident in registers
//   online softmax over keys, as in attention_fwd.hip: base 2, scale folded
//   into one FMA per score, lazy rescaling
//   O^T (D x 32 queries) += V^T . P^T     -- P^T split where it stands: the
//                                            S^T accumulator's registers are
//                                            the operand's contraction slots
// V is stored to LDS transposed, its keys in the order in which the
// accumulator holds them, so that both operands are 16-byte LDS reads.
//
// LDS holds two tiles of K and V (96 KB; 48 KB for 4 waves at D < 128), one
// barrier per tile; tile t+1 is split and stored, and t+2 loaded, in between
// the S products of tile t.
//
// What bounds it: the power limit, through the matrix cores and the vector
// work beside them (B4 H32 S4096 D128 causal: cores busy 66 % of cycles at
// 1.74 GHz, 4.3 vector instructions to a matrix one; without a limit the clock
// is 2.4 GHz).
// Tried against it and dropped: the two waves of a SIMD half a tile apart, so
// that one's softmax meets the other's products (a third V buffer; 2971
// against 2821 us there).  Against the fp32 instruction's kernel it replaced:
// B4 H32 S4096 D128 causal 3980 -> 2660 us (138 -> 207 TFLOP/s), B8 H16 S2048
// D64 causal 539 -> 388 (127 -> 177), B2 H8 S4096 D128 963 -> 624 (143 -> 220),
// 30 heads of 777 at D = 128 111 -> 86; error of O against float64 5.7e-7 ->
// 4.6e-7, 4.1e-7 -> 3.3e-7, 1.3e-6 -> 1.0e-6, 6.7e-7 -> 5.4e-7.
#include <math.h>

#include <type_traits>

#include "attention_fwd.h"
#include "common.h"
#include "mfma.h"
#include "split_bf16.h"

namespace ember {
namespace {

constexpr float kLn2 = 0.6931471805599453f;

template <int D, int NW>
struct Tile {
    static constexpr int NT = 64 * NW;
    static constexpr int KEYS = 8 * NT / D < 32 ? 32 : 8 * NT / D;
    static constexpr int KB = KEYS / 32;           // 32-key blocks
    static constexpr int UK = D / 8, UV = KEYS / 8;  // 16-byte units per K row / V^T row
    static constexpr int PLANE = KEYS * D / 8;     // units per plane (K or V)
    static constexpr int G = PLANE / NT;           // groups of 8 per thread (K or V)
    static constexpr int BUF = 3 * PLANE;
    static_assert(G >= 1 && G * NT == PLANE, "whole groups per thread");

    // Unit u of row r of a plane with U units per row; 16 neighbouring rows
    // of one u fall on different banks.
    template <int U>
    static __device__ __forceinline__ int unit(int r, int u)
    {
        return r * U + (u ^ ((U == 16 ? r : U == 8 ? r >> 1 : r >> 2) & (U - 1)));
    }
};

// One wave's 32 queries from row m0 on the fp32 matrix instruction, straight
// from global memory: for what the split cannot carry (split_bf16.h).
template <int D, bool CAUSAL>
__device__ __forceinline__ void rows_f32(const FwdArgs &a, int b, int hh, int bh, int m0)
{
    constexpr int DH = D / 2, DB = D / 32;
    const int lane = threadIdx.x & 63, h32 = lane >> 5, l32 = lane & 31;
    const int S = a.S, mq = m0 + l32;
    const int64_t base = (int64_t)b * a.in_sb + (int64_t)hh * a.in_sh;
    const float *qrow = a.q + base + (int64_t)min(mq, S - 1) * a.in_ss + h32 * DH;
    f32x16 oacc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) oacc[db] = zero16();
    float mrun = -INFINITY, lrun = 0.0f;
    const int kend = CAUSAL ? min(S, m0 + 32) : S;
    for (int n0 = 0; n0 < kend; n0 += 32) {
        const float *krow = a.k + base + (int64_t)min(n0 + l32, S - 1) * a.in_ss + h32 * DH;
        f32x16 s = zero16();
#pragma unroll 4
        for (int kk = 0; kk < DH; ++kk) s = mfma_32x32x2(krow[kk], qrow[kk], s);
        float tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int n = n0 + acc_row(i, h32);
            s[i] = (n < S) & (!CAUSAL | (n <= mq)) ? s[i] : -INFINITY;
            tmax = fmaxf(tmax, s[i]);
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32)) * a.c;
        if (__ballot(tmax > mrun + 8.0f) != 0) {
            const float mnew = fmaxf(mrun, tmax);
            const float alpha = __builtin_amdgcn_exp2f(mrun - mnew);
            mrun = mnew;
            lrun *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = s[i] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(fmaf(s[i], a.c, -mrun));
            lrun += s[i];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float *vrow = a.v + base + (int64_t)min(n0 + acc_row(i, h32), S - 1) * a.in_ss + l32;
#pragma unroll
            for (int db = 0; db < DB; ++db) oacc[db] = mfma_32x32x2(vrow[32 * db], s[i], oacc[db]);
        }
    }
    const float ltot = lrun + __shfl_xor(lrun, 32);
    if (mq < S) {
        const float inv = 1.0f / ltot;
        float *orow = a.o + (int64_t)b * a.out_sb + (int64_t)hh * a.out_sh + (int64_t)mq * a.out_ss;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) orow[32 * db + acc_row(i, h32)] = oacc[db][i] * inv;
        if (h32 == 0) a.lse[(int64_t)bh * S + mq] = (mrun + log2f(ltot)) * kLn2;
    }
}

// Query blocks of a workgroup (see launch_waves for which launch takes which):
//   kOne   one block of 32 NW queries, causally the long walks first;
//   kBoth  (causal, NW = 8) blocks nqb - 1 - p and p of 128 queries, half the
//          waves each: the second block's key tiles are the first ones of the first
//          block's, staged once for both;
//   kTurn  (causal, NW = 8) blocks nqb - 1 - p and p of 256 queries one after
//          the other: the same number of key tiles for every workgroup.
constexpr int kOne = 0, kBoth = 1, kTurn = 2;

template <int D, bool CAUSAL, int NW, int BLOCKS>
__global__ __launch_bounds__(64 * NW, NW == 4 && D < 128 ? 3 : 1) void attn_fwd_kernel(FwdArgs a)
{
    typedef Tile<D, NW> T;
    constexpr int DB = D / 32, KS = D / 16, KB = T::KB, NT = T::NT, G = T::G;
    constexpr int PF = D == 128 && NW == 8 ? 1 : 2;  // K operand register sets
    __shared__ u32x4 Ks[2 * T::BUF], Vs[2 * T::BUF];
    __shared__ int big;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h32 = lane >> 5;
    const int l32 = lane & 31;

    const int per_head = BLOCKS == kOne ? a.nqb : (a.nqb + 1) / 2;
    const int BH = (int)(gridDim.x / per_head);
    const int qbr = blockIdx.x / BH;
    const int bh = blockIdx.x - qbr * BH;
    const int b = bh / a.H;
    const int hh = bh - b * a.H;
    const int S = a.S;
    constexpr float kBig = 0x1p44f * kSplitScale;
    const float c = a.c / (kSplitScale * kSplitScale);
    const int64_t in_base = (int64_t)b * a.in_sb + (int64_t)hh * a.in_sh;
    const float *__restrict__ kbase = a.k + in_base;
    const float *__restrict__ vbase = a.v + in_base;

    auto run_block = [&](int qb) {
        // qb: the (first) block.  The waves of one SIMD (w and w + 4) take
        // rows 32 w and 32 (7 - w) of a 256-query block: equal causal work.
        constexpr int BQ = BLOCKS == kBoth ? 16 * NW : 32 * NW;
        const int q0 = BQ * qb;
        const bool second = BLOCKS == kBoth && w >= NW / 2;
        const int m0 = second ? BQ * (a.nqb - 1 - qb) + 32 * (w - NW / 2) : q0 + 32 * (w >= 4 ? 11 - w : w);
        const bool idle = second && qb == a.nqb - 1 - qb;  // an odd nqb's middle block is alone
        const int mq = m0 + l32;
        // O^T's columns carry 2^32 and the query's sign (split_bf16.h).
        const float pscale = flip(kSplitScale, sign_of(mq));
        const int kend = CAUSAL ? min(S, q0 + BQ) : S;
        const int ntiles = (kend + T::KEYS - 1) / T::KEYS;

        // Addresses derive from copies of the lane and thread index that each
        // tile makes opaque, so that the compiler computes them there and
        // keeps none of them live across the loop.
        int ln = lane, ti = tid;

        // ---- staging ----
        float kreg[G][8], vreg[G][8];
        float top = 0.0f;  // largest magnitude of the Q and K elements split, scaled
        auto load_k = [&](int n0, int g) {
            const int i = ti + NT * g, r = i / T::UK, u = i % T::UK;
            const float *src = kbase + (int64_t)min(n0 + r, S - 1) * a.in_ss + 8 * u;
            const f32x4 x = *(const f32x4 *)src, y = *(const f32x4 *)(src + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) kreg[g][j] = x[j], kreg[g][4 + j] = y[j];
        };
        auto load_v = [&](int n0, int g) {
            const int i = ti + NT * g, d = i % D;
            int uv = i / D;
            if (D >= 64) uv = __builtin_amdgcn_readfirstlane(uv);
            const int key = n0 + 32 * (uv / 4) + 16 * (uv / 2 % 2) + 4 * (uv % 2);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float *row = vbase + (int64_t)min(key + 8 * (j / 4) + j % 4, S - 1) * a.in_ss;
                vreg[g][j] = *(const float *)((const char *)row + 4u * (unsigned)d);
            }
        };
        unsigned part[3][2];
        // Pair i (of 4) of group g of K (v = false) or V; every second one
        // stores half a unit of each plane.
        auto split_store = [&](bool v, int g, int i, u32x4 *kn, u32x4 *vn) {
            const float x = (v ? vreg[g][2 * i] : kreg[g][2 * i]) * kSplitScale;
            const float y = (v ? vreg[g][2 * i + 1] : kreg[g][2 * i + 1]) * kSplitScale;
            if (!v) {
                top = fmaxf(top, fmaxf(fabsf(x), fabsf(y)));
                asm volatile("" : "+v"(top));  // here, so that x and y die here
            }
            split_pair(x, y, part[0][i & 1], part[1][i & 1], part[2][i & 1]);
            if (i & 1) {
                typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
                const int e = ti + NT * g;
                u32x2 *to = (u32x2 *)(v ? vn + T::template unit<T::UV>(e % D, e / D)
                                        : kn + T::template unit<T::UK>(e / T::UK, e % T::UK)) + i / 2;
#pragma unroll
                for (int pl = 0; pl < 3; ++pl) to[2 * pl * T::PLANE] = u32x2{part[pl][0], part[pl][1]};
            }
        };
        constexpr int NU = 8 * G;  // pairs to split per tile
        auto stage_unit = [&](int u, u32x4 *kn, u32x4 *vn) { split_store(u / 4 >= G, u / 4 % G, u % 4, kn, vn); };
        // The group whose last pair was unit u: its registers take the next tile.
        auto load_unit = [&](int u, int nnext) {
            if (u % 4 == 3) u / 4 >= G ? load_v(nnext, u / 4 % G) : load_k(nnext, u / 4 % G);
        };
        auto stage_all = [&](u32x4 *kn, u32x4 *vn, int nnext) {
#pragma unroll
            for (int u = 0; u < NU; ++u) stage_unit(u, kn, vn);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NU; ++u) load_unit(u, nnext);
        };
        auto tile_n0 = [&](int t) { return min(t, ntiles - 1) * T::KEYS; };  // past the end: the last again

#pragma unroll
        for (int g = 0; g < G; ++g) load_k(0, g), load_v(0, g);
        // Q^T's parts, the operand of k-step ks: d = 16 ks + 8 h32 .. + 7.
        Split8 qf[KS];
        {
            const float *src = a.q + in_base + (int64_t)min(mq, S - 1) * a.in_ss + 8 * h32;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float x[8];
                const f32x4 t0 = *(const f32x4 *)(src + 16 * ks), t1 = *(const f32x4 *)(src + 16 * ks + 4);
#pragma unroll
                for (int j = 0; j < 4; ++j) x[j] = t0[j] * kSplitScale, x[4 + j] = t1[j] * kSplitScale;
#pragma unroll
                for (int j = 0; j < 8; ++j) top = fmaxf(top, fabsf(x[j]));
                qf[ks] = split8(x);
            }
        }
        asm volatile("" : "+v"(top));
        if (tid == 0) big = a.c > 0.0f && a.c < 0x1p-94f;  // c below would be denormal
        stage_all(Ks, Vs, tile_n0(1));
        __syncthreads();

        f32x16 oacc[DB], sacc[KB];
#pragma unroll
        for (int db = 0; db < DB; ++db) oacc[db] = zero16();
        float mrun = -INFINITY, lrun = 0.0f;
        Split8 pf[2 * KB];

        // S^T of the tile in kt, with the staging of the next tile in between.
        auto scores = [&](const u32x4 *kt, u32x4 *kn, u32x4 *vn, int nnext) {
            Split8 kf[PF];
            auto read = [&](int c, Split8 &f) {
                const int ks = c / KB, blk = c % KB;
#pragma unroll
                for (int pl = 0; pl < 3; ++pl)
                    f.part[pl] = kt[pl * T::PLANE + 32 * blk * T::UK + T::template unit<T::UK>(ln & 31, 2 * ks + (ln >> 5))];
            };
            if (PF == 2) read(0, kf[0]);
#pragma unroll
            for (int c = 0; c < KS * KB; ++c) {
                if (PF == 1)
                    read(c, kf[0]);
                else if (c + 1 < KS * KB)
                    read(c + 1, kf[(c + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < 6; ++t) {
                    if (c < KB && t == 0) sacc[c] = zero16();
                    mfma_split_term(t, kf[c & (PF - 1)], qf[c / KB], sacc[c % KB]);
                }
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    if (u * (KS * KB) / NU == c) stage_unit(u, kn, vn);
                __builtin_amdgcn_sched_barrier(0);
                // Behind the barrier the old values are dead, so that the
                // loads need no second set of registers.
#pragma unroll
                for (int u = 0; u < NU; ++u)
                    if (u * (KS * KB) / NU == c) load_unit(u, nnext);
            }
        };
        auto softmax = [&](int n0) {
            const bool need_mask = (n0 + T::KEYS > S) || (CAUSAL && n0 + T::KEYS - 1 > m0);
            if (need_mask) {
#pragma unroll
                for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int n = n0 + 32 * blk + acc_row(i, ln >> 5);
                        const bool vis = (n < S) & (!CAUSAL | (n <= m0 + (ln & 31)));
                        sacc[blk][i] = vis ? sacc[blk][i] : -INFINITY;
                    }
            }
            float tmax = -INFINITY;
#pragma unroll
            for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                for (int i = 0; i < 16; i += 2) tmax = fmaxf(tmax, fmaxf(sacc[blk][i], sacc[blk][i + 1]));
            tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
            // Scaled tile max (scale >= 0, checked on the host).  The
            // reference max mrun is raised only when some lane's scores would
            // otherwise exceed it by more than 2^8: the result is the same
            // softmax, and most tiles skip the rescale of O.  Tile 0 holds
            // key 0, visible to every query, so it sets a finite mrun.
            const float tm2 = tmax * c;
            if (__ballot(tm2 > mrun + 8.0f) != 0) {
                const float mnew = fmaxf(mrun, tm2);
                const float alpha = __builtin_amdgcn_exp2f(mrun - mnew);
                mrun = mnew;
                lrun *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db) oacc[db] *= alpha;
            }
            // The tile's sum is added to the running one as a whole: fewer
            // roundings at the size of the total.
            float tsum = 0.0f;
            if (need_mask) {
#pragma unroll
                for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const float sv = sacc[blk][i];
                        sacc[blk][i] = sv == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(fmaf(sv, c, -mrun));
                        tsum += sacc[blk][i];
                    }
            } else {
#pragma unroll
                for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        sacc[blk][i] = __builtin_amdgcn_exp2f(fmaf(sacc[blk][i], c, -mrun));
                        tsum += sacc[blk][i];
                    }
            }
            // P^T's parts, with the query's sign.
#pragma unroll
            for (int blk = 0; blk < KB; ++blk)
#pragma unroll
                for (int i = 0; i < 16; i += 2) {
                    Split8 &f = pf[2 * blk + i / 8];
                    unsigned h, m, l;
                    split_pair(sacc[blk][i] * pscale, sacc[blk][i + 1] * pscale, h, m, l);
                    f.part[0][i / 2 % 4] = h;
                    f.part[1][i / 2 % 4] = m;
                    f.part[2][i / 2 % 4] = l;
                }
            lrun += tsum;
        };
        auto add_v = [&](const u32x4 *vt) {
            Split8 vf[2];
            auto read = [&](int c, Split8 &f) {
                const int s = c / DB, db = c % DB;
#pragma unroll
                for (int pl = 0; pl < 3; ++pl)
                    f.part[pl] = vt[pl * T::PLANE + 32 * db * T::UV + T::template unit<T::UV>(ln & 31, 2 * s + (ln >> 5))];
            };
            read(0, vf[0]);
#pragma unroll
            for (int c = 0; c < 2 * KB * DB; ++c) {
                if (c + 1 < 2 * KB * DB) read(c + 1, vf[(c + 1) & 1]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < 6; ++t) mfma_split_term(t, vf[c & 1], pf[c / DB], oacc[c % DB]);
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        // This wave's last tile; it stages the rest for the others.
        const int nmine = idle ? 0 : CAUSAL ? min(ntiles, (m0 + 32 + T::KEYS - 1) / T::KEYS) : ntiles;
        int t = 0;
        for (; t < nmine; ++t) {
            asm volatile("" : "+v"(ln), "+v"(ti));
            const int cur = (t & 1) * T::BUF, other = T::BUF - cur;
            scores(Ks + cur, Ks + other, Vs + other, tile_n0(t + 2));
            softmax(t * T::KEYS);
            add_v(Vs + cur);
            __syncthreads();
        }
        for (; CAUSAL && t < ntiles; ++t) {
            const int other = T::BUF - (t & 1) * T::BUF;
            stage_all(Ks + other, Vs + other, tile_n0(t + 2));
            __syncthreads();
        }

        // Q and K below 2^44: no score passes 2^95, with its scale fp32's
        // largest number.  (V and the weights show in O.)
        if (top >= kBig) big = 1;
        __syncthreads();
        const float ltot = lrun + __shfl_xor(lrun, 32);
        float probe = ltot * 0.0f;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) probe = fmaf(oacc[db][i], 0.0f, probe);
        if (idle) {
        } else if (__ballot(probe != 0.0f) != 0 || big) {
            rows_f32<D, CAUSAL>(a, b, hh, bh, m0);
        } else if (mq < S) {
            const float inv = 1.0f / (kSplitScale * kSplitScale) / (ltot * pscale) * kSplitScale;
            float *orow = a.o + (int64_t)b * a.out_sb + (int64_t)hh * a.out_sh + (int64_t)mq * a.out_ss;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 16; i += 4) {
                    f32x4 v;
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[j] = fmaf(oacc[db][i + j], inv, 0.0f);
                    *(f32x4 *)(orow + 32 * db + acc_row(i, h32)) = v;
                }
            if (h32 == 0) a.lse[(int64_t)bh * S + mq] = (mrun + log2f(ltot)) * kLn2;
        }
        if (BLOCKS == kTurn) __syncthreads();  // big and the buffers, before the next block
    };

    if constexpr (BLOCKS == kTurn) {
        // The middle block of an odd nqb alone.
        for (int r = qbr == a.nqb - 1 - qbr; r < 2; ++r) run_block(r == 0 ? a.nqb - 1 - qbr : qbr);
    } else {
        run_block(CAUSAL ? a.nqb - 1 - qbr : qbr);
    }
}

template <int D, bool CAUSAL, int NW, int BLOCKS>
int launch(FwdArgs args, int nqb)
{
    args.nqb = nqb;
    const int per_head = BLOCKS == kOne ? nqb : (nqb + 1) / 2;
    hipLaunchKernelGGL((attn_fwd_kernel<D, CAUSAL, NW, BLOCKS>), dim3((unsigned)(per_head * args.nbh)), dim3(64 * NW), 0, 0,
                       args);
    return launch_ok(BLOCKS == kBoth ? "attn_fwd_kernel_pairs" : "attn_fwd_kernel") ? EMBER_OK : EMBER_ERR_DEVICE;
}

template <int D, bool CAUSAL>
int launch_waves(const FwdArgs &args)
{
    const int ncu = device_cu_count();
    const double cus = ncu > 0 ? ncu : 256;
    const int nqb4 = (args.S + 127) / 128, nqb8 = (args.S + 255) / 256;
    if constexpr (CAUSAL) {
        // Both blocks of a pair at once where the pairs fit one round; beyond,
        // single blocks (65 heads of 1024 at D = 64: 76 us, 92 as pairs of
        // 64-query blocks in workgroups of four waves).  Measured (us: both /
        // 4 waves, one block / 8 waves, one block): 32 heads of 1024 at D =
        // 128 101 / 105 / 127, 64 heads 111 / 128 / 133, 32 of 2048 at D = 64
        // 110 / 128 / 148, 40 of 640 41 / 39 / 50.
        const double pairs = (double)((nqb4 + 1) / 2) * args.nbh;
        if (nqb4 >= 4 && pairs <= cus) return launch<D, CAUSAL, 8, kBoth>(args, nqb4);
    }
    // Workgroups of 4 waves while that spreads the queries better: relative
    // times of the busiest CU, in units of an 8-wave workgroup's walk.  One
    // 4-wave workgroup alone on its CU takes 0.7 of it (30 heads of 777 at
    // D = 128: 85 us against 117), and up to three share a CU at D < 128 (one
    // at D = 128: LDS and registers).  Measured at D = 64 (4 / 8 waves):
    // 256 heads of 300 38 / 58 us, 96 of 197 18 / 25, 48 of 777 non-causal
    // 73 / 66, 256 of 512 110 / 107; at D = 128: 64 of 700 148 / 100.
    const double b4 = (double)nqb4 * args.nbh / cus, b8 = (double)nqb8 * args.nbh / cus;
    const double x4 = CAUSAL ? fmax(1.0, b4) : ceil(b4), x8 = CAUSAL ? fmax(1.0, b8) : ceil(b8);
    if ((D == 128 ? 0.73 * x4 : fmax(0.7, 0.1 + 0.48 * x4)) < x8)
        return launch<D, CAUSAL, 4, kOne>(args, nqb4);
    if constexpr (CAUSAL && D >= 64) {
        // Two blocks in turn where that leaves every CU the same number of
        // pairs, or enough of them: 128 heads of 2048 at D = 64 405 -> 389
        // us, of 4096 at D = 128 2844 -> 2782 (D = 32: 938 -> 963, so not).
        const int64_t pairs = (int64_t)(nqb8 + 1) / 2 * args.nbh;
        if (nqb8 >= 2 && nqb8 % 2 == 0 && (pairs % (int64_t)cus == 0 || pairs >= 4 * (int64_t)cus))
            return launch<D, CAUSAL, 8, kTurn>(args, nqb8);
    }
    return launch<D, CAUSAL, 8, kOne>(args, nqb8);
}

}  // namespace

int launch_fwd_tiles(const FwdArgs &args, int D, bool causal)
{
    switch (D * 2 + (causal ? 1 : 0)) {
        case 64: return launch_waves<32, false>(args);
        case 65: return launch_waves<32, true>(args);
        case 128: return launch_waves<64, false>(args);
        case 129: return launch_waves<64, true>(args);
        case 256: return launch_waves<128, false>(args);
        default: return launch_waves<128, true>(args);
    }
}

}  // namespace ember
