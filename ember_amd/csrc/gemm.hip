// gemm.hip -- fp32 GEMM on gfx950 matrix cores behind Ember's matmul ABI.
//
// Replaces the reference's cuBLAS calls (src/tensor/operators_gpu.cu:114-136):
//   matmul(a, b, out, n, m, k):          out(n x m) = a(n x k) @ b(k x m)
//   matmul_batched(..., batch, n, m, k): the same per batch with strides
//                                        n*k, k*m, n*m
// and adds gemm_ex, which also takes either operand transposed in place
// (a stored k x n, b stored m x k: the weight- and input-gradient products of
// a Linear layer, ember/nn/layers.py:50-56, without materialising T(x)) and
// the fused epilogue of linear_fwd, all row-major fp32.
//
// Products run on the bf16 matrix cores at fp32 precision: every operand is
// split exactly into three bf16 parts (split_bf16.h), and six of the nine
// part products are accumulated in fp32.  One kernel covers every shape,
// orientation and alignment; choose_gemm (gemm_shape.h) picks its tile.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_shape.h"
#include "mfma.h"
#include "split_bf16.h"

namespace ember {
namespace {

struct GemmArgs {
    const float *a, *b;
    float *c;
    int n, m, k;
    int lda, ldb;        // row pitch of a and b as stored (k or n; m or k)
    int64_t sa, sb, sc;  // batch strides (elements)
    int tiles_n, tiles_m;
    int tile0;           // first tile of this launch
    int kchunk;          // split-K: k range of one blockIdx.z (multiple of 32)
    float *part;         // split-K partial sums [ksplit][batch][n][m]
    // Epilogue (all optional): out = act(acc + bias[col]) + residual, with
    // pre = acc + bias stored before the activation; residual and pre use
    // out's layout and batch stride.
    const float *bias;
    const float *residual;
    float *pre;
    int act;  // 0 none, 1 Ember's GELU
};

// Ember's GELU, 0.5*x*(1 + tanh(0.8*x)) (ember/nn/activations.py:58), in the
// order Ember's element-wise operators evaluate it.
__device__ __forceinline__ float gelu08(float x)
{
#pragma clang fp contract(off)
    return (x * 0.5f) * (tanhf(x * 0.8f) + 1.0f);
}

__device__ __forceinline__ float epilogue(const GemmArgs &g, float v, int64_t off, int col)
{
    if (g.bias) v += g.bias[col];
    if (g.pre) g.pre[off] = v;
    if (g.act == 1) v = gelu08(v);
    if (g.residual) v += g.residual[off];
    return v;
}

// One operand's share of a k-slab: R tile rows (rows of a, columns of b) by
// BK of k, loaded into registers by NT threads, split, and stored to LDS as
// three bf16 planes.  A thread holds G groups of 8 consecutive k of one row.
// KC: the operand is stored with k contiguous (a n x k, b m x k): a group is
// two 16-byte loads, and BK/8 neighbouring lanes share a row.  Otherwise (a
// k x n, b k x m) lanes run along the rows and a group is 8 dword loads, each
// 256 contiguous bytes per wave.  Either way a group's 8 elements are k
// neighbours, so its parts are stored as one 16-byte LDS write per plane.
// LDS: row r's 16-byte unit q of a plane sits at unit r * BK/8 + (q ^ swz(r)),
// with swz chosen so that 16 neighbouring rows of one q, which a quarter wave
// reads or writes together, fall on different banks.
template <int R, int BK, int NT, bool KC>
struct Operand {
    static constexpr int Q = BK / 8;             // 16-byte units per row and plane
    static constexpr int G = R * Q / NT;         // groups per thread
    static constexpr int kPlane = R * Q;         // units per plane
    static_assert(G >= 1 && G * NT == R * Q, "whole groups per thread");
    static_assert(Q == 2 || Q == 4, "swizzle below");
    static_assert(KC || R % 64 == 0, "a wave's lanes stay in one k row");

    const float *p[G];  // KC: this lane's group at the slab to load; else the wave's k row
    unsigned voff;      // !KC: this lane's byte offset from there
    int kq[G];          // the group's k offset within the slab
    float v[G][8];
    float f[G];         // kSplitScale with sign_of the group's row
    unsigned s[G][3][2];  // two split pairs: hi, mid, lo

    static __device__ __forceinline__ int unit(int r, int q)
    {
        return r * Q + (q ^ (Q == 2 ? (r >> 3) & 1 : (r >> 2) & 3));
    }
    static __device__ __forceinline__ int row_of(int tid, int g)
    {
        const int i = tid + NT * g;
        return KC ? i / Q : i % R;
    }
    static __device__ __forceinline__ int unit_of(int tid, int g)
    {
        const int i = tid + NT * g;
        return KC ? i % Q : i / R;
    }

    // base: the matrix; rows past `rows` re-read the last one (their results
    // are not stored).
    __device__ __forceinline__ void init(const float *base, int64_t ld, int row0, int rows, int kbeg, int tid)
    {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const int r = min(row_of(tid, g), rows - 1 - row0);
            int q = unit_of(tid, g);
            if (!KC) q = __builtin_amdgcn_readfirstlane(q);  // one k row per wave: scalar addresses
            kq[g] = 8 * q;
            f[g] = flip(kSplitScale, sign_of(row0 + row_of(tid, g)));
            p[g] = KC ? base + (int64_t)(row0 + r) * ld + kbeg + 8 * q : base + (int64_t)(kbeg + 8 * q) * ld + row0;
            if (!KC) voff = 4u * (unsigned)r;
        }
    }
    __device__ __forceinline__ float at(int g, int j, int64_t ld) const
    {
        if (KC) return p[g][j];
        return *(const float *)((const char *)(p[g] + j * ld) + voff);
    }
    // Loads group g of a whole slab.
    __device__ __forceinline__ void load_group(int64_t ld, int g)
    {
        typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
        if (KC) {
            const f32x4u x = *(const f32x4u *)p[g], y = *(const f32x4u *)(p[g] + 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[g][j] = x[j], v[g][4 + j] = y[j];
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[g][j] = at(g, j, ld);
        }
    }
    __device__ __forceinline__ void load(int64_t ld)
    {
#pragma unroll
        for (int g = 0; g < G; ++g) load_group(ld, g);
    }
    // Loads a partial slab of `len` k.
    __device__ __forceinline__ void load_part(int64_t ld, int len)
    {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int j = 0; j < 8; ++j) v[g][j] = kq[g] + j < len ? at(g, j, ld) : 0.0f;
    }
    // Moves on by k.
    __device__ __forceinline__ void advance(int64_t ld, int k)
    {
#pragma unroll
        for (int g = 0; g < G; ++g) p[g] += KC ? (int64_t)k : k * ld;
    }
    // Splits pair i (of 4) of group g; after every second one half a unit of
    // each plane is stored.
    __device__ __forceinline__ void split_store(int g, int i, u32x4 *__restrict__ lds, int tid)
    {
        split_pair(v[g][2 * i] * f[g], v[g][2 * i + 1] * f[g], s[g][0][i & 1], s[g][1][i & 1], s[g][2][i & 1]);
        if (i & 1) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            u32x2 *const to = (u32x2 *)lds + 2 * unit(row_of(tid, g), unit_of(tid, g)) + i / 2;
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) to[2 * pl * kPlane] = u32x2{s[g][pl][0], s[g][pl][1]};
        }
    }
    __device__ __forceinline__ void store(u32x4 *__restrict__ lds, int tid)
    {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
            for (int i = 0; i < 4; ++i) split_store(g, i, lds, tid);
    }
};

// A TM x TN block of out per workgroup of WR x WC waves, each 32*RB x 32*CB.
// What bounds it: the matrix cores, and at 4096^3 the power limit with them
// (78 % of cycles busy, at 1.64 GHz; the same launch on constant operands
// holds 2.28 GHz): 933 -> 584 us, 147 -> 235 TFLOP/s against the fp32
// instruction's kernel this replaced (573 to 627 us over cards).  Splitting costs 6.5 vector operations
// per element staged (2.6 per matrix instruction in the 256 x 256 tile, 4 are
// free beside one), so operands are split once, when they enter LDS, and not
// by each wave that reads them.
//   * k is walked in slabs of BK through two LDS buffers, one barrier per
//     slab: while slab s is multiplied, slab s+1 (in registers) is split and
//     stored to the other buffer and slab s+2 is requested.
//   * tiles are numbered so that the tiles one XCD runs (workgroup ids are
//     dealt to the 8 XCDs round-robin) are contiguous, and within that range
//     grouped 8 row tiles per b column panel for L2 reuse.
//   * split-K (g.part): blockIdx.z walks k in [z*kchunk, (z+1)*kchunk) and
//     stores its raw sums to part; gemm_splitk_reduce adds the splits in
//     order and applies the epilogue, so results do not depend on timing.
//   * a wave whose sums are not finite (split_bf16.h) computes its block
//     again from global memory with the fp32 instruction.
template <int TM, int TN, int WR, int WC, int BK, int PER_CU, bool TWO, bool TA, bool TB>
__global__ __launch_bounds__(64 * WR * WC, PER_CU) void gemm_split_kernel(GemmArgs g)
{
    constexpr int NT = 64 * WR * WC;
    constexpr int RB = TM / WR / 32, CB = TN / WC / 32;
    typedef Operand<TM, BK, NT, !TA> OA;
    typedef Operand<TN, BK, NT, TB> OB;
    
    __shared__ u32x4 As0[3 * OA::kPlane], As1[3 * OA::kPlane];
    __shared__ u32x4 Bs0[3 * OB::kPlane], Bs1[3 * OB::kPlane];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h32 = lane >> 5;
    const int l32 = lane & 31;
    const int wr = w / WC, wc = w % WC;

    const int ntiles = g.tiles_n * g.tiles_m;
    int tile = g.tile0 + blockIdx.x;
    if (ntiles % 8 == 0) tile = (tile % 8) * (ntiles / 8) + tile / 8;
    constexpr int GROUP = 8;
    const int per_group = GROUP * g.tiles_m;
    const int grp = tile / per_group;
    const int first = grp * GROUP;
    const int rows_in_grp = min(GROUP, g.tiles_n - first);
    const int in_grp = tile - grp * per_group;
    // Provably uniform, so that the operand addresses keep scalar parts.
    const int row0 = __builtin_amdgcn_readfirstlane((first + in_grp % rows_in_grp) * TM);
    const int col0 = __builtin_amdgcn_readfirstlane((in_grp / rows_in_grp) * TN);

    // Slab 0 takes what k leaves over, the others are whole, so that the loop
    // has no bounds on k and the short slab's guarded loads share the
    // prologue's wait.
    const KRange range = k_range(g.k, g.kchunk, blockIdx.z, BK);
    const int kbeg = range.beg, kend = range.end, nslab = range.slabs, first_k = range.first;
    const float *A = g.a + (int64_t)blockIdx.y * g.sa;
    const float *B = g.b + (int64_t)blockIdx.y * g.sb;

    // TWO: the five small products of a pair of operands are summed apart
    // from the large one, so that each sum is rounded less often.
    f32x16 acc[RB][CB], low[TWO ? RB : 1][TWO ? CB : 1];
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            acc[i][j] = zero16();
            if (TWO) low[i][j] = zero16();
        }

    OA oa;
    OB ob;
    const int arow = 32 * RB * wr + l32, bcol = 32 * CB * wc + l32;
    // Multiplies slab s (in as, bs) while slab s + 1 (in registers) is split
    // and stored to the other buffer and slab s + 2 is loaded.  Past the last
    // slab the last one is loaded again and not used: no branches here.
    // The products are cut into chunks of one b block; each chunk reads the
    // operands of the next one, the last, behind the barrier, those of the
    // next slab, and the chunks before it take an even share of the splitting.
    constexpr int KS = BK / 16, NC = KS * CB;
    static_assert(NC % 2 == 0, "b operands alternate between two register sets");
    constexpr int NU = 4 * (OA::G + OB::G);  // pairs to split
    constexpr int NS = (NC - 1) * RB * 6;    // products they are spread over
    Split8 af[2][RB], bf[2];
    auto read_a = [&](const u32x4 *__restrict__ as, int ks, Split8 (&f)[RB]) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int pl = 0; pl < 3; ++pl)
                f[rb].part[pl] = as[pl * OA::kPlane + 32 * rb * OA::Q + OA::unit(arow, 2 * ks + h32)];
    };
    auto read_b = [&](const u32x4 *__restrict__ bs, int ks, int cb, Split8 &f) {
#pragma unroll
        for (int pl = 0; pl < 3; ++pl)
            f.part[pl] = bs[pl * OB::kPlane + 32 * cb * OB::Q + OB::unit(bcol, 2 * ks + h32)];
    };
    auto step = [&](auto parity, auto only, int s, const u32x4 *__restrict__ as, const u32x4 *__restrict__ bs,
                    u32x4 *__restrict__ an, u32x4 *__restrict__ bn) {
        constexpr int PA = decltype(parity)::value;
        constexpr bool ONLY = decltype(only)::value;  // the one slab: nothing to stage
        const int k = s + 3 < nslab ? BK : 0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int ks = c / CB, cb = c % CB;
            if (c + 1 < NC) {
                if ((c + 1) % CB == 0) read_a(as, (c + 1) / CB, af[(PA + (c + 1) / CB) & 1]);
                read_b(bs, (c + 1) / CB, (c + 1) % CB, bf[(c + 1) & 1]);
            } else if (!ONLY) {
                __syncthreads();
                read_a(an, 0, af[(PA + KS) & 1]);
                read_b(bn, 0, 0, bf[0]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 6; ++t) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) {
                    const Split8 &x = af[(PA + ks) & 1][rb], &y = bf[c & 1];
                    if constexpr (TWO)
                        mfma_split_term(t, x, y, t == 5 ? acc[rb][cb] : low[rb][cb]);
                    else
                        mfma_split_term(t, x, y, acc[rb][cb]);
                    const int done = (c * 6 + t) * RB + rb;
#pragma unroll
                    for (int u = 0; u < NU; ++u) {
                        if (ONLY || done >= NS || u * NS / NU != done) continue;
                        if (u < 4 * OA::G) {
                            oa.split_store(u / 4, u % 4, an, tid);
                            if (u % 4 == 3) oa.load_group(g.lda, u / 4);
                        } else {
                            ob.split_store(u / 4 - OA::G, u % 4, bn, tid);
                            if (u % 4 == 3) ob.load_group(g.ldb, u / 4 - OA::G);
                        }
                    }
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        oa.advance(g.lda, k);
        ob.advance(g.ldb, k);
    };

    if (nslab > 0) {
        oa.init(A, g.lda, row0, g.n, kbeg, tid);
        ob.init(B, g.ldb, col0, g.m, kbeg, tid);
        if (first_k == BK) {
            oa.load(g.lda);
            ob.load(g.ldb);
        } else {
            oa.load_part(g.lda, first_k);
            ob.load_part(g.ldb, first_k);
        }
        if (nslab > 1) {
            oa.advance(g.lda, first_k);
            ob.advance(g.ldb, first_k);
        }
        oa.store(As0, tid);
        ob.store(Bs0, tid);
        if (nslab > 1) {
            oa.load(g.lda);
            ob.load(g.ldb);
            oa.advance(g.lda, nslab > 2 ? BK : 0);
            ob.advance(g.ldb, nslab > 2 ? BK : 0);
        }
        __syncthreads();
        read_a(As0, 0, af[0]);
        read_b(Bs0, 0, 0, bf[0]);
        // Two slabs per trip so that each buffer is a distinct LDS object:
        // the compiler then knows a store to one does not feed reads of the
        // other.
        typedef std::integral_constant<int, 0> zero;
        if (nslab == 1) step(zero{}, std::true_type{}, 0, As0, Bs0, As1, Bs1);
        for (int s = 0; nslab > 1;) {
            step(zero{}, std::false_type{}, s, As0, Bs0, As1, Bs1);
            if (++s == nslab) break;
            step(std::integral_constant<int, KS & 1>{}, std::false_type{}, s, As1, Bs1, As0, Bs0);
            if (++s == nslab) break;
        }
        __syncthreads();  // the operands read ahead, before the buffers are used again below
    }
    if (TWO) {
#pragma unroll
        for (int i = 0; i < RB; ++i)
#pragma unroll
            for (int j = 0; j < CB; ++j) acc[i][j] += low[i][j];
    }

    // Anything the split cannot carry (see split_bf16.h): do this wave's
    // block again with the fp32 instruction.
    float unscale = 1.0f / (kSplitScale * kSplitScale);
    if (nslab > 0) {
        float probe = 0.0f;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int i = 0; i < 16; ++i) probe = fmaf(acc[rb][cb][i], 0.0f, probe);
        if (__ballot(probe != 0.0f) != 0) {
            unscale = 1.0f;
            const float *ap[RB], *bp[CB];
            unsigned aneg[RB], bneg[CB];
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const int64_t r = min(row0 + arow + 32 * rb, g.n - 1);
                ap[rb] = A + (TA ? r : r * g.lda);
                aneg[rb] = sign_of(row0 + arow + 32 * rb);
            }
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const int64_t c = min(col0 + bcol + 32 * cb, g.m - 1);
                bp[cb] = B + (TB ? c * g.ldb : c);
                bneg[cb] = sign_of(col0 + bcol + 32 * cb);
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = zero16();
            for (int64_t k0 = kbeg; k0 < kend; k0 += 2) {
                const int64_t k = k0 + h32;
                float av[RB], bv[CB];
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
                    av[rb] = flip(k < kend ? ap[rb][TA ? k * g.lda : k] : 0.0f, aneg[rb]);
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
                    bv[cb] = flip(k < kend ? bp[cb][TB ? k : k * g.ldb] : 0.0f, bneg[cb]);
#pragma unroll
                for (int rb = 0; rb < RB; ++rb)
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = mfma_32x32x2(av[rb], bv[cb], acc[rb][cb]);
            }
        }
    }

    const int64_t zoff = g.part ? ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * g.sc
                                : (int64_t)blockIdx.y * g.sc;
    float *C = (g.part ? g.part : g.c) + zoff;
    const bool epi = !g.part && (g.bias || g.pre || g.act || g.residual);
    // Rows, columns and their signs derive from a lane index that the empty
    // asm makes opaque, so that the compiler does not compute them ahead of
    // the loop and spill.
    int el = lane;
    asm volatile("" : "+v"(el));
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const int col = col0 + 32 * (CB * wc + cb) + (el & 31);
        if (col >= g.m) continue;
        const float bias = epi && g.bias ? g.bias[col] : 0.0f;
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int row = row0 + 32 * (RB * wr + rb) + acc_row(i, el >> 5);
                if (row >= g.n) continue;
                const int64_t off = (int64_t)row * g.m + col;
                // Scale and sign come off by a multiplication, and a zero
                // sum stays +0.
                float v = fmaf(acc[rb][cb][i], flip(unscale, sign_of(row) ^ sign_of(col)), 0.0f);
                if (epi) {
                    // out = act(acc + bias) + residual, pre = acc + bias.
#pragma clang fp contract(off)
                    if (g.bias) v += bias;
                    if (g.pre) g.pre[zoff + off] = v;
                    if (g.act == 1) v = gelu08(v);
                    if (g.residual) v += g.residual[zoff + off];
                }
                C[off] = v;
            }
        }
    }
}

// out = epilogue(sum over z of part[z]), z in order; VEC: m % 4 == 0 and
// 16-byte aligned operands.
template <int V>
__global__ __launch_bounds__(256) void gemm_splitk_reduce(GemmArgs g, int ksplit, int64_t total)
{
    typedef float vec __attribute__((ext_vector_type(V)));
    const int64_t nv = total / V;
    for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < nv; q += (int64_t)gridDim.x * 256) {
        const int64_t off = V * q;
        vec s = *(const vec *)&g.part[off];
        for (int z = 1; z < ksplit; ++z) s += *(const vec *)&g.part[(int64_t)z * total + off];
        if (g.bias || g.pre || g.act || g.residual) {
            const int col = (int)(off % g.m);
#pragma unroll
            for (int c = 0; c < V; ++c) s[c] = epilogue(g, s[c], off + c, col + c);
        }
        *(vec *)&g.c[off] = s;
    }
}

// Tile-shape choice only: an unknown CU count falls back to MI355X's 256.
int num_cus()
{
    const int n = device_cu_count();
    return n > 0 ? n : 256;
}

template <int TM, int TN, int WR, int WC, int BK, int PER_CU, bool TWO, bool TA, bool TB>
void launch_tiles(GemmArgs &g, int batch, int ksplit)
{
    g.tiles_n = (int)ceil_div(g.n, TM);
    g.tiles_m = (int)ceil_div(g.m, TN);
    static_assert(kTilesPerLaunch % 8 == 0 && kTilesPerLaunch * 64 * WR * WC < int64_t(1) << 32, "threads of a grid in x");
    const int64_t tiles = (int64_t)g.tiles_n * g.tiles_m;
    for (int64_t t0 = 0; t0 < tiles; t0 += kTilesPerLaunch) {
        g.tile0 = (int)t0;
        hipLaunchKernelGGL((gemm_split_kernel<TM, TN, WR, WC, BK, PER_CU, TWO, TA, TB>),
                           dim3((unsigned)std::min(tiles - t0, kTilesPerLaunch), batch, ksplit), dim3(64 * WR * WC), 0, 0, g);
    }
}

template <bool TA, bool TB>
void launch_shape(GemmArgs &g, int batch, int ksplit, int shape)
{
    if (shape == 0)
        launch_tiles<256, 256, 4, 2, 16, 1, false, TA, TB>(g, batch, ksplit);
    else if (shape == 1)
        launch_tiles<128, 128, 4, 2, 32, 1, true, TA, TB>(g, batch, ksplit);
    else
        launch_tiles<64, 64, 2, 2, 32, 3, true, TA, TB>(g, batch, ksplit);
}

int gemm_launch(const float *a, const float *b, float *out, int batch, int n, int m, int k,
                const char *who, const float *bias = nullptr, const float *residual = nullptr,
                float *pre = nullptr, int act = 0, int ta = 0, int tb = 0)
{
    if (n < 0 || m < 0 || k < 0 || batch < 0) return record_error(EMBER_ERR_INVALID_ARGUMENT, who);
    if ((int64_t)n * m == 0 || batch == 0) return EMBER_OK;
    // k == 0: a and b are empty (null from alloc_memory(0)) and every output
    // is an empty sum, i.e. 0 before the epilogue, as in the reference's CPU
    // loop; the kernel never reads a or b then.
    if (!out || (k > 0 && (!a || !b))) return record_error(EMBER_ERR_INVALID_ARGUMENT, who);
    if (batch > 65535) return record_error(EMBER_ERR_UNSUPPORTED, who);
    GemmArgs g;
    g.a = a;
    g.b = b;
    g.c = out;
    g.n = n;
    g.m = m;
    g.k = k;
    g.lda = ta ? n : k;
    g.ldb = tb ? k : m;
    g.sa = (int64_t)n * k;
    g.sb = (int64_t)k * m;
    g.sc = (int64_t)n * m;
    g.kchunk = k;
    g.part = nullptr;
    g.bias = bias;
    g.residual = residual;
    g.pre = pre;
    g.act = act;

    const GemmChoice choice = choose_gemm(n, m, k, batch, num_cus());
    const int shape = choice.shape;
    int ksplit = choice.ksplit;
    const int64_t total = (int64_t)batch * n * m;
    if (ksplit > 1) {
        g.part = (float *)scratch(kScratchGemmSplit, (size_t)ksplit * total * sizeof(float), true);
        if (g.part)
            g.kchunk = (int)choice.kchunk;
        else
            ksplit = 1;  // no memory for the parts: one sum per element
    }
    if (ta)
        tb ? launch_shape<true, true>(g, batch, ksplit, shape) : launch_shape<true, false>(g, batch, ksplit, shape);
    else
        tb ? launch_shape<false, true>(g, batch, ksplit, shape) : launch_shape<false, false>(g, batch, ksplit, shape);
    if (!launch_ok(who)) return EMBER_ERR_DEVICE;
    if (ksplit > 1) {
        const bool vec = m % 4 == 0 && ((uintptr_t)out | (uintptr_t)pre | (uintptr_t)residual | (uintptr_t)bias) % 16 == 0;
        int64_t blocks = (total / (vec ? 4 : 1) + 255) / 256;
        if (blocks > 8 * num_cus()) blocks = 8 * num_cus();
        if (vec)
            hipLaunchKernelGGL(gemm_splitk_reduce<4>, dim3((unsigned)blocks), dim3(256), 0, 0, g, ksplit, total);
        else
            hipLaunchKernelGGL(gemm_splitk_reduce<1>, dim3((unsigned)blocks), dim3(256), 0, 0, g, ksplit, total);
        if (!launch_ok("gemm_splitk_reduce")) return EMBER_ERR_DEVICE;
    }
    return EMBER_OK;
}

}  // namespace
}  // namespace ember

extern "C" {

void matmul(const float *a, const float *b, float *out, int n, int m, int k)
{
    ember::gemm_launch(a, b, out, 1, n, m, k, "matmul");
}

void matmul_batched(const float *a, const float *b, float *out, int batch, int n, int m, int k)
{
    ember::gemm_launch(a, b, out, batch, n, m, k, "matmul_batched");
}

int linear_fwd(const float *a, const float *b, const float *bias, const float *residual,
               float *out, float *pre, int n, int m, int k, int act)
{
    if (act < 0 || act > 1) return ember::record_error(EMBER_ERR_INVALID_ARGUMENT, "linear_fwd");
    return ember::gemm_launch(a, b, out, 1, n, m, k, "linear_fwd", bias, residual, pre, act);
}

int gemm_ex(const float *a, const float *b, float *out, int batch, int n, int m, int k,
            int trans_a, int trans_b, const float *bias, const float *residual, float *pre, int act)
{
    if (act < 0 || act > 1 || (trans_a != 0 && trans_a != 1) || (trans_b != 0 && trans_b != 1))
        return ember::record_error(EMBER_ERR_INVALID_ARGUMENT, "gemm_ex");
    return ember::gemm_launch(a, b, out, batch, n, m, k, "gemm_ex", bias, residual, pre, act,
                              trans_a, trans_b);
}

}  // extern "C"
