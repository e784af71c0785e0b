// softmax.hip -- softmax along one axis in one launch, and the softmax
// cross-entropy loss (below).
//
// Ember's softmax(a, axis) is exp(a - amax(a, axis)) / sum(exp(...), axis)
// (ember/tensor/tensor.py:430-437), run by the reference as five launches
// (max_axis, sub_broadcasted, exponent_tensor, sum_axis, truediv_broadcasted)
// and four intermediate tensors.  Here each line along the axis is read once
// or three times and written once:
//   m = max over the line (fmaxf: any order gives the same value)
//   e = expf(x - m),  s = sum of e,  out = e * (1 / s)  (within 2 ulp of e / s)
// with the composed path's fp32 operations per element, except that the
// division is a multiply by the line's reciprocal.  The order of the sum also
// differs where lines are long: the last axis is reduced
// across a wave or a workgroup in a fixed tree order (deterministic);
// other axes are summed in index order as sum_axis does.
//   * last axis, L <= 2048: a wave per row, the row held in registers;
//   * last axis, L > 2048: a workgroup per row, three passes over the row
//     (the re-reads hit L2), float4 when rows are 16-byte aligned;
//   * other axes: a thread per (outer, inner) line, three passes, loads
//     coalesced across inner.
// HBM-bound: 8 bytes per element (read + write) on the first two paths.
#include <math.h>

#include <algorithm>

#include "common.h"
#include "host_sum.h"

namespace ember {
namespace {

__device__ __forceinline__ float wave_max(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ __forceinline__ float wave_sum(float v)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

template <int NV>
__global__ __launch_bounds__(256) void softmax_rows_wave(const float *__restrict__ a,
                                                         float *__restrict__ out, int rows, int L)
{
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row >= rows) return;
    const float *p = a + (int64_t)row * L;
    float *q = out + (int64_t)row * L;
    float v[NV];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = 64 * j + lane;
        v[j] = c < L ? p[c] : -INFINITY;
        m = fmaxf(m, v[j]);
    }
    m = wave_max(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = 64 * j + lane;
        const float e = c < L ? expf(v[j] - m) : 0.0f;
        v[j] = e;
        s += e;
    }
    // One correctly rounded reciprocal per row and a multiply per element
    // (within 2 ulp of the quotient) instead of an IEEE division per element.
    const float inv = 1.0f / wave_sum(s);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = 64 * j + lane;
        if (c < L) q[c] = v[j] * inv;
    }
}

// Block-wide reduction of one value per thread (256 threads); every thread
// gets the result.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float *red)
{
    v = MAX ? wave_max(v) : wave_sum(v);
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) red[w] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for (int i = 1; i < 4; ++i) r = MAX ? fmaxf(r, red[i]) : r + red[i];
    __syncthreads();
    return r;
}

template <bool VEC4>
__global__ __launch_bounds__(256) void softmax_rows_block(const float *__restrict__ a,
                                                          float *__restrict__ out, int L)
{
    __shared__ float red[4];
    const int t = threadIdx.x;
    const float *p = a + (int64_t)blockIdx.x * L;
    float *q = out + (int64_t)blockIdx.x * L;
    float m = -INFINITY;
    if (VEC4) {
        for (int c = 4 * t; c < L; c += 1024) {
            const float4 x = *(const float4 *)&p[c];
            m = fmaxf(m, fmaxf(fmaxf(x.x, x.y), fmaxf(x.z, x.w)));
        }
    } else {
        for (int c = t; c < L; c += 256) m = fmaxf(m, p[c]);
    }
    m = block_reduce<true>(m, red);
    float s = 0.0f;
    if (VEC4) {
        for (int c = 4 * t; c < L; c += 1024) {
            const float4 x = *(const float4 *)&p[c];
            s += expf(x.x - m);
            s += expf(x.y - m);
            s += expf(x.z - m);
            s += expf(x.w - m);
        }
    } else {
        for (int c = t; c < L; c += 256) s += expf(p[c] - m);
    }
    const float inv = 1.0f / block_reduce<false>(s, red);
    if (VEC4) {
        for (int c = 4 * t; c < L; c += 1024) {
            const float4 x = *(const float4 *)&p[c];
            float4 y;
            y.x = expf(x.x - m) * inv;
            y.y = expf(x.y - m) * inv;
            y.z = expf(x.z - m) * inv;
            y.w = expf(x.w - m) * inv;
            *(float4 *)&q[c] = y;
        }
    } else {
        for (int c = t; c < L; c += 256) q[c] = expf(p[c] - m) * inv;
    }
}

__global__ __launch_bounds__(256) void softmax_lines(const float *__restrict__ a,
                                                     float *__restrict__ out, int outer, int inner,
                                                     int L)
{
    const int64_t total = (int64_t)outer * inner;
    for (int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * 256) {
        const int64_t o = idx / inner, i = idx - o * inner;
        const int64_t base = o * L * inner + i;
        float m = a[base];
        for (int r = 1; r < L; ++r) m = fmaxf(m, a[base + (int64_t)r * inner]);
        float s = 0.0f;
        for (int r = 0; r < L; ++r) s += expf(a[base + (int64_t)r * inner] - m);
        // An IEEE division per element, as Ember's composition (a strided
        // line is latency-bound, so the reciprocal would save nothing here).
        for (int r = 0; r < L; ++r) {
            const int64_t off = base + (int64_t)r * inner;
            out[off] = expf(a[off] - m) / s;
        }
    }
}

template <int NV>
void launch_wave(const float *a, float *out, int rows, int L)
{
    hipLaunchKernelGGL(softmax_rows_wave<NV>, dim3((rows + 3) / 4), dim3(256), 0, 0, a, out, rows, L);
}

// ---- softmax cross-entropy ----
// Ember's CrossEntropyLoss (ember/loss/losses.py:29-56) composes nine
// element-wise, reduction and broadcast launches, each a pass over the logits'
// size; one pass here.  Per row: m = max, e = expf(x - m), s = sum of e, p = e
// * (1 / s) (nearer to the exact value than the composition's expf(logp),
// whose exponent has been rounded), grad = (p - t) / n, and the sum of t * logp
// with logp = (x - m) - logf(s), rounded as the composition's products and
// added in double.
//
// HBM-bound where rows are long: 16 bytes per element, two arrays read and two
// written.  A row is held in the registers of 16, 32 or 64 lanes (16 floats
// per lane at 1000 classes); a wave loads its next row's logits and targets
// before it works on the one it has, as the vector work (13 us of the 41 at
// 8192 x 1000 without that) otherwise has no loads beside it.  Rows longer
// than 4096 (1024 where they are not 16-byte aligned, one float per load) take
// a workgroup each and three passes, of which the second and third hit the
// caches.
// Measured, value and gradient with the sum read back, composed and here: 8192
// x 1000 179 and 45 us (the kernel 40 us without the next row's loads and with
// a second expf and a division per element, 30 with them: 4.4 TB/s).
constexpr int kLossBlocks = 1024;  // 4 workgroups of 4 waves per CU

template <int TPR>
__device__ __forceinline__ float group_max(float v)
{
#pragma unroll
    for (int o = TPR / 2; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
    return v;
}

template <int TPR>
__device__ __forceinline__ float group_sum(float v)
{
#pragma unroll
    for (int o = TPR / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

struct LossArgs {
    const float *x, *t;
    float *probs, *grad;
    double *partial;  // one per workgroup
    uint64_t *total;
    int rows, L;
    float n;
};

// a / n with r = 1 / n: the quotient corrected by its exact remainder
// (Markstein's method), and the special cases of a division; n within
// 2^-100 .. 2^100, so that r is an ordinary number.
__device__ __forceinline__ float divide_by(float a, float n, float r)
{
    const float q = a * r;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, n, a), r, q), n, a);
}

// The element's outputs; returns t * logp, rounded as the composition's product.
__device__ __forceinline__ float loss_element(float shifted, float logs, float e, float inv, float t, float n, float r,
                                              float &p, float &g)
{
#pragma clang fp contract(off)
    p = e * inv;
    g = divide_by(p - t, n, r);
    return t * (shifted - logs);
}

__device__ __forceinline__ void store_sum(double sum, const LossArgs &a)
{
    __shared__ double waves[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if ((threadIdx.x & 63) == 0) waves[threadIdx.x >> 6] = sum;
    __syncthreads();
    finish_sum((waves[0] + waves[1]) + (waves[2] + waves[3]), a.partial, a.total);
}

// TPR lanes per row, NV pieces of W neighbouring floats per lane (TPR * NV * W >= L).
template <int TPR, int NV, int W>
__global__ __launch_bounds__(256) void cross_entropy_rows(LossArgs a)
{
    typedef float piece __attribute__((ext_vector_type(W)));
    constexpr int RPB = 256 / TPR;
    const int sub = threadIdx.x % TPR;
    const float r = 1.0f / a.n;
    double sum = 0.0;
    piece xn[NV], tn[NV];  // the next row's
    auto load = [&](int64_t row) {  // up to a stride past the last row, which may be 2^31 - 1
        const int64_t base = row * a.L;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = W * (TPR * j + sub);
            if (row < a.rows && c < a.L) {
                xn[j] = *(const piece *)(a.x + base + c);
                tn[j] = *(const piece *)(a.t + base + c);
            } else {
                xn[j] = piece(-INFINITY);  // exp: 0
                tn[j] = piece(0.0f);
            }
        }
    };
    const int stride = gridDim.x * RPB;
    int64_t row = blockIdx.x * RPB + threadIdx.x / TPR;
    load(row);
    for (; row < a.rows; row += stride) {
        const int64_t base = row * a.L;
        piece x[NV], t[NV], e[NV];
#pragma unroll
        for (int j = 0; j < NV; ++j) x[j] = xn[j], t[j] = tn[j];
        load(row + stride);
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int i = 0; i < W; ++i) m = fmaxf(m, x[j][i]);
        m = group_max<TPR>(m);
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j)
#pragma unroll
            for (int i = 0; i < W; ++i) {
                x[j][i] -= m;
                e[j][i] = expf(x[j][i]);
                s += W * (TPR * j + sub) < a.L ? e[j][i] : 0.0f;  // a row of -inf: NaN from its own elements only
            }
        s = group_sum<TPR>(s);
        const float logs = logf(s), inv = 1.0f / s;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = W * (TPR * j + sub);
            if (c < a.L) {
                piece p, g;
#pragma unroll
                for (int i = 0; i < W; ++i) {
                    float pe, ge;
                    sum += (double)loss_element(x[j][i], logs, e[j][i], inv, t[j][i], a.n, r, pe, ge);
                    p[i] = pe, g[i] = ge;
                }
                *(piece *)(a.probs + base + c) = p;
                *(piece *)(a.grad + base + c) = g;
            }
        }
    }
    store_sum(sum, a);
}

__global__ __launch_bounds__(256) void cross_entropy_long(LossArgs a)
{
    __shared__ float red[4];
    const float r = 1.0f / a.n;
    double sum = 0.0;
    for (int64_t row = blockIdx.x; row < a.rows; row += gridDim.x) {
        const int64_t base = row * a.L;
        const float *x = a.x + base, *t = a.t + base;
        float m = -INFINITY, s = 0.0f;
        for (int c = threadIdx.x; c < a.L; c += 256) m = fmaxf(m, x[c]);
        m = block_reduce<true>(m, red);
        for (int c = threadIdx.x; c < a.L; c += 256) s += expf(x[c] - m);
        s = block_reduce<false>(s, red);
        const float logs = logf(s), inv = 1.0f / s;
        for (int c = threadIdx.x; c < a.L; c += 256) {
            float p, g;
            sum += (double)loss_element(x[c] - m, logs, expf(x[c] - m), inv, t[c], a.n, r, p, g);
            a.probs[base + c] = p;
            a.grad[base + c] = g;
        }
    }
    store_sum(sum, a);
}

template <int TPR, int NV, int W>
void launch_loss(const LossArgs &a, int blocks)
{
    hipLaunchKernelGGL((cross_entropy_rows<TPR, NV, W>), dim3(blocks), dim3(256), 0, 0, a);
}

}  // namespace
}  // namespace ember

extern "C" int softmax_axis(const float *a, float *out, int outer, int inner, int axis_dim)
{
    using namespace ember;
    if (outer < 0 || inner < 0 || axis_dim < 0) return record_error(EMBER_ERR_INVALID_ARGUMENT, "softmax_axis");
    if ((int64_t)outer * inner * axis_dim == 0) return EMBER_OK;
    if (!a || !out) return record_error(EMBER_ERR_INVALID_ARGUMENT, "softmax_axis");
    if (inner == 1) {
        const int L = axis_dim, rows = outer;
        if (L <= 64) launch_wave<1>(a, out, rows, L);
        else if (L <= 128) launch_wave<2>(a, out, rows, L);
        else if (L <= 256) launch_wave<4>(a, out, rows, L);
        else if (L <= 512) launch_wave<8>(a, out, rows, L);
        else if (L <= 1024) launch_wave<16>(a, out, rows, L);
        else if (L <= 2048) launch_wave<32>(a, out, rows, L);
        else if (L % 4 == 0 && (((uintptr_t)a | (uintptr_t)out) % 16) == 0)
            hipLaunchKernelGGL(softmax_rows_block<true>, dim3(rows), dim3(256), 0, 0, a, out, L);
        else
            hipLaunchKernelGGL(softmax_rows_block<false>, dim3(rows), dim3(256), 0, 0, a, out, L);
    } else {
        const int64_t total = (int64_t)outer * inner;
        int64_t blocks = (total + 255) / 256;
        if (blocks > 65536) blocks = 65536;
        hipLaunchKernelGGL(softmax_lines, dim3((unsigned)blocks), dim3(256), 0, 0, a, out, outer,
                           inner, axis_dim);
    }
    return launch_ok("softmax_axis") ? EMBER_OK : EMBER_ERR_DEVICE;
}

extern "C" int cross_entropy_loss(const float *logits, const float *target, float *probs, float *grad, int rows,
                                  int classes, float n, float *total)
{
    using namespace ember;
    if (rows < 0 || classes < 0 || !total) return record_error(EMBER_ERR_INVALID_ARGUMENT, "cross_entropy_loss");
    *total = 0.0f;
    if (rows == 0 || classes == 0) return EMBER_OK;
    if (!logits || !target || !probs || !grad) return record_error(EMBER_ERR_INVALID_ARGUMENT, "cross_entropy_loss");
    const int L = classes;
    const bool quads = L % 4 == 0 &&
                       (((uintptr_t)logits | (uintptr_t)target | (uintptr_t)probs | (uintptr_t)grad) & 15) == 0;
    const bool by_block = L > (quads ? 4096 : 1024);
    const int per_block = by_block ? 1 : L <= 16 ? 16 : L <= 32 ? 8 : 4;  // rows
    const int blocks = (int)std::min<int64_t>(((int64_t)rows + per_block - 1) / per_block, kLossBlocks);
    char *ws = (char *)scratch(kScratchSum, (size_t)blocks * sizeof(double) + 16);
    if (!ws) return EMBER_ERR_OUT_OF_MEMORY;
    const HostSum result((uint64_t *)(ws + (size_t)blocks * sizeof(double)), true);
    const bool ordinary = fabsf(n) >= 0x1p-100f && fabsf(n) <= 0x1p100f;  // divide_by
    const LossArgs a = {logits, target, probs, grad, (double *)ws, result.out(), rows, L, ordinary ? n : 1.0f};
    if (L <= 16) launch_loss<16, 1, 1>(a, blocks);
    else if (L <= 32) launch_loss<32, 1, 1>(a, blocks);
    else if (by_block) hipLaunchKernelGGL(cross_entropy_long, dim3(blocks), dim3(256), 0, 0, a);
    else if (quads) {
        if (L <= 256) launch_loss<64, 1, 4>(a, blocks);
        else if (L <= 512) launch_loss<64, 2, 4>(a, blocks);
        else if (L <= 1024) launch_loss<64, 4, 4>(a, blocks);
        else if (L <= 2048) launch_loss<64, 8, 4>(a, blocks);
        else launch_loss<64, 16, 4>(a, blocks);
    } else {
        if (L <= 64) launch_loss<64, 1, 1>(a, blocks);
        else if (L <= 128) launch_loss<64, 2, 1>(a, blocks);
        else if (L <= 256) launch_loss<64, 4, 1>(a, blocks);
        else if (L <= 512) launch_loss<64, 8, 1>(a, blocks);
        else launch_loss<64, 16, 1>(a, blocks);
    }
    if (!launch_ok("cross_entropy_loss")) return EMBER_ERR_DEVICE;
    const int64_t size = (int64_t)rows * L, part = int64_t(1) << 30;
    for (int64_t i = 0; !ordinary && i < size; i += part)
        truediv_scalar(grad + i, n, grad + i, (int)std::min(part, size - i));
    return result.read(total, "cross_entropy_loss");
}
