// host_sum.h -- sums that a caller gets as one host float: the last workgroup
// to finish adds the others' partial sums and writes the result to pinned host
// memory, where the caller waits for it.  What this saves is latency: a kernel
// of one workgroup, a device-to-host copy and the runtime's wait.  Measured, a
// call that finds the device idle: sum of 1000 floats 20.5 -> 12.4 us, of 2^20
// 20.7 -> 14.9.  (Waiting with hipStreamSynchronize instead of polling is
// slower than the copy: the step of a small classifier 107 against 87 us.)
#pragma once

#include "common.h"

namespace ember {
namespace {

// Workgroups of the running kernel that have stored their partial sum; 0
// between kernels (the last one resets it), and kernels on the null stream run
// one after another.  Many workgroups count in 16 groups, a cache line each,
// whose last ones count in the 17th: additions to one address take 10 ns each
// (cross-entropy of 8192 x 128 logits, 1024 workgroups: 28 us with one counter,
// 18 with the groups).
constexpr unsigned kSumGroups = 16, kSumLine = 32;
__device__ unsigned sums_stored[(kSumGroups + 1) * kSumLine];

// Counts one of `of` in counter i; true, and the counter 0 again, for the last.
__device__ __forceinline__ bool count_sum(unsigned i, unsigned of)
{
    unsigned *c = &sums_stored[i * kSumLine];
    if (__hip_atomic_fetch_add(c, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != of - 1) return false;
    __hip_atomic_store(c, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Called by all 256 threads of every workgroup.  mine: the workgroup's sum, in
// thread 0.  *out = 2^32 + the bits of the sum of partial[0 .. gridDim.x) in a fixed order: thread
// t adds every 256th from t, then a tree.
//
// The partial sums and the counter are device-scope relaxed atomics, which
// bypass this XCD's L2, and a workgroup counts itself after its store has been
// acknowledged (vmcnt 0).  A release fence would also write back the L2 with
// everything that the kernel has stored, once per workgroup.
__device__ __forceinline__ void finish_sum(double mine, double *partial, uint64_t *out)
{
    __shared__ double red[256];
    __shared__ int last;
    if (threadIdx.x == 0) {
        __hip_atomic_store(&partial[blockIdx.x], mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));  // vmcnt(0)
        asm volatile("" ::: "memory");
        const unsigned n = gridDim.x, g = blockIdx.x % kSumGroups;
        if (n <= 4 * kSumGroups)
            last = count_sum(kSumGroups, n);
        else
            last = count_sum(g, (n - g + kSumGroups - 1) / kSumGroups) && count_sum(kSumGroups, kSumGroups);
    }
    __syncthreads();
    if (!last) return;
    double s = 0.0;
    for (unsigned i = threadIdx.x; i < gridDim.x; i += 256)
        s += __hip_atomic_load(&partial[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = 128; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const uint64_t v = 1ull << 32 | __builtin_bit_cast(unsigned, (float)red[0]);
        __hip_atomic_store(out, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

}  // namespace

// Eight bytes of pinned host memory for a call's result, or, where there are
// none or the kernel also stores tensors, `res` in device memory.  The slot is
// written while the kernel's other stores may still be in flight or in an L2,
// and a caller may read its tensors on a stream of its own after the call:
// such calls wait for the whole kernel with the copy (cross-entropy 8192 x 1000
// 46 us; 37 without the wait, 58 polling and then hipStreamQuery until done).
class HostSum {
public:
    HostSum(uint64_t *res, bool stores_tensors) : slot_(stores_tensors ? nullptr : host_slot()), res_(res)
    {
        if (slot_) __atomic_store_n(slot_, 0, __ATOMIC_RELAXED);
    }
    ~HostSum()
    {
        if (slot_) release_host_slot(slot_);
    }
    HostSum(const HostSum &) = delete;
    HostSum &operator=(const HostSum &) = delete;
    uint64_t *out() const { return slot_ ? slot_ : res_; }
    // Waits for the kernel that writes the sum, and so for what was enqueued
    // before it, and reads the sum: polls the slot, and now and then asks the
    // runtime whether the stream still runs.
    int read(float *value, const char *who) const
    {
        uint64_t v = 0;
        if (!slot_) {
            if (!hip_ok(hipMemcpy(&v, res_, sizeof v, hipMemcpyDeviceToHost), who)) return EMBER_ERR_DEVICE;
        } else {
            for (unsigned polls = 1; (v = __atomic_load_n(slot_, __ATOMIC_ACQUIRE)) == 0; ++polls) {
                __builtin_ia32_pause();
                if (polls % 4096) continue;
                const hipError_t st = hipStreamQuery(nullptr);
                if (st == hipErrorNotReady) continue;
                if (!hip_ok(st, who)) return EMBER_ERR_DEVICE;
                v = __atomic_load_n(slot_, __ATOMIC_ACQUIRE);
                break;
            }
        }
        if (v >> 32 != 1) return record_error(EMBER_ERR_DEVICE, who);
        const unsigned bits = (unsigned)v;
        *value = __builtin_bit_cast(float, bits);
        return EMBER_OK;
    }

private:
    uint64_t *slot_, *res_;
};

}  // namespace ember
