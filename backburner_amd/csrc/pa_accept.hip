// pa_accept.hip - fused greedy acceptance of a draft block (the verify step's tail).
//
// No reference code exists for this in the checkout (the fork's LLAMA_BATCHED_ARGMAX, scripts/serve.sh:8-9, 281, and
// block verification, serve.sh:300-302). Semantics: a_i = argmax_j logits[i][j] with the lowest index on ties (numpy's
// rule, which also makes the first NaN win); k = the longest prefix with a_i == draft_i (i < n_rows-1); bonus = a_k.
//
// Layout: n_rows x splits workgroups; workgroup (row, sp) scans one or more segments of S values of its row (S and their count
// by the host's rule, accept_split),
// every thread issuing all its loads at once (S / 1024 16-byte loads, or S / 256 scalar ones when the vocab is not a
// multiple of 4); its lanes' best values become 64-bit keys (orderable value << 32 | ~index) so that one unsigned max picks the
// largest value and, among equal values, the lowest index. Each workgroup publishes its key with a write-through store and waits for
// it to complete before it counts itself done on a device-scope counter; the last one reads the keys with
// write-through loads, folds them per row and computes (k, bonus). No cache write-back or invalidate is needed: the
// keys never sit in an XCD's L2. The last workgroup resets the counter, so no memset is needed between calls.
#include "pa_attn.h"
#include "pa_common.h"

namespace pa_hip {

__device__ __forceinline__ unsigned long long accept_key(float x, uint32_t idx) {
    uint32_t u = __builtin_bit_cast(uint32_t, x);
    uint32_t k;
    if (x != x) k = 0xffffffffu;                 // NaN above everything (numpy.argmax returns the first NaN)
    else {
        if (u == 0x80000000u) u = 0u;            // -0 == +0
        k = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    }
    return ((unsigned long long) k << 32) | (unsigned long long) (0xffffffffu - idx);
}


__device__ __forceinline__ unsigned long long umax64(unsigned long long a, unsigned long long b) { return a > b ? a : b; }

// The best key of this wave's values of the segment [j0, j1) of row x (SEG / 256 values per thread: VEC consecutive ones 256 *
// VEC apart), every load issued at once. The thread's largest value first, then its first place where it is the wave's largest:
// about 3.5 vector instructions per value, where a 64-bit key each took fifteen (a workgroup is one wave per SIMD, so nothing
// hides them). A wave with a NaN anywhere goes over its values again by keys, which rank the first NaN above every value.
// us per call before and after: [17][151936] 9.05 / 7.5, [33][262144] 18.3 / 12.8, [5][50001] 9.3 / 6.85 (5.0 with the
// segments by accept_split).
template <int VEC, int SEG> __device__ __forceinline__ unsigned long long accept_best(const float * x, int64_t j0, int64_t j1, int t) {
    constexpr int NU = SEG / (256 * VEC);
    const uint32_t n = (uint32_t) (j1 - j0);                         // 1 .. SEG
    // buffer loads over the segment (values past it read 0 and become -inf in the one segment that has any): no branch per load
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc((void *) (x + j0), (short) 0, (int) (4 * n), 0x00020000);
    float v[NU][VEC];
    #pragma unroll
    for (int u = 0; u < NU; u++) {
        const uint32_t off = 4 * (VEC * t + 256 * VEC * u);
        if constexpr (VEC == 4) {
            const pa_f4 w = __builtin_bit_cast(pa_f4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0));
            v[u][0] = w[0]; v[u][1] = w[1]; v[u][2] = w[2]; v[u][3] = w[3];
        } else {
            v[u][0] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0));
        }
    }
    if (n < (uint32_t) SEG) {
        #pragma unroll
        for (int u = 0; u < NU; u++)
            #pragma unroll
            for (int e = 0; e < VEC; e++)
                if ((uint32_t) (VEC * t + 256 * VEC * u + e) >= n) v[u][e] = -INFINITY;
    }
    constexpr int NV = NU * VEC;
    float mx = -INFINITY;
    bool nan = false;
    #pragma unroll
    for (int i = 0; i < NV; i += 2) {
        const float a = v[i / VEC][i % VEC], b = v[(i + 1) / VEC][(i + 1) % VEC];
        mx = fmaxf(fmaxf(mx, a), b);
        nan |= __builtin_isunordered(a, b);
    }
    unsigned long long best = 0;
    if (!__any(nan)) {
        float wm = mx;
        #pragma unroll
        for (int off = 32; off > 0; off >>= 1) wm = fmaxf(wm, __shfl_xor(wm, off));
        if (mx == wm) {                                              // -0 == +0
            uint32_t at = 0;
            #pragma unroll
            for (int i = NV - 1; i >= 0; i--) at = v[i / VEC][i % VEC] == wm ? (uint32_t) (256 * VEC * (i / VEC) + i % VEC) : at;
            const uint32_t j = VEC * t + at;                         // past n: a thread without values, where all are -inf
            if (j < n) best = accept_key(wm, (uint32_t) j0 + j);
        }
    } else {
        #pragma unroll 1
        for (int u = 0; u < NU; u++) {
            const uint32_t j = VEC * t + 256 * VEC * u;
            #pragma unroll 1
            for (int e = 0; e < VEC; e++)
                if (j + e < n) best = umax64(best, accept_key(x[j0 + j + e], (uint32_t) j0 + j + e));
        }
    }
    return best;
}

// MANY: several segments per workgroup (the loop costs a call of one 0.5 us)
template <int SEG, bool MANY> __global__ __launch_bounds__(256) void accept_kernel(const AcceptArgs a) {
    __shared__ unsigned long long red[4];
    __shared__ bool last;
    const int row = blockIdx.x / a.splits, sp = blockIdx.x % a.splits;
    const float * x = a.logits + (size_t) row * (size_t) a.vocab;
    const int t = threadIdx.x;
    auto segment = [&](int64_t j0) {
        const int64_t j1 = min(a.vocab, j0 + SEG);
        return (a.vocab & 3) == 0 ? accept_best<4, SEG>(x, j0, j1, t) : accept_best<1, SEG>(x, j0, j1, t);
    };
    const int64_t s0 = (int64_t) sp * SEG * (MANY ? a.segs : 1);     // below vocab for every workgroup
    unsigned long long best = segment(s0);
    if constexpr (MANY)
        for (int c = 1; c < a.segs && s0 + (int64_t) c * SEG < a.vocab; c++) best = umax64(best, segment(s0 + (int64_t) c * SEG));
    for (int off = 32; off > 0; off >>= 1) best = umax64(best, __shfl_xor(best, off));
    if ((t & 63) == 0) red[t / 64] = best;
    __syncthreads();
    if (t == 0) {
        best = umax64(umax64(red[0], red[1]), umax64(red[2], red[3]));
        // write-through store (device scope), complete before the count below is made
        __hip_atomic_store(&a.part[row * a.splits + sp], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __builtin_amdgcn_s_waitcnt(0);
        const unsigned int done = __hip_atomic_fetch_add(a.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = done == (unsigned int) (a.n_rows * a.splits - 1);
    }
    __syncthreads();
    if (!last) return;
    // the last workgroup: every thread reads a share of all keys at once (write-through loads) and folds them into
    // its row's slot (LDS atomic max), then the accepted prefix
    __shared__ unsigned long long rk[64];
    __shared__ int32_t am[64];
    if (t < a.n_rows) rk[t] = 0;
    __syncthreads();
    const int nk = a.n_rows * a.splits;
    for (int i0 = 0; i0 < nk; i0 += 4 * 256) {
        unsigned long long k4[4];
        #pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + t + 256 * u;
            k4[u] = i < nk ? __hip_atomic_load(&a.part[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
        }
        #pragma unroll
        for (int u = 0; u < 4; u++) {
            const int i = i0 + t + 256 * u;
            if (i < nk) __hip_atomic_fetch_max(&rk[i / a.splits], k4[u], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    __syncthreads();
    if (t < a.n_rows) am[t] = (int32_t) (0xffffffffu - (uint32_t) (rk[t] & 0xffffffffu));
    __syncthreads();
    if (t == 0) {
        int k = 0;
        while (k < a.n_rows - 1 && am[k] == a.draft[k]) k++;
        a.out[0] = k;
        a.out[1] = am[k];
        __hip_atomic_store(a.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (t < a.n_rows) a.out[2 + t] = am[t];
}

hipError_t launch_accept(const AcceptArgs & a, hipStream_t st) {
    const dim3 grid((uint32_t) (a.n_rows * a.splits));
    if (a.seg == 4096 && a.segs == 1) hipLaunchKernelGGL((accept_kernel<4096, false>), grid, dim3(256), 0, st, a);
    else if (a.seg == 8192 && a.segs == 1) hipLaunchKernelGGL((accept_kernel<8192, false>), grid, dim3(256), 0, st, a);
    else if (a.seg == 16384 && a.segs == 1) hipLaunchKernelGGL((accept_kernel<16384, false>), grid, dim3(256), 0, st, a);
    else if (a.seg == 16384) hipLaunchKernelGGL((accept_kernel<16384, true>), grid, dim3(256), 0, st, a);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace pa_hip
