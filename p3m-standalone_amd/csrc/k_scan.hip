// Exclusive prefix sum of int counts, used by the counting sorts of the
// particle <-> mesh and real-space kernels.  Up to 4096 counts: one launch
// of one workgroup (runs of up to four counts per thread; longer serial runs
// lose to the launches below).  Beyond: per-block scans of 1024 elements, and
// the sums of the blocks before added.  Up to kDirectBlocks blocks each block
// adds those up itself; beyond, where that grows with the square of the
// blocks, their own prefix sums are made by a launch between the two.
#include <hip/hip_runtime.h>

#include "k_internal.hpp"

namespace {

constexpr int kBlock = 1024;

__device__ __forceinline__ int block_exclusive_scan(int v, int *sh, int &total) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    int x = v;
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off)
            x += y;
    }
    if (lane == 63)
        sh[wave] = x;
    __syncthreads();
    if (t < 64) {
        int w = (t < kBlock / 64) ? sh[t] : 0;
        for (int off = 1; off < 64; off <<= 1) {
            const int y = __shfl_up(w, off, 64);
            if (t >= off)
                w += y;
        }
        sh[64 + t] = w;
    }
    __syncthreads();
    total = sh[64 + kBlock / 64 - 1];
    const int before = (wave == 0) ? 0 : sh[64 + wave - 1];
    return before + x - v;
}

__global__ void __launch_bounds__(kBlock) k_scan_blocks(const int *__restrict__ in, int m,
                                                        int *__restrict__ out,
                                                        int *__restrict__ sums) {
    __shared__ int sh[128];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const int v = (i < m) ? in[i] : 0;
    int total;
    const int e = block_exclusive_scan(v, sh, total);
    if (i < m)
        out[i] = e;
    if (threadIdx.x == 0)
        sums[blockIdx.x] = total;
}

// Blocks up to which k_scan_add adds up the sums itself.  Whole scans, that
// way against a launch for the sums, us: 512 blocks 6.3 / 9.9, 1024 9.3 / 10.5,
// 2048 15.2 / 15.6, 4096 26.2 / 25.2, 16,384 113 / 85, 262,144 8336 / 1590.
constexpr int kDirectBlocks = 2048;

// single block: exclusive scan of nb block sums, 1024 a step with a carry
__global__ void __launch_bounds__(kBlock) k_scan_sums(int *__restrict__ sums, int nb) {
    __shared__ int sh[128];
    int carry = 0;
    for (int base = 0; base < nb; base += kBlock) {
        const int i = base + threadIdx.x;
        const int v = (i < nb) ? sums[i] : 0;
        int total;
        const int e = block_exclusive_scan(v, sh, total);
        if (i < nb)
            sums[i] = carry + e;
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0)
        sums[nb] = carry;
}

// the same from the sums' prefix sums
__global__ void __launch_bounds__(kBlock) k_scan_add_prefix(int *__restrict__ out, int m,
                                                            const int *__restrict__ sums, int nb) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < m)
        out[i] += sums[blockIdx.x];
    if (i == 0)
        out[m] = sums[nb];
}

// adds to each block's elements the sums of the blocks before it, which the
// block adds up itself (at most kDirectBlocks, two per thread)
__global__ void __launch_bounds__(kBlock) k_scan_add(int *__restrict__ out, int m,
                                                     const int *__restrict__ sums, int nb) {
    __shared__ int sh[kBlock / 64];
    int part = 0;
    for (int b = threadIdx.x; b < (int)blockIdx.x; b += kBlock)
        part += sums[b];
    for (int off = 32; off > 0; off >>= 1)
        part += __shfl_xor(part, off, 64);
    if ((threadIdx.x & 63) == 0)
        sh[threadIdx.x >> 6] = part;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; w++)
        before += sh[w];
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < m)
        out[i] += before;
    if ((int)blockIdx.x == nb - 1 && threadIdx.x == 0)
        out[m] = before + sums[nb - 1];
}

// one workgroup: thread t sums its run of ceil(m / 1024) consecutive counts,
// the run totals are scanned across the workgroup, and each thread writes its
// run's prefixes; total to out[m].  Each thread reads its run before writing
// it, so in and out may be the same array.
constexpr long kSmallScan = 4 * kBlock;

__global__ void __launch_bounds__(kBlock) k_scan_small(const int *in, int m, int *out) {
    __shared__ int sh[128];
    const int k = (m + kBlock - 1) / kBlock;
    const int b = min(m, (int)threadIdx.x * k), e = min(m, b + k);
    int sum = 0;
    for (int i = b; i < e; i++)
        sum += in[i];
    int total;
    int run = block_exclusive_scan(sum, sh, total);
    for (int i = b; i < e; i++) {
        const int v = in[i];
        out[i] = run;
        run += v;
    }
    if (threadIdx.x == 0)
        out[m] = total;
}

}  // namespace

size_t p3mk_scan_scratch_ints(long m) { return (size_t)((m + kBlock - 1) / kBlock) + 1; }

int p3mk_exclusive_scan(const int *count, long m, int *start, int *scratch, p3mk_queue *q) {
    hipStream_t s = p3mk_stream(q);
    const int nb = (int)((m + kBlock - 1) / kBlock);
    if (m <= 0)
        return p3mk_fill_zero(start, sizeof(int), q);
    if (m <= kSmallScan) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(kBlock), 0, s, count, (int)m, start);
        return p3mk_launch_check("scan");
    }
    hipLaunchKernelGGL(k_scan_blocks, dim3(nb), dim3(kBlock), 0, s, count, (int)m, start, scratch);
    P3MK_TRY(p3mk_launch_check("scan blocks"));
    if (nb > kDirectBlocks) {
        hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(kBlock), 0, s, scratch, nb);
        P3MK_TRY(p3mk_launch_check("scan sums"));
        hipLaunchKernelGGL(k_scan_add_prefix, dim3(nb), dim3(kBlock), 0, s, start, (int)m, scratch, nb);
        return p3mk_launch_check("scan add");
    }
    hipLaunchKernelGGL(k_scan_add, dim3(nb), dim3(kBlock), 0, s, start, (int)m, scratch, nb);
    return p3mk_launch_check("scan add");
}
