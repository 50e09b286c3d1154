// Stable order of up to some hundred thousand 63-bit keys in one to three launches, for the
// Morton orders of the j-set, of an i-set and of an irregular block.  The library's merge or
// radix sort takes 7 to 11 launches at these sizes, each shorter than the gap it costs.
//
//  * bsort_kernel: a work-group forms the keys of BRUN consecutive elements in LDS; every
//    thread counts the keys before its own among its wavefront's 64 (broadcast reads), then
//    searches the other seven sorted pieces side by side, and writes the sorted run.  A
//    bitonic network of 2048 keys took 25-34 us here (66 dependent LDS stages), counting
//    all 512 keys 10.5-13, this 7-11.
//  * bsort_rank_kernel: merges BWAY runs at a time: an element's place is its place in its
//    run plus, for every other run, the number of elements that come before it there, by
//    binary search, eight runs side by side so that their loads are in flight together (one
//    after the other 74 us at N = 50,021 where this takes 10.5; sixteen side by side or
//    three probes per step are no better: the cache reads of the searches bound it).
//
// Keys and order, N = 50,021: 55 us with the library's merge sort, 32 so.  N = 100,003: 50
// and 35.  Larger sets than BSORT_MAX would take a third merge and stay with the library.
#pragma once

#include "nb6_internal.h"

namespace nb6 {

constexpr int BRUN = 512;         // keys per first run = threads of bsort_kernel
constexpr int BWAY = 16;          // runs merged by one launch
constexpr int BSORT_MAX = BRUN * BWAY * BWAY;

// the low 21 bits of a with two zero bits between neighbours (one axis of a Morton key)
__device__ __forceinline__ unsigned long long spread21(unsigned long long a) {
    a &= 0x1fffffull;
    a = (a | (a << 32)) & 0x1f00000000ffffull;
    a = (a | (a << 16)) & 0x1f0000ff0000ffull;
    a = (a | (a << 8)) & 0x100f00f00f00f00full;
    a = (a | (a << 4)) & 0x10c30c30c30c30c3ull;
    a = (a | (a << 2)) & 0x1249249249249249ull;
    return a;
}

// a merge between: the keys go along
struct PutRun {
    unsigned long long *key;
    int *val;
    __device__ void put(int place, int e, unsigned long long k) const {
        key[place] = k;
        val[place] = e;
    }
};

// KEY: __device__ void begin(), run by every thread first (may synchronise the work-group),
//      then unsigned long long key(int element), below 2^63
// OUT: __device__ void put(int place, int element, unsigned long long key)
template <class KEY, class OUT>
__global__ __launch_bounds__(BRUN) void bsort_kernel(KEY kf, OUT out, int n) {
    __shared__ __attribute__((aligned(16))) unsigned long long sk[BRUN];
    const int t = threadIdx.x, lane = t & 63, e = blockIdx.x * BRUN + t;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    kf.begin();
    const unsigned long long k = e < n ? kf.key(e) : ~0ull >> 1;
    sk[t] = k;
    __syncthreads();
    // Equal keys of earlier elements come first: x <= k is x < k + 1 for them.  What stands
    // in for elements past n is the largest key and comes last.
    int r = 0;
    {
        const ulonglong2 *p = reinterpret_cast<const ulonglong2 *>(sk + w * 64);
#pragma unroll 16
        for (int q = 0; q < 32; q++) {
            const ulonglong2 x = p[q];
            r += x.x < k + (2 * q < lane);
            r += x.y < k + (2 * q + 1 < lane);
        }
    }
    __syncthreads();
    sk[w * 64 + r] = k;
    __syncthreads();
    constexpr int W = BRUN / 64;
    int pos[W];
#pragma unroll
    for (int b = 0; b < W; b++) pos[b] = 0;
#pragma unroll
    for (int s = 64; s > 0; s >>= 1) {
        unsigned long long x[W];
#pragma unroll
        for (int b = 0; b < W; b++) x[b] = sk[b * 64 + min(pos[b] + s, 64) - 1];
#pragma unroll
        for (int b = 0; b < W; b++)
            pos[b] = pos[b] + s <= 64 && x[b] < (b < w ? k + 1 : k) ? pos[b] + s : pos[b];
    }
#pragma unroll
    for (int b = 0; b < W; b++) r += b == w ? 0 : pos[b];
    if (e < n) out.put(blockIdx.x * BRUN + r, e, k);
}

// sorted runs of `run` keys (a multiple of 64; the last may be shorter) -> sorted runs of
// `run` * BWAY
template <class OUT>
__global__ __launch_bounds__(256) void bsort_rank_kernel(OUT out, int n, int run,
                                                         const unsigned long long *__restrict__ key,
                                                         const int *__restrict__ val) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e >= n) return;
    const int c = __builtin_amdgcn_readfirstlane(e / run), g = c / BWAY * BWAY;
    const unsigned long long k = key[e];
    const int v = val[e];
    int r = g * run + e - c * run;
    constexpr int U = 8;
#pragma unroll 1
    for (int b0 = g; b0 < g + BWAY && b0 * run < n; b0 += U) {
        const unsigned long long *p[U];
        int pos[U], len[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int b = b0 + u;
            len[u] = b == c ? 0 : max(0, min(run, n - b * run));
            p[u] = key + (len[u] > 0 ? b * run : 0);
            pos[u] = 0;
        }
        for (int s = run; s > 0; s >>= 1) {
            unsigned long long x[U];
#pragma unroll
            for (int u = 0; u < U; u++)
                x[u] = p[u][(unsigned)max(min(pos[u] + s, len[u]) - 1, 0)];
#pragma unroll
            for (int u = 0; u < U; u++)
                pos[u] += pos[u] + s <= len[u] && x[u] < (b0 + u < c ? k + 1 : k) ? s : 0;
        }
#pragma unroll
        for (int u = 0; u < U; u++) r += pos[u];
    }
    out.put(r, v, k);
}

// key, val: scratch of 2 n each
template <class KEY, class OUT>
void bsort(const KEY &kf, const OUT &out, int n, unsigned long long *key, int *val, hipStream_t s) {
    const dim3 ga((n + BRUN - 1) / BRUN), gr((n + 255) / 256);
    const PutRun a{key, val}, b{key + n, val + n};
    if (n <= BRUN) {
        hipLaunchKernelGGL((bsort_kernel<KEY, OUT>), ga, dim3(BRUN), 0, s, kf, out, n);
    } else {
        hipLaunchKernelGGL((bsort_kernel<KEY, PutRun>), ga, dim3(BRUN), 0, s, kf, a, n);
        if (n <= BRUN * BWAY) {
            hipLaunchKernelGGL(bsort_rank_kernel<OUT>, gr, dim3(256), 0, s, out, n, BRUN, a.key,
                               a.val);
        } else {
            hipLaunchKernelGGL(bsort_rank_kernel<PutRun>, gr, dim3(256), 0, s, b, n, BRUN, a.key,
                               a.val);
            hipLaunchKernelGGL(bsort_rank_kernel<OUT>, gr, dim3(256), 0, s, out, n, BRUN * BWAY,
                               b.key, b.val);
        }
    }
    NB6_HIP(hipGetLastError());
}

}  // namespace nb6
