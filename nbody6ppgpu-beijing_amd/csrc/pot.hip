// All-pairs potential for gfx950.
//
// Semantics follow gpupot (gpupot.gpu.cu:32-57, pot.avx.cpp:112-136):
//   phi_i = sum_{j, r_ij^2 > 0} m_j / r_ij   (positive; the self pair and any
//   coincident particle are skipped).
//
// Method (own): grid (i-blocks, j-chunks), 256 threads, two i-particles per lane (one in
// small calls).  j-tiles of 256 particles are staged in LDS as FP64 positions + FP32 mass.  The
// separation is formed in FP64 and rounded once to FP32 (v_add_f64 + v_cvt), so
// the relative error of dx is one FP32 rounding even for the tightest binaries
// (the reference reaches the same with float-float positions, cuda_share.h:45-54).
// r^2, v_rsq_f32 and m*rinv run in FP32 and are summed per tile with Kahan
// compensation (a tight binary can dominate a tile); tile sums are flushed into
// FP64, chunk partials are summed in FP64 by a second kernel.
#include "nb6_internal.h"

#include <algorithm>
#include <cmath>

namespace nb6 {

namespace {

constexpr int PT_THREADS = 256;
constexpr int PT_TJ = 256;   // (a thread per record of a tile)

struct PotParams {
    const double *__restrict__ xs;   // SoA [4][stride] x, y, z, m
    int n, stride;
    int i0, ni;
    int chunk_len;
    double *__restrict__ part;       // [nchunk][ni]
};

// One LDS tile against this lane's i, compensated (Kahan) FP32 sums from zero: one close
// pair (a tight binary) can dominate the tile sum.  CHECK: pairs with r2 = 0 (the particle
// itself, coincident ones) and with values that are not finite add nothing.  Four pairs at a
// time, their reciprocal square roots together and at raised priority: without it the two
// wavefronts that a SIMD issues side by side fall into step at these slow instructions and
// take turns afterwards (n = 262,144: 20.7 -> 20.2 ms; the same order without priority 21.2).
template <int IPL, bool CHECK>
__device__ __forceinline__ void pot_tile(const double4 *sJ, const double *xi, const double *yi,
                                         const double *zi, float *a32, float *c32) {
#pragma unroll
    for (int k = 0; k < IPL; k++) a32[k] = c32[k] = 0.f;
    constexpr int U = 4 / IPL;
#pragma unroll 2
    for (int j0 = 0; j0 < PT_TJ; j0 += U) {
        float mj[U], r2[U][IPL], ri[U][IPL];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const double4 b = sJ[j0 + u];
            mj[u] = __int_as_float(__double2loint(b.w));   // (stored as FP32)
#pragma unroll
            for (int k = 0; k < IPL; k++) {
                const float dx = (float)(b.x - xi[k]);
                const float dy = (float)(b.y - yi[k]);
                const float dz = (float)(b.z - zi[k]);
                r2[u][k] = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            }
        }
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 0; k < IPL; k++) ri[u][k] = __builtin_amdgcn_rsqf(r2[u][k]);
        __builtin_amdgcn_s_setprio(0);
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int k = 0; k < IPL; k++) {
                float q = ri[u][k];
                if (CHECK) q = r2[u][k] > 0.f ? q : 0.f;
                const float y = fmaf(mj[u], q, -c32[k]);
                const float t = a32[k] + y;
                c32[k] = (t - a32[k]) - y;
                a32[k] = t;
            }
    }
}

// Bound by VALU issue: per pair 3 FP64 subtractions and 3 conversions (half the FP32 rate),
// a reciprocal square root (a quarter) and 7 FP32 operations.  A pair with r2 = 0 would need a
// compare and a select in every pair (1.7 of 14.7 CU cycles); instead the tiles that hold the
// work-group's own particles are taken with the check, and elsewhere such a pair makes the
// reciprocal square root, and with it the tile's sum, infinite or NaN, and a wavefront that
// finds such a sum takes the tile again with the check (coincident particles, values that
// are not finite).  n = 262,144: 25.3 -> 22.7 ms, 21.2 with the launch shape of pot_launch.
template <int IPL>
__global__ __launch_bounds__(PT_THREADS) void pot_tile_kernel(PotParams p) {
    __shared__ double4 sJ[PT_TJ];
    const int tid = threadIdx.x;
    const int chunk = blockIdx.y;
    const int kbase = blockIdx.x * (PT_THREADS * IPL);
    const int st = p.stride;

    double xi[IPL], yi[IPL], zi[IPL];
    double a64[IPL];
#pragma unroll
    for (int k = 0; k < IPL; k++) {
        const int kk = kbase + k * PT_THREADS + tid;
        const int i = p.i0 + (kk < p.ni ? kk : 0);
        xi[k] = p.xs[0 * st + i]; yi[k] = p.xs[1 * st + i]; zi[k] = p.xs[2 * st + i];
        a64[k] = 0.0;
    }
    const int j0 = chunk * p.chunk_len;
    const int j1 = min(j0 + p.chunk_len, p.n);
    for (int jt = j0; jt < j1; jt += PT_TJ) {
        const int j = jt + tid;
        sJ[tid] = j < j1 ? make_double4(p.xs[0 * st + j], p.xs[1 * st + j], p.xs[2 * st + j],
                                        __hiloint2double(0, __float_as_int((float)p.xs[3 * st + j])))
                         : make_double4(1.0e17, 0.0, 0.0, 0.0);
        __syncthreads();
        float a32[IPL], c32[IPL];
        // (the tiles of its own particles need the check for certain)
        const int ib = p.i0 + kbase;
        bool fine = jt >= ib + PT_THREADS * IPL || jt + PT_TJ <= ib;
        if (fine) pot_tile<IPL, false>(sJ, xi, yi, zi, a32, c32);
#pragma unroll
        for (int k = 0; k < IPL; k++)
            fine = fine && fabsf(a32[k]) < INFINITY && c32[k] == c32[k];
        if (__ballot(!fine)) pot_tile<IPL, true>(sJ, xi, yi, zi, a32, c32);
#pragma unroll
        for (int k = 0; k < IPL; k++) a64[k] += (double)a32[k] - (double)c32[k];
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < IPL; k++) {
        const int kk = kbase + k * PT_THREADS + tid;
        if (kk < p.ni) p.part[(size_t)chunk * p.ni + kk] = a64[k];
    }
}

__global__ __launch_bounds__(64) void pot_sum_kernel(const double *__restrict__ part, int ni,
                                                     int nchunk, double *__restrict__ out) {
    const int k = blockIdx.x * 64 + threadIdx.x;
    if (k >= ni) return;
    double s = 0.0;
#pragma unroll 8
    for (int c = 0; c < nchunk; c++) s += part[(size_t)c * ni + k];
    out[k] = s;
}

DBuf g_part;

}  // namespace

int pot_launch(int n, int n_stride, const double *d_x, int i0, int ni, double *d_pot,
               hipStream_t s) {
    if (ni <= 0) return OK;
    if (n <= 0 || i0 < 0 || i0 + ni > n) {
        set_error(E_ARG, "gpupot: particle range outside [0, n)");
        return E_ARG;
    }
    const int tiles = (n + PT_TJ - 1) / PT_TJ;
    // Two i per lane, which share each LDS read, in 16,384 work-groups at least where there
    // are tiles enough (an uneven last round of 2048 cost 7 %: n = 262,144 22.7 -> 21.2 ms,
    // and 22.1 with one i per lane).  Below 4e8 pairs one i per lane, for more wavefronts:
    // n = 10,007 57 us against 69 with two, 40,000 585 us against 547; it was 220 us at
    // n = 10,007 with four i per lane in chunks of at least four tiles (90 work-groups).
    const int ipl = (long long)n * ni < 400000000ll ? 1 : 2;
    const int nib = (ni + PT_THREADS * ipl - 1) / (PT_THREADS * ipl);
    const int want = ((ipl == 1 ? 2048 : 16384) + nib - 1) / nib;
    int nchunk = std::max(1, std::min(want, tiles));
    const int clen = (tiles + nchunk - 1) / nchunk * PT_TJ;
    nchunk = (n + clen - 1) / clen;
    double *part = static_cast<double *>(g_part.get((size_t)nchunk * ni * sizeof(double)));
    PotParams p{d_x, n, n_stride, i0, ni, clen, part};
    KTimer &t = ktimer("pot");
    t.start(s);
    if (ipl == 2)
        hipLaunchKernelGGL(pot_tile_kernel<2>, dim3(nib, nchunk), dim3(PT_THREADS), 0, s, p);
    else
        hipLaunchKernelGGL(pot_tile_kernel<1>, dim3(nib, nchunk), dim3(PT_THREADS), 0, s, p);
    NB6_HIP(hipGetLastError());
    t.stop(s);
    hipLaunchKernelGGL(pot_sum_kernel, dim3((ni + 63) / 64), dim3(64), 0, s, part, ni, nchunk,
                       d_pot);
    NB6_HIP(hipGetLastError());
    return OK;
}

void pot_release() { g_part.release(); }

}  // namespace nb6
