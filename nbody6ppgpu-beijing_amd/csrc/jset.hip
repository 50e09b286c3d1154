// Device-side layout of the j-particles (what gpunb_send_ uploads).
//
// The reference packs j into FP32 absolute coordinates (Jparticle,
// gpunb.velocity.cu:58-93).  Here the j-set is kept in FP64 and re-ordered
// along a Morton (Z-order) curve on the device at every send, so that each tile
// of 256 consecutive j occupies a small region of space.  Every tile t has an
// origin (P_t, V_t): P_t the position of its middle record, V_t the mean velocity
// of its massive records (the middle record's own velocity would put the orbital
// velocity of a tight binary member into every relative velocity of the tile);
// the regular-force kernel streams
//   rec32[s] = { x - Px, y - Py, z - Pz, m,  vx - Vx, vy - Vy, vz - Vz, 0 }  (FP32)
// and forms the i side relative to the same origin in FP64, so the FP32
// separation carries the rounding error of the tile's extent, not of |x|.
// rec64 (sorted, AoS, 64 B) feeds the FP64 near-field / neighbour re-test, and
// perm[s] maps a sorted position back to the caller's 0-based j index.
#include "nb6_internal.h"

#include "block_sort.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cfloat>

namespace nb6 {

namespace {

// 21 bits per axis: a cluster with escapers far out still gets a fine order in its core
constexpr double MORTON_CELLS = 2097152.0;   // 2^21 per axis

__device__ __forceinline__ unsigned long long morton63(double x, double y, double z, double lx,
                                                       double ly, double lz, double sx, double sy,
                                                       double sz) {
    const double fx = (x - lx) * sx, fy = (y - ly) * sy, fz = (z - lz) * sz;
    // comparisons in FP64 first: NaN and far-outside values clamp without overflow
    const unsigned qx = fx > 0.0 ? (fx < MORTON_CELLS - 1.0 ? (unsigned)fx : 2097151u) : 0u;
    const unsigned qy = fy > 0.0 ? (fy < MORTON_CELLS - 1.0 ? (unsigned)fy : 2097151u) : 0u;
    const unsigned qz = fz > 0.0 ? (fz < MORTON_CELLS - 1.0 ? (unsigned)fz : 2097151u) : 0u;
    return spread21(qx) | (spread21(qy) << 1) | (spread21(qz) << 2);
}

constexpr int STATS_GROUPS = 512;

__device__ __forceinline__ void stat_identity(double *v) {
#pragma unroll
    for (int d = 0; d < 3; d++) {
        v[d] = DBL_MAX;
        v[3 + d] = -DBL_MAX;
    }
    v[6] = 0.0;
}
__device__ __forceinline__ void stat_add(double *v, double x, double y, double z, double m) {
    const double r[3] = {x, y, z};
#pragma unroll
    for (int d = 0; d < 3; d++) {
        v[d] = fmin(v[d], r[d]);
        v[3 + d] = fmax(v[3 + d], r[d]);
    }
    v[6] = fmax(v[6], m);
}
// bounds (lo[3], hi[3]) and maximum mass over the work-group's wavefronts, in every thread
__device__ __forceinline__ void stat_group(double *v, double (*sh)[8]) {
#pragma unroll
    for (int q = 0; q < 7; q++)
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const double u = __shfl_xor(v[q], o, 64);
            v[q] = q < 3 ? fmin(v[q], u) : fmax(v[q], u);
        }
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int q = 0; q < 7; q++) sh[threadIdx.x >> 6][q] = v[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 7; q++)
#pragma unroll
        for (int w = 0; w < (int)(blockDim.x >> 6); w++)
            v[q] = q < 3 ? fmin(v[q], sh[w][q]) : fmax(v[q], sh[w][q]);
}

// SoA [7][stride] (x y z vx vy vz m; null: aos is there already) -> AoS [n][8] (x y z m vx vy
// vz 0), and each work-group's bounds and maximum mass: part[group][7]
__global__ __launch_bounds__(256) void aos_stats_kernel(const double *__restrict__ soa, int n,
                                                        int stride, double *__restrict__ aos,
                                                        double *__restrict__ part) {
    __shared__ double sh[4][8];
    double v[7];
    stat_identity(v);
    for (int j = blockIdx.x * 256 + threadIdx.x; j < n; j += gridDim.x * 256) {
        double *o = aos + (size_t)j * 8;
        if (soa) {
            const size_t st = stride;
            const double x = soa[j], y = soa[st + j], z = soa[2 * st + j], m = soa[6 * st + j];
            o[0] = x; o[1] = y; o[2] = z; o[3] = m;
            o[4] = soa[3 * st + j]; o[5] = soa[4 * st + j]; o[6] = soa[5 * st + j];
            o[7] = 0.0;
            stat_add(v, x, y, z, m);
        } else {
            stat_add(v, o[0], o[1], o[2], o[3]);
        }
    }
    stat_group(v, sh);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < 7; q++) part[blockIdx.x * 7 + q] = v[q];
}

struct JStat {
    double v[7];             // lo[3], hi[3], maximum mass
};
__device__ __forceinline__ double morton_scale(const double *box, int d) {
    const double w = box[3 + d] - box[d];
    return w > 0.0 ? MORTON_CELLS / (w * (1.0 + 1e-12)) : 0.0;
}

// Morton keys of the AoS positions in their box, from the groups' bounds (every work-group
// reduces them: cheaper than a launch) or, with groups = 0, from `host`; the first
// work-group leaves the bounds and the maximum mass in stat[7]
struct JKeys {
    const double *in, *part;
    int groups;
    JStat host;
    double *stat;
    double v[7], sc[3];      // (device, from begin)
    __device__ void begin() {
        __shared__ double sh[16][8];
        stat_identity(v);
        if (groups > 0) {
            for (int g = threadIdx.x; g < groups; g += blockDim.x)
#pragma unroll
                for (int q = 0; q < 7; q++) {
                    const double u = part[g * 7 + q];
                    v[q] = q < 3 ? fmin(v[q], u) : fmax(v[q], u);
                }
            stat_group(v, sh);
        } else {
#pragma unroll
            for (int q = 0; q < 7; q++) v[q] = host.v[q];
        }
        if (blockIdx.x == 0 && threadIdx.x == 0)
#pragma unroll
            for (int q = 0; q < 7; q++) stat[q] = v[q];
#pragma unroll
        for (int d = 0; d < 3; d++) sc[d] = morton_scale(v, d);
    }
    __device__ unsigned long long key(int j) const {
        const double *r = in + (size_t)j * 8;
        return morton63(r[0], r[1], r[2], v[0], v[1], v[2], sc[0], sc[1], sc[2]);
    }
};
__global__ __launch_bounds__(256) void morton_kernel(JKeys kf, int n,
                                                     unsigned long long *__restrict__ key,
                                                     int *__restrict__ val) {
    kf.begin();
    for (int j = blockIdx.x * 256 + threadIdx.x; j < n; j += gridDim.x * 256) {
        key[j] = kf.key(j);
        val[j] = j;
    }
}

// Morton keys of i-particle positions (SoA rows 0-2) in the j-set's box (clamped)
struct IKeys {
    const double *ib;
    int stride;
    const double *box;
    __device__ void begin() {}
    __device__ unsigned long long key(int i) const {
        return morton63(ib[i], ib[(size_t)stride + i], ib[2 * (size_t)stride + i], box[0], box[1],
                        box[2], morton_scale(box, 0), morton_scale(box, 1), morton_scale(box, 2));
    }
};
struct PutOrder {
    int *order;
    __device__ void put(int place, int e, unsigned long long) const { order[place] = e; }
};

__global__ __launch_bounds__(256) void imorton_kernel(IKeys kf, int ni,
                                                      unsigned long long *__restrict__ key,
                                                      int *__restrict__ val) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ni) return;
    key[i] = kf.key(i);
    val[i] = i;
}

// v and the lane that the DPP pattern names (the lane's own value where there is none)
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_bound(float v, bool lo) {
    const int i = __float_as_int(v);
    const float u = __int_as_float(__builtin_amdgcn_update_dpp(i, i, CTRL, ROWS, 0xf, false));
    return lo ? fminf(v, u) : fmaxf(v, u);
}

// One work-group per tile: the records in sorted order (rec64), the tile's origin, its FP32
// records relative to the origin and their bounds (JSet::tbox), in one pass over the
// records.  P = position of the tile's middle record (its first in the padded layout), V =
// mean velocity of the tile's records with m > 0 (that record's velocity if there are none).
// Plain j-set (padoff null): position s holds the caller's record perm[s].  Padded layout of
// independent clusters: slot s of cluster c (padoff) holds record sorted[off[c] + s -
// padoff[c]] of the compact order, or past the cluster's last one a far massless record, and
// perm is written.  Four launches of separate kernels took 17 us at N = 50,021 where this
// takes 8.7.
__global__ __launch_bounds__(256) void tile_build_kernel(
    const double *__restrict__ in, int n, int *__restrict__ perm, const int *__restrict__ sorted,
    const int *__restrict__ off, const int *__restrict__ padoff, int nc,
    double *__restrict__ rec64, double *__restrict__ torg, float4 *__restrict__ rec32,
    float *__restrict__ tbox) {
    __shared__ double sh[4][4], rep[6], org[6];
    __shared__ float sb[4][16];
    const int t = blockIdx.x, k = threadIdx.x, lane = k & 63, w = k >> 6;
    const int s = t * JTILE + k;
    const int c = min(JTILE, n - t * JTILE);
    const int mid = padoff ? 0 : c / 2;
    int j = -1;
    if (padoff) {
        int cl = 0, hi = nc;             // the cluster with padoff[cl] <= tile start (uniform)
        while (hi - cl > 1) {
            const int m = (cl + hi) >> 1;
            if (padoff[m] <= t * JTILE) cl = m; else hi = m;
        }
        const int q = off[cl] + (s - padoff[cl]);
        if (q < off[cl + 1]) j = sorted[q];
        perm[s] = j;
    } else if (k < c) {
        j = perm[s];
    }
    double r[8] = {1.0e17, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (j >= 0) {
        const double2 *p = reinterpret_cast<const double2 *>(in + (size_t)j * 8);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const double2 u = p[q];
            r[2 * q] = u.x;
            r[2 * q + 1] = u.y;
        }
    }
    if (k < c) {
        double2 *o = reinterpret_cast<double2 *>(rec64 + (size_t)s * 8);
#pragma unroll
        for (int q = 0; q < 4; q++) o[q] = make_double2(r[2 * q], r[2 * q + 1]);
    }
    const bool use = k < c && r[3] > 0.0;
    double q[4] = {use ? r[4] : 0.0, use ? r[5] : 0.0, use ? r[6] : 0.0, use ? 1.0 : 0.0};
#pragma unroll
    for (int f = 0; f < 4; f++)
        for (int o = 32; o > 0; o >>= 1) q[f] += __shfl_xor(q[f], o, 64);
    if (lane == 0)
        for (int f = 0; f < 4; f++) sh[w][f] = q[f];
    if (k == mid) {
        rep[0] = r[0]; rep[1] = r[1]; rep[2] = r[2];
        rep[3] = r[4]; rep[4] = r[5]; rep[5] = r[6];
    }
    __syncthreads();
    if (k == 0) {
        double v[4];
        for (int f = 0; f < 4; f++) v[f] = (sh[0][f] + sh[1][f]) + (sh[2][f] + sh[3][f]);
        double *o = torg + (size_t)t * 8;
        for (int f = 0; f < 3; f++) {
            org[f] = rep[f];
            org[3 + f] = v[3] > 0.0 ? v[f] / v[3] : rep[3 + f];
            o[f] = org[f];
            o[3 + f] = org[3 + f];
        }
        o[6] = 0.0; o[7] = 0.0;
    }
    __syncthreads();
    const float4 a = make_float4((float)(r[0] - org[0]), (float)(r[1] - org[1]),
                                 (float)(r[2] - org[2]), (float)r[3]);
    const float4 b = make_float4((float)(r[4] - org[3]), (float)(r[5] - org[4]),
                                 (float)(r[6] - org[5]), 0.f);
    if (k < c) {
        rec32[2 * (size_t)s] = a;
        rec32[2 * (size_t)s + 1] = b;
    }
    // bounds: position lo[3], hi[3], velocity lo[3], hi[3], maximum mass, record count
    const bool in_box = k < c && fabsf(a.x) < 1.0e16f;
    float v[13] = {a.x, a.y, a.z, a.x, a.y, a.z, b.x, b.y, b.z, b.x, b.y, b.z, a.w};
#pragma unroll
    for (int f = 0; f < 13; f++) {
        const bool lo = f < 3 || (f >= 6 && f < 9);
        if (!in_box) v[f] = lo ? FLT_MAX : (f == 12 ? 0.f : -FLT_MAX);
        // (row_shr 1, 2, 4, 8, row_bcast 15, 31: lane 63 has seen every lane)
        v[f] = dpp_bound<0x111, 0xf>(v[f], lo);
        v[f] = dpp_bound<0x112, 0xf>(v[f], lo);
        v[f] = dpp_bound<0x114, 0xf>(v[f], lo);
        v[f] = dpp_bound<0x118, 0xf>(v[f], lo);
        v[f] = dpp_bound<0x142, 0xa>(v[f], lo);
        v[f] = dpp_bound<0x143, 0xc>(v[f], lo);
        if (lane == 63) sb[w][f] = v[f];
    }
    const unsigned long long held = __ballot(in_box);
    if (lane == 63) sb[w][13] = (float)__popcll(held);
    __syncthreads();
    if (k < TBOX) {
        float u = 0.f;
        if (k < 14) {
            const bool lo = k < 3 || (k >= 6 && k < 9);
            u = sb[0][k];
            for (int x = 1; x < 4; x++)
                u = k == 13 ? u + sb[x][k] : (lo ? fminf(u, sb[x][k]) : fmaxf(u, sb[x][k]));
        }
        tbox[(size_t)t * TBOX + k] = u;
    }
}

// plain streaming copy (used to calibrate HBM byte counters against a known size)
__global__ __launch_bounds__(256) void copy_kernel(const uint4 *__restrict__ src,
                                                   uint4 *__restrict__ dst, size_t n16) {
    for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n16; k += (size_t)gridDim.x * 256)
        dst[k] = src[k];
}

}  // namespace

void device_copy(void *dst, const void *src, size_t bytes, hipStream_t s) {
    const size_t n16 = bytes / 16;
    if (n16 == 0) return;
    const size_t blocks = std::min<size_t>((n16 + 255) / 256, 8192);
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, s,
                       static_cast<const uint4 *>(src), static_cast<uint4 *>(dst), n16);
    NB6_HIP(hipGetLastError());
}

void jset_reserve(JSet &js, int cap) {
    if (cap <= js.cap) return;
    js.cap = cap;
    const int ntile = (cap + JTILE - 1) / JTILE;
    js.in64.get((size_t)cap * 8 * sizeof(double));
    js.rec64.get((size_t)cap * 8 * sizeof(double));
    js.rec32.get((size_t)cap * 2 * sizeof(float4));
    js.torg.get((size_t)ntile * 8 * sizeof(double));
    js.perm.get((size_t)cap * sizeof(int));
    js.keys.get((size_t)cap * 2 * sizeof(unsigned long long));
    js.vals.get((size_t)cap * 2 * sizeof(int));
    js.stat.get((8 + 7 * STATS_GROUPS) * sizeof(double));   // stat[7], groups' parts
    js.tbox.get((size_t)ntile * TBOX * sizeof(float));
}

void jset_release(JSet &js) {
    js.in64.release(); js.rec64.release(); js.rec32.release(); js.torg.release();
    js.perm.release(); js.keys.release(); js.vals.release(); js.stat.release();
    js.sort_tmp.release(); js.tbox.release();
    js.cap = 0; js.n = 0; js.ntile = 0;
    if (js.read) (void)hipEventDestroy(js.read);
    if (js.built) (void)hipEventDestroy(js.built);
    js.read = js.built = nullptr;
    js.pending = js.recorded = false;
}

// The caller's input has been read, and in64 written, once the work queued so far is done; a
// send returns after that (its caller may then reuse the memory, on any stream), not after the
// whole build.
void jset_input_queued(JSet &js, hipStream_t s) {
    if (!js.read) NB6_HIP(hipEventCreateWithFlags(&js.read, hipEventDisableTiming));
    NB6_HIP(hipEventRecord(js.read, s));
}
void jset_input_wait(JSet &js) { NB6_HIP(hipEventSynchronize(js.read)); }

// A build is queued when its send returns.  Work on its own stream follows it there; work on
// another stream waits for an event after it.  The library's stream lives as long as the
// library, so there the event is recorded when another stream asks; a caller's stream can be
// gone by then and gets it at once.
namespace {
void record_built(const JSet &js) {
    if (!js.built) NB6_HIP(hipEventCreateWithFlags(&js.built, hipEventDisableTiming));
    NB6_HIP(hipEventRecord(js.built, js.stream));
    js.recorded = true;
}
void build_queued(JSet &js, hipStream_t s) {
    js.stream = s;
    js.pending = true;
    js.recorded = false;
    if (s != device().stream) record_built(js);
}
}  // namespace
void jset_ready(const JSet &js, hipStream_t s) {
    if (!js.pending || s == js.stream) return;
    // A captured call runs when its graph does, which the caller orders; a stream under capture
    // can neither wait for an event from outside nor may the thread wait for one meanwhile.
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    NB6_HIP(hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone) return;
    if (!js.recorded) record_built(js);
    const hipError_t e = hipEventQuery(js.built);
    if (e == hipErrorNotReady) {
        (void)hipGetLastError();
        NB6_HIP(hipStreamWaitEvent(s, js.built, 0));
        return;
    }
    NB6_HIP(e);
    js.pending = false;
}

namespace {
int stat_groups(int n) { return std::min(STATS_GROUPS, (n + 255) / 256); }

// from in64 and, with groups > 0, its groups' parts in js.stat (else host.v)
void build(JSet &js, int n, int groups, const JStat &host, hipStream_t s) {
    js.n = n;
    js.ntile = (n + JTILE - 1) / JTILE;
    if (n <= 0) return;
    unsigned long long *k0 = js.keys.as<unsigned long long>();
    unsigned long long *k1 = k0 + js.cap;
    int *v0 = js.vals.as<int>();
    int *v1 = js.perm.as<int>();
    double *stat = js.stat.as<double>();
    const JKeys kf{js.in64.as<double>(), stat + 8, groups, host, stat, {}, {}};
    if (n <= BSORT_MAX) {
        bsort(kf, PutOrder{v1}, n, k0, v0, s);
    } else {
        hipLaunchKernelGGL(morton_kernel, dim3(1024), dim3(256), 0, s, kf, n, k0, v0);
        NB6_HIP(hipGetLastError());
        size_t tb = 0;
        NB6_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k0, k1, v0, v1, n, 0, 63, s));
        void *tmp = js.sort_tmp.get(tb);
        NB6_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, v0, v1, n, 0, 63, s));
    }
    hipLaunchKernelGGL(tile_build_kernel, dim3(js.ntile), dim3(256), 0, s, js.in64.as<double>(), n,
                       v1, nullptr, nullptr, nullptr, 0, js.rec64.as<double>(), js.torg.as<double>(),
                       js.rec32.as<float4>(), js.tbox.as<float>());
    NB6_HIP(hipGetLastError());
    build_queued(js, s);
}
}  // namespace

// in64 holds n AoS records in the caller's order; box = {lo[3], hi[3]} or nullptr
void jset_build(JSet &js, int n, const double *box, double mmax, hipStream_t s) {
    JStat host{};
    int groups = 0;
    if (n > 0 && box) {
        for (int q = 0; q < 6; q++) host.v[q] = box[q];
        host.v[6] = mmax;
    } else if (n > 0) {
        groups = stat_groups(n);
        hipLaunchKernelGGL(aos_stats_kernel, dim3(groups), dim3(256), 0, s, nullptr, n, 0,
                           js.in64.as<double>(), js.stat.as<double>() + 8);
        NB6_HIP(hipGetLastError());
        jset_input_queued(js, s);
    }
    build(js, n, groups, host, s);
    if (groups > 0) jset_input_wait(js);     // in64 is written
}

void jset_build_clusters(JSet &js, int npad, const double *in, const int *sorted, const int *off,
                         const int *padoff, int nc, hipStream_t s) {
    js.n = npad;
    js.ntile = npad / JTILE;
    hipLaunchKernelGGL(tile_build_kernel, dim3(js.ntile), dim3(256), 0, s, in, npad,
                       js.perm.as<int>(), sorted, off, padoff, nc, js.rec64.as<double>(),
                       js.torg.as<double>(), js.rec32.as<float4>(), js.tbox.as<float>());
    NB6_HIP(hipGetLastError());
}

const int *jset_sort_i(const JSet &js, int ni, int stride, const double *d_i, RegfWork &w,
                       hipStream_t s) {
    unsigned long long *k0 =
        static_cast<unsigned long long *>(w.ikey.get((size_t)ni * 2 * sizeof(unsigned long long)));
    unsigned long long *k1 = k0 + ni;
    int *v0 = static_cast<int *>(w.ival.get((size_t)ni * 3 * sizeof(int)));
    int *v1 = v0 + 2 * (size_t)ni;
    const IKeys kf{d_i, stride, js.stat.as<double>()};
    if (ni <= BSORT_MAX) {
        bsort(kf, PutOrder{v1}, ni, k0, v0, s);
        return v1;
    }
    hipLaunchKernelGGL(imorton_kernel, dim3((ni + 255) / 256), dim3(256), 0, s, kf, ni, k0, v0);
    NB6_HIP(hipGetLastError());
    size_t tb = 0;
    NB6_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tb, k0, k1, v0, v1, ni, 0, 63, s));
    void *tmp = w.itmp.get(tb);
    NB6_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tb, k0, k1, v0, v1, ni, 0, 63, s));
    return v1;
}

namespace {
// row i of a [n][lmax] list array holds 1 + count ints (1 if the count is negative or
// above maxc); len[n] = 0 so that the exclusive scan's last entry is the total
__global__ __launch_bounds__(256) void row_len_kernel(const int *__restrict__ list, int n, int lmax,
                                                      int maxc, int *__restrict__ len) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i > n) return;
    int l = 0;
    if (i < n) {
        const int c = list[(size_t)i * lmax];
        l = 1 + (c > 0 && c <= maxc ? c : 0);
    }
    len[i] = l;
}

// one wavefront per row: copy its 1 + count ints to pack + off[i]
__global__ __launch_bounds__(256) void row_pack_kernel(const int *__restrict__ list, int n, int lmax,
                                                       const int *__restrict__ off,
                                                       int *__restrict__ pack) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= n) return;
    const int lane = threadIdx.x & 63;
    const int o = off[i], l = off[i + 1] - o;
    const int *src = list + (size_t)i * lmax;
    for (int k = lane; k < l; k += 64) pack[o + k] = src[k];
}
// The results of a small block straight into pinned host memory, one wavefront per row: the seven
// numbers side by side (out[8 i ..]) and the used part of the row's list.  Bound by the
// bus: copies of all of both arrays, most of it unused list, took 53 us at ni = 1024, lmax = 500
// (N = 65,536, send and force: 541 -> 475 us; N = 1024, ni = 40: 132 -> 114 us).
__global__ __launch_bounds__(256) void deliver_kernel(const double *__restrict__ res,
                                                      const int *__restrict__ list, int ni, int lmax,
                                                      int nnbmax, double *__restrict__ out,
                                                      int *__restrict__ rows) {
    const int lane = threadIdx.x & 63, i = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= ni) return;
    if (lane < 7) out[8 * (size_t)i + lane] = res[(size_t)lane * ni + i];
    const int *src = list + (size_t)i * lmax;
    int *dst = rows + (size_t)i * lmax;
    const int c = src[0], len = 1 + (c > 0 && c <= nnbmax ? c : 0);
    for (int k = lane; k < len; k += 64) dst[k] = src[k];
}

}  // namespace

void deliver_rows(const double *res, const int *list, int ni, int lmax, int nnbmax, double *out,
                  int *rows, hipStream_t s) {
    hipLaunchKernelGGL(deliver_kernel, dim3((ni + 3) / 4), dim3(256), 0, s, res, list, ni, lmax,
                       nnbmax, out, rows);
    NB6_HIP(hipGetLastError());
}

void pack_rows(const int *list, int n, int lmax, int maxc, int *len, int *off, int *pack,
               DBuf &tmp, hipStream_t s) {
    hipLaunchKernelGGL(row_len_kernel, dim3((n + 1 + 255) / 256), dim3(256), 0, s, list, n, lmax,
                       maxc, len);
    NB6_HIP(hipGetLastError());
    size_t tb = 0;
    NB6_HIP(hipcub::DeviceScan::ExclusiveSum(nullptr, tb, len, off, n + 1, s));
    void *t = tmp.get(tb);
    NB6_HIP(hipcub::DeviceScan::ExclusiveSum(t, tb, len, off, n + 1, s));
    hipLaunchKernelGGL(row_pack_kernel, dim3((n + 3) / 4), dim3(256), 0, s, list, n, lmax, off, pack);
    NB6_HIP(hipGetLastError());
}

void jset_from_soa(JSet &js, int n, int stride, const double *d_soa, hipStream_t s) {
    if (n <= 0) {
        build(js, n, 0, JStat{}, s);
        return;
    }
    jset_ready(js, s);
    const int groups = stat_groups(n);
    hipLaunchKernelGGL(aos_stats_kernel, dim3(groups), dim3(256), 0, s, d_soa, n, stride,
                       js.in64.as<double>(), js.stat.as<double>() + 8);
    NB6_HIP(hipGetLastError());
    jset_input_queued(js, s);
    build(js, n, groups, JStat{}, s);
    jset_input_wait(js);
}

}  // namespace nb6
