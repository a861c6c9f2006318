// pp_merge.hip -- the catalogue merger on the device: Lagrangian exclusion
// and volume reduction of a halo catalogue.
//
// Reference: merge_catalog (src/Merger/Merger.jl:21-79) over
// lagrangian_exclusion! / volume_reduction! / sphere_overlap and the 256^3
// spatial hash (src/Merger/Exclusion.jl:14-222).
//
// The reference walks the halos serially in descending radius order (stable
// sort); a surviving halo kills every surviving, not larger halo whose centre
// lies inside its radius.  That greedy pass is the same as: halo j survives
// iff no surviving halo earlier in the order contains j's centre (a halo
// earlier in the order is never smaller).  Here:
// * the halos are sorted by the cells of a grid of two cells a halo and
//   stay in that order: neighbours in space are neighbours in memory, and the
//   candidates of a row of cells are one run of the list (two loads, whatever
//   the row's length).  The reference's grid has 256 cells a side whatever the
//   catalogue, 10^4 cells for each halo of a small one;
// * several lanes share a halo and take its rows of cells in turn (one lane a
//   halo spent most of its time on the few largest radii);
// * "earlier in the order" compares radius and index, which needs no sort;
// * every halo k lists the later halos j it contains ("killer" edges k -> j,
//   stored by j);
// * rounds over the undecided halos settle them: j dies as soon as one of
//   its killers is known to survive, survives once all its killers are known
//   dead; the earliest undecided halo always settles, so the rounds end;
// * the reduction visits every overlapping surviving pair once, from its
//   larger member (whose cells within twice its radius hold every smaller
//   partner), with both cap volumes of sphere_overlap.  The larger member's
//   caps are summed in Float64 by its lanes; the smaller member's are added
//   by atomics as whole numbers of 2^-54 of its volume, finer than the 2^-53
//   to which Float64 subtracts them from it and the same in every order: the
//   result does not depend on thread timing, and no list of pairs is stored
//   or sorted.  (The sum stays under the 2^10 volumes that fit: a partner's
//   centre is outside of the halo and of the other partners, so that a cap
//   is under half the volume and at most a few hundred spheres touch it.)
//   The deficit is the reference's (which adds each pair from both sides and
//   halves) up to Float64 rounding;
// * the work space is the context's (it was 25 allocations a call).
// At 1.2 M halos with their records (a 600 Mpc/h box) a merge takes 1.7 ms
// instead of 41.1 ms.  What bounds it: the chains of
// dependent loads (cell, row, candidates) of k_pairs (0.38 ms, was 2 x 13 ms)
// and k_killers (0.18 and 0.24 ms, was 2 x 2.6 ms); an arithmetic half as
// long (Float32 distances before Float64 ones) changed neither.  At 300 to
// 700 halos 0.4 ms instead of 200 to 560 ms, most of it the empty cells.
#include <hipcub/hipcub.hpp>

#include <cmath>

#include "pp_common.h"

namespace pp {

constexpr int kMergeAxis = 1024;            // most cells on an axis
constexpr int64_t kMergeCells = 1ll << 27;  // most cells of a grid
// Lanes that share a halo's rows of cells.  k_killers / k_pairs over 1.2 M
// halos (median radius 1.5 in a 600^3 box, the largest 15) with 4, 8 and 16
// lanes for the first: 200, 216 and 257 us; 8, 16 and 32 for the second: 697,
// 616 and 733 us.  With the grid at 1, 2 and 4 cells a halo all kernels
// together are within 3 % (fewer candidates against more rows to look up); 2
// leaves room for clustering.
constexpr int kKillY = 4, kKillZ = 2, kKillLanes = kKillY * kKillZ;
constexpr int kPairY = 4, kPairZ = 4, kPairLanes = kPairY * kPairZ;
constexpr int kCellsPerHalo = 2;
constexpr int kBoundBlocks = 256;

struct MergeGeo {
    double o[3], inv;  // grid origin, 1 / cell size
    int nc[3];
};

struct MergeIn {
    const float *x, *y, *z, *r;
    int64_t n;
};

// the halos in cell order
struct MergeCells {
    const float4 *h;       // x, y, z, r
    const int32_t *id;     // position in the catalogue
    const int32_t *first;  // per cell, and one more: its first halo
    int64_t n;
};

// c cells from the origin: the cell, clamped to the grid (NaN: 0)
__device__ __forceinline__ int cell_clamp(double c, int nc)
{
    return c >= 1.0 ? (c < (double)nc ? (int)c : nc - 1) : 0;
}

// halo a comes before halo b: larger, or as large and earlier in the catalogue
__device__ __forceinline__ bool before(const MergeCells &C, int64_t a, float ra, int64_t b, float rb)
{
    return ra > rb || (ra == rb && C.id[a] < C.id[b]);
}

__device__ __forceinline__ double dist_of(const float4 &a, const float4 &b)
{
#pragma clang fp contract(off)
    const double dx = (double)b.x - (double)a.x, dy = (double)b.y - (double)a.y, dz = (double)b.z - (double)a.z;
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// whether a and b are further apart than R for certain (Float32: the sum of
// squares is right to 4e-7 of itself, the margin is 1e-5; radii whose squares
// would be denormal are left to Float64)
__device__ __forceinline__ bool apart(const float4 &a, const float4 &b, float R)
{
    const float dx = b.x - a.x, dy = b.y - a.y, dz = b.z - a.z;
    return R > 1e-15f && dx * dx + dy * dy + dz * dz > R * R * 1.00001f;
}

__device__ __forceinline__ int cell_between(float c, int lo, int hi)
{
    return max(lo, min((int)floorf(c), hi));
}

// fn(j, halo j) for every halo within R of halo p and others of the cells
// there.  LY x LZ lanes take the rows of cells in turn, each BATCH candidates
// of a row at once: the chain of loads is what bounds this.  Distances are in
// cells from p's own cell, in Float32 with margins over their rounding.
template <int LY, int LZ, int BATCH, class Fn>
__device__ __forceinline__ void around(const MergeCells &C, const MergeGeo &G, const float4 &p, double R, Fn fn)
{
    const double ux = ((double)p.x - G.o[0]) * G.inv, uy = ((double)p.y - G.o[1]) * G.inv,
                 uz = ((double)p.z - G.o[2]) * G.inv;
    const int cx = cell_clamp(ux, G.nc[0]), cy = cell_clamp(uy, G.nc[1]), cz = cell_clamp(uz, G.nc[2]);
    const float fx = (float)(ux - cx), fy = (float)(uy - cy), fz = (float)(uz - cz);
    const float u = fminf((float)(R * G.inv) * 1.000002f + 1e-5f, 4.0f * kMergeAxis);
    const int ly = threadIdx.x & (LY - 1), lz = threadIdx.x / LY & (LZ - 1);
    const int xl = -cx, xh = G.nc[0] - 1 - cx, yl = -cy, yh = G.nc[1] - 1 - cy, zl = -cz, zh = G.nc[2] - 1 - cz;
    const int y0 = cell_between(fy - u, yl, yh), y1 = cell_between(fy + u, yl, yh);
    const int z0 = cell_between(fz - u, zl, zh), z1 = cell_between(fz + u, zl, zh);
    if (y0 == y1 && z0 == z1) {
        // a sphere within one long row (small beside the cells, as where a few
        // far halos stretch the grid): the lanes share its candidates (100 k
        // halos and a far one 162 -> 51 ms; 1.2 M evenly spread 1.60 -> 1.63)
        const int64_t row = (int64_t)G.nc[0] * ((cy + y0) + (int64_t)G.nc[1] * (cz + z0)) + cx;
        const int32_t e0 = C.first[row + cell_between(fx - u, xl, xh)], e1 = C.first[row + cell_between(fx + u, xl, xh) + 1];
        if (e1 - e0 > 4 * LY * LZ) {
            for (int32_t q = threadIdx.x & (LY * LZ - 1); q < e1 - e0; q += LY * LZ) fn(e0 + q, C.h[e0 + q]);
            return;
        }
    }
    for (int z = z0 + lz; z <= z1; z += LZ)
        for (int y = y0 + ly; y <= y1; y += LY) {
            // the row's nearest point in y and z, and what that leaves of u in x
            const float gy = fmaxf(fmaxf((float)y - fy, fy - (float)(y + 1)), 0.0f);
            const float gz = fmaxf(fmaxf((float)z - fz, fz - (float)(z + 1)), 0.0f);
            const float w2 = u * u * 1.000002f - gy * gy - gz * gz;
            if (w2 < 0.0f) continue;
            const float w = sqrtf(w2) * 1.000002f + 1e-5f;
            const int64_t row = (int64_t)G.nc[0] * ((cy + y) + (int64_t)G.nc[1] * (cz + z)) + cx;
            const int32_t e1 = C.first[row + cell_between(fx + w, xl, xh) + 1];
            for (int32_t e = C.first[row + cell_between(fx - w, xl, xh)]; e < e1; e += BATCH) {
                float4 c[BATCH];
#pragma unroll
                for (int a = 0; a < BATCH; a++) c[a] = C.h[min(e + a, e1 - 1)];
#pragma unroll
                for (int a = 0; a < BATCH; a++)
                    if (e + a < e1) fn(e + a, c[a]);
            }
        }
}

// sphere_overlap (Exclusion.jl:64-96): cap volumes cut from spheres 1 and 2
__device__ __forceinline__ void sphere_caps(double d, double r1, double r2, double &v1, double &v2)
{
#pragma clang fp contract(off)
    v1 = v2 = 0.0;
    if (d >= r1 + r2 || d <= fabs(r1 - r2)) return;
    const double h1 = (r2 - r1 + d) * (r2 + r1 - d) / (2.0 * d);
    const double h2 = (r1 - r2 + d) * (r1 + r2 - d) / (2.0 * d);
    const double pi3 = 3.141592653589793 / 3.0;
    v1 = pi3 * (h1 * h1) * (3.0 * r1 - h1);
    v2 = pi3 * (h2 * h2) * (3.0 * r2 - h2);
}

// min/max of the positions and max radius of a block's lanes, in lane 0
__device__ __forceinline__ void bound_reduce(float (&red)[7][256], const float (&v)[7])
{
    for (int q = 0; q < 7; q++) red[q][threadIdx.x] = v[q];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w)
            for (int q = 0; q < 7; q++) {
                const float a = red[q][threadIdx.x], b = red[q][threadIdx.x + w];
                red[q][threadIdx.x] = (q & 1) || q == 6 ? fmaxf(a, b) : fminf(a, b);
            }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(256) k_merge_bounds(MergeIn H, float *__restrict__ part)
{
    __shared__ float red[7][256];
    float v[7] = {INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY, -INFINITY};
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < H.n; i += (int64_t)gridDim.x * 256) {
        v[0] = fminf(v[0], H.x[i]);
        v[1] = fmaxf(v[1], H.x[i]);
        v[2] = fminf(v[2], H.y[i]);
        v[3] = fmaxf(v[3], H.y[i]);
        v[4] = fminf(v[4], H.z[i]);
        v[5] = fmaxf(v[5], H.z[i]);
        v[6] = fmaxf(v[6], H.r[i]);
    }
    bound_reduce(red, v);
    if (threadIdx.x < 7) part[blockIdx.x * 7 + threadIdx.x] = red[threadIdx.x][0];
}

__global__ void __launch_bounds__(256) k_merge_bounds2(const float *__restrict__ part, int blocks,
                                                       double *__restrict__ out)
{
    __shared__ float red[7][256];
    float v[7] = {INFINITY, -INFINITY, INFINITY, -INFINITY, INFINITY, -INFINITY, -INFINITY};
    for (int b = threadIdx.x; b < blocks; b += 256)
        for (int q = 0; q < 7; q++)
            v[q] = (q & 1) || q == 6 ? fmaxf(v[q], part[b * 7 + q]) : fminf(v[q], part[b * 7 + q]);
    bound_reduce(red, v);
    if (threadIdx.x < 7) out[threadIdx.x] = (double)red[threadIdx.x][0];
}

__global__ void k_merge_keys(MergeIn H, MergeGeo G, float4 *__restrict__ h, int32_t *__restrict__ cell,
                             int32_t *__restrict__ iota)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < H.n; i += (int64_t)gridDim.x * blockDim.x) {
        const float4 p = make_float4(H.x[i], H.y[i], H.z[i], H.r[i]);
        const int cx = cell_clamp(((double)p.x - G.o[0]) * G.inv, G.nc[0]);
        const int cy = cell_clamp(((double)p.y - G.o[1]) * G.inv, G.nc[1]);
        const int cz = cell_clamp(((double)p.z - G.o[2]) * G.inv, G.nc[2]);
        h[i] = p;
        cell[i] = cx + G.nc[0] * (cy + G.nc[1] * cz);
        iota[i] = (int32_t)i;
    }
}

// the halos in cell order, their counters cleared
__global__ void k_merge_gather(const float4 *__restrict__ in, int64_t n, const int32_t *__restrict__ id,
                               float4 *__restrict__ h, int32_t *__restrict__ count, int32_t *__restrict__ state,
                               unsigned long long *__restrict__ frac)
{
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < n; p += (int64_t)gridDim.x * blockDim.x) {
        h[p] = in[id[p]];
        count[p] = 0;
        state[p] = 0;
        frac[p] = 0;
    }
}

// first[c] = the number of keys below c, c in [0, ncell]
__global__ void k_cell_first(const int32_t *__restrict__ key, int64_t n, int64_t ncell, int32_t *__restrict__ first)
{
    for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c <= ncell; c += (int64_t)gridDim.x * blockDim.x) {
        int64_t lo = 0, hi = n;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if ((int64_t)key[mid] < c) lo = mid + 1;
            else hi = mid;
        }
        first[c] = (int32_t)lo;
    }
}

// pass 1 edges: every later halo j inside halo k's radius; count them by j, or
// (FILL, which counts down to 0 again) write them into j's list
template <bool FILL>
__global__ void __launch_bounds__(256, 8) k_killers(MergeCells C, MergeGeo G, int32_t *__restrict__ count,
                                                 const int64_t *__restrict__ off, int32_t *__restrict__ edges)
{
    for (int64_t k = ((int64_t)blockIdx.x * 256 + threadIdx.x) / kKillLanes; k < C.n;
         k += (int64_t)gridDim.x * (256 / kKillLanes)) {
        const float4 hk = C.h[k];
        const double rk = (double)hk.w;
        if (!(rk > 0.0)) continue;
        around<kKillY, kKillZ, 1>(C, G, hk, rk, [&](int32_t j, const float4 &hj) {
            if (hj.w > hk.w || apart(hk, hj, hk.w) || !(dist_of(hk, hj) < rk) || !before(C, k, hk.w, j, hj.w))
                return;
            if constexpr (FILL) edges[off[j] + atomicSub(&count[j], 1) - 1] = (int32_t)k;
            else atomicAdd(&count[j], 1);
        });
    }
}

// one round: 0 undecided, 1 survives, 2 excluded (its radius becomes -1, which
// no pair has); *undecided = round if any is left
__global__ void k_decide(int64_t n, const int64_t *__restrict__ off, const int32_t *__restrict__ edges,
                         int32_t *state, float4 *__restrict__ h, int32_t *__restrict__ undecided, int32_t round)
{
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
        if (state[j] != 0) continue;
        bool all_dead = true, killed = false;
        for (int64_t e = off[j]; e < off[j + 1]; e++) {
            const int32_t s = __atomic_load_n(&state[edges[e]], __ATOMIC_RELAXED);
            if (s == 1) {
                killed = true;
                break;
            }
            if (s == 0) all_dead = false;
        }
        if (killed) {
            __atomic_store_n(&state[j], 2, __ATOMIC_RELAXED);
            h[j].w = -1.0f;
        } else if (all_dead) __atomic_store_n(&state[j], 1, __ATOMIC_RELAXED);
        else *undecided = round;
    }
}

// sum over a block of 256, in thread 0
__device__ __forceinline__ unsigned long long block_total(unsigned long long v)
{
    __shared__ unsigned long long part[4];
    for (int w = 32; w > 0; w >>= 1) v += __shfl_down(v, w, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    return part[0] + part[1] + part[2] + part[3];
}

constexpr double kSphere = 4.0 * 3.141592653589793 / 3.0;
constexpr double kFrac = 18014398509481984.0;  // 2^54

// pass 2 from the larger member i: the sum of its caps, every partner's cap
// added to the partner's whole numbers, the pairs counted
__global__ void __launch_bounds__(256, 6) k_pairs(MergeCells C, MergeGeo G, double *__restrict__ caps,
                                               unsigned long long *__restrict__ frac,
                                               unsigned long long *__restrict__ npair)
{
#pragma clang fp contract(off)
    unsigned long long found = 0;
    for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) / kPairLanes; i < C.n;
         i += (int64_t)gridDim.x * (256 / kPairLanes)) {
        const float4 hi = C.h[i];
        const double ri = (double)hi.w;
        double sum = 0.0;
        if (ri > 0.0)
            around<kPairY, kPairZ, 2>(C, G, hi, 2.0 * ri, [&](int32_t j, const float4 &hj) {
                if (hj.w > hi.w || apart(hi, hj, hi.w + hj.w)) return;
                const double rj = (double)hj.w, d = dist_of(hi, hj);
                if (!(d < ri + rj && d > fabs(ri - rj)) || !before(C, i, hi.w, j, hj.w)) return;
                double v1, v2;
                sphere_caps(d, ri, rj, v1, v2);
                sum += v1;
                atomicAdd(&frac[j], (unsigned long long)llrint(v2 / (kSphere * (rj * rj * rj)) * kFrac));
                found++;
            });
        for (int w = kPairLanes / 2; w > 0; w >>= 1) sum += __shfl_down(sum, w, kPairLanes);
        if ((threadIdx.x & (kPairLanes - 1)) == 0) caps[i] = sum;
    }
    const unsigned long long t = block_total(found);
    if (threadIdx.x == 0 && t) atomicAdd(npair, t);
}

// reduced radii: deficit = caps as the larger member + caps as the smaller
// (nothing for a number of pairs that is refused)
__global__ void __launch_bounds__(256) k_finalize(MergeCells C, const int32_t *__restrict__ state,
                                                  const unsigned long long *__restrict__ npair,
                                                  const double *__restrict__ caps,
                                                  const unsigned long long *__restrict__ frac,
                                                  int8_t *__restrict__ keep, float *__restrict__ new_r,
                                                  unsigned long long *__restrict__ nkept)
{
#pragma clang fp contract(off)
    if (*npair >> 31) return;
    unsigned long long kept = 0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < C.n; i += (int64_t)gridDim.x * 256) {
        const int32_t o = C.id[i];
        int8_t k = 0;
        float nr = 0.0f;
        if (state[i] == 1) {
            const double r = (double)C.h[i].w, v = kSphere * (r * r * r);
            const double vol = v - (caps[i] + (double)frac[i] / kFrac * v);
            if (!(vol <= 0.0)) {
                k = 1;
                nr = (float)pow(vol / kSphere, 1.0 / 3.0);
                kept++;
            }
        }
        keep[o] = k;
        new_r[o] = nr;
    }
    const unsigned long long t = block_total(kept);
    if (threadIdx.x == 0 && t) atomicAdd(nkept, t);
}

__global__ void k_merge_clear(unsigned long long *__restrict__ a, int n)
{
    if ((int)threadIdx.x < n) a[threadIdx.x] = 0;
}

struct I32ToI64 {
    __device__ __forceinline__ int64_t operator()(const int32_t &v) const { return (int64_t)v; }
};

// arrays of one call, carved out of a context buffer
struct Carve {
    char *p;
    size_t used = 0;
    template <class T> T *get(size_t n)
    {
        T *a = (T *)(p + used);
        used += (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~(size_t)255;
        return a;
    }
};

// a grid over the extents e with about kCellsPerHalo cells a halo
static void merge_grid(MergeGeo &G, const double (&e)[3], int64_t n)
{
    const double L = std::max(e[0], std::max(e[1], e[2]));
    G.inv = 0.0;
    G.nc[0] = G.nc[1] = G.nc[2] = 1;
    if (!(L > 0)) return;
    // a flat or linear catalogue counts as a cell of the finest grid thick
    double v = 1.0;
    for (int q = 0; q < 3; q++) v *= std::max(e[q] / L, 1.0 / kMergeAxis);
    const double most = (double)std::min<int64_t>(2 * kCellsPerHalo * n + 64, kMergeCells);
    for (double c = std::max(cbrt(v / ((double)n * kCellsPerHalo)), 1.0 / kMergeAxis);; c *= 1.25) {  // cell size over L
        double cells = 1.0;
        for (int q = 0; q < 3; q++) {
            G.nc[q] = std::min(kMergeAxis, std::max(1, (int)ceil(e[q] / L / c)));
            cells *= G.nc[q];
        }
        G.inv = 1.0 / (c * L);
        if (cells <= most) return;
    }
}

static int grid_n(pp_ctx *ctx, int64_t n, int block = 256)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>((n + block - 1) / block, (int64_t)ctx->num_cu * 16));
}

__global__ void k_fill_i64(int64_t *__restrict__ a, int64_t n, int64_t v)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) a[i] = v;
}

// off[0] = 0, off[q + 1] = counts[0] + ... + counts[q]; *total = off[n]
template <class It>
static int offsets(pp_ctx *ctx, It counts, int64_t *off, int64_t n, int64_t *total)
{
    hipLaunchKernelGGL(k_fill_i64, dim3(1), dim3(64), 0, ctx->stream, off, (int64_t)1, (int64_t)0);
    PP_HIP(hipGetLastError());
    size_t tmp = 0;
    PP_HIP(hipcub::DeviceScan::InclusiveSum(nullptr, tmp, counts, off + 1, (int)n, ctx->stream));
    PP_CHECK(ctx->d_cub.grow(tmp));
    PP_HIP(hipcub::DeviceScan::InclusiveSum(ctx->d_cub.ptr, tmp, counts, off + 1, (int)n, ctx->stream));
    PP_HIP(hipMemcpyAsync(total, off + n, sizeof(int64_t), hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

}  // namespace pp

using namespace pp;

extern "C" int pp_merge_halos(pp_ctx *ctx, int64_t n, const float *x, const float *y, const float *z,
                              const float *rthl, int on_device, int8_t *keep, float *new_rthl, int64_t *nkept)
{
    PP_ARG(ctx && x && y && z && rthl && keep && new_rthl && nkept, "NULL argument");
    PP_ARG(n >= 0 && n < (1ll << 31), "halo count %lld outside [0, 2^31)", (long long)n);
    *nkept = 0;
    if (n == 0) return PP_OK;
    PP_CHECK(ensure_device(ctx));
    hipStream_t s = ctx->stream;
    MergeIn H;
    H.n = n;
    if (on_device) {
        H.x = x;
        H.y = y;
        H.z = z;
        H.r = rthl;
    } else {
        PP_CHECK(ctx->d_merge_in.grow(4 * (size_t)n * sizeof(float)));
        float *d = ctx->d_merge_in.as<float>();
        const float *src[4] = {x, y, z, rthl};
        for (int q = 0; q < 4; q++) PP_HIP(hipMemcpyAsync(d + q * n, src[q], n * 4, hipMemcpyHostToDevice, s));
        H.x = d;
        H.y = d + n;
        H.z = d + 2 * n;
        H.r = d + 3 * n;
    }
    int8_t *d_keep = keep;
    float *d_nr = new_rthl;
    int32_t *cell, *iota, *cell_s, *id, *first, *cnt, *state;
    int64_t *off;
    float4 *h0, *h;
    double *caps, *d_b;
    float *d_part;
    unsigned long long *frac, *d_num;  // d_num: pairs, halos kept, round with undecided halos
    MergeGeo G{};
    int64_t ncell = std::min<int64_t>(2 * kCellsPerHalo * n + 64, kMergeCells);
    const auto layout = [&](Carve W) {
        cell = W.get<int32_t>(n);
        iota = W.get<int32_t>(n);
        cell_s = W.get<int32_t>(n);
        id = W.get<int32_t>(n);
        first = W.get<int32_t>(ncell + 1);
        cnt = W.get<int32_t>(n);
        state = W.get<int32_t>(n);
        off = W.get<int64_t>(n + 1);
        h0 = W.get<float4>(n);
        h = W.get<float4>(n);
        caps = W.get<double>(n);
        frac = W.get<unsigned long long>(n);
        d_b = W.get<double>(7);
        d_num = W.get<unsigned long long>(3);
        d_part = W.get<float>(7 * kBoundBlocks);
        if (!on_device) {
            d_keep = W.get<int8_t>(n);
            d_nr = W.get<float>(n);
        }
        return W.used;
    };
    PP_CHECK(ctx->d_merge.grow(layout(Carve{nullptr})));
    layout(Carve{ctx->d_merge.as<char>()});
    // domain (Merger.jl:40-50)
    double hb[7];
    const int nb = (int)std::min<int64_t>(kBoundBlocks, (n + 255) / 256);
    hipLaunchKernelGGL(k_merge_bounds, dim3(nb), dim3(256), 0, s, H, d_part);
    hipLaunchKernelGGL(k_merge_bounds2, dim3(1), dim3(256), 0, s, (const float *)d_part, nb, d_b);
    hipLaunchKernelGGL(k_merge_clear, dim3(1), dim3(64), 0, s, d_num, 3);
    PP_HIP(hipGetLastError());
    PP_HIP(hipMemcpyAsync(hb, d_b, sizeof(hb), hipMemcpyDeviceToHost, s));
    PP_HIP(hipStreamSynchronize(s));
    for (int q = 0; q < 7; q++) PP_ARG(std::isfinite(hb[q]), "non-finite position or radius in the catalogue");
    const double pad = 2.0 * hb[6];
    const double lo[3] = {hb[0] - pad, hb[2] - pad, hb[4] - pad}, hi[3] = {hb[1] + pad, hb[3] + pad, hb[5] + pad};
    PP_ARG(std::max(hi[0] - lo[0], std::max(hi[1] - lo[1], hi[2] - lo[2])) > 0, "degenerate catalogue extent");
    const double ext[3] = {hb[1] - hb[0], hb[3] - hb[2], hb[5] - hb[4]};
    for (int q = 0; q < 3; q++) G.o[q] = hb[2 * q];
    merge_grid(G, ext, n);
    ncell = (int64_t)G.nc[0] * G.nc[1] * G.nc[2];
    int bits = 1;
    while ((1ll << bits) < ncell) bits++;
    // halos in cell order, the first of every cell
    hipLaunchKernelGGL(k_merge_keys, dim3(grid_n(ctx, n)), dim3(256), 0, s, H, G, h0, cell, iota);
    PP_HIP(hipGetLastError());
    size_t tmp = 0;
    PP_HIP(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp, cell, cell_s, iota, id, (int)n, 0, bits, s));
    PP_CHECK(ctx->d_cub.grow(tmp));
    PP_HIP(hipcub::DeviceRadixSort::SortPairs(ctx->d_cub.ptr, tmp, cell, cell_s, iota, id, (int)n, 0, bits, s));
    hipLaunchKernelGGL(k_merge_gather, dim3(grid_n(ctx, n)), dim3(256), 0, s, (const float4 *)h0, n,
                       (const int32_t *)id, h, cnt, state, frac);
    hipLaunchKernelGGL(k_cell_first, dim3(grid_n(ctx, ncell + 1)), dim3(256), 0, s, (const int32_t *)cell_s, n, ncell, first);
    PP_HIP(hipGetLastError());
    const MergeCells C{h, id, first, n};
    // pass 1: killer edges by target, then rounds
    const int gk = grid_n(ctx, n * kKillLanes);
    hipLaunchKernelGGL(k_killers<false>, dim3(gk), dim3(256), 0, s, C, G, cnt, (const int64_t *)nullptr,
                       (int32_t *)nullptr);
    PP_HIP(hipGetLastError());
    int64_t nedge = 0;
    {
        hipcub::TransformInputIterator<int64_t, I32ToI64, const int32_t *> it(cnt, I32ToI64());
        PP_CHECK(offsets(ctx, it, off, n, &nedge));
    }
    PP_CHECK(ctx->d_merge_edges.grow((size_t)std::max<int64_t>(nedge, 1) * sizeof(int32_t)));
    int32_t *edges = ctx->d_merge_edges.as<int32_t>();
    hipLaunchKernelGGL(k_killers<true>, dim3(gk), dim3(256), 0, s, C, G, cnt, (const int64_t *)off, edges);
    PP_HIP(hipGetLastError());
    // a few rounds for every look at what is left; a round too many changes nothing
    constexpr int kRounds = 4;
    int32_t *d_und = (int32_t *)(d_num + 2);
    for (int64_t round = 0;; round += kRounds) {
        PP_ARG(round <= n, "exclusion rounds did not settle");
        int32_t last = 0;
        for (int q = 1; q <= kRounds; q++)
            hipLaunchKernelGGL(k_decide, dim3(grid_n(ctx, n)), dim3(256), 0, s, n, (const int64_t *)off,
                               (const int32_t *)edges, state, h, d_und, (int32_t)(round + q));
        PP_HIP(hipGetLastError());
        PP_HIP(hipMemcpyAsync(&last, d_und, 4, hipMemcpyDeviceToHost, s));
        PP_HIP(hipStreamSynchronize(s));
        if (last != (int32_t)(round + kRounds)) break;
    }
    // pass 2: caps of overlapping survivors, then the radii they leave
    hipLaunchKernelGGL(k_pairs, dim3(grid_n(ctx, n * kPairLanes)), dim3(256), 0, s, C, G, caps, frac, d_num);
    hipLaunchKernelGGL(k_finalize, dim3(std::min(grid_n(ctx, n), ctx->num_cu * 4)), dim3(256), 0, s, C, (const int32_t *)state,
                       (const unsigned long long *)d_num, (const double *)caps, (const unsigned long long *)frac, d_keep, d_nr, d_num + 1);
    PP_HIP(hipGetLastError());
    unsigned long long num[2];
    PP_HIP(hipMemcpyAsync(num, d_num, sizeof(num), hipMemcpyDeviceToHost, s));
    PP_HIP(hipStreamSynchronize(s));
    PP_ARG(num[0] < (1ull << 31), "too many overlapping pairs (%llu)", num[0]);
    if (!on_device) {
        PP_HIP(hipMemcpyAsync(keep, d_keep, n, hipMemcpyDeviceToHost, s));
        PP_HIP(hipMemcpyAsync(new_rthl, d_nr, n * 4, hipMemcpyDeviceToHost, s));
        PP_HIP(hipStreamSynchronize(s));
    }
    *nkept = (int64_t)num[1];
    return PP_OK;
}
