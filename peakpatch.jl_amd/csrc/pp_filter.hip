// pp_filter.hip -- k-space filter-bank multiply, rocFFT transforms and the
// 27-point local-maximum peak stencil.
//
// Reference: smooth_field (src/HaloFinder/Filters.jl:79-106), find_peaks
// (src/HaloFinder/PeakFind.jl:15-78), driver loop (src/Pipeline.jl:160-195,
// src/MultiResolution.jl:885-907), GPU counterpart peak_find_tile_gpu
// (ext/CUDAExt.jl:2959-3197).
//
// Design:
//  * window multiply: one pass over the complex half-spectrum, |k| and W in
//    Float64 (the top-hat cancels badly at small kR in Float32), product in
//    Float32 as the reference.  The 1/n^3 of the normalised irfft is folded
//    into the same pass (a power of two for power-of-two n, so bit-identical
//    to scaling after the transform).
//  * stencil: the inner cube is linearised k-outer / j / i-inner, exactly the
//    CPU loop order; pass 1 tests the cells into a bit mask (wave ballots) and
//    counts them by tile and plane, pass 2 writes each peak at the sum of the
//    counts before it.  The output order is therefore the CPU order,
//    deterministic, with no atomics.  The cap of max_peaks per filter
//    (PeakFind.jl:70-72) drops the tail of that order and masks only the kept
//    peaks, as the CPU early return does.
//  * the k^2 field at the peaks: line transforms (pp_fft.h) as far as the
//    peaks need them, on a second stream.
#include <cmath>
#include <mutex>

#include "pp_common.h"
#include "pp_fields.h"
#include "pp_noise.h"

namespace pp {

// ------------------------------------------------------------- window
// W depends on |k| only through kx^2 + ky^2 + kz^2 with kx = dk ix,
// ky = dk fy, kz = dk fz; negating fy or fz is exact, so the four elements
// (ix, +-fy, +-fz) share one Float64 evaluation bit for bit.  A thread takes
// one (ix, |fy|, |fz|) and scales its (up to) four mirror elements; the grid
// is (ix, |fy|) linearised in x and |fz| in y.  With two windows the thread
// reads each element once and writes both products.
struct WinSel {
    float2 *out;
    int wsmooth;  // PP_WINDOW_*; < 0: no output
    int pitch;    // elements of a row and of a plane of out
    size_t plane;
};

__device__ __forceinline__ double window_value(int wsmooth, double k, double fkR)
{
    if (wsmooth == PP_WINDOW_GAUSSIAN) {
        double t = fkR / 2.0;
        return exp(-(t * t) / 2.0);
    }
    if (wsmooth == PP_WINDOW_K2GAUSS) {
        double t = fkR / 2.0;
        return exp(-(t * t) / 2.0) * (k * k);
    }
    double s, c;
    sincos(fkR, &s, &c);
    return 3.0 * (s - fkR * c) / (fkR * fkR * fkR);
}

// a filter's window multiplication: gx x gz workgroups
struct WinJob {
    const float2 *in;
    WinSel a, b;
    int n, nk;
    double dk, Rf;
    float scale;
    int gx, gz;
};

__device__ __forceinline__ void window_block(const WinJob &J, int bx, int hz)
{
#pragma clang fp contract(off)
    const float2 *__restrict__ in = J.in;
    const WinSel &a = J.a, &b = J.b;
    const int n = J.n, nk = J.nk;
    const double dk = J.dk, Rf = J.Rf;
    const float scale = J.scale;
    const int half = n / 2;
    const int idx = bx * 256 + threadIdx.x;
    const int hy = idx / nk;
    const int ix = idx - hy * nk;
    if (hy > half) return;
    const int iy2 = hy == 0 ? 0 : n - hy, iz2 = hz == 0 ? 0 : n - hz;
    const int ny = iy2 == hy ? 1 : 2, nz = iz2 == hz ? 1 : 2;
    // the (up to) four elements are loaded before the Float64 window is
    // evaluated, so their latency hides behind it
    float2 vin[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int iy = (q & 1) ? iy2 : hy, iz = (q & 2) ? iz2 : hz;
        if ((q & 1) < ny && (q >> 1) < nz)
            vin[q] = in[(size_t)ix + (size_t)nk * ((size_t)iy + (size_t)n * (size_t)iz)];
    }
    const double kx = dk * (double)ix, ky = dk * (double)hy, kz = dk * (double)hz;
    const double k = sqrt(kx * kx + ky * ky + kz * kz);
    const double fkR = k * Rf;
    float wa = 1.f, wb = 1.f;
    const bool scaled = fkR != 0.0;
    if (scaled) {
        wa = (float)window_value(a.wsmooth, k, fkR);
        if (b.wsmooth >= 0) wb = (float)window_value(b.wsmooth, k, fkR);
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
        if ((q & 1) >= ny || (q >> 1) >= nz) continue;
        {
            const int iy = (q & 1) ? iy2 : hy, iz = (q & 2) ? iz2 : hz;
            const float2 v = vin[q];
            float2 r = v;
            if (scaled) { r.x = r.x * wa; r.y = r.y * wa; }
            r.x = r.x * scale;
            r.y = r.y * scale;
            a.out[ix + (size_t)a.pitch * iy + a.plane * iz] = r;
            if (b.wsmooth >= 0) {
                float2 s = v;
                if (scaled) { s.x = s.x * wb; s.y = s.y * wb; }
                s.x = s.x * scale;
                s.y = s.y * scale;
                b.out[ix + (size_t)b.pitch * iy + b.plane * iz] = s;
            }
        }
    }
}

__global__ void __launch_bounds__(256) k_window(WinJob J) { window_block(J, blockIdx.x, blockIdx.y); }

static int window_job(const void *in, void *out_a, int ws_a, const FftLayout *lay_a, void *out_b, int ws_b, int n,
                      double boxsize, double Rf, float scale, WinJob *J)
{
    const int nk = n / 2 + 1, half = n / 2;
    const long long per = (long long)nk * (half + 1);
    PP_ARG(per < (1ll << 31) && half + 1 <= 65535, "mesh %d too large for the window grid", n);
    const size_t plane = (size_t)nk * n;
    *J = WinJob{(const float2 *)in,
                {(float2 *)out_a, ws_a, lay_a ? lay_a->pitch : nk, lay_a ? lay_a->plane : plane},
                {(float2 *)out_b, out_b ? ws_b : -1, nk, plane},
                n, nk, 2.0 * M_PI / boxsize, Rf, scale, (int)((per + 255) / 256), half + 1};
    return PP_OK;
}

static int launch_window(pp_ctx *ctx, const WinJob &J)
{
    hipLaunchKernelGGL(k_window, dim3(J.gx, J.gz), dim3(256), 0, ctx->stream, J);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

static int launch_window(pp_ctx *ctx, const void *in, void *out, int n, double boxsize, double Rf,
                         int wsmooth, float scale)
{
    WinJob J;
    PP_CHECK(window_job(in, out, wsmooth, nullptr, nullptr, -1, n, boxsize, Rf, scale, &J));
    return launch_window(ctx, J);
}

// ------------------------------------------------------------- stencil
// One pass over the field per filter.  A workgroup takes a 64 x 16 tile of
// inner (x, y) columns and marches along z through kz planes: each
// plane's (64+2) x (16+2) neighbourhood is staged in LDS, two planes per
// barrier (four buffers), every column keeps the 3x3 (x, y) maxima of planes
// z-1, z, z+1 in registers, and the strict
// 27-point test "no neighbour above ff" is ff >= max of the 27 values.  A
// wave is one x-run of 64 cells of one row, so its ballot of accepted cells
// is one 64-bit word of the row's peak bit mask.  The mask byte is read only
// for cells that pass the field test.
//
// A second, small pass turns the bit mask into the output: the rank of a set
// bit is the exclusive sum of the words' popcounts in (k, j, x) order, the CPU
// loop's (k outer, j, i inner), the first max_peaks ranks are kept
// (PeakFind.jl:70-72) and only the kept peak cells are masked.  The first pass
// leaves every tile's count per plane; a plane's tiles of equal y are a run of
// words, so that a workgroup of the second pass, which takes a few runs, gets
// its first rank from one sum over the counts before (over their sums by
// workgroup where there are many), and no scan is launched between.  Scan,
// emission and bookkeeping were four launches of 15.4 us a filter at 128^3 and
// 23 us at 200^3; one of 4.2 and 8.1 us now, and the filter bank there is
// bound by the launches left (about 10 us of host each).
//
// Tiles are numbered x fastest, then y, then z, and handed out so that each
// XCD (workgroups go round-robin to the eight XCDs, each with its own L2)
// works through one contiguous run of them: neighbouring tiles share their
// halo rows and planes, and those lines are then read from HBM once per run
// instead of once per tile.
constexpr int kStencilBlock = 512;
constexpr int kStencilTY = 16;  // rows of the tile: each wave takes two, 8 apart
// Planes of a tile: most for a large grid (each tile reads two planes more
// than it tests), fewer while the tiles would leave CUs idle.
// k_peak_bits at 128^3 (an inner cube of 100^3): 21.6 us with 32 planes (56
// tiles), 8.3 with 8, 5.5 with 4, 5.6 with 2; at 200^3 24.5 with 32, 18 with a
// threshold of one tile a CU, 13.1 with three, 14 with six; from 384^3 on 32.
constexpr int kStencilKZ = 32, kStencilKZMin = 4;
constexpr int kStencilTilesPerCU = 3;
constexpr int kStencilXCD = 8;
constexpr int kEmitBlocks = 4096;    // at most, doubling the runs of one
constexpr int kEmitCounts = 1 << 14; // counts up to which k_peak_emit adds them up itself

struct StencilTiles {
    int nbx, nby, nbz, per_xcd;  // tiles along x, y, z; tiles per XCD run
    int kz;                      // planes of a tile
    int runs, nruns, per;        // (plane, tile row) runs of a workgroup and of all; counts of a workgroup
};

struct StencilGeom {
    int n1, n2, n3, nbuff;
    int in1, in2, in3;
    int words;            // 64-bit words per inner row, ceil(in1 / 64)
    long long nwords;     // words * in2 * in3
};

static StencilGeom stencil_geom(int n1, int n2, int n3, int nbuff)
{
    StencilGeom g;
    g.n1 = n1; g.n2 = n2; g.n3 = n3; g.nbuff = nbuff;
    g.in1 = std::max(0, n1 - 2 * nbuff);
    g.in2 = std::max(0, n2 - 2 * nbuff);
    g.in3 = std::max(0, n3 - 2 * nbuff);
    g.words = (g.in1 + 63) / 64;
    g.nwords = (long long)g.words * g.in2 * g.in3;
    return g;
}

// The staged (64+2) x (8+2) neighbourhood of a plane is 660 floats, three
// per thread at most.  Each thread's loads for plane z+3 are issued right
// after it stages plane z+1 (two planes in flight per thread), so the HBM
// latency hides behind the barrier and the comparisons of the planes
// between.
__global__ void __launch_bounds__(kStencilBlock) k_peak_bits(const float *__restrict__ d,
                                                             const int8_t *__restrict__ mask, StencilGeom g,
                                                             StencilTiles tl, float fcrit, uint64_t *__restrict__ bits,
                                                             int *__restrict__ counts)
{
    constexpr int LX = 64 + 2, LY = kStencilTY + 2, LN = LX * LY, NQ = (LN + kStencilBlock - 1) / kStencilBlock;
    __shared__ int found[kStencilKZ][kStencilBlock / 64];
    __shared__ float tile[4][LN];  // two pairs of planes: one pair staged while the other is read
    const int t = (int)(blockIdx.x % kStencilXCD) * tl.per_xcd + (int)(blockIdx.x / kStencilXCD);
    if (t >= tl.nbx * tl.nby * tl.nbz) return;  // the whole workgroup leaves before any barrier
    const int tbx = t % tl.nbx, tby = (t / tl.nbx) % tl.nby, tbz = t / (tl.nbx * tl.nby);
    const int lane = threadIdx.x & 63, wy = threadIdx.x >> 6;
    const int x0 = g.nbuff + 64 * tbx, y0 = g.nbuff + kStencilTY * tby;
    const int z0 = g.nbuff + tl.kz * tbz;
    const int z1 = min(z0 + tl.kz, g.nbuff + g.in3);  // planes z0..z1-1; z0-1..z1 are read
    const long long s12 = (long long)g.n1 * g.n2;
    const int x = x0 + lane;
    const int ya = y0 + wy, yb = ya + kStencilTY / 2;
    const bool xin = x < g.nbuff + g.in1;
    const bool ina = xin && ya < g.nbuff + g.in2, inb = xin && yb < g.nbuff + g.in2;
    // the plane elements each thread stages (clamped to the grid: clamped
    // cells only neighbour columns outside the inner cube)
    int off[NQ];
    bool has[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const int e = threadIdx.x + q * kStencilBlock;
        has[q] = e < LN;
        const int ly = e / LX, lx = e - ly * LX;
        const int gx = min(x0 - 1 + lx, g.n1 - 1), gy = min(y0 - 1 + ly, g.n2 - 1);
        off[q] = gx + gy * g.n1;
    }
    float ra[NQ], rb[NQ];
    auto load = [&](int z, float *r) {
        const float *p = d + (long long)z * s12;
#pragma unroll
        for (int q = 0; q < NQ; q++) r[q] = has[q] ? p[off[q]] : 0.0f;
    };
    auto store = [&](const float *r, int buf) {
#pragma unroll
        for (int q = 0; q < NQ; q++)
            if (has[q]) tile[buf][threadIdx.x + q * kStencilBlock] = r[q];
    };
    auto max9 = [&](int buf, int row, float &centre) {
        const float *t = tile[buf] + row * LX + lane;
        centre = t[LX + 1];
        float m = fmaxf(fmaxf(t[0], t[1]), t[2]);
        m = fmaxf(m, fmaxf(fmaxf(t[LX], t[LX + 1]), t[LX + 2]));
        m = fmaxf(m, fmaxf(fmaxf(t[2 * LX], t[2 * LX + 1]), t[2 * LX + 2]));
        return m;
    };
    const long long word_row = (long long)g.words * g.in2;
    float ca, cb, c1a, c1b, c2a, c2b;
    // planes z0-1 and z0 to buffers 2, 3; planes z0+1, z0+2 in flight
    load(z0 - 1, ra);
    load(z0, rb);
    store(ra, 2);
    store(rb, 3);
    load(z0 + 1, ra);
    if (z0 + 2 <= z1) load(z0 + 2, rb);
    __syncthreads();
    float pa = max9(2, wy, ca), pb = max9(2, wy + kStencilTY / 2, cb);
    float qa = max9(3, wy, ca), qb = max9(3, wy + kStencilTY / 2, cb);
    auto test = [&](int z, float c_a, float c_b, float mxa, float mxb) {
        bool ka = ina && c_a >= fcrit && !(c_a < mxa);
        bool kb = inb && c_b >= fcrit && !(c_b < mxb);
        if (ka) ka = mask[x + (long long)ya * g.n1 + (long long)z * s12] != 1;
        if (kb) kb = mask[x + (long long)yb * g.n1 + (long long)z * s12] != 1;
        const unsigned long long wa = __ballot(ka), wb = __ballot(kb);
        if (lane != 0) return;
        const long long base = (long long)(z - g.nbuff) * word_row + tbx;
        if (ya < g.nbuff + g.in2) bits[base + (long long)(ya - g.nbuff) * g.words] = wa;
        if (yb < g.nbuff + g.in2) bits[base + (long long)(yb - g.nbuff) * g.words] = wb;
        found[z - z0][wy] = __popcll(wa) + __popcll(wb);
    };
    // two planes per barrier: planes z+1, z+2 (in ra, rb) go to one pair of
    // buffers while z+3, z+4 are fetched; the pair written here was last
    // read two barriers ago
    for (int z = z0, k = 0; z < z1; z += 2, k ^= 1) {
        const int b1 = 2 * k, b2 = 2 * k + 1;
        store(ra, b1);
        if (z + 2 <= z1) store(rb, b2);
        if (z + 3 <= z1) load(z + 3, ra);
        if (z + 4 <= z1) load(z + 4, rb);
        __syncthreads();
        const float m1a = max9(b1, wy, c1a), m1b = max9(b1, wy + kStencilTY / 2, c1b);
        test(z, ca, cb, fmaxf(fmaxf(pa, qa), m1a), fmaxf(fmaxf(pb, qb), m1b));
        if (z + 1 < z1) {
            const float m2a = max9(b2, wy, c2a), m2b = max9(b2, wy + kStencilTY / 2, c2b);
            test(z + 1, c1a, c1b, fmaxf(fmaxf(qa, m1a), m2a), fmaxf(fmaxf(qb, m1b), m2b));
            pa = m1a; pb = m1b;
            qa = m2a; qb = m2b;
            ca = c2a; cb = c2b;
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < z1 - z0) {
        int sum = 0;
#pragma unroll
        for (int q = 0; q < kStencilBlock / 64; q++) sum += found[threadIdx.x][q];
        counts[((long long)(z0 - g.nbuff + threadIdx.x) * tl.nby + tby) * tl.nbx + tbx] = sum;
    }
}

struct PeakOut {
    int32_t *i, *j, *k, *filt;
    float *delta_s;
    long long capacity;
};

// before a call's first stencil
__global__ void k_stencil_clear(long long *counters, long long *base)
{
    if (threadIdx.x < 4) counters[threadIdx.x] = 0;
    if (threadIdx.x < 2) base[threadIdx.x] = 0;
}

// exclusive sum of v over the workgroup's 256 threads; *total gets the sum
__device__ __forceinline__ int block_offset(int v, int *wsum, int *total)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int s = v;
    for (int w = 1; w < 64; w <<= 1) {
        const int u = __shfl_up(s, w, 64);
        if (lane >= w) s += u;
    }
    __syncthreads();  // the sums of the call before have been read
    if (lane == 63) wsum[wave] = s;
    __syncthreads();
    int before = 0;
    for (int q = 0; q < 4; q++) before += q < wave ? wsum[q] : 0;
    *total = wsum[0] + wsum[1] + wsum[2] + wsum[3];
    return before + s - v;
}

// the counts' sums by workgroup of k_peak_emit
__global__ void __launch_bounds__(256) k_peak_sums(const int *__restrict__ counts, long long n, int per, int nsums,
                                                   int *__restrict__ sums)
{
    const int s = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (s >= nsums) return;
    const long long e = min((long long)(s + 1) * per, n);
    int sum = 0;
    for (long long q = (long long)s * per + (threadIdx.x & 63); q < e; q += 64) sum += counts[q];
    for (int w = 32; w > 0; w >>= 1) sum += __shfl_down(sum, w, 64);
    if ((threadIdx.x & 63) == 0) sums[s] = sum;
}

// counters[0] = peaks written so far (all filters), counters[1] = peaks found
// (capped per filter), counters[2] = first index of the current filter.  A
// workgroup writes the peaks of tl.runs runs; `before` holds `per` counts or
// sums for each workgroup.  The filter's first slot is base[parity]; the last
// workgroup leaves the next one in the other word (counters[0] itself would
// need every workgroup to have read it: a device-wide fence by each took 0.2
// ms at 512^3).  With WIN the workgroups from nemit on multiply the next
// filter's window, which needs nothing of this one's peaks.
template <bool WIN>
__global__ void __launch_bounds__(256) k_peak_emit(const float *__restrict__ d, int8_t *__restrict__ mask,
                                                   StencilGeom g, StencilTiles tl, const uint64_t *__restrict__ bits,
                                                   const int *__restrict__ before, int per,
                                                   long long *__restrict__ base, int parity,
                                                   long long *__restrict__ counters, long long max_peaks, int filt,
                                                   PeakOut o, long long *__restrict__ range, int nemit, WinJob J)
{
    if (WIN && (int)blockIdx.x >= nemit) {
        const int b = blockIdx.x - nemit, z = b / J.gx;
        window_block(J, b - z * J.gx, z);
        return;
    }
    __shared__ int wsum[4];
    int sum = 0, total;
    for (long long q = threadIdx.x, e = (long long)blockIdx.x * per; q < e; q += 256) sum += before[q];
    block_offset(sum, wsum, &total);
    long long first = total;  // rank of the workgroup's first peak
    const long long b0 = base[parity];
    auto word = [&](int run) {  // the run's first word
        const int z = run / tl.nby, ty = run - z * tl.nby;
        return ((long long)z * g.in2 + (long long)ty * kStencilTY) * g.words;
    };
    const int run1 = min((int)(blockIdx.x + 1) * tl.runs, tl.nruns);
    const long long w0 = word(blockIdx.x * tl.runs), w1 = run1 < tl.nruns ? word(run1) : g.nwords;
    for (long long w = w0 + threadIdx.x; w - (int)threadIdx.x < w1; w += 256) {
        uint64_t b = w < w1 ? bits[w] : 0;
        long long rank = first + block_offset(__popcll(b), wsum, &total);
        first += total;
        const long long row = w / g.words;
        const int wx = (int)(w - row * g.words);
        const int j = g.nbuff + (int)(row % g.in2), k = g.nbuff + (int)(row / g.in2);
        for (; b && rank < max_peaks; b &= b - 1, rank++) {
            const int i = g.nbuff + 64 * wx + __ffsll((unsigned long long)b) - 1;
            const long long c = i + (long long)j * g.n1 + (long long)k * g.n1 * g.n2;
            mask[c] = 1;
            const long long slot = b0 + rank;
            if (slot < o.capacity) {
                o.i[slot] = i;
                o.j[slot] = j;
                o.k[slot] = k;
                o.filt[slot] = filt;
                o.delta_s[slot] = d[c];
            }
        }
    }
    if ((int)blockIdx.x == nemit - 1 && threadIdx.x == 0) {
        const long long kept = first < max_peaks ? first : max_peaks;  // first: all of the filter's peaks
        base[parity ^ 1] = b0 + kept;
        counters[0] = b0 + kept;
        counters[1] += kept;
        counters[2] = b0;
        if (range) {  // this filter's peaks, for work that follows on another stream
            range[0] = b0;
            range[1] = b0 + kept;
        }
    }
}

// a filter's stencil over an empty inner cube
__global__ void k_stencil_none(long long *__restrict__ counters, long long *__restrict__ range)
{
    counters[2] = counters[0];
    if (range) range[0] = range[1] = counters[0];
}

__global__ void k_sample_field(const float *__restrict__ f, int n1, int n2, const int32_t *__restrict__ pi,
                               const int32_t *__restrict__ pj, const int32_t *__restrict__ pk,
                               float *__restrict__ out, const long long *__restrict__ counters,
                               long long capacity)
{
    long long lo = counters[2], hi = counters[0];
    if (hi > capacity) hi = capacity;
    for (long long s = lo + (long long)blockIdx.x * blockDim.x + threadIdx.x; s < hi;
         s += (long long)gridDim.x * blockDim.x)
        out[s] = f[pi[s] + (long long)pj[s] * n1 + (long long)pk[s] * n1 * n2];
}

// Device scratch of a call's stencils, carved from one buffer: the peak bit
// mask, the tiles' counts (as many as words at most), their sums, the slots.
struct StencilScratch {
    uint64_t *bits;
    int *counts, *sums;
    long long *base;
};

static size_t align256(size_t b) { return (b + 255) & ~(size_t)255; }

static size_t stencil_scratch_bytes(const StencilGeom &g)
{
    return align256((size_t)g.nwords * 8) + align256((size_t)g.nwords * 4) + align256(kEmitBlocks * sizeof(int)) + 256;
}

static StencilScratch stencil_carve(void *base, const StencilGeom &g)
{
    StencilScratch s;
    char *p = (char *)base;
    s.bits = (uint64_t *)p;
    p += align256((size_t)g.nwords * 8);
    s.counts = (int *)p;
    p += align256((size_t)g.nwords * 4);
    s.sums = (int *)p;
    p += align256(kEmitBlocks * sizeof(int));
    s.base = (long long *)p;
    return s;
}

// before a call's first stencil: a kernel rather than a memset node, so that
// a caller may capture the call in a HIP graph
static int stencil_clear(pp_ctx *ctx, const StencilScratch &s, long long *d_counters)
{
    hipLaunchKernelGGL(k_stencil_clear, dim3(1), dim3(64), 0, ctx->stream, d_counters, s.base);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

// Stencil over one field, the step-th of a call; peaks appended after
// counters[0].  The last launch also does the window of `next`: one launch less
// a filter, which takes ten filters at 128^3, bound by the host, from 0.90 to
// 0.84 ms and costs nothing at 512^3.
static int run_stencil(pp_ctx *ctx, const float *d_field, int8_t *d_mask, const StencilGeom &g,
                       float fcrit, long long max_peaks, int step, const PeakOut &o, long long *d_counters,
                       const StencilScratch &s, long long *range = nullptr, const WinJob *next = nullptr)
{
    PP_ARG(g.nwords < (1ll << 31), "inner cube too large for the stencil");
    if (g.nwords == 0) {
        hipLaunchKernelGGL(k_stencil_none, dim3(1), dim3(1), 0, ctx->stream, d_counters, range);
        PP_HIP(hipGetLastError());
        return next ? launch_window(ctx, *next) : PP_OK;
    }
    StencilTiles tl;
    tl.nbx = g.words;
    tl.nby = (g.in2 + kStencilTY - 1) / kStencilTY;
    long long ntiles = 0;
    for (tl.kz = kStencilKZ;; tl.kz /= 2) {
        tl.nbz = (g.in3 + tl.kz - 1) / tl.kz;
        ntiles = (long long)tl.nbx * tl.nby * tl.nbz;
        if (tl.kz <= kStencilKZMin || ntiles >= (long long)kStencilTilesPerCU * ctx->num_cu) break;
    }
    PP_ARG(ntiles < (1ll << 30), "inner cube too large for the stencil grid");
    tl.per_xcd = (int)((ntiles + kStencilXCD - 1) / kStencilXCD);
    tl.nruns = g.in3 * tl.nby;
    const long long ncounts = (long long)tl.nruns * tl.nbx;
    for (tl.runs = std::max(1, 256 / (kStencilTY * g.words)); (tl.nruns + tl.runs - 1) / tl.runs > kEmitBlocks;)
        tl.runs *= 2;
    const int blocks = (tl.nruns + tl.runs - 1) / tl.runs;
    tl.per = tl.runs * tl.nbx;
    hipLaunchKernelGGL(k_peak_bits, dim3((unsigned)tl.per_xcd * kStencilXCD), dim3(kStencilBlock), 0, ctx->stream,
                       d_field, (const int8_t *)d_mask, g, tl, fcrit, s.bits, s.counts);
    PP_HIP(hipGetLastError());
    const bool sums = ncounts > kEmitCounts;
    if (sums) {
        hipLaunchKernelGGL(k_peak_sums, dim3((blocks + 3) / 4), dim3(256), 0, ctx->stream, (const int *)s.counts,
                           ncounts, tl.per, blocks, s.sums);
        PP_HIP(hipGetLastError());
    }
    auto emit = [&](auto kern, long long more) {
        hipLaunchKernelGGL(kern, dim3((unsigned)(blocks + more)), dim3(256), 0, ctx->stream, d_field, d_mask, g, tl,
                           (const uint64_t *)s.bits, (const int *)(sums ? s.sums : s.counts), sums ? 1 : tl.per, s.base,
                           step & 1, d_counters, max_peaks, step, o, range, blocks, next ? *next : WinJob{});
    };
    if (next) emit(k_peak_emit<true>, (long long)next->gx * next->gz);
    else emit(k_peak_emit<false>, 0);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

// the state of a call's stencils in the context's scratch, cleared
static int stencil_start(pp_ctx *ctx, const StencilGeom &g, long long *d_counters, StencilScratch &s)
{
    PP_CHECK(ctx->d_scan.grow(stencil_scratch_bytes(g)));
    s = stencil_carve(ctx->d_scan.ptr, g);
    return stencil_clear(ctx, s, d_counters);
}

// ------------------------------------------- the k^2 field at the peaks
// With want_lapd every filter's k^2-Gaussian field is wanted at its new peaks
// only.  Its inverse transform (rocFFT: 1.46 ms at 512^3, after half of
// k_window's 0.31 ms) is done on line transforms (pp_fft.h) instead, as far as
// the peaks need it: the window goes into the z pass, planes and rows outside
// the inner cube are not written, modes whose window is zero in Float32 are not
// read, and only the row pairs that hold a peak are transformed along x, from
// where the peaks' values are taken without a field.  The passes run on the
// side stream beside the next filters' rocFFT kernels, which leave most of
// HBM's bandwidth free; only the last waits for its filter's stencil.
// pp_smooth_field with wsmooth = 3 takes the same passes over the whole grid
// and every mode, so both give the same bits (the peaks' spectrum is finite: a
// field with other modes has no peaks).
// Odd meshes stay with rocFFT, which rounds less in them (rms error at 25, 45,
// 81, 125, 135: 1.28, 1.22, 1.44, 1.43, 1.39e-7 against 1.37, 1.55, 1.66, 1.70,
// 1.78 on the lines; even ones, 64, 120, 128: 1.71, 1.73, 1.88 against 1.42,
// 1.66, 1.56).
static bool bank_lines(int n) { return n % 2 == 0 && line_supported(n); }

struct BankGeo {
    int n, lo, hi;      // planes [lo, hi)
    int ylo, yhi;       // rows [ylo, yhi): the inner ones and their partners in row pairs
    int cut;            // modes |i| > cut on any axis are left out
    int plain;          // radius 0: no window
    double mult2;       // k^2 = mult2 |i|^2
    float scale;
    const double *gauss; // exp(-(k Rf)^2 / 8) by index, n / 2 + 1
};

// exp(-(i dk R)^2 / 8) of every filter
__global__ void k_gauss_table(const double *__restrict__ Rf, int nfilt, int count, double dk, double *__restrict__ out)
{
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nfilt * count; t += gridDim.x * blockDim.x) {
        const int f = t / count, i = t - f * count;
        const double x = (double)i * dk * Rf[f] / 2.0;
        out[t] = exp(-(x * x) / 2.0);
    }
}

// rocFFT's spectrum (rows of n / 2 + 1) into rows of whole 128-byte lines
__global__ void __launch_bounds__(256) k_repack(const float2 *__restrict__ in, SpecGeo g, float2 *__restrict__ out)
{
    const long long rows = (long long)g.n * g.n;
    for (long long r = (long long)blockIdx.x * 4 + threadIdx.x / 64; r < rows; r += (long long)gridDim.x * 4) {
        const int z = (int)(r / g.n);
        const float2 *a = in + r * g.nk;
        float2 *b = out + g.row(z, (int)(r - (long long)z * g.n));
        for (int k = threadIdx.x % 64; k < g.nk; k += 64) b[k] = a[k];
    }
}

template <int M>
__global__ void __launch_bounds__(1024) k_bank_z(SpecGeo g, LineFft P, ColGrid C, BankGeo B,
                                                 const float2 *__restrict__ in, float2 *__restrict__ out)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    // the tile grid counts the rows |fy| <= cut: 0 .. cut, then -cut .. -1
    const int n = g.n, iy = t.plane <= B.cut || 2 * B.cut + 1 > n ? t.plane : n - (2 * B.cut + 1 - t.plane);
    const int fy = iy < (n + 1) / 2 ? iy : iy - n, ay = abs(fy), kx = min(t.kx, g.nk - 1), ixy = kx * kx + fy * fy;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const LineZ src(g, in, iy, t.kx);
    const double gxy = B.gauss[kx] * B.gauss[ay] * B.mult2;
    float2 X[kLineEpt];
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = min(t.jj + q * P.tj, n - 1), fz = e < (n + 1) / 2 ? e : e - n, az = abs(fz);
        X[q] = make_float2(0.f, 0.f);
        if (az <= B.cut) {
            const float2 v = *src.at(e);
            const int i2 = ixy + fz * fz;
            // the window in Float64, rounded once, as window_value's; k = 0: none
            const float f = i2 == 0 || B.plain ? 1.f : (float)(gxy * B.gauss[az] * (double)i2);
            X[q] = make_float2(v.x * f * B.scale, v.y * f * B.scale);
        }
    }
    line_run<1, M, false, false>(at, P, t.jj, X);
    const LineZ dst(g, out, iy, t.kx);
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = t.jj + q * P.tj;
        if (e >= B.lo && e < B.hi) *dst.at(e) = X[q];
    }
}

template <int M>
__global__ void __launch_bounds__(1024) k_bank_y(SpecGeo g, LineFft P, ColGrid C, BankGeo B, float2 *__restrict__ s)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const int n = g.n;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const LineY io(g, s, B.lo + t.plane, 0, 1, t.kx);
    float2 X[kLineEpt];
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = min(t.jj + q * P.tj, n - 1), fy = e < (n + 1) / 2 ? e : e - n;
        X[q] = abs(fy) <= B.cut ? *io.at(e) : make_float2(0.f, 0.f);
    }
    line_run<1, M, false, false>(at, P, t.jj, X);
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = t.jj + q * P.tj;
        if (e >= B.ylo && e < B.yhi) *io.at(e) = X[q];
    }
}

// the field at the peaks [range[0], range[1]), which come in the order of
// their rows: a line looks its row pair up and, if it holds peaks, transforms
// it as k_rows_inv does
template <int M>
__global__ void __launch_bounds__(512) k_bank_rows(SpecGeo g, LineFft P, BankGeo B, const float2 *__restrict__ s,
                                                   const int32_t *__restrict__ pi, const int32_t *__restrict__ pj,
                                                   const int32_t *__restrict__ pk, float *__restrict__ out,
                                                   const long long *__restrict__ range, long long capacity)
{
    extern __shared__ float2 lds[];
    const int n = g.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    // row pairs from the one that holds the first row of plane lo
    const long long r = 2 * ((long long)B.lo * n / 2 + (long long)blockIdx.x * (blockDim.x / P.tj) + line);
    const long long hi = min(range[1], capacity);
    auto row = [&](long long p) { return (long long)pk[p] * n + pj[p]; };
    long long lo = range[0], top = hi;
    while (lo < top) {  // the first peak of row r or later
        const long long mid = (lo + top) >> 1;
        if (row(mid) < r) lo = mid + 1;
        else top = mid;
    }
    const bool has = lo < hi && row(lo) <= r + 1;
    if (!__syncthreads_or(has)) return;
    const RowAddr at(lds + line * row_pitch(n));
    if (has) load_row_pair(at, P, g, s, r, true, jj, 0, false, Two{1.f, 0.f}, B.cut);
    __syncthreads();
    float2 x[kLineEpt];
    line_run<1, M, true, true>(at, P, jj, x);
    if (!has) return;
    for (long long p = lo + jj; p < hi && row(p) <= r + 1; p += P.tj) {
        const float2 v = at(pi[p]);
        out[p] = row(p) == r ? v.x : v.y;
    }
}

// Device buffers and launch shapes of the above for one pp_find_peaks call
struct Bank {
    GridPlan G;
    BankGeo B{};
    float2 *R = nullptr, *T = nullptr;
    double *tables = nullptr;
    long long *ranges = nullptr;
    double dk = 0;
};

// spec: delta_k as rocFFT leaves it, made on the main stream; planes and rows
// [lo, hi) are wanted
static int bank_start(pp_ctx *ctx, const void *spec, int n, int lo, int hi, double boxsize, const double *Rf, int nfilt,
                      Bank &K)
{
    PP_CHECK(grid_plan(ctx, n, &K.G));
    K.G.stream = ctx->side;
    const SpecGeo &g = K.G.g;
    const int count = n / 2 + 1;
    const size_t arr = g.size(n);
    PP_CHECK(ctx->d_spec.grow(2 * arr * sizeof(float2)));
    K.R = ctx->d_spec.as<float2>();
    K.T = K.R + arr;
    PP_CHECK(ctx->d_misc.grow((size_t)nfilt * (3 + count) * sizeof(double)));
    double *d_Rf = ctx->d_misc.as<double>();
    K.ranges = (long long *)(d_Rf + nfilt);
    K.tables = (double *)(K.ranges + 2 * nfilt);
    K.dk = 2.0 * M_PI / boxsize;
    K.B.n = n;
    K.B.lo = lo;
    K.B.hi = hi;
    K.B.ylo = std::max(0, lo - 1);
    K.B.yhi = std::min(n, hi + 1);
    K.B.mult2 = K.dk * K.dk;
    K.B.scale = (float)(1.0 / ((double)n * n * n));
    PP_HIP(hipEventRecord(ctx->ev_bank, ctx->stream));
    PP_HIP(hipStreamWaitEvent(ctx->side, ctx->ev_bank, 0));
    PP_HIP(hipMemcpyAsync(d_Rf, Rf, nfilt * sizeof(double), hipMemcpyHostToDevice, ctx->side));
    hipLaunchKernelGGL(k_gauss_table, dim3((nfilt * count + 255) / 256), dim3(256), 0, ctx->side, (const double *)d_Rf,
                       nfilt, count, K.dk, K.tables);
    PP_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_repack, dim3(ctx->num_cu * 16), dim3(256), 0, ctx->side, (const float2 *)spec, g, K.R);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

// main-stream work launched next runs after the side stream's so far
static int bank_join(pp_ctx *ctx)
{
    PP_HIP(hipEventRecord(ctx->ev_bank, ctx->side));
    PP_HIP(hipStreamWaitEvent(ctx->stream, ctx->ev_bank, 0));
    return PP_OK;
}

// The largest |i| on an axis at which k^2 exp(-(k R)^2 / 8), k = dk i, may still
// be other than zero in Float32.  With u = (k R)^2 / 8 the window is
// (8 / R^2) u exp(-u), which falls beyond u = 1 and rounds to zero from 2^-150
// on: u - ln u > ln(8 / R^2) + 150 ln 2, solved by iteration, with a per cent
// of the window to spare.
static int window_reach(double dk, double R, int half)
{
    if (!(fabs(R) > 0.0)) return half;
    const double L = log(8.0) - 2.0 * log(fabs(R)) + 150.0 * M_LN2;
    double u = 1000.0;
    for (int q = 0; q < 100; q++) u = std::max(1.0, L + log(u));
    const double c = sqrt(8.0 * (u + 0.01)) / (dk * fabs(R));
    return c < half ? (int)c + 1 : half;
}

// filter f's spectrum along z and y (needs no peaks)
static int bank_transform(pp_ctx *ctx, Bank &K, const double *Rf, int f, bool every_mode)
{
    const SpecGeo &g = K.G.g;
    const int n = g.n, half = n / 2;
    K.B.gauss = K.tables + (size_t)f * (half + 1);
    K.B.cut = every_mode ? half : window_reach(K.dk, Rf[f], half);
    K.B.plain = Rf[f] == 0.0;
    const int rows = std::min(n, 2 * K.B.cut + 1), bins = std::min(K.B.cut, g.nk - 1) + 1;
    if (K.B.hi <= K.B.lo) return PP_OK;
    const ColGrid cz = K.G.cs.grid(bins, rows, kColXCD), cy = K.G.ys.grid(bins, K.B.hi - K.B.lo, 1);
    PP_LINE_LAUNCH(K.G.col, k_bank_z, dim3(cz.blocks()), dim3(K.G.cs.block), K.G.cs.lds, ctx->side, g, K.G.col, cz, K.B,
                   (const float2 *)K.R, K.T);
    PP_LINE_LAUNCH(K.G.ycol, k_bank_y, dim3(cy.blocks()), dim3(K.G.ys.block), K.G.ys.lds, ctx->side, g, K.G.ycol, cy,
                   K.B, K.T);
    return PP_OK;
}

// ... and its values at filter f's peaks, once its stencil is done
static int bank_sample(pp_ctx *ctx, Bank &K, int f, const PeakOut &o, float *d_lapd)
{
    PP_HIP(hipEventRecord(ctx->ev_bank, ctx->stream));
    PP_HIP(hipStreamWaitEvent(ctx->side, ctx->ev_bank, 0));
    if (K.B.hi <= K.B.lo) return PP_OK;
    const long long n = K.G.g.n, pairs = (n * K.B.hi + 1) / 2 - n * K.B.lo / 2;
    const LineShape &S = K.G.rs;
    PP_LINE_LAUNCH(K.G.row, k_bank_rows, dim3((unsigned)((pairs + S.nl - 1) / S.nl)), dim3(S.block), S.lds, ctx->side,
                   K.G.g, K.G.row, K.B, (const float2 *)K.T, (const int32_t *)o.i, (const int32_t *)o.j,
                   (const int32_t *)o.k, d_lapd, (const long long *)(K.ranges + 2 * f), o.capacity);
    return PP_OK;
}

// ------------------------------------------- peak finding without allocation
// pp_find_peaks_field_noalloc keeps its counters and the stencil's bit mask and
// counts in `scratch`, a file-scope array every device the
// library runs on holds until the process ends.  Host code never passes the
// array's name to a kernel: it passes the device address hipGetSymbolAddress
// gives for the current device, taken once per device when a context is
// created there (noalloc_scratch_init).
static __device__ __align__(256) unsigned char scratch[PP_NOALLOC_SCRATCH_BYTES];
// Row words of the inner cube it is for, the bound callers know (12 bytes a
// word and 17 KB of sums; 64 words less than fit).
constexpr long long kNoallocWords = 8387136;

constexpr int kMaxDevices = 64;
static std::mutex g_scratch_mu;
static void *g_scratch_ptr[kMaxDevices];

int noalloc_scratch_init(int device)
{
    PP_ARG(device >= 0 && device < kMaxDevices, "device %d beyond the %d the library tracks", device, kMaxDevices);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return PP_OK;
    void *p = nullptr;
    PP_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    PP_ARG(p != nullptr, "no device address for the scratch array");
    g_scratch_ptr[device] = p;
    return PP_OK;
}

static void *noalloc_scratch(int device)
{
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return device >= 0 && device < kMaxDevices ? g_scratch_ptr[device] : nullptr;
}

static int alloc_peak_out(pp_ctx *ctx, long long cap, PeakOut &o, float **lapd, long long **counters)
{
    size_t per = cap > 0 ? (size_t)cap : 1;
    size_t bytes = per * (4 * sizeof(int32_t) + 2 * sizeof(float)) + 4 * sizeof(long long) + 256;
    PP_CHECK(ctx->d_peaks.grow(bytes));
    char *p = ctx->d_peaks.as<char>();
    *counters = (long long *)p;
    p += 256;
    o.i = (int32_t *)p; p += per * sizeof(int32_t);
    o.j = (int32_t *)p; p += per * sizeof(int32_t);
    o.k = (int32_t *)p; p += per * sizeof(int32_t);
    o.filt = (int32_t *)p; p += per * sizeof(int32_t);
    o.delta_s = (float *)p; p += per * sizeof(float);
    *lapd = (float *)p;
    o.capacity = cap;
    return PP_OK;
}

static int download_peaks(pp_ctx *ctx, const PeakOut &o, const float *d_lapd, const long long *d_counters,
                          pp_peaks *out)
{
    long long cnt[4];
    PP_HIP(hipMemcpyAsync(cnt, d_counters, sizeof cnt, hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    long long found = cnt[1];
    long long written = found < out->capacity ? found : out->capacity;
    out->needed = found;
    out->count = written;
    if (written > 0) {
        size_t b4 = (size_t)written * 4;
        if (out->i) PP_HIP(hipMemcpyAsync(out->i, o.i, b4, hipMemcpyDefault, ctx->stream));
        if (out->j) PP_HIP(hipMemcpyAsync(out->j, o.j, b4, hipMemcpyDefault, ctx->stream));
        if (out->k) PP_HIP(hipMemcpyAsync(out->k, o.k, b4, hipMemcpyDefault, ctx->stream));
        if (out->filt) PP_HIP(hipMemcpyAsync(out->filt, o.filt, b4, hipMemcpyDefault, ctx->stream));
        if (out->delta_s)
            PP_HIP(hipMemcpyAsync(out->delta_s, o.delta_s, b4, hipMemcpyDefault, ctx->stream));
        if (out->lapd_s && d_lapd)
            PP_HIP(hipMemcpyAsync(out->lapd_s, d_lapd, b4, hipMemcpyDefault, ctx->stream));
        PP_HIP(hipStreamSynchronize(ctx->stream));
    }
    if (found > out->capacity) {
        set_error("peak output capacity %lld too small: %lld peaks found", (long long)out->capacity, found);
        return PP_ERR_CAPACITY;
    }
    return PP_OK;
}

}  // namespace pp

using namespace pp;

extern "C" {

int pp_window_multiply(pp_ctx *ctx, const void *delta_k, void *out, int on_device, int n, double boxsize,
                       double Rf, int wsmooth, float scale)
{
    PP_ARG(ctx && delta_k && out, "NULL argument");
    PP_ARG(n >= 2 && boxsize > 0, "bad n=%d / boxsize", n);
    PP_ARG(wsmooth == 0 || wsmooth == 1 || wsmooth == 3, "wsmooth %d not in {0,1,3}", wsmooth);
    PP_CHECK(ensure_device(ctx));
    size_t bytes = (size_t)(n / 2 + 1) * n * n * sizeof(float2);
    if (on_device) return launch_window(ctx, delta_k, out, n, boxsize, Rf, wsmooth, scale);
    PP_CHECK(ctx->d_k1.grow(bytes));
    PP_HIP(hipMemcpyAsync(ctx->d_k1.ptr, delta_k, bytes, hipMemcpyHostToDevice, ctx->stream));
    PP_CHECK(launch_window(ctx, ctx->d_k1.ptr, ctx->d_k1.ptr, n, boxsize, Rf, wsmooth, scale));
    PP_HIP(hipMemcpyAsync(out, ctx->d_k1.ptr, bytes, hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

int pp_rfft(pp_ctx *ctx, const float *in, void *out, int on_device, int n)
{
    PP_ARG(ctx && in && out, "NULL argument");
    PP_ARG(n >= 2, "bad n=%d", n);
    PP_CHECK(ensure_device(ctx));
    PP_CHECK(fft_prepare(ctx, n));
    size_t rb = (size_t)n * n * n * sizeof(float), cb = (size_t)(n / 2 + 1) * n * n * sizeof(float2);
    void *din = (void *)in, *dout = out;
    if (!on_device) {
        PP_CHECK(ctx->d_field_a.grow(rb));
        PP_CHECK(ctx->d_k0.grow(cb));
        PP_HIP(hipMemcpyAsync(ctx->d_field_a.ptr, in, rb, hipMemcpyHostToDevice, ctx->stream));
        din = ctx->d_field_a.ptr;
        dout = ctx->d_k0.ptr;
    }
    void *ib[1] = {din}, *ob[1] = {dout};
    PP_FFT(rocfft_execute(ctx->fftp->r2c, ib, ob, ctx->fftp->info));
    if (!on_device) PP_HIP(hipMemcpyAsync(out, dout, cb, hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

int pp_smooth_field(pp_ctx *ctx, const void *delta_k, float *out, int on_device, int n, double boxsize,
                    double Rf, int wsmooth)
{
    PP_ARG(ctx && delta_k && out, "NULL argument");
    PP_ARG(n >= 2 && boxsize > 0, "bad n=%d / boxsize", n);
    PP_ARG(wsmooth == 0 || wsmooth == 1 || wsmooth == 3, "wsmooth %d not in {0,1,3}", wsmooth);
    PP_CHECK(ensure_device(ctx));
    PP_CHECK(fft_prepare(ctx, n));
    size_t rb = (size_t)n * n * n * sizeof(float), cb = (size_t)(n / 2 + 1) * n * n * sizeof(float2);
    const void *src = delta_k;
    if (!on_device) {
        PP_CHECK(ctx->d_k0.grow(cb));
        PP_HIP(hipMemcpyAsync(ctx->d_k0.ptr, delta_k, cb, hipMemcpyHostToDevice, ctx->stream));
        src = ctx->d_k0.ptr;
    }
    float inv = (float)(1.0 / ((double)n * n * n));
    float *dst = out;
    if (!on_device) {
        PP_CHECK(ctx->d_field_a.grow(rb));
        dst = ctx->d_field_a.as<float>();
    }
    if (wsmooth == PP_WINDOW_K2GAUSS && bank_lines(n)) {
        Bank K;
        PP_CHECK(bank_start(ctx, src, n, 0, n, boxsize, &Rf, 1, K));
        PP_CHECK(bank_transform(ctx, K, &Rf, 0, true));
        XArgs X{};
        X.top = K.B.cut;
        X.add(K.T, dst, 0, false, 1.0);
        PP_CHECK(rows_inv(K.G, X));
        PP_CHECK(bank_join(ctx));
        if (!on_device) PP_HIP(hipMemcpyAsync(out, dst, rb, hipMemcpyDeviceToHost, ctx->stream));
        PP_HIP(hipStreamSynchronize(ctx->stream));
        return PP_OK;
    }
    PP_CHECK(ctx->d_k1.grow(cb));
    PP_CHECK(launch_window(ctx, src, ctx->d_k1.ptr, n, boxsize, Rf, wsmooth, inv));
    void *ib[1] = {ctx->d_k1.ptr}, *ob[1] = {dst};
    PP_FFT(rocfft_execute(ctx->fftp->c2r, ib, ob, ctx->fftp->info));
    if (!on_device) PP_HIP(hipMemcpyAsync(out, dst, rb, hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

int pp_find_peaks_field(pp_ctx *ctx, const float *delta_s, int8_t *mask, int on_device, int n1, int n2,
                        int n3, int nbuff, float fcrit, int64_t max_peaks, pp_peaks *out)
{
    PP_ARG(ctx && delta_s && mask && out, "NULL argument");
    PP_ARG(n1 >= 3 && n2 >= 3 && n3 >= 3, "grid %dx%dx%d too small", n1, n2, n3);
    PP_ARG(nbuff >= 1, "nbuff must be >= 1 (the 27-point stencil reads one cell past the inner cube)");
    PP_ARG(out->capacity >= 0, "negative capacity");
    PP_CHECK(ensure_device(ctx));
    if (max_peaks <= 0) max_peaks = 2000000;
    const StencilGeom g = stencil_geom(n1, n2, n3, nbuff);
    size_t N = (size_t)n1 * n2 * n3;
    const float *d_f = delta_s;
    int8_t *d_m = mask;
    if (!on_device) {
        PP_CHECK(ctx->d_field_a.grow(N * sizeof(float)));
        PP_CHECK(ctx->d_mask.grow(N));
        PP_HIP(hipMemcpyAsync(ctx->d_field_a.ptr, delta_s, N * sizeof(float), hipMemcpyHostToDevice, ctx->stream));
        PP_HIP(hipMemcpyAsync(ctx->d_mask.ptr, mask, N, hipMemcpyHostToDevice, ctx->stream));
        d_f = ctx->d_field_a.as<float>();
        d_m = ctx->d_mask.as<int8_t>();
    }
    PeakOut o;
    float *d_lapd;
    long long *d_counters;
    PP_CHECK(alloc_peak_out(ctx, out->capacity, o, &d_lapd, &d_counters));
    StencilScratch S;
    PP_CHECK(stencil_start(ctx, g, d_counters, S));
    PP_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    PP_CHECK(run_stencil(ctx, d_f, d_m, g, fcrit, max_peaks, 0, o, d_counters, S));
    PP_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    if (!on_device) PP_HIP(hipMemcpyAsync(mask, d_m, N, hipMemcpyDeviceToHost, ctx->stream));
    int rc = download_peaks(ctx, o, nullptr, d_counters, out);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]);
    ctx->timing.peakfind_ms = ms;
    return rc;
}

int pp_find_peaks(pp_ctx *ctx, const float *delta, int on_device, int n, double boxsize, const double *Rf,
                  const float *fcrit, int nfilt, int wsmooth, int want_lapd, int nbuff,
                  int64_t max_peaks_per_filter, int8_t *mask_inout, pp_peaks *out)
{
    PP_ARG(ctx && delta && Rf && fcrit && out, "NULL argument");
    PP_ARG(n >= 3 && boxsize > 0 && nfilt >= 0, "bad n=%d / boxsize / nfilt", n);
    PP_ARG(nbuff >= 1, "nbuff must be >= 1");
    PP_ARG(wsmooth == 0 || wsmooth == 1 || wsmooth == 3, "wsmooth %d not in {0,1,3}", wsmooth);
    PP_ARG(out->capacity >= 0, "negative capacity");
    PP_CHECK(ensure_device(ctx));
    PP_CHECK(fft_prepare(ctx, n));
    if (max_peaks_per_filter <= 0) max_peaks_per_filter = 2000000;
    size_t N = (size_t)n * n * n;
    size_t rb = N * sizeof(float), cb = (size_t)(n / 2 + 1) * n * n * sizeof(float2);
    FftLayout lay;  // of each filter's spectrum
    PP_CHECK(fft_padded(*ctx->fftp, &lay));
    PP_CHECK(ctx->d_k0.grow(cb));
    PP_CHECK(ctx->d_k1.grow(lay.plane * n * sizeof(float2)));
    PP_CHECK(ctx->d_field_a.grow(rb));
    // the wsmooth = 3 field at the peaks: line transforms where the mesh has
    // them, else a second rocFFT inverse per filter
    const bool lines = want_lapd && bank_lines(n);
    if (want_lapd && !lines) {
        PP_CHECK(ctx->d_k2.grow(cb));
        PP_CHECK(ctx->d_field_b.grow(rb));
    }
    PP_CHECK(ctx->d_mask.grow(N));
    PP_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    const float *d_delta = delta;
    if (!on_device) {
        PP_HIP(hipMemcpyAsync(ctx->d_field_a.ptr, delta, rb, hipMemcpyHostToDevice, ctx->stream));
        d_delta = ctx->d_field_a.as<float>();
    }
    {
        void *ib[1] = {(void *)d_delta}, *ob[1] = {ctx->d_k0.ptr};
        PP_FFT(rocfft_execute(ctx->fftp->r2c, ib, ob, ctx->fftp->info));
    }
    int8_t *d_mask = ctx->d_mask.as<int8_t>();
    if (mask_inout)
        PP_HIP(hipMemcpyAsync(d_mask, mask_inout, N, hipMemcpyHostToDevice, ctx->stream));
    else
        PP_HIP(hipMemsetAsync(d_mask, 0, N, ctx->stream));
    PeakOut o;
    float *d_lapd;
    long long *d_counters;
    PP_CHECK(alloc_peak_out(ctx, out->capacity, o, &d_lapd, &d_counters));
    const StencilGeom g = stencil_geom(n, n, n, nbuff);
    StencilScratch S;
    PP_CHECK(stencil_start(ctx, g, d_counters, S));
    const float inv = (float)(1.0 / ((double)n * n * n));
    Bank K;
    if (lines && nfilt > 0) PP_CHECK(bank_start(ctx, ctx->d_k0.ptr, n, nbuff, n - nbuff, boxsize, Rf, nfilt, K));
    // one read of delta_k gives a filter's spectrum and, with want_lapd and no
    // line transform, the wsmooth = 3 spectrum sampled at the filter's new
    // peaks; without the latter it is formed beside the filter before's peaks
    const bool two = want_lapd && !lines;
    auto window = [&](int f, WinJob *J) {
        return window_job(ctx->d_k0.ptr, ctx->d_k1.ptr, wsmooth, &lay, two ? ctx->d_k2.ptr : nullptr, PP_WINDOW_K2GAUSS,
                          n, boxsize, Rf[f], inv, J);
    };
    for (int f = 0; f < nfilt; f++) {
        if (lines) PP_CHECK(bank_transform(ctx, K, Rf, f, false));
        WinJob J;
        if (f == 0 || two) {
            PP_CHECK(window(f, &J));
            PP_CHECK(launch_window(ctx, J));
        }
        const bool ahead = !two && f + 1 < nfilt;
        if (ahead) PP_CHECK(window(f + 1, &J));
        void *ib[1] = {ctx->d_k1.ptr}, *ob[1] = {ctx->d_field_a.ptr};
        PP_FFT(rocfft_execute(lay.c2r, ib, ob, ctx->fftp->info));
        PP_CHECK(run_stencil(ctx, ctx->d_field_a.as<float>(), d_mask, g, fcrit[f], max_peaks_per_filter, f,
                             o, d_counters, S, lines ? K.ranges + 2 * f : nullptr, ahead ? &J : nullptr));
        if (lines) {
            PP_CHECK(bank_sample(ctx, K, f, o, d_lapd));
        } else if (want_lapd) {
            void *ib2[1] = {ctx->d_k2.ptr}, *ob2[1] = {ctx->d_field_b.ptr};
            PP_FFT(rocfft_execute(ctx->fftp->c2r, ib2, ob2, ctx->fftp->info));
            hipLaunchKernelGGL(k_sample_field, dim3(ctx->num_cu * 4), dim3(256), 0, ctx->stream,
                               ctx->d_field_b.as<float>(), n, n, (const int32_t *)o.i, (const int32_t *)o.j,
                               (const int32_t *)o.k, d_lapd, (const long long *)d_counters, o.capacity);
            PP_HIP(hipGetLastError());
        }
    }
    if (lines) PP_CHECK(bank_join(ctx));
    PP_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    if (mask_inout) PP_HIP(hipMemcpyAsync(mask_inout, d_mask, N, hipMemcpyDeviceToHost, ctx->stream));
    int rc = download_peaks(ctx, o, want_lapd ? d_lapd : nullptr, d_counters, out);
    float ms = 0;
    (void)hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]);
    ctx->timing.peakfind_ms = ms;
    return rc;
}

int pp_find_peaks_field_noalloc(pp_ctx *ctx, const float *delta_s, int8_t *mask, int n1, int n2, int n3, int nbuff,
                                float fcrit, int64_t max_peaks, pp_peaks *out)
{
    PP_ARG(ctx && delta_s && mask && out, "NULL argument");
    PP_ARG(out->i && out->j && out->k && out->filt && out->delta_s, "every output array is required");
    PP_ARG(n1 >= 3 && n2 >= 3 && n3 >= 3, "grid %dx%dx%d too small", n1, n2, n3);
    PP_ARG(nbuff >= 1, "nbuff must be >= 1 (the 27-point stencil reads one cell past the inner cube)");
    PP_ARG(out->capacity >= 0, "negative capacity");
    PP_CHECK(ensure_device(ctx));
    if (max_peaks <= 0) max_peaks = 2000000;
    const StencilGeom g = stencil_geom(n1, n2, n3, nbuff);
    const size_t need = stencil_scratch_bytes(g) + 256;
    PP_ARG(g.nwords <= kNoallocWords && need <= (size_t)PP_NOALLOC_SCRATCH_BYTES,
           "inner cube %dx%dx%d has %lld words, more than the %lld the scratch of this entry point is for; use "
           "pp_find_peaks_field", g.in1, g.in2, g.in3, g.nwords, kNoallocWords);
    char *base = (char *)noalloc_scratch(ctx->device);
    if (!base) {
        set_error("no scratch address for device %d (context creation records it)", ctx->device);
        return PP_ERR_STATE;
    }
    long long *d_counters = (long long *)base;
    PeakOut o;
    o.i = out->i; o.j = out->j; o.k = out->k; o.filt = out->filt; o.delta_s = out->delta_s;
    o.capacity = out->capacity;
    const StencilScratch S = stencil_carve(base + 256, g);
    PP_CHECK(stencil_clear(ctx, S, d_counters));
    PP_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    PP_CHECK(run_stencil(ctx, delta_s, mask, g, fcrit, max_peaks, 0, o, d_counters, S));
    PP_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    long long cnt[4];
    PP_HIP(hipMemcpyAsync(cnt, d_counters, sizeof cnt, hipMemcpyDeviceToHost, ctx->stream));
    PP_HIP(hipStreamSynchronize(ctx->stream));
    float ms = 0;
    (void)hipEventElapsedTime(&ms, ctx->ev[0], ctx->ev[1]);
    ctx->timing.peakfind_ms = ms;
    out->needed = cnt[1];
    out->count = cnt[1] < out->capacity ? cnt[1] : out->capacity;
    if (cnt[1] > out->capacity) {
        set_error("peak output capacity %lld too small: %lld peaks found", (long long)out->capacity, cnt[1]);
        return PP_ERR_CAPACITY;
    }
    return PP_OK;
}

}  // extern "C"

// ------------------------------------------------------------ input noise
// fill_noise_threefry! (src/InitialConditions/RandomField.jl:46-81) over n3
// cells, one thread per counter pair (threefry_normals).
namespace pp {

__global__ void k_noise_threefry(float *__restrict__ out, int64_t n3, uint64_t seed)
{
    const int64_t npairs = (n3 + 1) / 2;
    for (int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; p < npairs; p += (int64_t)gridDim.x * blockDim.x) {
        double g1, g2;
        threefry_normals((uint64_t)p, seed, g1, g2);
        out[2 * p] = (float)g1;
        if (2 * p + 1 < n3) out[2 * p + 1] = (float)g2;
    }
}

int launch_noise(pp_ctx *ctx, float *out, int64_t ncells, uint64_t seed)
{
    if (ncells == 0) return PP_OK;
    const int64_t npairs = (ncells + 1) / 2;
    const int grid = (int)std::max<int64_t>(1, std::min<int64_t>((npairs + 255) / 256, (int64_t)ctx->num_cu * 16));
    hipLaunchKernelGGL(k_noise_threefry, dim3(grid), dim3(256), 0, ctx->stream, out, ncells, seed);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

}  // namespace pp

extern "C" int pp_fill_noise_threefry(pp_ctx *ctx, float *out, int64_t ncells, uint64_t seed)
{
    PP_ARG(ctx && out, "NULL argument");
    PP_ARG(ncells >= 0, "negative cell count");
    PP_CHECK(pp::ensure_device(ctx));
    return pp::launch_noise(ctx, out, ncells, seed);
}
