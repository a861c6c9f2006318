// pp_split.hip -- run_multitile_split's fields on the device: the coarse
// grid of the global white noise and, per tile, the Hoffman-Ribak residual,
// its isolated (zero-padded) convolution, the Catmull-Rom interpolation of
// the coarse fields and the tile-periodic 2LPT and k^2 fields.
//
// Reference: src/MultiResolution.jl:41-314 (building blocks), 596-667
// (phase 1a, the coarse fields), 719-850 (process_tile!'s phase 1b),
// 1239-1255 (_apply_kernel_inplace!); the reference's GPU path
// (ext/CUDAExt.jl:2480-2947) for the Hermitian planes of the isolated
// transform.
//
// Design.  Everything a tile needs is generated where it is used:
// * the coarse noise is a block sum over the global grid, one workgroup per
//   coarse cell, each lane walking counter pairs along rows (one Threefry
//   block gives both normals of a pair), Float64 partial sums reduced in a
//   fixed tree;
// * the isolated convolution of the residual runs on line transforms
//   (pp_fft.h) that never store the zero padding: the noise is drawn in the x
//   pass, the transfer functions sit between the forward and the inverse
//   transform of the z pass, and the last pass cuts the tile out and adds the
//   coarse field's Catmull-Rom interpolation, contracted along y and z once
//   per row;
// * meshes without a line transform (odd, or with a prime factor above 7) go
//   through an in-place (2n)^3 rocFFT transform of the padded residual (rows
//   padded to 2 (n+1) floats), one pass over the base spectrum per output
//   (Float64 transfer factor, the kx = 0 and Nyquist planes averaged with
//   their conjugate partners) and one pass that cuts and interpolates with
//   64 taps a cell;
// * 2LPT: the source is accumulated in real space in the reference's order,
//   one potential at a time (two spectra and two real fields resident).
#include <cmath>
#include <vector>

#include "pp_common.h"
#include "pp_fields.h"
#include "pp_kspace.h"
#include "pp_noise.h"

struct pp_coarse {
    int device = 0;
    pp_split_geom g{};
    int N = 0, nsub = 0, block = 0, npk = 0;
    double boxsize_full = 0;
    pp::DevBuf noise, delta, psi, pk;  // M^3 floats; 3 M^3 floats; the P(k) table
    pp::PkLog table{};                 // its logarithms, in pk
};

namespace pp {

// ------------------------------------------------------------ coarse noise
// _downsample_noise: coarse cell (I, J, K) sums the normals of fine cells
// I b .. I b + b - 1 (and likewise in y, z), 0-based.  Bound by the
// instructions of the normals: with M = 20, b = 41 (5.5e8 cells) the coarse
// fields take 1.98 ms (3.33 ms with the general functions and two divisions a
// pair): 248 vector instructions a pair, which keep the SIMDs issuing for 1.74
// ms at 2.4 GHz.
__global__ void __launch_bounds__(256) k_coarse_noise(float *__restrict__ out, int N, int M, int b, uint64_t seed,
                                                      double norm)
{
    __shared__ double red[256];
    const long long ncoarse = (long long)M * M * M;
    const int per_row = b / 2 + 1;  // counter pairs a row of b cells can touch
    // thread t takes pair t, t + 256, ... of the cell's b b per_row; the steps
    // of its pair q, row dj and plane dk (divisions would cost a quarter of
    // the normals)
    const int q0 = (int)threadIdx.x % per_row, dj0 = (int)threadIdx.x / per_row % b,
              dk0 = (int)threadIdx.x / per_row / b;
    const int sq = 256 % per_row, sj = 256 / per_row % b, sk = 256 / per_row / b;
    const long long NN = (long long)N * N, ss = (long long)sj * N + sk * NN, wrap = NN - (long long)b * N;
    for (long long c = blockIdx.x; c < ncoarse; c += gridDim.x) {
        const int I = (int)(c % M), J = (int)((c / M) % M), K = (int)(c / ((long long)M * M));
        double acc = 0.0;
        // idx - 1 of the row's first cell
        long long s = (long long)I * b + ((long long)(J * b + dj0) + (long long)(K * b + dk0) * N) * N;
        for (int q = q0, dj = dj0, dk = dk0; dk < b;) {
            const long long e = s + b - 1, p = (s >> 1) + q;
            if (p <= (e >> 1)) {
                double g1, g2;
                threefry_normals((uint64_t)p, seed, g1, g2);
                if (2 * p >= s) acc += g1;
                if (2 * p + 1 <= e) acc += g2;
            }
            q += sq;
            dj += sj;
            dk += sk;
            s += ss;
            if (q >= per_row) {
                q -= per_row;
                dj++;
                s += N;
            }
            if (dj >= b) {
                dj -= b;
                dk++;
                s += wrap;
            }
        }
        red[threadIdx.x] = acc;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) out[c] = (float)(red[0] / norm);
        __syncthreads();
    }
}

// ------------------------------------------------------ spectrum transfer
enum XferMode { XF_AMP = 0, XF_AMP_IK = 1, XF_PHI = 2, XF_MIK = 3, XF_K2 = 4 };

struct Xfer {
    KGrid g;
    long long total;
    int mode, a, b;
    int nyq_zero;  // zero k = 0's partners on the Nyquist planes (_apply_kernel_inplace!)
    int herm;      // average the kx = 0 / kx = Nyquist planes with their conjugate partners
    double dk3, n3;  // dk^3 and n^3 of the amplitude sqrt((P(k) dk^3) n^3)
    PkLog T;
};

// the mode at (ix, iy, iz) times its transfer factor, rounded to ComplexF32
__device__ __forceinline__ float2 xfer_mode(const Xfer &X, const float2 *__restrict__ src, int ix, int iy, int iz)
{
#pragma clang fp contract(off)
    const KGrid &g = X.g;
    const int fy = iy < (g.n + 1) / 2 ? iy : iy - g.n, fz = iz < (g.n + 1) / 2 ? iz : iz - g.n;
    double k[3] = {(double)ix * g.mult, (double)fy * g.mult, (double)fz * g.mult};
    const double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
    if (k2 == 0.0) return make_float2(0.f, 0.f);
    if (X.nyq_zero && (ix == g.nk - 1 || iy == g.n / 2 || iz == g.n / 2)) return make_float2(0.f, 0.f);
    const float2 v = src[ix + (long long)g.nk * (iy + (long long)g.n * iz)];
    switch (X.mode) {
    case XF_AMP: {
        const double amp = sqrt(pk_eval(X.T.lk, X.T.lp, X.T.np, sqrt(k2), X.T.even[0], X.T.even[1]) * X.dk3 * X.n3);
        return cmul(v, amp, 0.0);
    }
    case XF_AMP_IK: {
        const double amp = sqrt(pk_eval(X.T.lk, X.T.lp, X.T.np, sqrt(k2), X.T.even[0], X.T.even[1]) * X.dk3 * X.n3);
        return cmul(v, 0.0, amp * (k[X.a] / k2));
    }
    case XF_PHI:
        return cmul(v, -k[X.a] * k[X.b] / k2, 0.0);
    case XF_MIK:
        return cmul(v, 0.0, -k[X.a] / k2);
    default:
        return cmul(v, k2, 0.0);
    }
}

__global__ void __launch_bounds__(256) k_xfer(const float2 *__restrict__ src, float2 *__restrict__ dst, Xfer X)
{
#pragma clang fp contract(off)
    const KGrid &g = X.g;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < X.total;
         e += (long long)gridDim.x * blockDim.x) {
        const int ix = (int)(e % g.nk);
        const long long r = e / g.nk;
        const int iy = (int)(r % g.n), iz = (int)(r / g.n);
        float2 v = xfer_mode(X, src, ix, iy, iz);
        if (X.herm && (ix == 0 || ((g.n & 1) == 0 && ix == g.nk - 1))) {
            const int iyc = iy == 0 ? 0 : g.n - iy, izc = iz == 0 ? 0 : g.n - iz;
            if (iyc == iy && izc == iz) {
                v.y = 0.f;
            } else {
                const float2 p = xfer_mode(X, src, ix, iyc, izc);
                v = make_float2((v.x + p.x) * 0.5f, (v.y - p.y) * 0.5f);
            }
        }
        dst[e] = v;
    }
}

// out[i] = in[i] * s (the Float32 normalisation of an inverse transform;
// in may be out)
__global__ void __launch_bounds__(256) k_scale(const float *in, float *out, long long n, float s)
{
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x)
        out[e] = in[e] * s;
}

// ------------------------------------------------------------- tile stages
struct TileGeo {
    int n, N, M, b;
    int i0, j0, k0;  // 0-based global index of the tile's first cell (before the wrap), >= -nbuff
    float inv_b3;    // Float32(1 / sqrt(block^3))
    uint64_t seed;
};

// v in [-m, 2m) folded into [0, m) (mod1 of the reference, 0-based): tile
// cells lie within nbuff <= N of the global grid, Catmull-Rom taps within
// two cells of the coarse one (M >= 2)
__device__ __forceinline__ int wrap1(int v, int m) { return v < 0 ? v + m : (v >= m ? v - m : v); }

// residual into the zero-padded (2n)^3 real buffer of pitch 2 (n + 1), every
// float of every row written
__global__ void __launch_bounds__(256) k_residual_pad(float *__restrict__ R, TileGeo T,
                                                      const float *__restrict__ coarse)
{
    const int n2 = 2 * T.n, pitch = n2 + 2, half = pitch / 2;
    const long long total = (long long)half * n2 * n2;  // two floats per item, padding floats included
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int x = 2 * (int)(e % half);
        const long long r = e / half;
        const int y = (int)(r % n2), z = (int)(r / n2);
        float2 v = make_float2(0.f, 0.f);
        if (x < T.n && y < T.n && z < T.n) {
            const int gy = wrap1(T.j0 + y, T.N), gz = wrap1(T.k0 + z, T.N);
            const long long rowb = ((long long)gy + (long long)gz * T.N) * T.N;
            const long long crow = (long long)T.M * (gy / T.b + (long long)T.M * (gz / T.b));
            float out2[2];
            long long last_pair = -1;
            double g1 = 0, g2 = 0;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (x + h >= T.n) {  // odd n: the pair's second cell is padding
                    out2[h] = 0.f;
                    continue;
                }
                const int gx = wrap1(T.i0 + x + h, T.N);
                const long long idx0 = gx + rowb;  // idx - 1
                const long long pr = idx0 >> 1;
                if (pr != last_pair) {
                    threefry_normals((uint64_t)pr, T.seed, g1, g2);
                    last_pair = pr;
                }
                const float fine = (float)((idx0 & 1) ? g2 : g1);
                const float cm = coarse[gx / T.b + crow];
                out2[h] = fine - cm * T.inv_b3;
            }
            v = make_float2(out2[0], out2[1]);
        }
        *reinterpret_cast<float2 *>(R + x + (long long)pitch * (y + (long long)n2 * z)) = v;
    }
}

// Catmull-Rom weights of _catmull_rom, Float32
__device__ __forceinline__ void cr_weights(float t, float w[4])
{
#pragma clang fp contract(off)
    const float t2 = t * t, t3 = t2 * t;
    w[0] = (-0.5f * t3 + t2) - 0.5f * t;
    w[1] = (1.5f * t3 - 2.5f * t2) + 1.0f;
    w[2] = (-1.5f * t3 + 2.0f * t2) + 0.5f * t;
    w[3] = 0.5f * t3 - 0.5f * t2;
}

// 1-based coarse base index and fraction of 0-based global fine index g:
// f = (g + 1 - 0.5) / block + 0.5
__device__ __forceinline__ void cr_coord(int g, int b, int &i0, float &t)
{
    const double f = ((double)(g + 1) - 0.5) / (double)b + 0.5;
    const double fl = floor(f);
    i0 = (int)fl;
    t = (float)(f - fl);
}

// out = (padded inverse transform at the tile cell) * inv + Catmull-Rom of
// the coarse field.  LDS: the whole coarse field is first copied to LDS (its
// M^3 floats fit when M^3 <= kCoarseLds), so the 64 taps per cell are LDS reads.
constexpr int kCoarseLds = 16384;

template <bool LDS>
__global__ void __launch_bounds__(256) k_extract_add(const float *__restrict__ S, float inv, TileGeo T,
                                                     const float *__restrict__ coarse_g, float *__restrict__ out)
{
#pragma clang fp contract(off)
    const int n = T.n, n2 = 2 * n, pitch = n2 + 2, M = T.M;
    const long long total = (long long)n * n * n;
    extern __shared__ float coarse_s[];
    if (LDS) {
        for (int q = threadIdx.x; q < M * M * M; q += blockDim.x) coarse_s[q] = coarse_g[q];
        __syncthreads();
    }
    const float *coarse = LDS ? coarse_s : coarse_g;
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(e % n);
        const long long r = e / n;
        const int y = (int)(r % n), z = (int)(r / n);
        const float self = S[x + (long long)pitch * (y + (long long)n2 * z)] * inv;
        int bx, by, bz;
        float tx, ty, tz, wx[4], wy[4], wz[4];
        cr_coord(wrap1(T.i0 + x, T.N), T.b, bx, tx);
        cr_coord(wrap1(T.j0 + y, T.N), T.b, by, ty);
        cr_coord(wrap1(T.k0 + z, T.N), T.b, bz, tz);
        cr_weights(tx, wx);
        cr_weights(ty, wy);
        cr_weights(tz, wz);
        // taps mod1(b + d, M) for d = -1..2, 0-based (b in 0..M)
        int ii[4], jj[4], kk[4];
#pragma unroll
        for (int a = 0; a < 4; a++) {
            ii[a] = wrap1(bx + a - 2, M);
            jj[a] = wrap1(by + a - 2, M);
            kk[a] = wrap1(bz + a - 2, M);
        }
        float val = 0.0f;
        for (int c = 0; c < 4; c++) {
            for (int q = 0; q < 4; q++) {
                const float *row = coarse + (long long)M * (jj[q] + (long long)M * kk[c]);
#pragma unroll
                for (int a = 0; a < 4; a++) val = val + ((wx[a] * wy[q]) * wz[c]) * row[ii[a]];
            }
        }
        out[e] = self + val;
    }
}

// src = (delta * delta) * 0.5
__global__ void __launch_bounds__(256) k_src_init(const float *__restrict__ d, float *__restrict__ src, long long n)
{
#pragma clang fp contract(off)
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long long)gridDim.x * blockDim.x)
        src[e] = (d[e] * d[e]) * 0.5f;
}

// phi = t * inv; src = src - (phi * phi) * coef
__global__ void __launch_bounds__(256) k_src_sub(float *__restrict__ src, const float *__restrict__ t, long long n,
                                                 float inv, float coef)
{
#pragma clang fp contract(off)
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < n;
         e += (long long)gridDim.x * blockDim.x) {
        const float phi = t[e] * inv;
        src[e] = src[e] - (phi * phi) * coef;
    }
}

// ------------------------------------------------- isolated convolution
// The zero-padded transform of the residual with line transforms
// (pp_fft.h).  Half of every padded line is zero and half of every result is
// cut away, so a line of 2 n is two of n and no padding is ever stored or
// read: with w = exp(-i pi / n),
//   X[2 m]     = FFT_n(x)[m],        X[2 m + 1] = FFT_n(x w^j)[m],
//   y[j], j < n = IFFT_n(X[2 m])[j] + w^-j IFFT_n(X[2 m + 1])[j].
// A spectrum holds n z planes (real space along z) of 2 n rows.  The z pass
// transforms forward, applies the transfer and transforms back while a
// column is in LDS, so the (2 n)^3 spectrum never exists in memory; iy A goes to
// the upper half of A's rows, which the cut leaves free.  delta, psi_x, psi_y
// and psi_z come from the three arrays X, X / |i|^2 and iz X / |i|^2 (whole wave
// numbers i and factors in pairs, as in pp_fields.h).  Traffic at
// n = 512: 30 GB in place of 170.
constexpr int kLineCoarse = 512;  // coarse cells a side whose rows fit LDS beside a line
struct PadGeo {
    int n;
    SpecGeo g;  // nk = n + 1 bins, 2 n rows a plane
};

// half h (0 even, 1 odd bins) of the transform of x
template <int M, bool OUT_LDS, class A>
__device__ __forceinline__ void pad_forward(const A &at, const LineFft &P, int jj, const float2 x[kLineEpt],
                                            float2 X[kLineEpt], int h)
{
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) X[q] = h ? fmul(x[q], P.half[min(jj + q * P.tj, P.n - 1)]) : x[q];
    line_run<-1, M, false, OUT_LDS>(at, P, jj, X);
}

// y (+)= the inverse of half h: in x, or in LDS
template <int M, bool IN_LDS, class A>
__device__ __forceinline__ void pad_inverse(const A &at, const LineFft &P, int jj, float2 x[kLineEpt],
                                            float2 y[kLineEpt], int h)
{
    line_run<1, M, IN_LDS, false>(at, P, jj, x);
#pragma unroll
    for (int q = 0; q < kLineEpt; q++)
        y[q] = h ? fadd(y[q], fmulc(x[q], P.half[min(jj + q * P.tj, P.n - 1)])) : x[q];
}

// Residual of a row pair drawn into its line: fine normal minus coarse block
// mean.  A thread takes two cells of one Threefry counter pair where the row's
// parity and the wrap allow it.
__device__ __forceinline__ void residual_row(float *line, const TileGeo &T, const float *__restrict__ coarse, int y,
                                             int z, int jj, int tj)
{
    const int gy = wrap1(T.j0 + y, T.N), gz = wrap1(T.k0 + z, T.N);
    const long long rowb = ((long long)gy + (long long)gz * T.N) * T.N;
    const float *crow = coarse + (long long)T.M * (gy / T.b + (long long)T.M * (gz / T.b));
    const int par = (int)((wrap1(T.i0, T.N) + rowb) & 1);
    for (int m = jj; 2 * m - par < T.n; m += tj) {
        long long last = -1;
        double g1 = 0, g2 = 0;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int x = 2 * m - par + h;
            if (x < 0 || x >= T.n) continue;
            const int gx = wrap1(T.i0 + x, T.N);
            const long long idx = gx + rowb, pr = idx >> 1;
            if (pr != last) {
                threefry_normals((uint64_t)pr, T.seed, g1, g2);
                last = pr;
            }
            const float fine = (float)((idx & 1) ? g2 : g1), cm = crow[gx / T.b];
            line[2 * (x + (x >> 3))] = fine - cm * T.inv_b3;
        }
    }
}

// x-forward of the residual
template <int M>
__global__ void __launch_bounds__(512) k_pad_rows_noise(PadGeo G, LineFft P, TileGeo T,
                                                        const float *__restrict__ coarse, float2 *__restrict__ out)
{
    extern __shared__ float2 lds[];
    const int n = G.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, r = 2 * ((long long)blockIdx.x * (blockDim.x / P.tj) + line);
    float2 *row = lds + line * row_pitch(n);
    const RowAddr at(row);
    const bool live = r < rows, two = r + 1 < rows;
    const int z = (int)(r / n), y = (int)(r - (long long)z * n), z2 = (int)((r + 1) / n),
              y2 = (int)(r + 1 - (long long)z2 * n);
    if (live) residual_row((float *)row, T, coarse, y, z, jj, P.tj);
    if (two) residual_row((float *)row + 1, T, coarse, y2, z2, jj, P.tj);  // n is even, and so are the rows
    __syncthreads();
    float2 x[kLineEpt];
    line_get(at, P, jj, x);
    float2 *a = out + G.g.row(z, y), *b = out + G.g.row(z2, y2);
#pragma nounroll
    for (int h = 0; h < 2; h++) {
        int j2 = jj;
        asm volatile("" : "+v"(j2));
        float2 X[kLineEpt];
        pad_forward<M, true>(at, P, j2, x, X, h);
        if (!live) continue;
#pragma unroll
        for (int q = 0; q < kRowBins; q++) {
            const int m = j2 + q * P.tj, k = 2 * m + h;
            if (k > n) break;
            float2 va, vb;
            split_rows(at(m), at(h ? n - 1 - m : (m == 0 ? 0 : n - m)), va, vb);
            a[k] = va;
            if (two) b[k] = vb;
        }
    }
}

// y-forward, in place: n rows in, 2 n out
template <int M>
__global__ void __launch_bounds__(1024) k_pad_cols_y_fwd(PadGeo G, LineFft P, ColGrid C, float2 *__restrict__ s)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const int jj = t.jj, kx = t.kx;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    float2 x[kLineEpt];
    line_load(P, jj, x, LineY(G.g, s, t.plane, 0, 1, kx));
#pragma nounroll
    for (int h = 0; h < 2; h++) {
        int j2 = jj;
        asm volatile("" : "+v"(j2));
        float2 X[kLineEpt];
        pad_forward<M, false>(at, P, j2, x, X, h);
        line_store(P, j2, X, LineY(G.g, s, t.plane, h, 2, kx));
    }
}

struct PadZ {
    const float2 *in;
    float2 *out[3];  // X, X / |i|^2, iz X / |i|^2
    const Two *amp;  // by |i|^2
};

// z-forward, transfer, z-inverse
template <int M>
__global__ void __launch_bounds__(1024) k_pad_cols_z(PadGeo G, LineFft P, ColGrid C, PadZ A)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const int jj0 = t.jj, kxp = t.kx;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const int n = G.n, iy = t.plane, fy = iy < n ? iy : iy - 2 * n, kx = min(kxp, n), ixy = kx * kx + fy * fy;
    float2 X[2][kLineEpt];
    {
        float2 x[kLineEpt];
        line_load(P, jj0, x, LineZ(G.g, A.in, iy, kxp));
#pragma unroll
        for (int h = 0; h < 2; h++) {
            pad_forward<M, false>(at, P, jj0, x, X[h], h);
#pragma unroll
            for (int q = 0; q < kLineEpt; q++) {
                const int e = 2 * min(jj0 + q * P.tj, n - 1) + h, fz = e < n ? e : e - 2 * n;
                X[h][q] = ftimes(A.amp[ixy + fz * fz], X[h][q]);
            }
        }
    }
    for (int o = 0; o < 3; o++) {
        int jj = jj0;
        asm volatile("" : "+v"(jj));
        float2 y[kLineEpt];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float2 x[kLineEpt];
#pragma unroll
            for (int q = 0; q < kLineEpt; q++) {
                const int e = jj + q * P.tj, k = 2 * e + h, fz = k < n ? k : k - 2 * n, i2 = ixy + fz * fz;
                x[q] = X[h][q];
                if (o > 0) {
                    Two f = i2 == 0 ? Two{0.f, 0.f} : finverse((float)i2);
                    if (o == 2) f = ftimes(f, (float)fz);
                    x[q] = ftimes(f, x[q]);
                }
            }
            pad_inverse<M, false>(at, P, jj, x, y, h);
        }
        line_store(P, jj, y, LineZ(G.g, A.out[o], iy, kxp));
    }
}

struct PadY {
    float2 *s[3];
    int nvar[3];  // 1, or 2: times iy too, to rows n .. 2 n - 1
};

// y-inverse, in place: 2 n rows in, n (per power of ky) out
template <int M>
__global__ void __launch_bounds__(1024) k_pad_cols_y_inv(PadGeo G, LineFft P, ColGrid C, PadY A)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const int jj0 = t.jj, kx = t.kx;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const int n = G.n;
    float2 *s = A.s[blockIdx.y];
    float2 X[2][kLineEpt];
#pragma unroll
    for (int h = 0; h < 2; h++) line_load(P, jj0, X[h], LineY(G.g, s, t.plane, h, 2, kx));
    for (int o = 0; o < A.nvar[blockIdx.y]; o++) {
        int jj = jj0;
        asm volatile("" : "+v"(jj));
        float2 y[kLineEpt];
#pragma unroll
        for (int h = 0; h < 2; h++) {
            float2 x[kLineEpt];
#pragma unroll
            for (int q = 0; q < kLineEpt; q++) {
                const int e = jj + q * P.tj, k = 2 * e + h;
                const float f = o == 0 ? 1.f : (float)(k < n ? k : k - 2 * n);
                x[q] = make_float2(X[h][q].x * f, X[h][q].y * f);
            }
            pad_inverse<M, false>(at, P, jj, x, y, h);
        }
        const LineY w(G.g, s, t.plane, o * n, 1, kx);
        line_store(P, jj, y, w);
    }
}

struct PadX {
    struct Op {
        const float2 *in;
        int row0;       // first row of the plane
        int imag, pow;  // factor f, i f or i f ix
        Two f;
        const float *coarse;
        float *out;
    } op[4];
};

// Coarse row of tile row (y, z): the sum over the 4 x 4 taps along y and z,
// after which a cell takes four taps along x instead of 64
__device__ __forceinline__ void coarse_row(float *rc, const TileGeo &T, const float *__restrict__ coarse, int y, int z,
                                           int jj, int tj)
{
    int by, bz;
    float ty, tz, wy[4], wz[4];
    cr_coord(wrap1(T.j0 + y, T.N), T.b, by, ty);
    cr_coord(wrap1(T.k0 + z, T.N), T.b, bz, tz);
    cr_weights(ty, wy);
    cr_weights(tz, wz);
    for (int i = jj; i < T.M; i += tj) {
        float v = 0.f;
#pragma unroll
        for (int c = 0; c < 4; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const long long row = wrap1(by + q - 2, T.M) + (long long)T.M * wrap1(bz + c - 2, T.M);
                v += (wy[q] * wz[c]) * coarse[i + T.M * row];
            }
        rc[i] = v;
    }
}

// x-inverse of the row pairs, plus the interpolated coarse field
template <int M>
__global__ void __launch_bounds__(512) k_pad_rows_inv(PadGeo G, LineFft P, TileGeo T, PadX A)
{
    extern __shared__ float2 lds[];
    const int n = G.n, lines = blockDim.x / P.tj, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, r = 2 * ((long long)blockIdx.x * lines + line);
    const RowAddr at(lds + line * row_pitch(n));
    float *rc = (float *)(lds + lines * row_pitch(n)) + (size_t)line * 2 * T.M;
    const bool live = r < rows, two = r + 1 < rows;
    const PadX::Op &O = A.op[blockIdx.y];
    const int z = (int)(r / n), y = (int)(r - (long long)z * n), z2 = (int)((r + 1) / n),
              y2 = (int)(r + 1 - (long long)z2 * n);
    const float2 *a = O.in + G.g.row(z, O.row0 + y), *b = O.in + G.g.row(z2, O.row0 + y2);
    if (live) coarse_row(rc, T, O.coarse, y, z, jj, P.tj);
    if (two) coarse_row(rc + T.M, T, O.coarse, y2, z2, jj, P.tj);
    float2 v[kLineEpt];
#pragma nounroll
    for (int h = 0; h < 2; h++) {
        int j2 = jj;
        asm volatile("" : "+v"(j2));
        __syncthreads();
        if (live) {
            float2 va[kRowBins], vb[kRowBins];
#pragma unroll
            for (int q = 0; q < kRowBins; q++) {
                const int k = min(2 * (j2 + q * P.tj) + h, n);
                va[q] = a[k];
                vb[q] = two ? b[k] : make_float2(0.f, 0.f);
            }
#pragma unroll
            for (int q = 0; q < kRowBins; q++) {
                const int m = j2 + q * P.tj, k = 2 * m + h;
                if (k > n) break;
                const Two c = O.pow ? ftimes(O.f, (float)k) : O.f;
                const float2 p = ftimes(c, va[q]), s = ftimes(c, vb[q]);
                const float2 f1 = O.imag ? make_float2(-p.y, p.x) : p, f2 = O.imag ? make_float2(-s.y, s.x) : s;
                const int mc = h ? n - 1 - m : (m == 0 ? 0 : n - m);
                if (k == 0 || k == n) {  // real bins (mc = m)
                    at(m) = make_float2(f1.x, f2.x);
                } else {
                    at(m) = make_float2(f1.x - f2.y, f1.y + f2.x);
                    at(mc) = make_float2(f1.x + f2.y, f2.x - f1.y);
                }
            }
        }
        __syncthreads();
        float2 x[kLineEpt];
        pad_inverse<M, true>(at, P, j2, x, v, h);
    }
    if (!live) return;
    float *pa = O.out + r * n, *pb = pa + n;
    const unsigned b2 = 2u * (unsigned)T.b;
    const float ib2 = 1.f / (float)b2;
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = jj + q * P.tj;
        if (e >= n) break;
        // the base cell and fraction of (g + 1/2) / b + 1/2 (cr_coord), in integers
        const unsigned num = 2u * (unsigned)wrap1(T.i0 + e, T.N) + 1u + (unsigned)T.b, i = num / b2;
        float w[4];
        const float rem = (float)(num - i * b2), t0 = rem * ib2;
        cr_weights(__builtin_fmaf(__builtin_fmaf(-t0, (float)b2, rem), ib2, t0), w);  // rem / b2, rounded once
        float c1 = 0.f, c2 = 0.f;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const int c = wrap1((int)i + t - 2, T.M);
            c1 += w[t] * rc[c];
            c2 += w[t] * rc[T.M + c];
        }
        pa[e] = v[q].x + c1;
        if (two) pb[e] = v[q].y + c2;
    }
}

// pp_split_tile_fields with line transforms
static int split_tile_lines(pp_ctx *ctx, const pp_coarse *c, const TileGeo &T, pp_tile_fields *f)
{
    const pp_split_geom &G = c->g;
    const int n = G.nmesh, M = G.M;
    const long long n3 = (long long)n * n * n, M3 = (long long)M * M * M;
    const bool lpt2 = f->eta2x != nullptr;
    GridPlan D;
    PP_CHECK(grid_plan(ctx, n, &D));
    PadGeo Q;
    Q.n = n;
    Q.g = spec_geo(2 * n, 2 * n);
    // three padded spectra; then, in their place, those of the tile's grid.
    // Stream ordered and returned when the tile's fields are written, so a
    // context does not keep them between tiles
    const size_t pad = Q.g.size(n), arr = D.g.size(n);
    const int narr = 1 + (f->lapd ? 1 : 0) + (lpt2 ? 6 : 0);  // source or delta, then A .. iy B; L last
    const size_t need = std::max(3 * pad, (size_t)narr * arr) * sizeof(float2);
    void *arena = nullptr;
    hipError_t ea = hipMallocAsync(&arena, need, ctx->stream);
    if (ea != hipSuccess) {
        (void)hipGetLastError();
        set_error("hipMallocAsync of %zu B: %s", need, hipGetErrorString(ea));
        return ea == hipErrorOutOfMemory ? PP_ERR_OOM : PP_ERR_HIP;
    }
    struct Release {
        hipStream_t s;
        void *p;
        ~Release() { (void)hipFreeAsync(p, s); }
    } release{ctx->stream, arena};
    const long long count = amp_count(n);
    PP_CHECK(ctx->d_misc.grow(count * sizeof(Two)));
    Two *amp = ctx->d_misc.as<Two>();
    const int n2 = 2 * n;
    const double dx = (double)G.nmesh * G.alatt / n, dki = 2.0 * M_PI / (n2 * dx), mi = ((double)n2 * dki) / (double)n2;
    const double pad3 = (double)n2 * n2 * n2;
    PP_CHECK(amp_table(ctx, c->table, mi, dki * dki * dki, pad3, count, amp));
    float2 *s[3];
    for (int q = 0; q < 3; q++) s[q] = (float2 *)arena + pad * q;
    const long long pairs = ((long long)n * n + 1) / 2;
    const dim3 rgrid((unsigned)((pairs + D.rs.nl - 1) / D.rs.nl)), rblock(D.rs.block);
    const ColGrid cy = D.cs.grid(Q.g.nk, n, 1), cz = D.cs.grid(Q.g.nk, 2 * n, kColXCD);
    const dim3 gy(cy.blocks()), gz(cz.blocks()), cblock(D.cs.block);
    PP_LINE_LAUNCH(D.row, k_pad_rows_noise, rgrid, rblock, D.rs.lds, ctx->stream, Q, D.row, T, c->noise.as<float>(),
                   s[0]);
    PP_LINE_LAUNCH(D.col, k_pad_cols_y_fwd, gy, cblock, D.cs.lds, ctx->stream, Q, D.col, cy, s[0]);
    PadZ Z{s[0], {s[0], s[1], s[2]}, amp};
    PP_LINE_LAUNCH(D.col, k_pad_cols_z, gz, cblock, D.cs.lds, ctx->stream, Q, D.col, cz, Z);
    PadY Y{{s[0], s[1], s[2]}, {1, 2, 1}};
    PP_LINE_LAUNCH(D.col, k_pad_cols_y_inv, dim3(gy.x, 3), cblock, D.cs.lds, ctx->stream, Q, D.col, cy, Y);
    PadX X{};
    const float *psi = c->psi.as<float>();
    X.op[0] = PadX::Op{s[0], 0, 0, 0, two(1.0), c->delta.as<float>(), f->delta};
    X.op[1] = PadX::Op{s[1], 0, 1, 1, two(1.0 / mi), psi, f->etax};
    X.op[2] = PadX::Op{s[1], n, 1, 0, two(1.0 / mi), psi + M3, f->etay};
    X.op[3] = PadX::Op{s[2], 0, 1, 0, two(1.0 / mi), psi + 2 * M3, f->etaz};
    const size_t rlds = D.rs.lds + (size_t)D.rs.nl * 2 * M * sizeof(float);
    PP_LINE_LAUNCH(D.row, k_pad_rows_inv, dim3(rgrid.x, 4), rblock, rlds, ctx->stream, Q, D.row, T, X);
    if (!lpt2 && !f->lapd) {
        PP_HIP(hipStreamSynchronize(ctx->stream));
        return PP_OK;
    }
    // the tile-periodic k^2 and 2LPT fields from the combined delta
    float2 *t[8];
    for (int q = 0; q < narr; q++) t[q] = (float2 *)arena + arr * q;
    float2 *L = f->lapd ? t[narr - 1] : nullptr;
    const double dkt = 2.0 * M_PI / ((double)G.nmesh * G.alatt), mt = ((double)n * dkt) / (double)n;
    PP_CHECK(rows_real(D, f->delta, t[0]));
    PP_CHECK(cols_y_fwd(D, t[0]));
    ZArgs Z2{};
    Z2.in = t[0];
    YArgs Y2{};
    if (L) {
        Z2.add(L, Z_K2, 1);
        Y2.add(L, L, nullptr, nullptr);
    }
    if (lpt2) {
        Z2.add(t[0], Z_INV, 1);
        Z2.add(t[1], Z_INV_Z, 1);
        Z2.add(t[2], Z_INV_ZZ, 1);
        Y2.add(t[0], t[0], t[3], t[4]);
        Y2.add(t[1], t[1], t[5], nullptr);
        Y2.add(t[2], t[2], nullptr, nullptr);
    }
    PP_CHECK(cols_z(D, Z2));
    PP_CHECK(cols_y_inv(D, Y2));
    if (L) {
        XArgs X2{};
        X2.add(L, f->lapd, 0, false, mt * mt / (double)n3);
        PP_CHECK(rows_inv(D, X2));
    }
    if (lpt2) {
        float2 *src = t[6];
        SrcArgs S{};
        S.delta = f->delta;
        S.f = two(1.0 / (double)n3);
        S.out = src;
        src_inputs(S, t[0], t[3], t[4], t[1], t[5], t[2]);
        PP_CHECK(rows_src(D, S));
        float2 *w[3] = {src, t[0], t[1]};
        float *out[3] = {f->eta2x, f->eta2y, f->eta2z};
        PP_CHECK(second_order(D, w, mt, 1.0 / (double)n3, out));
    }
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

static int grid_for(pp_ctx *ctx, long long items)
{
    return (int)std::max<long long>(1, std::min<long long>((items + 255) / 256, (long long)ctx->num_cu * 16));
}

static int launch_xfer(pp_ctx *ctx, const void *src, void *dst, const Xfer &X)
{
    hipLaunchKernelGGL(k_xfer, dim3(grid_for(ctx, X.total)), dim3(256), 0, ctx->stream, (const float2 *)src,
                       (float2 *)dst, X);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

static Xfer make_xfer(int n, double dk, int mode, int a, int b, int nyq_zero, const pp_coarse *c)
{
    Xfer X{};
    X.g = KGrid{n, n / 2 + 1, ((double)n * dk) / (double)n};
    X.total = (long long)X.g.nk * n * n;
    X.mode = mode;
    X.a = a;
    X.b = b;
    X.nyq_zero = nyq_zero;
    X.herm = 1;
    X.dk3 = dk * dk * dk;
    X.n3 = (double)n * n * n;
    if (c) X.T = c->table;
    return X;
}

// Float32(1) / Float32(N): the scale of FFTW's normalised inverse on Float32 data
static float inv_count(long long count) { return 1.0f / (float)count; }

}  // namespace pp

using namespace pp;

extern "C" {

int pp_coarse_create(pp_ctx *ctx, const pp_split_geom *geom, const pp_pk_table *pk, pp_coarse **out)
{
    PP_ARG(ctx && geom && pk && out, "NULL argument");
    *out = nullptr;
    const pp_split_geom &G = *geom;
    PP_ARG(G.nmesh >= 4 && G.nbuff >= 0 && G.ntile >= 1 && G.M >= 2 && G.alatt > 0, "bad split geometry");
    const int nsub = G.nmesh - 2 * G.nbuff;
    PP_ARG(nsub >= 1, "nmesh %d leaves no core cells with nbuff %d", G.nmesh, G.nbuff);
    const long long N = (long long)nsub * G.ntile + 2ll * G.nbuff;
    PP_ARG(N % G.M == 0, "N=%lld must be divisible by M=%d", N, G.M);
    PP_ARG(N <= (1ll << 20) && (long long)G.M * G.M * G.M <= (1ll << 30), "global grid N=%lld too large", N);
    PP_ARG(pk->npk >= 2 && pk->k && pk->P, "P(k) table needs >= 2 rows");
    for (int q = 0; q < pk->npk; q++) {
        PP_ARG(pk->k[q] > 0 && pk->P[q] > 0, "P(k) table row %d not positive", q);
        PP_ARG(q == 0 || pk->k[q] > pk->k[q - 1], "P(k) table k not increasing at row %d", q);
    }
    PP_CHECK(ensure_device(ctx));
    pp_coarse *c = new pp_coarse();
    c->device = ctx->device;
    c->g = G;
    c->N = (int)N;
    c->nsub = nsub;
    c->block = (int)(N / G.M);
    c->boxsize_full = (double)N * G.alatt;
    c->npk = pk->npk;
    auto fail = [&](int rc) {
        pp_coarse_destroy(c);
        return rc;
    };
    const int M = G.M;
    const long long M3 = (long long)M * M * M;
    int rc = c->noise.grow(M3 * 4);
    if (rc == PP_OK) rc = c->delta.grow(M3 * 4);
    if (rc == PP_OK) rc = c->psi.grow(3 * M3 * 4);
    if (rc == PP_OK) rc = c->pk.grow(pk_log_doubles(pk->npk) * sizeof(double));
    if (rc != PP_OK) return fail(rc);
    rc = pk_log_device(ctx, pk, c->pk.as<double>(), &c->table);
    if (rc != PP_OK) return fail(rc);
    // 1. the coarse noise
    const int b = c->block;
    const double norm = sqrt((double)b * (double)b * (double)b);
    hipLaunchKernelGGL(k_coarse_noise, dim3((unsigned)std::min<long long>(M3, 1 << 20)), dim3(256), 0, ctx->stream,
                       c->noise.as<float>(), c->N, M, b, G.seed, norm);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        set_error("k_coarse_noise: %s", hipGetErrorString(e));
        return fail(PP_ERR_HIP);
    }
    // 2. its periodic convolutions on the coarse grid
    FftPlans *F = nullptr;
    rc = fft_plans(ctx, M, 0, &F);
    if (rc != PP_OK) return fail(rc);
    const long long ck = (long long)(M / 2 + 1) * M * M;
    rc = ctx->d_k0.grow(ck * 8);
    if (rc == PP_OK) rc = ctx->d_k1.grow(ck * 8);
    if (rc == PP_OK) rc = ctx->d_field_a.grow(M3 * 4);
    if (rc != PP_OK) return fail(rc);
    const double dk = 2.0 * M_PI / c->boxsize_full;
    const float inv = inv_count(M3);
    auto run = [&]() -> int {
        void *ib[1] = {c->noise.ptr}, *ob[1] = {ctx->d_k0.ptr};
        PP_FFT(rocfft_execute(F->r2c, ib, ob, F->info));
        for (int q = 0; q < 4; q++) {
            const Xfer X = make_xfer(M, dk, q == 0 ? XF_AMP : XF_AMP_IK, q == 0 ? 0 : q - 1, 0, 0, c);
            PP_CHECK(launch_xfer(ctx, ctx->d_k0.ptr, ctx->d_k1.ptr, X));
            void *ib2[1] = {ctx->d_k1.ptr}, *ob2[1] = {ctx->d_field_a.ptr};
            PP_FFT(rocfft_execute(F->c2r, ib2, ob2, F->info));
            float *dst = q == 0 ? c->delta.as<float>() : c->psi.as<float>() + (q - 1) * M3;
            hipLaunchKernelGGL(k_scale, dim3(grid_for(ctx, M3)), dim3(256), 0, ctx->stream,
                               (const float *)ctx->d_field_a.ptr, dst, M3, inv);
            PP_HIP(hipGetLastError());
        }
        PP_HIP(hipStreamSynchronize(ctx->stream));
        return PP_OK;
    };
    rc = run();
    if (rc != PP_OK) return fail(rc);
    *out = c;
    return PP_OK;
}

int pp_coarse_download(const pp_coarse *c, float *noise, float *delta, float *psix, float *psiy, float *psiz)
{
    PP_ARG(c, "NULL coarse field");
    PP_HIP(hipSetDevice(c->device));
    const size_t M3 = (size_t)c->g.M * c->g.M * c->g.M, b = M3 * 4;
    if (noise) PP_HIP(hipMemcpy(noise, c->noise.ptr, b, hipMemcpyDeviceToHost));
    if (delta) PP_HIP(hipMemcpy(delta, c->delta.ptr, b, hipMemcpyDeviceToHost));
    float *p[3] = {psix, psiy, psiz};
    for (int q = 0; q < 3; q++)
        if (p[q]) PP_HIP(hipMemcpy(p[q], c->psi.as<float>() + q * M3, b, hipMemcpyDeviceToHost));
    return PP_OK;
}

int pp_coarse_destroy(pp_coarse *c)
{
    if (!c) return PP_OK;
    (void)hipSetDevice(c->device);
    (void)hipDeviceSynchronize();
    c->noise.release();
    c->delta.release();
    c->psi.release();
    c->pk.release();
    delete c;
    return PP_OK;
}

int pp_split_tile_fields(pp_ctx *ctx, const pp_coarse *c, int it, int jt, int kt, pp_tile_fields *f)
{
    PP_ARG(ctx && c && f && f->delta && f->etax && f->etay && f->etaz, "NULL argument");
    PP_ARG(c->device == ctx->device, "coarse field on device %d, context on device %d", c->device, ctx->device);
    const pp_split_geom &G = c->g;
    PP_ARG(it >= 1 && jt >= 1 && kt >= 1 && it <= G.ntile && jt <= G.ntile && kt <= G.ntile,
           "tile (%d, %d, %d) outside 1..%d", it, jt, kt, G.ntile);
    const bool lpt2 = f->eta2x != nullptr;
    PP_ARG(!lpt2 || (f->eta2y && f->eta2z), "eta2 outputs come as a set of three");
    PP_CHECK(ensure_device(ctx));
    const int n = G.nmesh, n2 = 2 * n;
    TileGeo T;
    T.n = n;
    T.N = c->N;
    T.M = G.M;
    T.b = c->block;
    T.i0 = (it - 1) * c->nsub - G.nbuff;
    T.j0 = (jt - 1) * c->nsub - G.nbuff;
    T.k0 = (kt - 1) * c->nsub - G.nbuff;
    T.inv_b3 = (float)(1.0 / sqrt(pow((double)c->block, 3)));
    T.seed = G.seed;
    // the line passes pair rows of even length
    if (n % 2 == 0 && line_supported(n) && G.M <= kLineCoarse) return split_tile_lines(ctx, c, T, f);
    const long long n3 = (long long)n * n * n;
    // 1. residual -> padded buffer R; base spectrum in place
    FftPlans *Fi = nullptr;
    PP_CHECK(fft_plans(ctx, n2, 1, &Fi));
    // the two padded (2n)^3 buffers (the largest of the tile) are stream
    // ordered and returned when the tile's fields are written, so a context
    // does not keep them between tiles
    const size_t pad_floats = (size_t)(n2 + 2) * n2 * n2;
    float *R = nullptr, *S = nullptr;
    PP_HIP(hipMallocAsync((void **)&R, pad_floats * 4, ctx->stream));
    hipError_t ea = hipMallocAsync((void **)&S, pad_floats * 4, ctx->stream);
    if (ea != hipSuccess) {
        (void)hipFreeAsync(R, ctx->stream);
        set_error("hipMallocAsync of %zu B: %s", pad_floats * 4, hipGetErrorString(ea));
        return PP_ERR_HIP;
    }
    void *Wk = nullptr;
    struct Release {
        hipStream_t s;
        float *a, *b;
        void **w;
        ~Release()
        {
            (void)hipFreeAsync(a, s);
            (void)hipFreeAsync(b, s);
            if (*w) (void)hipFreeAsync(*w, s);
        }
    } release{ctx->stream, R, S, &Wk};
    if (Fi->work_need > 0) {
        PP_HIP(hipMallocAsync(&Wk, Fi->work_need, ctx->stream));
        PP_FFT(rocfft_execution_info_set_work_buffer(Fi->info, Wk, Fi->work_need));
    }
    hipLaunchKernelGGL(k_residual_pad, dim3(grid_for(ctx, (long long)(n + 1) * n2 * n2)), dim3(256), 0, ctx->stream, R, T,
                       (const float *)c->noise.ptr);
    PP_HIP(hipGetLastError());
    {
        void *io[1] = {R};
        PP_FFT(rocfft_execute(Fi->r2c, io, nullptr, Fi->info));
    }
    // 2. delta and psi: transfer, inverse in place, cut + interpolate
    const double dx = (double)G.nmesh * G.alatt / n;  // boxsize_local / n
    const double dki = 2.0 * M_PI / (n2 * dx);
    const float inv_i = inv_count((long long)n2 * n2 * n2);
    float *outs[4] = {f->delta, f->etax, f->etay, f->etaz};
    for (int q = 0; q < 4; q++) {
        const Xfer X = make_xfer(n2, dki, q == 0 ? XF_AMP : XF_AMP_IK, q == 0 ? 0 : q - 1, 0, 0, c);
        PP_CHECK(launch_xfer(ctx, R, S, X));
        void *io[1] = {S};
        PP_FFT(rocfft_execute(Fi->c2r, io, nullptr, Fi->info));
        const float *cf = q == 0 ? c->delta.as<float>() : c->psi.as<float>() + (long long)(q - 1) * G.M * G.M * G.M;
        const long long M3 = (long long)G.M * G.M * G.M;
        if (M3 <= kCoarseLds)
            hipLaunchKernelGGL(k_extract_add<true>, dim3(grid_for(ctx, n3)), dim3(256), M3 * sizeof(float),
                               ctx->stream, (const float *)S, inv_i, T, cf, outs[q]);
        else
            hipLaunchKernelGGL(k_extract_add<false>, dim3(grid_for(ctx, n3)), dim3(256), 0, ctx->stream,
                               (const float *)S, inv_i, T, cf, outs[q]);
        PP_HIP(hipGetLastError());
    }
    // 3. the tile-periodic 2LPT and k^2 fields from the combined delta
    if (lpt2 || f->lapd) {
        PP_CHECK(fft_prepare(ctx, n));
        const long long ckn = (long long)(n / 2 + 1) * n * n;
        PP_CHECK(ctx->d_k0.grow(ckn * 8));
        PP_CHECK(ctx->d_k1.grow(ckn * 8));
        PP_CHECK(ctx->d_field_a.grow(2 * n3 * 4));
        float *src = ctx->d_field_a.as<float>(), *tmp = src + n3;
        const double dkt = 2.0 * M_PI / ((double)G.nmesh * G.alatt);
        const float inv_t = inv_count(n3);
        FftPlans *F = ctx->fftp;
        auto c2r = [&](void *in, float *o) -> int {
            void *ib[1] = {in}, *ob[1] = {(void *)o};
            PP_FFT(rocfft_execute(F->c2r, ib, ob, F->info));
            return PP_OK;
        };
        auto r2c = [&](const float *in, void *o) -> int {
            void *ib[1] = {(void *)in}, *ob[1] = {o};
            PP_FFT(rocfft_execute(F->r2c, ib, ob, F->info));
            return PP_OK;
        };
        auto scale = [&](float *a) -> int {
            hipLaunchKernelGGL(k_scale, dim3(grid_for(ctx, n3)), dim3(256), 0, ctx->stream, (const float *)a, a, n3,
                               inv_t);
            PP_HIP(hipGetLastError());
            return PP_OK;
        };
        PP_CHECK(r2c(f->delta, ctx->d_k0.ptr));
        if (f->lapd) {
            PP_CHECK(launch_xfer(ctx, ctx->d_k0.ptr, ctx->d_k1.ptr, make_xfer(n, dkt, XF_K2, 0, 0, 1, nullptr)));
            PP_CHECK(c2r(ctx->d_k1.ptr, f->lapd));
            PP_CHECK(scale(f->lapd));
        }
        if (lpt2) {
            hipLaunchKernelGGL(k_src_init, dim3(grid_for(ctx, n3)), dim3(256), 0, ctx->stream, (const float *)f->delta,
                               src, n3);
            PP_HIP(hipGetLastError());
            const int A[6] = {0, 1, 2, 0, 0, 1}, B[6] = {0, 1, 2, 1, 2, 2};
            for (int q = 0; q < 6; q++) {
                PP_CHECK(launch_xfer(ctx, ctx->d_k0.ptr, ctx->d_k1.ptr, make_xfer(n, dkt, XF_PHI, A[q], B[q], 1, nullptr)));
                PP_CHECK(c2r(ctx->d_k1.ptr, tmp));
                hipLaunchKernelGGL(k_src_sub, dim3(grid_for(ctx, n3)), dim3(256), 0, ctx->stream, src,
                                   (const float *)tmp, n3, inv_t, q < 3 ? 0.5f : 1.0f);
                PP_HIP(hipGetLastError());
            }
            PP_CHECK(r2c(src, ctx->d_k0.ptr));
            float *e2[3] = {f->eta2x, f->eta2y, f->eta2z};
            for (int d = 0; d < 3; d++) {
                PP_CHECK(launch_xfer(ctx, ctx->d_k0.ptr, ctx->d_k1.ptr, make_xfer(n, dkt, XF_MIK, d, 0, 1, nullptr)));
                PP_CHECK(c2r(ctx->d_k1.ptr, e2[d]));
                PP_CHECK(scale(e2[d]));
            }
        }
    }
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

}  // extern "C"
