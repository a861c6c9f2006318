// pp_fields.hip -- the input fields of one tile on the device: Gaussian
// random field, 1LPT and 2LPT displacements and the k^2 ("Laplacian") field.
//
// Reference: run_tile's field generation (src/Pipeline.jl:110-206):
// generate_grf / _convolve_noise! (src/InitialConditions/RandomField.jl:
// 123-175) with fill_noise_threefry! (:46-81) and load_pk (src/
// InitialConditions/PowerSpectrum.jl:11-23); displacements_1lpt /
// displacements_2lpt (src/InitialConditions/LPT.jl:21-191);
// _compute_laplacian (src/Pipeline.jl:35-51).
//
// Design: line transforms in LDS (pp_fft.h) where the mesh has them: the noise
// is drawn in the x pass, the transfer functions sit between the forward and
// the inverse transform of the z pass, several outputs share a pass, and the
// 2LPT source is formed in the pass that brings its potentials to real space.
// Other meshes (lines_for) go through rocFFT (the context's
// cached plans) and one pass over the half spectrum per k-space step, which
// evaluates its Float64 factor per mode and rounds the product into Float32
// once, as the reference's Float64 factor times its ComplexF32 array does; the
// 1/n^3 of the normalised inverse transforms is folded into that factor (an
// exact power of two for power-of-two n), and the source is accumulated in
// real space in the reference's order, so only the diagonal potentials and the
// running sum are held at once.
#include <cmath>
#include <vector>

#include "pp_common.h"
#include "pp_fft.h"
#include "pp_fields.h"
#include "pp_kspace.h"
#include "pp_noise.h"

namespace pp {

// noise_k * sqrt(P(k) dk^3 n^3) / n^3, k = 0 zeroed (RandomField.jl:144-167)
__global__ void __launch_bounds__(256) k_grf_amp(float2 *__restrict__ a, KGrid g, long long total, double dk3,
                                                 double n3, double inv_n3, const double *__restrict__ lk,
                                                 const double *__restrict__ lp, int np, double lk0, double inv_dlk)
{
#pragma clang fp contract(off)
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        int ix, iy, iz;
        double kx, ky, kz;
        kvec(g, e, ix, iy, iz, kx, ky, kz);
        const double k2 = kx * kx + ky * ky + kz * kz;
        if (k2 == 0.0) {
            a[e] = make_float2(0.f, 0.f);
            continue;
        }
        const double amp = sqrt(pk_eval(lk, lp, np, sqrt(k2), lk0, inv_dlk) * dk3 * n3);
        a[e] = cmul(a[e], amp * inv_n3, 0.0);
    }
}

// one spectrum from delta_k: which = 0..2: psi_i = i k_i / k^2 (1LPT,
// Nyquist planes zeroed); 3..8: phi_ab = -k_a k_b / k^2 (ab = 11, 22, 33,
// 12, 13, 23); 9..11: psi2_i = -i k_i / k^2 (2LPT, Nyquist zeroed); all
// times scale
__global__ void __launch_bounds__(256) k_lpt(const float2 *__restrict__ in, float2 *__restrict__ out, KGrid g,
                                             long long total, int which, double scale)
{
#pragma clang fp contract(off)
    const int A[6] = {0, 1, 2, 0, 0, 1}, B[6] = {0, 1, 2, 1, 2, 2};
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        int ix, iy, iz;
        double k[3];
        kvec(g, e, ix, iy, iz, k[0], k[1], k[2]);
        const double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
        const bool nyq = ix == g.nk - 1 || iy == g.n / 2 || iz == g.n / 2;
        float2 r = make_float2(0.f, 0.f);
        if (which < 3) {
            if (k2 != 0.0 && !nyq) r = cmul(in[e], 0.0, k[which] / k2 * scale);
        } else if (which < 9) {
            const int q = which - 3;
            if (k2 != 0.0) r = cmul(in[e], -k[A[q]] * k[B[q]] / k2 * scale, 0.0);
        } else {
            if (k2 != 0.0 && !nyq) r = cmul(in[e], 0.0, -k[which - 9] / k2 * scale);
        }
        out[e] = r;
    }
}

// _compute_laplacian: k^2 delta_k with k and the product in Float32,
// then the two normalisations (exact powers of two for power-of-two n)
__global__ void __launch_bounds__(256) k_lapk(const float2 *__restrict__ in, float2 *__restrict__ out, int n, int nk,
                                              long long total, float dkf, float s1, float s2)
{
#pragma clang fp contract(off)
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const int ix = (int)(e % nk);
        const long long r = e / nk;
        const int iy = (int)(r % n), iz = (int)(r / n);
        const int nyq = n / 2;
        const float kx = (float)ix * dkf;
        const float ky = (float)(iy <= nyq ? iy : iy - n) * dkf;
        const float kz = (float)(iz <= nyq ? iz : iz - n) * dkf;
        const float k2 = kx * kx + ky * ky + kz * kz;
        const float2 v = in[e];
        out[e] = make_float2(v.x * k2 * s1 * s2, v.y * k2 * s1 * s2);
    }
}

// the 2LPT source, left to right in Float32: step 0: src = p11 p22 - p12^2;
// 1: src = src + p11 p33 - p13^2 (b = p33, c = p13); 2: src = src + p22 p33 -
// p23^2 (a = p22, b = p33, c = p23)
__global__ void __launch_bounds__(256) k_src2(float *__restrict__ src, const float *__restrict__ a,
                                              const float *__restrict__ b, const float *__restrict__ c, long long total,
                                              int step)
{
#pragma clang fp contract(off)
    for (long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x; e < total;
         e += (long long)gridDim.x * blockDim.x) {
        const float cc = c[e] * c[e];
        if (step == 0) src[e] = a[e] * b[e] - cc;
        else src[e] = (src[e] + a[e] * b[e]) - cc;
    }
}

int launch_noise(pp_ctx *ctx, float *out, int64_t ncells, uint64_t seed);  // pp_filter.hip

// ------------------------------------------------------- line-transform path
// The passes of a periodic grid with line transforms (pp_fft.h).

// spectra of a row pair from its transformed line
__device__ __forceinline__ void store_row_pair(const RowAddr &at, const LineFft &P, const SpecGeo &g, float2 *out,
                                               long long r, bool two, int jj)
{
    const long long z = r / g.n, z2 = (r + 1) / g.n;
    float2 *a = out + g.row((int)z, (int)(r - z * g.n)), *b = out + g.row((int)z2, (int)(r + 1 - z2 * g.n));
#pragma unroll
    for (int q = 0; q < kRowBins; q++) {
        const int k = jj + q * P.tj;
        if (k >= g.nk) break;
        float2 va, vb;
        split_rows(at(k), at(k == 0 ? 0 : g.n - k), va, vb);
        a[k] = va;
        if (two) b[k] = vb;
    }
}

// x-forward of the white noise, drawn where it is transformed: the 2 n cells
// of a row pair are n whole Threefry counter pairs
template <int M>
__global__ void __launch_bounds__(512) k_rows_noise(SpecGeo g, LineFft P, float2 *__restrict__ out, uint64_t seed)
{
    extern __shared__ float2 lds[];
    const int n = g.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, rp = (long long)blockIdx.x * (blockDim.x / P.tj) + line, r = 2 * rp;
    const RowAddr at(lds + line * row_pitch(n));
    const bool two = r + 1 < rows;
    if (r < rows) {
        for (int e = jj; e < n; e += P.tj) {
            double g1, g2;
            threefry_normals((uint64_t)(rp * n + e), seed, g1, g2);
            const int c1 = 2 * e, c2 = c1 + 1;
            const float v1 = (float)g1, v2 = (float)g2;
            if (c1 < n) at(c1).x = v1;
            else at(c1 - n).y = two ? v1 : 0.f;
            if (c2 < n) at(c2).x = v2;
            else at(c2 - n).y = two ? v2 : 0.f;
        }
    }
    __syncthreads();
    float2 x[kLineEpt];
    line_run<-1, M, true, true>(at, P, jj, x);
    if (r < rows) store_row_pair(at, P, g, out, r, two, jj);
}

// x-forward of a real field
template <int M>
__global__ void __launch_bounds__(512) k_rows_real(SpecGeo g, LineFft P, const float *__restrict__ in, float2 *__restrict__ out)
{
    extern __shared__ float2 lds[];
    const int n = g.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, r = 2 * ((long long)blockIdx.x * (blockDim.x / P.tj) + line);
    const RowAddr at(lds + line * row_pitch(n));
    const bool two = r + 1 < rows;
    float2 x[kLineEpt] = {};
    if (r < rows) {
        const float *pa = in + r * n, *pb = two ? pa + n : pa;
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) {
            const int e = min(jj + q * P.tj, n - 1);
            x[q] = make_float2(pa[e], pb[e]);
        }
    }
    line_run<-1, M, false, true>(at, P, jj, x);
    if (r < rows) store_row_pair(at, P, g, out, r, two, jj);
}

// y-forward, in place: planes of kz or z
template <int M>
__global__ void __launch_bounds__(1024) k_cols_y_fwd(SpecGeo g, LineFft P, ColGrid C, float2 *__restrict__ s)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const LineY io(g, s, t.plane, 0, 1, t.kx);
    float2 x[kLineEpt];
    line_load(P, t.jj, x, io);
    line_run<-1, M, false, false>(at, P, t.jj, x);
    line_store(P, t.jj, x, io);
}

// z-forward, transfer, z-inverse: one read of the spectrum gives every
// output.  The mode X (times its amplitude with A.amp) stays in registers
// while the outputs are formed one after the other in LDS.
template <int M>
__global__ void __launch_bounds__(1024) k_cols_z(SpecGeo g, LineFft P, ColGrid C, ZArgs A)
{
#pragma clang fp contract(off)
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const int n = g.n, iy = t.plane, half = n / 2;
    float2 X[kLineEpt];
    line_load(P, t.jj, X, LineZ(g, A.in, iy, t.kx));
    line_run<-1, M, false, false>(at, P, t.jj, X);
    const int kx = min(t.kx, g.nk - 1), fy = iy < (n + 1) / 2 ? iy : iy - n, ixy = kx * kx + fy * fy;
    const bool nyq_xy = kx == g.nk - 1 || iy == half;
    Two ik[kLineEpt];  // 1 / |i|^2
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = min(t.jj + q * P.tj, n - 1), fz = e < (n + 1) / 2 ? e : e - n, i2 = ixy + fz * fz;
        if (A.amp) X[q] = ftimes(A.amp[i2], X[q]);
        ik[q] = i2 == 0 ? Two{0.f, 0.f} : finverse((float)i2);
    }
    for (int o = 0; o < A.nout; o++) {
        const int kind = A.out[o].kind, nyq = A.out[o].nyq;
        int jj = t.jj;
        asm volatile("" : "+v"(jj));  // per-element values are formed anew, not held for every output
        float2 x[kLineEpt];
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) {
            const int e = jj + q * P.tj, fz = e < (n + 1) / 2 ? e : e - n;
            if (kind == Z_X) {
                x[q] = X[q];
            } else if (kind == Z_K2F) {
                // k and the product in Float32 (_compute_laplacian); the spectrum
                // holds the first of the two normalisations
                const float fx = (float)kx * A.dkf, fyf = (float)(iy <= half ? iy : iy - n) * A.dkf,
                            fzf = (float)(e <= half ? e : e - n) * A.dkf;
                const float f = (fx * fx + fyf * fyf + fzf * fzf) * A.scale;
                x[q] = make_float2(X[q].x * f, X[q].y * f);
            } else if (kind == Z_K2) {
                const float f = (float)(ixy + fz * fz);
                x[q] = make_float2(X[q].x * f, X[q].y * f);
            } else {
                const float iz = (float)fz;
                x[q] = ftimes(kind == Z_INV ? ik[q] : ftimes(ik[q], kind == Z_INV_Z ? iz : iz * iz), X[q]);
            }
            if (nyq && (nyq_xy || e == half)) x[q] = make_float2(0.f, 0.f);
        }
        line_run<1, M, false, false>(at, P, jj, x);
        line_store(P, jj, x, LineZ(g, A.out[o].p, iy, t.kx));
    }
}

__global__ void __launch_bounds__(256) k_amp_table(PkLog T, double mult2, double dk3, double n3, long long count,
                                                   Two *__restrict__ out)
{
#pragma clang fp contract(off)
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= count) return;
    const double k2 = (double)i * mult2;
    const double a =
        i == 0 ? 0.0 : sqrt(pk_eval(T.lk, T.lp, T.np, sqrt(k2), T.even[0], T.even[1]) * dk3 * n3) * (1.0 / n3);
    const float h = (float)a;
    out[i] = Two{h, isfinite(h) ? (float)(a - (double)h) : 0.f};
}

// logarithms of k and P (one block) and whether log k is evenly spaced, to
// 1e-9 of the spacing
__global__ void __launch_bounds__(1024) k_pk_log(const double *__restrict__ k, const double *__restrict__ P, int np,
                                                 double *lk, double *__restrict__ lp, double *__restrict__ even)
{
    __shared__ int uneven;
    if (threadIdx.x == 0) uneven = 0;
    for (int q = threadIdx.x; q < np; q += blockDim.x) {
        lk[q] = log(k[q]);
        lp[q] = log(P[q]);
    }
    __syncthreads();
    const double d = (lk[np - 1] - lk[0]) / (np - 1);
    bool off = np < 3 || !(d > 0.0);
    for (int q = 1 + threadIdx.x; q < np; q += blockDim.x) off = off || fabs((lk[q] - lk[q - 1]) - d) > 1e-9 * d;
    if (off) uneven = 1;
    __syncthreads();
    if (threadIdx.x == 0) {
        even[0] = lk[0];
        even[1] = uneven ? 0.0 : 1.0 / d;
    }
}

// y-inverse of the arrays of Y, each times the powers of iy asked for:
// z planes, grid y the arrays; an output may be its input
template <int M>
__global__ void __launch_bounds__(1024, M == kLineReg ? 8 : 4) k_cols_y_inv(SpecGeo g, LineFft P, ColGrid C, YArgs Y)
{
    extern __shared__ float2 lds[];
    const ColTile t = col_tile(C);
    if (t.plane < 0) return;
    const ColAddr<M != kLineAny> at(lds, t.l, C.logl);
    const YArgs::Arr &R = Y.arr[blockIdx.y];
    const int n = g.n;
    float2 X[kLineEpt];
    line_load(P, t.jj, X, LineY(g, R.in, t.plane, 0, 1, t.kx));
    for (int o = 0; o < 3; o++) {
        float2 *w = R.out[o];  // iy^o
        if (!w) continue;
        int jj = t.jj;
        asm volatile("" : "+v"(jj));
        float2 x[kLineEpt];
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) {
            const int e = jj + q * P.tj;
            const float iy = (float)(e < (n + 1) / 2 ? e : e - n), f = o == 0 ? 1.f : o == 1 ? iy : iy * iy;
            x[q] = make_float2(X[q].x * f, X[q].y * f);
        }
        line_run<1, M, false, false>(at, P, jj, x);
        line_store(P, jj, x, LineY(g, w, t.plane, 0, 1, t.kx));
    }
}

// x-inverse: grid (row pairs, outputs)
template <int M>
__global__ void __launch_bounds__(512) k_rows_inv(SpecGeo g, LineFft P, XArgs X)
{
    extern __shared__ float2 lds[];
    const int n = g.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, r = 2 * ((long long)blockIdx.x * (blockDim.x / P.tj) + line);
    const RowAddr at(lds + line * row_pitch(n));
    const bool two = r + 1 < rows;
    const XArgs::Op &O = X.op[blockIdx.y];
    if (r < rows) load_row_pair(at, P, g, O.in, r, two, jj, O.pow, O.imag, O.f, X.top);
    __syncthreads();
    float2 x[kLineEpt];
    line_run<1, M, true, false>(at, P, jj, x);
    if (r < rows) {
        float *pa = O.out + r * n, *pb = pa + n;
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) {
            const int e = jj + q * P.tj;
            if (e < n) {
                pa[e] = x[q].x;
                if (two) pb[e] = x[q].y;
            }
        }
    }
}

// The second-order source: the six potentials of a row pair one after the
// other through the same line, the running sum in registers, then its
// x-forward; only the source's spectrum is written.  The source is quadratic
// in the potentials, whose common sign is left out.  delta: null for
// run_tile's source p11 p22 + (p11 + p22) p33 - p12^2 - p13^2 - p23^2, else
// the split tiles' delta^2 / 2 - sum phi_dd^2 / 2 - sum phi_ab^2, in Float32.
template <int M>
__global__ void __launch_bounds__(512) k_rows_src(SpecGeo g, LineFft P, SrcArgs S)
{
#pragma clang fp contract(off)
    extern __shared__ float2 lds[];
    const int n = g.n, line = threadIdx.x / P.tj, jj = threadIdx.x - line * P.tj;
    const long long rows = (long long)n * n, r = 2 * ((long long)blockIdx.x * (blockDim.x / P.tj) + line);
    const RowAddr at(lds + line * row_pitch(n));
    const bool two = r + 1 < rows, live = r < rows;
    float2 src[kLineEpt], sum[kLineEpt];
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = min(jj + q * P.tj, n - 1);
        src[q] = sum[q] = make_float2(0.f, 0.f);
        if (S.delta && live) {
            const float d1 = S.delta[r * n + e], d2 = two ? S.delta[(r + 1) * n + e] : 0.f;
            src[q] = make_float2((d1 * d1) * 0.5f, (d2 * d2) * 0.5f);
        }
    }
    for (int v = 0; v < 6; v++) {  // 11 22 33 12 13 23
        int j2 = jj;
        asm volatile("" : "+v"(j2));
        __syncthreads();
        if (live) load_row_pair(at, P, g, S.in[v], r, two, j2, S.pow[v], false, S.f, g.nk);
        __syncthreads();
        float2 x[kLineEpt];
        line_run<1, M, true, false>(at, P, j2, x);
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) {
            const float2 p = x[q];
            if (S.delta || v >= 3) {
                const float co = v < 3 ? 0.5f : 1.0f;
                src[q].x = src[q].x - (p.x * p.x) * co;
                src[q].y = src[q].y - (p.y * p.y) * co;
            } else {
                src[q].x = src[q].x + sum[q].x * p.x;
                src[q].y = src[q].y + sum[q].y * p.y;
                sum[q] = fadd(sum[q], p);
            }
        }
    }
    if (!two) {
#pragma unroll
        for (int q = 0; q < kLineEpt; q++) src[q].y = 0.f;
    }
    line_run<-1, M, false, true>(at, P, jj, src);
    if (live) store_row_pair(at, P, g, S.out, r, two, jj);
}

// ---- launches
static unsigned row_blocks(const SpecGeo &g, const LineShape &s)
{
    const long long pairs = ((long long)g.n * g.n + 1) / 2;
    return (unsigned)((pairs + s.nl - 1) / s.nl);
}

int grid_plan(pp_ctx *ctx, int n, GridPlan *G)
{
    PP_CHECK(line_plan(ctx, n, &G->row));
    G->col = G->row;
    G->rs = row_shape(G->row);
    G->cs = col_shape(G->col, 512);
    // the y passes fit 64 registers, so that two workgroups of 1024 threads
    // (16 columns of a long line) share a CU; the z pass and the radices 5 and
    // 7 take more and keep to 512 threads
    G->ycol = G->col;
    G->ys = col_shape(G->ycol, G->col.mode == kLineReg ? 1024 : 512);
    G->g = spec_geo(n, n);
    G->stream = ctx->stream;
    return PP_OK;
}

int rows_real(const GridPlan &G, const float *in, float2 *out)
{
    PP_LINE_LAUNCH(G.row, k_rows_real, dim3(row_blocks(G.g, G.rs)), dim3(G.rs.block), G.rs.lds, G.stream, G.g, G.row, in,
                       out);
    return PP_OK;
}

int rows_noise(const GridPlan &G, uint64_t seed, float2 *out)
{
    PP_LINE_LAUNCH(G.row, k_rows_noise, dim3(row_blocks(G.g, G.rs)), dim3(G.rs.block), G.rs.lds, G.stream, G.g, G.row,
                       out, seed);
    return PP_OK;
}

int cols_y_fwd(const GridPlan &G, float2 *s)
{
    const ColGrid C = G.ys.grid(G.g.nk, G.g.n, 1);
    PP_LINE_LAUNCH(G.ycol, k_cols_y_fwd, dim3(C.blocks()), dim3(G.ys.block), G.ys.lds, G.stream, G.g, G.ycol, C, s);
    return PP_OK;
}

int cols_z(const GridPlan &G, const ZArgs &A)
{
    const ColGrid C = G.cs.grid(G.g.nk, G.g.n, kColXCD);
    PP_LINE_LAUNCH(G.col, k_cols_z, dim3(C.blocks()), dim3(G.cs.block), G.cs.lds, G.stream, G.g, G.col, C, A);
    return PP_OK;
}

int cols_y_inv(const GridPlan &G, const YArgs &Y)
{
    const ColGrid C = G.ys.grid(G.g.nk, G.g.n, 1);
    PP_LINE_LAUNCH(G.ycol, k_cols_y_inv, dim3(C.blocks(), Y.narr), dim3(G.ys.block), G.ys.lds, G.stream, G.g,
                   G.ycol, C, Y);
    return PP_OK;
}

int rows_inv(const GridPlan &G, const XArgs &X)
{
    PP_LINE_LAUNCH(G.row, k_rows_inv, dim3(row_blocks(G.g, G.rs), X.nop), dim3(G.rs.block), G.rs.lds, G.stream, G.g,
                       G.row, X);
    return PP_OK;
}

int rows_src(const GridPlan &G, const SrcArgs &S)
{
    PP_LINE_LAUNCH(G.row, k_rows_src, dim3(row_blocks(G.g, G.rs)), dim3(G.rs.block), G.rs.lds, G.stream, G.g, G.row, S);
    return PP_OK;
}

int amp_table(pp_ctx *ctx, const PkLog &T, double mult, double dk3, double n3, long long count, Two *out)
{
    hipLaunchKernelGGL(k_amp_table, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, ctx->stream, T, mult * mult,
                       dk3, n3, count, out);
    PP_HIP(hipGetLastError());
    return PP_OK;
}

int pk_log_device(pp_ctx *ctx, const pp_pk_table *pk, double *buf, PkLog *out)
{
    const int np = pk->npk;
    double *lk = buf, *lp = lk + np, *k = lp + np, *P = k + np, *even = P + np;
    PP_HIP(hipMemcpyAsync(k, pk->k, np * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    PP_HIP(hipMemcpyAsync(P, pk->P, np * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    hipLaunchKernelGGL(k_pk_log, dim3(1), dim3(1024), 0, ctx->stream, (const double *)k, (const double *)P, np, lk, lp,
                       even);
    PP_HIP(hipGetLastError());
    *out = PkLog{lk, lp, even, np};
    return PP_OK;
}

// The six potentials' arrays: y-inverses of X / |i|^2, iz X / |i|^2, iz^2 X / |i|^2
// times powers of iy, in the order 11 22 33 12 13 23 with their powers of ix
void src_inputs(SrcArgs &S, const float2 *a, const float2 *a1, const float2 *a2, const float2 *b, const float2 *b1,
                const float2 *c)
{
    const float2 *in[6] = {a, a2, c, a1, b, b1};
    const int pow[6] = {2, 0, 0, 1, 1, 0};
    for (int q = 0; q < 6; q++) {
        S.in[q] = in[q];
        S.pow[q] = pow[q];
    }
}

// eta2 = -i k / k^2 src_k from the x-spectrum of the source in s[0] (three
// arrays of work space)
int second_order(const GridPlan &G, float2 *const s[3], double mult, double scale, float *const out[3])
{
    PP_CHECK(cols_y_fwd(G, s[0]));
    ZArgs Z{};
    Z.in = s[0];
    Z.add(s[0], Z_INV, 1);
    Z.add(s[1], Z_INV_Z, 1);
    PP_CHECK(cols_z(G, Z));
    YArgs Y{};
    Y.add(s[0], s[0], s[2], nullptr);
    Y.add(s[1], s[1], nullptr, nullptr);
    PP_CHECK(cols_y_inv(G, Y));
    XArgs X{};
    X.add(s[0], out[0], 1, true, -scale / mult);
    X.add(s[2], out[1], 0, true, -scale / mult);
    X.add(s[1], out[2], 0, true, -scale / mult);
    return rows_inv(G, X);
}

// pp_make_tile_fields with line transforms.  The spectrum of delta is the
// noise's times the amplitude (rfft of its own inverse transform), so delta
// is not transformed again.
static int make_tile_lines(pp_ctx *ctx, int n, double boxsize, uint64_t seed, const pp_pk_table *pk, pp_tile_fields *f)
{
    const bool lpt2 = f->eta2x != nullptr;
    GridPlan G;
    PP_CHECK(grid_plan(ctx, n, &G));
    const size_t arr = G.g.size(n);  // complex values of one array
    // delta / source, A', B', iy A', L, and with 2LPT A, B, C, iy A, iy^2 A, iy B
    const int narr = 4 + (f->lapd ? 1 : 0) + (lpt2 ? 6 : 0);
    PP_CHECK(ctx->d_spec.grow(arr * narr * sizeof(float2)));
    float2 *s[11];
    for (int q = 0; q < narr; q++) s[q] = ctx->d_spec.as<float2>() + arr * q;
    float2 *L = f->lapd ? s[4] : nullptr, **W = s + 4 + (f->lapd ? 1 : 0);
    PP_CHECK(rows_noise(G, seed, s[0]));
    PP_CHECK(cols_y_fwd(G, s[0]));
    const double dk = 2.0 * M_PI / boxsize, mult = ((double)n * dk) / (double)n, n3 = (double)n * n * n;
    const long long count = amp_count(n / 2);
    PP_CHECK(ctx->d_misc.grow(pk_log_doubles(pk->npk) * sizeof(double) + count * sizeof(Two)));
    double *d_pk = ctx->d_misc.as<double>();
    Two *amp = (Two *)(d_pk + pk_log_doubles(pk->npk));
    PkLog T;
    PP_CHECK(pk_log_device(ctx, pk, d_pk, &T));
    PP_CHECK(amp_table(ctx, T, mult, dk * dk * dk, n3, count, amp));
    ZArgs Z{};
    Z.in = s[0];
    Z.amp = amp;
    Z.dkf = (float)dk;
    Z.scale = (float)(1.0 / n3);
    Z.add(s[0], Z_X, 0);
    Z.add(s[1], Z_INV, 1);
    Z.add(s[2], Z_INV_Z, 1);
    if (L) Z.add(L, Z_K2F, 0);
    if (lpt2) {
        Z.add(W[0], Z_INV, 0);
        Z.add(W[1], Z_INV_Z, 0);
        Z.add(W[2], Z_INV_ZZ, 0);
    }
    PP_CHECK(cols_z(G, Z));
    YArgs Y{};
    Y.add(s[0], s[0], nullptr, nullptr);
    Y.add(s[1], s[1], s[3], nullptr);
    Y.add(s[2], s[2], nullptr, nullptr);
    if (L) Y.add(L, L, nullptr, nullptr);
    if (lpt2) {
        Y.add(W[0], W[0], W[3], W[4]);
        Y.add(W[1], W[1], W[5], nullptr);
        Y.add(W[2], W[2], nullptr, nullptr);
    }
    PP_CHECK(cols_y_inv(G, Y));
    XArgs X{};
    X.add(s[0], f->delta, 0, false, 1.0);
    X.add(s[1], f->etax, 1, true, 1.0 / mult);
    X.add(s[3], f->etay, 0, true, 1.0 / mult);
    X.add(s[2], f->etaz, 0, true, 1.0 / mult);
    if (L) X.add(L, f->lapd, 0, false, 1.0);
    PP_CHECK(rows_inv(G, X));
    if (lpt2) {
        SrcArgs S{};
        S.f = two(1.0);
        S.out = s[0];
        src_inputs(S, W[0], W[3], W[4], W[1], W[5], W[2]);
        PP_CHECK(rows_src(G, S));
        float2 *w[3] = {s[0], s[1], s[2]};
        float *out[3] = {f->eta2x, f->eta2y, f->eta2z};
        PP_CHECK(second_order(G, w, mult, 1.0 / n3, out));
    }
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}

// Meshes on line transforms.  Odd multiples of 15 stay with rocFFT, which
// rounds less in them (the density's rms error at 45, 75, 135, 225, 375: 1.85,
// 2.05, 2.12, 2.26, 2.58e-7 against 2.04, 2.22, 2.38, 2.53, 2.67 on the lines);
// at the 73 other lengths measured between 16 and 512 no field's error on the
// lines is larger than 0.97 of rocFFT's, all fields together 0.48 to 0.78.
static bool lines_for(int n) { return line_supported(n) && (n % 2 == 0 || n % 15 != 0); }

}  // namespace pp

using namespace pp;

extern "C" int pp_make_tile_fields(pp_ctx *ctx, int n, double boxsize, uint64_t seed, const pp_pk_table *pk,
                                   pp_tile_fields *f)
{
    PP_ARG(ctx && pk && f && f->delta && f->etax && f->etay && f->etaz, "NULL argument");
    PP_ARG(n >= 4 && boxsize > 0, "bad n=%d / boxsize", n);
    PP_ARG(pk->npk >= 2 && pk->k && pk->P, "P(k) table needs >= 2 rows");
    const bool lpt2 = f->eta2x != nullptr;
    PP_ARG(!lpt2 || (f->eta2y && f->eta2z), "eta2 outputs come as a set of three");
    for (int q = 0; q < pk->npk; q++) {
        PP_ARG(pk->k[q] > 0 && pk->P[q] > 0, "P(k) table row %d not positive", q);
        PP_ARG(q == 0 || pk->k[q] > pk->k[q - 1], "P(k) table k not increasing at row %d", q);
    }
    PP_CHECK(ensure_device(ctx));
    if (lines_for(n)) {
        const int rc = make_tile_lines(ctx, n, boxsize, seed, pk, f);
        if (rc != PP_ERR_OOM) return rc;  // 44 to 50 B a cell are not there: rocFFT's route takes 24
    }
    PP_CHECK(fft_prepare(ctx, n));
    const int nk = n / 2 + 1;
    const long long total = (long long)nk * n * n;
    const size_t N = (size_t)n * n * n, cb = (size_t)total * sizeof(float2), rb = N * sizeof(float);
    // device buffers: the log P(k) table, delta_k, one work spectrum, and
    // with 2LPT four real fields (the diagonal potentials and the source)
    std::vector<double> lk(pk->npk), lp(pk->npk);
    for (int q = 0; q < pk->npk; q++) {
        lk[q] = log(pk->k[q]);
        lp[q] = log(pk->P[q]);
    }
    PP_CHECK(ctx->d_misc.grow(2 * pk->npk * sizeof(double)));
    double *d_lk = ctx->d_misc.as<double>(), *d_lp = d_lk + pk->npk;
    PP_HIP(hipMemcpyAsync(d_lk, lk.data(), pk->npk * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    PP_HIP(hipMemcpyAsync(d_lp, lp.data(), pk->npk * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
    PP_CHECK(ctx->d_k0.grow(cb));
    PP_CHECK(ctx->d_k1.grow(cb));
    float2 *dk0 = ctx->d_k0.as<float2>(), *dk1 = ctx->d_k1.as<float2>();
    const int grid = (int)std::min<long long>((total + 255) / 256, (long long)ctx->num_cu * 16);
    const double dk = 2.0 * M_PI / boxsize;
    KGrid g{n, nk, ((double)n * dk) / (double)n};
    const double inv_n3 = 1.0 / ((double)n * n * n);
    auto c2r = [&](void *in, float *out) -> int {
        void *ib[1] = {in}, *ob[1] = {(void *)out};
        PP_FFT(rocfft_execute(ctx->fftp->c2r, ib, ob, ctx->fftp->info));
        return PP_OK;
    };
    auto r2c = [&](const float *in, void *out) -> int {
        void *ib[1] = {(void *)in}, *ob[1] = {out};
        PP_FFT(rocfft_execute(ctx->fftp->r2c, ib, ob, ctx->fftp->info));
        return PP_OK;
    };
    // 1. delta: noise -> rfft -> sqrt(P dk^3 n^3) -> normalised irfft
    PP_CHECK(launch_noise(ctx, f->delta, (int64_t)N, seed));
    PP_CHECK(r2c(f->delta, dk0));
    hipLaunchKernelGGL(k_grf_amp, dim3(grid), dim3(256), 0, ctx->stream, dk0, g, total, dk * dk * dk,
                       (double)n * n * n, inv_n3, (const double *)d_lk, (const double *)d_lp, pk->npk, lk[0],
                       pk_uniform_inv_spacing(lk.data(), pk->npk));
    PP_HIP(hipGetLastError());
    PP_CHECK(c2r(dk0, f->delta));
    // 2. delta_k = rfft(delta), kept in dk0
    PP_CHECK(r2c(f->delta, dk0));
    auto lpt = [&](int which, float *out) -> int {
        hipLaunchKernelGGL(k_lpt, dim3(grid), dim3(256), 0, ctx->stream, (const float2 *)dk0, dk1, g, total, which,
                           inv_n3);
        PP_HIP(hipGetLastError());
        return c2r(dk1, out);
    };
    // 3. 1LPT
    PP_CHECK(lpt(0, f->etax));
    PP_CHECK(lpt(1, f->etay));
    PP_CHECK(lpt(2, f->etaz));
    // 4. Laplacian (before 2LPT reuses delta_k's buffer)
    if (f->lapd) {
        const float s = (float)inv_n3;
        hipLaunchKernelGGL(k_lapk, dim3(grid), dim3(256), 0, ctx->stream, (const float2 *)dk0, dk1, n, nk, total,
                           (float)dk, s, s);
        PP_HIP(hipGetLastError());
        PP_CHECK(c2r(dk1, f->lapd));
    }
    // 5. 2LPT: the source from the six potentials, then its gradient
    if (lpt2) {
        PP_CHECK(ctx->d_field_a.grow(4 * rb));
        float *p11 = ctx->d_field_a.as<float>(), *p22 = p11 + N, *p33 = p22 + N, *src = p33 + N;
        float *tmp = f->eta2x;  // the off-diagonal potentials pass through an output buffer
        PP_CHECK(lpt(3, p11));
        PP_CHECK(lpt(4, p22));
        PP_CHECK(lpt(6, tmp));  // p12
        hipLaunchKernelGGL(k_src2, dim3(grid), dim3(256), 0, ctx->stream, src, (const float *)p11, (const float *)p22,
                           (const float *)tmp, (long long)N, 0);
        PP_HIP(hipGetLastError());
        PP_CHECK(lpt(5, p33));
        PP_CHECK(lpt(7, tmp));  // p13
        hipLaunchKernelGGL(k_src2, dim3(grid), dim3(256), 0, ctx->stream, src, (const float *)p11, (const float *)p33,
                           (const float *)tmp, (long long)N, 1);
        PP_HIP(hipGetLastError());
        PP_CHECK(lpt(8, tmp));  // p23
        hipLaunchKernelGGL(k_src2, dim3(grid), dim3(256), 0, ctx->stream, src, (const float *)p22, (const float *)p33,
                           (const float *)tmp, (long long)N, 2);
        PP_HIP(hipGetLastError());
        PP_CHECK(r2c(src, dk0));
        PP_CHECK(lpt(9, f->eta2x));
        PP_CHECK(lpt(10, f->eta2y));
        PP_CHECK(lpt(11, f->eta2z));
    }
    PP_HIP(hipStreamSynchronize(ctx->stream));
    return PP_OK;
}
