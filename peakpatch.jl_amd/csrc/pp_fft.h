// pp_fft.h -- single-precision line transforms in LDS, the building block of
// the field kernels' three-dimensional transforms.
//
// A 3-D real transform here is three kinds of pass over a half spectrum
// S[kz][ky][kx] (kx fastest): rows along x, columns along y, columns along z.
// Every pass brings whole lines into LDS, transforms them there and lets the
// kernel around it do its own arithmetic on the way in and out, so transfer
// functions, several outputs of one input, the noise draw or a product of
// fields in real space cost no pass over memory of their own.  Each pass is
// bound by HBM: a line element is read and written once.
//
// * Columns: a workgroup takes 2^logl consecutive kx (a run of whole 64- or
//   128-byte pieces in every row) of one (ky or kz) plane.  In LDS the line
//   index is the fastest one, so the accesses of every stage are conflict
//   free whatever the radix.
// * Rows: two real rows travel as the real and imaginary part of one complex
//   line; the half spectra of both are separated (or joined) on the fly.
// * A line is transformed by Stockham stages of radix 8, 4, 2, 3, 5 and 7 (the
//   radices are chosen at run time, so one kernel serves every length up to
//   kLineMax with no larger prime factor).  A stage reads its inputs into
//   registers, then writes them back in place, so one buffer is enough.
//   Twiddles come from a table rounded from Float64 (append_roots), laid out as
//   the butterflies read them.  Vector instructions are the second bound beside
//   HBM (a radix-8 stage takes 14 per element, a pass has room for about a
//   hundred), so addresses advance by scalar strides and the kernels' own
//   Float64 factors are pairs of Float32 numbers (Two), wave numbers whole.
#pragma once

#include <cmath>

#include "pp_common.h"

namespace pp {

constexpr int kLineEpt = 8;    // line elements a thread holds
constexpr int kLineMax = 1024; // longest line
constexpr int kLineMin = 16;
constexpr int kRowBins = 5;    // bins of a half spectrum a thread handles, >= (n / 2 + 1) / tj

// One length's stages, passed to kernels by value.
struct LineFft {
    int n, nst;
    int tj;                  // threads per line, >= n / kLineEpt
    int mode;                // LineMode
    int rad[8], ns[8], nr[8], lin[8];  // radix, sub-length, butterflies; rows: constant strides
    unsigned magic[8];       // floor(2^22 / ns) + 1: j / ns = j magic >> 22 for j < 2048
    int two[8];              // a stage's twiddles exp(-2 pi i k r / (ns R)) at tw[two + k R + r]
    const float2 *tw;
    const float2 *half;      // exp(-pi i k / n), k < n
};

struct LinePlan {
    LineFft f{};
    unsigned long long last_use = 0;
    DevBuf buf;
};

bool line_supported(int n);                              // pp_context.hip
int line_plan(pp_ctx *ctx, int n, LineFft *out);         // a cached plan (the tables stay on the device)

// A half spectrum's layout: rows of pitch complex values, planes of z.
struct SpecGeo {
    int n, nk;
    int pitch;
    long long plane;
    __host__ __device__ long long row(int z, int y) const { return z * plane + (long long)y * pitch; }
    size_t size(int nz) const { return (size_t)plane * nz; }
};

inline SpecGeo spec_geo(int n, int rows)
{
    SpecGeo g;
    g.n = n;
    g.nk = n / 2 + 1;
    g.pitch = (g.nk + 15) / 16 * 16;  // whole tiles of columns: the kernels carry the padding along
    // three 128-byte lines on top keep the planes off a common power of two.
    // (Slabs of 16 z side by side, so that a column along z touches 32 places
    // instead of 512, change nothing: the passes are not bound by address
    // translation.)
    g.plane = (long long)g.pitch * rows + 48;
    return g;
}

// The arithmetic below is written out with its fused operations and without
// contraction by the compiler, so that a transform gives the same bits in every
// kernel it is part of.
#define PP_NO_CONTRACT _Pragma("clang fp contract(off)")

__device__ __forceinline__ float2 fmul(float2 a, float2 b)
{
    PP_NO_CONTRACT
    return make_float2(__builtin_fmaf(a.x, b.x, -(a.y * b.y)), __builtin_fmaf(a.x, b.y, a.y * b.x));
}
__device__ __forceinline__ float2 fmulc(float2 a, float2 b)  // a conj(b)
{
    PP_NO_CONTRACT
    return make_float2(__builtin_fmaf(a.x, b.x, a.y * b.y), __builtin_fmaf(a.y, b.x, -(a.x * b.y)));
}
__device__ __forceinline__ float2 fadd(float2 a, float2 b)
{
    PP_NO_CONTRACT
    return make_float2(a.x + b.x, a.y + b.y);
}
__device__ __forceinline__ float2 fsub(float2 a, float2 b)
{
    PP_NO_CONTRACT
    return make_float2(a.x - b.x, a.y - b.y);
}
// a + s b
__device__ __forceinline__ float2 faxpy(float s, float2 b, float2 a)
{
    return make_float2(__builtin_fmaf(s, b.x, a.x), __builtin_fmaf(s, b.y, a.y));
}
// A Float64 factor as the sum of two Float32 numbers, right to 2^-48: a complex
// value times it takes two instructions a component more than Float32's two and
// is rounded once, as the product in Float64 is (which takes conversions both
// ways besides).
struct Two {
    float h, l;
};
inline Two two(double v)
{
    const float h = (float)v;
    return Two{h, std::isfinite(h) ? (float)(v - (double)h) : 0.f};
}
__device__ __forceinline__ float2 ftimes(Two f, float2 x)
{
    PP_NO_CONTRACT
    return make_float2(__builtin_fmaf(f.h, x.x, f.l * x.x), __builtin_fmaf(f.h, x.y, f.l * x.y));
}
// times a whole number
__device__ __forceinline__ Two ftimes(Two f, float k)
{
    PP_NO_CONTRACT
    const float p = f.h * k;
    return Two{p, __builtin_fmaf(f.l, k, __builtin_fmaf(f.h, k, -p))};
}
// 1 / d of a whole number 0 < d < 2^24
__device__ __forceinline__ Two finverse(float d)
{
    const float r = __builtin_amdgcn_rcpf(d), h = __builtin_fmaf(__builtin_fmaf(-d, r, 1.f), r, r);
    return Two{h, __builtin_fmaf(-d, h, 1.f) * h};
}
// a + s b with a constant s to 48 bits
__device__ __forceinline__ float2 faxpy2(double s, float2 b, float2 a)
{
    const float h = (float)s, l = (float)(s - (double)h);
    return faxpy(h, b, l == 0.f ? a : faxpy(l, b, a));
}
// times -i (forward) or +i (inverse)
template <int SIGN> __device__ __forceinline__ float2 rot(float2 a)
{
    return SIGN < 0 ? make_float2(a.y, -a.x) : make_float2(-a.y, a.x);
}

template <int R, int SIGN> __device__ __forceinline__ void butterfly(float2 *v)
{
    if constexpr (R == 2) {
        const float2 a = v[0], b = v[1];
        v[0] = fadd(a, b);
        v[1] = fsub(a, b);
    } else if constexpr (R == 4) {
        const float2 a = fadd(v[0], v[2]), b = fsub(v[0], v[2]), c = fadd(v[1], v[3]), d = rot<SIGN>(fsub(v[1], v[3]));
        v[0] = fadd(a, c);
        v[1] = fadd(b, d);
        v[2] = fsub(a, c);
        v[3] = fsub(b, d);
    } else if constexpr (R == 8) {
        constexpr float h = 0.70710678118654752f;
        float2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        butterfly<4, SIGN>(e);
        butterfly<4, SIGN>(o);
        // odd half times exp(SIGN 2 pi i r / 8)
        const float2 o1 = fadd(o[1], rot<SIGN>(o[1])), o2 = rot<SIGN>(o[2]), o3 = fsub(rot<SIGN>(o[3]), o[3]);
        v[0] = fadd(e[0], o[0]);
        v[4] = fsub(e[0], o[0]);
        v[1] = faxpy(h, o1, e[1]);
        v[5] = faxpy(-h, o1, e[1]);
        v[2] = fadd(e[2], o2);
        v[6] = fsub(e[2], o2);
        v[3] = faxpy(h, o3, e[3]);
        v[7] = faxpy(-h, o3, e[3]);
    } else {
        // odd prime: the sums p and differences m of conjugate inputs; outputs
        // k and R - k are x0 + sum C p plus or minus i sum S m, as one chain of
        // fma each.  The constants are pairs: in Float32 alone they are half of
        // what such a stage is off (3e-8 of 5e-8), and the same in every mode.
        constexpr double C3[1] = {-0.5}, S3[1] = {0.86602540378443864676};
        constexpr double C5[2] = {0.30901699437494742410, -0.80901699437494742410},
                         S5[2] = {0.95105651629515357212, 0.58778525229247312917};
        constexpr double C7[3] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624},
                         S7[3] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
        const double *C = R == 3 ? C3 : R == 5 ? C5 : C7, *S = R == 3 ? S3 : R == 5 ? S5 : S7;
        constexpr int H = R / 2;
        float2 p[H], m[H], x0 = v[0], sum = v[0];
#pragma unroll
        for (int q = 0; q < H; q++) {
            p[q] = fadd(v[q + 1], v[R - 1 - q]);
            m[q] = rot<SIGN>(fsub(v[q + 1], v[R - 1 - q]));
            sum = fadd(sum, p[q]);
        }
        v[0] = sum;
#pragma unroll
        for (int k = 1; k <= H; k++) {
            float2 a = x0;
#pragma unroll
            for (int q = 0; q < H; q++) {
                const int t = (k * (q + 1)) % R, u = t <= H ? t : R - t;
                a = faxpy2(C[u - 1], p[q], a);
            }
            float2 b = a;
#pragma unroll
            for (int q = H - 1; q >= 0; q--) {
                const int t = (k * (q + 1)) % R, u = t <= H ? t : R - t;
                const double s = t <= H ? S[u - 1] : -S[u - 1];
                a = faxpy2(s, m[q], a);
                b = faxpy2(-s, m[q], b);
            }
            v[k] = a;
            v[R - k] = b;
        }
    }
}

// LDS addresses of this thread's line, in bytes.  Both layouts leave one
// element of padding every eight, so the strided writes of the first stage
// spread over the banks; a stage whose strides are whole eights (or whose
// outputs fill one eight) still advances by a constant.  Columns: element e of
// 2^logl interleaved lines; padded only for the lengths whose strides are
// always whole eights (the others' columns would lose more by it).
template <bool PAD> struct ColAddr {
    char *s;
    int logl;
    static constexpr bool kAlwaysLinear = true;
    __device__ __forceinline__ ColAddr(float2 *lds, int l, int logl) : s((char *)(lds + l)), logl(logl + 3) {}
    __device__ __forceinline__ int off(int e) const { return (PAD ? e + (e >> 3) : e) << logl; }
    __device__ __forceinline__ int step(int e) const { return (PAD ? e + (e >> 3) : e) << logl; }
    __device__ __forceinline__ int step1() const { return 1 << logl; }
    __device__ __forceinline__ float2 &at(int o) const { return *(float2 *)(s + o); }
    __device__ __forceinline__ float2 &operator()(int e) const { return at(off(e)); }
};
struct RowAddr {
    char *s;
    static constexpr bool kAlwaysLinear = false;
    __device__ __forceinline__ explicit RowAddr(float2 *line) : s((char *)line) {}
    __device__ __forceinline__ int off(int e) const { return (e + (e >> 3)) << 3; }
    __device__ __forceinline__ int step(int e) const { return (e + (e >> 3)) << 3; }
    __device__ __forceinline__ int step1() const { return 8; }  // within eight elements
    __device__ __forceinline__ float2 &at(int o) const { return *(float2 *)(s + o); }
    __device__ __forceinline__ float2 &operator()(int e) const { return at(off(e)); }
};
__host__ __device__ constexpr int row_pitch(int n) { return n + n / 8 + 1; }

template <int R, int SIGN, bool FIRST, bool LIN, class A>
__device__ __forceinline__ void line_stage(const A &at, const LineFft &P, int st, int jj)
{
    constexpr int B = (kLineEpt + R - 1) / R;
    const int nr = P.nr[st], ns = P.ns[st];
    // opaque, here and below, so that the addresses of every radix are not
    // formed ahead of the stage loop and held in registers (128 instead of 64)
    asm volatile("" : "+v"(jj));
    // the odd radices' twiddles are loaded where they are used: two or three
    // butterflies of them beside their values would cost half the occupancy
    constexpr bool kAhead = !FIRST && (R & (R - 1)) == 0;
    float2 v[B][R], w[kAhead ? B : 1][R];
    int o[B];
    const float2 *t[B];
    int rd = at.step(nr), wr = at.step(ns);
    asm volatile("" : "+s"(rd), "+s"(wr));
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int j = jj + b * P.tj;
        if (j < nr) {
            const int a = at.off(j);
#pragma unroll
            for (int r = 0; r < R; r++) v[b][r] = LIN ? at.at(a + r * rd) : at(j + r * nr);
            // the twiddles travel while the line's reads finish
            if constexpr (FIRST) {
                o[b] = j * R;
            } else {
                const int h = (int)(__umul24((unsigned)j, P.magic[st]) >> 22) * ns, k = j - h;
                o[b] = h * R + k;
                t[b] = P.tw + (unsigned)(P.two[st] + k * R);
                if constexpr (kAhead) {
#pragma unroll
                    for (int r = 1; r < R; r++) w[b][r] = t[b][r];
                }
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < B; b++) {
        const int j = jj + b * P.tj;
        if (j < nr) {
            if constexpr (!FIRST) {
#pragma unroll
                for (int r = 1; r < R; r++) {
                    const float2 u = kAhead ? w[kAhead ? b : 0][r] : t[b][r];
                    v[b][r] = SIGN < 0 ? fmul(v[b][r], u) : fmulc(v[b][r], u);
                }
            }
            butterfly<R, SIGN>(v[b]);
            const int a = at.off(o[b]);
#pragma unroll
            for (int r = 0; r < R; r++) {
                if (LIN) at.at(a + r * wr) = v[b][r];
                else at(o[b] + r * ns) = v[b][r];
            }
        }
    }
    __syncthreads();
}

template <int R, int SIGN, bool FIRST, class A>
__device__ __forceinline__ void line_stage_any(const A &at, const LineFft &P, int st, int jj)
{
    if (A::kAlwaysLinear || P.lin[st]) line_stage<R, SIGN, FIRST, true>(at, P, st, jj);
    else line_stage<R, SIGN, FIRST, false>(at, P, st, jj);
}

// A column in global memory.  LineZ: along z at row y.  LineY: along y (row0 +
// e stride) at plane z, by 32 bits from an address the workgroup shares.
struct LineZ {
    char *p;
    long long step;
    __device__ __forceinline__ LineZ(const SpecGeo &g, const float2 *s, int y, int kx)
        : p((char *)(s + g.row(0, y) + kx)), step(8 * g.plane)
    {
    }
    __device__ __forceinline__ float2 *at(int e) const { return (float2 *)(p + e * step); }
};
struct LineY {
    char *p;
    unsigned off, step;
    __device__ __forceinline__ LineY(const SpecGeo &g, const float2 *s, int z, int row0, int stride, int kx)
        : p((char *)(s + g.row(z, 0))), off(8u * (unsigned)(row0 * g.pitch + kx)), step(8u * (unsigned)(stride * g.pitch))
    {
    }
    __device__ __forceinline__ float2 *at(int e) const { return (float2 *)(p + (off + (unsigned)e * step)); }
};

// The eight elements e = jj + q tj of a thread from and to global memory
// (elements past the end: the last one, dropped by line_put and line_store).
// All loads are issued before the first is used.
template <class G> __device__ __forceinline__ void line_load(const LineFft &P, int jj, float2 x[kLineEpt], const G &g)
{
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) x[q] = *g.at(min(jj + q * P.tj, P.n - 1));
}
template <class A>
__device__ __forceinline__ void line_put(const A &at, const LineFft &P, int jj, const float2 x[kLineEpt])
{
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = jj + q * P.tj;
        if (e < P.n) at(e) = x[q];
    }
}
template <class A>
__device__ __forceinline__ void line_get(const A &at, const LineFft &P, int jj, float2 x[kLineEpt])
{
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) x[q] = at(min(jj + q * P.tj, P.n - 1));
}
template <class G> __device__ __forceinline__ void line_store(const LineFft &P, int jj, const float2 x[kLineEpt], const G &g)
{
#pragma unroll
    for (int q = 0; q < kLineEpt; q++) {
        const int e = jj + q * P.tj;
        if (e < P.n) *g.at(e) = x[q];
    }
}

// How a length is transformed (LineFft::mode):
//  kLineReg   n = 64 m without factors 5 and 7.  The first and the last stage
//             are of radix 8, whose butterflies take and give exactly the
//             elements e = jj + q tj that a thread holds, so a line enters and
//             leaves in registers: half the LDS traffic and barriers of 512 =
//             8 8 8.
//  kLineReg7  the same with factors 5 or 7 in between.  Their butterflies
//             need more registers, which the kernels of kLineReg are spared.
//  kLineAny   every other length: all stages through LDS.
enum LineMode { kLineReg = 0, kLineReg7 = 1, kLineAny = 2 };

template <int SIGN, bool FIRST, int M, class A>
__device__ __forceinline__ void line_radix(const A &at, const LineFft &P, int st, int jj)
{
    const int R = P.rad[st];
    if (R == 8) line_stage_any<8, SIGN, FIRST>(at, P, st, jj);
    else if (R == 4) line_stage_any<4, SIGN, FIRST>(at, P, st, jj);
    else if (R == 2) line_stage_any<2, SIGN, FIRST>(at, P, st, jj);
    else if (M == kLineReg || R == 3) line_stage_any<3, SIGN, FIRST>(at, P, st, jj);
    else if (R == 5) line_stage_any<5, SIGN, FIRST>(at, P, st, jj);
    else line_stage_any<7, SIGN, FIRST>(at, P, st, jj);
}

// Transforms every line of the workgroup (no scaling); all threads call it.
// Thread jj holds x[q] = element jj + q tj on the way in and out.  IN_LDS: the
// line is in LDS instead, visible to all.  OUT_LDS: it is left there, visible.
// LDS may be written by the caller only after a barrier of its own.
template <int SIGN, int M, bool IN_LDS, bool OUT_LDS, class A>
__device__ __forceinline__ void line_run(const A &at, const LineFft &P, int jj, float2 x[kLineEpt])
{
    if constexpr (M == kLineAny) {
        if constexpr (!IN_LDS) {
            __syncthreads();
            line_put(at, P, jj, x);
            __syncthreads();
        }
        line_radix<SIGN, true, M>(at, P, 0, jj);
        for (int st = 1; st < P.nst; st++) line_radix<SIGN, false, M>(at, P, st, jj);
        if constexpr (!OUT_LDS) line_get(at, P, jj, x);
    } else {
        asm volatile("" : "+v"(jj));
        const int wide = at.step(P.tj), one = at.step1();
        const int own = at.off(jj), first = at.off(8 * jj);
        if constexpr (IN_LDS) {
#pragma unroll
            for (int r = 0; r < 8; r++) x[r] = at.at(own + r * wide);
        }
        __syncthreads();
        butterfly<8, SIGN>(x);
#pragma unroll
        for (int r = 0; r < 8; r++) at.at(first + r * one) = x[r];
        __syncthreads();
        for (int st = 1; st + 1 < P.nst; st++) line_radix<SIGN, false, M>(at, P, st, jj);
        const float2 *t = P.tw + (unsigned)(P.two[P.nst - 1] + 8 * jj);
#pragma unroll
        for (int r = 0; r < 8; r++) x[r] = at.at(own + r * wide);
#pragma unroll
        for (int r = 1; r < 8; r++) x[r] = SIGN < 0 ? fmul(x[r], t[r]) : fmulc(x[r], t[r]);
        butterfly<8, SIGN>(x);
        if constexpr (OUT_LDS) {
#pragma unroll
            for (int r = 0; r < 8; r++) at.at(own + r * wide) = x[r];
            __syncthreads();
        }
    }
}

// kernel<mode> by the length
template <class K, class... Args>
int line_launch(K kernel, dim3 grid, dim3 block, size_t lds, hipStream_t stream, Args... args)
{
    if (lds > 64 * 1024)
        PP_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kernel, grid, block, lds, stream, args...);
    PP_HIP(hipGetLastError());
    return PP_OK;
}
#define PP_LINE_LAUNCH(P, kernel, grid, block, lds, stream, ...)                                                     \
    PP_CHECK((P).mode == kLineReg    ? line_launch(kernel<kLineReg>, grid, block, lds, stream, __VA_ARGS__)           \
             : (P).mode == kLineReg7 ? line_launch(kernel<kLineReg7>, grid, block, lds, stream, __VA_ARGS__)          \
                                     : line_launch(kernel<kLineAny>, grid, block, lds, stream, __VA_ARGS__))

// A workgroup's tile of columns: lines kx of one plane.  Tiles are numbered
// along kx first.  For the z passes each XCD takes one run of them (nx = 8;
// workgroups go round-robin to the eight XCDs), so the neighbours of an
// 8-column tile, which touch the other halves of its 128-byte lines, find them
// in the same L2 (4% of the z pass; the y passes, whose neighbours are one row
// apart, lose 8% by it and go without, nx = 1).
constexpr int kColXCD = 8;
struct ColGrid {
    int logl, nx, tiles, total, per;
    unsigned blocks() const { return (unsigned)(per * nx); }
};
struct ColTile {
    int l, jj, kx;  // kx up to the row's pitch: the padding is carried along
    int plane;      // < 0: no tile (the whole workgroup leaves)
};
__device__ __forceinline__ ColTile col_tile(const ColGrid &C)
{
    const int b = C.nx == 1 ? (int)blockIdx.x : (int)(blockIdx.x % kColXCD) * C.per + (int)(blockIdx.x / kColXCD);
    ColTile t;
    t.plane = b < C.total ? b / C.tiles : -1;
    t.l = threadIdx.x & ((1 << C.logl) - 1);
    t.jj = threadIdx.x >> C.logl;
    t.kx = ((b - t.plane * C.tiles) << C.logl) + t.l;
    return t;
}

// ------------------------------------------------------------- row joins
// Half spectra a, b of two real rows at bin k (0 < k < n / 2, or the bins of
// the DC and Nyquist with real values) as the complex line of both.
template <class A> __device__ __forceinline__ void join_rows(const A &at, int n, int k, float2 a, float2 b)
{
    PP_NO_CONTRACT
    const int kc = k == 0 ? 0 : n - k;
    if (kc == k) {  // DC and, for even n, Nyquist: real
        at(k) = make_float2(a.x, b.x);
    } else {
        at(k) = make_float2(a.x - b.y, a.y + b.x);
        at(kc) = make_float2(a.x + b.y, b.x - a.y);
    }
}

// bins k of both rows from the transformed complex line; kc: the line's bin
// that pairs with k
__device__ __forceinline__ void split_rows(float2 z, float2 zc, float2 &a, float2 &b)
{
    PP_NO_CONTRACT
    a = make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y - zc.y));
    b = make_float2(0.5f * (z.y + zc.y), 0.5f * (zc.x - z.x));
}

// ---------------------------------------------------------------- host side
// Workgroup shapes.  Columns: 2^logl lines of one plane, tj threads each.
// Rows: nl lines (row pairs), tj threads each.
struct LineShape {
    int logl, nl, block;
    size_t lds;
    ColGrid grid(int nk, int planes, int nx) const
    {
        ColGrid c;
        c.logl = logl;
        c.nx = nx;
        c.tiles = (nk + (1 << logl) - 1) >> logl;
        c.total = c.tiles * planes;
        c.per = (c.total + nx - 1) / nx;
        return c;
    }
};
LineShape col_shape(LineFft &P, int max_block);  // sets P.tj
LineShape row_shape(LineFft &P);

}  // namespace pp
