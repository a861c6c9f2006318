// pp_fields.h -- the passes of a periodic grid's transforms with line
// transforms (pp_fft.h), shared by the tile fields of run_tile
// (pp_fields.hip) and of run_multitile_split (pp_split.hip).
#pragma once

#include "pp_fft.h"

namespace pp {

// Transfer of one output of the z pass, i the whole wave numbers (k = mult i):
// X; X k^2 with k and the product as _compute_laplacian forms them, in Float32;
// X |i|^2; X / |i|^2, iz X / |i|^2, iz^2 X / |i|^2 (0 at k = 0).  The factors of
// ix and iy that a displacement or potential takes besides are constant along z
// and follow in the y and x passes, so three z-inverses serve the nine spectra
// of both orders.  Wave numbers and their squares are exact in Float32, the
// amplitude (from a table over |i|^2), 1 / |i|^2 and the field's constant (mult
// and the normalisation, in the x pass) are pairs (Two): a pass rounds a mode
// once, as a Float64 factor does, and no unit of length overflows on the way.
enum ZKind { Z_X = 0, Z_K2F, Z_K2, Z_INV, Z_INV_Z, Z_INV_ZZ };

struct ZArgs {
    const float2 *in;
    int nout;
    struct Out {
        float2 *p;
        int kind, nyq;  // nyq: the Nyquist planes are zeroed
    } out[7];
    const Two *amp;    // amplitude by |i|^2, or null
    float dkf, scale;  // Z_K2F's k of an index and normalisation
    void add(float2 *p, int kind, int nyq) { out[nout++] = Out{p, kind, nyq}; }
};

struct YArgs {
    int narr;
    struct Arr {
        const float2 *in;
        float2 *out[3];  // times 1, iy, iy^2; null: not wanted
    } arr[7];
    void add(const float2 *in, float2 *o0, float2 *o1, float2 *o2) { arr[narr++] = Arr{in, {o0, o1, o2}}; }
};

struct XArgs {
    int nop;
    struct Op {
        const float2 *in;
        float *out;
        int pow;    // power of ix
        bool imag;  // the factor is i f ix^pow, else f ix^pow
        Two f;
    } op[5];
    int top = 1 << 30;  // bins above it are zero and not read
    void add(const float2 *in, float *out, int pow, bool imag, double f) { op[nop++] = Op{in, out, pow, imag, two(f)}; }
};

struct SrcArgs {
    const float2 *in[6];  // potentials 11 22 33 12 13 23
    int pow[6];
    const float *delta;
    Two f;  // the potentials' constant
    float2 *out;
};

// The rows of a P(k) table (device, npk log k then npk log P) and, for rows
// evenly spaced in log k, {first log k, 1 / spacing}, else {.., 0}.
struct PkLog {
    const double *lk, *lp, *even;
    int np;
};
inline size_t pk_log_doubles(int npk) { return 4 * (size_t)npk + 2; }
// Copies the table into buf (pk_log_doubles values) and takes the logarithms
// there (on the host they took as long as a 128^3 tile's kernels).
int pk_log_device(pp_ctx *ctx, const pp_pk_table *pk, double *buf, PkLog *out);

// sqrt(P(k) dk^3 n^3) / n^3 at k^2 = mult^2 i for i = 0 .. 3 imax^2 (0 at i = 0).
// A mode's amplitude in the kernels was the bigger part of their Float64 work:
// the table holds a few hundred thousand values for the up to 10^9 modes of a
// grid.
inline long long amp_count(int imax) { return 3ll * imax * imax + 1; }
int amp_table(pp_ctx *ctx, const PkLog &T, double mult, double dk3, double n3, long long count, Two *out);

// the line of a row pair from an x-spectrum times f ix^pow or i f ix^pow; bins
// above top are zero
__device__ __forceinline__ void load_row_pair(const RowAddr &at, const LineFft &P, const SpecGeo &g,
                                              const float2 *in, long long r, bool two, int jj, int pow, bool imag,
                                              Two f, int top)
{
    const long long z = r / g.n, z2 = (r + 1) / g.n;
    const float2 *a = in + g.row((int)z, (int)(r - z * g.n)), *b = in + g.row((int)z2, (int)(r + 1 - z2 * g.n));
    float2 va[kRowBins], vb[kRowBins];
#pragma unroll
    for (int q = 0; q < kRowBins; q++) {
        const int k = jj + q * P.tj, kc = min(k, g.nk - 1);
        va[q] = k <= top ? a[kc] : make_float2(0.f, 0.f);
        vb[q] = two && k <= top ? b[kc] : make_float2(0.f, 0.f);
    }
#pragma unroll
    for (int q = 0; q < kRowBins; q++) {
        const int k = jj + q * P.tj;
        if (k >= g.nk) break;
        const float ix = (float)k;
        const Two c = pow == 0 ? f : ftimes(f, pow == 1 ? ix : ix * ix);
        const float2 u = ftimes(c, va[q]), v = ftimes(c, vb[q]);
        join_rows(at, g.n, k, imag ? make_float2(-u.y, u.x) : u, imag ? make_float2(-v.y, v.x) : v);
    }
}

struct GridPlan {
    LineFft row, col, ycol;
    LineShape rs, cs, ys;  // rows; columns along z; columns along y
    SpecGeo g;
    hipStream_t stream;
};

int grid_plan(pp_ctx *ctx, int n, GridPlan *G);
int rows_real(const GridPlan &G, const float *in, float2 *out);
int rows_noise(const GridPlan &G, uint64_t seed, float2 *out);
int cols_y_fwd(const GridPlan &G, float2 *s);
int cols_z(const GridPlan &G, const ZArgs &A);
int cols_y_inv(const GridPlan &G, const YArgs &Y);
int rows_inv(const GridPlan &G, const XArgs &X);
int rows_src(const GridPlan &G, const SrcArgs &S);
void src_inputs(SrcArgs &S, const float2 *a, const float2 *a1, const float2 *a2, const float2 *b, const float2 *b1,
                const float2 *c);
int second_order(const GridPlan &G, float2 *const s[3], double mult, double scale, float *const out[3]);

}  // namespace pp
