// grid_spectral.h -- the grid model's operator (OQ_K_FFT_GRID with K_fm and
// K_mf along strike) applied in the frequency domain: index arithmetic and
// block programs of the three kernels, over plain pointers.  Included by
// rhs.hip; also compiled for the host, one thread per block, by the
// bounds-checked emulation in tests/emul.
//
// Every block of the operator is a convolution (see MmGrid):
//   K_ff  along strike, length L >= 2 nx - 1 (real spectrum K[f][l][j]);
//   K_fm  out[b][a0 + m k] = sum_q sum_jx F[b][q][a0 + m (k - jx)] s[q][jx]:
//         for each residue a0 = a mod m of the fault row b a convolution over
//         the mantle columns, length P >= ceil(nx / m) + nxc - 1;
//   K_mf  out[q][jx] = sum_{b, a0} sum_k G[q][b][m (jx - k) - a0] s[b][a0 + m k]:
//         the transpose, same P;
//   K_mm  out[PO] = sum_PI T[PO][PI] * s[PI], 2D, P x Py (P >= 2 nxc - 1, Py >= 2 ny - 1).
// In the frequency domain they are products of a vector with one matrix per
// bin, f <= P / 2: F (Q columns, nxi m rows), G (nxi m columns, Q rows) and,
// per (fy, f), M (npl x npl), with Q = 6 ny nz mantle lines and npl = 6 nz
// planes.  One RHS is three launches: forward transforms (with the prologue),
// the products, inverse transforms (with the friction update).  At the
// composite model the products read 127 MB once and do 32 M multiply-adds
// instead of 251 M, so the middle launch streams.
//
// Taken wherever the transforms fit in LDS.  On one stream, against the
// convolution blocks: composite model 102 -> 38 us; lengths just past a power
// of two, which double P or Py: 34 x 8 patches over 17 x 17 x 2 cells 37 -> 26,
// 136 x 32 over 17 x 17 x 8 142 -> 76; small grids 24 x 8 over 4 x 4 x 2
// 25 -> 16 us; 1.46 times faster at the least of 17 grids.
//
// Rounding: in norm as the direct sums (2e-16), but a transform's error spreads
// over its outputs.  With slip rates over 16 decades every stress rate is
// within 7e-15 of its own sum |K||s| (direct sums 5e-16); with one patch at
// 1 m/s on a locked fault, where outputs fall off with distance, within 6e-13
// (7e-16).
//
// Spectra are stored column by column (rows fastest): a thread owns a row, a
// wavefront's loads are 1 KB of contiguous memory, the vector's entry is the
// same for all of them, and no sums cross lanes.
#pragma once

namespace oq {

struct GridSpec {
    int nx = 0, nxi = 0, m = 0, nr = 0;           // fault: patches along strike, dip rows, residues, ceil(nx / m)
    int nxc = 0, ny = 0, npl = 0, Q = 0, RF = 0;  // mantle: columns, rows, planes 6 nz, lines npl ny; RF = nxi m
    int P = 0, lgP = 0, H = 0;                    // strike transforms, H = P / 2 + 1 bins
    int Py = 0, lgPy = 0;
    int L = 0, lgL = 0, hb = 0;                   // K_ff transforms, hb = L / 2 + 1 bins
    int Lt = 0;                                   // twiddles: cos, sin of 2 pi k / Lt, k < Lt / 2
    int fq = 0, nfs = 0, gq = 0, ngs = 0;         // columns per chunk and chunks of the F and G products
    const double *tw = nullptr, *K = nullptr;
    const double2 *F = nullptr, *G = nullptr, *M = nullptr;
    // spectra of the source: Sm[f][q], Sf[f][row], S2[fy][f][PI], Sk[f][l];
    // of the result: Of[chunk][f][row], Og[chunk][f][q], Om[PO][fy][f], Ok[j][f]
    double2 *Sm = nullptr, *Sf = nullptr, *S2 = nullptr, *Sk = nullptr;
    double2 *Of = nullptr, *Og = nullptr, *Om = nullptr, *Ok = nullptr;
};

// doubles of LDS: twiddles, then the transforms of a fault row or of a plane
static inline int64_t gsp_lds(const GridSpec &g)
{
    const int64_t a = 2 * (int64_t)g.L + 2 * (int64_t)g.m * (g.P + 1);
    const int64_t b = 2 * (int64_t)g.ny * (g.P + 1) + 2 * (int64_t)g.H * (g.Py + 1);
    return g.Lt + (a > b ? a : b);
}

__device__ __forceinline__ int gsp_bitrev(int x, int bits) { return (int)(__brev((unsigned)x) >> (32 - bits)); }

// x1 <- x0 - w x1, x0 <- x0 + w x1 on registers
__device__ __forceinline__ void bfly(double &r0, double &i0, double &r1, double &i1, double wr, double wi)
{
    const double xr = r1 * wr - i1 * wi, xi = r1 * wi + i1 * wr;
    r1 = r0 - xr;
    i1 = i0 - xi;
    r0 += xr;
    i0 += xi;
}

// In-place radix-2 FFTs of `count` sequences of length L at `pitch`
// (bit-reversed input order), sign -1 (forward) or +1 (inverse), by the nt
// threads of the block.  cs, sn: the twiddles of length L at stride ts.
// Stages len, 2len and 4len run together: a thread that owns the eight
// entries p + k len/2 (k < 8) of a 4len-block holds every pair of the three
// stages, so three stages cost one barrier; one or two stages left over run
// the same way with two or four entries per thread.
__device__ __forceinline__ void lds_fft(double *re, double *im, int L, int count, int pitch, const double *cs,
                                        const double *sn, int ts, double sign, int tid, int nt)
{
    int len = 2;
    for (; 4 * len <= L; len <<= 3) {
        const int half = len >> 1, s1 = L / len * ts, s2 = s1 >> 1, s4 = s1 >> 2, per = L / 8;
        for (int w = tid; w < count * per; w += nt) {
            const int q = w / per, b = w - q * per, p = b & (half - 1), a0 = q * pitch + (b - p) * 8 + p;
            double r[8], i[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                r[k] = re[a0 + k * half];
                i[k] = im[a0 + k * half];
            }
            const double w1r = cs[p * s1], w1i = sign * sn[p * s1];
#pragma unroll
            for (int k = 0; k < 8; k += 2) bfly(r[k], i[k], r[k + 1], i[k + 1], w1r, w1i);  // stage len
#pragma unroll
            for (int k = 0; k < 2; ++k) {  // stage 2len: positions p, p + half
                const int x = (p + k * half) * s2;
                bfly(r[k], i[k], r[k + 2], i[k + 2], cs[x], sign * sn[x]);
                bfly(r[k + 4], i[k + 4], r[k + 6], i[k + 6], cs[x], sign * sn[x]);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {  // stage 4len: positions p + k half
                const int x = (p + k * half) * s4;
                bfly(r[k], i[k], r[k + 4], i[k + 4], cs[x], sign * sn[x]);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                re[a0 + k * half] = r[k];
                im[a0 + k * half] = i[k];
            }
        }
        __syncthreads();
    }
    if (2 * len <= L) {  // two stages left: len and 2len
        const int half = len >> 1, s1 = L / len * ts, s2 = s1 >> 1, per = L / 4;
        for (int w = tid; w < count * per; w += nt) {
            const int q = w / per, b = w - q * per, p = b & (half - 1), a0 = q * pitch + (b - p) * 4 + p, a1 = a0 + half,
                      a2 = a0 + len, a3 = a2 + half;
            double r0 = re[a0], i0 = im[a0], r1 = re[a1], i1 = im[a1];
            double r2 = re[a2], i2 = im[a2], r3 = re[a3], i3 = im[a3];
            const double w1r = cs[p * s1], w1i = sign * sn[p * s1];
            bfly(r0, i0, r1, i1, w1r, w1i);
            bfly(r2, i2, r3, i3, w1r, w1i);
            bfly(r0, i0, r2, i2, cs[p * s2], sign * sn[p * s2]);
            bfly(r1, i1, r3, i3, cs[(p + half) * s2], sign * sn[(p + half) * s2]);
            re[a0] = r0;
            im[a0] = i0;
            re[a1] = r1;
            im[a1] = i1;
            re[a2] = r2;
            im[a2] = i2;
            re[a3] = r3;
            im[a3] = i3;
        }
        __syncthreads();
    } else if (len <= L) {  // one stage left (len == L)
        const int half = len >> 1, step = L / len * ts, per = L / 2;
        for (int w = tid; w < count * per; w += nt) {
            const int q = w / per, b = w - q * per, p = b & (half - 1), a0 = q * pitch + (b - p) * 2 + p, a1 = a0 + half;
            double r0 = re[a0], i0 = im[a0], r1 = re[a1], i1 = im[a1];
            bfly(r0, i0, r1, i1, cs[p * step], sign * sn[p * step]);
            re[a0] = r0;
            im[a0] = i0;
            re[a1] = r1;
            im[a1] = i1;
        }
        __syncthreads();
    }
}

// Forward transforms of fault row b: src(n) = s of patch n of the row.
template <class Src>
__device__ __forceinline__ void gsp_fwd_fault(const GridSpec &g, int b, double *sh, int tid, int nt, Src src)
{
    const int ht = g.Lt / 2, pp = g.P + 1;
    double *cs = sh, *sn = cs + ht, *re = sn + ht, *im = re + g.L, *pr = im + g.L, *pi = pr + g.m * pp;
    for (int x = tid; x < ht; x += nt) {
        cs[x] = g.tw[x];
        sn[x] = g.tw[ht + x];
    }
    for (int n = tid; n < g.L; n += nt) {
        const int r = gsp_bitrev(n, g.lgL);
        re[r] = n < g.nx ? src(n) : 0.0;
        im[r] = 0.0;
    }
    for (int x = tid; x < g.m * g.P; x += nt) {
        const int k = x / g.m, a0 = x - k * g.m, r = a0 * pp + gsp_bitrev(k, g.lgP);  // patch x = a0 + m k
        pr[r] = x < g.nx ? src(x) : 0.0;
        pi[r] = 0.0;
    }
    __syncthreads();
    lds_fft(re, im, g.L, 1, g.L, cs, sn, g.Lt / g.L, -1.0, tid, nt);
    lds_fft(pr, pi, g.P, g.m, pp, cs, sn, g.Lt / g.P, -1.0, tid, nt);
    for (int f = tid; f < g.hb; f += nt) g.Sk[(int64_t)f * g.nxi + b] = double2{re[f], im[f]};
    for (int x = tid; x < g.H * g.m; x += nt) {
        const int f = x / g.m, a0 = x - f * g.m;
        g.Sf[(int64_t)f * g.RF + b * g.m + a0] = double2{pr[a0 * pp + f], pi[a0 * pp + f]};
    }
}

// Forward transforms of mantle plane PI: src(c) = s of cell c = ix + nxc jy.
template <class Src>
__device__ __forceinline__ void gsp_fwd_plane(const GridSpec &g, int PI, double *sh, int tid, int nt, Src src)
{
    const int ht = g.Lt / 2, pp = g.P + 1, pq = g.Py + 1;
    double *cs = sh, *sn = cs + ht, *pr = sn + ht, *pi = pr + g.ny * pp, *qr = pi + g.ny * pp, *qi = qr + g.H * pq;
    for (int x = tid; x < ht; x += nt) {
        cs[x] = g.tw[x];
        sn[x] = g.tw[ht + x];
    }
    for (int x = tid; x < g.ny * g.nxc; x += nt) {
        const int jy = x / g.nxc, ix = x - jy * g.nxc, r = jy * pp + gsp_bitrev(ix, g.lgP);
        pr[r] = src(x);
        pi[r] = 0.0;
    }
    const int nz = g.P - g.nxc;  // padding of a row
    for (int x = tid; x < g.ny * nz; x += nt) {
        const int jy = x / nz, r = jy * pp + gsp_bitrev(g.nxc + x - jy * nz, g.lgP);
        pr[r] = 0.0;
        pi[r] = 0.0;
    }
    __syncthreads();
    lds_fft(pr, pi, g.P, g.ny, pp, cs, sn, g.Lt / g.P, -1.0, tid, nt);
    for (int x = tid; x < g.H * g.Py; x += nt) {
        const int f = x >> g.lgPy, y = x & (g.Py - 1), r = f * pq + gsp_bitrev(y, g.lgPy);
        const bool in = y < g.ny;
        const double vr = in ? pr[y * pp + f] : 0.0, vi = in ? pi[y * pp + f] : 0.0;
        qr[r] = vr;
        qi[r] = vi;
        if (in) g.Sm[(int64_t)f * g.Q + PI * g.ny + y] = double2{vr, vi};
    }
    __syncthreads();
    lds_fft(qr, qi, g.Py, g.H, pq, cs, sn, g.Lt / g.Py, -1.0, tid, nt);
    for (int x = tid; x < g.H * g.Py; x += nt) {
        const int y = x / g.H, f = x - y * g.H;
        g.S2[(int64_t)x * g.npl + PI] = double2{qr[f * pq + y], qi[f * pq + y]};
    }
}

// acc += sum over columns [c0, c1) step cs of A[c * ld] * S[c]: A is the
// thread's row, S the same for every thread.
__device__ __forceinline__ double2 gsp_dot(const double2 *__restrict__ A, int64_t ld, const double2 *__restrict__ S,
                                           int c0, int c1, int cs)
{
    double xr = 0.0, xi = 0.0;
#pragma unroll 8
    for (int c = c0; c < c1; c += cs) {
        const double2 a = A[(int64_t)c * ld], s = S[c];
        xr += a.x * s.x - a.y * s.y;
        xi += a.x * s.y + a.y * s.x;
    }
    return double2{xr, xi};
}

// Blocks of the products, heaviest first.
struct GspBlocks {
    int f, g, m, k;  // block counts per role
};
static inline GspBlocks gsp_blocks(const GridSpec &g, int nt)
{
    return {g.H * ((g.RF + nt - 1) / nt) * g.nfs, g.H * ((g.Q + nt - 1) / nt) * g.ngs, g.Py * g.H, g.hb};
}

// F product: chunk idx % nfs of the columns, row block, bin.
__device__ __forceinline__ void gsp_mul_f(const GridSpec &g, int idx, int tid, int nt)
{
    const int c = idx % g.nfs, r1 = idx / g.nfs, nb = (g.RF + nt - 1) / nt, rb = r1 % nb, f = r1 / nb, row = rb * nt + tid;
    if (row >= g.RF) return;
    const int c0 = c * g.fq, c1 = c0 + g.fq < g.Q ? c0 + g.fq : g.Q;
    g.Of[((int64_t)c * g.H + f) * g.RF + row] =
        gsp_dot(g.F + (int64_t)f * g.Q * g.RF + row, g.RF, g.Sm + (int64_t)f * g.Q, c0, c1, 1);
}

__device__ __forceinline__ void gsp_mul_g(const GridSpec &g, int idx, int tid, int nt)
{
    const int c = idx % g.ngs, r1 = idx / g.ngs, nb = (g.Q + nt - 1) / nt, rb = r1 % nb, f = r1 / nb, row = rb * nt + tid;
    if (row >= g.Q) return;
    const int c0 = c * g.gq, c1 = c0 + g.gq < g.RF ? c0 + g.gq : g.RF;
    g.Og[((int64_t)c * g.H + f) * g.Q + row] =
        gsp_dot(g.G + (int64_t)f * g.Q * g.RF + row, g.Q, g.Sf + (int64_t)f * g.RF, c0, c1, 1);
}

// M product of bin w = fy H + f, in two phases (a barrier between them): the
// threads share the columns in nt / npl groups, then add the groups' sums.
__device__ __forceinline__ int gsp_groups(int rows, int nt) { return rows < nt ? nt / rows : 1; }

__device__ __forceinline__ void gsp_mul_m1(const GridSpec &g, int w, double2 *red, int tid, int nt)
{
    const int ng = gsp_groups(g.npl, nt);
    for (int x = tid; x < ng * g.npl; x += nt) {
        const int s = x / g.npl, PO = x - s * g.npl;
        red[x] = gsp_dot(g.M + (int64_t)w * g.npl * g.npl + PO, g.npl, g.S2 + (int64_t)w * g.npl, s, g.npl, ng);
    }
}

__device__ __forceinline__ void gsp_mul_m2(const GridSpec &g, int w, const double2 *red, int tid, int nt)
{
    const int ng = gsp_groups(g.npl, nt);
    for (int PO = tid; PO < g.npl; PO += nt) {
        double2 v = red[PO];
        for (int s = 1; s < ng; ++s) {
            v.x += red[s * g.npl + PO].x;
            v.y += red[s * g.npl + PO].y;
        }
        g.Om[(int64_t)PO * (g.Py * g.H) + w] = v;
    }
}

// K_ff product of bin f (real spectrum), the same two phases.
__device__ __forceinline__ void gsp_mul_k1(const GridSpec &g, int f, double2 *red, int tid, int nt)
{
    const int ng = gsp_groups(g.nxi, nt);
    const double2 *S = g.Sk + (int64_t)f * g.nxi;
    for (int x = tid; x < ng * g.nxi; x += nt) {
        const int s = x / g.nxi, j = x - s * g.nxi;
        const double *A = g.K + (int64_t)f * g.nxi * g.nxi + j;
        double xr = 0.0, xi = 0.0;
#pragma unroll 4
        for (int l = s; l < g.nxi; l += ng) {
            const double a = A[(int64_t)l * g.nxi];
            xr += a * S[l].x;
            xi += a * S[l].y;
        }
        red[x] = double2{xr, xi};
    }
}

__device__ __forceinline__ void gsp_mul_k2(const GridSpec &g, int f, const double2 *red, int tid, int nt)
{
    const int ng = gsp_groups(g.nxi, nt);
    for (int j = tid; j < g.nxi; j += nt) {
        double2 v = red[j];
        for (int s = 1; s < ng; ++s) {
            v.x += red[s * g.nxi + j].x;
            v.y += red[s * g.nxi + j].y;
        }
        g.Ok[(int64_t)j * g.hb + f] = v;
    }
}

// double2 entries of LDS that the two-phase products need
static inline int64_t gsp_red(const GridSpec &g, int nt)
{
    const int64_t a = g.npl < nt ? nt : g.npl, b = g.nxi < nt ? nt : g.nxi;
    return a > b ? a : b;
}

// bin f of a Hermitian spectrum of length n into bit-reversed order
__device__ __forceinline__ void gsp_put(double *re, double *im, int n, int lg, int f, double vr, double vi)
{
    const int r = gsp_bitrev(f, lg);
    re[r] = vr;
    im[r] = vi;
    if (f > 0 && 2 * f < n) {
        const int c = gsp_bitrev(n - f, lg);
        re[c] = vr;
        im[c] = -vi;
    }
}

// Inverse transforms of fault row b: out(n, tau) for its patches n < nx.
template <class Out>
__device__ __forceinline__ void gsp_inv_fault(const GridSpec &g, int b, double *sh, int tid, int nt, Out out)
{
    const int ht = g.Lt / 2, pp = g.P + 1;
    double *cs = sh, *sn = cs + ht, *re = sn + ht, *im = re + g.L, *pr = im + g.L, *pi = pr + g.m * pp;
    for (int x = tid; x < ht; x += nt) {
        cs[x] = g.tw[x];
        sn[x] = g.tw[ht + x];
    }
    for (int f = tid; f < g.hb; f += nt) {
        const double2 v = g.Ok[(int64_t)b * g.hb + f];
        gsp_put(re, im, g.L, g.lgL, f, v.x, v.y);
    }
    for (int x = tid; x < g.H * g.m; x += nt) {
        const int f = x / g.m, a0 = x - f * g.m;
        const double2 *o = g.Of + (int64_t)f * g.RF + b * g.m + a0;
        double vr = 0.0, vi = 0.0;
#pragma unroll 8
        for (int c = 0; c < g.nfs; ++c) {
            const double2 v = o[(int64_t)c * g.H * g.RF];
            vr += v.x;
            vi += v.y;
        }
        gsp_put(pr + a0 * pp, pi + a0 * pp, g.P, g.lgP, f, vr, vi);
    }
    __syncthreads();
    lds_fft(re, im, g.L, 1, g.L, cs, sn, g.Lt / g.L, 1.0, tid, nt);
    lds_fft(pr, pi, g.P, g.m, pp, cs, sn, g.Lt / g.P, 1.0, tid, nt);
    for (int n = tid; n < g.nx; n += nt) {
        const int k = n / g.m, a0 = n - k * g.m;
        out(n, re[n] / (double)g.L + pr[a0 * pp + k] / (double)g.P);
    }
}

// Inverse transforms of mantle plane PO: out(c, rate) for its cells c = ix + nxc jy.
template <class Out>
__device__ __forceinline__ void gsp_inv_plane(const GridSpec &g, int PO, double *sh, int tid, int nt, Out out)
{
    const int ht = g.Lt / 2, pp = g.P + 1, pq = g.Py + 1;
    double *cs = sh, *sn = cs + ht, *pr = sn + ht, *pi = pr + g.ny * pp, *qr = pi + g.ny * pp, *qi = qr + g.H * pq;
    for (int x = tid; x < ht; x += nt) {
        cs[x] = g.tw[x];
        sn[x] = g.tw[ht + x];
    }
    for (int x = tid; x < g.H * g.Py; x += nt) {
        const int y = x / g.H, f = x - y * g.H, r = f * pq + gsp_bitrev(y, g.lgPy);
        const double2 v = g.Om[(int64_t)PO * (g.Py * g.H) + x];
        qr[r] = v.x;
        qi[r] = v.y;
    }
    __syncthreads();
    lds_fft(qr, qi, g.Py, g.H, pq, cs, sn, g.Lt / g.Py, 1.0, tid, nt);
    for (int x = tid; x < g.H * g.ny; x += nt) {
        const int f = x / g.ny, jy = x - f * g.ny;
        const double2 *o = g.Og + (int64_t)f * g.Q + PO * g.ny + jy;
        double vr = qr[f * pq + jy] / (double)g.Py, vi = qi[f * pq + jy] / (double)g.Py;
#pragma unroll 8
        for (int c = 0; c < g.ngs; ++c) {
            const double2 v = o[(int64_t)c * g.H * g.Q];
            vr += v.x;
            vi += v.y;
        }
        gsp_put(pr + jy * pp, pi + jy * pp, g.P, g.lgP, f, vr, vi);
    }
    __syncthreads();
    lds_fft(pr, pi, g.P, g.ny, pp, cs, sn, g.Lt / g.P, 1.0, tid, nt);
    for (int x = tid; x < g.ny * g.nxc; x += nt) {
        const int jy = x / g.nxc, ix = x - jy * g.nxc;
        out(x, pr[jy * pp + ix] / (double)g.P);
    }
}

// cos and -sin of 2 pi k / n (n divides Lt) from the half table
__device__ __forceinline__ double2 gsp_phase(const GridSpec &g, int n, int64_t k)
{
    int64_t x = k % n;
    if (x < 0) x += n;
    x *= g.Lt / n;
    const int h = g.Lt / 2;
    return x < h ? double2{g.tw[x], -g.tw[h + x]} : double2{-g.tw[x - h], g.tw[h + (x - h)]};
}

// Bin f of residue a0 of K_fm's row of offsets (D entries Fr[a - m jx + m (nxc - 1)]).
__device__ __forceinline__ double2 gsp_tab_f(const GridSpec &g, const double *Fr, int64_t D, int a0, int f)
{
    double xr = 0.0, xi = 0.0;
    for (int t = -(g.nxc - 1); t < g.nr; ++t) {
        const int64_t dd = a0 + (int64_t)g.m * (t + g.nxc - 1);
        if (dd >= D) continue;
        const double2 e = gsp_phase(g, g.P, (int64_t)f * t);
        xr += Fr[dd] * e.x;
        xi += Fr[dd] * e.y;
    }
    return double2{xr, xi};
}

// Bin f of residue a0 of K_mf's row of offsets (Gr[m jx - a + nx - 1]).
__device__ __forceinline__ double2 gsp_tab_g(const GridSpec &g, const double *Gr, int64_t D, int a0, int f)
{
    double xr = 0.0, xi = 0.0;
    for (int t = -(g.nr - 1); t < g.nxc; ++t) {
        const int64_t e = (int64_t)g.m * t - a0 + g.nx - 1;
        if (e < 0 || e >= D) continue;
        const double2 p = gsp_phase(g, g.P, (int64_t)f * t);
        xr += Gr[e] * p.x;
        xi += Gr[e] * p.y;
    }
    return double2{xr, xi};
}

// Bin f along x of one row of a K_mm tile (Tr[m + nxp], |m| < nxc), and bin
// fy over the 2 ny - 1 rows' bins X[yy * H].
__device__ __forceinline__ double2 gsp_tab_mx(const GridSpec &g, const double *Tr, int nxp, int f)
{
    double xr = 0.0, xi = 0.0;
    for (int t = -(g.nxc - 1); t < g.nxc; ++t) {
        const double2 p = gsp_phase(g, g.P, (int64_t)f * t);
        xr += Tr[t + nxp] * p.x;
        xi += Tr[t + nxp] * p.y;
    }
    return double2{xr, xi};
}

__device__ __forceinline__ double2 gsp_tab_my(const GridSpec &g, const double2 *X, int fy)
{
    double xr = 0.0, xi = 0.0;
    for (int t = -(g.ny - 1); t < g.ny; ++t) {
        const double2 p = gsp_phase(g, g.Py, (int64_t)fy * t), v = X[(int64_t)(t + g.ny - 1) * g.H];
        xr += v.x * p.x - v.y * p.y;
        xi += v.x * p.y + v.y * p.x;
    }
    return double2{xr, xi};
}

// Lengths and chunks for a strike grid; nt threads per block of the products.
// False if a transform does not fit the LDS of a workgroup (lds_max bytes).
static inline bool gsp_shape(GridSpec &g, int64_t nx, int64_t nxi, int64_t m, int64_t nxc, int64_t ny, int64_t nz, int nt,
                             int64_t lds_max)
{
    const auto pow2 = [](int64_t n, int &lg) {
        int p = 2;
        for (lg = 1; p < n; p <<= 1) ++lg;
        return p;
    };
    if (nx * nxi > (1 << 24) || 6 * ny * nz * nxc > (1 << 24) || m > nx) return false;
    g.nx = (int)nx;
    g.nxi = (int)nxi;
    g.m = (int)m;
    g.nr = (int)((nx + m - 1) / m);
    g.nxc = (int)nxc;
    g.ny = (int)ny;
    g.npl = (int)(6 * nz);
    g.Q = g.npl * g.ny;
    g.RF = g.nxi * g.m;
    const int64_t need = (g.nr > g.nxc ? g.nr : g.nxc) + g.nxc - 1;
    g.P = pow2(need, g.lgP);
    g.H = g.P / 2 + 1;
    g.Py = pow2(2 * ny - 1, g.lgPy);
    g.L = pow2(2 * nx - 1, g.lgL);
    g.hb = g.L / 2 + 1;
    g.Lt = g.L > g.P ? g.L : g.P;
    if (g.Py > g.Lt) g.Lt = g.Py;
    if (gsp_lds(g) * 8 > lds_max || gsp_red(g, nt) * 16 > 64 * 1024) return false;
    // about 512 blocks per product, at least 16 columns each
    const auto chunks = [nt](int H, int rows, int cols, int &q, int &n) {
        int c = 512 / (H * ((rows + nt - 1) / nt));
        if (c > cols / 16) c = cols / 16;
        if (c < 1) c = 1;
        q = (cols + c - 1) / c;
        n = (cols + q - 1) / q;
    };
    chunks(g.H, g.RF, g.Q, g.fq, g.nfs);
    chunks(g.H, g.Q, g.RF, g.gq, g.ngs);
    return true;
}

}  // namespace oq
