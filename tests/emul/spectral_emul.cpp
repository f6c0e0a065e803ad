// The grid model's frequency-domain operator on the CPU: the block programs
// of oetqf.jl_amd/csrc/grid_spectral.h themselves (one thread per block for
// the transforms, the threads of a product one after another), over
// buffers of their exact sizes filled with NaN, against the direct sums of
// synthetic tables.  Built with the address and undefined-behaviour
// sanitizers, so an index out of range or an unfilled value ends it.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include <vector>

#define __device__
#define __forceinline__ inline
struct double2 { double x, y; };
static inline void __syncthreads() {}
static inline unsigned __brev(unsigned v)
{
    unsigned r = 0;
    for (int i = 0; i < 32; ++i) r |= ((v >> i) & 1u) << (31 - i);
    return r;
}
#include "../../oetqf.jl_amd/csrc/grid_spectral.h"

using namespace oq;
typedef std::vector<double> vd;
static const double NaN = std::numeric_limits<double>::quiet_NaN();

static int check(int nx, int nxi, int m, int nxc, int ny, int nz, int nt)
{
    GridSpec g;
    if (!gsp_shape(g, nx, nxi, m, nxc, ny, nz, nt, 160 * 1024)) {
        printf("%d x %d, m %d, %d x %d x %d: no shape\n", nx, nxi, m, nxc, ny, nz);
        return 1;
    }
    std::mt19937_64 rng(7);
    std::uniform_real_distribution<double> un(-1.0, 1.0);
    const auto rnd = [&](size_t n) { vd v(n); for (auto &x : v) x = un(rng); return v; };
    const int64_t D = nx + (int64_t)m * (nxc - 1);
    const int npl = 6 * nz, Q = npl * ny, Wp = 2 * nxc + 1, Wy = 2 * ny - 1;
    const vd F = rnd((size_t)nxi * Q * D), G = rnd((size_t)Q * nxi * D), st = rnd((size_t)nx * nxi * nxi),
             sf = rnd((size_t)nx * nxi), sm = rnd((size_t)Q * nxc);
    vd T = rnd((size_t)npl * npl * Wy * Wp);
    // twiddles
    vd tw((size_t)g.Lt);
    for (int k = 0; k < g.Lt / 2; ++k) {
        tw[k] = cos(2.0 * M_PI * k / g.Lt);
        tw[g.Lt / 2 + k] = sin(2.0 * M_PI * k / g.Lt);
    }
    g.tw = tw.data();
    const auto c2 = [](size_t n) { return std::vector<double2>(n, double2{NaN, NaN}); };
    auto sF = c2((size_t)g.H * Q * g.RF), sG = c2((size_t)g.H * Q * g.RF), sM = c2((size_t)g.Py * g.H * npl * npl);
    vd sK((size_t)g.hb * nxi * nxi);
    for (int f = 0; f < g.H; ++f)
        for (int q = 0; q < Q; ++q)
            for (int b = 0; b < nxi; ++b)
                for (int a0 = 0; a0 < m; ++a0) {
                    sF[((size_t)f * Q + q) * g.RF + b * m + a0] = gsp_tab_f(g, &F[((size_t)b * Q + q) * D], D, a0, f);
                    sG[((size_t)f * g.RF + b * m + a0) * Q + q] = gsp_tab_g(g, &G[((size_t)q * nxi + b) * D], D, a0, f);
                }
    for (int PO = 0; PO < npl; ++PO)
        for (int PI = 0; PI < npl; ++PI) {
            auto X = c2((size_t)Wy * g.H);
            for (int yy = 0; yy < Wy; ++yy)
                for (int f = 0; f < g.H; ++f)
                    X[(size_t)yy * g.H + f] = gsp_tab_mx(g, &T[(((size_t)PO * npl + PI) * Wy + yy) * Wp], nxc, f);
            for (int fy = 0; fy < g.Py; ++fy)
                for (int f = 0; f < g.H; ++f)
                    sM[((size_t)(fy * g.H + f) * npl + PI) * npl + PO] = gsp_tab_my(g, &X[f], fy);
        }
    for (int f = 0; f < g.hb; ++f)
        for (int l = 0; l < nxi; ++l)
            for (int j = 0; j < nxi; ++j) {
                double a = st[(size_t)nx * (j + nxi * l)];
                for (int k = 1; k < nx; ++k) a += 2.0 * st[k + (size_t)nx * (j + nxi * l)] * cos(2.0 * M_PI * ((int64_t)f * k % g.L) / g.L);
                sK[((size_t)f * nxi + l) * nxi + j] = a;
            }
    g.F = sF.data(); g.G = sG.data(); g.M = sM.data(); g.K = sK.data();
    auto Sm = c2((size_t)g.H * Q), Sf = c2((size_t)g.H * g.RF), S2 = c2((size_t)g.Py * g.H * npl), Sk = c2((size_t)g.hb * nxi);
    auto Of = c2((size_t)g.nfs * g.H * g.RF), Og = c2((size_t)g.ngs * g.H * Q), Om = c2((size_t)npl * g.Py * g.H),
         Ok = c2((size_t)nxi * g.hb);
    g.Sm = Sm.data(); g.Sf = Sf.data(); g.S2 = S2.data(); g.Sk = Sk.data();
    g.Of = Of.data(); g.Og = Og.data(); g.Om = Om.data(); g.Ok = Ok.data();
    vd lds((size_t)gsp_lds(g), NaN);
    for (int b = 0; b < nxi; ++b) {
        vd fresh((size_t)gsp_lds(g), NaN);
        gsp_fwd_fault(g, b, fresh.data(), 0, 1, [&](int n) { return sf[n + (size_t)nx * b]; });
    }
    for (int PI = 0; PI < npl; ++PI) {
        vd fresh((size_t)gsp_lds(g), NaN);
        gsp_fwd_plane(g, PI, fresh.data(), 0, 1, [&](int c) { return sm[c + (size_t)nxc * ny * PI]; });
    }
    const GspBlocks nb = gsp_blocks(g, nt);
    for (int i = 0; i < nb.f; ++i)
        for (int t = 0; t < nt; ++t) gsp_mul_f(g, i, t, nt);
    for (int i = 0; i < nb.g; ++i)
        for (int t = 0; t < nt; ++t) gsp_mul_g(g, i, t, nt);
    for (int i = 0; i < nb.m + nb.k; ++i) {
        auto red = c2((size_t)gsp_red(g, nt));
        for (int ph = 0; ph < 2; ++ph)
            for (int t = 0; t < nt; ++t) {
                if (i < nb.m) ph == 0 ? gsp_mul_m1(g, i, red.data(), t, nt) : gsp_mul_m2(g, i, red.data(), t, nt);
                else ph == 0 ? gsp_mul_k1(g, i - nb.m, red.data(), t, nt) : gsp_mul_k2(g, i - nb.m, red.data(), t, nt);
            }
    }
    vd tau((size_t)nx * nxi, NaN), ds((size_t)Q * nxc, NaN);
    for (int b = 0; b < nxi; ++b) {
        vd fresh((size_t)gsp_lds(g), NaN);
        gsp_inv_fault(g, b, fresh.data(), 0, 1, [&](int n, double v) { tau[n + (size_t)nx * b] = v; });
    }
    for (int PO = 0; PO < npl; ++PO) {
        vd fresh((size_t)gsp_lds(g), NaN);
        gsp_inv_plane(g, PO, fresh.data(), 0, 1, [&](int c, double v) { ds[c + (size_t)nxc * ny * PO] = v; });
    }
    // direct sums
    double e = 0.0, n2 = 0.0;
    for (int b = 0; b < nxi; ++b)
        for (int a = 0; a < nx; ++a) {
            double y = 0.0;
            for (int l = 0; l < nxi; ++l)
                for (int k = 0; k < nx; ++k) y += st[std::abs(a - k) + (size_t)nx * (b + nxi * l)] * sf[k + (size_t)nx * l];
            for (int q = 0; q < Q; ++q)
                for (int jx = 0; jx < nxc; ++jx)
                    y += F[((size_t)b * Q + q) * D + a - m * jx + m * (nxc - 1)] * sm[(size_t)q * nxc + jx];
            const double d = tau[a + (size_t)nx * b] - y;
            e += d * d;
            n2 += y * y;
        }
    const double ef = sqrt(e / n2);
    e = n2 = 0.0;
    for (int PO = 0; PO < npl; ++PO)
        for (int jy = 0; jy < ny; ++jy)
            for (int jx = 0; jx < nxc; ++jx) {
                const int q = PO * ny + jy;
                double y = 0.0;
                for (int b = 0; b < nxi; ++b)
                    for (int a = 0; a < nx; ++a)
                        y += G[((size_t)q * nxi + b) * D + m * jx - a + nx - 1] * sf[a + (size_t)nx * b];
                for (int PI = 0; PI < npl; ++PI)
                    for (int iy = 0; iy < ny; ++iy)
                        for (int ix = 0; ix < nxc; ++ix)
                            y += T[(((size_t)PO * npl + PI) * Wy + jy - iy + ny - 1) * Wp + jx - ix + nxc] *
                                 sm[((size_t)PI * ny + iy) * nxc + ix];
                const double d = ds[(size_t)q * nxc + jx] - y;
                e += d * d;
                n2 += y * y;
            }
    const double em = sqrt(e / n2);
    const bool ok = ef < 1e-13 && em < 1e-13;  // NaN fails
    printf("%d x %d, m %d, %d x %d x %d, %d threads: P %d Py %d L %d chunks %d %d: %.1e %.1e%s\n", nx, nxi, m, nxc, ny, nz, nt,
           g.P, g.Py, g.L, g.nfs, g.ngs, ef, em, ok ? "" : "  FAILED");
    return ok ? 0 : 1;
}

int main()
{
    int bad = 0;
    bad += check(16, 3, 4, 4, 4, 2, 256);
    bad += check(16, 3, 4, 4, 4, 2, 64);
    bad += check(9, 2, 1, 9, 5, 1, 256);
    bad += check(17, 3, 4, 4, 3, 2, 64);   // nx no multiple of m
    bad += check(5, 1, 2, 11, 2, 1, 64);   // mantle beyond the fault: P from the columns
    bad += check(33, 4, 3, 2, 1, 1, 64);
    bad += check(1, 1, 1, 1, 1, 1, 64);
    bad += check(2, 1, 1, 1, 2, 1, 64);
    bad += check(40, 20, 2, 12, 9, 1, 64);
    bad += check(12, 70, 3, 4, 2, 11, 64); // more dip rows and planes than threads
    bad += check(64, 4, 8, 8, 8, 2, 256);
    GridSpec g;  // transforms beyond the LDS are refused
    if (gsp_shape(g, 256, 64, 8, 64, 64, 8, 256, 160 * 1024) || gsp_shape(g, 2000, 4, 100, 20, 4, 2, 256, 64 * 1024)) ++bad;
    if (bad) return 1;
    printf("ok\n");
    return 0;
}
