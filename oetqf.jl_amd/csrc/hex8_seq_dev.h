// hex8_seq_dev.h -- the pair kernels' device code behind the operators of
// lockstep batches (ensembles and grouped batches): one thread per
// receiver-cell pair, six Gauss points per axis on boxes bisected to five
// half-diagonals, in a fixed order of operations.
//
// A batch stores its operator in FP32 or split FP16 and steps from rest, where
// the error estimates sit at the operator's rounding: an entry that rounds
// the other way changes a member's step sizes, and with them its state by
// several per cent after 48 steps (measured with the operator from the lane
// groups of hex8_dev.h, whose FP64 entries differ by 1e-13).  A run saved with
// one operator continues with the same steps only on the same bits, so batches
// keep this code (K_fm 46 ms and K_mm 22 ms at the composite model, against
// 25.8 and 16.8 ms); every other operator is assembled by hex8_dev.h.
#pragma once
#include <hip/hip_runtime.h>

#include "hex8_dev.h"

namespace oq {
namespace seq {

__constant__ double kGLX[7][6] = {
    {0}, {0.0}, {-0.5773502691896257645, 0.5773502691896257645},
    {-0.7745966692414833770, 0.0, 0.7745966692414833770},
    {-0.8611363115940525752, -0.3399810435848562648, 0.3399810435848562648, 0.8611363115940525752},
    {-0.9061798459386639928, -0.5384693101056830910, 0.0, 0.5384693101056830910, 0.9061798459386639928},
    {-0.9324695142031520278, -0.6612093864662645137, -0.2386191860831969086, 0.2386191860831969086,
     0.6612093864662645137, 0.9324695142031520278}};
__constant__ double kGLW[7][6] = {
    {0}, {2.0}, {1.0, 1.0},
    {0.5555555555555555556, 0.8888888888888888889, 0.5555555555555555556},
    {0.3478548451374538574, 0.6521451548625461426, 0.6521451548625461426, 0.3478548451374538574},
    {0.2369268850561890875, 0.4786286704993664680, 0.5688888888888888889, 0.4786286704993664680,
     0.2369268850561890875},
    {0.1713244923791703450, 0.3607615730481386076, 0.4679139345726910474, 0.4679139345726910474,
     0.3607615730481386076, 0.1713244923791703450}};

#define OQ_H8_NQ 6
#define OQ_H8_KAPPA 5.0

// Sub-box of the cuboid reached by `path` (depth bits, most significant
// first; 0 = lower half along the current longest axis).
__device__ __forceinline__ void h8_subbox(const double lo0[3], const double hi0[3],
                                          unsigned long long path, int depth,
                                          double lo[3], double hi[3])
{
#pragma unroll
    for (int a = 0; a < 3; ++a) { lo[a] = lo0[a]; hi[a] = hi0[a]; }
    for (int d = depth - 1; d >= 0; --d) {
        int amax = 0;
        double hm = hi[0] - lo[0];
        if (hi[1] - lo[1] > hm) { amax = 1; hm = hi[1] - lo[1]; }
        if (hi[2] - lo[2] > hm) { amax = 2; }
        const double mid = 0.5 * (hi[amax] + lo[amax]);
        if ((path >> d) & 1ull) lo[amax] = mid;
        else hi[amax] = mid;
    }
}

// Accumulates the 36 image stress combinations integrated over [lo0, hi0]
// into acc (depth-first over the bisection tree, lower child first).
__device__ void h8_image_integral(double x, double y, double z, const double lo0[3],
                                  const double hi0[3], double nu, double *acc)
{
    const double xi[3] = {x, y, -z};
    unsigned long long path = 0;
    int depth = 0;
    double Dk[36];
    for (;;) {
        double lo[3], hi[3], h[3], ctr[3], dist2 = 0.0, hd2 = 0.0;
        h8_subbox(lo0, hi0, path, depth, lo, hi);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            h[a] = 0.5 * (hi[a] - lo[a]);
            ctr[a] = 0.5 * (hi[a] + lo[a]);
            const double dd = fabs(xi[a] - ctr[a]) - h[a];
            if (dd > 0.0) dist2 += dd * dd;
            hd2 += h[a] * h[a];
        }
        if (depth < OQ_H8_MAXDEPTH && dist2 < OQ_H8_KAPPA * OQ_H8_KAPPA * hd2) {
            ++depth;
            path <<= 1;
            continue;
        }
        const double vol = h[0] * h[1] * h[2];
        for (int i = 0; i < OQ_H8_NQ; ++i)
            for (int j = 0; j < OQ_H8_NQ; ++j)
                for (int k = 0; k < OQ_H8_NQ; ++k) {
                    const double ys1 = ctr[0] + h[0] * kGLX[OQ_H8_NQ][i];
                    const double ys2 = ctr[1] + h[1] * kGLX[OQ_H8_NQ][j];
                    const double ys3 = ctr[2] + h[2] * kGLX[OQ_H8_NQ][k];
                    const double w = kGLW[OQ_H8_NQ][i] * kGLW[OQ_H8_NQ][j] * kGLW[OQ_H8_NQ][k] * vol;
                    hex8_image_stress_combos(x - ys1, y - ys2, z, ys3, nu, Dk);
#pragma unroll
                    for (int m = 0; m < 36; ++m) acc[m] += w * Dk[m];
                }
        // next leaf in depth-first order
        while (depth > 0 && (path & 1ull)) {
            path >>= 1;
            --depth;
        }
        if (depth == 0) break;
        path += 1;
    }
}

// Eshelby corner sums of the cuboid [lo, hi] at the receiver (x, y, z);
// returns whether the receiver lies inside the cuboid.
__device__ __forceinline__ bool hex8_kelvin(double x, double y, double z, const double lo[3], const double hi[3],
                            Hex8Kelvin &K)
{
    const double rv[3] = {x, y, z};
#pragma unroll
    for (int i = 0; i < 6; ++i) K.phi[i] = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        K.P4[a] = K.P22[a] = K.P211[a] = 0.0;
#pragma unroll
        for (int b = 0; b < 3; ++b) K.P31[a][b] = 0.0;
    }
    for (int s = 0; s < 8; ++s) {
        double X[3], sg = 1.0;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const int bit = (s >> a) & 1;
            X[a] = rv[a] - (bit ? hi[a] : lo[a]);
            if (bit) sg = -sg;
        }
        h8_kelvin_add(K, X, sg);
    }
    return x >= lo[0] && x < hi[0] && y >= lo[1] && y < hi[1] && z >= lo[2] && z < hi[2];
}

template <int FT>
__device__ void h8_image_traction(double x, double y, double z, const double lo0[3], const double hi0[3],
                                  double nu, double ca, double cb, double E[6])
{
    const double xi[3] = {x, y, -z};
    unsigned long long path = 0;
    int depth = 0;
    double Pk[12];
    for (;;) {
        double lo[3], hi[3], h[3], ctr[3], dist2 = 0.0, hd2 = 0.0;
        h8_subbox(lo0, hi0, path, depth, lo, hi);
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            h[a] = 0.5 * (hi[a] - lo[a]);
            ctr[a] = 0.5 * (hi[a] + lo[a]);
            const double dd = fabs(xi[a] - ctr[a]) - h[a];
            if (dd > 0.0) dist2 += dd * dd;
            hd2 += h[a] * h[a];
        }
        if (depth < OQ_H8_MAXDEPTH && dist2 < OQ_H8_KAPPA * OQ_H8_KAPPA * hd2) {
            ++depth;
            path <<= 1;
            continue;
        }
        const double vol = h[0] * h[1] * h[2];
        for (int i = 0; i < OQ_H8_NQ; ++i)
            for (int j = 0; j < OQ_H8_NQ; ++j)
                // one Gauss point per iteration: unrolled, the temporaries spill
#pragma unroll 1
                for (int k = 0; k < OQ_H8_NQ; ++k) {
                    const double ys1 = ctr[0] + h[0] * kGLX[OQ_H8_NQ][i];
                    const double ys2 = ctr[1] + h[1] * kGLX[OQ_H8_NQ][j];
                    const double ys3 = ctr[2] + h[2] * kGLX[OQ_H8_NQ][k];
                    const double w = kGLW[OQ_H8_NQ][i] * kGLW[OQ_H8_NQ][j] * kGLW[OQ_H8_NQ][k] * vol;
                    hex8_image_pairs<FT>(x - ys1, y - ys2, z, ys3, nu, Pk);
#pragma unroll
                    for (int q = 0; q < 6; ++q) E[q] += w * (ca * Pk[q] + cb * Pk[6 + q]);
                }
        while (depth > 0 && (path & 1ull)) {
            path >>= 1;
            --depth;
        }
        if (depth == 0) break;
        path += 1;
    }
}

// Per receiver-cell pair: everything independent of the eigenstrain.
struct Hex8Pair {
    Hex8Kelvin K;
    double D[36];  // image stress combinations, integrated (h8_image_integral)
    bool inside;
};

__device__ void hex8_pair(double x, double y, double z, double qx, double qy, double qz,
                          double T, double L, double W, double nu, Hex8Pair &P)
{
    const double lo[3] = {qx - T / 2.0, qy, qz - W};
    const double hi[3] = {qx + T / 2.0, qy + L, qz};
    // The image integral first: its quadrature loop then runs without the
    // 24 Kelvin sums live, which takes most of its register spills away.
#pragma unroll
    for (int m = 0; m < 36; ++m) P.D[m] = 0.0;
    h8_image_integral(x, y, z, lo, hi, nu, P.D);
    P.inside = hex8_kelvin(x, y, z, lo, hi, P.K);
}

// mv = the eigenstress C : e* of the unit eigenstrain p, as [xx xy xz yy yz zz]
__device__ __forceinline__ void hex8_moment(int p, double mu, double nu, double mv[6])
{
    const double lambda = 2.0 * mu * nu / (1.0 - 2.0 * nu);
#pragma unroll
    for (int q = 0; q < 6; ++q) mv[q] = 0.0;
    if (p == 0 || p == 3 || p == 5) {
        mv[0] = mv[3] = mv[5] = lambda;
        mv[p] += 2.0 * mu;
    } else {
        mv[p] = 2.0 * mu;
    }
}

// Stress s[6] for the unit eigenstrain component p from the Eshelby sums K
// and (IMG) the 54 image integrals D; without them, the full-space part
// plus the eigenstress inside the cuboid.
template <bool IMG>
__device__ __forceinline__ void hex8_stress_unit_body(const Hex8Kelvin &K, const double *D, bool inside, int p,
                                                      double mu, double nu, double s[6])
{
    const int pj[6] = {0, 0, 0, 1, 1, 2}, pk[6] = {0, 1, 2, 1, 2, 2};
    const double lambda = 2.0 * mu * nu / (1.0 - 2.0 * nu);
    const int j0 = pj[p], k0 = pk[p];
    double e[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
    e[j0][k0] = 1.0;
    e[k0][j0] = 1.0;
    const double tr = e[0][0] + e[1][1] + e[2][2];
    double m[3][3], mv[6], gu[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) m[i][j] = 2.0 * mu * e[i][j] + (i == j ? lambda * tr : 0.0);
    mv[0] = m[0][0]; mv[1] = m[0][1]; mv[2] = m[0][2];
    mv[3] = m[1][1]; mv[4] = m[1][2]; mv[5] = m[2][2];
    const double ck = 1.0 / (8.0 * M_PI * (1.0 - nu));
    const double ci = 1.0 / (16.0 * M_PI * mu * (1.0 - nu));
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int l = 0; l < 3; ++l) {
            double acc = 0.0;
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int k = 0; k < 3; ++k)
                    if (e[j][k] != 0.0) acc += e[j][k] * h8_psi(K, i, j, k, l);
#pragma unroll
            for (int k = 0; k < 3; ++k)
                if (e[i][k] != 0.0) acc -= 4.0 * (1.0 - nu) * e[i][k] * h8_phi(K, k, l);
            acc -= 2.0 * nu * tr * h8_phi(K, i, l);
            gu[i][l] = acc * ck;
        }
    // image part: the diagonal and the symmetric sums of its grad u
    double gi[6] = {0, 0, 0, 0, 0, 0};
    if (IMG) {
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            double g = 0.0;
#pragma unroll
            for (int q = 0; q < 6; ++q) g += D[6 * q + c] * mv[q];
            gi[c] = g * ci;
        }
    }
    const double div = gu[0][0] + gu[1][1] + gu[2][2] + (gi[0] + gi[1] + gi[2]);
    const double in = inside ? 1.0 : 0.0;
    s[0] = 2.0 * mu * (gu[0][0] + gi[0]) + lambda * div - in * m[0][0];
    s[1] = mu * (gu[0][1] + gu[1][0] + gi[3]) - in * m[0][1];
    s[2] = mu * (gu[0][2] + gu[2][0] + gi[4]) - in * m[0][2];
    s[3] = 2.0 * mu * (gu[1][1] + gi[1]) + lambda * div - in * m[1][1];
    s[4] = mu * (gu[1][2] + gu[2][1] + gi[5]) - in * m[1][2];
    s[5] = 2.0 * mu * (gu[2][2] + gi[2]) + lambda * div - in * m[2][2];
}

// Stress s[6] for the unit eigenstrain component p (0..5 = xx xy xz yy yz zz).
__device__ void hex8_stress_unit(const Hex8Pair &P, int p, double mu, double nu, double s[6])
{
    hex8_stress_unit_body<true>(P.K, P.D, P.inside, p, mu, nu, s);
}

// The same without the image part (the caller adds it).
__device__ void hex8_stress_unit_kelvin(const Hex8Kelvin &K, bool inside, int p, double mu, double nu, double s[6])
{
    hex8_stress_unit_body<false>(K, nullptr, inside, p, mu, nu, s);
}

}  // namespace seq
}  // namespace oq
