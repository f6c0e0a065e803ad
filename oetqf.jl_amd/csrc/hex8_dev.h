// hex8_dev.h -- device stress of a uniform eigenstrain in a cuboid of an
// elastic half-space (z <= 0, traction-free surface), FP64.
//
// Replaces GeoGreensFunctions.stress_vol_hex8! as called by the reference
// (src/BEM/GF.jl:215-221, 277-283): cuboid [qx-T/2, qx+T/2] x [qy, qy+L] x
// [qz-W, qz] ("T-L-W <=> x-y-z"), rotation 0, tensor strain components
// [xx xy xz yy yz zz], stress in the same order.
//
//   grad u = m : int_V d2G/dx dy,  m = C : e*,  G = G_Kelvin + G_image
//   - Kelvin part in closed form (Eshelby 1957 potentials phi = int 1/r,
//     psi = int r; their 2nd and 4th derivatives over a cuboid are corner
//     sums of log(R+X), atan and rational terms);
//   - image part of Mindlin's (1936) half-space solution (regular inside
//     the medium) by Gauss-Legendre quadrature, with the number of points on
//     each axis taken from the distance of the receiver's image point.
//
// The image kernel D[i][l][p] = d2 G_image_ij / dx_l dy_k summed over the
// moment pair p = (j, k) (without 1/(16 pi mu (1-nu))) enters only through
// the combinations a stress (36) or a fault's shear traction (12) takes,
// generated and simplified by oracle/derive/mindlin_image.py.
//
// GPU shape: everything that does not depend on the eigenstrain (the
// Eshelby tensors and the quadrature sums of the image combinations) is
// accumulated once per receiver-cell pair; the 6 unit eigenstrains the
// builders need are then contractions.  The reference calls the closed form
// once per unit eigenstrain (6x the geometric work).  A pair is the work of a
// group of lanes: they share its Gauss points, take one corner of the Eshelby
// sums each and one unit eigenstrain each.
#pragma once
#include <hip/hip_runtime.h>

#include "rhs_impl.h"

namespace oq {

#define OQ_IPOW(a, n) oq_ipow_dev((a), (n))
__device__ __forceinline__ double oq_ipow_dev(double a, int n)
{
    double r = 1.0;
    const int m = n < 0 ? -n : n;
    for (int i = 0; i < m; ++i) r *= a;
    return n < 0 ? 1.0 / r : r;
}

// The pair sums of the image kernel that the shear traction on a fault of
// type FT takes (P[p], P[6 + p] for eigenstrain pair p; see
// h8_image_traction), simplified as a whole before their common
// subexpressions are taken: about half the operations of the 24 kernel
// entries they are sums of.
template <int FT>
__device__ __forceinline__ void hex8_image_pairs(double X, double Y, double zr, double ys, double nu,
                                                 double *P)
{
    const double R = sqrt(X * X + Y * Y + (zr + ys) * (zr + ys));
    if constexpr (FT == 0) {
#include "hex8_image_trac0.inc"
    } else {
#include "hex8_image_trac1.inc"
    }
}

// log(R + xc) without cancellation for xc < 0 (one log: the lanes of a
// wavefront hold all eight corners, so every branch would run)
__device__ __forceinline__ double h8_logrx(double R, double xc, double rho2)
{
    const double d = R - xc, l = log(xc >= 0.0 ? R + xc : (rho2 > 0.0 ? rho2 / d : d));
    return xc < 0.0 && !(rho2 > 0.0) ? -l : l;
}

__device__ __forceinline__ double h8_atanq(double a, double b, double c, double R)
{
    const double num = a * b;
    if (c == 0.0) return num == 0.0 ? 0.0 : copysign(M_PI / 2.0, num);
    return atan(num / (c * R));
}

__device__ __forceinline__ double h8_ratio(double num, double den)
{
    return den == 0.0 ? 0.0 : num / den;
}

// Eshelby tensors summed over the 8 corners.
//   phi[ab] (a<=b, order 00 01 02 11 12 22)
//   psi by index counts: P4[a] = psi_aaaa, P31[a][b] = psi_aaab (a!=b),
//   P22[c] = psi_aabb with {a,b} = the pair excluding c, P211[a] = psi_aabc.
struct Hex8Kelvin {
    double phi[6];
    double P4[3], P31[3][3], P22[3], P211[3];
};

__device__ __forceinline__ void h8_kelvin_add(Hex8Kelvin &K, const double X[3], double sg)
{
    const double R = sqrt(X[0] * X[0] + X[1] * X[1] + X[2] * X[2]);
    if (R == 0.0) return;
    double A[3], L[3], rho2[3], B[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const int a = (c + 1) % 3, b = (c + 2) % 3;
        rho2[c] = X[a] * X[a] + X[b] * X[b];
        L[c] = h8_logrx(R, X[c], rho2[c]);
        A[c] = h8_atanq(X[a], X[b], X[c], R);
        B[c] = -X[a] * X[b] * h8_ratio(X[c], rho2[c] * R);  // psi_aabb
    }
    K.phi[0] += -sg * A[0];
    K.phi[3] += -sg * A[1];
    K.phi[5] += -sg * A[2];
    K.phi[1] += sg * L[2];
    K.phi[2] += sg * L[1];
    K.phi[4] += sg * L[0];
#pragma unroll
    for (int c = 0; c < 3; ++c) K.P22[c] += sg * B[c];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
        const int q = (p + 1) % 3, r = (p + 2) % 3;
        // psi_pppp = 2 phi_pp - psi_ppqq - psi_pprr
        K.P4[p] += sg * (-2.0 * A[p] - B[r] - B[q]);
        K.P211[p] += sg * (X[p] / R);
    }
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            if (p == q) continue;
            const int r = 3 - p - q;
            K.P31[p][q] += sg * (X[q] * X[q] * h8_ratio(X[r], rho2[r] * R) + L[r] - X[r] / R);
        }
}

__device__ __forceinline__ double h8_psi(const Hex8Kelvin &K, int i, int j, int k, int l)
{
    int cnt[3] = {0, 0, 0};
    cnt[i]++; cnt[j]++; cnt[k]++; cnt[l]++;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        if (cnt[a] == 4) return K.P4[a];
        if (cnt[a] == 3) {
            const int b = cnt[(a + 1) % 3] == 1 ? (a + 1) % 3 : (a + 2) % 3;
            return K.P31[a][b];
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if (cnt[a] == 0) return K.P22[a];
#pragma unroll
    for (int a = 0; a < 3; ++a)
        if (cnt[a] == 2) return K.P211[a];
    return 0.0;
}

__device__ __forceinline__ double h8_phi(const Hex8Kelvin &K, int a, int b)
{
    if (a > b) { const int t = a; a = b; b = t; }
    const int idx = a == 0 ? b : (a == 1 ? 2 + b : 5);
    return K.phi[idx];
}

// Gauss-Legendre rules of the image part: every axis of a box takes its own
// number of points n, 3 <= n <= 12, from how far the image singularity lies.
// With D the distance of the image point from the box centre along the axis
// and e the distance from the box across it, the integrand's nearest poles
// along the axis (half-length h, in units of h) lie at modulus
// r = sqrt(D^2 + e^2) / h or farther, so that n points leave an error of
// about rho^(-2n), rho + 1 / rho = 2 r.  kH8R2[n - 3] is the r^2 at which
// that reaches 3e-16; a box that needs more than 12 points on an axis is
// bisected along its axis of smallest r.
//
// Measured against extended precision over random pairs of five mesh pairs
// (composite, refined, coarse, touching the surface, thin layers): largest
// error of a pair's image sums 3e-12, of the blocks' 2-norms 4e-13; with six
// points on every axis and boxes bisected to five half-diagonals, 1.1e-10 and
// 1e-11.  Points per pair: composite K_fm 135 against 216, coarse 4 x 5 x 2
// cells 570 against 1,680 (the bisection tree of a close pair held up to 200
// boxes of 216 points, one after another).
#define OQ_H8_NMIN 3
#define OQ_H8_NMAX 12
#define OQ_H8_MAXDEPTH 48
#define OQ_H8_NGL 75  // points of the rules n = 3..12; rule n starts at n (n - 1) / 2 - 3

__constant__ double kH8R2[OQ_H8_NMAX - OQ_H8_NMIN + 1] = {37345.5, 1900.09, 318.565, 97.125, 41.7582, 22.295, 13.7696, 9.4242, 6.95304, 5.4276};

// (abscissa, weight)
__constant__ double2 kH8GL[OQ_H8_NGL] = {
    {-0.77459666924148340428, 0.55555555555555558023}, {0.0, 0.88888888888888883955}, {0.77459666924148340428,
    0.55555555555555558023},
    {-0.86113631159405257254, 0.34785484513745384971}, {-0.33998104358485625731, 0.65214515486254609478},
    {0.33998104358485625731, 0.65214515486254609478}, {0.86113631159405257254, 0.34785484513745384971},
    {-0.90617984593866396370, 0.23692688505618908490}, {-0.53846931010568310771, 0.47862867049936647090}, {0.0,
    0.56888888888888888840}, {0.53846931010568310771, 0.47862867049936647090}, {0.90617984593866396370,
    0.23692688505618908490},
    {-0.93246951420315205006, 0.17132449237917035667}, {-0.66120938646626448154, 0.36076157304813860627},
    {-0.23861918608319690471, 0.46791393457269103706}, {0.23861918608319690471, 0.46791393457269103706},
    {0.66120938646626448154, 0.36076157304813860627}, {0.93246951420315205006, 0.17132449237917035667},
    {-0.94910791234275848627, 0.12948496616886970290}, {-0.74153118559939446008, 0.27970539148927664463},
    {-0.40584515137739718416, 0.38183005050511892309}, {0.0, 0.41795918367346940325}, {0.40584515137739718416,
    0.38183005050511892309}, {0.74153118559939446008, 0.27970539148927664463}, {0.94910791234275848627,
    0.12948496616886970290},
    {-0.96028985649753628717, 0.10122853629037625867}, {-0.79666647741362672797, 0.22238103445337448205},
    {-0.52553240991632899082, 0.31370664587788726907}, {-0.18343464249564980784, 0.36268378337836199021},
    {0.18343464249564980784, 0.36268378337836199021}, {0.52553240991632899082, 0.31370664587788726907},
    {0.79666647741362672797, 0.22238103445337448205}, {0.96028985649753628717, 0.10122853629037625867},
    {-0.96816023950762608585, 0.08127438836157441227}, {-0.83603110732663576954, 0.18064816069485739591},
    {-0.61337143270059035771, 0.26061069640293543781}, {-0.32425342340380891581, 0.31234707704000286288}, {0.0,
    0.33023935500125978226}, {0.32425342340380891581, 0.31234707704000286288}, {0.61337143270059035771,
    0.26061069640293543781}, {0.83603110732663576954, 0.18064816069485739591}, {0.96816023950762608585,
    0.08127438836157441227},
    {-0.97390652851717174343, 0.06667134430868813799}, {-0.86506336668898453635, 0.14945134915058058689},
    {-0.67940956829902443559, 0.21908636251598204159}, {-0.43339539412924721340, 0.26926671930999634963},
    {-0.14887433898163121571, 0.29552422471475287002}, {0.14887433898163121571, 0.29552422471475287002},
    {0.43339539412924721340, 0.26926671930999634963}, {0.67940956829902443559, 0.21908636251598204159},
    {0.86506336668898453635, 0.14945134915058058689}, {0.97390652851717174343, 0.06667134430868813799},
    {-0.97822865814605697299, 0.05566856711617366310}, {-0.88706259976809531675, 0.12558036946490461205},
    {-0.73015200557404935644, 0.18629021092773426216}, {-0.51909612920681180714, 0.23319376459199048224},
    {-0.26954315595234495939, 0.26280454451024665152}, {0.0, 0.27292508677790061622}, {0.26954315595234495939,
    0.26280454451024665152}, {0.51909612920681180714, 0.23319376459199048224}, {0.73015200557404935644,
    0.18629021092773426216}, {0.88706259976809531675, 0.12558036946490461205}, {0.97822865814605697299,
    0.05566856711617366310},
    {-0.98156063424671924356, 0.04717533638651182776}, {-0.90411725637047490878, 0.10693932599531842664},
    {-0.76990267419430469253, 0.16007832854334622108}, {-0.58731795428661748293, 0.20316742672306592477},
    {-0.36783149899818018413, 0.23349253653835480571}, {-0.12523340851146891328, 0.24914704581340277323},
    {0.12523340851146891328, 0.24914704581340277323}, {0.36783149899818018413, 0.23349253653835480571},
    {0.58731795428661748293, 0.20316742672306592477}, {0.76990267419430469253, 0.16007832854334622108},
    {0.90411725637047490878, 0.10693932599531842664}, {0.98156063424671924356, 0.04717533638651182776}};

// Orders of the box [lo, hi] for the image point xi; returns the axis to
// bisect, or -1 if the box needs no bisection.
__device__ __forceinline__ int h8_orders(const double xi[3], const double lo[3], const double hi[3], int n[3])
{
    double D2[3], e2[3], h2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const double h = 0.5 * (hi[a] - lo[a]), D = fabs(xi[a] - 0.5 * (hi[a] + lo[a])), e = fmax(D - h, 0.0);
        h2[a] = h * h;
        D2[a] = D * D;
        e2[a] = e * e;
    }
    bool split = false;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        D2[a] += e2[(a + 1) % 3] + e2[(a + 2) % 3];
        n[a] = OQ_H8_NMIN;
#pragma unroll
        for (int q = 0; q < OQ_H8_NMAX - OQ_H8_NMIN; ++q) n[a] += D2[a] < kH8R2[q] * h2[a] ? 1 : 0;
        split = split || D2[a] < kH8R2[OQ_H8_NMAX - OQ_H8_NMIN] * h2[a];
    }
    if (!split) return -1;
    int ax = 0;  // smallest r^2 = D2 / h2
    if (D2[1] * h2[0] < D2[0] * h2[1]) ax = 1;
    if (D2[2] * h2[ax] < D2[ax] * h2[2]) ax = 2;
    return ax;
}

// Sum over the G lanes (8 or 64) of a pair's group, the same value in each.
template <int G>
__device__ __forceinline__ double h8_group_sum(double x)
{
    static_assert(G == 8 || G == 64, "a group is 8 lanes or a wavefront");
    if constexpr (G == 64) return wave_sum(x);
    x += dpp_f64<0xB1>(x);    // quad_perm [1,0,3,2]
    x += dpp_f64<0x4E>(x);    // quad_perm [2,3,0,1]
    return x + dpp_f64<0x141>(x);  // row_half_mirror
}

// Gauss points of the cuboid [lo0, hi0] for the receiver (x, y, z), dealt
// out to the G lanes of the pair's group: body(X, Y, ys, w) for lane g's
// points, X and Y the horizontal separations, ys the point's z, w its weight.
// Boxes of the bisection tree depth-first, lower child first; `path` holds
// the branches from the root.  gl: the rules in LDS.
template <int G, class F>
__device__ __forceinline__ void h8_points(double x, double y, double z, const double lo0[3], const double hi0[3],
                                          int g, const double2 *gl, F body)
{
    const double xi[3] = {x, y, -z};
    unsigned long long path = 0;
    int depth = 0;
    for (;;) {
        double lo[3], hi[3];
        int n[3], ax;
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = lo0[a];
            hi[a] = hi0[a];
        }
        ax = h8_orders(xi, lo, hi, n);
        for (int d = depth - 1; d >= 0; --d) {  // down the path (every inner box has an axis to bisect)
            const bool up = (path >> d) & 1ull;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const double mid = 0.5 * (hi[a] + lo[a]);
                if (a == ax && up) lo[a] = mid;
                if (a == ax && !up) hi[a] = mid;
            }
            ax = h8_orders(xi, lo, hi, n);
        }
        if (depth < OQ_H8_MAXDEPTH && ax >= 0) {
            ++depth;
            path <<= 1;
            continue;
        }
        double h[3], ctr[3];
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            h[a] = 0.5 * (hi[a] - lo[a]);
            ctr[a] = 0.5 * (hi[a] + lo[a]);
        }
        const double vol = h[0] * h[1] * h[2];
        const double2 *g0 = gl + (n[0] * (n[0] - 1) / 2 - 3), *g1 = gl + (n[1] * (n[1] - 1) / 2 - 3),
                      *g2 = gl + (n[2] * (n[2] - 1) / 2 - 3);
        const int n12 = n[1] * n[2], tot = n[0] * n12;
        const float r12 = 1.0f / (float)n12, r2 = 1.0f / (float)n[2];
        // one point per iteration: unrolled, the bodies' temporaries spill
#pragma unroll 1
        for (int t = g; t < tot; t += G) {
            // t < 1728: the rounded quotients of t + 1/2 are exact
            const int i = (int)(((float)t + 0.5f) * r12), u = t - i * n12;
            const int j = (int)(((float)u + 0.5f) * r2), k = u - j * n[2];
            const double2 p = g0[i], q = g1[j], s = g2[k];
            body(x - (ctr[0] + h[0] * p.x), y - (ctr[1] + h[1] * q.x), ctr[2] + h[2] * s.x, p.y * q.y * s.y * vol);
        }
        while (depth > 0 && (path & 1ull)) {
            path >>= 1;
            --depth;
        }
        if (depth == 0) break;
        path += 1;
    }
}

// The rules into LDS (all threads of the block; one barrier).
__device__ __forceinline__ void h8_load_rules(double2 *gl)
{
    for (int i = threadIdx.x; i < OQ_H8_NGL; i += blockDim.x) gl[i] = kH8GL[i];
    __syncthreads();
}

// The combinations of the image kernel that a stress takes: P[6 q + c] for
// moment pair q, c = D[0][0], D[1][1], D[2][2], D[0][1] + D[1][0],
// D[0][2] + D[2][0], D[1][2] + D[2][1] (the image part of grad u enters the
// stress only through its diagonal and symmetric sums), simplified as a
// whole before their common subexpressions are taken: about 60 % of the
// operations of the 54 kernel entries.
__device__ __forceinline__ void hex8_image_stress_combos(double X, double Y, double zr, double ys, double nu,
                                                         double *P)
{
    const double R = sqrt(X * X + Y * Y + (zr + ys) * (zr + ys));
#include "hex8_image_stress.inc"
}

// Adds wgt times corner s (0..7) of the Eshelby corner sums of the cuboid
// [lo, hi] at the receiver (x, y, z) to K.
__device__ __forceinline__ void hex8_kelvin_corner(double x, double y, double z, const double lo[3],
                                                   const double hi[3], int s, double wgt, Hex8Kelvin &K)
{
    const double X[3] = {x - ((s & 1) ? hi[0] : lo[0]), y - ((s & 2) ? hi[1] : lo[1]), z - ((s & 4) ? hi[2] : lo[2])};
    h8_kelvin_add(K, X, (__popc(s) & 1) ? -wgt : wgt);
}

__device__ __forceinline__ void hex8_kelvin_zero(Hex8Kelvin &K)
{
#pragma unroll
    for (int i = 0; i < 6; ++i) K.phi[i] = 0.0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        K.P4[a] = K.P22[a] = K.P211[a] = 0.0;
#pragma unroll
        for (int b = 0; b < 3; ++b) K.P31[a][b] = 0.0;
    }
}

template <int G>
__device__ __forceinline__ void hex8_kelvin_reduce(Hex8Kelvin &K)
{
#pragma unroll
    for (int i = 0; i < 6; ++i) K.phi[i] = h8_group_sum<G>(K.phi[i]);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        K.P4[a] = h8_group_sum<G>(K.P4[a]);
        K.P22[a] = h8_group_sum<G>(K.P22[a]);
        K.P211[a] = h8_group_sum<G>(K.P211[a]);
#pragma unroll
        for (int b = 0; b < 3; ++b)
            if (a != b) K.P31[a][b] = h8_group_sum<G>(K.P31[a][b]);
    }
}

__device__ __forceinline__ bool hex8_inside(double x, double y, double z, const double lo[3], const double hi[3])
{
    return x >= lo[0] && x < hi[0] && y >= lo[1] && y < hi[1] && z >= lo[2] && z < hi[2];
}

// The image integral contracted with the shear-traction functional of a
// fault receiver, for the 6 unit eigenstrains at once.  The traction is
// linear in grad u, tau = sum_il c_il (grad u)_il, and only four c_il are
// nonzero (FT 0, strike slip: tau = -s_xy sin d + s_xz cos d gives c_01 =
// c_10 = -mu sin d, c_02 = c_20 = mu cos d; FT 1, dip slip: tau = (s_zz -
// s_yy)/2 sin 2d + s_yz cos 2d gives c_22 = -c_11 = mu sin 2d, c_12 = c_21 =
// mu cos 2d).  So the quadrature accumulates E[q] = sum_il c_il D[i][l][q]
// (6 sums, from 24 of the 54 kernel terms; the other 30 and their common
// subexpressions are dead code) instead of all 54 integrals: ca, cb are the
// two coefficients above.  E: lane g's share.
template <int FT, int G>
__device__ __forceinline__ void h8_image_traction(double x, double y, double z, const double lo0[3],
                                                  const double hi0[3], double nu, double ca, double cb, int g,
                                                  const double2 *gl, double E[6])
{
    h8_points<G>(x, y, z, lo0, hi0, g, gl, [&](double X, double Y, double ys, double w) {
        double Pk[12];
        hex8_image_pairs<FT>(X, Y, z, ys, nu, Pk);
#pragma unroll
        for (int q = 0; q < 6; ++q) E[q] += w * (ca * Pk[q] + cb * Pk[6 + q]);
    });
}

// Adds wgt times lane g's share of the 36 image stress combinations
// integrated over [lo0, hi0] to acc.
template <int G>
__device__ __forceinline__ void h8_image_integral(double x, double y, double z, const double lo0[3],
                                                  const double hi0[3], double nu, double wgt, int g,
                                                  const double2 *gl, double acc[36])
{
    h8_points<G>(x, y, z, lo0, hi0, g, gl, [&](double X, double Y, double ys, double w) {
        double Dk[36];
        hex8_image_stress_combos(X, Y, z, ys, nu, Dk);
        w *= wgt;
#pragma unroll
        for (int m = 0; m < 36; ++m) acc[m] += w * Dk[m];
    });
}

// mv = the eigenstress C : e* of the unit eigenstrain p, as [xx xy xz yy yz zz]
__device__ __forceinline__ void hex8_moment(int p, double mu, double nu, double mv[6])
{
    const double lambda = 2.0 * mu * nu / (1.0 - 2.0 * nu);
    const bool diag = p == 0 || p == 3 || p == 5;
#pragma unroll
    for (int q = 0; q < 6; ++q) {
        const bool qd = q == 0 || q == 3 || q == 5;
        mv[q] = (diag && qd ? lambda : 0.0) + (p == q ? 2.0 * mu : 0.0);
    }
}

// Stress s[6] for the unit eigenstrain component p (0..5 = xx xy xz yy yz
// zz; any lane its own) from the Eshelby sums K and (IMG) the 36 image
// integrals D; without them, the full-space part plus the eigenstress inside
// the cuboid (in: 1 inside, 0 outside; a quadrature over the receiver passes
// its weighted sums of K, D and in).
template <bool IMG>
__device__ __forceinline__ void hex8_stress_unit(const Hex8Kelvin &K, const double *D, double in, int p, double mu,
                                                 double nu, double s[6])
{
    const double lambda = 2.0 * mu * nu / (1.0 - 2.0 * nu);
    // the unit eigenstrain: e[j][k] = e[k][j] = 1 for p's (j, k)
    const double e6[6] = {p == 0 ? 1.0 : 0.0, p == 1 ? 1.0 : 0.0, p == 2 ? 1.0 : 0.0,
                          p == 3 ? 1.0 : 0.0, p == 4 ? 1.0 : 0.0, p == 5 ? 1.0 : 0.0};
    const double e[3][3] = {{e6[0], e6[1], e6[2]}, {e6[1], e6[3], e6[4]}, {e6[2], e6[4], e6[5]}};
    const double tr = e6[0] + e6[3] + e6[5];
    double mv[6], gu[3][3];
    hex8_moment(p, mu, nu, mv);
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
                for (int k = 0; k < 3; ++k) acc += e[j][k] * h8_psi(K, i, j, k, l);
#pragma unroll
            for (int k = 0; k < 3; ++k) acc -= 4.0 * (1.0 - nu) * e[i][k] * h8_phi(K, k, l);
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
    s[0] = 2.0 * mu * (gu[0][0] + gi[0]) + lambda * div - in * mv[0];
    s[1] = mu * (gu[0][1] + gu[1][0] + gi[3]) - in * mv[1];
    s[2] = mu * (gu[0][2] + gu[2][0] + gi[4]) - in * mv[2];
    s[3] = 2.0 * mu * (gu[1][1] + gi[1]) + lambda * div - in * mv[3];
    s[4] = mu * (gu[1][2] + gu[2][1] + gi[5]) - in * mv[4];
    s[5] = 2.0 * mu * (gu[2][2] + gi[2]) + lambda * div - in * mv[5];
}

}  // namespace oq
