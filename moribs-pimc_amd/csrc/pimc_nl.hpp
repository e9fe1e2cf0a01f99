// pimc_nl.hpp -- non-linear rotors: Euler frames, the density-matrix look-up of rotden/rotpro,
// the 3D rotor-particle potential of vcord/vcalc and the TIP4P rotor-rotor energy of caleng.
//
// A rotor slice's rotation matrix is computed once when its angles change and cached as a
// Frame; rotden's relative Euler angles are then R1^T R2 of two cached frames, and vcord's body
// axes are the frame's columns.  Density factors and caleng are FP64; vcord/vcalc run in the
// pair precision R (float in production, double in parity runs).
#pragma once
#include "pimc_device.hpp"

namespace pimc {

constexpr double PI_D = 3.14159265358979323846;

// 1/sqrt(x) for x > 0: the hardware's estimate y (2^-23) times the binomial series of 1/sqrt(1 - e),
// e = 1 - x y^2, to second order: 1 + e/2 + 3 e^2/8, within an ulp or so; a square root and a division
// are four times the instructions.
__device__ __forceinline__ double rsqrt_fast(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// fmod(x, y) for y > 0: exact by one subtraction below 2 y, which is where a proposal's angle lies
__device__ __forceinline__ double fmod_near(double x, double y) {
    const double a = fabs(x);
    if (a >= 2.0 * y) return fmod(x, y);
    return a >= y ? copysign(a - y, x) : x;
}

// matpre (rotden.f:136-163) of (phi, theta = acos(cos theta), chi), as MCRot3Dstep passes the
// angles (mc_piqmc.cc:1019-1024).  Host and device build frames with the same expressions.
// cos(acos(cth)) is not cth to the last bit, and it has to stay: a link between near frames divides
// differences of products by the square of its small angle, and then meets the table's cells, whose
// interpolation is not continuous, so that a last bit here decides a move of some runs differently.
__host__ __device__ inline Frame make_frame(double phi, double cth, double chi) {
    double cp, sp, ct, st, ck, sk;
    sincos(phi, &sp, &cp);
    sincos(acos(cth), &st, &ct);
    sincos(chi, &sk, &ck);
    Frame f;
    f.m[0] = cp * ct * ck - sp * sk;   // (1,1)
    f.m[1] = sp * ct * ck + cp * sk;   // (2,1)
    f.m[2] = -st * ck;                 // (3,1)
    f.m[3] = -cp * ct * sk - sp * ck;  // (1,2)
    f.m[4] = -sp * ct * sk + cp * ck;  // (2,2)
    f.m[5] = st * sk;                  // (3,2)
    f.m[6] = cp * st;                  // (1,3)
    f.m[7] = sp * st;                  // (2,3)
    f.m[8] = ct;                       // (3,3)
    double d = 0.0;
    for (int i = 6; i < 9; ++i) d = d + f.m[i] * f.m[i];
    f.zn = sqrt(d);
    return f;
}

__device__ __forceinline__ double fm(const Frame& f, int i, int j) { return f.m[(j - 1) * 3 + (i - 1)]; }

__device__ __forceinline__ double within1(double v) {  // rotden.f:208-216
    if (v > 1.0) v = 1.0;
    if (v < -1.0) v = -1.0;
    return v;
}

// a / b, correctly rounded, from the correctly rounded inverse of b: the product, and its remainder
// (Markstein 1990); three instructions where a second division by the same b takes a dozen
__device__ __forceinline__ double quotient(double a, double b, double inv) {
    const double q = a * inv;
    return fma(fma(-q, b, a), inv, q);
}

// deleul (rotden.f:32-134): Euler angles, in radians, of the rotation whose elements r2(i, j) gives
template <typename M>
__device__ __forceinline__ void deleul(M r2, double& phi2, double& theta2, double& chi2) {
    const double small = 1.0e-08;
    const double cost = within1(r2(3, 3));
    theta2 = acos(cost);
    double cchi;
    bool chi_up, phi_up = true;  // whether the sine is positive
    phi2 = 0.0;
    if (fabs(1.0 - cost) < small) {
        cchi = r2(1, 1);
        chi_up = r2(2, 1) > 0.0;
    } else if (fabs(1.0 + cost) < small) {
        cchi = r2(2, 2);
        chi_up = r2(1, 2) > 0.0;
    } else {
        const double sint = sin(theta2), inv = 1.0 / sint;  // positive in this branch
        phi_up = r2(2, 3) > 0.0;
        phi2 = acos(within1(quotient(r2(1, 3), sint, inv)));
        cchi = quotient(-r2(3, 1), sint, inv);
        chi_up = r2(3, 2) > 0.0;
    }
    chi2 = acos(within1(cchi));
    if (!phi_up) phi2 = 2.0 * PI_D - phi2;
    if (!chi_up) chi2 = 2.0 * PI_D - chi2;
}

// element (i, j) of R(f1)^T R(f2)
__device__ __forceinline__ double rel_element(const Frame& f1, const Frame& f2, int i, int j) {
    double v = 0.0;
#pragma unroll
    for (int k = 1; k <= 3; ++k) v = v + fm(f1, k, i) * fm(f2, k, j);
    return v;
}

__device__ __forceinline__ double degrees(double x) { return quotient(x * 180.0, PI_D, 1.0 / PI_D); }

// rotden (rotden.f:1-31) with rotpro (rotpro_sub.f:1-64): corner value plus one forward
// difference per axis on the 1-degree grid, index (itheta*361 + iphi)*361 + ichi; E and E^2
// converted from cm^-1 to Kelvin.  Returns 1 for an out-of-range angle (the reference's istop).
// rho alone, for the moves: one 32-byte gather instead of three.  rotden_cell asks for a link's cell
// and leaves the rest to rho_value, so that a move can do other work while the gather is under way.
struct RhoCell {
    double4 r;
    double xc, xp, xt;
};

__device__ __forceinline__ double rho_value(const RhoCell& c) { return c.r.x + c.r.y * c.xc + c.r.z * c.xp + c.r.w * c.xt; }

template <typename M>
__device__ __forceinline__ int rotden_cell_of(M r2, const double4* __restrict__ tab, RhoCell& c) {
    double p2, t2, c2;
    deleul(r2, p2, t2, c2);
    const double phi = degrees(p2), theta = degrees(t2), chi = degrees(c2);
    int stop = 0;
    int ichi = (int)chi, iphi = (int)phi, ith = (int)theta;
    if (ichi > 360 || ichi < 0) { ichi = 0; stop = 1; }
    if (iphi > 360 || iphi < 0) { iphi = 0; stop = 1; }
    if (ith > 180 || ith < 0) { ith = 0; stop = 1; }
    c.r = tab[((long long)ith * 361 + iphi) * 361 + ichi];
    c.xc = chi - (double)ichi;
    c.xp = phi - (double)iphi;
    c.xt = theta - (double)ith;
    return stop;
}

// the link of a moved slice's frame f with the slice before it (side 0: f1 = other, f2 = f) or after
// it (side 1: f1 = f, f2 = other); the two rotations are each other's transposes
__device__ __forceinline__ int rotden_cell(const Frame& other, const Frame& f, int side, const double4* __restrict__ tab, RhoCell& c) {
    return rotden_cell_of([&](int i, int j) {
        const double a = rel_element(other, f, i, j), b = i == j ? a : rel_element(other, f, j, i);
        return side ? b : a;
    }, tab, c);
}

__device__ __forceinline__ int rotden_link(const Frame& other, const Frame& f, int side, const double4* __restrict__ tab, double& rho) {
    RhoCell c;
    const int stop = rotden_cell(other, f, side, tab, c);
    rho = rho_value(c);
    return stop;
}

__device__ inline int rotden_rho(const Frame& f1, const Frame& f2, const double4* __restrict__ tab, double& rho) {
    RhoCell c;
    const int stop = rotden_cell_of([&](int i, int j) { return rel_element(f1, f2, i, j); }, tab, c);
    rho = rho_value(c);
    return stop;
}

// rel (if not null) receives the relative Euler angles (phi, theta, chi) in radians
__device__ inline int rotden_frames(const Frame& f1, const Frame& f2, const double4* __restrict__ tab, double& rho,
                                    double& erot, double& esq, double* rel = nullptr) {
    const double wno2k = 0.6950356;
    double p2, t2, c2;
    deleul([&](int i, int j) { return rel_element(f1, f2, i, j); }, p2, t2, c2);
    if (rel) {
        rel[0] = p2;
        rel[1] = t2;
        rel[2] = c2;
    }
    const double phi = degrees(p2), theta = degrees(t2), chi = degrees(c2);
    int stop = 0;
    int ichi = (int)chi, iphi = (int)phi, ith = (int)theta;
    if (ichi > 360 || ichi < 0) { ichi = 0; stop = 1; }
    if (iphi > 360 || iphi < 0) { iphi = 0; stop = 1; }
    if (ith > 180 || ith < 0) { ith = 0; stop = 1; }
    const long long i0 = ((long long)ith * 361 + iphi) * 361 + ichi;
    const double xc = chi - (double)ichi, xp = phi - (double)iphi, xt = theta - (double)ith;
    const double4 r = tab[i0];
    rho = r.x + r.y * xc + r.z * xp + r.w * xt;
    const double4 e = tab[ROT3D_SIZE + i0];
    erot = (e.x + e.y * xc + e.z * xp + e.w * xt) / wno2k;
    const double4 q = tab[2 * ROT3D_SIZE + i0];
    esq = (q.x + q.y * xc + q.z * xp + q.w * xt) / (wno2k * wno2k);
    return stop;
}

template <typename R>
struct Lut3D {
    const vec4_t<R>* v;
    int nr, nth, nch;
    R rmin, rmax, rstep, inv_rstep;
};

__device__ __forceinline__ const float4* v3_ptr(const Tables3& T, float) { return T.v3f; }
__device__ __forceinline__ const double4* v3_ptr(const Tables3& T, double) { return T.v3d; }

template <typename R>
__device__ __forceinline__ Lut3D<R> lut3d(const Tables3& T, int tid) {
    Lut3D<R> L;
    if (tid < 0) {
        L.v = nullptr;
        L.nr = L.nth = L.nch = 2;
        L.rmin = L.rmax = L.rstep = L.inv_rstep = (R)1;
        return L;
    }
    const Tab3D t = T.t3[tid];
    L.v = v3_ptr(T, R()) + t.off;
    L.nr = t.nr;
    L.nth = t.nth;
    L.nch = t.nch;
    L.rmin = (R)t.rmin;
    L.rmax = (R)t.rmax;
    L.rstep = (R)t.rstep;
    L.inv_rstep = (R)(1.0 / t.rstep);
    return L;
}

// vcalc (vcalc.f:1-65): r in bohr clamped to the grid, theta and chi in degrees; corner value
// plus one forward difference per axis
template <typename R>
__device__ __forceinline__ R vcalc(const Lut3D<R>& L, R r, R theta, R chi) {
    if (r < L.rmin) r = L.rmin;
    if (r > L.rmax) r = L.rmax;
    int ir;
    if constexpr (std::is_same<R, float>::value) ir = (int)((r - L.rmin) * L.inv_rstep);
    else ir = (int)((r - L.rmin) / L.rstep);
    int ith = (int)theta, ich = (int)chi;
    if (ich > L.nch - 1) ich = L.nch - 1;
    if (ich < 0) ich = 0;
    if (ith > L.nth - 1) ith = L.nth - 1;
    if (ith < 0) ith = 0;
    if (ir > L.nr - 1) ir = L.nr - 1;  // r == rmax with rounding up
    const vec4_t<R> q = L.v[((long long)ir * L.nth + ith) * L.nch + ich];
    // the differences are zero at an axis' last point, where vcalc drops that term
    return q.x + (q.y / L.rstep) * (r - (L.rmin + (R)ir * L.rstep)) + q.z * (theta - (R)ith) + q.w * (chi - (R)ich);
}

// vcord (vcord.f:1-98): partner at the separation (rx, ry, rz) from the rotor centre with body frame f
template <typename R>
__device__ __forceinline__ R vcord_sep(const Lut3D<R>& L, const Frame& f, R rx, R ry, R rz) {
    const R pi = (R)PI_D;
    const R hx0 = (R)f.m[0], hx1 = (R)f.m[1], hx2 = (R)f.m[2];
    const R hy0 = (R)f.m[3], hy1 = (R)f.m[4], hy2 = (R)f.m[5];
    const R hz0 = (R)f.m[6], hz1 = (R)f.m[7], hz2 = (R)f.m[8];
    R dz = (R)0;
    dz = dz + hz0 * rx;
    dz = dz + hz1 * ry;
    dz = dz + hz2 * rz;
    R rr = (R)0;
    rr = rr + rx * rx;
    rr = rr + ry * ry;
    rr = rr + rz * rz;
    const R rn = sqrt(rr);
    R da = dz / ((R)f.zn * rn);
    if (da > (R)1) da = (R)1;
    if (da < (R)-1) da = (R)-1;
    R the = acos(da);
    R rdx = (R)0, rdy = (R)0;
    rdx = rdx + rx * hx0;
    rdx = rdx + ry * hx1;
    rdx = rdx + rz * hx2;
    rdy = rdy + rx * hy0;
    rdy = rdy + ry * hy1;
    rdy = rdy + rz * hy2;
    R chiw;
    if (fabs(rdx) < (R)1.0e-08) chiw = pi / (R)2;
    else chiw = atan(fabs(rdy / rdx));
    R chir;
    if (rdx >= (R)0 && rdy >= (R)0) chir = chiw;
    else if (rdx < (R)0 && rdy >= (R)0) chir = pi - chiw;
    else if (rdx < (R)0 && rdy < (R)0) chir = pi + chiw;
    else chir = (R)2 * pi - chiw;
    if (L.nch == 181) {
        chiw = chir;
        if (chir > pi) chiw = (R)2 * pi - chir;
    } else if (L.nch == 361) {
        chiw = chir;
    }
    const R rad = rn / (R)0.529177249;
    return vcalc<R>(L, rad, the * (R)180 / pi, chiw * (R)180 / pi);
}

// the same with partner and centre at their positions
template <typename R>
__device__ __forceinline__ R vcord_v(const Lut3D<R>& L, const Frame& f, double cx, double cy, double cz, double px,
                                     double py, double pz) {
    return vcord_sep<R>(L, f, (R)(px - cx), (R)(py - cy), (R)(pz - cz));
}

// vcord's geometry for the density bins (vcord.f:40-75), FP64: radret = |rpt - rcom| in
// Angstrom, theret = angle to the body z axis, chiret = azimuth about it in [0, 2 pi)
__device__ inline void vcord_geometry(const Frame& f, double cx, double cy, double cz, double px, double py, double pz,
                                      double& rad, double& the, double& chi) {
    const double rx = px - cx, ry = py - cy, rz = pz - cz;
    double dz = 0.0;
    dz = dz + f.m[6] * rx;
    dz = dz + f.m[7] * ry;
    dz = dz + f.m[8] * rz;
    double rr = 0.0;
    rr = rr + rx * rx;
    rr = rr + ry * ry;
    rr = rr + rz * rz;
    rad = sqrt(rr);
    the = acos(within1(dz / (f.zn * rad)));
    double rdx = 0.0, rdy = 0.0;
    rdx = rdx + rx * f.m[0];
    rdx = rdx + ry * f.m[1];
    rdx = rdx + rz * f.m[2];
    rdy = rdy + rx * f.m[3];
    rdy = rdy + ry * f.m[4];
    rdy = rdy + rz * f.m[5];
    const double chiw = fabs(rdx) < 1.0e-08 ? PI_D / 2.0 : atan(fabs(rdy / rdx));
    if (rdx >= 0.0 && rdy >= 0.0) chi = chiw;
    else if (rdx < 0.0 && rdy >= 0.0) chi = PI_D - chiw;
    else if (rdx < 0.0 && rdy < 0.0) chi = PI_D + chiw;
    else chi = 2 * PI_D - chiw;
}

// caleng (caleng_tip4p_gg.f:2-186): rigid TIP4P dimer in Kelvin, always FP64 (the Coulomb
// terms of distant pairs cancel to a small fraction of their size).  kcal2k is an INTEGER
// parameter there (implicit typing of names starting with k), so the LJ term is scaled by 503.
__device__ inline double caleng_v(double c1x, double c1y, double c1z, double c2x, double c2y, double c2z,
                                  const Frame& f1, const Frame& f2) {
    const double qm = -1.04, qh = 0.520, br2ang = 0.52917721092, hr2k = 3.1577465e5, kcal2k = 503.0;
    const double zo = 0.06562, zm = -0.08438, xh = 0.7557, zh = -0.5223;  // O and M on the z axis, H at (+-xh, 0, zh)
    double s1[4][3], s2[4][3];  // O, M, H1, H2
    auto sites = [&](double cx, double cy, double cz, const Frame& f, double (&s)[4][3]) {
        const double c[3] = {cx, cy, cz};
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double x = f.m[i], z = f.m[6 + i];
            s[0][i] = fma(z, zo, c[i]);
            s[1][i] = fma(z, zm, c[i]);
            s[2][i] = fma(z, zh, fma(x, xh, c[i]));
            s[3][i] = fma(z, zh, fma(x, -xh, c[i]));
        }
    };
    sites(c1x, c1y, c1z, f1, s1);
    sites(c2x, c2y, c2z, f2, s2);
    auto sq = [&](int a, int b) {
        const double x = s1[a][0] - s2[b][0], y = s1[a][1] - s2[b][1], z = s1[a][2] - s2[b][2];
        return fma(z, z, fma(y, y, x * x));
    };
    const double roo = sq(0, 0);
    const double roo4 = roo * roo, roo6 = 1.0 / (roo4 * roo);
    const double vlj = 6.e5 * (roo6 * roo6) - 610.0 * roo6;
    auto coulomb = [&](auto inverse) {  // of the inverse distance as a function of the squared one
        const double vmh = qm * qh * (inverse(sq(1, 2)) + inverse(sq(1, 3)) + inverse(sq(2, 1)) + inverse(sq(3, 1)));
        const double vhh = qh * qh * (inverse(sq(2, 2)) + inverse(sq(2, 3)) + inverse(sq(3, 2)) + inverse(sq(3, 3)));
        return vmh + vhh + qm * qm * inverse(sq(1, 1));
    };
    double v = coulomb([](double x) { return rsqrt_fast(x); });
    if (!(v == v)) v = coulomb([](double x) { return 1.0 / sqrt(x); });  // sites that coincide, or infinitely far
    return vlj * kcal2k + v * hr2k * br2ang;
}

}  // namespace pimc
