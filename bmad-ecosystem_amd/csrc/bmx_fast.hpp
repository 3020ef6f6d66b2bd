// Straight-line element operations for the common particle, and the runs that speculate on it.
//
// The maps of bmx_maps.hpp decide every rare case (a series domain left, a loss, an orbit too
// large) where it can arise, which costs each element several branches, mask changes and waits.
// The operations here are the same maps for the common case alone: branch-free code that only
// notes, per lane, whether a conservative test failed. What an element does to a particle is then
// defined once for all kernels: its operations if every test holds (and the momenta it leaves
// with are far from orbit_too_large's limit), else the general map, which decides what happens.
// A kernel may track many elements on their operations and look at the tests once at the end
// (a run): a lane that failed none has the result, and one that failed any goes back to where it
// entered the run and through the elements one by one. A particle on operations gets the same bits
// from every kernel, and its result never depends on the others in its wave. (The general maps are
// contracted by the compiler for each kernel they are built into: rf cavities, stepped elements
// and lanes that the operations refuse can differ between kernels in the last bits.)
//
// The operations are what an element's map is made of (bmx_table.hpp FastOp): one 64-byte record
// each, read by one scalar load. Sums and products are written as they are to be rounded
// (contraction is off and every fused multiply-add explicit), so that an operation gives the same
// bits wherever it is inlined.
//
// What bounds the kernels made of them: large beams, the issue of vector instructions (47 for 64
// passes of a particle through an element on the 901-element ring against 68 for the general maps,
// and 7.7 scalar ones against 26; counters over 1000 turns of 1e6 particles); few particles, the
// chain of dependent operations and the reads of their values, one line of 64 bytes ahead.
// 901-element ring, 10 turns, general maps -> operations: 1e6 particles 18.3 -> 11.3 ms, 1000
// particles 3.69 -> 1.32 ms with cell kernels; 150001 particles 8.9 -> 4.6 ms without. A run that
// refuses lanes costs its wave the run and the way element by element: beams with many particles
// beyond the tests' bounds that live on take up to 1.7 times as long as on the general maps alone.
#pragma once
#include <hip/hip_runtime.h>

#include "bmx_maps.hpp"

namespace bmx {

// The coordinates an operation changes.
struct FastP {
    double x, px, y, py, z;
};
__device__ __forceinline__ FastP fast_get(const Particle &p) { return {p.x, p.px, p.y, p.py, p.z}; }
__device__ __forceinline__ void fast_put(Particle &p, const FastP &f)
{
    p.x = f.x;
    p.px = f.px;
    p.y = f.y;
    p.py = f.py;
    p.z = f.z;
}

// The energy and its functions as the operations use them: Particle's own (a radiation kick
// inside a run changes them here first) and
//   ir2 = 1/(1+pz)^2,
//   bq = (beta - beta0)/beta0, the clock's path against the reference's, per length.
struct FastE {
    double pz, rel_p, inv_rp, ez, lez, ir2, bq;
};
__device__ __forceinline__ FastE fast_energy(const Particle &p, const Species &sp)
{
#pragma clang fp contract(off)
    return {p.pz, p.rel_p, p.inv_rp, p.ez, p.lez, p.inv_rp * p.inv_rp, (p.beta - sp.beta0) * sp.inv_beta0};
}
__device__ __forceinline__ void fast_put_energy(Particle &p, const FastE &en)
{
    p.pz = en.pz;
    p.rel_p = en.rel_p;
    p.inv_rp = en.inv_rp;
    p.ez = en.ez;
    p.lez = en.lez;
}

// One operation record, read with one 64-byte scalar load.
typedef double OpVec __attribute__((ext_vector_type(8)));
__device__ __forceinline__ OpVec load_op(CP r) { return *(const OpVec BMX_CONST *)r; }

// Bound of u = (px^2 + py^2)/(1+pz)^2 (angles below 44 mrad) in drifts and at both faces of bends:
// beyond the general maps' own series (31 mrad), so that a beam of large angles is not sent through a
// run and then element by element for lanes that those take by series. At 15.6 mrad, two terms fewer in
// the bend, 700 elements at angles of 8 mrad rms took 2.0 to 3.2 times as long as the general maps.
constexpr double kFastU2 = 0x1p-9;
// Bound of t = (k1 L^2/(1+pz))^2 of the short quadrupole series.
constexpr double kFastT = 0x1p-8;

// The exit aperture: x^2 + k2 y^2 < r2 (a centred ellipse, or no aperture), or |x| < k2 and
// |y| < r2 (a rectangle about the axis). NaN coordinates fail.
template <bool RECT>
__device__ __forceinline__ void fast_aperture(const FastP &f, double k2, double r2, LaneMask &bad)
{
#pragma clang fp contract(off)
    if constexpr (RECT) {
        bad |= lanes(!(fabs(f.x) < k2)) | lanes(!(fabs(f.y) < r2));
    } else {
        const double r = fma(f.y * f.y, k2, f.x * f.x);
        bad |= lanes(!(r < r2));
    }
}

// px^2 + py^2 <= (1+pz)^2 with room to spare, where no operation on the way tests it.
__device__ __forceinline__ void fast_unstable(const FastP &f, const FastE &en, LaneMask &bad)
{
    const double h = 0.5 * en.rel_p;
    bad |= lanes(!(fabs(f.px) < h)) | lanes(!(fabs(f.py) < h));
}

// track_a_drift.f90:25-116 by the series of 1/ps - 1 (drift_series with the terms that
// kFastU2 leaves: the first omitted one, 231/1024 u^6 of q, is below 1.3e-17, 2e-19 at 31 mrad).
__device__ __forceinline__ void fast_drift(FastP &f, const FastE &en, double L,
                                           LaneMask &bad)
{
#pragma clang fp contract(off)
    const double u = fma(f.py, f.py, f.px * f.px) * en.ir2;
    bad |= lanes(!(u < kFastU2));
    double h = fma(u, 0.24609375, 0.2734375);  // 63/256, 35/128
    h = fma(h, u, 0.3125);                      // 5/16
    h = fma(h, u, 0.375);                       // 3/8
    h = fma(h, u, 0.5);
    const double q = h * u;
    const double Li = L * en.inv_rp;
    const double w = fma(Li, q, Li);
    f.x = fma(f.px, w, f.x);
    f.y = fma(f.py, w, f.y);
    f.z = fma(L, en.ez - q, f.z);
}

// track_a_quadrupole.f90:17-148 (no multipoles, no fringe); b1 = k1 L, b1l = k1 L^2. The plane
// functions are those of quadrupole() (LONG: quad_series<5>, t <= kQuadTLim; else the terms that
// t <= kFastT leaves, the first omitted one, t^3/13! of sx, below 1e-17). The path length needs
// no matrix elements: with x'' = k x, d(x u)/ds = u^2 + k x^2 and u^2 - k x^2 is constant along
// the quadrupole, so
//   -1/2 int u^2 ds = -1/4 [ x1 u1 - x0 u0 + L (u0^2 - k x0^2) ],   u = px/(1+pz),
// which equals quad_mat2_calc.f90:56-61's z1 x^2 + z2 x px + z3 px^2 identically.
template <bool LONG>
__device__ __forceinline__ void fast_quad(FastP &f, const FastE &en, double L, double b1l, double b1,
                                          LaneMask &bad)
{
#pragma clang fp contract(off)
    const double W = b1l * en.inv_rp;
    const double t = W * W;
    double cx, cy, sx, sy;  // x focuses for b1 > 0: cos, sin(..)/(..) of the x plane, then y's
    if constexpr (LONG) {
        bad |= lanes(!(t <= kQuadTLim));
        const QuadFns s = quad_series<5>(W, t);
        cx = s.cxx;
        cy = s.cxy;
        sx = s.sxx;
        sy = s.sxy;
    } else {
        bad |= lanes(!(t <= kFastT));
        const double t2 = t * t;
        double a = fma(t, 0.041666666666666664, 1.0);    // 1/4!
        a = fma(2.48015873015873e-05, t2, a);             // 1/8!
        a = fma(2.08767569878681e-09, t2 * t, a);         // 1/12!
        double a1 = fma(t, 0.008333333333333333, 1.0);   // 1/5!
        a1 = fma(2.7557319223985893e-06, t2, a1);         // 1/9!
        double b = fma(t, 0.001388888888888889, 0.5);    // 1/6!, 1/2!
        b = fma(2.755731922398589e-07, t2, b);            // 1/10!
        double b3 = fma(t, 0.0011904761904761906, 1.0);  // 6/7!
        b3 = fma(1.5031265031265032e-07, t2, b3);         // 6/11!
        b3 = b3 * 0.16666666666666666;                    // 1/3!
        cx = fma(-W, b, a);
        cy = fma(W, b, a);
        sx = fma(-W, b3, a1);
        sy = fma(W, b3, a1);
    }
    const double Li = L * en.inv_rp;
    const double x = f.x, px = f.px, y = f.y, py = f.py;
    const double xp = fma(y, py, x * px);
    const double p2 = fma(py, py, px * px);
    double d = fma(b1, fma(-y, y, x * x), fma(Li, p2, -xp));
    f.x = fma(Li * sx, px, cx * x);
    f.px = fma(-(b1 * sx), x, cx * px);
    f.y = fma(Li * sy, py, cy * y);
    f.py = fma(b1 * sy, y, cy * py);
    d = fma(f.x, f.px, d);
    d = fma(f.y, f.py, d);
    f.z = fma(L, en.lez, fma(-0.25 * en.inv_rp, d, f.z));
}

// track_a_thick_multipole.f90:18-133 for one step of a normal sextupole: half kick, drift, half
// kick (two half kicks at one place make the full kick between two steps). b: the half-step
// strength, b2 = 2 b.
__device__ __forceinline__ void fast_sextupole(FastP &f, const FastE &en, double step, double b,
                                               double b2, LaneMask &bad)
{
#pragma clang fp contract(off)
    f.px = fma(-b, fma(-f.y, f.y, f.x * f.x), f.px);
    f.py = fma(b2, f.x * f.y, f.py);
    fast_drift(f, en, step, bad);
    f.px = fma(-b, fma(-f.y, f.y, f.x * f.x), f.px);
    f.py = fma(b2, f.x * f.y, f.py);
}

// track_a_bend.f90:18-333 for a sector bend with the simple Hwang edges and g_tot = g: the
// momentum form of sbend_momentum_form. With c = pz_s/(1+pz) = sqrt(1 - u) at each face, u =
// (px^2 + py^2)/(1+pz)^2, the orbit turns by theta + (phi_t - phi_f) with
//   sin(phi_t - phi_f) = (px_t c_f - px_f c_t)/((1+pz) (1 - w)),   w = (py/(1+pz))^2
// (ux^2 + c^2 = 1 - w at both faces), whose reciprocal is a short series and whose arcsine,
// below 0.089, another (to 3e-17, and 2e-17 of the angle where w is large): no division. The path length is h (theta + phi_t - phi_f)
// with h = (1+pz)/g, and against the clock's beta L/beta0 it leaves z only L (bq - pz) - h (phi_t
// - phi_f), without the difference of two terms of the size of L.
// near: some lane has |pz| < 1e-9; those that are all within 1e-9 of the zero orbit take the
// semi-linear body (:136-159).
template <class V>
__device__ __forceinline__ void fast_bend(FastP &f, const FastE &en, const V &r,
                                          const Species &sp, bool near, LaneMask &bad)
{
#pragma clang fp contract(off)
    const double g = r[0], ca = r[1], sa = r[2], omc = r[3], inv_g = r[4], L = r[5];
    const double gi = g * en.inv_rp, a = 0.5 * gi, ai = a * en.inv_rp;
    {
        const double pxy = f.px * f.y;
        f.x = fma(a, f.y * f.y, f.x);
        f.py = fma(-gi, pxy, f.py);
        f.z = fma(-ai, pxy * f.y, f.z);
    }
    const FastP in = f;
    const double x = f.x, px = f.px, py = f.py;
    const double py2 = py * py;
    const double w = py2 * en.ir2;
    const double su = fma(px, px, py2) * en.ir2;
    bad |= lanes(!(su < kFastU2));
    // sqrt(1 - u) - 1 = -u/2 - u^2/8 - u^3/16 - 5 u^4/128 - 7 u^5/256 - ...
    double m = fma(su, -0.02734375, -0.0390625);
    m = fma(m, su, -0.0625);
    m = fma(m, su, -0.125);
    m = fma(m, su, -0.5);
    m = m * su;
    const double v = fma(en.rel_p, m, en.pz);  // pz_s - 1
    const double pf = fma(fma(-g, x, v), sa, px * ca);
    const double sf = fma(pf, pf, py2) * en.ir2;
    bad |= lanes(!(sf < kFastU2));
    double n = fma(sf, -0.02734375, -0.0390625);
    n = fma(n, sf, -0.0625);
    n = fma(n, sf, -0.125);
    n = fma(n, sf, -0.5);
    n = n * sf;
    const double br = fma(px, sa, fma(v, omc, en.rel_p * (n - m)));
    f.x = fma(br, inv_g, x * ca);
    // 1/(1 - w): the first omitted term, w^6, is below 6e-17, and only where s is near zero
    double iv = 1.0 + w;
    iv = fma(w, iv, 1.0);
    iv = fma(w, iv, 1.0);
    iv = fma(w, iv, 1.0);
    iv = fma(w, iv, 1.0);
    const double s = fma(px, 1.0 + n, -(pf * (1.0 + m))) * (iv * en.inv_rp);
    const double s2 = s * s;
    double q = fma(s2, 0.017352764423076924, 0.022372159090909092);   // 231/13312, 63/2816
    q = fma(q, s2, 0.030381944444444444);                              // 35/1152
    q = fma(q, s2, 0.044642857142857144);                              // 5/112
    q = fma(q, s2, 0.075);                                              // 3/40
    q = fma(q, s2, 0.16666666666666666);                               // 1/6
    const double dphi = fma(q * s2, s, s);
    const double hd = inv_g * dphi;
    f.px = pf;
    f.y = fma(py, hd + L, f.y);
    f.z = fma(-en.rel_p, hd, fma(L, en.bq - en.pz, f.z));
    if (near) {
        const bool semi = (fabs(x * g) < 1e-9) & (fabs(px) < 1e-9) & (fabs(py) < 1e-9) &
                          (fabs(en.pz) < 1e-9);
        if (any_lane(semi)) {
            if (semi) {
                const double gam2 = sp.mc2_sq / (sqr(en.rel_p * sp.p0c) + sp.mc2_sq);
                const double ls = sa * inv_g, lc = omc * inv_g;  // L sinc, g L^2 cosc
                // L angle^2 sincc(angle), the path's change with the dispersion (|angle| <= 0.1)
                const double an2 = sqr(g * L);
                const double sincc = 1.0 / 6 + an2 * (-1.0 / 120 + an2 * (1.0 / 5040 - an2 / 362880));
                const double m56 = L * (gam2 - an2 * sincc);
                f.x = fma(ca, x, fma(ls, px, lc * en.pz));
                f.px = fma(-g * sa, x, fma(ca, px, sa * en.pz));
                f.y = fma(L, in.py, in.y);
                f.z = in.z - sa * x - lc * px + m56 * en.pz;
            }
        }
    }
    {
        const double pxy = f.px * f.y;
        f.x = fma(-a, f.y * f.y, f.x);
        f.py = fma(gi, pxy, f.py);
        f.z = fma(ai, pxy * f.y, f.z);
    }
}

// track_a_bend.f90:18-333 for a sector bend with a gradient (the k1 body map, :500-659), simple
// edges and g_tot = g. In each plane x'' = k x (about x_c in the horizontal one) with the plane
// functions as series in w = k L^2/(1+pz), |w| <= 1/16 (the first omitted term of C, w^7/14!, is
// below 5e-20): C = 1 + w D, D = 1/2 + w/4! + ..., S = 1 + w/3! + .... The second-order path
// length is fast_quad's; the first-order one is -g int x ds = -g (x_c L + L S r + L^2 D u).
// r: g, k_x = k1 + g^2, k1, g/k_x, L, L^2.
constexpr double kFastW = 1.0 / 16;
struct PlaneFns {
    double c, s, d;
};
__device__ __forceinline__ PlaneFns plane_fns(double w)
{
#pragma clang fp contract(off)
    double d = fma(w, 2.08767569878681e-09, 2.755731922398589e-07);  // 1/12!, 1/10!
    d = fma(d, w, 2.48015873015873e-05);                               // 1/8!
    d = fma(d, w, 0.001388888888888889);                               // 1/6!
    d = fma(d, w, 0.041666666666666664);                               // 1/4!
    d = fma(d, w, 0.5);
    double s = fma(w, 2.505210838544172e-08, 2.7557319223985893e-06);  // 1/11!, 1/9!
    s = fma(s, w, 0.0001984126984126984);                               // 1/7!
    s = fma(s, w, 0.008333333333333333);                                // 1/5!
    s = fma(s, w, 0.16666666666666666);                                 // 1/3!
    s = fma(s, w, 1.0);
    return {fma(w, d, 1.0), s, d};
}

template <class V>
__device__ __forceinline__ void fast_bend_k1(FastP &f, const FastE &en, const V &r, LaneMask &bad)
{
#pragma clang fp contract(off)
    const double g = r[0], kx = r[1], k1 = r[2], xcp = r[3], L = r[4], L2 = r[5];
    const double gi = g * en.inv_rp, a = 0.5 * gi, ai = a * en.inv_rp;
    {
        const double pxy = f.px * f.y;
        f.x = fma(a, f.y * f.y, f.x);
        f.py = fma(-gi, pxy, f.py);
        f.z = fma(-ai, pxy * f.y, f.z);
    }
    const double l2i = L2 * en.inv_rp, Li = L * en.inv_rp;
    const double wx = -(kx * l2i), wy = k1 * l2i;
    bad |= lanes(!(fabs(wx) <= kFastW)) | lanes(!(fabs(wy) <= kFastW));
    const PlaneFns X = plane_fns(wx), Y = plane_fns(wy);
    const double xc = xcp * en.pz;
    const double rx = f.x - xc, px = f.px, y = f.y, py = f.py;
    const double xp = fma(y, py, rx * px);
    const double p2 = fma(py, py, px * px);
    // L (u^2 - k x^2) (1+pz) with k = -k_x/(1+pz) and k1/(1+pz)
    double d = fma(Li, p2, -xp);
    d = fma(kx * L, rx * rx, d);
    d = fma(-(k1 * L), y * y, d);
    const double x1 = fma(Li * X.s, px, X.c * rx);
    const double px1 = fma(-(kx * (L * X.s)), rx, X.c * px);
    const double y1 = fma(Li * Y.s, py, Y.c * y);
    const double py1 = fma(k1 * (L * Y.s), y, Y.c * py);
    d = fma(x1, px1, d);
    d = fma(y1, py1, d);
    const double first = fma(L, fma(X.s, rx, xc), l2i * (X.d * px));
    f.x = x1 + xc;
    f.px = px1;
    f.y = y1;
    f.py = py1;
    f.z = fma(L, en.lez, fma(-0.25 * en.inv_rp, d, fma(-g, first, f.z)));
    {
        const double pxy = f.px * f.y;
        f.x = fma(-a, f.y * f.y, f.x);
        f.py = fma(gi, pxy, f.py);
        f.z = fma(ai, pxy * f.y, f.z);
    }
}

// The frame of an offset and tilted element, entering or leaving (offset_particle.f90:183-492
// without pitches or a longitudinal offset, whose drift to the face it then has none of):
// position and momenta turned by the tilt, the position then moved. r: cos, sin, move in x, in y.
template <class V>
__device__ __forceinline__ void fast_frame(FastP &f, const V &r)
{
#pragma clang fp contract(off)
    const double c = r[0], s = r[1], x = f.x, px = f.px;
    f.x = fma(c, x, fma(s, f.y, r[2]));
    f.y = fma(c, f.y, fma(-s, x, r[3]));
    f.px = fma(c, px, s * f.py);
    f.py = fma(c, f.py, -(s * px));
}

// The kernels whose map set carries the radiation kicks have this operation (bmx_maps.hpp).
struct RadAt {
    CP maps;          // the lattice's packed radiation maps
    uint32_t id;      // the particle's stream
    int32_t turn;
};

// The deviates of the columns `cols` of stoc_mat, in pairs (at: see fast_radiation).
__device__ __forceinline__ void rad_deviates(double *g, uint64_t at, uint32_t cols, const Species &sp,
                                             const RadAt &ra)
{
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    const int32_t edge = lo >> 24 & 1, ix1 = (int32_t)(hi >> 12);
#pragma unroll
    for (int b = 0; b < 3; b++) {
        g[2 * b] = g[2 * b + 1] = 0;
        if (cols >> (2 * b) & 3)
            gauss_pair(g[2 * b], g[2 * b + 1], ra.id, ra.turn, ix1, 4 * edge + b, sp.rad.key0, sp.rad.key1);
    }
}

// The kicked coordinates back in place; energy: pz may have changed.
__device__ __forceinline__ void rad_leave(FastP &f, FastE &en, const double *v, bool energy, const Species &sp,
                                          LaneMask &bad)
{
    f.x = v[0];
    f.px = v[1];
    f.y = v[2];
    f.py = v[3];
    f.z = v[4];
    bad |= lanes(!(v[5] > -0.5));
    if (energy) {
        en.pz = v[5];
        energy_functions(en.pz, en.bq, sp, en.rel_p, en.inv_rp, en.ez, en.lez);
        en.ir2 = en.inv_rp * en.inv_rp;
    }
}

// track1_radiation (radiation_mod.f90:61-147) at one end of an element, as rad_kick, on a map with
// its zero parts left out: `at` packs the map's first line in the lattice's radiation lines (low
// 24 bits), the edge (bit 24), the rows of damp_dmat and xfer_damp_vec that are not zero (bits 26-31), the
// rows and the columns of stoc_mat that are not (bits 32-37, 38-43), and the element's index (from
// bit 44). Lines of kFastOpLen values: ref_orb; then for each damping row its six coefficients and
// xfer_damp_vec; then for each stochastic row its coefficients. A row or column of zeros adds
// nothing to finite coordinates (others fail the tests), and a pair of deviates whose two columns
// are zero is not drawn: each pair comes from a counter of its own. The cell kernels have this
// written out instead, for the coefficients that are not zero in some cell (bmx_jit.cpp).
__device__ __forceinline__ void fast_radiation(FastP &f, FastE &en, uint64_t at, const Species &sp,
                                               const RadAt &ra, LaneMask &bad)
{
#pragma clang fp contract(off)
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)at);
    const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(at >> 32));
    CP m = ra.maps + (size_t)kFastOpLen * (lo & 0xFFFFFF);
    const uint32_t rows = lo >> 26, srows = hi & 63, scols = hi >> 6 & 63;
    double v[6] = {f.x, f.px, f.y, f.py, f.z, en.pz};
    bad |= lanes(!(fabs(f.z) < 1e30));
    const double rr = sp.rad.scale;
    if (sp.rad.flags & RAD_DAMP) {
        const OpVec ref = load_op(m);
        double d[6];
#pragma unroll
        for (int j = 0; j < 6; j++) d[j] = v[j] - ref[j];
        CP r = m + kFastOpLen;
#pragma unroll
        for (int i = 0; i < 6; i++) {
            if (rows >> i & 1) {
                const OpVec c = load_op(r);
                double s = c[0] * d[0];
#pragma unroll
                for (int j = 1; j < 6; j++) s = fma(c[j], d[j], s);
                v[i] = fma(rr, s, v[i]);
                if (!(sp.rad.flags & RAD_ZERO_AVERAGE)) v[i] = fma(rr, c[6], v[i]);
                r += kFastOpLen;
            }
        }
    }
    if (sp.rad.flags & RAD_FLUCT) {
        double g[6];
        rad_deviates(g, at, scols, sp, ra);
        CP r = m + kFastOpLen * (1 + __builtin_popcount(rows));
#pragma unroll
        for (int i = 0; i < 6; i++) {
            if (srows >> i & 1) {
                const OpVec c = load_op(r);
                double s = c[0] * g[0];
#pragma unroll
                for (int j = 1; j <= i; j++) s = fma(c[j], g[j], s);
                v[i] = fma(rr, s, v[i]);
                r += kFastOpLen;
            }
        }
    }
    rad_leave(f, en, v, (rows | srows) >> 5 & 1, sp, bad);
}

// An operation of kind `code` (FO_* with its FO_RECT and FO_UCHECK bits): values v[0..] as in its
// record, and the exit aperture's k2, r2. RAD: the map set carries the radiation kicks.
template <bool RAD, class V>
__device__ __forceinline__ void fast_op(FastP &f, FastE &en, uint32_t code, const V &v, double k2,
                                        double r2, const Species &sp, bool near, const RadAt &ra,
                                        LaneMask &bad)
{
    if (code & FO_UCHECK) fast_unstable(f, en, bad);
    switch (code & FO_KIND) {
    case FO_DRIFT: fast_drift(f, en, v[0], bad); break;
    case FO_QUAD: fast_quad<false>(f, en, v[0], v[1], v[2], bad); break;
    case FO_QUAD5: fast_quad<true>(f, en, v[0], v[1], v[2], bad); break;
    case FO_SEXT: fast_sextupole(f, en, v[0], v[1], v[2], bad); break;
    case FO_BEND: fast_bend(f, en, v, sp, near, bad); break;
    case FO_BEND_K1: fast_bend_k1(f, en, v, bad); break;
    case FO_KICK:
        f.px = f.px + v[0];
        f.py = f.py + v[1];
        return;
    case FO_FRAME: fast_frame(f, v); return;
    case FO_RAD:
        if constexpr (RAD) fast_radiation(f, en, __double_as_longlong(v[0]), sp, ra, bad);
        return;
    default: break;
    }
    if (code & FO_RECT) fast_aperture<true>(f, k2, r2, bad);
    else fast_aperture<false>(f, k2, r2, bad);
}

// Whether a lane of the wave may take the semi-linear bend before pz changes again (radiation
// kicks change it inside runs: there the bend itself looks).
template <int RARE>
__device__ __forceinline__ bool near_zero(const Particle &p)
{
    return maps_rad(RARE) || any_lane(fabs(p.pz) < 1e-9);
}

// The lane's bit of a mask.
__device__ __forceinline__ bool this_lane(LaneMask m) { return (m >> (threadIdx.x & 63)) & 1; }

// Keeps the loads written before it before it and those after it after it (arithmetic may cross).
__device__ __forceinline__ void load_fence() { __builtin_amdgcn_sched_barrier(0x1); }
// Waits for the scalar load of v here, so that the next one can be issued behind it: scalar
// loads return in any order, and waiting for one waits for every one in flight. (The word is
// taken through readfirstlane, so the wait compiles wherever the compiler holds v.)
__device__ __forceinline__ void arrive(const OpVec &v)
{
    const int32_t w = __builtin_amdgcn_readfirstlane((int32_t)__double_as_longlong(v[0]));
    asm volatile("" : : "s"(w));
    load_fence();
}

// What the next element by track_step starts from, read while the one before it is tracked: the
// element's operation codes and its first operation record. The records of a lattice follow one
// another in the order of its elements.
struct StepAhead {
    uint64_t codes[2];
    int32_t n_ops;
    CP r;       // the record in op
    OpVec op;
};

__device__ __forceinline__ void step_codes(StepAhead &s, const FastEle BMX_CONST *fe)
{
    s.codes[0] = fe->codes[0];
    s.codes[1] = fe->codes[1];
    s.n_ops = fe->n_ops;
}

__device__ __forceinline__ StepAhead step_at(const LatDesc &L, int32_t e)
{
    const FastEle BMX_CONST *fe = (const FastEle BMX_CONST *)L.fast + e;
    StepAhead s;
    step_codes(s, fe);
    s.r = (CP)L.ops + kFastOpLen * fe->op0;
    s.op = load_op(s.r);
    return s;
}

// One element for the active (live) lanes, by its definition: its operations where their tests
// hold, else the general map. RARE: the map set of elements on the rare path (bmx_maps.hpp).
// from_prev as track_element; e is wave-uniform. AHEAD: s is step_at(L, e) and becomes that of
// element e + 1 (of the last one again at the end of the lattice): a wave that goes through the
// elements one by one spends its time waiting for these tables, one read after the other, unless
// they are read ahead. Returns true when the particle was lost at the entrance aperture.
template <int RARE, bool AHEAD>
__device__ __forceinline__ bool track_step(Particle &p, FastE &en, const LatDesc &L, int32_t e,
                                           int32_t t_abs, bool from_prev, StepAhead &s)
{
    const CHdr h = (CHdr)L.hdr + 4 * e;
    const int32_t after = e + 1 < L.n_ele ? e + 1 : e;
    const FastEle BMX_CONST *fe = (const FastEle BMX_CONST *)L.fast + after;
    if constexpr (!AHEAD) step_codes(s, (const FastEle BMX_CONST *)L.fast + e);
    const int32_t n_ops = s.n_ops;
    LaneMask redo = ~(LaneMask)0;
    if (n_ops > 0) {
        const bool near = near_zero<RARE>(p);
        const RadAt ra = {(CP)L.rad, p.id, t_abs};
        FastP f = fast_get(p);
        FastE ef = en;
        LaneMask bad = 0;
        // an entrance test that repeats the exit test of an element not tracked before this one
        if (!from_prev && (h[1] & F_APE_ENT_SAME))
            bad = lanes(aperture_fails(p, h[1] & ~F_APE_CENTERED,
                                       (CP)L.prm + h[3] + ((h[1] & F_OFFSET) ? kOffsetLen : 0)));
        uint64_t w = s.codes[0];
        const uint64_t w1 = s.codes[1];
        if constexpr (!AHEAD) s.r = (CP)L.ops + kFastOpLen * ((const FastEle BMX_CONST *)L.fast + e)->op0;
        for (int32_t k = 0; k < n_ops; ++k) {
            k = __builtin_amdgcn_readfirstlane(k);
            OpVec v;
            if constexpr (AHEAD) {
                arrive(s.op);
                v = s.op;
                s.r += kFastOpLen;
                s.op = load_op(s.r);  // the table ends with a spare record
                if (k == 0) step_codes(s, fe);
                load_fence();
            } else {
                v = load_op(s.r);
                s.r += kFastOpLen;
            }
            const uint32_t code = (uint32_t)w & 255;
            w = k == 7 ? w1 : w >> 8;
            fast_op<maps_rad(RARE)>(f, ef, code, v, v[6], v[7], L.sp, near, ra, bad);
        }
        fast_unstable(f, ef, bad);
        if (!this_lane(bad)) {
            fast_put(p, f);
            if constexpr (maps_rad(RARE)) {
                en = ef;
                fast_put_energy(p, ef);
            }
        }
        redo = bad;
    }
    bool entrance = false;
    if (redo) {
        if (this_lane(redo)) {
            if (h[0] == K_RF || (h[1] & (F_OFFSET | F_APE_MOMENTUM | F_RARE_MAP))) {
                entrance = track_element<true, RARE>(p, load_ele(h), (CP)L.prm, L.sp, from_prev, e + 1, t_abs);
                en = fast_energy(p, L.sp);
            } else {
                entrance = track_element<true, MAPS_NO_RF>(p, load_ele(h), (CP)L.prm, L.sp, from_prev, e + 1, t_abs);
            }
        }
        if constexpr (AHEAD) s = step_at(L, after);  // read again, not held through the general maps
    }
    return entrance;
}

}  // namespace bmx
