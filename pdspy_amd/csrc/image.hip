// image.hip -- ray-traced images and their adjoint on gfx950: what RADMC-3D's
// camera computes for pdspy's Model.run_image (pdspy/modeling/Model.py:515-577,
// radmc3d/run.py:157-289), i.e. the formal solution
//     I = sum_k S_k (1 - exp(-dtau_k)) exp(-tau_k)
// along parallel rays, with S = B_nu(T) and absorption-only extinction
// (scattering_mode_max=0), or, given the scattering source's mean intensity J
// (scat.hip), extinction rho (kabs + ksca) and S = (rho kabs B + rho ksca J) /
// (rho kext) (isotropic scattering); plus blackbody point stars attenuated by
// the model (pdspy's nostar=False).  Pixel (j,k) is centred at
// ((k - nx/2) pix, (j - ny/2) pix) in the sky plane, the centring pdspy's
// zoomau produces (Model.py:522-527).
//
// Kernels: a per-cell prep pass (alpha and S per cell) so
// the ray loop reads 8 bytes per crossed cell; a ray's crossings split over
// lanes; the adjoint
// re-integrates each ray twice (first for I, then for dI/d dtau_k = e^-tau_k
// e^-dtau_k S_k - (I - I_<=k)) instead of storing tau, and accumulates
// dL/dalpha, dL/dS per cell as 64-bit fixed-point integers; a post pass applies
// the chain rule to log(rho_s) and T.
#include <algorithm>
#include <cmath>

#include "rt_internal.h"

using namespace rt;

struct CamParams {
    DevGrid g;
    float n[3];               // towards the observer
    double nd[3], ex[3], ey[3];
    double cpa, spa;
    double pix;      // au
    float pixf;
    int nx, ny, nsub, mode;
    int tw, th, ntx, nty;  // ray tiles: tw x th pixels, ntx per image row, nty rows of them
    unsigned hbits;   // adjoint LDS table: 2^hbits entries
    int lanes;        // lanes per ray (a power of two)
    float tau_stop;
    const float *alpha;  // [cell] per au
    const float *src;    // [cell]
    const float *csize;  // [cell] cell size for the sub-pixeling (au)
    unsigned long long *icount;  // cells crossed: [0] image rays, [1] adjoint sweeps
    const double *qs;  // adjoint: fixed-point units per unit of dL/dalpha, dL/dS
};

// adds the block's crossings n (summed over its threads) to *dst; every thread
// of the block calls it
__device__ __forceinline__ void count_crossings(unsigned long long *dst, uint32_t n) {
    __shared__ unsigned s_n;
    if (threadIdx.x == 0) s_n = 0u;
    __syncthreads();
    if (n) atomicAdd(&s_n, n);
    __syncthreads();
    if (threadIdx.x == 0 && s_n && dst) atomicAdd(dst, (unsigned long long)s_n);
}

// A camera ray is the line p0 + s d: p0 the point closest to the origin (in
// the sky plane through it), d = -n, s in [-S, S] inside the outer sphere.  All
// its crossings are known in closed form, so it is not marched from wall to
// wall:
//  * spheres: s = -+sqrt(R_i^2 - b^2), inwards down to the innermost one that
//    the ray meets, then outwards;
//  * cones: with z reflected so that z0 >= 0, u = z / r = cos(theta) rises
//    along the ray to u* = sqrt(z0^2 + dz^2 b^2) / b at s* = dz b^2 / z0 and
//    falls from there, so the walls met are those from the entry's down to u*'s
//    and back up to the exit's, wall c at s = (dz b^2 c -+ z0 Q) / (z0 c +- dz Q)
//    with Q = sqrt(z0^2 + b^2 (dz^2 - c^2)) (upper signs before s*, lower ones
//    after).  An equatorially mirrored grid is unfolded to 2 nt cells from pole
//    to pole;
//  * phi half-planes, in the order the ray turns about the axis.
// Each sequence is sorted and numbered, the k-th sphere or cone crossing costs
// one square root (and a quotient) whatever came before, in FP64, and the ray's
// segments are the merged sequence.  No test has to decide whether a wall is hit,
// so near-tangent rays need no care, and -- what it is done for -- a ray can be
// entered anywhere: `lanes` lanes take equal shares of the merged sequence (found
// by a binary search over the two sequences' counters) and combine their
// (optical depth, intensity) afterwards.  An image of 256 x 256 rays is 1024
// waves, one per SIMD, and a march of one ray per lane left it waiting on the
// longest chains (~700 crossings of ~6000 clocks: 1.47 ms); with 8 lanes per ray:
// 0.164 ms, paced by the FP64 instructions of the merge.
struct RayGeo {
    double b2, z0, dz, S;
    int nin, w;    // spheres met inwards (as many outwards); the innermost one
    int js, jt;    // theta cells of the entry and of u* (unfolded, flipped frame)
    int nA, nT;    // cone crossings before s*, and in all
    double x0, y0; // p0 in the equatorial plane (phi cells)
    bool flip;     // z reflected
};

// reciprocal: two Newton steps on the hardware's estimate
__device__ __forceinline__ double rcp_d(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// square root to a few ulp (positive arguments far from the ends of the range;
// anything below counts as 1e-280): Goldschmidt's iteration on the hardware's estimate
// of 1 / sqrt(x) and a last Newton step, without the library's scaling
__device__ __forceinline__ double sqrt_d(double x) {
    x = fmax(x, 1e-280);
    const double y = __builtin_amdgcn_rsq(x);
    double g = x * y, h = 0.5 * y;
    const double r = fma(-h, g, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    return fma(fma(-g, g, x), h, g);
}

// e^-x = s (1 + m) for x >= 0: s a power of two, m = e^r - 1 of the rest r of the
// division by ln 2 (in two parts), |r| < 0.36, or of -x itself below 0.5, by its series
// up to r^8 / 8!
__device__ __forceinline__ void exp_parts(float x, float &s, float &m) {
    const float y = x > 1000.f ? 1000.f : x;  // (NaN stays)
    const float n = y < 0.5f ? 0.f : rintf(y * -1.44269504f);
    float r = fmaf(n, -0.693145751953125f, -y);
    r = fmaf(n, -1.42860682e-6f, r);
    float p = 1.f / 40320.f;
    p = fmaf(p, r, 1.f / 5040.f);
    p = fmaf(p, r, 1.f / 720.f);
    p = fmaf(p, r, 1.f / 120.f);
    p = fmaf(p, r, 1.f / 24.f);
    p = fmaf(p, r, 1.f / 6.f);
    p = fmaf(p, r, 0.5f);
    m = fmaf(r, p * r, r);
    s = ldexpf(1.f, (int)n);
}

// 1 - e^-x to 7.2e-8 (rounding alone: 6e-8)
__device__ __forceinline__ float one_minus_exp(float x) {
    float s, m;
    exp_parts(x, s, m);
    return fmaf(-s, m, 1.f - s);
}

// cells of the unfolded theta axis, its walls' cosines (descending) and the
// grid's cell of an unfolded one
__device__ __forceinline__ int ntheta_u(const DevGrid &g) { return g.mirror ? 2 * g.nt : g.nt; }
__device__ __forceinline__ double cos_u(const DevGrid &g, bool flip, int j) {
    const int n = ntheta_u(g);
    const bool neg = g.mirror ? j > g.nt : flip;  // (one load, whichever side)
    const double c = g.ctd[neg ? n - j : j];
    return neg ? -c : c;
}
__device__ __forceinline__ int fold_u(const DevGrid &g, bool flip, int j) {
    const bool neg = g.mirror ? j >= g.nt : flip;
    return neg ? ntheta_u(g) - 1 - j : j;
}
// the unfolded cell j with cos(wall j) > u >= cos(wall j + 1)
__device__ __forceinline__ int find_u(const DevGrid &g, bool flip, double u) {
    int lo = 0, hi = ntheta_u(g);
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cos_u(g, flip, mid) > u)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// the crossing sequences of the ray with p0 at (q.x0, q.y0, q.z0) and q.b2; false:
// it misses the grid.  clear > 0: spheres of R^2 <= b^2 (1 + clear), which a march
// in FP32 may take for missed, are left out.
__device__ __forceinline__ bool ray_geometry(const CamParams &C, RayGeo &q, double clear) {
    const DevGrid &g = C.g;
    const double R = g.rwd[g.nr];
    q.dz = -C.nd[2];
    if (!(q.b2 < R * R)) return false;
    q.S = sqrt(R * R - q.b2);
    q.flip = q.z0 < 0.0;
    if (q.flip) {
        q.z0 = -q.z0;
        q.dz = -q.dz;
    }
    // innermost sphere met: the first with R_w > b
    int lo = -1, hi = g.nr;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        const double r = g.rwd[mid];
        if (r * r > q.b2 * (1.0 + clear))
            hi = mid;
        else
            lo = mid;
    }
    q.w = hi;
    q.nin = g.nr - hi;
    // theta cells of the entry, the turning point and the exit
    const double iR = rcp_d(R), b = sqrt(q.b2);
    const double us = (q.z0 - q.S * q.dz) * iR, ue = (q.z0 + q.S * q.dz) * iR;
    const double ut = sqrt(fma(q.z0, q.z0, q.dz * q.dz * q.b2)) * rcp_d(b);
    const double st = q.dz * q.b2;  // s* z0
    q.js = find_u(g, q.flip, us);
    const int je = find_u(g, q.flip, ue);
    // s* outside [-S, S]: u is monotonic there
    q.jt = st <= -q.S * q.z0 ? q.js : (st >= q.S * q.z0 ? je : find_u(g, q.flip, ut));
    q.jt = min(q.jt, min(q.js, je));
    q.nA = q.js - q.jt;
    q.nT = q.nA + je - q.jt;
    return true;
}

// p0 and b^2 of the ray through sky position (X, Y) (au)
__device__ __forceinline__ void ray_line(const CamParams &C, double X, double Y, RayGeo &q) {
    const double R = C.g.rwd[C.g.nr];
    double xp = X * C.cpa + Y * C.spa, yp = -X * C.spa + Y * C.cpa;
    // a ray through the origin is moved off it by 1e-12 of the grid's radius
    // (which direction it would turn to there is not defined)
    if (xp * xp + yp * yp < 1e-24 * R * R) yp = 1e-12 * R;
    q.x0 = xp * C.ex[0] + yp * C.ey[0];
    q.y0 = xp * C.ex[1] + yp * C.ey[1];
    q.z0 = xp * C.ex[2] + yp * C.ey[2];
    q.b2 = fma(q.x0, q.x0, fma(q.y0, q.y0, q.z0 * q.z0));
}

// the ray through sky position (X, Y) (au); false: it misses the grid
__device__ __forceinline__ bool ray_setup(const CamParams &C, double X, double Y, RayGeo &q) {
    ray_line(C, X, Y, q);
    return ray_geometry(C, q, 0.0);
}

// position of the k-th sphere crossing (k = 2 nin: the outer sphere)
__device__ __forceinline__ double sph_at(const CamParams &C, const RayGeo &q, int k) {
    const bool inw = k < q.nin;
    const double r = C.g.rwd[inw ? C.g.nr - 1 - k : q.w + k - q.nin];
    const double s = sqrt_d(fma(r, r, -q.b2));
    return inw ? -s : s;
}

// position of the k-th cone crossing (none left: beyond every sphere)
__device__ __forceinline__ double cone_at(const CamParams &C, const RayGeo &q, int k) {
    if (k >= q.nT) return 1e300;
    const bool A = k < q.nA;
    const double c = cos_u(C.g, q.flip, A ? q.js - k : q.jt + 1 + k - q.nA);
    const double Q = sqrt_d(fma(q.b2, fma(q.dz, q.dz, -c * c), q.z0 * q.z0));
    const double sQ = A ? -Q : Q;
    const double s = fma(q.dz * q.b2, c, q.z0 * sQ) * rcp_d(fma(q.z0, c, -q.dz * sQ));
    return s > -q.S ? (s < q.S ? s : q.S) : -q.S;   // (NaN: -S)
}

// position where the ray, turning in direction `up` about the axis, leaves phi
// cell ip; 1e300 if it never does
__device__ __forceinline__ double phi_at(const CamParams &C, const RayGeo &q, int ip, bool up, double s) {
    const int k = up ? ip + 1 : ip;
    const double cp = C.g.cp[k], sp = C.g.sp[k];
    const double dx = -C.nd[0], dy = -C.nd[1];
    const double den = dy * cp - dx * sp;
    if (up ? !(den > 0.0) : !(den < 0.0)) return 1e300;
    const double t = (q.x0 * sp - q.y0 * cp) * rcp_d(den);
    // In a cell of more than half a turn, a wall ahead of the cell may be one that the
    // line has passed behind the position (to come round into the cell by its other
    // end): it is not met again.  Such a position lies past the wall by what the other
    // cells turn at least.  One just past it is there because a share's first cell is
    // found in FP32, with angles good to 1e-6, and has yet to cross.
    if (t < s) {
        const double w = (double)C.g.pw[ip + 1] - (double)C.g.pw[ip];
        if (w > 3.1416) {
            const double x = fma(s, dx, q.x0), y = fma(s, dy, q.y0);
            const double sn = fabs(fma(y, cp, -(x * sp))), cs = fma(x, cp, y * sp);
            if (!(sn <= fmin(4e-6, 0.5 * (6.283185307179586 - w)) * cs)) return 1e300;
        }
    }
    return fmax(t, s);
}

// Lane `l` of `L` walks its share of the ray's segments: f(cell, length) for each
// of them that lies in a cell, until f returns true.
template <class F>
__device__ __forceinline__ void walk_ray(const CamParams &C, const RayGeo &q, int l, int L, F f) {
    const DevGrid &g = C.g;
    const int NR = 2 * q.nin + 1, M = NR + q.nT;
    const int m0 = (int)(((long long)M * l) / L), m1 = (int)(((long long)M * (l + 1)) / L);
    if (m0 >= m1) return;
    // the first m0 crossings: kr spheres and kt cones (a sphere first on a tie)
    int lo = max(0, m0 - q.nT), hi = min(m0, NR);
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (sph_at(C, q, mid) <= cone_at(C, q, m0 - 1 - mid))
            lo = mid + 1;
        else
            hi = mid;
    }
    int kr = lo, kt = m0 - lo;
    if (kr >= NR) return;  // cones beyond the outer sphere by rounding
    double s = -q.S;
    if (kr > 0) s = fmax(s, sph_at(C, q, kr - 1));
    if (kt > 0) s = fmax(s, cone_at(C, q, kt - 1));
    double sr = sph_at(C, q, kr), st = cone_at(C, q, kt);
    int ir = kr <= q.nin ? g.nr - 1 - kr : q.w - 1 + kr - q.nin;
    int it = fold_u(g, q.flip, kt <= q.nA ? q.js - kt : q.jt + kt - q.nA);
    int ip = 0;
    double sp = 1e300;
    int nphi = g.np;  // a ray turns by less than a whole turn: each wall once at most
    bool up = true;
    if (g.np > 1) {
        up = q.x0 * -C.nd[1] - q.y0 * -C.nd[0] >= 0.0;
        float ph = atan2f((float)(q.y0 - s * C.nd[1]), (float)(q.x0 - s * C.nd[0]));
        if (ph < 0.f) ph += 6.28318530718f;
        ip = search_walls(g.pw, g.np, ph);
        sp = phi_at(C, q, ip, up, s);
    }
    for (int n = m1 - m0; n > 0;) {
        double sn = fmin(sr, st);
        const bool phi = sp < sn;
        sn = fmax(phi ? sp : sn, s);
        if (ir >= 0)
            if (f(ir + g.nr * (it + g.nt * ip), (float)(sn - s))) return;
        s = sn;
        if (phi) {
            ip = up ? (ip + 1 < g.np ? ip + 1 : 0) : (ip > 0 ? ip - 1 : g.np - 1);
            sp = --nphi > 0 ? phi_at(C, q, ip, up, s) : 1e300;
            continue;
        }
        --n;
        if (sr <= st) {
            ++kr;
            if (kr >= NR) return;
            ir = kr <= q.nin ? g.nr - 1 - kr : q.w - 1 + kr - q.nin;
            sr = sph_at(C, q, kr);
        } else {
            ++kt;
            it = fold_u(g, q.flip, kt <= q.nA ? q.js - kt : q.jt + kt - q.nA);
            st = cone_at(C, q, kt);
        }
    }
}

// ---- the march of the adjoint.  A gradient's value hangs on which cell a piece
// of a ray is charged to: where a ray grazes a cone for long, a shift of the wall
// by an ulp of the radius (1e-5 au at 200 au) moves up to 1e-3 of a cell's
// gradient to its neighbour, and either is as good.  The adjoint keeps the FP32
// march from wall to wall (next_wall) that defines those gradients, and takes
// from the sequences above only where a lane's share begins: at a radial
// crossing, where the march sets its position on the line again (put_on_sphere) and
// so depends on nothing before it.
struct CamRay {
    float x0, y0, z0;  // p0 (au)
    double b2;         // |p0|^2
};

// the ray's line in FP32; false: it misses the grid
__device__ __forceinline__ bool cam_line(const CamParams &C, float X, float Y, CamRay &cr) {
    const float cpa = (float)C.cpa, spa = (float)C.spa;
    const float xp = fmaf(cpa, X, spa * Y), yp = fmaf(-spa, X, cpa * Y);
    cr.x0 = fmaf((float)C.ex[0], xp, (float)C.ey[0] * yp);
    cr.y0 = fmaf((float)C.ex[1], xp, (float)C.ey[1] * yp);
    cr.z0 = fmaf((float)C.ex[2], xp, (float)C.ey[2] * yp);
    const double x = cr.x0, y = cr.y0, z = cr.z0, R = C.g.rwd[C.g.nr];
    cr.b2 = fma(z, z, fma(x, x, y * y));
    return cr.b2 < R * R;
}

// puts p on the line at the sphere of wall iw, inbound or outbound
__device__ __forceinline__ void put_on_sphere(const DevGrid &g, const CamRay &cr, int iw, bool inw,
                                              Pos &p) {
    const double rw = g.rwd[iw];
    float s = (float)sqrt(fmax(fma(rw, rw, -cr.b2), 0.0));
    if (inw) s = -s;
    p.x = fmaf(s, p.dx, cr.x0);
    p.y = fmaf(s, p.dy, cr.y0);
    p.z = fmaf(s, p.dz, cr.z0);
}

// Lane l of L marches its share: from the sphere its equal part of the merged
// crossings begins at (the ray's entry for lane 0) to the one where the next
// lane's does.  `at` counts the spheres passed as RayGeo does.  imin: the innermost
// shell of the exact line (a sphere it is tangent to is met or missed as there).
template <class F>
__device__ __forceinline__ void march_ray(const CamParams &C, const CamRay &cr, const RayGeo &q,
                                          int imin, int l, int L, F f) {
    const DevGrid &g = C.g;
    const int NR = 2 * q.nin + 1, M = NR + q.nT;
    int at[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int m0 = (int)(((long long)M * (l + e)) / L);
        int lo = max(0, m0 - q.nT), hi = min(m0, NR);
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sph_at(C, q, mid) <= cone_at(C, q, m0 - 1 - mid))
                lo = mid + 1;
            else
                hi = mid;
        }
        at[e] = l + e == L ? NR : lo;
    }
    if (at[0] >= at[1]) return;
    Pos p;
    p.dx = -C.n[0];
    p.dy = -C.n[1];
    p.dz = -C.n[2];
    const int k = at[0];
    p.ir = k <= q.nin ? g.nr - 1 - k : q.w - 1 + k - q.nin;
    if (k <= q.nin)
        put_on_sphere(g, cr, g.nr - k, true, p);
    else
        put_on_sphere(g, cr, p.ir, false, p);
    p.it = p.ip = 0;
    p.hemi = 1;
    locate_angles<1>(g, p);
    uint32_t nzero = 0;
    for (int guard = 0; guard < (1 << 24); ++guard) {
        int kind;
        const float tw = next_wall<1, true>(g, p, kind, p.ir <= imin);
        const float rcell = g.rw[p.ir + 1];
        if (p.ir >= 0 && f(cell_index(g, p), tw)) return;
        if (kind == W_RIN || kind == W_ROUT || kind == W_HOLE) {
            const bool inw = kind == W_RIN;
            const int ir = kind == W_HOLE ? 0 : p.ir + (inw ? -1 : 1);
            p.ir = ir;
            if ((inw ? min(g.nr - 1 - ir, q.nin) : q.nin + ir - q.w + 1) >= at[1]) return;
            put_on_sphere(g, cr, inw ? ir + 1 : ir, inw, p);
            if (kind == W_HOLE) locate_angles<1>(g, p);
        } else {
            cross_wall(g, p, tw, kind);
        }
        if (unstick(g, p, tw, rcell, nzero) && p.ir >= g.nr) return;
    }
}

// what a lane's share of a ray adds up to
template <class A>
struct RaySum {
    A I;          // its own emission, attenuated from its own front on
    float tau;    // its own optical depth
    float tau0;   // optical depth in front of it
    A front;      // attenuation in front of it (0: the ray has ended there, tau_stop)
    float lmin;   // smallest cell size on the part traced (LMIN)
};

// 1 - e^-dtau and e^-dtau as two numbers that sum to 1
__device__ __forceinline__ void absorb(float dtau, double &om, double &e) {
    float s, m;
    exp_parts(dtau, s, m);
    om = fma(-(double)s, (double)m, 1.0 - (double)s);
    e = fma((double)s, (double)m, (double)s);
}

// The formal solution along the ray by L neighbouring lanes; every lane gets the
// ray's value (the intensity, or tau).  A ray ends once its optical depth
// exceeds tau_stop: the share it ends in is walked again with the optical depth
// in front of it, the shares behind it count for nothing.  A: type the intensity
// is summed in; in double (the adjoint) the attenuation is the running product
// of the segments' e^-dtau, so that emission and attenuation of a segment add up
// to what comes in, whatever their rounding.
template <bool LMIN, class A, class W>
__device__ __forceinline__ A trace_ray(const CamParams &C, const W &walk, bool act, int l, int L,
                                       RaySum<A> &r, uint32_t &nseg) {
    r.I = 0;
    r.tau = r.tau0 = 0.f;
    r.front = 1;
    r.lmin = RT_INF;
    uint32_t ns = 0;
    A att = 1;
    const bool inten = C.mode == 0;
    auto share = [&](float tau0) {
        float tau = 0.f, lm = RT_INF;
        A I = 0;
        att = 1;
        ns = 0;
        walk([&](int c, float ds) {
            ++ns;
            if (LMIN) lm = fminf(lm, C.csize[c]);
            const float dtau = C.alpha[c] * ds;
            if (inten) {
                if (sizeof(A) == 8) {
                    double om, e;
                    absorb(dtau, om, e);
                    I = fma((A)(att * om), (A)C.src[c], I);
                    att *= (A)e;
                } else {
                    I = fma((A)(__expf(-tau) * one_minus_exp(dtau)), (A)C.src[c], I);
                }
            }
            tau += dtau;
            return inten && tau0 + tau > C.tau_stop;
        });
        r.I = I;
        r.tau = tau;
        r.lmin = lm;
    };
    if (act) share(0.f);
    if (L > 1) {
        float t = r.tau;
        A f = att;
        for (int o = 1; o < L; o <<= 1) {
            const float v = __shfl_up(t, o, L);
            const A w = __shfl_up(f, o, L);
            if (l >= o) {
                t += v;
                f *= w;
            }
        }
        t = __shfl_up(t, 1, L);
        f = __shfl_up(f, 1, L);
        r.tau0 = l > 0 ? t : 0.f;
        // The ray ends in the first share that takes it over tau_stop.  What lies
        // behind must not count, whatever it is: that share, walked with the optical
        // depth in front of it unknown, may have gone on into cells whose opacity or
        // source is not finite, and so have those after it (hence NaN is "over" too).
        const bool over = inten && !(r.tau0 + r.tau <= C.tau_stop);
        const uint64_t ends = __ballot(over) >> (__lane_id() - l);
        if (inten) {
            const bool past = (ends & ((1ull << l) - 1ull)) != 0ull;
            if (act && over && !past && l > 0) share(r.tau0);
            r.front = past ? (A)0 : sizeof(A) == 8 ? (l > 0 ? f : (A)1) : (A)__expf(-r.tau0);
            if (past) {
                r.I = 0;
                r.lmin = RT_INF;
                ns = 0;
            }
        }
        A x = inten ? r.I * r.front : (A)r.tau;
        for (int o = 1; o < L; o <<= 1) x += __shfl_xor(x, o, L);
        if (LMIN)
            for (int o = 1; o < L; o <<= 1) r.lmin = fminf(r.lmin, __shfl_xor(r.lmin, o, L));
        nseg += ns;
        return x;
    }
    nseg += ns;
    return inten ? r.I : (A)r.tau;
}

// pixel of the n-th ray group: the image's tiles in order, the tile's pixels
__device__ __forceinline__ bool tile_pixel(const CamParams &C, unsigned n, int &j, int &k) {
    const unsigned tp = (unsigned)(C.tw * C.th), tile = n / tp, t = n - tile * tp;
    const int ty = (int)tile / C.ntx, tx = (int)tile - ty * C.ntx;
    const int dy = (int)t / C.tw, dx = (int)t - dy * C.tw;
    k = tx * C.tw + dx;
    j = ty * C.th + dy;
    return k < C.nx && j < C.ny;
}

__device__ __forceinline__ double sky_x(const CamParams &C, int k, int b) {
    return ((double)(k - C.nx / 2) + ((b + 0.5) / C.nsub - 0.5)) * C.pix;
}
__device__ __forceinline__ double sky_y(const CamParams &C, int j, int a) {
    return ((double)(j - C.ny / 2) + ((a + 0.5) / C.nsub - 0.5)) * C.pix;
}

// (in FP32, as the adjoint's march takes them)
__device__ __forceinline__ float sky_f(const CamParams &C, int k, int n, int b) {
    return ((float)(k - n / 2) + ((b + 0.5f) / C.nsub - 0.5f)) * C.pixf;
}

#define IMG_BS 256
#define IMG_LANES 524288u  // lanes a launch is spread over, if the rays allow
#define IMG_MAXL 32         // at most this many of them per ray

__global__ void __launch_bounds__(IMG_BS) k_image(CamParams C, float *img) {
    int j, k;
    uint32_t nseg = 0;
    const int L = C.lanes, l = (int)(threadIdx.x & (unsigned)(L - 1));
    const unsigned n = (blockIdx.x * IMG_BS + threadIdx.x) / (unsigned)L;
    const bool in = tile_pixel(C, n, j, k);
    float acc = 0.f;
    for (int a = 0; a < C.nsub; ++a)
        for (int b = 0; b < C.nsub; ++b) {
            RayGeo q;
            RaySum<float> r;
            const bool act = in && ray_setup(C, sky_x(C, k, b), sky_y(C, j, a), q);
            auto walk = [&](auto f) { walk_ray(C, q, l, L, f); };
            acc += trace_ray<false>(C, walk, act, l, L, r, nseg);
        }
    if (in && l == 0) img[j * C.nx + k] = acc / (float)(C.nsub * C.nsub);
    count_crossings(C.icount, nseg);
}

// The adjoint's per-cell sums are 64-bit fixed-point integers (units in
// C.qs, set by k_adj_scale): integer adds commute, so the gradient does not
// depend on the order in which rays and blocks add to a cell -- it is
// bit-reproducible, as the thermal tallies are.  They are first gathered in a
// small open-addressing table in LDS: the rays of one block are neighbours on
// the sky and cross mostly the same cells, so each cell then costs one global
// atomic per block instead of one per ray.  Entries: 2^hbits keys (cell index,
// -1 = empty) and two sums; a contribution that finds no slot in 8 probes goes
// straight to global memory.
typedef unsigned long long u64;
__device__ __forceinline__ void adj_add(int c, long long va, long long vs, int *key, u64 *ga,
                                        u64 *gs, unsigned hbits, double *g_alpha,
                                        double *g_src) {
    const unsigned mask = (1u << hbits) - 1u;
    unsigned slot = ((unsigned)c * 2654435761u) >> (32u - hbits);
    for (int probe = 0; probe < 8; ++probe) {
        int cur = __hip_atomic_load(&key[slot], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (cur == -1) {
            int exp = -1;
            __hip_atomic_compare_exchange_strong(&key[slot], &exp, c, __ATOMIC_RELAXED,
                                                 __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            cur = exp == -1 ? c : exp;
        }
        if (cur == c) {
            __hip_atomic_fetch_add(&ga[slot], (u64)va, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(&gs[slot], (u64)vs, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            return;
        }
        slot = (slot + 1u) & mask;
    }
    atomicAdd((u64 *)&g_alpha[c], (u64)va);
    atomicAdd((u64 *)&g_src[c], (u64)vs);
}

// the block's LDS table into the global sums
__device__ __forceinline__ void adj_flush(const int *key, const u64 *ga, const u64 *gs,
                                          unsigned H, double *g_alpha, double *g_src) {
    for (unsigned i = threadIdx.x; i < H; i += blockDim.x) {
        const int c = key[i];
        if (c >= 0) {
            if (ga[i]) atomicAdd((u64 *)&g_alpha[c], ga[i]);
            if (gs[i]) atomicAdd((u64 *)&g_src[c], gs[i]);
        }
    }
}

// gI times the gradient of the ray through sky (X, Y) ((Xf, Yf) in FP32) w.r.t. the per-cell
// alpha and S, by L neighbouring lanes: the ray is integrated for I, then each
// lane sweeps its share again front to back recomputing tau (nothing is stored
// per segment).  What lies behind segment k, R_k = I - I_<=k, is what the same
// sums leave of the lane's own share (the sweep repeats the integration's
// operations, in FP64, so no rounding is left over where R_k is small) plus the
// shares behind it.
__device__ __forceinline__ void adjoint_ray(const CamParams &C, double X, double Y, float Xf,
                                            float Yf, float gI, int l, int L, int *key, u64 *ga, u64 *gs, double *g_alpha,
                                            double *g_src, uint32_t &nseg) {
    RayGeo q;
    CamRay cr;
    RaySum<double> r;
    int imin = 0;
    bool act = gI != 0.f && cam_line(C, Xf, Yf, cr);
    if (act) {
        ray_line(C, X, Y, q);
        const double b2 = q.b2;
        q.x0 = cr.x0;
        q.y0 = cr.y0;
        q.z0 = cr.z0;
        q.b2 = cr.b2;
        if (cr.b2 == 0.0) ray_line(C, X, Y, q);  // (for the shares only)
        act = ray_geometry(C, q, 1e-4);
        if (act) {
            imin = q.w - 1;
            for (; imin >= 0; --imin) {
                const double w = C.g.rwd[imin];
                if (!(w * w > b2)) break;
            }
        }
    }
    uint32_t nfwd = 0;
    auto walk = [&](auto f) { march_ray(C, cr, q, imin, l, L, f); };
    (void)trace_ray<false>(C, walk, act, l, L, r, nfwd);
    double behind = r.I * r.front;
    if (L > 1) {
        double x = behind;
        for (int o = 1; o < L; o <<= 1) {
            const double v = __shfl_down(x, o, L);
            if (l + o < L) x += v;
        }
        behind = __shfl_down(x, 1, L);
    }
    if (l == L - 1) behind = 0.0;
    if (!act || r.front == 0.0) return;
    const double qa = C.qs[0] * (double)gI, qsrc = C.qs[1] * (double)gI;
    float tau = 0.f;
    double cum = 0.0, att = 1.0;
    walk([&](int c, float ds) {
        ++nseg;
        const float dtau = C.alpha[c] * ds;
        const double S = C.src[c];
        double om, e;
        absorb(dtau, om, e);
        const double em = att * om;
        cum = fma(em, S, cum);
        att *= e;
        const double dI_ddtau = r.front * fma(att, S, cum - r.I) - behind;
        adj_add(c, __double2ll_rn(dI_ddtau * (double)ds * qa),
                __double2ll_rn(r.front * em * qsrc), key, ga, gs, C.hbits, g_alpha, g_src);
        tau += dtau;
        return r.tau0 + tau > C.tau_stop;
    });
}

__global__ void __launch_bounds__(IMG_BS) k_image_adj(CamParams C, const float *dimg, double *g_alpha,
                                                      double *g_src) {
    extern __shared__ u64 adj_lds[];
    const unsigned H = 1u << C.hbits;
    u64 *ga = adj_lds, *gs = adj_lds + H;
    int *key = (int *)(adj_lds + 2 * H);
    for (unsigned i = threadIdx.x; i < H; i += blockDim.x) {
        key[i] = -1;
        ga[i] = 0ull;
        gs[i] = 0ull;
    }
    __syncthreads();
    int j, k;
    const int L = C.lanes, l = (int)(threadIdx.x & (unsigned)(L - 1));
    const bool in = tile_pixel(C, (blockIdx.x * IMG_BS + threadIdx.x) / (unsigned)L, j, k);
    const float gI = in ? dimg[j * C.nx + k] / (float)(C.nsub * C.nsub) : 0.f;
    uint32_t nseg = 0;
    for (int a = 0; a < C.nsub; ++a)
        for (int b = 0; b < C.nsub; ++b)
            adjoint_ray(C, sky_x(C, k, b), sky_y(C, j, a), sky_f(C, k, C.nx, b),
                        sky_f(C, j, C.ny, a), gI, l, L, key, ga, gs, g_alpha, g_src, nseg);
    __syncthreads();
    adj_flush(key, ga, gs, H, g_alpha, g_src);
    count_crossings(C.icount ? C.icount + 1 : nullptr, nseg);
}

// ---------------------------------------------------------------- sub-pixels
// Recursive sub-pixeling (RADMC-3D's camera_nrrefine / camera_refine_criterion,
// as pdspy leaves them at RADMC-3D's defaults): a (sub)pixel of side d whose
// central ray crosses a cell of size l with d > crit l is replaced by the mean
// of its 2 x 2 sub-pixels.  Done breadth first over a node pool: every node of
// level L is traced by ref_lanes of the level's size, the first of which hands its
// four children (at most RT_MAX_REFINE levels deep) their slots in level L + 1 with
// one atomic per wavefront; the values are then averaged bottom-up, level by level.  Siblings
// are summed in a fixed order, so the image does not depend on the order in
// which slots were handed out.  The adjoint hands each leaf ray the pixel's
// cotangent divided by 4 per level and runs the per-ray reverse sweep.
#define RT_REF_DEAD 1.0e30f  // sky position of a node with no ray (tile padding, no room)

struct RefArgs {
    float2 *xy;       // sky position of the node's central ray (au)
    float *val;       // its value (intensity or tau)
    int *child;       // first of its four children, -1: a leaf
    float *gw;        // adjoint: its cotangent
    unsigned *ctl;    // control words (RT_REF_*)
    unsigned cap;     // pool size (nodes)
    float crit;       // refine criterion
    int nref;         // levels that may split
    float d0;         // side of a level-0 node (au): pixel / nsub
    unsigned n0;      // level-0 nodes: every tile's pixels x nsub^2
    unsigned nray0;   // those of them that lie in the image
    int ns2;          // nsub^2
};

// level-0 node i: tiles in order, the tile's pixels, then the pixel's nsub^2
// sub-rays, so the rays of a wavefront are neighbours on the sky
__device__ __forceinline__ bool node0_pixel(const CamParams &C, int ns2, unsigned i, int &j, int &k,
                                            int &a, int &b) {
    const unsigned tp = (unsigned)(C.tw * C.th);
    const unsigned sub = i % (unsigned)ns2, q = i / (unsigned)ns2;
    const unsigned t = q / tp, r = q - t * tp;
    const int ty = (int)t / C.ntx, tx = (int)t - ty * C.ntx;
    const int dy = (int)r / C.tw, dx = (int)r - dy * C.tw;
    k = tx * C.tw + dx;
    j = ty * C.th + dy;
    a = (int)sub / C.nsub;
    b = (int)sub - a * C.nsub;
    return k < C.nx && j < C.ny;
}

__device__ __forceinline__ unsigned pixel_node0(const CamParams &C, int ns2, int j, int k, int sub) {
    const int ty = j / C.th, tx = k / C.tw;
    const unsigned t = (unsigned)(ty * C.ntx + tx);
    const unsigned r = (unsigned)((j - ty * C.th) * C.tw + (k - tx * C.tw));
    return (t * (unsigned)(C.tw * C.th) + r) * (unsigned)ns2 + (unsigned)sub;
}

__global__ void k_ref_init(CamParams C, RefArgs R) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0) {
        R.ctl[0] = R.n0;
        R.ctl[1] = 0u;
        for (int L = 1; L <= RT_MAX_REFINE + 1; ++L) R.ctl[1 + L] = R.n0;
        R.ctl[RT_REF_RAYS] = 0u;
    }
    if (i >= R.n0) return;
    int j, k, a, b;
    float2 xy = make_float2(RT_REF_DEAD, RT_REF_DEAD);  // tile padding: no ray
    if (node0_pixel(C, R.ns2, i, j, k, a, b)) {
        xy.x = sky_f(C, k, C.nx, b);
        xy.y = sky_f(C, j, C.ny, a);
    }
    R.xy[i] = xy;
}

// lanes per ray for n rays: about four waves per SIMD, and no more than a ray's
// crossings are worth.  A ray's sums are rounded by its shares, so n is a number
// that the image alone decides: the nodes that tiles add beyond its edges are
// not counted
__device__ __host__ __forceinline__ int ref_lanes(unsigned n) {
    int L = 1;
    while (L < IMG_MAXL && (size_t)n * (size_t)(2 * L) <= IMG_LANES) L *= 2;
    return L;
}

// traces level L: value of every node, children for those that split
__global__ void __launch_bounds__(256) k_ref_trace(CamParams C, RefArgs R, int L) {
    const unsigned start = R.ctl[1 + L], end = R.ctl[2 + L];
    const float d = ldexpf(R.d0, -L);
    const bool may_split = L < R.nref;
    const int lane = __lane_id();
    unsigned nrays = 0;
    uint32_t nseg = 0;
    const int LN = ref_lanes(L == 0 ? R.nray0 : end > start ? end - start : 0u),
              l = (int)(threadIdx.x & (unsigned)(LN - 1));
    const unsigned per = blockDim.x / (unsigned)LN;  // nodes of a block
    for (unsigned base = start + blockIdx.x * per; base < end; base += gridDim.x * per) {
        const unsigned i = base + threadIdx.x / (unsigned)LN;
        const bool act = i < end;
        float2 xy = make_float2(RT_REF_DEAD, RT_REF_DEAD);
        if (act) xy = R.xy[i];
        RayGeo q;
        RaySum<float> r;
        const bool ray = act && xy.x < 0.5f * RT_REF_DEAD && ray_setup(C, xy.x, xy.y, q);
        auto walk = [&](auto f) { walk_ray(C, q, l, LN, f); };
        const float I = trace_ray<true>(C, walk, ray, l, LN, r, nseg);
        const bool first = act && l == 0;
        if (first) R.val[i] = I;
        if (first && ray) ++nrays;
        const bool want = first && may_split && d > R.crit * r.lmin;
        const uint64_t mk = __ballot(want);
        int ch = -1;
        if (mk) {
            const int cnt = __popcll(mk);
            const int leader = __ffsll((unsigned long long)mk) - 1;
            // slots are only handed out while the pool has room (the count
            // stays within a wavefront's 256 slots of the pool size)
            unsigned b0 = R.cap;
            if (lane == leader && __hip_atomic_load(&R.ctl[0], __ATOMIC_RELAXED,
                                                    __HIP_MEMORY_SCOPE_AGENT) < R.cap)
                b0 = atomicAdd(&R.ctl[0], 4u * (unsigned)cnt);
            b0 = __shfl(b0, leader);
            if (want) {
                const unsigned c0 = b0 + 4u * (unsigned)__popcll(mk & ((1ull << lane) - 1ull));
                if (b0 < R.cap && c0 + 4u <= R.cap) {
                    ch = (int)c0;
                    const float h = 0.25f * d;
                    R.xy[c0] = make_float2(xy.x - h, xy.y - h);
                    R.xy[c0 + 1] = make_float2(xy.x + h, xy.y - h);
                    R.xy[c0 + 2] = make_float2(xy.x - h, xy.y + h);
                    R.xy[c0 + 3] = make_float2(xy.x + h, xy.y + h);
                } else {
                    // no room: this node stays a leaf; slots of its that lie in
                    // the pool become rayless orphans of the next level
                    if (b0 < R.cap)
                        for (unsigned q = 0; q < 4u; ++q)
                            if (c0 + q < R.cap) {
                                R.xy[c0 + q] = make_float2(RT_REF_DEAD, RT_REF_DEAD);
                                R.gw[c0 + q] = 0.f;
                            }
                    atomicAdd(&R.ctl[RT_REF_UNSPLIT], 1u);
                }
            }
        }
        if (first) R.child[i] = ch;
    }
    for (int off = 32; off > 0; off >>= 1) nrays += __shfl_down(nrays, off);
    if (lane == 0 && nrays) atomicAdd(&R.ctl[RT_REF_RAYS], nrays);
    count_crossings(C.icount, nseg);
}

// level L + 1 ends where the slots handed out so far end
__global__ void k_ref_close(RefArgs R, int L) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        const unsigned c = R.ctl[0];
        R.ctl[3 + L] = c < R.cap ? c : R.cap;
    }
}

__global__ void __launch_bounds__(256) k_ref_combine(RefArgs R, int L) {
    const unsigned start = R.ctl[1 + L], end = R.ctl[2 + L];
    for (unsigned i = start + blockIdx.x * blockDim.x + threadIdx.x; i < end;
         i += gridDim.x * blockDim.x) {
        const int c = R.child[i];
        if (c >= 0) R.val[i] = 0.25f * (((R.val[c] + R.val[c + 1]) + R.val[c + 2]) + R.val[c + 3]);
    }
}

__global__ void __launch_bounds__(256) k_ref_out(CamParams C, RefArgs R, float *img) {
    const int pix = blockIdx.x * blockDim.x + threadIdx.x;
    if (pix >= C.nx * C.ny) return;
    const int j = pix / C.nx, k = pix - j * C.nx;
    float acc = 0.f;
    for (int sub = 0; sub < R.ns2; ++sub) acc += R.val[pixel_node0(C, R.ns2, j, k, sub)];
    img[pix] = acc / (float)R.ns2;
}

__global__ void __launch_bounds__(256) k_ref_gw0(CamParams C, RefArgs R, const float *dimg) {
    const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= R.n0) return;
    int j, k, a, b;
    R.gw[i] = node0_pixel(C, R.ns2, i, j, k, a, b) ? dimg[j * C.nx + k] / (float)R.ns2 : 0.f;
}

__global__ void __launch_bounds__(256) k_ref_down(RefArgs R, int L) {
    const unsigned start = R.ctl[1 + L], end = R.ctl[2 + L];
    for (unsigned i = start + blockIdx.x * blockDim.x + threadIdx.x; i < end;
         i += gridDim.x * blockDim.x) {
        const int c = R.child[i];
        if (c >= 0) {
            const float g = 0.25f * R.gw[i];
            R.gw[c] = g;
            R.gw[c + 1] = g;
            R.gw[c + 2] = g;
            R.gw[c + 3] = g;
        }
    }
}

// the leaves' reverse sweeps; each block gathers a chunk of leaves' cell
// gradients in its LDS table before the global atomics, as k_image_adj does
__global__ void __launch_bounds__(256) k_ref_adj(CamParams C, RefArgs R, double *g_alpha,
                                                 double *g_src) {
    extern __shared__ u64 adj_lds[];
    const unsigned H = 1u << C.hbits;
    u64 *ga = adj_lds, *gs = adj_lds + H;
    int *key = (int *)(adj_lds + 2 * H);
    const unsigned n = R.ctl[0] < R.cap ? R.ctl[0] : R.cap;
    uint32_t nseg = 0;
    const int LN = ref_lanes(n - R.n0 + R.nray0), l = (int)(threadIdx.x & (unsigned)(LN - 1));
    const unsigned per = blockDim.x / (unsigned)LN;
    for (unsigned base = blockIdx.x * per; base < n; base += gridDim.x * per) {
        for (unsigned t = threadIdx.x; t < H; t += blockDim.x) {
            key[t] = -1;
            ga[t] = 0ull;
            gs[t] = 0ull;
        }
        __syncthreads();
        const unsigned i = base + threadIdx.x / (unsigned)LN;
        float g = 0.f;
        float2 xy = make_float2(0.f, 0.f);
        if (i < n && R.child[i] < 0) {
            xy = R.xy[i];
            g = xy.x < 0.5f * RT_REF_DEAD ? R.gw[i] : 0.f;
        }
        adjoint_ray(C, xy.x, xy.y, xy.x, xy.y, g, l, LN, key, ga, gs, g_alpha, g_src, nseg);
        __syncthreads();
        adj_flush(key, ga, gs, H, g_alpha, g_src);
        __syncthreads();
    }
    count_crossings(C.icount ? C.icount + 1 : nullptr, nseg);
}

// point-source fluxes (erg/s/cm^2/Hz/sr over one pixel) passed by value
struct StarArg {
    float f[RT_MAX_STAR];
};

// Point stars: one block per star.  The star's pixel gets F e^-tau, tau along
// the ray from the star to the observer.  A star at the origin (pdspy's
// default) sees the grid along a radial ray: it stays in one (theta, phi) cell
// column and crosses every shell over its full width, so tau is a sum over the
// shells that the block's lanes share; any other star walks its ray cell by
// cell on one lane.  For the adjoint (img NULL) each cell on the ray gets
// -dimg F e^-tau l in g_alpha.
__global__ void k_stars(CamParams C, int nstar, const float *spos, StarArg sflux, float *img,
                        const float *dimg, double *g_alpha) {
    const int s = blockIdx.x;
    if (s >= nstar) return;
    const int lane = threadIdx.x;
    float qx = spos[3 * s], qy = spos[3 * s + 1], qz = spos[3 * s + 2];
    const float exx = (float)C.ex[0], exy = (float)C.ex[1], exz = (float)C.ex[2];
    const float eyx = (float)C.ey[0], eyy = (float)C.ey[1], eyz = (float)C.ey[2];
    const float cpa = (float)C.cpa, spa = (float)C.spa;
    float xp = qx * exx + qy * exy + qz * exz;
    float yp = qx * eyx + qy * eyy + qz * eyz;
    float X = xp * cpa - yp * spa;
    float Y = xp * spa + yp * cpa;
    int k = (int)floorf(X / C.pixf + 0.5f) + C.nx / 2;
    int j = (int)floorf(Y / C.pixf + 0.5f) + C.ny / 2;
    if (k < 0 || k >= C.nx || j < 0 || j >= C.ny) return;
    const DevGrid &g = C.g;
    if (qx == 0.f && qy == 0.f && qz == 0.f) {
        // radial ray: the (theta, phi) column of the direction
        Pos p;
        const float rm = 0.5f * (g.rw[0] + g.rw[1]);
        p.x = rm * C.n[0];
        p.y = rm * C.n[1];
        p.z = rm * C.n[2];
        p.dx = C.n[0];
        p.dy = C.n[1];
        p.dz = C.n[2];
        locate(g, p);
        const size_t col = (size_t)g.nr * (p.it + (size_t)g.nt * p.ip);
        float part = 0.f;
        for (int ir = lane; ir < g.nr; ir += blockDim.x)
            part += C.alpha[col + ir] * (g.rw[ir + 1] - g.rw[ir]);
        for (int off = 32; off > 0; off >>= 1) part += __shfl_xor(part, off);
        const float Is = sflux.f[s] * __expf(-part);
        if (img) {
            if (lane == 0) atomicAdd(&img[j * C.nx + k], Is);
            return;
        }
        const float gI = dimg[j * C.nx + k];
        if (gI == 0.f) return;
        const double qa = C.qs[0];
        for (int ir = lane; ir < g.nr; ir += blockDim.x)
            atomicAdd((u64 *)&g_alpha[col + ir],
                      (u64)__double2ll_rn((double)(-gI * Is * (g.rw[ir + 1] - g.rw[ir])) * qa));
        return;
    }
    if (lane != 0) return;
    Pos p;
    p.x = qx;
    p.y = qy;
    p.z = qz;
    p.dx = C.n[0];
    p.dy = C.n[1];
    p.dz = C.n[2];
    locate(g, p);
    float tau = 0.f;
    Pos p0 = p;
    uint32_t nzero = 0;
    for (int guard = 0; guard < (1 << 24) && p.ir < g.nr; ++guard) {
        int kind;
        float tw = next_wall<1>(g, p, kind);
        const float rcell = g.rw[p.ir + 1];
        if (p.ir >= 0) tau += C.alpha[cell_index(g, p)] * tw;
        if (cross_wall(g, p, tw, kind)) break;
        unstick(g, p, tw, rcell, nzero);
    }
    float Is = sflux.f[s] * __expf(-tau);
    if (img) {
        atomicAdd(&img[j * C.nx + k], Is);
        return;
    }
    float gI = dimg[j * C.nx + k];
    if (gI == 0.f) return;
    p = p0;
    nzero = 0;
    for (int guard = 0; guard < (1 << 24) && p.ir < g.nr; ++guard) {
        int kind;
        float tw = next_wall<1>(g, p, kind);
        const float rcell = g.rw[p.ir + 1];
        if (p.ir >= 0)
            atomicAdd((u64 *)&g_alpha[cell_index(g, p)],
                      (u64)__double2ll_rn((double)(-gI * Is * tw) * C.qs[0]));
        if (cross_wall(g, p, tw, kind)) break;
        unstick(g, p, tw, rcell, nzero);
    }
}

struct KapArg {
    float k[RT_MAX_SPEC];   // absorption opacity at the camera wavelength
    float ks[RT_MAX_SPEC];  // scattering opacity (0 without a scattering source)
};

// alpha (per au) and the source function per cell: B_nu(T), or with a
// scattering source J (isotropic) (rho kabs B + rho ksca J) / (rho kext)
__global__ void k_cam_prep(const float *rho, int S, int ncell, KapArg kap, float lenu, const float *T,
                           float pre, float hnu_k, int mode, const float *J, float *alpha,
                           float *src) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    float aa = 0.f, as = 0.f;
    for (int s = 0; s < S; ++s) {
        const float r = rho[(size_t)s * ncell + c];
        aa = fmaf(r, kap.k[s], aa);
        as = fmaf(r, kap.ks[s], as);
    }
    const float a = aa + as;
    alpha[c] = a * lenu;
    float S_ = 0.f;
    if (mode == 0) {
        const float B = planck_f(pre, hnu_k, T[c]);
        S_ = J ? (a > 0.f ? (aa * B + as * J[c]) / a : 0.f) : B;
    }
    src[c] = S_;
}

// chain rule to log rho_s and T.  With a scattering source (J held fixed):
// d alpha / d log rho_s = rho_s kext_s, dS / d log rho_s = rho_s (kabs_s B +
// ksca_s J - S kext_s) / (rho kext), dS / dT = (rho kabs / rho kext) dB/dT.
__global__ void k_cam_post(const double *g_alpha, const double *g_src, const double *qs,
                           const float *rho, int S, int ncell, KapArg kap, float lenu,
                           const float *T, float pre, float hnu_k, const float *J,
                           const float *src, float *g_logrho, float *g_T) {
    int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= ncell) return;
    // the fixed-point sums back to FP64
    const double qa = qs[0], qsrc = qs[1];
    const double ga = qa > 0.0 ? (double)((const long long *)g_alpha)[c] / qa : 0.0;
    const double gsv = qsrc > 0.0 ? (double)((const long long *)g_src)[c] / qsrc : 0.0;
    if (!J) {
        for (int s = 0; s < S; ++s)
            g_logrho[(size_t)s * ncell + c] =
                (float)(ga * (double)rho[(size_t)s * ncell + c] * (double)kap.k[s] * (double)lenu);
        g_T[c] = (float)(gsv * (double)dplanck_f(pre, hnu_k, T[c]));
        return;
    }
    const double gs = gsv;
    double aa = 0.0, a = 0.0;
    for (int s = 0; s < S; ++s) {
        const double r = rho[(size_t)s * ncell + c];
        aa += r * (double)kap.k[s];
        a += r * ((double)kap.k[s] + (double)kap.ks[s]);
    }
    const double B = planck_f(pre, hnu_k, T[c]), Jc = J[c], Sc = src[c];
    for (int s = 0; s < S; ++s) {
        const double r = rho[(size_t)s * ncell + c];
        const double ke = (double)kap.k[s] + (double)kap.ks[s];
        const double dS = a > 0.0 ? r * ((double)kap.k[s] * B + (double)kap.ks[s] * Jc - Sc * ke) / a
                                  : 0.0;
        g_logrho[(size_t)s * ncell + c] = (float)(ga * r * ke * (double)lenu + gs * dS);
    }
    g_T[c] = (float)(gs * (a > 0.0 ? aa / a : 0.0) * (double)dplanck_f(pre, hnu_k, T[c]));
}

__global__ void k_zero_f64(double *p, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// Units of the adjoint's fixed-point sums, from bounds that hold whatever rays
// an image traces.  The cotangents of all rays sum to at most ||dimg||_1 (the
// rays of a pixel share its dL/dI, sub-pixels a quarter of their parent's).  A
// contribution to dL/dalpha_c is g dI/d(dtau) l with |dI/d(dtau)| <= S_max
// (the largest source: I and every emission term lie in [0, S_max]) and
// l <= 2 R_out; a star adds g F l with F its pixel flux.  A ray crosses a cell
// at most 4 times.  So |sum_c| <= 8 R_out max(S_max, F) (1 + nstar) ||dimg||_1
// for alpha and 4 ||dimg||_1 for S, and units of 2^-61 of those bounds keep
// every partial sum below 2^61.  One block; the reductions run in a fixed
// order, so the units (and with them the gradient) are bit-reproducible.
// 1024 lanes with eight loads in flight each: 69 us with 256 lanes, one load at a
// time, at 256 x 256 pixels, 9.5 us now.
#define ADJ_SC 1024
__global__ void __launch_bounds__(ADJ_SC) k_adj_scale(const float *dimg, int npix, const float *src,
                                                      int ncell, float fstar, int nstar,
                                                      float rout, double *qs) {
    __shared__ double s_l1[ADJ_SC];
    __shared__ float s_max[ADJ_SC];
    const int t = threadIdx.x;
    double l1 = 0.0;
    float smax = fstar;
    for (int i = t; i < npix; i += 8 * ADJ_SC) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = dimg[min(i + e * ADJ_SC, npix - 1)];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            if (i + e * ADJ_SC < npix) l1 += fabs((double)x[e]);
    }
    for (int i = t; i < ncell; i += 8 * ADJ_SC) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = src[min(i + e * ADJ_SC, ncell - 1)];
#pragma unroll
        for (int e = 0; e < 8; ++e) smax = fmaxf(smax, x[e]);
    }
    s_l1[t] = l1;
    s_max[t] = smax;
    __syncthreads();
    for (int h = ADJ_SC / 2; h > 0; h >>= 1) {
        if (t < h) {
            s_l1[t] += s_l1[t + h];
            s_max[t] = fmaxf(s_max[t], s_max[t + h]);
        }
        __syncthreads();
    }
    if (t == 0) {
        const double two61 = 2305843009213693952.0;
        const double ba = 8.0 * (double)rout * (double)s_max[0] * (1.0 + nstar) * s_l1[0];
        const double bs = 4.0 * s_l1[0];
        qs[0] = ba > 0.0 ? two61 / ba : 0.0;
        qs[1] = bs > 0.0 ? two61 / bs : 0.0;
    }
}

static inline unsigned nblk(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

// opacity at the camera wavelength: log-log interpolation of the model's table
// (power-law extrapolation beyond the ends)
static double kappa_at(const rt_model *m, const std::vector<double> &tab, int s, double lam);

double kappa_at_lambda(const rt_model *m, const std::vector<double> &tab, int s, double lam) {
    return kappa_at(m, tab, s, lam);
}

static double kappa_at(const rt_model *m, const std::vector<double> &tab, int s, double lam) {
    const int nl = m->nlam;
    const double *k = &tab[(size_t)s * nl];
    if (nl == 1) return k[0];
    int i = 0;
    if (lam <= m->lam[0])
        i = 0;
    else if (lam >= m->lam[nl - 1])
        i = nl - 2;
    else
        while (i < nl - 2 && m->lam[i + 1] < lam) ++i;
    double l0 = std::log(m->lam[i]), l1 = std::log(m->lam[i + 1]);
    if (!(k[i] > 0) || !(k[i + 1] > 0)) {
        double w = (lam - m->lam[i]) / (m->lam[i + 1] - m->lam[i]);
        return k[i] + w * (k[i + 1] - k[i]);
    }
    double w = (std::log(lam) - l0) / (l1 - l0);
    return std::exp(std::log(k[i]) + w * (std::log(k[i + 1]) - std::log(k[i])));
}

// per-cell scratch of the camera kernels (allocated once per model) and the
// cells' sizes for the sub-pixeling: the least of dr, r_c dtheta and (with phi
// cells) r_c sin(theta_c) dphi at the cell centre, in au
int image_buffers(rt_model *m) {
    rt_ctx *ctx = m->ctx;
    size_t nc = (size_t)m->ncell;
    if (!m->d_alpha) {
        HIPCHK(ctx, hipMalloc(&m->d_alpha, nc * sizeof(float)));
        HIPCHK(ctx, hipMalloc(&m->d_src, nc * sizeof(float)));
        HIPCHK(ctx, hipMalloc(&m->d_galpha, nc * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&m->d_gsrc, nc * sizeof(double)));
        HIPCHK(ctx, hipMalloc(&m->d_qscale, 2 * sizeof(double)));
    }
    if (!m->d_csize) {
        std::vector<float> cs(nc);
        for (int ip = 0; ip < m->np; ++ip)
            for (int it = 0; it < m->nt; ++it)
                for (int ir = 0; ir < m->nr; ++ir) {
                    const double rc = 0.5 * (m->rw[ir] + m->rw[ir + 1]);
                    double l = m->rw[ir + 1] - m->rw[ir];
                    l = std::min(l, rc * (m->tw[it + 1] - m->tw[it]));
                    if (m->np > 1)
                        l = std::min(l, rc * std::sin(0.5 * (m->tw[it] + m->tw[it + 1])) *
                                            (m->pw[ip + 1] - m->pw[ip]));
                    cs[(size_t)ir + (size_t)m->nr * (it + (size_t)m->nt * ip)] =
                        (float)(l / RT_LEN_UNIT);
                }
        HIPCHK(ctx, hipMalloc(&m->d_csize, nc * sizeof(float)));
        HIPCHK(ctx, hipMemcpy(m->d_csize, cs.data(), nc * sizeof(float), hipMemcpyHostToDevice));
    }
    return RT_OK;
}

int refine_reserve(rt_ctx *ctx, size_t n) {
    RefinePool &P = ctx->ref;
    if (n > ((size_t)1 << 30)) return set_err(ctx, RT_E_LIMIT, "sub-pixel pool of %zu nodes > 2^30", n);
    if (P.cap >= n && P.ctl) return RT_OK;
    HIPCHK(ctx, hipStreamSynchronize(ctx->stream));
    void *old[] = {P.xy, P.val, P.child, P.gw};
    for (void *q : old)
        if (q) (void)hipFree(q);
    P.xy = nullptr;
    P.val = nullptr;
    P.child = nullptr;
    P.gw = nullptr;
    P.cap = 0;
    if (hipMalloc(&P.xy, n * sizeof(float2)) != hipSuccess ||
        hipMalloc(&P.val, n * sizeof(float)) != hipSuccess ||
        hipMalloc(&P.child, n * sizeof(int)) != hipSuccess ||
        hipMalloc(&P.gw, n * sizeof(float)) != hipSuccess)
        return set_err(ctx, RT_E_NOMEM, "sub-pixel pool of %zu nodes", n);
    if (!P.ctl) {
        HIPCHK(ctx, hipMalloc(&P.ctl, RT_REF_NCTL * sizeof(unsigned)));
        std::vector<unsigned> z(RT_REF_NCTL, 0u);
        HIPCHK(ctx, hipMemcpy(P.ctl, z.data(), RT_REF_NCTL * sizeof(unsigned), hipMemcpyHostToDevice));
    }
    P.cap = n;
    return RT_OK;
}

static int setup_camera(rt_model *m, const rt_camera *cam, CamParams &C, KapArg &kap, float &pre,
                        float &hnu_k) {
    rt_ctx *ctx = m->ctx;
    if (!cam || cam->nx < 1 || cam->ny < 1 || !(cam->pix_cm > 0) || !(cam->lam_um > 0))
        return set_err(ctx, RT_E_ARG, "invalid camera");
    if (cam->mode != 0 && cam->mode != 1) return set_err(ctx, RT_E_ARG, "camera mode must be 0 or 1");
    const double d2r = M_PI / 180.0;
    double i = cam->incl_deg * d2r, ph = cam->phi_deg * d2r, pa = cam->posang_deg * d2r;
    double n[3] = {std::sin(i) * std::sin(ph), -std::sin(i) * std::cos(ph), std::cos(i)};
    double ex[3] = {std::cos(ph), std::sin(ph), 0.0};
    double ey[3] = {n[1] * ex[2] - n[2] * ex[1], n[2] * ex[0] - n[0] * ex[2], n[0] * ex[1] - n[1] * ex[0]};
    C.g = dev_grid(m);
    C.icount = ctx->d_icount;
    for (int a = 0; a < 3; ++a) {
        C.n[a] = (float)n[a];
        C.nd[a] = n[a];
        C.ex[a] = ex[a];
        C.ey[a] = ey[a];
    }
    C.cpa = std::cos(pa);
    C.spa = std::sin(pa);
    C.pix = cam->pix_cm / RT_LEN_UNIT;
    C.pixf = (float)C.pix;
    C.nx = cam->nx;
    C.ny = cam->ny;
    C.nsub = cam->nsub > 0 ? cam->nsub : 1;
    C.mode = cam->mode;
    // ray tile: neighbouring rays run in tile_w x tile_h pixels (default 8 x 8; 64
    // wide if only the height is given).  Sub-pixelled images keep every tile's pixels
    // in their node pool, which is as large as its caller made it under capture: theirs
    // is 64 x 1 where that takes fewer (64 x 1 pixels: 64 nodes, 512 with 8 x 8 tiles)
    C.tw = cam->tile_w > 0 ? cam->tile_w : (cam->tile_h > 0 ? 64 : 8);
    if (cam->tile_w <= 0 && cam->tile_h <= 0 && cam->nrefine > 0) {
        auto up = [](int n, int t) { return (size_t)((n + t - 1) / t) * t; };
        if (up(C.nx, 64) * C.ny < up(C.nx, 8) * up(C.ny, 8)) C.tw = 64;
    }
    C.th = cam->tile_h > 0 ? cam->tile_h : 64 / C.tw;
    if (C.th < 1) C.th = 1;
    if (C.tw * C.th > 256 || (C.tw * C.th) % 64)
        return set_err(ctx, RT_E_ARG, "ray tile %d x %d: need a multiple of 64 pixels, at most 256",
                       C.tw, C.th);
    C.ntx = (C.nx + C.tw - 1) / C.tw;
    C.nty = (C.ny + C.th - 1) / C.th;
    C.hbits = 11;
    C.lanes = ref_lanes((unsigned)std::min<size_t>((size_t)C.nx * C.ny, 1u << 30));
    C.tau_stop = (float)(cam->tau_stop > 0 ? cam->tau_stop : 40.0);
    for (int s = 0; s < RT_MAX_SPEC; ++s) {
        kap.k[s] = s < m->nspec ? (float)kappa_at(m, m->kabs, s, cam->lam_um) : 0.f;
        kap.ks[s] = (s < m->nspec && cam->d_jscat) ? (float)kappa_at(m, m->ksca, s, cam->lam_um)
                                                   : 0.f;
    }
    double nu = 2.99792458e10 / (cam->lam_um * 1e-4);
    pre = (float)(2.0 * 6.6260755e-27 * nu * nu * nu / (2.99792458e10 * 2.99792458e10));
    hnu_k = (float)(6.6260755e-27 * nu / 1.380658e-16);
    int rc = image_buffers(m);
    if (rc) return rc;
    C.alpha = m->d_alpha;
    C.src = m->d_src;
    C.csize = m->d_csize;
    return 0;
}

static bool stream_capturing(hipStream_t sm) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return hipStreamIsCapturing(sm, &st) == hipSuccess && st == hipStreamCaptureStatusActive;
}

// The sub-pixelled image (d_img) or, with d_dimg, the gradients w.r.t. the
// per-cell alpha and S accumulated into m->d_galpha / m->d_gsrc.  Outside a
// graph capture a pool too small for the refinement is grown and the image
// traced again; inside one the pool must have been reserved (rt_refine_reserve)
// and a sub-pixel without room stays a leaf (counted for rt_refine_stats).
static int refine_run(rt_model *m, const rt_camera *cam, CamParams C, float *d_img,
                      const float *d_dimg) {
    rt_ctx *ctx = m->ctx;
    hipStream_t sm = ctx->stream;
    const int nref = std::min(cam->nrefine, RT_MAX_REFINE);
    const int ns2 = C.nsub * C.nsub;
    const unsigned ntiles = (unsigned)(C.ntx * C.nty);
    const size_t n0 = (size_t)ntiles * (size_t)(C.tw * C.th) * (size_t)ns2;
    const bool capturing = stream_capturing(sm);
    // a fresh pool starts at 2^21 nodes (40 MB); a reserved one is used as
    // it is while it holds the pixels' rays twice
    size_t want = ctx->ref.cap ? std::max(ctx->ref.cap, 2 * n0)
                               : std::max((size_t)1 << 21, 8 * n0);
    if (capturing) {
        if (ctx->ref.cap < 2 * n0)
            return set_err(ctx, RT_E_ARG, "sub-pixel pool (%zu nodes) too small to capture an image "
                                          "of %zu rays: reserve it first", ctx->ref.cap, n0);
        want = ctx->ref.cap;
    }
    const unsigned gblk = (unsigned)(ctx->n_cu > 0 ? 8 * ctx->n_cu : 2048);
    for (;;) {
        int rc = refine_reserve(ctx, want);
        if (rc) return rc;
        RefinePool &P = ctx->ref;
        RefArgs R{P.xy, P.val, P.child, P.gw, P.ctl, (unsigned)P.cap,
                  (float)(cam->refine_crit > 0 ? cam->refine_crit : 1.0), nref, C.pixf / C.nsub,
                  (unsigned)n0, (unsigned)((size_t)C.nx * C.ny * ns2), ns2};
        hipLaunchKernelGGL(k_ref_init, dim3(nblk(n0, 256)), dim3(256), 0, sm, C, R);
        for (int L = 0; L <= nref; ++L) {
            hipLaunchKernelGGL(k_ref_trace, dim3(gblk), dim3(256), 0, sm, C, R, L);
            if (L < nref) hipLaunchKernelGGL(k_ref_close, dim3(1), dim3(64), 0, sm, R, L);
        }
        if (!capturing) {
            unsigned uns = 0;
            HIPCHK(ctx, hipMemcpyAsync(&uns, P.ctl + RT_REF_UNSPLIT, sizeof(uns),
                                       hipMemcpyDeviceToHost, sm));
            HIPCHK(ctx, hipStreamSynchronize(sm));
            if (uns && P.cap < ((size_t)1 << 30)) {
                unsigned z = 0;
                HIPCHK(ctx, hipMemcpy(P.ctl + RT_REF_UNSPLIT, &z, sizeof(z), hipMemcpyHostToDevice));
                want = std::min((size_t)1 << 30, 4 * P.cap);
                continue;  // trace again in a larger pool
            }
        }
        if (!d_dimg) {
            for (int L = nref - 1; L >= 0; --L)
                hipLaunchKernelGGL(k_ref_combine, dim3(gblk), dim3(256), 0, sm, R, L);
            hipLaunchKernelGGL(k_ref_out, dim3(nblk((size_t)C.nx * C.ny, 256)), dim3(256), 0, sm, C,
                               R, d_img);
        } else {
            hipLaunchKernelGGL(k_ref_gw0, dim3(nblk(n0, 256)), dim3(256), 0, sm, C, R, d_dimg);
            for (int L = 0; L < nref; ++L)
                hipLaunchKernelGGL(k_ref_down, dim3(gblk), dim3(256), 0, sm, R, L);
            const CamParams &Ca = C;
            const size_t lds = (size_t)(1u << Ca.hbits) * (2 * sizeof(u64) + sizeof(int));
            hipLaunchKernelGGL(k_ref_adj, dim3(gblk), dim3(256), lds, sm, Ca, R, m->d_galpha,
                               m->d_gsrc);
        }
        HIPCHK(ctx, hipGetLastError());
        return RT_OK;
    }
}

// blocks of k_image / k_image_adj: every pixel of every tile, C.lanes lanes each
static unsigned image_blocks(const CamParams &C) {
    return nblk((size_t)C.ntx * C.nty * (size_t)(C.tw * C.th) * (size_t)C.lanes, IMG_BS);
}

static void star_fluxes(const rt_model *m, const rt_camera *cam, StarArg &fl) {
    double nu = 2.99792458e10 / (cam->lam_um * 1e-4);
    for (int s = 0; s < RT_MAX_STAR; ++s) fl.f[s] = 0.f;
    for (int s = 0; s < m->nstar && s < RT_MAX_STAR; ++s) {
        double R = m->stars[5 * s], T = m->stars[5 * s + 1];
        double x = 6.6260755e-27 * nu / (1.380658e-16 * T);
        double B = 2.0 * 6.6260755e-27 * nu * nu * nu / (2.99792458e10 * 2.99792458e10) / std::expm1(x);
        fl.f[s] = (float)(M_PI * R * R * B / (cam->pix_cm * cam->pix_cm));
    }
}

int image_run(rt_model *m, const rt_camera *cam, const float *d_T, const float *d_rho, float *d_img) {
    rt_ctx *ctx = m->ctx;
    CamParams C{};
    KapArg kap{};
    float pre, hnu_k;
    int rc = setup_camera(m, cam, C, kap, pre, hnu_k);
    if (rc) return rc;
    if (!d_T && cam->mode == 0) return set_err(ctx, RT_E_ARG, "temperature pointer is NULL");
    const float *rho = d_rho ? d_rho : m->d_rho;
    hipStream_t sm = ctx->stream;
    hipLaunchKernelGGL(k_cam_prep, dim3(nblk(m->ncell, 256)), dim3(256), 0, sm, rho, m->nspec,
                       m->ncell, kap, (float)RT_LEN_UNIT, d_T, pre, hnu_k, cam->mode,
                       cam->d_jscat, m->d_alpha, m->d_src);
    if (cam->nrefine > 0) {
        rc = refine_run(m, cam, C, d_img, nullptr);
        if (rc) return rc;
    } else {
        hipLaunchKernelGGL(k_image, dim3(image_blocks(C)), dim3(IMG_BS), 0, sm, C, d_img);
    }
    if (cam->incl_star && cam->mode == 0 && m->nstar > 0) {
        StarArg fl;
        star_fluxes(m, cam, fl);
        hipLaunchKernelGGL(k_stars, dim3(m->nstar), dim3(64), 0, sm, C, m->nstar, m->d_spos, fl, d_img,
                           (const float *)nullptr, (double *)nullptr);
    }
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}

int image_adjoint_run(rt_model *m, const rt_camera *cam, const float *d_T, const float *d_rho,
                      const float *d_dimg, float *d_g_logrho, float *d_g_T) {
    rt_ctx *ctx = m->ctx;
    if (cam && cam->mode != 0) return set_err(ctx, RT_E_ARG, "adjoint needs mode 0 (intensity)");
    CamParams C{};
    KapArg kap{};
    float pre, hnu_k;
    int rc = setup_camera(m, cam, C, kap, pre, hnu_k);
    if (rc) return rc;
    if (!d_T || !d_dimg || !d_g_logrho || !d_g_T) return set_err(ctx, RT_E_ARG, "NULL pointer");
    const float *rho = d_rho ? d_rho : m->d_rho;
    hipStream_t sm = ctx->stream;
    size_t nc = (size_t)m->ncell;
    hipLaunchKernelGGL(k_cam_prep, dim3(nblk(nc, 256)), dim3(256), 0, sm, rho, m->nspec, m->ncell,
                       kap, (float)RT_LEN_UNIT, d_T, pre, hnu_k, 0, cam->d_jscat, m->d_alpha,
                       m->d_src);
    hipLaunchKernelGGL(k_zero_f64, dim3(nblk(nc, 256)), dim3(256), 0, sm, m->d_galpha, nc);
    hipLaunchKernelGGL(k_zero_f64, dim3(nblk(nc, 256)), dim3(256), 0, sm, m->d_gsrc, nc);
    const bool stars = cam->incl_star && m->nstar > 0;
    StarArg fl;
    star_fluxes(m, cam, fl);
    float fmax_star = 0.f;
    for (int s = 0; stars && s < m->nstar && s < RT_MAX_STAR; ++s) fmax_star = std::max(fmax_star, fl.f[s]);
    hipLaunchKernelGGL(k_adj_scale, dim3(1), dim3(ADJ_SC), 0, sm, d_dimg, C.nx * C.ny, m->d_src,
                       m->ncell, fmax_star, stars ? m->nstar : 0,
                       (float)(m->rw[m->nr] / RT_LEN_UNIT), m->d_qscale);
    C.qs = m->d_qscale;
    if (cam->nrefine > 0) {
        rc = refine_run(m, cam, C, nullptr, d_dimg);
        if (rc) return rc;
    } else {
        const size_t adj_lds = (size_t)(1u << C.hbits) * (2 * sizeof(u64) + sizeof(int));
        hipLaunchKernelGGL(k_image_adj, dim3(image_blocks(C)), dim3(IMG_BS), adj_lds, sm, C, d_dimg,
                           m->d_galpha, m->d_gsrc);
    }
    if (stars)
        hipLaunchKernelGGL(k_stars, dim3(m->nstar), dim3(64), 0, sm, C, m->nstar, m->d_spos, fl,
                           (float *)nullptr, d_dimg, m->d_galpha);
    hipLaunchKernelGGL(k_cam_post, dim3(nblk(nc, 256)), dim3(256), 0, sm, m->d_galpha, m->d_gsrc,
                       (const double *)m->d_qscale, rho, m->nspec, m->ncell, kap,
                       (float)RT_LEN_UNIT, d_T, pre, hnu_k, cam->d_jscat, m->d_src, d_g_logrho,
                       d_g_T);
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}
