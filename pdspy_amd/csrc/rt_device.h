// rt_device.h -- device helpers shared by the gfx950 kernels: Philox4x32-10,
// the spherical-grid traversal (FP32 with FP64 re-evaluation of near-tangent
// sphere/cone crossings), Planck functions and wave-level helpers.
//
// Geometry follows the grids pdspy writes for RADMC-3D (radmc3d/write.py:198-244):
// r walls (lengths in au on the device), theta walls in [0, pi/2] with an
// equatorial mirror (the lower half-space folds onto the upper one) or [0, pi],
// phi walls over [0, 2 pi].  Cells are indexed c = ir + nr*(it + nt*ip)
// (r fastest, dust_density.inp order, write.py:259-264).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define RT_INF 3.0e38f

namespace rt {

// ---------------------------------------------------------------- Philox
// Salmon, Moraes, Dror & Shaw, "Parallel random numbers: as easy as 1, 2, 3"
// (SC'11): 10 rounds of the 4x32 bijection, Weyl key schedule.

__device__ __forceinline__ void philox_block(uint32_t c0, uint32_t c1, uint32_t c2,
                                             uint32_t c3, uint32_t k0, uint32_t k1,
                                             uint32_t out[4]) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r > 0) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        // one 64-bit product per pair of halves (v_mad_u64_u32): the high and
        // low words taken separately cost two quarter-rate multiplies each
        const uint64_t m0 = (uint64_t)0xD2511F53u * c0, m1 = (uint64_t)0xCD9E8D57u * c2;
        uint32_t hi0 = (uint32_t)(m0 >> 32), lo0 = (uint32_t)m0;
        uint32_t hi1 = (uint32_t)(m1 >> 32), lo1 = (uint32_t)m1;
        uint32_t n0 = hi1 ^ c1 ^ k0, n2 = hi0 ^ c3 ^ k1;
        c0 = n0;
        c1 = lo1;
        c2 = n2;
        c3 = lo0;
    }
    out[0] = c0;
    out[1] = c1;
    out[2] = c2;
    out[3] = c3;
}

// uniform in (0,1) from the top 24 bits of a word, exact in FP32
__device__ __forceinline__ float u24(uint32_t x) {
    return ((float)(x >> 8) + 0.5f) * (1.0f / 16777216.0f);
}

// The random numbers of a packet come in events: event k (k = 0 at emission,
// then one per interaction and one per modified-random-walk step) uses the 8
// uniforms of the blocks with counter (k, pid_lo, pid_hi, 0) and
// (k, pid_lo, pid_hi, 1) under key = seed.  A fixed number of Philox blocks per
// event keeps the wavefront from re-running the generator at every draw.
__device__ __forceinline__ void rng8(uint64_t seed, uint64_t pid, uint32_t k, float u[8]) {
    uint32_t a[4], b[4];
    philox_block(k, (uint32_t)pid, (uint32_t)(pid >> 32), 0u, (uint32_t)seed,
                 (uint32_t)(seed >> 32), a);
    philox_block(k, (uint32_t)pid, (uint32_t)(pid >> 32), 1u, (uint32_t)seed,
                 (uint32_t)(seed >> 32), b);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        u[i] = u24(a[i]);
        u[4 + i] = u24(b[i]);
    }
}

// ---------------------------------------------------------------- grid
struct DevGrid {
    int nr, nt, np, mirror, ncell;
    const float *rw;    // nr+1 radial walls (au)
    const float *rw2;   // their squares
    const double *rwd;  // FP64 walls
    const float *tw;    // nt+1 theta walls
    const float *ct;    // cos of theta walls (ct[nt] = 0 exactly in mirror mode)
    const float *st;    // sin
    const double *ctd;  // FP64 cos/sin for the near-tangent re-evaluation
    const double *std_;
    const float *pw;    // np+1 phi walls
    const float *cp;
    const float *sp;
};

// x a + y b with one rounding of the first product less: which of the two a
// compiler fuses depends on the code around an inlined call, and a packet's
// whole history on the last bit, so the choice is written out.  XF = 1: x a is
// the fused one.  (next_wall's XF is the caller's: the thermal packets take 0,
// the scattering source's 1.)
template <int XF>
__device__ __forceinline__ float sum2(float x, float a, float y, float b) {
    return XF ? fmaf(x, a, y * b) : fmaf(y, b, x * a);
}
template <int XF>
__device__ __forceinline__ double sum2(double x, double a, double y, double b) {
    return XF ? fma(x, a, y * b) : fma(y, b, x * a);
}

enum { W_NONE = 0, W_ROUT, W_RIN, W_TLO, W_THI, W_PLO, W_PHI, W_HOLE };

struct Pos {
    float x, y, z, dx, dy, dz;
    int ir, it, ip, hemi;  // ir = -1: inner hole; ir = nr: outside
};

__device__ __forceinline__ int cell_index(const DevGrid &g, const Pos &p) {
    return p.ir + g.nr * (p.it + g.nt * p.ip);
}

__device__ __forceinline__ int search_walls(const float *w, int n, float v) {
    // i in [0, n-1] with w[i] <= v < w[i+1], clamped
    if (v <= w[0]) return 0;
    if (v >= w[n]) return n - 1;
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (w[mid] <= v)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

template <int XF = 1>
__device__ __forceinline__ void locate_angles(const DevGrid &g, Pos &p) {
    float rho = sqrtf(sum2<XF>(p.x, p.x, p.y, p.y));
    if (g.mirror) {
        p.hemi = (p.z >= 0.f) ? 1 : -1;
        p.it = search_walls(g.tw, g.nt, atan2f(rho, fabsf(p.z)));
    } else {
        p.hemi = 1;
        p.it = search_walls(g.tw, g.nt, atan2f(rho, p.z));
    }
    if (g.np > 1) {
        float ph = atan2f(p.y, p.x);
        if (ph < 0.f) ph += 6.28318530718f;
        p.ip = search_walls(g.pw, g.np, ph);
    } else {
        p.ip = 0;
    }
}

// Cell of the position.  Every index is written once at the end (separate
// early returns writing different fields would keep Pos out of registers).
template <int XF = 1>
__device__ __forceinline__ void locate(const DevGrid &g, Pos &p) {
    float rr = fmaf(p.z, p.z, sum2<XF>(p.x, p.x, p.y, p.y));
    const bool hole = rr < g.rw2[0], outside = !hole && rr >= g.rw2[g.nr];
    int ir;
    Pos q = p;
    q.it = 0;
    q.ip = 0;
    q.hemi = (g.mirror && p.z < 0.f) ? -1 : 1;
    if (hole) {
        ir = -1;
    } else if (outside) {
        ir = g.nr;
    } else {
        ir = search_walls(g.rw, g.nr, sqrtf(rr));
        locate_angles<XF>(g, q);
    }
    p.ir = ir;
    p.it = q.it;
    p.ip = q.ip;
    p.hemi = q.hemi;
}

__device__ __forceinline__ float sph_out(float b, float rr, float R2) {
    float c = rr - R2;
    float D = fmaxf(fmaf(b, b, -c), 0.f);
    float sq = sqrtf(D);
    float t = (b <= 0.f) ? (sq - b) : (-c / (b + sq));
    return fmaxf(t, 0.f);
}

// inner sphere, moving inwards (b < 0), where the discriminant is small against
// b^2: FP64 from the FP32 position, so that hit or miss is decided consistently
template <int XF>
__device__ __forceinline__ float sph_in_d(const Pos &p, double Rd) {
    const double xd = p.x, yd = p.y, zd = p.z;
    double bd = fma(zd, (double)p.dz, sum2<XF>(xd, (double)p.dx, yd, (double)p.dy));
    double rrd = fma(zd, zd, sum2<XF>(xd, xd, yd, yd));
    double cd = fma(-Rd, Rd, rrd);
    double Dd = fma(bd, bd, -cd);
    if (Dd < 0.0) return RT_INF;
    double t = cd / (sqrt(Dd) - bd);
    return t > 0.0 ? (float)t : 0.f;
}

// Exit through the cone at polar angle th (folded frame): f = rho^2 cos^2 -
// z^2 sin^2; root with f' > 0 is (-B+sqrt(D))/A, with f' < 0 is (-B-sqrt(D))/A;
// on the nappe sign(z) = sign(cos th) the sign of dtheta/dt is
// sign(f') * sign(cos th).  req = -1 leaves towards smaller theta, +1 larger.
// A ray whose cell index is consistent with its position always meets its
// exit root ahead of it.  When a radial and a theta crossing lie within FP32
// resolution of each other, the ray can take the radial one first and stand a
// hair past the cone while the index still names the cell before it: the exit
// root is then just behind the position (the ray moving through the wall in
// the req direction), or, near tangency, missing while f already has the far
// side's sign.  The wall is then crossed at once (t = 0); rejecting it would
// leave the theta index behind for the rest of the ray.
__device__ __forceinline__ float cone_root(double A, double B, double C, double D,
                                           int want_plus) {
    double sq = sqrt(D);
    double t;
    if (want_plus)
        t = (B < 0) ? (-B + sq) / A : -C / (B + sq);
    else
        t = (B > 0) ? -(B + sq) / A : C / (-B + sq);
    return (float)t;
}

// what a ray and all cones have in common, in the folded frame
struct ConeRay {
    float z, dz, rr;
    float dd, xd, rho2;     // dx^2 + dy^2, x dx + y dy, x^2 + y^2
    float dz2, zdz, z2;
};

// the same in FP64, for the cone of cos/sin cthd, sthd (near tangency)
template <int XF>
__device__ __forceinline__ float cone_hit_d(float x, float y, float z, float dx, float dy, float dz,
                                            double cthd, double sthd, float sreq) {
    double c2d = cthd * cthd, s2d = sthd * sthd;
    const double xd = x, yd = y, zd = z, dxd = dx, dyd = dy, dzd = dz;
    double Ad = fma(sum2<XF>(dxd, dxd, dyd, dyd), c2d, -(dzd * dzd * s2d));
    double Bd = fma(sum2<XF>(xd, dxd, yd, dyd), c2d, -(zd * dzd * s2d));
    double Cd = fma(sum2<XF>(xd, xd, yd, yd), c2d, -(zd * zd * s2d));
    double Dd = fma(Bd, Bd, -(Ad * Cd));
    // no crossing: f keeps the sign of C along the whole line
    if (Dd < 0.0) return Cd * sreq > 0.0 ? 0.f : RT_INF;
    return cone_root(Ad, Bd, Cd, Dd, sreq > 0.f);
}

// Without branches but for the near-tangent one: a wave's lanes differ in
// every one of these cases, so each branch was taken by some of them, and a
// branch on a lone lane costs as much as the ten instructions it skips.
template <int XF>
__device__ __forceinline__ float cone_hit(const Pos &p, const ConeRay &q, float cth, float sth,
                                          const double *cthd, const double *sthd, int req,
                                          bool there) {
    const float c2 = cth * cth, s2 = sth * sth;
    const float A = fmaf(q.dd, c2, -(q.dz2 * s2));
    const float B = fmaf(q.xd, c2, -(q.zdz * s2));
    const float C = fmaf(q.rho2, c2, -(q.z2 * s2));
    // a ray lying in the cone (direction and position on it, as a radial ray
    // through the origin along a wall angle): it never leaves through it
    const bool lies = fabsf(A) <= 1e-6f && fabsf(C) <= 1e-6f * (q.rho2 + q.z2);
    const float D = fmaf(B, B, -(A * C));
    const float sreq = (float)(cth > 0.f ? req : -req);
    // the root as one quotient: (-B + sq) / A or -C / (B + sq) for the larger,
    // -(B + sq) / A or C / (-B + sq) for the other
    const float sq = sqrtf(D);
    const float s = sreq > 0.f ? B : -B;
    const bool direct = s < 0.f;   // no cancellation in -B +- sq
    const float u = sreq > 0.f ? (direct ? -B + sq : -C) : (direct ? -(B + sq) : C);
    const float v = direct ? A : s + sq;
    float t = u / v;
    // no crossing, clear of rounding (|A| <= 1, |B| <= r, |C| <= r^2, so D is
    // good to a few ulp of r^2): as the FP64 test would find
    const bool clear = D < -1e-5f * q.rr;
    t = clear ? (C * sreq > 0.f ? 0.f : RT_INF) : t;
    if (there && !lies && !clear && D < 1e-4f * B * B)
        t = cone_hit_d<XF>(p.x, p.y, q.z, p.dx, p.dy, q.dz, *cthd, *sthd, sreq);
    t = t >= 0.f ? t : (B * sreq > 0.f ? 0.f : RT_INF);
    const float zh = fmaf(t, q.dz, q.z);
    return !there || lies || !(t < RT_INF) || zh * cth < 0.f ? RT_INF : t;
}

// Exit through the phi half-plane (cos ph, sin ph); a crossing just behind
// the position (the ray already past the wall, moving through it) is taken at
// once, as for the cones.
__device__ __forceinline__ float phi_hit(float x, float y, float dx, float dy, float cph,
                                         float sph, int req) {
    float g0 = fmaf(y, cph, -(x * sph));
    float g1 = fmaf(dy, cph, -(dx * sph));
    const float t = fmaxf(-g0 / g1, 0.f);
    float xh = fmaf(t, dx, x), yh = fmaf(t, dy, y);
    const bool hit = (req < 0 ? g1 < 0.f : g1 > 0.f) && !(fmaf(xh, cph, yh * sph) < 0.f);
    return hit ? t : RT_INF;
}

// distance to the next wall of the current cell and which wall it is.  noin: the
// inner sphere is not met.  EQ: a cone that is a plane but for the rounding of
// pi/2 -- the equator of a grid over [0, pi] -- is taken as the plane (its
// quadratic has a double root).
template <int XF, bool EQ = false>
__device__ __forceinline__ float next_wall(const DevGrid &g, const Pos &p, int &kind,
                                           bool noin = false) {
    const bool in = p.ir >= 0;
    const int i = in ? p.ir : 0, j = p.it;
    // the walls' words first: one wait for all of them
    const float R2o = g.rw2[p.ir + 1], R2i = g.rw2[i];
    const float ctl = g.ct[j], stl = g.st[j], cth = g.ct[j + 1], sth = g.st[j + 1];
    ConeRay q;
    q.dd = sum2<XF>(p.dx, p.dx, p.dy, p.dy);
    q.xd = sum2<XF>(p.x, p.dx, p.y, p.dy);
    q.rho2 = sum2<XF>(p.x, p.x, p.y, p.y);
    const float rr = fmaf(p.z, p.z, q.rho2);
    const float b = fmaf(p.z, p.dz, q.xd);
    q.rr = rr;
    q.z = p.hemi > 0 ? p.z : -p.z;
    q.dz = p.hemi > 0 ? p.dz : -p.dz;
    q.dz2 = __fmul_rn(q.dz, q.dz);
    q.zdz = __fmul_rn(q.z, q.dz);
    q.z2 = __fmul_rn(q.z, q.z);
    // outer sphere (from the inner hole: its wall)
    float tb = sph_out(b, rr, R2o);
    kind = in ? W_ROUT : W_HOLE;
    // inner sphere.  A discriminant below -1e-5 (r^2 + R^2), twenty times its
    // FP32 rounding bound, is a miss without the FP64 check
    {
        const float c = rr - R2i;
        const float D = fmaf(b, b, -c);
        const bool cand = in && !noin && b < 0.f && !(D < -1e-5f * (rr + R2i));
        float t = fmaxf(c / (sqrtf(D) - b), 0.f);
        if (cand && D < 1e-4f * b * b) t = sph_in_d<XF>(p, g.rwd[i]);
        const bool hit = cand && t < tb;
        tb = hit ? t : tb;
        kind = hit ? W_RIN : kind;
    }
    // lower cone; the equatorial plane of a full-sphere grid is left upwards
    // (a crossing behind the position is taken at once)
    {
        const bool plane = !g.mirror && (EQ ? fabsf(ctl) < 1e-6f : ctl == 0.f);
        float t = cone_hit<XF>(p, q, ctl, stl, g.ctd + j, g.std_ + j, -1, in && j > 0 && !plane);
        if (!g.mirror && plane && in && j > 0 && p.dz > 0.f) t = fmaxf(-p.z / p.dz, 0.f);
        const bool hit = t < tb;
        tb = hit ? t : tb;
        kind = hit ? W_TLO : kind;
    }
    // upper cone, or the mirror plane under the last row of cells
    {
        const bool last = j + 1 == g.nt;
        const bool plane = !g.mirror && (EQ ? fabsf(cth) < 1e-6f : cth == 0.f);
        float t = cone_hit<XF>(p, q, cth, sth, g.ctd + j + 1, g.std_ + j + 1, +1,
                               in && !last && !plane);
        const bool fold = g.mirror ? last && q.dz < 0.f : plane && !last && p.dz < 0.f;
        const float tp = fmaxf(-q.z / q.dz, 0.f);
        t = in && fold ? tp : t;
        const bool hit = t < tb;
        tb = hit ? t : tb;
        kind = hit ? W_THI : kind;
    }
    if (g.np > 1) {
        const int k = p.ip;
        float t = phi_hit(p.x, p.y, p.dx, p.dy, g.cp[k], g.sp[k], -1);
        bool hit = in && t < tb;
        tb = hit ? t : tb;
        kind = hit ? W_PLO : kind;
        t = phi_hit(p.x, p.y, p.dx, p.dy, g.cp[k + 1], g.sp[k + 1], +1);
        hit = in && t < tb;
        tb = hit ? t : tb;
        kind = hit ? W_PHI : kind;
    }
    return tb;
}

__device__ __forceinline__ void snap_radius(Pos &p, float R) {
    float r = sqrtf(fmaf(p.z, p.z, sum2<1>(p.x, p.x, p.y, p.y)));
    if (r > 0.f) {
        float f = R / r;
        p.x *= f;
        p.y *= f;
        p.z *= f;
    }
}

// move by t, cross the wall; returns true when the packet leaves the grid.
// The cell indices change by +-1 through selects (no branch writes through a
// pointer into the packet state, which would keep it out of registers).
__device__ __forceinline__ bool cross_wall(const DevGrid &g, Pos &p, float t, int kind) {
    p.x = fmaf(t, p.dx, p.x);
    p.y = fmaf(t, p.dy, p.y);
    p.z = fmaf(t, p.dz, p.z);
    if (kind == W_HOLE) {
        snap_radius(p, g.rw[0]);
        p.ir = 0;
        locate_angles(g, p);
        return false;
    }
    const bool mirror_hit = kind == W_THI && g.mirror && p.it + 1 == g.nt;
    const int dir_r = (kind == W_ROUT ? 1 : 0) - (kind == W_RIN ? 1 : 0);
    const int dir_t = (kind == W_THI && !mirror_hit ? 1 : 0) - (kind == W_TLO ? 1 : 0);
    const int dir_p = (kind == W_PHI ? 1 : 0) - (kind == W_PLO ? 1 : 0);
    p.ir += dir_r;
    if (p.ir >= g.nr) return true;
    // the wall crossed: inner wall of the new cell going out, outer going in
    if (dir_r != 0) snap_radius(p, g.rw[dir_r > 0 ? p.ir : p.ir + 1]);
    p.it += dir_t;
    if (mirror_hit) {
        p.z = 0.f;
        p.hemi = -p.hemi;
    }
    int ip = p.ip + dir_p;
    p.ip = ip < 0 ? g.np - 1 : (ip >= g.np ? 0 : ip);
    return false;
}

// Ping-pong guard.  A ray almost tangent to a sphere or cone can find the wall
// it has just crossed again at a distance below FP32 resolution and bounce
// between two cells without moving.  After 8 consecutive crossings shorter
// than 2^-20 r (r: outer radius of the cell the step started in) the position
// is advanced by 2^-16 r along the ray and its cell is found again from the
// position.  Returns true when it moved the packet.
__device__ __forceinline__ bool unstick(const DevGrid &g, Pos &p, float tw, float rcell,
                                        uint32_t &nzero) {
    if (tw > rcell * 9.5367431640625e-07f) {
        nzero = 0;
        return false;
    }
    if (++nzero < 8u) return false;
    nzero = 0;
    float d = rcell * 1.52587890625e-05f;
    p.x = fmaf(d, p.dx, p.x);
    p.y = fmaf(d, p.dy, p.y);
    p.z = fmaf(d, p.dz, p.z);
    locate<0>(g, p);
    return true;
}

// ---------------------------------------------------------------- physics
// pdspy CGS constants (pdspy/constants/physics.py)
#define RT_H 6.6260755e-27
#define RT_C 2.99792458e10
#define RT_K 1.380658e-16

// isotropic direction: cos(theta) = 2 u1 - 1, azimuth 2 pi u2
__device__ __forceinline__ void iso_dir(float u1, float u2, float &dx, float &dy, float &dz) {
    float mu = 2.f * u1 - 1.f;
    float s, c;
    sincospif(2.f * u2, &s, &c);
    float st = sqrtf(fmaxf(0.f, 1.f - mu * mu));
    dx = st * c;
    dy = st * s;
    dz = mu;
}

// rotate the unit vector (dx,dy,dz) by polar angle (cosine ct) and azimuth
// 2 pi u2 about itself
__device__ __forceinline__ void rotate_dir(float ct, float u2, float &dx, float &dy, float &dz) {
    float sps, cps;
    sincospif(2.f * u2, &sps, &cps);
    float st = sqrtf(fmaxf(0.f, 1.f - ct * ct));
    float ux = dx, uy = dy, uz = dz;
    if (fabsf(uz) > 0.99999f) {
        dx = st * cps;
        dy = st * sps;
        dz = (uz > 0.f ? 1.f : -1.f) * ct;
    } else {
        // (fused as written: which of two products a compiler fuses depends on
        // the code around an inlined call, and a packet's history on the last bit)
        float s = sqrtf(fmaf(-uz, uz, 1.f));
        dx = fmaf(ux, ct, st * fmaf(ux * uz, cps, -(uy * sps)) / s);
        dy = fmaf(uy, ct, st * fmaf(uy * uz, cps, ux * sps) / s);
        dz = fmaf(uz, ct, -(st * cps * s));
    }
    float n = rsqrtf(fmaf(dz, dz, fmaf(dx, dx, dy * dy)));
    dx *= n;
    dy *= n;
    dz *= n;
}

// Henyey-Greenstein scattering about the current direction: cosine from u1,
// azimuth 2 pi u2
__device__ __forceinline__ void hg_dir(float u1, float u2, float g, float &dx, float &dy,
                                       float &dz) {
    float u = u1;
    float ct;
    if (fabsf(g) < 1e-6f) {
        ct = 2.f * u - 1.f;
    } else {
        float f = (1.f - g * g) / (1.f - g + 2.f * g * u);
        ct = (1.f + g * g - f * f) / (2.f * g);
    }
    ct = fminf(1.f, fmaxf(-1.f, ct));
    rotate_dir(ct, u2, dx, dy, dz);
}

// perpendicular distance to the nearest wall of the current cell that bounds
// the medium; the equatorial mirror and the polar axis are not walls.  Cone at
// theta_j: r sin|theta - theta_j| = |rho cos theta_j - z sin theta_j| while
// |theta - theta_j| <= pi/2 (else the axis, r); phi half-plane at phi_k:
// |y cos phi_k - x sin phi_k| while |phi - phi_k| <= pi/2 (else rho).
__device__ __forceinline__ float wall_dist(const DevGrid &g, const Pos &p) {
    float r = sqrtf(fmaf(p.z, p.z, fmaf(p.x, p.x, p.y * p.y)));
    float d = fminf(r - g.rw[p.ir], g.rw[p.ir + 1] - r);
    float rho = sqrtf(fmaf(p.x, p.x, p.y * p.y));
    float zf = g.mirror ? fabsf(p.z) : p.z;
    int j = p.it;
    if (j > 0) {
        float sn = fmaf(rho, g.ct[j], -(zf * g.st[j]));
        float cs = fmaf(zf, g.ct[j], rho * g.st[j]);
        d = fminf(d, cs >= 0.f ? fabsf(sn) : r);
    }
    if (j + 1 < g.nt) {
        float sn = fmaf(rho, g.ct[j + 1], -(zf * g.st[j + 1]));
        float cs = fmaf(zf, g.ct[j + 1], rho * g.st[j + 1]);
        d = fminf(d, cs >= 0.f ? fabsf(sn) : r);
    }
    if (g.np > 1) {
        int k = p.ip;
        float sn = fmaf(p.y, g.cp[k], -(p.x * g.sp[k]));
        float cs = fmaf(p.x, g.cp[k], p.y * g.sp[k]);
        d = fminf(d, cs >= 0.f ? fabsf(sn) : rho);
        sn = fmaf(p.y, g.cp[k + 1], -(p.x * g.sp[k + 1]));
        cs = fmaf(p.x, g.cp[k + 1], p.y * g.sp[k + 1]);
        d = fminf(d, cs >= 0.f ? fabsf(sn) : rho);
    }
    return d;
}

// table value at the fractional temperature-row coordinate x
__device__ __forceinline__ float trow(const float *tab, int ntemp, float x) {
    x = fminf(fmaxf(x, 0.f), (float)(ntemp - 1));
    int lo = min((int)x, ntemp - 2);
    float w = x - (float)lo;
    return fmaf(w, tab[lo + 1] - tab[lo], tab[lo]);
}

// diffusion escape law: y(xi) with P(y) = xi, tabulated on a uniform grid of
// logit(xi) over [-lmax, lmax] (24-bit uniforms stay inside it)
__device__ __forceinline__ float mrw_escape_y(const float *Y, int ny, float lmax, float xi) {
    float L = __logf(xi) - __logf(1.f - xi);
    float f = (L + lmax) * ((float)(ny - 1) / (2.f * lmax));
    f = fminf(fmaxf(f, 0.f), (float)(ny - 1));
    int k = min((int)f, ny - 2);
    float w = f - (float)k;
    return fmaf(w, Y[k + 1] - Y[k], Y[k]);
}

// a[i] for i < 4 without dynamic register indexing
__device__ __forceinline__ float pick4(const float (&a)[4], int i) {
    return i == 0 ? a[0] : i == 1 ? a[1] : i == 2 ? a[2] : a[3];
}

// B_nu(T) in FP32 from h nu/k (pdspy/misc/B_nu.py:4-6); pre = 2 h nu^3 / c^2
__device__ __forceinline__ float planck_f(float pre, float hnu_k, float T) {
    if (!(T > 0.f)) return 0.f;
    float x = hnu_k / T;
    if (x > 80.f) return pre * __expf(-x);
    return pre / expm1f(x);
}

// dB_nu/dT (pdspy/misc/dB_nu.py:4-7 up to sign) = pre * x e^x / (T (e^x-1)^2)
__device__ __forceinline__ float dplanck_f(float pre, float hnu_k, float T) {
    if (!(T > 0.f)) return 0.f;
    float x = hnu_k / T;
    if (x > 80.f) return pre * x * __expf(-x) / T;
    float e = expm1f(x);
    return pre * x * (e + 1.f) / (T * e * e);
}

// ---------------------------------------------------------------- waves
__device__ __forceinline__ int lane_id() { return __lane_id(); }

}  // namespace rt
