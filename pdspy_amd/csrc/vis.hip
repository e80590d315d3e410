// vis.hip -- model visibilities and chi^2 on gfx950.
//
// V(u,v) = sum_jk I[j][k] exp(-2 pi i (u x_k + v y_j)) with x_k = (k - nx/2) dxy,
// y_j = (j - ny/2) dxy, times the phase-centre shift exp(-2 pi i (u dra + v ddec)).
// On the pixel-conjugate grid this is pdspy's imtovis (imaging/imtovis.py:13-24,
// fftshift(fft2(ifftshift(I)))); at arbitrary (u,v) it is the exact sampler
// behind interpolate_model (interferometry/interpolate_model.py:20-27), and the
// gridded sampler further down samples it as galario does.
// chi^2 = sum w ((Re_d - Re_m)^2 + (Im_d - Im_m)^2) (libinterferometry.pyx:619-633).
//
// Both directions of the exact DFT run on the matrix cores over the image folded
// about its centre (c_x, c_y) = the middle of its pixel positions: with
// x_k - c_x = +-X_m and y_j - c_y = +-Y_l the four pixels of a (l, m) pair enter as
// their sums and differences, with cosines and sines of X_m and Y_l alone --
// half the multiplications of the plain sum, and real ones.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "rt_internal.h"

#define VIS_BS 256
// More rows are an error of rt_vis_dft, as they were when its kernel held whole columns
// in LDS; this one has no such bound, but a call that was refused stays refused
#define VIS_MAXROWS 1024
#define VIS_TK 32  // columns (of the folded image) per staged tile
#define VIS_REF 8  // matrix-core steps between exact phasors

typedef float vf4 __attribute__((ext_vector_type(4)));
typedef float vf16 __attribute__((ext_vector_type(16)));

// cos and sin of 2 pi a, a reduced in FP64
__device__ __forceinline__ void phasor(double a, float &c, float &s) {
    sincospif(2.f * (float)(a - rint(a)), &s, &c);
}

// entries of a folded axis of n pixels and the first one's distance from the
// centre (pixels): pixel n/2 + l lies at l + off, its partner at -(l + off)
__device__ __host__ __forceinline__ int fold_n(int n) { return (n + 1) / 2; }
__device__ __forceinline__ double fold_off(int n) { return (n & 1) ? 0.0 : 0.5; }
__device__ __forceinline__ int fold_lo(int n, int l) { return (n & 1) ? n / 2 - l : n / 2 - 1 - l; }

// V(u,v): with the folded planes EE, EO, OE, OO (E: sum, O: difference; first
// letter rows), a = 2 pi u X_m, b = 2 pi v Y_l,
//   Re V = sum_l cos b (sum_m EE cos a) - sin b (sum_m OO sin a)
//   Im V = -sum_l cos b (sum_m EO sin a) + sin b (sum_m OE cos a)
// times the shift of the centre.  The inner sums are four products
// [32 rows x m] x [m x 32 points] with v_mfma_f32_32x32x2f32: a lane holds its
// point's cos a or sin a of one column (rotated by two pixels a step, exact
// every VIS_REF steps, so no table is needed), the folded rows come from LDS, one
// 16-byte read per step for all four.  2 nx ny flops per point: 6.5 GFLOP
// at 256 x 256 and 5e4 points, 42 us at the FP32 matrix peak; 411 us with plain sums
// on the vector units, 101 now (1e6 points: 5005 and 1445), the phasors' rotation and
// the staging between barriers taking the rest.  4 / NRS groups of 32
// points per workgroup share the staged rows; with NRS = 4 the four waves take
// every fourth 32 rows of one group of points instead (few points: the GPU would
// be short of waves), added in order.
template <int NRS>
__global__ void __launch_bounds__(VIS_BS) k_vis(const float *img, int nx, int ny, const double *u,
                                                const double *v, int K, double dxy, double dra,
                                                double ddec, float *re, float *im) {
    constexpr int NP = 4 / NRS;
    __shared__ vf4 pl[NRS][32][VIS_TK + 1];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, rs = w % NRS, pg = w / NRS;
    const int i32 = lane & 31, kh = lane >> 5;
    const int q = (blockIdx.x * NP + pg) * 32 + i32;
    const int hx = fold_n(nx), hy = fold_n(ny);
    const double ox = fold_off(nx), oy = fold_off(ny);
    const double uq = q < K ? u[q] : 0.0, vq = q < K ? v[q] : 0.0;
    const double ud = uq * dxy, vd = vq * dxy;
    float c2, s2, c1, s1;  // two columns, one row
    phasor(2.0 * ud, c2, s2);
    phasor(vd, c1, s1);
    float sr = 0.f, si = 0.f;
    const int nt = (hy + 32 * NRS - 1) / (32 * NRS);
    for (int t = 0; t < nt; ++t) {
        const int l0 = (t * NRS + rs) * 32;
        vf16 pee = {}, poo = {}, peo = {}, poe = {};
        for (int m0 = 0; m0 < hx; m0 += VIS_TK) {
            __syncthreads();
            for (int e = pg * 64 + lane; e < 32 * VIS_TK; e += NP * 64) {
                const int l = l0 + e / VIS_TK, m = m0 + e % VIS_TK;
                float a = 0.f, b = 0.f, c = 0.f, d = 0.f;
                if (l < hy && m < hx) {
                    const int jp = ny / 2 + l, jm = fold_lo(ny, l), kp = nx / 2 + m,
                              km = fold_lo(nx, m);
                    const bool two_r = jm != jp, two_c = km != kp;
                    a = img[(size_t)jp * nx + kp];
                    if (two_c) b = img[(size_t)jp * nx + km];
                    if (two_r) c = img[(size_t)jm * nx + kp];
                    if (two_r && two_c) d = img[(size_t)jm * nx + km];
                }
                const float ab = a + b, cd = c + d, am = a - b, cm = c - d;
                vf4 o = {ab + cd, am - cm, am + cm, ab - cd};  // EE, OO, EO, OE
                pl[rs][e / VIS_TK][e % VIS_TK] = o;
            }
            __syncthreads();
            const int ns = min(VIS_TK, (hx - m0 + 1) & ~1) / 2;
            float ca = 1.f, sa = 0.f;
            for (int st = 0; st < ns; ++st) {
                const int m = 2 * st + kh;
                if (st % VIS_REF == 0) {
                    phasor(ud * ((double)(m0 + m) + ox), ca, sa);
                } else {
                    const float nc = ca * c2 - sa * s2;
                    sa = fmaf(ca, s2, sa * c2);
                    ca = nc;
                }
                const vf4 f = pl[rs][i32][m];
                pee = __builtin_amdgcn_mfma_f32_32x32x2f32(f[0], ca, pee, 0, 0, 0);
                poo = __builtin_amdgcn_mfma_f32_32x32x2f32(f[1], sa, poo, 0, 0, 0);
                peo = __builtin_amdgcn_mfma_f32_32x32x2f32(f[2], sa, peo, 0, 0, 0);
                poe = __builtin_amdgcn_mfma_f32_32x32x2f32(f[3], ca, poe, 0, 0, 0);
            }
        }
        // lane: point i32, rows l0 + 8 g + 4 kh .. + 3 in elements 4 g .. 4 g + 3
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float cb, sb;
            phasor(vd * ((double)(l0 + 8 * g + 4 * kh) + oy), cb, sb);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 4 * g + e;
                sr += cb * pee[r] - sb * poo[r];
                si -= cb * peo[r] + sb * poe[r];
                const float nc = cb * c1 - sb * s1;
                sb = fmaf(cb, s1, sb * c1);
                cb = nc;
            }
        }
    }
    sr += __shfl_xor(sr, 32);
    si += __shfl_xor(si, 32);
    if (NRS > 1) {
        __syncthreads();
        float *red = (float *)&pl[0][0][0];  // [NRS][2][32]
        if (kh == 0) {
            red[rs * 64 + i32] = sr;
            red[rs * 64 + 32 + i32] = si;
        }
        __syncthreads();
        sr = si = 0.f;
#pragma unroll
        for (int r = 0; r < NRS; ++r) {
            sr += red[r * 64 + i32];
            si += red[r * 64 + 32 + i32];
        }
    }
    if (rs == 0 && kh == 0 && q < K) {
        // the image's phase centre lies ox, oy pixels past the folding centre
        double sn, cs;
        sincospi(-2.0 * (uq * dra + vq * ddec - ox * ud - oy * vd), &sn, &cs);
        re[q] = (float)(sr * cs - si * sn);
        im[q] = (float)(sr * sn + si * cs);
    }
}

// ---- the transpose: g[j][k] = Re sum_q H_q exp(-i (+-a_qm +- b_ql)) about the
// folding centre, H_q = (gre_q - i gim_q) times the shift, a = 2 pi u X_m, b = 2 pi v
// Y_l.  With
//   P1 = sum Hr cos a cos b, P2 = sum Hr sin a sin b,
//   P3 = sum Hi sin a cos b, P4 = sum Hi cos a sin b
// the pixel at signs (s, t) of (X, Y) is P1 - s t P2 + s P3 + t P4: four products
// [l x q] x [q x m] on v_mfma_f32_32x32x2f32, half the multiplications of the
// plain sum.  A workgroup takes 64 x 64 entries (l, m) -- four waves of 32 x 32 --
// and a share of the points, 32 at a time: their cosines and sines go through
// LDS once (16 entries per lane, exact every 8, rotated in between) and serve
// 64 x 64 x 4 products, so the matrix cores set the pace.  The folded image has
// few such tiles, so the points are split over the CUs (adj_split);
// their partial planes are added in order by k_vis_adj_sum.
// 256 x 256 pixels, 5e4 points: 467 us with k_vis_adj, 111 now; 1024 x 1024: 7446
// and 1219.
// An accumulator takes 64 chunks and is then added to the share's sum: a large
// image has few shares (8 at 1024 x 1024, one from about 2450 x 2450 on), and the
// rounding of an FP32 sum grows with the root of its number of terms.  2048 x 2048, 1e6
// points, rms error over rms gradient: 1.3e-5 in one sum per share, 9e-7 now.
#define VA_CH 32   // points per chunk
#define VA_SUM 64  // chunks per accumulator
// below this many pixel x point products k_vis_adj, which needs no scratch and one
// launch, is the faster one: 22 against 27 us at 256 x 256 and 2e3 points, 51
// against 31 at 5e3 (smaller images count as 256 x 256: they take as long)
#define VIS_ADJ_MIN (65536.0 * 3072.0)

struct AdjSplit {
    int tx, ty, splits, per;  // tiles, shares of the points, chunks per share
    int wpc;                  // workgroups per CU (2 or 3)
};

// Shares that fill two workgroups per CU, which is what the registers allow at full
// speed, or three, 5 % slower each (some are spilled), where that comes out
// ahead: a launch takes its rounds of them.  2300 x 2300 pixels (324 tiles): two shares
// at three per CU 4.1 ms, one at two 5.8; 300 x 300 (9 tiles): 56 shares, 504
// workgroups at two per CU, 0.38 ms, 57 shares 0.44.
static AdjSplit adj_split(const rt_ctx *ctx, int nx, int ny, int K) {
    AdjSplit a;
    a.tx = (fold_n(nx) + 63) / 64;
    a.ty = (fold_n(ny) + 63) / 64;
    const long tiles = (long)a.tx * a.ty, chunks = ((long)K + VA_CH - 1) / VA_CH;
    double best = 0.0;
    long s = 1;
    for (int wpc = 2; wpc <= 3; ++wpc) {
        const long c = (long)wpc * ctx->n_cu, n = std::max(1l, std::min(c / tiles, (chunks + 3) / 4));
        const double cost = (double)((tiles * n + c - 1) / c) * wpc / n * (wpc == 3 ? 1.05 : 1.0);
        if (wpc == 2 || cost < best) {
            best = cost;
            s = n;
            a.wpc = wpc;
        }
    }
    a.per = (int)((chunks + s - 1) / s);
    a.splits = (int)((chunks + a.per - 1) / a.per);
    return a;
}

static bool adj_tiled(int nx, int ny, int K) {
    return std::max(65536.0, (double)nx * ny) * K >= VIS_ADJ_MIN;
}

// at most 3 n_cu workgroups' planes: 48 MiB on 256 CUs
size_t vis_adjoint_workspace(const rt_ctx *ctx, int nx, int ny, int K) {
    if (nx < 1 || ny < 1 || !adj_tiled(nx, ny, K)) return 0;
    const AdjSplit a = adj_split(ctx, nx, ny, K);
    return a.splits > 1 ? (size_t)a.tx * a.ty * a.splits * 4 * 64 * 64 * sizeof(float) : 0;
}

// the four pixels of the folded entry (l, m)
__device__ __forceinline__ void unfold_pixels(int l, int m, int nx, int ny, float p1, float p2,
                                              float p3, float p4, float *gimg) {
    if (l >= fold_n(ny) || m >= fold_n(nx)) return;
    const int jp = ny / 2 + l, jm = fold_lo(ny, l), kp = nx / 2 + m, km = fold_lo(nx, m);
    gimg[(size_t)jp * nx + kp] = (p1 - p2) + (p3 + p4);
    if (km != kp) gimg[(size_t)jp * nx + km] = (p1 + p2) + (p4 - p3);
    if (jm != jp) gimg[(size_t)jm * nx + kp] = (p1 + p2) + (p3 - p4);
    if (jm != jp && km != kp) gimg[(size_t)jm * nx + km] = (p1 - p2) - (p3 + p4);
}

// WPC: workgroups per CU the registers are kept for
template <int WPC>
__global__ void __launch_bounds__(256, WPC) k_vis_adj_part(const float *gre, const float *gim, int nx,
                                                      int ny, const double *u, const double *v,
                                                      int K, double dxy, double dra, double ddec,
                                                      int per, float *part, float *gimg) {
    __shared__ float2 ra[VA_CH][64 + 1], ca[VA_CH][64 + 1];  // rows: cos b, sin b; columns: cos a, sin a
    __shared__ float2 H[VA_CH];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int i32 = lane & 31, kh = lane >> 5, wr = (w >> 1) * 32, wc = (w & 1) * 32;
    const int l0 = blockIdx.y * 64, m0 = blockIdx.x * 64;
    const double ox = fold_off(nx), oy = fold_off(ny);
    vf16 p1 = {}, p2 = {}, p3 = {}, p4 = {}, t1 = {}, t2 = {}, t3 = {}, t4 = {};
    // table: lane of point tp, 16 rows (tg < 4) or columns
    const int tp = threadIdx.x >> 3, tg = threadIdx.x & 7;
    const int c0 = blockIdx.z * per, c1 = min(c0 + per, (K + VA_CH - 1) / VA_CH);
    for (int c = c0; c < c1; ++c) {
        const int q = c * VA_CH + tp;
        const double uq = q < K ? u[q] : 0.0, vq = q < K ? v[q] : 0.0;
        __syncthreads();
        {
            const bool row = tg < 4;
            const int e0 = (tg & 3) * 16;
            const double f = (row ? vq : uq) * dxy;
            const double base = (row ? (double)l0 + oy : (double)m0 + ox) + e0;
            float2(*tab)[64 + 1] = row ? ra : ca;
            float cs, sn, c1s, s1s;
            phasor(f, c1s, s1s);
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                if (e % 8 == 0) {
                    phasor(f * (base + e), cs, sn);
                } else {
                    const float nc = cs * c1s - sn * s1s;
                    sn = fmaf(cs, s1s, sn * c1s);
                    cs = nc;
                }
                tab[tp][e0 + e] = make_float2(cs, sn);
            }
            if (tg == 0) {
                float hr = 0.f, hi = 0.f;
                if (q < K) {
                    double s, cc;
                    sincospi(-2.0 * (uq * dra + vq * ddec - (ox * uq + oy * vq) * dxy), &s, &cc);
                    const float gr = gre[q], gi = gim[q];
                    hr = (float)(gr * cc + gi * s);
                    hi = (float)(gr * s - gi * cc);
                }
                H[tp] = make_float2(hr, hi);
            }
        }
        __syncthreads();
#pragma unroll 4
        for (int st = 0; st < VA_CH / 2; ++st) {
            const int k = 2 * st + kh;
            const float2 r = ra[k][wr + i32], a = ca[k][wc + i32], h = H[k];
            p1 = __builtin_amdgcn_mfma_f32_32x32x2f32(r.x, h.x * a.x, p1, 0, 0, 0);
            p2 = __builtin_amdgcn_mfma_f32_32x32x2f32(r.y, h.x * a.y, p2, 0, 0, 0);
            p3 = __builtin_amdgcn_mfma_f32_32x32x2f32(r.x, h.y * a.y, p3, 0, 0, 0);
            p4 = __builtin_amdgcn_mfma_f32_32x32x2f32(r.y, h.y * a.x, p4, 0, 0, 0);
        }
        if ((c - c0) % VA_SUM == VA_SUM - 1 || c == c1 - 1) {
            t1 += p1;
            t2 += p2;
            t3 += p3;
            t4 += p4;
            p1 = p2 = p3 = p4 = vf16{};
        }
    }
    if (!part) {  // one share: no planes
#pragma unroll
        for (int r = 0; r < 16; ++r)
            unfold_pixels(l0 + wr + 8 * (r >> 2) + 4 * kh + (r & 3), m0 + wc + i32, nx, ny, t1[r],
                          t2[r], t3[r], t4[r], gimg);
        return;
    }
    // [share][tile][plane][64][64]
    float *o = part + (((size_t)blockIdx.z * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x) *
                          (4 * 64 * 64);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int at = (wr + 8 * (r >> 2) + 4 * kh + (r & 3)) * 64 + wc + i32;
        o[at] = t1[r];
        o[at + 4096] = t2[r];
        o[at + 2 * 4096] = t3[r];
        o[at + 3 * 4096] = t4[r];
    }
}

// one folded entry (l, m) per lane: the shares' planes added in order, four pixels
__global__ void __launch_bounds__(256) k_vis_adj_sum(const float *part, int splits, int nx, int ny,
                                                     float *gimg) {
    const int tx = gridDim.x, ty = gridDim.y;
    const int e = blockIdx.z * 256 + threadIdx.x;  // of the tile's 64 x 64
    const int l = blockIdx.y * 64 + e / 64, m = blockIdx.x * 64 + e % 64;
    const float *p = part + ((size_t)blockIdx.y * tx + blockIdx.x) * (4 * 4096) + e;
    float p1 = 0.f, p2 = 0.f, p3 = 0.f, p4 = 0.f;
    const size_t step = (size_t)tx * ty * (4 * 4096);
#pragma unroll 4
    for (int s = 0; s < splits; ++s, p += step) {
        p1 += p[0];
        p2 += p[4096];
        p3 += p[2 * 4096];
        p4 += p[3 * 4096];
    }
    unfold_pixels(l, m, nx, ny, p1, p2, p3, p4, gimg);
}

#define ADJ_T 16
#define ADJ_CH 64
#define ADJ_G 4   // point groups per tile: each takes every ADJ_G-th chunk of points
#define ADJ_BS (ADJ_T * ADJ_T * ADJ_G)

// g[j][k] = Re sum_q H_q a_qk b_qj,  H_q = (gre_q - i gim_q) shift_q,
// a_qk = exp(-2 pi i u_q x_k), b_qj = exp(-2 pi i v_q y_j)
// One workgroup per 16x16 tile, ADJ_G groups of 256 lanes; group g takes the
// chunks g, g + ADJ_G, ... of the points, builds the chunk's phasor tables in
// LDS, and each of its four waves adds 16 of the chunk's points to its own copy
// of the tile on the matrix cores.  The 16 copies are added in wave order, so
// the result does not depend on scheduling.
__global__ void __launch_bounds__(ADJ_BS) k_vis_adj(const float *gre, const float *gim, int nx,
                                                    int ny, const double *u, const double *v,
                                                    int K, double dxy, double dra, double ddec,
                                                    float *gimg) {
    __shared__ float Ha_r[ADJ_G][ADJ_CH][ADJ_T], Ha_i[ADJ_G][ADJ_CH][ADJ_T];
    __shared__ float b_r[ADJ_G][ADJ_CH][ADJ_T], b_i[ADJ_G][ADJ_CH][ADJ_T];
    __shared__ float H_r[ADJ_G][ADJ_CH], H_i[ADJ_G][ADJ_CH];
    __shared__ float sa_c[ADJ_G][ADJ_CH], sa_s[ADJ_G][ADJ_CH], sb_c[ADJ_G][ADJ_CH],
        sb_s[ADJ_G][ADJ_CH];
    __shared__ double s_u[ADJ_G][ADJ_CH], s_v[ADJ_G][ADJ_CH];  // u dxy, v dxy
    const int g = threadIdx.x / (ADJ_T * ADJ_T), lt = threadIdx.x - g * (ADJ_T * ADJ_T);
    const int tx = lt % ADJ_T, ty = lt / ADJ_T;
    const int k0 = blockIdx.x * ADJ_T, j0 = blockIdx.y * ADJ_T;
    const int k = k0 + tx, j = j0 + ty;
    // matrix-core layout: wave wv of the group, lane = mq * 16 + mc
    const int wv = lt >> 6, mq = (lt >> 4) & 3, mc = lt & 15;
    vf4 acc4 = {0.f, 0.f, 0.f, 0.f};
    // loader: 4 threads per point, 4 consecutive columns / rows each
    const int lq = lt >> 2, ll = (lt & 3) * 4;
    const int nch = (K + ADJ_CH - 1) / ADJ_CH;
    // the setup lanes' point data, loaded one round ahead so that the loads
    // are in flight while the round before runs (the barrier waits for none)
    double pu = 0.0, pv = 0.0;
    float pgr = 0.f, pgi = 0.f;
    if (lt < ADJ_CH && g * ADJ_CH + lt < K) {
        const int q = g * ADJ_CH + lt;
        pu = u[q];
        pv = v[q];
        pgr = gre[q];
        pgi = gim[q];
    }
    for (int c0 = 0; c0 < nch; c0 += ADJ_G) {
        const int q0 = (c0 + g) * ADJ_CH;  // past K for some groups in the last round
        const double cu = pu, cv = pv;
        const float gr = pgr, gi = pgi;
        if (lt < ADJ_CH && q0 + ADJ_G * ADJ_CH + lt < K) {
            const int qn = q0 + ADJ_G * ADJ_CH + lt;
            pu = u[qn];
            pv = v[qn];
            pgr = gre[qn];
            pgi = gim[qn];
        }
        __syncthreads();
        // per point: the cotangent with the phase-centre shift and the
        // one-pixel steps of its column and row phasors
        if (lt < ADJ_CH) {
            const int q = q0 + lt;
            float hr = 0.f, hi = 0.f, s1 = 0.f, c1 = 1.f, s2 = 0.f, c2 = 1.f;
            double su = 0.0, sv = 0.0;
            if (q < K) {
                double s, c;
                sincospi(-2.0 * (cu * dra + cv * ddec), &s, &c);
                // H = (gre - i gim) * (c + i s)
                hr = (float)(gr * c + gi * s);
                hi = (float)(gr * s - gi * c);
                su = cu * dxy;
                sv = cv * dxy;
                phasor(-su, c1, s1);
                phasor(-sv, c2, s2);
            }
            H_r[g][lt] = hr;
            H_i[g][lt] = hi;
            sa_c[g][lt] = c1;
            sa_s[g][lt] = s1;
            sb_c[g][lt] = c2;
            sb_s[g][lt] = s2;
            s_u[g][lt] = su;
            s_v[g][lt] = sv;
        }
        __syncthreads();
        {
            const int q = q0 + lq;
            float hr = 0.f, hi = 0.f, ar = 0.f, ai = 0.f, br = 0.f, bi = 0.f;
            float dac = 1.f, das = 0.f, dbc = 1.f, dbs = 0.f;
            if (q < K) {
                hr = H_r[g][lq];
                hi = H_i[g][lq];
                phasor(-s_u[g][lq] * (double)(k0 + ll - nx / 2), ar, ai);
                phasor(-s_v[g][lq] * (double)(j0 + ll - ny / 2), br, bi);
                dac = sa_c[g][lq];
                das = sa_s[g][lq];
                dbc = sb_c[g][lq];
                dbs = sb_s[g][lq];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                Ha_r[g][lq][ll + e] = hr * ar - hi * ai;
                Ha_i[g][lq][ll + e] = hr * ai + hi * ar;
                b_r[g][lq][ll + e] = br;
                b_i[g][lq][ll + e] = bi;
                // next column / row: rotate by one pixel step
                const float nar = ar * dac - ai * das;
                ai = fmaf(ar, das, ai * dac);
                ar = nar;
                const float nbr = br * dbc - bi * dbs;
                bi = fmaf(br, dbs, bi * dbc);
                br = nbr;
            }
        }
        __syncthreads();
        // the tile's update by the wave's 16 points on the matrix cores:
        // G[j][k] += sum_q b_r[q][j] Ha_r[q][k] - b_i[q][j] Ha_i[q][k], four points
        // per v_mfma_f32_16x16x4f32 (A[j][q] from lane q*16 + j, B[q][k] from
        // lane q*16 + k)
#pragma unroll
        for (int st = 0; st < ADJ_CH / 16; ++st) {
            const int qq = wv * 16 + st * 4 + mq;
            acc4 = __builtin_amdgcn_mfma_f32_16x16x4f32(b_r[g][qq][mc], Ha_r[g][qq][mc], acc4, 0, 0, 0);
            acc4 = __builtin_amdgcn_mfma_f32_16x16x4f32(-b_i[g][qq][mc], Ha_i[g][qq][mc], acc4, 0, 0, 0);
        }
    }
    // the 16 waves' tiles (lane q*16 + k holds rows 4q..4q+3 of column k),
    // added in wave order; the phasor buffers are free now
    __syncthreads();
    float *red = &Ha_r[0][0][0];
    const int w16 = g * 4 + wv;
#pragma unroll
    for (int r = 0; r < 4; ++r) red[w16 * (ADJ_T * ADJ_T) + (4 * mq + r) * ADJ_T + mc] = acc4[r];
    __syncthreads();
    if (g == 0 && k < nx && j < ny) {
        float sum = red[lt];
        for (int h = 1; h < 4 * ADJ_G; ++h) sum += red[h * (ADJ_T * ADJ_T) + lt];
        gimg[(size_t)j * nx + k] = sum;
    }
}

// ---- gridded sampler: galario's method (Tazzari, Beaujean & Testi 2018,
// MNRAS 476, 4527: Fourier transform of the image on its pixel-conjugate grid,
// bilinear interpolation at each (u,v), then the phase-centre shift), which is
// what pdspy's interpolate_model calls (interpolate_model.py:20-27).
// F[b][a] = sum_jk I[j][k] w_nx((a - nx/2)(k - nx/2)) w_ny((b - ny/2)(j - ny/2)),
// w_n(r) = exp(-2 pi i r / n), is the exact DFT at u_a = (a - nx/2) / (nx dxy),
// v_b = (b - ny/2) / (ny dxy); it is computed as two passes of 1D transforms
// with integer phase indices into one twiddle table per axis, so every twiddle
// is exact to FP32 rounding.  Work:
// [A: ny x nx float2][F: ny x nx float2][twiddles: nx + ny float2] (of A one half
// is used).
#define GRID_BS 256
#define GRID_MAXN 4096

__global__ void __launch_bounds__(GRID_BS) k_grid_twiddles(int nx, int ny, float2 *tw) {
    const int i = blockIdx.x * GRID_BS + threadIdx.x;
    if (i >= nx + ny) return;
    const int n = i < nx ? nx : ny, r = i < nx ? i : i - nx;
    double s, c;
    sincospi(-2.0 * (double)r / (double)n, &s, &c);
    tw[i] = make_float2((float)c, (float)s);
}

// The transform on the grid, folded in both image and grid axes about their node 0
// (index n/2): with the planes EE, OE, EO, OO over k = 0..nx/2, l = 0..ny/2 (E: sum,
// O: difference of the pixels at +-; first letter rows), angles a k of 2 pi / nx and
// b l of 2 pi / ny,
//   rows:    X0 = sum_l EE cos bl, X1 = sum_l OE sin bl, X2 = sum_l EO cos bl,
//            X3 = sum_l OO sin bl                                 (FIRST)
//   columns: F1 = sum_k X0 cos ak, F2 = sum_k X3 sin ak, F3 = sum_k X2 sin ak,
//            F4 = sum_k X1 cos ak
// and the node (sgn_a a, sgn_b b) is (F1 - sgn_a sgn_b F2) - i (sgn_a F3 + sgn_b F4):
// a quarter of the plain sums' multiplications, on v_mfma_f32_16x16x4f32.  A
// workgroup makes 16 x (16 * GRID_NB) entries of the four planes, its four waves
// taking every fourth group of four terms; a lane's value operand is read from
// L2 where the sum is (64-byte runs), its cosines and sines from the twiddle
// table in LDS.  1024 x 1024: 32 + 29 us (572 with the
// plain sums), 7 us each at the FP32 matrix peak; the operands' address and
// fold instructions pace it.  Measured without effect: rotated instead of looked-up
// phases, the loads of 4 or 8 groups ahead, 16 x 64 entries; 16 x 16 entries: 34 us.
#define GRID_NB 2

template <bool FIRST>
__global__ void __launch_bounds__(GRID_BS) k_grid_dft(const float *src, const float2 *twg, int nx,
                                                      int ny, int flip, float *X, float2 *F) {
    __shared__ __align__(16) float sm[4 * 16 * GRID_NB * 64];  // twiddles, then the waves' sums
    static_assert(sizeof(sm) >= GRID_MAXN * sizeof(float2), "the table fits");
    float2 *tw = (float2 *)sm;
    const int n = FIRST ? ny : nx;  // the transformed axis
    for (int i = threadIdx.x; i < n; i += GRID_BS) tw[i] = twg[i];
    __syncthreads();
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i16 = lane & 15, kh = lane >> 4;
    const int cx = nx / 2, cy = ny / 2, hx = cx + 1, hy = cy + 1;  // E entries
    const int ox = (nx - 1) / 2, oy = (ny - 1) / 2;                // O entries (1, 2, ..)
    // X0 [hx][hy], X1 [hx][oy], X2 [ox][hy], X3 [ox][oy]: nx ny floats
    float *X1 = X + (size_t)hx * hy, *X2 = X1 + (size_t)hx * oy, *X3 = X2 + (size_t)ox * hy;
    const int v0 = blockIdx.x * 16, f0 = blockIdx.y * (16 * GRID_NB);
    const int vi = v0 + i16, h = FIRST ? hy : hx;
    int r[GRID_NB], dr[GRID_NB];
    vf4 acc[GRID_NB][4];
#pragma unroll
    for (int b = 0; b < GRID_NB; ++b) {
        const int f = f0 + 16 * b + i16;
        r[b] = (f * (4 * w + kh)) % n;
        dr[b] = (16 * f) % n;
#pragma unroll
        for (int p = 0; p < 4; ++p) acc[b][p] = vf4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll 4
    for (int t0 = 4 * w; t0 < h; t0 += 16) {
        const int t = t0 + kh;
        float x[4] = {0.f, 0.f, 0.f, 0.f};
        if (FIRST) {
            const int jp = cy + t, jm = cy - t, kp = cx + vi, km = cx - vi;
            const bool rp = jp < ny, rm = t > 0 && jm >= 0, cp = kp < nx, cm = vi > 0 && km >= 0;
            const float *ip = src + (size_t)(flip ? ny - 1 - jp : jp) * nx;
            const float *im = src + (size_t)(flip ? ny - 1 - jm : jm) * nx;
            const float pp = rp && cp ? ip[kp] : 0.f, pm = rp && cm ? ip[km] : 0.f;
            const float mp = rm && cp ? im[kp] : 0.f, mm = rm && cm ? im[km] : 0.f;
            const float e = pp + pm, d = pp - pm, em = mp + mm, dm = mp - mm;
            x[0] = e + em;
            x[1] = e - em;
            x[2] = d + dm;
            x[3] = d - dm;
        } else {
            const bool ek = t < hx, ok = t > 0 && t <= ox, eb = vi < hy, ob = vi > 0 && vi <= oy;
            if (ek && eb) x[0] = X[(size_t)t * hy + vi];
            if (ek && ob) x[1] = X1[(size_t)t * oy + vi - 1];
            if (ok && eb) x[2] = X2[(size_t)(t - 1) * hy + vi];
            if (ok && ob) x[3] = X3[(size_t)(t - 1) * oy + vi - 1];
        }
#pragma unroll
        for (int b = 0; b < GRID_NB; ++b) {
            const float c = tw[r[b]].x, s = -tw[r[b]].y;
            acc[b][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[0], c, acc[b][0], 0, 0, 0);
            acc[b][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[1], FIRST ? s : c, acc[b][1], 0, 0, 0);
            acc[b][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[2], FIRST ? c : s, acc[b][2], 0, 0, 0);
            acc[b][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[3], s, acc[b][3], 0, 0, 0);
            r[b] += dr[b];
            if (r[b] >= n) r[b] -= n;
        }
    }
    // the four waves' sums, in order; wave w finishes elements e = 2w, 2w + 1, .. of a lane
    __syncthreads();
#pragma unroll
    for (int b = 0; b < GRID_NB; ++b)
#pragma unroll
        for (int p = 0; p < 4; ++p)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                sm[((w * GRID_NB + b) * 16 + p * 4 + e) * 64 + lane] = acc[b][p][e];
    __syncthreads();
    for (int z = w; z < 4 * GRID_NB; z += 4) {
        const int b = z >> 2, e = z & 3;
        const int v = v0 + 4 * kh + e, f = f0 + 16 * b + i16;  // row, column of the products
        float o[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const float *q = sm + (b * 16 + p * 4 + e) * 64 + lane;
            constexpr int W = GRID_NB * 16 * 64;
            o[p] = (q[0] + q[W]) + (q[2 * W] + q[3 * W]);
        }
        if (FIRST) {
            const bool ek = v < hx, ok = v > 0 && v <= ox, eb = f < hy, ob = f > 0 && f <= oy;
            if (ek && eb) X[(size_t)v * hy + f] = o[0];
            if (ek && ob) X1[(size_t)v * oy + f - 1] = o[1];
            if (ok && eb) X2[(size_t)(v - 1) * hy + f] = o[2];
            if (ok && ob) X3[(size_t)(v - 1) * oy + f - 1] = o[3];
        } else if (v < hy && f < hx) {
            // o: F1, F4, F3, F2
            const float pr = o[0] - o[3], mr = o[0] + o[3], ps = o[1] + o[2], ds = o[2] - o[1];
            const int bp = cy + v, bm = cy - v, ap = cx + f, am = cx - f;
            if (bp < ny && ap < nx) F[(size_t)bp * nx + ap] = make_float2(pr, -ps);
            if (bp < ny && f > 0) F[(size_t)bp * nx + am] = make_float2(mr, ds);
            if (v > 0 && ap < nx) F[(size_t)bm * nx + ap] = make_float2(mr, -ds);
            if (v > 0 && f > 0) F[(size_t)bm * nx + am] = make_float2(pr, ps);
        }
    }
}

// position of a (u,v) coordinate on a grid axis of step 1 / s, the product and the
// sum rounded one by one: the check and the sampler agree to the last bit
__device__ __forceinline__ double grid_pos(double u, double s, int n) {
#pragma clang fp contract(off)
    return u * s + (double)(n / 2);
}

// *outside |= 1 if a point's four nodes are not all on the grid (NaN: not either).
// One pass over (u, v), 16 bytes a point, for what was fifteen elementwise passes and
// a reduction: 63 us of kernels at 1e6 points, 8 us now (zeroing included).
__global__ void __launch_bounds__(GRID_BS) k_grid_outside(int nx, int ny, double dxy,
                                                          const double *u, const double *v, int K,
                                                          double usgn, int *outside) {
    const double sx = (double)nx * dxy, sy = (double)ny * dxy;
    bool bad = false;
    for (int q = blockIdx.x * GRID_BS + threadIdx.x; q < K; q += gridDim.x * GRID_BS) {
        const double fa = grid_pos(usgn * u[q], sx, nx);
        const double fb = grid_pos(usgn * v[q], sy, ny);
        bad |= !(fa >= 0.0 && fa < (double)(nx - 1) && fb >= 0.0 && fb < (double)(ny - 1));
    }
    if (__any(bad) && (threadIdx.x & 63) == 0) atomicOr(outside, 1);
}

int vis_grid_outside_run(rt_ctx *ctx, int nx, int ny, double dxy, const double *d_u,
                         const double *d_v, int K, int conv, int *d_outside) {
    if (nx < 0 || ny < 0 || K < 0 || (K > 0 && (!d_u || !d_v)) || !d_outside)
        return set_err(ctx, RT_E_ARG, "vis grid: invalid sizes or NULL (u,v)");
    if (K == 0) return RT_OK;
    const int nb = std::min((K - 1) / GRID_BS + 1, 8 * ctx->n_cu);
    hipLaunchKernelGGL(k_grid_outside, dim3(nb), dim3(GRID_BS), 0, ctx->stream, nx, ny, dxy, d_u,
                       d_v, K, conv == 1 ? -1.0 : 1.0, d_outside);
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}

// one (u,v) point per lane: bilinear interpolation between the four grid nodes
// around (usgn u, usgn v), then the phase-centre shift at (u, v); a point whose
// four nodes are not all on the grid gets NaN
__global__ void __launch_bounds__(GRID_BS) k_grid_sample(const float2 *F, int nx, int ny,
                                                         double dxy, const double *u,
                                                         const double *v, int K, double usgn,
                                                         double dra, double ddec, float *re,
                                                         float *im) {
    const int q = blockIdx.x * GRID_BS + threadIdx.x;
    if (q >= K) return;
    const double uq = u[q], vq = v[q];
    const double fa = grid_pos(usgn * uq, (double)nx * dxy, nx);
    const double fb = grid_pos(usgn * vq, (double)ny * dxy, ny);
    const double a0 = floor(fa), b0 = floor(fb);
    if (!(a0 >= 0.0 && a0 <= (double)(nx - 2) && b0 >= 0.0 && b0 <= (double)(ny - 2))) {
        re[q] = __builtin_nanf("");
        im[q] = __builtin_nanf("");
        return;
    }
    const size_t o = (size_t)b0 * nx + (size_t)a0;
    const float2 f00 = F[o], f01 = F[o + 1], f10 = F[o + nx], f11 = F[o + nx + 1];
    const double ta = fa - a0, tb = fb - b0;
    const double w00 = (1.0 - ta) * (1.0 - tb), w01 = ta * (1.0 - tb), w10 = (1.0 - ta) * tb,
                 w11 = ta * tb;
    const double sr = w00 * f00.x + w01 * f01.x + w10 * f10.x + w11 * f11.x;
    const double si = w00 * f00.y + w01 * f01.y + w10 * f10.y + w11 * f11.y;
    double s, c;
    sincospi(-2.0 * (uq * dra + vq * ddec), &s, &c);
    re[q] = (float)(sr * c - si * s);
    im[q] = (float)(sr * s + si * c);
}

size_t vis_grid_workspace(int nx, int ny) {
    return sizeof(float2) * (2 * (size_t)nx * ny + (size_t)nx + ny);
}

// Scratch of the allocation-free gridded sampler (rt_vis_grid_noalloc): the
// workspace of an image of up to VIS_NOALLOC_MAXN x VIS_NOALLOC_MAXN pixels
// (16.8 MB), one copy per GPU for the life of the process.  Host code never
// passes the array's name to a kernel: it is a host-side stand-in, and the
// device address of each GPU's copy is looked up once per device.
#define VIS_NOALLOC_MAXN 1024
static __device__ __align__(256) float2 scratch[2 * VIS_NOALLOC_MAXN * VIS_NOALLOC_MAXN +
                                                 2 * VIS_NOALLOC_MAXN];
#define VIS_MAX_DEVICES 64
static void *g_scratch_ptr[VIS_MAX_DEVICES];
static std::mutex g_scratch_mu;

// with `device` current: the device address of this GPU's scratch array
int vis_scratch_init(rt_ctx *ctx, int device) {
    if (device < 0 || device >= VIS_MAX_DEVICES)
        return set_err(ctx, RT_E_LIMIT, "device %d beyond the %d the library supports", device,
                       VIS_MAX_DEVICES);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return RT_OK;
    void *ptr = nullptr;
    hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
        return set_err(ctx, RT_E_HIP, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[device] = ptr;
    return RT_OK;
}

int vis_grid_noalloc_run(rt_ctx *ctx, const float *d_img, int nx, int ny, double dxy,
                         const double *d_u, const double *d_v, int K, double dra, double ddec,
                         float *d_re, float *d_im) {
    if (nx > VIS_NOALLOC_MAXN || ny > VIS_NOALLOC_MAXN)
        return set_err(ctx, RT_E_LIMIT, "rt_vis_grid_noalloc: %d x %d image exceeds its scratch "
                                        "(at most %d x %d pixels); use rt_vis_grid", nx, ny,
                       VIS_NOALLOC_MAXN, VIS_NOALLOC_MAXN);
    void *ptr = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (ctx->device >= 0 && ctx->device < VIS_MAX_DEVICES) ptr = g_scratch_ptr[ctx->device];
    }
    if (!ptr) return set_err(ctx, RT_E_HIP, "rt_vis_grid_noalloc: scratch of device %d not set up",
                             ctx->device);
    // every scratch word the kernels read is written first in the same call
    // (twiddles, row pass, column pass), so nothing needs clearing
    return vis_grid_run(ctx, d_img, nx, ny, dxy, d_u, d_v, K, dra, ddec, d_re, d_im, ptr, 0);
}

// conv 0: the imtovis convention above.  conv 1: pdspy's galario call
// (interpolate_model.py:23-27): galario's sampleImage of image[::-1] with the
// imaginary part negated.  galario samples G = transform of image[::-1] at
// (u, v) and multiplies by exp(+2 pi i (u dra + v ddec)); for a real image
// conj(G(u, v)) = G(-u, -v) holds node by node, hence also for the bilinear
// interpolant, so the negated imaginary part is G interpolated at (-u, -v)
// times exp(-2 pi i (u dra + v ddec)).
int vis_grid_run(rt_ctx *ctx, const float *d_img, int nx, int ny, double dxy, const double *d_u,
                 const double *d_v, int K, double dra, double ddec, float *d_re, float *d_im,
                 void *d_work, int conv) {
    if (nx < 2 || ny < 2 || nx > GRID_MAXN || ny > GRID_MAXN || K < 0 || !(dxy > 0))
        return set_err(ctx, RT_E_ARG, "vis grid: invalid sizes (2 <= nx, ny <= %d)", GRID_MAXN);
    if (K == 0) return RT_OK;
    if (!d_img || !d_u || !d_v || !d_re || !d_im)
        return set_err(ctx, RT_E_ARG, "vis grid: NULL image, (u,v) or output");
    float2 *ws = (float2 *)d_work;
    if (!ws) HIPCHK(ctx, hipMallocAsync((void **)&ws, vis_grid_workspace(nx, ny), ctx->stream));
    float *A = (float *)ws;  // the folded rows' transforms
    float2 *F = ws + (size_t)nx * ny, *tw = ws + 2 * (size_t)nx * ny;
    hipLaunchKernelGGL(k_grid_twiddles, dim3((nx + ny + GRID_BS - 1) / GRID_BS), dim3(GRID_BS), 0,
                       ctx->stream, nx, ny, tw);
    const int hx = nx / 2 + 1, hy = ny / 2 + 1, FW = 16 * GRID_NB;
    hipLaunchKernelGGL(k_grid_dft<true>, dim3((hx + 15) / 16, (hy + FW - 1) / FW), dim3(GRID_BS), 0,
                       ctx->stream, d_img, tw + nx, nx, ny, conv == 1 ? 1 : 0, A, F);
    hipLaunchKernelGGL(k_grid_dft<false>, dim3((hy + 15) / 16, (hx + FW - 1) / FW), dim3(GRID_BS), 0,
                       ctx->stream, d_img, tw, nx, ny, 0, A, F);
    hipLaunchKernelGGL(k_grid_sample, dim3((K + GRID_BS - 1) / GRID_BS), dim3(GRID_BS), 0,
                       ctx->stream, F, nx, ny, dxy, d_u, d_v, K, conv == 1 ? -1.0 : 1.0, dra, ddec,
                       d_re, d_im);
    if (!d_work) HIPCHK(ctx, hipFreeAsync(ws, ctx->stream));
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}

#define CHI_BS 256

__global__ void __launch_bounds__(CHI_BS) k_chisq(const float *dre, const float *dim, const float *w,
                                                  const float *mre, const float *mim, int K,
                                                  double *partial, float *gre, float *gim) {
    __shared__ double sh[CHI_BS];
    int q = blockIdx.x * CHI_BS + threadIdx.x;
    double x = 0.0;
    if (q < K) {
        double a = (double)dre[q] - mre[q], b = (double)dim[q] - mim[q];
        x = (a * a + b * b) * (double)w[q];
        if (gre) {
            gre[q] = (float)(-2.0 * w[q] * a);
            gim[q] = (float)(-2.0 * w[q] * b);
        }
    }
    sh[threadIdx.x] = x;
    __syncthreads();
    for (int s = CHI_BS / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = sh[0];
}

// fixed-order final sum (deterministic)
__global__ void __launch_bounds__(CHI_BS) k_sum(const double *partial, int n, double *out) {
    __shared__ double sh[CHI_BS];
    double x = 0.0;
    for (int i = threadIdx.x; i < n; i += CHI_BS) x += partial[i];
    sh[threadIdx.x] = x;
    __syncthreads();
    for (int s = CHI_BS / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s) sh[threadIdx.x] += sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}

int vis_run(rt_ctx *ctx, const float *d_img, int nx, int ny, double dxy, const double *d_u,
            const double *d_v, int K, double dra, double ddec, float *d_re, float *d_im) {
    if (nx < 1 || ny < 1 || ny > VIS_MAXROWS || K < 0 || !(dxy > 0))
        return set_err(ctx, RT_E_ARG, "vis: invalid sizes (ny <= %d)", VIS_MAXROWS);
    if (K == 0) return RT_OK;
    if (!d_img || !d_u || !d_v || !d_re || !d_im)
        return set_err(ctx, RT_E_ARG, "vis: NULL image, (u,v) or output");
    // rows split over the waves while that takes no more than one workgroup per CU (256 x
    // 256: 31 against 67 us at 5e3 points, 70 against 69 at 2e4, 142 against 101 at 5e4;
    // 128 x 128: 17 against 20, 35 against 21); up to 64 rows there is one tile of them
    const int nb = (K + 127) / 128;
    if ((K + 31) / 32 <= ctx->n_cu && ny > 64)
        hipLaunchKernelGGL(k_vis<4>, dim3((K + 31) / 32), dim3(VIS_BS), 0, ctx->stream, d_img, nx,
                           ny, d_u, d_v, K, dxy, dra, ddec, d_re, d_im);
    else
        hipLaunchKernelGGL(k_vis<1>, dim3(nb), dim3(VIS_BS), 0, ctx->stream, d_img, nx, ny, d_u,
                           d_v, K, dxy, dra, ddec, d_re, d_im);
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}

// whether calls on this stream are being recorded (or it cannot be told: a capture
// elsewhere that the null stream would join)
static bool capturing(hipStream_t sm) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return !HipMem::ok(hipStreamIsCapturing(sm, &st)) || st != hipStreamCaptureStatusNone;
}

int vis_adjoint_run(rt_ctx *ctx, const float *d_gre, const float *d_gim, int nx, int ny, double dxy,
                    const double *d_u, const double *d_v, int K, double dra, double ddec,
                    float *d_g_img, void *ws) {
    if (nx < 1 || ny < 1 || K < 0 || !(dxy > 0)) return set_err(ctx, RT_E_ARG, "vis adjoint: invalid sizes");
    const hipStream_t sm = ctx->stream;
    const size_t need = vis_adjoint_workspace(ctx, nx, ny, K);
    auto tiled = [&](void *part) {
        const AdjSplit a = adj_split(ctx, nx, ny, K);
        hipLaunchKernelGGL(a.wpc == 3 ? k_vis_adj_part<3> : k_vis_adj_part<2>,
                           dim3(a.tx, a.ty, a.splits), dim3(256), 0, sm, d_gre, d_gim, nx, ny, d_u,
                           d_v, K, dxy, dra, ddec, a.per, (float *)part, d_g_img);
        if (part)
            hipLaunchKernelGGL(k_vis_adj_sum, dim3(a.tx, a.ty, 16), dim3(256), 0, sm,
                               (const float *)part, a.splits, nx, ny, d_g_img);
    };
    bool done = false;
    if (need == 0 ? adj_tiled(nx, ny, K) : ws != nullptr) {
        tiled(need ? ws : nullptr);
        done = true;
    } else if (need > 0 && !capturing(sm)) {
        // (a capture can neither allocate nor wait on an event from outside)
        done = ctx->vis_ws.with(sm, need, tiled);
    }
    if (!done) {
        dim3 grid((nx + ADJ_T - 1) / ADJ_T, (ny + ADJ_T - 1) / ADJ_T);
        hipLaunchKernelGGL(k_vis_adj, grid, dim3(ADJ_BS), 0, sm, d_gre, d_gim, nx, ny, d_u, d_v, K,
                           dxy, dra, ddec, d_g_img);
    }
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}

size_t chisq_workspace(int K) { return (size_t)((K + CHI_BS - 1) / CHI_BS); }

int chisq_run(rt_ctx *ctx, const float *dre, const float *dim, const float *w, const float *mre,
              const float *mim, int K, double *out, float *gre, float *gim, double *ws) {
    if (K < 1 || !out) return set_err(ctx, RT_E_ARG, "chisq: invalid arguments");
    if ((gre == nullptr) != (gim == nullptr)) return set_err(ctx, RT_E_ARG, "chisq: gre/gim both or neither");
    int nb = (int)chisq_workspace(K);
    double *partial = ws;
    if (!partial) HIPCHK(ctx, hipMallocAsync((void **)&partial, sizeof(double) * nb, ctx->stream));
    hipLaunchKernelGGL(k_chisq, dim3(nb), dim3(CHI_BS), 0, ctx->stream, dre, dim, w, mre, mim, K,
                       partial, gre, gim);
    hipLaunchKernelGGL(k_sum, dim3(1), dim3(CHI_BS), 0, ctx->stream, partial, nb, out);
    if (!ws) HIPCHK(ctx, hipFreeAsync(partial, ctx->stream));
    HIPCHK(ctx, hipGetLastError());
    return RT_OK;
}
