// geo.hip -- exact price of the geometric control variate of the Asian call, FP64 on gfx950.
//
// For an expiry's Asian functional A = sum_j w_j X_{t_j} (weights from the run schedule, sum W)
// the control variate is G = c e^L with c = W S0 and L = sum_j v_j ln(X_{t_j}/S0), v = w / W.
// Under the Heston model
//   phi(s) = E[e^{sL}] = exp(A_0 + B_0 v0)
// by a backward recursion over the grid points: at t_j the log-price coefficient a grows by s v_j;
// over (t_{j-1}, t_j] the Riccati equations of exp(A + a y + B V),
//   B' = sigma^2 B^2 / 2 + (rho sigma a - kappa) B + (a^2 - a) / 2,   A' = kappa theta B + r a,
// are solved in closed form from the running B (no cancellation as sigma -> 0, see geo_cf).
// The call price is Lewis' inversion
//   E[(c e^L - K)^+] = c (phi(1) - e^{k/2}/pi int_0^inf Re(e^{iuk} phi(1/2 - iu)) / (u^2 + 1/4) du),
// k = ln(K / c), by 64-node Gauss-Legendre panels of width h (host-chosen from the scale of L and
// the strikes) until the characteristic function has decayed below 1e-15 u0 on a whole panel
// starting at u0 (the integral's remaining tail is then below 1e-15).
//
// Work items are (request, expiry, block of <= 64 strikes), in up to three rounds. Pass 1 of a
// round evaluates the next p0 panels of every unconverged item at once, one workgroup or, where
// there are enough of them, one wavefront per panel (lane q: node q, a recursion over the expiry's grid,
// a few hundred to a few thousand steps; lane i: strike i's panel sum over the 64 nodes in a
// fixed order), plus E[e^L] in the first round;
// p0 is the host's estimate of where the characteristic function has decayed. Pass 2 gives each
// item one workgroup: lane i adds strike i's panel sums in panel order, keeps them for the next
// round if the decay was not reached, and in the last round evaluates further panels itself;
// every price is therefore the same fixed-order sum whatever p0 is. Runs once per batch, before
// the path kernels.
#include <hip/hip_runtime.h>

// Products are fused within an expression only, by the front end: two kernels evaluate the same panels
// and have to agree in every bit.
#pragma clang fp contract(on)

#include "cplx_device.hpp"
#include "kernels.hpp"
#include "layout.hpp"
#include "math_f64.hpp"

namespace hexo {
namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kGeoHelpers = 7;
constexpr int kGeoWaves = kGeoHelpers + 1;

struct GeoShared {
    Cplx pre[2][kGeoHelpers][3][64];  // B-, e, Z of a chunk's steps, lane by lane
    Cplx z[2][kGeoHelpers][64];
    Cplx A[2][kGeoHelpers][64];
    double node[3][64];  // weighted phi and u of a panel's nodes
    double part[kGeoWaves][64];
    double mag;
};

struct GeoWaveShared {
    Cplx A[2][kGeoHelpers][64];
    double node[3][64];
};

__device__ __forceinline__ double cabs_(Cplx z) { return hypot(z.re, z.im); }
__device__ __forceinline__ double norm2(Cplx z) { return __builtin_fma(z.re, z.re, z.im * z.im); }
// z / w, inv_w2 = 1 / |w|^2: the operands here are far from the ends of the range
__device__ __forceinline__ Cplx div_by(Cplx z, Cplx w, double inv_w2) { return inv_w2 * (z * conj(w)); }

// phi(s) over points 0..n of pts = (t_j, v_j) pairs, lane by lane.
// With beta = kappa - rho sigma a, d = sqrt(beta^2 - sigma^2 (a^2 - a)), the stable root
// B- = (a^2 - a)/(beta + d) (or (beta - d)/sigma^2 when beta + d is the smaller),
// e = e^{-d tau}, Z = sigma^2 (1 - e) / (2d) and z = Z (B- - B):
//   B(tau) = B- - (B- - B) e / (1 + z),   A(tau) = A + r a tau + kappa theta (B- tau - (2/sigma^2) log(1 + z)).
// A's sums, the logarithms apart, run over every seventh step: a helper's below.
//
// What of a step does not depend on the running B; its part of A but for the logarithm is added to dA.
struct GeoStep {
    Cplx Bm, e, Z;
};
struct GeoModel {
    double kappa, kth, rs, s2, r;
    __device__ explicit GeoModel(const DevReq& R)
        : kappa(R.kappa), kth(R.kappa * R.theta), rs(R.rho * R.sigma), s2(R.sigma * R.sigma), r(R.r_drift) {}
};
__device__ __forceinline__ GeoStep geo_prepare(const GeoModel& M, double tau, Cplx a, Cplx& dA) {
    const double s2 = M.s2;
    const Cplx bt = cx(__builtin_fma(-M.rs, a.re, M.kappa), -M.rs * a.im);
    const Cplx q = a * a - a, bt2 = bt * bt;
    // d = principal root of d2, |d|^2 = |d2|
    const Cplx d2 = cx(__builtin_fma(-s2, q.re, bt2.re), __builtin_fma(-s2, q.im, bt2.im));
    const double r = sqrt(norm2(d2));
    const double t = sqrt(0.5 * (r + fabs(d2.re))), o = r > 0.0 ? 0.5 * div_f64(d2.im, t) : 0.0;
    const Cplx d = d2.re >= 0.0 ? Cplx{t, o} : Cplx{fabs(o), copysign(t, d2.im)};
    const Cplx bp = bt + d, bm = bt - d;
    const double bp2 = norm2(bp);
    GeoStep p;
    p.Bm = bp2 >= norm2(bm) ? div_by(q, bp, div_f64(1.0, bp2)) : (1.0 / s2) * bm;
    const Cplx x = cexpm1(-tau * d);  // e - 1
    p.e = cx(1.0 + x.re, x.im);
    p.Z = (-0.5 * s2 * div_f64(1.0, r)) * (x * conj(d));
    const double ra = M.r * tau, kt = M.kth * tau;
    dA = cx(__builtin_fma(kt, p.Bm.re, __builtin_fma(ra, a.re, dA.re)),
            __builtin_fma(kt, p.Bm.im, __builtin_fma(ra, a.im, dA.im)));
    return p;
}
// B over the step; returns z.
__device__ __forceinline__ Cplx geo_advance(Cplx Bm, Cplx e, Cplx Z, Cplx& B) {
    const Cplx y = Bm - B, z = Z * y;
    const Cplx v = cx(__builtin_fma(Z.re, y.re, __builtin_fma(-Z.im, y.im, 1.0)), z.im);
    const double inv = div_f64(1.0, norm2(v));
    const Cplx t = (y * e) * conj(v);
    B = Cplx{__builtin_fma(-inv, t.re, Bm.re), __builtin_fma(-inv, t.im, Bm.im)};
    return z;
}
// A: the helpers' sums of dA, then of the logarithms.
__device__ __forceinline__ Cplx geo_phi(const DevReq& R, const Cplx (&A)[2][kGeoHelpers][64], Cplx B,
                                        int lane) {
    const double k2 = 2.0 * R.kappa * R.theta / (R.sigma * R.sigma);
    Cplx dA = cx(0.0), lg = cx(0.0);
#pragma unroll
    for (int h = 0; h < kGeoHelpers; ++h) {
        dA = dA + A[0][h][lane];
        lg = lg + A[1][h][lane];
    }
    return cexp((dA - k2 * lg) + R.v0 * B);
}

// By a wavefront, the sums of a lane in LDS: at 250 registers two wavefronts share a SIMD, and a batch
// with panels enough to fill them needs no helpers to wait for (324 items of 2 steps 972 -> 200 us, of
// 252 steps 11.3 -> 7.7 ms against a workgroup per panel; the rule is in engine.cpp).
__device__ Cplx geo_cf_wave(const DevReq& R, const double* pts, uint32_t n, Cplx s,
                            Cplx (&A)[2][kGeoHelpers][64], int lane) {
#pragma unroll
    for (int h = 0; h < kGeoHelpers; ++h) A[0][h][lane] = A[1][h][lane] = cx(0.0);
    const GeoModel M(R);
    Cplx B = cx(0.0);
    double S = 0.0;  // sum of the weights from point n down
    uint32_t h = 0;
    for (uint32_t j = n; j > 0; --j) {
        S += pts[2 * j + 1];
        Cplx dA = A[0][h][lane];
        const GeoStep p = geo_prepare(M, pts[2 * j] - pts[2 * (j - 1)], S * s, dA);
        A[0][h][lane] = dA;
        A[1][h][lane] = A[1][h][lane] + clog1p(geo_advance(p.Bm, p.e, p.Z, B));
        h = h + 1 == kGeoHelpers ? 0 : h + 1;
    }
    return geo_phi(R, A, B, lane);
}

// By a workgroup; wavefront kGeoHelpers returns it. The recursion over an expiry's grid is one chain of
// steps, and 87 panels (one expiry) leave a wavefront alone on its SIMD, where it issues an instruction
// every 7 cycles or so: 0.9 us a step when one wavefront did all of it. Most of a step does not depend on
// the running B. So 7 wavefronts prepare the steps of a chunk (one each) and take the logarithms of an
// earlier one, and the eighth runs the rest: 35 instructions in place of 500. 252 steps, one expiry, 87
// panels: 450 -> 105 us for the first pass; 2,000 steps 2.9 -> 0.65 ms.
__device__ Cplx geo_cf(const DevReq& R, const double* pts, uint32_t n, Cplx s, GeoShared& sh, int w, int lane) {
    const uint32_t chunks = (n + kGeoHelpers - 1) / kGeoHelpers;
    const GeoModel M(R);
    Cplx dA = cx(0.0), lg = cx(0.0), B = cx(0.0);
    double S = 0.0;     // sum of the weights from point n down to jn + 1
    uint32_t jn = n;
    if (w == kGeoHelpers) __builtin_amdgcn_s_setprio(2);  // the others wait for it
    for (uint32_t it = 0; it < chunks + 2; ++it) {
        if (w < kGeoHelpers) {
            if (it >= 2 && (it - 2) * kGeoHelpers + w < n) lg = lg + clog1p(sh.z[it & 1][w][lane]);
            const uint32_t i = it * kGeoHelpers + w;
            if (i < n) {
                const uint32_t j = n - i;  // the step from point j to j - 1
                for (; jn >= j; --jn) S += pts[2 * jn + 1];
                const GeoStep p = geo_prepare(M, pts[2 * j] - pts[2 * (j - 1)], S * s, dA);
                sh.pre[it & 1][w][0][lane] = p.Bm;
                sh.pre[it & 1][w][1][lane] = p.e;
                sh.pre[it & 1][w][2][lane] = p.Z;
            }
        } else if (it >= 1 && it <= chunks) {
            const uint32_t m = min((uint32_t)kGeoHelpers, n - (it - 1) * kGeoHelpers);
#pragma unroll
            for (uint32_t h = 0; h < (uint32_t)kGeoHelpers; ++h) {
                if (h < m) {
                    const auto& pre = sh.pre[(it - 1) & 1][h];
                    sh.z[(it - 1) & 1][h][lane] = geo_advance(pre[0][lane], pre[1][lane], pre[2][lane], B);
                }
            }
        }
        __syncthreads();
    }
    if (w < kGeoHelpers) {
        sh.A[0][w][lane] = dA;
        sh.A[1][w][lane] = lg;
    }
    __syncthreads();
    if (w < kGeoHelpers) return cx(0.0);
    __builtin_amdgcn_s_setprio(0);
    return geo_phi(R, sh.A, B, lane);
}

__device__ __forceinline__ void wave_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wave_max(double x) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) x = fmax(x, __shfl_xor(x, m));
    return x;  // every lane holds the wave's maximum
}

// A panel's sums. Node q, u_q = (p + (x_q + 1)/2) h, has phi(1/2 - i u_q) weighted by
// w_q (h/2) / (u_q^2 + 1/4); strike i's Re(e^{i u_q k_i} weighted phi) is summed over parts of 8 nodes,
// and the eight parts are added in order. Up to 32 strikes are taken eight at a time, a lane per strike
// and node of a part, whose nodes are added by a fixed tree: a lane per strike that goes through the nodes
// has eight sine-cosine pairs for one strike too, most of the time of a panel of a short grid (324
// items of 2 steps and a strike 1,007 -> 819 us). With more it saves less than the exchanges cost (222
// items of 28 steps, whole call: 21 strikes 3,788 -> 3,708 us, 40 strikes 3,868 -> 3,892).
//
// Panel 0 holds the integrand's 1/(u^2 + 1/4) peak at u = 0, which 64 nodes integrate to 1e-13
// over [0, 16] but only to 1e-4 over [0, 120]: it is summed as n_sub = min(64, ceil(h / 16))
// sub-panels of 64 nodes (wave-uniform, in order). The other panels keep width h.
constexpr int kPartNodes = 8;
constexpr uint32_t kTreeStrikes = 32;

__device__ __forceinline__ uint32_t first_panel_parts(double h) {
    return (uint32_t)fmin(64.0, ceil(h / 16.0));
}

// The panel's nodes as (Re, Im of the weighted phi, u), one a lane.
__device__ __forceinline__ double node_u(const GeoArgs& a, uint32_t panel, double h, int lane) {
    return ((double)panel + 0.5 * (a.gl[lane] + 1.0)) * h;
}
__device__ __forceinline__ void store_node(const GeoArgs& a, double (&node)[3][64], Cplx phi, double u,
                                           double h, int lane) {
    const double f = 0.5 * h * a.gl[64 + lane] / (u * u + 0.25);
    node[0][lane] = f * phi.re;
    node[1][lane] = f * phi.im;
    node[2][lane] = u;
}
__device__ __forceinline__ double node_value(const double (&node)[3][64], int q, double k) {
    double sn, cs;
    sincos(node[2][q] * k, &sn, &cs);
    return cs * node[0][q] - sn * node[1][q];
}
// Part v for the strike of the lane: in every one of its eight lanes with the tree, else in lane i.
__device__ __forceinline__ double tree_part(const double (&node)[3][64], int v, double k, int lane) {
    double part = node_value(node, v * kPartNodes + lane % kPartNodes, k);
#pragma unroll
    for (int m = 1; m < kPartNodes; m <<= 1) part += __shfl_xor(part, m);
    return part;
}
__device__ __forceinline__ double lane_part(const double (&node)[3][64], int v, double k) {
    double part = 0.0;
    for (int q = v * kPartNodes; q < (v + 1) * kPartNodes; ++q) part += node_value(node, q, k);
    return part;
}

// Panel p of an item by a workgroup, a part each wavefront; lane i of wavefront kGeoHelpers returns strike
// i's sum, and the maximum of |phi| over the panel in *mag.
__device__ double panel_sum(const GeoArgs& a, const DevGeo& G, const DevReq& R, const double* pts, uint32_t p, int w,
                            int lane, double k, bool has_k, GeoShared& sh, double* mag) {
    static_assert(kGeoWaves * kPartNodes == 64, "a part per wavefront");
    const uint32_t n_sub = p == 0 ? first_panel_parts(G.h) : 1u;
    const double hs = G.h / (double)n_sub;
    double sum = 0.0, mg = 0.0;
    for (uint32_t j = 0; j < n_sub; ++j) {
        const double u = node_u(a, p + j, hs, lane);  // p = 0 or j = 0
        const Cplx ph = geo_cf(R, pts, G.n_pts, cx(0.5, -u), sh, w, lane);  // ends the use of node and part before
        if (w == kGeoHelpers) {
            store_node(a, sh.node, ph, u, hs, lane);
            mg = fmax(mg, wave_max(cabs_(ph)));
        }
        __syncthreads();
        if (G.n_strikes > kTreeStrikes) {
            sh.part[w][lane] = lane_part(sh.node, w, k);
        } else {
            for (uint32_t i0 = 0; i0 < G.n_strikes; i0 += 8) {
                const int i = (int)i0 + lane / kPartNodes;
                const double part = tree_part(sh.node, w, __shfl(k, i), lane);
                if (lane % kPartNodes == 0) sh.part[w][i] = part;
            }
        }
        __syncthreads();
        if (w == kGeoHelpers && has_k) {
#pragma unroll
            for (int v = 0; v < kGeoWaves; ++v) sum += sh.part[v][lane];
        }
    }
    *mag = mg;
    return sum;
}

// By a wavefront, the same bits.
__device__ double panel_sum_wave(const GeoArgs& a, const DevGeo& G, const DevReq& R, const double* pts, uint32_t p,
                                 int lane, double k, bool has_k, GeoWaveShared& sh, double* mag) {
    const uint32_t n_sub = p == 0 ? first_panel_parts(G.h) : 1u;
    const double hs = G.h / (double)n_sub;
    double sum = 0.0, mg = 0.0;
    for (uint32_t j = 0; j < n_sub; ++j) {
        const double u = node_u(a, p + j, hs, lane);
        const Cplx ph = geo_cf_wave(R, pts, G.n_pts, cx(0.5, -u), sh.A, lane);
        wave_sync_lds();  // the last sub-panel's nodes have been read
        store_node(a, sh.node, ph, u, hs, lane);
        mg = fmax(mg, wave_max(cabs_(ph)));
        wave_sync_lds();
        if (G.n_strikes > kTreeStrikes) {
            if (has_k)
                for (int v = 0; v < kGeoWaves; ++v) sum += lane_part(sh.node, v, k);
        } else {
            for (uint32_t i0 = 0; i0 < G.n_strikes; i0 += 8) {
                const int i = (int)i0 + lane / kPartNodes;
                const double ki = __shfl(k, i);
                double t = __shfl(sum, i);
                for (int v = 0; v < kGeoWaves; ++v) t += tree_part(sh.node, v, ki, lane);
                t = __shfl(t, lane % 8 * kPartNodes);  // strike i0 + lane % 8's
                if ((uint32_t)lane / 8u == i0 / 8u && has_k) sum = t;
            }
        }
    }
    *mag = mg;
    return sum;
}

__device__ __forceinline__ void strike_of(const GeoArgs& a, const DevGeo& G, int lane, double& K, double& k,
                                          bool& has_k) {
    const bool in = (uint32_t)lane < G.n_strikes;
    K = in ? a.opts[G.opt + (uint32_t)lane].k_abs : 0.0;
    has_k = K > 0.0;  // K <= 0: max(G - K, 0) = G - K needs no integral
    k = has_k ? log(K / G.c) : 0.0;
}

// Per-item state between rounds (kGeoState doubles): each strike's integral so far, E[e^L], the
// panels summed so far, whether the sum has converged and whether the last panel summed was below
// the stop rule's bound.
constexpr int kGeoState = 64 + 4;
constexpr int kGeoRounds = 3;  // parallel rounds of p0 panels before the serial continuation

// Pass 1 of round r: every workgroup (k_geo_panels) or wavefront (k_geo_panels_wave) evaluates one panel
// of one unconverged item (round r covers that item's panels done .. done + p0 - 1) and stores each
// strike's panel sum; in the first round the item's last one evaluates E[e^L] instead.
// The grid is items x panels, without those past an item's p0: found from a prefix sum over the items, a
// workgroup's item cost it nine dependent loads at 324 items. z and y: the items, x: the panels.
constexpr uint32_t kGridItems = 65535;  // the most blocks in y and z of a grid
struct PanelWork {
    uint32_t item, p;
    size_t slot;  // in panel and panel_max
    bool e1;      // E[e^L]
    bool none;
};
__device__ __forceinline__ PanelWork panel_work(const GeoArgs& a, uint32_t round, uint32_t j) {
    PanelWork k{blockIdx.z * kGridItems + blockIdx.y, j, 0, false, true};
    if (k.item >= a.n_items) return k;
    const DevGeo& G = a.items[k.item];
    if (j > G.p0) return k;
    k.slot = (size_t)G.slot_begin + j;
    k.e1 = j == G.p0;
    if (round > 0) {
        const double* st = a.state + (size_t)k.item * kGeoState;
        if (k.e1 || st[66] != 0.0) return k;  // E[e^L] is known; or the item has converged
        k.p += (uint32_t)st[65];
    }
    k.none = !k.e1 && k.p >= G.max_panels;
    return k;
}

__global__ __launch_bounds__(64 * kGeoWaves) void k_geo_panels(GeoArgs a, uint32_t round) {
    __shared__ GeoShared sh;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const PanelWork job = panel_work(a, round, blockIdx.x);
    if (job.none) return;
    const DevGeo& G = a.items[job.item];
    const DevReq& R = a.reqs[G.req];
    const double* pts = a.pts + 2 * (size_t)G.pts_begin;
    if (job.e1) {
        const Cplx e1 = geo_cf(R, pts, G.n_pts, cx(1.0), sh, w, lane);
        if (w == kGeoHelpers && lane == 0) a.panel_max[job.slot] = e1.re;
        return;
    }
    double K, k, mag;
    bool has_k;
    strike_of(a, G, lane, K, k, has_k);
    const double sum = panel_sum(a, G, R, pts, job.p, w, lane, k, has_k, sh, &mag);
    if (w != kGeoHelpers) return;
    a.panel[job.slot * 64 + (uint32_t)lane] = sum;
    if (lane == 0) a.panel_max[job.slot] = mag;
}

// (248 registers, two wavefronts a SIMD; three or four spill 35 values.)
constexpr int kPanelWaves = 4;
__global__ __launch_bounds__(64 * kPanelWaves, 2) void k_geo_panels_wave(GeoArgs a, uint32_t round) {
    __shared__ GeoWaveShared sh[kPanelWaves];
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const PanelWork job = panel_work(a, round, blockIdx.x * kPanelWaves + (uint32_t)w);
    if (job.none) return;  // whole wavefronts, which share nothing
    const DevGeo& G = a.items[job.item];
    const DevReq& R = a.reqs[G.req];
    const double* pts = a.pts + 2 * (size_t)G.pts_begin;
    if (job.e1) {
        const Cplx e1 = geo_cf_wave(R, pts, G.n_pts, cx(1.0), sh[w].A, lane);
        if (lane == 0) a.panel_max[job.slot] = e1.re;
        return;
    }
    double K, k, mag;
    bool has_k;
    strike_of(a, G, lane, K, k, has_k);
    const double sum = panel_sum_wave(a, G, R, pts, job.p, lane, k, has_k, sh[w], &mag);
    a.panel[job.slot * 64 + (uint32_t)lane] = sum;
    if (lane == 0) a.panel_max[job.slot] = mag;
}

// Pass 2 of round r: one workgroup per item; lane i of wavefront kGeoHelpers adds strike i's panel sums in
// panel order up to the second of the first two consecutive panels (after the first) whose |phi| stays
// below 1e-15 u0, u0 a panel's start: beyond u0 the integrand |phi| / (u^2 + 1/4) leaves at most
// sup|phi| / u0 to the integral, and two panels in a row guard against a dip of a non-monotone
// |phi|. An unconverged item keeps its sums for the next round; in the last round the workgroup
// evaluates further panels itself. Nearly all converge in the first round, and the host reads the
// prices back before it runs the paths: it launches the other rounds only where a price is
// kGeoUnfinished (four empty launches were 19 us of a request's 355). The price is the same ordered sum
// whatever p0 and the number of rounds are.
__global__ __launch_bounds__(64 * kGeoWaves) void k_geo_sum(GeoArgs a, uint32_t round) {
    __shared__ GeoShared sh;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const uint32_t item = blockIdx.x;
    const DevGeo& G = a.items[item];
    const DevReq& R = a.reqs[G.req];
    const double* pts = a.pts + 2 * (size_t)G.pts_begin;
    double* st = a.state + (size_t)item * kGeoState;
    // every wavefront follows the same decisions; all have read the state before it is written
    const bool done = round > 0 && st[66] != 0.0;
    const double e1 = round == 0 ? a.panel_max[G.slot_begin + G.p0] : st[64];  // E[e^L]
    double integ = round == 0 ? 0.0 : st[lane];
    const uint32_t base = round == 0 ? 0u : (uint32_t)st[65];
    bool below = round == 0 ? false : st[67] != 0.0;  // the previous panel was below the bound
    __syncthreads();
    if (done) return;
    double K, k;
    bool has_k;
    strike_of(a, G, lane, K, k, has_k);
    bool converged = false;
    uint32_t p = base;
    for (uint32_t j = 0; j < G.p0 && p < G.max_panels && !converged; ++j, ++p) {
        integ += a.panel[(size_t)(G.slot_begin + j) * 64 + (uint32_t)lane];
        const bool now = p > 0 && a.panel_max[G.slot_begin + j] < 1e-15 * (double)p * G.h;
        converged = now && below;
        below = now;
    }
    const bool last = round + 1 == kGeoRounds;
    if (!converged && !last && p < G.max_panels) {
        if (w != kGeoHelpers) return;
        st[lane] = integ;
        if ((uint32_t)lane < G.n_strikes) a.geo[G.out + (uint64_t)lane] = kGeoUnfinished;
        if (lane == 0) {
            st[64] = e1;
            st[65] = (double)p;
            st[66] = 0.0;
            st[67] = below ? 1.0 : 0.0;
        }
        return;
    }
    for (; p < G.max_panels && !converged; ++p) {
        double mag;
        integ += panel_sum(a, G, R, pts, p, w, lane, k, has_k, sh, &mag);
        if (w == kGeoHelpers && lane == 0) sh.mag = mag;
        __syncthreads();
        const bool now = p > 0 && sh.mag < 1e-15 * (double)p * G.h;  // rewritten after the next panel's barriers
        converged = now && below;
        below = now;
    }
    if (w != kGeoHelpers) return;
    if (lane == 0) st[66] = 1.0;  // later rounds skip the item
    if ((uint32_t)lane >= G.n_strikes) return;
    double price;
    if (!converged)
        price = __builtin_nan("");
    else if (has_k)
        price = G.c * (e1 - exp(0.5 * k) / kPi * integ);
    else
        price = G.c * e1 - K;  // max(G - K, 0) = G - K
    a.geo[G.out + (uint64_t)lane] = price;
}

}  // namespace

size_t geo_state_doubles(uint32_t n_items) { return (size_t)n_items * kGeoState; }

hipError_t launch_geo(const GeoArgs& a, bool first, hipStream_t st) {
    if (a.n_items == 0) return hipSuccess;
    for (uint32_t r = first ? 0u : 1u; r < (first ? 1u : (uint32_t)kGeoRounds); ++r) {
        const uint32_t per_item = a.max_p0 + 1, rows = a.n_items < kGridItems ? a.n_items : kGridItems;
        const uint32_t layers = (a.n_items + kGridItems - 1) / kGridItems;
        if (a.by_wave)
            k_geo_panels_wave<<<dim3((per_item + kPanelWaves - 1) / kPanelWaves, rows, layers),
                                64 * kPanelWaves, 0, st>>>(a, r);
        else
            k_geo_panels<<<dim3(per_item, rows, layers), 64 * kGeoWaves, 0, st>>>(a, r);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        k_geo_sum<<<a.n_items, 64 * kGeoWaves, 0, st>>>(a, r);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace hexo
