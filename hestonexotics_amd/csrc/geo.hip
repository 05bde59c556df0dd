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
// round evaluates the next p0 panels of every unconverged item at once, one workgroup per panel
// (lane q: node q, a recursion over the expiry's grid, a few hundred to a few thousand steps;
// lane i: strike i's panel sum over the 64 nodes in a fixed order), plus E[e^L] in the first round;
// p0 is the host's estimate of where the characteristic function has decayed. Pass 2 gives each
// item one workgroup: lane i adds strike i's panel sums in panel order, keeps them for the next
// round if the decay was not reached, and in the last round evaluates further panels itself;
// every price is therefore the same fixed-order sum whatever p0 is. Runs once per batch, before
// the path kernels.
#include <hip/hip_runtime.h>

#include "cplx_device.hpp"
#include "kernels.hpp"
#include "layout.hpp"
#include "math_f64.hpp"

namespace hexo {
namespace {

constexpr double kPi = 3.14159265358979323846;
// The recursion over an expiry's grid is one chain of steps, and 87 panels (one expiry) leave a wavefront
// alone on its SIMD, where it issues an instruction every 7 cycles or so: 0.9 us a step when one
// wavefront did all of it. Most of a step does not depend on the running B: a is known from the
// weights, and with it beta, d, B-, e and Z below; and log(1 + z) only adds to A. So 7 wavefronts
// prepare the steps of a chunk (one each) and take the logarithms of an earlier one, and the eighth
// runs the rest, B' = B- - (B- - B) e / (1 + z): 35 instructions in place of 500. 252 steps, one
// expiry, 87 panels: 450 -> 106 us for the first pass; 2,000 steps 2.9 -> 0.65 ms; 40 expiries, where
// the chip is full either way, 3.6 -> 2.9 ms.
constexpr int kGeoHelpers = 7;
constexpr int kGeoWaves = kGeoHelpers + 1;

struct GeoShared {
    Cplx pre[2][kGeoHelpers][3][64];  // B-, e, Z of a chunk's steps, lane by lane
    Cplx z[2][kGeoHelpers][64];
    Cplx A[kGeoHelpers][64];
    double node[3][64];  // weighted phi and u of a panel's nodes
    double part[kGeoWaves][64];
    double mag;
};

__device__ __forceinline__ double cabs_(Cplx z) { return hypot(z.re, z.im); }
__device__ __forceinline__ double norm2(Cplx z) { return __builtin_fma(z.re, z.re, z.im * z.im); }
// z / w, inv_w2 = 1 / |w|^2: the operands here are far from the ends of the range
__device__ __forceinline__ Cplx div_by(Cplx z, Cplx w, double inv_w2) { return inv_w2 * (z * conj(w)); }

// phi(s) over points 0..n of pts = (t_j, v_j) pairs, by a whole workgroup, lane by lane; wavefront
// kGeoHelpers returns it.
// With beta = kappa - rho sigma a, d = sqrt(beta^2 - sigma^2 (a^2 - a)), the stable root
// B- = (a^2 - a)/(beta + d) (or (beta - d)/sigma^2 when beta + d is the smaller),
// e = e^{-d tau}, Z = sigma^2 (1 - e) / (2d) and z = Z (B- - B):
//   B(tau) = B- - (B- - B) e / (1 + z),   A(tau) = A + r a tau + kappa theta (B- tau - (2/sigma^2) log(1 + z)).
__device__ Cplx geo_cf(const DevReq& R, const double* pts, uint32_t n, Cplx s, GeoShared& sh, int w, int lane) {
    const double s2 = R.sigma * R.sigma, kth = R.kappa * R.theta, rs = R.rho * R.sigma, kap = R.kappa;
    const double k2 = 2.0 * kth / s2;
    const uint32_t chunks = (n + kGeoHelpers - 1) / kGeoHelpers;
    Cplx A = cx(0.0), B = cx(0.0);
    double S = 0.0;     // sum of the weights from point n down to jn + 1
    uint32_t jn = n;
    if (w == kGeoHelpers) __builtin_amdgcn_s_setprio(2);  // the others wait for it
    for (uint32_t it = 0; it < chunks + 2; ++it) {
        if (w < kGeoHelpers) {
            if (it >= 2 && (it - 2) * kGeoHelpers + w < n) A = A - k2 * clog1p(sh.z[it & 1][w][lane]);
            const uint32_t i = it * kGeoHelpers + w;
            if (i < n) {
                const uint32_t j = n - i;  // the step from point j to j - 1
                for (; jn >= j; --jn) S += pts[2 * jn + 1];
                const double tau = pts[2 * j] - pts[2 * (j - 1)];
                const Cplx a = S * s;
                const Cplx bt = cx(kap) - rs * a;
                const Cplx q = a * a - a;
                // d = principal root of d2, |d|^2 = |d2|
                const Cplx d2 = bt * bt - s2 * q;
                const double r = sqrt(norm2(d2));
                const double t = sqrt(0.5 * (r + fabs(d2.re))), o = r > 0.0 ? 0.5 * div_f64(d2.im, t) : 0.0;
                const Cplx d = d2.re >= 0.0 ? Cplx{t, o} : Cplx{fabs(o), copysign(t, d2.im)};
                const Cplx bp = bt + d, bm = bt - d;
                const double bp2 = norm2(bp);
                const Cplx Bm = bp2 >= norm2(bm) ? div_by(q, bp, div_f64(1.0, bp2)) : (1.0 / s2) * bm;
                const Cplx om = -1.0 * cexpm1(-tau * d);
                A = A + (R.r_drift * tau) * a + (kth * tau) * Bm;
                sh.pre[it & 1][w][0][lane] = Bm;
                sh.pre[it & 1][w][1][lane] = cx(1.0) - om;
                sh.pre[it & 1][w][2][lane] = div_by((0.5 * s2) * om, d, div_f64(1.0, r));
            }
        } else if (it >= 1 && it <= chunks) {
            const uint32_t m = min((uint32_t)kGeoHelpers, n - (it - 1) * kGeoHelpers);
#pragma unroll
            for (uint32_t h = 0; h < (uint32_t)kGeoHelpers; ++h) {
                if (h < m) {
                    const Cplx Bm = sh.pre[(it - 1) & 1][h][0][lane];
                    const Cplx y = Bm - B, z = sh.pre[(it - 1) & 1][h][2][lane] * y;
                    const Cplx v = cx(1.0 + z.re, z.im);
                    sh.z[(it - 1) & 1][h][lane] = z;
                    B = Bm - div_by(y * sh.pre[(it - 1) & 1][h][1][lane], v, div_f64(1.0, norm2(v)));
                }
            }
        }
        __syncthreads();
    }
    if (w < kGeoHelpers) sh.A[w][lane] = A;
    __syncthreads();
    if (w < kGeoHelpers) return cx(0.0);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int h = 0; h < kGeoHelpers; ++h) A = A + sh.A[h][lane];
    return cexp(A + R.v0 * B);
}

__device__ __forceinline__ double wave_max(double x) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) x = fmax(x, __shfl_xor(x, m));
    return x;  // every lane holds the wave's maximum
}

// Panel p of an item, by one workgroup: lane q evaluates node q, u_q = (p + (x_q + 1)/2) h, and
// phi(1/2 - i u_q) weighted by w_q (h/2) / (u_q^2 + 1/4); then each wavefront sums
// Re(e^{i u_q k_i} weighted phi) over 8 nodes for every strike i, and wavefront kGeoHelpers adds and
// returns the eight sums in order, with the maximum of |phi| over the panel in *mag. Up to 32 strikes
// are taken eight at a time, a lane per strike and node, the nodes added by a fixed tree: a lane per
// strike that goes through the nodes has eight sine-cosine pairs for one strike too, most of the
// time of a panel of a short grid (324 items of 2 steps and a strike 1,007 -> 819 us). With more it
// saves less than the exchanges cost (222 items of 28 steps, whole call: 21 strikes 3,788 -> 3,708 us, 40
// strikes 3,868 -> 3,892).
// Panel 0 holds the integrand's 1/(u^2 + 1/4) peak at u = 0, which 64 nodes integrate to 1e-13
// over [0, 16] but only to 1e-4 over [0, 120]: it is summed as n_sub = min(64, ceil(h / 16))
// sub-panels of 64 nodes (wave-uniform, in order). The other panels keep width h.
__device__ __forceinline__ uint32_t first_panel_parts(double h) {
    return (uint32_t)fmin(64.0, ceil(h / 16.0));
}

__device__ double panel_sum(const GeoArgs& a, const DevGeo& G, const DevReq& R, const double* pts, uint32_t p, int w,
                            int lane, double k, bool has_k, GeoShared& sh, double* mag) {
    const uint32_t n_sub = p == 0 ? first_panel_parts(G.h) : 1u;
    const double hs = G.h / (double)n_sub;
    constexpr int kNodes = 64 / kGeoWaves;  // per wavefront
    constexpr uint32_t kTreeStrikes = 32;
    double sum = 0.0, mg = 0.0;
    for (uint32_t j = 0; j < n_sub; ++j) {
        const double u = ((double)(p + j) + 0.5 * (a.gl[lane] + 1.0)) * hs;  // p = 0 or j = 0
        const Cplx ph = geo_cf(R, pts, G.n_pts, cx(0.5, -u), sh, w, lane);  // ends the use of node and part before
        if (w == kGeoHelpers) {
            const double f = 0.5 * hs * a.gl[64 + lane] / (u * u + 0.25);
            sh.node[0][lane] = f * ph.re;
            sh.node[1][lane] = f * ph.im;
            sh.node[2][lane] = u;
            mg = fmax(mg, wave_max(cabs_(ph)));
        }
        __syncthreads();
        if (G.n_strikes > kTreeStrikes) {
            double part = 0.0;
            if (has_k) {
                for (int q = w * kNodes; q < (w + 1) * kNodes; ++q) {
                    double sn, cs;
                    sincos(sh.node[2][q] * k, &sn, &cs);
                    part += cs * sh.node[0][q] - sn * sh.node[1][q];
                }
            }
            sh.part[w][lane] = part;
        } else {
            const int q = w * kNodes + lane % kNodes;
            for (int i = lane / kNodes; i - lane / kNodes < (int)G.n_strikes; i += 64 / kNodes) {
                const double ki = __shfl(k, i);
                double sn, cs;
                sincos(sh.node[2][q] * ki, &sn, &cs);
                double part = cs * sh.node[0][q] - sn * sh.node[1][q];
#pragma unroll
                for (int m = 1; m < kNodes; m <<= 1) part += __shfl_xor(part, m);
                if (lane % kNodes == 0) sh.part[w][i] = part;
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

// Pass 1 of round r: every workgroup evaluates one panel of one unconverged item (round r covers
// that item's panels done .. done + p0 - 1) and stores each strike's panel sum; in the first round the
// item's last workgroup evaluates E[e^L] instead.
// The grid is items x panels, without those past an item's p0: found from a prefix sum over the items, a
// workgroup's item cost it nine dependent loads at 324 items. Item by item, or where all grids are short
// panel by panel, so that the first panels, which take longest, begin first: 324 items of 2, 6, 12,
// 24, 52, 252 steps 913/831, 1,103/1,076, 1,314/1,298, 1,744/1,764, 2,971/3,001, 10,864/11,534 us.
constexpr uint32_t kShortGrid = 16;     // points
constexpr uint32_t kGridItems = 65535;  // the most blocks in y and z of a grid
__global__ __launch_bounds__(64 * kGeoWaves) void k_geo_panels(GeoArgs a, uint32_t round) {
    __shared__ GeoShared sh;
    const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63u);
    const bool panels_first = a.max_pts <= kShortGrid;
    const uint32_t item = panels_first ? blockIdx.x : blockIdx.z * kGridItems + blockIdx.y;
    const uint32_t j = panels_first ? blockIdx.y : blockIdx.x;
    if (item >= a.n_items) return;
    const DevGeo& G = a.items[item];
    if (j > G.p0) return;
    const uint32_t wv = G.wave_begin + j;
    const DevReq& R = a.reqs[G.req];
    const double* pts = a.pts + 2 * (size_t)G.pts_begin;
    const double* st = a.state + (size_t)item * kGeoState;
    uint32_t base = 0;
    if (round > 0) {
        if (j == G.p0 || st[66] != 0.0) return;  // E[e^L] is known; or the item has converged
        base = (uint32_t)st[65];
    } else if (j == G.p0) {
        const Cplx e1 = geo_cf(R, pts, G.n_pts, cx(1.0), sh, w, lane);
        if (w == kGeoHelpers && lane == 0) a.panel_max[wv] = e1.re;
        return;
    }
    const uint32_t p = base + j;
    if (p >= G.max_panels) return;
    double K, k, mag;
    bool has_k;
    strike_of(a, G, lane, K, k, has_k);
    const double sum = panel_sum(a, G, R, pts, p, w, lane, k, has_k, sh, &mag);
    if (w != kGeoHelpers) return;
    a.panel[(size_t)wv * 64 + (uint32_t)lane] = sum;
    if (lane == 0) a.panel_max[wv] = mag;
}

// Pass 2 of round r: one workgroup per item; lane i of wavefront kGeoHelpers adds strike i's panel sums in panel order up
// to the second of the first two consecutive panels (after the first) whose |phi| stays below
// 1e-15 u0, u0 a panel's start: beyond u0 the integrand |phi| / (u^2 + 1/4) leaves at most
// sup|phi| / u0 to the integral, and two panels in a row guard against a dip of a non-monotone
// |phi|. An unconverged item keeps its sums for the next round; in the last round the workgroup
// evaluates further panels itself. Nearly all converge in the first round, and the host reads the
// prices back before it runs the paths: it launches the other rounds only where a price is
// kGeoUnfinished (four empty launches were 19 us of a request's 355). The price is the same ordered sum whatever p0 and the number of
// rounds are.
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
    const double e1 = round == 0 ? a.panel_max[G.wave_begin + G.p0] : st[64];  // E[e^L]
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
        integ += a.panel[(size_t)(G.wave_begin + j) * 64 + (uint32_t)lane];
        const bool now = p > 0 && a.panel_max[G.wave_begin + j] < 1e-15 * (double)p * G.h;
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
        const uint32_t per_item = a.max_p0 + 1;
        const dim3 grid = a.max_pts <= kShortGrid ? dim3(a.n_items, per_item)
                                                  : dim3(per_item, a.n_items < kGridItems ? a.n_items : kGridItems,
                                                         (a.n_items + kGridItems - 1) / kGridItems);
        k_geo_panels<<<grid, 64 * kGeoWaves, 0, st>>>(a, r);
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
        k_geo_sum<<<a.n_items, 64 * kGeoWaves, 0, st>>>(a, r);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace hexo
