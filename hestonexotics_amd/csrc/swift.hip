// swift.hip -- SWIFT European pricer on gfx950, FP64 throughout.
//
// The Shannon-wavelet (SWIFT) method of the reference (src/SWIFT.cpp:18-118): payoff
// coefficients of the call on the truncated log-price range, two Fourier transforms to the
// density coefficients c_j, then price = Re sum_j chf(u_j) c_j e^{-rT} K e^{-i u_j x} with
// x = rT + log(S/K) (src/SWIFT.cpp:102-117). The reference uses FFTW for the transforms and
// Eigen for the final 6 x J by J x K product.
//
// A call is three kernels and one wait: k_swift_transform takes each chain from its inputs to its
// density coefficients in one workgroup (the dynamic grid, the payoff coefficients and both
// transforms in LDS), k_swift_chf forms the pricing matrix, k_swift_sum contracts it with the strikes.
// Chains whose transforms exceed the LDS (J > kSwiftFftMaxJ) get their grid only and go
// through direct sums (one wavefront per output) between the same outer stages.
//
// Gradients (SWIFT::price_opts_grad, the calibration Jacobian) come from the same
// characteristic-function expression evaluated in forward-mode dual arithmetic carrying all five
// parameter directions, instead of hand-derived partials (src/HDistribution.cpp:47-84).
//
// Long maturities with high vol-of-vol truncate the log-price at 14-16, and payoff coefficients of
// size S e^upper cancel in the transforms and in the sum: two evaluations that round differently
// anywhere agree to eps S e^upper only. The stages therefore keep one order of operations (radix-2
// butterflies in time, sums over j in 16 phases, phases re-evaluated every 16 steps).
#include "swift.hpp"
#include "swift_grid.hpp"
#include "cplx_device.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>

namespace hexo {
namespace {

constexpr double kPi = 3.14159265358979323846;

// Plain complex versions of the elementary functions, so that the characteristic-function
// expression below instantiates for Cplx (values) and for Dual5 (values and partials).
__device__ __forceinline__ Cplx dsqrt(Cplx a) { return csqrt(a); }
__device__ __forceinline__ Cplx dexp(Cplx a) { return cexp(a); }
__device__ __forceinline__ Cplx dlog(Cplx a) { return clog(a); }
__device__ __forceinline__ Cplx dsinh(Cplx a) { return csinh(a); }
__device__ __forceinline__ Cplx dcosh(Cplx a) { return ccosh(a); }

// Value and the five partial derivatives (forward-mode, all parameter directions at once).
struct Dual5 {
    Cplx v, d[5];
};
__device__ __forceinline__ Dual5 d5const(Cplx v) {
    Dual5 r;
    r.v = v;
#pragma unroll
    for (int k = 0; k < 5; ++k) r.d[k] = cx(0.0);
    return r;
}
__device__ __forceinline__ Dual5 d5var(double v, int dir) {
    Dual5 r = d5const(cx(v));
    r.d[dir] = cx(1.0);
    return r;
}
__device__ __forceinline__ Dual5 operator+(Dual5 a, const Dual5& b) {
    a.v = a.v + b.v;
#pragma unroll
    for (int k = 0; k < 5; ++k) a.d[k] = a.d[k] + b.d[k];
    return a;
}
__device__ __forceinline__ Dual5 operator-(Dual5 a, const Dual5& b) {
    a.v = a.v - b.v;
#pragma unroll
    for (int k = 0; k < 5; ++k) a.d[k] = a.d[k] - b.d[k];
    return a;
}
__device__ __forceinline__ Dual5 operator*(const Dual5& a, const Dual5& b) {
    Dual5 r;
    r.v = a.v * b.v;
#pragma unroll
    for (int k = 0; k < 5; ++k) r.d[k] = a.d[k] * b.v + a.v * b.d[k];
    return r;
}
__device__ __forceinline__ Dual5 operator*(Cplx s, Dual5 a) {
    a.v = s * a.v;
#pragma unroll
    for (int k = 0; k < 5; ++k) a.d[k] = s * a.d[k];
    return a;
}
__device__ __forceinline__ Dual5 operator*(double s, Dual5 a) { return cx(s) * a; }
__device__ __forceinline__ Dual5 operator/(const Dual5& a, const Dual5& b) {
    Dual5 r;
    r.v = a.v / b.v;
    const Cplx ib = cx(1.0) / b.v;
#pragma unroll
    for (int k = 0; k < 5; ++k) r.d[k] = (a.d[k] - r.v * b.d[k]) * ib;
    return r;
}
// f(a) with f'(a.v) = df
__device__ __forceinline__ Dual5 d5apply(const Dual5& a, Cplx f, Cplx df) {
    Dual5 r;
    r.v = f;
#pragma unroll
    for (int k = 0; k < 5; ++k) r.d[k] = df * a.d[k];
    return r;
}
__device__ __forceinline__ Dual5 dsqrt(const Dual5& a) {
    const Cplx s = csqrt(a.v);
    return d5apply(a, s, cx(0.5) / s);
}
__device__ __forceinline__ Dual5 dexp(const Dual5& a) {
    const Cplx e = cexp(a.v);
    return d5apply(a, e, e);
}
__device__ __forceinline__ Dual5 dlog(const Dual5& a) { return d5apply(a, clog(a.v), cx(1.0) / a.v); }
__device__ __forceinline__ Dual5 dsinh(const Dual5& a) { return d5apply(a, csinh(a.v), ccosh(a.v)); }
__device__ __forceinline__ Dual5 dcosh(const Dual5& a) { return d5apply(a, ccosh(a.v), csinh(a.v)); }

__device__ __forceinline__ void set_const(Cplx& x, Cplx c) { x = c; }
__device__ __forceinline__ void set_const(Dual5& x, Cplx c) { x = d5const(c); }

// The Heston characteristic function of the reference's parameterisation (HDistribution::Helpers
// and chf, src/HDistribution.cpp:12-38) at real u, generic over the number type: Cplx gives the
// value, Dual5 the value and its five partial derivatives.
template <typename D>
__device__ __forceinline__ D chf_expr(const D& v0, const D& vm, const D& rho, const D& kappa, const D& sigma,
                                      double tau, double u) {
    const Cplx iu = cx(0.0, u);
    const D xi = kappa + iu * (sigma * rho);
    D fac;  // the constant u^2 - i u
    set_const(fac, cx(u * u, -u));
    const D d = dsqrt(xi * xi + (sigma * sigma) * fac);
    const D half = (0.5 * tau) * d;
    const D sh = dsinh(half), ch = dcosh(half);
    const D a1 = fac * sh;
    const D a2 = (d / v0) * ch + (xi / v0) * sh;
    const D A = a1 / a2;
    const D den = (d + xi) + (d - xi) * dexp((-tau) * d);
    const D Dl = dlog((2.0 * d) / den) + (0.5 * tau) * (kappa - d);
    const D t1 = cx(0.0, tau * u) * ((kappa * vm) * rho) / sigma;
    const D t3 = 2.0 * ((Dl * kappa) * vm) / (sigma * sigma);
    return dexp((t1 - A) + t3);
}

// chf(u) and its gradient in (v0, theta, rho, kappa, sigma) in one pass.
__device__ Dual5 heston_chf5(const double (&p)[5], double tau, double u) {
    return chf_expr<Dual5>(d5var(p[0], 0), d5var(p[1], 1), d5var(p[2], 2), d5var(p[3], 3), d5var(p[4], 4), tau, u);
}

__device__ __forceinline__ uint32_t find_chain(const uint64_t* end, uint32_t n, uint64_t t) {
    uint32_t lo = 0, hi = n - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (end[mid] > t)
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo;
}

__device__ __forceinline__ int64_t pmod(int64_t a, int64_t n) { return ((a % n) + n) % n; }

__device__ __forceinline__ double u_of(const DevSwift& R, uint32_t j) {
    return kPi * (2.0 * (double)j + 1.0) / (2.0 * (double)R.J) * R.exp2_m;
}

// Twiddle tables e^{2 pi i k / 4J}, k < 4J, one per distinct J of the call.
__global__ __launch_bounds__(256) void k_swift_twiddle(SwiftArgs a, uint64_t total) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint32_t ti = find_chain(a.tab_end, a.n_tables, t);
    const SwiftTable& T = a.tables[ti];
    const uint32_t k = (uint32_t)(t - (ti ? a.tab_end[ti - 1] : 0ull));
    double s, c;
    sincospi((double)k / (2.0 * (double)T.J), &s, &c);
    a.tw[T.off + k] = Cplx{c, s};
}

// Payoff coefficients of the call on [max(lower, 0), upper] (src/SWIFT.cpp:41-58):
// H(upper) - H(max(lower, 0)) with H(y) = -i e^{-i u y} (1/u - e^y / (i + u)).
__device__ __forceinline__ Cplx payoff_at(const DevSwift& R, uint32_t k) {
    const double u = u_of(R, k);
    const double ylo = R.lower > 0.0 ? R.lower : 0.0;
    const Cplx iu1 = cx(u, 1.0);  // i + u
    const Cplx inv_u = cx(1.0 / u);
    const Cplx mi = cx(0.0, -1.0);
    const Cplx hu = mi * cexp(cx(0.0, -u * R.upper)) * (inv_u - cx(exp(R.upper)) / iu1);
    const Cplx hl = mi * cexp(cx(0.0, -u * ylo)) * (inv_u - cx(exp(ylo)) / iu1);
    return hu - hl;
}

__global__ __launch_bounds__(256) void k_swift_payoff(SwiftArgs a, uint64_t total) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint32_t ri = find_chain(a.j_end, a.n_req, t);
    const DevSwift& R = a.reqs[ri];
    const uint32_t k = (uint32_t)(t - (ri ? a.j_end[ri - 1] : 0ull));
    a.pay[R.pay_off + k] = payoff_at(R, k);
}

// First transform (src/SWIFT.cpp:59-70): for each wavelet index i in [k1, k2], the length-2J
// backward DFT of the zero-padded payoff coefficients at i mod 2J, rotated by e^{i pi i / 2J}:
// dens_i = Re(e^{i pi i/2J} sum_j pay_j e^{2 pi i j i / 2J}) sqrt(2^m) / J.
// Direct sum: one wavefront per i, lane l sums j = l, l+64, ... in
// order (twiddle tw[(2 j i2) mod 4J]), a fixed xor butterfly combines the lanes.
__global__ __launch_bounds__(256) void k_swift_dens(SwiftArgs a, uint64_t total) {
    const uint64_t w = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64u;  // wave-uniform
    const uint32_t lane = threadIdx.x % 64u;
    if (w >= total) return;
    const uint32_t ri = find_chain(a.dens_end, a.n_req, w);
    const DevSwift& R = a.reqs[ri];
    const int64_t il = (int64_t)(w - (ri ? a.dens_end[ri - 1] : 0ull));
    const int64_t i = R.k1 + il;
    const int64_t n4 = 4 * (int64_t)R.J;
    const Cplx* tw = a.tw + R.tw_off;
    const Cplx* pay = a.pay + R.pay_off;
    const int64_t step = 2 * pmod(i, 2 * (int64_t)R.J);  // index advance per unit of j
    const int64_t stride = (64 * step) % n4;             // per lane iteration
    int64_t idx = ((int64_t)lane * step) % n4;
    double re = 0.0, im = 0.0;
    for (uint32_t j = lane; j < R.J; j += 64u) {
        const Cplx q = pay[j] * tw[idx];
        re += q.re;
        im += q.im;
        idx += stride;
        if (idx >= n4) idx -= n4;
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        re += __shfl_xor(re, m);
        im += __shfl_xor(im, m);
    }
    if (lane != 0) return;
    const Cplx rot = tw[pmod(i, n4)];
    a.dens[R.dens_off + (uint64_t)il] = (rot * Cplx{re, im}).re * R.sqrt_exp2_m / (double)R.J;
}

// Second transform (src/SWIFT.cpp:71-72): the length-4J real forward DFT of dens at the odd bin
// 2j+1, conjugated and scaled: c_j = conj(sum_i dens_i e^{-2 pi i (i mod 4J)(2j+1)/4J}) sqrt(2^m)/J.
// Direct sum: one wavefront per j, lanes strided over i as above.
__global__ __launch_bounds__(256) void k_swift_coeff(SwiftArgs a, uint64_t total) {
    const uint64_t w = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64u;  // wave-uniform
    const uint32_t lane = threadIdx.x % 64u;
    if (w >= total) return;
    const uint32_t ri = find_chain(a.j_end, a.n_req, w);
    const DevSwift& R = a.reqs[ri];
    const uint32_t j = (uint32_t)(w - (ri ? a.j_end[ri - 1] : 0ull));
    const int64_t n4 = 4 * (int64_t)R.J;
    const Cplx* tw = a.tw + R.tw_off;
    const double* dens = a.dens + R.dens_off;
    const int64_t k = 2 * (int64_t)j + 1;  // < n4
    const int64_t stride = (64 * k) % n4;
    int64_t idx = (pmod(R.k1 + (int64_t)lane, n4) * k) % n4;
    double re = 0.0, im = 0.0;
    for (int64_t i = R.k1 + (int64_t)lane; i <= R.k2; i += 64) {
        const double d = dens[i - R.k1];
        const Cplx t = tw[idx];
        re += d * t.re;
        im -= d * t.im;  // conj(tw)
        idx += stride;
        if (idx >= n4) idx -= n4;
    }
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        re += __shfl_xor(re, m);
        im += __shfl_xor(im, m);
    }
    if (lane != 0) return;
    a.coeff[R.coeff_off + j] = (R.sqrt_exp2_m / (double)R.J) * Cplx{re, -im};
}

// Pricing matrix (src/SWIFT.cpp:106-110): row 0 = chf(u_j) c_j, rows 1..5 = d chf / d p_k c_j.
// A chain has as many workgroups as the largest J needs; those past its own J return at once. A
// workgroup's number modulo 8 is its XCD, so that the ones of a short chain (the first few) begin at
// another XCD for each chain, and for each run of 8 chains: calibration batches repeat 8 or so
// maturities, and with each maturity on an XCD of its own 512 chains took 63 us instead of 55.
__global__ __launch_bounds__(256) void k_swift_chf(SwiftArgs a, uint32_t blocks) {
    const uint32_t ri = blockIdx.x / blocks;
    const DevSwift& R = a.reqs[ri];
    const uint32_t j = ((blockIdx.x + ri + ri / 8u) & (blocks - 1u)) * blockDim.x + threadIdx.x;  // blocks: 2^k
    if (j >= R.J) return;
    const double p[5] = {R.p[0], R.p[1], R.p[2], R.p[3], R.p[4]};
    const double u = u_of(R, j);
    const Cplx c = a.coeff[R.coeff_off + j];
    Cplx* pm = a.pm + R.pm_off;
    // the value row comes from the plain evaluation in both modes, so prices do not depend on
    // whether gradients were asked for
    pm[j] = chf_expr<Cplx>(cx(p[0]), cx(p[1]), cx(p[2]), cx(p[3]), cx(p[4]), R.T, u) * c;
    if (R.rows == 6) {
        const Dual5 f = heston_chf5(p, R.T, u);
#pragma unroll
        for (int k = 0; k < 5; ++k) pm[(uint64_t)(k + 1) * R.J + j] = f.d[k] * c;
    }
}

// Final contraction (src/SWIFT.cpp:111-117): out[s][row] = Re sum_j pm[row][j] e^{-rT} K_s e^{-i u_j x_s}.
// One workgroup per (chain, group of NS x 16 strikes): thread (s, p) = (tid % 16, tid / 16) owns
// strikes s, s + 16, ... and sums j = p, p+16, ... in order; the pricing matrix is staged through LDS
// in chunks of 256 j, the next one on its way in registers meanwhile; the 16 partial sums of a strike
// are added in a fixed order. With one strike a thread the LDS (6 x 16 B per lane and j) and not the
// FP64 units set the pace; two share each read.
constexpr int kSumChunk = 256;
constexpr int kSumLanes = 16;
constexpr uint32_t kSumPhases = 256 / kSumLanes;
// A long chain is bound by its serial sums, though (J = 4,096 alone: 77 us with one group of 256
// threads, 65 with the next chunk in registers, 54 with its six rows on three groups): G groups.
template <int NS, int ROWS, int G>
__global__ __launch_bounds__(256 * G) void k_swift_sum(SwiftArgs a) {
    constexpr int RG = ROWS / G;  // rows per group
    __shared__ union {
        Cplx pm[ROWS][kSumChunk];
        double part[ROWS][NS][256];
    } sh;
    const DevSwift& R = a.reqs[a.block_chain[blockIdx.x]];
    const uint32_t J = R.J;
    if (J == 0) return;  // not priced in this pass; uniform over the workgroup
    const uint32_t o0 = a.block_strike[blockIdx.x];
    const uint32_t tid = threadIdx.x % 256u, row0 = threadIdx.x / 256u * RG;
    const uint32_t sl = tid % kSumLanes, ph = tid / kSumLanes;
    const Cplx* pm = a.pm + R.pm_off + (uint64_t)row0 * J;
    Cplx next[RG];
    if (tid < J) {
#pragma unroll
        for (int k = 0; k < RG; ++k) next[k] = pm[(uint64_t)k * J + tid];
    }
    double x[NS], scale[NS];
    Cplx rot[NS], z[NS];
    double acc[RG][NS];
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        const uint32_t so = o0 + i * kSumLanes + sl;
        const bool on = so < R.n_strikes;
        const double K = a.strikes[R.strike_off + (on ? so : o0)];
        x[i] = __builtin_fma(R.r, R.T, log(R.S0 / K));
        scale[i] = on ? R.disc * K : 0.0;
        // e^{-i u_j x} along j = p, p+16, ...: rotation by e^{-i 16 (u_{j+1} - u_j) x}, re-anchored with
        // a direct evaluation every 16 steps (rounding grows by at most 16 ulps)
        double sr, cr;
        sincos(-((double)kSumPhases * kPi / (double)J * R.exp2_m) * x[i], &sr, &cr);
        rot[i] = Cplx{cr, sr};
#pragma unroll
        for (int k = 0; k < RG; ++k) acc[k][i] = 0.0;
    }
    constexpr int kUnroll = NS * RG <= 3 ? 4 : NS == 1 ? 2 : 1;
    for (uint32_t jc = 0; jc < J; jc += kSumChunk) {
        const uint32_t n = min((uint32_t)kSumChunk, J - jc);
        __syncthreads();  // the previous chunk has been consumed
        if (tid < n) {
#pragma unroll
            for (int k = 0; k < RG; ++k) sh.pm[row0 + k][tid] = next[k];
        }
        __syncthreads();
        if (jc + kSumChunk + tid < J) {
#pragma unroll
            for (int k = 0; k < RG; ++k) next[k] = pm[(uint64_t)k * J + jc + kSumChunk + tid];
        }
        if (ph < n) {
            const double u = u_of(R, jc + ph);
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                double sn, cs;
                sincos(-u * x[i], &sn, &cs);
                z[i] = Cplx{cs, sn};
            }
        }
        // the products are written out as one rounding and one fused step each, so that every
        // instance gives the same bits
#pragma unroll kUnroll
        for (uint32_t jj = ph; jj < n; jj += kSumPhases) {
            double er[NS], ei[NS];
#pragma unroll
            for (int i = 0; i < NS; ++i) {
                er[i] = scale[i] * z[i].re;
                ei[i] = scale[i] * z[i].im;
                z[i] = Cplx{__builtin_fma(z[i].re, rot[i].re, -__dmul_rn(z[i].im, rot[i].im)),
                            __builtin_fma(z[i].re, rot[i].im, __dmul_rn(z[i].im, rot[i].re))};
            }
#pragma unroll
            for (int k = 0; k < RG; ++k) {
                const Cplx c = sh.pm[row0 + k][jj];
#pragma unroll
                for (int i = 0; i < NS; ++i)
                    acc[k][i] = __dadd_rn(acc[k][i], __builtin_fma(er[i], c.re, -__dmul_rn(ei[i], c.im)));
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < RG; ++k)
#pragma unroll
        for (int i = 0; i < NS; ++i) sh.part[row0 + k][i][tid] = acc[k][i];
    __syncthreads();
    // Each output's 16 phases in order, by one thread: the prices, then the gradients as they lie in
    // memory (strike, row): they go over the host link, where a wavefront's stores want to be contiguous.
    constexpr uint32_t kStrikes = NS * kSumLanes;
    const uint32_t t = threadIdx.x, g = t - kStrikes;
    const uint32_t s_out = t < kStrikes ? t : g / 5u, k = t < kStrikes ? 0u : 1u + g % 5u;
    if (t >= kStrikes * ROWS || o0 + s_out >= R.n_strikes) return;
    const double* part = sh.part[k][s_out / kSumLanes];
    double v = 0.0;
    for (uint32_t p = 0; p < kSumPhases; ++p) v += part[p * kSumLanes + s_out % kSumLanes];
    const uint64_t o = R.out_off + o0;
    if (t < kStrikes)
        a.prices[o + t] = v;
    else
        a.grads[o * 5 + g] = v;
}

// ------------------------------------------------------------------------------------------
// A chain from its inputs to its density coefficients, one per workgroup
// ------------------------------------------------------------------------------------------
// e^{2 pi i k / 4 kSwiftFftMaxJ}, k < 4 kSwiftFftMaxJ: every smaller transform's roots are a stride
// of it. Filled once per context.
__global__ __launch_bounds__(256) void k_swift_roots(Cplx* roots) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= 4u * kSwiftFftMaxJ) return;
    double s, c;
    sincospi((double)k / (2.0 * (double)kSwiftFftMaxJ), &s, &c);
    roots[k] = Cplx{c, s};
}

// The scale of a chain's dynamic grid (SwiftParameters ctor, src/SWIFT.cpp:21-35) by one wavefront. The lanes
// first find the chain's extreme strikes (and whether every strike is finite and positive). The
// reference loops m = 0, 1, ... while int_error(m) > trunc and keeps one past the first m that
// stops it (src/HDistribution.cpp:8-11: |chf(2^m pi) + chf(-2^m pi)| / (4 2^m pi^2 T)); here lane m
// evaluates scale m for m = 0..30 at once and the lowest lane whose error does not exceed trunc (a
// NaN error stops the loop too) is that first m. chf(-u) is the conjugate of chf(u), to the last
// bit, so the sum is twice the real part. Lanes past the first evaluate scales the loop never
// reaches; their values are not used. The result is the same in every lane.
// Returns the status so far; m and the extreme strikes where it is kSwiftGridOk.
__device__ int32_t swift_scale_wave(const SwiftChainIn& q, const double* ks, int lane, uint32_t& m, double& kmin,
                                    double& kmax) {
    double lo = INFINITY, hi = -INFINITY;
    bool bad = false;
    for (uint32_t i = (uint32_t)lane; i < q.n_strikes; i += 64) {
        const double k = ks[i];
        bad |= !(k > 0.0 && k < INFINITY);
        lo = fmin(lo, k);
        hi = fmax(hi, k);
    }
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        lo = fmin(lo, __shfl_xor(lo, s));
        hi = fmax(hi, __shfl_xor(hi, s));
    }
    kmin = lo;
    kmax = hi;
    m = 0;
    if (__builtin_amdgcn_ballot_w64(bad)) return kSwiftGridBadStrike;
    if (q.fixed) return kSwiftGridOk;
    bool stop = false;
    if (lane <= 30) {
        const double e2m = ::ldexp(1.0, lane);
        const Cplx f =
            chf_expr<Cplx>(cx(q.p[0]), cx(q.p[1]), cx(q.p[2]), cx(q.p[3]), cx(q.p[4]), q.T, e2m * kPi);
        stop = !(::fabs(2.0 * f.re) / (4.0 * e2m * kPi * kPi * q.T) > q.trunc);
    }
    const uint64_t mask = __builtin_amdgcn_ballot_w64(stop);
    if (mask == 0) return kSwiftGridNoScale;
    m = (uint32_t)__builtin_ctzll(mask) + 1u;
    return kSwiftGridOk;
}

// One radix-2 butterfly with the root e^{SIGN i phi}, w = e^{i phi}: (x0, x1) to
// (x0 + x1 e, x0 - x1 e). The fused products are written out: left to the compiler, their choice
// (and so the last bits of prices that cancel heavily) would change with the code around them.
template <int SIGN>
__device__ __forceinline__ void butterfly(Cplx& x0, Cplx& x1, Cplx w) {
    const Cplx u = x0;
    Cplx v;
    if (SIGN > 0) {
        v.re = __builtin_fma(w.re, x1.re, -__dmul_rn(w.im, x1.im));
        v.im = __builtin_fma(w.im, x1.re, __dmul_rn(w.re, x1.im));
    } else {
        v.re = __builtin_fma(w.re, x1.re, __dmul_rn(w.im, x1.im));
        v.im = __builtin_fma(w.re, x1.im, -__dmul_rn(w.im, x1.re));
    }
    x0 = Cplx{__dadd_rn(u.re, v.re), __dadd_rn(u.im, v.im)};
    x1 = Cplx{__dsub_rn(u.re, v.re), __dsub_rn(u.im, v.im)};
}

// In-place transform of length N = 2^logN in LDS, sum x_n e^{+-2 pi i n k / N}, bit-reversed order to
// natural, from stage s on: radix-2 decimation in time, two stages per pass over the LDS (a pass and
// its barrier cost more than the butterflies).
template <int SIGN, uint32_t THREADS>
__device__ __forceinline__ void fft_lds(Cplx* x, uint32_t logN, uint32_t s, const Cplx* __restrict__ roots) {
    const uint32_t N = 1u << logN;
    for (; s + 2 <= logN; s += 2) {
        const uint32_t h = 1u << s, st = 2u * kSwiftFftMaxJ >> s;  // roots[st k] = e^{2 pi i k / 2h}
        for (uint32_t b = threadIdx.x; b < N / 4; b += THREADS) {
            const uint32_t k = b & (h - 1u), i = 4 * b - 3 * k;  // (b / h) 4h + k
            Cplx x0 = x[i], x1 = x[i + h], x2 = x[i + 2 * h], x3 = x[i + 3 * h];
            const Cplx w = roots[st * k];
            butterfly<SIGN>(x0, x1, w);
            butterfly<SIGN>(x2, x3, w);
            butterfly<SIGN>(x0, x2, roots[(st / 2) * k]);
            butterfly<SIGN>(x1, x3, roots[(st / 2) * (k + h)]);
            x[i] = x0;
            x[i + h] = x1;
            x[i + 2 * h] = x2;
            x[i + 3 * h] = x3;
        }
        __syncthreads();
    }
    if (s < logN) {  // s = logN - 1
        const uint32_t h = 1u << s, st = 2u * kSwiftFftMaxJ >> s;
        for (uint32_t k = threadIdx.x; k < h; k += THREADS) {
            Cplx x0 = x[k], x1 = x[k + h];
            butterfly<SIGN>(x0, x1, roots[st * k]);
            x[k] = x0;
            x[k + h] = x1;
        }
        __syncthreads();
    }
}

// Each of a call's chains from its inputs to its density coefficients.
//
// As a kernel per stage, the grids first, this was five launches and a host round trip for the
// layout between the grids and the rest. Here a chain's data stays in its CU: the payoff
// coefficients go straight to their bit-reversed places, the second transform's input is
// elementwise in the first's output, and two radix-2 stages share a pass over the LDS. A chain is
// bound by the serial chain of its stages (a lone one of J = 512: 21 us of the 39 us that the five
// kernels took; 1,024 threads for the largest J no faster than 512), so that a batch wants several on
// a CU: with MAX_J = 1,024, 32 KiB and 256 threads four fit, of the largest J one.
template <uint32_t MAX_J, uint32_t THREADS>
__global__ __launch_bounds__(THREADS) void k_swift_transform(SwiftChainArgs a) {
    extern __shared__ Cplx lds_c[];  // 2 MAX_J values
    __shared__ DevSwift R;
    __shared__ double width_s, k_s[2];
    __shared__ uint32_t scale_s;
    __shared__ int32_t status_s;
    const uint32_t slot = blockIdx.x, ci = a.order ? a.order[slot] : slot;
    const SwiftChainIn& q = a.chains[ci];
    // one wavefront each, at the same time: the scale and the range's width; the others hand what the
    // contraction needs on to device memory
    if (threadIdx.x < 64) {
        uint32_t m;
        double kmin, kmax;
        const int32_t status = swift_scale_wave(q, a.strikes + q.strike_off, (int)threadIdx.x, m, kmin, kmax);
        if (threadIdx.x == 0) {
            scale_s = m;
            status_s = status;
            k_s[0] = kmin;
            k_s[1] = kmax;
        }
    } else if (threadIdx.x < 128) {
        const double c = swift_grid_width(q.p, q.T);
        if (threadIdx.x == 64) width_s = c;
    } else {
        const uint32_t t = threadIdx.x - 128u;
        for (uint32_t k = t; k < q.n_strikes; k += THREADS - 128u) a.dev_strikes[q.strike_off + k] = a.strikes[q.strike_off + k];
        for (uint32_t b = t; b * a.strike_block < q.n_strikes; b += THREADS - 128u) {
            a.block_chain[q.block_off + b] = slot;
            a.block_strike[q.block_off + b] = b * a.strike_block;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        SwiftGridOut o{};
        o.status = status_s;
        if (status_s == kSwiftGridOk && q.fixed) {
            o.g = q.grid;
        } else if (status_s == kSwiftGridOk) {
            const SwiftGridIn in{{q.p[0], q.p[1], q.p[2], q.p[3], q.p[4]}, q.T, q.r, q.S0, k_s[0], k_s[1], q.trunc};
            o.status = swift_grid_finish(in, width_s, scale_s, o.g, o.J_wanted);
        }
        DevSwift r{};
#pragma unroll
        for (int i = 0; i < 5; ++i) r.p[i] = q.p[i];
        r.S0 = q.S0;
        r.r = q.r;
        r.T = q.T;
        r.disc = q.disc;
        r.exp2_m = (double)o.g.exp2_m;
        r.sqrt_exp2_m = o.g.sqrt_exp2_m;
        r.lower = o.g.lower;
        r.upper = o.g.upper;
        r.k1 = o.g.k1;
        r.k2 = o.g.k2;
        r.n_strikes = q.n_strikes;
        r.rows = a.rows;
        r.strike_off = r.out_off = q.strike_off;
        if (o.status == kSwiftGridOk && o.g.J <= MAX_J) {
            r.J = o.g.J;
            r.coeff_off = (uint64_t)slot * MAX_J;
            r.pm_off = r.coeff_off * a.rows;
        }
        R = r;
        a.recs[slot] = r;
        a.grids[ci] = o;
    }
    __syncthreads();
    const uint32_t J = R.J;
    if (J == 0) return;  // uniform
    const double norm = R.sqrt_exp2_m / (double)J;
    const uint32_t N = 2u * J, logN = 32u - (uint32_t)__builtin_clz(N) - 1u;
    // payoff coefficients, zero-padded to 2J, into bit-reversed order (the padding lands on the odd
    // places, so that the first stage copies each value onto its neighbour), then the first transform
    // (src/SWIFT.cpp:59-70)
    for (uint32_t j = threadIdx.x; j < J; j += THREADS) {
        const uint32_t b = __builtin_bitreverse32(j) >> (32u - logN);
        lds_c[b] = lds_c[b + 1] = payoff_at(R, j);
    }
    __syncthreads();
    fft_lds<+1, THREADS>(lds_c, logN, 1, a.roots);
    // Wavelet index i (k1 <= i <= k2) has density Re(e^{i pi i/2J} F_{i mod 2J}) norm, and the length-4J
    // real transform's odd bins (src/SWIFT.cpp:71-72) are the length-2J transform of
    // z_n = y_n + y_{n+2J}, y_n = x_n e^{-i pi n/2J} with x_n the density at i = n mod 4J. Both terms are
    // the same product (e^{i pi (n+2J)/2J} = -e^{i pi n/2J}) of values at n: no density array, only the
    // bit reversal in front of the second transform, through registers.
    const uint32_t rs = kSwiftFftMaxJ / J;
    const uint32_t wrap = 2u * N - 1u, k1 = (uint32_t)R.k1, span = (uint32_t)R.k2 - k1;  // mod 4J
    constexpr uint32_t kOwn = 2u * MAX_J / THREADS;
    Cplx y[kOwn];
#pragma unroll
    for (uint32_t e = 0; e < kOwn; ++e) {
        const uint32_t n = threadIdx.x + e * THREADS;
        if (n < N) {
            const Cplx t = a.roots[rs * n];
            const double dens = __builtin_fma(t.re, lds_c[n].re, -__dmul_rn(t.im, lds_c[n].im)) * norm;
            const bool h0 = ((n - k1) & wrap) <= span, h1 = ((n + N - k1) & wrap) <= span;
            Cplx v = (h0 || h1) ? dens * conj(t) : cx(0.0);
            if (h0 && h1) v = Cplx{__builtin_fma(dens, t.re, v.re), __builtin_fma(dens, -t.im, v.im)};
            y[e] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t e = 0; e < kOwn; ++e) {
        const uint32_t n = threadIdx.x + e * THREADS;
        if (n < N) lds_c[__builtin_bitreverse32(n) >> (32u - logN)] = y[e];
    }
    __syncthreads();
    fft_lds<-1, THREADS>(lds_c, logN, 0, a.roots);
    for (uint32_t j = threadIdx.x; j < J; j += THREADS) a.coeff[R.coeff_off + j] = norm * conj(lds_c[j]);
}

// Copies two ranges of 16-byte words from fine-grained pinned host memory to the device (a call's
// tables and its strikes), so the pricing kernels read them from HBM.
__global__ __launch_bounds__(256) void k_swift_stage(const uint4* s0, uint4* d0, uint64_t n0, const uint4* s1,
                                                     uint4* d1, uint64_t n1) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n0 + n1; i += stride) {
        if (i < n0)
            d0[i] = s0[i];
        else
            d1[i - n0] = s1[i - n0];
    }
}

inline dim3 grid_of(uint64_t n, uint32_t block) { return dim3((uint32_t)((n + block - 1) / block)); }

}  // namespace

hipError_t launch_swift_large(const SwiftArgs& a, const SwiftTotals& t, hipStream_t st) {
    k_swift_twiddle<<<grid_of(t.tw, 256), 256, 0, st>>>(a, t.tw);
    k_swift_payoff<<<grid_of(t.j, 256), 256, 0, st>>>(a, t.j);
    k_swift_dens<<<grid_of(t.dens * 64u, 256), 256, 0, st>>>(a, t.dens);
    k_swift_coeff<<<grid_of(t.j * 64u, 256), 256, 0, st>>>(a, t.j);
    return launch_swift_prices(a, HEXO_SWIFT_MAX_J, st);
}

hipError_t launch_swift_prices(const SwiftArgs& a, uint32_t max_J, hipStream_t st) {
    const uint32_t blocks = max_J / 256u;
    k_swift_chf<<<a.n_req * blocks, 256, 0, st>>>(a, blocks);
    if (a.strike_block > kSumLanes)
        a.grads ? k_swift_sum<2, 6, 1><<<a.n_blocks, 256, 0, st>>>(a) : k_swift_sum<2, 1, 1><<<a.n_blocks, 256, 0, st>>>(a);
    else if (!a.grads)
        k_swift_sum<1, 1, 1><<<a.n_blocks, 256, 0, st>>>(a);
    else if (a.split_rows)
        k_swift_sum<1, 6, 3><<<a.n_blocks, 768, 0, st>>>(a);
    else
        k_swift_sum<1, 6, 1><<<a.n_blocks, 256, 0, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_swift_roots(Cplx* roots, hipStream_t st) {
    k_swift_roots<<<grid_of(4ull * kSwiftFftMaxJ, 256), 256, 0, st>>>(roots);
    return hipGetLastError();
}

template <uint32_t MAX_J, uint32_t THREADS>
hipError_t launch_transform(const SwiftChainArgs& a, hipStream_t st) {
    const int lds = (int)(sizeof(Cplx) * 2 * MAX_J);
    // the kernel's dynamic LDS limit, raised once per device
    static std::atomic<uint64_t> lds_set{0};  // bit d: done on device d
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const uint64_t bit = 1ull << (dev & 63);
    if (!(lds_set.load() & bit)) {
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(k_swift_transform<MAX_J, THREADS>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) return e;
        lds_set.fetch_or(bit);
    }
    k_swift_transform<MAX_J, THREADS><<<a.n_req, THREADS, lds, st>>>(a);
    return hipGetLastError();
}

hipError_t launch_swift_transform(const SwiftChainArgs& a, hipStream_t st) {
    return a.max_J == kSwiftSmallJ ? launch_transform<kSwiftSmallJ, 256>(a, st) : launch_transform<kSwiftFftMaxJ, 512>(a, st);
}

hipError_t launch_swift_stage(const void* s0, void* d0, size_t bytes0, const void* s1, void* d1, size_t bytes1,
                              hipStream_t st) {
    if (bytes0 % 16 || bytes1 % 16) return hipErrorInvalidValue;
    const uint64_t n0 = bytes0 / 16, n1 = bytes1 / 16;
    if (n0 + n1 == 0) return hipSuccess;
    const uint32_t blocks = (uint32_t)std::min<uint64_t>((n0 + n1 + 255) / 256, 1024);
    k_swift_stage<<<blocks, 256, 0, st>>>(static_cast<const uint4*>(s0), static_cast<uint4*>(d0), n0,
                                          static_cast<const uint4*>(s1), static_cast<uint4*>(d1), n1);
    return hipGetLastError();
}

}  // namespace hexo
