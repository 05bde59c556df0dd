// swift_host.cpp -- host side of the SWIFT European pricer: validation, the dynamic grid (the
// reference's SwiftParameters constructor, src/SWIFT.cpp:21-35) for hexo_swift_grid_for (a call's
// grids are chosen on the GPU, swift.hip), the layout of one call's chains in the context's
// pinned stages, and the C entry points hexo_swift_grid_for / hexo_swift_price.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/hexo.h"
#include "engine.hpp"
#include "swift.hpp"
#include "swift_grid.hpp"

namespace {

using cd = std::complex<double>;
constexpr double kPi = 3.14159265358979323846;

// The reference's characteristic function (src/HDistribution.cpp:12-38), for the truncation test.
cd heston_chf(const double p[5], double tau, double u) {
    const double v0 = p[0], theta = p[1], rho = p[2], kappa = p[3], sigma = p[4];
    const cd iu(0.0, u);
    const cd xi = kappa + sigma * rho * iu;
    const cd fac = u * u - iu;
    const cd d = std::sqrt(xi * xi + sigma * sigma * fac);
    const cd sh = std::sinh(d * (tau * 0.5)), ch = std::cosh(d * (tau * 0.5));
    const cd A = fac * sh / (d / v0 * ch + xi / v0 * sh);
    const cd D = std::log(2.0 * d / (d + xi + (d - xi) * std::exp(-d * tau))) + (kappa - d) * (tau * 0.5);
    return std::exp(kappa * theta * rho * tau * iu / sigma - A + 2.0 * D * kappa * theta / (sigma * sigma));
}

// Truncation error of scale m (HDistribution::int_error, src/HDistribution.cpp:8-11).
double int_error(const double p[5], double tau, unsigned m) {
    const double e2m = std::exp2((double)m);
    return std::abs(heston_chf(p, tau, e2m * kPi) + heston_chf(p, tau, -e2m * kPi)) / (4.0 * e2m * kPi * kPi * tau);
}

bool finite_pos(double x) { return std::isfinite(x) && x > 0.0; }

// Everything but the strikes' values.
int check_chain(const hexo_swift_request& q, std::string& err) {
    if (!(finite_pos(q.v0) && finite_pos(q.theta) && finite_pos(q.kappa) && finite_pos(q.sigma) &&
          std::isfinite(q.rho) && q.rho > -1.0 && q.rho < 1.0)) {
        err = "Heston parameters out of range (v0, theta, kappa, sigma > 0, |rho| < 1)";
        return HEXO_ERR_INVALID;
    }
    if (!finite_pos(q.S0) || !finite_pos(q.T) || !std::isfinite(q.r)) {
        err = "S0 and T must be positive, r finite";
        return HEXO_ERR_INVALID;
    }
    if (q.n_strikes == 0 || !q.strikes) {
        err = "a chain needs at least one strike";
        return HEXO_ERR_INVALID;
    }
    if (q.flags & ~HEXO_SWIFT_FIXED_GRID) {
        err = "unknown flags";
        return HEXO_ERR_INVALID;
    }
    if (!(q.flags & HEXO_SWIFT_FIXED_GRID) && !(q.trunc > 0.0 && q.trunc < 1.0)) {
        err = "trunc must be in (0, 1)";
        return HEXO_ERR_INVALID;
    }
    return HEXO_OK;
}

int check_strikes(const hexo_swift_request& q, std::string& err) {
    for (uint32_t i = 0; i < q.n_strikes; ++i)
        if (!finite_pos(q.strikes[i])) {
            err = "strikes must be positive";
            return HEXO_ERR_INVALID;
        }
    return HEXO_OK;
}

int check_request(const hexo_swift_request& q, std::string& err) {
    const int rc = check_chain(q, err);
    return rc ? rc : check_strikes(q, err);
}

int check_grid(const hexo_swift_grid& g, std::string& err) {
    const uint32_t J = g.J;
    if (J == 0 || (J & (J - 1)) || J > HEXO_SWIFT_MAX_J) {
        err = "J must be a power of two <= HEXO_SWIFT_MAX_J";
        return HEXO_ERR_INVALID;
    }
    if (g.m > 30 || g.exp2_m != (1u << g.m) || g.reserved != 0 || !(g.sqrt_exp2_m > 0.0) ||
        !std::isfinite(g.lower) || !std::isfinite(g.upper) || !(g.lower < g.upper)) {
        err = "inconsistent SWIFT grid";
        return HEXO_ERR_INVALID;
    }
    // the density input of length 4J must hold every wavelet index once (no aliasing)
    if (g.k2 < g.k1 || (int64_t)g.k2 - (int64_t)g.k1 + 1 > 4 * (int64_t)J) {
        err = "wavelet index range must satisfy k1 <= k2 < k1 + 4J";
        return HEXO_ERR_INVALID;
    }
    return HEXO_OK;
}

// The extreme strikes and the rest of a chain's grid-choice inputs.
hexo::SwiftGridIn grid_input(const hexo_swift_request& q) {
    hexo::SwiftGridIn in{{q.v0, q.theta, q.rho, q.kappa, q.sigma}, q.T, q.r, q.S0, q.strikes[0], q.strikes[0], q.trunc};
    for (uint32_t i = 1; i < q.n_strikes; ++i) {
        in.kmin = std::min(in.kmin, q.strikes[i]);
        in.kmax = std::max(in.kmax, q.strikes[i]);
    }
    return in;
}

int grid_status(int32_t status, double J_wanted, std::string& err) {
    switch (status) {
        case hexo::kSwiftGridOk: return HEXO_OK;
        case hexo::kSwiftGridNoScale: err = "no wavelet scale reaches the truncation precision"; break;
        case hexo::kSwiftGridOverflow: err = "SWIFT index range overflows"; break;
        case hexo::kSwiftGridBadStrike: err = "strikes must be positive"; break;
        default: err = "SWIFT grid needs J = " + std::to_string(J_wanted) + " (outside [1, HEXO_SWIFT_MAX_J])"; break;
    }
    return HEXO_ERR_INVALID;
}

// SwiftParameters constructor (src/SWIFT.cpp:21-35) on the host.
int dynamic_grid(const hexo_swift_request& q, hexo_swift_grid& g, std::string& err) {
    const hexo::SwiftGridIn in = grid_input(q);
    unsigned m = 0;
    // the reference loops `while (int_error(m++) > trunc)`: m ends one past the first scale
    // whose error bound is below trunc
    while (int_error(in.p, q.T, m++) > q.trunc)
        if (m > 30) return grid_status(hexo::kSwiftGridNoScale, 0.0, err);
    double J = 0.0;
    return grid_status(hexo::swift_grid_finish(in, hexo::swift_grid_width(in.p, in.T), m, g, J), J, err);
}

// Grows one of the context's SWIFT device buffers to at least `bytes` (kept for the context's
// lifetime, so calls of a calibration loop allocate nothing).
int grow_device(hexo_ctx* ctx, void*& buf, size_t& cap, size_t bytes) {
    if (bytes <= cap) return HEXO_OK;
    // the previous buffer may still be read by work queued on the stream
    if (hipStreamSynchronize(ctx->stream) != hipSuccess) return ctx->set_error(HEXO_ERR_HIP, "stream sync failed");
    if (buf) (void)hipFree(buf);
    buf = nullptr;
    cap = 0;
    const size_t want = bytes + bytes / 2;
    if (hipMalloc(&buf, want) != hipSuccess) {
        buf = nullptr;
        return ctx->set_error(HEXO_ERR_NOMEM, "hipMalloc failed");
    }
    cap = want;
    return HEXO_OK;
}

int grid_of(const hexo_swift_request& q, hexo_swift_grid& g, std::string& err) {
    int rc = check_request(q, err);
    if (rc) return rc;
    if (q.flags & HEXO_SWIFT_FIXED_GRID)
        g = q.grid;
    else if ((rc = dynamic_grid(q, g, err)))
        return rc;
    return check_grid(g, err);
}

}  // namespace

extern "C" int hexo_swift_grid_for(const hexo_swift_request* req, hexo_swift_grid* out) {
    if (!req || !out) return HEXO_ERR_INVALID;
    std::string err;
    return grid_of(*req, *out, err);
}

namespace {

// A chain's J up to a factor (J / 1.3, mostly within a factor of 2): the frequency where the
// characteristic function, e^{-u sqrt(1 - rho^2) (v0 + kappa theta T) / sigma} far out, has fallen to
// trunc, times the width of the log-price range, about 20 standard deviations and the strikes'. Only
// the order and the class of a chain's workgroup depend on it.
double size_estimate(const hexo_swift_request& q) {
    if (q.flags & HEXO_SWIFT_FIXED_GRID) return 0.6 * q.grid.J;  // 1,024 below the line at 640, 2,048 above it
    const double u = -std::log(q.trunc) * q.sigma / ((q.v0 + q.kappa * q.theta * q.T) * std::sqrt(1.0 - q.rho * q.rho));
    const double size = u * (0.5 + 20.0 * std::sqrt(std::max(q.v0, q.theta) * q.T));
    return std::isfinite(size) ? size : 1e300;  // ordered in any case
}

// How the contraction of a pass with `blocks` groups of 16 strikes (of long chains, or in price_large; as
// many as would take as long if all chains were the longest) divides its work: the six gradient rows on
// three groups of threads while half the CUs have nothing, two strikes a thread where one fills them
// and a half and most of the second ones exist. Kernel, us:
// split / plain / two strikes, 33 strikes a chain with gradients, J = 4,096, at 24, 96, 192, 384, 768,
// 3,000 groups: 56/65/80, 62/68/82, 70/71/84, 129/93/91, 195/140/124, 761/530/410; 5 strikes, 1,000
// groups 271/196/224. 512 calibration chains, whose 676 groups of J up to 4,096 count as fewer than 384:
// whole call 306 us, 318 with two strikes a thread.
struct SumShape {
    uint32_t strike_block;
    bool split_rows;
};
SumShape sum_shape(const hexo_ctx* ctx, uint64_t blocks, uint64_t n_strikes, uint32_t n_chains) {
    const uint64_t cus = (uint64_t)ctx->prop.multiProcessorCount;
    const bool two = 2 * blocks > 3 * cus && n_strikes > 16ull * n_chains;
    return {two ? hexo::kSwiftStrikeBlock2 : hexo::kSwiftStrikeBlock, 2 * blocks <= cus};
}

// The most chains of a pass. A pass is three kernels in a row, each with its own end on a half-empty
// chip: 5,000 chains of 30 strikes with gradients 1,754, 1,598, 1,500 us at 256, 512, 1,024 large
// (and four times as many small) ones, 2,000 of 21 755, 666, 581.
constexpr uint32_t kBigPass = 1024, kSmallPass = 4096;

// Quarter octaves of the size estimate, the longest last, from kSizeBig (640) on chains that may
// exceed kSwiftSmallJ: the estimate is within a factor of 2 of J / 1.3 for nearly all, and of 6,000
// calibration chains none with J = 2,048 was below 678. One that is after all runs once more.
constexpr int kSizeClasses = 64, kSizeBig = 24;
int size_class(double size) {
    auto octave4 = [](double x) {
        uint64_t b;
        std::memcpy(&b, &x, 8);
        return (int64_t)(b >> 50);  // exponent and the top two bits of the mantissa
    };
    return (int)std::clamp<int64_t>(octave4(size) - octave4(640.0) + kSizeBig, 0, kSizeClasses - 1);
}

// Chains whose transforms exceed the LDS (J > kSwiftFftMaxJ), given their grids, through the direct
// sums. idx: the chains; results go to their places in the pinned arrays.
// Called with the context locked, its stream idle.
int price_large(hexo_ctx* ctx, const hexo_swift_request* reqs, const std::vector<uint32_t>& idx,
                const std::vector<hexo_swift_grid>& grids, const std::vector<uint64_t>& strike_off, uint64_t n_strk,
                const double* h_strikes, double* h_prices, double* h_grads) {
    auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    hipStream_t st = ctx->stream;
    const uint32_t n = (uint32_t)idx.size(), rows = h_grads ? 6u : 1u;
    std::vector<hexo::DevSwift> recs(n);
    std::vector<hexo::SwiftTable> tables;
    std::vector<uint64_t> ends(2 * (size_t)n);  // j, dens
    std::vector<uint32_t> blk_chain, blk_strike;
    uint64_t n_pay = 0, n_dens = 0, n_pm = 0, n_blocks = 0, n_own = 0;
    for (uint32_t i : idx) {
        n_blocks += (reqs[i].n_strikes + hexo::kSwiftStrikeBlock - 1u) / hexo::kSwiftStrikeBlock;
        n_own += reqs[i].n_strikes;
    }
    const SumShape shape = sum_shape(ctx, n_blocks, n_own, n);
    hexo::SwiftTotals tot{0, 0, 0};
    for (uint32_t i = 0; i < n; ++i) {
        const hexo_swift_request& q = reqs[idx[i]];
        const hexo_swift_grid& g = grids[idx[i]];
        hexo::DevSwift& R = recs[i];
        std::memset(&R, 0, sizeof(R));
        R.p[0] = q.v0;
        R.p[1] = q.theta;
        R.p[2] = q.rho;
        R.p[3] = q.kappa;
        R.p[4] = q.sigma;
        R.S0 = q.S0;
        R.r = q.r;
        R.T = q.T;
        R.disc = std::exp(-q.r * q.T);
        R.n_strikes = q.n_strikes;
        R.rows = rows;
        R.strike_off = strike_off[idx[i]];
        R.out_off = strike_off[idx[i]];
        R.exp2_m = (double)g.exp2_m;
        R.sqrt_exp2_m = g.sqrt_exp2_m;
        R.lower = g.lower;
        R.upper = g.upper;
        R.k1 = g.k1;
        R.k2 = g.k2;
        R.J = g.J;
        // one twiddle table per distinct J
        size_t t = 0;
        while (t < tables.size() && tables[t].J != g.J) ++t;
        if (t == tables.size()) {
            tables.push_back(hexo::SwiftTable{g.J, 0, tot.tw});
            tot.tw += 4ull * g.J;
        }
        R.tw_off = tables[t].off;
        R.pay_off = n_pay;
        R.coeff_off = n_pay;
        R.dens_off = n_dens;
        R.pm_off = n_pm;
        const uint64_t nk = (uint64_t)((int64_t)g.k2 - (int64_t)g.k1 + 1);
        tot.dens += nk;
        n_pay += g.J;
        n_dens += nk;
        n_pm += (uint64_t)rows * g.J;
        tot.j += g.J;
        for (uint32_t o = 0; o < q.n_strikes; o += shape.strike_block) {
            blk_chain.push_back(i);
            blk_strike.push_back(o);
        }
        ends[i] = tot.j;
        ends[n + i] = tot.dens;
    }
    std::vector<uint64_t> tab_end(tables.size());
    for (size_t t = 0; t < tables.size(); ++t) tab_end[t] = tables[t].off + 4ull * tables[t].J;
    const uint32_t n_tab = (uint32_t)tables.size();
    const size_t b_strk = align(8 * n_strk), b_recs = align(sizeof(hexo::DevSwift) * n),
                 b_tabs = align(sizeof(hexo::SwiftTable) * n_tab), b_tabend = align(8 * (size_t)n_tab),
                 b_ends = align(sizeof(uint64_t) * 2 * (size_t)n), b_blk = align(4 * blk_chain.size()), b_tw = align(16 * tot.tw), b_pay = align(16 * n_pay),
                 b_dens = align(8 * n_dens), b_coeff = align(16 * n_pay), b_pm = align(16 * n_pm);
    const size_t in_bytes = b_recs + b_tabs + b_tabend + b_ends + 2 * b_blk;
    // device: [tables | strikes | work arrays]
    const size_t total = in_bytes + b_strk + b_tw + b_pay + b_dens + b_coeff + b_pm;
    if (!ctx->swift_large_host.reserve(in_bytes)) return ctx->set_error(HEXO_ERR_NOMEM, "hipHostMalloc failed");
    if (int rc = grow_device(ctx, ctx->swift_dev, ctx->swift_dev_bytes, total)) return rc;
    unsigned char* host = reinterpret_cast<unsigned char*>(ctx->swift_large_host.p);
    std::memset(host, 0, in_bytes);
    size_t off = 0;
    std::memcpy(host + off, recs.data(), sizeof(hexo::DevSwift) * n);
    off += b_recs;
    std::memcpy(host + off, tables.data(), sizeof(hexo::SwiftTable) * n_tab);
    off += b_tabs;
    std::memcpy(host + off, tab_end.data(), 8 * (size_t)n_tab);
    off += b_tabend;
    std::memcpy(host + off, ends.data(), sizeof(uint64_t) * 2 * (size_t)n);
    off += b_ends;
    std::memcpy(host + off, blk_chain.data(), 4 * blk_chain.size());
    off += b_blk;
    std::memcpy(host + off, blk_strike.data(), 4 * blk_strike.size());
    unsigned char* dev = reinterpret_cast<unsigned char*>(ctx->swift_dev);
    hexo::SwiftArgs a{};
    off = 0;
    a.reqs = reinterpret_cast<const hexo::DevSwift*>(dev + off);
    a.n_req = n;
    off += b_recs;
    a.tables = reinterpret_cast<const hexo::SwiftTable*>(dev + off);
    a.n_tables = n_tab;
    off += b_tabs;
    a.tab_end = reinterpret_cast<const uint64_t*>(dev + off);
    off += b_tabend;
    const uint64_t* d_ends = reinterpret_cast<const uint64_t*>(dev + off);
    a.j_end = d_ends;
    a.dens_end = d_ends + n;
    off += b_ends;
    a.block_chain = reinterpret_cast<const uint32_t*>(dev + off);
    off += b_blk;
    a.block_strike = reinterpret_cast<const uint32_t*>(dev + off);
    a.n_blocks = (uint32_t)blk_chain.size();
    a.strike_block = shape.strike_block;
    a.split_rows = shape.split_rows;
    off += b_blk;
    double* d_strikes = reinterpret_cast<double*>(dev + off);
    a.strikes = d_strikes;
    off += b_strk;
    a.tw = reinterpret_cast<hexo::Cplx*>(dev + off);
    off += b_tw;
    a.pay = reinterpret_cast<hexo::Cplx*>(dev + off);
    off += b_pay;
    a.dens = reinterpret_cast<double*>(dev + off);
    off += b_dens;
    a.coeff = reinterpret_cast<hexo::Cplx*>(dev + off);
    off += b_coeff;
    a.pm = reinterpret_cast<hexo::Cplx*>(dev + off);
    a.prices = h_prices;
    a.grads = h_grads;
    if (hexo::launch_swift_stage(host, dev, in_bytes, h_strikes, d_strikes, b_strk, st) != hipSuccess ||
        hexo::launch_swift_large(a, tot, st) != hipSuccess || hipStreamSynchronize(st) != hipSuccess) {
        (void)hipStreamSynchronize(st);
        return ctx->set_error(HEXO_ERR_HIP, "SWIFT launch failed");
    }
    return HEXO_OK;
}

}  // namespace

extern "C" int hexo_swift_price(hexo_ctx* ctx, const hexo_swift_request* reqs, uint32_t n, double* prices, double* grads,
                                hexo_swift_grid* grids_used) {
    if (!ctx) return HEXO_ERR_INVALID;
    if (!reqs || !prices || n == 0) return ctx->set_error(HEXO_ERR_INVALID, "requests and prices must be non-NULL");
    std::string err;
    std::vector<uint64_t> strike_off(n);
    uint64_t n_strk = 0, n_blocks = 0;
    for (uint32_t i = 0; i < n; ++i) {
        int rc = check_chain(reqs[i], err);
        if (!rc && (reqs[i].flags & HEXO_SWIFT_FIXED_GRID)) rc = check_grid(reqs[i].grid, err);
        if (rc) return ctx->set_error(rc, "swift request " + std::to_string(i) + ": " + err);
        strike_off[i] = n_strk;
        n_strk += reqs[i].n_strikes;
        n_blocks += (reqs[i].n_strikes + hexo::kSwiftStrikeBlock - 1u) / hexo::kSwiftStrikeBlock;
    }
    if (n_blocks >= (1ull << 31)) return ctx->set_error(HEXO_ERR_INVALID, "too many strikes in one call");
    std::lock_guard<std::recursive_mutex> lock(ctx->mu);
    if (hipSetDevice(ctx->device) != hipSuccess) return ctx->set_error(HEXO_ERR_HIP, "hipSetDevice failed");
    auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    hipStream_t st = ctx->stream;
    // The kernels read their inputs from and write the grids and results to two fine-grained pinned
    // stages, in place: [strikes | chains | chain order] and [grids | prices | gradients].
    const size_t b_strk = align(8 * n_strk), b_chain = align(sizeof(hexo::SwiftChainIn) * n), b_blk = align(4 * n_blocks);
    const size_t b_grid = align(sizeof(hexo::SwiftGridOut) * n), b_prices = align(8 * n_strk);
    if (!ctx->swift_in_host.reserve(b_strk + b_chain + 4 * (size_t)n) ||
        !ctx->swift_host.reserve(b_grid + b_prices + (grads ? 40 * n_strk : 0)))
        return ctx->set_error(HEXO_ERR_NOMEM, "hipHostMalloc failed");
    unsigned char* in = reinterpret_cast<unsigned char*>(ctx->swift_in_host.p);
    unsigned char* out = reinterpret_cast<unsigned char*>(ctx->swift_host.p);
    double* h_strikes = reinterpret_cast<double*>(in);
    hexo::SwiftChainIn* chains = reinterpret_cast<hexo::SwiftChainIn*>(in + b_strk);
    uint32_t* order = reinterpret_cast<uint32_t*>(in + b_strk + b_chain);
    hexo::SwiftGridOut* gout = reinterpret_cast<hexo::SwiftGridOut*>(out);
    double* h_prices = reinterpret_cast<double*>(out + b_grid);
    double* h_grads = grads ? reinterpret_cast<double*>(out + b_grid + b_prices) : nullptr;
    for (uint32_t i = 0; i < n; ++i) {
        const hexo_swift_request& q = reqs[i];
        std::memcpy(h_strikes + strike_off[i], q.strikes, 8 * q.n_strikes);
        hexo::SwiftChainIn& c = chains[i];
        c = hexo::SwiftChainIn{{q.v0, q.theta, q.rho, q.kappa, q.sigma}, q.T, q.r, q.S0, q.trunc, std::exp(-q.r * q.T),
                               strike_off[i], 0, q.n_strikes, (q.flags & HEXO_SWIFT_FIXED_GRID) ? 1u : 0u, q.grid};
    }
    // More chains than CUs: by size, the longest transforms first (J ranges over a factor of 32 in a
    // calibration batch, and one of 4,096 begun last holds up the rest), and those that will not
    // exceed kSwiftSmallJ several to a CU. The others' chain of kernels is as long as the rest of the
    // batch takes, so it runs beside it on a stream of its own.
    // Sorted into quarter octaves of the estimate only: comparing 5,000 chains took 160 us of the host.
    const bool sorted = n > (uint32_t)ctx->prop.multiProcessorCount;
    uint32_t n_big = n;
    std::vector<uint8_t> key(sorted ? n : 0);
    if (sorted) {
        uint32_t count[kSizeClasses] = {}, first[kSizeClasses];
        for (uint32_t i = 0; i < n; ++i) ++count[key[i] = (uint8_t)size_class(size_estimate(reqs[i]))];
        uint32_t at = 0;
        for (int k = kSizeClasses - 1; k >= 0; at += count[k--]) {
            first[k] = at;
            if (k == kSizeBig) n_big = at + count[k];
        }
        for (uint32_t i = 0; i < n; ++i) order[first[key[i]]++] = i;
    }
    auto fail = [&](int code, const std::string& msg) {
        // drain what was queued before the pinned stages are reused
        (void)hipStreamSynchronize(st);
        if (ctx->swift_stream) (void)hipStreamSynchronize(ctx->swift_stream);
        return ctx->set_error(code, msg);
    };
    if (!ctx->swift_roots) {
        if (hipMalloc(&ctx->swift_roots, sizeof(hexo::Cplx) * 4 * hexo::kSwiftFftMaxJ) != hipSuccess) {
            ctx->swift_roots = nullptr;
            return ctx->set_error(HEXO_ERR_NOMEM, "hipMalloc failed");
        }
        // (read on both streams, so it has to be complete)
        if (hexo::launch_swift_roots(static_cast<hexo::Cplx*>(ctx->swift_roots), st) != hipSuccess ||
            hipStreamSynchronize(st) != hipSuccess) {
            (void)hipFree(ctx->swift_roots);
            ctx->swift_roots = nullptr;
            return fail(HEXO_ERR_HIP, "SWIFT launch failed");
        }
    }
    if (n_big && n_big < n && !ctx->swift_stream &&
        hipStreamCreateWithFlags(&ctx->swift_stream, hipStreamNonBlocking) != hipSuccess) {
        ctx->swift_stream = nullptr;
        return ctx->set_error(HEXO_ERR_HIP, "hipStreamCreate failed");
    }
    // Work arrays of each class for a pass of the call's chains, each chain with room for the largest J of
    // its class: no second look at J, and the two streams share nothing that is written. At most
    // 2 x 470 MB with gradients, 2 x 134 MB without. (How many chains each class gets changes from call to
    // call of a calibration; n does not.)
    const uint32_t rows = grads ? 6u : 1u;
    const uint32_t big_pass = std::min(n, kBigPass), small_pass = std::min(n, kSmallPass);
    const size_t row_bytes[2] = {sizeof(hexo::Cplx) * hexo::kSwiftFftMaxJ * big_pass,
                                 n_big < n ? sizeof(hexo::Cplx) * hexo::kSwiftSmallJ * small_pass : 0};
    const size_t b_recs[2] = {align(sizeof(hexo::DevSwift) * big_pass), align(sizeof(hexo::DevSwift) * small_pass)};
    if (int rc = grow_device(ctx, ctx->swift_dev, ctx->swift_dev_bytes,
                             b_strk + 2 * b_blk + b_recs[0] + b_recs[1] + (row_bytes[0] + row_bytes[1]) * (1 + rows)))
        return rc;
    unsigned char* dev = reinterpret_cast<unsigned char*>(ctx->swift_dev);
    double* dev_strikes = reinterpret_cast<double*>(dev);
    uint32_t* block_chain = reinterpret_cast<uint32_t*>(dev + b_strk);
    uint32_t* block_strike = reinterpret_cast<uint32_t*>(dev + b_strk + b_blk);
    // the next pass of a class of chains, order[k .. end), its contraction workgroups numbered from blk on
    uint32_t blk = 0;
    auto run = [&](int small, uint32_t& k, uint32_t end, hipStream_t s) {
        const uint32_t m = std::min(end - k, small ? small_pass : big_pass), b0 = blk;
        SumShape shape{hexo::kSwiftStrikeBlock, false};
        if (small) {
            // Two strikes a thread where the call would already fill the device with one (2 workgroups a
            // CU) and most of the second ones exist. 1,000 chains of J = 512 and 64 strikes with gradients:
            // 107 us instead of 147.
            if (n_blocks > 2ull * ctx->prop.multiProcessorCount && n_strk > 16ull * n)
                shape.strike_block = hexo::kSwiftStrikeBlock2;
        } else if (sorted) {
            uint64_t blocks[kSizeClasses] = {}, strikes = 0;
            for (uint32_t i = k; i < k + m; ++i) {
                const uint32_t ns = chains[order[i]].n_strikes;
                blocks[key[order[i]]] += (ns + hexo::kSwiftStrikeBlock - 1u) / hexo::kSwiftStrikeBlock;
                strikes += ns;
            }
            double longest = 0.0;
            for (int c = 0; c <= key[order[k]]; ++c)
                longest += (double)blocks[c] * std::exp2(0.25 * (c - key[order[k]]));
            shape = sum_shape(ctx, (uint64_t)longest, strikes, m);
        }
        hexo::SwiftChainArgs c{};
        c.chains = chains;
        c.order = sorted ? order + k : nullptr;
        c.strikes = h_strikes;
        c.roots = static_cast<const hexo::Cplx*>(ctx->swift_roots);
        c.grids = gout;
        c.dev_strikes = dev_strikes;
        c.block_chain = block_chain;
        c.block_strike = block_strike;
        c.recs = reinterpret_cast<hexo::DevSwift*>(dev + b_strk + 2 * b_blk + (small ? b_recs[0] : 0));
        c.coeff = reinterpret_cast<hexo::Cplx*>(dev + b_strk + 2 * b_blk + b_recs[0] + b_recs[1] + (small ? row_bytes[0] * (1 + rows) : 0));
        c.n_req = m;
        c.max_J = small ? hexo::kSwiftSmallJ : hexo::kSwiftFftMaxJ;
        c.rows = rows;
        c.strike_block = shape.strike_block;
        for (uint32_t i = k; i < k + m; ++i) {
            hexo::SwiftChainIn& q = chains[sorted ? order[i] : i];
            q.block_off = blk;
            blk += (q.n_strikes + c.strike_block - 1u) / c.strike_block;
        }
        k += m;
        hexo::SwiftArgs a{};
        a.reqs = c.recs;
        a.n_req = m;
        a.strikes = dev_strikes;
        a.block_chain = block_chain + b0;
        a.block_strike = block_strike + b0;
        a.n_blocks = blk - b0;
        a.strike_block = c.strike_block;
        a.split_rows = shape.split_rows;
        a.coeff = c.coeff;
        a.pm = c.coeff + row_bytes[small] / sizeof(hexo::Cplx);
        a.prices = h_prices;
        a.grads = h_grads;
        return hexo::launch_swift_transform(c, s) == hipSuccess && hexo::launch_swift_prices(a, c.max_J, s) == hipSuccess;
    };
    // the two classes' passes in turn, so that both streams have work from the start
    const bool beside = n_big && n_big < n;
    bool ok = true;
    for (uint32_t big = 0, small = n_big; ok && (big < n_big || small < n);) {
        if (big < n_big) ok = run(0, big, n_big, beside ? ctx->swift_stream : st);
        if (ok && small < n) ok = run(1, small, n, st);
    }
    if (!ok || (beside && hipStreamSynchronize(ctx->swift_stream) != hipSuccess) || hipStreamSynchronize(st) != hipSuccess)
        return fail(HEXO_ERR_HIP, "SWIFT launch failed");
    // chains that were larger than their class
    uint32_t missed = 0;
    for (uint32_t k = n_big; k < n; ++k)
        if (gout[order[k]].status == hexo::kSwiftGridOk && gout[order[k]].g.J > hexo::kSwiftSmallJ &&
            gout[order[k]].g.J <= hexo::kSwiftFftMaxJ)
            order[missed++] = order[k];
    blk = 0;
    for (uint32_t k = 0; ok && k < missed;) ok = run(0, k, missed, st);
    if (!ok || (missed && hipStreamSynchronize(st) != hipSuccess)) return fail(HEXO_ERR_HIP, "SWIFT launch failed");
    std::vector<hexo_swift_grid> grids(n);
    std::vector<uint32_t> large;
    for (uint32_t i = 0; i < n; ++i) {
        int rc = grid_status(gout[i].status, gout[i].J_wanted, err);
        if (!rc) rc = check_grid(grids[i] = gout[i].g, err);
        if (rc) return ctx->set_error(rc, "swift request " + std::to_string(i) + ": " + err);
        if (grids[i].J > hexo::kSwiftFftMaxJ) large.push_back(i);
    }
    if (!large.empty())
        if (int rc = price_large(ctx, reqs, large, grids, strike_off, n_strk, h_strikes, h_prices, h_grads)) return rc;
    std::memcpy(prices, h_prices, 8 * n_strk);
    if (grads) std::memcpy(grads, h_grads, 40 * n_strk);
    if (grids_used) std::memcpy(grids_used, grids.data(), sizeof(hexo_swift_grid) * n);
    return HEXO_OK;
}
