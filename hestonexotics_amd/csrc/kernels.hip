// kernels.hip -- HIP kernels of the Heston QE Monte-Carlo path for gfx950.
//
// k_path_fp32  fused FP32 path kernel: Philox4x32-10 -> inverse normal -> QE step -> Asian/European
//              finalisation -> per-tile payoff sums. Replaces the reference's OpenMP path loop
//              and scheme (src/HSimulation.tpp:23-49, :52-86), the option policies
//              (src/inc/AsianContract.h:25-47, src/inc/VanillaContract.h:24-39) and the RNG ring
//              refills (src/RNG.cpp:28-43, src/as241.f90:85-118).
// k_path_fp32_split  the same paths with the draws and the steps on different waves, for batches
//              that leave k_path_fp32's persistent grid short of work.
// k_path_fp64, k_path_fp64_split  the plain FP64 kernel, the same path in the reference's own FP64
//              form, and its division into drawing and stepping waves for small batches.
// k_reduce_*   cross-tile reduction in a fixed order and the estimator (price, standard error);
//              replaces the racy `prices[...] +=` of src/HSimulation.tpp:40,47-48.
//
// Work distribution: a persistent grid of independent wavefronts. Each wave takes a work item
// (request, PPT consecutive 64-path tiles) from an atomic queue; items are ordered longest request
// first. Lane l of the wave runs path tile*64 + l of each of its PPT tiles. At every expiry the
// wave transposes its paths' (A, X_T) through LDS so that lanes work over (option, 8-path group)
// pairs; each tile's sums therefore depend only on its 64 paths, never on the launch shape.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"
#include "layout.hpp"

// No implicit FMA contraction in this file: every fused multiply-add is written out. With contraction
// the compiler fuses a product into a later add only where both land in one basic block, which depends
// on how each instance of a kernel is laid out (one FP32 path per thread flattens the quadratic branch
// and turned tt - 1 into fma(m^2, 1/s2h, -1); a branch added to the FP64 step changed which of its
// sums were fused), so results would change by an ulp with the launch shape or the batch that a
// request is in.
#pragma clang fp contract(off)

namespace hexo {

namespace {

constexpr uint32_t kEuropean = 2u;
constexpr uint32_t kAsianGeoCV = 4u;
constexpr uint32_t kGeoAsian = 8u;
constexpr uint32_t kTrapezoid = 4u;
constexpr uint32_t kMartingale = 8u;
constexpr uint32_t kCvRegression = 16u;
constexpr uint32_t kPrecFP64 = 0u;
constexpr uint32_t kPrecComp = 2u;

__device__ __forceinline__ void wave_sync_lds() {
    // LDS traffic of one wave is processed in order; this keeps the compiler from moving the
    // transpose's reads above its writes.
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// Work item -> (sorted request position). item_end is a prefix sum over the sorted requests.
__device__ __forceinline__ uint32_t find_sorted(const uint32_t* item_end, uint32_t n, uint32_t item) {
    uint32_t lo = 0, hi = n - 1;
    while (lo < hi) {
        const uint32_t mid = (lo + hi) >> 1;
        if (item_end[mid] > item)
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo;
}

// Takes the wave's next work item. Every lane executes the atomic (lane 0 adds 1, the others 0)
// and the wave keeps lane 0's ticket, so there is no divergent region around the atomic: with
// `if (lane == 0) atomicAdd(...)` followed by a broadcast, the loop structurizer may move the
// broadcast into a loop that lanes 1..63 re-enter without lane 0, repeating one item forever.
__device__ __forceinline__ uint32_t next_item(uint32_t* counter, int lane) {
    const uint32_t old = atomicAdd(counter, lane == 0 ? 1u : 0u);
    return uniform(old);
}

// Compensated (Neumaier) FP32 accumulation.
struct CompF {
    float s, c;
    __device__ __forceinline__ void add(float x) {
        const float t = s + x;
        c += (__builtin_fabsf(s) >= __builtin_fabsf(x)) ? (s - t) + x : (x - t) + s;
        s = t;
    }
    // x^2 enters every sum unrounded. (Fused by the compiler in some of them only, a wave's first square
    // had its rounding error counted twice: standard errors off by 1.1e-8 on average, now 4.9e-9.)
    __device__ __forceinline__ void add_square(float x) {
        const float t = __builtin_fmaf(x, x, s);
        c += (__builtin_fabsf(s) >= x * x) ? __builtin_fmaf(x, x, s - t) : __builtin_fmaf(x, x, -t) + s;
        s = t;
    }
    __device__ __forceinline__ void merge(float s2, float c2) {
        const float t = s + s2;
        const float e = (__builtin_fabsf(s) >= __builtin_fabsf(s2)) ? (s - t) + s2 : (s2 - t) + s;
        s = t;
        c = c + c2 + e;
    }
};

// Per-expiry tile reduction. vals[j*64 + p] holds (A, X_T) of path p of sub-tile j (in the
// kernel's units); paths beyond n_paths hold values whose payoff is 0 (FP32: -inf; FP64: masked).
// Output o of the request is payoff-major: o = pay * n_opts + option. The summation order of a
// tile's 64 payoffs depends only on the number of strikes of the expiry (a property of the
// request), never on the launch shape:
//  * many strikes (>= kWideStrikes): lane i takes strike i and sums the 64 paths in path order,
//    reading each path's values as an LDS broadcast;
//  * few strikes: lane (o = lane/8, g = lane%8) sums paths 8g..8g+7 of output o in path order and
//    the 8 group sums are combined by a fixed xor tree.
constexpr uint32_t kWideStrikes = 48;

template <typename Acc>
struct TileSums;

template <>
struct TileSums<double> {  // FP64 sums (HEXO_FP32 and the FP64 kernel)
    double s = 0.0, ss = 0.0;
    __device__ __forceinline__ void add(double x) {
        s += x;
        ss = __builtin_fma(x, x, ss);
    }
    __device__ __forceinline__ void combine(const TileSums& o) {
        s += o.s;
        ss += o.ss;
    }
    __device__ __forceinline__ void poison() { s = ss = __builtin_nan(""); }
    __device__ __forceinline__ void load(const void* partials, size_t slot) {
        const double2 v = reinterpret_cast<const double2*>(partials)[slot];
        s = v.x;
        ss = v.y;
    }
    __device__ __forceinline__ void tree8() {
#pragma unroll
        for (int m = 1; m < 8; m <<= 1) {
            s += __shfl_xor(s, m);
            ss += __shfl_xor(ss, m);
        }
    }
    __device__ __forceinline__ void store(void* partials, size_t slot) const {
        reinterpret_cast<double2*>(partials)[slot] = make_double2(s, ss);
    }
    __device__ __forceinline__ TileSums of_lane(int l) const {
        TileSums t;
        t.s = __shfl(s, l);
        t.ss = __shfl(ss, l);
        return t;
    }
};

template <>
struct TileSums<float> {  // compensated FP32 sums (HEXO_FP32_COMPENSATED)
    CompF s{0.f, 0.f}, ss{0.f, 0.f};
    __device__ __forceinline__ void add(float x) {
        s.add(x);
        ss.add_square(x);
    }
    __device__ __forceinline__ void combine(const TileSums& o) {
        s.merge(o.s.s, o.s.c);
        ss.merge(o.ss.s, o.ss.c);
    }
    __device__ __forceinline__ void poison() { s = ss = CompF{__builtin_nanf(""), 0.0f}; }
    __device__ __forceinline__ void load(const void* partials, size_t slot) {
        const float4 v = reinterpret_cast<const float4*>(partials)[slot];
        s = CompF{v.x, v.y};
        ss = CompF{v.z, v.w};
    }
    __device__ __forceinline__ void tree8() {
#pragma unroll
        for (int m = 1; m < 8; m <<= 1) {
            const float s2 = __shfl_xor(s.s, m), c2 = __shfl_xor(s.c, m);
            const float q2 = __shfl_xor(ss.s, m), d2 = __shfl_xor(ss.c, m);
            s.merge(s2, c2);
            ss.merge(q2, d2);
        }
    }
    __device__ __forceinline__ void store(void* partials, size_t slot) const {
        reinterpret_cast<float4*>(partials)[slot] = make_float4(s.s, s.c, ss.s, ss.c);
    }
    __device__ __forceinline__ TileSums of_lane(int l) const {
        TileSums t;
        t.s = CompF{__shfl(s.s, l), __shfl(s.c, l)};
        t.ss = CompF{__shfl(ss.s, l), __shfl(ss.c, l)};
        return t;
    }
};

// The level of the chunk tree ((t0 + t1) + (t2 + t3)) that N consecutive tiles of one chunk form
// (layout.hpp, kChunkTiles): t0 for one tile, t0 + t1 for two, the whole tree for four.
template <int N, typename Acc>
__device__ __forceinline__ TileSums<Acc> chunk_level(TileSums<Acc> (&t)[N]) {
    static_assert(N == 1 || N == 2 || N == kChunkTiles, "tiles per stored partial: 1, 2 or 4");
    if constexpr (N >= 2) t[0].combine(t[1]);
    if constexpr (N == 4) {
        t[2].combine(t[3]);
        t[0].combine(t[2]);
    }
    return t[0];
}

// Payoff kind of output block `pay` of a request: the pay-th set bit of its payoffs (outputs are
// payoff-major in bit order: Asian, European, Asian with the geometric control variate, the
// geometric call).
__device__ __forceinline__ uint32_t payoff_kind(uint32_t payoffs, uint32_t pay) {
    uint32_t b = payoffs;
    for (uint32_t i = 0; i < pay; ++i) b &= b - 1u;
    return b & (~b + 1u);
}

// Payoff of one path for strike K and payoff kind. Path values: the FP32 kernel's float2 (A, X_T)
// or float4 (A, X_T, G, -) in units of S0, paths beyond n_paths holding -inf; the FP64 kernel's
// double4 (A, X_T, G, -) with an explicit validity flag. The control-variate payoff is the
// arithmetic minus the geometric call payoff. max(., 0) turns a NaN value into 0: tiles holding a
// NaN value are marked by the path kernel instead (NanBits) and their sums set to NaN.
__device__ __forceinline__ float payoff_of(float2 v, uint32_t kind, float K, bool) {
    return __builtin_fmaxf((kind == kEuropean ? v.y : v.x) - K, 0.0f);
}
__device__ __forceinline__ float payoff_of(float4 v, uint32_t kind, float K, bool) {
    const float pg = __builtin_fmaxf(v.z - K, 0.0f);
    const float pa = __builtin_fmaxf((kind == kEuropean ? v.y : v.x) - K, 0.0f);
    return kind == kGeoAsian ? pg : kind == kAsianGeoCV ? pa - pg : pa;
}
__device__ __forceinline__ double payoff_of(double4 v, uint32_t kind, double K, bool valid) {
    const double pg = __builtin_fmax(v.z - K, 0.0);
    const double pa = __builtin_fmax((kind == kEuropean ? v.y : v.x) - K, 0.0);
    const double pay = kind == kGeoAsian ? pg : kind == kAsianGeoCV ? pa - pg : pa;
    return valid ? pay : 0.0;
}

// NaN marks of a wave's tiles at one expiry, wave-uniform: bit 3j + c is set when a path of tile j
// (within n_paths) has a NaN value in component c (0: A, 1: X_T, 2: G). A path whose price left the
// floating-point range (inf - inf in the finalisation) has one; the sums of every output of the
// tile that reads that component are then NaN, as the NaN payoff would have made them, instead of
// silently dropping the path.
struct NanBits {
    uint32_t bits = 0;
    __device__ __forceinline__ void mark(int j, bool valid, float A, float xt, float G) {
        const bool na = valid && A != A, nx = valid && xt != xt, ng = valid && G != G;
        bits |= (__builtin_amdgcn_ballot_w64(na) ? 1u : 0u) << (3 * j);
        bits |= (__builtin_amdgcn_ballot_w64(nx) ? 2u : 0u) << (3 * j);
        bits |= (__builtin_amdgcn_ballot_w64(ng) ? 4u : 0u) << (3 * j);
    }
    __device__ __forceinline__ void mark(int j, bool valid, double A, double xt, double G) {
        const bool na = valid && A != A, nx = valid && xt != xt, ng = valid && G != G;
        bits |= (__builtin_amdgcn_ballot_w64(na) ? 1u : 0u) << (3 * j);
        bits |= (__builtin_amdgcn_ballot_w64(nx) ? 2u : 0u) << (3 * j);
        bits |= (__builtin_amdgcn_ballot_w64(ng) ? 4u : 0u) << (3 * j);
    }
    // whether outputs of payoff `kind` of tile j read a NaN value
    __device__ __forceinline__ bool hit(int j, uint32_t kind) const {
        const uint32_t c = kind == kEuropean ? 2u : kind == kGeoAsian ? 4u : kind == kAsianGeoCV ? 5u : 1u;
        return ((bits >> (3 * j)) & c) != 0u;
    }
};

// Stores a wave's PPT tile sums of output o: the chunk tree's level for PPT tiles (1, 2 or 4), or,
// for 3 paths per thread (which does not divide a chunk), every tile's own sum, from which the
// group reduction builds the same tree.
template <int PPT, typename Acc>
__device__ __forceinline__ void store_tile_sums(const PathArgs& a, const DevReq& R, uint32_t tile0, uint32_t n_out,
                                                uint32_t o, bool active, TileSums<Acc> (&t)[PPT]) {
    if constexpr (kChunkTiles % PPT == 0) {
        const TileSums<Acc> c = chunk_level<PPT, Acc>(t);
        if (active) c.store(a.partials, (size_t)R.partial_base + (size_t)(tile0 / PPT) * n_out + o);
    } else {
#pragma unroll
        for (int j = 0; j < PPT; ++j)
            if (active && tile0 + (uint32_t)j < R.n_tiles)
                t[j].store(a.partials, (size_t)R.partial_base + (size_t)(tile0 + (uint32_t)j) * n_out + o);
    }
}

template <int PPT, typename ValT, typename Acc>
__device__ __forceinline__ void reduce_tiles_impl(const PathArgs& a, const DevReq& R, const DevFin& F,
                                                  uint32_t tile0, int lane, const ValT* vals, NanBits nan) {
    using KT = decltype(ValT{}.x);
    const uint32_t nk = F.n_strikes;
    const uint32_t n_out = R.n_opts * R.n_pay;
    for (uint32_t pay = 0; pay < R.n_pay; ++pay) {
        const uint32_t kind = payoff_kind(R.payoffs, pay);  // wave-uniform
        if (nk >= kWideStrikes) {
            for (uint32_t kb = 0; kb < nk; kb += kTile) {
                const uint32_t kj = kb + (uint32_t)lane;
                const bool active = kj < nk;
                const DevOpt& opt = a.opts[R.opt_begin + F.opt_begin + (active ? kj : 0u)];
                const KT K = sizeof(KT) == 4 ? (KT)opt.k_rel : (KT)opt.k_abs;
                const uint32_t o = pay * R.n_opts + F.opt_begin + kj;
                TileSums<Acc> t[PPT];
#pragma unroll
                for (int j = 0; j < PPT; ++j) {
                    const uint32_t tile = tile0 + (uint32_t)j;
                    if (tile >= R.n_tiles) continue;  // absent tiles are zero sums
                    const uint64_t nv = R.n_paths - (uint64_t)tile * kTile;
                    for (int p = 0; p < kTile; ++p)
                        t[j].add((Acc)payoff_of(vals[j * kTile + p], kind, K, (uint64_t)p < nv));
                    if (nan.hit(j, kind)) t[j].poison();
                }
                store_tile_sums<PPT, Acc>(a, R, tile0, n_out, o, active, t);
            }
        } else {
            const int g = lane & 7;
            for (uint32_t kb = 0; kb < nk; kb += 8) {
                const uint32_t kj = kb + (uint32_t)(lane >> 3);
                const bool active = kj < nk;
                const DevOpt& opt = a.opts[R.opt_begin + F.opt_begin + (active ? kj : 0u)];
                const KT K = sizeof(KT) == 4 ? (KT)opt.k_rel : (KT)opt.k_abs;
                const uint32_t o = pay * R.n_opts + F.opt_begin + kj;
                TileSums<Acc> t[PPT];
#pragma unroll
                for (int j = 0; j < PPT; ++j) {
                    const uint32_t tile = tile0 + (uint32_t)j;
                    if (tile >= R.n_tiles) continue;  // absent tiles are zero sums
                    const uint64_t nv = R.n_paths - (uint64_t)tile * kTile;
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const int p = g * 8 + i;
                        t[j].add((Acc)payoff_of(vals[j * kTile + p], kind, K, (uint64_t)p < nv));
                    }
                    t[j].tree8();  // every lane of the 8-lane group ends with the same bits
                    if (nan.hit(j, kind)) t[j].poison();
                }
                store_tile_sums<PPT, Acc>(a, R, tile0, n_out, o, g == 0 && active, t);
            }
        }
    }
}

template <int PPT, typename ValT>
__device__ __forceinline__ void reduce_tiles(const PathArgs& a, const DevReq& R, const DevFin& F, uint32_t tile0,
                                             int lane, const ValT* vals, NanBits nan) {
    if (std::is_same<decltype(ValT{}.x), float>::value && R.precision == kPrecComp)
        reduce_tiles_impl<PPT, ValT, float>(a, R, F, tile0, lane, vals, nan);
    else
        reduce_tiles_impl<PPT, ValT, double>(a, R, F, tile0, lane, vals, nan);
}

__device__ __forceinline__ void count_flush(unsigned long long* counts, uint32_t c0, uint32_t c1, uint32_t c2,
                                            uint32_t c3, int lane) {
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) {
        c0 += __shfl_xor(c0, m);
        c1 += __shfl_xor(c1, m);
        c2 += __shfl_xor(c2, m);
        c3 += __shfl_xor(c3, m);
    }
    // all lanes hold the wave total after the butterfly; only lane 0 contributes it (no divergent region)
    const bool first = lane == 0;
    atomicAdd(&counts[0], first ? (unsigned long long)c0 : 0ull);
    atomicAdd(&counts[1], first ? (unsigned long long)c1 : 0ull);
    atomicAdd(&counts[2], first ? (unsigned long long)c2 : 0ull);
    atomicAdd(&counts[3], first ? (unsigned long long)c3 : 0ull);
}

// ------------------------------------------------------------------------------------------
// FP32 path kernel
// ------------------------------------------------------------------------------------------
struct SegF {
    float omd, th, c1h, c2h, g0, ka, kb, k3;
    float mA, ma, mh, mr;
};

// Per-wave LDS scratch of the FP32 kernel: the transpose of the per-path values at expiries, 4 words
// per path ((A, X_T) or, with the geometric payoffs, (A, X_T, G, -)).
template <int PPT>
struct WaveLds {
    static constexpr int kWords = 4 * PPT * kTile;  // 32-bit words
};

struct StepCount {
    uint32_t quad = 0, exp = 0, central = 0, tail = 0;
};

// The step's conditional moments from V (src/HSimulation.tpp:58-62): d0 = th - V, m = V + omd d0
// (exactly th at V = th, whatever the roundings), s2h = s2 / 2 (from the halved constants: the
// same bits as s2, scaled), m^2, tt = 2 / psi = m^2 / s2h and the branch: quadratic when
// psi < 1.5, i.e. tt > 4/3. tt is formed before the branch because the quadratic branch starts
// from it; the exponential branch does not use it.
template <int PPT>
__device__ __forceinline__ void qe_moments_fp32(const float (&V)[PPT], const SegF& c, float (&d0)[PPT],
                                                float (&m)[PPT], float (&s2h)[PPT], float (&m2)[PPT],
                                                float (&tt)[PPT], bool (&quad)[PPT]) {
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        d0[j] = c.th - V[j];
        m[j] = __builtin_fmaf(c.omd, d0[j], V[j]);
        s2h[j] = __builtin_fmaf(V[j], c.c1h, c.c2h);
        m2[j] = m[j] * m[j];
        tt[j] = m2[j] * __builtin_amdgcn_rcpf(s2h[j]);  // finite by the FP32 validation bound
        quad[j] = tt[j] > 4.0f / 3.0f;
    }
}

// The update of one step given its moments and normals: the variance by the quadratic branch
// a (b + Z_V)^2 or the exponential branch, then the log-price step (MART: Andersen's
// martingale-corrected form, falling back per path and step to the plain step where
// E[exp(A V')] does not exist; GEO: also Y before the step and the run's sum of Y).
//
// FLAT evaluates the quadratic branch on every lane and enters one branch per step, for the lanes in
// the exponential one, instead of two per path. The stepping waves of the split kernel run it (1e6
// stiff paths with the martingale correction x 512 steps: 1.80 ms against 2.05); at the persistent
// kernel's issue limit it costs 2% (64 uneven requests 5.18 ms against 5.07).
template <bool FLAT, int PPT, bool MART, bool GEO>
__device__ __forceinline__ void qe_update_fp32(float (&V)[PPT], float (&Y)[PPT], float (&X)[PPT], float (&Xp)[PPT],
                                               float (&P)[PPT], float (&Yp)[PPT], float (&PY)[PPT],
                                               const uint32_t (&wv)[PPT], const float (&zv)[PPT],
                                               const float (&zx)[PPT], const float (&d0)[PPT], const float (&m)[PPT],
                                               const float (&s2h)[PPT], const float (&m2)[PPT], const float (&tt)[PPT],
                                               const bool (&quad)[PPT], const SegF& c) {
    // One path's draw: dm = V' - m and, MART: A m - ln E[exp(A V')] = fs f(ft) + corr with
    // f(t) = t - ln(1 + t), in natural log units; mok: the expectation exists
    struct Draw {
        float dm, ft = 0.0f, fs = 0.0f, corr = 0.0f;
        bool mok = false;
    };
    auto quadratic = [&](int j, Draw& o) __attribute__((always_inline)) {
        const float tm1 = tt[j] - 1.0f;
        const float b2 = tm1 + __builtin_amdgcn_sqrtf(tt[j] * tm1);
        const float b = __builtin_amdgcn_sqrtf(b2);
        // V' = a (b + Z)^2 with a = m / (1 + b^2), taken as V' - m = a (Z (Z + 2 b) - 1): its
        // mean is 0 whatever the rounding of a and b, so the scheme's E[V'] = m holds exactly
        // (a biased mean would move the variance's mean-reversion level by (bias) / (kappa dt))
        const float aq = m[j] * __builtin_amdgcn_rcpf(__builtin_fmaf(b, b, 1.0f));
        // near b + Z = 0, m + (V' - m) can round a few ulp of m below 0 where a (b + Z)^2 is
        // >= 0: harmless to the moments, and the diffusion below takes |k3 (V + V')|
        o.dm = aq * __builtin_fmaf(zv[j], __builtin_fmaf(2.0f, b, zv[j]), -1.0f);
        if constexpr (MART) {
            // x = 2 A a < 1: A m - ln E[exp(A V')] = -(f(-x) + x^2 b^2 / (1 - x)) / 2
            const float x = (c.mA + c.mA) * aq;
            o.mok = x < 1.0f;
            o.ft = -x;
            o.fs = -0.5f;
            o.corr = -0.5f * (x * x) * b2 * __builtin_amdgcn_rcpf(1.0f - x);
        }
    };
    auto exponential = [&](int j, Draw& o) __attribute__((always_inline)) {
        // p = (psi-1)/(psi+1), beta = 2/(m (psi+1)); V' = ln((1-p)/(1-U))/beta if U > p, else 0.
        // With sm = s2 + m^2: 1-p = 2m^2/sm and 1/beta = sm/(2m).
        const float sm = __builtin_fmaf(2.0f, s2h[j], m2[j]);
        // (1-U) sm, 1 - U from ~k; the complement is taken here (asm: not hoisted in front of the
        // branch, where every lane would pay for it; the wait state as at the asm helpers in
        // device.hpp)
        uint32_t nk;
        asm("s_nop 0\n\tv_not_b32 %0, %1" : "=v"(nk) : "v"(wv[j]));
        const float lhs = uniform_f32(nk) * sm;
        const float tm2 = m2[j] + m2[j];
        const float lg = __builtin_amdgcn_logf(tm2 * rcp_refined(lhs));
        const float ib = sm * rcp_refined(m[j]);  // 2 / beta
        const float v = ib * (0.5f * 0.693147180559945309f) * lg;
        // U > p exactly when (1-p)/(1-U) > 1, i.e. when the log is positive: V' = max(v, 0)
        o.dm = __builtin_fmaxf(v, 0.0f) - m[j];
        if constexpr (MART) {
            // cA = A / beta < 1, r1 = (1-p) / (1 - cA) = 2 m^2 / (sm (1 - cA)), y = r1 cA:
            // A m - ln E[exp(A V')] = f(y) - r1 cA^2
            const float cA = (0.5f * c.mA) * ib;
            o.mok = cA < 1.0f;
            const float r1 = tm2 * __builtin_amdgcn_rcpf(__builtin_fmaf(-cA, sm, sm));
            o.ft = r1 * cA;
            o.fs = 1.0f;
            o.corr = -o.ft * cA;
        }
    };
    Draw flat[FLAT ? PPT : 1];
    if constexpr (FLAT) {
        bool any_exp = false;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            quadratic(j, flat[j]);
            any_exp |= !quad[j];
        }
        if (__builtin_amdgcn_ballot_w64(any_exp)) {
#pragma unroll
            for (int j = 0; j < PPT; ++j)
                if (!quad[j]) exponential(j, flat[j]);
        }
    }
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        Draw o;
        if constexpr (FLAT)
            o = flat[j];
        else if (quad[j])
            quadratic(j, o);
        else
            exponential(j, o);
        const float dm = o.dm, ft = o.ft, fs = o.fs, corr = o.corr;
        const bool mok = o.mok;
        // The reference's log-price step multiplies V' - V by rho/sigma and V + V' - 2 th by
        // kappa rho dt / (2 sigma). As differences of FP32 variances they would carry ulp(V) errors
        // amplified by 1/sigma (prices tens of percent off at sigma = 1e-6, or at sigma = 1e-4
        // with dt = 2e-7). Written on V' - m and th - V, each term has its own size:
        // K1 V + K2 V' = (K1 + K2) th + K2 (V' - m) - (K1 + K2 e^{-kappa dt}) (th - V), the first
        // part in g0, the coefficients ka = K2 and kb (O(dt), formed in FP64) in the segment.
        const float Vn = m[j] + dm;
        const float sum = V[j] + Vn;
        float inc = __builtin_fmaf(c.ka, dm, __builtin_fmaf(c.kb, d0[j], c.g0));
        if constexpr (MART) {
            // f(t) = t - ln(1 + t): its series through t^7 for |t| < 1/16 (relative error < 2e-8),
            // else from the rounded 1 + t. The direct form alone would return f = t wherever 1 + t
            // rounds to 1, a one-signed error of up to 6e-8 per step where t stays small.
            const float t2 = ft * ft;
            float h = __builtin_fmaf(ft, -1.0f / 7.0f, 1.0f / 6.0f);
            h = __builtin_fmaf(ft, h, -0.2f);
            h = __builtin_fmaf(ft, h, 0.25f);
            h = __builtin_fmaf(ft, h, -1.0f / 3.0f);
            h = __builtin_fmaf(ft, h, 0.5f);
            const float fdir = __builtin_fmaf(-0.693147180559945309f, __builtin_amdgcn_logf(1.0f + ft), ft);
            const float f = __builtin_fabsf(ft) < 0.0625f ? t2 * h : fdir;
            const float cl = __builtin_fmaf(fs, f, corr) * 1.44269504088896341f;
            const float im = __builtin_fmaf(c.ma, dm, __builtin_fmaf(-c.mh, sum, c.mr)) + cl;
            inc = mok ? im : inc;
        }
        const float sq = __builtin_amdgcn_sqrtf(__builtin_fabsf(c.k3 * sum));
        if constexpr (GEO) Yp[j] = Y[j];
        Y[j] = __builtin_fmaf(sq, zx[j], Y[j] + inc);
        Xp[j] = X[j];
        X[j] = __builtin_amdgcn_exp2f(Y[j]);
        P[j] += X[j];
        if constexpr (GEO) PY[j] += Y[j];
        V[j] = Vn;
    }
}

// Branch statistics (COUNT): quad / exp per step; central / tail per normal drawn (Z_V only where
// the variance branch is quadratic).
__device__ __forceinline__ void count_step(StepCount& cnt, bool valid, bool quad, bool tv, bool tx) {
    if (!valid) return;
    cnt.quad += quad ? 1u : 0u;
    cnt.exp += quad ? 0u : 1u;
    cnt.central += (quad && !tv ? 1u : 0u) + (tx ? 0u : 1u);
    cnt.tail += (quad && tv ? 1u : 0u) + (tx ? 1u : 0u);
}

// One QE step for the PPT paths of a lane (Andersen's QE scheme as in src/HSimulation.tpp:52-86):
// the normals Z_V (quadratic lanes only: the exponential branch reads the word as a uniform) and
// Z_X, then the update. Y is log2(X/S0); X = 2^Y; P accumulates X for the Asian sum.
template <int PPT, bool COUNT, bool MART, bool GEO>
__device__ __forceinline__ void qe_step_fp32(float (&V)[PPT], float (&Y)[PPT], float (&X)[PPT], float (&Xp)[PPT],
                                             float (&P)[PPT], float (&Yp)[PPT], float (&PY)[PPT],
                                             const uint32_t (&wv)[PPT], const uint32_t (&wx)[PPT],
                                             const SegF& c, const bool (&valid)[PPT], StepCount& cnt,
                                             const NormalVregs& nv) {
    float d0[PPT], m[PPT], s2h[PPT], m2[PPT], tt[PPT], zv[PPT], zx[PPT];
    bool quad[PPT];
    qe_moments_fp32<PPT>(V, c, d0, m, s2h, m2, tt, quad);
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        bool tv, tx;
        // Z_V with its tail polynomial wherever the word needs it, also on the rare exponential-
        // branch lanes that do not read it: the branch on the quadratic test then comes once, at
        // the variance update, instead of also in front of the tail polynomial
        zv[j] = normal_word_f32(wv[j], true, nv, tv);
        zx[j] = normal_word_f32(wx[j], true, nv, tx);
        if constexpr (COUNT) count_step(cnt, valid[j], quad[j], tv, tx);
    }
    qe_update_fp32<false, PPT, MART, GEO>(V, Y, X, Xp, P, Yp, PY, wv, zv, zx, d0, m, s2h, m2, tt, quad, c);
}

// Philox4x32-10 (device.hpp philox4x32_10) of the path counter {blk, plo, phi, 0} with the step
// pair blk, the path's high word phi and the key wave-uniform. The rounds are the same; the values
// that stay wave-uniform through the first three rounds are marked so (readfirstlane), which keeps
// their products on the scalar unit: both of round 1's, one each of rounds 2 and 3.
__device__ __forceinline__ u32x4 philox_path(uint32_t blk, uint32_t plo, uint32_t phi, uint32_t k0, uint32_t k1) {
    // round 1: c0 = blk, c2 = phi, c3 = 0 uniform
    uint64_t p0 = (uint64_t)kPhiloxM0 * blk, p1 = (uint64_t)kPhiloxM1 * phi;
    uint32_t c0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), plo, k0, 0x96);
    uint32_t c1 = uniform((uint32_t)p1);
    uint32_t c2 = uniform((uint32_t)(p0 >> 32)) ^ uniform(k1);
    uint32_t c3 = uniform((uint32_t)p0);
    k0 += kPhiloxW0;
    k1 += kPhiloxW1;
    // round 2: c2 uniform; the new c0 and c1 are uniform
    p0 = (uint64_t)kPhiloxM0 * c0;
    p1 = (uint64_t)kPhiloxM1 * c2;
    c0 = uniform((uint32_t)(p1 >> 32)) ^ c1 ^ uniform(k0);
    c1 = uniform((uint32_t)p1);
    c2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
    c3 = (uint32_t)p0;
    k0 += kPhiloxW0;
    k1 += kPhiloxW1;
    // round 3: c0 uniform; the new c3 is uniform
    p0 = (uint64_t)kPhiloxM0 * c0;
    p1 = (uint64_t)kPhiloxM1 * c2;
    c0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
    c1 = (uint32_t)p1;
    c2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
    c3 = uniform((uint32_t)p0);
    k0 += kPhiloxW0;
    k1 += kPhiloxW1;
#pragma unroll
    for (int r = 3; r < 10; ++r) {
        p0 = (uint64_t)kPhiloxM0 * c0;
        p1 = (uint64_t)kPhiloxM1 * c2;
        const uint32_t n0 = __builtin_amdgcn_bitop3_b32((uint32_t)(p1 >> 32), c1, k0, 0x96);
        const uint32_t n2 = __builtin_amdgcn_bitop3_b32((uint32_t)(p0 >> 32), c3, k1, 0x96);
        c0 = n0;
        c1 = (uint32_t)p1;
        c2 = n2;
        c3 = (uint32_t)p0;
        k0 += kPhiloxW0;
        k1 += kPhiloxW1;
    }
    return u32x4{c0, c1, c2, c3};
}

template <int PPT>
__device__ __forceinline__ void philox_block(uint32_t blk, const uint32_t (&plo)[PPT], const uint32_t (&phi)[PPT],
                                             uint32_t key0, uint32_t key1, uint32_t (&w0)[PPT], uint32_t (&w1)[PPT],
                                             uint32_t (&w2)[PPT], uint32_t (&w3)[PPT]) {
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        const u32x4 r = philox_path(blk, plo[j], phi[j], key0, key1);
        w0[j] = r.x;
        w1[j] = r.y;
        w2[j] = r.z;
        w3[j] = r.w;
    }
}

// A chunk's draws in the split kernel (below), step-major: (Z_V, Z_X) and the word of Z_V (the
// exponential branch's uniform).
template <uint32_t C>
struct DrawChunk {
    float2 z[C][kTile];
    uint32_t w[C][kTile];
};
template <>
struct DrawChunk<0> {};

__device__ __forceinline__ void workgroup_sync_lds() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// The paths of a lane through the request's runs. C = 0: the draws are made here, a counter block per
// two steps; else they come in chunks of C steps from the drawing waves (PPT = 1).
template <uint32_t C, int PPT, bool DEBUG, bool COUNT, bool MART, bool GEO>
__device__ __forceinline__ void path_fp32(const PathArgs& a, uint32_t ri, uint32_t tile0, int lane, uint32_t* lds,
                                          const DrawChunk<C>* buf = nullptr) {
    const DevReq& R = a.reqs[ri];
    const uint64_t n_paths = R.n_paths;
    const uint32_t key0 = R.seed_lo, key1 = R.seed_hi;
    float V[PPT], Y[PPT], X[PPT], Xp[PPT], P[PPT], acc[PPT], Xs[PPT];
    float Yp[PPT], PY[PPT], accY[PPT], Ys[PPT];  // GEO: the same accumulation on Y = log2(X/S0)
    uint32_t plo[PPT], phi[PPT], sv[PPT], sx[PPT];
    bool valid[PPT];
    StepCount cnt;
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
        const uint64_t pl = (uint64_t)(tile0 + (uint32_t)j) * kTile + (uint64_t)lane;
        valid[j] = pl < n_paths;
        const uint64_t gp = R.path_offset + pl;
        plo[j] = (uint32_t)gp;
        // path_offset is a multiple of 64, so a tile never straddles 2^32: the high word is
        // wave-uniform and the first Philox rounds run partly on the scalar unit
        phi[j] = uniform((uint32_t)((R.path_offset + (uint64_t)(tile0 + (uint32_t)j) * kTile) >> 32));
        V[j] = R.v0_f;
        Y[j] = 0.0f;
        X[j] = 1.0f;
        Xp[j] = 1.0f;
        P[j] = 0.0f;
        acc[j] = 0.0f;
        Xs[j] = 1.0f;
        Yp[j] = PY[j] = accY[j] = Ys[j] = 0.0f;
        sv[j] = sx[j] = 0u;
    }
    const NormalVregs nv = normal_vregs();
    uint32_t k = 0;  // global step index; step k uses words 2k, 2k+1 of the path's stream
    const uint32_t n_segs = R.n_segs;
    for (uint32_t s = 0; s < n_segs; ++s) {
        const DevSeg& S = a.segs[R.seg_begin + s];
        const SegF c{S.omd, S.th, S.c1h, S.c2h, S.g0, S.ka, S.kb, S.k3, S.mA, S.ma, S.mh, S.mr};
        const uint32_t n = S.n_steps;
        if constexpr (C == 0) {
            uint32_t i = 0;
            if ((k & 1u) && n > 0) {  // second half of a block opened by the previous run
                qe_step_fp32<PPT, COUNT, MART, GEO>(V, Y, X, Xp, P, Yp, PY, sv, sx, c, valid, cnt, nv);
                ++i;
                ++k;
            }
            for (; i + 2 <= n; i += 2, k += 2) {
                uint32_t w0[PPT], w1[PPT], w2[PPT], w3[PPT];
                philox_block<PPT>(k >> 1, plo, phi, key0, key1, w0, w1, w2, w3);
                qe_step_fp32<PPT, COUNT, MART, GEO>(V, Y, X, Xp, P, Yp, PY, w0, w1, c, valid, cnt, nv);
                qe_step_fp32<PPT, COUNT, MART, GEO>(V, Y, X, Xp, P, Yp, PY, w2, w3, c, valid, cnt, nv);
            }
            if (i < n) {
                uint32_t w0[PPT], w1[PPT];
                philox_block<PPT>(k >> 1, plo, phi, key0, key1, w0, w1, sv, sx);
                qe_step_fp32<PPT, COUNT, MART, GEO>(V, Y, X, Xp, P, Yp, PY, w0, w1, c, valid, cnt, nv);
                ++k;
            }
        } else {
            auto step = [&](float2 z, uint32_t w) {
                float d0[1], m[1], s2h[1], m2[1], tt[1];
                bool quad[1];
                qe_moments_fp32<1>(V, c, d0, m, s2h, m2, tt, quad);
                const uint32_t wv[1] = {w};
                const float zv[1] = {z.x}, zx[1] = {z.y};
                qe_update_fp32<true, 1, MART, GEO>(V, Y, X, Xp, P, Yp, PY, wv, zv, zx, d0, m, s2h, m2, tt, quad, c);
            };
            for (uint32_t left = n; left;) {
                const uint32_t at = k % C;
                if (at == 0) workgroup_sync_lds();
                const DrawChunk<C>& d = buf[k / C % 2u];
                if (at == 0 && left >= C) {  // a whole chunk: its draws in registers, no loop
                    float2 z[C];
                    uint32_t w[C];
#pragma unroll
                    for (uint32_t t = 0; t < C; ++t) {
                        z[t] = d.z[t][lane];
                        w[t] = d.w[t][lane];
                    }
#pragma unroll
                    for (uint32_t t = 0; t < C; ++t) step(z[t], w[t]);
                    k += C;
                    left -= C;
                } else {
                    const uint32_t end = min(C, at + left);
                    for (uint32_t t = at; t < end; ++t) step(d.z[t][lane], d.w[t][lane]);
                    k += end - at;
                    left -= end - at;
                }
            }
        }
        // Asian accumulation of the run's interior steps b..e-1:
        // delta * (X_{b-1}/2 + X_b + ... + X_{e-2} + X_{e-1}/2) = delta * (P - X_e + (Xs - Xp)/2)
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            acc[j] = __builtin_fmaf(S.delta_f, (P[j] - X[j]) + 0.5f * (Xs[j] - Xp[j]), acc[j]);
            if constexpr (GEO) accY[j] = __builtin_fmaf(S.delta_f, (PY[j] - Y[j]) + 0.5f * (Ys[j] - Yp[j]), accY[j]);
        }
        // per-path values at an expiry: (A, X_T), with GEO (A, X_T, G, -); the wave's LDS region
        // holds 4 words per path either way
        using Val = typename std::conditional<GEO, float4, float2>::type;
        Val* vals = reinterpret_cast<Val*>(lds);
        for (uint32_t f = 0; f < S.fin_count; ++f) {
            const DevFin& F = a.fins[S.fin_begin + f];
            const float w = F.w_f, invT = F.invT_f;
            NanBits nan;
#pragma unroll
            for (int j = 0; j < PPT; ++j) {
                const float dX = X[j] - Xp[j];
                const float xt = __builtin_fmaf(dX, w, Xp[j]);
                const float A = (R.flags & kTrapezoid) ? (acc[j] + F.hwdt_f * (Xp[j] + xt)) * invT
                                                       : __builtin_fmaf(dX, w, acc[j]) * invT;
                // paths beyond n_paths carry -inf: every payoff max(0, . - K) is then 0
                if constexpr (GEO) {
                    // the same functional on Y, normalised by its weight sum W: G/S0 = W 2^(L/W)
                    const float dY = Y[j] - Yp[j];
                    const float L = (R.flags & kTrapezoid)
                                        ? (accY[j] + F.hwdt_f * (Yp[j] + __builtin_fmaf(dY, w, Yp[j]))) * invT
                                        : __builtin_fmaf(dY, w, accY[j]) * invT;
                    const float G = F.gW_f * __builtin_amdgcn_exp2f(L * F.gInvW_f);
                    vals[j * kTile + lane] =
                        valid[j] ? make_float4(A, xt, G, 0.0f) : make_float4(-INFINITY, -INFINITY, -INFINITY, 0.0f);
                    nan.mark(j, valid[j], A, xt, G);
                } else {
                    vals[j * kTile + lane] = valid[j] ? make_float2(A, xt) : make_float2(-INFINITY, -INFINITY);
                    nan.mark(j, valid[j], A, xt, 0.0f);
                }
                if constexpr (DEBUG) {
                    if (valid[j] && a.finals) {
                        const uint64_t pl = (uint64_t)(tile0 + (uint32_t)j) * kTile + (uint64_t)lane;
                        double* out = a.finals + (pl * R.n_exp + F.chain) * 2;
                        out[0] = (double)A * R.S0;
                        out[1] = (double)xt * R.S0;
                    }
                }
            }
            wave_sync_lds();
            reduce_tiles<PPT>(a, R, F, tile0, lane, vals, nan);
            wave_sync_lds();
        }
        const float hn = 0.5f * S.dnext_f;
#pragma unroll
        for (int j = 0; j < PPT; ++j) {
            acc[j] = __builtin_fmaf(hn, X[j] + Xp[j], acc[j]);
            Xs[j] = X[j];
            P[j] = 0.0f;
            if constexpr (GEO) {
                accY[j] = __builtin_fmaf(hn, Y[j] + Yp[j], accY[j]);
                Ys[j] = Y[j];
                PY[j] = 0.0f;
            }
        }
    }
    if constexpr (COUNT) count_flush(a.counts, cnt.quad, cnt.exp, cnt.central, cnt.tail, lane);
}

// The workgroup's LDS, aligned for path_fp32's values of an expiry. Without the geometric average these are
// float2: declared 16-byte aligned, its reads of two of them become single 16-byte ones, and the 512
// uneven requests take 682.5 ms against 676.5.
template <bool GEO>
__device__ __forceinline__ uint32_t* path_lds() {
    if constexpr (GEO) {
        extern __shared__ __align__(16) uint32_t lds_16[];
        static_assert(__alignof__(lds_16) >= alignof(float4));
        return lds_16;
    } else {
        extern __shared__ __align__(8) uint32_t lds_8[];
        static_assert(__alignof__(lds_8) >= alignof(float2));
        return lds_8;
    }
}

// Registers for 5 waves per SIMD at 2 paths per lane (96), 4 with the martingale step: it needs 114,
// and held to 96 it spilled 22 (4e6 paths x 252 steps 2.58 -> 2.48 ms, 2^20 stiff paths x 2,048 steps
// 7.15 -> 6.90). With the geometric average as well it spills as much, but its payoff sums want
// the fifth wave more (1,000 strikes x 3 payoffs x 52 steps, 3.5e6 paths 3.79 -> 3.30 ms with it).
template <int PPT, bool DEBUG, bool COUNT, bool MART, bool GEO>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(PPT == 2 && (!MART || GEO) ? 5 : 4, 8))) void k_path_fp32(PathArgs a) {
    const int lane = (int)(threadIdx.x & 63u);
    // the wave's LDS region, at a wave-uniform address
    uint32_t* lds = path_lds<GEO>() + uniform(threadIdx.x >> 6) * WaveLds<PPT>::kWords;
    for (;;) {
        const uint32_t item = next_item(a.counter, lane);
        if (item >= a.total_items) break;
        const uint32_t sp = uniform(find_sorted(a.item_end, a.n_sorted, item));
        const uint32_t first = sp ? a.item_end[sp - 1] : 0u;
        const uint32_t ri = uniform(a.order[sp]);
        path_fp32<0, PPT, DEBUG, COUNT, MART, GEO>(a, ri, uniform((item - first) * (uint32_t)PPT), lane, lds);
    }
}
// ------------------------------------------------------------------------------------------
// FP32 path kernel with drawing and stepping waves
// ------------------------------------------------------------------------------------------
// One workgroup per 64-path tile. NP waves draw the normals of a chunk of C steps (Philox and the
// inverse normals, 57 of a step's 100 instructions) into one LDS buffer while the stepping wave
// runs the variance and log-price recursion over the chunk before it from the other.
//
// Why: a wave alone issues one vector instruction in 6.5 to 7.7 cycles however independent they are
// (1 or 2 paths per lane: 720 and 670 cycles per path-step, 86 instructions), a SIMD needs four or
// five waves to reach its 3.1; and a request's time axis cannot be split, so a batch of up to
// 5 waves x 2 tiles per SIMD (650,000 paths) left k_path_fp32 short of waves or of work for its last
// round. Here a tile is two or three waves, each with its part of the step. Kernel times, k_path_fp32
// (2 paths per lane) against this one, base parameters x 252 steps: 1e4 paths 144 -> 34 us,
// 1e5 159 -> 97, 4e5 323 -> 234, 1e6 593 -> 541; martingale step 2e5 paths 245 -> 176 us;
// the 8 x 64 grid at 1e6 paths 1802 -> 1718 us. The stepping wave's priority is raised: the tile
// waits for it (400k paths 240 -> 234 us, the grid at a quarter of its paths 501 -> 478).
// Drawing wave `part` of NP: counter blocks part, part + NP, ... of every chunk. Every wave of the
// workgroup meets ceil(n_steps / C) barriers: here after each chunk drawn, in the stepping wave
// before each chunk stepped, so that a buffer is rewritten only after its chunk has been consumed.
template <uint32_t NP, uint32_t C>
__device__ __forceinline__ void draw_fp32(const DevReq& R, uint32_t tile, int lane, uint32_t part, DrawChunk<C>* buf) {
    static_assert(C % (2 * NP) == 0, "whole counter blocks per wave and chunk");
    const uint64_t first = R.path_offset + (uint64_t)tile * kTile;  // tiles never straddle 2^32
    const uint32_t plo = (uint32_t)first + (uint32_t)lane, phi = uniform((uint32_t)(first >> 32));
    const uint32_t key0 = R.seed_lo, key1 = R.seed_hi, n_steps = R.n_steps;
    const NormalVregs nv = normal_vregs();
    for (uint32_t k = 0, c = 0; k < n_steps; k += C, ++c) {
        DrawChunk<C>& d = buf[c & 1u];
#pragma unroll
        for (uint32_t b = 0; b < C / 2; b += NP) {
            const uint32_t t = 2 * (b + part);  // the block's first step; past n_steps the draws are unused
            const u32x4 r = philox_path((k + t) >> 1, plo, phi, key0, key1);
            const uint32_t w[4] = {r.x, r.y, r.z, r.w};
            float z[4];
            normals_f32<4>(w, z, nv);
            d.z[t][lane] = make_float2(z[0], z[1]);
            d.w[t][lane] = w[0];
            d.z[t + 1][lane] = make_float2(z[2], z[3]);
            d.w[t + 1][lane] = w[2];
        }
        workgroup_sync_lds();
    }
}

// A wave's role in its workgroup of n waves: 0 steps, the others draw. The stepping wave's place
// varies with the tile, so that the waves of one role do not gather on the same SIMDs.
__device__ __forceinline__ uint32_t stepping_first(uint32_t wave, uint32_t item, uint32_t n) {
    return (wave + (uint32_t)__builtin_popcount(item * 0x9E3779B1u >> 16)) % n;
}

template <uint32_t NP, uint32_t C, bool MART, bool GEO>
__global__ __launch_bounds__(64 * (NP + 1)) void k_path_fp32_split(PathArgs a) {
    __shared__ DrawChunk<C> buf[2];
    __shared__ __align__(16) uint32_t vals[WaveLds<1>::kWords];
    static_assert(__alignof__(vals) >= alignof(float4), "path_fp32 stores float4 there");
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t item = blockIdx.x;
    const uint32_t sp = uniform(find_sorted(a.item_end, a.n_sorted, item));
    const uint32_t tile = uniform(item - (sp ? a.item_end[sp - 1] : 0u));
    const uint32_t ri = uniform(a.order[sp]);
    const uint32_t role = stepping_first(uniform(threadIdx.x >> 6), item, NP + 1);
    if (role == 0) {
        __builtin_amdgcn_s_setprio(2);
        path_fp32<C, 1, false, false, MART, GEO>(a, ri, tile, lane, vals, buf);
    } else {
        draw_fp32<NP, C>(a.reqs[ri], tile, lane, role - 1, buf);
    }
}
// ------------------------------------------------------------------------------------------
// Plain FP64 path kernel: the reference's step and policies in FP64 (src/HSimulation.tpp:52-86) with
// the expressions that depend on the run only (e^-kappa dt, the variance's coefficients, K0..K4)
// taken from the run's record.
//
// Bound by FP64 issue (4 cycles per wave instruction, 16 per v_rcp/v_rsq_f64): about 1,200 cycles
// per wave and step at 3 waves per SIMD. With the constants recomputed every step, the library's
// division, root, exp and log and the tail normals evaluated for every word it was 2,700: 1e6
// paths x 252 steps 4.93 -> 2.11 ms, 1e5 x 252 0.715 -> 0.382 ms (kernel, base parameters), a
// 64-request batch of daily steps 42.9 -> 19.1 ms. Held to 4 waves per SIMD (128 registers) the
// constants spill and it is 10% slower at 1e6 paths, 25% at 1e5.
// ------------------------------------------------------------------------------------------
struct SegD {
    double e, s2v, s2c, k0, k1, k2, k3, delta;
};

__device__ __forceinline__ bool qe_step_fp64(const DevReq& R, const SegD& c, double& V, double& logX, uint32_t wv,
                                             double zv, double zx) {
    const double m = __builtin_fma(V - R.theta, c.e, R.theta);
    const double s2 = __builtin_fabs(__builtin_fma(V, c.s2v, c.s2c));
    const double m2 = m * m;
    const double Vp = V;
    const bool quad = s2 < 1.5 * m2;  // psi = s2 / m^2 < 1.5
    const bool tiny = s2 < 1e-290;    // so that (s2 + m^2)(1 - U) is normal where this is false
    double aq = 0.0, bp2 = 0.0, sm = 0.0;
    const auto variance = [&](auto div) {
        if (quad) {
            const double tt = div(m2 + m2, s2);  // 2 / psi
            const double tm1 = tt - 1.0;
            bp2 = tm1 + sqrt_f64(tt * tm1);
            aq = div_f64(m, 1.0 + bp2);
            const double bz = sqrt_f64(bp2) + zv;
            V = aq * bz * bz;
        } else {
            // p = (psi - 1)/(psi + 1), beta = 2/(m (psi + 1)): with sm = s2 + m^2, 1 - p = 2 m^2/sm and
            // 1/beta = sm/(2 m). U > p exactly when arg = (1 - p)/(1 - U) > 1; 1 - U comes from ~k
            sm = s2 + m2;
            const double arg = div(m2 + m2, sm * uniform_f64(~wv));
            const double v = log_f64(arg) * div_f64(sm, m + m);
            V = arg > 1.0 ? v : 0.0;
        }
    };
    // div_f64's reciprocal of a subnormal divisor overflows. One test of the wave a step: one at each
    // division took 0.4% more (the 512 uneven requests' quarter of paths 779.8 against 772.7 ms, with
    // the martingale correction's condition below; 768 with no test)
    if (__builtin_amdgcn_ballot_w64(tiny))
        variance([&](double a, double b) {
            const double q = div_f64(a, b);
            return tiny ? a / b : q;
        });
    else
        variance([](double a, double b) { return div_f64(a, b); });
    double k0 = c.k0;
    if (R.flags & kMartingale) {
        // Andersen's martingale-corrected K0* = -ln E[exp(A V') | V] - (K1 + K3/2) V, A = K2 + K4/2
        const double A = __builtin_fma(0.5, c.k3, c.k2), K1h = __builtin_fma(0.5, c.k3, c.k1);
        double lnM = 0.0;
        bool exists;
        if (quad) {
            exists = 2.0 * A * aq < 1.0;
            lnM = A * bp2 * aq / (1.0 - 2.0 * A * aq) - 0.5 * ::log1p(-2.0 * A * aq);
        } else {
            const double beta = (m + m) / sm;
            const double omp = (m2 + m2) / sm;  // 1 - p
            // where m^2 and s2 underflow to 0 there is no psi and omp is NaN: the uncorrected step
            exists = A < beta && omp >= 0.0;
            lnM = ::log((1.0 - omp) + beta * omp / (beta - A));
        }
        if (exists) k0 = __builtin_fma(R.r_drift, c.delta, __builtin_fma(-K1h, Vp, -lnM));
    }
    // V = V' = 0 makes the diffusion's variance 0: the floor keeps the root finite and moves nothing
    const double var = __builtin_fmax(__builtin_fma(c.k3, Vp, c.k3 * V), 1e-300);
    logX = __builtin_fma(sqrt_f64(var), zx, __builtin_fma(c.k2, V, __builtin_fma(c.k1, Vp, logX + k0)));
    return quad;
}

__device__ __forceinline__ bool central_f64(uint32_t k) { return !is_tail_f64(centred_f64(k)); }

// The normals of a counter block's four words. The central rational runs on every lane; the tail
// (a logarithm, a root and another rational, 15% of the words, so that nearly every wave has a lane
// in it for every word) runs once for all four words: their tail words are queued in LDS, 38 of
// the 256 on average, and each lane takes one (`queue`: this wave's 256 slots of 8 bytes).
__device__ __forceinline__ void normals4_f64(const u32x4& w, double (&z)[4], double* queue, int lane) {
    const uint32_t k[4] = {w.x, w.y, w.z, w.w};
    double q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = centred_f64(k[i]);
    uint32_t* words = reinterpret_cast<uint32_t*>(queue);  // a slot's first half: the folded word
    uint32_t pos[4], n = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool t = is_tail_f64(q[i]);
        const uint64_t mask = __builtin_amdgcn_ballot_w64(t);
        pos[i] = __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, n));
        if (t) words[2 * pos[i]] = k[i] ^ (uint32_t)((int32_t)k[i] >> 31);
        n += (uint32_t)__builtin_popcountll(mask);
    }
    normals_central_f64(q, z);
    wave_sync_lds();
    for (uint32_t b = 0; b < n; b += kTile) {  // wave-uniform
        const uint32_t t = b + (uint32_t)lane;
        if (t < n) queue[t] = normal_tail_f64(words[2 * t]);
    }
    wave_sync_lds();
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (is_tail_f64(q[i])) z[i] = __builtin_copysign(queue[pos[i]], q[i]);
    wave_sync_lds();  // the slots are rewritten by the next block, or by the values of an expiry
}

// e^y; the fast form covers every price within e^+-700, the library's the rest.
__device__ __forceinline__ double price_exp_f64(double y) {
    double x = exp_f64(y);
    const bool out = !(__builtin_fabs(y) < 700.0);
    if (__builtin_amdgcn_ballot_w64(out)) x = out ? ::exp(y) : x;
    return x;
}

// A chunk's draws in the FP64 split kernel (below), as DrawChunk.
template <uint32_t C>
struct DrawChunk64 {
    double2 z[C][kTile];
    uint32_t w[C][kTile];
};
template <>
struct DrawChunk64<0> {};

template <uint32_t C, bool DEBUG, bool COUNT>
__device__ __forceinline__ void path_fp64(const PathArgs& a, uint32_t ri, uint32_t tile, int lane, double4* vals,
                                          const DrawChunk64<C>* buf = nullptr) {
    const DevReq& R = a.reqs[ri];
    const bool geo = (R.payoffs & (kAsianGeoCV | kGeoAsian)) != 0;  // wave-uniform
    double accY = 0.0, yp = 0.0;  // the Asian accumulation on y = ln(X/S0); y before the last step
    const uint64_t pl = (uint64_t)tile * kTile + (uint64_t)lane;
    const bool valid = pl < R.n_paths;
    const uint64_t gp = R.path_offset + pl;
    const uint32_t plo = (uint32_t)gp, phi = uniform((uint32_t)((R.path_offset + (uint64_t)tile * kTile) >> 32));
    double V = R.v0, logX = R.log_S0, X = R.S0, Xp = R.S0, acc = 0.0;
    double z[4] = {};  // the counter block's normals: Z_V, Z_X of its two steps
    u32x4 w{};
    uint32_t k = 0;
    uint32_t cq = 0, ce = 0, cc = 0, ct = 0;
    for (uint32_t s = 0; s < R.n_segs; ++s) {
        const DevSeg& S = a.segs[R.seg_begin + s];
        const SegD c{S.e, S.s2v, S.s2c, S.dk0, S.dk1, S.dk2, S.dk3, S.delta};
        const uint32_t n = S.n_steps;
        for (uint32_t i = 0; i < n; ++i, ++k) {
            if constexpr (C != 0) {
                if (k % C == 0) workgroup_sync_lds();
                const DrawChunk64<C>& d = buf[k / C % 2u];
                const double2 zz = d.z[k % C][lane];
                z[0] = zz.x;
                z[1] = zz.y;
                w.x = d.w[k % C][lane];
            } else if ((k & 1u) == 0u) {
                w = philox4x32_10(k >> 1, plo, phi, 0u, R.seed_lo, R.seed_hi);
                normals4_f64(w, z, reinterpret_cast<double*>(vals), lane);
            } else {
                w.x = w.z;
                w.y = w.w;
                z[0] = z[2];
                z[1] = z[3];
            }
            yp = logX - R.log_S0;
            const bool quad = qe_step_fp64(R, c, V, logX, w.x, z[0], z[1]);
            Xp = X;
            X = price_exp_f64(logX);
            if constexpr (COUNT) {
                if (valid) {
                    cq += quad ? 1u : 0u;
                    ce += quad ? 0u : 1u;
                    const bool cv = central_f64(w.x), cx = central_f64(w.y);
                    cc += (quad && cv ? 1u : 0u) + (cx ? 1u : 0u);
                    ct += (quad && !cv ? 1u : 0u) + (cx ? 0u : 1u);
                }
            }
            if (i + 1u < n) {
                acc = __builtin_fma(c.delta * 0.5, X + Xp, acc);  // AAsianCallNonAdaptive::accumulate_value
                if (geo) accY = __builtin_fma(c.delta * 0.5, (logX - R.log_S0) + yp, accY);
            }
        }
        for (uint32_t f = 0; f < S.fin_count; ++f) {
            const DevFin& F = a.fins[S.fin_begin + f];
            const double xt = Xp + (X - Xp) * (F.T - F.tp) / F.dt;
            const double A = (R.flags & kTrapezoid) ? (acc + (F.T - F.tp) * 0.5 * (Xp + xt)) / F.T
                                                    : (acc + (X - Xp) * (F.T - F.tp) / F.dt) / F.T;
            double G = 0.0;
            if (geo) {
                // the same functional on y, normalised by its weight sum W: G = W S0 exp(L / W)
                const double y = logX - R.log_S0, wf = (F.T - F.tp) / F.dt;
                const double yt = __builtin_fma(y - yp, wf, yp);
                const double L = (R.flags & kTrapezoid) ? (accY + (F.T - F.tp) * 0.5 * (yp + yt)) / F.T
                                                        : (accY + (y - yp) * wf) / F.T;
                G = F.gW * R.S0 * ::exp(L / F.gW);
            }
            vals[lane] = make_double4(A, xt, G, 0.0);
            NanBits nan;
            nan.mark(0, valid, A, xt, G);
            if constexpr (DEBUG) {
                if (valid && a.finals) {
                    double* out = a.finals + (pl * R.n_exp + F.chain) * 2;
                    out[0] = A;
                    out[1] = xt;
                }
            }
            wave_sync_lds();
            reduce_tiles<1>(a, R, F, tile, lane, vals, nan);
            wave_sync_lds();
        }
        acc = __builtin_fma(S.dnext * 0.5, X + Xp, acc);
        if (geo) accY = __builtin_fma(S.dnext * 0.5, (logX - R.log_S0) + yp, accY);
    }
    if constexpr (COUNT) count_flush(a.counts, cq, ce, cc, ct, lane);
}

template <bool DEBUG, bool COUNT>
__global__ __launch_bounds__(256) void k_path_fp64(PathArgs a) {
    extern __shared__ double4 lds_d4[];
    const int lane = (int)(threadIdx.x & 63u);
    double4* vals = lds_d4 + (threadIdx.x >> 6) * kTile;
    for (;;) {
        const uint32_t item = next_item(a.counter, lane);
        if (item >= a.total_items) break;
        const uint32_t sp = uniform(find_sorted(a.item_end, a.n_sorted, item));
        const uint32_t first = sp ? a.item_end[sp - 1] : 0u;
        const uint32_t ri = uniform(a.order[sp]);
        path_fp64<0, DEBUG, COUNT>(a, ri, uniform(item - first), lane, vals);
    }
}

// ------------------------------------------------------------------------------------------
// FP64 path kernel with drawing and stepping waves (k_path_fp32_split's division of a tile's work)
// ------------------------------------------------------------------------------------------
// A lone wave of k_path_fp64 takes 2,600 cycles per step, of which its SIMD needs 1,200 for the
// instructions: up to a few tiles per SIMD the time is the wave's. Drawing (half of the work) on
// waves of their own: 1e4 paths x 252 steps 272 -> 120 us, 5e4 286 -> 195, 1e5 385 -> 314,
// 2e5 593 -> 502. Beyond 13 tiles per CU (3,328) k_path_fp64 is as fast (3e5 716 against 734 us,
// stiff parameters 938 against 845): its three waves per SIMD are full, and the LDS traffic is not
// free.
constexpr uint32_t kChunkSteps64 = 4;

template <uint32_t NP>
__device__ __forceinline__ void draw_fp64(const DevReq& R, uint32_t tile, int lane, uint32_t part,
                                          DrawChunk64<kChunkSteps64>* buf, double* queue) {
    constexpr uint32_t C = kChunkSteps64;
    static_assert(C % (2 * NP) == 0, "whole counter blocks per wave and chunk");
    const uint64_t first = R.path_offset + (uint64_t)tile * kTile;  // tiles never straddle 2^32
    const uint32_t plo = (uint32_t)first + (uint32_t)lane, phi = uniform((uint32_t)(first >> 32));
    const uint32_t n_steps = R.n_steps;
    for (uint32_t k = 0, c = 0; k < n_steps; k += C, ++c) {
        DrawChunk64<C>& d = buf[c & 1u];
        for (uint32_t b = 0; b < C / 2; b += NP) {
            const uint32_t t = 2 * (b + part);
            const u32x4 w = philox4x32_10((k + t) >> 1, plo, phi, 0u, R.seed_lo, R.seed_hi);
            double z[4];
            normals4_f64(w, z, queue, lane);
            d.z[t][lane] = make_double2(z[0], z[1]);
            d.w[t][lane] = w.x;
            d.z[t + 1][lane] = make_double2(z[2], z[3]);
            d.w[t + 1][lane] = w.z;
        }
        workgroup_sync_lds();  // as in draw_fp32: ceil(n_steps / C) barriers in every wave
    }
}

// One drawing wave: 4 waves per SIMD (128 registers, 18 spilled constants) against the 3 of an
// unconstrained build: 2e5 paths x 252 steps 552 -> 516 us. Two, for at most half a tile per SIMD,
// have no use for them.
template <uint32_t NP>
__global__ __launch_bounds__(64 * (NP + 1)) __attribute__((amdgpu_waves_per_eu(NP == 1 ? 4 : 3))) void k_path_fp64_split(
    PathArgs a) {
    __shared__ DrawChunk64<kChunkSteps64> buf[2];
    __shared__ double queue[NP][4 * kTile];
    __shared__ double4 vals[kTile];
    const int lane = (int)(threadIdx.x & 63u);
    const uint32_t item = blockIdx.x;
    const uint32_t sp = uniform(find_sorted(a.item_end, a.n_sorted, item));
    const uint32_t tile = uniform(item - (sp ? a.item_end[sp - 1] : 0u));
    const uint32_t ri = uniform(a.order[sp]);
    const uint32_t role = stepping_first(uniform(threadIdx.x >> 6), item, NP + 1);
    if (role == 0) {
        __builtin_amdgcn_s_setprio(2);
        path_fp64<kChunkSteps64, false, false>(a, ri, tile, lane, vals, buf);
    } else {
        draw_fp64<NP>(a.reqs[ri], tile, lane, role - 1, buf, queue[role - 1]);
    }
}

// ------------------------------------------------------------------------------------------
// Reduction: pass A sums each 64-tile group of a (request, output) in tile order; pass B sums
// the groups in order and forms the estimator. Both orders depend only on the request.
// ------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t find_req(const uint64_t* end, uint32_t n, uint64_t t) {
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

// Stored partial `slot` of output o, or a zero sum past the request's last stored one.
template <typename Acc>
__device__ __forceinline__ TileSums<Acc> stored_sum(const ReduceArgs& a, const DevReq& R, uint32_t n_out,
                                                    uint32_t n_slots, uint32_t slot, uint32_t o) {
    TileSums<Acc> t;
    if (slot < n_slots) t.load(a.partials, (size_t)R.partial_base + (size_t)slot * n_out + o);
    return t;
}

// The sum of one chunk of tiles: completes the tree ((t0 + t1) + (t2 + t3)) from the level the path
// kernel stored (store_tiles tiles per partial), so a chunk's bits do not depend on the paths per
// thread the request ran with.
template <typename Acc>
__device__ __forceinline__ TileSums<Acc> chunk_sum(const ReduceArgs& a, const DevReq& R, uint32_t n_out, uint32_t c,
                                                   uint32_t o) {
    const uint32_t st = R.store_tiles;
    const uint32_t n_slots = (R.n_tiles + st - 1) / st;
    if (st == kChunkTiles) return stored_sum<Acc>(a, R, n_out, n_slots, c, o);
    if (st == 2) {
        TileSums<Acc> t[2] = {stored_sum<Acc>(a, R, n_out, n_slots, 2 * c, o),
                              stored_sum<Acc>(a, R, n_out, n_slots, 2 * c + 1, o)};
        t[0].combine(t[1]);
        return t[0];
    }
    TileSums<Acc> t[kChunkTiles];
#pragma unroll
    for (int i = 0; i < kChunkTiles; ++i) t[i] = stored_sum<Acc>(a, R, n_out, n_slots, kChunkTiles * c + i, o);
    return chunk_level<kChunkTiles, Acc>(t);
}

__device__ __forceinline__ uint32_t chunks_of(const DevReq& R) { return (R.n_tiles + kChunkTiles - 1) / kChunkTiles; }
constexpr uint32_t kGroupChunks = kGroupTiles / kChunkTiles;

// Sums the chunks of one 64-tile group in chunk order.
template <typename Acc>
__device__ __forceinline__ TileSums<Acc> group_sum(const ReduceArgs& a, const DevReq& R, uint32_t n_out, uint32_t g,
                                                   uint32_t o) {
    TileSums<Acc> acc;
    const uint32_t end = min((g + 1) * kGroupChunks, chunks_of(R));
    for (uint32_t c = g * kGroupChunks; c < end; ++c) acc.combine(chunk_sum<Acc>(a, R, n_out, c, o));
    return acc;
}

__global__ __launch_bounds__(256) void k_reduce_groups(ReduceArgs a, uint64_t total) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const uint32_t ri = find_req(a.group_end, a.n_req, t);
    const uint64_t local = t - (ri ? a.group_end[ri - 1] : 0ull);
    const DevReq& R = a.reqs[ri];
    const uint32_t n_out = R.n_opts * R.n_pay;
    const uint32_t g = (uint32_t)(local / n_out);
    const uint32_t o = (uint32_t)(local - (uint64_t)g * n_out);
    const size_t gslot = (size_t)R.group_base + (size_t)g * n_out + o;
    if (R.precision == kPrecComp)
        group_sum<float>(a, R, n_out, g, o).store(a.groups, gslot);
    else
        group_sum<double>(a, R, n_out, g, o).store(a.groups, gslot);
}

// Sum and sum of squares of an output over the request's groups (sums[first + g stride]), on one
// wavefront: lane l sums groups l, l + 64, l + 128, ... in order and the 64 lane sums are combined by a fixed xor
// butterfly (every lane ends with the same bits). The order depends only on the request's group
// count, never on the launch.
__device__ __forceinline__ void output_sums(const void* sums, size_t first, uint32_t stride, const DevReq& R,
                                            uint32_t lane, double& s, double& ss) {
    if (R.precision == kPrecComp) {
        const float4* p = reinterpret_cast<const float4*>(sums);
        CompF cs{0.f, 0.f}, css{0.f, 0.f};
        for (uint32_t g = lane; g < R.n_groups; g += kTile) {
            const float4 v = p[first + (size_t)g * stride];
            cs.merge(v.x, v.y);
            css.merge(v.z, v.w);
        }
#pragma unroll
        for (int m = 1; m < kTile; m <<= 1) {
            const float s2 = __shfl_xor(cs.s, m), c2 = __shfl_xor(cs.c, m);
            const float q2 = __shfl_xor(css.s, m), d2 = __shfl_xor(css.c, m);
            cs.merge(s2, c2);
            css.merge(q2, d2);
        }
        s = (double)cs.s + (double)cs.c;
        ss = (double)css.s + (double)css.c;
    } else {
        const double2* p = reinterpret_cast<const double2*>(sums);
        s = 0.0;
        ss = 0.0;
        for (uint32_t g = lane; g < R.n_groups; g += kTile) {
            const double2 v = p[first + (size_t)g * stride];
            s += v.x;
            ss += v.y;
        }
#pragma unroll
        for (int m = 1; m < kTile; m <<= 1) {
            s += __shfl_xor(s, m);
            ss += __shfl_xor(ss, m);
        }
    }
}

// Sample mean and variance (n - 1 denominator, clamped at 0) from a sum and a sum of squares.
__device__ __forceinline__ void mean_var(double s, double ss, double n, double& mean, double& var) {
    mean = s / n;
    var = n > 1.0 ? __builtin_fma(-(n * mean), mean, ss) / (n - 1.0) : 0.0;
    var = var > 0.0 ? var : 0.0;
}

// The group sums of output o into LDS by a workgroup of 256 threads: 16 lanes take the chunks of a
// group, and combine them in chunk order.
template <typename Acc>
__device__ __forceinline__ void group_sums_lds(const ReduceArgs& a, const DevReq& R, uint32_t o, void* sums) {
    static_assert(kGroupChunks == 16, "a group's chunks are the 16 lanes of a row");
    const uint32_t n_out = R.n_opts * R.n_pay, n_chunks = chunks_of(R), i = threadIdx.x % 16u;
    for (uint32_t g0 = 0; g0 < R.n_groups; g0 += 16) {
        const uint32_t g = g0 + threadIdx.x / 16u, c = g * kGroupChunks + i;
        TileSums<Acc> t, acc;
        if (c < n_chunks) t = chunk_sum<Acc>(a, R, n_out, c, o);
#pragma unroll
        for (uint32_t k = 0; k < kGroupChunks; ++k) {
            const TileSums<Acc> u = t.of_lane((int)((threadIdx.x & 48u) + k));
            if (g * kGroupChunks + k < n_chunks) acc.combine(u);
        }
        if (i == 0 && g < R.n_groups) acc.store(sums, g);
    }
}

// One wavefront per output, or for small batches (SMALL, at most kSmallGroups groups a request) one
// workgroup, whose threads form the group sums of what the output reads first: one kernel in place of
// two, and a group's chunks in parallel lanes instead of one thread's serial loads (a request of 63
// tiles: 11.5 us with the gap between them -> 6.8). In larger batches a wavefront's loads a whole row
// of outputs apart cost more.
// A control-variate output adds the exact geometric price to the mean of A - G; with kCvRegression
// it is A - beta (G - E[G]) instead, beta = Cov(A, G) / Var G from the same paths' Asian (block 0)
// and geometric outputs of the option: Cov from Var(A - G) = Var A + Var G - 2 Cov(A, G), variance
// Var A - beta Cov(A, G).
template <bool SMALL>
__global__ __launch_bounds__(256) void k_reduce_final(ReduceArgs a, uint64_t total) {
    __shared__ double2 lds[SMALL ? 3 : 1][SMALL ? kSmallGroups : 1];
    const uint64_t t = SMALL ? blockIdx.x : ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / (uint64_t)kTile;  // wave-uniform
    const uint32_t lane = threadIdx.x % (uint32_t)kTile;
    if (t >= total) return;
    const uint32_t ri = find_req(a.out_end, a.n_req, t);
    const uint32_t o = (uint32_t)(t - (ri ? a.out_end[ri - 1] : 0ull));
    const DevReq& R = a.reqs[ri];
    const uint32_t opt = o % R.n_opts, n_out = R.n_opts * R.n_pay;
    const bool cv = a.geo && payoff_kind(R.payoffs, o / R.n_opts) == kAsianGeoCV;
    const bool reg = cv && (R.flags & kCvRegression);  // request-uniform
    const uint32_t outs[3] = {o, opt, (uint32_t)__popc(R.payoffs & (kGeoAsian - 1u)) * R.n_opts + opt};
    if constexpr (SMALL) {
        for (int k = 0; k < (reg ? 3 : 1); ++k) {
            if (R.precision == kPrecComp)
                group_sums_lds<float>(a, R, outs[k], lds[k]);
            else
                group_sums_lds<double>(a, R, outs[k], lds[k]);
        }
        __syncthreads();
        if (threadIdx.x >= (uint32_t)kTile) return;
    }
    auto sums = [&](int k, double& s, double& ss) {
        if constexpr (SMALL)
            output_sums(lds[k], 0, 1, R, lane, s, ss);
        else
            output_sums(a.groups, (size_t)R.group_base + outs[k], n_out, R, lane, s, ss);
    };
    double s, ss, sa = 0.0, ssa = 0.0, sg = 0.0, ssg = 0.0;
    sums(0, s, ss);
    if (reg) {
        sums(1, sa, ssa);
        sums(2, sg, ssg);
    }
    if (lane != 0) return;
    const double disc = a.opts[R.opt_begin + opt].disc;
    const double scale = (R.precision == kPrecFP64) ? 1.0 : R.S0;
    const double n = (double)R.n_paths;
    double mean, var;
    mean_var(s, ss, n, mean, var);
    double price = __builtin_fma(scale, mean, cv ? a.geo[R.out_base + o] : 0.0);
    if (reg) {
        double ma, va, mg, vg;
        mean_var(sa, ssa, n, ma, va);
        mean_var(sg, ssg, n, mg, vg);
        const double cov = 0.5 * (va + vg - var);
        const double beta = vg > 0.0 ? cov / vg : 0.0;
        price = __builtin_fma(scale, ma, -(beta * __builtin_fma(scale, mg, -a.geo[R.out_base + o])));
        var = __builtin_fma(-beta, cov, va);
        var = var > 0.0 ? var : 0.0;
    }
    a.prices[R.out_base + o] = disc * price;
    if (a.std_errs) a.std_errs[R.out_base + o] = scale * disc * ::sqrt(var / n);
}

// ------------------------------------------------------------------------------------------
// Component kernels for the parity tests and measurement.
// ------------------------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t* p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_fill_u64(unsigned long long* p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

__global__ void k_rng_fill(uint32_t* out, uint64_t seed, uint32_t stream, uint64_t path0, uint64_t n_paths,
                           uint64_t word0, uint64_t n_words) {
    const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n_paths * n_words) return;
    const uint64_t i = t / n_words, j = t - i * n_words;
    const uint64_t w = word0 + j, path = path0 + i;
    const u32x4 b = philox4x32_10((uint32_t)(w >> 2), (uint32_t)path, (uint32_t)(path >> 32), stream, (uint32_t)seed,
                                  (uint32_t)(seed >> 32));
    const uint32_t e = (uint32_t)(w & 3u);
    out[t] = e == 0 ? b.x : e == 1 ? b.y : e == 2 ? b.z : b.w;
}

__global__ void k_philox(const uint32_t* ctr, const uint32_t* key, uint64_t n, uint32_t* out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const u32x4 b = philox4x32_10(ctr[4 * i], ctr[4 * i + 1], ctr[4 * i + 2], ctr[4 * i + 3], key[2 * i], key[2 * i + 1]);
    out[4 * i] = b.x;
    out[4 * i + 1] = b.y;
    out[4 * i + 2] = b.z;
    out[4 * i + 3] = b.w;
}

__global__ void k_normals_fp32(const uint32_t* words, uint64_t n, double* out) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] = (double)normal_f32(words[i]);
}

// Words 4t .. 4t + 3 by thread t, as the FP64 path kernels take a lane's counter block. Words past n
// (central ones) fill the last wavefront up.
__global__ __launch_bounds__(256) void k_normals_fp64(const uint32_t* words, uint64_t n, double* out) {
    __shared__ double queue[4][4 * kTile];
    const uint64_t i = 4 * ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x);
    uint32_t k[4];
    for (uint32_t j = 0; j < 4; ++j) k[j] = i + j < n ? words[i + j] : 0x80000000u;
    double z[4];
    normals4_f64(u32x4{k[0], k[1], k[2], k[3]}, z, queue[threadIdx.x >> 6], (int)(threadIdx.x & 63u));
    for (uint32_t j = 0; j < 4; ++j)
        if (i + j < n) out[i + j] = z[j];
}

__global__ void k_copy(const float4* __restrict__ src, float4* __restrict__ dst, uint64_t n) {
    uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = src[i];
}

inline dim3 grid_for(uint64_t n, uint32_t block) { return dim3((uint32_t)((n + block - 1) / block)); }

}  // namespace

// ------------------------------------------------------------------------------------------
// Launch wrappers (host)
// ------------------------------------------------------------------------------------------
const void* path_kernel_symbol(uint32_t precision, uint32_t ppt, PathMode mode, bool mart, bool geo) {
    if (precision == kPrecFP64) {
        switch (mode) {
            case PathMode::Normal: return reinterpret_cast<const void*>(&k_path_fp64<false, false>);
            case PathMode::Debug: return reinterpret_cast<const void*>(&k_path_fp64<true, false>);
            case PathMode::Count: return reinterpret_cast<const void*>(&k_path_fp64<false, true>);
        }
        return nullptr;
    }
#define HEXO_PPT_MODES(P, M, G)                                                                          \
    switch (mode) {                                                                                      \
        case PathMode::Normal: return reinterpret_cast<const void*>(&k_path_fp32<P, false, false, M, G>); \
        case PathMode::Debug: return reinterpret_cast<const void*>(&k_path_fp32<P, true, false, M, G>);   \
        case PathMode::Count: return reinterpret_cast<const void*>(&k_path_fp32<P, false, true, M, G>);   \
    }                                                                                                    \
    return nullptr;
#define HEXO_PPT_CASE(P)                    \
    case P:                                 \
        if (mart && geo) {                  \
            HEXO_PPT_MODES(P, true, true)   \
        }                                   \
        if (mart) {                         \
            HEXO_PPT_MODES(P, true, false)  \
        }                                   \
        if (geo) {                          \
            HEXO_PPT_MODES(P, false, true)  \
        }                                   \
        HEXO_PPT_MODES(P, false, false)
    switch (ppt) {
        HEXO_PPT_CASE(1)
        HEXO_PPT_CASE(2)
        HEXO_PPT_CASE(3)
        HEXO_PPT_CASE(4)
        default: return nullptr;
    }
#undef HEXO_PPT_CASE
#undef HEXO_PPT_MODES
}

size_t path_lds_bytes(uint32_t precision, uint32_t ppt, uint32_t block) {
    const size_t waves = block / kTile;
    // FP32: per wave the transpose of the per-path values at expiries (4 words per path, WaveLds);
    // FP64: 64 double4 per wave
    return precision == kPrecFP64 ? waves * kTile * sizeof(double4) : waves * 4 * ppt * kTile * sizeof(uint32_t);
}

hipError_t launch_paths_split(uint32_t precision, uint32_t n_draw, const PathArgs& a, bool mart, bool geo,
                              hipStream_t st) {
    if (n_draw != 1 && n_draw != 2) return hipErrorInvalidValue;
    if (precision == kPrecFP64) {
        if (n_draw == 2)
            k_path_fp64_split<2><<<a.total_items, 192, 0, st>>>(a);
        else
            k_path_fp64_split<1><<<a.total_items, 128, 0, st>>>(a);
        return hipGetLastError();
    }
#define HEXO_SPLIT(M, G)                                                           \
    if (n_draw == 2)                                                               \
        k_path_fp32_split<2, 8, M, G><<<a.total_items, 192, 0, st>>>(a);           \
    else                                                                           \
        k_path_fp32_split<1, 4, M, G><<<a.total_items, 128, 0, st>>>(a);
    if (mart && geo) {
        HEXO_SPLIT(true, true)
    } else if (mart) {
        HEXO_SPLIT(true, false)
    } else if (geo) {
        HEXO_SPLIT(false, true)
    } else {
        HEXO_SPLIT(false, false)
    }
#undef HEXO_SPLIT
    return hipGetLastError();
}

hipError_t launch_paths(uint32_t precision, uint32_t ppt, PathMode mode, uint32_t grid, uint32_t block,
                        hipStream_t st, const PathArgs& a, bool mart, bool geo) {
    const size_t lds = path_lds_bytes(precision, ppt, block);
    if (precision == kPrecFP64) {
        switch (mode) {
            case PathMode::Normal: k_path_fp64<false, false><<<grid, block, lds, st>>>(a); break;
            case PathMode::Debug: k_path_fp64<true, false><<<grid, block, lds, st>>>(a); break;
            case PathMode::Count: k_path_fp64<false, true><<<grid, block, lds, st>>>(a); break;
        }
        return hipGetLastError();
    }
#define HEXO_LAUNCH_M(P, M, G)                                                                      \
    switch (mode) {                                                                                 \
        case PathMode::Normal: k_path_fp32<P, false, false, M, G><<<grid, block, lds, st>>>(a); break; \
        case PathMode::Debug: k_path_fp32<P, true, false, M, G><<<grid, block, lds, st>>>(a); break;   \
        case PathMode::Count: k_path_fp32<P, false, true, M, G><<<grid, block, lds, st>>>(a); break;   \
    }
#define HEXO_LAUNCH(P)                  \
    if (mart && geo) {                  \
        HEXO_LAUNCH_M(P, true, true)    \
    } else if (mart) {                  \
        HEXO_LAUNCH_M(P, true, false)   \
    } else if (geo) {                   \
        HEXO_LAUNCH_M(P, false, true)   \
    } else {                            \
        HEXO_LAUNCH_M(P, false, false)  \
    }
    switch (ppt) {
        case 1: HEXO_LAUNCH(1) break;
        case 2: HEXO_LAUNCH(2) break;
        case 3: HEXO_LAUNCH(3) break;
        case 4: HEXO_LAUNCH(4) break;
        default: return hipErrorInvalidValue;
    }
#undef HEXO_LAUNCH
#undef HEXO_LAUNCH_M
    return hipGetLastError();
}

hipError_t launch_reduce(const ReduceArgs& a, uint64_t n_group_threads, uint64_t n_out_threads, bool small,
                         hipStream_t st) {
    if (small) {
        if (n_out_threads) k_reduce_final<true><<<(uint32_t)n_out_threads, 256, 0, st>>>(a, n_out_threads);
        return hipGetLastError();
    }
    if (n_group_threads) k_reduce_groups<<<grid_for(n_group_threads, 256), 256, 0, st>>>(a, n_group_threads);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // one wavefront per output
    if (n_out_threads) k_reduce_final<false><<<grid_for(n_out_threads * kTile, 256), 256, 0, st>>>(a, n_out_threads);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t st) {
    k_fill_u32<<<grid_for(n, 256), 256, 0, st>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_zero_u64(unsigned long long* p, uint32_t n, hipStream_t st) {
    k_fill_u64<<<grid_for(n, 256), 256, 0, st>>>(p, n);
    return hipGetLastError();
}

hipError_t launch_rng_fill(uint32_t* out, uint64_t seed, uint32_t stream, uint64_t path0, uint64_t n_paths,
                           uint64_t word0, uint64_t n_words, hipStream_t st) {
    k_rng_fill<<<grid_for(n_paths * n_words, 256), 256, 0, st>>>(out, seed, stream, path0, n_paths, word0, n_words);
    return hipGetLastError();
}

hipError_t launch_philox(const uint32_t* ctr, const uint32_t* key, uint64_t n, uint32_t* out, hipStream_t st) {
    k_philox<<<grid_for(n, 256), 256, 0, st>>>(ctr, key, n, out);
    return hipGetLastError();
}

hipError_t launch_normals(const uint32_t* words, uint64_t n, uint32_t precision, double* out, hipStream_t st) {
    if (precision == kPrecFP64)
        k_normals_fp64<<<grid_for((n + 3) / 4, 256), 256, 0, st>>>(words, n, out);
    else
        k_normals_fp32<<<grid_for(n, 256), 256, 0, st>>>(words, n, out);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, uint64_t bytes, uint32_t grid, hipStream_t st) {
    k_copy<<<grid, 256, 0, st>>>(reinterpret_cast<const float4*>(src), reinterpret_cast<float4*>(dst), bytes / 16);
    return hipGetLastError();
}

}  // namespace hexo
