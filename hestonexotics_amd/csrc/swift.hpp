// swift.hpp -- device layout and launch wrappers of the SWIFT European pricer (FP64).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "cplx.hpp"
#include "swift_grid.hpp"

namespace hexo {

// Chains with J up to this size run both transforms in one workgroup's LDS (16 B x 2J = 128 KiB);
// larger ones use direct sums.
constexpr uint32_t kSwiftFftMaxJ = 4096;
// Chains expected to stay at or below this share a CU with others (32 KiB each).
constexpr uint32_t kSwiftSmallJ = 1024;
// Strikes of one chain summed by one workgroup of the final contraction: one or two per thread.
constexpr uint32_t kSwiftStrikeBlock = 16, kSwiftStrikeBlock2 = 32;

// One chain's inputs, read by the kernels from pinned host memory.
struct SwiftChainIn {
    double p[5];  // v0, theta, rho, kappa, sigma
    double T, r, S0, trunc, disc;
    uint64_t strike_off;
    uint32_t block_off;  // first of its workgroups in the contraction
    uint32_t n_strikes;
    uint32_t fixed;        // use `grid` instead of choosing one
    hexo_swift_grid grid;  // checked by the host
};

// One chain (expiry) of a SWIFT call: model, grid and the offsets of its slices in the work arrays.
// Written by k_swift_transform, for chains with larger J by the host (swift_host.cpp). J = 0: not
// priced in this pass.
struct DevSwift {
    double p[5];  // v0, theta, rho, kappa, sigma
    double S0, r, T, disc;
    double exp2_m, sqrt_exp2_m, lower, upper;
    int32_t k1, k2;
    uint32_t J, n_strikes;
    uint32_t rows;  // 1 (prices) or 6 (prices and the five partials)
    uint32_t pad;
    uint64_t strike_off;  // doubles
    uint64_t tw_off;      // Cplx, 4J: e^{2 pi i k / 4J}; shared by the chains with the same J
    uint64_t pay_off;     // Cplx, J: payoff coefficients
    uint64_t dens_off;    // doubles, k2 - k1 + 1
    uint64_t coeff_off;   // Cplx, J: density coefficients
    uint64_t pm_off;      // Cplx, rows x J: pricing matrix
    uint64_t out_off;     // doubles: prices; grads at 5x that offset in the grads array
};

// One twiddle table (per distinct J of the call).
struct SwiftTable {
    uint32_t J;
    uint32_t pad0;
    uint64_t off;  // Cplx
};

struct SwiftArgs {
    const DevSwift* reqs;
    uint32_t n_req;
    uint32_t n_tables;
    const SwiftTable* tables;
    const double* strikes;
    const uint32_t* block_chain;   // per workgroup of the contraction: its chain
    const uint32_t* block_strike;  // and the first of its (up to strike_block) strikes
    uint32_t n_blocks, strike_block;
    bool split_rows;  // gradients: three times the threads on a strike
    Cplx* tw;
    Cplx* pay;
    double* dens;
    Cplx* coeff;
    Cplx* pm;
    double* prices;
    double* grads;  // null when no request asks for gradients
    // direct sums: inclusive prefix sums of the per-kernel thread (or wavefront) counts
    const uint64_t* tab_end;   // over tables: 4J
    const uint64_t* j_end;     // over chains: J
    const uint64_t* dens_end;  // over chains: k2 - k1 + 1
};

struct SwiftTotals {
    uint64_t tw, j, dens;
};

// A pass over n_req chains. The k-th has slot k of recs and of the work arrays, max_J values (times
// rows) each.
struct SwiftChainArgs {
    const SwiftChainIn* chains;
    const uint32_t* order;  // k -> chain; null: in order
    const double* strikes;
    const Cplx* roots;  // e^{2 pi i k / 4 kSwiftFftMaxJ}
    SwiftGridOut* grids;
    double* dev_strikes;  // the call's strikes and contraction workgroups (SwiftArgs), filled in
    uint32_t* block_chain;
    uint32_t* block_strike;
    DevSwift* recs;
    Cplx* coeff;
    uint32_t n_req;
    uint32_t max_J;  // kSwiftSmallJ or kSwiftFftMaxJ
    uint32_t rows, strike_block;
};

// The roots table of SwiftChainArgs (4 kSwiftFftMaxJ values).
hipError_t launch_swift_roots(Cplx* roots, hipStream_t st);
// Chains to their grids and records and, where J <= max_J, their density coefficients.
hipError_t launch_swift_transform(const SwiftChainArgs& a, hipStream_t st);
// Prices (and gradients) from the density coefficients of chains with J up to max_J.
hipError_t launch_swift_prices(const SwiftArgs& a, uint32_t max_J, hipStream_t st);
// Chains given their grids from payoffs to prices, the transforms by direct sums.
hipError_t launch_swift_large(const SwiftArgs& a, const SwiftTotals& t, hipStream_t st);
// Copies bytes0 from s0 to d0 and bytes1 from s1 to d1 (multiples of 16; the sources may be
// fine-grained pinned host memory) in one kernel.
hipError_t launch_swift_stage(const void* s0, void* d0, size_t bytes0, const void* s1, void* d1, size_t bytes1,
                              hipStream_t st);

}  // namespace hexo
