// Rules by which the host runtime chooses a launch, on sizes only (no device needed).
#pragma once
#include <algorithm>
#include <cstddef>

namespace hcg {

// Sizes of a certifier's split tapes.
struct CertSplit {
    long coefs;    // coefficients of one parameter vector
    long doubles;  // its table
    long saved;    // operations that every evaluation of a candidate saves by the table
    long ops;      // operations of the coefficients' programs
};

// Most bytes of coefficient tables a certification call allocates.
constexpr size_t kCertTableBytes = (size_t)4 << 30;

// Whether a certification call evaluates the parameter-only coefficients once per parameter vector, into
// tables, or whole tapes per candidate.  Below a full GPU a call takes the latency of one candidate's
// evaluations, which the tables shorten by a time proportional to `saved`; a table costs a time proportional to
// its programs' operations (and about 8 for each program's tables and stores) however many candidates
// read it.  The first limit is where the two meet, with the second part of the saving (a few operations
// cost as much as none) taken off; the other one allows a vector for every 16 candidates on a full
// GPU.  Both lie below the smallest number of vectors at which tables lost, with refinement or without.
// Whole tapes / tables, kernel ms, FP64 test only, candidates each on a vector of its own unless stated:
//   n = 10, 718 coefficients: 4,096 60.6 / 11.8, 16,384 61.6 / 22, 262,144 81 / 360 (limit 27,000 + 1/16)
//   n = 6, 418 coefficients:  8,192 27.0 / 6.9, 16,384 27.3 / 12.1, 65,536 30.8 / 44.8 (limit 24,400 + 1/16)
//   n = 4, 130 coefficients:  8,192 2.2 / 1.1, 16,384 2.2 / 1.7, 65,536 2.7 / 4.3 (limit 8,800 + 1/16)
//   n = 3, 63 coefficients, products of parameters: 4,096 1.05 / 0.60, 16,384 1.07 / 1.27, 65,536
//   1.34 / 3.75; 262,144 on 24,576 vectors 3.9 / 3.5, on 65,536 4.0 / 5.7 (limit 4,100 + 1/16)
inline bool certify_with_tables(long nsol, long ngroups, const CertSplit& s) {
    if ((size_t)ngroups > kCertTableBytes / (sizeof(double) * (size_t)s.doubles)) return false;
    const long few = (40000 * s.saved - 3000000) / (s.ops + 8 * s.coefs);
    return ngroups <= (few > 0 ? few : 0) + (nsol + 15) / 16;
}

// Workgroups of a tracker launch, and how many lanes (per-lane layout) or groups (lane-group layout) of
// each wave take paths.
struct LaunchShape {
    long workgroups;
    int per_wave;
};

// Per-lane kernels, one wave per workgroup.  A batch with fewer than 64 paths per CU is spread over up to one
// wave per CU instead of filling 64 lanes of fewer waves: the lanes of a wave wait for each other's
// branches, and the CUs are free.  Every wave has the same number of lanes, so just past a multiple of the
// CU count up to half of the CUs stay free (257 paths on 256 CUs: 129 waves of two).  Four waves per CU
// touch more lines of private memory (a line holds one dword of 32 lanes), which costs more than it
// gives at n = 10 and less at n = 8.  Full waves / one wave per CU / four per CU, measured: two-variable
// parameter homotopy, 2,000 paths 0.29 / 0.21 / 0.29 ms; dense n = 4, 81 paths 6.9 / 5.1 / 5.3; dense n = 8,
// 400 paths 119.7 / 95.0 / 94.1, 6,561 paths 141.8 / 138.3 / 135.7; parameter batch n = 10, 100 paths
// 43.9 / 35.3 / 37.5, 1,024 paths 49.0 / 47.6 / 61.9, 4,096 paths 43.6 / 45.0 / 59.8.
inline LaunchShape lane_shape(long ncu, int waves_per_eu, int blocks_per_cu, long npaths) {
    const long slots = ncu * (blocks_per_cu > 0 ? blocks_per_cu : 4 * waves_per_eu);  // every wave slot of the CU's 4 SIMDs
    const long waves = std::max<long>(1, std::min(slots, std::max((npaths + 63) / 64, std::min(npaths, ncu))));
    const long lanes = std::max<long>(1, std::min<long>(64, (npaths + waves - 1) / waves));
    return {std::max<long>(1, std::min<long>(slots, (npaths + lanes - 1) / lanes)), (int)lanes};
}

// Lane-group kernels, workgroups of `waves` waves with `most` groups each: as few groups of a wave as one wave per
// SIMD allows, since the groups of a wave wait for each other's evaluations; at most blocks_per_cu workgroups
// per CU (default 2).  As above, just past a step half of the CUs stay free (1,025 paths with two groups
// per wave: 129 workgroups).  All groups of a wave / this rule, measured: n = 15, 64 paths 114.8 / 108.0 ms,
// 2,048 paths 144.5 / 132.1, 5,000 paths (all groups either way) 166; n = 22, 100 paths 296 / 280, 601 paths
// 354 / 320.
inline LaunchShape group_shape(long ncu, int waves, int most, int blocks_per_cu, long total) {
    const long slots = ncu * waves;
    const long groups = std::max<long>(1, std::min<long>(most, (total + slots - 1) / slots));
    const long grid = std::min<long>((total + groups * waves - 1) / (groups * waves), ncu * (blocks_per_cu > 0 ? blocks_per_cu : 2));
    return {std::max<long>(1, grid), (int)groups};
}

}  // namespace hcg
