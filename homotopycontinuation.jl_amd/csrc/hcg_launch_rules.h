// Rules by which the host runtime chooses a launch, on sizes only (no device needed).
#pragma once
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

}  // namespace hcg
