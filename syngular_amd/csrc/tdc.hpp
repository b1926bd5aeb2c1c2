// Direct phase of the blocked Gram eigen-solver (tdc.hip).
#pragma once
#include <vector>

#include "tjacobi.hpp"

namespace syn {

// Orders the direct phase takes.
constexpr int64_t kTdcMin = 17;
constexpr int64_t kTdcMax = 2048;
bool tdc_takes(int64_t nv);
// Orders whose reduction runs over work-groups that wait for each other.
bool tdc_waits(int64_t nv);

// Runs the direct phase on problems that tdc_takes(); host holds the same
// items as the device table, w set to disjoint regions of at least
// tj_work<16>(nv) doubles and counter to an entry each, cleared.  polls bounds
// every wait of a work-group for another (0: the phase's own bounds).  On return
// (stream order) g is rt g rt^T and rt the eigenvector rows, or g as it was and rt
// the identity for a matrix with no entry that passes the sweeps' rotation test
// (threshold tol), one that the phase cannot take (zero, not finite, far out of
// range) or whose reduction gave up waiting; counter is set to 1 for the last.
int tdc_launch(const syn_gbj_item *items, const std::vector<syn_gbj_item> &host, int polls, double tol,
               hipStream_t st);

}  // namespace syn
