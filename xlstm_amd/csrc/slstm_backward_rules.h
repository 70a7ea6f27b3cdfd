// Decisions of the reverse kernels that spread a head over several compute units, in plain C++ without a GPU's anything: the tests
// compile this file for the host and walk through it.
#pragma once

#ifdef __HIPCC__
#define XS_RULE __host__ __device__ constexpr
#else
#define XS_RULE constexpr
#endif

namespace {

// Whether a call has to be flagged as failed because of where a group's workgroups ran.  `seen`: the XCDs they found themselves on, one
// bit each.  Their exchange goes through ONE XCD's L2; a group of one workgroup, and a call with the recurrent gradient cut, in
// which nothing reaches the step before, exchange nothing and may run anywhere.
XS_RULE bool bwd_exchange_torn(int members, bool cut, unsigned int seen) { return members > 1 && !cut && (seen & (seen - 1u)) != 0u; }

}  // namespace
