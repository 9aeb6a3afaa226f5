// The symmetric softened self sums (soft_sym.hip): S and a of every member over its halo.
#pragma once
#include "halma_common.h"

namespace halma {

// Whether the path takes a halo of n members (its slots grow with the halo: 2^21 at most).
bool soft_sym_takes(int64_t n);
size_t soft_sym_bytes(int64_t H, const int64_t* off);

// rows: (x, y, z, m) from member off[0] on; pot (may be null) and acc (3 per member, may be
// null) likewise from that member on.  Haloes it does not take are left out.
int soft_sym_run(int64_t H, const int64_t* off, const float4* rows, float e2, double* pot,
                 double* acc, void* ws, size_t ws_bytes, hipStream_t st);

}  // namespace halma
