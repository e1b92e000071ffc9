// Matrix-core transforms of the Reed-Solomon encoder (implemented in ntt_mx.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "ntt.h"

namespace whir {

// Device tables of one shape, built by the caller (ntt.hip) and shared by all messages:
//   row[c*C2 + i2] = w_N^(c C1 i2), post[(c*C2 + t2)*C1 + i1] = w_N^(i1 (c + Q t2)),
//   pre[c*C + i] = w_N^(c i).
struct MxTables {
  const uint64_t* row = nullptr;
  const uint64_t* post = nullptr;
  const uint64_t* pre = nullptr;
};

// Whether the matrix-core kernels transform cosets of 2^logC elements, and how: the
// four-step split's log C1 (0: one pass).
bool mx_split(int logC, int* logC1);
void mx_prepare();  // builds the constant tables (not during a stream capture)
void mx_encode(int D, const RsArgs& a, const MxTables& t, uint64_t* scratch, hipStream_t st);

}  // namespace whir
