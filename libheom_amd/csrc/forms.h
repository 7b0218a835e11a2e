// Launchers of the operator kernels by form (one fused operator pass each),
// instantiated for <float, false> (FP32 operator) and <double, true> (every
// operand complex128).  They return the number of error-norm partials written.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace hamd {

template <typename R, bool F64>
int launch_hilb(const FormDev& d, const StageArgs& A, hipStream_t st);
// 4 <= N <= 16, diagonal V, few ADOs with many links (d.slinks)
template <typename R, bool F64>
int launch_hilb_split(const FormDev& d, const StageArgs& A, hipStream_t st);
// 16 < N <= 64 on matrix cores: diagonal V (d.mfma 1, 2), dense V (d.mfma 3)
template <typename R, bool F64>
int launch_hilb_mfma(const FormDev& d, const StageArgs& A, hipStream_t st);
template <typename R, bool F64>
int launch_hilb_mfma_dense(const FormDev& d, const StageArgs& A, hipStream_t st);
template <typename R, bool F64>
int launch_batch(const FormDev& d, const StageArgs& A, hipStream_t st);
template <typename R, bool F64>
int launch_redfield(const FormDev& d, const StageArgs& A, hipStream_t st);

#define HAMD_FORM_INSTANCES(f)                                              \
  template int f<float, false>(const FormDev&, const StageArgs&, hipStream_t); \
  template int f<double, true>(const FormDev&, const StageArgs&, hipStream_t);

}  // namespace hamd
