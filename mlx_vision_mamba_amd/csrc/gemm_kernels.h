// float32 matrix products on the bf16 matrix units: geometry and launch
// entry points (gemm.hip), used by the C ABI (capi.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mvm {

struct GemmGeom {
  int32_t M, N, K;
  int32_t batch;
  int32_t lda, ldb;
  int64_t ldc;
  int64_t sa, sb, sc;    // batch strides
  int32_t seg;           // B segment length along k (K when there is one)
  int64_t seg_stride;
  int32_t a_km, b_km;    // 1: k is the contiguous index
  int32_t cfg;           // tile shape (gemm.hip)
  int32_t nsplit, kper;  // the sum over k in nsplit parts of kper
};

// picks the tile shape and (when nsplit is 0) the split of k; below 32 values
// of k no operand is loaded in vectors, so any alignment will do
void gemm_plan(GemmGeom& g);
// float32 elements of the partial-product buffer (0 without a split)
int64_t gemm_partial_floats(const GemmGeom& g);
// add: nullptr, or what is added to the products, laid out as C (may be C)
hipError_t launch_gemm(const GemmGeom& g, const float* A, const float* B, const float* add, float* C,
                       float* part, hipStream_t s);

}  // namespace mvm
