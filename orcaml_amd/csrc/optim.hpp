// The optimizers' per-element arithmetic, shared by their passes (fused.hip) and by the
// weight-gradient products that update what they produce (gemm_tile.hpp).
#pragma once

#include "runtime.hpp"

namespace orca_hip {
namespace {

__device__ __forceinline__ void adamw_elem(float& p, float g, float& m, float& v, const AdamWScalars& k) {
  float d = p * k.decay;                // p * (1 - lr*wd)
  float mn = (m * k.b1) + (g * k.omb1); // m*b1 + g*(1-b1)
  float vn = (v * k.b2) + ((g * g) * k.omb2);
  float mh = mn * k.c1;
  float vh = vn * k.c2;
  float den = sqrtf(vh) + k.eps;
  float u = (mh / den) * k.lr;
  p = d - u;
  m = mn;
  v = vn;
}

}  // namespace
}  // namespace orca_hip
