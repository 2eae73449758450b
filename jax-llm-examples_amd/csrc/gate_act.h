// The activations of gated units.  ACT 0: silu, z / (1 + exp(-z)); 1: the tanh form of gelu, 0.5 z (1 + tanh(sqrt(2 /
// pi) (z + 0.044715 z^3))).
#pragma once

#include "common.h"

namespace jle {

template <int ACT>
__device__ __forceinline__ float gate_act(float g) {
  if (ACT == 1) return 0.5f * g * (1.0f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
  return g / (1.0f + expf(-g));
}

}  // namespace jle
