// The spherical-harmonic operators, forward and backward, each one C++ call and one autograd node.
#pragma once
#include "torch_util.hpp"

namespace fsgs_host {

// Basis values [B,(degree+1)^2] of the directions dirs[B,>=3]; no value: not a call for this layer (another type, device, layout or
// dimension, a mode that asks for more than the values, a degree out of range), the Python operator pair takes or refuses it.
OptTensor sh_encode(const Tensor& dirs, int64_t degree);

// Colours [P,3] of the coefficients sh[P,F,3] seen along dirs[P,3] (positions, with campos[3]); no value: as above.
OptTensor sh_to_rgb(const Tensor& sh, const Tensor& dirs, const OptTensor& campos, int64_t degree, bool clamp);

}  // namespace fsgs_host
