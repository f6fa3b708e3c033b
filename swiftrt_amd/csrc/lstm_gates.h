// The gate arithmetic of an LSTM cell, for translation units without floating-point contraction.
#pragma once
#include "gemm_common.h"

namespace srt {

template <typename T>
__device__ __forceinline__ float gate_sigmoid(float a) {
  if constexpr (T::dtype == srtReal32F) return 1.0f / (1.0f + expf(-a));
  return __fdividef(1.0f, 1.0f + __expf(-a));
}
template <typename T>
__device__ __forceinline__ float gate_tanh(float a) {
  if constexpr (T::dtype == srtReal32F) return tanhf(a);
  return activation16_ct<srtActivationTanh>(0.0f, a);
}
template <typename T>
__device__ __forceinline__ float gate_round(float a) { return T::to_float(T::from_float(a)); }

// cell' = cell * sigmoid(forget) + sigmoid(input) * tanh(update),  hidden' = tanh(cell') * sigmoid(output), every intermediate rounded
// to the element type: bit for bit what the element-wise operations it stands for give (16-bit types: their fast forms).
template <typename T, typename S>
__device__ __forceinline__ void lstm_gate(float input, float update, float forget, float output, float cell, S* new_cell, S* new_hidden) {
  const float in = gate_round<T>(gate_sigmoid<T>(input)), up = gate_round<T>(gate_tanh<T>(update));
  const float share = gate_round<T>(gate_sigmoid<T>(forget)), out = gate_round<T>(gate_sigmoid<T>(output));
  const float kept = gate_round<T>(cell * share), added = gate_round<T>(in * up);
  *new_cell = T::from_float(kept + added);
  *new_hidden = T::from_float(gate_round<T>(gate_tanh<T>(T::to_float(*new_cell))) * out);
}

}  // namespace srt
