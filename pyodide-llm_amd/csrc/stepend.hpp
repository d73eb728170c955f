// stepend.hpp — the end of a replayed step, run by the block that chooses the step's token (the last stage of the greedy
// choice, the draw): two launches of their own before, 1.3 us of a replayed step each.
#pragma once

#include "kernels.hpp"

namespace ple {

// whether the step that chose `token` with largest logit `value` ends the call: a token that is not one (the draw's
// SAMPLE_NOT_FINITE or SAMPLE_DECLINED), a largest logit that is not finite, or a stop token
__device__ __forceinline__ bool halts(int32_t token, float value, const RunParams *params) {
  if (token < 0 || !__builtin_isfinite(value)) return true;
  const int ns = params->n_stops;
  for (int j = 0; j < RUN_STOPS_MOST; ++j)
    if (j < ns && params->stops[j] == token) return true;
  return false;
}

// The whole block (nt threads) calls it with the same token and value: where the step ends the call and none before it
// did, state[STATE_HALTED] = step + 1, and its logits are kept apart where the round's later replays overwrite the step's
// own; then the token and the value into ids / values at the step, the token appended to the penalty's window (a ring of
// RUN_WINDOW once full) and made the next step's input (a valid one after a step that chose none), the position and the
// step advanced. The kept logits are copied by this one block, U float4 a thread in flight (both buffers lie on 16 bytes):
// 128,256 logits 10 us by the greedy choice's 256 threads, 9 by the draw's 1024 (35 and 14 with a float a load).
template <int U>
__device__ __forceinline__ void step_end(const StepEnd &e, int32_t token, float value, int tid, int nt) {
  int32_t *const state = e.state;
  const int32_t step = state[STATE_STEP];
  const bool ends = state[STATE_HALTED] == 0 && halts(token, value, e.params);
  __syncthreads();  // (every thread has read the state)
  if (ends && step + 1 < e.params->steps) {
    typedef float Four __attribute__((ext_vector_type(4)));  // (an array of float4 goes to scratch)
    const Four *const from = reinterpret_cast<const Four *>(e.logits);
    Four *const to = reinterpret_cast<Four *>(e.kept);
    const int n4 = e.n >> 2;
    for (int base = tid; base < n4; base += U * nt) {
      Four v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = from[min(base + u * nt, n4 - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (base + u * nt < n4) to[base + u * nt] = v[u];
    }
    for (int i = 4 * n4 + tid; i < e.n; i += nt) e.kept[i] = e.logits[i];
  }
  if (tid != 0) return;
  e.ids[step] = token;
  e.values[step] = value;
  if (ends) state[STATE_HALTED] = step + 1;
  if (token >= 0) {
    const int32_t count = state[STATE_WINDOW];
    if (count < RUN_WINDOW) {
      e.window[count] = token;
      state[STATE_WINDOW] = count + 1;
    } else {
      const int32_t head = state[STATE_HEAD];
      e.window[head] = token;
      state[STATE_HEAD] = head + 1 == RUN_WINDOW ? 0 : head + 1;
    }
  }
  e.tokens[0] = token >= 0 ? token : 0;
  state[STATE_POS] = state[STATE_POS] + 1;
  state[STATE_STEP] = step + 1;
}

}  // namespace ple
