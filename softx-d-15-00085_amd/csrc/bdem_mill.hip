/*
 * bdem_mill.hip - the lifters' turn as a launch of its own (bdem_turn.hpp),
 * for the steps that sort in full.
 */
#include "bdem_turn.hpp"

namespace bdem {

__global__ __launch_bounds__(TURN_THREADS) void k_turn_lifters(TurnArgs t) {
  __shared__ bdem_float3 tv[TURN_THREADS];
  turn_lifters_block(t.params, t, tv);
}

void launch_turn_lifters(const TurnArgs& t, hipStream_t st) {
  hipLaunchKernelGGL(k_turn_lifters, dim3(1), dim3(TURN_THREADS), 0, st, t);
}

}  // namespace bdem
