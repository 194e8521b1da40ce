// Prefill SwiGLU up-projection and logits GEMMs.
#include "gemm_launch.hpp"

namespace hb {

hipError_t gemm_swiglu(const f16* W, const f16* X, int N, int T, int K, const EpiSwiGLU& e,
                       hipStream_t st, int kw) {
  return launch_gemm(W, X, N, T, K, e, st, kw);
}
// The head's weights come from HBM: every layer's pass through the memory-side
// cache between two calls, while the time model was fitted to repeated launches.
// With one 256-token tile it picks 128x256, and 192x256, with a third fewer blocks
// that each read the same activations, gains more than it loses. 32000 columns,
// logits + loss, us, 128x256 -> 192x256. Models on streams of their own, whose work
// fills the compute units that 167 blocks leave free: K 4096 at 130 / 200 / 256 tokens
// 78 / 84 / 88 -> 67 / 70 / 73, K 2560 at 190 57.7 -> 48.4, K 1536 37.6 -> 31.7. Models
// in turn on one stream, 136 / 200 / 256 tokens: K 8192 166 / 171 / 175 ->
// 159 / 167 / 173, K 4096 87.3 / 91.1 / 95.4 -> 83.6 / 87.7 / 92.4, K 2048
// 51.7 / 55.6 / 59.6 -> 50.1 / 53.9 / 57.2, and the other way K 2560 59.2 / 63.0 / 67.0
// -> 59.7 / 65.5 / 71.3, K 1536 43.1 / 46.1 / 48.8 -> 43.4 / 47.6 / 50.9.
// (One model's weights read again at once: K 4096 at 200 83.8 -> 80.8, K 2560 50.2 -> 52.3.)
hipError_t gemm_logits(const f16* W, const f16* X, int N, int T, int K, const EpiLogits& e,
                       hipStream_t st, int kw) {
  if (!gemm_fits(N, T, K)) return hipErrorInvalidValue;
  GemmChoice c = gemm_tile(N, T, K, 1);
  if (T > 128 && T <= 256 && c.tile == GEMM_128x256) c.tile = GEMM_192x256;
  return launch_choice(c, W, X, N, T, K, e, st, kw);
}

}  // namespace hb
