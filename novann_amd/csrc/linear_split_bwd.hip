// The split-K products of the Linear backward, operands K-major as the
// backward receives them (linear_split.h): no transposed copies.
#include "linear_split.h"

namespace novaq {

bool linear_split_bwd_supported(int64_t D_in, int64_t D_out) { return D_in >= 4 && D_out >= 4; }

int linear_split_wcol_launch(const float* grad, int64_t M, int64_t K, const void* w_q, int w_dtype,
                             const float* w_scale, int64_t N, float* y, hipStream_t stream) {
  Epilogue ep{};
  ep.out_dtype = F32;
  const auto* g = reinterpret_cast<const uint8_t*>(grad);
  const auto* w = static_cast<const uint8_t*>(w_q);
  switch (w_dtype) {
    case E4M3: return split_launch<F32, false, E4M3, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    case E5M2: return split_launch<F32, false, E5M2, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    case E2M1: return split_launch<F32, false, E2M1, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    case BF16: return split_launch<F32, false, BF16, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    case F16: return split_launch<F32, false, F16, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    case F32: return split_launch<F32, false, F32, true>(g, nullptr, M, K, w, w_scale, ep, N, y, nullptr, stream);
    default: return NOVAQ_EDTYPE;
  }
}

int linear_split_tn_launch(const float* a, const float* b, int64_t M, int64_t N, int64_t K,
                           float* c, float* colsum, hipStream_t stream) {
  Epilogue ep{};
  ep.out_dtype = F32;
  return split_launch<F32, true, F32, true>(reinterpret_cast<const uint8_t*>(a), nullptr, M, K,
                                            reinterpret_cast<const uint8_t*>(b), nullptr, ep, N, c,
                                            colsum, stream);
}

}  // namespace novaq
