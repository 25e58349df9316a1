// Prefill-width grouped expert GEMM (q4 G = 128 experts, BF16 activations) on the matrix cores.
#pragma once
#include "qmm.hpp"

namespace sx::gg {

// Tokens from which the grouped entry points take this kernel (the reference switches its grouped path to the WMMA
// tiles at prefill width; at verify width buckets hold a few slots and the register tiles' one pass over the weights wins).
constexpr int64_t kPrefillMinTokens = 32;

bool eligible(int bits, int64_t G, int64_t K, int act);
// Tokens from which launch_dense's tiles can be the faster ones for a dense linear (the rule is in api_qmm.hip): below,
// their blocks leave most of the chip idle. 4096 x 4096, the register tiles against the K-split tiles (gs_kernel): q4
// 12.4 / 23.0 us at M = 64, 17.2 / 23.1 at 96, 26.5 / 21.2 at 200; q8 16.9 / 26.0 at 48.
constexpr int64_t kDenseMinTokens = 96, kDenseMinTokensQ8 = 48;
constexpr int64_t dense_min_tokens(int bits) { return bits == 8 ? kDenseMinTokensQ8 : kDenseMinTokens; }
// Up to this many tokens launch_dense splits K over each block's waves (gs_kernel: 64 x 64 tiles, a quarter of the steps
// each); above, 128-token units (gw_kernel). 4096 x 4096, gs_kernel / gw_kernel: q4 25.0 / 33.6 us at M = 256, 47.4 / 40.1
// at 512; q8 28.7 / 55.3, 55.3 / 58.6. Where gs_kernel needs three rounds and more (q4
// 8192 x 2560 M = 512 59.7 / 32.1) gw_kernel would be faster from fewer tokens, but its sums over the whole K round more
// (FP32 outputs 2.9e-6 against 1.7e-6 of the norm), so those stay.
constexpr int64_t kDenseSplitMaxTokens = 512;
// The dense linears the tiles take: eligible's q4, and q8 (G = 64, K % 256 == 0, K <= 4096, BF16 x).
bool eligible_dense(int bits, int64_t G, int64_t K, int act);
// A dense linear at prefill width: y [M, w->N] (BF16 or FP32) = x [M, K] (BF16) . deq(w)^T (eligible_dense(bits, G, K,
// BF16)), in gs_kernel's blocks of 64 tokens x 64 rows up to kDenseSplitMaxTokens tokens, above in gw_kernel's units of 128
// tokens x 256 rows.
hipError_t launch_dense(const void *x, const sx_qview *w, void *y, int64_t M, int out_act, hipStream_t stream);
// mode: qmm::SWIGLU (h [S, N/2], BF16), qmm::GATHER (y [S, N], BF16), qmm::COMBINE (FP32 partials [S, N]); N = w->N / E.
hipError_t launch(int mode, const void *x, const sx_qview *w, void *y, const int32_t *ws, int64_t M, int64_t A,
                  int64_t E, hipStream_t stream);

}  // namespace sx::gg
