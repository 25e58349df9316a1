// Dequantizing GEMM with the activations of a tile resident in registers (reg_tiles.hip): the grouped experts with a
// few slots each.
#pragma once
#include "qmm.hpp"

namespace sx::rt {

// Slots an expert up to which the grouped entry points take these tiles where the 64-slot tiles (gemm_grouped.hpp) take
// the shape too: a tile is 16 slots, and a bucket's further tiles read its weights again. gate_up at d = 4096, I = 1024,
// 512 experts top-10 against gg_kernel: 13.7 slots an expert 578 / 592 us, 14.6 604 / 594, 15.6 651 / 600; d = 2560, I =
// 640: 14.0 240 / 269, 15.6 275 / 271.
constexpr int64_t kMaxSlotsAnExpert = 14;

// The grouped experts: q4 G = 128, BF16 activations, K of 2 .. 32 spans of 128 codes; N rows an expert.
bool eligible_grouped(int bits, int64_t G, int64_t N, int64_t K, int64_t M, int64_t A, int64_t E, int act);
// mode: qmm::SWIGLU (h [S, N/2]), qmm::GATHER (y [S, N]), qmm::COMBINE (FP32 partials [S, N]); N = w->N / E.
hipError_t launch_grouped(int mode, const void *x, const sx_qview *w, void *y, const int32_t *ws, int64_t M, int64_t A,
                          int64_t E, hipStream_t stream);

// A dense linear: q4 G = 128 / q8 G = 64, K of whole spans up to 4096, BF16 or FP32 x (act / out_act as linear's).
bool eligible_dense(int bits, int64_t G, int64_t N, int64_t K, int64_t M, int act);
hipError_t launch_dense(int bits, const void *x, const sx_qview *w, void *y, int64_t M, int act, int out_act,
                        hipStream_t stream);
// A dense block (an eligible shape): K slices, spans a slice, output units (32 rows) it works on at once.
struct Block {
    int slices, spans, units;
};
Block dense_block(int bits, int64_t K, int act);

}  // namespace sx::rt
