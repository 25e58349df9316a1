// Dequantizing GEMM with a tile's activations resident in registers: grouped experts with a few slots each (q4 G = 128,
// BF16 x), from a handful of tokens to about 14 slots an expert; and dense linears (q4 G = 128, q8 G = 64, BF16 or FP32 x)
// that dense_ks does not take: other K than a power of two of spans, more than 16 rows, up to prefill width (short K stays
// with qmm where that is the faster one: the rules are in api_qmm.hip).
//
// What bounds it: the experts' codes, read once a 16-slot tile; the work is weight streaming (4.7 - 5.4 TB/s of codes,
// scales and mins against 6.35 for a plain streaming read; leaving out the dequant, the MFMAs or the SwiGLU changes no
// time). So the split is made for the stream:
//   - a block's Q waves split K into Q slices of four spans (a span: 128 codes, one quantization group, 64 bytes of a
//     row), so that a tile of 16 weight rows is one contiguous piece of memory read by the block at once, and a wave
//     keeps its slice of the tile's 16 activation rows in registers as MFMA operands (64 VGPRs): the K loop has no
//     LDS traffic and no activation loads. A row of 20 spans gets five waves, not eight: spans read by two slices, and
//     128-byte lines split between two waves' loads, cost as much as any other request (K = 2560, 512 experts: eight
//     slices of three spans 4.3 TB/s, five of four 5.0; K = 2048: eight slices of three 2.7, four of four 5.4).
//   - two blocks a compute unit of at most 128 registers, each with one tile of rows in flight a wave, a slot's reload
//     two spans after its unpack (more in flight is slower: lag 0 277 us against 225 for K = 2560, I = 640, M = 200).
//   - the grid is the resident blocks; each takes an equal run of the (tile, round) sequence, to within one round
//     (P units of 16 weight rows times gate and up), and the next tile's first weights are in flight while the last
//     round of the one before computes. A grid of (tile, part) blocks was up to 10 % slower: its last wave is nearly
//     empty, and the dispatcher deals blocks to a die's shader engines in turn, so that a grid whose every other block
//     exits at once left half of the engines idle.
// The Q partial tiles of a round meet in LDS after one barrier (only LDS operations are waited for) and are summed in
// K order by the waves that made them, SwiGLU and the store included.
//   sum_k x * (code * s + m) = s * D + (m - 128 s) * sum_span x with D from v_mfma_f32_16x16x32_bf16 on (128 + code),
// added span by span (qmm_impl.hpp; the second term kept for the end, as gg_kernel does, is 1.6 times as far from 64 bits).
// gate_up + SwiGLU at d = 4096, I = 1024, 512 experts top-10: M = 10 110 -> 88 us (qmm), 64 425 -> 291 (gg_kernel), 200
// 570 -> 413; d = 2560, I = 640 with the shared expert: M = 6 40.6 -> 21.6, 24 210 -> 71, 200 254 -> 180; down + combine
// (K = 640, qmm before): M = 200 136 -> 116, 2048 375 -> 338.
// Dense: the tokens in tiles of 16 (FP32 rows: five tokens as three exact BF16 planes each, fifteen operand rows, so that
// the K loop and its registers are the BF16 ones), the weight streamed once a tile, from the caches after the first.
// Before (qmm) and after, three weights in turn: q4 8192 x 2560 M = 24 19.5 -> 9.4 us, M = 64 36.8 -> 14.2; q8 2560 x 4096
// FP32 rows M = 37 42.0 -> 23.9, 7680 x 2560 FP32 rows M = 128 247 -> 92; the q8 head 248,320 x 2560 at M = 6 228 -> 134 (0.68
// GB: 5.1 TB/s), 151,936 x 4096 at M = 16 380 -> 129.
#include "reg_tiles_impl.hpp"

namespace sx::rt {

bool eligible_grouped(int bits, int64_t G, int64_t N, int64_t K, int64_t M, int64_t A, int64_t E, int act) {
    if (!(bits == 4 && G == 128 && K % 128 == 0 && K >= 256 && K <= 4096 && act == SX_ACT_BF16)) return false;
    // 32-bit offsets into an expert's rows and a 32-bit (tile, round) sequence
    return N * (K / 2) < (int64_t(1) << 32) && (M * A / 16 + E + 2) * (N / 16 + 1) < (int64_t(1) << 31) && N < (1 << 22);
}

hipError_t launch_grouped(int mode, const void *x, const sx_qview *w, void *y, const int32_t *ws, int64_t M, int64_t A,
                          int64_t E, hipStream_t stream) {
    detail::Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y, p.ws = ws;
    p.A = A, p.N = w->N / E, p.K = w->K, p.E = (int)E, p.nspan = (int)(w->K / 128);
    const int split = detail::split_of(p.nspan, detail::kSplits4);
    if (split < 0) return hipErrorInvalidValue;
    const int P = detail::lanes_of(4, detail::kSplits4[split].q, false);
    const int64_t out_rows = mode == qmm::SWIGLU ? p.N / 2 : p.N, unit = mode == qmm::SWIGLU ? 16 : 32;
    const int64_t units = (out_rows + unit - 1) / unit;
    p.rounds = (int)((units + P - 1) / P);
    const int64_t S = M * A, most = std::min<int64_t>(S, S / 16 + E + 2) * p.rounds;
    if (mode == qmm::COMBINE) return detail::go<4, qmm::COMBINE, uint16_t, float>(p, split, most, stream);
    if (mode == qmm::SWIGLU) return detail::go<4, qmm::SWIGLU, uint16_t, uint16_t>(p, split, most, stream);
    return detail::go<4, qmm::GATHER, uint16_t, uint16_t>(p, split, most, stream);
}

bool eligible_dense(int bits, int64_t G, int64_t N, int64_t K, int64_t M, int act) {
    const int64_t span = bits == 4 ? 128 : 64, nspan = K / span;
    if (G != span || K % span != 0 || K > 4096) return false;
    if ((bits == 4 ? detail::split_of((int)nspan, detail::kSplits4) : detail::split_of((int)nspan, detail::kSplits8)) < 0)
        return false;
    const int64_t tiles = act == SX_ACT_F32 ? (M + 4) / 5 : (M + 15) / 16;
    return N * (K * bits / 8) < (int64_t(1) << 32) && tiles * (N / 32 + 1) < (int64_t(1) << 31) && N < (1 << 27);
}

Block dense_block(int bits, int64_t K, int act) {
    const detail::Split s = bits == 4 ? detail::kSplits4[detail::split_of((int)(K / 128), detail::kSplits4)]
                                      : detail::kSplits8[detail::split_of((int)(K / 64), detail::kSplits8)];
    return {s.q, s.spw, detail::lanes_of(bits, s.q, act == SX_ACT_F32)};
}

hipError_t launch_dense(int bits, const void *x, const sx_qview *w, void *y, int64_t M, int act, int out_act,
                        hipStream_t stream) {
    detail::Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y;
    p.A = 1, p.N = w->N, p.K = w->K, p.E = 1, p.nspan = (int)(w->K / (bits == 4 ? 128 : 64)), p.dense_M = M;
    return bits == 4 ? detail::dense_q4(p, act, out_act, stream) : detail::dense_q8(p, act, out_act, stream);
}

}  // namespace sx::rt
