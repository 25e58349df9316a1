// C-ABI entry points of the dequantizing GEMMs: dense linear (q4 / q8) and the per-slot and grouped MoE experts.
// Host-side preconditions follow the reference launchers (kernels/linear_q4.hip:353-440, linear_q8.hip:192-223,
// moe_grouped.hip:476-556); the work runs in qmm_impl.hpp.
#include "common.hpp"
#include "gemm_grouped.hpp"
#include "dense_ks.hpp"
#include "qmm.hpp"
#include "reg_tiles.hpp"

#include <algorithm>
#include <cmath>

namespace sx {
namespace {

using qmm::Params;

constexpr int64_t kMaxN = 0x7fffffff;
constexpr int64_t kMaxK = 1 << 24;
constexpr size_t kLdsBudget = 56 * 1024;  // x staging per block: 2 blocks (8 waves) a CU of the 160 KB

// Checks of a weight view shared by every entry point (linear_q4.hip:353-362).
int check_view(const char *fn, const sx_qview *w, int bits) {
    if (w == nullptr) {
        set_error(cat(fn, ": null weight view"));
        return SX_EINVAL;
    }
    if (!(w->q && w->scale && w->minv)) {
        set_error(cat(fn, ": null weight pointer (q=", (const void *)w->q, ", scale=", w->scale, ", min=", w->minv, ")"));
        return SX_EINVAL;
    }
    if (!(w->G == 32 || w->G == 64 || w->G == 128)) {
        set_error(cat(fn, ": group size ", w->G, " unsupported (32, 64 or 128)"));
        return SX_EINVAL;
    }
    if (!(w->N >= 1 && w->N <= kMaxN)) {
        set_error(cat(fn, ": N = ", w->N, ", expected 1..", kMaxN));
        return SX_EINVAL;
    }
    if (!(w->K >= w->G && w->K <= kMaxK && w->K % w->G == 0)) {
        set_error(cat(fn, ": K = ", w->K, " must be a positive multiple of group size ", w->G, " and <= ", kMaxK));
        return SX_EINVAL;
    }
    if (!aligned(w->q, 16)) {
        set_error(cat(fn, ": code array ", (const void *)w->q, " must be 16-byte aligned for vector loads"));
        return SX_EINVAL;
    }
    return SX_OK;
}

// Activation rows one block stages in LDS: up to `want` (<= 16), as many as fit the budget.
int rows_that_fit(int bits, int nsplit, int64_t K, int64_t G, int want, size_t budget = kLdsBudget) {
    int r = want < 16 ? want : 16;
    while (r > 1 && qmm::lds_bytes(bits, nsplit, K, G, r, 1) > budget) --r;
    return r;
}

// Tiles a block covers: 4 waves x tiles a wave, enough waves for the chip (~8 a CU) but no more than the work.
int tiles_per_chunk(int64_t total_tiles, int cus) {
    const int64_t waves = (int64_t)cus * 8;
    int64_t tpw = (total_tiles + waves - 1) / waves;
    tpw = tpw < 1 ? 1 : tpw > 16 ? 16 : tpw;
    return (int)(tpw * qmm::kWaves);
}

int launch_qmm(const char *fn, int mode, int bits, int act_x, int act_y, Params &p, int64_t units, int64_t rows_out,
               int64_t grid_y, hipStream_t stream) {
    const int64_t tiles = (rows_out + qmm::kTile - 1) / qmm::kTile;
    p.tiles_per_chunk = tiles_per_chunk(tiles * units, device_cus());
    p.nchunks = (int)((tiles + p.tiles_per_chunk - 1) / p.tiles_per_chunk);
    const int64_t gx = units * p.nchunks;
    SX_CHECK(gx >= 1 && gx <= 0x7fffffff && grid_y <= 65535, fn, " grid ", gx, " x ", grid_y, " out of range");
    SX_HIP(qmm::launch(mode, bits, act_x, act_y, p, dim3((unsigned)gx, (unsigned)grid_y), stream), fn);
    return SX_OK;
}

enum Kernel { kKSplit, kRegTiles, kWideTiles, kQmm };

// Whether qmm takes a dense linear rather than the register tiles, which read a tile's rows of x into each wave's registers
// first: at short K that costs more than the tile's weights. The lines are in qmm's blocks a compute unit (staged rows x 4
// waves' weight tiles a block), which its time follows. Both sides measured, qmm / register tiles in us:
//   - on qmm's straight-line path: up to three blocks a compute unit (two at K = 2048), FP32 rows four and at K = 512 any
//     number. q8 5120 x 512 M = 24 5.3 / 11.8, 8192 x 1024 M = 37 9.5 / 11.9, 14000 x 2048 M = 24 15.7 / 16.4, M = 32 22.9 /
//     16.6; q4 8192 x 1024 M = 64 7.8 / 9.6, 14000 x 1024 M = 95 18.4 / 14.8; FP32 rows, q8 5120 x 1024 M = 37 13.8 /
//     18.9, 8192 x 512 M = 200 26.9 / 38.9, 8192 x 1024 M = 128 47.4 / 42.2. At K = 4096 only as one block a compute unit
//     where the register tiles need two rounds (5120 x 4096 M = 17 q4 10.1 / 11.6, q8 15.0 / 17.1);
//   - on its general path below K = 1024, where a block of register tiles holds more than four times the x it needs (each
//     of its output units has its own, and slices may overlap), for one round of blocks (two where it holds more than 8 KB
//     a row): q8 5120 x 768 M = 24 10.3 / 11.3, 14000 x 768 M = 24 14.7 / 12.1; q4 5120 x 640 M = 37 8.1 / 10.9, 5120 x 640 M =
//     200 19.0 / 14.0. FP32 rows, which the register tiles read in more tiles: two rounds, with a bar that rises with the
//     rows qmm stages, less where the register tiles need a second round: q8 5120 x 768 M = 6 12.9 / 14.3, 5120 x 896 M = 32
//     15.8 / 19.1, 1000 x 896 M = 24 15.8 / 14.4; slices that overlap by half any number (q8 5120 x 320 M = 200 20.7 / 28.5);
//   - FP32 rows whose 5-token tiles are more than an eighth of the chip, so that a block passes from tile to tile and
//     reads x again: q4 2560 x 512 M = 300 17.4 / 23.8, 1000 x 1152 M = 200 16.9 / 22.3; and a single FP32 row up to K = 1280
//     (q4 8192 x 1152 M = 1 10.4 / 11.1).
bool qmm_is_faster(int bits, const sx_qview *w, int64_t M, int act, int cus) {
    const bool f32 = act == SX_ACT_F32;
    const int64_t K = w->K, span = bits == 4 ? 128 : 64, nspan = K / span;
    const rt::Block b = rt::dense_block(bits, K, act);
    const int64_t reg_tiles = (M + (f32 ? 4 : 15)) / (f32 ? 5 : 16);
    const int64_t reg_rounds = reg_tiles * (((w->N + 31) / 32 + b.units - 1) / b.units);  // of one block
    const int rows = rows_that_fit(bits, f32 ? 3 : 1, K, w->G, (int)(M < 16 ? M : 16));
    const int64_t tiles = (w->N + qmm::kTile - 1) / qmm::kTile, per_block = tiles_per_chunk(tiles, cus);
    // qmm's blocks, each counted by the tiles its waves work through
    const int64_t blocks = (M + rows - 1) / rows * ((tiles + per_block - 1) / per_block) * (per_block / qmm::kWaves);
    if (qmm::straight_line(bits, K, w->G, f32, rows)) {
        if (f32 && K <= 512) return true;
        if (K <= 2048 && blocks <= std::min<int64_t>(f32 ? 4 : 3, 4096 / K) * cus) return true;
        return !f32 && blocks <= cus && reg_rounds > cus;
    }
    const int64_t held = (int64_t)b.slices * b.spans * b.units;  // spans of x in a block's registers
    if (held <= 16 || (f32 && held * span <= 2048)) return false;  // K = 256: little x (q4 5120 x 256 M = 24 6.8 / 6.2)
    if (!f32) return K < 1024 && 2 * held > 9 * nspan && blocks <= (held * span > 4096 ? 2 : 1) * cus;
    if (reg_tiles > cus / 8 && reg_rounds > cus &&
        ((K <= 512 && blocks <= 3 * cus) || (K > 1024 && K <= 1280 && blocks <= 2 * cus)))
        return true;
    if (K >= 1024) return M == 1 && K <= 1280 && blocks <= cus;
    if (80 * held <= (320 + (reg_rounds > cus ? 4 : bits == 4 ? 7 : 10) * rows) * nspan) return false;
    return blocks <= 2 * cus || 2 * b.slices * b.spans >= 3 * nspan;
}

// Which kernel takes a dense linear. Up to 16 rows with a power of two of spans: dense_ks. Otherwise the register tiles
// where they take the shape (reg_tiles.hpp), against
//   - the 64-token tiles (from dense_min_tokens tokens): above kDenseSplitMaxTokens tokens those; up to there by the two
//     kernels' times, each linear in its rounds: gs_kernel's 64 x 64 blocks in whole waves of the chip (4096 x 4096, q4
//     21 us a wave, q8 27), the register tiles' (16 tokens x 32 rows) units a compute unit (q4 7 us and 2.3 each at K =
//     4096, q8 9 and 4.6), with a fifth in gs_kernel's favour. Both sides measured, register tiles / gs_kernel: q4 4096
//     x 4096 M = 128 16.2 / 20.4 us, M = 200 26.5 / 21.2; 12288 x 4096 M = 400 98.9 / 120.1; 8192 x 2560 M = 128 18.8 /
//     15.2; q8 4096 x 4096 M = 48 16.9 / 26.0, 12288 x 4096 M = 64 34.2 / 28.0;
//   - qmm at short K (qmm_is_faster).
Kernel dense_kernel(int bits, const sx_qview *w, int64_t M, int act, int out_act, int cus) {
    const int64_t N = w->N, K = w->K;
    if (dks::eligible(bits, w->G, N, K, M, act, out_act, cus)) return kKSplit;
    const bool wide = M >= gg::dense_min_tokens(bits) && gg::eligible_dense(bits, w->G, K, act) && aligned(w->scale, 4) &&
                      aligned(w->minv, 4);
    if (!rt::eligible_dense(bits, w->G, N, K, M, act)) return wide ? kWideTiles : kQmm;
    if (wide) {
        if (M > gg::kDenseSplitMaxTokens) return kWideTiles;
        const double units = (double)((M + 15) / 16) * (double)((N + 31) / 32) / cus, k = K / 4096.0;
        const int64_t blocks = (M + 63) / 64 * ((N + 63) / 64);
        const double waves = (double)((blocks + cus - 1) / cus);
        const double reg = bits == 4 ? 7 + 2.3 * k * units : 9 + 4.6 * k * ceil(units);
        const double split = waves * (bits == 4 ? 6 + 15 * k : 4 + 23 * k);
        return reg * 1.2 < split ? kRegTiles : kWideTiles;
    }
    return qmm_is_faster(bits, w, M, act, cus) ? kQmm : kRegTiles;
}

int linear(const char *fn, int bits, const void *x, const sx_qview *w, void *y, int64_t M, int act, int out_act,
           sx_stream stream) {
    SX_CHECK(x != nullptr && y != nullptr, fn, " null pointer (x=", x, ", y=", y, ")");
    if (int rc = check_view(fn, w, bits)) return rc;
    SX_CHECK(M >= 1 && M <= 65535ll * 8, fn, " M (rows of x) = ", M, ", expected 1..", 65535ll * 8);
    SX_CHECK(aligned(x, 16), fn, " x ", x, " must be 16-byte aligned for vector loads");
    SX_CHECK(act == SX_ACT_F32 || act == SX_ACT_BF16, fn, " unsupported activation dtype ", act);
    SX_CHECK(out_act == act || (act == SX_ACT_BF16 && out_act == SX_ACT_F32), fn, " output dtype ", out_act,
             " with input ", act, " unsupported (same dtype, or BF16 -> F32)");
    SX_CHECK(apart(x, M * w->K * act_bytes(act), y, M * w->N * act_bytes(out_act)), fn, " output y [", y, ", +",
             M * w->N * act_bytes(out_act), " B) overlaps input x [", x, ", +", M * w->K * act_bytes(act), " B)");
    switch (dense_kernel(bits, w, M, act, out_act, device_cus())) {
    case kKSplit: {  // decode width: K split over a block
        dks::Params d{};
        d.x = x, d.q = w->q, d.scale = w->scale, d.minv = w->minv, d.y = y, d.M = (int)M, d.N = w->N, d.K = w->K;
        SX_HIP(dks::launch(bits, w->G, act, out_act, d, device_cus(), stream_of(stream)), fn);
        return SX_OK;
    }
    case kRegTiles:
        SX_HIP(rt::launch_dense(bits, x, w, y, M, act, out_act, stream_of(stream)), fn);
        return SX_OK;
    case kWideTiles:  // prefill width
        SX_HIP(gg::launch_dense(x, w, y, M, out_act, stream_of(stream)), fn);
        return SX_OK;
    case kQmm: break;
    }
    const int nsplit = act == SX_ACT_F32 ? 3 : 1;
    const int rows = rows_that_fit(bits, nsplit, w->K, w->G, (int)(M < 16 ? M : 16));
    SX_CHECK(qmm::lds_bytes(bits, nsplit, w->K, w->G, rows, 1) <= 160 * 1024, fn, " K = ", w->K,
             " too long to stage one activation row in LDS");
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y;
    p.M = M, p.A = 1, p.E = 1, p.N = w->N, p.K = w->K, p.G = (int)w->G, p.max_rows = rows;
    return launch_qmm(fn, qmm::DENSE, bits, act, out_act, p, 1, w->N, (M + rows - 1) / rows, stream_of(stream));
}

int experts_common(const char *fn, const void *x, const sx_qview *w, int64_t E, int64_t M, int64_t A, void *y,
                   int act) {
    SX_CHECK(x != nullptr && y != nullptr, fn, " null pointer (x=", x, ", y=", y, ")");
    if (int rc = check_view(fn, w, 4)) return rc;
    SX_CHECK(E >= 1 && w->N % E == 0, fn, " weight has ", w->N, " rows, not a multiple of E = ", E, " experts");
    SX_CHECK(M >= 1 && M <= 65535, fn, " M (tokens) = ", M, ", expected 1..65535");
    SX_CHECK(A >= 1 && A <= 64 && A <= E, fn, " A (active experts per token) = ", A, ", expected 1..min(64, E=", E, ")");
    SX_CHECK(aligned(x, 16), fn, " input ", x, " must be 16-byte aligned");
    SX_CHECK(act == SX_ACT_F32 || act == SX_ACT_BF16, fn, " unsupported activation dtype ", act);
    return SX_OK;
}

// The route workspace checks of moe_grouped.hip:476-497, plus the header E read back from nothing: the layout is
// recomputed on the host from (M, A, E).
int grouped_common(const char *fn, const void *x, const sx_qview *w, int64_t E, int64_t M, int64_t A, const void *ws,
                   size_t ws_bytes, void *y, int act, int math) {
    if (int rc = experts_common(fn, x, w, E, M, A, y, act)) return rc;
    SX_CHECK(ws != nullptr, fn, " null workspace");
    SX_CHECK(E <= 1023 && M * A <= (1 << 20), fn, " E = ", E, " (<= 1023), M*A = ", M * A, " (<= 2^20)");
    size_t need = 0;
    if (int rc = sx_moe_route_workspace_bytes(M, A, E, &need)) return rc;
    SX_CHECK(ws_bytes >= need, fn, " workspace of ", ws_bytes, " bytes, needs ", need, " for M = ", M, ", A = ", A,
             ", E = ", E);
    SX_CHECK(math == SX_MOE_F32 || math == SX_MOE_WMMA_BF16 || math == SX_MOE_WMMA_F16, fn, " unknown math ", math);
    return SX_OK;
}

// Which kernel takes a grouped call: the 64-slot tiles from kPrefillMinTokens tokens and more than kMaxSlotsAnExpert
// slots an expert on average, the register tiles otherwise (and where the 64-slot ones do not take the shape), qmm for
// the rest (other group sizes, FP32 activations, long K) and, below kPrefillMinTokens tokens, on its straight-line path
// with few weight tiles (16 rows of one slot tile) a compute unit: K = 1024 up to 21; K = 2048, where the register tiles
// are the faster ones while every block is alone on its compute unit (up to 4), 4 to 9. Measured, qmm / register tiles in
// us (weight tiles a compute unit): down, E = 8 4096 x 1024 A = 2 M = 2 (4) 8.5 / 10.2, M = 24 (13) 11.9 / 16.1; E = 32 2048 x
// 1024 A = 4 M = 31 (20.5) 16.6 / 17.0; E = 512 4096 x 1024 A = 10 M = 2 (20) 18.4 / 21.4, M = 4 (40) 31.1 / 25.7, M = 12 (120)
// 61.0 / 48.9; gate_up, E = 128 d = 2048 I = 768 A = 8 M = 1 (3) 9.6 / 8.2, M = 2 (6) 10.0 / 11.6, M = 4 (12) 16.5 / 14.5; E = 64
// d = 2048 I = 512 A = 8 M = 4 (8) 11.4 / 12.1.
// The rule looks at the weight's rows alone, so that a gather and its SwiGLU form run the same kernel (the same bits).
Kernel grouped_kernel(const sx_qview *w, int64_t M, int64_t A, int64_t E, int act, int cus) {
    const bool wide = M >= gg::kPrefillMinTokens && gg::eligible(4, w->G, w->K, act) && aligned(w->scale, 4) &&
                      aligned(w->minv, 4);
    if (!rt::eligible_grouped(4, w->G, w->N / E, w->K, M, A, E, act)) return wide ? kWideTiles : kQmm;
    if (wide && M * A > rt::kMaxSlotsAnExpert * E) return kWideTiles;
    const int64_t S = M * A, slot_tiles = std::min(S, S / 16 + E + 2);
    const int64_t tiles = slot_tiles * ((w->N / E + qmm::kTile - 1) / qmm::kTile);
    const bool few = w->K <= 1024 ? tiles <= 21 * cus : w->K <= 2048 && tiles > 4 * cus && tiles <= 9 * cus;
    if (M < gg::kPrefillMinTokens && few && qmm::straight_line(4, w->K, w->G, false, 12)) return kQmm;
    return kRegTiles;
}

const char *kernel_name(Kernel k, bool k_split) {
    switch (k) {
    case kKSplit: return "k_split";
    case kRegTiles: return "register_tiles";
    case kWideTiles: return k_split ? "wide_tiles_k_split" : "wide_tiles";
    default: return "qmm";
    }
}

}  // namespace
}  // namespace sx

using namespace sx;

extern "C" {

int sx_linear_q4(const void *x, const sx_qview *w, void *y, int64_t M, int act, int out_act, sx_stream stream) {
    return linear("sx_linear_q4", 4, x, w, y, M, act, out_act, stream);
}

int sx_linear_q8(const void *x, const sx_qview *w, void *y, int64_t M, int act, int out_act, sx_stream stream) {
    return linear("sx_linear_q8", 8, x, w, y, M, act, out_act, stream);
}

const char *sx_linear_kernel(const sx_qview *w, int bits, int64_t M, int act, int out_act, int cus) {
    const char *fn = "sx_linear_kernel";
    if (!(bits == 4 || bits == 8) || M < 1) {
        set_error(cat(fn, ": bits = ", bits, " (4 or 8), M = ", M, " (>= 1)"));
        return nullptr;
    }
    if (check_view(fn, w, bits)) return nullptr;
    return kernel_name(dense_kernel(bits, w, M, act, out_act, cus > 0 ? cus : device_cus()),
                       M <= gg::kDenseSplitMaxTokens);
}

const char *sx_experts_grouped_kernel(const sx_qview *w, int64_t E, int64_t M, int64_t A, int act, int cus) {
    const char *fn = "sx_experts_grouped_kernel";
    if (check_view(fn, w, 4)) return nullptr;
    if (!(E >= 1 && w->N % E == 0 && M >= 1 && A >= 1 && A <= E)) {
        set_error(cat(fn, ": E = ", E, " of ", w->N, " rows, M = ", M, ", A = ", A));
        return nullptr;
    }
    return kernel_name(grouped_kernel(w, M, A, E, act, cus > 0 ? cus : device_cus()), false);
}

int sx_mtp_head_pick(const void *x, const sx_qview *w, int bits, float *logits, const uint32_t *router_err,
                     const uint32_t *expert_err, const uint32_t *attn_err, const unsigned long long *emb_err,
                     sx_mtp_pick_t *out, void *workspace, size_t workspace_bytes, sx_stream stream) {
    const char *fn = "sx_mtp_head_pick";
    SX_CHECK(bits == 4 || bits == 8, fn, " bits = ", bits, ", expected 4 or 8");
    SX_CHECK(x && logits && router_err && expert_err && attn_err && emb_err && out && workspace, fn, " null pointer");
    if (int rc = check_view(fn, w, bits)) return rc;
    SX_CHECK(aligned(x, 16), fn, " x ", x, " must be 16-byte aligned for vector loads");
    SX_CHECK(apart(x, w->K * 2, logits, w->N * 4), fn, " logits overlap x");
    SX_CHECK(workspace_bytes >= sizeof(pick::Workspace), fn, " workspace ", workspace_bytes, " bytes, need ",
             sizeof(pick::Workspace));
    SX_CHECK(aligned(workspace, 16), fn, " workspace must be 16-byte aligned");
    const pick::Args pa{static_cast<pick::Workspace *>(workspace), router_err, expert_err, attn_err, emb_err, out};
    const int cus = device_cus();
    if (cus <= pick::kMaxParts && dks::eligible(bits, w->G, w->N, w->K, 1, SX_ACT_BF16, SX_ACT_F32, cus)) {
        dks::Params d{};
        d.x = x, d.q = w->q, d.scale = w->scale, d.minv = w->minv, d.y = logits, d.M = 1, d.N = w->N, d.K = w->K;
        d.pick = pa;
        SX_HIP(dks::launch(bits, w->G, SX_ACT_BF16, SX_ACT_F32, d, cus, stream_of(stream)), fn);
        return SX_OK;
    }
    // other shapes: the GEMV, then the pick over the logits
    if (int rc = linear(fn, bits, x, w, logits, 1, SX_ACT_BF16, SX_ACT_F32, stream)) return rc;
    return sx_mtp_pick_ws(logits, w->N, router_err, expert_err, attn_err, emb_err, out, workspace, workspace_bytes,
                          stream);
}

int sx_linear_q4_experts_gather(const void *x, const sx_qview *w, int64_t E, const int32_t *ids, int64_t M, int64_t A,
                                void *y, int act, uint32_t *err, sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_gather";
    if (int rc = experts_common(fn, x, w, E, M, A, y, act)) return rc;
    SX_CHECK(ids != nullptr && err != nullptr, fn, " null pointer (ids=", (const void *)ids, ", err=", (void *)err, ")");
    const int64_t N = w->N / E, es = act_bytes(act);
    SX_CHECK(apart(x, M * w->K * es, y, M * A * N * es), fn, " output overlaps input");
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y, p.ids = ids, p.err = err;
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G, p.max_rows = 1;
    return launch_qmm(fn, qmm::SLOT_GATHER, 4, act, act, p, M * A, N, 1, stream_of(stream));
}

int sx_linear_q4_experts_gather_swiglu(const void *x, const sx_qview *w, int64_t E, const int32_t *ids, int64_t M,
                                       int64_t A, void *h, int act, uint32_t *err, sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_gather_swiglu";
    if (int rc = experts_common(fn, x, w, E, M, A, h, act)) return rc;
    SX_CHECK(ids != nullptr && err != nullptr, fn, " null pointer (ids=", (const void *)ids, ", err=", (void *)err, ")");
    const int64_t N = w->N / E, es = act_bytes(act);
    SX_CHECK(N % 2 == 0, fn, " SwiGLU gather needs an even row count per expert ([gate | up]), got ", N);
    SX_CHECK(apart(x, M * w->K * es, h, M * A * (N / 2) * es), fn, " output overlaps input");
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = h, p.ids = ids, p.err = err;
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G, p.max_rows = 1;
    return launch_qmm(fn, qmm::SLOT_SWIGLU, 4, act, act, p, M * A, N / 2, 1, stream_of(stream));
}

int sx_linear_q4_experts_combine(const void *h, const sx_qview *w, int64_t E, const int32_t *ids, const float *coef,
                                 int64_t M, int64_t A, void *y, int act, uint32_t *err, sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_combine";
    if (int rc = experts_common(fn, h, w, E, M, A, y, act)) return rc;
    SX_CHECK(ids != nullptr && err != nullptr && coef != nullptr, fn, " null pointer (ids=", (const void *)ids,
             ", coef=", (const void *)coef, ", err=", (void *)err, ")");
    const int64_t N = w->N / E, es = act_bytes(act);
    SX_CHECK(apart(h, M * A * w->K * es, y, M * N * es), fn, " output overlaps input");
    const int nsplit = act == SX_ACT_F32 ? 3 : 1;
    SX_CHECK(qmm::lds_bytes(4, nsplit, w->K, w->G, (int)A, (int)A) <= 96 * 1024, fn, " A x K = ", A, " x ", w->K,
             " activation rows exceed the LDS the per-token combine stages");
    Params p{};
    p.x = h, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y, p.ids = ids, p.coef = coef, p.err = err;
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G, p.max_rows = (int)A;
    return launch_qmm(fn, qmm::SLOT_COMBINE, 4, act, act, p, M, N, 1, stream_of(stream));
}

int sx_linear_q4_experts_gather_grouped(const void *x, const sx_qview *w, int64_t E, const void *ws, size_t ws_bytes,
                                        int64_t M, int64_t A, void *y, int act, int math, sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_gather_grouped";
    if (int rc = grouped_common(fn, x, w, E, M, A, ws, ws_bytes, y, act, math)) return rc;
    const int64_t N = w->N / E, es = act_bytes(act), S = M * A;
    SX_CHECK(apart(x, M * w->K * es, y, S * N * es), fn, " y overlaps x");
    const Kernel kernel = grouped_kernel(w, M, A, E, act, device_cus());
    const int32_t *route = static_cast<const int32_t *>(ws);
    if (kernel != kQmm) {
        SX_HIP(kernel == kRegTiles ? rt::launch_grouped(qmm::GATHER, x, w, y, route, M, A, E, stream_of(stream))
                                   : gg::launch(qmm::GATHER, x, w, y, route, M, A, E, stream_of(stream)), fn);
        return SX_OK;
    }
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y, p.ws = static_cast<const int32_t *>(ws);
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G;
    p.max_rows = rows_that_fit(4, act == SX_ACT_F32 ? 3 : 1, w->K, w->G, (int)(S < 16 ? S : 16));
    const int64_t units = S < S / 16 + E + 2 ? S : S / 16 + E + 2;  // tiles: at most one a slot
    return launch_qmm(fn, qmm::GATHER, 4, act, act, p, units, N, 1, stream_of(stream));
}

int sx_linear_q4_experts_gather_swiglu_grouped(const void *x, const sx_qview *w, int64_t E, const void *ws,
                                               size_t ws_bytes, int64_t M, int64_t A, void *h, int act,
                                               sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_gather_swiglu_grouped";
    if (int rc = grouped_common(fn, x, w, E, M, A, ws, ws_bytes, h, act, SX_MOE_F32)) return rc;
    const int64_t N = w->N / E, es = act_bytes(act), S = M * A;
    SX_CHECK(N % 2 == 0, fn, " SwiGLU gather needs an even row count per expert ([gate | up]), got ", N);
    SX_CHECK(apart(x, M * w->K * es, h, S * (N / 2) * es), fn, " h overlaps x");
    const Kernel kernel = grouped_kernel(w, M, A, E, act, device_cus());
    const int32_t *route = static_cast<const int32_t *>(ws);
    if (kernel != kQmm) {
        SX_HIP(kernel == kRegTiles ? rt::launch_grouped(qmm::SWIGLU, x, w, h, route, M, A, E, stream_of(stream))
                                   : gg::launch(qmm::SWIGLU, x, w, h, route, M, A, E, stream_of(stream)), fn);
        return SX_OK;
    }
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = h, p.ws = static_cast<const int32_t *>(ws);
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G;
    p.max_rows = rows_that_fit(4, act == SX_ACT_F32 ? 3 : 1, w->K, w->G, (int)(S < 16 ? S : 16));
    const int64_t units = S < S / 16 + E + 2 ? S : S / 16 + E + 2;
    return launch_qmm(fn, qmm::SWIGLU, 4, act, act, p, units, N / 2, 1, stream_of(stream));
}

int sx_linear_q4_experts_combine_grouped(const void *h, const sx_qview *w, int64_t E, const int32_t *ids,
                                         const float *coef, const void *ws, size_t ws_bytes, float *partial, int64_t M,
                                         int64_t A, void *y, int act, int math, sx_stream stream) {
    const char *fn = "sx_linear_q4_experts_combine_grouped";
    if (int rc = grouped_common(fn, h, w, E, M, A, ws, ws_bytes, y, act, math)) return rc;
    SX_CHECK(ids != nullptr && coef != nullptr && partial != nullptr, fn, " null pointer (ids=", (const void *)ids,
             ", coef=", (const void *)coef, ", partial=", (void *)partial, ")");
    const int64_t N = w->N / E, es = act_bytes(act), S = M * A;
    SX_CHECK(apart(y, M * N * es, h, S * w->K * es), fn, " y overlaps h");
    SX_CHECK(apart(y, M * N * es, partial, S * N * 4), fn, " y overlaps partial");
    SX_CHECK(apart(partial, S * N * 4, h, S * w->K * es), fn, " partial overlaps h");
    const Kernel kernel = grouped_kernel(w, M, A, E, act, device_cus());
    const int32_t *route = static_cast<const int32_t *>(ws);
    if (kernel != kQmm) {
        SX_HIP(kernel == kRegTiles ? rt::launch_grouped(qmm::COMBINE, h, w, partial, route, M, A, E, stream_of(stream))
                                   : gg::launch(qmm::COMBINE, h, w, partial, route, M, A, E, stream_of(stream)), fn);
        return combine_reduce(partial, ids, coef, M, A, E, N, y, act, stream_of(stream));
    }
    Params p{};
    p.x = h, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = partial, p.ws = static_cast<const int32_t *>(ws);
    p.M = M, p.A = A, p.E = E, p.N = N, p.K = w->K, p.G = (int)w->G;
    p.max_rows = rows_that_fit(4, act == SX_ACT_F32 ? 3 : 1, w->K, w->G, (int)(S < 16 ? S : 16));
    const int64_t units = S < S / 16 + E + 2 ? S : S / 16 + E + 2;
    if (int rc = launch_qmm(fn, qmm::COMBINE, 4, act, act, p, units, N, 1, stream_of(stream))) return rc;
    return combine_reduce(partial, ids, coef, M, A, E, N, y, act, stream_of(stream));
}

}  // extern "C"
