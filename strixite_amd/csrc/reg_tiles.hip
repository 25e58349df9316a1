// Dequantizing GEMM with a tile's activations resident in registers: grouped experts with a few slots each (q4 G = 128,
// BF16 x), from a handful of tokens to about 14 slots an expert.
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
//   sum_k x * (code * s + m) = s * D + (m - 128 s) * sum_span x with D from v_mfma_f32_16x16x32_bf16 on (128 + code)
// (qmm_impl.hpp); the second term of four spans is one MFMA of both sides' three BF16 terms (24 bits, as gg_kernel's).
// gate_up + SwiGLU at d = 4096, I = 1024, 512 experts top-10: M = 10 110 -> 88 us (qmm), 64 425 -> 291 (gg_kernel), 200
// 570 -> 413; d = 2560, I = 640 with the shared expert: M = 6 40.6 -> 21.6, 24 210 -> 71, 200 254 -> 180; down + combine
// (K = 640, qmm before): M = 200 136 -> 116, 2048 375 -> 338.
#include "reg_tiles.hpp"
#include "qmm_impl.hpp"

#include <algorithm>
#include <utility>

namespace sx::rt {
namespace {

using qmm::detail::bf16x8;
using qmm::detail::f32x4;

constexpr int kSpanBytes = 64;  // a weight row's span: 16 bytes a lane, 4 lanes
constexpr int kLag = 2;         // a slot's reload goes out two slots after its unpack

struct Params {
    const void *x;
    const uint8_t *q;
    const uint16_t *scale, *minv;
    void *y;
    const int32_t *ws;  // grouped: the route workspace (dense_M == 0)
    int64_t A, N, K;    // slots a token; rows an expert (SWIGLU: 2I); K
    int E, nspan, rounds;
    int64_t dense_M;    // > 0: a dense linear over dense_M token rows
};

// SPW BF16 words (a row's scales or mins of a wave's spans) at any 2-byte alignment
template <int SPW>
struct Win {
    uint32_t d[(SPW + 1) / 2];
    __device__ __forceinline__ void load(const uint16_t *p) {
        if constexpr (SPW >= 8) {
            uint4 v;
            __builtin_memcpy(&v, p, 16);
            d[0] = v.x, d[1] = v.y, d[2] = v.z, d[3] = v.w;
            rest<8>(p);
        } else if constexpr (SPW >= 4) {
            uint2 v;
            __builtin_memcpy(&v, p, 8);
            d[0] = v.x, d[1] = v.y;
            rest<4>(p);
        } else {
            rest<0>(p);
        }
    }
    template <int AT>
    __device__ __forceinline__ void rest(const uint16_t *p) {
        if constexpr (SPW - AT >= 2) {
            uint32_t v;
            __builtin_memcpy(&v, p + AT, 4);
            d[AT / 2] = v;
            rest<AT + 2>(p);
        } else if constexpr (SPW - AT == 1) {
            d[AT / 2] = p[AT];
        }
    }
    __device__ __forceinline__ float at(int s) const {
        return __uint_as_float((s & 1) ? (d[s >> 1] & 0xFFFF0000u) : (d[s >> 1] << 16));
    }
};

// A lane's value by its quarter g of the wave (by value: a conditional between array elements is one between addresses)
__device__ __forceinline__ float pick4(float a, float b, float c, float d, int g) {
    const float lo = (g & 1) ? b : a, hi = (g & 1) ? d : c;
    return (g & 2) ? hi : lo;
}
// FP32 -> BF16 as store_act rounds (nearest even), by the conversion instruction
__device__ __forceinline__ float bf16_rounded(float v) { return (float)(__bf16)v; }
__device__ __forceinline__ void put(float *y, int64_t i, float v) { y[i] = v; }
__device__ __forceinline__ void put(uint16_t *y, int64_t i, float v) { y[i] = __builtin_bit_cast(uint16_t, (__bf16)v); }
__device__ __forceinline__ uint32_t pick2(uint32_t a, uint32_t b, bool second) { return second ? b : a; }

// Q K slices of SPW spans, P output units a round: blocks of Q P waves.
constexpr int lanes_of(int q) { return q >= 5 ? 1 : 8 / q; }  // P
constexpr int blocks_a_cu(int ns, int q, int spw) { return ns > 1 || spw > 4 ? 1 : 2; }

template <int BITS, int MODE, int NS, int Q, int SPW, typename TY>
__global__ void __launch_bounds__(Q *lanes_of(Q) * 64, blocks_a_cu(NS, Q, SPW) == 2 ? 4 : 2)
    rt_kernel(Params p) {
    using F = qmm::detail::Fmt<BITS>;
    constexpr int NM = F::kMfmas;          // MFMAs a span
    constexpr int kSpan = F::kSpanCodes;
    constexpr int NC = (SPW + 3) / 4;      // span terms: MFMAs of four spans
    constexpr int NU = 4 * NS;             // output units of a tile pair: (set, v)
    constexpr int P = lanes_of(Q), kWaves = Q * P;
    constexpr int kUnitRows = MODE == qmm::SWIGLU ? 16 : 32;  // output rows of a unit (SWIGLU: features)
    __shared__ float red[2][kWaves][2][NU][64];  // [round & 1][wave][tile][unit][lane]
    __shared__ int s_out[2][16 * NS];            // [tile & 1]

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, g = lane >> 4;
    const int ip = wave / Q, kq = wave % Q;
    const int64_t K = p.K;
    const int nspan = p.nspan, E = p.E, rounds = p.rounds;
    const int64_t Nrows = MODE == qmm::SWIGLU ? p.N / 2 : p.N;
    const int64_t rowbytes = K * BITS / 8;
    const int units = (int)((Nrows + kUnitRows - 1) / kUnitRows);
    const int s0 = kq * SPW, w0 = min(s0, nspan - SPW);

    // ---- the block's share of the (tile, round) sequence, to within one round of every other block's ----
    const int32_t *ws = p.ws, *offsets = ws + 4, *slots = nullptr, *tile_bucket = nullptr, *tile_start = nullptr;
    unsigned n_tiles;
    if (p.dense_M > 0) {
        n_tiles = (unsigned)((p.dense_M + 16 * NS - 1) / (16 * NS));
    } else {
        const int S = ws[1];
        n_tiles = (unsigned)ws[0];
        slots = offsets + E + 2, tile_bucket = slots + S, tile_start = tile_bucket + S / 16 + E + 2;
    }
    const unsigned W = n_tiles * (unsigned)rounds, G = gridDim.x, blk = blockIdx.x, per = W / G, rem = W - per * G;
    const unsigned wa = blk * per + min(blk, rem), wn = per + (blk < rem ? 1u : 0u);
    if (wn == 0) return;
    int t = (int)(wa / (unsigned)rounds), r = (int)(wa - (unsigned)t * rounds);
    int left = (int)wn;  // rounds still to do, this tile's included

    // ---- a tile: its bucket, slots in lanes, rows of x ----
    int T = 0, bucket = 0, slot[NS];
    auto tile_at = [&](int t_) __attribute__((always_inline)) {
        if (p.dense_M > 0) {
            const int64_t t0 = (int64_t)t_ * (16 * NS);
            T = (int)min((int64_t)(16 * NS), p.dense_M - t0);
#pragma unroll
            for (int s = 0; s < NS; ++s) slot[s] = (int)t0 + min(16 * s + n16, T - 1);
        } else {
            bucket = __builtin_amdgcn_readfirstlane(tile_bucket[t_]);
            const int st = tile_start[t_];
            T = __builtin_amdgcn_readfirstlane(min(16 * NS, offsets[bucket + 1] - st));
#pragma unroll
            for (int s = 0; s < NS; ++s) slot[s] = slots[st + min(16 * s + n16, T - 1)];
        }
    };
    uint4 xr[NS][SPW][NM];
    auto load_x = [&]() __attribute__((always_inline)) {
        const uint16_t *x = static_cast<const uint16_t *>(p.x);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int64_t xrow = p.dense_M > 0 || MODE == qmm::COMBINE ? slot[s] : slot[s] / (int)p.A;
            const uint16_t *xp = x + xrow * K + (int64_t)w0 * kSpan + g * (kSpan / 4);
#pragma unroll
            for (int so = 0; so < SPW; ++so)
#pragma unroll
                for (int m = 0; m < NM; ++m) xr[s][so][m] = *reinterpret_cast<const uint4 *>(xp + so * kSpan + m * 8);
        }
    };

    // ---- this wave's weights: unit r P + ip of a round, spans w0 .. w0 + SPW - 1, through uniform bases and 32-bit
    // lane offsets (an expert's or the dense weight's code bytes < 2^32: checked by the host) ----
    const uint8_t *bq[2];
    const uint16_t *bs[2], *bm[2];
    auto base_at = [&](int bk) {
        const int64_t row_base = (int64_t)min(bk, E - 1) * p.N;  // invalid ids' tile: a valid expert, its results unused
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int64_t rb = row_base + (MODE == qmm::SWIGLU ? w * Nrows : 0);
            bq[w] = p.q + rb * rowbytes + (int64_t)w0 * kSpanBytes;
            bs[w] = p.scale + rb * nspan + w0;
            bm[w] = p.minv + rb * nspan + w0;
        }
    };
    constexpr int NO = MODE == qmm::SWIGLU ? 1 : 2;  // gate and up rows share their offsets
    uint32_t oq[NO], os[NO];
    auto place = [&](int r_) {
        const int f = min(r_ * P + ip, units - 1);
#pragma unroll
        for (int w = 0; w < NO; ++w) {
            const uint32_t n = min((uint32_t)(f * kUnitRows + 16 * w + n16), (uint32_t)Nrows - 1);
            oq[w] = n * (uint32_t)rowbytes + g * 16, os[w] = n * (uint32_t)nspan;
        }
    };
    // tiles in flight a wave: both of a round, or (one slot set, two blocks a compute unit: fewer registers) the next one
    constexpr int PF = NS == 1 ? 1 : 2;
    uint4 ring[PF][SPW];
    Win<SPW> sw[PF], mw[PF];
    auto issue_slot = [&](int w, int so) {
        ring[w % PF][so] = *reinterpret_cast<const uint4 *>(bq[w] + so * kSpanBytes + oq[w * (NO - 1)]);
    };
    auto issue_window = [&](int w) {
        sw[w % PF].load(bs[w] + os[w * (NO - 1)]), mw[w % PF].load(bm[w] + os[w * (NO - 1)]);
    };

    // ---- the A operands and the span-term operand of the loaded rows ----
    bf16x8 aop[NS][SPW][NM], xt[NS][NC];
    auto take_x = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float sums[4 * NC];
#pragma unroll
            for (int so = 0; so < 4 * NC; ++so) sums[so] = 0.f;
            const bool row_on = 16 * s + n16 < T;
#pragma unroll
            for (int so = 0; so < SPW; ++so) {
                const bool on = row_on && w0 + so >= s0;  // a span the slice before has too: zeros here
                float sum = 0.f;
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    const uint4 raw = on ? xr[s][so][m] : uint4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t d = qmm::detail::dword(raw, e);
                        sum += __uint_as_float(d << 16) + __uint_as_float(d & 0xFFFF0000u);
                    }
                    if constexpr (BITS == 4)
                        aop[s][so][m] = __builtin_bit_cast(
                            bf16x8, uint4{__builtin_amdgcn_perm(raw.z, raw.x, 0x05040100u), __builtin_amdgcn_perm(raw.z, raw.x, 0x07060302u),
                                          __builtin_amdgcn_perm(raw.w, raw.y, 0x05040100u), __builtin_amdgcn_perm(raw.w, raw.y, 0x07060302u)});
                    else
                        aop[s][so][m] = __builtin_bit_cast(bf16x8, raw);
                }
                sum += __shfl_xor(sum, 16);
                sum += __shfl_xor(sum, 32);
                sums[so] = sum;
                __builtin_amdgcn_sched_barrier(0);  // span by span: the loaded and the permuted rows do not all live at once
            }
            // lane (slot n16, g) holds span 4 c + g's sum as [x0 x0 x0 x1 x1 x2 0 0]
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const float v = pick4(sums[4 * c], sums[4 * c + 1], sums[4 * c + 2], sums[4 * c + 3], g);
                const __bf16 a = (__bf16)v;
                const float q1 = v - (float)a;
                const __bf16 b = (__bf16)q1;
                const __bf16 d = (__bf16)(q1 - (float)b);
                xt[s][c] = bf16x8{a, a, a, b, b, d, (__bf16)0.f, (__bf16)0.f};
            }
        }
    };

    // ---- the end of a round: the Q partial tiles summed in K order and stored ----
    // unit u (set, v) of a tile pair by the wave u % Q of its slices
    auto epilogue = [&](int r_, int buf, int tb) __attribute__((always_inline)) {
        const int f = r_ * P + ip;
        if (f >= units) return;
#pragma unroll
        for (int j = 0; j < (NU + Q - 1) / Q; ++j) {
            const int u = kq + j * Q;
            if (u >= NU) break;
            float a0 = 0.f, a1 = 0.f;
#pragma unroll
            for (int qq = 0; qq < Q; ++qq) {
                a0 += red[buf][ip * Q + qq][0][u][lane];
                a1 += red[buf][ip * Q + qq][1][u][lane];
            }
            const int row = 16 * (u >> 2) + 4 * g + (u & 3);
            if (row >= T) continue;
            if (bucket == E && p.dense_M == 0) a0 = a1 = qnan();  // invalid ids (reported by the grouping)
            const int64_t o = (int64_t)s_out[tb][row] * Nrows, n = (int64_t)f * kUnitRows + n16;
            TY *y = static_cast<TY *>(p.y);
            if constexpr (MODE == qmm::SWIGLU) {
                const float gv = bf16_rounded(a0), uv = bf16_rounded(a1);
                if (n < Nrows) put(y, o + n, bf16_rounded(silu(gv)) * uv);
            } else {
                if (n < Nrows) put(y, o + n, a0);
                if (n + 16 < Nrows) put(y, o + n + 16, a1);
            }
        }
    };

    tile_at(t);
    base_at(bucket);
    place(r);
#pragma unroll
    for (int w = 0; w < PF; ++w) {
        issue_window(w);
#pragma unroll
        for (int so = 0; so < SPW; ++so) issue_slot(w, so);
    }
    __builtin_amdgcn_sched_barrier(0);
    int buf = 0, tb = 0;
    for (;;) {
        load_x();
        if (wave == 0 && g == 0)  // read after the first round's barrier
#pragma unroll
            for (int s = 0; s < NS; ++s) s_out[tb][16 * s + n16] = slot[s];
        const int r1 = min(rounds, r + left);
        left -= r1 - r;
        // the tile after this one, for the loads that run ahead (none: this one's last round again, never used)
        const int next_bucket = left > 0 && p.dense_M == 0 ? __builtin_amdgcn_readfirstlane(tile_bucket[t + 1]) : bucket;
        take_x();
        for (; r < r1; ++r, buf ^= 1) {
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const Win<SPW> cs = sw[w % PF], cm_ = mw[w % PF];
                // the tile whose loads this one issues: the round's other tile (PF = 1, the first) or the next round's
                const int nw = PF == 1 ? 1 - w : w;
                if (w == (PF == 1 ? 1 : 0)) {
                    const bool last = r + 1 == r1;
                    if (last) base_at(next_bucket);
                    place(last ? (left > 0 ? 0 : r) : r + 1);
                }
                issue_window(nw);
                __builtin_amdgcn_sched_barrier(0);
                f32x4 acc[NS];
                // the span terms first: sum over the spans of (min - off scale)[row] * sum x[slot], both sides split
                // into three BF16 terms, the six products down to 2^-16 of the whole, as one MFMA of four spans
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    float sv, mv;
                    {
                        constexpr int top = (SPW + 1) / 2 - 1;
                        const int i0 = min(2 * c, top), i1 = min(2 * c + 1, top);
                        const uint32_t sd = pick2(cs.d[i0], cs.d[i1], g & 2), md = pick2(cm_.d[i0], cm_.d[i1], g & 2);
                        const int sh = (g & 1) ? 0 : 16;
                        sv = __uint_as_float((sd << sh) & 0xFFFF0000u), mv = __uint_as_float((md << sh) & 0xFFFF0000u);
                    }
                    const float cmv = fmaf(-F::kOff, sv, mv);
                    const __bf16 a = (__bf16)cmv;
                    const float q1 = cmv - (float)a;
                    const __bf16 b = (__bf16)q1;
                    const __bf16 d = (__bf16)(q1 - (float)b);
                    const bf16x8 bt = bf16x8{a, b, d, a, b, a, (__bf16)0.f, (__bf16)0.f};
#pragma unroll
                    for (int s = 0; s < NS; ++s)
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xt[s][c], bt, c == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[s], 0, 0, 0);
                }
                // a span's codes are unpacked while the MFMAs of the one before run; a slot's reload goes out kLag
                // spans after its unpack, pinned there (left to the scheduler the reloads sink below the whole round)
                // (NS = 1: four waves a SIMD cover each other's MFMAs; one operand unpacked at a time keeps two blocks
                // a compute unit within 128 registers)
                constexpr int NB = NS == 1 ? 1 : 2;
                bf16x8 bop[NB][NM];
                auto unpack = [&](int so) __attribute__((always_inline)) {
#pragma unroll
                    for (int m = 0; m < NM; ++m) bop[so % NB][m] = qmm::detail::codes_b<BITS>(ring[w % PF][so], m);
                };
                if (NB == 2) unpack(0);
#pragma unroll
                for (int so = 0; so < SPW; ++so) {
                    if (so >= kLag) issue_slot(nw, so - kLag);
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 D[NS];
#pragma unroll
                    for (int m = 0; m < NM; ++m) {
                        if (NB == 1) bop[0][m] = qmm::detail::codes_b<BITS>(ring[w % PF][so], m);
#pragma unroll
                        for (int s = 0; s < NS; ++s)
                            D[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aop[s][so][m], bop[so % NB][m], m == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : D[s], 0, 0, 0);
                        if (NB == 1) __builtin_amdgcn_sched_barrier(0);
                    }
                    if (NB == 2 && so + 1 < SPW) unpack(so + 1);
                    const float s_ = cs.at(so);
#pragma unroll
                    for (int s = 0; s < NS; ++s)
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[s][v] = fmaf(s_, D[s][v], acc[s][v]);
                }
#pragma unroll
                for (int so = SPW - kLag; so < SPW; ++so) issue_slot(nw, so);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < NS; ++s)
#pragma unroll
                    for (int v = 0; v < 4; ++v) red[buf][wave][w][4 * s + v][lane] = acc[s][v];
            }
            // every wave's partial tiles of this round are in LDS (the loads in flight stay in flight); the next write
            // to this half of red comes after the next round's barrier, when these reads are done
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            epilogue(r, buf, tb);
        }
        if (left <= 0) break;
        // the next tile: its first round's weights are on their way already
        ++t, r = 0, tb ^= 1;
        tile_at(t);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the loads past the last round land before the wave exits
}

// K slices and spans a wave for nspan spans. The slices cover whole 128-byte lines (pairs of spans) of an even row:
// spans two slices both read, and lines split between them, cost as much as any other request.
struct Split {
    int q, spw;
};
constexpr Split kSplits4[] = {{1, 2}, {1, 3}, {1, 4}, {1, 5}, {2, 4}, {3, 4}, {4, 4}, {5, 4}, {6, 4}, {7, 4}, {8, 4}};

template <int N>
int split_of(int nspan, const Split (&s)[N]) {  // the fewest spare spans
    int best = -1, cost = 1 << 30;
    for (int i = 0; i < N; ++i) {
        const int spare = s[i].spw * s[i].q - nspan;
        if (s[i].spw <= nspan && spare >= 0 && spare < cost) cost = spare, best = i;
    }
    return best;
}

template <int MODE, int NS, typename TY>
hipError_t go4(const Params &p, int split, int64_t most, hipStream_t stream) {
    auto one = [&](auto i_tag) {
        constexpr Split S = kSplits4[decltype(i_tag)::value];
        if (split != decltype(i_tag)::value) return;
        const int64_t blocks = (int64_t)device_cus() * blocks_a_cu(NS, S.q, S.spw);
        hipLaunchKernelGGL((rt_kernel<4, MODE, NS, S.q, S.spw, TY>), dim3((unsigned)std::min(blocks, most)),
                           dim3(S.q * lanes_of(S.q) * 64), 0, stream, p);
    };
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (one(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, (int)(sizeof(kSplits4) / sizeof(kSplits4[0]))>{});
    return hipGetLastError();
}

}  // namespace

bool eligible_grouped(int bits, int64_t G, int64_t N, int64_t K, int64_t M, int64_t A, int64_t E, int act) {
    if (!(bits == 4 && G == 128 && K % 128 == 0 && K >= 256 && K <= 4096 && act == SX_ACT_BF16)) return false;
    // 32-bit offsets into an expert's rows and a 32-bit (tile, round) sequence
    return N * (K / 2) < (int64_t(1) << 32) && (M * A / 16 + E + 2) * (N / 16 + 1) < (int64_t(1) << 31);
}

hipError_t launch_grouped(int mode, const void *x, const sx_qview *w, void *y, const int32_t *ws, int64_t M, int64_t A,
                          int64_t E, hipStream_t stream) {
    Params p{};
    p.x = x, p.q = w->q, p.scale = w->scale, p.minv = w->minv, p.y = y, p.ws = ws;
    p.A = A, p.N = w->N / E, p.K = w->K, p.E = (int)E, p.nspan = (int)(w->K / 128);
    const int split = split_of(p.nspan, kSplits4);
    if (split < 0) return hipErrorInvalidValue;
    const int P = lanes_of(kSplits4[split].q);
    const int64_t out_rows = mode == qmm::SWIGLU ? p.N / 2 : p.N, unit = mode == qmm::SWIGLU ? 16 : 32;
    const int64_t units = (out_rows + unit - 1) / unit;
    p.rounds = (int)((units + P - 1) / P);
    const int64_t S = M * A, most = std::min<int64_t>(S, S / 16 + E + 2) * p.rounds;
    if (mode == qmm::COMBINE) return go4<qmm::COMBINE, 1, float>(p, split, most, stream);
    if (mode == qmm::SWIGLU) return go4<qmm::SWIGLU, 1, uint16_t>(p, split, most, stream);
    return go4<qmm::GATHER, 1, uint16_t>(p, split, most, stream);
}

}  // namespace sx::rt
