// The register-tile kernel (see reg_tiles.hip for the scheme), instantiated for the grouped experts in reg_tiles.hip and
// for dense linears in reg_dense_q4.hip and reg_dense_q8.hip, so that the instantiations compile in parallel.
#pragma once
#include "reg_tiles.hpp"
#include "qmm_impl.hpp"

#include <algorithm>
#include <utility>

namespace sx::rt {
namespace detail {

using qmm::detail::bf16x8;
using qmm::detail::f32x4;

constexpr int kSpanBytes = 64;  // a weight row's span: 16 bytes a lane, 4 lanes
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

// FP32 -> BF16 as store_act rounds (nearest even), by the conversion instruction
__device__ __forceinline__ float bf16_rounded(float v) { return (float)(__bf16)v; }
__device__ __forceinline__ void put(float *y, int64_t i, float v) { y[i] = v; }
__device__ __forceinline__ void put(uint16_t *y, int64_t i, float v) { y[i] = __builtin_bit_cast(uint16_t, (__bf16)v); }

// Q K slices of SPW spans, P output units a round: blocks of Q P waves. Eight waves where P can fill them up; past four
// slices one unit, but two for q8's five (K = 2112 .. 2560, BF16 rows): five waves are two on one SIMD and one on each of
// the others, ten are three or two on each. One unit / two, us: 248320 x 2560 M = 24 218 / 203, 248320 x 2112 M = 64 411 /
// 332, 14000 x 2112 M = 200 80 / 68; where a block has a single round two cost more (4096 x 2560 M = 16 9.4 / 14.5, M = 1
// 8.1 / 10.8; qmm 19.7 and 16.0).
constexpr int lanes_of(int bits, int q, bool f32) { return q < 5 ? 8 / q : bits == 8 && q == 5 && !f32 ? 2 : 1; }  // P
// Blocks a compute unit: two of at most 128 registers where the operands leave room (a wave's 512 codes of 16 rows are
// 64 registers; q8 has twice the code and scale registers in flight, FP32 rows twice the loads), else one.
constexpr int blocks_a_cu(int bits, int spw, bool f32) { return bits == 4 && spw <= 4 && !f32 ? 2 : 1; }
constexpr int waves_a_simd(int bits, int q, int spw, bool f32) {
    return blocks_a_cu(bits, spw, f32) == 2 ? 4 : (q * lanes_of(bits, q, f32) + 3) / 4;
}
// A slot's reload goes out kLag slots after its unpack (fewer bytes in flight a compute unit stream faster).
constexpr int lag_of(int spw) { return spw >= 8 ? 6 : 2; }

// FP32 rows (TX float): the 16 operand rows of a tile are 5 tokens x 3 exact BF16 planes (row 3 t + p: hi, mid, lo), so
// the K loop is the BF16 one, and the planes' results are added with the slices' at the end.
template <int BITS, int MODE, int Q, int SPW, typename TX, typename TY>
__global__ void __launch_bounds__(Q *lanes_of(BITS, Q, sizeof(TX) == 4) * 64, waves_a_simd(BITS, Q, SPW, sizeof(TX) == 4))
    rt_kernel(Params p) {
    constexpr bool FX = sizeof(TX) == 4;
    constexpr int kTok = FX ? 5 : 16;      // tokens (slots) a tile
    constexpr int kLag = lag_of(SPW);
    using F = qmm::detail::Fmt<BITS>;
    constexpr int NM = F::kMfmas;          // MFMAs a span
    constexpr int kSpan = F::kSpanCodes;
    constexpr int P = lanes_of(BITS, Q, FX), kWaves = Q * P;
    constexpr int kUnitRows = MODE == qmm::SWIGLU ? 16 : 32;  // output rows of a unit (SWIGLU: features)
    __shared__ float red[2][kWaves][2][4][64];  // [round & 1][wave][tile][v][lane]
    __shared__ __attribute__((aligned(16))) float xsum[kWaves][SPW][16];  // the wave's span sums of the operand rows
    __shared__ int s_out[2][16];                // [tile & 1]

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
        n_tiles = (unsigned)((p.dense_M + kTok - 1) / kTok);
    } else {
        const int S = ws[1];
        n_tiles = (unsigned)ws[0];
        slots = offsets + E + 2, tile_bucket = slots + S, tile_start = tile_bucket + S / 16 + E + 2;
    }
    // (few tiles: a whole number of blocks each, at an eighth of them idle at most, so that no block takes up a second
    // tile's activations)
    const unsigned G = gridDim.x, blk = blockIdx.x, R = (unsigned)rounds, bpt = G / max(n_tiles, 1u);
    unsigned wa, wn;
    if (bpt >= 8) {
        const unsigned bt = blk / bpt, i = blk - bt * bpt;
        if (bt >= n_tiles) return;
        const unsigned f0 = i * R / bpt;  // R < 2^23 where a tile has this many blocks (checked by the host)
        wa = bt * R + f0, wn = (i + 1) * R / bpt - f0;
    } else {
        const unsigned W = n_tiles * R, per = W / G, rem = W - per * G;
        wa = blk * per + min(blk, rem), wn = per + (blk < rem ? 1u : 0u);
    }
    if (wn == 0) return;
    int t = (int)(wa / (unsigned)rounds), r = (int)(wa - (unsigned)t * rounds);
    int left = (int)wn;  // rounds still to do, this tile's included

    // ---- a tile: its bucket, slots in lanes, rows of x ----
    int T = 0, bucket = 0, slot = 0;
    const int tok = FX ? n16 / 3 : n16;  // the operand row's token
    auto tile_at = [&](int t_) __attribute__((always_inline)) {
        if (p.dense_M > 0) {
            const int64_t t0 = (int64_t)t_ * kTok;
            T = (int)min((int64_t)kTok, p.dense_M - t0);
            slot = (int)t0 + min(tok, T - 1);
        } else {
            bucket = __builtin_amdgcn_readfirstlane(tile_bucket[t_]);
            const int st = tile_start[t_];
            T = __builtin_amdgcn_readfirstlane(min(16, offsets[bucket + 1] - st));
            slot = slots[st + min(n16, T - 1)];
        }
    };
    qmm::detail::Raw8<TX> xr[SPW][NM];
    auto load_x = [&]() __attribute__((always_inline)) {
        const int64_t xrow = p.dense_M > 0 || MODE == qmm::COMBINE ? slot : slot / (int)p.A;
        const TX *xp = static_cast<const TX *>(p.x) + xrow * K + (int64_t)w0 * kSpan + g * (kSpan / 4);
#pragma unroll
        for (int so = 0; so < SPW; ++so)
#pragma unroll
            for (int m = 0; m < NM; ++m) xr[so][m] = qmm::detail::load_raw8<TX>(xp + so * kSpan + m * 8);
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
    uint4 ring[SPW];  // one tile in flight a wave
    Win<SPW> sw, mw;
    auto issue_slot = [&](int w, int so) {
        ring[so] = *reinterpret_cast<const uint4 *>(bq[w] + so * kSpanBytes + oq[w * (NO - 1)]);
    };
    auto issue_window = [&](int w) { sw.load(bs[w] + os[w * (NO - 1)]), mw.load(bm[w] + os[w * (NO - 1)]); };

    // ---- the loaded rows as A operands, and their span sums ----
    bf16x8 aop[SPW][NM];
    auto take_x = [&]() __attribute__((always_inline)) {
        const bool row_on = tok < T && (!FX || n16 < 15);
        const int plane = n16 % 3;
#pragma unroll
        for (int so = 0; so < SPW; ++so) {
            const bool on = row_on && w0 + so >= s0;  // a span the slice before has too: zeros here
            float sum = 0.f;
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                if constexpr (FX) {
                    float v[8];
                    qmm::detail::unpack8(xr[so][m], v);
                    bf16x8 o;
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float x = on ? v[e] : 0.f;
                        const __bf16 hi = (__bf16)x;
                        const float r1 = x - (float)hi;
                        const __bf16 mid = (__bf16)r1;
                        const float r2 = r1 - (float)mid;
                        const __bf16 mine = (__bf16)(plane == 0 ? x : plane == 1 ? r1 : r2);
                        o[qmm::detail::lds_pos<BITS>(e)] = mine;
                        sum += (float)mine;
                    }
                    aop[so][m] = o;
                } else {
                    const uint4 raw = on ? xr[so][m] : uint4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t d = qmm::detail::dword(raw, e);
                        sum += __uint_as_float(d << 16) + __uint_as_float(d & 0xFFFF0000u);
                    }
                    if constexpr (BITS == 4)
                        aop[so][m] = __builtin_bit_cast(
                            bf16x8, uint4{__builtin_amdgcn_perm(raw.z, raw.x, 0x05040100u), __builtin_amdgcn_perm(raw.z, raw.x, 0x07060302u),
                                          __builtin_amdgcn_perm(raw.w, raw.y, 0x05040100u), __builtin_amdgcn_perm(raw.w, raw.y, 0x07060302u)});
                    else
                        aop[so][m] = __builtin_bit_cast(bf16x8, raw);
                }
            }
            sum += __shfl_xor(sum, 16);
            sum += __shfl_xor(sum, 32);
            if (g == 0) xsum[wave][so][n16] = sum;  // read by this wave alone (its LDS operations keep their order)
            __builtin_amdgcn_sched_barrier(0);  // span by span: the loaded and the permuted rows do not all live at once
        }
    };

    // ---- the end of a round: the Q partial tiles summed in K order and stored ----
    // D row 4 g + v of a tile pair by the wave v % Q of its slices, the four quarters of a wave at once (FP32 rows: token
    // 4 j + g by the wave j % Q, the token's three planes added too)
    constexpr int NJ = FX ? 2 : 4;
    auto epilogue = [&](int r_, int buf, int tb) __attribute__((always_inline)) {
        const int f = r_ * P + ip;
        if (f >= units) return;
#pragma unroll
        for (int i = 0; i < (NJ + Q - 1) / Q; ++i) {
            const int j = kq + i * Q;
            if (j >= NJ) break;
            const int row = FX ? 4 * j + g : 4 * g + j;  // token of the tile
            float a0 = 0.f, a1 = 0.f;
#pragma unroll
            for (int qq = 0; qq < Q; ++qq) {
                if constexpr (FX) {
#pragma unroll
                    for (int pl = 2; pl >= 0; --pl) {
                        const int rr = min(3 * row + pl, 15), at = (rr >> 2) * 16 + n16;
                        a0 += red[buf][ip * Q + qq][0][rr & 3][at];
                        a1 += red[buf][ip * Q + qq][1][rr & 3][at];
                    }
                } else {
                    a0 += red[buf][ip * Q + qq][0][j][lane];
                    a1 += red[buf][ip * Q + qq][1][j][lane];
                }
            }
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
    issue_window(0);
#pragma unroll
    for (int so = 0; so < SPW; ++so) issue_slot(0, so);
    __builtin_amdgcn_sched_barrier(0);
    int buf = 0, tb = 0;
    for (;;) {
        load_x();
        // the tile's output rows, read after the first round's barrier
        if (wave == 0 && g == 0) {
            if constexpr (FX) {
                if (n16 < T) s_out[tb][n16] = t * kTok + n16;
            } else {
                s_out[tb][n16] = slot;
            }
        }
        const int r1 = min(rounds, r + left);
        left -= r1 - r;
        // the tile after this one, for the loads that run ahead (none: this one's last round again, never used)
        const int next_bucket = left > 0 && p.dense_M == 0 ? __builtin_amdgcn_readfirstlane(tile_bucket[t + 1]) : bucket;
        take_x();
        for (; r < r1; ++r, buf ^= 1) {
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const Win<SPW> cs = sw, cm_ = mw;
                // the tile whose loads this one issues: the round's second or the next round's first
                const int nw = 1 - w;
                if (w == 1) {
                    const bool last = r + 1 == r1;
                    if (last) base_at(next_bucket);
                    place(last ? (left > 0 ? 0 : r) : r + 1);
                }
                issue_window(nw);
                __builtin_amdgcn_sched_barrier(0);
                f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
                // a slot's reload is pinned kLag spans after its unpack (left to the scheduler the reloads sink below the
                // whole round), and one operand is unpacked at a time (the other waves of the SIMD cover its MFMA)
#pragma unroll
                for (int so = 0; so < SPW; ++so) {
                    if (so >= kLag) issue_slot(nw, so - kLag);
                    __builtin_amdgcn_sched_barrier(0);
                    f32x4 D = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int m = 0; m < NM; ++m) {
                        const bf16x8 bop = qmm::detail::codes_b<BITS>(ring[so], m);
                        D = __builtin_amdgcn_mfma_f32_16x16x32_bf16(aop[so][m], bop, D, 0, 0, 0);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    const float4 xs4 = *reinterpret_cast<const float4 *>(&xsum[wave][so][4 * g]);
                    const float xv[4] = {xs4.x, xs4.y, xs4.z, xs4.w};
                    const float s_ = cs.at(so), cm = fmaf(-F::kOff, s_, cm_.at(so));
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[v] = fmaf(s_, D[v], fmaf(cm, xv[v], acc[v]));
                }
#pragma unroll
                for (int so = SPW > kLag ? SPW - kLag : 0; so < SPW; ++so) issue_slot(nw, so);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int v = 0; v < 4; ++v) red[buf][wave][w][v][lane] = acc[v];
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
constexpr Split kSplits8[] = {{1, 4}, {1, 8}, {2, 5}, {2, 8}, {3, 8}, {4, 8}, {5, 8}, {6, 8}, {7, 8}, {8, 8}};
template <int BITS>
constexpr auto &splits() {
    if constexpr (BITS == 4) return kSplits4;
    else return kSplits8;
}

template <int N>
int split_of(int nspan, const Split (&s)[N]) {  // the fewest spare spans
    int best = -1, cost = 1 << 30;
    for (int i = 0; i < N; ++i) {
        const int spare = s[i].spw * s[i].q - nspan;
        if (s[i].spw <= nspan && spare >= 0 && spare < cost) cost = spare, best = i;
    }
    return best;
}

// The launch of a split: the resident blocks, at most one a unit of work (most).
template <int BITS, int MODE, typename TX, typename TY>
hipError_t go(const Params &p, int split, int64_t most, hipStream_t stream) {
    constexpr auto &table = splits<BITS>();
    auto one = [&](auto i_tag) {
        constexpr Split S = table[decltype(i_tag)::value];
        if (split != decltype(i_tag)::value) return;
        const int cus = device_cus();
        int64_t blocks = (int64_t)cus * blocks_a_cu(BITS, S.spw, sizeof(TX) == 4);
        // A dense weight's tiles share their codes in the caches, and a block's first cost is its activations: one block
        // a compute unit (4096 x 4096, M = 64: 11.5 us against 16.2 with two), except small blocks with three or more
        // units a compute unit (7680 x 2560, five waves, M = 400: 40.8 us against 46.5 with one).
        if (p.dense_M > 0 && (S.q * lanes_of(BITS, S.q, sizeof(TX) == 4) >= 8 || most < 3 * cus)) blocks = cus;
        hipLaunchKernelGGL((rt_kernel<BITS, MODE, S.q, S.spw, TX, TY>), dim3((unsigned)std::min(blocks, most)),
                           dim3(S.q * lanes_of(BITS, S.q, sizeof(TX) == 4) * 64), 0, stream, p);
    };
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (one(std::integral_constant<int, I>{}), ...);
    }(std::make_integer_sequence<int, (int)(sizeof(table) / sizeof(table[0]))>{});
    return hipGetLastError();
}

// A dense linear (reg_dense_q4.hip, reg_dense_q8.hip): p without rounds, act / out_act as linear's.
template <int BITS>
hipError_t dense(Params p, int act, int out_act, hipStream_t stream) {
    const int split = split_of(p.nspan, splits<BITS>());
    if (split < 0) return hipErrorInvalidValue;
    const int P = lanes_of(BITS, splits<BITS>()[split].q, act == SX_ACT_F32), tok = act == SX_ACT_F32 ? 5 : 16;
    p.rounds = (int)(((p.N + 31) / 32 + P - 1) / P);
    const int64_t most = (p.dense_M + tok - 1) / tok * p.rounds;
    if (act == SX_ACT_F32) return go<BITS, qmm::GATHER, float, float>(p, split, most, stream);
    if (out_act == SX_ACT_F32) return go<BITS, qmm::GATHER, uint16_t, float>(p, split, most, stream);
    return go<BITS, qmm::GATHER, uint16_t, uint16_t>(p, split, most, stream);
}

hipError_t dense_q4(const Params &p, int act, int out_act, hipStream_t stream);
hipError_t dense_q8(const Params &p, int act, int out_act, hipStream_t stream);

}  // namespace detail
}  // namespace sx::rt
