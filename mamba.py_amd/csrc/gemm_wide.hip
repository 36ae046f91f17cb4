// y (T x M) = x (T x K) . W^T in bfloat16 for many rows, W as (M x K) or as (K x M), by tiles of 256 x 256, for gfx950.
//
// A product of a layer has a short K (768: 24 slices of 32), so what a tile does before its first product and after its last is a third
// of it, and its tiles are a few rounds of the chip and a part of one.  Here a workgroup (one a CU, four waves, 128 x 128 a wave with 256
// accumulators) walks tile after tile without a break in its loads: the last slices of a tile request the first ones of the next, the results
// leave by stores that the next products do not wait for, and the part of a round that is left is cut into tiles of half the rows where that is
// shorter.
//
// Operands go from memory to LDS directly, 16 bytes a lane, in chunks of 64 k of x or of W (32 KB), in turn; five chunks are in LDS.  A stage of
// 64 k is multiplied in two steps: in the first its second half's operands are read between the products and the next chunk of x is requested,
// in the second the next stage's, and a chunk of W: 2 to 3 steps before the one barrier of a stage at which it has to be there.  (In slices of
// 32 k, whose loads are 64 bytes of 16 rows and whose barriers twice as many, 8192 x 8192 x 8192 took 820 us.)
// Rows of 128 bytes (k fast) are rotated by parts of 16 bytes so that eight lanes in eight rows read from different banks; W as (K x M) is
// read by ds_read_b64_tr_b16 from rows of 512 bytes, rotated by 32.  The rows of W are dealt to the operands so that a lane's results of two
// operands are eight neighbours in y, and four lanes have 64 bytes.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kTileSide = 256, kHalf = 128, kStageK = 64, kRing = 5, kCUs = 256;

struct GemmParams {
    const void *x, *w;
    void* y;
    int64_t x_pitch, w_pitch, y_pitch;
    int T, M, K;
    int tiles_t, tiles_m;
    int full, half;  // tiles of 256 x 256, the first ones; the others, in halves of 128 rows of x
};

// In place, see wgrad_wide.hip; what reads a sum has 19 wait states before it.
__device__ __forceinline__ void multiply(f32x4& c, const u32x4& a, const u32x4& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void multiply_first(f32x4& c, const u32x4& a, const u32x4& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(c) : "v"(a), "v"(b));
}

// TAIL: K is not whole stages, and two of them at least.
template <bool KXM, bool TAIL>
__global__ void __launch_bounds__(256, 1) gemm_wide_kernel(const GemmParams p) {
    constexpr int kChunk = kTileSide * kStageK * 2;
    constexpr uint32_t kNowhere = 0x80000000u;
    __shared__ alignas(16) char lds[kRing * kChunk];
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int wt = wave & 1, wm = wave >> 1, fr = lane & 15, fq = lane >> 4;
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;

    // The workgroup's tiles: one of every round.  An XCD takes neighbouring ones: strips of four columns of tiles, row by row.
    struct Tile {
        int t0, m0, half;  // half: 128 rows; t0 < 0: none
    };
    auto place = [&](int tile, Tile& g) {
        const int strip = tile / (4 * p.tiles_t), wide = min(4, p.tiles_m - strip * 4), in = tile - strip * 4 * p.tiles_t;
        const int tt = in / wide;
        g.t0 = tt * kTileSide;
        g.m0 = (strip * 4 + in - tt * wide) * kTileSide;
    };
    const int rounds = (p.full + kCUs - 1) / kCUs;
    int round = 0;
    auto next_tile = [&] {
        for (;; ++round) {
            Tile g{-1, 0, 0};
            const bool whole = round < rounds;
            const int begin = (whole ? round : round - rounds) * kCUs, some = min(kCUs, (whole ? p.full : p.half) - begin), per = (some + 7) / 8, at = xcd * per + slot;
            if (some <= 0) return g;
            if (slot >= per || at >= some) continue;
            place(whole ? begin + at : p.full + (begin + at) / 2, g);
            if (!whole) {
                g.t0 += (begin + at) % 2 * kHalf;
                g.half = 1;
                if (g.t0 >= p.T) continue;
            }
            ++round;
            return g;
        }
    };

    // by what the parts of a row of W are rotated: the eight rows that lanes read together differ in it
    auto turn = [](int row) { return (row & 3) | (row >> 3 & 1) << 2; };
    // loads of a chunk: wave w rows 64 * w + 8 * i + lane / 8 (W as (K x M): 16 * w + 2 * i + lane / 32), i = 0 .. 7
    uint32_t off_x[8], off_w[8];
    const int kx = ((lane & 7) ^ (lane >> 3)) * 8;
    int kw[KXM ? 8 : 2], cw[KXM ? 8 : 1];  // first k of the lane's part, and column
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = 64 * wave + 8 * i + (lane >> 3);
        off_x[i] = ((uint32_t)row * (uint32_t)p.x_pitch + (uint32_t)kx) * 2u;
        if constexpr (KXM) {
            kw[i] = 16 * wave + 2 * i + (lane >> 5);
            cw[i] = ((lane & 31) ^ (2 * turn(kw[i]))) * 8;
            off_w[i] = ((uint32_t)kw[i] * (uint32_t)p.w_pitch + (uint32_t)cw[i]) * 2u;
        } else {
            kw[i & 1] = ((lane & 7) ^ turn(row)) * 8;
            off_w[i] = ((uint32_t)row * (uint32_t)p.w_pitch + (uint32_t)kw[i & 1]) * 2u;
        }
    }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds) + (uint32_t)wave * 8192u;
    u32x4 window_x, window_w;
    int next_k = 0, cols = 0;  // of the next stage to request; columns of W as (K x M) from the tile's first on
    auto aim = [&](const Tile& g) {
        next_k = 0;
        const bool some = g.t0 >= 0;
        const int64_t t0 = some ? g.t0 : 0, rows = some ? min((int64_t)(g.half ? kHalf : kTileSide), p.T - t0) : 0;
        window_x = lds_window(static_cast<const char*>(p.x) + t0 * p.x_pitch * 2, some ? (uint32_t)(((rows - 1) * p.x_pitch + p.K) * 2) : 0u);
        if constexpr (KXM) {
            cols = p.M - g.m0;
            window_w = lds_window(static_cast<const char*>(p.w) + (int64_t)g.m0 * 2, some ? (uint32_t)(((p.K - 1) * p.w_pitch + p.M - g.m0) * 2) : 0u);
        } else {
            const int64_t of = min(kTileSide, p.M - g.m0);
            window_w = lds_window(static_cast<const char*>(p.w) + g.m0 * p.w_pitch * 2, some ? (uint32_t)(((of - 1) * p.w_pitch + p.K) * 2) : 0u);
        }
    };
    // Load i of the next chunk of x or W, in two parts with a product between them: where to (in place `to`), and the load (k beyond the last: zeros).
    // (A lone wave issues an instruction every five clocks, and a product takes sixteen: with all of it behind one, loads cost a tenth of the time.)
    // (m0 is where a load finds its place: the value is handed from one to the other in it, so that the compiler leaves it there)
    uint32_t spot;
    auto aim_load = [&](int i, uint32_t to) { asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(spot) : "s"(to), "n"(i * 1024) : "scc"); };
    auto load = [&](const u32x4& window, uint32_t off, uint32_t k) {
        asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(off), "s"(window), "s"(k), "{m0}"(spot) : "memory");
    };
    auto load_x = [&](int i) { load(window_x, TAIL && next_k + kx >= p.K ? kNowhere : off_x[i], (uint32_t)next_k * 2u); };
    auto load_w = [&](int i) {
        const bool none = (TAIL && next_k + kw[KXM ? i : i & 1] >= p.K) || (KXM && cw[KXM ? i : 0] >= cols);
        load(window_w, none ? kNowhere : off_w[i], KXM ? (uint32_t)next_k * (uint32_t)p.w_pitch * 2u : (uint32_t)next_k * 2u);
    };

    // reads: 16 x 32 of x as rows 16 * i + fr, of W as rows 32 * (j / 2) + 8 * (fr / 4) + 4 * (j % 2) + fr % 4, eight k from 8 * fq of either half of a
    // stage
    uint32_t at_x[2], at_w[KXM ? 4 : 2];
    auto set_x = [&](int half) {
#pragma unroll
        for (int h = 0; h < 2; ++h) at_x[h] = (uint32_t)((wt * (half ? kHalf / 2 : kHalf) + fr) * 128 + ((4 * h + fq) ^ (fr & 7)) * 16);
    };
    if constexpr (KXM) {
        const int row = 8 * fq + (fr >> 2), c = fr & 3;
#pragma unroll
        for (int j = 0; j < 4; ++j) at_w[j] = (uint32_t)(row * 512 + wm * 256 + (((2 * j + (c >> 1)) ^ turn(row)) * 32) + (c & 1) * 16);
    } else {
#pragma unroll
        for (int h = 0; h < 2; ++h) at_w[h] = (uint32_t)((wm * 128 + 8 * (fr >> 2) + (fr & 3)) * 128 + ((4 * h + fq) ^ (fr & 7)) * 16);
    }
    const auto base = (__attribute__((address_space(3))) char*)lds;
    u32x4 ox[2][8], ow[2][8];  // of the first and the second half of a stage
    auto read_x = [&](uint32_t from, int h, int i) { ox[h][i] = *(__attribute__((address_space(3))) u32x4*)(base + at_x[h] + from + i * 2048); };
    auto read_w = [&](uint32_t from, int h, int j) {
        if constexpr (KXM) {
            typedef __attribute__((address_space(3))) i16x4* P;
            struct { i16x4 v[2]; } r;
#pragma unroll
            for (int q = 0; q < 2; ++q) r.v[q] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((P)(base + at_w[j >> 1] + from + (j & 1) * 8 + (32 * h + 4 * q) * 512));
            ow[h][j] = __builtin_bit_cast(u32x4, r);
        } else {
            ow[h][j] = *(__attribute__((address_space(3))) u32x4*)(base + at_w[h] + from + (j >> 1) * 4096 + (j & 1) * 512);
        }
    };

    f32x4 acc[8][8];  // [of W][of x]
    int stores = 0;   // of the tile before, issued behind the loads of two stages
    int place_x = 0;  // of the stage's chunk of x; that of W is the next place
    auto ahead = [](int place, int n) { return place + n >= kRing ? place + n - kRing : place + n; };
    // The first half of a stage is multiplied, its second half read, and the chunk of x requested that is two stages on; then the second half, the first
    // half of the next stage, and a chunk of W.
    auto step = [&](auto first, auto narrow, auto second) {
        constexpr bool kFirst = decltype(first)::value, kNarrow = decltype(narrow)::value;
        constexpr int h = decltype(second)::value, kX = kNarrow ? 4 : 8;
        if constexpr (h == 1) {
            // the next stage is there (behind it: a chunk, and the stores of the tile before), and all waves have read this one
            if (kFirst && stores == 32) asm volatile("s_waitcnt vmcnt(40) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else if (kFirst && stores == 16) asm volatile("s_waitcnt vmcnt(24) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        }
        const uint32_t to = lds0 + (uint32_t)(h == 0 ? ahead(place_x, 4) : place_x) * kChunk;  // (the first chunk of this stage's, read)
        const int from = h == 0 ? place_x : ahead(place_x, 2);
        const uint32_t from_x = (uint32_t)from * kChunk, from_w = (uint32_t)ahead(from, 1) * kChunk;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
#pragma unroll
            for (int i = 0; i < kX; ++i) {
                if (kFirst && h == 0) multiply_first(acc[j][i], ow[h][j], ox[h][i]);
                else multiply(acc[j][i], ow[h][j], ox[h][i]);
                // (one of the others behind a product each: it issues while the product runs; done some way before the wait for them)
                constexpr int kReads = kX == 8 ? 3 : 1, kFetches = kX == 8 ? 7 : 4;
                const int at = j * kX + i, n = at / kReads;
                if (at % kReads == 0 && n < 16) {
                    if (n & 1) read_x(from_x, h ^ 1, n >> 1);
                    else read_w(from_w, h ^ 1, n >> 1);
                }
                if (at % kFetches == 0 && at / kFetches < 8) aim_load(at / kFetches, to);
                if (at % kFetches == 1 && at / kFetches < 8) {
                    if (h == 0) load_x(at / kFetches);
                    else load_w(at / kFetches);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if constexpr (h == 1) {
            next_k += kStageK;
            place_x = ahead(place_x, 2);
        }
    };
    auto leave = [&](const Tile& g, auto half) {
        constexpr bool kNarrow = decltype(half)::value;
        constexpr int kX = kNarrow ? 4 : 8;
        asm volatile("s_nop 15\n\ts_nop 3");
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int i = 0; i < kX; ++i) asm volatile("" : "+a"(acc[j][i]));
        const int64_t rows = min((int64_t)(kNarrow ? kHalf : kTileSide), (int64_t)p.T - g.t0);
        const rsrc_t out = make_rsrc(static_cast<char*>(p.y) + (int64_t)g.t0 * p.y_pitch * 2, (uint32_t)(((rows - 1) * p.y_pitch + p.M) * 2));
        const int col = g.m0 + 128 * wm + 8 * fq;
        uint32_t at = ((uint32_t)(wt * (kNarrow ? kHalf / 2 : kHalf) + fr) * (uint32_t)p.y_pitch + (uint32_t)col) * 2u;
#pragma unroll
        for (int i = 0; i < kX; ++i) {
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                bf16x8 v;
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = static_cast<__bf16>(acc[2 * c + (e >> 2)][i][e & 3]);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), out, col + 32 * c < p.M ? at + 64u * c : kNowhere, 0, 0);
            }
            at += 32u * (uint32_t)p.y_pitch;
        }
        stores = 4 * kX;
    };
    const int stages = max(2, (p.K + kStageK - 1) / kStageK);
    const std::integral_constant<int, 0> one; const std::integral_constant<int, 1> two;

    Tile g = next_tile();
    if (g.t0 < 0) return;
    aim(g);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            aim_load(i & 7, lds0 + (uint32_t)(2 * s + (i >> 3)) * kChunk);
            asm volatile("s_nop 0");
            if (i < 8) load_x(i);
            else load_w(i & 7);
        }
        next_k += kStageK;
    }
    set_x(g.half);
    asm volatile("s_waitcnt vmcnt(16)\n\ts_barrier" ::: "memory");
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        read_x(0, 0, i);
        read_w(kChunk, 0, i);
    }
    auto walk = [&](auto narrow, const Tile& tile, const Tile& then) {
        if (stages == 2) aim(then);
        step(std::true_type{}, narrow, one);
        step(std::true_type{}, narrow, two);
        for (int q = 1; q < stages; ++q) {
            if (q + 2 == stages) aim(then);
            step(std::false_type{}, narrow, one);
            if (q + 1 == stages) set_x(then.half);
            step(std::false_type{}, narrow, two);
        }
        leave(tile, narrow);
    };
    for (;;) {
        const Tile then = next_tile();
        if (g.half) walk(std::true_type{}, g, then);
        else walk(std::false_type{}, g, then);
        if (then.t0 < 0) break;
        g = then;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

}  // namespace

}  // namespace mpa

using namespace mpa;

namespace {

// Microseconds of a tile and of a half one over a K of so many stages, measured with all CUs busy.
float tile_us(int stages) { return 1.45f * (float)stages + 5.0f; }
float half_us(int stages) { return 0.8f * (float)stages + 3.0f; }

int gemm_check(const mpa_gemm* s) {
    if (!s || !s->x || !s->weight || !s->y) return MPA_ERR_NULL_POINTER;
    constexpr int64_t kMost = (int64_t)1 << 24, kBytes = (int64_t)1 << 31;
    if (s->T <= 0 || s->M <= 0 || s->K <= 0 || s->T > kMost || s->M > kMost || s->K > kMost || s->M % 8 || s->K % 8) return MPA_ERR_BAD_SHAPE;
    const int64_t inner = s->weight_kxm ? s->M : s->K, rows = s->weight_kxm ? s->K + kStageK : kTileSide;
    if (s->x_pitch < s->K || s->weight_pitch < inner || s->y_pitch < s->M || s->x_pitch % 8 || s->weight_pitch % 8 || s->y_pitch % 8) return MPA_ERR_BAD_STRIDE;
    if (s->x_pitch > kMost || s->weight_pitch > kMost || s->y_pitch > kMost || kTileSide * s->x_pitch * 2 >= kBytes || rows * s->weight_pitch * 2 >= kBytes ||
        kTileSide * s->y_pitch * 2 >= kBytes || ((s->T + kTileSide - 1) / kTileSide) * ((s->M + kTileSide - 1) / kTileSide) >= (int64_t)1 << 29)
        return MPA_ERR_BAD_SHAPE;
    if (!aligned_to(s->x, 16) || !aligned_to(s->weight, 16) || !aligned_to(s->y, 16)) return MPA_ERR_MISALIGNED;
    return MPA_OK;
}

// Tiles, and the time of a call.  What is left behind whole rounds of the chip becomes halves where that is shorter than a round of whole ones.
float gemm_plan(const mpa_gemm* s, GemmParams& p) {
    p.x = s->x; p.w = s->weight; p.y = s->y;
    p.x_pitch = s->x_pitch; p.w_pitch = s->weight_pitch; p.y_pitch = s->y_pitch;
    p.T = (int)s->T; p.M = (int)s->M; p.K = (int)s->K;
    p.tiles_t = (p.T + kTileSide - 1) / kTileSide;
    p.tiles_m = (p.M + kTileSide - 1) / kTileSide;
    const int all = p.tiles_t * p.tiles_m, rest = all % kCUs, stages = (p.K + kStageK - 1) / kStageK;
    const float halves = (float)((2 * rest + kCUs - 1) / kCUs) * half_us(stages);
    const bool cut = rest > 0 && halves < tile_us(stages);
    p.full = cut ? all - rest : all;
    p.half = cut ? 2 * rest : 0;
    return (float)((p.full + kCUs - 1) / kCUs) * tile_us(stages) + (cut ? halves : 0.0f);
}

}  // namespace

// Against the library, at 2800 products of 64 to 70 000 rows, 128 to 128 000 columns and a K of 64 to 4096 (W as M x K and, up to 4096 columns, as
// K x M), among them the products of a layer of widths 64 to 1024 (W as M x K: 4d x d, d x 2d; as K x M: 2d x d, d x 4d) and 50 280 x d; its time
// over the library's:
//   K up to 512       0.3 to 1.03 (14 of 1094 up to 1.12, 2048 columns or more by two rounds or three), layers 0.4 to 0.96 (one of 155 1.05).  Not where it is slower: 2048 columns or more in whole tiles over more
//                     than one round, K 64 to 256 (0.57 to 1.42: y is what takes the time, and the library is as fast there), and more than 51 200
//                     columns by a K below 128 (up to 1.18).
//   rows of x or W that are not whole 128 bytes (K % 64), or of y (M % 64; up to 4000 rows or 4096 columns): 0.4 to 1.02
//                     where tiles fill the chip.  The library runs these at 400 to 900 TFLOP/s, 700 is what it is taken for, and 18 us at least (host).
//                     With W as M x K in whole tiles it reaches up to 1340 (0.83 to 1.22): taken for 1400, which leaves its parts of rounds.  Of more than
//                     51 200 columns some are 1.01 to 1.14.
//   others            both take tiles of this size, and whole rounds of them are 0 to 9 % faster there; where this kernel saves a part of a
//                     round by halves, up to K = 1024 (a longer sum leaves the first loads and the stores a smaller part): 0.61 to 0.98
extern "C" int mpa_gemm_faster(const mpa_gemm* s) {
    if (gemm_check(s) != MPA_OK) return 0;
    GemmParams p{};
    const float us = gemm_plan(s, p);
    constexpr int64_t kMostM = 51200;
    const bool whole = s->M % kTileSide == 0;
    if (s->K <= 512) {
        const int tiles = p.tiles_t * p.tiles_m, most = tiles <= 2 * kCUs && !s->weight_kxm ? 384 : 256;
        if (whole && s->M >= 2048 && s->K <= most && s->K % 64 == 0 && tiles > kCUs) return 0;
        return s->M <= kMostM || s->K >= 128;
    }
    if (s->K % 64 || (s->M % 64 && (s->M <= 4096 || s->T <= 4096))) {
        const float rate = whole && !s->weight_kxm ? 1.4f : 0.7f;
        return s->M <= kMostM && us + 3.0f < std::max(18.0f, 6.0f + 2e-9f * (float)s->T * (float)s->M * (float)s->K / rate);
    }
    return s->K <= 1024 && us <= 0.93f * (float)((p.tiles_t * p.tiles_m + kCUs - 1) / kCUs) * tile_us((p.K + kStageK - 1) / kStageK);
}

extern "C" int mpa_gemm_run(const mpa_gemm* s, void* stream) {
    const int rc = gemm_check(s);
    if (rc != MPA_OK) return rc;
    GemmParams p{};
    gemm_plan(s, p);
    const int grid = p.full >= kCUs ? kCUs : (std::max(p.full, std::min(p.half, kCUs)) + 7) / 8 * 8;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const bool tail = p.K % kStageK || p.K < 2 * kStageK;
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), 0, st, p); };
    if (s->weight_kxm) tail ? run(gemm_wide_kernel<true, true>) : run(gemm_wide_kernel<true, false>);
    else tail ? run(gemm_wide_kernel<false, true>) : run(gemm_wide_kernel<false, false>);
    return check_launch();
}
