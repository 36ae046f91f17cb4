// Weight gradients out = P^T . Q in bfloat16 (P (T, M), Q (T, N), T thousands of rows) by tiles of 256 x 256, for gfx950.
//
// What bounds such a product is the way of its operands: a tile of 128 x 128 reads 32 KB for 2 MFLOP, and the chip's L2s gave 11 TB/s to
// the kernel of such tiles (layer.hip), with the matrix cores 28 % busy.  A tile of 256 x 256 reads half of that, and a wave with 128 x 128
// of it reads LDS at half the rate too (32 KB for 64 products of 16 x 16 x 32: half of what LDS delivers in their time).
//
// Rows go from memory to LDS directly, 16 bytes a lane, as they are: a stage is 32 rows of 256 columns of P and Q (32 KB), four
// stages a workgroup.  The matrix cores want the summation index (the row) fast; ds_read_b64_tr_b16 turns 4 x 16 blocks as it reads.
// The 32-byte parts of a row are rotated by the row (part ^ (row & 7), by the order in which lanes load), so that the eight
// rows of a half wave fall on different banks.  While a stage is multiplied the operands of the next one are read, and
// the stage after the next two is on its way; one barrier a stage.  Four waves, one a SIMD, with 256 accumulators a lane.
//
// The output is cut into tiles, T into `splits` parts, whose partial tiles a second kernel adds in a fixed order.  What is left of a
// job beside its whole tiles and has 128 rows or columns at most is made of tiles of 128 x 256 (`narrow`): half the products for
// three quarters of the rows.
//
// The four products of a layer, sums included, here and by the 128 x 128 tiles: width 768, 8000 rows 74 and 94 us, 32 768 rows 225 and
// 352; width 1024, 16 384 rows 191 and 320 (1140 TFLOP/s); width 2048, 2500 rows 160 and 210.  With the reads and loads of
// a stage in front of its products instead of between them 16 384 rows took 228.
#include "wgrad.h"

#include <algorithm>

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short i16x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int kWide = 256, kNarrow = 128, kSlice = 32, kRing = 4, kMaxSplits = 16;
constexpr uint32_t kNoColumn = 0x80000000u;  // an offset beyond every window
constexpr int kFullFloats = kWide * kWide, kNarrowFloats = kNarrow * kWide;

// Tiles of one kind of one job: `a` is the operand that gives the tile's rows (the narrow one of a narrow tile), `b` its columns.
struct Region {
    const void *a, *b;
    int64_t lda, ldb;
    int a_cols, b_cols, a0;  // columns of the operands; the first of `a` that the region takes
    int a_blocks, b_blocks;  // blocks of kWide (narrow: one of kNarrow) columns
    int first;               // number of its first tile among those of its kind
    int swapped;             // `a` is Q: rows of the tile are columns of the output
    int keep, gap_at, gap;
    void* out;
};
constexpr int kMaxRegions = 3 * MPA_WGRAD_MAX_JOBS;
struct WideParams {
    Region region[kMaxRegions];  // those of whole tiles first
    int full_regions, regions;
    int full, narrow;            // tiles
    int splits[2];                // parts of T, of whole tiles and of narrow ones
    int full_per, narrow_per;     // workgroups of either kind per XCD
    int64_t T;
    float* part;  // [splits[0]][full][256][256], [splits[1]][narrow][128][256]
};

// slices of a part of T: whole rounds of the ring
__host__ __device__ inline int slices_per(int64_t T, int splits) {
    const int64_t slices = (T + kSlice - 1) / kSlice;
    return (int)(((slices + splits - 1) / splits + kRing - 1) / kRing * kRing);
}

// Workgroup -> part of T and tile; the narrow ones come last.  Workgroups go to the eight XCDs in turn: an XCD takes a run of neighbouring tiles of
// one part of T, which share their rows in its L2.
__device__ __forceinline__ bool wide_work(const WideParams& p, bool& narrow, int& split, int& tile, int& region) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    narrow = slot >= p.full_per;
    const int q = narrow ? xcd * p.narrow_per + slot - p.full_per : xcd * p.full_per + slot;
    const int tiles = narrow ? p.narrow : p.full;
    if (q >= tiles * p.splits[narrow]) return false;
    split = q / tiles;
    tile = q - split * tiles;
    region = narrow ? p.full_regions : 0;
    const int end = narrow ? p.regions : p.full_regions;
    while (region + 1 < end && tile >= p.region[region + 1].first) ++region;
    return true;
}
// block of `a` and of `b`: neighbouring tiles share that of the operand with more of them
__device__ __forceinline__ void region_tile(const Region& r, int local, int& ta, int& tb) {
    if (r.a_blocks >= r.b_blocks) {
        ta = local / r.b_blocks;
        tb = local - ta * r.b_blocks;
    } else {
        tb = local / r.a_blocks;
        ta = local - tb * r.a_blocks;
    }
}

// (Written out: with the accumulators in place.  Left to the compiler, 256 of them leave it no register to move one through, and the
// loop was half copies.  Its operands come from LDS, whose loads the compiler waits for; what reads a sum has the waits at the loop's end before it.)
__device__ __forceinline__ void multiply(f32x4& c, const bf16x8& a, const bf16x8& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// One tile over the rows from t_begin to t_end.  NARROW: 128 columns of `a`, of which every wave takes all and a quarter of those of `b`.
template <bool NARROW>
__device__ __forceinline__ void wide_tile(const Region& g, int ta, int tb, int64_t t_begin, int64_t t_end, float* out, char* lds) {
    constexpr int kStageBytes = 2 * kSlice * kWide * 2, kOperand = kSlice * kWide * 2, kPitch = kWide * 2;
    constexpr int kA = 8, kB = NARROW ? 4 : 8;  // operands of 16 columns a wave
    constexpr int kLoads = 8;                   // of a stage and wave: four for each operand, two rows each
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int a_begin = g.a0 + ta * kWide, b_begin = tb * kWide;
    // the wave's rows of a stage are 8 * wave .. + 7; position (row, part) of LDS holds the row's part ^ 2 * (row & 7)
    uint32_t off[2][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = 8 * wave + 2 * i + (lane >> 5), part = (lane & 31) ^ (2 * (row & 7));
        const int ca = a_begin + 8 * part, cb = b_begin + 8 * part;
        // (columns beyond the operand's last: of its last eight, into results that are not stored)
        off[0][i] = NARROW && part >= kNarrow / 8 ? kNoColumn : ((uint32_t)row * (uint32_t)g.lda + (uint32_t)min(ca, g.a_cols - 8)) * 2u;
        off[1][i] = ((uint32_t)row * (uint32_t)g.ldb + (uint32_t)min(cb, g.b_cols - 8)) * 2u;
    }
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)lds) + (uint32_t)wave * (8 * kPitch);
    // the next slice to request; rows from t_end on read as zeros
    const char* src[2] = {static_cast<const char*>(g.a) + t_begin * g.lda * 2, static_cast<const char*>(g.b) + t_begin * g.ldb * 2};
    int64_t left[2] = {(t_end - t_begin) * g.lda * 2, (t_end - t_begin) * g.ldb * 2};
    // (a window ends at 2^31 bytes, where the columns that a narrow tile does not have are; a slice of 32 rows is shorter, see wide_plan)
    const int64_t ahead[2] = {kSlice * 2 * g.lda, kSlice * 2 * g.ldb};
    u32x4 window[2];
    auto aim = [&] {
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            window[o] = lds_window(src[o], left[o] <= 0 ? 0u : left[o] > kNoColumn ? kNoColumn : (uint32_t)left[o]);
            src[o] += ahead[o];
            left[o] -= ahead[o];
        }
    };
    // load i of the stage that aim() was called for, in two parts with a product between them: where to, and the load.  (A lone wave
    // issues an instruction every five clocks, and a product takes sixteen.)
    // (m0 is where a load finds its place: the value is handed from one to the other in it, so that the compiler leaves it there)
    uint32_t spot;
    auto aim_load = [&](int i, uint32_t to) { asm volatile("s_add_u32 %0, %1, %2" : "={m0}"(spot) : "s"(to), "n"((i >> 2) * kOperand + (i & 3) * 2 * kPitch) : "scc"); };
    auto load = [&](int i) { asm volatile("buffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(off[i >> 2][i & 3]), "s"(window[i >> 2]), "{m0}"(spot) : "memory"); };
    // reads: lane -> row 4 * (lane / 16) + lane % 16 / 4 of the first sixteen (the other sixteen behind them), four columns from 4 * (lane % 4)
    const int rowl = 4 * (lane >> 4) + ((lane & 15) >> 2), r7 = rowl & 7;
    uint32_t at_a[kA], at_b[kB];
    const uint32_t base = (uint32_t)(rowl * kPitch + (lane & 3) * 8);
#pragma unroll
    for (int i = 0; i < kA; ++i) at_a[i] = base + (NARROW ? 0u : (uint32_t)(wave >> 1) * 256u) + (uint32_t)((i ^ r7) * 32);
#pragma unroll
    for (int i = 0; i < kB; ++i)
        at_b[i] = base + kOperand + (NARROW ? (uint32_t)(wave >> 1) * 256u + (uint32_t)(((4 * (wave & 1) + i) ^ r7) * 32) : (uint32_t)(wave & 1) * 256u + (uint32_t)((i ^ r7) * 32));
    typedef __attribute__((address_space(3))) i16x4* LdsPtr;
    auto lds_base = (__attribute__((address_space(3))) char*)lds;
    auto read = [&](i16x4& v, uint32_t at, int buf, int half) {
        v = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsPtr)(lds_base + at + buf * kStageBytes + half * 16 * kPitch));
    };
    struct Operand { i16x4 half[2]; };
    f32x4 acc[kB][kA] = {};
    Operand a[2][kA], b[2][kB];
    const int slices = (int)((t_end - t_begin + kSlice - 1) / kSlice);
#pragma unroll
    for (int s = 0; s < kRing; ++s) {
        aim();
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            aim_load(i, lds0 + (uint32_t)(s * kStageBytes));
            asm volatile("s_nop 0");
            load(i);
        }
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((kRing - 1) * kLoads) : "memory");
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        read(a[0][i >> 1].half[i & 1], at_a[i >> 1], 0, i & 1);
        if (i < 2 * kB) read(b[0][i >> 1].half[i & 1], at_b[i >> 1], 0, i & 1);
    }
    // Stage s (operands in set s % 2) is multiplied in eight groups, between which the operands of the next stage are read and the loads of
    // stage s + kRing are issued into its own buffer, which all waves have read behind the barrier.
    auto step = [&](int buf) {
        const int x = buf & 1, y = x ^ 1;
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((kRing - 2) * kLoads) : "memory");
        aim();
        const uint32_t to = lds0 + (uint32_t)(buf * kStageBytes);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#pragma unroll
            for (int j = 0; j < kB; ++j) {
                multiply(acc[j][i], __builtin_bit_cast(bf16x8, b[x][j]), __builtin_bit_cast(bf16x8, a[x][i]));
                // (one of the others behind a product each: it issues while the product runs; the reads done some way before the wait for them)
                constexpr int kFetches = NARROW ? 4 : 8;
                const int at = i * kB + j, n = at;
                if (n < 2 * (kA + kB)) {
                    const int o = n >> 1, half = n & 1;
                    if (o < kB) read(b[y][o].half[half], at_b[o], (buf + 1) % kRing, half);
                    else read(a[y][o - kB].half[half], at_a[o - kB], (buf + 1) % kRing, half);
                }
                if (at % kFetches == 0 && at / kFetches < kLoads) aim_load(at / kFetches, to);
                if (at % kFetches == 1 && at / kFetches < kLoads) load(at / kFetches);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    static_assert(kRing == 4, "the loop's steps");
    // (whole rounds of the ring: slices beyond the last are of zeros.  The last products' results are 19 wait states away from whatever
    // the compiler does with them.)
    int s = 0;
    do {
        step(0);
        step(1);
        step(2);
        step(3);
        asm volatile("s_nop 15\n\ts_nop 3");
    } while ((s += kRing) < slices);
#pragma unroll
    for (int j = 0; j < kB; ++j)
#pragma unroll
        for (int i = 0; i < kA; ++i) asm volatile("" : "+a"(acc[j][i]));
    const int row0 = NARROW ? 0 : 128 * (wave >> 1), col0 = NARROW ? 64 * wave : 128 * (wave & 1);
#pragma unroll
    for (int i = 0; i < kA; ++i)
#pragma unroll
        for (int j = 0; j < kB; ++j)
            *reinterpret_cast<f32x4*>(out + (row0 + 16 * i + (lane & 15)) * kWide + col0 + 16 * j + 4 * (lane >> 4)) = acc[j][i];
}

__global__ void __launch_bounds__(256, 1) wgrad_wide_kernel(const WideParams p) {
    __shared__ alignas(16) char lds[kRing * 2 * kSlice * kWide * 2];
    bool narrow;
    int split, tile, region;
    if (!wide_work(p, narrow, split, tile, region)) return;
    const Region& g = p.region[region];
    int ta, tb;
    region_tile(g, tile - g.first, ta, tb);
    const int64_t per = (int64_t)slices_per(p.T, p.splits[narrow]) * kSlice;
    const int64_t t_begin = min(p.T, split * per), t_end = min(p.T, (split + 1) * per);
    if (!narrow) wide_tile<false>(g, ta, tb, t_begin, t_end, p.part + ((int64_t)split * p.full + tile) * kFullFloats, lds);
    else wide_tile<true>(g, ta, tb, t_begin, t_end, p.part + (int64_t)p.splits[0] * p.full * kFullFloats + ((int64_t)split * p.narrow + tile) * kNarrowFloats, lds);
}

// Sum over the parts of T, in order.  A thread takes eight neighbouring columns of a row of a tile; blocks of a tile are 8 rows.
__global__ void __launch_bounds__(256) wgrad_wide_sum_kernel(const WideParams p) {
    const int full_blocks = p.full * (kWide / 8);
    const bool narrow = (int)blockIdx.x >= full_blocks;
    const int q = narrow ? (int)blockIdx.x - full_blocks : (int)blockIdx.x, per = (narrow ? kNarrow : kWide) / 8;
    const int tile = q / per, row = (q - tile * per) * 8 + (int)(threadIdx.x >> 5), col = 8 * (int)(threadIdx.x & 31);
    int region = narrow ? p.full_regions : 0;
    const int end = narrow ? p.regions : p.full_regions;
    while (region + 1 < end && tile >= p.region[region + 1].first) ++region;
    const Region& g = p.region[region];
    int ta, tb;
    region_tile(g, tile - g.first, ta, tb);
    const int ra = g.a0 + ta * kWide + row, cb = tb * kWide + col;
    if (ra >= g.a_cols || cb >= g.b_cols) return;
    const int64_t pitch = (int64_t)(narrow ? p.narrow * kNarrowFloats : p.full * (int64_t)kFullFloats);
    const float* src = p.part + (narrow ? (int64_t)p.splits[0] * p.full * kFullFloats + (int64_t)tile * kNarrowFloats : (int64_t)tile * kFullFloats) + row * kWide + col;
    f32x4 s[2] = {};
    constexpr int kSome = 4;
    const int splits = p.splits[narrow];
    for (int k0 = 0; k0 < splits; k0 += kSome) {
        f32x4 v[kSome][2];
#pragma unroll
        for (int k = 0; k < kSome; ++k) {
            const f32x4* from = reinterpret_cast<const f32x4*>(src + min(k0 + k, splits - 1) * pitch);
            v[k][0] = from[0];
            v[k][1] = from[1];
        }
#pragma unroll
        for (int k = 0; k < kSome; ++k) {
            if (k0 + k >= splits) break;
            s[0] += v[k][0];
            s[1] += v[k][1];
        }
    }
    bf16_t* const out = static_cast<bf16_t*>(g.out);
    if (!g.swapped) {
        if (ra >= g.gap_at && ra < g.gap_at + g.gap) return;
        bf16_t* const to = out + (int64_t)(ra >= g.gap_at ? ra - g.gap : ra) * g.keep + cb;
        if (g.keep % 8 == 0 && cb + 8 <= g.keep && (reinterpret_cast<uintptr_t>(g.out) & 15) == 0) {
            bf16x8 r;
#pragma unroll
            for (int c = 0; c < 8; ++c) r[c] = static_cast<__bf16>(s[c >> 2][c & 3]);
            *reinterpret_cast<bf16x8*>(to) = r;
        } else {
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (cb + c < g.keep) to[c] = from_float<bf16_t>(s[c >> 2][c & 3]);
        }
    } else if (ra < g.keep) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int m = cb + c;
            if (m < g.b_cols && (m < g.gap_at || m >= g.gap_at + g.gap))
                out[(int64_t)(m >= g.gap_at ? m - g.gap : m) * g.keep + ra] = from_float<bf16_t>(s[c >> 2][c & 3]);
        }
    }
}

// Regions and parts of T.
bool wide_plan(WideParams& p, const mpa_wgrad_job* jobs, int n, int64_t T, float other_us) {
    p.regions = p.full = p.narrow = 0;
    p.T = T;
    for (int i = 0; i < n; ++i)
        if (std::max(jobs[i].ldp, jobs[i].ldq) >= (int64_t)kNoColumn / (kSlice * 2)) return false;
    auto add = [&](const mpa_wgrad_job& s, bool swapped, int a0, int a_blocks, int b_blocks, int& tiles) {
        if (a_blocks == 0 || b_blocks == 0) return;
        Region& r = p.region[p.regions++];
        r.a = swapped ? s.q : s.p; r.b = swapped ? s.p : s.q;
        r.lda = swapped ? s.ldq : s.ldp; r.ldb = swapped ? s.ldp : s.ldq;
        r.a_cols = (int)(swapped ? s.cols : s.rows); r.b_cols = (int)(swapped ? s.rows : s.cols);
        r.a0 = a0;
        r.a_blocks = a_blocks; r.b_blocks = b_blocks;
        r.first = tiles;
        r.swapped = swapped;
        r.keep = (int)s.keep_cols;
        r.gap_at = s.gap ? (int)s.gap_at : (int)s.rows; r.gap = (int)s.gap;
        r.out = s.out;
        tiles += a_blocks * b_blocks;
    };
    // blocks of 256 columns of an operand that whole tiles take; the rest, if it is 128 or fewer, is left to narrow ones
    auto blocks = [](int64_t cols) { return (int)(cols / kWide + (cols % kWide > kNarrow)); };
    auto rest = [](int64_t cols) { return cols % kWide > 0 && cols % kWide <= kNarrow; };
    for (int i = 0; i < n; ++i) add(jobs[i], false, 0, blocks(jobs[i].rows), blocks(jobs[i].cols), p.full);
    p.full_regions = p.regions;
    for (int i = 0; i < n; ++i) {
        const int m = blocks(jobs[i].rows), c = blocks(jobs[i].cols);
        if (rest(jobs[i].rows)) add(jobs[i], false, m * kWide, 1, c + rest(jobs[i].cols), p.narrow);
        if (rest(jobs[i].cols)) add(jobs[i], true, c * kWide, 1, m, p.narrow);
    }
    // Parts of T by an estimate of the time: a slice of a whole tile takes 0.72 us, of a narrow one 0.45, after 4 for the first
    // loads and the sums' way out; one workgroup a CU, the narrow ones on the CUs that the last round of whole ones leaves; the sums of the parts are
    // read at 4.5 TB/s.
    constexpr int kCUs = 256;
    constexpr float kOnceUs = 13.0f;  // two launches, what the sums take beyond their bytes, and 5 us for being sure (4: 6000 rows of width 512 42.2 us -> 44.5)
    const int64_t slices = (T + kSlice - 1) / kSlice;
    float best = 1e30f;
    for (int s = 1; s <= kMaxSplits && (s == 1 || (slices >= 8 * s && p.full * (s - 1) <= 2 * kCUs)); ++s) {
        const int64_t nf = (int64_t)p.full * s, rounds = (nf + kCUs - 1) / kCUs;
        const int left = (int)(rounds * kCUs - nf);
        const float t_full = p.full ? 4.0f + 0.72f * (float)slices_per(T, s) : 0.0f, walk = (float)rounds * t_full;
        const int some[] = {1, 2, 4, 8, kMaxSplits, p.narrow ? std::min(left / p.narrow, kMaxSplits) : 0};
        for (int sn : some) {
            if (sn < 1 || (sn > 1 && (p.narrow == 0 || slices < 8 * sn))) continue;
            const float t_narrow = 4.0f + 0.45f * (float)slices_per(T, sn);
            const int64_t nn = (int64_t)p.narrow * sn, fit = left * std::max<int64_t>(t_full >= t_narrow, (int64_t)(t_full / t_narrow));
            const float us = walk + (nn > fit ? (float)((nn - fit + kCUs - 1) / kCUs) * t_narrow : 0.0f) + (float)(0.262 * (double)nf + 0.131 * (double)nn) / 4.5f;
            if (us < best) {
                best = us;
                p.splits[0] = s;
                p.splits[1] = sn;
            }
        }
    }
    p.full_per = (int)(((int64_t)p.full * p.splits[0] + 7) / 8);
    p.narrow_per = (int)(((int64_t)p.narrow * p.splits[1] + 7) / 8);
    return best + kOnceUs < other_us;
}

size_t wide_bytes(const WideParams& p) { return ((size_t)p.splits[0] * p.full * kFullFloats + (size_t)p.splits[1] * p.narrow * kNarrowFloats) * sizeof(float); }

}  // namespace

size_t wgrad_wide_bytes(const mpa_wgrad_job* jobs, int n, int64_t T, float other_us) {
    WideParams p;
    return wide_plan(p, jobs, n, T, other_us) ? wide_bytes(p) : 0;
}

int wgrad_wide_run(const mpa_wgrad_job* jobs, int n, int64_t T, float other_us, void* workspace, size_t workspace_bytes, hipStream_t st) {
    WideParams p;
    if (!wide_plan(p, jobs, n, T, other_us)) return kNotWide;
    if (workspace_bytes < wide_bytes(p)) return MPA_ERR_WORKSPACE;
    p.part = static_cast<float*>(workspace);
    hipLaunchKernelGGL(wgrad_wide_kernel, dim3((unsigned)(8 * (p.full_per + p.narrow_per))), dim3(256), 0, st, p);
    hipLaunchKernelGGL(wgrad_wide_sum_kernel, dim3((unsigned)(p.full * (kWide / 8) + p.narrow * (kNarrow / 8))), dim3(256), 0, st, p);
    return check_launch();
}

}  // namespace mpa
