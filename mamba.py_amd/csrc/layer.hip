// Kernels of a layer's training pass around the library GEMMs, for gfx950:
//
//   wgrad      weight gradients out = P^T . Q of several projections in one launch (P (T, M) the
//              gradient of a projection's output, Q (T, N) its input, T = batch * length rows)
//   cast       up to a dozen conversions of small matrices in one launch: the float32 and padded forms of a layer's
//              parameters before a pass, the float32 gradients of its small parameters in their own types after it
//
// wgrad.  The sum runs over thousands of rows and gives a matrix of a few hundred rows and columns, so
// a kernel that parallelises over the output alone leaves most of the chip idle: as library GEMMs
// the four products of a layer at width 768 and 8000 rows (3072 x 768, 768 x 1536, 80 x 1536,
// 1536 x 48) took 88 + 80 + 80 + 54 us.  Here the 128 x 128 output tiles of all of them are one grid,
// cut over T into `splits` parts that a second kernel adds in a fixed order.
#include "wgrad.h"

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kWgTile = 128;

struct WgradJob {
    const void *p, *q;
    int64_t ldp, ldq;
    int M, N;
    int tiles_n, first_tile;  // tiles of this job: first_tile + tm * tiles_n + tn (p_major) or tn * tiles_m + tm
    int tiles_m, p_major;
    int keep, gap_at, gap;  // output columns kept; output row r comes from row r (+ gap from gap_at on) of P^T Q
    void* out;
};
struct WgradParams {
    WgradJob job[MPA_WGRAD_MAX_JOBS];
    int jobs, tiles, splits;
    int64_t T;
    float* part;  // [splits][tiles][128][128] in the order of the kernel's tiles
};

__device__ __forceinline__ int wgrad_find(const WgradParams& p, int tile) {
    int j = 0;
    while (j + 1 < p.jobs && tile >= p.job[j + 1].first_tile) ++j;
    return j;
}
__device__ __forceinline__ void wgrad_tile_at(const WgradJob& j, int tile, int& tm, int& tn) {
    const int local = tile - j.first_tile;
    if (j.p_major) {
        tm = local / j.tiles_n;
        tn = local - tm * j.tiles_n;
    } else {
        tn = local / j.tiles_m;
        tm = local - tn * j.tiles_m;
    }
}

// Workgroup -> (tile, split).  The chip hands workgroups to its 8 XCDs in turn and each has its own L2:
// an XCD works on one split of T and on a run of neighbouring tiles, which share their P or Q panel
// (the wider of the two is the outer index of the run), so that an L2 fetches its part of the wide
// operand once and of the narrow one once.
__device__ __forceinline__ bool wgrad_work(const WgradParams& p, int& tile, int& split) {
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int groups = 8 / p.splits, per = (p.tiles + groups - 1) / groups;
    split = xcd / groups;
    tile = (xcd % groups) * per + slot;
    return slot < per && tile < p.tiles;
}

// bfloat16.  Both operands have the summation index as their slow dimension, the matrix cores want it
// fast: a lane loads eight neighbouring columns of eight rows (16 bytes each), turns the 8 x 8 block with
// v_perm and stores eight 16-byte units (8 rows of one column), each the operand of one lane, into LDS.
// The units of a panel lie in the order column % 8, column / 8: neighbouring lanes write
// neighbouring units, and a 16-row operand tile is 16 neighbouring units (its rows are then every
// eighth column of the matrix, which only the order of the partial sums has to know).
// 64 rows of T per step, loads of the two steps after it in registers meanwhile: waves 0 and 1 bring the rows of P,
// 2 and 3 those of Q; each wave computes 64 x 64 outputs.  (Loads within branches, and one step ahead: 99 us for the four
// products above, 87 now; the matrix cores are busy 28 % of it, LDS 29 %, and the panels come from L2 at 11 TB/s.)
constexpr int kWgStep = 64;
__device__ __forceinline__ int wg_unit_to_col(int u) { return 8 * (u & 15) + (u >> 4); }

__global__ void __launch_bounds__(256, 2) wgrad_bf16_kernel(const WgradParams p) {
    __shared__ u32x4 lds[2][2][8][kWgTile];  // [buffer][P, Q][group of 8 rows][unit]
    int tile, split;
    if (!wgrad_work(p, tile, split)) return;
    const WgradJob& job = p.job[wgrad_find(p, tile)];
    int tm, tn;
    wgrad_tile_at(job, tile, tm, tn);
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int64_t steps = (p.T + kWgStep - 1) / kWgStep, per = (steps + p.splits - 1) / p.splits;
    const int64_t t_begin = split * per * kWgStep, t_end = min(p.T, (split + 1) * per * kWgStep);
    // this lane's columns and rows of a step
    const int o = wave >> 1, g = 4 * (wave & 1) + (lane >> 4);
    const int64_t ld = o ? job.ldq : job.ldp;
    const char* const src = static_cast<const char*>(o ? job.q : job.p);
    const uint32_t off = ((uint32_t)(8 * g) * (uint32_t)ld + (uint32_t)min((o ? tn : tm) * kWgTile + 8 * (lane & 15), (o ? job.N : job.M) - 8)) * 2u;
    u32x4 raw[2][8];
    auto request = [&](u32x4(&v)[8], int64_t t) {  // (rows from t_end on read as zeros)
        const rsrc_t rows = make_rsrc(src + t * ld * 2, window_bytes((t_end - t) * ld, 0, 2));
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = __builtin_amdgcn_raw_buffer_load_b128(rows, off + (uint32_t)r * (uint32_t)ld * 2u, 0, 0);
    };
    auto stage = [&](const u32x4(&v)[8], int buf) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            u32x4 unit;
            // halves c % 2 of words c / 2 of two rows
#pragma unroll
            for (int r = 0; r < 4; ++r)
                unit[r] = __builtin_amdgcn_perm(v[2 * r + 1][c >> 1], v[2 * r][c >> 1], c & 1 ? 0x07060302u : 0x05040100u);
            lds[buf][o][g][16 * c + (lane & 15)] = unit;
        }
    };
    f32x4 acc[4][4] = {};
    const int mu = 64 * (wave >> 1), nu = 64 * (wave & 1);  // the wave's units of P and Q
    request(raw[0], t_begin);
    request(raw[1], t_begin + kWgStep);
    auto multiply = [&](int buf) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            bf16x8 a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[i] = __builtin_bit_cast(bf16x8, lds[buf][0][4 * k + (lane >> 4)][mu + 16 * i + (lane & 15)]);
                b[i] = __builtin_bit_cast(bf16x8, lds[buf][1][4 * k + (lane >> 4)][nu + 16 * i + (lane & 15)]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    };
    // One barrier a step: behind it the step's operands are in LDS, and the other buffer, which all have read, takes the next step's
    // while the products run.  (The loop has one exit, or every wait in it would be one for all loads in flight; steps
    // beyond the last are of zeros.)
    stage(raw[0], 0);
    request(raw[0], t_begin + 2 * kWgStep);
    for (int64_t t = t_begin; t < t_end; t += 2 * kWgStep) {
#pragma unroll
        for (int buf = 0; buf < 2; ++buf) {
            __syncthreads();
            stage(raw[buf ^ 1], buf ^ 1);
            request(raw[buf ^ 1], t + (3 + buf) * kWgStep);
            multiply(buf);
            __builtin_amdgcn_sched_barrier(0);  // (nothing of the next step before its loads are waited for)
        }
    }
    float* out = p.part + ((int64_t)split * p.tiles + tile) * kWgTile * kWgTile;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                out[(mu + 16 * i + 4 * (lane >> 4) + r) * kWgTile + nu + 16 * j + (lane & 15)] = acc[i][j][r];
}

// float32.  The matrix-core operand of four rows x 16 columns is what a row-major panel in LDS gives as
// it is; rows are 16 floats longer than the tile so that the four rows of an operand fall on different
// banks.  The products that come here are narrow (the wide ones are left to the GEMM library), and a
// float32 product keeps a wave busy 16 times as long as a bfloat16 one: 64 x 64 tiles, 32 x 32 per wave,
// make enough waves (128 x 128 tiles: 54 us for 96 x 2048 and 2048 x 64 over 4096 rows).
constexpr int kWgTileF = 64, kWgStepF = 32, kWgPitch = kWgTileF + 16;
__global__ void __launch_bounds__(256) wgrad_f32_kernel(const WgradParams p) {
    __shared__ float lds[2][2][kWgStepF][kWgPitch];
    int tile, split;
    if (!wgrad_work(p, tile, split)) return;
    const WgradJob& job = p.job[wgrad_find(p, tile)];
    int tm, tn;
    wgrad_tile_at(job, tile, tm, tn);
    const int lane = threadIdx.x & 63, wave = wave_id();
    const int64_t steps = (p.T + kWgStepF - 1) / kWgStepF, per = (steps + p.splits - 1) / p.splits;
    const int64_t t_begin = split * per * kWgStepF, t_end = min(p.T, (split + 1) * per * kWgStepF);
    const int cq = 4 * (threadIdx.x & 15), r0 = threadIdx.x >> 4;  // four columns of rows r0 and r0 + 16
    const char* const src[2] = {static_cast<const char*>(job.p), static_cast<const char*>(job.q)};
    const int64_t ld[2] = {job.ldp, job.ldq};
    const uint32_t off[2] = {((uint32_t)r0 * (uint32_t)job.ldp + (uint32_t)min(tm * kWgTileF + cq, job.M - 4)) * 4u,
                             ((uint32_t)r0 * (uint32_t)job.ldq + (uint32_t)min(tn * kWgTileF + cq, job.N - 4)) * 4u};
    constexpr int kAhead = 4;  // steps in flight
    f32x4 raw[kAhead][2][2];
    auto request = [&](f32x4(&v)[2][2], int64_t t) {  // (rows from t_end on read as zeros)
#pragma unroll
        for (int o = 0; o < 2; ++o) {
            const rsrc_t rows = make_rsrc(src[o] + t * ld[o] * 4, window_bytes((t_end - t) * ld[o], 0, 4));
#pragma unroll
            for (int r = 0; r < 2; ++r)
                v[o][r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, off[o] + (uint32_t)(16 * r) * (uint32_t)ld[o] * 4u, 0, 0));
        }
    };
    f32x4 acc[2][2] = {};
    const int mu = 32 * (wave >> 1), nu = 32 * (wave & 1);
#pragma unroll
    for (int i = 0; i < kAhead; ++i) request(raw[i], t_begin + i * kWgStepF);
    auto stage = [&](const f32x4(&v)[2][2], int buf) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int r = 0; r < 2; ++r) *reinterpret_cast<f32x4*>(&lds[buf][o][r0 + 16 * r][cq]) = v[o][r];
    };
    auto multiply = [&](int buf) {
#pragma unroll
        for (int k = 0; k < kWgStepF / 4; ++k) {
            float a[2], b[2];
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                a[n] = lds[buf][0][4 * k + (lane >> 4)][mu + 16 * n + (lane & 15)];
                b[n] = lds[buf][1][4 * k + (lane >> 4)][nu + 16 * n + (lane & 15)];
            }
#pragma unroll
            for (int n = 0; n < 2; ++n)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[n][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[n], b[j], acc[n][j], 0, 0, 0);
        }
    };
    int64_t t = t_begin;
    for (; t + (kAhead - 1) * kWgStepF < t_end; t += kAhead * kWgStepF) {
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            stage(raw[i], i & 1);
            __syncthreads();
            request(raw[i], t + (kAhead + i) * kWgStepF);
            multiply(i & 1);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int i = 0; i < kAhead - 1; ++i) {
        if (t + i * kWgStepF >= t_end) break;  // uniform over the block
        stage(raw[i], i & 1);
        __syncthreads();
        multiply(i & 1);
    }
    float* out = p.part + ((int64_t)split * p.tiles + tile) * kWgTileF * kWgTileF;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                out[(mu + 16 * i + 4 * (lane >> 4) + r) * kWgTileF + nu + 16 * j + (lane & 15)] = acc[i][j][r];
}

// Sum over the splits, in order; a thread takes kCols neighbouring output columns of one row of a tile.
template <typename IO>
__global__ void __launch_bounds__(256) wgrad_sum_kernel(const WgradParams p) {
    constexpr bool UNITS = sizeof(IO) == 2;
    constexpr int kTileIO = UNITS ? kWgTile : kWgTileF, kCols = UNITS ? 8 : 4, kGroups = kTileIO / kCols;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int tile = (int)(id / (kTileIO * kGroups)), local = (int)(id % (kTileIO * kGroups));
    const WgradJob& job = p.job[wgrad_find(p, tile)];
    int tm, tn;
    wgrad_tile_at(job, tile, tm, tn);
    const int u = local / kGroups, q = local % kGroups;
    const int row_in = tm * kTileIO + (UNITS ? wg_unit_to_col(u) : u), col = tn * kTileIO + kCols * q;
    if (row_in >= job.M || (row_in >= job.gap_at && row_in < job.gap_at + job.gap) || col >= job.keep) return;
    const float* src = p.part + (int64_t)tile * kTileIO * kTileIO + u * kTileIO;
    const int64_t pitch = (int64_t)p.tiles * kTileIO * kTileIO;
    float s[kCols] = {};
    for (int k = 0; k < p.splits; ++k) {
        const float* v = src + k * pitch;
#pragma unroll
        for (int c = 0; c < kCols; ++c) s[c] += v[UNITS ? kGroups * c + q : kCols * q + c];
    }
    const int row = row_in >= job.gap_at ? row_in - job.gap : row_in;
    IO* out = static_cast<IO*>(job.out) + (int64_t)row * job.keep + col;
#pragma unroll
    for (int c = 0; c < kCols; ++c)
        if (col + c < job.keep) out[c] = from_float<IO>(s[c]);
}

static int wgrad_tile(int io_dtype) { return io_dtype == MPA_F32 ? kWgTileF : kWgTile; }

static int wgrad_params(WgradParams& p, const mpa_wgrad_job* jobs, int n, int64_t T, int io_dtype) {
    if (!jobs) return MPA_ERR_NULL_POINTER;
    if (n <= 0 || n > MPA_WGRAD_MAX_JOBS || T <= 0) return MPA_ERR_BAD_SHAPE;
    if (io_dtype != MPA_F32 && io_dtype != MPA_BF16) return MPA_ERR_BAD_DTYPE;
    p.jobs = n;
    p.T = T;
    int64_t tiles = 0;
    const int tile = wgrad_tile(io_dtype);
    for (int i = 0; i < n; ++i) {
        const mpa_wgrad_job& s = jobs[i];
        WgradJob& j = p.job[i];
        const int64_t v = io_dtype == MPA_BF16 ? 8 : 4;  // elements of a 16-byte load
        if (s.rows < v || s.cols < v || s.rows % v || s.cols % v || s.rows > 1 << 20 || s.cols > 1 << 20 || s.keep_cols < 1 ||
            s.keep_cols > s.cols || s.gap < 0 || s.gap_at < 0 || s.gap_at + s.gap > s.rows)
            return MPA_ERR_BAD_SHAPE;
        if (s.ldp < s.rows || s.ldq < s.cols || s.ldp % v || s.ldq % v) return MPA_ERR_BAD_STRIDE;
        j.p = s.p; j.q = s.q; j.out = s.out;
        j.ldp = s.ldp; j.ldq = s.ldq;
        j.M = (int)s.rows; j.N = (int)s.cols;
        j.keep = (int)s.keep_cols;
        j.gap_at = s.gap ? (int)s.gap_at : j.M; j.gap = (int)s.gap;
        j.tiles_m = (j.M + tile - 1) / tile;
        j.tiles_n = (j.N + tile - 1) / tile;
        j.p_major = j.tiles_m >= j.tiles_n;
        j.first_tile = (int)tiles;
        tiles += (int64_t)j.tiles_m * j.tiles_n;
        if (tiles > 1 << 20) return MPA_ERR_BAD_SHAPE;
    }
    p.tiles = (int)tiles;
    // parts of T: as few as give about two workgroups per CU (each part writes and reads back all partial
    // tiles), none shorter than 128 rows
    int s = 1;
    while (s < 8 && tiles * s < 400 && T / (2 * s) >= 128) s *= 2;
    p.splits = s;
    return MPA_OK;
}

static size_t wgrad_bytes(const WgradParams& p, int io_dtype) {
    return (size_t)p.splits * p.tiles * wgrad_tile(io_dtype) * wgrad_tile(io_dtype) * sizeof(float);
}

// Estimated time of the bfloat16 kernels here, against which wgrad_wide.hip measures its tiles: a step of 64 rows takes 0.75 us with one workgroup
// a CU and 1.27 with two, the sums of the parts come at 4.5 TB/s, and 10 us are launches and latencies.  (Layers of a width and a number of
// rows, here and there: 768 x 8000 94 and 74 us, 1024 x 16384 319 and 191, 512 x 8192 49 and 47, 640 x 4000 46 and 45; 768 x 2048 35 and 38,
// 256 x 16000 35 and 41, 128 x 4096 17 and 23.)
static float wgrad_bf16_us(const WgradParams& p) {
    const float workgroups = (float)p.tiles * (float)p.splits, steps = (float)((p.T + kWgStep - 1) / kWgStep) / (float)p.splits;
    return 10.0f + 0.0146f * workgroups + steps * (workgroups <= 256.0f ? 0.75f : 1.27f * (workgroups <= 512.0f ? 1.0f : workgroups / 512.0f));
}

// ---- small parameters ---------------------------------------------------------------------------

struct CastParams {
    mpa_cast_job job[MPA_CAST_MAX_JOBS];
    unsigned first[MPA_CAST_MAX_JOBS];  // block of every job
    int jobs;
};
// Rows x cols elements a job, row pitches of its own on either side; a block has 1024 of them, a thread four, requested
// together.  Bound by its launch and two memory latencies.  (With up to six elements a thread one after the other, found by
// 64-bit divisions, and as many blocks for the smallest job as for the largest, the forms of a layer of width 768 took 5.9 us, now 4.6.)
template <typename I>
__global__ void __launch_bounds__(256) cast_kernel(const CastParams p) {
    int k = 0;
    while (k + 1 < p.jobs && blockIdx.x >= p.first[k + 1]) ++k;
    const mpa_cast_job& j = p.job[k];
    const I n = (I)(j.rows * j.cols), cols = (I)j.cols, i0 = ((I)(blockIdx.x - p.first[k]) * 256 + threadIdx.x) * 4;
    if (i0 >= n) return;
    I r = i0 / cols, c = i0 - r * cols;
    float v[4];
    int64_t at[4], from[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // (beyond the last element: the last one)
        from[e] = (int64_t)r * j.src_pitch + c;
        at[e] = (int64_t)r * j.dst_pitch + c;
        if (i0 + e + 1 < n && ++c == cols) {
            c = 0;
            ++r;
        }
    }
    if (j.op == MPA_CAST_ZERO) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = 0.0f;
    } else if (j.src_dtype == MPA_F32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = static_cast<const float*>(j.src)[from[e]];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_float(static_cast<const bf16_t*>(j.src)[from[e]]);
    }
    if (j.op == MPA_CAST_TIMES) {
        const float* const factor = static_cast<const float*>(j.factor);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= factor[i0 + e < n ? i0 + e : n - 1];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (i0 + e >= n) break;
        if (j.op == MPA_CAST_NEG_EXP) v[e] = -expf(v[e]);
        if (j.dst_dtype == MPA_F32) static_cast<float*>(j.dst)[at[e]] = v[e];
        else static_cast<bf16_t*>(j.dst)[at[e]] = from_float<bf16_t>(v[e]);
    }
}

}  // namespace mpa

using namespace mpa;

extern "C" size_t mpa_wgrad_workspace_bytes(const mpa_wgrad_job* jobs, int32_t n, int64_t T, int32_t io_dtype) {
    WgradParams p{};
    if (wgrad_params(p, jobs, n, T, io_dtype) != MPA_OK) return 0;
    if (const size_t wide = io_dtype == MPA_BF16 ? wgrad_wide_bytes(jobs, n, T, wgrad_bf16_us(p)) : 0) return wide;
    return wgrad_bytes(p, io_dtype);
}

extern "C" int mpa_wgrad(const mpa_wgrad_job* jobs, int32_t n, int64_t T, int32_t io_dtype, void* workspace, size_t workspace_bytes,
                         void* stream) {
    WgradParams p{};
    const int rc = wgrad_params(p, jobs, n, T, io_dtype);
    if (rc != MPA_OK) return rc;
    const size_t es = dtype_size(io_dtype);
    for (int i = 0; i < n; ++i) {
        if (!p.job[i].p || !p.job[i].q || !p.job[i].out) return MPA_ERR_NULL_POINTER;
        if (!aligned_to(p.job[i].p, 16) || !aligned_to(p.job[i].q, 16) || !aligned_to(p.job[i].out, es)) return MPA_ERR_MISALIGNED;
    }
    if (!workspace) return MPA_ERR_NULL_POINTER;
    if (!aligned_to(workspace, 256)) return MPA_ERR_MISALIGNED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (io_dtype == MPA_BF16) {
        const int wide = wgrad_wide_run(jobs, n, T, wgrad_bf16_us(p), workspace, workspace_bytes, st);
        if (wide != kNotWide) return wide;
    }
    if (workspace_bytes < wgrad_bytes(p, io_dtype)) return MPA_ERR_WORKSPACE;
    p.part = static_cast<float*>(workspace);
    const int groups = 8 / p.splits, per = (p.tiles + groups - 1) / groups;
    const dim3 grid((unsigned)(8 * per)), sums((unsigned)(io_dtype == MPA_F32 ? kWgTileF * kWgTileF / 4 / 256 * p.tiles : kWgTile * kWgTile / 8 / 256 * p.tiles));
    if (io_dtype == MPA_F32) {
        hipLaunchKernelGGL(wgrad_f32_kernel, grid, dim3(256), 0, st, p);
        hipLaunchKernelGGL(wgrad_sum_kernel<float>, sums, dim3(256), 0, st, p);
    } else {
        hipLaunchKernelGGL(wgrad_bf16_kernel, grid, dim3(256), 0, st, p);
        hipLaunchKernelGGL(wgrad_sum_kernel<bf16_t>, sums, dim3(256), 0, st, p);
    }
    return check_launch();
}

extern "C" int mpa_cast(const mpa_cast_job* jobs, int32_t n, void* stream) {
    if (!jobs) return MPA_ERR_NULL_POINTER;
    if (n <= 0 || n > MPA_CAST_MAX_JOBS) return MPA_ERR_BAD_SHAPE;
    CastParams p{};
    p.jobs = n;
    int64_t blocks = 0;
    bool wide = false;  // a job of 2^31 elements
    for (int i = 0; i < n; ++i) {
        const mpa_cast_job& j = jobs[i];
        if (!j.src || !j.dst || (j.op == MPA_CAST_TIMES && !j.factor)) return MPA_ERR_NULL_POINTER;
        if (j.rows <= 0 || j.cols <= 0 || j.src_pitch < j.cols || j.dst_pitch < j.cols) return MPA_ERR_BAD_SHAPE;
        for (int dt : {j.src_dtype, j.dst_dtype})
            if (dt != MPA_F32 && dt != MPA_BF16) return MPA_ERR_BAD_DTYPE;
        if (!aligned_to(j.src, dtype_size(j.src_dtype)) || !aligned_to(j.dst, dtype_size(j.dst_dtype))) return MPA_ERR_MISALIGNED;
        p.job[i] = j;
        p.first[i] = (unsigned)blocks;
        blocks += (j.rows * j.cols + 1023) / 1024;
        wide |= j.rows * j.cols >= (int64_t)1 << 31;
        if (blocks >= (int64_t)1 << 31) return MPA_ERR_BAD_SHAPE;
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (wide) hipLaunchKernelGGL(cast_kernel<int64_t>, dim3((unsigned)blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(cast_kernel<uint32_t>, dim3((unsigned)blocks), dim3(256), 0, st, p);
    return check_launch();
}
