// y (T x M) = x (T x K) . W (M x K)^T for the projections of a layer over a short sequence, for gfx950.
//
// A prompt of a few hundred steps gives products of a few GFLOP: what they cost is latency (a library
// call of 8-12 us on the device and 18 us on the host each), not arithmetic.  The kernels here
// run one tile per workgroup, as many workgroups as the shape offers, and take over the element-wise work around
// the product: with `residual` the sum y + residual is stored, with `ssq_out` the partial sums of squares of its rows;
// with `ssq`, those of x, the rows of x are normalised on their way into LDS (x * rstd * weight, rounded, as the norm
// kernel rounds; a form for callers of the C interface).  Between the layers of a stack the norm is in two places instead: out_proj
// stores the rows of the stream times the next norm's weight as well, rounded once as a normalised row is, and in_proj multiplies its
// product with their rstd.  The residual stream between bfloat16 layers can be float32: x (with `ssq`), y and residual each have a flag.
//
// Tile: BT steps x BM rows of W per workgroup, each wave 32 * RT x 32 of it (2 * RT x 2 MFMA tiles of 16 x 16, W as the left
// operand, so that a lane's four results are neighbours in y) over its share of K.  K runs in stages of 128 bytes per
// share: a stage is in LDS in 16-byte parts, rotated by the row (part ^ (row & 7)) so that the operand reads, one row
// per lane, fall on different banks.  Rows that are multiplied as they stand in memory (with a factor or without) go to LDS directly, three stages:
// two are on their way while one is multiplied, by one barrier a stage.  What has to be changed between memory and LDS (rows that are
// normalised, W by columns) passes through D sets of registers, two stages in LDS.
//
// Width 768, recorded in a graph with the operands of 24 layers, through registers / directly / the library's product alone:
//              in_proj with the rows' factor   out_proj, residual, scaled rows   x_proj         dt_proj
//   32 steps          6.4 /  5.9 /  7.0 us           7.8 /  6.2 /  7.2            6.9 / 5.4      3.6 / 3.2
//   512               9.6 /  8.2 /  9.0              9.1 /  8.0 /  7.9            7.3 / 5.7      3.8 / 3.4
//   2048             23.4 / 24.3 / 17.1             19.4 / 18.5 / 17.0            7.6 / 6.6      6.3 / 5.8
// (In a whole pass of 512 steps, under the profiler, they are 10.3 and 9.2.  The third stage in LDS leaves two workgroups a CU instead of three of 64 x
// 128: in_proj in 640 to 768 such tiles is 2 to 6 % slower for it, out_proj of the same steps 5 to 7 % faster.)  What bounds the short
// ones is latency: the launch, the first rows from memory, a barrier a stage, the way of the results.  Besides, the kernels save the norm between the
// layers (6 us) and three quarters of the host time (24 layers of library calls: 2.1 ms, all of it host).
// float32 runs the same tiles with sixteen times less of the matrix unit's rate (16x16x4, 150 TFLOP/s): the same host
// time is saved, until the product itself is longer than a library call (a training layer of 1614 steps and width 424
// 0.69 ms, 0.81 with library calls; 168 steps of ten layers of width 640 without gradients 0.63 and 0.85 ms).
#include "common.h"
#include "row_offset.h"

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// What a 16-byte part holds: kVec elements; a stage is 8 parts of every row.
template <typename IO>
struct LinearOps;
template <>
struct LinearOps<bf16_t> {
    static constexpr int kVec = 8;
    typedef bf16x4 Out;
    static __device__ __forceinline__ float get(const Out& v, int e) { return static_cast<float>(v[e]); }
    static __device__ __forceinline__ void set(Out& v, int e, float f) { v[e] = static_cast<__bf16>(f); }
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
    static __device__ __forceinline__ u32x4 scale(const u32x4& v, float rs, const f32x4 (&w)[2]) {
        bf16x8 x = __builtin_bit_cast(bf16x8, v);
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = static_cast<__bf16>(static_cast<float>(x[e]) * rs * w[e >> 2][e & 3]);
        return __builtin_bit_cast(u32x4, x);
    }
    static __device__ __forceinline__ u32x4 scale_f32(const u32x4& lo, const u32x4& hi, float rs, const f32x4 (&w)[2]) {
        bf16x8 x;
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = static_cast<__bf16>(__uint_as_float(e < 4 ? lo[e] : hi[e - 4]) * rs * w[e >> 2][e & 3]);
        return __builtin_bit_cast(u32x4, x);
    }
};
template <>
struct LinearOps<float> {
    static constexpr int kVec = 4;
    typedef f32x4 Out;
    static __device__ __forceinline__ float get(const Out& v, int e) { return v[e]; }
    static __device__ __forceinline__ void set(Out& v, int e, float f) { v[e] = f; }
    // (four products of one k per lane group; the groups' k are those of the part, whatever their order)
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4& b, f32x4& c) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[e]), __uint_as_float(b[e]), c, 0, 0, 0);
    }
    static __device__ __forceinline__ u32x4 scale(const u32x4& v, float rs, const f32x4 (&w)[1]) {
        u32x4 x;
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __float_as_uint(__uint_as_float(v[e]) * rs * w[0][e]);
        return x;
    }
};

// (one word next to the sizes, in registers from the start: a scalar load at the end of the kernel is a latency by itself)
enum LinearFlags {
    kAccumulate = 1,   // the residual is added before the result is rounded
    kYF32 = 2,         // y is float32 whatever IO is
    kResidualF32 = 4,  // so is the residual
    kXLarger = 8,      // x has more bytes than W
    kBySteps = 16,     // tiles walk W first: set by the launch
    kRowsWrap = 32,    // rows beyond the last have to be kept outside of the windows: set by the launch
};
struct LinearParams {
    const void *x, *w, *bias;
    int64_t x_pitch, y_pitch;
    int T, M, K;
    int flags;  // LinearFlags
    int tiles, tiles_per_xcd, inner;  // of the launch: all, an XCD's share, those of the dimension that is walked first
    uint32_t inner_inv;
    void* y;
    const float* ssq;  // [in_parts][T]
    int in_parts;
    float inv_d, eps;
    const float* norm_w;  // [K], with ssq
    const void* residual;
    float* ssq_out;  // [M/32 rounded up][T]
    const float* y_weight;  // [M]
    void* y_scaled;         // [T][M]: y * y_weight
};

// How x comes: as it is, to be normalised, float32 (IO is bfloat16) and to be normalised, or as it is, its rows' rstd a
// factor of the product.
enum LinearX { kPlainX = 0, kNormX = 1, kNormXF32 = 2, kFactor = 3 };

constexpr int linear_threads(int BT, int BM, int KS, int RT) { return BT / (32 * RT) * (BM / 32) * KS * kWave; }

template <typename IO, int BT, int BM, int KS, int RT, int D, int XMODE, bool NN>
__global__ void __launch_bounds__(linear_threads(BT, BM, KS, RT)) linear_kernel(const LinearParams p) {
    typedef LinearOps<IO> Ops;
    constexpr bool NORM = XMODE == kNormX || XMODE == kNormXF32, XF32 = XMODE == kNormXF32;
    static_assert(!XF32 || sizeof(IO) == 2, "float32 x of a bfloat16 product");
    constexpr uint32_t kXES = XF32 ? 4 : sizeof(IO);  // bytes of an element of x
    constexpr int kVec = Ops::kVec, kStep = 8 * kVec;  // k of a stage and share
    constexpr uint32_t kES = sizeof(IO);
    constexpr int kThreads = linear_threads(BT, BM, KS, RT), kWavesM = BM / 32;
    static_assert(BM * 8 * KS % kThreads == 0, "a load instruction reads W or x");
    constexpr int kRows = BT + BM, kParts = 8 * KS, kLoads = kRows * kParts / kThreads, kStage = kRows * kParts;  // 16-byte parts
    static_assert(D % 2 == 0, "a set of registers always goes to the same buffer");
    // Rows as they are in memory go to LDS directly, kBuffers - 1 stages ahead; W by columns and rows to be scaled pass through registers.
    constexpr bool kDirect = !NN && !NORM;
    constexpr int kBuffers = kDirect ? 3 : 2;
    __shared__ u32x4 lds[kBuffers][kStage];
    asm volatile("" ::"s"(p.x), "s"(p.w), "s"(p.bias), "s"(p.x_pitch), "s"(p.y_pitch), "s"(p.T), "s"(p.M), "s"(p.K), "s"(p.flags), "s"(p.y), "s"(p.ssq),
                 "s"(p.in_parts), "s"(p.tiles), "s"(p.tiles_per_xcd), "s"(p.inner), "s"(p.inner_inv), "s"(p.inv_d), "s"(p.eps), "s"(p.residual), "s"(p.ssq_out), "s"(p.y_weight), "s"(p.y_scaled));
    // Blocks of one XCD (every eighth) take neighbouring tiles and share one operand's rows in its L2: those of W, whose
    // tiles' steps they walk first, or of x where that is the larger one (each XCD reads the other operand whole) and tiles
    // are many (17 layers of width 528, 4038 steps: 2.27 -> 2.17 ms; below two rounds of tiles it made no difference).
    // (the division by tiles of the inner dimension as a product with its reciprocal, rounded up: exact below 2^16 tiles)
    const int flags = p.flags;
    const int tile = (int)(blockIdx.x & 7) * p.tiles_per_xcd + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= p.tiles_per_xcd || tile >= p.tiles) return;  // uniform over the block
    const int major = p.inner_inv ? (int)__umulhi((uint32_t)tile, p.inner_inv) : tile / p.inner, minor = tile - major * p.inner;
    const bool by_steps = flags & kBySteps;
    const int m0 = (by_steps ? minor : major) * BM, t0 = (by_steps ? major : minor) * BT;
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int ks = wave % KS, wm = wave / KS % kWavesM, wt = wave / KS / kWavesM;

    // (buffer loads: a part beyond K gets an offset beyond the window and reads as zero without a branch, which
    // would make every wait one for all loads in flight)
    const rsrc_t rw = make_rsrc(p.w, (uint32_t)p.M * (uint32_t)p.K * kES);  // (both forms of W are dense)
    const rsrc_t rx = make_rsrc(p.x, ((uint32_t)(p.T - 1) * (uint32_t)p.x_pitch + (uint32_t)p.K) * kXES);
    constexpr int kWLoads = BM * kParts / kThreads;  // the loads of W; those of x follow
    constexpr int kRowsPer = sizeof(IO) == 2 ? 2 : 1;  // rows of W that make a word in LDS
    uint32_t off[kLoads];
    int koff[kLoads], at[kLoads];
    // Direct loads: a wave fetches for its own share of K, 64 places of LDS (eight rows) at a time, W's rows first; a lane's part of K is the
    // same in all of them.  (Rows beyond the last are read as zeros: they are
    // beyond the window.  Their results are not stored.)
    constexpr int kShareWaves = kThreads / kWave / KS, kRowStep = 8 * kShareWaves;
    static_assert(!kDirect || (BM % kRowStep == 0 && kRows % kRowStep == 0), "a load instruction reads W or x");
    const int share_wave = wave / KS, part_of = (lane & 7) ^ (lane >> 3);
    const int kl = (ks * 8 + part_of) * kVec;
    const u32x4 win_w = lds_window(p.w, (uint32_t)p.M * (uint32_t)p.K * kES), win_x = lds_window(p.x, ((uint32_t)(p.T - 1) * (uint32_t)p.x_pitch + (uint32_t)p.K) * kES);
#pragma unroll
    for (int i = 0; kDirect && i < kLoads; ++i) {
        const bool isw = i * kRowStep < BM;
        const uint32_t pitch = isw ? (uint32_t)p.K : (uint32_t)p.x_pitch;
        if (i == 0 || i * kRowStep == BM) off[i] = kES * (kl + (uint32_t)((isw ? m0 : t0) + share_wave * 8 + (lane >> 3)) * pitch);
        else off[i] = off[i - 1] + kES * kRowStep * pitch;
    }
    // (a choice for every row is 24 instructions of a wave at most, 70 ns of every launch)
    if (kDirect && (flags & kRowsWrap)) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const bool isw = i * kRowStep < BM;
            off[i] = row_offset((isw ? m0 : t0 - BM) + i * kRowStep + share_wave * 8 + (lane >> 3), isw ? p.M : p.T, off[i]);
        }
    }
#pragma unroll
    for (int i = 0; !kDirect && i < kLoads; ++i) {
        const int c = threadIdx.x + i * kThreads, row = c / kParts, part = c % kParts;
        if (NN && i < kWLoads) {
            // eight columns of two neighbouring rows of W (K x M), or four of one: see store_transposed
            const int item = threadIdx.x + i / kRowsPer * kThreads, col = item % (BM / kVec) * kVec;
            koff[i] = item / (BM / kVec) * kRowsPer + i % kRowsPer;
            off[i] = kES * ((uint32_t)koff[i] * (uint32_t)p.M + (uint32_t)min(m0 + col, p.M - kVec));
            at[i] = 0;
            continue;
        }
        koff[i] = part * kVec;
        off[i] = row < BM ? kES * (koff[i] + (uint32_t)min(m0 + row, p.M - 1) * (uint32_t)p.K)
                          : kXES * (koff[i] + (uint32_t)min(t0 + row - BM, p.T - 1) * (uint32_t)p.x_pitch);
        at[i] = (part >> 3) * (kRows * 8) + row * 8 + ((part & 7) ^ (row & 7));
    }
    // first of the four columns of the result that a lane holds of tile i
    auto column = [&](int i) {
        const int u = wm * 32 + i * 16 + (lane >> 4) * 4;
        return m0 + (NN && kVec == 8 ? u % (BM / 2) * 2 + u / (BM / 2) * 4 : u);
    };
    const int steps = (p.K + kStep * KS - 1) / (kStep * KS);
    struct Stage {
        u32x4 v[kLoads];
        u32x4 hi[XF32 ? kLoads - kWLoads : 1];  // float32 x: the second half of a part
        f32x4 w[kVec / 4];  // NORM: norm weight of the thread's k (the same in all its parts)
    };
    const rsrc_t rn = make_rsrc(p.norm_w, (uint32_t)p.K * 4u);
    float rs[kLoads - kWLoads];  // rstd of the rows of x the thread stages
    Stage r[D];
    // (a stage beyond the last, and what lies beyond K: zeros)
    const uint32_t lds0 = (uint32_t)reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) void*)&lds[0][0]) + (uint32_t)(ks * (kRows * 8) + share_wave * kWave) * 16u;
    auto fetch = [&](int s, int buf) {
        const int k = s * kStep * KS;
        const bool some = k + kl < p.K;
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            load_to_lds(i * kRowStep < BM ? win_w : win_x, some ? off[i] : kNoRow, (uint32_t)k * kES, lds0 + (uint32_t)(buf * kStage + i * kShareWaves * kWave) * 16u);
    };
    auto load = [&](Stage& st, int s) {
        u32x4(&v)[kLoads] = st.v;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            const int k = s * kStep * KS;
            const uint32_t at_k = (i < kWLoads ? kES : kXES) * (uint32_t)k * (NN && i < kWLoads ? (uint32_t)p.M : 1u);
            const uint32_t at = k + koff[i] < p.K ? off[i] + at_k : 0xffffffe0u;
            v[i] = __builtin_amdgcn_raw_buffer_load_b128(i < kWLoads ? rw : rx, at, 0, 0);
            if constexpr (XF32) {
                if (i >= kWLoads) st.hi[i - kWLoads] = __builtin_amdgcn_raw_buffer_load_b128(rx, at + 16, 0, 0);
            }
        }
        if constexpr (NORM) {
#pragma unroll
            for (int h = 0; h < kVec / 4; ++h)
                st.w[h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rn, 4u * (uint32_t)(s * kStep * KS + koff[0] + 4 * h), 0, 0));
        }
    };
    // W with K as its slow dimension: a word of LDS holds two neighbouring k of a column, or one in float32; a lane writes
    // those of its eight (four) columns.  Column 8*c + 4*h + e goes to row h*BM/2 + 4*c + e (4*c + e to row 4*c + e), so
    // that a lane's four results are neighbours again, and the parts of that row are rotated by row ^ row/4: the words
    // of a wave then meet two to a bank, the operand reads as without.
    auto store_transposed = [&](const Stage& st, int i, int buf) {
        const int item = threadIdx.x + i / kRowsPer * kThreads, c = item % (BM / kVec), kw = item / (BM / kVec);
        uint32_t* const words = reinterpret_cast<uint32_t*>(lds[buf] + kw / 32 * (kRows * 8));
#pragma unroll
        for (int e = 0; e < kVec; ++e) {
            const int u = (e >> 2) * (BM / 2) + 4 * c + (e & 3);
            uint32_t v;
            if constexpr (sizeof(IO) == 2)
                v = __builtin_amdgcn_perm(st.v[i + 1][e >> 1], st.v[i][e >> 1], e & 1 ? 0x07060302u : 0x05040100u);
            else v = st.v[i][e];
            words[u * 32 + ((kw % 32 >> 2) ^ ((u ^ u >> 2) & 7)) * 4 + (kw & 3)] = v;
        }
    };
    auto store = [&](const Stage& st, int buf) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            u32x4 v = st.v[i];
            if (NN && i < kWLoads) {
                if (i % kRowsPer == 0) store_transposed(st, i, buf);
                continue;
            }
            if constexpr (XF32) {
                if (i >= kWLoads) v = Ops::scale_f32(v, st.hi[i - kWLoads], rs[i - kWLoads], st.w);
            } else if constexpr (NORM) {
                if (i >= kWLoads) v = Ops::scale(v, rs[i - kWLoads], st.w);
            }
            lds[buf][at[i]] = v;
        }
    };
    f32x4 acc[2][2 * RT] = {};  // [rows of W][steps]
    const int fr = lane & 15, fq = lane >> 4;
    auto compute = [&](int buf) {
        const u32x4* base = lds[buf] + ks * (kRows * 8);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
            const int part = (kk * 4 + fq) ^ (fr & 7);  // of x, and of W unless it is transposed
            u32x4 a[2], b[2 * RT];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int u = wm * 32 + i * 16 + fr;
                a[i] = base[u * 8 + (NN ? (kk * 4 + fq) ^ ((u ^ u >> 2) & 7) : part)];
            }
#pragma unroll
            for (int j = 0; j < 2 * RT; ++j) b[j] = base[(BM + (wt * RT * 2 + j) * 16 + fr) * 8 + part];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2 * RT; ++j) Ops::mma(a[i], b[j], acc[i][j]);
        }
    };
    // step of the lane's results of tile j
    auto step = [&](int j) { return t0 + (wt * RT * 2 + j) * 16 + fr; };
    float factor[2 * RT];
    if constexpr (XMODE == kFactor) {
        // Requested in front of the stages, so that their sum is in no one's way: the four lanes of a step share its partial sums, eight
        // each at a time (a width of 1024).
        constexpr int kSome = 8;
        const rsrc_t rq = make_rsrc(p.ssq, (uint32_t)p.in_parts * (uint32_t)p.T * 4u);
#pragma unroll
        for (int j = 0; j < 2 * RT; ++j) factor[j] = 0.0f;
        int q0 = 0;
        auto request = [&](float(&v)[2 * RT][kSome]) {
#pragma unroll
            for (int j = 0; j < 2 * RT; ++j)
#pragma unroll
                for (int i = 0; i < kSome; ++i) {
                    const int q = q0 + 4 * i + fq;
                    const uint32_t at = q < p.in_parts ? ((uint32_t)q * (uint32_t)p.T + (uint32_t)min(step(j), p.T - 1)) * 4u : 0xffffffe0u;
                    v[j][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rq, at, 0, 0));
                }
        };
        auto sum = [&](const float(&v)[2 * RT][kSome]) {
#pragma unroll
            for (int j = 0; j < 2 * RT; ++j)
#pragma unroll
                for (int i = 0; i < kSome; ++i) factor[j] += v[j][i];
        };
        float v[2 * RT][kSome];
        request(v);
        fetch(0, 0);
        fetch(1, 1);
        sum(v);
        for (q0 = 4 * kSome; q0 < p.in_parts; q0 += 4 * kSome) {
            request(v);
            sum(v);
        }
#pragma unroll
        for (int j = 0; j < 2 * RT; ++j) {
            factor[j] += __shfl_xor(factor[j], 16);
            factor[j] += __shfl_xor(factor[j], 32);
            factor[j] = __builtin_amdgcn_rsqf(factor[j] * p.inv_d + p.eps);
        }
    } else if constexpr (kDirect) {
        fetch(0, 0);
        fetch(1, 1);
    } else {
#pragma unroll
        for (int i = 0; i < D; ++i) load(r[i], i);
    }
    if constexpr (NORM) {
        // The eight lanes of a row share its partial sums, four each requested together (up to a width of 1024 all of them: one
        // after the other they were three latencies in front of the product at width 768: 128 steps 38.9 -> 37.7 us a layer).
        constexpr int kRowsOf = kLoads - kWLoads, kSome = 4;
        float s[kRowsOf] = {};
        for (int q0 = 0; q0 < p.in_parts; q0 += 8 * kSome) {
            float v[kRowsOf][kSome];
#pragma unroll
            for (int i = 0; i < kRowsOf; ++i)
#pragma unroll
                for (int j = 0; j < kSome; ++j) {
                    const int t = min(t0 + (int)(threadIdx.x + (i + kWLoads) * kThreads) / kParts - BM, p.T - 1), q = q0 + (int)(threadIdx.x % 8) + 8 * j;
                    v[i][j] = p.ssq[(int64_t)min(q, p.in_parts - 1) * p.T + t];
                }
#pragma unroll
            for (int i = 0; i < kRowsOf; ++i)
#pragma unroll
                for (int j = 0; j < kSome; ++j) s[i] += q0 + (int)(threadIdx.x % 8) + 8 * j < p.in_parts ? v[i][j] : 0.0f;
        }
#pragma unroll
        for (int i = 0; i < kRowsOf; ++i) {
            s[i] += __shfl_xor(s[i], 1);
            s[i] += __shfl_xor(s[i], 2);
            s[i] += __shfl_xor(s[i], 4);
            rs[i] = __builtin_amdgcn_rsqf(s[i] * p.inv_d + p.eps);
        }
    }
    if constexpr (kDirect) {
        // A stage's loads are in flight while the two before it are multiplied.  Its wave waits for its own, the barrier for all waves', and
        // for the reads of the buffer that is filled next.
        auto ready = [&] { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kLoads) : "memory"); };
        int s0 = 0;
        for (; s0 + kBuffers <= steps; s0 += kBuffers) {
#pragma unroll
            for (int i = 0; i < kBuffers; ++i) {
                ready();
                fetch(s0 + i + 2, (i + 2) % kBuffers);
                compute(i);
            }
        }
#pragma unroll
        for (int i = 0; i < kBuffers - 1; ++i) {
            if (s0 + i >= steps) break;
            ready();
            fetch(s0 + i + 2, (i + 2) % kBuffers);
            compute(i);
        }
        if constexpr (KS > 1) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    } else {
        store(r[0], 0);
        load(r[0], D);
        __syncthreads();
        // (whole groups of D stages without a branch, so that every wait is for the one stage it needs; loads and
        // stores beyond the last stage are of zeros)
        int s0 = 0;
        for (; s0 + D <= steps; s0 += D) {
#pragma unroll
            for (int i = 0; i < D; ++i) {
                store(r[(i + 1) % D], (i + 1) & 1);
                load(r[(i + 1) % D], s0 + i + 1 + D);
                compute(i & 1);
                __syncthreads();
            }
        }
#pragma unroll
        for (int i = 0; i < D - 1; ++i) {
            if (s0 + i >= steps) break;
            store(r[(i + 1) % D], (i + 1) & 1);
            compute(i & 1);
            __syncthreads();
        }
    }
    // The lane's part of the residual and the weights of its scaled rows, requested at once and before the shares of K are added (one memory latency and
    // not four; what lies beyond T or M is read from within and not used).
    f32x4 res[2][2 * RT] = {}, next[2] = {};
    if (p.y_scaled && ks == 0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) next[i] = *reinterpret_cast<const f32x4*>(p.y_weight + min(column(i), p.M - 4));
    }
    if (p.residual && ks == 0) {
        typename Ops::Out narrow[2][2 * RT];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2 * RT; ++j) {
                const int64_t o = (int64_t)min(step(j), p.T - 1) * p.y_pitch + min(column(i), p.M - 4);
                if (flags & kResidualF32) res[i][j] = *reinterpret_cast<const f32x4*>(static_cast<const float*>(p.residual) + o);
                else narrow[i][j] = *reinterpret_cast<const typename Ops::Out*>(static_cast<const IO*>(p.residual) + o);
            }
        if (!(flags & kResidualF32)) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2 * RT; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) res[i][j][e] = Ops::get(narrow[i][j], e);
        }
    }
    constexpr int kTiles = 4 * RT;
    if constexpr (KS > 1) {
        static_assert(kThreads / kWave * kTiles * kWave <= kBuffers * kStage, "the shares of K use the stages' memory");
        // (the stages are done with: the last barrier)
        f32x4* part = reinterpret_cast<f32x4*>(&lds[0][0]);
        if (ks > 0) {
#pragma unroll
            for (int i = 0; i < kTiles; ++i) part[(wave * kTiles + i) * kWave + lane] = acc[i / (2 * RT)][i % (2 * RT)];
        }
        __syncthreads();
        if (ks > 0) return;
#pragma unroll
        for (int q = 1; q < KS; ++q)
#pragma unroll
            for (int i = 0; i < kTiles; ++i) acc[i / (2 * RT)][i % (2 * RT)] += part[((wave + q) * kTiles + i) * kWave + lane];
    }
    float ss[2 * RT] = {};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int m = column(i);
        if (m >= p.M) continue;
        typename Ops::Out bias = {};
        if (p.bias) bias = *reinterpret_cast<const typename Ops::Out*>(static_cast<const IO*>(p.bias) + m);
#pragma unroll
        for (int j = 0; j < 2 * RT; ++j) {
            const int t = step(j);
            if (t >= p.T) continue;
            const int64_t o = (int64_t)t * p.y_pitch + m;
            // (a factor of zero: squares beyond float32, and the sum may be an infinity; a normalised row is zeros)
            if constexpr (XMODE == kFactor) acc[i][j] = factor[j] == 0.0f ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[i][j] * factor[j];
            f32x4 f;
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = acc[i][j][e] + Ops::get(bias, e);
            if (flags & kAccumulate) f += res[i][j];
            if (sizeof(IO) == 4 || (flags & kYF32)) {
                if (p.residual && !(flags & kAccumulate)) f += res[i][j];
                *reinterpret_cast<f32x4*>(static_cast<float*>(p.y) + o) = f;
            } else {
                typename Ops::Out v;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    Ops::set(v, e, f[e]);
                    if (p.residual && !(flags & kAccumulate)) Ops::set(v, e, Ops::get(v, e) + res[i][j][e]);
                    f[e] = Ops::get(v, e);
                }
                *reinterpret_cast<typename Ops::Out*>(static_cast<IO*>(p.y) + o) = v;
            }
            if (p.y_scaled) {
                typename Ops::Out v;
#pragma unroll
                for (int e = 0; e < 4; ++e) Ops::set(v, e, f[e] * next[i][e]);
                *reinterpret_cast<typename Ops::Out*>(static_cast<IO*>(p.y_scaled) + (int64_t)t * p.M + m) = v;
            }
            if (p.ssq_out) {
#pragma unroll
                for (int e = 0; e < 4; ++e) ss[j] = __builtin_fmaf(f[e], f[e], ss[j]) + (f[e] - f[e]);  // (NaN with an infinity)
            }
        }
    }
    if (p.ssq_out) {
#pragma unroll
        for (int j = 0; j < 2 * RT; ++j) {
            const int t = step(j), q = m0 / 32 + wm;
            float s = ss[j];
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (fq == 0 && t < p.T && q * 32 < p.M) p.ssq_out[(int64_t)q * p.T + t] = s;
        }
    }
}

// What a call asks for beside the sizes.
struct LinearForm {
    bool nn, x_f32, factor;
};
template <typename IO, int BT, int BM, int KS, int RT = 1>
static int launch_linear(LinearParams p, const LinearForm& f, hipStream_t st) {
    const int nt = (p.T + BT - 1) / BT, nm = (p.M + BM - 1) / BM, per = (nt * nm + 7) / 8;
    const bool by_steps = (p.flags & kXLarger) && nt * nm >= 512;
    if (by_steps) p.flags |= kBySteps;
    if (rows_wrap(p.T, BT, p.x_pitch, sizeof(IO)) || rows_wrap(p.M, BM, p.K, sizeof(IO))) p.flags |= kRowsWrap;
    p.tiles = nt * nm;
    p.tiles_per_xcd = per;
    p.inner = by_steps ? nm : nt;
    p.inner_inv = p.tiles < 1 << 16 && p.inner > 1 ? (uint32_t)((((uint64_t)1 << 32) + p.inner - 1) / p.inner) : 0;
    const dim3 grid((unsigned)per * 8), block(linear_threads(BT, BM, KS, RT));
    auto run = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, p); };
    if (f.nn) run(linear_kernel<IO, BT, BM, KS, RT, 2, kPlainX, true>);
    else if (!p.ssq) run(linear_kernel<IO, BT, BM, KS, RT, 2, kPlainX, false>);
    else if (f.factor) run(linear_kernel<IO, BT, BM, KS, RT, 2, kFactor, false>);
    else if (sizeof(IO) == 2 && f.x_f32) run(linear_kernel<IO, BT, BM, KS, RT, 2, sizeof(IO) == 2 ? kNormXF32 : kNormX, false>);
    else run(linear_kernel<IO, BT, BM, KS, RT, 2, kNormX, false>);
    return check_launch();
}

// The largest tile that gives most CUs one (a tile's traffic per product falls with its size), smaller ones
// with K split over more waves (512 steps of a layer of width 768: in_proj 9.0 us with 64 x 128, 9.9 with 64 x
// 64, 15 with 32 x 32; out_proj 7.9 us with 64 x 32 on eight waves, 10.8 with 64 x 64; x_proj 6.7 and 10.2 us).
// Where those are more than one round and tiles twice as long are not, these (bfloat16, in_proj: 1024 steps of width 768
// 12.8 us for 14.4, 1400 of 512 10.7 for 11.7, 2048 of 400 11.0 for 12.1; in one round the small ones: 700 of 640 9.1 for 11.4; with
// more than one round of either there is no difference).  Of the plain products in training it makes no difference (four layers of
// 1400 steps of width 512, forward and backward, 862 us of kernels and 863), and they take them by the same rule.
// Tiles of 32 x 32 with K in four shares fill a CU's LDS: where they are more than a round of the CUs, 64 x 32 at any number (out_proj, 400 steps of width
// 640: 10.3 us in 260 tiles of 32 x 32, 7.5 in 140; 9.3 with two stages in LDS, of which a CU has two.  700 of 392 9.8 and 6.7, x_proj, 4950
// of 128, 7.2 and 4.7; float32 0.73 to 0.83 of the time, input gradients 0.74 to 0.94).
template <typename IO>
static int dispatch_linear(const LinearParams& p, const LinearForm& f, hipStream_t st) {
    auto tiles = [&](int bt, int bm) { return (int64_t)((p.T + bt - 1) / bt) * ((p.M + bm - 1) / bm); };
    constexpr int kFull = 160;
    if constexpr (sizeof(IO) == 2) {
        constexpr int kCUs = 256;
        if (!f.nn && tiles(64, 128) > kCUs && tiles(128, 128) <= kCUs) return launch_linear<IO, 128, 128, 1, 2>(p, f, st);
    }
    if (tiles(64, 128) >= kFull) return launch_linear<IO, 64, 128, 1>(p, f, st);
    if (p.K <= 128) return launch_linear<IO, 64, 64, 1>(p, f, st);  // (one or two stages: nothing to split)
    const bool one = p.K >= 1024;
    if (tiles(64, 64) >= kFull) return one && tiles(64, 64) <= 256 ? launch_linear<IO, 64, 64, 2>(p, f, st) : launch_linear<IO, 64, 64, 1>(p, f, st);
    if (tiles(64, 32) >= kFull || tiles(32, 32) > 256) return one && tiles(64, 32) <= 256 ? launch_linear<IO, 64, 32, 4>(p, f, st) : launch_linear<IO, 64, 32, 2>(p, f, st);
    return launch_linear<IO, 32, 32, 4>(p, f, st);
}

}  // namespace mpa

using namespace mpa;

extern "C" int mpa_linear_run(const mpa_linear* s, void* stream) {
    if (s && s->x_ssq && !s->norm_weight) return MPA_ERR_NULL_POINTER;
    return mpa_linear_run_scaled(s, nullptr, nullptr, stream);
}

extern "C" int mpa_linear_run_scaled(const mpa_linear* s, const float* y_weight, void* y_scaled, void* stream) {
    if (!s || !s->x || !s->weight || !s->y || !y_weight != !y_scaled) return MPA_ERR_NULL_POINTER;
    const int wide = MPA_LINEAR_X_F32 | MPA_LINEAR_Y_F32 | MPA_LINEAR_RESIDUAL_F32, io = s->io_dtype & ~wide;
    if (io != MPA_F32 && io != MPA_BF16) return MPA_ERR_BAD_DTYPE;
    const bool f32 = io == MPA_F32;
    const bool x_f32 = !f32 && (s->io_dtype & MPA_LINEAR_X_F32), y_f32 = f32 || (s->io_dtype & MPA_LINEAR_Y_F32);
    const bool residual_f32 = f32 || (s->io_dtype & MPA_LINEAR_RESIDUAL_F32);
    const bool factor = s->x_ssq && !s->norm_weight;
    if (x_f32 && (!s->x_ssq || factor)) return MPA_ERR_BAD_DTYPE;
    const int vec = f32 ? 4 : 8;
    if (s->weight_kxm && (s->x_ssq || s->y_ssq || y_scaled || s->M % vec)) return MPA_ERR_BAD_SHAPE;
    // (x and the weight are addressed with 32-bit byte offsets)
    if (s->T <= 0 || s->M <= 0 || s->K <= 0 || s->K % vec || s->x_pitch % vec || s->M % 4 || s->y_pitch % 4 || s->x_pitch < s->K ||
        s->y_pitch < s->M || s->T > 1 << 24 || s->M > 1 << 24 || s->K > 1 << 24 || s->T * s->x_pitch >= (int64_t)1 << 29 ||
        s->M * s->K >= (int64_t)1 << 29 || (s->x_ssq && (s->ssq_parts <= 0 || s->ssq_parts > 1 << 20)) ||
        (factor && s->ssq_parts * s->T >= (int64_t)1 << 29))
        return MPA_ERR_BAD_SHAPE;
    if (!aligned_to(s->x, 16) || !aligned_to(s->weight, 16) || !aligned_to(s->bias, f32 ? 16 : 8) || !aligned_to(s->y, y_f32 ? 16 : 8) ||
        !aligned_to(s->residual, residual_f32 ? 16 : 8) || !aligned_to(s->norm_weight, 16) || !aligned_to(s->x_ssq, 4) || !aligned_to(s->y_ssq, 4) ||
        !aligned_to(y_weight, 16) || !aligned_to(y_scaled, f32 ? 16 : 8))
        return MPA_ERR_MISALIGNED;
    LinearParams p{};
    p.x = s->x; p.w = s->weight; p.bias = s->bias;
    p.x_pitch = s->x_pitch; p.y_pitch = s->y_pitch;
    p.T = (int)s->T; p.M = (int)s->M; p.K = (int)s->K;
    p.y = s->y;
    p.ssq = s->x_ssq; p.in_parts = (int)s->ssq_parts;
    p.inv_d = 1.0f / (float)s->K; p.eps = s->eps; p.norm_w = s->norm_weight;
    p.residual = s->residual;
    p.ssq_out = s->y_ssq;
    p.y_weight = y_weight; p.y_scaled = y_scaled;
    p.flags = (s->accumulate ? kAccumulate : 0) | (y_f32 ? kYF32 : 0) | (residual_f32 ? kResidualF32 : 0) |
              (s->T * (x_f32 || f32 ? 4 : 2) > s->M * (f32 ? 4 : 2) ? kXLarger : 0);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const LinearForm form{s->weight_kxm != 0, x_f32, factor};
    return f32 ? dispatch_linear<float>(p, form, st) : dispatch_linear<bf16_t>(p, form, st);
}
