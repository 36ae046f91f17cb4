// One decode step of a whole residual layer (norm, in_proj, convolution, x_proj, dt_proj, state
// update, gate, out_proj) in three or four launches, for gfx950.
//
// At decode batch sizes every operation of a layer is a pass over a weight matrix of a few MB or
// over the recurrent state: 2-3 us of memory time next to ~1.6 us of launch time per graph node.
// Run as library GEMMs between element-wise kernels, a layer is seven or more launches of 4-7 us
// (24 layers at width 768, bfloat16: 1.00 ms for one sequence, 1.24 ms for 64).  Here the
// element-wise work rides in the products:
//
//   decode_in_kernel   RMSNorm, in_proj, and for the x half the convolution over the rolling
//                      window with bias and silu
//   decode_xproj_kernel  x_proj (float32 partial sums over ranges of K); in a small call decode_in does it
//   decode_ssm_kernel  dt_proj, softplus, state update, readout, gate
//   decode_out_kernel  out_proj, residual add, and what the next layer's norm needs
//
// decode_out writes the new residual row and, for the next layer, that row times its norm weight and
// the row's partial sums of squares, so only the first layer's in_proj has to form them; a row's
// rstd is a factor of the finished product.
//
// The products are `W (rows x K) . X^T (K x batch)` with batch <= MPA_DECODE_MAX_BATCH: a workgroup
// owns MT tiles of 16 rows of W and NT tiles of 16 sequences, its waves split K, and the partial tiles meet
// in LDS.  A contraction may be summed in any order, so a wave takes 128 bytes of each of its rows at
// a time: eight lanes load one row's piece (lanes in different rows, as the MFMA operand has them, cost
// an address per lane: in_proj of 64 sequences at width 2560, float32, took 95 us that way, 55 us by pieces), and a
// 2 KB exchange through the wave's own LDS turns rows into operands.  Activations that these kernels
// write for each other are stored in operand order.  The unused columns of a batch below 16 cost nothing that
// matters: the kernels wait for the weights, not for the matrix pipe.  What the epilogue needs is
// requested before the product, so that its latency is not added to the weights'.
#include "common.h"

#include <type_traits>

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// What a lane holds of 32 k of a row (or a sequence): eight consecutive ones.
template <typename IO>
struct Frag;
template <>
struct Frag<bf16_t> {
    static constexpr int kVec = 8, kOps = 2;  // of a 16-byte access; operands of a piece of 128 bytes
    typedef u32x4 Op;
    static __device__ __forceinline__ void unpack(const u32x4& v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __uint_as_float(v[i] << 16);
            f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ Op pack(const float (&f)[8]) {
        bf16x8 r;
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = static_cast<__bf16>(f[i]);
        return __builtin_bit_cast(u32x4, r);
    }
    static __device__ __forceinline__ Op from(const u32x4 (&v)[1]) { return v[0]; }
    template <int NT>
    static __device__ __forceinline__ void mma(const Op& a, const Op (&b)[NT], f32x4 (&c)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
            c[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                           __builtin_bit_cast(bf16x8, b[t]), c[t], 0, 0, 0);
    }
};
template <>
struct Frag<float> {
    static constexpr int kVec = 4, kOps = 1;
    struct Op {
        u32x4 half[2];
    };
    static __device__ __forceinline__ void unpack(const u32x4& v, float (&f)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(v[i]);
    }
    static __device__ __forceinline__ Op pack(const float (&f)[8]) {
        Op r;
#pragma unroll
        for (int i = 0; i < 8; ++i) r.half[i >> 2][i & 3] = __float_as_uint(f[i]);
        return r;
    }
    static __device__ __forceinline__ Op from(const u32x4 (&v)[2]) { return Op{{v[0], v[1]}}; }
    // eight products of one k per lane group: together the 32 k that the four lane groups hold (the
    // tiles in the inner loop: products of one tile depend on each other).  As three bfloat16 parts and six 16-bit products, a third of
    // the matrix unit's time, it was 0 to 8 % slower: cutting the operands is vector work, and the loads are what is waited for.
    template <int NT>
    static __device__ __forceinline__ void mma(const Op& a, const Op (&b)[NT], f32x4 (&c)[NT]) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a.half[i >> 2][i & 3]), __uint_as_float(b[t].half[i >> 2][i & 3]),
                                                            c[t], 0, 0, 0);
    }
};

__device__ __forceinline__ u32x4 ld16(const void* p) { return *static_cast<const u32x4*>(p); }

// Loads that may not be wanted are buffer loads at an offset beyond the window, which read zero: a load within a branch makes the
// compiler wait for all loads in flight at the next use of any (the product loop then had one memory latency for every
// piece of a wave; 64 sequences through in_proj at width 2560, float32, 56 us).
__device__ __forceinline__ uint32_t wanted(uint32_t at, bool ok) {
    asm("" : "+v"(at));  // (formed either way: or the choice becomes a branch around its arithmetic, and around the load)
    return ok ? at : 0xffffffe0u;
}
__device__ __forceinline__ u32x4 ld16(rsrc_t r, uint32_t at, bool ok) { return __builtin_amdgcn_raw_buffer_load_b128(r, wanted(at, ok), 0, 0); }
__device__ __forceinline__ float ld_f32(rsrc_t r, uint32_t at, bool ok) {
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, wanted(at, ok), 0, 0));
}
template <typename IO>
__device__ __forceinline__ IO ld_io(rsrc_t r, uint32_t i, bool ok) {
    const uint32_t at = wanted(i * (uint32_t)sizeof(IO), ok);
    if constexpr (sizeof(IO) == 4) return __builtin_bit_cast(IO, __builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0));
    else return __builtin_bit_cast(IO, __builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0));
}
// window of n elements, none without a pointer
__device__ __forceinline__ rsrc_t window(const void* p, int64_t n, int es) { return make_rsrc(p, p ? (uint32_t)(n * es) : 0u); }

// Operand order of activations (batch x K): tiles of 16 sequences x 32 values of k, lane (sequence % 16) + 16 * (k / 8 % 4)
// holding eight consecutive k (float32: in two halves, 1 KB of lanes each).
template <typename IO>
__device__ __forceinline__ int64_t frag_at(int b, int k, int K) {
    constexpr int kVec = Frag<IO>::kVec;
    const int64_t tile = (int64_t)(b >> 4) * ((K + 31) / 32) + k / 32;
    return (tile * (8 / kVec) + k % 8 / kVec) * (64 * kVec) + ((b & 15) + 16 * (k % 32 / 8)) * kVec + k % kVec;
}
__host__ __device__ inline int64_t frag_bytes(int64_t batch, int64_t K, int es) { return (batch + 15) / 16 * ((K + 31) / 32) * 512 * es; }
// One value of an activation; the last four of a float32 row whose eight are not whole bring the zeros after them.
template <typename IO>
__device__ __forceinline__ void frag_store(void* base, int b, int k, int K, IO v) {
    IO* const to = static_cast<IO*>(base) + frag_at<IO>(b, k, K);
    *to = v;
    if constexpr (sizeof(IO) == 4) {
        if (k % 8 < 4 && k + 4 >= K) to[256] = 0.0f;
    }
}
template <typename IO>
__device__ __forceinline__ float frag_load(const void* base, int b, int k, int K) {
    return load_as_float<IO>(base, frag_at<IO>(b, k, K));
}
// Activations in operand order.
template <typename IO, int NT>
struct FragAct {
    static constexpr int kLoads = 8 / Frag<IO>::kVec;
    struct Raw {
        u32x4 x[kLoads];
    };
    rsrc_t r;
    uint32_t at[NT];
    bool live[NT];
    __device__ __forceinline__ void setup(const void* base, int b0, int batch, int K, int lane) {
        r = make_rsrc(base, (uint32_t)frag_bytes(batch, K, sizeof(IO)));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            at[t] = (uint32_t)(sizeof(IO) * frag_at<IO>(b0 + t * 16, 0, K)) + lane * 16;
            live[t] = b0 + t * 16 + (lane & 15) < batch;  // (one sequence then reads a sixteenth of its tile)
        }
    }
    __device__ __forceinline__ void request(Raw& v, int t, int chunk, int, int, bool ok) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) v.x[i] = ld16(r, at[t] + (uint32_t)(chunk * kLoads + i) * 1024u, ok && live[t]);
    }
    __device__ __forceinline__ typename Frag<IO>::Op operand(const Raw& v, int) { return Frag<IO>::from(v.x); }
};

// Rows of X as the caller has them (zeros for a column without a sequence), as they are or (NORM) times
// the norm weight, with the sums of squares.
template <typename IO, int NT, bool NORM>
struct RowAct {
    static constexpr int kVec = Frag<IO>::kVec, kLoads = 8 / kVec;
    struct Raw {
        u32x4 x[kLoads];
        f32x4 w[NORM ? 2 : 1];
    };
    rsrc_t r, rw;
    uint32_t at[NT];
    bool live[NT], gain;
    float ss[NT];
    __device__ __forceinline__ void setup(const void* base, const float* w, int b0, int batch, int K, int lane) {
        r = window(base, (int64_t)batch * K, sizeof(IO));
        rw = window(w, K, 4);
        gain = w != nullptr;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int b = b0 + t * 16 + (lane & 15);
            live[t] = b < batch;
            at[t] = (uint32_t)b * (uint32_t)K * (uint32_t)sizeof(IO);
            ss[t] = 0.0f;
        }
    }
    __device__ __forceinline__ void request(Raw& v, int t, int, int k, int K, bool ok) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) v.x[i] = ld16(r, at[t] + (uint32_t)(k + i * kVec) * (uint32_t)sizeof(IO), ok && live[t] && k + i * kVec < K);
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < 2; ++i) v.w[i] = __builtin_bit_cast(f32x4, ld16(rw, (uint32_t)(k + 4 * i) * 4u, k + 4 * i < K));
        }
    }
    __device__ __forceinline__ typename Frag<IO>::Op operand(const Raw& v, int t) {
        if constexpr (!NORM) return Frag<IO>::from(v.x);
        float f[8];
#pragma unroll
        for (int i = 0; i < kLoads; ++i) {
            float u[kVec];
            Frag<IO>::unpack(v.x[i], u);
#pragma unroll
            for (int j = 0; j < kVec; ++j) f[i * kVec + j] = u[j];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            ss[t] = __builtin_fmaf(f[i], f[i], ss[t]);
            if (gain) f[i] *= v.w[i >> 2][i & 3];
        }
        return Frag<IO>::pack(f);
    }
};

// What a wave of decode_product keeps in LDS: two slots of MT x 16 rows x 128 bytes for the exchange, then
// its MT x NT partial tiles (lane l holds rows 4*(l/16) .. +3 of column l%16 of each).
template <int MT, int NT>
struct alignas(16) WaveLds {
    static constexpr int kMT = MT;
    float v[MT * (NT > 4 ? 256 * NT : 1024)];
};
template <int NW, typename L>
__device__ __forceinline__ float tile_sum(const L (&lds)[NW], int row, int b) {
    const int at = ((b >> 4) * L::kMT + (row >> 4)) * 256 + ((row % 16 >> 2) * 16 + (b & 15)) * 4 + (row & 3);
    float s = lds[0].v[at];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += lds[w].v[at];
    return s;
}

// Rows n0 .. n0+16*MT-1 of `W . x^T` for NT batch tiles, over the 128-byte pieces first + wave, + NW, ...
// below `last` of the rows of W; the wave leaves its partial tiles in its LDS.  U pieces are in flight (`more` issues the caller's own
// loads behind them), each with its activations: loads return in the order they were issued, so
// activations requested later than weights of pieces further on would wait for those as well.
template <typename IO, int NW, int U, int MT, int NT, typename ACT, typename MORE>
__device__ __forceinline__ void decode_product(WaveLds<MT, NT>& lds, const void* W, int rows, int K, int n0, int first, int last, int wave,
                                               int lane, ACT& act, MORE&& more) {
    constexpr int kVec = Frag<IO>::kVec, kES = sizeof(IO);
    char* const slot = reinterpret_cast<char*>(lds.v);
    // lane -> 16 bytes of row 8*i + lane/8: the piece's eight 16-byte parts are stored rotated by the row
    // (part ^ (row & 7)), so that the operand reads, one row per lane, fall on different banks
    const uint32_t part = ((lane & 7) ^ (lane >> 3)) * 16u;
    const int left = rows - n0;
    const rsrc_t rw = make_rsrc(static_cast<const IO*>(W) + (int64_t)n0 * K, (uint32_t)min(left, 16 * MT) * (uint32_t)K * kES);
    uint32_t row[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) row[i] = (uint32_t)min(8 * i + (lane >> 3), left - 1) * (uint32_t)K * kES + part;
    constexpr int kOps = Frag<IO>::kOps, kReads = 2 / kOps;  // operands of a piece; 16-byte parts of one
    const int kl = 8 * (lane >> 4);
    int frag[kOps][kReads];
#pragma unroll
    for (int h = 0; h < kOps; ++h)
#pragma unroll
        for (int i = 0; i < kReads; ++i) frag[h][i] = (lane & 15) * 128 + ((((lane >> 4) * kReads + i + 4 * h) ^ (lane & 7)) << 4);
    const int count = first + wave < last ? (last - first - wave + NW - 1) / NW : 0;  // pieces of this wave
    const int k_end = min(last * 8 * kVec, K);

    struct Piece {
        u32x4 w[2 * MT];
        typename ACT::Raw a[NT][kOps];
    };
    Piece r[U];
    auto request = [&](Piece& v, int s) {
        const int piece = first + wave + s * NW;
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) v.w[i] = ld16(rw, row[i] + (uint32_t)piece * 128u, (uint32_t)piece * 128u + part < (uint32_t)k_end * kES);
#pragma unroll
        for (int h = 0; h < kOps; ++h) {
            const int chunk = kOps * piece + h, k = chunk * 32 + kl;
#pragma unroll
            for (int t = 0; t < NT; ++t) act.request(v.a[t][h], t, chunk, k, K, k < k_end);
        }
    };
    f32x4 acc[MT][NT] = {};
    auto multiply = [&](const Piece& v, int u) {
        char* const at = slot + (u & 1) * (2048 * MT);
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) *reinterpret_cast<u32x4*>(at + i * 1024 + lane * 16) = v.w[i];
#pragma unroll
        for (int h = 0; h < kOps; ++h) {
            typename Frag<IO>::Op x[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) x[t] = act.operand(v.a[t][h], t);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                u32x4 raw[kReads];
#pragma unroll
                for (int i = 0; i < kReads; ++i) raw[i] = *reinterpret_cast<const u32x4*>(at + m * 2048 + frag[h][i]);
                Frag<IO>::mma(Frag<IO>::from(raw), x, acc[m]);
            }
        }
    };
#pragma unroll
    for (int u = 0; u < U; ++u) request(r[u], u);
    more();
    // (whole groups without a branch; what is requested beyond the last piece are zeros)
    int s = 0;
    for (; s + U <= count; s += U) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            multiply(r[u], u);
            request(r[u], s + u + U);
        }
    }
#pragma unroll
    for (int u = 0; u < U - 1; ++u) {
        if (s + u >= count) break;  // uniform over the wave
        multiply(r[u], u);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&lds.v[(t * MT + m) * 256 + 4 * lane]) = acc[m][t];
}

struct DecodeParams {
    int batch, d, ED, N, R, K;  // K: convolution taps
    float eps;
    int splits, ssq_tiles;  // partial sums of x_proj; row tiles of d (partial sums of squares)
    const void* x;
    const void* xw;        // x times the norm weight in operand order, or null: formed from x
    const float* ssq;      // [ssq_tiles][batch] partial sums of squares of the rows of x, with xw
    const float* norm_w;
    const void *in_w, *in_b;
    const float *conv_w, *conv_b;
    const void *xp_w, *dt_w;
    const float *dt_b, *A, *D;
    const void *out_w, *out_b;
    const float* h_in;
    float* h_out;
    const void* win_in;
    void* win_out;
    void *xs, *z, *g;  // in the workspace: convolved x, gate (batch, ED), gated readout; xs and g in operand order
    float* dbc;        // [splits][batch][R + 2N]
    void* y;
    const float* next_w;  // norm weight of the next layer, with y_w and ssq_out
    void* y_w;
    float* ssq_out;
};

// What decode_in_kernel does with x: as it is, normalised here, or normalised by the kernel before.
enum { kInPlain, kInNorm, kInReady };

// grid: (row tiles) x (batch tile groups), batch groups of one row tile eight blocks apart: the
// blocks of an XCD (every eighth) then meet the same rows of W again in their own L2.
template <int NT>
__device__ __forceinline__ void decode_tile(int row_tiles, int groups, int& rt, int& bt) {
    const int id = blockIdx.x;
    if (groups == 1) {
        rt = id;
        bt = 0;
        return;
    }
    const int span = 8 * groups, g = id / span, in = id - g * span;
    rt = g * 8 + (in & 7);
    bt = (in >> 3) * NT;
}

// XP: also the workgroup's share of x_proj, its 16 channels' product with all rows of x_proj's weight, as one
// more partial sum of dbc; a thread owns one row and every so many sequences (there are as many threads as rows, or more).
template <typename IO, int MT, int NT, int NW, int U, int MODE, bool XP = false>
__global__ void __launch_bounds__(NW* kWave) decode_in_kernel(const DecodeParams p, int row_tiles, int groups) {
    constexpr int kThreads = NW * kWave, kRows = MT * 16, kAll = NT * 16 * kRows, kOuts = (kAll + kThreads - 1) / kThreads;
    static_assert(!XP || MT == 1, "x_proj by 16 channels");
    __shared__ WaveLds<MT, NT> tile[NW];
    __shared__ float ssq[NW][NT][16];
    __shared__ float xl[XP ? NT * 16 : 1][16];  // convolved x of the tile
    int rt, bt;
    decode_tile<NT>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;  // uniform over the block
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * kRows, b0 = bt * 16, rows = 2 * p.ED;
    const int pieces = (p.d + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    // the epilogue's operands: thread -> outputs (row o % kRows, sequence o / kRows)
    IO win[kOuts][3];
    float cw[kOuts][4], cb[kOuts], ib[kOuts];
    float ss[NT] = {};
    const int P = p.R + 2 * p.N;
    u32x4 xw[XP ? 16 / Frag<IO>::kVec : 1];
    // wave w, lane group q: partial sums of squares 4w + q, 4w + q + 4*NW, ... of column lane % 16, four requested together and the
    // first four ahead of the product
    const rsrc_t rs = window(p.ssq, (int64_t)p.ssq_tiles * p.batch, 4);
    float sq[NT][4];
    auto request_sums = [&](int q0) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int b = b0 + t * 16 + (lane & 15), q = q0 + 4 * (wave + NW * i) + (lane >> 4);
                sq[t][i] = ld_f32(rs, (uint32_t)(q * p.batch + b) * 4u, b < p.batch && q < p.ssq_tiles);
            }
    };
    auto more = [&] {
        if constexpr (XP) {
            // (a part beyond the last channel is read at the row's start and meets zeros)
            const IO* row = static_cast<const IO*>(p.xp_w) + (int64_t)(threadIdx.x % P) * p.ED;
#pragma unroll
            for (int i = 0; i < 16 / Frag<IO>::kVec; ++i) {
                const int k = n0 + i * Frag<IO>::kVec;
                xw[i] = ld16(row + (k < p.ED ? k : 0));
            }
        }
        const rsrc_t rb = window(p.in_b, rows, sizeof(IO)), rwin = window(p.win_in, (int64_t)p.batch * p.ED * (p.K - 1), sizeof(IO)),
                     rcw = window(p.conv_w, (int64_t)p.ED * p.K, 4), rcb = window(p.conv_b, p.ED, 4);
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % kRows, b = b0 + o / kRows;
            const bool some = o < kAll && n < rows && b < p.batch, conv = some && n < p.ED;
            ib[i] = to_float(ld_io<IO>(rb, n, some));
#pragma unroll
            for (int j = 0; j < 3; ++j) win[i][j] = ld_io<IO>(rwin, (uint32_t)(b * p.ED + n) * (uint32_t)(p.K - 1) + j, conv && j < p.K - 1);
#pragma unroll
            for (int j = 0; j < 4; ++j) cw[i][j] = ld_f32(rcw, (uint32_t)(n * p.K + j) * 4u, conv && j < p.K);
            cb[i] = ld_f32(rcb, (uint32_t)n * 4u, conv);
        }
        if constexpr (MODE == kInReady) request_sums(0);
    };
    if constexpr (MODE == kInReady) {
        FragAct<IO, NT> act;
        act.setup(p.xw, b0, p.batch, p.d, lane);
        decode_product<IO, NW, U>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
        for (int q0 = 0;; request_sums(q0)) {
#pragma unroll
            for (int t = 0; t < NT; ++t) ss[t] += (sq[t][0] + sq[t][1]) + (sq[t][2] + sq[t][3]);
            if ((q0 += 16 * NW) >= p.ssq_tiles) break;
        }
    } else {
        RowAct<IO, NT, MODE == kInNorm> act;
        act.setup(p.x, p.norm_w, b0, p.batch, p.d, lane);
        decode_product<IO, NW, U>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
#pragma unroll
        for (int t = 0; t < NT; ++t) ss[t] = act.ss[t];
    }
    if constexpr (MODE != kInPlain) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            float s = ss[t];
            s += __shfl_xor(s, 16);
            s += __shfl_xor(s, 32);
            if (lane < 16) ssq[wave][t][lane] = s;
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOuts; ++i) {
        const int o = threadIdx.x + i * kThreads, row = o % kRows, bl = o / kRows, n = n0 + row, b = b0 + bl;
        if (o >= kAll || n >= rows || b >= p.batch) continue;
        float v = tile_sum(tile, row, bl);
        if constexpr (MODE != kInPlain) {
            float s = ssq[0][bl >> 4][bl & 15];
#pragma unroll
            for (int w = 1; w < NW; ++w) s += ssq[w][bl >> 4][bl & 15];
            v *= __builtin_amdgcn_rsqf(s / (float)p.d + p.eps);
        }
        const IO vr = from_float<IO>(v + ib[i]);
        if (n >= p.ED) {
            static_cast<IO*>(p.z)[(int64_t)b * p.ED + n - p.ED] = vr;
            continue;
        }
        // newest tap first, then the window from its newest input backwards
        const int last = p.K - 2;
        IO* wo = static_cast<IO*>(p.win_out) + ((int64_t)b * p.ED + n) * (p.K - 1);
        float c = cb[i];
#pragma unroll
        for (int j = 3; j >= 0; --j)
            if (j == p.K - 1) c = __builtin_fmaf(cw[i][j], to_float(vr), c);
            else if (j < p.K - 1) c = __builtin_fmaf(cw[i][j], to_float(win[i][j < 3 ? j : 2]), c);
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j <= last) wo[j] = j < last ? win[i][j < 2 ? j + 1 : 2] : vr;
        c *= sigmoid_f(c);
        const IO cr = from_float<IO>(c);
        frag_store<IO>(p.xs, b, n, p.ED, cr);
        if constexpr (XP) xl[bl][row] = to_float(cr);
    }
    if constexpr (XP) {
        if (n0 >= p.ED) return;  // uniform over the block
        if (n0 + 16 > p.ED)
            for (int o = threadIdx.x; o < kAll; o += kThreads)
                if (n0 + o % 16 >= p.ED) xl[o / 16][o % 16] = 0.0f;
        __syncthreads();
        const int G = kThreads / P, g = threadIdx.x / P, nb = min(p.batch - b0, NT * 16);
        if (g >= G) return;
        for (int b = g; b < nb; b += G) {
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < 16 / Frag<IO>::kVec; ++i) {
                float w[Frag<IO>::kVec];
                Frag<IO>::unpack(xw[i], w);
#pragma unroll
                for (int e = 0; e < Frag<IO>::kVec; ++e) s = __builtin_fmaf(w[e], xl[b][i * Frag<IO>::kVec + e], s);
            }
            p.dbc[((int64_t)rt * p.batch + b0 + b) * P + threadIdx.x % P] = s;
        }
    }
}

// Rows of x times the norm weight in operand order, and their sums of squares: what decode_out of a layer before
// would have left.  One workgroup per sequence.
template <typename IO>
__global__ void __launch_bounds__(256) decode_scale_kernel(const DecodeParams p, void* xw, float* ssq) {
    constexpr int kVec = Frag<IO>::kVec;
    __shared__ float part[4];
    const int b = blockIdx.x;
    const IO* row = static_cast<const IO*>(p.x) + (int64_t)b * p.d;
    float ss = 0.0f;
    for (int k = threadIdx.x * 8; k < p.d; k += 256 * 8) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; i += kVec) {  // (zeros beyond d)
            float v[kVec];
            Frag<IO>::unpack(k + i < p.d ? ld16(row + k + i) : u32x4{0, 0, 0, 0}, v);
#pragma unroll
            for (int j = 0; j < kVec; ++j) f[i + j] = v[j];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            ss = __builtin_fmaf(f[i], f[i], ss);
            if (p.norm_w && k + i < p.d) f[i] *= p.norm_w[k + i];
        }
        u32x4* to = reinterpret_cast<u32x4*>(static_cast<IO*>(xw) + frag_at<IO>(b, k, p.d));
        if constexpr (sizeof(IO) == 2) to[0] = Frag<IO>::pack(f);
        else
#pragma unroll
            for (int i = 0; i < 8; ++i) to[64 * (i >> 2)][i & 3] = __float_as_uint(f[i]);
    }
#pragma unroll
    for (int o = 1; o < kWave; o *= 2) ss += __shfl_xor(ss, o);
    if ((threadIdx.x & (kWave - 1)) == 0) part[wave_id()] = ss;
    __syncthreads();
    if (threadIdx.x == 0) ssq[b] = (part[0] + part[1]) + (part[2] + part[3]);
}

template <typename IO, int NW>
__global__ void __launch_bounds__(NW* kWave) decode_xproj_kernel(const DecodeParams p, int row_tiles, int groups) {
    __shared__ WaveLds<1, 1> tile[NW];
    int rt, bt;
    decode_tile<1>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id(), rows = p.R + 2 * p.N;
    const int pieces = (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    const int per = (pieces + gridDim.y - 1) / gridDim.y, first = (int)blockIdx.y * per;
    FragAct<IO, 1> act;
    act.setup(p.xs, bt * 16, p.batch, p.ED, lane);
    decode_product<IO, NW, 2>(tile[wave], p.xp_w, rows, p.ED, rt * 16, first, min(pieces, first + per), wave, lane, act, [] {});
    __syncthreads();
    const int o = threadIdx.x, n = rt * 16 + (o & 15), b = bt * 16 + (o >> 4);
    if (o < 256 && n < rows && b < p.batch) p.dbc[((int64_t)blockIdx.y * p.batch + b) * rows + n] = tile_sum(tile, o & 15, o >> 4);
}

// y = out_proj(g) [+ x]; with next_w also y * next_w and the sums of squares of 16 columns each
template <typename IO, int MT, int NT, int NW, int U, bool RES>
__global__ void __launch_bounds__(NW* kWave) decode_out_kernel(const DecodeParams p, int row_tiles, int groups) {
    constexpr int kThreads = NW * kWave, kRows = MT * 16, kAll = NT * 16 * kRows, kOuts = (kAll + kThreads - 1) / kThreads;
    __shared__ WaveLds<MT, NT> tile[NW];
    int rt, bt;
    decode_tile<NT>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * kRows, b0 = bt * 16;
    float bias[kOuts], xv[kOuts], nw[kOuts];
    auto more = [&] {
        const rsrc_t rb = window(p.out_b, p.d, sizeof(IO)), rx = window(RES ? p.x : nullptr, (int64_t)p.batch * p.d, sizeof(IO)),
                     rn = window(RES ? p.next_w : nullptr, p.d, 4);
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % kRows, b = b0 + o / kRows;
            const bool ok = o < kAll && n < p.d && b < p.batch;
            bias[i] = to_float(ld_io<IO>(rb, n, ok));
            xv[i] = to_float(ld_io<IO>(rx, (uint32_t)(b * p.d + n), ok));
            nw[i] = ld_f32(rn, (uint32_t)n * 4u, ok);
        }
    };
    FragAct<IO, NT> act;
    act.setup(p.g, b0, p.batch, p.ED, lane);
    decode_product<IO, NW, U>(tile[wave], p.out_w, p.d, p.ED, n0, 0, (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec), wave,
                                      lane, act, more);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOuts; ++i) {
        const int o = threadIdx.x + i * kThreads, row = o % kRows, bl = o / kRows, n = n0 + row, b = b0 + bl;
        if (o >= kAll) break;  // uniform over a wave
        const bool ok = n < p.d && b < p.batch;
        const int64_t at = (int64_t)b * p.d + n;
        IO v = from_float<IO>(tile_sum(tile, row, bl) + bias[i]);
        if constexpr (RES) {
            v = from_float<IO>(to_float(v) + xv[i]);
            if (p.next_w) {
                const float f = ok ? to_float(v) : 0.0f;
                float s = f * f;
                s += __shfl_xor(s, 1);
                s += __shfl_xor(s, 2);
                s += __shfl_xor(s, 4);
                s += __shfl_xor(s, 8);
                if (ok) frag_store<IO>(p.y_w, b, n, p.d, from_float<IO>(f * nw[i]));
                if (ok && row % 16 == 0) p.ssq_out[(int64_t)(n / 16) * p.batch + b] = s;
            }
        }
        if (ok) static_cast<IO*>(p.y)[at] = v;
    }
}

// DTV consecutive values of a row of dt_proj
template <typename IO, int DTV>
struct DtVec {  // one element
    typedef IO Raw;
    static __device__ __forceinline__ Raw load(const IO* p) { return *p; }
    static __device__ __forceinline__ void unpack(const Raw& r, float (&w)[DTV]) { w[0] = to_float(r); }
};
template <>
struct DtVec<bf16_t, 4> {
    typedef u32x2 Raw;
    static __device__ __forceinline__ Raw load(const bf16_t* p) { return *reinterpret_cast<const u32x2*>(p); }
    static __device__ __forceinline__ void unpack(const Raw& v, float (&w)[4]) {
        w[0] = __uint_as_float(v[0] << 16);
        w[1] = __uint_as_float(v[0] & 0xffff0000u);
        w[2] = __uint_as_float(v[1] << 16);
        w[3] = __uint_as_float(v[1] & 0xffff0000u);
    }
};
template <>
struct DtVec<float, 4> {
    typedef u32x4 Raw;
    static __device__ __forceinline__ Raw load(const float* p) { return ld16(p); }
    static __device__ __forceinline__ void unpack(const Raw& v, float (&w)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = __uint_as_float(v[i]);
    }
};

// A thread owns a quarter of the states and of the dt_rank of one channel, for BT sequences: the
// quarter sums of dt_proj meet in a quad (two exchanges), after which every lane of the quad has
// delta and goes on with its own states.  State loads are issued before the dt_proj sum.
// MANY: dbc comes as many partial sums (see xproj_fused); otherwise as eight at most (see decode_splits).
template <typename IO, int BT, bool N16, int DTV, bool MANY>
__global__ void __launch_bounds__(256) decode_ssm_kernel(const DecodeParams p) {
    extern __shared__ float dbc[];  // [BT][R + 2N], as many times as threads allow while it is summed
    const int P = p.R + 2 * p.N;
    const int b0 = blockIdx.y * BT;
    const int part = threadIdx.x & 3, ch = blockIdx.x * 64 + (threadIdx.x >> 2);
    const bool live = ch < p.ED;
    const int d = live ? ch : p.ED - 1;
    f32x4 h[BT], a16;
    float xv[BT], zv[BT];
    if constexpr (N16) a16 = *reinterpret_cast<const f32x4*>(p.A + (int64_t)d * 16 + 4 * part);
#pragma unroll
    for (int t = 0; t < BT; ++t) {
        const int64_t row = (int64_t)min(b0 + t, p.batch - 1) * p.ED + d;
        if constexpr (N16)
            h[t] = p.h_in ? *reinterpret_cast<const f32x4*>(p.h_in + row * 16 + 4 * part) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        xv[t] = frag_load<IO>(p.xs, min(b0 + t, p.batch - 1), d, p.ED);
        zv[t] = load_as_float<IO>(p.z, row);
    }
    const float Dv = p.D[d], bias = p.dt_b ? p.dt_b[d] : 0.0f;
    // the first rows of dt_proj are requested here, ahead of the barriers
    typedef DtVec<IO, DTV> Dt;
    constexpr int kPre = 3;
    const IO* wr = static_cast<const IO*>(p.dt_w) + (int64_t)d * p.R;
    typename Dt::Raw pre[kPre];
#pragma unroll
    for (int i = 0; i < kPre; ++i) pre[i] = Dt::load(wr + min(DTV * (part + 4 * i), p.R - DTV));
    if constexpr (!MANY) {
        const rsrc_t parts = window(p.dbc, (int64_t)p.splits * p.batch * P, 4);
        for (int i = threadIdx.x; i < BT * P; i += 256) {
            const int t = i / P, b = b0 + t;
            float v[8], s = 0.0f;  // (requested together)
#pragma unroll
            for (int q = 0; q < 8; ++q)
                v[q] = ld_f32(parts, (uint32_t)((q * p.batch + b) * P + (i - t * P)) * 4u, b < p.batch && q < p.splits);
#pragma unroll
            for (int q = 0; q < 8; ++q) s += v[q];
            dbc[i] = s;
        }
        __syncthreads();
    } else {
        static_assert(BT == 1, "small calls take one sequence per workgroup");
        // thread -> (output, every G-th of the partial sums), 8, 16 or 32 requested together (width 768 has 32
        // of them: 13.9 -> 13.4 us a layer; in two turns of 16 they were two memory latencies)
        const int G = max(256 / P, 1), g = G > 1 ? threadIdx.x / P : 0;
        const auto sum = [&](const float* src, auto some) {
            constexpr int kSome = decltype(some)::value;
            const int64_t pitch = (int64_t)p.batch * P;
            float s = 0.0f;
            for (int q0 = g; q0 < p.splits; q0 += kSome * G) {
                float v[kSome];
#pragma unroll
                for (int j = 0; j < kSome; ++j) v[j] = src[min(q0 + j * G, p.splits - 1) * pitch];
#pragma unroll
                for (int j = 0; j < kSome; ++j)
                    if (q0 + j * G < p.splits) s += v[j];
            }
            return s;
        };
        for (int i = G > 1 ? threadIdx.x % P : threadIdx.x; i < P && g < G; i += 256) {
            const float* src = p.dbc + (int64_t)b0 * P + i;
            const float s = p.splits <= 8 * G    ? sum(src, std::integral_constant<int, 8>())
                            : p.splits <= 16 * G ? sum(src, std::integral_constant<int, 16>())
                                                 : sum(src, std::integral_constant<int, 32>());
            dbc[g * P + i] = s;
        }
        __syncthreads();
        if (G > 1) {
            float s = 0.0f;
            if ((int)threadIdx.x < P)
                for (int q = 0; q < G; ++q) s += dbc[q * P + threadIdx.x];
            __syncthreads();
            if ((int)threadIdx.x < P) dbc[threadIdx.x] = s;
            __syncthreads();
        }
    }
    float dl[BT] = {};
    auto dt_dot = [&](const typename Dt::Raw& raw, int r) {
        float w[DTV];
        Dt::unpack(raw, w);
#pragma unroll
        for (int t = 0; t < BT; ++t)
#pragma unroll
            for (int i = 0; i < DTV; ++i) dl[t] = __builtin_fmaf(w[i], dbc[t * P + r + i], dl[t]);
    };
#pragma unroll
    for (int i = 0; i < kPre; ++i)
        if (DTV * (part + 4 * i) < p.R) dt_dot(pre[i], DTV * (part + 4 * i));
    for (int r = DTV * (part + 4 * kPre); r < p.R; r += 4 * DTV) dt_dot(Dt::load(wr + r), r);
#pragma unroll
    for (int t = 0; t < BT; ++t) {
        const int b = b0 + t;
        float s = dl[t];
        s += __shfl_xor(s, 1);
        s += __shfl_xor(s, 2);
        const float delta = softplus_f(s + bias), dl2 = delta * kLog2e, u = delta * xv[t];
        const float* Bv = dbc + t * P + p.R;
        const float* Cv = Bv + p.N;
        const int64_t row = (int64_t)min(b, p.batch - 1) * p.ED + d;
        const bool mine = live && b < p.batch;
        float acc = 0.0f;
        auto states = [&](int n, f32x4 hv, const f32x4& av) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                hv[i] = __builtin_fmaf(u, Bv[n + i], fast_exp2(dl2 * av[i]) * hv[i]);
                acc = __builtin_fmaf(Cv[n + i], hv[i], acc);
            }
            if (mine) *reinterpret_cast<f32x4*>(p.h_out + row * p.N + n) = hv;
        };
        if constexpr (N16) {
            states(4 * part, h[t], a16);
        } else {
            for (int n = 4 * part; n < p.N; n += 16)
                states(n,
                       p.h_in ? *reinterpret_cast<const f32x4*>(p.h_in + row * p.N + n) : f32x4{0.0f, 0.0f, 0.0f, 0.0f},
                       *reinterpret_cast<const f32x4*>(p.A + (int64_t)d * p.N + n));
        }
        acc += __shfl_xor(acc, 1);
        acc += __shfl_xor(acc, 2);
        if (mine && part == 0)
            frag_store<IO>(p.g, b, d, p.ED, from_float<IO>(__builtin_fmaf(Dv, xv[t], acc) * zv[t] * sigmoid_f(zv[t])));
    }
}

static int decode_validate(const mpa_decode_layer* s) {
    if (!s) return MPA_ERR_NULL_POINTER;
    if (s->io_dtype != MPA_F32 && s->io_dtype != MPA_BF16) return MPA_ERR_BAD_DTYPE;
    const int64_t vec = s->io_dtype == MPA_BF16 ? 8 : 4;
    if (s->batch <= 0 || s->batch > MPA_DECODE_MAX_BATCH || s->d_model <= 0 || s->dim <= 0 || s->dt_rank <= 0 ||
        s->dstate <= 0 || s->dstate > MPA_MAX_DSTATE || s->d_conv < 2 || s->d_conv > 4)
        return MPA_ERR_BAD_SHAPE;
    if (s->d_model % vec || s->dim % vec || s->dstate % 4 || s->d_model > 1 << 20 || s->dim > 1 << 20 || s->dt_rank > 2048)
        return MPA_ERR_BAD_SHAPE;
    return MPA_OK;
}

// K ranges of x_proj: its few rows give few workgroups, so K is cut until about 128 of them run
// (each with at least one piece per wave); the state kernel adds the partial sums as it reads them.
constexpr int kXprojWaves = 8;
static bool xproj_fused(int ED, int P, int batch);
static int decode_splits(const mpa_decode_layer* s) {
    if (xproj_fused((int)s->dim, (int)(s->dt_rank + 2 * s->dstate), (int)s->batch)) return (int)((s->dim + 15) / 16);
    const int64_t piece = s->io_dtype == MPA_BF16 ? 64 : 32;
    const int64_t tiles = ((s->dt_rank + 2 * s->dstate + 15) / 16) * ((s->batch + 15) / 16);
    const int64_t by_k = (s->dim + piece * kXprojWaves - 1) / (piece * kXprojWaves);
    int64_t n = (128 + tiles - 1) / tiles;
    n = n < by_k ? n : by_k;
    return (int)(n < 1 ? 1 : n > 8 ? 8 : n);
}

static size_t round256(size_t v) { return (v + 255) / 256 * 256; }

static dim3 decode_grid(int64_t row_tiles, int64_t groups, int splits) {
    return dim3((unsigned)((row_tiles + 7) / 8 * 8 * groups), (unsigned)splits);
}

// Workgroup tiles (row tiles x batch tiles, waves, pieces in flight of each), from sweeps over fourteen of them at widths 768 to
// 2560 and batches 1 to 128.  in_proj: one 16 x 16 tile on eight waves, two pieces, is best or within 3 % while its tiles are
// fewer than 1536; from there two batch tiles (64 x 2560: float32 128 -> 115 us a layer, bfloat16 80 -> 75).  Larger tiles read less
// and lose to the second workgroup that their registers cost (4 x 4: 124 and 77).
constexpr int kManyTiles = 1536;

// in_proj does its share of x_proj for one batch tile while the partial sums that it leaves, one per 16 channels, are
// few: they cost the state kernel less than a launch then (a layer of width 768 in bfloat16, one sequence: 16.3 ->
// 14.9 us, 16 sequences 18.2 -> 17.1; width 256 13.1 -> 11.3; but width 2560 in float32, eight times the partial
// sums, 56 -> 72).
static bool xproj_fused(int ED, int P, int batch) { return batch <= 16 && P <= 512 && (int64_t)((ED + 15) / 16) * P <= 16384; }

template <typename IO, int MODE>
static int launch_in(const DecodeParams& p, hipStream_t st) {
    const int rt = (2 * p.ED + 15) / 16, bt = (p.batch + 15) / 16;
    if (xproj_fused(p.ED, p.R + 2 * p.N, p.batch)) {
        // (float32 rows have twice the pieces.  From 704 columns on fewer waves with more pieces in flight, a measured line: 1 x 768 20.2 ->
        // 19.0 us a layer, but below it eight waves are 1 to 3 % faster at every width tried, 12 layers of 1 x 700 210 us and 215, of
        // 16 x 576 229 and 235.  Up to 512 columns a wave has two pieces at most, and the second is better requested as the first is
        // used: 6 layers of 1 x 512 118.7 us with both in flight, 116.0.  Four waves have a thread for 256 rows of x_proj; more of them
        // take eight at any width.)
        if (sizeof(IO) == 4 && p.d >= 704 && p.R + 2 * p.N <= 256) hipLaunchKernelGGL((decode_in_kernel<IO, 1, 1, 4, 4, MODE, true>), decode_grid(rt, bt, 1), dim3(256), 0, st, p, rt, bt);
        else if (sizeof(IO) == 4 && p.d > 256 && p.d <= 512) hipLaunchKernelGGL((decode_in_kernel<IO, 1, 1, 8, 1, MODE, true>), decode_grid(rt, bt, 1), dim3(512), 0, st, p, rt, bt);
        else hipLaunchKernelGGL((decode_in_kernel<IO, 1, 1, 8, 2, MODE, true>), decode_grid(rt, bt, 1), dim3(512), 0, st, p, rt, bt);
    } else if (rt * bt < kManyTiles) {
        hipLaunchKernelGGL((decode_in_kernel<IO, 1, 1, 8, 2, MODE>), decode_grid(rt, bt, 1), dim3(512), 0, st, p, rt, bt);
    } else {
        const int groups = (bt + 1) / 2;
        // (four waves where eight would have two pieces each or fewer: 128 x 1000 in bfloat16 14.2 us on eight, 11.2 on four)
        if (p.d * (int)sizeof(IO) <= 2048) hipLaunchKernelGGL((decode_in_kernel<IO, 1, 2, 4, 2, MODE>), decode_grid(rt, groups, 1), dim3(256), 0, st, p, rt, groups);
        else hipLaunchKernelGGL((decode_in_kernel<IO, 1, 2, 8, 2, MODE>), decode_grid(rt, groups, 1), dim3(512), 0, st, p, rt, groups);
    }
    return check_launch();
}

template <typename IO>
static int launch_xproj(const DecodeParams& p, hipStream_t st) {
    const int rt = (p.R + 2 * p.N + 15) / 16, bt = (p.batch + 15) / 16;
    hipLaunchKernelGGL((decode_xproj_kernel<IO, kXprojWaves>), decode_grid(rt, bt, p.splits), dim3(kXprojWaves * kWave), 0, st, p, rt, bt);
    return check_launch();
}

// out_proj has half the rows and twice the K: sixteen waves while one workgroup per CU is all there is (1 x 2560 float32: 56 us a
// layer, 58 on eight), then two batch tiles on eight waves, and from 512 tiles two row tiles as well (64 x 1536: float32 61 -> 58 us a
// layer, 64 x 2560 123 -> 120; bfloat16 42 -> 40 and 80 -> 75).
template <typename IO, bool RES>
static int launch_out(const DecodeParams& p, hipStream_t st) {
    const int rt = (p.d + 15) / 16, bt = (p.batch + 15) / 16, groups = (bt + 1) / 2, pairs = (rt + 1) / 2;
    if (rt * bt <= 256) hipLaunchKernelGGL((decode_out_kernel<IO, 1, 1, 16, 2, RES>), decode_grid(rt, bt, 1), dim3(1024), 0, st, p, rt, bt);
    else if (rt * bt < 512) hipLaunchKernelGGL((decode_out_kernel<IO, 1, 2, 8, 2, RES>), decode_grid(rt, groups, 1), dim3(512), 0, st, p, rt, groups);
    else hipLaunchKernelGGL((decode_out_kernel<IO, 2, 2, 8, 2, RES>), decode_grid(pairs, groups, 1), dim3(512), 0, st, p, pairs, groups);
    return check_launch();
}

template <typename IO, int BT, bool MANY = false>
static int launch_ssm(const DecodeParams& p, hipStream_t st) {
    const dim3 grid((p.ED + 63) / 64, (p.batch + BT - 1) / BT);
    const int outs = BT * (p.R + 2 * p.N);
    const size_t lds = (size_t)(outs < 256 ? 256 : outs) * sizeof(float);
    if (lds > 48 * 1024) return MPA_ERR_BAD_SHAPE;
    const bool v4 = p.R % 4 == 0 && aligned_to(p.dt_w, 4 * sizeof(IO));
#define MPA_SSM(N16_, V_) hipLaunchKernelGGL((decode_ssm_kernel<IO, BT, N16_, V_, MANY>), grid, dim3(256), lds, st, p)
    if (p.N == 16) { if (v4) MPA_SSM(true, 4); else MPA_SSM(true, 1); }
    else { if (v4) MPA_SSM(false, 4); else MPA_SSM(false, 1); }
#undef MPA_SSM
    return check_launch();
}

// A first layer whose in_proj has many tiles: each of them would normalise its sequences again, and read them by
// rows (64 x 2560, float32: 88 us, 62 + 4 with the rows prepared).
static bool scale_first(int ED, int batch) { return (2 * ED + 15) / 16 * ((batch + 15) / 16) >= kManyTiles; }

template <typename IO>
static int decode_launch(DecodeParams p, bool norm, void* xw, float* ssq, hipStream_t st) {
    if (norm && !p.xw && scale_first(p.ED, p.batch)) {
        hipLaunchKernelGGL((decode_scale_kernel<IO>), dim3(p.batch), dim3(256), 0, st, p, xw, ssq);
        const int e = check_launch();
        if (e != MPA_OK) return e;
        p.xw = xw; p.ssq = ssq; p.ssq_tiles = 1;
    }
    int rc = !norm ? launch_in<IO, kInPlain>(p, st) : p.xw ? launch_in<IO, kInReady>(p, st) : launch_in<IO, kInNorm>(p, st);
    if (rc != MPA_OK) return rc;
    const bool fused = xproj_fused(p.ED, p.R + 2 * p.N, p.batch);
    if (!fused) rc = launch_xproj<IO>(p, st);
    if (rc != MPA_OK) return rc;
    // sequences per workgroup: four (weights and A read once for them) while that leaves two
    // workgroups per CU; one where dbc is many partial sums, whose summing takes all threads
    const int64_t cols = (p.ED + 63) / 64;
    rc = fused ? launch_ssm<IO, 1, true>(p, st)
         : cols * ((p.batch + 3) / 4) >= 512 ? launch_ssm<IO, 4>(p, st)
         : cols * ((p.batch + 1) / 2) >= 512 ? launch_ssm<IO, 2>(p, st) : launch_ssm<IO, 1>(p, st);
    if (rc != MPA_OK) return rc;
    return norm ? launch_out<IO, true>(p, st) : launch_out<IO, false>(p, st);
}

}  // namespace mpa

using namespace mpa;

extern "C" size_t mpa_decode_scaled_bytes(const mpa_decode_layer* s) {
    return decode_validate(s) == MPA_OK ? (size_t)frag_bytes(s->batch, s->d_model, (int)dtype_size(s->io_dtype)) : 0;
}

static size_t decode_scaled_ws(const mpa_decode_layer* s) {
    return s->norm && scale_first((int)s->dim, (int)s->batch)
               ? (size_t)frag_bytes(s->batch, s->d_model, (int)dtype_size(s->io_dtype)) + round256(s->batch * sizeof(float)) : 0;
}

extern "C" size_t mpa_decode_layer_workspace_bytes(const mpa_decode_layer* s) {
    if (decode_validate(s) != MPA_OK) return 0;
    const size_t act = (size_t)frag_bytes(s->batch, s->dim, (int)dtype_size(s->io_dtype));
    return 3 * act + round256((size_t)decode_splits(s) * s->batch * (s->dt_rank + 2 * s->dstate) * sizeof(float)) + decode_scaled_ws(s);
}

extern "C" int mpa_decode_layer_step(const mpa_decode_layer* s, const void* x, const void* x_scaled, const float* x_ssq, void* y,
                                     const float* next_norm_weight, void* y_scaled, float* y_ssq, const float* h_in, float* h_out,
                                     const void* window_in, void* window_out, void* workspace, size_t workspace_bytes, void* stream) {
    int rc = decode_validate(s);
    if (rc != MPA_OK) return rc;
    if (!x || !y || !h_out || !window_in || !window_out || !workspace || !s->in_weight || !s->conv_weight || !s->x_weight ||
        !s->dt_weight || !s->A || !s->D || !s->out_weight || (x_scaled && !x_ssq) || (next_norm_weight && (!y_scaled || !y_ssq)))
        return MPA_ERR_NULL_POINTER;
    if (!s->norm && (x_scaled || next_norm_weight)) return MPA_ERR_BAD_SHAPE;
    const size_t es = dtype_size(s->io_dtype);
    const void* wide[] = {x, x_scaled, y_scaled, s->in_weight, s->x_weight, s->out_weight, s->norm_weight, s->A, h_in, h_out};
    for (const void* q : wide)
        if (q && !aligned_to(q, 16)) return MPA_ERR_MISALIGNED;
    const void* narrow[] = {y, window_in, window_out, s->in_bias, s->out_bias, s->dt_weight};
    for (const void* q : narrow)
        if (q && !aligned_to(q, es)) return MPA_ERR_MISALIGNED;
    const void* words[] = {s->conv_weight, s->conv_bias, s->dt_bias, s->D, next_norm_weight, x_ssq, y_ssq};
    for (const void* q : words)
        if (q && !aligned_to(q, 4)) return MPA_ERR_MISALIGNED;
    if (!aligned_to(workspace, 256)) return MPA_ERR_MISALIGNED;
    if (workspace_bytes < mpa_decode_layer_workspace_bytes(s)) return MPA_ERR_WORKSPACE;
    DecodeParams p{};
    p.batch = (int)s->batch; p.d = (int)s->d_model; p.ED = (int)s->dim; p.N = (int)s->dstate; p.R = (int)s->dt_rank;
    p.K = s->d_conv; p.eps = s->eps; p.splits = decode_splits(s); p.ssq_tiles = (p.d + 15) / 16;
    p.x = x; p.xw = x_scaled; p.ssq = x_ssq; p.norm_w = s->norm_weight;
    p.in_w = s->in_weight; p.in_b = s->in_bias; p.conv_w = s->conv_weight; p.conv_b = s->conv_bias;
    p.xp_w = s->x_weight; p.dt_w = s->dt_weight; p.dt_b = s->dt_bias; p.A = s->A; p.D = s->D;
    p.out_w = s->out_weight; p.out_b = s->out_bias;
    p.h_in = h_in; p.h_out = h_out; p.win_in = window_in; p.win_out = window_out;
    p.y = y; p.next_w = next_norm_weight; p.y_w = y_scaled; p.ssq_out = y_ssq;
    const size_t act = (size_t)frag_bytes(s->batch, s->dim, (int)es);
    char* ws = static_cast<char*>(workspace);
    p.xs = ws; p.z = ws + act; p.g = ws + 2 * act; p.dbc = reinterpret_cast<float*>(ws + 3 * act);
    hipStream_t st = static_cast<hipStream_t>(stream);
    char* const xw = ws + mpa_decode_layer_workspace_bytes(s) - decode_scaled_ws(s);
    float* const ssq = reinterpret_cast<float*>(xw + frag_bytes(s->batch, s->d_model, (int)es));
    return s->io_dtype == MPA_F32 ? decode_launch<float>(p, s->norm != 0, xw, ssq, st) : decode_launch<bf16_t>(p, s->norm != 0, xw, ssq, st);
}
