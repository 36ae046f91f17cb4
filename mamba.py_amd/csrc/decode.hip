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
// owns 16 rows of W and up to NT tiles of 16 sequences, its waves split K, and the partial tiles meet
// in LDS.  A contraction may be summed in any order, so a wave takes 128 bytes of each of its rows at
// a time: eight lanes load one row's piece (lanes in different rows, as the MFMA operand has them, cost
// an address per lane: in_proj of 64 sequences at width 2560, float32, took 95 us that way, 55 us now), and a
// 2 KB exchange through the wave's own LDS turns rows into operands.  Activations that these kernels
// write for each other are stored in operand order.  The unused columns of a batch below 16 cost nothing that
// matters: the kernels wait for the weights, not for the matrix pipe.  What the epilogue needs is
// requested before the product, so that its latency is not added to the weights'.
#include "common.h"

namespace mpa {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Operand fragment of one lane: kVec consecutive k of one row, loaded with one 16-byte access.
template <typename IO>
struct Frag;
template <>
struct Frag<bf16_t> {
    static constexpr int kVec = 8;
    static __device__ __forceinline__ void unpack(const u32x4& v, float (&f)[8]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f[2 * i] = __uint_as_float(v[i] << 16);
            f[2 * i + 1] = __uint_as_float(v[i] & 0xffff0000u);
        }
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[8]) {
        bf16x8 r;
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = static_cast<__bf16>(f[i]);
        return __builtin_bit_cast(u32x4, r);
    }
    template <int NT>
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4 (&b)[NT], f32x4 (&c)[NT]) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
            c[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                           __builtin_bit_cast(bf16x8, b[t]), c[t], 0, 0, 0);
    }
};
template <>
struct Frag<float> {
    static constexpr int kVec = 4;
    static __device__ __forceinline__ void unpack(const u32x4& v, float (&f)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(v[i]);
    }
    static __device__ __forceinline__ u32x4 pack(const float (&f)[4]) {
        u32x4 r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = __float_as_uint(f[i]);
        return r;
    }
    // four products of one k per lane group: together the 16 k that the four lane groups hold (the
    // tiles in the inner loop: products of one tile depend on each other)
    template <int NT>
    static __device__ __forceinline__ void mma(const u32x4& a, const u32x4 (&b)[NT], f32x4 (&c)[NT]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
                c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i]), __uint_as_float(b[t][i]), c[t],
                                                            0, 0, 0);
    }
};

__device__ __forceinline__ u32x4 ld16(const void* p) { return *static_cast<const u32x4*>(p); }

// Operand order of activations (batch x K): tiles of 16 sequences x kChunk values of k, lane
// (sequence % 16) + 16 * (k / kVec % 4) of a tile holding kVec consecutive k.
template <typename IO>
__device__ __forceinline__ int64_t frag_at(int b, int k, int K) {
    constexpr int kVec = Frag<IO>::kVec, kChunk = 4 * kVec;
    const int chunks = (K + kChunk - 1) / kChunk;
    return (((int64_t)(b >> 4) * chunks + k / kChunk) * 64 + (b & 15) + 16 * (k % kChunk / kVec)) * kVec + k % kVec;
}
__host__ __device__ inline int64_t frag_bytes(int64_t batch, int64_t K, int es) {
    return (batch + 15) / 16 * ((K * es + 63) / 64) * 1024;
}

// Activations in operand order.
template <typename IO, int NT>
struct FragAct {
    typedef u32x4 Raw;
    const IO* x[NT];
    __device__ __forceinline__ void setup(const void* base, int b0, int batch, int K, int lane) {
#pragma unroll
        for (int t = 0; t < NT; ++t)  // (a tile beyond the batch repeats the last one: its products are not used)
            x[t] = static_cast<const IO*>(base) + frag_at<IO>(min(b0 + t * 16, batch - 1) & ~15, 0, K) + lane * Frag<IO>::kVec;
    }
    __device__ __forceinline__ void request(Raw& r, int t, int chunk, int, bool ok) {
        r = ok ? ld16(x[t] + (int64_t)chunk * 64 * Frag<IO>::kVec) : u32x4{0, 0, 0, 0};
    }
    __device__ __forceinline__ u32x4 operand(const Raw& r, int) { return r; }
};

// Rows of X as the caller has them (null: a column without a sequence), as they are or (NORM) times
// the norm weight, with the sums of squares.
template <typename IO, int NT, bool NORM>
struct RowAct {
    static constexpr int kVec = Frag<IO>::kVec;
    struct Raw {
        u32x4 x;
        float w[NORM ? kVec : 1];
    };
    const IO* x[NT];
    const float* w;  // null: no gain
    float ss[NT];
    __device__ __forceinline__ void setup(const void* base, int b0, int batch, int K, int lane) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int b = b0 + t * 16 + (lane & 15);
            x[t] = b < batch ? static_cast<const IO*>(base) + (int64_t)b * K : nullptr;
            ss[t] = 0.0f;
        }
    }
    __device__ __forceinline__ void request(Raw& r, int t, int, int k, bool ok) {
        r.x = ok && x[t] ? ld16(x[t] + k) : u32x4{0, 0, 0, 0};
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < kVec; i += 4) {
                const f32x4 v = ok && w ? *reinterpret_cast<const f32x4*>(w + k + i) : f32x4{1.0f, 1.0f, 1.0f, 1.0f};
#pragma unroll
                for (int j = 0; j < 4; ++j) r.w[i + j] = v[j];
            }
        }
    }
    __device__ __forceinline__ u32x4 operand(const Raw& r, int t) {
        if constexpr (!NORM) return r.x;
        float f[kVec];
        Frag<IO>::unpack(r.x, f);
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            ss[t] = __builtin_fmaf(f[i], f[i], ss[t]);
            f[i] *= r.w[i];
        }
        return Frag<IO>::pack(f);
    }
};

// What a wave of decode_product keeps in LDS: two slots of 16 rows x 128 bytes for the exchange, then
// its partial tiles (lane l holds rows 4*(l/16) .. +3 of column l%16 of each).
struct alignas(16) WaveLds {
    float v[1024];
};
template <int NW>
__device__ __forceinline__ float tile_sum(const WaveLds (&lds)[NW], int row, int b) {
    const int at = (b >> 4) * 256 + ((row >> 2) * 16 + (b & 15)) * 4 + (row & 3);
    float s = lds[0].v[at];
#pragma unroll
    for (int w = 1; w < NW; ++w) s += lds[w].v[at];
    return s;
}

// Rows n0 .. n0+15 of `W . x^T` for NT batch tiles, over the 128-byte pieces first + wave, + NW, ...
// below `last` of the rows of W; the wave leaves its partial tiles in its LDS.  Two groups of U pieces
// are in flight (`more` issues the caller's own loads behind the first), each with its activations: loads return in the order they were issued, so
// activations requested later than weights of pieces further on would wait for those as well.
template <typename IO, int NT, int NW, int U, typename ACT, typename MORE>
__device__ __forceinline__ void decode_product(WaveLds& lds, const void* W, int rows, int K, int n0, int first, int last, int wave,
                                               int lane, ACT& act, MORE&& more) {
    constexpr int kVec = Frag<IO>::kVec, kPiece = 8 * kVec;
    char* const slot = reinterpret_cast<char*>(lds.v);
    // lane -> 16 bytes of row 8*i + lane/8: the piece's eight 16-byte parts are stored rotated by the row
    // (part ^ (row & 7)), so that the operand reads, one row per lane, fall on different banks
    const int part = (lane & 7) ^ (lane >> 3), kw = part * kVec;
    const IO* wrow[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) wrow[i] = static_cast<const IO*>(W) + (int64_t)min(n0 + 8 * i + (lane >> 3), rows - 1) * K;
    const int kl = kVec * (lane >> 4);
    int frag[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) frag[h] = (lane & 15) * 128 + ((((lane >> 4) + 4 * h) ^ (lane & 7)) << 4);
    const int count = first + wave < last ? (last - first - wave + NW - 1) / NW : 0;  // pieces of this wave

    u32x4 w[2][U][2];
    typename ACT::Raw a[2][U][NT][2];
    auto request = [&](int buf, int s) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int piece = first + wave + (s + u) * NW;
            const bool some = s + u < count;
#pragma unroll
            for (int i = 0; i < 2; ++i)
                w[buf][u][i] = some && piece * kPiece + kw < K ? ld16(wrow[i] + piece * kPiece + kw) : u32x4{0, 0, 0, 0};
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int k = (2 * piece + h) * 4 * kVec + kl;
#pragma unroll
                for (int t = 0; t < NT; ++t) act.request(a[buf][u][t][h], t, 2 * piece + h, k, some && k < K);
            }
        }
    };
    f32x4 acc[NT] = {};
    auto group = [&](int buf, int s0) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s0 + u >= count) break;  // uniform over the wave
            char* const at = slot + (u & 1) * 2048;
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(at + i * 1024 + lane * 16) = w[buf][u][i];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u32x4 wf = *reinterpret_cast<const u32x4*>(at + frag[h]);
                u32x4 x[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) x[t] = act.operand(a[buf][u][t][h], t);
                Frag<IO>::mma(wf, x, acc);
            }
        }
    };
    request(0, 0);
    more();
    for (int s = 0; s < count; s += 2 * U) {
        request(1, s + U);
        group(0, s);
        request(0, s + 2 * U);
        group(1, s + U);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4*>(&lds.v[t * 256 + 4 * lane]) = acc[t];
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
// more partial sum of dbc; a thread owns one row and every so many sequences.
template <typename IO, int NT, int NW, int U, int MODE, bool XP = false>
__global__ void __launch_bounds__(NW* kWave) decode_in_kernel(const DecodeParams p, int row_tiles, int groups) {
    constexpr int kThreads = NW * kWave, kAll = NT * 256, kOuts = (kAll + kThreads - 1) / kThreads;
    __shared__ WaveLds tile[NW];
    __shared__ float ssq[NW][NT][16];
    __shared__ float xl[XP ? NT * 16 : 1][16];  // convolved x of the tile
    int rt, bt;
    decode_tile<NT>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;  // uniform over the block
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * 16, b0 = bt * 16, rows = 2 * p.ED;
    const int pieces = (p.d + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    // the epilogue's operands: thread -> outputs (row o % 16, sequence o / 16)
    IO win[kOuts][3];
    float cw[kOuts][4], cb[kOuts], ib[kOuts];
    float ss[NT] = {};
    const int P = p.R + 2 * p.N;
    u32x4 xw[XP ? 16 / Frag<IO>::kVec : 1];
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
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % 16, b = b0 + o / 16;
            ib[i] = cb[i] = 0.0f;
            if (o >= kAll || n >= rows || b >= p.batch) continue;
            if (p.in_b) ib[i] = load_as_float<IO>(p.in_b, n);
            if (n >= p.ED) continue;
            const IO* wi = static_cast<const IO*>(p.win_in) + ((int64_t)b * p.ED + n) * (p.K - 1);
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j < p.K - 1) win[i][j] = wi[j];
#pragma unroll
            for (int j = 0; j < 4; ++j) cw[i][j] = j < p.K ? p.conv_w[(int64_t)n * p.K + j] : 0.0f;
            if (p.conv_b) cb[i] = p.conv_b[n];
        }
        if constexpr (MODE == kInReady) {
            // wave w, lane group q: partial sums 4w + q, 4w + q + 4*NW, ... of column lane % 16
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int b = b0 + t * 16 + (lane & 15);
                if (b < p.batch)
                    for (int q = 4 * wave + (lane >> 4); q < p.ssq_tiles; q += 4 * NW) ss[t] += p.ssq[(int64_t)q * p.batch + b];
            }
        }
    };
    if constexpr (MODE == kInReady) {
        FragAct<IO, NT> act;
        act.setup(p.xw, b0, p.batch, p.d, lane);
        decode_product<IO, NT, NW, U>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
    } else {
        RowAct<IO, NT, MODE == kInNorm> act;
        act.w = p.norm_w;
        act.setup(p.x, b0, p.batch, p.d, lane);
        decode_product<IO, NT, NW, U>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
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
        const int o = threadIdx.x + i * kThreads, row = o % 16, bl = o / 16, n = n0 + row, b = b0 + bl;
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
        static_cast<IO*>(p.xs)[frag_at<IO>(b, n, p.ED)] = cr;
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
    for (int k = threadIdx.x * kVec; k < p.d; k += 256 * kVec) {
        float f[kVec];
        Frag<IO>::unpack(ld16(row + k), f);
#pragma unroll
        for (int i = 0; i < kVec; ++i) {
            ss = __builtin_fmaf(f[i], f[i], ss);
            if (p.norm_w) f[i] *= p.norm_w[k + i];
        }
        *reinterpret_cast<u32x4*>(static_cast<IO*>(xw) + frag_at<IO>(b, k, p.d)) = Frag<IO>::pack(f);
    }
#pragma unroll
    for (int o = 1; o < kWave; o *= 2) ss += __shfl_xor(ss, o);
    if ((threadIdx.x & (kWave - 1)) == 0) part[wave_id()] = ss;
    __syncthreads();
    if (threadIdx.x == 0) ssq[b] = (part[0] + part[1]) + (part[2] + part[3]);
}

template <typename IO, int NW>
__global__ void __launch_bounds__(NW* kWave) decode_xproj_kernel(const DecodeParams p, int row_tiles, int groups) {
    __shared__ WaveLds tile[NW];
    int rt, bt;
    decode_tile<1>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id(), rows = p.R + 2 * p.N;
    const int pieces = (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    const int per = (pieces + gridDim.y - 1) / gridDim.y, first = (int)blockIdx.y * per;
    FragAct<IO, 1> act;
    act.setup(p.xs, bt * 16, p.batch, p.ED, lane);
    decode_product<IO, 1, NW, 1>(tile[wave], p.xp_w, rows, p.ED, rt * 16, first, min(pieces, first + per), wave, lane, act, [] {});
    __syncthreads();
    const int o = threadIdx.x, n = rt * 16 + (o & 15), b = bt * 16 + (o >> 4);
    if (o < 256 && n < rows && b < p.batch) p.dbc[((int64_t)blockIdx.y * p.batch + b) * rows + n] = tile_sum(tile, o & 15, o >> 4);
}

// y = out_proj(g) [+ x]; with next_w also y * next_w and the sums of squares of 16 columns each
template <typename IO, int NT, int NW, int U, bool RES>
__global__ void __launch_bounds__(NW* kWave) decode_out_kernel(const DecodeParams p, int row_tiles, int groups) {
    constexpr int kThreads = NW * kWave, kAll = NT * 256, kOuts = (kAll + kThreads - 1) / kThreads;
    __shared__ WaveLds tile[NW];
    int rt, bt;
    decode_tile<NT>(row_tiles, groups, rt, bt);
    if (rt >= row_tiles) return;
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * 16, b0 = bt * 16;
    float bias[kOuts], xv[kOuts], nw[kOuts];
    auto more = [&] {
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % 16, b = b0 + o / 16;
            const bool ok = o < kAll && n < p.d && b < p.batch;
            bias[i] = ok && p.out_b ? load_as_float<IO>(p.out_b, n) : 0.0f;
            xv[i] = RES && ok ? load_as_float<IO>(p.x, (int64_t)b * p.d + n) : 0.0f;
            nw[i] = RES && ok && p.next_w ? p.next_w[n] : 0.0f;
        }
    };
    FragAct<IO, NT> act;
    act.setup(p.g, b0, p.batch, p.ED, lane);
    decode_product<IO, NT, NW, U>(tile[wave], p.out_w, p.d, p.ED, n0, 0, (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec), wave,
                                      lane, act, more);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOuts; ++i) {
        const int o = threadIdx.x + i * kThreads, row = o % 16, bl = o / 16, n = n0 + row, b = b0 + bl;
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
                if (ok) static_cast<IO*>(p.y_w)[frag_at<IO>(b, n, p.d)] = from_float<IO>(f * nw[i]);
                if (ok && row == 0) p.ssq_out[(int64_t)rt * p.batch + b] = s;
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
// MANY: dbc comes as many partial sums (see xproj_fused).
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
        xv[t] = load_as_float<IO>(p.xs, frag_at<IO>(min(b0 + t, p.batch - 1), d, p.ED));
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
        for (int i = threadIdx.x; i < BT * P; i += 256) {
            const int t = i / P, b = b0 + t;
            float s = 0.0f;
            if (b < p.batch)
                for (int q = 0; q < p.splits; ++q) s += p.dbc[((int64_t)q * p.batch + b) * P + (i - t * P)];
            dbc[i] = s;
        }
        __syncthreads();
    } else {
        static_assert(BT == 1, "small calls take one sequence per workgroup");
        // thread -> (output, every G-th of the partial sums), sixteen requested together
        const int G = max(256 / P, 1), g = G > 1 ? threadIdx.x / P : 0;
        for (int i = G > 1 ? threadIdx.x % P : threadIdx.x; i < P && g < G; i += 256) {
            const float* src = p.dbc + (int64_t)b0 * P + i;
            const int64_t pitch = (int64_t)p.batch * P;
            float s = 0.0f;
            for (int q0 = g; q0 < p.splits; q0 += 16 * G) {
                float v[16];
#pragma unroll
                for (int j = 0; j < 16; ++j) v[j] = src[min(q0 + j * G, p.splits - 1) * pitch];
#pragma unroll
                for (int j = 0; j < 16; ++j)
                    if (q0 + j * G < p.splits) s += v[j];
            }
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
            store_from_float<IO>(p.g, frag_at<IO>(b, d, p.ED), __builtin_fmaf(Dv, xv[t], acc) * zv[t] * sigmoid_f(zv[t]));
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

// Workgroup tiles, from a sweep over row tiles, batch tiles, waves and pieces in flight at widths 768 and
// 2560 and batches 1, 64 and 128.  One 16 x 16 tile on eight waves, one piece ahead (U = 1), is best or
// within 5 % nearly everywhere: more tiles or pieces per wave cost the registers of a second workgroup
// per CU, which hides more (in_proj at 64 x 768, bfloat16: 6.1 us, 8.7 us with U = 2).  in_proj with more
// than 1536 tiles takes two batch tiles per workgroup (128 x 768: 8.6 us on four waves, 10.0 with one
// tile), on eight waves where K is long (64 x 2560, float32: 55 us, 62 on four).
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
        hipLaunchKernelGGL((decode_in_kernel<IO, 1, 8, 1, MODE, true>), decode_grid(rt, bt, 1), dim3(512), 0, st, p, rt, bt);
    } else if (rt * bt < kManyTiles) {
        hipLaunchKernelGGL((decode_in_kernel<IO, 1, 8, 1, MODE>), decode_grid(rt, bt, 1), dim3(512), 0, st, p, rt, bt);
    } else {
        const int groups = (bt + 1) / 2;
        const dim3 grid = decode_grid(rt, groups, 1);
        if (p.d > 16 * 8 * Frag<IO>::kVec) hipLaunchKernelGGL((decode_in_kernel<IO, 2, 8, 1, MODE>), grid, dim3(512), 0, st, p, rt, groups);
        else hipLaunchKernelGGL((decode_in_kernel<IO, 2, 4, 1, MODE>), grid, dim3(256), 0, st, p, rt, groups);
    }
    return check_launch();
}

template <typename IO>
static int launch_xproj(const DecodeParams& p, hipStream_t st) {
    const int rt = (p.R + 2 * p.N + 15) / 16, bt = (p.batch + 15) / 16;
    hipLaunchKernelGGL((decode_xproj_kernel<IO, kXprojWaves>), decode_grid(rt, bt, p.splits), dim3(kXprojWaves * kWave), 0, st, p, rt, bt);
    return check_launch();
}

// out_proj has half the rows and twice the K: sixteen waves while one workgroup per CU is all there is
// (1 x 768: 4.6 us, 4.8 on eight; 1 x 2560 float32: 16.2, 18.7).
template <typename IO, bool RES>
static int launch_out(const DecodeParams& p, hipStream_t st) {
    const int rt = (p.d + 15) / 16, bt = (p.batch + 15) / 16;
    const dim3 grid = decode_grid(rt, bt, 1);
    if (rt * bt <= 256) hipLaunchKernelGGL((decode_out_kernel<IO, 1, 16, 1, RES>), grid, dim3(1024), 0, st, p, rt, bt);
    else hipLaunchKernelGGL((decode_out_kernel<IO, 1, 8, 1, RES>), grid, dim3(512), 0, st, p, rt, bt);
    return check_launch();
}

template <typename IO, int BT>
static int launch_ssm(const DecodeParams& p, hipStream_t st) {
    const dim3 grid((p.ED + 63) / 64, (p.batch + BT - 1) / BT);
    const int outs = BT * (p.R + 2 * p.N);
    const size_t lds = (size_t)(outs < 256 ? 256 : outs) * sizeof(float);
    if (lds > 48 * 1024) return MPA_ERR_BAD_SHAPE;
    const bool v4 = p.R % 4 == 0 && aligned_to(p.dt_w, 4 * sizeof(IO));
    const bool many = BT == 1 && xproj_fused(p.ED, p.R + 2 * p.N, p.batch);
#define MPA_SSM(N16_, V_)                                                                                              \
    do {                                                                                                               \
        if (many) hipLaunchKernelGGL((decode_ssm_kernel<IO, 1, N16_, V_, true>), grid, dim3(256), lds, st, p);         \
        else hipLaunchKernelGGL((decode_ssm_kernel<IO, BT, N16_, V_, false>), grid, dim3(256), lds, st, p);            \
    } while (0)
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
    if (!xproj_fused(p.ED, p.R + 2 * p.N, p.batch)) rc = launch_xproj<IO>(p, st);
    if (rc != MPA_OK) return rc;
    // sequences per workgroup: four (weights and A read once for them) while that leaves two
    // workgroups per CU
    const int64_t cols = (p.ED + 63) / 64;
    rc = cols * ((p.batch + 3) / 4) >= 512 ? launch_ssm<IO, 4>(p, st)
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
