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
template <typename IO>
__device__ __forceinline__ auto ld_bits(rsrc_t r, uint32_t at) {
    if constexpr (sizeof(IO) == 4) return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, at, 0, 0);
    else return (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, at, 0, 0);
}
__device__ __forceinline__ float ld_f32(rsrc_t r, uint32_t at, bool ok) {
    asm("" : "+v"(at));  // (formed either way: or the choice becomes a branch around its arithmetic, and around the load)
    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, ok ? at : 0xffffffe0u, 0, 0));
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
template <typename IO>
__device__ __forceinline__ float frag_load(const void* base, int b, int k, int K) {
    return load_as_float<IO>(base, frag_at<IO>(b, k, K));
}
// An offset beyond any window here (they are below 2 GB): the load reads zero, with a scalar offset on top as well.
constexpr uint32_t kNowhere = 0x80000000u;
// (formed either way: or the choice becomes a branch around its arithmetic, and around the load)
__device__ __forceinline__ uint32_t where(bool ok, uint32_t at) {
    asm("" : "+v"(at));
    return ok ? at : kNowhere;
}

// Activations in operand order; request() takes a chunk of 32 k, of which `left` are wanted (any number, also below zero).  Offsets
// within a chunk are formed once, the chunk is a scalar offset.
template <typename IO, int NT>
struct FragAct {
    static constexpr int kLoads = 8 / Frag<IO>::kVec;
    struct Raw {
        u32x4 x[kLoads];
    };
    rsrc_t r;
    uint32_t at[NT];
    int kl;
    __device__ __forceinline__ void setup(const void* base, int b0, int batch, int K, int lane) {
        const uint32_t tile = (uint32_t)((K + 31) / 32) * (512u * sizeof(IO));
        r = make_rsrc(static_cast<const char*>(base) + (int64_t)(b0 >> 4) * tile, (uint32_t)(((batch - b0 + 15) >> 4) * tile));
        kl = 8 * (lane >> 4);
#pragma unroll
        for (int t = 0; t < NT; ++t)  // (one sequence then reads a sixteenth of its tile)
            at[t] = b0 + t * 16 + (lane & 15) < batch ? t * tile + lane * 16u : kNowhere;
    }
    __device__ __forceinline__ void request(Raw& v, int t, int chunk, int left) {
        const uint32_t from = kl < left ? at[t] : kNowhere;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) v.x[i] = __builtin_amdgcn_raw_buffer_load_b128(r, from + i * 1024u, (uint32_t)(chunk * kLoads) * 1024u, 0);
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
    int kl;
    bool gain;
    float ss[NT];
    __device__ __forceinline__ void setup(const void* base, const float* w, int b0, int batch, int K, int lane) {
        r = window(base, (int64_t)batch * K, sizeof(IO));
        rw = window(w, K, 4);
        gain = w != nullptr;
        kl = 8 * (lane >> 4);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int b = b0 + t * 16 + (lane & 15);
            at[t] = b < batch ? ((uint32_t)b * (uint32_t)K + kl) * (uint32_t)sizeof(IO) : kNowhere;
            ss[t] = 0.0f;
        }
    }
    __device__ __forceinline__ void request(Raw& v, int t, int chunk, int left) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            v.x[i] = __builtin_amdgcn_raw_buffer_load_b128(r, (kl + i * kVec < left ? at[t] : kNowhere) + i * 16u, (uint32_t)chunk * 32u * (uint32_t)sizeof(IO), 0);
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
                v.w[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rw, kl + 4 * i < left ? (uint32_t)(kl + 4 * i) * 4u : kNowhere, (uint32_t)chunk * 128u, 0));
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
    float s[NW];
#pragma unroll
    for (int w = 0; w < NW; ++w) s[w] = lds[w].v[at];
#pragma unroll
    for (int o = 1; o < NW; o *= 2)  // (pairs: additions in a row are 9 clocks each)
#pragma unroll
        for (int w = 0; w + o < NW; w += 2 * o) s[w] += s[w + o];
    return s[0];
}
// sum over the 16 lanes of a row, in all of them
__device__ __forceinline__ float row_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x124, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x122, 0xf, 0xf, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x121, 0xf, 0xf, true));
    return v;
}

// Rows n0 .. n0+16*MT-1 of `W . x^T` for NT batch tiles, over the 128-byte pieces first + wave, + NW, ...
// below `last` of the rows of W; the wave leaves its partial tiles in its LDS.  U pieces are in flight (`more` issues the caller's own
// loads behind them), each with its activations: loads return in the order they were issued, so
// activations requested later than weights of pieces further on would wait for those as well.
// ONCE: no wave has more than U pieces, and there is no loop.
// What a wave does before its first load and between the last one's arrival and its result is time that nothing hides (a wave
// issues an instruction every five clocks at best, and a step of one sequence is a chain of such kernels): offsets of lanes are formed
// once, pieces are scalar offsets, what lies beyond the rows or beyond K reads zero.
template <typename IO, int NW, int U, bool ONCE, int MT, int NT, typename ACT, typename MORE>
__device__ __forceinline__ void decode_product(WaveLds<MT, NT>& lds, const void* W, int rows, int K, int n0, int first, int last, int wave,
                                               int lane, ACT& act, MORE&& more) {
    constexpr int kVec = Frag<IO>::kVec, kES = sizeof(IO);
    char* const slot = reinterpret_cast<char*>(lds.v);
    // lane -> 16 bytes of row 8*i + lane/8: the piece's eight 16-byte parts are stored rotated by the row
    // (part ^ (row & 7)), so that the operand reads, one row per lane, fall on different banks
    const int part = ((lane & 7) ^ (lane >> 3)) * 16;
    // (a scalar, which the compiler's v_med3 is not: every load would be a loop over the lanes' descriptors)
    const uint32_t rows_left = (uint32_t)__builtin_amdgcn_readfirstlane(max(min(rows - n0, 16 * MT), 0));
    const rsrc_t rw = make_rsrc(static_cast<const IO*>(W) + (int64_t)n0 * K, rows_left * (uint32_t)K * kES);
    uint32_t row[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) row[i] = (uint32_t)(lane >> 3) * (uint32_t)K * kES + part + (uint32_t)(8 * i * K) * kES;
    constexpr int kOps = Frag<IO>::kOps, kReads = 2 / kOps;  // operands of a piece; 16-byte parts of one
    const int k_end = min(last * 8 * kVec, K);

    struct Piece {
        u32x4 w[2 * MT];
        typename ACT::Raw a[NT][kOps];
    };
    Piece r[U];
    auto request = [&](Piece& v, int s) {
        const int piece = first + wave + s * NW;
        const bool ok = part < k_end * kES - piece * 128;
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) v.w[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, ok ? row[i] : kNowhere, (uint32_t)piece * 128u, 0);
#pragma unroll
        for (int h = 0; h < kOps; ++h) {
            const int chunk = kOps * piece + h;
#pragma unroll
            for (int t = 0; t < NT; ++t) act.request(v.a[t][h], t, chunk, k_end - chunk * 32);
        }
    };
    f32x4 acc[MT][NT] = {};
    int frag[kOps][kReads];
#pragma unroll
    for (int h = 0; h < kOps; ++h)
#pragma unroll
        for (int i = 0; i < kReads; ++i) frag[h][i] = (lane & 15) * 128 + ((((lane >> 4) * kReads + i + 4 * h) ^ (lane & 7)) << 4);
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
    if constexpr (ONCE) {
        // (all pieces; what lies beyond the last are zeros)
#pragma unroll
        for (int u = 0; u < U; ++u) multiply(r[u], u);
    } else {
        const int count = first + wave < last ? (last - first - wave + NW - 1) / NW : 0;  // pieces of this wave
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
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m) *reinterpret_cast<f32x4*>(&lds.v[(t * MT + m) * 256 + 4 * lane]) = acc[m][t];
}

struct DecodeParams {
    int batch, d, ED, N, R, K;  // K: convolution taps
    int P4;         // dt_rank + 2 d_state to a multiple of four: pitch of dbc
    uint32_t span_inv;  // of a launch's tiles, see decode_tile
    int groups;
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
    float* dbc;        // [splits][batch][P4]
    void* y;
    const float* next_w;  // norm weight of the next layer, with y_w and ssq_out
    void* y_w;
    float* ssq_out;
};

// What decode_in_kernel does with x: as it is, normalised here, or normalised by the kernel before.
enum { kInPlain, kInNorm, kInReady };

// grid: (row tiles) x (batch tile groups), batch groups of one row tile eight blocks apart: the
// blocks of an XCD (every eighth) then meet the same rows of W again in their own L2.  (id / (8 * groups) as a product with
// span_inv = 2^32 / (8 * groups) rounded up, exact below 2^25 blocks.)  A tile beyond the last has no rows: it reads zeros and stores nothing.
template <int NT>
__device__ __forceinline__ void decode_tile(const DecodeParams& p, int& rt, int& bt) {
    const uint32_t id = blockIdx.x, g = __umulhi(id, p.span_inv), in = id - g * 8u * (uint32_t)p.groups;
    rt = (int)(g * 8 + (in & 7));
    bt = (int)(in >> 3) * NT;
}

template <typename IO>
__device__ __forceinline__ void st_io(rsrc_t r, uint32_t at, IO v) {
    if constexpr (sizeof(IO) == 4) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, at, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, v), r, at, 0, 0);
}
// byte offset of an activation in operand order, and its store (with the zeros after the last four of a float32 row whose eight are not whole)
template <typename IO>
__device__ __forceinline__ uint32_t frag_offset(int b, int k, int K) {
    constexpr uint32_t kVec = Frag<IO>::kVec;
    const uint32_t tile = (uint32_t)(b >> 4) * (uint32_t)((K + 31) / 32) + ((uint32_t)k >> 5);
    return (uint32_t)sizeof(IO) * (tile * 512u + ((uint32_t)k % 8 / kVec) * (64 * kVec) + ((b & 15) + 16 * ((uint32_t)k % 32 / 8)) * kVec + (uint32_t)k % kVec);
}
template <typename IO>
__device__ __forceinline__ void frag_store_at(rsrc_t r, uint32_t at, int k, int K, IO v) {
    st_io<IO>(r, at, v);
    if constexpr (sizeof(IO) == 4) st_io<float>(r, k % 8 < 4 && k + 4 >= K ? at + 1024u : kNowhere, 0.0f);
}
// n / d for n < 2^20: (n + 1/2) / d is at least 1 / 2d from a whole number, and off by n / d * 2^-22 at most
__device__ __forceinline__ int div_small(int n, int d) { return (int)(((float)n + 0.5f) * __builtin_amdgcn_rcpf((float)d)); }

// XP: also the workgroup's share of x_proj, its 16 channels' product with all rows of x_proj's weight, as one
// more partial sum of dbc; a thread owns one row and every so many sequences (there are as many threads as rows, or more).
template <typename IO, int MT, int NT, int NW, int U, bool ONCE, int MODE, bool XP = false>
__global__ void __launch_bounds__(NW* kWave) decode_in_kernel(const DecodeParams p) {
    constexpr int kThreads = NW * kWave, kRows = MT * 16, kAll = NT * 16 * kRows, kOuts = (kAll + kThreads - 1) / kThreads;
    static_assert(!XP || MT == 1, "x_proj by 16 channels");
    __shared__ WaveLds<MT, NT> tile[NW];
    __shared__ float ssq[NW][NT][16];
    __shared__ alignas(16) float xl[XP ? NT * 16 : 1][16];  // convolved x of the tile
    // (all arguments requested at once: the compiler otherwise loads some where they are used, each a round trip in a step's chain)
    asm volatile("" ::"s"(p.batch), "s"(p.d), "s"(p.ED), "s"(p.N), "s"(p.R), "s"(p.K), "s"(p.P4), "s"(p.span_inv), "s"(p.groups), "s"(p.eps),
                 "s"(p.ssq_tiles), "s"(p.x), "s"(p.xw), "s"(p.ssq), "s"(p.norm_w), "s"(p.in_w), "s"(p.in_b), "s"(p.conv_w), "s"(p.conv_b), "s"(p.xp_w),
                 "s"(p.win_in), "s"(p.win_out), "s"(p.xs), "s"(p.z), "s"(p.dbc));
    int rt, bt;
    decode_tile<NT>(p, rt, bt);
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * kRows, b0 = bt * 16, rows = 2 * p.ED;
    const int pieces = (p.d + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    // the epilogue's operands: thread -> outputs (row o % kRows, sequence o / kRows), and where its results go
    IO win[kOuts][3], ib[kOuts];
    float cw[kOuts][4], cb[kOuts];
    uint32_t to_win[kOuts], to_z[kOuts], to_xs[kOuts];
    float ss[NT] = {};
    const int P = p.R + 2 * p.N;
    int xrow = 0, xgroup = 0;
    u32x4 xw[XP ? 16 / Frag<IO>::kVec : 1];
    // wave w, lane group q: partial sums of squares 4w + q, 4w + q + 4*NW, ... of column lane % 16, up to a width of 1024 requested together
    // and ahead of the product
    constexpr int kSums = NW >= 16 ? 1 : 16 / NW;
    const rsrc_t rs = window(p.ssq, (int64_t)p.ssq_tiles * p.batch, 4);
    float sq[NT][kSums];
    auto request_sums = [&](int q0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int b = b0 + t * 16 + (lane & 15);
            const uint32_t at = ((uint32_t)(q0 + 4 * wave + (lane >> 4)) * (uint32_t)p.batch + (uint32_t)b) * 4u, step = 16u * NW * (uint32_t)p.batch;
#pragma unroll
            for (int i = 0; i < kSums; ++i)  // (beyond the last row of sums is beyond the window)
                sq[t][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, where(b < p.batch, at + i * step), 0, 0));
        }
    };
    const rsrc_t rwo = window(p.win_out, (int64_t)p.batch * p.ED * (p.K - 1), sizeof(IO)), rz = window(p.z, (int64_t)p.batch * p.ED, sizeof(IO)),
                 rxs = make_rsrc(p.xs, (uint32_t)frag_bytes(p.batch, p.ED, sizeof(IO)));
    auto more = [&] {
        if constexpr (MODE == kInReady) request_sums(0);
        const rsrc_t rb = window(p.in_b, rows, sizeof(IO)), rwin = window(p.win_in, (int64_t)p.batch * p.ED * (p.K - 1), sizeof(IO)),
                     rcw = window(p.conv_w, (int64_t)p.ED * p.K, 4), rcb = window(p.conv_b, p.ED, 4);
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % kRows, b = b0 + o / kRows;
            const bool some = (kOuts * kThreads == kAll || o < kAll) && n < rows && b < p.batch, conv = some && n < p.ED;
            const uint32_t at = (uint32_t)b * (uint32_t)p.ED + (uint32_t)n;
            to_win[i] = where(conv, at * (uint32_t)(p.K - 1) * (uint32_t)sizeof(IO));
            to_z[i] = where(some && n >= p.ED, (at - (uint32_t)p.ED) * (uint32_t)sizeof(IO));
            to_xs[i] = where(conv, frag_offset<IO>(b, n, p.ED));
            ib[i] = __builtin_bit_cast(IO, ld_bits<IO>(rb, (uint32_t)n * (uint32_t)sizeof(IO)));
            // (taps that the layer does not have are read from what follows, and not used)
#pragma unroll
            for (int j = 0; j < 3; ++j) win[i][j] = __builtin_bit_cast(IO, ld_bits<IO>(rwin, to_win[i] + j * (uint32_t)sizeof(IO)));
            const uint32_t cat = where(conv, (uint32_t)(n * p.K) * 4u);
#pragma unroll
            for (int j = 0; j < 4; ++j) cw[i][j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rcw, cat + 4u * j, 0, 0));
            cb[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rcb, (uint32_t)n * 4u, 0, 0));
        }
        if constexpr (XP) {
            xgroup = div_small(threadIdx.x, P);
            xrow = (int)threadIdx.x - xgroup * P;
            const rsrc_t rx = window(p.xp_w, (int64_t)P * p.ED, sizeof(IO));
#pragma unroll
            for (int i = 0; i < 16 / Frag<IO>::kVec; ++i) {  // (zeros beyond the last channel)
                const int k = n0 + i * Frag<IO>::kVec;
                xw[i] = __builtin_amdgcn_raw_buffer_load_b128(rx, where(k < p.ED, (uint32_t)(xrow * p.ED + k) * (uint32_t)sizeof(IO)), 0, 0);
            }
        }
    };
    if constexpr (MODE == kInReady) {
        FragAct<IO, NT> act;
        act.setup(p.xw, b0, p.batch, p.d, lane);
        decode_product<IO, NW, U, ONCE>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
        for (int q0 = 0;; request_sums(q0)) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < kSums; ++i) ss[t] += sq[t][i];
            if ((q0 += 4 * NW * kSums) >= p.ssq_tiles) break;
        }
    } else {
        RowAct<IO, NT, MODE == kInNorm> act;
        act.setup(p.x, p.norm_w, b0, p.batch, p.d, lane);
        decode_product<IO, NW, U, ONCE>(tile[wave], p.in_w, rows, p.d, n0, 0, pieces, wave, lane, act, more);
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
        const int o = threadIdx.x + i * kThreads, row = o % kRows, bl = o / kRows, n = n0 + row;
        if (kOuts * kThreads != kAll && o >= kAll) break;  // uniform over a wave
        float v = tile_sum(tile, row, bl);
        if constexpr (MODE != kInPlain) {
            float s = ssq[0][bl >> 4][bl & 15];
#pragma unroll
            for (int w = 1; w < NW; ++w) s += ssq[w][bl >> 4][bl & 15];
            v *= __builtin_amdgcn_rsqf(s / (float)p.d + p.eps);
        }
        const IO vr = from_float<IO>(v + to_float(ib[i]));
        if (n0 >= p.ED) {  // uniform over the block
            st_io<IO>(rz, to_z[i], vr);
            continue;
        }
        // newest tap first, then the window from its newest input backwards
        float c = cb[i];
        IO keep[3] = {win[i][1], win[i][2], vr};  // the window after this step
        if (p.K == 4) {
            c = __builtin_fmaf(cw[i][3], to_float(vr), c);
#pragma unroll
            for (int j = 2; j >= 0; --j) c = __builtin_fmaf(cw[i][j], to_float(win[i][j]), c);
        } else if (p.K == 3) {
            c = __builtin_fmaf(cw[i][2], to_float(vr), c);
            c = __builtin_fmaf(cw[i][1], to_float(win[i][1]), c);
            c = __builtin_fmaf(cw[i][0], to_float(win[i][0]), c);
            keep[1] = vr;
        } else {
            c = __builtin_fmaf(cw[i][1], to_float(vr), c);
            c = __builtin_fmaf(cw[i][0], to_float(win[i][0]), c);
            keep[0] = vr;
        }
        c *= sigmoid_f(c);
        const IO cr = from_float<IO>(c);
        if constexpr (XP) xl[bl][row] = n < p.ED ? to_float(cr) : 0.0f;
        frag_store_at<IO>(rxs, to_xs[i], n, p.ED, cr);
        st_io<IO>(rz, to_z[i], vr);  // (of a tile with the last channels of x and the first of z)
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (j < p.K - 1) st_io<IO>(rwo, to_win[i] + j * (uint32_t)sizeof(IO), keep[j]);
    }
    if constexpr (XP) {
        if (n0 >= p.ED) return;  // uniform over the block
        __syncthreads();
        const int G = div_small(kThreads, P), nb = min(p.batch - b0, NT * 16);
        if (xgroup >= G) return;
        float w[16];
#pragma unroll
        for (int i = 0; i < 16 / Frag<IO>::kVec; ++i) {
            float part[Frag<IO>::kVec];
            Frag<IO>::unpack(xw[i], part);
#pragma unroll
            for (int e = 0; e < Frag<IO>::kVec; ++e) w[i * Frag<IO>::kVec + e] = part[e];
        }
        for (int b = xgroup; b < nb; b += G) {
            float s[4] = {};  // (four chains of four)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[i] = __builtin_fmaf(w[4 * i + e], xl[b][4 * i + e], s[i]);
            p.dbc[((int64_t)rt * p.batch + b0 + b) * p.P4 + xrow] = (s[0] + s[1]) + (s[2] + s[3]);
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

template <typename IO, int NW, int U, bool ONCE>
__global__ void __launch_bounds__(NW* kWave) decode_xproj_kernel(const DecodeParams p) {
    __shared__ WaveLds<1, 1> tile[NW];
    // (all arguments requested at once: the compiler otherwise loads some where they are used, each a round trip in a step's chain)
    asm volatile("" ::"s"(p.batch), "s"(p.ED), "s"(p.N), "s"(p.R), "s"(p.P4), "s"(p.span_inv), "s"(p.groups), "s"(p.splits), "s"(p.xp_w), "s"(p.xs), "s"(p.dbc));
    int rt, bt;
    decode_tile<1>(p, rt, bt);
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id(), rows = p.R + 2 * p.N;
    const int pieces = (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec);
    const int per = (pieces + p.splits - 1) / p.splits, first = (int)blockIdx.y * per;
    const int o = threadIdx.x, n = rt * 16 + (o & 15), b = bt * 16 + (o >> 4);
    const rsrc_t rd = make_rsrc(p.dbc + (int64_t)blockIdx.y * p.batch * p.P4, (uint32_t)(p.batch * p.P4) * 4u);
    const uint32_t to = where(o < 256 && n < rows && b < p.batch, (uint32_t)(b * p.P4 + n) * 4u);
    FragAct<IO, 1> act;
    act.setup(p.xs, bt * 16, p.batch, p.ED, lane);
    decode_product<IO, NW, U, ONCE>(tile[wave], p.xp_w, rows, p.ED, rt * 16, first, min(pieces, first + per), wave, lane, act, [] {});
    __syncthreads();
    if (wave >= 4) return;
    st_io<float>(rd, to, tile_sum(tile, o & 15, o >> 4));
}

// y = out_proj(g) [+ x]; with next_w also y * next_w and the sums of squares of 16 columns each
template <typename IO, int MT, int NT, int NW, int U, bool ONCE, bool RES>
__global__ void __launch_bounds__(NW* kWave) decode_out_kernel(const DecodeParams p) {
    constexpr int kThreads = NW * kWave, kRows = MT * 16, kAll = NT * 16 * kRows, kOuts = (kAll + kThreads - 1) / kThreads;
    __shared__ WaveLds<MT, NT> tile[NW];
    // (all arguments requested at once: the compiler otherwise loads some where they are used, each a round trip in a step's chain)
    asm volatile("" ::"s"(p.batch), "s"(p.d), "s"(p.ED), "s"(p.span_inv), "s"(p.groups), "s"(p.x), "s"(p.out_w), "s"(p.out_b), "s"(p.g), "s"(p.y), "s"(p.next_w),
                 "s"(p.y_w), "s"(p.ssq_out));
    int rt, bt;
    decode_tile<NT>(p, rt, bt);
    const int lane = threadIdx.x & (kWave - 1), wave = wave_id();
    const int n0 = rt * kRows, b0 = bt * 16;
    IO bias[kOuts], xv[kOuts];
    float nw[kOuts];
    uint32_t to[kOuts], to_yw[kOuts], to_ssq[kOuts];  // of y, y_w and ssq_out
    const bool next = RES && p.next_w;
    const rsrc_t ry = window(p.y, (int64_t)p.batch * p.d, sizeof(IO)), ryw = make_rsrc(p.y_w, next ? (uint32_t)frag_bytes(p.batch, p.d, sizeof(IO)) : 0u),
                 rso = window(next ? p.ssq_out : nullptr, (int64_t)((p.d + 15) / 16) * p.batch, 4);
    auto more = [&] {
        const rsrc_t rb = window(p.out_b, p.d, sizeof(IO)), rx = window(RES ? p.x : nullptr, (int64_t)p.batch * p.d, sizeof(IO)),
                     rn = window(RES ? p.next_w : nullptr, p.d, 4);
#pragma unroll
        for (int i = 0; i < kOuts; ++i) {
            const int o = threadIdx.x + i * kThreads, n = n0 + o % kRows, b = b0 + o / kRows;
            const bool ok = (kOuts * kThreads == kAll || o < kAll) && n < p.d && b < p.batch;
            to[i] = where(ok, (uint32_t)(b * p.d + n) * (uint32_t)sizeof(IO));
            to_yw[i] = where(ok, frag_offset<IO>(b, n, p.d));
            to_ssq[i] = where(ok && n % 16 == 0, (uint32_t)((n >> 4) * p.batch + b) * 4u);
            bias[i] = __builtin_bit_cast(IO, ld_bits<IO>(rb, (uint32_t)n * (uint32_t)sizeof(IO)));
            xv[i] = __builtin_bit_cast(IO, ld_bits<IO>(rx, to[i]));
            nw[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rn, (uint32_t)n * 4u, 0, 0));
        }
    };
    FragAct<IO, NT> act;
    act.setup(p.g, b0, p.batch, p.ED, lane);
    decode_product<IO, NW, U, ONCE>(tile[wave], p.out_w, p.d, p.ED, n0, 0, (p.ED + 8 * Frag<IO>::kVec - 1) / (8 * Frag<IO>::kVec), wave,
                                    lane, act, more);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOuts; ++i) {
        const int o = threadIdx.x + i * kThreads, row = o % kRows, bl = o / kRows, n = n0 + row;
        if (kOuts * kThreads != kAll && o >= kAll) break;  // uniform over a wave
        IO v = from_float<IO>(tile_sum(tile, row, bl) + to_float(bias[i]));
        if constexpr (RES) {
            v = from_float<IO>(to_float(v) + to_float(xv[i]));
            if (next) {
                const float f = n < p.d ? to_float(v) : 0.0f;
                frag_store_at<IO>(ryw, to_yw[i], n, p.d, from_float<IO>(f * nw[i]));
                st_io<float>(rso, to_ssq[i], row_sum(f * f));
            }
        }
        st_io<IO>(ry, to[i], v);
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
    // (all arguments requested at once: the compiler otherwise loads some where they are used, each a round trip in a step's chain)
    asm volatile("" ::"s"(p.batch), "s"(p.ED), "s"(p.N), "s"(p.R), "s"(p.P4), "s"(p.splits), "s"(p.dt_w), "s"(p.dt_b), "s"(p.A), "s"(p.D), "s"(p.h_in), "s"(p.h_out),
                 "s"(p.xs), "s"(p.z), "s"(p.g), "s"(p.dbc));
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
        const rsrc_t parts = window(p.dbc, (int64_t)p.splits * p.batch * p.P4, 4);
        for (int i = threadIdx.x; i < BT * P; i += 256) {
            const int t = div_small(i, P), b = b0 + t;
            float v[8], s = 0.0f;  // (requested together)
#pragma unroll
            for (int q = 0; q < 8; ++q)
                v[q] = ld_f32(parts, (uint32_t)((q * p.batch + b) * p.P4 + (i - t * P)) * 4u, b < p.batch && q < p.splits);
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
            const int64_t pitch = (int64_t)p.batch * p.P4;
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
            const float* src = p.dbc + (int64_t)b0 * p.P4 + i;
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
            frag_store_at<IO>(make_rsrc(p.g, (uint32_t)frag_bytes(p.batch, p.ED, sizeof(IO))), frag_offset<IO>(b, d, p.ED), d, p.ED,
                              from_float<IO>(__builtin_fmaf(Dv, xv[t], acc) * zv[t] * sigmoid_f(zv[t])));
    }
}

// The same where dbc comes as many partial sums, 16 states: a row of 16 lanes owns CH channels of one sequence, a lane one of their states and
// a sixteenth of dt_rank.  For one sequence it is a chain of latencies, and short: the partial sums in 16-byte parts,
// eight or fewer to a thread, three products, one exponential and two sums over a row of lanes (four states a lane, a thread
// for every output and 32 partial sums each: 3.4 us from the first instruction to the last, 1400 instructions).
template <typename IO, int CH>
__global__ void __launch_bounds__(256) decode_ssm_row_kernel(const DecodeParams p) {
    extern __shared__ float lds[];  // [groups][P4] partial sums; then their sums in front
    // (all arguments requested at once: the compiler otherwise loads some where they are used, each a round trip in a step's chain)
    asm volatile("" ::"s"(p.batch), "s"(p.ED), "s"(p.R), "s"(p.P4), "s"(p.splits), "s"(p.dt_w), "s"(p.dt_b), "s"(p.A), "s"(p.D), "s"(p.h_in), "s"(p.h_out), "s"(p.xs),
                 "s"(p.z), "s"(p.g), "s"(p.dbc));
    const int b = blockIdx.y, n = threadIdx.x & 15, parts4 = p.P4 >> 2;
    const int G = div_small(256, parts4), g = div_small(threadIdx.x, parts4), quad = (int)threadIdx.x - g * parts4;
    const rsrc_t rp = make_rsrc(p.dbc + (int64_t)b * p.P4, (uint32_t)(((p.splits - 1) * p.batch + 1) * p.P4) * 4u);
    const uint32_t pitch = (uint32_t)(p.batch * p.P4) * 4u;
    const uint32_t at = g < G ? (uint32_t)g * pitch + (uint32_t)quad * 16u : kNowhere;
    constexpr int kSome = 8, kPre = 4;
    u32x4 v[kSome];
    auto request = [&](int q0) {  // (beyond the last partial sum is beyond the window)
#pragma unroll
        for (int i = 0; i < kSome; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(rp, at == kNowhere ? kNowhere : at + (uint32_t)(q0 + i * G) * pitch, 0, 0);
    };
    request(0);
    IO xv[CH], zv[CH], w[CH][kPre];
    float h[CH], a[CH], Dv[CH], bias[CH];
    const rsrc_t rx = make_rsrc(p.xs, (uint32_t)frag_bytes(p.batch, p.ED, sizeof(IO))), rz = window(p.z, (int64_t)p.batch * p.ED, sizeof(IO)),
                 rw = window(p.dt_w, (int64_t)p.ED * p.R, sizeof(IO)), rA = window(p.A, (int64_t)p.ED * 16, 4), rD = window(p.D, p.ED, 4),
                 rb = window(p.dt_b, p.ED, 4), rg = make_rsrc(p.g, (uint32_t)frag_bytes(p.batch, p.ED, sizeof(IO)));
    const int64_t row0 = (int64_t)b * p.ED;
    const rsrc_t rh = window(p.h_in ? p.h_in + row0 * 16 : nullptr, (int64_t)p.ED * 16, 4), ro = make_rsrc(p.h_out + row0 * 16, (uint32_t)p.ED * 64u);
    int ch[CH];
    uint32_t frag[CH];
#pragma unroll
    for (int j = 0; j < CH; ++j) {  // (a channel beyond the last is beyond the windows of its rows)
        const int d = ch[j] = (blockIdx.x * CH + j) * 16 + (threadIdx.x >> 4);
        frag[j] = d < p.ED ? frag_offset<IO>(b, d, p.ED) : kNowhere;
        xv[j] = __builtin_bit_cast(IO, ld_bits<IO>(rx, frag[j]));
        zv[j] = __builtin_bit_cast(IO, ld_bits<IO>(rz, d < p.ED ? (uint32_t)(row0 + d) * (uint32_t)sizeof(IO) : kNowhere));
        h[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rh, (uint32_t)(d * 16 + n) * 4u, 0, 0));
        a[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rA, (uint32_t)(d * 16 + n) * 4u, 0, 0));
        Dv[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rD, (uint32_t)d * 4u, 0, 0));
        bias[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, (uint32_t)d * 4u, 0, 0));
#pragma unroll
        for (int i = 0; i < kPre; ++i)
            w[j][i] = __builtin_bit_cast(IO, ld_bits<IO>(rw, n + 16 * i < p.R ? (uint32_t)(d * p.R + n + 16 * i) * (uint32_t)sizeof(IO) : kNowhere));
    }
    f32x4 s = {};
    for (int q0 = 0;; request(q0)) {
        f32x4 t[kSome];
#pragma unroll
        for (int i = 0; i < kSome; ++i) t[i] = __builtin_bit_cast(f32x4, v[i]);
#pragma unroll
        for (int o = 1; o < kSome; o *= 2)
#pragma unroll
            for (int i = 0; i < kSome; i += 2 * o) t[i] += t[i + o];
        s += t[0];
        if ((q0 += kSome * G) >= p.splits) break;
    }
    float* const sums = lds + G * p.P4;
    if (g < G) *reinterpret_cast<f32x4*>(lds + g * p.P4 + quad * 4) = s;
    __syncthreads();
    for (int i = threadIdx.x; i < p.P4; i += 256) {
        float t[4] = {};
        for (int q = 0; q < G; q += 4)
#pragma unroll
            for (int e = 0; e < 4; ++e) t[e] += q + e < G ? lds[(q + e) * p.P4 + i] : 0.0f;
        sums[i] = (t[0] + t[1]) + (t[2] + t[3]);
    }
    __syncthreads();
    const float Bn = sums[p.R + n], Cn = sums[p.R + 16 + n];
    float low[kPre];
#pragma unroll
    for (int i = 0; i < kPre; ++i) low[i] = n + 16 * i < p.R ? sums[n + 16 * i] : 0.0f;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
        float dl = 0.0f;
#pragma unroll
        for (int i = 0; i < kPre; ++i) dl = __builtin_fmaf(to_float(w[j][i]), low[i], dl);
        for (int r = n + 16 * kPre; r < p.R; r += 16)
            dl = __builtin_fmaf(to_float(__builtin_bit_cast(IO, ld_bits<IO>(rw, (uint32_t)(ch[j] * p.R + r) * (uint32_t)sizeof(IO)))), sums[r], dl);
        const float delta = softplus_f(row_sum(dl) + bias[j]), x = to_float(xv[j]), z = to_float(zv[j]);
        const float hn = __builtin_fmaf(delta * x, Bn, fast_exp2(delta * kLog2e * a[j]) * h[j]);
        st_io<float>(ro, (uint32_t)(ch[j] * 16 + n) * 4u, hn);
        const float y = row_sum(Cn * hn);
        frag_store_at<IO>(rg, n == 0 ? frag[j] : kNowhere, ch[j], p.ED, from_float<IO>(__builtin_fmaf(Dv[j], x, y) * z * sigmoid_f(z)));
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

// grid of a product: sets what decode_tile reads
static dim3 decode_grid(DecodeParams& p, int row_tiles, int groups, int splits = 1) {
    p.groups = groups;
    p.span_inv = (uint32_t)((((uint64_t)1 << 32) + 8 * groups - 1) / (8 * groups));
    return dim3((unsigned)(groups == 1 ? row_tiles : (row_tiles + 7) / 8 * 8 * groups), (unsigned)splits);
}
// 128-byte pieces of a row of K elements
template <typename IO>
static int pieces_of(int K) { return (K + 128 / (int)sizeof(IO) - 1) / (128 / (int)sizeof(IO)); }

// One tile of rows and sequences: all pieces of a wave are in flight at once and nothing loops while four waves have three pieces each at
// most, then eight (layers of 1 x 768: bfloat16 13.8 us on eight looping waves -> 10.8, float32 17.0 -> 13.6; 64 x 768 20.8 -> 17.2;
// 1 x 256 10.8 -> 9.5, all with the other changes of the same kernels).  Above, as measured before: float32 four waves with more pieces in flight.
template <typename IO, int MODE>
static int launch_in(DecodeParams p, hipStream_t st) {
    const int rt = (2 * p.ED + 15) / 16, bt = (p.batch + 15) / 16, P = p.R + 2 * p.N, pieces = pieces_of<IO>(p.d);
    const bool fused = xproj_fused(p.ED, P, p.batch);
#define MPA_IN(MT_, NT_, NW_, U_, ONCE_, XP_, GROUPS_) \
    hipLaunchKernelGGL((decode_in_kernel<IO, MT_, NT_, NW_, U_, ONCE_, MODE, XP_>), decode_grid(p, rt, GROUPS_), dim3(NW_ * kWave), 0, st, p)
    if (fused) {
        // (Four waves have a thread for 256 rows of x_proj; more of them take eight at any width.)
        if (pieces <= 12 && P <= 256) MPA_IN(1, 1, 4, 3, true, true, bt);
        else if (pieces <= 24) MPA_IN(1, 1, 8, 3, true, true, bt);
        else if (sizeof(IO) == 4 && P <= 256) MPA_IN(1, 1, 4, 4, false, true, bt);
        else MPA_IN(1, 1, 8, 2, false, true, bt);
    } else if (rt * bt < kManyTiles) {
        if (pieces <= 12) MPA_IN(1, 1, 4, 3, true, false, bt);
        else if (pieces <= 24) MPA_IN(1, 1, 8, 3, true, false, bt);
        else MPA_IN(1, 1, 8, 2, false, false, bt);
    } else {
        const int groups = (bt + 1) / 2;
        // (four waves where eight would have two pieces each or fewer: 128 x 1000 in bfloat16 14.2 us on eight, 11.2 on four)
        if (p.d * (int)sizeof(IO) <= 2048) MPA_IN(1, 2, 4, 2, false, false, groups);
        else MPA_IN(1, 2, 8, 2, false, false, groups);
    }
#undef MPA_IN
    return check_launch();
}

template <typename IO>
static int launch_xproj(DecodeParams p, hipStream_t st) {
    const int rt = (p.R + 2 * p.N + 15) / 16, bt = (p.batch + 15) / 16, per = (pieces_of<IO>(p.ED) + p.splits - 1) / p.splits;
    const dim3 grid = decode_grid(p, rt, bt, p.splits);
    if (per <= kXprojWaves) hipLaunchKernelGGL((decode_xproj_kernel<IO, kXprojWaves, 1, true>), grid, dim3(kXprojWaves * kWave), 0, st, p);
    else hipLaunchKernelGGL((decode_xproj_kernel<IO, kXprojWaves, 2, false>), grid, dim3(kXprojWaves * kWave), 0, st, p);
    return check_launch();
}

// out_proj has half the rows and twice the K: while one workgroup per CU is all there is, as many waves as have three pieces each
// (see launch_in), or sixteen (1 x 2560 float32: 56 us a layer, 58 on eight), then two batch tiles on eight waves, and from 512 tiles two row tiles as well (64 x 1536: float32 61 -> 58 us a
// layer, 64 x 2560 123 -> 120; bfloat16 42 -> 40 and 80 -> 75).
template <typename IO, bool RES>
static int launch_out(DecodeParams p, hipStream_t st) {
    const int rt = (p.d + 15) / 16, bt = (p.batch + 15) / 16, groups = (bt + 1) / 2, pairs = (rt + 1) / 2, pieces = pieces_of<IO>(p.ED);
#define MPA_OUT(MT_, NT_, NW_, U_, ONCE_, TILES_, GROUPS_) \
    hipLaunchKernelGGL((decode_out_kernel<IO, MT_, NT_, NW_, U_, ONCE_, RES>), decode_grid(p, TILES_, GROUPS_), dim3(NW_ * kWave), 0, st, p)
    if (rt * bt <= 256) {
        if (pieces <= 12) MPA_OUT(1, 1, 4, 3, true, rt, bt);
        else if (pieces <= 24) MPA_OUT(1, 1, 8, 3, true, rt, bt);
        else if (pieces <= 48) MPA_OUT(1, 1, 16, 3, true, rt, bt);
        else MPA_OUT(1, 1, 16, 2, false, rt, bt);
    } else if (rt * bt < 512) MPA_OUT(1, 2, 8, 2, false, rt, groups);
    else MPA_OUT(2, 2, 8, 2, false, pairs, groups);
#undef MPA_OUT
    return check_launch();
}

template <typename IO, int BT, bool MANY = false>
static int launch_ssm(const DecodeParams& p, hipStream_t st) {
    if constexpr (MANY) {
        if (p.N == 16) {
            const int G = 256 / (p.P4 / 4);
            const size_t lds = (size_t)(G + 1) * p.P4 * sizeof(float);
            const int tiles = (p.ED + 15) / 16;
            // (four channels a lane from two workgroups per CU on: the sums of dbc are then formed a quarter as often)
            if (tiles * p.batch <= 512) hipLaunchKernelGGL((decode_ssm_row_kernel<IO, 1>), dim3(tiles, p.batch), dim3(256), lds, st, p);
            else hipLaunchKernelGGL((decode_ssm_row_kernel<IO, 4>), dim3((tiles + 3) / 4, p.batch), dim3(256), lds, st, p);
            return check_launch();
        }
    }
    const dim3 grid((p.ED + 63) / 64, (p.batch + BT - 1) / BT);
    const int outs = BT * (p.R + 2 * p.N);
    const size_t lds = (size_t)(outs < 256 ? 256 : outs) * sizeof(float);
    if (lds > 48 * 1024) return MPA_ERR_BAD_SHAPE;
    const bool v4 = p.R % 4 == 0 && aligned_to(p.dt_w, 4 * sizeof(IO));
#define MPA_SSM(N16_, V_) hipLaunchKernelGGL((decode_ssm_kernel<IO, BT, N16_, V_, MANY>), grid, dim3(256), lds, st, p)
    if constexpr (!MANY) {
        if (p.N == 16) { if (v4) MPA_SSM(true, 4); else MPA_SSM(true, 1); return check_launch(); }
    }
    if (v4) MPA_SSM(false, 4); else MPA_SSM(false, 1);
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
    return 3 * act + round256((size_t)decode_splits(s) * s->batch * ((s->dt_rank + 2 * s->dstate + 3) / 4 * 4) * sizeof(float)) + decode_scaled_ws(s);
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
    p.P4 = (p.R + 2 * p.N + 3) / 4 * 4;
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
