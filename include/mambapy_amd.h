/* C ABI of libmambapy_amd.so: hand-written gfx950 (MI355X) kernels for the selective-scan
 * hot path of alxndrTL/mamba.py.
 *
 * The reference has no FFI for this path: its operator boundary is a set of Python
 * symbols (cited per entry point below).  Each entry point here is what a ctypes binding
 * placed behind that symbol calls.  Conventions:
 *   - every pointer is a DEVICE pointer unless stated otherwise; the library allocates
 *     and frees nothing, outputs and workspaces are caller-allocated;
 *   - `stream` is a hipStream_t passed as void* (NULL = the null stream); all work is
 *     enqueued on it and nothing synchronises the device;
 *   - sizes are in elements, strides are ELEMENT strides of the tensor they describe;
 *   - io_dtype selects the storage type of x, delta, B, C, z, y, dy and of their
 *     gradients (delta and its gradient may be float32 next to bfloat16 tensors, see
 *     MPA_DELTA_F32); A, D, delta_bias, the recurrent state and every accumulation are float32;
 *   - the return value is MPA_OK or one of the MPA_ERR_* codes; nothing is thrown.
 * All entry points are reentrant: nothing is read from the environment, every choice the
 * library makes is a function of the arguments (the workspace queries and the calls they size
 * therefore always agree).  They keep no global state, with two exceptions: a per-device flag
 * that remembers that a kernel's dynamic-LDS limit has been raised, and mpa_sscan_fwd_noalloc,
 * which owns a static device array per GPU and the address of it (see there).
 */
#ifndef MAMBAPY_AMD_H
#define MAMBAPY_AMD_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define MPA_VERSION 20100 /* major*10000 + minor*100 + patch: 2.1.0 */

enum mpa_status {
    MPA_OK = 0,
    MPA_ERR_NULL_POINTER = 1,  /* a required pointer is NULL */
    MPA_ERR_BAD_SHAPE = 2,     /* non-positive size, d_state above the supported maximum, ... */
    MPA_ERR_BAD_DTYPE = 3,     /* io_dtype is not one of mpa_dtype */
    MPA_ERR_BAD_STRIDE = 4,    /* a stride the kernels cannot honour (see each entry point) */
    MPA_ERR_MISALIGNED = 5,    /* a pointer is not aligned to its element size */
    MPA_ERR_WORKSPACE = 6,     /* workspace_bytes is smaller than the *_workspace_bytes query */
    MPA_ERR_LAUNCH = 7         /* hipGetLastError() reported a launch failure */
};

enum mpa_dtype { MPA_F32 = 0, MPA_BF16 = 1 };

/* Number of time steps between two saved states (see mpa_sscan_fwd: h_ckpt). */
#define MPA_CKPT_STEPS 16
/* Largest supported d_state (N). */
#define MPA_MAX_DSTATE 256

/* Shape and layout of one selective-scan call.  Logical shapes (mambapy/mamba.py:275-282):
 *   x, delta, z, y, dy, dx, ddelta : (batch, seqlen, dim)      dim = ED = d_inner
 *   A : (dim, dstate) contiguous float32;  D, delta_bias : (dim) contiguous float32
 *   B, C, dB, dC : (batch, seqlen, dstate), innermost stride 1
 * u_* strides apply to x;  z_* to z;  d_* to delta;  y_* to y, dy, y_pregate;  g_* to dx, ddelta, dz;
 * bc_* to B and C;  dbc_* to dB and dC.
 * The reference calls this path both with fresh channel-contiguous tensors
 * (tests/compare_seq_pscan.py:24-29: strides (L*ED, ED, 1)) and, from MambaBlock.forward,
 * with time-contiguous views (mambapy/mamba.py:217-221, 247, 264: strides (ED*L, 1, L)) and
 * with B, C that are slices of one projection (mamba.py:245: row stride dt_rank+2N).
 * Both layouts are honoured without a copy. */
typedef struct mpa_sscan_shape {
    int64_t batch, seqlen, dim, dstate;
    int32_t io_dtype; /* enum mpa_dtype */
    int32_t flags;    /* bit set of MPA_SSCAN_* */
    int64_t u_sb, u_sl, u_sd;
    int64_t z_sb, z_sl, z_sd;
    int64_t d_sb, d_sl, d_sd;
    int64_t y_sb, y_sl, y_sd;
    int64_t g_sb, g_sl, g_sd;
    int64_t bc_sb, bc_sl;
    int64_t dbc_sb, dbc_sl;
    /* Launch plan.  0 = chosen by the library from the shape (the normal case); a caller that
     * tunes or tests may pin the decomposition.  The same values must be given to a call and
     * to the workspace query that sizes it. */
    int32_t plan_states_per_lane; /* states of d_state kept by one lane: a power of two */
    int32_t plan_segments;        /* pieces the sequence is cut into (1 = never cut) */
    int32_t plan_flags;           /* bit set of MPA_PLAN_* */
    int32_t delta_dtype;          /* 0: delta and ddelta have io_dtype; MPA_DELTA_F32: see below */
} mpa_sscan_shape;

/* mpa_sscan_shape.delta_dtype: delta (read) and ddelta (written) are float32 whatever io_dtype is
 * (d_* and g_* remain element strides).  This is the call the reference makes under
 * torch.autocast: softplus leaves delta in float32 while x, B, C are bfloat16
 * (mambapy/mamba.py:264-265 with :284-287).  Fast kernels only: mpa_sscan_bwd returns
 * MPA_ERR_BAD_DTYPE where it would need its general kernel. */
#define MPA_DELTA_F32 1

/* delta = softplus(delta + delta_bias) is applied inside the kernel (mamba.py:264-265);
 * without the flag `delta` is used as given and delta_bias must be NULL. */
#define MPA_SSCAN_DELTA_SOFTPLUS 1
/* The recurrence runs from the last step to the first: h[t] = a[t]*h[t+1] + ..., h0 is the
 * state before step seqlen-1 and h_last the state after step 0.  Equal to flipping x, delta,
 * z, B, C along time, scanning, and flipping y back, which is how the reference's
 * bidirectional block obtains its backward direction (mambapy/vim.py:228-261: xz.flip([1])
 * in, y_b.flip([1]) out) at the price of those copies. */
#define MPA_SSCAN_REVERSE 2

/* mpa_sscan_bwd: use the general backward kernel even where the fast one applies. */
#define MPA_PLAN_BWD_GENERAL 1
/* Test hook: the bounded waits inside the kernels behave as if they had run out (see
 * mpa_sscan_bwd); every kernel still runs to its end. */
#define MPA_PLAN_EXPIRE_WAITS 2
/* Channels of a batch row that one workgroup of the forward owns: 64 always, 48, 32 or 16 wherever the kernels have
 * that form (none of the bits: the library picks, see mpa_sscan_fwd). */
#define MPA_PLAN_GROUP_64 4
#define MPA_PLAN_GROUP_48 8
#define MPA_PLAN_GROUP_32 16
#define MPA_PLAN_GROUP_16 32

int mpa_version(void);
/* Host string naming the GPU architecture the kernels were compiled for ("gfx950"). */
const char* mpa_arch(void);
/* Host string: hash of the kernel sources this library was built from (16 hex digits, "unknown"
 * when the build did not say).  Measurements that are kept next to the sources (hardware-counter
 * summaries) quote it, so that a reader can tell whether they describe the kernels that run. */
const char* mpa_source_hash(void);
/* Host string describing a status code. */
const char* mpa_status_string(int status);

/* ---- fused selective scan, forward ------------------------------------------------------
 * Replaces MambaBlock.selective_scan(x, delta, A, B, C, D) (mambapy/mamba.py:274-295) and
 * its sequential twin selective_scan_seq (:297-327): discretisation exp(delta*A) /
 * delta*B*x, the scan that mambapy/pscan.py:151-186 performs on materialised
 * (B,L,ED,N) tensors, and the readout y = C.h + D*x, in one pass that never writes a
 * (B,L,ED,N) tensor.  Any seqlen >= 1 (no power-of-two padding, cf. pscan.py:165-174).
 *   z        optional: y is multiplied by silu(z) (mamba.py:229-231); NULL = no gate.
 *   h0       optional (batch, dim, dstate) float32 initial state; NULL = zeros (mamba.py:314).
 *   h_ckpt   optional float32 buffer of mpa_sscan_ckpt_elems() elements: the state after
 *            every MPA_CKPT_STEPS-th step, consumed by mpa_sscan_bwd; NULL when no
 *            gradient is needed.
 *   h_last   optional (batch, dim, dstate) float32: state after the last step, in the
 *            layout of the decode cache `h` (mamba.py:335, 341).
 *   y_pregate  optional, only with z: the output before the gate (C.h + D*x), io_dtype, strides
 *            of y.  mpa_sscan_bwd needs it on its fast path; NULL when no gradient is needed.
 *   workspace  scratch of mpa_sscan_fwd_workspace_bytes() bytes.
 * d_state above 64 runs in passes over blocks of 64 states, each adding its readout to y (in
 * y_pregate when that is given) in io_dtype.
 * When batch * dim/64 workgroups would cover a fraction of the chip, the sequence is cut into
 * segments that run side by side (end states of all segments from zero, a carry pass, then the
 * real pass from the true initial states); checkpoints, h_last and y are the same as without the
 * cut up to float32 rounding.
 * A workgroup owns 64, 48, 32 or 16 channels of a batch row (48: two states per lane, not cut): the library takes
 * the width and the number of segments that an estimate of the time, from measured tile times, puts first.
 */
int mpa_sscan_fwd(const mpa_sscan_shape* s, const void* x, const void* delta, const float* A,
                  const void* B, const void* C, const float* D, const void* z,
                  const float* delta_bias, const float* h0, void* y, void* y_pregate,
                  float* h_ckpt, float* h_last, void* workspace, size_t workspace_bytes,
                  void* stream);

/* Number of float32 elements of the h_ckpt buffer for this shape. */
int64_t mpa_sscan_ckpt_elems(const mpa_sscan_shape* s);

/* Bytes of the scratch `workspace` of mpa_sscan_fwd (256-byte aligned; holds B and C
 * repacked as float32 in the order the scan waves read them, or the per-segment states of a
 * cut sequence; contents are dead after the call).  with_ckpt = 1 for a call that passes
 * h_ckpt, 0 for one that does not (the two are cut differently). */
size_t mpa_sscan_fwd_workspace_bytes(const mpa_sscan_shape* s, int with_ckpt);

/* ---- fused selective scan, forward, with dt_proj inside ------------------------------------------
 * mpa_sscan_fwd without gradients for a layer whose delta = rows . dt_weight^T (mambapy/mamba.py:246-247): `rows`
 * (batch, seqlen, dt_rank), strides d_sb, d_sl and 1, takes delta's place, dt_weight is (dim, dt_rank) contiguous, 16-byte
 * aligned; delta is rounded to bfloat16 as dt_proj's output is, and not written.  bfloat16, dt_rank = MPA_PROJ_RANK (a
 * narrower one padded with zeros), dstate <= 16, x with unit channel stride, with z, not reversed, states per lane
 * not pinned.  Workspace as mpa_sscan_fwd.
 */
#define MPA_PROJ_RANK 64
int mpa_sscan_fwd_proj(const mpa_sscan_shape* s, const void* x, const void* rows, const void* dt_weight, int64_t dt_rank,
                       const float* A, const void* B, const void* C, const float* D, const void* z,
                       const float* delta_bias, const float* h0, void* y, float* h_last, void* workspace,
                       size_t workspace_bytes, void* stream);

/* ---- fused selective scan, forward, for callers that cannot allocate ------------------------
 * No counterpart in the reference.  It is for callers that cannot provide a workspace because they
 * cannot call hipMalloc: code under HIP graph capture, tight serving loops, harnesses that forbid
 * allocation.  Same arguments and results as mpa_sscan_fwd (bit for bit) without `workspace`: the
 * scratch is a static device array of MPA_NOALLOC_SCRATCH_BYTES that the library owns, one copy on
 * every GPU it runs on, held until the process ends.  The call allocates and frees nothing.
 * A shape whose mpa_sscan_fwd_workspace_bytes() exceeds MPA_NOALLOC_SCRATCH_BYTES is refused with
 * MPA_ERR_WORKSPACE before anything is launched (sequences cut into segments need
 * 2 * batch * segments * dim * min(dstate, 64) floats and a little more, which fits for any shape unless the
 * caller pins the segments; one that pins 16 or 32 states per lane needs the packed B/C of the whole
 * sequence).  All calls on one GPU share that GPU's array: calls that overlap
 * on one GPU (different streams or threads) race; calls on one stream are ordered.
 * The first call on a device looks up the array's address and raises the kernels' dynamic-LDS limit
 * (host calls that do not belong into a stream capture): make one call per device and kernel variant
 * (same dtype, gate and states per lane) before capturing.
 */
#define MPA_NOALLOC_SCRATCH_BYTES (16u << 20)
int mpa_sscan_fwd_noalloc(const mpa_sscan_shape* s, const void* x, const void* delta, const float* A,
                          const void* B, const void* C, const float* D, const void* z,
                          const float* delta_bias, const float* h0, void* y, void* y_pregate,
                          float* h_ckpt, float* h_last, void* stream);

/* ---- fused selective scan, backward -----------------------------------------------------
 * Replaces what autograd records for mamba.py:284-293 plus PScan.backward
 * (mambapy/pscan.py:188-224): given dy it writes dx, ddelta (io_dtype), dB, dC (io_dtype),
 * dA (dim, dstate) and dD (dim) (float32, overwritten, not accumulated).
 * h_ckpt is the buffer mpa_sscan_fwd filled for the same inputs.  The gate z, delta_bias /
 * MPA_SSCAN_DELTA_SOFTPLUS and h0 must be the ones given to the forward call; dz (io_dtype,
 * u-strides of g_*) is required when z is given, ddelta is then the gradient w.r.t. the
 * raw (pre-softplus) delta, and ddelta_bias (dim) float32 is written when delta_bias is
 * given.  y_pregate (strides of dy) is what the forward call wrote for the same inputs; with z
 * and y_pregate == NULL the pre-gate output is recomputed by a slower, more general kernel.
 * `workspace` needs mpa_sscan_bwd_workspace_bytes() bytes, 256-byte aligned.
 * d_state up to MPA_MAX_DSTATE; above 16 the call runs in passes over blocks of 16 states (the
 * states are independent given x, delta, B, C), dx and ddelta being summed over the passes in
 * io_dtype.  Short batches of long sequences are cut into segments as in the forward call (the
 * carry runs from the end).
 * One kernel waits, with a bound, for a counter in shared memory; the wait cannot run out
 * unless the hardware scheduler misbehaves, and if it ever does the call does not return clean
 * numbers: dA of every channel whose sums may have been damaged is NaN.
 */
int mpa_sscan_bwd(const mpa_sscan_shape* s, const void* x, const void* delta, const float* A,
                  const void* B, const void* C, const float* D, const void* z,
                  const float* delta_bias, const float* h0, const void* dy,
                  const void* y_pregate, const float* h_ckpt, void* dx, void* ddelta, float* dA, void* dB, void* dC,
                  float* dD, void* dz, float* ddelta_bias, void* workspace,
                  size_t workspace_bytes, void* stream);

size_t mpa_sscan_bwd_workspace_bytes(const mpa_sscan_shape* s);

/* ---- causal depthwise convolution along time (+ bias, + SiLU) ------------------------------
 * Replaces, in MambaBlock.forward (mambapy/mamba.py:217-221),
 *     x.transpose(1,2) -> Conv1d(ED, ED, kernel, groups=ED, padding=kernel-1)(.)[:, :, :L]
 *       -> transpose(1,2) -> silu
 * on the (batch, seqlen, dim) tensor directly (any element strides: the caller passes the x half
 * of the in_proj output, mamba.py:213-214, without a copy), and its gradient.  weight is the
 * Conv1d weight (dim, 1, kernel) viewed as (dim, kernel) float32, bias (dim) float32 or NULL.
 * window_in  optional (batch, dim, kernel-1), io_dtype: the inputs before step 0 (the decode
 *            cache of mamba.py:344-346, 379), NULL = zeros (the reference's left padding).
 * window_out optional (batch, dim, kernel-1): the last kernel-1 inputs, i.e. the cache to
 *            continue from with MambaBlock.step.
 * y has the y_* strides, dy too; dx the g_* strides; dweight (dim, kernel), dbias (dim) float32,
 * overwritten.  No gradient flows into window_in.  window_out may equal window_in (the rolling
 * cache of a decode loop, updated in place: every (batch, channel) row is read and written by
 * one thread).
 */
#define MPA_CONV_SILU 1
typedef struct mpa_conv_shape {
    int64_t batch, seqlen, dim;
    int32_t kernel;   /* d_conv, 2..4 */
    int32_t io_dtype; /* enum mpa_dtype */
    int32_t flags;    /* bit set of MPA_CONV_* */
    int32_t reserved;
    int64_t x_sb, x_sl, x_sd;
    int64_t y_sb, y_sl, y_sd;
    int64_t g_sb, g_sl, g_sd;
} mpa_conv_shape;

int mpa_conv1d_fwd(const mpa_conv_shape* s, const void* x, const float* weight, const float* bias,
                   const void* window_in, void* y, void* window_out, void* stream);
int mpa_conv1d_bwd(const mpa_conv_shape* s, const void* x, const float* weight, const float* bias,
                   const void* window_in, const void* dy, void* dx, float* dweight, float* dbias,
                   void* workspace, size_t workspace_bytes, void* stream);
size_t mpa_conv1d_bwd_workspace_bytes(const mpa_conv_shape* s);

/* mpa_conv1d_fwd, and x_proj (mambapy/mamba.py:242) of its output in the same launch: proj (rows x dim, rows of dim elements)
 * times y, as batch * seqlen rows of `rows` elements, out_pitch apart, followed by out_cols - rows zeros.  Bfloat16, four
 * taps, MPA_CONV_SILU, x and y with unit stride along dim, dim a multiple of 32, strides of 8, `rows` a multiple of 4 up to
 * MPA_CONV_PROJ_COLS, a batch row under 1 GiB: mpa_conv1d_proj_suits() says so (1) or not (0, and the call returns
 * MPA_ERR_BAD_SHAPE).  x, y and proj 16-byte, out 8-byte aligned, out_pitch a multiple of 4. */
#define MPA_CONV_PROJ_COLS 96
int mpa_conv1d_proj_suits(const mpa_conv_shape* s, int64_t rows);
int mpa_conv1d_proj_fwd(const mpa_conv_shape* s, const void* x, const float* weight, const float* bias, const void* window_in, void* y,
                        void* window_out, const void* proj, int64_t rows, void* out, int64_t out_cols, int64_t out_pitch, void* stream);

/* ---- RMSNorm --------------------------------------------------------------------------------
 * Replaces RMSNorm.forward (mambapy/mamba.py:427-433): y = x * rsqrt(mean(x^2, -1) + eps) * weight
 * on `rows` contiguous rows of `d` elements (io_dtype; d a multiple of 4 (float32) / 8 (bfloat16),
 * d <= 2048 / 4096), weight (d) float32 or NULL (the muP variant has none), and its gradient:
 * dx (io_dtype) and dweight (d) float32, overwritten.  rstd (rows) float32 is an optional output.
 * Pointers to x, y, dy, dx must be 16-byte aligned.
 *
 * The residual add of the layer stack (mambapy/mamba.py:106-112: mixer(norm(x)) + x, read by the
 * next layer's norm) can be folded in: with `residual` (rows x d, io_dtype) the forward writes
 * sum_out = x + residual (rounded to io_dtype, as the separate add would be) and normalises that
 * row; the backward then takes the sum as its `x` and `dsum`, the gradient that reaches the sum
 * from its other users, and returns dx = (gradient through the norm) + dsum, which is the gradient
 * of both x and residual.  residual, sum_out and dsum may be NULL (plain RMSNorm).
 * io_dtype | MPA_NORM_WEIGHT_BF16: weight and dweight are bfloat16.
 */
#define MPA_NORM_WEIGHT_BF16 256
int mpa_rmsnorm_fwd(const void* x, const void* residual, const void* weight, void* y, void* sum_out,
                    float* rstd, int64_t rows, int64_t d, float eps, int32_t io_dtype, void* stream);
int mpa_rmsnorm_bwd(const void* x, const void* weight, const void* dy, const void* dsum, void* dx,
                    void* dweight, int64_t rows, int64_t d, float eps, int32_t io_dtype,
                    void* workspace, size_t workspace_bytes, void* stream);
size_t mpa_rmsnorm_bwd_workspace_bytes(int64_t rows, int64_t d);

/* ---- generic first-order scan -----------------------------------------------------------
 * Replaces pscan = PScan.apply (mambapy/pscan.py:226; forward :151-186, backward :188-224)
 * for callers that hold materialised A, X of logical shape (batch, seqlen, dim, dstate):
 * H[t] = A[t]*H[t-1] + X[t], H[-1] = 0.  Strides are (sb, sl, sd, sn) element strides, one
 * set per tensor; any seqlen.  H is a new tensor: inputs are never modified
 * (pscan.py:167-174 clones).  Backward: gradX[t] = gradH[t] + A[t+1]*gradX[t+1],
 * gradA[t] = H[t-1]*gradX[t], gradA[0] = 0 (pscan.py:216-222).
 * The reference's scan has O(log L) depth at any batch size (pscan.py:36-92); here one lane owns
 * one (dim, dstate) recurrence, and when batch*dim*dstate offers too few lanes to keep the memory
 * system busy the sequence is cut into pieces that run side by side (aggregate pass, carry pass,
 * main pass).  `workspace` (mpa_pscan_workspace_bytes() bytes, 256-byte aligned) holds the
 * per-piece aggregates; contents are dead after the call.
 */
typedef struct mpa_pscan_shape {
    int64_t batch, seqlen, dim, dstate;
    int32_t io_dtype;
    int32_t reverse;          /* 1: scan from the last step to the first (pscan.py:94-149) */
    int64_t a_st[4];          /* A     (sb, sl, sd, sn) */
    int64_t x_st[4];          /* X or gradH */
    int64_t h_st[4];          /* H (output of fwd, input of bwd) */
    int64_t ga_st[4];         /* gradA */
    int64_t gx_st[4];         /* gradX */
    int32_t plan_chunks;      /* pieces the sequence is cut into; 0 = chosen from the shape, 1 = never cut */
    int32_t reserved;         /* 0 */
} mpa_pscan_shape;

size_t mpa_pscan_workspace_bytes(const mpa_pscan_shape* s);
int mpa_pscan_fwd(const mpa_pscan_shape* s, const void* A, const void* X, void* H, void* workspace,
                  size_t workspace_bytes, void* stream);
int mpa_pscan_bwd(const mpa_pscan_shape* s, const void* A, const void* H, const void* gradH,
                  void* gradA, void* gradX, void* workspace, size_t workspace_bytes, void* stream);

/* ---- decode step --------------------------------------------------------------------------
 * Replaces the state update and readout of MambaBlock.ssm_step (mambapy/mamba.py:400-412)
 * for one token: h' = exp(delta*A)*h + delta*B*x ; y = C.h' + D*x, optionally
 * delta = softplus(delta + delta_bias) (mamba.py:398) and y *= silu(z) (mamba.py:373-375).
 *   x, delta, y : (batch, dim) io_dtype contiguous;  z : (batch, dim) with row stride z_stride (it
 *   is a half of the in_proj output, mamba.py:356-357);  B, C : (batch, dstate) io_dtype,
 *   row stride bc_stride;  h_in, h_out : (batch, dim, dstate) float32 contiguous.
 * h_in == NULL means zeros (mamba.py:405-406).  h_out may equal h_in (in-place update);
 * with distinct buffers h_in is left untouched, which is the reference's behaviour
 * (ssm_step returns a new tensor).
 */
int mpa_ssm_step(const void* x, const void* delta, const float* A, const void* B, const void* C,
                 const float* D, const void* z, const float* delta_bias, const float* h_in,
                 float* h_out, void* y, int64_t batch, int64_t dim, int64_t dstate,
                 int64_t bc_stride, int64_t z_stride, int32_t io_dtype, int32_t delta_softplus,
                 void* stream);

/* ---- decode step of a whole layer -----------------------------------------------------------
 * Replaces, for one token of each of up to MPA_DECODE_MAX_BATCH sequences, the chain that
 * ResidualBlock.step / MambaBlock.step run (mambapy/mamba.py:114-125, 351-414): RMSNorm, in_proj, the
 * convolution over the rolling window with silu, x_proj, dt_proj, the state update with softplus, the
 * gate, out_proj, residual add; three or four launches.
 *   x, y : (batch, d_model) io_dtype contiguous.  norm = 1: y = x + block(rmsnorm(x)), the residual block;
 *     norm = 0: y = block(x), the mixer alone.  y may not alias x.
 *   x_scaled, x_ssq  optional (norm = 1): x times norm_weight in io_dtype, in the order in which the matrix
 *     cores take it (mpa_decode_scaled_bytes() bytes), and ceil(d_model / 16) rows of `batch` partial
 *     sums of squares of x, as the call of the layer before wrote them; NULL: formed here.
 *   next_norm_weight, y_scaled, y_ssq  optional: the same two for the layer after, whose norm weight is given.
 *   h_in (NULL: zeros), h_out : (batch, dim, dstate) float32;  window_in, window_out : (batch, dim,
 *     d_conv-1) io_dtype.  The outputs may be the inputs (in-place update).
 * Weights: in_weight (2*dim, d_model), x_weight (dt_rank + 2*dstate, dim), dt_weight (dim, dt_rank),
 * out_weight (d_model, dim), biases of in_proj / out_proj in io_dtype or NULL; norm_weight (d_model),
 * conv_weight (dim, d_conv), conv_bias, dt_bias (dim), A (dim, dstate), D (dim) float32 (norm_weight and the
 * biases may be NULL).  d_model and dim are multiples of 4 (float32) / 8 (bfloat16), dstate of 4.
 */
#define MPA_DECODE_MAX_BATCH 128
typedef struct mpa_decode_layer {
    int64_t batch, d_model, dim, dstate, dt_rank;
    int32_t d_conv, io_dtype;
    int32_t norm;
    float eps;
    const float* norm_weight;
    const void *in_weight, *in_bias;
    const float *conv_weight, *conv_bias;
    const void *x_weight, *dt_weight;
    const float *dt_bias, *A, *D;
    const void *out_weight, *out_bias;
} mpa_decode_layer;

size_t mpa_decode_layer_workspace_bytes(const mpa_decode_layer* s);
size_t mpa_decode_scaled_bytes(const mpa_decode_layer* s);
int mpa_decode_layer_step(const mpa_decode_layer* s, const void* x, const void* x_scaled, const float* x_ssq, void* y,
                          const float* next_norm_weight, void* y_scaled, float* y_ssq, const float* h_in, float* h_out,
                          const void* window_in, void* window_out, void* workspace, size_t workspace_bytes,
                          void* stream);

/* ---- projections of a short sequence -----------------------------------------------------------
 * y (T x M) = x (T x K) . weight (M x K)^T + bias, io_dtype with float32 sums, around it the norm and the
 * residual add of a pre-norm stack (mambapy/mamba.py:114-125):
 *   norm_weight, x_ssq  optional: `ssq_parts` rows of T partial sums of squares of the rows of x, which are
 *     multiplied by 1 / sqrt(sum / K + eps) and by norm_weight (K, float32) and rounded before the product.  (For callers with rows
 *     that are not yet scaled; this package's own stacks use mpa_linear_run_scaled, which is faster.)
 *   weight_kxm  the weight is (K x M), M a multiple of 4 (float32) / 8: y = x . weight, the product of a projection's backward;
 *     without norm_weight and y_ssq.
 *   residual  optional: (T x M), added to the rounded product or, with `accumulate`, before it is rounded; may be y.
 *   y_ssq  optional: ceil(M / 32) rows of T partial sums of squares of y (NaN with an infinity among them).
 *   io_dtype | MPA_LINEAR_X_F32 (with x_ssq), _Y_F32, _RESIDUAL_F32: x, y or residual are float32 in a bfloat16
 *     call (nothing is rounded on its way into a float32 y).
 * Rows of x are x_pitch apart, those of y and residual y_pitch.  K and x_pitch are multiples of 4 (float32) / 8
 * (bfloat16), M and y_pitch of 4; x, weight and norm_weight 16-byte aligned, the rest four elements.
 */
#define MPA_LINEAR_X_F32 256
#define MPA_LINEAR_Y_F32 512
#define MPA_LINEAR_RESIDUAL_F32 1024
typedef struct mpa_linear {
    int64_t T, M, K, x_pitch, y_pitch;
    const void *x, *weight, *bias;
    void* y;
    const float *norm_weight, *x_ssq;
    int64_t ssq_parts;
    float eps;
    int32_t io_dtype, weight_kxm, accumulate;
    const void* residual;
    float* y_ssq;
} mpa_linear;
int mpa_linear_run(const mpa_linear* s, void* stream);
/* The same between the layers of a stack, where the norm's weight is applied to the rows as they are written and their
 * 1 / rms to the product of them:
 *   y_weight, y_scaled  optional: y * y_weight (M, float32), rounded to io_dtype, in rows of M.
 *   x_ssq without norm_weight: x holds such rows, and the product is multiplied by 1 / sqrt(sum / K + eps) of its row
 *     before bias and residual; where the sum is an infinity (squares beyond float32) it is zero, whatever the product is.  Not
 *     with weight_kxm or a float32 x in a bfloat16 call.
 * y_weight is 16-byte aligned, y_scaled four elements.
 */
int mpa_linear_run_scaled(const mpa_linear* s, const float* y_weight, void* y_scaled, void* stream);

/* ---- weight gradients --------------------------------------------------------------------------
 * out = P^T . Q for up to MPA_WGRAD_MAX_JOBS pairs of matrices of T rows: what autograd forms for the
 * projections of a layer (mambapy/mamba.py:210, 244, 247, 232), P the gradient of a projection's output
 * (rows columns, row stride ldp), Q its input (cols columns, row stride ldq), io_dtype; sums in float32,
 * added in a fixed order.  out is (rows - gap, keep_cols) contiguous, io_dtype: columns from keep_cols on
 * and the `gap` rows from gap_at on (padding of P and Q) are left out.  rows, cols and the strides are
 * multiples of 4 (float32) / 8 (bfloat16), P and Q 16-byte aligned.
 */
#define MPA_WGRAD_MAX_JOBS 4
typedef struct mpa_wgrad_job {
    const void *p, *q;
    int64_t ldp, ldq;
    int64_t rows, cols, keep_cols, gap_at, gap;
    void* out;
} mpa_wgrad_job;
size_t mpa_wgrad_workspace_bytes(const mpa_wgrad_job* jobs, int32_t n, int64_t T, int32_t io_dtype);
int mpa_wgrad(const mpa_wgrad_job* jobs, int32_t n, int64_t T, int32_t io_dtype, void* workspace,
              size_t workspace_bytes, void* stream);

/* ---- products of many rows -----------------------------------------------------------------------
 * y (T x M) = x (T x K) . W^T in bfloat16, sums in float32, rounded once: the projections of a layer over long sequences and their
 * input gradients (mambapy/mamba.py:210, 232).  weight is (M, K), or (K, M) with weight_kxm; pitches are of rows, in elements.  M, K and
 * the pitches are multiples of 8, pointers 16-byte aligned; bounds: T, M and K at most 2^24, 256 rows of x, of y and of a weight (M, K)
 * below 2^31 bytes, and all of a weight (K, M).
 * mpa_gemm_faster: 1 where it is expected to be faster than the GEMM library, 0 where not and for calls that mpa_gemm_run refuses.
 */
typedef struct mpa_gemm {
    const void *x, *weight;
    void* y;
    int64_t T, M, K, x_pitch, weight_pitch, y_pitch;
    int32_t weight_kxm;
} mpa_gemm;
int mpa_gemm_faster(const mpa_gemm* s);
int mpa_gemm_run(const mpa_gemm* s, void* stream);

/* ---- conversions of small matrices ----------------------------------------------------------------
 * Up to MPA_CAST_MAX_JOBS copies of rows x cols elements between float32 and bfloat16 in one launch, each
 * optionally through -exp(v) (A from A_log, mambapy/mamba.py:239) or v * factor (float32, contiguous);
 * MPA_CAST_ZERO writes zeros (src is not read).
 */
#define MPA_CAST_MAX_JOBS 12
enum mpa_cast_op { MPA_CAST_COPY = 0, MPA_CAST_NEG_EXP = 1, MPA_CAST_TIMES = 2, MPA_CAST_ZERO = 3 };
typedef struct mpa_cast_job {
    const void* src;
    void* dst;
    const float* factor;
    int64_t rows, cols, src_pitch, dst_pitch;
    int32_t src_dtype, dst_dtype, op, reserved;
} mpa_cast_job;
int mpa_cast(const mpa_cast_job* jobs, int32_t n, void* stream);

/* ---- wide float32 products ---------------------------------------------------------------------------
 * y (T x M) = x (T x K) . w (M x K)^T [+ bias] in float32 on the 16-bit matrix cores: each operand is cut into two
 * float16 parts per value with one power of two per row, mpa_split_run, and up to MPA_SPLIT_MAX_PRODUCTS products of cut operands
 * run in one launch, mpa_split_product.  A value keeps 2^-23 of itself, 2^-20 (from K = 2048 on K / 64 * 2^-24) where it is below 2^-28 of
 * its row's largest; a row with values more than 2^31 (K / 1024 * 2^31) apart, zeros aside, or with an infinity is multiplied
 * in float32 (split.hip).
 *
 * An operand has `rows` rows of length k: element (row, i) is src[row * pitch + i], or with by_cols
 * src[i * pitch + row].  The fast dimension's size and the pitch are multiples of 4, src is 16-byte aligned.  `split`
 * (256-byte aligned, mpa_split_bytes bytes: 4 bytes a value of rows rounded up to 32, k to 32, and a little) receives the parts.  A
 * product takes w with M rows, a multiple of 4, and x with T rows, and reads their parts only.  y and bias are 16-byte
 * aligned, y_pitch a multiple of 4.  The workspace (16-byte aligned) may be NULL where its query says 0.
 */
#define MPA_SPLIT_MAX_OPERANDS 8
#define MPA_SPLIT_MAX_PRODUCTS 4
typedef struct mpa_split_operand {
    const float* src;
    int64_t rows, k, pitch;
    int32_t by_cols, reserved;
    void* split;
} mpa_split_operand;
typedef struct mpa_split_job {
    mpa_split_operand w, x;
    const float* bias;
    float* y;
    int64_t y_pitch;
} mpa_split_job;
size_t mpa_split_bytes(int64_t rows, int64_t k);
int mpa_split_run(const mpa_split_operand* operands, int32_t n, void* stream);
size_t mpa_split_product_workspace_bytes(const mpa_split_job* jobs, int32_t n);
int mpa_split_product(const mpa_split_job* jobs, int32_t n, void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* MAMBAPY_AMD_H */
