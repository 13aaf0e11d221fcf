// nsm_mlp.hip -- the surrogate network of the ensemble estimator: a fully
// connected network with GELU between layers, BF16 weights and activations,
// FP32 accumulation on gfx950's matrix cores (v_mfma_f32_16x16x32_bf16),
// FP32 master parameters trained by Adam.  Kernels and the nsm_mlp_* C ABI.
//
// Layer l (1..L) with width d_l: Z_l = H_{l-1} W_l^T + b_l (FP32), hidden
// layers H_l = bf16(gelu(Z_l)), output Y = Z_L.  H_0 = bf16(x).  Gradients of
// the mean squared error over batch and outputs run the same GEMM kernel:
// G_L = 2 (Y - T) / (B d_L); for l = L..1: D_l = bf16(G_l),
// dW_l = D_l^T H_{l-1}, db_l = sum_b G_l (FP32), and below the first layer
// G_{l-1} = (D_l W_l) * gelu'(Z_{l-1}).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/nimblesm_amd.h"

namespace nsm {
int set_last_error(int status, const char* msg);
}

namespace {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float  f32x4 __attribute__((ext_vector_type(4)));

int fail(int status, const char* fmt, ...)
{
  char    buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  return nsm::set_last_error(status, buf);
}

#define MLP_HIP(call)                                                                              \
  do {                                                                                             \
    hipError_t _e = (call);                                                                        \
    if (_e != hipSuccess) return fail(NSM_ERR_HIP, "%s: %s", #call, hipGetErrorString(_e));        \
  } while (0)

#define MLP_LAUNCHED()                                                                             \
  do {                                                                                             \
    hipError_t _e = hipGetLastError();                                                             \
    if (_e != hipSuccess) return fail(NSM_ERR_HIP, "kernel launch: %s", hipGetErrorString(_e));    \
  } while (0)

// GELU with the error function, and its derivative
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float x)
{
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// ---------------------------------------------------------------------------
// GEMM: C[m][n] = sum_k A(m, k) B(k, n), A(m, k) = a[m a_m + k a_k],
// B(k, n) = b[k b_k + n b_n] (BF16), FP32 accumulation, with an epilogue.
// The network's products are small (M <= a few thousand rows, N, K <= 512),
// so a product's time is the latency of its loads, not its multiplies: a
// 256-thread workgroup computes a 32 x 32 tile of C (four waves of one
// 16 x 16 MFMA tile each) and stages up to 256 of K at once, every load of
// that range in flight together, so a product with K <= 256 waits for one
// round trip to memory instead of one per 32 of K.
// MFMA 16x16x32 operand layout: lane l holds row (A) / column (B) l % 16 and
// k = 8 (l / 16) .. 8 (l / 16) + 7; the result holds column l % 16, rows
// 4 (l / 16) .. 4 (l / 16) + 3.
// ---------------------------------------------------------------------------
constexpr int kTile = 32, kKStep = 32, kKStage = 256, kPad = 8, kGemmThreads = 256;
// chunks of 8 values one thread loads per operand and K stage
constexpr int kChunks = kTile * kKStage / 8 / kGemmThreads;
// weight-gradient products (K = batch) longer than this are split into at
// most kMaxSplits K ranges summed by k_split_sum
constexpr int kSplitAbove = 1024, kMaxSplits = 8;

enum Epilogue {
  kStoreC     = 0,  // C = v (FP32)
  kHidden     = 1,  // z = v + bias: C = z (FP32), H = bf16(gelu(z))
  kOutput     = 2,  // C = v + bias (FP32)
  kBackHidden = 3,  // g = v * gelu'(Z): G = g (FP32), D = bf16(g)
};

// How an operand tile is staged: 16-byte loads along k (contiguous in k),
// 16-byte loads along m / n written transposed into LDS (contiguous in m /
// n), or one element at a time.
enum Staging { kAlongK = 1, kAlongMN = 2, kScalar = 0 };

struct GemmArgs {
  int          M, N, K;
  const bf16*  a;
  int64_t      a_m, a_k;
  const bf16*  b;
  int64_t      b_k, b_n;
  float*       c;  // [M][ldc]; split-K: split z writes c + z * split_stride
  int64_t      ldc;
  const float* bias;  // [N]
  bf16*        h;     // [M][ldc]
  const float* z;     // [M][ldc]: pre-activation (kBackHidden)
  int          a_stage, b_stage;
  int          k_chunk;  // K range of one split (multiple of kKStep)
  int64_t      split_stride;
};

// One operand's share of a K stage: the 32 rows r0.. of the M or N side and
// k in [k0, k0 + 32 nk32) are cut into chunks of 8 values; chunk c of
// thread t is t + 256 c.  AlongK / scalar: chunk = (row, 8 k); AlongMN:
// chunk = (k, 8 rows).  Values past R or K are zero.
struct StageRegs {
  bf16x8 v[kChunks];
};

__device__ __forceinline__ void chunk_coords(int mode, int q, int& r, int& k)
{
  if (mode == kAlongMN) {
    k = q >> 2;
    r = (q & 3) * 8;
  } else {
    r = q & (kTile - 1);
    k = (q >> 5) * 8;
  }
}

__device__ __forceinline__ void stage_load(const bf16* p, int64_t s_r, int64_t s_k, int mode, int r0, int R, int k0,
                                           int K, int nchunks, StageRegs& g)
{
#pragma unroll
  for (int c = 0; c < kChunks; c++) {
    const int q = (int)threadIdx.x + c * kGemmThreads;
    if (q >= nchunks) continue;
    int rl, kl;
    chunk_coords(mode, q, rl, kl);
    const int r = r0 + rl, k = k0 + kl;
    if (mode == kAlongK) {
      if (r < R && k + 8 <= K) {
        g.v[c] = *reinterpret_cast<const bf16x8*>(p + (int64_t)r * s_r + k);
        continue;
      }
#pragma unroll
      for (int j = 0; j < 8; j++) g.v[c][j] = (r < R && k + j < K) ? p[(int64_t)r * s_r + (k + j)] : (bf16)0.0f;
    } else if (mode == kAlongMN) {
      if (k < K && r + 8 <= R) {
        g.v[c] = *reinterpret_cast<const bf16x8*>(p + (int64_t)k * s_k + r);
        continue;
      }
#pragma unroll
      for (int j = 0; j < 8; j++) g.v[c][j] = (k < K && r + j < R) ? p[(int64_t)k * s_k + (r + j)] : (bf16)0.0f;
    } else {
#pragma unroll
      for (int j = 0; j < 8; j++)
        g.v[c][j] = (r < R && k + j < K) ? p[(int64_t)r * s_r + (int64_t)(k + j) * s_k] : (bf16)0.0f;
    }
  }
}

template <int kLd>
__device__ __forceinline__ void stage_store(const StageRegs& g, int mode, int nchunks, bf16 (*S)[kLd])
{
#pragma unroll
  for (int c = 0; c < kChunks; c++) {
    const int q = (int)threadIdx.x + c * kGemmThreads;
    if (q >= nchunks) continue;
    int r, k;
    chunk_coords(mode, q, r, k);
    if (mode == kAlongMN) {
#pragma unroll
      for (int j = 0; j < 8; j++) S[r + j][k] = g.v[c][j];
    } else {
      *reinterpret_cast<bf16x8*>(&S[r][k]) = g.v[c];
    }
  }
}

// Tile (bx, by) of C (columns 32 bx.., rows 32 by..) over split bz of the
// K range, by the whole workgroup (bx, by, bz uniform).
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, int mode, int bx, int by, int bz)
{
  constexpr int kLd = kKStage + kPad;
  __shared__ __attribute__((aligned(16))) bf16 As[kTile][kLd];
  __shared__ __attribute__((aligned(16))) bf16 Bs[kTile][kLd];
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  const int m0 = by * kTile, n0 = bx * kTile;
  const int wm = wave >> 1, wn = wave & 1;
  const int kb = bz * g.k_chunk, ke = min(g.K, kb + g.k_chunk);
  f32x4     acc = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = kb; k0 < ke; k0 += kKStage) {
    const int nk32    = (min(kKStage, ke - k0) + kKStep - 1) / kKStep;  // 32-wide steps of this stage
    const int nchunks = kTile * nk32 * kKStep / 8;
    StageRegs ra, rb;
    stage_load(g.a, g.a_m, g.a_k, g.a_stage, m0, g.M, k0, ke, nchunks, ra);
    stage_load(g.b, g.b_n, g.b_k, g.b_stage, n0, g.N, k0, ke, nchunks, rb);
    if (k0 > kb) __syncthreads();  // the previous stage's LDS reads are done
    stage_store<kLd>(ra, g.a_stage, nchunks, As);
    stage_store<kLd>(rb, g.b_stage, nchunks, Bs);
    __syncthreads();
    for (int s = 0; s < nk32; s++) {
      const bf16x8 af  = *reinterpret_cast<const bf16x8*>(&As[wm * 16 + (lane & 15)][s * kKStep + 8 * (lane >> 4)]);
      const bf16x8 bfr = *reinterpret_cast<const bf16x8*>(&Bs[wn * 16 + (lane & 15)][s * kKStep + 8 * (lane >> 4)]);
      acc              = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr, acc, 0, 0, 0);
    }
  }

  float* const c = g.c + (int64_t)bz * g.split_stride;
  const int    n = n0 + wn * 16 + (lane & 15);
#pragma unroll
  for (int r = 0; r < 4; r++) {
    const int m = m0 + wm * 16 + 4 * (lane >> 4) + r;
    if (m >= g.M || n >= g.N) continue;
    const int64_t o = (int64_t)m * g.ldc + n;
    float         v = acc[r];
    if (mode == kStoreC) {
      c[o] = v;
    } else if (mode == kHidden) {
      v += g.bias[n];
      c[o]   = v;
      g.h[o] = (bf16)gelu(v);
    } else if (mode == kOutput) {
      c[o] = v + g.bias[n];
    } else {  // kBackHidden
      const float gr = v * gelu_grad(g.z[o]);
      c[o]           = gr;
      g.h[o]         = (bf16)gr;
    }
  }
}

// Row tiles run along the grid's x dimension (up to 2^31 - 1 workgroups; y
// and z are limited to 65535), column tiles along y, K ranges along z.
__global__ __launch_bounds__(kGemmThreads) void k_gemm_bf16(GemmArgs g, int mode)
{
  gemm_tile(g, mode, (int)blockIdx.y, (int)blockIdx.x, (int)blockIdx.z);
}

// db[n] = sum over the batch of G[b][n] for the four columns 4 w .. 4 w + 3
// of workgroup w: one wave per column, lane l sums rows l, l + 64, ... in
// ascending order, then a fixed shuffle tree
__device__ __forceinline__ void bias_grad_columns(const float* __restrict__ G, int64_t B, int N,
                                                  float* __restrict__ db, int w)
{
  const int n = w * 4 + (int)(threadIdx.x >> 6);
  if (n >= N) return;
  const int lane = (int)threadIdx.x & 63;
  float     s    = 0.0f;
  for (int64_t b = lane; b < B; b += 64) s += G[b * N + n];
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) s += __shfl_down(s, m, 64);
  if (lane == 0) db[n] = s;
}

// The independent parts of one layer's backward pass in one launch:
// workgroups [0, tiles[0]) compute tiles of product 0 (the weight
// gradient), the next tiles[1] tiles of product 1 (the input gradient,
// absent below the first layer), the rest the bias gradient.  Products are
// unsplit (K = batch <= kSplitAbove).
struct LayerBackward {
  GemmArgs     prod[2];
  int          mode[2];
  int          tiles[2], tiles_x[2];
  const float* G;  // [B][N] FP32 gradient of the layer's output
  int64_t      B;
  int          N;
  float*       db;
};

__global__ __launch_bounds__(kGemmThreads) void k_layer_backward(LayerBackward lb)
{
  int w = (int)blockIdx.x;
#pragma unroll
  for (int q = 0; q < 2; q++) {
    if (w < lb.tiles[q]) {  // uniform across the workgroup
      gemm_tile(lb.prod[q], lb.mode[q], w % lb.tiles_x[q], w / lb.tiles_x[q], 0);
      return;
    }
    w -= lb.tiles[q];
  }
  bias_grad_columns(lb.G, lb.B, lb.N, lb.db, w);
}

// out[i] = sum over splits s of part[s * stride + i], ascending s
__global__ __launch_bounds__(256) void k_split_sum(const float* __restrict__ part, int splits, int64_t stride,
                                                   int64_t n, float* __restrict__ out)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float s = 0.0f;
  for (int z = 0; z < splits; z++) s += part[(int64_t)z * stride + i];
  out[i] = s;
}

// FP32 -> BF16 (round to nearest even), n values
__global__ __launch_bounds__(256) void k_to_bf16(const float* __restrict__ x, bf16* __restrict__ y, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = (bf16)x[i];
}

// Gradient G = 2 (y - t) / n of the mean squared error over n outputs (also
// as BF16), and per workgroup the sum of squared errors (fixed tree).
constexpr int kMseBlocks = 64;
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ y, const float* __restrict__ t, int64_t n,
                                             float* __restrict__ grad, bf16* __restrict__ grad_bf,
                                             double* __restrict__ partial)
{
  __shared__ double red[256];
  double            s     = 0.0;
  const float       scale = 2.0f / (float)n;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    const float e = y[i] - t[i];
    s += (double)e * (double)e;
    const float gr = scale * e;
    grad[i]        = gr;
    grad_bf[i]     = (bf16)gr;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// loss of pass p = sum of its `count` partials (ascending) / n, for passes
// 0 .. gridDim.x - 1 (partial[p count + b])
__global__ __launch_bounds__(64) void k_mse_total(const double* __restrict__ partial, int count, int64_t n,
                                                  double* __restrict__ loss_out)
{
  if (threadIdx.x != 0) return;
  const double* p = partial + (int64_t)blockIdx.x * count;
  double        s = 0.0;
  for (int b = 0; b < count; b++) s += p[b];
  loss_out[blockIdx.x] = s / (double)n;
}

// bias gradient alone (batches longer than kSplitAbove)
__global__ __launch_bounds__(256) void k_bias_grad(const float* __restrict__ G, int64_t B, int N,
                                                   float* __restrict__ db)
{
  bias_grad_columns(G, B, N, db, (int)blockIdx.x);
}

// Adam on the FP32 master parameters; BF16 copies for the forward pass.
struct Adam {
  float *p, *m1, *m2;
  bf16*  p_bf;
  float  lr, b1, b2, c1, c2, eps;
};

struct AdamState {
  float p, m1, m2;
};
__device__ __forceinline__ AdamState adam_load(const Adam& o, int64_t i) { return {o.p[i], o.m1[i], o.m2[i]}; }

// parameter i in state t with gradient gi; its new BF16 value.  The fused
// multiply-adds are written out, so every kernel rounds alike.
__device__ __forceinline__ bf16 adam_update(const Adam& o, int64_t i, const AdamState& t, float gi)
{
  const float a  = __builtin_fmaf(1.0f - o.b1, gi, o.b1 * t.m1);
  const float v  = __builtin_fmaf(gi, (1.0f - o.b2) * gi, o.b2 * t.m2);
  o.m1[i]        = a;
  o.m2[i]        = v;
  const float pi = t.p - o.lr * (a / o.c1) / (sqrtf(v / o.c2) + o.eps);
  o.p[i]         = pi;
  return o.p_bf[i] = (bf16)pi;
}

__global__ __launch_bounds__(256) void k_adam(Adam o, const float* __restrict__ g, int64_t n)
{
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) adam_update(o, i, adam_load(o, i), g[i]);
}

// ---------------------------------------------------------------------------
// Small networks (at most kRowLayers layers, no width above kRowWidth): a
// training pass in two launches instead of ten, a forward pass in one.
//
// Layer by layer such a pass is a chain of launches that each wait for a
// few loads: at batch 512 the products of the 4-256-256-256-64 network are
// 0.46 GFLOP, under a microsecond of the matrix cores, and took 69 us.  But
// the rows of a batch are independent until the weight gradients: a
// workgroup takes a few rows (training: 4, 8 or 16, train_group; prediction:
// 4, 16 or 32, forward_rows) through every layer forward, the loss and the
// input gradients back (k_rows), activations in LDS, one wave per 16 columns
// of a layer's output and the next layer's weights on their way to registers
// while a layer computes.  It leaves H_l and D_l transposed, so that the
// weight-gradient products read both operands along the batch, 16 bytes per
// lane, straight into MFMA operands; k_weights forms every weight and bias
// gradient in one launch and applies Adam to each where it is formed.
// Products use the MFMA steps, K ranges and summation orders of the
// layer-by-layer kernels: gradients and outputs are the same bits (the loss
// adds its FP64 squares by rows).
//
// Weights are kept twice, in BF16 and padded to multiples of 32 with zeros:
// wf [np][kp] with k along the input (forward), wt [kp][np] with k along the
// output (input gradients), each in MFMA operand order (operand_index).
// Padded columns of a layer's output and of its gradient are 0 by selection:
// their zero weights make a NaN of an infinite value, which the next product
// would carry to every column.  Rows past the batch, up to Bp (a multiple of
// 32), are stored as 0 in H and D.
//
// Training iteration of the 4-256-256-256-64 network, layer by layer and
// here: batch 64 54 -> 19 us, 512 66 -> 23 us, 1024 100 -> 29 us, 2048 185 ->
// 37 us, 4096 243 -> 56 us, 16384 693 -> 205 us.  At 512 (128 workgroups of 4 rows): k_rows 15 us, of
// which about 4 are weight loads (one CU reads the 0.6 MB of both copies from
// L2) and 3 the stores of H, D and G, the rest the chain of seven dependent
// products; k_weights 8 us, one round of loads per 16 K steps and Adam.
// ---------------------------------------------------------------------------
constexpr int kRowWidth = 256, kRowLayers = 4, kRowThreads = 1024, kRowSteps = kRowWidth / kKStep;

// Place of element (r, k) of an operand of `steps` k steps stored in MFMA
// operand order: 16 rows x 32 k are one contiguous block of 1 KB, lane
// r % 16 + 16 (k % 32 / 8) holding 16 bytes of it.  A wave's operand load is
// then 1 KB in lane order; from rows at a stride it took four times as long
// (consecutive lanes in different cache lines), and a pass of k_rows 27 us.
__device__ __forceinline__ int64_t operand_index(int64_t r, int64_t k, int64_t steps)
{
  return ((r >> 4) * steps + (k >> 5)) * 512 + ((r & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

struct RowLayer {
  int          din, dout, kp, np;  // widths, and rounded up to 32
  int64_t      w_off, b_off;       // in the flat parameter array
  bf16 *       wf, *wt;
  const float* bias;
  bf16 *       ht, *dt;  // H of the layer's input [kp][Bp], D of its output [np][Bp], in operand order
  float*       gt;       // G of its output [Bp][np]
};

struct RowArgs {
  int64_t      B, Bp;
  const float* x;        // [B][d_0]
  const float* target;   // [B][d_L] (training)
  float*       y;        // [B][d_L] (forward only)
  double*      partial;  // squared error per workgroup (training)
  float        scale;    // 2 / (B d_L)
  RowLayer     l[kRowLayers];
};

// One wave's columns of a layer's weights: lane c + 16 q holds column c,
// k = 32 s + 8 q .. + 7 in v[s].
struct RowWeights {
  bf16x8 v[kRowSteps];
};

// Every load is executed whatever the layer's size (past its columns or its
// last k step the indices are clamped): with no branch around them the waits
// for one layer's weights leave the next layer's in flight.
__device__ __forceinline__ void load_weights(const bf16* w, int ld, int cols, int wave, int lane, RowWeights& f)
{
  const bf16x8* p = reinterpret_cast<const bf16x8*>(w + (int64_t)min(wave, cols / 16 - 1) * 16 * ld) + lane;
#pragma unroll
  for (int s = 0; s < kRowSteps; s++) f.v[s] = p[64 * min(s, ld / kKStep - 1)];
}

// Rows of a workgroup in the matrix-core tiles: tile t's accumulator lane
// c + 16 q holds column c of tile rows 4 q .. 4 q + 3, of which the first
// kPer are rows 4 kPer t + kPer q + r of the workgroup (the others repeat the
// last of them and are not used).
template <int kPer, int kRT, int kLd>
__device__ __forceinline__ void row_product(const bf16 (*act)[kLd], const RowWeights& f, int kp, int lane,
                                            f32x4 (&acc)[kRT])
{
  const int m = lane & 15, row = (m >> 2) * kPer + min(m & 3, kPer - 1);
#pragma unroll
  for (int t = 0; t < kRT; t++) {
    const bf16* p = &act[4 * kPer * t + row][8 * (lane >> 4)];
    bf16x8      v[kRowSteps];
#pragma unroll
    for (int s = 0; s < kRowSteps; s++) v[s] = *reinterpret_cast<const bf16x8*>(p + min(s * kKStep, kp - kKStep));
    acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (kp == kRowWidth) {  // uniform
#pragma unroll
      for (int s = 0; s < kRowSteps; s++)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[s], f.v[s], acc[t], 0, 0, 0);
    } else {
#pragma unroll
      for (int s = 0; s < kRowSteps - 1; s++)
        if (s * kKStep < kp) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[s], f.v[s], acc[t], 0, 0, 0);
    }
  }
}

// kL layers, 4 kPer kRT rows per workgroup
template <int kL, int kPer, int kRT, bool kTrain>
__global__ __launch_bounds__(kRowThreads) void k_rows(RowArgs a)
{
  constexpr int kRows = 4 * kPer * kRT, kLd = kRowWidth + kPad;
  typedef float  fvec __attribute__((ext_vector_type(kPer)));
  typedef __bf16 bvec __attribute__((ext_vector_type(kPer)));
  __shared__ __attribute__((aligned(16))) bf16 act[2][kRows][kLd];
  __shared__ double                            red[kRowThreads / 64];
  const int     tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int     col = wave * 16 + (lane & 15), row0 = kPer * (lane >> 4);
  const int64_t b0  = (int64_t)blockIdx.x * kRows;

  RowWeights w;
  load_weights(a.l[0].wf, a.l[0].kp, a.l[0].np, wave, lane, w);
  {
    const int din = a.l[0].din, kp = a.l[0].kp;
    for (int i = tid; i < kRows * kp; i += kRowThreads) {
      const int  r = i & (kRows - 1), k = i / kRows;
      const bool ok = b0 + r < a.B && k < din;
      const bf16 v  = ok ? (bf16)a.x[(b0 + r) * din + k] : (bf16)0.0f;
      act[0][r][k]  = v;
      if (kTrain) a.l[0].ht[operand_index(k, b0 + r, a.Bp / kKStep)] = v;
    }
  }
  float gp[kL][kRT][kPer];  // gelu'(z) of the hidden layers (training)
  float bias[kL], tgt[kRT][kPer];
#pragma unroll
  for (int l = 0; l < kL; l++) bias[l] = a.l[l].bias[min(col, a.l[l].dout - 1)];
  if (kTrain)
#pragma unroll
    for (int t = 0; t < kRT; t++)
#pragma unroll
      for (int r = 0; r < kPer; r++)
        tgt[t][r] = a.target[min(b0 + 4 * kPer * t + row0 + r, a.B - 1) * a.l[kL - 1].dout +
                             min(col, a.l[kL - 1].dout - 1)];
  __syncthreads();

#pragma unroll
  for (int l = 0; l < kL; l++) {
    const RowLayer& y  = a.l[l];
    const RowLayer& up = a.l[l + 1 < kL ? l + 1 : l];
    RowWeights next;
    if (l + 1 < kL)
      load_weights(up.wf, up.kp, up.np, wave, lane, next);
    else if (kTrain && kL > 1)
      load_weights(y.wt, y.np, y.kp, wave, lane, next);
    double sq = 0.0;
    if (wave * 16 < y.np) {
      f32x4 acc[kRT];
      row_product<kPer, kRT, kLd>(act[l & 1], w, y.kp, lane, acc);
#pragma unroll
      for (int t = 0; t < kRT; t++) {
        const int     rl = 4 * kPer * t + row0;  // first of the lane's kPer rows
        const int64_t at = operand_index(col, b0 + rl, a.Bp / kKStep);
        bvec          hv;
        fvec          gv;
#pragma unroll
        for (int r = 0; r < kPer; r++) {
          const bool  ok = b0 + rl + r < a.B;
          const float z  = col < y.dout ? acc[t][r] + bias[l] : 0.0f;
          if (l + 1 < kL) {
            if (kTrain) gp[l][t][r] = gelu_grad(z);
            const bf16 h                  = (bf16)gelu(z);
            act[(l + 1) & 1][rl + r][col] = h;
            hv[r]                         = ok ? h : (bf16)0.0f;
          } else if (!kTrain) {
            if (ok && col < y.dout) a.y[(b0 + rl + r) * y.dout + col] = z;
          } else {
            const float e = ok && col < y.dout ? z - tgt[t][r] : 0.0f;
            sq += (double)e * (double)e;
            gv[r]                         = a.scale * e;
            hv[r]                         = (bf16)gv[r];
            act[(l + 1) & 1][rl + r][col] = hv[r];
          }
        }
        if (kTrain && l + 1 < kL) {
          *reinterpret_cast<bvec*>(up.ht + at) = hv;
        } else if (kTrain) {
#pragma unroll
          for (int r = 0; r < kPer; r++) y.gt[(b0 + rl + r) * y.np + col] = gv[r];
          *reinterpret_cast<bvec*>(y.dt + at) = hv;
        }
      }
    }
    if (kTrain && l == kL - 1) {
#pragma unroll
      for (int m = 32; m > 0; m >>= 1) sq += __shfl_down(sq, m, 64);
      if (lane == 0) red[wave] = sq;
    }
    if (kTrain || l + 1 < kL) __syncthreads();
    w = next;
  }
  if (!kTrain) return;
  if (tid == 0) {
    double s = 0.0;
    for (int i = 0; i < kRowThreads / 64; i++) s += red[i];
    a.partial[blockIdx.x] = s;
  }

  // G of layer l - 1's output = (D_l W_l) gelu'(z), its D in act
#pragma unroll
  for (int l = kL - 1; l > 0; l--) {
    const RowLayer& y    = a.l[l];
    const RowLayer& dst  = a.l[l > 0 ? l - 1 : 0];
    const int       from = (kL - 1 - l + (kL & 1)) & 1;  // act[kL & 1] holds D of the last layer
    RowWeights      next;
    if (l > 1) load_weights(dst.wt, dst.np, dst.kp, wave, lane, next);
    if (wave * 16 < y.kp) {
      f32x4 acc[kRT];
      row_product<kPer, kRT, kLd>(act[from], w, y.np, lane, acc);
#pragma unroll
      for (int t = 0; t < kRT; t++) {
        const int     rl = 4 * kPer * t + row0;
        const int64_t at = operand_index(col, b0 + rl, a.Bp / kKStep);
        bvec          dv;
        fvec          gv;
#pragma unroll
        for (int r = 0; r < kPer; r++) {
          gv[r] = b0 + rl + r < a.B && col < y.din ? acc[t][r] * gp[l > 0 ? l - 1 : 0][t][r] : 0.0f;
          dv[r] = (bf16)gv[r];
          act[from ^ 1][rl + r][col] = dv[r];
        }
#pragma unroll
        for (int r = 0; r < kPer; r++) dst.gt[(b0 + rl + r) * dst.np + col] = gv[r];
        *reinterpret_cast<bvec*>(dst.dt + at) = dv;
      }
    }
    if (l > 1) __syncthreads();
    w = next;
  }
}

// Weight and bias gradients of every layer from H and D: workgroups
// [0, tiles[0]) take 32 x 32 tiles of the first layer's weights (four waves
// of 16 x 16), the next tiles[1] the second's, ..., then four bias columns
// each.  The K range (batch) is cut and summed as mlp_gemm's split-K does.
// kUpdate: Adam on each parameter where its gradient is formed, else the
// gradients go to g.
struct WeightArgs {
  int      layers;
  int      tiles[kRowLayers], tiles_x[kRowLayers];
  int64_t  B, Bp;
  int      splits, k_chunk;
  float*   g;
  Adam     adam;
  RowLayer l[kRowLayers];
};

template <bool kUpdate>
__global__ __launch_bounds__(256) void k_weights(WeightArgs a)
{
  const int lane = (int)threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
  int       w    = (int)blockIdx.x;
#pragma unroll
  for (int l = 0; l < kRowLayers; l++) {
    if (l >= a.layers) break;
    const RowLayer& y = a.l[l];
    if (w >= a.tiles[l]) {
      w -= a.tiles[l];
      continue;
    }
    const int m0 = (w / a.tiles_x[l]) * 32 + (wave >> 1) * 16, n0 = (w % a.tiles_x[l]) * 32 + (wave & 1) * 16;
    if (m0 >= y.dout || n0 >= y.din) return;  // uniform across the wave
    const bf16x8* pd = reinterpret_cast<const bf16x8*>(y.dt + m0 * a.Bp) + lane;
    const bf16x8* ph = reinterpret_cast<const bf16x8*>(y.ht + n0 * a.Bp) + lane;
    // this lane's four parameters, loaded beside the operands
    const int     k = n0 + (lane & 15), n4 = m0 + 4 * (lane >> 4);
    const int64_t i0 = y.w_off + (int64_t)n4 * y.din + k;
    AdamState     old[4];
    if (kUpdate)
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (k < y.din && n4 + r < y.dout) old[r] = adam_load(a.adam, i0 + (int64_t)r * y.din);
    f32x4 sum{0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < a.splits; z++) {
      const int kb = z * a.k_chunk, ke = (int)min(a.Bp, (int64_t)kb + a.k_chunk);
      f32x4     acc{0.f, 0.f, 0.f, 0.f};
      constexpr int kFlight = 16;  // steps whose loads are in flight together
      for (int k0 = kb; k0 < ke; k0 += kFlight * kKStep) {
        bf16x8 d[kFlight], h[kFlight];
#pragma unroll
        for (int s = 0; s < kFlight; s++) {
          const int k = min(k0 + s * kKStep, ke - kKStep);
          d[s]        = pd[2 * k];
          h[s]        = ph[2 * k];
        }
#pragma unroll
        for (int s = 0; s < kFlight; s++)
          if (k0 + s * kKStep < ke) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d[s], h[s], acc, 0, 0, 0);
      }
      if (a.splits == 1)
        sum = acc;
      else
#pragma unroll
        for (int r = 0; r < 4; r++) sum[r] += acc[r];
    }
    if (k >= y.din) return;
    bf16x4 v;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int64_t i = i0 + (int64_t)r * y.din;
      v[r]            = (bf16)0.0f;
      if (n4 + r >= y.dout) continue;
      if (kUpdate) {
        v[r]                               = adam_update(a.adam, i, old[r], sum[r]);
        y.wf[operand_index(n4 + r, k, y.kp / kKStep)] = v[r];
      } else {
        a.g[i] = sum[r];
      }
    }
    if (kUpdate) *reinterpret_cast<bf16x4*>(y.wt + operand_index(k, n4, y.np / kKStep)) = v;
    return;
  }
  // bias columns, as bias_grad_columns sums them
  int n = 4 * w + wave;
#pragma unroll
  for (int l = 0; l < kRowLayers; l++) {
    if (l >= a.layers) break;
    const RowLayer& y = a.l[l];
    if (n >= y.dout) {
      n -= y.dout;
      continue;
    }
    float s = 0.0f;
    for (int64_t b = lane; b < a.B; b += 64) s += y.gt[b * y.np + n];
#pragma unroll
    for (int m = 32; m > 0; m >>= 1) s += __shfl_down(s, m, 64);
    if (lane == 0) {
      if (kUpdate)
        adam_update(a.adam, y.b_off + n, adam_load(a.adam, y.b_off + n), s);
      else
        a.g[y.b_off + n] = s;
    }
    return;
  }
}

// BF16 weights W [dout][din] into the padded copies
__global__ __launch_bounds__(256) void k_pack(const bf16* __restrict__ W, RowLayer y)
{
  const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (i >= y.din * y.dout) return;
  const int  n = i / y.din, k = i % y.din;
  const bf16 v = W[i];
  y.wf[operand_index(n, k, y.kp / kKStep)] = v;
  y.wt[operand_index(k, n, y.np / kKStep)] = v;
}

inline unsigned blocks_of(int64_t n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
struct nsm_mlp {
  int                  device = 0;
  hipStream_t          stream = nullptr;
  std::vector<int>     width;              // d_0 .. d_L
  std::vector<int64_t> w_off, b_off;       // offsets of W_l, b_l in the flat parameter array
  int64_t              num_params = 0;
  float*               p   = nullptr;      // FP32 master parameters
  bf16*                pb  = nullptr;      // BF16 copy
  float*               g   = nullptr;      // gradients
  float *              m1 = nullptr, *m2 = nullptr;
  int64_t              adam_t = 0;
  // activations for a batch of `cap` rows
  int64_t              cap = 0;
  std::vector<float*>  z;   // Z_l, l = 1..L   [cap][d_l] (index l-1)
  std::vector<bf16*>   h;   // H_l, l = 0..L-1 [cap][d_l]
  float*               gf = nullptr;  // G (FP32) [cap][max d]
  bf16*                gb = nullptr;  // D (BF16) [cap][max d]
  float*               gf2 = nullptr;
  bf16*                gb2 = nullptr;
  float*               x32 = nullptr;  // input [cap][d_0]
  float*               t32 = nullptr;  // targets [cap][d_L]
  double*              loss = nullptr; // [loss_cap]
  int64_t              loss_cap = 0;
  double*              loss_part = nullptr;  // [min(passes, kLossChunk)][partials per pass]
  int64_t              loss_part_cap = 0;
  float*               split = nullptr;      // split-K partial products
  int64_t              split_cap = 0;

  // small networks (k_rows, k_weights): padded BF16 weights, transposed
  // activations and gradients of a batch of row_cap rows
  bool                  rows = false;
  std::vector<RowLayer> row;
  bf16*                 row_weights = nullptr;
  bool                  row_stale   = false;  // pb is newer than the padded copies
  char*                 row_batch   = nullptr;
  int64_t               row_cap     = 0;
  float*                y32         = nullptr;  // output [y_cap][d_L] of k_rows' forward pass
  int64_t               y_cap       = 0;
  int64_t               x_cap = 0, t_cap = 0;   // rows of x32, t32

  int L() const { return (int)width.size() - 1; }
  int max_width() const { return *std::max_element(width.begin(), width.end()); }
};

namespace {

// staging mode of an operand with rows at stride s_r and k at stride s_k
int staging(const bf16* p, int64_t s_r, int64_t s_k)
{
  const bool aligned = ((uintptr_t)p % 16) == 0;
  if (aligned && s_k == 1 && s_r % 8 == 0) return kAlongK;
  if (aligned && s_r == 1 && s_k % 8 == 0) return kAlongMN;
  return kScalar;
}

// Staging modes and K ranges of a product cut into `splits` K ranges
// (clamped to its 32-wide steps); returns the split count.
int prepare(GemmArgs& a, int splits)
{
  a.a_stage = staging(a.a, a.a_m, a.a_k);
  a.b_stage = staging(a.b, a.b_n, a.b_k);
  splits    = std::max(1, std::min(splits, (a.K + kKStep - 1) / kKStep));
  a.k_chunk = ((a.K + splits - 1) / splits + kKStep - 1) / kKStep * kKStep;
  return splits;
}

// C = A B with the epilogue `mode`.  splits > 1 (kStoreC only): the K range
// is cut into `splits` parts written to net->split (one M x N block each)
// and summed in ascending order into a.c.
int mlp_gemm(nsm_mlp* net, GemmArgs a, int mode, int splits = 1)
{
  splits         = prepare(a, splits);
  float* final_c = a.c;
  const int64_t mn = (int64_t)a.M * a.ldc;
  if (splits > 1) {
    if (mode != kStoreC || mn * splits > net->split_cap) return fail(NSM_ERR_STATE, "split-K scratch too small");
    a.c            = net->split;
    a.split_stride = mn;
  }
  const dim3 grid(blocks_of(a.M, kTile), blocks_of(a.N, kTile), (unsigned)splits);
  hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(kGemmThreads), 0, net->stream, a, mode);
  MLP_LAUNCHED();
  if (splits > 1) {
    hipLaunchKernelGGL(k_split_sum, dim3(blocks_of(mn, 256)), dim3(256), 0, net->stream, net->split, splits, mn, mn,
                       final_c);
    MLP_LAUNCHED();
  }
  return NSM_OK;
}

void free_batch(nsm_mlp* net)
{
  for (auto* q : net->z) (void)hipFree(q);
  for (auto* q : net->h) (void)hipFree(q);
  net->z.clear();
  net->h.clear();
  for (void* q : {(void*)net->gf, (void*)net->gb, (void*)net->gf2, (void*)net->gb2})
    if (q) (void)hipFree(q);
  net->gf = nullptr;
  net->gb = nullptr;
  net->gf2 = nullptr;
  net->gb2 = nullptr;
  net->cap = 0;
}

// `*buf` of at least rows * width values
template <typename T>
int ensure_rows(T** buf, int64_t* cap, int64_t rows, int64_t width)
{
  if (rows <= *cap) return NSM_OK;
  if (*buf) MLP_HIP(hipFree(*buf));
  *buf = nullptr;
  *cap = 0;
  MLP_HIP(hipMalloc((void**)buf, (size_t)(rows * width) * sizeof(T)));
  *cap = rows;
  return NSM_OK;
}

int ensure_batch(nsm_mlp* net, int64_t B)
{
  if (B <= net->cap) return NSM_OK;
  free_batch(net);
  const int     L  = net->L();
  const int64_t mw = net->max_width();
  net->z.assign((size_t)L, nullptr);
  net->h.assign((size_t)L, nullptr);
  for (int l = 0; l < L; l++) {
    MLP_HIP(hipMalloc((void**)&net->z[(size_t)l], (size_t)(B * net->width[(size_t)l + 1]) * sizeof(float)));
    MLP_HIP(hipMalloc((void**)&net->h[(size_t)l], (size_t)(B * net->width[(size_t)l]) * sizeof(bf16)));
  }
  MLP_HIP(hipMalloc((void**)&net->gf, (size_t)(B * mw) * sizeof(float)));
  MLP_HIP(hipMalloc((void**)&net->gb, (size_t)(B * mw) * sizeof(bf16)));
  MLP_HIP(hipMalloc((void**)&net->gf2, (size_t)(B * mw) * sizeof(float)));
  MLP_HIP(hipMalloc((void**)&net->gb2, (size_t)(B * mw) * sizeof(bf16)));
  net->cap = B;
  return NSM_OK;
}

// Forward pass of B rows already in x32 (converted to BF16 into h[0] unless
// convert_input is false: training converts once); output Z_L in z[L-1].
int forward(nsm_mlp* net, int64_t B, bool convert_input = true)
{
  const int L  = net->L();
  const int d0 = net->width[0];
  if (convert_input) {
    hipLaunchKernelGGL(k_to_bf16, dim3(blocks_of(B * d0, 256)), dim3(256), 0, net->stream, net->x32, net->h[0],
                       B * d0);
    MLP_LAUNCHED();
  }
  for (int l = 1; l <= L; l++) {
    const int din = net->width[(size_t)l - 1], dout = net->width[(size_t)l];
    GemmArgs  a{};
    a.M    = (int)B;
    a.N    = dout;
    a.K    = din;
    a.a    = net->h[(size_t)l - 1];
    a.a_m  = din;
    a.a_k  = 1;
    a.b    = net->pb + net->w_off[(size_t)l - 1];  // B(k, n) = W_l[n][k]
    a.b_k  = 1;
    a.b_n  = din;
    a.c    = net->z[(size_t)l - 1];
    a.ldc  = dout;
    a.bias = net->p + net->b_off[(size_t)l - 1];
    a.h    = l < L ? net->h[(size_t)l] : nullptr;
    int st = mlp_gemm(net, a, l < L ? kHidden : kOutput);
    if (st) return st;
  }
  return NSM_OK;
}

// Gradients of every parameter into net->g from the forward pass against
// t32; the pass's kMseBlocks squared-error partials go to `partial`
// (device; k_mse_total turns them into the loss).  With at most
// kSplitAbove batch rows each layer is one launch (k_layer_backward: weight
// gradient, input gradient and bias gradient side by side), else one per
// product.
int backward(nsm_mlp* net, int64_t B, double* partial)
{
  const int L  = net->L();
  const int dL = net->width[(size_t)L];
  hipLaunchKernelGGL(k_mse, dim3(kMseBlocks), dim3(256), 0, net->stream, net->z[(size_t)L - 1], net->t32, B * dL,
                     net->gf, net->gb, partial);
  MLP_LAUNCHED();
  float* gcur = net->gf;
  bf16*  dcur = net->gb;
  float* gnext = net->gf2;
  bf16*  dnext = net->gb2;
  for (int l = L; l >= 1; l--) {
    const int din = net->width[(size_t)l - 1], dout = net->width[(size_t)l];
    // dW_l[n][k] = sum_b D_l[b][n] H_{l-1}[b][k]
    GemmArgs a{};
    a.M   = dout;
    a.N   = din;
    a.K   = (int)B;
    a.a   = dcur;
    a.a_m = 1;
    a.a_k = dout;
    a.b   = net->h[(size_t)l - 1];
    a.b_k = din;
    a.b_n = 1;
    a.c   = net->g + net->w_off[(size_t)l - 1];
    a.ldc = din;
    // G_{l-1}[b][k] = (sum_n D_l[b][n] W_l[n][k]) gelu'(Z_{l-1}[b][k])
    GemmArgs d{};
    d.M   = (int)B;
    d.N   = din;
    d.K   = dout;
    d.a   = dcur;
    d.a_m = dout;
    d.a_k = 1;
    d.b   = net->pb + net->w_off[(size_t)l - 1];
    d.b_k = din;
    d.b_n = 1;
    d.c   = gnext;
    d.ldc = din;
    d.h   = dnext;
    d.z   = l > 1 ? net->z[(size_t)l - 2] : nullptr;
    float* const db = net->g + net->b_off[(size_t)l - 1];
    if (B <= kSplitAbove) {
      LayerBackward lb{};
      lb.prod[0]    = a;
      lb.mode[0]    = kStoreC;
      prepare(lb.prod[0], 1);
      lb.tiles_x[0] = (int)blocks_of(a.N, kTile);
      lb.tiles[0]   = lb.tiles_x[0] * (int)blocks_of(a.M, kTile);
      if (l > 1) {
        lb.prod[1]    = d;
        lb.mode[1]    = kBackHidden;
        prepare(lb.prod[1], 1);
        lb.tiles_x[1] = (int)blocks_of(d.N, kTile);
        lb.tiles[1]   = lb.tiles_x[1] * (int)blocks_of(d.M, kTile);
      }
      lb.G  = gcur;
      lb.B  = B;
      lb.N  = dout;
      lb.db = db;
      const unsigned grid = (unsigned)(lb.tiles[0] + lb.tiles[1]) + blocks_of(dout, 4);
      hipLaunchKernelGGL(k_layer_backward, dim3(grid), dim3(kGemmThreads), 0, net->stream, lb);
      MLP_LAUNCHED();
    } else {
      const int splits = (int)std::min<int64_t>(kMaxSplits, (B + kSplitAbove - 1) / kSplitAbove);
      int       st     = mlp_gemm(net, a, kStoreC, splits);
      if (st) return st;
      hipLaunchKernelGGL(k_bias_grad, dim3(blocks_of(dout, 4)), dim3(256), 0, net->stream, gcur, B, dout, db);
      MLP_LAUNCHED();
      if (l > 1 && (st = mlp_gemm(net, d, kBackHidden))) return st;
    }
    std::swap(gcur, gnext);
    std::swap(dcur, dnext);
  }
  return NSM_OK;
}

// ---- small networks: k_rows and k_weights
// Training batches up to kRowBatch rows; longer ones, and other networks, run
// layer by layer.  The line is where the measurements it was drawn from ended,
// no crossover: us per iteration layer by layer / in two
// launches, 4-256-256-256-64 16,384 rows 693 / 205, 32,768 1348 / 445, 131,072
// 6896 / 2156; 3-16-1 16,385 rows 251 / 123, 131,072 1786 / 780.
constexpr int64_t kRowBatch = 16384;
// A prediction of more rows goes layer by layer where no width passes 32: then
// 2 of k_rows' 16 waves have columns, and with every CU busy that costs more
// than the launches.  Layer by layer / k_rows: 3-16-1, 16,384 rows 46 / 47 us,
// 60,000 81 / 92, 1e6 829 / 1059; 4-32-32-8, 16,384 76 / 74, 60,000 200 / 213,
// 1e6 3.05 / 3.40 ms; 8-33-33-33-4, 60,000 198 / 188 us, 1e6 3.17 / 3.20 ms;
// 4-64-64-8, 60,000 215 / 215 us, 1e6 3.41 / 3.41 ms.
constexpr int kNarrow = 32;

bool fits_rows(const std::vector<int>& width)
{
  return (int)width.size() - 1 <= kRowLayers && *std::max_element(width.begin(), width.end()) <= kRowWidth;
}

// padded weights (zeroed once: the padding is never written)
int create_rows(nsm_mlp* net)
{
  int64_t total = 0;
  net->row.resize((size_t)net->L());
  for (int l = 0; l < net->L(); l++) {
    RowLayer& y = net->row[(size_t)l];
    y           = RowLayer{};
    y.din       = net->width[(size_t)l];
    y.dout      = net->width[(size_t)l + 1];
    y.kp        = (y.din + 31) / 32 * 32;
    y.np        = (y.dout + 31) / 32 * 32;
    y.w_off     = net->w_off[(size_t)l];
    y.b_off     = net->b_off[(size_t)l];
    y.bias      = net->p + y.b_off;
    total += 2 * (int64_t)y.kp * y.np;
  }
  MLP_HIP(hipMalloc((void**)&net->row_weights, (size_t)total * sizeof(bf16)));
  MLP_HIP(hipMemsetAsync(net->row_weights, 0, (size_t)total * sizeof(bf16), net->stream));
  bf16* q = net->row_weights;
  for (RowLayer& y : net->row) {
    y.wf = q;
    y.wt = q + (int64_t)y.kp * y.np;
    q += 2 * (int64_t)y.kp * y.np;
  }
  net->rows      = true;
  net->row_stale = true;
  return NSM_OK;
}

int pack_rows(nsm_mlp* net)
{
  if (!net->row_stale) return NSM_OK;
  for (const RowLayer& y : net->row) {
    hipLaunchKernelGGL(k_pack, dim3(blocks_of((int64_t)y.din * y.dout, 256)), dim3(256), 0, net->stream,
                       net->pb + y.w_off, y);
    MLP_LAUNCHED();
  }
  net->row_stale = false;
  return NSM_OK;
}

template <int kPer, int kRT, bool kTrain>
int launch_rows(nsm_mlp* net, const RowArgs& a, int64_t rows)
{
  const dim3 g(blocks_of(rows, 4 * kPer * kRT)), b(kRowThreads);
  switch (net->L()) {
    case 1: hipLaunchKernelGGL((k_rows<1, kPer, kRT, kTrain>), g, b, 0, net->stream, a); break;
    case 2: hipLaunchKernelGGL((k_rows<2, kPer, kRT, kTrain>), g, b, 0, net->stream, a); break;
    case 3: hipLaunchKernelGGL((k_rows<3, kPer, kRT, kTrain>), g, b, 0, net->stream, a); break;
    default: hipLaunchKernelGGL((k_rows<4, kPer, kRT, kTrain>), g, b, 0, net->stream, a);
  }
  MLP_LAUNCHED();
  return NSM_OK;
}

// forward pass of the B rows in x32 into y32
int forward_rows(nsm_mlp* net, int64_t B)
{
  int st = pack_rows(net);
  if (st || (st = ensure_rows(&net->y32, &net->y_cap, B, net->width.back()))) return st;
  RowArgs a{};
  a.B = a.Bp = B;
  a.x = net->x32;
  a.y = net->y32;
  std::copy(net->row.begin(), net->row.end(), a.l);
  // 4, 16 or 32 rows per workgroup: few while that spreads the call over more
  // CUs, many to share the weight loads once every CU has a workgroup
  if (B <= 1024) return launch_rows<1, 1, false>(net, a, B);
  return B <= 4096 ? launch_rows<4, 1, false>(net, a, B) : launch_rows<4, 2, false>(net, a, B);
}

// Rows per workgroup of a training pass: 4 while that leaves at most one
// workgroup per CU of 256 (a workgroup's time is its chain of products and
// hardly depends on its rows), then 8, then 16.
int train_group(int64_t B) { return B <= 1024 ? 4 : B <= 2048 ? 8 : 16; }

int64_t row_padded(int64_t B) { return (B + 31) / 32 * 32; }

int64_t row_partials(int64_t B) { return row_padded(B) / train_group(B); }

// activations and gradients of a training pass of B rows
int ensure_row_batch(nsm_mlp* net, int64_t B)
{
  int64_t per_row = 0;  // bytes
  for (const RowLayer& y : net->row) per_row += 2 * y.kp + 6 * y.np;
  return ensure_rows(&net->row_batch, &net->row_cap, row_padded(B), per_row);
}

// One pass over the B rows in x32, t32 (after ensure_row_batch): squared-error partials
// (row_partials(B) of them) and gradients, which go to net->g, or through
// Adam when `adam` is given.
int train_rows(nsm_mlp* net, int64_t B, double* partial, const Adam* adam)
{
  int st = pack_rows(net);
  if (st) return st;
  const int64_t Bp = row_padded(B);
  char* q = net->row_batch;  // every array a multiple of 64 bytes
  for (RowLayer& y : net->row) {
    y.ht = (bf16*)q, q += 2 * y.kp * Bp;
    y.dt = (bf16*)q, q += 2 * y.np * Bp;
    y.gt = (float*)q, q += 4 * y.np * Bp;
  }
  RowArgs a{};
  a.B       = B;
  a.Bp      = Bp;
  a.x       = net->x32;
  a.target  = net->t32;
  a.partial = partial;
  a.scale   = 2.0f / (float)(B * net->width.back());
  std::copy(net->row.begin(), net->row.end(), a.l);
  switch (train_group(B)) {
    case 4: st = launch_rows<1, 1, true>(net, a, Bp); break;
    case 8: st = launch_rows<2, 1, true>(net, a, Bp); break;
    default: st = launch_rows<4, 1, true>(net, a, Bp);
  }
  if (st) return st;

  WeightArgs w{};
  w.layers = net->L();
  w.B      = B;
  w.Bp     = Bp;
  GemmArgs split{};
  split.K   = (int)B;
  w.splits  = prepare(split, B <= kSplitAbove ? 1 : (int)std::min<int64_t>(kMaxSplits, (B + kSplitAbove - 1) / kSplitAbove));
  w.k_chunk = split.k_chunk;
  w.g       = net->g;
  unsigned grid = 0;
  int      cols = 0;
  for (int l = 0; l < net->L(); l++) {
    w.l[l]       = net->row[(size_t)l];
    w.tiles_x[l] = w.l[l].kp / 32;
    w.tiles[l]   = w.tiles_x[l] * (w.l[l].np / 32);
    grid += (unsigned)w.tiles[l];
    cols += w.l[l].dout;
  }
  grid += blocks_of(cols, 4);
  if (adam) {
    w.adam = *adam;
    hipLaunchKernelGGL(k_weights<true>, dim3(grid), dim3(256), 0, net->stream, w);
  } else {
    hipLaunchKernelGGL(k_weights<false>, dim3(grid), dim3(256), 0, net->stream, w);
  }
  MLP_LAUNCHED();
  return NSM_OK;
}

uint64_t splitmix(uint64_t& s)
{
  uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
  z          = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z          = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}

int upload_params(nsm_mlp* net, const float* host)
{
  MLP_HIP(hipMemcpyAsync(net->p, host, (size_t)net->num_params * sizeof(float), hipMemcpyHostToDevice,
                         net->stream));
  hipLaunchKernelGGL(k_to_bf16, dim3(blocks_of(net->num_params, 256)), dim3(256), 0, net->stream, net->p, net->pb,
                     net->num_params);
  MLP_LAUNCHED();
  net->row_stale = true;
  MLP_HIP(hipMemsetAsync(net->m1, 0, (size_t)net->num_params * sizeof(float), net->stream));
  MLP_HIP(hipMemsetAsync(net->m2, 0, (size_t)net->num_params * sizeof(float), net->stream));
  net->adam_t = 0;
  MLP_HIP(hipStreamSynchronize(net->stream));
  return NSM_OK;
}

int load_rows(nsm_mlp* net, int64_t B, const float* x, const float* t)
{
  int st = ensure_rows(&net->x32, &net->x_cap, B, net->width[0]);
  if (st || (t && (st = ensure_rows(&net->t32, &net->t_cap, B, net->width.back())))) return st;
  MLP_HIP(hipMemcpyAsync(net->x32, x, (size_t)(B * net->width[0]) * sizeof(float), hipMemcpyHostToDevice,
                         net->stream));
  if (t)
    MLP_HIP(hipMemcpyAsync(net->t32, t, (size_t)(B * net->width.back()) * sizeof(float), hipMemcpyHostToDevice,
                           net->stream));
  return NSM_OK;
}

// squared-error partials of up to kLossChunk passes are kept on the device
// and turned into losses by one k_mse_total launch per chunk
constexpr int kLossChunk = 4096;

// losses for `passes` forward/backward passes and `per_pass` partials for
// min(passes, kLossChunk) of them
int ensure_loss(nsm_mlp* net, int64_t passes, int64_t per_pass)
{
  int st = ensure_rows(&net->loss, &net->loss_cap, passes, 1);
  if (st) return st;
  return ensure_rows(&net->loss_part, &net->loss_part_cap, std::min<int64_t>(passes, kLossChunk) * per_pass, 1);
}

}  // namespace

extern "C" {

int nsm_mlp_create(int num_layers, const int* widths, uint64_t seed, nsm_mlp** out)
{
  if (!out || !widths) return fail(NSM_ERR_ARG, "null argument");
  *out = nullptr;
  if (num_layers < 1 || num_layers > 16) return fail(NSM_ERR_ARG, "1 to 16 layers");
  for (int l = 0; l <= num_layers; l++)
    if (widths[l] < 1 || widths[l] > 4096) return fail(NSM_ERR_ARG, "layer widths must be in [1, 4096]");
  nsm_mlp* net = new nsm_mlp();
  net->width.assign(widths, widths + num_layers + 1);
  int64_t off = 0;
  for (int l = 1; l <= num_layers; l++) {
    net->w_off.push_back(off);
    off += (int64_t)widths[l] * widths[l - 1];
    net->b_off.push_back(off);
    off += widths[l];
  }
  net->num_params = off;
  auto cleanup    = [&](int st) {
    nsm_mlp_destroy(net);
    return st;
  };
  if (hipGetDevice(&net->device) != hipSuccess) return cleanup(fail(NSM_ERR_HIP, "no HIP device"));
  if (hipStreamCreateWithFlags(&net->stream, hipStreamNonBlocking) != hipSuccess)
    return cleanup(fail(NSM_ERR_HIP, "hipStreamCreate failed"));
  const size_t n = (size_t)net->num_params;
  int64_t max_w = 0;
  for (int l = 1; l <= num_layers; l++) max_w = std::max<int64_t>(max_w, (int64_t)widths[l] * widths[l - 1]);
  net->split_cap = kMaxSplits * max_w;
  if (hipMalloc((void**)&net->p, n * 4) != hipSuccess || hipMalloc((void**)&net->pb, n * 2) != hipSuccess ||
      hipMalloc((void**)&net->g, n * 4) != hipSuccess || hipMalloc((void**)&net->m1, n * 4) != hipSuccess ||
      hipMalloc((void**)&net->m2, n * 4) != hipSuccess ||
      hipMalloc((void**)&net->split, (size_t)net->split_cap * 4) != hipSuccess)
    return cleanup(fail(NSM_ERR_NOMEM, "device allocation of the parameters failed"));
  if (fits_rows(net->width)) {
    const int rst = create_rows(net);
    if (rst) return cleanup(rst);
  }
  // uniform(-a, a) weights with a = sqrt(6 / (fan_in + fan_out)), zero biases
  std::vector<float> init(n, 0.0f);
  uint64_t           s = seed;
  for (int l = 1; l <= num_layers; l++) {
    const double a = std::sqrt(6.0 / (double)(widths[l - 1] + widths[l]));
    for (int64_t i = 0; i < (int64_t)widths[l] * widths[l - 1]; i++) {
      const double u = (double)(splitmix(s) >> 11) * (1.0 / 9007199254740992.0);
      init[(size_t)(net->w_off[(size_t)l - 1] + i)] = (float)((2.0 * u - 1.0) * a);
    }
  }
  int st = upload_params(net, init.data());
  if (st) return cleanup(st);
  *out = net;
  return NSM_OK;
}

int nsm_mlp_destroy(nsm_mlp* net)
{
  if (!net) return NSM_OK;
  (void)hipSetDevice(net->device);
  if (net->stream) (void)hipStreamSynchronize(net->stream);
  free_batch(net);
  for (void* q : {(void*)net->p, (void*)net->pb, (void*)net->g, (void*)net->m1, (void*)net->m2, (void*)net->loss,
                  (void*)net->loss_part, (void*)net->split, (void*)net->x32, (void*)net->t32, (void*)net->y32,
                  (void*)net->row_weights, (void*)net->row_batch})
    if (q) (void)hipFree(q);
  if (net->stream) (void)hipStreamDestroy(net->stream);
  delete net;
  return NSM_OK;
}

int nsm_mlp_num_parameters(nsm_mlp* net, int64_t* n)
{
  if (!net || !n) return fail(NSM_ERR_ARG, "null argument");
  *n = net->num_params;
  return NSM_OK;
}

int nsm_mlp_get_parameters(nsm_mlp* net, float* out)
{
  if (!net || !out) return fail(NSM_ERR_ARG, "null argument");
  MLP_HIP(hipSetDevice(net->device));
  MLP_HIP(hipMemcpyAsync(out, net->p, (size_t)net->num_params * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  MLP_HIP(hipStreamSynchronize(net->stream));
  return NSM_OK;
}

int nsm_mlp_set_parameters(nsm_mlp* net, const float* in)
{
  if (!net || !in) return fail(NSM_ERR_ARG, "null argument");
  MLP_HIP(hipSetDevice(net->device));
  return upload_params(net, in);
}

int nsm_mlp_forward(nsm_mlp* net, int64_t batch, const float* x, float* y)
{
  if (!net || (batch > 0 && (!x || !y))) return fail(NSM_ERR_ARG, "null argument");
  if (batch < 0 || batch > (1 << 24)) return fail(NSM_ERR_ARG, "batch out of range");
  if (batch == 0) return NSM_OK;
  MLP_HIP(hipSetDevice(net->device));
  int st = load_rows(net, batch, x, nullptr);
  const bool rows = net->rows && (batch <= kRowBatch || net->max_width() > kNarrow);
  if (st || (st = rows ? forward_rows(net, batch) : ensure_batch(net, batch))) return st;
  if (!rows && (st = forward(net, batch))) return st;
  MLP_HIP(hipMemcpyAsync(y, rows ? net->y32 : net->z.back(), (size_t)(batch * net->width.back()) * sizeof(float),
                         hipMemcpyDeviceToHost, net->stream));
  MLP_HIP(hipStreamSynchronize(net->stream));
  return NSM_OK;
}

int nsm_mlp_loss_gradients(nsm_mlp* net, int64_t batch, const float* x, const float* t, double* loss, float* grad)
{
  if (!net || !x || !t || !loss || !grad) return fail(NSM_ERR_ARG, "null argument");
  if (batch < 1 || batch > (1 << 24)) return fail(NSM_ERR_ARG, "batch out of range");
  MLP_HIP(hipSetDevice(net->device));
  int st = load_rows(net, batch, x, t);
  if (st) return st;
  const int64_t n = batch * net->width.back();
  const bool    rows     = net->rows && batch <= kRowBatch;
  const int64_t per_pass = rows ? row_partials(batch) : kMseBlocks;
  if ((st = ensure_loss(net, 1, per_pass)) || (st = rows ? ensure_row_batch(net, batch) : ensure_batch(net, batch)))
    return st;
  if (rows)
    st = train_rows(net, batch, net->loss_part, nullptr);
  else if (!(st = forward(net, batch)))
    st = backward(net, batch, net->loss_part);
  if (st) return st;
  hipLaunchKernelGGL(k_mse_total, dim3(1), dim3(64), 0, net->stream, net->loss_part, (int)per_pass, n, net->loss);
  MLP_LAUNCHED();
  MLP_HIP(hipMemcpyAsync(loss, net->loss, sizeof(double), hipMemcpyDeviceToHost, net->stream));
  MLP_HIP(hipMemcpyAsync(grad, net->g, (size_t)net->num_params * sizeof(float), hipMemcpyDeviceToHost,
                         net->stream));
  MLP_HIP(hipStreamSynchronize(net->stream));
  return NSM_OK;
}

int nsm_mlp_train(nsm_mlp* net, int64_t batch, const float* x, const float* t, int iterations, double lr,
                  double lr_final, double* loss_history)
{
  if (!net || !x || !t) return fail(NSM_ERR_ARG, "null argument");
  if (batch < 1 || batch > (1 << 24) || iterations < 0) return fail(NSM_ERR_ARG, "invalid batch or iterations");
  if (!(lr > 0.0) || !(lr_final > 0.0)) return fail(NSM_ERR_ARG, "learning rates must be positive");
  MLP_HIP(hipSetDevice(net->device));
  int st = load_rows(net, batch, x, t);
  if (st) return st;
  const bool    rows     = net->rows && batch <= kRowBatch;
  const int64_t per_pass = rows ? row_partials(batch) : kMseBlocks;
  // every buffer before the first step: a call without memory trains nothing
  if ((st = ensure_loss(net, iterations, per_pass)) ||
      (st = rows ? ensure_row_batch(net, batch) : ensure_batch(net, batch)))
    return st;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int it = 0; it < iterations; it++) {
    // cosine decay from lr to lr_final
    const double c   = 0.5 * (1.0 + std::cos(M_PI * (double)it / (double)std::max(iterations - 1, 1)));
    const float  lri = (float)(lr_final + (lr - lr_final) * c);
    net->adam_t++;
    const float c1 = (float)(1.0 - std::pow((double)b1, (double)net->adam_t));
    const float c2 = (float)(1.0 - std::pow((double)b2, (double)net->adam_t));
    const Adam    adam{net->p, net->m1, net->m2, net->pb, lri, b1, b2, c1, c2, eps};
    double* const partial = net->loss_part + (int64_t)(it % kLossChunk) * per_pass;
    if (rows) {
      if ((st = train_rows(net, batch, partial, &adam))) return st;
    } else {
      if ((st = forward(net, batch, it == 0)) || (st = backward(net, batch, partial))) return st;
      hipLaunchKernelGGL(k_adam, dim3(blocks_of(net->num_params, 256)), dim3(256), 0, net->stream, adam, net->g,
                         net->num_params);
      MLP_LAUNCHED();
      net->row_stale = true;
    }
    // the losses of a full chunk of iterations (or of the last one)
    if ((it + 1) % kLossChunk == 0 || it + 1 == iterations) {
      const int first = it - it % kLossChunk;
      hipLaunchKernelGGL(k_mse_total, dim3((unsigned)(it + 1 - first)), dim3(64), 0, net->stream, net->loss_part,
                         (int)per_pass, batch * net->width.back(), net->loss + first);
      MLP_LAUNCHED();
    }
  }
  if (loss_history && iterations > 0)
    MLP_HIP(hipMemcpyAsync(loss_history, net->loss, (size_t)iterations * sizeof(double), hipMemcpyDeviceToHost,
                           net->stream));
  MLP_HIP(hipStreamSynchronize(net->stream));
  return NSM_OK;
}

}  // extern "C"
