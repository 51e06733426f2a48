// Multilayer perceptron on MFMA: BF16 operands, FP32 accumulation.
//
// The network maps a chemistry state and time step to the increment of the
// state over that step; it is trained on the GPU with the kernels below
// (forward, mean-squared-error loss, backward, Adam) and evaluated by the
// surrogate step.  Layers: nin -> hidden (GELU) x nhl -> nout, all linear
// layers y = x W^T + b with W[out][in] row-major.  Widths are padded to
// multiples of 64 (the GEMM tile); padded weights, biases and activations
// stay exactly zero, so the padded network computes the unpadded one.
//
// Networks whose widths fit a workgroup's LDS row (all at most 256; the ones of
// this repository have 64, 256 and 64) take fused kernels: one launch for the
// whole forward pass (mlp_infer_kernel: a tile of rows goes through all layers
// with its activations in LDS, the weights come from L2 as MFMA fragments), and
// three for a training step (forward, loss and input gradients; all weight
// gradients, split over the batch; their sums and Adam).  Wider networks go
// layer by layer through the product kernel:
//
// GEMM: C[M][N] = sum_k A(m,k) B(k,n) on 64x64 output tiles, 4 waves per
// workgroup, each wave 32x32 as 2x2 v_mfma_f32_16x16x32_bf16 blocks, K in
// steps of 32 staged through LDS.  Operands are addressed by element strides
// so the three products of a layer (x W^T, dY W, dY^T x) use the same kernel
// with no transposed copies; the load path is chosen by which stride is 1.
// Entry points: include/tiger_mlp.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/tiger_mlp.h"

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg) {
  g_err = msg;
  return code;
}

#define HIP_TRY(x)                                                                           \
  do {                                                                                       \
    hipError_t e_ = (x);                                                                     \
    if (e_ != hipSuccess) return fail(TGR_MLP_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kTile = 64;   // output tile (M and N)
constexpr int kKStep = 32;  // K per LDS stage
constexpr int kLdsRow = kKStep + 8;  // bf16 elements per LDS row (80 B: 16-byte aligned, staggered banks)

// round to nearest even; NaN stays a quiet NaN (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// GELU(x) = x Phi(x) with the normal CDF through erf; derivative Phi(x) + x phi(x)
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

__device__ __forceinline__ float gelu_grad(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// both, with one erf; the same values
__device__ __forceinline__ float gelu_both(float x, float& d) {
  const float c = 1.0f + erff(x * 0.70710678118654752f);
  d = 0.5f * c + x * 0.39894228040143268f * expf(-0.5f * x * x);
  return 0.5f * x * c;
}

// four outputs of a row, aligned as floats are: the caller's array may be a view
// that starts anywhere in a larger one (the hardware takes the store as one
// instruction either way)
typedef float row4 __attribute__((ext_vector_type(4), aligned(4)));

enum Act { kNone = 0, kGelu = 1, kGeluGrad = 2 };

struct GemmArgs {
  const uint16_t* A;
  int64_t sam, sak;  // A(m,k) = A[m*sam + k*sak]
  const uint16_t* B;
  int64_t sbk, sbn;  // B(k,n) = B[k*sbk + n*sbn]
  int M, N, K;       // multiples of 64, 64, 32
  const float* bias;  // [N] or null
  int act;
  const float* aux;  // kGeluGrad: pre-activation, aux[m*ldaux + n]
  int64_t ldaux;
  float* pre;  // kGelu: pre-activation out (or null)
  int64_t ldpre;
  float* out_f;  // fp32 out (or null)
  int64_t ldf;
  uint16_t* out_h;  // bf16 out (or null)
  int64_t ldh;
  int n_valid;  // columns n >= n_valid are written as 0
  int ksplit;   // > 1: workgroup z sums K range z of ksplit into out_f + z * M * ldf (no epilogue)
};

// AK: A's k stride is 1 (else its m stride is 1); BK: B's k stride is 1 (else its n stride is 1).
template <bool AK, bool BK>
__global__ __launch_bounds__(256) void gemm_bf16_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[kTile * kLdsRow];
  __shared__ __attribute__((aligned(16))) uint16_t Bs[kTile * kLdsRow];
  const int t = threadIdx.x;
  const int lane = t & 63, w = t >> 6;
  const int m0 = blockIdx.y * kTile, n0 = blockIdx.x * kTile;
  const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
  const int kchunk = g.K / g.ksplit;
  const int kbeg = blockIdx.z * kchunk, kend = kbeg + kchunk;
  f32x4 acc[2][2];
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int k0 = kbeg; k0 < kend; k0 += kKStep) {
    // global -> registers: 8 bf16 of A and 8 of B per thread (16-byte loads)
    uint4 ra, rb;
    int ar, ac, br, bc;
    if (AK) {  // row m = t/4, k chunk (t%4)*8
      ar = t >> 2;
      ac = (t & 3) * 8;
      ra = *reinterpret_cast<const uint4*>(g.A + (int64_t)(m0 + ar) * g.sam + (k0 + ac));
    } else {  // k = t/8, m chunk (t%8)*8
      ar = (t & 7) * 8;
      ac = t >> 3;
      ra = *reinterpret_cast<const uint4*>(g.A + (int64_t)(k0 + ac) * g.sak + (m0 + ar));
    }
    if (BK) {
      br = t >> 2;
      bc = (t & 3) * 8;
      rb = *reinterpret_cast<const uint4*>(g.B + (int64_t)(n0 + br) * g.sbn + (k0 + bc));
    } else {
      br = (t & 7) * 8;
      bc = t >> 3;
      rb = *reinterpret_cast<const uint4*>(g.B + (int64_t)(k0 + bc) * g.sbk + (n0 + br));
    }
    __syncthreads();  // previous stage's reads are done
    if (AK) {
      *reinterpret_cast<uint4*>(&As[ar * kLdsRow + ac]) = ra;
    } else {
      const uint16_t* e = reinterpret_cast<const uint16_t*>(&ra);
      for (int i = 0; i < 8; ++i) As[(ar + i) * kLdsRow + ac] = e[i];
    }
    if (BK) {
      *reinterpret_cast<uint4*>(&Bs[br * kLdsRow + bc]) = rb;
    } else {
      const uint16_t* e = reinterpret_cast<const uint16_t*>(&rb);
      for (int i = 0; i < 8; ++i) Bs[(br + i) * kLdsRow + bc] = e[i];
    }
    __syncthreads();
    // MFMA 16x16x32: lane l holds row (l%16) of A and column (l%16) of B,
    // k = (l/16)*8 .. +8 of this stage (the same k split for A and B)
    const int r = lane & 15, kq = (lane >> 4) * 8;
    bf16x8 a[2], b[2];
    for (int i = 0; i < 2; ++i)
      a[i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&As[(wm + i * 16 + r) * kLdsRow + kq]));
    for (int j = 0; j < 2; ++j)
      b[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(&Bs[(wn + j * 16 + r) * kLdsRow + kq]));
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
  }

  // epilogue: lane l holds rows (l/16)*4 + 0..3, column l%16 of each 16x16 block
  if (g.ksplit > 1) {  // partial sums of this K range
    float* part = g.out_f + (int64_t)blockIdx.z * g.M * g.ldf;
    for (int i = 0; i < 2; ++i)
      for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn + j * 16 + (lane & 15);
        for (int q = 0; q < 4; ++q) part[(int64_t)(m0 + wm + i * 16 + (lane >> 4) * 4 + q) * g.ldf + col] = acc[i][j][q];
      }
    return;
  }
  for (int i = 0; i < 2; ++i)
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + wn + j * 16 + (lane & 15);
      const float bias = g.bias ? g.bias[col] : 0.0f;
      for (int q = 0; q < 4; ++q) {
        const int row = m0 + wm + i * 16 + (lane >> 4) * 4 + q;
        float v = acc[i][j][q] + bias;
        if (g.act == kGelu) {
          if (g.pre) g.pre[(int64_t)row * g.ldpre + col] = v;
          v = gelu(v);
        } else if (g.act == kGeluGrad) {
          v *= gelu_grad(g.aux[(int64_t)row * g.ldaux + col]);
        }
        if (col >= g.n_valid) v = 0.0f;
        if (g.out_f) g.out_f[(int64_t)row * g.ldf + col] = v;
        if (g.out_h) g.out_h[(int64_t)row * g.ldh + col] = f2bf(v);
      }
    }
}

// Mean-squared error over the first nout columns of out[B][ld] against
// tgt[B][nout]: dY = 2 (out - tgt) / (B nout) (0 in the padded columns) as
// fp32 and bf16, and per-block partial sums of the squared error.
__global__ __launch_bounds__(256) void mse_grad_kernel(const float* out, int64_t ld, const float* tgt, int nout,
                                                      int64_t B, float* dyf, uint16_t* dyh, float* part) {
  __shared__ float red[256];
  const float scale = 2.0f / ((float)B * (float)nout);
  float s = 0.0f;
  const int64_t total = B * ld;
  for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
    const int64_t row = e / ld;
    const int col = (int)(e - row * ld);
    float d = 0.0f;
    if (col < nout) d = out[e] - tgt[row * nout + col];
    s += d * d;
    dyf[e] = scale * d;
    dyh[e] = f2bf(scale * d);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

// loss = sum(part[0:n]) / count, one workgroup
__global__ __launch_bounds__(256) void finish_loss_kernel(const float* part, int n, float inv_count, float* loss) {
  __shared__ float red[256];
  float s = 0.0f;
  for (int i = threadIdx.x; i < n; i += 256) s += part[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = red[0] * inv_count;
}

// part[chunk][n] = sum over the rows of chunk `blockIdx.y` of y[row][n]; 64
// columns per workgroup, 4 row groups
__global__ __launch_bounds__(256) void colsum_kernel(const float* y, int64_t ld, int64_t rows, int64_t rows_per_chunk,
                                                    float* part, int n) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), rg = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.y * rows_per_chunk;
  const int64_t r1 = r0 + rows_per_chunk < rows ? r0 + rows_per_chunk : rows;
  float s = 0.0f;
  for (int64_t r = r0 + rg; r < r1; r += 4) s += y[r * ld + c];
  red[rg][threadIdx.x & 63] = s;
  __syncthreads();
  if (rg == 0) part[(int64_t)blockIdx.y * n + c] = (red[0][c & 63] + red[1][c & 63]) + (red[2][c & 63] + red[3][c & 63]);
}

// out[i] = sum_z part[z][i], i < n (split-K and chunked column sums)
__global__ __launch_bounds__(256) void sum_parts_kernel(const float* part, int nparts, int64_t n, float* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    float s = 0.0f;
    for (int z = 0; z < nparts; ++z) s += part[(int64_t)z * n + i];
    out[i] = s;
  }
}

// Adam with bias correction folded into lr_t and eps_t; keeps the bf16 copy in step
__global__ __launch_bounds__(256) void adam_kernel(float* p, const float* gr, float* m, float* v, uint16_t* pb,
                                                  int64_t n, float lr_t, float b1, float b2, float eps_t) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr_t * mi / (sqrtf(vi) + eps_t);
    p[i] = pi;
    pb[i] = f2bf(pi);
  }
}

__global__ __launch_bounds__(256) void to_bf16_kernel(const float* p, uint16_t* pb, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    pb[i] = f2bf(p[i]);
}

// ---- fused passes (widths at most kWide) --------------------------------------

constexpr int kWide = 256;           // widest layer of the fused kernels
constexpr int kActRow = kWide + 8;   // bf16 elements per activation row in LDS (528 B: staggered banks)
constexpr int kFusedWaves = 8;       // inference: a wave per 32 columns
constexpr int kTrainWaves = kWide / 16;
constexpr int kMaxLin = 17;

struct FusedArgs {
  const uint16_t* x;  // [B][fin[0]]
  int64_t B;          // rows, a multiple of 64
  int nlin, nout;
  int fin[kMaxLin], fout[kMaxLin];
  int64_t offw[kMaxLin], offb[kMaxLin];  // in the flat parameter vector
  const float* p;        // parameters (biases)
  const uint16_t *pb, *pt;  // bf16 weights W[out][in] and transposed [in][out], same offsets
  float* out;            // inference: [B][fout.back()]
  // training
  const float* tgt;   // [B][nout]
  float scale;        // 2 / (B nout)
  float* dact;        // [nlin - 1][B][hidden], GELU' at the hidden pre-activations
  float* dyf;         // output gradients of layer l at offd[l] B, [B][fout[l]]
  uint16_t* xt;       // inputs of every layer, transposed: [sum fin][B]
  uint16_t* dt;       // output gradients of every layer, transposed: [sum fout][B]
  int offx[kMaxLin], offd[kMaxLin];  // first row of layer l in xt / dt
  int ks[kMaxLin];    // slices of the batch in the weight gradient of layer l
  int nch, rpc;       // row chunks of the bias gradients and their rows
  float* bpart;       // [nch][sum fout] column sums of the output gradients
  float* lpart;       // [workgroups] sums of squared errors
};

__device__ __forceinline__ bf16x8 frag(const uint16_t* q) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(q));
}

// acc[i][j] = the weight rows n0 + 128 j .. of W[.][K] (K a multiple of 64) times
// rows 16 i .. of As: the wave's column tiles j with 128 j + n0 < N.  As is the
// MFMA's N operand, so a lane ends with four consecutive columns of one row.
template <int MT>
__device__ __forceinline__ void tile_product(f32x4 (&acc)[MT][2], const uint16_t* As, const uint16_t* W, int K, int n0,
                                             int N, int lane) {
  const int r = lane & 15, kq = (lane >> 4) * 8;
  const bool on[2] = {n0 < N, n0 + 128 < N};
  const uint16_t* w0 = W + (int64_t)(n0 + r) * K + kq;
  const uint16_t* w1 = w0 + (int64_t)128 * K;
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (!on[0]) return;
  // the next 64 of K are loaded while these multiply
  bf16x8 b[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    b[0][h] = frag(w0 + 32 * h);
    if (on[1]) b[1][h] = frag(w1 + 32 * h);
  }
  for (int k0 = 0; k0 < K; k0 += 64) {
    bf16x8 c[2][2];
    const int kn = k0 + 64 < K ? k0 + 64 : 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      c[0][h] = frag(w0 + kn + 32 * h);
      if (on[1]) c[1][h] = frag(w1 + kn + 32 * h);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const bf16x8 a = frag(As + (i * 16 + r) * kActRow + k0 + 32 * h + kq);
        acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0][h], a, acc[i][0], 0, 0, 0);
        if (on[1]) acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[1][h], a, acc[i][1], 0, 0, 0);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      b[0][h] = c[0][h];
      if (on[1]) b[1][h] = c[1][h];
    }
  }
}

__device__ __forceinline__ void load_rows(uint16_t* As, const uint16_t* x, int64_t row0, int rows, int width) {
  const int per = width / 8;
  for (int e = threadIdx.x; e < rows * per; e += blockDim.x) {
    const int row = e / per, c = (e - row * per) * 8;
    *reinterpret_cast<uint4*>(As + row * kActRow + c) =
        *reinterpret_cast<const uint4*>(x + (row0 + row) * width + c);
  }
}

// Inference: 16 MT rows through all layers.  262,144 rows of the 64-256-256-256-256-64
// network: 603 -> 397 us, 303 TFLOP/s on the padded widths.  A wave's weight loads,
// LDS fragments, products and GELU follow one another, and the other waves of its
// SIMD overlap them in part only.  GELU is the layered pass's, by erf: a polynomial
// with the hardware's reciprocal and exponential took 355 us (six waves a SIMD
// 422), but was three times as far from GELU for positive arguments, and the
// outputs are those of the layered pass to the last bit this way.
template <int MT>
__global__ __launch_bounds__(64 * kFusedWaves) void mlp_infer_kernel(FusedArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[16 * MT * kActRow];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t row0 = (int64_t)blockIdx.x * 16 * MT;
  load_rows(As, g.x, row0, 16 * MT, g.fin[0]);
  __syncthreads();
  for (int l = 0; l < g.nlin; ++l) {
    const int N = g.fout[l], n0 = w * 16;
    f32x4 acc[MT][2];
    tile_product<MT>(acc, As, g.pb + g.offw[l], g.fin[l], n0, N, lane);
    __syncthreads();  // every wave has read As
    const bool last = l == g.nlin - 1;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int col = n0 + 128 * j + (lane >> 4) * 4;  // and the next three
      if (n0 + 128 * j >= N) break;
      const float4 bias = *reinterpret_cast<const float4*>(g.p + g.offb[l] + col);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int row = i * 16 + (lane & 15);
        float v[4] = {acc[i][j][0] + bias.x, acc[i][j][1] + bias.y, acc[i][j][2] + bias.z, acc[i][j][3] + bias.w};
        if (last) {
#pragma unroll
          for (int q = 0; q < 4; ++q)
            if (col + q >= g.nout) v[q] = 0.0f;
          *reinterpret_cast<row4*>(g.out + (row0 + row) * N + col) = row4{v[0], v[1], v[2], v[3]};
        } else {
          ushort4 h;
          h.x = f2bf(gelu(v[0]));
          h.y = f2bf(gelu(v[1]));
          h.z = f2bf(gelu(v[2]));
          h.w = f2bf(gelu(v[3]));
          *reinterpret_cast<ushort4*>(As + row * kActRow + col) = h;
        }
      }
    }
    __syncthreads();
  }
}

// Training: forward, loss and the gradient of every layer's output for 16 MT
// rows, a wave per 16 columns.  A chain of 2 nlin - 1 products of a few hundred
// cycles each, so latency is what counts: a wave loads its whole share of the
// next product's weights (16 columns, at most 256 deep) before it finishes the
// present one, and GELU' is formed with GELU (one erf).  Leaves the layers'
// inputs and output gradients transposed in HBM (rows in the fast index, four a
// lane), which is what the weight gradients' products contract over.  4,096 rows:
// 48 us; a training step 323 -> 89 us (33 launches before), of it the weight
// gradients 22 and the sums with Adam 9 us.
template <int MT>
__global__ __launch_bounds__(64 * kTrainWaves) void mlp_train_kernel(FusedArgs g) {
  __shared__ __attribute__((aligned(16))) uint16_t As[16 * MT * kActRow];
  __shared__ float red[kTrainWaves];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t row0 = (int64_t)blockIdx.x * 16 * MT;
  const int n0 = w * 16, r = lane & 15, kq = (lane >> 4) * 8, rq = (lane >> 4) * 4;
  const int col = n0 + r;  // the lane's column; its rows are 16 i + rq .. + 3
  const int hidden = g.fout[0], nstep = 2 * g.nlin - 1;
  bf16x8 wf[kWide / 32];
  // forward steps 0 .. nlin - 1 (layer l = step), then backward steps for the
  // inputs of layers nlin - 1 .. 1
  auto load_weights = [&](int step) {
    const bool fwd = step < g.nlin;
    const int l = fwd ? step : nstep - step;
    const int K = fwd ? g.fin[l] : g.fout[l], N = fwd ? g.fout[l] : g.fin[l];
    if (n0 >= N) return;
    const uint16_t* q = (fwd ? g.pb : g.pt) + g.offw[l] + (int64_t)col * K + kq;
#pragma unroll
    for (int h = 0; h < kWide / 32; ++h)
      if (32 * h < K) wf[h] = frag(q + 32 * h);
  };
#pragma unroll
  for (int h = 0; h < kWide / 32; ++h) wf[h] = bf16x8{};
  load_weights(0);
  load_rows(As, g.x, row0, 16 * MT, g.fin[0]);
  __syncthreads();
  for (int e = threadIdx.x; e < 4 * MT * g.fin[0]; e += blockDim.x) {
    const int f = e / (4 * MT), q = (e - f * 4 * MT) * 4;
    const uint16_t* a = As + q * kActRow + f;
    *reinterpret_cast<ushort4*>(g.xt + (int64_t)f * g.B + row0 + q) =
        ushort4{a[0], a[kActRow], a[2 * kActRow], a[3 * kActRow]};
  }
  float lsum = 0.0f;
  for (int step = 0; step < nstep; ++step) {
    const bool fwd = step < g.nlin, last = step == g.nlin - 1;
    const int l = fwd ? step : nstep - step;
    const int K = fwd ? g.fin[l] : g.fout[l], N = fwd ? g.fout[l] : g.fin[l];
    const bool on = n0 < N;
    // what the epilogue needs from HBM
    float bias = 0.0f, ga[MT][4];
    if (on && fwd) bias = g.p[g.offb[l] + col];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int64_t row = row0 + i * 16 + rq + q;
        ga[i][q] = 0.0f;
        if (last && col < g.nout) ga[i][q] = g.tgt[row * g.nout + col];
        if (!fwd && on) ga[i][q] = g.dact[((int64_t)(l - 1) * g.B + row) * hidden + col];
      }
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (on) {
#pragma unroll
      for (int h = 0; h < kWide / 32; ++h)
        if (32 * h < K) {
#pragma unroll
          for (int i = 0; i < MT; ++i)
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag(As + (i * 16 + r) * kActRow + 32 * h + kq), wf[h],
                                                             acc[i], 0, 0, 0);
        }
    }
    if (step + 1 < nstep) load_weights(step + 1);
    __syncthreads();  // every wave has read As
    if (on) {
      const int ld = fwd ? l : l - 1;  // layer whose output gradient this is, after the forward steps
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        const int64_t row = row0 + i * 16 + rq;
        ushort4 h;
        uint16_t* hv = reinterpret_cast<uint16_t*>(&h);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v = acc[i][q] + bias;
          if (last) {  // gradient of the mean squared error
            const float d = col < g.nout ? v - ga[i][q] : 0.0f;
            lsum += d * d;
            v = g.scale * d;
          } else if (fwd) {
            float dv;
            v = gelu_both(v, dv);
            g.dact[((int64_t)l * g.B + row + q) * hidden + col] = dv;
          } else {
            v *= ga[i][q];
          }
          if (last || !fwd) g.dyf[(int64_t)g.offd[ld] * g.B + (row + q) * g.fout[ld] + col] = v;
          hv[q] = f2bf(v);
          As[(i * 16 + rq + q) * kActRow + col] = hv[q];
        }
        uint16_t* to = fwd && !last ? g.xt + (int64_t)(g.offx[l + 1] + col) * g.B
                                    : g.dt + (int64_t)(g.offd[ld] + col) * g.B;
        *reinterpret_cast<ushort4*>(to + row) = h;
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int d = 1; d < 64; d *= 2) lsum += __shfl_xor(lsum, d);
  if (lane == 0) red[w] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float s = 0.0f;
    for (int q = 0; q < kTrainWaves; ++q) s += red[q];
    g.lpart[blockIdx.x] = s;
  }
}

// Weight gradients of all layers, dW[o][i] = sum_b dt[o][b] xt[i][b], on 64 x 64
// tiles, K = the batch in ks[l] slices; both operands have the batch in the
// fast index, so the fragments come straight from L2.  The workgroups past the
// slices sum 64 columns of the output gradients over a chunk of rows each, for
// the biases.
__global__ __launch_bounds__(256) void wgrad_kernel(FusedArgs g, int64_t nparam, float* part, int slices) {
  int l = 0, t = blockIdx.x;
  if (t >= slices) {
    __shared__ float red[4][64];
    t -= slices;
    const int nb = g.offd[g.nlin - 1] + g.fout[g.nlin - 1], ch = t / (nb / 64), c0 = (t % (nb / 64)) * 64;
    while (c0 >= g.offd[l] + g.fout[l]) ++l;
    const int c = threadIdx.x & 63, rg = threadIdx.x >> 6;
    const float* y = g.dyf + (int64_t)g.offd[l] * g.B + c0 - g.offd[l] + c;
    const int64_t r1 = (int64_t)(ch + 1) * g.rpc < g.B ? (int64_t)(ch + 1) * g.rpc : g.B;
    float s = 0.0f;
#pragma unroll 8
    for (int64_t r = (int64_t)ch * g.rpc + rg; r < r1; r += 4) s += y[r * g.fout[l]];
    red[rg][c] = s;
    __syncthreads();
    if (rg == 0) g.bpart[(int64_t)ch * nb + c0 + c] = (red[0][c] + red[1][c]) + (red[2][c] + red[3][c]);
    return;
  }
  for (;; ++l) {
    const int n = (g.fout[l] / 64) * (g.fin[l] / 64) * g.ks[l];
    if (t < n) break;
    t -= n;
  }
  const int tn = g.fin[l] / 64, nt = (g.fout[l] / 64) * tn, z = t / nt;
  t -= z * nt;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = lane & 15, kq = (lane >> 4) * 8;
  const int m0 = (t / tn) * 64 + (w >> 1) * 32, n0 = (t % tn) * 64 + (w & 1) * 32;
  const int64_t kc = g.B / g.ks[l];  // a multiple of 32
  const uint16_t* a = g.dt + (int64_t)(g.offd[l] + m0 + r) * g.B + kc * z + kq;
  const uint16_t* b = g.xt + (int64_t)(g.offx[l] + n0 + r) * g.B + kc * z + kq;
  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i) acc[i][0] = acc[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k0 = 0; k0 < (int)kc; k0 += 32) {
    bf16x8 fa[2], fb[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      fa[i] = frag(a + i * 16 * g.B + k0);
      fb[i] = frag(b + i * 16 * g.B + k0);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
  }
  float* to = part + nparam * z + g.offw[l];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        to[(int64_t)(m0 + i * 16 + (lane >> 4) * 4 + q) * g.fin[l] + n0 + j * 16 + r] = acc[i][j][q];
}

struct AdamArgs {
  float *p, *g, *m, *v;
  uint16_t *pb, *pt;
  float lr_t, b1, b2, eps_t;
  int update;  // 0: gradients into g only; 1: Adam (g not written); 2: bf16 copies only
};

// The gradient sums and Adam (bias correction folded into lr_t and eps_t) on
// 32 x 32 tiles of the weights, which leave through LDS transposed too; the
// last workgroups take 256 biases each, the very last the loss.
__global__ __launch_bounds__(256) void finish_kernel(FusedArgs f, AdamArgs o, const float* part, int64_t nparam,
                                                     int nwg, float inv_count, float* loss, int ntile) {
  __shared__ uint16_t tile[32][34];
  __shared__ float red[256];
  int t = blockIdx.x;
  if (t < ntile) {
    int l = 0;
    for (;; ++l) {
      const int n = (f.fout[l] / 32) * (f.fin[l] / 32);
      if (t < n) break;
      t -= n;
    }
    const int tn = f.fin[l] / 32, o0 = (t / tn) * 32, i0 = (t % tn) * 32;
    const int c = threadIdx.x & 31, r = threadIdx.x >> 5;
    float gr[4] = {0.f, 0.f, 0.f, 0.f};
    int64_t at[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) at[e] = f.offw[l] + (int64_t)(o0 + r + 8 * e) * f.fin[l] + i0 + c;
    if (o.update < 2) {
#pragma unroll 8
      for (int z = 0; z < f.ks[l]; ++z)
#pragma unroll
        for (int e = 0; e < 4; ++e) gr[e] += part[(int64_t)z * nparam + at[e]];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (o.update == 0) {
        o.g[at[e]] = gr[e];
        continue;
      }
      float pi = o.p[at[e]];
      if (o.update == 1) {
        const float mi = o.b1 * o.m[at[e]] + (1.0f - o.b1) * gr[e];
        const float vi = o.b2 * o.v[at[e]] + (1.0f - o.b2) * gr[e] * gr[e];
        o.m[at[e]] = mi;
        o.v[at[e]] = vi;
        pi = pi - o.lr_t * mi / (sqrtf(vi) + o.eps_t);
        o.p[at[e]] = pi;
      }
      const uint16_t h = f2bf(pi);
      o.pb[at[e]] = h;
      tile[r + 8 * e][c] = h;
    }
    if (o.update == 0) return;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o.pt[f.offw[l] + (int64_t)(i0 + r + 8 * e) * f.fout[l] + o0 + c] = tile[c][r + 8 * e];
    return;
  }
  t -= ntile;
  const int nb = f.offd[f.nlin - 1] + f.fout[f.nlin - 1];
  if (t * 256 < nb) {
    const int col = t * 256 + threadIdx.x;
    if (col >= nb) return;
    float s = 0.0f;
    if (o.update < 2) {
#pragma unroll 8
      for (int z = 0; z < f.nch; ++z) s += f.bpart[(int64_t)z * nb + col];
    }
    int l = 0;
    while (col >= f.offd[l] + f.fout[l]) ++l;
    const int64_t at = f.offb[l] + col - f.offd[l];
    if (o.update == 0) {
      o.g[at] = s;
      return;
    }
    float pi = o.p[at];
    if (o.update == 1) {
      const float mi = o.b1 * o.m[at] + (1.0f - o.b1) * s;
      const float vi = o.b2 * o.v[at] + (1.0f - o.b2) * s * s;
      o.m[at] = mi;
      o.v[at] = vi;
      pi = pi - o.lr_t * mi / (sqrtf(vi) + o.eps_t);
      o.p[at] = pi;
    }
    o.pb[at] = f2bf(pi);
    return;
  }
  float s = 0.0f;  // the loss
  for (int z = threadIdx.x; z < nwg; z += 256) s += f.lpart[z];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = red[0] * inv_count;
}

int round_up(int x, int m) { return (x + m - 1) / m * m; }

}  // namespace

struct tgr_mlp {
  int nin = 0, nout = 0, hidden = 0, nhl = 0, nlin = 0;
  std::vector<int> fin, fout;        // padded fan-in / fan-out per linear layer
  std::vector<int64_t> offw, offb;   // offsets in the flat parameter vector
  int64_t nparam = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;
  uint16_t* pb = nullptr;
  uint16_t* pt = nullptr;  // fused passes: the weights of pb transposed, same offsets
  bool fused = false;      // all widths at most kWide
  int n_cu = 1;
  int64_t step = 0;
  // fused training workspace for wcap rows, and the fewest rows that there was no
  // memory for
  int64_t wcap = 0, refused = INT64_MAX;
  float *wdact = nullptr, *wdyf = nullptr, *wpart = nullptr, *wbias = nullptr;
  uint16_t *wxt = nullptr, *wdt = nullptr;
  // batch workspace
  int64_t cap = 0;
  std::vector<float*> pre;      // [nlin-1] hidden pre-activations, fp32 [cap][hidden]
  std::vector<uint16_t*> act;   // [nlin] act[0] unused (input), act[l] bf16 [cap][fin[l]]
  float* out = nullptr;         // [cap][fout.back()]
  float* dyf[2] = {nullptr, nullptr};
  uint16_t* dyh[2] = {nullptr, nullptr};
  float* part = nullptr;
  float* loss = nullptr;
  float* kpart = nullptr;  // split-K / column-sum partials
  int64_t kpart_n = 0;
  static constexpr int kLossBlocks = 256;
  static constexpr int kMaxSplit = 32;

  int sum_fin() const { int n = 0; for (int v : fin) n += v; return n; }
  int sum_fout() const { int n = 0; for (int v : fout) n += v; return n; }

  void free_fused() {
    for (void* q : {(void*)wdact, (void*)wdyf, (void*)wpart, (void*)wbias, (void*)wxt, (void*)wdt})
      if (q) (void)hipFree(q);
    wdact = wdyf = wpart = wbias = nullptr;
    wxt = wdt = nullptr;
    wcap = 0;
  }

  int ensure_fused(int64_t rows) {
    if (!loss) HIP_TRY(hipMalloc(&loss, sizeof(float)));
    if (rows <= wcap) return 0;
    free_fused();
    HIP_TRY(hipMalloc(&wdact, sizeof(float) * rows * hidden * (nlin - 1)));
    HIP_TRY(hipMalloc(&wdyf, sizeof(float) * rows * sum_fout()));
    HIP_TRY(hipMalloc(&wxt, sizeof(uint16_t) * rows * sum_fin()));
    HIP_TRY(hipMalloc(&wdt, sizeof(uint16_t) * rows * sum_fout()));
    HIP_TRY(hipMalloc(&wpart, sizeof(float) * kMaxSplit * nparam));
    // column sums of kMaxSplit row chunks, then the squared errors of every workgroup
    HIP_TRY(hipMalloc(&wbias, sizeof(float) * (kMaxSplit * sum_fout() + rows / 16)));
    wcap = rows;
    return 0;
  }

  void free_ws() {
    for (float* q : pre) (void)hipFree(q);
    for (size_t l = 1; l < act.size(); ++l) (void)hipFree(act[l]);
    pre.clear();
    act.clear();
    for (void* q : {(void*)out, (void*)dyf[0], (void*)dyf[1], (void*)dyh[0], (void*)dyh[1], (void*)part,
                    (void*)kpart})
      if (q) (void)hipFree(q);
    kpart = nullptr;
    kpart_n = 0;
    out = nullptr;
    dyf[0] = dyf[1] = nullptr;
    dyh[0] = dyh[1] = nullptr;
    part = nullptr;
    cap = 0;
  }

  int ensure(int64_t rows) {
    if (rows <= cap) return 0;
    free_ws();
    const int wmax = std::max(hidden, std::max(fin[0], fout.back()));
    pre.assign(nlin - 1, nullptr);
    act.assign(nlin, nullptr);
    for (int l = 0; l < nlin - 1; ++l) HIP_TRY(hipMalloc(&pre[l], sizeof(float) * rows * hidden));
    for (int l = 1; l < nlin; ++l) HIP_TRY(hipMalloc(&act[l], sizeof(uint16_t) * rows * fin[l]));
    HIP_TRY(hipMalloc(&out, sizeof(float) * rows * fout.back()));
    for (int i = 0; i < 2; ++i) {
      HIP_TRY(hipMalloc(&dyf[i], sizeof(float) * rows * wmax));
      HIP_TRY(hipMalloc(&dyh[i], sizeof(uint16_t) * rows * wmax));
    }
    HIP_TRY(hipMalloc(&part, sizeof(float) * kLossBlocks));
    if (!loss) HIP_TRY(hipMalloc(&loss, sizeof(float)));
    // partials of the weight-gradient products (at most kMaxSplit slices of
    // the largest weight matrix) followed by those of the bias column sums
    // (at most kMaxSplit rows of the widest layer)
    kpart_n = (int64_t)kMaxSplit * ((int64_t)wmax * wmax + wmax);
    HIP_TRY(hipMalloc(&kpart, sizeof(float) * kpart_n));
    cap = rows;
    return 0;
  }
};

namespace {

int launch_gemm(const GemmArgs& a, hipStream_t s) {
  if (a.M % kTile || a.N % kTile || a.K % kKStep || a.M <= 0 || a.N <= 0 || a.K <= 0)
    return fail(TGR_MLP_E_ARG, "gemm: M, N must be positive multiples of 64 and K of 32");
  const bool ak = a.sak == 1, bk = a.sbk == 1;
  if (!ak && a.sam != 1) return fail(TGR_MLP_E_ARG, "gemm: A needs a unit stride in m or k");
  if (!bk && a.sbn != 1) return fail(TGR_MLP_E_ARG, "gemm: B needs a unit stride in k or n");
  // 16-byte loads: the other stride and the base must keep 8-element alignment
  if ((ak ? a.sam : a.sak) % 8 || (bk ? a.sbn : a.sbk) % 8 || ((uintptr_t)a.A & 15) || ((uintptr_t)a.B & 15))
    return fail(TGR_MLP_E_ARG, "gemm: operands must be 16-byte aligned with strides that are multiples of 8");
  const int ks = a.ksplit > 1 ? a.ksplit : 1;
  if (a.K % (ks * kKStep)) return fail(TGR_MLP_E_ARG, "gemm: K must split into multiples of 32");
  dim3 grid(a.N / kTile, a.M / kTile, ks), block(256);
  if (ak && bk) gemm_bf16_kernel<true, true><<<grid, block, 0, s>>>(a);
  else if (ak) gemm_bf16_kernel<true, false><<<grid, block, 0, s>>>(a);
  else if (bk) gemm_bf16_kernel<false, true><<<grid, block, 0, s>>>(a);
  else gemm_bf16_kernel<false, false><<<grid, block, 0, s>>>(a);
  HIP_TRY(hipGetLastError());
  return 0;
}

GemmArgs plain_args() {
  GemmArgs a;
  memset(&a, 0, sizeof(a));
  a.act = kNone;
  a.ksplit = 1;
  return a;
}

// Slices of the batch (K) of a weight-gradient product of n 64 x 64 tiles: the
// weight matrices alone give only n workgroups
int batch_slices(int64_t n, int64_t B) {
  int ks = 1;
  while (ks < tgr_mlp::kMaxSplit && n * ks < 512 && B % (2 * ks * kKStep) == 0 && B / (2 * ks) >= 128) ks *= 2;
  return ks;
}

// Row chunks of a bias gradient (column sums of the output gradients)
int bias_chunks(int64_t B) { return (int)std::min<int64_t>(tgr_mlp::kMaxSplit, (B + 255) / 256); }

FusedArgs fused_args(const tgr_mlp* h, const uint16_t* x, int64_t B) {
  FusedArgs a;
  memset(&a, 0, sizeof(a));
  a.x = x;
  a.B = B;
  a.nlin = h->nlin;
  a.nout = h->nout;
  for (int l = 0; l < h->nlin; ++l) {
    a.fin[l] = h->fin[l];
    a.fout[l] = h->fout[l];
    a.offw[l] = h->offw[l];
    a.offb[l] = h->offb[l];
    a.offx[l] = l ? a.offx[l - 1] + h->fin[l - 1] : 0;
    a.offd[l] = l ? a.offd[l - 1] + h->fout[l - 1] : 0;
  }
  a.p = h->p;
  a.pb = h->pb;
  a.pt = h->pt;
  return a;
}

// Rows of a workgroup of the fused passes, as 16-row tiles: the weights are
// read from L2 once per workgroup, so as many as leave every CU a workgroup.
int row_tiles(const tgr_mlp* h, int64_t B) {
  int mt = 4;
  while (mt > 1 && B / (16 * mt) < h->n_cu) mt /= 2;
  return mt;
}

int forward_fused(tgr_mlp* h, const uint16_t* x, int64_t B, float* out, hipStream_t s) {
  FusedArgs a = fused_args(h, x, B);
  a.out = out;
  const int mt = row_tiles(h, B);
  const dim3 grid((unsigned)(B / (16 * mt))), block(64 * kFusedWaves);
  if (mt == 4) mlp_infer_kernel<4><<<grid, block, 0, s>>>(a);
  else if (mt == 2) mlp_infer_kernel<2><<<grid, block, 0, s>>>(a);
  else mlp_infer_kernel<1><<<grid, block, 0, s>>>(a);
  HIP_TRY(hipGetLastError());
  return 0;
}

// Whether a batch is trained by the fused pass.  Its workspace takes a third more
// memory than the layered pass's (12.8 and 9.5 KB a row of the 64-256-256-256-256-64
// network); where it is not to be had, the layered pass gives the same parameters.
bool trains_fused(tgr_mlp* h, int64_t B) {
  if (!h->fused || B >= h->refused) return false;
  if (!h->ensure_fused(B)) return true;
  (void)hipGetLastError();
  g_err.clear();
  h->free_fused();
  h->refused = B;
  return false;
}

// One pass over the batch: loss and gradients, then o (Adam, or gradients into h->g)
int train_fused(tgr_mlp* h, const uint16_t* x, const float* tgt, int64_t B, const AdamArgs& o, hipStream_t s) {
  FusedArgs a = fused_args(h, x, B);
  a.tgt = tgt;
  a.scale = 2.0f / ((float)B * (float)h->nout);
  a.dact = h->wdact;
  a.dyf = h->wdyf;
  a.xt = h->wxt;
  a.dt = h->wdt;
  const int mt = row_tiles(h, B);
  const int nwg = (int)(B / (16 * mt)), nb = h->sum_fout();
  a.bpart = h->wbias;
  a.lpart = h->wbias + tgr_mlp::kMaxSplit * nb;
  a.nch = bias_chunks(B);
  a.rpc = (int)((B + a.nch - 1) / a.nch);
  const dim3 grid((unsigned)nwg), block(64 * kTrainWaves);
  if (mt == 4) mlp_train_kernel<4><<<grid, block, 0, s>>>(a);
  else if (mt == 2) mlp_train_kernel<2><<<grid, block, 0, s>>>(a);
  else mlp_train_kernel<1><<<grid, block, 0, s>>>(a);
  // slices of the batch until a layer has 512 workgroups, as in loss_and_grad
  int tiles = 0, slices = 0;
  for (int l = 0; l < h->nlin; ++l) {
    const int n = (h->fout[l] / 64) * (h->fin[l] / 64);
    a.ks[l] = batch_slices(n, B);
    tiles += n;
    slices += n * a.ks[l];
  }
  hipLaunchKernelGGL(wgrad_kernel, dim3(slices + nb / 64 * a.nch), dim3(256), 0, s, a, h->nparam, h->wpart, slices);
  hipLaunchKernelGGL(finish_kernel, dim3(tiles * 4 + (nb + 255) / 256 + 1), dim3(256), 0, s, a, o, h->wpart, h->nparam, nwg,
                     1.0f / ((float)B * (float)h->nout), h->loss, tiles * 4);
  HIP_TRY(hipGetLastError());
  return 0;
}

AdamArgs adam_args(const tgr_mlp* h, int update) {
  AdamArgs o;
  memset(&o, 0, sizeof(o));
  o.p = h->p;
  o.g = h->g;
  o.m = h->m;
  o.v = h->v;
  o.pb = h->pb;
  o.pt = h->pt;
  o.update = update;
  return o;
}

// both bf16 copies of the weights of a network of the fused passes
int refresh_copies(tgr_mlp* h, hipStream_t s) {
  int tiles = 0;
  for (int l = 0; l < h->nlin; ++l) tiles += (h->fout[l] / 32) * (h->fin[l] / 32);
  hipLaunchKernelGGL(finish_kernel, dim3(tiles + (h->sum_fout() + 255) / 256), dim3(256), 0, s, fused_args(h, nullptr, 0),
                     adam_args(h, 2), (const float*)nullptr, h->nparam, 0, 0.0f, (float*)nullptr, tiles);
  HIP_TRY(hipGetLastError());
  return 0;
}

// forward over B rows of x (bf16 [B][fin[0]]); keep_pre: store the hidden
// pre-activations that the backward needs
int forward(tgr_mlp* h, const uint16_t* x, int64_t B, float* out, int64_t ldo, bool keep_pre, hipStream_t s) {
  const uint16_t* in = x;
  for (int l = 0; l < h->nlin; ++l) {
    GemmArgs a = plain_args();
    a.A = in;
    a.sam = h->fin[l];
    a.sak = 1;
    a.B = h->pb + h->offw[l];  // W[out][in]: B(k=in, n=out) = W[n*fin + k]
    a.sbk = 1;
    a.sbn = h->fin[l];
    a.M = (int)B;
    a.N = h->fout[l];
    a.K = h->fin[l];
    a.bias = h->p + h->offb[l];
    a.n_valid = h->fout[l];
    if (l < h->nlin - 1) {
      a.act = kGelu;
      a.pre = keep_pre ? h->pre[l] : nullptr;
      a.ldpre = h->hidden;
      a.out_h = h->act[l + 1];
      a.ldh = h->fin[l + 1];
    } else {
      a.out_f = out;
      a.ldf = ldo;
      a.n_valid = h->nout;
    }
    int rc = launch_gemm(a, s);
    if (rc) return rc;
    in = h->act[l + 1];
  }
  return 0;
}

// loss and gradient into h->g for targets tgt[B][nout]
int loss_and_grad(tgr_mlp* h, const uint16_t* x, const float* tgt, int64_t B, hipStream_t s) {
  int rc = h->ensure(B);
  if (rc) return rc;
  const int ldo = h->fout.back();
  if ((rc = forward(h, x, B, h->out, ldo, true, s))) return rc;
  hipLaunchKernelGGL(mse_grad_kernel, dim3(tgr_mlp::kLossBlocks), dim3(256), 0, s, h->out, (int64_t)ldo, tgt,
                     h->nout, B, h->dyf[0], h->dyh[0], h->part);
  hipLaunchKernelGGL(finish_loss_kernel, dim3(1), dim3(256), 0, s, h->part, tgr_mlp::kLossBlocks,
                     1.0f / ((float)B * (float)h->nout), h->loss);
  HIP_TRY(hipGetLastError());
  int cur = 0;
  for (int l = h->nlin - 1; l >= 0; --l) {
    const int no = h->fout[l], ni = h->fin[l];
    const uint16_t* xin = l == 0 ? x : h->act[l];
    // dW[o][i] = sum_b dY[b][o] x[b][i]
    GemmArgs a = plain_args();
    a.A = h->dyh[cur];
    a.sam = 1;
    a.sak = no;
    a.B = xin;
    a.sbk = ni;
    a.sbn = 1;
    a.M = no;
    a.N = ni;
    a.K = (int)B;
    a.ldf = ni;
    a.n_valid = ni;
    const int ks = batch_slices((int64_t)(no / 64) * (ni / 64), B);
    a.ksplit = ks;
    a.out_f = ks > 1 ? h->kpart : h->g + h->offw[l];
    if ((rc = launch_gemm(a, s))) return rc;
    if (ks > 1)
      hipLaunchKernelGGL(sum_parts_kernel, dim3(256), dim3(256), 0, s, h->kpart, ks, (int64_t)no * ni,
                         h->g + h->offw[l]);
    // bias gradient: column sums of dY in row chunks, then the chunk sums
    const int64_t nch = bias_chunks(B);
    const int64_t rpc = (B + nch - 1) / nch;
    hipLaunchKernelGGL(colsum_kernel, dim3(no / 64, (unsigned)nch), dim3(256), 0, s, h->dyf[cur], (int64_t)no, B,
                       rpc, h->kpart + (int64_t)tgr_mlp::kMaxSplit * no * ni, no);
    hipLaunchKernelGGL(sum_parts_kernel, dim3(1), dim3(256), 0, s, h->kpart + (int64_t)tgr_mlp::kMaxSplit * no * ni,
                       (int)nch, (int64_t)no, h->g + h->offb[l]);
    HIP_TRY(hipGetLastError());
    if (l == 0) break;
    // dY_prev = (dY W) * gelu'(pre_prev)
    GemmArgs d = plain_args();
    d.A = h->dyh[cur];
    d.sam = no;
    d.sak = 1;
    d.B = h->pb + h->offw[l];  // B(k=o, n=i) = W[k*ni + n]
    d.sbk = ni;
    d.sbn = 1;
    d.M = (int)B;
    d.N = ni;
    d.K = no;
    d.act = kGeluGrad;
    d.aux = h->pre[l - 1];
    d.ldaux = h->hidden;
    d.out_f = h->dyf[cur ^ 1];
    d.ldf = ni;
    d.out_h = h->dyh[cur ^ 1];
    d.ldh = ni;
    d.n_valid = ni;
    if ((rc = launch_gemm(d, s))) return rc;
    cur ^= 1;
  }
  return 0;
}

// the fused passes load x in 16-byte pieces, as the product kernel does (which
// checks its operands itself)
int check_input(const uint16_t* x) {
  return (uintptr_t)x & 15 ? fail(TGR_MLP_E_ARG, "the input rows must be 16-byte aligned") : 0;
}

constexpr int64_t kInferChunk = 262144;  // rows per inference pass (a multiple of 64)

int check_batch(const tgr_mlp* h, int64_t B) {
  if (!h) return fail(TGR_MLP_E_ARG, "null network");
  if (B <= 0 || B % 64) return fail(TGR_MLP_E_ARG, "batch rows must be a positive multiple of 64");
  if (B > (int64_t)1 << 26) return fail(TGR_MLP_E_ARG, "batch too large");
  return 0;
}

}  // namespace

extern "C" {

int tgr_mlp_create(int nin, int nout, int hidden, int n_hidden_layers, tgr_mlp** out) {
  if (!out) return fail(TGR_MLP_E_ARG, "null output pointer");
  *out = nullptr;
  if (nin < 1 || nout < 1 || hidden < 64 || hidden % 64 || n_hidden_layers < 1 || n_hidden_layers > 16 ||
      nin > 4096 || nout > 4096 || hidden > 4096)
    return fail(TGR_MLP_E_ARG, "bad network shape (hidden must be a multiple of 64)");
  tgr_mlp* h = new tgr_mlp();
  h->nin = nin;
  h->nout = nout;
  h->hidden = hidden;
  h->nhl = n_hidden_layers;
  h->nlin = n_hidden_layers + 1;
  for (int l = 0; l < h->nlin; ++l) {
    h->fin.push_back(l == 0 ? round_up(nin, 64) : hidden);
    h->fout.push_back(l == h->nlin - 1 ? round_up(nout, 64) : hidden);
    h->offw.push_back(h->nparam);
    h->nparam += (int64_t)h->fin[l] * h->fout[l];
    h->offb.push_back(h->nparam);
    h->nparam += h->fout[l];
  }
  h->fused = hidden <= kWide && h->fin[0] <= kWide && h->fout.back() <= kWide;
  int dev = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) != hipSuccess || hipGetDeviceProperties(&prop, dev) != hipSuccess) {
    delete h;
    return fail(TGR_MLP_E_HIP, "device query failed");
  }
  h->n_cu = prop.multiProcessorCount;
  const size_t n = h->nparam;
  if (hipMalloc(&h->p, n * 4) != hipSuccess || hipMalloc(&h->g, n * 4) != hipSuccess ||
      hipMalloc(&h->m, n * 4) != hipSuccess || hipMalloc(&h->v, n * 4) != hipSuccess ||
      hipMalloc(&h->pb, n * 2) != hipSuccess || hipMalloc(&h->pt, n * 2) != hipSuccess) {
    tgr_mlp_destroy(h);
    return fail(TGR_MLP_E_NOMEM, "hipMalloc failed");
  }
  if (hipMemset(h->p, 0, n * 4) != hipSuccess || hipMemset(h->g, 0, n * 4) != hipSuccess ||
      hipMemset(h->m, 0, n * 4) != hipSuccess || hipMemset(h->v, 0, n * 4) != hipSuccess ||
      hipMemset(h->pb, 0, n * 2) != hipSuccess || hipMemset(h->pt, 0, n * 2) != hipSuccess) {
    tgr_mlp_destroy(h);
    return fail(TGR_MLP_E_HIP, "hipMemset failed");
  }
  *out = h;
  return 0;
}

int tgr_mlp_destroy(tgr_mlp* h) {
  if (!h) return 0;
  h->free_ws();
  h->free_fused();
  for (void* q : {(void*)h->p, (void*)h->g, (void*)h->m, (void*)h->v, (void*)h->pb, (void*)h->pt, (void*)h->loss})
    if (q) (void)hipFree(q);
  delete h;
  return 0;
}

int tgr_mlp_layout(const tgr_mlp* h, int64_t* nparam, int* in_pad, int* out_pad) {
  if (!h) return fail(TGR_MLP_E_ARG, "null network");
  if (nparam) *nparam = h->nparam;
  if (in_pad) *in_pad = h->fin[0];
  if (out_pad) *out_pad = h->fout.back();
  return 0;
}

int tgr_mlp_shape(const tgr_mlp* h, int* nin, int* nout, int* hidden, int* n_hidden_layers) {
  if (!h) return fail(TGR_MLP_E_ARG, "null network");
  if (nin) *nin = h->nin;
  if (nout) *nout = h->nout;
  if (hidden) *hidden = h->hidden;
  if (n_hidden_layers) *n_hidden_layers = h->nhl;
  return 0;
}

int tgr_mlp_set_params(tgr_mlp* h, const float* host) {
  if (!h || !host) return fail(TGR_MLP_E_ARG, "null argument");
  // padded entries must be zero for the padded network to equal the unpadded one
  for (int l = 0; l < h->nlin; ++l) {
    const int ni = l == 0 ? h->nin : h->fin[l], no = l == h->nlin - 1 ? h->nout : h->fout[l];
    for (int o = 0; o < h->fout[l]; ++o) {
      for (int i = 0; i < h->fin[l]; ++i)
        if ((o >= no || i >= ni) && host[h->offw[l] + (int64_t)o * h->fin[l] + i] != 0.0f)
          return fail(TGR_MLP_E_ARG, "nonzero weight in the padding of layer " + std::to_string(l));
      if (o >= no && host[h->offb[l] + o] != 0.0f)
        return fail(TGR_MLP_E_ARG, "nonzero bias in the padding of layer " + std::to_string(l));
    }
  }
  HIP_TRY(hipMemcpy(h->p, host, h->nparam * 4, hipMemcpyHostToDevice));
  if (h->fused) {
    const int rc = refresh_copies(h, 0);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL(to_bf16_kernel, dim3(256), dim3(256), 0, 0, h->p, h->pb, h->nparam);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemset(h->m, 0, h->nparam * 4));
  HIP_TRY(hipMemset(h->v, 0, h->nparam * 4));
  h->refused = INT64_MAX;
  HIP_TRY(hipDeviceSynchronize());
  h->step = 0;
  return 0;
}

int tgr_mlp_get_params(const tgr_mlp* h, float* host) {
  if (!h || !host) return fail(TGR_MLP_E_ARG, "null argument");
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(host, h->p, h->nparam * 4, hipMemcpyDeviceToHost));
  return 0;
}

int tgr_mlp_forward(tgr_mlp* h, const uint16_t* x, int64_t B, float* out, void* stream) {
  int rc = check_batch(h, B);
  if (rc) return rc;
  if (!x || !out) return fail(TGR_MLP_E_ARG, "null argument");
  if ((rc = check_input(x))) return rc;
  if (h->fused) return forward_fused(h, x, B, out, (hipStream_t)stream);
  // inference in row chunks: the workspace stays at most kInferChunk rows
  const int64_t chunk = std::min<int64_t>(B, kInferChunk);
  if ((rc = h->ensure(chunk))) return rc;
  const int ldo = h->fout.back();
  for (int64_t r0 = 0; r0 < B; r0 += chunk) {
    const int64_t rows = std::min<int64_t>(chunk, B - r0);
    if ((rc = forward(h, x + r0 * h->fin[0], rows, out + r0 * ldo, ldo, false, (hipStream_t)stream))) return rc;
  }
  return 0;
}

int tgr_mlp_gradients(tgr_mlp* h, const uint16_t* x, const float* tgt, int64_t B, float* grad_host,
                      float* loss_host, void* stream) {
  int rc = check_batch(h, B);
  if (rc) return rc;
  if (!x || !tgt) return fail(TGR_MLP_E_ARG, "null argument");
  if ((rc = check_input(x))) return rc;
  hipStream_t s = (hipStream_t)stream;
  if ((rc = trains_fused(h, B) ? train_fused(h, x, tgt, B, adam_args(h, 0), s) : loss_and_grad(h, x, tgt, B, s)))
    return rc;
  HIP_TRY(hipStreamSynchronize(s));
  if (grad_host) HIP_TRY(hipMemcpy(grad_host, h->g, h->nparam * 4, hipMemcpyDeviceToHost));
  if (loss_host) HIP_TRY(hipMemcpy(loss_host, h->loss, 4, hipMemcpyDeviceToHost));
  return 0;
}

int tgr_mlp_train_step(tgr_mlp* h, const uint16_t* x, const float* tgt, int64_t B, float lr, float beta1,
                       float beta2, float eps, float* loss_host, void* stream) {
  int rc = check_batch(h, B);
  if (rc) return rc;
  if (!x || !tgt) return fail(TGR_MLP_E_ARG, "null argument");
  if ((rc = check_input(x))) return rc;
  if (!(lr > 0.0f) || !(beta1 >= 0.0f && beta1 < 1.0f) || !(beta2 >= 0.0f && beta2 < 1.0f) || !(eps > 0.0f))
    return fail(TGR_MLP_E_ARG, "bad optimiser settings");
  hipStream_t s = (hipStream_t)stream;
  const bool fused = trains_fused(h, B);
  if (!fused && (rc = loss_and_grad(h, x, tgt, B, s))) return rc;
  h->step += 1;
  const double c1 = 1.0 - std::pow((double)beta1, (double)h->step);
  const double c2 = 1.0 - std::pow((double)beta2, (double)h->step);
  const float lr_t = (float)(lr * std::sqrt(c2) / c1);
  const float eps_t = (float)(eps * std::sqrt(c2));
  if (fused) {
    AdamArgs o = adam_args(h, 1);
    o.lr_t = lr_t;
    o.b1 = beta1;
    o.b2 = beta2;
    o.eps_t = eps_t;
    if ((rc = train_fused(h, x, tgt, B, o, s))) {
      h->step -= 1;
      return rc;
    }
  } else {
    hipLaunchKernelGGL(adam_kernel, dim3(512), dim3(256), 0, s, h->p, h->g, h->m, h->v, h->pb, h->nparam, lr_t, beta1,
                       beta2, eps_t);
    HIP_TRY(hipGetLastError());
    if (h->fused && (rc = refresh_copies(h, s))) return rc;
  }
  if (loss_host) {
    HIP_TRY(hipStreamSynchronize(s));
    HIP_TRY(hipMemcpy(loss_host, h->loss, 4, hipMemcpyDeviceToHost));
  }
  return 0;
}

int tgr_mlp_gemm_bf16(const uint16_t* A, int64_t sam, int64_t sak, const uint16_t* B, int64_t sbk, int64_t sbn,
                      int M, int N, int K, float* C, int64_t ldc, void* stream) {
  if (!A || !B || !C) return fail(TGR_MLP_E_ARG, "null argument");
  GemmArgs a = plain_args();
  a.A = A;
  a.sam = sam;
  a.sak = sak;
  a.B = B;
  a.sbk = sbk;
  a.sbn = sbn;
  a.M = M;
  a.N = N;
  a.K = K;
  a.out_f = C;
  a.ldf = ldc;
  a.n_valid = N;
  return launch_gemm(a, (hipStream_t)stream);
}

const char* tgr_mlp_last_error(void) { return g_err.c_str(); }

}  // extern "C"
