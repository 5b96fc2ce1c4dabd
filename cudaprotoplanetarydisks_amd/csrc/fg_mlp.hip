// MLP emulator: BF16 weights and activations, FP32 accumulation, on the
// gfx950 matrix cores (v_mfma_f32_16x16x32_bf16), with training (MSE loss,
// backpropagation, Adam) and inference.  It maps disk parameters to
// ring-averaged profiles (cudaprotoplanetarydisks_amd/emulator.py); no
// reference counterpart.
//
// Every dense layer is one GEMM C = A B (M x K times K x N) with a fused
// epilogue:
//   forward hidden   Z = H W^T + b,  H' = bf16(GELU(Z))
//   (kept in FP32 for the way back: GELU'(Z) by k_mlp_rows, Z by k_gemm_bf16)
//   forward output   Y = H W^T + b                          (FP32)
//   backward         dZ_below = (dZ W) * GELU'(Z_below)     (FP32 + BF16)
//   weight gradient  dW = dZ^T H                            (FP32)
// Master weights, gradients and Adam moments are FP32; the BF16 weight
// copies the GEMMs read are refreshed by the optimizer step.
//
// Networks whose widths fit in LDS (mlp_fits_rows) run two kernels per
// training step: k_mlp_rows takes 4 to 16 batch rows a workgroup through every
// layer forward and back, k_mlp_weights forms every weight gradient and
// applies Adam to it where it stands.  Wider networks, and fg_bf16_gemm,
// run k_gemm_bf16 layer by layer: operands addressed by (row stride, column
// stride), a 256-thread workgroup per 64 x 64 tile as four waves of 2 x 2
// MFMA blocks, 64 x 32 slices of A and B^T staged in LDS.  Both accumulate
// every output over k in the same 32-wide MFMA steps, so their products are the
// same bits.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "fg_internal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short bf16_t;

#define GT 64  // output tile (rows and columns)
#define GK 32  // k per MFMA step
#define GKP (GK + 8)  // LDS row length (16-byte aligned rows, fewer bank conflicts)
#define MLP_MAX_LAYERS 8

__device__ __forceinline__ bf16_t f2bf(float f) {  // round to nearest even
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (bf16_t)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float((unsigned)h << 16); }

// GELU(x) = x Phi(x) and its derivative Phi(x) + x phi(x)
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float x) {
  return 0.5f * (1.0f + erff(x * 0.70710678118654752f)) + x * 0.39894228040143268f * expf(-0.5f * x * x);
}

// both at once, each from the same operations
__device__ __forceinline__ float gelu_both(float x, float &d) {
  const float e = 1.0f + erff(x * 0.70710678118654752f);
  d = 0.5f * e + x * 0.39894228040143268f * expf(-0.5f * x * x);
  return 0.5f * x * e;
}

enum { EPI_STORE = 0, EPI_GELU = 1, EPI_GELU_BACK = 2 };

struct gemm_args {
  const bf16_t *A;
  long sai, sak;  // A[i][k] = A[i*sai + k*sak]
  const bf16_t *B;
  long sbk, sbj;  // B[k][j] = B[k*sbk + j*sbj]
  int M, N, K;
  int mode;
  const float *bias;   // EPI_STORE / EPI_GELU (may be NULL)
  float *C;            // FP32 result (Y, Z or dZ), row stride ldc
  bf16_t *Cb;          // BF16 copy (GELU(Z) or dZ; optional for EPI_STORE)
  const float *Zprev;  // EPI_GELU_BACK: pre-activation below, row stride ldc
  int ldc;
};

__global__ __launch_bounds__(256) void k_gemm_bf16(gemm_args g) {
  __shared__ __attribute__((aligned(16))) bf16_t As[GT][GKP];  // As[i][k]
  __shared__ __attribute__((aligned(16))) bf16_t Bs[GT][GKP];  // Bs[j][k] (B transposed)
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int i0 = blockIdx.y * GT, j0 = blockIdx.x * GT;
  const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
  const int lr = lane & 15, kq = (lane >> 4) * 8;
  f32x4 acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < g.K; k0 += GK) {
    for (int e = tid; e < GT * GK; e += 256) {
      const int r = e / GK, k = e % GK, gi = i0 + r, gk = k0 + k;
      As[r][k] = (gi < g.M && gk < g.K) ? g.A[gi * g.sai + gk * g.sak] : (bf16_t)0;
    }
    for (int e = tid; e < GT * GK; e += 256) {
      const int c = e / GK, k = e % GK, gj = j0 + c, gk = k0 + k;
      Bs[c][k] = (gj < g.N && gk < g.K) ? g.B[gk * g.sbk + gj * g.sbj] : (bf16_t)0;
    }
    __syncthreads();
    bf16x8 a[2], b[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      a[t] = *(const bf16x8 *)&As[wi + 16 * t + lr][kq];
      b[t] = *(const bf16x8 *)&Bs[wj + 16 * t + lr][kq];
    }
#pragma unroll
    for (int ti = 0; ti < 2; ti++)
#pragma unroll
      for (int tj = 0; tj < 2; tj++) acc[ti][tj] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ti], b[tj], acc[ti][tj], 0, 0, 0);
    __syncthreads();
  }
  // lane holds D[4*(lane/16) + v][lane%16] of each 16 x 16 block
#pragma unroll
  for (int ti = 0; ti < 2; ti++)
#pragma unroll
    for (int tj = 0; tj < 2; tj++)
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int i = i0 + wi + 16 * ti + 4 * (lane >> 4) + v;
        const int j = j0 + wj + 16 * tj + lr;
        if (i >= g.M || j >= g.N) continue;
        const long o = (long)i * g.ldc + j;
        float x = acc[ti][tj][v];
        if (g.mode == EPI_GELU_BACK) {
          x *= gelu_d(g.Zprev[o]);
          g.C[o] = x;
          g.Cb[o] = f2bf(x);
        } else {
          if (g.bias) x += g.bias[j];
          g.C[o] = x;
          if (g.mode == EPI_GELU)
            g.Cb[o] = f2bf(gelu(x));
          else if (g.Cb)
            g.Cb[o] = f2bf(x);
        }
      }
}

__global__ void k_f32_to_bf16(const float *src, bf16_t *dst, long n) {
  const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (l < n) dst[l] = f2bf(src[l]);
}

// MSE over the batch: dY = 2 (Y - T) / n (FP32 and BF16), loss into
// *loss (a fixed-order tree over one workgroup)
__global__ __launch_bounds__(1024) void k_mse(const float *Y, const float *T, long n, float *dY, bf16_t *dYb,
                                              float *loss) {
  __shared__ float red[1024];
  const float scale = 2.0f / (float)n;
  float s = 0.f;
  for (long l = threadIdx.x; l < n; l += 1024) {
    const float d = Y[l] - T[l];
    s += d * d;
    const float g = scale * d;
    dY[l] = g;
    dYb[l] = f2bf(g);
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = 512; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = red[0] / (float)n;
}

// bias gradient: column sums of dZ (rows in order)
__global__ void k_colsum(const float *dZ, int rows, int cols, float *db) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= cols) return;
  float s = 0.f;
  for (int i = 0; i < rows; i++) s += dZ[(long)i * cols + j];
  db[j] = s;
}

// Adam (bias-corrected), then the BF16 copy of the weights
__global__ void k_adam(float *w, const float *gr, float *m, float *v, bf16_t *wb, long n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  const long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n) return;
  const float g = gr[l];
  const float mm = b1 * m[l] + (1.f - b1) * g;
  const float vv = b2 * v[l] + (1.f - b2) * g * g;
  m[l] = mm;
  v[l] = vv;
  const float x = w[l] - lr * (mm / c1) / (sqrtf(vv / c2) + eps);
  w[l] = x;
  wb[l] = f2bf(x);
}

// ------------------------------------------------- networks in LDS -----
// (pointers to global memory: as generic ones, loaded from memory, every access
// would be a flat instruction)
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) float mlp_f;
typedef __attribute__((address_space(1))) bf16_t mlp_b;
typedef __attribute__((address_space(1))) bf16x8 mlp_b8;
typedef __attribute__((address_space(1))) u32x2 mlp_u2;

// Matrices that the MFMAs read as operands are stored tile by tile in the
// operand's own order: a tile is 16 columns x 32 of the contracted index k,
// lane (c % 16) + 16 (k % 32 / 8) holding eight consecutive k of column c, so
// that a wave's operand is one contiguous kilobyte.  (Row by row, a lane's 16
// bytes lie a row apart from its neighbour's and each takes a cache access of
// its own: 5.1 us a layer in k_mlp_rows.)  Tiles of a column block follow
// each other in k, ksteps of them; whatever no weight or value fills is zero.
#define MLP_TILE 512
__device__ __forceinline__ long mlp_tile(int c, int k, int ksteps) {
  return ((long)(c >> 4) * ksteps + (k >> 5)) * MLP_TILE + ((c & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

// One dense layer as the two kernels below see it, in device memory (uniform
// loads, two cache lines a layer).  kp and np are K and N rounded up to 128
// (whole groups of four steps); the batch is padded to ldb, a multiple of 32.
struct mlp_layer {
  int K, N, kp, np;
  mlp_f *bias;     // in the flat parameters
  mlp_b *Wb, *Wt;  // tiles of W: columns n over k, and columns k over n
  mlp_f *Z;        // batch x N: GELU' of the pre-activations; the last layer's output
  mlp_f *dZ;       // batch x N: their gradients
  mlp_b *Ht;       // tiles of the layer's input: columns k over the batch
  mlp_b *dZt;      // tiles of the gradients: columns n over the batch
};

// One wave's work in k_mlp_weights
enum { JOB_LOSS = 0, JOB_BIAS = 1, JOB_WEIGHT = 2 };
struct mlp_job {
  int kind, n0, k0, K, N, kp, np, unused;
  long at;  // the bias or weight matrix in the flat parameters
  mlp_b *Wb, *Wt, *Ht, *dZt;
  mlp_f *dZ;
};

#define MLP_ROWS_TPB 1024  // 16 waves, one 16-column block of the layer each
#define MLP_PAD 8          // LDS row padding (16 bytes)

// the squared error's partial sums (k_mlp_weights) to one number, in the
// order of k_mse's tree; one workgroup of MLP_ROWS_TPB threads
__device__ __forceinline__ void mlp_loss_tree(const float *lossp, long n, float *red, float *loss) {
  red[threadIdx.x] = lossp[threadIdx.x];
  __syncthreads();
  for (int w = MLP_ROWS_TPB / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = red[0] / (float)n;
}

// One wave's weights for the first 8 steps (256 of k) of a 16-column block,
// and its column's bias: loaded a layer ahead, so that their latency passes
// behind the layer before and its barrier.
struct mlp_ahead {
  bf16x8 b[8];
  float bias;
  // tile: the block's first tile
  __device__ __forceinline__ void load(const mlp_b *tile, int kp) {
    const mlp_b *q = tile + (threadIdx.x & 63) * 8;
#pragma unroll
    for (int u = 0; u < 4; u++) b[u] = *(const mlp_b8 *)(q + MLP_TILE * u);
    if (kp > 128) {
#pragma unroll
      for (int u = 4; u < 8; u++) b[u] = *(const mlp_b8 *)(q + MLP_TILE * u);
    }
  }
};

// A 16 x 16 block of act (this lane's row in LDS) times a weight copy's
// column block, k < kp, the first 256 of k loaded ahead: one accumulator,
// 32-wide steps in increasing k
__device__ __forceinline__ f32x4 mlp_block(const bf16_t *act, const mlp_ahead &w, const mlp_b *tile, int kp) {
  const int lane = threadIdx.x & 63;
  const bf16_t *a = act + (lane >> 4) * 8;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 4; u++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)(a + 32 * u), w.b[u], acc, 0, 0, 0);
  if (kp > 128) {
#pragma unroll
    for (int u = 4; u < 8; u++)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)(a + 32 * u), w.b[u], acc, 0, 0, 0);
  }
  const mlp_b *b = tile + lane * 8;
#pragma unroll 2
  for (int k = 256; k < kp; k += 128) {
    bf16x8 bv[4];
#pragma unroll
    for (int u = 0; u < 4; u++) bv[u] = *(const mlp_b8 *)(b + (long)k * (MLP_TILE / 32) + MLP_TILE * u);
#pragma unroll
    for (int u = 0; u < 4; u++)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*(const bf16x8 *)(a + k + 32 * u), bv[u], acc, 0, 0, 0);
  }
  return acc;
}

// V consecutive k of one column of a tile
template <int V>
__device__ __forceinline__ void mlp_store_rows(mlp_b *t, const bf16_t (&h)[V]) {
  if constexpr (V == 4)
    *(mlp_u2 *)t = u32x2{h[0] | (unsigned)h[1] << 16, h[2] | (unsigned)h[3] << 16};
  else if constexpr (V == 2)
    *(__attribute__((address_space(1))) unsigned *)t = h[0] | (unsigned)h[1] << 16;
  else
    *t = h[0];
}

// Forward pass of 4 V rows through every layer and, when TRAIN, the MSE
// gradient back through every layer.  Rows are independent of each other,
// so one workgroup carries its rows through the whole network: the
// activations stay in LDS (BF16), the weights stream from L2 straight into
// MFMA operands, and a layer costs one
// barrier instead of a launch.
// The MFMA block has 16 rows; row r of it holds the workgroup's row
// (r / 4) V + min(r % 4, V - 1), so that with few rows every lane still has
// V results: GELU (erff, ~100 instructions) on them and the weights'
// passage through the CU's L1 (1.3 MB both ways for the emulator network)
// are what bounds the kernel, the products are not.  GELU' is formed on the
// way up, where erff is at hand, and kept for the way back.
// 512 rows of 5-256-256-256-256-512: 28 us; with k_mlp_weights 41 us a
// training step, where fourteen k_gemm_bf16, five k_colsum (114 us each), k_mse
// and k_adam took 1160 us.  Forward alone, 128 rows: 13 us, was 5 x 24 us; 18 us
// with its rows and output in pinned host memory.
// Workgroups are dispatched round-robin over the 8 XCDs; each XCD takes a
// contiguous run of rows, so that the tiles they fill together are written
// through one L2 (with neighbouring rows on different XCDs, k_mlp_weights
// read the partly written lines 55 us slower).
// The last workgroup of a launch with loss != NULL reduces the previous
// step's loss partials instead.  Y: where a forward pass's output goes (NULL:
// Z of the last layer).
template <int V, bool TRAIN>
__global__ __launch_bounds__(MLP_ROWS_TPB) void k_mlp_rows(const mlp_layer *__restrict__ net, int L,
                                                           const float *__restrict__ X, const float *__restrict__ T,
                                                           int batch, int ldb, int ld, const float *lossp,
                                                           float *loss, float *Y) {
  extern __shared__ __attribute__((aligned(16))) bf16_t lds_mlp[];
  if (TRAIN && loss && blockIdx.x == gridDim.x - 1) {
    mlp_loss_tree(lossp, (long)batch * net[L - 1].N, (float *)lds_mlp, loss);
    return;
  }
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int lr = lane & 15, rq = V * (lane >> 4);  // this lane's column and first row of a block
  const int per = (int)gridDim.x / 8;  // (the grid is 8 per, plus the one above)
  const int i0 = ((int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8)) * 4 * V;
  const int bsteps = ldb / 32;
  if (i0 >= (TRAIN ? (batch + 31) / 32 * 32 : batch)) return;
  const int jw = wave * 16 + lr;  // its column in the wave's first block
  bf16_t *cur = lds_mlp, *nxt = lds_mlp + 4 * V * ld;
  const int arow = ((lr >> 2) * V + min(lr & 3, V - 1)) * ld;  // its MFMA row in LDS
  mlp_ahead ah;
  // what the wave's first block of pass q reads: q < L forward layer q, then
  // back through layers L - 1 .. 1
  auto ahead = [&](int q) {
    if (q < L) {
      const mlp_layer &n = net[q];
      if (wave * 16 < n.np) ah.load(n.Wb + (long)wave * (n.kp / 32) * MLP_TILE, n.kp);
      ah.bias = n.bias[min(jw, n.N - 1)];
    } else if (TRAIN && q < 2 * L - 1) {
      const mlp_layer &n = net[2 * L - 1 - q];
      if (wave * 16 < n.kp) ah.load(n.Wt + (long)wave * (n.np / 32) * MLP_TILE, n.np);
    }
  };
  ahead(0);
  {
    const int K = net[0].K, kp = net[0].kp;
    for (int e = tid; e < 4 * V * kp; e += MLP_ROWS_TPB) {
      const int r = e / kp, k = e - r * kp;
      const bool in = i0 + r < batch && k < K;
      const bf16_t h = in ? f2bf(X[(long)(i0 + r) * K + k]) : (bf16_t)0;
      cur[r * ld + k] = h;
      if (TRAIN && k < K) net[0].Ht[mlp_tile(k, i0 + r, bsteps)] = h;
    }
  }
  __syncthreads();
  for (int l = 0; l < L; l++) {
    const mlp_layer n = net[l];
    const bool last = l == L - 1;
    const float scale = 2.0f / (float)((long)batch * n.N);
    mlp_b *tr = TRAIN ? (last ? n.dZt : net[l + 1].Ht) : nullptr;
    if (wave * 16 >= n.np) ahead(l + 1);  // (a wave without a block here)
    for (int j0 = wave * 16; j0 < n.np; j0 += MLP_ROWS_TPB / 4) {
      const int j = j0 + lr, jc = min(j, n.N - 1);
      const mlp_b *tile = n.Wb + (long)(j0 / 16) * (n.kp / 32) * MLP_TILE;
      if (j0 != wave * 16) {  // (a wave's first block was loaded ahead)
        ah.load(tile, n.kp);
        ah.bias = n.bias[jc];
      }
      float t[V];
      if (TRAIN && last) {
#pragma unroll
        for (int v = 0; v < V; v++) t[v] = T[(long)min(i0 + rq + v, batch - 1) * n.N + jc];
      }
      const f32x4 acc = mlp_block(cur + arow, ah, tile, n.kp);
      const float bj = ah.bias;
      if (j0 + MLP_ROWS_TPB / 4 >= n.np) ahead(l + 1);
      bf16_t h[V];
#pragma unroll
      for (int v = 0; v < V; v++) {
        const int i = i0 + rq + v;
        const bool in = i < batch && j < n.N;
        const float x = acc[v] + bj;
        const long o = (long)i * n.N + j;
        h[v] = 0;
        if (!last) {
          float d;
          const float y = gelu_both(x, d);
          if (in) {
            h[v] = f2bf(y);
            if (TRAIN) n.Z[o] = d;
          }
        } else if (in) {
          (!TRAIN && Y ? (mlp_f *)Y : n.Z)[o] = x;
          if (TRAIN) {  // dY = 2 (Y - T) / n
            const float d = x - t[v];
            const float gd = scale * d;
            n.dZ[o] = gd;
            h[v] = f2bf(gd);
          }
        }
        if (TRAIN || !last) nxt[(rq + v) * ld + j] = h[v];
      }
      if (TRAIN && j < n.N) mlp_store_rows<V>(tr + mlp_tile(j, i0 + rq, bsteps), h);
    }
    __syncthreads();
    bf16_t *s = cur;
    cur = nxt;
    nxt = s;
  }
  if constexpr (TRAIN) {
    for (int l = L - 1; l >= 1; l--) {  // dZ below = (dZ W) * GELU'(Z below)
      const mlp_layer n = net[l], below = net[l - 1];
      if (wave * 16 >= n.kp) ahead(2 * L - l);
      for (int j0 = wave * 16; j0 < n.kp; j0 += MLP_ROWS_TPB / 4) {
        const int j = j0 + lr, jc = min(j, n.K - 1);
        const mlp_b *tile = n.Wt + (long)(j0 / 16) * (n.np / 32) * MLP_TILE;
        if (j0 != wave * 16) ah.load(tile, n.np);
        float d[V];  // (this lane stored them on the way up)
#pragma unroll
        for (int v = 0; v < V; v++) d[v] = below.Z[(long)min(i0 + rq + v, batch - 1) * n.K + jc];
        const f32x4 acc = mlp_block(cur + arow, ah, tile, n.np);
        if (j0 + MLP_ROWS_TPB / 4 >= n.kp) ahead(2 * L - l);
        bf16_t h[V];
#pragma unroll
        for (int v = 0; v < V; v++) {
          const int i = i0 + rq + v;
          h[v] = 0;
          if (i < batch && j < n.K) {
            const float x = acc[v] * d[v];
            below.dZ[(long)i * n.K + j] = x;
            h[v] = f2bf(x);
          }
          nxt[(rq + v) * ld + j] = h[v];
        }
        if (j < n.K) mlp_store_rows<V>(below.dZt + mlp_tile(j, i0 + rq, bsteps), h);
      }
      __syncthreads();
      bf16_t *s = cur;
      cur = nxt;
      nxt = s;
    }
  }
}

struct adam_args {
  float lr, b1, b2, eps, c1, c2;
};

// one parameter's Adam step (bias-corrected): its moments updated, its new
// value returned
__device__ __forceinline__ float adam_step(float p, float &m, float &v, float g, const adam_args &a) {
  m = a.b1 * m + (1.f - a.b1) * g;
  v = a.b2 * v + (1.f - a.b2) * g * g;
  return p - a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
}

#define MLP_CS_U 128  // rows a lane has in flight in a column sum
#define MLP_LS_U 64   // values of each array in the squared error's sums

// Everything of a training step after k_mlp_rows, one wave per job, the
// long sequential ones first:
//   - 16 waves: the squared error's 1024 partial sums (k_mse's order);
//   - 64 columns per wave: the bias gradient (rows in order) and its step;
//   - 32 x 32 weights per wave: dW = dZ^T H over the batch as 2 x 2 MFMA
//     blocks, 32 rows per step, then Adam on the accumulators and both BF16
//     copies of the new weights.
// ADAM false stores the gradient instead (fg_mlp_gradient).  Every operand
// is stored in tiles over the batch, so the fragments load straight from
// memory, and a job's new weights fill whole tiles of both copies; 32 x 32
// weights a job give the 330k-weight network 330 waves, where the 64 x 64 workgroups of
// k_gemm_bf16 gave 4 to 32 a layer.  Bound: the latency of reading what
// other XCDs have just written, a few round trips deep, so every job has as
// much in flight as its registers hold.
// 512 rows of that network: 13 us (20 us with half as many loads in flight).
template <bool ADAM>
__global__ __launch_bounds__(64) void k_mlp_weights(const mlp_job *__restrict__ jobs, const float *__restrict__ Y,
                                                    const float *__restrict__ T, int nout, int batch, int ldb,
                                                    mlp_f *p, mlp_f *g, mlp_f *m, mlp_f *v, mlp_f *lossp,
                                                    adam_args ad) {
  const int lane = threadIdx.x;
  const mlp_job job = jobs[blockIdx.x];
  if (job.kind == JOB_LOSS) {
    const long n = (long)batch * nout;
    const int t = job.n0 + lane;
    float s = 0.f;
    // whole chunks without a condition on the sums: loads that only a
    // condition needs sink into it, one latency each
    long l0 = t;
    for (; l0 - t + (long)MLP_ROWS_TPB * MLP_LS_U <= n; l0 += (long)MLP_ROWS_TPB * MLP_LS_U) {
      float y[MLP_LS_U], z[MLP_LS_U];
#pragma unroll
      for (int u = 0; u < MLP_LS_U; u++) {
        y[u] = Y[l0 + (long)MLP_ROWS_TPB * u];
        z[u] = T[l0 + (long)MLP_ROWS_TPB * u];
      }
#pragma unroll
      for (int u = 0; u < MLP_LS_U; u++) {
        const float d = y[u] - z[u];
        s += d * d;
      }
    }
    for (; l0 < n; l0 += MLP_ROWS_TPB) {
      const float d = Y[l0] - T[l0];
      s += d * d;
    }
    lossp[t] = s;
    return;
  }
  if (job.kind == JOB_BIAS) {
    const int j = job.n0 + lane, jc = min(j, job.N - 1);
    const mlp_f *dZ = job.dZ + jc;
    const long q = job.at + jc;
    float pv = 0.f, mv = 0.f, vv = 0.f;
    if (ADAM) {
      pv = p[q];
      mv = m[q];
      vv = v[q];
    }
    float s = 0.f;
    int i0 = 0;
    for (; i0 + MLP_CS_U <= batch; i0 += MLP_CS_U) {
      float x[MLP_CS_U];
#pragma unroll
      for (int u = 0; u < MLP_CS_U; u++) x[u] = dZ[(long)(i0 + u) * job.N];
#pragma unroll
      for (int u = 0; u < MLP_CS_U; u++) s += x[u];
    }
#pragma unroll 16
    for (; i0 < batch; i0++) s += dZ[(long)i0 * job.N];
    if (j < job.N) {
      if constexpr (ADAM) {
        p[q] = adam_step(pv, mv, vv, s, ad);
        m[q] = mv;
        v[q] = vv;
      } else {
        g[q] = s;
      }
    }
    return;
  }
  const int n0 = job.n0, k0 = job.k0, N = job.N, K = job.K;
  const int lr = lane & 15, kq = (lane >> 4) * 8, rq = 4 * (lane >> 4);
  // a lane holds rows n0 + 16 x + rq .. + 3 of column k0 + 16 y + lr of each
  // block; the parameters and moments of all of them load together, first
  float pv[2][2][4], mv[2][2][4], vv[2][2][4];
  if constexpr (ADAM) {
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++)
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int n = min(n0 + 16 * x + rq + u, N - 1), k = min(k0 + 16 * y + lr, K - 1);
          const long q = job.at + (long)n * K + k;
          pv[x][y][u] = p[q];
          mv[x][y][u] = m[q];
          vv[x][y][u] = v[q];
        }
  }
  const long bs = (long)(ldb / 32) * MLP_TILE;  // a column block of the batch's tiles
  const mlp_b *a0 = job.dZt + n0 / 16 * bs + lane * 8, *a1 = a0 + bs;
  const mlp_b *b0 = job.Ht + k0 / 16 * bs + lane * 8, *b1 = b0 + bs;
  f32x4 acc[2][2] = {};
#pragma unroll 8
  for (long b = 0; b < (long)(batch + 31) / 32 * MLP_TILE; b += MLP_TILE) {
    const bf16x8 av[2] = {*(const mlp_b8 *)(a0 + b), *(const mlp_b8 *)(a1 + b)};
    const bf16x8 bv[2] = {*(const mlp_b8 *)(b0 + b), *(const mlp_b8 *)(b1 + b)};
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
      for (int y = 0; y < 2; y++) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[x], bv[y], acc[x][y], 0, 0, 0);
  }
#pragma unroll
  for (int x = 0; x < 2; x++)
#pragma unroll
    for (int y = 0; y < 2; y++) {
      const int k = k0 + 16 * y + lr, nq = n0 + 16 * x + rq;
      if (k >= K) continue;
      bf16_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int n = nq + u;
        if (n >= N) continue;
        const long q = job.at + (long)n * K + k;
        if constexpr (ADAM) {
          const float pn = adam_step(pv[x][y][u], mv[x][y][u], vv[x][y][u], acc[x][y][u], ad);
          p[q] = pn;
          m[q] = mv[x][y][u];
          v[q] = vv[x][y][u];
          w[u] = f2bf(pn);
          job.Wb[mlp_tile(n, k, job.kp / 32)] = w[u];
        } else {
          g[q] = acc[x][y][u];
        }
      }
      if (ADAM && nq < N) mlp_store_rows<4>(job.Wt + mlp_tile(k, nq, job.np / 32), w);
    }
}

// the last step's loss partials (grid of one workgroup)
__global__ __launch_bounds__(MLP_ROWS_TPB) void k_mlp_loss(const float *lossp, long n, float *loss) {
  __shared__ float red[MLP_ROWS_TPB];
  mlp_loss_tree(lossp, n, red, loss);
}

// both BF16 copies of the weights (layer blockIdx.y; p: its FP32 weights
// precede its bias)
__global__ void k_mlp_copies(const mlp_layer *__restrict__ net) {
  const mlp_layer n = net[blockIdx.y];
  const long q = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (long)n.N * n.K) return;
  const int i = (int)(q / n.K), k = (int)(q - (long)i * n.K);
  const bf16_t w = f2bf(n.bias[q - (long)n.N * n.K]);
  n.Wb[mlp_tile(i, k, n.kp / 32)] = w;
  n.Wt[mlp_tile(k, i, n.np / 32)] = w;
}

// ------------------------------------------------------------ host ----
struct fg_mlp {
  int L;                        // dense layers
  int width[MLP_MAX_LAYERS + 1];  // width[0] inputs ... width[L] outputs
  int max_batch;
  long nparam;
  long offW[MLP_MAX_LAYERS], offb[MLP_MAX_LAYERS];
  hipStream_t stream;
  float *p, *g, *m, *v;  // parameters, gradients, Adam moments (FP32)
  bf16_t *pb;            // BF16 parameters
  bf16_t *H[MLP_MAX_LAYERS];     // BF16 layer inputs (H[0] = x)
  // Z[L-1]: the output.  Below it what the way back needs: with net (networks in
  // LDS) GELU' of the pre-activations, left by a training pass alone; without it
  // the pre-activations
  float *Z[MLP_MAX_LAYERS];
  float *dZ[MLP_MAX_LAYERS];     // FP32 gradients of the pre-activations
  bf16_t *dZb[MLP_MAX_LAYERS];   // and their BF16 copies
  float *X, *T;                  // FP32 batch inputs and targets
  float *loss;                   // per-step losses of the last fg_mlp_train call
  int loss_cap;
  long step;                     // Adam steps taken
  // networks in LDS (mlp_fits_rows): the kernels' view of the arrays, the
  // padded arrays it points to in one allocation, and fg_mlp_train's
  // samples (kept for the next call, grown when a larger set comes, given back
  // after a call whose set takes more than MLP_KEEP_BYTES)
  mlp_layer *net;                // device copy; NULL: layer by layer
  mlp_job *jobs;                 // k_mlp_weights's work list, njobs entries
  int njobs;
  char *padded;
  float *lossp;                  // MLP_ROWS_TPB partial sums of the squared error
  int ld, ldb;                   // LDS row length of k_mlp_rows, row length of the transposes
  float *Xall, *Tall;
  size_t all_cap;                // samples they hold
  // small forward passes: pinned host memory that k_mlp_rows reads its rows from
  // and writes its output to, and its device alias.  Allocated with the network,
  // while its device is the current one; NULL where it could not be: rows are copied
  float *h_io, *d_io;
};
// Bytes of it at most, as it stays pinned while the network lives.  The two copies
// cost a call more than the kernel's own way over the bus (us per fg_mlp_forward of
// 5-256x4-512 with and without them: 1 row 39 and 27, 128 rows 50 and 38, 512 rows 97
// and 82, 1024 rows 158 and 136, 2000 rows, 4.1 MB, 266 and 245; beyond the bound the
// gain is 6 to 8 %: 3000 rows 386 and 370).  A network's first call: 128 rows 52
// and 43, 2000 rows 270 and 275; fg_mlp_create takes 1.13 ms with it, 1.10 without.
#define MLP_IO_BYTES (4 << 20)
// Bytes of fg_mlp_train's samples that a network keeps between calls
#define MLP_KEEP_BYTES (64 << 20)

// Rows per workgroup of k_mlp_rows, 4 V: few, so that the chip's CUs share
// the GELUs, until every CU has a workgroup; then more rows for each passage
// of the weights.  Microseconds per training step with 4, 8, 16 rows:
// batch 512 40.6, 42.2, 53.5; 1024 53.1, 53.9, 64.8; 2048 95.7, 76.2, 86.0;
// 4096 176, 135, 122.
static int mlp_rows_v(int batch) { return batch <= 4 * 256 ? 1 : batch <= 8 * 256 ? 2 : 4; }

// k_mlp_rows keeps two sets of up to 16 activation rows in LDS: networks up
// to 896 wide fit 64 KB.  Wider ones run layer by layer (k_gemm_bf16).
static int mlp_rows_ld(const fg_mlp *m) {
  int kp = 0;
  for (int l = 0; l <= m->L; l++) kp = std::max(kp, (m->width[l] + 127) / 128 * 128);
  return kp + MLP_PAD;
}
static bool mlp_fits_rows(int ld) { return (size_t)2 * 16 * ld * sizeof(bf16_t) <= 65536; }
static size_t mlp_rows_lds(int ld, int v) {  // (the loss tree of the last workgroup reuses it)
  return std::max((size_t)2 * 4 * v * ld * sizeof(bf16_t), (size_t)MLP_ROWS_TPB * sizeof(float));
}

static fg_status mlp_gemm(fg_mlp *m, const gemm_args &g) {
  dim3 grid((g.N + GT - 1) / GT, (g.M + GT - 1) / GT);
  hipLaunchKernelGGL(k_gemm_bf16, grid, dim3(256), 0, m->stream, g);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

static uint64_t mix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
  x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
  return x ^ (x >> 31);
}

extern "C" fg_status fg_mlp_set_params(fg_mlp *m, const float *params);

extern "C" fg_status fg_mlp_destroy(fg_mlp *m) {
  if (!m) return FG_OK;
  (void)hipStreamSynchronize(m->stream);
  void *ptrs[] = {m->p, m->g, m->m, m->v, m->pb, m->X, m->T, m->loss, m->net, m->jobs, m->padded, m->lossp, m->Xall, m->Tall};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  for (int l = 0; l < MLP_MAX_LAYERS; l++) {
    void *q[] = {m->H[l], m->Z[l], m->dZ[l], m->dZb[l]};
    for (void *x : q)
      if (x) (void)hipFree(x);
  }
  if (m->h_io) (void)hipHostFree(m->h_io);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return FG_OK;
}

#define MLP_TRY(call)              \
  do {                             \
    hipError_t e_ = (call);        \
    if (e_ != hipSuccess) {        \
      fg_set_error("mlp: %s", hipGetErrorString(e_)); \
      fg_mlp_destroy(m);           \
      return FG_E_HIP;             \
    }                              \
  } while (0)

// widths[0..nlayers]: inputs, hidden widths, outputs.  Weights drawn
// uniform in +-sqrt(6 / (fan_in + fan_out)) from seed, biases zero.
extern "C" fg_status fg_mlp_create(const int *widths, int nlayers, int max_batch, unsigned long long seed,
                                   int device, fg_mlp **out) {
  if (!widths || !out || nlayers < 1 || nlayers > MLP_MAX_LAYERS || max_batch < 1) {
    fg_set_error("fg_mlp_create: bad argument");
    return FG_E_INVALID;
  }
  for (int l = 0; l <= nlayers; l++)
    if (widths[l] < 1 || widths[l] > 65536) {
      fg_set_error("fg_mlp_create: width %d", widths[l]);
      return FG_E_INVALID;
    }
  FG_HIP(hipSetDevice(device));
  fg_mlp *m = new fg_mlp();
  m->L = nlayers;
  for (int l = 0; l <= nlayers; l++) m->width[l] = widths[l];
  m->max_batch = max_batch;
  long off = 0;
  for (int l = 0; l < nlayers; l++) {
    m->offW[l] = off;
    off += (long)widths[l + 1] * widths[l];
    m->offb[l] = off;
    off += widths[l + 1];
  }
  m->nparam = off;
  MLP_TRY(hipStreamCreate(&m->stream));
  const size_t P = (size_t)off;
  MLP_TRY(hipMalloc((void **)&m->p, P * 4));
  MLP_TRY(hipMalloc((void **)&m->g, P * 4));
  MLP_TRY(hipMalloc((void **)&m->m, P * 4));
  MLP_TRY(hipMalloc((void **)&m->v, P * 4));
  MLP_TRY(hipMemset(m->m, 0, P * 4));
  MLP_TRY(hipMemset(m->v, 0, P * 4));
  MLP_TRY(hipMemset(m->g, 0, P * 4));
  m->ld = mlp_rows_ld(m);
  const bool rows = mlp_fits_rows(m->ld);
  if (!rows) MLP_TRY(hipMalloc((void **)&m->pb, P * 2));
  for (int l = 0; l < nlayers; l++) {
    const size_t in = (size_t)max_batch * widths[l], outn = (size_t)max_batch * widths[l + 1];
    MLP_TRY(hipMalloc((void **)&m->Z[l], outn * 4));
    MLP_TRY(hipMalloc((void **)&m->dZ[l], outn * 4));
    if (rows) continue;
    MLP_TRY(hipMalloc((void **)&m->H[l], in * 2));
    MLP_TRY(hipMalloc((void **)&m->dZb[l], outn * 2));
  }
  if (rows) {
    m->ldb = (max_batch + 31) / 32 * 32;
    mlp_layer net[MLP_MAX_LAYERS] = {};
    size_t at[MLP_MAX_LAYERS][4], end = 0;
    auto take = [&](size_t count) {  // (256-byte aligned pieces)
      const size_t o = end;
      end += (count * sizeof(bf16_t) + 255) / 256 * 256;
      return o;
    };
    for (int l = 0; l < nlayers; l++) {
      mlp_layer &n = net[l];
      n.K = widths[l];
      n.N = widths[l + 1];
      n.kp = (n.K + 127) / 128 * 128;
      n.np = (n.N + 127) / 128 * 128;
      at[l][0] = take((size_t)n.np * n.kp);
      at[l][1] = take((size_t)n.kp * n.np);
      at[l][2] = take((size_t)n.kp * m->ldb);
      at[l][3] = take((size_t)n.np * m->ldb);
    }
    MLP_TRY(hipMalloc((void **)&m->padded, end));
    MLP_TRY(hipMemset(m->padded, 0, end));  // the padding stays zero
    MLP_TRY(hipMalloc((void **)&m->lossp, MLP_ROWS_TPB * sizeof(float)));
    std::vector<mlp_job> jobs;
    for (int t = 0; t < MLP_ROWS_TPB; t += 64) {
      mlp_job j{};
      j.kind = JOB_LOSS;
      j.n0 = t;
      jobs.push_back(j);
    }
    for (int l = 0; l < nlayers; l++) {
      mlp_layer &n = net[l];
      n.Wb = (mlp_b *)(m->padded + at[l][0]);
      n.Wt = (mlp_b *)(m->padded + at[l][1]);
      n.Ht = (mlp_b *)(m->padded + at[l][2]);
      n.dZt = (mlp_b *)(m->padded + at[l][3]);
      n.bias = (mlp_f *)(m->p + m->offb[l]);
      n.Z = (mlp_f *)m->Z[l];
      n.dZ = (mlp_f *)m->dZ[l];
    }
    auto push = [&](int kind, int l, int n0, int k0) {
      const mlp_layer &n = net[l];
      jobs.push_back({kind, n0, k0, n.K, n.N, n.kp, n.np, 0, kind == JOB_BIAS ? m->offb[l] : m->offW[l], n.Wb, n.Wt, n.Ht,
                      n.dZt, n.dZ});
    };
    for (int l = 0; l < nlayers; l++)
      for (int n0 = 0; n0 < widths[l + 1]; n0 += 64) push(JOB_BIAS, l, n0, 0);
    for (int l = 0; l < nlayers; l++)
      for (int n0 = 0; n0 < widths[l + 1]; n0 += 32)
        for (int k0 = 0; k0 < widths[l]; k0 += 32) push(JOB_WEIGHT, l, n0, k0);
    m->njobs = (int)jobs.size();
    MLP_TRY(hipMalloc((void **)&m->net, sizeof net));
    MLP_TRY(hipMemcpy(m->net, net, sizeof net, hipMemcpyHostToDevice));
    MLP_TRY(hipMalloc((void **)&m->jobs, jobs.size() * sizeof(mlp_job)));
    MLP_TRY(hipMemcpy(m->jobs, jobs.data(), jobs.size() * sizeof(mlp_job), hipMemcpyHostToDevice));
    const size_t most = (size_t)max_batch * (widths[0] + widths[nlayers]) * 4;
    void *h = nullptr, *d = nullptr;
    if (hipHostMalloc(&h, std::min(most, (size_t)MLP_IO_BYTES), hipHostMallocCoherent | hipHostMallocMapped) !=
            hipSuccess ||
        hipHostGetDevicePointer(&d, h, 0) != hipSuccess) {
      if (h) (void)hipHostFree(h);
      h = d = nullptr;
      (void)hipGetLastError();  // (a later launch's check would report it)
    }
    m->h_io = (float *)h;
    m->d_io = (float *)d;
  }
  MLP_TRY(hipMalloc((void **)&m->X, (size_t)max_batch * widths[0] * 4));
  MLP_TRY(hipMalloc((void **)&m->T, (size_t)max_batch * widths[nlayers] * 4));
  std::vector<float> host(P, 0.0f);
  uint64_t state = seed;
  for (int l = 0; l < nlayers; l++) {
    const double lim = sqrt(6.0 / (double)(widths[l] + widths[l + 1]));
    for (long q = 0; q < (long)widths[l + 1] * widths[l]; q++) {
      state = mix64(state);
      const double u = (double)(state >> 11) * (1.0 / 9007199254740992.0);
      host[m->offW[l] + q] = (float)((2.0 * u - 1.0) * lim);
    }
  }
  fg_status st = fg_mlp_set_params(m, host.data());
  if (st) {
    fg_mlp_destroy(m);
    return st;
  }
  *out = m;
  return FG_OK;
}

extern "C" fg_status fg_mlp_set_params(fg_mlp *m, const float *params) {
  if (!m || !params) return FG_E_INVALID;
  FG_HIP(hipMemcpyAsync(m->p, params, m->nparam * 4, hipMemcpyHostToDevice, m->stream));
  if (m->net) {
    long most = 0;
    for (int l = 0; l < m->L; l++) most = std::max(most, (long)m->width[l] * m->width[l + 1]);
    hipLaunchKernelGGL(k_mlp_copies, dim3(fg_blocks(most, 256), m->L), dim3(256), 0, m->stream, m->net);
  } else {
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(fg_blocks(m->nparam, 256)), dim3(256), 0, m->stream, m->p, m->pb,
                       m->nparam);
  }
  FG_LAUNCH_CHECK();
  FG_HIP(hipStreamSynchronize(m->stream));
  return FG_OK;
}

extern "C" long fg_mlp_nparam(const fg_mlp *m) { return m ? m->nparam : 0; }

extern "C" fg_status fg_mlp_get_params(fg_mlp *m, float *params) {
  if (!m || !params) return FG_E_INVALID;
  FG_HIP(hipMemcpyAsync(params, m->p, m->nparam * 4, hipMemcpyDeviceToHost, m->stream));
  FG_HIP(hipStreamSynchronize(m->stream));
  return FG_OK;
}

// networks in LDS: forward pass of `batch` rows of x (device); output in
// y, or Z[L-1] without it.  With t (device targets) also the gradients of the
// pre-activations; *prev_loss, when not NULL, takes the loss of the step
// before this one.
template <int V>
static fg_status mlp_rows_launch(fg_mlp *m, const float *x, const float *t, int batch, float *prev_loss, float *y) {
  const size_t lds = mlp_rows_lds(m->ld, V);
  if (t) {
    // rows up to the next multiple of 32 are written (as zeros), which the
    // weight gradients' last step over the batch reads
    const int blocks = fg_blocks((batch + 31) / 32 * (32 / (4 * V)), 8) * 8 + (prev_loss ? 1 : 0);
    hipLaunchKernelGGL((k_mlp_rows<V, true>), dim3(blocks), dim3(MLP_ROWS_TPB), lds, m->stream, m->net, m->L, x, t,
                       batch, m->ldb, m->ld, m->lossp, prev_loss, nullptr);
  } else {
    hipLaunchKernelGGL((k_mlp_rows<V, false>), dim3(fg_blocks(fg_blocks(batch, 4 * V), 8) * 8), dim3(MLP_ROWS_TPB), lds,
                       m->stream, m->net, m->L, x, nullptr, batch, m->ldb, m->ld, nullptr, nullptr, y);
  }
  FG_LAUNCH_CHECK();
  return FG_OK;
}
static fg_status mlp_rows(fg_mlp *m, const float *x, const float *t, int batch, float *prev_loss,
                          float *y = nullptr) {
  switch (mlp_rows_v(batch)) {
    case 1: return mlp_rows_launch<1>(m, x, t, batch, prev_loss, y);
    case 2: return mlp_rows_launch<2>(m, x, t, batch, prev_loss, y);
    default: return mlp_rows_launch<4>(m, x, t, batch, prev_loss, y);
  }
}

// the weight gradients of mlp_rows(x, t): stored (adam NULL), or applied
static fg_status mlp_weights(fg_mlp *m, const float *t, int batch, const adam_args *adam) {
  auto kernel = adam ? k_mlp_weights<true> : k_mlp_weights<false>;
  hipLaunchKernelGGL(kernel, dim3(m->njobs), dim3(64), 0, m->stream, m->jobs, m->Z[m->L - 1], t, m->width[m->L],
                     batch, m->ldb, (mlp_f *)m->p, (mlp_f *)m->g, (mlp_f *)m->m, (mlp_f *)m->v, (mlp_f *)m->lossp,
                     adam ? *adam : adam_args{});
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// the loss of the last mlp_weights
static fg_status mlp_loss(fg_mlp *m, int batch, float *loss) {
  hipLaunchKernelGGL(k_mlp_loss, dim3(1), dim3(MLP_ROWS_TPB), 0, m->stream, m->lossp, (long)batch * m->width[m->L],
                     loss);
  FG_LAUNCH_CHECK();
  return FG_OK;
}

// forward pass of the batch in m->X (rows = batch); output in Z[L-1]
static fg_status mlp_forward(fg_mlp *m, int batch) {
  const int L = m->L;
  if (m->net) return mlp_rows(m, m->X, nullptr, batch, nullptr);
  hipLaunchKernelGGL(k_f32_to_bf16, dim3(fg_blocks((long)batch * m->width[0], 256)), dim3(256), 0, m->stream, m->X,
                     m->H[0], (long)batch * m->width[0]);
  FG_LAUNCH_CHECK();
  for (int l = 0; l < L; l++) {
    const int K = m->width[l], N = m->width[l + 1];
    gemm_args g{};
    g.A = m->H[l];
    g.sai = K;
    g.sak = 1;
    g.B = m->pb + m->offW[l];  // B[k][j] = W[j][k]
    g.sbk = 1;
    g.sbj = K;
    g.M = batch;
    g.N = N;
    g.K = K;
    g.bias = m->p + m->offb[l];
    g.C = m->Z[l];
    g.ldc = N;
    if (l < L - 1) {
      g.mode = EPI_GELU;
      g.Cb = m->H[l + 1];
    } else {
      g.mode = EPI_STORE;
      g.Cb = nullptr;
    }
    if (fg_status s = mlp_gemm(m, g)) return s;
  }
  return FG_OK;
}

// gradients of the MSE of Z[L-1] against m->T into m->g; loss to *loss_dev
static fg_status mlp_backward(fg_mlp *m, int batch, float *loss_dev) {
  const int L = m->L;
  const long nout = (long)batch * m->width[L];
  hipLaunchKernelGGL(k_mse, dim3(1), dim3(1024), 0, m->stream, m->Z[L - 1], m->T, nout, m->dZ[L - 1],
                     m->dZb[L - 1], loss_dev);
  FG_LAUNCH_CHECK();
  for (int l = L - 1; l >= 0; l--) {
    const int K = m->width[l], N = m->width[l + 1];
    // dW = dZ^T H: M = N rows, N = K columns, contraction over the batch
    gemm_args gw{};
    gw.A = m->dZb[l];
    gw.sai = 1;
    gw.sak = N;
    gw.B = m->H[l];
    gw.sbk = K;
    gw.sbj = 1;
    gw.M = N;
    gw.N = K;
    gw.K = batch;
    gw.mode = EPI_STORE;
    gw.C = m->g + m->offW[l];
    gw.ldc = K;
    if (fg_status s = mlp_gemm(m, gw)) return s;
    hipLaunchKernelGGL(k_colsum, dim3(fg_blocks(N, 256)), dim3(256), 0, m->stream, m->dZ[l], batch, N,
                       m->g + m->offb[l]);
    FG_LAUNCH_CHECK();
    if (l == 0) break;
    // dZ below = (dZ W) * GELU'(Z below)
    gemm_args gb{};
    gb.A = m->dZb[l];
    gb.sai = N;
    gb.sak = 1;
    gb.B = m->pb + m->offW[l];  // B[k][j] = W[k][j]
    gb.sbk = K;
    gb.sbj = 1;
    gb.M = batch;
    gb.N = K;
    gb.K = N;
    gb.mode = EPI_GELU_BACK;
    gb.C = m->dZ[l - 1];
    gb.Cb = m->dZb[l - 1];
    gb.Zprev = m->Z[l - 1];
    gb.ldc = K;
    if (fg_status s = mlp_gemm(m, gb)) return s;
  }
  return FG_OK;
}

static fg_status check_batch(fg_mlp *m, int batch) {
  if (!m || batch < 1 || batch > m->max_batch) {
    fg_set_error("mlp: batch %d outside 1..%d", batch, m ? m->max_batch : 0);
    return FG_E_INVALID;
  }
  return FG_OK;
}

// y[batch x outputs] = MLP(x[batch x inputs]), row-major FP32
extern "C" fg_status fg_mlp_forward(fg_mlp *m, const float *x, int batch, float *y) {
  if (fg_status s = check_batch(m, batch)) return s;
  const size_t nx = (size_t)batch * m->width[0], ny = (size_t)batch * m->width[m->L];
  // (NULL goes the way of the copies, which refuse it)
  if (m->h_io && x && y && (nx + ny) * 4 <= MLP_IO_BYTES) {
    std::memcpy(m->h_io, x, nx * 4);
    if (fg_status s = mlp_rows(m, m->d_io, nullptr, batch, nullptr, m->d_io + nx)) return s;
    FG_HIP(hipStreamSynchronize(m->stream));
    std::memcpy(y, m->h_io + nx, ny * 4);
    return FG_OK;
  }
  FG_HIP(hipMemcpyAsync(m->X, x, (size_t)batch * m->width[0] * 4, hipMemcpyHostToDevice, m->stream));
  if (fg_status s = mlp_forward(m, batch)) return s;
  FG_HIP(hipMemcpyAsync(y, m->Z[m->L - 1], (size_t)batch * m->width[m->L] * 4, hipMemcpyDeviceToHost, m->stream));
  FG_HIP(hipStreamSynchronize(m->stream));
  return FG_OK;
}

// MSE loss and its gradient with respect to every parameter (flat, in the
// fg_mlp_get_params order) for one batch; no update
extern "C" fg_status fg_mlp_gradient(fg_mlp *m, const float *x, const float *t, int batch, float *grad,
                                     float *loss) {
  if (fg_status s = check_batch(m, batch)) return s;
  FG_HIP(hipMemcpyAsync(m->X, x, (size_t)batch * m->width[0] * 4, hipMemcpyHostToDevice, m->stream));
  FG_HIP(hipMemcpyAsync(m->T, t, (size_t)batch * m->width[m->L] * 4, hipMemcpyHostToDevice, m->stream));
  if (!m->loss) {
    FG_HIP(hipMalloc((void **)&m->loss, 4));
    m->loss_cap = 1;
  }
  if (m->net) {
    if (fg_status s = mlp_rows(m, m->X, m->T, batch, nullptr)) return s;
    if (fg_status s = mlp_weights(m, m->T, batch, nullptr)) return s;
    if (fg_status s = mlp_loss(m, batch, m->loss)) return s;
  } else {
    if (fg_status s = mlp_forward(m, batch)) return s;
    if (fg_status s = mlp_backward(m, batch, m->loss)) return s;
  }
  if (grad) FG_HIP(hipMemcpyAsync(grad, m->g, m->nparam * 4, hipMemcpyDeviceToHost, m->stream));
  if (loss) FG_HIP(hipMemcpyAsync(loss, m->loss, 4, hipMemcpyDeviceToHost, m->stream));
  FG_HIP(hipStreamSynchronize(m->stream));
  return FG_OK;
}

static void mlp_free_samples(fg_mlp *m) {
  if (m->Xall) (void)hipFree(m->Xall);
  if (m->Tall) (void)hipFree(m->Tall);
  m->Xall = m->Tall = nullptr;
  m->all_cap = 0;
}

// `steps` Adam steps on the n samples (x: n x inputs, t: n x outputs),
// cycling through consecutive batches of `batch` rows (n a multiple of
// batch); losses[s] = the loss of step s before its update
extern "C" fg_status fg_mlp_train(fg_mlp *m, const float *x, const float *t, int n, int batch, int steps, float lr,
                                  float *losses) {
  if (fg_status s = check_batch(m, batch)) return s;
  if (n < batch || n % batch || steps < 1) {
    fg_set_error("fg_mlp_train: n %d must be a positive multiple of batch %d", n, batch);
    return FG_E_INVALID;
  }
  const int din = m->width[0], dout = m->width[m->L];
  fg_status st = FG_OK;
  if (m->all_cap < (size_t)n) {
    mlp_free_samples(m);
    hipError_t e = hipMalloc((void **)&m->Xall, (size_t)n * din * 4);
    if (e == hipSuccess) e = hipMalloc((void **)&m->Tall, (size_t)n * dout * 4);
    if (e != hipSuccess) mlp_free_samples(m);
    FG_HIP(e);
    m->all_cap = (size_t)n;
  }
  if (m->loss_cap < steps) {
    if (m->loss) (void)hipFree(m->loss);
    m->loss = nullptr;
    m->loss_cap = 0;
    if (hipMalloc((void **)&m->loss, (size_t)steps * 4) != hipSuccess)
      st = FG_E_NOMEM;
    else
      m->loss_cap = steps;
  }
  if (!st && (hipMemcpyAsync(m->Xall, x, (size_t)n * din * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess ||
              hipMemcpyAsync(m->Tall, t, (size_t)n * dout * 4, hipMemcpyHostToDevice, m->stream) != hipSuccess))
    st = FG_E_HIP;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  const int nb = n / batch;
  for (int s = 0; s < steps && !st; s++) {
    const int q = s % nb;
    const float *xs = m->Xall + (size_t)q * batch * din, *ts = m->Tall + (size_t)q * batch * dout;
    // (counted once its gradients stand, or, with both in one, its update)
    const float taken = (float)(m->step + 1), c1 = 1.0f - powf(b1, taken), c2 = 1.0f - powf(b2, taken);
    if (m->net) {
      const adam_args adam = {lr, b1, b2, eps, c1, c2};
      if ((st = mlp_rows(m, xs, ts, batch, s > 0 ? m->loss + s - 1 : nullptr))) break;
      if (!(st = mlp_weights(m, ts, batch, &adam))) m->step++;
      continue;
    }
    if (hipMemcpyAsync(m->X, xs, (size_t)batch * din * 4, hipMemcpyDeviceToDevice, m->stream) != hipSuccess ||
        hipMemcpyAsync(m->T, ts, (size_t)batch * dout * 4, hipMemcpyDeviceToDevice, m->stream) != hipSuccess) {
      st = FG_E_HIP;
      break;
    }
    if ((st = mlp_forward(m, batch))) break;
    if ((st = mlp_backward(m, batch, m->loss + s))) break;
    m->step++;
    hipLaunchKernelGGL(k_adam, dim3(fg_blocks(m->nparam, 256)), dim3(256), 0, m->stream, m->p, m->g, m->m, m->v,
                       m->pb, m->nparam, lr, b1, b2, eps, c1, c2);
    if (hipGetLastError() != hipSuccess) st = FG_E_HIP;
  }
  if (!st && m->net) st = mlp_loss(m, batch, m->loss + steps - 1);
  if (!st && losses &&
      hipMemcpyAsync(losses, m->loss, (size_t)steps * 4, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    st = FG_E_HIP;
  (void)hipStreamSynchronize(m->stream);
  if (m->all_cap * (size_t)(din + dout) * 4 > MLP_KEEP_BYTES) mlp_free_samples(m);
  if (st && st != FG_E_NOMEM) fg_set_error("fg_mlp_train: HIP error");
  return st;
}

// C[M x N] = A[M x K] B[K x N] with A, B rounded to BF16 and FP32
// accumulation (the layer GEMM on its own, for tests and tools)
extern "C" fg_status fg_bf16_gemm(const float *A, const float *B, int M, int N, int K, float *C) {
  if (!A || !B || !C || M < 1 || N < 1 || K < 1) return FG_E_INVALID;
  float *dA = nullptr, *dB = nullptr, *dC = nullptr;
  bf16_t *bA = nullptr, *bB = nullptr;
  hipStream_t st = nullptr;
  fg_status rc = FG_OK;
  const size_t nA = (size_t)M * K, nB = (size_t)K * N, nC = (size_t)M * N;
  if (hipStreamCreate(&st) != hipSuccess || hipMalloc((void **)&dA, nA * 4) != hipSuccess ||
      hipMalloc((void **)&dB, nB * 4) != hipSuccess || hipMalloc((void **)&dC, nC * 4) != hipSuccess ||
      hipMalloc((void **)&bA, nA * 2) != hipSuccess || hipMalloc((void **)&bB, nB * 2) != hipSuccess ||
      hipMemcpyAsync(dA, A, nA * 4, hipMemcpyHostToDevice, st) != hipSuccess ||
      hipMemcpyAsync(dB, B, nB * 4, hipMemcpyHostToDevice, st) != hipSuccess) {
    rc = FG_E_HIP;
  } else {
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(fg_blocks((long)nA, 256)), dim3(256), 0, st, dA, bA, (long)nA);
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(fg_blocks((long)nB, 256)), dim3(256), 0, st, dB, bB, (long)nB);
    gemm_args g{};
    g.A = bA;
    g.sai = K;
    g.sak = 1;
    g.B = bB;
    g.sbk = N;
    g.sbj = 1;
    g.M = M;
    g.N = N;
    g.K = K;
    g.mode = EPI_STORE;
    g.C = dC;
    g.ldc = N;
    hipLaunchKernelGGL(k_gemm_bf16, dim3((N + GT - 1) / GT, (M + GT - 1) / GT), dim3(256), 0, st, g);
    if (hipGetLastError() != hipSuccess ||
        hipMemcpyAsync(C, dC, nC * 4, hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      rc = FG_E_HIP;
  }
  if (rc) fg_set_error("fg_bf16_gemm: HIP error");
  void *ptrs[] = {dA, dB, dC, bA, bB};
  for (void *q : ptrs)
    if (q) (void)hipFree(q);
  if (st) (void)hipStreamDestroy(st);
  return rc;
}
