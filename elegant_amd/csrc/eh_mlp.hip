/*
 * ehd_mlp.hip - a small multilayer perceptron trained and evaluated on the GPU.
 *
 * It proposes dynamic-aperture boundaries: inputs are a test particle's start
 * (x0, y0, delta) and the lattice variant's error summary, the output is the
 * probability that the particle survives.  FP32 throughout; FP64 tracking of
 * the proposed points decides the answer.
 *
 * Kernels: one LDS-tiled FP32 GEMM (64x64 output tile per 256-thread
 * workgroup, 4x4 per thread, K staged in 16-wide slabs) with transpose
 * variants for the forward pass (Y = X W^T + b), the data gradient
 * (dX = dY W) and the weight gradient (dW = dY^T X); fused bias/ReLU
 * epilogues; the loss gradient of binary cross-entropy on logits; Adam.
 */
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include "../../include/elegant_hip.h"
#include "eh_device.h"
#include "ehd_internal.h"

#define TM 64
#define TN 64
#define TK 16

/* C[M,N] = op(A) op(B) (+ bias[N]) (ReLU), row-major.
 * TA = 0: A is [M,K] (lda);  TA = 1: A is [K,M] (lda), use A^T.
 * TB = 0: B is [K,N] (ldb);  TB = 1: B is [N,K] (ldb), use B^T. */
template <int TA, int TB>
__global__ void __launch_bounds__(256) gemm_f32(const float *__restrict__ A, const float *__restrict__ B,
                                                float *__restrict__ C, const float *__restrict__ bias, int M, int N,
                                                int K, int lda, int ldb, int ldc, int relu, int accumulate,
                                                int kslice, int64_t c_slice) {
  __shared__ float As[TK][TM + 4];
  __shared__ float Bs[TK][TN + 4];
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  /* split K: slice z covers [z kslice, (z+1) kslice) and writes its partial
   * product to C + z c_slice */
  const int kb = blockIdx.z * kslice, ke = kb + kslice < K ? kb + kslice : K;
  C += blockIdx.z * c_slice;
  float acc[4][4] = {{0}};
  for (int k0 = kb; k0 < ke; k0 += TK) {
    for (int e = threadIdx.x; e < TK * TM; e += 256) {
      int kk = e / TM, mm = e % TM;
      int gm = m0 + mm, gk = k0 + kk;
      float v = 0.f;
      if (gm < M && gk < ke)
        v = TA ? A[(size_t)gk * lda + gm] : A[(size_t)gm * lda + gk];
      As[kk][mm] = v;
    }
    for (int e = threadIdx.x; e < TK * TN; e += 256) {
      int kk = e / TN, nn = e % TN;
      int gn = n0 + nn, gk = k0 + kk;
      float v = 0.f;
      if (gn < N && gk < ke)
        v = TB ? B[(size_t)gn * ldb + gk] : B[(size_t)gk * ldb + gn];
      Bs[kk][nn] = v;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TK; kk++) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++)
        a[i] = As[kk][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; j++)
        b[j] = Bs[kk][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
          acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int gm = m0 + ty * 4 + i;
    if (gm >= M)
      continue;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int gn = n0 + tx * 4 + j;
      if (gn >= N)
        continue;
      float v = acc[i][j];
      if (bias)
        v += bias[gn];
      if (relu)
        v = v > 0.f ? v : 0.f;
      float *dst = &C[(size_t)gm * ldc + gn];
      *dst = accumulate ? *dst + v : v;
    }
  }
}

/* out[i] = sum over s of part[s][i], s in order (deterministic split-K) */
__global__ void reduce_slices(const float *__restrict__ part, int S, int64_t count, float *out) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count)
    return;
  float v = 0.f;
  for (int s = 0; s < S; s++)
    v += part[(int64_t)s * count + i];
  out[i] = v;
}

/* partial column sums of dz[rows, cols]: slice blockIdx.y of rowsl rows,
 * 64 columns per workgroup, 4 row lanes per column combined in LDS */
__global__ void __launch_bounds__(256) col_sum_part(const float *__restrict__ dz, float *part, int rows, int cols,
                                                    int rowsl) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), lane = threadIdx.x >> 6;
  const int r0 = blockIdx.y * rowsl, r1 = r0 + rowsl < rows ? r0 + rowsl : rows;
  float v = 0.f;
  if (c < cols)
    for (int r = r0 + lane; r < r1; r += 4)
      v += dz[(size_t)r * cols + c];
  red[lane][threadIdx.x & 63] = v;
  __syncthreads();
  if (lane == 0 && c < cols)
    part[(size_t)blockIdx.y * cols + c] = ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) +
                                          red[3][threadIdx.x];
}

/* the minibatch from the resident training set: rows perm[0..B) of X, y */
__global__ void gather_batch(const float *__restrict__ X, const float *__restrict__ y,
                             const int32_t *__restrict__ perm, int B, int nin, float *xb, float *yb) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (int64_t)B * nin)
    return;
  const int i = (int)(e / nin), k = (int)(e % nin);
  const int32_t j = perm[i];
  xb[e] = X[(size_t)j * nin + k];
  if (k == 0)
    yb[i] = y[j];
}

/* acc[0] += the batch loss (sum of the block partials in order) */
__global__ void loss_accumulate(const float *__restrict__ part, int nb, float *acc) {
  if (threadIdx.x != 0 || blockIdx.x != 0)
    return;
  float s = 0.f;
  for (int k = 0; k < nb; k++)
    s += part[k];
  acc[0] += s;
}

/* dZ *= (H > 0): ReLU derivative with the layer's output H */
__global__ void relu_mask(float *dz, const float *h, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && !(h[i] > 0.f))
    dz[i] = 0.f;
}

/* binary cross-entropy on logits, mean over the batch: loss partials and dz = (sigmoid(z) - y)/B */
__global__ void bce_grad(const float *z, const float *y, float *dz, float *loss_part, int B) {
  __shared__ float red[256];
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  float l = 0.f;
  if (i < B) {
    float zi = z[i], yi = y[i];
    float sp = zi > 0 ? zi + log1pf(expf(-zi)) : log1pf(expf(zi)); /* softplus */
    l = sp - yi * zi;
    float sg = 1.f / (1.f + expf(-zi));
    dz[i] = (sg - yi) / (float)B;
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
      red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0)
    loss_part[blockIdx.x] = red[0] / (float)B;
}

__global__ void sigmoid_k(const float *z, float *p, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = 1.f / (1.f + expf(-z[i]));
}

__global__ void adam_k(float *w, const float *g, float *m, float *v, int64_t n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n)
    return;
  float gi = g[i];
  float mi = b1 * m[i] + (1.f - b1) * gi;
  float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

/* ---- the fused path: hidden <= 256, inputs <= 256 ----
 *
 * A training step is three kernels: mlp_rows takes 16 samples per workgroup
 * through all layers and back (activations stay in LDS; they and the layers'
 * gradients are also written out), mlp_wgrad contracts those over the batch
 * into partial gradients, mlp_update sums the partials in order and applies
 * Adam.  The products run on the matrix cores in FP32 (v_mfma_f32_16x16x4f32).
 *
 * The results are the general path's bit for bit: one such instruction is
 * four FMAs in the order of its contraction index, each rounded, so every sum
 * is taken in the order that gemm_f32, col_sum_part, bce_grad and
 * reduce_slices take it (ascending from zero, the batch in ksplit's slices,
 * column sums in slices of 64 rows).  Adam divides by the root of the squared
 * gradient, so another order of a sum shows in the weights: 1.4e-3 of their
 * norm after 64 steps of 4096 samples.
 *
 * What bounds it: 3.3 GFLOP per step of 4096 samples is 22 us at the 150
 * TFLOP/s of a large FP32 product; a step takes 65 us (38 + 19 + 8), the
 * general path's 35 launches 470.  mlp_rows reads 1.3 MB of weights per
 * workgroup from L2, all workgroups in the same order (with the order of the
 * sums free it took 35).
 *
 * Layouts.  HS = hidden rounded up to 64, XS = inputs rounded up to 64; padded
 * weights are zero, so padded activations and gradients are zero.  A
 * contraction is cut into chunks of 16, product m of the four that a chunk
 * takes has elements 4 m .. 4 m + 3 (element 4 m + g in the lanes l / 16 = g),
 * and a lane loads its elements of all four products as one 16-byte load.  So
 * element k of a chunk is kept at place mlp_place(k) of it: in the weights,
 * one 1 KB block per tile of 16 outputs and chunk (wf for the forward
 * products, wb for the ones going back), and in the rows of activations and
 * gradients, in LDS and in memory. */
typedef float f4 __attribute__((ext_vector_type(4)));

static __host__ __device__ __forceinline__ int mlp_place(int k) { return (k & ~15) | (k & 3) << 2 | (k >> 2 & 3); } /* its own inverse */

struct mlp_net {
  const float *wf[3], *wb[3]; /* wb[0] unused */
  const float *bias[3], *w4, *b4;
  int nin, hidden, xc, xs;    /* xc: input chunks of 16 */
};

struct mlp_batch {
  const float *X, *y;
  const int32_t *perm;        /* sample indices, or NULL */
  float *xb, *h[3], *dz[3];   /* [rows][xs] and [rows][HS] */
  float *dz4, *lrow;          /* per row: the output's gradient and the loss */
  float *prob;                /* prediction */
  int rows;
};

/* acc[mt][t] += rows of a (LDS, stride lda) x tile wave + 4 t of wt, over kc
 * chunks, D of them in flight: a workgroup is alone on its CU, one wave per
 * SIMD. */
template <int NT, int MT, int D>
static __device__ __forceinline__ void rows_mm(const float *a, int lda, const float *__restrict__ wt, int kc,
                                               f4 (&acc)[MT][NT]) {
  int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  /* opaque: the addresses of every layer's chunks are otherwise computed ahead
   * of the loop over rows and spilled */
  asm volatile("" : "+v"(lane));
  const float *ar = a + (lane & 15) * lda + 4 * (lane >> 4);
  const float *w0 = wt + (size_t)wave * kc * 256 + 4 * lane;
  f4 b[D][NT];
#pragma unroll
  for (int u = 0; u < D; u++)
#pragma unroll
    for (int t = 0; t < NT; t++)
      b[u][t] = *(const f4 *)(w0 + ((size_t)4 * t * kc + (u < kc ? u : 0)) * 256);
  f4 av[2][MT]; /* the next chunk's rows are read while a chunk's products run */
#pragma unroll
  for (int m = 0; m < MT; m++)
    av[0][m] = *(const f4 *)(ar + 16 * m * lda);
  for (int c = 0; c < kc; c += D) {
#pragma unroll
    for (int u = 0; u < D; u++) {
      const int ca = c + u + 1 < kc ? c + u + 1 : 0, cl = c + u + D < kc ? c + u + D : 0; /* rows, weights to load */
#pragma unroll
      for (int m = 0; m < MT; m++)
        av[D > 1 ? (u + 1) & 1 : 1][m] = *(const f4 *)(ar + 16 * m * lda + 16 * ca);
#pragma unroll
      for (int k = 0; k < 4; k++)
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int t = 0; t < NT; t++)
            acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[D > 1 ? u & 1 : 0][m][k], b[u][t][k], acc[m][t], 0, 0, 0);
#pragma unroll
      for (int t = 0; t < NT; t++)
        b[u][t] = *(const f4 *)(w0 + ((size_t)4 * t * kc + cl) * 256);
      if (D == 1)
#pragma unroll
        for (int m = 0; m < MT; m++)
          av[0][m] = av[1][m];
    }
  }
}

/* rows [0, 16 MT) of an LDS buffer to global rows r0.. of width HS, as far as
 * rows exist */
template <int HS>
static __device__ __forceinline__ void rows_out(const float *a, int lda, float *g, int r0, int nr, int rows) {
  for (int e = threadIdx.x; e < nr * (HS / 4); e += 256) {
    const int r = e / (HS / 4), c = e % (HS / 4) * 4;
    if (r0 + r < rows)
      *(f4 *)(g + (size_t)(r0 + r) * HS + c) = *(const f4 *)(a + r * lda + c);
  }
}

/* TRAIN: forward, loss, backward of 16 rows at a time (MT = 1); else the
 * probabilities of 16 MT rows.  Workgroups stride over the batch. */
template <int NT, int MT, bool TRAIN>
__global__ void __launch_bounds__(256, TRAIN ? 1 : 2) mlp_rows(mlp_net N, mlp_batch Q) {
  constexpr int HS = 64 * NT, R = 16 * MT, LD = HS + 4, LX = 260;
  __shared__ float sx[TRAIN ? R * LX : R * (LX > LD ? LX : LD)];
  __shared__ float sh[TRAIN ? 3 : 1][R * LD];
  __shared__ float sd[R], sy[R];
  __shared__ __attribute__((aligned(16))) float sw[HS]; /* the last layer's weights, placed */
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  /* biases and the last layer's weights, loaded once and together (indices
   * clamped, no load behind a branch): each would cost a trip to L2 where it
   * is used */
  float bias[3][NT];
  const int pt = mlp_place(tid), pc = mlp_place(lane & 15);
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int t = 0; t < NT; t++) {
      const int c = 16 * (wave + 4 * t) + (lane & 15);
      bias[l][t] = N.bias[l][c < N.hidden ? c : 0];
    }
  float b4 = N.b4[0], w4c = N.w4[pt < N.hidden ? pt : 0];
  w4c = pt < N.hidden ? w4c : 0.f;
  if (tid < HS)
    sw[tid] = w4c;
#pragma unroll
  for (int l = 0; l < 3; l++)
#pragma unroll
    for (int t = 0; t < NT; t++)
      bias[l][t] = 16 * (wave + 4 * t) + (lane & 15) < N.hidden ? bias[l][t] : 0.f;
  for (int r0 = blockIdx.x * R; r0 < Q.rows; r0 += gridDim.x * R) {
    /* the rows' inputs, zero beyond the net's and beyond the batch: 16 threads
     * per row, the sample's index first, then its inputs together */
    {
      const int q = tid & 15, xw = TRAIN ? N.xs : 16 * N.xc;
      int64_t j[MT];
#pragma unroll
      for (int m = 0; m < MT; m++) {
        const int r = r0 + 16 * m + (tid >> 4), rc = r < Q.rows ? r : Q.rows - 1;
        j[m] = Q.perm ? Q.perm[rc] : rc;
      }
      float yv = 0.f;
      if (TRAIN)
        yv = Q.y[j[0]];
      for (int k0 = 0; k0 < xw; k0 += 64) {
        float v[MT][4];
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int k = k0 + q + 16 * u;
            v[m][u] = Q.X[j[m] * N.nin + (k < N.nin ? k : N.nin - 1)];
          }
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const int k = k0 + q + 16 * u, r = 16 * m + (tid >> 4);
            const bool on = r0 + r < Q.rows && k < N.nin;
            if (k < xw) {
              sx[r * LX + mlp_place(k)] = on ? v[m][u] : 0.f;
              if (TRAIN && r0 + r < Q.rows)
                Q.xb[(size_t)(r0 + r) * N.xs + mlp_place(k)] = on ? v[m][u] : 0.f;
            }
          }
      }
      if (TRAIN && q == 0)
        sy[tid >> 4] = yv;
    }
    __syncthreads();
#pragma unroll
    for (int l = 0; l < 3; l++) {
      /* prediction alternates between two buffers */
      const float *in = l == 0 ? sx : (TRAIN ? sh[l - 1] : (l == 1 ? sh[0] : sx));
      float *out = TRAIN ? sh[l] : (l == 1 ? sx : sh[0]);
      const int lin = l == 0 ? LX : LD;
      f4 acc[MT][NT];
#pragma unroll
      for (int m = 0; m < MT; m++)
#pragma unroll
        for (int t = 0; t < NT; t++)
          acc[m][t] = (f4){0.f, 0.f, 0.f, 0.f};
      if (l == 0)
        rows_mm<NT, MT, 1>(in, lin, N.wf[l], N.xc, acc);
      else
        rows_mm<NT, MT, 4>(in, lin, N.wf[l], HS / 16, acc);
#pragma unroll
      for (int t = 0; t < NT; t++) {
        const int c = 16 * (wave + 4 * t) + pc;
        const float b = bias[l][t];
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
          for (int i = 0; i < 4; i++) {
            const float v = acc[m][t][i] + b;
            out[(16 * m + 4 * (lane >> 4) + i) * LD + c] = v > 0.f ? v : 0.f;
          }
      }
      __syncthreads();
      if (TRAIN)
        rows_out<HS>(sh[l], LD, Q.h[l], r0, R, Q.rows);
    }
    /* the last layer: a thread per row, as its sum has one order */
    const float *h3 = TRAIN ? sh[2] : sh[0];
    if (tid < R) {
      const float *h = h3 + tid * LD;
      float v = 0.f;
#pragma unroll 2
      for (int c = 0; c < HS; c += 16) {
        f4 a[4], w[4];
#pragma unroll
        for (int g = 0; g < 4; g++) {
          a[g] = *(const f4 *)(h + c + 4 * g);
          w[g] = *(const f4 *)(sw + c + 4 * g);
        }
#pragma unroll
        for (int k = 0; k < 16; k++)
          v = fmaf(a[k & 3][k >> 2], w[k & 3][k >> 2], v);
      }
      const int r = r0 + tid;
      const float z = v + b4;
      if (!TRAIN) {
        if (r < Q.rows)
          Q.prob[r] = 1.f / (1.f + expf(-z));
      } else {
        float d = 0.f;
        if (r < Q.rows) {
          const float yi = sy[tid];
          const float sp = z > 0 ? z + log1pf(expf(-z)) : log1pf(expf(z)); /* softplus */
          Q.lrow[r] = sp - yi * z;
          d = (1.f / (1.f + expf(-z)) - yi) / (float)Q.rows;
          Q.dz4[r] = d;
        }
        sd[tid] = d;
      }
    }
    __syncthreads();
    if (TRAIN) {
      /* dz3 in place of h3, then dz2 in place of h2, dz1 of h1 */
      if (tid < HS)
#pragma unroll
        for (int r = 0; r < R; r++)
          sh[2][r * LD + tid] = sh[2][r * LD + tid] > 0.f ? fmaf(sd[r], w4c, 0.f) : 0.f;
      __syncthreads();
#pragma unroll
      for (int l = 2; l >= 0; l--) {
        rows_out<HS>(sh[l], LD, Q.dz[l], r0, R, Q.rows);
        if (l > 0) {
          f4 acc[MT][NT];
#pragma unroll
          for (int m = 0; m < MT; m++)
#pragma unroll
            for (int t = 0; t < NT; t++)
              acc[m][t] = (f4){0.f, 0.f, 0.f, 0.f};
          rows_mm<NT, MT, 4>(sh[l], LD, N.wb[l], HS / 16, acc);
#pragma unroll
          for (int t = 0; t < NT; t++) {
            const int c = 16 * (wave + 4 * t) + pc;
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
              for (int i = 0; i < 4; i++) {
                float *h = &sh[l - 1][(16 * m + 4 * (lane >> 4) + i) * LD + c];
                *h = *h > 0.f ? acc[m][t][i] : 0.f;
              }
          }
          __syncthreads();
        }
      }
    }
    __syncthreads();
  }
}

/* The partial gradients: how the batch is cut for each layer (as ksplit cuts
 * it for the general path, the column sums in slices of 64 rows) and where the
 * partials lie. */
struct mlp_cut {
  int hidden, nin, hs, xs;
  int S[4], rows[4];          /* slices of the weights' contractions and their rows */
  int rs, nb;                 /* slices of 64 rows; blocks of 256 rows of the loss */
  float *pw[4];               /* [S][hs][xs or hs] of the tiled layers, [S][hs] of the last */
  float *pb[4];               /* bias gradients [rs][hs], of the last layer [rs] */
  float *loss;                /* [nb] */
  int first[4], wgs[3];       /* first workgroup of the tiled layers' parts, and of what follows; workgroups per slice */
  int nbias, nlast;           /* workgroups of the column sums and of the last layer's weights */
};

/* Workgroups [first[l], first[l + 1]) take layer 2 - l: partial weight
 * gradients dW[n][k] = sum over a slice of the batch of dz[b][n] in[b][k].  A
 * wave takes a tile of 64 x 32 (8 products of 16 x 16) and four rows of the
 * batch per step, its operands straight from memory, 16 and 8 bytes per load:
 * tile row 4 i + rt is row i of product rt, so a lane's elements feed as many
 * products.  The 32 tiles and 16 slices of a layer of 256 make 512 waves, two
 * such layers one per SIMD of the device (with tiles of 64 x 64 half of them
 * would be idle).  The tiles of one slice read the same rows, so a slice stays
 * on one XCD (workgroups go round the 8 of them).  The workgroups after them
 * make the column sums, the last layer's weight gradients and the loss. */
typedef float f2 __attribute__((ext_vector_type(2)));
#define WG_D 8
__global__ void __launch_bounds__(256, 2) mlp_wgrad(mlp_batch Q, mlp_cut C) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  int blk = (int)blockIdx.x;
  if (blk < C.first[3]) {
    const int l = blk < C.first[1] ? 2 : (blk < C.first[2] ? 1 : 0);
    const int hs = C.hs, ks = l ? hs : C.xs, kn = ((l ? C.hidden : C.nin) + 31) / 32;
    const int tiles = (C.hidden + 63) / 64 * kn;
    blk -= C.first[2 - l];
    const int j = blk / 8, slice = blk % 8 + 8 * (j / C.wgs[l]), tile = 4 * (j % C.wgs[l]) + wave;
    if (slice >= C.S[l] || tile >= tiles)
      return;
    const int n0 = tile / kn * 64, k0 = tile % kn * 32;
    const int b0 = slice * C.rows[l], b1 = b0 + C.rows[l] < Q.rows ? b0 + C.rows[l] : Q.rows;
    const int g = lane >> 4, ca = 4 * (lane & 15), cb = 2 * (lane & 15), last = Q.rows - 1;
    const float *pa = Q.dz[l] + n0 + ca, *pb = (l ? Q.h[l - 1] : Q.xb) + k0 + cb;
    f4 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int k = 0; k < 2; k++)
        acc[i][k] = (f4){0.f, 0.f, 0.f, 0.f};
    /* WG_D steps' operands in flight; rows past the slice count as zero */
    f4 av[WG_D];
    f2 bv[WG_D];
#pragma unroll
    for (int u = 0; u < WG_D; u++) {
      const int r = b0 + 4 * u + g, rc = r < last ? r : last;
      av[u] = *(const f4 *)(pa + (size_t)rc * hs);
      bv[u] = *(const f2 *)(pb + (size_t)rc * ks);
    }
    for (int b = b0; b < b1; b += 4 * WG_D) {
#pragma unroll
      for (int u = 0; u < WG_D; u++) {
        f4 a = av[u];
        f2 v = bv[u];
        if (b + 4 * u + g >= b1) {
          a = (f4){0.f, 0.f, 0.f, 0.f};
          v = (f2){0.f, 0.f};
        }
        const int r = b + 4 * WG_D + 4 * u + g, rc = r < last ? r : last;
        av[u] = *(const f4 *)(pa + (size_t)rc * hs);
        bv[u] = *(const f2 *)(pb + (size_t)rc * ks);
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int k = 0; k < 2; k++)
            acc[i][k] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], v[k], acc[i][k], 0, 0, 0);
      }
    }
    float *o = C.pw[l] + (size_t)slice * hs * ks;
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const f2 v = {acc[i][0][r], acc[i][1][r]};
        *(f2 *)(o + (size_t)(n0 + 4 * (4 * g + r) + i) * ks + k0 + cb) = v;
      }
    return;
  }
  blk -= C.first[3];
  __shared__ float red[256];
  if (blk < C.nbias) {
    /* column sums of 64 rows and 64 columns: four interleaved rows */
    const int cg = C.hs / 64, slice = blk / (3 * cg), l = blk / cg % 3, c = blk % cg * 64 + lane;
    const int r0 = slice * 64, r1 = r0 + 64 < Q.rows ? r0 + 64 : Q.rows;
    const float *p = Q.dz[l] + c;
    float s = 0.f;
#pragma unroll 16
    for (int r = r0 + wave; r < r1; r += 4)
      s += p[(size_t)r * C.hs];
    red[tid] = s;
    __syncthreads();
    if (wave == 0)
      C.pb[l][(size_t)slice * C.hs + c] = ((red[lane] + red[64 + lane]) + red[128 + lane]) + red[192 + lane];
    return;
  }
  blk -= C.nbias;
  if (blk < C.nlast) {
    const int r0 = blk * C.rows[3], r1 = r0 + C.rows[3] < Q.rows ? r0 + C.rows[3] : Q.rows;
    if (tid >= C.hs)
      return;
    const float *p = Q.h[2] + tid;
    float s = 0.f;
#pragma unroll 8
    for (int r = r0; r < r1; r++)
      s = fmaf(Q.dz4[r], p[(size_t)r * C.hs], s);
    C.pw[3][(size_t)blk * C.hs + tid] = s;
    return;
  }
  blk -= C.nlast;
  if (blk < C.nb) {
    /* the loss of 256 rows, in a tree */
    const int r = blk * 256 + tid;
    red[tid] = r < Q.rows ? Q.lrow[r] : 0.f;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
      if (tid < w)
        red[tid] += red[tid + w];
      __syncthreads();
    }
    if (tid == 0)
      C.loss[blk] = red[0] / (float)Q.rows;
    return;
  }
  blk -= C.nb;
  /* the output gradient's sums over 64 rows */
  const int slice = blk * 64 + lane, r1 = slice * 64 + 64 < Q.rows ? slice * 64 + 64 : Q.rows;
  float s = 0.f;
  for (int r = slice * 64 + wave; r < r1; r += 4)
    s += Q.dz4[r];
  red[tid] = s;
  __syncthreads();
  if (wave == 0 && slice < C.rs)
    C.pb[3][slice] = ((red[lane] + red[64 + lane]) + red[128 + lane]) + red[192 + lane];
}

struct mlp_param {
  float *w, *g, *m, *v;       /* parameters, gradients out (or NULL), Adam moments */
  float *wf[3], *wb[3];
  int64_t woff[4], boff[4];
  int nin, hidden, hs, xs, xc;
  float lr, b1, b2, eps, c1, c2;
};

/* where weight (n, k) of layer l lies in the tiled copies */
static __device__ __forceinline__ void mlp_tiles(const mlp_param &P, int l, int n, int k, float w) {
  const int kc = l == 0 ? P.xc : P.hs / 16;
  P.wf[l][((size_t)(n / 16) * kc + k / 16) * 256 + 4 * ((n % 16) + 16 * (k % 4)) + k % 16 / 4] = w;
  if (l > 0)
    P.wb[l][((size_t)(k / 16) * (P.hs / 16) + n / 16) * 256 + 4 * ((k % 16) + 16 * (n % 4)) + n % 16 / 4] = w;
}

static __device__ __forceinline__ float mlp_step(const mlp_param &P, int64_t p, float gi) {
  const float mi = P.b1 * P.m[p] + (1.f - P.b1) * gi;
  const float vi = P.b2 * P.v[p] + (1.f - P.b2) * gi * gi;
  P.m[p] = mi;
  P.v[p] = vi;
  const float w = P.w[p] - P.lr * (mi / P.c1) / (sqrtf(vi / P.c2) + P.eps);
  P.w[p] = w;
  return w;
}

/* layer, row and column of weight i of the three tiled layers */
static __device__ __forceinline__ int mlp_where(const mlp_param &P, int64_t i, int &n, int &k) {
  const int64_t w0 = (int64_t)P.hidden * P.nin, w1 = (int64_t)P.hidden * P.hidden;
  const int l = i < w0 ? 0 : (i < w0 + w1 ? 1 : 2), in = l ? P.hidden : P.nin;
  const int q = (int)(i - (l == 0 ? 0 : (l == 1 ? w0 : w0 + w1)));
  n = q / in;
  k = q % in;
  return l;
}

/* the tiled copies from the parameters, with zeros as their padding: tiles
 * holds wf[0], wf[1], wb[1], wf[2], wb[2] */
__global__ void __launch_bounds__(256) mlp_retile(mlp_param P, float *tiles, int len) {
  const int i = (int)(blockIdx.x * 256 + threadIdx.x), w0 = P.hs * 16 * P.xc, w1 = P.hs * P.hs;
  if (i >= len)
    return;
  const int b = i < w0 ? 0 : 1 + (i - w0) / w1, j = i < w0 ? i : (i - w0) % w1; /* which of the five, and where in it */
  const int l = (b + 1) / 2, kc = l ? P.hs / 16 : P.xc, in = l ? P.hidden : P.nin;
  const int lane = j % 256 / 4, r = j / 256 / kc * 16 + lane % 16, c = j / 256 % kc * 16 + j % 4 * 4 + lane / 16;
  const int back = l && b % 2 == 0, n = back ? c : r, k = back ? r : c;
  tiles[i] = n < P.hidden && k < in ? P.w[P.woff[l] + (int64_t)n * in + k] : 0.f;
}

__global__ void mlp_zero(float *p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n)
    p[i] = 0.f;
}

/* p[0] + p[stride] + ... from zero, in order, n terms */
static __device__ __forceinline__ float sum_in_order(const float *p, int n, size_t stride) {
  float s = 0.f;
  int u = 0;
  for (; u + 8 <= n; u += 8) {
    float t[8];
#pragma unroll
    for (int e = 0; e < 8; e++)
      t[e] = p[(size_t)(u + e) * stride];
#pragma unroll
    for (int e = 0; e < 8; e++)
      s += t[e];
  }
  for (; u < n; u++)
    s += p[(size_t)u * stride];
  return s;
}

/* The partial gradients summed in order, then Adam (or, with P.g, the
 * gradients themselves): the first nwb workgroups take the weights of the
 * tiled layers, the others the rest, 64 entries each so that their chains of
 * sums run beside each other.  The loss is added to *loss. */
__global__ void __launch_bounds__(256) mlp_update(mlp_param P, mlp_cut C, int64_t nw, int nwb, float *loss) {
  if ((int)blockIdx.x < nwb) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= nw)
      return;
    int n, k;
    const int l = mlp_where(P, i, n, k);
    const int ks = l ? P.hs : P.xs;
    const float g = sum_in_order(C.pw[l] + (size_t)mlp_place(n) * ks + mlp_place(k), C.S[l], (size_t)P.hs * ks);
    const int64_t p = P.woff[l] + (int64_t)n * (l ? P.hidden : P.nin) + k;
    if (P.g)
      P.g[p] = g;
    else
      mlp_tiles(P, l, n, k, mlp_step(P, p, g));
    return;
  }
  const int c = ((int)blockIdx.x - nwb) * 64 + (int)threadIdx.x, l = c / P.hs, e = c % P.hs;
  if (threadIdx.x >= 64 || c > 4 * P.hs + 1)
    return;
  if (c == 4 * P.hs + 1) {
    *loss += sum_in_order(C.loss, C.nb, 1);
    return;
  }
  float g;
  int64_t p;
  if (c == 4 * P.hs) {
    g = sum_in_order(C.pb[3], C.rs, 1);
    p = P.boff[3];
  } else {
    if (e >= P.hidden)
      return;
    g = l < 3 ? sum_in_order(C.pb[l] + mlp_place(e), C.rs, P.hs) : sum_in_order(C.pw[3] + mlp_place(e), C.S[3], P.hs);
    p = (l < 3 ? P.boff[l] : P.woff[3]) + e;
  }
  if (P.g)
    P.g[p] = g;
  else
    mlp_step(P, p, g);
}

/* ------------------------------------------------------------ host side */

#define MLP_LAYERS 4

struct ehd_mlp {
  ehd_dev *d;
  int32_t nin, hidden;
  int32_t in_dim[MLP_LAYERS], out_dim[MLP_LAYERS];
  int64_t woff[MLP_LAYERS], boff[MLP_LAYERS], nparams;
  float *params, *grads, *adam_m, *adam_v;
  float *act[MLP_LAYERS + 1]; /* act[0] = input, act[l+1] = output of layer l */
  float *dact[MLP_LAYERS + 1];
  float *labels, *loss_part;
  int32_t cap;
  int64_t step;
  float *part;           /* split-K and column-sum partials */
  int64_t part_cap;
  float *Xd, *yd;        /* the resident training set */
  int32_t *permd;        /* its sample order, epochs x n */
  float *eloss;          /* per-epoch loss sums */
  int64_t data_cap, y_cap, perm_cap, eloss_cap;
  /* the fused path */
  int fused, hs, xs, xc;
  int tiles_stale;       /* the parameters were set: wf, wb to be filled */
  float *tiles;          /* wf[0], wf[1], wb[1], wf[2], wb[2] */
  float *fbuf;           /* xb, h[3], dz[3] for fcap rows */
  int64_t fcap;
  float *fpart;          /* partial gradients and losses */
  int64_t fpart_cap;
  float *floss;
  float *pin[2], *pout[2]; /* prediction: two chunks of inputs and of probabilities, the second of a call of more */
  int64_t pin_cap[2], pout_cap[2];
  hipStream_t pstream;   /* the copies of such a call */
  hipEvent_t pev[4];
  char msg[256];
};

/* two row tiles per workgroup (half the weight reads) once one each fills
 * the device twice */
template <int NT> static void rows_predict(hipStream_t st, const mlp_net &N, const mlp_batch &Q) {
  if (Q.rows > 16 * 512)
    hipLaunchKernelGGL((mlp_rows<NT, 2, false>), dim3((Q.rows + 31) / 32), dim3(256), 0, st, N, Q);
  else
    hipLaunchKernelGGL((mlp_rows<NT, 1, false>), dim3((Q.rows + 15) / 16), dim3(256), 0, st, N, Q);
}

extern "C" {

static int mlp_fail(ehd_mlp *m, hipError_t e, const char *what) {
  snprintf(m->d->msg, sizeof(m->d->msg), "%s: %s", what, hipGetErrorString(e));
  return EH_ERR_HIP;
}

#define MCHK(call)                                                                                                     \
  do {                                                                                                                 \
    hipError_t e_ = (call);                                                                                            \
    if (e_ != hipSuccess)                                                                                              \
      return mlp_fail(m, e_, #call);                                                                                   \
  } while (0)

/* S > 1 splits K into S slices whose partial products go to C + z c_slice */
static void launch_gemm_s(ehd_mlp *m, int ta, int tb, const float *A, const float *B, float *C, const float *bias,
                          int M, int N, int K, int lda, int ldb, int ldc, int relu, int acc, int S, int64_t c_slice) {
  const int kslice = (K + S - 1) / S;
  dim3 grid((N + TN - 1) / TN, (M + TM - 1) / TM, S);
  if (!ta && tb)
    hipLaunchKernelGGL((gemm_f32<0, 1>), grid, dim3(256), 0, m->d->stream, A, B, C, bias, M, N, K, lda, ldb, ldc,
                       relu, acc, kslice, c_slice);
  else if (!ta && !tb)
    hipLaunchKernelGGL((gemm_f32<0, 0>), grid, dim3(256), 0, m->d->stream, A, B, C, bias, M, N, K, lda, ldb, ldc,
                       relu, acc, kslice, c_slice);
  else
    hipLaunchKernelGGL((gemm_f32<1, 0>), grid, dim3(256), 0, m->d->stream, A, B, C, bias, M, N, K, lda, ldb, ldc,
                       relu, acc, kslice, c_slice);
}

static void launch_gemm(ehd_mlp *m, int ta, int tb, const float *A, const float *B, float *C, const float *bias, int M,
                        int N, int K, int lda, int ldb, int ldc, int relu, int acc) {
  launch_gemm_s(m, ta, tb, A, B, C, bias, M, N, K, lda, ldb, ldc, relu, acc, 1, 0);
}

/* K slices for a weight-gradient GEMM of M x N over K = batch: enough
 * workgroups to fill the device (about 256), slices of at least 64 */
static int ksplit(int M, int N, int K) {
  int tiles = ((M + TM - 1) / TM) * ((N + TN - 1) / TN);
  int S = 256 / tiles;
  if (S > K / 64)
    S = K / 64;
  return S < 1 ? 1 : S;
}

static int ensure_batch(ehd_mlp *m, int32_t B) {
  if (B <= m->cap)
    return EH_OK;
  for (int l = 0; l <= MLP_LAYERS; l++) {
    if (m->act[l])
      MCHK(hipFree(m->act[l]));
    if (m->dact[l])
      MCHK(hipFree(m->dact[l]));
    m->act[l] = m->dact[l] = NULL;
  }
  if (m->labels)
    MCHK(hipFree(m->labels));
  if (m->loss_part)
    MCHK(hipFree(m->loss_part));
  for (int l = 0; l <= MLP_LAYERS; l++) {
    int w = l == 0 ? m->nin : m->out_dim[l - 1];
    MCHK(hipMalloc((void **)&m->act[l], sizeof(float) * (size_t)B * w));
    MCHK(hipMalloc((void **)&m->dact[l], sizeof(float) * (size_t)B * w));
  }
  MCHK(hipMalloc((void **)&m->labels, sizeof(float) * B));
  MCHK(hipMalloc((void **)&m->loss_part, sizeof(float) * ((B + 255) / 256)));
  m->cap = B;
  {
    /* partials of the split-K weight gradients and of the column sums */
    int64_t need = 0;
    for (int l = 0; l < MLP_LAYERS; l++) {
      int64_t w = (int64_t)ksplit(m->out_dim[l], m->in_dim[l], B) * m->out_dim[l] * m->in_dim[l];
      int64_t c = (int64_t)((B + 63) / 64) * m->out_dim[l];
      need = w > need ? w : need;
      need = c > need ? c : need;
    }
    if (need > m->part_cap) {
      if (m->part)
        MCHK(hipFree(m->part));
      m->part = NULL;
      m->part_cap = 0;
      MCHK(hipMalloc((void **)&m->part, sizeof(float) * need));
      m->part_cap = need;
    }
  }
  return EH_OK;
}

void ehd_mlp_destroy(ehd_mlp *m);

#define FUSED_WGS 512 /* most workgroups of mlp_rows in training */

static size_t tiles_len(const ehd_mlp *m) { return (size_t)m->hs * 16 * m->xc + 4 * (size_t)m->hs * m->hs; }

int ehd_mlp_create(ehd_dev *d, int32_t nin, int32_t hidden, const float *init, ehd_mlp **out) {
  ehd_mlp *m = (ehd_mlp *)calloc(1, sizeof(ehd_mlp));
  if (!m)
    return EH_ERR_NOMEM;
  m->d = d;
  m->nin = nin;
  m->hidden = hidden;
  int64_t off = 0;
  for (int l = 0; l < MLP_LAYERS; l++) {
    m->in_dim[l] = l == 0 ? nin : hidden;
    m->out_dim[l] = l == MLP_LAYERS - 1 ? 1 : hidden;
    m->woff[l] = off;
    off += (int64_t)m->in_dim[l] * m->out_dim[l];
    m->boff[l] = off;
    off += m->out_dim[l];
  }
  m->nparams = off;
  if (hipSetDevice(d->device) != hipSuccess || hipMalloc((void **)&m->params, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void **)&m->grads, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void **)&m->adam_m, sizeof(float) * off) != hipSuccess ||
      hipMalloc((void **)&m->adam_v, sizeof(float) * off) != hipSuccess) {
    ehd_mlp_destroy(m);
    return EH_ERR_NOMEM;
  }
  if (hipMemcpy(m->params, init, sizeof(float) * off, hipMemcpyHostToDevice) != hipSuccess ||
      hipMemset(m->adam_m, 0, sizeof(float) * off) != hipSuccess ||
      hipMemset(m->adam_v, 0, sizeof(float) * off) != hipSuccess) {
    ehd_mlp_destroy(m);
    return EH_ERR_HIP;
  }
  if ((hidden + 63) / 64 <= 4 && (nin + 63) / 64 <= 4) {
    m->fused = 1;
    m->hs = (hidden + 63) / 64 * 64;
    m->xs = (nin + 63) / 64 * 64;
    m->xc = (nin + 15) / 16;
    m->tiles_stale = 1;
    if (hipMalloc((void **)&m->tiles, sizeof(float) * (tiles_len(m) + 1)) != hipSuccess) {
      ehd_mlp_destroy(m);
      return EH_ERR_NOMEM;
    }
    m->floss = m->tiles + tiles_len(m);
  }
  *out = m;
  return EH_OK;
}

int64_t ehd_mlp_nparams(const ehd_mlp *m) { return m->nparams; }

/* teardown: errors are ignored, there is nothing left to undo */
void ehd_mlp_destroy(ehd_mlp *m) {
  if (!m)
    return;
  (void)hipSetDevice(m->d->device);
  (void)hipStreamSynchronize(m->d->stream);
  if (m->pstream) {
    (void)hipStreamSynchronize(m->pstream);
    (void)hipStreamDestroy(m->pstream);
  }
  for (int k = 0; k < 4; k++)
    if (m->pev[k])
      (void)hipEventDestroy(m->pev[k]);
  void *bufs[16] = {m->params, m->grads, m->adam_m, m->adam_v, m->part,   m->Xd,      m->yd,     m->permd, m->eloss,
                    m->tiles,  m->fbuf,  m->fpart,  m->pin[0], m->pin[1], m->pout[0], m->pout[1]};
  for (int k = 0; k < 16; k++)
    if (bufs[k])
      (void)hipFree(bufs[k]);
  for (int l = 0; l <= MLP_LAYERS; l++) {
    if (m->act[l])
      (void)hipFree(m->act[l]);
    if (m->dact[l])
      (void)hipFree(m->dact[l]);
  }
  if (m->labels)
    (void)hipFree(m->labels);
  if (m->loss_part)
    (void)hipFree(m->loss_part);
  free(m);
}

static void forward(ehd_mlp *m, int B) {
  for (int l = 0; l < MLP_LAYERS; l++) {
    int last = l == MLP_LAYERS - 1;
    launch_gemm(m, 0, 1, m->act[l], m->params + m->woff[l], m->act[l + 1], m->params + m->boff[l], B,
                m->out_dim[l], m->in_dim[l], m->in_dim[l], m->in_dim[l], m->out_dim[l], last ? 0 : 1, 0);
  }
}

/* the sum of nb partial losses on the device, which is waited for */
static int batch_loss(ehd_mlp *m, const float *part, int nb, float *loss) {
  float *h = (float *)malloc(sizeof(float) * nb);
  if (!h)
    return EH_ERR_NOMEM;
  hipError_t e = hipMemcpyAsync(h, part, sizeof(float) * nb, hipMemcpyDeviceToHost, m->d->stream);
  const hipError_t w = hipStreamSynchronize(m->d->stream);
  e = e ? e : w;
  double s = 0;
  for (int k = 0; k < nb; k++)
    s += h[k];
  free(h);
  if (e)
    return mlp_fail(m, e, "reading the loss");
  *loss = (float)s;
  return EH_OK;
}

/* gradient of the mean BCE over the batch into m->grads.  The loss: into
 * *loss (synchronizing) when loss is given, else added to the device word
 * loss_acc when that is given.  Weight gradients dW = dZ^T X are split over
 * K (the batch) so that even the 19- and 1-wide layers fill the device; the
 * slices and the bias gradients' row slices are summed in a fixed order. */
static int backward(ehd_mlp *m, int B, float *loss, float *loss_acc) {
  int nb = (B + 255) / 256;
  hipLaunchKernelGGL(bce_grad, dim3(nb), dim3(256), 0, m->d->stream, m->act[MLP_LAYERS], m->labels,
                     m->dact[MLP_LAYERS], m->loss_part, B);
  if (loss_acc)
    hipLaunchKernelGGL(loss_accumulate, dim3(1), dim3(64), 0, m->d->stream, m->loss_part, nb, loss_acc);
  for (int l = MLP_LAYERS - 1; l >= 0; l--) {
    const int M = m->out_dim[l], N = m->in_dim[l];
    const int S = ksplit(M, N, B);
    const int64_t cnt = (int64_t)M * N;
    /* dW = dZ^T X */
    if (S > 1) {
      launch_gemm_s(m, 1, 0, m->dact[l + 1], m->act[l], m->part, NULL, M, N, B, M, N, N, 0, 0, S, cnt);
      hipLaunchKernelGGL(reduce_slices, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, m->d->stream, m->part, S,
                         cnt, m->grads + m->woff[l]);
    } else
      launch_gemm(m, 1, 0, m->dact[l + 1], m->act[l], m->grads + m->woff[l], NULL, M, N, B, M, N, N, 0, 0);
    /* db = column sums of dZ, in row slices of 64 */
    {
      const int rs = (B + 63) / 64;
      hipLaunchKernelGGL(col_sum_part, dim3((unsigned)((M + 63) / 64), (unsigned)rs), dim3(256), 0, m->d->stream,
                         m->dact[l + 1], m->part, B, M, 64);
      hipLaunchKernelGGL(reduce_slices, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, m->d->stream, m->part, rs,
                         (int64_t)M, m->grads + m->boff[l]);
    }
    if (l > 0) {
      /* dX = dZ W, then the ReLU mask of the previous layer's output */
      launch_gemm(m, 0, 0, m->dact[l + 1], m->params + m->woff[l], m->dact[l], NULL, B, N, M, M, N, N, 0, 0);
      int64_t n = (int64_t)B * N;
      hipLaunchKernelGGL(relu_mask, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->d->stream, m->dact[l],
                         m->act[l], n);
    }
  }
  return loss ? batch_loss(m, m->loss_part, nb, loss) : EH_OK;
}

static mlp_net fused_net(const ehd_mlp *m) {
  mlp_net N;
  const size_t w0 = (size_t)m->hs * 16 * m->xc, w1 = (size_t)m->hs * m->hs;
  N.wf[0] = m->tiles;
  N.wf[1] = m->tiles + w0;
  N.wb[1] = m->tiles + w0 + w1;
  N.wf[2] = m->tiles + w0 + 2 * w1;
  N.wb[2] = m->tiles + w0 + 3 * w1;
  N.wb[0] = NULL;
  for (int l = 0; l < 3; l++)
    N.bias[l] = m->params + m->boff[l];
  N.w4 = m->params + m->woff[3];
  N.b4 = m->params + m->boff[3];
  N.nin = m->nin;
  N.hidden = m->hidden;
  N.xc = m->xc;
  N.xs = m->xs;
  return N;
}

static mlp_param fused_param(const ehd_mlp *m) {
  mlp_param P;
  const mlp_net N = fused_net(m);
  memset(&P, 0, sizeof P);
  P.w = m->params;
  P.m = m->adam_m;
  P.v = m->adam_v;
  for (int l = 0; l < 3; l++) {
    P.wf[l] = (float *)N.wf[l];
    P.wb[l] = (float *)N.wb[l];
  }
  for (int l = 0; l < MLP_LAYERS; l++) {
    P.woff[l] = m->woff[l];
    P.boff[l] = m->boff[l];
  }
  P.nin = m->nin;
  P.hidden = m->hidden;
  P.hs = m->hs;
  P.xs = m->xs;
  P.xc = m->xc;
  return P;
}

static int64_t fused_weights(const ehd_mlp *m) { return (int64_t)m->hidden * m->nin + 2 * (int64_t)m->hidden * m->hidden; }

/* the tiled weights, filled after the parameters were set from outside */
static void fused_tiles(ehd_mlp *m) {
  if (!m->tiles_stale)
    return;
  const int len = (int)tiles_len(m);
  hipLaunchKernelGGL(mlp_retile, dim3((len + 255) / 256), dim3(256), 0, m->d->stream, fused_param(m), m->tiles, len);
  m->tiles_stale = 0;
}

static int grow_dev(ehd_mlp *m, void **p, int64_t *cap, int64_t count, size_t sz);

/* buffers for batches of B rows, the batch that uses them and how it is cut */
static int fused_batch(ehd_mlp *m, int32_t B, mlp_batch *Q, mlp_cut *C) {
  const int64_t hs = m->hs, xs = m->xs;
  int rc = grow_dev(m, (void **)&m->fbuf, &m->fcap, B * (xs + 6 * hs + 2), sizeof(float));
  if (rc)
    return rc;
  memset(Q, 0, sizeof *Q);
  Q->xb = m->fbuf;
  for (int l = 0; l < 3; l++) {
    Q->h[l] = m->fbuf + (size_t)B * (xs + l * hs);
    Q->dz[l] = m->fbuf + (size_t)B * (xs + (3 + l) * hs);
  }
  Q->dz4 = m->fbuf + (size_t)B * (xs + 6 * hs);
  Q->lrow = Q->dz4 + B;
  Q->rows = B;
  memset(C, 0, sizeof *C);
  C->hidden = m->hidden;
  C->nin = m->nin;
  C->hs = m->hs;
  C->xs = m->xs;
  C->rs = (B + 63) / 64;
  C->nb = (B + 255) / 256;
  int64_t need = 0, pw[4];
  for (int l = 0; l < MLP_LAYERS; l++) {
    C->S[l] = ksplit(m->out_dim[l], m->in_dim[l], B);
    C->rows[l] = (B + C->S[l] - 1) / C->S[l];
    C->S[l] = (B + C->rows[l] - 1) / C->rows[l]; /* the slices that have rows */
    pw[l] = need;
    need += C->S[l] * (l == 0 ? hs * xs : (l < 3 ? hs * hs : hs));
  }
  const int64_t pb = need, loss = pb + C->rs * (3 * hs + 1);
  rc = grow_dev(m, (void **)&m->fpart, &m->fpart_cap, loss + C->nb, sizeof(float));
  if (rc)
    return rc;
  for (int l = 0; l < MLP_LAYERS; l++) {
    C->pw[l] = m->fpart + pw[l];
    C->pb[l] = m->fpart + pb + C->rs * l * hs;
  }
  C->loss = m->fpart + loss;
  for (int l = 2; l >= 0; l--) {
    const int kn = (m->in_dim[l] + 31) / 32;
    C->wgs[l] = ((m->hidden + 63) / 64 * kn + 3) / 4;
    C->first[3 - l] = C->first[2 - l] + 8 * C->wgs[l] * ((C->S[l] + 7) / 8);
  }
  C->nbias = C->rs * 3 * (m->hs / 64);
  C->nlast = C->S[3];
  return EH_OK;
}

/* one batch: gradients to P.g, or an Adam step; its loss is added to *loss */
static void fused_step(ehd_mlp *m, const mlp_param &P, const mlp_batch &Q, const mlp_cut &C, float *loss) {
  const mlp_net N = fused_net(m);
  hipStream_t st = m->d->stream;
  int wgs = (Q.rows + 15) / 16;
  if (wgs > FUSED_WGS)
    wgs = FUSED_WGS;
  switch (m->hs / 64) {
  case 1:
    hipLaunchKernelGGL((mlp_rows<1, 1, true>), dim3(wgs), dim3(256), 0, st, N, Q);
    break;
  case 2:
    hipLaunchKernelGGL((mlp_rows<2, 1, true>), dim3(wgs), dim3(256), 0, st, N, Q);
    break;
  case 3:
    hipLaunchKernelGGL((mlp_rows<3, 1, true>), dim3(wgs), dim3(256), 0, st, N, Q);
    break;
  default:
    hipLaunchKernelGGL((mlp_rows<4, 1, true>), dim3(wgs), dim3(256), 0, st, N, Q);
  }
  hipLaunchKernelGGL(mlp_wgrad, dim3(C.first[3] + C.nbias + C.nlast + C.nb + (C.rs + 63) / 64), dim3(256), 0, st, Q, C);
  const int64_t nw = fused_weights(m);
  const int nwb = (int)((nw + 255) / 256), nvb = (4 * m->hs + 2 + 63) / 64;
  hipLaunchKernelGGL(mlp_update, dim3(nwb + nvb), dim3(256), 0, st, P, C, nw, nwb, loss);
}

static int fused_grad(ehd_mlp *m, const float *X, const float *y, int32_t B, float *grad, float *loss);
static int fused_predict(ehd_mlp *m, const float *X, int64_t n, float *prob);

int ehd_mlp_grad(ehd_mlp *m, const float *X, const float *y, int32_t B, float *grad, float *loss) {
  int rc;
  MCHK(hipSetDevice(m->d->device));
  if (m->fused)
    return fused_grad(m, X, y, B, grad, loss);
  if ((rc = ensure_batch(m, B)))
    return rc;
  MCHK(hipMemcpyAsync(m->act[0], X, sizeof(float) * (size_t)B * m->nin, hipMemcpyHostToDevice, m->d->stream));
  MCHK(hipMemcpyAsync(m->labels, y, sizeof(float) * B, hipMemcpyHostToDevice, m->d->stream));
  forward(m, B);
  if ((rc = backward(m, B, loss, NULL)))
    return rc;
  MCHK(hipGetLastError());
  MCHK(hipMemcpyAsync(grad, m->grads, sizeof(float) * m->nparams, hipMemcpyDeviceToHost, m->d->stream));
  MCHK(hipStreamSynchronize(m->d->stream));
  return EH_OK;
}

/* grow a device buffer to hold count elements of size sz */
static int grow_dev(ehd_mlp *m, void **p, int64_t *cap, int64_t count, size_t sz) {
  if (count <= *cap)
    return EH_OK;
  if (*p)
    MCHK(hipFree(*p));
  *p = NULL;
  *cap = 0;
  MCHK(hipMalloc(p, sz * (size_t)(count > 0 ? count : 1)));
  *cap = count;
  return EH_OK;
}

static int queue_grad(ehd_mlp *m, const float *X, const float *y, int32_t B, float *grad, mlp_cut &C) {
  mlp_batch Q;
  int rc = fused_batch(m, B, &Q, &C);
  if (!rc)
    rc = grow_dev(m, (void **)&m->Xd, &m->data_cap, (int64_t)B * m->nin, sizeof(float));
  if (!rc)
    rc = grow_dev(m, (void **)&m->yd, &m->y_cap, B, sizeof(float));
  if (rc)
    return rc;
  Q.X = m->Xd;
  Q.y = m->yd;
  mlp_param P = fused_param(m);
  P.g = m->grads;
  MCHK(hipMemcpyAsync(m->Xd, X, sizeof(float) * (size_t)B * m->nin, hipMemcpyHostToDevice, m->d->stream));
  MCHK(hipMemcpyAsync(m->yd, y, sizeof(float) * B, hipMemcpyHostToDevice, m->d->stream));
  fused_tiles(m);
  hipLaunchKernelGGL(mlp_zero, dim3(1), dim3(64), 0, m->d->stream, m->floss, (int64_t)1);
  fused_step(m, P, Q, C, m->floss);
  MCHK(hipGetLastError());
  MCHK(hipMemcpyAsync(grad, m->grads, sizeof(float) * m->nparams, hipMemcpyDeviceToHost, m->d->stream));
  return EH_OK;
}

static int fused_grad(ehd_mlp *m, const float *X, const float *y, int32_t B, float *grad, float *loss) {
  mlp_cut C;
  const int rc = queue_grad(m, X, y, B, grad, C);
  if (!rc && loss)
    return batch_loss(m, C.loss, C.nb, loss);
  const hipError_t e = hipStreamSynchronize(m->d->stream);
  return rc || !e ? rc : mlp_fail(m, e, "gradient");
}

/* chunks of rows: the copies of the next chunk's inputs and the last one's
 * probabilities run beside a chunk's kernel */
#define PRED_ROWS 32768

/* each one made where it is missing: a call that failed half way is
 * completed by the next */
static int predict_set_up(ehd_mlp *m, int64_t n) {
  const int64_t rows = n < PRED_ROWS ? n : PRED_ROWS;
  for (int k = 0; k < (n > PRED_ROWS ? 2 : 1); k++) {
    int rc = grow_dev(m, (void **)&m->pin[k], &m->pin_cap[k], rows * m->nin, sizeof(float));
    if (!rc)
      rc = grow_dev(m, (void **)&m->pout[k], &m->pout_cap[k], rows, sizeof(float));
    if (rc)
      return rc;
  }
  if (n <= PRED_ROWS)
    return EH_OK;
  if (!m->pstream)
    MCHK(hipStreamCreateWithFlags(&m->pstream, hipStreamNonBlocking));
  for (int k = 0; k < 4; k++)
    if (!m->pev[k])
      MCHK(hipEventCreateWithFlags(&m->pev[k], hipEventDisableTiming));
  return EH_OK;
}

static void predict_launch(const ehd_mlp *m, const mlp_net &N, const mlp_batch &Q) {
  hipStream_t st = m->d->stream;
  switch (m->hs / 64) {
  case 1:
    rows_predict<1>(st, N, Q);
    break;
  case 2:
    rows_predict<2>(st, N, Q);
    break;
  case 3:
    rows_predict<3>(st, N, Q);
    break;
  default:
    rows_predict<4>(st, N, Q);
  }
}

static int predict_chunks(ehd_mlp *m, const float *X, int64_t n, float *prob) {
  hipStream_t st = m->d->stream;
  fused_tiles(m);
  const mlp_net N = fused_net(m);
  int rc = n > 0 ? predict_set_up(m, n) : EH_OK;
  if (rc || n <= 0)
    return rc;
  if (n <= PRED_ROWS) {
    /* nothing to run beside: one stream, no events (a net of 16 on one row
     * takes 38 us instead of 48, its first prediction 90 instead of 210) */
    mlp_batch Q;
    memset(&Q, 0, sizeof Q);
    Q.X = m->pin[0];
    Q.prob = m->pout[0];
    Q.rows = (int)n;
    MCHK(hipMemcpyAsync(m->pin[0], X, sizeof(float) * (size_t)n * m->nin, hipMemcpyHostToDevice, st));
    predict_launch(m, N, Q);
    MCHK(hipGetLastError());
    MCHK(hipMemcpyAsync(prob, m->pout[0], sizeof(float) * (size_t)n, hipMemcpyDeviceToHost, st));
    return EH_OK;
  }
  int64_t done = 0; /* probabilities copied out */
  int c = 0;
  for (int64_t s0 = 0; s0 < n; s0 += PRED_ROWS, c++) {
    const int b = (int)(n - s0 < PRED_ROWS ? n - s0 : PRED_ROWS), k = c & 1;
    mlp_batch Q;
    memset(&Q, 0, sizeof Q);
    Q.X = m->pin[k];
    Q.prob = m->pout[k];
    Q.rows = b;
    /* chunk c - 2's kernel is done with this buffer (its results were copied) */
    MCHK(hipMemcpyAsync(m->pin[k], X + (size_t)s0 * m->nin, sizeof(float) * (size_t)b * m->nin, hipMemcpyHostToDevice,
                        m->pstream));
    MCHK(hipEventRecord(m->pev[k], m->pstream));
    MCHK(hipStreamWaitEvent(st, m->pev[k], 0));
    predict_launch(m, N, Q);
    MCHK(hipGetLastError());
    MCHK(hipEventRecord(m->pev[2 + k], st));
    if (c > 0) {
      const int64_t p0 = done;
      MCHK(hipStreamWaitEvent(m->pstream, m->pev[2 + (k ^ 1)], 0));
      MCHK(hipMemcpyAsync(prob + p0, m->pout[k ^ 1], sizeof(float) * PRED_ROWS, hipMemcpyDeviceToHost, m->pstream));
      done = s0;
    }
  }
  MCHK(hipStreamWaitEvent(m->pstream, m->pev[2 + ((c - 1) & 1)], 0));
  MCHK(hipMemcpyAsync(prob + done, m->pout[(c - 1) & 1], sizeof(float) * (size_t)(n - done), hipMemcpyDeviceToHost,
                      m->pstream));
  return EH_OK;
}

/* also after a failure nothing queued may still use the caller's arrays */
static int fused_predict(ehd_mlp *m, const float *X, int64_t n, float *prob) {
  const int rc = predict_chunks(m, X, n, prob);
  const hipError_t p = m->pstream ? hipStreamSynchronize(m->pstream) : hipSuccess, s = hipStreamSynchronize(m->d->stream);
  if (rc)
    return rc;
  return p || s ? mlp_fail(m, p ? p : s, "prediction") : EH_OK;
}

/* minibatch Adam over n samples (X row-major [n, nin]) for the given epochs;
 * the sample order per epoch is the given permutation table (epochs x n).
 * The training set and the order are copied to the device once; each step
 * gathers its minibatch on the device, the losses are summed on the device,
 * and the host waits once, at the end. */
int ehd_mlp_train(ehd_mlp *m, const float *X, const float *y, int64_t n, const int64_t *perm, int32_t epochs,
                  int32_t B, float lr, float *losses) {
  int rc;
  const int64_t nsteps = n / B;
  MCHK(hipSetDevice(m->d->device));
  if (n > 0x7fffffff)
    return EH_ERR_INVALID;
  mlp_batch Q;
  mlp_cut C;
  if ((rc = m->fused ? fused_batch(m, B, &Q, &C) : ensure_batch(m, B)))
    return rc;
  if ((rc = grow_dev(m, (void **)&m->Xd, &m->data_cap, n * m->nin, sizeof(float))) ||
      (rc = grow_dev(m, (void **)&m->yd, &m->y_cap, n, sizeof(float))) ||
      (rc = grow_dev(m, (void **)&m->permd, &m->perm_cap, (int64_t)epochs * n, sizeof(int32_t))) ||
      (rc = grow_dev(m, (void **)&m->eloss, &m->eloss_cap, epochs, sizeof(float))))
    return rc;
  {
    int32_t *p32 = (int32_t *)malloc(sizeof(int32_t) * (size_t)((int64_t)epochs * n > 0 ? (int64_t)epochs * n : 1));
    if (!p32)
      return EH_ERR_NOMEM;
    for (int64_t k = 0; k < (int64_t)epochs * n; k++)
      p32[k] = (int32_t)perm[k];
    MCHK(hipMemcpyAsync(m->Xd, X, sizeof(float) * (size_t)(n * m->nin), hipMemcpyHostToDevice, m->d->stream));
    MCHK(hipMemcpyAsync(m->yd, y, sizeof(float) * (size_t)n, hipMemcpyHostToDevice, m->d->stream));
    MCHK(hipMemcpyAsync(m->permd, p32, sizeof(int32_t) * (size_t)((int64_t)epochs * n), hipMemcpyHostToDevice,
                        m->d->stream));
    MCHK(hipStreamSynchronize(m->d->stream));
    free(p32);
  }
  if (epochs > 0)
    hipLaunchKernelGGL(reduce_slices, dim3((unsigned)((epochs + 255) / 256)), dim3(256), 0, m->d->stream, m->eloss,
                       0, (int64_t)epochs, m->eloss); /* zero the per-epoch sums (a kernel, no memset) */
  if (m->fused) {
    mlp_param P = fused_param(m);
    P.lr = lr;
    P.b1 = 0.9f;
    P.b2 = 0.999f;
    P.eps = 1e-8f;
    Q.X = m->Xd;
    Q.y = m->yd;
    fused_tiles(m);
    for (int ep = 0; ep < epochs; ep++)
      for (int64_t st = 0; st < nsteps; st++) {
        Q.perm = m->permd + (int64_t)ep * n + st * B;
        m->step++;
        P.c1 = 1.f - powf(0.9f, (float)m->step);
        P.c2 = 1.f - powf(0.999f, (float)m->step);
        fused_step(m, P, Q, C, m->eloss + ep);
      }
  }
  for (int ep = 0; ep < epochs && !m->fused; ep++) {
    for (int64_t st = 0; st < nsteps; st++) {
      const int64_t e = (int64_t)B * m->nin;
      hipLaunchKernelGGL(gather_batch, dim3((unsigned)((e + 255) / 256)), dim3(256), 0, m->d->stream, m->Xd, m->yd,
                         m->permd + (int64_t)ep * n + st * B, B, m->nin, m->act[0], m->labels);
      forward(m, B);
      if ((rc = backward(m, B, NULL, m->eloss + ep)))
        return rc;
      m->step++;
      float c1 = 1.f - powf(0.9f, (float)m->step), c2 = 1.f - powf(0.999f, (float)m->step);
      hipLaunchKernelGGL(adam_k, dim3((unsigned)((m->nparams + 255) / 256)), dim3(256), 0, m->d->stream, m->params,
                         m->grads, m->adam_m, m->adam_v, m->nparams, lr, 0.9f, 0.999f, 1e-8f, c1, c2);
    }
  }
  MCHK(hipGetLastError());
  if (losses && epochs > 0) {
    MCHK(hipMemcpyAsync(losses, m->eloss, sizeof(float) * epochs, hipMemcpyDeviceToHost, m->d->stream));
    MCHK(hipStreamSynchronize(m->d->stream));
    for (int ep = 0; ep < epochs; ep++)
      losses[ep] = nsteps ? losses[ep] / (float)nsteps : 0.f;
  }
  MCHK(hipStreamSynchronize(m->d->stream));
  return EH_OK;
}

int ehd_mlp_predict(ehd_mlp *m, const float *X, int64_t n, float *prob) {
  int rc;
  const int32_t B = 8192;
  MCHK(hipSetDevice(m->d->device));
  if (m->fused)
    return fused_predict(m, X, n, prob);
  if ((rc = ensure_batch(m, B)))
    return rc;
  for (int64_t s0 = 0; s0 < n; s0 += B) {
    int32_t b = (int32_t)(n - s0 < B ? n - s0 : B);
    MCHK(hipMemcpyAsync(m->act[0], X + (size_t)s0 * m->nin, sizeof(float) * (size_t)b * m->nin,
                        hipMemcpyHostToDevice, m->d->stream));
    forward(m, b);
    hipLaunchKernelGGL(sigmoid_k, dim3((b + 255) / 256), dim3(256), 0, m->d->stream, m->act[MLP_LAYERS],
                       m->dact[MLP_LAYERS], (int64_t)b);
    MCHK(hipMemcpyAsync(prob + s0, m->dact[MLP_LAYERS], sizeof(float) * b, hipMemcpyDeviceToHost, m->d->stream));
  }
  MCHK(hipStreamSynchronize(m->d->stream));
  return EH_OK;
}

int ehd_mlp_params(ehd_mlp *m, float *buf, int set) {
  MCHK(hipSetDevice(m->d->device));
  if (set)
    m->tiles_stale = 1;
  if (set)
    MCHK(hipMemcpy(m->params, buf, sizeof(float) * m->nparams, hipMemcpyHostToDevice));
  else
    MCHK(hipMemcpy(buf, m->params, sizeof(float) * m->nparams, hipMemcpyDeviceToHost));
  return EH_OK;
}
}
