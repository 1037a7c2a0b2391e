// Per-column MLP that predicts the initial iterate of the HEVI Newton solve
// (no counterpart in the reference, whose Newton loop starts from q^n and
// stops after one iteration).  Dense layers n_in -> H -> H -> H -> n_out with
// ReLU, BF16 operands on the matrix cores (v_mfma_f32_16x16x16_bf16) with
// FP32 accumulation, FP32 master weights and Adam.
//
// All products are "NT" GEMMs, C[m][n] = sum_k A[m][k] B[n][k]:
//   forward     Z  = X  W^T        (A = X [B x K],    B = W  [N x K])
//   input grad  dX = dZ W          (A = dZ [B x N],   B = W^T [K x N])
//   weight grad dW = dZ^T X        (A = dZ^T [N x B], B = X^T [K x B])
// A BF16 operand lies in memory as the matrix instruction's fragments: 16 rows
// x 32 k per 1 KB block, lane l's two quadruples of k (row l % 16, k = 4 (l /
// 16) + 0..3 and 16 + that) together, rows and k padded to 32 with zeros.  A
// wavefront's load of a fragment pair is one contiguous 16 bytes per lane, and
// an accumulator tile stored as it lies in registers is a fragment of the
// product's transpose: the kernel that forms an activation or a gradient
// writes both forms the later products read, and Adam writes the weights'.
//
// Bound: launches and the latency of the loads (the network of the HEVI guess
// has 0.4 million weights).  Training step of the 641-256-256-256-320 network
// with 512 rows: 49 launches, 314 us -> 11 launches, 75 us.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "fedg_internal.h"
#include "fedg_mlp.h"

namespace fedg {
namespace {

typedef short short4_ __attribute__((ext_vector_type(4)));
typedef short short8_ __attribute__((ext_vector_type(8)));
typedef float float4_ __attribute__((ext_vector_type(4)));

// round to nearest even
__device__ __forceinline__ uint16_t f2bf(float x) {
  uint32_t u = __float_as_uint(x);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16) | ((u & 0xffffu) ? 0x40 : 0);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

inline __host__ __device__ int pad32(int k) { return (k + 31) / 32 * 32; }

// position of (row, k) in a fragment-ordered matrix of KB = pad32(K) / 32 blocks per row block
__device__ __forceinline__ size_t frag(int row, int k, int KB) {
  return (((size_t)(row >> 4) * KB + (k >> 5)) * 64 + ((k >> 2) & 3) * 16 + (row & 15)) * 8 + ((k >> 4) & 1) * 4 +
         (k & 3);
}

// acc = the (16 T) x (16 T) tile of row blocks ra.. of A and rb.. of B over KB
// pairs of 16-deep products, k ascending.  U pairs are in flight while the U
// before them are multiplied.
template <int T>
__device__ __forceinline__ void gemm_tile(const uint16_t* __restrict__ A, int ra, const uint16_t* __restrict__ B, int rb,
                                          int KB, float4_ (&acc)[T][T]) {
  constexpr int U = T == 1 ? 8 : 4;
  const int lane = threadIdx.x & 63;
  const short8_* pa[T];
  const short8_* pb[T];
#pragma unroll
  for (int a = 0; a < T; ++a) {
    pa[a] = reinterpret_cast<const short8_*>(A) + (size_t)(ra + a) * KB * 64 + lane;
    pb[a] = reinterpret_cast<const short8_*>(B) + (size_t)(rb + a) * KB * 64 + lane;
#pragma unroll
    for (int b = 0; b < T; ++b) acc[a][b] = (float4_){0.f, 0.f, 0.f, 0.f};
  }
  short8_ fa[2][U][T], fb[2][U][T];
  auto load = [&](int s, int k) {
    if (k >= KB) return;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int kk = (k + u < KB ? k + u : KB - 1) * 64;
#pragma unroll
      for (int a = 0; a < T; ++a) {
        fa[s][u][a] = pa[a][kk];
        fb[s][u][a] = pb[a][kk];
      }
    }
  };
  auto multiply = [&](int s, int k) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (k + u >= KB) break;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int a = 0; a < T; ++a)
#pragma unroll
          for (int b = 0; b < T; ++b) {
            const short8_ x = fa[s][u][a], y = fb[s][u][b];
            const short4_ xh = h ? __builtin_shufflevector(x, x, 4, 5, 6, 7) : __builtin_shufflevector(x, x, 0, 1, 2, 3);
            const short4_ yh = h ? __builtin_shufflevector(y, y, 4, 5, 6, 7) : __builtin_shufflevector(y, y, 0, 1, 2, 3);
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(xh, yh, acc[a][b], 0, 0, 0);
          }
    }
  };
  load(0, 0);
  for (int k = 0; k < KB; k += 2 * U) {
    load(1, k + U);
    multiply(0, k);
    load(0, k + 2 * U);
    multiply(1, k + U);
  }
}

// stores a tile's values val(a, b, i, row, col) (zero in the padding): fp32
// [M x N] (f32), fragments of the matrix (d) and of its transpose (t); null
// pointers are skipped.  Accumulator layout: rows 4 (lane / 16) + i of column
// lane % 16.
template <int T, typename F>
__device__ __forceinline__ void store_tile(int ra, int rb, int M, int N, float* __restrict__ f32, uint16_t* __restrict__ d,
                                           uint16_t* __restrict__ t, F val) {
  const int lane = threadIdx.x & 63, q = lane >> 4, c = lane & 15;
  const int KBd = pad32(N) / 32, KBt = pad32(M) / 32;
#pragma unroll
  for (int a = 0; a < T; ++a)
#pragma unroll
    for (int b = 0; b < T; ++b) {
      const int row0 = (ra + a) * 16 + q * 4, col = (rb + b) * 16 + c;
      short4_ h;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool in = row0 + i < M && col < N;
        const float v = in ? val(a, b, i, row0 + i, col) : 0.f;
        if (in && f32) f32[(size_t)(row0 + i) * N + col] = v;
        h[i] = (short)f2bf(v);
        if (d) d[frag(row0 + i, col, KBd)] = (uint16_t)h[i];
      }
      if (t) *reinterpret_cast<short4_*>(t + frag(col, row0, KBt)) = h;
    }
}

// the wavefront's tile of a product of M x N results in tiles of 16 T, the four
// wavefronts of a block along n; false past the last one
template <int T>
__device__ __forceinline__ bool tile_of(int blk, int M, int N, int& ra, int& rb) {
  const int tn = pad32(N) / (16 * T), tm = pad32(M) / (16 * T);
  const int t = blk * 4 + (threadIdx.x >> 6);
  ra = t / tn * T;
  rb = t % tn * T;
  return t < tn * tm;
}
template <int T>
inline unsigned tile_blocks(int M, int N) {
  return (unsigned)(((size_t)(pad32(N) / (16 * T)) * (pad32(M) / (16 * T)) + 3) / 4);
}

// one layer forward, [Bn x K] -> [Bn x N]: bias, ReLU (act), the outputs in the forms asked for
template <int T>
__global__ void __launch_bounds__(256) forward_kernel(const uint16_t* __restrict__ X, const uint16_t* __restrict__ W,
                                                      const float* __restrict__ bias, int Bn, int N, int K, int act,
                                                      float* __restrict__ f32, uint16_t* __restrict__ d,
                                                      uint16_t* __restrict__ t) {
  int ra, rb;
  if (!tile_of<T>(blockIdx.x, Bn, N, ra, rb)) return;
  float4_ acc[T][T];
  gemm_tile<T>(X, ra, W, rb, pad32(K) / 32, acc);
  store_tile<T>(ra, rb, Bn, N, f32, d, t, [&](int a, int b, int i, int, int col) {
    float v = acc[a][b][i] + bias[col];
    if (act) v = v > 0.f ? v : 0.f;
    return v;
  });
}

// a 32 x 32 tile of a matrix [R x C] with values val(r, c) into its fragments
// (d) and its transpose's (t), 16 bytes per lane; block of 256 threads
template <typename F>
__device__ __forceinline__ void pack_tile(int br, int bc, int R, int C, uint16_t* __restrict__ d, uint16_t* __restrict__ t,
                                          F val) {
  __shared__ float tile[32][33];
  const int r0 = br * 32, c0 = bc * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
#pragma unroll
  for (int j = 0; j < 32; j += 8) {
    const int r = r0 + j + ty, c = c0 + tx;
    tile[j + ty][tx] = (r < R && c < C) ? val(r, c) : 0.f;
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int row = (w & 1) * 16 + (lane & 15), k0 = (lane >> 4) * 4;
  uint16_t* const y = w < 2 ? d : t;
  if (!y) return;
  short8_ h;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int k = k0 + (i & 3) + (i >> 2) * 16;
    h[i] = (short)f2bf(w < 2 ? tile[row][k] : tile[k][row]);
  }
  const int KB = (w < 2 ? pad32(C) : pad32(R)) / 32;
  *reinterpret_cast<short8_*>(y + frag((w < 2 ? r0 : c0) + row, (w < 2 ? c0 : r0) + k0, KB)) = h;
}

// fp32 [R x C] -> fragments
__global__ void __launch_bounds__(256) pack_kernel(const float* __restrict__ x, int R, int C, uint16_t* __restrict__ d,
                                                   uint16_t* __restrict__ t) {
  const int tn = pad32(C) / 32;
  pack_tile(blockIdx.x / tn, blockIdx.x % tn, R, C, d, t, [&](int r, int c) { return x[(size_t)r * C + c]; });
}

// column sums of dZ [Bn x N] -> db[N]: 16 columns x 16 row groups per 256
// threads, the groups' partial sums added in group order
__device__ __forceinline__ void column_sums(int blk, const float* __restrict__ dZ, float* __restrict__ db, int Bn, int N) {
  __shared__ float part[16][16];
  const int tx = threadIdx.x & 15, g = threadIdx.x >> 4;
  const int c = blk * 16 + tx;
  float s = 0.f;
  if (c < N) {
    int b = g;
    for (; b + 112 < Bn; b += 128) {
      float a[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) a[u] = dZ[(size_t)(b + 16 * u) * N + c];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += a[u];
    }
    for (; b < Bn; b += 16) s += dZ[(size_t)b * N + c];
  }
  part[g][tx] = s;
  __syncthreads();
  if (g == 0 && c < N) {
    float t = part[0][tx];
    for (int k = 1; k < 16; ++k) t += part[k][tx];
    db[c] = t;
  }
}

// One layer backward from dZ [Bn x N]: the blocks before nW form the weight
// gradient [N x K], those before nX the bias gradient, the rest the gradient
// of the layer's input behind its ReLU, dX (H > 0) with H = X [Bn x K].
struct BackArgs {
  int Bn, N, K;
  int nW, nX;
  const uint16_t *dZ, *dZt, *Xt, *Wt;  // fragments
  const float *dZ32, *H;
  float *dW, *db;
  float* dX32;
  uint16_t *dX, *dXt;
};
template <int T>
__global__ void __launch_bounds__(256) backward_kernel(const BackArgs p) {
  int blk = blockIdx.x, ra, rb;
  if (blk < p.nW) {
    if (!tile_of<1>(blk, p.N, p.K, ra, rb)) return;
    float4_ acc[1][1];
    gemm_tile<1>(p.dZt, ra, p.Xt, rb, pad32(p.Bn) / 32, acc);
    store_tile<1>(ra, rb, p.N, p.K, p.dW, nullptr, nullptr, [&](int a, int b, int i, int, int) { return acc[a][b][i]; });
  } else if (blk < p.nX) {
    column_sums(blk - p.nW, p.dZ32, p.db, p.Bn, p.N);
  } else {
    if (!tile_of<T>(blk - p.nX, p.Bn, p.K, ra, rb)) return;
    float4_ acc[T][T];
    gemm_tile<T>(p.dZ, ra, p.Wt, rb, pad32(p.N) / 32, acc);
    store_tile<T>(ra, rb, p.Bn, p.K, p.dX32, p.dX, p.dXt, [&](int a, int b, int i, int row, int col) {
      return p.H[(size_t)row * p.K + col] > 0.f ? acc[a][b][i] : 0.f;
    });
  }
}

// mean squared error: dY = 2 (Y - T) / (Bn N) (blocks from 256 on, one 32 x 32
// tile each) and the first 256 blocks' partial sums of (Y-T)^2
__global__ void __launch_bounds__(256) mse_kernel(const float* __restrict__ Y, const float* __restrict__ T,
                                                  float* __restrict__ dY, uint16_t* __restrict__ d,
                                                  uint16_t* __restrict__ dt, int Bn, int N, float* __restrict__ partial) {
  const long n = (long)Bn * N;
  if (blockIdx.x >= 256) {
    const int tn = pad32(N) / 32, b = blockIdx.x - 256;
    const float sc = 2.f / (float)n;
    pack_tile(b / tn, b % tn, Bn, N, d, dt, [&](int r, int c) {
      const size_t o = (size_t)r * N + c;
      const float e = Y[o] - T[o];
      dY[o] = sc * e;
      return sc * e;
    });
    return;
  }
  __shared__ float s[256];
  float acc = 0.f;
  for (long t = (long)blockIdx.x * 256 + threadIdx.x; t < n; t += 256 * 256) {
    const float e = Y[t] - T[t];
    acc += e * e;
  }
  s[threadIdx.x] = acc;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = s[0];
}

// the layers' places in the parameter vector and the fragments of their weights
struct Layers {
  int nl;
  int N[8], K[8];
  long woff[8];
  uint16_t *W[8], *Wt[8];
};

__global__ void adam_kernel(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                            float* __restrict__ v, long n, float lr, float b1, float b2, float eps, float c1,
                            float c2, const Layers L) {
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const float gt = g[t];
  const float mt = b1 * m[t] + (1.f - b1) * gt;
  const float vt = b2 * v[t] + (1.f - b2) * gt * gt;
  m[t] = mt;
  v[t] = vt;
  const float pt = p[t] - lr * (mt / c1) / (sqrtf(vt / c2) + eps);
  p[t] = pt;
  int l = 0;
  while (l + 1 < L.nl && t >= L.woff[l + 1]) ++l;
  const long e = t - L.woff[l];
  if (e >= (long)L.N[l] * L.K[l]) return;  // a bias
  // 64-bit division only where the layer needs it: it is most of the kernel's instructions
  const int r = e >> 32 ? (int)(e / L.K[l]) : (int)((uint32_t)e / (uint32_t)L.K[l]);
  const int k = (int)(e - (long)r * L.K[l]);
  const uint16_t h = f2bf(pt);
  L.W[l][frag(r, k, pad32(L.K[l]) / 32)] = h;
  L.Wt[l][frag(k, r, pad32(L.N[l]) / 32)] = h;
}

inline unsigned nblk(long n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

struct MlpImpl {
  int nl;                 // layers
  int dims[8];            // dims[0] = n_in, ..., dims[nl] = n_out
  float* params;          // all W (N x K, unpadded) then b, fp32 master copy
  float* grads;
  float* m;
  float* v;
  long nparam;
  long woff[8], boff[8];
  Layers lay;             // dims, offsets, BF16 fragments of the weights and of their transposes
  bool packed;            // the fragments are those of params
  int cap, cap_train;     // rows the workspaces hold: forward; and backward
  uint16_t* hb[8];        // fragments of the layers' inputs [B x dims[l]]
  uint16_t* hbt[8];       // of their transposes (backward only, as all that follow)
  float* act[8];          // act[l], l >= 1: outputs of layer l - 1, fp32
  float* dact[8];         // gradients w.r.t. act
  uint16_t* dzb[2];       // fragments of dact, of the layer in work and of the one below
  uint16_t* dzbt[2];
  float* partial;         // the loss's partial sums, host memory the GPU writes
  long step;
  hipStream_t stream;
};

static int mlp_hip(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    set_error(std::string(what) + ": " + hipGetErrorString(e));
    return FEDG_ERR_HIP;
  }
  return FEDG_OK;
}
#define MLP_TRY(x)                   \
  do {                               \
    int rc_ = (x);                   \
    if (rc_ != FEDG_OK) return rc_;  \
  } while (0)

int mlp_create(int n_in, int n_hidden, int n_hidden_layers, int n_out, unsigned seed, MlpImpl** out) {
  if (n_in < 1 || n_hidden < 1 || n_hidden_layers < 1 || n_hidden_layers > 6 || n_out < 1) {
    set_error("mlp: bad layer sizes");
    return FEDG_ERR_ARG;
  }
  MlpImpl* p = new MlpImpl();
  memset(p, 0, sizeof(*p));
  p->nl = n_hidden_layers + 1;
  p->dims[0] = n_in;
  for (int l = 1; l <= n_hidden_layers; ++l) p->dims[l] = n_hidden;
  p->dims[p->nl] = n_out;
  long off = 0;
  for (int l = 0; l < p->nl; ++l) {
    p->woff[l] = off;
    off += (long)p->dims[l + 1] * p->dims[l];
  }
  for (int l = 0; l < p->nl; ++l) {
    p->boff[l] = off;
    off += p->dims[l + 1];
  }
  p->nparam = off;
  // He-uniform initialisation, zero biases
  std::vector<float> h((size_t)off, 0.f);
  std::mt19937 rng(seed);
  for (int l = 0; l < p->nl; ++l) {
    const float lim = std::sqrt(6.f / (float)p->dims[l]) * (l == p->nl - 1 ? 0.1f : 1.f);
    std::uniform_real_distribution<float> U(-lim, lim);
    for (long t = 0; t < (long)p->dims[l + 1] * p->dims[l]; ++t) h[p->woff[l] + t] = U(rng);
  }
  int rc = mlp_hip(hipStreamCreate(&p->stream), "hipStreamCreate");
  auto al = [&](void** q, size_t bytes) {
    if (rc == FEDG_OK) rc = mlp_hip(hipMalloc(q, bytes), "hipMalloc");
    if (rc == FEDG_OK) rc = mlp_hip(hipMemset(*q, 0, bytes), "hipMemset");
  };
  al((void**)&p->params, sizeof(float) * off);
  al((void**)&p->grads, sizeof(float) * off);
  al((void**)&p->m, sizeof(float) * off);
  al((void**)&p->v, sizeof(float) * off);
  if (rc == FEDG_OK) rc = mlp_hip(hipHostMalloc((void**)&p->partial, sizeof(float) * 256, hipHostMallocDefault), "hipHostMalloc");
  Layers& L = p->lay;
  L.nl = p->nl;
  for (int l = 0; l < p->nl; ++l) {
    L.N[l] = p->dims[l + 1];
    L.K[l] = p->dims[l];
    L.woff[l] = p->woff[l];
    const size_t sz = sizeof(uint16_t) * (size_t)pad32(L.N[l]) * pad32(L.K[l]);
    al((void**)&L.W[l], sz);  // cleared: the padding stays zero
    al((void**)&L.Wt[l], sz);
  }
  if (rc == FEDG_OK) rc = mlp_hip(hipMemcpy(p->params, h.data(), sizeof(float) * off, hipMemcpyHostToDevice), "upload");
  if (rc != FEDG_OK) {
    mlp_destroy(p);
    return rc;
  }
  *out = p;
  return FEDG_OK;
}

void mlp_destroy(MlpImpl* p) {
  if (!p) return;
  void* bufs[] = {p->params, p->grads, p->m, p->v, p->dzb[0], p->dzb[1], p->dzbt[0], p->dzbt[1]};
  for (void* b : bufs)
    if (b) (void)hipFree(b);
  for (int l = 0; l < 8; ++l)
    for (void* b : {(void*)p->lay.W[l], (void*)p->lay.Wt[l], (void*)p->hb[l], (void*)p->hbt[l], (void*)p->act[l],
                    (void*)p->dact[l]})
      if (b) (void)hipFree(b);
  if (p->partial) (void)hipHostFree(p->partial);
  if (p->stream) (void)hipStreamDestroy(p->stream);
  delete p;
}

// workspaces for B rows, forward only or with the backward pass
static int mlp_reserve(MlpImpl* p, int B, bool train) {
  int rc = FEDG_OK;
  auto al = [&](auto*& q, size_t n) {
    if (q) (void)hipFree(q);
    q = nullptr;
    if (rc == FEDG_OK) rc = mlp_hip(hipMalloc((void**)&q, sizeof(*q) * n), "hipMalloc");
  };
  const int cap = pad32(B);
  if (B > p->cap) {
    p->cap = 0;
    for (int l = 0; l < p->nl; ++l) al(p->hb[l], (size_t)cap * pad32(p->dims[l]));
    if (rc == FEDG_OK) p->cap = cap;
  }
  if (train && B > p->cap_train) {
    p->cap_train = 0;
    size_t wmax = 0;
    for (int l = 1; l <= p->nl; ++l) wmax = std::max(wmax, (size_t)pad32(p->dims[l]));
    for (int l = 0; l <= p->nl; ++l) {
      if (l < p->nl) al(p->hbt[l], (size_t)cap * pad32(p->dims[l]));
      if (l > 0) al(p->act[l], (size_t)cap * p->dims[l]);
      if (l > 0) al(p->dact[l], (size_t)cap * p->dims[l]);
    }
    for (int s = 0; s < 2; ++s) {
      al(p->dzb[s], (size_t)cap * wmax);
      al(p->dzbt[s], (size_t)cap * wmax);
    }
    if (rc == FEDG_OK) p->cap_train = cap;
  }
  return rc;
}

static int mlp_pack(MlpImpl* p, const float* x, int R, int C, uint16_t* d, uint16_t* t) {
  hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((size_t)(pad32(C) / 32) * (pad32(R) / 32))), dim3(256), 0,
                     p->stream, x, R, C, d, t);
  return mlp_hip(hipGetLastError(), "pack_kernel");
}

// fragments of the weights from the fp32 masters, where Adam has not written them
static int mlp_sync_weights(MlpImpl* p) {
  if (p->packed) return FEDG_OK;
  const Layers& L = p->lay;
  for (int l = 0; l < p->nl; ++l) MLP_TRY(mlp_pack(p, p->params + p->woff[l], L.N[l], L.K[l], L.W[l], L.Wt[l]));
  p->packed = true;
  return FEDG_OK;
}

// 32 x 32 tiles per wavefront (half the loads per product) once they give every
// SIMD two; below, four times as many wavefronts of 16 x 16 hide the latency.
// Forward, 641-256-256-256-320, wide / narrow: 2048 rows (512 wide tiles in a
// hidden layer) 47.8 / 37.8 us, 4096 rows 52.6 / 50.2, 8192 rows (2048 tiles)
// 67.1 / 71.9, 65536 rows 363 / 413 us.  Loss and gradients, the backward pass
// wide / narrow: 2048 rows 85 / 84 us, 4096 rows 125 / 128, 8192 rows 199 / 205,
// 65536 rows 1907 / 1934 us; 1024-wide layers, 8192 rows 889 / 936 us.
static bool wide_tiles(int M, int N) { return (long)(pad32(M) / 32) * (pad32(N) / 32) >= 2048; }

// forward of B rows of X (device fp32 [B x n_in]) into Y; train: what the backward pass reads as well
static int mlp_fwd(MlpImpl* p, const float* X, float* Y, int B, bool train) {
  MLP_TRY(mlp_pack(p, X, B, p->dims[0], p->hb[0], train ? p->hbt[0] : nullptr));
  for (int l = 0; l < p->nl; ++l) {
    const bool last = l == p->nl - 1;
    const int K = p->dims[l], N = p->dims[l + 1];
    const bool wide = wide_tiles(B, N);
    hipLaunchKernelGGL(wide ? forward_kernel<2> : forward_kernel<1>, dim3(wide ? tile_blocks<2>(B, N) : tile_blocks<1>(B, N)),
                       dim3(256), 0, p->stream, p->hb[l], p->lay.W[l], p->params + p->boff[l], B, N, K, last ? 0 : 1,
                       last ? Y : train ? p->act[l + 1] : nullptr, last ? nullptr : p->hb[l + 1],
                       !last && train ? p->hbt[l + 1] : nullptr);
    MLP_TRY(mlp_hip(hipGetLastError(), "forward_kernel"));
  }
  return FEDG_OK;
}

// backward from dact[nl] and its fragments dzb[0], dzbt[0] (set by the loss); gradients into p->grads
static int mlp_bwd(MlpImpl* p, int B) {
  int s = 0;
  for (int l = p->nl - 1; l >= 0; --l, s ^= 1) {
    BackArgs a{};
    a.Bn = B;
    a.N = p->dims[l + 1];
    a.K = p->dims[l];
    a.dZ = p->dzb[s];
    a.dZt = p->dzbt[s];
    a.Xt = p->hbt[l];
    a.Wt = p->lay.Wt[l];
    a.dZ32 = p->dact[l + 1];
    a.dW = p->grads + p->woff[l];
    a.db = p->grads + p->boff[l];
    a.nW = tile_blocks<1>(a.N, a.K);
    a.nX = a.nW + (a.N + 15) / 16;
    unsigned blocks = a.nX;
    const bool wide = l > 0 && wide_tiles(B, a.K);  // of the input gradient, which the first layer has none of
    if (l > 0) {
      a.H = p->act[l];
      a.dX32 = p->dact[l];
      a.dX = l > 1 ? p->dzb[s ^ 1] : nullptr;  // no product reads the first layer's
      a.dXt = p->dzbt[s ^ 1];
      blocks += wide ? tile_blocks<2>(B, a.K) : tile_blocks<1>(B, a.K);
    }
    hipLaunchKernelGGL(wide ? backward_kernel<2> : backward_kernel<1>, dim3(blocks), dim3(256), 0, p->stream, a);
    MLP_TRY(mlp_hip(hipGetLastError(), "backward_kernel"));
  }
  return FEDG_OK;
}

int mlp_forward(MlpImpl* p, const float* X, float* Y, int B) {
  MLP_TRY(mlp_reserve(p, B, false));
  MLP_TRY(mlp_sync_weights(p));
  MLP_TRY(mlp_fwd(p, X, Y, B, false));
  return mlp_hip(hipStreamSynchronize(p->stream), "sync");
}

int mlp_loss_grad(MlpImpl* p, const float* X, const float* T, int B, float* loss) {
  MLP_TRY(mlp_reserve(p, B, true));
  MLP_TRY(mlp_sync_weights(p));
  MLP_TRY(mlp_fwd(p, X, p->act[p->nl], B, true));
  const int N = p->dims[p->nl];
  const long n = (long)B * N;
  hipLaunchKernelGGL(mse_kernel, dim3(256 + (unsigned)((size_t)(pad32(B) / 32) * (pad32(N) / 32))), dim3(256), 0, p->stream,
                     p->act[p->nl], T, p->dact[p->nl], p->dzb[0], p->dzbt[0], B, N, p->partial);
  MLP_TRY(mlp_hip(hipGetLastError(), "mse_kernel"));
  MLP_TRY(mlp_bwd(p, B));
  MLP_TRY(mlp_hip(hipStreamSynchronize(p->stream), "sync"));
  double s = 0.0;
  for (int b = 0; b < 256; ++b) s += p->partial[b];
  if (loss) *loss = (float)(s / (double)n);
  return FEDG_OK;
}

int mlp_adam(MlpImpl* p, float lr, float b1, float b2, float eps) {
  p->step += 1;
  const float c1 = 1.f - std::pow(b1, (float)p->step), c2 = 1.f - std::pow(b2, (float)p->step);
  hipLaunchKernelGGL(adam_kernel, dim3(nblk(p->nparam, 256)), dim3(256), 0, p->stream, p->params, p->grads, p->m,
                     p->v, p->nparam, lr, b1, b2, eps, c1, c2, p->lay);
  MLP_TRY(mlp_hip(hipGetLastError(), "adam_kernel"));
  p->packed = true;
  return FEDG_OK;
}

long mlp_param_count(const MlpImpl* p) { return p->nparam; }
int mlp_get(MlpImpl* p, float* params_host, float* grads_host) {
  MLP_TRY(mlp_hip(hipStreamSynchronize(p->stream), "sync"));
  if (params_host) MLP_TRY(mlp_hip(hipMemcpy(params_host, p->params, sizeof(float) * p->nparam, hipMemcpyDeviceToHost), "copy"));
  if (grads_host) MLP_TRY(mlp_hip(hipMemcpy(grads_host, p->grads, sizeof(float) * p->nparam, hipMemcpyDeviceToHost), "copy"));
  return FEDG_OK;
}
int mlp_set(MlpImpl* p, const float* params_host) {
  MLP_TRY(mlp_hip(hipStreamSynchronize(p->stream), "sync"));
  MLP_TRY(mlp_hip(hipMemcpy(p->params, params_host, sizeof(float) * p->nparam, hipMemcpyHostToDevice), "copy"));
  MLP_TRY(mlp_hip(hipMemset(p->m, 0, sizeof(float) * p->nparam), "memset"));
  MLP_TRY(mlp_hip(hipMemset(p->v, 0, sizeof(float) * p->nparam), "memset"));
  p->step = 0;
  p->packed = false;
  return FEDG_OK;
}
int mlp_dims(const MlpImpl* p, int* n_in, int* n_out) {
  if (n_in) *n_in = p->dims[0];
  if (n_out) *n_out = p->dims[p->nl];
  return FEDG_OK;
}
hipStream_t mlp_stream(const MlpImpl* p) { return p->stream; }

}  // namespace fedg
