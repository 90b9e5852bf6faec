// MLP cost model (include/op2amd_costmodel.h): forward, backward and Adam as
// HIP kernels.  Every product of the forward and backward passes (the dense
// layers, the weight and bias gradients, the back-propagated deltas) runs on
// the matrix cores (v_mfma_f32_16x16x4f32, FP32 in and out); the weight
// gradients, which reduce over the samples, are split over the samples in
// fixed chunks whose partials are summed in chunk order, so the gradients are
// deterministic.
//
// Networks of 64 hidden units and up to 64 inputs (the cost model's has 22) run an epoch as three launches instead of thirteen: k_rows takes 16
// samples per wave through the forward pass, the loss gradient and both
// backward products with every operand in LDS, k_wgrads forms the weight
// gradients' partials of all three layers, k_adam sums them and steps.
// Launches bound the thirteen (8 us each, most under 2 us of work).  Every
// output goes through the same matrix instructions in the same order in both
// forms: the same bits.  2,371 samples, per epoch: 106 us
// in thirteen launches, 23 in three (k_rows 12.7, k_wgrads 7.2, k_adam 4.0).
#include "op2amd_costmodel.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <type_traits>
#include <vector>

#define MCHECK(x)                                                            \
  do {                                                                       \
    hipError_t e_ = (x);                                                     \
    if (e_ != hipSuccess) {                                                  \
      printf("op2hip mlp: %s failed at %s:%d: %s\n", #x, __FILE__, __LINE__, \
             hipGetErrorString(e_));                                         \
      exit(-1);                                                              \
    }                                                                        \
  } while (0)

struct op2amd_mlp {
  int nin, H, np;
  float *P = nullptr, *G = nullptr, *M = nullptr, *V = nullptr;  // device
  // device work buffers, grown on demand
  int cap = 0;
  float *X = nullptr, *T = nullptr, *Z1 = nullptr, *A1 = nullptr, *Z2 = nullptr,
        *A2 = nullptr, *Y = nullptr, *DY = nullptr, *D2 = nullptr, *D1 = nullptr,
        *PK = nullptr, *loss = nullptr;  // PK: split partials of the gradients
  int adam_t = 0;
  float wd = 0.f;  // decoupled weight decay
  float *host = nullptr;  // pinned, host_cap values: small forward passes' x and y
  size_t host_cap = 0;
  hipStream_t st = nullptr;
  // parameter offsets
  int oW1, ob1, oW2, ob2, oW3, ob3;
};

namespace {

int blocks(long long n, int bs) { return (int)((n + bs - 1) / bs); }

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kSplit = 256;  // samples per split of a weight-gradient product

int splits_for(int n) { return (n + kSplit - 1) / kSplit; }

// C(m, n) = sum over k of a(m, k) b(k, n), k in split blockIdx.z's range
// [z kchunk, (z + 1) kchunk) of [0, K), with
//   a(m, k) = A[m sam + k sak] for m < ma, 1 for ma <= m < M (a row of ones
//             gives the bias gradient next to the weight gradient),
//   b(k, n) = B[k sbk + n sbn],
// on the matrix cores: each wave one 16x16 tile of C, four k per
// v_mfma_f32_16x16x4f32 (A operand: lane l holds a(l % 16, l / 16); B
// operand: b(l / 16, l % 16); result: lane l, element v holds
// C(4 (l / 16) + v, l % 16)).  Operands outside the matrices are zeros.
// Epilogue: EP 0 stores split z's partial at C + z M N; EP 1 stores
// Z = C + bias[n] and, when R is given, R = relu(Z); EP 2 stores C where
// mask(m, n) > 0, else 0.  C, R and mask are row-major M x N.
template <int EP>
__global__ void __launch_bounds__(256)
    k_gemm(const float *__restrict A, int sam, int sak, int ma, const float *__restrict B,
           int sbk, int sbn, float *__restrict C, float *__restrict R,
           const float *__restrict aux, int M, int N, int K, int kchunk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i0 = (blockIdx.x * 4 + wave) * 16, j0 = blockIdx.y * 16;
  if (i0 >= M) return;  // the whole wave: no barriers below
  const int k_lo = blockIdx.z * kchunk, k_hi = min(K, k_lo + kchunk);
  const int ia = i0 + (lane & 15), kk = lane >> 4, jb = j0 + (lane & 15);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = k_lo; k0 < k_hi; k0 += 4) {
    const int k = k0 + kk;
    float a = 0.f, b = 0.f;
    if (k < k_hi) {
      if (ia < ma)
        a = A[(size_t)ia * sam + (size_t)k * sak];
      else if (ia < M)
        a = 1.f;
      if (jb < N) b = B[(size_t)k * sbk + (size_t)jb * sbn];
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0);
  }
  const int j = j0 + (lane & 15);
  if (j >= N) return;
  for (int v = 0; v < 4; ++v) {
    const int i = i0 + 4 * (lane >> 4) + v;
    if (i >= M) break;
    const size_t o = (size_t)i * N + j;
    if (EP == 0) {
      C[(size_t)blockIdx.z * M * N + o] = acc[v];
    } else if (EP == 1) {
      const float z = acc[v] + aux[j];
      C[o] = z;
      if (R) R[o] = z > 0.f ? z : 0.f;
    } else {
      C[o] = aux[o] > 0.f ? acc[v] : 0.f;
    }
  }
}

// out[i] = sum over splits z, in order, of P[z MN + i]
__global__ void k_split_sum(const float *__restrict P, int splits, int MN,
                            float *__restrict out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= MN) return;
  float s = P[i];
  for (int z = 1; z < splits; ++z) s += P[(size_t)z * MN + i];
  out[i] = s;
}

// ---- small networks: whole rows per wave ----
constexpr int kHidden = 64, kMaxInputs = 64;
// LDS rows of 64 values: 4 banks on from the last, so 16 rows of 4 values (an
// operand read down a column) meet no bank twice; W1, read only along rows of
// 16 values, 16 banks on
constexpr int kRowStride = 68, kW1Stride = 80;
constexpr int kRowWaves = 2;          // waves (of 16 samples) per workgroup
// Forward passes of up to so many values of x read them from, and write y to,
// pinned host memory instead of copying both ways: 21.5 us against 39.9 at 23
// rows of 22 values, 30.2 against 46.5 at 2,979; at 5,958 the copies are level
// (54.3 against 53.5), each workgroup's reads being one trip over the link.
constexpr long long kHostInputs = 65536;

// How k_rows and k_wgrads see the parameters.
struct Net {
  int nin, H, np, oW1, ob1, oW2, ob2, oW3, ob3;
};

// NT 16x16 tiles side by side: rows of `a` (LDS, stride kRowStride) times
// B(k, n) = W[k sk + n sn] (LDS), tile t's column n = 16 t + lane % 16, k < K
// (a multiple of four), four k per instruction in ascending order as k_gemm.
// The tiles share their rows' operand and keep the matrix core busy over one
// another's latency.
template <int NT>
__device__ __forceinline__ void tiles_product(const float *a, const float *W, int sk, int sn,
                                              int K, int lane, f32x4 *acc) {
  const int row = lane & 15, kk = lane >> 4;
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const float *ak = a + row * kRowStride + kk, *wk = W + kk * sk + row * sn;
  auto steps = [&](auto count) {  // that many steps, their operands read first
    constexpr int S = decltype(count)::value;
    float av[S], bv[S][NT];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      av[s] = ak[4 * s];
#pragma unroll
      for (int t = 0; t < NT; ++t) bv[s][t] = wk[4 * s * sk + 16 * t * sn];
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], bv[s][t], acc[t], 0, 0, 0);
    ak += 4 * S;
    wk += 4 * S * sk;
  };
  int k = 0;
  for (; k + 16 <= K; k += 16) steps(std::integral_constant<int, 4>());
  for (; k < K; k += 4) steps(std::integral_constant<int, 1>());
}

// LDS written by a lane of this wave before and read by another after (or read
// before and written after): the hardware keeps a wave's LDS accesses in order,
// the fences make the compiler do so too.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// 16 samples per wave: Y, and with BACK the samples' A1, A2, DY, D2 and D1,
// which the weight gradients are formed from.  The parameters and the rows'
// activations stay in LDS (25 KiB and 8.5 KiB a wave for the cost model's).  X and Y may be pinned
// host memory.  Rows past n hold zeros and are not stored.
template <bool BACK>
__global__ void __launch_bounds__(64 * kRowWaves)
    k_rows(Net g, const float *__restrict P, const float *X, const float *__restrict T, float *Y,
           float *__restrict A1, float *__restrict A2, float *__restrict DY,
           float *__restrict D2, float *__restrict D1, int n) {
  extern __shared__ float lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, r4 = 4 * (lane >> 4);
  const int i0 = (blockIdx.x * kRowWaves + wave) * 16;
  constexpr unsigned H = kHidden;  // (unsigned: rows and columns by shifts)
  float *w1 = lds, *w2 = w1 + ((g.nin + 3) & ~3) * kW1Stride, *vec = w2 + H * kRowStride;  // vec: b1 b2 W3 b3
  float *u = vec + 3 * H + 4 + wave * 2 * 16 * kRowStride;  // x, then A2, then D2
  float *v = u + 16 * kRowStride;                                     // A1
  // every load is issued before the first is waited for; the parameters as
  // 16-byte pieces, 16 to a row of 64 (every block of them starts at one)
  constexpr int kT = 64 * kRowWaves, kRowQ = kHidden / 4;
  const float4 *pq = reinterpret_cast<const float4 *>(P);
  const int tid = threadIdx.x, q1 = g.nin * kRowQ;
  float4 p1[kMaxInputs * kRowQ / kT], p2[kHidden * kRowQ / kT], pv = {0.f, 0.f, 0.f, 0.f};
  float xx[16];
#pragma unroll
  for (int s = 0; s < kMaxInputs * kRowQ / kT; ++s)
    if (tid + s * kT < q1) p1[s] = pq[tid + s * kT];
#pragma unroll
  for (int s = 0; s < kHidden * kRowQ / kT; ++s) p2[s] = pq[g.oW2 / 4 + tid + s * kT];
  // b1, then b2, W3 and b3 (the allocation is padded to a whole last piece)
  if (tid <= 3 * kRowQ) pv = pq[tid < kRowQ ? g.ob1 / 4 + tid : g.ob2 / 4 + tid - kRowQ];
#pragma unroll
  for (int r = 0; r < 16; ++r)
    xx[r] = lane < g.nin && i0 + r < n ? X[(size_t)(i0 + r) * g.nin + lane] : 0.f;
#pragma unroll
  for (int s = 0; s < kMaxInputs * kRowQ / kT; ++s) {
    const int q = tid + s * kT;
    if (q < ((g.nin + 3) & ~3) * kRowQ)  // zeros past nin, up to a whole step of four
      *reinterpret_cast<float4 *>(w1 + q / kRowQ * kW1Stride + q % kRowQ * 4) =
          q < q1 ? p1[s] : float4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int s = 0; s < kHidden * kRowQ / kT; ++s) {
    const int q = tid + s * kT;
    *reinterpret_cast<float4 *>(w2 + q / kRowQ * kRowStride + q % kRowQ * 4) = p2[s];
  }
  if (tid <= 3 * kRowQ) reinterpret_cast<float4 *>(vec)[tid] = pv;
#pragma unroll
  for (int r = 0; r < 16; ++r)
    if (lane < ((g.nin + 3) & ~3)) u[r * kRowStride + lane] = xx[r];
  const float *b1 = vec, *b2 = vec + H, *w3 = vec + 2 * H, *b3 = vec + 3 * H;
  __syncthreads();
  // the waves go on apart: u and v are the wave's own, the weights are only read
  constexpr int NT = kHidden / 16;
  f32x4 acc[NT];
  tiles_product<NT>(u, w1, kW1Stride, 1, (g.nin + 3) & ~3, lane, acc);
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = 16 * t + col;
    for (int e = 0; e < 4; ++e) {
      const float z = acc[t][e] + b1[j], a = z > 0.f ? z : 0.f;
      v[(r4 + e) * kRowStride + j] = a;
      if (BACK && i0 + r4 + e < n) A1[(size_t)(i0 + r4 + e) * H + j] = a;
    }
  }
  wave_sync();
  tiles_product<NT>(v, w2, kRowStride, 1, H, lane, acc);
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = 16 * t + col;
    for (int e = 0; e < 4; ++e) {
      const float z = acc[t][e] + b2[j], a = z > 0.f ? z : 0.f;
      u[(r4 + e) * kRowStride + j] = a;
      if (BACK && i0 + r4 + e < n) A2[(size_t)(i0 + r4 + e) * H + j] = a;
    }
  }
  wave_sync();
  // one output column: the other lanes' products (of W3's neighbours) are unused
  f32x4 y;
  tiles_product<1>(u, w3, 1, 0, H, lane, &y);
  float dy[4];
  for (int e = 0; e < 4; ++e) {  // column 0's lanes hold y
    const int i = i0 + r4 + e;
    const float ye = y[e] + *b3;
    dy[e] = 0.f;
    if (col == 0 && i < n) {
      Y[i] = ye;
      if (BACK) DY[i] = dy[e] = 2.f * (ye - T[i]) / (float)n;
    }
  }
  if (!BACK) return;
  // D2 = (dy W3^T) where A2 > 0 (its Z2 > 0), over A2: lane l of the product's
  // first operand wants row l % 16's dy, which lane 16 (row / 4) holds
  const float d0 = __shfl(dy[0], (lane & 12) << 2), d1 = __shfl(dy[1], (lane & 12) << 2),
              d2 = __shfl(dy[2], (lane & 12) << 2), d3 = __shfl(dy[3], (lane & 12) << 2);
  const float dr = (lane & 3) == 0 ? d0 : (lane & 3) == 1 ? d1 : (lane & 3) == 2 ? d2 : d3;
  wave_sync();  // y's product has read u
  for (int t = 0; t < NT; ++t) {
    const int j = 16 * t + col;
    f32x4 d = {0.f, 0.f, 0.f, 0.f};
    d = __builtin_amdgcn_mfma_f32_16x16x4f32(lane < 16 ? dr : 0.f,
                                               lane < 16 ? w3[j] : 0.f, d, 0, 0, 0);
    for (int e = 0; e < 4; ++e) {
      float *a = u + (r4 + e) * kRowStride + j;
      *a = *a > 0.f ? d[e] : 0.f;
      if (i0 + r4 + e < n) D2[(size_t)(i0 + r4 + e) * H + j] = *a;
    }
  }
  wave_sync();
  // D1 = (D2 W2^T) where A1 > 0
  tiles_product<NT>(u, w2, 1, kRowStride, H, lane, acc);
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int j = 16 * t + col;
    for (int e = 0; e < 4; ++e)
      if (i0 + r4 + e < n)
        D1[(size_t)(i0 + r4 + e) * H + j] = v[(r4 + e) * kRowStride + j] > 0.f ? acc[t][e] : 0.f;
  }
}

// The weight gradients' partials of all layers: one 16x16 tile of one layer's
// [A^T; 1] D over one split of kSplit samples per workgroup (a wave), as
// k_gemm<0>: split blockIdx.x's partial of parameter q at PK[split np + q].
__global__ void __launch_bounds__(64)
    k_wgrads(Net g, const float *__restrict X, const float *__restrict A1,
             const float *__restrict A2, const float *__restrict D1,
             const float *__restrict D2, const float *__restrict DY, float *__restrict PK,
             int n) {
  const int lane = threadIdx.x, H = g.H;
  const int nt = (H + 15) / 16, t1 = ((g.nin + 16) / 16) * nt, t2 = ((H + 16) / 16) * nt;
  int t = blockIdx.y;
  const float *A = X, *D = D1;
  int K = g.nin, N = H, at = g.oW1;
  if (t >= t1 + t2) {
    t -= t1 + t2;
    A = A2;
    D = DY;
    K = H;
    N = 1;
    at = g.oW3;
  } else if (t >= t1) {
    t -= t1;
    A = A1;
    D = D2;
    K = H;
    at = g.oW2;
  }
  const int cols = (N + 15) / 16, i0 = t / cols * 16, j0 = t % cols * 16, M = K + 1;
  const int k_lo = blockIdx.x * kSplit, k_hi = min(n, k_lo + kSplit);
  const int ia = i0 + (lane & 15), kk = lane >> 4, jb = j0 + (lane & 15);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = k_lo; k0 < k_hi; k0 += 128) {
    float a[32], b[32];
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const int k = k0 + 4 * s + kk;
      a[s] = k < k_hi ? (ia < K ? A[(size_t)k * K + ia] : ia < M ? 1.f : 0.f) : 0.f;
      b[s] = k < k_hi && jb < N ? D[(size_t)k * N + jb] : 0.f;
    }
#pragma unroll
    for (int s = 0; s < 32; ++s)
      if (k0 + 4 * s < k_hi)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s], b[s], acc, 0, 0, 0);
  }
  if (jb >= N) return;
  for (int e = 0; e < 4; ++e) {
    const int i = i0 + 4 * (lane >> 4) + e;
    if (i < M) PK[(size_t)blockIdx.x * g.np + at + i * N + jb] = acc[e];
  }
}

dim3 gemm_grid(int M, int N, int splits) {
  return dim3((unsigned)(((M + 15) / 16 + 3) / 4), (unsigned)((N + 15) / 16), (unsigned)splits);
}

// DY[n] = 2 (Y[n] - T[n]) / N
__global__ void k_dloss(const float *__restrict Y, const float *__restrict T,
                        float *__restrict DY, int N) {
  int n = blockIdx.x * blockDim.x + threadIdx.x;
  if (n < N) DY[n] = 2.f * (Y[n] - T[n]) / (float)N;
}

// loss = mean (Y - T)^2, one workgroup, lanes in order then a tree
__global__ void k_loss(const float *__restrict Y, const float *__restrict T,
                       float *__restrict loss, int N) {
  __shared__ float sh[256];
  float s = 0.f;
  for (int n = threadIdx.x; n < N; n += blockDim.x) {
    float d = Y[n] - T[n];
    s += d * d;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int o = blockDim.x / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) *loss = sh[0] / (float)N;
}

// Adam with decoupled weight decay `wd` (AdamW; wd = 0 is plain Adam).
// splits > 0: G is first formed as the sum of its splits' partials PK, in order.
__global__ void k_adam(float *__restrict P, const float *__restrict G,
                       float *__restrict M, float *__restrict V, int np, float lr,
                       float c1, float c2, float wd, const float *__restrict PK, int splits) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= np) return;
  float g = splits ? PK[i] : G[i];
  for (int z0 = 1; z0 < splits; z0 += 8) {  // eight loads in flight, added in order
    float t[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) t[z] = z0 + z < splits ? PK[(size_t)(z0 + z) * np + i] : 0.f;
#pragma unroll
    for (int z = 0; z < 8; ++z)
      if (z0 + z < splits) g += t[z];
  }
  float m = 0.9f * M[i] + 0.1f * g;
  float v = 0.999f * V[i] + 0.001f * g * g;
  M[i] = m;
  V[i] = v;
  float p = P[i];
  P[i] = p - lr * (m / c1) / (sqrtf(v / c2) + 1e-8f) - lr * wd * p;
}

void ensure(op2amd_mlp *m, int n) {
  if (n <= m->cap) return;
  float **bufs[] = {&m->X, &m->T, &m->Z1, &m->A1, &m->Z2, &m->A2, &m->Y, &m->DY, &m->D2, &m->D1,
                    &m->PK};
  for (float **b : bufs)
    if (*b) MCHECK(hipFree(*b));
  const size_t H = m->H;
  MCHECK(hipMalloc(&m->X, sizeof(float) * n * m->nin));
  MCHECK(hipMalloc(&m->T, sizeof(float) * n));
  MCHECK(hipMalloc(&m->Z1, sizeof(float) * n * H));
  MCHECK(hipMalloc(&m->A1, sizeof(float) * n * H));
  MCHECK(hipMalloc(&m->Z2, sizeof(float) * n * H));
  MCHECK(hipMalloc(&m->A2, sizeof(float) * n * H));
  MCHECK(hipMalloc(&m->Y, sizeof(float) * n));
  MCHECK(hipMalloc(&m->DY, sizeof(float) * n));
  MCHECK(hipMalloc(&m->D2, sizeof(float) * n * H));
  MCHECK(hipMalloc(&m->D1, sizeof(float) * n * H));
  // split partials of the largest gradient product, (max(nin, H) + 1) x H, or
  // of all parameters (small networks)
  MCHECK(hipMalloc(&m->PK, sizeof(float) * splits_for(n) *
                               std::max((size_t)(std::max(m->nin, m->H) + 1) * H, (size_t)m->np)));
  m->cap = n;
}

// Z = A W + b (A: n x K, W: K x Mo), R = relu(Z) when R is given
void dense(op2amd_mlp *m, const float *A, int n, int K, const float *W, const float *b,
           int Mo, float *Z, float *R) {
  k_gemm<1><<<gemm_grid(n, Mo, 1), 256, 0, m->st>>>(A, K, 1, n, W, Mo, 1, Z, R, b, n, Mo, K, K);
}

// [dW; db] = [A^T; 1] D over the n samples (A: n x K, D: n x Mo) into the
// (K + 1) x Mo block G (W's gradient, then b's, as the parameters are laid out)
void wgrad(op2amd_mlp *m, const float *A, int n, int K, const float *D, int Mo, float *G) {
  const int sp = splits_for(n), M = K + 1;
  k_gemm<0><<<gemm_grid(M, Mo, sp), 256, 0, m->st>>>(A, 1, K, K, D, Mo, 1, m->PK, nullptr,
                                                       nullptr, M, Mo, n, kSplit);
  k_split_sum<<<blocks((long long)M * Mo, 256), 256, 0, m->st>>>(m->PK, sp, M * Mo, G);
}

// Din = (D W^T) where Z > 0, else 0 (D: n x Mo, W: K x Mo, Z and Din: n x K)
void back(op2amd_mlp *m, const float *D, int n, int Mo, const float *W, int K, const float *Z,
          float *Din) {
  k_gemm<2><<<gemm_grid(n, K, 1), 256, 0, m->st>>>(D, Mo, 1, n, W, 1, Mo, Din, nullptr, Z, n, K,
                                                     Mo, Mo);
}

bool small_net(const op2amd_mlp *m) { return m->nin <= kMaxInputs && m->H == kHidden; }

Net net_of(const op2amd_mlp *m) {
  return Net{m->nin, m->H, m->np, m->oW1, m->ob1, m->oW2, m->ob2, m->oW3, m->ob3};
}

template <bool BACK>
void rows(op2amd_mlp *m, const float *x, float *y, int n) {
  const size_t lds = sizeof(float) * ((size_t)((m->nin + 3) & ~3) * kW1Stride + m->H * kRowStride +
                                      3 * m->H + 4 + kRowWaves * 2 * 16 * kRowStride);
  k_rows<BACK><<<blocks(n, 16 * kRowWaves), 64 * kRowWaves, lds, m->st>>>(
      net_of(m), m->P, x, m->T, y, m->A1, m->A2, m->DY, m->D2, m->D1, n);
}

void wgrads(op2amd_mlp *m, int n) {
  const int nt = (m->H + 15) / 16;
  const int tiles = ((m->nin + 16) / 16 + (m->H + 16) / 16) * nt + (m->H + 16) / 16;
  k_wgrads<<<dim3(splits_for(n), tiles), 64, 0, m->st>>>(net_of(m), m->X, m->A1, m->A2, m->D1,
                                                        m->D2, m->DY, m->PK, n);
}

void forward(op2amd_mlp *m, int n) {
  const int H = m->H;
  float *P = m->P;
  if (small_net(m)) {
    rows<false>(m, m->X, m->Y, n);
    return;
  }
  dense(m, m->X, n, m->nin, P + m->oW1, P + m->ob1, H, m->Z1, m->A1);
  dense(m, m->A1, n, H, P + m->oW2, P + m->ob2, H, m->Z2, m->A2);
  dense(m, m->A2, n, H, P + m->oW3, P + m->ob3, 1, m->Y, nullptr);
}

void backward(op2amd_mlp *m, int n) {
  const int H = m->H;
  float *P = m->P, *G = m->G;
  k_dloss<<<blocks(n, 256), 256, 0, m->st>>>(m->Y, m->T, m->DY, n);
  wgrad(m, m->A2, n, H, m->DY, 1, G + m->oW3);
  back(m, m->DY, n, 1, P + m->oW3, H, m->Z2, m->D2);
  wgrad(m, m->A1, n, H, m->D2, H, G + m->oW2);
  back(m, m->D2, n, H, P + m->oW2, H, m->Z1, m->D1);
  wgrad(m, m->X, n, m->nin, m->D1, H, G + m->oW1);
}

void upload(op2amd_mlp *m, const float *x, const float *t, int n) {
  ensure(m, n);
  MCHECK(hipMemcpyAsync(m->X, x, sizeof(float) * n * m->nin, hipMemcpyHostToDevice, m->st));
  if (t) MCHECK(hipMemcpyAsync(m->T, t, sizeof(float) * n, hipMemcpyHostToDevice, m->st));
}

}  // namespace

extern "C" op2amd_mlp *op2amd_mlp_create(int nin, int hidden, uint64_t seed) {
  int ndev = 0;
  if (nin < 1 || hidden < 1 || hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0)
    return nullptr;
  op2amd_mlp *m = new op2amd_mlp();
  m->nin = nin;
  m->H = hidden;
  m->oW1 = 0;
  m->ob1 = m->oW1 + nin * hidden;
  m->oW2 = m->ob1 + hidden;
  m->ob2 = m->oW2 + hidden * hidden;
  m->oW3 = m->ob2 + hidden;
  m->ob3 = m->oW3 + hidden;
  m->np = m->ob3 + 1;
  MCHECK(hipStreamCreateWithFlags(&m->st, hipStreamNonBlocking));
  MCHECK(hipMalloc(&m->P, sizeof(float) * (m->np + 3)));  // (read in whole 16-byte pieces)
  MCHECK(hipMalloc(&m->G, sizeof(float) * m->np));
  MCHECK(hipMalloc(&m->M, sizeof(float) * m->np));
  MCHECK(hipMalloc(&m->V, sizeof(float) * m->np));
  MCHECK(hipMalloc(&m->loss, sizeof(float)));
  MCHECK(hipMemset(m->M, 0, sizeof(float) * m->np));
  MCHECK(hipMemset(m->V, 0, sizeof(float) * m->np));
  MCHECK(hipDeviceSynchronize());  // null-stream work done before m->st uses it
  // He initialisation: normal(0, sqrt(2/fan_in)) by Box-Muller on SplitMix64
  std::vector<float> p(m->np, 0.f);
  uint64_t s = seed;
  auto uni = [&]() {
    uint64_t z = (s += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return ((double)(z >> 11) + 0.5) * 0x1.0p-53;
  };
  auto normal = [&]() { return std::sqrt(-2.0 * std::log(uni())) * std::cos(2 * M_PI * uni()); };
  for (int i = 0; i < nin * hidden; ++i) p[m->oW1 + i] = (float)(normal() * std::sqrt(2.0 / nin));
  for (int i = 0; i < hidden * hidden; ++i) p[m->oW2 + i] = (float)(normal() * std::sqrt(2.0 / hidden));
  for (int i = 0; i < hidden; ++i) p[m->oW3 + i] = (float)(normal() * std::sqrt(1.0 / hidden));
  MCHECK(hipMemcpy(m->P, p.data(), sizeof(float) * m->np, hipMemcpyHostToDevice));
  return m;
}

extern "C" void op2amd_mlp_destroy(op2amd_mlp *m) {
  if (!m) return;
  float *bufs[] = {m->P, m->G, m->M, m->V, m->loss, m->X, m->T, m->Z1, m->A1,
                   m->Z2, m->A2, m->Y, m->DY, m->D2, m->D1, m->PK};
  for (float *b : bufs)
    if (b) (void)hipFree(b);
  if (m->host) (void)hipHostFree(m->host);
  if (m->st) (void)hipStreamDestroy(m->st);
  delete m;
}

extern "C" int op2amd_mlp_num_params(const op2amd_mlp *m) { return m->np; }

extern "C" int op2amd_mlp_get_params(const op2amd_mlp *m, float *out) {
  MCHECK(hipStreamSynchronize(m->st));
  MCHECK(hipMemcpy(out, m->P, sizeof(float) * m->np, hipMemcpyDeviceToHost));
  return 0;
}

extern "C" int op2amd_mlp_set_params(op2amd_mlp *m, const float *in) {
  MCHECK(hipStreamSynchronize(m->st));
  MCHECK(hipMemcpy(m->P, in, sizeof(float) * m->np, hipMemcpyHostToDevice));
  return 0;
}

extern "C" int op2amd_mlp_forward(op2amd_mlp *m, const float *x, int n, float *y) {
  if (n < 1) return 1;
  const long long in = (long long)n * m->nin;
  if (small_net(m) && in <= kHostInputs) {  // y after x
    if ((size_t)(in + n) > m->host_cap) {
      if (m->host) MCHECK(hipHostFree(m->host));
      m->host_cap = ((size_t)(in + n) + 4095) / 4096 * 4096;
      MCHECK(hipHostMalloc((void **)&m->host, sizeof(float) * m->host_cap, hipHostMallocDefault));
    }
    std::memcpy(m->host, x, sizeof(float) * in);
    rows<false>(m, m->host, m->host + in, n);
    MCHECK(hipGetLastError());
    MCHECK(hipStreamSynchronize(m->st));
    std::memcpy(y, m->host + in, sizeof(float) * n);
    return 0;
  }
  upload(m, x, nullptr, n);
  forward(m, n);
  MCHECK(hipMemcpyAsync(y, m->Y, sizeof(float) * n, hipMemcpyDeviceToHost, m->st));
  MCHECK(hipStreamSynchronize(m->st));
  return 0;
}

extern "C" int op2amd_mlp_loss_grad(op2amd_mlp *m, const float *x, const float *t, int n,
                                    float *loss, float *grad) {
  if (n < 1) return 1;
  upload(m, x, t, n);
  if (small_net(m)) {
    rows<true>(m, m->X, m->Y, n);
    wgrads(m, n);
    k_split_sum<<<blocks(m->np, 256), 256, 0, m->st>>>(m->PK, splits_for(n), m->np, m->G);
  } else {
    forward(m, n);
    backward(m, n);
  }
  k_loss<<<1, 256, 0, m->st>>>(m->Y, m->T, m->loss, n);
  MCHECK(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->st));
  MCHECK(hipMemcpyAsync(grad, m->G, sizeof(float) * m->np, hipMemcpyDeviceToHost, m->st));
  MCHECK(hipStreamSynchronize(m->st));
  return 0;
}

extern "C" int op2amd_mlp_set_weight_decay(op2amd_mlp *m, float wd) {
  if (!m || wd < 0.f) return 1;
  m->wd = wd;
  return 0;
}

extern "C" int op2amd_mlp_train(op2amd_mlp *m, const float *x, const float *t, int n,
                                int epochs, float lr, float *final_loss) {
  if (n < 1) return 1;
  upload(m, x, t, n);
  const bool small = small_net(m);
  for (int e = 0; e < epochs; ++e) {
    if (small) {
      rows<true>(m, m->X, m->Y, n);
      wgrads(m, n);
    } else {
      forward(m, n);
      backward(m, n);
    }
    ++m->adam_t;
    float c1 = 1.f - std::pow(0.9f, (float)m->adam_t);
    float c2 = 1.f - std::pow(0.999f, (float)m->adam_t);
    k_adam<<<blocks(m->np, 256), 256, 0, m->st>>>(m->P, m->G, m->M, m->V, m->np, lr, c1, c2,
                                                  m->wd, m->PK, small ? splits_for(n) : 0);
  }
  forward(m, n);
  k_loss<<<1, 256, 0, m->st>>>(m->Y, m->T, m->loss, n);
  float l = 0.f;
  MCHECK(hipMemcpyAsync(&l, m->loss, sizeof(float), hipMemcpyDeviceToHost, m->st));
  MCHECK(hipStreamSynchronize(m->st));
  if (final_loss) *final_loss = l;
  return 0;
}
