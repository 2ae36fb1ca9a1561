// Multilayer perceptron for the SCFT warm start: training (forward, backward,
// Adam) and inference on the GPU.  Weights are kept as an FP32 master copy for
// the optimiser and a BF16 copy that feeds the matrix cores; every GEMM takes
// BF16 operands (activations are rounded to BF16 when loaded) and accumulates
// in FP32 with v_mfma_f32_16x16x32_bf16.  SiLU hidden activations, linear
// output, mean-squared-error loss.  No counterpart in the reference.
#include <hip/hip_runtime.h>

#include <cmath>
#include <memory>
#include <random>
#include <type_traits>
#include <vector>

#include "../../include/cfft_hip.h"
#include "common.hpp"

using namespace cfft;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u;
  std::memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}

__device__ inline float silu(float z) { return z / (1.0f + expf(-z)); }
__device__ inline float dsilu(float z) {
  const float s = 1.0f / (1.0f + expf(-z));
  return s * (1.0f + z * (1.0f - s));
}

// Operands of C(m, n) = sum_k A(m, k) B(k, n): x is the index that C keeps (m
// or n), FP32 values are rounded to BF16 when loaded, BF16 values are used as
// stored.  A lane's fragment is kf = 8 values of k at each of its TX indices.
//   ContigK  element (x, k) at p[x * ld + k]: TX rows of 16, a lane reads 8
//            neighbours along k
//   StrideK  element (x, k) at p[k * ld + x]: a lane reads TX neighbours along
//            x in each of its 8 rows, so its TX sub-tiles interleave and 16
//            lanes cover 16 TX neighbours
// Rows of C past the edge read the last valid one and are not stored; the
// vector loads are aligned to an element only (any width, any offset).
constexpr int kf = 8, kChunk = 32, kMaxWaves = 8;

template <typename T, int TX>
struct ContigK {
  static constexpr int tx = TX;
  using Elem = T;
  const T* p;
  long ld;
  __device__ static int at(int x0, int i, int r, int) { return x0 + 16 * i + r; }
  __device__ static bool own(int x0, int i, int r, int X) { return x0 + 16 * i + r < X; }
  template <bool TAIL>
  __device__ __forceinline__ void load(T (&v)[TX][kf], int x0, int r, int X, int k, int K) const {
    typedef T Vec __attribute__((ext_vector_type(kf), aligned(sizeof(T))));
#pragma unroll
    for (int i = 0; i < TX; ++i) {
      const T* q = p + (long)min(x0 + 16 * i + r, X - 1) * ld;
      if constexpr (TAIL) {
#pragma unroll
        for (int j = 0; j < kf; ++j) {
          const T u = q[min(k + j, K - 1)];
          v[i][j] = k + j < K ? u : T(0);
        }
      } else {
        const Vec u = *reinterpret_cast<const Vec*>(q + k);
#pragma unroll
        for (int j = 0; j < kf; ++j) v[i][j] = u[j];
      }
    }
  }
};

template <typename T, int TX>
struct StrideK {
  static constexpr int tx = TX;
  using Elem = T;
  const T* p;
  long ld;
  // needs X >= TX: the last lane's neighbours start at X - TX at most
  __device__ static int at(int x0, int i, int r, int X) { return min(x0 + TX * r, X - TX) + i; }
  __device__ static bool own(int x0, int i, int r, int X) { return at(x0, i, r, X) >= x0 + TX * r; }
  template <bool TAIL>
  __device__ __forceinline__ void load(T (&v)[TX][kf], int x0, int r, int X, int k, int K) const {
    typedef T Vec __attribute__((ext_vector_type(TX), aligned(sizeof(T))));
    const T* q = p + min(x0 + TX * r, X - TX);
#pragma unroll
    for (int j = 0; j < kf; ++j) {
      const Vec u = *reinterpret_cast<const Vec*>(q + (long)(TAIL ? min(k + j, K - 1) : k + j) * ld);
#pragma unroll
      for (int i = 0; i < TX; ++i) v[i][j] = !TAIL || k + j < K ? u[i] : T(0);
    }
  }
};

__device__ __forceinline__ short to_bf(float v) { return (short)f2bf(v); }
__device__ __forceinline__ short to_bf(uint16_t v) { return (short)v; }

template <int TX, typename T>
__device__ __forceinline__ void frag(s16x8 (&f)[TX], const T (&v)[TX][kf]) {
#pragma unroll
  for (int i = 0; i < TX; ++i) {
#pragma unroll
    for (int j = 0; j < kf; ++j) f[i][j] = to_bf(v[i][j]);
  }
}

// Epilogues of C = A B (M x N):
//   GRAD       out0 = C (weight gradient); out1 = sum_k B(k, n) (bias gradient)
//   BIAS_SILU  out0 = Z = C + b, out1 = silu(Z)
//   BIAS       out0 = C + b
//   MSE        Y = C + b, out0 = 2 (Y - aux) * scale; part[block] = sum (Y - aux)^2
//   DSILU      out0 = C * silu'(aux) (backward)
enum { EP_GRAD, EP_BIAS_SILU, EP_BIAS, EP_MSE, EP_DSILU };

struct Ep {
  float* out0;
  float* out1;
  const float* bias;  // N
  const float* aux;   // M x N, row-major
  double* part;
  long ldo;  // row stride of out0 / out1 / aux
  float scale;
};

// One workgroup per tile of 16 TM x 16 TN; its waves take the chunks of 32
// along k in turn, one v_mfma_f32_16x16x32_bf16 per sub-tile and chunk, and
// their partial tiles are added in LDS in wave order.  A batch of tens of rows
// against layers of hundreds leaves some hundred tiles, so the time is one
// chain of loads: splitting k keeps that chain at two chunks for K = 512, and
// each lane's loads are vectors without a branch.  64 rows, 512 x 512 layer:
// 27 -> 4.1 us (one wave per tile and 2-byte loads in one chain over k before),
// weight gradient with its column sums 42 -> 5.0 us.  An empty kernel takes 2.
// Lane l of the MFMA holds A(row l%16, k 8(l/16)+j), B(k 8(l/16)+j, col l%16),
// j < 8, and D(row 4(l/16)+j, col l%16), j < 4.
struct Shape {
  int M, N, K;
};

template <int T>
struct GemmLds {
  float red[kMaxWaves][T][4][64];
  float csum[kMaxWaves][2][16];
  double lsum[kMaxWaves];
};

template <int EP, typename OA, typename OB, int T>
__device__ __forceinline__ void gemm_tile(const OA& A, const OB& B, const Shape& sh, const Ep& ep, unsigned tile,
                                          GemmLds<T>& lds) {
  constexpr int TM = OA::tx, TN = OB::tx;
  static_assert(TM * TN <= T && TN <= 2, "sub-tiles");
  auto& red = lds.red;
  auto& csum = lds.csum;
  auto& lsum = lds.lsum;
  const int M = sh.M, N = sh.N, K = sh.K;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int nw = min((int)(blockDim.x >> 6), (K + kChunk - 1) / kChunk);  // waves with a chunk
  const int tiles_n = (N + 16 * TN - 1) / (16 * TN);
  const int m0 = (int)(tile / tiles_n) * 16 * TM, n0 = (int)(tile % tiles_n) * 16 * TN;
  const int r = lane & 15, kl = (lane >> 4) * kf;
  const bool sum_b = EP == EP_GRAD && m0 == 0;
  f32x4 acc[TM][TN] = {};
  float cs[TN] = {};
  auto chunk = [&](auto tail, int k0) {
    typename OA::Elem va[TM][kf];
    typename OB::Elem vb[TN][kf];
    A.template load<decltype(tail)::value>(va, m0, r, M, k0 + kl, K);
    B.template load<decltype(tail)::value>(vb, n0, r, N, k0 + kl, K);
    if constexpr (EP == EP_GRAD) {
      if (sum_b) {
#pragma unroll
        for (int i = 0; i < TN; ++i) {
#pragma unroll
          for (int j = 0; j < kf; ++j) cs[i] += vb[i][j];
        }
      }
    }
    s16x8 a[TM], b[TN];
    frag(a, va);
    frag(b, vb);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[i]),
                                                            __builtin_bit_cast(bf16x8, b[j]), acc[i][j], 0, 0, 0);
      }
    }
  };
  const int full = K / kChunk;
  if (wave < nw) {
#pragma unroll 2
    for (int c = wave; c < full; c += nw) chunk(std::false_type{}, c * kChunk);
    if (full * kChunk < K && full % nw == wave) chunk(std::true_type{}, full * kChunk);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) red[wave][i * TN + j][q][lane] = acc[i][j][q];
      }
    }
  }
  if constexpr (EP == EP_GRAD) {
    if (sum_b && wave < nw) {
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        cs[i] += __shfl_xor(cs[i], 16);
        cs[i] += __shfl_xor(cs[i], 32);
        if (lane < 16) csum[wave][i][lane] = cs[i];
      }
    }
  }
  __syncthreads();
  double loss = 0.0;
  for (int e = threadIdx.x; e < 256 * TM * TN; e += blockDim.x) {
    const int t = e >> 8, q = (e >> 6) & 3, rm = 4 * ((e & 63) >> 4) + q, rn = e & 15;
    float v = 0.f;
    for (int w = 0; w < nw; ++w) v += red[w][t][q][e & 63];
    if (!OA::own(m0, t / TN, rm, M) || !OB::own(n0, t % TN, rn, N)) continue;
    const int row = OA::at(m0, t / TN, rm, M), col = OB::at(n0, t % TN, rn, N);
    const long o = (long)row * ep.ldo + col;
    if constexpr (EP == EP_GRAD) {
      ep.out0[o] = v;
    } else if constexpr (EP == EP_DSILU) {
      ep.out0[o] = v * dsilu(ep.aux[o]);
    } else {
      v += ep.bias[col];
      if constexpr (EP == EP_MSE) {
        const float d = v - ep.aux[o];
        ep.out0[o] = 2.0f * d * ep.scale;
        loss += (double)d * d;
      } else {
        ep.out0[o] = v;
        if constexpr (EP == EP_BIAS_SILU) ep.out1[o] = silu(v);
      }
    }
  }
  if constexpr (EP == EP_GRAD) {
    if (sum_b) {
      for (int e = threadIdx.x; e < 16 * TN; e += blockDim.x) {
        float v = 0.f;
        for (int w = 0; w < nw; ++w) v += csum[w][e >> 4][e & 15];
        if (OB::own(n0, e >> 4, e & 15, N)) ep.out1[OB::at(n0, e >> 4, e & 15, N)] = v;
      }
    }
  }
  if constexpr (EP == EP_MSE) {
    for (int d = 1; d < 64; d <<= 1) loss += __shfl_xor(loss, d);
    if (lane == 0) lsum[wave] = loss;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < (int)(blockDim.x >> 6); ++w) loss += lsum[w];
      ep.part[tile] = loss;
    }
  }
}

template <int EP, typename OA, typename OB>
__global__ void __launch_bounds__(64 * kMaxWaves) k_gemm(OA A, OB B, Shape sh, Ep ep) {
  __shared__ GemmLds<OA::tx * OB::tx> lds;
  gemm_tile<EP>(A, B, sh, ep, blockIdx.x, lds);
}

// Backward of one layer, both products in one launch (they only share dZ): the
// first `n_w` workgroups take tiles of the weight gradient, the others those of
// the input's gradient.
template <typename OW, typename OD>
__global__ void __launch_bounds__(64 * kMaxWaves) k_back(OW in, OW dz, Shape shw, Ep epw, unsigned n_w,
                                                         ContigK<float, 1> dzk, OD w, Shape shd, Ep epd) {
  __shared__ GemmLds<OW::tx * OW::tx> lds;
  if (blockIdx.x < n_w) gemm_tile<EP_GRAD>(in, dz, shw, epw, blockIdx.x, lds);
  else gemm_tile<EP_DSILU>(dzk, w, shd, epd, blockIdx.x - n_w, lds);
}

// Adam on the FP32 master parameters; refreshes the BF16 copy.
__global__ void k_adam(float* __restrict__ w, uint16_t* __restrict__ wb, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ v, long n, float lr, float b1, float b2,
                       float eps, float c1, float c2) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
}

__global__ void k_to_bf16(const float* __restrict__ w, uint16_t* __restrict__ wb, long n) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i < n) wb[i] = f2bf(w[i]);
}

// Device words into mapped host memory, four per thread as 16-byte stores.
__global__ void __launch_bounds__(256) k_words(const float* __restrict__ src, float* __restrict__ dst, long n) {
  const long i = 4 * (blockIdx.x * 256L + threadIdx.x);
  typedef float Vec __attribute__((ext_vector_type(4), aligned(4)));
  if (i + 4 <= n) {
    *reinterpret_cast<f32x4*>(dst + i) = *reinterpret_cast<const Vec*>(src + i);
  } else {
    for (long j = i; j < n; ++j) dst[j] = src[j];
  }
}

__global__ void k_gather_rows(const float* __restrict__ src, const int* __restrict__ idx, float* __restrict__ dst,
                              int rows, int cols) {
  const long i = blockIdx.x * (long)blockDim.x + threadIdx.x;
  if (i >= (long)rows * cols) return;
  const int r = (int)(i / cols), c = (int)(i % cols);
  dst[i] = src[(long)idx[r] * cols + c];
}

}  // namespace

namespace {

long tiles(long n, int w) { return (n + w - 1) / w; }

// Page-locked host memory.  Copies of the caller's pageable arrays go through
// it in pieces, written by a kernel: 2.6 MB of gradients take 110 us this way
// (one piece copied to the caller while the next is written), 220 us as an
// asynchronous copy of the runtime.  Pieces of 256 KiB, 512 KiB and 1 MiB
// measured 207, 178 and 224 us for the whole gradient call.
struct HostBuf {
  void* p = nullptr;
  void alloc(size_t n) {
    release();
    hip_check(hipHostMalloc(&p, n, hipHostMallocDefault), "hipHostMalloc");
  }
  void release() {
    if (p) (void)hipHostFree(p);
    p = nullptr;
  }
  ~HostBuf() { release(); }
};
constexpr int kSlots = 4;
constexpr size_t kSlot = 512 << 10;

}  // namespace

struct cfft_mlp {
  int L = 0;                 // weight layers
  std::vector<int> dims;     // L + 1
  std::vector<long> woff, boff;
  long n_params = 0;         // weights then biases, all layers
  int max_rows = 0;
  DevBuf w, wb, g, m, v;     // FP32 master, BF16 copy, gradient, Adam moments
  DevBuf Z, H;               // per layer pre/post activations (max_rows x dims[l+1])
  DevBuf dA, dB;             // backward ping-pong (max_rows x max dim)
  DevBuf X, T, xt;           // training set; the batch's inputs, then its targets
  HostBuf part;              // squared error per tile of the output layer, written by the kernel
  HostBuf stage;             // kSlots pieces of kSlot bytes between the caller's arrays and the device
  hipEvent_t slot_done[kSlots] = {};
  long n_data = 0;
  long step = 0;
  hipStream_t stream = nullptr;
  std::vector<long> zoff;
  ~cfft_mlp() {
    for (hipEvent_t e : slot_done)
      if (e) (void)hipEventDestroy(e);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

void ensure_rows(cfft_mlp* p, int rows) {
  if (rows <= p->max_rows) return;
  p->max_rows = 0;  // until every buffer is there: a failed allocation leaves some without memory
  long tot = 0;
  p->zoff.assign(p->L + 1, 0);
  for (int l = 0; l < p->L; ++l) {
    p->zoff[l] = tot;
    tot += (long)rows * p->dims[l + 1];
  }
  p->zoff[p->L] = tot;
  p->Z.alloc(4 * tot);
  p->H.alloc(4 * tot);
  int dmax = 0;
  for (int d : p->dims) dmax = std::max(dmax, d);
  p->dA.alloc(4L * rows * dmax);
  p->dB.alloc(4L * rows * dmax);
  p->xt.alloc(4L * rows * (p->dims[0] + p->dims[p->L]));
  p->part.alloc(8L * tiles(rows, 16) * tiles(p->dims[p->L], 16));
  p->max_rows = rows;
}

float* Zl(cfft_mlp* p, int l) { return static_cast<float*>(p->Z.p) + p->zoff[l]; }
float* Hl(cfft_mlp* p, int l) { return static_cast<float*>(p->H.p) + p->zoff[l]; }
const uint16_t* Wb(cfft_mlp* p, int l) { return static_cast<const uint16_t*>(p->wb.p) + p->woff[l]; }
const float* Bias(cfft_mlp* p, int l) { return static_cast<const float*>(p->w.p) + p->boff[l]; }

// Launches one GEMM; returns its workgroup count.
template <int EP, typename OA, typename OB>
int gemm(cfft_mlp* p, OA A, OB B, int M, int N, int K, const Ep& ep) {
  const long grid = tiles(M, 16 * OA::tx) * tiles(N, 16 * OB::tx);
  const int waves = (int)std::min<long>(kMaxWaves, tiles(K, kChunk));
  hipLaunchKernelGGL((k_gemm<EP, OA, OB>), dim3((unsigned)grid), dim3(64 * waves), 0, p->stream, A, B,
                     Shape{M, N, K}, ep);
  hip_check(hipGetLastError(), "k_gemm");
  return (int)grid;
}

// Both products of layer l's backward: dW_l = in^T dZ (K x N) with db_l = column
// sums of dZ, and dZ_{l-1} = (dZ_l W_l^T) * silu'(Z_{l-1}) (rows x K) unless l = 0.
template <int TX>
void back(cfft_mlp* p, int l, const float* in, const float* dz, float* dz_in, int rows) {
  const int K = p->dims[l], N = p->dims[l + 1];
  float* g = static_cast<float*>(p->g.p);
  const StrideK<float, TX> A{in, K}, B{dz, N};
  Ep ew{};
  ew.out0 = g + p->woff[l];
  ew.out1 = g + p->boff[l];
  ew.ldo = N;
  if (l == 0) {
    gemm<EP_GRAD>(p, A, B, K, N, rows, ew);
    return;
  }
  Ep ed{};
  ed.out0 = dz_in;
  ed.aux = Zl(p, l - 1);
  ed.ldo = K;
  const ContigK<float, 1> D{dz, N};
  const ContigK<uint16_t, 1> W{Wb(p, l), N};
  const long nw = tiles(K, 16 * TX) * tiles(N, 16 * TX), nd = tiles(rows, 16) * tiles(K, 16);
  const int waves = (int)std::min<long>(kMaxWaves, tiles(std::max(rows, N), kChunk));
  hipLaunchKernelGGL((k_back<StrideK<float, TX>, ContigK<uint16_t, 1>>), dim3((unsigned)(nw + nd)), dim3(64 * waves),
                     0, p->stream, A, B, Shape{K, N, rows}, ew, (unsigned)nw, D, W, Shape{rows, K, N}, ed);
  hip_check(hipGetLastError(), "k_back");
}

// Enqueues the caller's array `src` to the device, through the staging pieces
// at byte `at` where it fits (the stream is idle when a call begins).
void copy_in(cfft_mlp* p, void* dst, const void* src, size_t bytes, size_t at) {
  if (at + bytes <= kSlots * kSlot) {
    char* h = static_cast<char*>(p->stage.p) + at;
    std::memcpy(h, src, bytes);
    src = h;
  }
  hip_check(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, p->stream), "H2D");
}

// Device array to the caller's, through the staging pieces in turn; the stream's
// work is done on return.
void copy_out(cfft_mlp* p, float* dst, const void* src, size_t bytes) {
  const size_t n = (bytes + kSlot - 1) / kSlot;
  auto part = [&](size_t i) { return std::min(kSlot, bytes - i * kSlot); };
  auto slot = [&](size_t i) { return static_cast<float*>(p->stage.p) + (i % kSlots) * (kSlot / 4); };
  auto fetch = [&](size_t i) {
    const long words = (long)part(i) / 4;
    hipLaunchKernelGGL(k_words, dim3(nblk(words, 1024)), dim3(256), 0, p->stream,
                       static_cast<const float*>(src) + i * (kSlot / 4), slot(i), words);
    hip_check(hipGetLastError(), "k_words");
    hip_check(hipEventRecord(p->slot_done[i % kSlots], p->stream), "hipEventRecord");
  };
  for (size_t i = 0; i < std::min<size_t>(n, kSlots); ++i) fetch(i);
  for (size_t i = 0; i < n; ++i) {
    hip_check(hipEventSynchronize(p->slot_done[i % kSlots]), "hipEventSynchronize");
    std::memcpy(dst + i * (kSlot / 4), slot(i), part(i));
    if (i + kSlots < n) fetch(i + kSlots);
  }
}

// Layer l on `rows` inputs at `in`; W of layer l is K x N row-major.
template <int EP>
int layer(cfft_mlp* p, int l, const float* in, int rows, Ep ep) {
  const int K = p->dims[l], N = p->dims[l + 1];
  ep.bias = Bias(p, l);
  ep.ldo = N;
  const ContigK<float, 1> A{in, K};
  return N >= 2 ? gemm<EP>(p, A, StrideK<uint16_t, 2>{Wb(p, l), N}, rows, N, K, ep)
                : gemm<EP>(p, A, StrideK<uint16_t, 1>{Wb(p, l), N}, rows, N, K, ep);
}

// The hidden layers on `rows` inputs at x; returns the last layer's input.
const float* hidden(cfft_mlp* p, const float* x, int rows) {
  const float* in = x;
  for (int l = 0; l + 1 < p->L; ++l) {
    Ep ep{};
    ep.out0 = Zl(p, l);
    ep.out1 = Hl(p, l);
    layer<EP_BIAS_SILU>(p, l, in, rows, ep);
    in = Hl(p, l);
  }
  return in;
}

// Forward on `rows` inputs at x (device, rows x dims[0]); the output is Z of
// the last layer.
void forward(cfft_mlp* p, const float* x, int rows) {
  Ep ep{};
  ep.out0 = Zl(p, p->L - 1);
  layer<EP_BIAS>(p, p->L - 1, hidden(p, x, rows), rows, ep);
}

// Forward against the targets t: dY at dA and the squared errors per tile in
// `part`; returns their count.
int forward_loss(cfft_mlp* p, const float* x, const float* t, int rows) {
  Ep ep{};
  ep.out0 = static_cast<float*>(p->dA.p);
  ep.aux = t;
  ep.part = static_cast<double*>(p->part.p);
  ep.scale = 1.0f / (float)((long)rows * p->dims[p->L]);
  return layer<EP_MSE>(p, p->L - 1, hidden(p, x, rows), rows, ep);
}

// Backward from dY (rows x dims[L]) at dA; fills the gradient buffer.
void backward(cfft_mlp* p, const float* x, int rows) {
  float* cur = static_cast<float*>(p->dA.p);  // dZ of layer l
  float* nxt = static_cast<float*>(p->dB.p);
  for (int l = p->L - 1; l >= 0; --l) {
    const float* in = l == 0 ? x : Hl(p, l - 1);
    if (p->dims[l] >= 2 && p->dims[l + 1] >= 2) back<2>(p, l, in, cur, nxt, rows);
    else back<1>(p, l, in, cur, nxt, rows);
    std::swap(cur, nxt);
  }
}

// Mean squared error from the `parts` tile sums of forward_loss, once the
// stream is idle.
double mean_loss(const cfft_mlp* p, int parts, int rows) {
  const double* h = static_cast<const double*>(p->part.p);
  double s = 0.0;
  for (int i = 0; i < parts; ++i) s += h[i];
  return s / (double)((long)rows * p->dims[p->L]);
}

}  // namespace

extern "C" {

int cfft_mlp_create(int32_t n_layers, const int32_t* dims, uint64_t seed, cfft_mlp** out) {
  return guarded([&] {
    require(n_layers >= 1 && dims && out, CFFT_ERR_INVALID, "bad argument");
    *out = nullptr;
    std::lock_guard<std::recursive_mutex> guard(setup_mutex());
    std::unique_ptr<cfft_mlp> p(new cfft_mlp());
    p->L = n_layers;
    p->dims.assign(dims, dims + n_layers + 1);
    for (int d : p->dims) require(d >= 1, CFFT_ERR_INVALID, "layer widths must be positive");
    long off = 0;
    for (int l = 0; l < p->L; ++l) {
      p->woff.push_back(off);
      off += (long)p->dims[l] * p->dims[l + 1];
    }
    for (int l = 0; l < p->L; ++l) {
      p->boff.push_back(off);
      off += p->dims[l + 1];
    }
    p->n_params = off;
    hip_check(hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking), "hipStreamCreate");
    for (hipEvent_t& e : p->slot_done) {
      hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    }
    p->stage.alloc(kSlots * kSlot);
    // He-style initialisation (normal, std sqrt(2 / fan_in)), zero biases
    std::vector<float> w(p->n_params, 0.f);
    std::mt19937_64 rng(seed);
    for (int l = 0; l < p->L; ++l) {
      std::normal_distribution<float> nd(0.f, std::sqrt(2.0f / p->dims[l]));
      for (long i = 0; i < (long)p->dims[l] * p->dims[l + 1]; ++i) w[p->woff[l] + i] = nd(rng);
    }
    p->w.alloc(4 * p->n_params);
    p->wb.alloc(2 * p->n_params);
    p->g.alloc(4 * p->n_params);
    p->m.alloc(4 * p->n_params);
    p->v.alloc(4 * p->n_params);
    hip_check(hipMemcpy(p->w.p, w.data(), 4 * p->n_params, hipMemcpyHostToDevice), "upload");
    hip_check(hipMemset(p->m.p, 0, 4 * p->n_params), "memset");
    hip_check(hipMemset(p->v.p, 0, 4 * p->n_params), "memset");
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(p->n_params, 256)), dim3(256), 0, p->stream,
                       static_cast<const float*>(p->w.p), static_cast<uint16_t*>(p->wb.p), p->n_params);
    hip_check(hipStreamSynchronize(p->stream), "sync");
    *out = p.release();
  });
}

int cfft_mlp_info(const cfft_mlp* p, int64_t* n_params) {
  return guarded([&] {
    require(p && n_params, CFFT_ERR_INVALID, "null argument");
    *n_params = p->n_params;
  });
}

int cfft_mlp_get_params(cfft_mlp* p, float* out) {
  return guarded([&] {
    require(p && out, CFFT_ERR_INVALID, "null argument");
    hip_check(hipMemcpyAsync(out, p->w.p, 4 * p->n_params, hipMemcpyDeviceToHost, p->stream), "D2H");
    hip_check(hipStreamSynchronize(p->stream), "sync");
  });
}

int cfft_mlp_set_params(cfft_mlp* p, const float* in) {
  return guarded([&] {
    require(p && in, CFFT_ERR_INVALID, "null argument");
    hip_check(hipMemcpyAsync(p->w.p, in, 4 * p->n_params, hipMemcpyHostToDevice, p->stream), "H2D");
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(p->n_params, 256)), dim3(256), 0, p->stream,
                       static_cast<const float*>(p->w.p), static_cast<uint16_t*>(p->wb.p), p->n_params);
    hip_check(hipMemsetAsync(p->m.p, 0, 4 * p->n_params, p->stream), "memset");
    hip_check(hipMemsetAsync(p->v.p, 0, 4 * p->n_params, p->stream), "memset");
    p->step = 0;
    hip_check(hipStreamSynchronize(p->stream), "sync");
  });
}

int cfft_mlp_forward(cfft_mlp* p, const float* x, int32_t rows, float* y) {
  return guarded([&] {
    require(p && x && y && rows >= 1, CFFT_ERR_INVALID, "bad argument");
    ensure_rows(p, rows);
    copy_in(p, p->xt.p, x, 4L * rows * p->dims[0], 0);
    forward(p, static_cast<const float*>(p->xt.p), rows);
    copy_out(p, y, Zl(p, p->L - 1), 4L * rows * p->dims[p->L]);
  });
}

int cfft_mlp_gradient(cfft_mlp* p, const float* x, const float* t, int32_t rows, double* loss, float* grad) {
  return guarded([&] {
    require(p && x && t && rows >= 1, CFFT_ERR_INVALID, "bad argument");
    ensure_rows(p, rows);
    float* xb = static_cast<float*>(p->xt.p);
    float* tb = xb + (long)rows * p->dims[0];
    const size_t nx = 4L * rows * p->dims[0], nt = 4L * rows * p->dims[p->L];
    copy_in(p, xb, x, nx, 0);
    copy_in(p, tb, t, nt, nx);
    const int parts = forward_loss(p, xb, tb, rows);
    backward(p, xb, rows);
    if (grad) copy_out(p, grad, p->g.p, 4 * p->n_params);
    else hip_check(hipStreamSynchronize(p->stream), "sync");
    const double l = mean_loss(p, parts, rows);
    if (loss) *loss = l;
  });
}

int cfft_mlp_train(cfft_mlp* p, const float* X, const float* T, int64_t n, int32_t epochs, int32_t batch,
                   float lr, uint64_t seed, double* loss_per_epoch) {
  return guarded([&] {
    require(p && X && T && n >= 1 && epochs >= 0 && batch >= 1, CFFT_ERR_INVALID, "bad argument");
    const int din = p->dims[0], dout = p->dims[p->L];
    ensure_rows(p, batch);
    p->X.alloc(4L * n * din);
    p->T.alloc(4L * n * dout);
    hip_check(hipMemcpyAsync(p->X.p, X, 4L * n * din, hipMemcpyHostToDevice, p->stream), "H2D");
    hip_check(hipMemcpyAsync(p->T.p, T, 4L * n * dout, hipMemcpyHostToDevice, p->stream), "H2D");
    std::mt19937_64 rng(seed);
    std::vector<int> perm(n);
    for (long i = 0; i < n; ++i) perm[i] = (int)i;
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    DevBuf perm_dev;
    perm_dev.alloc(4L * n);
    for (int ep = 0; ep < epochs; ++ep) {
      // the previous epoch's gathers have read the device copy before it is replaced
      hip_check(hipStreamSynchronize(p->stream), "sync");
      std::shuffle(perm.begin(), perm.end(), rng);
      hip_check(hipMemcpyAsync(perm_dev.p, perm.data(), 4L * n, hipMemcpyHostToDevice, p->stream), "H2D");
      double lsum = 0.0;
      long seen = 0;
      for (long s0 = 0; s0 < n; s0 += batch) {
        const int rows = (int)std::min<long>(batch, n - s0);
        float* xb = static_cast<float*>(p->xt.p);
        float* tb = xb + (long)rows * din;
        const int* idx = static_cast<const int*>(perm_dev.p) + s0;
        hipLaunchKernelGGL(k_gather_rows, dim3(nblk((long)rows * din, 256)), dim3(256), 0, p->stream,
                           static_cast<const float*>(p->X.p), idx, xb, rows, din);
        hipLaunchKernelGGL(k_gather_rows, dim3(nblk((long)rows * dout, 256)), dim3(256), 0, p->stream,
                           static_cast<const float*>(p->T.p), idx, tb, rows, dout);
        hip_check(hipGetLastError(), "k_gather_rows");
        const int parts = forward_loss(p, xb, tb, rows);
        backward(p, xb, rows);
        ++p->step;
        const float c1 = 1.f - std::pow(b1, (float)p->step), c2 = 1.f - std::pow(b2, (float)p->step);
        hipLaunchKernelGGL(k_adam, dim3(nblk(p->n_params, 256)), dim3(256), 0, p->stream,
                           static_cast<float*>(p->w.p), static_cast<uint16_t*>(p->wb.p),
                           static_cast<const float*>(p->g.p), static_cast<float*>(p->m.p),
                           static_cast<float*>(p->v.p), p->n_params, lr, b1, b2, eps, c1, c2);
        hip_check(hipGetLastError(), "k_adam");
        hip_check(hipStreamSynchronize(p->stream), "sync");
        lsum += mean_loss(p, parts, rows) * rows;
        seen += rows;
      }
      if (loss_per_epoch) loss_per_epoch[ep] = lsum / (double)seen;
    }
    hip_check(hipStreamSynchronize(p->stream), "sync");
  });
}

int cfft_mlp_destroy(cfft_mlp* p) {
  return guarded([&] {
    if (!p) return;
    std::lock_guard<std::recursive_mutex> guard(setup_mutex());
    if (p->stream) (void)hipStreamSynchronize(p->stream);
    delete p;
  });
}

}  // extern "C"
