// Learned Newton predictor network: an MLP with BF16 weights and activations
// and FP32 accumulation on the CDNA matrix cores, with hand-written forward,
// backward (mean masked squared error) and Adam kernels.  It has no
// counterpart in the reference: it proposes the Newton initial guess that
// OneStep::obtainPredictor (src/TimeIntegrationPKG/N_TIA_OneStep.C:135)
// computes by polynomial extrapolation, which stays the fallback.
//
// Layout (all row-major, rows = samples):
//   parameters  per layer l: W_l [out_l][in_l] then b_l [out_l]; one FP32
//               master vector, one BF16 copy (the GEMM operand), FP32
//               gradients and Adam moments of the same layout
//   activations X [rows][in] bf16; Z_l [rows][width] fp32 (pre-activation,
//               kept for the backward pass); H_l [rows][width] bf16
//   output      Y [rows][out] fp32 (last layer linear)
// Every dimension is a multiple of 64 (rows, widths) so the 64-wide tiles of
// the GEMM need no edge handling; the host checks this before each launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <random>
#include <vector>

#include "xg_internal.h"

#define HIPCHK(x)                          \
  do {                                     \
    hipError_t e_ = (x);                   \
    if (e_ != hipSuccess) return XG_E_HIP; \
  } while (0)

namespace xgm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ unsigned short f2bf(float f) {
  // round to nearest even; NaN stays NaN
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((unsigned)h << 16); }

// GELU, erf form: z * Phi(z); derivative Phi(z) + z * phi(z)
__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_d(float z) {
  return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * 0.39894228040143268f * expf(-0.5f * z * z);
}

enum Epi { EPI_F32 = 0, EPI_BIAS_F32 = 1, EPI_BIAS_GELU = 2, EPI_GELU_BWD = 3, EPI_BIAS_GELU_H = 4 };

struct GemmArgs {
  int M, N, K;
  const unsigned short* A; int lda;   // A(m,k) = TA ? A[k*lda+m] : A[m*lda+k]
  const unsigned short* B; int ldb;   // B(n,k) = TB ? B[k*ldb+n] : B[n*ldb+k]
  float* C; int ldc;                  // EPI_F32 / EPI_BIAS_F32 output; EPI_BIAS_GELU: Z
  const float* bias;
  unsigned short* H;                  // EPI_BIAS_GELU(_H: without Z, which only the backward pass reads): gelu(Z)
                                      // bf16; EPI_GELU_BWD: dZ bf16
  const float* Zin;                   // EPI_GELU_BWD: pre-activation of this layer
};

constexpr int BN = 64, BK = 64;

// Place of (row, k) in a staged tile: rows of 64 halves without padding, the
// eight 16-byte groups of a row exchanged by the row's bits so that no LDS access
// of the product meets a bank twice as often as it must: 16 consecutive rows at
// one group (operand reads) fall on 16 different quads of banks, and so do the
// rows 8 apart that a transposed operand's pairs are stored to (with rows padded
// to 72 halves those eight fell on one bank: weight gradients of 2048 rows 40 us,
// 23 now).
__device__ __forceinline__ int lds_at(int row, int k) {
  const int f = ((row >> 3) ^ (((row >> 1) & 3) << 1)) & 7;
  return row * BK + (((k >> 3) ^ f) << 3) + (k & 7);
}

// A tile of T rows (of A or B as the product reads them) by BK of k, from
// memory to registers and from there to LDS.  Straight operands are rows of
// consecutive k: 16-byte loads and stores.  Transposed ones hold consecutive
// rows per k: a thread loads eight rows at k and k + 1 and writes the pairs, so
// that loads are whole 128-byte lines and stores 4 bytes.
template <bool TR, int T>
struct Stage {
  static constexpr int N = T * BK / 8 / 256;      // 16-byte loads per thread
  u32x4 v[N];
  __device__ __forceinline__ void load(const unsigned short* p, int ld, int r0, int k0, int t) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (!TR) {
        const int r = (t >> 3) + 32 * i, k = (t & 7) * 8;
        v[i] = *reinterpret_cast<const u32x4*>(p + (size_t)(r0 + r) * ld + k0 + k);
      } else {
        const int r = (t & 7) * 8 + 64 * (i >> 1), k = (t >> 3) * 2 + (i & 1);
        v[i] = *reinterpret_cast<const u32x4*>(p + (size_t)(k0 + k) * ld + r0 + r);
      }
    }
  }
  __device__ __forceinline__ void store(unsigned short* lds, int t) const {
    if (!TR) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        *reinterpret_cast<u32x4*>(&lds[lds_at((t >> 3) + 32 * i, (t & 7) * 8)]) = v[i];
    } else {
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        const u32x4 a = v[i], b = v[i + 1];
        const int r = (t & 7) * 8 + 32 * i, k = (t >> 3) * 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // rows 2 j and 2 j + 1: (k, k + 1) side by side
          *reinterpret_cast<unsigned*>(&lds[lds_at(r + 2 * j, k)]) = __builtin_amdgcn_perm(b[j], a[j], 0x05040100u);
          *reinterpret_cast<unsigned*>(&lds[lds_at(r + 2 * j + 1, k)]) = __builtin_amdgcn_perm(b[j], a[j], 0x07060302u);
        }
      }
    }
  }
};

// C = A B^T on BM x 64 tiles (BM 64 or 128): 4 waves, each (BM / 2) x 32 as
// BM / 64 blocks of v_mfma_f32_32x32x16_bf16 (A: lane l holds row l%32, k =
// 8*(l/32)..+7; B likewise by column; D register r of lane l is row 8*(r/4) +
// 4*(l/32) + r%4, column l%32).  At these sizes a tile's chain of k steps bounds
// the product (8 to 32 steps of 64, one or two tiles per CU), so two steps are in
// flight from memory in registers while LDS holds two, with one barrier per step
// (four in flight take the registers of more tiles per CU: forward of 8192 rows
// 72 us against 75, training on 8192 rows 294 us a step against 328); and the tiles
// that share rows of A sit on one XCD (consecutive workgroups go to the eight
// XCDs in turn), so that A crosses to one L2 only.  Forward of 4096 rows (1600 ->
// 3 x 512 -> 256) 50.2 us, 78.5 with one 64 x 64 x 32 step at a time.  Every
// element accumulates k in ascending order of 16 whatever the tile, so the tile
// size does not change a result.
constexpr int kAhead = 2;
constexpr long long kWideTiles = 512;   // (the dispatch of 128-row tiles)

template <bool TA, bool TB, int EPI, int BM>
__device__ __forceinline__ void gemm_tile(const GemmArgs& g, int id, unsigned short (*As)[BM * BK],
                                          unsigned short (*Bs)[BN * BK]) {
  constexpr int MI = BM / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // workgroup id -> tile: ids id, id + 8, ... (one XCD) walk the columns of a row of tiles
  const int nt = g.N / BN, mt = g.M / BM;
  const int full = mt / 8 * 8 * nt;               // ids of whole groups of eight tile rows
  int tm, tn;
  if (id < full) {
    const int q = id / 8;
    tm = q / nt * 8 + id % 8;
    tn = q % nt;
  } else {
    tm = mt / 8 * 8 + (id - full) / nt;
    tn = (id - full) % nt;
  }
  const int m0 = tm * BM, n0 = tn * BN;
  f32x16 acc[MI] = {};
  Stage<TA, BM> sa[kAhead];
  Stage<TB, BN> sb[kAhead];
  // Loads are never skipped (past the end they repeat the last step's): a
  // branch around one makes the compiler wait for all that are in flight.
  const int klast = g.K - BK;
#pragma unroll
  for (int d = 0; d < kAhead; ++d) {
    sa[d].load(g.A, g.lda, m0, min(d * BK, klast), tid);
    sb[d].load(g.B, g.ldb, n0, min(d * BK, klast), tid);
  }
  auto multiply = [&](const unsigned short* at, const unsigned short* bt) {
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(&bt[lds_at(wn * 32 + (lane & 31), kk + 8 * (lane >> 5))]);
#pragma unroll
      for (int i = 0; i < MI; ++i) {
        const bf16x8 a =
            *reinterpret_cast<const bf16x8*>(&at[lds_at((wm * MI + i) * 32 + (lane & 31), kk + 8 * (lane >> 5))]);
        acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i], 0, 0, 0);
      }
    }
  };
  int k0 = 0;
  for (; k0 + kAhead * BK < g.K; k0 += kAhead * BK) {
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
      sa[d].store(As[d & 1], tid);
      sb[d].store(Bs[d & 1], tid);
      const int k = min(k0 + (d + kAhead) * BK, klast);
      sa[d].load(g.A, g.lda, m0, k, tid);
      sb[d].load(g.B, g.ldb, n0, k, tid);
      __syncthreads();
      multiply(As[d & 1], Bs[d & 1]);
      // (else the later steps' operands are waited for and packed here too)
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the epilogue's operands, beside the last steps
  const int col = n0 + wn * 32 + (lane & 31);
  const int row0 = m0 + wm * MI * 32 + 4 * (lane >> 5);
  float bias = 0.0f, zin[MI * 16];
  if (EPI == EPI_BIAS_F32 || EPI == EPI_BIAS_GELU || EPI == EPI_BIAS_GELU_H) bias = g.bias[col];
  if (EPI == EPI_GELU_BWD)
#pragma unroll
    for (int r = 0; r < MI * 16; ++r)
      zin[r] = g.Zin[(size_t)(row0 + (r >> 4) * 32 + 8 * ((r & 15) >> 2) + (r & 3)) * g.ldc + col];
#pragma unroll
  for (int d = 0; d < kAhead; ++d) {
    if (k0 + d * BK >= g.K) break;
    sa[d].store(As[d & 1], tid);
    sb[d].store(Bs[d & 1], tid);
    __syncthreads();
    multiply(As[d & 1], Bs[d & 1]);
  }
  // ---- epilogue
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = row0 + i * 32 + 8 * (r >> 2) + (r & 3);
      const size_t o = (size_t)row * g.ldc + col;
      const float v = acc[i][r];
      if (EPI == EPI_F32) {
        g.C[o] = v;
      } else if (EPI == EPI_BIAS_F32) {
        g.C[o] = v + bias;
      } else if (EPI == EPI_BIAS_GELU) {
        const float z = v + bias;
        g.C[o] = z;
        g.H[o] = f2bf(gelu(z));
      } else if (EPI == EPI_BIAS_GELU_H) {
        g.H[o] = f2bf(gelu(v + bias));
      } else {
        g.H[o] = f2bf(v * gelu_d(zin[i * 16 + r]));
      }
    }
}

template <bool TA, bool TB, int EPI, int BM>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) unsigned short As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BN * BK];
  gemm_tile<TA, TB, EPI, BM>(g, blockIdx.x, As, Bs);
}

// loss = sum_rows sum_j mask (y - t)^2 / count, dY = 2 mask (y - t) / count
// (bf16), per-block partial sums of the loss (deterministic two-pass sum)
__global__ void k_mse(int n, int count, const float* y, const float* t, const float* mask, unsigned short* dy,
                      double* partial) {
  __shared__ double red[256];
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double l = 0.0;
  if (i < n) {
    const float d = (y[i] - t[i]) * mask[i];
    l = (double)d * d;
    dy[i] = f2bf(2.0f * d / (float)count);
  }
  red[threadIdx.x] = l;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

// bias gradients: column sums of a bf16 [rows][N] matrix, two passes (chunks of
// 256 rows, then over chunks).  The chunk pass is bound by its loads' latency:
// eight rows in flight.
__device__ __forceinline__ void colsum_part(int rows, int N, const unsigned short* d, float* part, int bx, int by,
                                            float* red) {
  const int col = bx * 64 + (threadIdx.x & 63);
  const int r0 = by * 256 + (threadIdx.x >> 6) * 64;
  float s = 0.0f;
  // (rows are a multiple of 64: a wavefront's 64 rows all exist or none does)
  if (r0 < rows)
    for (int r = r0; r < r0 + 64; r += 8) {
      unsigned short v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = d[(size_t)(r + q) * N + col];
#pragma unroll
      for (int q = 0; q < 8; ++q) s += bf2f(v[q]);
    }
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 64) {
    const float t = red[threadIdx.x] + red[threadIdx.x + 64] + red[threadIdx.x + 128] + red[threadIdx.x + 192];
    part[(size_t)by * N + col] = t;
  }
}

// Weight gradients dW_l = d_l^T in_l and the bias gradients' chunk sums of up
// to kGroup layers in one launch, after the chain of activation gradients: a
// layer alone has 32 to 200 tiles for 256 CUs and each is a chain of rows / 64
// steps, so layers one after another left most of the chip idle (1600 -> 3 x 512
// -> 256 over 2048 rows: 87 us and four launches of column sums, 18, one after
// another; 23 together).
constexpr int kGroup = 8;
struct WgradArgs {
  int n, rows;
  int tile0[kGroup + 1], col0[kGroup + 1];   // first product tile and first column-sum block of each layer
  GemmArgs g[kGroup];
  float* part[kGroup];
};

template <int BM>
__global__ void __launch_bounds__(256) k_wgrad(WgradArgs w) {
  __shared__ __attribute__((aligned(16))) unsigned short As[2][BM * BK];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BN * BK];
  int id = blockIdx.x, l = 0;
  if (id < w.tile0[w.n]) {
    while (id >= w.tile0[l + 1]) ++l;
    gemm_tile<true, true, EPI_F32, BM>(w.g[l], id - w.tile0[l], As, Bs);
  } else {
    id -= w.tile0[w.n];
    while (id >= w.col0[l + 1]) ++l;
    id -= w.col0[l];
    const int nb = w.g[l].M / 64;
    colsum_part(w.rows, w.g[l].M, w.g[l].A, w.part[l], id % nb, id / nb, reinterpret_cast<float*>(As));
  }
}

// layer blockIdx.y: its N columns' partial sums at `off` of part, the sums at
// boff of g; the last row's first block sums the loss's partials into pinned memory
struct ColLayer { int N; long long off, boff; };
__global__ void __launch_bounds__(256) k_grad_fin(int chunks, int n_layers, const ColLayer* layers, const float* part,
                                                 float* g, int n_loss, const double* lpart, double* loss) {
  if ((int)blockIdx.y == n_layers) {
    if (blockIdx.x) return;
    __shared__ double red[256];
    double s = 0.0;
    for (int i = threadIdx.x; i < n_loss; i += 256) s += lpart[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
      if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
      __syncthreads();
    }
    if (threadIdx.x == 0) *loss = red[0];
    return;
  }
  const ColLayer L = layers[blockIdx.y];
  const int col = blockIdx.x * blockDim.x + threadIdx.x;
  if (col >= L.N) return;
  float s = 0.0f;
  for (int c = 0; c < chunks; ++c) s += part[L.off + (size_t)c * L.N + col];
  g[L.boff + col] = s;
}

// Adam on the FP32 master parameters, refreshing the BF16 copy
__global__ void k_adam(long long n, float* w, unsigned short* wb, const float* g, float* m, float* v, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  wb[i] = f2bf(wi);
}
__global__ void k_to_bf16(long long n, const float* w, unsigned short* wb) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) wb[i] = f2bf(w[i]);
}

inline unsigned nblk(long long n, unsigned b = 256) { return (unsigned)((n + b - 1) / b); }

template <class T>
struct Buf {
  T* p = nullptr;
  ~Buf() { if (p) (void)hipFree(p); }
  hipError_t alloc(size_t n) {
    if (p) { (void)hipFree(p); p = nullptr; }
    return n ? hipMalloc((void**)&p, n * sizeof(T)) : hipSuccess;
  }
};

}  // namespace xgm

using namespace xgm;

struct xg_mlp {
  int in_dim = 0, width = 0, hidden = 0, out_dim = 0, max_rows = 0;
  int n_layers = 0;                       // hidden + 1
  std::vector<int> din, dout;             // per layer
  std::vector<long long> woff, boff;      // parameter offsets
  long long n_params = 0;
  long long adam_t = 0;
  hipStream_t stream = nullptr;
  Buf<float> w, g, m, v, Y, part, Zall;
  Buf<unsigned short> wb, Hall, dH, dY;
  Buf<double> lpart;
  double* loss_sum = nullptr;             // pinned
  std::vector<ColLayer> col_layer;        // per layer: its partial column sums in `part`
  Buf<ColLayer> d_col;
  // Z_l / H_l at offset l * max_rows * width
  float* Z(int l) { return Zall.p + (size_t)l * max_rows * width; }
  unsigned short* H(int l) { return Hall.p + (size_t)l * max_rows * width; }
  // gradient with respect to layer l's output before its activation
  unsigned short* D(int l) { return l + 1 == n_layers ? dY.p : dH.p + (size_t)l * max_rows * width; }
  ~xg_mlp() {
    if (stream) (void)hipStreamDestroy(stream);
    if (loss_sum) (void)hipHostFree(loss_sum);
  }

  template <bool TA, bool TB, int EPI>
  int gemm(const GemmArgs& a) {
    if (a.M % 64 || a.N % BN || a.K % BK || a.M <= 0 || a.N <= 0 || a.K <= 0) return XG_E_ARG;
    // 128-row tiles read B half as often, but their chain per step is longer: from
    // two tiles per CU (256 of them) on (forward of 4096 rows, one per CU: 58.6 us
    // against 52 with 64-row tiles; of 8192 rows 78 against 80.5)
    if (a.M % 128 == 0 && (long long)(a.N / BN) * (a.M / 128) >= kWideTiles)
      hipLaunchKernelGGL((k_gemm<TA, TB, EPI, 128>), dim3(a.N / BN * (a.M / 128)), dim3(256), 0, stream, a);
    else
      hipLaunchKernelGGL((k_gemm<TA, TB, EPI, 64>), dim3(a.N / BN * (a.M / 64)), dim3(256), 0, stream, a);
    HIPCHK(hipGetLastError());
    return XG_OK;
  }

  // forward of `rows` samples; Y fp32; with keep, Z stays for the backward pass
  int forward(int rows, const unsigned short* X, float* Yout, bool keep) {
    return forward_on(rows, X, Yout, keep, stream);
  }
  int forward_on(int rows, const unsigned short* X, float* Yout, bool keep, hipStream_t s) {
    hipStream_t own = stream;
    stream = s;
    const int st = forward_layers(rows, X, Yout, keep);
    stream = own;
    return st;
  }
  int forward_layers(int rows, const unsigned short* X, float* Yout, bool keep) {
    const unsigned short* in = X;
    for (int l = 0; l < n_layers; ++l) {
      GemmArgs a{};
      a.M = rows; a.N = dout[l]; a.K = din[l];
      a.A = in; a.lda = din[l];
      a.B = wb.p + woff[l]; a.ldb = din[l];
      a.bias = w.p + boff[l];
      int st;
      if (l + 1 < n_layers) {
        a.C = Z(l); a.ldc = width; a.H = H(l);
        st = keep ? gemm<false, false, EPI_BIAS_GELU>(a) : gemm<false, false, EPI_BIAS_GELU_H>(a);
        in = H(l);
      } else {
        a.C = Yout; a.ldc = out_dim;
        st = gemm<false, false, EPI_BIAS_F32>(a);
      }
      if (st != XG_OK) return st;
    }
    return XG_OK;
  }

  // backward of the loss whose output gradient is in dY (bf16 [rows][out]): the
  // gradients with respect to each layer's output first, then all weights'
  int backward(int rows, const unsigned short* X) {
    for (int l = n_layers - 1; l > 0; --l) {
      // d(pre-activation of layer l-1) = (d_l W_l) * gelu'(Z_{l-1})
      GemmArgs b{};
      b.M = rows; b.N = din[l]; b.K = dout[l];
      b.A = D(l); b.lda = dout[l];
      b.B = wb.p + woff[l]; b.ldb = din[l];
      b.H = D(l - 1); b.ldc = width; b.Zin = Z(l - 1);
      const int st = gemm<false, true, EPI_GELU_BWD>(b);
      if (st != XG_OK) return st;
    }
    const int chunks = (rows + 255) / 256;
    for (int l0 = 0; l0 < n_layers; l0 += kGroup) {
      WgradArgs w{};
      w.n = std::min(kGroup, n_layers - l0);
      w.rows = rows;
      bool wide = true;
      long long big = 0;
      for (int j = 0; j < w.n; ++j) {
        const int l = l0 + j;
        // C[dout][din] = sum_m d[m][o] in[m][i]
        GemmArgs& a = w.g[j];
        a.M = dout[l]; a.N = din[l]; a.K = rows;
        a.A = D(l); a.lda = dout[l];
        a.B = l == 0 ? X : H(l - 1); a.ldb = din[l];
        a.C = g.p + woff[l]; a.ldc = din[l];
        w.part[j] = part.p + col_layer[l].off;
        wide = wide && a.M % 128 == 0;
        big += (long long)(a.N / BN) * (a.M / 128);
      }
      const int bm = wide && big >= kWideTiles ? 128 : 64;
      for (int j = 0; j < w.n; ++j) {
        w.tile0[j + 1] = w.tile0[j] + w.g[j].N / BN * (w.g[j].M / bm);
        w.col0[j + 1] = w.col0[j] + w.g[j].M / 64 * chunks;
      }
      const dim3 grid(w.tile0[w.n] + w.col0[w.n]);
      if (bm == 128) hipLaunchKernelGGL(k_wgrad<128>, grid, dim3(256), 0, stream, w);
      else hipLaunchKernelGGL(k_wgrad<64>, grid, dim3(256), 0, stream, w);
    }
    hipLaunchKernelGGL(k_grad_fin, dim3(nblk(std::max(width, out_dim)), n_layers + 1), dim3(256), 0, stream, chunks,
                       n_layers, d_col.p, part.p, g.p, (int)nblk((long long)rows * out_dim), lpart.p, loss_sum);
    HIPCHK(hipGetLastError());
    return XG_OK;
  }
};

namespace xg {
int mlp_forward_on_stream(xg_mlp* net, int rows, const unsigned short* x, float* y, void* stream) {
  if (!net || rows <= 0 || rows > net->max_rows || rows % 64) return XG_E_ARG;
  return net->forward_on(rows, x, y, false, (hipStream_t)stream);
}
int mlp_dims(const xg_mlp* net, int* in_dim, int* out_dim, int* max_rows) {
  if (!net) return XG_E_ARG;
  *in_dim = net->in_dim; *out_dim = net->out_dim; *max_rows = net->max_rows;
  return XG_OK;
}
}  // namespace xg

extern "C" {

int xg_mlp_create(int in_dim, int width, int hidden_layers, int out_dim, int max_rows, unsigned long long seed,
                  xg_mlp** out) {
  if (!out || in_dim <= 0 || width <= 0 || out_dim <= 0 || hidden_layers < 1 || max_rows <= 0) return XG_E_ARG;
  if (in_dim % 64 || width % 64 || out_dim % 64 || max_rows % 64) return XG_E_ARG;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return XG_E_NOGPU;
  auto net = std::make_unique<xg_mlp>();
  net->in_dim = in_dim; net->width = width; net->hidden = hidden_layers; net->out_dim = out_dim;
  net->max_rows = max_rows;
  net->n_layers = hidden_layers + 1;
  long long off = 0;
  for (int l = 0; l < net->n_layers; ++l) {
    const int di = l == 0 ? in_dim : width, dn = l + 1 < net->n_layers ? width : out_dim;
    net->din.push_back(di); net->dout.push_back(dn);
    net->woff.push_back(off); off += (long long)di * dn;
    net->boff.push_back(off); off += dn;
  }
  net->n_params = off;
  // uniform(-1/sqrt(in), 1/sqrt(in)) weights, zero biases; the output layer
  // scaled by 0.1 so an untrained net proposes almost no correction
  std::vector<float> h(off, 0.0f);
  std::mt19937_64 rng(seed);
  for (int l = 0; l < net->n_layers; ++l) {
    const float a = 1.0f / std::sqrt((float)net->din[l]) * (l + 1 == net->n_layers ? 0.1f : 1.0f);
    std::uniform_real_distribution<float> u(-a, a);
    for (long long i = 0; i < (long long)net->din[l] * net->dout[l]; ++i) h[net->woff[l] + i] = u(rng);
  }
  if (hipStreamCreate(&net->stream) != hipSuccess) return XG_E_HIP;
  HIPCHK(net->w.alloc(off)); HIPCHK(net->g.alloc(off)); HIPCHK(net->m.alloc(off)); HIPCHK(net->v.alloc(off));
  HIPCHK(net->wb.alloc(off));
  HIPCHK(net->Zall.alloc((size_t)hidden_layers * max_rows * width));
  HIPCHK(net->Hall.alloc((size_t)hidden_layers * max_rows * width));
  // (a layer's each: the weight gradients of all layers are formed together)
  HIPCHK(net->dH.alloc((size_t)hidden_layers * max_rows * width));
  HIPCHK(net->dY.alloc((size_t)max_rows * out_dim));
  HIPCHK(net->Y.alloc((size_t)max_rows * out_dim));
  long long col_off = 0;
  for (int l = 0; l < net->n_layers; ++l) {
    net->col_layer.push_back(ColLayer{net->dout[l], col_off, net->boff[l]});
    col_off += (long long)((max_rows + 255) / 256) * net->dout[l];
  }
  HIPCHK(net->part.alloc((size_t)col_off));
  HIPCHK(net->d_col.alloc(net->col_layer.size()));
  HIPCHK(hipMemcpy(net->d_col.p, net->col_layer.data(), sizeof(ColLayer) * net->col_layer.size(), hipMemcpyHostToDevice));
  HIPCHK(net->lpart.alloc(nblk((long long)max_rows * out_dim)));
  HIPCHK(hipHostMalloc((void**)&net->loss_sum, sizeof(double), hipHostMallocDefault));
  HIPCHK(hipMemcpy(net->w.p, h.data(), off * sizeof(float), hipMemcpyHostToDevice));
  HIPCHK(hipMemset(net->m.p, 0, off * sizeof(float)));
  HIPCHK(hipMemset(net->v.p, 0, off * sizeof(float)));
  HIPCHK(hipMemset(net->g.p, 0, off * sizeof(float)));
  hipLaunchKernelGGL(k_to_bf16, dim3(nblk(off)), dim3(256), 0, net->stream, off, net->w.p, net->wb.p);
  HIPCHK(hipStreamSynchronize(net->stream));
  *out = net.release();
  return XG_OK;
}

int xg_mlp_destroy(xg_mlp* net) {
  if (!net) return XG_E_ARG;
  delete net;
  return XG_OK;
}

int xg_mlp_params(xg_mlp* net, int set, float* params, long long* count) {
  if (!net) return XG_E_ARG;
  if (count) *count = net->n_params;
  if (!params) return XG_OK;
  if (set) {
    HIPCHK(hipMemcpyAsync(net->w.p, params, net->n_params * sizeof(float), hipMemcpyHostToDevice, net->stream));
    hipLaunchKernelGGL(k_to_bf16, dim3(nblk(net->n_params)), dim3(256), 0, net->stream, net->n_params, net->w.p,
                       net->wb.p);
    HIPCHK(hipMemsetAsync(net->m.p, 0, net->n_params * sizeof(float), net->stream));
    HIPCHK(hipMemsetAsync(net->v.p, 0, net->n_params * sizeof(float), net->stream));
    net->adam_t = 0;
  } else {
    HIPCHK(hipMemcpyAsync(params, net->w.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  }
  HIPCHK(hipStreamSynchronize(net->stream));
  return XG_OK;
}

int xg_mlp_forward(xg_mlp* net, int rows, const unsigned short* x_dev, float* y_dev) {
  if (!net || !x_dev || !y_dev || rows <= 0 || rows > net->max_rows || rows % 64) return XG_E_ARG;
  int st = net->forward(rows, x_dev, y_dev, false);
  if (st != XG_OK) return st;
  HIPCHK(hipStreamSynchronize(net->stream));
  return XG_OK;
}

int xg_mlp_loss_backward(xg_mlp* net, int rows, const unsigned short* x_dev, const float* t_dev,
                         const float* mask_dev, int count, double* loss, float* grads) {
  if (!net || !x_dev || !t_dev || !mask_dev || rows <= 0 || rows > net->max_rows || rows % 64 || count <= 0)
    return XG_E_ARG;
  int st = net->forward(rows, x_dev, net->Y.p, true);
  if (st != XG_OK) return st;
  const long long n = (long long)rows * net->out_dim;
  hipLaunchKernelGGL(k_mse, dim3(nblk(n)), dim3(256), 0, net->stream, (int)n, count, net->Y.p, t_dev, mask_dev,
                     net->dY.p, net->lpart.p);
  HIPCHK(hipGetLastError());
  st = net->backward(rows, x_dev);
  if (st != XG_OK) return st;
  if (grads) HIPCHK(hipMemcpyAsync(grads, net->g.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  HIPCHK(hipStreamSynchronize(net->stream));
  if (loss) *loss = *net->loss_sum / count;
  return XG_OK;
}

int xg_mlp_adam(xg_mlp* net, float lr, float beta1, float beta2, float eps) {
  if (!net || !(lr > 0.0f)) return XG_E_ARG;
  net->adam_t += 1;
  const float c1 = 1.0f - std::pow(beta1, (float)net->adam_t), c2 = 1.0f - std::pow(beta2, (float)net->adam_t);
  hipLaunchKernelGGL(k_adam, dim3(nblk(net->n_params)), dim3(256), 0, net->stream, net->n_params, net->w.p,
                     net->wb.p, net->g.p, net->m.p, net->v.p, lr, beta1, beta2, eps, c1, c2);
  HIPCHK(hipGetLastError());
  return XG_OK;
}

int xg_mlp_sync(xg_mlp* net) {
  if (!net) return XG_E_ARG;
  HIPCHK(hipStreamSynchronize(net->stream));
  return XG_OK;
}

}  // extern "C"
