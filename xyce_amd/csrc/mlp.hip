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

constexpr int BN = 64, BK = 64, LDS_K = BK + 8;

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
        *reinterpret_cast<u32x4*>(&lds[((t >> 3) + 32 * i) * LDS_K + (t & 7) * 8]) = v[i];
    } else {
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        const u32x4 a = v[i], b = v[i + 1];
        unsigned short* to = lds + ((t & 7) * 8 + 32 * i) * LDS_K + (t >> 3) * 2;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // rows 2 j and 2 j + 1: (k, k + 1) side by side
          *reinterpret_cast<unsigned*>(to + (2 * j) * LDS_K) = __builtin_amdgcn_perm(b[j], a[j], 0x05040100u);
          *reinterpret_cast<unsigned*>(to + (2 * j + 1) * LDS_K) = __builtin_amdgcn_perm(b[j], a[j], 0x07060302u);
        }
      }
    }
  }
};

// C = A B^T on BM x 64 tiles (BM 64 or 128): 4 waves, each (BM / 2) x 32 as
// BM / 64 blocks of v_mfma_f32_32x32x16_bf16 (A: lane l holds row l%32, k =
// 8*(l/32)..+7; B likewise by column; D register r of lane l is row 8*(r/4) +
// 4*(l/32) + r%4, column l%32).  At these sizes a tile's chain of k steps bounds
// the product (8 to 32 steps of 64, one or two tiles per CU), so four steps are
// in flight from memory in registers while LDS holds two, with one barrier per
// step; and the tiles that share rows of A sit on one XCD (consecutive
// workgroups go to the eight XCDs in turn), so that A crosses to one L2 only.
// Forward of 4096 rows (1600 -> 3 x 512 -> 256) 53.0 us, 78.5 with one 64 x 64 x 32
// step at a time; weight gradient 512 x 1600 over 2048 rows 22 us, 53.  Every element accumulates k in ascending order of
// 16 whatever the tile, so the tile size does not change a result.
constexpr int kAhead = 4;

template <bool TA, bool TB, int EPI, int BM>
__global__ void __launch_bounds__(256) k_gemm(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) unsigned short As[2][BM * LDS_K];
  __shared__ __attribute__((aligned(16))) unsigned short Bs[2][BN * LDS_K];
  constexpr int MI = BM / 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // workgroup id -> tile: ids id, id + 8, ... (one XCD) walk the columns of a row of tiles
  const int nt = g.N / BN, mt = g.M / BM, id = blockIdx.x;
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
#pragma unroll
  for (int d = 0; d < kAhead; ++d)
    if (d * BK < g.K) {
      sa[d].load(g.A, g.lda, m0, d * BK, tid);
      sb[d].load(g.B, g.ldb, n0, d * BK, tid);
    }
  for (int k0 = 0; k0 < g.K; k0 += kAhead * BK) {
#pragma unroll
    for (int d = 0; d < kAhead; ++d) {
      const int k = k0 + d * BK;
      if (k >= g.K) break;
      unsigned short *at = As[d & 1], *bt = Bs[d & 1];
      sa[d].store(at, tid);
      sb[d].store(bt, tid);
      if (k + kAhead * BK < g.K) {
        sa[d].load(g.A, g.lda, m0, k + kAhead * BK, tid);
        sb[d].load(g.B, g.ldb, n0, k + kAhead * BK, tid);
      }
      __syncthreads();
      // ---- matrix cores
#pragma unroll
      for (int kk = 0; kk < BK; kk += 16) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(&bt[(wn * 32 + (lane & 31)) * LDS_K + kk + 8 * (lane >> 5)]);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          const bf16x8 a =
              *reinterpret_cast<const bf16x8*>(&at[((wm * MI + i) * 32 + (lane & 31)) * LDS_K + kk + 8 * (lane >> 5)]);
          acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[i], 0, 0, 0);
        }
      }
    }
  }
  // ---- epilogue
  const int col = n0 + wn * 32 + (lane & 31);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = m0 + (wm * MI + i) * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      const size_t o = (size_t)row * g.ldc + col;
      const float v = acc[i][r];
      if (EPI == EPI_F32) {
        g.C[o] = v;
      } else if (EPI == EPI_BIAS_F32) {
        g.C[o] = v + g.bias[col];
      } else if (EPI == EPI_BIAS_GELU) {
        const float z = v + g.bias[col];
        g.C[o] = z;
        g.H[o] = f2bf(gelu(z));
      } else if (EPI == EPI_BIAS_GELU_H) {
        g.H[o] = f2bf(gelu(v + g.bias[col]));
      } else {
        g.H[o] = f2bf(v * gelu_d(g.Zin[o]));
      }
    }
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
__global__ void k_sum(int n, const double* p, double* out) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += p[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int st = 128; st > 0; st >>= 1) {
    if (threadIdx.x < st) red[threadIdx.x] += red[threadIdx.x + st];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[0] = red[0];
}

// bias gradients: column sums of a bf16 [rows][N] matrix, two passes (chunks of
// 256 rows, then over chunks; the second for all layers in one launch).  The
// chunk pass is bound by its loads' latency: eight rows in flight
// (2048 x 512: 4.4 us, 9.9 one row at a time).
__global__ void k_colsum_part(int rows, int N, const unsigned short* d, float* part) {
  const int col = blockIdx.x * 64 + (threadIdx.x & 63);
  const int r0 = blockIdx.y * 256 + (threadIdx.x >> 6) * 64;
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
  __shared__ float red[256];
  red[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x < 64) {
    const float t = red[threadIdx.x] + red[threadIdx.x + 64] + red[threadIdx.x + 128] + red[threadIdx.x + 192];
    part[(size_t)blockIdx.y * N + col] = t;
  }
}
// layer blockIdx.y: its N columns' partial sums at `off` of part, the sums at boff of g
struct ColLayer { int N; long long off, boff; };
__global__ void k_colsum_fin(int chunks, const ColLayer* layers, const float* part, float* g) {
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
  Buf<double> lpart, lsum;
  std::vector<ColLayer> col_layer;        // per layer: its partial column sums in `part`
  Buf<ColLayer> d_col;
  // Z_l / H_l at offset l * max_rows * width
  float* Z(int l) { return Zall.p + (size_t)l * max_rows * width; }
  unsigned short* H(int l) { return Hall.p + (size_t)l * max_rows * width; }
  ~xg_mlp() { if (stream) (void)hipStreamDestroy(stream); }

  template <bool TA, bool TB, int EPI>
  int gemm(const GemmArgs& a) {
    if (a.M % 64 || a.N % BN || a.K % BK || a.M <= 0 || a.N <= 0 || a.K <= 0) return XG_E_ARG;
    // 128-row tiles read B half as often, but their chain per step is longer: from
    // two tiles per CU (256 of them) on (forward of 8192 rows 78 us against 80.5
    // with 64-row tiles, of 4096 rows 61 against 53.6)
    if (a.M % 128 == 0 && (long long)(a.N / BN) * (a.M / 128) >= 512)
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

  // partial column sums of layer l's gradient (k_colsum_fin adds the chunks)
  int colsum(int rows, int l, const unsigned short* d) {
    hipLaunchKernelGGL(k_colsum_part, dim3(dout[l] / 64, (rows + 255) / 256), dim3(256), 0, stream, rows, dout[l], d,
                       part.p + col_layer[l].off);
    HIPCHK(hipGetLastError());
    return XG_OK;
  }

  // backward of the loss whose output gradient is in dY (bf16 [rows][out])
  int backward(int rows, const unsigned short* X) {
    const unsigned short* dcur = dY.p;   // gradient w.r.t. this layer's output (pre-activation)
    for (int l = n_layers - 1; l >= 0; --l) {
      const unsigned short* in = l == 0 ? X : H(l - 1);
      // dW_l = dcur^T in : C[dout][din] = sum_m dcur[m][o] in[m][i]
      GemmArgs a{};
      a.M = dout[l]; a.N = din[l]; a.K = rows;
      a.A = dcur; a.lda = dout[l];
      a.B = in; a.ldb = din[l];
      a.C = g.p + woff[l]; a.ldc = din[l];
      int st = gemm<true, true, EPI_F32>(a);
      if (st != XG_OK) return st;
      st = colsum(rows, l, dcur);
      if (st != XG_OK) return st;
      if (l == 0) break;
      // d(pre-activation of layer l-1) = (dcur W_l) * gelu'(Z_{l-1})
      GemmArgs b{};
      b.M = rows; b.N = din[l]; b.K = dout[l];
      b.A = dcur; b.lda = dout[l];
      b.B = wb.p + woff[l]; b.ldb = din[l];
      unsigned short* dst = dH.p + (size_t)((l - 1) & 1) * max_rows * width;
      b.H = dst; b.ldc = width; b.Zin = Z(l - 1);
      st = gemm<false, true, EPI_GELU_BWD>(b);
      if (st != XG_OK) return st;
      dcur = dst;
    }
    hipLaunchKernelGGL(k_colsum_fin, dim3(nblk(std::max(width, out_dim)), n_layers), dim3(256), 0, stream, (rows + 255) / 256,
                       d_col.p, part.p, g.p);
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
  HIPCHK(net->dH.alloc((size_t)2 * max_rows * width));
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
  HIPCHK(net->lsum.alloc(1));
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
  hipLaunchKernelGGL(k_sum, dim3(1), dim3(256), 0, net->stream, (int)nblk(n), net->lpart.p, net->lsum.p);
  HIPCHK(hipGetLastError());
  st = net->backward(rows, x_dev);
  if (st != XG_OK) return st;
  double l = 0.0;
  HIPCHK(hipMemcpyAsync(&l, net->lsum.p, sizeof(double), hipMemcpyDeviceToHost, net->stream));
  if (grads) HIPCHK(hipMemcpyAsync(grads, net->g.p, net->n_params * sizeof(float), hipMemcpyDeviceToHost, net->stream));
  HIPCHK(hipStreamSynchronize(net->stream));
  if (loss) *loss = l / count;
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
