// Multifrontal numeric LU for large systems (power-grid meshes, gate
// arrays): the factorisation that AmesosSolver::doSolve
// (src/LinearAlgebraServicesPKG/N_LAS_AmesosSolver.C:216-478) gets from KLU,
// restructured for the GPU.  The symbolic analysis (maximum transversal,
// approximate minimum degree, elimination tree) is the one the level-
// scheduled path uses; here the columns of L are grouped into supernodes,
// each with a dense frontal matrix, and the elimination tree of supernodes
// is processed level by level (all fronts of a level in one launch):
//
//   assemble  F_s = A entries of s's columns + extend-add of the children's
//             Schur complements (the j-th children of a level in launch j,
//             rows split over workgroups: a fixed order)
//   factor    dense LU of the pivot block, L21, U12 and the Schur complement
//             F22 -= L21 U12; small fronts one workgroup each, large fronts
//             blocked by 32-column panels (diagonal block in LDS, row-parallel
//             triangular solves for L21 and U12, tiled update over the GPU)
//
// Static pivots, as in the level-scheduled path, with KLU's threshold test
// (|l_ij| <= 1/0.001, finite nonzero pivots) on every column.
//
// Layout in HBM: fronts row-major, one after another (fo[s]); factors stay in
// the fronts (F11 = L11\U11, F21 = L21, F12 = U12); per-front solve vectors
// (vo[s]); index lists in B (permuted) numbering.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <stdexcept>
#include <type_traits>
#include <vector>

#include "xg_internal.h"

namespace xg {

// ---------------------------------------------------------------------------
// plan (host)
// ---------------------------------------------------------------------------
int mf_plan(const LuSymbolic& s, const int* rowptr, const int* colind, MfPlan& p) {
  const int n = s.n;
  const int ns = (int)s.sfirst.size() - 1;
  if (ns < 1 || (int)s.sparent.size() != ns || (int)s.srow_ptr.size() != ns + 1 || s.sfirst[ns] != n) return XG_E_SETUP;
  p = MfPlan();
  p.n = n;
  p.ns = ns;
  p.sfirst = s.sfirst;
  p.sparent = s.sparent;
  std::vector<int> snode(n);
  for (int t = 0; t < ns; ++t)
    for (int k = p.sfirst[t]; k < p.sfirst[t + 1]; ++k) snode[k] = t;
  // front index lists: pivots, then the rows below
  p.iptr.assign(ns + 1, 0);
  p.m.resize(ns);
  for (int t = 0; t < ns; ++t) {
    p.m[t] = (p.sfirst[t + 1] - p.sfirst[t]) + (s.srow_ptr[t + 1] - s.srow_ptr[t]);
    p.iptr[t + 1] = p.iptr[t] + p.m[t];
    p.max_m = std::max<long long>(p.max_m, p.m[t]);
    if (p.sparent[t] >= 0 && p.sparent[t] <= t) return XG_E_SETUP;
  }
  p.idx.resize(p.iptr[ns]);
  for (int t = 0; t < ns; ++t) {
    int q = p.iptr[t];
    for (int c = p.sfirst[t]; c < p.sfirst[t + 1]; ++c) p.idx[q++] = c;
    for (int r = s.srow_ptr[t]; r < s.srow_ptr[t + 1]; ++r) p.idx[q++] = s.srow[r];
  }
  p.cptr.assign(ns + 1, 0);
  for (int t = 0; t < ns; ++t) if (p.sparent[t] >= 0) p.cptr[p.sparent[t] + 1]++;
  for (int t = 0; t < ns; ++t) p.cptr[t + 1] += p.cptr[t];
  p.clist.resize(p.cptr[ns]);
  {
    std::vector<int> f(p.cptr.begin(), p.cptr.end() - 1);
    for (int t = 0; t < ns; ++t) if (p.sparent[t] >= 0) p.clist[f[p.sparent[t]]++] = t;
  }
  std::vector<int> lvl(ns, 0);
  int maxl = 0;
  for (int t = 0; t < ns; ++t) {       // children come before parents
    for (int c = p.cptr[t]; c < p.cptr[t + 1]; ++c) lvl[t] = std::max(lvl[t], lvl[p.clist[c]] + 1);
    maxl = std::max(maxl, lvl[t]);
  }
  p.lvl_ptr.assign(maxl + 2, 0);
  for (int t = 0; t < ns; ++t) p.lvl_ptr[lvl[t] + 1]++;
  for (int l = 0; l <= maxl; ++l) p.lvl_ptr[l + 1] += p.lvl_ptr[l];
  p.lvl_s.resize(ns);
  {
    std::vector<int> f(p.lvl_ptr.begin(), p.lvl_ptr.end() - 1);
    for (int t = 0; t < ns; ++t) p.lvl_s[f[lvl[t]]++] = t;
  }
  // extend-add maps: each row below a front's pivots, located in its parent
  p.eptr.assign(ns + 1, 0);
  for (int t = 0; t < ns; ++t) p.eptr[t + 1] = p.eptr[t] + (p.m[t] - (p.sfirst[t + 1] - p.sfirst[t]));
  p.emap.resize(p.eptr[ns]);
  for (int t = 0; t < ns; ++t) {
    const int np = p.sfirst[t + 1] - p.sfirst[t];
    const int nu = p.m[t] - np;
    if (nu == 0) continue;
    const int pa = p.sparent[t];
    if (pa < 0) return XG_E_SETUP;
    const int* pb = p.idx.data() + p.iptr[pa];
    const int* pe = p.idx.data() + p.iptr[pa + 1];
    const int npa = p.sfirst[pa + 1] - p.sfirst[pa];
    for (int a = 0; a < nu; ++a) {
      const int r = p.idx[p.iptr[t] + np + a];
      // the parent's list is pivots (ascending) then rows (ascending)
      int loc = -1;
      if (r >= p.sfirst[pa] && r < p.sfirst[pa + 1]) loc = r - p.sfirst[pa];
      else {
        const int* f = std::lower_bound(pb + npa, pe, r);
        if (f != pe && *f == r) loc = (int)(f - pb);
      }
      if (loc < 0) return XG_E_SETUP;   // structures must nest
      p.emap[p.eptr[t] + a] = loc;
    }
  }
  // front and vector offsets, flops
  p.fo.assign(ns + 1, 0);
  p.vo.assign(ns + 1, 0);
  for (int t = 0; t < ns; ++t) {
    p.fo[t + 1] = p.fo[t] + (long long)p.m[t] * p.m[t];
    p.vo[t + 1] = p.vo[t] + p.m[t];
    const double np = p.sfirst[t + 1] - p.sfirst[t], mm = p.m[t];
    for (double k = 0; k < np; ++k) p.flops += 2.0 * (mm - k - 1) * (mm - k - 1) + (mm - k - 1);
  }
  // A entries by front row: entry (i,j) of B goes to the front whose pivots
  // hold min(i,j)
  std::vector<int> arow_of(s.nnz_a), acol_of(s.nnz_a);
  p.arow.assign((size_t)p.vo[ns] + 1, 0);
  for (int r = 0; r < n; ++r) {
    const int i = s.rinv[r];
    for (int k = rowptr[r]; k < rowptr[r + 1]; ++k) {
      const int j = s.pinv[colind[k]];
      const int t = snode[std::min(i, j)];
      const int* b = p.idx.data() + p.iptr[t];
      const int np = p.sfirst[t + 1] - p.sfirst[t];
      auto local = [&](int g) -> int {
        if (g >= p.sfirst[t] && g < p.sfirst[t + 1]) return g - p.sfirst[t];
        const int* e = p.idx.data() + p.iptr[t + 1];
        const int* f = std::lower_bound(b + np, e, g);
        return (f != e && *f == g) ? (int)(f - b) : -1;
      };
      const int li = local(i), lj = local(j);
      if (li < 0 || lj < 0) return XG_E_SETUP;
      arow_of[k] = p.vo[t] + li;
      acol_of[k] = lj;
      ++p.arow[arow_of[k] + 1];
    }
  }
  for (size_t q = 1; q < p.arow.size(); ++q) p.arow[q] += p.arow[q - 1];
  p.acol.resize(s.nnz_a);
  p.aslot.resize(s.nnz_a);
  {
    std::vector<int> f(p.arow.begin(), p.arow.end() - 1);
    for (int k = 0; k < s.nnz_a; ++k) {
      const int q = f[arow_of[k]]++;
      p.acol[q] = acol_of[k];
      p.aslot[q] = k;
    }
  }
  return XG_OK;
}

// ---------------------------------------------------------------------------
// kernels
// ---------------------------------------------------------------------------
// what a kernel needs to know of a front and of a child, each in one load
struct MfFront {
  long long fo;                 // its elements (row-major, order m)
  int m, np;                    // order, pivots
  int first, idx;               // first column, index list
  int c0, c1;                   // children
  int vo, pad;                  // its rows' slots in the front vectors and in arow
};
struct MfChild {
  long long src;                // the Schur complement's first element
  int ld, nu;                   // its row stride and order
  int em, vsrc;                 // parent positions of its rows; their slots in the front vectors
};
struct MfDev {
  const int* sfirst; const int* m; const long long* fo; const int* iptr; const int* idx;
  const int* cptr; const int* clist; const int* eptr; const int* emap; const int* vo;
  const MfFront* front; const MfChild* child;
  const int* arow; const int* acol; const int* aslot;
};

constexpr int kMfTiny = 64;     // fronts up to this order: one wavefront, the front in LDS
constexpr int kMfPanel = 32;    // panel width of the blocked factorisation (64 spills the register panel)
constexpr int kMfSolveBlock = 1024;

// f(0), f(1), ... f(N - 1) with the index a constant in each
template <int N, int K = 0, class F>
__device__ __forceinline__ void mf_for(const F& f) {
  if constexpr (K < N) {
    f(std::integral_constant<int, K>{});
    mf_for<N, K + 1>(f);
  }
}
#define MF_INLINE __attribute__((always_inline))

// value of v in lane `src` (wave-uniform) of the wavefront
__device__ __forceinline__ double mf_bcast(double v, int src) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b & 0xffffffffull), src);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), src);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ float mf_bcast(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

template <class T>
__device__ __forceinline__ T mf_wave_sum(T v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Larger fronts: blocked by panels of kMfPanel columns, one launch per panel
// index over all fronts of a level.  Launch j (p0 = 32 j) does two things at
// once: the rank-32 update by panel j - 1 and the factorisation of panel j.
//   panel entries {front, i, -1, slot}: blocks 2 i and 2 i + 1 of the front's
//     64-row blocks of L21 and 64-column blocks of U12.  Wavefronts 1 and 2
//     apply panel j - 1's update to a block each (matrix cores) while wavefront
//     0 updates and factors the 32 x 32 diagonal block in registers (lane t
//     owns row t, the pivot row broadcast with readlane); wavefronts 1 and 2
//     then solve their blocks by substitution.  Every workgroup of a front
//     factors the diagonal block for itself, so no workgroup waits for
//     another; the first stores the factors in the front's dbuf slot (the
//     others may still be reading the unfactored block), and launch j + 1
//     copies them into the front.
//   update entries {front, tile row, tile column, slot}: a 96 x 64 tile of the
//     rest, -= L U of panel j - 1.
//   copy entries {front, 0, -2, slot}: only the copy of panel j - 1's diagonal.
// The launch after the last panel holds the update entries of the Schur
// complement.  The chain of panels is what bounds a tree's top: one launch per
// panel instead of a panel and an update launch, and no operand passes through
// LDS on its way to the matrix cores, so that a step is one round of loads, the
// diagonal's 32 dependent pivots and a substitution (16.8 us where the two
// launches took 31.6, on the 865-order root of a 512 x 512 grid; 10.7 to 20 us
// with FP32 factors and up to 720 workgroups).
//
// v_mfma_{f64,f32}_16x16x4: lane l holds A's row l % 16, column l / 16 of the
// 16 x 4 block, B's row l / 16, column l % 16 of the 4 x 16 block; accumulator
// register r of lane l: column l % 16, row l / 16 + 4 r for FP64 and
// 4 (l / 16) + r for FP32.
typedef double mf_d4 __attribute__((ext_vector_type(4)));
typedef float mf_f4 __attribute__((ext_vector_type(4)));
template <class T> struct MfAcc;
template <> struct MfAcc<double> {
  typedef mf_d4 V;
  static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
  static __device__ __forceinline__ V mma(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <> struct MfAcc<float> {
  typedef mf_f4 V;
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
  static __device__ __forceinline__ V mma(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// acc = F[i0.., j0..] - F[i0.., q0..q0+kw) F[q0..q0+kw, j0..) on NA x NB blocks
// of 16 x 16 by one wavefront (i0 < i1, j0 < j1).  Rows from i1 and columns from
// j1 on repeat the last one (the caller drops them), so that no load is conditional; addresses
// are a uniform base and a 32-bit offset.  Every load is issued before the
// first product.
template <class T>
__device__ __forceinline__ T mf_at(const T* base, unsigned byte_off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + byte_off);
}

template <class T, int NA, int NB>
__device__ __forceinline__ void mf_update_blocks(const T* Fs, long long ld, int i0, int i1, int j0, int j1, int q0,
                                                 int kw, int lane, typename MfAcc<T>::V (&acc)[NA][NB]) {
  const int lr = lane & 15, lk = lane >> 4;
  const unsigned row = (unsigned)ld * sizeof(T);
  unsigned cj[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) cj[b] = (unsigned)(min(j0 + 16 * b + lr, j1 - 1) - j0) * sizeof(T);
  const T* C = Fs + i0 * ld + j0;
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned o = (unsigned)(min(i0 + 16 * a + MfAcc<T>::row(lk, r), i1 - 1) - i0) * row;
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b][r] = mf_at(C, o + cj[b]);
    }
  if (kw <= 0) return;
  T l[NA][kMfPanel / 4], u[NB][kMfPanel / 4];
  const T* Lb = Fs + i0 * ld + q0;
  const T* Ub = Fs + q0 * ld + j0;
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    const unsigned o = (unsigned)(min(i0 + 16 * a + lr, i1 - 1) - i0) * row;
#pragma unroll
    for (int k = 0; k < kMfPanel / 4; ++k) l[a][k] = mf_at(Lb, o + (unsigned)min(4 * k + lk, kw - 1) * (unsigned)sizeof(T));
  }
#pragma unroll
  for (int k = 0; k < kMfPanel / 4; ++k) {
    const unsigned o = (unsigned)min(4 * k + lk, kw - 1) * row;
#pragma unroll
    for (int b = 0; b < NB; ++b) u[b][k] = mf_at(Ub, o + cj[b]);
  }
#pragma unroll
  for (int k = 0; k < kMfPanel / 4; ++k) {
    const bool in = 4 * k + lk < kw;
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const T lv = in ? -l[a][k] : (T)0;
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b] = MfAcc<T>::mma(lv, u[b][k], acc[a][b]);
    }
  }
}

// reciprocal of a pivot in four stages that run between the products of a row
// update: the hardware estimate of the mantissa's reciprocal, two Newton steps
// (one for FP32), the exponent (apart, so that no step over- or underflows)
template <class T> struct MfRecip;
template <> struct MfRecip<double> {
  double p, m, x;
  __device__ __forceinline__ void stage(int i) {
    if (i == 0) { m = __builtin_amdgcn_frexp_mant(p); x = __builtin_amdgcn_rcp(m); }
    if (i == 1 || i == 2) x = fma(fma(-m, x, 1.0), x, x);
    if (i == 3) x = __builtin_amdgcn_ldexp(x, -__builtin_amdgcn_frexp_exp(p));
  }
};
template <> struct MfRecip<float> {
  float p, m, x;
  __device__ __forceinline__ void stage(int i) {
    if (i == 0) { m = __builtin_amdgcn_frexp_mantf(p); x = __builtin_amdgcn_rcpf(m); }
    if (i == 2) x = fmaf(fmaf(-m, x, 1.0f), x, x);
    if (i == 3) x = __builtin_amdgcn_ldexpf(x, -__builtin_amdgcn_frexp_expf(p));
  }
};

// row[q] -= l * (row k's element q) for q in [q0, N), the lanes' rows in
// registers: eight broadcasts before the products that use them (a broadcast
// is usable two cycles after it issues), the next pivot's reciprocal in between
template <int N, class T>
__device__ __forceinline__ void mf_row_update(T (&v)[N], T l, int k, int q0, MfRecip<T>& rec) {
#pragma unroll
  for (int c = 0; c < N; c += 8) {
    T u[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (c + q >= q0 && c + q < N) u[q] = mf_bcast(v[c + q < N ? c + q : 0], k);
    if (c + 7 >= q0) __builtin_amdgcn_sched_barrier(0);
    if (c >= N - 32) rec.stage((c - (N - 32)) / 8);
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (c + q >= q0 && c + q < N) v[c + q < N ? c + q : 0] -= l * u[q];
  }
}

// right-looking LU of the rows in registers (lane t: row t), pivots [0, NP) of
// N columns; lanes from `rows` on count for nothing.  first: lowest column with
// a bad pivot or a multiplier beyond KLU's threshold; rd: lane k's reciprocal
// of pivot k.  Constant trip counts keep the rows in registers.
template <int N, int NP, class T>
__device__ __forceinline__ void mf_factor_rows(T (&v)[N], int lane, int rows, int np, int& first, bool& hard, T& rd) {
  MfRecip<T> rec;
  T piv = mf_bcast(v[0], 0);
  rec.p = piv;
#pragma unroll
  for (int i = 0; i < 4; ++i) rec.stage(i);
  mf_for<NP>([&](auto kc) MF_INLINE {
    constexpr int k = kc, k1 = k + 1 < N ? k + 1 : k;
    if (k >= np) return;
    const T rp = rec.x;
    if (!(fabs((double)piv) > 0.0) || !isfinite((double)piv)) { first = min(first, k); hard = true; }
    if (lane == k) rd = rp;
    const bool upd = lane > k && lane < rows;
    const T l = upd ? v[k] * rp : (T)0;
    if (upd) v[k] = l;
    if (!(fabs((double)l) <= 1.0e3)) first = min(first, k);
    if constexpr (k1 > k) v[k1] -= l * mf_bcast(v[k1], k);
    piv = mf_bcast(v[k1], k1);
    rec.p = piv;
    mf_row_update<N>(v, l, k, k + 2, rec);
    __builtin_amdgcn_sched_barrier(0);
  });
}

// LDS written by a wavefront's lanes is visible to its other lanes
__device__ __forceinline__ void mf_wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Assembly of a larger front: A's entries plus the children's Schur
// complements, one child after another in their fixed order, so that every
// element receives the same sums in the same order on every refactor.  One
// workgroup per range of rows and columns (entries {front, first row, rows,
// offset into alo}, {first column, columns, 0, 0}; at most kMfAsm elements, held
// in LDS until they are complete, so a front is written once and never cleared
// or read back).  Wavefront w owns the rows with index % 4 = w: no wavefront
// waits for another.  alo holds, per entry and child, the child's rows [x, y)
// that land in the range; a child's rows map to increasing parent rows.  Per
// child and 256 columns a wavefront issues the loads of up to four rows at
// once (512 x 512 grid, all levels: 263 us with A's entries in, where clearing the
// fronts, scattering A and adding the children in memory took 400).
constexpr int kMfAsmRows = 16;
constexpr int kMfAsm = 4096;

template <class T>
__global__ void __launch_bounds__(256) k_mf_assemble(MfDev d, const int4* ent, const int2* alo, const double* vals,
                                                     T* F) {
  __shared__ T R[kMfAsm];
  const int4 e = ent[2 * blockIdx.x], ec = ent[2 * blockIdx.x + 1];
  const MfFront f = d.front[e.x];
  const int r0 = e.y, rows = e.z, j0 = ec.x, w = ec.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int i = wave; i < rows; i += 4) {
    for (int j = lane; j < w; j += 64) R[i * w + j] = (T)0;
    mf_wave_fence();
    const int* ar = d.arow + f.vo + r0 + i;
    for (int q = ar[0] + lane; q < ar[1]; q += 64) {
      const int j = d.acol[q] - j0;
      // (an entry listed twice in a row adds up)
      if (j >= 0 && j < w) atomicAdd(&R[i * w + j], (T)vals[d.aslot[q]]);
    }
  }
  mf_wave_fence();
  const int2* lo = alo + e.w;
  for (int c = f.c0; c < f.c1; ++c) {
    const MfChild ch = d.child[c];
    const int2 ab = lo[c - f.c0];
    if (ab.x >= ab.y) continue;
    const int* em = d.emap + ch.em;
    // slot k: the child's row that lands on this wavefront's row 4 k + wave
    const int er = ab.x + lane < ab.y ? em[ab.x + lane] - r0 : -1;
    int a[kMfAsmRows / 4];
#pragma unroll
    for (int k = 0; k < kMfAsmRows / 4; ++k) {
      const unsigned long long hit = __ballot(er == 4 * k + wave);
      a[k] = hit ? ab.x + (int)__builtin_ctzll(hit) : -1;
    }
    const T* Fc = F + ch.src;
    for (int c0 = lane; c0 - lane < ch.nu; c0 += 256) {
      int eb[4];
      T cv[kMfAsmRows / 4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = c0 + 64 * q;
        const int j = b < ch.nu ? em[b] - j0 : -1;
        eb[q] = j < w ? j : -1;
      }
#pragma unroll
      for (int k = 0; k < kMfAsmRows / 4; ++k) {
        if (a[k] < 0) continue;
        const T* crow = Fc + (long long)a[k] * ch.ld;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int b = c0 + 64 * q;
          cv[k][q] = b < ch.nu ? crow[b] : (T)0;
        }
      }
#pragma unroll
      for (int k = 0; k < kMfAsmRows / 4; ++k) {
        if (a[k] < 0) continue;
        T* prow = R + (4 * k + wave) * w;
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (eb[q] >= 0) prow[eb[q]] += cv[k][q];
      }
    }
    mf_wave_fence();
  }
  T* Fs = F + f.fo + (long long)r0 * f.m + j0;
  for (int i = wave; i < rows; i += 4)
    for (int j = lane; j < w; j += 64) Fs[(long long)i * f.m + j] = R[i * w + j];
}

// Fronts of order at most N (32 or 64): one wavefront per front.  A's entries
// and the children's updates are added in LDS (row stride N + 1), one child
// after another; then lane t holds row t in registers and the pivot rows are
// broadcast from there: a pivot costs its reciprocal and the row updates, no
// LDS traffic (512 x 512 grid, all levels: 300 us, 656 with the elimination in LDS).
template <class T, int N>
__global__ void __launch_bounds__(64) k_mf_factor_tiny(MfDev d, const int* list, const double* vals, T* F, int* bad) {
  constexpr int ld = N + 1;
  __shared__ T A[N * ld];
  const MfFront f = d.front[list[blockIdx.x]];
  const int ms = f.m, np = f.np, t = threadIdx.x;
  if (t < ms) {
    T* row = A + t * ld;
    for (int j = 0; j < ms; ++j) row[j] = (T)0;
    const int q1 = d.arow[f.vo + t + 1];
    for (int q = d.arow[f.vo + t]; q < q1; ++q) row[d.acol[q]] += (T)vals[d.aslot[q]];
  }
  mf_wave_fence();
  // a child's update has at most ms rows and columns: lane t adds column t
  for (int c = f.c0; c < f.c1; ++c) {
    const MfChild ch = d.child[c];
    const int nu = ch.nu;
    const int eb = t < nu ? d.emap[ch.em + t] : 0;   // parent position of the child's row/column t
    const T* cb = F + ch.src + t;
    for (int a = 0; a < nu; a += 16) {
      T v[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) v[q] = (t < nu && a + q < nu) ? cb[(long long)(a + q) * ch.ld] : (T)0;
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        if (a + q >= nu) break;
        const int pr = __builtin_amdgcn_readlane(eb, a + q);
        if (t < nu) A[pr * ld + eb] += v[q];
      }
    }
    mf_wave_fence();
  }
  T v[N];
  const T* own = A + (t < N ? t : 0) * ld;
#pragma unroll
  for (int q = 0; q < N; ++q) v[q] = (t < ms && q < ms) ? own[q] : (T)0;
  int first = N;
  bool hard = false;
  T rd = (T)0;
  mf_factor_rows<N, N>(v, t, ms, np, first, hard, rd);
  if (t < ms) {
    T* row = A + t * ld;
#pragma unroll
    for (int q = 0; q < N; ++q) row[q] = v[q];
  }
  mf_wave_fence();
  T* Fs = F + f.fo;
  for (int i = 0; i < ms; ++i)
    if (t < ms) Fs[(long long)i * ms + t] = A[i * ld + t];
  if (first < np) atomicMin(bad, f.first + first + 1);
  if (__any(hard) && t == 0) atomicOr(bad + 1, 1);
}

constexpr int kMfStep = 192;              // threads of a step workgroup: three wavefronts
constexpr int kMfTileRows = 96;           // rows of an update tile: 32 per wavefront
constexpr int kMfDs = kMfPanel + 2;       // row stride of the diagonal factors in LDS (16-byte pairs)
constexpr int kMfTile = 64 * (kMfPanel + 1) > kMfPanel * 65 ? 64 * (kMfPanel + 1) : kMfPanel * 65;

template <class T>
__global__ void __launch_bounds__(kMfStep) __attribute__((amdgpu_waves_per_eu(2))) k_mf_step(MfDev d, const int4* ent, int p0, T* F, T* dbuf, int half,
                                                     int* bad) {
  constexpr int PW = kMfPanel;
  __shared__ __attribute__((aligned(16))) T Du[PW * kMfDs];   // U11 by rows
  __shared__ __attribute__((aligned(16))) T Dl[PW * kMfDs];   // L11 by columns; the updated block before it is factored
  __shared__ T Rd[PW];
  __shared__ T Ts[2][kMfTile];
  const int4 e = ent[blockIdx.x];
  const int s = e.x, slot = e.w;
  const int ms = d.m[s], np = d.sfirst[s + 1] - d.sfirst[s];
  const int base = min(np, p0 + PW), q0 = p0 - PW, kw = q0 >= 0 ? min(PW, np - q0) : 0;
  T* Fs = F + d.fo[s];
  const long long ld = ms;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 15, lk = lane >> 4;
  typedef typename MfAcc<T>::V V;
  if (kw > 0 && e.y == 0 && e.z <= 0) {
    // the front's first entry: panel j - 1's diagonal factors into the front
    const T* db = dbuf + ((long long)slot * 2 + (half ^ 1)) * PW * PW;
    for (int x = t; x < PW * PW; x += kMfStep) {
      const int i = x / PW, j = x % PW;
      if (i < kw && j < kw) Fs[(q0 + i) * ld + q0 + j] = db[x];
    }
  }
  if (e.z == -2) return;
  if (e.z >= 0) {
    const int i0 = base + e.y * kMfTileRows + 32 * wave, j0 = base + e.z * 64;
    if (i0 >= ms) return;      // these rows of the tile lie beyond the front
    V acc[2][4];
    mf_update_blocks<T, 2, 4>(Fs, ld, i0, ms, j0, ms, q0, kw, lane, acc);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int gi = i0 + 16 * a + MfAcc<T>::row(lk, r), gj = j0 + 16 * b + lr;
          if (gi < ms && gj < ms) Fs[gi * ld + gj] = acc[a][b][r];
        }
    return;
  }
  // ---- the diagonal (wavefront 0) and two blocks (wavefronts 1, 2) of panel j
  const int pw = base - p0, rest = ms - base, nrb = (rest + 63) / 64;
  const int blk = 2 * e.y + wave - 1;
  const bool has = wave > 0 && blk < 2 * nrb, lower = blk < nrb;
  T* Tl = Ts[wave > 1];
  const int o0 = base + (lower ? blk : blk - nrb) * 64;     // first row or column of the block
  if (wave == 0) {
    V acc[2][2];
    mf_update_blocks<T, 2, 2>(Fs, ld, p0, base, p0, base, q0, kw, lane, acc);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * a + MfAcc<T>::row(lk, r), j = 16 * b + lr;
          // beyond the panel's width: the identity
          Dl[i * kMfDs + j] = (i < pw && j < pw) ? acc[a][b][r] : (i == j ? (T)1 : (T)0);
        }
  } else if (has && lower) {
    V acc[4][2];
    mf_update_blocks<T, 4, 2>(Fs, ld, o0, ms, p0, base, q0, kw, lane, acc);
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          Tl[(16 * a + MfAcc<T>::row(lk, r)) * (PW + 1) + 16 * b + lr] = acc[a][b][r];
  } else if (has) {
    V acc[2][4];
    mf_update_blocks<T, 2, 4>(Fs, ld, p0, base, o0, ms, q0, kw, lane, acc);
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 4; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r) Tl[(16 * a + MfAcc<T>::row(lk, r)) * 65 + 16 * b + lr] = acc[a][b][r];
  }
  mf_wave_fence();          // each wavefront reads back its own tile: no wait for the others
  int failed = PW;          // first column whose pivot or multiplier fails
  bool hard = false;
  T v[PW];
  if (wave == 0) {
    const int row = lane & 31;
#pragma unroll
    for (int q = 0; q < PW; ++q) v[q] = Dl[row * kMfDs + q];
    T rd = (T)1;
    mf_factor_rows<PW, PW>(v, lane, PW, PW, failed, hard, rd);
    if (lane < PW) Rd[lane] = rd;
  } else if (has && lower) {
#pragma unroll
    for (int q = 0; q < PW; ++q) v[q] = Tl[lane * (PW + 1) + q];
  } else if (has) {
#pragma unroll
    for (int q = 0; q < PW; ++q) v[q] = Tl[q * 65 + lane];
  }
  __syncthreads();
  if (wave == 0 && lane < PW) {
#pragma unroll
    for (int q = 0; q < PW; ++q) {
      Du[lane * kMfDs + q] = v[q];
      Dl[q * kMfDs + lane] = v[q];
    }
    if (e.y == 0) {
      T* db = dbuf + ((long long)slot * 2 + half) * PW * PW + lane * PW;
#pragma unroll
      for (int q = 0; q < PW; ++q) db[q] = v[q];
    }
  }
  __syncthreads();
  if (has) {
    if (lower) {
      const bool valid = o0 + lane < ms;
      // row k + 1 of U11 is read while row k is applied (z, zero, is tied to
      // v[k] so that at most two rows are held in registers)
      int z = 0;
      T u[PW], un[PW];
#pragma unroll
      for (int q = 0; q < PW; ++q) u[q] = Du[q];
      T r = Rd[0];
      mf_for<PW>([&](auto kc) MF_INLINE {
        constexpr int k = kc, k1 = k + 1 < PW ? k + 1 : k;
        asm volatile("" : "+v"(z) : "v"(v[k]));
        const T rn = Rd[k1 + z];
#pragma unroll
        for (int q = k + 2; q < PW; ++q) un[q] = Du[z + k1 * kMfDs + q];
        v[k] *= r;
        if (valid && !(fabs((double)v[k]) <= 1.0e3)) failed = min(failed, k);
#pragma unroll
        for (int q = k + 1; q < PW; ++q) v[q] -= v[k] * u[q];
#pragma unroll
        for (int q = k + 2; q < PW; ++q) u[q] = un[q];
        r = rn;
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int q = 0; q < PW; ++q) Tl[lane * (PW + 1) + q] = v[q];
    } else {
      const int c = o0 + lane;
      int z = 0;
      T u[PW], un[PW];
#pragma unroll
      for (int q = 0; q < PW; ++q) u[q] = Dl[q];
      mf_for<PW>([&](auto kc) MF_INLINE {
        constexpr int k = kc, k1 = k + 1 < PW ? k + 1 : k;
        asm volatile("" : "+v"(z) : "v"(v[k]));
#pragma unroll
        for (int q = k + 2; q < PW; ++q) un[q] = Dl[z + k1 * kMfDs + q];
#pragma unroll
        for (int q = k + 1; q < PW; ++q) v[q] -= u[q] * v[k];
#pragma unroll
        for (int q = k + 2; q < PW; ++q) u[q] = un[q];
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int q = 0; q < PW; ++q)
        if (c < ms && q < pw) Fs[(p0 + q) * ld + c] = v[q];
    }
  }
  __syncthreads();
  // the L21 blocks, row by row
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    const int b = 2 * e.y + w, r0 = base + b * 64;
    if (b >= nrb) break;
    for (int x = t; x < 64 * PW; x += kMfStep) {
      const int i = x / PW, q = x % PW;
      if (r0 + i < ms && q < pw) Fs[(r0 + i) * ld + p0 + q] = Ts[w][i * (PW + 1) + q];
    }
  }
  if (failed < pw) atomicMin(bad, d.sfirst[s] + p0 + failed + 1);
  if (__any(hard) && lane == 0) atomicOr(bad + 1, 1);
}

// sums over c in [c0, c1) of F[r + k][c] v[c] for the rows r .. r + nr - 1
// (nr <= 4, wave-uniform) of a row-major front, by one wavefront: every lane
// keeps eight loads in flight (four rows, two column blocks), so the four rows
// share their memory round trips; row k's sum is returned in out[k] in every
// lane
template <class T>
__device__ __forceinline__ void mf_rows_dot4(const T* Fs, long long ms, int r, int nr, const T* v, int c0, int c1,
                                             int lane, T out[4]) {
  const T* row[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) row[k] = Fs + (long long)(r + (k < nr ? k : 0)) * ms;
  T a[4], b[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) { a[k] = (T)0; b[k] = (T)0; }
  int c = c0 + lane;
  for (; c + 64 < c1; c += 128) {
    const T v0 = v[c], v1 = v[c + 64];
    T f0[4], f1[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) { f0[k] = row[k][c]; f1[k] = row[k][c + 64]; }
#pragma unroll
    for (int k = 0; k < 4; ++k) { a[k] += f0[k] * v0; b[k] += f1[k] * v1; }
  }
  if (c < c1) {
    const T v0 = v[c];
#pragma unroll
    for (int k = 0; k < 4; ++k) a[k] += row[k][c] * v0;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) out[k] = mf_wave_sum(a[k] + b[k]);
}

// ---- solves.  V holds, per front, the vector of its index list: y on the
// pivot rows, the update for the parent below them.

// sum the children's updates into the front's vector Vl (LDS)
template <class T>
__device__ __forceinline__ void mf_gather_children(const MfDev& d, int s, const T* V, T* Vl) {
  for (int c = d.cptr[s]; c < d.cptr[s + 1]; ++c) {
    const int ch = d.clist[c];
    const int npc = d.sfirst[ch + 1] - d.sfirst[ch], nu = d.m[ch] - npc;
    const T* Vc = V + d.vo[ch];
    const int* em = d.emap + d.eptr[ch];
    for (int a = threadIdx.x; a < nu; a += blockDim.x) Vl[em[a]] += Vc[npc + a];
    __syncthreads();
  }
}

// forward, fronts of order <= 64: one wavefront, lane i owns row i
template <class T>
__global__ void __launch_bounds__(64) k_mf_fwd_tiny(MfDev d, const int* list, const T* F, T* V, const double* b,
                                                    T* yg) {
  __shared__ T Vl[kMfTiny];
  const int s = list[blockIdx.x];
  const int ms = d.m[s], np = d.sfirst[s + 1] - d.sfirst[s];
  const T* Fs = F + d.fo[s];
  const int* ix = d.idx + d.iptr[s];
  const int t = threadIdx.x;
  Vl[t] = t < np ? (T)b[ix[t]] : (T)0;
  __syncthreads();
  mf_gather_children(d, s, V, Vl);
  T v = Vl[t];
  for (int k = 0; k < np; ++k) {
    const T yk = mf_bcast(v, k);
    if (t > k && t < ms) v -= Fs[(long long)t * ms + k] * yk;
  }
  if (t < ms) V[d.vo[s] + t] = v;
  if (t < np) yg[ix[t]] = v;
}

// forward, larger fronts: one workgroup per front, the vector in LDS; the
// unit-lower L11 by 64-row blocks (rows updated by a row-wise product with the
// solved part, then the block's triangle solved by one wavefront from LDS),
// then the rows below the pivots updated by L21 y
template <class T>
__global__ void __launch_bounds__(kMfSolveBlock) k_mf_fwd_big(MfDev d, const int* list, const T* F, T* V,
                                                             const double* b, T* yg, int ldsv) {
  extern __shared__ unsigned char mf_sm[];
  T* Bl = reinterpret_cast<T*>(mf_sm);          // 64 x 65 block
  const int s = list[blockIdx.x];
  T* Vl = ldsv ? Bl + 64 * 65 : V + d.vo[s];    // the front's vector (ms)
  const int ms = d.m[s], np = d.sfirst[s + 1] - d.sfirst[s];
  const T* Fs = F + d.fo[s];
  const int* ix = d.idx + d.iptr[s];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = blockDim.x >> 6;
  for (int i = t; i < ms; i += blockDim.x) Vl[i] = i < np ? (T)b[ix[i]] : (T)0;
  __syncthreads();
  mf_gather_children(d, s, V, Vl);
  for (int b0 = 0; b0 < np; b0 += 64) {
    const int bw = min(64, np - b0);
    if (b0 > 0) {
      for (int rr = 4 * wave; rr < bw; rr += 4 * nw) {
        const int nr = min(4, bw - rr);
        T acc[4];
        mf_rows_dot4(Fs, ms, b0 + rr, nr, Vl, 0, b0, lane, acc);
        if (lane == 0)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < nr) Vl[b0 + rr + k] -= acc[k];
      }
    }
    {
      T v[64 * 64 / kMfSolveBlock];
#pragma unroll
      for (int it = 0; it < 64 * 64 / kMfSolveBlock; ++it) {
        const int x = t + it * kMfSolveBlock, i = x >> 6, j = x & 63;
        v[it] = (i < bw && j < i) ? Fs[(long long)(b0 + i) * ms + b0 + j] : (T)0;
      }
#pragma unroll
      for (int it = 0; it < 64 * 64 / kMfSolveBlock; ++it) {
        const int x = t + it * kMfSolveBlock;
        Bl[(x >> 6) * 65 + (x & 63)] = v[it];
      }
    }
    __syncthreads();
    if (wave == 0) {
      T v = lane < bw ? Vl[b0 + lane] : (T)0;
      for (int k = 0; k < bw; ++k) {
        const T yk = mf_bcast(v, k);
        if (lane > k && lane < bw) v -= Bl[lane * 65 + k] * yk;
      }
      if (lane < bw) Vl[b0 + lane] = v;
    }
    __syncthreads();
  }
  for (int rr = np + 4 * wave; rr < ms; rr += 4 * nw) {
    const int nr = min(4, ms - rr);
    T acc[4];
    mf_rows_dot4(Fs, ms, rr, nr, Vl, 0, np, lane, acc);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < nr) Vl[rr + k] -= acc[k];
  }
  __syncthreads();
  if (ldsv)
    for (int i = t; i < ms; i += blockDim.x) V[d.vo[s] + i] = Vl[i];
  for (int i = t; i < np; i += blockDim.x) yg[ix[i]] = Vl[i];
}

// backward, fronts of order <= 64 (roots first): x = U11^-1 (y - U12 x_below)
template <class T>
__global__ void __launch_bounds__(64) k_mf_bwd_tiny(MfDev d, const int* list, const T* F, T* x) {
  __shared__ T Xl[kMfTiny];
  const int s = list[blockIdx.x];
  const int ms = d.m[s], np = d.sfirst[s + 1] - d.sfirst[s];
  const T* Fs = F + d.fo[s];
  const int* ix = d.idx + d.iptr[s];
  const int t = threadIdx.x;
  if (t < ms) Xl[t] = x[ix[t]];           // y on the pivot rows, solved x below
  __syncthreads();
  T v = Xl[t];
  if (t < np) {
    const T* row = Fs + (long long)t * ms;
    int u = np;
    for (; u + 4 <= ms; u += 4) {
      const T f0 = row[u], f1 = row[u + 1], f2 = row[u + 2], f3 = row[u + 3];
      v -= f0 * Xl[u];
      v -= f1 * Xl[u + 1];
      v -= f2 * Xl[u + 2];
      v -= f3 * Xl[u + 3];
    }
    for (; u < ms; ++u) v -= row[u] * Xl[u];
  }
  // each lane's pivot reciprocal first (in parallel), so that the serial
  // sweep multiplies instead of dividing
  const T rd = t < np ? (T)1 / Fs[(long long)t * ms + t] : (T)0;
  for (int k = np - 1; k >= 0; --k) {
    const T xk = mf_bcast(v, k) * mf_bcast(rd, k);
    if (t == k) v = xk;
    else if (t < k) v -= Fs[(long long)t * ms + k] * xk;
  }
  if (t < np) x[ix[t]] = v;
}

// backward, larger fronts: rows minus U12 x_below (row-wise products), then
// U11 by 64-row blocks from the bottom
template <class T>
__global__ void __launch_bounds__(kMfSolveBlock) k_mf_bwd_big(MfDev d, const int* list, const T* F, T* V, T* x,
                                                             int ldsv) {
  extern __shared__ unsigned char mf_sm[];
  T* Bl = reinterpret_cast<T*>(mf_sm);          // 64 x 65 block
  const int s = list[blockIdx.x];
  T* Xl = ldsv ? Bl + 64 * 65 : V + d.vo[s];    // scratch (ms); V is not read by the backward solve
  const int ms = d.m[s], np = d.sfirst[s + 1] - d.sfirst[s];
  const T* Fs = F + d.fo[s];
  const int* ix = d.idx + d.iptr[s];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, nw = blockDim.x >> 6;
  for (int i = t; i < ms; i += blockDim.x) Xl[i] = x[ix[i]];
  __syncthreads();
  for (int rr = 4 * wave; rr < np; rr += 4 * nw) {
    const int nr = min(4, np - rr);
    T acc[4];
    mf_rows_dot4(Fs, ms, rr, nr, Xl, np, ms, lane, acc);
    if (lane == 0)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (k < nr) Xl[rr + k] -= acc[k];
  }
  __syncthreads();
  for (int b1 = np; b1 > 0; b1 -= 64) {
    const int b0 = max(0, b1 - 64), bw = b1 - b0;
    if (b1 < np) {
      for (int rr = 4 * wave; rr < bw; rr += 4 * nw) {
        const int nr = min(4, bw - rr);
        T acc[4];
        mf_rows_dot4(Fs, ms, b0 + rr, nr, Xl, b1, np, lane, acc);
        if (lane == 0)
#pragma unroll
          for (int k = 0; k < 4; ++k)
            if (k < nr) Xl[b0 + rr + k] -= acc[k];
      }
    }
    {
      T v[64 * 64 / kMfSolveBlock];
#pragma unroll
      for (int it = 0; it < 64 * 64 / kMfSolveBlock; ++it) {
        const int x = t + it * kMfSolveBlock, i = x >> 6, j = x & 63;
        v[it] = (i < bw && j >= i && j < bw) ? Fs[(long long)(b0 + i) * ms + b0 + j] : (T)0;
      }
#pragma unroll
      for (int it = 0; it < 64 * 64 / kMfSolveBlock; ++it) {
        const int x = t + it * kMfSolveBlock;
        Bl[(x >> 6) * 65 + (x & 63)] = v[it];
      }
    }
    __syncthreads();
    if (wave == 0) {
      T v = lane < bw ? Xl[b0 + lane] : (T)0;
      const T rd = lane < bw ? (T)1 / Bl[lane * 65 + lane] : (T)0;
      for (int k = bw - 1; k >= 0; --k) {
        const T xk = mf_bcast(v, k) * mf_bcast(rd, k);
        if (lane == k) v = xk;
        else if (lane < k) v -= Bl[lane * 65 + k] * xk;
      }
      if (lane < bw) Xl[b0 + lane] = v;
    }
    __syncthreads();
  }
  for (int i = t; i < np; i += blockDim.x) x[ix[i]] = Xl[i];
}

template <class T>
__global__ void k_mf_perm_in(int n, const int* prow, const double* b, double* bp) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) bp[i] = b[prow[i]];
}
template <class T>
__global__ void k_mf_perm_out(int n, const int* pcol, const T* xp, double* x, int* nan_flag) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n) {
    const double v = (double)xp[j];
    x[pcol[j]] = v;
    if (!isfinite(v)) atomicOr(nan_flag, 1);
  }
}

// ---------------------------------------------------------------------------
// host driver
// ---------------------------------------------------------------------------
#define MFCHK(x)                           \
  do {                                     \
    hipError_t e_ = (x);                   \
    if (e_ != hipSuccess) return XG_E_HIP; \
  } while (0)

template <class T>
struct DevVec {
  T* p = nullptr;
  ~DevVec() { if (p) (void)hipFree(p); }
  hipError_t up(const std::vector<T>& v, hipStream_t s) {
    if (p) { (void)hipFree(p); p = nullptr; }
    if (v.empty()) return hipSuccess;
    hipError_t e = hipMalloc((void**)&p, v.size() * sizeof(T));
    if (e != hipSuccess) return e;
    return hipMemcpyAsync(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice, s);
  }
  hipError_t alloc(size_t n) {
    if (p) { (void)hipFree(p); p = nullptr; }
    return n ? hipMalloc((void**)&p, n * sizeof(T)) : hipSuccess;
  }
};

// The refactor and the solve are fixed launch sequences for a given plan and
// set of buffers: each is captured once into a hipGraph and replayed.
struct MfGraph {
  const void* key[8] = {};
  hipGraphExec_t exec = nullptr;
};

struct MfLu::Impl {
  MfPlan P;
  hipStream_t st = nullptr;
  std::vector<MfGraph> graphs;
  ~Impl() {
    for (auto& g : graphs)
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
  }
  DevVec<int> sfirst, m, iptr, idx, cptr, clist, eptr, emap, vo, prow, pcol, bad, arow, acol, aslot;
  DevVec<long long> fo;
  DevVec<MfFront> front;
  DevVec<MfChild> child;
  DevVec<double> F64, V64, y64, b64;
  DevVec<float> F32, V32, y32;
  DevVec<int> tiny_list, big_list;
  DevVec<int4> aent;              // assembly entries of the larger fronts, two each
  DevVec<int2> alo;               // per entry and child: the child's rows in the entry's range
  DevVec<int4> sent;              // entries of the panel steps
  DevVec<double> dbuf;            // diagonal-block factors, two 32 x 32 slots per larger front of a level
  std::vector<int> tiny_off, tiny_half, big_off;   // fronts up to order 32 at [tiny_off, tiny_half), up to 64 from there
  int big_maxm = 0;
  std::vector<int> aoff;          // per level: offset into aent
  struct Step { int p0, off, cnt; };
  std::vector<std::vector<Step>> steps;   // per level: its panel steps
  MfDev dev() const {
    MfDev d;
    d.sfirst = sfirst.p; d.m = m.p; d.fo = fo.p; d.iptr = iptr.p; d.idx = idx.p; d.cptr = cptr.p;
    d.clist = clist.p; d.eptr = eptr.p; d.emap = emap.p; d.vo = vo.p;
    d.front = front.p; d.child = child.p; d.arow = arow.p; d.acol = acol.p; d.aslot = aslot.p;
    return d;
  }
};

MfLu::MfLu() : impl_(new Impl) {}
MfLu::~MfLu() { delete impl_; }

int MfLu::setup(const LuSymbolic& s, const int* rowptr, const int* colind, void* stream, bool want_fp32) {
  Impl& I = *impl_;
  I.st = (hipStream_t)stream;
  int rc = mf_plan(s, rowptr, colind, I.P);
  if (rc != XG_OK) return rc;
  const MfPlan& P = I.P;
  // every index a kernel reads is checked here
  for (int v : P.idx) if (v < 0 || v >= P.n) return XG_E_SETUP;
  for (int k : P.aslot) if (k < 0 || k >= s.nnz_a) return XG_E_SETUP;
  for (int c : P.clist) if (c < 0 || c >= P.ns) return XG_E_SETUP;
  for (int t = 0; t < P.ns; ++t) {
    if (P.m[t] < P.sfirst[t + 1] - P.sfirst[t] || P.sfirst[t + 1] <= P.sfirst[t]) return XG_E_SETUP;
    for (int e = P.eptr[t]; e < P.eptr[t + 1]; ++e) {
      if (P.sparent[t] < 0 || P.emap[e] < 0 || P.emap[e] >= P.m[P.sparent[t]]) return XG_E_SETUP;
      if (e > P.eptr[t] && P.emap[e] <= P.emap[e - 1]) return XG_E_SETUP;   // assembly bisects the map
    }
  }
  std::vector<MfFront> fr(P.ns);
  std::vector<MfChild> chv(P.clist.size());
  for (int t = 0; t < P.ns; ++t) {
    const int np = P.sfirst[t + 1] - P.sfirst[t];
    fr[t] = MfFront{P.fo[t], P.m[t], np, P.sfirst[t], P.iptr[t], P.cptr[t], P.cptr[t + 1], P.vo[t], 0};
    for (int i = 0; i < P.m[t]; ++i)
      for (int q = P.arow[P.vo[t] + i]; q < P.arow[P.vo[t] + i + 1]; ++q)
        if (P.acol[q] < 0 || P.acol[q] >= P.m[t]) return XG_E_SETUP;
  }
  for (size_t c = 0; c < P.clist.size(); ++c) {
    const int t = P.clist[c], np = P.sfirst[t + 1] - P.sfirst[t];
    chv[c] = MfChild{P.fo[t] + (long long)np * P.m[t] + np, P.m[t], P.m[t] - np, P.eptr[t], P.vo[t] + np};
  }
  hipStream_t st = I.st;
  MFCHK(I.front.up(fr, st)); MFCHK(I.child.up(chv, st));
  MFCHK(I.arow.up(P.arow, st)); MFCHK(I.acol.up(P.acol, st)); MFCHK(I.aslot.up(P.aslot, st));
  MFCHK(I.sfirst.up(P.sfirst, st)); MFCHK(I.m.up(P.m, st)); MFCHK(I.iptr.up(P.iptr, st)); MFCHK(I.idx.up(P.idx, st));
  MFCHK(I.cptr.up(P.cptr, st)); MFCHK(I.clist.up(P.clist, st)); MFCHK(I.eptr.up(P.eptr, st));
  MFCHK(I.emap.up(P.emap, st)); MFCHK(I.vo.up(P.vo, st)); MFCHK(I.fo.up(P.fo, st));
  MFCHK(I.prow.up(s.perm_row, st)); MFCHK(I.pcol.up(s.perm_col, st));
  MFCHK(I.bad.alloc(2));
  MFCHK(I.F64.alloc(P.fo[P.ns])); MFCHK(I.V64.alloc(P.vo[P.ns])); MFCHK(I.y64.alloc(P.n)); MFCHK(I.b64.alloc(P.n));
  if (want_fp32) { MFCHK(I.F32.alloc(P.fo[P.ns])); MFCHK(I.V32.alloc(P.vo[P.ns])); MFCHK(I.y32.alloc(P.n)); }
  // per level: tiny fronts (one launch), larger fronts (blocked panels, all
  // fronts of the level in each panel launch)
  const int nl = (int)P.lvl_ptr.size() - 1;
  std::vector<int> tl, bl;
  std::vector<int4> se;
  int max_slots = 1;
  I.tiny_off.assign(nl + 1, 0);
  I.big_off.assign(nl + 1, 0);
  I.tiny_half.assign(nl, 0);
  I.steps.assign(nl, {});
  I.big_maxm = 0;
  for (int l = 0; l < nl; ++l) {
    I.tiny_off[l] = (int)tl.size();
    I.big_off[l] = (int)bl.size();
    int maxp = 0;
    std::vector<int> mid;
    for (int q = P.lvl_ptr[l]; q < P.lvl_ptr[l + 1]; ++q) {
      const int t = P.lvl_s[q];
      if (P.m[t] <= kMfTiny) {
        (P.m[t] <= kMfTiny / 2 ? tl : mid).push_back(t);
      } else {
        bl.push_back(t);
        I.big_maxm = std::max(I.big_maxm, P.m[t]);
        maxp = std::max(maxp, (P.sfirst[t + 1] - P.sfirst[t] + kMfPanel - 1) / kMfPanel);
      }
    }
    I.tiny_half[l] = (int)tl.size();
    tl.insert(tl.end(), mid.begin(), mid.end());
    const int nb = (int)bl.size() - I.big_off[l];
    max_slots = std::max(max_slots, nb);
    for (int j = 0; nb > 0 && j <= maxp; ++j) {
      Impl::Step S{j * kMfPanel, (int)se.size(), 0};
      // the panels first (they are the longer chain), then the update tiles
      for (int pass = 0; pass < 2; ++pass)
        for (int slot = 0; slot < nb; ++slot) {
          const int t = bl[I.big_off[l] + slot];
          const int np = P.sfirst[t + 1] - P.sfirst[t];
          if (S.p0 >= np + kMfPanel) continue;                 // finished at an earlier step
          const int rest = P.m[t] - std::min(np, S.p0 + kMfPanel);
          const int nrb = (rest + 63) / 64;
          if (pass == 0) {
            if (S.p0 < np)
              for (int i = 0; i < std::max(1, nrb); ++i) se.push_back(make_int4(t, i, -1, slot));
            else if (rest == 0) se.push_back(make_int4(t, 0, -2, slot));
          } else if (j > 0) {
            // after the last panel tile (0, 0) copies the diagonal
            for (int ti = 0; ti * kMfTileRows < rest; ++ti)
              for (int tj = 0; tj < nrb; ++tj) se.push_back(make_int4(t, ti, tj, slot));
          }
        }
      S.cnt = (int)se.size() - S.off;
      I.steps[l].push_back(S);
    }
  }
  I.tiny_off[nl] = (int)tl.size();
  I.big_off[nl] = (int)bl.size();
  MFCHK(I.tiny_list.up(tl, st));
  MFCHK(I.big_list.up(bl, st));
  MFCHK(I.sent.up(se, st));
  MFCHK(I.dbuf.alloc((size_t)max_slots * 2 * kMfPanel * kMfPanel));
  // assembly of the larger fronts, ranges of rows and columns (the tiny fronts
  // assemble themselves inside their factor kernel)
  std::vector<int4> ae;
  std::vector<int2> lo;
  I.aoff.assign(nl + 1, 0);
  for (int l = 0; l < nl; ++l) {
    I.aoff[l] = (int)ae.size() / 2;
    for (int b = I.big_off[l]; b < I.big_off[l + 1]; ++b) {
      const int t = bl[b], m = P.m[t];
      const int w = std::min(m, kMfAsm / 4), rows = std::min(kMfAsmRows, kMfAsm / w);
      for (int r0 = 0; r0 < m; r0 += rows) {
        const int off = (int)lo.size();
        for (int c = P.cptr[t]; c < P.cptr[t + 1]; ++c) {
          const int ch = P.clist[c];
          const int* eb = P.emap.data() + P.eptr[ch];
          const int* ee = P.emap.data() + P.eptr[ch + 1];
          lo.push_back(make_int2((int)(std::lower_bound(eb, ee, r0) - eb), (int)(std::lower_bound(eb, ee, r0 + rows) - eb)));
        }
        for (int j0 = 0; j0 < m; j0 += w) {
          ae.push_back(make_int4(t, r0, std::min(rows, m - r0), off));
          ae.push_back(make_int4(j0, std::min(w, m - j0), 0, 0));
        }
      }
    }
  }
  I.aoff[nl] = (int)ae.size() / 2;
  MFCHK(I.aent.up(ae, st));
  MFCHK(I.alo.up(lo, st));
  MFCHK(hipStreamSynchronize(st));
  return XG_OK;
}

double MfLu::flops() const { return impl_->P.flops; }
long long MfLu::front_elements() const { return impl_->P.fo.empty() ? 0 : impl_->P.fo[impl_->P.ns]; }
int MfLu::levels() const { return (int)impl_->P.lvl_ptr.size() - 1; }
int MfLu::supernodes() const { return impl_->P.ns; }

template <class T>
__global__ void k_mf_flag_init(int* bad) {
  bad[0] = 0x7fffffff;
  bad[1] = 0;
}

// the launches of one refactor (no host work: the sequence is captured)
template <class T>
static int mf_factor_enqueue(MfLu::Impl& I, const double* vals_dev, int nnz, T* F) {
  const MfPlan& P = I.P;
  hipStream_t st = I.st;
  hipLaunchKernelGGL(k_mf_flag_init<T>, dim3(1), dim3(1), 0, st, I.bad.p);
  const MfDev d = I.dev();
  T* dbuf = reinterpret_cast<T*>(I.dbuf.p);
  const int nl = (int)P.lvl_ptr.size() - 1;
  for (int l = 0; l < nl; ++l) {
    const int na = I.aoff[l + 1] - I.aoff[l];
    if (na)
      hipLaunchKernelGGL(k_mf_assemble<T>, dim3(na), dim3(256), 0, st, d, I.aent.p + 2 * I.aoff[l], I.alo.p, vals_dev, F);
    const int n32 = I.tiny_half[l] - I.tiny_off[l], n64 = I.tiny_off[l + 1] - I.tiny_half[l];
    if (n32)
      hipLaunchKernelGGL((k_mf_factor_tiny<T, kMfTiny / 2>), dim3(n32), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l],
                         vals_dev, F, I.bad.p);
    if (n64)
      hipLaunchKernelGGL((k_mf_factor_tiny<T, kMfTiny>), dim3(n64), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_half[l],
                         vals_dev, F, I.bad.p);
    for (const auto& S : I.steps[l])
      hipLaunchKernelGGL(k_mf_step<T>, dim3(S.cnt), dim3(kMfStep), 0, st, d, I.sent.p + S.off, S.p0, F, dbuf,
                         (S.p0 / kMfPanel) & 1, I.bad.p);
  }
  MFCHK(hipGetLastError());
  return XG_OK;
}

// Replays the graph captured for `key`, capturing it on first use.
template <class Enqueue>
static int mf_replay(MfLu::Impl& I, const void* const* key, int nkey, Enqueue enqueue) {
  MfGraph* g = nullptr;
  for (auto& c : I.graphs)
    if (std::equal(key, key + nkey, c.key)) { g = &c; break; }
  if (!g) {
    hipGraph_t graph = nullptr;
    MFCHK(hipStreamBeginCapture(I.st, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue();
    hipError_t e = hipStreamEndCapture(I.st, &graph);
    if (rc != XG_OK) { if (graph) (void)hipGraphDestroy(graph); return rc; }
    MFCHK(e);
    MfGraph ng;
    std::copy(key, key + nkey, ng.key);
    e = hipGraphInstantiate(&ng.exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    MFCHK(e);
    I.graphs.push_back(ng);
    g = &I.graphs.back();
  }
  MFCHK(hipGraphLaunch(g->exec, I.st));
  return XG_OK;
}

template <class T>
static int mf_factor_t(MfLu::Impl& I, const double* vals_dev, int nnz, T* F, int* bad_out, int* hard_out) {
  const void* key[8] = {(const void*)1, vals_dev, F, (const void*)(long long)nnz, nullptr, nullptr, nullptr, nullptr};
  int rc = mf_replay(I, key, 8, [&] { return mf_factor_enqueue<T>(I, vals_dev, nnz, F); });
  if (rc != XG_OK) return rc;
  int res[2];
  MFCHK(hipMemcpyAsync(res, I.bad.p, sizeof(res), hipMemcpyDeviceToHost, I.st));
  MFCHK(hipStreamSynchronize(I.st));
  *bad_out = res[0] == 0x7fffffff ? 0 : res[0];
  *hard_out = res[1];
  return XG_OK;
}

template <class T>
static int mf_solve_enqueue(MfLu::Impl& I, const T* F, T* V, T* y, double* bp, const double* b_dev, double* x_dev,
                            int* nan_flag) {
  const MfPlan& P = I.P;
  hipStream_t st = I.st;
  const MfDev d = I.dev();
  const int n = P.n;
  // the larger fronts keep their vector in LDS when it fits in 64 KB with the
  // 64x65 block, else in their slice of V
  const size_t blk_bytes = 64 * 65 * sizeof(T);
  const bool ldsv = blk_bytes + (size_t)I.big_maxm * sizeof(T) <= 65536;
  const size_t big_lds = blk_bytes + (ldsv ? (size_t)I.big_maxm * sizeof(T) : 0);
  hipLaunchKernelGGL(k_mf_perm_in<T>, dim3((n + 255) / 256), dim3(256), 0, st, n, I.prow.p, b_dev, bp);
  const int nl = (int)P.lvl_ptr.size() - 1;
  for (int l = 0; l < nl; ++l) {
    const int nt = I.tiny_off[l + 1] - I.tiny_off[l], nb = I.big_off[l + 1] - I.big_off[l];
    if (nt)
      hipLaunchKernelGGL(k_mf_fwd_tiny<T>, dim3(nt), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l], F, V,
                         bp, y);
    if (nb)
      hipLaunchKernelGGL(k_mf_fwd_big<T>, dim3(nb), dim3(kMfSolveBlock), big_lds, st, d, I.big_list.p + I.big_off[l],
                         F, V, bp, y, (int)ldsv);
  }
  for (int l = nl - 1; l >= 0; --l) {
    const int nt = I.tiny_off[l + 1] - I.tiny_off[l], nb = I.big_off[l + 1] - I.big_off[l];
    if (nb)
      hipLaunchKernelGGL(k_mf_bwd_big<T>, dim3(nb), dim3(kMfSolveBlock), big_lds, st, d, I.big_list.p + I.big_off[l],
                         F, V, y, (int)ldsv);
    if (nt)
      hipLaunchKernelGGL(k_mf_bwd_tiny<T>, dim3(nt), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l], F, y);
  }
  hipLaunchKernelGGL(k_mf_perm_out<T>, dim3((n + 255) / 256), dim3(256), 0, st, n, I.pcol.p, y, x_dev, nan_flag);
  MFCHK(hipGetLastError());
  return XG_OK;
}

template <class T>
static int mf_solve_t(MfLu::Impl& I, const T* F, T* V, T* y, double* bp, const double* b_dev, double* x_dev,
                      int* nan_flag) {
  const void* key[8] = {(const void*)2, F, V, y, bp, b_dev, x_dev, nan_flag};
  return mf_replay(I, key, 8, [&] { return mf_solve_enqueue<T>(I, F, V, y, bp, b_dev, x_dev, nan_flag); });
}

int MfLu::factor(const double* vals_dev, int nnz, bool fp32, int* bad, int* hard) {
  Impl& I = *impl_;
  if (fp32) {
    if (!I.F32.p) return XG_E_ARG;
    return mf_factor_t<float>(I, vals_dev, nnz, I.F32.p, bad, hard);
  }
  return mf_factor_t<double>(I, vals_dev, nnz, I.F64.p, bad, hard);
}

int MfLu::solve(const double* b_dev, double* x_dev, bool fp32, int* nan_flag) {
  Impl& I = *impl_;
  if (fp32) {
    if (!I.F32.p) return XG_E_ARG;
    return mf_solve_t<float>(I, I.F32.p, I.V32.p, I.y32.p, I.b64.p, b_dev, x_dev, nan_flag);
  }
  return mf_solve_t<double>(I, I.F64.p, I.V64.p, I.y64.p, I.b64.p, b_dev, x_dev, nan_flag);
}

static size_t round32(size_t v) { return (v + 31) & ~(size_t)31; }

size_t MfLu::solve_work_doubles() const {
  const MfPlan& P = impl_->P;
  return round32((size_t)P.vo[P.ns]) + 2 * round32((size_t)P.n);
}

int MfLu::solve_ext(const double* b_dev, double* x_dev, int* nan_flag, double* work) {
  Impl& I = *impl_;
  const MfPlan& P = I.P;
  double* V = work;
  double* y = V + round32((size_t)P.vo[P.ns]);
  double* bp = y + round32((size_t)P.n);
  return mf_solve_t<double>(I, I.F64.p, V, y, bp, b_dev, x_dev, nan_flag);
}

}  // namespace xg
