// Multifrontal numeric LU for large systems (power-grid meshes, gate
// arrays): the factorisation that AmesosSolver::doSolve
// (src/LinearAlgebraServicesPKG/N_LAS_AmesosSolver.C:216-478) gets from KLU,
// restructured for the GPU.  The symbolic analysis (mf_analyse: maximum
// transversal, the cheapest of minimum degree and nested dissection, a tree of
// supernodes merged where that adds few zeros) gives each supernode a dense
// frontal matrix; the tree is processed level by level (all fronts of a level in
// the same launches):
//
//   assemble  F_s = A entries of s's rows and columns + extend-add of the
//             children's Schur complements, in LDS, in a fixed order
//   factor    dense LU of the pivot block, L21, U12 and the Schur complement
//             F22 -= L21 U12; fronts of order <= 64 by one wavefront each (with
//             their assembly), larger ones by 32-column panels, one launch per
//             panel that updates by the panel before and factors its own
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
  // every row and column is eliminated once, by one front; with the nesting of the
  // rows and the place of every entry of A, checked below, the fronts hold all fill
  if ((int)s.perm_row.size() != n || (int)s.perm_col.size() != n || (int)s.rinv.size() != n || (int)s.pinv.size() != n)
    return XG_E_SETUP;
  if (s.sfirst[0] != 0) return XG_E_SETUP;
  for (int t = 0; t < ns; ++t)
    if (s.sfirst[t + 1] <= s.sfirst[t]) return XG_E_SETUP;
  for (int i = 0; i < n; ++i) {
    const int r = s.perm_row[i], c = s.perm_col[i];
    if (r < 0 || r >= n || c < 0 || c >= n || s.rinv[r] != i || s.pinv[c] != i) return XG_E_SETUP;
  }
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
  const MfFront* front; const MfChild* child; const int* emap;
  const int* bidx; const int* xidx;      // of the fronts' rows: index into b, into x
  const int* arow; const int* acol; const int* aslot;
};

constexpr int kMfTiny = 64;     // fronts up to this order: one wavefront, the front in LDS
constexpr int kMfPanel = 32;    // panel width of the blocked factorisation (64 spills the register panel)

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

// Sums over the wavefront, of four values at once: lanes of row k (16 k to 16 k +
// 15) get the sum of the k-th.  Halves and rows are exchanged between two
// registers (so that one addition serves two values), the rest within rows; the
// order of each sum is the butterfly's (lane distances 32, 16, 8, 4, 2, 1).  In
// registers, as a butterfly through LDS takes 48 accesses where this takes none
// (solve of a 64-row block by 13 wavefronts: 6300 cycles of sums, 1300 now).
__device__ __forceinline__ void mf_swap32(unsigned& a, unsigned& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
__device__ __forceinline__ void mf_swap16(unsigned& a, unsigned& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
// upper half of a <-> lower half of b (odd rows of a <-> even rows of b), added
template <int N, class T>
__device__ __forceinline__ T mf_fold(T a, T b) {
  constexpr int W = sizeof(T) / 4;
  unsigned ua[W], ub[W];
  __builtin_memcpy(ua, &a, sizeof(T));
  __builtin_memcpy(ub, &b, sizeof(T));
#pragma unroll
  for (int w = 0; w < W; ++w) {
    if (N == 32) mf_swap32(ua[w], ub[w]);
    else mf_swap16(ua[w], ub[w]);
  }
  __builtin_memcpy(&a, ua, sizeof(T));
  __builtin_memcpy(&b, ub, sizeof(T));
  return a + b;
}
template <int N, class T>
__device__ __forceinline__ T mf_add_ror(T v) {
  constexpr int W = sizeof(T) / 4;
  int u[W];
  __builtin_memcpy(u, &v, sizeof(T));
#pragma unroll
  for (int w = 0; w < W; ++w) u[w] = __builtin_amdgcn_update_dpp(0, u[w], 0x120 + N, 0xf, 0xf, true);
  T o;
  __builtin_memcpy(&o, u, sizeof(T));
  return v + o;
}
template <class T>
__device__ __forceinline__ T mf_sum4(T v0, T v1, T v2, T v3) {
  T s = mf_fold<16>(mf_fold<32>(v0, v2), mf_fold<32>(v1, v3));
  s = mf_add_ror<8>(s);
  s = mf_add_ror<4>(s);
  s = mf_add_ror<2>(s);
  return mf_add_ror<1>(s);
}
// x[r + k] -= the sum of acc[k], k < min(nr, NR)
template <int NR, class T>
__device__ __forceinline__ void mf_sub_sums(T* x, int r, int nr, int lane, const T (&acc)[NR]) {
  static_assert(NR == 4 || NR == 5, "");
  const T s = mf_sum4(acc[0], acc[1], acc[2], acc[3]);
  const int k = lane >> 4;
  if ((lane & 15) == 0 && k < nr) x[r + k] -= s;
  if (NR == 5) {
    const T s4 = mf_sum4(acc[NR - 1], acc[NR - 1], acc[NR - 1], acc[NR - 1]);
    if (lane == 0 && 4 < nr) x[r + 4] -= s4;
  }
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
// diagonal's 32 dependent pivots and a substitution (12.4 us where the two
// launches took 31.6, on the 865-order root of a 512 x 512 grid, of which the 32
// pivots take 4.3; mean over all its steps 13.2, 14.4 with the loads of C and L
// waited for before U's and the substitution's rows read one ahead).
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
// first product.  The products are summed apart and subtracted once: an entry is
// rounded once per panel, where with the entry as the first summand every product
// rounds it (error of a solve, 300 x 77 mesh with FP32 factors: 1.12e-6, 0.98e-6
// so; 512 x 512 mesh in FP64: 1.99e-15, 1.74e-15; same time).
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
  typename MfAcc<T>::V old[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const unsigned o = (unsigned)(min(i0 + 16 * a + MfAcc<T>::row(lk, r), i1 - 1) - i0) * row;
#pragma unroll
      for (int b = 0; b < NB; ++b) old[a][b][r] = mf_at(C, o + cj[b]);
    }
  if (kw <= 0) {
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b] = old[a][b];
    return;
  }
  // step k of the product takes the columns 8 lk + k of L (a lane's eight lie
  // next to each other in memory) and the same rows of U
  T l[NA][kMfPanel / 4], u[NB][kMfPanel / 4];
  const T* Lb = Fs + i0 * ld + q0;
  const T* Ub = Fs + q0 * ld + j0;
  // (in pairs, the last of an odd kw with the one before it: no branch, which
  // would have the loads before it waited for; a front's last row may be read one
  // value past its end, the buffer has it)
  typedef T Pair __attribute__((ext_vector_type(2), aligned(sizeof(T))));
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    const unsigned o = (unsigned)(min(i0 + 16 * a + lr, i1 - 1) - i0) * row;
#pragma unroll
    for (int k = 0; k < kMfPanel / 4; k += 2) {
      const unsigned c = (unsigned)max(min(8 * lk + k, kw - 2), 0);
      const Pair p = *reinterpret_cast<const Pair*>(reinterpret_cast<const char*>(Lb) + o + c * (unsigned)sizeof(T));
      l[a][k] = p.x;
      l[a][k + 1] = p.y;
    }
  }
#pragma unroll
  for (int k = 0; k < kMfPanel / 4; ++k) {
    const unsigned o = (unsigned)min(8 * lk + k, kw - 1) * row;
#pragma unroll
    for (int b = 0; b < NB; ++b) u[b][k] = mf_at(Ub, o + cj[b]);
  }
  // (L's signs and its columns past kw only here, behind U's loads)
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int k = 0; k < kMfPanel / 4; ++k)
#pragma unroll
    for (int a = 0; a < NA; ++a) {
      const int c = 8 * lk + k;
      const T lv = c < kw ? ((k & 1) == 0 && c > 0 && c == kw - 1 ? l[a][k | 1] : l[a][k]) : (T)0;
#pragma unroll
      for (int b = 0; b < NB; ++b) acc[a][b] = MfAcc<T>::mma(lv, u[b][k], k == 0 ? typename MfAcc<T>::V{} : acc[a][b]);
    }
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = old[a][b] - acc[a][b];
}

__device__ __forceinline__ double mf_fma(double a, double b, double c) { return fma(a, b, c); }
__device__ __forceinline__ float mf_fma(float a, float b, float c) { return fmaf(a, b, c); }

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

// right-looking LU of the rows in registers (lane t: row t), the first np <= N
// pivots; rd: lane k's reciprocal of pivot k.  Constant trip counts keep the
// rows in registers.  A multiplier is the product with the reciprocal and the
// correction of its remainder: rounded once, as a division (the product alone
// rounds twice: errors of solves on meshes about 5 % larger, for 1.7 % of the
// refactor's time on a 512 x 512 mesh).
template <int N, class T>
__device__ __forceinline__ void mf_factor_rows(T (&v)[N], int lane, int np, T& rd) {
  MfRecip<T> rec;
  rec.p = mf_bcast(v[0], 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) rec.stage(i);
  mf_for<N>([&](auto kc) MF_INLINE {
    constexpr int k = kc, k1 = k + 1 < N ? k + 1 : k;
    if (k >= np) return;
    const T rp = rec.x;
    rd = lane == k ? rp : rd;
    const T pv = rec.p, q = v[k] * rp;
    const T l = lane > k ? mf_fma(mf_fma(-q, pv, v[k]), rp, q) : (T)0;
    v[k] = lane > k ? l : v[k];
    if constexpr (k1 > k) v[k1] -= l * mf_bcast(v[k1], k);
    rec.p = mf_bcast(v[k1], k1);
    mf_row_update<N>(v, l, k, k + 2, rec);
    __builtin_amdgcn_sched_barrier(0);
  });
}

__device__ __forceinline__ unsigned mf_abs_high(double v) {
  return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu;
}
__device__ __forceinline__ unsigned mf_abs_high(float v) { return __float_as_uint(v) & 0x7fffffffu; }

// pivots up to here have a reciprocal that overflows
template <class T> constexpr T kMfNoPivot = (T)0x1p-1024;
template <> constexpr float kMfNoPivot<float> = 0x1p-128f;

// the lowest of the first np columns of factored rows (lane t: row t, t < rows;
// also in memory, at(k)) with a bad pivot or a multiplier beyond KLU's
// threshold, or N.  The high words of absolute values order like the values, NaN
// last: one maximum over the multipliers and the pivot's word tell whether
// anything has to be looked at.
template <int N, class T, class At>
__device__ __forceinline__ int mf_check_rows(const T (&v)[N], int lane, int rows, int np, const At& at, bool& hard) {
  unsigned top = 0, piv = mf_abs_high((T)1);
  // (the comparisons are made here: kept from the factorisation they would spill)
  asm volatile("" : "+v"(lane), "+v"(np));
  const int lim = min(lane, np), own = lane < np ? lane : -1;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const unsigned h = mf_abs_high(v[k]);
    top = max(top, lim > k ? h : 0);
    piv = own == k ? h : piv;
  }
  const bool look = lane < rows && (top >= mf_abs_high((T)1.0e3) || piv <= mf_abs_high(kMfNoPivot<T>) || piv >= mf_abs_high((T)INFINITY));
  int first = N;
  if (__any(look) && lane < rows)
    for (int k = min(min(np, N) - 1, lane); k >= 0; --k) {
      const double a = fabs((double)at(k));
      const bool p = lane == k;
      if (p ? !(a > (double)kMfNoPivot<T>) || !isfinite(a) : !(a <= 1.0e3)) { first = k; hard |= p; }
    }
  return first;
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
// offset into parts}, {first column, columns, parts, 0}; at most kMfAsm elements, held
// in LDS until they are complete, so a front is written once and never cleared
// or read back).  Wavefront w owns the rows with index % 4 = w: no wavefront
// waits for another.  The parts are the children with rows in the range (a front
// with a supply row has many others), their positions loaded one part ahead; a
// child's rows map to increasing parent rows.  Per part and 256 columns a wavefront
// issues the loads of up to four rows at once; a part is a round trip, which bounds
// fronts of many children (512 x 512 grid, all levels: 242 us with A's entries in,
// where clearing the fronts, scattering A and adding the children in memory took
// 400; roots of a 2000-gate array 42 us).
constexpr int kMfAsmRows = 16;
// a child in a range: its Schur complement, and its rows [a, b) that land there
struct MfPart { long long src; int ld, nu, em, a, b, pad; };
constexpr int kMfAsm = 4096;

template <class T>
__global__ void __launch_bounds__(256) k_mf_assemble(MfDev d, const int4* ent, const MfPart* parts, const double* vals,
                                                     T* F) {
  __shared__ T R[kMfAsm];
  const int4 e = ent[2 * blockIdx.x], ec = ent[2 * blockIdx.x + 1];
  const MfFront f = d.front[e.x];
  const int r0 = e.y, rows = e.z, j0 = ec.x, w = ec.y;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const MfPart* part = parts + e.w;
  const int n_part = ec.z;
  MfPart next{};
  int next_er = -1, next_eb[4] = {-1, -1, -1, -1};
  auto fetch = [&](int c) MF_INLINE {
    if (c >= n_part) return;
    next = part[c];
    const int* em = d.emap + next.em;
    next_er = next.a + lane < next.b ? em[next.a + lane] - r0 : -1;
#pragma unroll
    for (int q = 0; q < 4; ++q) next_eb[q] = lane + 64 * q < next.nu ? em[lane + 64 * q] - j0 : -1;
  };
  fetch(0);
  // A's entries, the wavefront's rows side by side (each is three dependent loads)
  constexpr int NR = kMfAsmRows / 4;
  int q0[NR], q1[NR], col[NR], slot[NR];
  T av[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const int i = min(4 * k + wave, rows - 1);
    q0[k] = d.arow[f.vo + r0 + i];
    q1[k] = 4 * k + wave < rows ? d.arow[f.vo + r0 + i + 1] : q0[k];
  }
#pragma unroll
  for (int k = 0; k < NR; ++k) {
    const bool in = q0[k] + lane < q1[k];
    col[k] = in ? d.acol[q0[k] + lane] - j0 : -1;
    slot[k] = in ? d.aslot[q0[k] + lane] : 0;
  }
#pragma unroll
  for (int k = 0; k < NR; ++k) av[k] = q0[k] + lane < q1[k] ? (T)vals[slot[k]] : (T)0;
  for (int i = wave; i < rows; i += 4)
    for (int j = lane; j < w; j += 64) R[i * w + j] = (T)0;
  mf_wave_fence();
  // (an entry listed twice in a row adds up)
#pragma unroll
  for (int k = 0; k < NR; ++k)
    if (col[k] >= 0 && col[k] < w) atomicAdd(&R[(4 * k + wave) * w + col[k]], av[k]);
#pragma unroll
  for (int k = 0; k < NR; ++k)
    for (int q = q0[k] + 64 + lane; q < q1[k]; q += 64) {
      const int j = d.acol[q] - j0;
      if (j >= 0 && j < w) atomicAdd(&R[(4 * k + wave) * w + j], (T)vals[d.aslot[q]]);
    }
  mf_wave_fence();
  // (the next child's positions are loaded beside this one's values)
  for (int c = 0; c < n_part; ++c) {
    const MfPart ch = next;
    const int er = next_er;
    int ebn[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) ebn[q] = next_eb[q];
    const int* em = d.emap + ch.em;
    // slot k: the child's row that lands on this wavefront's row 4 k + wave
    int a[kMfAsmRows / 4];
#pragma unroll
    for (int k = 0; k < kMfAsmRows / 4; ++k) {
      const unsigned long long hit = __ballot(er == 4 * k + wave);
      a[k] = hit ? ch.a + (int)__builtin_ctzll(hit) : -1;
    }
    const T* Fc = F + ch.src;
    for (int c0 = lane; c0 - lane < ch.nu; c0 += 256) {
      int eb[4];
      T cv[kMfAsmRows / 4][4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int b = c0 + 64 * q;
        const int j = c0 == lane ? ebn[q] : b < ch.nu ? em[b] - j0 : -1;
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
      if (c0 == lane) fetch(c + 1);
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
// LDS traffic (512 x 512 grid, all levels: 297 us, 656 with the elimination in LDS).
template <class T, int N>
__global__ void __launch_bounds__(64) k_mf_factor_tiny(MfDev d, const int* list, const double* vals, T* F, int* bad, int* fail) {
  constexpr int ld = N + 1;
  __shared__ T A[N * ld];
  const MfFront f = d.front[list[blockIdx.x]];
  const int ms = f.m, np = f.np, t = threadIdx.x;
  MfChild next{};
  int next_e = 0;                                    // parent position of its row/column t
  auto fetch = [&](int c) MF_INLINE {
    if (c >= f.c1) return;
    next = d.child[c];
    next_e = t < next.nu ? d.emap[next.em + t] : 0;
  };
  fetch(f.c0);
  if (t < ms) {
    T* row = A + t * ld;
    const int qa = d.arow[f.vo + t], qb = d.arow[f.vo + t + 1];
    for (int j = 0; j < ms; ++j) row[j] = (T)0;
    // eight entries at a time: their positions, then their values
    for (int q = qa; q < qb; q += 8) {
      int col[8], slot[8];
      T av[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int p = min(q + i, qb - 1);
        col[i] = d.acol[p];
        slot[i] = d.aslot[p];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) av[i] = (T)vals[slot[i]];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (q + i < qb) row[col[i]] += av[i];
    }
  }
  mf_wave_fence();
  // a child's update has at most ms rows and columns: lane t adds column t; the
  // next child's positions are loaded beside this one's values
  for (int c = f.c0; c < f.c1; ++c) {
    const MfChild ch = next;
    const int nu = ch.nu, eb = next_e;
    const T* cb = F + ch.src + t;
    for (int a = 0; a < nu; a += 16) {
      T v[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) v[q] = (t < nu && a + q < nu) ? cb[(long long)(a + q) * ch.ld] : (T)0;
      if (a == 0) fetch(c + 1);
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
  bool hard = false;
  T rd = (T)0;
  mf_factor_rows<N>(v, t, np, rd);
  if (t < ms) {
    T* row = A + t * ld;
#pragma unroll
    for (int q = 0; q < N; ++q) row[q] = v[q];
  }
  mf_wave_fence();
  const int first = mf_check_rows<N>(v, t, ms, np, [&](int k) MF_INLINE { return A[t * ld + k]; }, hard);
  T* Fs = F + f.fo;
#pragma unroll 8
  for (int i = 0; i < ms; ++i)
    if (t < ms) Fs[(long long)i * ms + t] = A[i * ld + t];
  if (first < np) { atomicMin(bad, f.first + first + 1); *fail = 1; }
  if (__any(hard) && t == 0) atomicOr(bad + 1, 1);
}

constexpr int kMfStep = 192;              // threads of a step workgroup: three wavefronts
constexpr int kMfTileRows = 96;           // rows of an update tile: 32 per wavefront
constexpr int kMfDs = kMfPanel + 2;       // row stride of the diagonal factors in LDS (16-byte pairs)
constexpr int kMfTile = 64 * (kMfPanel + 1) > kMfPanel * 65 ? 64 * (kMfPanel + 1) : kMfPanel * 65;

// an entry and its front's numbers, so that the kernel's first loads are its tiles
struct MfStep { int y, z, w, m, np, first; long long fo; };

template <class T>
__global__ void __launch_bounds__(kMfStep) __attribute__((amdgpu_waves_per_eu(2))) k_mf_step(const MfStep* ent, int p0, T* F, T* dbuf, int half, int* bad,
                                                     int* fail) {
  constexpr int PW = kMfPanel;
  __shared__ __attribute__((aligned(16))) T Du[PW * kMfDs];   // U11 by rows
  __shared__ __attribute__((aligned(16))) T Dl[PW * kMfDs];   // L11 by columns; the updated block before it is factored
  __shared__ T Ts[2][kMfTile];
  const MfStep e = ent[blockIdx.x];
  const int slot = e.w, ms = e.m, np = e.np;
  const int base = min(np, p0 + PW), q0 = p0 - PW, kw = q0 >= 0 ? min(PW, np - q0) : 0;
  T* Fs = F + e.fo;
  const long long ld = ms;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, lr = lane & 15, lk = lane >> 4;
  typedef typename MfAcc<T>::V V;
  // the front's first entry: panel j - 1's diagonal factors into the front
  auto copy_diagonal = [&](int t0, int nt) MF_INLINE {
    if (kw <= 0 || e.y != 0 || e.z > 0) return;
    const T* db = dbuf + ((long long)slot * 2 + (half ^ 1)) * PW * PW;
    for (int x = t0; x < PW * PW; x += nt) {
      const int i = x / PW, j = x % PW;
      if (i < kw && j < kw) Fs[(q0 + i) * ld + q0 + j] = db[x];
    }
  };
  if (e.z != -1) copy_diagonal(t, kMfStep);
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
    __builtin_amdgcn_s_setprio(3);       // the others wait for this wavefront: its loads first
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
  if (wave > 0) copy_diagonal(t - 64, kMfStep - 64);      // (beside the diagonal's pivots)
  mf_wave_fence();          // each wavefront reads back its own tile: no wait for the others
  int failed = PW;          // first column whose pivot or multiplier fails
  bool hard = false;
  T v[PW];
  if (wave == 0) {
    const int row = lane & 31;
#pragma unroll
    for (int q = 0; q < PW; ++q) v[q] = Dl[row * kMfDs + q];
    T rd = (T)1;
    mf_factor_rows<PW>(v, lane, PW, rd);
    if (lane < PW) Du[lane * kMfDs + PW] = rd;      // the pivots' reciprocals behind the rows
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
  }
  __syncthreads();
  if (wave == 0)
    failed = mf_check_rows<PW>(v, lane, PW, PW, [&](int k) MF_INLINE { return Du[lane * kMfDs + k]; }, hard);
  if (wave == 0 && e.y == 0 && lane < PW) {
    T* db = dbuf + ((long long)slot * 2 + half) * PW * PW + lane * PW;
#pragma unroll
    for (int q = 0; q < PW; ++q) db[q] = v[q];
  }
  if (has) {
    // the factors' rows come two values at a time from LDS, two rows ahead of the
    // one applied (one ahead for the first, longest ones: registers); a row's
    // address is tied to v[k], so that no more are held
    typedef T Pair __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(3))) T* Lds;
    typedef const __attribute__((address_space(3))) Pair* LdsPair;
    constexpr int K2 = 8;                         // from here on two rows ahead
    Lds pd = (Lds)(lower ? Du : Dl);
    T u[3][PW];
    T rr[3] = {(T)1, (T)1, (T)1};
    auto fetch = [&](auto kc) MF_INLINE {
      constexpr int k = kc;
      if constexpr (k < PW) {
#pragma unroll
        for (int q = (k + 1) & ~1; q < PW; q += 2) {
          const Pair p = *(LdsPair)(pd + k * kMfDs + q);
          u[k % 3][q] = p.x;
          u[k % 3][q + 1] = p.y;
        }
        if (lower) rr[k % 3] = pd[k * kMfDs + PW];
      }
    };
    auto ahead = [&](auto kc) MF_INLINE {
      constexpr int k = kc;
      asm volatile("" : "+v"(pd) : "v"(v[k]));
      if constexpr (k <= K2) fetch(std::integral_constant<int, k + 1>{});
      if constexpr (k >= K2) fetch(std::integral_constant<int, k + 2>{});
    };
    fetch(std::integral_constant<int, 0>{});
    if (lower) {
      const bool valid = o0 + lane < ms;
      mf_for<PW>([&](auto kc) MF_INLINE {
        constexpr int k = kc;
        ahead(kc);
        v[k] *= rr[k % 3];
        if (valid && !(fabs((double)v[k]) <= 1.0e3)) failed = min(failed, k);
#pragma unroll
        for (int q = k + 1; q < PW; ++q) v[q] -= v[k] * u[k % 3][q];
        __builtin_amdgcn_sched_barrier(0);
      });
      // the lane's row of L21: 32 values next to each other
      if (valid) {
        T* to = Fs + (o0 + lane) * ld + p0;
        if (pw == PW) {
          typedef T Pair8 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
#pragma unroll
          for (int q = 0; q < PW; q += 2) *reinterpret_cast<Pair8*>(to + q) = Pair8{v[q], v[q + 1]};
        } else {
#pragma unroll
          for (int q = 0; q < PW; ++q)
            if (q < pw) to[q] = v[q];
        }
      }
    } else {
      const int c = o0 + lane;
      mf_for<PW>([&](auto kc) MF_INLINE {
        constexpr int k = kc;
        ahead(kc);
#pragma unroll
        for (int q = k + 1; q < PW; ++q) v[q] -= u[k % 3][q] * v[k];
        __builtin_amdgcn_sched_barrier(0);
      });
#pragma unroll
      for (int q = 0; q < PW; ++q)
        if (c < ms && q < pw) Fs[(p0 + q) * ld + c] = v[q];
    }
  }
  if (failed < pw) { atomicMin(bad, e.first + p0 + failed + 1); *fail = 1; }
  if (__any(hard) && lane == 0) atomicOr(bad + 1, 1);
}

// ---- solves.  V holds, per front, the vector of its index list: y on the
// pivot rows, the update for the parent below them.  The right-hand side is
// read, and the solution written, in A's numbering.

// partial sums of this lane (to be added over the wavefront) of F[r + k][c] x(c)
// over c in [c0, c1), for the NR rows from r on (rows from nr on repeat the
// last): 4 NR loads in flight, so the rows share their memory round trips
template <int NR, class T, class X>
__device__ __forceinline__ void mf_rows_part(const T* Fs, long long ld, int r, int nr, int c0, int c1, int lane,
                                             const X& x, T (&acc)[NR]) {
  const T* row[NR];
#pragma unroll
  for (int k = 0; k < NR; ++k) { row[k] = Fs + (long long)(r + min(k, nr - 1)) * ld; acc[k] = (T)0; }
  for (int c = c0; c < c1; c += 256) {
    T xv[4], f[NR][4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (c + 64 * q >= c1) break;
      const int jj = min(c + 64 * q + lane, c1 - 1);
#pragma unroll
      for (int k = 0; k < NR; ++k) f[k][q] = row[k][jj];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int j = c + 64 * q + lane;
      if (c + 64 * q >= c1) break;
      xv[q] = j < c1 ? x(j) : (T)0;
#pragma unroll
      for (int k = 0; k < NR; ++k) acc[k] += f[k][q] * xv[q];
    }
  }
}

// forward, fronts of order <= 64: one wavefront, lane i owns row i; sixteen
// columns of the rows are loaded before the pivots that use them
template <class T>
__global__ void __launch_bounds__(64) k_mf_fwd_tiny(MfDev d, const int* list, const T* F, T* V, const double* b) {
  __shared__ T Vl[kMfTiny];
  const MfFront f = d.front[list[blockIdx.x]];
  const int ms = f.m, np = f.np, t = threadIdx.x;
  Vl[t] = t < np ? (T)b[d.bidx[f.idx + t]] : (T)0;
  mf_wave_fence();
  // the next child's values are loaded while this one's are added
  MfChild ch{};
  int e = -1;
  T v = (T)0;
  auto fetch = [&](int c) MF_INLINE {
    e = -1;
    if (c >= f.c1) return;
    ch = d.child[c];
    if (t < ch.nu) { e = d.emap[ch.em + t]; v = V[ch.vsrc + t]; }
  };
  fetch(f.c0);
  for (int c = f.c0; c < f.c1; ++c) {
    const int ec = e;
    const T vc = v;
    fetch(c + 1);
    if (ec >= 0) Vl[ec] += vc;
    mf_wave_fence();
  }
  v = Vl[t];
  const T* row = F + f.fo + (long long)min(t, ms - 1) * ms;
  for (int k0 = 0; k0 < np; k0 += 16) {
    T l[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) l[q] = row[min(k0 + q, np - 1)];
    __builtin_amdgcn_sched_barrier(0);
    // (coefficients of no effect set to zero off the chain of steps; those of the
    // lanes past the front too, whose values every other lane gets times zero)
#pragma unroll
    for (int q = 0; q < 16; ++q)
      if (!(k0 + q < np && t > k0 + q && t < ms)) l[q] = (T)0;
#pragma unroll
    for (int q = 0; q < 16; ++q) v -= l[q] * mf_bcast(v, k0 + q);
  }
  if (t < ms) V[f.vo + t] = v;
}

// backward, fronts of order <= 64 (roots first): x = U11^-1 (y - U12 x_below)
template <class T>
__global__ void __launch_bounds__(64) k_mf_bwd_tiny(MfDev d, const int* list, const T* F, const T* V, double* x,
                                                    int* nan_flag) {
  const MfFront f = d.front[list[blockIdx.x]];
  const int ms = f.m, np = f.np, t = threadIdx.x;
  const int g = t < ms ? d.xidx[f.idx + t] : 0;
  // lane t: y of pivot t, or the solved x of row t below the pivots
  T v = t < np ? V[f.vo + t] : t < ms ? (T)x[g] : (T)0;
  const T* row = F + f.fo + (long long)min(t, np - 1) * ms;
  // each lane's pivot reciprocal first (in parallel): the sweep multiplies
  const T rd = t < np ? (T)1 / row[t] : (T)1;
  for (int k1 = ms; k1 > 0; k1 -= 16) {
    T u[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) u[q] = row[max(k1 - 1 - q, 0)];
    __builtin_amdgcn_sched_barrier(0);
    // (coefficients of no effect set to zero off the chain of steps; a branch in
    // it would keep it from being unrolled)
#pragma unroll
    for (int q = 0; q < 16; ++q)
      if (!(t < k1 - 1 - q && t < np)) u[q] = (T)0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int k = max(k1 - 1 - q, 0);
      v -= u[q] * (mf_bcast(v, k) * mf_bcast(rd, k));
    }
  }
  v *= rd;
  if (t < np) {
    x[g] = (double)v;
    if (!isfinite((double)v)) *nan_flag = 1;
  }
}

// Larger fronts: one workgroup per front solves the pivot block (L11 or U11) by
// 64-row blocks with the vector in LDS.  While wavefront 0 solves a block's
// triangle (64 dependent steps), wavefronts 1 to 13 form the products of the
// next block's rows (five each) with everything solved before this block, load
// those rows' part inside it, and the next triangle; so between two triangles
// stands one 64 x 64 product from registers.  The rows outside the pivot block
// (L21 y, U12 x_below) are split over the GPU by the _rows kernels where they
// have more than kMfSplit elements, which one workgroup would need longer for
// than a launch takes (5 us).  What bounds a block is one CU's reads (64 rows of
// the solved columns at 27 bytes a cycle) above 128 solved columns, the triangle
// below (64 steps of 55 cycles).  512 x 512 grid, all levels, forward and
// backward: 0.59 ms; 0.78 with the sums as butterflies through LDS and whole
// 256-column chunks read, 1.08 with the triangle's steps rolled, 1.38 before the
// overlap and the split.
constexpr int kMfSolve = 1024;
constexpr int kMfSplit = 49152;
constexpr int kMfTri = 64 * 65;
constexpr int kMfNext = 5;                     // rows of the next block per wavefront

// the triangle at b0 into `tri` by wavefronts w, w + nw, ..., straight to LDS (a
// row is one or two loads of a dword per lane; no registers, so the products'
// loads follow at once).  mf_tri_wait: before the barrier that publishes it.
template <class T>
__device__ __forceinline__ void mf_load_tri(const T* Fs, long long ld, int b0, int bw, int w, int nw, int lane, T* tri) {
  constexpr int D = sizeof(T) / 4;
  for (int i = __builtin_amdgcn_readfirstlane(w); i < bw; i += nw) {
    const char* src = reinterpret_cast<const char*>(Fs + (b0 + i) * ld + b0);
#pragma unroll
    for (int h = 0; h < D; ++h) {
      const int q = 64 * h + lane;
      __builtin_amdgcn_global_load_lds(
          (const __attribute__((address_space(1))) void*)(src + (min(q / D, bw - 1) * D + q % D) * 4),
          (__attribute__((address_space(3))) void*)(reinterpret_cast<char*>(tri + i * 65) + 256 * h), 4, 0, 0);
    }
  }
}
__device__ __forceinline__ void mf_tri_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// A 64-row triangle by one wavefront, lane i holding row i's unknown: a row's
// coefficients come from LDS sixteen at a time, the next ones under way, those of
// no effect set to zero before, so that a step is a broadcast and a multiply-add
// (a loop the compiler keeps rolled waits for LDS in each: 64 rows 5 us more)
template <bool UPPER, class T>
__device__ __forceinline__ T mf_triangle(const T* tri, int bw, int lane, T v) {
  const T* row = tri + lane * 65;
  const T rd = UPPER && lane < bw ? (T)1 / row[lane] : (T)1;
  T l[2][16];
  auto fetch = [&](int c, T (&to)[16]) MF_INLINE {
#pragma unroll
    for (int q = 0; q < 16; ++q) to[q] = row[UPPER ? 63 - (16 * c + q) : 16 * c + q];
  };
  fetch(0, l[0]);
  mf_for<4>([&](auto cc) MF_INLINE {
    constexpr int c = cc;
    if constexpr (c < 3) fetch(c + 1, l[(c + 1) & 1]);
    // (opaque: else all 64 steps' masks are kept over the calls, in spilled registers)
    int ln = lane < bw ? lane : UPPER ? 64 : -1, w = bw;
    asm volatile("" : "+v"(ln), "+s"(w));
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int j = UPPER ? 63 - (16 * c + q) : 16 * c + q;
      if (!(UPPER ? ln < j && j < w : ln > j)) l[c & 1][q] = (T)0;
    }
    mf_for<16>([&](auto qc) MF_INLINE {
      constexpr int q = qc, j = UPPER ? 63 - (16 * c + q) : 16 * c + q;
      v -= l[c & 1][q] * (UPPER ? mf_bcast(v, j) * mf_bcast(rd, j) : mf_bcast(v, j));
    });
    __builtin_amdgcn_sched_barrier(0);
  });
  return UPPER ? v * rd : v;
}

template <class T, bool LDSV>
__global__ void __launch_bounds__(kMfSolve) k_mf_fwd_big(MfDev d, const int2* list, const T* F, T* V, const double* b) {
  extern __shared__ unsigned char mf_sm[];
  T* tri = reinterpret_cast<T*>(mf_sm);
  const int2 en = list[blockIdx.x];             // front, rows below the pivots left to k_mf_fwd_rows
  const MfFront f = d.front[en.x];
  T* x = LDSV ? tri + 2 * kMfTri : V + f.vo;    // the front's vector
  const int ms = f.m, np = f.np;
  const long long ld = ms;
  const T* Fs = F + f.fo;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  mf_load_tri(Fs, ld, 0, min(64, np), wave, kMfSolve / 64, lane, tri);
  for (int i = t; i < ms; i += kMfSolve) x[i] = i < np ? (T)b[d.bidx[f.idx + i]] : (T)0;
  mf_tri_wait();
  __syncthreads();
  for (int c = f.c0; c < f.c1; ++c) {
    const MfChild ch = d.child[c];
    for (int a = t; a < ch.nu; a += kMfSolve) x[d.emap[ch.em + a]] += V[ch.vsrc + a];
    __syncthreads();
  }
  if (en.y && LDSV)
    for (int i = np + t; i < ms; i += kMfSolve) V[f.vo + i] = x[i];
  const int nb = (np + 63) / 64;
  for (int k = 0; k < nb; ++k) {
    const int b0 = 64 * k, r = b0 + 64 + kMfNext * (wave - 1);
    const bool mine = wave > 0 && kMfNext * (wave - 1) < 64 && r < np;
    const int nr = min(kMfNext, min(np, b0 + 128) - r);
    T acc[kMfNext], pre[kMfNext];
    if (wave == 0) {
      const int bw = min(64, np - b0);
      const T v = mf_triangle<false>(tri + (k & 1) * kMfTri, bw, lane, lane < bw ? x[b0 + lane] : (T)0);
      if (lane < bw) x[b0 + lane] = v;
    } else {
      if (k + 1 < nb)
        mf_load_tri(Fs, ld, b0 + 64, min(64, np - b0 - 64), wave - 1, kMfSolve / 64 - 1, lane, tri + ((k + 1) & 1) * kMfTri);
      if (mine) {
#pragma unroll
        for (int i = 0; i < kMfNext; ++i) pre[i] = Fs[(r + min(i, nr - 1)) * ld + b0 + lane];
        mf_rows_part<kMfNext>(Fs, ld, r, nr, 0, b0, lane, [&](int j) MF_INLINE { return x[j]; }, acc);
      }
      mf_tri_wait();
    }
    __syncthreads();
    if (mine) {
      const T y = x[b0 + lane];
#pragma unroll
      for (int i = 0; i < kMfNext; ++i) acc[i] += pre[i] * y;
      mf_sub_sums<kMfNext>(x, r, nr, lane, acc);
    }
    __syncthreads();
  }
  if (!en.y)
    for (int r = np + 4 * wave; r < ms; r += 4 * (kMfSolve / 64)) {
      const int nr = min(4, ms - r);
      T acc[4];
      mf_rows_part<4>(Fs, ld, r, nr, 0, np, lane, [&](int j) MF_INLINE { return x[j]; }, acc);
      mf_sub_sums<4>(x, r, nr, lane, acc);
    }
  if (!LDSV) return;
  __syncthreads();
  for (int i = t; i < (en.y ? np : ms); i += kMfSolve) V[f.vo + i] = x[i];
}

// rows below the pivots of a split front, 16 per workgroup (entries {front, row})
template <class T>
__global__ void __launch_bounds__(256) k_mf_fwd_rows(MfDev d, const int2* ent, const T* F, T* V) {
  const int2 en = ent[blockIdx.x];
  const MfFront f = d.front[en.x];
  const int lane = threadIdx.x & 63, r = en.y + 4 * (threadIdx.x >> 6), nr = min(4, f.m - r);
  if (nr <= 0) return;
  T* v = V + f.vo;
  T acc[4];
  mf_rows_part<4>(F + f.fo, f.m, r, nr, 0, f.np, lane, [&](int j) MF_INLINE { return v[j]; }, acc);
  mf_sub_sums<4>(v, r, nr, lane, acc);
}

// pivot rows of a split front minus U12 x_below, 16 per workgroup
template <class T>
__global__ void __launch_bounds__(256) k_mf_bwd_rows(MfDev d, const int2* ent, const T* F, T* V, const double* x) {
  const int2 en = ent[blockIdx.x];
  const MfFront f = d.front[en.x];
  const int lane = threadIdx.x & 63, r = en.y + 4 * (threadIdx.x >> 6), nr = min(4, f.np - r);
  if (nr <= 0) return;
  const int* ix = d.xidx + f.idx;
  T acc[4];
  mf_rows_part<4>(F + f.fo, f.m, r, nr, f.np, f.m, lane, [&](int j) MF_INLINE { return (T)x[ix[j]]; }, acc);
  mf_sub_sums<4>(V + f.vo, r, nr, lane, acc);
}

template <class T, bool LDSV>
__global__ void __launch_bounds__(kMfSolve) k_mf_bwd_big(MfDev d, const int2* list, const T* F, T* V, double* xg,
                                                        int* nan_flag) {
  extern __shared__ unsigned char mf_sm[];
  T* tri = reinterpret_cast<T*>(mf_sm);
  const int2 en = list[blockIdx.x];             // front, U12 x_below already subtracted by k_mf_bwd_rows
  const MfFront f = d.front[en.x];
  T* x = LDSV ? tri + 2 * kMfTri : V + f.vo;
  const int ms = f.m, np = f.np;
  const long long ld = ms;
  const T* Fs = F + f.fo;
  const int* ix = d.xidx + f.idx;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int nb = (np + 63) / 64;
  mf_load_tri(Fs, ld, 64 * (nb - 1), np - 64 * (nb - 1), wave, kMfSolve / 64, lane, tri + ((nb - 1) & 1) * kMfTri);
  for (int i = t; i < (en.y ? np : ms); i += kMfSolve)
    if (i >= np) x[i] = (T)xg[ix[i]];
    else if (LDSV) x[i] = V[f.vo + i];
  mf_tri_wait();
  __syncthreads();
  if (!en.y && ms > np) {
    for (int r = 4 * wave; r < np; r += 4 * (kMfSolve / 64)) {
      const int nr = min(4, np - r);
      T acc[4];
      mf_rows_part<4>(Fs, ld, r, nr, np, ms, lane, [&](int j) MF_INLINE { return x[j]; }, acc);
      mf_sub_sums<4>(x, r, nr, lane, acc);
    }
    __syncthreads();
  }
  for (int k = nb - 1; k >= 0; --k) {
    const int b0 = 64 * k, bw = min(64, np - b0);
    const int i0 = kMfNext * (wave - 1), r = b0 - 64 + i0;
    const bool mine = wave > 0 && i0 < 64 && k > 0;
    const int nr = min(kMfNext, 64 - i0);
    T acc[kMfNext], pre[kMfNext];
    if (wave == 0) {
      const T v = mf_triangle<true>(tri + (k & 1) * kMfTri, bw, lane, lane < bw ? x[b0 + lane] : (T)0);
      if (lane < bw) x[b0 + lane] = v;
    } else {
      if (k > 0)
        mf_load_tri(Fs, ld, b0 - 64, 64, wave - 1, kMfSolve / 64 - 1, lane, tri + ((k - 1) & 1) * kMfTri);
      if (mine) {
#pragma unroll
        for (int i = 0; i < kMfNext; ++i) pre[i] = Fs[(r + min(i, nr - 1)) * ld + b0 + min(lane, bw - 1)];
        mf_rows_part<kMfNext>(Fs, ld, r, nr, b0 + bw, np, lane, [&](int j) MF_INLINE { return x[j]; }, acc);
      }
      mf_tri_wait();
    }
    __syncthreads();
    if (mine) {
      const T y = lane < bw ? x[b0 + lane] : (T)0;
#pragma unroll
      for (int i = 0; i < kMfNext; ++i) acc[i] += pre[i] * y;
      mf_sub_sums<kMfNext>(x, r, nr, lane, acc);
    }
    __syncthreads();
  }
  bool bad = false;
  for (int i = t; i < np; i += kMfSolve) {
    const double v = (double)x[i];
    xg[ix[i]] = v;
    bad |= !isfinite(v);
  }
  if (bad) *nan_flag = 1;
}

__global__ void k_mf_flag_init(int* bad) {
  bad[0] = 0x7fffffff;
  bad[1] = 0;
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
  int* fail = nullptr;            // pinned: raised by a factorisation whose pivots fail
  ~Impl() {
    if (fail) (void)hipHostFree(fail);
    for (auto& g : graphs)
      if (g.exec) (void)hipGraphExecDestroy(g.exec);
  }
  DevVec<int> emap, bidx, xidx, bad, arow, acol, aslot;
  DevVec<MfFront> front;
  DevVec<MfChild> child;
  DevVec<double> F64, V64;
  DevVec<float> F32, V32;
  DevVec<int> tiny_list;
  DevVec<int2> big_list;          // larger fronts {front, 1: rows outside the pivot block split over the GPU}
  DevVec<int2> frow, brow;        // entries of those rows {front, first row}
  DevVec<int4> aent;              // assembly entries of the larger fronts, two each
  DevVec<MfPart> parts;           // per entry: the children with rows in its range
  DevVec<MfStep> sent;            // entries of the panel steps
  DevVec<double> dbuf;            // diagonal-block factors, two 32 x 32 slots per larger front of a level
  std::vector<int> tiny_off, tiny_half, big_off;   // fronts up to order 32 at [tiny_off, tiny_half), up to 64 from there
  int big_maxm = 0;
  std::vector<int> frow_off, brow_off;   // per level
  std::vector<int> aoff;          // per level: offset into aent
  struct Step { int p0, off, cnt; };
  std::vector<std::vector<Step>> steps;   // per level: its panel steps
  MfDev dev() const {
    MfDev d;
    d.emap = emap.p; d.bidx = bidx.p; d.xidx = xidx.p;
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
      if (e > P.eptr[t] && P.emap[e] <= P.emap[e - 1]) return XG_E_SETUP;   // the parts below are bisected from it
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
  MFCHK(I.emap.up(P.emap, st));
  std::vector<int> bi(P.idx.size()), xi(P.idx.size());
  for (size_t q = 0; q < P.idx.size(); ++q) { bi[q] = s.perm_row[P.idx[q]]; xi[q] = s.perm_col[P.idx[q]]; }
  MFCHK(I.bidx.up(bi, st)); MFCHK(I.xidx.up(xi, st));
  MFCHK(I.bad.alloc(2));
  if (!I.fail) MFCHK(hipHostMalloc((void**)&I.fail, sizeof(int), hipHostMallocDefault));
  hipLaunchKernelGGL(k_mf_flag_init, dim3(1), dim3(1), 0, st, I.bad.p);
  MFCHK(I.F64.alloc(P.fo[P.ns] + 1)); MFCHK(I.V64.alloc(P.vo[P.ns]));
  if (want_fp32) { MFCHK(I.F32.alloc(P.fo[P.ns] + 1)); MFCHK(I.V32.alloc(P.vo[P.ns])); }
  // per level: tiny fronts (one launch), larger fronts (blocked panels, all
  // fronts of the level in each panel launch)
  const int nl = (int)P.lvl_ptr.size() - 1;
  std::vector<int> tl, bl;
  std::vector<int2> bl2, fre, bre;
  I.frow_off.assign(nl + 1, 0);
  I.brow_off.assign(nl + 1, 0);
  std::vector<MfStep> se;
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
    I.frow_off[l] = (int)fre.size();
    I.brow_off[l] = (int)bre.size();
    for (int q = I.big_off[l]; q < (int)bl.size(); ++q) {
      const int t = bl[q], m = P.m[t], np = P.sfirst[t + 1] - P.sfirst[t];
      const bool split = (long long)np * (m - np) > kMfSplit;
      bl2.push_back(make_int2(t, split));
      for (int r = np; split && r < m; r += 16) fre.push_back(make_int2(t, r));
      for (int r = 0; split && r < np; r += 16) bre.push_back(make_int2(t, r));
    }
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
          auto add = [&](int y, int z) { se.push_back(MfStep{y, z, slot, P.m[t], np, P.sfirst[t], P.fo[t]}); };
          if (pass == 0) {
            if (S.p0 < np)
              for (int i = 0; i < std::max(1, nrb); ++i) add(i, -1);
            else if (rest == 0) add(0, -2);
          } else if (j > 0) {
            // after the last panel tile (0, 0) copies the diagonal
            for (int ti = 0; ti * kMfTileRows < rest; ++ti)
              for (int tj = 0; tj < nrb; ++tj) add(ti, tj);
          }
        }
      S.cnt = (int)se.size() - S.off;
      I.steps[l].push_back(S);
    }
  }
  I.tiny_off[nl] = (int)tl.size();
  I.big_off[nl] = (int)bl.size();
  MFCHK(I.tiny_list.up(tl, st));
  I.frow_off[nl] = (int)fre.size();
  I.brow_off[nl] = (int)bre.size();
  MFCHK(I.big_list.up(bl2, st));
  MFCHK(I.frow.up(fre, st));
  MFCHK(I.brow.up(bre, st));
  MFCHK(I.sent.up(se, st));
  MFCHK(I.dbuf.alloc((size_t)max_slots * 2 * kMfPanel * kMfPanel));
  // assembly of the larger fronts, ranges of rows and columns (the tiny fronts
  // assemble themselves inside their factor kernel)
  std::vector<int4> ae;
  std::vector<MfPart> parts;
  I.aoff.assign(nl + 1, 0);
  for (int l = 0; l < nl; ++l) {
    I.aoff[l] = (int)ae.size() / 2;
    for (int b = I.big_off[l]; b < I.big_off[l + 1]; ++b) {
      const int t = bl[b], m = P.m[t];
      const int w = std::min(m, kMfAsm / 4), rows = std::min(kMfAsmRows, kMfAsm / w);
      for (int r0 = 0; r0 < m; r0 += rows) {
        const int off = (int)parts.size();
        for (int c = P.cptr[t]; c < P.cptr[t + 1]; ++c) {
          const int ch = P.clist[c];
          const int* eb = P.emap.data() + P.eptr[ch];
          const int* ee = P.emap.data() + P.eptr[ch + 1];
          const int x = (int)(std::lower_bound(eb, ee, r0) - eb), y = (int)(std::lower_bound(eb, ee, r0 + rows) - eb);
          if (x < y) parts.push_back(MfPart{chv[c].src, chv[c].ld, chv[c].nu, chv[c].em, x, y, 0});
        }
        for (int j0 = 0; j0 < m; j0 += w) {
          ae.push_back(make_int4(t, r0, std::min(rows, m - r0), off));
          ae.push_back(make_int4(j0, std::min(w, m - j0), (int)parts.size() - off, 0));
        }
      }
    }
  }
  I.aoff[nl] = (int)ae.size() / 2;
  MFCHK(I.aent.up(ae, st));
  MFCHK(I.parts.up(parts, st));
  MFCHK(hipStreamSynchronize(st));
  return XG_OK;
}

double MfLu::flops() const { return impl_->P.flops; }
long long MfLu::front_elements() const { return impl_->P.fo.empty() ? 0 : impl_->P.fo[impl_->P.ns]; }
int MfLu::levels() const { return (int)impl_->P.lvl_ptr.size() - 1; }
int MfLu::supernodes() const { return impl_->P.ns; }

// the launches of one refactor (no host work: the sequence is captured)
template <class T>
static int mf_factor_enqueue(MfLu::Impl& I, const double* vals_dev, int nnz, T* F) {
  const MfPlan& P = I.P;
  hipStream_t st = I.st;
  const MfDev d = I.dev();
  T* dbuf = reinterpret_cast<T*>(I.dbuf.p);
  const int nl = (int)P.lvl_ptr.size() - 1;
  for (int l = 0; l < nl; ++l) {
    const int na = I.aoff[l + 1] - I.aoff[l];
    if (na)
      hipLaunchKernelGGL(k_mf_assemble<T>, dim3(na), dim3(256), 0, st, d, I.aent.p + 2 * I.aoff[l], I.parts.p, vals_dev, F);
    const int n32 = I.tiny_half[l] - I.tiny_off[l], n64 = I.tiny_off[l + 1] - I.tiny_half[l];
    if (n32)
      hipLaunchKernelGGL((k_mf_factor_tiny<T, kMfTiny / 2>), dim3(n32), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l],
                         vals_dev, F, I.bad.p, I.fail);
    if (n64)
      hipLaunchKernelGGL((k_mf_factor_tiny<T, kMfTiny>), dim3(n64), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_half[l],
                         vals_dev, F, I.bad.p, I.fail);
    for (const auto& S : I.steps[l])
      hipLaunchKernelGGL(k_mf_step<T>, dim3(S.cnt), dim3(kMfStep), 0, st, I.sent.p + S.off, S.p0, F, dbuf,
                         (S.p0 / kMfPanel) & 1, I.bad.p, I.fail);
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
static int mf_factor_t(MfLu::Impl& I, const double* vals_dev, int nnz, T* F) {
  const void* key[8] = {(const void*)1, vals_dev, F, (const void*)(long long)nnz, nullptr, nullptr, nullptr, nullptr};
  *I.fail = 0;
  return mf_replay(I, key, 8, [&] { return mf_factor_enqueue<T>(I, vals_dev, nnz, F); });
}

template <class T>
static int mf_solve_enqueue(MfLu::Impl& I, const T* F, T* V, const double* b_dev, double* x_dev, int* nan_flag) {
  const MfPlan& P = I.P;
  hipStream_t st = I.st;
  const MfDev d = I.dev();
  // the larger fronts keep their vector in LDS when it fits beside the two
  // triangles, else in their slice of V
  const size_t tri = 2 * kMfTri * sizeof(T);
  const bool ldsv = tri + (size_t)I.big_maxm * sizeof(T) <= 150 * 1024;
  const size_t lds = tri + (ldsv ? (size_t)I.big_maxm * sizeof(T) : 0);
  const int nl = (int)P.lvl_ptr.size() - 1;
  for (int l = 0; l < nl; ++l) {
    const int nt = I.tiny_off[l + 1] - I.tiny_off[l], nb = I.big_off[l + 1] - I.big_off[l];
    const int nr = I.frow_off[l + 1] - I.frow_off[l];
    if (nt) hipLaunchKernelGGL(k_mf_fwd_tiny<T>, dim3(nt), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l], F, V, b_dev);
    if (nb && ldsv)
      hipLaunchKernelGGL((k_mf_fwd_big<T, true>), dim3(nb), dim3(kMfSolve), lds, st, d, I.big_list.p + I.big_off[l], F, V,
                         b_dev);
    else if (nb)
      hipLaunchKernelGGL((k_mf_fwd_big<T, false>), dim3(nb), dim3(kMfSolve), lds, st, d, I.big_list.p + I.big_off[l], F,
                         V, b_dev);
    if (nr) hipLaunchKernelGGL(k_mf_fwd_rows<T>, dim3(nr), dim3(256), 0, st, d, I.frow.p + I.frow_off[l], F, V);
  }
  for (int l = nl - 1; l >= 0; --l) {
    const int nt = I.tiny_off[l + 1] - I.tiny_off[l], nb = I.big_off[l + 1] - I.big_off[l];
    const int nr = I.brow_off[l + 1] - I.brow_off[l];
    if (nr)
      hipLaunchKernelGGL(k_mf_bwd_rows<T>, dim3(nr), dim3(256), 0, st, d, I.brow.p + I.brow_off[l], F, V,
                         (const double*)x_dev);
    if (nb && ldsv)
      hipLaunchKernelGGL((k_mf_bwd_big<T, true>), dim3(nb), dim3(kMfSolve), lds, st, d, I.big_list.p + I.big_off[l], F, V,
                         x_dev, nan_flag);
    else if (nb)
      hipLaunchKernelGGL((k_mf_bwd_big<T, false>), dim3(nb), dim3(kMfSolve), lds, st, d, I.big_list.p + I.big_off[l], F,
                         V, x_dev, nan_flag);
    if (nt)
      hipLaunchKernelGGL(k_mf_bwd_tiny<T>, dim3(nt), dim3(64), 0, st, d, I.tiny_list.p + I.tiny_off[l], F, (const T*)V,
                         x_dev, nan_flag);
  }
  MFCHK(hipGetLastError());
  return XG_OK;
}

template <class T>
static int mf_solve_t(MfLu::Impl& I, const T* F, T* V, const double* b_dev, double* x_dev, int* nan_flag) {
  const void* key[8] = {(const void*)2, F, V, b_dev, x_dev, nan_flag, nullptr, nullptr};
  return mf_replay(I, key, 8, [&] { return mf_solve_enqueue<T>(I, F, V, b_dev, x_dev, nan_flag); });
}

int MfLu::factor_begin(const double* vals_dev, int nnz, bool fp32) {
  Impl& I = *impl_;
  if (fp32) {
    if (!I.F32.p) return XG_E_ARG;
    return mf_factor_t<float>(I, vals_dev, nnz, I.F32.p);
  }
  return mf_factor_t<double>(I, vals_dev, nnz, I.F64.p);
}

// The kernels raise the pinned flag and leave the details on the device, where
// they are looked at (and cleared) only then.
int MfLu::factor_end(int* bad, int* hard) {
  Impl& I = *impl_;
  *bad = *hard = 0;
  if (!*I.fail) return XG_OK;
  int res[2];
  MFCHK(hipMemcpyAsync(res, I.bad.p, sizeof(res), hipMemcpyDeviceToHost, I.st));
  hipLaunchKernelGGL(k_mf_flag_init, dim3(1), dim3(1), 0, I.st, I.bad.p);
  MFCHK(hipStreamSynchronize(I.st));
  *bad = res[0] == 0x7fffffff ? 0 : res[0];
  *hard = res[1];
  return XG_OK;
}

int MfLu::factor(const double* vals_dev, int nnz, bool fp32, int* bad, int* hard) {
  const int rc = factor_begin(vals_dev, nnz, fp32);
  if (rc != XG_OK) return rc;
  MFCHK(hipStreamSynchronize(impl_->st));
  return factor_end(bad, hard);
}

int MfLu::solve(const double* b_dev, double* x_dev, bool fp32, int* nan_flag) {
  Impl& I = *impl_;
  if (fp32) {
    if (!I.F32.p) return XG_E_ARG;
    return mf_solve_t<float>(I, I.F32.p, I.V32.p, b_dev, x_dev, nan_flag);
  }
  return mf_solve_t<double>(I, I.F64.p, I.V64.p, b_dev, x_dev, nan_flag);
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
  // launched one by one: a captured graph would be allocated with the first call
  // (131 x 97 mesh 211 us, 206 replayed; gate array of 298 55 us, 58 replayed)
  MFCHK(hipMemcpyAsync(bp, b_dev, sizeof(double) * P.n, hipMemcpyDeviceToDevice, I.st));
  const int rc = mf_solve_enqueue<double>(I, I.F64.p, V, bp, y, nan_flag);
  if (rc != XG_OK) return rc;
  MFCHK(hipMemcpyAsync(x_dev, y, sizeof(double) * P.n, hipMemcpyDeviceToDevice, I.st));
  return XG_OK;
}

}  // namespace xg
