// Internal kernel launchers shared by the translation units of libhps_mi355x.
#pragma once

#include "hps_common.h"

namespace hps {

// D[b] = alpha * op(A[b]) @ B[b] + beta * C[b]   (row-major, per batch element)
// op(A) = A (M x K, lda) or, with transA, A^H where A is stored K x M (lda);
// B: K x N (ldb), C/D: M x N (ldc/ldd).  s* are batch strides (0 broadcasts).
// C may be null when beta == 0.  C and D may alias.
template <typename T>
struct GemmArgs {
  int M = 0, N = 0, K = 0;
  double alpha = 1.0, beta = 0.0;
  const T* A = nullptr;
  long lda = 0, sA = 0;
  const T* B = nullptr;
  long ldb = 0, sB = 0;
  const T* C = nullptr;
  long ldc = 0, sC = 0;
  T* D = nullptr;
  long ldd = 0, sD = 0;
  int batch = 1;
  // two-level batches: element b is matrix b / nin, part b % nin of it, and a
  // part's operands lie s*2 apart inside the matrix
  int nin = 1;
  long sA2 = 0, sB2 = 0, sC2 = 0, sD2 = 0;
  int transA = 0;
  // sum2 (real types, not transA): sum over 32 k at a time and add the sums up,
  // for products with much cancellation -- the rounding of a long chain grows
  // with its length.  A hint: shapes without that kernel sum in one chain.
  int sum2 = 0;
  // triA: A is a packed 32 x 32 diagonal-block inverse used as its unit-lower
  // part (1) or its upper part (2); needs K <= 32.  D may then alias B.
  int triA = 0;
};

__host__ __device__ inline long batch_offset(int b, int nin, long s, long s2) {
  return nin == 1 ? (long)b * s : (long)(b / nin) * s + (long)(b % nin) * s2;
}

template <typename T>
hipError_t gemm(const GemmArgs<T>& a, hipStream_t s);

// The products of row blocks of one A with row blocks of one B: blk holds
// n_blk host-side rectangles (r0, nr, k0, nk); block u is
// D[r0 : r0 + nr] = alpha A[r0 : r0 + nr, k0 : k0 + nk] B[k0 : k0 + nk] + beta C[r0 : r0 + nr]
// with a's N, leading dimensions, batch strides, alpha and beta (a.M and
// a.K are not read).  The blocks must write disjoint rows of D.
template <typename T>
hipError_t gemm_grouped(const GemmArgs<T>& a, int n_blk, const int* blk, hipStream_t s);

// In-place batched LU with partial pivoting of the n x n block of each A[b]
// (row stride lda, batch stride sA): P A = L U.  perm[b*n + i] is the row of
// A that became row i of P A.  dinv[b] (dinv_elems(n) values) receives the
// packed inverses of the 32 x 32 diagonal blocks.  scratch holds
// getrf_scratch_bytes(n, batch) bytes.  info[b] = 0, or j+1 for the first
// column j whose pivot candidates are all exactly zero.
size_t getrf_scratch_bytes(int n, int batch);
size_t dinv_elems(int n);
// natural: register-sized matrices without row exchanges, checked in the kernel:
// a matrix with a multiplier above 64 (or not finite) gets info = -1 and must be
// refactored with pivoting.
template <typename T>
hipError_t getrf_ws(int n, T* A, long lda, long sA, int* perm, T* dinv, int* scratch, int* info, int batch,
                    hipStream_t s, bool natural = false);

// X = A^{-1} R from getrf_ws's factors.  R (n x nrhs, row stride ldr, batch
// stride sR) is read only; X must not alias R.
template <typename T>
hipError_t getrs_perm(int n, int nrhs, const T* LU, long lda, long sA, const int* perm, const T* dinv, const T* R,
                      long ldr, long sR, T* X, long ldx, long sX, int batch, hipStream_t s);

// X = A^{-1} P^T X in place, X already gathered by the permutation
// (X[i] = R[perm[i]]): the triangular solves of getrs_perm's blocked path.
template <typename T>
hipError_t getrs_inplace(int n, int nrhs, const T* LU, long lda, long sA, const T* dinv, T* X, long ldx, long sX,
                         int batch, hipStream_t s);

// smallest matrix that pivoted factorisations cut into column blocks of 512
constexpr int LU_WIDE_MIN = 3072;

// Few-column solves (at most 16 columns) of matrices too large for one
// workgroup, in fewer than 128 matrices: the refinement's up passes through
// the top merge levels' low-precision factors.  form_fewinv writes the
// inverses of the FEWINV_NB x FEWINV_NB diagonal blocks of L (unit lower) and
// U of every matrix: inv holds batch * fewinv_elems(n) elements (all the L
// block inverses, then all the U ones), ws fewinv_workspace_elems(n, batch)
// elements.  getrs_perm_fewinv solves X = A^{-1} R with them (Y: n x nrhs
// scratch per matrix, row stride nrhs); R, X and Y must not alias.  Eligible:
// n > 256 and a multiple of 32.
constexpr int FEWINV_NB = 256;
inline bool fewinv_eligible(int n) { return n > 256 && n % 32 == 0; }
inline int fewinv_blocks(int n) { return (n + FEWINV_NB - 1) / FEWINV_NB; }
inline size_t fewinv_elems(int n) {
  return fewinv_eligible(n) ? 2 * (size_t)fewinv_blocks(n) * FEWINV_NB * FEWINV_NB : 0;
}
inline size_t fewinv_workspace_elems(int n, int batch) {
  return fewinv_eligible(n) ? (size_t)batch * fewinv_blocks(n) * (FEWINV_NB * FEWINV_NB + FEWINV_NB * 32) : 0;
}
template <typename T>
hipError_t form_fewinv(int n, const T* LU, long lda, long sA, const T* dinv, T* inv, T* ws, int batch, hipStream_t s);
template <typename T>
hipError_t getrs_perm_fewinv(int n, int nrhs, const T* LU, long lda, long sA, const int* perm, const T* inv,
                             const T* R, long ldr, long sR, T* X, long ldx, long sX, T* Y, int batch, hipStream_t s);

// ---------------------------------------------------------------------------
// Natural-order LU and many-column solves by blocks (lu_blocks.h)
// ---------------------------------------------------------------------------
// The elimination's block structure: stages of `cnt` equal diagonal blocks
// (groups) that do not couple to one another.  Group i of a stage couples,
// among the later unknowns, to the runs (s[j], ns[j]) only, and its right-hand
// sides are nonzero in nc columns from c0 + i c_step only.
constexpr int LUB_NB = 128;       // block of the elimination inside a group
constexpr int LUB_MAX_CNT = 4;    // groups per stage
constexpr int LUB_MAX_STAGES = 3;
constexpr int LUB_MAX_RUNS = 4;
struct LuGroup {
  int nrun = 0;
  int s[LUB_MAX_RUNS] = {}, ns[LUB_MAX_RUNS] = {};
};
struct LuStage {
  int cnt = 1, size = 0, r0 = 0;  // groups, unknowns of a group, first unknown of the stage
  int c0 = 0, nc = 0, c_step = 0;
  LuGroup g[LUB_MAX_CNT];
};
// Largest multiplier that an elimination without row exchanges accepts, and the
// one for DtN matrices by blocks.  The matrices of definite problems stay below 8
// (anisotropy 100, coefficient jumps of 1000, strong advection).  DtN Helmholtz
// problems past the first eigenvalues reach any size, and the blocks' explicit
// 64- and 128-wide inverses amplify growth: with multipliers up to 16 the
// solution's error is up to 3.3 times that of pivoting everywhere, with 17 to 64
// mostly below 5, but up to 2300 times (120 problems, p = 6 .. 16; no norm of the
// inverses tells the two apart).  ItI merges reach 15 to 58 with eta below k / 20
// and lose nothing (ratio 0.94 to 1.01, 40 problems).
constexpr double LU_NOPIV_BOUND = 64.0;
constexpr double LU_DTN_BOUND = 16.0;
struct LuPlan {
  int n = 0, nstage = 0;
  double bound = LU_NOPIV_BOUND;  // largest multiplier
  int nbmax = LUB_NB;  // widest block
  LuStage st[LUB_MAX_STAGES];
};
// One dense group of n unknowns.  Many matrices (LUB_MANY) take blocks of 64:
// their launches are full either way, and a block's inverse, half of it zero,
// costs operations and traffic in proportion to its width (the ItI leaf stage of
// 16384 leaves, p = 16: 32.7 ms, with blocks of 128 36.0 ms).  Few matrices keep
// 128: their chain of launches is half as long.
constexpr int LUB_MANY = 1024;
inline LuPlan lu_plan_dense(int n, int ncols, int batch) {
  LuPlan p;
  p.n = n;
  if (batch >= LUB_MANY) p.nbmax = 64;
  p.nstage = 1;
  p.st[0].size = n;
  p.st[0].nc = ncols;
  return p;
}
// 2D DtN merge, unknowns in the order of the interfaces a|b, c|d, b|c, d|a (m
// each), columns by child: the first two do not couple
inline LuPlan lu_plan_quad(int m) {
  LuPlan p;
  p.n = 4 * m;
  p.nstage = 2;
  p.st[0].cnt = 2;
  p.st[0].size = m;
  p.st[0].nc = p.st[0].c_step = 4 * m;
  for (int i = 0; i < 2; ++i) {
    p.st[0].g[i].nrun = 1;
    p.st[0].g[i].s[0] = p.st[0].g[i].ns[0] = 2 * m;
  }
  p.st[1].size = p.st[1].r0 = 2 * m;
  p.st[1].nc = 8 * m;
  return p;
}
// 3D DtN merge (children a .. h, columns by child): the x-interfaces a|b, d|c of
// the upper slab and e|f, h|g of the lower one (group 2 z + y), the y-interfaces
// of each slab (two groups), the z-interfaces at y- and at y+
inline LuPlan lu_plan_oct(int m) {
  LuPlan p;
  p.n = 12 * m;
  p.nstage = 3;
  p.st[0].cnt = 4;
  p.st[0].size = m;
  p.st[0].nc = p.st[0].c_step = 6 * m;
  for (int i = 0; i < 4; ++i) {
    LuGroup& g = p.st[0].g[i];
    g.nrun = 2;
    g.s[0] = 4 * m + (i / 2) * 2 * m;
    g.s[1] = 8 * m + (i % 2) * 2 * m;
    g.ns[0] = g.ns[1] = 2 * m;
  }
  p.st[1].cnt = 2;
  p.st[1].size = 2 * m;
  p.st[1].r0 = 4 * m;
  p.st[1].nc = p.st[1].c_step = 12 * m;
  for (int i = 0; i < 2; ++i) {
    p.st[1].g[i].nrun = 1;
    p.st[1].g[i].s[0] = 8 * m;
    p.st[1].g[i].ns[0] = 4 * m;
  }
  p.st[2].size = 4 * m;
  p.st[2].r0 = 8 * m;
  p.st[2].nc = 24 * m;
  return p;
}
// A group is cut into blocks of nbmax from its end, so that the trailing
// products of every step are whole tiles; the first block takes the remainder
// (with 64-wide blocks one of up to 16 joins the first whole block: 196 unknowns
// are 68 + 64 + 64, where 64 + 64 + 64 + 4 left 132 and 68 unknowns to nine and
// four 64 x 64 tiles).  A level of 1024 float64 merges of 68, 72, 80 unknowns,
// joined / in a block of its own: 920 / 990, 960 / 1026, 1090 / 1145 us; 132 and
// 144 unknowns 3062 / 3174, 3344 / 3425.  From 84 to 96 unknowns (20 to 32 over)
// joining would still gain 3 to 4 %.
inline int lub_first(const LuPlan& p, int size) {
  if (size <= p.nbmax) return size;
  const int r = size % p.nbmax;
  return r == 0 ? p.nbmax : (p.nbmax < LUB_NB && r <= 16 ? p.nbmax + r : r);
}
inline int lub_blocks(const LuPlan& p, int size) { return 1 + (size - lub_first(p, size)) / p.nbmax; }
// row stride (and rows) of a stored block inverse
inline int lub_ld(const LuPlan& p, int size) {
  const int f = lub_first(p, size), m = size > p.nbmax && f < p.nbmax ? p.nbmax : f;
  return (m + 31) / 32 * 32;
}
// elements of the block inverses that a solve needs and of the factorisation's
// scratch, bytes of its integer scratch
inline size_t lub_inv_elems(const LuPlan& p, int batch) {
  size_t t = 0;
  for (int i = 0; i < p.nstage; ++i)
    t += (size_t)p.st[i].cnt * lub_blocks(p, p.st[i].size) * 2 * lub_ld(p, p.st[i].size) * lub_ld(p, p.st[i].size);
  return t * batch;
}
inline size_t lub_tmp_elems(const LuPlan& p, int batch) {
  size_t m = 0;
  for (int i = 0; i < p.nstage; ++i) {
    const LuStage& s = p.st[i];
    const size_t t = (size_t)s.cnt * lub_ld(p, s.size) * ((size_t)(s.size + p.n - s.r0 - s.cnt * s.size) + 32);
    m = m > t ? m : t;
  }
  return m * batch;
}
size_t lub_scratch_bytes(const LuPlan& p, int batch);

// A = L U in natural order, in place (batch matrices, row stride lda, batch
// stride sA); perm becomes the identity, dinv as getrf_ws's, inv the inverses
// of every block's L and U (lub_inv_elems), tmp lub_tmp_elems elements.
// info[b] = -1 where a multiplier exceeds the plan's bound or a pivot is zero, not finite or
// without a normal reciprocal (the matrix then needs pivoting), else 0.
template <typename T>
hipError_t lu_blocks_factor(const LuPlan& plan, T* A, long lda, long sA, int* perm, T* dinv, T* inv, T* tmp,
                            int* scratch, int* info, int batch, hipStream_t s);
// B = A^{-1} B; X is scratch of B's shape.  cols: the right-hand sides have the
// plan's column structure (otherwise they are dense).
template <typename T>
hipError_t lu_blocks_solve(const LuPlan& plan, const T* A, long lda, long sA, const T* inv, T* B, long ldb, long sB,
                           T* X, long ldx, long sX, int nrhs, bool cols, int batch, hipStream_t s);

// X = A^{-H} R from getrf_ws's factors (A^H = U^H L^H P).  W is n x nrhs
// scratch per batch element (row stride nrhs); X, W and R must not alias.
template <typename T>
hipError_t getrs_conjt(int n, int nrhs, const T* LU, long lda, long sA, const int* perm, const T* dinv, const T* R,
                       long ldr, long sR, T* X, long ldx, long sX, T* W, int batch, hipStream_t s);

// dst[b][r][c] = alpha * src[b][r][c]; src == nullptr writes zeros; a batch
// stride of 0 on src broadcasts.
template <typename T>
hipError_t add2d(int rows, int cols, double alpha, const T* src, long lds, long ss, T* dst, long ldd, long sd,
                 int batch, hipStream_t s);

template <typename T>
hipError_t copy2d(int rows, int cols, double alpha, const T* src, long lds, long ss, T* dst, long ldd, long sd,
                  int batch, hipStream_t s);

}  // namespace hps
