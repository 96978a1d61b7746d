// Natural-order LU by blocks and the many-column solves with it (included by
// lu.hip).
//
// Without row exchanges a block column needs no tall panel: the diagonal block
// (at most 128 wide) is factored by itself, the inverses of its L and U are
// formed, and everything else is a product -- L21 = A21 inv(U11), U12 =
// inv(L11) A12, the trailing update -- at the matrix cores' rate.  The
// solves use the same inverses.  Tall panels of 32 columns instead updated the
// block column with K = 32 products, which are bound by reading and writing
// their C tile.
//
// A plan (LuPlan) adds the block zeros of nested dissection: the 3D merge's
// four x-interfaces do not couple, then the two y-slabs do not, so a stage's
// groups go through every launch together (two-level batches) and the zero
// blocks are left out: 3696 m^3 operations for LU and right-hand sides of a 3D
// merge with m unknowns an interface, 8064 m^3 densely.
//
// Measured when this came in, one build + solve, panels and dense solves before / this:
// 3D p = 10, L = 3 with 4 sources (12288 unknowns at the root) 287 / 173 ms, 2D
// elliptic p = 16, L = 6 with 16 sources 21.3 / 18.0 ms, 2D Helmholtz p = 16,
// L = 7 complex128 172 / 170 ms, complex64 113 / 115 ms (its solves had
// 512-wide block inverses already).  The first block takes a group's remainder
// and blocks of at most 64 are multiplied in place: elliptic case 16.6 / 15.9 ms,
// ItI leaves below (16384 of 196 + 60 unknowns) 35.4 / 32.7 ms.
#pragma once

namespace hps {

// Parts up to which the unpivoted panel kernel takes the diagonal blocks (its
// workgroups repeat the diagonal block, up to five of them a part), above it one
// workgroup a part with its rows in registers: the repeated work has to stay
// small beside the GPU's 256 CUs.  A level of merges with 112 unknowns each
// (float64 DtN; complex128 ItI), spread / one workgroup: 16 merges 246 / 318; 437
// / 528 us, 96 merges 339 / 404; 821 / 898, 256 merges 631 / 683; 1705 / 1728, 512
// merges 1129 / 1158; 3160 / 3088: the two meet between 256 and 512 parts, so
// levels of 97 to 256 give up 1 to 14 %.
constexpr int LUB_SPREAD_PARTS = 96;

// widest block whose products with its inverses run in place: the GEMM's tile
constexpr int LUB_INPLACE = 64;

// Inverses of L (unit lower, blockIdx.x < nq) and U of nb x nb diagonal
// blocks, nb <= 128: one workgroup per 32-column strip of one inverse, the strip
// in LDS.  Block row i of inv(L)'s strip s is -inv(L_ii) sum_{s <= q < i}
// L_iq X_q (U: from the diagonal upwards), every product 32 x 32 on the matrix
// cores, one 16 x 16 tile a wave.  db: the packed 32 x 32 inverses (part
// stride nq blocks).  Writes whole columns, zeros included; ldi x ldi storage,
// inv(U) after inv(L).
template <typename T, int NBMAX>
__global__ __launch_bounds__(256) void block_inverse_kernel(int nb, const T* A, long lda, long sA, int nin, long sA2,
                                                            const T* db, T* inv, int ldi, long sI, long sI2, int batch) {
  using R = typename real_of<T>::type;
  using M = Mfma<R>;
  using acc_t = typename M::acc_t;
  __shared__ T X[NBMAX][LU_NB + 1];
  __shared__ T W[LU_NB][LU_NB + 1];
  const int nq = (nb + LU_NB - 1) / LU_NB;
  const bool upper = (int)blockIdx.x >= nq;
  const int s = (int)blockIdx.x % nq;
  const int tid = threadIdx.x;
  const int wave = tid >> 6, li = tid & 15, lk = (tid & 63) >> 4;
  const int tr = 16 * (wave >> 1) + li, tc = 16 * (wave & 1) + li;
  for (int b = blockIdx.y; b < batch; b += gridDim.y) {
    const T* Ab = A + batch_offset(b, nin, sA, sA2);
    const T* d = db + (long)b * nq * LU_NB * LU_NB;
    T* out = inv + batch_offset(b, nin, sI, sI2) + (upper ? ldi * ldi : 0);
    // entry (r, c) of the triangular inverse of diagonal block i
    auto tri = [&](int i, int r, int c) {
      const T v = d[((long)i * LU_NB + r) * LU_NB + c];
      if (upper) return s_sel(c >= r, v, s_zero<T>());
      return s_sel(c < r, v, s_sel(c == r && i * LU_NB + r < nb, s_one<T>(), s_zero<T>()));
    };
    for (int idx = tid; idx < LU_NB * LU_NB; idx += 256) {
      const int r = idx / LU_NB, c = idx % LU_NB;
      X[s * LU_NB + r][c] = tri(s, r, c);
    }
    __syncthreads();
    // the pairs (i, q) of the strip in one sequence: the next pair's factor
    // entries (and, with a block row's first pair, its diagonal inverse) are
    // requested before the current pair's product
    const int steps = upper ? s : nq - 1 - s;
    auto load = [&](int i, int q, T (&a)[LU_NB / 4]) {
      const int row = i * LU_NB + tr;
#pragma unroll
      for (int k = 0; k < LU_NB / 4; ++k) {
        const int col = q * LU_NB + 4 * k + lk;
        const bool in = row < nb && col < nb;
        a[k] = Ab[in ? (long)row * lda + col : 0];
        a[k] = s_sel(in, a[k], s_zero<T>());
      }
    };
    T a[LU_NB / 4], an[LU_NB / 4], di[LU_NB / 4];
    if (steps > 0) load(upper ? s - 1 : s + 1, s, a);
    for (int t = 1; t <= steps; ++t) {
      const int i = upper ? s - t : s + t;
      const int q0 = upper ? i + 1 : s, q1 = upper ? s + 1 : i;
#pragma unroll
      for (int k = 0; k < LU_NB / 4; ++k) di[k] = tri(i, tr, 4 * k + lk);
      acc_t re = acc_t{0, 0, 0, 0}, im = acc_t{0, 0, 0, 0};
      for (int q = q0; q < q1; ++q) {
        const int i2 = upper ? i - 1 : i + 1;
        if (q + 1 < q1)
          load(i, q + 1, an);
        else if (t < steps)
          load(i2, upper ? i2 + 1 : s, an);
#pragma unroll
        for (int k = 0; k < LU_NB / 4; ++k) mma_step<T>(a[k], X[q * LU_NB + 4 * k + lk][tc], re, im);
#pragma unroll
        for (int k = 0; k < LU_NB / 4; ++k) a[k] = an[k];
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        W[16 * (wave >> 1) + M::out_row(lk, r)][tc] = make_val<T>(re[r], is_cplx<T>::value ? im[r] : R(0));
      __syncthreads();
      re = im = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < LU_NB / 4; ++k) mma_step<T>(di[k], W[4 * k + lk][tc], re, im);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        X[i * LU_NB + 16 * (wave >> 1) + M::out_row(lk, r)][tc] =
            s_neg(make_val<T>(re[r], is_cplx<T>::value ? im[r] : R(0)));
      __syncthreads();
    }
    const int r0 = upper ? 0 : s * LU_NB, r1 = upper ? (s + 1) * LU_NB : nb;
    for (int idx = tid; idx < nb * LU_NB; idx += 256) {
      const int r = idx / LU_NB, c = idx % LU_NB;
      if (s * LU_NB + c < nb) out[r * ldi + s * LU_NB + c] = r >= r0 && r < r1 ? X[r][c] : s_zero<T>();
    }
    __syncthreads();  // X is rewritten for the next part
  }
}

// Packed inverses of the 32 x 32 diagonal blocks of a factored matrix
// (absolute block positions, which the groups' own blocks need not share).
template <typename T>
__global__ __launch_bounds__(256) void dinv_from_factors_kernel(int n, const T* A, long lda, long sA, T* dinv,
                                                                int batch) {
  __shared__ T D[LU_NB][LU_NB + 1];
  const int k = blockIdx.x * LU_NB;
  const int nb = n - k < LU_NB ? n - k : LU_NB;
  for (int b = blockIdx.y; b < batch; b += gridDim.y) {
    const T* Akk = A + (long)b * sA + (long)k * lda + k;
    for (int idx = threadIdx.x; idx < LU_NB * LU_NB; idx += 256) {
      const int r = idx / LU_NB, c = idx % LU_NB;
      D[r][c] = r < nb && c < nb ? Akk[(long)r * lda + c] : s_zero<T>();
    }
    __syncthreads();
    invert_diag_block<T>(&D[0][0], LU_NB + 1, dinv + ((long)b * gridDim.x + blockIdx.x) * LU_NB * LU_NB, LU_NB, nb);
    __syncthreads();
  }
}

// perm = identity, info = 0, arrivals = 0
static __global__ __launch_bounds__(256) void lu_blocks_init_kernel(int n, int batch, int parts, int* perm, int* info,
                                                                    int* arrivals) {
  const long total = (long)n * batch;
  for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    perm[i] = (int)(i % n);
    if (i < batch) info[i] = 0;
    if (i < parts) arrivals[i] = 0;  // parts <= n batch: a group has at least one unknown
  }
}

// rows x cols of tmp (row stride ldt) back into the matrix; CHECK: the values
// are multipliers
template <typename T, bool CHECK>
__global__ __launch_bounds__(256) void panel_back_kernel(int rows, int cols, const T* tmp, long ldt, long sT, T* A,
                                                         long lda, long sA, int nin, long sA2,
                                                         typename real_of<T>::type bound, int* info, int batch) {
  const auto bound2 = bound * bound;
  const int total = rows * cols;
  for (int b = blockIdx.y; b < batch; b += gridDim.y) {
    const T* t = tmp + (long)b * sT;
    T* a = A + batch_offset(b, nin, sA, sA2);
    bool ok = true;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
      const int r = idx / cols, c = idx - r * cols;
      const T v = t[(long)r * ldt + c];
      a[(long)r * lda + c] = v;
      if (CHECK) ok = ok && s_mod2(v) <= bound2;
    }
    if (!ok) info[b / nin] = -1;
  }
}

// info of the matrices whose multipliers (rows x cols at A) pass the bound
template <typename T>
__global__ __launch_bounds__(256) void panel_check_kernel(int rows, int cols, const T* A, long lda, long sA, int nin,
                                                          long sA2, typename real_of<T>::type bound, int* info,
                                                          int batch) {
  const auto bound2 = bound * bound;
  const int total = rows * cols;
  for (int b = blockIdx.y; b < batch; b += gridDim.y) {
    const T* a = A + batch_offset(b, nin, sA, sA2);
    bool ok = true;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < total; idx += gridDim.x * 256) {
      const int r = idx / cols, c = idx - r * cols;
      ok = ok && s_mod2(a[(long)r * lda + c]) <= bound2;
    }
    if (!ok) info[b / nin] = -1;
  }
}

// X[:, c] = 0 for the columns outside [c0, c0 + nc)
template <typename T>
__global__ __launch_bounds__(256) void zero_outside_kernel(int rows, int cols, int c0, int c_step, int nc, T* X,
                                                           long ldx, long sX, int nin, long sX2, int batch) {
  const int out = cols - nc;
  for (int b = blockIdx.y; b < batch; b += gridDim.y) {
    T* x = X + batch_offset(b, nin, sX, sX2);
    const int cb = c0 + (b % nin) * c_step;
    for (long idx = (long)blockIdx.x * 256 + threadIdx.x; idx < (long)rows * out; idx += (long)gridDim.x * 256) {
      const int r = (int)(idx / out), c = (int)(idx - (long)r * out);
      x[(long)r * ldx + (c < cb ? c : c + nc)] = s_zero<T>();
    }
  }
}

#if HPS_LU_TYPES & 1
size_t lub_scratch_bytes(const LuPlan& p, int batch) {
  int cnt = 1;
  for (int i = 0; i < p.nstage; ++i) cnt = cnt > p.st[i].cnt ? cnt : p.st[i].cnt;
  // pivots and swap tables that the panel kernels write, arrival counters
  return (size_t)batch * cnt * (LUB_NB + SWTAB + 1) * sizeof(int);
}
#endif

// The parts of a stage in one launch: nin groups of each of batch matrices.
template <typename T>
struct Parts {
  const T* p;
  long ld, s, s2;  // row stride, matrix stride, group stride
};

template <typename T>
static hipError_t mul(int M, int N, int K, double alpha, Parts<T> A, Parts<T> B, double beta, Parts<T> D, int nin,
                      int batch, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  GemmArgs<T> g;
  g.M = M;
  g.N = N;
  g.K = K;
  g.alpha = alpha;
  g.beta = beta;
  g.A = A.p;
  g.lda = A.ld;
  g.sA = A.s;
  g.sA2 = A.s2;
  g.B = B.p;
  g.ldb = B.ld;
  g.sB = B.s;
  g.sB2 = B.s2;
  g.C = beta != 0.0 ? D.p : nullptr;
  g.ldc = D.ld;
  g.sC = D.s;
  g.sC2 = D.s2;
  g.D = const_cast<T*>(D.p);
  g.ldd = D.ld;
  g.sD = D.s;
  g.sD2 = D.s2;
  g.nin = nin;
  g.batch = batch * nin;
  return gemm<T>(g, s);
}

// LU of the nb x nb diagonal blocks (nb <= 128) of nin parts of batch matrices;
// db receives the packed 32 x 32 inverses, part by part.
template <typename T>
static hipError_t diag_block_lu(int nb, Parts<T> A, T* db, int* arrivals, int* scratch, int* info,
                                typename real_of<T>::type bound, int nin, int batch, hipStream_t s) {
  const int parts = nin * batch;
  int* ipiv = scratch;  // the panel kernels' pivots and swap tables, not used here
  int* swtab = ipiv + (long)parts * nb;
  T* a = const_cast<T*>(A.p);
  for (int k = 0; k < nb; k += LU_NB) {
    const int kb = nb - k < LU_NB ? nb - k : LU_NB, m = nb - k;
    const double pf = flop_mult<T>() * parts * ((double)m * kb * kb - (double)kb * kb * kb / 3.0);
    // few parts: the unpivoted panel; many: one workgroup a part
    if (parts <= LUB_SPREAD_PARTS) {
      static const std::string nm_np = std::string("getrf_panel_nopiv<") + tname<T>() + ">";
      prof::Scope ps(s, nm_np.c_str(), pf, 2.0 * sizeof(T) * (double)m * kb * parts);
      const int row_wgs = m - kb > 0 ? ceil_div(m - kb, NOPIV_ROWS) : 1;
      const int u12_wgs = ceil_div(m - kb, LU_NB);
      hipLaunchKernelGGL((getrf_panel_nopiv_kernel<T>), dim3(row_wgs + u12_wgs, parts), dim3(256), 0, s, nb, a, A.ld,
                         A.s, k, kb, ipiv, db, arrivals, info, row_wgs, nb, nin, A.s2, bound);
      HPS_LU_CHECK(hipGetLastError());
    } else {
      {
        static const std::string nm_rows = std::string("getrf_panel_rows_nopiv<") + tname<T>() + ">";
        prof::Scope ps(s, nm_rows.c_str(), pf, 2.0 * sizeof(T) * (double)m * kb * parts);
        hipLaunchKernelGGL((getrf_panel_rows_kernel<T, 1, 128, true>), dim3(parts), dim3(128), 0, s, nb, a, A.ld, A.s,
                           k, kb, ipiv, info, db, swtab, nin, A.s2, bound);
        HPS_LU_CHECK(hipGetLastError());
      }
      if (m - kb > 0) {
        static const std::string nm = std::string("getrf_u12<") + tname<T>() + ">";
        HPS_LU_CHECK(trsm_block<T>(false, nb, m - kb, db, a + k + kb, A.ld, A.s, k, kb, parts, s, nm, nin, A.s2));
      }
    }
    const long o = (long)(k + kb) * A.ld;
    HPS_LU_CHECK(mul<T>(m - kb, m - kb, kb, -1.0, {a + o + k, A.ld, A.s, A.s2},
                        {a + (long)k * A.ld + k + kb, A.ld, A.s, A.s2}, 1.0, {a + o + k + kb, A.ld, A.s, A.s2}, nin,
                        batch, s));
  }
  return hipSuccess;
}

template <typename T>
hipError_t lu_blocks_factor(const LuPlan& plan, T* A, long lda, long sA, int* perm, T* dinv, T* inv, T* tmp,
                            int* scratch, int* info, int batch, hipStream_t s) {
  const int n = plan.n;
  const auto bound = typename real_of<T>::type(plan.bound);
  if (n <= 0 || batch <= 0) return hipSuccess;
  int cnt = 1;
  for (int i = 0; i < plan.nstage; ++i) cnt = cnt > plan.st[i].cnt ? cnt : plan.st[i].cnt;
  int* arrivals = scratch;  // zero between panels
  scratch += (long)batch * cnt;
  const unsigned igrid = ceil_div((long)batch * n, 256);
  hipLaunchKernelGGL(lu_blocks_init_kernel, dim3(igrid < 4096 ? igrid : 4096), dim3(256), 0, s, n, batch, batch * cnt,
                     perm, info, arrivals);
  HPS_LU_CHECK(hipGetLastError());
  const bool single = plan.nstage == 1 && plan.st[0].cnt == 1 && lub_blocks(plan, n) == 1;
  const long sI = lub_inv_elems(plan, 1);
  T* ginv = inv;
  for (int is = 0; is < plan.nstage; ++is) {
    const LuStage& st = plan.st[is];
    const int nin = st.cnt, parts = nin * batch, size = st.size;
    const int nb0 = lub_ld(plan, size);
    const int end = st.r0 + nin * size;  // first unknown after the stage
    const int rest = n - end;
    // 32 x 32 inverses of the current block (a single block's are dinv itself), then the panels
    T* db = single ? dinv : tmp;
    T* pan = tmp + (long)parts * nb0 * LU_NB;
    const long gs = (long)size * (lda + 1);               // diagonal step from group to group
    const long gr = (long)size * lda, gc = (long)size;    // row and column step
    const long sI2 = (long)lub_blocks(plan, size) * 2 * nb0 * nb0;
    T* a0 = A + (long)st.r0 * (lda + 1);
    const int first = lub_first(plan, size);
    for (int k = 0, blk = 0, nb = first; k < size; k += nb, nb = plan.nbmax, ++blk) {
      const int below = size - k - nb;   // rows (columns) of the group after the block
      const int m = below + rest;
      T* akk = a0 + (long)k * (lda + 1);
      T* li = ginv + (long)blk * 2 * nb0 * nb0;
      const T* ui = li + nb0 * nb0;
      HPS_LU_CHECK(diag_block_lu<T>(nb, {akk, lda, sA, gs}, db, arrivals, scratch, info, bound, nin, batch, s));
      {
        static const std::string nm = std::string("block_inverse<") + tname<T>() + ">";
        prof::Scope ps(s, nm.c_str(), flop_mult<T>() * parts * 2.0 / 3.0 * (double)nb * nb * nb,
                       sizeof(T) * 3.0 * (double)nb * nb * parts);
        const dim3 igrid(2 * ceil_div(nb, LU_NB), parts < 65535 ? parts : 65535);
        if (nb <= 64)  // less LDS: more workgroups a CU
          hipLaunchKernelGGL((block_inverse_kernel<T, 64>), igrid, dim3(256), 0, s, nb, akk, lda, sA, nin, gs, db, li,
                             nb0, sI, sI2, parts);
        else
          hipLaunchKernelGGL((block_inverse_kernel<T, LUB_NB>), igrid, dim3(256), 0, s, nb, akk, lda, sA, nin, gs, db,
                             li, nb0, sI, sI2, parts);
        HPS_LU_CHECK(hipGetLastError());
      }
      if (m == 0) continue;
      static const std::string nmc = std::string("panel_back<") + tname<T>() + ">";
      const dim3 bgrid(ceil_div((long)m * nb, 1024) < 1024 ? ceil_div((long)m * nb, 1024) : 1024,
                       parts < 65535 ? parts : 65535);
      const long sP = (long)m * nb;
      // L21 = A21 inv(U11): the group's rows, then the later unknowns' rows;
      // U12 = inv(L11) A12, the same way by columns
      const Parts<T> u{ui, nb0, sI, sI2}, l{li, nb0, sI, sI2};
      T* arc = A + (long)end * lda + st.r0 + k;    // later rows, the block's columns
      T* acr = A + (long)(st.r0 + k) * lda + end;  // the block's rows, later columns
      if (nb <= LUB_INPLACE && (below == 0 || below > 2) && (rest == 0 || rest > 2)) {
        // one tile holds the block's width, so every workgroup has read all that
        // it overwrites (its rows of A21, its columns of A12) before it writes
        // (one or two columns of A12 take the GEMV kernel, which is not so)
        HPS_LU_CHECK(mul<T>(below, nb, nb, 1.0, {akk + (long)nb * lda, lda, sA, gs}, u, 0.0,
                            {akk + (long)nb * lda, lda, sA, gs}, nin, batch, s));
        HPS_LU_CHECK(mul<T>(rest, nb, nb, 1.0, {arc, lda, sA, gc}, u, 0.0, {arc, lda, sA, gc}, nin, batch, s));
        HPS_LU_CHECK(mul<T>(nb, below, nb, 1.0, l, {akk + nb, lda, sA, gs}, 0.0, {akk + nb, lda, sA, gs}, nin, batch, s));
        HPS_LU_CHECK(mul<T>(nb, rest, nb, 1.0, l, {acr, lda, sA, gr}, 0.0, {acr, lda, sA, gr}, nin, batch, s));
        for (int seg = 0; seg < 2; ++seg) {
          const int rows = seg == 0 ? below : rest;
          if (rows <= 0) continue;
          static const std::string nmk = std::string("panel_check<") + tname<T>() + ">";
          prof::Scope ps(s, nmk.c_str(), 0.0, sizeof(T) * (double)rows * nb * parts);
          hipLaunchKernelGGL((panel_check_kernel<T>), bgrid, dim3(256), 0, s, rows, nb,
                             seg == 0 ? akk + (long)nb * lda : arc, lda, sA, nin, seg == 0 ? gs : gc, bound, info, parts);
          HPS_LU_CHECK(hipGetLastError());
        }
      } else {
        HPS_LU_CHECK(mul<T>(below, nb, nb, 1.0, {akk + (long)nb * lda, lda, sA, gs}, u, 0.0,
                            {pan, nb, sP * nin, sP}, nin, batch, s));
        HPS_LU_CHECK(mul<T>(rest, nb, nb, 1.0, {arc, lda, sA, gc}, u, 0.0, {pan + (long)below * nb, nb, sP * nin, sP},
                            nin, batch, s));
        // (with one group the two segments are neighbours and go back together)
        auto back = [&](bool rows, int first_, int count, T* dst, long step) -> hipError_t {
          if (count <= 0) return hipSuccess;
          prof::Scope ps(s, nmc.c_str(), 0.0, 2.0 * sizeof(T) * (double)count * nb * parts);
          if (rows)
            hipLaunchKernelGGL((panel_back_kernel<T, true>), bgrid, dim3(256), 0, s, count, nb,
                               pan + (long)first_ * nb, (long)nb, sP, dst, lda, sA, nin, step, bound, info, parts);
          else
            hipLaunchKernelGGL((panel_back_kernel<T, false>), bgrid, dim3(256), 0, s, nb, count, pan + first_, (long)m,
                               sP, dst, lda, sA, nin, step, bound, info, parts);
          return hipGetLastError();
        };
        HPS_LU_CHECK(back(true, 0, nin == 1 ? m : below, akk + (long)nb * lda, gs));
        if (nin > 1) HPS_LU_CHECK(back(true, below, rest, arc, gc));
        HPS_LU_CHECK(mul<T>(nb, below, nb, 1.0, l, {akk + nb, lda, sA, gs}, 0.0, {pan, m, sP * nin, sP}, nin, batch, s));
        HPS_LU_CHECK(mul<T>(nb, rest, nb, 1.0, l, {acr, lda, sA, gr}, 0.0, {pan + below, m, sP * nin, sP}, nin, batch, s));
        HPS_LU_CHECK(back(false, 0, nin == 1 ? m : below, akk + nb, gs));
        if (nin > 1) HPS_LU_CHECK(back(false, below, rest, acr, gr));
      }
      // the group's trailing block, the later rows in its columns and its rows
      // in the later columns; the later unknowns' own block waits for the whole
      // group (one product with K = size)
      const Parts<T> lg{akk + (long)nb * lda, lda, sA, gs}, ug{akk + nb, lda, sA, gs};
      const Parts<T> lr{arc, lda, sA, gc}, ur{acr, lda, sA, gr};
      HPS_LU_CHECK(mul<T>(below, below, nb, -1.0, lg, ug, 1.0, {akk + (long)nb * (lda + 1), lda, sA, gs}, nin, batch, s));
      HPS_LU_CHECK(mul<T>(rest, below, nb, -1.0, lr, ug, 1.0, {lr.p + nb, lda, sA, gc}, nin, batch, s));
      HPS_LU_CHECK(mul<T>(below, rest, nb, -1.0, lg, ur, 1.0, {ur.p + (long)nb * lda, lda, sA, gr}, nin, batch, s));
    }
    // the later unknowns' block, run by run; neighbouring groups that share both runs in one product
    for (int i = 0; i < nin; ++i) {
      const LuGroup& g = st.g[i];
      for (int x = 0; x < g.nrun; ++x)
        for (int y = 0; y < g.nrun; ++y) {
          auto has = [&](int j) {
            bool hx = false, hy = false;
            for (int t = 0; t < st.g[j].nrun; ++t) {
              hx = hx || (st.g[j].s[t] == g.s[x] && st.g[j].ns[t] == g.ns[x]);
              hy = hy || (st.g[j].s[t] == g.s[y] && st.g[j].ns[t] == g.ns[y]);
            }
            return hx && hy;
          };
          if (i > 0 && has(i - 1)) continue;  // done with the group before
          int j = i + 1;
          while (j < nin && has(j)) ++j;
          const long k0 = st.r0 + (long)i * size;
          HPS_LU_CHECK(mul<T>(g.ns[x], g.ns[y], (j - i) * size, -1.0, {A + (long)g.s[x] * lda + k0, lda, sA, 0},
                              {A + k0 * lda + g.s[y], lda, sA, 0}, 1.0, {A + (long)g.s[x] * lda + g.s[y], lda, sA, 0},
                              1, batch, s));
        }
    }
    ginv += nin * sI2;
  }
  if (single) return hipSuccess;
  static const std::string nmd = std::string("dinv_form<") + tname<T>() + ">";
  prof::Scope ps(s, nmd.c_str(), 0.0, 2.0 * sizeof(T) * (double)n * LU_NB * batch);
  hipLaunchKernelGGL((dinv_from_factors_kernel<T>), dim3(ceil_div(n, LU_NB), batch < 65535 ? batch : 65535), dim3(256),
                     0, s, n, A, lda, sA, dinv, batch);
  return hipGetLastError();
}

template <typename T>
hipError_t lu_blocks_solve(const LuPlan& plan, const T* A, long lda, long sA, const T* inv, T* B, long ldb, long sB,
                           T* X, long ldx, long sX, int nrhs, bool cols, int batch, hipStream_t s) {
  if (plan.n <= 0 || nrhs <= 0 || batch <= 0) return hipSuccess;
  const long sI = lub_inv_elems(plan, 1);
  long ginv[LUB_MAX_STAGES];
  long off = 0;
  // forward: X = inv(L) B, group by group in the columns where B is not zero
  for (int is = 0; is < plan.nstage; ++is) {
    const LuStage& st = plan.st[is];
    const int nin = st.cnt, size = st.size, nb0 = lub_ld(plan, size);
    const long sI2 = (long)lub_blocks(plan, size) * 2 * nb0 * nb0;
    ginv[is] = off;
    off += nin * sI2;
    const int c0 = cols ? st.c0 : 0, nc = cols ? st.nc : nrhs, cs = cols ? st.c_step : 0;
    const long gb = (long)size * ldb + cs, gx = (long)size * ldx + cs;
    T* b0 = B + (long)st.r0 * ldb + c0;
    T* x0 = X + (long)st.r0 * ldx + c0;
    const T* a0 = A + (long)st.r0 * (lda + 1);
    for (int k = 0, blk = 0, nb = lub_first(plan, size); k < size; k += nb, nb = plan.nbmax, ++blk) {
      const Parts<T> x{x0 + (long)k * ldx, ldx, sX, gx};
      HPS_LU_CHECK(mul<T>(nb, nc, nb, 1.0, {inv + ginv[is] + (long)blk * 2 * nb0 * nb0, nb0, sI, sI2},
                          {b0 + (long)k * ldb, ldb, sB, gb}, 0.0, x, nin, batch, s));
      HPS_LU_CHECK(mul<T>(size - k - nb, nc, nb, -1.0,
                          {a0 + (long)(k + nb) * lda + k, lda, sA, (long)size * (lda + 1)}, x, 1.0,
                          {b0 + (long)(k + nb) * ldb, ldb, sB, gb}, nin, batch, s));
    }
    if (nc < nrhs) {
      hipLaunchKernelGGL((zero_outside_kernel<T>), dim3(256, nin * batch < 65535 ? nin * batch : 65535), dim3(256), 0,
                         s, size, nrhs, c0, cs, nc, X + (long)st.r0 * ldx, ldx, sX, nin, (long)size * ldx,
                         nin * batch);
      HPS_LU_CHECK(hipGetLastError());
    }
    for (int i = 0; i < nin; ++i)
      for (int t = 0; t < st.g[i].nrun; ++t) {
        const long k0 = st.r0 + (long)i * size;
        const int r = st.g[i].s[t];
        HPS_LU_CHECK(mul<T>(st.g[i].ns[t], nc, size, -1.0, {A + (long)r * lda + k0, lda, sA, 0},
                            {x0 + (long)i * gx, ldx, sX, 0}, 1.0, {B + (long)r * ldb + c0 + (long)i * cs, ldb, sB, 0},
                            1, batch, s));
      }
  }
  // backward: B = inv(U) X, all columns
  for (int is = plan.nstage - 1; is >= 0; --is) {
    const LuStage& st = plan.st[is];
    const int nin = st.cnt, size = st.size, nb0 = lub_ld(plan, size);
    const long sI2 = (long)lub_blocks(plan, size) * 2 * nb0 * nb0;
    for (int i = 0; i < nin; ++i)
      for (int t = 0; t < st.g[i].nrun; ++t) {
        const long k0 = st.r0 + (long)i * size;
        const int r = st.g[i].s[t];
        HPS_LU_CHECK(mul<T>(size, nrhs, st.g[i].ns[t], -1.0, {A + k0 * lda + r, lda, sA, 0},
                            {B + (long)r * ldb, ldb, sB, 0}, 1.0, {X + k0 * ldx, ldx, sX, 0}, 1, batch, s));
      }
    const T* a0 = A + (long)st.r0 * (lda + 1);
    for (int blk = lub_blocks(plan, size) - 1; blk >= 0; --blk) {
      const int first = lub_first(plan, size);
      const int k = blk == 0 ? 0 : first + (blk - 1) * plan.nbmax, nb = blk == 0 ? first : plan.nbmax;
      const Parts<T> b{B + (long)(st.r0 + k) * ldb, ldb, sB, (long)size * ldb};
      HPS_LU_CHECK(mul<T>(nb, nrhs, nb, 1.0,
                          {inv + ginv[is] + (long)(2 * blk + 1) * nb0 * nb0, nb0, sI, sI2},
                          {X + (long)(st.r0 + k) * ldx, ldx, sX, (long)size * ldx}, 0.0, b, nin, batch, s));
      HPS_LU_CHECK(mul<T>(k, nrhs, nb, -1.0, {a0 + k, lda, sA, (long)size * (lda + 1)}, b, 1.0,
                          {X + (long)st.r0 * ldx, ldx, sX, (long)size * ldx}, nin, batch, s));
    }
  }
  return hipSuccess;
}

}  // namespace hps
