// ItI leaves with real coefficients, by static condensation (included by
// hps_capi.hip).
//
// The leaf matrix B = [G; A_int] is complex only through the boundary columns of
// the impedance rows G = N + i eta I: the collocation rows and G's interior
// columns are real.  Eliminating the interior first,
//   X = A_ii^{-1} [A_ib | f_i]                 real, ni unknowns
//   S = G_b - G_i X_b                          complex, nb unknowns
//   Y_b = S^{-1} P,  v_b = -S^{-1} G_i X_f     boundary values
//   Y_i = -X_b Y_b,  v_i = X_f - X_b v_b
//   T = Z Y_b,  h = Z v_b + Q_i X_f,  Z = Q_b - Q_i X_b
// costs 19 Mflop a leaf at p = 16 where the LU of B and its solves cost 81
// (complex operations four times), and the factors kept for later solves are
// a third as large.  A complex right-hand side is two real columns: the
// interleaved array read as real, without a copy.
//
// A_ii is the leaf's Dirichlet problem, singular where k^2 is one of its
// eigenvalues (leaf side h with k h >= sqrt(2) pi) and indefinite above the
// first.  While it is definite, its multipliers stay below 2.2, those of S
// mostly below 3 and the entries of X_b, which extend boundary values into the
// leaf, below 1.2, and T is as exact as through the factorisation of B:
// error ratio 0.4 to 1.1 at p = 8, 11 and 16 up to k h = 4.2.  Past the first
// eigenvalue elimination without row exchanges loses up to two digits, often
// with X_b still of size 1 (p = 16: ratio 100 at k h = 4.5, multipliers of 20).  A
// leaf that passes one of the bounds below (or is not finite) gets info = -1, and
// the caller takes the factorisation of B for it: with them the ratio stays below
// 1.5 also for strong advection and small eta, where S is hard to eliminate.
//
// Measured, by the LU of B / condensed: leaf stage at p = 16, L = 7 (16384
// leaves) 55 / 31 ms in complex128, 32 / 19 ms in complex64; Helmholtz build +
// solve there 158 / 135 and, mixed, 107 / 88 ms; gradient at L = 6 43 / 37 ms.  Bound by the real products (12.5 ms, tiles of
// 64 x 64 on 60 .. 196 rows) and the passes between them.
#pragma once

namespace hps {

constexpr double LEAF_EXT_BOUND = 2.0;     // entries of X_b
constexpr double LEAF_INNER_BOUND = 4.0;   // multipliers of A_ii
constexpr double LEAF_BORDER_BOUND = 10.0;  // multipliers of S

// S = G_b - R[:nb, :nb], RB = [P | -R[:nb, nb:]], Z = Q_b - R[nb:, :nb],
// h = R[nb:, nb:]; R (nb + nq, nb + 2 nsrc) real, the sources' columns (re, im)
template <typename C, typename R>
__global__ __launch_bounds__(256) void condense_kernel(int nb, int nq, int nsrc, const R* Rp, const C* Gb,
                                                       const C* Qb, const C* P, C* S, C* RB, C* Z, C* h, int nl) {
  const int wr = nb + 2 * nsrc, wb = nq + nsrc;
  const int nS = nb * nb, nRB = nb * wb, nZ = nq * nb, nh = nq * nsrc;
  for (int l = blockIdx.y; l < nl; l += gridDim.y) {
    const R* r = Rp + (long)l * (nb + nq) * wr;
    for (int idx = blockIdx.x * 256 + threadIdx.x; idx < nS + nRB + nZ + nh; idx += gridDim.x * 256) {
      if (idx < nS) {
        const int i = idx / nb, j = idx - i * nb;
        const C g = Gb[idx];
        S[(long)l * nS + idx] = C{g.re - r[i * wr + j], g.im};
      } else if (idx < nS + nRB) {
        const int e = idx - nS, i = e / wb, j = e - i * wb;
        const R* q = r + i * wr + nb + 2 * (j - nq);
        RB[(long)l * nRB + e] = j < nq ? P[i * nq + j] : C{-q[0], -q[1]};
      } else if (idx < nS + nRB + nZ) {
        const int e = idx - nS - nRB, i = e / nb, j = e - i * nb;
        const C q = Qb[e];
        Z[(long)l * nZ + e] = C{q.re - r[(nb + i) * wr + j], q.im};
      } else {
        const int e = idx - nS - nRB - nZ, i = e / nsrc, j = e - i * nsrc;
        const R* q = r + (nb + i) * wr + nb + 2 * j;
        h[(long)l * nh + e] = C{q[0], q[1]};
      }
    }
  }
}

// info[l] = -1 where the extension X (ni rows of nb entries, row stride ld)
// passes the bound or either factorisation was rejected
template <typename R>
__global__ __launch_bounds__(256) void extension_check_kernel(int ni, int nb, const R* X, long ld, const int* info_s,
                                                              int* info) {
  const int l = blockIdx.x;
  const R* x = X + (long)l * ni * ld;
  bool ok = info_s[l] == 0;
  for (int idx = threadIdx.x; idx < ni * nb; idx += 256) {
    const int i = idx / nb, j = idx - i * nb;
    ok = ok && fabs(x[(long)i * ld + j]) <= R(LEAF_EXT_BOUND);
  }
  if (!ok) info[l] = -1;
}

// info[l] = -1 where zeroth / (xx + yy) of the leaf's n points passes the limit
// or is not a number (yy may be null)
template <typename R>
__global__ __launch_bounds__(256) void mark_indefinite_kernel(int n, const R* zeroth, const R* xx, const R* yy,
                                                              R limit, int* info, int nl) {
  for (int l = blockIdx.x; l < nl; l += gridDim.x) {
    bool ok = true;
    for (int i = threadIdx.x; i < n; i += 256) {
      const long at = (long)l * n + i;
      ok = ok && zeroth[at] / (yy ? xx[at] + yy[at] : xx[at]) <= limit;
    }
    if (!ok) info[l] = -1;  // every writer writes the same value
  }
}

}  // namespace hps

struct CondensedWs {
  size_t R, S_inv, A_inv, A_tmp, A_x, S_tmp, RB, S_x, Z, info_s, ints, total;
};

// regions of the workspace for chunks of m leaves (elements of the real type e, complex 2 e)
static CondensedWs condensed_ws(size_t e, int nl, int n, int nb, int nq, int nsrc) {
  const int m = nl < LEAF_CHUNK ? nl : LEAF_CHUNK;
  const int ni = n - nb, wr = nb + 2 * nsrc, wb = nq + nsrc;
  const LuPlan pa = lu_plan_dense(ni, wr, m), ps = lu_plan_dense(nb, wb, m);
  CondensedWs w;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t o = at;
    at += align_up(bytes);
    return o;
  };
  w.R = take((size_t)m * (nb + nq) * wr * e);
  w.A_inv = take(lub_inv_elems(pa, m) * e);
  w.A_tmp = take(lub_tmp_elems(pa, m) * e);
  w.A_x = take((size_t)m * ni * wr * e);
  w.S_inv = take(lub_inv_elems(ps, m) * 2 * e);
  w.S_tmp = take(lub_tmp_elems(ps, m) * 2 * e);
  w.RB = take((size_t)m * nb * wb * 2 * e);
  w.S_x = take((size_t)m * nb * wb * 2 * e);
  w.Z = take((size_t)m * nq * nb * 2 * e);
  w.info_s = take((size_t)m * sizeof(int));
  w.ints = take(std::max(lub_scratch_bytes(pa, m), lub_scratch_bytes(ps, m)));
  w.total = at;
  return w;
}

size_t hps_leaf_condensed_workspace(int dtype, int nl, int n, int nb, int nq, int nsrc) {
  return condensed_ws(dtype_size(dtype) / 2, nl, n, nb, nq, nsrc).total;
}

template <typename C>
static int leaf_condensed_t(hps_handle_t h, int nl_all, int n, int nb, int nq, int nsrc, int ncoef, const int* coef_ops,
                            const void* coeffs, const void* diffops, const void* GQ, const void* Gb, const void* Qb,
                            const void* Pv, const void* source, void* Yv, void* Tv, void* vv, void* hv, void* aluv,
                            int* aperm, void* adinvv, void* Xv, void* sluv, int* sperm, void* sdinvv, int* info,
                            char* ws) {
  using R = typename real_of<C>::type;
  hipStream_t s = h->stream;
  const int ni = n - nb, wr = nb + 2 * nsrc, wb = nq + nsrc;
  const CondensedWs o = condensed_ws(sizeof(R), nl_all, n, nb, nq, nsrc);
  const int m = nl_all < LEAF_CHUNK ? nl_all : LEAF_CHUNK;  // every chunk takes the first one's plan
  LuPlan pa = lu_plan_dense(ni, wr, m), ps = lu_plan_dense(nb, wb, m);
  pa.bound = LEAF_INNER_BOUND;
  ps.bound = LEAF_BORDER_BOUND;
  CoefOps co;
  for (int i = 0; i < 16; ++i) co.op[i] = i < ncoef ? coef_ops[i] : 0;
  {
    // A_int for every leaf at once
    HPS_PROF("leaf_assemble", R, 2.0 * ncoef * (double)ni * n * nl_all,
             sizeof(R) * ((double)ni * n * nl_all + (double)ncoef * n * nl_all));
    dim3 g(ni, ceil_div(nl_all, ASM_LEAVES) < 65535 ? ceil_div(nl_all, ASM_LEAVES) : 65535);
    hipLaunchKernelGGL((assemble_kernel<R>), g, dim3(256), 0, s, n, nl_all, ncoef, co, (const R*)coeffs,
                       (const R*)diffops, nb, ni, 0, n, (R*)aluv, (long)n, (long)ni * n);
    HPS_CHECK_HIP(h, hipGetLastError());
  }
  R* R1 = (R*)(ws + o.R);
  C* RB = (C*)(ws + o.RB);
  C* Z = (C*)(ws + o.Z);
  int* info_s = (int*)(ws + o.info_s);
  int* ints = (int*)(ws + o.ints);
  for (int l0 = 0; l0 < nl_all; l0 += LEAF_CHUNK) {
    const int nl = nl_all - l0 < LEAF_CHUNK ? nl_all - l0 : LEAF_CHUNK;
    R* alu = (R*)aluv + (long)l0 * ni * n;
    R* X = (R*)Xv + (long)l0 * ni * wr;
    C* slu = (C*)sluv + (long)l0 * nb * nb;
    C* Y = (C*)Yv + (long)l0 * n * nq;
    C* T = (C*)Tv + (long)l0 * nq * nq;
    C* v = nsrc ? (C*)vv + (long)l0 * n * nsrc : nullptr;
    C* hh = nsrc ? (C*)hv + (long)l0 * nq * nsrc : nullptr;
    const C* f = source ? (const C*)source + (long)l0 * n * nsrc : nullptr;
    const long sX = (long)ni * wr, sRB = (long)nb * wb;
    // X = A_ii^{-1} [A_ib | f_i]
    HPS_CHECK_HIP(h, copy2d<R>(ni, nb, 1.0, alu, n, (long)ni * n, X, wr, sX, nl, s));
    if (nsrc)
      HPS_CHECK_HIP(h, copy2d<R>(ni, 2 * nsrc, 1.0, f ? (const R*)(f + (long)nb * nsrc) : nullptr, 2 * nsrc,
                                 2 * (long)n * nsrc, X + nb, wr, sX, nl, s));
    R* ainv = (R*)(ws + o.A_inv);
    HPS_CHECK_HIP(h, lu_blocks_factor<R>(pa, alu + nb, n, (long)ni * n, aperm + (long)l0 * ni,
                                         (R*)adinvv + (long)l0 * dinv_elems(ni), ainv, (R*)(ws + o.A_tmp), ints,
                                         info + l0, nl, s));
    HPS_CHECK_HIP(h, lu_blocks_solve<R>(pa, alu + nb, n, (long)ni * n, ainv, X, wr, sX, (R*)(ws + o.A_x), wr, sX, wr,
                                        false, nl, s));
    // [G_i; Q_i] X, then the boundary system
    // (derivatives: sums with cancellation, whose rounding decides T's)
    {
      GemmArgs<R> g;
      g.M = nb + nq;
      g.N = wr;
      g.K = ni;
      g.A = (const R*)GQ;
      g.lda = ni;
      g.B = X;
      g.ldb = wr;
      g.sB = sX;
      g.D = R1;
      g.ldd = wr;
      g.sD = (long)(nb + nq) * wr;
      g.batch = nl;
      g.sum2 = 1;
      HPS_CHECK_HIP(h, gemm<R>(g, s));
    }
    {
      const int total = nb * nb + nb * wb + nq * nb + nq * nsrc;
      HPS_PROF("leaf_condense", C, 0.0, sizeof(C) * 1.5 * (double)total * nl);
      hipLaunchKernelGGL((condense_kernel<C, R>), dim3(ceil_div(total, 256) < 16 ? ceil_div(total, 256) : 16,
                                                       nl < 65535 ? nl : 65535),
                         dim3(256), 0, s, nb, nq, nsrc, R1, (const C*)Gb, (const C*)Qb, (const C*)Pv, slu, RB, Z, hh,
                         nl);
      HPS_CHECK_HIP(h, hipGetLastError());
    }
    C* sinv = (C*)(ws + o.S_inv);
    HPS_CHECK_HIP(h, lu_blocks_factor<C>(ps, slu, nb, (long)nb * nb, sperm + (long)l0 * nb,
                                         (C*)sdinvv + (long)l0 * dinv_elems(nb), sinv, (C*)(ws + o.S_tmp), ints, info_s,
                                         nl, s));
    HPS_CHECK_HIP(h, lu_blocks_solve<C>(ps, slu, nb, (long)nb * nb, sinv, RB, wb, sRB, (C*)(ws + o.S_x), wb, sRB, wb,
                                        false, nl, s));
    {
      HPS_PROF("leaf_check", R, 0.0, sizeof(R) * (double)ni * nb * nl);
      hipLaunchKernelGGL((extension_check_kernel<R>), dim3(nl), dim3(256), 0, s, ni, nb, X, (long)wr, info_s,
                         info + l0);
      HPS_CHECK_HIP(h, hipGetLastError());
    }
    // Y and v: boundary rows from the solve, interior rows through X
    HPS_CHECK_HIP(h, copy2d<C>(nb, nq, 1.0, RB, wb, sRB, Y, nq, (long)n * nq, nl, s));
    HPS_CHECK_HIP(h, gemm_call<R>(s, ni, 2 * nq, nb, -1.0, X, wr, sX, (const R*)RB, 2 * wb, 2 * sRB, 0.0, nullptr, 0, 0,
                                  (R*)(Y + (long)nb * nq), 2 * nq, 2 * (long)n * nq, nl));
    if (nsrc) {
      HPS_CHECK_HIP(h, copy2d<C>(nb, nsrc, 1.0, RB + nq, wb, sRB, v, nsrc, (long)n * nsrc, nl, s));
      HPS_CHECK_HIP(h, gemm_call<R>(s, ni, 2 * nsrc, nb, -1.0, X, wr, sX, (const R*)(RB + nq), 2 * wb, 2 * sRB, 1.0,
                                    X + nb, wr, sX, (R*)(v + (long)nb * nsrc), 2 * nsrc, 2 * (long)n * nsrc, nl));
    }
    // T and h
    HPS_CHECK_HIP(h, gemm_call<C>(s, nq, nq, nb, 1.0, Z, nb, (long)nq * nb, RB, wb, sRB, 0.0, nullptr, 0, 0, T, nq,
                                  (long)nq * nq, nl));
    if (nsrc)
      HPS_CHECK_HIP(h, gemm_call<C>(s, nq, nsrc, nb, 1.0, Z, nb, (long)nq * nb, RB + nq, wb, sRB, 1.0, hh, nsrc,
                                    (long)nq * nsrc, hh, nsrc, (long)nq * nsrc, nl));
  }
  return HPS_OK;
}

int hps_mark_indefinite(hps_handle_t h, int dtype, int nl, int n, const void* zeroth, const void* xx, const void* yy,
                        double limit, int* info) {
  if (!h) return HPS_ERR_ARG;
  HPS_ARG(h, dtype == HPS_F64 || dtype == HPS_F32, "real coefficients required");
  HPS_ARG(h, nl > 0 && n > 0, "bad leaf sizes");
  HPS_ARG(h, zeroth && xx && info, "null pointer");
  const dim3 grid(nl < 65535 ? nl : 65535);
  if (dtype == HPS_F64)
    hipLaunchKernelGGL((mark_indefinite_kernel<double>), grid, dim3(256), 0, h->stream, n, (const double*)zeroth,
                       (const double*)xx, (const double*)yy, limit, info, nl);
  else
    hipLaunchKernelGGL((mark_indefinite_kernel<float>), grid, dim3(256), 0, h->stream, n, (const float*)zeroth,
                       (const float*)xx, (const float*)yy, (float)limit, info, nl);
  HPS_CHECK_HIP(h, hipGetLastError());
  return HPS_OK;
}

int hps_leaf_condensed(hps_handle_t h, int dtype, int nl, int n, int nb, int nq, int nsrc, int ncoef,
                       const int* coef_ops, const void* coeffs, const void* diffops, const void* GQ, const void* Gb,
                       const void* Qb, const void* P, const void* source, void* Y, void* T, void* v, void* hvec,
                       void* alu, int* aperm, void* adinv, void* X, void* slu, int* sperm, void* sdinv, int* info,
                       void* ws, size_t ws_bytes) {
  if (!h) return HPS_ERR_ARG;
  HPS_ARG(h, dtype == HPS_C128 || dtype == HPS_C64, "condensed leaves are complex");
  HPS_ARG(h, nl > 0 && n > nb && nb > 0 && nq > 0 && nsrc >= 0, "bad leaf sizes");
  HPS_ARG(h, ncoef > 0 && ncoef <= 16 && coef_ops, "1..16 coefficients required");
  HPS_ARG(h, coeffs && diffops && GQ && Gb && Qb && P && Y && T && alu && aperm && adinv && X && slu && sperm &&
                 sdinv && info,
          "null pointer");
  HPS_ARG(h, nsrc == 0 || (v && hvec), "v/h required when nsrc > 0");
  if (ws_bytes < hps_leaf_condensed_workspace(dtype, nl, n, nb, nq, nsrc)) {
    h->err = "condensed leaf workspace too small";
    return HPS_ERR_WORKSPACE;
  }
  auto fn = dtype == HPS_C128 ? leaf_condensed_t<c128> : leaf_condensed_t<c64>;
  return fn(h, nl, n, nb, nq, nsrc, ncoef, coef_ops, coeffs, diffops, GQ, Gb, Qb, P, source, Y, T, v, hvec, alu, aperm,
            adinv, X, slu, sperm, sdinv, info, (char*)ws);
}
