// ks_ksp.hip -- the linear solves of shift-and-invert on the device.
//
// STSINVERT applies (A - sigma I)^-1 by an inner Krylov solve (the reference's
// STApply_Sinvert -> KSPSolve, src/sys/classes/st/impls/sinvert/sinvert.c:16-30,
// with KSPCG and PCJACOBI as in src/eps/tutorials/ex11.c's test 2).  PETSc is not
// part of the reference tree; the solver here is the preconditioned conjugate
// gradient method in PETSc's KSPCG form (Hestenes-Stiefel recurrences, the
// preconditioned residual norm |B r| for the test rnorm <= max(rtol |B b|, abstol))
// with B = diag(A - sigma I)^-1 (zero diagonal entries replaced by 1, as PCJACOBI
// does), and for an indefinite shifted matrix BiCGStab (van der Vorst 1992) in
// PETSc's KSPBCGS form with the same left preconditioner.  Every scalar of a
// recurrence and the convergence test stay on the device, so the host enqueues
// iterations in chunks and reads one small state block per chunk; once a solve
// has converged or failed the later launches exit at their first instruction.
//
// Small solves are bound by their launches (a dependent launch costs 3-4 us, a
// pass over a vector of 65,000 rows less), so an iteration takes as few as its
// sums allow: two for CG, three for BiCGStab.  A kernel begins by adding the
// previous one's per-workgroup partial sums (every workgroup adds the same
// values in the same order) and takes the recurrence's scalars from them, and
// the vector a product needs is formed on the fly where its entries are
// gathered.  256 x 255 grid, one CG iteration: 24.3 us with a launch for each
// operation and each sum, 10.8 us so (BiCGStab 41.3 and 16.5).
#include <algorithm>
#include <cstring>
#include <new>
#include <vector>

#include "ks_internal.hpp"

namespace {

#define KS_PCG_BLOCKS 512        // workgroups of the vector kernels
#define KS_KSP_SPMV_BLOCKS 2048  // workgroups of the products (each walks row blocks)

// The solver state.  Two copies at the end of the workspace: a kernel reads one,
// its first workgroup writes the other, the next kernel reads that one.
struct ksp_state {
  double sc[12];
  int32_t its, reason, sconv, maxits;   // reason: 0 while iterating, > 0 converged, < 0 failed
};
static_assert(2 * sizeof(ksp_state) <= 64 * sizeof(double), "the solver states take 64 doubles");
enum { S_RZ = 0, S_RZOLD, S_PQ,                                          // CG
       S_RHO = 0, S_RHOOLD, S_ALPHA, S_OMEGA, S_SS,                      // BiCGStab
       S_TTOL = 8, S_RNORM };

#define KS_FOR_ROWS(i, n) for (int i = blockIdx.x * KS_BLOCK + threadIdx.x; i < n; i += gridDim.x * KS_BLOCK)

// workgroup sums of NV values, to every thread: a butterfly in each wave, then the waves in order
template <int NV>
__device__ __forceinline__ void all_sum(double (&v)[NV], double (&lds)[KS_WAVES][NV]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int j = 0; j < NV; j++) v[j] = ks_wave_sum(v[j]);
  if (lane == 0)
#pragma unroll
    for (int j = 0; j < NV; j++) lds[wave][j] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; j++) {
    v[j] = lds[0][j];
#pragma unroll
    for (int w = 1; w < KS_WAVES; w++) v[j] += lds[w][j];
  }
}

// this thread's share of the np partial sums part[NV b + j]
template <int NV>
__device__ __forceinline__ void load_partials(const double *__restrict__ part, int np, double (&v)[NV]) {
#pragma unroll
  for (int j = 0; j < NV; j++) v[j] = 0.0;
  for (int q = threadIdx.x; q < np; q += KS_BLOCK)
#pragma unroll
    for (int j = 0; j < NV; j++) v[j] += part[NV * q + j];
}

template <int NV>
__device__ __forceinline__ void store_partials(double (&v)[NV], double *__restrict__ part, double (&lds)[KS_WAVES][NV],
                                               int b) {
  all_sum(v, lds);
  if (threadIdx.x == 0)
#pragma unroll
    for (int j = 0; j < NV; j++) part[NV * b + j] = v[j];
}

// the state field by field (copied whole it passes through scratch memory)
__device__ __forceinline__ void load_state(ksp_state &s, const ksp_state *in) {
#pragma unroll
  for (int j = 0; j < 12; j++) s.sc[j] = in->sc[j];
  s.its = in->its;
  s.reason = in->reason;
  s.sconv = in->sconv;
  s.maxits = in->maxits;
}
__device__ __forceinline__ void publish(const ksp_state &s, ksp_state *out) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
#pragma unroll
    for (int j = 0; j < 12; j++) out->sc[j] = s.sc[j];
    out->its = s.its;
    out->reason = s.reason;
    out->sconv = s.sconv;
    out->maxits = s.maxits;
  }
}

// dinv[i] = 1 / (a_ii - sigma), 1 where that is zero; all ones without a preconditioner
__global__ __launch_bounds__(KS_BLOCK) void k_jacobi(const int32_t *__restrict__ rowptr,
                                                    const int32_t *__restrict__ colidx,
                                                    const double *__restrict__ val, int n, double sigma, int jacobi,
                                                    double *__restrict__ dinv) {
  KS_FOR_ROWS(i, n) {
    double d = 0.0;
    if (jacobi) {
      for (int32_t e = rowptr[i]; e < rowptr[i + 1]; e++)
        if (colidx[e] == i) d += val[e];
      d -= sigma;
    }
    dinv[i] = (d == 0.0) ? 1.0 : 1.0 / d;
  }
}

// the end of a CG iteration from the new z.r (t[0]) and z.z (t[1]), and its tests: p^T (A - sigma I) p
// <= 0 (KSP_DIVERGED_INDEFINITE_MAT, -8), |B r| <= ttol (1), the iteration limit (-3)
__device__ __forceinline__ void cg_decide(ksp_state &s, const double (&t)[2]) {
  s.sc[S_RZOLD] = s.sc[S_RZ];
  s.sc[S_RZ] = t[0];
  s.sc[S_RNORM] = sqrt(t[1]);
  s.its += 1;
  if (!(s.sc[S_PQ] > 0.0)) s.reason = -8;
  else if (s.sc[S_RNORM] <= s.sc[S_TTOL]) s.reason = 1;
  else if (s.its >= s.maxits) s.reason = -3;
}

// the end of a BiCGStab iteration from (r, r) and (rhat, r): converged (1), breakdown (-5), limit (-3)
__device__ __forceinline__ void bcgs_decide(ksp_state &s, const double (&t)[2]) {
  s.its += 1;
  if (s.sconv) {
    s.sc[S_RNORM] = sqrt(s.sc[S_SS]);
    s.reason = 1;
    return;
  }
  s.sc[S_RNORM] = sqrt(t[0]);
  if (s.sc[S_RNORM] <= s.sc[S_TTOL]) s.reason = 1;
  else {
    s.sc[S_RHOOLD] = s.sc[S_RHO];
    s.sc[S_RHO] = t[1];
    if (t[1] == 0.0 || s.sc[S_OMEGA] == 0.0) s.reason = -5;
    else if (s.its >= s.maxits) s.reason = -3;
  }
}

// a b rounded by itself (not contracted into a sum), so an entry formed for a
// neighbour's product is the entry its own row stores
__device__ __forceinline__ double rounded_product(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}

// The vector w of a product and what is summed with its result y:
//   KSP_CG  w = B r + beta p_old            sums (w, y)
//   KSP_P   w = r + beta (p_old - omega v)  sums (rhat, y)
//   KSP_S   w = r - alpha v                 sums (w, y), (y, y), (w, w)
// ksp_take adds up the previous kernel's sums (where they end an iteration or
// give alpha), moves the state on and leaves w's two scalars in c.
enum { KSP_CG, KSP_P, KSP_S };
template <int MODE>
struct ksp_form {
  static constexpr int NI = MODE == KSP_S ? 1 : 2;   // sums taken
  const double *__restrict__ r, *__restrict__ p, *__restrict__ v, *__restrict__ dinv;
  double c1 = 0.0, c2 = 0.0;
  struct in { double a, b, c; };                     // the entries w_i is formed from
  __device__ __forceinline__ in load(int i) const {
    in e = {r[i], 0.0, 0.0};
    if (MODE == KSP_CG) e.b = p[i], e.c = dinv[i];
    else if (MODE == KSP_P) e.b = p[i], e.c = v[i];
    else e.b = v[i];
    return e;
  }
  __device__ __forceinline__ double value(const in &e) const {
    if (MODE == KSP_CG) {
      const double z = rounded_product(e.c, e.a);
      return c2 != 0.0 ? z + c1 * e.b : z;           // c2 0: the first iteration (p_old is unset)
    }
    if (MODE == KSP_P) return e.a + c1 * (e.b - c2 * e.c);
    return e.a - c1 * e.b;
  }
  // t: this thread's share of the previous kernel's sums
  __device__ __forceinline__ void take(ksp_state &s, double (&t)[NI], bool sums, double (&lds)[KS_WAVES][NI]) {
    if (!s.reason && sums) {
      all_sum(t, lds);
      if constexpr (MODE == KSP_CG) cg_decide(s, t);
      else if constexpr (MODE == KSP_P) bcgs_decide(s, t);
      else if (t[0] == 0.0) s.reason = -5;           // (rhat, v) = 0
      else s.sc[S_ALPHA] = s.sc[S_RHO] / t[0];
    }
    if (MODE == KSP_CG) {
      c1 = s.its ? s.sc[S_RZ] / s.sc[S_RZOLD] : 0.0;
      c2 = s.its ? 1.0 : 0.0;
    } else if (MODE == KSP_P) {
      c1 = (s.sc[S_RHO] / s.sc[S_RHOOLD]) * (s.sc[S_ALPHA] / s.sc[S_OMEGA]);
      c2 = s.sc[S_OMEGA];
    } else c1 = s.sc[S_ALPHA];
  }
};

struct ksp_prod {
  const int32_t *blk, *rowptr, *colidx;
  const double *val;
  int nblocks, n;
  const double *r, *p, *v, *rh, *dinv;
  double *w, *y;
  double sigma;
  const ksp_state *in;
  ksp_state *out;
  const double *pin;   // the previous kernel's partial sums (npin of them)
  int npin, decide;    // decide: they end an iteration (else the state is decided)
  double *pout;
};

// w by itself, for long vectors: with FUSE a product gathers up to three vectors
// where it gathers one of w
template <int MODE>
__global__ __launch_bounds__(KS_BLOCK) void k_ksp_vector(ksp_prod a) {
  __shared__ double lin[KS_WAVES][ksp_form<MODE>::NI];
  ksp_form<MODE> f = {a.r, a.p, a.v, a.dinv};
  ksp_state s;
  load_state(s, a.in);
  const bool sums = MODE == KSP_S || a.decide;
  double t[ksp_form<MODE>::NI];
  load_partials(a.pin, sums ? a.npin : 0, t);
  f.take(s, t, sums, lin);
  publish(s, a.out);
  if (s.reason) return;
  double *__restrict__ w = a.w;
  KS_FOR_ROWS(i, a.n) w[i] = f.value(f.load(i));
}

// The product of an iteration, y = (A - sigma I) w, times diag(dinv) where the
// preconditioner is applied here (PC; for CG it is part of w), and its sums
// (without PC -- ILU(0), B applied by later launches -- only (w, w)).  FUSE: w is
// formed where it is gathered and stored for the rows of the workgroup, and the
// kernel moves the state on; else w is there and the state is only read.
// The row blocks and the order of a row's sum are those of k_spmv_csr.  A row
// block's entries are fetched before the previous block (or the first one's
// scalars) is worked on.
template <int MODE, bool PC, bool FUSE>
__global__ __launch_bounds__(KS_BLOCK) void k_ksp_product(ksp_prod a) {
  constexpr int NV = MODE == KSP_S ? 3 : 1, NI = ksp_form<MODE>::NI, PER = KS_SPMV_NNZ / KS_BLOCK;
  __shared__ double prod[KS_SPMV_NNZ];
  __shared__ double lin[KS_WAVES][NI], lout[KS_WAVES][NV], red[KS_WAVES];
  const int tid = threadIdx.x, nblocks = a.nblocks;
  const double *__restrict__ val = a.val, *__restrict__ rh = a.rh, *__restrict__ dinv = a.dinv;
  const int32_t *__restrict__ colidx = a.colidx, *__restrict__ rowptr = a.rowptr, *__restrict__ blk = a.blk;
  double *__restrict__ w = a.w, *__restrict__ y = a.y;
  const double *wr = a.w;
  const double sigma = a.sigma;
  ksp_form<MODE> f = {a.r, a.p, a.v, a.dinv};
  using ent = typename ksp_form<MODE>::in;
  ksp_state s;
  double t[NI];
  const bool sums = FUSE && (MODE == KSP_S || a.decide);
  load_state(s, a.in);
  load_partials(a.pin, sums ? a.npin : 0, t);
  // the block at hand
  int r0, r1, p0, p1;
  bool longrow;
  double va[PER];
  ent en[FUSE ? PER : 1];
  double xw[FUSE ? 1 : PER];
  auto fetch = [&](int g) __attribute__((always_inline)) {
    const int b = ks_xcd_block(g, nblocks);
    r0 = blk[b];
    r1 = blk[b + 1];
    p0 = rowptr[r0];
    p1 = rowptr[r1];
    longrow = r1 - r0 == 1 && p1 - p0 > KS_SPMV_NNZ;
    if (longrow || p1 == p0) return;
    int ci[PER];
#pragma unroll
    for (int u = 0; u < PER; u++) {
      const int q = min(p0 + tid + u * KS_BLOCK, p1 - 1);
      ci[u] = colidx[q];
      va[u] = val[q];
    }
#pragma unroll
    for (int u = 0; u < PER; u++) {
      if constexpr (FUSE) en[u] = f.load(ci[u]);
      else xw[u] = wr[ci[u]];
    }
  };
  fetch(blockIdx.x);
  if (FUSE) {
    f.take(s, t, sums, lin);
    publish(s, a.out);
  }
  if (s.reason) return;
  double o[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) o[j] = 0.0;
  auto row = [&](int i, double sum) __attribute__((always_inline)) {
    const double wi = FUSE ? f.value(f.load(i)) : wr[i];
    double yi = sum - sigma * wi;
    if (PC && MODE != KSP_CG) yi *= dinv[i];
    if (FUSE) w[i] = wi;
    y[i] = yi;
    if (MODE == KSP_CG) o[0] += wi * yi;
    else if (MODE == KSP_P) o[0] += PC ? rh[i] * yi : 0.0;
    else {
      o[0] += PC ? wi * yi : 0.0;
      o[NV > 1 ? 1 : 0] += PC ? yi * yi : 0.0;
      o[NV > 2 ? 2 : 0] += wi * wi;
    }
  };
  for (int g = blockIdx.x; g < nblocks; g += gridDim.x) {
    const int nrows = r1 - r0, R0 = r0, P0 = p0, P1 = p1;
    const bool lng = longrow;
    if (!lng && P1 > P0) {
#pragma unroll
      for (int u = 0; u < PER; u++) {
        double x;
        if constexpr (FUSE) x = f.value(en[u]);
        else x = xw[u];
        prod[tid + u * KS_BLOCK] = va[u] * x;
      }
    }
    __syncthreads();
    if (g + (int)gridDim.x < nblocks) fetch(g + gridDim.x);
    if (lng) {   // a long row: the whole workgroup strides over it
      double x = 0.0;
      for (int q = P0 + tid; q < P1; q += KS_BLOCK) {
        const int c = colidx[q];
        x += val[q] * (FUSE ? f.value(f.load(c)) : wr[c]);
      }
      const double tot = ks_block_sum(x, red);
      if (tid == 0) row(R0, tot);
    } else {
      int tpr = 1;
      while (tpr < 64 && nrows * (tpr << 1) <= KS_BLOCK) tpr <<= 1;
      const int lr = tid / tpr, sub = tid & (tpr - 1);
      if (lr < nrows) {
        const int rs = rowptr[R0 + lr] - P0, re = rowptr[R0 + lr + 1] - P0;
        double x = 0.0;
        for (int q = rs + sub; q < re; q += tpr) x += prod[q];
        for (int off = tpr >> 1; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
        if (sub == 0) row(R0 + lr, x);
      }
    }
    __syncthreads();
  }
  // a workgroup with one row block leaves its sums at that block's place
  if (PC || MODE == KSP_S)
    store_partials(o, a.pout, lout, gridDim.x == (unsigned)nblocks ? ks_xcd_block(blockIdx.x, nblocks) : blockIdx.x);
}

// ---------------------------------------------------------------- CG
// x = 0, r = b; partials of z.r and z.z, z = B r
__global__ __launch_bounds__(KS_BLOCK) void k_pcg_start(int n, const double *__restrict__ b, double *__restrict__ x,
                                                       double *__restrict__ r, const double *__restrict__ dinv,
                                                       double *__restrict__ part) {
  __shared__ double lds[KS_WAVES][2];
  double t[2] = {0.0, 0.0};
  KS_FOR_ROWS(i, n) {
    const double ri = b[i], zi = dinv[i] * ri;
    x[i] = 0.0;
    r[i] = ri;
    t[0] += zi * ri;
    t[1] += zi * zi;
  }
  store_partials(t, part, lds, blockIdx.x);
}

// a = rz / pq; x += a p; r -= a q; partials of z.r and z.z, z = B r
__global__ __launch_bounds__(KS_BLOCK) void k_pcg_xr(int n, const double *__restrict__ p,
                                                    const double *__restrict__ q, double *__restrict__ x,
                                                    double *__restrict__ r, const double *__restrict__ dinv,
                                                    const ksp_state *in, ksp_state *out,
                                                    const double *__restrict__ pin, int npin,
                                                    double *__restrict__ pout) {
  __shared__ double lin[KS_WAVES][1], lds[KS_WAVES][2];
  ksp_state s;
  load_state(s, in);
  if (s.reason) {
    publish(s, out);
    return;
  }
  double pq[1];
  load_partials<1>(pin, npin, pq);
  all_sum(pq, lin);
  s.sc[S_PQ] = pq[0];
  publish(s, out);
  const double a = s.sc[S_RZ] / pq[0];
  double t[2] = {0.0, 0.0};
  KS_FOR_ROWS(i, n) {
    x[i] += a * p[i];
    const double ri = r[i] - a * q[i], zi = dinv[i] * ri;
    r[i] = ri;
    t[0] += zi * ri;
    t[1] += zi * zi;
  }
  store_partials(t, pout, lds, blockIdx.x);
}

// The first state of a solve (start), or the end of a chunk's last iteration:
// the decision the next product would take, for the host to read
template <bool BCGS>
__global__ __launch_bounds__(KS_BLOCK) void k_ksp_decide(const double *__restrict__ part, int np, const ksp_state *in,
                                                        ksp_state *out, int start, double rtol, double abstol,
                                                        int maxits) {
  __shared__ double lds[KS_WAVES][2];
  ksp_state s = {};
  if (!start) load_state(s, in);
  if (!s.reason) {
    double t[2];
    load_partials<2>(part, np, t);
    all_sum(t, lds);
    if (start) {
      const double rnorm0 = sqrt(BCGS ? t[0] : t[1]);
      s.sc[BCGS ? S_RHO : S_RZ] = t[0];   // BiCGStab: (rhat, r) with rhat = r; CG: z.r
      if (BCGS) s.sc[S_RHOOLD] = s.sc[S_ALPHA] = s.sc[S_OMEGA] = 1.0;
      s.sc[S_RNORM] = rnorm0;
      s.sc[S_TTOL] = fmax(rtol * rnorm0, abstol);
      s.maxits = maxits;
      s.reason = rnorm0 <= s.sc[S_TTOL] ? 1 : 0;
    } else if (BCGS) bcgs_decide(s, t);
    else cg_decide(s, t);
  }
  publish(s, out);
}

// ---------------------------------------------------------------- BiCGStab
// x = 0, r = B b, rhat = r, p = v = 0; partials of r.r
__global__ __launch_bounds__(KS_BLOCK) void k_bcgs_start(int n, const double *__restrict__ b, double *__restrict__ x,
                                                        double *__restrict__ r, double *__restrict__ rh,
                                                        double *__restrict__ p, double *__restrict__ v,
                                                        const double *__restrict__ dinv, double *__restrict__ part) {
  __shared__ double lds[KS_WAVES][2];
  double t[2] = {0.0, 0.0};
  KS_FOR_ROWS(i, n) {
    const double ri = dinv ? dinv[i] * b[i] : b[i];   // no dinv: b holds B b already
    x[i] = 0.0;
    r[i] = ri;
    rh[i] = ri;
    p[i] = 0.0;
    v[i] = 0.0;
    t[0] += ri * ri;
  }
  store_partials(t, part, lds, blockIdx.x);
}

// ILU(0): the sums of a product after B was applied to it: (rhat, y), or
// (w, y) and (y, y) with the (w, w) that the product left in ww
template <int NV>
__global__ __launch_bounds__(KS_BLOCK) void k_bcgs_dots(int n, const double *__restrict__ h,
                                                       const double *__restrict__ y, const ksp_state *S,
                                                       const double *__restrict__ ww, int nww,
                                                       double *__restrict__ part) {
  __shared__ double lds[KS_WAVES][NV];
  if (S->reason) return;
  double t[NV];
#pragma unroll
  for (int j = 0; j < NV; j++) t[j] = 0.0;
  KS_FOR_ROWS(i, n) {
    const double yi = y[i];
    t[0] += h[i] * yi;
    if (NV > 1) t[NV > 1 ? 1 : 0] += yi * yi;
  }
  if (NV > 2)   // the product's partials, dealt to the workgroups
    for (int q = blockIdx.x * KS_BLOCK + threadIdx.x; q < nww; q += gridDim.x * KS_BLOCK)
      t[NV > 2 ? 2 : 0] += ww[3 * q + 2];
  store_partials(t, part, lds, blockIdx.x);
}

// omega = (t, s) / (t, t); x += alpha p + omega s, r = s - omega t (or x += alpha p alone when |s| <= ttol);
// partials of (r, r) and (rhat, r)
__global__ __launch_bounds__(KS_BLOCK) void k_bcgs_x(int n, double *__restrict__ x, const double *__restrict__ p,
                                                    const double *__restrict__ sv, const double *__restrict__ tv,
                                                    double *__restrict__ r, const double *__restrict__ rh,
                                                    const ksp_state *in, ksp_state *out,
                                                    const double *__restrict__ pin, int npin,
                                                    double *__restrict__ pout) {
  __shared__ double lin[KS_WAVES][3], lds[KS_WAVES][2];
  ksp_state s;
  load_state(s, in);
  if (s.reason) {
    publish(s, out);
    return;
  }
  double d[3];
  load_partials<3>(pin, npin, d);
  all_sum(d, lin);
  s.sc[S_SS] = d[2];
  s.sconv = sqrt(d[2]) <= s.sc[S_TTOL] ? 1 : 0;
  if (!s.sconv) {
    if (d[1] == 0.0) s.reason = -5;   // (t, t) = 0
    else s.sc[S_OMEGA] = d[0] / d[1];
  }
  publish(s, out);
  if (s.reason) return;
  const double a = s.sc[S_ALPHA], om = s.sc[S_OMEGA];
  double t[2] = {0.0, 0.0};
  if (s.sconv) {
    KS_FOR_ROWS(i, n) x[i] += a * p[i];
  } else {
    KS_FOR_ROWS(i, n) {
      x[i] += a * p[i] + om * sv[i];
      const double ri = sv[i] - om * tv[i];
      r[i] = ri;
      t[0] += ri * ri;
      t[1] += rh[i] * ri;
    }
  }
  store_partials(t, pout, lds, blockIdx.x);
}

// ---------------------------------------------------------------- ILU(0)
// lu = values of A - sigma I on A's pattern
__global__ __launch_bounds__(KS_BLOCK) void k_ilu0_init(const int32_t *__restrict__ rowptr,
                                                       const int32_t *__restrict__ colidx,
                                                       const double *__restrict__ val, int n, double sigma,
                                                       double *__restrict__ lu) {
  KS_FOR_ROWS(i, n)
    for (int32_t q = rowptr[i]; q < rowptr[i + 1]; q++) lu[q] = val[q] - (colidx[q] == i ? sigma : 0.0);
}

// row i of the IKJ factorization (Saad, Algorithm 10.4); the rows it reads (its
// L part) belong to earlier levels.  The operations of a row are the oracle's,
// in the same order.
__device__ __forceinline__ void ilu0_factor_row(int i, const int32_t *__restrict__ rowptr,
                                               const int32_t *__restrict__ colidx, const int32_t *__restrict__ diag,
                                               double *lu, int *zero_pivot) {
  const int32_t re = rowptr[i + 1];
  for (int32_t q = rowptr[i]; q < diag[i]; q++) {
    const int k = colidx[q];
    const double ukk = lu[diag[k]];
    if (ukk == 0.0) {
      atomicExch(zero_pivot, 1);
      return;
    }
    const double lik = lu[q] / ukk;
    lu[q] = lik;
    int32_t u = diag[k] + 1;
    const int32_t ke = rowptr[k + 1];
    for (int32_t r = q + 1; r < re; r++) {
      const int j = colidx[r];
      while (u < ke && colidx[u] < j) u++;
      if (u < ke && colidx[u] == j) lu[r] -= lik * lu[u];
    }
  }
}

// one level: a thread per row of the level
__global__ __launch_bounds__(64) void k_ilu0_factor_level(const int32_t *__restrict__ rows, int cnt,
                                                         const int32_t *__restrict__ rowptr,
                                                         const int32_t *__restrict__ colidx,
                                                         const int32_t *__restrict__ diag, double *__restrict__ lu,
                                                         int *zero_pivot) {
  const int t = blockIdx.x * 64 + threadIdx.x;
  if (t < cnt) ilu0_factor_row(rows[t], rowptr, colidx, diag, lu, zero_pivot);
}

// Every level in one workgroup, a barrier (which orders its global stores) between
// them: for narrow levels of short rows a launch a level costs more than the level.
// Wider levels, or rows whose chains of merges are long, are better spread over the
// chip.  The whole set-up, a launch a level / one launch: 128 x 127 grid 1.83 / 1.56
// ms, 256 x 255 (levels of up to 255 rows) 4.35 / 4.14, 512 x 511 (511) 10.9 / 11.8,
// tridiagonal 2,000 rows 5.3 / 2.7; nine-point 100 x 100 4.45 / 4.07; seven-point 16^3
// (192) 0.62 / 0.57, 32^3 (768) 1.58 / 1.95; 27-point 40^3 33 / 44; random graphs of 20
// entries a row 9.6 / 10.1.
#define KS_ILU_WG 256        // rows of a level, at most
#define KS_ILU_WG_ROW 9      // entries of a row, at most
__global__ __launch_bounds__(KS_ILU_WG) void k_ilu0_factor(const int32_t *__restrict__ rows,
                                                          const int32_t *__restrict__ lptr, int nlev,
                                                          const int32_t *__restrict__ rowptr,
                                                          const int32_t *__restrict__ colidx,
                                                          const int32_t *__restrict__ diag, double *lu,
                                                          int *zero_pivot) {
  for (int l = 0; l < nlev; l++) {
    const int r = lptr[l] + (int)threadIdx.x;
    if (r < lptr[l + 1]) ilu0_factor_row(rows[r], rowptr, colidx, diag, lu, zero_pivot);
    __syncthreads();
  }
}

// One triangular solve of y = (L U)^-1 y in one launch (LOWER: the unit lower
// factor, forward; else the upper factor, backward), in place, one wavefront per
// row: row i goes to wavefront i (forward) or n-1-i (backward), so a row waits
// only for rows of lower-numbered wavefronts, dispatched before it.  The lanes
// take the row's entries of its factor part (64 at a time), wait until each
// entry's column is solved and load its value; lane order then subtracts them
// in column order, as the oracle's loop does.  A solved value is published as
// two 64-bit words, each a 32-bit half of the double beside the solve's epoch,
// written and polled with agent-scope atomics: a reader takes a value once both
// words carry the current epoch, so no fence is needed.  Waits are bounded
// (KS_ILU_SPIN polls, or sooner once another wait has run out): then bit 1 of
// *err is set and the row goes on, so every row publishes and every wavefront
// exits; the solve reports the failure.  Skipped like the products when the
// solver's state says so (the state is read once, at the start).
#define KS_ILU_SPIN (1 << 26)
template <bool LOWER>
__global__ __launch_bounds__(KS_BLOCK) void k_ilu0_sf(int n, const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ colidx,
                                                     const int32_t *__restrict__ diag, const double *__restrict__ lu,
                                                     double *y, unsigned long long *slot, unsigned epoch, int *err,
                                                     const ksp_state *S) {
  if (S && S->reason) return;
  const int w = blockIdx.x * KS_WAVES + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (w >= n) return;
  const int i = LOWER ? w : n - 1 - w;
  const int q0 = LOWER ? rowptr[i] : diag[i] + 1, q1 = LOWER ? diag[i] : rowptr[i + 1];
  const unsigned long long tag = (unsigned long long)epoch << 32;
  double s = y[i];
  for (int qb = q0; qb < q1; qb += 64) {
    const int q = qb + lane;
    double a = 0.0, v = 0.0;
    if (q < q1) {
      a = lu[q];
      const unsigned long long *sl = slot + 2 * (size_t)colidx[q];
      unsigned long long lo, hi;
      int spins = 0;
      for (;;) {
        lo = __hip_atomic_load(sl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        hi = __hip_atomic_load(sl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((lo >> 32) == epoch && (hi >> 32) == epoch) break;
        // past the bound, or once another wait has run out, the row goes on (and publishes)
        if (++spins > KS_ILU_SPIN || ((spins & 1023) == 0 && (__hip_atomic_load(err, __ATOMIC_RELAXED,
                                                                                  __HIP_MEMORY_SCOPE_AGENT) & 2))) {
          atomicOr(err, 2);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      v = __longlong_as_double((long long)(((hi & 0xffffffffull) << 32) | (lo & 0xffffffffull)));
    }
    const int cnt = q1 - qb < 64 ? q1 - qb : 64;
    for (int t = 0; t < cnt; t++) s -= ks_readlane_f64(a, t) * ks_readlane_f64(v, t);
  }
  const double x = LOWER ? s : s / lu[diag[i]];
  if (lane == 0) {
    y[i] = x;
    const unsigned long long bits = (unsigned long long)__double_as_longlong(x);
    __hip_atomic_store(slot + 2 * (size_t)i, tag | (bits & 0xffffffffull), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(slot + 2 * (size_t)i + 1, tag | (bits >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The same solve by one workgroup, one barrier a level, for dependency graphs
// that are deep and narrow (a grid in natural order).  k_ilu0_sf hands a value
// from row to row through memory, about 1.3 us a level whatever the level's
// width; here the solved values stay in a ring in LDS and a level costs an LDS
// round trip and a barrier.  Rows are laid out in level order, ns to a step and
// each level padded to whole steps (row -1), their entries in E columns of a
// fixed width (absent: coefficient 0 on the ring's zero slot), so every load is
// coalesced and its address known in advance: KS_ILU_PD steps are in flight in
// registers and the barrier waits for LDS only.  Threads past ns repeat the
// step's last row and store nothing.  A row's subtractions keep k_ilu0_sf's
// order, so the results are its bits.
// 128 x 127 five-point grid (254 levels): one application of both factors 673
// us by k_ilu0_sf, 106 us by levels (0.21 us a level).
#define KS_ILU_PD 8
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
template <bool LOWER, int E, int NT>
__global__ __launch_bounds__(NT) void k_ilu0_levels(int nsteps, int ns, int ring, const int32_t *__restrict__ rowid,
                                                   const int32_t *__restrict__ dep, const double *__restrict__ coef,
                                                   const double *__restrict__ dg, double *y, const ksp_state *S) {
  if (S && S->reason) return;
  extern __shared__ double xs[];   // ring values, then the zero slot
  const int t = threadIdx.x, ts = min(t, ns - 1);
  const bool own = t < ns;
  const int np = nsteps * ns;      // at most KS_ILU_PAD times n
  if (t == 0) xs[ring] = 0.0;
  int rnext[KS_ILU_PD], r[KS_ILU_PD], d[KS_ILU_PD][E];
  double c[KS_ILU_PD][E], b[KS_ILU_PD], g[KS_ILU_PD];
  auto at = [&](int s) { return min(s, nsteps - 1) * ns + ts; };
  auto load = [&](int j, int s) {   // step s into slot j; its rows were loaded KS_ILU_PD steps before
    const int p = at(s);
    r[j] = rnext[j];
    b[j] = y[max(r[j], 0)];
#pragma unroll
    for (int e = 0; e < E; e++) {
      d[j][e] = dep[e * np + p];
      c[j][e] = coef[e * np + p];
    }
    if (!LOWER) g[j] = dg[p];
    rnext[j] = rowid[at(s + KS_ILU_PD)];
  };
#pragma unroll
  for (int j = 0; j < KS_ILU_PD; j++) rnext[j] = rowid[at(j)];
#pragma unroll
  for (int j = 0; j < KS_ILU_PD; j++) load(j, j);
  lds_barrier();
  for (int s0 = 0; s0 < nsteps; s0 += KS_ILU_PD) {
#pragma unroll
    for (int j = 0; j < KS_ILU_PD; j++) {
      const int s = s0 + j;
      if (s >= nsteps) break;
      double v[E], x = b[j];
#pragma unroll
      for (int e = 0; e < E; e++) v[e] = xs[d[j][e]];
#pragma unroll
      for (int e = 0; e < E; e++) x -= c[j][e] * v[e];
      if (!LOWER) x /= g[j];
      if (own) {
        xs[(s * ns + t) & (ring - 1)] = x;
        if (r[j] >= 0) y[r[j]] = x;
      }
      load(j, s + KS_ILU_PD);
      lds_barrier();
    }
  }
}

// coef[e][p] = the factor entry behind slot (e, p), dg[p] = its row's pivot
__global__ __launch_bounds__(KS_BLOCK) void k_ilu0_pack(int np, int E, const int32_t *__restrict__ src,
                                                       const int32_t *__restrict__ rowid,
                                                       const int32_t *__restrict__ diag,
                                                       const double *__restrict__ lu, double *__restrict__ coef,
                                                       double *__restrict__ dg) {
  KS_FOR_ROWS(p, np) {
    for (int e = 0; e < E; e++) {
      const int q = src[(size_t)e * np + p];
      coef[(size_t)e * np + p] = q >= 0 ? lu[q] : 0.0;
    }
    dg[p] = rowid[p] >= 0 ? lu[diag[rowid[p]]] : 1.0;
  }
}

inline int ksp_blocks(int n) {
  int b = (n + KS_BLOCK - 1) / KS_BLOCK;
  if (b > KS_PCG_BLOCKS) b = KS_PCG_BLOCKS;
  return b < 1 ? 1 : b;
}

// iterations enqueued between two reads of the solver state: a read costs the
// stream about 12 us, a launch after the solve's end about 2 us
inline int ksp_chunk(int done) { return std::min(64, std::max(8, done / 4)); }

// waits for the stream, then the iteration count, the outcome and |B r|
static int read_state(ks_ctx ctx, const ksp_state *S, int *its, int *reason, double *rnorm) {
  ksp_state h;
  KS_HIP(hipMemcpyAsync(ctx->h_scalar, S, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
  KS_HIP(hipStreamSynchronize(ctx->stream));
  std::memcpy(&h, ctx->h_scalar, sizeof(h));
  *its = h.its;
  *reason = h.reason;
  *rnorm = h.sc[S_RNORM];
  return KS_OK;
}

// the two states and the partial sums of a solve: a kernel that moves the state
// on reads in() and writes out(), then step()
struct ksp_run {
  ks_ctx ctx;
  ksp_state *S;
  double *part;        // 3 regions, used in turn
  int cur = 0, nb = 0, nprod = 0;
  const ksp_state *in() const { return S + cur; }
  ksp_state *out() const { return S + (cur ^ 1); }
  void step() { cur ^= 1; }
  double *region(int k) const { return part + (size_t)k * 3 * KS_KSP_SPMV_BLOCKS; }
};

inline ksp_run ksp_begin(ks_ctx ctx, ks_csr A, double *state, int nb) {
  static_assert(9 * KS_KSP_SPMV_BLOCKS <= (size_t)KS_MAXB * KS_NCOLP, "partials exceed the workspace");
  static_assert(KS_PCG_BLOCKS <= KS_KSP_SPMV_BLOCKS, "a region holds three sums of every workgroup");
  ksp_run R;
  R.ctx = ctx;
  R.S = (ksp_state *)state;
  R.part = ctx->d_partial;
  R.nb = nb;
  R.nprod = std::min(A->nblocks, KS_KSP_SPMV_BLOCKS);
  return R;
}

// Products of up to this many entries form their vector as they gather it, one
// launch fewer; beyond, the two or three gathers an entry cost more than the
// launch.  us an iteration, formed inside / by itself: CG 256 x 255 grid (325,000
// entries) 10.8 / 12.2, random graph of 900,000 entries 24.6 / 18.5, 512 x 511 grid
// (1.3 million) 19.5 / 18.3; BiCGStab 16.6 / 20.2, 40.5 / 29.9, 30.8 / 31.6; CG on
// 2048 x 2047 (21 million) 186 / 154.
#define KS_KSP_FUSE_NNZ 500000
template <int MODE, bool PC>
void ksp_product(ksp_run &R, ks_csr A, double sigma, const double *r, const double *p, const double *v,
                 const double *rh, const double *dinv, double *w, double *y, int kin, int npin, int decide, int kout) {
  const double n = A->nrows;
  const bool fuse = A->nnz <= KS_KSP_FUSE_NNZ;
  ksp_prod a = {A->d_blk, A->d_rowptr, A->d_colidx, (const double *)A->d_val, A->nblocks, A->nrows, r, p, v, rh, dinv,
                w, y, sigma, R.in(), R.out(), R.region(kin), npin, decide, R.region(kout)};
  if (!fuse) {
    hipLaunchKernelGGL(k_ksp_vector<MODE>, dim3(R.nb), dim3(KS_BLOCK), 0, R.ctx->stream, a);
    a.in = R.out();
  }
  ks_prof_begin(R.ctx, KS_PROF_SPMV, (double)A->nnz * 12.0 + (n + 1.0) * 4.0 + 8.0 * n * (fuse ? 5.0 : 2.0),
                2.0 * (double)A->nnz, false);
  if (fuse)
    hipLaunchKernelGGL((k_ksp_product<MODE, PC, true>), dim3(R.nprod), dim3(KS_BLOCK), 0, R.ctx->stream, a);
  else
    hipLaunchKernelGGL((k_ksp_product<MODE, PC, false>), dim3(R.nprod), dim3(KS_BLOCK), 0, R.ctx->stream, a);
  ks_prof_end(R.ctx);
  R.step();
}

}  // namespace

struct ks_ilu_s {
  int n = 0;
  std::vector<int> lptr, uptr;        // level starts (host): the factorization's schedule; the
                                      // backward solve's depth (ks_ilu0_levels)
  int32_t *d_lrows = nullptr, *d_diag = nullptr;
  double *d_lu = nullptr;
  int *d_flag = nullptr;              // bit 0: a zero pivot; bit 1: a solve's wait ran out
  unsigned long long *d_slot = nullptr;   // [n][2] published values of the triangular solves
  unsigned epoch = 0;
  const int32_t *d_rowptr = nullptr, *d_colidx = nullptr;   // the operator's pattern (borrowed)
  // one factor in level order for k_ilu0_levels (nsteps 0: k_ilu0_sf takes it)
  struct lvl {
    int nsteps = 0, ns = 0, nt = 0, E = 0, ring = 0;
    size_t np() const { return (size_t)nsteps * ns; }   // slots
    size_t nidx() const { return np() * (2 * E + 1); }
    size_t nval() const { return np() * (E + 1); }
    int32_t *d_idx = nullptr;      // rowid[np], dep[E][np], src[E][np]
    double *d_val = nullptr;       // dg[np], then coef[E][np]
  } lo, up;
  int32_t *d_lvl = nullptr;        // both layouts' d_idx
};

namespace {

#define KS_ILU_EMAX 4          // entries a row in the level-ordered layout
#define KS_ILU_RING 16384      // solved values held in LDS (128 KB), at most

template <bool LOWER, int E, int NT>
void launch_levels(ks_ctx ctx, const ks_ilu_s::lvl &L, double *y, const ksp_state *S) {
  const size_t np = L.np();
  hipLaunchKernelGGL((k_ilu0_levels<LOWER, E, NT>), dim3(1), dim3(NT), sizeof(double) * (L.ring + 1), ctx->stream,
                     L.nsteps, L.ns, L.ring, (const int32_t *)L.d_idx, (const int32_t *)L.d_idx + np,
                     (const double *)L.d_val + np, (const double *)L.d_val, y, S);
}
template <bool LOWER>
void apply_levels(ks_ctx ctx, const ks_ilu_s::lvl &L, double *y, const ksp_state *S) {
#define KS_ILU_NT(X)                                           \
  case X:                                                      \
    if (L.E == 2) launch_levels<LOWER, 2, X>(ctx, L, y, S);    \
    else launch_levels<LOWER, 4, X>(ctx, L, y, S);             \
    break;
  switch (L.nt) {
    KS_ILU_NT(64) KS_ILU_NT(128) KS_ILU_NT(256) KS_ILU_NT(512)
    default: launch_levels<LOWER, 2, 1024>(ctx, L, y, S);   // leaves 128 VGPRs, enough for two entries a row
  }
#undef KS_ILU_NT
}

// y = (L U)^-1 y on the context stream: two launches, the forward and the
// backward solve, by levels where the factors have that layout, else each a
// new epoch of the published values
void ilu0_apply(ks_ctx ctx, ks_ilu M, double *y, const ksp_state *S) {
  const int blocks = (M->n + KS_WAVES - 1) / KS_WAVES;
  if (M->lo.nsteps && M->up.nsteps) {
    apply_levels<true>(ctx, M->lo, y, S);
    apply_levels<false>(ctx, M->up, y, S);
    return;
  }
  M->epoch += 1;
  hipLaunchKernelGGL(k_ilu0_sf<true>, dim3(blocks), dim3(KS_BLOCK), 0, ctx->stream, M->n, M->d_rowptr,
                     M->d_colidx, (const int32_t *)M->d_diag, (const double *)M->d_lu, y, M->d_slot, M->epoch,
                     M->d_flag, S);
  M->epoch += 1;
  hipLaunchKernelGGL(k_ilu0_sf<false>, dim3(blocks), dim3(KS_BLOCK), 0, ctx->stream, M->n, M->d_rowptr,
                     M->d_colidx, (const int32_t *)M->d_diag, (const double *)M->d_lu, y, M->d_slot, M->epoch,
                     M->d_flag, S);
}

// rows grouped by level (stable in row order) and the level starts
void group_levels(const std::vector<int> &lev, std::vector<int32_t> &rows, std::vector<int> &ptr) {
  int nl = 0;
  for (int v : lev) nl = v + 1 > nl ? v + 1 : nl;
  ptr.assign(nl + 1, 0);
  for (int v : lev) ptr[v + 1]++;
  for (int l = 0; l < nl; l++) ptr[l + 1] += ptr[l];
  std::vector<int> fill(ptr.begin(), ptr.end() - 1);
  rows.resize(lev.size());
  for (size_t i = 0; i < lev.size(); i++) rows[fill[lev[i]]++] = (int32_t)i;
}

// The level-ordered layout of one factor (entries q0(i) .. q1(i)-1 of row i),
// appended to idx: which row, which ring slots and which factor entries stand in
// every slot.  A step holds the widest level, up to what a workgroup takes, but
// is halved while the padding of narrower levels makes more than KS_ILU_PAD slots a
// row: a slot takes 44 or 76 bytes, and steps of at least 256 rows whatever the
// levels took 22 GB for a tridiagonal matrix of 1,000,000 rows.  Returns false, and
// the factors keep k_ilu0_sf, where a row has more than KS_ILU_EMAX entries, a
// dependency lies further back than the ring, or the levels are so wide that the
// steps outnumber them KS_ILU_STEPS times (k_ilu0_sf has the whole chip for them).
// A BiCGStab iteration (four triangular solves), k_ilu0_sf / by levels: five-point
// grids 64 x 63 592 / 118 us, 128 x 127 1449 / 236, 256 x 255 7.1 / 0.82 ms, 512 x
// 511 48.9 / 3.0 ms; seven-point grids 16^3 283 / 97 us, 64^3 (levels 1380 rows wide
// on average) 10.7 / 2.9 ms; a tridiagonal matrix of 20,000 rows 84.8 / 16.6 ms.
#define KS_ILU_STEPS 4
#define KS_ILU_PAD 4
template <typename Q0, typename Q1>
bool level_layout(int n, const std::vector<int32_t> &rows, const std::vector<int> &ptr, const int32_t *ci, Q0 q0, Q1 q1,
                  ks_ilu_s::lvl &L, std::vector<int32_t> &idx) {
  const int nl = (int)ptr.size() - 1;
  int emax = 0, wmax = 0;
  for (int i = 0; i < n; i++) emax = std::max(emax, (int)(q1(i) - q0(i)));
  for (int l = 0; l < nl; l++) wmax = std::max(wmax, ptr[l + 1] - ptr[l]);
  if (emax > KS_ILU_EMAX) return false;
  const int E = emax <= 2 ? 2 : KS_ILU_EMAX, ntmax = E > 2 ? 512 : 1024;
  int ns = 1;
  while (ns < wmax && ns < ntmax) ns *= 2;
  auto count = [&](int w) {
    int64_t k = 0;
    for (int l = 0; l < nl; l++) k += (ptr[l + 1] - ptr[l] + w - 1) / w;
    return k;
  };
  int64_t steps = count(ns);
  while (steps * ns > KS_ILU_PAD * (int64_t)n) steps = count(ns /= 2);   // one row a step: n slots
  if (steps > (int64_t)KS_ILU_STEPS * nl || steps * ns * E >= (1 << 29)) return false;
  const int np = (int)steps * ns;
  std::vector<int> pos(n);
  const size_t at = idx.size();
  idx.resize(at + (size_t)np * (2 * E + 1), -1);
  int32_t *id = idx.data() + at, *dep = id + np, *src = dep + (size_t)np * E;
  int s = 0, ring = 64;
  while (ring < ns) ring *= 2;
  for (int l = 0; l < nl; l++) {
    for (int k = ptr[l]; k < ptr[l + 1]; k++) {
      const int i = rows[k], p = s * ns + (k - ptr[l]), end = (p / ns + 1) * ns;
      pos[i] = p;
      id[p] = i;
      size_t e = p;
      for (int32_t q = q0(i); q < q1(i); q++, e += np) {
        const int back = end - pos[ci[q]];   // slots written from the entry's value to the end of this step
        while (ring < back && ring <= KS_ILU_RING) ring *= 2;
        if (ring > KS_ILU_RING) return false;
        dep[e] = pos[ci[q]];
        src[e] = q;
      }
    }
    s += (ptr[l + 1] - ptr[l] + ns - 1) / ns;
  }
  for (size_t k = 0; k < (size_t)np * E; k++) dep[k] = dep[k] < 0 ? ring : (dep[k] & (ring - 1));
  L.nsteps = (int)steps;
  L.ns = ns;
  L.nt = std::max(ns, 64);
  L.E = E;
  L.ring = ring;
  return true;
}

// the diagonal entries of a pattern whose rows list increasing columns
int find_diagonals(int n, const int32_t *rp, const int32_t *ci, int32_t *diag) {
  for (int i = 0; i < n; i++) {
    diag[i] = -1;
    for (int32_t q = rp[i]; q < rp[i + 1]; q++) {
      KS_CHECK((q == rp[i] || ci[q] > ci[q - 1]) && ci[q] >= 0 && ci[q] < n, KS_ERR_ARG,
               "ILU(0) needs increasing column indices (row %d)", i);
      if (ci[q] == i) diag[i] = q;
    }
    KS_CHECK(diag[i] >= 0, KS_ERR_ARG, "ILU(0) needs the diagonal entry of row %d", i);
  }
  return KS_OK;
}

// the rows by level and the level starts: forward (row i after the rows of its L
// part) or backward (after its U part)
void factor_levels(bool lower, int n, const int32_t *rp, const int32_t *ci, const int32_t *diag, std::vector<int> &lev,
                   std::vector<int32_t> &rows, std::vector<int> &ptr) {
  lev.assign(n, 0);
  if (lower) {
    for (int i = 0; i < n; i++)
      for (int32_t q = rp[i]; q < diag[i]; q++) lev[i] = std::max(lev[i], lev[ci[q]] + 1);
  } else {
    for (int i = n - 1; i >= 0; i--)
      for (int32_t q = diag[i] + 1; q < rp[i + 1]; q++) lev[i] = std::max(lev[i], lev[ci[q]] + 1);
  }
  group_levels(lev, rows, ptr);
}

bool factor_layout(bool lower, int n, const int32_t *rp, const int32_t *ci, const int32_t *diag,
                   const std::vector<int32_t> &rows, const std::vector<int> &ptr, ks_ilu_s::lvl &L,
                   std::vector<int32_t> &idx) {
  if (lower)
    return level_layout(n, rows, ptr, ci, [&](int i) { return rp[i]; }, [&](int i) { return diag[i]; }, L, idx);
  return level_layout(n, rows, ptr, ci, [&](int i) { return diag[i] + 1; }, [&](int i) { return rp[i + 1]; }, L, idx);
}

// Uploads both layouts and packs the factors' values.  KS_ERR_NOMEM where there is no
// room for them: then nothing is held or enqueued.
int levels_pack(ks_ctx ctx, ks_ilu M, const std::vector<int32_t> &idx) {
  int e = ks_malloc((void **)&M->d_lvl, sizeof(int32_t) * idx.size());
  if (!e) e = ks_malloc((void **)&M->lo.d_val, sizeof(double) * (M->lo.nval() + M->up.nval()));
  if (e) {
    if (M->d_lvl) (void)ks_free(M->d_lvl);
    M->d_lvl = nullptr;
    return e;
  }
  KS_HIP(hipMemcpyAsync(M->d_lvl, idx.data(), sizeof(int32_t) * idx.size(), hipMemcpyHostToDevice, ctx->stream));
  M->lo.d_idx = M->d_lvl;
  M->up.d_idx = M->d_lvl + M->lo.nidx();
  M->up.d_val = M->lo.d_val + M->lo.nval();
  for (ks_ilu_s::lvl *L : {&M->lo, &M->up}) {
    const int np = (int)L->np();
    hipLaunchKernelGGL(k_ilu0_pack, dim3(ksp_blocks(np)), dim3(KS_BLOCK), 0, ctx->stream, np, L->E,
                       (const int32_t *)L->d_idx + (size_t)np * (L->E + 1), (const int32_t *)L->d_idx,
                       (const int32_t *)M->d_diag, (const double *)M->d_lu, L->d_val + np, L->d_val);
  }
  KS_HIP(hipGetLastError());
  return KS_OK;
}

}  // namespace

int ks_ilu0_create(ks_ctx ctx, ks_csr A, double sigma, ks_ilu *out) {
  KS_CHECK(ctx && A && out, KS_ERR_ARG, "null ILU argument");
  KS_CHECK(A->vprec == KS_F64 && A->nrows == A->ncols, KS_ERR_ARG, "ILU(0) needs a square FP64 matrix");
  *out = nullptr;
  const int n = A->nrows;
  const int64_t nnz = A->nnz;
  std::vector<int32_t> rp(n + 1), ci(nnz), diag(n);
  KS_HIP(hipMemcpyAsync(rp.data(), A->d_rowptr, sizeof(int32_t) * (n + 1), hipMemcpyDeviceToHost, ctx->stream));
  KS_HIP(hipMemcpyAsync(ci.data(), A->d_colidx, sizeof(int32_t) * nnz, hipMemcpyDeviceToHost, ctx->stream));
  KS_HIP(hipStreamSynchronize(ctx->stream));
  KS_TRY(find_diagonals(n, rp.data(), ci.data(), diag.data()));
  std::vector<int> lev;
  std::vector<int32_t> lrows, urows;
  ks_ilu M = new ks_ilu_s();
  M->n = n;
  M->d_rowptr = A->d_rowptr;
  M->d_colidx = A->d_colidx;
  factor_levels(true, n, rp.data(), ci.data(), diag.data(), lev, lrows, M->lptr);
  factor_levels(false, n, rp.data(), ci.data(), diag.data(), lev, urows, M->uptr);
  int e = KS_OK;
  // the rows by level and the level starts
  lrows.insert(lrows.end(), M->lptr.begin(), M->lptr.end());
  if (!e) e = ks_malloc((void **)&M->d_lrows, sizeof(int32_t) * lrows.size());
  if (!e) e = ks_malloc((void **)&M->d_diag, sizeof(int32_t) * n);
  if (!e) e = ks_malloc((void **)&M->d_lu, sizeof(double) * (nnz > 0 ? nnz : 1));
  if (!e) e = ks_malloc((void **)&M->d_flag, sizeof(int));
  if (!e) e = ks_malloc((void **)&M->d_slot, sizeof(unsigned long long) * 2 * (size_t)n);
  if (!e) e = ks_memset_zero(ctx, M->d_slot, sizeof(unsigned long long) * 2 * (size_t)n);
  if (e) {
    ks_ilu0_destroy(M);
    return e;
  }
  hipStream_t st = ctx->stream;
  KS_HIP(hipMemcpyAsync(M->d_lrows, lrows.data(), sizeof(int32_t) * lrows.size(), hipMemcpyHostToDevice, st));
  KS_HIP(hipMemcpyAsync(M->d_diag, diag.data(), sizeof(int32_t) * n, hipMemcpyHostToDevice, st));
  KS_TRY(ks_memset_zero(ctx, M->d_flag, sizeof(int)));
  hipLaunchKernelGGL(k_ilu0_init, dim3(ksp_blocks(n)), dim3(KS_BLOCK), 0, st, A->d_rowptr, A->d_colidx,
                     (const double *)A->d_val, n, sigma, M->d_lu);
  const int nlev = (int)M->lptr.size() - 1;
  int wmax = 0, emax = 0;
  for (int l = 0; l < nlev; l++) wmax = std::max(wmax, M->lptr[l + 1] - M->lptr[l]);
  for (int i = 0; i < n; i++) emax = std::max(emax, rp[i + 1] - rp[i]);
  if (wmax <= KS_ILU_WG && emax <= KS_ILU_WG_ROW) {
    hipLaunchKernelGGL(k_ilu0_factor, dim3(1), dim3(KS_ILU_WG), 0, st, (const int32_t *)M->d_lrows,
                       (const int32_t *)M->d_lrows + n, nlev, A->d_rowptr, A->d_colidx, (const int32_t *)M->d_diag,
                       M->d_lu, M->d_flag);
  } else {
    for (int l = 0; l < nlev; l++) {
      const int cnt = M->lptr[l + 1] - M->lptr[l];
      hipLaunchKernelGGL(k_ilu0_factor_level, dim3((cnt + 63) / 64), dim3(64), 0, st,
                         (const int32_t *)M->d_lrows + M->lptr[l], cnt, A->d_rowptr, A->d_colidx,
                         (const int32_t *)M->d_diag, M->d_lu, M->d_flag);
    }
  }
  KS_HIP(hipGetLastError());
  // The level-ordered layouts, made while the device factors; without room for them,
  // here or on the device, the rows wait for each other (k_ilu0_sf)
  std::vector<int32_t> idx;
  bool by_levels = false;
  try {
    by_levels = factor_layout(true, n, rp.data(), ci.data(), diag.data(), lrows, M->lptr, M->lo, idx) &&
                factor_layout(false, n, rp.data(), ci.data(), diag.data(), urows, M->uptr, M->up, idx);
  } catch (const std::bad_alloc &) {
  }
  if (by_levels) {
    e = levels_pack(ctx, M, idx);
    if (e && e != KS_ERR_NOMEM) {
      (void)hipStreamSynchronize(st);
      ks_ilu0_destroy(M);
      return e;
    }
    by_levels = !e;
  }
  if (!by_levels) M->lo.nsteps = M->up.nsteps = 0;
  // the last pivot, and a zero pivot met on the way
  int flag = 0;
  double ulast = 0.0;
  KS_HIP(hipMemcpyAsync(&flag, M->d_flag, sizeof(int), hipMemcpyDeviceToHost, st));
  KS_HIP(hipMemcpyAsync(&ulast, M->d_lu + diag[n - 1], sizeof(double), hipMemcpyDeviceToHost, st));
  KS_HIP(hipStreamSynchronize(st));
  if (flag || ulast == 0.0) {
    fprintf(stderr, "ks_hip: ILU(0) met a zero pivot\n");
    ks_ilu0_destroy(M);
    return KS_ERR_PIVOT;
  }
  *out = M;
  return KS_OK;
}

int ks_ilu0_destroy(ks_ilu M) {
  if (!M) return KS_OK;
  if (M->d_lrows) (void)ks_free(M->d_lrows);
  if (M->d_slot) (void)ks_free(M->d_slot);
  if (M->d_diag) (void)ks_free(M->d_diag);
  if (M->d_lu) (void)ks_free(M->d_lu);
  if (M->d_flag) (void)ks_free(M->d_flag);
  if (M->d_lvl) (void)ks_free(M->d_lvl);
  if (M->lo.d_val) (void)ks_free(M->lo.d_val);
  delete M;
  return KS_OK;
}

int ks_ilu0_layout(int n, const int32_t *rowptr, const int32_t *colidx, int lower, ks_ilu_layout *out) {
  KS_CHECK(n > 0 && rowptr && colidx && out && rowptr[0] == 0, KS_ERR_ARG, "bad ILU layout arguments");
  *out = ks_ilu_layout{};
  try {
    std::vector<int32_t> diag(n), rows, idx;
    std::vector<int> lev, ptr;
    ks_ilu_s::lvl L;
    KS_TRY(find_diagonals(n, rowptr, colidx, diag.data()));
    factor_levels(lower != 0, n, rowptr, colidx, diag.data(), lev, rows, ptr);
    if (!factor_layout(lower != 0, n, rowptr, colidx, diag.data(), rows, ptr, L, idx)) return KS_OK;
    out->step = L.ns;
    out->threads = L.nt;
    out->entries = L.E;
    out->ring = L.ring;
    out->bytes = (int64_t)(sizeof(int32_t) * L.nidx() + sizeof(double) * L.nval());
  } catch (const std::bad_alloc &) {
    return KS_ERR_NOMEM;
  }
  return KS_OK;
}

int ks_ilu0_levels(ks_ilu M, int *nlower, int *nupper) {
  KS_CHECK(M && nlower && nupper, KS_ERR_ARG, "null argument");
  *nlower = (int)M->lptr.size() - 1;
  *nupper = (int)M->uptr.size() - 1;
  return KS_OK;
}

int ks_pcg_jacobi(ks_ctx ctx, ks_csr A, double sigma, int jacobi, double *d_dinv) {
  KS_CHECK(ctx && A && d_dinv, KS_ERR_ARG, "null argument");
  KS_CHECK(A->vprec == KS_F64 && A->nrows == A->ncols, KS_ERR_ARG, "the inner solve needs a square FP64 matrix");
  hipLaunchKernelGGL(k_jacobi, dim3(ksp_blocks(A->nrows)), dim3(KS_BLOCK), 0, ctx->stream, A->d_rowptr, A->d_colidx,
                     (const double *)A->d_val, A->nrows, sigma, jacobi, d_dinv);
  KS_HIP(hipGetLastError());
  return KS_OK;
}

int ks_pcg_solve(ks_ctx ctx, ks_csr A, double sigma, const double *d_dinv, const double *d_b, double *d_x,
                 double rtol, double abstol, int maxits, double *d_work, int *its, double *rnorm, int *reason) {
  KS_CHECK(ctx && A && d_dinv && d_b && d_x && d_work && its && rnorm && reason, KS_ERR_ARG, "null PCG argument");
  KS_CHECK(A->vprec == KS_F64 && A->nrows == A->ncols, KS_ERR_ARG, "PCG needs a square FP64 matrix");
  KS_CHECK(maxits > 0, KS_ERR_ARG, "PCG needs maxits > 0");
  const int n = A->nrows, nb = ksp_blocks(n);
  double *r = d_work, *p = r + n, *pn = p + n, *q = pn + n;
  ksp_run R = ksp_begin(ctx, A, q + n, nb);
  hipStream_t st = ctx->stream;
  const dim3 g(nb), b1(KS_BLOCK), one(1);
  hipLaunchKernelGGL(k_pcg_start, g, b1, 0, st, n, d_b, d_x, r, d_dinv, R.region(0));
  hipLaunchKernelGGL(k_ksp_decide<false>, one, b1, 0, st, (const double *)R.region(0), nb, R.in(), R.out(), 1, rtol,
                     abstol, maxits);
  R.step();
  for (int done = 0;;) {
    KS_TRY(read_state(ctx, R.in(), its, reason, rnorm));
    if (*reason || done >= maxits) break;
    const int chunk = ksp_chunk(done);
    for (int c = 0; c < chunk; c++) {
      ksp_product<KSP_CG, true>(R, A, sigma, r, p, nullptr, nullptr, d_dinv, pn, q, 0, nb, c > 0, 1);
      hipLaunchKernelGGL(k_pcg_xr, g, b1, 0, st, n, (const double *)pn, (const double *)q, d_x, r, d_dinv, R.in(),
                         R.out(), (const double *)R.region(1), R.nprod, R.region(0));
      R.step();
      std::swap(p, pn);
    }
    hipLaunchKernelGGL(k_ksp_decide<false>, one, b1, 0, st, (const double *)R.region(0), nb, R.in(), R.out(), 0, rtol,
                       abstol, maxits);
    R.step();
    KS_HIP(hipGetLastError());
    done += chunk;
  }
  if (!*reason) *reason = -3;   // KSP_DIVERGED_ITS
  return KS_OK;
}

namespace {

// BiCGStab with B = diag(d_dinv) (ilu null) or B = (L U)^-1 (ilu).  The six
// vectors of the workspace: r and rhat keep their places; p and v are formed
// from their old values into two others, which s and t then take back, so the
// pairs change places every iteration.
int bcgs_solve(ks_ctx ctx, ks_csr A, double sigma, const double *d_dinv, const ks_ilu ilu, const double *d_b,
               double *d_x, double rtol, double abstol, int maxits, double *d_work, int *its, double *rnorm,
               int *reason) {
  KS_CHECK(maxits > 0, KS_ERR_ARG, "BiCGStab needs maxits > 0");
  const int n = A->nrows, nb = ksp_blocks(n);
  double *r = d_work, *rh = r + n, *p = rh + n, *v = p + n, *sv = v + n, *t = sv + n;
  ksp_run R = ksp_begin(ctx, A, t + n, nb);
  hipStream_t st = ctx->stream;
  const dim3 g(nb), b1(KS_BLOCK), one(1);
  if (ilu) {
    KS_TRY(ks_memcpy_dtod(ctx, r, d_b, sizeof(double) * n));
    ilu0_apply(ctx, ilu, r, nullptr);                                                // r = B b
    hipLaunchKernelGGL(k_bcgs_start, g, b1, 0, st, n, (const double *)r, d_x, r, rh, p, v, (const double *)nullptr,
                       R.region(0));
  } else {
    hipLaunchKernelGGL(k_bcgs_start, g, b1, 0, st, n, d_b, d_x, r, rh, p, v, d_dinv, R.region(0));
  }
  hipLaunchKernelGGL(k_ksp_decide<true>, one, b1, 0, st, (const double *)R.region(0), nb, R.in(), R.out(), 1, rtol,
                     abstol, maxits);
  R.step();
  for (int done = 0;;) {
    KS_TRY(read_state(ctx, R.in(), its, reason, rnorm));
    if (*reason || done >= maxits) break;
    const int chunk = ksp_chunk(done);
    for (int c = 0; c < chunk; c++) {
      double *pn = sv, *vn = t, *sn = p, *tn = v;
      if (ilu) {
        ksp_product<KSP_P, false>(R, A, sigma, r, p, v, rh, nullptr, pn, vn, 0, nb, c > 0, 1);
        ilu0_apply(ctx, ilu, vn, R.in());                                            // v = B (A - sigma I) p
        hipLaunchKernelGGL(k_bcgs_dots<1>, g, b1, 0, st, n, (const double *)rh, (const double *)vn, R.in(),
                           (const double *)nullptr, 0, R.region(1));
        ksp_product<KSP_S, false>(R, A, sigma, r, nullptr, vn, nullptr, nullptr, sn, tn, 1, nb, 0, 2);
        ilu0_apply(ctx, ilu, tn, R.in());                                            // t = B (A - sigma I) s
        hipLaunchKernelGGL(k_bcgs_dots<3>, g, b1, 0, st, n, (const double *)sn, (const double *)tn, R.in(),
                           (const double *)R.region(2), R.nprod, R.region(1));
        hipLaunchKernelGGL(k_bcgs_x, g, b1, 0, st, n, d_x, (const double *)pn, (const double *)sn, (const double *)tn,
                           r, (const double *)rh, R.in(), R.out(), (const double *)R.region(1), nb, R.region(0));
      } else {
        ksp_product<KSP_P, true>(R, A, sigma, r, p, v, rh, d_dinv, pn, vn, 0, nb, c > 0, 1);
        ksp_product<KSP_S, true>(R, A, sigma, r, nullptr, vn, nullptr, d_dinv, sn, tn, 1, R.nprod, 0, 2);
        hipLaunchKernelGGL(k_bcgs_x, g, b1, 0, st, n, d_x, (const double *)pn, (const double *)sn, (const double *)tn,
                           r, (const double *)rh, R.in(), R.out(), (const double *)R.region(2), R.nprod, R.region(0));
      }
      R.step();
      sv = sn;
      t = tn;
      p = pn;
      v = vn;
    }
    hipLaunchKernelGGL(k_ksp_decide<true>, one, b1, 0, st, (const double *)R.region(0), nb, R.in(), R.out(), 0, rtol,
                       abstol, maxits);
    R.step();
    KS_HIP(hipGetLastError());
    done += chunk;
  }
  if (!*reason) *reason = -3;
  return KS_OK;
}

}  // namespace

int ks_bcgs_solve(ks_ctx ctx, ks_csr A, double sigma, const double *d_dinv, const double *d_b, double *d_x,
                  double rtol, double abstol, int maxits, double *d_work, int *its, double *rnorm, int *reason) {
  KS_CHECK(ctx && A && d_dinv && d_b && d_x && d_work && its && rnorm && reason, KS_ERR_ARG,
           "null BiCGStab argument");
  KS_CHECK(A->vprec == KS_F64 && A->nrows == A->ncols, KS_ERR_ARG, "BiCGStab needs a square FP64 matrix");
  return bcgs_solve(ctx, A, sigma, d_dinv, nullptr, d_b, d_x, rtol, abstol, maxits, d_work, its, rnorm, reason);
}

int ks_bcgs_solve_ilu(ks_ctx ctx, ks_csr A, double sigma, ks_ilu M, const double *d_b, double *d_x, double rtol,
                      double abstol, int maxits, double *d_work, int *its, double *rnorm, int *reason) {
  KS_CHECK(ctx && A && M && d_b && d_x && d_work && its && rnorm && reason, KS_ERR_ARG,
           "null BiCGStab argument");
  KS_CHECK(A->vprec == KS_F64 && A->nrows == A->ncols && M->n == A->nrows, KS_ERR_ARG,
           "BiCGStab with ILU(0) needs the square FP64 matrix the factors were made from");
  KS_CHECK(M->d_rowptr == A->d_rowptr, KS_ERR_ARG, "the ILU(0) factors belong to another matrix");
  const int e = bcgs_solve(ctx, A, sigma, nullptr, M, d_b, d_x, rtol, abstol, maxits, d_work, its, rnorm, reason);
  if (e) return e;
  // the triangular solves' waits all met (bit 1 of the flag word); the solve has synchronized
  int flag = 0;
  KS_HIP(hipMemcpyAsync(&flag, M->d_flag, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  KS_HIP(hipStreamSynchronize(ctx->stream));
  KS_CHECK(!(flag & 2), KS_ERR_TIMEOUT, "an ILU(0) triangular solve's wait ran out of polls");
  return KS_OK;
}
