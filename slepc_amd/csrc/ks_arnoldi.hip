// ks_arnoldi.hip -- a whole Arnoldi/Lanczos expansion of a small problem in one launch.
//
// Column by column the expansion of BVMatArnoldi / BVMatLanczos
// (src/sys/classes/bv/interface/bvkrylov.c:88-97) is seven dependent launches of 4-6
// us each, whatever the size: the product, the dots, two fused DGKS passes and
// their three finishes.  Here the workgroups stay: workgroup b owns the rows of the
// matrix' row block b (at most 256) for the whole expansion, and the workgroups
// exchange what a step needs -- the new vector's entries and the dots -- through
// epoch-tagged words (ks_pub_store), so nothing is fenced.  A step of the common
// two passes costs three exchanges, which and the latency of loading V bound it (V itself
// comes from L2).  Measured, a step, launches -> this: graph Laplacian of 2,000 rows,
// columns 16..32, 39.9 -> 15.4 us, 64..128 43.7 -> 30.6; convection-diffusion on 150 x
// 150 (88 workgroups) 39.0 -> 16.1 and 48.2 -> 27.5; on 220 x 220 (190) 42.9 -> 19.0 and
// 57.1 -> 34.3.
//
// A word is rewritten only after every workgroup has read it: the sums alternate
// between two areas, and a workgroup writes an area again two exchanges later, when it
// has seen the sums of the exchange between, which every workgroup gave after reading
// the first; the vector's words are rewritten a step later, after that step's dots.
// Every wait is bounded (KS_EXP_SPIN polls unless ks_ctx_expand_polls says otherwise, or
// sooner once *err shows another ran out): then the status carries KS_ERR_TIMEOUT, no
// total goes out that a value is missing from, every workgroup leaves the kernel, and
// the caller expands with the launches (the start column and those before it are not
// touched).  Beside work that keeps the chip full each such launch costs 0.1 s and more,
// so the context then leaves a growing number of expansions to the launches at once.
// The workgroups wait on each other, so they must be able to run at the
// same time: up to KS_EXP_MAXG2 of them two fit a CU, up to KS_EXP_MAXG three, so that
// one launch of each of the four hardware queues HIP uses fits the chip.
#include "ks_internal.hpp"

namespace {

#define KS_EXP_MAXG 192            // workgroups, at most
#define KS_EXP_MAXG2 128           // of the form of which two fit a CU
#define KS_EXP_MAXK 128            // columns orthogonalized against, at most
// Up to KS_EXP_DIRECT workgroups every one adds up all sums itself; more add a column's
// each and exchange the totals.  A step at columns 16..32, direct against that: 9
// workgroups 17.1 against 18.5 us, 36 workgroups 23.3 against 19.2 (64..128: 51.8 against
// 30.7).
#define KS_EXP_DIRECT 16
#define KS_EXP_SPIN (1 << 18)      // polls of about half a microsecond
#define KS_EXP_CB 8                // columns of a wavefront's batch
#define KS_EXP_PER (KS_SPMV_NNZ / KS_BLOCK)
static_assert(KS_SPMV_ROWS == KS_BLOCK, "a thread a row");

struct exp_args {
  int n, ld, nc, j0, m, G, polls;
  const int32_t *blk, *rowptr, *colidx;
  const void *val;
  void *V;
  double *buf;
  int ldbuf, refine;
  double eta, deftol;
  ks_status *st;
  unsigned long long *part, *tot, *vec;   // [2][MAXK + 1][MAXG][2], [2][MAXK + 1][2], [n][2]
  unsigned *err;                          // the last launch (its first epoch) whose wait ran out
  unsigned epoch;                         // the first of this launch
};

// *err == launch: another wait of this launch has run out
__device__ __forceinline__ double exp_wait(const unsigned long long *w, unsigned epoch, unsigned *err, unsigned launch,
                                           int polls, int &dead) {
  for (int spins = 0; !dead;) {
    const unsigned long long lo = ks_pub_load(w), hi = ks_pub_load(w + 1);
    if ((unsigned)(lo >> 32) == epoch && (unsigned)(hi >> 32) == epoch) return ks_pub_f64(lo, hi);
    if (++spins > polls ||
        ((spins & 255) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == launch)) {
      __hip_atomic_store(err, launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dead = 1;
    }
    __builtin_amdgcn_s_sleep(1);
  }
  return 0.0;
}

// the sum over each aligned group of GP lanes (a power of two), in every lane
__device__ __forceinline__ double group_sum(double v, int GP) {
  if (GP > 32) v = ks_lane_xor_add<32>(v);
  if (GP > 16) v = ks_lane_xor_add<16>(v);
  if (GP > 8) v = ks_lane_xor_add<8>(v);
  if (GP > 4) v = ks_lane_xor_add<4>(v);
  if (GP > 2) v = ks_lane_xor_add<2>(v);
  if (GP > 1) v = ks_lane_xor_add<1>(v);
  return v;
}

// WGS: workgroups that fit a CU.  2 leaves the registers to keep the last batch of V's
// columns from the dots to the update.
template <typename T, typename VT, int WGS>
__global__ __launch_bounds__(KS_BLOCK, WGS) void k_expand(exp_args a) {
  __shared__ double prod[KS_SPMV_NNZ];
  __shared__ double wl[KS_SPMV_ROWS];                  // this workgroup's rows of the vector
  __shared__ double red[KS_WAVES][KS_SPMV_ROWS];
  __shared__ double tot[KS_EXP_MAXK + 1], hacc[KS_EXP_MAXK + 1];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.x, G = a.G;
  const T *V = (const T *)a.V;
  unsigned *const err = a.err;
  const unsigned launch = a.epoch;
  const size_t ld = (size_t)a.ld;
  if (!a.st->active) return;
  const int r0 = a.blk[b], nrows = a.blk[b + 1] - r0, p0 = a.rowptr[r0], cnt = a.rowptr[r0 + nrows] - p0;
  // this thread's entries of the row block: their columns are kept for every step
  // (-1: none), their values loaded while the step waits for the vector
  int ci[KS_EXP_PER];
#pragma unroll
  for (int u = 0; u < KS_EXP_PER; u++) {
    const int p = tid + u * KS_BLOCK;
    ci[u] = p < cnt ? a.colidx[p0 + p] : -1;
  }
  int tpr = 1;   // threads a row in the product's sums
  while (tpr < 64 && nrows * (tpr << 1) <= KS_BLOCK) tpr <<= 1;
  const int lr = tid / tpr, sub = tid & (tpr - 1);
  int rs = 0, re = 0;
  if (lr < nrows) {
    rs = a.rowptr[r0 + lr] - p0;
    re = a.rowptr[r0 + lr + 1] - p0;
  }
  int GP = 1;    // lanes that hold one column's sums of all workgroups (G <= 64)
  while (GP < G && GP < 64) GP <<= 1;
  // byte offsets of rows lane, lane + 64, ... of the block (past its end: its last, whose dots get a zero)
  unsigned rowoff[4];
#pragma unroll
  for (int q = 0; q < 4; q++) rowoff[q] = (unsigned)(r0 + min(64 * q + lane, nrows - 1)) * (unsigned)sizeof(T);
  unsigned ep = a.epoch;
  int par = 0, dead = 0;
  long passes = 0;
  int breakdown = -1, error = 0, lastcol = -1, lastpass = 0, lindep = 0;
  double nrm = 0.0, onrm = 0.0, sumsq = 0.0;

  int pt = p0 + tid;
#pragma unroll 1
  for (int j = a.j0; j < a.m; j++) {
    // what the addresses of a step are made from, opaque here: computed before the
    // loop and kept they would not leave the registers WGS asks for
#pragma unroll
    for (int u = 0; u < KS_EXP_PER; u++) asm volatile("" : "+v"(ci[u]));
#pragma unroll
    for (int q = 0; q < 4; q++) asm volatile("" : "+v"(rowoff[q]));
    asm volatile("" : "+v"(pt));
    const int col = j + 1, kk = a.nc + col;        // storage column kk, against the kk before it
    const int cw = (kk + KS_WAVES - 1) / KS_WAVES; // columns of a wavefront
    const int c0 = wave * cw, c1 = min(kk, c0 + cw), nb = (cw + KS_EXP_CB - 1) / KS_EXP_CB;
    const T *x = V + (size_t)(kk - 1) * ld;
    double vb[KS_EXP_CB][4];
    auto load_batch = [&](int bt) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < KS_EXP_CB; u++) {
        const int c = c0 + bt * KS_EXP_CB + u;
        const char *vc = (const char *)(V + (size_t)min(c, kk - 1) * ld);   // past the wavefront's columns: not used
#pragma unroll
        for (int q = 0; q < 4; q++) vb[u][q] = (double)*(const T *)(vc + rowoff[q]);
      }
    };
    // ---- w = A v: the previous step's vector as its workgroups publish it
    {
      double xv[KS_EXP_PER];
      VT va[KS_EXP_PER];
#pragma unroll
      for (int u = 0; u < KS_EXP_PER; u++) va[u] = ci[u] >= 0 ? ((const VT *)a.val)[pt + u * KS_BLOCK] : (VT)0;
      if (j == a.j0) {
#pragma unroll
        for (int u = 0; u < KS_EXP_PER; u++) xv[u] = ci[u] >= 0 ? (double)x[ci[u]] : 0.0;
      } else {
        const unsigned long long tag0 = (unsigned long long)ep << 32;
        // all entries at once, again while some are not there (rarely)
        for (int spins = 0;;) {
          bool ok = true;
#pragma unroll
          for (int u = 0; u < KS_EXP_PER; u++) {
            unsigned long long lo = tag0, hi = tag0;
            if (ci[u] >= 0) {
              lo = ks_pub_load(a.vec + 2 * (size_t)ci[u]);
              hi = ks_pub_load(a.vec + 2 * (size_t)ci[u] + 1);
            }
            xv[u] = ks_pub_f64(lo, hi);
            ok = ok && (unsigned)(lo >> 32) == ep && (unsigned)(hi >> 32) == ep;
          }
          if (ok) break;
          if (++spins > a.polls || ((spins & 255) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == launch)) {
            __hip_atomic_store(err, launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            dead = 1;
            break;
          }
          __builtin_amdgcn_s_sleep(1);
        }
      }
#pragma unroll
      for (int u = 0; u < KS_EXP_PER; u++) prod[tid + u * KS_BLOCK] = (double)va[u] * xv[u];
    }

    if (__syncthreads_or(dead)) break;
    if (lr < nrows) {
      double s = 0.0;
#pragma unroll 2
      for (int q = rs + sub; q < re; q += tpr) s += prod[q];
      for (int off = tpr >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
      if (sub == 0) wl[lr] = (double)(T)s;
    }
    for (int c = tid; c <= kk; c += KS_BLOCK) hacc[c] = 0.0;
    __syncthreads();
    // ---- the passes: dots (with the vector's own), then the update, as DGKS asks
    int l = 0, fin = 0;
    double scale = 1.0;
    lindep = 0;
#pragma unroll 1
    for (;;) {
      // this workgroup's sums of columns c0 .. c1-1 and, by wavefront 0, |w|^2
      ep++;
      par ^= 1;
#pragma unroll
      for (int q = 0; q < 4; q++) asm volatile("" : "+v"(rowoff[q]));
      unsigned long long *P = a.part + (size_t)par * (KS_EXP_MAXK + 1) * KS_EXP_MAXG * 2;
      double wq[4];
#pragma unroll
      for (int q = 0; q < 4; q++) wq[q] = 64 * q + lane < nrows ? wl[64 * q + lane] : 0.0;
#pragma unroll 1
      for (int bt = 0; bt < nb; bt++) {
        load_batch(bt);
        double d[KS_EXP_CB];
#pragma unroll
        for (int u = 0; u < KS_EXP_CB; u++)
          d[u] = (vb[u][0] * wq[0] + vb[u][1] * wq[1]) + (vb[u][2] * wq[2] + vb[u][3] * wq[3]);
        ks_multi_sum<KS_EXP_CB>::run(d, lane);
        const int c = c0 + bt * KS_EXP_CB + ks_multi_sum<KS_EXP_CB>::index(lane, 0);
        if (ks_multi_sum<KS_EXP_CB>::leader(lane) && c < c1) ks_pub_store_f64(P + 2 * ((size_t)c * G + b), ep, d[0]);
      }
      if (wave == 0) {
        const double s = ks_wave_sum((wq[0] * wq[0] + wq[1] * wq[1]) + (wq[2] * wq[2] + wq[3] * wq[3]));
        if (lane == 0) ks_pub_store_f64(P + 2 * ((size_t)kk * G + b), ep, s);
      }
      // the totals, in every workgroup
      if (G <= KS_EXP_DIRECT) {
        const int cpl = 64 / GP, cs = lane / GP, g = lane & (GP - 1);   // columns a wavefront adds at once
#pragma unroll 1
        for (int c = wave * cpl; c <= kk; c += KS_WAVES * cpl) {
          const int cc = c + cs;
          double s = 0.0;
          if (cc <= kk && g < G) s = exp_wait(P + 2 * ((size_t)cc * G + g), ep, err, launch, a.polls, dead);
          s = group_sum(s, GP);
          if (g == 0 && cc <= kk) tot[cc] = s;
        }
      } else {   // a wavefront a column, then everyone reads the kk + 1 totals
        unsigned long long *Q = a.tot + (size_t)par * (KS_EXP_MAXK + 1) * 2;
#pragma unroll 1
        for (int c = b + wave * G; c <= kk; c += KS_WAVES * G) {
          double s = 0.0;
#pragma unroll
          for (int q = 0; q < KS_EXP_MAXG / 64; q++)
            if (lane + 64 * q < G) s += exp_wait(P + 2 * ((size_t)c * G + lane + 64 * q), ep, err, launch, a.polls, dead);
          s = ks_wave_sum(s);
          if (!__any(dead) && lane == 0) ks_pub_store_f64(Q + 2 * c, ep, s);
        }
        if (tid <= kk) tot[tid] = exp_wait(Q + 2 * tid, ep, err, launch, a.polls, dead);
      }
      if (__syncthreads_or(dead)) break;
      // ---- the decisions of BVOrthogonalizeGS (bvorthog.c:91-217), alike in every workgroup
      const double self = tot[kk];
      double sq = 0.0;
      for (int c = lane; c < kk; c += 64) sq += tot[c] * tot[c];
      sq = ks_wave_sum(sq);
      if (l == 0) {
        if (self < -a.deftol) {
          error = KS_ERR_INNER;
          break;
        }
        onrm = self < 0.0 ? 0.0 : sqrt(self);
      } else {
        const double exact = sqrt(self);
        bool more = false;
        if (a.refine == KS_REFINE_NEVER) {
          nrm = exact;
          lindep = !(nrm != 0.0);
        } else if (a.refine == KS_REFINE_ALWAYS && l < 2) {
          more = true;
        } else {
          nrm = onrm * onrm - sumsq;
          nrm = nrm <= 0.0 ? exact : sqrt(nrm);
          if (a.refine == KS_REFINE_IFNEEDED && l < 3 && nrm != 0.0 && fabs(nrm) < a.eta * fabs(onrm)) more = true;
          else lindep = !(nrm != 0.0 && fabs(nrm) >= a.eta * fabs(onrm));
        }
        if (!more) {
          fin = 1;
          scale = (!lindep && nrm != 1.0) ? 1.0 / nrm : 1.0;
          break;
        }
        onrm = exact;
      }
      sumsq = sq;
      // the pass's outcome is known before it when its estimate is positive (and
      // another pass does not follow): then it needs no dots
      if (a.refine != KS_REFINE_NEVER && !(a.refine == KS_REFINE_ALWAYS && l + 1 < 2)) {
        const double e2 = onrm * onrm - sumsq;
        if (e2 > 0.0) {
          const double e = sqrt(e2);
          if (!(a.refine == KS_REFINE_IFNEEDED && l + 1 < 3 && e < a.eta * fabs(onrm))) {
            nrm = e;
            lindep = !(nrm >= a.eta * fabs(onrm));
            scale = (!lindep && nrm != 1.0) ? 1.0 / nrm : 1.0;
            fin = 1;
          }
        }
      }
      // ---- w -= V c, h += c
      double s[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
      for (int bt = nb - 1; bt >= 0; bt--) {
        if (WGS != 2 || bt != nb - 1) load_batch(bt);   // the last one is here from the dots
#pragma unroll
        for (int u = 0; u < KS_EXP_CB; u++) {
          const int c = c0 + bt * KS_EXP_CB + u;
          const double cf = c < c1 ? tot[c] : 0.0;
#pragma unroll
          for (int q = 0; q < 4; q++) s[q] += vb[u][q] * cf;
        }
      }
#pragma unroll
      for (int q = 0; q < 4; q++) red[wave][64 * q + lane] = s[q];
      for (int c = tid; c < kk; c += KS_BLOCK) hacc[c] += tot[c];
      __syncthreads();
      if (tid < nrows) {
        static_assert(KS_WAVES == 4, "added in pairs");
        wl[tid] = (double)(T)(wl[tid] - ((red[0][tid] + red[1][tid]) + (red[2][tid] + red[3][tid])));
      }
      __syncthreads();
      l++;
      passes++;
      if (fin) break;
    }
    if (!fin) break;   // an error or a wait that ran out
    // ---- the column, stored and published for the next product
    ep++;
    if (tid < nrows) {
      const T v = scale == 1.0 ? (T)wl[tid] : (T)(wl[tid] * scale);
      ((T *)a.V)[(size_t)kk * ld + r0 + tid] = v;
      if (!lindep && j + 1 < a.m) ks_pub_store_f64(a.vec + 2 * (size_t)(r0 + tid), ep, (double)v);
    }
    if (b == 0) {
      double *h = a.buf + (size_t)col * a.ldbuf;
      for (int c = tid; c <= kk; c += KS_BLOCK) h[c] = c < kk ? hacc[c] : (lindep ? 0.0 : nrm);
    }
    lastcol = col;
    lastpass = l;
    if (lindep) {
      breakdown = col;
      break;
    }
    __syncthreads();   // the column's stores before the next step's loads of it; hacc read before it is cleared
  }
  if (__syncthreads_or(dead)) {
    if (tid == 0) {
      a.st->error = KS_ERR_TIMEOUT;
      a.st->active = 0;
    }
  } else if (b == 0 && tid == 0) {
    ks_status *st = a.st;
    if (error) st->error = error;
    if (error || breakdown >= 0) st->active = 0;
    st->breakdown_col = breakdown;
    st->col = lastcol;
    st->pass_done = lastpass;
    st->done = 1;
    st->lindep = lindep;
    st->total_passes += passes;
    st->onrm = onrm;
    st->sumsq = sumsq;
    st->nrm = st->beta_last = nrm;
    st->scale = 1.0;
    st->prescale_col = st->defer_col = st->halt_col = -1;
  }
}

// the exchange areas of a context, made by its first expansion (none: there is no room for them);
// the epochs of its words start at 0
int exp_areas(ks_ctx ctx, unsigned long long **w) {
  const size_t words = 2 * (2 * (size_t)(KS_EXP_MAXK + 1) * (KS_EXP_MAXG + 1) + (size_t)KS_EXP_MAXG * KS_SPMV_ROWS) + 8;
  if (!ctx->d_exp) {
    if (hipMalloc((void **)&ctx->d_exp, words * sizeof(unsigned long long)) != hipSuccess) {
      (void)hipGetLastError();
      *w = ctx->d_exp = nullptr;
      return KS_OK;
    }
    ctx->exp_epoch = 0;
  }
  if (ctx->exp_epoch == 0 || ctx->exp_epoch > 0xf0000000u) {
    KS_TRY(ks_memset_zero(ctx, ctx->d_exp, words * sizeof(unsigned long long)));
    ctx->exp_epoch = 1;
  }
  *w = ctx->d_exp;
  return KS_OK;
}

}  // namespace

extern "C" int ks_ctx_expand_polls(ks_ctx ctx, int polls) {
  KS_CHECK(ctx && polls >= 0, KS_ERR_ARG, "bad number of polls");
  ctx->exp_polls = polls;
  ctx->exp_hold = ctx->exp_back = 0;
  return KS_OK;
}

extern "C" int ks_arnoldi_expand(ks_ctx ctx, ks_csr A, ks_prec prec, int n, void *V, int ld, int nc, int k, int m,
                                 double *d_buf, int ldbuf, ks_refine refine, double eta, int *taken) {
  KS_CHECK(ctx && A && V && d_buf && taken, KS_ERR_ARG, "null expansion argument");
  KS_CHECK(n > 0 && ld >= n && nc >= 0 && k >= 0 && m > k && ldbuf > nc + m && n == A->nrows && n == A->ncols,
           KS_ERR_ARG, "bad expansion sizes n=%d ld=%d nc=%d k=%d m=%d ldbuf=%d", n, ld, nc, k, m, ldbuf);
  KS_CHECK(refine >= KS_REFINE_IFNEEDED && refine <= KS_REFINE_ALWAYS, KS_ERR_ARG, "bad refinement type");
  *taken = 0;
  if (ctx->prof || ctx->capturing) return KS_OK;   // per-kernel events, or a replay that would repeat the epochs
  if (A->variant != 0 || A->nblocks > KS_EXP_MAXG || nc + m > KS_EXP_MAXK || m > n - 1) return KS_OK;
  if (ctx->exp_hold > 0) {   // a launch's workgroups could not all run (ks_status_get)
    ctx->exp_hold--;
    return KS_OK;
  }
  exp_args a = {};
  unsigned long long *w;
  KS_TRY(exp_areas(ctx, &w));
  if (!w) return KS_OK;
  a.n = n;
  a.ld = ld;
  a.nc = nc;
  a.j0 = k;
  a.m = m;
  a.G = A->nblocks;
  a.polls = ctx->exp_polls ? ctx->exp_polls : KS_EXP_SPIN;
  a.blk = A->d_blk;
  a.rowptr = A->d_rowptr;
  a.colidx = A->d_colidx;
  a.val = A->d_val;
  a.V = V;
  a.buf = d_buf;
  a.ldbuf = ldbuf;
  a.refine = refine;
  a.eta = eta;
  a.deftol = 10.0 * 2.220446049250313e-16;
  a.st = ctx->d_status;
  a.part = w;
  a.tot = a.part + 2 * (size_t)(KS_EXP_MAXK + 1) * KS_EXP_MAXG * 2;
  a.vec = a.tot + 2 * (size_t)(KS_EXP_MAXK + 1) * 2;
  a.err = (unsigned *)(a.vec + 2 * (size_t)KS_EXP_MAXG * KS_SPMV_ROWS);
  a.epoch = ctx->exp_epoch;
  ctx->exp_epoch += 8u * (unsigned)(m - k) + 8u;   // at most five exchanges a step
  const dim3 g(a.G), t(KS_BLOCK);
#define KS_EXP_LAUNCH(T, VT)                                                            \
  do {                                                                                  \
    if (a.G <= KS_EXP_MAXG2) hipLaunchKernelGGL((k_expand<T, VT, 2>), g, t, 0, ctx->stream, a); \
    else hipLaunchKernelGGL((k_expand<T, VT, 3>), g, t, 0, ctx->stream, a);             \
  } while (0)
  if (prec == KS_F64 && A->vprec == KS_F64) KS_EXP_LAUNCH(double, double);
  else if (prec == KS_F64) KS_EXP_LAUNCH(double, float);
  else if (A->vprec == KS_F64) KS_EXP_LAUNCH(float, double);
  else KS_EXP_LAUNCH(float, float);
#undef KS_EXP_LAUNCH
  KS_HIP(hipGetLastError());
  ctx->exp_live = true;
  *taken = 1;
  return KS_OK;
}
