// ks_tsqr.hip -- TSQR of a tall-skinny FP64 panel on one GPU (BVOrthogonalize
// with block types TSQR and TSQRCHOL; the reference's BVOrthogonalize_TSQR /
// _TSQRCHOL, src/sys/classes/bv/interface/bvorthog.c:615-663, factor the panel
// with LAPACK on each process and reduce the triangular factors across
// processes, bvlapack.c:347-560).
//
// Here the row blocks are workgroups.  The panel's rows are cut into leaves of
// rb rows (a multiple of 64, at least 2k); a workgroup loads its leaf into LDS,
// factors it by Householder reflections (dgeqr2's steps) and, for TSQR, forms its
// explicit Q in place (dorg2r's steps) and writes it back over the leaf.  The
// leaves' k x k factors, stacked f at a time (256 rows where LDS holds them), are
// the rows of the next level, factored by the same kernel, until one node
// remains: its R is the panel's.  For TSQR the Q of the panel is then the leaf
// Q times the product of the slices of the node Q's on the leaf's path to the
// root: a top-down pass forms that k x k product per leaf and a last pass
// multiplies each leaf by its own.
//
// Every level is one launch; the sums inside a workgroup run in a fixed order,
// so a factorization is deterministic.  The workspace (the node levels and the
// per-leaf products, about 1.5 n k doubles in all) is the context's.
#include "ks_internal.hpp"

namespace {

// A workgroup of NW wavefronts factors a node.  Lane l of every wavefront holds
// rows l, l + 64, ... of the node's matrix, which stays in LDS column-major
// (stride 64 R; a row a lane, so no bank conflicts).  In a column step each
// wavefront forms the reflector itself, in registers, and applies it to its own
// columns, eight at a time (columns 8 g .. 8 g + 7 belong to wavefront g mod NW);
// the sums over rows are lane exchanges, eight columns together by recursive
// halving (ks_multi_sum), so a step has one barrier.  The steps are a chain of
// latencies: NW spreads a step's columns over the SIMDs where k has enough.
// 500,000 x 32 with Q (four wavefronts sharing a column step's sums through
// three barriers, 64-row nodes, before; now): leaves and nodes 4.8 -> 0.78 ms, the
// call 8.26 -> 1.17 ms; R alone 3.51 -> 0.70; 500,000 x 8 548 -> 236 us; 500,000 x
// 60 23.1 -> 5.0 ms.
#define KS_TSQR_CB 8   // columns updated together

// rows j+1.. of the column at aj, as the reflector's vector with 1 at row j
template <int R>
__device__ __forceinline__ void tsqr_vector(const double *aj, int j, int lane, double scal, double (&v)[R]) {
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int r = 64 * q + lane;
    const double x = aj[r];
    v[q] = r > j ? x * scal : (r == j ? 1.0 : 0.0);
  }
}

// this wavefront's columns beyond j of A become (I - t v v^T) times themselves
template <int R, int NW>
__device__ __forceinline__ void tsqr_reflect(double *A, int k, int j, double t, const double (&v)[R], int lane,
                                             int wave) {
  using MS = ks_multi_sum<KS_TSQR_CB>;
  constexpr int rb = 64 * R;
  for (int g = (j + 1) / KS_TSQR_CB; g * KS_TSQR_CB < k; g++) {
    if (g % NW != wave) continue;
    const int c = g * KS_TSQR_CB;
    double x[KS_TSQR_CB][R], d[KS_TSQR_CB];
#pragma unroll
    for (int u = 0; u < KS_TSQR_CB; u++) {
      const double *ac = A + (size_t)min(c + u, k - 1) * rb + lane;
      d[u] = 0.0;
#pragma unroll
      for (int q = 0; q < R; q++) {
        x[u][q] = ac[64 * q];
        d[u] += v[q] * x[u][q];
      }
    }
    MS::run(d, lane);   // eight totals: lane 8 m holds total m
#pragma unroll
    for (int u = 0; u < KS_TSQR_CB; u++) {
      const double s = t * ks_readlane_f64(d[0], 8 * u);
      if (c + u > j && c + u < k) {
        double *ac = A + (size_t)(c + u) * rb + lane;
#pragma unroll
        for (int q = 0; q < R; q++) ac[64 * q] = x[u][q] - s * v[q];
      }
    }
  }
}

// Householder QR of the 64 R x k matrix A: R in the upper triangle, the
// reflectors' vectors below it (v_0 = 1 implicit), their factors in tau.  dlarfg:
// beta = -sign(alpha) |(alpha, x)|, tau = (beta - alpha) / beta, v = x / (alpha -
// beta); tau = 0 when x = 0.  A column is written by its wavefront after the
// step's barrier, when every wavefront has read it.
template <int R, int NW>
__device__ __forceinline__ void tsqr_geqr2(double *A, int k, double *tau, int lane, int wave) {
  constexpr int rb = 64 * R;
  for (int j = 0; j < k; j++) {
    double *aj = A + (size_t)j * rb;
    double s = 0.0;
#pragma unroll
    for (int q = 0; q < R; q++) {
      const double x = aj[64 * q + lane];
      s += 64 * q + lane > j ? x * x : 0.0;
    }
    const double xnorm2 = ks_wave_sum(s), alpha = aj[j];
    double t = 0.0, scal = 0.0, beta = alpha;
    if (xnorm2 > 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xnorm2), alpha);
      t = (beta - alpha) / beta;
      scal = 1.0 / (alpha - beta);
    }
    double v[R];
    tsqr_vector<R>(aj, j, lane, scal, v);
    if (t != 0.0) tsqr_reflect<R, NW>(A, k, j, t, v, lane, wave);
    __syncthreads();
    if ((j / KS_TSQR_CB) % NW == wave) {
      if (lane == 0) tau[j] = t;
      if (t != 0.0)
#pragma unroll
        for (int q = 0; q < R; q++)
          if (64 * q + lane >= j) aj[64 * q + lane] = 64 * q + lane == j ? beta : v[q];
    }
  }
  __syncthreads();
}

// dorg2r on the factored A: the first k columns of H_0 ... H_{k-1}, in place
template <int R, int NW>
__device__ __forceinline__ void tsqr_org2r(double *A, int k, const double *tau, int lane, int wave) {
  constexpr int rb = 64 * R;
  for (int j = k - 1; j >= 0; j--) {
    double *aj = A + (size_t)j * rb;
    const double t = tau[j];
    double v[R];
    tsqr_vector<R>(aj, j, lane, 1.0, v);
    if (t != 0.0) tsqr_reflect<R, NW>(A, k, j, t, v, lane, wave);
    __syncthreads();
    if ((j / KS_TSQR_CB) % NW == wave)   // the wavefront that will update this column from the next step on
#pragma unroll
      for (int q = 0; q < R; q++) {
        const int r = 64 * q + lane;
        aj[r] = r == j ? 1.0 - t : -t * v[q];   // rows above j: v = 0
      }
  }
  __syncthreads();
}

// One level: block b factors rows [b rb, min(b rb + rb, nrows)) of the level's
// matrix (block b's rows start at base + b bstride, leading dimension ld; rows
// past nrows, and rows rb .. 64 R - 1 of the node, count as zero).  Its R goes to
// rout: block b's k x k factor at rows (b % rf) k of the (rf k) x k matrix number
// b / rf, leading dimension rf k.  FORM_Q: its explicit Q overwrites its rows.
template <bool FORM_Q, int R, int NW>
__global__ __launch_bounds__(64 * NW) void k_tsqr_level(double *base, long ld, long bstride, int rb, long nrows,
                                                        int k, double *rout, int rf) {
  extern __shared__ double lds[];
  double *A = lds, *tau = A + (size_t)64 * R * k;
  const int b = blockIdx.x, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double *in = base + (size_t)b * bstride;
  const long r0 = (long)b * rb;
  const int valid = (int)min((long)rb, nrows - r0);
  for (int c = wave; c < k; c += NW)
#pragma unroll
    for (int q = 0; q < R; q++) {
      const int r = 64 * q + lane;
      A[(size_t)c * 64 * R + r] = r < valid ? in[r + (size_t)c * ld] : 0.0;
    }
  __syncthreads();
  tsqr_geqr2<R, NW>(A, k, tau, lane, wave);
  double *Rf = rout + (size_t)(b / rf) * ((size_t)rf * k * k) + (size_t)(b % rf) * k;
  const long ldr = (long)rf * k;
  for (int j = wave; j < k; j += NW)
    for (int i = lane; i < k; i += 64) Rf[i + (size_t)j * ldr] = i <= j ? A[(size_t)j * 64 * R + i] : 0.0;
  if (FORM_Q) {
    __syncthreads();
    tsqr_org2r<R, NW>(A, k, tau, lane, wave);
    for (int c = wave; c < k; c += NW)
#pragma unroll
      for (int q = 0; q < R; q++) {
        const int r = 64 * q + lane;
        if (r < valid) in[r + (size_t)c * ld] = A[(size_t)c * 64 * R + r];
      }
  }
}

// Top-down: child b of the level below takes M_child[b] = S(b) M_parent[b / f],
// S(b) the k x k slice at rows (b % f) k of its parent's Q (leading dimension
// f k); M_parent = I at the root.  Both factors pass through LDS.  kp > 0 (the
// leaves' products): stored by rows with stride kp, zeros past column k.
#define KS_TSQR_NT 256
__global__ __launch_bounds__(KS_TSQR_NT) void k_tsqr_down(const double *Q, int f, int k, const double *Mpar,
                                                          double *Mch, int kp) {
  extern __shared__ double lds[];
  double *S = lds, *P = lds + k * k;
  const int b = blockIdx.x, p = b / f, t = b % f;
  const long ldq = (long)f * k;
  const double *Sg = Q + (size_t)p * ((size_t)f * k * k) + (size_t)t * k;
  for (int e = threadIdx.x; e < k * k; e += KS_TSQR_NT) {
    const int i = e % k, j = e / k;
    S[e] = Sg[i + (size_t)j * ldq];
    if (Mpar) P[e] = Mpar[(size_t)p * k * k + e];
  }
  __syncthreads();
  double *out = Mch + (size_t)b * k * (kp ? kp : k);
  for (int e = threadIdx.x; e < k * k; e += KS_TSQR_NT) {
    const int i = e % k, j = e / k;
    double a = 0.0;
    if (Mpar)
      for (int c = 0; c < k; c++) a += S[i + c * k] * P[c + j * k];
    else
      a = S[e];
    if (kp) out[(size_t)i * kp + j] = a;
    else out[e] = a;
  }
  for (int e = threadIdx.x; e < k * (kp - k); e += KS_TSQR_NT) out[(size_t)(e / (kp - k)) * kp + k + e % (kp - k)] = 0.0;
}

// Rows [64 g, 64 g + 64) of V times M of their leaf (rb rows a leaf), in place: a
// row a lane, its k products in registers, M's entries wave-uniform (scalar
// loads), the row's values loaded eight columns ahead.  Reads and writes V once:
// 500,000 x 32 in 100 us (2.6 TB/s; through LDS with M from global memory 664).
template <int K>
__global__ __launch_bounds__(64) void k_tsqr_apply(double *V, long ld, int n, int rb, int k,
                                                   const double *__restrict__ M) {
  const int row = blockIdx.x * 64 + threadIdx.x, rc = min(row, n - 1);
  const double *__restrict__ Mb = M + (size_t)(blockIdx.x * 64 / rb) * k * K;
  double acc[K];
#pragma unroll
  for (int j = 0; j < K; j++) acc[j] = 0.0;
  for (int c0 = 0; c0 < k; c0 += 8) {
    double x[8];
#pragma unroll
    for (int u = 0; u < 8; u++) x[u] = V[rc + (size_t)min(c0 + u, k - 1) * ld];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      if (c0 + u < k) {
        const double *m = Mb + (size_t)(c0 + u) * K;
#pragma unroll
        for (int j = 0; j < K; j++) acc[j] += x[u] * m[j];
      }
    }
  }
  if (row < n)
#pragma unroll
    for (int j = 0; j < K; j++)
      if (j < k) V[row + (size_t)j * ld] = acc[j];
}

template <bool FORM_Q, int NW>
void launch_level(hipStream_t st, long cnt, int R, double *base, long ld, long bstride, int rb, long nrows, int k,
                  double *rout, int rf) {
  const size_t lds = sizeof(double) * ((size_t)64 * R + 1) * k;
  const dim3 g((unsigned)cnt), w(64 * NW);
#define KS_TSQR_R(X)                                                                                                \
  case X:                                                                                                           \
    hipLaunchKernelGGL((k_tsqr_level<FORM_Q, X, NW>), g, w, lds, st, base, ld, bstride, rb, nrows, k, rout, rf);     \
    break;
  switch (R) { KS_TSQR_R(1) KS_TSQR_R(2) KS_TSQR_R(3) KS_TSQR_R(4) }
#undef KS_TSQR_R
}

// one wavefront for every eight columns, up to eight
template <bool FORM_Q>
void launch_level_k(hipStream_t st, long cnt, int R, double *base, long ld, long bstride, int rb, long nrows, int k,
                    double *rout, int rf) {
  if (k <= 8) launch_level<FORM_Q, 1>(st, cnt, R, base, ld, bstride, rb, nrows, k, rout, rf);
  else if (k <= 16) launch_level<FORM_Q, 2>(st, cnt, R, base, ld, bstride, rb, nrows, k, rout, rf);
  else if (k <= 32) launch_level<FORM_Q, 4>(st, cnt, R, base, ld, bstride, rb, nrows, k, rout, rf);
  else launch_level<FORM_Q, 8>(st, cnt, R, base, ld, bstride, rb, nrows, k, rout, rf);
}

// columns of the leaves' products, padded to what k_tsqr_apply is built for
inline int apply_cols(int k) { return k <= 8 ? 8 : (k <= 16 ? 16 : (k + 31) / 32 * 32); }

}  // namespace

extern "C" int ks_bv_tsqr(ks_ctx ctx, int n, double *d_V, int ld, int k, int form_q, double *R, int ldr) {
  KS_CHECK(ctx && d_V && R, KS_ERR_ARG, "null TSQR argument");
  KS_CHECK(k >= 1 && n >= k && ld >= n && ldr >= k, KS_ERR_ARG, "TSQR needs 1 <= k <= n <= ld and ldr >= k");
  int dev = 0, maxlds = 0;
  KS_HIP(hipGetDevice(&dev));
  KS_HIP(hipDeviceGetAttribute(&maxlds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
  const int rmin = (2 * k + 63) / 64;   // rows of a leaf / 64, at least
  const size_t lds_level = sizeof(double) * ((size_t)64 * rmin + 1) * k;
  KS_CHECK(lds_level <= (size_t)maxlds, KS_ERR_ARG,
           "TSQR of %d columns needs %zu bytes of LDS per workgroup (the device has %d)", k, lds_level, maxlds);
  // Longer leaves make a shallower tree, as long as they still fill the chip
  // (KS_TSQR_LEAVES of them) and a CU holds several; the nodes above, too few to
  // fill it, take as many children as 256 rows of LDS hold.  500,000 x 32 with
  // leaves of 128 rows 1165 us, of 64 rows (a line at 7000) 1510.
  int r0 = rmin, rn = rmin;
#define KS_TSQR_LEAVES 2048
  while (r0 < 4 && sizeof(double) * 64 * (r0 + 1) * k <= 32768 && n / (64 * (r0 + 1)) >= KS_TSQR_LEAVES) r0++;
  while (rn < 4 && sizeof(double) * ((size_t)64 * (rn + 1) + 1) * k <= (size_t)maxlds) rn++;
  const int rb = 64 * r0, f = 64 * rn / k;
  // level sizes: cnt[0] leaves, cnt[l] nodes of level l
  std::vector<long> cnt(1, ((long)n + rb - 1) / rb);
  while (cnt.back() > 1) cnt.push_back((cnt.back() + f - 1) / f);
  const int L = (int)cnt.size() - 1, kp = apply_cols(k);
  KS_CHECK(cnt[0] <= 0x7fffffffL && kp <= 96, KS_ERR_ARG, "TSQR panel too large");
  const size_t node = (size_t)f * k * k;
  // workspace: the panel's R, the node levels, the levels' products (the leaves' padded)
  std::vector<size_t> buf(L + 1, 0), mat(L + 1, 0);
  size_t words = (size_t)k * k;
  for (int l = 1; l <= L; l++) buf[l] = words, words += node * (size_t)cnt[l];
  if (form_q)
    for (int l = 0; l < L; l++) mat[l] = words, words += (size_t)k * (l ? k : kp) * (size_t)cnt[l];
  double *ws = nullptr;
  KS_TRY(ks_ws_take(ctx, sizeof(double) * words, (void **)&ws));
  hipStream_t st = ctx->stream;
  // leaves, then node levels: level l factors the cnt[l-1] factors of the level below, f per node
  for (int l = 0; l <= L; l++) {
    double *base = l ? ws + buf[l] : d_V, *rout = l < L ? ws + buf[l + 1] : ws;
    const long ldb = l ? (long)f * k : ld, stride = l ? (long)node : rb, nrows = l ? cnt[l - 1] * k : n;
    const int rows = l ? f * k : rb, rf = l < L ? f : 1;
    if (form_q) launch_level_k<true>(st, cnt[l], l ? rn : r0, base, ldb, stride, rows, nrows, k, rout, rf);
    else launch_level_k<false>(st, cnt[l], l ? rn : r0, base, ldb, stride, rows, nrows, k, rout, rf);
  }
  if (form_q && L > 0) {
    for (int l = L; l >= 1; l--)
      hipLaunchKernelGGL(k_tsqr_down, dim3((unsigned)cnt[l - 1]), dim3(KS_TSQR_NT), sizeof(double) * 2 * k * k, st,
                         (const double *)ws + buf[l], f, k, l < L ? (const double *)ws + mat[l] : nullptr,
                         ws + mat[l - 1], l == 1 ? kp : 0);
    const dim3 g((n + 63) / 64), w(64);
    const double *Mb = ws + mat[0];
#define KS_TSQR_K(X) \
  case X: hipLaunchKernelGGL(k_tsqr_apply<X>, g, w, 0, st, d_V, (long)ld, n, rb, k, Mb); break;
    switch (kp) { KS_TSQR_K(8) KS_TSQR_K(16) KS_TSQR_K(32) KS_TSQR_K(64) KS_TSQR_K(96) }
#undef KS_TSQR_K
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpy2DAsync(R, sizeof(double) * (size_t)ldr, ws, sizeof(double) * (size_t)k,
                                            sizeof(double) * (size_t)k, (size_t)k, hipMemcpyDeviceToHost, st);
  hipError_t es = hipStreamSynchronize(st);   // nothing may still use the workspace
  if (e == hipSuccess) e = es;
  ks_ws_give(ctx, ws);
  KS_CHECK(e == hipSuccess, KS_ERR_HIP, "TSQR launch failed: %s", hipGetErrorString(e));
  return KS_OK;
}
