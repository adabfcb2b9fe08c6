// ks_internal.hpp -- shared pieces of libks_hip.so (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <map>
#include <vector>

#include "../../include/ks_hip.h"

#define KS_BLOCK 256                 // threads per block of the reduction kernels
#define KS_WAVES (KS_BLOCK / 64)
#define KS_MAXB 8192                 // maximum blocks of one row-partitioned reduction
#ifndef KS_GS_SPLITMAX
#define KS_GS_SPLITMAX 128           // Gram-Schmidt against <= this many columns: column-split kernel
#endif
// Loads of data a kernel streams exactly once (basis columns in a sweep): the
// nontemporal hint keeps them from displacing what is reused in L2 (the vector
// being orthogonalized, partial sums).  Measured on the split sweeps at
// n = 2^21: 5.0-5.2 -> 5.3-5.5 TB/s for k = 24..96.
template <typename T>
__device__ __forceinline__ T ks_stream_load(const T *p) {
  return __builtin_nontemporal_load(p);
}
typedef float ks_float2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float2 ks_stream_load2(const float *p) {
  const ks_float2v v = __builtin_nontemporal_load((const ks_float2v *)p);
  return make_float2(v.x, v.y);
}

#ifndef KS_GS_SPLIT_BLOCKS
#define KS_GS_SPLIT_BLOCKS 1024      // workgroups of the column-split Gram-Schmidt (FP64 basis)
#endif
#ifndef KS_GS_SPLIT_BLOCKS32
#define KS_GS_SPLIT_BLOCKS32 2048    // the same for an FP32 basis
#endif
#ifndef KS_GS_WIDE_BLOCKS
#define KS_GS_WIDE_BLOCKS 512        // workgroups (eight wavefronts) of the sweep over more columns than that
#endif
#ifndef KS_GS_RPL2_MAXCW
#define KS_GS_RPL2_MAXCW 12          // FP64 column-split sweeps with <= this many columns per wave: 2 rows per lane
#endif
#ifndef KS_GS_REGMAX
#define KS_GS_REGMAX 16              // Gram-Schmidt against <= this many columns: register-resident kernel
#endif
#ifndef KS_GS_REG_BLOCKS
#define KS_GS_REG_BLOCKS 512         // workgroups of the register-resident Gram-Schmidt
#endif
#ifndef KS_GS_BATCH
#define KS_GS_BATCH 8                // column loads in flight per thread in the Gram-Schmidt sweep
#endif
#define KS_NCOLP (KS_MAX_COLS + 2)   // partial row width: columns + self dot + spare
#ifndef KS_SPMV_NNZ
#define KS_SPMV_NNZ 2048             // products staged in LDS per SpMV row block (a multiple of KS_BLOCK)
#endif
#define KS_SPMV_ROWS 256             // rows per SpMV row block (one per thread)

#define KS_HIP(call)                                                                    \
  do {                                                                                  \
    hipError_t _e = (call);                                                             \
    if (_e != hipSuccess) {                                                             \
      fprintf(stderr, "ks_hip: %s failed: %s (%s:%d)\n", #call, hipGetErrorString(_e),  \
              __FILE__, __LINE__);                                                      \
      return KS_ERR_HIP;                                                                \
    }                                                                                   \
  } while (0)

#define KS_TRY(call)          \
  do {                        \
    int _e = (call);          \
    if (_e) return _e;        \
  } while (0)

#define KS_CHECK(cond, code, ...)                                                       \
  do {                                                                                  \
    if (!(cond)) {                                                                      \
      fprintf(stderr, "ks_hip: " __VA_ARGS__);                                          \
      fputc('\n', stderr);                                                              \
      return (code);                                                                    \
    }                                                                                   \
  } while (0)

struct ks_prof_rec {
  int cls;
  int ran_slot;            // index into the device ran-flag array, -1 if always runs
  double bytes, flops;
  hipEvent_t ev0, ev1;
};

struct ks_ctx_s {
  hipStream_t stream = nullptr;
  ks_status *d_status = nullptr;
  double *d_partial = nullptr;     // [KS_MAXB][KS_NCOLP]
  double *d_sums = nullptr;        // k_gs_fin's column sums [KS_NCOLP] ...
  unsigned *d_counter = nullptr;   // ... and its ticket, zero between launches
  unsigned long long *d_finpub = nullptr;   // k_gs_fin_pub's epoch and epoch-tagged sums [1 + 2 * KS_NCOLP]
  double *d_coef1 = nullptr;                // first-pass coefficients kept for a deferred store [KS_NCOLP]
  double *d_scalar = nullptr;      // small device scratch (norm results)
  double *h_scalar = nullptr;      // pinned host scratch
  ks_status *h_status = nullptr;   // pinned mirror of d_status, filled by ks_status_post
  unsigned long long *d_exp = nullptr;      // the exchange areas of ks_arnoldi_expand, and ...
  unsigned exp_epoch = 0;                   // ... the next launch's first epoch
  int exp_polls = 0;                        // ks_ctx_expand_polls
  bool exp_live = false;                    // the status of an expansion's launch has not been read
  int exp_hold = 0, exp_back = 0;           // expansions left to the launches, and how many after the last time-out
  // a call's workspace, kept for the next call on the context (ks_ws_take)
  void *d_ws = nullptr;
  size_t ws_bytes = 0;
  // profiling
  bool prof = false;
  unsigned prof_mask = ~0u;   // classes that get events while prof is on
  bool prof_open = false;     // the last ks_prof_begin recorded its start event
  bool capturing = false;     // between ks_graph_begin and ks_graph_end
  std::vector<ks_prof_rec> recs;
  std::vector<hipEvent_t> event_pool;
  int *d_ran = nullptr;            // per-launch "did work" flags
  int ran_cap = 0, ran_used = 0;
  ks_prof_entry acc[KS_PROF_NCLASS] = {};
};

// first-fit arena over [base, base+size), blocks aligned to KS_POOL_ALIGN
#define KS_POOL_ALIGN 256
struct ks_arena {
  char *base = nullptr;
  size_t size = 0, used = 0, peak = 0;
  std::map<size_t, size_t> free_;   // offset -> length, coalesced
  std::map<size_t, size_t> taken;   // offset -> length
  void init(char *b, size_t n) {
    base = b; size = n; used = peak = 0;
    free_.clear(); taken.clear();
    if (n) free_[0] = n;
  }
  bool owns(const void *p) const { return base && (const char *)p >= base && (const char *)p < base + size; }
  void *take(size_t n) {
    n = (n + KS_POOL_ALIGN - 1) / KS_POOL_ALIGN * KS_POOL_ALIGN;
    for (auto it = free_.begin(); it != free_.end(); ++it) {
      if (it->second < n) continue;
      size_t off = it->first, len = it->second;
      free_.erase(it);
      if (len > n) free_[off + n] = len - n;
      taken[off] = n;
      used += n;
      if (used > peak) peak = used;
      return base + off;
    }
    return nullptr;
  }
  bool give(const void *p) {
    size_t off = (size_t)((const char *)p - base);
    auto t = taken.find(off);
    if (t == taken.end()) return false;
    size_t len = t->second;
    taken.erase(t);
    used -= len;
    auto nx = free_.lower_bound(off);
    if (nx != free_.end() && off + len == nx->first) { len += nx->second; free_.erase(nx); }
    auto nxt = free_.lower_bound(off);
    if (nxt != free_.begin()) {
      auto pv = std::prev(nxt);
      if (pv->first + pv->second == off) { pv->second += len; return true; }
    }
    free_[off] = len;
    return true;
  }
  size_t largest() const {
    size_t m = 0;
    for (auto &f : free_) m = f.second > m ? f.second : m;
    return m;
  }
};

struct ks_pool_s {
  ks_arena dev, host;
};

struct ks_csr_s {
  int nrows = 0, ncols = 0, max_row = 0, nblocks = 0, variant = 0;
  int64_t nnz = 0;
  ks_prec vprec = KS_F64;
  int32_t *d_rowptr = nullptr, *d_colidx = nullptr, *d_blk = nullptr;
  void *d_val = nullptr;
};

// A workspace for one call on ctx: while no pool is current, the context's own
// (kept up to KS_WS_KEEP bytes: allocating and freeing 75 MB costs a call about
// 0.5 ms), else a block of the pool.  A call takes at most one and has waited for
// the stream, or enqueues nothing after its own work that uses it, when it gives
// it back.
#define KS_WS_KEEP ((size_t)256 << 20)
int ks_ws_take(ks_ctx ctx, size_t bytes, void **p);
void ks_ws_give(ks_ctx ctx, void *p);

// ---------------------------------------------------------------- grouped launches (serving)
#define KS_GROUP_MAX 16   // solves per grouped launch
// members' SpMVs: workgroups b0[m] .. b0[m+1]-1 run member m's row blocks
struct ks_grp_spmv {
  int nmem;
  int b0[KS_GROUP_MAX + 1];
  const int32_t *blk[KS_GROUP_MAX], *rowptr[KS_GROUP_MAX], *colidx[KS_GROUP_MAX];
  const double *val[KS_GROUP_MAX];
  const double *x[KS_GROUP_MAX];
  double *y[KS_GROUP_MAX];
  const ks_status *st[KS_GROUP_MAX];
};
// members' Gram-Schmidt of one column each (FP64 basis)
struct ks_grp_gs_member {
  const double *V;
  double *w, *cbuf, *hcol, *partial, *sums;
  ks_status *st;
  unsigned *counter;
  unsigned long long *pub;         // the context's epoch-tagged finish area (k+2 finishing workgroups), or null
  double *coef1;                   // first-pass coefficient copy for a deferred store (null: none)
  long ld;
  int n, k, rpb, nb, col;
  int cw;                          // the member's own column split (as when it is grouped alone)
};
struct ks_grp_gs {
  int nmem;
  int b0_gs[KS_GROUP_MAX + 1];     // sweep workgroups
  int b0_fin[KS_GROUP_MAX + 1];    // finishing workgroups (k+2 per member, k+1 with a ticket)
  int b0_sc[KS_GROUP_MAX + 1];     // scaling workgroups
  ks_grp_gs_member m[KS_GROUP_MAX];
};
void ks_group_launch_spmv(hipStream_t stream, const ks_grp_spmv &g);
void ks_group_launch_gs(hipStream_t stream, const ks_grp_gs &g, int refine, double eta);
int ks_gs_split_geometry(int n, int k, int *cw, int *rpb, int *nb);   // KS_ERR_RANGE beyond the split kernel
int ks_csr_blocks(ks_csr A, const int32_t **blk, const int32_t **rowptr, const int32_t **colidx, const void **val,
                  int *nblocks, ks_prec *vprec);
int ks_ew_blocks(int n);

// ---------------------------------------------------------------- profiling hooks
// begin() returns a pointer to the device ran-flag for gated kernels (or null).
extern "C" int *ks_prof_begin(ks_ctx ctx, int cls, double bytes, double flops, bool gated);
extern "C" void ks_prof_end(ks_ctx ctx);

// ---------------------------------------------------------------- device helpers
// Workgroups go to the 8 XCDs round-robin (workgroup i to XCD i mod 8), each
// XCD with its own L2.  Row block ks_xcd_block(i) gives XCD x a contiguous eighth
// of the row blocks, so the x entries a block gathers from neighbouring rows
// (a stencil's +-1, +-nx, +-nx*ny) are mostly in the L2 its XCD already filled.
// A bijection on [0, nb) for any nb.
#ifndef KS_SPMV_XCD
#define KS_SPMV_XCD 1
#endif
__device__ __forceinline__ int ks_xcd_block(int i, int nb) {
  if (!KS_SPMV_XCD) return i;
  const int q = nb >> 3, r = nb & 7, x = i & 7, j = i >> 3;
  return x < r ? x * (q + 1) + j : r * (q + 1) + (x - r) * q + j;
}

// lane k's value of v, to every lane (k wave-uniform), as two 32-bit readlanes
__device__ __forceinline__ double ks_readlane_f64(double v, int k) {
  const long long bits = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_readlane((int)bits, k), hi = __builtin_amdgcn_readlane((int)(bits >> 32), k);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Epoch-tagged publication: a 64-bit word holds a 32-bit payload (low half)
// and the epoch it was written in (high half), stored and loaded as one relaxed
// agent-scope atomic, so a reader that sees the current epoch sees the payload
// written with it, with no fence on either side.  A double takes two words.
__device__ __forceinline__ void ks_pub_store(unsigned long long *w, unsigned epoch, unsigned payload) {
  __hip_atomic_store(w, ((unsigned long long)epoch << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void ks_pub_store_f64(unsigned long long *w, unsigned epoch, double x) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(x);
  ks_pub_store(w, epoch, (unsigned)(b & 0xffffffffull));
  ks_pub_store(w + 1, epoch, (unsigned)(b >> 32));
}
__device__ __forceinline__ unsigned long long ks_pub_load(const unsigned long long *w) {
  return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double ks_pub_f64(unsigned long long lo, unsigned long long hi) {
  return __longlong_as_double((long long)(((hi & 0xffffffffull) << 32) | (lo & 0xffffffffull)));
}

// Exchanges between lanes l and l ^ OFF without the LDS pipe (a __shfl_xor is a
// ds_bpermute, about 100 cycles; these are a few).  32 and 16 use gfx950's lane
// swaps: ks_lane_swap leaves {a of the lower half, b of the lower half} in a and
// {a of the upper half, b of the upper half} in b, so a + b holds, in the lower
// lanes, a's sum over the pair and, in the upper lanes, b's.
template <int OFF>
__device__ __forceinline__ void ks_lane_swap(double &a, double &b) {
  static_assert(OFF == 32 || OFF == 16, "lane swaps exist for 32 and 16");
  const long long x = __double_as_longlong(a), y = __double_as_longlong(b);
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  u2 lo, hi;
  if constexpr (OFF == 32) {
    lo = __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  } else {
    lo = __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);
    hi = __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);
  }
  a = __longlong_as_double(((long long)hi.x << 32) | lo.x);
  b = __longlong_as_double(((long long)hi.y << 32) | lo.y);
}
template <int OFF>
__device__ __forceinline__ int ks_lane_xor32(int v) {
  static_assert(OFF == 8 || OFF == 4 || OFF == 2 || OFF == 1, "within a row of 16 lanes");
  if constexpr (OFF == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false);         // row_ror:8
  else if constexpr (OFF == 4) {
    const int t = __builtin_amdgcn_update_dpp(0, v, 0x104, 0xf, 0x5, false);                        // row_shl:4
    return __builtin_amdgcn_update_dpp(t, v, 0x114, 0xf, 0xa, false);                               // row_shr:4
  } else if constexpr (OFF == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4e, 0xf, 0xf, false);   // quad_perm 2301
  else return __builtin_amdgcn_update_dpp(0, v, 0xb1, 0xf, 0xf, false);                             // quad_perm 1032
}
// lane l ^ OFF's value
template <int OFF>
__device__ __forceinline__ double ks_lane_xor(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = ks_lane_xor32<OFF>((int)x), hi = ks_lane_xor32<OFF>((int)(x >> 32));
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// v plus lane l ^ OFF's value
template <int OFF>
__device__ __forceinline__ double ks_lane_xor_add(double v) {
  if constexpr (OFF >= 16) {
    double a = v, b = v;
    ks_lane_swap<OFF>(a, b);
    return a + b;
  } else return v + ks_lane_xor<OFF>(v);
}

// the sum over the wave's 64 lanes, in every lane
__device__ __forceinline__ double ks_wave_sum(double v) {
  v = ks_lane_xor_add<32>(v);
  v = ks_lane_xor_add<16>(v);
  v = ks_lane_xor_add<8>(v);
  v = ks_lane_xor_add<4>(v);
  v = ks_lane_xor_add<2>(v);
  return ks_lane_xor_add<1>(v);
}

// Wave sums of M values per lane by recursive halving: at each step the lanes
// of an xor pair keep opposite halves of their values and add the partner's
// copy of the half they keep, so M values cost about M + 3 log2(64) exchanges
// instead of 6 M.  While M stays even the halving continues (offsets 32, 16,
// ...); the values left are then summed over the remaining lane bits.  On
// return v[i] of lane l holds the wave total of value ks_multi_sum<M>::index(l, i).
// Fixed pairing and order, so the result does not depend on timing.
template <int M, int OFF>
struct ks_multi_halve {
  // every index below is a compile-time constant, so v stays in registers
  __device__ static __forceinline__ void run(double *v, int lane) {
    if constexpr (OFF >= 1) {
      if constexpr (M % 2 == 0) {
        constexpr int half = M / 2;
#pragma unroll
        for (int i = 0; i < half; i++) {
          if constexpr (OFF >= 16) {
            ks_lane_swap<OFF>(v[i], v[half + i]);
            v[i] += v[half + i];
          } else {
            const bool up = (lane & OFF) != 0;
            const double keep = up ? v[half + i] : v[i];
            const double give = up ? v[i] : v[half + i];
            v[i] = keep + ks_lane_xor<OFF>(give);
          }
        }
        ks_multi_halve<half, OFF / 2>::run(v, lane);
      } else {
#pragma unroll
        for (int i = 0; i < M; i++) v[i] = ks_lane_xor_add<OFF>(v[i]);
        ks_multi_halve<M, OFF / 2>::run(v, lane);   // M stays odd
      }
    }
  }
};

template <int M>
struct ks_multi_sum {
  static constexpr int halvings(int m, int off) { return (m % 2 == 0 && off >= 1) ? 1 + halvings(m / 2, off / 2) : 0; }
  static constexpr int H = halvings(M, 32);    // halving steps
  static constexpr int R = M >> H;             // values left per lane
  __device__ static __forceinline__ void run(double *v, int lane) { ks_multi_halve<M, 32>::run(v, lane); }
  // which of the M values lane's v[i] holds after run()
  __device__ static __forceinline__ int index(int lane, int i) {
    int base = 0, m = M;
#pragma unroll
    for (int s = 0; s < H; s++) {
      const int half = m >> 1;
      if (lane & (32 >> s)) base += half;
      m = half;
    }
    return base + i;
  }
  // the lane that stores: lowest lane of its group of equal totals
  __device__ static __forceinline__ bool leader(int lane) { return (lane & ((64 >> H) - 1)) == 0; }
};

// Block-wide sum of one double; result valid in thread 0.  sh: >= KS_WAVES doubles.
__device__ __forceinline__ double ks_block_sum(double v, double *sh) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  v = ks_wave_sum(v);
  __syncthreads();
  if (lane == 0) sh[wave] = v;
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 0; w < KS_WAVES; w++) s += sh[w];
  }
  return s;
}

// rows per thread (1,2,4,8,16) and block count for a row-partitioned reduction
inline void ks_rows_split(int n, int *rpt, int *nblocks) {
  int r = 1;
  while (r < 16 && (int64_t)(n + KS_BLOCK * r - 1) / (KS_BLOCK * r) > 1024) r <<= 1;
  int64_t nb = (n + (int64_t)KS_BLOCK * r - 1) / ((int64_t)KS_BLOCK * r);
  if (nb < 1) nb = 1;
  *rpt = r;
  *nblocks = (int)nb;
}

