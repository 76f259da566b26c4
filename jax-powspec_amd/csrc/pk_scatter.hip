// Particle -> mesh mass assignment: reference stencil (src/mas.py:88-153 and :5-87),
// textbook CIC and TSC.
//
// Sorted owner-computes deposit on row-bundle tiles (1 x ty x n cells, full z rows):
//   1. count:  each block takes a chunk of particles (one block per CU) and histograms their
//              keys (tile, y-class) in LDS, or their x planes when the keys do not fit.
//   2. column: scans of the [blocks][groups] count matrix give every (block, group) its
//              offset inside the group, and the totals.  Groups are what the place sorts by:
//              keys on a small mesh, else x planes (keys are x-plane major).
//   3. place:  the blocks scan the group totals into starts (each its own copy), re-read their
//              chunk and write each record into its group's range (start + block offset + an
//              LDS rank).  Groups = keys: the sort is done.  Groups = x planes:
//      a. plane keys (only where the count could not take keys): one block per plane counts
//                the plane's keys and scans them into key starts;
//      b. fine:  blocks take consecutive segments of the plane-grouped records, histogram
//                their keys over the segment's window of planes in LDS, reserve one run per
//                key with a global atomic and write each key's records as one run.
//      Owner-computes deposits sum in fixed point, so the order inside a key (atomic order)
//      does not change any result.
//   4. deposit: one block per tile stages its ty full rows in LDS (zeros or mesh_in), walks
//              its own buckets plus the neighbour buckets that spill into it (the whole
//              x - 1 / x + 1 tiles, the boundary-row classes of the y neighbours), adds every
//              stencil corner that falls inside with LDS atomics (64-bit fixed point) and
//              writes each row once with coalesced stores: no global atomics, no zero fill.
//   5. atomic: the (normally empty) irregular bucket is added with global atomics.
// A direct mode (tile[0] == 0) adds every particle with global atomics instead.
#include "pk_particles.h"

namespace pk {

// ------------------------------------------------------------------------------------
// small utility kernels (fills instead of hipMemset so a captured graph has no memset node)
// ------------------------------------------------------------------------------------
__global__ void k_fill_f64(double* __restrict__ p, int n, double v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}
__global__ void k_copy_or_zero(const float* src, float* dst, int64_t n) {  // src may alias dst
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    dst[i] = src ? src[i] : 0.0f;
}

constexpr int CNT_NT = 1024;
constexpr int CNT_UNROLL = 8;

// Batched wrappers: blockIdx.y selects the job; blocks beyond the job's own extent return
// at once (the whole block, so no barrier is left waiting).
#define PK_JOB_OR_RETURN(jobs, limit_expr)                              \
  const Job& j = (jobs)[blockIdx.y];                                    \
  if (!j.active || (int)blockIdx.x >= (limit_expr)) return;

// ------------------------------------------------------------------------------------
// 1. count: LDS histogram of one chunk -> matrix row; FP64 weight sum per block
// ------------------------------------------------------------------------------------
struct CountShared {
  double red[CNT_NT];
  unsigned wmax_bits;
};

// AOS / W: the job's input layout and weights, fixed per instantiation (no branch between the
// loads of a thread's particles)
template <int AOS, int W, int ST = -1>
__device__ __forceinline__ void bucket_count_body(const Job& j, int bx, CountShared& sh) {
  // chunks of <= 65535 particles: key k -> 16-bit half (k & 1) of word k >> 1 (half the
  // LDS); larger chunks: one 32-bit counter per key
  extern __shared__ unsigned hist[];
  double* red = sh.red;
  unsigned& wmax_bits = sh.wmax_bits;
  const ScatterArgs a = j.a;
  const TileGeom g = j.g;
  const int tid = threadIdx.x;
  const bool packed = g.chunk <= 65535;
  const int ncol = count_columns(g, a.n);
  unsigned* row = j.mat + (size_t)bx * ncol;
  const bool planes = g.sort == SORT_PLANES;
  {
    const int words = packed ? (ncol + 1) >> 1 : ncol;
    for (int i = tid; i < words; i += CNT_NT) hist[i] = 0u;
  }
  if (tid == 0) wmax_bits = 0u;
  // block 0 clears the estimate's statistics (written from the scans on; no separate fill)
  if (bx == 0 && tid < PK_STATS_LEN) j.stats[tid] = 0.0;
  __syncthreads();
  const int64_t lo = (int64_t)bx * g.chunk;
  const int64_t hi = min(lo + (int64_t)g.chunk, a.np);
  double ws = 0.0;
  float wm = 0.0f, mid = 0.0f;   // mid: the least middle coordinate, if negative
  // CNT_UNROLL particles per thread and iteration: their loads are all in flight before
  // the first key is computed
  for (int64_t i0 = lo + tid; i0 < hi; i0 += (int64_t)CNT_NT * CNT_UNROLL) {
    float px[CNT_UNROLL], py[CNT_UNROLL], pz[CNT_UNROLL], w[CNT_UNROLL];
    // indexes clamped to the chunk: the loads need no branch (the extra ones repeat the
    // last particle and are not counted)
#pragma unroll
    for (int u = 0; u < CNT_UNROLL; ++u)
      load_particle<AOS, W, true>(a, min(i0 + (int64_t)u * CNT_NT, hi - 1), px[u], py[u], pz[u], w[u]);
    __builtin_amdgcn_sched_barrier(0);   // every load issued before the first key
#pragma unroll
    for (int u = 0; u < CNT_UNROLL; ++u) {
      if (i0 + (int64_t)u * CNT_NT >= hi) continue;
      const int key = planes ? row_plane<ST>(a, px[u], py[u], pz[u]) : row_tile_key<ST>(a, g, px[u], py[u], pz[u]);
      if (key >= 0) {
        if (packed) atomicAdd(&hist[key >> 1], 1u << (16 * (key & 1)));
        else atomicAdd(&hist[key], 1u);
        ws += (double)w[u];
        wm = fmaxf(wm, fabsf(w[u]));
        if ((ST >= 0 ? ST : a.stencil) == PK_STENCIL_CIC_REF) mid = fminf(mid, __builtin_amdgcn_fmed3f(px[u], py[u], pz[u]));
      }
    }
  }
  wm *= corner_weight_bound(mid);
  atomicMax(&wmax_bits, __float_as_uint(wm));   // non-negative floats order like their bits
  __syncthreads();
  if (tid == 0) j.wmax[bx] = (double)__uint_as_float(wmax_bits);
  auto count_of = [&](int k) { return packed ? (hist[k >> 1] >> (16 * (k & 1))) & 0xffffu : hist[k]; };
  for (int k = tid; k < ncol; k += CNT_NT) row[k] = count_of(k);
  if (g.sort == SORT_MIXED) {   // the block's x planes: sums over their keys
    const int kpp = g.nyt * g.ncls;
    for (int p = tid; p <= a.n; p += CNT_NT) {
      unsigned sum = 0;
      int q = p % kpp;   // rotated: the lanes' keys fall into different banks
      for (int i = 0; p < a.n && i < kpp; ++i) {
        sum += count_of(p * kpp + q);
        q = q + 1 == kpp ? 0 : q + 1;
      }
      j.pmat[(size_t)bx * (a.n + 1) + p] = p < a.n ? sum : count_of(g.nkeys - 1);
    }
  }
  const double t = block_sum_f64(ws, red, CNT_NT);
  if (tid == 0) j.wsum[bx] = t;
}
template <int AOS, int W, int ST>
__global__ void __launch_bounds__(CNT_NT) k_bucket_count(Job j) {
  __shared__ CountShared sh;
  bucket_count_body<AOS, W, ST>(j, blockIdx.x, sh);
}
__global__ void __launch_bounds__(CNT_NT) k_bucket_count_jobs(const Job* __restrict__ jobs) {
  __shared__ CountShared sh;
  PK_JOB_OR_RETURN(jobs, j.g.nblk);
  // block-uniform choice of the instantiation for this job's layout and weights
  const bool w = j.a.w != nullptr;
  if (j.a.aos) {
    if (w) bucket_count_body<1, 1>(j, blockIdx.x, sh);
    else bucket_count_body<1, 0>(j, blockIdx.x, sh);
  } else {
    if (w) bucket_count_body<0, 1>(j, blockIdx.x, sh);
    else bucket_count_body<0, 0>(j, blockIdx.x, sh);
  }
}

// ------------------------------------------------------------------------------------
// 2. columns of the count matrix: offsets of the blocks inside each group, totals
// ------------------------------------------------------------------------------------
constexpr int COL_NT = 256;
constexpr int COL_KEYS = 32;                  // columns per block: one 128-byte segment per row
constexpr int COL_SUBS = COL_NT / COL_KEYS;   // threads per column, each over a run of rows
constexpr int COL_ROWS = 32;                  // rows per thread and pass (loads in flight)

// Thread (sub, column) walks rows [sub * COL_ROWS, +COL_ROWS) of each pass of COL_SUBS *
// COL_ROWS rows: the run sums of a column's threads meet in LDS, so one pass costs one round
// trip to memory instead of a walk down the whole column.  SCAN: the counts become the
// exclusive sums of the rows above; otherwise the matrix is only summed.
template <bool SCAN>
__device__ __forceinline__ void column_body(unsigned* mat, int ncol, int nblk, int* totals, int bx) {
  __shared__ unsigned part[COL_SUBS][COL_KEYS];
  const int kk = threadIdx.x % COL_KEYS, sub = threadIdx.x / COL_KEYS;
  const int k = bx * COL_KEYS + kk;
  const bool on = k < ncol;
  unsigned carry = 0;
  for (int r0 = 0; r0 < nblk; r0 += COL_SUBS * COL_ROWS) {   // block-uniform
    const int rb = r0 + sub * COL_ROWS;
    unsigned c[COL_ROWS];
    unsigned sum = 0;
#pragma unroll
    for (int u = 0; u < COL_ROWS; ++u) {
      c[u] = (on && rb + u < nblk) ? mat[(size_t)(rb + u) * ncol + k] : 0u;
      sum += c[u];
    }
    part[sub][kk] = sum;
    __syncthreads();
    unsigned run = carry, total = 0;
#pragma unroll
    for (int t = 0; t < COL_SUBS; ++t) {
      const unsigned v = part[t][kk];
      if (t < sub) run += v;
      total += v;
    }
    __syncthreads();   // part is reused by the next pass
    if constexpr (SCAN) {
#pragma unroll
      for (int u = 0; u < COL_ROWS; ++u) {
        if (on && rb + u < nblk) {
          mat[(size_t)(rb + u) * ncol + k] = run;
          run += c[u];
        }
      }
    }
    carry += total;
  }
  if (on && sub == 0) totals[k] = (int)carry;
}

// sums the weight partials into stats[3] = sum(w) / n^3 and sets the fixed-point scale
// aux[0] = S, aux[1] = 1 / S from max |w|
__device__ __forceinline__ void weight_stats_body(const Job& j) {
  __shared__ double shd[COL_NT / 64 + 1];
  __shared__ unsigned long long wmax_bits;
  double ws = 0.0, wm = 0.0;
  if (threadIdx.x == 0) wmax_bits = 0ull;
  for (int i = threadIdx.x; i < j.g.nblk; i += COL_NT) {
    ws += j.wsum[i];
    wm = fmax(wm, j.wmax[i]);
  }
  const double t = block_sum_f64_waves<COL_NT>(ws, shd);   // ends with a barrier
  atomicMax(&wmax_bits, (unsigned long long)__double_as_longlong(wm));
  __syncthreads();
  if (threadIdx.x == 0) {
    const double n = (double)j.a.n;
    j.stats[3] = t / (n * n * n);
    // fixed-point scale S = 2^30 / 2^e, max |w| corner_weight_bound < 2^e: every deposit
    // |rint(w W S)| < 2^31, so it converts through int32
    int e = 0;
    const double wmax = __longlong_as_double((long long)wmax_bits);
    if (wmax > 0.0 && wmax < 1e300) (void)frexp(wmax, &e);
    if (e < -96) e = -96;   // S is used in float
    j.aux[0] = ldexp(1.0, 30 - e);
    j.aux[1] = ldexp(1.0, e - 30);
  }
}

// blocks: the groups' columns, the keys' columns (sums only) where the groups are the planes
// of counted keys, and one for the weights
__host__ __device__ inline int column_blocks(const TileGeom& g, int n) {
  return (group_count(g, n) + COL_KEYS - 1) / COL_KEYS +
         (g.sort == SORT_MIXED ? (g.nkeys + COL_KEYS - 1) / COL_KEYS : 0) + 1;
}
__device__ __forceinline__ void columns_body(const Job& j, int bx) {
  const TileGeom& g = j.g;
  const int G = group_count(g, j.a.n);
  const int ng = (G + COL_KEYS - 1) / COL_KEYS;
  if (bx == column_blocks(g, j.a.n) - 1) weight_stats_body(j);
  else if (bx >= ng) column_body<false>(j.mat, g.nkeys, g.nblk, j.totals, bx - ng);
  else if (g.sort == SORT_MIXED) column_body<true>(j.pmat, G, g.nblk, j.ptotals, bx);
  else column_body<true>(j.mat, G, g.nblk, j.totals, bx);
}
__global__ void __launch_bounds__(COL_NT) k_columns(Job j) { columns_body(j, blockIdx.x); }
__global__ void __launch_bounds__(COL_NT) k_columns_jobs(const Job* __restrict__ jobs) {
  PK_JOB_OR_RETURN(jobs, column_blocks(j.g, j.a.n));
  columns_body(j, blockIdx.x);
}

// ------------------------------------------------------------------------------------
// 3. place (both passes): rounds of records are ranked per destination run in LDS, staged
// there in destination order and written by consecutive lanes to consecutive addresses, so
// a wave's stores touch a few runs instead of one line per lane
// ------------------------------------------------------------------------------------

// Exclusive scan of the counts a[0, len) in LDS by the whole block of NT threads (each takes
// a contiguous span): f(i, count, prefix) for every entry, in the thread that owns it.
// Returns the grand total.  Every thread must call it (it holds a barrier).
template <int NT, class F>
__device__ __forceinline__ unsigned block_scan_apply(const unsigned* a, int len, unsigned* wtot, F&& f) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int per = (len + NT - 1) / NT;
  const int i0 = min(tid * per, len), i1 = min(i0 + per, len);
  unsigned own = 0;
  for (int i = i0; i < i1; ++i) own += a[i];
  unsigned incl = own;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const unsigned v = __shfl_up(incl, off, 64);
    if (lane >= off) incl += v;
  }
  if (lane == 63) wtot[wv] = incl;
  __syncthreads();
  unsigned pre = 0, total = 0;
#pragma unroll
  for (int k = 0; k < NT / 64; ++k) {
    const unsigned t = wtot[k];
    if (k < wv) pre += t;
    total += t;
  }
  unsigned e = pre + incl - own;
  for (int i = i0; i < i1; ++i) {
    const unsigned c = a[i];
    f(i, c, e);
    e += c;
  }
  return total;
}

// ------------------------------------------------------------------------------------
// 3. place by group: group start + block offset inside the group + LDS rank
// ------------------------------------------------------------------------------------
constexpr int PLACE_PER = 7;                     // most particles per thread and round
constexpr size_t PLACE_LDS = 150 * 1024;         // tables + staging
// particles per round: 20 staged bytes each (x, y, z, w, destination) next to three tables
// of one word per group, a multiple of the block size
__host__ __device__ constexpr int place_round(int groups) {
  return (int)((PLACE_LDS - 12 * (size_t)groups) / 20) / CNT_NT * CNT_NT > CNT_NT * PLACE_PER
             ? CNT_NT * PLACE_PER
             : (int)((PLACE_LDS - 12 * (size_t)groups) / 20) / CNT_NT * CNT_NT;
}
size_t place_lds(int groups) { return 12 * (size_t)groups + 20 * (size_t)place_round(groups); }

// Every block scans the group totals into its own group starts (no launch and no round trip
// between the column scan and the place) and adds its offsets: dest[] (lcnt: scratch).  The
// starts that later passes read go to memory too: key_start (groups = keys: by block 0;
// planes of counted keys: each block the keys of some planes), or plane_start.
template <int ST>
__device__ __forceinline__ void place_starts(const Job& j, int bx, unsigned* dest, unsigned* lcnt, unsigned* wtot) {
  const TileGeom& g = j.g;
  const int n = j.a.n, G = group_count(g, n), tid = threadIdx.x;
  const unsigned* row = (g.sort == SORT_MIXED ? j.pmat : j.mat) + (size_t)bx * G;
  const int* tot = g.sort == SORT_MIXED ? j.ptotals : j.totals;
  for (int i = tid; i < G; i += CNT_NT) {
    lcnt[i] = (unsigned)tot[i];
    dest[i] = row[i];
  }
  __syncthreads();
  int* starts = g.sort == SORT_KEYS ? j.key_start : j.plane_start;
  const bool write = bx == 0 && g.sort != SORT_MIXED;
  const unsigned all = block_scan_apply<CNT_NT>(lcnt, G, wtot, [&](int i, unsigned, unsigned e) {
    dest[i] += e;
    lcnt[i] = e;
    if (write) starts[i] = (int)e;
  });
  if (write && tid == 0) starts[G] = (int)all;
  if (g.sort == SORT_MIXED) {
    __syncthreads();   // lcnt: plane starts
    const int kpp = g.nyt * g.ncls, lane = tid & 63;
    constexpr int NW = CNT_NT / 64;
    // one wave per plane; the planes are dealt over the blocks' waves
    for (int p = bx * NW + (tid >> 6); p <= n; p += g.nblk * NW) {
      const int k0 = p * kpp, kn = p < n ? kpp : 1;
      int run = (int)lcnt[p];
      for (int q0 = 0; q0 < kn; q0 += 64) {
        const int q = q0 + lane;
        const int c = q < kn ? j.totals[k0 + q] : 0;
        int incl = c;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const int v = __shfl_up(incl, off, 64);
          if (lane >= off) incl += v;
        }
        if (q < kn) {
          j.key_start[k0 + q] = run + incl - c;
          j.koff[k0 + q] = 0u;   // the fine pass counts each key's records from zero
        }
        run += __shfl(incl, 63, 64);
      }
      if (p == n && lane == 0) j.key_start[g.nkeys] = run;
    }
  }
  __syncthreads();   // dest complete, lcnt free
}

template <int AOS, int W, int ST = -1>
__device__ __forceinline__ void bucket_place_body(const Job& j, int bx, unsigned* wtot) {
  extern __shared__ unsigned lds[];
  const ScatterArgs a = j.a;
  const TileGeom g = j.g;
  const int tid = threadIdx.x;
  const int G = group_count(g, a.n);
  const bool by_key = g.sort == SORT_KEYS;
  const int S = place_round(G);     // particles per round
  unsigned* dest = lds;             // next write position of each group for this block
  unsigned* lcnt = lds + G;         // the round's count, then local start, of each group
  unsigned* delta = lds + 2 * G;    // global position - local slot, per group
  float* sx = reinterpret_cast<float*>(lds + 3 * G);
  float* sy = sx + S;
  float* sz = sy + S;
  float* sw = sz + S;
  unsigned* sd = reinterpret_cast<unsigned*>(sw + S);   // global position of each slot
  void* out = by_key ? j.sorted : j.staged;
  const int64_t lo = (int64_t)bx * g.chunk;
  const int64_t hi = min(lo + (int64_t)g.chunk, a.np);
  const bool has_w = a.w != nullptr;
  // software pipeline: the next round's particles load while this round is ranked, staged
  // and stored
  float px[PLACE_PER], py[PLACE_PER], pz[PLACE_PER], w[PLACE_PER];
  // indexes clamped to the chunk: no branch between the loads (the extra loads repeat the
  // chunk's last particle and are not placed)
  auto load_round = [&](int64_t r0, float* x, float* y, float* z, float* ww) {
#pragma unroll
    for (int u = 0; u < PLACE_PER; ++u)
      load_particle<AOS, W, true>(a, min(r0 + (int64_t)u * CNT_NT + tid, hi - 1), x[u], y[u], z[u], ww[u]);
  };
  if (lo < hi) load_round(lo, px, py, pz, w);
  place_starts<ST>(j, bx, dest, lcnt, wtot);
  if (lo >= hi) return;   // whole block: an empty chunk
  for (int64_t r0 = lo; r0 < hi; r0 += S) {   // block-uniform
    int pl[PLACE_PER];
#pragma unroll
    for (int u = 0; u < PLACE_PER; ++u) {
      const int64_t i = r0 + (int64_t)u * CNT_NT + tid;
      pl[u] = (u * CNT_NT >= S || i >= hi) ? -1
              : by_key                   ? row_tile_key<ST>(a, g, px[u], py[u], pz[u])
                                         : row_plane<ST>(a, px[u], py[u], pz[u]);
    }
    float nx[PLACE_PER], ny[PLACE_PER], nz[PLACE_PER], nw[PLACE_PER];
    load_round(r0 + S, nx, ny, nz, nw);
    for (int q = tid; q < G; q += CNT_NT) lcnt[q] = 0u;
    __syncthreads();
    unsigned rk[PLACE_PER];
#pragma unroll
    for (int u = 0; u < PLACE_PER; ++u)
      if (pl[u] >= 0) rk[u] = atomicAdd(&lcnt[pl[u]], 1u);
    __syncthreads();
    const unsigned m = block_scan_apply<CNT_NT>(lcnt, G, wtot, [&](int p, unsigned c, unsigned e) {
      lcnt[p] = e;
      if (c) {   // this thread alone owns group p here
        const unsigned b = dest[p];
        dest[p] = b + c;
        delta[p] = b - e;
      }
    });
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PLACE_PER; ++u)
      if (pl[u] >= 0) {
        const unsigned slot = lcnt[pl[u]] + rk[u];
        sx[slot] = px[u];
        sy[slot] = py[u];
        sz[slot] = pz[u];
        sw[slot] = w[u];
        sd[slot] = delta[pl[u]] + slot;
      }
    __syncthreads();
    for (int q = tid; q < (int)m; q += CNT_NT) store_record(out, sd[q], has_w, sx[q], sy[q], sz[q], sw[q]);
#pragma unroll
    for (int u = 0; u < PLACE_PER; ++u) {
      px[u] = nx[u];
      py[u] = ny[u];
      pz[u] = nz[u];
      w[u] = nw[u];
    }
    __syncthreads();   // the staging is read before the next round overwrites it
  }
}
template <int AOS, int W, int ST>
__global__ void __launch_bounds__(CNT_NT) k_bucket_place(Job j) {
  __shared__ unsigned wtot[CNT_NT / 64];
  bucket_place_body<AOS, W, ST>(j, blockIdx.x, wtot);
}
__global__ void __launch_bounds__(CNT_NT) k_bucket_place_jobs(const Job* __restrict__ jobs) {
  __shared__ unsigned wtot[CNT_NT / 64];
  PK_JOB_OR_RETURN(jobs, j.g.nblk);
  const bool w = j.a.w != nullptr;
  if (j.a.aos) {
    if (w) bucket_place_body<1, 1>(j, blockIdx.x, wtot);
    else bucket_place_body<1, 0>(j, blockIdx.x, wtot);
  } else {
    if (w) bucket_place_body<0, 1>(j, blockIdx.x, wtot);
    else bucket_place_body<0, 0>(j, blockIdx.x, wtot);
  }
}

// the plain launches' instantiation for a job's layout, weights and stencil
template <template <int, int, int> class Pick, int AOS, int W>
auto pick_st(const ScatterArgs& a) -> decltype(Pick<0, 0, 0>::k) {
  if (a.stencil == PK_STENCIL_CIC_REF) return Pick<AOS, W, PK_STENCIL_CIC_REF>::k;
  if (a.stencil == PK_STENCIL_CIC) return Pick<AOS, W, PK_STENCIL_CIC>::k;
  return Pick<AOS, W, PK_STENCIL_TSC>::k;
}
template <template <int, int, int> class Pick>
auto pick_aw(const ScatterArgs& a) -> decltype(Pick<0, 0, 0>::k) {
  const bool w = a.w != nullptr;
  if (a.aos) return w ? pick_st<Pick, 1, 1>(a) : pick_st<Pick, 1, 0>(a);
  return w ? pick_st<Pick, 0, 1>(a) : pick_st<Pick, 0, 0>(a);
}
template <int AOS, int W, int ST> struct CountK { static constexpr void (*k)(Job) = k_bucket_count<AOS, W, ST>; };
template <int AOS, int W, int ST> struct PlaceK { static constexpr void (*k)(Job) = k_bucket_place<AOS, W, ST>; };

// ------------------------------------------------------------------------------------
// 3a. the keys of one x plane's records, counted in LDS and scanned into key starts (where the
// count took planes; block n takes the irregular key)
// ------------------------------------------------------------------------------------
constexpr int PKEY_NT = 1024;
constexpr int PKEY_UNROLL = 8;
__device__ __forceinline__ void plane_keys_body(const Job& j, int p) {
  extern __shared__ unsigned lds[];   // [keys per plane]
  __shared__ unsigned wtot[PKEY_NT / 64];
  const ScatterArgs a = j.a;
  const TileGeom g = j.g;
  const int tid = threadIdx.x;
  const int lo = j.plane_start[p], hi = j.plane_start[p + 1];
  if (p == a.n) {
    if (tid == 0) {
      j.key_start[g.nkeys - 1] = lo;
      j.key_start[g.nkeys] = hi;
      j.koff[g.nkeys - 1] = 0u;
    }
    return;
  }
  const int kpp = g.nyt * g.ncls;
  for (int i = tid; i < kpp; i += PKEY_NT) lds[i] = 0u;
  __syncthreads();
  const int stride = a.w != nullptr ? 4 : 3;
  const float* y = static_cast<const float*>(j.staged) + 1;   // y of record i at y[i stride]
  for (int64_t i0 = lo + tid; i0 < hi; i0 += PKEY_NT * PKEY_UNROLL) {
    float py[PKEY_UNROLL];
#pragma unroll
    for (int u = 0; u < PKEY_UNROLL; ++u) py[u] = y[min(i0 + u * PKEY_NT, (int64_t)hi - 1) * stride];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < PKEY_UNROLL; ++u)
      if (i0 + u * PKEY_NT < hi) atomicAdd(&lds[row_key_in_plane(a, g, py[u])], 1u);
  }
  __syncthreads();
  block_scan_apply<PKEY_NT>(lds, kpp, wtot, [&](int q, unsigned, unsigned e) {
    j.key_start[p * kpp + q] = lo + (int)e;
    j.koff[p * kpp + q] = 0u;
  });
}
__global__ void __launch_bounds__(PKEY_NT) k_plane_keys(Job j) { plane_keys_body(j, blockIdx.x); }
__global__ void __launch_bounds__(PKEY_NT) k_plane_keys_jobs(const Job* __restrict__ jobs) {
  const Job& j = jobs[blockIdx.y];
  if (!j.active || j.g.sort != SORT_PLANES) return;
  plane_keys_body(j, blockIdx.x);
}

// ------------------------------------------------------------------------------------
// 3b. fine place: a segment of the plane-grouped records -> one run per (segment, key)
// ------------------------------------------------------------------------------------
constexpr int FINE_NT = 256;                      // small blocks, several per CU: their
constexpr int FINE_PER = 6;                       // load, rank and store phases overlap
constexpr int FINE_SEG = FINE_NT * FINE_PER;      // records per block
constexpr int FINE_WIN = 1024;                    // keys of the LDS window
constexpr size_t FINE_LDS = (size_t)FINE_SEG * 20;   // staging: x, y, z, w, destination

int fine_place_blocks(int64_t np) { return (int)((np > 0 ? np + FINE_SEG - 1 : FINE_SEG) / FINE_SEG); }

template <int ST = -1>
__device__ __forceinline__ void fine_place_body(const Job& j, int bx) {
  extern __shared__ unsigned lds[];
  __shared__ unsigned cnt[FINE_WIN];     // per key of the window: count, then local start
  __shared__ unsigned delta[FINE_WIN];   // global position - local slot
  __shared__ unsigned wtot[FINE_NT / 64];
  __shared__ int win[2];
  const ScatterArgs a = j.a;
  const TileGeom g = j.g;
  const int tid = threadIdx.x;
  const int64_t total = j.key_start[g.nkeys];   // records kept
  const int64_t s0 = (int64_t)bx * FINE_SEG;
  if (s0 >= total) return;   // whole block
  const int64_t s1 = min(s0 + (int64_t)FINE_SEG, total);
  const bool has_w = a.w != nullptr;
  const unsigned kpp = (unsigned)(g.nyt * g.ncls);
  float* sx = reinterpret_cast<float*>(lds);
  float* sy = sx + FINE_SEG;
  float* sz = sy + FINE_SEG;
  float* sw = sz + FINE_SEG;
  unsigned* sd = reinterpret_cast<unsigned*>(sw + FINE_SEG);
  // the records are grouped by plane, so the first and last records bound the segment's planes
  if (tid < 2) {
    const float4 r = load_record(j.staged, (size_t)(tid == 0 ? s0 : s1 - 1), has_w);
    win[tid] = row_plane<ST>(a, r.x, r.y, r.z);
  }
  float4 r[FINE_PER];
  int key[FINE_PER];
#pragma unroll
  for (int u = 0; u < FINE_PER; ++u)   // clamped: no branch between the loads
    r[u] = load_record_stream(j.staged, (size_t)min(s0 + tid + (int64_t)u * FINE_NT, s1 - 1), has_w);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < FINE_PER; ++u) {
    const int64_t i = s0 + tid + (int64_t)u * FINE_NT;
    r[u].w = record_weight(r[u], has_w);
    key[u] = i < s1 ? row_tile_key<ST>(a, g, r[u].x, r[u].y, r[u].z) : -1;   // of the plane the place saw
  }
  __syncthreads();
  const int kbase = win[0] * (int)kpp;
  const int wlen = min((win[1] + 1) * (int)kpp, g.nkeys) - kbase;
  if (wlen > FINE_WIN) {
    // a sparse segment spanning too many planes (small catalogues): one global atomic each
#pragma unroll
    for (int u = 0; u < FINE_PER; ++u)
      if (key[u] >= 0) {
        const unsigned at = (unsigned)j.key_start[key[u]] + atomicAdd(&j.koff[key[u]], 1u);
        store_record(j.sorted, at, has_w, r[u].x, r[u].y, r[u].z, r[u].w);
      }
    return;
  }
  for (int q = tid; q < wlen; q += FINE_NT) cnt[q] = 0u;
  __syncthreads();
  unsigned rank[FINE_PER];
#pragma unroll
  for (int u = 0; u < FINE_PER; ++u)
    if (key[u] >= 0) rank[u] = atomicAdd(&cnt[key[u] - kbase], 1u);
  __syncthreads();
  const unsigned m = block_scan_apply<FINE_NT>(cnt, wlen, wtot, [&](int q, unsigned c, unsigned e) {
    cnt[q] = e;
    if (c) delta[q] = (unsigned)j.key_start[kbase + q] + atomicAdd(&j.koff[kbase + q], c) - e;
  });
  __syncthreads();
#pragma unroll
  for (int u = 0; u < FINE_PER; ++u)
    if (key[u] >= 0) {
      const int q = key[u] - kbase;
      const unsigned slot = cnt[q] + rank[u];
      sx[slot] = r[u].x;
      sy[slot] = r[u].y;
      sz[slot] = r[u].z;
      sw[slot] = r[u].w;
      sd[slot] = delta[q] + slot;
    }
  __syncthreads();
  for (int q = tid; q < (int)m; q += FINE_NT) store_record(j.sorted, sd[q], has_w, sx[q], sy[q], sz[q], sw[q]);
}
template <int ST>
__global__ void __launch_bounds__(FINE_NT) k_fine_place(Job j) { fine_place_body<ST>(j, blockIdx.x); }
__global__ void __launch_bounds__(FINE_NT) k_fine_place_jobs(const Job* __restrict__ jobs) {
  const Job& j = jobs[blockIdx.y];
  if (!j.active || j.g.sort == SORT_KEYS) return;
  fine_place_body(j, blockIdx.x);
}

// ------------------------------------------------------------------------------------
// 4. deposit (mesh mode): one block per row-bundle tile
// ------------------------------------------------------------------------------------
constexpr int DEP_NT = 1024;
constexpr int DEP_U = 4;                                             // records in flight per thread
constexpr int DEP_CELLS = (int)(FIXED_LDS_MAX / 8 / DEP_NT);         // cells per thread, at most

// One block per tile.  Bound by memory latency (one 128 KB block per CU leaves 16 waves): the
// base mesh is read into registers before the deposit and every load and store of the flush
// is in flight together (one cell at a time, each waiting for its read, the kernel took 1036
// us at 512^3 with 2e7 weighted particles; now 454).
// FIXED: 64-bit fixed-point cells (at most DEP_CELLS per thread), else float.
// V4: rows and mesh pointers allow 16-byte accesses.
template <bool FIXED, bool V4, int ST>
__global__ void __launch_bounds__(DEP_NT) k_rows_deposit(ScatterArgs a, TileGeom g, const int* __restrict__ key_start,
                                                         const void* __restrict__ sorted, const double* __restrict__ aux,
                                                         const float* mesh_in, float* mesh_out,
                                                         double* __restrict__ tile_mass) {
  extern __shared__ unsigned long long acc_q[];   // [ty][n]: 64-bit fixed point, or float when !FIXED
  float* acc_f = reinterpret_cast<float*>(acc_q);
  __shared__ TileBuckets B;
  __shared__ double red[DEP_NT / 64 + 1];
  __shared__ long long redi[DEP_NT / 64 + 1];
  const int tid = threadIdx.x;
  const int n = a.n;
  const int xt = blockIdx.x / g.nyt, yt = blockIdx.x % g.nyt;
  const int y0 = yt * g.ty;
  const int cells = g.ty * n;
  const size_t gbase = ((size_t)xt * n + y0) * n;   // rows y0 .. y0+ty-1 are contiguous
  constexpr bool tsc = ST == PK_STENCIL_TSC;
  // the tile buckets hold no irregular record (those are added with global atomics)
  const int nbk = tile_bucket_count(g, n, tsc, false);
  int lo = 0, hi = 0;
  if (tid < nbk) {
    const int key = tile_bucket_key(g, n, tsc, xt, yt, tid);
    lo = key_start[key];
    hi = key_start[key + 1];
  }
  // mesh_in may alias mesh_out: a thread reads its cells here and writes the same ones below
  constexpr int W = V4 ? 4 : 1, PER = DEP_CELLS / W;
  typedef float fw __attribute__((ext_vector_type(W)));
  fw base[FIXED ? PER : 1];
  if constexpr (FIXED) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = (tid + u * DEP_NT) * W;
      base[u] = 0.0f;
      if (mesh_in && i < cells) base[u] = *reinterpret_cast<const fw*>(mesh_in + gbase + i);
    }
  }
  for (int i = tid; i < cells; i += DEP_NT) {
    if (FIXED) acc_q[i] = 0ull;
    else acc_f[i] = 0.0f;
  }
  publish_buckets(B, nbk, lo, hi);
  __syncthreads();
  const float scale = (float)aux[0];
  const int total = B.pre[B.nbk];
  const bool has_w = a.w != nullptr;
  for (int idx0 = tid; idx0 < total; idx0 += DEP_NT * DEP_U) {
    float4 r[DEP_U];
#pragma unroll
    for (int u = 0; u < DEP_U; ++u) r[u] = bucket_record(B, sorted, idx0 + u * DEP_NT, has_w);
    __builtin_amdgcn_sched_barrier(0);   // every load issued before the first deposit
#pragma unroll
    for (int u = 0; u < DEP_U; ++u) {
      if (idx0 + u * DEP_NT >= total) continue;
      auto add = [&](int iy, int iz, float wt) {
        const int ly = iy - y0;
        if ((unsigned)ly >= (unsigned)g.ty) return;
        if (FIXED) atomicAdd(&acc_q[ly * n + iz], to_fixed(wt));
        else atomicAdd(&acc_f[ly * n + iz], wt);
      };
      // the weight carries the power-of-two scale: each corner is (W w) S exactly
      const float w = record_weight(r[u], has_w) * (FIXED ? scale : 1.0f);
      if (ST == PK_STENCIL_CIC_REF) ref_corners_on_x_regular(a, r[u].x, r[u].y, r[u].z, w, xt, add);
      else for_each_corner_on_x<ST>(a, r[u].x, r[u].y, r[u].z, w, xt, add);
    }
  }
  __syncthreads();
  const double inv = aux[1];
  if constexpr (FIXED) {
    long long isum = 0;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int i = (tid + u * DEP_NT) * W;
      if (i >= cells) continue;
      fw v;
#pragma unroll
      for (int e = 0; e < W; ++e) {
        const long long q = (long long)acc_q[i + e];
        isum += q;
        v[e] = (float)((double)q * inv);
      }
      if (mesh_in) v += base[u];
      *reinterpret_cast<fw*>(mesh_out + gbase + i) = v;
    }
    const long long t = block_sum_i64_waves<DEP_NT>(isum, redi);   // exact
    if (tid == 0) tile_mass[blockIdx.x] = (double)t * inv;
  } else {
    double msum = 0.0;
    for (int i = tid; i < cells; i += DEP_NT) {
      const float v = acc_f[i];
      msum += (double)v;
      mesh_out[gbase + i] = mesh_in ? mesh_in[gbase + i] + v : v;
    }
    const double m = block_sum_f64_waves<DEP_NT>(msum, red);
    if (tid == 0) tile_mass[blockIdx.x] = m;
  }
}

template <bool FIXED, bool V4> auto rows_deposit_st(int stencil) -> decltype(&k_rows_deposit<FIXED, V4, 0>) {
  if (stencil == PK_STENCIL_CIC_REF) return k_rows_deposit<FIXED, V4, PK_STENCIL_CIC_REF>;
  if (stencil == PK_STENCIL_CIC) return k_rows_deposit<FIXED, V4, PK_STENCIL_CIC>;
  return k_rows_deposit<FIXED, V4, PK_STENCIL_TSC>;
}

// ------------------------------------------------------------------------------------
// 5. global-atomic deposit: all particles (direct mode) or the irregular bucket
// ------------------------------------------------------------------------------------
constexpr int ATM_NT = 256;

__global__ void __launch_bounds__(ATM_NT) k_atomic_deposit(ScatterArgs a, const void* __restrict__ sorted,
                                                           const int* __restrict__ range, float* __restrict__ mesh,
                                                           double* __restrict__ stats) {
  __shared__ double red[ATM_NT];
  int64_t lo = 0, hi = a.np;
  if (range) {
    lo = range[0];
    hi = range[1];
  }
  const int n = a.n;
  double msum = 0.0;
  for (int64_t i = lo + blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < hi; i += (int64_t)gridDim.x * blockDim.x) {
    float px, py, pz, w;
    if (sorted) {
      const float4 r = load_record(sorted, (size_t)i, a.w != nullptr);
      px = r.x; py = r.y; pz = r.z; w = r.w;
    } else {
      load_particle(a, i, px, py, pz, w);
    }
    if (!pos_ok(px, py, pz)) continue;
    for_each_corner(a, px, py, pz, w, [&](int ix, int iy, int iz, float wt) {
      atomicAdd(&mesh[((size_t)ix * n + iy) * n + iz], wt);
      msum += (double)wt;
    });
  }
  const double m = block_sum_f64(msum, red, ATM_NT);
  if (threadIdx.x == 0 && m != 0.0) atomicAdd(&stats[2], m);
}

// ------------------------------------------------------------------------------------
// mass finalize: stats[0] = M (fixed-order sum of tile masses + atomic part), stats[1] = n^3 / M
// ------------------------------------------------------------------------------------
// fixed-order FP64 sum of the tile masses: each thread adds its slots in order (eight
// loads in flight per step), then wave butterflies and the wave totals
constexpr int MASS_NT = 1024;
__device__ __forceinline__ void mass_finalize_body(const Job& j, int ntiles) {
  __shared__ double red[MASS_NT / 64 + 1];
  constexpr int MU = 8;
  double s = 0.0;
  for (int i0 = threadIdx.x; i0 < ntiles; i0 += MASS_NT * MU) {
    double v[MU];
#pragma unroll
    for (int u = 0; u < MU; ++u) {
      const int i = i0 + u * MASS_NT;
      v[u] = i < ntiles ? j.tile_mass[i] : 0.0;
    }
#pragma unroll
    for (int u = 0; u < MU; ++u) s += v[u];
  }
  const double m = block_sum_f64_waves<MASS_NT>(s, red) + j.stats[2];
  if (threadIdx.x == 0) {
    const double n = (double)j.a.n;
    j.stats[0] = m;
    j.stats[1] = n * n * n / m;
  }
  if (j.tile_sq != nullptr) {   // fused tiles: the sum of (rho - c)^2 in a fixed order -> aux[2]
    double q = 0.0;
    for (int i = threadIdx.x; i < ntiles; i += MASS_NT) q += j.tile_sq[i];
    const double tq = block_sum_f64_waves<MASS_NT>(q, red);
    if (threadIdx.x == 0) j.aux[2] = tq;
  }
}
__global__ void __launch_bounds__(MASS_NT) k_mass_finalize(Job j, int ntiles) { mass_finalize_body(j, ntiles); }


// ------------------------------------------------------------------------------------
// host side
// ------------------------------------------------------------------------------------
constexpr size_t LDS_MAX = 160 * 1024;
// Sort by the keys themselves up to this many (SORT_KEYS): the fine pass is saved, but a round's
// records spread over more runs and more of the LDS goes to tables.  Whole estimates, us, by key
// against by plane and then by key (SORT_MIXED): 1025 keys (128^3) 72 / 80 with 1e6 particles
// and 585 / 668 with 3e7; 3457 keys (192^3 TSC) 235 / 242 with 5e6 and 996 / 1009 with 3e7;
// 4097 keys (256^3) 136 / 138 with 1e6 but 526 / 516 with 2e7.
constexpr long SORT_KEYS_MAX = 4000;
// Count keys up to this many (SORT_MIXED: 32-bit counters in LDS), x planes beyond (n = 768 and
// 1024, tiles of few rows).  Counting planes alone reads the staged records once more for their
// keys: 384^3 with 3e7 particles took 1101 us that way against 1004.  Keys that do not fit LDS
// went to per-block tables in HBM before (global atomics): 1314 us of counting and 77 us of
// column scan at 1024^3 with 3e7 particles, against 70 + 6 us and 95 us for the plane keys.
constexpr long COUNT_KEYS_MAX = (LDS_MAX - 16384) / 4;
constexpr long KEYS_MAX = 1L << 24;
constexpr int CHUNK_MIN = 4096;          // smallest counting chunk (small catalogues)
constexpr int CHUNK_MAX = 1 << 22;       // largest (32-bit LDS counters above 65535)

static int largest_divisor_le(int n, int cap) {
  for (int d = cap < n ? cap : n; d >= 2; --d)
    if (n % d == 0) return d;
  return n;
}

static int sort_of(long nkeys) {
  return nkeys <= SORT_KEYS_MAX ? SORT_KEYS : nkeys <= COUNT_KEYS_MAX ? SORT_MIXED : SORT_PLANES;
}

SortScratch sort_scratch(const TileGeom& g, int n) {
  return {count_columns(g, n), g.sort == SORT_MIXED, g.sort == SORT_PLANES, g.sort != SORT_KEYS};
}

SortScratch batch_sort_scratch(const TileGeom& cap, int n) {
  SortScratch r = sort_scratch(cap, n);
  for (int ncls = 2; ncls < cap.ncls; ++ncls) {
    TileGeom g = cap;
    g.ncls = ncls;
    g.nkeys = cap.ntiles * ncls + 1;
    g.sort = sort_of(g.nkeys);
    const SortScratch s = sort_scratch(g, n);
    r = {s.columns > r.columns ? s.columns : r.columns, r.mixed || s.mixed, r.planes || s.planes, r.staged || s.staged};
  }
  return r;
}

void set_chunk(TileGeom* g, int64_t np, int64_t chunk) {
  if (chunk < CHUNK_MIN) chunk = CHUNK_MIN;
  if (chunk > CHUNK_MAX) chunk = CHUNK_MAX;
  g->chunk = (int)chunk;
  g->nblk = (int)((np + chunk - 1) / chunk);
  if (g->nblk < 1) g->nblk = 1;
}

int make_tile_geom(int n, int64_t np, int stencil, const int* tile, TileGeom* g, bool* direct) {
  *direct = false;
  *g = TileGeom{};
  int ty = 0;
  if (tile) {
    if (tile[0] == 0) {
      *direct = true;
      return PK_OK;
    }
    ty = tile[1];
    if (tile[0] != 1 || (tile[2] != 0 && tile[2] != n))
      return set_error(PK_E_INVALID, "sorted deposit tiles are (1, ty, n) row bundles, got (%d, %d, %d)", tile[0],
                       tile[1], tile[2]);
    if (ty < 1 || ty > n || n % ty != 0) return set_error(PK_E_INVALID, "rows per tile %d must divide n=%d", ty, n);
    if (ty < 2 && n >= 2) return set_error(PK_E_INVALID, "rows per tile must be >= 2");
  } else {
    // largest divisor <= 32 whose rows fit the 64-bit fixed-point deposit (n <= 512: 32;
    // 768 and 1024: 16)
    ty = largest_divisor_le(n, 32);
    while (ty > 2 && ((size_t)ty * n * 8 > FIXED_LDS_MAX || n % ty != 0)) --ty;
    if (n % ty != 0) {   // no divisor's rows fit (odd sides above 127 without one up to 32): global atomics
      *direct = true;
      return PK_OK;
    }
  }
  g->ty = ty;
  g->nyt = n / ty;
  // exact for y * ty < 2^32 (y < n <= 4096): the multiplier exceeds 2^32 / ty by under 1
  g->ty_mul = (unsigned)((0xffffffffull + (unsigned long long)ty) / (unsigned long long)ty);
  g->ncls = stencil == PK_STENCIL_TSC ? 3 : 2;
  const long ntiles = (long)n * g->nyt;
  const long nkeys = ntiles * g->ncls + 1;
  const size_t rows_bytes = (size_t)ty * n * sizeof(float);
  if (rows_bytes > LDS_MAX - 8192) return set_error(PK_E_INVALID, "tile of %d rows x %d needs too much LDS", ty, n);
  g->ntiles = (int)ntiles;
  g->nkeys = (int)nkeys;
  g->fixed = (size_t)ty * n * 8 <= FIXED_LDS_MAX ? 1 : 0;
  g->sort = sort_of(nkeys);
  // one counting / placing block per CU when the catalogue is large (a second, partial
  // round of blocks would cost a whole round), at least CHUNK_MIN particles per block
  int dev = 0;
  (void)hipGetDevice(&dev);
  const int64_t ncu = num_cus(dev);
  set_chunk(g, np, (np + ncu - 1) / ncu);
  if (g->nblk < 1) g->nblk = 1;
  if (nkeys > KEYS_MAX) return set_error(PK_E_INVALID, "too many buckets");
  return PK_OK;
}

namespace {
int grid_for(int64_t items, int nt, int cap) {
  int64_t gsz = (items + nt - 1) / nt;
  if (gsz < 1) gsz = 1;
  if (gsz > cap) gsz = cap;
  return (int)gsz;
}

template <typename K> int allow_lds(K kernel, size_t bytes) {
  return bytes <= 65536 ? PK_OK : allow_dynamic_lds(reinterpret_cast<const void*>(kernel), bytes);
}

size_t hist_lds(const TileGeom& g, int n) {
  const size_t ncol = (size_t)count_columns(g, n);
  return g.chunk <= 65535 ? (ncol + 1) / 2 * 4 : ncol * 4;
}
// keys of one plane: at most 3 n / 2 words (24 KB at n = 4096)
size_t plane_keys_lds(const TileGeom& g) { return (size_t)g.nyt * g.ncls * sizeof(unsigned); }
}  // namespace

int sort_column_blocks(const TileGeom& g, int n) { return column_blocks(g, n); }

size_t carve_scatter(Job& j, bool direct, const SortScratch& need, void* base) {
  size_t off = 0;
  char* b = static_cast<char*>(base);
  auto take = [&](size_t bytes) -> void* {
    void* p = b ? b + off : nullptr;
    off += align_up(bytes);
    return p;
  };
  const TileGeom& g = j.g;
  double* st = static_cast<double*>(take(PK_STATS_LEN * sizeof(double)));
  if (!j.stats) j.stats = st;
  if (!direct) {
    const size_t planes = (size_t)j.a.n + 1;   // and the irregular key
    j.mat = static_cast<unsigned*>(take((size_t)g.nblk * need.columns * sizeof(unsigned)));
    j.pmat = static_cast<unsigned*>(take(need.mixed ? g.nblk * planes * sizeof(unsigned) : 0));
    j.totals = static_cast<int*>(take((size_t)need.columns * sizeof(int)));
    j.ptotals = static_cast<int*>(take(need.mixed ? planes * sizeof(int) : 0));
    j.key_start = static_cast<int*>(take(((size_t)g.nkeys + 1) * sizeof(int)));
    j.plane_start = static_cast<int*>(take(need.planes ? (planes + 1) * sizeof(int) : 0));
    j.wsum = static_cast<double*>(take((size_t)g.nblk * sizeof(double)));
    j.wmax = static_cast<double*>(take((size_t)g.nblk * sizeof(double)));
    j.aux = static_cast<double*>(take(AUX_LEN * sizeof(double)));
    j.koff = static_cast<unsigned*>(take((size_t)g.nkeys * sizeof(unsigned)));
    j.sorted = take((size_t)(j.a.np > 0 ? j.a.np : 1) * sizeof(float4));
    j.staged = take(need.staged ? (size_t)(j.a.np > 0 ? j.a.np : 1) * sizeof(float4) : 0);
    j.tile_mass = static_cast<double*>(take((size_t)g.ntiles * sizeof(double)));
    j.tile_sq = static_cast<double*>(take((size_t)g.ntiles * sizeof(double)));
  }
  return off;
}

size_t scatter_workspace_bytes(const TileGeom& g, bool direct, int n, int64_t np) {
  Job j{};
  j.g = g;
  j.a.np = np;
  j.a.n = n;
  return carve_scatter(j, direct, sort_scratch(g, n), nullptr);
}

int mass_finalize(const Job& j, hipStream_t s) {
  StageTimer t(ST_MASS, s);
  hipLaunchKernelGGL(k_mass_finalize, dim3(1), dim3(MASS_NT), 0, s, j, j.tile_mass ? j.g.ntiles : 0);
  return check_hip(hipGetLastError(), "mass finalize launch");
}

int scatter_run(Job& j, bool direct, const float* mesh_in, float* mesh_out, void* ws, size_t ws_bytes,
                hipStream_t s) {
  const size_t need = carve_scatter(j, direct, sort_scratch(j.g, j.a.n), ws);
  if (ws_bytes < need) return set_error(PK_E_WORKSPACE, "scatter workspace %zu < %zu bytes", ws_bytes, need);
  const ScatterArgs& a = j.a;
  const TileGeom& g = j.g;
  const int64_t ncell = (int64_t)a.n * a.n * a.n;
  if (direct) {
    {
      StageTimer t(ST_FILL, s);
      hipLaunchKernelGGL(k_fill_f64, dim3(1), dim3(PK_STATS_LEN), 0, s, j.stats, PK_STATS_LEN, 0.0);
      hipLaunchKernelGGL(k_copy_or_zero, dim3(grid_for(ncell, 256, 16384)), dim3(256), 0, s, mesh_in, mesh_out,
                         ncell);
      int e = check_hip(hipGetLastError(), "scatter fill launch");
      if (e) return e;
    }
    if (!mesh_out) return set_error(PK_E_INVALID, "direct mode needs a mesh");
    if (a.np > 0) {
      StageTimer t(ST_ATOMIC, s);
      hipLaunchKernelGGL(k_atomic_deposit, dim3(grid_for(a.np, ATM_NT, 65535)), dim3(ATM_NT), 0, s, a,
                         (const void*)nullptr, (const int*)nullptr, mesh_out, j.stats);
      int e = check_hip(hipGetLastError(), "atomic deposit launch");
      if (e) return e;
    }
    j.tile_mass = nullptr;
    j.tile_sq = nullptr;
    return mass_finalize(j, s);
  }
  {
    StageTimer t(ST_SORT_COUNT, s);
    const size_t lds = hist_lds(g, a.n);
    const auto kc = pick_aw<CountK>(a);
    int e = allow_lds(kc, lds);
    if (e) return e;
    hipLaunchKernelGGL(kc, dim3(g.nblk), dim3(CNT_NT), lds, s, j);
    e = check_hip(hipGetLastError(), "bucket count launch");
    if (e) return e;
  }
  {
    StageTimer t(ST_SCAN, s);
    hipLaunchKernelGGL(k_columns, dim3(column_blocks(g, a.n)), dim3(COL_NT), 0, s, j);
    int e = check_hip(hipGetLastError(), "scan launch");
    if (e) return e;
  }
  {
    StageTimer t(ST_SORT_PLACE, s);
    const size_t lds = place_lds(group_count(g, a.n));
    const auto kp = pick_aw<PlaceK>(a);
    int e = allow_lds(kp, lds);
    if (e) return e;
    hipLaunchKernelGGL(kp, dim3(g.nblk), dim3(CNT_NT), lds, s, j);
    e = check_hip(hipGetLastError(), "bucket place launch");
    if (e) return e;
  }
  if (g.sort == SORT_PLANES) {
    StageTimer t(ST_SCAN, s);
    hipLaunchKernelGGL(k_plane_keys, dim3(a.n + 1), dim3(PKEY_NT), plane_keys_lds(g), s, j);
    int e = check_hip(hipGetLastError(), "plane keys launch");
    if (e) return e;
  }
  if (g.sort != SORT_KEYS) {
    StageTimer t(ST_SORT_FINE, s);
    const auto kf = a.stencil == PK_STENCIL_CIC_REF ? k_fine_place<PK_STENCIL_CIC_REF>
                    : a.stencil == PK_STENCIL_CIC   ? k_fine_place<PK_STENCIL_CIC>
                                                    : k_fine_place<PK_STENCIL_TSC>;
    int e = allow_lds(kf, FINE_LDS);
    if (e) return e;
    hipLaunchKernelGGL(kf, dim3(fine_place_blocks(a.np)), dim3(FINE_NT), FINE_LDS, s, j);
    e = check_hip(hipGetLastError(), "fine place launch");
    if (e) return e;
  }
  if (!mesh_out) return PK_OK;   // the caller deposits (fused with the z pass)
  {
    StageTimer t(ST_DEPOSIT, s);
    const size_t lds = (size_t)g.ty * a.n * (g.fixed ? 8 : 4);
    auto aligned = [](const float* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool v4 = a.n % 4 == 0 && aligned(mesh_in) && aligned(mesh_out);
    const auto kd = !g.fixed ? rows_deposit_st<false, false>(a.stencil)
                    : v4     ? rows_deposit_st<true, true>(a.stencil)
                             : rows_deposit_st<true, false>(a.stencil);
    int e = allow_lds(kd, lds);
    if (e) return e;
    hipLaunchKernelGGL(kd, dim3(g.ntiles), dim3(DEP_NT), lds, s, a, g, (const int*)j.key_start, (const void*)j.sorted,
                       (const double*)j.aux, mesh_in, mesh_out, j.tile_mass);
    e = check_hip(hipGetLastError(), "row deposit launch");
    if (e) return e;
  }
  if (a.stencil == PK_STENCIL_CIC_REF && a.np > 0) {
    StageTimer t(ST_ATOMIC, s);
    hipLaunchKernelGGL(k_atomic_deposit, dim3(64), dim3(ATM_NT), 0, s, a, (const void*)j.sorted,
                       (const int*)(j.key_start + g.nkeys - 1), mesh_out, j.stats);
    int e = check_hip(hipGetLastError(), "irregular deposit launch");
    if (e) return e;
  }
  j.tile_sq = nullptr;   // mesh tiles: the z pass sums the squares
  return mass_finalize(j, s);
}

int scatter_sort_jobs(const Job* jobs, const BatchDims& d, hipStream_t s) {
  const int nj = d.njobs;
  {
    StageTimer t(ST_SORT_COUNT, s);
    const size_t lds = (size_t)d.lds_keys * 4;   // any job may count with 32-bit counters
    int e = allow_lds(k_bucket_count_jobs, lds);
    if (e) return e;
    hipLaunchKernelGGL(k_bucket_count_jobs, dim3(d.max_nblk, nj), dim3(CNT_NT), lds, s, jobs);
    e = check_hip(hipGetLastError(), "batch bucket count launch");
    if (e) return e;
  }
  {
    StageTimer t(ST_SCAN, s);
    hipLaunchKernelGGL(k_columns_jobs, dim3(d.max_col, nj), dim3(COL_NT), 0, s, jobs);
    int e = check_hip(hipGetLastError(), "batch scan launch");
    if (e) return e;
  }
  {
    StageTimer t(ST_SORT_PLACE, s);
    // at least what any job's groups take (its rounds shrink as its groups grow)
    const size_t lds = PLACE_LDS;
    int e = allow_lds(k_bucket_place_jobs, lds);
    if (e) return e;
    hipLaunchKernelGGL(k_bucket_place_jobs, dim3(d.max_nblk, nj), dim3(CNT_NT), lds, s, jobs);
    e = check_hip(hipGetLastError(), "batch bucket place launch");
    if (e) return e;
  }
  if (d.planes) {
    StageTimer t(ST_SCAN, s);
    // at most 3 n / 2 keys per plane, whatever the job's tile
    hipLaunchKernelGGL(k_plane_keys_jobs, dim3(d.n + 1, nj), dim3(PKEY_NT), (size_t)6 * d.n, s, jobs);
    int e = check_hip(hipGetLastError(), "batch plane keys launch");
    if (e) return e;
  }
  if (!d.fine) return PK_OK;
  StageTimer t(ST_SORT_FINE, s);
  int e = allow_lds(k_fine_place_jobs, FINE_LDS);
  if (e) return e;
  hipLaunchKernelGGL(k_fine_place_jobs, dim3(d.max_fblk, nj), dim3(FINE_NT), FINE_LDS, s, jobs);
  return check_hip(hipGetLastError(), "batch fine place launch");
}


}  // namespace pk
