// Seeded lognormal mock generator: Gaussian half spectrum (src/gauss_field.py:5-80),
// Poisson population of a density field (src/gauss_field.py:83-110,
// src/populate_field.py:4-29) with the lognormal step of tests/create_lognormal.py:50-51
// fused in, and an optional Zel'dovich redshift-space shift along z.
//
// Population passes:
//   sum   : FP64 per-block sums of rho = exp(bias * field) (or field) -> fixed-order total
//   count : Poisson counts per cell (one byte each, saturated) -> per-block totals ->
//           exclusive scan (block offsets)
//   emit  : the block scans its cells' stored counts and finds its particles' cells in LDS,
//           then one thread per particle: draws, offset, shift, wrap, the (x, y, z) record
// A block owns POP_CELLS consecutive cells in C order (the count visits them in rounds of
// 2 POP_NT, a thread taking a pair, whose two Poisson draws share one Philox block), so
// particles come out in cell order and every offset is a prefix sum.  Emitting per particle
// rather than per cell keeps the random-number and FP64 work free of the divergence of
// sparse cells (most cells hold no particle).
#include "pk_common.h"
#include "pk_internal.h"
#include "pk_mock.h"

namespace pk {

namespace {
constexpr int AMP_NT = 256;
constexpr int SPEC_NT = 256;
constexpr int POP_NT = 256;
constexpr int POP_ROUNDS = 8;
constexpr int POP_CELLS = 2 * POP_NT * POP_ROUNDS;
constexpr int TOP_NT = 1024;
constexpr int TOP_ROWS = 8;   // block totals per thread in flight
constexpr int MISC_LEN = 4;   // [0] rate scale, [1] total (as int64 bits), [2] sum rho, [3] lengths of the lists of dense and of saturated blocks (two ints)

int64_t pop_blocks(int n) {
  const int64_t nc = (int64_t)n * n * n;
  return (nc + POP_CELLS - 1) / POP_CELLS;
}
}  // namespace

size_t gauss_table_len(int n) { return (size_t)3 * (size_t)(n / 2) * (size_t)(n / 2) + 1; }

size_t populate_ws_bytes(int n) {
  const size_t nb = (size_t)pop_blocks(n);
  const size_t npair = ((size_t)n * n * n + 1) / 2;
  return align_up(nb * sizeof(double)) + align_up(nb * sizeof(long long)) + align_up(MISC_LEN * sizeof(double)) +
         align_up(npair * sizeof(uint16_t));
}

// ------------------------------------------------------------------------------------
// amplitude table: sqrt(P(k_F sqrt(m)) (n^2/L)^3), the bisection and linear
// interpolation of src/gauss_field.py:39-47 (end segments extrapolate)
// ------------------------------------------------------------------------------------
__global__ void __launch_bounds__(AMP_NT) k_amp_table(const double* __restrict__ kf, const double* __restrict__ pkf,
                                                      int nk, double kpref, double units, int mmax,
                                                      float* __restrict__ amp) {
  const int m = blockIdx.x * AMP_NT + threadIdx.x;
  if (m > mmax) return;
  const double kmod = sqrt((double)m) * kpref;
  int lo = 0, hi = nk - 1;
  while (hi - lo > 1) {
    const int l = (lo + hi) >> 1;
    if (kf[l] < kmod) lo = l;
    else hi = l;
  }
  const double P = (pkf[hi] - pkf[lo]) / (kf[hi] - kf[lo]) * (kmod - kf[lo]) + pkf[lo];
  amp[m] = (float)sqrt(P * units);
}

int gauss_table(int n, double box, const double* kf, const double* pkf, int nk, float* amp, hipStream_t s) {
  const int mmax = (int)gauss_table_len(n) - 1;
  const double kpref = 2.0 * M_PI / box;
  const double u = (double)n * (double)n / box;
  const double units = u * u * u;
  hipLaunchKernelGGL(k_amp_table, dim3((mmax + AMP_NT) / AMP_NT), dim3(AMP_NT), 0, s, kf, pkf, nk, kpref, units, mmax,
                     amp);
  return check_hip(hipGetLastError(), "amplitude table launch");
}

// the stored half spectrum itself, [kz][kx][ky]
__global__ void __launch_bounds__(SPEC_NT) k_gauss_spectrum(FieldGen g, float2* __restrict__ spec, int64_t total) {
  const int n = g.n;
  const int64_t nn = (int64_t)n * n;
  for (int64_t i = (int64_t)blockIdx.x * SPEC_NT + threadIdx.x; i < total; i += (int64_t)gridDim.x * SPEC_NT) {
    const int kz = (int)(i / nn);
    const int r = (int)(i - (int64_t)kz * nn);
    spec[i] = gauss_mode(g, r / n, r % n, kz);
  }
}

int gauss_spectrum(const FieldGen& g, float2* spec, hipStream_t s) {
  const int64_t total = (int64_t)(g.n / 2 + 1) * g.n * g.n;
  int64_t blocks = (total + SPEC_NT - 1) / SPEC_NT;
  int dev = 0;
  (void)hipGetDevice(&dev);
  const int64_t cap = (int64_t)num_cus(dev) * 32;
  if (blocks > cap) blocks = cap;
  hipLaunchKernelGGL(k_gauss_spectrum, dim3((unsigned)blocks), dim3(SPEC_NT), 0, s, g, spec, total);
  return check_hip(hipGetLastError(), "Gaussian spectrum launch");
}

// ------------------------------------------------------------------------------------
// population
// ------------------------------------------------------------------------------------
struct PopWs {
  double* rsum;      // [nblk]
  long long* boff;   // [nblk] counts, then exclusive offsets
  double* misc;      // [MISC_LEN]
  uint16_t* cnt;     // [ncell / 2] counts of cell pairs (two saturated bytes)
};

static PopWs carve_pop(void* ws, int n) {
  const size_t nb = (size_t)pop_blocks(n);
  char* p = static_cast<char*>(ws);
  PopWs w;
  w.rsum = reinterpret_cast<double*>(p);
  p += align_up(nb * sizeof(double));
  w.boff = reinterpret_cast<long long*>(p);
  p += align_up(nb * sizeof(long long));
  w.misc = reinterpret_cast<double*>(p);
  p += align_up(MISC_LEN * sizeof(double));
  w.cnt = reinterpret_cast<uint16_t*>(p);
  return w;
}

struct PopK {
  const float* field;
  const float* psi;
  int64_t ncell;
  int n;
  int nblk;
  double bias;
  double mean_obj;   // cell volume * density
  double box, H, growth;
  uint32_t k0, k1;
  double* rsum;
  long long* boff;
  double* misc;
  uint16_t* cnt;
  long long* total;  // caller's device int64 (nullable)
  float* pos;
  long long capacity;
};

__device__ __forceinline__ double cell_rho(float v, double bias) {
  return bias != 0.0 ? exp(bias * (double)v) : (double)v;
}

// first cell of round k of this thread: a block owns POP_CELLS consecutive cells in C
// order, visited in POP_ROUNDS rounds of 2 POP_NT cells; thread t takes the pair
// (2t, 2t + 1) of each round
__device__ __forceinline__ int64_t pop_pair(int k) {
  return (int64_t)blockIdx.x * POP_CELLS + (int64_t)k * (2 * POP_NT) + 2 * (int64_t)threadIdx.x;
}

__device__ __forceinline__ long long block_sum_i64(long long v, long long* red) {
  constexpr int NW = POP_NT / 64;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  long long t = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) t += red[i];
  return t;
}

// exclusive prefix of v over the block (int64) and the block total; sh holds NT / 64
// entries and is free again only after the caller's next barrier
template <int NT>
__device__ __forceinline__ long long block_scan_i64(long long v, long long* sh, long long& total) {
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  long long incl = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const long long t = __shfl_up(incl, off, 64);
    if (lane >= off) incl += t;
  }
  if (lane == 63) sh[w] = incl;
  __syncthreads();
  long long before = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    const long long x = sh[i];
    if (i < w) before += x;
    tot += x;
  }
  total = tot;
  return before + incl - v;
}

__global__ void __launch_bounds__(POP_NT) k_pop_sum(PopK a) {
  __shared__ double red[POP_NT / 64 + 1];
  float v[2 * POP_ROUNDS];
#pragma unroll
  for (int k = 0; k < POP_ROUNDS; ++k) {
    const int64_t c = pop_pair(k);
    v[2 * k] = c < a.ncell ? a.field[c] : 0.0f;
    v[2 * k + 1] = c + 1 < a.ncell ? a.field[c + 1] : 0.0f;
  }
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < POP_ROUNDS; ++k) {
    const int64_t c = pop_pair(k);
    if (c < a.ncell) s += cell_rho(v[2 * k], a.bias);
    if (c + 1 < a.ncell) s += cell_rho(v[2 * k + 1], a.bias);
  }
  const double t = block_sum_f64_waves<POP_NT>(s, red);
  if (threadIdx.x == 0) a.rsum[blockIdx.x] = t;
}

// fixed-order total of the block sums -> rate scale = cell volume * density / mean(rho)
__global__ void __launch_bounds__(TOP_NT) k_pop_scale(PopK a) {
  __shared__ double red[TOP_NT / 64 + 1];
  double s = 0.0;
  for (int b0 = threadIdx.x; b0 < a.nblk; b0 += TOP_NT * TOP_ROWS) {
    double v[TOP_ROWS];
#pragma unroll
    for (int r = 0; r < TOP_ROWS; ++r) v[r] = b0 + r * TOP_NT < a.nblk ? a.rsum[b0 + r * TOP_NT] : 0.0;
#pragma unroll
    for (int r = 0; r < TOP_ROWS; ++r) s += v[r];
  }
  const double t = block_sum_f64_waves<TOP_NT>(s, red);
  if (threadIdx.x == 0) {
    a.misc[0] = a.mean_obj / (t / (double)a.ncell);
    a.misc[2] = t;
    a.misc[3] = 0.0;   // no block is listed yet
  }
}

// counts of the pair (c, c + 1); cells beyond the mesh count 0
__device__ __forceinline__ void pair_counts(const PopK& a, int64_t c, double scale, int& n0, int& n1) {
  const double l0 = c < a.ncell ? cell_rho(a.field[c], a.bias) * scale : 0.0;
  const double l1 = c + 1 < a.ncell ? cell_rho(a.field[c + 1], a.bias) * scale : 0.0;
  poisson_pair(l0, l1, (uint64_t)c, a.k0, a.k1, n0, n1);
}

// orders a wave's LDS writes before its lanes' later reads of them
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// How a block of cells is emitted (k_pop_emit): by the most particles that EMIT_PER consecutive cells
// (one thread of the emitting block) hold, at most EMIT_OWN or more, and whether a count is saturated
enum { EMIT_SPARSE = 0, EMIT_DENSE = 1, EMIT_SATURATED = 2 };
constexpr int EMIT_PER = POP_CELLS / POP_NT;   // cells per thread
constexpr int EMIT_OWN = 64;

// The field's sums are spent once the rate scale is known: their place holds [nblk] block routes and
// [nblk] block numbers, the dense ones from the front and the saturated ones from the back; misc[3]
// their two lengths.
__device__ __forceinline__ int* pop_route(const PopK& a) { return reinterpret_cast<int*>(a.rsum); }
__device__ __forceinline__ int* pop_listed(const PopK& a, bool sat, int i) {
  return reinterpret_cast<int*>(a.rsum) + a.nblk + (sat ? a.nblk - 1 - i : i);
}
__device__ __forceinline__ int* pop_list_length(const PopK& a, bool sat) {
  return reinterpret_cast<int*>(a.misc + 3) + (sat ? 1 : 0);
}

// particles of the 16 cells whose stored counts are (lo, hi)
__device__ __forceinline__ int bytes_sum(uint64_t lo, uint64_t hi) {
  uint32_t s = __builtin_amdgcn_sad_u8((uint32_t)lo, 0u, 0u);
  s = __builtin_amdgcn_sad_u8((uint32_t)(lo >> 32), 0u, s);
  s = __builtin_amdgcn_sad_u8((uint32_t)hi, 0u, s);
  return (int)__builtin_amdgcn_sad_u8((uint32_t)(hi >> 32), 0u, s);
}
// whether a byte of v is 255
__device__ __forceinline__ bool any_saturated(uint64_t v) {
  constexpr uint64_t LOW = 0x7f7f7f7f7f7f7f7full, TOP = 0x8080808080808080ull;
  return (((v & LOW) + 0x0101010101010101ull) & v & TOP) != 0;
}

// Most cells hold no particle, and u <= 1 - lambda decides that without exp(-lambda): 1 - lambda
// <= exp(-lambda), and the margin of 2^-50 covers the rounding of both.  The other cells go to a
// list in LDS, whose draws (the exponential and the inversion loop, or the rejection) then
// run with full waves.  Counts equal those of a draw per cell.  512^3 cells, 2e7 particles, bias 1 of
// a unit Gaussian field: a draw per cell 692 us, one list per block 582, a list per wave (no round
// waits for another wave) 547; 64^3 cells with half a particle each: 11.8, 15.4 and 13.3 us.
constexpr int CNT_LIST = 256;   // entries per wave; a round adds at most 128
__global__ void __launch_bounds__(POP_NT) k_pop_count(PopK a) {
  constexpr int NW = POP_NT / 64;
  __shared__ long long red[NW];
  __shared__ double list_l[NW][CNT_LIST], list_u[NW][CNT_LIST];
  __shared__ uint16_t list_c[NW][CNT_LIST];
  __shared__ __align__(16) uint8_t cnt[POP_CELLS];   // saturated: 255 means "recount"
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const double scale = a.misc[0];
  const int64_t c0 = (int64_t)blockIdx.x * POP_CELLS;
  static_assert(EMIT_PER == 16, "one 16-byte access of counts per thread");
  reinterpret_cast<uint4*>(cnt)[tid] = make_uint4(0u, 0u, 0u, 0u);
  float f0, f1;
  auto load = [&](int k) {
    const int64_t c = pop_pair(k);
    f0 = c < a.ncell ? a.field[c] : 0.0f;
    f1 = c + 1 < a.ncell ? a.field[c + 1] : 0.0f;
  };
  load(0);
  __syncthreads();
  long long s = 0;   // counts: at most 2^42 in a block
  int have = 0;      // the wave's listed cells
#pragma unroll 1
  for (int k = 0; k < POP_ROUNDS; ++k) {
    const int64_t c = pop_pair(k);
    const double lam[2] = {c < a.ncell ? cell_rho(f0, a.bias) * scale : 0.0,
                           c + 1 < a.ncell ? cell_rho(f1, a.bias) * scale : 0.0};
    if (k + 1 < POP_ROUNDS) load(k + 1);
    const Philox4 w = rng_block((uint64_t)c >> 1, 0, TAG_POISSON, a.k0, a.k1);
    const double u[2] = {uniform_f64(w.x, w.y), uniform_f64(w.z, w.w)};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const bool draw = lam[e] > 0.0 && !(u[e] + 0x1p-50 <= 1.0 - lam[e]);
      const uint64_t m = __ballot(draw);
      if (draw) {
        const int at = have + __popcll(m & ((1ull << lane) - 1));
        list_l[wv][at] = lam[e];
        list_u[wv][at] = u[e];
        list_c[wv][at] = (uint16_t)(c + e - c0);
      }
      have += __popcll(m);
    }
    if (have > CNT_LIST - 128 || k + 1 == POP_ROUNDS) {   // wave-uniform
      wave_lds_fence();
      for (int i = lane; i < have; i += 64) {
        const int at = list_c[wv][i];
        const int n = poisson_draw(list_l[wv][i], list_u[wv][i], (uint64_t)(c0 + at), a.k0, a.k1);
        cnt[at] = (uint8_t)min(n, 255);
        s += n;
      }
      wave_lds_fence();
      have = 0;
    }
  }
  __syncthreads();
  const ulonglong2 mine = reinterpret_cast<const ulonglong2*>(cnt)[tid];
  if (bytes_sum(mine.x, mine.y) > EMIT_OWN) s += 1ll << 43;              // at most 2^51 in a block
  if (any_saturated(mine.x) || any_saturated(mine.y)) s += 1ll << 52;
  // whole pairs, the mesh's last one too (its second cell counts 0)
  const int64_t pairs = min((int64_t)POP_CELLS, a.ncell - c0 + 1) / 2;
  if (pairs == POP_CELLS / 2) {
    reinterpret_cast<ulonglong2*>(a.cnt + c0 / 2)[tid] = mine;
  } else {
    for (int i = tid; i < pairs; i += POP_NT) a.cnt[c0 / 2 + i] = reinterpret_cast<const uint16_t*>(cnt)[i];
  }
  const long long t = block_sum_i64(s, red);
  if (tid == 0) {
    a.boff[blockIdx.x] = t & ((1ll << 43) - 1);
    const int route = t >> 52 ? EMIT_SATURATED : t >> 43 ? EMIT_DENSE : EMIT_SPARSE;
    pop_route(a)[blockIdx.x] = route;
    const bool sat = route == EMIT_SATURATED;
    if (route != EMIT_SPARSE) *pop_listed(a, sat, atomicAdd(pop_list_length(a, sat), 1)) = blockIdx.x;
  }
}

// block totals -> exclusive block offsets (in place); grand total to misc[1] and *total.  Rows
// of TOP_NT consecutive totals, TOP_ROWS of them in flight: their wave scans, then one scan of
// the (row, wave) totals.  32768 totals (512^3): 60 us walking contiguous runs per thread ->
// 30 us.
__global__ void __launch_bounds__(TOP_NT) k_pop_scan(PopK a) {
  constexpr int NW = TOP_NT / 64, NE = NW * TOP_ROWS;
  static_assert(NE == 128, "two entries per lane of the scanning wave");
  __shared__ long long wt[NE];   // totals of (row, wave), then their exclusive prefix
  __shared__ long long tot;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  long long carry = 0;
  for (int b0 = 0; b0 < a.nblk; b0 += TOP_NT * TOP_ROWS) {   // block-uniform
    long long v[TOP_ROWS], incl[TOP_ROWS];
#pragma unroll
    for (int r = 0; r < TOP_ROWS; ++r) {
      const int i = b0 + r * TOP_NT + tid;
      v[r] = i < a.nblk ? a.boff[i] : 0;
    }
#pragma unroll
    for (int r = 0; r < TOP_ROWS; ++r) {
      incl[r] = v[r];
      if (b0 + r * TOP_NT < a.nblk) {   // block-uniform
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
          const long long t = __shfl_up(incl[r], off, 64);
          if (lane >= off) incl[r] += t;
        }
      }
      if (lane == 63) wt[r * NW + w] = incl[r];
    }
    __syncthreads();
    if (w == 0) {
      const long long e0 = wt[2 * lane], e1 = wt[2 * lane + 1];
      long long run = e0 + e1;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const long long t = __shfl_up(run, off, 64);
        if (lane >= off) run += t;
      }
      wt[2 * lane] = run - e0 - e1;
      wt[2 * lane + 1] = run - e1;
      if (lane == 63) tot = run;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < TOP_ROWS; ++r) {
      const int i = b0 + r * TOP_NT + tid;
      if (i < a.nblk) a.boff[i] = carry + wt[r * NW + w] + incl[r] - v[r];
    }
    carry += tot;
    __syncthreads();   // wt and tot are rewritten by the next rows
  }
  if (tid == 0) {
    reinterpret_cast<long long*>(a.misc)[1] = carry;
    if (a.total) *a.total = carry;
  }
}

// periodic wrap into [0, L) in FP64, rounded to float32 (a value that rounds up to L
// becomes 0); values already inside skip the division
__device__ __forceinline__ float wrap_box(double r, double box) {
  double u = r;
  if (!(u >= 0.0 && u < box)) {
    u = r - box * floor(r / box);
    if (u < 0.0) u += box;
    if (u >= box) u -= box;
  }
  const float f = (float)u;
  return f >= (float)box ? 0.0f : f;
}

// One particle: output slot p, cell c
__device__ __forceinline__ void emit_particle(const PopK& a, long long p, uint32_t c) {
  const uint32_t n = (uint32_t)a.n;
  const uint32_t iz = c % n, cy = c / n;
  const uint32_t iy = cy % n, ix = cy / n;
  const Philox4 w = rng_block((uint64_t)p, 0, TAG_DISP, a.k0, a.k1);
  const double shift = (a.psi != nullptr && a.growth != 0.0) ? a.growth * (double)a.psi[c] : 0.0;
  typedef float f3 __attribute__((ext_vector_type(3), aligned(4)));
  const f3 f = {wrap_box(((double)ix + 0.5 + tri_offset(w.x)) * a.H, a.box),
                wrap_box(((double)iy + 0.5 + tri_offset(w.y)) * a.H, a.box),
                wrap_box(((double)iz + 0.5 + tri_offset(w.z)) * a.H + shift, a.box)};
  *reinterpret_cast<f3*>(a.pos + 3 * p) = f;
}

// stored counts of the thread's EMIT_PER consecutive cells of block blk
__device__ __forceinline__ ulonglong2 load_counts(const PopK& a, int blk) {
  const int64_t mine = (int64_t)blk * POP_CELLS + (int64_t)threadIdx.x * EMIT_PER;
  if (mine + EMIT_PER <= a.ncell) return reinterpret_cast<const ulonglong2*>(a.cnt)[mine / EMIT_PER];
  ulonglong2 v = {0, 0};
  for (int i = 0; i < EMIT_PER; ++i)
    if (mine + i < a.ncell) {
      const uint64_t pair = a.cnt[(mine + i) >> 1];   // the cell's byte of its pair
      (i < 8 ? v.x : v.y) |= ((i & 1 ? pair >> 8 : pair) & 255u) << (8 * (i & 7));
    }
  return v;
}

// Emission, by what the block's cells hold.  Bound by the draws and FP64 arithmetic of the particles
// where the finding of their cells keeps up: a thread that lists its cells' particles one by one holds
// up its block once they are many (64^3 cells of 40 particles: 1112 us, against 225 to mark the slots
// from the waves and 84 to emit), so blocks with more than EMIT_OWN in the cells of one thread go by
// bisection (119 us there).  Whole calls, us, marking / listing alone / both ways as here:
// 64^3 cells of 40: 395 / 1226 / 208; of 300: 2346 / 36000 / 1233; 128^3, 1 per cell, bias 2: 147 /
// 216 / 130; 256^3 of 2: 565 / 473 / 447 (EMIT_OWN 32: 514); 256^3 of 0.15: 175 / 140 / 124; 64^3 of a half:
// 54 / 64 / 58.  At 512^3 with 2e7 particles marking and emitting take 407 + 158 us, this 251 + 4.
// Sparse blocks: a thread scans its 16 cells' counts (one 16-byte load), the block scans the threads'
// sums, every thread lists its particles' cells in LDS (EMIT_WIN slots at a time), and the lanes then
// take consecutive particles.
constexpr int EMIT_WIN = 4096;
__device__ __forceinline__ void emit_sparse(const PopK& a, int blk, uint16_t* list) {
  __shared__ long long sh[POP_NT / 64];
  const int64_t c0 = (int64_t)blk * POP_CELLS;
  const long long base = a.boff[blk];
  const ulonglong2 v = load_counts(a, blk);
  const int own = bytes_sum(v.x, v.y);
  long long sum;
  const int first = (int)block_scan_i64<POP_NT>(own, sh, sum);   // this thread's first slot
  const int total = (int)sum;
  for (int w0 = 0; w0 < total; w0 += EMIT_WIN) {   // block-uniform
    const int w1 = min(w0 + EMIT_WIN, total);
    if (own > 0 && first < w1 && first + own > w0) {
      int s = first;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        uint64_t left = h ? v.y : v.x;
#pragma unroll 1
        while (left) {
          const int k = (__ffsll((unsigned long long)left) - 1) >> 3;
          const int end = s + (int)((left >> (8 * k)) & 255u);
          left &= ~(255ull << (8 * k));
          for (int q = max(s, w0); q < min(end, w1); ++q) list[q - w0] = (uint16_t)(threadIdx.x * EMIT_PER + 8 * h + k);
          s = end;
        }
      }
    }
    __syncthreads();
#pragma unroll 1
    for (int s = w0 + threadIdx.x; s < w1; s += POP_NT) {
      const long long p = base + s;
      if (p >= a.capacity) break;
      emit_particle(a, p, (uint32_t)(c0 + list[s - w0]));
    }
    __syncthreads();   // the list is read before the next window overwrites it
  }
}

// Windows first, first + step, ... of EMIT_WIN particles of block blk: pre holds every cell's first
// slot, clipped to the window, and a particle finds its cell by bisection.  SAT: the block holds
// saturated counts, which are drawn again into LDS (big); in a kernel of its own, since the draws take
// 132 registers against 60.
constexpr int EMIT_SPLIT = 16;        // emitting blocks that share the windows of one block
constexpr int EMIT_DENSE_MAX = 512;   // blocks emitted at a time
template <bool SAT>
__device__ __forceinline__ void emit_dense(const PopK& a, int blk, int first, int step, uint16_t* pre, int* big) {
  __shared__ long long sh[POP_NT / 64];
  const int tid = threadIdx.x;
  const int64_t c0 = (int64_t)blk * POP_CELLS;
  const long long base = a.boff[blk];
  const ulonglong2 v = load_counts(a, blk);
  auto stored = [&](int i) { return (int)(((i < 8 ? v.x : v.y) >> (8 * (i & 7))) & 255u); };
  long long own = 0;
  if constexpr (SAT) {
#pragma unroll 1
    for (int i = 0; i < EMIT_PER; ++i) {
      int n = stored(i);
      if (n == 255) {
        const int64_t c = c0 + tid * EMIT_PER + i;
        int n0, n1;
        pair_counts(a, c & ~(int64_t)1, a.misc[0], n0, n1);
        n = c & 1 ? n1 : n0;
      }
      big[i * POP_NT + tid] = n;
      own += n;
    }
  } else {
    own = bytes_sum(v.x, v.y);
  }
  long long total;
  const long long mine = block_scan_i64<POP_NT>(own, sh, total);
  for (long long w0 = (long long)first * EMIT_WIN; w0 < total; w0 += (long long)step * EMIT_WIN) {   // block-uniform
    long long p = mine - w0;
    uint32_t* out = reinterpret_cast<uint32_t*>(pre) + tid * (EMIT_PER / 2);
#pragma unroll 1
    for (int i = 0; i < EMIT_PER; i += 2) {
      const uint32_t e = (uint32_t)min(max(p, 0ll), (long long)EMIT_WIN);
      p += SAT ? big[i * POP_NT + tid] : stored(i);
      const uint32_t o = (uint32_t)min(max(p, 0ll), (long long)EMIT_WIN);
      p += SAT ? big[(i + 1) * POP_NT + tid] : stored(i + 1);
      out[i / 2] = e | o << 16;
    }
    __syncthreads();
    const int last = (int)min((long long)EMIT_WIN, total - w0);
#pragma unroll 1
    for (int s = tid; s < last; s += POP_NT) {
      const long long q = base + w0 + s;
      if (q >= a.capacity) break;
      int cell = 0;   // the last cell whose first slot is not above s
#pragma unroll
      for (int half = POP_CELLS / 2; half > 0; half >>= 1) cell += pre[cell + half] <= s ? half : 0;
      emit_particle(a, q, (uint32_t)(c0 + cell));
    }
    __syncthreads();   // the window's slots are read before the next one's are written
  }
}
// the blocks of one list, dealt over nx EMIT_SPLIT emitting blocks: consecutive ones take
// different dense blocks, so that the few windows of a not very dense one lie on all XCDs
template <bool SAT>
__device__ __forceinline__ void emit_dense_blocks(const PopK& a, int bx, int nx, uint16_t* pre, int* big) {
  const int count = *pop_list_length(a, SAT);
  for (int d = bx % nx; d < count; d += nx) {   // block-uniform
    const int blk = *pop_listed(a, SAT, d), first = bx / nx;
    const long long end = blk + 1 < a.nblk ? a.boff[blk + 1] : reinterpret_cast<const long long*>(a.misc)[1];
    if ((long long)first * EMIT_WIN < end - a.boff[blk]) emit_dense<SAT>(a, blk, first, EMIT_SPLIT, pre, big);
  }
}
// one sparse block each, then the nx EMIT_SPLIT blocks that take the dense ones (those first, the idle ones
// of them held the sparse blocks up: 128^3 of 1 42 against 33 us, 256^3 of 2 324 against 309)
__global__ void __launch_bounds__(POP_NT) k_pop_emit(PopK a, int nx) {
  __shared__ __align__(16) uint16_t lds[EMIT_WIN > POP_CELLS ? EMIT_WIN : POP_CELLS];
  const int bx = blockIdx.x;
  if (bx >= a.nblk) emit_dense_blocks<false>(a, bx - a.nblk, nx, lds, nullptr);
  else if (pop_route(a)[bx] == EMIT_SPARSE) emit_sparse(a, bx, lds);
}
__global__ void __launch_bounds__(POP_NT) k_pop_emit_saturated(PopK a, int nx) {
  __shared__ __align__(16) uint16_t pre[POP_CELLS];
  __shared__ int big[POP_CELLS];
  emit_dense_blocks<true>(a, blockIdx.x, nx, pre, big);
}

namespace {
PopK make_pop(const float* field, const float* psi, int n, double box, double density, double bias, double growth,
              uint64_t seed, void* ws, long long* total, float* pos, long long capacity) {
  PopK a{};
  a.field = field;
  a.psi = psi;
  a.n = n;
  a.ncell = (int64_t)n * n * n;
  a.nblk = (int)pop_blocks(n);
  a.bias = bias;
  a.box = box;
  a.H = box / (double)n;
  a.mean_obj = a.H * a.H * a.H * density;
  a.growth = growth;
  a.k0 = (uint32_t)seed;
  a.k1 = (uint32_t)(seed >> 32);
  const PopWs w = carve_pop(ws, n);
  a.rsum = w.rsum;
  a.boff = w.boff;
  a.misc = w.misc;
  a.cnt = w.cnt;
  a.total = total;
  a.pos = pos;
  a.capacity = capacity;
  return a;
}
}  // namespace

int populate_count(const float* field, int n, double box, double density, double bias, uint64_t seed, void* ws,
                   int64_t* total, hipStream_t s) {
  const PopK a = make_pop(field, nullptr, n, box, density, bias, 0.0, seed, ws, reinterpret_cast<long long*>(total),
                          nullptr, 0);
  hipLaunchKernelGGL(k_pop_sum, dim3(a.nblk), dim3(POP_NT), 0, s, a);
  hipLaunchKernelGGL(k_pop_scale, dim3(1), dim3(TOP_NT), 0, s, a);
  hipLaunchKernelGGL(k_pop_count, dim3(a.nblk), dim3(POP_NT), 0, s, a);
  hipLaunchKernelGGL(k_pop_scan, dim3(1), dim3(TOP_NT), 0, s, a);
  return check_hip(hipGetLastError(), "population count launch");
}

int populate_place(const float* field, const float* psi, double growth, int n, double box, double bias, uint64_t seed,
                   void* ws, float* pos, int64_t capacity, hipStream_t s) {
  if (capacity == 0) return PK_OK;
  const PopK a = make_pop(field, psi, n, box, 0.0, bias, growth, seed, ws, nullptr, pos, (long long)capacity);
  const int nx = a.nblk < EMIT_DENSE_MAX ? a.nblk : EMIT_DENSE_MAX;
  hipLaunchKernelGGL(k_pop_emit, dim3(nx * EMIT_SPLIT + a.nblk), dim3(POP_NT), 0, s, a, nx);
  hipLaunchKernelGGL(k_pop_emit_saturated, dim3(nx * EMIT_SPLIT), dim3(POP_NT), 0, s, a, nx);
  return check_hip(hipGetLastError(), "population place launch");
}

}  // namespace pk
