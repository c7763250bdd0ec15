// Block output-stationary convolution (fp16, wide rows): every output row is summed in registers over all kernel
// offsets and stored once.  Rows are visited in an order that puts equal neighbour patterns side by side inside
// windows of the storage order (pce_osb_order), so that a 16-row block can leave out the offsets none of its rows has.
#include <math.h>
#include <string.h>

#include "pce_tile.h"

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// ---- row order -----------------------------------------------------------------------------------------------------
// perm[n] | bmask[ceil(n / 16)]: inside every window of OSB_WINDOW rows the rows sorted by their neighbour pattern,
// and the union of the patterns of every 16 consecutive rows of that order.
// The window keeps rows that are near in space near in the order (the gathers of a tile hit its XCD's L2).
#define OSB_WINDOW 8192
#define OSB_MAX_KV 27
#define OSB_ORDER_THREADS 1024

// position of an offset's bit in the sort key of a 3x3x3 kernel, most significant first: corners, edges, faces,
// centre.  Rare bits first keep the blocks' unions small: 12.9 offsets per 256 rows on the 680 k-row level of the
// indoor scenes against 17.8 in natural order (6.2 offsets per row), 14.4 against 14.8 on a 89 k-row LiDAR level.
__device__ constexpr int osb_key_bit27(int kp) {
  int pos = 0;
  const int dist = (kp / 9 != 1) + (kp / 3 % 3 != 1) + (kp % 3 != 1);
  for (int i = 0; i < 27; ++i) {
    const int d = (i / 9 != 1) + (i / 3 % 3 != 1) + (i % 3 != 1);
    if (d > dist || (d == dist && i < kp)) ++pos;
  }
  return 26 - pos;
}

// The orders of several tables are one launch: they are wanted together (a network's levels), and each alone leaves most of the
// machine idle, a workgroup a window: with the plans four levels of a 100 k-voxel scan 38 us, 140 one after the other, six of eight
// indoor scenes 70 and 278.
struct OsbOrderJob {
  const int *nbr;
  const unsigned *known;
  unsigned centre;
  int kv, n, window0;   // its first workgroup
  int *perm;
  unsigned *bmask;
  int *plans;
};
struct OsbOrderJobs {
  OsbOrderJob job[PCE_OSB_ORDER_MAX];
  int count;
};

// One workgroup per window: the rows' patterns (known, or 27 table reads per row), then a radix sort of (key, row) in LDS,
// three passes of 9 bits.  The key is the rank of the pattern in the reflected Gray code, in which
// consecutive patterns differ in one bit.  The sort is stable by construction: a wavefront ranks its entries of a digit by
// ballots (the lanes of one LDS atomic have no promised order), so the order of a cloud is the same in every run, and the
// entries behind the last row of the cloud, which share their key with a pattern of offset 0 alone, stay behind every row.
// Bound by the ballots and the LDS counters, not by memory: with the plan 36 us for 72 k rows of a random cloud as for
// 100 k of a scan (ranked by LDS atomics, whose lanes met at few counters: 36 and 43).
// SHORT: a cloud of one window that is not full, where a thread has per = rows / 1024 entries instead of eight (with the plan
// 31 -> 15 us on 700 rows, 21 on 3 k, 29 on 6 k; in a full window the conditions would cost 1 us of 33).
template <bool SHORT>
__global__ void __launch_bounds__(OSB_ORDER_THREADS) osb_order_kernel(OsbOrderJobs jobs) {
  constexpr int PER = OSB_WINDOW / OSB_ORDER_THREADS, WAVES = OSB_ORDER_THREADS / 64, BITS = 9, BINS = 1 << BITS;
  __shared__ unsigned keys[OSB_WINDOW];
  __shared__ unsigned masks[OSB_WINDOW];
  __shared__ unsigned short rows[OSB_WINDOW];
  __shared__ unsigned hist[BINS * WAVES];
  __shared__ unsigned wave_sum[WAVES];
  int which = 0;
  while (which + 1 < jobs.count && (int)blockIdx.x >= jobs.job[which + 1].window0) ++which;
  const int *__restrict__ nbr = jobs.job[which].nbr;
  const unsigned *__restrict__ known = jobs.job[which].known;
  int *__restrict__ perm = jobs.job[which].perm;
  unsigned *__restrict__ bmask = jobs.job[which].bmask;
  const unsigned centre = jobs.job[which].centre;
  const int kv = jobs.job[which].kv, n = jobs.job[which].n;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int r0 = ((int)blockIdx.x - jobs.job[which].window0) * OSB_WINDOW, cnt = n - r0 < OSB_WINDOW ? n - r0 : OSB_WINDOW;
  const int per = SHORT ? (cnt + OSB_ORDER_THREADS - 1) / OSB_ORDER_THREADS : PER;
  unsigned m[PER];
  if (known) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int li = i * OSB_ORDER_THREADS + t;
      m[i] = known[r0 + (li < cnt ? li : 0)];
    }
  } else {
#pragma unroll
    for (int i = 0; i < PER; ++i) m[i] = 0;
    for (int kp = 0; kp < kv; ++kp) {
      int v[PER];
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int li = i * OSB_ORDER_THREADS + t;
        v[i] = nbr[(long long)kp * n + r0 + (li < cnt ? li : 0)];
      }
#pragma unroll
      for (int i = 0; i < PER; ++i) m[i] |= (unsigned)(v[i] >= 0) << kp;
    }
  }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (SHORT && i >= per) break;
    const int li = i * OSB_ORDER_THREADS + t;
    const bool ok = li < cnt;
    const unsigned pat = m[i] | centre;
    unsigned k = 0;
    if (kv == 27) {
#pragma unroll
      for (int kp = 0; kp < 27; ++kp) k |= ((pat >> kp) & 1u) << osb_key_bit27(kp);
    } else {
      k = pat;
    }
    k ^= k >> 1;
    k ^= k >> 2;
    k ^= k >> 4;
    k ^= k >> 8;
    k ^= k >> 16;
    masks[li] = ok ? pat : 0u;
    keys[li] = ok ? k : (1u << 27) - 1;
    rows[li] = (unsigned short)li;
  }
  // where a digit's counter of a wavefront lies: the counters one wavefront updates fall into different banks
  auto counter = [](int d, int w) { return d * WAVES + ((w + (d >> 2)) & (WAVES - 1)); };
  for (int shift = 0; shift < 3 * BITS; shift += BITS) {
    for (int i = t; i < BINS * WAVES; i += OSB_ORDER_THREADS) hist[i] = 0;
    __syncthreads();
    unsigned key[PER], pos[PER];
    unsigned short rw[PER];
    // rank among the wavefront's entries of one digit: the lanes below with the same digit, behind those of the entries
    // before (a counter per (digit, wavefront), updated by the first lane of a digit)
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int at = (wave * per + (!SHORT || i < per ? i : 0)) * 64 + lane;
      key[i] = keys[at];
      rw[i] = rows[at];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (SHORT && i >= per) break;
      const unsigned d = (key[i] >> shift) & (BINS - 1);
      unsigned long long peers = ~0ull;
#pragma unroll
      for (int b = 0; b < BITS; ++b) {
        const unsigned mine = (unsigned)((int)(d << (31 - b)) >> 31);   // the bit of this lane, in all bits
        peers &= ~(__ballot(mine != 0) ^ (mine | (unsigned long long)mine << 32));
      }
      const int before = __popcll(peers & ((1ull << lane) - 1));
      unsigned *count = &hist[counter(d, wave)];
      pos[i] = *count + before;
      __builtin_amdgcn_wave_barrier();
      if (before == 0) *count = pos[i] + __popcll(peers);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    __syncthreads();
    // exclusive scan over (digit, wavefront)
    constexpr int HP = BINS * WAVES / OSB_ORDER_THREADS;
    unsigned v[HP], sum = 0;
#pragma unroll
    for (int j = 0; j < HP; ++j) {
      v[j] = sum;
      sum += hist[counter((t * HP + j) / WAVES, (t * HP + j) % WAVES)];
    }
    unsigned inc = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const unsigned up = __shfl_up(inc, o, 64);
      if (lane >= o) inc += up;
    }
    if (lane == 63) wave_sum[wave] = inc;
    __syncthreads();
    unsigned base = inc - sum;
    for (int w = 0; w < wave; ++w) base += wave_sum[w];
#pragma unroll
    for (int j = 0; j < HP; ++j) hist[counter((t * HP + j) / WAVES, (t * HP + j) % WAVES)] = base + v[j];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (SHORT && i >= per) break;
      const unsigned d = (key[i] >> shift) & (BINS - 1);
      const unsigned p = hist[counter(d, wave)] + pos[i];
      keys[p] = key[i];
      rows[p] = rw[i];
    }
    __syncthreads();
  }
  for (int i = 0; i < per; ++i) {
    const int p = i * OSB_ORDER_THREADS + t;
    const int li = rows[p];
    unsigned m = p < cnt ? masks[li] : 0u;
    if (p < cnt) perm[r0 + p] = r0 + li;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) m |= __shfl_xor(m, o, 64);
    if ((lane & 15) == 0 && p < cnt) bmask[(r0 + p) >> 4] = m;
  }
}

// ---- plan ---------------------------------------------------------------------------------------------------------
// The tiles of a layer differ in cost (the offsets their rows have together) and a launch holds 512 workgroups, so a
// layer of a few hundred tiles ends with most of the machine waiting for the last ones.  A plan deals the (tile, column
// slab) items to the eight XCDs: contiguous ranges of equal cost; inside a range the last OSB_TAIL items heaviest first
// (the others in storage order, neighbours in space beside each other in time); and where the items do not fill the last
// round of OSB_SLOTS workgroups, the ones left over are cut into parts of their offsets whose sums a second
// kernel adds up.  72 k rows of a random cloud, 256 -> 256 channels (564 items): 220 us with the items in storage order,
// 194 us with the plan.
#define OSB_ROWS 128        // rows of a tile: eight blocks of 16
#define OSB_SLOTS 64        // workgroups an XCD holds: 32 compute units, two each
#define OSB_TAIL 192
#define OSB_MAX_CUT 48      // items of an XCD that may be cut
#define OSB_MAX_PARTS 8
#define OSB_MAX_SLABS 4

// ints of a plan: cut items {item, parts} [8][OSB_MAX_CUT] | items {item, part | parts << 8 | slot << 16} [8][cap];
// item -1: none
__host__ __device__ static inline long long osb_plan_cap(long long tiles, int slabs) { return (tiles / 8 + tiles / 16 + 3) * slabs + OSB_SLOTS; }
__host__ __device__ static inline long long osb_plan_elems(long long tiles, int slabs) {
  return 2 * (8 * OSB_MAX_CUT) + 2 * 8 * osb_plan_cap(tiles, slabs);
}
// the plans for one, two, ... column slabs lie behind one another
__host__ __device__ static inline long long osb_plan_offset(long long tiles, int slabs) {
  long long at = 0;
  for (int s = 1; s < slabs; ++s) at += osb_plan_elems(tiles, s);
  return at;
}

// One workgroup per XCD and column slab count of an order.
__global__ void __launch_bounds__(1024) osb_plan_kernel(OsbOrderJobs jobs) {
  const unsigned *__restrict__ bmask = jobs.job[blockIdx.z].bmask;
  int *__restrict__ plans = jobs.job[blockIdx.z].plans;
  const int n = jobs.job[blockIdx.z].n, tiles = (n + OSB_ROWS - 1) / OSB_ROWS;
  __shared__ unsigned sums[16];
  __shared__ int bound[2];
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, x = blockIdx.x;
  const int slabs = blockIdx.y + 1, cap = (int)osb_plan_cap(tiles, slabs);
  int *plan = plans + osb_plan_offset(tiles, slabs);
  const int blocks = (n + 15) >> 4;
  auto cost = [&](int tile) {
    unsigned m = 0;
    for (int b = tile * 8; b < tile * 8 + 8; ++b) m |= b < blocks ? bmask[b] : 0u;
    return __popc(m) + 1;   // one more for what a tile costs whatever its offsets
  };
  // range of this XCD: tiles whose cost prefix lies in [x, x + 1) eighths of the total, kept within a sixteenth of the
  // equal split by count so that the lists have a known length
  const int per = (tiles + 1023) / 1024, t0 = t * per, t1 = t0 + per < tiles ? t0 + per : tiles;
  unsigned sum = 0;
  for (int i = t0; i < t1; ++i) sum += cost(i);
  unsigned inc = sum;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned up = __shfl_up(inc, o, 64);
    if (lane >= o) inc += up;
  }
  if (lane == 63) sums[wave] = inc;
  __syncthreads();
  unsigned base = inc - sum, total = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) base += sums[w];
    total += sums[w];
  }
  for (int k = 0; k < 2; ++k) {
    const unsigned want = (unsigned)((unsigned long long)total * (x + k) / 8);
    if (t0 < t1 && base <= want && want < base + sum) {
      unsigned at = base;
      int i = t0;
      while (i < t1 && at < want) at += cost(i++);
      bound[k] = i;
    }
    if (x + k == 8 && t == 0) bound[k] = tiles;
  }
  __syncthreads();
  int lim[2];
  for (int k = 0; k < 2; ++k) {
    const int even = (int)((long long)tiles * (x + k) / 8), slack = tiles / 32;
    int b = x + k == 0 ? 0 : (x + k == 8 ? tiles : bound[k]);
    b = b < even - slack ? even - slack : (b > even + slack ? even + slack : b);
    lim[k] = x + k == 0 ? 0 : (x + k == 8 ? tiles : b);
  }
  const int lo = lim[0], m = (lim[1] - lim[0]) * slabs;
  // what does not fill the last round of workgroups is cut
  const int round = m / OSB_SLOTS * OSB_SLOTS, left = m - round;
  const int cut = left <= OSB_MAX_CUT && left > 0 ? left : 0;
  int parts = cut ? OSB_SLOTS / cut : 1;
  parts = parts > OSB_MAX_PARTS ? OSB_MAX_PARTS : parts;
  const int n_cut = parts > 1 ? cut : 0;
  int *cuts = plan + x * (2 * OSB_MAX_CUT);
  int *items = plan + 8 * (2 * OSB_MAX_CUT) + (long long)x * 2 * cap;
  const int n_items = m - n_cut + n_cut * parts;
  for (int i = n_items + t; i < cap; i += 1024) {   // workgroups without an item
    items[2 * i] = -1;
    items[2 * i + 1] = 0;
  }
  for (int i = n_cut + t; i < OSB_MAX_CUT; i += 1024) {
    cuts[2 * i] = -1;
    cuts[2 * i + 1] = 0;
  }
  auto put = [&](int pos, int item) {
    if (pos < m - n_cut) {
      items[2 * pos] = item;
      items[2 * pos + 1] = 1 << 8;
    } else {
      const int c = pos - (m - n_cut);
      cuts[2 * c] = item;
      cuts[2 * c + 1] = parts;
      for (int p = 0; p < parts; ++p) {
        const int at = m - n_cut + c * parts + p;
        items[2 * at] = item;
        items[2 * at + 1] = p | (parts << 8) | ((x * OSB_SLOTS + c * parts + p) << 16);
      }
    }
  };
  const int tail = m < OSB_TAIL ? m / slabs : OSB_TAIL / slabs, head = lim[1] - lim[0] - tail;   // in tiles
  for (int i = t; i < head; i += 1024)
    for (int sl = 0; sl < slabs; ++sl) put(i * slabs + sl, (lo + i) * slabs + sl);
  // the tail by cost, heaviest first: every tile's place is the number of tiles in front of it
  __shared__ int costs[OSB_TAIL];
  if (t < tail) costs[t] = cost(lo + head + t);
  __syncthreads();
  if (t < tail) {
    const int c = costs[t];
    int pos = 0;
    for (int i = 0; i < tail; ++i) pos += costs[i] > c || (costs[i] == c && i < t);
    for (int sl = 0; sl < slabs; ++sl) put((head + pos) * slabs + sl, (lo + head + t) * slabs + sl);
  }
}

static long long osb_mask_offset(long long n) { return (n + 63) / 64 * 64; }
static long long osb_plans_offset(long long n) { return (osb_mask_offset(n) + (n + 15) / 16 + 63) / 64 * 64; }

extern "C" int64_t pce_osb_order_elems(int64_t n) {
  return n <= 0 ? 0 : osb_plans_offset(n) + osb_plan_offset(pce_div_up(n, OSB_ROWS), OSB_MAX_SLABS + 1);
}

extern "C" int pce_osb_order_batch(const pce_osb_order_problem_t *problems, int32_t count, pce_stream_t stream) {
  if (!problems || count < 1 || count > PCE_OSB_ORDER_MAX) PCE_FAIL(PCE_EINVAL, "pce_osb_order: 1..%d tables per call", PCE_OSB_ORDER_MAX);
  OsbOrderJobs jobs;
  memset(&jobs, 0, sizeof(jobs));
  jobs.count = count;
  int64_t windows = 0;
  // A window is full, or there are several of one table: then the full ones take the time, and a choice per workgroup in one kernel
  // costs them more than it saves (a surface's tables of 20.7 k, 10.3 k, 3 k, 0.8 k and 0.2 k rows 34.1 us together, 34.5 so; the first
  // alone 34.0).
  bool whole = false;
  for (int i = 0; i < count; ++i) {
    const pce_osb_order_problem_t &p = problems[i];
    const int64_t n = p.n_rows;
    if (!p.nbr_dev || !p.order_dev) PCE_FAIL(PCE_EINVAL, "pce_osb_order: null pointer");
    if (p.kv <= 0 || p.kv > OSB_MAX_KV || p.mid >= p.kv)
      PCE_FAIL(PCE_EINVAL, "pce_osb_order: kv=%d outside [1, %d] or mid=%d", (int)p.kv, OSB_MAX_KV, (int)p.mid);
    if (n <= 0 || n >= (1ll << 31) / OSB_MAX_SLABS - OSB_WINDOW) PCE_FAIL(PCE_ECAPACITY, "pce_osb_order: n=%lld", (long long)n);
    if (p.order_elems < pce_osb_order_elems(n))
      PCE_FAIL(PCE_EWORKSPACE, "pce_osb_order: order holds %lld elements, needs %lld", (long long)p.order_elems, (long long)pce_osb_order_elems(n));
    OsbOrderJob &q = jobs.job[i];
    q.nbr = p.nbr_dev;
    q.known = (const unsigned *)p.mask_dev;
    q.centre = p.mid >= 0 ? 1u << p.mid : 0u;
    q.kv = p.kv;
    q.n = (int)n;
    q.window0 = (int)windows;
    q.perm = p.order_dev;
    q.bmask = (unsigned *)p.order_dev + osb_mask_offset(n);
    q.plans = p.order_dev + osb_plans_offset(n);
    windows += pce_div_up(n, OSB_WINDOW);
    whole |= n > OSB_WINDOW - OSB_ORDER_THREADS;
  }
  if (windows >= (1ll << 31)) PCE_FAIL(PCE_ECAPACITY, "pce_osb_order: too many rows");
  hipStream_t s = (hipStream_t)stream;
  if (whole)
    hipLaunchKernelGGL(osb_order_kernel<false>, dim3((unsigned)windows), dim3(OSB_ORDER_THREADS), 0, s, jobs);
  else
    hipLaunchKernelGGL(osb_order_kernel<true>, dim3((unsigned)windows), dim3(OSB_ORDER_THREADS), 0, s, jobs);
  PCE_LAUNCH_CHECK("osb_order");
  hipLaunchKernelGGL(osb_plan_kernel, dim3(8, OSB_MAX_SLABS, (unsigned)count), dim3(1024), 0, s, jobs);
  PCE_LAUNCH_CHECK("osb_plan");
  return PCE_OK;
}

extern "C" int pce_osb_order(const int32_t *nbr, const int32_t *mask, int32_t mid, int32_t kv, int64_t n, int32_t *order,
                             int64_t order_elems, pce_stream_t stream) {
  const pce_osb_order_problem_t p = {nbr, mask, mid, kv, n, order, order_elems};
  return pce_osb_order_batch(&p, 1, stream);
}

// ---- the convolution -----------------------------------------------------------------------------------------------
struct OsbArgs {
  const int *perm;
  const unsigned *bmask;
  float *part;          // partial sums of split items
  unsigned a_bytes;     // extent of the feature rows: gathers of a missing row lie beyond it and read as zero
  const int *plan;
  int cap;              // items per XCD in the plan
  int whole;            // no item is cut: the first part of a cut one does all of it
};

#define OSB_RB (OSB_ROWS / 16)
#define OSB_KC 64          // input channels per step: 128 bytes of a row, one line
#define OSB_ST 4           // stages of the ring of feature rows
#define OSB_STAGE (OSB_ROWS * OSB_KC / 8)   // 16-byte pieces per stage
#define OSB_A_LOADS (OSB_STAGE / 256)
#define OSB_MISSING 0xF0000000u

// 16 bytes per lane, global -> LDS: byte `off` of the range [base, base + bytes) to `dst` + 16 lane.  A lane whose offset
// lies beyond the range reads nothing and writes zero.  `base`, `bytes` and `dst` are uniform over the wavefront.
__device__ __forceinline__ void copy16_to_lds(const void *base, unsigned bytes, unsigned off, half8 *dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void *)base, 0, bytes, 0x00020000),
                                           (__attribute__((address_space(3))) void *)dst, 16, off, 0, 0, 0);
}
__device__ __forceinline__ unsigned lds_addr(const void *p) { return (unsigned)(uintptr_t)(__attribute__((address_space(3))) void *)p; }
// a load the compiler does not track: the caller waits by hand
__device__ __forceinline__ void load16_raw(u32x4 &v, unsigned off, const void *base) {
  asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(v) : "v"(off), "s"(base) : "memory");
}
// where the piece `p` of row `r` of a stage sits among the row's eight: sixteen consecutive rows read at one p meet
// sixteen different quarters of the bank row
__device__ __forceinline__ int osb_slot(int r, int p) { return p ^ ((r >> 1) & 7); }

// the fragments of one 16-row block (two 32-channel steps): request, and wait until at most N younger reads are out
#define OSB_READ(F_, RB_)                                                                                       \
  asm volatile("ds_read_b128 %0, %2 offset:%4\n\tds_read_b128 %1, %3 offset:%4"                                  \
               : "=&v"(F_[0]), "=&v"(F_[1]) : "v"(ra0), "v"(ra1), "n"((RB_) * 16 * OSB_KC * 2) : "memory")
#define OSB_WAIT(F_, N_) asm volatile("s_waitcnt lgkmcnt(" #N_ ")" : "+v"(F_[0]), "+v"(F_[1]) : : "memory")

// Sums of 16-row blocks -> finished rows in memory.  They go through the wavefront's LDS region in fp32, so that bias,
// residual and activation are applied to the eight consecutive columns a lane stores, and a residual is read as whole lines
// the way the rows are written (as 32 bytes of 16 rows an instruction, each block waited for: 566 us, 523 so), up to
// OSB_AHEAD blocks before it is added.
#define OSB_AHEAD 4
template <int CB>
struct OsbOut {
  static constexpr int LD = CB * 16 + 4;             // floats per row of the region
  static constexpr int PPR = CB * 2;                 // 16-byte pieces of a finished row
  static constexpr int ITS = (16 * PPR + 63) / 64;
  half8 bias[ITS], res[OSB_AHEAD][ITS];
  ActK act;
  static __device__ __forceinline__ int row(int it, int lane) { return (it * 64 + lane) / PPR; }
  static __device__ __forceinline__ int col(int it, int lane) { return (it * 64 + lane) % PPR * 8; }
  // rows: the output rows of the tile's blocks (-1: none)
  __device__ __forceinline__ void request(int rb, const int *rows, const TileArgs &a, int nw, int lane) {
    if (!a.res) return;
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int r = row(it, lane), c = nw + col(it, lane), dst = rows[rb * 16 + (r & 15)];
      const bool ok = r < 16 && dst >= 0 && c < a.c_out;
      res[rb % OSB_AHEAD][it] = *reinterpret_cast<const half8 *>((const half_t *)a.res + (ok ? (long long)dst * a.c_out + c : 0ll));
    }
  }
  __device__ __forceinline__ void init(int blocks, const int *rows, const TileArgs &a, int nw, int lane) {
    act = act_coeffs(a.act, a.slope, a.act != PCE_ACT_NONE);
#pragma unroll
    for (int rb = 0; rb < OSB_AHEAD; ++rb)
      if (rb < blocks) request(rb, rows, a, nw, lane);
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int c = nw + col(it, lane);
      half8 b = {0, 0, 0, 0, 0, 0, 0, 0};
      if (a.bias && c < a.c_out) b = *reinterpret_cast<const half8 *>((const half_t *)a.bias + c);
      bias[it] = b;
    }
  }
  __device__ __forceinline__ void store(const f32x4 (&acc)[CB], int rb, const int *rows, const TileArgs &a, int nw, float *region, int lane) {
    const int l16 = lane & 15, q = lane >> 4;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) *reinterpret_cast<f32x4 *>(region + l16 * LD + cb * 16 + q * 4) = acc[cb];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int r = row(it, lane), c = nw + col(it, lane), dst = rows[rb * 16 + (r & 15)];
      const float *from = region + (r & 15) * LD + col(it, lane);
      const f32x4 v[2] = {*reinterpret_cast<const f32x4 *>(from), *reinterpret_cast<const f32x4 *>(from + 4)};
      half8 y;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        float x = v[i / 4][i % 4] + (float)bias[it][i];
        if (a.res) x += (float)res[rb % OSB_AHEAD][it][i];
        y[i] = (half_t)act_apply(x, act);
      }
      if (r < 16 && dst >= 0 && c < a.c_out)
        store_maybe_stream(reinterpret_cast<half8 *>((half_t *)a.out + (long long)dst * a.ldo + c), y, a.stream);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
};

// Zeros stand for a row's missing neighbour in the matrix products, and zero times a weight that is not finite is NaN.  Where a
// sum of the wavefront is NaN and one of its weights is not finite, the NaN sums of rows that miss such an offset are formed
// again, neighbour by neighbour.  `all`: the offsets the sums run over.  Costs a comparison per sum otherwise (256 -> 256 on
// 72 k rows: 178.4 us, 177.8 without), and the weights once more in a tile with a NaN (NaN features in a hundredth of those
// rows, which is nearly every tile: 193 us -> 395, 128 -> 192: 103 -> 160).
template <int CB>
__device__ __forceinline__ void osb_redo_nan(f32x4 (&acc)[OSB_RB][CB], const TileArgs &a, unsigned all, const int *rows, int nw, int lane) {
  bool nan = false;
#pragma unroll
  for (int rb = 0; rb < OSB_RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int i = 0; i < 4; ++i) nan |= acc[rb][cb][i] != acc[rb][cb][i];
  if (!__any(nan)) return;
  const int l16 = lane & 15, q = lane >> 4, n = (int)a.n_rows;
  const half8 *wp = (const half8 *)a.Wp;
  unsigned bad = 0;   // the offsets with a weight that is not finite in this wavefront's columns
  for (unsigned rest = all; rest; rest &= rest - 1) {
    const int kp = __ffs(rest) - 1;
    bool here = false;
    for (int k8 = q; k8 < a.k8_total; k8 += 4)
      for (int cb = 0; cb < CB; ++cb) {
        const int c = nw + cb * 16 + l16;
        const half8 w = wp[((long long)kp * a.k8_total + k8) * a.n_pad + (c < a.n_pad ? c : a.n_pad - 1)];
#pragma unroll
        for (int j = 0; j < 8; ++j) here |= !(fabsf((float)w[j]) <= 65504.f);
      }
    if (__any(here)) bad |= 1u << kp;
  }
  if (!bad) return;
#pragma clang loop unroll(disable)
  for (int e = 0; e < OSB_RB * CB * 4; ++e) {
    float v = 0.f;
    int at = e;   // (opaque, here and below: otherwise the comparisons are made once and fill the scalar registers)
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int rb = 0; rb < OSB_RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) v = (rb * CB + cb) * 4 + i == at ? acc[rb][cb][i] : v;
    const int row = rows[e / (4 * CB) * 16 + l16], c = nw + e / 4 % CB * 16 + q * 4 + e % 4;
    const bool mine = v != v && row >= 0 && c < a.c_out;
    if (!__any(mine)) continue;
    bool misses = false, live = mine;
    float sum = 0.f;
    for (int pass = 0; pass < 2; ++pass) {   // those offsets first: a sum they make NaN is done
      for (unsigned rest = pass == 0 ? bad : all & ~bad; rest && __any(live); rest &= rest - 1) {
        const int kp = __ffs(rest) - 1;
        const int nb = live ? a.nbr[(long long)kp * n + row] : -1;
        if (pass == 0) misses |= nb < 0;
        if (nb >= 0) {
          const half8 *f = (const half8 *)((const half_t *)a.A + (long long)nb * a.lda), *w = wp + (long long)kp * a.k8_total * a.n_pad + c;
          for (int k8 = 0; k8 < a.k8_total; ++k8) {
            const half8 x = f[k8], y = w[(long long)k8 * a.n_pad];
#pragma unroll
            for (int j = 0; j < 8; ++j) sum += (float)x[j] * (float)y[j];
          }
          live = !(sum != sum);
        }
      }
      live = live && misses;
    }
    v = mine && misses ? sum : v;
    asm volatile("" : "+v"(at));
#pragma unroll
    for (int rb = 0; rb < OSB_RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[rb][cb][i] = (rb * CB + cb) * 4 + i == at ? v : acc[rb][cb][i];
  }
}

// Bound by the matrix cores and by what keeps them from running: the gathers' L2 latency and the LDS reads (a wavefront
// reads 1 KB per 16-row block and step for CB matrix instructions of 16 clocks; four of them share the LDS port, so below
// CB = 4 the reads alone take as long as the instructions).  A tile of 128 rows holds its sums in registers (8 * CB
// tiles of 16x16 per wavefront) over all its offsets, so no partial row goes to memory and each weight tile is read
// once per 128 rows.  Two workgroups per compute unit; the four wavefronts of one share the rows and split the columns: the
// weights of a wavefront are its own, go straight to registers and need no LDS.  Chunks of 64 channels outside, offsets inside:
// the same rows' 128-byte pieces are gathered for 27 offsets in a row and stay in the L2.
// fp16, pairs per row in brackets, against the dataflow that was taken before: 256 -> 256 on 72 k rows (9) 180 us against 278
// (deferred scatter), matrix cores busy for 59 % of the cycles a compute unit has workgroups and 49 % of the launch (the
// blocks multiply 2.0 times the useful products); the layers of the eight indoor scenes' network 15.7 ms
// against 25.
// TAIL: the last chunk of input channels has 32 of them.
template <int CB, bool TAIL>
__global__ void __launch_bounds__(256, 2) osb_kernel(TileArgs a, OsbArgs o) {
  constexpr int COLS = 4 * CB * 16;
  constexpr int W_LOADS = 2 * CB;
  constexpr int NW = CB == 2 ? 4 : CB == 3 ? 3 : 2;   // steps whose weights are held or on their way: what the registers allow
  // younger operations that may be out where a step's weights must have landed (those of the NW - 1 steps behind it, with the copies
  // between) and where the next step's rows must have (the copies of one step, and the weights issued around them)
  constexpr int OUT_W = (NW - 1) * (OSB_A_LOADS + W_LOADS), OUT_A = OSB_A_LOADS + 2 * W_LOADS;
  static_assert(OUT_W <= 63 && OUT_A <= 63, "vmcnt is a 6-bit counter");
  __shared__ __attribute__((aligned(128))) half8 lds[OSB_ST * OSB_STAGE];
  // byte offset of the neighbour row at every offset; the four rows whose pieces a lane gathers lie side by side
  __shared__ __attribute__((aligned(16))) unsigned src[OSB_MAX_KV + 1][OSB_ROWS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  // item of this workgroup: workgroups are dealt to the XCDs round robin
  const int xcd = blockIdx.x % PCE_XCDS, at = blockIdx.x / PCE_XCDS;
  const int2 it = ((const int2 *)(o.plan + 8 * (2 * OSB_MAX_CUT)))[(long long)xcd * o.cap + at];
  if (it.x < 0) return;
  const int part = it.y & 255, parts = o.whole ? 1 : (it.y >> 8) & 255, slot = it.y >> 16;
  if (o.whole && part > 0) return;
  const int tile = it.x / a.slabs;
  const int nw = (it.x % a.slabs) * COLS + wave * CB * 16;   // first column of this wavefront
  const int n = (int)a.n_rows;

  unsigned own[OSB_RB], all = 0;
#pragma unroll
  for (int rb = 0; rb < OSB_RB; ++rb) {
    const int b = tile * OSB_RB + rb;
    own[rb] = b * 16ll < n ? o.bmask[b] : 0u;
    all |= own[rb];
  }
  if (parts > 1) {   // this part's share of the tile's offsets, consecutive ones
    const int bits = __popc(all), lo = part * bits / parts, hi = (part + 1) * bits / parts;
    unsigned keep = 0, rest = all;
    for (int i = 0; i < hi; ++i) {
      const unsigned low = rest & (0u - rest);
      if (i >= lo) keep |= low;
      rest ^= low;
    }
    all = keep;
  }
  __shared__ int rows[OSB_ROWS];
  {
    const int r = threadIdx.x & (OSB_ROWS - 1), half = threadIdx.x / OSB_ROWS;
    const long long p = (long long)tile * OSB_ROWS + r;
    const int row = p < n ? o.perm[p] : -1;
    if (half == 0) rows[r] = row;
    // The offsets some row of the tile has go to the two halves of the workgroup in turn; every table read of the thread is
    // requested before the first one is used.  The other offsets' entries are not read (of 27 offsets a tile of the 951 k-row
    // level of the indoor scenes has 7: 614 us with all of them, 566 without).
    int nb[(OSB_MAX_KV + 1) / 2], kp[(OSB_MAX_KV + 1) / 2];
    unsigned left = all;
#pragma unroll
    for (int i = 0; i < (OSB_MAX_KV + 1) / 2; ++i) {
      const unsigned b0 = left & (0u - left);
      left ^= b0;
      const unsigned b1 = left & (0u - left);
      left ^= b1;
      const unsigned mine = half ? b1 : b0;
      kp[i] = mine ? __ffs(mine) - 1 : -1;
      if (b0) nb[i] = a.nbr[(long long)(mine ? kp[i] : 0) * n + (row >= 0 ? row : 0)];
    }
    const int at = (r & ~31) + (r & 7) * 4 + ((r >> 3) & 3);
#pragma unroll
    for (int i = 0; i < (OSB_MAX_KV + 1) / 2; ++i)
      if (kp[i] >= 0) src[kp[i]][at] = row >= 0 && nb[i] >= 0 ? (unsigned)nb[i] * (unsigned)(a.lda * 2) : OSB_MISSING;
    if (half) src[OSB_MAX_KV][at] = OSB_MISSING;   // what the steps behind the last one read
  }
  const int kch = (a.c_in + OSB_KC - 1) / OSB_KC;
  const int steps = __popc(all) * kch;
  f32x4 acc[OSB_RB][CB];
#pragma unroll
  for (int rb = 0; rb < OSB_RB; ++rb)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[rb][cb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // this lane's weight fragments: columns of its blocks, k = 8 q .. of a 32-channel step
  unsigned woff[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) {
    const int c = nw + cb * 16 + l16;
    woff[cb] = (unsigned)((q * a.n_pad + (c < a.n_pad ? c : a.n_pad - 1)) * 16);
  }
  unsigned gp[OSB_A_LOADS];   // this lane's piece of its four rows
#pragma unroll
  for (int i = 0; i < OSB_A_LOADS; ++i) gp[i] = osb_slot(wave * 32 + i * 8 + lane / 8, lane & 7) * 16;
  const unsigned src_addr = lds_addr(&src[0][wave * 32 + lane / 8 * 4]);
  const unsigned row_addr = lds_addr(lds) + l16 * (OSB_KC * 2) + osb_slot(l16, q) * 16;
  __syncthreads();

  // The steps run over all offsets for one chunk of 64 channels, then over all of them for the next: the workgroups of
  // an XCD then share one line of each of their rows and one chunk of the weights at a time, which fit its L2 together
  // (256 channels: 2 MB, all of them 8).
  unsigned rest = all;
  int chunk = 0;
#define OSB_NEXT(K_, C_)               /* the cursor's step, and on; behind the last one a row table without rows */     \
  {                                                                                                                     \
    K_ = chunk < kch ? __builtin_ctz(rest) : OSB_MAX_KV;                                                                \
    C_ = chunk;                                                                                                         \
    rest &= rest - 1;                                                                                                   \
    if (rest == 0) {                                                                                                    \
      rest = all;                                                                                                       \
      ++chunk;                                                                                                          \
    }                                                                                                                   \
  }
  u32x4 as;
  u32x4 wf[NW][W_LOADS] = {};
#define OSB_SRC(K_) asm volatile("ds_read_b128 %0, %1" : "=&v"(as) : "v"(src_addr + (K_) * (OSB_ROWS * 4)) : "memory")
#define OSB_ISSUE_A(ST_, C_)                                                                                            \
  _Pragma("unroll") for (int i = 0; i < OSB_A_LOADS; ++i)                                                               \
      copy16_to_lds(a.A, o.a_bytes, as[i] + gp[i] + (C_) * (OSB_KC * 2), lds + (ST_) * OSB_STAGE + (wave * OSB_A_LOADS + i) * 64);
#define OSB_ISSUE_W(B_, K_, C_)                                                                                         \
  {                                                                                                                     \
    const int kp = (C_) < kch ? (K_) : 0, c = (C_) < kch ? (C_) : 0;                                                    \
    const char *wb = (const char *)a.Wp + (long long)(kp * a.k8_total + c * (OSB_KC / 8)) * a.n_pad * 16;               \
    const char *wb1 = wb + (TAIL && c + 1 == kch ? 0 : 4 * a.n_pad * 16);                                             \
    _Pragma("unroll") for (int cb = 0; cb < CB; ++cb) load16_raw(wf[B_][cb], woff[cb], wb);                             \
    _Pragma("unroll") for (int cb = 0; cb < CB; ++cb) load16_raw(wf[B_][CB + cb], woff[cb], wb1);                       \
  }
  // at most N_ operations are out: this step's weights have landed
#define OSB_WEIGHTS(B_, N_)                                                                                             \
  {                                                                                                                     \
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N_) : "memory");                                                         \
    _Pragma("unroll") for (int i = 0; i < W_LOADS; ++i) asm volatile("" : "+v"(wf[B_][i]) : : "memory");                \
  }
  // the next step's rows have landed in every wavefront, and every wavefront is done with the stage that is filled next
#define OSB_ROWS_LANDED(N_) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" : : "n"(N_) : "memory");
#define OSB_BLOCK(F_, RB_, B_)                                                                                          \
  if ((own[RB_] >> k0) & 1u) {                                                                                          \
    _Pragma("unroll") for (int cb = 0; cb < CB; ++cb)                                                                   \
        acc[RB_][cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wf[B_][cb]), __builtin_bit_cast(half8, F_[0]), acc[RB_][cb], 0, 0, 0); \
    if (!half_step) {                                                                                                   \
      _Pragma("unroll") for (int cb = 0; cb < CB; ++cb)                                                                 \
          acc[RB_][cb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, wf[B_][CB + cb]), __builtin_bit_cast(half8, F_[1]), acc[RB_][cb], 0, 0, 0); \
    }                                                                                                                   \
  }
  // A step begins with its first four blocks' fragments on their way; in its middle the next step's rows are there, and their first
  // blocks are requested between the last four blocks' products.  (With all of it at the head of a step, the
  // products waited from the barrier to the first fragments: 256 -> 256 on 72 k rows 179.4 us, 176.9 so; the layers of the eight indoor
  // scenes' network 9.2 ms, 9.0.)
#define OSB_STEP(B_, N_)                                                                                                \
  {                                                                                                                     \
    OSB_WEIGHTS(B_, OUT_W)                                                                                              \
    const unsigned ra0 = row_addr + (t & (OSB_ST - 1)) * (OSB_STAGE * 16), ra1 = ra0 ^ 64;                              \
    const bool half_step = TAIL && c0 + 1 == kch;                                                                       \
    OSB_WAIT(f0, 6); OSB_BLOCK(f0, 0, B_) OSB_READ(f0, 4);                                                              \
    OSB_WAIT(f1, 6); OSB_BLOCK(f1, 1, B_) OSB_READ(f1, 5);                                                              \
    OSB_WAIT(f2, 6); OSB_BLOCK(f2, 2, B_) OSB_READ(f2, 6);                                                              \
    OSB_WAIT(f3, 6); OSB_BLOCK(f3, 3, B_) OSB_READ(f3, 7);                                                              \
    asm volatile("" : "+v"(as) : : "memory");                                                                           \
    OSB_ROWS_LANDED(N_)                                                                                                 \
    OSB_ISSUE_A((t + 3) & (OSB_ST - 1), c3)                                                                             \
    int k4, c4;                                                                                                         \
    OSB_NEXT(k4, c4)                                                                                                    \
    OSB_SRC(k4);                                                                                                        \
    {                                                                                                                   \
      const unsigned ra0 = row_addr + ((t + 1) & (OSB_ST - 1)) * (OSB_STAGE * 16), ra1 = ra0 ^ 64;                      \
      OSB_WAIT(f0, 7); OSB_BLOCK(f0, 4, B_) OSB_READ(f0, 0);                                                            \
      OSB_WAIT(f1, 7); OSB_BLOCK(f1, 5, B_) OSB_READ(f1, 1);                                                            \
      OSB_WAIT(f2, 7); OSB_BLOCK(f2, 6, B_) OSB_READ(f2, 2);                                                            \
      OSB_WAIT(f3, 7); OSB_BLOCK(f3, 7, B_) OSB_READ(f3, 3);                                                            \
    }                                                                                                                   \
    __builtin_amdgcn_sched_barrier(0);                                                                                  \
    if (NW == 2) OSB_ISSUE_W(B_, k2, c2)                                                                                \
    if (NW == 3) OSB_ISSUE_W(B_, k3, c3)                                                                                \
    if (NW == 4) OSB_ISSUE_W(B_, k4, c4)                                                                                \
    k0 = k1; c0 = c1; k1 = k2; c1 = c2; k2 = k3; c2 = c3; k3 = k4; c3 = c4;                                             \
  }
  if (steps > 0) {
    // steps t, t + 1, t + 2 (feature rows on their way) and t + 3 (their addresses)
    int k0, c0, k1, c1, k2, c2, k3, c3;
    OSB_NEXT(k0, c0)
    OSB_NEXT(k1, c1)
    OSB_NEXT(k2, c2)
    OSB_NEXT(k3, c3)
    OSB_ISSUE_W(0, k0, c0)
    OSB_ISSUE_W(1, k1, c1)
    if (NW > 2) OSB_ISSUE_W(NW > 2 ? 2 : 0, k2, c2)
    if (NW > 3) OSB_ISSUE_W(NW > 3 ? 3 : 0, k3, c3)
    OSB_SRC(k0);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(as) : : "memory");
    OSB_ISSUE_A(0, c0)
    OSB_SRC(k1);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(as) : : "memory");
    OSB_ISSUE_A(1, c1)
    OSB_SRC(k2);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(as) : : "memory");
    OSB_ISSUE_A(2, c2)
    OSB_SRC(k3);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(as) : : "memory");
    // the first step's rows and the weights of the first NW are there once two steps' copies are out
    OSB_ROWS_LANDED(2 * OSB_A_LOADS)
    u32x4 f0[2], f1[2], f2[2], f3[2];
    {
      const unsigned ra0 = row_addr, ra1 = ra0 ^ 64;
      OSB_READ(f0, 0); OSB_READ(f1, 1); OSB_READ(f2, 2); OSB_READ(f3, 3);
    }
    int t = 0;
    OSB_STEP(0, OSB_A_LOADS)
    if (++t < steps) OSB_STEP(1, OSB_A_LOADS + W_LOADS)
    if (++t < steps) OSB_STEP(2 % NW, OUT_A)
    for (++t; t < steps; ++t) {
      OSB_STEP(3 % NW, OUT_A)
      if (++t < steps) OSB_STEP(4 % NW, OUT_A)
      if (NW > 2 && ++t < steps) OSB_STEP(5 % NW, OUT_A)
      if (NW > 3 && ++t < steps) OSB_STEP(6 % NW, OUT_A)
    }
    // the reads behind the last step
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f0[0]), "+v"(f0[1]), "+v"(f1[0]), "+v"(f1[1]), "+v"(f2[0]), "+v"(f2[1]), "+v"(f3[0]), "+v"(f3[1]),
                 "+v"(as) : : "memory");
  }
  // the copies and loads behind the last step end before their destinations are used for anything else
#pragma unroll
  for (int b = 0; b < NW; ++b)
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i) asm volatile("s_waitcnt vmcnt(0)" : "+v"(wf[b][i]) : : "memory");
#undef OSB_STEP
#undef OSB_BLOCK
#undef OSB_ROWS_LANDED
#undef OSB_WEIGHTS
#undef OSB_ISSUE_W
#undef OSB_ISSUE_A
#undef OSB_SRC
#undef OSB_NEXT
  osb_redo_nan<CB>(acc, a, all, rows, nw, lane);
  if (parts > 1) {
    // partial sums as they lie in the registers: [slot][wavefront][block][column block][lane] of 16 bytes
    f32x4 *dst = (f32x4 *)o.part + ((long long)slot * 4 + wave) * (OSB_RB * CB * 64) + lane;
#pragma unroll
    for (int rb = 0; rb < OSB_RB; ++rb)
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) dst[(rb * CB + cb) * 64] = acc[rb][cb];
    return;
  }
  __syncthreads();  // the ring becomes the epilogue staging area
  OsbOut<CB> out;
  out.init(OSB_RB, rows, a, nw, lane);
  float *region = (float *)lds + wave * (16 * OsbOut<CB>::LD);
#pragma unroll
  for (int rb = 0; rb < OSB_RB; ++rb) {
    out.store(acc[rb], rb, rows, a, nw, region, lane);
    if (rb + OSB_AHEAD < OSB_RB) out.request(rb + OSB_AHEAD, rows, a, nw, lane);
  }
}

// Sums the parts of the cut items in their order and finishes the rows: a workgroup per item and 16-row block, a wavefront
// per column group.
template <int CB>
__global__ void __launch_bounds__(256) osb_reduce_kernel(TileArgs a, OsbArgs o) {
  __shared__ __attribute__((aligned(16))) float lds[4][16 * OsbOut<CB>::LD];
  __shared__ int rows[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x % PCE_XCDS, c = blockIdx.x / PCE_XCDS / OSB_RB, rb = blockIdx.x / PCE_XCDS % OSB_RB;
  const int *cut = o.plan + (x * OSB_MAX_CUT + c) * 2;
  const int item = cut[0], parts = cut[1];
  if (item < 0) return;
  const int nw = (item % a.slabs) * (4 * CB * 16) + wave * CB * 16;
  const long long p0 = (long long)(item / a.slabs) * OSB_ROWS + rb * 16;
  if (threadIdx.x < 16) rows[threadIdx.x] = p0 + threadIdx.x < a.n_rows ? o.perm[p0 + threadIdx.x] : -1;
  __syncthreads();
  if (p0 >= a.n_rows || nw >= a.c_out) return;
  OsbOut<CB> out;
  out.init(1, rows, a, nw, lane);
  f32x4 acc[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const f32x4 *from = (const f32x4 *)o.part + ((long long)(x * OSB_SLOTS + c * parts) * 4 + wave) * (OSB_RB * CB * 64) + rb * CB * 64 + lane;
  f32x4 v[OSB_MAX_PARTS][CB];
#pragma unroll
  for (int k = 0; k < OSB_MAX_PARTS; ++k)
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) v[k][cb] = from[(long long)(k < parts ? k : 0) * (4 * OSB_RB * CB * 64) + cb * 64];
#pragma unroll
  for (int k = 0; k < OSB_MAX_PARTS; ++k)
    if (k < parts) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] += v[k][cb];
    }
  out.store(acc, 0, rows, a, nw, lds[wave], lane);
}

// column blocks of 16 per wavefront (four wavefronts beside one another) and column slabs of a layer
static void osb_shape(int64_t n, int c_out, int *cb, int *slabs) {
  *slabs = (int)pce_div_up(c_out, 256);
  *cb = (int)pce_div_up(c_out, *slabs * 64);
  if (*cb < 2) *cb = 2;
  // few tiles: 128 columns each make twice the items (27 k rows of 19 pairs, 256 -> 256: 104 us against 107; 806 rows:
  // 20 against 27)
  if (pce_div_up(n, OSB_ROWS) * *slabs <= 256 && c_out <= 128 * OSB_MAX_SLABS) *cb = 2;
  *slabs = (int)pce_div_up(c_out, *cb * 64);
}

extern "C" int pce_conv_osb_takes(int32_t dtype, int32_t c_in, int32_t c_out, int32_t kv) {
  return dtype == PCE_F16 && c_in >= 64 && c_in % 32 == 0 && c_out >= 72 && c_out % 8 == 0 && c_out <= 256 * OSB_MAX_SLABS && kv >= 2 && kv <= OSB_MAX_KV;
}

// Pairs per row from which this kernel leads on deferred scatter.  Its time hardly depends on them, as long as the patterns
// are as mixed as those of a random cloud (a tile then meets 21 to 24 of 27 offsets; on walls and scans fewer, so it leads
// earlier there): it follows the rows and the product of the widths, while deferred scatter's follows the pairs.  The line is
// where the two met on random clouds of 0.6 k to 0.8 M rows, 1 to 13 pairs per row and 26 pairs of widths: highest at 12 k to
// 20 k rows, where deferred scatter's launches are long enough and its partial rows still in the caches, lower for fewer rows
// (one launch against several) and for more (partial rows in memory), and the higher the more input channels are gathered
// for each offset.  Crossings: 128 -> 192 7 at 15 k rows, 4 at 40 k, below 1.8 from 95 k; 192 -> 192 4 at 2 k, 9 at 15 k, 5
// at 40 k; 256 -> 256 10 at 15 k, 6 at 60 k, below 1.8 from 150 k; 512 -> 512 10 to 13 up to 30 k, 6 to 7 beyond.  Of 3920
// layers on random clouds, LiDAR and indoor pyramids 1660 take this kernel: 19 of them 2 to 16 % slower than the other
// choice, the mean 1.53 times faster.
static double osb_from(double n, int c_in, int c_out) {
  const double prod = (double)c_in * c_out;
  const int c = (c_in + OSB_KC - 1) / OSB_KC * OSB_KC;   // channels it multiplies
  double from = 7.5 + 4.0 * log2(c / 128.0);
  from = from < 7.5 ? 7.5 : from > 13.0 || prod >= 262144 ? 13.0 : from;
  const bool narrow = c_out <= 128 && c >= 160;          // much to gather, short partial rows
  if (n < 12000)
    from *= pow(n / 12000, prod >= 131072 ? 0.05 : c >= 384 ? 0.2 : 0.25);
  else if (n > 20000)
    from *= pow(20000 / n, narrow ? (c_in < 192 ? 0.35 : 0.4) : c >= 384 ? 0.55 : c >= 256 ? 0.6 : 0.7);
  if (c >= 256 && c_out >= 2 * c && c_out <= 512) from *= 0.8;   // long partial rows
  double least = c_out <= 128 ? 1.85 : (c > 256 && prod > 65536) || prod > 131072 ? 1.8 + (prod - 65536) / 38000 : 1.5;
  if (least > 9.5) least = 9.5;
  return from > least ? from : least;
}

// Submanifold layers this kernel leads on: from osb_from() on against deferred scatter, and wherever the general selector
// would take the dense tiles, which multiply every offset (128 -> 128 at 7 pairs per row on 20 k rows 0.76 of their time, at
// 19 on 27 k 0.85; not with 64 and 96 channels on 12 k to 50 k rows with 11 and more: 64 -> 192
// at 12 on 16 k rows 1.21).  On the widths the ordered rows of the K-stepped kernel take as well: to 128 columns from five pairs per
// row on 60 k rows and more (0.65-0.95 of their time), to fewer from five to twelve on a million pairs and more (0.78-0.98;
// 96 -> 96 with 0.4 to 0.9 million 1.05-1.26), from 112 channels where the dense tiles are the other choice.
extern "C" int pce_conv_osb_leads(int64_t n_out, int64_t n_pairs, int32_t c_in, int32_t c_out, int32_t kv, int32_t mid, int32_t dtype) {
  if (n_out <= 0 || mid < 0 || !pce_conv_osb_takes(dtype, c_in, c_out, kv)) return 0;
  const double n = (double)n_out, rho = (double)n_pairs / n;
  const bool dense = pce_select_dataflow(n_out, n_out, n_pairs, c_in, c_out, kv, mid, 0, dtype) == PCE_DATAFLOW_OS;
  if (!pce_conv_oso_takes(dtype, c_in, c_out, kv, mid))
    return dense ? c_in >= 128 || rho < 11.0 || n_out < 12000 || n_out >= 50000 : rho >= osb_from(n, c_in, c_out);
  if (c_in >= 112) return dense && (n_out >= 60000 || (n_out >= 25000 && rho >= 9.0));
  return c_out >= 128 ? n_out >= 60000 && rho >= 5.0 : rho >= 5.0 && rho <= 12.0 && n_pairs >= 1000000;
}

extern "C" int pce_select_layer(int64_t n_in, int64_t n_out, int64_t n_pairs, int32_t c_in, int32_t c_out, int32_t kv, int32_t mid,
                                int32_t transposed, int32_t dtype) {
  if (mid >= 0 && (!transposed || kv % 2 == 1) && n_in * c_in * 2 < (int64_t)OSB_MISSING &&
      pce_conv_osb_leads(n_out, n_pairs, c_in, c_out, kv, mid, dtype))
    return PCE_DATAFLOW_OSB;
  return pce_select_dataflow(n_in, n_out, n_pairs, c_in, c_out, kv, mid, transposed, dtype);
}

extern "C" int64_t pce_conv_osb_workspace_bytes(int64_t n_out, int32_t c_out) {
  int cb, slabs;
  osb_shape(n_out, c_out, &cb, &slabs);
  return (int64_t)8 * OSB_SLOTS * OSB_ROWS * cb * 64 * 4;
}

// Whether cutting items pays for the second launch (5-8 us): the steps a tile is expected to take, from the pairs per
// row (tiles of sorted rows meet two to three times as many offsets as a row has), at about half a microsecond each.
static bool osb_cuts(int64_t n_out, int64_t n_pairs, int c_in, int kv, long long items) {
  const double rho = n_pairs >= 0 ? (double)n_pairs / (double)n_out + 1.0 : kv;
  const double steps = (rho * 2.5 < kv ? rho * 2.5 : kv) * (double)pce_div_up(c_in, OSB_KC);
  return steps >= 24 && items < 16 * 8 * OSB_SLOTS;
}

extern "C" int64_t pce_conv_osb_scratch_bytes(int64_t n_out, int64_t n_pairs, int32_t c_in, int32_t c_out, int32_t kv) {
  if (n_out <= 0 || c_out <= 0) return 0;
  int cb, slabs;
  osb_shape(n_out, c_out, &cb, &slabs);
  return osb_cuts(n_out, n_pairs, c_in, kv, pce_div_up(n_out, OSB_ROWS) * slabs) ? pce_conv_osb_workspace_bytes(n_out, c_out) : 0;
}

extern "C" int pce_conv_fwd_osb(const void *in, const void *wp, void *out, int32_t dtype, int64_t n_in, int64_t n_out, int64_t n_pairs,
                                int32_t c_in, int32_t c_out, int32_t kv, const int32_t *nbr, const int32_t *order, void *ws, int64_t ws_bytes,
                                const pce_epilogue_t *epilogue, pce_stream_t stream) {
  int rc = check_common("pce_conv_fwd_osb", in, wp, out, dtype, n_in, n_out, c_in, c_out, kv, -1);
  if (rc) return rc;
  if (!pce_conv_osb_takes(dtype, c_in, c_out, kv))
    PCE_FAIL(PCE_EINVAL, "pce_conv_fwd_osb: dtype %d, %d -> %d channels, %d offsets: see pce_conv_osb_takes", dtype, c_in, c_out, kv);
  if (!nbr || !order) PCE_FAIL(PCE_EINVAL, "pce_conv_fwd_osb: null neighbour table or order");
  Epi e;
  if ((rc = read_epilogue("pce_conv_fwd_osb", epilogue, out, &e, c_in, c_out))) return rc;
  TileArgs a = base_args<half_t>(in, nullptr, wp, kv, c_in, c_out, e.lda);
  set_out<half_t>(&a, out, false, n_out, e.ldo);
  set_epi(&a, e);
  a.nbr = nbr;
  a.n_rows = n_out;
  if (!a.a_vec || !a.o_vec || !aligned16(wp) || !epi_aligned(e)) PCE_FAIL(PCE_EINVAL, "pce_conv_fwd_osb: pointers must be 16-byte aligned");
  const int64_t a_bytes = ((n_in - 1) * (int64_t)a.lda + c_in) * 2;
  if (a_bytes >= (int64_t)OSB_MISSING || n_out >= (1ll << 31) / OSB_MAX_SLABS - OSB_WINDOW)
    PCE_FAIL(PCE_ECAPACITY, "pce_conv_fwd_osb: %lld bytes of features, %lld rows", (long long)a_bytes, (long long)n_out);
  int cb, slabs;
  osb_shape(n_out, c_out, &cb, &slabs);
  const bool cuts = osb_cuts(n_out, n_pairs, c_in, kv, pce_div_up(n_out, OSB_ROWS) * slabs);
  if (ws ? !aligned16(ws) || ws_bytes < pce_conv_osb_workspace_bytes(n_out, c_out) : cuts)
    PCE_FAIL(PCE_EWORKSPACE, "pce_conv_fwd_osb: workspace of %lld bytes, needs %lld", (long long)ws_bytes, (long long)pce_conv_osb_workspace_bytes(n_out, c_out));
  const long long tiles = pce_div_up(n_out, OSB_ROWS);
  OsbArgs o = {};
  o.perm = order;
  o.bmask = (const unsigned *)order + osb_mask_offset(n_out);
  o.plan = order + osb_plans_offset(n_out) + osb_plan_offset(tiles, slabs);
  o.cap = (int)osb_plan_cap(tiles, slabs);
  o.part = (float *)ws;
  o.a_bytes = (unsigned)a_bytes;
  o.whole = !cuts;
  a.slabs = slabs;
  hipStream_t s = (hipStream_t)stream;
  const unsigned grid = (unsigned)(8 * o.cap);
#define OSB_CASE(CB_)                                                                                    \
  if (cb == CB_) {                                                                                       \
    if (c_in % OSB_KC)                                                                                   \
      hipLaunchKernelGGL((osb_kernel<CB_, true>), dim3(grid), dim3(256), 0, s, a, o);                    \
    else                                                                                                 \
      hipLaunchKernelGGL((osb_kernel<CB_, false>), dim3(grid), dim3(256), 0, s, a, o);                   \
    PCE_LAUNCH_CHECK("osb");                                                                             \
    if (!o.whole) {                                                                                      \
      hipLaunchKernelGGL((osb_reduce_kernel<CB_>), dim3(8 * OSB_MAX_CUT * OSB_RB), dim3(256), 0, s, a, o); \
      PCE_LAUNCH_CHECK("osb_reduce");                                                                    \
    }                                                                                                    \
  }
  OSB_CASE(2)
  OSB_CASE(3)
  OSB_CASE(4)
#undef OSB_CASE
  return PCE_OK;
}
