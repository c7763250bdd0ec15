// Types, tile arguments, epilogues and argument checks shared by the convolution translation units.
#pragma once
#include "pce_common.h"

typedef _Float16 half_t;
typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T, int N>
struct VecOfC;
template <>
struct VecOfC<half_t, 8> { typedef half8 type; };
template <>
struct VecOfC<float, 4> { typedef f32x4 type; };
template <>
struct VecOfC<half_t, 4> { typedef _Float16 type __attribute__((ext_vector_type(4))); };

// plain store, or one with the non-temporal hint (see store_rows_via_lds) when the host asked for it
template <typename V>
__device__ __forceinline__ void store_maybe_stream(V *p, const V &v, bool stream) {
  if (stream)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

enum {
  MODE_FOD = 0,      // A row = imap[pair], out row = omap[pair]
  MODE_BUF = 1,      // A row = out row = quantised pair row (staging buffer)
  MODE_DENSE = 2,    // A row = out row = tile row, one fixed weight
  MODE_OS = 3,       // out row = tile row, A row = nbr[kp][row], loop over all offsets
  MODE_FOD_BUF = 4   // A row = imap[pair], out row = oslot[pair] (partial-row buffer in output-CSR order)
};
enum {
  EPI_ATOMIC_F32 = 0,  // fp32 atomic add, one column per lane
  EPI_ROWS = 1,        // store T, 16 bytes per lane along the row
  EPI_ROWS_F32 = 2,    // store fp32 (accumulator of the atomic dataflow), 16 bytes per lane
  EPI_ROWS_CSR = 3     // EPI_ROWS plus the sum of partial rows buf[ocsr[row] .. ocsr[row+1])
};

#define PCE_ROUTE_HEAD 4  // ints in front of the pair destinations of a routing array (pce_pair_route)
#define MAX_KV_ARGS 32  // kpos / qkpos travel in the kernel arguments up to this kernel volume

struct TileArgs {
  const void *A;
  const void *W;
  const void *Wp;  // fp16 weights in LDS-image order, or null
  void *out;
  const int *imap;
  const int *omap;
  const int *kpos;
  const int *qkpos;
  const int *nbr;
  const int *ocsr;
  const int *oslot;
  const void *buf;
  long long n_rows;  // MODE_DENSE / MODE_OS: rows of the output
  long long a_rows;  // MODE_OS: rows of A (0: not stated)
  long long items;   // (tile, column slab) work items of the launch
  int slabs;         // column slabs per tile
  int groups;        // MODE_OS, small_f32_kernel (not tile_gemm_kernel): groups of offsets whose sums are added up from zero (0, 1: one)
  int parts;         // MODE_OS: shares of the offsets, blockIdx.y; the sums of share p at out + p * n_rows * c_out (0, 1: one)
  int kv, c_in, c_out;
  int lda, ldo;      // elements between consecutive rows of A and of `out` (rows of buf, res and out_alt are dense)
  int w_fixed;
  int mode, epi;
  int a_vec, w_vec, o_vec, b_vec;  // 16-byte accesses allowed on A rows / W rows / out rows / buf rows
  int k8_total, n_pad;             // packed weight extents
  int host_pos;                    // kpos_h / qkpos_h are valid
  const void *bias;                // fused epilogue of the launch that stores output rows: out = act(acc + bias + res)
  const void *res;
  int act;
  float slope;
  int act_alone_only;               // apply the activation only to rows without partial rows (ocsr tells)
  int stream;                       // output rows leave with the non-temporal hint (set_out)
  void *out_alt;                    // routed pair tiles: destination d < n_split is row d of `out` (a finished output
  int n_split;                      // row, takes the epilogue), d >= n_split is row d - n_split of `out_alt`
  int kpos_h[MAX_KV_ARGS + 1];
  int qkpos_h[MAX_KV_ARGS + 1];
};

// XCD-aware work mapping.  Workgroups are dealt to the 8 XCDs round-robin in launch order and each
// XCD has its own L2.  Neighbouring tiles read overlapping feature rows, so every XCD gets one
// contiguous range of the (tile, column slab) items instead of every eighth one.  The launch is one-
// dimensional with ceil8(items) workgroups; returns false for the padding workgroups.
#define PCE_XCDS 8
__device__ __forceinline__ bool xcd_item(long long items, int slabs, bool remap, long long *tile, int *slab) {
  long long lid = blockIdx.x;
  long long per = (items + PCE_XCDS - 1) / PCE_XCDS;
  long long item = remap ? (lid % PCE_XCDS) * per + lid / PCE_XCDS : lid;
  if ((remap && lid / PCE_XCDS >= per) || item >= items) return false;
  *tile = item / slabs;
  *slab = (int)(item % slabs);
  return true;
}

// Row epilogue, first step: the two lanes of a row (g = 0, 1) exchange 4-column pieces so that each
// ends with 8 consecutive columns per 16-column group: lane g owns columns 16*h + 8*g + 0..7,
// h = 0, 1, of every 32-column block.
template <int NB>
__device__ __forceinline__ void gather_row_pieces(const f32x16 (&acc)[NB], float (&V)[NB][2][8], int g) {
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int qa = 2 * h, qb = 2 * h + 1;  // lane g=0 keeps piece qa, lane g=1 keeps piece qb
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (NB > 2) {
          // wide tiles: a shuffle and two selects (the swap below costs the kernels that hold 64 accumulators per lane
          // a tenth of a network forward)
          float lo = acc[nb][4 * qa + i], hi = acc[nb][4 * qb + i];
          float recv = __shfl_xor(g == 0 ? hi : lo, 32, PCE_WAVE);
          V[nb][h][i] = g == 0 ? lo : recv;
          V[nb][h][4 + i] = g == 0 ? recv : hi;
        } else {
          // one instruction swaps the upper half of `lo` with the lower half of `hi`: lanes 0-31 then hold (own lo,
          // partner's lo), lanes 32-63 (partner's hi, own hi)
          auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[nb][4 * qa + i]), __float_as_uint(acc[nb][4 * qb + i]), false, false);
          V[nb][h][i] = __uint_as_float(r[0]);
          V[nb][h][4 + i] = __uint_as_float(r[1]);
        }
      }
    }
  }
}

// Per-wavefront LDS region, in 16-byte pieces: big enough for 16 fp32 rows or 32 fp16 rows of the
// output tile with 8 elements of padding per row.  It first stages partial rows, then the finished
// rows on their way to memory.
template <int NB>
struct WaveLds {
  static constexpr int NT = NB * 32;
  static constexpr int PIECES = 4 * (NT + 8);
};

// ---- fused epilogue: out = act(acc + bias + residual) -------------------------------------------
// Written without branches: with `act` a kernel argument the compiler turned the three-way form into scalar
// compares, jumps and a reload of the slope around every element of an unrolled epilogue.  The two
// coefficients depend on `act` alone and are hoisted out of the loops.
struct ActK {
  float mul;      // what a non-positive value is multiplied by ...
  unsigned keep;  // ... and whether the product survives
};
// `on` may differ from lane to lane (rows that get their activation in a later pass): it goes into the
// coefficients, not into a test around every element
__device__ __forceinline__ ActK act_coeffs(int act, float slope, bool on) {
  ActK k;
  k.mul = (on && act == PCE_ACT_LEAKY_RELU) ? slope : 1.f;
  k.keep = (on && act == PCE_ACT_RELU) ? 0u : ~0u;
  return k;
}
__device__ __forceinline__ float act_apply(float v, const ActK &k) {
  const float t = __uint_as_float(__float_as_uint(v * k.mul) & k.keep);
  return v > 0.f ? v : t;  // no activation: t == v
}
__device__ __forceinline__ float act_apply(float v, int act, float slope) { return act_apply(v, act_coeffs(act, slope, true)); }
// derivative of the activation where its output is `out` (ReLU and LeakyReLU with a positive slope keep the sign)
__device__ __forceinline__ float act_slope_at(float out, int act, float slope) {
  const float neg = act == PCE_ACT_RELU ? 0.f : (act == PCE_ACT_LEAKY_RELU ? slope : 1.f);
  return out > 0.f ? 1.f : neg;
}

// eight consecutive elements of a row of T as floats; VEC: the address is 16-byte aligned
template <typename T, bool VEC>
__device__ __forceinline__ void add8(float (&v)[8], const T *p, int valid) {
  if (VEC) {
    if (sizeof(T) == 2) {
      half8 x = *reinterpret_cast<const half8 *>(p);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += (float)x[j];
    } else {
      f32x4 x0 = *reinterpret_cast<const f32x4 *>(p), x1 = *reinterpret_cast<const f32x4 *>(p + 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] += (float)x0[j];
        v[4 + j] += (float)x1[j];
      }
    }
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < valid) v[j] += (float)p[j];
  }
}

// one 16-byte-aligned piece of eight elements of T, loaded whole (two 16-byte loads for fp32)
template <typename T>
struct Piece8;
template <>
struct Piece8<half_t> {
  half8 x;
  __device__ __forceinline__ void load(const half_t *p) { x = *reinterpret_cast<const half8 *>(p); }
  __device__ __forceinline__ float at(int j) const { return (float)x[j]; }
};
template <>
struct Piece8<float> {
  f32x4 x0, x1;
  __device__ __forceinline__ void load(const float *p) {
    x0 = *reinterpret_cast<const f32x4 *>(p);
    x1 = *reinterpret_cast<const f32x4 *>(p + 4);
  }
  __device__ __forceinline__ float at(int j) const { return j < 4 ? x0[j] : x1[j - 4]; }
};

// on the row pieces of the tile epilogue (lane g of row `orow` owns columns n0 + 32*nb + 16*h + 8*g + 0..7).
// VEC: every piece is 16-byte aligned and lies wholly inside or outside the row.  The pieces of the bias, then
// those of the residual row, are requested together from addresses that are valid for every lane (a lane
// without a row or column reads the base and drops the value), so that a lane waits once per operand: loads
// guarded piece by piece were issued and waited for one after the other, sixteen round trips at the end of
// every workgroup of a 128-column tile.
// Used where the register budget is fixed by the launch bounds anyway (the pipelined kernel: 128 registers, four
// workgroups per CU); in the tile kernel and the barrier-free kernel the addresses and pieces in flight cost a
// resident wavefront (output-stationary tile kernel at 128 columns: 97 -> 145 us), so those keep the guarded form.
// NBB: column blocks whose pieces are in flight together (8 registers per block for fp16 rows, 16 for fp32).
template <typename T, int NB, bool VEC, int NBB>
__device__ __forceinline__ void epilogue_row_pieces_batched(float (&V)[NB][2][8], const TileArgs &a, int orow, int n0, int g,
                                                            bool with_act) {
  const T *bias = (const T *)a.bias;
  const T *res = (const T *)a.res;
  if (VEC) {
#pragma unroll
    for (int op = 0; op < 2; ++op) {
      const T *base = op == 0 ? bias : res;
      if (!base) continue;
      const long long row_off = op == 0 ? 0ll : (long long)(orow >= 0 ? orow : 0) * a.c_out;
#pragma unroll
      for (int nb0 = 0; nb0 < NB; nb0 += NBB) {
        Piece8<T> x[NBB][2];
#pragma unroll
        for (int nb = 0; nb < NBB; ++nb)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            int c0 = n0 + (nb0 + nb) * 32 + 16 * h + 8 * g;
            bool ok = nb0 + nb < NB && orow >= 0 && c0 < a.c_out;
            x[nb][h].load(ok ? base + row_off + c0 : base);
          }
#pragma unroll
        for (int nb = 0; nb < NBB; ++nb)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if (nb0 + nb >= NB) continue;
            int c0 = n0 + (nb0 + nb) * 32 + 16 * h + 8 * g;
            bool ok = orow >= 0 && c0 < a.c_out;
#pragma unroll
            for (int j = 0; j < 8; ++j) V[nb0 + nb][h][j] += ok ? x[nb][h].at(j) : 0.f;
          }
      }
    }
  } else {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        int c0 = n0 + nb * 32 + 16 * h + 8 * g;
        int valid = a.c_out - c0;
        if (valid > 0 && orow >= 0) {
          if (bias) add8<T, false>(V[nb][h], bias + c0, valid);
          if (res) add8<T, false>(V[nb][h], res + (long long)orow * a.c_out + c0, valid);
        }
      }
  }
  const ActK k = act_coeffs(a.act, a.slope, with_act);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) V[nb][h][j] = act_apply(V[nb][h][j], k);
}

// the same with every piece guarded and added as it arrives: fewest registers
template <typename T, int NB, bool VEC>
__device__ __forceinline__ void epilogue_row_pieces(float (&V)[NB][2][8], const TileArgs &a, int orow, int n0, int g,
                                                    bool with_act) {
  const T *bias = (const T *)a.bias;
  const T *res = (const T *)a.res;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      int c0 = n0 + nb * 32 + 16 * h + 8 * g;
      int valid = a.c_out - c0;
      if (valid > 0 && orow >= 0) {
        if (bias) add8<T, VEC>(V[nb][h], bias + c0, valid);
        if (res) add8<T, VEC>(V[nb][h], res + (long long)orow * a.c_out + c0, valid);
      }
      if (with_act) {
#pragma unroll
        for (int j = 0; j < 8; ++j) V[nb][h][j] = act_apply(V[nb][h][j], a.act, a.slope);
      }
    }
}

// element-wise stores straight from the row pieces (rows that are not 16-byte multiples)
template <typename TO, int NB>
__device__ __forceinline__ void store_row_pieces_slow(const float (&V)[NB][2][8], TO *out, int orow, const TileArgs &a,
                                                      int n0, int g) {
  if (orow < 0) return;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        int col = n0 + nb * 32 + 16 * h + 8 * g + j;
        if (col < a.c_out) out[(long long)orow * a.ldo + col] = (TO)V[nb][h][j];
      }
}

// Finished rows -> memory through the wavefront's LDS region: the lane that owns (row, 8 columns)
// writes its pieces; then 16 bytes per lane are read back along the rows, so that NT*sizeof(TO)/16
// consecutive lanes store one full row segment (whole 128-byte lines at 64 fp16 channels).
// a.stream: the stores carry the non-temporal hint.  Rows kept as ordinary dirty lines are written back in one
// burst when the kernel ends (2.3 of 9.3 us on the 150 k-voxel layer); streamed out they leave while the kernel
// runs, but the next layer then finds none of them in the L2 of its XCD.  The host decides per launch (set_out).
template <typename TO, int NB, int ROWS = (sizeof(TO) == 2 ? 32 : 16), bool SPLIT = false>
__device__ __forceinline__ void store_rows_via_lds(const float (&V)[NB][2][8], void *region, TO *out, int orow,
                                                   const TileArgs &a, int n0, int lane, int l32, int g, bool stream,
                                                   int ld_out = -1) {   // row stride of `out` where it is not a.ldo
  constexpr int NT = NB * 32;
  constexpr int EPP = 16 / sizeof(TO);              // elements per piece
  constexpr int LDP = (NT + 8) / EPP;               // row stride in pieces; ROWS rows per pass
  constexpr int PPR = NT / EPP;                     // pieces per row
  constexpr int ITS = ROWS * PPR / 64;
  typedef typename VecOfC<TO, EPP>::type OV;
  OV *R = (OV *)region;
#pragma unroll
  for (int pass = 0; pass < 32 / ROWS; ++pass) {
    if ((l32 / ROWS) == pass) {
      int lr = l32 % ROWS;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          int c0 = nb * 32 + 16 * h + 8 * g;  // first of this lane's 8 columns
          if (sizeof(TO) == 2) {
            OV y;
#pragma unroll
            for (int j = 0; j < 8; ++j) y[j % EPP] = (TO)V[nb][h][j];
            R[lr * LDP + c0 / EPP] = y;
          } else {
            OV y0, y1;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              y0[j] = (TO)V[nb][h][j];
              y1[j] = (TO)V[nb][h][4 + j];
            }
            R[lr * LDP + c0 / EPP] = y0;
            R[lr * LDP + c0 / EPP + 1] = y1;
          }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      int idx = it * 64 + lane;
      int lr = idx / PPR, ch = idx - lr * PPR;
      int dst = __shfl(orow, pass * ROWS + lr, PCE_WAVE);
      int col = n0 + ch * EPP;
      OV y = R[lr * LDP + ch];
      TO *base = out;
      int ld = ld_out >= 0 ? ld_out : a.ldo;
      if (SPLIT && dst >= a.n_split) {
        base = (TO *)a.out_alt;
        dst -= a.n_split;
        ld = a.c_out;
      }
      if (dst >= 0 && col < a.c_out) {
        OV *dp = reinterpret_cast<OV *>(base + (long long)dst * ld + col);
        if (stream)
          __builtin_nontemporal_store(y, dp);
        else
          *dp = y;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

// Stage selection exists in the measurement build only (libpcengine_amd_measure.so, compiled with
// -DPCE_MEASURE): there a benchmark can run one kernel of a dataflow alone or pick a kernel family.  The
// product library compiles every test below to `true` and keeps no such state.
#ifdef PCE_MEASURE
extern unsigned g_stage_mask;
static inline bool stage_on(int bit) { return (g_stage_mask >> bit) & 1u; }
#else
static constexpr bool stage_on(int) { return true; }
#endif

// Output rows leave with the non-temporal hint when the tensor they belong to is larger than PCE_STREAM_MIN_BYTES:
// a tensor that size is written back from the L2s in one burst at the end of the kernel anyway, and streaming it
// out while the kernel runs hides that (150 k rows x 64 channels, 19 MB: 9.3 -> 7.0 us); a smaller one is better
// left in the L2 of the XCD that wrote it, where the next layer's tiles of the same rows find it.
#define PCE_STREAM_MIN_BYTES (16ll << 20)
static inline int stream_policy(long long bytes) {
  return stage_on(10) && (!stage_on(11) || bytes >= PCE_STREAM_MIN_BYTES);
}


static inline bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

static inline int check_common(const char *fn, const void *in, const void *w, const void *out, int dtype, int64_t n_in,
                        int64_t n_out, int c_in, int c_out, int kv, int mid) {
  if (!in || !w || !out) PCE_FAIL(PCE_EINVAL, "%s: null feature / weight pointer", fn);
  if (dtype != PCE_F16 && dtype != PCE_F32) PCE_FAIL(PCE_EINVAL, "%s: dtype must be PCE_F16 or PCE_F32", fn);
  if (n_in <= 0 || n_out <= 0 || c_in <= 0 || c_out <= 0 || kv <= 0)
    PCE_FAIL(PCE_EINVAL, "%s: sizes must be positive (n_in=%lld n_out=%lld c_in=%d c_out=%d kv=%d)", fn, (long long)n_in, (long long)n_out, c_in, c_out, kv);
  if (n_in >= (1ll << 31) || n_out >= (1ll << 31)) PCE_FAIL(PCE_ECAPACITY, "%s: row count exceeds int32", fn);
  if (mid >= kv) PCE_FAIL(PCE_EINVAL, "%s: mid=%d >= kv=%d", fn, mid, kv);
  if (mid >= 0 && n_in != n_out) PCE_FAIL(PCE_EINVAL, "%s: a centre offset needs n_in == n_out", fn);
  return PCE_OK;
}

// features / weights / packed weights / sizes common to every launch of one layer
template <typename T>
static inline TileArgs base_args(const void *in, const void *w, const void *wp, int kv, int c_in, int c_out, int lda = 0) {
  constexpr int VEC = sizeof(T) == 2 ? 8 : 4;
  TileArgs a = {};
  a.A = in;
  a.W = w;
  a.Wp = sizeof(T) == 2 ? wp : nullptr;
  a.kv = kv;
  a.c_in = c_in;
  a.c_out = c_out;
  a.lda = lda > 0 ? lda : c_in;
  a.ldo = c_out;
  a.k8_total = (c_in + 7) / 8;
  a.n_pad = (c_out + 31) / 32 * 32;
  a.a_vec = (c_in % VEC == 0) && aligned16(in);
  a.w_vec = (c_out % VEC == 0) && aligned16(w);
  return a;
}

// `rows` = rows of the tensor `out` points to (0: not known, no streaming)
template <typename T>
static inline void set_out(TileArgs *a, void *out, bool f32out, long long rows = 0, int ldo = 0) {
  // a lane of the row epilogue owns 8 consecutive columns, whatever the element type
  a->out = out;
  a->ldo = ldo > 0 ? ldo : a->c_out;
  a->o_vec = (a->c_out % 8 == 0) && aligned16(out);
  a->stream = rows > 0 ? stream_policy(rows * a->c_out * (f32out ? 4 : (long long)sizeof(T))) : 0;
}

struct Epi {
  const void *bias, *res;
  int act;
  float slope;
  int lda, ldo;   // row strides of the input and output matrices in elements, 0 = dense
  bool any() const { return bias || res || act != PCE_ACT_NONE; }
};

static inline int read_epilogue(const char *fn, const pce_epilogue_t *e, const void *out, Epi *o, int c_in = 0, int c_out = 0) {
  o->bias = o->res = nullptr;
  o->act = PCE_ACT_NONE;
  o->slope = 0.f;
  o->lda = o->ldo = 0;
  if (!e) return PCE_OK;
  // row strides: only the entry points that pass their channel counts take them
  if ((e->ld_in != 0 && e->ld_in != c_in) || (e->ld_out != 0 && e->ld_out != c_out)) {
    if (c_in <= 0) PCE_FAIL(PCE_EINVAL, "%s: this entry point takes dense feature matrices only (ld_in=%lld, ld_out=%lld)", fn, (long long)e->ld_in, (long long)e->ld_out);
    if ((e->ld_in != 0 && (e->ld_in < c_in || e->ld_in % 8)) || (e->ld_out != 0 && (e->ld_out < c_out || e->ld_out % 8)) ||
        e->ld_in >= (1ll << 31) || e->ld_out >= (1ll << 31))
      PCE_FAIL(PCE_EINVAL, "%s: row strides (ld_in=%lld, ld_out=%lld) must be multiples of 8 elements, at least the channel counts (%d, %d)", fn, (long long)e->ld_in, (long long)e->ld_out, c_in, c_out);
    o->lda = (int)e->ld_in;
    o->ldo = (int)e->ld_out;
  }
  if (e->act != PCE_ACT_NONE && e->act != PCE_ACT_RELU && e->act != PCE_ACT_LEAKY_RELU)
    PCE_FAIL(PCE_EINVAL, "%s: unknown activation %d", fn, (int)e->act);
  if (e->residual && e->residual == out) PCE_FAIL(PCE_EINVAL, "%s: the residual must not alias the output", fn);
  o->bias = e->bias;
  o->res = e->residual;
  o->act = e->act;
  o->slope = e->slope;
  return PCE_OK;
}

static inline void set_epi(TileArgs *a, const Epi &e) {
  a->bias = e.bias;
  a->res = e.res;
  a->act = e.act;
  a->slope = e.slope;
}

static inline bool epi_aligned(const Epi &e) { return aligned16(e.bias) && aligned16(e.res); }
