// The per-row sparse read as a masked sweep on the matrix cores, for many query rows (the
// reference's prefill: every row has its own list, read_kernel_tiled.py:30-156).
//
// The gather read fetches each row's list for itself: at 32k rows of 4612 keys that is 576 GB
// through the L2s (12.5 TB/s, 46 ms) for a cache of 134 MB. Rows that are neighbours list much
// of the same cache, so here 256 query columns (32-row blocks times the kv-head's query group)
// sweep the 64-key tiles any of their rows lists, and each row's list, as a bitmap over the
// cache rows, masks the softmax weights: the keys outside it weigh exactly zero.
//
//   row_bits_kernel     turns 32 rows' lists into bitmaps (bits [block][tile][row], 64 bits
//                       each) and flags, per block and tile, whether any row lists a key there,
//                       and the rows that list a key twice (a bitmap cannot count);
//   tile_finite_kernel  flags the 64-key tiles whose K or V holds a value that is not finite
//                       (a masked product would not be zero there);
//   rows_mfma_kernel    the sweep, 256 columns a workgroup;
//   rows_rest_kernel    the gather read of the rows the sweep leaves out: a duplicate in the
//                       list, a flagged tile among the workgroup's, or too few listed keys for
//                       the tiles they are spread over.
//
// A slab of query rows at a time, so that the bitmaps (and the list of units left) stay under kSlabBytes.
#include <math.h>

#include "lsa_abi_common.h"
#include "lsa_mfma_dev.h"
#include "lsa_read_dev.h"

using namespace lsa;

namespace {

constexpr int kTile = 64;              // keys of a tile
constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int NB = 4;                  // K and V tile buffers each
constexpr int kBlockRows = 32;         // query rows of a bitmap block (and columns of a wave)
constexpr int kMaxTiles = 4096;        // tiles of a cache (262144 rows)
constexpr int64_t kSlabBytes = 64 << 20;
constexpr int kXcds = 8;
constexpr int64_t kRestGrid = 16384;   // most workgroups that gather what is left (a multiple of kXcds)

struct RowsArgs {
  const void* q;
  const void* k;
  const void* v;
  void* out;
  const int32_t* ids;
  const int32_t* lengths;
  int64_t Tq, Tk;
  int64_t kv_sb, kv_st, kv_sh;
  int Hq, Hkv, W;
  int per_head;        // lists per (row, kv-head); 0: one list a row, shared by the heads
  int64_t u0;          // first row tile of the slab (row tile u = batch * n_rt + tile)
  int n_u;             // row tiles of the slab
  int n_rt;            // row tiles a batch row
  int rb;              // 32-row blocks of a row tile (8 / query group)
  int n_tile;          // 64-key tiles of the cache
  uint64_t* bits;      // [block][tile][32 rows]
  uint8_t* any;        // [block][tile]
  uint8_t* dup;        // [block][32 rows]
  int2* listed;        // [block]: keys its rows list (rows without duplicates), tiles they lie in
  int* left_n;         // [kXcds]: units (row, kv-head) of the slab left to the gather, by list
  int32_t* left;       // [kXcds][left_cap]: them, (row of the slab's row tiles) * kv-heads + kv-head
  int left_cap;
  const uint8_t* odd;  // [batch of K][kv-head][tile]: 1 a value that is not finite, or kUnseen
  float scale_log2;
  int empty_nan;
};

// The list index of query row t of batch b for kv-head g.
__device__ __forceinline__ int64_t list_of(const RowsArgs& a, int64_t b, int64_t t, int g) {
  const int64_t row = b * a.Tq + t;
  return a.per_head ? row * a.Hkv + g : row;
}

// ---------------------------------------------------------------- what is swept

// Listed keys a swept tile under which the gather reads a workgroup's rows faster: the sweep
// takes a CU ~2.6 us a tile (D 64: 1.9), the gather ~7.9 ns a listed key (D 64: 2.7, 3.8, 5.9
// and 12.3 ns at query groups 1, 2, 4 and 8).
template <int D, int GQ>
__device__ constexpr int sparse_keys() {
  return D == 128 ? 330 : (GQ == 1 ? 700 : (GQ == 2 ? 500 : (GQ == 4 ? 320 : 155)));
}

// Whether the sweep serves any row of the slab. The host chose it by sizes; the lists may still be
// short or scattered. A workgroup whose rows list enough keys a tile is swept, but the sweep takes
// at least its longest workgroup, so a slab of which only some are is read by the gather altogether where
// that is faster: 2048 rows of 0 to 4612 keys over 32768, 32 heads on 8, D 128, one workgroup in
// seven dense enough: 2.78 ms, 1.47 by this rule, 1.40 by the gather alone. Every workgroup of a
// kernel that asks finds the same; of more than 256 lists it looks at evenly spaced ones (an odd step,
// so that they are not all of one kv-head). Every thread calls both parts, a barrier between them.
enum Verdict { kGather, kSweep, kNothing };  // kNothing: no keys but duplicates' are listed
template <int D, int GQ, int THREADS>
struct SlabVerdict {
  static constexpr int RB = kWaves / GQ, WAVES = THREADS / LSA_WAVE;
  typedef float Red[WAVES][4];
  int keys = 0, tiles = 0, step;

  __device__ __forceinline__ explicit SlabVerdict(const RowsArgs& a) {
    const int units = a.n_u * (a.per_head ? a.Hkv : 1);
    step = units <= LSA_BLOCK ? 1 : (units / LSA_BLOCK + 1) | 1;
    const int64_t i = (int64_t)threadIdx.x * step;
    if (threadIdx.x < LSA_BLOCK && i < units) {
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const int2 x = a.listed[i * RB + r];
        keys += x.x;
        tiles = max(tiles, x.y);  // at least these
      }
    }
  }
  __device__ __forceinline__ void add_up(Red& red) const {
    const bool ok = (float)keys >= (float)tiles * (float)sparse_keys<D, GQ>();
    const float dense = wave_sum(ok ? (float)keys : 0.0f), thin = wave_sum(ok ? 0.0f : (float)keys);
    const float t = wave_sum(ok ? (float)tiles : 0.0f), longest = wave_max(ok ? (float)tiles : 0.0f);
    if (threadIdx.x % LSA_WAVE == 0) {
      float* x = red[threadIdx.x / LSA_WAVE];
      x[0] = dense; x[1] = thin; x[2] = t; x[3] = longest;
    }
  }
  __device__ __forceinline__ Verdict verdict(const RowsArgs& a, const Red& red) const {
    constexpr float SPARSE = (float)sparse_keys<D, GQ>(), CUS = 256.0f;
    float dense = 0.0f, thin = 0.0f, t = 0.0f, longest = 0.0f;
#pragma unroll
    for (int x = 0; x < WAVES; ++x) {
      dense += red[x][0]; thin += red[x][1]; t += red[x][2];
      longest = fmaxf(longest, red[x][3]);
    }
    if (dense + thin == 0.0f) return kNothing;
    const float all = (a.per_head ? 1.0f : (float)a.Hkv) * (float)step;  // workgroups a list seen
    const bool pays = 3.0f * thin <= dense || (dense > 0.0f && all * dense >= SPARSE * fmaxf(all * t, CUS * longest));
    return pays ? kSweep : kGather;
  }
};

// ---------------------------------------------------------------- tiles that are not finite

template <typename T>
__device__ __forceinline__ bool odd16(const uint4& x) {  // any of 8 elements infinite or NaN
  constexpr uint32_t E = __is_same(T, bf16_t) ? 0x7F80u : 0x7C00u;
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
  bool bad = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) bad |= (w[i] & E) == E || (w[i] & (E << 16)) == (E << 16);
  return bad;
}

// grid (tile, kv-head, batch of K). HBM-bound: one read of K and V, by the first slab that is swept.
constexpr uint8_t kUnseen = 2;  // a tile not looked at: no slab so far was swept
template <typename T, int D, int GQ>
__global__ __launch_bounds__(LSA_BLOCK) void tile_finite_kernel(RowsArgs a, uint8_t* odd) {
  constexpr int SEGS = D / 8, N = kTile * SEGS / LSA_BLOCK;
  __shared__ int bad[LSA_WAVES];
  using V = SlabVerdict<D, GQ, LSA_BLOCK>;
  __shared__ typename V::Red red;
  const int tile = blockIdx.x, g = blockIdx.y, b = blockIdx.z;
  uint8_t* state = odd + ((int64_t)b * gridDim.y + g) * a.n_tile + tile;
  if (a.u0 != 0 && *state != kUnseen) return;  // uniform
  const V slab(a);
  slab.add_up(red);
  __syncthreads();
  if (slab.verdict(a, red) != kSweep) {
    if (threadIdx.x == 0) *state = kUnseen;
    return;
  }
  const T* kb = (const T*)a.k + b * a.kv_sb + g * a.kv_sh;
  const T* vb = (const T*)a.v + b * a.kv_sb + g * a.kv_sh;
  uint4 x[2 * N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int i = n * LSA_BLOCK + threadIdx.x;
    const int64_t row = min((int64_t)tile * kTile + i / SEGS, a.Tk - 1);
    const int64_t off = row * a.kv_st + (i % SEGS) * 8;
    x[2 * n] = *(const uint4*)(kb + off);
    x[2 * n + 1] = *(const uint4*)(vb + off);
  }
  bool o = false;
#pragma unroll
  for (int n = 0; n < 2 * N; ++n) o |= odd16<T>(x[n]);
  const uint64_t m = __ballot(o);
  if ((threadIdx.x & 63) == 0) bad[threadIdx.x / 64] = m != 0;
  __syncthreads();
  if (threadIdx.x == 0) *state = (uint8_t)(bad[0] | bad[1] | bad[2] | bad[3]);
}

// ---------------------------------------------------------------- bitmaps

constexpr int kBitThreads = 1024;
constexpr int kSegKeys = 32768;                  // cache rows whose bits are in LDS at once
constexpr int kSegWords = kSegKeys / 32 + 2;     // dwords of a row in LDS (two of padding: conflict-free columns)

struct BitLds {
  uint32_t w[kBlockRows][kSegWords];
  int dup[kBlockRows], len[kBlockRows];
  int tiles;
};

// One 32-row block (grid: row tile of the slab, kv-head when lists are per head, block). Two
// rows a wave; a list is read once per kSegKeys cache rows. LDS-atomic bound.
__global__ __launch_bounds__(kBitThreads) void row_bits_kernel(RowsArgs a) {
  __shared__ BitLds sh;
  const int tid = threadIdx.x, lane = tid & 63, w = tid / 64;
  const int64_t blk = blockIdx.x;
  const int rb = (int)(blk % a.rb);
  const int64_t x = blk / a.rb;
  const int g = a.per_head ? (int)(x % a.Hkv) : 0;
  const int64_t u = a.u0 + (a.per_head ? x / a.Hkv : x);
  const int64_t b = u / a.n_rt;
  const int64_t t0 = ((u % a.n_rt) * a.rb + rb) * kBlockRows;
  if (tid < kBlockRows) sh.dup[tid] = sh.len[tid] = 0;
  if (tid == 0) sh.tiles = 0;
  if (blk == 0 && tid < kXcds) a.left_n[tid] = 0;
  for (int64_t k0 = 0; k0 < a.Tk; k0 += kSegKeys) {
    for (int i = tid; i < kBlockRows * kSegWords; i += kBitThreads) (&sh.w[0][0])[i] = 0;
    __syncthreads();
#pragma unroll
    for (int rr = 0; rr < 2; ++rr) {
      const int r = 2 * w + rr;
      const int64_t t = t0 + r;
      if (t < a.Tq) {
        const int64_t li = list_of(a, b, t, g);
        int n = a.lengths[li];
        n = n < 0 ? 0 : (n > a.W ? a.W : n);
        if (lane == 0) sh.len[r] = n;
        const int32_t* list = a.ids + li * a.W;
        bool twice = false;
        for (int j0 = 0; j0 < n; j0 += 8 * 64) {
          int32_t id[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) {  // unconditional (clamped): all in flight
            const int j = j0 + 64 * e + lane;
            const int32_t v = list[j < n ? j : n - 1];
            id[e] = j < n ? v : -1;
          }
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int64_t o = (int64_t)id[e] - k0;
            if (id[e] >= 0 && id[e] < a.Tk && o >= 0 && o < kSegKeys) {
              const uint32_t bit = 1u << (o & 31);
              twice |= (atomicOr(&sh.w[r][o >> 5], bit) & bit) != 0;
            }
          }
        }
        if (__any(twice) && lane == 0) sh.dup[r] = 1;
      }
    }
    __syncthreads();
    const int tiles = (int)min((int64_t)kSegKeys / kTile, (a.Tk - k0 + kTile - 1) / kTile);
    const int tile0 = (int)(k0 / kTile);
    int on = 0;
    for (int i = tid; i < tiles * kBlockRows; i += kBitThreads) {  // 64 lanes: two tiles of 32 rows
      const int tile = i / kBlockRows, r = i % kBlockRows;
      const uint64_t word = *(const uint64_t*)&sh.w[r][2 * tile];
      a.bits[(blk * a.n_tile + tile0 + tile) * kBlockRows + r] = word;
      const uint64_t m = __ballot(word != 0);
      if (r == 0) {
        const int any = ((lane ? m >> 32 : m) & 0xFFFFFFFFull) != 0;
        a.any[blk * a.n_tile + tile0 + tile] = (uint8_t)any;
        on += any;
      }
    }
    on = wave_sum(on);
    if (lane == 0) atomicAdd(&sh.tiles, on);
    __syncthreads();
  }
  if (tid < LSA_WAVE) {
    const bool dup = tid < kBlockRows && sh.dup[tid] != 0;
    if (tid < kBlockRows) a.dup[blk * kBlockRows + tid] = (uint8_t)dup;
    const int keys = wave_sum(tid < kBlockRows && !dup ? sh.len[tid] : 0);
    if (tid == 0) a.listed[blk] = make_int2(keys, sh.tiles);
  }
}

// ---------------------------------------------------------------- the sweep
//
// A workgroup is 8 waves of 32 query columns; K and V tiles go from memory straight to LDS
// (dma16), four buffers each. A wave's step is two phases: M, the last tile's P V products and
// this tile's scores (matrix cores, LDS reads and the loads ahead), and V, this tile's weights
// (vector unit). The waves form two groups of four, one wave of each on every SIMD, half a step
// apart (phase_barrier twice a step), so one group's matrix work runs beside the other's vector
// work instead of all waves wanting the same unit at once.
//
// What bounds it (counters, 32k rows of the reference's lists, 4288 keys a row on average, Hq 32,
// Hkv 8, D 128): a step of both groups takes ~5530 cycles of a SIMD against 3072 of matrix work.
// Matrix cores busy 55% of the cycles, vector unit 48% (~330 instructions a wave's V, 32 of them
// exponentials), both at once 17%; waves wait 18%, no LDS bank conflicts; the five loads of an M
// cost issue time wherever they stand. 10.7 ms against 46.2 for the gather; 403 M matrix
// instructions, 13.2 TFLOP with both halves of every swept pair: 1235 TFLOP/s.


template <int D>
struct alignas(1024) SweepLds {
  uint16_t k[NB][kTile * D];  // 16-byte segments of a row permuted by kseg
  uint16_t v[NB][kTile * D];  // by vseg
  uint64_t mask[kWaves][NB][kBlockRows];
  uint16_t act[kMaxTiles];    // the tiles swept, ascending
  int wsum[kWaves], wbad[kWaves];
  typename SlabVerdict<D, 1, kThreads>::Red red;
  int n_act, left0;
};

// Which LDS segment of row r holds its segment 0 (XOR): K rows are read 16 rows to a
// 16-lane group at one segment, V rows (transposing reads) 8 rows at 64 bytes each.
template <int D> __device__ __forceinline__ int kseg(int r) { return D == 128 ? r & 15 : (r >> 1) & 7; }
template <int D> __device__ __forceinline__ int vseg(int r) { return D == 128 ? (r & 3) << 2 : ((r >> 1) & 1) << 2; }

// 1024 (256) bytes from base + voff (a lane's) to LDS address `lds` + 16 (4) * lane, counted
// by vmcnt. Written as instructions, so that the compiler does not drain the counter before
// the LDS reads it cannot tell apart from these writes; the waits are wait_vm's.
__device__ __forceinline__ void dma16(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
__device__ __forceinline__ void dma4(uint32_t lds, const void* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(voff), "s"(base)
               : "memory", "m0");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// What a weight's 16-bit half leaves out, exact in fp32: x - pair.lo (lo) and x - pair.hi (hi),
// one dot product with (-1, 0) or (0, -1) each. The constants are kept opaque: as an inline
// operand this compiler gives the packed bf16 pair (-1, 0) the encoding of -1.0, which the
// instruction reads as the fp32 bits (0, -1).
template <typename T>
struct Rest {
  static constexpr uint32_t ONE = __is_same(T, bf16_t) ? 0xBF80u : 0xBC00u;
  uint32_t c_lo = ONE, c_hi = ONE << 16;
  __device__ __forceinline__ Rest() { asm("" : "+s"(c_lo), "+s"(c_hi)); }
  static __device__ __forceinline__ float dot(uint32_t pair, uint32_t c, float x) {
    if constexpr (__is_same(T, bf16_t))
      return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), __builtin_bit_cast(bf16x2_t, c), x, false);
    else
      return __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2_t, pair), __builtin_bit_cast(f16x2_t, c), x, false);
  }
  __device__ __forceinline__ float lo(uint32_t pair, float x) const { return dot(pair, c_lo, x); }
  __device__ __forceinline__ float hi(uint32_t pair, float x) const { return dot(pair, c_hi, x); }
};

// All ones where bit `bit` of w is set, else 0 (written as an instruction: with an AND it is two
// where the compiler's compare and select are three).
__device__ __forceinline__ uint32_t bit_mask(uint32_t w, int bit) {
  uint32_t m;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(m) : "v"(w), "ns"(bit));
  return m;
}

// A wave's 32 query columns: LDS addresses, the matrix products, and the weights of a tile. The
// gather read multiplies fp32 weights, so here a weight enters the matrix cores as the sum of
// two 16-bit halves (one alone would cost 2^-9 of it); the normaliser adds up the fp32 weights.
// bf16 halves are within 2^-17 of the weight at any size (fp32's exponents). fp16 halves are
// within 2^-23, but end at 2^-24: weights below that would count in the normaliser alone, and
// rows of one large and many small weights lost all the small ones (4612 keys of 2^-25 beside one of
// 1 read 0 for 1.4e-4). So fp16 weights are kept as high as their range allows: the largest is 2^BIAS
// when the reference moves and stays below 2^TOP, and the smallest step of a half is 2^-36 of it
// (8192 rows of 4612 keys, 32 heads on 8: D 128 827 -> 890 us, D 64 595 -> 660 to 690, the columns moved
// one by one). Measured against
// 64 bits, 4096 rows of up to 2308 keys: 2.1e-4 in fp16 and 1.7e-3 in bf16, as the gather.
template <typename T, int D>
struct Sweep {
  using M = Mfma<T>;
  using op_t = typename M::op_t;
  static constexpr int KS = D / 16, DB = D / 32, SEGS = D / 8, ROWB = 2 * D;
  static constexpr int KPI = 1024 / ROWB;            // keys a dma16 moves
  static constexpr int NI = kTile / (KPI * kWaves);  // dma16s a wave a tile, K and V each
  // log2 of a column's largest weight when its reference moves, and of the weight that moves it
  static constexpr bool HALF = !__is_same(T, bf16_t);
  static constexpr float BIAS = HALF ? 12.0f : 0.0f, TOP = HALF ? 15.0f : 8.0f;

  const lds_char *kl, *vl;
  uint32_t kbase, vbase;
  int jj;
  op_t qop[KS];
  f32x16_t o[DB], sc[2];
  uint32_t ph[2][8], pl[2][8];  // the weights' halves, two a word
  float m_run, l_run;  // the weights' reference, 2^BIAS below the largest score when it moved; their sum
  Rest<T> rest;

  __device__ __forceinline__ void init(const void* k_tiles, const void* v_tiles, const T* qrow) {
    const int lane = threadIdx.x & 63, hh = lane / 32, ln = lane % 32;
    kl = (const lds_char*)k_tiles;
    vl = (const lds_char*)v_tiles;
    jj = (lane % 16) / 4;
    kbase = (uint32_t)(ln * ROWB) + (uint32_t)((hh ^ kseg<D>(ln)) * 16);  // segment 2 s is this one's XOR 2 s
    vbase = (uint32_t)((4 * hh + jj) * ROWB + 32 * (ln / 16) + 8 * (lane % 4));
#pragma unroll
    for (int s = 0; s < KS; ++s) qop[s] = __builtin_bit_cast(op_t, *(const uint4*)(qrow + 16 * s + 8 * hh));
#pragma unroll
    for (int d = 0; d < DB; ++d) {
#pragma unroll
      for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    }
    m_run = kNegBig;
    l_run = 0.0f;
  }
  // Makes the compiler wait for the query rows here, ahead of a loop that counts loads itself.
  __device__ __forceinline__ void settle_queries() {
#pragma unroll
    for (int s = 0; s < KS; ++s) asm volatile("" ::"v"(qop[s]));
  }
  // Phase M as groups of matrix operations, each with its LDS operands in a buffer of `op`:
  // groups 0 .. 3 are O^T += V^T P^T of the last tile (16 keys each), groups 4 .. the scores of
  // the next (two 16-dim steps each). A group's operands are read while the two groups before
  // it compute, so the matrix cores do not wait for the LDS.
  static constexpr int NG = 4 + KS / 2;
  op_t op[3][4];
  __device__ __forceinline__ void load_group(int gi, int tile_v, int tile_k) {
    if (gi < 4) {  // V^T of keys 16 gi .. + 15: dims 32 d + ln at keys {4 hh .. + 3, 8 + 4 hh .. + 3}
      const lds_char* vt = vl + (tile_v & (NB - 1)) * (kTile * ROWB) + vbase;
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        const lds_char* vd = vt + (uint32_t)(64 * (D == 128 ? (d ^ jj) : (d ^ (jj >> 1))));
        const uint2 lo = v_column4(vd, 16 * gi * ROWB);
        const uint2 hi = v_column4(vd, (16 * gi + 8) * ROWB);
        op[gi % 3][d] = __builtin_bit_cast(op_t, make_uint4(lo.x, lo.y, hi.x, hi.y));
      }
    } else if (gi < NG) {  // K rows of both halves at dims 16 s .. + 15, s = 2 (gi - 4) and the next
      const lds_char* kt = kl + (tile_k & (NB - 1)) * (kTile * ROWB);
      typedef __attribute__((address_space(3))) const op_t lds_op;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        op[gi % 3][e] = *(lds_op*)(kt + (kbase ^ (uint32_t)(32 * (2 * (gi - 4) + e / 2))) + (e % 2) * 32 * ROWB);
    }
  }
  __device__ __forceinline__ void run_group(int gi) {
    if (gi < 4) {
      const int h = gi / 2, sp = gi % 2;
      const op_t pb = __builtin_bit_cast(op_t, make_uint4(ph[h][4 * sp], ph[h][4 * sp + 1], ph[h][4 * sp + 2], ph[h][4 * sp + 3]));
#pragma unroll
      for (int d = 0; d < DB; ++d) o[d] = M::run(op[gi % 3][d], pb, o[d]);
      const op_t qb = __builtin_bit_cast(op_t, make_uint4(pl[h][4 * sp], pl[h][4 * sp + 1], pl[h][4 * sp + 2], pl[h][4 * sp + 3]));
#pragma unroll
      for (int d = 0; d < DB; ++d) o[d] = M::run(op[gi % 3][d], qb, o[d]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int s = 2 * (gi - 4) + e / 2;
        sc[e % 2] = M::run(op[gi % 3][e], qop[s], sc[e % 2]);
      }
    }
  }
  // Tile i's scores, sc[h]: keys 32 h + 8 (r / 4) + 4 hh + r % 4 of column ln (groups 4 .. ;
  // the first two loaded by load_scores(i)).
  __device__ __forceinline__ void load_scores(int i) {
    load_group(4, i, i);
    load_group(5, i, i);
  }
  // hook(g), g = 0, 1, .., is called once a group (loads ahead: the matrix cores stay busy while
  // they issue).
  template <typename Hook>
  __device__ __forceinline__ void run_scores(int i, Hook&& hook) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r = 0; r < 16; ++r) sc[h][r] = 0.0f;
    }
#pragma unroll
    for (int gi = 4; gi < NG; ++gi) {
      load_group(gi + 2, i, i);
      hook(gi - 4);
      __builtin_amdgcn_sched_barrier(0);
      run_group(gi);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Tile i's P V product (its first groups loaded by load_pv(i)); loads tile i + 1's scores.
  __device__ __forceinline__ void load_pv(int i) {
    __builtin_amdgcn_sched_barrier(0);
    load_group(0, i, i);
    load_group(1, i, i);
  }
  template <typename Hook>
  __device__ __forceinline__ void run_pv(int i, Hook&& hook) {
#pragma unroll
    for (int gi = 0; gi < 4; ++gi) {
      load_group(gi + 2, i, i + 1);
      hook(gi);
      __builtin_amdgcn_sched_barrier(0);
      run_group(gi);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // p = exp2(s * scale - m) of the tile's keys, +0 where the key's bit of wd (this lane's keys of
  // each half: bit 8 (r / 4) + r % 4) is clear. Eight scores at a time, one operation of all of
  // them after the other: one wave a SIMD makes weights, so a chain of dependent instructions
  // would leave the unit idle between them (16k rows: 3.15 ms with four at a time, 2.98 with
  // eight, 3.00 with sixteen).
  // top: the largest upper halves of even and odd keys, as bits (weights are not negative, so the
  // bits order as they do); fp16.
  typedef unsigned short u16x2_t __attribute__((ext_vector_type(2)));
  __device__ __forceinline__ void weights(const uint32_t (&wd)[2], float scale_log2, float (&ls)[2], u16x2_t& top) {
    constexpr int E = 8;
    ls[0] = ls[1] = 0.0f;
    top = {0, 0};
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int r0 = 0; r0 < 16; r0 += E) {
        float p[E], q[E];
        uint32_t m[E];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < E; ++e) p[e] = fmaf(sc[h][r0 + e], scale_log2, -m_run);
#pragma unroll
        for (int e = 0; e < E; ++e) p[e] = fast_exp2(p[e]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < E; ++e) m[e] = bit_mask(wd[h], 8 * ((r0 + e) / 4) + e % 4);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < E; ++e) p[e] = __uint_as_float(__float_as_uint(p[e]) & m[e]);
        __builtin_amdgcn_sched_barrier(0);
        uint32_t* pair = &ph[h][r0 / 2];
#pragma unroll
        for (int e = 0; e < E; e += 2) pair[e / 2] = M::pack2(p[e], p[e + 1]);
#pragma unroll
        for (int e = 0; e < E; ++e) ls[e & 1] += p[e];
        if constexpr (HALF) {
#pragma unroll
          for (int e = 0; e < E / 2; ++e) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2_t, pair[e]));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < E; e += 2) {
          q[e] = rest.lo(pair[e / 2], p[e]);
          q[e + 1] = rest.hi(pair[e / 2], p[e + 1]);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int e = 0; e < E; e += 2) pl[h][(r0 + e) / 2] = M::pack2(q[e], q[e + 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  // The weights of a tile and its share of the normaliser. The reference moves lazily: the weights
  // are made against the current one, and only where a weight may have reached 2^TOP (bf16: a
  // lane's 32 weights together, which costs no instruction; fp16, whose range leaves no room for
  // that, the largest one) are the column maxima taken and, where a column's did, its state
  // rescaled and the weights made again. So every weight stays below 2^TOP, and most tiles take
  // no maximum. A column moves by its own weights alone: its row's bits do not depend on the
  // other rows of the wave (the same weights made twice are the same, and the others' tiles add zero);
  // with all columns moved together when one does, bf16 rows took up to 1% less, fp16 rows 4%.
  __device__ __forceinline__ void softmax(uint64_t mask, float scale_log2) {
    const int hh = (threadIdx.x & 63) / 32;
    const uint32_t wd[2] = {(uint32_t)mask >> (4 * hh), (uint32_t)(mask >> 32) >> (4 * hh)};
    float ls[2];
    u16x2_t top;
    weights(wd, scale_log2, ls, top);
    static_assert(TOP == (HALF ? 15.0f : 8.0f), "the test is against 2^TOP");
    const bool over = HALF ? max(top.x, top.y) >= 0x7800 : !(ls[0] + ls[1] < 256.0f);
    if (__builtin_expect(__any(over), 0)) {
      float mx = -INFINITY;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, (wd[h] >> (8 * (r / 4) + r % 4)) & 1u ? sc[h][r] : -INFINITY);
      }
      mx = over ? mx : -INFINITY;
      const float mt = fmaxf(mx, lane_xor(mx, 32)) * scale_log2;
      const bool moves = mt > m_run + TOP;
      if (__builtin_expect(__any(moves), 0)) {
        const float mn = moves ? mt - BIAS : m_run;
        const float alpha = fast_exp2(m_run - mn);
        m_run = mn;
        l_run *= alpha;
#pragma unroll
        for (int d = 0; d < DB; ++d) {
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
        }
        weights(wd, scale_log2, ls, top);
      }
    }
    l_run += ls[0] + ls[1];
  }
  // The normalised output row (lane: 4 dims of every 8 of its column), `empty` where no key weighed.
  __device__ __forceinline__ void store(T* op, float empty) const {
    const int hh = (threadIdx.x & 63) / 32;
    const float lt = l_run + lane_xor(l_run, 32);
    const float inv = 1.0f / lt;
    const bool none = !(lt > 0.0f);  // as the gather: a sum that is not a number counts as none
    if (op == nullptr) return;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        float x[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = none ? empty : o[d][4 * r4 + c] * inv;
        uint2 y;
        y.x = M::pack2(x[0], x[1]);
        y.y = M::pack2(x[2], x[3]);
        *(uint2*)(op + 32 * d + 8 * r4 + 4 * hh) = y;
      }
    }
  }
};

template <typename T, int D, int GQ>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void rows_mfma_kernel(RowsArgs a) {
  using S = Sweep<T, D>;
  constexpr int RB = kWaves / GQ;  // 32-row blocks of the workgroup
  constexpr int SEGS = S::SEGS, ROWB = S::ROWB, KPI = S::KPI, NI = S::NI;
  constexpr int PER = 2 * NI + 1;     // loads a wave issues a step
  constexpr int KLAST = S::NG - 4 - 1;  // the last score group
  __shared__ SweepLds<D> sh;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid / 64);
  const int ln = lane % 32;
  const int g = (int)(blockIdx.x % a.Hkv);
  const int ul = a.n_u - 1 - (int)(blockIdx.x / a.Hkv);  // later rows list more: longest first
  const int64_t u = a.u0 + ul;
  const int64_t b = u / a.n_rt;
  const int hl = w % GQ, rb = w / GQ;
  const int64_t t = ((u % a.n_rt) * RB + rb) * kBlockRows + ln;  // this lane's query row
  const int64_t blk0 = (a.per_head ? (int64_t)ul * a.Hkv + g : ul) * RB;
  const T* kb = (const T*)a.k + b * a.kv_sb + (int64_t)g * a.kv_sh;
  const T* vb = (const T*)a.v + b * a.kv_sb + (int64_t)g * a.kv_sh;

  // the tiles any of the workgroup's rows lists, and whether one of them is not finite
  {
    const SlabVerdict<D, GQ, kThreads> slab(a);  // its loads and the next are in flight until the tiles are listed
    int keys = 0;
#pragma unroll
    for (int r = 0; r < RB; ++r) keys += a.listed[blk0 + r].x;
    const bool dup = tid < RB * kBlockRows && a.dup[blk0 * kBlockRows + tid];
    bool not_finite = false;
    const uint8_t* odd = a.odd + ((a.kv_sb ? b : 0) * a.Hkv + g) * a.n_tile;
    int base = 0;
    for (int c0 = 0; c0 < a.n_tile; c0 += kThreads) {
      const int tile = c0 + tid;
      const int tc = tile < a.n_tile ? tile : 0;
      int on = 0;
#pragma unroll
      for (int r = 0; r < RB; ++r) on |= a.any[(blk0 + r) * a.n_tile + tc];
      const bool use = tile < a.n_tile && on;
      not_finite |= use && odd[tc];
      const uint64_t m = __ballot(use);
      if (lane == 0) sh.wsum[w] = __popcll(m);
      __syncthreads();
      int before = 0, total = 0;
#pragma unroll
      for (int x = 0; x < kWaves; ++x) {
        before += x < w ? sh.wsum[x] : 0;
        total += sh.wsum[x];
      }
      if (use) sh.act[base + before + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)tile;
      base += total;
      __syncthreads();
    }
    slab.add_up(sh.red);
    const bool wave_bad = __any(not_finite);
    if (lane == 0) sh.wbad[w] = wave_bad;
    __syncthreads();
    bool bad = false;
#pragma unroll
    for (int x = 0; x < kWaves; ++x) bad |= sh.wbad[x] != 0;
    const bool all = bad || keys < base * sparse_keys<D, GQ>() || slab.verdict(a, sh.red) == kGather;  // uniform
    if (tid == 0) sh.n_act = all ? -1 : base;
    // the rows the gather reads: all, or the ones that list a key twice
    const int64_t tr = (u % a.n_rt) * RB * kBlockRows + tid;
    const bool left = tid < RB * kBlockRows && tr < a.Tq && (all || dup);
    const uint64_t m = __ballot(left);
    if (lane == 0) sh.wsum[w] = __popcll(m);
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int x = 0; x < kWaves; ++x) {
      before += x < w ? sh.wsum[x] : 0;
      total += sh.wsum[x];
    }
    if (total > 0) {  // uniform
      const int c = (int)(((int64_t)ul * a.Hkv + g) % kXcds);
      if (tid == 0) sh.left0 = atomicAdd(&a.left_n[c], total);
      __syncthreads();
      const int at = sh.left0 + before + __popcll(m & ((1ull << lane) - 1));
      if (left) a.left[(int64_t)c * a.left_cap + at] = (int32_t)(((int64_t)ul * RB * kBlockRows + tid) * a.Hkv + g);
    }
  }
  const int n = __builtin_amdgcn_readfirstlane(sh.n_act);
  if (n < 0) return;  // uniform

  const bool row_ok = t < a.Tq;
  const int64_t qrow = ((b * a.Tq + (row_ok ? t : 0)) * a.Hq + (int64_t)g * GQ + hl) * D;
  S sw;
  sw.init(&sh.k[0][0], &sh.v[0][0], (const T*)a.q + qrow);

  if (n > 0) {
    // loads: wave w moves keys [8 w, 8 w + 8) of a K and a V tile, and its own 32 masks
    const uint32_t st = (uint32_t)a.kv_st * 2u;
    uint32_t kvo[NI], vvo[NI];
    auto offsets = [&](int limit) {  // rows at or past `limit` read the row before it
#pragma unroll
      for (int x = 0; x < NI; ++x) {
        const int r = (w * NI + x) * KPI + lane / SEGS;
        const uint32_t row = (uint32_t)min(r, limit - 1) * st;
        kvo[x] = row + (uint32_t)(((lane % SEGS) ^ kseg<D>(r)) * 16);
        vvo[x] = row + (uint32_t)(((lane % SEGS) ^ vseg<D>(r)) * 16);
      }
    };
    const int last_rows = (int)(a.Tk - (int64_t)(a.n_tile - 1) * kTile);  // rows of the cache's last tile
    const uint32_t k_lds = (uint32_t)(uintptr_t)(lds_char*)&sh.k[0][0];
    const uint32_t v_lds = (uint32_t)(uintptr_t)(lds_char*)&sh.v[0][0];
    const uint32_t m_lds = (uint32_t)(uintptr_t)(lds_char*)&sh.mask[w][0][0];
    const uint64_t* bits = a.bits + (blk0 + rb) * a.n_tile * kBlockRows;
    // Part x (of NI) of this wave's share of tile i's K or V rows, its i-th tile being `tile`.
    auto move = [&](uint32_t lds, const T* src, int i, int tile, int x, const uint32_t (&vo)[NI]) {
      dma16(lds + (uint32_t)(i & (NB - 1)) * (kTile * ROWB) + (uint32_t)(w * NI + x) * 1024u,
            src + (int64_t)tile * kTile * a.kv_st, vo[x]);
    };
    auto load = [&](bool values, int i, int tile, int x) {
      const bool part = tile == a.n_tile - 1 && last_rows < kTile;  // uniform
      if (part) offsets(last_rows);
      if (values) move(v_lds, vb, i, tile, x, vvo);
      else move(k_lds, kb, i, tile, x, kvo);
      if (part) offsets(kTile);
    };
    auto load_mask = [&](int i, int tile) {
      dma4(m_lds + (uint32_t)(i & (NB - 1)) * 256u, bits + (int64_t)tile * kBlockRows, (uint32_t)lane * 4u);
    };
    auto tile_at = [&](int i) { return __builtin_amdgcn_readfirstlane((int)sh.act[i < n ? i : n - 1]); };

    auto mask_of = [&](int i) {
      typedef __attribute__((address_space(3))) const uint64_t lds_u8;
      return *(lds_u8*)((const lds_char*)&sh.mask[w][0][0] + (i & (NB - 1)) * 256 + ln * 8);
    };

    // Two groups of four waves, one wave of each on every SIMD, half a step apart: while one
    // group's waves feed the matrix cores (the last tile's P V, this tile's scores), the other
    // group's make weights. Group 0 runs M(i) in half-step 2 i and V(i) in 2 i + 1, group 1 one
    // half-step later, so K(i) is read in half-steps 2 i, 2 i + 1 and V(i) in 2 i + 2, 2 i + 3.
    // In M(i) a wave loads K(i + 3) into the buffer of K(i - 1) (last read in half-step 2 i - 1),
    // V(i + 2) into that of V(i - 2) (likewise) and its masks of tile i + 3. What a phase reads
    // was loaded two or more of every wave's M phases before the barrier ahead of it: V(i) is read
    // from the end of V(i) on (half-step 2 i + 1 at the earliest) and K(i + 1) from half-step
    // 2 i + 2 on, both loaded in M(i - 2). So at the end of M(i) the loads of M(i) and M(i - 1) may
    // be outstanding, at the end of V(i) those of M(i).
    offsets(kTile);
    int t2 = 0, t3;
    for (int j = 0; j < 3; ++j) {
      t2 = tile_at(j);
#pragma unroll
      for (int x = 0; x < NI; ++x) {
        load(false, j, t2, x);
        if (j < 2) load(true, j, t2, x);
      }
      load_mask(j, t2);
    }
    t3 = tile_at(3);
    sw.settle_queries();
    wait_vm<0>();
#pragma unroll
    for (int x = 0; x < NI; ++x) load(false, 3, t3, x);  // M(0)'s
    phase_barrier();
    const bool late = w >= kWaves / 2;
    if (late) phase_barrier();
    sw.load_scores(0);
    for (int i = 0;;) {
      sw.run_scores(i, [&](int x) {
        if (x < NI) load(true, i + 2, t2, x);
        if (x == KLAST) load_mask(i + 3, t3);
      });
      const uint64_t mask = mask_of(i);
      wait_vm<2 * PER>();
      phase_barrier();
      t2 = t3;
      t3 = tile_at(i + 4);
      sw.softmax(mask, a.scale_log2);
      sw.load_pv(i);
      wait_vm<PER>();
      phase_barrier();
      sw.run_pv(i, [&](int x) {
        if (x < NI) load(false, i + 4, t3, x);
      });
      if (++i == n) break;
    }
    if (!late) phase_barrier();
    wait_vm<0>();  // no load may land after the workgroup's LDS is given back
  }

  sw.store(row_ok ? (T*)a.out + qrow : nullptr, a.empty_nan ? NAN : 0.0f);
}

// ---------------------------------------------------------------- the rows left to the gather

// The units (row, kv-head) the sweep left, from their lists, so that wherever they lie they spread over
// the chip; up to kRestGrid of them a workgroup each, as their lengths may differ. The rows of a
// (row tile, kv-head), which list much the same, are in one list, and a list goes to the workgroups of one
// XCD (consecutive ones are on different XCDs), whose L2 then serves them all; where the lists
// differ much in length, the workgroups take them one after the other instead. All units left, 32
// heads on 8, D 128 (us; a workgroup of the gather alone for each unit / this call, with the bitmaps and a sweep
// that finds nothing to do / before, when a workgroup read all it found in 256 neighbouring
// units): 1024 rows of 1024 keys, one twice 301 / 329 / 3550, of 16 keys of 1024 60 / 79 / 900; 2048
// rows of 0 to 4612 keys of 32768 1400 / 1465 / 8970. Taking units one by one from a counter costs
// ~26 ns each across the XCDs (1024 rows of 16 keys: 650 us). 2048 workgroups: the last figure is
// 1800, but with nothing left they are 1.5 us less.
template <typename T, int D, int GQ>
__global__ __launch_bounds__(LSA_BLOCK) __attribute__((amdgpu_waves_per_eu(GQ == 8 ? 2 : 3))) void rows_rest_kernel(
    RowsArgs a) {
  using S = ReadShape<T, D, GQ>;
  constexpr int RT = kWaves / GQ * kBlockRows;
  __shared__ ReadLds<D, GQ, kMaxSplits> sh;
  const int lp = (threadIdx.x & 63) % S::LPT;
  int most = 0, total = 0;
#pragma unroll
  for (int c = 0; c < kXcds; ++c) {
    most = max(most, a.left_n[c]);
    total += a.left_n[c];
  }
  const bool even = most <= 2 * (total / kXcds);
  const int end = even ? most * kXcds : total;
  for (int i = blockIdx.x; i < end; i += gridDim.x) {  // uniform
    int c = even ? i % kXcds : 0, p = even ? i / kXcds : i;
    if (even) {
      if (p >= a.left_n[c]) continue;
    } else {
      while (p >= a.left_n[c]) p -= a.left_n[c++];
    }
    const uint32_t j = (uint32_t)__builtin_amdgcn_readfirstlane(a.left[(int64_t)c * a.left_cap + p]);
    const int g = (int)(j % (uint32_t)a.Hkv);
    const uint32_t x = j / (uint32_t)a.Hkv;
    const int64_t u = a.u0 + x / RT;
    const int64_t b = u / a.n_rt, t = (u % a.n_rt) * RT + x % RT;
    const int64_t li = list_of(a, b, t, g);
    int n = a.lengths[li];
    n = n < 0 ? 0 : (n > a.W ? a.W : n);
    T* outp = (T*)a.out + ((b * a.Tq + t) * a.Hq + (int64_t)g * GQ) * D;
    if (n == 0) {
      for (int o = threadIdx.x; o < GQ * D; o += LSA_BLOCK) store_out<T>(outp + o, a.empty_nan ? NAN : 0.0f);
      continue;
    }
    const int32_t* list = a.ids + li * a.W;
    const T* kb = (const T*)a.k + b * a.kv_sb + g * a.kv_sh + lp * S::VEC;
    const T* vb = (const T*)a.v + b * a.kv_sb + g * a.kv_sh + lp * S::VEC;
    AttnState<T, D, GQ> st;
    attend_span<T, D, GQ>((const T*)a.q + (outp - (T*)a.out), kb, vb, a.kv_st, a.Tk, 0, n,
                          [&](int s) {
                            const int32_t id = list[s < n ? s : n - 1];
                            return s < n ? id : -1;
                          },
                          a.scale_log2, st);
    __syncthreads();  // the last unit is done with sh
    finish_span<T, D, GQ, kMaxSplits, true>(sh, st, true, outp, nullptr, a.empty_nan);
  }
}

// ---------------------------------------------------------------- host

struct Layout {
  int gq, rb;
  int64_t n_rt, n_tile, u_total, slab_u, blocks;
  int64_t left_cap;
  size_t bits, any, dup, listed, left_n, left, odd, total;
};

Layout layout_of(int64_t B, int64_t Tq, int64_t Tk, int32_t Hq, int32_t Hkv, int per_head) {
  Layout l;
  l.gq = Hq / Hkv;
  l.rb = kWaves / l.gq;
  l.n_rt = (Tq + l.rb * kBlockRows - 1) / (l.rb * kBlockRows);
  l.n_tile = (Tk + kTile - 1) / kTile;
  l.u_total = B * l.n_rt;
  const int64_t per_u = (int64_t)l.rb * (per_head ? Hkv : 1);  // blocks a row tile
  const int64_t units_u = (int64_t)l.rb * kBlockRows * Hkv;     // (row, kv-head) units a row tile
  const int64_t most = per_u * l.n_tile * kBlockRows * 8;       // bytes of bitmaps a row tile
  const int64_t fit = kSlabBytes / (most > units_u * 4 ? most : units_u * 4);
  l.slab_u = fit < 1 ? 1 : (fit < l.u_total ? fit : l.u_total);
  l.blocks = l.slab_u * per_u;
  auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
  l.bits = 0;
  l.any = l.bits + up((size_t)l.blocks * l.n_tile * kBlockRows * 8);
  l.dup = l.any + up((size_t)l.blocks * l.n_tile);
  l.listed = l.dup + up((size_t)l.blocks * kBlockRows);
  l.left_n = l.listed + up((size_t)l.blocks * sizeof(int2));
  l.left = l.left_n + up(kXcds * sizeof(int));
  l.left_cap = (l.slab_u * Hkv + kXcds - 1) / kXcds * l.rb * kBlockRows;
  l.odd = l.left + up((size_t)(kXcds * l.left_cap) * sizeof(int32_t));
  l.total = l.odd + up((size_t)B * Hkv * l.n_tile);
  return l;
}

template <typename T, int D, int GQ>
void launch_slab(const RowsArgs& a, const Layout& l, int64_t kv_batches, uint8_t* odd, hipStream_t s) {
  const int64_t per_u = (int64_t)l.rb * (a.per_head ? a.Hkv : 1);
  row_bits_kernel<<<dim3((unsigned)(a.n_u * per_u)), kBitThreads, 0, s>>>(a);
  const dim3 tiles((unsigned)l.n_tile, (unsigned)a.Hkv, (unsigned)kv_batches);
  tile_finite_kernel<T, D, GQ><<<tiles, LSA_BLOCK, 0, s>>>(a, odd);
  rows_mfma_kernel<T, D, GQ><<<dim3((unsigned)(a.n_u * a.Hkv)), kThreads, 0, s>>>(a);
  const int64_t units = (int64_t)a.n_u * l.rb * kBlockRows * a.Hkv;
  rows_rest_kernel<T, D, GQ><<<dim3((unsigned)(units < kRestGrid ? units : kRestGrid)), LSA_BLOCK, 0, s>>>(a);
}

template <typename T, int D>
void launch_rows(RowsArgs a, const Layout& l, int64_t kv_batches, uint8_t* odd, hipStream_t s) {
  for (int64_t u = 0; u < l.u_total; u += l.slab_u) {
    a.u0 = u;
    a.n_u = (int)(l.u_total - u < l.slab_u ? l.u_total - u : l.slab_u);
    switch (l.gq) {
      case 1: launch_slab<T, D, 1>(a, l, kv_batches, odd, s); break;
      case 2: launch_slab<T, D, 2>(a, l, kv_batches, odd, s); break;
      case 4: launch_slab<T, D, 4>(a, l, kv_batches, odd, s); break;
      default: launch_slab<T, D, 8>(a, l, kv_batches, odd, s); break;
    }
  }
}

bool rows_fit(int dtype, int64_t B, int64_t Tq, int64_t Tk, int32_t Hq, int32_t Hkv, int32_t D, int32_t W) {
  if (!(dtype == LSA_BF16 || dtype == LSA_F16) || !(D == 64 || D == 128)) return false;
  if (B < 1 || Tq < 1 || Tk < 1 || Hkv < 1 || Hq < Hkv || Hq % Hkv || W < 1) return false;
  const int gq = Hq / Hkv;
  if (!(gq == 1 || gq == 2 || gq == 4 || gq == 8)) return false;
  return Tk <= (int64_t)kMaxTiles * kTile && B <= 65535 && Hkv <= 65535;
}

}  // namespace

extern "C" size_t lsa_read_rows_scratch_bytes(int dtype, int64_t B, int64_t Tq, int64_t Tk, int32_t Hq, int32_t Hkv,
                                              int32_t D, int32_t W, int ids_per_head) {
  if (!rows_fit(dtype, B, Tq, Tk, Hq, Hkv, D, W)) return 0;
  return layout_of(B, Tq, Tk, Hq, Hkv, ids_per_head ? 1 : 0).total;
}

extern "C" int lsa_read_rows(const void* q, const void* k, const void* v, int dtype, int64_t B, int64_t Tq, int64_t Tk,
                             int32_t Hq, int32_t Hkv, int32_t D, int64_t kv_batch_stride, int64_t kv_token_stride,
                             int64_t kv_head_stride, const int32_t* ids, const int32_t* lengths, int32_t W,
                             int ids_per_head, float scale, int empty_nan, void* scratch, size_t scratch_bytes,
                             void* out, void* stream) {
  LSA_REQUIRE(q && k && v && ids && lengths && out, LSA_ERR_NULL, "lsa_read_rows: NULL pointer");
  LSA_REQUIRE(rows_fit(dtype, B, Tq, Tk, Hq, Hkv, D, W), LSA_ERR_SHAPE, "lsa_read_rows: shape not served");
  LSA_REQUIRE(scale > 0.0f && isfinite(scale), LSA_ERR_SHAPE, "lsa_read_rows: scale must be positive and finite");
  const uintptr_t mis = ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) & 15;
  LSA_REQUIRE(mis == 0, LSA_ERR_ALIGN, "lsa_read_rows: q/k/v/out must be 16-byte aligned");
  LSA_REQUIRE(kv_batch_stride >= 0 && kv_token_stride >= D && kv_head_stride >= D && kv_token_stride < (1 << 24),
              LSA_ERR_SHAPE, "lsa_read_rows: K/V strides");
  LSA_REQUIRE(((kv_batch_stride | kv_token_stride | kv_head_stride) * 2) % 16 == 0, LSA_ERR_ALIGN,
              "lsa_read_rows: K/V strides must keep rows 16-byte aligned");
  const Layout l = layout_of(B, Tq, Tk, Hq, Hkv, ids_per_head ? 1 : 0);
  LSA_REQUIRE(scratch && ((uintptr_t)scratch & 255) == 0 && scratch_bytes >= l.total, LSA_ERR_WORKSPACE,
              "lsa_read_rows: scratch %zu < %zu bytes", scratch_bytes, l.total);
  LSA_REQUIRE(l.blocks <= 0x7FFFFFFF && l.slab_u * l.rb * kBlockRows * Hkv <= 0x7FFFFFFF, LSA_ERR_SHAPE,
              "lsa_read_rows: too many rows");
  RowsArgs a;
  char* ws = (char*)scratch;
  a.q = q; a.k = k; a.v = v; a.out = out; a.ids = ids; a.lengths = lengths;
  a.Tq = Tq; a.Tk = Tk; a.kv_sb = kv_batch_stride; a.kv_st = kv_token_stride; a.kv_sh = kv_head_stride;
  a.Hq = Hq; a.Hkv = Hkv; a.W = W; a.per_head = ids_per_head ? 1 : 0;
  a.u0 = 0; a.n_u = 0; a.n_rt = (int)l.n_rt; a.rb = l.rb; a.n_tile = (int)l.n_tile;
  a.bits = (uint64_t*)(ws + l.bits); a.any = (uint8_t*)(ws + l.any); a.dup = (uint8_t*)(ws + l.dup);
  a.listed = (int2*)(ws + l.listed); a.left_n = (int*)(ws + l.left_n); a.left = (int32_t*)(ws + l.left);
  a.left_cap = (int)l.left_cap; a.odd = (const uint8_t*)(ws + l.odd);
  a.scale_log2 = scale * kLog2e; a.empty_nan = empty_nan ? 1 : 0;
  const int64_t kv_batches = kv_batch_stride ? B : 1;
  uint8_t* odd = (uint8_t*)(ws + l.odd);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == LSA_BF16) {
    if (D == 64) launch_rows<bf16_t, 64>(a, l, kv_batches, odd, s);
    else launch_rows<bf16_t, 128>(a, l, kv_batches, odd, s);
  } else {
    if (D == 64) launch_rows<_Float16, 64>(a, l, kv_batches, odd, s);
    else launch_rows<_Float16, 128>(a, l, kv_batches, odd, s);
  }
  LSA_LAUNCHED("lsa_read_rows");
  return LSA_OK;
}
