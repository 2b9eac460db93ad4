// Bucket-table build on the GPU: contiguous Ward-style segments from the keys.
//
// The index build that precedes the select+read path (the reference builds its bucket tables
// with build_buckets_gpu, pipeline.py:71-116: pooled keys merged by the Ward cost into
// buckets, centroids from the member keys). Here the buckets stay contiguous - every
// bucket is a run of consecutive positions, so a table is its span ends and the decode
// expands a pick from them - and merges adjacent segments only:
//
//   1. pools: the keys of one table (one (batch, kv-head)) cut into pools of `pool`
//      consecutive positions (the last one shorter); a pool's key sum in fp64, positions in
//      order;
//   2. merges: while more than `target` segments remain, the adjacent pair (a, b) with the
//      smallest Ward cost  n_a n_b / (n_a + n_b) * |s_a / n_a - s_b / n_b|^2  merges into
//      one (ties to the leftmost pair; pairs over `max_size` positions never merge);
//   3. out: the segment start positions, [target + 1] per table (the last entry = T).
//
// Every cost is computed in one fixed order of fp64 operations, with no contraction into
// fused multiply-adds: the squared differences d = 0..D-1 fold into 64 partials
// (partial l = sum over k of sq[l + 64 k], k ascending), then halve 32, 16, .., 1 (partial l
// += partial l + h). Costs, sizes and the segment links of a table sit in LDS, the fp64 sums in
// a global scratch buffer.
#include <float.h>
#include <math.h>

#include "lsa_abi_common.h"
#include "lsa_device.h"
#include "lsa_select_dev.h"

using namespace lsa;

namespace {

constexpr int kPoolThreads = 256;
constexpr int kMergeThreads = 1024;
constexpr int kMaxPools = 4096;  // LDS-resident segment state per table, 64 groups of costs
constexpr int kSmallPools = 512;
constexpr int kRecips = 2048;  // reciprocals of 0 .. in LDS; larger counts are divided

// fp64 key sum of every (table, pool, dim): positions of the pool in order.
template <typename KT>
__global__ __launch_bounds__(kPoolThreads) void pool_sums_kernel(const KT* keys, int64_t T, int kv_heads, int D,
                                                                 int64_t kv_sb, int64_t kv_st, int64_t kv_sh,
                                                                 int pool, int npool, double* sums) {
#pragma clang fp contract(off)
  const int64_t per_table = (int64_t)npool * D;
  const int64_t x = (int64_t)blockIdx.x * kPoolThreads + threadIdx.x;
  const int64_t table = blockIdx.y;
  if (x >= per_table) return;
  const int p = (int)(x / D), d = (int)(x % D);
  const KT* kb = keys + (table / kv_heads) * kv_sb + (table % kv_heads) * kv_sh;
  const int64_t t0 = (int64_t)p * pool;
  const int64_t t1 = t0 + pool < T ? t0 + pool : T;
  double s = 0.0;
  for (int64_t t = t0; t < t1; ++t) s = s + (double)elem<KT>::load(kb, t * kv_st + d);
  sums[table * per_table + x] = s;
}

// Ward cost of adjacent segments a < b (sums at sa / sb, sizes na / nb) on one wave; every
// lane returns it. +inf when the merged segment would exceed max_size.
__device__ double pair_cost(const double* sa, const double* sb, int na, int nb, int D, int max_size) {
#pragma clang fp contract(off)
  if (na + nb > max_size) return INFINITY;
  const int lane = threadIdx.x & (LSA_WAVE - 1);
  const double fa = (double)na, fb = (double)nb;
  double part = 0.0;
  for (int d = lane; d < D; d += LSA_WAVE) {
    const double diff = sa[d] / fa - sb[d] / fb;
    const double sq = diff * diff;
    part = part + sq;
  }
#pragma unroll
  for (int h = LSA_WAVE / 2; h >= 1; h >>= 1) {
    const double other = __shfl_down(part, h, LSA_WAVE);
    if (lane < h) part = part + other;
  }
  const double total = __shfl(part, 0, LSA_WAVE);
  const double w = (fa * fb) / (fa + fb);
  return w * total;
}

// ---------------------------------------------------------------- the merge loop
//
// The loop is one dependent chain (a merge decides the next), so it runs on one wave with no
// barrier, and what counts is the chain's length. Costs sit in LDS as their bits (a cost is not
// negative, so the bits order as the values; NaN sorts past infinity), in groups of 64
// positions whose minimum and its place lane g of the wave holds: the next pair is one wave
// reduction over the lanes, and a merge renews only the groups it touched (one or two). Every
// cross-lane step is DPP or a row swap. A merge reads the sums of the four segments around it in
// one round trip; the quotients s / n need no division (quotient), the two weights
// n_a n_b / (n_a + n_b) and the new segment's reciprocal are divided while the sums are in flight.
//
// Latency-bound: 32k positions x 8 tables (1536 merges of 2048 pools each, D 128): 1.1 us a merge
// against 3.45 for a workgroup of 16 waves with three barriers a merge; the build 5.5 -> 1.8 ms.

constexpr uint32_t kInfHi = 0x7FF00000u;  // the high word of +infinity

// A live segment, named by its first pool: its neighbours (-1: none) and positions (0: merged into
// an earlier one).
struct alignas(8) Seg {
  int16_t prv, nxt;
  int32_t size;
};

// RN(x / n) for n a positive integer and y = RN(1 / n): x y is within 1.5 ulp, the first
// correction makes it faithful, and by Markstein's theorem (faithful quotient, correctly rounded
// reciprocal, exact remainder by FMA) the second rounds correctly. Not for x infinite (NaN there:
// the costs it enters are inadmissible either way).
__device__ __forceinline__ double quotient(double x, double n, double y) {
  double q = x * y;
  q = fma(fma(-q, n, x), y, q);
  return fma(fma(-q, n, x), y, q);
}

// The halving folds of two sets of 64 partials at once (partial l += partial l + h, h = 32 .. 1):
// a's total in lanes 0 .. 31, b's in lanes 32 .. 63.
template <int CTRL>
__device__ __forceinline__ double add_dpp(double x) {
  const uint64_t u = __builtin_bit_cast(uint64_t, x);
  const uint64_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)u, CTRL, 0xF, 0xF, true);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(u >> 32), CTRL, 0xF, 0xF, true);
  return x + __builtin_bit_cast(double, hi << 32 | lo);
}
__device__ __forceinline__ double fold2(double a, double b) {
  const auto word = [](double x, int k) { return __uint_as_float((uint32_t)(__builtin_bit_cast(uint64_t, x) >> (32 * k))); };
  const auto whole = [](float lo, float hi) {
    return __builtin_bit_cast(double, (uint64_t)__float_as_uint(hi) << 32 | __float_as_uint(lo));
  };
  float al = word(a, 0), ah = word(a, 1), bl = word(b, 0), bh = word(b, 1);
  row_swap32(al, bl);  // [a lower, b lower], [a upper, b upper]
  row_swap32(ah, bh);
  double x = whole(al, ah) + whole(bl, bh);
  float xl = word(x, 0), xh = word(x, 1), yl = xl, yh = xh;
  row_swap16(xl, yl);  // rows [0, 0, 2, 2], [1, 1, 3, 3]
  row_swap16(xh, yh);
  x = whole(xl, xh) + whole(yl, yh);
  x = add_dpp<0x128>(x);     // row_ror:8
  x = add_dpp<0x124>(x);     // row_ror:4, lanes now repeating every 8
  x = add_dpp<kDppXor2>(x);
  return add_dpp<kDppXor1>(x);
}

__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  return (uint32_t)wave_reduce_bits((int)x, -1, [](int p, int q) { return (uint32_t)p < (uint32_t)q ? p : q; });
}

// The lowest lane that holds the wave's smallest k.
__device__ __forceinline__ int lane_of_min(uint64_t k, uint32_t* min_hi) {
  const uint32_t hi = (uint32_t)(k >> 32), mh = wave_min_u32(hi);
  uint64_t at = __ballot(hi == mh);
  if (at & (at - 1)) {  // uniform: equal high words
    const uint32_t lo = hi == mh ? (uint32_t)k : 0xFFFFFFFFu;
    at &= __ballot(lo == wave_min_u32(lo));
  }
  *min_hi = mh;
  return __ffsll((long long)at) - 1;
}

// The greedy adjacent merge of one table: the workgroup's waves make the first costs, wave 0
// merges. KD: dims a lane holds (D <= 64 KD); 0: any D, walked 64 at a time. MAXP: pools the LDS
// holds (80 KiB at kMaxPools; small tables leave room for more of them on a CU).
template <int KD, int MAXP>
__global__ __launch_bounds__(kMergeThreads) void ward_merge_kernel(double* sums, int64_t T, int D, int pool,
                                                                   int npool, int target, int max_size,
                                                                   int32_t* starts, int32_t* status,
                                                                   int32_t* failed_any) {
#pragma clang fp contract(off)
  __shared__ Seg seg[MAXP];
  __shared__ uint64_t cost[MAXP];
  __shared__ double recip[kRecips];  // RN(1 / n)
  const int tid = threadIdx.x, lane = tid & (LSA_WAVE - 1), w = tid / LSA_WAVE, waves = blockDim.x / LSA_WAVE;
  const int64_t table = blockIdx.x;
  const int groups = (npool + LSA_WAVE - 1) / LSA_WAVE;
  double* ts = sums + table * (int64_t)npool * D;
  for (int i = tid; i < npool; i += blockDim.x) {
    const int64_t t0 = (int64_t)i * pool;
    Seg x;
    x.size = (int)((t0 + pool < T ? t0 + pool : T) - t0);
    x.nxt = (int16_t)(i + 1 < npool ? i + 1 : -1);
    x.prv = (int16_t)(i - 1);
    seg[i] = x;
  }
  for (int i = tid; i < kRecips; i += blockDim.x) recip[i] = 1.0 / (double)(i > 0 ? i : 1);
  __syncthreads();
  for (int i = w; i < groups * LSA_WAVE; i += waves) {
    const double c = i + 1 < npool ? pair_cost(ts + (int64_t)i * D, ts + (int64_t)(i + 1) * D, seg[i].size,
                                               seg[i + 1].size, D, max_size)
                                   : INFINITY;
    if (lane == 0) cost[i] = __builtin_bit_cast(uint64_t, c);
  }
  __syncthreads();
  if (w != 0) return;

  uint64_t gkey = (uint64_t)kInfHi << 32;  // lane g: the smallest cost of group g and its place
  int gidx = 0;
  auto set_group = [&](int g, uint64_t k) {  // k: the group's costs, one a lane
    uint32_t mh;
    const int l = lane_of_min(k, &mh);
    const uint32_t ml = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, l);
    if (lane == g) {
      gkey = (uint64_t)mh << 32 | ml;
      gidx = g * LSA_WAVE + l;
    }
  };
  for (int g = 0; g < groups; ++g) set_group(g, cost[g * LSA_WAVE + lane]);

  int failed = 0;
  for (int alive = npool; alive > target; --alive) {
    uint32_t mh;
    const int l = lane_of_min(gkey, &mh);
    if (mh >= kInfHi) {  // no pair can merge under max_size
      failed = 1;
      break;
    }
    const int i = __builtin_amdgcn_readlane(gidx, l);
    const Seg si = seg[i];
    const int a = __builtin_amdgcn_readfirstlane((int)si.prv), j = __builtin_amdgcn_readfirstlane((int)si.nxt);
    const Seg sj = seg[j], sa = seg[a >= 0 ? a : i];
    const int b = __builtin_amdgcn_readfirstlane((int)sj.nxt);
    const Seg sb = seg[b >= 0 ? b : i];
    const int g = i / LSA_WAVE;
    const uint64_t kg = cost[g * LSA_WAVE + lane];  // the group's costs, renewed below
    const double* pi = ts + (int64_t)i * D;
    const double* pj = ts + (int64_t)j * D;
    const double* pa = ts + (int64_t)(a >= 0 ? a : i) * D;
    const double* pb = ts + (int64_t)(b >= 0 ? b : i) * D;
    const int n = si.size + sj.size;
    const double fa = (double)sa.size, fb = (double)sb.size, fn = (double)n;
    double part_a = 0.0, part_b = 0.0;
    double rcp = 0.0, rcp_a = 0.0, rcp_b = 0.0, wa = 0.0, wb = 0.0;
    auto divide = [&] {  // while the sums are in flight; a division takes ~350 cycles, a read ~130
      const int na = sa.size + n, nb = n + sb.size;
      if (max(na, nb) < kRecips) {  // uniform; sizes are positive
        rcp = recip[n];
        rcp_a = recip[sa.size];
        rcp_b = recip[sb.size];
        wa = quotient(fa * fn, (double)na, recip[na]);
        wb = quotient(fn * fb, (double)nb, recip[nb]);
      } else {
        rcp = 1.0 / fn;
        rcp_a = 1.0 / fa;
        rcp_b = 1.0 / fb;
        wa = (fa * fn) / (fa + fn);
        wb = (fn * fb) / (fn + fb);
      }
    };
    auto add = [&](double xi, double xj, double xa, double xb, int d) {
      const double s = xi + xj;
      const double m = quotient(s, fn, rcp);
      const double da = quotient(xa, fa, rcp_a) - m, db = m - quotient(xb, fb, rcp_b);
      const double qa = da * da, qb = db * db;
      if (d < D) {
        ts[(int64_t)i * D + d] = s;
        part_a = part_a + qa;
        part_b = part_b + qb;
      }
    };
    if constexpr (KD > 0) {
      double xi[KD], xj[KD], xa[KD], xb[KD];
#pragma unroll
      for (int k = 0; k < KD; ++k) {  // unconditional (clamped): all in flight
        const int d = lane + LSA_WAVE * k, dc = d < D ? d : 0;
        xi[k] = pi[dc]; xj[k] = pj[dc]; xa[k] = pa[dc]; xb[k] = pb[dc];
      }
      divide();
#pragma unroll
      for (int k = 0; k < KD; ++k) add(xi[k], xj[k], xa[k], xb[k], lane + LSA_WAVE * k);
    } else {
      divide();
      for (int d = lane; d < (D + LSA_WAVE - 1) / LSA_WAVE * LSA_WAVE; d += LSA_WAVE) {
        const int dc = d < D ? d : 0;
        add(pi[dc], pj[dc], pa[dc], pb[dc], d);
      }
    }
    const double x = fold2(part_a, part_b);
    const bool right = lane >= 32;
    const bool pair = right ? b >= 0 && n + sb.size <= max_size : sa.size + n <= max_size;
    const double c = pair ? (right ? wb : wa) * x : INFINITY;
    const uint64_t u = __builtin_bit_cast(uint64_t, c);
    const uint64_t ca = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), 0) << 32 |
                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 0);
    const uint64_t ci = (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(u >> 32), 32) << 32 |
                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)u, 32);
    if (lane == 0) {  // uniform values
      cost[i] = ci;
      cost[j] = (uint64_t)kInfHi << 32;
      if (a >= 0) cost[a] = ca;
      seg[i].nxt = (int16_t)b;
      seg[i].size = n;
      seg[j].size = 0;
      if (b >= 0) seg[b].prv = (int16_t)i;
    }
    __builtin_amdgcn_wave_barrier();
    // the group of i from its costs as read before, the new ones put in; the groups of a and j
    // where they are others
    const int here = g * LSA_WAVE + lane;
    uint64_t k = here == a ? ca : kg;
    k = here == i ? ci : (here == j ? (uint64_t)kInfHi << 32 : k);
    set_group(g, k);
    if (a >= 0 && a / LSA_WAVE != g) set_group(a / LSA_WAVE, cost[a / LSA_WAVE * LSA_WAVE + lane]);
    if (j / LSA_WAVE != g) set_group(j / LSA_WAVE, cost[j / LSA_WAVE * LSA_WAVE + lane]);
  }

  int32_t* out = starts + table * (int64_t)(target + 1);
  if (failed) {
    // the even cut: valid, increasing positions for every kernel that reads the table later
    for (int r = lane; r < target; r += LSA_WAVE) out[r] = (int32_t)((int64_t)r * T / target);
  } else {
    int before = 0;
    for (int g = 0; g < groups; ++g) {
      const int i = g * LSA_WAVE + lane;
      const uint64_t m = __ballot(i < npool && seg[i < npool ? i : 0].size > 0);
      if ((m >> lane) & 1) out[before + __popcll(m & ((1ull << lane) - 1))] = i * pool;
      before += __popcll(m);
    }
  }
  if (lane == 0) {
    status[table] = failed;
    // system scope: the word may live in pinned host memory
    if (failed && failed_any) __hip_atomic_store(failed_any, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    out[target] = (int32_t)T;
  }
}

}  // namespace

extern "C" size_t lsa_ward_segments_scratch_bytes(int64_t tables, int64_t T, int32_t D, int32_t pool) {
  if (tables < 0 || T < 0 || D < 1 || pool < 1) return 0;
  const int64_t npool = (T + pool - 1) / pool;
  return (size_t)(tables * npool * D) * sizeof(double);
}

extern "C" int lsa_ward_segments(const void* keys, int k_dtype, int64_t B, int64_t T, int32_t kv_heads, int32_t D,
                                 int64_t kv_sb, int64_t kv_st, int64_t kv_sh, int32_t pool, int32_t target,
                                 int32_t max_size, void* scratch, size_t scratch_bytes, int32_t* starts,
                                 int32_t* status, int32_t* failed, void* stream) {
  LSA_REQUIRE(keys && scratch && starts && status, LSA_ERR_NULL, "lsa_ward_segments: NULL pointer");
  LSA_REQUIRE(k_dtype == LSA_F32 || k_dtype == LSA_BF16 || k_dtype == LSA_F16, LSA_ERR_DTYPE,
              "lsa_ward_segments: dtype %d", k_dtype);
  LSA_REQUIRE(B >= 1 && T >= 1 && kv_heads >= 1 && D >= 1 && D <= kMergeThreads && pool >= 1 && target >= 1,
              LSA_ERR_SHAPE, "lsa_ward_segments: bad sizes");
  LSA_REQUIRE(T < (1ll << 31), LSA_ERR_SHAPE, "lsa_ward_segments: T = %lld does not fit int32 positions",
              (long long)T);
  const int64_t npool = (T + pool - 1) / pool;
  LSA_REQUIRE(npool <= kMaxPools, LSA_ERR_SHAPE,
              "lsa_ward_segments: %lld pools exceed %d (raise the pool size)", (long long)npool, kMaxPools);
  LSA_REQUIRE(target <= npool, LSA_ERR_SHAPE, "lsa_ward_segments: target %d exceeds the %lld pools", target,
              (long long)npool);
  LSA_REQUIRE(max_size >= pool, LSA_ERR_SHAPE, "lsa_ward_segments: max_size %d below the pool size %d", max_size,
              pool);
  const int64_t tables = B * kv_heads;
  LSA_REQUIRE(tables <= 65535, LSA_ERR_SHAPE, "lsa_ward_segments: too many tables");
  const size_t need = lsa_ward_segments_scratch_bytes(tables, T, D, pool);
  LSA_REQUIRE(scratch_bytes >= need, LSA_ERR_SHAPE, "lsa_ward_segments: scratch %zu bytes, needs %zu", scratch_bytes,
              need);
  hipStream_t s = (hipStream_t)stream;
  double* sums = (double*)scratch;
  const dim3 grid((unsigned)((npool * D + kPoolThreads - 1) / kPoolThreads), (unsigned)tables);
  LSA_DISPATCH_QT(k_dtype, {
    pool_sums_kernel<QT><<<grid, kPoolThreads, 0, s>>>((const QT*)keys, T, kv_heads, D, kv_sb, kv_st, kv_sh, pool,
                                                       (int)npool, sums);
  })
  LSA_LAUNCHED("lsa_ward_segments (pool sums)");
  // enough waves that the first costs take a few rounds
  const int threads = npool >= 1024 ? kMergeThreads : (npool >= 256 ? 512 : 256);
  const dim3 tg((unsigned)tables);
#define LSA_MERGE(KD)                                                                                             \
  if (npool <= kSmallPools)                                                                                       \
    ward_merge_kernel<KD, kSmallPools><<<tg, threads, 0, s>>>(sums, T, D, pool, (int)npool, target, max_size, starts, \
                                                              status, failed);                                    \
  else                                                                                                            \
    ward_merge_kernel<KD, kMaxPools><<<tg, threads, 0, s>>>(sums, T, D, pool, (int)npool, target, max_size, starts,   \
                                                            status, failed);
  if (D <= 64) {
    LSA_MERGE(1)
  } else if (D <= 128) {
    LSA_MERGE(2)
  } else if (D <= 256) {
    LSA_MERGE(4)
  } else {
    LSA_MERGE(0)
  }
#undef LSA_MERGE
  LSA_LAUNCHED("lsa_ward_segments (merge)");
  return LSA_OK;
}
