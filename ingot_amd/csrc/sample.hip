// Temperature > 0 verification by rejection sampling, and the verify-row chooser, on gfx950.
//
// Reference: Shaders/zz_sample.metal:1-281 (topk64_part / topk64_merge: per row the 64 best logits, ties to the lower
// id, and the max and Σ exp((x − max)/T) over the whole vocabulary; sample_dist: temperature → top-k → min-p → top-p
// over the 64 candidates; spec_accept_sample: draft d of row i accepted with probability p_i(d), otherwise the token is
// drawn from p_i without d, so the emitted tokens follow the target distribution exactly) and spec_rows_choose
// (Shaders/yy_model.metal:644-675, SpecRows.swift: the rows with the best expected tokens per cost).
//
// MI355X design: a 64-entry list is one value per lane of a wave, sorted by a bitonic network of lane exchanges; two
// lists merge as the better of list[l] and batch[63 − l], a bitonic sequence holding the 64 best that six exchange stages
// sort. The vocabulary is streamed twice (a bound, then the few logits that reach it) so that only ≈ 200 values a row are
// ever sorted; the acceptance holds one candidate per lane and one row per wave.
#include <cfloat>
#include <cmath>

#include "ih_internal.h"
#include "lanes.h"

namespace ih {

constexpr int SK = IH_TOPK;      // candidates per row
constexpr int SPG = 32;          // chunks (workgroups) per row
constexpr int SPT = 256;         // threads per chunk workgroup (SPG chunks of interleaved 64-logit blocks)
constexpr uint32_t NO_ID = 0xFFFFFFFFu;

// (v, i) ranks before (w, j): larger value, ties to the lower id (tk_better, yy_model.metal:503).
__device__ __forceinline__ bool tk_better(float v, uint32_t i, float w, uint32_t j) {
  return (v > w) | ((v == w) & (i < j));  // no short circuit: compares and masks, no branches
}

// Compare-exchange with lane ^ J: the lane ends with the better of the pair if keep_better, else the worse. The
// partner's value and id come through DPP / row-swap lane patterns (lane_xor), not an LDS round trip; every lane of
// the wave is active wherever these run.
template <int J>
__device__ __forceinline__ void cx(float& v, uint32_t& id, bool keep_better) {
  const float ov = lane_xor<J>(v);
  const uint32_t oi = __float_as_uint(lane_xor<J>(__uint_as_float(id)));
  const bool take = (keep_better & tk_better(ov, oi, v, id)) | (!keep_better & tk_better(v, id, ov, oi));
  v = take ? ov : v;
  id = take ? oi : id;
}

// Bitonic sort of one value per lane into descending rank order (lane 0 the best).
__device__ __forceinline__ void sort64(float& v, uint32_t& id, int lane) {
#define IH_CX(K, J) cx<J>(v, id, (((lane & (J)) == 0) == ((lane & (K)) == 0)))
  IH_CX(2, 1);
  IH_CX(4, 2); IH_CX(4, 1);
  IH_CX(8, 4); IH_CX(8, 2); IH_CX(8, 1);
  IH_CX(16, 8); IH_CX(16, 4); IH_CX(16, 2); IH_CX(16, 1);
  IH_CX(32, 16); IH_CX(32, 8); IH_CX(32, 4); IH_CX(32, 2); IH_CX(32, 1);
  IH_CX(64, 32); IH_CX(64, 16); IH_CX(64, 8); IH_CX(64, 4); IH_CX(64, 2); IH_CX(64, 1);
#undef IH_CX
}

// The 64 best of two descending lists (the list in v/id, the other in bv/bi), descending, in v/id.
// x of lane 63 − lane (= lane ^ 63): the row mirror (i ^ 15 within 16 lanes), then the row swaps 16 and 32.
__device__ __forceinline__ float rev64(float x) {
  return lane_xor<32>(lane_xor<16>(__int_as_float(dpp_mov<0x140>(__float_as_int(x)))));
}

__device__ __forceinline__ void merge64(float& v, uint32_t& id, float bv, uint32_t bi, int lane) {
  const float rv = rev64(bv);
  const uint32_t ri = __float_as_uint(rev64(__uint_as_float(bi)));
  const bool take = tk_better(rv, ri, v, id);
  v = take ? rv : v;
  id = take ? ri : id;
  // v is now bitonic (descending, then ascending); six half-cleaners sort it.
  cx<32>(v, id, (lane & 32) == 0);
  cx<16>(v, id, (lane & 16) == 0);
  cx<8>(v, id, (lane & 8) == 0);
  cx<4>(v, id, (lane & 4) == 0);
  cx<2>(v, id, (lane & 2) == 0);
  cx<1>(v, id, (lane & 1) == 0);
}

// Online (max, Σ exp((x − max)/T)) of one lane over a batch of values (the max starts at −FLT_MAX, as the reference's,
// so −inf logits add exp(−inf) = 0; NaN logits and values past the row are passed as not ok): one exponential per value
// and one per batch. exp(0) is taken as exactly 1 where either operand is the new max.
template <int N>
__device__ __forceinline__ void lse_batch(const float (&c)[N], const bool (&ok)[N], float it, float& mt, float& s) {
  float nm = mt;
#pragma unroll
  for (int u = 0; u < N; ++u) nm = ok[u] ? fmaxf(nm, c[u]) : nm;
  s = mt == nm ? s : s * __expf((mt - nm) * it);
#pragma unroll
  for (int u = 0; u < N; ++u) s += !ok[u] ? 0.f : (c[u] == nm ? 1.0f : __expf((c[u] - nm) * it));
  mt = nm;
}

// The 64 best of a row in three launches. A row is cut into blocks of 64 consecutive logits, block b belonging to chunk b
// mod SPG (interleaved, so that a masked or ordered stretch of the vocabulary falls on every chunk).
//   1. topk64_bound_kernel, one workgroup per (chunk, row): the chunk's (max, Σ exp) and its second best value. The
//      smallest of the 32 second bests is a value that at least 64 logits of the row reach.
//   2. topk64_collect_kernel, the same workgroups: the chunk's logits that reach it, in any order, to the chunk's own
//      slots (≈ 170 of 151936 per row for independent logits; one list per row behind a global counter took 38 µs).
//   3. topk64_final_kernel, one workgroup per row: the candidates sorted.
// A chunk with more candidates than slots (many logits equal to the bound, e.g. a vocabulary masked with one finite value)
// hands on those above the bound and the first 64 equal to it; one with more than 64 above it, its best 64. Values below
// −FLT_MAX and NaN are never candidates; missing entries are (−FLT_MAX, NO_ID).
// A 17 × 151936 round: bound 6.9, collect 4.3, final 7.9 µs, against 28 + 9 for running best-64 lists per chunk and their
// merge, whose sorting networks were one long dependency chain per wave. With all but 40 logits of a row at −1e9: 23.4 µs
// (81 where one workgroup scanned such a row, 23.0 by the lists).
constexpr int CCAP = 128;        // candidates kept per chunk (sorted logits: one block of 64)
struct TopScratch {
  float* thr;    // [rows][SPG] second best of each chunk
  float2* pz;    // [rows][SPG] (max, Σ exp)
  unsigned* cnt; // [rows][SPG] candidates; crowded: above the bound | equal << 8 | equal in the first block << 16
  uint2* cand;   // [rows][SPG][CCAP] (value bits, id); crowded: above the bound from 0, equal to it from SK
};

__global__ __launch_bounds__(SPT) void topk64_bound_kernel(const float* __restrict__ x, int ldx, int V, float temp,
                                                           TopScratch t) {
  constexpr int NB = 8;  // loads in flight per lane
  __shared__ float r1[SPT / 64], r2[SPT / 64], rm[SPT / 64], rs[SPT / 64];
  const int g = blockIdx.x, row = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float it = 1.0f / temp;
  const float* xr = x + size_t(row) * ldx;
  float a1 = -FLT_MAX, a2 = -FLT_MAX, mt = -FLT_MAX, s = 0.f;
  constexpr int STRIDE = 64 * SPG * (SPT / 64);  // elements between a wave's blocks
  for (int base = 64 * (g + SPG * wave); base < V; base += STRIDE * NB) {
    float c[NB];
    bool ok[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) c[u] = xr[min(base + STRIDE * u + lane, V - 1)];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      ok[u] = base + STRIDE * u + lane < V && c[u] == c[u];
      const float v = ok[u] ? c[u] : -FLT_MAX;
      a2 = fmaxf(a2, fminf(a1, v));
      a1 = fmaxf(a1, v);
    }
    lse_batch<NB>(c, ok, it, mt, s);
  }
  // The two best and the (max, sum) of the wave, then of the workgroup.
  auto two = [&](float b1, float b2) {
    a2 = fmaxf(fminf(a1, b1), fmaxf(a2, b2));
    a1 = fmaxf(a1, b1);
  };
  float m = mt;
  auto step = [&](auto hc) {
    constexpr int H = decltype(hc)::value;
    two(lane_xor<H>(a1), lane_xor<H>(a2));
    m = fmaxf(m, lane_xor<H>(m));
  };
  step(std::integral_constant<int, 32>{});
  step(std::integral_constant<int, 16>{});
  step(std::integral_constant<int, 8>{});
  step(std::integral_constant<int, 4>{});
  step(std::integral_constant<int, 2>{});
  step(std::integral_constant<int, 1>{});
  float ss = s * __expf((mt - m) * it);
  ss += lane_xor<32>(ss);
  ss += lane_xor<16>(ss);
  ss += lane_xor<8>(ss);
  ss += lane_xor<4>(ss);
  ss += lane_xor<2>(ss);
  ss += lane_xor<1>(ss);
  if (lane == 0) {
    r1[wave] = a1;
    r2[wave] = a2;
    rm[wave] = m;
    rs[wave] = ss;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  float M = rm[0];
  for (int w = 1; w < SPT / 64; ++w) {
    two(r1[w], r2[w]);
    M = fmaxf(M, rm[w]);
  }
  float Z = 0.f;
  for (int w = 0; w < SPT / 64; ++w) Z += rs[w] * __expf((rm[w] - M) * it);
  t.thr[row * SPG + g] = a2;
  t.pz[row * SPG + g] = make_float2(M, Z);
}

// The NW lists of a workgroup (one per wave, descending in v/id) merged into wave 0's.
template <int NW>
__device__ __forceinline__ void merge_waves(float& v, uint32_t& id, float (*sv)[SK], uint32_t (*si)[SK], int wave,
                                            int lane) {
#pragma unroll
  for (int n = NW / 2; n >= 1; n >>= 1) {  // waves n … 2n − 1 hand theirs to waves 0 … n − 1
    if (wave >= n && wave < 2 * n) {
      sv[wave][lane] = v;
      si[wave][lane] = id;
    }
    __syncthreads();
    if (wave < n) merge64(v, id, sv[wave + n][lane], si[wave + n][lane], lane);
  }
}

__global__ __launch_bounds__(SPT) void topk64_collect_kernel(const float* __restrict__ x, int ldx, int V, TopScratch t) {
  constexpr int NB = 8;
  __shared__ unsigned count;
  const int g = blockIdx.x, row = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* xr = x + size_t(row) * ldx;
  uint2* cand = t.cand + (size_t(row) * SPG + g) * CCAP;
  if (threadIdx.x == 0) count = 0u;
  __syncthreads();
  float thr = t.thr[row * SPG + (lane & (SPG - 1))];
  thr = fminf(thr, lane_xor<16>(thr));
  thr = fminf(thr, lane_xor<8>(thr));
  thr = fminf(thr, lane_xor<4>(thr));
  thr = fminf(thr, lane_xor<2>(thr));
  thr = fminf(thr, lane_xor<1>(thr));
  constexpr int STRIDE = 64 * SPG * (SPT / 64);
  for (int base = 64 * (g + SPG * wave); base < V; base += STRIDE * NB) {
    float c[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) c[u] = xr[min(base + STRIDE * u + lane, V - 1)];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = base + STRIDE * u + lane;
      const bool take = i < V && c[u] >= thr;  // NaN compares false
      const unsigned long long mask = __ballot(take);
      if (mask == 0ull) continue;  // uniform
      unsigned at = 0;
      if (lane == 0) at = atomicAdd(&count, unsigned(__popcll(mask)));
      at = __builtin_amdgcn_readfirstlane(at) + unsigned(__popcll(mask & ((1ull << lane) - 1ull)));
      if (take && at < CCAP) cand[at] = make_uint2(__float_as_uint(c[u]), uint32_t(i));
    }
  }
  __syncthreads();
  const unsigned n = count;  // uniform
  if (n <= unsigned(CCAP)) {
    if (threadIdx.x == 0) t.cnt[row * SPG + g] = n;
    return;
  }
  // Too many: the values above the bound to slots 0 …, of those equal to it the first 64 in order to slots SK … (block j of
  // the chunk is wave j mod 4's).
  constexpr int NW = SPT / 64;
  __shared__ unsigned above, eqb[NW * NB];
  unsigned taken = 0, first = 0;  // uniform: equal values so far (to 64), those of the chunk's first block
  if (threadIdx.x == 0) above = 0u;
  __syncthreads();
  for (int b0 = 64 * g; b0 < V; b0 += STRIDE * NB) {  // uniform over the workgroup
    const int base = b0 + 64 * SPG * wave;
    float c[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) c[u] = xr[min(base + STRIDE * u + lane, V - 1)];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = base + STRIDE * u + lane;
      const unsigned long long mask = __ballot(i < V && c[u] > thr);
      if (mask) {
        unsigned at = 0;
        if (lane == 0) at = atomicAdd(&above, unsigned(__popcll(mask)));
        at = __builtin_amdgcn_readfirstlane(at) + unsigned(__popcll(mask & ((1ull << lane) - 1ull)));
        if ((mask >> lane & 1ull) && at < SK) cand[at] = make_uint2(__float_as_uint(c[u]), uint32_t(i));
      }
      const unsigned long long eq = __ballot(i < V && c[u] == thr);
      if (lane == 0) eqb[NW * u + wave] = unsigned(__popcll(eq));
    }
    if (taken >= SK) continue;
    __syncthreads();
    unsigned e = lane < NW * NB ? eqb[lane] : 0u, sum = e;
#pragma unroll
    for (int d = 1; d < NW * NB; d <<= 1) {
      const unsigned o = __shfl_up(sum, d);
      if (lane >= d) sum += o;
    }
    if (b0 == 64 * g) first = min(__builtin_amdgcn_readlane(e, 0), unsigned(SK));
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int j = NW * u + wave, i = base + STRIDE * u + lane;
      const unsigned before = taken + __builtin_amdgcn_readlane(sum, j) - __builtin_amdgcn_readlane(e, j);
      if (before >= SK) continue;
      const unsigned long long eq = __ballot(i < V && c[u] == thr);
      const unsigned at = before + unsigned(__popcll(eq & ((1ull << lane) - 1ull)));
      if ((eq >> lane & 1ull) && at < SK) cand[SK + at] = make_uint2(__float_as_uint(c[u]), uint32_t(i));
    }
    taken = min(taken + __builtin_amdgcn_readlane(sum, NW * NB - 1), unsigned(SK));
    __syncthreads();
  }
  __syncthreads();
  const unsigned na = above;  // uniform
  if (na <= SK) {
    if (threadIdx.x == 0) t.cnt[row * SPG + g] = na | taken << 8 | first << 16;
    return;
  }
  // More than 64 above the bound as well: the chunk's best 64, by a running list per wave. A block enters its wave's list
  // only if one of its values beats the list's last entry (a lane's batch in LDS: a register file has no index).
  __shared__ float sv[NW][SK];
  __shared__ uint32_t si[NW][SK];
  __shared__ float batch[NB][SPT];
  float v = -FLT_MAX;
  uint32_t id = NO_ID;
  auto enters = [&](float b, uint32_t bid) {
    const float tv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
    const uint32_t ti = uint32_t(__builtin_amdgcn_readlane(int(id), 63));
    return __any(tk_better(b, bid, tv, ti));
  };
  for (int base = 64 * (g + SPG * wave); base < V; base += STRIDE * NB) {
    float c[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) c[u] = xr[min(base + STRIDE * u + lane, V - 1)];
    unsigned need = 0;  // uniform: the batch's blocks that may enter
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int i = base + STRIDE * u + lane;
      c[u] = i < V && c[u] > thr ? c[u] : -INFINITY;
      batch[u][threadIdx.x] = c[u];
      need |= enters(c[u], uint32_t(i)) ? 1u << u : 0u;
    }
    for (; need; need &= need - 1) {
      const int u = __builtin_ctz(need);
      float b = batch[u][threadIdx.x];
      uint32_t bid = b == -INFINITY ? NO_ID : uint32_t(base + STRIDE * u + lane);
      b = b == -INFINITY ? -FLT_MAX : b;
      if (!enters(b, bid)) continue;
      sort64(b, bid, lane);
      merge64(v, id, b, bid, lane);
    }
  }
  merge_waves<NW>(v, id, sv, si, wave, lane);
  if (wave == 0) cand[lane] = make_uint2(__float_as_uint(v), id);
  if (threadIdx.x == 0) t.cnt[row * SPG + g] = unsigned(SK);
}

constexpr int FT = 512;  // threads of the final kernel
__global__ __launch_bounds__(FT) void topk64_final_kernel(const float* __restrict__ x, int ldx, int V, float temp,
                                                          TopScratch t, uint32_t* __restrict__ idx,
                                                          float* __restrict__ val, float* __restrict__ z) {
  __shared__ float sv[FT / 64][SK];
  __shared__ uint32_t si[FT / 64][SK];
  __shared__ uint2 list[SPG * CCAP];
  const int row = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // The chunks' counts, one per lane of the lower half: candidates; in crowded chunks those above the bound, those equal to
  // it and how many of these lie in the chunk's first block. The first blocks of all chunks are the row's first logits, so
  // where they hold 64 equal values no others are needed. Then where each chunk's candidates start in the row's list.
  const unsigned cw = lane < SPG ? t.cnt[row * SPG + lane] : 0u, cn = cw & 255u, e0 = cw >> 16;
  auto scan = [&](unsigned x) {
#pragma unroll
    for (int d = 1; d < SPG; d <<= 1) {
      const unsigned o = __shfl_up(x, d);
      if (lane >= d) x += o;
    }
    return x;
  };
  unsigned eq = cw >> 8 & 255u;
  if (__any(eq != 0u)) {
    const unsigned upto = scan(e0);
    if (__builtin_amdgcn_readlane(upto, SPG - 1) >= SK) eq = min(e0, unsigned(max(0, SK - int(upto - e0))));
  }
  const unsigned at = scan(cn + eq), n = __builtin_amdgcn_readlane(at, SPG - 1);
  for (int g = wave; g < SPG; g += FT / 64) {
    const unsigned cg = __builtin_amdgcn_readlane(cn, g), eg = __builtin_amdgcn_readlane(eq, g);
    const unsigned ag = __builtin_amdgcn_readlane(at, g) - cg - eg;
    const uint2* cand = t.cand + (size_t(row) * SPG + g) * CCAP;
    for (unsigned k = lane; k < cg + eg; k += 64) list[ag + k] = cand[k < cg ? k : SK + k - cg];
  }
  __syncthreads();
  const float it = 1.0f / temp;
  float v = -FLT_MAX;
  uint32_t id = NO_ID;
  bool first = true;
  for (unsigned b = 64 * wave; b < n; b += FT) {  // a batch of 64 candidates, one per lane, into the wave's list
    const uint2 w = b + lane < n ? list[b + lane] : make_uint2(__float_as_uint(-FLT_MAX), NO_ID);
    float c = __uint_as_float(w.x);
    uint32_t cid = w.y;
    sort64(c, cid, lane);
    if (first) {
      v = c;
      id = cid;
      first = false;
    } else {
      merge64(v, id, c, cid, lane);
    }
  }
  merge_waves<FT / 64>(v, id, sv, si, wave, lane);
  if (wave != 0) return;
  idx[size_t(row) * SK + lane] = id;
  val[size_t(row) * SK + lane] = v;
  const float2 p = lane < SPG ? t.pz[size_t(row) * SPG + lane] : make_float2(-FLT_MAX, 0.f);
  float M = p.x;
  M = fmaxf(M, lane_xor<16>(M));
  M = fmaxf(M, lane_xor<8>(M));
  M = fmaxf(M, lane_xor<4>(M));
  M = fmaxf(M, lane_xor<2>(M));
  M = fmaxf(M, lane_xor<1>(M));
  float Z = lane < SPG ? p.y * __expf((p.x - M) * it) : 0.f;
  Z += lane_xor<16>(Z);
  Z += lane_xor<8>(Z);
  Z += lane_xor<4>(Z);
  Z += lane_xor<2>(Z);
  Z += lane_xor<1>(Z);
  if (lane == 0) {
    z[2 * row] = M;
    z[2 * row + 1] = Z;
  }
}

// v[0] + v[1] + … + v[63] of a value per lane, added in that order (as the reference's sequential loop rounds; lanes past
// the count hold 0, which adds exactly nothing). Constant lane numbers: the reads run ahead of the chain of additions.
__device__ __forceinline__ float ordered_sum(float v) {
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < SK; ++j) s += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
  return s;
}

// Probabilities of a row's candidates after temperature, top-k, min-p and top-p, renormalised; returns how many
// remain (sample_dist, zz_sample.metal:196-226). One candidate (ci, cv) per lane: exponentials and divisions run on all
// lanes at once, every sum over j = 0, 1, … in order.
__device__ __forceinline__ int sample_dist(uint32_t ci, float cv, float M, float Z, const ih_sample_params& p, int lane,
                                           float& pr) {
  const float it = 1.0f / p.temp;
  // Lanes 0 … k − 1 of a mask's leading ones.
  auto leading = [](unsigned long long m) { return m == ~0ull ? 64 : int(__builtin_ctzll(~m)); };
  int n = leading(__ballot(ci != NO_ID));  // the leading candidates that exist
  const float e = __expf((cv - M) * it);
  float tot = Z;
  if (p.top_k > 0 && p.top_k < n) n = p.top_k;
  if (p.top_k > 0) tot = ordered_sum(lane < n ? e : 0.f);
  pr = lane < n ? e / tot : 0.f;
  if (p.min_p > 0.f) {
    const float thr = p.min_p * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pr), 0));
    n = leading(__ballot(lane == 0 || (lane < n && pr >= thr)));
    pr = lane < n ? pr : 0.f;
    const float sm = ordered_sum(pr);
    if (lane < n) pr /= sm;
  }
  if (p.top_p < 1.f) {
    // The first prefix that reaches top_p ends the set: as many prefixes as do not, and one more.
    float c = 0.f;
    int below = 0;
#pragma unroll
    for (int j = 0; j < SK; ++j) {
      c += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pr), j));
      below += j < n && !(c >= p.top_p) ? 1 : 0;
    }
    n = max(min(below + 1, n), 1);
    pr = lane < n ? pr : 0.f;
  }
  const float sm = ordered_sum(pr);
  pr = lane < n ? pr / sm : 0.f;
  return n;
}

// Acceptance by rejection (spec_accept_sample, zz_sample.metal:241-281): rows' candidates idx/val [rows][64] and
// (max, Z) [rows][2]; uniforms rnd[round · IH_RND_PER_ROUND + 2i] (accept) and [… + 2i + 1] (resample) of row i. Writes the record
// and advances the state as the greedy acceptance does (vtok[0] = the new anchor; the history as in accept_kernel).
// Wave w builds the distributions of rows w and w + 16, a candidate per lane (one lane per row with all its candidates
// took 19 µs: 64 divisions and three ordered sums in a row); wave 0 then finds the first rejected row with one ballot and
// walks that row's candidates to the drawn token (sample_pick, zz_sample.metal:228-239).
constexpr int AS_WAVES = 16;
__global__ __launch_bounds__(64 * AS_WAVES) void accept_sample_kernel(uint32_t* st, uint32_t* vtok, const uint32_t* cidx,
                                                                      const float* cval, const float* z, uint32_t* rec,
                                                                      const float* rnd, ih_sample_params p, int ring,
                                                                      int rows, uint32_t* hist, int hist_cap) {
  __shared__ float prs[IH_MAX_ROWS][SK];
  __shared__ int ns[IH_MAX_ROWS];
  __shared__ float qs[IH_MAX_ROWS];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t nr = rows ? uint32_t(rows) : min(max(st[6], 1u), uint32_t(IH_MAX_ROWS));
  const uint32_t round = st[5], p0 = st[0];
  // Wave 0's walk: the round's uniforms and block, one per lane, requested before the distributions.
  const float un = wave == 0 && lane < 2 * int(nr) ? rnd[size_t(round) * IH_RND_PER_ROUND + lane] : 0.f;
  const uint32_t tok = lane < int(nr) ? vtok[lane] : NO_ID;
  for (uint32_t i = wave; i < nr; i += AS_WAVES) {
    const uint32_t ci = cidx[i * SK + lane];
    float pr;
    const int n = sample_dist(ci, cval[i * SK + lane], z[2 * i], z[2 * i + 1], p, lane, pr);
    const uint32_t d = i + 1 < nr ? uint32_t(__builtin_amdgcn_readlane(int(tok), i + 1)) : NO_ID;
    const unsigned long long hit = __ballot(lane < n && ci == d);
    prs[i][lane] = pr;
    if (lane == 0) ns[i] = n;
    if (hit == 0ull ? lane == 0 : lane == int(__builtin_ctzll(hit))) qs[i] = hit == 0ull ? 0.f : pr;
  }
  __syncthreads();
  if (wave != 0) return;
  // Row i accepts its draft if its uniform 2i is below the draft's probability; the last row has no draft.
  const float u = __shfl(un, 2 * min(lane, IH_MAX_ROWS - 1));
  const unsigned long long okm = __ballot(lane + 1 < int(nr) && u < qs[min(lane, IH_MAX_ROWS - 1)]);
  const int m = int(__builtin_ctzll(~okm));  // < 64: at most 16 rows have a draft
  const uint32_t skip = m + 1 < int(nr) ? uint32_t(__builtin_amdgcn_readlane(int(tok), m + 1)) : NO_ID;
  const float q = m + 1 < int(nr) ? qs[m] : 0.f;
  const float ur = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(un), 2 * m + 1));
  // A token of row m without `skip` (whose mass is q): the first candidate whose ordered sum passes the target, else the
  // last one.
  const uint32_t ci = cidx[m * SK + lane];
  const float pr = prs[m][lane], target = ur * (1.0f - q);
  const int n = ns[m];
  const float part = lane < n && ci != skip ? pr : 0.f;
  float sum = 0.f;
  int pick = 0;  // prefixes that do not pass the target; the skipped candidate adds nothing, so it never is the first
#pragma unroll
  for (int j = 0; j < SK; ++j) {
    sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(part), j));
    pick += sum > target ? 0 : 1;
  }
  const unsigned long long valid = __ballot(lane < n && ci != skip);
  if (pick >= n) pick = valid ? 63 - int(__builtin_clzll(valid)) : 0;
  const uint32_t next = uint32_t(__builtin_amdgcn_readlane(int(ci), pick));
  // Emitted tokens: the accepted drafts, then `next`.
  const uint32_t draft = uint32_t(__shfl(int(tok), min(lane + 1, 63)));  // every lane active
  const uint32_t out = lane == m ? next : draft;
  uint32_t* r = rec + (round % uint32_t(ring)) * IH_REC_STRIDE;
  if (lane <= m) {
    r[1 + lane] = out;
    if (hist && p0 + 1 + lane < uint32_t(hist_cap)) hist[p0 + 1 + lane] = out;
  }
  if (lane != 0) return;
  r[0] = uint32_t(m);
  r[IH_REC_ROWS] = nr;
  r[IH_REC_P] = p0;
  st[3] = p0;
  st[2] = uint32_t(m) + 1;
  st[0] = p0 + uint32_t(m) + 1;
  st[1] = uint32_t(m) + 1;
  st[4] = next;
  st[5] = round + 1;
  vtok[0] = next;
}

// Verification rows of the round (spec_rows_choose, yy_model.metal:654-675): with draft t's calibrated acceptance
// q_t = sigmoid(a_g · logit(conf_t) + b_g) (g = min(t, 3)), expected tokens E(k) = 1 + Σ_{i<k−1} Π_{t≤i} q_t, the
// k in [kmin, kmax] with the highest E(k) / cost(k) goes to st[6].
__global__ void rows_choose_kernel(uint32_t* st, const float* conf, ih_rows_params p) {
  if (threadIdx.x != 0 || blockIdx.x != 0) return;
  float acc = 1.f, lp = 1.f, bv = -1.f;
  uint32_t best = uint32_t(p.kmax);
  for (int t = 0; t + 1 < p.kmax; ++t) {
    const int g = min(t, 3);
    const float c = fminf(fmaxf(conf[t], 1e-6f), 1.0f - 1e-6f);
    const float q = 1.0f / (1.0f + __expf(-(p.a[g] * __logf(c / (1.0f - c)) + p.b[g])));
    lp *= q;
    acc += lp;
    const int k = t + 2;
    if (k >= p.kmin) {
      const float v = acc / p.cost[k];
      if (v > bv) {
        bv = v;
        best = uint32_t(k);
      }
    }
  }
  st[6] = best;
}

int ensure_samp(ih_ctx* c, size_t bytes) {
  if (c->samp_bytes >= bytes) return IH_OK;
  ++c->gen;
  IH_HIP(hipStreamSynchronize(c->stream));
  if (c->samp) IH_HIP(hipFree(c->samp));
  c->samp = nullptr;
  c->samp_bytes = 0;
  if (hipMalloc(&c->samp, bytes) != hipSuccess) return fail(IH_ENOMEM, "sampling scratch allocation failed");
  c->samp_bytes = bytes;
  return IH_OK;
}

int launch_topk64(ih_ctx* c, const float* x, int ldx, int rows, int V, float temp, uint32_t* idx, float* val,
                  float* z) {
  TopScratch t;
  const size_t np = size_t(rows) * SPG, nc = np * CCAP;
  IH_TRY(ensure_samp(c, nc * sizeof(uint2) + np * (sizeof(float2) + sizeof(float) + sizeof(unsigned))));
  t.cand = static_cast<uint2*>(c->samp);
  t.pz = reinterpret_cast<float2*>(t.cand + nc);
  t.thr = reinterpret_cast<float*>(t.pz + np);
  t.cnt = reinterpret_cast<unsigned*>(t.thr + np);
  {
    TimedLaunch tl(c, TC_ARGMAX, double(rows) * V * 4);
    tlaunch(tl, topk64_bound_kernel, dim3(SPG, rows), dim3(SPT), 0, c->stream, x, ldx, V, temp, t);
    IH_HIP(hipGetLastError());
  }
  topk64_collect_kernel<<<dim3(SPG, rows), SPT, 0, c->stream>>>(x, ldx, V, t);
  IH_HIP(hipGetLastError());
  topk64_final_kernel<<<rows, FT, 0, c->stream>>>(x, ldx, V, temp, t, idx, val, z);
  IH_HIP(hipGetLastError());
  return IH_OK;
}

int launch_accept_sample(ih_ctx* c, uint32_t* st, uint32_t* vtok, const uint32_t* idx, const float* val,
                         const float* z, uint32_t* rec, const float* rnd, const ih_sample_params& p, int ring, int rows,
                         uint32_t* hist, int hist_cap) {
  accept_sample_kernel<<<1, 64 * AS_WAVES, 0, c->stream>>>(st, vtok, idx, val, z, rec, rnd, p, ring, rows, hist, hist_cap);
  IH_HIP(hipGetLastError());
  return IH_OK;
}

}  // namespace ih

using namespace ih;

extern "C" {

int ih_topk64_dev(ih_ctx* c, const float* logits_dev, int ldl, int rows, int V, float temp, uint32_t* idx_dev,
                  float* val_dev, float* z_dev) {
  IH_CHECK(c && logits_dev && idx_dev && val_dev && z_dev, IH_EINVAL, "ih_topk64_dev: null argument");
  IH_CHECK(rows >= 1 && rows <= 256 && V >= 1 && ldl >= V, IH_EINVAL, "ih_topk64_dev: bad shape");
  IH_CHECK(temp > 0.f && std::isfinite(temp), IH_EINVAL, "ih_topk64_dev: temperature must be positive");
  return launch_topk64(c, logits_dev, ldl, rows, V, temp, idx_dev, val_dev, z_dev);
}

int ih_spec_accept_sample_dev(ih_ctx* c, uint32_t* st_dev, uint32_t* vtok_dev, const uint32_t* idx_dev,
                              const float* val_dev, const float* z_dev, uint32_t* rec_dev, const float* rnd_dev,
                              const ih_sample_params* p, int ring, int rows) {
  IH_CHECK(c && st_dev && vtok_dev && idx_dev && val_dev && z_dev && rec_dev && rnd_dev && p, IH_EINVAL,
           "ih_spec_accept_sample_dev: null argument");
  IH_CHECK(ring >= 1 && rows >= 0 && rows <= IH_MAX_ROWS, IH_EINVAL, "ih_spec_accept_sample_dev: bad ring or rows");
  IH_CHECK(p->temp > 0.f && p->top_p > 0.f && p->top_k >= 0 && p->min_p >= 0.f, IH_EINVAL,
           "ih_spec_accept_sample_dev: need temp > 0, top_p > 0, top_k >= 0, min_p >= 0");
  return launch_accept_sample(c, st_dev, vtok_dev, idx_dev, val_dev, z_dev, rec_dev, rnd_dev, *p, ring, rows, nullptr,
                              0);
}

int ih_spec_rows_choose_dev(ih_ctx* c, uint32_t* st_dev, const float* conf_dev, const ih_rows_params* p) {
  IH_CHECK(c && st_dev && conf_dev && p, IH_EINVAL, "ih_spec_rows_choose_dev: null argument");
  IH_CHECK(p->kmin >= 2 && p->kmin <= p->kmax && p->kmax <= IH_MAX_ROWS, IH_EINVAL,
           "ih_spec_rows_choose_dev: need 2 <= kmin <= kmax <= 17");
  rows_choose_kernel<<<1, 64, 0, c->stream>>>(st_dev, conf_dev, *p);
  IH_HIP(hipGetLastError());
  return IH_OK;
}

}  // extern "C"
