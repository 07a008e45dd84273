// Verify-block attention over the int8 KV cache on gfx950: prework (RoPE, Hadamard, int8 K/V write), split-key
// flash-decoding on MFMA, and the fixed-order reduction of the splits.
//
// Reference: AttentionLayer.encode pieces prework → attn → reduce (Sources/Ingot/Layers/Attention.swift:398-525);
// kernels vattn_prework_i8 (Shaders/verify_attn_nax.metal:47-146), pattn_i8<RG, DEC=true> (Shaders/verify_attn_pf.metal:
// 49-398) and vattn_reduce (Shaders/verify_attn.metal:149-192).
//
// Cache: K and V int8 in 32-slot blocks laid out as MFMA operands (k_index, v_index in attn_args.h), one fp16 scale per
// token and head, symmetric. K holds H·k (orthonormal Walsh–Hadamard of the roped key) when hadk is set, and q is rotated
// the same way, so (Hq)·(Hk) = q·k.
//
// MI355X design: one workgroup of 16 waves per (key split, KV head, 80 query rows); the split size C is fixed per cache
// so that all splits of all heads are one workgroup per CU. A split goes in rounds of three 32-key steps, one per key
// class: 15 waves hold one (16-query tile, class) each, every wave stages a sixteenth of the next round (int8 → fp16
// fragments in LDS, two rounds of loads in flight). Sᵀ = K·Qᵀ (v_mfma_f32_16x16x32_f16, keys as rows so each lane holds
// 4 keys of one query), online softmax in base 2 per query column, P stays in registers as the B operand of
// Oᵀ += Vᵀ·Pᵀ. The classes are merged in LDS; a split writes O/l in fp16 with its (reference, sum) and the reduction
// merges the splits in a fixed order. Blocks of at most 32 query rows, and larger ones whose tiles in pairs are at most one
// workgroup per CU, take a kernel of three waves per tile that reads the cache straight into MFMA operands
// (attn_few_kernel); both run the same attn_step and attn_merge. A query's result
// does not depend on the other rows of the block: steps and classes are counted from fixed key positions, the split
// boundaries are fixed multiples of C, and every row is reduced in the same order whatever tile it falls in.
//
// What bounds it: no one unit. A 1056-key split of 80 rows (32K positions, 8 KV heads of 128, 27.5 µs) by its counters: a
// wave lives 22.5 µs, in which a SIMD's vector ALU is busy for 11.9 (conversion, softmax), a CU's LDS for 11.3 (no bank
// conflicts), a SIMD's matrix core for 4.3, and the HBM stream takes 9.9 at 6.9 TB/s; the rest is the wait for the first
// loads and the merge, during which none of them works. One tile per wave at 16 waves (four
// per SIMD, 128 VGPRs) overlaps them better than two or three tiles per wave at eight (28.7 against 33.2 µs, and
// 54.5 → 32.7 µs with 64-dim heads over 64K positions, where one wave per tile left three SIMDs with one tile).

#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdlib>

#include "act.h"
#include "attn_args.h"
#include "ih_internal.h"
#include "lanes.h"
#include "qmm_common.h"

namespace ih {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// AttnArgs: attn_args.h.

// ---------------------------------------------------------------------------------------------------------------
// One Walsh–Hadamard butterfly stage over lanes at distance H.
template <int H, int NE>
__device__ __forceinline__ void wht_stage(float (&x)[NE], int lane) {
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const float o = lane_xor<H>(x[e]);
    x[e] = (lane & H) ? o - x[e] : x[e] + o;
  }
}

// Prework: vattn_prework_i8 (verify_attn_nax.metal:47-146) without QK-norm and gate (the configurations have neither):
// RoPE on all HD dims (non-interleaved halves, angle pos·θ^(−i/(HD/2)) evaluated in double once per step into the
// table a.rope), orthonormal WHT of q and k when hadk (Sylvester order: stages h = 1, 2, 4, …, HD/2 with
// x[d] ← x[d] + x[d^h] where d & h = 0 and x[d^h] − x[d] where d & h ≠ 0, then ×1/√HD), int8 quantisation of k and v
// per (token, head): sc = fp16(amax/127) (1 when amax = 0), q = clamp(rint(x/sc), ±127), written at slot P + t.
// One wave per (head slot, token), lane l holding dims l + 64e: the RoPE partner of dim d is d ± HD/2 (the lane's
// other value at HD 128, the lane 32 away at HD 64), WHT stages h < 64 are lane exchanges (lane_xor) and h = 64 is
// in-lane — no LDS, no barrier. Grid (KVH, (G + 2)·B), one wave per workgroup: workgroup (kvh, j) takes token
// j / (G + 2) and, by j mod (G + 2), one of the group's G q heads, its k head or its v head. Consecutive workgroup ids
// go round-robin over the 8 XCDs, so with 8 KV heads a group's q and new K/V rows are written on XCD kvh, where the
// attention kernel's splits of that KV head run.
template <int HD>
__global__ __launch_bounds__(64) void prework_kernel(AttnArgs a) {
  constexpr int NE = HD / 64, RH = HD / 2;
  const int kvh = blockIdx.x, u = int(blockIdx.y) % (a.G + 2), t = int(blockIdx.y) / (a.G + 2);
  const int slot = u < a.G ? kvh * a.G + u : (u == a.G ? a.QH + kvh : a.QH + a.KVH + kvh);
  const int lane = threadIdx.x & 63;
  if (a.pos_dev && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) {
    const uint32_t p = a.pos_dev[0];
    if (p < uint32_t(a.pos_min) || p > uint32_t(a.pos_max)) a.flag_dev[0] = 1u;
  }
  if (slot >= a.QH + 2 * a.KVH) return;  // wave-uniform
  const bool isq = slot < a.QH, isk = !isq && slot < a.QH + a.KVH;
  // Column of the head in the projection row: q heads QS apart (a gated head is [q | gate]), then k heads, v heads.
  const int col = isq ? slot * a.QS : a.QH * a.QS + (slot - a.QH) * HD;
  const float* row = a.proj + size_t(t) * a.ldp + col;
  float x[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) x[e] = row[lane + 64 * e];
  if (a.qkv_bias) {
#pragma unroll
    for (int e = 0; e < NE; ++e) x[e] += a.qkv_bias[col + lane + 64 * e];
  }
  if ((isq || isk) && a.qnorm) {
    // QK-norm: x · rsqrt(mean x² + eps) · w over the head, before RoPE (the AT_QKN branch of vattn_prework_i8).
    float ss = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e) ss += x[e] * x[e];
    ss += lane_xor<32>(ss);
    ss += lane_xor<16>(ss);
    ss += lane_xor<8>(ss);
    ss += lane_xor<4>(ss);
    ss += lane_xor<2>(ss);
    ss += lane_xor<1>(ss);
    const float r = rsqrtf(ss / float(HD) + a.eps);
    const uint16_t* w = isq ? a.qnorm : a.knorm;
#pragma unroll
    for (int e = 0; e < NE; ++e) x[e] = x[e] * r * dbf16(w[lane + 64 * e]);
  }
  if (isq || isk) {
    if (a.rot == HD) {
      const float2 cs = a.rope[t * RH + (lane % RH)];
      if constexpr (NE == 2) {
        const float xl = x[0], xh = x[1];
        x[0] = xl * cs.x - xh * cs.y;
        x[1] = xh * cs.x + xl * cs.y;
      } else {
        const float o = lane_xor<RH>(x[0]);
        x[0] = lane < RH ? x[0] * cs.x - o * cs.y : x[0] * cs.x + o * cs.y;
      }
    } else {
      // Partial RoPE (AT_ROT < HD): dim d < rot pairs with d ± rot/2, read from the lane and element that hold it; the
      // dims from rot on keep their value.
      const int rh = a.rot >> 1;
      float y[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int d = lane + 64 * e, dp = d < rh ? d + rh : d - rh;
        float o = __shfl(x[0], dp & 63);
        if constexpr (NE == 2) {
          const float o1 = __shfl(x[1], dp & 63);
          o = (dp >> 6) ? o1 : o;
        }
        y[e] = x[e];
        if (d < a.rot) {
          const float2 cs = a.rope[t * rh + (d % rh)];
          y[e] = d < rh ? x[e] * cs.x - o * cs.y : x[e] * cs.x + o * cs.y;
        }
      }
#pragma unroll
      for (int e = 0; e < NE; ++e) x[e] = y[e];
    }
    if (a.hadk) {
      wht_stage<1>(x, lane);
      wht_stage<2>(x, lane);
      wht_stage<4>(x, lane);
      wht_stage<8>(x, lane);
      wht_stage<16>(x, lane);
      wht_stage<32>(x, lane);
      if constexpr (NE == 2) {
        const float x0 = x[0], x1 = x[1];
        x[0] = x0 + x1;
        x[1] = x0 - x1;
      }
#pragma unroll
      for (int e = 0; e < NE; ++e) x[e] *= HD == 128 ? 0.088388347648318441f : 0.125f;
    }
    if (isq) {
      const int kvh = slot / a.G;
      __half* q = a.q + (size_t(kvh) * a.Qpad + t * a.G + slot % a.G) * HD;
#pragma unroll
      for (int e = 0; e < NE; ++e) q[lane + 64 * e] = __float2half_rn(x[e]);
      return;
    }
  }
  // K or V: symmetric int8 with one fp16 scale per (token, head).
  float am = 0.f;
#pragma unroll
  for (int e = 0; e < NE; ++e) am = fmaxf(am, fabsf(x[e]));
  am = fmaxf(am, lane_xor<32>(am));
  am = fmaxf(am, lane_xor<16>(am));
  am = fmaxf(am, lane_xor<8>(am));
  am = fmaxf(am, lane_xor<4>(am));
  am = fmaxf(am, lane_xor<2>(am));
  am = fmaxf(am, lane_xor<1>(am));
  const __half sc16 = __float2half_rn(am > 0.f ? am / 127.0f : 1.0f);
  const float sc = __half2float(sc16);
  const int h = isk ? slot - a.QH : slot - a.QH - a.KVH;
  const int pos = attn_pos(a).P + t, kpos = a.ring ? pos % a.ring : pos;
  if (!a.ring && pos >= a.cap) return;  // a device position beyond the range the step was sized for (flagged)
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int d = lane + 64 * e;
    const uint8_t qv = kv_byte(fminf(127.f, fmaxf(-127.f, rintf(x[e] / sc))));
    if (isk) a.kc[k_index(h, kpos, d, HD, a.vld)] = qv;
    else a.vc[v_index(h, kpos, d, HD, a.vld)] = qv;
  }
  if (lane == 0) (isk ? a.ks : a.vs)[size_t(h) * a.vld + kpos] = sc16;
}

// ---------------------------------------------------------------------------------------------------------------
// Four cache bytes u = v + 128 ∈ [1, 255] → four exact fp16 values v: interleaved with the byte 0x64 they read as the
// halves 1024 + u; minus 1152 gives v.
__device__ __forceinline__ void u8x4_to_h(unsigned w, __half2& lo, __half2& hi) {
  const unsigned l = __builtin_amdgcn_perm(0x64646464u, w, 0x04010400u);
  const unsigned h = __builtin_amdgcn_perm(0x64646464u, w, 0x04030402u);
  const __half2 off = __halves2half2(__float2half(1152.f), __float2half(1152.f));
  lo = __hsub2(__builtin_bit_cast(__half2, l), off);
  hi = __hsub2(__builtin_bit_cast(__half2, h), off);
}

// Max over the 4 lanes of a query column (lanes j, j + 16, j + 32, j + 48) with the gfx950 lane swaps (no LDS round
// trip, unlike a shuffle).
__device__ __forceinline__ float row_max4(float x) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(y), __float_as_uint(y), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

constexpr int ATT_WAVES = 16, ATT_THREADS = 64 * ATT_WAVES;
constexpr int STEP = 32;        // keys of a step: one 32-slot block of the cache
constexpr int NCLS = 3;         // key classes of a split: step s belongs to class s mod 3
constexpr int WTILES = 5;       // 16-query tiles of a workgroup (80 query rows): 15 of the 16 waves multiply
constexpr float RAISE = 4.f;    // log2 of how far a row's max may pass its exponents' reference

// Eight cache values (two words, memory order) → fp16, exact.
__device__ __forceinline__ u32x4 u8x8_to_f16(unsigned w0, unsigned w1) {
  __half2 lo, hi;
  u32x4 v;
  u8x4_to_h(w0, lo, hi);
  v.x = __builtin_bit_cast(unsigned, lo);
  v.y = __builtin_bit_cast(unsigned, hi);
  u8x4_to_h(w1, lo, hi);
  v.z = __builtin_bit_cast(unsigned, lo);
  v.w = __builtin_bit_cast(unsigned, hi);
  return v;
}

// LDS of a workgroup: two buffers of a round's keys (three steps, one per class) as fp16 MFMA fragments and their
// scales. After the rounds the key buffers hold the merge's partial sums.
template <int HD>
struct AttnLds {
  static constexpr int NU = HD / 32;      // 1 KB cache units of a step's K, and of its V
  u32x4 kv[2][NCLS][2][2 * NU][64];       // K: [16-key group · HD/32 + 32-dim chunk][lane]; V: [16-dim tile][lane]
  float sc[2][NCLS][2][STEP];             // K and V scales of the step's keys
  float2 ml[NCLS][WTILES][16];
  __device__ f32x4 (*part())[64] { return reinterpret_cast<f32x4(*)[64]>(&kv[0][0][0][0][0]); }
  static_assert(sizeof(kv) >= size_t(WTILES) * (HD / 16) * (NCLS - 1) * 1024, "the merge fits the key buffers");
};

// A tile's state in one key class: O (lane (j, qd) holds dims 16dt + 4qd + i of query j), the exponents' reference and
// the lane's part of the sum.
template <int HD>
struct TileState {
  f32x4 o[HD / 16];
  float mrun, lsum;
};
// What the keys of a step are masked by: the lane's query sees keys lo … hi; every query of the tile sees all_lo …
// all_hi (uniform).
struct TileMask {
  int lo, hi, all_lo, all_hi;
};

// The products and the online softmax of one step (32 keys from key0) for one tile: kf(h, c) and vf(dt) are the step's
// MFMA fragments (16-key group h, 32-dim chunk c; 16-dim tile dt), ks and vs the scales of the lane's keys 16h + 4qd + i.
// Both kernels below run exactly this, so a row's bits do not depend on which of them a block takes.
template <int HD, typename KF, typename VF>
__device__ __forceinline__ void attn_step(TileState<HD>& st, const f16x8 (&qf)[HD / 32], const TileMask& mk, int key0,
                                          int qd, float sc, KF kf, const f32x4 (&ks)[2], const f32x4 (&vs)[2], VF vf) {
  // The fused multiply-adds are the written ones only.
#pragma clang fp contract(off)
  // Sᵀ of the two 16-key groups (keys as rows: lane (j, qd) gets keys 16h + 4qd + i of query j).
  f32x4 sa[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int c = 0; c < HD / 32; ++c)
#pragma unroll
    for (int h = 0; h < 2; ++h) sa[h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf(h, c), qf[c], sa[h], 0, 0, 0);
  // Online softmax in base 2. Scores stay in units of 1/scale: exp2(s·scale − m·scale) is one fused multiply-add and the
  // exponential.
  f32x4 sv[2] = {sa[0] * ks[0], sa[1] * ks[1]};
  if (!(key0 + STEP - 1 <= mk.all_hi && key0 >= mk.all_lo)) {  // uniform: some row does not see every key
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = key0 + 16 * h + 4 * qd + i;
        sv[h][i] = key <= mk.hi && key >= mk.lo ? sv[h][i] : -INFINITY;
      }
  }
  float mx = -INFINITY;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) mx = fmaxf(mx, sv[h][i]);
  mx = row_max4(mx);
  // The reference of a row's exponents is its first visible step's max, moved only when a later max passes it by RAISE
  // in log2 units: most steps then leave O as it is (a new max somewhere among 16 rows would rescale it nearly every
  // step). Weights stay ≤ 2^RAISE; times a V scale above 65504 / 2^RAISE one may pass the range of the fp16 product, and
  // the reduction then takes the row's split without it (split_in_fp32).
  const bool raise = mx * sc > fmaf(st.mrun, sc, RAISE) || st.mrun == -INFINITY;
  const float mnew = raise ? mx : st.mrun;
  const float alpha = raise && mnew != -INFINITY ? __builtin_amdgcn_exp2f((st.mrun - mnew) * sc) : 1.f;
  st.mrun = mnew;
  // A row that has seen no key yet takes exponents against 0, not −inf (exp2(−inf + inf) would be NaN).
  const float mref = mnew == -INFINITY ? 0.f : mnew * sc;
  float ps = 0.f;
  f16x8 pb;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // v_exp_f32 directly: exp2(−inf) = 0, and the arguments need no range reduction.
      const float pv = __builtin_amdgcn_exp2f(fmaf(sv[h][i], sc, -mref));
      ps += pv;
      // The product rounds to fp32 and then to fp16 wherever this is inlined (a fused conversion rounds once).
      float w = pv * vs[h][i];
      asm("" : "+v"(w));
      pb[4 * h + i] = (_Float16)w;
    }
  st.lsum = fmaf(st.lsum, alpha, ps);
  if (__any(raise)) {
#pragma unroll
    for (int dt = 0; dt < HD / 16; ++dt) st.o[dt] *= alpha;
  }
  // Oᵀ += Vᵀ·Pᵀ: a lane's eight keys of a dim are eight consecutive bytes of the block (v_index).
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt)
    st.o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf(dt), pb, st.o[dt], 0, 0, 0);
}

// Merge of the classes of tile lt of a workgroup and the split's output: every class's (reference, sum) per row through
// LDS, its O scaled by 2^(m − M) / L; then the 16-dim tile dt is added by class dt mod 3 (its own part first, then the
// following classes') and written. The order depends on the dim only. Every wave of the workgroup calls it (two
// barriers; `live`: the wave holds a tile). part: LDS for the other classes' parts, free of earlier readers.
template <int HD>
__device__ __forceinline__ void attn_merge(const AttnArgs& a, TileState<HD>& st, bool live, int kvh, int sidx, int cls,
                                           int lt, int m, int lane, float2 (*sml)[WTILES][16], f32x4 (*part)[64]) {
#pragma clang fp contract(off)
  constexpr int NDT = HD / 16;
  const int j = lane & 15, qd = lane >> 4, Q = a.G * a.B;
  const float sc = a.scale_log2;
  if (live) {
    float l = st.lsum;
    l += lane_xor<16>(l);
    l += lane_xor<32>(l);
    // A weight that overflowed leaves no dim of its row finite: any one tells. The NaN sum reaches the reduction; the
    // partial itself stays finite, for lanes of the reduction that read it in an idle place.
    if (!(fabsf(st.o[0][0]) < INFINITY)) {
      l = NAN;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) st.o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (qd == 0) sml[cls][lt][j] = make_float2(st.mrun, l);
  }
  __syncthreads();
  if (live) {
    float2 ml[NCLS];
    float M = -INFINITY, sum = 0.f;
#pragma unroll
    for (int c = 0; c < NCLS; ++c) {
      ml[c] = sml[c][lt][j];
      M = fmaxf(M, ml[c].x);
    }
#pragma unroll
    for (int c = 0; c < NCLS; ++c)
      sum += ml[c].x == -INFINITY ? 0.f : ml[c].y * __builtin_amdgcn_exp2f((ml[c].x - M) * sc);
    const float f = st.mrun == -INFINITY || !(sum > 0.f) ? 0.f : __builtin_amdgcn_exp2f((st.mrun - M) * sc) / sum;
    if (cls == 0 && qd == 0 && m < Q)
      a.ml[(size_t(kvh) * a.nsplit + sidx) * a.Qpad + m] = make_float2(M * sc, sum);
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      st.o[dt] *= f;
      const int k = (cls - dt % NCLS + NCLS) % NCLS;  // 0: this class adds the tile
      if (k != 0) part[(lt * NDT + dt) * (NCLS - 1) + k - 1][lane] = st.o[dt];
    }
  }
  __syncthreads();
  if (live) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) {
      if (dt % NCLS != cls) continue;  // uniform
      f32x4 v = st.o[dt];
#pragma unroll
      for (int k = 0; k < NCLS - 1; ++k) v += part[(lt * NDT + dt) * (NCLS - 1) + k][lane];
      if (m >= Q) continue;
      uint2 w;
      w.x = __builtin_bit_cast(unsigned, __floats2half2_rn(v[0], v[1]));
      w.y = __builtin_bit_cast(unsigned, __floats2half2_rn(v[2], v[3]));
      *reinterpret_cast<uint2*>(a.opart + ((size_t(kvh) * a.nsplit + sidx) * a.Qpad + m) * HD + 16 * dt + 4 * qd) = w;
    }
  }
}

// A wave's tile: its queries' fragments (chunk c of a lane's K bytes are dims 64·(c / 2) + 16·qd + 8·(c mod 2) …; q is
// read the same way), its masks and its empty state.
template <int HD>
__device__ __forceinline__ void attn_tile(const AttnArgs& a, int kvh, int P, int m0, int lane, f16x8 (&qf)[HD / 32],
                                          TileMask& mk, TileState<HD>& st) {
  const int j = lane & 15, qd = lane >> 4, m = m0 + j, Q = a.G * a.B;
#pragma unroll
  for (int c = 0; c < HD / 32; ++c)
    qf[c] = __builtin_bit_cast(
        f16x8, *reinterpret_cast<const u32x4*>(a.q + (size_t(kvh) * a.Qpad + min(m, a.Qpad - 1)) * HD + 64 * (c >> 1) +
                                               16 * qd + 8 * (c & 1)));
#pragma unroll
  for (int dt = 0; dt < HD / 16; ++dt) st.o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  st.mrun = -INFINITY;
  st.lsum = 0.f;
  mk.hi = m < Q ? P + m / a.G : -1;  // last visible key (causal); −1: a padding row sees nothing
  mk.lo = a.window > 0 ? mk.hi - a.window + 1 : -2147483647;
  // Up to the tile's first row's causal limit (none if it has padding rows), from its last row's window start.
  mk.all_hi = m0 + 15 < Q ? P + m0 / a.G : -1;
  mk.all_lo = a.window > 0 ? P + min(m0 + 15, Q - 1) / a.G - a.window + 1 : -2147483647;
}

// Keys of a split: its first key, the end, its steps and the rounds r0 … r1 − 1 of three steps (one per class) that are
// run. Steps are counted from the split's own first key. In a sliding-window layer every row's window starts at or after
// P − window + 1: the rounds wholly before it are masked for every row and left out.
struct SplitKeys {
  int kbase, k1, nsteps, r0, r1;
};
__device__ __forceinline__ SplitKeys split_keys(const AttnArgs& a, const AttnPos& ap, int sidx) {
  SplitKeys k;
  k.kbase = (sidx + ap.s0) * a.C;
  k.k1 = min(k.kbase + a.C, ap.P + a.B);
  k.nsteps = (k.k1 - k.kbase + STEP - 1) / STEP;
  k.r0 = a.window > 0 ? max(0, ap.P - a.window + 1 - k.kbase) / (STEP * NCLS) : 0;
  k.r1 = (k.nsteps + NCLS - 1) / NCLS;
  return k;
}

// Full blocks: one workgroup of 16 waves per (split of C keys, KV head, 80 query rows of the head's group), the keys
// shared through LDS.
template <int HD, bool RING>
__global__ __launch_bounds__(ATT_THREADS) void attn_kernel(AttnArgs a) {
  constexpr int NC = HD / 32;  // MFMA K steps of Sᵀ
  constexpr int NU = HD / 32;
  constexpr int UNITS = NCLS * 2 * NU, UPW = (UNITS + ATT_WAVES - 1) / ATT_WAVES;  // units of a round, per wave
  __shared__ AttnLds<HD> L;
  const AttnPos ap = attn_pos(a);
  // Grid (KV head, split): consecutive workgroup ids go round-robin over the 8 XCDs, so with 8 KV heads every split of
  // head h runs on XCD h and the head's queries are fetched into one L2 instead of all eight.
  const int sidx = blockIdx.y, kvh = blockIdx.x;
  if (sidx >= ap.nsplit) return;  // launched for a later position than the step's (chained rounds): no keys
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int qd = lane >> 4;
  const SplitKeys sk = split_keys(a, ap, sidx);
  const size_t hrow = size_t(kvh) * a.vld;

  // Wave w < 15 multiplies tile w mod 5 over the steps of class w / 5. Its queries are requested ahead of the keys: the
  // wait for the first round then covers them.
  const int lt = wave % WTILES, cls = wave / WTILES;
  const int m0 = 16 * (WTILES * int(blockIdx.z) + lt);
  const bool live = cls < NCLS && m0 < a.G * a.B;  // uniform
  f16x8 qf[NC];
  TileMask mk;
  TileState<HD> st;
  attn_tile<HD>(a, kvh, ap.P, m0, lane, qf, mk, st);

  // Staging: a round's cache bytes go out one 1 KB unit (16 bytes per lane) at a time over the 16 waves, unit u = (step
  // u / 2NU, K or V, unit); the last six waves read the steps' scales. Steps past the last are read as the last one.
  // Every wave issues the same buffer loads without a branch (an offset out of range reads as zero and touches no
  // memory), so that the compiler's wait counts cover exactly one round.
  struct Stage {
    u32x4 b[UPW];
    unsigned short s;
  };
  __amdgpu_buffer_rsrc_t rkv[UPW];
  unsigned ukv[UPW];
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    const int u = wave + ATT_WAVES * i;
    rkv[i] = make_rsrc(((u / NU) & 1 ? a.vc : a.kc) + hrow * HD, unsigned(a.vld) * HD);
    ukv[i] = u < UNITS ? unsigned((lane & 15) * 64 + qd * 16) : OOB;
  }
  const int scu = wave - (ATT_WAVES - 2 * NCLS);  // scale unit of the last waves: (class, K or V)
  const __amdgpu_buffer_rsrc_t rsc = make_rsrc(((scu & 1) ? a.vs : a.ks) + hrow, unsigned(a.vld) * 2);
  const int ring = a.ring;
  auto slot_of = [&](int r, int c) {
    const int key = sk.kbase + STEP * min(NCLS * r + c, sk.nsteps - 1);
    return RING ? key % ring : key;
  };
  auto load = [&](Stage& g, int r) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
      const int u = min(wave + ATT_WAVES * i, UNITS - 1);
      g.b[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rkv[i], ukv[i], slot_of(r, u / (2 * NU)) * HD + (u % NU) * 1024, 0));
    }
    g.s = __builtin_amdgcn_raw_buffer_load_b16(rsc, scu >= 0 && lane < STEP ? unsigned(lane) * 2u : OOB,
                                               slot_of(r, max(scu, 0) >> 1) * 2, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto store = [&](const Stage& g, int r, int buf) {
#pragma unroll
    for (int i = 0; i < UPW; ++i) {
      const int u = wave + ATT_WAVES * i, c = u / (2 * NU), kv = (u / NU) & 1;
      if (u < UNITS) {
        // K: a 16-key group's 64-dim half is two 32-dim chunks; V: a 32-dim pair is two 16-dim tiles.
        L.kv[buf][c][kv][2 * (u % NU)][lane] = u8x8_to_f16(g.b[i][0], g.b[i][1]);
        L.kv[buf][c][kv][2 * (u % NU) + 1][lane] = u8x8_to_f16(g.b[i][2], g.b[i][3]);
      }
    }
    if (scu >= 0 && lane < STEP) {
      // Keys past the split's end may hold anything: their scores are masked and their scales zeroed, so that
      // 0 · scale stays 0.
      const bool ok = sk.kbase + STEP * (NCLS * r + (scu >> 1)) + lane < sk.k1;
      L.sc[buf][scu >> 1][scu & 1][lane] = ok ? __half2float(__ushort_as_half(g.s)) : 0.f;
    }
  };
  auto multiply = [&](int r, int buf) {
    const int s = NCLS * r + cls;
    if (!live || s >= sk.nsteps) return;  // uniform
    f32x4 ks[2], vs[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ks[h] = *reinterpret_cast<const f32x4*>(&L.sc[buf][cls][0][16 * h + 4 * qd]);
      vs[h] = *reinterpret_cast<const f32x4*>(&L.sc[buf][cls][1][16 * h + 4 * qd]);
    }
    attn_step<HD>(
        st, qf, mk, sk.kbase + STEP * s, qd, a.scale_log2,
        [&](int h, int c) { return __builtin_bit_cast(f16x8, L.kv[buf][cls][0][h * NC + c][lane]); }, ks, vs,
        [&](int dt) { return __builtin_bit_cast(f16x8, L.kv[buf][cls][1][dt][lane]); });
  };

  // Round r is multiplied from buffer (r − r0) mod 2 while round r + 1 is converted into the other one (last read in
  // round r − 1, before its barrier) and rounds r + 2 and r + 3 are on their way.
  Stage sg[2];
  load(sg[0], sk.r0);
  load(sg[1], sk.r0 + 1);
  store(sg[0], sk.r0, 0);
  load(sg[0], sk.r0 + 2);
  __syncthreads();
  for (int r = sk.r0; r < sk.r1; r += 2) {
    if (r + 1 < sk.r1) store(sg[1], r + 1, 1);
    load(sg[1], r + 3);
    multiply(r, 0);
    __syncthreads();
    if (r + 1 >= sk.r1) break;
    if (r + 2 < sk.r1) store(sg[0], r + 2, 0);
    load(sg[0], r + 4);
    multiply(r + 1, 1);
    __syncthreads();
  }
  attn_merge<HD>(a, st, live, kvh, sidx, cls, lt, m0 + (lane & 15), lane, L.ml, L.part());
}

// Small blocks: one workgroup per (split, KV head, FEW tiles), three waves per tile, one per class, each reading its steps'
// cache bytes straight into the MFMA operand registers: no staging, no barrier before the merge. One row at 611
// positions: 4.6 µs against 7.7 in the kernel above, whose 16 waves mostly stage. More tiles read and convert every byte
// once per FEW of them; that wins as long as the launch is one workgroup per CU at most, since one of the kernel above
// then leaves CUs idle or is mostly latency (8 heads per KV head, 4 KV heads of 128, 8 rows: 1000 positions 57.8 → 55.2 µs
// a layer, 16000 65.2 → 62.2; 12 rows at 1000 65.3 → 62.2, at 2000 in 64-key splits, three workgroups for two CUs, 65.9 → 66.2).
constexpr int FEW = 2;
template <int HD, bool RING>
__global__ __launch_bounds__(64 * NCLS * FEW) void attn_few_kernel(AttnArgs a) {
  constexpr int NC = HD / 32, NU = HD / 32, NH = HD / 64;
  __shared__ f32x4 part[FEW * (HD / 16) * (NCLS - 1)][64];
  __shared__ float2 sml[NCLS][WTILES][16];
  const AttnPos ap = attn_pos(a);
  const int sidx = blockIdx.y, kvh = blockIdx.x;  // as in attn_kernel
  if (sidx >= ap.nsplit) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int qd = lane >> 4, lt = wave / NCLS, cls = wave % NCLS, m0 = 16 * (FEW * int(blockIdx.z) + lt);
  const bool live = m0 < a.G * a.B;  // uniform
  const SplitKeys sk = split_keys(a, ap, sidx);
  const size_t hrow = size_t(kvh) * a.vld;
  const unsigned l16 = unsigned(lane & 15) * 64u + unsigned(qd) * 16u;
  const int ring = a.ring;
  uint4 kr[NU], vr[NU];
  uint2 sr[2][2], sn[2][2];  // [K, V][16-key group]: the scales of the lane's four keys
  auto slot_of = [&](int s) {
    const int key = sk.kbase + STEP * min(s, sk.nsteps - 1);
    return RING ? key % ring : key;
  };
  auto load_k = [&](int s, uint2 (&d)[2][2]) {
    const int slot = slot_of(s);
    const uint8_t* p = a.kc + (hrow + slot) * HD;
#pragma unroll
    for (int i = 0; i < NU; ++i) kr[i] = *reinterpret_cast<const uint4*>(p + i * 1024 + l16);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      d[0][h] = *reinterpret_cast<const uint2*>(a.ks + hrow + slot + 16 * h + 4 * qd);
      d[1][h] = *reinterpret_cast<const uint2*>(a.vs + hrow + slot + 16 * h + 4 * qd);
    }
  };
  auto load_v = [&](int s) {
    const uint8_t* p = a.vc + (hrow + slot_of(s)) * HD;
#pragma unroll
    for (int i = 0; i < NU; ++i) vr[i] = *reinterpret_cast<const uint4*>(p + i * 1024 + l16);
  };
  f16x8 qf[NC];
  TileMask mk;
  TileState<HD> st;
  int s = NCLS * sk.r0 + cls;
  load_k(s, sr);
  attn_tile<HD>(a, kvh, ap.P, m0, lane, qf, mk, st);
  load_v(s);
  for (; live && s < sk.nsteps; s += NCLS) {
    const int key0 = sk.kbase + STEP * s;
    f32x4 sc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned w = i < 2 ? sr[x][h].x : sr[x][h].y;
          const float f = __half2float(__ushort_as_half((unsigned short)(w >> (16 * (i & 1)))));
          sc[x][h][i] = key0 + 16 * h + 4 * qd + i < sk.k1 ? f : 0.f;  // keys past the end: see attn_kernel
        }
    f16x8 kf[2][NC];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const uint4& w = kr[h * NH + (c >> 1)];
        kf[h][c] = __builtin_bit_cast(f16x8, (c & 1) ? u8x8_to_f16(w.z, w.w) : u8x8_to_f16(w.x, w.y));
      }
    load_k(s + NCLS, sn);
    attn_step<HD>(
        st, qf, mk, key0, qd, a.scale_log2, [&](int h, int c) { return kf[h][c]; }, sc[0], sc[1],
        [&](int dt) {
          const uint4& w = vr[dt >> 1];
          return __builtin_bit_cast(f16x8, (dt & 1) ? u8x8_to_f16(w.z, w.w) : u8x8_to_f16(w.x, w.y));
        });
    load_v(s + NCLS);
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int h = 0; h < 2; ++h) sr[x][h] = sn[x][h];
  }
  attn_merge<HD>(a, st, live, kvh, sidx, cls, lt, m0 + (lane & 15), lane, sml, part);
}

// ---------------------------------------------------------------------------------------------------------------
// One row's split again, by a whole wave: softmax over its visible keys in fp32 with weights of at most 1, for rows whose
// weights times V scales passed fp16 in the kernels above (their limit would otherwise be a sixteenth of what the cache
// holds: values of 5e5). O / l in fp16 as those write it, the lane's eight dims 8dg … in raw; returns (reference, sum).
// A test of the scales in every step instead, or a second pass inside those kernels, cost 0.5 to 1 % of a step's time;
// this costs nothing measurable (dense, 17 rows at 8K: 2238 µs a step with and without).
template <int HD>
__device__ __forceinline__ float2 split_in_fp32(const AttnArgs& a, int kvh, int m, int sidx, int lane, int dg, uint4& raw) {
  constexpr int NE = HD / 64;
  const AttnPos ap = attn_pos(a);
  const SplitKeys sk = split_keys(a, ap, sidx);
  const int row = ap.P + m / a.G;
  const int k0 = max(sk.kbase, a.window > 0 ? row - a.window + 1 : 0), k1 = min(sk.k1, row + 1);
  float q[NE], o[NE], M = -INFINITY, l = 0.f;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    q[e] = __half2float(a.q[(size_t(kvh) * a.Qpad + m) * HD + lane + 64 * e]);
    o[e] = 0.f;
  }
  for (int key = k0; key < k1; ++key) {
    const int slot = a.ring ? key % a.ring : key;
    const size_t hs = size_t(kvh) * a.vld + slot;
    float s = 0.f;
#pragma unroll
    for (int e = 0; e < NE; ++e) s = fmaf(q[e], float(a.kc[k_index(kvh, slot, lane + 64 * e, HD, a.vld)]) - 128.f, s);
    s += lane_xor<32>(s);
    s += lane_xor<16>(s);
    s += lane_xor<8>(s);
    s += lane_xor<4>(s);
    s += lane_xor<2>(s);
    s += lane_xor<1>(s);
    s *= __half2float(a.ks[hs]) * a.scale_log2;
    const float Mn = fmaxf(M, s), c = M == -INFINITY ? 0.f : exp2f(M - Mn), p = Mn == -INFINITY ? 0.f : exp2f(s - Mn);
    const float w = p * __half2float(a.vs[hs]);
    l = fmaf(l, c, p);
#pragma unroll
    for (int e = 0; e < NE; ++e)
      o[e] = fmaf(w, float(a.vc[v_index(kvh, slot, lane + 64 * e, HD, a.vld)]) - 128.f, o[e] * c);
    M = Mn;
  }
  unsigned h[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int d = 8 * dg + i;
    float v = __shfl(o[0], d & 63);
    if constexpr (NE == 2) {
      const float v1 = __shfl(o[1], d & 63);
      v = d >= 64 ? v1 : v;
    }
    h[i] = __half_as_ushort(__float2half_rn(l > 0.f ? v / l : 0.f));
  }
  raw = make_uint4(h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16);
  return make_float2(M, l);
}

// Reduction of the splits (vattn_reduce, verify_attn.metal:149-192): M = max over splits (and the sink), L = Σ e^(m−M)·l
// (+ e^(sink−M)), o = Σ e^(m−M)·l·ō / L with ō = O/l the split's normalised partial; written into the o_proj
// activation layout (column h·HD + d). One wave per (row, q head): lane = (split group sg, 8-dim group dg); a lane
// merges splits sg, sg + SG, … in batches of NB whose loads are all issued before any is used (a load per trip of a
// runtime loop would wait out a memory latency per split), keeping a running (M, L, o) rescaled per batch; then the
// SG groups are merged by a fixed butterfly. Grid (B, QH/w), 64·w threads (w = 1 by default).
template <int HD>
__global__ __launch_bounds__(64) void attn_reduce_kernel(AttnArgs a, uint4* __restrict__ frag, int nkb, int ntile) {
  constexpr int DG = HD / 8, SG = 64 / DG, NB = 8;
  static_assert(DG == 8 || DG == 16, "the split-group merge below runs the stages 8/16/32 of HD 64 and 128");
  // Grid (KVH, B·G), one wave per workgroup: workgroup (kvh, j) merges q head kvh·G + j mod G of token j / G, on the
  // XCD where that KV head's splits ran and wrote their partials (consecutive workgroup ids go round-robin over the 8
  // XCDs; the attention grid is (KV head, split)).
  const int kvh = blockIdx.x, t = int(blockIdx.y) / a.G, h = kvh * a.G + int(blockIdx.y) % a.G;
  const int lane = threadIdx.x & 63;
  const int dg = lane % DG, sg = lane / DG;
  const int m = t * a.G + h % a.G;
  float M = -INFINITY, L = 0.f;
  float o[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = 0.f;
  const int nsplit = attn_pos(a).nsplit;
  for (int s0 = sg; s0 < nsplit; s0 += NB * SG) {
    float2 v[NB];
    uint4 raw[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int s = s0 + i * SG;
      const bool ok = s < nsplit;
      const size_t idx = (size_t(kvh) * a.nsplit + (ok ? s : 0)) * a.Qpad + m;
      v[i] = a.ml[idx];
      raw[i] = *reinterpret_cast<const uint4*>(a.opart + idx * HD + 8 * dg);
      if (!ok) v[i].x = -INFINITY;  // an empty split (m = −inf, l = 0) has weight 0
    }
    float Mb = M;
#pragma unroll
    for (int i = 0; i < NB; ++i) Mb = fmaxf(Mb, v[i].x);
    const float ca = M == -INFINITY ? 0.f : exp2f(M - Mb);
    L *= ca;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= ca;
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const float w = v[i].x == -INFINITY ? 0.f : exp2f(v[i].x - Mb) * v[i].y;
      L += w;
      const unsigned rw[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float2 f = __half22float2(__builtin_bit_cast(__half2, rw[e]));
        o[2 * e] += w * f.x;
        o[2 * e + 1] += w * f.y;
      }
    }
    M = Mb;
  }
  // Merge the split groups (lanes dg + DG·sg): butterfly over sg, fixed order.
  auto merge = [&](auto xc) {
    constexpr int X = decltype(xc)::value;
    const float Mo = lane_xor<X>(M), Lo = lane_xor<X>(L);
    const float Mn = fmaxf(M, Mo);
    const float ca = M == -INFINITY ? 0.f : exp2f(M - Mn), cb = Mo == -INFINITY ? 0.f : exp2f(Mo - Mn);
    L = L * ca + Lo * cb;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float oo = lane_xor<X>(o[e]);
      o[e] = o[e] * ca + oo * cb;
    }
    M = Mn;
  };
  if constexpr (DG <= 8) merge(std::integral_constant<int, 8>{});
  merge(std::integral_constant<int, 16>{});
  merge(std::integral_constant<int, 32>{});
  if (__builtin_expect(__any(L != L), 0)) {
    // Some split's weights overflowed: the row once more, that split in fp32, the splits in order. The arguments are read
    // again here from the kernel's argument segment, which they head: hoisted, their loads cost every launch 0.2 µs.
    const AttnArgs* ac = (const AttnArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(ac));
    M = -INFINITY;
    L = 0.f;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
    for (int s = 0; s < nsplit; ++s) {
      const size_t idx = (size_t(kvh) * a.nsplit + s) * a.Qpad + m;
      float2 f = a.ml[idx];
      uint4 raw = *reinterpret_cast<const uint4*>(a.opart + idx * HD + 8 * dg);
      if (f.y != f.y) f = split_in_fp32<HD>(*ac, kvh, m, s, lane, dg, raw);  // uniform
      if (f.x == -INFINITY) continue;
      const float Mn = fmaxf(M, f.x), c = M == -INFINITY ? 0.f : exp2f(M - Mn), w = exp2f(f.x - Mn) * f.y;
      const unsigned rw[4] = {raw.x, raw.y, raw.z, raw.w};
      L = L * c + w;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float2 h = __half22float2(__builtin_bit_cast(__half2, rw[e >> 1]));
        o[e] = o[e] * c + w * ((e & 1) ? h.y : h.x);
      }
      M = Mn;
    }
  }
  if (sg != 0) return;
  // The sink is a last split with weight e^(sink−M) and no value, merged after the splits' tree so that its place
  // does not depend on which split a window starts in (the same bits for a row whatever the block's P).
  if (a.sinks) {
    const float ms = a.sinks[h] * 1.4426950408889634f;
    const float Mn = fmaxf(M, ms);
    const float ca = M == -INFINITY ? 0.f : exp2f(M - Mn);
    L = L * ca + exp2f(ms - Mn);
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= ca;
  }
  const float inv = L > 0.f ? 1.0f / L : 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= inv;
  if (a.QS != HD) {
    // Gated attention (AT_GATED): × sigmoid(gate), the gate being the second half of the q head's projection.
    const float* g = a.proj + size_t(t) * a.ldp + size_t(h) * a.QS + HD + 8 * dg;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] *= 1.0f / (1.0f + expf(-g[e]));
  }
  frag_store_chunk(frag, nkb, ntile, t, (h * HD) / 8 + dg, o);
}

int launch_prework(ih_ctx* c, const AttnArgs& a) {
  TimedLaunch tl(c, TC_PREWORK, double(a.B) * (a.QH + 2 * a.KVH) * a.HD * 4 + double(a.B) * a.KVH * (2 * a.HD + 4) +
                                    double(a.B) * a.QH * a.HD * 2);
  // One wave (one (head slot, token)) per workgroup (config 1: 2.306 against 2.312 ms per step with four).
  IH_CHECK(a.QH == a.G * a.KVH, IH_EINVAL, "attention prework: q heads must be G per KV head");
  const dim3 grid(a.KVH, (a.G + 2) * a.B);
  if (a.HD == 128) tlaunch(tl, prework_kernel<128>, grid, dim3(64), 0, c->stream, a);
  else if (a.HD == 64) tlaunch(tl, prework_kernel<64>, grid, dim3(64), 0, c->stream, a);
  else return fail(IH_EINVAL, "attention prework: head_dim must be 64 or 128");
  IH_HIP(hipGetLastError());
  return IH_OK;
}

int launch_attention(ih_ctx* c, const AttnArgs& a) {
  const int Q = a.G * a.B;
  const int qtiles = (Q + 15) / 16;
  IH_CHECK(qtiles <= 16, IH_EINVAL, "attention: at most 256 query rows per KV head");
  IH_CHECK(a.C > 0 && a.C % STEP == 0, IH_EINVAL, "attention: unsupported key chunk");
  IH_CHECK(size_t(a.vld) * a.HD < (size_t(1) << 31), IH_EINVAL, "attention: a KV head's cache must be below 2 GiB");
  const bool few = qtiles <= FEW || a.KVH * a.nsplit * ((qtiles + FEW - 1) / FEW) <= c->cu_count, ring = a.ring != 0;
  const int per = few ? FEW : WTILES;
  const dim3 grid(a.KVH, a.nsplit, (qtiles + per - 1) / per);
  const dim3 block(few ? 64 * NCLS * std::min(FEW, qtiles) : ATT_THREADS);
  // Algorithmic bytes: the int8 K and V and their fp16 scales of every key the launched splits cover, and q.
  const double keys = double(a.P + a.B) - double(a.s0) * a.C;
  TimedLaunch tl(c, TC_ATTN, double(a.KVH) * keys * (2 * a.HD + 4) + double(a.KVH) * Q * a.HD * 2);
  auto run = [&](auto hd, auto rg) {
    constexpr int HD = decltype(hd)::value;
    constexpr bool RG = decltype(rg)::value;
    tlaunch(tl, few ? attn_few_kernel<HD, RG> : attn_kernel<HD, RG>, grid, block, 0, c->stream, a);
  };
  using I128 = std::integral_constant<int, 128>;
  using I64 = std::integral_constant<int, 64>;
  if (a.HD == 128) ring ? run(I128{}, std::true_type{}) : run(I128{}, std::false_type{});
  else if (a.HD == 64) ring ? run(I64{}, std::true_type{}) : run(I64{}, std::false_type{});
  else return fail(IH_EINVAL, "attention: head_dim must be 64 or 128");
  IH_HIP(hipGetLastError());
  return IH_OK;
}

int launch_attn_reduce(ih_ctx* c, const AttnArgs& a, ActBuf& out) {
  TimedLaunch tl(c, TC_REDUCE, double(a.KVH) * a.nsplit * a.G * a.B * (2 * a.HD + 8) + double(a.B) * a.QH * a.HD * 2);
  // One wave (one (row, q head)) per workgroup: B·QH small workgroups spread over more CUs than four-wave ones
  // (config 1: 0.146 against 0.149 ms per step).
  IH_CHECK(a.QH == a.G * a.KVH, IH_EINVAL, "attention reduce: q heads must be G per KV head");
  const dim3 grid(a.KVH, a.B * a.G);
  uint4* of = static_cast<uint4*>(out.frag);
  if (a.HD == 128) tlaunch(tl, attn_reduce_kernel<128>, grid, dim3(64), 0, c->stream, a, of, out.nkb, out.ntile);
  else if (a.HD == 64) tlaunch(tl, attn_reduce_kernel<64>, grid, dim3(64), 0, c->stream, a, of, out.nkb, out.ntile);
  else return fail(IH_EINVAL, "attention reduce: head_dim must be 64 or 128");
  IH_HIP(hipGetLastError());
  return IH_OK;
}

}  // namespace ih
