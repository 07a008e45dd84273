// The few-row int4 product kernel, its epilogues and its launch by shape, instantiated by qmm.hip (activations in the
// fragment layout, the round's fused epilogues) and qmm_rows.hip (bf16 rows as the caller holds them). See qmm.hip.
#pragma once
#include "act.h"
#include "ih_internal.h"
#include "qmm_common.h"

namespace ih {

// ---------------------------------------------------------------------------------------------------------------
struct QmmParams {
  const uint4* w;          // packed words of the expert
  const uint2* s;          // packed scale/bias of the expert
  const uint4* xa;         // activation fragments, or (XN) bf16 rows of ldx elements
  int ldx, K;              // XN
  void* y;
  int ldy, M, N, Npad, nkb;
  // The nibble-decode constants 0x000F000F and 0x43004300, passed as arguments so that they live in SGPRs and the
  // compiler can use the three-operand v_and_or_b32 (gfx9 VOP3 takes no literal constants).
  unsigned kmask, kbias;
  // RMSNorm factor of the input rows (modes QM_F32_SCALE, QM_GLU_ACT): r_t = 1/sqrt(Σ ss_in[t][j] / D + eps).
  const float* ss_in;
  int nss_in, D;
  float eps;
  // QM_RESID_ACT: h[m][n] += v (fp32, the y pointer), then the next activation bf16(h ⊙ nw) and the sum-of-squares
  // partial of this workgroup's columns, ss_out[t][blockIdx.x].
  const uint16_t* nw;
  const float* bias;  // QM_RESID_ACT: h += v + bias[n] when not null
  uint4* act_out;
  int act_nkb;
  float* ss_out;
  // QM_GLU_ACT: gated activation kind and clip.
  int glu;
  float limit;
  int act_f16;  // the next activation in fp16 (the input of MXFP4 experts) instead of bf16
  // K split over workgroups (gridDim.y > 1): partial sums [split][MAX_TOK][Npad], added in split order by the last
  // workgroup of a row group to arrive, which runs the epilogue; arrival counters, one per row group (zero between
  // launches).
  float* part;
  unsigned* ctr;
};

// The epilogue of the R tiles tile0 … tile0+R−1 of a workgroup of nthr threads, given val(m, r, rn) = the finished
// product of token m and row rn of tile r. rsc holds the RMSNorm factors (modes QM_F32_SCALE, QM_GLU_ACT); ssu is
// LDS scratch of MAX_TOK·2R floats; wg indexes this workgroup's sum-of-squares partial (QM_RESID_ACT).
// QM_RESID_ACT: a thread's first work item (token m, 8 columns) of the residual epilogue, its h and norm weights
// loaded at kernel entry so that their latency overlaps the main loop.
struct ResidPrefetch {
  float h[8];
  float nw[8];
};
template <int R>
__device__ __forceinline__ void resid_prefetch(ResidPrefetch& pf, const QmmParams& p, int tile0) {
  constexpr int nch = 2 * R;
  const int u = threadIdx.x;
  if (u >= p.M * nch) return;
  const int m = u / nch, cl = u % nch, col0 = (tile0 + (cl >> 1)) * 16 + 8 * (cl & 1);
  const float* hrow = static_cast<const float*>(p.y) + size_t(m) * p.ldy;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int col = min(col0 + j, p.N - 1);
    pf.h[j] = hrow[col];
    pf.nw[j] = bf16f(p.nw[col]);
  }
}

template <int R, int MODE, typename V>
__device__ __forceinline__ void qmm_epilogue(const QmmParams& p, int tile0, V val, const float* rsc, float* ssu,
                                             int nthr, int wg, const ResidPrefetch* rpf = nullptr) {
  if constexpr (MODE == QM_RESID_ACT) {
    // h += v for the 16R columns, the next activation bf16(h ⊙ nw) in 8-column chunks, and Σh² per token.
    constexpr int nch = 2 * R;
    for (int u = threadIdx.x; u < p.M * nch; u += nthr) {
      const int m = u / nch, cl = u % nch, r = cl >> 1, half = cl & 1;
      const int col0 = (tile0 + r) * 16 + 8 * half;
      const bool pre = rpf && u == int(threadIdx.x);
      float v[8], ss = 0.f;
      float* hrow = static_cast<float*>(p.y) + size_t(m) * p.ldy;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int col = col0 + j;
        float hv = 0.f;
        if (col < p.N) {
          hv = (pre ? rpf->h[j] : hrow[col]) + (p.bias ? val(m, r, 8 * half + j) + p.bias[col] : val(m, r, 8 * half + j));
          hrow[col] = hv;
        }
        ss += hv * hv;
        v[j] = col < p.N ? hv * (pre ? rpf->nw[j] : bf16f(p.nw[col])) : 0.f;
      }
      ssu[m * nch + cl] = ss;
      if (col0 < p.N) frag_store(p.act_f16 != 0, p.act_out, p.act_nkb, MAX_TOK / 16, m, col0 / 8, v);
    }
    __syncthreads();
    if (int(threadIdx.x) < p.M) {
      float ss = 0.f;
      for (int cl = 0; cl < nch; ++cl) ss += ssu[threadIdx.x * nch + cl];
      p.ss_out[threadIdx.x * SS_CAP + wg] = ss;
    }
    return;
  }
  if constexpr (MODE == QM_GLU_ACT) {
    // Interleaved gate|up tiles: rows 0–7 gate, 8–15 up of the same 8 columns (chunk tile0 + r of the output).
    for (int u = threadIdx.x; u < p.M * R; u += nthr) {
      const int m = u / R, r = u % R;
      const float rs_ = rsc[m];
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = glu_f(val(m, r, j) * rs_, val(m, r, 8 + j) * rs_, p.glu, p.limit);
      const int chunk = tile0 + r;
      if (chunk * 8 < p.N / 2) frag_store(p.act_f16 != 0, p.act_out, p.act_nkb, MAX_TOK / 16, m, chunk, v);
    }
    return;
  }
  for (int u = threadIdx.x; u < p.M * 16 * R; u += nthr) {
    const int m = u / (16 * R), rr = u % (16 * R), r = rr >> 4, rn = rr & 15;
    const int row = (tile0 + r) * 16 + rn;
    if (row >= p.N) continue;
    float v = val(m, r, rn);
    if constexpr (MODE == QM_F32_SCALE) v *= rsc[m];
    if constexpr (MODE == QM_BF16) {
      static_cast<unsigned short*>(p.y)[size_t(m) * p.ldy + row] = f2bf(v);
    } else if constexpr (MODE == QM_F32_ADD) {
      float* o = static_cast<float*>(p.y) + size_t(m) * p.ldy + row;
      *o = *o + v;
    } else {
      static_cast<float*>(p.y)[size_t(m) * p.ldy + row] = v;
    }
  }
}

// Eight consecutive bf16 values → the fragment's element order {0,4,1,5,2,6,3,7}.
__device__ __forceinline__ u32x4 frag_order(const u32x4& v) {
  return u32x4{__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
               __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
}

// T: MFMA token tiles loaded from memory (tokens 0–15, and 16–31 when T = 2); X16 (with T = 1, M = 17): token 16 as
// a second tile whose A operand comes from LDS.
//
// Workgroup (blockIdx.x, blockIdx.y) = KW waves over the 16·R rows of tiles R·blockIdx.x …; the K range is split over
// gridDim.y workgroups and, inside one, over its waves: wave w streams the KPW consecutive K-blocks from
// (blockIdx.y·KW + w)·KPW through a D-deep register ring (the loads of K-block i + D go out as K-block i is
// multiplied). R tiles per wave share each x fragment, so x traffic per weight byte falls as 1/R (one tile per wave
// re-reads x ~4× the weight bytes from L2).
// VALU budget. At M = 17 the products are cheap on MFMA; the VALU work per 16 × 128 tile (nibble decode 28, the
// per-group affine map 20, scale words 6) is ~55 % of the tile's HBM time at full speed, so nothing else may run on
// the VALU in the loop: every K-dependent offset is a scalar (buffer loads take the K-block as soffset, the LDS reads
// as an immediate of an unrolled trip), and the ring's last D K-blocks are peeled rather than guarded.
// The KW partial sums are added in wave order through LDS; with gridDim.y > 1 the last workgroup of a row group to arrive
// adds the splits in order. A row's summation order depends only on (N, K), never on M.
// KPW1 > 0: the second half of the waves (the second wave of each SIMD at KW = 8) take KPW1 K-blocks each instead of
// KPW. A CU's loads come back roughly in issue order, so those waves receive their first stage after the first half's
// first two stages; with fewer K-blocks they still end with the first half.
// XN: the activations are the caller's bf16 rows (16-byte aligned), permuted to the fragment order with four v_perm_b32
// per MFMA step as they are used; a step past K reads as zero. A separate launch that rearranged them cost more than the
// product of a small matrix (8 × 4096 × 4096: 3.6 + 4.7 µs). With gridDim.z = 2 (T = 1, more than 17 rows) workgroup z
// takes rows 16z … as a product of its own, with its own partial sums and arrival counts. RAG: see QmmShape.
template <int T, int R, int KW, bool X16, int D, int KPW, int MODE, int KPW1 = 0, bool XN = false, bool RAG = false>
__global__ __launch_bounds__(64 * KW) void qmm_int4_kernel(QmmParams p) {
  if constexpr (XN && T == 1 && !X16) {
    if (gridDim.z > 1) {
      const int z = int(blockIdx.z);
      p.xa = reinterpret_cast<const uint4*>(reinterpret_cast<const uint16_t*>(p.xa) + size_t(16 * z) * p.ldx);
      p.y = static_cast<char*>(p.y) + size_t(16 * z) * p.ldy * (MODE == QM_BF16 ? 2 : 4);
      p.M = min(16, p.M - 16 * z);
      if (gridDim.y > 1) {
        p.part += size_t(16 * z) * p.Npad;
        p.ctr += z * int(gridDim.x);
      }
    }
  }
  static_assert(KPW % D == 0 && KPW1 % D == 0, "the ring depth divides the K-blocks of a wave");
  // The wave index is uniform: readfirstlane keeps it (and everything derived from it) in scalar registers.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n = lane & 15, qd = lane >> 4;
  const int tile0 = blockIdx.x * R;
  constexpr int nk = KPW;                                // K-blocks of a wave of the first half (the LDS stride)
  constexpr int HALF = KW / 2;
  const int nkr = (KPW1 == 0 || wave < HALF) ? KPW : KPW1;  // K-blocks of this wave
  const int kwg = int(blockIdx.y) * (KPW1 ? HALF * (KPW + KPW1) : KW * nk);  // first K-block of the workgroup
  const int kb0 = kwg + (KPW1 == 0 ? wave * nk : wave < HALF ? wave * KPW : HALF * KPW + (wave - HALF) * KPW1);
  const unsigned tiles_total = unsigned(p.Npad / 16) * unsigned(p.nkb);
  const unsigned wlim = tiles_total * 1024u;
  const unsigned xlim = XN ? (unsigned(p.M - 1) * unsigned(p.ldx) + unsigned(p.K)) * 2u : unsigned(MAX_TOK) * p.nkb * 256u;
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(p.w, wlim), rsb = make_rsrc(p.s, tiles_total * 128u),
                               rx = make_rsrc(p.xa, xlim);
  const unsigned km = vgpr_of(p.kmask), kbias = p.kbias;
  const unsigned shv[3] = {vgpr_of(4u), vgpr_of(8u), vgpr_of(12u)};  // 64-bit nibble shifts (nib_bf16_pair)

  // Epilogue inputs that another kernel just wrote, requested ahead of the weight stages (consumed after the main loop).
  // Rows per wave of the RMSNorm prefetch: M ≤ 16 (T = 1), 17 (X16) or 32 (T = 2); more than eight (one-wave
  // workgroups) are read after the loop instead.
  constexpr int NR = ((T == 2 ? 32 : X16 ? 17 : 16) + KW - 1) / KW;
  constexpr bool RMS = MODE == QM_F32_SCALE || MODE == QM_GLU_ACT, RMS_PRE = RMS && NR <= 8;
  RmsPrefetch<RMS_PRE ? NR : 1> rpf;
  ResidPrefetch hpf;
  unsigned xoff[T];
#pragma unroll
  for (int tt = 0; tt < T; ++tt)
    xoff[tt] = 16 * tt + n >= p.M ? OOB
               : XN ? unsigned(16 * tt + n) * unsigned(p.ldx) * 2u + qd * 16u
                    : unsigned(tt) * 4096u + n * 64u + qd * 16u;
  // XN: the offset bit that makes step t of K-block kb read as zero past K (K is a multiple of 64).
  auto past_k = [&](int kb, int t) { return XN && kb * KBLK + 32 * t >= p.K ? OOB : 0u; };
  const unsigned woff = unsigned(lane) * 16u;

  u32x4 wv[D][R], xv[D][T][4];
  // One ring stage: the weight tiles and x of K-block kb. Every offset that depends on kb is a scalar.
  auto load_stage = [&](int d, int kb) {
    kb = kb < p.nkb ? kb : p.nkb - 1;  // a ragged last wave re-reads the last K-block; its scales are zero
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tt = 0; tt < T; ++tt)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        xv[d][tt][t] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       rx, xoff[tt] | past_k(kb, t), XN ? kb * (2 * KBLK) + 64 * t : kb * (MAX_TOK / 16) * 4096 + 1024 * t, 0));
#pragma unroll
    for (int r = 0; r < R; ++r)
      wv[d][r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                               rw, woff, ((tile0 + r) * p.nkb + kb) * 1024, 0));
    __builtin_amdgcn_sched_barrier(0);
  };
  // With the asymmetric split (two waves per SIMD), every wave's first stage goes out before anything else of the
  // workgroup: a CU's loads come back roughly in issue order at its share of the bandwidth, and the second half's
  // first stages would otherwise queue behind the first half's staging loads and second stages. The barrier orders
  // only the issue. (With one wave per SIMD the staging loads go first: they are small and the first products wait
  // for them.)
  // The same for the seven-wave split-K shapes (down at K = 14336: 2.318 → 2.310 ms per step); at 16 waves (qkv, o) it
  // loses (2.347).
  constexpr bool FS = KPW1 > 0 || KW == 7;
  if constexpr (FS) {
    load_stage(0, kb0);
    __syncthreads();
  }
  if constexpr (RMS_PRE)
    if (p.ss_in) rms_prefetch(rpf, p.ss_in, SS_CAP, p.M, wave, KW, lane);
  if constexpr (MODE == QM_RESID_ACT) resid_prefetch<R>(hpf, p, tile0);

  // Wave-private staging in LDS: the scale/bias words of the R tiles over this wave's K-blocks ([r][i][row] 8 bytes)
  // and token 16 of those K-blocks as [i][t][row ∈ {token 16, zeros}][qd] 16 bytes, so that lane (n, qd) reads
  // row n ≠ 0 ? zeros : token 16 from an address that depends on the K-block only through an immediate. The loads go
  // out first and only they are waited for before the LDS writes; no barrier: one wave's LDS operations complete in
  // order and no other wave reads the region (a workgroup barrier here made every wave wait for the slowest wave's
  // staging, queued behind all of the workgroup's first weight stages).
  __shared__ u32x4 ssb[KW][R * nk * 8];
  __shared__ u32x4 s16[KW][X16 ? nk * 32 : 1];
  __shared__ float rsc[MAX_TOK];
  constexpr int nsb = R * nk * 8;
  constexpr int NSB = (nsb + 63) / 64, N16 = X16 ? (nk * 16 + 63) / 64 : 1;
  u32x4 vsb[NSB], v16[N16];
#pragma unroll
  for (int j = 0; j < NSB; ++j) {
    const int e = j * 64 + lane, r = e / (nk * 8), i = (e >> 3) % nk;
    const unsigned off = (unsigned(tile0 + r) * unsigned(p.nkb) + unsigned(kb0 + i)) * 128u + unsigned(e & 7) * 16u;
    const bool in = e < nsb && i < nkr && kb0 + i < p.nkb;  // K-blocks past the matrix: zero scale and bias
    vsb[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsb, in ? off : OOB, 0, 0));
  }
  if constexpr (X16) {
#pragma unroll
    for (int j = 0; j < N16; ++j) {
      const int e = j * 64 + lane, i = e >> 4, t = (e >> 2) & 3, q = e & 3;
      const unsigned off = XN ? 16u * unsigned(p.ldx) * 2u + unsigned(kb0 + i) * (2u * KBLK) + 64u * t + 16u * q
                              : unsigned(kb0 + i) * unsigned(MAX_TOK / 16) * 4096u + 4096u + 1024u * t + 16u * q;
      const bool in = i < nkr && kb0 + i < p.nkb && (!XN || (kb0 + i) * KBLK + 32 * t < p.K);
      v16[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rx, in ? off : OOB, 0, 0));
    }
  }

  const bool idle = RAG && kb0 >= p.nkb;  // uniform: no K-blocks, the wave only adds its zeros
  if (!idle) {
#pragma unroll
    for (int d = FS ? 1 : 0; d < D; ++d) load_stage(d, kb0 + d);
  }

  // The RMSNorm factors of the input rows, while the first stages are on their way: their partials were requested
  // first, so waiting for them does not wait for the weights, and no accumulator is live yet.
  if constexpr (RMS_PRE) {
    if (p.ss_in) rms_finish(rpf, p.ss_in, SS_CAP, p.nss_in, p.D, p.eps, p.M, rsc, wave, KW, lane);
  }

#pragma unroll
  for (int j = 0; j < NSB; ++j) {
    const int e = j * 64 + lane;
    if (e < nsb) ssb[wave][e] = vsb[j];
  }
  if constexpr (X16) {
#pragma unroll
    for (int j = 0; j < N16; ++j) {
      const int e = j * 64 + lane, i = e >> 4, t = (e >> 2) & 3, q = e & 3;
      if (i < nk) {
        s16[wave][(i * 4 + t) * 8 + q] = XN ? frag_order(v16[j]) : v16[j];
        s16[wave][(i * 4 + t) * 8 + 4 + q] = u32x4{0u, 0u, 0u, 0u};
      }
    }
  }

  f32x4 acc[R][T];
  float acc16[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    acc16[r] = 0.f;
#pragma unroll
    for (int tt = 0; tt < T; ++tt) acc[r][tt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u});
  const f32x4 zero4 = f32x4{0.f, 0.f, 0.f, 0.f};
  const u32x4* const s16l = &s16[wave][0] + (n ? 4 : 0) + qd;  // this lane's row of the token-16 staging
  const uint2* const sbl = reinterpret_cast<const uint2*>(&ssb[wave][0]) + n;  // row n of the staged scale words

  // Products of ring stage d (K-block kl of this wave, 0 ≤ kl < nk).
  auto compute = [&](int d, int kl) {
    if constexpr (XN) {
#pragma unroll
      for (int tt = 0; tt < T; ++tt)
#pragma unroll
        for (int t = 0; t < 4; ++t) xv[d][tt][t] = frag_order(xv[d][tt][t]);
    }
    u32x4 x16[X16 ? 4 : 1];
    if constexpr (X16) {
#pragma unroll
      for (int t = 0; t < 4; ++t) x16[t] = s16l[(kl * 4 + t) * 8];
    }
    // Σx per group and token (ones operand), in the D layout of the products: lane (n, qd) gets tokens 4qd … 4qd+3.
    f32x4 xs[T][2];
#pragma unroll
    for (int tt = 0; tt < T; ++tt)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xv[d][tt][2 * g]), ones, zero4,
                                                          0, 0, 0);
        xs[tt][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xv[d][tt][2 * g + 1]), ones,
                                                            z, 0, 0, 0);
      }
    // Token 16: a second token tile whose only live row is token 16; its Σx per group lands in element 0 of the
    // qd = 0 lanes, like every other output of that token.
    float xs16[2] = {0.f, 0.f};
    if constexpr (X16) {
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        f32x4 z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x16[2 * g]), ones, zero4, 0, 0,
                                                          0);
        z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x16[2 * g + 1]), ones, z, 0, 0, 0);
        xs16[g] = z[0];
      }
    }
    // The scale/bias words of all R tiles, requested together before the first product so that one LDS latency per
    // K-block is exposed instead of one per tile (the fence after each tile keeps later reads from being hoisted).
    uint2 sbv[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sbv[r] = sbl[(r * nk + kl) * 16];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint2 sb = sbv[r];
      const float s0 = __uint_as_float(sb.x << 16), s1 = __uint_as_float(sb.y << 16);
      const float c0 = fmaf(-128.f, s0, __uint_as_float(sb.x & 0xFFFF0000u));
      const float c1 = fmaf(-128.f, s1, __uint_as_float(sb.y & 0xFFFF0000u));
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        bf16x8 w0, w1;
        nib_bf16_pair(wv[d][r][2 * g], wv[d][r][2 * g + 1], km, kbias, shv, w0, w1);
        const float sg = g ? s1 : s0, cg = g ? c1 : c0;
#pragma unroll
        for (int tt = 0; tt < T; ++tt) {
          f32x4 tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xv[d][tt][2 * g]), w0,
                                                              zero4, 0, 0, 0);
          tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, xv[d][tt][2 * g + 1]), w1, tmp, 0,
                                                        0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][tt][e] = fmaf(sg, tmp[e], fmaf(cg, xs[tt][g][e], acc[r][tt][e]));
        }
        if constexpr (X16) {
          f32x4 tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x16[2 * g]), w0, zero4, 0,
                                                              0, 0);
          tmp = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x16[2 * g + 1]), w1, tmp, 0, 0,
                                                        0);
          acc16[r] = fmaf(sg, tmp[0], fmaf(cg, xs16[g], acc16[r]));
        }
      }
      // One tile at a time: without the fence the scheduler decodes every tile's nibbles ahead of the products and
      // the decoded operands (16 VGPRs per tile) exhaust the register file at R = 7.
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // The ring: trips of D K-blocks, each multiplied from its stage and the stage refilled D K-blocks ahead, then the
  // last D K-blocks without refills (nk is a multiple of D, which the launch checks; nk = D loads everything at
  // entry).
  if (!idle) {
    int i = 0;
#pragma unroll 1
    for (; i < nkr - D; i += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        compute(d, i + d);
        load_stage(d, kb0 + i + d + D);
      }
    }
#pragma unroll
    for (int d = 0; d < D; ++d) {
      compute(d, i + d);
    }
  }

  // Partial sums of every wave → LDS [wave][r][tt][e][lane] (+ token 16 [wave][r][row]), then fixed-order sums.
  constexpr int NEL = R * T * 4 * 64;
  constexpr int NEL16 = X16 ? R * 16 : 0;
  constexpr int WST = NEL + NEL16;
  __shared__ float red[KW * WST];
  __shared__ float ssu[MAX_TOK * 2 * R];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int tt = 0; tt < T; ++tt)
#pragma unroll
      for (int e = 0; e < 4; ++e) red[wave * WST + ((r * T + tt) * 4 + e) * 64 + lane] = acc[r][tt][e];
  if constexpr (X16) {
    if (lane < 16) {
#pragma unroll
      for (int r = 0; r < R; ++r) red[wave * WST + NEL + r * 16 + lane] = acc16[r];
    }
  }
  // Without the entry prefetch (one-wave workgroups, more rows than a wave prefetches): the RMSNorm factors once the
  // accumulators are in LDS (their loads and shuffles would otherwise keep every accumulator live across them).
  if constexpr (RMS && !RMS_PRE) {
    if (p.ss_in) rms_factors(p.ss_in, SS_CAP, p.nss_in, p.D, p.eps, p.M, rsc, wave, KW, lane);
  }
  __syncthreads();
  // Sum over waves, in wave order, of every partial at once (independent, coalesced LDS reads spread over the whole
  // workgroup), into wave 0's slots; the epilogue then reads one value per output.
  if constexpr (KW > 1) {
    for (int i = threadIdx.x; i < WST; i += 64 * KW) {
      float v = red[i];
#pragma unroll
      for (int w = 1; w < KW; ++w) v += red[w * WST + i];
      red[i] = v;
    }
    __syncthreads();
  }
  // The finished output (token m, tile r, row rn of the tile).
  auto val = [&](int m, int r, int rn) -> float {
    int i;
    if (X16 && m == 16) {
      i = NEL + r * 16 + rn;
    } else {
      const int tt = m >> 4, mm = m & 15;
      i = ((r * T + tt) * 4 + (mm & 3)) * 64 + 16 * (mm >> 2) + rn;
    }
    return red[i];
  };
  if (gridDim.y > 1) {
    // K split over gridDim.y workgroups: each writes its partial sums with agent-coherent stores (they bypass the
    // XCD's L2, so no cache write-back is needed), then counts itself in on the row group's counter; the last to
    // arrive adds the partials in split order (its own from LDS) and runs the epilogue, the others exit. No
    // workgroup waits for another, and the sum's order depends only on the split, not on who arrives last.
    const int nsp = int(gridDim.y), me = int(blockIdx.y);
    const unsigned sstride = unsigned(MAX_TOK) * unsigned(p.Npad);  // floats per split
    const __amdgpu_buffer_rsrc_t rp = make_rsrc(p.part, unsigned(nsp) * sstride * 4u);
    // Quads of 4 consecutive rows of one token: slot of (m, 4q) in red, byte offset in a split's partials.
    auto quad = [&](int u, int& i, unsigned& off) {
      const int m = u / (4 * R), rr = 4 * (u % (4 * R)), r = rr >> 4, rn = rr & 15;
      if (X16 && m == 16) {
        i = NEL + r * 16 + rn;
      } else {
        const int tt = m >> 4, mm = m & 15;
        i = ((r * T + tt) * 4 + (mm & 3)) * 64 + 16 * (mm >> 2) + rn;
      }
      off = (unsigned(m) * unsigned(p.Npad) + unsigned(tile0 * 16 + rr)) * 4u;
    };
    constexpr int SC1 = 16;  // cache policy: agent-coherent (sc1)
    for (int u = threadIdx.x; u < p.M * 4 * R; u += 64 * KW) {
      int i;
      unsigned off;
      quad(u, i, off);
      const f32x4 v = f32x4{red[i], red[i + 1], red[i + 2], red[i + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), rp, off, unsigned(me) * sstride * 4u,
                                             SC1);
    }
    __builtin_amdgcn_s_waitcnt(0);  // every partial store of this thread has completed
    __syncthreads();
    __shared__ unsigned arrived;
    if (threadIdx.x == 0) {
      arrived = __hip_atomic_fetch_add(p.ctr + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (arrived == unsigned(nsp - 1))
        __hip_atomic_store(p.ctr + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (arrived != unsigned(nsp - 1)) return;  // workgroup-uniform
    // Ordering without agent-scope fences (an agent-scope release writes back the XCD's L2, ~15 µs per launch; an
    // acquire, which invalidates the CU's caches, measured 0.14 ms per configuration-1 step): every writer's
    // partials are agent-coherent stores (sc1: they bypass the XCD's L2), completed (waitcnt 0) before its barrier
    // and its count, so they are at the coherence point before the count that reports them; the reads below are
    // sc1 loads (they do not hit stale lines of this CU's caches), issued after the workgroup barrier that follows
    // the count (a workgroup-scope acquire: the compiler cannot hoist them above it) and under the branch on the
    // count's value (the hardware issues no load of a branch before the branch resolves).
    // The sums, in split order, into wave 0's partial slots (each thread reads back only slots it owns).
    for (int u = threadIdx.x; u < p.M * 4 * R; u += 64 * KW) {
      int i;
      unsigned off;
      quad(u, i, off);
      f32x4 v = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int sp = 0; sp < nsp; ++sp) {
        const f32x4 x = sp == me ? f32x4{red[i], red[i + 1], red[i + 2], red[i + 3]}
                                 : __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                                                 rp, off, unsigned(sp) * sstride * 4u, SC1));
        v += x;
      }
      red[i] = v[0];
      red[i + 1] = v[1];
      red[i + 2] = v[2];
      red[i + 3] = v[3];
    }
    __syncthreads();
  }
  qmm_epilogue<R, MODE>(p, tile0, val, rsc, ssu, 64 * KW, blockIdx.x, &hpf);
}

// Launch shape: see qmm_shape (qmm.hip). ragged: the K range need not be tiled exactly; waves past its end are idle and
// a wave that runs past it re-reads the last K-block with zero scales.
struct QmmShape { int R, KW, D, kpw, ks, kpw1 = 0, ragged = 0; };
constexpr int qmm_ring_depth(int kpw) { return kpw % 2 == 0 ? 2 : kpw <= 3 ? kpw : 1; }

// Whether a shape's LDS fits with T token tiles (and token 16 on its own): only those are instantiated. Two tiles of
// (7, 8, 6) do not: the caller's rows past 17 go as two groups of 16 there (qmm_setup).
constexpr bool qmm_fits(int T, int R, int KW, bool X16, int KPW) {
  return 4 * KW * (R * T * 256 + (X16 ? R * 16 : 0)) + 4 * MAX_TOK * (2 * R + 1) + R * KW * KPW * 128 +
             (X16 ? KW * KPW * 512 : 0) <= 128 * 1024;
}

// Instantiated launch shapes (R, KW, KPW; ring depth qmm_ring_depth(KPW)) for each epilogue. Epilogues are compile-time:
// the code of every mode in one kernel raised its register demand past the ring's (302 VGPRs at R = 7, KW = 4).
template <int T, bool X16, int MODE, bool XN = false>
static bool qmm_dispatch_mode(const TimedLaunch& tl, QmmShape sh, dim3 grid, hipStream_t st, const QmmParams& p) {
#define IH_QMM_CASE(R_, KW_, KPW_)                                                                          \
  if constexpr (qmm_fits(T, R_, KW_, X16, KPW_)) {                                                        \
    if (sh.R == R_ && sh.KW == KW_ && sh.kpw == KPW_ && sh.kpw1 == 0 && !sh.ragged) {                                     \
      tlaunch(tl, qmm_int4_kernel<T, R_, KW_, X16, qmm_ring_depth(KPW_), KPW_, MODE, 0, XN>, grid,            \
              dim3(64 * KW_), 0, st, p);                                                                                       \
      return true;                                                                                          \
    }                                                                                                       \
  }
  // K = 4096 (32 K-blocks); K = 14336 (112; (4,7,4) and (2,7,8) split it over 4 and 2 workgroups); K = 2048 (16);
  // K = 2880 (23, ragged); and the one-wave fallback.
  IH_QMM_CASE(1, 16, 2) IH_QMM_CASE(2, 16, 2) IH_QMM_CASE(2, 8, 4) IH_QMM_CASE(4, 8, 4) IH_QMM_CASE(4, 4, 8)
  IH_QMM_CASE(7, 4, 8) IH_QMM_CASE(1, 14, 8) IH_QMM_CASE(1, 8, 14) IH_QMM_CASE(4, 4, 2) IH_QMM_CASE(2, 8, 2)
  IH_QMM_CASE(4, 8, 2) IH_QMM_CASE(2, 8, 3) IH_QMM_CASE(4, 8, 3) IH_QMM_CASE(4, 7, 4) IH_QMM_CASE(2, 7, 8)
  IH_QMM_CASE(1, 1, 1) IH_QMM_CASE(2, 1, 1) IH_QMM_CASE(4, 1, 1) IH_QMM_CASE(7, 1, 1)
#undef IH_QMM_CASE
  // Asymmetric K split (KPW for the first half of the waves, KPW1 for the second): gate|up at two waves per SIMD.
#define IH_QMM_CASE1(R_, KW_, KPW_, KPW1_)                                                                       \
  if constexpr (qmm_fits(T, R_, KW_, X16, KPW_)) {                                                        \
    if (sh.R == R_ && sh.KW == KW_ && sh.kpw == KPW_ && sh.kpw1 == KPW1_) {                                \
      tlaunch(tl, qmm_int4_kernel<T, R_, KW_, X16, 2, KPW_, MODE, KPW1_, XN>, grid, dim3(64 * KW_), 0, st, p);   \
      return true;                                                                                          \
    }                                                                                                       \
  }
  IH_QMM_CASE1(7, 8, 6, 2)
#undef IH_QMM_CASE1
  if constexpr (XN && T == 1) {
#define IH_QMM_CASER(R_, KW_, KPW_)                                                                                 \
  if constexpr (qmm_fits(T, R_, KW_, X16, KPW_)) {                                                                \
    if (sh.ragged && sh.R == R_ && sh.KW == KW_ && sh.kpw == KPW_) {                                                \
      tlaunch(tl, qmm_int4_kernel<T, R_, KW_, X16, qmm_ring_depth(KPW_), KPW_, MODE, 0, true, true>, grid,          \
              dim3(64 * KW_), 0, st, p);                                                                            \
      return true;                                                                                                  \
    }                                                                                                               \
  }
    IH_QMM_CASER(1, 16, 1) IH_QMM_CASER(1, 16, 2) IH_QMM_CASER(1, 16, 3) IH_QMM_CASER(1, 16, 4) IH_QMM_CASER(1, 14, 8)
    IH_QMM_CASER(2, 16, 1) IH_QMM_CASER(2, 16, 2) IH_QMM_CASER(2, 16, 4) IH_QMM_CASER(2, 14, 8)
    IH_QMM_CASER(4, 8, 2) IH_QMM_CASER(4, 8, 3) IH_QMM_CASER(4, 8, 4) IH_QMM_CASER(4, 8, 8)
#undef IH_QMM_CASER
  }
  return false;  // not an instantiated shape
}

// qmm_rows.hip: the launch on bf16 rows (more than 17: two token tiles, or grid.z = 2 groups of 16).
bool qmm_rows_dispatch(const TimedLaunch& tl, QmmShape sh, dim3 grid, hipStream_t st, const QmmParams& p, int M,
                       int mode);

}  // namespace ih
