// Few-row quantized matmul of the verify step on gfx950: Y[M ≤ 32, N] (+)= X[M, K] · dequant(W)ᵀ, with the epilogues
// of the round fused in (RMSNorm scale, residual add, gated activation, next activation's layout).
//
// Reference: VQMV.encode → vnax_qmv_nf1_sg32 (Sources/Ingot/Layers/Linear.swift:263-445,
// Sources/Ingot/Shaders/verify_nax.metal:102-176); the arithmetic it stands for is qmv_acc
// (Sources/Ingot/Shaders/verify.metal:89-105): y = Σ_groups s·Σ x·q + b·Σ x.
//
// MI355X design (not a translation of the Metal kernel):
//   - HBM-bound at M ≤ 17 (≈ 2·M / 0.5625 ≤ 60 FLOP/B). Each wave streams its weight tiles with one contiguous
//     1024-byte dwordx4 buffer load per 16×128 tile (layout in ih_internal.h), the next K-block in flight while the
//     current one is multiplied, and dequantizes in registers.
//   - The products run on MFMA v_mfma_f32_16x16x32_bf16 with the tokens as the A operand (16 tokens × 32 K) and the
//     weights as B (32 K × 16 rows). A nibble q becomes the bf16 128 + q with one v_and_or_b32 per pair
//     ((w >> 4c) & 0x000F000F | 0x43004300), so the MFMA sums Σ x·(128 + q) exactly in fp32 per group of 64; one more
//     MFMA against a ones operand gives Σ x per group and token in the same layout, and the affine map is applied
//     once per group and output: y += s·acc + (b − 128·s)·Σx. No rounding of the dequantised weight.
//   - Token 16 (the 17th row of a k = 16 block) is the only live row of a second MFMA token tile whose A operand
//     comes from LDS (token 16 staged once per workgroup, zeros for the other rows), so it costs no extra
//     vector-memory instructions and one output element of VALU work. Each MFMA output element depends only on its
//     own A row, so its bits are those of the M > 17 path (two full token tiles) and never depend on M.
//   - K is split over the waves of a workgroup (a split chosen from (N, K) only, never from M) and the partial sums are
//     added in wave order in LDS: deterministic and row-invariant (row r's bits do not depend on M).
#include "act.h"
#include "ih_internal.h"
#include "qmm_common.h"
#include "qmm_kernel.h"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <cstdlib>

namespace ih {

// ---------------------------------------------------------------------------------------------------------------
// Repack an MLX int4 g64 matrix ([E][N][K/8] words, [E][N][K/64] bf16 scales and biases) into the tile layout.
// Grid (Npad/16 · nkb, E), 64 threads: lane L = 16·qd + n. With il8, rows are interleaved by eights for a gate|up pair
// (N = 2I, gate rows 0…I−1, up rows I…2I−1): tile t holds gate rows 8t…8t+7 then up rows 8t…8t+7, so one tile's
// outputs are the gate and up of the same 8 columns.
__global__ void pack_int4_kernel(const uint32_t* __restrict__ w, const uint16_t* __restrict__ s,
                                 const uint16_t* __restrict__ b, uint4* __restrict__ wp, uint2* __restrict__ sp, int N,
                                 int K, int Npad, int nkb, int il8) {
  const int lane = threadIdx.x, n = lane & 15, qd = lane >> 4;
  const int tile = blockIdx.x / nkb, kb = blockIdx.x % nkb, e = blockIdx.y;
  const int prow = tile * 16 + n;
  const int row = il8 ? (n < 8 ? 8 * tile + n : N / 2 + 8 * tile + n - 8) : prow;
  const bool live = il8 ? (8 * tile + (n & 7) < N / 2) : row < N;
  const int wpr = K / 8, gpr = K / 64;
  const size_t ebase_w = size_t(e) * N * wpr, ebase_s = size_t(e) * N * gpr;
  unsigned v[4];
  for (int t = 0; t < 4; ++t) {
    int wi = kb * 16 + 4 * t + qd;
    v[t] = (live && wi < wpr) ? w[ebase_w + size_t(row) * wpr + wi] : 0u;
  }
  const size_t tb = (size_t(e) * (Npad / 16) + tile) * nkb + kb;
  wp[tb * 64 + lane] = make_uint4(v[0], v[1], v[2], v[3]);
  if (qd == 0) {
    unsigned s0 = 0, b0 = 0, s1 = 0, b1 = 0;
    if (live) {
      int g0 = 2 * kb, g1 = 2 * kb + 1;
      if (g0 < gpr) { s0 = s[ebase_s + size_t(row) * gpr + g0]; b0 = b[ebase_s + size_t(row) * gpr + g0]; }
      if (g1 < gpr) { s1 = s[ebase_s + size_t(row) * gpr + g1]; b1 = b[ebase_s + size_t(row) * gpr + g1]; }
    }
    sp[tb * 16 + n] = make_uint2(s0 | (b0 << 16), s1 | (b1 << 16));
  }
}

// ---------------------------------------------------------------------------------------------------------------
// bf16 rows that are not 16-byte aligned → aligned rows of ld elements, one thread per eight (K is a multiple of 64):
// grid (⌈K / 512⌉, M), 64 threads. (With one workgroup per row and an element per thread and trip, 16 rows at an odd
// element through 4096 × 4096 took 11.0 µs a call, with this 8.5.)
__global__ __launch_bounds__(64) void align_rows_kernel(const uint16_t* __restrict__ x, int ldx, int K,
                                                        uint16_t* __restrict__ out, int ld) {
  const int i = blockIdx.y, c = 8 * (blockIdx.x * 64 + threadIdx.x);
  if (c >= K) return;
  const uint16_t* p = x + size_t(i) * ldx + c;
  unsigned w[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) w[e] = unsigned(p[2 * e]) | unsigned(p[2 * e + 1]) << 16;
  *reinterpret_cast<uint4*>(out + size_t(i) * ld + c) = make_uint4(w[0], w[1], w[2], w[3]);
}

// ---------------------------------------------------------------------------------------------------------------
// Launch shape for an (Npad, nkb) matrix: R row tiles per wave, KW waves per workgroup, ring depth D, kpw K-blocks per
// wave, and ks = nkb / (KW·kpw) workgroups splitting K. KW, kpw and ks come from the shape only, never from M, so each
// row's summation order is fixed. The K range tiles exactly (ks·KW·kpw = nkb, kpw a multiple of D), or, in one split, the
// last wave runs past the end by less than its kpw: its K-blocks past the matrix re-stream the last block (clamped,
// so every load stays inside the matrix) with zero scale and bias words, which add exactly nothing.
static bool qmm_shape_ok(const QmmShape& sh, int Npad, int nkb) {
  const int span = sh.kpw1 ? sh.KW / 2 * (sh.kpw + sh.kpw1) : sh.KW * sh.kpw;
  return sh.R >= 1 && sh.KW >= 1 && sh.D >= 1 && sh.kpw >= sh.D && sh.kpw % sh.D == 0 && sh.kpw <= 32 &&
         sh.R * sh.kpw <= 64 && (Npad / 16) % sh.R == 0 &&
         (sh.ks * span == nkb || (sh.ks == 1 && span > nkb && span - nkb < sh.kpw) || (sh.ragged && sh.ks * span >= nkb));
}
// The instantiated (R, KW, KPW) shapes (qmm_dispatch_mode lists the same set).
static constexpr int kQmmShapes[][3] = {{1, 16, 2}, {2, 16, 2}, {2, 8, 4}, {4, 4, 8}, {4, 8, 4}, {7, 4, 8},
                                        {1, 8, 14}, {1, 14, 8}, {4, 4, 2}, {2, 8, 2}, {4, 8, 2}, {1, 1, 1},
                                        {2, 1, 1},  {4, 1, 1},  {7, 1, 1},  {2, 8, 3},  {4, 8, 3}};
static QmmShape qmm_shape_sym(int Npad, int nkb, int M);
// The symmetric choice below, except that seven-tile workgroups over 32 K-blocks (gate|up at K = 4096) run at two
// waves per SIMD with the asymmetric split (7,8,6,2): the loop's VALU work issues ~2× faster per SIMD with two waves,
// and the second wave of each SIMD, whose first stage arrives ~3 µs later, takes a third of the K-blocks of the first.
static QmmShape qmm_shape(int Npad, int nkb, int M) {
  const QmmShape sh = qmm_shape_sym(Npad, nkb, M);
  if (sh.R == 7 && sh.KW == 4 && sh.kpw == 8 && sh.ks == 1) return QmmShape{7, 8, 2, 6, 1, 2};
  // One-tile workgroups over 112 K-blocks (down at K = 14336): every workgroup reads the whole 487 KB activation from
  // L2, which bounds the kernel; two-tile workgroups with K split in two read half as much per CU, and the split's
  // reduction in the last-arriving workgroup costs less than that saves (config 1: 2.375 → 2.342 ms per step).
  if (sh.R == 1 && sh.KW == 8 && sh.kpw == 14 && sh.ks == 1 && nkb == 112 && Npad % 32 == 0) {
    const QmmShape s2{2, 7, qmm_ring_depth(8), 8, 2};
    if (qmm_shape_ok(s2, Npad, nkb)) return s2;
  }
  return sh;
}
// Products of the caller's rows whose K-block count no exact shape tiles: the smallest span of the row-tile class that
// covers K (waves past the end idle), or the largest one in as many splits as it takes. One wave per workgroup and
// K-block, the general shape below, leaves the sum of all the splits to the last workgroup (2880 × 4160: 15.8 µs in two
// launches against 5). Four row tiles are taken from 2048 on (vocabulary-sized N), where they were measured first. Below,
// down to 513, they are faster for most sizes as well (17 rows, two against four: 8256 × 1600 8.1 and 6.4 µs, 11008 × 4160
// 14.6 and 13.3, 32000 × 4160 28.3 and 26.2, but 24576 × 4160 21.8 and 25.7; at 384 tiles 8.2 and 13.0).
static QmmShape qmm_shape_ragged(int Npad, int nkb) {
  static constexpr int one[5][2] = {{16, 1}, {16, 2}, {16, 3}, {16, 4}, {14, 8}};
  static constexpr int two[4][2] = {{16, 1}, {16, 2}, {16, 4}, {14, 8}};  // (16, 3) spills with two row tiles
  static constexpr int four[4][2] = {{8, 2}, {8, 3}, {8, 4}, {8, 8}};
  const int NT = Npad / 16, R = NT >= 2048 ? 4 : NT > 256 ? 2 : 1, n = R == 1 ? 5 : 4;
  const auto* v = R == 4 ? four : R == 2 ? two : one;
  int i = 0;
  while (i + 1 < n && v[i][0] * v[i][1] < nkb) ++i;
  const int span = v[i][0] * v[i][1];
  return QmmShape{R, v[i][0], qmm_ring_depth(v[i][1]), v[i][1], (nkb + span - 1) / span, 0, 1};
}
static QmmShape qmm_shape_sym(int Npad, int nkb, int M) {
  const int NT = Npad / 16;
  // Rows: R tiles per wave share x, and the workgroup count NT / R should be about one round over the 256 CUs (a
  // partial second round doubles the time of the CUs that run it): 7 for gate|up (1792 tiles → 256 workgroups), 2
  // for qkv (192), 1 for o and down (256). Above 512 tiles every CU has several workgroups' work whatever R is, and four
  // tiles per wave read half as much x per weight as two (17 rows, K = 4096: 11008 rows 12.9 → 9.5 µs, 16384 13.4 →
  // 10.2, 24576 19.7 → 16.1, 32000 26.6 → 18.9; at 8192 rows two tiles are better, 7.4 against 9.4).
  int rp[4] = {1, 2, 0, 0};
  if (NT % 7 == 0 && NT / 7 >= 192 && NT / 7 <= 320) { rp[0] = 7; rp[1] = 4; rp[2] = 2; rp[3] = 1; }
  else if (NT > 512) {
    // At K ≤ 2048 the x of four tiles is no longer what binds, and two fill the rounds better where four leave a quarter
    // of the last one's CUs idle (20480 × 2048: 9.5 against 10.5 µs; 32000 × 2048, where they do not, 12.1 against 10.9).
    auto fill = [](int wgs) { return double(wgs) / ((wgs + 255) / 256 * 256); };
    const bool two = nkb <= 16 && fill(NT / 2) > 1.25 * fill(NT / 4);
    rp[0] = two ? 2 : 4;
    rp[1] = two ? 4 : 2;
    rp[2] = 1;
  }
  else if (NT > 256) { rp[0] = 2; rp[1] = 1; }
  // K: the whole range in one workgroup when a shape tiles it (16 waves × 2 K-blocks at K = 4096; a ring of 8 or 14
  // K-blocks per wave for longer K), else split over workgroups.
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1) {
      // K too long for one workgroup: eight waves over four tiles (two where that leaves CUs idle), the span whose
      // workgroups fill their rounds over the CUs best. Every workgroup reads its whole K range of x from L2, so one
      // tile per wave reads several times the weights' bytes in x (17 rows: 4096 × 12288 20.5 → 11.7 µs, 4096 × 8192
      // 14.3 → 9.6, 8192 × 8192 15.6 → 12.5; 16 rows: 4096 × 20480 30.9 → 15.8).
      QmmShape best{};
      double fill = 0;
      for (int R : {4, 2}) {
        for (int kpw : {4, 3, 2}) {
          const QmmShape sh{R, 8, qmm_ring_depth(kpw), kpw, nkb / (8 * kpw)};
          if (nkb % (8 * kpw) || !qmm_shape_ok(sh, Npad, nkb)) continue;
          const int wgs = NT / R * sh.ks, rounds = (wgs + 255) / 256;
          if (wgs < (R == 4 ? 192 : 128) || wgs <= fill * rounds * 256) continue;
          fill = double(wgs) / (rounds * 256);
          best = sh;
        }
        if (best.R) return best;
      }
    }
    for (int R : rp) {
      if (R == 0) continue;
      for (const auto& c : kQmmShapes) {
        if (c[0] != R || c[1] == 1) continue;
        const int span = c[1] * c[2];
        if (nkb % span) continue;
        const QmmShape sh{R, c[1], qmm_ring_depth(c[2]), c[2], nkb / span};
        if ((pass == 0 && sh.ks != 1) || !qmm_shape_ok(sh, Npad, nkb)) continue;
        return sh;
      }
    }
  }
  // K-block counts without a fitting factor: one split whose last wave runs past the end by less than its kpw. One token
  // tile leaves less x to share, and two row tiles per wave win there (K = 2880, 9 rows: 32000 11.1 against 12.5 µs, 50257
  // 20.7 against 23.9, 201088 74.7 against 80.4; 17 rows: 20.0, 36.1 and 125.8 against 14.9, 32.1 and 101.5). Only the
  // row tiles follow M (not for the residual epilogue, see qmm_setup): the waves and their K-blocks, which order a row's
  // sums, stay.
  for (int R : rp)
    if (R)
      for (const auto& c : kQmmShapes) {
        if (c[0] != R || c[1] == 1) continue;
        QmmShape sh{R, c[1], qmm_ring_depth(c[2]), c[2], 1};
        if (c[1] * c[2] <= nkb || !qmm_shape_ok(sh, Npad, nkb)) continue;
        if (R == 4 && NT >= 1024 && M <= 16)
          for (const auto& t : kQmmShapes)
            if (t[0] == 2 && t[1] == sh.KW && t[2] == sh.kpw) sh.R = 2;
        return sh;
      }
  // Otherwise one wave per workgroup, one K-block per wave.
  for (int R : rp)
    if (R && (Npad / 16) % R == 0) return QmmShape{R, 1, 1, 1, nkb};
  return QmmShape{1, 1, 1, 1, nkb};
}

// The fused modes of the round on fragment activations.
template <int T, bool X16>
static bool qmm_dispatch(const TimedLaunch& tl, QmmShape sh, dim3 grid, hipStream_t st, const QmmParams& p, int mode) {
  switch (mode) {
    case QM_F32: return qmm_dispatch_mode<T, X16, QM_F32>(tl, sh, grid, st, p);
    case QM_F32_SCALE: return qmm_dispatch_mode<T, X16, QM_F32_SCALE>(tl, sh, grid, st, p);
    case QM_RESID_ACT: return qmm_dispatch_mode<T, X16, QM_RESID_ACT>(tl, sh, grid, st, p);
    case QM_GLU_ACT: return qmm_dispatch_mode<T, X16, QM_GLU_ACT>(tl, sh, grid, st, p);
    default: return false;
  }
}

// Split-K partial sums: grown on demand, the stream drained before an old buffer is freed.
static int ensure_qpart(ih_ctx* c, size_t bytes) {
  if (!c->qctr) {
    // Arrival counters of the in-kernel split-K reduction: zeroed once; the last workgroup of a row group resets its
    // counter, so they are zero between launches.
    ++c->gen;
    if (hipMalloc(&c->qctr, QCTR_CAP * sizeof(unsigned)) != hipSuccess)
      return fail(IH_ENOMEM, "qmm: split-K counter allocation failed");
    IH_TRY(fill(c, c->qctr, 0, QCTR_CAP * sizeof(unsigned)));
  }
  if (c->qpart_bytes >= bytes) return IH_OK;
  ++c->gen;
  IH_HIP(hipStreamSynchronize(c->stream));
  if (c->qpart) IH_HIP(hipFree(c->qpart));
  c->qpart = nullptr;
  c->qpart_bytes = 0;
  if (hipMalloc(&c->qpart, bytes) != hipSuccess) return fail(IH_ENOMEM, "qmm: split-K partial allocation failed");
  c->qpart_bytes = bytes;
  return IH_OK;
}

// The launch's shape (an override of the matrix size first), its K split and the weight side of its parameters. `rows`:
// the caller's rows (qmm_rows.hip).
static int qmm_setup(ih_ctx* c, const ih_qmat* W, int expert, int M, int mode, bool rows, QmmShape& sh, QmmParams& p,
                     dim3& grid) {
  IH_CHECK(W->format == QF_INT4, IH_EINVAL, "qmm: int4 matrix expected");
  IH_CHECK(M >= 1 && M <= MAX_TOK, IH_EINVAL, "qmm: M must be in 1..32");
  // The residual epilogue writes a sum-of-squares partial per workgroup: its row tiles, which group the columns of the
  // next RMSNorm's sum, must not follow M either.
  sh = qmm_shape(W->Npad, W->nkb, mode == QM_RESID_ACT ? MAX_TOK : M);
  if (rows && sh.KW == 1) sh = qmm_shape_ragged(W->Npad, W->nkb);
  for (const auto& o : c->qmm_shapes) {
    if (o[0] != W->N || o[1] != W->K) continue;
    const int span = o[5] ? o[3] / 2 * (o[4] + o[5]) : o[3] * o[4];
    sh = QmmShape{o[2], o[3], o[5] ? 2 : qmm_ring_depth(o[4]), o[4], std::max(1, W->nkb / std::max(1, span)), o[5]};
  }
  IH_CHECK(qmm_shape_ok(sh, W->Npad, W->nkb), IH_EINVAL, "qmm: launch shape does not tile the matrix");
  const size_t tiles_per_e = size_t(W->Npad / 16) * W->nkb;
  p = QmmParams{};
  p.w = static_cast<const uint4*>(W->w) + tiles_per_e * 64 * expert;
  p.s = static_cast<const uint2*>(W->s) + tiles_per_e * 16 * expert;
  p.M = M;
  p.N = W->N;
  p.K = W->K;
  p.Npad = W->Npad;
  p.nkb = W->nkb;
  p.kmask = 0x000F000Fu;
  p.kbias = 0x43004300u;
  // More than 17 of the caller's rows: two token tiles of one product, or two products of 16 rows where the registers
  // (ragged shapes of 16 waves) or the LDS of two do not fit.
  const bool two = rows && M > 17 && (sh.ragged || !qmm_fits(2, sh.R, sh.KW, false, sh.kpw));
  grid = dim3(W->Npad / (16 * sh.R), sh.ks, two ? 2 : 1);
  if (sh.ks > 1) {
    IH_TRY(ensure_qpart(c, size_t(sh.ks) * MAX_TOK * W->Npad * sizeof(float)));
    p.part = c->qpart;
    IH_CHECK(int(grid.x * grid.z) <= QCTR_CAP, IH_EINVAL, "qmm: too many row groups for the split-K counters");
    p.ctr = c->qctr;
  }
  return IH_OK;
}

int launch_qmm_ex(ih_ctx* c, const ih_qmat* W, int expert, const ActBuf& a, int M, const QmmEpilogue& ep) {
  IH_CHECK(a.nkb == W->nkb && !a.f16, IH_EINVAL, "qmm: activation K does not match the matrix");
  QmmShape sh;
  QmmParams p;
  dim3 grid;
  IH_TRY(qmm_setup(c, W, expert, M, ep.mode, false, sh, p, grid));
  p.xa = static_cast<const uint4*>(a.frag);
  p.y = ep.y;
  p.ldy = ep.ldy;
  if (ep.mode == QM_F32_SCALE || ep.mode == QM_GLU_ACT) {
    IH_CHECK(a.ss && a.nss > 0, IH_EINVAL, "qmm: the input activation carries no RMSNorm sums");
    p.ss_in = a.ss;
    p.nss_in = a.nss;
    p.D = a.K;
    p.eps = ep.eps;
  }
  if (ep.mode == QM_RESID_ACT) {
    IH_CHECK(ep.act_out && ep.act_out->nkb * KBLK >= W->N && ep.nw, IH_EINVAL, "qmm: residual epilogue needs an output");
    IH_CHECK(int(grid.x) <= ep.act_out->ss_cap, IH_EINVAL, "qmm: too many workgroups for the RMSNorm partials");
    p.nw = ep.nw;
    p.bias = ep.bias;
    p.act_out = static_cast<uint4*>(ep.act_out->frag);
    p.act_nkb = ep.act_out->nkb;
    p.act_f16 = ep.act_out->f16 ? 1 : 0;
    p.ss_out = ep.act_out->ss;
    ep.act_out->nss = int(grid.x);
  }
  if (ep.mode == QM_GLU_ACT) {
    IH_CHECK(ep.act_out && ep.act_out->nkb * KBLK >= W->N / 2 && W->il8, IH_EINVAL,
             "qmm: gated epilogue needs an interleaved gate|up matrix and an output");
    p.act_out = static_cast<uint4*>(ep.act_out->frag);
    p.act_nkb = ep.act_out->nkb;
    p.act_f16 = ep.act_out->f16 ? 1 : 0;
    p.glu = ep.glu;
    p.limit = ep.limit;
  }
  // Algorithmic bytes: the matrix in its MLX format, x (bf16) read, y written (read too when accumulating).
  TimedLaunch tl(c, TC_QMM, double(W->algo_bytes) + double(M) * W->K * 2 +
                                double(M) * W->N * (ep.mode == QM_RESID_ACT ? 8 : 4));
  bool ok;
  if (M > 17) ok = qmm_dispatch<2, false>(tl, sh, grid, c->stream, p, ep.mode);
  else if (M == 17) ok = qmm_dispatch<1, true>(tl, sh, grid, c->stream, p, ep.mode);
  else ok = qmm_dispatch<1, false>(tl, sh, grid, c->stream, p, ep.mode);
  IH_CHECK(ok, IH_EINVAL, "qmm: launch shape not instantiated");
  IH_HIP(hipGetLastError());
  return IH_OK;
}

int launch_qmm_rows(ih_ctx* c, const ih_qmat* W, const uint16_t* x, int ldx, int M, void* y, int ldy, int out_mode) {
  QmmShape sh;
  QmmParams p;
  dim3 grid;
  IH_TRY(qmm_setup(c, W, 0, M, out_mode, true, sh, p, grid));
  // The kernel reads 16-byte pieces of the rows through 32-bit offsets; other rows are copied to aligned scratch first,
  // and so are rows that the output overwrites (some workgroups store while others still read x).
  const uintptr_t x0 = reinterpret_cast<uintptr_t>(x), y0 = reinterpret_cast<uintptr_t>(y);
  const uintptr_t x1 = x0 + (size_t(M - 1) * ldx + W->K) * 2;
  const uintptr_t y1 = y0 + (size_t(M - 1) * ldy + W->N) * (out_mode == QM_BF16 ? 2 : 4);
  if (x0 % 16 != 0 || ldx % 8 != 0 || (x0 < y1 && y0 < x1) ||
      (size_t(M - 1) * ldx + W->K) * 2 >= (size_t(1) << 31)) {
    IH_TRY(ensure_act(c, c->act, W->K, false));
    uint16_t* rows = static_cast<uint16_t*>(c->act.frag);
    align_rows_kernel<<<dim3((W->K + 511) / 512, M), 64, 0, c->stream>>>(x, ldx, W->K, rows, W->nkb * KBLK);
    IH_HIP(hipGetLastError());
    x = rows;
    ldx = W->nkb * KBLK;
  }
  p.xa = reinterpret_cast<const uint4*>(x);
  p.ldx = ldx;
  p.y = y;
  p.ldy = ldy;
  TimedLaunch tl(c, TC_QMM, double(W->algo_bytes) + double(M) * W->K * 2 +
                                double(M) * W->N * (out_mode == QM_BF16 ? 2 : out_mode == QM_F32_ADD ? 8 : 4));
  IH_CHECK(qmm_rows_dispatch(tl, sh, grid, c->stream, p, M, out_mode), IH_EINVAL, "qmm: launch shape not instantiated");
  IH_HIP(hipGetLastError());
  return IH_OK;
}

int launch_qmm(ih_ctx* c, const ih_qmat* W, int expert, const ActBuf& a, int M, void* y, int ldy, int out_mode) {
  QmmEpilogue ep;
  ep.mode = out_mode;
  ep.y = y;
  ep.ldy = ldy;
  return launch_qmm_ex(c, W, expert, a, M, ep);
}

static int qmat_alloc(ih_ctx* c, ih_qmat* q) {
  const size_t tiles = size_t(q->E) * (q->Npad / 16) * q->nkb;
  q->wbytes = tiles * 1024;
  q->sbytes = tiles * (q->format == QF_INT4 ? 128 : 64);
  if (hipMalloc(&q->w, q->wbytes) != hipSuccess) return fail(IH_ENOMEM, "qmat: weight allocation failed");
  if (hipMalloc(&q->s, q->sbytes) != hipSuccess) return fail(IH_ENOMEM, "qmat: scale allocation failed");
  return IH_OK;
}

int pack_int4(ih_ctx* c, ih_qmat* q, const uint32_t* w, const uint16_t* s, const uint16_t* b) {
  dim3 grid((q->Npad / 16) * q->nkb, q->E);
  pack_int4_kernel<<<grid, 64, 0, c->stream>>>(w, s, b, static_cast<uint4*>(q->w), static_cast<uint2*>(q->s), q->N,
                                               q->K, q->Npad, q->nkb, q->il8);
  IH_HIP(hipGetLastError());
  return IH_OK;
}

static ih_qmat* new_qmat_int4(ih_ctx* c, int E, int N, int K) {
  ih_qmat* q = new ih_qmat();
  q->ctx = c;
  q->format = QF_INT4;
  q->E = E;
  q->N = N;
  q->K = K;
  q->Npad = (N + 255) / 256 * 256;
  q->nkb = (K + KBLK - 1) / KBLK;
  q->ktail = (K % KBLK) ? 1 : 0;
  q->algo_bytes = size_t(N) * K / 2 + size_t(N) * (K / 64) * 4;
  return q;
}

int qmat_int4_create_dev(ih_ctx* c, const void* w, const void* s, const void* b, int E, int N, int K, int il8,
                         ih_qmat** out) {
  IH_CHECK(c && w && s && b && out, IH_EINVAL, "ih_qmat_int4_create_dev: null argument");
  IH_CHECK(E >= 1 && N >= 1 && K >= 64 && K % 64 == 0, IH_EINVAL,
           "ih_qmat_int4_create_dev: need E, N >= 1 and K a positive multiple of 64");
  IH_CHECK(!il8 || N % 16 == 0, IH_EINVAL, "qmat: an interleaved gate|up matrix needs N a multiple of 16");
  *out = nullptr;
  ih_qmat* q = new_qmat_int4(c, E, N, K);
  q->il8 = il8;
  int st = qmat_alloc(c, q);
  if (st == IH_OK) st = pack_int4(c, q, static_cast<const uint32_t*>(w), static_cast<const uint16_t*>(s),
                                  static_cast<const uint16_t*>(b));
  if (st != IH_OK) {
    ih_qmat_free(q);
    return st;
  }
  *out = q;
  return IH_OK;
}

}  // namespace ih

using namespace ih;

extern "C" {

int ih_qmat_int4_create_dev(ih_ctx* c, const void* w, const void* s, const void* b, int E, int N, int K,
                            ih_qmat** out) {
  return qmat_int4_create_dev(c, w, s, b, E, N, K, 0, out);
}

int ih_qmat_int4_create(ih_ctx* c, const uint32_t* w, const uint16_t* s, const uint16_t* b, int E, int N, int K,
                        ih_qmat** out) {
  IH_CHECK(c && w && s && b && out, IH_EINVAL, "ih_qmat_int4_create: null argument");
  IH_CHECK(E >= 1 && N >= 1 && K >= 64 && K % 64 == 0, IH_EINVAL,
           "ih_qmat_int4_create: need E, N >= 1 and K a positive multiple of 64");
  const size_t wb = size_t(E) * N * (K / 8) * 4, sb = size_t(E) * N * (K / 64) * 2;
  void *dw = nullptr, *ds = nullptr, *db = nullptr;
  int st = IH_OK;
  if (hipMalloc(&dw, wb) != hipSuccess || hipMalloc(&ds, sb) != hipSuccess || hipMalloc(&db, sb) != hipSuccess)
    st = fail(IH_ENOMEM, "ih_qmat_int4_create: staging allocation failed");
  if (st == IH_OK && (hipMemcpyAsync(dw, w, wb, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
                      hipMemcpyAsync(ds, s, sb, hipMemcpyHostToDevice, c->stream) != hipSuccess ||
                      hipMemcpyAsync(db, b, sb, hipMemcpyHostToDevice, c->stream) != hipSuccess))
    st = fail(IH_EDEVICE, "ih_qmat_int4_create: upload failed");
  if (st == IH_OK) st = ih_qmat_int4_create_dev(c, dw, ds, db, E, N, K, out);
  (void)hipStreamSynchronize(c->stream);
  if (dw) (void)hipFree(dw);
  if (ds) (void)hipFree(ds);
  if (db) (void)hipFree(db);
  return st;
}

int ih_qmat_free(ih_qmat* q) {
  if (!q) return IH_OK;
  if (q->ctx) (void)hipStreamSynchronize(q->ctx->stream);
  if (q->w) (void)hipFree(q->w);
  if (q->s) (void)hipFree(q->s);
  delete q;
  return IH_OK;
}

size_t ih_qmat_bytes(const ih_qmat* q) { return q ? q->algo_bytes * q->E : 0; }

int ih_qmm_shape_override(ih_ctx* c, int N, int K, int R, int KW, int kpw) {
  IH_CHECK(c && N >= 1 && K >= 64, IH_EINVAL, "ih_qmm_shape_override: null context or empty matrix");
  IH_CHECK(R >= 0 && KW >= 0 && kpw >= 0, IH_EINVAL, "ih_qmm_shape_override: negative shape");
  auto& v = c->qmm_shapes;
  for (size_t i = 0; i < v.size();) {
    if (v[i][0] == N && v[i][1] == K) v.erase(v.begin() + i);
    else ++i;
  }
  if (R > 0) v.push_back({N, K, R, KW, kpw, 0});
  ++c->gen;  // recorded steps launched the previous shapes
  return IH_OK;
}

int ih_qmm_int4(ih_ctx* c, const ih_qmat* W, const void* x, int ldx, int M, void* y, int ldy, int out_mode) {
  IH_CHECK(c && W && x && y, IH_EINVAL, "ih_qmm_int4: null argument");
  IH_CHECK(M >= 1 && M <= MAX_TOK, IH_EINVAL, "ih_qmm_int4: M must be in 1..32");
  IH_CHECK(ldx >= W->K && ldy >= W->N, IH_EINVAL, "ih_qmm_int4: leading dimension smaller than the row");
  IH_CHECK(out_mode >= 0 && out_mode <= 2, IH_EINVAL, "ih_qmm_int4: out_mode must be 0, 1 or 2");
  IH_CHECK(W->E == 1, IH_EINVAL, "ih_qmm_int4: stacked experts need the gathered entry point");
  return launch_qmm_rows(c, W, static_cast<const uint16_t*>(x), ldx, M, y, ldy, out_mode);
}

}  // extern "C"
