// FlashAttention-2 backward, FP32, CDNA4 MFMA: three atomics-free stages.
//
// Semantics follow Transformer_kernels/flash_attention.cuh:175-504:
//   delta_i = sum_d O_id dO_id                                   (:175-213)
//   P_ij = e^{S_ij - L_i},  dP_ij = dO_i . v_j,  dS_ij = P_ij (dP_ij - delta_i)
//   dQ_i = s * sum_j dS_ij k_j                                   (:216-354)
//   dV_j = sum_i P_ij dO_i,  dK_j = s * sum_i dS_ij q_i          (:357-504)
// with S = s q.k, s = 1/sqrt(hs), and the causal mask j > i.  Each output row is owned by
// exactly one lane, so there are no atomics and results are deterministic.
//
// gfx950 design (same MFMA layout trick as the forward kernel):
//  * dQ stage: a wave owns 32 query rows and keeps q, dO, L and delta of its rows in
//    registers.  It computes S^T = K Q^T and dP^T = V dO^T (one query row per lane), forms
//    dS^T in registers and feeds it straight into dQ^T += K^T dS^T.
//  * dK/dV stage: a wave owns 32 key rows and keeps k and v in registers, as three bfloat16
//    parts (all its products run on the BF16 matrix pipe, split_bf16.hpp).  It computes
//    S = Q K^T and dP = dO V^T (one key row per lane) and feeds P and dS straight into
//    dV^T += dO^T P and dK^T += Q^T dS.  Unlike the reference, causal tiles above the
//    diagonal are skipped here too (the reference computes kvEnd but never uses it).
//  * dQ streams K and V global -> registers -> LDS, double buffered, one barrier per tile;
//    dK/dV streams Q, dO, L and delta global -> LDS and splits each stage in LDS.
//
// Stored-dS schedule (cta_flash_attention_bwd given a workspace): the reference's dQ stage
// recomputes S and dP, so the three stages run seven tile GEMMs.  With HBM to spare, the
// dK/dV kernel also writes every 32x32 dS tile it forms to a workspace, transposed through
// LDS into the order the dQ kernel reads, and a lean dQ kernel computes dQ = s * dS K from
// it: five GEMMs, still without atomics and bitwise deterministic.  The workspace holds
// whole heads (the lower-triangular tiles only when causal); heads are processed in chunks
// when the caller's workspace cannot hold them all.
#include "cta_common.hpp"
#include "split_bf16.hpp"

namespace cta {
namespace {

struct RowStrides {
  int64_t b, h, t;
};
struct LStrides {
  int64_t b, h, t;
};

// ------------------------------------------------------------------------------------
// Stage 1: delta.  G = hs/4 lanes share one row (one float4 each).
template <int HS>
__global__ __launch_bounds__(256) void fa2_bwd_delta_kernel(const float* __restrict__ O,
                                                            const float* __restrict__ dO,
                                                            float* __restrict__ delta, int nh,
                                                            int T, int64_t rows, RowStrides so,
                                                            RowStrides sdo) {
  constexpr int G = HS / 4;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = gid / G;
  const int c4 = (int)(gid % G);
  float acc = 0.0f;
  if (row < rows) {
    const int64_t bh = row / T;
    const int t = (int)(row - bh * T);
    const int64_t b = bh / nh, h = bh - b * nh;
    const float4 o = ld4(O + b * so.b + h * so.h + (int64_t)t * so.t + 4 * c4);
    const float4 g = ld4(dO + b * sdo.b + h * sdo.h + (int64_t)t * sdo.t + 4 * c4);
    acc = o.x * g.x + o.y * g.y + o.z * g.z + o.w * g.w;
  }
#pragma unroll
  for (int off = G / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
  if (row < rows && c4 == 0) delta[row] = acc;
}

template <int HS>
struct BwdTile;
template <> struct BwdTile<32> { static constexpr int BN = 64; static constexpr int MINW = 2; };
template <> struct BwdTile<64> { static constexpr int BN = 64; static constexpr int MINW = 2; };
template <> struct BwdTile<128> { static constexpr int BN = 32; static constexpr int MINW = 1; };

// Waves per SIMD that the dK/dV stage's registers are held to: k's and v's parts and two
// accumulator sets are 160 registers at hs 64, 320 at hs 128.
template <int HS>
constexpr int kDkdvMinWaves = HS == 128 ? 1 : 2;

// ------------------------------------------------------------------------------------
// Stage 2: dQ.  Workgroup = 128 query rows; K/V tiles streamed through LDS.
// FORM_DELTA: the kernel forms delta = rowsum(O dO) from its own rows (O through strides so),
// with fa2_bwd_delta_kernel's products and summation order (the same bits), uses it and writes
// it for the dK/dV stage that follows; otherwise it reads delta.
template <int HS, bool CAUSAL, bool FORM_DELTA = false>
__global__ __launch_bounds__(256, BwdTile<HS>::MINW) void fa2_bwd_dq_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    const float* __restrict__ dO, const float* __restrict__ Lg, float* __restrict__ delta,
    float* __restrict__ dQ, int nh, int T, int BH, int n_qtiles, RowStrides sq, RowStrides sk,
    RowStrides sv, RowStrides sdo, LStrides sl, RowStrides sdq, float scale, float scale_log2,
    const float* __restrict__ Og = nullptr, RowStrides so = {}, int heads_per_xcd = 0) {
  constexpr int BN = BwdTile<HS>::BN;
  constexpr int BM = 128;
  constexpr int H2 = HS / 2;
  constexpr int KP = HS + 4;  // both K and V rows are read as 16-byte row segments
  constexpr int TILE = BN * KP;
  constexpr int F4_ROW = HS / 4;
  constexpr int LOADS = BN * F4_ROW / 256;
  static_assert(BN * F4_ROW % 256 == 0, "tile must split evenly over 256 threads");
  __shared__ __attribute__((aligned(16))) float smem[2 * 2 * TILE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = wave_index();
  const int half = lane >> 5, col = lane & 31;
  // Head-major items over XCDs; causal items are query-tile pairs (n-1-p, p) of equal cost, or
  // (heads_per_xcd > 0) single query tiles longest first per XCD (lpt_tile).
  int bh, qa, qb = -1;  // the item's query tiles, in pass order (qb < 0: one pass)
  if (CAUSAL && heads_per_xcd > 0) {
    int rank;
    lpt_tile(blockIdx.x, heads_per_xcd, bh, rank);
    qa = n_qtiles - 1 - rank;
  } else {
    const int per_head = CAUSAL ? (n_qtiles + 1) / 2 : n_qtiles;
    const int w = xcd_work_item(blockIdx.x, BH * per_head);
    if (w >= BH * per_head) return;
    bh = w / per_head;
    const int p = w - bh * per_head;
    qa = CAUSAL ? n_qtiles - 1 - p : p;
    if (CAUSAL && n_qtiles - 1 - p != p) qb = p;
  }
  const int b = bh / nh, h = bh - b * nh;

  const float* Kb = K + b * sk.b + h * sk.h;
  const float* Vb = V + b * sv.b + h * sv.h;

  const int n_pass = qb >= 0 ? 2 : 1;
  for (int pass = 0; pass < n_pass; ++pass) {
  const int qt = pass == 0 ? qa : qb;
  const int i0 = qt * BM + wave * 32;
  const int my_i = i0 + col;

  float qf[H2], dof[H2];
  float l2 = 0.0f, dl = 0.0f;  // L_i * log2(e) and delta_i of this lane's row
  float part[FORM_DELTA ? H2 / 4 : 1];  // delta's per-chunk products (FORM_DELTA)
  if (my_i < T) {
    const float* qp = Q + b * sq.b + h * sq.h + (int64_t)my_i * sq.t + half * H2;
    const float* gp = dO + b * sdo.b + h * sdo.h + (int64_t)my_i * sdo.t + half * H2;
#pragma unroll
    for (int c = 0; c < H2 / 4; ++c) {
      const float4 x = ld4(qp + 4 * c);
      const float4 g = ld4(gp + 4 * c);
      qf[4 * c + 0] = x.x; qf[4 * c + 1] = x.y; qf[4 * c + 2] = x.z; qf[4 * c + 3] = x.w;
      dof[4 * c + 0] = g.x; dof[4 * c + 1] = g.y; dof[4 * c + 2] = g.z; dof[4 * c + 3] = g.w;
    }
    l2 = Lg[b * sl.b + h * sl.h + (int64_t)my_i * sl.t] * kLog2e;
    if constexpr (FORM_DELTA) {
      // The delta kernel's per-float4 products (chunk c = half * H2/4 + u of the row), then its
      // xor tree over chunks: offset H2/4 pairs the two wave halves, the smaller ones chunks
      // u and u ^ off of this lane.
      const float* op = Og + b * so.b + h * so.h + (int64_t)my_i * so.t + half * H2;
#pragma unroll
      for (int c = 0; c < H2 / 4; ++c) {
        const float4 o = ld4(op + 4 * c);
        const float4 g = make_float4(dof[4 * c], dof[4 * c + 1], dof[4 * c + 2], dof[4 * c + 3]);
        part[c] = o.x * g.x + o.y * g.y + o.z * g.z + o.w * g.w;
      }
    } else {
      dl = delta[(int64_t)bh * T + my_i];
    }
  } else {
#pragma unroll
    for (int c = 0; c < H2; ++c) { qf[c] = 0.0f; dof[c] = 0.0f; }
  }
  if constexpr (FORM_DELTA) {
    // Rows past T: every chunk 0 (both halves take part in the exchange).
#pragma unroll
    for (int c = 0; c < H2 / 4; ++c) {
      if (my_i >= T) part[c] = 0.0f;
      part[c] = part[c] + xor32(part[c]);
    }
#pragma unroll
    for (int off = H2 / 8; off >= 1; off >>= 1)
#pragma unroll
      for (int c = 0; c < off; ++c) part[c] = part[c] + part[c + off];
    dl = part[0];
    if (my_i < T && half == 0) delta[(int64_t)bh * T + my_i] = dl;
  }

  f32x16 dqacc[HS / 32];
#pragma unroll
  for (int d = 0; d < HS / 32; ++d) dqacc[d] = zero16();

  const int kv_end = CAUSAL ? min(T, (qt + 1) * BM) : T;
  const int n_stages = (kv_end + BN - 1) / BN;

  float4 kst[LOADS], vst[LOADS];
  // K/V rows of a stage through buffer resources over its valid rows: past T they read zero.
  auto gload = [&](int stage) {
    const int j0 = stage * BN;
    const int rows = min(BN, T - j0);
    const __amdgpu_buffer_rsrc_t rk = rows_rsrc(Kb + (int64_t)j0 * sk.t, rows, sk.t, HS);
    const __amdgpu_buffer_rsrc_t rv = rows_rsrc(Vb + (int64_t)j0 * sv.t, rows, sv.t, HS);
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int f = tid + 256 * u;
      const int r = f / F4_ROW, c4 = f % F4_ROW;
      kst[u] = ld4_buffer(rk, (r * (int)sk.t + 4 * c4) * 4);
      vst[u] = ld4_buffer(rv, (r * (int)sv.t + 4 * c4) * 4);
    }
  };
  auto lstore = [&](int buf) {
    float* ks = smem + buf * 2 * TILE;
    float* vs = ks + TILE;
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int f = tid + 256 * u;
      const int r = f / F4_ROW, c4 = f % F4_ROW;
      st4(ks + r * KP + 4 * c4, kst[u]);
      st4(vs + r * KP + 4 * c4, vst[u]);
    }
  };

  gload(0);
  lstore(0);
  __syncthreads();

  for (int s = 0; s < n_stages; ++s) {
    const int buf = s & 1;
    if (s + 1 < n_stages) gload(s + 1);
    const float* ks = smem + buf * 2 * TILE;
    const float* vs = ks + TILE;

#pragma unroll
    for (int sub = 0; sub < BN / 32; ++sub) {
      const int jj0 = s * BN + sub * 32;
      if (jj0 >= T) continue;
      if (CAUSAL && jj0 > i0 + 31) continue;

      f32x16 sacc = zero16(), pacc = zero16();
      const float* krow = ks + (sub * 32 + col) * KP + half * H2;
      const float* vrow = vs + (sub * 32 + col) * KP + half * H2;
#pragma unroll
      for (int c = 0; c < H2 / 4; ++c) {
        const float4 kv = ld4(krow + 4 * c);
        const float4 vv = ld4(vrow + 4 * c);
        sacc = mfma32(kv.x, qf[4 * c + 0], sacc);
        pacc = mfma32(vv.x, dof[4 * c + 0], pacc);
        sacc = mfma32(kv.y, qf[4 * c + 1], sacc);
        pacc = mfma32(vv.y, dof[4 * c + 1], pacc);
        sacc = mfma32(kv.z, qf[4 * c + 2], sacc);
        pacc = mfma32(vv.z, dof[4 * c + 2], pacc);
        sacc = mfma32(kv.w, qf[4 * c + 3], sacc);
        pacc = mfma32(vv.w, dof[4 * c + 3], pacc);
      }

      const bool need_mask = (CAUSAL && jj0 + 31 > i0) || (jj0 + 32 > T);
      // dS^T (overwrites sacc): P (dP - delta), masked entries give exactly 0.
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float p = fast_exp2(fmaf(sacc[r], scale_log2, -l2));
        if (need_mask) {
          const int j = jj0 + mfma_row(r, half);
          if ((CAUSAL && j > my_i) || j >= T) p = 0.0f;
        }
        sacc[r] = p * (pacc[r] - dl);
      }

      // K^T operand (key row R(kk, half), column d*32 + col) from a lane base pointer.
      const float* kcol = ks + (sub * 32 + 4 * half) * KP + col;
#pragma unroll
      for (int kk = 0; kk < 16; ++kk) {
#pragma unroll
        for (int d = 0; d < HS / 32; ++d)
          dqacc[d] = mfma32(kcol[(8 * (kk >> 2) + (kk & 3)) * KP + d * 32], sacc[kk], dqacc[d]);
      }
    }

    if (s + 1 < n_stages) lstore(buf ^ 1);
    __syncthreads();
  }

  if (my_i < T) {
    float* op = dQ + b * sdq.b + h * sdq.h + (int64_t)my_i * sdq.t;
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int dc = d * 32 + 8 * g + 4 * half;
        st4(op + dc, make_float4(dqacc[d][4 * g + 0] * scale, dqacc[d][4 * g + 1] * scale,
                                 dqacc[d][4 * g + 2] * scale, dqacc[d][4 * g + 3] * scale));
      }
    }
  }
  }  // pass
}

// ------------------------------------------------------------------------------------
// Stored dS tiles (ds_tile_index, cta_common.hpp).  An FP32 tile holds its 1024 floats in the
// order of the wave that consumes it: lane l = 32*h + c reads float4 g at offset 256*g + 4*l,
// which holds dS[32*ib + c][32*jb + 8*g + 4*h + e] for e = 0..3 — the B operand of the
// 32x32x2 MFMA for contraction steps kk = 4*g + e.
constexpr int kDsTileFloats = 1024;
constexpr int kDsPitch = 40;  // LDS pitch of the per-wave transpose: halves 4 rows apart hit disjoint banks

// The matrix pipe rounds small addends of a large accumulator downward.  The six products of parts
// summed over a head of T = 8192 left dQ and dK a mean error of -2.9e-7 of their RMS, which sums
// over the tokens (bias gradients) show as 18 times what independent roundings leave.  So the
// stages enter the sum with one sign for kFlipRows rows and the other for the next: the sum is
// negated in between, and what was rounded down in one run is rounded up in the next (8e-9).  dP's
// own sums, short but cancelling against delta, take theirs from the block of 32 keys.  (Summing
// each tile apart and adding it in FP32 has the same effect; its registers cost dK/dV 5-12%.)
constexpr int kFlipRows = 256;

// ------------------------------------------------------------------------------------
// Stage 3: dK, dV.  Workgroup = 128 key rows, each of its four waves owning 32 of them and each
// lane one key row's k and v, as three bfloat16 parts in registers.  All four products run on
// the BF16 matrix pipe (split_bf16.hpp; six products of parts, smallest first): 3072 matrix
// cycles per 32x32 tile at hs 64 where the FP32 MFMA takes 8192, which it kept 85% busy.
//
// Q, dO (O), L and delta stream through LDS in stages of 32 query rows: copied global -> LDS in
// FP32 (no staging registers) while the stage before is computed, then split once per workgroup
// into four images in MFMA operand order, Q and dO by rows (S, dP) and by columns (dK, dV).  One
// image set (48 KiB at hs 64) and one FP32 stage leave room for two workgroups a CU, which hide
// each other's two barriers a stage; a second image set would leave one.
// B4 H32 N4096 D64 causal: 4.2 -> 3.2 ms with the dS store (2.7 without), MFMA busy 53% at
// 1.84 GHz; B2 H16 T1999 D128 0.44 ms.  (hs 64 spills 44-60 bytes outside the stage loop.)
// The rest is VALU work (the splits and the softmax, about 600 instructions a tile, in long runs
// between the MFMAs), the barriers and the chip's power limit.
//
// Heads [bh_base, bh_base + BH) are processed; with STORE_DS every dS tile is also written
// to dsw (heads indexed from bh_base), transposed through LDS half a tile at a time.
//
// FOLD: delta is not read from a delta stage's output but computed here, per query stage, from
// the stage's dO tile and an O tile streamed beside it (delta_i = O_i . dO_i, the reference's
// flash_attention_bwd_delta, flash_attention.cuh:175-213, folded in).  Every key tile of a head
// recomputes it.
//
// SPLIT: each work item (key-tile pair, or tile) is run by two workgroups, part 0 and part 1,
// each over one half of the item's query stages (in the item's stage order, across its passes);
// every dS tile is still stored once, by the part that forms it.  Part 0 writes its partial dK
// and dV to dK / dV, part 1 densely to part_ws (dK, then dV, of all BH heads); zeros where a
// part saw no query stage.  fa2_bwd_dkdv_sum_kernel then adds part 1 to part 0.
//
// k, v, P, dS, and Q and dO but for the rows of Q in S, are scaled before they are split, so the
// parts hold every bit of them (split_bf16.hpp; Q's rows: kMaxScoreFactor).  Sums that are not
// finite (infinities, NaN, operands above 2^103, dK or dV above 2^79, dP above 2^79), or |k| above
// kMaxScoreFactor, run the pass again on FP32 MFMAs: a P or dS that is not finite leaves its key's
// dV or dK not finite, so these two are all that is looked at.  With every pass run again the
// backward takes 2.3 to 2.6 times as long.
template <int HS, bool CAUSAL, bool STORE_DS, bool FOLD, bool SPLIT = false>
__global__ __launch_bounds__(256, kDkdvMinWaves<HS>) void fa2_bwd_dkdv_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V,
    const float* __restrict__ dO, const float* __restrict__ O, const float* __restrict__ Lg,
    const float* __restrict__ delta, float* __restrict__ dK, float* __restrict__ dV,
    float* __restrict__ dsw, int nh, int T, int bh_base, int BH, int n_ktiles, RowStrides sq,
    RowStrides sk, RowStrides sv, RowStrides sdo, RowStrides so, LStrides sl, RowStrides sdk,
    RowStrides sdv, float scale, float scale_log2, float* __restrict__ part_ws = nullptr,
    int heads_per_xcd = 0) {
  constexpr int BN = 32, WAVES = 4, THREADS = 64 * WAVES;
  constexpr int BM = 32 * WAVES;  // key rows per workgroup, 32 per wave
  constexpr int TILE = BN * HS;     // an FP32 tile: dense rows (convert reads whole runs of them)
  constexpr int NT = FOLD ? 3 : 2;  // tiles per stage: Q, dO (and O when folding delta)
  constexpr int RPC = 256 / HS;     // rows of a 1 KiB async copy
  constexpr int RVEC = 64;  // L and delta of a stage, each padded to one wave
  // Images, each of three parts: Q by rows, dO by rows, Q by columns, dO by columns, in units of
  // eight values of one part (16 bytes).  By rows: unit (d8, row) = d 8 d8 .. 8 d8 + 7 of a row,
  // at d8 * 32 + (row ^ (d8 & 7)).  By columns: unit (d, sh) = the eight query rows that half
  // sh & 1 takes in step sh >> 1 (16 st + 4 half + 0..3 and + 8..11, the order in which a lane
  // holds P and dS), at (d/32, sh, d % 32).
  constexpr int PART = BN * HS * 2, IMAGE = 3 * PART;
  constexpr int UNITS = BN * HS / 8;  // of one part of one image
  static_assert(4 * UNITS % THREADS == 0 && UNITS % 64 == 0, "whole waves share an image");
  constexpr int XPOSE = STORE_DS ? WAVES * 16 * kDsPitch : 0;
  __shared__ __attribute__((aligned(16))) char images[4 * IMAGE];
  __shared__ __attribute__((aligned(16))) float raw[NT * TILE];
  __shared__ __attribute__((aligned(16))) float rvec[2][2 * RVEC];  // by parity of the step
  __shared__ __attribute__((aligned(16))) float xpose_all[XPOSE > 0 ? XPOSE : 4];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = wave_index();
  const int half = lane >> 5, col = lane & 31;
  // Head-major items over XCDs; causal items are key-tile pairs (p, n-1-p) of equal cost, or
  // (heads_per_xcd > 0, unsplit) single key tiles longest first per XCD (lpt_tile).
  int bh_local, part = 0;
  int ka, kb = -1;  // the item's key tiles, in pass order (kb < 0: one pass)
  if (CAUSAL && !SPLIT && heads_per_xcd > 0) {
    lpt_tile(blockIdx.x, heads_per_xcd, bh_local, ka);  // key tile 0 is the longest
  } else {
    const int per_head = CAUSAL ? (n_ktiles + 1) / 2 : n_ktiles;
    const int n_items = BH * per_head * (SPLIT ? 2 : 1);
    const int w = xcd_work_item(blockIdx.x, n_items);
    if (w >= n_items) return;
    const int item = SPLIT ? w >> 1 : w;
    part = SPLIT ? w & 1 : 0;  // the two parts of an item are neighbours: one XCD
    bh_local = item / per_head;
    const int p = item - bh_local * per_head;
    ka = p;
    if (CAUSAL && n_ktiles - 1 - p != p) kb = n_ktiles - 1 - p;
  }
  const int bh = bh_base + bh_local;
  const int b = bh / nh, h = bh - b * nh;

  const float* Qb = Q + b * sq.b + h * sq.h;
  const float* Kb = K + b * sk.b + h * sk.h;
  const float* Vb = V + b * sv.b + h * sv.h;
  const float* dOb = dO + b * sdo.b + h * sdo.h;
  const float* Ob = FOLD ? O + b * so.b + h * so.h : nullptr;
  const float* Lb = Lg + b * sl.b + h * sl.h;
  const float* Db = FOLD ? nullptr : delta + (int64_t)bh * T;
  const int nb = (T + 31) / 32;
  // Byte offset of this lane's 16 bytes in a copy's first row, for the tile's row stride.
  auto lane_off = [&](int64_t st) { return ((lane * 4 / HS) * (int)st + lane * 4 % HS) * 4; };
  const int off_q = lane_off(sq.t), off_g = lane_off(sdo.t), off_o = FOLD ? lane_off(so.t) : 0;
  float* xpose = xpose_all + (STORE_DS ? wave * 16 * kDsPitch : 0);  // this wave's half dS tile
  float* dsh = STORE_DS ? dsw + (int64_t)bh_local * ds_tiles_per_head(T, CAUSAL) * kDsTileFloats
                        : nullptr;

  // The FP32 stage starts as zeros, so the rows that no copy writes are finite.
#pragma unroll 4
  for (int e = 4 * tid; e < NT * TILE; e += 4 * THREADS) st4(raw + e, zero4());
  __syncthreads();

  const int n_pass = kb >= 0 ? 2 : 1;
  auto kt_of = [&](int pass) { return pass == 0 ? ka : kb; };
  const int n_stages = (T + BN - 1) / BN;
  // first query stage that can see the keys of tile kt
  auto q_begin_of = [&](int kt) { return CAUSAL ? (kt * BM / BN) : 0; };
  // SPLIT: this part's positions [g0, g1) in the item's list of steps (pass 0's, then pass 1's).
  int g0 = 0, g1 = 0, pos = 0;
  if constexpr (SPLIT) {
    int total = 0;
    for (int pass = 0; pass < n_pass; ++pass) total += n_stages - q_begin_of(kt_of(pass));
    g0 = part ? (total + 1) / 2 : 0;
    g1 = part ? total : (total + 1) / 2;
  }
  int slot = 0;  // which of rvec the coming step reads
  for (int pass = 0; pass < n_pass; ++pass) {
  const int kt = kt_of(pass);
  const int j0 = kt * BM + wave * 32;  // first key row of this wave
  const int my_j = j0 + col;

  // k's and v's parts, the B operands of S and dP: step st, d 16 st + 8 half + 0..7.
  // v takes a sign that alternates over the blocks of 32 keys, and with it dP (kFlipRows).
  bf16x8 kp[HS / 16][3], vp[HS / 16][3];
  float kmax = 0.0f;
  const float v_sign = (j0 >> 5) & 1 ? -1.0f : 1.0f;
#pragma unroll
  for (int st = 0; st < HS / 16; ++st) {
    auto load = [&](const float* src, float sign, bf16x8 (&p)[3]) {
      const float4 x = my_j < T ? ld4(src) : zero4(), y = my_j < T ? ld4(src + 4) : zero4();
      const float v[8] = {sign * x.x, sign * x.y, sign * x.z, sign * x.w,
                          sign * y.x, sign * y.y, sign * y.z, sign * y.w};
      split_bf16<true>(v, p);
      float m = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) m = fmaxf(fmaxf(m, fabsf(v[e])), fabsf(v[e + 1]));
      return m;
    };
    kmax = fmaxf(kmax, load(Kb + (int64_t)my_j * sk.t + 16 * st + 8 * half, 1.0f, kp[st]));
    load(Vb + (int64_t)my_j * sv.t + 16 * st + 8 * half, v_sign, vp[st]);
  }
  // The pass runs again on FP32 MFMAs.  (The vote is taken here: left to the end of the pass, it
  // would keep k in registers.)
  bool odd = __any(kmax >= kMaxScoreFactor);

  f32x16 dkacc[HS / 32], dvacc[HS / 32];
#pragma unroll
  for (int d = 0; d < HS / 32; ++d) { dkacc[d] = zero16(); dvacc[d] = zero16(); }

  const int q_begin = q_begin_of(kt);

  // Async copies of a stage into the FP32 tiles.  Each tile is read through a buffer resource
  // over its valid rows (base and extent are scalar), so the lane's offset serves every copy; rows past T are out of range and leave finite rows in LDS, masked to P = 0.
  auto issue = [&](int stage, float* rv) {
    const int r0 = stage * BN;
    const int rows = min(BN, T - r0);
    auto copy = [&](const float* base, int64_t st, int off, float* tile) {
      const __amdgpu_buffer_rsrc_t rs = rows_rsrc(base + (int64_t)r0 * st, rows, st, HS);
#pragma unroll
      for (int u = 0; u < BN / RPC / WAVES; ++u) {
        const int pc = wave + WAVES * u;
        async_copy16_buffer(rs, off + pc * RPC * (int)st * 4, tile + pc * 256);
      }
    };
    copy(Qb, sq.t, off_q, raw);
    copy(dOb, sdo.t, off_g, raw + TILE);
    if (FOLD) copy(Ob, so.t, off_o, raw + 2 * TILE);
    if (wave == 0) {  // lanes past BN fill the padding
      const int64_t i = min(r0 + lane, T - 1);
      async_copy4(Lb + i * sl.t, rv);
      if (!FOLD) async_copy4(Db + i, rv + RVEC);
    }
  };
  // The four images from the FP32 tiles, one unit (three parts) at a time.
  auto convert = [&]() {
#pragma unroll
    for (int u = 0; u < 4 * UNITS / THREADS; ++u) {
      // unit f of image img: a constant where a step of the workgroup stays in one image
      const int img = UNITS >= THREADS
                          ? THREADS * u / UNITS
                          : THREADS / UNITS * u + __builtin_amdgcn_readfirstlane(tid / UNITS);
      const int f = UNITS >= THREADS ? tid + THREADS * u % UNITS : tid % UNITS;
      const float* src = raw + (img & 1) * TILE;
      float x[8];
      int at;
      if (img < 2) {
        const int r = f / (HS / 8), d8 = f % (HS / 8);
        const float4 lo = ld4(src + r * HS + 8 * d8), hi = ld4(src + r * HS + 8 * d8 + 4);
        x[0] = lo.x; x[1] = lo.y; x[2] = lo.z; x[3] = lo.w;
        x[4] = hi.x; x[5] = hi.y; x[6] = hi.z; x[7] = hi.w;
        at = d8 * 32 + (r ^ (d8 & 7));
      } else {
        const int d = f % HS, sh = f / HS;
        const float* c = src + (16 * (sh >> 1) + 4 * (sh & 1)) * HS + d;
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = c[(8 * (j >> 2) + (j & 3)) * HS];
        at = (d >> 5) * 128 + sh * 32 + (d & 31);
      }
      bf16x8 p[3];
      if (img == 0) split_bf16(x, p);
      else split_bf16<true>(x, p);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        *reinterpret_cast<bf16x8*>(images + img * IMAGE + q * PART + at * 16) = p[q];
    }
  };
  // FOLD: delta of the stage from its O and dO tiles, THREADS / BN lanes per row.  Rows past T
  // are masked (P = 0).
  auto fold_delta = [&](float* rv) {
    constexpr int LPR = THREADS / BN;  // lanes per row (consecutive lanes of one wave)
    constexpr int DPL = HS / LPR;      // d values per lane
    static_assert(THREADS % BN == 0 && DPL % 4 == 0 && LPR <= 64, "delta split");
    const int r = tid / LPR, seg = tid % LPR;
    const float* orow = raw + 2 * TILE + r * HS + seg * DPL;
    const float* grow = raw + TILE + r * HS + seg * DPL;
    float acc = 0.0f;
#pragma unroll
    for (int c = 0; c < DPL / 4; ++c) {
      const float4 o4 = ld4(orow + 4 * c), g4 = ld4(grow + 4 * c);
      acc = fmaf(o4.x, g4.x, acc);
      acc = fmaf(o4.y, g4.y, acc);
      acc = fmaf(o4.z, g4.z, acc);
      acc = fmaf(o4.w, g4.w, acc);
    }
#pragma unroll
    for (int off = LPR / 2; off >= 1; off >>= 1) acc += __shfl_xor(acc, off);
    if (seg == 0) rv[RVEC + r] = acc;
  };
  // Tiles whose every query row precedes every key row, or without a key row, are skipped (dS = 0,
  // nothing stored).
  auto live = [&](int ii0) { return j0 < T && !(CAUSAL && ii0 + 31 < j0); };
  // S (query rows ii0 + R(r, half), key my_j) -> y P, P = e^{S - L} = 2^{S c - L log2(e)}, with
  // the rows' L log2(e) in ls; masked entries and key rows past T give exactly 0.
  auto probabilities = [&](f32x16& sacc, int ii0, const float* ls, float c, float y) {
    // A separate block behind a wave-uniform branch: inside the exponential loop the test is
    // if-converted into per-element predication that every tile pays for.
    if ((CAUSAL && ii0 < j0 + 31) || (ii0 + 32 > T) || (j0 + 32 > T)) {
      asm volatile("");  // a side effect keeps the block from being speculated into selects
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int i = ii0 + mfma_row(r, half);
        if ((CAUSAL && my_j > i) || i >= T || my_j >= T) sacc[r] = -INFINITY;
      }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 lv = ld4(ls + 8 * g + 4 * half);
      const float lr[4] = {lv.x, lv.y, lv.z, lv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sacc[4 * g + e] = y * fast_exp2(fmaf(sacc[4 * g + e], c, -lr[e]));
    }
  };
  // dP -> y dS = y P (dP u - delta), y and u powers of two.  Rounded to FP32 before it is split:
  // fused into the split's first subtraction (where nothing stores dS) it would give the schedules
  // different bits.
  auto score_gradients = [&](const f32x16& p, f32x16& pacc, const float* ds, float u) {
#pragma clang fp contract(off)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 dv = ld4(ds + 8 * g + 4 * half);
      const float dr[4] = {dv.x, dv.y, dv.z, dv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e)
        pacc[4 * g + e] = p[4 * g + e] * fmaf(pacc[4 * g + e], u, -dr[e]);
    }
  };
  // Lane (col, half) holds dS[ii0 + R(r, half)][j0 + col]: through the wave's transpose buffer
  // as [query][key], 16 queries at a time, and out one query row per lane in whole 256-byte runs.
  // dsv holds dS / u.
  auto store_ds = [&](const f32x16& dsv, int ii0, float u) {
    float* gt = dsh + ds_tile_index(ii0 / 32, j0 / 32, nb, CAUSAL) * kDsTileFloats;
    const int gs = lane >> 5, hs = (lane >> 4) & 1, c = lane & 15;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      wave_lds_fence();
#pragma unroll
      for (int r = 0; r < 8; ++r) xpose[mfma_row(r, half) * kDsPitch + col] = dsv[8 * hh + r] * u;
      wave_lds_fence();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int g = 2 * k + gs;
        st4_stream(gt + 256 * g + 4 * (32 * hs + 16 * hh + c),
                   ld4(xpose + c * kDsPitch + 8 * g + 4 * hs));
      }
    }
    wave_lds_fence();
  };

  // Stage order.  With a causal mask the first (long) pass walks its query stages downward
  // from the last and the second (short) pass upward from its first, so every workgroup of a
  // head in its first pass reads query stage n-1-t at step t and every one in its second pass
  // reads stage t - 4 (t counted from the item's start): the workgroups of a head share each
  // streamed Q / dO stage in L2 instead of each reading it at a different time.
  const int n_steps = n_stages - q_begin;
  // the steps [i_begin, i_end) of this pass that this part runs (all of them unless SPLIT)
  const int i_begin = SPLIT ? min(max(g0 - pos, 0), n_steps) : 0;
  const int i_end = SPLIT ? min(max(g1 - pos, 0), n_steps) : n_steps;
  pos += n_steps;
  // (the long tile of a pair walks down: a property of the tile, so single tiles match pairs)
  const bool down = CAUSAL && kt <= n_ktiles - 1 - kt;
  auto stage_at = [&](int i) { return down ? n_stages - 1 - i : q_begin + i; };
  if (i_begin < i_end) issue(stage_at(i_begin), rvec[slot]);
  constexpr int kFlip = kFlipRows / BN;
  float y = kSplitScale;  // the scale, and now and then the sign, of P and dS in the sums

  for (int run = i_begin; run < i_end; run += kFlip) {
  if (run > i_begin) {
    y = -y;
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) { dkacc[d] = -dkacc[d]; dvacc[d] = -dvacc[d]; }
  }
  for (int i = run; i < min(run + kFlip, i_end); ++i) {
    // the stage's copies have landed, and every wave is done with the images
    vm_wait_all();
    __syncthreads();
    convert();
    float* const rv = rvec[slot];
    if (tid < BN) rv[tid] *= kLog2e;
    if (FOLD) fold_delta(rv);
    slot ^= 1;
    __syncthreads();
    if (i + 1 < i_end) issue(stage_at(i + 1), rvec[slot]);

    const int ii0 = stage_at(i) * BN;
    if (!live(ii0)) continue;

    // S and dP tiles: lane holds column my_j, rows ii0 + R(r, half)
    f32x16 sacc = zero16(), pacc = zero16();
#pragma unroll
    for (int st = 0; st < HS / 16; ++st) {
      const int d8 = 2 * st + half;
      const char* at = images + (d8 * 32 + (col ^ (d8 & 7))) * 16;
      bf16x8 qa[3], ga[3];
#pragma unroll
      for (int q = 2; q >= 0; --q) {
        qa[q] = *reinterpret_cast<const bf16x8*>(at + q * PART);
        ga[q] = *reinterpret_cast<const bf16x8*>(at + IMAGE + q * PART);
      }
#pragma unroll
      for (int p = 0; p < 6; ++p) {
        sacc = mfma_bf16(qa[kSplitA[p]], kp[st][kSplitB[p]], sacc);
        pacc = mfma_bf16(ga[kSplitA[p]], vp[st][kSplitB[p]], pacc);
      }
    }
    // X^T += (image's columns) Y over the 32 query rows, two steps of 16
    auto accumulate = [&](f32x16 (&acc)[HS / 32], const char* image, const f32x16& y) {
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = y[8 * st + e];
        bf16x8 yp[3];
        split_bf16(x, yp);
#pragma unroll
        for (int d0 = 0; d0 < HS / 32; d0 += 2) {
          constexpr int ND = HS / 32 < 2 ? 1 : 2;  // two chains
          bf16x8 a[ND][3];
#pragma unroll
          for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int q = 2; q >= 0; --q)
              a[d][q] = *reinterpret_cast<const bf16x8*>(
                  image + q * PART + ((d0 + d) * 128 + (2 * st + half) * 32 + col) * 16);
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int d = 0; d < ND; ++d)
              acc[d0 + d] = mfma_bf16(a[d][kSplitA[p]], yp[kSplitB[p]], acc[d0 + d]);
        }
      }
    };
    probabilities(sacc, ii0, rv, scale_log2 * kSplitUnscale, y);
    accumulate(dvacc, images + 3 * IMAGE, sacc);
    score_gradients(sacc, pacc, rv + RVEC, v_sign * (kSplitUnscale * kSplitUnscale));
    if (STORE_DS) store_ds(pacc, ii0, y * (kSplitUnscale * kSplitUnscale));
    accumulate(dkacc, images + 2 * IMAGE, pacc);
  }
  }  // run

  y *= kSplitUnscale * kSplitUnscale * kSplitUnscale;
#pragma unroll
  for (int d = 0; d < HS / 32; ++d) {
    odd |= not_finite(dkacc[d]) || not_finite(dvacc[d]);
    dkacc[d] *= y;
    dvacc[d] *= y;
  }
  vm_wait_all();  // dS tiles that a second run stores again are stored in order
  if (__syncthreads_or(odd)) {
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) { dkacc[d] = zero16(); dvacc[d] = zero16(); }
    for (int i = i_begin; i < i_end; ++i) {
      const int ii0 = stage_at(i) * BN;
      float* const rv = rvec[slot];
      __syncthreads();
      for (int f = tid; f < BN * HS / 4; f += THREADS) {
        const int r = f / (HS / 4), c4 = f % (HS / 4) * 4;
        const int64_t t = ii0 + r;
        st4(raw + r * HS + c4, t < T ? ld4(Qb + t * sq.t + c4) : zero4());
        st4(raw + TILE + r * HS + c4, t < T ? ld4(dOb + t * sdo.t + c4) : zero4());
        if (FOLD) st4(raw + 2 * TILE + r * HS + c4, t < T ? ld4(Ob + t * so.t + c4) : zero4());
      }
      if (tid < BN) {
        const int64_t t = min(ii0 + tid, T - 1);
        rv[tid] = Lb[t * sl.t] * kLog2e;
        if (!FOLD) rv[RVEC + tid] = Db[t];
      }
      __syncthreads();
      if (FOLD) {
        fold_delta(rv);
        __syncthreads();
      }
      if (!live(ii0)) continue;
      f32x16 sacc = zero16(), pacc = zero16();
      const int64_t jc = min(my_j, T - 1);
      const float* k = Kb + jc * sk.t + half * (HS / 2);
      const float* v = Vb + jc * sv.t + half * (HS / 2);
      const float* qrow = raw + col * HS + half * (HS / 2);
#pragma unroll 2
      for (int c = 0; c < HS / 2; c += 4) {
        const float4 q4 = ld4(qrow + c), g4 = ld4(qrow + TILE + c), k4 = ld4(k + c), v4 = ld4(v + c);
        sacc = mfma32(q4.x, k4.x, sacc);
        pacc = mfma32(g4.x, v4.x, pacc);
        sacc = mfma32(q4.y, k4.y, sacc);
        pacc = mfma32(g4.y, v4.y, pacc);
        sacc = mfma32(q4.z, k4.z, sacc);
        pacc = mfma32(g4.z, v4.z, pacc);
        sacc = mfma32(q4.w, k4.w, sacc);
        pacc = mfma32(g4.w, v4.w, pacc);
      }
      probabilities(sacc, ii0, rv, scale_log2, 1.0f);
      score_gradients(sacc, pacc, rv + RVEC, 1.0f);
      if (STORE_DS) store_ds(pacc, ii0, 1.0f);
#pragma unroll
      for (int d = 0; d < HS / 32; ++d)
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
          const float* a = raw + mfma_row(kk, half) * HS + d * 32 + col;
          dvacc[d] = mfma32(a[TILE], sacc[kk], dvacc[d]);
          dkacc[d] = mfma32(a[0], pacc[kk], dkacc[d]);
        }
    }
    __syncthreads();
  }

  if (my_j < T) {
    float* dkp = dK + b * sdk.b + h * sdk.h + (int64_t)my_j * sdk.t;
    float* dvp = dV + b * sdv.b + h * sdv.h + (int64_t)my_j * sdv.t;
    if (SPLIT && part) {
      dkp = part_ws + ((int64_t)bh * T + my_j) * HS;
      dvp = dkp + (int64_t)(bh_base + BH) * T * HS;
    }
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int dc = d * 32 + 8 * g + 4 * half;
        st4(dkp + dc, make_float4(dkacc[d][4 * g + 0] * scale, dkacc[d][4 * g + 1] * scale,
                                  dkacc[d][4 * g + 2] * scale, dkacc[d][4 * g + 3] * scale));
        st4(dvp + dc, make_float4(dvacc[d][4 * g + 0], dvacc[d][4 * g + 1], dvacc[d][4 * g + 2],
                                  dvacc[d][4 * g + 3]));
      }
    }
  }
  }  // pass: the check above is a barrier, so the next pass may refill LDS
}

// dK += part 1's dK, dV += part 1's dV, row by row in a fixed order (part 0, then part 1), after
// a split dK/dV stage; dK / dV through their strides, part 1 dense in part_ws.  HS / 4 lanes
// per row, one float4 each.
template <int HS>
__global__ __launch_bounds__(256) void fa2_bwd_dkdv_sum_kernel(float* __restrict__ dK,
                                                               float* __restrict__ dV,
                                                               const float* __restrict__ part_ws,
                                                               int nh, int T, int64_t rows,
                                                               RowStrides sdk, RowStrides sdv) {
  constexpr int G = HS / 4;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = gid / G;
  if (row >= rows) return;
  const int c4 = (int)(gid % G);
  const int64_t bh = row / T;
  const int t = (int)(row - bh * T);
  const int64_t b = bh / nh, h = bh - b * nh;
  float* kp = dK + b * sdk.b + h * sdk.h + (int64_t)t * sdk.t + 4 * c4;
  float* vp = dV + b * sdv.b + h * sdv.h + (int64_t)t * sdv.t + 4 * c4;
  const float4 a = ld4(kp), c = ld4(part_ws + row * HS + 4 * c4);
  const float4 x = ld4(vp), y = ld4(part_ws + (rows + row) * HS + 4 * c4);
  st4(kp, make_float4(a.x + c.x, a.y + c.y, a.z + c.z, a.w + c.w));
  st4(vp, make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w));
}

// dQ += part 1's dQ, row by row (part 0, then part 1), after a split dQ-from-dS stage; dQ
// through its strides, part 1 dense in part_ws.  HS / 4 lanes per row, one float4 each.
template <int HS>
__global__ __launch_bounds__(256) void fa2_bwd_dq_sum_kernel(float* __restrict__ dQ,
                                                             const float* __restrict__ part_ws,
                                                             int nh, int T, int64_t rows,
                                                             RowStrides sdq) {
  constexpr int G = HS / 4;
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t row = gid / G;
  if (row >= rows) return;
  const int c4 = (int)(gid % G);
  const int64_t bh = row / T;
  const int t = (int)(row - bh * T);
  const int64_t b = bh / nh, h = bh - b * nh;
  float* qp = dQ + b * sdq.b + h * sdq.h + (int64_t)t * sdq.t + 4 * c4;
  const float4 a = ld4(qp), c = ld4(part_ws + row * HS + 4 * c4);
  st4(qp, make_float4(a.x + c.x, a.y + c.y, a.z + c.z, a.w + c.w));
}

// ------------------------------------------------------------------------------------
// dQ from stored dS tiles: dQ^T += K^T dS^T, one 32x32 tile per MFMA chain.  Workgroup =
// 32 * WAVES query rows (WAVES = 4, or 2 for short causal heads).  The product runs on the BF16
// matrix pipe, six products of three-part operands (split_bf16.hpp; 768 matrix cycles a tile at
// hs 64, 2048 on the FP32 MFMA).  K stages go global -> registers -> split -> LDS, double
// buffered; each wave streams its own dS tiles from the workspace straight into registers,
// one stage ahead, and splits them there as the B operand.  What bounds it is mostly the read of
// dS, at the chip's power limit: B1 H32 N8192 D64 2.29 -> 1.67-1.89 ms (4.5-5.3 TB/s, MFMA busy 52%),
// B4 H32 N4096 causal 1.26 -> 0.92-0.98 ms.
// A stage is 64 keys, or 32 where two buffers of 64 would hold the CU to fewer than three
// workgroups of four waves (hs 128; two-wave workgroups).  Heads [bh_base, bh_base + BH).
// Operands are scaled before they are split (split_bf16.hpp); sums that are not finite run the pass
// again on FP32 MFMAs.
// SPLIT (small grids, heads from 0): each item's key stages (pass 0's, then pass 1's) are
// split over two workgroups, neighbours in the XCD order; part 0 writes dQ, part 1 its
// partial dQ densely into part_ws, and fa2_bwd_dq_sum_kernel adds the two in that order.
__device__ __forceinline__ float f4_at(const float4& v, int e) {
  return e == 0 ? v.x : e == 1 ? v.y : e == 2 ? v.z : v.w;
}

template <int HS, bool CAUSAL, int WAVES = 4, bool SPLIT = false>
__global__ __launch_bounds__(64 * WAVES, 2) void fa2_bwd_dq_ds_kernel(
    const float* __restrict__ K, const float* __restrict__ dsw, float* __restrict__ dQ, int nh,
    int T, int bh_base, int BH, int n_qtiles, RowStrides sk, RowStrides sdq, float scale,
    float* __restrict__ part_ws = nullptr, int heads_per_xcd = 0) {
  constexpr int BN = HS == 128 || WAVES == 2 ? 32 : 64;
  constexpr int NSUB = BN / 32;
  constexpr int THREADS = 64 * WAVES;
  constexpr int BM = 32 * WAVES;  // query rows per workgroup, 32 per wave
  // LDS image of a K stage in units of eight values of one part (16 bytes): unit (sub, d, sh) =
  // the eight keys of sub's that half sh & 1 takes in step sh >> 1 (16 st + 4 half + 0..3 and
  // + 8..11: the keys of a lane's two dS float4), at (sub, d/32, sh, d % 32).
  constexpr int PART = BN * HS * 2;
  constexpr int STAGE = 3 * PART;
  constexpr int NU = BN * HS / 8 / THREADS;
  static_assert(BN * HS / 8 % THREADS == 0, "units must split evenly over the workgroup");
  constexpr int KP = HS + 8;  // row pitch of the FP32 stage (second run)
  static_assert(BN * KP * 4 <= 2 * STAGE, "the FP32 stage fits");
  __shared__ __attribute__((aligned(16))) char smem[2 * STAGE];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = wave_index();
  const int half = lane >> 5, col = lane & 31;
  // Head-major items over XCDs; causal items are query-tile pairs (n-1-p, p) of equal cost, or
  // (heads_per_xcd > 0, unsplit) single query tiles longest first per XCD (lpt_tile).
  int bh_local, part = 0;
  int qa, qb = -1;  // the item's query tiles, in pass order (qb < 0: one pass)
  if (CAUSAL && !SPLIT && heads_per_xcd > 0) {
    int rank;
    lpt_tile(blockIdx.x, heads_per_xcd, bh_local, rank);
    qa = n_qtiles - 1 - rank;
  } else {
    const int per_head = CAUSAL ? (n_qtiles + 1) / 2 : n_qtiles;
    const int n_items = BH * per_head * (SPLIT ? 2 : 1);
    const int w = xcd_work_item(blockIdx.x, n_items);
    if (w >= n_items) return;
    const int item = SPLIT ? w >> 1 : w;
    part = SPLIT ? w & 1 : 0;
    bh_local = item / per_head;
    const int p = item - bh_local * per_head;
    qa = CAUSAL ? n_qtiles - 1 - p : p;
    if (CAUSAL && n_qtiles - 1 - p != p) qb = p;
  }
  const int bh = bh_base + bh_local;
  const int b = bh / nh, h = bh - b * nh;
  const float* Kb = K + b * sk.b + h * sk.h;
  const int nb = (T + 31) / 32;
  const float* dsh = dsw + (int64_t)bh_local * ds_tiles_per_head(T, CAUSAL) * kDsTileFloats;

  const int n_pass = qb >= 0 ? 2 : 1;
  auto qt_of = [&](int pass) { return pass == 0 ? qa : qb; };
  auto stages_of = [&](int qt) {
    const int kv_end = CAUSAL ? min(T, (qt + 1) * BM) : T;
    return (kv_end + BN - 1) / BN;
  };
  // SPLIT: this part's positions [g0, g1) in the item's list of stages (pass 0's, then pass 1's).
  int g0 = 0, g1 = 0, pos = 0;
  if constexpr (SPLIT) {
    int total = 0;
    for (int pass = 0; pass < n_pass; ++pass) total += stages_of(qt_of(pass));
    g0 = part ? (total + 1) / 2 : 0;
    g1 = part ? total : (total + 1) / 2;
  }
  for (int pass = 0; pass < n_pass; ++pass) {
  const int qt = qt_of(pass);
  const int i0 = qt * BM + wave * 32;
  const int my_i = i0 + col;
  const int ib = i0 / 32;  // query block of this wave

  f32x16 acc[HS / 32];
#pragma unroll
  for (int d = 0; d < HS / 32; ++d) acc[d] = zero16();

  const int n_stages = stages_of(qt);
  // the stages [s_begin, s_end) of this pass that this part runs (all of them unless SPLIT)
  const int s_begin = SPLIT ? min(max(g0 - pos, 0), n_stages) : 0;
  const int s_end = SPLIT ? min(max(g1 - pos, 0), n_stages) : n_stages;
  pos += n_stages;

  // Every stage issues the same loads, unconditionally (K through a buffer resource, dS from
  // clamped in-bounds tiles), and the stage count is padded to even (padded stages compute
  // nothing).  The compiler can then
  // count the loads in flight exactly: the MFMAs of stage s wait only for stage s's dS, not
  // for the stage s+1 loads issued ahead of them.
  float kst[NU][8];
  // K rows through a buffer resource over the stage's valid rows (none for a padded stage):
  // keys past T read as zero, as they must, since they meet finite dS columns.
  auto gload = [&](int stage) {
    const int j0 = stage * BN;
    const int rows = min(BN, T - j0);
    const __amdgpu_buffer_rsrc_t rk = rows_rsrc(Kb + (int64_t)j0 * sk.t, rows, sk.t, HS);
    const int st = (int)sk.t * 4;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int f = tid + THREADS * u;
      const int d = f % HS, sh = f / HS;  // sh: over the stage's 16-key steps and halves
      const int at = (16 * (sh >> 1) + 4 * (sh & 1)) * st + 4 * d;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        kst[u][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
            rk, at, (8 * (j >> 2) + (j & 3)) * st, 0));
    }
  };
  auto lstore = [&](int buf) {
    char* ks = smem + buf * STAGE;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int f = tid + THREADS * u;
      const int d = f % HS, sh = f / HS;
      bf16x8 p[3];
      split_bf16<true>(kst[u], p);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        *reinterpret_cast<bf16x8*>(
            ks + q * PART +
            (((sh >> 2) * (HS / 32) + (d >> 5)) * 128 + (sh & 3) * 32 + (d & 31)) * 16) = p[q];
    }
  };
  // A stored tile exists for query block ib and key block jb iff both lie inside the head and,
  // with a causal mask, jb <= ib (the wave-uniform skip of the dK/dV stage).
  auto has_tile = [&](int jb) { return ib < nb && jb < nb && (!CAUSAL || jb <= ib); };
  // Tiles that do not exist are read from the row's last stored tile (clamped block indices,
  // equal to (ib, jb) whenever has_tile(jb)); compute() skips them.
  const int ibc = min(ib, nb - 1);
  auto dsload = [&](int stage, float4 (&dr)[NSUB][4]) {
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub) {
      const int jbc = min(stage * NSUB + sub, CAUSAL ? ibc : nb - 1);
      const float* src = dsh + ds_tile_index(ibc, jbc, nb, CAUSAL) * kDsTileFloats + 4 * lane;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        dr[sub][g] = ld4_stream(src + 256 * g);
      }
    }
  };
  constexpr int kFlip = kFlipRows / BN;  // even
  float y = kSplitScale;  // the scale, and now and then the sign, of dS in the sums
  auto compute = [&](int stage, const char* ks, const float4 (&dr)[NSUB][4]) {
    if (stage >= s_end) return;  // a padded stage (or, split, the other part's)
#pragma unroll
    for (int sub = 0; sub < NSUB; ++sub) {
      if (!has_tile(stage * NSUB + sub)) continue;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const float4 lo = dr[sub][2 * st], hi = dr[sub][2 * st + 1];
        const float x[8] = {y * lo.x, y * lo.y, y * lo.z, y * lo.w,
                            y * hi.x, y * hi.y, y * hi.z, y * hi.w};
        bf16x8 dp[3];
        split_bf16(x, dp);
#pragma unroll
        for (int d0 = 0; d0 < HS / 32; d0 += 2) {
          constexpr int ND = HS / 32 < 2 ? 1 : 2;  // two chains
          bf16x8 a[ND][3];
#pragma unroll
          for (int d = 0; d < ND; ++d)
#pragma unroll
            for (int q = 2; q >= 0; --q)
              a[d][q] = *reinterpret_cast<const bf16x8*>(
                  ks + q * PART +
                  ((sub * (HS / 32) + d0 + d) * 128 + (2 * st + half) * 32 + col) * 16);
#pragma unroll
          for (int p = 0; p < 6; ++p)
#pragma unroll
            for (int d = 0; d < ND; ++d)
              acc[d0 + d] = mfma_bf16(a[d][kSplitA[p]], dp[kSplitB[p]], acc[d0 + d]);
        }
      }
    }
  };
  auto step = [&](int s, const float4 (&cur)[NSUB][4], float4 (&nxt)[NSUB][4]) {
    const int buf = (s - s_begin) & 1;
    gload(s + 1);
    dsload(s + 1, nxt);
    compute(s, smem + buf * STAGE, cur);
    lstore(buf ^ 1);
    __syncthreads();
  };

  if (s_end > s_begin) {
    float4 dA[NSUB][4], dB[NSUB][4];
    dsload(s_begin, dA);
    gload(s_begin);
    lstore(0);
    __syncthreads();
    // Unrolled by two so the two dS register sets swap roles without copies.
    const int s_end2 = s_begin + ((s_end - s_begin + 1) & ~1);
    for (int run = s_begin; run < s_end2; run += kFlip) {
      if (run > s_begin) {
        y = -y;
#pragma unroll
        for (int d = 0; d < HS / 32; ++d) acc[d] = -acc[d];
      }
      for (int s = run; s < min(run + kFlip, s_end2); s += 2) {
        step(s, dA, dB);
        step(s + 1, dB, dA);
      }
    }
  }

  bool odd = false;
  y *= kSplitUnscale * kSplitUnscale * kSplitUnscale;
#pragma unroll
  for (int d = 0; d < HS / 32; ++d) {
    odd |= not_finite(acc[d]);
    acc[d] *= y;
  }
  if (__syncthreads_or(odd)) {
    float* const ks = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) acc[d] = zero16();
    for (int s = s_begin; s < s_end; ++s) {
      __syncthreads();
      for (int f = tid; f < BN * HS / 4; f += THREADS) {
        const int r = f / (HS / 4), c4 = f % (HS / 4) * 4;
        const int64_t j = (int64_t)s * BN + r;
        st4(ks + r * KP + c4, j < T ? ld4(Kb + j * sk.t + c4) : zero4());
      }
      __syncthreads();
      float4 dr[NSUB][4];
      dsload(s, dr);
#pragma unroll
      for (int sub = 0; sub < NSUB; ++sub) {
        if (!has_tile(s * NSUB + sub)) continue;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk)
#pragma unroll
          for (int d = 0; d < HS / 32; ++d)
            acc[d] = mfma32(ks[(sub * 32 + mfma_row(kk, half)) * KP + d * 32 + col],
                            f4_at(dr[sub][kk >> 2], kk & 3), acc[d]);
      }
    }
    __syncthreads();
  }

  if (my_i < T) {
    float* op = dQ + b * sdq.b + h * sdq.h + (int64_t)my_i * sdq.t;
    if (SPLIT && part) op = part_ws + ((int64_t)bh * T + my_i) * HS;
#pragma unroll
    for (int d = 0; d < HS / 32; ++d) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int dc = d * 32 + 8 * g + 4 * half;
        st4(op + dc, make_float4(acc[d][4 * g + 0] * scale, acc[d][4 * g + 1] * scale,
                                 acc[d][4 * g + 2] * scale, acc[d][4 * g + 3] * scale));
      }
    }
  }
  }  // pass: the check above is a barrier, so the next pass may refill LDS
}

RowStrides rs(const int64_t* s) { return RowStrides{s[0], s[1], s[2]}; }

template <int HS>
void launch_delta(const float* o, const float* d_o, float* delta, int nh, int T, int64_t rows,
                  RowStrides so, RowStrides sdo, hipStream_t st) {
  const int64_t threads = rows * (HS / 4);
  const unsigned grid = (unsigned)((threads + 255) / 256);
  hipLaunchKernelGGL((fa2_bwd_delta_kernel<HS>), dim3(grid), dim3(256), 0, st, o, d_o, delta, nh,
                     T, rows, so, sdo);
}

// With o != nullptr the kernel forms delta from O (strides so) and writes it into `delta`.
template <int HS, bool CAUSAL>
void launch_dq(const float* q, const float* k, const float* v, const float* d_o, const float* l,
               float* delta, float* dq, int nh, int T, int BH, RowStrides sq,
               RowStrides sk, RowStrides sv, RowStrides sdo, LStrides sl, RowStrides sdq,
               float scale, hipStream_t st, const float* o = nullptr, RowStrides so = {}) {
  const int n_qtiles = (T + 127) / 128;
  const int64_t items = (int64_t)(CAUSAL ? (n_qtiles + 1) / 2 : n_qtiles) * BH;
  const int lpt = CAUSAL ? lpt_heads(BH, n_qtiles, 4, BwdTile<HS>::MINW) : 0;
  const dim3 grid(lpt > 0 ? (unsigned)(BH * n_qtiles) : xcd_grid(items));
  if (o != nullptr) {
    hipLaunchKernelGGL((fa2_bwd_dq_kernel<HS, CAUSAL, true>), grid, dim3(256), 0, st, q, k, v,
                       d_o, l, delta, dq, nh, T, BH, n_qtiles, sq, sk, sv, sdo, sl, sdq, scale,
                       scale * kLog2e, o, so, lpt);
    return;
  }
  hipLaunchKernelGGL((fa2_bwd_dq_kernel<HS, CAUSAL>), grid, dim3(256), 0, st, q, k, v, d_o, l,
                     delta, dq, nh, T, BH, n_qtiles, sq, sk, sv, sdo, sl, sdq, scale,
                     scale * kLog2e, nullptr, RowStrides{}, lpt);
}

// dK/dV for heads [bh_base, bh_base + n_heads), written through strides sdk / sdv; with
// STORE_DS the dS tiles go to dsw; with FOLD delta comes from O (strides so) instead of the
// delta array.  Four waves (128 keys) per workgroup.
// part_ws (heads [0, n_heads) with bh_base = 0 only): run the split form and its sum pass.
template <int HS, bool CAUSAL, bool STORE_DS, bool FOLD = false>
void launch_dkdv(const float* q, const float* k, const float* v, const float* d_o,
                 const float* l, const float* delta, float* dk, float* dv, float* dsw, int nh,
                 int T, int bh_base, int n_heads, RowStrides sq, RowStrides sk, RowStrides sv,
                 RowStrides sdo, LStrides sl, RowStrides sdk, RowStrides sdv, float scale,
                 hipStream_t st, const float* o = nullptr, RowStrides so = {},
                 float* part_ws = nullptr) {
  constexpr int WAVES = 4;
  const int n_ktiles = (T + 32 * WAVES - 1) / (32 * WAVES);
  const int64_t items = (int64_t)(CAUSAL ? (n_ktiles + 1) / 2 : n_ktiles) * n_heads;
  if (part_ws != nullptr) {
    hipLaunchKernelGGL((fa2_bwd_dkdv_kernel<HS, CAUSAL, STORE_DS, FOLD, true>),
                       dim3(xcd_grid(2 * items)), dim3(64 * WAVES), 0, st, q, k, v, d_o, o, l,
                       delta, dk, dv, dsw, nh, T, bh_base, n_heads, n_ktiles, sq, sk, sv, sdo,
                       so, sl, sdk, sdv, scale, scale * kLog2e, part_ws);
    const int64_t rows = (int64_t)n_heads * T;
    hipLaunchKernelGGL((fa2_bwd_dkdv_sum_kernel<HS>),
                       dim3((unsigned)((rows * (HS / 4) + 255) / 256)), dim3(256), 0, st, dk,
                       dv, part_ws, nh, T, rows, sdk, sdv);
    return;
  }
  const int lpt = CAUSAL ? lpt_heads(n_heads, n_ktiles, WAVES, kDkdvMinWaves<HS>) : 0;
  hipLaunchKernelGGL((fa2_bwd_dkdv_kernel<HS, CAUSAL, STORE_DS, FOLD>),
                     dim3(lpt > 0 ? (unsigned)(n_heads * n_ktiles) : xcd_grid(items)),
                     dim3(64 * WAVES), 0, st, q, k, v, d_o, o, l, delta, dk, dv, dsw, nh, T,
                     bh_base, n_heads, n_ktiles, sq, sk, sv, sdo, so, sl, sdk, sdv, scale,
                     scale * kLog2e, nullptr, lpt);
}

// part_ws (heads [0, n_heads) with bh_base = 0 only): run the split form and its sum pass.
template <int HS, bool CAUSAL>
void launch_dq_ds(const float* k, const float* dsw, float* dq, int nh, int T, int bh_base,
                  int n_heads, RowStrides sk, RowStrides sdq, float scale, hipStream_t st,
                  float* part_ws = nullptr) {
  auto run = [&]<int WAVES>() {
    const int n_qtiles = (T + 32 * WAVES - 1) / (32 * WAVES);
    const int64_t items = (int64_t)(CAUSAL ? (n_qtiles + 1) / 2 : n_qtiles) * n_heads;
    if (part_ws != nullptr) {
      hipLaunchKernelGGL((fa2_bwd_dq_ds_kernel<HS, CAUSAL, WAVES, true>),
                         dim3(xcd_grid(2 * items)), dim3(64 * WAVES), 0, st, k, dsw, dq, nh, T,
                         bh_base, n_heads, n_qtiles, sk, sdq, scale, part_ws);
      const int64_t rows = (int64_t)n_heads * T;
      hipLaunchKernelGGL((fa2_bwd_dq_sum_kernel<HS>),
                         dim3((unsigned)((rows * (HS / 4) + 255) / 256)), dim3(256), 0, st, dq,
                         part_ws, nh, T, rows, sdq);
      return;
    }
    const int lpt = CAUSAL ? lpt_heads(n_heads, n_qtiles, WAVES, 2) : 0;
    hipLaunchKernelGGL((fa2_bwd_dq_ds_kernel<HS, CAUSAL, WAVES>),
                       dim3(lpt > 0 ? (unsigned)(n_heads * n_qtiles) : xcd_grid(items)),
                       dim3(64 * WAVES), 0, st, k, dsw, dq, nh, T, bh_base, n_heads, n_qtiles, sk,
                       sdq, scale, nullptr, lpt);
  };
  // Short causal heads (hs 64, T <= 512): two waves (64 query rows) per workgroup.  Two waves
  // against four: T64 64 heads 5.9 and 6.6 us; T256 B64 H6 27.7 and 32.3, 64 heads 12.5 and 12.1;
  // T512 B64 H6 69.4 and 69.1, 128 heads 29.7 and 30.9, 64 heads 22.3 and 20.6.  Beyond: T768 128
  // heads 55.6 and 56.6, 16 heads 29.6 and 27.0; T1024 256 heads 168 and 150.
  if constexpr (HS == 64 && CAUSAL) {
    if (T <= 512) {
      run.template operator()<2>();
      return;
    }
  }
  run.template operator()<4>();
}

// The stored-dS dK/dV stage splits each item's query stages over two workgroups when its grid
// would hold fewer than two waves per SIMD (1024 SIMDs) and a full column of queries gives each
// part at least kSplitMinStages stages (T >= 1024; 2048 at hs 32, whose stages are half the work),
// as the forward does.
constexpr int kSimds = 1024;
constexpr int kSplitMinStages = 16;

template <int HS, bool CAUSAL>
bool dkdv_split(int T, int BH) {
  const int n_ktiles = (T + 127) / 128;
  const int64_t items = (int64_t)(CAUSAL ? (n_ktiles + 1) / 2 : n_ktiles) * BH;
  return items * 4 < 2 * kSimds && T / (HS == 32 ? 64 : 32) >= 2 * kSplitMinStages;
}

// Runs f.template operator()<HS, CAUSAL>() for the runtime head size and mask flag.
template <typename F>
void dispatch_hs_causal(int64_t hs, int causal, F&& f) {
  if (hs == 32) { if (causal) f.template operator()<32, true>(); else f.template operator()<32, false>(); }
  else if (hs == 64) { if (causal) f.template operator()<64, true>(); else f.template operator()<64, false>(); }
  else { if (causal) f.template operator()<128, true>(); else f.template operator()<128, false>(); }
}

bool l_ok(const float* l, const int64_t* s) { return l != nullptr && s != nullptr; }

}  // namespace
}  // namespace cta

using namespace cta;

extern "C" int cta_flash_attention_bwd_delta(const float* o, const int64_t* o_strides,
                                             const float* d_o, const int64_t* do_strides,
                                             int64_t B, int64_t nh, int64_t T, int64_t hs,
                                             float* delta, void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (!delta) return fail(CTA_ERR_INVALID_ARGUMENT, "null delta pointer");
  if (!attn_layout_ok(o, o_strides) || !attn_layout_ok(d_o, do_strides))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned O/dO");
  const int64_t rows = B * nh * T;
  hipStream_t st = as_stream(stream);
  if (hs == 32) launch_delta<32>(o, d_o, delta, (int)nh, (int)T, rows, rs(o_strides), rs(do_strides), st);
  else if (hs == 64) launch_delta<64>(o, d_o, delta, (int)nh, (int)T, rows, rs(o_strides), rs(do_strides), st);
  else launch_delta<128>(o, d_o, delta, (int)nh, (int)T, rows, rs(o_strides), rs(do_strides), st);
  return check_launch("flash_attention_bwd_delta");
}

namespace {
int check_bwd_inputs(const float* q, const int64_t* qs, const float* k, const int64_t* ks,
                     const float* v, const int64_t* vs, const float* d_o, const int64_t* dos,
                     const float* l, const int64_t* ls, const float* delta) {
  if (!attn_layout_ok(q, qs) || !attn_layout_ok(k, ks) || !attn_layout_ok(v, vs) ||
      !attn_layout_ok(d_o, dos))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned Q/K/V/dO");
  if (!l_ok(l, ls) || !delta) return fail(CTA_ERR_INVALID_ARGUMENT, "null L or delta pointer");
  return CTA_OK;
}
}  // namespace

namespace {
// Strides of a dense (B, nh, T, hs) output.
RowStrides dense_out(int64_t nh, int64_t T, int64_t hs) { return {nh * T * hs, T * hs, hs}; }

// With o != nullptr, dQ forms delta itself (from O, strides so) and writes it into `delta`.
int bwd_dq_impl(const float* q, const int64_t* q_strides, const float* k,
                const int64_t* k_strides, const float* v, const int64_t* v_strides,
                const float* d_o, const int64_t* do_strides, const float* l,
                const int64_t* l_strides, float* delta, int64_t B, int64_t nh, int64_t T,
                int64_t hs, int causal, float* dq, RowStrides sdq, hipStream_t st,
                const float* o = nullptr, RowStrides so = {}) {
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  const LStrides sl{l_strides[0], l_strides[1], l_strides[2]};
  const int BH = (int)(B * nh);
  dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
    launch_dq<HS, C>(q, k, v, d_o, l, delta, dq, (int)nh, (int)T, BH, rs(q_strides),
                     rs(k_strides), rs(v_strides), rs(do_strides), sl, sdq, scale, st, o, so);
  });
  return check_launch("flash_attention_bwd_dq");
}

int bwd_dkdv_impl(const float* q, const int64_t* q_strides, const float* k,
                  const int64_t* k_strides, const float* v, const int64_t* v_strides,
                  const float* d_o, const int64_t* do_strides, const float* l,
                  const int64_t* l_strides, const float* delta, int64_t B, int64_t nh, int64_t T,
                  int64_t hs, int causal, float* dk, RowStrides sdk, float* dv, RowStrides sdv,
                  hipStream_t st) {
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  const LStrides sl{l_strides[0], l_strides[1], l_strides[2]};
  const int BH = (int)(B * nh);
  dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
    launch_dkdv<HS, C, false>(q, k, v, d_o, l, delta, dk, dv, nullptr, (int)nh, (int)T, 0, BH,
                              rs(q_strides), rs(k_strides), rs(v_strides), rs(do_strides), sl,
                              sdk, sdv, scale, st);
  });
  return check_launch("flash_attention_bwd_dkdv");
}
}  // namespace

extern "C" int cta_flash_attention_bwd_dq(const float* q, const int64_t* q_strides,
                                          const float* k, const int64_t* k_strides,
                                          const float* v, const int64_t* v_strides,
                                          const float* d_o, const int64_t* do_strides,
                                          const float* l, const int64_t* l_strides,
                                          const float* delta, int64_t B, int64_t nh, int64_t T,
                                          int64_t hs, int causal, float* dq, void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (int rc = check_bwd_inputs(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                                l_strides, delta))
    return rc;
  if (!dq || !aligned16(dq)) return fail(CTA_ERR_LAYOUT, "dQ must be a 16-byte aligned pointer");
  // (read only: without O the kernel reads delta)
  return bwd_dq_impl(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l, l_strides,
                     const_cast<float*>(delta), B, nh, T, hs, causal, dq, dense_out(nh, T, hs),
                     as_stream(stream));
}

extern "C" int cta_flash_attention_bwd_dq_delta(
    const float* q, const int64_t* q_strides, const float* k, const int64_t* k_strides,
    const float* v, const int64_t* v_strides, const float* o, const int64_t* o_strides,
    const float* d_o, const int64_t* do_strides, const float* l, const int64_t* l_strides,
    int64_t B, int64_t nh, int64_t T, int64_t hs, int causal, float* delta, float* dq,
    void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (!attn_layout_ok(o, o_strides))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned O/dO");
  if (int rc = check_bwd_inputs(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                                l_strides, delta))
    return rc;
  if (!dq || !aligned16(dq)) return fail(CTA_ERR_LAYOUT, "dQ must be a 16-byte aligned pointer");
  return bwd_dq_impl(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l, l_strides,
                     delta, B, nh, T, hs, causal, dq, dense_out(nh, T, hs), as_stream(stream), o,
                     rs(o_strides));
}

extern "C" int cta_flash_attention_bwd_dkdv(const float* q, const int64_t* q_strides,
                                            const float* k, const int64_t* k_strides,
                                            const float* v, const int64_t* v_strides,
                                            const float* d_o, const int64_t* do_strides,
                                            const float* l, const int64_t* l_strides,
                                            const float* delta, int64_t B, int64_t nh, int64_t T,
                                            int64_t hs, int causal, float* dk, float* dv,
                                            void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (int rc = check_bwd_inputs(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                                l_strides, delta))
    return rc;
  if (!dk || !dv || !aligned16(dk) || !aligned16(dv))
    return fail(CTA_ERR_LAYOUT, "dK/dV must be 16-byte aligned pointers");
  const RowStrides dense = dense_out(nh, T, hs);
  return bwd_dkdv_impl(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l, l_strides,
                       delta, B, nh, T, hs, causal, dk, dense, dv, dense, as_stream(stream));
}

extern "C" int64_t cta_flash_attention_bwd_workspace(int64_t B, int64_t nh, int64_t T,
                                                     int64_t hs, int causal) {
  if (B <= 0 || nh <= 0 || T <= 0 || (hs != 32 && hs != 64 && hs != 128)) return 0;
  return B * nh * ds_tiles_per_head(T, causal != 0) * kDsTileFloats * (int64_t)sizeof(float);
}

extern "C" int64_t cta_flash_attention_bwd_split_workspace(int64_t B, int64_t nh, int64_t T,
                                                           int64_t hs, int causal) {
  if (B <= 0 || nh <= 0 || T <= 0 || (hs != 32 && hs != 64 && hs != 128) ||
      B * nh > ((int64_t)1 << 24) || T > ((int64_t)1 << 24))
    return 0;
  bool split = false;
  dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() { split = dkdv_split<HS, C>((int)T, (int)(B * nh)); });
  return split ? 2 * B * nh * T * hs * (int64_t)sizeof(float) : 0;
}

extern "C" int cta_flash_attention_bwd_dkdv_store_ds(
    const float* q, const int64_t* q_strides, const float* k, const int64_t* k_strides,
    const float* v, const int64_t* v_strides, const float* d_o, const int64_t* do_strides,
    const float* l, const int64_t* l_strides, const float* delta, int64_t B, int64_t nh,
    int64_t T, int64_t hs, int causal, float* dk, float* dv, float* ds_workspace,
    void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (int rc = check_bwd_inputs(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                                l_strides, delta))
    return rc;
  if (!dk || !dv || !aligned16(dk) || !aligned16(dv) || !ds_workspace || !aligned16(ds_workspace))
    return fail(CTA_ERR_LAYOUT, "dK/dV and the dS workspace must be 16-byte aligned pointers");
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  const LStrides sl{l_strides[0], l_strides[1], l_strides[2]};
  hipStream_t st = as_stream(stream);
  dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
    launch_dkdv<HS, C, true>(q, k, v, d_o, l, delta, dk, dv, ds_workspace, (int)nh, (int)T, 0,
                             (int)(B * nh), rs(q_strides), rs(k_strides), rs(v_strides),
                             rs(do_strides), sl, dense_out(nh, T, hs), dense_out(nh, T, hs),
                             scale, st);
  });
  return check_launch("flash_attention_bwd_dkdv_store_ds");
}

extern "C" int cta_flash_attention_bwd_dq_from_ds(const float* k, const int64_t* k_strides,
                                                  const float* ds_workspace, int64_t B,
                                                  int64_t nh, int64_t T, int64_t hs, int causal,
                                                  float* dq, void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (!attn_layout_ok(k, k_strides))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned K");
  if (!dq || !aligned16(dq) || !ds_workspace || !aligned16(ds_workspace))
    return fail(CTA_ERR_LAYOUT, "dQ and the dS workspace must be 16-byte aligned pointers");
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  hipStream_t st = as_stream(stream);
  dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
    launch_dq_ds<HS, C>(k, ds_workspace, dq, (int)nh, (int)T, 0, (int)(B * nh), rs(k_strides),
                        dense_out(nh, T, hs), scale, st);
  });
  return check_launch("flash_attention_bwd_dq_from_ds");
}

extern "C" int cta_flash_attention_bwd_strided(
    const float* q, const int64_t* q_strides, const float* k, const int64_t* k_strides,
    const float* v, const int64_t* v_strides, const float* o, const int64_t* o_strides,
    const float* d_o, const int64_t* do_strides, const float* l, const int64_t* l_strides,
    int64_t B, int64_t nh, int64_t T, int64_t hs, int causal, float* dq,
    const int64_t* dq_strides, float* dk, const int64_t* dk_strides, float* dv,
    const int64_t* dv_strides, float* delta, float* workspace, int64_t workspace_bytes,
    void* stream) {
  const int64_t head_bytes = cta_flash_attention_bwd_workspace(1, 1, T, hs, causal);
  const bool stored = workspace != nullptr && head_bytes != 0 && workspace_bytes >= head_bytes;
  if (stored) {
    if (int rc = cta_flash_attention_bwd_delta(o, o_strides, d_o, do_strides, B, nh, T, hs,
                                               delta, stream))
      return rc;
  } else {
    // the recompute schedule's dQ stage forms delta itself: the delta pass's checks only
    if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
    if (B * nh * T > 0 && (!attn_layout_ok(o, o_strides) || !attn_layout_ok(d_o, do_strides)))
      return fail(CTA_ERR_LAYOUT,
                  "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                  "aligned O/dO");
  }
  if (B * nh * T == 0) return CTA_OK;
  if (int rc = check_bwd_inputs(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                                l_strides, delta))
    return rc;
  if (!attn_layout_ok(dq, dq_strides) || !attn_layout_ok(dk, dk_strides) ||
      !attn_layout_ok(dv, dv_strides))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned dQ/dK/dV");
  const RowStrides sdq = rs(dq_strides), sdk = rs(dk_strides), sdv = rs(dv_strides);
  hipStream_t st = as_stream(stream);
  if (!stored) {
    // The reference's schedule: dQ recomputes S and dP, and forms delta for dK/dV on the way
    // (no delta launch).
    if (int rc = bwd_dq_impl(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                             l_strides, delta, B, nh, T, hs, causal, dq, sdq, st, o,
                             rs(o_strides)))
      return rc;
    return bwd_dkdv_impl(q, q_strides, k, k_strides, v, v_strides, d_o, do_strides, l,
                         l_strides, delta, B, nh, T, hs, causal, dk, sdk, dv, sdv, st);
  }
  if (!aligned16(workspace))
    return fail(CTA_ERR_LAYOUT, "the workspace must be a 16-byte aligned pointer");
  // Stored-dS schedule over chunks of equal head counts that fit the workspace.
  const int BH = (int)(B * nh);
  const int64_t fit = std::min<int64_t>(BH, workspace_bytes / head_bytes);
  const int64_t n_chunks = (BH + fit - 1) / fit;
  const int chunk = (int)((BH + n_chunks - 1) / n_chunks);
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  const LStrides sl{l_strides[0], l_strides[1], l_strides[2]};
  // A small grid's dK/dV and dQ-from-dS stages split over twice the workgroups when the
  // workspace also holds the split's partial sums after every head's dS tiles (dK, dV; then,
  // once the dK/dV sum pass has read them, dQ in the same place).
  const int64_t ds_all = cta_flash_attention_bwd_workspace(B, nh, T, hs, causal);
  const int64_t split = cta_flash_attention_bwd_split_workspace(B, nh, T, hs, causal);
  float* part_ws = split > 0 && n_chunks == 1 && workspace_bytes >= ds_all + split
                       ? workspace + ds_all / (int64_t)sizeof(float)
                       : nullptr;
  for (int h0 = 0; h0 < BH; h0 += chunk) {
    const int n = std::min(chunk, BH - h0);
    dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
      launch_dkdv<HS, C, true>(q, k, v, d_o, l, delta, dk, dv, workspace, (int)nh, (int)T, h0, n,
                               rs(q_strides), rs(k_strides), rs(v_strides), rs(do_strides), sl,
                               sdk, sdv, scale, st, nullptr, {}, part_ws);
      launch_dq_ds<HS, C>(k, workspace, dq, (int)nh, (int)T, h0, n, rs(k_strides), sdq, scale,
                          st, part_ws);
    });
    if (int rc = check_launch("flash_attention_bwd")) return rc;
  }
  return CTA_OK;
}

extern "C" int cta_flash_attention_bwd(const float* q, const int64_t* q_strides, const float* k,
                                       const int64_t* k_strides, const float* v,
                                       const int64_t* v_strides, const float* o,
                                       const int64_t* o_strides, const float* d_o,
                                       const int64_t* do_strides, const float* l,
                                       const int64_t* l_strides, int64_t B, int64_t nh,
                                       int64_t T, int64_t hs, int causal, float* dq, float* dk,
                                       float* dv, float* delta, float* workspace,
                                       int64_t workspace_bytes, void* stream) {
  const int64_t ds[4] = {nh * T * hs, T * hs, hs, 1};  // dense (B, nh, T, hs) outputs
  return cta_flash_attention_bwd_strided(q, q_strides, k, k_strides, v, v_strides, o, o_strides,
                                         d_o, do_strides, l, l_strides, B, nh, T, hs, causal, dq,
                                         ds, dk, ds, dv, ds, delta, workspace, workspace_bytes,
                                         stream);
}

extern "C" int cta_flash_attention_bwd_fold_delta(
    const float* q, const int64_t* q_strides, const float* k, const int64_t* k_strides,
    const float* v, const int64_t* v_strides, const float* o, const int64_t* o_strides,
    const float* d_o, const int64_t* do_strides, const float* l, const int64_t* l_strides,
    int64_t B, int64_t nh, int64_t T, int64_t hs, int causal, float* dq, float* dk, float* dv,
    float* workspace, int64_t workspace_bytes, void* stream) {
  if (int rc = check_attn_sizes(B, nh, T, hs)) return rc;
  if (B * nh * T == 0) return CTA_OK;
  if (!attn_layout_ok(q, q_strides) || !attn_layout_ok(k, k_strides) ||
      !attn_layout_ok(v, v_strides) || !attn_layout_ok(o, o_strides) ||
      !attn_layout_ok(d_o, do_strides))
    return fail(CTA_ERR_LAYOUT,
                "flash_attention_bwd needs unit d-stride, strides divisible by 4, time strides below 2^23 and 16-byte "
                "aligned Q/K/V/O/dO");
  if (!l_ok(l, l_strides)) return fail(CTA_ERR_INVALID_ARGUMENT, "null L pointer");
  const int64_t head_bytes = cta_flash_attention_bwd_workspace(1, 1, T, hs, causal);
  if (workspace == nullptr || workspace_bytes < head_bytes)
    return fail(CTA_ERR_INVALID_ARGUMENT,
                "flash_attention_bwd_fold_delta needs a dS workspace of at least one head (" +
                    std::to_string(head_bytes) + " bytes)");
  if (!dq || !dk || !dv || !aligned16(dq) || !aligned16(dk) || !aligned16(dv) ||
      !aligned16(workspace))
    return fail(CTA_ERR_LAYOUT, "dQ/dK/dV and the workspace must be 16-byte aligned pointers");
  const int BH = (int)(B * nh);
  const int64_t fit = std::min<int64_t>(BH, workspace_bytes / head_bytes);
  const int64_t n_chunks = (BH + fit - 1) / fit;
  const int chunk = (int)((BH + n_chunks - 1) / n_chunks);
  const float scale = 1.0f / std::sqrt(static_cast<float>(hs));
  const LStrides sl{l_strides[0], l_strides[1], l_strides[2]};
  hipStream_t st = as_stream(stream);
  for (int h0 = 0; h0 < BH; h0 += chunk) {
    const int n = std::min(chunk, BH - h0);
    dispatch_hs_causal(hs, causal, [&]<int HS, bool C>() {
      launch_dkdv<HS, C, true, true>(q, k, v, d_o, l, nullptr, dk, dv, workspace, (int)nh,
                                     (int)T, h0, n, rs(q_strides), rs(k_strides), rs(v_strides),
                                     rs(do_strides), sl, dense_out(nh, T, hs),
                                     dense_out(nh, T, hs), scale, st, o, rs(o_strides));
      launch_dq_ds<HS, C>(k, workspace, dq, (int)nh, (int)T, h0, n, rs(k_strides),
                          dense_out(nh, T, hs), scale, st);
    });
    if (int rc = check_launch("flash_attention_bwd_fold_delta")) return rc;
  }
  return CTA_OK;
}
