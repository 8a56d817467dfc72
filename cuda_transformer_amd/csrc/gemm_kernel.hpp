// Strided, batched FP32 GEMM on CDNA4 MFMA, and the linear layer's C entry points.
//
//   out[z][m][n] = alpha * sum_k A[z][m][k] * B[z][k][n]  (+ bias[n])  (causal: -inf for n > m)
//
// optionally followed by a GELU stage (erf or tanh form) in the epilogue (the GPT MLP's
// fc1 -> GELU forward and fc2 -> GELU backward products, each one pass over the output instead
// of two).
//
// This one kernel backs the reference's fused_multiply_add (Transformer_kernels/
// fused_multiply_add.cuh:10-92, launched from Transformer_launchers/linear_layer.cu:28-70),
// its strided batched cuda_bmm (batched_matrix_multiply.cuh:9-75) and the two GEMM stages of
// the naive attention (causal_self_attention_fwd.cuh:9-127).  Every operand is addressed
// through strides, so transposed views (W^T, x^T in the linear backward) need no copies.
// The batch index z is split as (z / zin, z % zin) with a stride per level, which lets
// the naive attention address heads inside a packed (B, T, 3C) tensor directly.
//
// FP32 products on the BF16 matrix pipe.  A float is the exact sum of three bfloat16 numbers
// (8 + 8 + 8 significant bits: x0 = bf16(x), x1 = bf16(x - x0), x2 = x - x0 - x1), so
//   a b = a0 b0 + (a0 b1 + a1 b0) + (a0 b2 + a1 b1 + a2 b0) + O(2^-26 |a b|)
// and six v_mfma_f32_32x32x16_bf16 (32 cycles, 16 k) take the place of eight
// v_mfma_f32_32x32x2_f32 (64 cycles, 2 k each): 192 instead of 512 matrix cycles.  The products
// of 8-bit significands are exact and accumulate in FP32, a0 b0 apart from the other five; with
// one rounding of the large accumulator per 16 k instead of sixteen the result is closer to the
// exact product than the FP32 MFMA's (relative error at K = 768, N(0,1) operands: 1.6e-7 against
// 5.0e-7; K = 8192: 5.7e-7 against 1.6e-6).
// Sustained on all CUs, from registers, the six products reach 305-312 TFLOP/s of FP32 work (the
// chip's power limit), the FP32 MFMA 154.
// Operands are scaled by 2^24 before the split (split_bf16.hpp), so that the parts hold every float
// below 2^103 exactly, subnormals included, and products keep their bits down to where FP32's own
// end.  Sums above 2^79 overflow, infinities and larger operands give NaN: a workgroup whose tile
// comes out with a value that is not finite discards it and runs the tile again with FP32 MFMAs
// (exact_tile), so such operands give what FP32 arithmetic gives, in up to 2.7 times the time
// (8192 x 3072 x 768 with an infinity in every tile: 195-201 -> 528 us).
//
// gfx950 design: workgroup tile 128x128 of four 64x64 waves, 64x128 of four 32x64 or 64x64 of
// four 32x32, two or three workgroups (waves per SIMD) on a CU.  A lane loads eight k of one row
// (two dwordx4 where k is contiguous in memory, eight dwords otherwise), scales and splits them
// (13 VALU instructions per pair, beside the MFMAs) and stores one 16-byte unit per
// part: LDS holds [part][k half][row][8 k], which is the MFMA operand order, so operand reads
// and stores are contiguous 16-byte accesses with no bank conflict and no padding to speak of.
// Loads and the epilogue's stores go through buffer resources: scalar bases with fixed per-lane
// offsets, and the buffer's range check zeroes (loads) or drops (stores) what lies outside the
// operand, so the K loop and the epilogue carry no per-element address arithmetic or bounds
// tests.  What bounds it: 8192 x 3072 x 768 runs at 192-199 TFLOP/s (FP32 MFMA: 142), the matrix
// pipe 60% busy at 1.77 GHz, at the chip's power limit (on all-zero operands the same kernel takes
// 142 us instead of 195-201), so bytes moved per product and the splits' instructions cost time too.
//
// This header holds the kernel templates and the per-tile launcher; gemm_tiles_*.hip each
// instantiate a few tile types (gemm_launch_<tile>), so the build compiles them in parallel, and
// gemm.hip picks the tile and holds the C entry points.
#pragma once

#include "cta_common.hpp"
#include "gemm.hpp"
#include "split_bf16.hpp"

namespace cta {

// How an operand's slices are loaded: k contiguous with rows a multiple of 16 bytes apart
// (kVecK), k contiguous with any row stride or length (kAnyK), rows contiguous (kVecMN: m of A,
// n of B; any alignment), any strides whose slices 32-bit offsets reach (kStrided), or any strides
// at all (kScalar, only ever for both operands).
enum LoadMode { kVecK = 0, kVecMN = 1, kScalar = 2, kAnyK = 3, kStrided = 4 };

namespace {

constexpr int kGemmK = 16;  // K-slice: one k step of the 32x32x16 MFMA

// Workgroup tile BM x BN, WM x WN waves; each wave owns a (BM/WM) x (BN/WN) block of 32x32 MFMA
// tiles.
template <int BM_, int BN_, int WM_, int WN_>
struct GemmTile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_;
  static constexpr int THREADS = 64 * WM * WN;
  static constexpr int MB = BM / WM / 32;  // MFMA tiles per wave along m
  static constexpr int NB = BN / WN / 32;  // ... along n
  // LDS bytes of one part of an operand's slice: two k halves of 16 bytes per row, the second
  // 64 bytes further so that lanes writing both halves of a row use different banks.
  static constexpr int plane(int rows) { return 2 * (rows * 16 + 64); }
  static constexpr int A_BYTES = 3 * plane(BM), B_BYTES = 3 * plane(BN);
  static constexpr int BUF_BYTES = A_BYTES + B_BYTES;  // double buffered
  static_assert(MB >= 1 && NB >= 1, "bad GEMM tile");
  static_assert(kGemmK * (BM + BN) * 4 <= 2 * BUF_BYTES, "exact_tile's slices fit");
};

// One operand's K-slice in registers: unit u of the slice is eight k (half h: k = 8h .. 8h + 7)
// of one row; a thread holds units tid, tid + THREADS, ...  `rows` indexes m (A) or n (B); the
// operand is row-major in (row, k) when kVecK or kAnyK, (k, row) when kVecMN.
template <int ROWS, int THREADS>
struct Slice {
  static constexpr int UNITS = 2 * ROWS;
  static constexpr int N = (UNITS + THREADS - 1) / THREADS;
  static_assert(UNITS % 64 == 0, "whole waves hold a unit or none");
  float v[N][8];
};

// Row and k half of unit f: in memory order, so that a wave's loads are contiguous.
template <int MODE, int ROWS>
__device__ __forceinline__ void unit_coords(int f, int& r, int& h) {
  if (MODE == kVecMN) { r = f % ROWS; h = f / ROWS; }
  else { r = f >> 1; h = f & 1; }
}

// Vector modes read through buffer loads: each lane's byte offset within a slice is fixed for
// the whole K loop, and each slice only moves the resource's base and extent (scalar work), so
// the loop carries no per-load address arithmetic.  Reads outside the resource return zero,
// which zeroes k past the end of the K range and slices past the last one; rows past R read
// zero (kVecK, kAnyK) or in-bounds values that only feed output rows/columns never stored
// (kVecMN).  On a ragged last slice a kVecK lane whose k lies past the end moves its offset out
// of range; kAnyK, whose end may fall inside a lane's four k, loads that slice by single dwords
// (its whole slices are dwordx4 loads too: buffer loads need only 4-byte alignment).  kStrided
// loads every slice by single dwords, rows past the end moved out of range, and zeroes k past the
// end in registers (2048 x 3072 x 768 with every second column of a wider x: 103 us, 132 with
// kScalar loads of both operands; with every second column of a wider W 69 and 134).
template <int MODE, int ROWS, int THREADS>
struct LoadPlan {
  using S = Slice<ROWS, THREADS>;
  static constexpr int N = S::N;
  const float* base;  // (row0, k0) of the tile
  int64_t s_row, s_k;
  int rows;           // valid rows from row0: min(ROWS, R - row0) (kVecK) or R - row0 (kVecMN)
  int row0, kb, R, ke;
  int voff[N];        // vector modes: byte offset of the lane's unit within a slice
  int kq;             // not kVecMN: the unit's first k within a slice (the same for all its units)
  __device__ __forceinline__ void init(const float* b, int64_t sr, int64_t sk, int r0, int k0,
                                       int R_, int K_, int tid) {
    s_row = sr; s_k = sk; row0 = r0; kb = k0; R = R_; ke = K_;
    if (MODE == kVecK || MODE == kAnyK || MODE == kStrided) {
      base = b + (int64_t)r0 * sr + (int64_t)k0 * (MODE == kStrided ? sk : 1);
      rows = min(ROWS, R_ - r0);
    } else if (MODE == kVecMN) {
      base = b + (int64_t)k0 * sk + r0;
      rows = R_ - r0;
    } else {
      base = b;
    }
    kq = (tid & 1) * 8;
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int f = tid + THREADS * u;
      int r, h;
      unit_coords<MODE, ROWS>(f, r, h);
      voff[u] = MODE == kVecMN     ? (int)(((int64_t)(8 * h) * sk + r) * 4)
                : MODE == kStrided ? (int)(((int64_t)r * sr + 8 * h * sk) * 4)
                                   : (int)(((int64_t)r * sr + 8 * h) * 4);
      if (f >= S::UNITS || (MODE == kStrided && r >= rows)) voff[u] = (int)0x80000000;
    }
  }
  static __device__ __forceinline__ void coords(int f, int& r, int& h) {
    unit_coords<MODE, ROWS>(f, r, h);
  }
  // Slice t (k from kb + t * kGemmK) into registers.
  __device__ __forceinline__ void load(S& L, int t, int tid) const {
    const int k0 = kb + t * kGemmK;
    const int klim = min(kGemmK, ke - k0);  // <= 0 past the end: nothing in range
    if (MODE == kScalar) {
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const int f = tid + THREADS * u;
        int r, h;
        unit_coords<MODE, ROWS>(f, r, h);
        const int gr = row0 + r, gk = k0 + 8 * h;
#pragma unroll
        for (int e = 0; e < 8; ++e)
          L.v[u][e] = (gr < R && gk + e < ke && f < S::UNITS)
                          ? base[(int64_t)gr * s_row + (int64_t)(gk + e) * s_k] : 0.0f;
      }
      return;
    }
    // 32 bits reach (pick_mode), and the product by 0 or 1 stays scalar arithmetic: a conditional
    // becomes a branch that splits the K loop's schedule (64 more VGPRs where both operands load
    // dwords, scratch in some kStrided kernels).
    const float* bt = base + (int64_t)t * kGemmK * (MODE == kVecK || MODE == kAnyK ? 1 : s_k);
    const int last = MODE == kVecK || MODE == kAnyK ? (rows - 1) * (int)s_row + klim
                     : MODE == kVecMN               ? (klim - 1) * (int)s_k + rows
                                      : (rows - 1) * (int)s_row + (klim - 1) * (int)s_k + 1;
    const int nbytes = last * 4 * min(max(klim, 0), 1);
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(bt), (short)0, nbytes, 0x00020000);
    if (MODE == kAnyK && klim < kGemmK) {  // uniform
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e)
          L.v[u][e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rs, kq + e < klim ? voff[u] + 4 * e : (int)0x80000000, 0, 0));
      return;
    }
#pragma unroll
    for (int u = 0; u < N; ++u) {
      if (MODE == kVecK || MODE == kAnyK) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
          const int vo = MODE == kAnyK || kq + 4 * q < klim ? voff[u] + 16 * q : (int)0x80000000;
          const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, vo, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) L.v[u][4 * q + e] = __uint_as_float(w[e]);
        }
      } else {
        const int kbytes = (int)(s_k * 4);
#pragma unroll
        for (int e = 0; e < 8; ++e)
          L.v[u][e] = __uint_as_float(
              __builtin_amdgcn_raw_buffer_load_b32(rs, voff[u], e * kbytes, 0));
      }
    }
  }
  // kStrided: what slice t, in registers, holds past the end of K (other elements of the operand).
  __device__ __forceinline__ void mask(S& L, int t) const {
    if constexpr (MODE == kStrided) {
      const int klim = ke - (kb + t * kGemmK) - kq;
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) L.v[u][e] = e < klim ? L.v[u][e] : 0.0f;
    }
  }
};

// Splits a slice and stores its parts: LDS image [part][half][row][8 k], part p at p * PLANE.
template <int MODE, int ROWS, int THREADS, int PLANE>
__device__ __forceinline__ void store_slice(const Slice<ROWS, THREADS>& L, char* lds, int tid) {
  using S = Slice<ROWS, THREADS>;
#pragma unroll
  for (int u = 0; u < S::N; ++u) {
    const int f = tid + THREADS * u;
    if (S::UNITS % THREADS != 0 && f >= S::UNITS) continue;  // wave-uniform
    int r, h;
    unit_coords<MODE, ROWS>(f, r, h);
    bf16x8 p[3];
    split_bf16<true>(L.v[u], p);
    char* at = lds + h * (PLANE / 2) + r * 16;
#pragma unroll
    for (int q = 0; q < 3; ++q) *reinterpret_cast<bf16x8*>(at + q * PLANE) = p[q];
  }
}

// One wave's operand fragments of one K-slice: the three parts of each MFMA tile row (A) or
// column (B); lane half h supplies k = 8h .. 8h + 7.
template <class TL>
struct Frags {
  bf16x8 a[TL::MB][3], b[TL::NB][3];
};

template <class TL>
__device__ __forceinline__ void read_frags(const char* buf, Frags<TL>& f, int wm, int wn,
                                           int half, int col) {
  constexpr int PA = TL::plane(TL::BM), PB = TL::plane(TL::BN);
  const char* ap = buf + half * (PA / 2) + (wm * (TL::BM / TL::WM) + col) * 16;
  const char* bp = buf + TL::A_BYTES + half * (PB / 2) + (wn * (TL::BN / TL::WN) + col) * 16;
  // the parts that the next slice's first products take come first
#pragma unroll
  for (int q = 2; q >= 0; --q) {
#pragma unroll
    for (int i = 0; i < TL::MB; ++i)
      f.a[i][q] = *reinterpret_cast<const bf16x8*>(ap + q * PA + i * 512);
#pragma unroll
    for (int j = 0; j < TL::NB; ++j)
      f.b[j][q] = *reinterpret_cast<const bf16x8*>(bp + q * PB + j * 512);
  }
}

// Products [P0, P1) of the six of a slice, smallest first, in the same order for every
// accumulator and tile type (a fused GELU product gives the bits of the plain one).  a0 b0 has
// an accumulator of its own: the matrix pipe rounds small addends of a large accumulator
// downward, which with one accumulator left a mean error of -4e-8 of the result's RMS at K = 768
// (-4e-7 at 8192; column sums of such results showed it), and with two none that could be
// measured, and a relative error of 1.6e-7 (5.7e-7) where one gives 4.2e-7 (1.4e-6).
template <class TL, int P0, int P1>
__device__ __forceinline__ void mma_products(const Frags<TL>& f, f32x16 (&acc)[TL::MB][TL::NB],
                                             f32x16 (&low)[TL::MB][TL::NB]) {
#pragma unroll
  for (int p = P0; p < P1; ++p)
#pragma unroll
    for (int i = 0; i < TL::MB; ++i)
#pragma unroll
      for (int j = 0; j < TL::NB; ++j) {
        f32x16& c = p == 5 ? acc[i][j] : low[i][j];
        c = mfma_bf16(f.a[i][kSplitA[p]], f.b[j][kSplitB[p]], c);
      }
}

// Stores a wave's block of one output tile.  RAW: the accumulators as they are (split-K
// partials); otherwise alpha, bias, the causal mask (MASK) and the pointwise stage ACT.  `Cz`
// and `Xz` are the batch's output and aux planes, row stride srow.  The block is stored through
// buffer stores from its origin: a lane's column is a fixed per-lane offset (moved out of range
// when the column lies past N), each row's offset is scalar, and rows past M fall outside the
// resource, so the stores need no per-element bounds tests or 64-bit address arithmetic.
// One element of the epilogue: v = alpha * acc + bias, the mask, the gradient stages (xg: the
// aux value), then the value stored to C (cv) and, for the forward GELU stages, to aux (xv).
template <int ACT, bool RAW, bool MASK>
__device__ __forceinline__ void epilogue_value(float a, float bias, float xg,
                                               const GemmEpilogue& ep, bool masked, float& cv,
                                               float& xv) {
  float val = a;
  if (!RAW) {
    val = fmaf(ep.alpha, val, bias);
    if (MASK && masked) val = -INFINITY;
    if constexpr (ACT == kActGeluGrad) val = gelu_grad(xg, val);
    else if constexpr (ACT == kActGeluTanhGrad) val = gelu_tanh_grad(xg, val);
    else if constexpr (ACT == kActMulAux) val = val * xg;
  }
  // The derivative forms store gelu'(v) (its product with g = 1.0 is exact, so a later
  // kActMulAux stage gives gelu_grad(v, g) bit for bit) and gelu(v).
  cv = val;
  if (!RAW && ACT == kActGeluDeriv) cv = gelu_grad(val, 1.0f);
  if (!RAW && ACT == kActGeluTanhDeriv) cv = gelu_tanh_grad(val, 1.0f);
  xv = 0.0f;
  if (!RAW && (ACT == kActGelu || ACT == kActGeluDeriv)) xv = gelu_f(val);
  if (!RAW && (ACT == kActGeluTanh || ACT == kActGeluTanhDeriv)) xv = gelu_tanh_f(val);
}

// The wave's block when it spans 2^31 bytes or more (row strides of 2^22 floats and up), which
// 32-bit buffer offsets cannot address: plain stores through 64-bit addresses with explicit
// row and column bounds, the same values as block_store's.
template <class TL, int ACT, bool RAW, bool MASK>
__device__ __forceinline__ void block_store_wide(const f32x16 (&acc)[TL::MB][TL::NB], float* Cz,
                                              float* Xz, int64_t srow, const GemmEpilogue& ep,
                                              int M, int N, int mw, int nw, int half, int col) {
  constexpr bool kGrad =
      !RAW && (ACT == kActGeluGrad || ACT == kActGeluTanhGrad || ACT == kActMulAux);
  constexpr bool kAux = !RAW && (ACT == kActGelu || ACT == kActGeluDeriv ||
                                 ACT == kActGeluTanh || ACT == kActGeluTanhDeriv);
#pragma unroll
  for (int j = 0; j < TL::NB; ++j) {
    const int n = nw + j * 32 + col;
    if (n >= N) continue;
    const float bias = (!RAW && ep.bias) ? ep.bias[(int64_t)n * ep.bias_stride] : 0.0f;
#pragma unroll
    for (int i = 0; i < TL::MB; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = mw + i * 32 + mfma_row(r, half);
        if (m >= M) continue;
        const int64_t at = (int64_t)m * srow + n;
        const float xg = kGrad ? Xz[at] : 0.0f;
        float cv, xv;
        epilogue_value<ACT, RAW, MASK>(acc[i][j][r], bias, xg, ep, n > m, cv, xv);
        Cz[at] = cv;
        if (kAux) Xz[at] = xv;
      }
    }
  }
}

template <class TL, int ACT, bool RAW, bool MASK>
__device__ __forceinline__ void block_store(const f32x16 (&acc)[TL::MB][TL::NB], float* Cz,
                                            float* Xz, int64_t srow, const GemmEpilogue& ep,
                                            int M, int N, int mw, int nw, int half, int col) {
  constexpr int MB = TL::MB, NB = TL::NB;
  constexpr int WROWS = TL::BM / TL::WM, WCOLS = TL::BN / TL::WN;
  constexpr bool kGrad =
      !RAW && (ACT == kActGeluGrad || ACT == kActGeluTanhGrad || ACT == kActMulAux);
  const int64_t span = ((int64_t)(min(WROWS, M - mw) - 1) * srow + min(WCOLS, N - nw)) * 4;
  if (span >= ((int64_t)1 << 31) || (int64_t)WROWS * srow * 4 >= ((int64_t)1 << 31)) {
    block_store_wide<TL, ACT, RAW, MASK>(acc, Cz, Xz, srow, ep, M, N, mw, nw, half, col);
    return;
  }
  float* Cb = Cz + (int64_t)mw * srow + nw;
  float* Xb = Xz ? Xz + (int64_t)mw * srow + nw : Cb;
  const int nbytes = (int)span;
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(Cb, (short)0, nbytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(Xb, (short)0, nbytes, 0x00020000);
  const int row_bytes = (int)(srow * 4);
  int vo[NB];
  float bv[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = nw + j * 32 + col;
    bv[j] = (!RAW && ep.bias && n < N) ? ep.bias[(int64_t)n * ep.bias_stride] : 0.0f;
    vo[j] = n < N ? 4 * half * row_bytes + (j * 32 + col) * 4 : (int)0x80000000;
  }
  // The gradient stages read the pre-activations (kActMulAux: the saved derivatives): all of
  // the block's loads are issued before its first store, so their latencies overlap.  Each
  // element's aux value is read before any store, so dx may alias it.
  float xg[kGrad ? MB : 1][kGrad ? NB : 1][16];
  if constexpr (kGrad) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          xg[i][j][r] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              rx, vo[j], (i * 32 + 8 * (r >> 2) + (r & 3)) * row_bytes, 0));
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = nw + j * 32 + col;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int so = (i * 32 + 8 * (r >> 2) + (r & 3)) * row_bytes;
        float cv, xv;
        epilogue_value<ACT, RAW, MASK>(acc[i][j][r], bv[j], kGrad ? xg[i][j][r] : 0.0f, ep,
                                       n > mw + i * 32 + mfma_row(r, half), cv, xv);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(cv), rc, vo[j], so, 0);
        if (!RAW && (ACT == kActGelu || ACT == kActGeluDeriv || ACT == kActGeluTanh ||
                     ACT == kActGeluTanhDeriv))
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(xv), rx, vo[j], so, 0);
      }
    }
  }
}

// The tile's sums with FP32 MFMAs, for operands or sums that the parts cannot hold: the same
// loads, FP32 slices in LDS as [k][row], one buffer.  Every thread of the workgroup calls it.
template <class TL, class PA, class PB>
__device__ __forceinline__ void exact_tile(const PA& pa, const PB& pb, typename PA::S& la,
                                           typename PB::S& lb, float* smem, int nk, int tid,
                                           int tid_b, int wm, int wn, int half, int col,
                                           f32x16 (&acc)[TL::MB][TL::NB]) {
  constexpr int BM = TL::BM, BN = TL::BN;
#pragma unroll
  for (int i = 0; i < TL::MB; ++i)
#pragma unroll
    for (int j = 0; j < TL::NB; ++j) acc[i][j] = zero16();
  float* const as = smem;
  float* const bs = smem + kGemmK * BM;
  auto put = [&](const auto& plan, const auto& L, float* lds, int rows, int id) {
    using S = std::remove_cvref_t<decltype(L)>;
#pragma unroll
    for (int u = 0; u < S::N; ++u) {
      const int f = id + TL::THREADS * u;
      if (f >= S::UNITS) continue;
      int r, h;
      plan.coords(f, r, h);
#pragma unroll
      for (int e = 0; e < 8; ++e) lds[(8 * h + e) * rows + r] = L.v[u][e];
    }
  };
  for (int t = 0; t < nk; ++t) {
    pa.load(la, t, tid);
    pb.load(lb, t, tid_b);
    pa.mask(la, t);
    pb.mask(lb, t);
    __syncthreads();
    put(pa, la, as, BM, tid);
    put(pb, lb, bs, BN, tid_b);
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kGemmK / 2; ++e) {
      float a[TL::MB], b[TL::NB];
#pragma unroll
      for (int i = 0; i < TL::MB; ++i)
        a[i] = as[(2 * e + half) * BM + wm * (BM / TL::WM) + i * 32 + col];
#pragma unroll
      for (int j = 0; j < TL::NB; ++j)
        b[j] = bs[(2 * e + half) * BN + wn * (BN / TL::WN) + j * 32 + col];
#pragma unroll
      for (int i = 0; i < TL::MB; ++i)
#pragma unroll
        for (int j = 0; j < TL::NB; ++j) acc[i][j] = mfma32(a[i], b[j], acc[i][j]);
    }
  }
}

// split_ws == nullptr: out = alpha * A B (+ bias, mask) written through C.
// split_ws != nullptr: blockIdx.z = s * Z + z covers K range [s*kchunk, (s+1)*kchunk) and the raw
// partial sum goes to split_ws[s][z][m][n] (dense); gemm_splitk_reduce finishes the epilogue.
// CS (Z == 1, B in kVecMN mode): the workgroups of the first row of tiles also sum B's columns
// over their K range, into ep.colsum or, split, into row s of the [S][N] block that follows
// the partial products.
template <class TL, int AMODE, int BMODE, bool CS = false>
__global__ __launch_bounds__(TL::THREADS, 2) void gemm_kernel(GemmOperand A, GemmOperand B,
                                                              GemmOut C, GemmEpilogue ep, int M,
                                                              int N, int K, int zin, int Z,
                                                              int kchunk,
                                                              float* __restrict__ split_ws) {
  constexpr int BM = TL::BM, BN = TL::BN, THREADS = TL::THREADS;
  constexpr int MB = TL::MB, NB = TL::NB;
  __shared__ __attribute__((aligned(16))) char smem[2 * TL::BUF_BYTES];
  const int tid = threadIdx.x;
  // Where half of the threads hold an operand's slice (the 64x64 tile), the other half holds B's.
  const int tid_b = 2 * BM + 2 * BN <= THREADS ? tid ^ (2 * BM) : tid;
  const int lane = tid & 63, wave = wave_index();
  const int half = lane >> 5, col = lane & 31;
  const int wm = wave / TL::WN, wn = wave % TL::WN;

  // Without a K split: the output tiles of all batches in one row-major list (batch, m, n; n
  // fastest), each XCD walking a contiguous run of it, so the workgroups that share an A row
  // block run on one XCD and read it into one L2.  Split along K: tile (x, y), z = split * Z +
  // batch.
  int n0, m0, z, split;
  if (split_ws == nullptr) {
    const int ntn = (N + BN - 1) / BN, ntiles = ntn * ((M + BM - 1) / BM);
    const int w = xcd_work_item(blockIdx.x, ntiles * Z);
    if (w >= ntiles * Z) return;
    z = w / ntiles;
    const int t = w - z * ntiles;
    n0 = (t % ntn) * BN;
    m0 = (t / ntn) * BM;
    split = 0;
  } else {
    n0 = blockIdx.x * BN;
    m0 = blockIdx.y * BM;
    z = blockIdx.z % Z;
    split = blockIdx.z / Z;
  }
  const int zo = z / zin, zi = z - zo * zin;
  const float* Ab = A.p + zo * A.s_outer + zi * A.s_inner;
  const float* Bb = B.p + zo * B.s_outer + zi * B.s_inner;
  const int kb = split * kchunk;
  const int ke = min(K, kb + kchunk);

  // A rows are m with (s_row, s_col) = (m, k); B "rows" are n with (n, k) = (s_col, s_row).
  // Global loads run two K-slices ahead of the MFMAs (two register sets, alternating), so a
  // slice's loads have two slices of MFMA work to arrive; LDS is double buffered.  Vector-mode
  // reads past K, or past the last slice, return zero.
  using PlanA = LoadPlan<AMODE, BM, THREADS>;
  using PlanB = LoadPlan<BMODE, BN, THREADS>;
  constexpr int PA = TL::plane(BM), PB = TL::plane(BN);
  PlanA pa;
  PlanB pb;
  pa.init(Ab, A.s_row, A.s_col, m0, kb, M, ke, tid);
  pb.init(Bb, B.s_col, B.s_row, n0, kb, N, ke, tid_b);
  typename PlanA::S la0, la1;
  typename PlanB::S lb0, lb1;
  const int nk = (ke - kb + kGemmK - 1) / kGemmK;
  static_assert(!CS || BMODE == kVecMN, "column sums come from n-contiguous B slices");

  // CS: a lane's B unit holds the same column and k half in every slice, so the lane sums its
  // values as the slices pass through its registers (slices past the end are zero), one sum per
  // k of the unit: sixteen short chains a column, combined after the loop.
  float cs[CS ? PlanB::N : 1][8];
  auto add_cs = [&](const typename PlanB::S& lb) {
    if constexpr (CS) {
#pragma unroll
      for (int u = 0; u < PlanB::N; ++u)
#pragma unroll
        for (int e = 0; e < 8; ++e) cs[u][e] += lb.v[u][e];
    }
  };
#pragma unroll
  for (int u = 0; u < (CS ? PlanB::N : 1); ++u)
#pragma unroll
    for (int e = 0; e < 8; ++e) cs[u][e] = 0.0f;

  f32x16 acc[MB][NB], low[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) { acc[i][j] = zero16(); low[i][j] = zero16(); }

  // Slice count rounded up to even: slices past the end read nothing in range, so they are
  // stored as zeros and add nothing.  The loop then has no conditional loads or stores, which
  // keeps the compiler's wait counts exact (a load issued two slices ahead is not waited for
  // until its LDS store).
  const int nk2 = (nk + 1) & ~1;
  char* const buf0 = smem;
  char* const buf1 = smem + TL::BUF_BYTES;
  pa.load(la0, 0, tid);
  pb.load(lb0, 0, tid_b);
  pa.load(la1, 1, tid);
  pb.load(lb1, 1, tid_b);
  pa.mask(la0, 0);
  pb.mask(lb0, 0);
  store_slice<AMODE, BM, THREADS, PA>(la0, buf0, tid);
  store_slice<BMODE, BN, THREADS, PB>(lb0, buf0 + TL::A_BYTES, tid_b);
  add_cs(lb0);
  __syncthreads();

  // Each slice's MFMAs run in two parts around the barrier that publishes the next slice.  The
  // first part (the three smallest products) carries the next-but-one slice's global loads and
  // the next slice's split and LDS stores; right after the barrier the wave issues the next
  // slice's fragment reads, which complete under the second part, so no wave waits on LDS
  // latency before its MFMAs.  A buffer is rewritten only after the barrier that follows every
  // wave's reads of it (the barrier waits for outstanding LDS reads).
  Frags<TL> f0, f1;
  read_frags<TL>(buf0, f0, wm, wn, half, col);
  auto slice = [&](Frags<TL>& cur, Frags<TL>& nxt, typename PlanA::S& la_far,
                   typename PlanB::S& lb_far, typename PlanA::S& la_next,
                   typename PlanB::S& lb_next, char* nbuf, int t_far) {
    pa.load(la_far, t_far, tid);
    pb.load(lb_far, t_far, tid_b);
    mma_products<TL, 0, 3>(cur, acc, low);
    pa.mask(la_next, t_far - 1);
    pb.mask(lb_next, t_far - 1);
    store_slice<AMODE, BM, THREADS, PA>(la_next, nbuf, tid);
    store_slice<BMODE, BN, THREADS, PB>(lb_next, nbuf + TL::A_BYTES, tid_b);
    add_cs(lb_next);
    if constexpr (PlanA::S::UNITS % THREADS == 0 && PlanB::S::UNITS % THREADS == 0 &&
                  !(AMODE == kStrided && BMODE == kVecK)) {
      // Each MFMA takes the pipe for eight vector instructions' time: the slice's splits go
      // between them, evenly.  Left alone, the scheduler ran most of every second slice's after
      // the last MFMA (4096 x 3072 x 1536: 214 us, 198 so; one workgroup a CU, 2048 x 2048 x 2048:
      // 107 and 98).  Strided A beside W^T's rows is left to the scheduler: its eight single loads a
      // unit, issued between the MFMAs too, and full registers wait (2048 x 768 x 3072: 116 us
      // interleaved, 106 not).
      constexpr int kMfmas = 6 * MB * NB;
      constexpr int kValu = 52 * (PlanA::N + PlanB::N);
#pragma unroll
      for (int i = 0; i < kMfmas; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, (kValu + kMfmas - 1) / kMfmas, 0);  // VALU
      }
    }
    __syncthreads();
    read_frags<TL>(nbuf, nxt, wm, wn, half, col);
    mma_products<TL, 3, 6>(cur, acc, low);
  };
  for (int t = 0; t < nk2; t += 2) {
    // slice t in f0; slices t+2 (set 0) and t+1 (set 1, stored below) in flight
    slice(f0, f1, la0, lb0, la1, lb1, buf1, t + 2);
    slice(f1, f0, la1, lb1, la0, lb0, buf0, t + 3);
  }

  // Sums that are not finite (see the top): the whole workgroup runs the tile again.
  bool odd = false;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      acc[i][j] += low[i][j];
      odd |= not_finite(acc[i][j]);
      acc[i][j] *= kSplitUnscale * kSplitUnscale;
    }
  if (__syncthreads_or(odd))
    exact_tile<TL>(pa, pb, la0, lb0, reinterpret_cast<float*>(smem), nk, tid, tid_b, wm, wn, half,
                   col, acc);

  if constexpr (CS) {
    if (m0 == 0) {  // workgroup-uniform
      // Units f and f + BN hold the two k halves of column f.
      float* const half1 = reinterpret_cast<float*>(smem);
      auto unit_sum = [&](int u) {
        return ((cs[u][0] + cs[u][1]) + (cs[u][2] + cs[u][3])) +
               ((cs[u][4] + cs[u][5]) + (cs[u][6] + cs[u][7]));
      };
      __syncthreads();  // every wave is done with the slices
#pragma unroll
      for (int u = 0; u < PlanB::N; ++u) {
        const int f = tid_b + THREADS * u;
        if (f >= BN && f < 2 * BN) half1[f - BN] = unit_sum(u);
      }
      __syncthreads();
      float* out = split_ws ? split_ws + (int64_t)gridDim.z * M * N + (int64_t)split * N
                            : ep.colsum;
#pragma unroll
      for (int u = 0; u < PlanB::N; ++u) {
        const int f = tid_b + THREADS * u;
        if (f < BN && n0 + f < N) out[n0 + f] = unit_sum(u) + half1[f];
      }
    }
  }

  const int mw = m0 + wm * (BM / TL::WM), nw = n0 + wn * (BN / TL::WN);
  if (mw >= M || nw >= N) return;
  if (split_ws != nullptr) {
    float* Pz = split_ws + ((int64_t)split * Z + z) * M * N;
    block_store<TL, kActNone, true, false>(acc, Pz, nullptr, N, ep, M, N, mw, nw, half, col);
    return;
  }
  float* Cz = C.p + zo * C.s_outer + zi * C.s_inner;
  float* Xz = ep.aux ? ep.aux + zo * C.s_outer + zi * C.s_inner : nullptr;
  // The pointwise stage is a scalar branch here, outside the K loop: one kernel per tile and
  // operand order instead of one per stage.
  auto store = [&]<int ACT, bool MASK>() {
    block_store<TL, ACT, false, MASK>(acc, Cz, Xz, C.s_row, ep, M, N, mw, nw, half, col);
  };
  if constexpr (CS) {
    store.template operator()<kActNone, false>();
    return;
  }
  if (ep.causal_mask) store.template operator()<kActNone, true>();
  else if (ep.act == kActNone) store.template operator()<kActNone, false>();
  else if (ep.act == kActGelu) store.template operator()<kActGelu, false>();
  else if (ep.act == kActGeluGrad) store.template operator()<kActGeluGrad, false>();
  else if (ep.act == kActGeluTanh) store.template operator()<kActGeluTanh, false>();
  else if (ep.act == kActGeluTanhGrad) store.template operator()<kActGeluTanhGrad, false>();
  else if (ep.act == kActGeluDeriv) store.template operator()<kActGeluDeriv, false>();
  else if (ep.act == kActGeluTanhDeriv) store.template operator()<kActGeluTanhDeriv, false>();
  else store.template operator()<kActMulAux, false>();
}

// Fixed-order sum of the split-K partials plus the epilogue of gemm_kernel; with ep.colsum also
// of the per-split column sums stored after them.
__global__ __launch_bounds__(256) void gemm_splitk_reduce(const float* __restrict__ ws, int S,
                                                          int Z, int M, int N, GemmOut C,
                                                          GemmEpilogue ep, int zin) {
  const int64_t total = (int64_t)Z * M * N;
  const int64_t plane = total;
  const int64_t all = total + (ep.colsum ? N : 0);
  for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < all;
       e += (int64_t)gridDim.x * 256) {
    if (e >= total) {
      const float* p = ws + (int64_t)S * plane + (e - total);
      float t = p[0];
      for (int s = 1; s < S; ++s) t += p[(int64_t)s * N];
      ep.colsum[e - total] = t;
      continue;
    }
    float acc = ws[e];
    for (int s = 1; s < S; ++s) acc += ws[(int64_t)s * plane + e];
    const int64_t z = e / ((int64_t)M * N);
    const int64_t mn = e - z * M * N;
    const int m = (int)(mn / N), n = (int)(mn - (int64_t)m * N);
    const int64_t zo = z / zin, zi = z - zo * zin;
    float val = fmaf(ep.alpha, acc, ep.bias ? ep.bias[(int64_t)n * ep.bias_stride] : 0.0f);
    if (ep.causal_mask && n > m) val = -INFINITY;
    const int64_t off = zo * C.s_outer + zi * C.s_inner + (int64_t)m * C.s_row + n;
    if (ep.act == kActGeluGrad) val = gelu_grad(ep.aux[off], val);
    if (ep.act == kActGeluTanhGrad) val = gelu_tanh_grad(ep.aux[off], val);
    if (ep.act == kActMulAux) val = val * ep.aux[off];
    C.p[off] = ep.act == kActGeluDeriv       ? gelu_grad(val, 1.0f)
               : ep.act == kActGeluTanhDeriv ? gelu_tanh_grad(val, 1.0f)
                                             : val;
    if (ep.act == kActGelu || ep.act == kActGeluDeriv) ep.aux[off] = gelu_f(val);
    if (ep.act == kActGeluTanh || ep.act == kActGeluTanhDeriv) ep.aux[off] = gelu_tanh_f(val);
  }
}

// Load mode of an operand.  A: (s_row, s_col) = (m, k); B: (k, n).  `rows` is M for A and N for
// B.
int pick_mode(const GemmOperand& op, bool is_a, int64_t rows, int64_t K) {
  const int64_t s_k = is_a ? op.s_col : op.s_row;
  const int64_t s_mn = is_a ? op.s_row : op.s_col;
  // The buffer loads address a slice with 32-bit byte offsets and rely on rows (kVecK, kAnyK) or
  // k rows (kVecMN) not overlapping, so that reads past the valid range fall outside it.
  constexpr int64_t kMaxBytes = (int64_t)1 << 31;
  if (s_k == 1 && K >= 1 && s_mn >= K && (255 * s_mn + 64) * 4 < kMaxBytes) {
    // dwordx4 loads of a ragged end need it to fall between float4s
    const bool quads = K % 4 == 0 && aligned16(op.p) && s_mn % 4 == 0 && op.s_outer % 4 == 0 &&
                       op.s_inner % 4 == 0;
    return quads ? kVecK : kAnyK;
  }
  if (s_mn == 1 && rows >= 1 && s_k >= rows &&
      (63 * s_k + std::max<int64_t>(rows, 256)) * 4 < kMaxBytes)
    return kVecMN;
  if (s_k >= 0 && s_mn >= 0 && (127 * s_mn + 15 * s_k + 1) * 4 < kMaxBytes) return kStrided;
  return kScalar;
}

template <class TL, int AM, bool CS>
void dispatch_b(int bm, dim3 grid, hipStream_t st, const GemmOperand& A, const GemmOperand& B,
                const GemmOut& C, const GemmEpilogue& ep, int M, int N, int K, int zin, int Z,
                int kchunk, float* ws) {
  const dim3 block(TL::THREADS);
  if constexpr (CS) {  // the launcher has checked bm == kVecMN
    hipLaunchKernelGGL((gemm_kernel<TL, AM, kVecMN, true>), grid, block, 0, st, A, B, C, ep, M, N,
                       K, zin, Z, kchunk, ws);
    return;
  }
  if (bm == kVecK)
    hipLaunchKernelGGL((gemm_kernel<TL, AM, kVecK>), grid, block, 0, st, A, B, C, ep, M, N, K,
                       zin, Z, kchunk, ws);
  else if (bm == kAnyK)
    hipLaunchKernelGGL((gemm_kernel<TL, AM, kAnyK>), grid, block, 0, st, A, B, C, ep, M, N, K,
                       zin, Z, kchunk, ws);
  else if (bm == kStrided)
    hipLaunchKernelGGL((gemm_kernel<TL, AM, kStrided>), grid, block, 0, st, A, B, C, ep, M, N, K,
                       zin, Z, kchunk, ws);
  else
    hipLaunchKernelGGL((gemm_kernel<TL, AM, kVecMN>), grid, block, 0, st, A, B, C, ep, M, N, K,
                       zin, Z, kchunk, ws);
}

template <class TL, bool CS = false>
void dispatch_a(int am, int bm, dim3 grid, hipStream_t st, const GemmOperand& A,
                const GemmOperand& B, const GemmOut& C, const GemmEpilogue& ep, int M, int N,
                int K, int zin, int Z, int kchunk, float* ws) {
  // kScalar loads any layout: one kernel of it serves wherever either operand needs it
  if (!CS && (am == kScalar || bm == kScalar)) {
    hipLaunchKernelGGL((gemm_kernel<TL, kScalar, kScalar>), grid, dim3(TL::THREADS), 0, st, A, B,
                       C, ep, M, N, K, zin, Z, kchunk, ws);
    return;
  }
  if (am == kVecK)
    dispatch_b<TL, kVecK, CS>(bm, grid, st, A, B, C, ep, M, N, K, zin, Z, kchunk, ws);
  else if (am == kAnyK)
    dispatch_b<TL, kAnyK, CS>(bm, grid, st, A, B, C, ep, M, N, K, zin, Z, kchunk, ws);
  else if (am == kStrided)
    dispatch_b<TL, kStrided, CS>(bm, grid, st, A, B, C, ep, M, N, K, zin, Z, kchunk, ws);
  else if (am == kVecMN)
    dispatch_b<TL, kVecMN, CS>(bm, grid, st, A, B, C, ep, M, N, K, zin, Z, kchunk, ws);
  else if constexpr (CS)
    dispatch_b<TL, kScalar, true>(bm, grid, st, A, B, C, ep, M, N, K, zin, Z, kchunk, ws);
}

// K splits for a GEMM whose output tiles alone cannot fill the 256 CUs (1 = no split).  The
// busiest CU runs ceil(tiles S / 256) workgroups of ceil(K / S) each, and the split adds a
// round trip of S partial outputs through HBM; S in [1, 32] (at least 256 of K per split)
// minimises the sum.  Costs are in seconds at ~1.2 TFLOP/s per CU and ~5 TB/s of HBM.  E.g. the
// 768 x 3072 x 8192 weight gradient: 144 tiles, S = 5 (234 us + 17 us of reduction; S = 7, which
// the FP32 MFMA's 0.4 TFLOP/s gave, 235 + 20).
template <class TL>
int64_t splitk_factor(int64_t M, int64_t N, int64_t K, int64_t Z) {
  const int64_t tiles = ((M + TL::BM - 1) / TL::BM) * ((N + TL::BN - 1) / TL::BN) * Z;
  if (tiles >= 256 || K < 1024) return 1;
  constexpr double kCuFlops = 1.2e12, kHbmBytes = 5e12;
  const double tile_flop_per_k = 2.0 * TL::BM * TL::BN;
  int64_t best = 1;
  double best_cost = 0.0;
  for (int64_t s = 1; s <= 32 && (s == 1 || K / s >= 256); ++s) {
    const int64_t kchunk = ((K + s - 1) / s + kGemmK - 1) / kGemmK * kGemmK;
    const int64_t rounds = (tiles * s + 255) / 256;
    const double cost = (double)rounds * kchunk * tile_flop_per_k / kCuFlops +
                        (s > 1 ? 8.0 * s * M * N * Z / kHbmBytes : 0.0);
    if (s == 1 || cost < best_cost) { best = s; best_cost = cost; }
  }
  return best;
}

template <class TL>
int gemm_launch_tile(const GemmOperand& A, const GemmOperand& B, const GemmOut& C,
                     const GemmEpilogue& ep, int64_t M, int64_t N, int64_t K, int64_t Z,
                     int64_t zin, hipStream_t st, float* workspace, int64_t workspace_floats) {
  if (M <= 0 || N <= 0 || Z <= 0) return CTA_OK;
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX || Z > 65535 || zin <= 0)
    return fail(CTA_ERR_INVALID_ARGUMENT, "GEMM size out of range");
  int64_t S = splitk_factor<TL>(M, N, K, Z);
  const int64_t cs_floats = ep.colsum ? N : 0;  // per split
  if (S > 1 && (workspace == nullptr || workspace_floats < S * (Z * M * N + cs_floats))) S = 1;
  const int64_t kchunk =
      S > 1 ? ((K + S - 1) / S + kGemmK - 1) / kGemmK * kGemmK : std::max<int64_t>(K, 1);
  const int64_t ntiles = ((N + TL::BN - 1) / TL::BN) * ((M + TL::BM - 1) / TL::BM);
  if (ntiles * Z > INT32_MAX - kNumXcds || Z * S > 65535)
    return fail(CTA_ERR_INVALID_ARGUMENT, "GEMM grid too large");
  const dim3 grid = S > 1 ? dim3((unsigned)((N + TL::BN - 1) / TL::BN),
                                 (unsigned)((M + TL::BM - 1) / TL::BM), (unsigned)(Z * S))
                          : dim3(xcd_grid(ntiles * Z), 1, 1);
  if (grid.y > 65535) return fail(CTA_ERR_INVALID_ARGUMENT, "GEMM grid too large");
  float* ws = S > 1 ? workspace : nullptr;
  const int am = pick_mode(A, true, M, K);
  const int bm = pick_mode(B, false, N, K);
  const int iM = (int)M, iN = (int)N, iK = (int)K, izin = (int)zin, iZ = (int)Z, ikc = (int)kchunk;
  if (ep.colsum) {
    if (Z != 1 || bm != kVecMN || ep.act != kActNone || ep.causal_mask)
      return fail(CTA_ERR_INVALID_ARGUMENT,
                  "GEMM column sums need one batch, an n-contiguous B and no pointwise stage");
    dispatch_a<TL, true>(am, bm, grid, st, A, B, C, ep, iM, iN, iK, izin, iZ, ikc, ws);
  } else {
    if (ep.causal_mask && ep.act != kActNone)
      return fail(CTA_ERR_INVALID_ARGUMENT, "GEMM with both a mask and a pointwise stage");
    dispatch_a<TL>(am, bm, grid, st, A, B, C, ep, iM, iN, iK, izin, iZ, ikc, ws);
  }
  if (S > 1) {
    const int64_t total = Z * M * N + cs_floats;
    const unsigned rgrid = (unsigned)std::min<int64_t>((total + 255) / 256, 8192);
    hipLaunchKernelGGL(gemm_splitk_reduce, dim3(rgrid), dim3(256), 0, st, ws, (int)S, (int)Z,
                       (int)M, (int)N, C, ep, (int)zin);
  }
  return check_launch("gemm");
}

using WideTile = GemmTile<128, 128, 2, 2>;
using NarrowTile = GemmTile<64, 128, 2, 2>;
using SmallTile = GemmTile<64, 64, 2, 2>;

}  // namespace

// One launcher per tile type (defined in gemm_tiles_*.hip): gemm_launch_tile of that tile.
int gemm_launch_wide(const GemmOperand& A, const GemmOperand& B, const GemmOut& C,
                     const GemmEpilogue& ep, int64_t M, int64_t N, int64_t K, int64_t Z,
                     int64_t zin, hipStream_t st, float* workspace, int64_t workspace_floats);
int gemm_launch_narrow(const GemmOperand& A, const GemmOperand& B, const GemmOut& C,
                       const GemmEpilogue& ep, int64_t M, int64_t N, int64_t K, int64_t Z,
                       int64_t zin, hipStream_t st, float* workspace, int64_t workspace_floats);
int gemm_launch_small(const GemmOperand& A, const GemmOperand& B, const GemmOut& C,
                      const GemmEpilogue& ep, int64_t M, int64_t N, int64_t K, int64_t Z,
                      int64_t zin, hipStream_t st, float* workspace, int64_t workspace_floats);

}  // namespace cta
