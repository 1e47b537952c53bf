// Row-invariant linear layer for gfx950: C[M, N] = X[M, K] . W[N, K]^T.
//
// Replaces linear / _gemm of respect/kernels/gemm.py:11-41 (FixedLinear,
// respect/kernels/patch.py:26-37): bf16 inputs, fp32 accumulation, output in
// bf16 (the layers) or fp32 (the vocabulary projection, patch.py:23).
//
// Reduction order of every output element, fixed by (N, K) only:
//   K is cut into S equal chunks (S from splits(N, K), never from M); each
//   chunk is a chain of v_mfma_f32_16x16x32_bf16 over its 32-wide k-blocks in
//   increasing k; the chunk results are added in chunk order,
//   ((c0 + c1) + c2) + ..., then rounded once to the output type.
// So a row's output bits do not depend on how many rows the call carries.
//
// Work split (gemm_kernel: few rows; gemm_wide_kernel takes calls of many, with
// its own comment): workgroup = (16 W output columns, chunk s, 64-row tile), W = 4,
// 6 or 8 waves of 16 columns each (the host picks W per shape for speed; the
// chunk count S comes from 64-column tiles whatever W is, so W never changes
// a bit of the result).  W -- the large operand, read exactly once -- goes
// straight from HBM into the MFMA A operand registers (lane (n16, g4) loads
// W[col n16][k + 8 g4, +8): 16 contiguous bytes), in rounds of 8 k-blocks
// requested 3 rounds ahead.  X (at most 64 rows) is shared by the block's
// waves: each round of it is copied into LDS with direct-to-LDS loads laid
// out as MFMA B fragments (one conflict-free ds_read_b128 per 16-row tile and
// k-block).  The output tile D[n][m] comes back as 4 consecutive columns per
// lane.
//
// x may also come in the tiled layout (row stride RSPX_TILED, tiled_offset in
// common.h): a 64-row block's k-block is then four 1 KB operand tiles, and
// each direct-to-LDS load copies one whole tile instead of 16 rows x 64 B
// (gemm_kernel, gate/up [64 x 4096] . [24576 x 4096]^T on MI355X: 46 instead of 53
// us; gemm_wide_kernel loads row-major x in whole lines: 37.2 and 37.3).
// The LDS image, and so every result bit, is the same in both layouts.  The
// SwiGLU epilogue can write its output tiled for the next layer.
//
// S > 1 writes fp32 chunk partials [S][M][N] into the caller's workspace and
// a second kernel sums them in chunk order and rounds.
//
// W may also come in a tiled layout (row stride RSPX_TILED; written by
// rspx_linear_tile_weight from the row-major matrix): 16-row slabs of
// 16 K + kWSlabPad elements, slab n / 16 holding the K / 32 tiles of its rows
// one after the other, tile k / 32 holding element (n, k) at
// (n % 16 + 16 ((k % 32) / 8)) 8 + k % 8 -- lane n % 16 + 16 g of a wave
// loads its MFMA A operand (row n % 16, k 8 g .. 8 g + 7) as 16 contiguous
// bytes of one 1 KB tile.  The TCP (vector L1) then handles one 8 KB piece per
// wave and round instead of 16 rows of 512 bytes on 16 pages (q/k/v, o,
// gate/up, down at 64 rows, tiled x: 12.3 / 9.1 / 37.2 / 20.7 us instead of 13.2 /
// 9.9 / 43.6 / 24.2; one row 11.0 / 7.9 / 34.9 / 18.7 instead of 11.3 / 8.5 /
// 34.4 / 19.5).  The same bits as the row-major W.

#include "common.h"
#include "respect_amd.h"

namespace rspx {

namespace gemm {

constexpr int kSplitCols = 64;  // column tile the chunk count S is derived from
constexpr int kRows = 64;       // rows per workgroup (4 MFMA tiles)
constexpr int kRoundKB = 8;    // k-blocks of 32 per round
constexpr int kRoundK = 32 * kRoundKB;

typedef __attribute__((address_space(3))) void lds_void_t;
typedef __attribute__((address_space(3))) char lds_char_t;

__device__ __forceinline__ void x_dma16(__amdgpu_buffer_rsrc_t r, int voff, lds_char_t* dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void_t*)dst, 16, voff, 0, 0, 0);
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, int64_t nbytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0,
                                           (int)(nbytes > 0 ? nbytes : 0), 0x00020000);
}

struct Args {
  const uint16_t* x; int64_t sx;  // [M, K]
  const uint16_t* w; int64_t sw;  // [N, K]
  void* out; int64_t so;          // [M, N]: bf16 or fp32 (S == 1)
  float* part;                    // [S][M][N] fp32 (S > 1)
  int M, N, K, S, KC, out_fp32;
  int to_part;                    // write chunk partials even when S == 1
  int silu;                       // S == 1: columns (2i, 2i + 1) are (gate_i, up_i); out[m][i] = SwiGLU
  int x_tiled;                    // x in the tiled layout (sx unused)
  int out_tiled;                  // silu: out in the tiled layout of [M, N / 2] (so unused)
};

constexpr int kXResRounds = 4;   // X-resident blocks: K chunks of at most 4 rounds (128 KB of LDS)
// Elements after each 16-row slab of a tiled W.  Slabs of 4096 or 12288
// columns are a multiple of 128 KB long, so without it every wave's stream
// starts at the same offset modulo the memory-channel interleave; 128 bytes
// spread them (on MI355X, 64 rows: gate/up [24576, 4096] 40.2 instead of 41.7
// us with no pad, down [4096, 12288] 23.4 vs 24.1, vocabulary 238 vs 250; pads
// of 32, 128, 256, 512, 1024 and 2048 elements measured no better).
constexpr int kWSlabPad = 64;
constexpr int kOOB = 0x7ffffff0;  // a buffer offset past any descriptor: loads return 0, touch nothing
constexpr int kOOBRow = 0x40000000;  // the same for a whole lane chunk (k-block steps added stay below 2^31)

__device__ __forceinline__ void vm_wait0() { __builtin_amdgcn_s_waitcnt(0x0F70); }
__device__ __forceinline__ void raw_barrier() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc[t] += W . X^T over one round: X B-fragments of row tile t, k-block kb
// from LDS buffer xb, W A-fragments from registers wf.
template <int MT>
__device__ __forceinline__ void round_compute(const lds_char_t* xb, const u32x4 (&wf)[kRoundKB], f32x4 (&acc)[4],
                                              int lane) {
#pragma unroll
  for (int kb = 0; kb < kRoundKB; ++kb) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const u32x4 xf = *(const __attribute__((address_space(3))) u32x4*)(xb + (kb * 4 + t) * 1024 + 16 * lane);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[kb]),
                                                       __builtin_bit_cast(bf16x8, xf), acc[t], 0, 0, 0);
    }
  }
}

// X chunks of round rr into LDS buffer xb: the NC = 8 MT chunks c of a round
// (k-block kb = c / MT, row tile t = c % MT: rows 16 t + n16, k [8 g4, +8) of
// the block; only the MT row tiles the block computes) are spread over the W
// waves, wave w taking c = w, w + W, ...; chunk (kb, t) lands at
// (4 kb + t) KB of the buffer whatever MT is; xo[t] is this lane's offset of
// row tile t.  Rounds past the chunk and rows past M use out-of-range
// offsets: zeros, no memory traffic.  Wave w issues the same
// ceil((NC - w) / W) X chunks and 8 W loads per round on every path, so the
// waits below are exact counts.  xkb: bytes between consecutive k-blocks of
// one lane's chunk (64 row-major, 4096 tiled).
template <int W, int MT>
__device__ __forceinline__ void issue_x(__amdgpu_buffer_rsrc_t rx, const int (&xo)[4], int xkb, int rr, int nr,
                                        lds_char_t* xb, int w) {
  constexpr int NC = 8 * MT;
  const bool live = rr < nr;
  if constexpr (NC % W == 0 && W % MT == 0) {
    // Every chunk of wave w is row tile w % MT, whose offset the caller put in xo[0].
#pragma unroll
    for (int j = 0; j < NC / W; ++j) {
      const int kb = w / MT + (W / MT) * j;
      x_dma16(rx, live ? xo[0] + xkb * (rr * kRoundKB + kb) : kOOB, xb + (kb * 4 + w % MT) * 1024);
    }
  } else {
#pragma unroll
    for (int j = 0; j < (NC + W - 1) / W; ++j) {
      const int c = w + W * j;
      const int kb = c / MT, t = c % MT;
      if (c < NC) x_dma16(rx, live ? xo[t] + xkb * (rr * kRoundKB + kb) : kOOB, xb + (kb * 4 + t) * 1024);
    }
  }
  asm volatile("" ::: "memory");
}

// WKB: bytes between a lane's consecutive k-blocks of W (64 row-major, 1024
// tiled).
template <int WKB>
__device__ __forceinline__ void issue_w(__amdgpu_buffer_rsrc_t rw, int woff, int rr, int nr, u32x4 (&wf)[kRoundKB]) {
  const bool live = rr < nr;
#pragma unroll
  for (int kb = 0; kb < kRoundKB; ++kb)
    wf[kb] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                           rw, live ? woff + WKB * (rr * kRoundKB + kb) : kOOB, 0, 0));
  asm volatile("" ::: "memory");
}

// s_waitcnt vmcnt(n), 0 <= n <= 63 (a compile-time constant for 4 and 8
// waves, where one case remains; a per-wave value for 6 waves).
#define RSPX_VMW(v) __builtin_amdgcn_s_waitcnt(((v) & 15) | (((v) >> 4) << 14) | 0x70 | 0xF00)
__device__ __forceinline__ void vm_wait_n(int n) {
  switch (n) {
    case 0: RSPX_VMW(0); break;
    case 1: RSPX_VMW(1); break;
    case 2: RSPX_VMW(2); break;
    case 3: RSPX_VMW(3); break;
    case 4: RSPX_VMW(4); break;
    case 5: RSPX_VMW(5); break;
    case 6: RSPX_VMW(6); break;
    case 7: RSPX_VMW(7); break;
    case 8: RSPX_VMW(8); break;
    case 9: RSPX_VMW(9); break;
    case 10: RSPX_VMW(10); break;
    case 11: RSPX_VMW(11); break;
    case 12: RSPX_VMW(12); break;
    case 13: RSPX_VMW(13); break;
    case 14: RSPX_VMW(14); break;
    case 15: RSPX_VMW(15); break;
    case 16: RSPX_VMW(16); break;
    case 17: RSPX_VMW(17); break;
    case 18: RSPX_VMW(18); break;
    case 19: RSPX_VMW(19); break;
    case 20: RSPX_VMW(20); break;
    case 21: RSPX_VMW(21); break;
    case 22: RSPX_VMW(22); break;
    case 23: RSPX_VMW(23); break;
    case 24: RSPX_VMW(24); break;
    case 25: RSPX_VMW(25); break;
    case 26: RSPX_VMW(26); break;
    case 27: RSPX_VMW(27); break;
    case 28: RSPX_VMW(28); break;
    case 29: RSPX_VMW(29); break;
    case 30: RSPX_VMW(30); break;
    case 31: RSPX_VMW(31); break;
    case 32: RSPX_VMW(32); break;
    case 33: RSPX_VMW(33); break;
    case 34: RSPX_VMW(34); break;
    case 35: RSPX_VMW(35); break;
    case 36: RSPX_VMW(36); break;
    case 37: RSPX_VMW(37); break;
    case 38: RSPX_VMW(38); break;
    case 39: RSPX_VMW(39); break;
    case 40: RSPX_VMW(40); break;
    case 41: RSPX_VMW(41); break;
    case 42: RSPX_VMW(42); break;
    case 43: RSPX_VMW(43); break;
    case 44: RSPX_VMW(44); break;
    case 45: RSPX_VMW(45); break;
    case 46: RSPX_VMW(46); break;
    case 47: RSPX_VMW(47); break;
    case 48: RSPX_VMW(48); break;
    case 49: RSPX_VMW(49); break;
    case 50: RSPX_VMW(50); break;
    case 51: RSPX_VMW(51); break;
    case 52: RSPX_VMW(52); break;
    case 53: RSPX_VMW(53); break;
    case 54: RSPX_VMW(54); break;
    case 55: RSPX_VMW(55); break;
    case 56: RSPX_VMW(56); break;
    case 57: RSPX_VMW(57); break;
    case 58: RSPX_VMW(58); break;
    case 59: RSPX_VMW(59); break;
    case 60: RSPX_VMW(60); break;
    case 61: RSPX_VMW(61); break;
    case 62: RSPX_VMW(62); break;
    default: RSPX_VMW(63); break;
  }
}

// Columns n .. n + 3 of output row m (chunk s): the fp32 chunk partial, the
// SwiGLU of the two (gate, up) column pairs, or the result in fp32 or bf16.
__device__ __forceinline__ void store_tile(const Args& A, int s, int m, int n, f32x4 v) {
  if (m >= A.M) return;
  if (A.S > 1 || A.to_part) {
    *reinterpret_cast<f32x4*>(A.part + ((size_t)s * A.M + m) * A.N + n) = v;
  } else if (A.out_fp32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(A.out) + (int64_t)m * A.so + n) = v;
  } else if (A.silu) {
    // The bf16 gate/up values rspx_linear would store, then rspx_silu_mul's
    // arithmetic: bf16(bf16(silu(g)) * u) for columns n / 2 and n / 2 + 1.
    const uint32_t p0 = pack_bf16x2(v[0], v[1]);
    const uint32_t p1 = pack_bf16x2(v[2], v[3]);
    const float a0 = round_bf16(silu_f32(bf16_lo(p0))), a1 = round_bf16(silu_f32(bf16_lo(p1)));
    uint16_t* dst = static_cast<uint16_t*>(A.out) +
                    (A.out_tiled ? tiled_offset(m, n / 2, A.N / 2) : (int64_t)m * A.so + n / 2);
    *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2(a0 * bf16_hi(p0), a1 * bf16_hi(p1));
  } else {
    u32x2 o;
    o[0] = pack_bf16x2(v[0], v[1]);
    o[1] = pack_bf16x2(v[2], v[3]);
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(A.out) + (int64_t)m * A.so + n) = o;
  }
}

// Pipeline: W (the HBM stream) is requested 3 rounds ahead into a ring of 4
// register buffers, X (L2-resident) 1 round ahead into 2 LDS buffers.  Round
// r issues X(r + 1) and W(r + 3), then waits until X(r) and W(r) have landed.
// NR > 0: the NR rounds are unrolled at compile time, so every wait count is
// exact and the compiler's own waits for the W registers never drain the
// prefetch; NR == 0: a run-time loop (any round count, shallower prefetch).
//
// XRES (NR <= kXResRounds): the block's whole X chunk is copied into LDS up
// front (NR x 32 KB), so the main loop streams W with no X loads and no
// barriers.  The LDS image and the MFMA chain are those of the two-buffer
// form: the same bits.
//
// WT: W in the tiled layout (w row stride RSPX_TILED): a wave's 16 bytes per
// lane of a k-block are one 1 KB tile and its k-blocks follow each other, so
// a round of W is 8 KB in one piece instead of 16 rows x 512 bytes.  The MFMA
// operands, and so every bit, are the same.
template <int MT, int NR, int W, bool XRES = false, bool WT = false>
__global__ __launch_bounds__(64 * W) void gemm_kernel(Args A) {
  constexpr int WKB = WT ? 1024 : 64;
  static_assert(!XRES || (NR > 0 && NR <= kXResRounds), "X-resident blocks hold at most kXResRounds rounds");
  constexpr int kCols = 16 * W;
  __shared__ __attribute__((aligned(16))) char xs[XRES ? NR : 2][kRoundKB * 4 * 1024];  // 32 KB each
  constexpr int XB = kRoundKB * 4 * 1024;
  const int lane = __lane_id();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // X chunks this wave issues per round: a constant when W divides 8 MT, so
  // every wait count below is one too (a run-time count leaves the compiler's
  // own waits for the W registers conservative).
  constexpr int NC = 8 * MT;
  const int XPW = NC % W == 0 ? NC / W : (NC - w + W - 1) / W;
  const int n16 = lane & 15, g4 = lane >> 4;
  // Grid (column tile, K chunk, 64-row tile): no index divisions.  The
  // arguments the prologue needs are requested in one batch.
  const int nt = blockIdx.x, s = blockIdx.y, mt = blockIdx.z;
  asm volatile("" ::"s"(A.x), "s"(A.w), "s"(A.sx), "s"(A.sw), "s"(A.M), "s"(A.N), "s"(A.K), "s"(A.KC),
               "s"(A.x_tiled));
  const int col = nt * kCols + 16 * w;        // this wave's first column
  const int row0 = mt * kRows;
  const int k0 = s * A.KC;
  const int nr = NR > 0 ? NR : A.KC / kRoundK;
  const bool has_cols = col < A.N;            // N % 16 == 0: whole tiles only

  // X: rows [row0, M) from column k0.  W: this wave's 16 rows, columns
  // [k0, k0 + KC) (no bytes at all for a wave past N).
  // Tiled x: this block's chunk is (K - k0) / 32 k-blocks of four 1 KB tiles;
  // a wave whose tile lies past M loads nothing (rows past M inside a tile are
  // read but only reach output rows that are never stored).
  const int mrows = min(kRows, A.M - row0);
  // xoff[t]: this lane's offset of row tile t; when every chunk of a wave is
  // one row tile (issue_x), only its offset, kept in xoff[0].
  __amdgpu_buffer_rsrc_t rx;
  int xoff[4], xkb;
  auto tile_off = [&](int t) {
    return A.x_tiled ? (16 * t < mrows ? 1024 * t + 16 * lane : kOOBRow)
                     : 2 * ((16 * t + n16) * (int)A.sx + 8 * g4);
  };
  if (A.x_tiled) {
    rx = rsrc(A.x + (int64_t)mt * kRows * A.K + (int64_t)(k0 / 32) * 2048, (int64_t)(A.K - k0) * 128);
    xkb = 4096;
  } else {
    rx = rsrc(A.x + (int64_t)row0 * A.sx + k0, 2 * ((int64_t)(mrows - 1) * A.sx + (A.K - k0)));
    xkb = 64;
  }
  if constexpr (NC % W == 0 && W % MT == 0) {
    xoff[0] = tile_off(w % MT);
    xoff[1] = xoff[2] = xoff[3] = 0;
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t) xoff[t] = tile_off(t);
  }
  const __amdgpu_buffer_rsrc_t rw =
      WT ? rsrc(A.w + (int64_t)(has_cols ? col / 16 : 0) * ((A.K / 32) * 512 + kWSlabPad) + (k0 / 32) * 512,
                has_cols ? A.KC * 32 : 0)
         : rsrc(A.w + (int64_t)(has_cols ? col : 0) * A.sw + k0, has_cols ? 2 * (15 * A.sw + A.KC) : 0);
  const int woff = WT ? 16 * lane : 2 * (n16 * (int)A.sw + 8 * g4);

  lds_char_t* xl = (lds_char_t*)xs[0];
  f32x4 acc[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};

  if constexpr (XRES) {
    u32x4 wbuf[4][kRoundKB];
#pragma unroll
    for (int rr = 0; rr < NR; ++rr) issue_x<W, MT>(rx, xoff, xkb, rr, nr, xl + rr * XB, w);
    issue_w<WKB>(rw, woff, 0, nr, wbuf[0]);
    if constexpr (NR > 1) issue_w<WKB>(rw, woff, 1, nr, wbuf[1]);
    if constexpr (NR > 2) issue_w<WKB>(rw, woff, 2, nr, wbuf[2]);
    vm_wait_n(8 * (1 + (1 < NR) + (2 < NR)));  // every X chunk (issued before the W rounds) landed
    raw_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (r + 3 < NR) issue_w<WKB>(rw, woff, r + 3, nr, wbuf[(r + 3) & 3]);
      vm_wait_n(8 * ((r + 1 < NR) + (r + 2 < NR) + (r + 3 < NR)));  // W(r) landed
      round_compute<MT>(xl + r * XB, wbuf[r & 3], acc, lane);
    }
  } else if constexpr (NR > 0) {
    // Only loads whose data is used are issued (the compiler would drop the
    // others and the counts below would be off).  Exact wait per round: the
    // loads issued after the later of X(r) and W(r).
    u32x4 wbuf[4][kRoundKB];
    issue_x<W, MT>(rx, xoff, xkb, 0, nr, xl, w);
    issue_w<WKB>(rw, woff, 0, nr, wbuf[0]);
    if constexpr (NR > 1) issue_w<WKB>(rw, woff, 1, nr, wbuf[1]);
    if constexpr (NR > 2) issue_w<WKB>(rw, woff, 2, nr, wbuf[2]);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      if (r + 1 < NR) issue_x<W, MT>(rx, xoff, xkb, r + 1, nr, xl + ((r + 1) & 1) * XB, w);
      if (r + 3 < NR) issue_w<WKB>(rw, woff, r + 3, nr, wbuf[(r + 3) & 3]);
      const int younger = r == 0 ? 8 * ((1 < NR) + (2 < NR) + (3 < NR)) + XPW * (1 < NR)
                                 : 8 * ((r + 2 < NR) + (r + 3 < NR)) + XPW * (r + 1 < NR);
      vm_wait_n(younger);
      raw_barrier();
      round_compute<MT>(xl + (r & 1) * XB, wbuf[r & 3], acc, lane);
      raw_barrier();
    }
  } else {
    u32x4 wa[kRoundKB], wb[kRoundKB];
    issue_x<W, MT>(rx, xoff, xkb, 0, nr, xl, w);
    issue_w<WKB>(rw, woff, 0, nr, wa);
    for (int r = 0; r < nr; r += 2) {
      issue_x<W, MT>(rx, xoff, xkb, r + 1, nr, xl + XB, w);
      issue_w<WKB>(rw, woff, r + 1, nr, wb);
      vm_wait_n(8 + XPW);
      raw_barrier();
      round_compute<MT>(xl, wa, acc, lane);
      raw_barrier();
      if (r + 1 >= nr) break;
      issue_x<W, MT>(rx, xoff, xkb, r + 2, nr, xl, w);
      issue_w<WKB>(rw, woff, r + 2, nr, wa);
      vm_wait_n(8 + XPW);
      raw_barrier();
      round_compute<MT>(xl + XB, wb, acc, lane);
      raw_barrier();
    }
  }
  vm_wait0();
  if (!has_cols) return;

  // D[n][m]: lane (n16, g4) holds columns col + 4 g4 + e of row 16 t + n16.
#pragma unroll
  for (int t = 0; t < MT; ++t) store_tile(A, s, row0 + 16 * t + n16, col + 4 * g4, acc[t]);
}

// Many rows: workgroup = (16 W CT output columns, chunk s, 16 MT rows), W waves of
// CT 16-column tiles, every wave over all MT row tiles.  The same MFMA
// chain per element as gemm_kernel, in the same k order: the same bits.
//
// What bounds it: at one 16-column tile per wave (gemm_kernel) a k-block's X
// fragments (1 KB of LDS reads per MFMA) take twice the time of its MFMAs, and
// every 64 rows read W again.  A wave that owns CT column tiles reads an X
// fragment once for CT MFMAs, and MT = 8 row tiles read a W fragment once for 8.
// W still goes from memory straight into registers (each fragment is read by one
// wave only), X through an LDS ring; both are requested 3 rounds of KB k-blocks
// ahead, one barrier per round: the barrier that publishes round r's X also says
// that every wave is done with round r - 1, whose buffer then takes round r + 3.
//
// Tiles of one column slice and chunk follow each other on one XCD
// (workgroups are dealt round-robin over the 8 XCDs), so its L2 reads the slice of
// W from memory once for all row tiles.
//
// Row-major operands: an operand tile of 16 rows is 64 bytes of each, half a cache
// line, and the loads of a round took twice the line requests of the tiled layouts.
// Over pairs of k-blocks every load takes 8 rows of 128 bytes instead; x goes to LDS
// in swizzled 16-byte pieces, w is put on its lanes by two DPP moves per register
// pair.  x and w row-major, 128 rows: q/k/v 20.4 -> 16.7 us, o 17.4 -> 12.9, gate/up
// 65.2 -> 51, down 46.9 -> 32.1 (tiled 15.6 / 11.9 / 45.8 / 27.1); 512 rows, gate/up
// 177 -> 133.  Three column tiles of row-major w hold two rounds only (four would not
// fit the registers): half as far ahead, but 132.6 instead of 176.0 us there.  With
// tiled w three and four column tiles keep single k-block rounds of W beside pairs of
// X: row-major x then costs nothing (512 rows, down 50.8 us against 51.9 tiled, 61.9
// with half lines; 1024 rows, gate/up 184 against 178 and 223).
//
// 512 rows, q/k/v [6144, 4096], o [4096, 4096], gate/up [24576, 4096] and down
// [4096, 12288], tiled: 35.6 / 23.0 / 103 / 49 us (0.72 / 0.75 / 1.0 / 1.05 PFLOP/s)
// instead of 77.7 / 44.9 / 257 / 132 us in 64-row tiles of gemm_kernel.  At 33 .. 64
// rows (CT = 1) its gain is the deeper X ring and the single barrier per round; use_wide
// has the figures.
// KB: k-blocks of a round of W, RING: rounds of W in registers.  X comes in pairs of
// k-blocks: one a round (KB = 2, RING of them in LDS), or one every other round (KB =
// 1, four in LDS, one barrier per pair).
template <int MT, int CT, int W, bool WT, int KB, int RING>
__global__ __launch_bounds__(64 * W, 2) void gemm_wide_kernel(Args A, int units, int mtiles) {
  constexpr int NC = 2 * MT;              // 1 KB X chunks of a pair
  constexpr int XL = (NC + W - 1) / W;    // chunks a wave requests per pair (those past NC read nothing)
  constexpr int WL = KB * CT;             // W loads of a wave per round
  constexpr int WKB = WT ? 1024 : 64;     // bytes between a lane's consecutive k-blocks of W
  constexpr int XRING = KB == 2 ? RING : 4;
  static_assert((KB == 2 || RING == 4) && (RING - 2) * (XL + WL) < 64 && XL + 2 * WL < 64, "vmcnt range");
  __shared__ __attribute__((aligned(16))) char xs[(XRING * NC + 1) * 1024];   // the last KB takes chunks past NC
  const int lane = __lane_id();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, g4 = lane >> 4;
  // Workgroup id -> (unit = column slice and chunk, row tile): ids equal mod 8 share an XCD.
  const int j = blockIdx.x >> 3;
  const int unit = (blockIdx.x & 7) + 8 * (j / mtiles), mt = j % mtiles;
  if (unit >= units) return;
  const int s = unit % A.S, nt = unit / A.S;
  const int col = 16 * CT * (nt * W + w);       // this wave's first column
  const int row0 = mt * 16 * MT;
  const int k0 = s * A.KC;
  const int nr = A.KC / (32 * KB);              // a multiple of RING (the host checks it)
  const int ncol = min(CT, (A.N - col + 15) / 16);   // column tiles of this wave inside N (may be <= 0)

  // X: lane offset of the wave's chunk jj of a pair, c = w + W jj: of row tile t =
  // c % MT the k-block kb = c / MT (tiled x: one operand tile), or, row-major x, the
  // rows 8 kb .. + 7 over both k-blocks, 128 bytes each, whose 16-byte pieces take
  // XOR-swizzled places so that the fragment reads below hit all banks.  It lands in
  // the (2 t + kb)-th KB of the pair's slot.
  const int mrows = min(16 * MT, A.M - row0);
  const int t0 = row0 / 16;                      // first 16-row tile
  const __amdgpu_buffer_rsrc_t rx =
      A.x_tiled ? rsrc(A.x + (int64_t)(t0 >> 2) * 64 * A.K, (int64_t)(((t0 + MT - 1) >> 2) - (t0 >> 2) + 1) * A.K * 128)
                : rsrc(A.x + (int64_t)row0 * A.sx + k0, 2 * ((int64_t)(mrows - 1) * A.sx + (A.K - k0)));
  const int xkb = A.x_tiled ? 4096 : 64;
  int xo[XL];
#pragma unroll
  for (int jj = 0; jj < XL; ++jj) {
    const int c = w + W * jj, kb = c / MT, t = c % MT;
    int o;
    if (A.x_tiled) {
      const int T = t0 + t;
      o = (((T >> 2) - (t0 >> 2)) * (A.K >> 5) + (k0 >> 5) + kb) * 4096 + (T & 3) * 1024 + 16 * lane;
    } else {
      o = 2 * (16 * t + 8 * kb + (lane >> 3)) * (int)A.sx + 16 * ((lane & 7) ^ (4 * kb + g4));
    }
    xo[jj] = c < NC && 16 * t < mrows ? o : kOOBRow;
  }
  const __amdgpu_buffer_rsrc_t rw =
      WT ? rsrc(A.w + (int64_t)(col / 16) * ((A.K / 32) * 512 + kWSlabPad) + (k0 / 32) * 512,
                ncol > 0 ? (int64_t)(ncol - 1) * (A.K * 32 + 2 * kWSlabPad) + A.KC * 32 : 0)
         : rsrc(A.w + (int64_t)(ncol > 0 ? col : 0) * A.sw + k0,
                ncol > 0 ? 2 * ((int64_t)(16 * ncol - 1) * A.sw + A.KC) : 0);
  // Row-major w, two k-blocks a round: load j takes the rows 8 j .. + 7 over both,
  // 128 bytes each; w_operands puts the pieces on their lanes.
  constexpr bool WL2 = !WT && KB == 2;
  const int woff = WT ? 16 * lane
                   : WL2 ? 2 * (n16 & 7) * (int)A.sw + 16 * (4 * (n16 >> 3) + g4) : 2 * (n16 * (int)A.sw + 8 * g4);
  const int wcol = WT ? A.K * 32 + 2 * kWSlabPad : 32 * (int)A.sw;   // bytes between column tiles

  lds_char_t* xl = (lds_char_t*)xs;
  f32x4 acc[MT][CT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wf[RING][KB][CT];

  auto issue_w = [&](int rr, u32x4 (&wr)[KB][CT]) {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
        wr[kb][c] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                       rw, woff + c * wcol + (WL2 ? 128 * rr + 16 * kb * (int)A.sw : WKB * (KB * rr + kb)), 0, 0));
    asm volatile("" ::: "memory");
  };
  auto issue_x = [&](int pair, int slot) {
#pragma unroll
    for (int jj = 0; jj < XL; ++jj) {
      const int c = w + W * jj;
      x_dma16(rx, xo[jj] + xkb * 2 * pair, xl + (c < NC ? slot * NC + (c % MT) * 2 + c / MT : XRING * NC) * 1024);
    }
    asm volatile("" ::: "memory");
  };
  // Fragment (kb, t): lane (n16, g4) reads row n16, 16-byte piece 4 kb + g4.
  int xr[2];
#pragma unroll
  for (int kb = 0; kb < 2; ++kb)
    xr[kb] = A.x_tiled ? 1024 * kb + 16 * lane : 128 * n16 + 16 * ((4 * kb + g4) ^ (n16 >> 1));
  // Loads j = 0, 1 of row-major w hold, on lane (n16, g4), row 8 j + n16 % 8, piece
  // 4 (n16 / 8) + g4; operand kb takes row n16, piece 4 kb + g4: half of each 16
  // lanes from its own register, half from the other's lane n16 + 8 (mod 16).
  auto w_operands = [&](u32x4& w0, u32x4& w1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int a = (int)w0[i], b = (int)w1[i];
      w0[i] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x128, 0xf, 0xc, false);   // row_ror:8, lanes 8 .. 15
      w1[i] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x128, 0xf, 0x3, false);   // row_ror:8, lanes 0 .. 7
    }
  };
  // The X fragments of a k-block are read two row tiles ahead of their MFMAs.
  auto compute = [&](u32x4 (&wr)[KB][CT], int slot, int kb0) {
    if constexpr (WL2) {
#pragma unroll
      for (int c = 0; c < CT; ++c) w_operands(wr[0][c], wr[KB - 1][c]);
    }
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      u32x4 xf[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xf[t] = *(const __attribute__((address_space(3))) u32x4*)(xl + (slot * NC + 2 * t) * 1024 + xr[kb0 + kb]);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wr[kb][c]),
                                                              __builtin_bit_cast(bf16x8, xf[t]), acc[t][c], 0, 0, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);   // LDS reads
#pragma unroll
    for (int t = 0; t < MT * KB; ++t) {
      __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);   // MFMAs
      if (t + 3 < MT * KB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };
  if constexpr (KB == 2) {
    // Round rr's W into ring slot rr % RING, then its X: with X issued last, a count
    // that covers round rr's X covers its W too.
    auto issue = [&](int rr, int slot) {
      issue_w(rr, wf[slot]);
      issue_x(rr, slot);
    };
    constexpr int PER = XL + WL;   // loads a wave issues per round
#pragma unroll
    for (int r = 0; r < RING - 1; ++r) issue(r, r);
    int r = 0;
    for (; r + RING < nr; r += RING) {
#pragma unroll
      for (int u = 0; u < RING; ++u) {
        vm_wait_n((RING - 2) * PER);   // round r + u has landed (this wave's part)
        raw_barrier();       // every wave's part, and every wave is done with round r + u - 1
        issue(r + u + RING - 1, (u + RING - 1) % RING);
        compute(wf[u], u, 0);
      }
    }
    // The last RING rounds: one more to request.
#pragma unroll
    for (int u = 0; u < RING; ++u) {
      vm_wait_n((RING - 1 - (u > 0 ? u : 1)) * PER);
      raw_barrier();
      if (u == 0) issue(r + RING - 1, RING - 1);
      compute(wf[u], u, 0);
    }
  } else {
    // W three rounds ahead, X two pairs ahead.  Round r waits until what was issued
    // after its W is all that is in flight: rounds r - 2 and r - 1 issued W, the even
    // one of them X before it.  X of pair r / 2 is older than W of round r.
    issue_x(0, 0);
    issue_w(0, wf[0]);
    issue_x(1, 1);
    issue_w(1, wf[1]);
    issue_w(2, wf[2]);
    int r = 0;
    for (; r + 8 < nr; r += 8) {
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        vm_wait_n(XL + 2 * WL);
        if (u % 2 == 0) {
          raw_barrier();   // every wave's part of the pair, and every wave is done with the pair before
          issue_x((r + u) / 2 + 2, (u / 2 + 2) % 4);
        }
        issue_w(r + u + 3, wf[(u + 3) % 4]);
        compute(wf[u % 4], u / 2, u % 2);
      }
    }
    // The last eight rounds request up to their end.
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      vm_wait_n(u < 5 ? XL + 2 * WL : (7 - u) * WL);
      if (u % 2 == 0) {
        raw_barrier();
        if (u + 4 < 8) issue_x((r + u) / 2 + 2, (u / 2 + 2) % 4);
      }
      if (u + 3 < 8) issue_w(r + u + 3, wf[(u + 3) % 4]);
      compute(wf[u % 4], u / 2, u % 2);
    }
  }
#pragma unroll
  for (int c = 0; c < CT; ++c)
    if (c < ncol)
#pragma unroll
      for (int t = 0; t < MT; ++t) store_tile(A, s, row0 + 16 * t + n16, col + 16 * c + 4 * g4, acc[t][c]);
}

#undef RSPX_VMW

// out[m][n] = round(((p0 + p1) + p2) + ...), 4 columns per thread.  Grid:
// x = 256-thread blocks along a row, y = rows from row0 (at most 65535 per
// launch), so no thread divides to find its row.
template <int SC>
__global__ __launch_bounds__(256) void reduce_kernel(const float* part, int S, int M, int N, void* out, int64_t so,
                                                     int out_fp32, int row0) {
  const int n = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= N) return;
  const int m = row0 + blockIdx.y;
  const f32x4 v = sum_parts4<SC>(part + (int64_t)m * N + n, S, (int64_t)M * N);
  if (out_fp32) {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + (int64_t)m * so + n) = v;
  } else {
    u32x2 o;
    o[0] = pack_bf16x2(v[0], v[1]);
    o[1] = pack_bf16x2(v[2], v[3]);
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + (int64_t)m * so + n) = o;
  }
}

// Any shape outside gemm_kernel's (N % 16 != 0 or K % 256 != 0): one chain
// of v_mfma_f32_16x16x32_bf16 over the 32-wide k-blocks of K in increasing k,
// rounded once -- an order fixed by K alone, so a row's bits never depend on
// M.  Workgroup = 64 CT columns (4 waves of CT 16-column tiles) times 16 MT rows.
//
// What bounded it: one k-block at a time from memory into the MFMA registers, a
// memory latency per k-block, and every wave reading all of X by itself.  Now W
// fragments go into a ring of registers 3 rounds of KB k-blocks ahead, and X is
// shared: the waves load a round's fragments 3 rounds ahead, one part each, and
// put them into one of two LDS buffers a round before use.  X passes through
// registers, not direct-to-LDS loads, because a lane's 8 k may start at any 2-byte
// address and end past K.  No load reaches past a row's K elements and none sits
// under a branch (a load under one makes the compiler drain all before it): a
// group that K cuts, or a round past K, loads the row's last 8 elements.  What K
// leaves past its whole rounds is taken once at the end, such a group shifted into
// place with zeros past K, so that it adds exact zeros to the chain.  Rows past M and columns past N read the last row or column;
// their results are not stored.
//
// 77 x 4864 x 896: 21.3 -> 8.0 us (1.1 TB/s of 9.6 MB); 23 x 9976 x 6596, rows not
// 16-byte aligned: 304 -> 39.6 us (3.3 TB/s); 512 x 9976 x 6596: 3.10 -> 0.192 ms
// (350 TFLOP/s); 1024 x 5504 x 4416: 469 -> 118 us (422 TFLOP/s).
struct AnyArgs {
  const uint16_t* x; int64_t sx;  // [M, K]
  const uint16_t* w; int64_t sw;  // [N, K]
  void* out; int64_t so;          // [M, N], bf16 or fp32
  int M, N, K, out_fp32;
};

// The 16 bytes at p, any 2-byte address (one instruction on this target).
__device__ __forceinline__ u32x4 any_load(const uint16_t* p) {
  u32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// Elements k .. k + 7 of a row, zero past K, from v = the 8 elements at min(k, K - 8).
__device__ __forceinline__ u32x4 any_cut(u32x4 v, int k, int K) {
  const int s = max(0, k + 8 - K);   // elements past K
  if (s & 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (v[i] >> 16) | (i < 3 ? v[i + 1 < 4 ? i + 1 : 3] << 16 : 0u);
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t x = 0u;
#pragma unroll
    for (int j = i; j < 4; ++j) x = j - i == s >> 1 ? v[j] : x;
    o[i] = x;
  }
  return o;
}

template <int MT, int CT> constexpr int any_kb() { return CT * MT >= 16 ? 1 : CT == 1 && MT <= 2 ? 4 : 2; }   // k-blocks of a round

template <int MT, int CT, int KB = any_kb<MT, CT>()>
__global__ __launch_bounds__(256, 2) void gemm_any_kernel(AnyArgs A, int units, int mtiles) {
  constexpr int NC = KB * MT;           // 1 KB X fragments of a round
  constexpr int XL = (NC + 3) / 4;      // fragments a wave loads per round
  __shared__ __attribute__((aligned(16))) char xs[2 * XL * 4 * 1024];
  const int lane = __lane_id();
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n16 = lane & 15, g4 = lane >> 4;
  const int j = blockIdx.x >> 3;        // as gemm_wide_kernel: the row tiles of a column slice on one XCD
  const int nt = (blockIdx.x & 7) + 8 * (j / mtiles), mt = j % mtiles;
  if (nt >= units) return;
  const int col = nt * 64 * CT + 16 * CT * w, row0 = mt * 16 * MT;
  const int K = A.K, nkb = (K + 31) >> 5, nr = K / (32 * KB);   // nr: whole rounds

  const uint16_t* wp[CT];
#pragma unroll
  for (int c = 0; c < CT; ++c) wp[c] = A.w + (int64_t)min(col + 16 * c + n16, A.N - 1) * A.sw;
  const uint16_t* xp[XL];
  int xk[XL];                           // k of the lane's fragment jj (w + 4 jj: k-block c / MT, row tile c % MT)
#pragma unroll
  for (int jj = 0; jj < XL; ++jj) {
    const int c = w + 4 * jj;
    xp[jj] = A.x + (int64_t)min(row0 + 16 * (c % MT) + n16, A.M - 1) * A.sx;
    xk[jj] = c < NC ? 32 * (c / MT) + 8 * g4 : 0x40000000;   // past any K: zeros
  }
  lds_char_t* xl = (lds_char_t*)xs;
  typedef __attribute__((address_space(3))) u32x4 lds_u32x4_t;
  f32x4 acc[MT][CT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int c = 0; c < CT; ++c) acc[t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wf[4][KB][CT], xr[2][XL];

  auto load_w = [&](int r, u32x4 (&f)[KB][CT]) {
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int c = 0; c < CT; ++c) f[kb][c] = any_load(wp[c] + min(32 * (KB * r + kb) + 8 * g4, K - 8));
    asm volatile("" ::: "memory");   // the loads stay in this order, so the waits for them are exact
  };
  auto load_x = [&](int r, u32x4 (&f)[XL]) {
#pragma unroll
    for (int jj = 0; jj < XL; ++jj) f[jj] = any_load(xp[jj] + min(32 * KB * r + xk[jj], K - 8));
    asm volatile("" ::: "memory");
  };
  auto put_x = [&](int r, const u32x4 (&f)[XL]) {
#pragma unroll
    for (int jj = 0; jj < XL; ++jj)
      *(lds_u32x4_t*)(xl + ((r & 1) * XL * 4 + w + 4 * jj) * 1024 + 16 * lane) = f[jj];
  };
  auto compute = [&](int r, int n, const u32x4 (&f)[KB][CT]) {   // the round's first n k-blocks
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
      if (kb >= n) break;
      u32x4 xf[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t)
        xf[t] = *(const lds_u32x4_t*)(xl + ((r & 1) * XL * 4 + kb * MT + t) * 1024 + 16 * lane);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int c = 0; c < CT; ++c)
          acc[t][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f[kb][c]),
                                                              __builtin_bit_cast(bf16x8, xf[t]), acc[t][c], 0, 0, 0);
    }
  };
  load_x(0, xr[0]);
  load_w(0, wf[0]);
  load_x(1, xr[1]);
  load_w(1, wf[1]);
  put_x(0, xr[0]);
  load_x(2, xr[0]);
  load_w(2, wf[2]);
  int r0 = 0;
  for (; r0 + 4 <= nr; r0 += 4) {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int r = r0 + u;
      raw_barrier();   // round r's X is in LDS; every wave is done with round r - 1's buffer
      put_x(r + 1, xr[(u + 1) & 1]);
      load_x(r + 3, xr[(u + 1) & 1]);
      load_w(r + 3, wf[(u + 3) & 3]);
      compute(r, KB, wf[u]);
    }
  }
  // Up to three more whole rounds, already requested (a way out of the middle of
  // the loop would blur its waits).
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    if (r0 + u >= nr) break;
    raw_barrier();
    put_x(r0 + u + 1, xr[(u + 1) & 1]);
    compute(r0 + u, KB, wf[u]);
  }
  if (KB * nr < nkb) {
    // What is left of K, less than a round.
    load_x(nr, xr[0]);
    load_w(nr, wf[0]);
#pragma unroll
    for (int jj = 0; jj < XL; ++jj) xr[0][jj] = any_cut(xr[0][jj], 32 * KB * nr + xk[jj], K);
    raw_barrier();   // every wave is done with the buffer
    put_x(nr, xr[0]);
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int c = 0; c < CT; ++c) wf[0][kb][c] = any_cut(wf[0][kb][c], 32 * (KB * nr + kb) + 8 * g4, K);
    raw_barrier();
    compute(nr, nkb - KB * nr, wf[0]);
  }
  // acc[t][c][e] = D[column 16 c + 4 g4 + e][row 16 t + n16] of the wave's tiles.
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = row0 + 16 * t + n16;
    if (m >= A.M) continue;
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = col + 16 * c + 4 * g4 + e;
        if (n >= A.N) continue;
        if (A.out_fp32)
          static_cast<float*>(A.out)[(int64_t)m * A.so + n] = acc[t][c][e];
        else
          static_cast<uint16_t*>(A.out)[(int64_t)m * A.so + n] = f32_to_bf16_rne(acc[t][c][e]);
      }
  }
}

// Short K (8 .. 32 U): nothing to pipeline, so each wave loads its W fragments and all X
// fragments at once, straight into the MFMA registers: one memory round trip, no LDS, no
// barriers.  Workgroup = 64 columns (4 waves of 16) times 16 MT rows; the same chain.
template <int MT, int U>
__global__ __launch_bounds__(256) void gemm_short_kernel(AnyArgs A) {
  const int lane = __lane_id(), wv = threadIdx.x >> 6;
  const int n16 = lane & 15, g4 = lane >> 4;
  const int n0 = blockIdx.x * 64 + wv * 16, m0 = blockIdx.y * 16 * MT, K = A.K;
  if (n0 >= A.N) return;   // whole wave; no barriers below
  const uint16_t* wp = A.w + (int64_t)min(n0 + n16, A.N - 1) * A.sw;
  const uint16_t* xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = A.x + (int64_t)min(m0 + 16 * t + n16, A.M - 1) * A.sx;
  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  u32x4 wf[U], xf[U][MT];
#pragma unroll
  for (int kb = 0; kb < U; ++kb) {
    const int k = min(32 * kb + 8 * g4, K - 8);
    wf[kb] = any_load(wp + k);
#pragma unroll
    for (int t = 0; t < MT; ++t) xf[kb][t] = any_load(xp[t] + k);
  }
#pragma unroll
  for (int kb = 0; kb < U; ++kb) {
    const int k = 32 * kb;
    if (k >= K) break;
    if (k + 32 > K) {
      wf[kb] = any_cut(wf[kb], k + 8 * g4, K);
#pragma unroll
      for (int t = 0; t < MT; ++t) xf[kb][t] = any_cut(xf[kb][t], k + 8 * g4, K);
    }
#pragma unroll
    for (int t = 0; t < MT; ++t)
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf[kb]),
                                                       __builtin_bit_cast(bf16x8, xf[kb][t]), acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int m = m0 + 16 * t + n16;
    if (m >= A.M) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = n0 + 4 * g4 + e;
      if (n >= A.N) continue;
      if (A.out_fp32)
        static_cast<float*>(A.out)[(int64_t)m * A.so + n] = acc[t][e];
      else
        static_cast<uint16_t*>(A.out)[(int64_t)m * A.so + n] = f32_to_bf16_rne(acc[t][e]);
    }
  }
}

// K < 8: no row holds a 16-byte group.  One 16 x 16 tile per wave, its elements
// loaded one by one into the single k-block of the chain.  Grid: x = column tiles, y =
// row tiles from row0 on (at most 65535 per launch): tiles counted along x alone would
// reach the 2^32 threads that a grid dimension may have at 2^34 outputs.
__global__ __launch_bounds__(64) void gemm_small_k_kernel(AnyArgs A, int row0) {
  const int lane = __lane_id(), n16 = lane & 15, g4 = lane >> 4;
  const int n0 = 16 * (int)blockIdx.x;
  const int64_t m0 = row0 + 16 * (int64_t)blockIdx.y;
  u32x4 wf = {0u, 0u, 0u, 0u}, xf = wf;
  if (g4 == 0) {
#pragma unroll
    for (int j = 0; j < 7; ++j) {
      if (j >= A.K) break;
      if (n0 + n16 < A.N) wf[j / 2] |= (uint32_t)A.w[(int64_t)(n0 + n16) * A.sw + j] << (16 * (j & 1));
      if (m0 + n16 < A.M) xf[j / 2] |= (uint32_t)A.x[(m0 + n16) * A.sx + j] << (16 * (j & 1));
    }
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wf), __builtin_bit_cast(bf16x8, xf), acc, 0, 0,
                                                0);
  const int64_t m = m0 + n16;
  if (m >= A.M) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int n = n0 + 4 * g4 + e;
    if (n >= A.N) continue;
    if (A.out_fp32) static_cast<float*>(A.out)[m * A.so + n] = acc[e];
    else static_cast<uint16_t*>(A.out)[m * A.so + n] = f32_to_bf16_rne(acc[e]);
  }
}

}  // namespace gemm

// Chunk count of the K reduction: a function of (N, K) only.  More chunks
// until the grid has >= 256 workgroups per 64-row tile, at most 8, each chunk
// a whole number of 256-wide rounds.
static int linear_splits(int N, int K) {
  const int nt = (N + gemm::kSplitCols - 1) / gemm::kSplitCols;
  int S = 1;
  while (nt * S < 256 && S < 8 && K % (gemm::kRoundK * 2 * S) == 0) S *= 2;
  return S;
}

// W [N, K] (row stride sw) into the tiled layout: one thread per 16 bytes of
// the output, the slab pads written as zeros.
__global__ __launch_bounds__(256) void tile_weight_kernel(const uint16_t* w, int64_t sw, int N, int K,
                                                         uint16_t* out) {
  const int64_t slab = (int64_t)K * 16 + gemm::kWSlabPad;   // elements per slab
  const int64_t per = slab / 8;                              // 16-byte units per slab
  const int64_t u = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (u >= (int64_t)(N / 16) * per) return;
  const int s = (int)(u / per);
  const int64_t j = u - s * per;                             // unit inside the slab
  u32x4 v = {0u, 0u, 0u, 0u};
  if (j < (int64_t)K * 2) {
    const int t = (int)(j >> 6), lane = (int)(j & 63);
    const int n = 16 * s + (lane & 15), k = 32 * t + 8 * (lane >> 4);
    v = *reinterpret_cast<const u32x4*>(w + (int64_t)n * sw + k);
  }
  *reinterpret_cast<u32x4*>(out + u * 8) = v;
}

}  // namespace rspx

using namespace rspx;

extern "C" int64_t rspx_linear_tiled_weight_elems(int N, int K) {
  if (N <= 0 || K <= 0 || N % 16 != 0 || K % 32 != 0) return -1;
  return (int64_t)(N / 16) * ((int64_t)K * 16 + gemm::kWSlabPad);
}

extern "C" int rspx_linear_tile_weight(const void* w, int64_t sw, int N, int K, void* out, void* stream) {
  if (N <= 0 || K <= 0 || !w || !out || sw < K) return RSPX_EINVAL;
  if (N % 16 != 0 || K % 32 != 0) return RSPX_EUNSUPPORTED;
  if ((reinterpret_cast<uintptr_t>(w) & 15u) || (reinterpret_cast<uintptr_t>(out) & 15u) || sw % 8)
    return RSPX_EALIGN;
  const int64_t units = rspx_linear_tiled_weight_elems(N, K) / 8;
  if ((units + 255) / 256 > 0x7fffffff) return RSPX_EUNSUPPORTED;
  hipLaunchKernelGGL(tile_weight_kernel, dim3((unsigned)((units + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(w), sw, N, K,
                     static_cast<uint16_t*>(out));
  return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
}

// Shapes gemm_kernel takes; every other (N, K) runs gemm_any_kernel (one
// K chain).  The choice depends on (N, K) only.
static bool linear_fast_shape(int N, int K) { return N % 16 == 0 && K % gemm::kRoundK == 0; }

extern "C" int rspx_linear_splits(int N, int K) {
  if (N <= 0 || K <= 0) return -1;
  return linear_fast_shape(N, K) ? linear_splits(N, K) : 1;
}

extern "C" int64_t rspx_linear_workspace_bytes(int M, int N, int K) {
  if (M < 0 || N <= 0 || K <= 0) return -1;
  const int S = rspx_linear_splits(N, K);
  return S > 1 ? (int64_t)S * M * N * (int64_t)sizeof(float) : 0;
}

namespace rspx {
// The chunk sums of a split product that no consumer takes, and the launch status.
static int reduce_launch(const gemm::Args& a, hipStream_t s) {
  if (a.S > 1 && !a.to_part) {
    const unsigned bx = (unsigned)((a.N / 4 + 255) / 256);
    for (int row0 = 0; row0 < a.M; row0 += 65535) {
      const dim3 rg(bx, (unsigned)min(a.M - row0, 65535));
      RSPX_WITH_SPLITS(a.S, SC,
                       hipLaunchKernelGGL((gemm::reduce_kernel<SC>), rg, dim3(256), 0, s, a.part, a.S, a.M, a.N, a.out,
                                          a.so, a.out_fp32, row0));
    }
  }
  return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
}

// Waves of a workgroup and 16-column tiles per wave, for gemm_wide_kernel and
// gemm_any_kernel: the least time for the busiest CU, workgroups per CU times a
// workgroup's time (tiles: row tiles times K chunks).  Narrower waves read each X
// fragment for fewer MFMAs, so 1 .. 4 column tiles cost 14 : 24 : 31 : 40 and not
// 1 : 2 : 3 : 4 (512 rows, o projection [4096, 4096]: 33.1 / 27.5 / 32.6 / 23.0 us
// at 1 .. 4 with 4 / 2 / 2 / 1 workgroups per CU; 512 rows, gate/up [24576, 4096]:
// 144.8 / 115.8 / 103.3 / 116.7 us with 6 / 3 / 2 / 2; 128 rows, q/k/v [6144, 4096]:
// 20.1 / 16.5 / 19.3 / 22.2 us with 2 / 1 / 1 / 1; 512 rows, [9976, 6596]: 216 / 259
// / - / 192 us with 3 / 2 / - / 1).  Six waves of one tile (96 columns, 22) fill the
// chip with one workgroup per CU where 64 columns take two and 128 leave CUs idle:
// gate/up at 64 rows 37.2 us instead of 47.0 (4 x 1) and 40.2 (4 x 2), at 128 rows 45.6
// instead of 61.0 and 50.3.
//
// Row-major w costs more the more column tiles a wave has (4 do not fit its two
// k-blocks a round, and two workgroups per CU hide its shallower ring), so there the
// costs are 15 : 24 : 36 and 21 for six waves, a lone workgroup 1.2 of its share (512
// rows, gate/up: 132.6 us at 4 x 3, 138.1 at 4 x 2, 153.4 at 6 x 1; 256 rows: 102.0 /
// 94.9 / 84.6; 512 rows, o: 40.4 / 30.9 / 38.4, 36.1 at 4 x 1, 33.6 at 4 x 4).
struct WaveTile { int waves, ct; };
enum class TileFor { kTiledW, kRowsW, kAny };
static WaveTile wave_tile(int N, int64_t tiles, TileFor use) {
  static const struct { WaveTile t; int cost, cost_rows; } kTiles[] = {
      {{4, 4}, 40, 0}, {{4, 3}, 31, 36}, {{4, 2}, 24, 24}, {{6, 1}, 22, 21}, {{4, 1}, 14, 15}};
  WaveTile best{4, 1};
  int64_t t_best = -1;
  for (const auto& c : kTiles) {
    if (use == TileFor::kAny ? c.t.ct == 3 || c.t.waves == 6 : use == TileFor::kRowsW && c.t.ct == 4) continue;
    const int cols = 16 * c.t.waves * c.t.ct;
    const int64_t n = ((int64_t)((N + cols - 1) / cols) * tiles + 255) / 256;   // workgroups of the busiest CU
    const int64_t t = use == TileFor::kRowsW ? (n > 1 ? 5 * n : 6) * c.cost_rows : n * c.cost;
    if (t_best < 0 || t < t_best) { best = c.t; t_best = t; }
  }
  return best;
}

// 31-bit byte offsets inside a 128-row tile of x and a wave's 64 rows of w.
static bool wide_fits(const gemm::Args& a) {
  return (a.x_tiled || (int64_t)128 * a.sx * 2 < (1ll << 30)) && (a.sw == kTiled || (int64_t)64 * a.sw * 2 < (1ll << 30)) &&
         (int64_t)a.K * 384 < (1ll << 30);
}

// Whether gemm_wide_kernel runs the call.  Always above 64 rows, except that tiled
// operands whose chunk is one round of gemm_kernel stay there while neither grid is
// large ([4096, 1024]: 96 rows 5.3 us against 5.6, 128 rows 5.8 / 6.4; [576, 512],
// 1024 rows 4.8 / 5.5; but [6144, 1024], 96 rows 8.7 / 7.5), or are split with at most
// one workgroup per CU ([1024, 1024], 836 rows: 13.9 / 16.4; [6912, 512], 235 rows: 14.5 /
// 15.9; with two [3840, 1024], 613 rows: 25.1 / 24.1).  For 33 .. 64 rows where waves of one
// column tile make one workgroup for most CUs and its chunk has eight rounds or more:
// q/k/v [6144, 4096], o [4096, 4096], gate/up [24576, 4096] and down [4096, 12288], tiled,
// at 64 rows 12.3 / 9.1 / 37.2 / 20.7 us instead of 13.7 / 10.3 / 39.7 / 23.3 in
// gemm_kernel, at 48 rows 11.7 / 8.6 / 36.1 / 19.6 instead of 12.1 / 9.6 / 36.9 / 21.8, at
// 32 rows 11.4 / 8.3 / 35.7 / 19.0 and 11.2 / 8.5 / 36.1 / 19.3; row-major at 64 rows 13.1 /
// 9.8 / 44.5 / 25.4 instead of 16.3 / 11.7 / 47.6 / 28.1.  Tiled x with row-major w is the
// slower one there (gate/up, 48 rows: 43.6 / 40.6).  Below 208 workgroups tiled operands
// gain or lose up to a quarter with no rule in the sizes ([9184, 8704], 35 rows 43.7 / 35.3;
// [12544, 2304], 55 rows 15.2 / 17.1), mostly gain.  gemm_kernel keeps more bytes of W in
// flight per wave, which counts in short chunks and small grids ([4096, 1024], 64 rows: 5.1
// against 5.3; [1024, 3072], 64 workgroups, 48 rows: 5.9 / 6.1), and shares X between 128
// columns in large ones (vocabulary [151936, 4096]: 239 / 252).
static bool use_wide(const gemm::Args& a, WaveTile t) {
  if (!wide_fits(a) || a.M <= 32) return false;
  const bool w_tiled = a.sw == kTiled;
  const int cols = 16 * t.waves;
  const int64_t wgs = (int64_t)((a.N + cols - 1) / cols) * a.S;   // of one row tile
  if (a.M > gemm::kRows) {
    if (a.KC != gemm::kRoundK || !a.x_tiled || !w_tiled) return true;
    if (a.S > 1) return (int64_t)((a.N + cols * t.ct - 1) / (cols * t.ct)) * a.S * ((a.M + 127) / 128) > 256;
    return !(t.ct == 1 && t.waves == 4 && wgs * ((a.M + gemm::kRows - 1) / gemm::kRows) <= 512);
  }
  return t.ct == 1 && a.KC >= 512 && wgs > 128 && wgs <= 256 && (w_tiled || !a.x_tiled);
}

static int wide_launch(const gemm::Args& a, WaveTile wt, int mtiles, hipStream_t s) {
  const int cols = 16 * wt.waves * wt.ct;
  const int64_t units = (int64_t)((a.N + cols - 1) / cols) * a.S;
  // Lower row tiles while the grid stays within one workgroup per CU ([1024, 3072],
  // tiled / row-major, 128 rows: 7.0 / 11.7 us in one tile, 4.7 / 6.1 in four).
  // Units are dealt over the 8 XCDs of 32 CUs, so the XCD with the most of them counts
  // (374 rows of [1280, 3840], row-major, 20 units: in 12 tiles, 36 workgroups on four XCDs,
  // 33.1 us; in 10 20.1; 64-row tiles of gemm_kernel 29.5).
  if (wt.ct == 1 && units < 256) mtiles = max(mtiles, min((int)(32 / ((units + 7) / 8)), (a.M + 31) / 32));
  const int mt = ((a.M + mtiles - 1) / mtiles + 15) / 16;
  mtiles = (a.M + 16 * mt - 1) / (16 * mt);
  const int64_t wgs = (units + 7) / 8 * 8 * mtiles;
  if (wgs > 0x7fffffff) return RSPX_EUNSUPPORTED;
  const dim3 g((unsigned)wgs), b(64 * wt.waves);
  const bool w_tiled = a.sw == kTiled;
#define RSPX_WIDE(MTV, CTV, WV, WTV, KBV, RV) \
  hipLaunchKernelGGL((gemm::gemm_wide_kernel<MTV, CTV, WV, WTV, KBV, RV>), g, b, 0, s, a, (int)units, mtiles)
#define RSPX_WIDE_12(MTV, CTV, WV)                  \
  if (w_tiled) RSPX_WIDE(MTV, CTV, WV, true, 2, 4); \
  else RSPX_WIDE(MTV, CTV, WV, false, 2, 4);
#define RSPX_WIDE_1(MTV)                                 \
  if (wt.waves == 6) { RSPX_WIDE_12(MTV, 1, 6) }         \
  else { RSPX_WIDE_12(MTV, 1, 4) }
#define RSPX_WIDE_CT(MTV)                                                      \
  if (wt.ct == 4) RSPX_WIDE(MTV, 4, 4, true, 1, 4);   /* tiled w only */       \
  else if (wt.ct == 3) {                                                       \
    if (!w_tiled) RSPX_WIDE(MTV, 3, 4, false, 2, 2);                           \
    else RSPX_WIDE(MTV, 3, 4, true, 1, 4);                                     \
  } else if (wt.ct == 2) { RSPX_WIDE_12(MTV, 2, 4) }                           \
  else { RSPX_WIDE_1(MTV) }
  switch (mt) {
    case 8: RSPX_WIDE_CT(8) break;
    case 7: RSPX_WIDE_CT(7) break;
    case 6: RSPX_WIDE_CT(6) break;
    case 5: RSPX_WIDE_CT(5) break;
    case 4: RSPX_WIDE_1(4) break;   // one-tile waves: use_wide's rule, or lower row tiles
    case 3: RSPX_WIDE_1(3) break;
    default: RSPX_WIDE_1(2) break;
  }
#undef RSPX_WIDE_CT
#undef RSPX_WIDE_1
#undef RSPX_WIDE_12
#undef RSPX_WIDE
  return reduce_launch(a, s);
}

static int linear_launch(const void* x, int64_t sx, const void* w, int64_t sw, void* out, int64_t so, int M, int N,
                         int K, int out_fp32, float* part, int to_part, hipStream_t s, int silu = 0) {
  const int S = linear_splits(N, K);
  gemm::Args a;
  a.x = static_cast<const uint16_t*>(x); a.sx = sx;
  a.w = static_cast<const uint16_t*>(w); a.sw = sw;
  a.out = out; a.so = so;
  a.part = part;
  a.M = M; a.N = N; a.K = K; a.S = S; a.KC = K / S; a.out_fp32 = out_fp32 ? 1 : 0; a.to_part = to_part;
  a.silu = silu;
  a.x_tiled = sx == kTiled;
  a.out_tiled = silu && so == kTiled;
  const int MTILES = (M + gemm::kRows - 1) / gemm::kRows;
  if (MTILES > 65535) return RSPX_EUNSUPPORTED;
  // gemm_wide_kernel: row tiles of at most 128 rows, all of the same height.
  const int mtiles = (M + 127) / 128;
  const WaveTile wt = wave_tile(N, (int64_t)S * mtiles, sw == kTiled ? TileFor::kTiledW : TileFor::kRowsW);
  if (use_wide(a, wt)) return wide_launch(a, wt, mtiles, s);
  // 8 waves (128 columns) share each X round between twice the columns; worth
  // it while the grid keeps >= 192 workgroups, and for the widest layers
  // (the vocabulary head) only when the X block is large (many rows).
  const int wg8 = (N + 127) / 128 * S;
  // An 8-wave grid that leaves CUs idle: 6 waves (96 columns) fill them
  // (gate/up [64 x 4096] . [24576 x 4096]^T: 192 -> 256 workgroups, 47.7 ->
  // 42.2 us, one row 38.9 -> 34.8 us; q/k/v [6144 x 4096], 4 K chunks: 15.4 ->
  // 14.8 us with X resident).  The vocabulary head gained nothing from it.
  const int wg6 = (N + 95) / 96 * S;
  const int waves = (N % 96 == 0 && wg8 < 256 && wg6 >= 256 && wg6 <= 512) ? 6
                    : (wg8 >= 192 && (M >= 32 || wg8 < 1024)) ? 8 : 4;
  const int NT = (N + 16 * waves - 1) / (16 * waves);
  const int mt = (MTILES > 1 || M >= 64) ? 4 : (M + 15) / 16;  // row tiles per 64-row tile
  // X-resident blocks pay where X is large against each block's W slice and
  // the grid is one wave of 6- or 8-wave blocks (q/k/v [64 x 4096] .
  // [6144 x 4096]^T: 17.5 -> 16.7 us at 8 waves); for 4-wave blocks and for
  // one row they cost a little.
  const bool xres = waves >= 6 && M >= 32;
  const int nr = a.KC / gemm::kRoundK;
  const dim3 g((unsigned)NT, (unsigned)S, (unsigned)MTILES), b(64 * waves);
#define RSPX_GEMM_NR(MTV, WV, WTV)                                                                       \
  switch (nr) {                                                                                          \
    case 1: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 1, WV, false, WTV>), g, b, 0, s, a); break;       \
    case 2: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 2, WV, false, WTV>), g, b, 0, s, a); break;       \
    case 3: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 3, WV, false, WTV>), g, b, 0, s, a); break;       \
    case 4:                                                                                              \
      if (xres) hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 4, WV, true, WTV>), g, b, 0, s, a);           \
      else hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 4, WV, false, WTV>), g, b, 0, s, a);               \
      break;                                                                                             \
    case 6: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 6, WV, false, WTV>), g, b, 0, s, a); break;       \
    case 8: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 8, WV, false, WTV>), g, b, 0, s, a); break;       \
    case 12: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 12, WV, false, WTV>), g, b, 0, s, a); break;     \
    case 16: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 16, WV, false, WTV>), g, b, 0, s, a); break;     \
    default: hipLaunchKernelGGL((gemm::gemm_kernel<MTV, 0, WV, false, WTV>), g, b, 0, s, a); break;      \
  }
#define RSPX_GEMM_MT(WV, WTV)                                                                            \
  if (mt == 4) { RSPX_GEMM_NR(4, WV, WTV) }                                                              \
  else if (mt == 3) { RSPX_GEMM_NR(3, WV, WTV) }                                                         \
  else if (mt == 2) { RSPX_GEMM_NR(2, WV, WTV) }                                                         \
  else { RSPX_GEMM_NR(1, WV, WTV) }
#define RSPX_GEMM_W(WV)                                                                                  \
  if (sw == kTiled) { RSPX_GEMM_MT(WV, true) }                                                           \
  else { RSPX_GEMM_MT(WV, false) }
  if (waves == 6) { RSPX_GEMM_W(6) }
  else if (waves == 8) { RSPX_GEMM_W(8) }
  else { RSPX_GEMM_W(4) }
#undef RSPX_GEMM_W
#undef RSPX_GEMM_MT
#undef RSPX_GEMM_NR
  return reduce_launch(a, s);
}

static int linear_check(const void* x, int64_t sx, const void* w, int64_t sw, int M, int N, int K) {
  if (M < 0 || N <= 0 || K <= 0) return RSPX_EINVAL;
  if (N % 16 != 0 || K % gemm::kRoundK != 0) return RSPX_EUNSUPPORTED;
  if (M == 0) return RSPX_OK;
  if (!x || !w) return RSPX_EINVAL;
  const bool xt = sx == kTiled, wt = sw == kTiled;
  if ((!xt && sx < K) || (!wt && sw < K)) return RSPX_EINVAL;
  auto al = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  if (!al(x) || !al(w) || (!xt && sx % 8) || (!wt && sw % 8)) return RSPX_EALIGN;
  if ((!xt && (int64_t)64 * sx * 2 >= (1ll << 31)) || (!wt && (int64_t)16 * sw * 2 >= (1ll << 31)) ||
      (int64_t)K * 128 >= (1ll << 30))
    return RSPX_EUNSUPPORTED;
  return RSPX_OK;
}
}  // namespace rspx

// Any (N, K): row-major x and w with rows of at least K elements (2-byte
// aligned, any stride below 2^24 elements), out [M, N] with row stride so.
static int linear_any(const void* x, int64_t sx, const void* w, int64_t sw, void* out, int64_t so, int M, int N,
                      int K, int out_fp32, hipStream_t s) {
  if (M < 0 || N <= 0 || K <= 0) return RSPX_EINVAL;
  if (M == 0) return RSPX_OK;
  if (!x || !w || !out) return RSPX_EINVAL;
  if (sx == kTiled || sw == kTiled) return RSPX_EUNSUPPORTED;  // the tiled layouts need N % 16, K % 32
  if (sx < K || sw < K || so < N) return RSPX_EINVAL;
  auto al = [](const void* p, unsigned a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
  if (!al(x, 2) || !al(w, 2) || !al(out, out_fp32 ? 4 : 2)) return RSPX_EALIGN;
  // Rows are addressed with 64-bit pointers.  What these limits bound is K (a row is at least
  // K elements: K < 2^24), so that the kernels' int offsets inside a row, three rounds past K
  // and beside the 0x40000000 that stands for no fragment, stay below 2^31; the M limit, that
  // row numbers do.
  if (((int64_t)gemm::kRows * sx + K) * 2 >= (1ll << 31) - 64 || ((int64_t)16 * sw + K) * 2 >= (1ll << 31) - 64)
    return RSPX_EUNSUPPORTED;
  if ((M + gemm::kRows - 1) / gemm::kRows > 65535) return RSPX_EUNSUPPORTED;
  gemm::AnyArgs a{static_cast<const uint16_t*>(x), sx, static_cast<const uint16_t*>(w), sw, out, so, M, N, K,
                  out_fp32 ? 1 : 0};
  if (K < 8) {
    constexpr int kRowsPerLaunch = 16 * 65535;
    for (int row0 = 0; row0 < M; row0 += kRowsPerLaunch) {
      const dim3 g((unsigned)((N + 15) / 16), (unsigned)((min(M - row0, kRowsPerLaunch) + 15) / 16));
      hipLaunchKernelGGL(gemm::gemm_small_k_kernel, g, dim3(64), 0, s, a, row0);
    }
    return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
  }
  // Short K: gemm_short_kernel, in row tiles as high as leave a workgroup to every CU.
  // gemm_any_kernel spends a barrier and an LDS pass on a chain of one or two memory round
  // trips (1 x 64 x 64: 3.81 us against 1.93; 760 x 6496 x 8: 20.8 / 14.5; 10 x 96 x 128:
  // 3.20 / 2.43; 1 x 64 x 192: 3.87 / 2.78).  Above 128 it wins with more than two row tiles,
  // which it reads once for four waves (82 x 8256 x 192: 6.9 / 11.4; 279 x 3296 x 192: 7.3 /
  // 11.7); from 65 to 128 with more than two it is up to 15 % ahead or behind.
  const int nt = (N + 63) / 64;
  int ms = min((M + 15) / 16, 4);
  while (ms > 1 && (int64_t)nt * ((M + 16 * ms - 17) / (16 * ms - 16)) <= 256) --ms;
  if (K <= 128 || (K <= 256 && ms <= 2)) {
    const dim3 g((unsigned)nt, (unsigned)((M + 16 * ms - 1) / (16 * ms)));
    const int u = (K + 31) / 32;   // k-blocks
#define RSPX_SHORT(MTV, UV) hipLaunchKernelGGL((gemm::gemm_short_kernel<MTV, UV>), g, dim3(256), 0, s, a)
#define RSPX_SHORT_U(MTV)           \
  if (u <= 1) RSPX_SHORT(MTV, 1);      \
  else if (u <= 2) RSPX_SHORT(MTV, 2); \
  else if (u <= 4) RSPX_SHORT(MTV, 4); \
  else RSPX_SHORT(MTV <= 2 ? MTV : 2, 8);
    if (ms == 1) { RSPX_SHORT_U(1) }
    else if (ms == 2) { RSPX_SHORT_U(2) }
    else if (ms == 3) { RSPX_SHORT_U(3) }
    else { RSPX_SHORT_U(4) }
#undef RSPX_SHORT
#undef RSPX_SHORT_U
    return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
  }
  // Row tiles of 1, 2, 4, 6 or 8 16-row tiles and 1, 2 or 4 column tiles a wave
  // (wave_tile); where that leaves CUs without a workgroup, lower row tiles
  // while the grid stays within one workgroup per CU (77 x 4864 x 896: 12.1 -> 8.0
  // us, 64 x 5000 x 2600: 25.9 -> 18.3; up to two per CU: 10.7, 26.6).
  const int mtiles = (M + 127) / 128, rows = (M + mtiles - 1) / mtiles;
  const int ct = wave_tile(N, mtiles, TileFor::kAny).ct;
  const int64_t units = (N + 64 * ct - 1) / (64 * ct);
  int mt = rows <= 16 ? 1 : rows <= 32 ? 2 : rows <= 64 ? 4 : rows <= 96 ? 6 : 8;
  auto row_tiles = [&](int t) { return (M + 16 * t - 1) / (16 * t); };
  while (ct == 1 && mt > 1 && units * row_tiles(mt == 6 ? 4 : mt / 2) <= 256) mt = mt == 6 ? 4 : mt / 2;
  const int64_t mtl = row_tiles(mt);
  const int64_t wgs = (units + 7) / 8 * 8 * mtl;
  if (wgs > 0x7fffffff) return RSPX_EUNSUPPORTED;
  const dim3 g((unsigned)wgs), b(256);
#define RSPX_ANY(MTV, CTV) \
  hipLaunchKernelGGL((gemm::gemm_any_kernel<MTV, CTV>), g, b, 0, s, a, (int)units, (int)mtl);
#define RSPX_ANY_MT(CTV)                                \
  if (mt == 1) { RSPX_ANY(1, CTV) }                     \
  else if (mt == 2) { RSPX_ANY(2, CTV) }                \
  else if (mt == 4) { RSPX_ANY(4, CTV) }                \
  else if (mt == 6) { RSPX_ANY(6, CTV) }                \
  else { RSPX_ANY(8, CTV) }
  // One and two row tiles of one column tile take rounds of four k-blocks; of two where
  // those come out even and the K is short, since what K leaves to the end is a memory round
  // trip of its own (2 x 448 x 576: 5.93 us with four, 4.58 with two).
  const bool halves = K % 128 == 64 && K <= 640;
  if (ct == 1 && mt <= 2 && halves) {
    if (mt == 1) hipLaunchKernelGGL((gemm::gemm_any_kernel<1, 1, 2>), g, b, 0, s, a, (int)units, (int)mtl);
    else hipLaunchKernelGGL((gemm::gemm_any_kernel<2, 1, 2>), g, b, 0, s, a, (int)units, (int)mtl);
  } else if (ct == 1) { RSPX_ANY_MT(1) }
  else if (ct == 2) { RSPX_ANY_MT(2) }
  else { RSPX_ANY_MT(4) }
#undef RSPX_ANY
#undef RSPX_ANY_MT
  return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
}

extern "C" int rspx_linear(const void* x, int64_t sx, const void* w, int64_t sw, void* out, int64_t so, int M, int N,
                           int K, int out_fp32, void* workspace, int64_t workspace_bytes, void* stream) {
  if (N > 0 && K > 0 && !linear_fast_shape(N, K))
    return linear_any(x, sx, w, sw, out, so, M, N, K, out_fp32, static_cast<hipStream_t>(stream));
  int rc = linear_check(x, sx, w, sw, M, N, K);
  if (rc != RSPX_OK || M == 0) return rc;
  if (!out) return RSPX_EINVAL;
  if (so < N) return RSPX_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out) & 15u) || so % 4) return RSPX_EALIGN;
  const int S = linear_splits(N, K);
  const int64_t need = S > 1 ? (int64_t)S * M * N * (int64_t)sizeof(float) : 0;
  if (need > 0 && (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 15u)))
    return RSPX_EWORKSPACE;
  return linear_launch(x, sx, w, sw, out, so, M, N, K, out_fp32, static_cast<float*>(workspace), 0,
                       static_cast<hipStream_t>(stream));
}

extern "C" int rspx_linear_silu(const void* x, int64_t sx, const void* w, int64_t sw, void* out, int64_t so, int M,
                                int N, int K, void* stream) {
  int rc = linear_check(x, sx, w, sw, M, N, K);
  if (rc != RSPX_OK || M == 0) return rc;
  const bool ot = so == kTiled;
  if (!out || N % 32 != 0 || (!ot && so < N / 2) || (ot && (N / 2) % 32 != 0)) return RSPX_EINVAL;
  if ((reinterpret_cast<uintptr_t>(out) & 15u) || (!ot && so % 8)) return RSPX_EALIGN;
  if (linear_splits(N, K) != 1) return RSPX_EUNSUPPORTED;
  return linear_launch(x, sx, w, sw, out, so, M, N, K, 0, nullptr, 0, static_cast<hipStream_t>(stream), 1);
}

extern "C" int rspx_linear_partials(const void* x, int64_t sx, const void* w, int64_t sw, float* part, int M, int N,
                                    int K, void* stream) {
  int rc = linear_check(x, sx, w, sw, M, N, K);
  if (rc != RSPX_OK || M == 0) return rc;
  if (!part || (reinterpret_cast<uintptr_t>(part) & 15u)) return RSPX_EINVAL;
  return linear_launch(x, sx, w, sw, nullptr, N, M, N, K, 1, part, 1, static_cast<hipStream_t>(stream));
}
