// SwiGLU for gfx950: y = bf16(bf16(silu(g)) * u), silu(g) = g / (1 + exp(-g)).
//
// Replaces silu_mul of respect/system/fused.py:106-123 (and the stock
// act_fn(gate) * up of the HF MLP): silu is computed in fp32 and rounded to
// bf16, then multiplied by u in fp32 and rounded again -- the rounding points
// of PyTorch's bf16 F.silu(g) * u.  No reduction: each element depends on its
// own g and u only, so rows never influence each other.
//
// Two bf16 per thread (4-byte loads of g and u, one 4-byte store), four from kWide and
// eight from kWider elements on, where cols, the strides and the pointers allow it, else
// one (the same values).  Grid: x = blocks along a row, y = rows (one launch per 65535
// rows), so a thread finds its row and column without a division.  Stores are
// non-temporal: not kept in L2, they shorten the write-back at the kernel's end.  What
// bounds it: one memory round trip in small calls, where more elements per thread only
// lengthen the chain and leave fewer wavefronts ([64, 2 x 12288] 3.02 / 3.19 / 3.47 us with
// 2 / 4 / 8 elements, [16, 2 x 3072] 2.10 / 2.15 / 2.33, [1, 2 x 4096] 2.06 / 2.08 / 2.15);
// and bandwidth in large ones, where four bytes per load kept too little in flight
// ([3072, 2 x 12288] 56.2 us with 2, 40.6 with 4 (5.6 TB/s), [2048, 2 x 6144] 15.3 / 13.9).
// The first line lies near 1.5 M elements ([512, 2 x 2816] 3.88 / 3.89, [128, 2 x 12288] 3.93
// / 3.90; graph replays over rotating inputs).  Eight elements come with non-temporal loads,
// which leave what the caller's next kernels read in the caches: alone no faster than
// four (40.7 us, and [2048, 2 x 6144] 14.5), but one layer's element-wise work over
// 3072 tokens takes 106.8 us instead of 111.7; rows that leave more than a sixth of
// their 2048-element blocks empty keep four ([2511, 2 x 2112] 7.7 / 10.6).  g and u may be
// strided views (e.g. the two halves of a packed [rows, 2F] gate/up).
#include "common.h"
#include "respect_amd.h"

namespace rspx {

__device__ __forceinline__ float swiglu1(float g, float u) { return round_bf16(silu_f32(g)) * u; }

constexpr int swiglu_threads(int V) { return V >= 4 ? 256 : 512; }
constexpr int64_t kWide = 3 << 19, kWider = 1 << 24;   // elements
constexpr int kMaxGridY = 65535;

// V elements per thread: 8, 4, 2 or 1.
template <int V>
__global__ __launch_bounds__(swiglu_threads(V)) void silu_mul_kernel(const uint16_t* g, int64_t sg, const uint16_t* u,
                                                                     int64_t su, uint16_t* y, int64_t sy, int row0,
                                                                     int units) {
  // Every argument in one scalar-load batch, ahead of the index arithmetic.
  asm volatile("" ::"s"(g), "s"(sg), "s"(u), "s"(su), "s"(y), "s"(sy), "s"(row0), "s"(units));
  const int unit = blockIdx.x * swiglu_threads(V) + threadIdx.x;
  if (unit >= units) return;
  const int c = unit * V;
  const int row = row0 + blockIdx.y;
  if constexpr (V == 8) {
    const u32x4 gw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(g + row * sg + c));
    const u32x4 uw = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(u + row * su + c));
    u32x4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      o[i] = pack_bf16x2(swiglu1(bf16_lo(gw[i]), bf16_lo(uw[i])), swiglu1(bf16_hi(gw[i]), bf16_hi(uw[i])));
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(y + row * sy + c));
  } else if constexpr (V == 4) {
    const u32x2 gw = *reinterpret_cast<const u32x2*>(g + row * sg + c);
    const u32x2 uw = *reinterpret_cast<const u32x2*>(u + row * su + c);
    u32x2 o;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      o[i] = pack_bf16x2(swiglu1(bf16_lo(gw[i]), bf16_lo(uw[i])), swiglu1(bf16_hi(gw[i]), bf16_hi(uw[i])));
    __builtin_nontemporal_store(o, reinterpret_cast<u32x2*>(y + row * sy + c));
  } else if constexpr (V == 2) {
    const uint32_t gw = *reinterpret_cast<const uint32_t*>(g + row * sg + c);
    const uint32_t uw = *reinterpret_cast<const uint32_t*>(u + row * su + c);
    __builtin_nontemporal_store(pack_bf16x2(swiglu1(bf16_lo(gw), bf16_lo(uw)), swiglu1(bf16_hi(gw), bf16_hi(uw))),
                                reinterpret_cast<uint32_t*>(y + row * sy + c));
  } else {
    __builtin_nontemporal_store(
        f32_to_bf16_rne(swiglu1(bf16_to_f32(g[row * sg + c]), bf16_to_f32(u[row * su + c]))), y + row * sy + c);
  }
}
}  // namespace rspx

using namespace rspx;

extern "C" int rspx_silu_mul(const void* g, int64_t sg, const void* u, int64_t su, void* y, int64_t sy, int rows,
                             int cols, void* stream) {
  if (rows < 0 || cols < 0) return RSPX_EINVAL;
  if ((int64_t)rows * cols == 0) return RSPX_OK;
  if (!g || !u || !y) return RSPX_EINVAL;
  auto al = [](const void* p, unsigned a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) == 0; };
  if (!al(g, 2) || !al(u, 2) || !al(y, 2)) return RSPX_EALIGN;
  auto fits = [&](int v) {
    return cols % v == 0 && al(g, 2 * v) && al(u, 2 * v) && al(y, 2 * v) && sg % v == 0 && su % v == 0 && sy % v == 0;
  };
  const int64_t n = (int64_t)rows * cols;
  const bool full = 5 * (((int64_t)cols + 2047) / 2048 * 2048) <= 6 * (int64_t)cols;   // blocks of eight elements per thread
  const int v = n >= kWider && full && fits(8) ? 8 : n >= kWide && fits(4) ? 4 : fits(2) ? 2 : 1;
  const int units = cols / v;
  const unsigned bx = (unsigned)((units + swiglu_threads(v) - 1) / swiglu_threads(v));
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const uint16_t* G = static_cast<const uint16_t*>(g);
  const uint16_t* U = static_cast<const uint16_t*>(u);
  uint16_t* Y = static_cast<uint16_t*>(y);
  for (int row0 = 0; row0 < rows; row0 += kMaxGridY) {   // one launch per 65535 rows
    const dim3 grid(bx, (unsigned)min(rows - row0, kMaxGridY));
    const dim3 b(swiglu_threads(v));
    if (v == 8) hipLaunchKernelGGL(silu_mul_kernel<8>, grid, b, 0, s, G, sg, U, su, Y, sy, row0, units);
    else if (v == 4) hipLaunchKernelGGL(silu_mul_kernel<4>, grid, b, 0, s, G, sg, U, su, Y, sy, row0, units);
    else if (v == 2) hipLaunchKernelGGL(silu_mul_kernel<2>, grid, b, 0, s, G, sg, U, su, Y, sy, row0, units);
    else hipLaunchKernelGGL(silu_mul_kernel<1>, grid, b, 0, s, G, sg, U, su, Y, sy, row0, units);
  }
  return hipGetLastError() == hipSuccess ? RSPX_OK : RSPX_ELAUNCH;
}
