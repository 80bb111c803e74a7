// In-order fp16 implicit GEMM for layers with few output pixels (20x20 and
// 13x13 maps, single frames): the same convolution and packed operands as
// igemm_kernel.h, one accumulator chain per output as there.
//
// The sums of fp16 layers keep one order, so K cannot be split over waves as
// igemm_ks.h does, and such a layer walks its k-steps one after another: with
// weights staged in LDS and 64 pixels a workgroup, 100-220 ns a step on a few
// dozen CUs.  Here a workgroup is one wave that owns 16 pixels x 16 CB
// channels and shares nothing: both operands go straight to registers
// (weights are 1 KB contiguous a fragment) through a ring of 8 to 16 k-steps,
// so that many steps' loads are in flight and no barrier stands between them.
// A step is then bound by the instructions of its one wave: addresses are
// kept in scalar registers and worked out once for up to four k-steps of a
// tap (per lane and k-step, as igemm_ks.h does it, they cost 60 instructions
// and gained nothing).  Two waves a workgroup were no faster.  20 x 20 128 ->
// 128 3x3 on one frame: 8.8 -> 5.2 us, 40 x 40 128 -> 256 3x3/2 8.9 -> 5.3 us,
// the batch-5 416 x 416 fp16 detector graph 383 -> 337 us.
#pragma once

#include "igemm_kernel.h"

namespace dw {

// fp16 only; false if no kernel exists for the tile (bc 16, 32 or 64).
bool igemm_launch_fp_f16(hipStream_t st, const IgemmArgs& a, const TileCfg& t);

namespace ig {


// G: k-steps that lie in one tap together (c_in a multiple of 32 G), whose
// loads share their address arithmetic.
template <int CB, int G>
__global__ __launch_bounds__(64) void igemm_fp_kernel(const IgemmArgs a) {
  constexpr int BC = 16 * CB;
  constexpr int A = CB == 1 ? 16 : CB == 2 ? 12 : 8;  // k-steps in flight
  __shared__ __align__(8) uint16_t s_bias[BC];
  const int lane = threadIdx.x;
  const int ctiles = a.cout_pad / BC;
  const int pt = (int)blockIdx.x / ctiles;
  const int c0 = ((int)blockIdx.x - pt * ctiles) * BC, p0 = pt * 16;
  if (a.bias_h && lane < BC) s_bias[lane] = c0 + lane < a.cout ? a.bias_h[c0 + lane] : (uint16_t)0;
  int pbase[1];
  uint32_t tmask[1];
  pixel_setup<1>(a, p0, lane, true, pbase, tmask);
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, a.x_bytes, 0x00020000);
  const int xlane = pbase[0] * 2 + (lane >> 4) * 16;
  const uint32_t wlane = (lane & 15) * 64 + (lane >> 4) * 16;
  const size_t wstep = (size_t)a.cout_pad * 64;
  const int ksteps = a.ksteps, tap_bytes = a.cin * 2, xps = a.x_pix_stride * 2, row_skip = (a.w - a.kw) * xps, kws = a.kw;
  v4i wf[A][CB];
  u32x4 xf[A];
  // the next k-steps to load: their number and weights, their tap, the tap's
  // byte offset from the pixel's top-left tap, its column and the first byte
  // of the tap, all in scalar registers; past the end the last weights
  // against zeros
  const uint8_t* wk = a.wpk + (size_t)c0 * 64;
  int nk = 0, ntap = 0, noff = 0, nkw = 0, nci = 0;
  auto load = [&](int u) {
    const uint32_t bit = nk < ksteps ? 1u << ntap : 0u;
    const int off = (tmask[0] & bit) ? xlane + (noff + nci) : (int)0x80000000;
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        wf[u + g][cb] = *reinterpret_cast<const v4i*>(wk + g * wstep + (wlane + cb * 1024));
      xf[u + g] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xrsrc, off, g * 64, 0));
    }
    nk += G;
    wk += nk < ksteps ? G * wstep : 0;
    nci += 64 * G;
    const bool tap_end = nci == tap_bytes;
    nci = tap_end ? 0 : nci;
    ntap += tap_end;
    nkw += tap_end;
    noff += tap_end ? xps : 0;
    const bool row_end = nkw == kws;
    nkw = row_end ? 0 : nkw;
    noff += row_end ? row_skip : 0;
    __builtin_amdgcn_sched_barrier(0);  // the loads stay in ring order
  };
  v4f acc[CB][1];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb][0] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int u = 0; u < A; u += G) load(u);
  for (int kb = 0; kb < ksteps; kb += A) {
#pragma unroll
    for (int u = 0; u < A; u += G) {
      if (kb + u < ksteps) {
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int cb = 0; cb < CB; ++cb)
            acc[cb][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wf[u + g][cb]),
                                                                __builtin_bit_cast(v8h, xf[u + g]), acc[cb][0], 0, 0, 0);
      }
      load(u);
    }
  }
  const EpiLds ep{nullptr, nullptr, nullptr, a.bias_h ? s_bias : nullptr};
  igemm_store<2, BC, 1, EPV_GENERIC>(a, ep, acc, c0, p0, lane, nullptr, nullptr);
}

template <int CB>
void launch_fp(hipStream_t st, const IgemmArgs& a) {
  const unsigned wgs = (unsigned)(((a.m + 15) / 16) * (a.cout_pad / (16 * CB)));
  if (a.cin % 128 == 0)
    hipLaunchKernelGGL((igemm_fp_kernel<CB, 4>), dim3(wgs), dim3(64), 0, st, a);
  else if (a.cin % 64 == 0)
    hipLaunchKernelGGL((igemm_fp_kernel<CB, 2>), dim3(wgs), dim3(64), 0, st, a);
  else
    hipLaunchKernelGGL((igemm_fp_kernel<CB, 1>), dim3(wgs), dim3(64), 0, st, a);
}

}  // namespace ig
}  // namespace dw
