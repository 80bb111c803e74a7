// Split-K int8 implicit GEMM for layers with few output pixels (one frame's
// 20x20 and 40x40 maps, classifier tails): the same convolution and packed
// operands as igemm_kernel.h, another split of the work.
//
// Such a layer gives the other kernels a few dozen workgroups, each walking
// all of K through its CU's memory path (a wave instruction of im2col rows
// touches 16 half-used lines), one 100-200 ns k-step after another.  Here a
// workgroup owns 16 pixels x 16 CB channels and its NW waves take a
// contiguous part of K each: NW times as many CUs share the loads, and a
// wave issues kKsAhead k-steps of both operands before its first matrix
// instruction, so a layer of up to NW * kKsAhead k-steps waits for memory
// once.  Nothing is shared before the sums, so the weights go from the
// packed rows (1 KB contiguous a fragment) straight to registers.  The int32
// partial sums meet in LDS, wave cb adds those of channel block cb and runs
// the epilogue; integer sums are the same in any order, so the bytes are the
// other kernels'.  20 x 20 128 -> 128 3x3 on one frame: 6.4 -> 4.0 us; one
// 640x640 frame of the detector graph 292 -> 268 us, 16 classifier images 144
// -> 122 us.
#pragma once

#include "igemm_kernel.h"

namespace dw {

// int8 only; false if no kernel exists for the tile (bc 16 or 32, pb = NW 4, 8 or 16).
bool igemm_launch_ks_i8(hipStream_t st, const IgemmArgs& a, const TileCfg& t);

namespace ig {

constexpr int kKsAhead = 5;

template <int CB, int NW>
__global__ __launch_bounds__(NW * 64) void igemm_ks_kernel(const IgemmArgs a) {
  __shared__ v4i red[NW][CB][64];
  __shared__ __align__(4) uint8_t s_lut[256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ctiles = a.cout_pad / (16 * CB);
  const int pt = (int)blockIdx.x / ctiles;
  const int c0 = ((int)blockIdx.x - pt * ctiles) * 16 * CB, p0 = pt * 16;
  const bool second = a.y2 != nullptr && c0 >= a.split;  // a sibling GEMM's second conv
  const uint8_t* lut = second ? a.lut2 : a.lut;
  // the epilogue's operands, on their way under everything else: the table
  // (into LDS before the sums meet), and in the waves that run it (one
  // channel block each) the residual and the channels' values
  const uint32_t lut4 = lut && wave == NW - 1 ? reinterpret_cast<const uint32_t*>(lut)[lane] : 0u;
  const int p = p0 + (lane & 15), cl = wave * 16 + 4 * (lane >> 4), ch = c0 + cl;
  const bool mine = wave < CB && p < a.m && ch < a.cout;
  int4 bi = make_int4(0, 0, 0, 0);
  float4 ms = make_float4(0, 0, 0, 0);
  uint32_t rres = 0;
  if (mine && a.epi == EPI_QU8) {
    if (a.bias_i) bi = *reinterpret_cast<const int4*>(a.bias_i + ch);
    ms = *reinterpret_cast<const float4*>(a.mscale + ch);
    if (a.res)
      rres = *reinterpret_cast<const uint32_t*>((const uint8_t*)a.res + (size_t)p * a.r_pix_stride + a.r_c_off + ch);
  }
  int pbase[1];
  uint32_t tmask[1];
  pixel_setup<1>(a, p0, lane, true, pbase, tmask);
  const int kelems = a.kh * a.kw * a.cin;
  const int per = (a.ksteps + NW - 1) / NW, k0 = wave * per, k1 = min(a.ksteps, k0 + per);
  const __amdgpu_buffer_rsrc_t xrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, a.x_bytes, 0x00020000);
  const uint8_t* wl = a.wpk + (size_t)(c0 + (lane & 15)) * 64 + (lane >> 4) * 16;
  v4i acc[CB];
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) acc[cb] = v4i{0, 0, 0, 0};
  for (int kb = k0; kb < k1; kb += kKsAhead) {
    v4i wf[kKsAhead][CB];
    u32x4 xf[kKsAhead];
    uint32_t key[kKsAhead];
#pragma unroll
    for (int u = 0; u < kKsAhead; ++u) {
      // past the wave's part: the last weights again against zeros
      const int ks = min(kb + u, k1 - 1);
      const bool live = kb + u < k1;
#pragma unroll
      for (int cb = 0; cb < CB; ++cb)
        wf[u][cb] = *reinterpret_cast<const v4i*>(wl + ((size_t)ks * a.cout_pad + cb * 16) * 64);
      const int e = ks * 64 + (lane >> 4) * 16;
      const int tap = div_small(min(e, kelems - 1), a.cin, a.r_cin);
      const int ci = e - tap * a.cin;
      const int kh = div_small(tap, a.kw, a.r_kw);
      const int kw = tap - kh * a.kw;
      const bool in = live & (e < kelems) & (((tmask[0] >> tap) & 1u) != 0);
      const int off = pbase[0] + (kh * a.w + kw) * a.x_pix_stride + ci;
      xf[u] = __builtin_bit_cast(u32x4,
                                 __builtin_amdgcn_raw_buffer_load_b128(xrsrc, in ? off : (int)0x80000000, 0, 0));
      key[u] = in ? a.xxor : live ? a.xpad : 0u;
    }
    __builtin_amdgcn_sched_barrier(0);  // every load before the first matrix instruction
#pragma unroll
    for (int u = 0; u < kKsAhead; ++u) {
      const v4i b = __builtin_bit_cast(v4i, xf[u] ^ key[u]);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) acc[cb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(wf[u][cb], b, acc[cb], 0, 0, 0);
    }
  }
#pragma unroll
  for (int cb = 0; cb < CB; ++cb) red[wave][cb][lane] = acc[cb];
  if (lut && wave == NW - 1) reinterpret_cast<uint32_t*>(s_lut)[lane] = lut4;
  __syncthreads();
  if (!mine) return;
  v4i sum = red[0][wave][lane];
#pragma unroll
  for (int w = 1; w < NW; ++w) sum += red[w][wave][lane];
  if (a.epi != EPI_QU8) {
    const EpiLds none{nullptr, nullptr, nullptr, nullptr};
    epilogue4<1>(a, none, sum, ch, cl, p);
    return;
  }
  const int accs[4] = {sum[0] + bi.x, sum[1] + bi.y, sum[2] + bi.z, sum[3] + bi.w};
  const float mss[4] = {ms.x, ms.y, ms.z, ms.w};
  uint32_t out = 0;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    int qi = requant_u8(accs[r], mss[r], (float)a.y_zp);
    if (lut) qi = s_lut[qi];
    if (a.res) qi = qadd_u8(qi, (rres >> (8 * r)) & 0xff, a);
    out |= (uint32_t)qi << (8 * r);
  }
  uint8_t* y = second ? (uint8_t*)a.y2 + (size_t)p * a.y2_pix_stride + a.y2_c_off - a.split
                      : (uint8_t*)a.y + (size_t)p * a.y_pix_stride + a.y_c_off;
  *reinterpret_cast<uint32_t*>(y + ch) = out;
  if (a.y_up) {
    // the nearest 2x upsample: the same values at the pixel's four pixels
    const int hw = a.ho * a.wo, nn = div_small(p, hw, a.r_hwo), r = p - nn * hw;
    const int oh = div_small(r, a.wo, a.r_wo), ow = r - oh * a.wo;
    uint8_t* u = (uint8_t*)a.y_up + ((size_t)(nn * 2 * a.ho + 2 * oh) * (2 * a.wo) + 2 * ow) * a.up_pix_stride +
                 a.up_c_off + ch;
    const size_t upr = (size_t)2 * a.wo * a.up_pix_stride;
    *reinterpret_cast<uint32_t*>(u) = out;
    *reinterpret_cast<uint32_t*>(u + a.up_pix_stride) = out;
    *reinterpret_cast<uint32_t*>(u + upr) = out;
    *reinterpret_cast<uint32_t*>(u + upr + a.up_pix_stride) = out;
  }
}

template <int CB, int NW>
void launch_ks(hipStream_t st, const IgemmArgs& a) {
  const unsigned wgs = (unsigned)(((a.m + 15) / 16) * (a.cout_pad / (16 * CB)));
  hipLaunchKernelGGL((igemm_ks_kernel<CB, NW>), dim3(wgs), dim3(NW * 64), 0, st, a);
}

}  // namespace ig
}  // namespace dw
