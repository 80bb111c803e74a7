// Depthwise 3x3, stride 1 or 2, over f16 or f32 NHWC, in the reference's
// accumulation order (dwconv3_tile_kernel in k_dwtile.hip is the packed-f16
// alternative of the fp16 graphs).
//
// A thread owns 4 channels of 2 output columns and marches down the image:
// every input row of its 4 (stride 2: 5) columns is loaded and widened once,
// then goes into the chains of all the output rows that it is a tap row of
// (at stride 1 the third taps of one, the second of the next and the first of
// the one after).  The chains stay in registers between rows, so no window is
// kept and no input is read twice down a block of rows; the next row's loads
// are in flight while one is summed.  (4 columns a thread widen a quarter
// less but need 138 registers, not 103: 24.4 against 22.2 us below.)
// ROW1 is a block of a single output row, of 4 columns, all of its input
// loaded up front: shorter where there are few threads (4.7 us against 5.1 us
// for a march of 2 rows on 1 x 20 x 20 x 256).
//
// Bound by the vector ALUs in f16 (of 3.7 instructions a tap and value, one
// is the FMA, the rest widening, rounding, bias and SiLU), by memory in f32:
// 32 x 40 x 40 x 384 f16 22.2 us, 3.5 TB/s (32.7 us as one row of 4 columns a
// thread with its whole window loaded and decoded), f32 34 us, 4.6 TB/s (86 us
// as one pixel a thread, each tap read under its own condition).
//
// Each output is the reference's sum: taps in (kh, kw) order, fmaf in f32.
// Loads are buffer loads; rows and columns outside the image are sent past
// the buffer and read zeros.  In f16 such a tap adds an exact +0, which
// leaves the sum as the reference's skip does (weights are finite and no
// product of two f16 values underflows, so the running sum is never -0); in
// f32 the chain keeps its value.  The offsets are 32-bit: x spans at most
// 2^30 bytes, so that one or two times kBad (2^30) lies past it.
//
// f16 subnormals are widened to half their value, as the reference does: a
// wave that loaded none skips that.  Bias: the reference adds in f32 and
// rounds to f16; for f16 operands that is the correctly rounded f16 sum (f32
// holds 2 * 11 + 2 bits), so two channels are added by one packed f16 add,
// unless a sum or the bias is an f16 subnormal.  SiLU: as silu_f16_pk_lite
// (fp16 tolerance).
#include "direct_util.h"

#include <algorithm>

namespace dw {
namespace {

constexpr int kCpt = 4;  // channels of a thread
constexpr int kBad = 0x40000000;

struct Dw3Args {
  DwArgs d;
  int segs, rblocks, rows, x_bytes;
};

// The row of NC columns x 4 channels as loaded.
template <bool H, int NC>
struct RawRow {
  uint32_t v[NC][H ? 2 : 4];
};

// h2f of N x 4 f16 values, of which a wave rarely holds a subnormal.
template <int N>
__device__ __forceinline__ void widen_f16(const uint32_t (&h)[N][2], float (&f)[N][4]) {
  // any subnormal: (2|h| - 2) mod 2^16 < 0x7fe, both halves at once (one
  // packed multiply-add, one packed min per register)
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  uint32_t mn = 0xffffffffu;
  const uint32_t two = 0x00020002u, m2 = 0xfffefffeu;
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      uint32_t t;
      asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(t) : "v"(h[i][e]), "v"(two), "s"(m2));
      mn = __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(us2, mn),
                                                                  __builtin_bit_cast(us2, t)));
      f[i][2 * e] = h2f_ieee(h[i][e] & 0xffff);
      f[i][2 * e + 1] = h2f_ieee(h[i][e] >> 16);
    }
  if (__any((mn & 0xffffu) < 0x7feu || (mn >> 16) < 0x7feu)) {
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) f[i][c] = fabsf(f[i][c]) < 6.103515625e-05f ? f[i][c] * 0.5f : f[i][c];
  }
}

// silu_f16_pk_lite with each scaled argument in one instruction.
__device__ __forceinline__ h16x2 silu_mix(h16x2 x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  const float e0 = __builtin_amdgcn_exp2f(fma_mix_hf0<0>(u, -1.44269502f));
  const float e1 = __builtin_amdgcn_exp2f(fma_mix_hf0<1>(u, -1.44269502f));
  return x * pk_f2h(__builtin_amdgcn_rcpf(1.0f + e0), __builtin_amdgcn_rcpf(1.0f + e1));
}

// SEG: output columns of a thread.
template <bool H, int SW, int SEG, bool ROW1, int ACT>
__global__ __launch_bounds__(256) void dwconv3_kernel(const Dw3Args p) {
  constexpr int NC = SW * (SEG - 1) + 3;
  constexpr int ES = H ? 2 : 4;
  const DwArgs& a = p.d;
  const int groups = a.c / kCpt;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.n * p.rblocks * p.segs * groups) return;
  const int g = t % groups;
  int rest = t / groups;
  const int sg = rest % p.segs;
  rest /= p.segs;
  const int rb = rest % p.rblocks;
  const int nn = rest / p.rblocks;
  const int c0 = g * kCpt, ow0 = sg * SEG;
  const int rows = ROW1 ? 1 : p.rows;
  const int oh0 = rb * rows;

  const __amdgpu_buffer_rsrc_t xrs =
      __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, p.x_bytes, 0x00020000);
  const int ps = a.x_pix_stride * ES;
  const int iw0 = ow0 * SW - a.pl;
  int colo[NC];
#pragma unroll
  for (int q = 0; q < NC; ++q) colo[q] = (unsigned)(iw0 + q) < (unsigned)a.w ? (iw0 + q) * ps : kBad;
  int ih = oh0 * SW - a.pt;  // next row to load
  const int img = nn * a.h;
  const int coff = (a.x_c_off + c0) * ES;
  auto load = [&](RawRow<H, NC>& r) {
    const int rowo = (unsigned)ih < (unsigned)a.h ? (img + ih) * a.w * ps + coff : kBad;
    ++ih;
#pragma unroll
    for (int q = 0; q < NC; ++q) {
      if constexpr (H) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(xrs, rowo + colo[q], 0, 0);
        r.v[q][0] = v[0];
        r.v[q][1] = v[1];
      } else {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(xrs, rowo + colo[q], 0, 0);
#pragma unroll
        for (int c = 0; c < 4; ++c) r.v[q][c] = v[c];
      }
    }
  };

  RawRow<H, NC> raw[ROW1 ? 3 : 1];
  float wv[9][kCpt];
  float bf[kCpt];          // f32 bias
  uint2 br = make_uint2(0, 0);  // f16 bias
  if constexpr (H) {
    uint32_t wr[9][2];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const uint2 w2 = *reinterpret_cast<const uint2*>((const uint16_t*)a.wt + (size_t)k * a.c + c0);
      wr[k][0] = w2.x;
      wr[k][1] = w2.y;
    }
    if (a.bias) br = *reinterpret_cast<const uint2*>((const uint16_t*)a.bias + c0);
#pragma unroll
    for (int i = 0; i < (ROW1 ? 3 : 1); ++i) load(raw[i]);
    widen_f16<9>(wr, wv);
  } else {
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const float4 w4 = *reinterpret_cast<const float4*>((const float*)a.wt + (size_t)k * a.c + c0);
      wv[k][0] = w4.x; wv[k][1] = w4.y; wv[k][2] = w4.z; wv[k][3] = w4.w;
    }
    if (a.bias) {
      const float4 b4 = *reinterpret_cast<const float4*>((const float*)a.bias + c0);
      bf[0] = b4.x; bf[1] = b4.y; bf[2] = b4.z; bf[3] = b4.w;
    }
#pragma unroll
    for (int i = 0; i < (ROW1 ? 3 : 1); ++i) load(raw[i]);
  }
  const uint16_t bh[kCpt] = {(uint16_t)(br.x & 0xffff), (uint16_t)(br.x >> 16), (uint16_t)(br.y & 0xffff),
                             (uint16_t)(br.y >> 16)};
  bool bias_sub = false;
#pragma unroll
  for (int c = 0; c < kCpt; ++c) bias_sub |= (uint16_t)((bh[c] & 0x7fff) - 1) < 0x3ff;

  // The widened current row, and which of its values lie in the image.
  float x[NC][kCpt];
  bool in[NC];
  auto widen = [&](const RawRow<H, NC>& r, int row) {
    if constexpr (H) {
      widen_f16<NC>(r.v, x);
    } else {
      const bool row_in = (unsigned)row < (unsigned)a.h;
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        in[q] = row_in & (colo[q] != kBad);
#pragma unroll
        for (int c = 0; c < kCpt; ++c) x[q][c] = __builtin_bit_cast(float, r.v[q][c]);
      }
    }
  };

  // The three taps of row kh on the chains of one output row.
  auto taps = [&](int kh, float (&to)[SEG][kCpt], const float (&from)[SEG][kCpt]) {
#pragma unroll
    for (int j = 0; j < SEG; ++j)
#pragma unroll
      for (int c = 0; c < kCpt; ++c) {
        float s = from[j][c];
#pragma unroll
        for (int kw = 0; kw < 3; ++kw) {
          const int q = SW * j + kw;
          const float v = fmaf(x[q][c], wv[kh * 3 + kw][c], s);
          s = H || in[q] ? v : s;
        }
        to[j][c] = s;
      }
  };

  uint8_t* yrow = (uint8_t*)a.y + ((((size_t)nn * a.ho + oh0) * a.wo + ow0) * a.y_pix_stride + a.y_c_off + c0) * ES;
  const size_t yps = (size_t)a.y_pix_stride * ES, yrs = yps * a.wo;
  int oh = oh0;  // of the next finished row
  auto finish = [&](const float (&acc)[SEG][kCpt]) {
    if (oh < a.ho) {
      if constexpr (H) {
        // the conv result rounded to f16 (the reference's store)
        h16x2 r[SEG][2];
        float amin = 1.0f;
#pragma unroll
        for (int j = 0; j < SEG; ++j) {
          float v[kCpt];
#pragma unroll
          for (int c = 0; c < kCpt; ++c) {
            v[c] = acc[j][c];
            asm("" : "+v"(v[c]));  // rounded to f32 before the conversion
            amin = fminf(amin, fabsf(v[c]));
          }
          r[j][0] = h16x2{(_Float16)v[0], (_Float16)v[1]};
          r[j][1] = h16x2{(_Float16)v[2], (_Float16)v[3]};
        }
        if (a.bias) {
          if (__any(bias_sub || amin < 6.103515625e-05f)) {
#pragma unroll
            for (int j = 0; j < SEG; ++j)
#pragma unroll
              for (int h = 0; h < 2; ++h)
                r[j][h] = pk_make(f16_add_bits(pk_lo(r[j][h]), bh[2 * h]), f16_add_bits(pk_hi(r[j][h]), bh[2 * h + 1]));
          } else {
#pragma unroll
            for (int j = 0; j < SEG; ++j) {
              r[j][0] = r[j][0] + __builtin_bit_cast(h16x2, br.x);
              r[j][1] = r[j][1] + __builtin_bit_cast(h16x2, br.y);
            }
          }
        }
#pragma unroll
        for (int j = 0; j < SEG; ++j) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            if constexpr (ACT == ACT_SILU) r[j][h] = silu_mix(r[j][h]);
            if constexpr (ACT == ACT_RELU)
              r[j][h] = pk_make(f16_act_bits(pk_lo(r[j][h]), ACT_RELU), f16_act_bits(pk_hi(r[j][h]), ACT_RELU));
          }
          if (ow0 + j < a.wo)
            *reinterpret_cast<uint2*>(yrow + j * yps) =
                make_uint2(__builtin_bit_cast(uint32_t, r[j][0]), __builtin_bit_cast(uint32_t, r[j][1]));
        }
      } else {
#pragma unroll
        for (int j = 0; j < SEG; ++j) {
          float o[kCpt];
#pragma unroll
          for (int c = 0; c < kCpt; ++c) {
            float v = acc[j][c];
            if (a.bias) v = v + bf[c];
            if constexpr (ACT == ACT_RELU) v = dx::relu_ref(v);
            if constexpr (ACT == ACT_SILU) {
              const float s = 1.0f / (1.0f + expf(-v));
              v = v * s;
            }
            o[c] = v;
          }
          if (ow0 + j < a.wo) *reinterpret_cast<float4*>(yrow + j * yps) = make_float4(o[0], o[1], o[2], o[3]);
        }
      }
    }
    ++oh;
    yrow += yrs;
  };

  const float zero[SEG][kCpt] = {};
  float s0[SEG][kCpt], s1[SEG][kCpt];  // chains with their first, and first two, tap rows summed
  int row = ih - (ROW1 ? 3 : 1);
  if constexpr (ROW1) {
    widen(raw[0], row);
    taps(0, s0, zero);
    widen(raw[1], row + 1);
    taps(1, s0, s0);
    widen(raw[2], row + 2);
    taps(2, s0, s0);
    finish(s0);
  } else {
    auto next = [&] {  // the next input row, the one after it on its way
      widen(raw[0], row++);
      load(raw[0]);
    };
    next();
    taps(0, s0, zero);
    if constexpr (SW == 1) {
      next();
      taps(1, s1, s0);
      taps(0, s0, zero);
#pragma unroll 1
      for (int i = 2; i < rows; ++i) {
        next();
        taps(2, s1, s1);
        finish(s1);
        taps(1, s1, s0);
        taps(0, s0, zero);
      }
      next();
      taps(2, s1, s1);
      finish(s1);
      taps(1, s1, s0);
      widen(raw[0], row);
      taps(2, s1, s1);
      finish(s1);
    } else {
#pragma unroll 1
      for (int i = 1; i < rows; ++i) {
        next();
        taps(1, s0, s0);
        next();
        taps(2, s1, s0);
        taps(0, s0, zero);
        finish(s1);
      }
      next();
      taps(1, s0, s0);
      widen(raw[0], row);
      taps(2, s0, s0);
      finish(s0);
    }
  }
}

template <bool H, int SW, int SEG, bool ROW1>
void launch_act(hipStream_t st, const Dw3Args& p, unsigned blocks) {
  if (p.d.act == ACT_RELU)
    hipLaunchKernelGGL((dwconv3_kernel<H, SW, SEG, ROW1, ACT_RELU>), dim3(blocks), dim3(256), 0, st, p);
  else if (p.d.act == ACT_SILU)
    hipLaunchKernelGGL((dwconv3_kernel<H, SW, SEG, ROW1, ACT_SILU>), dim3(blocks), dim3(256), 0, st, p);
  else if (!H || p.d.act == ACT_NONE)  // (f32: a value that names no activation is none, as in dwconv_kernel)
    hipLaunchKernelGGL((dwconv3_kernel<H, SW, SEG, ROW1, ACT_NONE>), dim3(blocks), dim3(256), 0, st, p);
  else
    fail(-2, "depthwise: no kernel for this activation");
}

}  // namespace

bool launch_dwconv3(hipStream_t st, const DwArgs& a, int dtype) {
  const int es = dtype == F16 ? 2 : 4;
  const size_t al = 4 * es;  // a thread's four channels
  const long long x_bytes = ((long long)a.n * a.h * a.w - 1) * a.x_pix_stride * es + (long long)(a.x_c_off + a.c) * es;
  if (a.kh != 3 || a.kw != 3 || (a.sw != 1 && a.sw != 2) || a.sh != a.sw || a.c % kCpt != 0 || x_bytes > (1ll << 30) ||
      (uintptr_t)a.x % al != 0 || (uintptr_t)a.y % al != 0 || (uintptr_t)a.wt % al != 0 || (uintptr_t)a.bias % al != 0 ||
      a.x_pix_stride % 4 != 0 || a.x_c_off % 4 != 0 || a.y_pix_stride % 4 != 0 || a.y_c_off % 4 != 0)
    return false;
  Dw3Args p{a};
  p.x_bytes = (int)x_bytes;
  const long long pairs = (long long)a.n * a.ho * ((a.wo + 1) / 2) * (a.c / kCpt);
  if (pairs >= (1ll << 31)) return false;
  // rows of a march: as many as leave 1.5 waves on each of the 1024 SIMDs, up
  // to 12 (beyond, nothing is gained: 22.2 against 22.6 us with 16 on 32 x 40
  // x 40 x 384 f16); with fewer than 2, one row of output a thread
  const int rows = (int)std::min<long long>(12, pairs / 64 / 1536);
  const bool row1 = rows < 2 || a.ho < 2;
  p.rblocks = row1 ? a.ho : (a.ho + rows - 1) / rows;
  p.rows = (a.ho + p.rblocks - 1) / p.rblocks;
  // a map of one or two columns takes threads of as many, which do not compute
  // the columns beside it (19 x 126 x 1 x 136 f16: 6.2 us with 4, 4.6 with 1)
  const int seg = a.wo == 1 ? 1 : a.wo == 2 || !row1 ? 2 : 4;
  p.segs = (a.wo + seg - 1) / seg;
  const unsigned blocks = (unsigned)(((long long)a.n * p.rblocks * p.segs * (a.c / kCpt) + 255) / 256);
#define DW_D3(H_, SW_)                                             \
  if ((dtype == F16) == H_ && a.sw == SW_) {                       \
    if (row1)                                                      \
      seg == 1   ? launch_act<H_, SW_, 1, true>(st, p, blocks)     \
      : seg == 2 ? launch_act<H_, SW_, 2, true>(st, p, blocks)     \
                 : launch_act<H_, SW_, 4, true>(st, p, blocks);    \
    else                                                           \
      seg == 1 ? launch_act<H_, SW_, 1, false>(st, p, blocks)      \
               : launch_act<H_, SW_, 2, false>(st, p, blocks);     \
  }
  DW_D3(true, 1)
  DW_D3(true, 2)
  DW_D3(false, 1)
  DW_D3(false, 2)
#undef DW_D3
  DW_HIP(hipGetLastError());
  return true;
}

}  // namespace dw
