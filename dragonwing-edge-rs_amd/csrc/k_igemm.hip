// Implicit-GEMM convolution on CDNA4 matrix cores: tile selection, launch
// dispatch and weight packing.  The kernels are igemm_kernel.h, the
// persistent igemm_sk.h for small K, the streamed-weight igemm_stream.h for
// long K, the row-, band- and wide-tile kernels (igemm_rows.h, igemm_band.h,
// igemm_wide.h); their instantiations live in the k_igemm_*.hip files so
// that they compile in parallel.
#include "igemm_band.h"
#include "igemm_fp.h"
#include "igemm_ks.h"
#include "igemm_rows.h"
#include "igemm_sk.h"
#include "igemm_stream.h"
#include "igemm_wide.h"

#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>

namespace dw {
namespace {

// ---------------------------------------------------------------------------
// Weight packing: HWIO [K][cout] -> [ksteps][cout_pad][64 bytes], zero filled,
// with the QLinearConv's per-channel values in the same pass.
// ---------------------------------------------------------------------------

// The multipliers of one launch's channels, passed by value: they live in
// the caller's host array, and as kernel arguments they need no copy that
// the host would have to wait for.  With the other 64 bytes of arguments they
// fill 4 KB.
constexpr int kPrepChannels = 1008;
struct PrepScales {
  float m[kPrepChannels];
};
struct QconvPrep {
  const int* bias;  // int32 [cout] or null
  int* bias_out;    // (bias ? bias[c] : 0) + corr * sum_k w[k][c]
  float* ms_out;    // the multipliers as the epilogue reads them
  int corr, c0;     // c0: first channel of the launch
};

// A workgroup owns 16 channels; a wave takes whole k-steps of 64 bytes of K.
// Lane (kg, quad) reads one dword of weights per row (4 int8 channels; a
// uint2 for f16) for the rows its output dword holds, transposes them in
// registers (v_perm) and stores 4 dwords, one per channel: each store
// instruction writes four whole 64-byte rows.  The channel sums of the
// QLinearConv bias come from the transposed dwords (one dot4 each), reduced
// over the 16 lanes of a quad and the waves.  Bound by the lines a
// workgroup touches (16 bytes of each row's line) and two trips to memory:
// 16 waves with kPackAhead k-steps of loads in flight each.  2304 x 256
// takes 7.3 us against 5.1 us for a byte per thread plus 232 us for a thread
// summing a whole channel; 1152 x 256 5.3 us against 5.1 + 117 us.
//
// SUM: bias' needs the channel sums (corr != 0), so a workgroup walks all of
// K.  A zero point of 128 (activations around zero) needs none: the k-steps
// then spread over the grid, four to a workgroup, and its first row writes
// bias' and the multipliers: 2304 x 256 in 3.4 us, its whole QLinearConv at
// 20 x 20 12.4 -> 9.5 us.  Other zero points stay at the figures above.
template <int ESZ, bool Q, bool SUM>
__device__ __forceinline__ void pack_weights_body(const uint8_t* __restrict__ w, uint8_t* __restrict__ out, int K,
                                                  int cout, int cout_pad, int ksteps, const QconvPrep& q,
                                                  const float* m) {
  constexpr int RK = 4 / ESZ;  // rows of K in one output dword
  constexpr int kPackAhead = SUM ? 3 : 1;  // k-steps a wave loads before it stores the first
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const int kg = lane & 15, quad = lane >> 4;
  const int cb = blockIdx.x * 16 + (Q ? q.c0 : 0);  // first channel of the workgroup
  const int c = cb + quad * 4;
  const bool in = c < cout;  // cout % 4 == 0: all four channels or none
  int sum[4] = {0, 0, 0, 0};
  // the last threads' operands, fetched under the weight loads
  [[maybe_unused]] float m_ch = 0.0f;
  [[maybe_unused]] int bias_ch = 0;
  if constexpr (Q)
    if ((SUM || blockIdx.y == 0) && threadIdx.x < 16 && cb + (int)threadIdx.x < cout) {
      m_ch = m[blockIdx.x * 16 + threadIdx.x];
      bias_ch = q.bias ? q.bias[cb + threadIdx.x] : 0;
    }
  const int step = gridDim.y * waves;
  for (int s0 = blockIdx.y * waves + wave; s0 < ksteps; s0 += kPackAhead * step) {
    // past K or c_out the last row or the first channels are read and
    // replaced by zeros (a load under a condition would be a branch, waited
    // for by itself)
    uint32_t r[kPackAhead][4];
#pragma unroll
    for (int u = 0; u < kPackAhead; ++u) {
      const int k0 = (s0 + u * step) * (64 / ESZ) + kg * RK;
#pragma unroll
      for (int j = 0; j < RK; ++j) {
        const size_t at = (size_t)(k0 + j < K ? k0 + j : K - 1) * cout + (in ? c : 0);
        if constexpr (ESZ == 1) {
          r[u][j] = *reinterpret_cast<const uint32_t*>(w + at);
        } else {
          const uint2 v = *reinterpret_cast<const uint2*>(w + at * 2);
          r[u][2 * j] = v.x;
          r[u][2 * j + 1] = v.y;
        }
      }
    }
#pragma unroll
    for (int u = 0; u < kPackAhead; ++u) {
      const int k0 = (s0 + u * step) * (64 / ESZ) + kg * RK;
#pragma unroll
      for (int j = 0; j < 4; ++j) r[u][j] = in && k0 + j * RK / 4 < K ? r[u][j] : 0u;
    }
#pragma unroll
    for (int u = 0; u < kPackAhead; ++u) {
      const int s = s0 + u * step;
      if (s >= ksteps) break;
      uint32_t d[4];
      if constexpr (ESZ == 1) {
        const uint32_t t0 = __builtin_amdgcn_perm(r[u][1], r[u][0], 0x05010400u);
        const uint32_t t1 = __builtin_amdgcn_perm(r[u][1], r[u][0], 0x07030602u);
        const uint32_t t2 = __builtin_amdgcn_perm(r[u][3], r[u][2], 0x05010400u);
        const uint32_t t3 = __builtin_amdgcn_perm(r[u][3], r[u][2], 0x07030602u);
        d[0] = __builtin_amdgcn_perm(t2, t0, 0x05040100u);
        d[1] = __builtin_amdgcn_perm(t2, t0, 0x07060302u);
        d[2] = __builtin_amdgcn_perm(t3, t1, 0x05040100u);
        d[3] = __builtin_amdgcn_perm(t3, t1, 0x07060302u);
      } else {
        d[0] = __builtin_amdgcn_perm(r[u][2], r[u][0], 0x05040100u);
        d[1] = __builtin_amdgcn_perm(r[u][2], r[u][0], 0x07060302u);
        d[2] = __builtin_amdgcn_perm(r[u][3], r[u][1], 0x05040100u);
        d[3] = __builtin_amdgcn_perm(r[u][3], r[u][1], 0x07060302u);
      }
      uint8_t* o = out + ((size_t)s * cout_pad + c) * 64 + kg * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        *reinterpret_cast<uint32_t*>(o + j * 64) = d[j];
        if constexpr (SUM) sum[j] = __builtin_amdgcn_sdot4((int)d[j], 0x01010101, sum[j], false);
      }
    }
  }
  const int t = threadIdx.x, ch = cb + t;
  if constexpr (SUM) {
    __shared__ int red[16][16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int x = 1; x < 16; x <<= 1) sum[j] += __shfl_xor(sum[j], x);
      if (kg == 0) red[wave][quad * 4 + j] = sum[j];
    }
    __syncthreads();
    if (t < 16 && ch < cout) {
      uint32_t total = 0;
      for (int v = 0; v < waves; ++v) total += (uint32_t)red[v][t];
      q.bias_out[ch] = (int)((uint32_t)bias_ch + (uint32_t)q.corr * total);
      q.ms_out[ch] = m_ch;
    }
  } else if constexpr (Q) {
    if (blockIdx.y == 0 && t < 16 && ch < cout) {
      q.bias_out[ch] = bias_ch;
      q.ms_out[ch] = m_ch;
    }
  }
}

template <int ESZ>
__global__ __launch_bounds__(1024) void pack_weights_kernel(const uint8_t* w, uint8_t* out, int K, int cout,
                                                            int cout_pad, int ksteps) {
  pack_weights_body<ESZ, false, false>(w, out, K, cout, cout_pad, ksteps, QconvPrep{}, nullptr);
}

template <bool SUM>
__global__ __launch_bounds__(1024) void qconv_prep_kernel(const uint8_t* w, uint8_t* out, int K, int cout,
                                                          int cout_pad, int ksteps, QconvPrep q, PrepScales m) {
  pack_weights_body<1, true, SUM>(w, out, K, cout, cout_pad, ksteps, q, m.m);
}

int channel_tile(int cout) {
  if (cout > 96) return 128;
  if (cout > 80) return 96;
  if (cout > 64) return 80;
  if (cout > 48) return 64;
  if (cout > 32) return 48;
  if (cout > 16) return 32;
  return 16;
}

// LDS for the weight chunk of one workgroup: two workgroups fit a CU.
constexpr int kWeightLds = 65536;

// Prefetch depth of the im2col ring: deeper for narrow pixel tiles, whose
// k-steps are short, so about the same time's worth of loads is in flight.
int ring_depth(int pb) { return pb == 4 ? 4 : (pb == 2 ? 6 : 8); }

bool tile_ok(const IgemmArgs& a, int bc, int pb) {
  const int bcs[] = {128, 96, 80, 64, 48, 32, 16};
  bool known = false;
  for (int b : bcs) known |= b == bc;
  return known && (pb == 1 || pb == 2 || pb == 4) && bc <= channel_tile(a.cout) && a.cout_pad % bc == 0;
}

TileCfg make_tile(const IgemmArgs& a, int bc, int pb) {
  const int kchunk = std::max(1, std::min(a.ksteps, kWeightLds / (bc * 64)));
  return {bc, pb, ring_depth(pb), kchunk, 0};
}

// The persistent small-K kernel: all of K in at most 4 k-steps, instantiated
// for these channel and pixel tiles.
bool sk_ok(const IgemmArgs& a, int bc, int pb, int tpw) {
  return tpw > 0 && a.ksteps >= 1 && a.ksteps <= 4 && (pb == 2 || pb == 4) &&
         (bc == 128 || bc == 64 || bc == 32 || bc == 16) && tile_ok(a, bc, pb);
}

TileCfg make_sk_tile(const IgemmArgs& a, int bc, int pb, int tpw) {
  TileCfg t = make_tile(a, bc, pb);
  t.kchunk = a.ksteps;
  t.tpw = tpw;
  return t;
}

// The streamed-weight kernel (tpw = -1): two or more k-steps, and its
// weight ring and k-slice table fit LDS.
bool st_ok(const IgemmArgs& a, int bc, int pb) {
  return tile_ok(a, bc, pb) && a.ksteps >= 2 && ig::st_lds_bytes(bc, a.ksteps, ring_depth(pb)) <= 160 * 1024;
}

TileCfg make_st_tile(const IgemmArgs& a, int bc, int pb) {
  TileCfg t = make_tile(a, bc, pb);
  t.tpw = -1;
  return t;
}

// The row-tile kernel (tpw = -2): int8 3x3, stride 1, padding 1 (same-size
// output), whole rows of 320 output pixels per workgroup (W divides 320, and
// the row count per tile divides H), channel tiles up to 96 (register
// budget), the input tile within the start-up loads and LDS.
bool rows_ok(const IgemmArgs& a, int bc) {
  const int es = a.epi == EPI_F16 ? 2 : 1;
  if (a.kh != 3 || a.kw != 3 || a.sh != 1 || a.sw != 1 || a.pt != 1 || a.pl != 1) return false;
  if (a.ho != a.h || a.wo != a.w || (a.cin * es) % 16 != 0 || a.w <= 0 || ig::kRowsPix % a.w != 0) return false;
  const int r = ig::kRowsPix / a.w;
  if (a.h % r != 0 || bc > 96 || !tile_ok(a, bc, 4)) return false;
  if ((r + 2) * (a.w + 2) * (a.cin * es / 16) > ig::kRowsFill * 256) return false;
  return ig::rows_lds_bytes(bc, a.ksteps, a.w, a.cin, es) <= 160 * 1024;
}

TileCfg make_rows_tile(const IgemmArgs& a, int bc) {
  TileCfg t = make_tile(a, bc, 4);
  t.kchunk = a.ksteps;
  t.tpw = -2;
  return t;
}

// The wide-tile kernel (tpw = -3): input rows of whole 128-byte units
// (c_in % 128 == 0 int8, % 64 == 0 fp16; 16-byte aligned views), 256-pixel
// workgroups of 64, 128 or 256 channels.
bool wide_ok(const IgemmArgs& a, int bc) {
  const int es = a.epi == EPI_F16 ? 2 : 1;
  if ((a.cin * es) % 128 != 0 || (a.x_pix_stride * es) % 16 != 0 || (a.x_c_off * es) % 16 != 0) return false;
  if (!(bc == 256 || bc == 128 || bc == 64) || a.cout_pad % bc != 0 || a.ksteps % 2 != 0) return false;
  if (bc > 64 && a.cout <= bc / 2) return false;  // half the tile would be padding
  return ig::wide_lds_bytes(bc, a.ksteps) <= 160 * 1024;
}

TileCfg make_wide_tile(const IgemmArgs& a, int bc) {
  TileCfg t = make_tile(a, std::min(bc, 128), 4);
  t.bc = bc;
  t.kchunk = a.ksteps;
  t.tpw = -3;
  return t;
}

// The band-tile kernel (tpw = -4: 8 waves, -5: 16 waves; pb = its band
// height R): 3x3, stride 1 or 2 on both axes, padding 1 (the output map
// (h - 1) / s + 1 by (w - 1) / s + 1), R whole output rows (R divides the
// output height) of at least one 16-pixel block per wave, the input tile
// within the start-up loads, everything within LDS.
int band_waves(int tpw) { return tpw == -5 ? 16 : 8; }

bool band_ok(const IgemmArgs& a, int bc, int rows, int tpw = -4) {
  const int es = a.epi == EPI_F16 ? 2 : 1;
  const int nw = band_waves(tpw);
  const int s = a.sh;
  // DW_BAND_S2=0: no stride-2 band tiles (plan comparisons)
  static const bool s2_on = !(getenv("DW_BAND_S2") && atoi(getenv("DW_BAND_S2")) == 0);
  if (a.kh != 3 || a.kw != 3 || !(s == 1 || (s == 2 && s2_on)) || a.sw != s || a.pt != 1 || a.pl != 1) return false;
  if (a.h <= 0 || a.w <= 0 || a.ho != (a.h - 1) / s + 1 || a.wo != (a.w - 1) / s + 1) return false;
  if ((a.cin * es) % 16 != 0) return false;
  if (!(bc == 128 || bc == 80 || bc == 64 || bc == 32 || bc == 16) || a.cout_pad % bc != 0) return false;
  // 16 waves over 64 channels: only the u8 requantize and table epilogues
  // without a residual fit 128 VGPRs
  if (nw == 16 && bc > 64 && !(es == 1 && a.epi == EPI_QU8 && !a.res && !a.h_wfrag)) return false;
  if (rows < 1 || a.ho % rows != 0 || rows * a.wo < 16 * nw) return false;
  const int cu = a.cin * es / 16;
  if ((long)ig::band_tile_rows(rows, s) * ig::band_tile_w(a.wo, s) * cu > ig::kBandFill * 512) return false;
  return ig::band_lds_bytes(bc, a.ksteps, rows, a.wo, cu, nw, s) <= 160 * 1024;
}

TileCfg make_band_tile(const IgemmArgs& a, int bc, int rows, int tpw = -4) {
  TileCfg t = make_tile(a, bc, 4);
  t.pb = rows;
  t.kchunk = a.ksteps;
  t.tpw = tpw;
  return t;
}

// Band heights worth timing for a channel tile and wave count: those that
// give between 96 and 768 workgroups (about one a CU up to three), at most 5.
int band_heights(const IgemmArgs& a, int bc, int tpw, int* rows, int max) {
  int n = 0;
  for (int r = 1; r <= a.ho && n < max; ++r) {
    if (!band_ok(a, bc, r, tpw)) continue;
    const long wgs = (long)a.n * (a.ho / r) * (a.cout_pad / bc);
    if (wgs >= 96 && wgs <= 768) rows[n++] = r;
  }
  return n;
}

// The split-K kernel (tpw = -6; pb = its waves): int8, 16 or 32 channels, at
// least a k-step for every wave.
bool ks_ok(const IgemmArgs& a, int bc, int waves) {
  return a.epi != EPI_F16 && !a.h_wfrag && (bc == 16 || bc == 32) && a.cout_pad % bc == 0 &&
         (waves == 4 || waves == 8 || waves == 16) && a.ksteps >= waves;
}

// 16-pixel tiles that are few: at most four workgroups a CU.
bool ks_few(const IgemmArgs& a, int bc) { return (long)((a.m + 15) / 16) * (a.cout_pad / bc) <= 1024; }

TileCfg make_ks_tile(const IgemmArgs& a, int bc, int waves) {
  TileCfg t = make_tile(a, bc, 1);
  t.pb = waves;
  t.tpw = -6;
  return t;
}

// The in-order fp16 kernel (tpw = -7): 16, 32 or 64 channels of 16 pixels, taps
// of whole k-steps.
bool fp_ok(const IgemmArgs& a, int bc) {
  return a.epi == EPI_F16 && !a.h_wfrag && (bc == 16 || bc == 32 || bc == 64) && a.cout_pad % bc == 0 &&
         a.cin % 32 == 0 && a.ksteps == a.kh * a.kw * (a.cin / 32);
}

// Its tiles that are few: at most a wave a SIMD.
bool fp_few(const IgemmArgs& a, int bc) { return (long)((a.m + 15) / 16) * (a.cout_pad / bc) <= 1024; }

TileCfg make_fp_tile(const IgemmArgs& a, int bc) {
  TileCfg t = make_tile(a, bc, 1);
  t.tpw = -7;
  return t;
}

// A detect head's 1x1 fused into the epilogue (a.h_wfrag): one tile holds
// every channel (64 or 80) on the staged kernel (with room for the regroup
// rows in its weight chunk), the row-tile or the band-tile kernel.
bool head_tile_ok(const IgemmArgs& a, const TileCfg& t) {
  if (!(t.bc == 64 || t.bc == 80) || a.cout_pad != t.bc) return false;
  if (t.tpw == -2) return rows_ok(a, t.bc);
  if (t.tpw == -4) return band_ok(a, t.bc, t.pb);
  return t.tpw == 0 && tile_ok(a, t.bc, t.pb) && t.kchunk * t.bc * 64 >= ig::xpose_bytes(t.bc);
}

// Microseconds that a launch of the staged (fam 0), streamed-weight (1) or
// wide-tile (2) kernel is expected to take, for launches that no tuner timed
// (the op functions): a sum of what one workgroup cannot overlap (start-up, a
// latency per k-step, the epilogue of its tile) and of what a CU's share of
// the workgroups costs in matrix instructions, im2col loads, weight reads and
// epilogues per k-step, with the share both as the mean (tiles / 256) and as
// the busiest CU's whole tiles.  The coefficients are a non-negative least
// squares fit (relative error 8-12%) to the timings of 475 int8 and 337 fp16
// convolutions with 1-32 images of 7-160 rows and columns, 16-512 input and
// 16-1000 output channels, 1x1 and 3x3, strides 1 and 2.  Choosing among up to
// 50 tiles is host time of every untimed launch, so the arguments are what
// the candidates share: 0.3 us (0.9-2.2 us with each tile laid out first).
float tile_cost(int esize, int fam, int ksteps, int bc, int pb, int wgs) {
  static const float kFit[2][3][15] = {
      {{3.254f, 0.1118f, 0.003944f, 0.01639f, 0.002887f, 0.04835f, 0.08821f, 0.002636f, 0.0154f, 0, 0.01487f,
        0.002478f, 0.01127f, 0.01528f, 0.08366f},
       {3.93f, 0.08103f, 0, 0.01531f, 0, 0.06327f, 0.5737f, 0.002326f, 0, 0, 0, 0.0008586f, 0.04129f, 0.01257f,
        0.1047f},
       {3.394f, 0, 0, 0, 0, 0, 1.221f, 0.00399f, 0, 0, 0, 0.006569f, 0.05407f, 0, 0.08989f}},
      {{3.626f, 0.07469f, 0.005534f, 0, 0.003169f, 0.01053f, 0.0151f, 0.001067f, 0.01693f, 0, 0.06502f,
        0.004994f, 0.02329f, 0.01432f, 0.03708f},
       {3.885f, 0.0769f, 0, 0, 0, 0, 0.5448f, 0.002746f, 0.009312f, 0, 0, 0.003492f, 0.03948f, 0.01009f, 0.1019f},
       {3.033f, 0, 0, 0, 0, 0, 1.406f, 0.002105f, 0, 0, 0.04805f, 0.008186f, 0.03759f, 0, 0.05602f}}};
  const float ks = (float)ksteps, b = (float)bc / 16.0f, p = (float)pb;
  const float kb = ks * b, kp = ks * p, bp = b * p, kbp = kb * p;
  const float mean = (float)wgs * (1.0f / 256.0f), full = (float)((wgs + 255) >> 8);
  const float* c = kFit[esize == 1 ? 0 : 1][fam];
  const float one = (c[0] + c[1] * ks) + (c[2] * kb + c[3] * kp) + (c[4] * kbp + c[5] * bp);
  const float share = c[6] + (c[7] * kbp + c[8] * kp) + (c[9] * kb + c[10] * bp);
  const float busiest = (c[11] * kbp + c[12] * kp) + (c[13] * kb + c[14] * bp);
  return one + mean * share + full * busiest;
}

// The same for the split-K kernel of `waves` waves (fit to 493 timings, 6%):
// its batches of loads, and the busiest CU's waves and batches.
float ks_cost(const IgemmArgs& a, int bc, int waves, int wgs) {
  const float mean = (float)wgs / 256.0f, full = (float)((wgs + 255) / 256), nw = (float)waves;
  const int per = (a.ksteps + waves - 1) / waves;
  const float batches = (float)((per + ig::kKsAhead - 1) / ig::kKsAhead);
  return 2.907f + 0.0054f * nw + 0.619f * batches + 0.01647f * mean * (float)a.ksteps * ((float)bc / 16.0f) +
         full * (0.05115f * batches + 0.0971f * nw);
}

// The same for the in-order fp16 kernel (fit to 63 timings, 10%): its chain of
// k-steps, shorter where up to four share their addresses, and the CUs' loads.
float fp_cost(const IgemmArgs& a, int bc, int waves) {
  const float mean = (float)waves / 256.0f, full = (float)((waves + 255) / 256);
  const float ks = (float)a.ksteps, cb = (float)bc / 16.0f, shared = a.cin % 128 == 0 ? 4.0f : a.cin % 64 == 0 ? 2.0f : 1.0f;
  return 3.367f + 0.0554f * ks / shared + mean * (0.4539f + 0.0518f * cb + 0.01781f * ks) + 0.01207f * full * ks * cb;
}

// Tile shape for a problem: an override from DW_IGEMM_TILE (tests and
// tuning runs), an explicit choice (a.tile_bc / a.tile_pb, set by the graph
// runtime's tuner), else the tile that tile_cost expects to be fastest.  The
// weight slice of the channel tile is staged in chunks of at most kWeightLds
// bytes.
TileCfg pick_any(const IgemmArgs& a);
struct TilePick {
  int bc, pb, tpw;
};

// A launch that also writes an upsampled copy (a.y_up) takes any tile whose
// epilogue is igemm_store's; the persistent small-K kernel's is its own, so
// its tiles become the staged kernel's of the same shape.
TileCfg pick(const IgemmArgs& a) {
  TileCfg t = pick_any(a);
  if (a.y_up && t.tpw > 0) t = make_tile(a, t.bc, t.pb);
  return t;
}

TileCfg pick_any(const IgemmArgs& a) {
  if (a.h_wfrag) {
    // a DW_IGEMM_TILE row- or band-tile override, else the tuner's choice
    // when it is a head tile, else the staged kernel with the widest pixel
    // tile that fits
    if (const char* env = getenv("DW_IGEMM_TILE")) {
      int v0 = 0, v1 = 0, v2 = 0;
      if (sscanf(env, "%d,%d,%d", &v0, &v1, &v2) == 3 && (v2 == -2 || v2 == -4)) {
        const TileCfg t = v2 == -2 ? make_rows_tile(a, v0) : make_band_tile(a, v0, v1);
        if (head_tile_ok(a, t)) return t;
      }
    }
    if (a.tile_bc) {
      const TileCfg t = a.tile_tpw == -2   ? make_rows_tile(a, a.tile_bc)
                        : a.tile_tpw == -4 ? make_band_tile(a, a.tile_bc, a.tile_pb)
                                           : make_tile(a, a.tile_bc, a.tile_pb);
      if (head_tile_ok(a, t)) return t;
    }
    for (int pb : {4, 2, 1}) {
      const TileCfg t = make_tile(a, a.cout_pad, pb);
      if (head_tile_ok(a, t)) return t;
    }
    return make_tile(a, a.cout_pad, 1);  // launch_igemm refuses it
  }
  if (const char* env = getenv("DW_IGEMM_TILE")) {
    int v0 = 0, v1 = 0, v2 = 0;
    const int nv = sscanf(env, "%d,%d,%d", &v0, &v1, &v2);
    if (nv == 3 && sk_ok(a, v0, v1, v2)) return make_sk_tile(a, v0, v1, v2);
    if (nv == 3 && v2 == -1 && st_ok(a, v0, v1)) return make_st_tile(a, v0, v1);
    if (nv == 3 && v2 == -2 && rows_ok(a, v0)) return make_rows_tile(a, v0);
    if (nv == 3 && v2 == -3 && wide_ok(a, v0)) return make_wide_tile(a, v0);
    if (nv == 3 && (v2 == -4 || v2 == -5) && band_ok(a, v0, v1, v2)) return make_band_tile(a, v0, v1, v2);
    if (nv == 3 && v2 == -6 && ks_ok(a, v0, v1)) return make_ks_tile(a, v0, v1);
    if (nv == 3 && v2 == -7 && fp_ok(a, v0)) return make_fp_tile(a, v0);
    if (nv >= 2 && tile_ok(a, v0, v1)) return make_tile(a, v0, v1);
    if (nv == 1 && tile_ok(a, channel_tile(a.cout), v0)) return make_tile(a, channel_tile(a.cout), v0);
  }
  if (a.tile_bc && sk_ok(a, a.tile_bc, a.tile_pb, a.tile_tpw)) return make_sk_tile(a, a.tile_bc, a.tile_pb, a.tile_tpw);
  if (a.tile_bc && a.tile_tpw == -1 && st_ok(a, a.tile_bc, a.tile_pb)) return make_st_tile(a, a.tile_bc, a.tile_pb);
  if (a.tile_bc && a.tile_tpw == -2 && rows_ok(a, a.tile_bc)) return make_rows_tile(a, a.tile_bc);
  if (a.tile_bc && a.tile_tpw == -3 && wide_ok(a, a.tile_bc)) return make_wide_tile(a, a.tile_bc);
  if (a.tile_bc && (a.tile_tpw == -4 || a.tile_tpw == -5) && band_ok(a, a.tile_bc, a.tile_pb, a.tile_tpw))
    return make_band_tile(a, a.tile_bc, a.tile_pb, a.tile_tpw);
  if (a.tile_bc && a.tile_tpw == -6 && ks_ok(a, a.tile_bc, a.tile_pb)) return make_ks_tile(a, a.tile_bc, a.tile_pb);
  if (a.tile_bc && a.tile_tpw == -7 && fp_ok(a, a.tile_bc)) return make_fp_tile(a, a.tile_bc);
  if (a.tile_bc && tile_ok(a, a.tile_bc, a.tile_pb)) return make_tile(a, a.tile_bc, a.tile_pb);
  // The widest channel tile and the widest pixel tile (16 * pb pixels per
  // wave) that still gives about two workgroups per CU reads the input least
  // often, but leaves CUs idle on small maps and makes long workgroups of
  // deep layers; it stays unless another tile is expected to take clearly less
  // (how clearly stands below).  On 5000 convolutions kept out of the fits
  // (those above and 5x5, up to 720 channels) the choice is 1.22x faster
  // (geometric mean), 0.5% of them are more than 3% slower, the worst 14%; with
  // 95% of its time enough for every tile that was 2.3%, the worst 36%.  20 x
  // 20, 256 -> 256 3x3, one image: 15.8 -> 9.2 us.
  const int bc = channel_tile(a.cout);
  const int ctiles = a.cout_pad / bc;
  TileCfg best = make_tile(a, bc, 1);
  for (int pb : {4, 2, 1}) {
    const long wgs = (long)((a.m + 64 * pb - 1) / (64 * pb)) * ctiles;
    if (wgs >= 512) {
      best = make_tile(a, bc, pb);
      break;
    }
  }
  if (a.y2 || a.y_up) return best;  // the graph runtime's fused launches
  const int esize = a.epi == EPI_F16 ? 2 : 1;
  // 64 PB-pixel tiles: (m + 64 PB - 1) / (64 PB) for PB = 1, 2, 4
  auto pixel_tiles = [&](int pb) { return (a.m + 64 * pb - 1) >> (pb == 4 ? 8 : pb == 2 ? 7 : 6); };
  const float base = tile_cost(esize, 0, a.ksteps, best.bc, best.pb, pixel_tiles(best.pb) * ctiles);
  float least = 0.95f * base;
  TilePick f{};
  auto consider = [&](float c, int b, int p, int tpw) {
    if (c < least) {
      least = c;
      f = {b, p, tpw};
    }
  };
  for (int b : {128, 96, 80, 64, 48, 32, 16}) {
    if (b > bc || a.cout_pad % b != 0) continue;  // tile_ok, for each pixel tile
    const int ct = a.cout_pad / b;
    for (int p : {4, 2, 1}) {
      const int wgs = pixel_tiles(p) * ct;
      consider(tile_cost(esize, 0, a.ksteps, b, p, wgs), b, p, 0);
      if (a.ksteps >= 2 && ig::st_lds_bytes(b, a.ksteps, ring_depth(p)) <= 160 * 1024)  // st_ok
        consider(tile_cost(esize, 1, a.ksteps, b, p, wgs), b, p, -1);
    }
  }
  for (int b : {256, 128, 64})
    if (wide_ok(a, b)) consider(tile_cost(esize, 2, a.ksteps, b, 4, pixel_tiles(4) * (a.cout_pad / b)), b, 4, -3);
  // A tile of 64 pixels in place of one, or the wide kernel's, is believed at 95%
  // (at 85 to 95% 1% of 690 such choices were more than 3% slower); one of more
  // pixels, or of fewer than the first's, is not (22% of 430), the streamed
  // kernel's least; and K beyond the fits, which end at 512 channels of 3x3,
  // counts for less.
  const bool deep = a.ksteps > (esize == 1 ? 72 : 144);
  const bool near = f.tpw == -3 || (f.pb == 1 && best.pb == 1);
  const float enough = deep ? 0.7f : near ? 0.95f : f.tpw == -1 ? 0.8f : 0.85f;
  if (f.bc && least >= enough * base) {
    least = 0.95f * base;
    f = {};
  }
  // Tiles of 16 pixels where they are few, against 95% of the best above
  // (least when nothing above was chosen is that already).
  // Split K (int8: a sum of integers is the same in any order; fp16 layers
  // keep one order for every plan): a fifth of the int8 layers above, those
  // 1.30x faster, and the best tile 4.6% away instead of 11%.  20 x 20, 256 ->
  // 256 3x3, one image: 9.2 -> 5.5 us.
  // In order (fp16): half of 29 layers of up to 1024 such waves, those 1.37x
  // faster; below four k-steps there is no chain to shorten (7 x 21 96 -> 92
  // 1x1 of 5 images: 4.8 against 3.9 us).
  if (f.bc) least *= 0.95f;
  if (deep) least = std::min(least, 0.7f * base);
  const int p16 = (a.m + 15) >> 4;
  for (int b : {16, 32, 64}) {
    if (a.cout_pad % b != 0) continue;
    const long tiles = (long)p16 * (a.cout_pad / b);
    if (tiles > 1024) continue;  // ks_few, fp_few
    if (esize == 2) {
      if (a.ksteps >= 4 && fp_ok(a, b)) consider(fp_cost(a, b, (int)tiles), b, 1, -7);
    } else {
      for (int nw : {4, 8, 16})
        if (ks_ok(a, b, nw))  // (four workgroups a CU are short of loads: up to 18% slower than expected to win by 25%)
          consider(ks_cost(a, b, nw, (int)tiles) * (tiles > 768 ? 1.3f : 1.0f), b, nw, -6);
    }
  }
  if (!f.bc) return best;
  return f.tpw == 0    ? make_tile(a, f.bc, f.pb)
         : f.tpw == -1 ? make_st_tile(a, f.bc, f.pb)
         : f.tpw == -3 ? make_wide_tile(a, f.bc)
         : f.tpw == -6 ? make_ks_tile(a, f.bc, f.pb)
                       : make_fp_tile(a, f.bc);
}

// Epilogue specialisation for the arguments.
int epilogue_variant(const IgemmArgs& a, int esize) {
  if (esize != 1 || a.epi != EPI_QU8) return EPV_GENERIC;
  if (a.h_wfrag) return EPV_QU8_LUT_HEAD;
  if (!a.lut) return a.res ? EPV_GENERIC : EPV_QU8;
  return a.res ? EPV_QU8_LUT_RES : EPV_QU8_LUT;
}

}  // namespace

int igemm_channel_tile(int cout) { return channel_tile(cout); }

bool igemm_sibling_tile_ok(const IgemmArgs& a, int bc, int tpw, int esize) {
  const bool common = !a.res && !a.y_up && !a.h_wfrag && bc > 0 && a.split > 0 && a.split % bc == 0 &&
                      a.split < a.cout && a.y2_pix_stride % 4 == 0 && a.y2_c_off % 4 == 0;
  if (esize == 1)  // the u8 table epilogue (its table staged per channel tile)
    return common && a.epi == EPI_QU8 && a.lut && a.lut2 &&
           (tpw == 0 || tpw == -1 || tpw == -4 || tpw == -5 || tpw == -6);
  // fp16: the store chooses the view per channel tile; every kernel but the
  // persistent small-K one
  return common && esize == 2 && a.epi == EPI_F16 && tpw <= 0;
}

int igemm_candidates(const IgemmArgs& a, int* bc, int* pb, int* tpw, int max) {
  int n = 0;
  if (a.h_wfrag) {
    for (int p : {4, 2, 1})
      if (n < max && head_tile_ok(a, make_tile(a, a.cout_pad, p))) {
        bc[n] = a.cout_pad;
        pb[n] = p;
        tpw[n] = 0;
        ++n;
      }
    if (n < max && head_tile_ok(a, make_rows_tile(a, a.cout_pad))) {
      bc[n] = a.cout_pad;
      pb[n] = 4;
      tpw[n] = -2;
      ++n;
    }
    int rows[8];
    const int nr = band_heights(a, a.cout_pad, -4, rows, 8);
    for (int i = 0; i < nr && n < max; ++i)
      if (head_tile_ok(a, make_band_tile(a, a.cout_pad, rows[i]))) {
        bc[n] = a.cout_pad;
        pb[n] = rows[i];
        tpw[n] = -4;
        ++n;
      }
    return n;
  }
  for (int b : {16, 32})
    for (int nw : {4, 8, 16})
      if (n < max && ks_ok(a, b, nw) && ks_few(a, b)) {
        bc[n] = b;
        pb[n] = nw;
        tpw[n] = -6;
        ++n;
      }
  for (int b : {16, 32, 64})
    if (n < max && fp_ok(a, b) && fp_few(a, b)) {
      bc[n] = b;
      pb[n] = 1;
      tpw[n] = -7;
      ++n;
    }
  // band tiles (8 and 16 waves): the widest channel tile, and 64 or 80
  // channels when that splits a wider layer in two or more (80: a sibling
  // GEMM whose first conv has 80 channels)
  {
    const int bw = std::min(a.cout_pad, 128);
    for (int tw : {-4, -5})
      for (int j = 0; j < 3; ++j) {
        const int b = j == 0 ? bw : (j == 1 ? 64 : 80);
        if (j > 0 && (bw <= b || a.cout_pad % b != 0)) continue;
        int rows[8];
        const int nr = band_heights(a, b, tw, rows, 8);
        for (int i = 0; i < nr && n < max; ++i) {
          bc[n] = b;
          pb[n] = rows[i];
          tpw[n] = tw;
          ++n;
        }
      }
  }
  for (int b : {256, 128, 64})
    if (n < max && wide_ok(a, b)) {
      bc[n] = b;
      pb[n] = 4;
      tpw[n] = -3;
      ++n;
    }
  for (int b : {128, 96, 80, 64, 48, 32, 16})
    for (int p : {4, 2, 1}) {
      if (n < max && tile_ok(a, b, p)) {
        bc[n] = b;
        pb[n] = p;
        tpw[n] = 0;
        ++n;
      }
      if (n < max && st_ok(a, b, p)) {
        bc[n] = b;
        pb[n] = p;
        tpw[n] = -1;
        ++n;
      }
      if (n < max && p == 4 && rows_ok(a, b)) {
        bc[n] = b;
        pb[n] = p;
        tpw[n] = -2;
        ++n;
      }
      // persistent variants that still leave a workgroup for every CU
      const long tiles = (long)((a.m + 64 * p - 1) / (64 * p)) * (a.cout_pad / std::max(b, 1));
      for (int t : {2, 4, 8})
        if (n < max && sk_ok(a, b, p, t) && tiles / t >= 256) {
          bc[n] = b;
          pb[n] = p;
          tpw[n] = t;
          ++n;
        }
    }
  return n;
}

const char* igemm_tile_name(const IgemmArgs& a, int esize) {
  static thread_local char buf[64];
  const TileCfg t = pick(a);
  if (t.tpw > 0)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_p%d_t%d", esize == 1 ? "i8" : "f16", t.bc, 64 * t.pb, t.tpw);
  else if (t.tpw == -1)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_p%d_st", esize == 1 ? "i8" : "f16", t.bc, 64 * t.pb);
  else if (t.tpw == -2)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_rows", esize == 1 ? "i8" : "f16", t.bc);
  else if (t.tpw == -3)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_wide", esize == 1 ? "i8" : "f16", t.bc);
  else if (t.tpw == -4)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_band%d", esize == 1 ? "i8" : "f16", t.bc, t.pb);
  else if (t.tpw == -5)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_band%dw16", esize == 1 ? "i8" : "f16", t.bc, t.pb);
  else if (t.tpw == -6)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_ks%d", esize == 1 ? "i8" : "f16", t.bc, t.pb);
  else if (t.tpw == -7)
    snprintf(buf, sizeof buf, "igemm_%s_c%d_fp", esize == 1 ? "i8" : "f16", t.bc);
  else
    snprintf(buf, sizeof buf, "igemm_%s_c%d_p%d", esize == 1 ? "i8" : "f16", t.bc, 64 * t.pb);
  if (a.h_wfrag) strncat(buf, "_head", sizeof buf - strlen(buf) - 1);
  if (a.y_up) strncat(buf, "_up", sizeof buf - strlen(buf) - 1);
  if (a.y2) strncat(buf, "_sib", sizeof buf - strlen(buf) - 1);
  return buf;
}

void launch_igemm(hipStream_t st, const IgemmArgs& a_in, int esize) {
  const TileCfg t = pick(a_in);
  if (a_in.cout_pad % t.bc != 0) fail(-4, "igemm: cout_pad not a multiple of the channel tile");
  if (a_in.m >= (1 << 24)) fail(-2, "igemm: more than 2^24 output pixels in one launch");
  if (a_in.kh * a_in.kw > 31) fail(-2, "igemm: more than 31 filter taps");
  IgemmArgs a = a_in;
  a.kchunk = t.kchunk;
  const long long xb = (long long)a.n * a.h * a.w * a.x_pix_stride * esize;
  if (xb >= (1ll << 31)) fail(-2, "igemm: input view larger than 2 GB");
  a.x_bytes = (int)xb;
  const size_t lds = t.tpw > 0     ? ig::sk_lds_bytes(t.bc, a.ksteps)
                     : t.tpw == -1 ? ig::st_lds_bytes(t.bc, a.ksteps, t.pd)
                     : t.tpw == -2 ? ig::rows_lds_bytes(t.bc, a.ksteps, a.w, a.cin, esize)
                     : t.tpw == -3 ? ig::wide_lds_bytes(t.bc, a.ksteps)
                     : t.tpw == -4 || t.tpw == -5
                         ? ig::band_lds_bytes(t.bc, a.ksteps, t.pb, a.wo, a.cin * esize / 16, band_waves(t.tpw), a.sh)
                     : t.tpw <= -6 ? 0
                                   : ig::lds_bytes(t, a.ksteps);
  if (lds > 160 * 1024) fail(-2, "igemm: k-slice table does not fit LDS");
  if ((long long)a.ho * a.wo >= (1ll << 23)) fail(-2, "igemm: more than 2^23 output pixels per image");
  if ((long long)a.ksteps * a.cout_pad * 64 >= (1ll << 32)) fail(-2, "igemm: packed weights larger than 4 GB");
  a.r_cin = 1.0f / (float)a.cin;
  a.r_kw = 1.0f / (float)a.kw;
  a.r_hwo = 1.0f / (float)(a.ho * a.wo);
  a.r_wo = 1.0f / (float)a.wo;
  // u8 output and residual views, addressed by the persistent kernel's
  // buffer stores and loads
  const long long yb = a.epi == EPI_QU8 ? (long long)a.m * a.y_pix_stride : 0;
  const long long rb = a.epi == EPI_QU8 && a.res ? (long long)a.m * a.r_pix_stride : 0;
  if (yb >= (1ll << 31) || rb >= (1ll << 31)) fail(-2, "igemm: output view larger than 2 GB");
  a.y_bytes = (int)yb;
  a.r_bytes = (int)rb;
  a.tile_tpw = t.tpw;
  a.band_rows = t.tpw == -4 || t.tpw == -5 ? t.pb : 0;
  if (a.y_up && (esize == 1 ? (a.epi != EPI_QU8 || a.h_wfrag || (a.res && !a.lut) || a.up_pix_stride % 4 != 0 ||
                                a.up_c_off % 4 != 0)
                             : (a.epi != EPI_F16 || a.up_pix_stride % 4 != 0 || a.up_c_off % 4 != 0)))
    fail(-2, "igemm: an upsampled copy needs a u8 table, requantize or f16 epilogue and aligned views");
  // a sibling GEMM: a kernel whose workgroup keeps one channel tile and
  // stores through igemm_store (staged, streamed-weight, band), the table
  // epilogue, and tiles that do not straddle the split
  if (a.y2 && !igemm_sibling_tile_ok(a, t.bc, t.tpw, esize))
    fail(-2, "igemm: a sibling GEMM needs the table epilogue and a staged, streamed or band tile within one conv");
  bool ok;
  if (esize == 1 && a.h_wfrag) {
    if (a.epi != EPI_QU8 || !a.lut || a.res || !head_tile_ok(a, t))
      fail(-2, "igemm: the fused head 1x1 needs a table epilogue and a tile of every channel");
    ok = igemm_launch_head_i8(st, a, t);
  } else if (esize == 1) {
    const int epv = epilogue_variant(a, esize);
    const bool ab = epv == EPV_GENERIC || epv == EPV_QU8;
    if (t.tpw > 0)
      ok = ab ? igemm_launch_sk_i8_a(st, a, t, epv) : igemm_launch_sk_i8_b(st, a, t, epv);
    else if (t.tpw == -1)
      ok = ab ? igemm_launch_st_i8_a(st, a, t, epv) : igemm_launch_st_i8_b(st, a, t, epv);
    else if (t.tpw == -2)
      ok = ab ? igemm_launch_rows_i8_a(st, a, t, epv) : igemm_launch_rows_i8_b(st, a, t, epv);
    else if (t.tpw == -3)
      ok = ab ? igemm_launch_wide_i8_a(st, a, t, epv) : igemm_launch_wide_i8_b(st, a, t, epv);
    else if (t.tpw == -4 || t.tpw == -5)
      ok = ab ? igemm_launch_band_i8_a(st, a, t, epv) : igemm_launch_band_i8_b(st, a, t, epv);
    else if (t.tpw == -6)
      ok = igemm_launch_ks_i8(st, a, t);
    else
      ok = ab ? igemm_launch_i8_a(st, a, t, epv) : igemm_launch_i8_b(st, a, t, epv);
  } else {
    ok = t.tpw > 0     ? igemm_launch_sk_f16(st, a, t)
         : t.tpw == -1 ? igemm_launch_st_f16(st, a, t)
         : t.tpw == -2 ? igemm_launch_rows_f16(st, a, t)
         : t.tpw == -3 ? igemm_launch_wide_f16(st, a, t)
         : t.tpw == -7 ? igemm_launch_fp_f16(st, a, t)
         : t.tpw == -4 || t.tpw == -5 ? igemm_launch_band_f16(st, a, t)
                       : igemm_launch_f16(st, a, t);
  }
  if (!ok) fail(-2, "igemm: no kernel for tile");
  DW_HIP(hipGetLastError());
}

void launch_pack_weights(hipStream_t st, const void* w_hwio, void* wpk, int K, int cout,
                         int cout_pad, int ksteps, int esize) {
  if (cout % 4 != 0 || cout_pad % 16 != 0) fail(-4, "pack_weights: c_out must be a multiple of 4, its padding of 16");
  // no sums to complete: the k-steps spread over the grid, four to a workgroup
  const dim3 grid((unsigned)(cout_pad / 16), (unsigned)((ksteps + 3) / 4)), block(64 * std::min(ksteps, 4));
  if (esize == 1)
    hipLaunchKernelGGL(pack_weights_kernel<1>, grid, block, 0, st, (const uint8_t*)w_hwio, (uint8_t*)wpk, K, cout,
                       cout_pad, ksteps);
  else
    hipLaunchKernelGGL(pack_weights_kernel<2>, grid, block, 0, st, (const uint8_t*)w_hwio, (uint8_t*)wpk, K, cout,
                       cout_pad, ksteps);
  DW_HIP(hipGetLastError());
}

void launch_qconv_prep(hipStream_t st, const void* w_hwio, void* wpk, const int* bias, int* bias_out, float* ms_out,
                       const float* m_host, int K, int cout, int cout_pad, int ksteps, int corr) {
  if (cout % 4 != 0 || cout_pad % 16 != 0) fail(-4, "qconv_prep: c_out must be a multiple of 4, its padding of 16");
  const bool sum = corr != 0;
  const dim3 block(64 * std::min(ksteps, sum ? 16 : 4));
  const unsigned rows = sum ? 1 : (unsigned)((ksteps + 3) / 4);
  // a launch holds the multipliers of kPrepChannels channels; the last one
  // also packs the padding channels, which have none
  for (int c0 = 0; c0 < cout; c0 += kPrepChannels) {
    PrepScales m;
    memcpy(m.m, m_host + c0, sizeof(float) * std::min(kPrepChannels, cout - c0));
    const QconvPrep q{bias, bias_out, ms_out, corr, c0};
    const int groups = (c0 + kPrepChannels < cout ? kPrepChannels : cout_pad - c0) / 16;
    hipLaunchKernelGGL(sum ? qconv_prep_kernel<true> : qconv_prep_kernel<false>, dim3(groups, rows), block, 0, st,
                       (const uint8_t*)w_hwio, (uint8_t*)wpk, K, cout, cout_pad, ksteps, q, m);
  }
  DW_HIP(hipGetLastError());
}

}  // namespace dw
