// fp32 convolution in the reference's accumulation order, any shape: per
// output acc = 0; for kh, for kw (taps outside the image skipped), for ic:
// acc = fma(x, w, acc) (crates/dragonwing-cpu/src/ops.rs:1356-1436), then the
// bias pass and the activation.  The chains allow no matrix instruction and
// no split of K, so the kernel is a register-tiled product on the vector
// ALUs: K runs in the chains' order and only outputs are parallel.
//
// A workgroup of 256 threads owns 32 PX output pixels x 8 CH channels.  K is
// walked in chunks of at most KC values that never mix parts of taps: whole
// taps (c_in <= KC; as many as fit) or KC channels of one tap.  A chunk's
// im2col values and weights go to LDS with K innermost, in two buffers, the
// next chunk's loads in flight while the current one is summed.  A thread
// holds PX x CH chains and reads 16 bytes (4 steps of K) of each of its
// pixels and channels at a time: PX + CH reads feed 4 PX CH FMAs.  The row
// stride KC + 4 puts the 8 pixels (or channels) that a wave reads together
// on different banks.
//
// A tap outside a pixel's image must leave its chains alone (its weights may
// be infinite): they are kept and put back after the tap, in tiles that have
// such a pixel.
//
// Bound by the FMA rate where there are many pixels (16 x 80 x 80, 64 -> 64
// 3x3, 7.5 GFLOP: 140 us, 54 TFLOP/s, against 280 us for the 16 x 16 LDS
// window kernel), by the latency of the chunks where there are few (2 x 53 x
// 75 x 48 -> 40: 18 us, against 27.4 us for a thread per pixel reading global
// memory at the pixel stride; 1 x 18 x 50 x 78 -> 171: 22 against 148 us).
#include "direct_util.h"

#include <algorithm>
#include <type_traits>

namespace dw {
namespace {

struct CfArgs {
  const float* x;
  const float* w;  // HWIO
  const float* bias;
  float* y;
  int n, h, wd, cin, cout, kh, kw, sh, sw, pt, pl, ho, wo, m;
  int xs, ys;      // pixel strides
  int seg, segp;   // channels of a segment (a tap's part of a chunk), rounded up to 4
  int taps_chunk;  // segments in a chunk
  int segs_tap;    // segments of a tap (1 if whole taps fit)
  int chunks;
  int wtap, wrow;  // rows of the weights between two taps, and more between two rows of taps
  int act;
  int x_bytes, w_bytes;
};

// Steps of K in a chunk of a tile with px pixels a thread, and the whole taps
// that it holds (0: a tap takes several chunks).
__host__ __device__ constexpr int cf_k(int px) { return px == 4 ? 32 : px == 2 ? 64 : 128; }
int cf_taps(int cin, int taps, int px) { return cin <= cf_k(px) ? std::min(taps, cf_k(px) / ((cin + 3) & ~3)) : 0; }
int cf_chunks(int cin, int taps, int px) {
  const int t = cf_taps(cin, taps, px);
  return t ? (taps + t - 1) / t : taps * ((cin + cf_k(px) - 1) / cf_k(px));
}

template <int PX, int CH, bool VEC>
struct CfTile {
  static constexpr int kK = cf_k(PX);
  static constexpr int kLd = kK + 4;
  static constexpr int kPix = 32 * PX, kCh = 8 * CH;
  static constexpr int kV = VEC ? 4 : 1;             // input values of one load
  static constexpr int kRows = 256 * kV / kK;        // pixels that the workgroup loads at a time
  static constexpr int kXLoads = kPix / kRows, kWLoads = kCh * kK / 256;
  // waves a SIMD that the registers are to allow
  static constexpr int kWaves = PX * CH <= 5 ? 4 : PX * CH <= 10 ? 3 : 2;
};

// VEC: c_in % 4 == 0 and 16-byte aligned pixels, so the input comes in four
// channels at a time.  CUT: columns of the filter are left out between its rows
// (a test of it a chunk costs the other layers 1%).
template <int PX, int CH, bool VEC, bool CUT>
__global__ __launch_bounds__(256, (CfTile<PX, CH, VEC>::kWaves)) void conv_f32_kernel(const CfArgs a) {
  using T = CfTile<PX, CH, VEC>;
  constexpr int K = T::kK, LD = T::kLd, V = T::kV;
  using XV = std::conditional_t<VEC, float4, float>;
  __shared__ __align__(16) float sx[2][T::kPix * LD];
  __shared__ __align__(16) float sw[2][T::kCh * LD];
  __shared__ int4 pix[T::kPix];  // element offset of the window's corner, its row and column
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int p0 = blockIdx.x * T::kPix, c0 = blockIdx.y * T::kCh;
  const int taps = a.kh * a.kw;
  bool out = false;
  if (t < T::kPix) {
    const int p = min(p0 + t, a.m - 1);  // past the end: the last pixel again, not stored
    const int hw = a.ho * a.wo, nn = p / hw, r = p - nn * hw, oh = r / a.wo, ow = r - oh * a.wo;
    const int ih = oh * a.sh - a.pt, iw = ow * a.sw - a.pl;
    pix[t] = make_int4(((nn * a.h + ih) * a.wd + iw) * a.xs, ih, iw, 0);
    out = ih < 0 || iw < 0 || ih + a.kh > a.h || iw + a.kw > a.wd;
  }
  const bool border = __syncthreads_or(out);

  // The thread's part of every chunk's loads: V steps of K of kXLoads
  // pixels, and kWLoads weights with channels across the threads.  Only the
  // address is computed: places outside an image, a row or the channels
  // read whatever lies there (or zero, past the buffers), which no chain
  // reads or keeps.
  const int kk = t % (K / V) * V, prow = t / (K / V);
  const int ktl = kk / a.segp, kic = kk - ktl * a.segp;
  int xo[T::kXLoads], wo[T::kWLoads];
#pragma unroll
  for (int i = 0; i < T::kXLoads; ++i) xo[i] = pix[prow + i * T::kRows].x;
#pragma unroll
  for (int i = 0; i < T::kWLoads; ++i) {
    const int idx = t + 256 * i, k = idx / T::kCh, tl = k / a.segp;
    wo[i] = (tl * a.wtap + k - tl * a.segp) * a.cout + c0 + idx % T::kCh;
  }
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)a.x, (short)0, a.x_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void*)a.w, (short)0, a.w_bytes, 0x00020000);
  XV xv[T::kXLoads];
  float wv[T::kWLoads];
  auto load = [&](int chunk) {
    const int tap0 = a.segs_tap > 1 ? chunk / a.segs_tap : chunk * a.taps_chunk;
    const int ic0 = a.segs_tap > 1 ? (chunk - tap0 * a.segs_tap) * a.seg : 0;
    const int tap = tap0 + ktl;
    const int kh = tap / a.kw, kw = tap - kh * a.kw;
    const int koff = (kh * a.wd + kw) * a.xs + ic0 + kic;
    const int woff = (tap0 * a.wtap + ic0 + (CUT ? tap0 / a.kw * a.wrow : 0)) * a.cout;
#pragma unroll
    for (int i = 0; i < T::kXLoads; ++i) {
      if constexpr (VEC)
        xv[i] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(xr, (xo[i] + koff) * 4, 0, 0));
      else
        xv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, (xo[i] + koff) * 4, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < T::kWLoads; ++i)
      wv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(wr, (wo[i] + woff) * 4, 0, 0));
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int i = 0; i < T::kXLoads; ++i)
      *reinterpret_cast<XV*>(&sx[buf][(prow + i * T::kRows) * LD + kk]) = xv[i];
#pragma unroll
    for (int i = 0; i < T::kWLoads; ++i) {
      const int idx = t + 256 * i;
      sw[buf][(idx % T::kCh) * LD + idx / T::kCh] = wv[i];
    }
  };

  const int pl = lane & 7, cl = lane >> 3, row0 = wave * 8 * PX + pl;  // rows row0 + 8 i, channels cl + 8 j
  int ih0[PX], iw0[PX];
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    ih0[i] = pix[row0 + 8 * i].y;
    iw0[i] = pix[row0 + 8 * i].z;
  }
  float acc[PX][CH] = {};
  int kh = 0, kw = 0, tap = 0, ic = 0;  // of the next segment to sum
  load(0);
  store(0);
  __syncthreads();
  for (int chunk = 0; chunk < a.chunks; ++chunk) {
    const int buf = chunk & 1;
    const bool more = chunk + 1 < a.chunks;
    if (more) load(chunk + 1);
    for (int s = 0; s < a.taps_chunk && tap < taps; ++s) {
      const float* xs = &sx[buf][row0 * LD + s * a.segp];
      const float* ws = &sw[buf][cl * LD + s * a.segp];
      float keep[PX][CH];
      if (border) {
#pragma unroll
        for (int i = 0; i < PX; ++i)
#pragma unroll
          for (int j = 0; j < CH; ++j) keep[i][j] = acc[i][j];
      }
      const int steps = min(a.seg, a.cin - ic);
#pragma unroll 2
      for (int k = 0; k + 4 <= steps; k += 4) {
        float4 xq[PX], wq[CH];
#pragma unroll
        for (int i = 0; i < PX; ++i) xq[i] = *reinterpret_cast<const float4*>(xs + 8 * i * LD + k);
#pragma unroll
        for (int j = 0; j < CH; ++j) wq[j] = *reinterpret_cast<const float4*>(ws + 8 * j * LD + k);
#pragma unroll
        for (int i = 0; i < PX; ++i)
#pragma unroll
          for (int j = 0; j < CH; ++j) {
            acc[i][j] = fmaf(xq[i].x, wq[j].x, acc[i][j]);
            acc[i][j] = fmaf(xq[i].y, wq[j].y, acc[i][j]);
            acc[i][j] = fmaf(xq[i].z, wq[j].z, acc[i][j]);
            acc[i][j] = fmaf(xq[i].w, wq[j].w, acc[i][j]);
          }
      }
      if constexpr (!VEC)
        for (int k = steps & ~3; k < steps; ++k) {
          float x1[PX];
#pragma unroll
          for (int i = 0; i < PX; ++i) x1[i] = xs[8 * i * LD + k];
#pragma unroll
          for (int j = 0; j < CH; ++j) {
            const float w1 = ws[8 * j * LD + k];
#pragma unroll
            for (int i = 0; i < PX; ++i) acc[i][j] = fmaf(x1[i], w1, acc[i][j]);
          }
        }
      if (border) {
#pragma unroll
        for (int i = 0; i < PX; ++i) {
          const bool in = (unsigned)(ih0[i] + kh) < (unsigned)a.h && (unsigned)(iw0[i] + kw) < (unsigned)a.wd;
#pragma unroll
          for (int j = 0; j < CH; ++j) acc[i][j] = in ? acc[i][j] : keep[i][j];
        }
      }
      ic += a.seg;
      if (ic >= a.cin) {
        ic = 0;
        ++tap;
        if (++kw == a.kw) {
          kw = 0;
          ++kh;
        }
      }
    }
    if (more) store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < PX; ++i) {
    const int p = p0 + row0 + 8 * i;
    if (p >= a.m) continue;
    float* y = a.y + (size_t)p * a.ys;
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int ch = c0 + cl + 8 * j;
      if (ch >= a.cout) continue;
      float v = acc[i][j];
      if (a.bias) v = v + a.bias[ch];
      if (a.act == ACT_RELU) {
        v = dx::relu_ref(v);
      } else if (a.act == ACT_SILU) {
        const float sg = 1.0f / (1.0f + expf(-v));
        v = v * sg;
      }
      y[ch] = v;
    }
  }
}

template <int PX, int CH, bool VEC, bool CUT = false>
void launch_tile(hipStream_t st, CfArgs a) {
  using T = CfTile<PX, CH, VEC>;
  const int taps = a.kh * a.kw, whole = cf_taps(a.cin, taps, PX);
  a.seg = whole ? a.cin : T::kK;
  a.segp = (a.seg + 3) & ~3;
  a.taps_chunk = whole ? whole : 1;
  if (CUT)
    while (a.kw % a.taps_chunk) --a.taps_chunk;
  a.segs_tap = whole ? 1 : (a.cin + T::kK - 1) / T::kK;
  a.chunks = whole ? (taps + a.taps_chunk - 1) / a.taps_chunk : taps * a.segs_tap;
  hipLaunchKernelGGL((conv_f32_kernel<PX, CH, VEC, CUT>),
                     dim3((unsigned)((a.m + T::kPix - 1) / T::kPix), (unsigned)((a.cout + T::kCh - 1) / T::kCh)),
                     dim3(256), 0, st, a);
  DW_HIP(hipGetLastError());
}

// The tile that is expected to be done first, in microseconds: what a
// workgroup's chunks and FMAs cost alone, and what the busiest CU's
// workgroups cost its FMAs, LDS reads and barriers.  The coefficients are a
// non-negative least squares fit (14%) to 12 tiles on 33 convolutions of
// 180 to 205k pixels, 3-256 input and 16-256 output channels; the choice
// is 5% off the best tile (geometric mean).  A chunk of K that is a few
// hundred nanoseconds of latency whatever it holds asks for small tiles
// and long chunks on few pixels (20 x 20, 128 -> 128: 18.5 us at 1 x 1
// against 46.7 us at 2 x 4, with a repacking launch that is gone), FMAs per LDS read for large ones on many (16
// x 80 x 80, 64 -> 64: 140 us at 4 x 4 against 243 us at 1 x 2).
bool cf_cut(const DirectArgs& d, const CfWindow& win) { return win.kw > 1 && win.kh > 1 && win.kw < d.kw; }
struct CfChoice {
  int px, ch;
  long long wgs;
};
// Cut filters take tiles of one pixel a thread: their maps are small.
CfChoice cf_choose(const DirectArgs& d, const CfWindow& win) {
  const int taps = win.kh * win.kw;
  CfChoice best{};
  float least = 0;
  const float kt = (float)taps * (float)d.cin / 64.0f;
  for (int p : {1, 2, 4})
    for (int c : {1, 2, 3, 4, 5}) {
      if ((c == 1 || cf_cut(d, win)) && p > 1) continue;
      const long long wgs = (((long long)d.m + 32 * p - 1) / (32 * p)) * ((d.cout + 8 * c - 1) / (8 * c));
      const float mean = (float)wgs / 256.0f, full = (float)((wgs + 255) / 256);
      const float chunks = (float)cf_chunks(d.cin, taps, p), fmas = kt * (float)(p * c);
      const float cost = 0.448f * chunks + 0.103f * fmas +
                         full * (0.0779f * fmas + 0.0043f * kt * (float)(p + c) + 0.242f * chunks) + 0.682f * mean;
      if (!best.px || cost < least) {
        least = cost;
        best = {p, c, wgs};
      }
    }
  return best;
}

// The filter's rows or columns first..last that meet the image of n rows at
// one of the no outputs at least.
struct CfSpan {
  int first, count;
};
CfSpan cf_span(int taps, int n, int no, int stride, int pad) {
  auto met = [&](int k) {
    const int o = std::max(0, (pad - k + stride - 1) / stride);  // the first output whose tap k is not above the image
    return o < no && o * stride - pad + k >= 0 && o * stride - pad + k < n;
  };
  int first = 0, last = taps - 1;
  while (first < last && !met(first)) ++first;
  while (first < last && !met(last)) --last;
  return {first, last - first + 1};
}

}  // namespace

// A small map under a large filter: the taps that no output has in its image
// are cut off (18 maps of one pixel, 47 -> 99 7x7, are a 1x1: 46.9 -> 7 us).
CfWindow conv_f32_window(const DirectArgs& d) {
  const CfSpan r = cf_span(d.kh, d.h, d.ho, d.sh, d.pt), c = cf_span(d.kw, d.w, d.wo, d.sw, d.pl);
  return {r.first, r.count, c.first, c.count};
}

bool conv_f32_reaches(const DirectArgs& d) {
  // 32-bit byte offsets into the input and the weights, also for the windows
  // and chunks that reach past them
  const long long xe = ((long long)d.n * d.h * d.w - 1) * d.x_pix_stride + d.cin;
  const long long we = (long long)d.kh * d.kw * d.cin * d.cout;
  const long long edge = ((long long)(d.pt + d.kh + 64) * d.w + d.pl + d.kw) * d.x_pix_stride + 64;
  const long long wedge = (64ll * d.cin + 128ll * d.kw + 64) * d.cout + d.cout;
  return d.m > 0 && d.cout <= 8 * 65535 && xe + edge < (1ll << 29) && we + wedge < (1ll << 29);
}

// The same kind of sum for layers of up to 24 input or 4 output channels,
// where the tile's per-tap work (a tap is a segment of few steps, kept and put
// back at the borders) and its eight channels a row of threads weigh: a
// robust fit (15%) to 627 of them.
float conv_f32_cost(const DirectArgs& d, const CfWindow& w) {
  const int taps = w.kh * w.kw;
  const CfChoice t = cf_choose(d, w);
  const float chunks = (float)cf_chunks(d.cin, taps, t.px), segs = cf_taps(d.cin, taps, t.px) ? (float)taps : chunks;
  const float kt = (float)taps * (float)d.cin / 64.0f, pc = (float)(t.px * t.ch);
  const float mean = (float)t.wgs / 256.0f, full = (float)((t.wgs + 255) / 256);
  return 3.26f + 0.673f * chunks + 0.0476f * segs + 0.0542f * kt * pc +
         full * (0.0782f * segs + 0.108f * kt * (float)(t.px + t.ch) + 0.0398f * kt * pc) + 0.139f * mean * pc;
}

void launch_conv_f32(hipStream_t st, const DirectArgs& d) {
  if (d.in_kind != 0 || d.out_kind != 0 || !conv_f32_reaches(d)) fail(-4, "conv_f32: not a problem of this kernel");
  const long long xe = ((long long)d.n * d.h * d.w - 1) * d.x_pix_stride + d.cin;
  const long long we = (long long)d.kh * d.kw * d.cin * d.cout;
  const CfWindow win = conv_f32_window(d);
  const long long wc = (long long)d.cin * d.cout, w0 = (win.kh0 * d.kw + win.kw0) * wc;
  CfArgs a{};
  a.x = (const float*)d.x + d.x_c_off;
  a.w = d.wf + w0;
  // one column: its taps are as far apart as rows; several: a chunk stays in a row
  a.wtap = (win.kw == 1 ? d.kw : 1) * d.cin;
  a.wrow = (d.kw - win.kw) * d.cin;
  a.bias = d.bias_f;
  a.y = (float*)d.y + d.y_c_off;
  a.n = d.n; a.h = d.h; a.wd = d.w; a.cin = d.cin; a.cout = d.cout; a.kh = win.kh; a.kw = win.kw;
  a.sh = d.sh; a.sw = d.sw; a.pt = d.pt - win.kh0; a.pl = d.pl - win.kw0; a.ho = d.ho; a.wo = d.wo; a.m = d.m;
  a.xs = d.x_pix_stride;
  a.ys = d.y_pix_stride;
  a.act = d.act;
  a.x_bytes = (int)(xe * 4);
  a.w_bytes = (int)((we - w0) * 4);
  const auto [px, ch, wgs] = cf_choose(d, win);
  const bool vec = d.cin % 4 == 0 && d.x_pix_stride % 4 == 0 && (uintptr_t)a.x % 16 == 0;
  const bool cut = cf_cut(d, win);
#define DW_CUT(C) \
  if (cut && ch == C) return vec ? launch_tile<1, C, true, true>(st, a) : launch_tile<1, C, false, true>(st, a);
  DW_CUT(1) DW_CUT(2) DW_CUT(3) DW_CUT(4) DW_CUT(5)
#undef DW_CUT
#define DW_CF(P, C) \
  if (px == P && ch == C) vec ? launch_tile<P, C, true>(st, a) : launch_tile<P, C, false>(st, a);
  DW_CF(1, 1) DW_CF(1, 2) DW_CF(1, 3) DW_CF(1, 4) DW_CF(1, 5)
  DW_CF(2, 2) DW_CF(2, 3) DW_CF(2, 4) DW_CF(2, 5)
  DW_CF(4, 2) DW_CF(4, 3) DW_CF(4, 4) DW_CF(4, 5)
#undef DW_CF
}

}  // namespace dw
