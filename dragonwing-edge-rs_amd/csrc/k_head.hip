// Classifier-head ops: Gemm (f32, f16, int8) with the reference's
// accumulation order, GlobalAveragePool and Softmax over rows.  These are
// small ops (a classifier's last layers: batch x 1280 -> 1000, a 7 x 7
// pool), so a Gemm or pool output is one thread's sum in the reference
// order, and what bounds them is how many bytes are in flight beside it.
#include "dw_common.h"
#include "dw_device.h"

#include <algorithm>
#include <type_traits>

namespace dw {
namespace {

// Workgroups of up to 256 threads in x: HIP refuses 2^32 threads or more there.
constexpr long long kMaxGridX = 1 << 23;

// C[i][j] = sum over p of A[i][p] * B[p][j].  f32: fma chain from +0 in p
// order (gemm_f32_naive, ops.rs:273-290).  F16: operands widened with the
// reference decode (h2f), the same chain, f2h of the sum (gemm_fp16,
// ops.rs:461-479).  TB (the graph runtime's transposed path, onnx
// runtime.rs:1220-1233, :1256-1266): B is [n][k] and each step is a multiply
// then an add, each rounded.  bias (blen values): the stored sum plus
// bias[j % blen] (f32 add; f16: F16 of the widened sum).
//
// A workgroup owns 8 x 16 outputs, one chain per thread, and stages 256
// steps of K at a time (A as [row][k], B as [k / 4][column][4], both widened
// to f32) in two LDS buffers: the next chunk's 48 loads a thread are in
// flight while the current one is summed from two 16-byte LDS reads per four
// steps.  A head of 32 x 1280 -> 1000 is bound by the chain (1280 dependent
// steps), the LDS reads beside it and the latency of five chunks; 252
// workgroups of 8 x 16 outputs each read an 80 KB slab of B.  12.1 us, against
// 144 us (290 us with B from HBM) for a thread walking its chain from global
// memory, and 16.8 us for 16 x 16 outputs a workgroup.
constexpr int kGemmR = 8, kGemmC = 16;  // rows and columns of a tile
constexpr int kGemmThreads = kGemmR * kGemmC;
constexpr int kGemmK = 256;          // steps of K in one chunk
constexpr int kGemmLd = kGemmK + 4;  // row stride of A in LDS: four rows read together fall on different banks
__device__ __forceinline__ unsigned umin(unsigned a, unsigned b) { return a < b ? a : b; }
template <bool F16, bool TB>
__global__ __launch_bounds__(kGemmThreads) void gemm_exact_kernel(const void* A, const void* B, void* Cm, int m,
                                                                  int n, int k, const void* bias, int blen) {
  __shared__ __align__(16) float sa[2][kGemmR * kGemmLd];
  __shared__ __align__(16) float sb[2][kGemmK * kGemmC];
  using E = std::conditional_t<F16, uint16_t, float>;
  const E* a = (const E*)A;
  const E* b = (const E*)B;
  const unsigned t = threadIdx.x, i0 = blockIdx.y * kGemmR, j0 = (blockIdx.z * gridDim.x + blockIdx.x) * kGemmC;
  const unsigned um = m, un = n, uk = k;
  if (j0 >= un) return;  // the last grid z's workgroups past the columns
  const unsigned lr = t / kGemmC, lc = t % kGemmC;  // the thread's output; (k quad, column) when it loads B
  auto widen = [](E v) -> float {
    if constexpr (F16) return h2f(v);
    return v;
  };
  // Loads of chunk p0: A's rows (and TB's rows of B) with k across the
  // threads, two values a row each; B's [k][n] rows with columns across 16
  // threads.  Places outside the matrices load the last row, column or step
  // instead, which nothing reads: a load under a condition would be a branch,
  // waited for by itself.
  E ra[2 * kGemmR], rb[2 * kGemmC];
  auto load = [&](unsigned p0) {
    const unsigned last = uk - 1 - p0;
    const unsigned pk[2] = {umin(t, last), umin(t + kGemmThreads, last)};
    const E* ak = a + p0;
#pragma unroll
    for (int r = 0; r < 2 * kGemmR; ++r) ra[r] = ak[(size_t)umin(i0 + (r >> 1), um - 1) * uk + pk[r & 1]];
    if constexpr (TB) {
      const E* bk = b + p0;
#pragma unroll
      for (int q = 0; q < 2 * kGemmC; ++q) rb[q] = bk[(size_t)umin(j0 + (q >> 1), un - 1) * uk + pk[q & 1]];
    } else {
      const E* bk = b + (size_t)p0 * un + umin(j0 + lc, un - 1);
#pragma unroll
      for (int q = 0; q < 2 * kGemmC; ++q) rb[q] = bk[(size_t)umin(4 * (lr + kGemmR * (q >> 2)) + (q & 3), last) * un];
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int r = 0; r < 2 * kGemmR; ++r) sa[buf][(r >> 1) * kGemmLd + t + (r & 1) * kGemmThreads] = widen(ra[r]);
    if constexpr (TB) {
#pragma unroll
      for (int q = 0; q < 2 * kGemmC; ++q) {
        const unsigned p = t + (q & 1) * kGemmThreads;
        sb[buf][((p >> 2) * kGemmC + (q >> 1)) * 4 + (p & 3)] = widen(rb[q]);
      }
    } else {
#pragma unroll
      for (int q = 0; q < kGemmC / 2; ++q)
        *reinterpret_cast<float4*>(&sb[buf][((lr + kGemmR * q) * kGemmC + lc) * 4]) =
            make_float4(widen(rb[4 * q]), widen(rb[4 * q + 1]), widen(rb[4 * q + 2]), widen(rb[4 * q + 3]));
    }
  };
  float acc = 0.0f;
  load(0);
  store(0);
  __syncthreads();
  for (unsigned p0 = 0, buf = 0; p0 < uk; p0 += kGemmK, buf ^= 1) {
    const bool more = uk - p0 > kGemmK;
    if (more) load(p0 + kGemmK);
    const float* pa = &sa[buf][lr * kGemmLd];
    const float* pb = &sb[buf][lc * 4];
    const int steps = (int)umin(kGemmK, uk - p0);
    auto step = [&](float x, float y) {
      if constexpr (TB) {
        float prod = x * y;
        asm("" : "+v"(prod));  // rounded product, then the add
        acc = acc + prod;
      } else {
        acc = fmaf(x, y, acc);
      }
    };
#pragma unroll 8
    for (int p = 0; p + 4 <= steps; p += 4) {
      const float4 x = *reinterpret_cast<const float4*>(pa + p);
      const float4 y = *reinterpret_cast<const float4*>(pb + p * kGemmC);
      step(x.x, y.x);
      step(x.y, y.y);
      step(x.z, y.z);
      step(x.w, y.w);
    }
    for (int p = steps & ~3; p < steps; ++p) step(pa[p], pb[(p & ~3) * kGemmC + (p & 3)]);
    if (more) store(buf ^ 1);
    __syncthreads();
  }
  const unsigned i = i0 + lr, j = j0 + lc;
  if (i >= um || j >= un) return;
  if constexpr (F16) {
    uint16_t hb = f2h(acc);
    if (bias) hb = f16_add_bits(hb, ((const uint16_t*)bias)[j % blen]);
    ((uint16_t*)Cm)[(size_t)i * n + j] = hb;
  } else {
    if (bias) acc = acc + ((const float*)bias)[j % blen];
    ((float*)Cm)[(size_t)i * n + j] = acc;
  }
}

// The same sums with a thread per output straight from memory (j across the
// lanes: B's rows coalesced, A's value the same in every lane).  The tiles
// above cost about 2 us for 1024 workgroups before their first step; on many
// outputs of few steps that is the whole product.
template <bool F16, bool TB>
__global__ __launch_bounds__(256) void gemm_thread_kernel(const void* A, const void* B, void* Cm, int m, int n, int k,
                                                          const void* bias, int blen) {
  using E = std::conditional_t<F16, uint16_t, float>;
  const int j = blockIdx.x * 256 + threadIdx.x;
  const int i = blockIdx.y;
  if (j >= n || i >= m) return;
  const E* a = (const E*)A + (size_t)i * k;
  const E* b = (const E*)B + (TB ? (size_t)j * k : (size_t)j);
  const size_t bs = TB ? 1 : (size_t)n;  // B's step along p
  auto widen = [](E v) -> float {
    if constexpr (F16) return h2f(v);
    return v;
  };
  float acc = 0.0f;
  for (int p = 0; p < k; ++p) {
    const float x = widen(a[p]), y = widen(b[p * bs]);
    if constexpr (TB) {
      float prod = x * y;
      asm("" : "+v"(prod));  // rounded product, then the add
      acc = acc + prod;
    } else {
      acc = fmaf(x, y, acc);
    }
  }
  if constexpr (F16) {
    uint16_t hb = f2h(acc);
    if (bias) hb = f16_add_bits(hb, ((const uint16_t*)bias)[j % blen]);
    ((uint16_t*)Cm)[(size_t)i * n + j] = hb;
  } else {
    if (bias) acc = acc + ((const float*)bias)[j % blen];
    ((float*)Cm)[(size_t)i * n + j] = acc;
  }
}

// Whether a thread per output is expected to be done before the tiles, in
// microseconds: a chain of K steps that the waves in flight lengthen (of a
// transposed B, the more so the further apart its rows lie), against the tiles'
// workgroups, and their chains where they fill the chip more than once.  Fitted
// (7-30%) to 746 products of up to 4096 rows and 8192 columns with K of 8 to
// 290, both kernels timed at each; the thread has the benefit of the doubt.  The
// choice is more than 5% slower than a thread per output in 6 of them, the
// worst 19%.  1024 x 1024 f32 with K = 8
// 4.4 against 17.9 us, with K = 64 14.9 against 20.6 us; 3721 x 1616 with K = 75
// 104 against 120 us; 32 x 1000 with K = 8 3.9 against 3.6 us, with K = 128 13.8
// against 3.8 us.  Above 128 steps it won nowhere.
bool gemm_by_threads(int dtype, bool trans_b, int m, int n, int k) {
  if (k > 128) return false;
  struct Fit {
    float start, tile, step, round;  // tiles: a call, a tile, its step, a step of 1024 tiles
    float tstart, tstep, wave;       // threads: a call, a step, a wave's step
  };
  static const Fit fits[2][2] = {{{3.59f, 1.65e-3f, 6.93e-6f, 1.77e-3f, 2.29f, 0.0654f, 1.12e-5f},
                                  {2.94f, 2.33e-3f, 8.9e-6f, 1.07e-2f, 1.76f, 0.0756f, 5.7e-5f}},
                                 {{3.44f, 2.43e-3f, 2.72e-6f, 3.88e-3f, 2.13f, 0.0839f, 1.5e-5f},
                                  {3.0f, 2.43e-3f, 9.8e-6f, 1.36e-2f, 1.83f, 0.082f, 5.7e-5f}}};
  const Fit& f = fits[dtype == F16][trans_b];
  const int rows = (m - 1) / kGemmR + 1, cols = (n - 1) / kGemmC + 1;
  const float tiles = (float)rows * (float)cols, rounds = (float)(((long long)rows * cols + 1023) / 1024);
  const float steps = (float)k, row_bytes = steps * (dtype == F16 ? 2.0f : 4.0f);
  const float waves = (float)m * (float)((n - 1) / 64 + 1) * (trans_b ? std::max(1.0f, row_bytes / 36.0f) : 1.0f);
  return f.tstart + steps * (f.tstep + f.wave * waves) <
         (trans_b ? 1.1f : 1.05f) * (f.start + tiles * (f.tile + f.step * steps) + f.round * steps * rounds);
}

// int32 sum of i8 products (gemm_i8_scalar, ops.rs:2981-2995); integer
// addition wraps like the reference's release build, in any order.
__global__ __launch_bounds__(256) void gemm_i8_kernel(const int8_t* A, const int8_t* B, int32_t* Cm, int m, int n,
                                                      int k) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  const int i = blockIdx.y;
  if (j >= n || i >= m) return;
  const int8_t* a = A + (size_t)i * k;
  const int8_t* b = B + j;
  uint32_t acc = 0;
  for (int p = 0; p < k; ++p) acc += (uint32_t)((int32_t)a[p] * (int32_t)b[(size_t)p * n]);
  Cm[(size_t)i * n + j] = (int32_t)acc;
}

// NHWC global average pool (CpuGraphRuntime::dispatch_global_avg_pool,
// onnx runtime.rs:1109-1175): thread (batch, channel) sums its h x w values
// in row-major order in f32 and divides by h * w (correctly rounded); f16
// widens with the reference decode and rounds the mean to f16.
// The sum is one ordered chain, so what counts is the loads in flight: AHEAD are
// issued before the first is added (past the end the last value again, not
// added; 16, or 4 and 1 for the few pixels that would be loaded again and
// again), and workgroups of one wave spread a small batch over the CUs (T = 64;
// 256 where they are so many that their dispatch, 0.5 ns each, counts).
// 32 x 7 x 7 x 1280 f32: 6.9-13.6 us before, 5.0 us.
constexpr int kGapAhead = 16;
template <bool F16, int T, int AHEAD>
__global__ __launch_bounds__(T) void global_avg_pool_kernel(const void* X, void* Y, int n, int hw, int c) {
  using E = std::conditional_t<F16, uint16_t, float>;
  const int ch = blockIdx.x * T + threadIdx.x;
  const int b = blockIdx.y;
  if (ch >= c || b >= n) return;
  const E* x = (const E*)X + (size_t)b * hw * c + ch;
  auto widen = [](E v) -> float {
    if constexpr (F16) return h2f(v);
    return v;
  };
  float sum = 0.0f;
  unsigned s0 = 0;
  for (; s0 + AHEAD <= (unsigned)hw; s0 += AHEAD) {
    E v[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) v[j] = x[(size_t)(s0 + j) * c];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) sum += widen(v[j]);
  }
  if (AHEAD > 1 && s0 < (unsigned)hw) {
    E v[AHEAD];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) v[j] = x[(size_t)umin(s0 + j, hw - 1) * c];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) sum = s0 + j < (unsigned)hw ? sum + widen(v[j]) : sum;
  }
  const float mean = __fdiv_rn(sum, (float)hw);
  if constexpr (F16)
    ((uint16_t*)Y)[(size_t)b * c + ch] = f2h(mean);
  else
    ((float*)Y)[(size_t)b * c + ch] = mean;
}

// Reductions over a group of G consecutive threads (G up to 64: lanes of a
// wave; 256: the workgroup, through LDS).
template <int G, typename Op>
__device__ __forceinline__ float group_reduce(float v, Op op) {
#pragma unroll
  for (int x = 1; x < (G < 64 ? G : 64); x <<= 1) v = op(v, __shfl_xor(v, x));
  if constexpr (G == 256) {
    __shared__ float part[4];
    __syncthreads();  // an earlier reduction's reads are done
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = v;
    __syncthreads();
    v = op(op(part[0], part[1]), op(part[2], part[3]));
  }
  return v;
}

// Softmax over rows of n (softmax_f32, ops.rs:1609-1638): the max from -inf
// (fmaxf: a NaN operand loses, as f32::max), e = exp(x - max), out = e *
// (1 / sum).  The sum is a tree over the threads' partial sums, whose
// rounding error is below the reference's serial sum's; exp is the device
// expf, so outputs agree with the host's to within a few ulps.  The f16 form
// (CpuGraphRuntime::dispatch_softmax, runtime.rs:1311-1322) widens every
// input with the reference decode, runs the f32 softmax and rounds each
// output once to f16.
// G threads share a row, so that its loads are coalesced and in flight
// together; a row of up to kSoftmaxRegs * G values is read once and stays in
// registers.  A classifier's 32 x 1000 (128 KB, launch latency bound) takes
// 4.6 us, against 391 us for a thread per row walking it three times.
constexpr int kSoftmaxRegs = 8;
template <bool H, int G>
__global__ __launch_bounds__(256) void softmax_rows_kernel(const void* X, void* Y, int rows, int n) {
  // (grid y: a launch's threads in x stay below 2^32)
  const size_t r = ((size_t)blockIdx.y * gridDim.x + blockIdx.x) * (256 / G) + threadIdx.x / G;
  const int l = threadIdx.x % G;
  const bool live = r < (size_t)rows;  // a dead group runs along (its lanes' wave reduces together)
  const size_t base = (live ? r : 0) * n;
  auto ld = [&](int i) -> float {
    if constexpr (H) return h2f(((const uint16_t*)X)[base + i]);
    return ((const float*)X)[base + i];
  };
  auto st = [&](int i, float v) {
    if (!live) return;
    if constexpr (H)
      ((uint16_t*)Y)[base + i] = f2h(v);
    else
      ((float*)Y)[base + i] = v;
  };
  auto fmx = [](float a, float b) { return fmaxf(a, b); };
  auto add = [](float a, float b) { return a + b; };
  float mx = -INFINITY, sum = 0.0f;
  if (n <= kSoftmaxRegs * G) {
    float v[kSoftmaxRegs];
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j) v[j] = j * G + l < n ? ld(j * G + l) : -INFINITY;
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j) mx = fmaxf(mx, v[j]);
    mx = group_reduce<G>(mx, fmx);
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j)
      if (j * G + l < n) {
        v[j] = expf(v[j] - mx);
        sum += v[j];
      }
    const float inv = __fdiv_rn(1.0f, group_reduce<G>(sum, add));
#pragma unroll
    for (int j = 0; j < kSoftmaxRegs; ++j)
      if (j * G + l < n) st(j * G + l, v[j] * inv);
  } else {
    for (int i = l; i < n; i += G) mx = fmaxf(mx, ld(i));
    mx = group_reduce<G>(mx, fmx);
    for (int i = l; i < n; i += G) sum += expf(ld(i) - mx);
    const float inv = __fdiv_rn(1.0f, group_reduce<G>(sum, add));
    for (int i = l; i < n; i += G) st(i, expf(ld(i) - mx) * inv);
  }
}

// QLinearGlobalAveragePool over NHWC u8: per (batch, channel) the h x w
// values minus the input zero point are summed as an int32, then
// y = clamp(rint((float)sum * M) + y_zp, 0, 255) with M = (x_scale / y_scale)
// / (h * w) in f32 (rint: round half to even).
__device__ __forceinline__ uint8_t qgap_out(int acc, float m, int y_zp) {
  const float q = rintf((float)acc * m) + (float)y_zp;
  return (uint8_t)fminf(fmaxf(q, 0.0f), 255.0f);
}

// A workgroup owns 64 * 4 bytes of channels (a dword of four channels a lane,
// c % 4 == 0) of one image; its four waves take a quarter of the pixels each,
// kGapAhead loads in flight, and the sums (integers, any order) meet in LDS.
// 32 x 7 x 7 x 1280: 7.1 us for a byte a thread walking all pixels, 3.0 us.
__global__ __launch_bounds__(256) void qlinear_gap_kernel(const uint8_t* X, uint8_t* Y, int n, int hw, int c,
                                                          int x_zp, float m, int y_zp) {
  __shared__ __align__(16) uint32_t part[4][64][4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch = (blockIdx.x * 64 + lane) * 4, b = blockIdx.y;
  const uint8_t* x = X + (size_t)b * hw * c + (ch < c ? ch : 0);
  // bytes 0 and 2, 1 and 3 in 16-bit halves: 257 pixels before one overflows
  uint32_t tot[4] = {0, 0, 0, 0};
  for (int s0 = wave * kGapAhead; s0 < hw; s0 += 4 * kGapAhead) {
    uint32_t v[kGapAhead], even = 0, odd = 0;
#pragma unroll
    for (int j = 0; j < kGapAhead; ++j)
      v[j] = *reinterpret_cast<const uint32_t*>(x + (size_t)(s0 + j < hw ? s0 + j : hw - 1) * c);
#pragma unroll
    for (int j = 0; j < kGapAhead; ++j) {
      const uint32_t w = s0 + j < hw ? v[j] : 0u;
      even += w & 0x00ff00ffu;
      odd += (w >> 8) & 0x00ff00ffu;
    }
    tot[0] += even & 0xffffu;
    tot[1] += odd & 0xffffu;
    tot[2] += even >> 16;
    tot[3] += odd >> 16;
  }
  *reinterpret_cast<uint4*>(part[wave][lane]) = make_uint4(tot[0], tot[1], tot[2], tot[3]);
  __syncthreads();
  if (wave != 0 || ch >= c) return;
  uint32_t out = 0;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const uint32_t sum = part[0][lane][j] + part[1][lane][j] + part[2][lane][j] + part[3][lane][j];
    out |= (uint32_t)qgap_out((int)(sum - (uint32_t)hw * (uint32_t)x_zp), m, y_zp) << (8 * j);
  }
  *reinterpret_cast<uint32_t*>(Y + (size_t)b * c + ch) = out;
}

// The same for channel counts that are no multiple of 4, and for a few pixels,
// which leave three of the four waves nothing: a byte a thread.
template <int T>
__global__ __launch_bounds__(T) void qlinear_gap_byte_kernel(const uint8_t* X, uint8_t* Y, int n, int hw, int c,
                                                             int x_zp, float m, int y_zp) {
  const int ch = blockIdx.x * T + threadIdx.x;
  const int b = blockIdx.y;
  if (ch >= c || b >= n) return;
  const uint8_t* x = X + (size_t)b * hw * c + ch;
  int acc = 0;
#pragma unroll 8
  for (int s = 0; s < hw; ++s) acc += (int)x[(size_t)s * c] - x_zp;
  Y[(size_t)b * c + ch] = qgap_out(acc, m, y_zp);
}

// dst[c][r] = src[r][c] for a rows x cols byte matrix (32 x 32 tiles through LDS).
__global__ __launch_bounds__(256) void transpose_u8_kernel(const uint8_t* src, uint8_t* dst, int rows, int cols) {
  __shared__ uint8_t t[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;
    if (r < rows && c < cols) t[k][tx] = src[(size_t)r * cols + c];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k, r = r0 + tx;
    if (r < rows && c < cols) dst[(size_t)c * rows + r] = t[tx][k];
  }
}

}  // namespace

void launch_gemm_ex(hipStream_t st, int dtype, const void* a, const void* b, void* c, int m, int n, int k,
                    bool trans_b, const void* bias, int blen) {
  if (m > 65535) fail(-2, "gemm: more than 65535 rows");
  const long long cols = ((long long)n + kGemmC - 1) / kGemmC, gx = std::min(cols, kMaxGridX);
  const dim3 g((unsigned)gx, (unsigned)((m + kGemmR - 1) / kGemmR), (unsigned)((cols + gx - 1) / gx));
  const bool threads = gemm_by_threads(dtype, trans_b, m, n, k);
  const dim3 gt((unsigned)((n - 1) / 256 + 1), (unsigned)m);
  auto launch = [&](auto* tile, auto* thread) {
    if (threads)
      hipLaunchKernelGGL(thread, gt, dim3(256), 0, st, a, b, c, m, n, k, bias, blen);
    else
      hipLaunchKernelGGL(tile, g, dim3(kGemmThreads), 0, st, a, b, c, m, n, k, bias, blen);
  };
  if (dtype == F32 && !trans_b)
    launch(gemm_exact_kernel<false, false>, gemm_thread_kernel<false, false>);
  else if (dtype == F32)
    launch(gemm_exact_kernel<false, true>, gemm_thread_kernel<false, true>);
  else if (dtype == F16 && !trans_b)
    launch(gemm_exact_kernel<true, false>, gemm_thread_kernel<true, false>);
  else if (dtype == F16)
    launch(gemm_exact_kernel<true, true>, gemm_thread_kernel<true, true>);
  else
    fail(-2, "gemm: dtype");
  DW_HIP(hipGetLastError());
}

void launch_gemm(hipStream_t st, int dtype, const void* a, const void* b, void* c, int m, int n, int k) {
  const dim3 g((unsigned)((n + 255) / 256), (unsigned)m);
  if (dtype == F32 || dtype == F16)
    return launch_gemm_ex(st, dtype, a, b, c, m, n, k, false, nullptr, 1);
  if (dtype == I8)
    hipLaunchKernelGGL(gemm_i8_kernel, g, dim3(256), 0, st, (const int8_t*)a, (const int8_t*)b, (int32_t*)c, m, n,
                       k);
  else
    fail(-2, "gemm: dtype");
  DW_HIP(hipGetLastError());
}

namespace {
// Threads of a pool's workgroups, of which each takes a channel: a wave, unless
// that makes so many workgroups that they take longer to dispatch than to run
// (4096 images of 1 x 1 x 1024 f32: 20.2 us in waves, 9.7 us in fours).
int pool_threads(int n, int c) { return c > 64 && (long long)n * ((c - 1) / 64 + 1) >= 4096 ? 256 : 64; }
}  // namespace

void launch_global_avg_pool(hipStream_t st, int dtype, const void* x, void* y, int n, int hw, int c) {
  if (dtype != F32 && dtype != F16) fail(-2, "global average pool: dtype");
  const int t = pool_threads(n, c);
  auto launch = [&](auto* wave, auto* four) {
    hipLaunchKernelGGL(t == 64 ? wave : four, dim3((unsigned)((c - 1) / t + 1), (unsigned)n), dim3(t), 0, st, x, y, n, hw,
                       c);
  };
  if (dtype == F32)
    hw > 12  ? launch(global_avg_pool_kernel<false, 64, 16>, global_avg_pool_kernel<false, 256, 16>)
    : hw > 2 ? launch(global_avg_pool_kernel<false, 64, 4>, global_avg_pool_kernel<false, 256, 4>)
             : launch(global_avg_pool_kernel<false, 64, 1>, global_avg_pool_kernel<false, 256, 1>);
  else
    hw > 12  ? launch(global_avg_pool_kernel<true, 64, 16>, global_avg_pool_kernel<true, 256, 16>)
    : hw > 2 ? launch(global_avg_pool_kernel<true, 64, 4>, global_avg_pool_kernel<true, 256, 4>)
             : launch(global_avg_pool_kernel<true, 64, 1>, global_avg_pool_kernel<true, 256, 1>);
  DW_HIP(hipGetLastError());
}

void launch_softmax_rows(hipStream_t st, const float* x, float* y, int rows, int n) {
  launch_softmax_rows_t(st, F32, x, y, rows, n);
}

namespace {
// Four values a thread up to a row of 16, which many short rows ask for (the
// kernel's time is its slots then: 262144 rows of 1 value 3.7 us with a
// thread a row, 19.6 us with 16; of 8, 6.6 us with 2, 20.5 us with 16; of 16,
// 8.5 us with 4, 20.6 us with 16); beyond, the smallest group that keeps a row
// in registers: a classifier's 1000 classes take a workgroup.
template <bool H>
void launch_softmax(hipStream_t st, const void* x, void* y, int rows, int n) {
  const int g = n <= 4 ? 1 : n <= 8 ? 2 : n <= 16 ? 4 : n <= kSoftmaxRegs * 16 ? 16 : n <= kSoftmaxRegs * 64 ? 64 : 256;
  auto* k = g == 1    ? softmax_rows_kernel<H, 1>
            : g == 2  ? softmax_rows_kernel<H, 2>
            : g == 4  ? softmax_rows_kernel<H, 4>
            : g == 16 ? softmax_rows_kernel<H, 16>
            : g == 64 ? softmax_rows_kernel<H, 64>
                      : softmax_rows_kernel<H, 256>;
  const long long blocks = ((long long)rows * g + 255) / 256;
  const long long gx = std::min(blocks, kMaxGridX);
  hipLaunchKernelGGL(k, dim3((unsigned)gx, (unsigned)((blocks + gx - 1) / gx)), dim3(256), 0, st, x, y, rows, n);
  DW_HIP(hipGetLastError());
}
}  // namespace

void launch_softmax_rows_t(hipStream_t st, int dtype, const void* x, void* y, int rows, int n) {
  if (dtype == F32)
    launch_softmax<false>(st, x, y, rows, n);
  else if (dtype == F16)
    launch_softmax<true>(st, x, y, rows, n);
  else
    fail(-2, "softmax: dtype");
}

}  // namespace dw

namespace dw {

void launch_qlinear_gap(hipStream_t st, const uint8_t* x, uint8_t* y, int n, int hw, int c, int x_zp, float m,
                        int y_zp) {
  // (4096 images of 1 x 1 x 1024: 8.7 us with a byte a thread, 9.4 us with four and the sums in LDS)
  if (c % 4 == 0 && hw > 4) {
    hipLaunchKernelGGL(qlinear_gap_kernel, dim3((unsigned)((c + 255) / 256), (unsigned)n), dim3(256), 0, st, x, y, n, hw,
                       c, x_zp, m, y_zp);
  } else {
    const int t = pool_threads(n, c);
    hipLaunchKernelGGL(t == 64 ? qlinear_gap_byte_kernel<64> : qlinear_gap_byte_kernel<256>,
                       dim3((unsigned)((c - 1) / t + 1), (unsigned)n), dim3(t), 0, st, x, y, n, hw, c, x_zp, m, y_zp);
  }
  DW_HIP(hipGetLastError());
}

void launch_transpose_u8(hipStream_t st, const void* src, void* dst, int rows, int cols) {
  const dim3 g((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32));
  hipLaunchKernelGGL(transpose_u8_kernel, g, dim3(256), 0, st, (const uint8_t*)src, (uint8_t*)dst, rows, cols);
  DW_HIP(hipGetLastError());
}

}  // namespace dw
