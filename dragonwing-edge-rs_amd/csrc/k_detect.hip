// YOLOv8 detect tail and post-processing on the GPU.
//
// detect_tail_kernel: the exported graph's tail after the three head convs
// (ultralytics Detect in inference): per anchor, DFL (softmax over each
// side's reg_max bins, then the 1x1 expectation with weights 0..reg_max-1),
// dist2bbox (anchor -/+ distances, centre and size) times the level's
// stride, and the sigmoid of every class logit, written as [n][4 + nc][A]
// f32 (the [1, 84, 8400] layout of an export).  Each step is the reference
// f32 op the exported graph applies: softmax_f32 (ops.rs:1609-1638), the
// conv's fma chain (ops.rs:1356-1436), sub/add/div/mul, sigmoid_f32
// (ops.rs:1866-1870).  exp is the device's expf (a few ulps from the host
// libm's), everything else is IEEE single-rounded.
//
// Post-processing (postprocess_yolo, onnx postprocess.rs:279-305), per image:
//   pp_candidates_kernel  decode_detections_v8 (:78-146) for every anchor:
//                         best class, threshold, corners, clamp; a 64-bit
//                         sort key (confidence descending, anchor ascending);
//   pp_nms_kernel         one workgroup per image: the keys over the threshold
//                         gathered and bitonically sorted in registers or LDS
//                         (the reference's stable sort by confidence),
//                         a stable partition by class, greedy NMS per class
//                         on LDS-resident boxes, one wave per class
//                         (nms, :214-243; nms_agnostic as one class), and the
//                         kept detections written in sorted order with their
//                         sorted positions.
// The reference then removes the suppressed entries with swap_remove from
// the back, which reorders the survivors; the host applies that order to
// the kept list (a permutation of the survivors, no arithmetic).
#include "dw_common.h"
#include "dw_device.h"

#include <type_traits>

namespace dw {
namespace {

struct TailLevels {
  const void* x[4];
  int h[4], w[4];
  int start[4];  // first anchor of the level
  int tile0[4];  // first 64-anchor tile of the level
  int pix[4];    // elements per pixel
  float stride[4];
  int levels;
  int A;
};

template <bool H>
__device__ __forceinline__ float tail_ld(const void* p, size_t i) {
  if constexpr (H)
    return h2f(((const uint16_t*)p)[i]);
  else
    return ((const float*)p)[i];
}

// One side's DFL from its logits ld(0..reg_max-1): softmax, then the
// expectation's fma chain.  R > 0: reg_max as a constant, so that the
// exponentials stay in registers; 0: any reg_max, each computed twice.
template <int R, typename Ld>
__device__ __forceinline__ float dfl_side(int reg_max, Ld ld) {
  float mx = -INFINITY, sum = 0.0f, acc = 0.0f;
  if constexpr (R > 0) {
    float e[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
      e[k] = ld(k);
      mx = fmaxf(mx, e[k]);
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
      e[k] = expf(e[k] - mx);
      sum += e[k];
    }
    const float inv = __fdiv_rn(1.0f, sum);
#pragma unroll
    for (int k = 0; k < R; ++k) acc = fmaf(e[k] * inv, (float)k, acc);
  } else {
    for (int k = 0; k < reg_max; ++k) mx = fmaxf(mx, ld(k));
    for (int k = 0; k < reg_max; ++k) sum += expf(ld(k) - mx);
    const float inv = __fdiv_rn(1.0f, sum);
    for (int k = 0; k < reg_max; ++k) acc = fmaf(expf(ld(k) - mx) * inv, (float)k, acc);
  }
  return acc;
}

// Row j of the box (centre x, centre y, width, height) of the anchor at grid
// cell (gx, gy), from its four distances.
__device__ __forceinline__ float box_row(int j, const float d[4], int gx, int gy, float st) {
  const float ax = (float)gx + 0.5f, ay = (float)gy + 0.5f;
  const float lo = j & 1 ? ay - d[1] : ax - d[0];
  const float hi = j & 1 ? ay + d[3] : ax + d[2];
  return (j < 2 ? __fdiv_rn(lo + hi, 2.0f) : hi - lo) * st;
}
__device__ __forceinline__ float sigmoid_rn(float v) { return __fdiv_rn(1.0f, 1.0f + expf(-v)); }

// A workgroup takes 64 consecutive anchors of one level and image: their
// pixels, 288 contiguous bytes each for an f16 head of 144 channels, are read
// as whole lines (every load of a thread in flight together), widened once
// and kept in LDS as f32 with an odd row stride, so that 64 lanes at one
// channel of 64 anchors fall on different banks.  A wave owns one box side
// (its DFL, then one box row) and a quarter of the classes; every output row
// is written as 64 consecutive floats.  Bound by exp and the divisions once
// the bytes stream (624 B an anchor): eight 640x640 images (42 MB) take
// 22 us, against 83 us for a thread per anchor reading its own pixel two
// bytes at a time.
constexpr int kTailAnchors = 64;
// dwords a thread may hold: 192 f16 or 160 f32 channels
__host__ __device__ constexpr int tail_loads(bool h) { return h ? 24 : 40; }
template <bool H, int R>
__global__ __launch_bounds__(256) void detect_tail_tile_kernel(TailLevels L, float* out, int nc, int reg_max) {
  extern __shared__ float tile[];  // [64][ld], then the distances [4][64]
  const int chans = 4 * reg_max + nc, ld = chans | 1;
  float* dist = tile + kTailAnchors * ld;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, b = blockIdx.y;
  int s = 0;
  while (s + 1 < L.levels && (int)blockIdx.x >= L.tile0[s + 1]) ++s;
  const int hw = L.h[s] * L.w[s];
  const int a0 = ((int)blockIdx.x - L.tile0[s]) * kTailAnchors;  // first anchor in the level
  const int live = min(kTailAnchors, hw - a0);
  // dword i of the tile: anchor i / dw, its dword i % dw; 256 dwords further
  // on is (256 / dw, 256 % dw) further on
  const int dw = H ? chans / 2 : chans, pixdw = H ? L.pix[s] / 2 : L.pix[s];
  const uint32_t* x = (const uint32_t*)L.x[s] + ((size_t)b * hw + a0) * (size_t)pixdw;
  const int sa = 256 / dw, sr = 256 % dw;
  // all of a thread's dwords on their way before the first is stored: N of them,
  // for the tiles that have few (few channels, or a map's last tile)
  auto stage = [&](auto count) {
    constexpr int N = decltype(count)::value;
    uint32_t v[N];
    int a = t / dw, r = t % dw;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      v[i] = x[a < live ? (size_t)a * pixdw + r : 0];
      a += sa;
      r += sr;
      if (r >= dw) {
        r -= dw;
        ++a;
      }
    }
    a = t / dw;
    r = t % dw;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (a < live) {
        if constexpr (H) {
          tile[a * ld + 2 * r] = h2f((uint16_t)v[i]);
          tile[a * ld + 2 * r + 1] = h2f((uint16_t)(v[i] >> 16));
        } else {
          tile[a * ld + r] = __builtin_bit_cast(float, v[i]);
        }
      }
      a += sa;
      r += sr;
      if (r >= dw) {
        r -= dw;
        ++a;
      }
    }
  };
  if (live * dw <= 2 * 256)
    stage(std::integral_constant<int, 2>{});
  else if (live * dw <= 8 * 256)
    stage(std::integral_constant<int, 8>{});
  else
    stage(std::integral_constant<int, tail_loads(H)>{});
  __syncthreads();
  const float* row = tile + min(lane, live - 1) * ld;  // idle lanes repeat the last anchor
  dist[wave * 64 + lane] = dfl_side<R>(reg_max, [&](int k) { return row[wave * reg_max + k]; });
  const size_t A = (size_t)L.A;
  float* o = out + (size_t)b * (4 + nc) * A + L.start[s] + a0 + lane;
  for (int c = wave; c < nc; c += 4) {
    const float v = sigmoid_rn(row[4 * reg_max + c]);
    if (lane < live) o[(size_t)(4 + c) * A] = v;
  }
  __syncthreads();
  const float d[4] = {dist[lane], dist[64 + lane], dist[128 + lane], dist[192 + lane]};
  const int gy = (a0 + lane) / L.w[s], gx = (a0 + lane) - gy * L.w[s];
  const float v = box_row(wave, d, gx, gy, L.stride[s]);
  if (lane < live) o[(size_t)wave * A] = v;
}

// A thread per anchor, straight from memory: any head (channels that do not
// pair into dwords, or more than a thread of the tile kernel holds), and those
// that tail_by_tiles leaves to it.
template <bool H>
__global__ __launch_bounds__(256) void detect_tail_kernel(TailLevels L, float* out, int nc, int reg_max) {
  const int a = blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.y;
  if (a >= L.A) return;
  int s = 0;
  while (s + 1 < L.levels && a >= L.start[s + 1]) ++s;
  const int local = a - L.start[s];
  const int gy = local / L.w[s];
  const int gx = local - gy * L.w[s];
  const size_t px = (((size_t)b * L.h[s] + gy) * L.w[s] + gx) * (size_t)L.pix[s];
  const void* x = L.x[s];
  const size_t A = (size_t)L.A;
  float* o = out + (size_t)b * (4 + nc) * A + a;
  float d[4];
  for (int j = 0; j < 4; ++j)
    d[j] = dfl_side<0>(reg_max, [&](int k) { return tail_ld<H>(x, px + (size_t)j * reg_max + k); });
  for (int j = 0; j < 4; ++j) o[(size_t)j * A] = box_row(j, d, gx, gy, L.stride[s]);
  for (int c = 0; c < nc; ++c) o[(size_t)(4 + c) * A] = sigmoid_rn(tail_ld<H>(x, px + (size_t)4 * reg_max + c));
}

// ---------------------------------------------------------------------------
// post-processing

struct PPArgs {
  const float* raw;  // [n][4 + nc][A]
  int nc, A;
  float sx, sy, img_w, img_h, conf, iou;
  int agnostic;
  int nmax;          // capacity of the per-image arrays below
  unsigned long long* keys;  // [n][A]
  DwDetection* det;          // [n][A], per anchor
  int* sorted_anchor;        // [n][nmax]
  int* part_pos;             // [n][nmax]
  DwKept* kept;              // every image's kept detections, one image after another
  int* counts;               // [n][4]: candidates, kept, overflow, first of the image's in `kept`
  int* cursor;               // entries of `kept` taken
};

__global__ __launch_bounds__(256) void pp_candidates_kernel(PPArgs p) {
  const int a = blockIdx.x * 256 + threadIdx.x;
  const int b = blockIdx.y;
  if (a >= p.A) return;
  const size_t A = (size_t)p.A;
  const float* r = p.raw + (size_t)b * (4 + p.nc) * A + a;
  const float cx = r[0], cy = r[A], w = r[2 * A], h = r[3 * A];
  // the class rows 16 at a time, so that their loads are in flight together
  // (past the last class its value again, which is not greater)
  int best = 0;
  float best_conf = 0.0f;
  for (int c0 = 0; c0 < p.nc; c0 += 16) {
    float v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = r[(size_t)(4 + min(c0 + j, p.nc - 1)) * A];
#pragma unroll
    for (int j = 0; j < 16; ++j)
      if (v[j] > best_conf) {
        best_conf = v[j];
        best = c0 + j;
      }
  }
  if (a == 0 && b == 0) *p.cursor = 0;  // for pp_nms_kernel, which follows
  unsigned long long key = ~0ull;
  if (!(best_conf < p.conf)) {
    const float hw = __fdiv_rn(w, 2.0f), hh = __fdiv_rn(h, 2.0f);
    float x1 = (cx - hw) * p.sx, y1 = (cy - hh) * p.sy;
    float x2 = (cx + hw) * p.sx, y2 = (cy + hh) * p.sy;
    x1 = fminf(fmaxf(x1, 0.0f), p.img_w);
    y1 = fminf(fmaxf(y1, 0.0f), p.img_h);
    x2 = fminf(fmaxf(x2, 0.0f), p.img_w);
    y2 = fminf(fmaxf(y2, 0.0f), p.img_h);
    DwDetection d;
    d.bbox[0] = x1;
    d.bbox[1] = y1;
    d.bbox[2] = x2;
    d.bbox[3] = y2;
    d.class_id = (uint32_t)best;
    d.confidence = best_conf;
    p.det[(size_t)b * A + a] = d;
    // confidence >= +0, so its bits order like its value
    key = ((unsigned long long)(0xFFFFFFFFu - __float_as_uint(best_conf)) << 32) | (unsigned)a;
  }
  p.keys[(size_t)b * A + a] = key;
}

// Detection::area and iou (postprocess.rs:28-32, :36-55), each operation
// rounded as written (no contraction).
__device__ __forceinline__ float box_area(float4 d) {
  return fmaxf(d.z - d.x, 0.0f) * fmaxf(d.w - d.y, 0.0f);
}
__device__ __forceinline__ float box_iou(float4 a, float aa, float4 b) {
  const float x1 = fmaxf(a.x, b.x), y1 = fmaxf(a.y, b.y);
  const float x2 = fminf(a.z, b.z), y2 = fminf(a.w, b.w);
  const float inter = fmaxf(x2 - x1, 0.0f) * fmaxf(y2 - y1, 0.0f);
  const float uni = aa + box_area(b) - inter;
  return uni > 0.0f ? __fdiv_rn(inter, uni) : 0.0f;
}

constexpr int kNmsThreads = 1024;
constexpr int kNmsPer = (kPPMaxCandidates + kNmsThreads - 1) / kNmsThreads;

// LDS layout (bytes), phase by phase:
//   [0, 16 nmax)            sort keys (at most 16384 of 8 bytes), then class ids
//                           of the sorted candidates (u16), then the boxes in
//                           class-partitioned order (float4)
//   [16 nmax, 17 nmax)      keep flags (partitioned order)
//   then 1024 ints          per-class counts / scan scratch
//   then 1024 ints          per-class offsets
//   then nmax / 32 words    kept bitmap over sorted positions
//   then 4 ints             candidate count, next class, first kept entry
__host__ __device__ constexpr size_t nms_lds_bytes(int nmax) {
  return (size_t)17 * nmax + 2 * 1024 * 4 + (size_t)((nmax + 31) / 32) * 4 + 16;
}

// Inclusive scan over the workgroup's threads (wsum: an int per wave).
__device__ __forceinline__ int block_scan(int v, int* wsum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int add = __shfl_up(v, d);
    v += lane >= d ? add : 0;
  }
  __syncthreads();  // an earlier scan's reads are done
  if (lane == 63) wsum[wave] = v;
  __syncthreads();
  for (int w = 0; w < kNmsThreads / 64 - 1; ++w) v += w < wave ? wsum[w] : 0;
  return v;
}

// One workgroup per image, a chain of short phases between barriers, so its
// time is their latencies: sorting only the candidates (a few hundred, in
// registers) and scanning through lane shuffles, eight 640x640 frames of
// about 350 candidates take 31 us, against 243 us with a sort of 16384 keys.
__global__ __launch_bounds__(kNmsThreads) void pp_nms_kernel(PPArgs p) {
  __shared__ int wsum[kNmsThreads / 64];
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int nmax = p.nmax;
  unsigned long long* sk = (unsigned long long*)smem;
  uint16_t* scls = (uint16_t*)smem;
  float4* sbox = (float4*)smem;
  volatile uint8_t* keep = smem + (size_t)16 * nmax;
  int* scnt = (int*)(smem + (size_t)17 * nmax);
  int* soff = scnt + 1024;
  uint32_t* kbits = (uint32_t*)(soff + 1024);
  int* sn = (int*)(kbits + (nmax + 31) / 32);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x;
  const int A = p.A;
  const int ncls = p.agnostic ? 1 : p.nc;

  if (tid == 0) {
    sn[0] = 0;
    sn[1] = 0;
  }
  __syncthreads();
  // The keys over the threshold, gathered in any order (they are distinct,
  // so the sort decides): a few hundred of 8400 on an ordinary frame.
  // All loads first: at most 16384 anchors, 16 a thread.
  {
    unsigned long long key[16384 / kNmsThreads];
#pragma unroll
    for (int u = 0; u < 16384 / kNmsThreads; ++u)
      key[u] = p.keys[(size_t)b * A + min(u * kNmsThreads + tid, A - 1)];
#pragma unroll
    for (int u = 0; u < 16384 / kNmsThreads; ++u) {
      const bool in = u * kNmsThreads + tid < A && key[u] != ~0ull;
      const unsigned long long m = __ballot(in);
      if (m) {
        int at = 0;
        if (lane == 0) at = atomicAdd(&sn[0], __popcll(m));
        at = __shfl(at, 0);
        if (in) sk[at + __popcll(m & ((1ull << lane) - 1))] = key[u];
      }
    }
  }
  __syncthreads();
  const int n = sn[0];
  // bitonic sort, ascending: confidence descending, then anchor ascending
  int S = 64;
  while (S < n) S <<= 1;
  if (S <= kNmsThreads) {
    // a key per thread: partners in the same wave trade through lane
    // shuffles, only the others through LDS and barriers (6 of 45 steps at 512)
    unsigned long long key = tid < n ? sk[tid] : ~0ull;
    __syncthreads();
    for (int k = 2; k <= S; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        unsigned long long other;
        if (j >= 64) {
          sk[tid] = key;
          __syncthreads();
          other = sk[tid ^ j];
          __syncthreads();
        } else {
          other = __shfl_xor(key, j);
        }
        // the lower place of an ascending pair keeps the smaller key
        const bool low = ((tid & j) == 0) == ((tid & k) == 0);
        key = (key < other) == low ? key : other;
      }
    sk[tid] = key;
    __syncthreads();
  } else {
    for (int i = n + tid; i < S; i += kNmsThreads) sk[i] = ~0ull;
    __syncthreads();
    for (int k = 2; k <= S; k <<= 1)
      for (int j = k >> 1; j > 0; j >>= 1) {
        for (int i = tid; i < S; i += kNmsThreads) {
          const int ixj = i ^ j;
          if (ixj > i) {
            const unsigned long long u = sk[i], v = sk[ixj];
            if ((u > v) == ((i & k) == 0)) {
              sk[i] = v;
              sk[ixj] = u;
            }
          }
        }
        __syncthreads();
      }
  }
  int* cnt = p.counts + 4 * b;
  if (n > nmax) {
    if (tid == 0) {
      cnt[0] = n;
      cnt[1] = 0;
      cnt[2] = 1;
      cnt[3] = 0;
    }
    return;
  }
  // sorted candidates: anchors to global, classes kept in registers
  int my_cls[kNmsPer];
#pragma unroll
  for (int t = 0; t < kNmsPer; ++t) {
    const int q = tid + t * kNmsThreads;
    my_cls[t] = -1;
    if (q < n) {
      const int a = (int)(unsigned)(sk[q] & 0xFFFFFFFFull);
      p.sorted_anchor[(size_t)b * nmax + q] = a;
      my_cls[t] = p.agnostic ? 0 : (int)p.det[(size_t)b * A + a].class_id;
    }
  }
  for (int c = tid; c < 1024; c += kNmsThreads) scnt[c] = 0;
  for (int w = tid; w < (nmax + 31) / 32; w += kNmsThreads) kbits[w] = 0;
  __syncthreads();  // keys no longer read
#pragma unroll
  for (int t = 0; t < kNmsPer; ++t) {
    const int q = tid + t * kNmsThreads;
    if (q < n) {
      scls[q] = (uint16_t)my_cls[t];
      atomicAdd(&scnt[my_cls[t]], 1);
    }
  }
  __syncthreads();
  // exclusive scan of the class counts (ncls <= 1024)
  const int v = tid < ncls ? scnt[tid] : 0;
  soff[tid] = block_scan(v, wsum) - v;
  __syncthreads();
  // stable partition by class: one wave per class, ballots over the sorted order
  for (int c = wave; c < ncls; c += kNmsThreads / 64) {
    int cursor = soff[c];
    for (int q0 = 0; q0 < n; q0 += 64) {
      const int q = q0 + lane;
      const bool m = q < n && (int)scls[q] == c;
      const unsigned long long bal = __ballot(m);
      if (m) {
        const int rank = __popcll(bal & ((1ull << lane) - 1));
        p.part_pos[(size_t)b * nmax + cursor + rank] = q;
      }
      cursor += __popcll(bal);
    }
  }
  __syncthreads();
  // boxes in partitioned order
  for (int q = tid; q < n; q += kNmsThreads) {
    const int sp = p.part_pos[(size_t)b * nmax + q];
    const int a = p.sorted_anchor[(size_t)b * nmax + sp];
    const DwDetection d = p.det[(size_t)b * A + a];
    sbox[q] = make_float4(d.bbox[0], d.bbox[1], d.bbox[2], d.bbox[3]);
    keep[q] = 1;
  }
  __syncthreads();
  // greedy suppression per class, one wave per class (taken in turn)
  for (;;) {
    int c = 0;
    if (lane == 0) c = atomicAdd(&sn[1], 1);
    c = __shfl(c, 0);
    if (c >= ncls) break;
    const int s0 = soff[c], e0 = s0 + scnt[c];
    for (int i = s0; i < e0; ++i) {
      if (!keep[i]) continue;
      const float4 bi = sbox[i];
      const float ai = box_area(bi);
      for (int j = i + 1 + lane; j < e0; j += 64)
        if (keep[j] && box_iou(bi, ai, sbox[j]) > p.iou) keep[j] = 0;
    }
  }
  __syncthreads();
  for (int q = tid; q < n; q += kNmsThreads)
    if (keep[q]) {
      const int sp = p.part_pos[(size_t)b * nmax + q];
      atomicOr(&kbits[sp >> 5], 1u << (sp & 31));
    }
  __syncthreads();
  // kept detections in sorted order: contiguous ranges per thread, block scan
  const int per = (n + kNmsThreads - 1) / kNmsThreads;
  const int q0 = tid * per, q1 = min(n, q0 + per);
  int mine = 0;
  for (int q = q0; q < q1; ++q) mine += (kbits[q >> 5] >> (q & 31)) & 1;
  const int upto = block_scan(mine, wsum);
  if (tid == kNmsThreads - 1) {
    const int first = atomicAdd(p.cursor, upto);
    sn[2] = first;
    cnt[0] = n;
    cnt[1] = upto;
    cnt[2] = 0;
    cnt[3] = first;
  }
  __syncthreads();
  int k = sn[2] + upto - mine;
  for (int q = q0; q < q1; ++q)
    if ((kbits[q >> 5] >> (q & 31)) & 1) {
      const int a = p.sorted_anchor[(size_t)b * nmax + q];
      p.kept[k].det = p.det[(size_t)b * A + a];
      p.kept[k].pos = q;
      ++k;
    }
}

// Whether the tiles are expected to be done before a thread per anchor, in
// microseconds: their workgroups, each of which has a start and costs by its
// channels however few its anchors are, against the waves that walk every
// channel of their anchors (and a side's logits three times).  Fitted (14-30%) to
// 12 heads of 6 to 144 channels on 12 batches of 1 to 20000 images with 1 to
// 8400 anchors, both kernels timed at each; the thread has the benefit of the
// doubt, which leaves the choice at most 1.2x from it.  20000 images of 3
// anchors, 6 channels in f32: 18.5 against 67 us (1 x 8400 of 144: 47 against
// 12); 32 of 8400 anchors, 6 channels 7.4 against 10.5 us.
bool tail_by_tiles(int dtype, int n, int anchors, int tiles, int reg_max, int chans) {
  const float k = (float)n / 1000.0f, wg = k * (float)tiles, all = k * (float)anchors, ch = (float)chans;
  const float blocks = k * (float)((anchors + 255) / 256), waves = k * (float)((anchors + 63) / 64);
  const bool h = dtype == F16;
  const float tile = h ? 6.6f + wg * (0.75f + 0.0354f * ch) + 0.00029f * all * ch + 0.0051f * ch
                       : 6.5f + wg * (0.82f + 0.0390f * ch) + 0.00093f * all * ch + 0.0073f * ch;
  const float thread = h ? 3.5f + 0.22f * blocks + 0.0578f * waves * ch + 0.0007f * all * ch + 0.1925f * ch +
                               0.118f * waves * (float)reg_max
                         : 4.0f + 0.0566f * waves * ch + 0.0027f * all * ch + 0.1621f * ch +
                               0.083f * waves * (float)reg_max;
  return 1.2f * tile <= thread;
}

}  // namespace

void launch_detect_tail(hipStream_t st, int dtype, const DetectTailArgs& t, float* out, int n) {
  TailLevels L{};
  if (t.levels < 1 || t.levels > 4) fail(-2, "detect tail: 1 to 4 levels");
  int a = 0;
  for (int s = 0; s < t.levels; ++s) {
    L.x[s] = t.x[s];
    L.h[s] = t.h[s];
    L.w[s] = t.w[s];
    L.pix[s] = t.pix[s];
    L.stride[s] = t.stride[s];
    L.start[s] = a;
    a += t.h[s] * t.w[s];
  }
  L.levels = t.levels;
  L.A = a;
  if (dtype != F16 && dtype != F32) fail(-2, "detect tail: f16 or f32 inputs");
  // The tile kernel reads dwords: f16 channels in pairs on 4-byte addresses,
  // 64 anchors' dwords within its loads of 256 threads.
  const int es = dtype == F16 ? 2 : 4, chans = 4 * t.reg_max + t.nc;
  const size_t lds = ((size_t)kTailAnchors * (chans | 1) + 4 * kTailAnchors) * 4;
  int tiles = 0;
  bool tile = (chans * es) % 4 == 0 && chans * es / 4 * kTailAnchors <= tail_loads(dtype == F16) * 256;
  for (int s = 0; s < t.levels; ++s) {
    L.tile0[s] = tiles;
    tiles += (t.h[s] * t.w[s] + kTailAnchors - 1) / kTailAnchors;
    tile = tile && (t.pix[s] * es) % 4 == 0 && (uintptr_t)t.x[s] % 4 == 0;
  }
  if (tile && tail_by_tiles(dtype, n, a, tiles, t.reg_max, chans)) {
    auto* k = dtype == F16 ? (t.reg_max == 16 ? detect_tail_tile_kernel<true, 16> : detect_tail_tile_kernel<true, 0>)
                           : (t.reg_max == 16 ? detect_tail_tile_kernel<false, 16> : detect_tail_tile_kernel<false, 0>);
    hipLaunchKernelGGL(k, dim3((unsigned)tiles, (unsigned)n), dim3(256), lds, st, L, out, t.nc, t.reg_max);
  } else {
    auto* k = dtype == F16 ? detect_tail_kernel<true> : detect_tail_kernel<false>;
    hipLaunchKernelGGL(k, dim3((unsigned)((a + 255) / 256), (unsigned)n), dim3(256), 0, st, L, out, t.nc, t.reg_max);
  }
  DW_HIP(hipGetLastError());
}

size_t pp_nms_lds_bytes(int nmax) { return nms_lds_bytes(nmax) + kNmsThreads / 64 * sizeof(int); }

void launch_yolo_postprocess(hipStream_t st, const PostprocessArgs& a) {
  PPArgs p{};
  p.raw = a.raw;
  p.nc = a.nc;
  p.A = a.A;
  p.sx = a.sx;
  p.sy = a.sy;
  p.img_w = a.img_w;
  p.img_h = a.img_h;
  p.conf = a.conf;
  p.iou = a.iou;
  p.agnostic = a.agnostic;
  p.nmax = a.nmax;
  if (a.A > 16384 || (size_t)16 * a.nmax < (size_t)16384 * 8) fail(-2, "postprocess: too many anchors to sort");
  if (a.nmax > kPPMaxCandidates) fail(-1, "postprocess: capacity");
  p.keys = a.keys;
  p.det = a.det;
  p.sorted_anchor = a.sorted_anchor;
  p.part_pos = a.part_pos;
  p.kept = a.kept;
  p.counts = a.counts;
  p.cursor = a.cursor;
  hipLaunchKernelGGL(pp_candidates_kernel, dim3((unsigned)((a.A + 255) / 256), (unsigned)a.n), dim3(256), 0, st,
                     p);
  DW_HIP(hipGetLastError());
  hipLaunchKernelGGL(pp_nms_kernel, dim3((unsigned)a.n), dim3(kNmsThreads), nms_lds_bytes(a.nmax), st, p);
  DW_HIP(hipGetLastError());
}

}  // namespace dw
