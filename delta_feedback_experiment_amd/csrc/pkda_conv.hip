// Fused Q/K/V short convolution + SiLU + per-head L2 normalisation for gfx950,
// forward and backward: the producer of the PKDA recurrence's q, k, v.
//
// Reference: delta_feedback::pkda_qkv_conv and its backward
// (delta_feedback_experiment/fla_ops.py:134-249); the same function in
// portable form is PreconditionedKDA._causal_conv + _l2norm
// (delta_feedback_experiment/pkda.py:37-44,197-220,290-316).  Per channel c of
// x [B, T, C] and token t, with W taps and zero history before t = 0:
//
//   a[t, c] = sum_{w < W} weight[c, w] x[t - (W - 1) + w, c]
//   y[t, c] = silu(a[t, c])
//   out     = y / sqrt(sum_{head} y^2 + eps)   for c < norm_channels (q and k)
//           = y                                 otherwise (v)
//
// all in FP32, cast once to the output dtype; channels [0, P), [P, 2P),
// [2P, 3P) leave as the three slabs q, k, v [B, T, P].
//
// Layout and threads: one thread owns 4 consecutive channels (8 bytes of a
// BF16 token row, 512 bytes a wave) and walks a tile of tokens with the W - 1
// previous rows in registers, so each row of x is read once (plus a W - 1 row
// halo per tile) with fully coalesced loads, a group of four rows ahead of the
// one computed; whole groups run without a row test, so the windows slide by
// renaming and not by register moves.  The head's sum of squares is a DPP
// reduction over the head_dim / 4 lanes that share the head; the forward's and
// the token kernel's add as lanes of eight channels would, so that Q and K do not
// depend on the split (five operations a row, 1 to 2 % of the forward).  The backward
// recomputes a and y for its tile plus the W - 1 rows after it (the rows whose
// gradient reaches the tile's x).  dw is summed per tile in registers and the
// tiles in a fixed order by a second kernel: deterministic.
//
// Bounds: HBM, with the VALU close behind (90 operations a thread and row
// forward, 125 backward).  B8 T4096, 3 x 1,024 channels, W = 4, BF16: forward
// 82 us for 403 MB (4.9 TB/s, the card's copy rate 5.2), backward 144 for 604
// MB and 25 of dw partials (4.4 TB/s, 112 VGPRs, four waves a SIMD).  Eight
// channels a thread, row tests and IEEE divisions in the sigmoids took 105
// and 184 (227 VGPRs, two waves); eight channels in today's form 80 and 190,
// but 15.4 us against 14 on 3 rows of 1,000 tokens.
#include "pkda_common.h"
#include "pkda_reduce.h"

#include <type_traits>

namespace pkda {
namespace {

// A workgroup's piece of a row is 2 KB of BF16 and 4 KB of FP32 with 256 threads,
// contiguous; half of that costs FP32 6 to 10 % (8 x 4,096 rows of 3,072 channels,
// forward 169 us against 154, backward 284 against 264; 8 x 4,000 rows 162
// against 150 and 296 against 266), BF16 up to 1 %.
constexpr int kConvThreads = 256;
constexpr int kCh = 4;          // channels of a thread
constexpr int kGroup = 4;       // token rows loaded together
constexpr int kTileFwd = 32;    // longest tiles, tokens
constexpr int kTileBwd = 64;
constexpr int kFillWaves = 4096;  // four waves on every SIMD

// Tokens of a workgroup's tile: the longest of long_tile, long_tile / 2 and
// long_tile / 4 whose waves fill the chip, else the last.  A long tile reads
// and recomputes fewer halo rows, a short one puts more waves on a small
// call: one row of 200 tokens, 768 channels, goes 4.6 us forward (tile 8) against
// 6.6 (tile 16), 10.0 backward (tile 16) against 16.0 (tile 32); 3 rows of 1,000,
// 3,072 channels, 14 either way and 21 to 23 against 27; 8 rows of 4,096,
// 6,144 channels, take the long tiles, 190 and 306 us, 3 % faster than half.
inline int conv_tile(int B, int T, int C, int long_tile) {
  const int64_t waves = (C + 64 * kCh - 1) / (64 * kCh);
  int tile = long_tile;
  while (tile > long_tile / 4 && waves * B * ((T + tile - 1) / tile) < kFillWaves) tile /= 2;
  return tile;
}

struct ConvParams {
  const void* x;
  const void* weight;
  int w_dtype;
  const void* dq;  // backward: gradients of the three slabs
  const void* dk;
  const void* dv;
  void* q;         // forward outputs
  void* k;
  void* v;
  void* dx;        // backward outputs
  float* dw_part;  // [tiles, C, W] FP32
  void* dw;        // [C, W] in w_dtype
  const int32_t* slot;   // cached rows: row -> history slot, or null
  const void* hist_in;   // [pool, W - 1, C] or null (zero history)
  void* hist_out;        // [pool, W - 1, C] or null
  int B, T, C, P, head_dim, norm_channels, x_dtype;
  float eps;
  int tile, tiles_per_row;
};

// CH elements kept as raw 16-byte pieces or one 8-byte piece (unpacked when
// used), so a prefetched row costs a register for each two BF16 elements.
template <typename T, int CH>
struct RawRow {
  static constexpr int N = CH * (int)sizeof(T) / 4;  // 32-bit words
  static_assert(N == 2 || N % 4 == 0, "8 bytes or whole 16-byte pieces");
  uint32_t r[N];
  __device__ __forceinline__ void load(const T* p) {
    if constexpr (N == 2) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      r[0] = v.x; r[1] = v.y;
    } else {
#pragma unroll
      for (int i = 0; i < N / 4; ++i) {
        const uint4 v = reinterpret_cast<const uint4*>(p)[i];
        r[4 * i] = v.x; r[4 * i + 1] = v.y; r[4 * i + 2] = v.z; r[4 * i + 3] = v.w;
      }
    }
  }
  __device__ __forceinline__ void store(T* p) const {
    if constexpr (N == 2) {
      *reinterpret_cast<uint2*>(p) = make_uint2(r[0], r[1]);
    } else {
#pragma unroll
      for (int i = 0; i < N / 4; ++i)
        reinterpret_cast<uint4*>(p)[i] = make_uint4(r[4 * i], r[4 * i + 1], r[4 * i + 2], r[4 * i + 3]);
    }
  }
  __device__ __forceinline__ void unpack(float* x) const {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        x[2 * i] = __uint_as_float(r[i] << 16);
        x[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
      }
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = __uint_as_float(r[i]);
    }
  }
  __device__ __forceinline__ void pack(const float* x) {
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int i = 0; i < N; ++i)
        r[i] = static_cast<uint32_t>(f32_to_bf16(x[2 * i])) | (static_cast<uint32_t>(f32_to_bf16(x[2 * i + 1])) << 16);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) r[i] = __float_as_uint(x[i]);
    }
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = 0u;
  }
};
template <typename T, int CH>
__device__ __forceinline__ void store_row(T* p, const float* x) {
  RawRow<T, CH> v;
  v.pack(x);
  v.store(p);
}

// Sum over the G lanes of one head (G a power of two, lanes aligned to G;
// the lanes of a head are active together).
template <int G>
__device__ __forceinline__ float head_sum(float x) {
  if constexpr (G <= 16) return lane_group_sum<G>(x);
  else return lane_half_sum(x);
}

// The slab (q, k or v) and the offset inside it of channel c.
template <typename T>
__device__ __forceinline__ T* slab_ptr(void* q, void* k, void* v, int P, int c, int64_t row, int& off) {
  const int s = c / P;
  off = c - s * P;
  T* base = static_cast<T*>(s == 0 ? q : s == 1 ? k : v);
  return base + row * P;
}
template <typename T>
__device__ __forceinline__ const T* slab_ptr(const void* q, const void* k, const void* v, int P, int c, int64_t row,
                                             int& off) {
  const int s = c / P;
  off = c - s * P;
  const T* base = static_cast<const T*>(s == 0 ? q : s == 1 ? k : v);
  return base + row * P;
}

// The CH W taps of this thread's channels are contiguous: one branch on the
// dtype (uniform) around straight-line loads, so they go out together (a
// per-element dtype test made each load wait for the one before).
template <int CH, int W>
__device__ __forceinline__ void load_weights(const ConvParams& p, int c0, float (&wt)[CH][W]) {
  const int64_t base = (int64_t)c0 * W;
  if (p.w_dtype == PKDA_BF16) {
    const bf16_t* w8 = static_cast<const bf16_t*>(p.weight) + base;
#pragma unroll
    for (int j = 0; j < CH; ++j)
#pragma unroll
      for (int w = 0; w < W; ++w) wt[j][w] = bf16_to_f32(w8[j * W + w]);
  } else {
    const float* w8 = static_cast<const float*>(p.weight) + base;
#pragma unroll
    for (int j = 0; j < CH; ++j)
#pragma unroll
      for (int w = 0; w < W; ++w) wt[j][w] = w8[j * W + w];
  }
}

// ---------------------------------------------------------------------------
// forward
// ---------------------------------------------------------------------------
template <typename T, int W, int D>
__global__ __launch_bounds__(kConvThreads) void qkv_conv_fwd_kernel(ConvParams p) {
  constexpr int CH = kCh, G = D / CH;
  const int tpr = p.tiles_per_row;
  const int b = blockIdx.x / tpr;
  const int t0 = (blockIdx.x - b * tpr) * p.tile;
  const int t1 = min(t0 + p.tile, p.T);
  const int c0 = (blockIdx.y * kConvThreads + threadIdx.x) * CH;
  if (c0 >= p.C) return;  // whole heads: the lanes of one head leave together
  const bool norm = c0 < p.norm_channels;
  float wt[CH][W];
  load_weights<CH, W>(p, c0, wt);
  const T* xs = static_cast<const T*>(p.x) + (int64_t)b * p.T * p.C + c0;
  float hist[W > 1 ? W - 1 : 1][CH];  // x at t - (W - 1) .. t - 1
  {
    // the halo rows load unconditionally (row 0 stands in before the row's
    // start) and are replaced below where t < 0, so no branch holds them back
    RawRow<T, CH> hr[W > 1 ? W - 1 : 1];
#pragma unroll
    for (int w = 0; w < W - 1; ++w) hr[w].load(xs + (int64_t)max(t0 - (W - 1) + w, 0) * p.C);
#pragma unroll
    for (int w = 0; w < W - 1; ++w) {
      const int t = t0 - (W - 1) + w;
      if (t >= 0) {
        hr[w].unpack(hist[w]);
      } else if (p.hist_in) {  // the row's cached projections before its first token
        const int64_t sb = p.slot ? p.slot[b] : b;
        RawRow<T, CH> h;
        h.load(static_cast<const T*>(p.hist_in) + (sb * (W - 1) + (W - 1) + t) * p.C + c0);
        h.unpack(hist[w]);
      } else {
#pragma unroll
        for (int j = 0; j < CH; ++j) hist[w][j] = 0.f;
      }
    }
  }
  int off;
  T* out = slab_ptr<T>(p.q, p.k, p.v, p.P, c0, (int64_t)b * p.T, off) + off;
  // tokens in groups of kGroup rows, the next group's loads in flight while
  // the current one computes
  using Row = RawRow<T, CH>;
  Row xa[kGroup], xb[kGroup];
  auto load_group = [&](int tg, Row (&dst)[kGroup]) {  // rows past the tile clamp (never used)
#pragma unroll
    for (int i = 0; i < kGroup; ++i) dst[i].load(xs + (int64_t)min(tg + i, t1 - 1) * p.C);
  };
  auto step = [&](int t, const Row& xr) {
    float xt[CH], y[CH];
    xr.unpack(xt);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      float a = wt[j][W - 1] * xt[j];
#pragma unroll
      for (int w = 0; w < W - 1; ++w) a += wt[j][w] * hist[w][j];
      y[j] = a * sigmoid_fast(a);
    }
    if (norm) {
      const float r = rsqrtf(lane_pair_squares<G>(y) + p.eps);
#pragma unroll
      for (int j = 0; j < CH; ++j) y[j] *= r;
    }
    store_row<T, CH>(out + (int64_t)t * p.P, y);
#pragma unroll
    for (int w = 0; w + 1 < W - 1; ++w)
#pragma unroll
      for (int j = 0; j < CH; ++j) hist[w][j] = hist[w + 1][j];
    if (W > 1)
#pragma unroll
      for (int j = 0; j < CH; ++j) hist[W > 1 ? W - 2 : 0][j] = xt[j];
  };
  load_group(t0, xa);
  int tg = t0;
  for (; tg + kGroup <= t1; tg += kGroup) {  // whole groups: no row test
    load_group(tg + kGroup, xb);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) step(tg + i, xa[i]);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) xa[i] = xb[i];
  }
#pragma unroll
  for (int i = 0; i + 1 < kGroup; ++i)  // a row's last, partial group
    if (tg + i < t1) step(tg + i, xa[i]);
  // a row that is one tile (a decode token, a short prompt) leaves its
  // history here: hist holds its last W - 1 rows of history ++ x, and this
  // thread read its slot's old history at the start (in place is safe)
  if constexpr (W > 1) {
    if (p.hist_out && tpr == 1) {
      const int64_t sb = p.slot ? p.slot[b] : b;
#pragma unroll
      for (int w = 0; w < W - 1; ++w) store_row<T, CH>(static_cast<T*>(p.hist_out) + (sb * (W - 1) + w) * p.C + c0, hist[w]);
    }
  }
}

// ---------------------------------------------------------------------------
// backward
//   n = y r, r = (sum y^2 + eps)^-1/2:  dy = r (dn - n sum(n dn))   (q, k)
//   da = dy silu'(a),  silu'(a) = s (1 + a (1 - s)),  s = sigmoid(a)
//   dx[t] = sum_w weight[w] da[t + W - 1 - w],  dw[w] += da[t] x[t - (W - 1) + w]
// ---------------------------------------------------------------------------
template <typename T, int W, int D>
__global__ __launch_bounds__(kConvThreads) void qkv_conv_bwd_kernel(ConvParams p) {
  constexpr int CH = kCh, G = D / CH;
  const int b = blockIdx.x / p.tiles_per_row;
  const int tile = blockIdx.x;
  const int t0 = (blockIdx.x - b * p.tiles_per_row) * p.tile;
  const int t1 = min(t0 + p.tile, p.T);
  const int c0 = (blockIdx.y * kConvThreads + threadIdx.x) * CH;
  if (c0 >= p.C) return;
  const bool norm = c0 < p.norm_channels;
  float wt[CH][W];
  load_weights<CH, W>(p, c0, wt);
  const T* xs = static_cast<const T*>(p.x) + (int64_t)b * p.T * p.C + c0;
  int off;
  const T* dn_base = slab_ptr<T>(p.dq, p.dk, p.dv, p.P, c0, (int64_t)b * p.T, off) + off;
  T* dxs = static_cast<T*>(p.dx) + (int64_t)b * p.T * p.C + c0;

  float hist[W][CH];   // x at t - (W - 1) .. t (hist[W - 1] = x[t] once loaded)
  float dwin[W][CH];   // da at t - (W - 1) .. t
  float dw[CH][W];
#pragma unroll
  for (int w = 0; w < W; ++w)
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      dwin[w][j] = 0.f;
      dw[j][w] = 0.f;
    }
  {
    // halo rows unconditionally (row 0 stands in before the row's start, then zeroed)
    RawRow<T, CH> hr[W > 1 ? W - 1 : 1];
#pragma unroll
    for (int w = 0; w < W - 1; ++w) hr[w].load(xs + (int64_t)max(t0 - (W - 1) + w, 0) * p.C);
#pragma unroll
    for (int w = 0; w < W - 1; ++w) {
      hr[w].unpack(hist[w]);
      if (t0 - (W - 1) + w < 0)
#pragma unroll
        for (int j = 0; j < CH; ++j) hist[w][j] = 0.f;
    }
  }
  using Row = RawRow<T, CH>;
  Row xa[kGroup], xb[kGroup], na[kGroup], nb[kGroup];
  auto load_group = [&](int tg, Row (&dx_)[kGroup], Row (&dn_)[kGroup]) {
    // rows past the row's end clamp (never used): no branch holds a load back
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      const int t = min(tg + i, p.T - 1);
      dx_[i].load(xs + (int64_t)t * p.C);
      dn_[i].load(dn_base + (int64_t)t * p.P);
    }
  };
  // row t: its da (zero when not LIVE, past the row's end), its share of dw
  // when it is the tile's own, and dx of row t - (W - 1), whose da are then
  // all known
  auto step = [&](auto live, auto own, int t, const Row& xr, const Row& nr) {
    float da[CH];
    if constexpr (decltype(live)::value) {
      xr.unpack(hist[W - 1]);
      float dn[CH];
      nr.unpack(dn);
      float y[CH], slope[CH];  // silu(a) and silu'(a) = s + y (1 - s)
      float ss = 0.f;
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        float a = wt[j][0] * hist[0][j];
#pragma unroll
        for (int w = 1; w < W; ++w) a += wt[j][w] * hist[w][j];
        const float sg = sigmoid_fast(a);
        y[j] = a * sg;
        slope[j] = sg + y[j] * (1.f - sg);
        ss += y[j] * y[j];
      }
      if (norm) {
        // dy = r (dn - n nd) with n = y r, nd = sum n dn = r sum y dn
        const float r = rsqrtf(head_sum<G>(ss) + p.eps);
        float yd = 0.f;
#pragma unroll
        for (int j = 0; j < CH; ++j) yd += y[j] * dn[j];
        const float f = r * r * (r * head_sum<G>(yd));
#pragma unroll
        for (int j = 0; j < CH; ++j) dn[j] = r * dn[j] - y[j] * f;
      }
#pragma unroll
      for (int j = 0; j < CH; ++j) da[j] = dn[j] * slope[j];
      if constexpr (decltype(own)::value) {
#pragma unroll
        for (int j = 0; j < CH; ++j)
#pragma unroll
          for (int w = 0; w < W; ++w) dw[j][w] += da[j] * hist[w][j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < CH; ++j) da[j] = 0.f;
    }
    // slide the windows: dwin holds da[t - (W - 1) .. t]
#pragma unroll
    for (int w = 0; w + 1 < W; ++w)
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        dwin[w][j] = dwin[w + 1][j];
        hist[w][j] = hist[w + 1][j];
      }
#pragma unroll
    for (int j = 0; j < CH; ++j) dwin[W - 1][j] = da[j];
    const int s = t - (W - 1);
    if (s >= t0) {
      float dx[CH];
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        float acc = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) acc += wt[j][w] * dwin[W - 1 - w][j];
        dx[j] = acc;
      }
      store_row<T, CH>(dxs + (int64_t)s * p.C, dx);
    }
  };
  static_assert(W - 1 <= kGroup, "the group after the tile holds its halo rows");
  using Yes = std::true_type;
  using No = std::false_type;
  load_group(t0, xa, na);
  int tg = t0;
  for (; tg + kGroup <= t1; tg += kGroup) {  // whole groups: no row test
    load_group(tg + kGroup, xb, nb);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) step(Yes{}, Yes{}, tg + i, xa[i], na[i]);
#pragma unroll
    for (int i = 0; i < kGroup; ++i) {
      xa[i] = xb[i];
      na[i] = nb[i];
    }
  }
  const int rem = t1 - tg;  // a row's last, partial group: its tile ends the row
#pragma unroll
  for (int i = 0; i + 1 < kGroup; ++i)
    if (i < rem) step(Yes{}, Yes{}, tg + i, xa[i], na[i]);
  // the W - 1 rows after the tile, whose da reach its dx
#pragma unroll
  for (int i = 0; i < W - 1; ++i) {
    if (t1 + i < p.T) step(Yes{}, No{}, t1 + i, xa[i], na[i]);  // rem == 0: the group holds them
    else step(No{}, No{}, t1 + i, xa[i], na[i]);
  }
  float* part = p.dw_part + ((int64_t)tile * p.C + c0) * W;
#pragma unroll
  for (int j = 0; j < CH; ++j)
#pragma unroll
    for (int w = 0; w < W; ++w) part[j * W + w] = dw[j][w];
}

// ---------------------------------------------------------------------------
// decode tokens: rows of one token, each continuing its slot's history.  A
// thread owns 4 channels of one row: it loads its W - 1 history rows, new
// projection row and (last: the rows' loads wait for the slot) weights before
// computing; out = the normalised silu(conv),
// and the slot's history shifts by one row in place (each thread reads its
// channels' rows before writing them).  Bound by the latency of one round of
// loads, so a row a thread: 256 rows of 3 x 4,096 channels, histories among 512
// slots, 12 us, 4 of 3 x 1,024 3.3 (two rows a thread 10 and 30 % more; eight
// rows of eight channels, the earlier form, 18 and 5.5).
// ---------------------------------------------------------------------------
template <typename T, int W, int D>
__global__ __launch_bounds__(kConvThreads) void qkv_conv_token_kernel(ConvParams p) {
  constexpr int CH = kCh, G = D / CH;
  const int c0 = (blockIdx.y * kConvThreads + threadIdx.x) * CH;
  if (c0 >= p.C) return;
  const bool norm = c0 < p.norm_channels;
  const int b = blockIdx.x;
  const int64_t sb = p.slot ? p.slot[b] : b;
  RawRow<T, CH> hr[W - 1], xr;
  xr.load(static_cast<const T*>(p.x) + (int64_t)b * p.C + c0);
#pragma unroll
  for (int w = 0; w < W - 1; ++w) {
    if (p.hist_in) {
      hr[w].load(static_cast<const T*>(p.hist_in) + (sb * (W - 1) + w) * p.C + c0);
    } else {
      hr[w].zero();
    }
  }
  float wt[CH][W];
  load_weights<CH, W>(p, c0, wt);
  float xt[CH], hist[W - 1][CH];
  xr.unpack(xt);
#pragma unroll
  for (int w = 0; w < W - 1; ++w) hr[w].unpack(hist[w]);
  float y[CH];
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    float a = wt[j][W - 1] * xt[j];
#pragma unroll
    for (int w = 0; w < W - 1; ++w) a += wt[j][w] * hist[w][j];
    y[j] = a * sigmoid_fast(a);
  }
  if (norm) {
    const float rn = rsqrtf(lane_pair_squares<G>(y) + p.eps);
#pragma unroll
    for (int j = 0; j < CH; ++j) y[j] *= rn;
  }
  int off;
  T* out = slab_ptr<T>(p.q, p.k, p.v, p.P, c0, (int64_t)b, off) + off;
  store_row<T, CH>(out, y);
  if (p.hist_out) {
    T* ho = static_cast<T*>(p.hist_out) + sb * (W - 1) * p.C + c0;
#pragma unroll
    for (int w = 0; w + 1 < W - 1; ++w) store_row<T, CH>(ho + (int64_t)w * p.C, hist[w + 1]);
    store_row<T, CH>(ho + (int64_t)(W - 2) * p.C, xt);
  }
}

// ---------------------------------------------------------------------------
// cached rows longer than one forward tile: the history left for the next
// call, the last W - 1 rows of history ++ x.  One thread per 4 channels of
// one row reads every row it needs before writing any, so history_out may
// alias history_in; it runs after the forward kernel (whose first tile of a
// row reads history_in) on the same stream.
// ---------------------------------------------------------------------------
template <typename T, int W>
__global__ __launch_bounds__(kConvThreads) void qkv_conv_history_kernel(ConvParams p) {
  constexpr int CH = kCh;
  const int b = blockIdx.x;
  const int c0 = (blockIdx.y * kConvThreads + threadIdx.x) * CH;
  if (c0 >= p.C) return;
  const int64_t sb = p.slot ? p.slot[b] : b;
  const T* xs = static_cast<const T*>(p.x) + (int64_t)b * p.T * p.C + c0;
  RawRow<T, CH> rows[W - 1];
#pragma unroll
  for (int j = 0; j < W - 1; ++j) {
    const int t = p.T - (W - 1) + j;  // position relative to the row's first token
    if (t >= 0) {
      rows[j].load(xs + (int64_t)t * p.C);
    } else if (p.hist_in) {
      rows[j].load(static_cast<const T*>(p.hist_in) + (sb * (W - 1) + (W - 1) + t) * p.C + c0);
    } else {
      rows[j].zero();
    }
  }
#pragma unroll
  for (int j = 0; j < W - 1; ++j) rows[j].store(static_cast<T*>(p.hist_out) + (sb * (W - 1) + j) * p.C + c0);
}

template <typename T, int W, int D>
int launch_conv(const ConvParams& p, bool backward, hipStream_t s) {
  constexpr int CB = kConvThreads * kCh;  // channels of a workgroup
  const int cblocks = (p.C + CB - 1) / CB;
  const dim3 grid(p.B * p.tiles_per_row, cblocks);
  if (!backward) {
    if constexpr (W > 1) {
      if (p.T == 1 && (p.hist_in || p.hist_out)) {  // decode tokens
        hipLaunchKernelGGL((qkv_conv_token_kernel<T, W, D>), dim3(p.B, cblocks), dim3(kConvThreads), 0, s, p);
        return launch_status("pkda_qkv_conv_fwd(token)");
      }
    }
    if (p.T > 0) {
      hipLaunchKernelGGL((qkv_conv_fwd_kernel<T, W, D>), grid, dim3(kConvThreads), 0, s, p);
      if (int st = launch_status("pkda_qkv_conv_fwd")) return st;
    }
    if constexpr (W > 1) {
      if (p.hist_out && p.tiles_per_row != 1) {  // else the forward kernel wrote it
        hipLaunchKernelGGL((qkv_conv_history_kernel<T, W>), dim3(p.B, cblocks), dim3(kConvThreads), 0, s, p);
        return launch_status("pkda_qkv_conv_fwd(history)");
      }
    }
    return 0;
  }
  hipLaunchKernelGGL((qkv_conv_bwd_kernel<T, W, D>), grid, dim3(kConvThreads), 0, s, p);
  if (int st = launch_status("pkda_qkv_conv_bwd")) return st;
  return launch_column_sums(column_sum(p.dw_part, p.B * p.tiles_per_row, p.C * W, p.C * W, p.dw, p.w_dtype), {}, s,
                            "pkda_qkv_conv_bwd(dw)");
}

template <typename T, int D>
int dispatch_w(const ConvParams& p, int W, bool backward, hipStream_t s) {
  switch (W) {
    case 1: return launch_conv<T, 1, D>(p, backward, s);
    case 2: return launch_conv<T, 2, D>(p, backward, s);
    case 3: return launch_conv<T, 3, D>(p, backward, s);
    case 4: return launch_conv<T, 4, D>(p, backward, s);
    default: set_error("conv_size %d not built (1..4)", W); return PKDA_EUNSUPPORTED;
  }
}

template <typename T>
int dispatch(const ConvParams& p, int W, bool backward, hipStream_t s) {
  switch (p.head_dim) {
    case 32: return dispatch_w<T, 32>(p, W, backward, s);
    case 64: return dispatch_w<T, 64>(p, W, backward, s);
    case 128: return dispatch_w<T, 128>(p, W, backward, s);
    default: set_error("head_dim %d not built (32, 64, 128)", p.head_dim); return PKDA_EUNSUPPORTED;
  }
}

int conv_call(const pkda_qkv_conv_args* a, void* stream, bool backward) {
  PKDA_REQUIRE(a != nullptr, PKDA_EINVAL, "null args");
  PKDA_REQUIRE(a->struct_size == (int32_t)sizeof(pkda_qkv_conv_args), PKDA_EINVAL, "pkda_qkv_conv_args size mismatch");
  PKDA_REQUIRE(a->dtype == PKDA_F32 || a->dtype == PKDA_BF16, PKDA_EUNSUPPORTED, "dtype %d", a->dtype);
  PKDA_REQUIRE(a->w_dtype == PKDA_F32 || a->w_dtype == PKDA_BF16, PKDA_EUNSUPPORTED, "weight dtype %d", a->w_dtype);
  PKDA_REQUIRE(a->batch >= 0 && a->seqlen >= 0 && a->width > 0, PKDA_EINVAL, "sizes");
  PKDA_REQUIRE(a->head_dim == 32 || a->head_dim == 64 || a->head_dim == 128, PKDA_EUNSUPPORTED, "head_dim %d",
               a->head_dim);
  PKDA_REQUIRE(a->width % a->head_dim == 0, PKDA_EINVAL, "slab width %d is not a multiple of head_dim %d", a->width,
               a->head_dim);
  PKDA_REQUIRE(a->norm_channels >= 0 && a->norm_channels <= 3 * a->width && a->norm_channels % a->head_dim == 0,
               PKDA_EINVAL, "norm_channels %d", a->norm_channels);
  PKDA_REQUIRE(a->conv_size >= 1 && a->conv_size <= 4, PKDA_EUNSUPPORTED, "conv_size %d (1..4)", a->conv_size);
  ConvParams p;
  p.B = a->batch;
  p.T = a->seqlen;
  p.P = a->width;
  p.C = 3 * a->width;
  p.head_dim = a->head_dim;
  p.norm_channels = a->norm_channels;
  p.x_dtype = a->dtype;
  p.eps = a->eps;
  p.tile = backward ? conv_tile(p.B, p.T, p.C, kTileBwd) : conv_tile(p.B, p.T, p.C, kTileFwd);
  p.tiles_per_row = (a->seqlen + p.tile - 1) / p.tile;
  p.x = a->x;
  p.weight = a->weight;
  p.w_dtype = a->w_dtype;
  p.q = a->q; p.k = a->k; p.v = a->v;
  p.dq = a->dq; p.dk = a->dk; p.dv = a->dv;
  p.dx = a->dx; p.dw = a->dw; p.dw_part = a->dw_part;
  p.slot = a->slot_idx;
  p.hist_in = a->history_in;
  p.hist_out = a->history_out;
  const bool cached = a->history_in || a->history_out;
  PKDA_REQUIRE(!backward || !cached, PKDA_EUNSUPPORTED, "conv histories are a forward (cached rows) feature");
  PKDA_REQUIRE(!cached || a->conv_size > 1, PKDA_EINVAL, "conv_size 1 keeps no history");
  PKDA_REQUIRE(!a->slot_idx || a->pool_size > 0, PKDA_EINVAL, "slot-indexed histories need pool_size > 0");
  if (p.B == 0 || (p.T == 0 && !(a->history_out && !backward))) {
    PKDA_REQUIRE(!backward || a->dw, PKDA_EINVAL, "null dw");
    return 0;  // an empty batch: nothing to launch (dw is the caller's zeros)
  }
  if (backward) {
    PKDA_REQUIRE(a->x && a->weight && a->dq && a->dk && a->dv && a->dx && a->dw && a->dw_part, PKDA_EINVAL,
                 "null tensor");
  } else {
    PKDA_REQUIRE(p.T == 0 || (a->x && a->weight && a->q && a->k && a->v), PKDA_EINVAL, "null tensor");
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  return a->dtype == PKDA_BF16 ? dispatch<bf16_t>(p, a->conv_size, backward, s)
                               : dispatch<float>(p, a->conv_size, backward, s);
}

}  // namespace
}  // namespace pkda

extern "C" int64_t pkda_qkv_conv_workspace(int32_t batch, int32_t seqlen, int32_t width, int32_t conv_size) {
  const int tile = pkda::conv_tile(batch, seqlen, 3 * width, pkda::kTileBwd);
  const int64_t tiles = (int64_t)batch * ((seqlen + tile - 1) / tile);
  return tiles * 3 * (int64_t)width * conv_size;
}

extern "C" int pkda_qkv_conv_fwd(const pkda_qkv_conv_args* args, void* stream) {
  return pkda::conv_call(args, stream, false);
}

extern "C" int pkda_qkv_conv_bwd(const pkda_qkv_conv_args* args, void* stream) {
  return pkda::conv_call(args, stream, true);
}
