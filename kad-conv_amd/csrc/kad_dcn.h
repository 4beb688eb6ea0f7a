// Shared pieces of the deformable-convolution kernels: tile geometry, sample records and bilinear
// geometry, MFMA fragments per data type, buffer loads, and the fused squeeze-excitation tail.
#pragma once
#include "kad_common.h"

namespace kad {

constexpr int DCN_TILE = 128;                      // output pixels per tile
constexpr int DCN_NOFF = 18;                       // offset channels (2 x 9 taps)
constexpr int DCN_SE_LDS = 48 * 1024;              // fused SE scratch limit (kad_dcn_args.se_*)

enum { MODE_EXT = 0, MODE_FUSED = 1, MODE_PLAIN = 2 };

struct DcnGeom {
  int ho, wo, th, tw, tiles_x, tiles, grid_x, nchunk, cout_pad;
  int fh, fw;        // 3x3 footprint of a tile: (th - 1) * stride + 3 rows, likewise columns
  float inv_tw, inv_fw;
};

// Tile shape for an Ho x Wo output: TH x TW <= tile pixels minimising the
// padded pixel count; ties prefer squarer tiles (smaller halo).
inline void pick_tile(int ho, int wo, int* th_out, int* tw_out, int tile = DCN_TILE) {
  long best = -1;
  int bth = tile / 16, btw = 16;
  for (int tw = 4; tw <= 64; ++tw) {
    const int th = tile / tw;
    if (th < 1) break;
    const long cost = (long)ceil_div(ho, th) * ceil_div(wo, tw) * tile * 64 + (th > tw ? th - tw : tw - th);
    if (best < 0 || cost < best) {
      best = cost;
      bth = th;
      btw = tw;
    }
  }
  *th_out = bth;
  *tw_out = btw;
}

inline DcnGeom make_geom(const kad_dcn_args& a, int ho, int wo, int tile = DCN_TILE) {
  DcnGeom g;
  g.ho = ho;
  g.wo = wo;
  pick_tile(ho, wo, &g.th, &g.tw, tile);
  g.tiles_x = ceil_div(wo, g.tw);
  g.tiles = ceil_div(ho, g.th) * g.tiles_x;
  g.grid_x = round_up(a.n * g.tiles, 8);  // flattened (image, tile), padded to whole XCD rounds
  g.nchunk = ceil_div(a.cin, 32);
  g.cout_pad = round_up(a.cout, 16);
  g.fh = (g.th - 1) * a.stride + 3;
  g.fw = (g.tw - 1) * a.stride + 3;
  g.inv_tw = 1.f / (float)g.tw;
  g.inv_fw = 1.f / (float)g.fw;
  return g;
}

// ---- samples ----------------------------------------------------------------------------------
// The kernels keep a record per (tap, pixel) in LDS: where its top-left corner lies, the corner steps, and
// the four corner weights times the mask (sample_geom), in 16-bit paths as fp16: uint2 {w00 | w01, w10 | w11}.
__device__ __forceinline__ unsigned pack_h2(float a, float b) {
  const half2_t h{(half_t)a, (half_t)b};
  return __builtin_bit_cast(unsigned, h);
}

// ---- A fragment from four corners ------------------------------------------------------------
template <typename T> struct DcnFrag;

template <> struct DcnFrag<half_t> {
  typedef half8_t frag;
  static __device__ __forceinline__ frag blend(const half8_t& v0, const half8_t& v1, const half8_t& v2,
                                               const half8_t& v3, const uint2& w) {
    const half2_t w01 = __builtin_bit_cast(half2_t, w.x), w23 = __builtin_bit_cast(half2_t, w.y);
    frag r = v0 * w01[0];
    r += v1 * w01[1];
    r += v2 * w23[0];
    r += v3 * w23[1];
    return r;
  }
  static __device__ __forceinline__ floatx4 mma(const frag& a, const frag& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

template <> struct DcnFrag<bf16_t> {
  typedef bf16x8_t frag;
  static __device__ __forceinline__ frag blend(const bf16x8_t& v0, const bf16x8_t& v1, const bf16x8_t& v2,
                                               const bf16x8_t& v3, const uint2& w) {
    const half2_t w01 = __builtin_bit_cast(half2_t, w.x), w23 = __builtin_bit_cast(half2_t, w.y);
    const float a = (float)w01[0], b = (float)w01[1], c = (float)w23[0], d = (float)w23[1];
    frag r;
#pragma unroll
    for (int j = 0; j < 8; ++j)
      r[j] = (bf16_t)(a * (float)v0[j] + b * (float)v1[j] + c * (float)v2[j] + d * (float)v3[j]);
    return r;
  }
  static __device__ __forceinline__ floatx4 mma(const frag& a, const frag& b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

struct f32x8 { floatx4 lo, hi; };

template <> struct DcnFrag<float> {
  typedef f32x8 frag;
  // 8 MFMA steps of k=4: step j consumes slot j of every lane group, i.e.
  // k = 8 * group + j on both operands.
  static __device__ __forceinline__ floatx4 mma(const frag& a, const frag& b, floatx4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.lo[j], b.lo[j], c, 0, 0, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.hi[j], b.hi[j], c, 0, 0, 0);
    return c;
  }
};

template <typename T>
__device__ __forceinline__ typename DcnFrag<T>::frag ld8(const T* p) {
  typedef typename DcnFrag<T>::frag F;
  if constexpr (sizeof(T) == 4) {
    F r;
    r.lo = *(const floatx4*)p;
    r.hi = *(const floatx4*)(p + 4);
    return r;
  } else {
    return *(const F*)p;
  }
}

template <typename T>
__device__ __forceinline__ void st8(T* p, const typename DcnFrag<T>::frag& v) {
  if constexpr (sizeof(T) == 4) {
    *(floatx4*)p = v.lo;
    *(floatx4*)(p + 4) = v.hi;
  } else {
    *(typename DcnFrag<T>::frag*)p = v;
  }
}

template <typename T>
__device__ __forceinline__ typename DcnFrag<T>::frag zero8() {
  typedef typename DcnFrag<T>::frag F;
  if constexpr (sizeof(T) == 4) {
    F r;
    r.lo = floatx4{0.f, 0.f, 0.f, 0.f};
    r.hi = r.lo;
    return r;
  } else {
    return F{};
  }
}

// Bilinear geometry of one sample at (py, px) (torchvision's rule): clamped
// top-left corner, corner steps (0 or 1 per axis) and the four weights times m;
// all weights 0 for a dead sample.
__device__ __forceinline__ void sample_geom(float py, float px, float m, int h, int w, int& cy0, int& cx0, int& sy,
                                            int& sx, float* wt) {
  cy0 = cx0 = sy = sx = 0;
  wt[0] = wt[1] = wt[2] = wt[3] = 0.f;
  if (py > -1.f && py < (float)h && px > -1.f && px < (float)w) {
    const float fy = floorf(py), fx = floorf(px);
    const int y0 = (int)fy, x0 = (int)fx, y1 = y0 + 1, x1 = x0 + 1;
    const float ly = py - fy, lx = px - fx, hy = 1.f - ly, hx = 1.f - lx;
    const bool vy0 = y0 >= 0, vy1 = y1 <= h - 1, vx0 = x0 >= 0, vx1 = x1 <= w - 1;
    cy0 = vy0 ? y0 : 0;
    const int cy1 = vy1 ? y1 : h - 1;
    cx0 = vx0 ? x0 : 0;
    const int cx1 = vx1 ? x1 : w - 1;
    sy = cy1 - cy0;
    sx = cx1 - cx0;
    wt[0] = (vy0 && vx0) ? hy * hx * m : 0.f;
    wt[1] = (vy0 && vx1) ? hy * lx * m : 0.f;
    wt[2] = (vy1 && vx0) ? ly * hx * m : 0.f;
    wt[3] = (vy1 && vx1) ? ly * lx * m : 0.f;
  }
}

// ---- buffer loads ------------------------------------------------------------------------------
// A raw buffer load returns 0 for a byte offset at or past the descriptor's
// size, so pieces outside the image (padding ring, channels past Cin, unused
// staging slots) are staged as zeros with no branch; per-thread byte offsets are
// computed once per block and only shifted per channel chunk.
template <typename T>
__device__ __forceinline__ typename DcnFrag<T>::frag buf_ld8(__amdgpu_buffer_rsrc_t r, uint32_t voff) {
  typedef typename DcnFrag<T>::frag F;
  if constexpr (sizeof(T) == 4) {
    F f;
    f.lo = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
    f.hi = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r, voff + 16, 0, 0));
    return f;
  } else {
    return __builtin_bit_cast(F, __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 0));
  }
}

// ---- fused squeeze-excitation of one image ------------------------------------------------------
// Cross-block exchange without fences.  A device-scope release fence writes
// back the whole L2 of the XCD (8 XCDs, each with its own L2), which costs
// microseconds per block; atomic read-modify-writes, by contrast, are
// performed at the memory-side coherence point for every XCD.  So every step
// of the exchange is a relaxed device-scope RMW whose returned value the
// thread waits for (the RMW has then been performed):
//  - each block stores its GAP partials with atomic exchanges and waits;
//  - after a barrier, thread 0 increments the image's arrival counter;
//  - the block that completes the count resets it (exchange with 0) and reads
//    every partial of the image with device-scope atomic loads (coherent across
//    XCDs: they do not return a stale line of the reader's L2).
// se_tail then forms g = se_inv_count * column sums of the [tiles][Cout]
// partials in a fixed order (thread (slice s, channel c) takes tiles s,
// s + nsl, ...; the slices are then added in order), so the result does not
// depend on which block came last; then att = sigmoid(W2 relu(W1 g + b1) + b2)
// with 4 lanes per output and a shuffle reduction.  lds: Cout + hid + THREADS floats (Cout + hid where one
// slice takes every tile: its sums are formed in g itself).
// (dev_load / rmw_store: kad_common.h)

// se_tail_any covers every size; se_tail below the usual ones.
template <int THREADS>
__device__ __forceinline__ void se_tail_any(const float* __restrict__ partial, const float* __restrict__ w1,
                                        const float* __restrict__ b1, const float* __restrict__ w2,
                                        const float* __restrict__ b2, float* __restrict__ att, float inv_count, int C,
                                        int hid, int n, int tiles, float* lds) {
  constexpr int PB = 16;   // loads in flight per thread per batch
  constexpr int LPO = 4;   // lanes per MLP output (shuffle-reduced)
  constexpr int OPP = THREADS / LPO;  // outputs per pass
  const int tid = threadIdx.x;
  float* g = lds;          // [C]
  float* hb = g + C;       // [hid]
  const float* pn = partial + (int64_t)n * tiles * C;
  const int nsl = C < THREADS ? THREADS / C : 1;
  float* red = nsl > 1 ? hb + hid : g;  // [nsl][C]: at most THREADS floats behind hb, or g's own
  for (int e = tid; e < nsl * C; e += THREADS) {
    const int s = e / C, ch = e - s * C;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int t0 = s; t0 < tiles; t0 += PB * nsl) {
      float v[PB];
#pragma unroll
      for (int u = 0; u < PB; ++u) {
        const int t = t0 + u * nsl;
        v[u] = t < tiles ? dev_load(pn + (int64_t)t * C + ch) : 0.f;
      }
#pragma unroll
      for (int u = 0; u < PB; ++u) acc[u & 3] += v[u];
    }
    red[e] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
  __syncthreads();
  for (int ch = tid; ch < C; ch += THREADS) {
    float v = 0.f;
    for (int s = 0; s < nsl; ++s) v += red[s * C + ch];
    g[ch] = v * inv_count;
  }
  __syncthreads();
  const int part = tid & (LPO - 1);
  // out[o] = act(sum_k w[o][k] in[k] + b[o]): LPO lanes per output, each taking k = part, part + LPO, ...
  auto layer = [&](const float* __restrict__ w, const float* __restrict__ b, const float* in, int nin, int nout,
                   bool relu, float* dst) {
    for (int o0 = 0; o0 < nout; o0 += OPP) {
      const int o = o0 + tid / LPO;
      const float* wr = w + (int64_t)(o < nout ? o : 0) * nin;
      float acc = 0.f;
      for (int k0 = part; k0 < nin; k0 += PB * LPO) {
        float wv[PB];
#pragma unroll
        for (int u = 0; u < PB; ++u) {
          const int k = k0 + u * LPO;
          wv[u] = (o < nout && k < nin) ? wr[k] : 0.f;
        }
#pragma unroll
        for (int u = 0; u < PB; ++u) {
          const int k = k0 + u * LPO;
          acc += wv[u] * in[k < nin ? k : 0];
        }
      }
      acc += __shfl_xor(acc, 1);
      acc += __shfl_xor(acc, 2);
      if (o < nout && part == 0) {
        const float v = acc + (b ? b[o] : 0.f);
        dst[o] = relu ? fmaxf(v, 0.f) : sigmoidf_(v);
      }
    }
  };
  layer(w1, b1, g, C, hid, true, hb);
  __syncthreads();
  layer(w2, b2, hb, hid, C, false, att + (int64_t)n * C);
}

// The tail is a chain of round trips to memory, alone on its CU.  Where both weight matrices are small
// (C hid <= 16 THREADS floats, and one fits the LDS beside the partials: C = 90 with 512 threads) they are
// requested at its start, beside the partials, as contiguous 16-byte pieces: read row by row, 4 or 16
// lanes to a row, their 64-byte sectors were each requested several times over, at one sector in 2.4
// clocks.  W1 goes to LDS, W2 waits in registers until layer 1 is done with it.
// LDSF: floats of LDS at lds.
template <int THREADS, int LDSF>
__device__ __forceinline__ void se_tail(const float* __restrict__ partial, const float* __restrict__ w1,
                                        const float* __restrict__ b1, const float* __restrict__ w2,
                                        const float* __restrict__ b2, float* __restrict__ att, float inv_count, int C,
                                        int hid, int n, int tiles, float* lds) {
  constexpr int NP = 4;    // 16-byte pieces of a matrix per thread
  constexpr int PB = 8;    // partials in flight per thread
  constexpr int LPO = 4;   // lanes per MLP output
  const int cw = round_up(C * hid, 4), cp = round_up(C, 4), hp = round_up(hid, 4);
  if (cw > 4 * NP * THREADS || C > THREADS || cw + cp + hp + THREADS > LDSF) {
    se_tail_any<THREADS>(partial, w1, b1, w2, b2, att, inv_count, C, hid, n, tiles, lds);
    return;
  }
  const int tid = threadIdx.x;
  float* wl = lds;        // [C hid]
  float* g = wl + cw;     // [C]
  float* hb = g + cp;     // [hid]
  float* red = hb + hp;   // [nsl][C]
  const __amdgpu_buffer_rsrc_t r1 = make_rsrc(w1, (uint32_t)(C * hid * 4)), r2 = make_rsrc(w2, (uint32_t)(C * hid * 4));
  floatx4 wa[NP], wb[NP];
#pragma unroll
  for (int u = 0; u < NP; ++u)
    wa[u] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r1, (tid + u * THREADS) * 16, 0, 0));
#pragma unroll
  for (int u = 0; u < NP; ++u)
    wb[u] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(r2, (tid + u * THREADS) * 16, 0, 0));
  const int nsl = THREADS / C, s = tid / C, ch = tid - s * C;
  const float* pn = partial + (int64_t)n * tiles * C;
  if (s < nsl) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int t0 = s; t0 < tiles; t0 += PB * nsl) {
      float v[PB];
#pragma unroll
      for (int u = 0; u < PB; ++u) {
        const int t = t0 + u * nsl;
        v[u] = dev_load(pn + (t < tiles ? t : t0) * C + ch);
        if (t >= tiles) v[u] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < PB; ++u) acc[u & 3] += v[u];
    }
    red[tid] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  }
  auto put = [&](const floatx4 (&w)[NP]) {
#pragma unroll
    for (int u = 0; u < NP; ++u)
      if ((tid + u * THREADS) * 4 < cw) *(floatx4*)(wl + (tid + u * THREADS) * 4) = w[u];
  };
  put(wa);
  __syncthreads();
  if (tid < C) {
    float v = 0.f;
    for (int i = 0; i < nsl; ++i) v += red[i * C + tid];
    g[tid] = v * inv_count;
  }
  __syncthreads();
  // layer 0: hb = relu(W1 g + b1); layer 1: att = sigmoid(W2 hb + b2)
  const int part = tid & (LPO - 1);
#pragma unroll 1
  for (int l = 0; l < 2; ++l) {
    const int nin = l ? hid : C, nout = l ? C : hid;
    const float* in = l ? hb : g;
    const float* b = l ? b2 : b1;
#pragma unroll 1
    for (int o = tid / LPO; o < round_up(nout, THREADS / LPO); o += THREADS / LPO) {
      const int oc = o < nout ? o : nout - 1;
      const float bias = b ? b[oc] : 0.f;
      float acc = 0.f;
#pragma unroll 8
      for (int k = part; k < nin; k += LPO) acc += wl[oc * nin + k] * in[k];
      acc += __shfl_xor(acc, 1);
      acc += __shfl_xor(acc, 2);
      if (part == 0 && o < nout) {
        if (l)
          att[(int64_t)n * C + o] = sigmoidf_(acc + bias);
        else
          hb[o] = fmaxf(acc + bias, 0.f);
      }
    }
    __syncthreads();
    if (l == 0) {
      put(wb);
      __syncthreads();
    }
  }
}

// Several independent problems of one instantiation (same dtype, mode and column-fragment count)
// in one grid: problem p owns blocks [start[p], start[p + 1]) (its grid_x x ny blocks, start a
// multiple of 8 so a block's XCD, id % 8, is its tile order's).  The three branches of a KAD-Conv
// layer run their DSCs this way, as one launch instead of three concurrent streams.
struct DcnGroup {
  kad_dcn_args a[KAD_DCN_GROUP_MAX];
  DcnGeom g[KAD_DCN_GROUP_MAX];
  int start[KAD_DCN_GROUP_MAX + 1];
  int ny[KAD_DCN_GROUP_MAX];
  int count;
};

// kad_dcn_gather.h's kernels, one translation unit per data type: 0 or a KAD_E* code.
template <typename T> int dcn_gather(const kad_dcn_args& a, const DcnGeom& g, int mode, hipStream_t st);
template <typename T> int dcn_gather_group(const DcnGroup& grp, int nbf, hipStream_t st);

}  // namespace kad
