// Modulated deformable 3x3 convolution with its samples gathered from L1 / L2 (kad_dcn_fwd and
// kad_dsc_fwd).  Semantics at kad_dcn.hip's head; here is the kernel's own shape.
//
// GEMM view: out[p, co] = sum_k S[p, k] * Wt[k, co]; a k-step is one tap x CH input channels, CH the
// channels of 64 bytes (32 16-bit, 16 fp32), so a sample's k-step is a 64-byte piece of each corner.
//
//  * Block = 8 waves x one tile of up to 128 output pixels x 16 NBF output channels.  Per k-step the
//    block builds the sampled tile A [128][64 B] and the weight tile B [16 NBF][64 B] in LDS (both
//    double-buffered, 16-byte pieces XOR-swizzled by row: a fragment read hits distinct banks) and
//    multiplies them on MFMA, 4 x 2 waves taking 32 pixels x 8 NBF channels each (NBF = 1: 8 x 1 waves of
//    16 pixels; with 32 columns for 16 fp32 DCN 512 -> 16 [8, 25, 25] took 162 us, with 16 126).
//  * A piece (pixel p, 16 bytes g) belongs to thread 4 p + g: four lanes read one corner's 64
//    consecutive bytes, which L1 serves as one request (37 TB/s measured over the chip, 8 KB
//    footprints).  In the MFMA operand's own lane order (16 pixels, then the piece) every lane of a
//    quad touches another line: 15 TB/s.
//  * Loads run two k-steps ahead in registers, are blended, and enter LDS one k-step ahead; one
//    barrier per k-step.  Taps are the outer loop: a tap's k-steps walk along the same corners' lines.
//  * No input region is staged: samples may lie anywhere at one cost, a block needs 48 to 55 KB of LDS (fp32
//    with 96 columns 57, with 128 77: the epilogue's tile) and at most 128 registers, and two share a CU.
//    The kernel this one replaced staged the region a tile samples (147 KB, one block per CU; samples beyond
//    it in a pass of their own) and read every weight fragment for 16 pixels only: it was bound by LDS reads
//    and by its serial phases.
//
// Measured (alone, 10 launches in a graph; this kernel / the replaced one, us): fp16 [8, 128, 100, 100] DSC
// 77 / 105, branch 0 of KADConv(256) at 100 x 100 (86 channels) 58 / 84; fp32 [4, 128, 100, 100] DSC 204 / 417.
// By clock64 stamps a block of 86 channels takes 34k cycles for its 27 k-steps when two share the CU (620 per
// k-step and block; the loads alone take about 600 through L1's 64 B / clk) and 27k alone, and some 30k for
// conv_offset, records, epilogue and squeeze-excitation.
#pragma once
#include <type_traits>

#include "kad_dcn.h"

namespace kad {

constexpr int DG_THREADS = 512, DG_WAVES = 8;
constexpr int DG_DEPTH = 2;  // k-steps of loads in flight
constexpr int DG_FROWS = 24;  // LDS rows per tap of conv_offset's 18 filters

// MFMA and blend on 16-byte pieces (8 16-bit or 4 fp32 channels)
template <typename T> struct DgOps {
  typedef typename DcnFrag<T>::frag frag;
  typedef uint2 weights;  // 4 x fp16
  static constexpr int E = 8;
  static __device__ __forceinline__ weights pack(const float* w) {
    return make_uint2(pack_h2(w[0], w[1]), pack_h2(w[2], w[3]));
  }
  static __device__ __forceinline__ frag blend(const frag (&v)[4], const weights& w) {
    return DcnFrag<T>::blend(v[0], v[1], v[2], v[3], w);
  }
  static __device__ __forceinline__ floatx4 mma(const frag& a, const frag& b, floatx4 c) {
    return DcnFrag<T>::mma(a, b, c);
  }
};
template <> struct DgOps<float> {
  typedef floatx4 frag;
  typedef floatx4 weights;
  static constexpr int E = 4;
  static __device__ __forceinline__ weights pack(const float* w) { return floatx4{w[0], w[1], w[2], w[3]}; }
  static __device__ __forceinline__ frag blend(const frag (&v)[4], const weights& w) {
    return v[0] * w[0] + v[1] * w[1] + v[2] * w[2] + v[3] * w[3];
  }
  // step j takes element j of every lane group: k = 4 group + j on both operands
  static __device__ __forceinline__ floatx4 mma(const frag& a, const frag& b, floatx4 c) {
#pragma unroll
    for (int j = 0; j < 4; ++j) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], c, 0, 0, 0);
    return c;
  }
};

template <typename T, int NBF, int MODE> struct DgCfg {
  static_assert((NBF == 1 || NBF % 2 == 0) && DG_THREADS == 4 * DCN_TILE, "wave grid; one A piece per thread");
  static constexpr int WCOL = NBF == 1 ? 1 : 2, WPX = DG_WAVES / WCOL;  // wave grid: columns x pixels
  static constexpr int MF = DCN_TILE / 16 / WPX, NW = NBF / WCOL;
  static constexpr int NB = NBF * 16;
  static constexpr int CH = 64 / (int)sizeof(T);                 // channels per k-step
  static constexpr int A_BYTES = DCN_TILE * 64, B_BYTES = NB * 64;
  static constexpr int REC_BYTES = 9 * DCN_TILE * (4 + (int)sizeof(typename DgOps<T>::weights));
  static constexpr int MAIN = 2 * (A_BYTES + B_BYTES) + REC_BYTES;
  // epilogue tile: [DCN_TILE][SROW] for NHWC, [NB][PROW] for NCHW
  static constexpr int SROW = NB + 16 / (int)sizeof(T), PROW = DCN_TILE + 16;
  static constexpr int STAGE = (DCN_TILE * SROW > NB * PROW ? DCN_TILE * SROW : NB * PROW) * (int)sizeof(T);
  static constexpr int EPI = STAGE + (WPX + 3) * NB * 4;
  // FUSED: one 64-byte plane of the 3x3 footprint (at most 645 pixels at stride <= 2) and filters
  static constexpr int OFFS = MODE == MODE_FUSED ? (645 + 9 * DG_FROWS) * 64 : 0;
  static constexpr int max4(int a, int b, int c, int d) {
    const int x = a > b ? a : b, y = c > d ? c : d;
    return x > y ? x : y;
  }
  static constexpr int SU = (max4(MAIN, EPI, OFFS, DCN_SE_LDS) + 15) / 16 * 16;
};

// 16-byte piece g of row r of a [rows][64 B] tile sits at slot g ^ ((r >> 1) & 3): eight consecutive
// lanes of a fragment read (rows r .. r + 7, one g) then cover 128 bytes of distinct banks.
__device__ __forceinline__ int dg_piece(int r, int g) { return r * 64 + ((g ^ ((r >> 1) & 3)) << 4); }

// conv_offset over the tile: oacc[b] = offset channel 16 b + row of pixels 16 wave ..
// Per 64-byte channel plane: the 3x3 footprint [fpix][64 B] and the filters [9 x 18][64 B] go through
// registers into LDS (two buffers where they fit su), the next plane's loads in flight while a plane's
// nine k-steps run; one barrier per plane.  A tap's filters take 24 rows, so that their swizzle does
// not depend on the tap.
template <typename T, int SU>
__device__ __forceinline__ void dg_offset_conv(floatx4 (&oacc)[2], __amdgpu_buffer_rsrc_t rx, const kad_dcn_args& a,
                                               const DcnGeom& g, int fy0, int fx0, unsigned char* su) {
  typedef DgOps<T> Ops;
  typedef typename Ops::frag frag;
  constexpr int CH = 64 / (int)sizeof(T), ROWB = 32 * (int)sizeof(T), HALF = ROWB / 64;
  constexpr int RS = DG_THREADS / 4;                     // rows between a thread's pieces
  constexpr int NF = (264 + RS - 1) / RS;                // footprint rows per thread at stride 1
  constexpr int NW = (9 * DCN_NOFF + RS - 1) / RS;       // filter rows per thread
  const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, grp = lane >> 4, gq = tid & 3, pq = tid >> 2;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fpix = g.fh * g.fw, npx = g.th * g.tw;
  const int cin8 = round_up(a.cin, 8), nst = ceil_div(a.cin, CH);
  const __amdgpu_buffer_rsrc_t rwo = make_rsrc(a.off_wpack, (uint32_t)(32 * g.nchunk * 9 * ROWB));
  int pl = wave * 16 + row;
  if (pl >= npx) pl = 0;  // padding lane: any pixel of the tile, result discarded
  const int ppy = (int)(((float)pl + 0.5f) * g.inv_tw);
  const int apix = (ppy * g.fw + pl - ppy * g.tw) * a.stride;  // its (0, 0) tap in the footprint
  const int plane = (fpix + 9 * DG_FROWS) * 64;
  const bool two = 2 * plane <= SU;
  auto foot_off = [&](int e) {  // byte offset of footprint pixel e's piece, or out of range
    const int qy = (int)(((float)e + 0.5f) * g.inv_fw), qx = e - qy * g.fw;
    const int gy = fy0 + qy, gx = fx0 + qx;
    return e < fpix && gy >= 0 && gy < a.h && gx >= 0 && gx < a.w
               ? (uint32_t)((gy * a.w + gx) * a.x_cs * (int)sizeof(T) + gq * 16) : KAD_OOB;
  };
  uint32_t fo[NF], wo[NW];
#pragma unroll
  for (int u = 0; u < NF; ++u) fo[u] = foot_off(pq + RS * u);
#pragma unroll
  for (int u = 0; u < NW; ++u) {
    const int e = pq + RS * u, k = e / DCN_NOFF, col = e - k * DCN_NOFF;
    wo[u] = e < 9 * DCN_NOFF ? (uint32_t)((col * g.nchunk * 9 + k) * ROWB + gq * 16) : KAD_OOB;
  }
  frag vf[NF], vw[NW];
  auto load = [&](int s) {  // plane s
    const uint32_t oob = s * CH + gq * Ops::E < cin8 ? 0u : KAD_OOB;
    const uint32_t so = (uint32_t)((s / HALF) * 9 * ROWB + (s % HALF) * 64);
#pragma unroll
    for (int u = 0; u < NF; ++u)
      vf[u] = __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rx, fo[u] | oob, s * 64, 0));
#pragma unroll
    for (int u = 0; u < NW; ++u)
      vw[u] = __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rwo, wo[u], so, 0));
  };
  load(0);
#pragma unroll 1
  for (int s = 0; s < nst; ++s) {
    unsigned char* foot = su + (two && (s & 1) ? plane : 0);
    unsigned char* filt = foot + fpix * 64;
#pragma unroll
    for (int u = 0; u < NF; ++u)
      if (pq + RS * u < fpix) *(frag*)(foot + dg_piece(pq + RS * u, gq)) = vf[u];
#pragma unroll
    for (int u = 0; u < NW; ++u) {
      const int e = pq + RS * u, k = e / DCN_NOFF;
      if (e < 9 * DCN_NOFF) *(frag*)(filt + dg_piece(e + k * (DG_FROWS - DCN_NOFF), gq)) = vw[u];
    }
    for (int e = pq + RS * NF; e < fpix; e += RS) {  // the rest of a stride-2 footprint
      const uint32_t o = s * CH + gq * Ops::E < cin8 ? foot_off(e) : KAD_OOB;
      *(frag*)(foot + dg_piece(e, gq)) =
          __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rx, o, s * 64, 0));
    }
    if (s + 1 < nst) load(s + 1);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    int ap = apix;
    asm volatile("" : "+v"(ap));  // the taps' addresses are formed per plane, not kept over the loop
    // columns past the 18 filters repeat the last two: their results are not used
    const unsigned char* f0 = filt + dg_piece(row, grp);
    const unsigned char* f1 = filt + dg_piece(16 + (row & 1), grp);
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const frag b0 = *(const frag*)(f0 + k * DG_FROWS * 64);
      const frag b1 = *(const frag*)(f1 + k * DG_FROWS * 64);
      const int toff = (k / 3) * g.fw + k % 3;
      const frag af = *(const frag*)(foot + dg_piece(ap + toff, grp));
      oacc[0] = Ops::mma(af, b0, oacc[0]);
      oacc[1] = Ops::mma(af, b1, oacc[1]);
    }
    if (!two) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  }
  __syncthreads();  // planes consumed: the caller reuses su
}

template <typename T, int NBF, int MODE>
__device__ __forceinline__ void dg_block(const kad_dcn_args& a, const DcnGeom& g, const int bx, const int by,
                                         const int ny) {
  typedef DgOps<T> Ops;
  typedef typename Ops::frag frag;
  typedef typename Ops::weights weights;
  typedef DgCfg<T, NBF, MODE> C;
  constexpr int MF = C::MF, NW = C::NW, NB = C::NB, CH = C::CH;
  constexpr int ROWB = 32 * (int)sizeof(T), HALF = ROWB / 64;  // bytes of a packed weight row; k-steps in it
  constexpr int KS = DG_THREADS / DCN_TILE, PPT = (9 + KS - 1) / KS;  // samples per thread: taps tid / 128 + KS u
  __shared__ __align__(16) unsigned char s_u[C::SU];

  // XCD-aware tile order over (image, tile) flattened: block b runs on XCD b % 8, which takes a
  // contiguous run of it, so neighbouring tiles share their samples' lines through one L2
  const int q = (bx & 7) * (g.grid_x >> 3) + (bx >> 3);
  if (q >= a.n * g.tiles) return;  // whole block, before any barrier
  const int n = q / g.tiles, tile = q - n * g.tiles;
  const int co0 = by * NB;
  const int tyi = tile / g.tiles_x;
  const int ty0 = tyi * g.th, tx0 = (tile - tyi * g.tiles_x) * g.tw;
  const int P = g.ho * g.wo, npx = g.th * g.tw;
  const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wpx = wave / C::WCOL, wcol = wave % C::WCOL;
  const T* xb = (const T*)a.x + (int64_t)n * a.h * a.w * a.x_cs;
  const int cin8 = round_up(a.cin, 8);
  const int pxb = a.x_cs * (int)sizeof(T), rowb = a.w * pxb;
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(xb, (uint32_t)(a.h * rowb));
  const __amdgpu_buffer_rsrc_t rwp = make_rsrc(a.wpack, (uint32_t)(g.cout_pad * g.nchunk * 9 * ROWB));

  // ---- 0. independent loads ------------------------------------------------------------------------
  float par[4] = {0.f, 1.f, 0.f, 1.f};
  if (tid < NB) {
    const int co = co0 + tid;
    if (co < a.cout) {
      if (a.bias) par[0] = a.bias[co];
      if (a.post_mul) par[1] = a.post_mul[co];
      if (a.post_add) par[2] = a.post_add[co];
      if (a.post_scale) par[3] = a.post_scale[co];
    }
  }
  const int ppl = tid % DCN_TILE;
  const int ppy = (int)(((float)ppl + 0.5f) * g.inv_tw), ppx = ppl - ppy * g.tw;
  const int poy = ty0 + ppy, pox = tx0 + ppx;
  const bool plive = ppl < npx && poy < g.ho && pox < g.wo;
  const int64_t pp = (int64_t)poy * g.wo + pox;
  float pre_dy[PPT], pre_dx[PPT], pre_m[PPT];
#pragma unroll
  for (int u = 0; u < PPT; ++u) {
    const int k = tid / DCN_TILE + KS * u;
    pre_dy[u] = pre_dx[u] = 0.f;
    pre_m[u] = 1.f;
    if (k < 9 && plive) {
      if constexpr (MODE == MODE_EXT) {
        pre_dy[u] = a.offset[n * a.off_sn + pp * a.off_sp + (2 * k) * a.off_sc];
        pre_dx[u] = a.offset[n * a.off_sn + pp * a.off_sp + (2 * k + 1) * a.off_sc];
      }
      if (a.mask) pre_m[u] = a.mask[n * a.mask_sn + pp * a.mask_sp + k * a.mask_sc];
    }
  }

  // ---- 1. FUSED: offsets = conv_offset(x) over the tile -> [DCN_TILE][18] fp32 in s_u ---------------------
  if constexpr (MODE == MODE_FUSED) {
    floatx4 oacc[2] = {floatx4{0.f, 0.f, 0.f, 0.f}, floatx4{0.f, 0.f, 0.f, 0.f}};
    dg_offset_conv<T, C::SU>(oacc, rx, a, g, ty0 * a.stride - a.pad, tx0 * a.stride - a.pad, s_u);
    float* s_off = (float*)s_u;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int ch = b * 16 + row;
      if (ch < DCN_NOFF) {
        const float ob = a.off_bias ? a.off_bias[ch] : 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i) s_off[(wave * 16 + grp * 4 + i) * DCN_NOFF + ch] = oacc[b][i] + ob;
      }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
      const int k = tid / DCN_TILE + KS * u;
      if (k < 9) {
        pre_dy[u] = s_off[ppl * DCN_NOFF + 2 * k];
        pre_dx[u] = s_off[ppl * DCN_NOFF + 2 * k + 1];
      }
    }
    __syncthreads();  // offsets read: s_u is free
  }

  // ---- 2. sample records: top-left corner's byte offset (| sx | sy << 1) and corner weights ----------
  unsigned char* sA = s_u;                                     // [2][DCN_TILE][64 B]
  unsigned char* sB = s_u + 2 * C::A_BYTES;                    // [2][NB][64 B]
  weights* s_rw = (weights*)(sB + 2 * C::B_BYTES);             // [9][DCN_TILE]
  unsigned* s_ro = (unsigned*)(s_rw + 9 * DCN_TILE);                 // [9][DCN_TILE]
#pragma unroll
  for (int u = 0; u < PPT; ++u) {
    const int k = tid / DCN_TILE + KS * u;
    if (k >= 9) break;
    float w[4] = {0.f, 0.f, 0.f, 0.f};
    int cy0 = 0, cx0 = 0, sy = 0, sx = 0;
    if (plive) {
      const int ky = k / 3, kx = k - (k / 3) * 3;
      sample_geom((float)(poy * a.stride - a.pad + ky) + pre_dy[u], (float)(pox * a.stride - a.pad + kx) + pre_dx[u],
                  pre_m[u], a.h, a.w, cy0, cx0, sy, sx, w);
    }
    const bool dead = w[0] == 0.f && w[1] == 0.f && w[2] == 0.f && w[3] == 0.f;
    // a dead sample reads out of range (zeros); pxb is a multiple of 16, so the low bits are free
    s_ro[k * DCN_TILE + ppl] = dead ? KAD_OOB : (uint32_t)(cy0 * rowb + cx0 * pxb) | (unsigned)sx | ((unsigned)sy << 1);
    s_rw[k * DCN_TILE + ppl] = Ops::pack(w);
  }
  __syncthreads();

  // ---- 3. k-steps -------------------------------------------------------------------------------------
  const int gq = tid & 3, pq = tid >> 2;  // this thread's piece, and its first pixel / weight row
  const uint32_t bvo = pq < NB && co0 + pq < g.cout_pad ? (uint32_t)((co0 + pq) * g.nchunk * 9 * ROWB + gq * 16) : KAD_OOB;
  // ring of k-steps in flight: corners, their blend weights, weight piece
  frag cr[DG_DEPTH][4], br[DG_DEPTH];
  weights wr[DG_DEPTH];
  // the tap whose loads are issued: corner offsets and blend weights; ron / rwn: the next tap's record
  uint32_t vo[4];
  weights rw, rwn;
  unsigned ron;
  auto read_rec = [&](int k) {
    ron = s_ro[k * DCN_TILE + pq];
    rwn = s_rw[k * DCN_TILE + pq];
  };
  auto set_tap = [&]() {
    const uint32_t o = (ron & ~3u) + gq * 16;
    const uint32_t dx = (ron & 1u) ? (uint32_t)pxb : 0u, dy = (ron & 2u) ? (uint32_t)rowb : 0u;
    vo[0] = o;
    vo[1] = o + dx;
    vo[2] = o + dy;
    vo[3] = o + dy + dx;
    rw = rwn;
  };
  const int nst = ceil_div(a.cin, CH), total = 9 * nst;
  int ik = 0, is = -1;  // the k-step issued last: tap, 64-byte step of its channels
  // Past the last k-step the ring takes steps of zeros (out-of-range loads): the loop needs no
  // conditional loads, so the compiler's wait counts stay exact.
  auto issue = [&](int slot) {
    if (++is == nst) {
      is = 0;
      ++ik;
      set_tap();
      if (ik < 8) read_rec(ik + 1);
    }
    const uint32_t end = ik < 9 ? 0u : KAD_OOB;
    const uint32_t so = ik < 9 ? (uint32_t)(((is / HALF) * 9 + ik) * ROWB + (is % HALF) * 64) : 0u;
    br[slot] = __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rwp, bvo | end, so, 0));
    const uint32_t oob = is * CH + gq * Ops::E < cin8 ? end : KAD_OOB;  // channels past Cin read zeros
#pragma unroll
    for (int j = 0; j < 4; ++j)
      cr[slot][j] = __builtin_bit_cast(frag, __builtin_amdgcn_raw_buffer_load_b128(rx, vo[j] | oob, is * 64, 0));
    wr[slot] = rw;
  };
  auto put = [&](int slot, int buf) {  // k-step of ring slot `slot` into LDS buffer buf
    if (NB == DCN_TILE || pq < NB) *(frag*)(sB + buf * C::B_BYTES + dg_piece(pq, gq)) = br[slot];
    *(frag*)(sA + buf * C::A_BYTES + dg_piece(pq, gq)) = Ops::blend(cr[slot], wr[slot]);
  };
  floatx4 acc[MF][NW];
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int f = 0; f < NW; ++f) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};

  read_rec(0);
  set_tap();
  read_rec(1);
#pragma unroll
  for (int d = 0; d < DG_DEPTH; ++d) issue(d);
  put(0, 0);
  // the barriers of the k-steps wait for LDS traffic only: the loads in flight stay in flight
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  int buf = 0;
  for (int t = 0; t < total; t += DG_DEPTH) {
#pragma unroll
    for (int d = 0; d < DG_DEPTH; ++d) {
      frag af[MF], bf[NW];
#pragma unroll
      for (int f = 0; f < NW; ++f)
        bf[f] = *(const frag*)(sB + buf * C::B_BYTES + dg_piece((wcol * NW + f) * 16 + row, grp));
#pragma unroll
      for (int m = 0; m < MF; ++m)
        af[m] = *(const frag*)(sA + buf * C::A_BYTES + dg_piece((wpx * MF + m) * 16 + row, grp));
      issue(d);
#pragma unroll
      for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int f = 0; f < NW; ++f) acc[m][f] = Ops::mma(af[m], bf[f], acc[m][f]);
      buf ^= 1;
      put((d + 1) % DG_DEPTH, buf);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }

  // ---- 4. epilogue: values -> LDS tile -> row-contiguous stores; GAP partials ------------------------
  constexpr int SROW = C::SROW, PROW = C::PROW;
  const bool nchw = a.out_layout == KAD_NCHW;
  T* ost = (T*)s_u;
  float(*s_par)[NB] = (float(*)[NB])(s_u + C::STAGE);         // shift, mul, scale
  float(*gap_red)[NB] = s_par + 3;                            // [WPX][NB]
  if (tid < NB) {  // v = acc * mul + (bias * mul + add)
    s_par[0][tid] = par[0] * par[1] + par[2];
    s_par[1][tid] = par[1];
    s_par[2][tid] = par[3];
  }
  __syncthreads();
  unsigned pix_ok = 0u;
#pragma unroll
  for (int m = 0; m < MF; ++m)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int pl = (wpx * MF + m) * 16 + grp * 4 + i;
      const int oyl = (int)(((float)pl + 0.5f) * g.inv_tw);
      if (pl < npx && ty0 + oyl < g.ho && tx0 + pl - oyl * g.tw < g.wo) pix_ok |= 1u << (m * 4 + i);
    }
  // the activation as a template argument: a per-value branch would put every value's chain in a
  // basic block of its own, and the scheduler could not interleave the independent chains
  auto epilogue = [&](auto act) {
    constexpr int ACT = decltype(act)::value;
#pragma unroll
    for (int f = 0; f < NW; ++f) {
      const int col = (wcol * NW + f) * 16 + row;
      float gs = 0.f;
      const bool co_ok = co0 + col < a.cout;
      const float shift = s_par[0][col], mul = s_par[1][col], scl = s_par[2][col];
#pragma unroll
      for (int m = 0; m < MF; ++m)
{
        const int pl = (wpx * MF + m) * 16 + grp * 4;
        struct alignas(4 * sizeof(T)) Quad { T v[4]; } o;  // four consecutive pixels of one channel
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v = fmaf(acc[m][f][i], mul, shift);
          if constexpr (ACT == KAD_ACT_SILU) v = v * sigmoidf_(v);
          else if constexpr (ACT == KAD_ACT_RELU) v = fmaxf(v, 0.f);
          v *= scl;
          o.v[i] = from_f32<T>(v);
          if (co_ok && ((pix_ok >> (m * 4 + i)) & 1u)) gs += to_f32(o.v[i]);
        }
        if (nchw) {
          *(Quad*)(ost + col * PROW + pl) = o;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) ost[(pl + i) * SROW + col] = o.v[i];
        }
      }
      if (a.gap_partial) {
        gs = sum_xor32(sum_xor16(gs));
        if (grp == 0) gap_red[wpx][col] = gs;
      }
    }
  };
  if (a.relu == KAD_ACT_SILU) epilogue(std::integral_constant<int, KAD_ACT_SILU>{});
  else if (a.relu) epilogue(std::integral_constant<int, KAD_ACT_RELU>{});
  else epilogue(std::integral_constant<int, KAD_ACT_NONE>{});
  __syncthreads();
  T* out = (T*)a.out;
  constexpr int VEC = 16 / (int)sizeof(T);
  const bool vec_ok = a.out_layout == KAD_NHWC && (a.out_cs * (int)sizeof(T)) % 16 == 0 && ((uintptr_t)a.out & 15) == 0;
  if (vec_ok) {
    constexpr int VPP = NB / VEC;  // 16-byte vectors per pixel
    for (int j = tid; j < DCN_TILE * VPP; j += DG_THREADS) {
      const int pl = j / VPP, v = j - pl * VPP;
      const int oyl = (int)(((float)pl + 0.5f) * g.inv_tw);
      const int oy = ty0 + oyl, ox = tx0 + pl - oyl * g.tw;
      const int co = co0 + v * VEC;
      if (pl >= npx || oy >= g.ho || ox >= g.wo || co >= a.cout) continue;
      const T* src = ost + pl * SROW + v * VEC;
      T* dst = out + ((int64_t)n * P + (int64_t)oy * g.wo + ox) * a.out_cs + co;
      if (co + VEC <= a.cout) {
        *(intx4*)dst = *(const intx4*)src;
      } else {
        for (int e = 0; e < a.cout - co; ++e) dst[e] = src[e];
      }
    }
  } else if (a.out_layout == KAD_NHWC) {
    for (int j = tid; j < DCN_TILE * NB; j += DG_THREADS) {
      const int pl = j / NB, col = j - pl * NB;
      const int oyl = (int)(((float)pl + 0.5f) * g.inv_tw);
      const int oy = ty0 + oyl, ox = tx0 + pl - oyl * g.tw;
      const int co = co0 + col;
      if (pl >= npx || oy >= g.ho || ox >= g.wo || co >= a.cout) continue;
      out[((int64_t)n * P + (int64_t)oy * g.wo + ox) * a.out_cs + co] = ost[pl * SROW + col];
    }
  } else {  // NCHW: consecutive lanes along the tile's pixels; a thread keeps its pixel for every channel
    constexpr int CSTEP = DG_THREADS / DCN_TILE;
    const int pl = tid % DCN_TILE, col0 = tid / DCN_TILE;
    const int oyl = (int)(((float)pl + 0.5f) * g.inv_tw);
    const int oy = ty0 + oyl, ox = tx0 + pl - oyl * g.tw;
    if (pl < npx && oy < g.ho && ox < g.wo) {
      T* dst = out + ((int64_t)n * a.out_cs + co0 + col0) * P + (int64_t)oy * g.wo + ox;
      const T* src = ost + col0 * PROW + pl;
      const int ncol = a.cout - co0 < NB ? a.cout - co0 : NB;
#pragma unroll 4
      for (int col = col0; col < ncol; col += CSTEP) {
        *dst = *src;
        dst += (int64_t)CSTEP * P;
        src += CSTEP * PROW;
      }
    }
  }
  if (a.gap_partial && tid < NB) {
    const int co = co0 + tid;
    if (co < a.cout) {
      float v = 0.f;
#pragma unroll
      for (int i = 0; i < C::WPX; ++i) v += gap_red[i][tid];
      float* dst = a.gap_partial + ((int64_t)n * g.tiles + tile) * a.cout + co;
      if (a.se_att)
        rmw_store(dst, v);  // read by another block of this launch (fused SE)
      else
        *dst = v;
    }
  }

  // ---- 5. fused squeeze-excitation: the image's last block runs the MLP (protocol at se_tail) ---------
  if (a.se_att && a.gap_partial) {
    __shared__ int s_last;
    // Each thread has waited for its own exchange's return and the epilogue tile is free: the
    // barriers wait for LDS traffic only, not for the output stores' acknowledgements.
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (tid == 0) {
      const unsigned total = (unsigned)g.tiles * ny;
      const unsigned prev = __hip_atomic_fetch_add(a.se_count + n, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const int last = prev + 1u == total;
      if (last) {
        const unsigned z = __hip_atomic_exchange(a.se_count + n, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("" ::"v"(z));
      }
      s_last = last;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (s_last)
      se_tail<DG_THREADS, C::SU / 4>(a.gap_partial, a.se_w1, a.se_b1, a.se_w2, a.se_b2, a.se_att, a.se_inv_count, a.cout, a.se_hid,
                          n, g.tiles, (float*)s_u);
  }
}

template <typename T, int NBF, int MODE>
__global__ __launch_bounds__(DG_THREADS, 4) void dg_kernel(kad_dcn_args a, DcnGeom g) {
  dg_block<T, NBF, MODE>(a, g, blockIdx.x, blockIdx.y, gridDim.y);
}

template <typename T, int NBF>
__global__ __launch_bounds__(DG_THREADS, 4) void dg_group_kernel(DcnGroup grp) {
  const int id = blockIdx.x;
  int p = 0;
#pragma unroll
  for (int i = 1; i < KAD_DCN_GROUP_MAX; ++i)
    if (i < grp.count && id >= grp.start[i]) p = i;
  if (id >= grp.start[p + 1]) return;
  const int local = id - grp.start[p];
  const int gx = grp.g[p].grid_x;
  dg_block<T, NBF, MODE_FUSED>(grp.a[p], grp.g[p], local % gx, local / gx, grp.ny[p]);
}

template <typename T, int NBF>
static int dg_launch(const kad_dcn_args& a, const DcnGeom& g, int mode, hipStream_t st) {
  const dim3 grid(g.grid_x, ceil_div(a.cout, NBF * 16));
  if (mode == MODE_FUSED)
    hipLaunchKernelGGL((dg_kernel<T, NBF, MODE_FUSED>), grid, dim3(DG_THREADS), 0, st, a, g);
  else
    hipLaunchKernelGGL((dg_kernel<T, NBF, MODE_EXT>), grid, dim3(DG_THREADS), 0, st, a, g);
  return check_launch(mode == MODE_FUSED ? "kad_dsc_fwd" : "kad_dcn_fwd");
}

// Columns by Cout alone: 16, 32, 64, 96 or blocks of 128.  The padding of 33 .. 48 channels to 64 columns and of
// 65 .. 80 to 96 costs less than a form of 48 or 80 would gain: the replaced kernel had those, and DSC took (us,
// it / this) 48 channels fp16 [8, 50, 50] 40 / 35, bf16 48 / 43, fp32 82 / 62; 80 channels 51 / 44, 71 / 59, 150 / 104.
template <typename T> int dcn_gather(const kad_dcn_args& a, const DcnGeom& g, int mode, hipStream_t st) {
  if (a.cout <= 16) return dg_launch<T, 1>(a, g, mode, st);
  switch (ceil_div(a.cout, 32)) {
    case 1: return dg_launch<T, 2>(a, g, mode, st);
    case 2: return dg_launch<T, 4>(a, g, mode, st);
    case 3: return dg_launch<T, 6>(a, g, mode, st);
    default: return dg_launch<T, 8>(a, g, mode, st);
  }
}

template <typename T, int NBF> static int dg_launch_group(const DcnGroup& grp, hipStream_t st) {
  hipLaunchKernelGGL((dg_group_kernel<T, NBF>), dim3(grp.start[grp.count]), dim3(DG_THREADS), 0, st, grp);
  return check_launch("kad_dsc_fwd_group");
}

template <typename T> int dcn_gather_group(const DcnGroup& grp, int nbf, hipStream_t st) {
  if (nbf == 1) return dg_launch_group<T, 1>(grp, st);
  switch ((nbf + 1) / 2) {
    case 1: return dg_launch_group<T, 2>(grp, st);
    case 2: return dg_launch_group<T, 4>(grp, st);
    case 3: return dg_launch_group<T, 6>(grp, st);
    default: return dg_launch_group<T, 8>(grp, st);
  }
}

}  // namespace kad
