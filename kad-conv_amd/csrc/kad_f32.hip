// fp32 1x1 GEMM (kad_gemm1x1_fwd) and 3x3 convolution (kad_conv_fwd, kad_conv3x3_fwd) on MFMA.
//
// Block = 4 waves; a wave's tile is 32 pixels x 32 output channels (2 x 2 fragments of
// v_mfma_f32_16x16x4f32, 16 instructions of 32 clocks per k-step of 16 input channels of one tap).  The
// waves are 2 x 2 tiles (KS = 1: 64 x 64 per block), 2 x 1 tiles x 2 shares of the k-steps (KS = 2), or
// one tile x 4 shares (KS = 4), the shares added through LDS at the end in a fixed order: a map of few
// pixels has few tiles, and splitting k keeps the matrix cores of more CUs busy.
// Per step the block brings KS k-steps of both operands through registers into LDS (16-byte pieces,
// XOR-swizzled rows of 64 bytes; double-buffered), two steps ahead of the MFMAs.  NCHW input keeps its
// pixel runs: [16 channels][pixels], read with four 4-byte reads per fragment (the row pitch puts the
// lane groups' channels on distinct banks).
// Bound by the matrix cores (157 TFLOP/s) where the grid fills the chip, by the round trips of a step
// where it does not.  The kernels it replaced loaded single floats, 4 bytes per lane: KAD-CNet-S in
// fp32, one 512 x 512 image, 10.4 -> 3.3 ms; 1x1 512 -> 512 on [16, 512, 50, 50] runs at 111 TFLOP/s.
#include <type_traits>

#include "kad_common.h"

namespace kad {

typedef floatx4 __attribute__((aligned(4))) floatx4u;

enum { F32_GEMM_NHWC = 0, F32_CONV_NHWC = 1, F32_GEMM_NCHW = 2 };

struct F32Args {
  const float* x;
  const float* w;
  const float* bias;
  float* out;
  int n, cin, cout, colim;   // colim: output channels written (past cout: zeros)
  int h, w_, x_cs, stride, pad;
  int ho, wo, out_cs;        // NHWC output stride
  int spt, taps;             // k-steps per tap, taps
  int wrow;                  // floats per packed weight row
  int act;                   // KAD_ACT_*
  int P;                     // output pixels per image, or of the batch
};

template <int KS> struct F32Cfg {
  static constexpr int PXB = KS == 4 ? 32 : 64, COB = KS == 1 ? 64 : 32;
  static constexpr int NA = KS * PXB * 4 / 256, NB = KS * COB * 4 / 256;  // pieces per thread
  static constexpr int PITCH = PXB + 4;                                   // floats, NCHW operand rows
  static constexpr int A_FLOATS = KS * (16 * PITCH > PXB * 16 ? 16 * PITCH : PXB * 16), B_FLOATS = KS * COB * 16;
};

template <int KS, int MODE>
__global__ __launch_bounds__(256, 3) void f32_kernel(F32Args a) {
  typedef F32Cfg<KS> C;
  constexpr int PXB = C::PXB, COB = C::COB, NA = C::NA, NB = C::NB, D = 2;
  __shared__ __align__(16) float sA[2][C::A_FLOATS];
  __shared__ __align__(16) float sB[2][C::B_FLOATS];
  const int tid = threadIdx.x, lane = tid & 63, row = lane & 15, grp = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = blockIdx.z, p0 = blockIdx.x * PXB, co0 = blockIdx.y * COB;
  const int P = a.P;
  // wave -> pixel tile, channel tile, share of k
  const int wks = KS == 1 ? 0 : KS == 2 ? wave >> 1 : wave;
  const int wpx = KS == 4 ? 0 : wave & 1, wco = KS == 1 ? wave >> 1 : 0;

  // one descriptor per block: the tile's rows (NHWC GEMM), the image (conv, NCHW)
  const float* xb;
  uint32_t xbytes;
  if constexpr (MODE == F32_GEMM_NHWC) {
    xb = a.x + (int64_t)p0 * a.x_cs;
    const int rows = P - p0 < PXB ? P - p0 : PXB;
    xbytes = (uint32_t)(((int64_t)(rows - 1) * a.x_cs + a.cin) * 4);
  } else if constexpr (MODE == F32_CONV_NHWC) {
    xb = a.x + (int64_t)n * a.h * a.w_ * a.x_cs;
    xbytes = (uint32_t)(((int64_t)(a.h * a.w_ - 1) * a.x_cs + round_up(a.cin, 4)) * 4);
  } else {
    xb = a.x + (int64_t)n * a.cin * P;
    xbytes = (uint32_t)((int64_t)a.cin * P * 4);
  }
  const __amdgpu_buffer_rsrc_t rx = make_rsrc(xb, xbytes);
  const __amdgpu_buffer_rsrc_t rw = make_rsrc(a.w, (uint32_t)((int64_t)a.cout * a.wrow * 4));

  // this thread's pieces: slice of the step's KS k-steps (wave-uniform), row, 16-byte piece g
  int ak[NA], ac[NA], bk[NB], bc[NB];   // tap and 16-channel step of the piece's next load
  int ar[NA], ay[NA], ax[NA];           // conv: input row / column of tap (0, 0); else the piece's fixed offset in ar
  int br[NB];
  int alds[NA], blds[NB];
  const int g = tid & 3;
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int e = tid + u * 256, sl = __builtin_amdgcn_readfirstlane(e / (PXB * 4)), q = e % (PXB * 4);
    ak[u] = 0;
    ac[u] = sl;
    if constexpr (MODE == F32_GEMM_NCHW) {
      const int c = q / (PXB / 4), px = (q % (PXB / 4)) * 4;
      ar[u] = p0 + px < P ? (c * P + p0 + px) * 4 : -1;
      ay[u] = c;
      alds[u] = sl * (16 * C::PITCH) + c * C::PITCH + px;
    } else {
      const int r = q >> 2, p = p0 + r;
      alds[u] = sl * PXB * 16 + r * 16 + ((g ^ ((r >> 1) & 3)) << 2);
      if constexpr (MODE == F32_GEMM_NHWC) {
        ar[u] = p < P ? (r * a.x_cs + g * 4) * 4 : -1;
      } else {
        const int oy = p / a.wo, ox = p - oy * a.wo;
        ay[u] = p < P ? oy * a.stride - a.pad : -0x10000;
        ax[u] = ox * a.stride - a.pad;
      }
    }
  }
#pragma unroll
  for (int u = 0; u < NB; ++u) {
    const int e = tid + u * 256, sl = __builtin_amdgcn_readfirstlane(e / (COB * 4)), r = (e % (COB * 4)) >> 2;
    bk[u] = 0;
    bc[u] = sl;
    br[u] = co0 + r < a.cout ? ((co0 + r) * a.wrow + g * 4) * 4 : -1;
    blds[u] = sl * COB * 16 + r * 16 + ((g ^ ((r >> 1) & 3)) << 2);
  }
  auto norm = [&](int& k, int& c) {
    while (c >= a.spt) {
      c -= a.spt;
      ++k;
    }
  };
#pragma unroll
  for (int u = 0; u < NA; ++u) norm(ak[u], ac[u]);
#pragma unroll
  for (int u = 0; u < NB; ++u) norm(bk[u], bc[u]);

  floatx4 va[D][NA], vb[D][NB];
  auto issue = [&](int slot) {  // past the last k-step: zeros
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      uint32_t o = KAD_OOB;
      const int k = ak[u], c = ac[u];
      if constexpr (MODE == F32_GEMM_NHWC) {
        if (k == 0 && ar[u] >= 0 && c * 16 + g * 4 < a.cin) o = (uint32_t)(ar[u] + c * 64);
      } else if constexpr (MODE == F32_CONV_NHWC) {
        const int ky = k / 3, iy = ay[u] + ky, ix = ax[u] + k - ky * 3;
        if (k < 9 && iy >= 0 && iy < a.h && ix >= 0 && ix < a.w_ && c * 16 + g * 4 < a.cin)
          o = (uint32_t)(((iy * a.w_ + ix) * a.x_cs + c * 16 + g * 4) * 4);
      } else {
        if (k == 0 && ar[u] >= 0 && c * 16 + ay[u] < a.cin) o = (uint32_t)(ar[u] + c * 64 * P);
      }
      va[slot][u] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rx, o, 0, 0));
      ac[u] += KS;
      norm(ak[u], ac[u]);
    }
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int k = bk[u], c = bc[u];
      uint32_t o = KAD_OOB;
      if (k < a.taps && br[u] >= 0)
        o = (uint32_t)(br[u] + (MODE == F32_CONV_NHWC ? ((c >> 1) * 9 + k) * 128 + (c & 1) * 64 : c * 64));
      vb[slot][u] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(rw, o, 0, 0));
      bc[u] += KS;
      norm(bk[u], bc[u]);
    }
  };
  auto put = [&](int slot, int buf) {
#pragma unroll
    for (int u = 0; u < NA; ++u) *(floatx4*)(sA[buf] + alds[u]) = va[slot][u];
#pragma unroll
    for (int u = 0; u < NB; ++u) *(floatx4*)(sB[buf] + blds[u]) = vb[slot][u];
  };
  floatx4 acc[2][2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int f = 0; f < 2; ++f) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int steps = ceil_div(a.taps * a.spt, KS);
#pragma unroll
  for (int d = 0; d < D; ++d) issue(d);
  put(0, 0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  int buf = 0;
  for (int t = 0; t < steps; t += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      floatx4 xf[2], wf[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if constexpr (MODE == F32_GEMM_NCHW) {
          const float* s = sA[buf] + wks * (16 * C::PITCH) + grp * 4 * C::PITCH + wpx * 32 + m * 16 + row;
#pragma unroll
          for (int j = 0; j < 4; ++j) xf[m][j] = s[j * C::PITCH];
        } else {
          const int r = wpx * 32 + m * 16 + row;
          xf[m] = *(const floatx4*)(sA[buf] + wks * PXB * 16 + r * 16 + ((grp ^ ((r >> 1) & 3)) << 2));
        }
      }
#pragma unroll
      for (int f = 0; f < 2; ++f) {
        const int r = wco * 32 + f * 16 + row;
        wf[f] = *(const floatx4*)(sB[buf] + wks * COB * 16 + r * 16 + ((grp ^ ((r >> 1) & 3)) << 2));
      }
      issue(d);
      // rows of the product along the output's contiguous axis: channels (NHWC) or pixels (NCHW)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int m = 0; m < 2; ++m)
#pragma unroll
          for (int f = 0; f < 2; ++f)
            acc[m][f] = MODE == F32_GEMM_NCHW
                            ? __builtin_amdgcn_mfma_f32_16x16x4f32(xf[m][j], wf[f][j], acc[m][f], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f32_16x16x4f32(wf[f][j], xf[m][j], acc[m][f], 0, 0, 0);
      buf ^= 1;
      put((d + 1) % D, buf);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    }
  }

  // shares of k: added by wave 0 of the tile in share order
  if constexpr (KS > 1) {
    constexpr int RED = 64 * 16;  // floats of a wave's tile
    float* red = &sA[0][0] + (wpx * (KS - 1) + (wks > 0 ? wks - 1 : 0)) * RED;
    static_assert((KS == 4 ? 3 : 2) * RED <= 2 * C::A_FLOATS, "partial tiles fit");
    if (wks > 0) {
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int f = 0; f < 2; ++f) *(floatx4*)(red + (m * 2 + f) * 256 + lane * 4) = acc[m][f];
    }
    __syncthreads();
    if (wks > 0) return;
#pragma unroll
    for (int s = 0; s < KS - 1; ++s)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int f = 0; f < 2; ++f) acc[m][f] += *(const floatx4*)(red + s * RED + (m * 2 + f) * 256 + lane * 4);
  }

  auto epilogue = [&](auto act) {
    constexpr int ACT = decltype(act)::value;
    auto fn = [&](float v) {
      if constexpr (ACT == KAD_ACT_SILU) return v * sigmoidf_(v);
      else if constexpr (ACT == KAD_ACT_RELU) return fmaxf(v, 0.f);
      else return v;
    };
#pragma unroll
    for (int f = 0; f < 2; ++f) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if constexpr (MODE == F32_GEMM_NCHW) {
          const int co = co0 + wco * 32 + f * 16 + row, p = p0 + wpx * 32 + m * 16 + grp * 4;
          if (co >= a.cout || p >= P) continue;
          const float b = a.bias ? a.bias[co] : 0.f;
          floatx4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) o[i] = fn(acc[m][f][i] + b);
          float* dst = a.out + ((int64_t)n * a.cout + co) * P + p;
          if (p + 4 <= P) {
            *(floatx4u*)dst = o;  // planes of any size: 4-byte aligned
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (p + i < P) dst[i] = o[i];
          }
        } else {
          const int co = co0 + wco * 32 + f * 16 + grp * 4, p = p0 + wpx * 32 + m * 16 + row;
          if (co >= a.colim || p >= P) continue;
          floatx4 o;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float b = a.bias && co + i < a.cout ? a.bias[co + i] : 0.f;
            o[i] = fn(acc[m][f][i] + b);
          }
          float* dst = a.out + ((int64_t)n * P + p) * a.out_cs + co;
          if (co + 4 <= a.colim && a.out_cs % 4 == 0 && ((uintptr_t)a.out & 15) == 0) {
            *(floatx4*)dst = o;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (co + i < a.colim) dst[i] = o[i];
          }
        }
      }
    }
  };
  if (a.act == KAD_ACT_SILU) epilogue(std::integral_constant<int, KAD_ACT_SILU>{});
  else if (a.act == KAD_ACT_RELU) epilogue(std::integral_constant<int, KAD_ACT_RELU>{});
  else epilogue(std::integral_constant<int, KAD_ACT_NONE>{});
}

// Time of a launch with B blocks, in tenths of an iteration that has a CU's matrix cores to itself: each block
// runs its share of the k-steps (two per round of the loop) and about `over` iterations of prologue, sum of the
// shares and epilogue; a CU's blocks take its matrix cores in turn, and below three of them each one's round
// trips show.
static int64_t f32_cost(int64_t B, int iters, int over) {
  const int64_t q = (B + 255) / 256;  // blocks on the fullest CU
  return (10 * q + (q == 1 ? 8 : q == 2 ? 4 : 2)) * (round_up(iters, 2) + over);
}

// The split of k that f32_cost makes fastest.  Over 593 GEMMs and convolutions (8 .. 768 channels, 256 .. 160000
// pixels, each split timed) its choice is 0.4% off the best on average and 7% at worst; going by block counts
// alone (512 blocks for KS = 1, then 2) was 13% off, most for one step of channels and for up to 32 columns (us):
// conv 256 -> 20 [8, 100, 100] 209 -> 126, 40 -> 72 there 87 -> 80, 1x1 16 -> 16 [8, 50, 50] 7.6 -> 4.7.
template <int MODE>
static void f32_launch(const F32Args& a, int images, hipStream_t st) {
  const int ncol = a.colim, steps = a.taps * a.spt;
  const int p64 = ceil_div(a.P, 64), p32 = ceil_div(a.P, 32), c64 = ceil_div(ncol, 64), c32 = ceil_div(ncol, 32);
  const int64_t t1 = f32_cost((int64_t)images * p64 * c64, steps, 5);
  const int64_t t2 = f32_cost((int64_t)images * p64 * c32, ceil_div(steps, 2), 6);
  const int64_t t4 = f32_cost((int64_t)images * p32 * c32, ceil_div(steps, 4), 8);
  if (t4 <= t1 && t4 <= t2)
    hipLaunchKernelGGL((f32_kernel<4, MODE>), dim3(p32, c32, images), dim3(256), 0, st, a);
  else if (t2 <= t1)
    hipLaunchKernelGGL((f32_kernel<2, MODE>), dim3(p64, c32, images), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((f32_kernel<1, MODE>), dim3(p64, c64, images), dim3(256), 0, st, a);
}

int gemm_f32(const kad_gemm_args& a, hipStream_t st) {
  const int64_t P = (int64_t)a.h * a.w;
  if (a.dtype != KAD_F32 || a.pool != 1 || a.in_layout != a.out_layout) return 1;
  const int cin_pad = round_up(a.cin, 32);
  if ((int64_t)a.cout * cin_pad * 4 >= (1ll << 31) || a.n > 65535) return 1;
  F32Args f{};
  f.x = (const float*)a.x;
  f.w = (const float*)a.wpack;
  f.bias = a.bias;
  f.out = (float*)a.out;
  f.n = a.n;
  f.cin = a.cin;
  f.cout = f.colim = a.cout;
  f.spt = ceil_div(a.cin, 16);
  f.taps = 1;
  f.wrow = cin_pad;
  f.act = a.act ? KAD_ACT_SILU : KAD_ACT_NONE;
  if (a.in_layout == KAD_NCHW) {
    // runs of four pixels, 4-byte aligned (the last of a plane may reach into the next: columns past P
    // are not stored); one image's input and offsets within 31 bits
    if ((int64_t)round_up(a.cin, 16) * P * 4 >= (1ll << 31)) return 1;
    f.P = (int)P;
    f32_launch<F32_GEMM_NCHW>(f, a.n, st);
  } else {
    // whole 16-byte channel pieces: channels past Cin belong to others
    const int64_t M = P * a.n;
    if ((uintptr_t)a.x % 16 != 0 || a.cin % 4 != 0 || a.x_cs % 4 != 0 || M >= (1ll << 30) || (int64_t)64 * a.x_cs * 4 >= (1ll << 31)) return 1;
    f.x_cs = a.x_cs;
    f.out_cs = a.out_cs;
    f.colim = round_up(a.cout, 8) < a.out_cs ? round_up(a.cout, 8) : a.out_cs;
    f.P = (int)M;
    f32_launch<F32_GEMM_NHWC>(f, 1, st);
  }
  return check_launch("kad_gemm1x1_fwd");
}

int conv_f32(const kad_dcn_args& a, int ho, int wo, hipStream_t st) {
  if (a.dtype != KAD_F32 || a.out_layout != KAD_NHWC || a.post_mul || a.post_add || a.post_scale || a.gap_partial ||
      a.n > 65535)
    return 1;
  // Up to 16 output channels half of each 32-column tile is empty, and the general kernel computes 16.  It is
  // the faster one for a single whole 32-channel chunk and where it needs one round of the chip and this one
  // more (us, this / general): 32 -> 16 [8, 50, 50] 12.3 / 8.6, [16, 100, 100] 40 / 37; 16 -> 16 [8, 50, 50]
  // 9.5 / 8.7, 64 -> 16 17.5 / 14.2; but [16, 50, 50] 12 / 16 and 25 / 27.
  if (a.cout <= 16 && ((a.cin > 16 && a.cin <= 32) || (a.n * (int64_t)ceil_div(ho * wo, 64) > 256 &&
                                                       a.n * (int64_t)kad_dcn_tiles(ho, wo) <= 256)))
    return 1;
  F32Args f{};
  f.x = (const float*)a.x;
  f.w = (const float*)a.wpack;
  f.bias = a.bias;
  f.out = (float*)a.out;
  f.n = a.n;
  f.cin = round_up(a.cin, 8);  // the padding channels hold zeros
  f.cout = f.colim = a.cout;
  f.h = a.h;
  f.w_ = a.w;
  f.x_cs = a.x_cs;
  f.stride = a.stride;
  f.pad = a.pad;
  f.ho = ho;
  f.wo = wo;
  f.out_cs = a.out_cs;
  f.spt = ceil_div(a.cin, 16);
  f.taps = 9;
  f.wrow = ceil_div(a.cin, 32) * 288;
  f.act = a.relu == KAD_ACT_SILU ? KAD_ACT_SILU : a.relu ? KAD_ACT_RELU : KAD_ACT_NONE;
  f.P = ho * wo;
  f32_launch<F32_CONV_NHWC>(f, a.n, st);
  return check_launch("kad_conv_fwd");
}

}  // namespace kad
