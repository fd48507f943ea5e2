// unet_kernels.hip -- BF16 MFMA kernels of the pressure warm-start U-Net (gfx950).
//
// Tensors are channels-last (B, D, H, W, C) in bf16 with a channel stride and
// offset, so a decoder's concatenated input is one buffer that the skip
// connection and the upsampled path write into side by side. All three 3x3x3
// convolution products -- forward, input gradient and weight gradient -- run on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation.
//
// MFMA 16x16x32 lane layout (wave64): lane l supplies row (l % 16) of A and
// column (l % 16) of B, each with the 8 consecutive k values 8*(l/16) .. +7; it
// receives C rows 4*(l/16) .. +3 of column (l % 16).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cstdlib>

#include "unet_internal.h"

namespace aqu {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kXCD = 8;

__device__ __forceinline__ float bf2f(__bf16 v) { return (float)v; }
__device__ __forceinline__ __bf16 f2bf(float v) { return (__bf16)v; }  // round to nearest even

__device__ __forceinline__ int xcd_block() {
  const int nb = gridDim.x, bid = blockIdx.x;
  const int per = nb / kXCD, rem = nb % kXCD;
  const int xcd = bid % kXCD, k = bid / kXCD;
  return xcd * per + min(xcd, rem) + k;
}

struct VoxelPos {
  int b, d, h, w;
};
__device__ __forceinline__ VoxelPos vox_of(const Vol& v, long long id) {
  VoxelPos p;
  p.w = (int)(id % v.W);
  long long t = id / v.W;
  p.h = (int)(t % v.H);
  t /= v.H;
  p.d = (int)(t % v.D);
  p.b = (int)(t / v.D);
  return p;
}
__device__ __forceinline__ long long vox_id(const Vol& v, int b, int d, int h, int w) {
  return (((long long)b * v.D + d) * v.H + h) * v.W + w;
}

// ------------------------------------------------------------------ conv 3x3x3, implicit GEMM
// Y[v, n] = sum_{tap, c} X[v + off(tap), c] * Wk[n, tap*CIN + c], zero padding outside
// the volume. M = voxels, N = COUT, K = 27*CIN in slices of 32.
//
// k_conv3 gathers its input per tap from memory, one fragment of 16 voxels and one
// 16-channel output tile per wave: for extents that would leave most of k_conv3_tile's tiles
// empty (conv3_tile_fits), and the reference for its forward pass, run at every extent under
// AQUNET_NO_TILE=1 (read at every launch).
static bool conv3_tile_enabled() {
  const char* e = std::getenv("AQUNET_NO_TILE");
  return !(e && e[0] == '1');
}

template <int CIN, int COUT>
__global__ __launch_bounds__(256) void k_conv3(Vol v, const __bf16* __restrict__ X, int xs, int xo,
                                               const __bf16* __restrict__ Wk,
                                               const float* __restrict__ bias, __bf16* __restrict__ Y, int ys,
                                               int yo) {
  constexpr int K = 27 * CIN;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const int n = (int)blockIdx.y * 16 + r;
  const long long V = (long long)v.B * v.D * v.H * v.W;
  const long long wbase = ((long long)xcd_block() * 4 + wave) * 16;
  if (wbase >= V) return;
  const bool vok = wbase + r < V;
  const VoxelPos p = vox_of(v, vok ? wbase + r : 0);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const bf16x8 zero8 = {};
  for (int k0 = 0; k0 < K; k0 += 32) {
    const int k = k0 + q * 8;
    const bool kok = k < K;
    const int tap = k / CIN, c = k - tap * CIN;
    const int zd = p.d + tap / 9 - 1, zh = p.h + (tap / 3) % 3 - 1, zw = p.w + tap % 3 - 1;
    bf16x8 a = zero8;
    if (kok && vok && zd >= 0 && zd < v.D && zh >= 0 && zh < v.H && zw >= 0 && zw < v.W)
      a = *(const bf16x8*)(X + vox_id(v, p.b, zd, zh, zw) * xs + xo + c);
    const bf16x8 bw = kok ? *(const bf16x8*)(Wk + (long long)n * K + k) : zero8;
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bw, acc, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const long long o = wbase + q * 4 + i;
    if (o < V) Y[o * ys + yo + n] = f2bf(fmaxf(acc[i] + bias[n], 0.f));
  }
}

// ------------------------------------------------------------------ conv 3x3x3, input tile in LDS
// The convolutions of the forward pass and, with flipped transposed weights, the input
// gradients. A block owns output tiles of TD x 8 x 16 voxels (d, h, w) of one batch item
// and NTB 16-channel output tiles (channel group blockIdx.y). An input tile with its
// one-voxel halo, (TD+2) x 10 x 18 voxels, is staged in LDS CH input channels at a time
// (zero outside the volume), so each input value is read from memory about 2.5 times per
// layer instead of once per tap; the fragments of all 27 taps then come from LDS. A
// block walks several tiles when there are many: the next tile's (or channel chunk's)
// pieces are loaded into registers while the current one is multiplied. Wave w owns the
// rows h = 2w, 2w + 1 of every plane, so it holds whole 2 x 2 x 2 groups when TD = 2.
// 8 x 64^3, before (16-bit stores, weights refetched, one tile per block; gradients by
// gathering per tap, FP32, with separate upsampling, pooling and ReLU passes) and now:
// forward 16 -> 16 104 -> 67 us, 32 -> 32 at 32^3 38 -> 31 us, 96 -> 32 93 -> 84 us, 48 -> 16
// 232 -> 230 us; gradients 16 -> 16 147 + 77 -> 69 us, 48 -> 16 277 + 90 -> 169 us. The
// fragments' LDS reads (1 KB per MFMA with one channel tile) bound the 16-channel layers.
// The weights are the MFMA's first operand (rows = output channels): lane (r, q) then
// holds channels 4q .. 4q + 3 of voxel r, one 8- or 16-byte store. LDS voxels sit
// VS bf16 apart so that the 16-byte reads of 8 consecutive lanes fall in distinct banks.
// The k order is (chunk, tap, channel within the chunk), the order of k_conv3 when
// CH = CIN. Extents that are no multiples of the tile compute partial tiles.
enum { kConvFwd, kConvF32, kConvMask, kConvUp };
struct ConvOut {
  const float* bias;  // kConvFwd: + bias, ReLU, bf16
  void* y;            // bf16 (kConvFwd, kConvMask) or FP32 (kConvF32; kConvUp: channels below `split`)
  int ys, yo;         // its channel stride and offset
  const __bf16* m;    // kConvMask / kConvUp: the ReLU outputs whose sign gates the gradient
  int ms, mo;
  int split;          // kConvUp: first channel of the upsampled part
  __bf16* up;         // kConvUp: gated gradient of the coarse tensor, dense
};

// Offset (in LDS bf16) of tap t from tap 0.
template <int IH, int IW, int VS>
__device__ constexpr int tap_off(int t) {
  return (((t / 9) * IH + (t / 3) % 3) * IW + t % 3) * VS;
}

// Waves per SIMD the registers must allow: what the tile's LDS leaves room for, at most 3
// (four 16-channel variants spill at 128 registers).
constexpr int conv_waves(int CH, int TD) {
  const int n = 160 * 1024 / ((TD + 2) * 180 * (CH <= 16 ? CH : CH + 8) * 2);
  return CH == 48 ? 1 : CH >= 32 && n > 2 ? 2 : n > 3 ? 3 : n;
}

template <int CIN, int COUT, int CH, int TD, int NTB, int EPI>
__global__ __launch_bounds__(256, conv_waves(CH, TD)) void k_conv3_tile(Vol v, int ntiles, const __bf16* __restrict__ X, int xs, int xo,
                                                    const __bf16* __restrict__ Wk, ConvOut out) {
  constexpr int TH = 8, TW = 16;
  constexpr int ID = TD + 2, IH = TH + 2, IW = TW + 2;
  constexpr int NV = ID * IH * IW;
  constexpr int VS = CH <= 16 ? CH : CH + 8;     // LDS voxel stride (bf16)
  constexpr int MF = 2 * TD;                      // 16-voxel rows per wave
  constexpr int NSL = (27 * CH + 31) / 32;        // k slices per chunk
  constexpr int NC = CIN / CH;
  constexpr int K = 27 * CIN;
  constexpr int PV = CH / 8;                      // 16-byte pieces per voxel
  constexpr int NP = (NV * PV + 255) / 256;       // pieces per thread
  constexpr int TPS = CH >= 32 ? 1 : 32 / CH;     // taps per slice
  static_assert(CIN % CH == 0 && CH % 8 == 0 && (CH < 32 ? 32 % CH == 0 : CH % 32 == 0 || CH == 48), "channel chunks");
  __shared__ __align__(16) __bf16 sX[NV * VS];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  const int n0 = (int)blockIdx.y * NTB * 16;
  const int ntw = (v.W + TW - 1) / TW, nth = (v.H + TH - 1) / TH, ntd = (v.D + TD - 1) / TD;
  const bf16x8 zero8 = {};
  struct Org {
    int b, d0, h0, w0;
  };
  auto org_of = [&](int t) {
    Org o;
    o.w0 = (t % ntw) * TW;
    t /= ntw;
    o.h0 = (t % nth) * TH;
    t /= nth;
    o.d0 = (t % ntd) * TD;
    o.b = t / ntd;
    return o;
  };
  bf16x8 rp[NP];
  auto load = [&](const Org& o, int cc) {
    const __bf16* base = X + vox_id(v, o.b, o.d0 - 1, o.h0 - 1, o.w0 - 1) * xs + xo + cc;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int e = i * 256 + (int)threadIdx.x;
      const int vx = e / PV, j = e - vx * PV;
      const int iw = vx % IW, ih = (vx / IW) % IH, id = vx / (IW * IH);
      const bool ok = (NP * 256 == NV * PV || e < NV * PV) && (unsigned)(o.d0 - 1 + id) < (unsigned)v.D &&
                      (unsigned)(o.h0 - 1 + ih) < (unsigned)v.H && (unsigned)(o.w0 - 1 + iw) < (unsigned)v.W;
      rp[i] = ok ? *(const bf16x8*)(base + (long long)((id * v.H + ih) * v.W + iw) * xs + j * 8) : zero8;
    }
  };
  // lane bases: the voxel fragment's, and the weight row's
  const __bf16* lx = &sX[(2 * wave * IW + r) * VS + (CH >= 32 ? q : q & (PV - 1)) * 8];
  const __bf16* lw = Wk + (long long)(n0 + r) * K +
                     (CH >= 32 ? q * 8 : (q / PV) * CIN + (q & (PV - 1)) * 8);
  // Layers whose weight fragments fit beside the rest keep them in registers across the
  // block's tiles; the others read them again per tile (wofs hides the invariance).
  constexpr bool kKeepW = NC * NSL * NTB * 4 <= (TD == 1 ? 108 : 56);
  int wofs = 0;
  f32x4 acc[MF][NTB];
  auto slice = [&](int s, int cc) {
    bf16x8 w[NTB];
    // the slice's first tap and, for CH > 32, the channel it starts at
    constexpr int SPT = CH > 32 ? 1 : 0;
    const int k = s * 32;
    const int tap = k / CH, ch = SPT ? k - tap * CH : 0;
    int off;
    bool ok = true;
    if (CH == 48) {  // slices straddle taps: the lane's own
      const int kl = k + q * 8, t = kl / CH, c = kl - t * CH;
      ok = kl < 27 * CH;
      off = ok ? tap_off<IH, IW, VS>(t) + c - q * 8 : 0;
    } else if (CH >= 32) {
      off = tap_off<IH, IW, VS>(tap) + ch;
    } else {
      const int last = min(tap + TPS - 1, 26);
      off = tap_off<IH, IW, VS>(tap);
      if (q / PV >= 1) off = tap_off<IH, IW, VS>(min(tap + 1, last));
      if (TPS == 4) {
        if (q == 2) off = tap_off<IH, IW, VS>(min(tap + 2, last));
        if (q == 3) off = tap_off<IH, IW, VS>(min(tap + 3, last));
      }
      ok = tap + TPS <= 27 || tap + q / PV < 27;
    }
    const int wo = CH >= 32 ? (CH == CIN ? k : tap * CIN + cc + ch) : tap * CIN + cc;
#pragma unroll
    for (int n = 0; n < NTB; ++n) {
      const __bf16* p = lw + wofs + (long long)n * 16 * K + wo;
      w[n] = ok ? *(const bf16x8*)p : zero8;
    }
#pragma unroll
    for (int f = 0; f < MF; ++f) {
      const int fo = ((f >> 1) * IH + (f & 1)) * IW * VS;
      bf16x8 x = *(const bf16x8*)(lx + off + fo);
      if (!ok) x = zero8;
#pragma unroll
      for (int n = 0; n < NTB; ++n) acc[f][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[n], x, acc[f][n], 0, 0, 0);
    }
  };
  const int nb = gridDim.x;
  int t = xcd_block();
  Org o = org_of(t);
  load(o, 0);
  for (; t < ntiles; t += nb) {
    const Org cur = o;
#pragma unroll
    for (int f = 0; f < MF; ++f)
#pragma unroll
      for (int n = 0; n < NTB; ++n) acc[f][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ci = 0; ci < NC; ++ci) {
      if (!kKeepW) asm volatile("" : "+s"(wofs));
      __syncthreads();  // every wave is done with the previous chunk
#pragma unroll
      for (int i = 0; i < NP; ++i) {
        const int e = i * 256 + (int)threadIdx.x;
        const int vx = e / PV, j = e - vx * PV;
        if (NP * 256 == NV * PV || e < NV * PV) *(bf16x8*)&sX[vx * VS + j * 8] = rp[i];
      }
      __syncthreads();
      if (ci + 1 < NC) {
        load(cur, (ci + 1) * CH);
      } else if (t + nb < ntiles) {
        o = org_of(t + nb);
        load(o, 0);
      }
#pragma unroll
      for (int s = 0; s < NSL; ++s) slice(s, ci * CH);
    }
    const int w = cur.w0 + r;
    if (EPI != kConvUp) {
#pragma unroll
      for (int f = 0; f < MF; ++f) {
        const int d = cur.d0 + (f >> 1), h = cur.h0 + 2 * wave + (f & 1);
        if (d >= v.D || h >= v.H || w >= v.W) continue;
        const long long vi = vox_id(v, cur.b, d, h, w);
#pragma unroll
        for (int n = 0; n < NTB; ++n) {
          const int c = n0 + n * 16 + q * 4;
          f32x4 a = acc[f][n];
          if (EPI == kConvF32) {
            *(f32x4*)((float*)out.y + vi * out.ys + out.yo + c) = a;
            continue;
          }
          bf16x4 y;
          if (EPI == kConvFwd) {
            const f32x4 bs = *(const f32x4u*)(out.bias + c);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = f2bf(fmaxf(a[j] + bs[j], 0.f));
          } else {
            const bf16x4 m = *(const bf16x4*)(out.m + vi * out.ms + out.mo + c);
#pragma unroll
            for (int j = 0; j < 4; ++j) y[j] = f2bf(bf2f(m[j]) > 0.f ? a[j] : 0.f);
          }
          *(bf16x4*)((__bf16*)out.y + vi * out.ys + out.yo + c) = y;
        }
      }
    } else {
      // Concatenated input: the skip part is stored as it is; the upsampled part's
      // gradient is the sum of its eight children, (d, h, w) order, this wave's 2 x 2 rows
      // and lane pairs along w.
      const int h = cur.h0 + 2 * wave;
      const bool in = cur.d0 < v.D && h < v.H && w < v.W;  // extents are even: whole groups
      const long long vi = vox_id(v, cur.b, cur.d0, h, w);
      const Vol vc{v.B, v.D / 2, v.H / 2, v.W / 2};
      const long long vcI = vox_id(vc, cur.b, cur.d0 >> 1, h >> 1, w >> 1);
      const int cup = COUT - out.split;
#pragma unroll
      for (int n = 0; n < NTB; ++n) {
        const int c = n0 + n * 16 + q * 4;
        if (n0 + n * 16 < out.split) {
          if (in)
#pragma unroll
            for (int f = 0; f < MF; ++f)
              *(f32x4*)((float*)out.y + (vi + ((long long)(f >> 1) * v.H + (f & 1)) * v.W) * out.ys + out.yo + c) = acc[f][n];
          continue;
        }
        float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int f = 0; f < MF; ++f)
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            s[j] += acc[f][n][j];
            s[j] += __shfl_xor(acc[f][n][j], 1, 64);
          }
        if (in && !(r & 1)) {
          const int cc = c - out.split;
          const bf16x4 m = *(const bf16x4*)(out.m + vcI * out.ms + out.mo + cc);
          bf16x4 y;
#pragma unroll
          for (int j = 0; j < 4; ++j) y[j] = f2bf(bf2f(m[j]) > 0.f ? s[j] : 0.f);
          *(bf16x4*)(out.up + vcI * cup + cc) = y;
        }
      }
    }
  }
}

// Output tiles per launch: enough blocks to fill the chip, each walking several tiles
// when there are more (kConvBlocks: 4 blocks of 256 threads per CU).
constexpr int kConvBlocks = 1024;
template <int CIN, int COUT, int CH, int TD, int NTB, int EPI>
static void conv3_tile_launch(const Vol& v, const __bf16* X, int xs, int xo, const __bf16* Wk, const ConvOut& out,
                              hipStream_t s) {
  const long long tiles = (long long)v.B * ((v.D + TD - 1) / TD) * ((v.H + 7) / 8) * ((v.W + 15) / 16);
  const unsigned nb = (unsigned)std::min<long long>(tiles, std::max(8, kConvBlocks / (COUT / (16 * NTB)) / 8 * 8));
  hipLaunchKernelGGL((k_conv3_tile<CIN, COUT, CH, TD, NTB, EPI>), dim3(nb, COUT / (16 * NTB)), dim3(256), 0, s, v,
                     (int)tiles, X, xs, xo, Wk, out);
}

// Tile depth and channel tiles per block: two planes and two channel tiles where the
// launch still has at least 512 blocks (two per CU), else one.
template <int CIN, int COUT, int CH, int EPI>
static void conv3_tile_pick(const Vol& v, const __bf16* X, int xs, int xo, const __bf16* Wk, const ConvOut& out,
                            hipStream_t s) {
  constexpr bool kDeep = 4 * 180 * (CH + 8) * 2 <= 80 * 1024;  // two blocks' two-plane tiles fit a CU's LDS
  const long long tiles1 = (long long)v.B * v.D * ((v.H + 7) / 8) * ((v.W + 15) / 16);
  const bool td2 = kDeep && v.D % 2 == 0 && tiles1 / 2 * (COUT / 16) >= 512;
  const bool ntb2 = COUT >= 32 && (td2 ? tiles1 / 2 : tiles1) * (COUT / 32) >= 512;
  constexpr int TD2 = kDeep ? 2 : 1, NT2 = COUT >= 32 ? 2 : 1;
  if (td2 && ntb2)
    conv3_tile_launch<CIN, COUT, CH, TD2, NT2, EPI>(v, X, xs, xo, Wk, out, s);
  else if (td2)
    conv3_tile_launch<CIN, COUT, CH, TD2, 1, EPI>(v, X, xs, xo, Wk, out, s);
  else if (ntb2)
    conv3_tile_launch<CIN, COUT, CH, 1, NT2, EPI>(v, X, xs, xo, Wk, out, s);
  else
    conv3_tile_launch<CIN, COUT, CH, 1, 1, EPI>(v, X, xs, xo, Wk, out, s);
}

// Whether a layer's forward pass takes less time on tiles of 8 x 16 rows and columns: not where
// over half of their voxels lie outside and these come to more than the launch itself costs.
// Whole networks, us, gathered / tiled: 1 x 4096 x 4 x 4 271 / 585, 1 x 256 x 256 x 4 528 / 784,
// 1 x 96 x 96 x 4 388 / 433, 1 x 64 x 64 x 4 272 / 249, 1 x 256 x 4 x 4 195 / 149, 1 x 128 x 128 x 8
// 364 / 346, 1 x 256 x 256 x 12 1,156 / 1,037.
static bool conv3_tile_fits(const Vol& v, int cin, int cout) {
  const long long rows = (long long)v.B * v.D, padded = rows * ((v.H + 7) / 8 * 8) * ((v.W + 15) / 16 * 16);
  return padded <= 2 * rows * v.H * v.W || padded * cin * cout <= 1 << 26;
}

// Layers with more than 32 input channels are staged in chunks where the extents divide
// into tiles, and whole otherwise: the two orders of k that the forward pass has always
// had there.
template <int CIN, int COUT>
static void conv3_fwd_t(const Vol& v, const __bf16* X, int xs, int xo, const __bf16* Wk,
                        const float* bias, __bf16* Y, int ys, int yo, hipStream_t s) {
  constexpr int CH = CIN <= 32 ? CIN : CIN % 32 == 0 ? 32 : 16;
  if (!conv3_tile_enabled() || !conv3_tile_fits(v, CIN, COUT)) {
    const long long V = (long long)v.B * v.D * v.H * v.W;
    hipLaunchKernelGGL((k_conv3<CIN, COUT>), dim3((unsigned)((V + 63) / 64), COUT / 16), dim3(256), 0, s, v, X, xs,
                       xo, Wk, bias, Y, ys, yo);
    return;
  }
  const ConvOut out{bias, Y, ys, yo, nullptr, 0, 0, 0, nullptr};
  if (CH == CIN || (v.W % 16 == 0 && v.H % 8 == 0))
    conv3_tile_pick<CIN, COUT, CH, kConvFwd>(v, X, xs, xo, Wk, out, s);
  else
    conv3_tile_pick<CIN, COUT, CIN, kConvFwd>(v, X, xs, xo, Wk, out, s);
}

void conv3_forward(int cin, int cout, const Vol& v, const __bf16* X, int xs, int xo, const __bf16* Wk,
                   const float* bias, __bf16* Y, int ys, int yo, hipStream_t s) {
#define AQU_FWD(CI, CO) \
  if (cin == CI && cout == CO) return conv3_fwd_t<CI, CO>(v, X, xs, xo, Wk, bias, Y, ys, yo, s);
  AQU_FWD(8, 16) AQU_FWD(16, 16) AQU_FWD(16, 32) AQU_FWD(32, 32) AQU_FWD(32, 64) AQU_FWD(64, 64)
  AQU_FWD(96, 32) AQU_FWD(48, 16)
#undef AQU_FWD
}

// Input gradient: dX[v, c] = sum_{tap, n} dYpre[v - off(tap), n] * W[n, tap, c], computed as a
// convolution of dYpre (cout channels) with Wt[c, tap', n] = W[n, 26 - tap', c].
// dX in FP32 (the pooled layers, whose gradient is added to another).
void conv3_dgrad(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* Wt, float* dX, hipStream_t s) {
  const ConvOut out{nullptr, dX, cin, 0, nullptr, 0, 0, 0, nullptr};
  if (cin == 16 && cout == 32) return conv3_tile_pick<32, 16, 32, kConvF32>(v, dY, 32, 0, Wt, out, s);
  if (cin == 32 && cout == 64) return conv3_tile_pick<64, 32, 64, kConvF32>(v, dY, 64, 0, Wt, out, s);
}
// The same through the ReLU whose outputs are M: dYpre of the layer below, bf16, dense.
void conv3_dgrad_relu(int c, const Vol& v, const __bf16* dY, const __bf16* Wt, const __bf16* M, int ms, int mo,
                      __bf16* dYpre, hipStream_t s) {
  const ConvOut out{nullptr, dYpre, c, 0, M, ms, mo, 0, nullptr};
  if (c == 16) return conv3_tile_pick<16, 16, 16, kConvMask>(v, dY, 16, 0, Wt, out, s);
  if (c == 32) return conv3_tile_pick<32, 32, 32, kConvMask>(v, dY, 32, 0, Wt, out, s);
  if (c == 64) return conv3_tile_pick<64, 64, 64, kConvMask>(v, dY, 64, 0, Wt, out, s);
}
// The same for a concatenated input of `cin` channels: the skip part's gradient (the first
// cin/3 channels) in FP32, the upsampled part's through its upsampling and ReLU (outputs
// M, dense, half extents) to dYpre of that layer.
void conv3_dgrad_concat(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* Wt, float* skip,
                        const __bf16* M, __bf16* up, hipStream_t s) {
  const int split = cin / 3;
  const ConvOut out{nullptr, skip, split, 0, M, cin - split, 0, split, up};
  if (cin == 48 && cout == 16) return conv3_tile_launch<16, 48, 16, 2, 3, kConvUp>(v, dY, 16, 0, Wt, out, s);
  if (cin == 96 && cout == 32) return conv3_tile_launch<32, 96, 32, 2, 2, kConvUp>(v, dY, 32, 0, Wt, out, s);
}

// ------------------------------------------------------------------ weight gradient
// dW[n, tap, c] = sum_v dYpre[v, n] * X[v + off(tap), c]: per tap an MFMA GEMM
// (COUT x CIN) with K = voxels, one w row of up to RW voxels at a time. The rows are
// dealt round-robin to `nsplit` splits; a one-wave block owns a split, one (dd, dh)
// pair of taps and 16*NTB input channels, and keeps the three dw taps' accumulators
// over all its rows. Both operands have K as their strided dimension (channels-last),
// so a row is staged in LDS as it lies in memory -- 16-byte pieces, one zero voxel
// either side -- and read transposed (ds_read_b64_tr_b16: lane i of 16 receives element
// i of four consecutive voxels); a dw shift is then an address offset, and one staged X
// row serves three taps. The next row's pieces are loaded into registers while the
// current one is multiplied. Partial sums go to `part` [split][tap][COUT][CIN] and are
// folded in split order by k_fold_wgrad.
// Bound by LDS reads (1 KB per MFMA when COUT = 16). 8 x 64^3 (the training batch),
// 48 -> 16: 5,880 -> 228 us, 16 -> 16: 1,878 -> 132 us, 96 -> 32 at 32^3: 3,166 -> 113 us
// against one tap per block with 2-byte transposing LDS stores.
constexpr int kWgRow = 64;  // longest row the staging holds

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Eight consecutive k (rows of the LDS tile, `stride` bf16 apart) of column lane % 16,
// for lane group q = lane / 16: the MFMA operand layout. p: the tile's first row and
// column; lane i of a group addresses row i / 4, columns 4 (i % 4) .. +3.
__device__ __forceinline__ bf16x8 lds_read_k8(const __bf16* p, int stride, int lane) {
  const __bf16* a = p + (8 * (lane >> 4) + ((lane & 15) >> 2)) * stride + 4 * (lane & 3);
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)a);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(a + 4 * stride));
  return __builtin_bit_cast(bf16x8, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// LDS row stride for C channels: 64 channels are padded so that the four voxels a lane
// group reads at once fall in distinct banks.
constexpr int wg_stride(int C) { return C == 64 ? 80 : C; }

template <int CIN, int COUT, int NTB, int RW>
__global__ __launch_bounds__(64) void k_conv3_wgrad(Vol v, const __bf16* __restrict__ dY,
                                                    const __bf16* __restrict__ X, int xs, int xo,
                                                    float* __restrict__ part, int nsplit) {
  constexpr int MT = COUT / 16, KCH = RW / 32;
  constexpr int XC = 16 * NTB;                          // staged input channels
  constexpr int XP = (CIN < 16 ? CIN : XC) / 8;         // 16-byte pieces per voxel
  constexpr int XST = wg_stride(XC), YST = wg_stride(COUT);
  constexpr int NX = (RW * XP + 63) / 64, NY = RW * (COUT / 8) / 64;  // pieces per lane
  static_assert(NY * 64 == RW * (COUT / 8), "whole pieces per lane");
  __shared__ __align__(16) __bf16 sX[(RW + 2) * XST];
  __shared__ __align__(16) __bf16 sY[RW * YST];
  const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
  const int split = xcd_block();  // neighbouring splits hold neighbouring rows: one XCD
  const int dd = (int)blockIdx.y / 3 - 1, dh = (int)blockIdx.y % 3 - 1;
  const int c0 = (int)blockIdx.z * XC;
  const bf16x8 zero8 = {};
  for (int e = lane; e < (RW + 2) * XST / 8; e += 64) *(bf16x8*)&sX[e * 8] = zero8;
  for (int e = lane; e < RW * YST / 8; e += 64) *(bf16x8*)&sY[e * 8] = zero8;
  f32x4 acc[3][MT][NTB];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int n = 0; n < NTB; ++n) acc[t][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nrows = v.B * v.D * v.H;  // rows of at least 4 voxels: fits 32 bits with the tensors in memory
  bf16x8 rx[NX], ry[NY];
  auto load = [&](int row) {
    const int h = row % v.H, t = row / v.H;
    const int d = t % v.D, b = t / v.D;
    const int sd = d + dd, sh = h + dh;
    const bool ok = sd >= 0 && sd < v.D && sh >= 0 && sh < v.H;
    const __bf16* py = dY + vox_id(v, b, d, h, 0) * COUT;
    const __bf16* px = X + vox_id(v, b, ok ? sd : d, ok ? sh : h, 0) * xs + xo + c0;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = i * 64 + lane, w = e / XP, j = e - w * XP;
      rx[i] = ok && w < v.W ? *(const bf16x8*)(px + (long long)w * xs + j * 8) : zero8;
    }
#pragma unroll
    for (int i = 0; i < NY; ++i) {
      const int e = i * 64 + lane, w = e / (COUT / 8);
      ry[i] = w < v.W ? *(const bf16x8*)(py + e * 8) : zero8;
    }
  };
  load(split);
  const int kch = (v.W + 31) / 32;
  for (int row = split; row < nrows; row += nsplit) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int e = i * 64 + lane, w = e / XP, j = e - w * XP;
      if (NX * 64 == RW * XP || w < RW) *(bf16x8*)&sX[(w + 1) * XST + j * 8] = rx[i];
    }
#pragma unroll
    for (int i = 0; i < NY; ++i) {
      const int e = i * 64 + lane, w = e / (COUT / 8), j = e - w * (COUT / 8);
      *(bf16x8*)&sY[w * YST + j * 8] = ry[i];
    }
    __syncthreads();
    if (row + nsplit < nrows) load(row + nsplit);
#pragma unroll
    for (int kc = 0; kc < KCH; ++kc) {
      if (kc >= kch) break;
      bf16x8 a[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m) a[m] = lds_read_k8(&sY[kc * 32 * YST + m * 16], YST, lane);
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int n = 0; n < NTB; ++n) {
          bf16x8 x = lds_read_k8(&sX[(kc * 32 + t) * XST + n * 16], XST, lane);
          // voxel W is outside: its dw = -1 source, voxel W - 1, is not (dY is 0 there,
          // but 0 times an infinity is not)
          if (t == 0 && v.W - kc * 32 < 32) {
#pragma unroll
            for (int j = 0; j < 8; ++j)
              if (kc * 32 + q * 8 + j == v.W) x[j] = f2bf(0.f);
          }
#pragma unroll
          for (int m = 0; m < MT; ++m)
            acc[t][m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], x, acc[t][m][n], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int n = 0; n < NTB; ++n) {
      const int c = c0 + n * 16 + r;
      if (c >= CIN) continue;
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          part[(((long long)split * 27 + blockIdx.y * 3 + t) * COUT + m * 16 + q * 4 + j) * CIN + c] = acc[t][m][n][j];
    }
}

// Bias gradient partials: per-block sums of dYpre over vox_per_block voxels. A channel's
// voxels are dealt to 256 / C slots, each summed in voxel order by one thread (two
// channels per thread, kBiasAhead loads in flight), then the slots in order.
constexpr int kBiasBlocks = 512, kBiasAhead = 16;
__global__ __launch_bounds__(128) void k_bias_part(long long V, int C, const __bf16* __restrict__ dYpre,
                                                   float* __restrict__ bpart, int vox_per_block) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  __shared__ float red[256];
  const int C2 = C / 2, slots = 256 / C;
  const int slot = (int)threadIdx.x / C2, c = ((int)threadIdx.x - slot * C2) * 2;
  const long long v0 = (long long)blockIdx.x * vox_per_block;
  const int nv = (int)std::max<long long>(0, std::min<long long>(vox_per_block, V - v0));
  const __bf16* p = dYpre + v0 * C + c;
  float a0 = 0.f, a1 = 0.f;
  int i = slot;
  for (; i + (kBiasAhead - 1) * slots < nv; i += kBiasAhead * slots) {
    bf16x2 t[kBiasAhead];
#pragma unroll
    for (int k = 0; k < kBiasAhead; ++k) t[k] = *(const bf16x2*)(p + (long long)(i + k * slots) * C);
#pragma unroll
    for (int k = 0; k < kBiasAhead; ++k) a0 += bf2f(t[k][0]), a1 += bf2f(t[k][1]);
  }
  for (; i < nv; i += slots) {
    const bf16x2 t = *(const bf16x2*)(p + (long long)i * C);
    a0 += bf2f(t[0]), a1 += bf2f(t[1]);
  }
  red[slot * C + c] = a0;
  red[slot * C + c + 1] = a1;
  __syncthreads();
  if ((int)threadIdx.x < C) {
    float s = 0.f;
    for (int k = 0; k < slots; ++k) s += red[k * C + threadIdx.x];
    bpart[(long long)blockIdx.x * C + threadIdx.x] = s;
  }
}

// Sum of base[e], base[stride + e], ... over `rows` values, in order, kFoldAhead loads in
// flight together: a chain of round trips and of additions, so as few of the former as
// registers allow. base and stride are the block's, so that the rows' addresses are scalar.
// Per layer of a 2 x 24 x 20 x 28 batch (256 splits, 512 bias rows): 32 loads 10.2 us, 128
// 7.7. (Four groups of lanes taking 128 bias rows each at once: 8.2.)
constexpr int kFoldAhead = 128;
__device__ __forceinline__ float fold_column(const float* __restrict__ base, uint32_t e, long long stride, int rows) {
  float s = 0.f;
  int r = 0;
  for (; r + kFoldAhead <= rows; r += kFoldAhead) {
    float t[kFoldAhead];
#pragma unroll
    for (int k = 0; k < kFoldAhead; ++k) t[k] = (base + (r + k) * stride)[e];
#pragma unroll
    for (int k = 0; k < kFoldAhead; ++k) s += t[k];
  }
  for (; r + 8 <= rows; r += 8) {
    float t[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) t[k] = (base + (r + k) * stride)[e];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += t[k];
  }
  for (; r < rows; ++r) s += (base + r * stride)[e];
  return s;
}
// dW[n][tap*CIN + c] = sum over splits (in order) of part[split][tap][n][c], and the bias
// gradient db[n] likewise of bpart[block][n].
__global__ __launch_bounds__(64) void k_fold_wgrad(const float* __restrict__ part, const float* __restrict__ bpart,
                                                   int nsplit, int cin, int cout, float* __restrict__ dW,
                                                   float* __restrict__ db) {
  const int total = 27 * cout * cin;  // a multiple of 64: a block folds weights or biases
  const bool isw = (int)blockIdx.x * 64 < total;
  const int e = (int)(blockIdx.x * 64 + threadIdx.x) - (isw ? 0 : total);
  if (!isw && e >= cout) return;
  const float s = fold_column(isw ? part : bpart, (uint32_t)e, isw ? total : cout, isw ? nsplit : kBiasBlocks);
  if (!isw) {
    db[e] = s;
    return;
  }
  const int c = e % cin, t2 = e / cin;
  const int n = t2 % cout, tap = t2 / cout;
  dW[n * 27 * cin + tap * cin + c] = s;
}

template <int CIN, int COUT, int NTB>
static void wgrad_t(const Vol& v, const __bf16* dY, const __bf16* X, int xs, int xo, float* part,
                    float* bpart, int nsplit, float* dW, float* db, hipStream_t s) {
  // a split without rows would only add zeros
  nsplit = std::min(nsplit, v.B * v.D * v.H);
  const dim3 grid(nsplit, 9, (CIN + 16 * NTB - 1) / (16 * NTB));
  if (v.W > 32)
    hipLaunchKernelGGL((k_conv3_wgrad<CIN, COUT, NTB, 64>), grid, dim3(64), 0, s, v, dY, X, xs, xo, part, nsplit);
  else
    hipLaunchKernelGGL((k_conv3_wgrad<CIN, COUT, NTB, 32>), grid, dim3(64), 0, s, v, dY, X, xs, xo, part, nsplit);
  const long long V = (long long)v.B * v.D * v.H * v.W;
  hipLaunchKernelGGL(k_bias_part, dim3(kBiasBlocks), dim3(128), 0, s, V, COUT, dY, bpart,
                     (int)((V + kBiasBlocks - 1) / kBiasBlocks));
  const int total = 27 * CIN * COUT + COUT;
  hipLaunchKernelGGL(k_fold_wgrad, dim3((total + 63) / 64), dim3(64), 0, s, part, bpart, nsplit, CIN, COUT, dW, db);
}

void conv3_wgrad(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* X, int xs, int xo,
                 float* part, float* bpart, int nsplit, float* dW, float* db, hipStream_t s) {
#define AQU_WG(CI, CO, NTB) \
  if (cin == CI && cout == CO) return wgrad_t<CI, CO, NTB>(v, dY, X, xs, xo, part, bpart, nsplit, dW, db, s);
  AQU_WG(8, 16, 1) AQU_WG(16, 16, 1) AQU_WG(16, 32, 1) AQU_WG(32, 32, 2) AQU_WG(32, 64, 2) AQU_WG(64, 64, 2)
  AQU_WG(96, 32, 3) AQU_WG(48, 16, 3)
#undef AQU_WG
}

// ------------------------------------------------------------------ skip connections backward
// dYpre of a layer whose output goes to a skip connection (gradient dS, FP32, dense) and
// to an average pooling (gradient dP of the pooled tensor, vo): (dS + dP / 8) * (Y > 0) as
// bf16, 8 channels per thread.
__global__ void k_skip_bwd(Vol v, int C8, const __bf16* __restrict__ Y, int ys, const float* __restrict__ dS,
                           const float* __restrict__ dP, __bf16* __restrict__ dYpre) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long vv = e / C8;
  if (vv >= (long long)v.B * v.D * v.H * v.W) return;
  const int c = (int)(e - vv * C8) * 8;
  const VoxelPos p = vox_of(v, vv);
  const Vol vo{v.B, v.D / 2, v.H / 2, v.W / 2};
  const float* pp = dP + vox_id(vo, p.b, p.d >> 1, p.h >> 1, p.w >> 1) * (C8 * 8) + c;
  const bf16x8 y = *(const bf16x8*)(Y + vv * ys + c);
  const f32x4 s0 = *(const f32x4*)(dS + e * 8), s1 = *(const f32x4*)(dS + e * 8 + 4);
  const f32x4 p0 = *(const f32x4*)pp, p1 = *(const f32x4*)(pp + 4);
  bf16x8 o;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float g = (k < 4 ? s0[k & 3] : s1[k & 3]) + (k < 4 ? p0[k & 3] : p1[k & 3]) * 0.125f;
    o[k] = f2bf(bf2f(y[k]) > 0.f ? g : 0.f);
  }
  *(bf16x8*)(dYpre + e * 8) = o;
}
void skip_bwd(const Vol& v, int C, const __bf16* Y, int ys, const float* dS, const float* dP, __bf16* dYpre,
              hipStream_t s) {
  const long long n8 = (long long)v.B * v.D * v.H * v.W * (C / 8);
  hipLaunchKernelGGL(k_skip_bwd, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, s, v, C / 8, Y, ys, dS, dP, dYpre);
}

// out[c] = sum over rows (in order) of part[row][c], C <= 64. 512 rows: 14.7 -> 6.1 us against
// staging them in LDS.
__global__ __launch_bounds__(64) void k_fold_rows(const float* __restrict__ part, int rows, int C,
                                                  float* __restrict__ out) {
  if ((int)threadIdx.x < C) out[threadIdx.x] = fold_column(part, threadIdx.x, C, rows);
}

// ------------------------------------------------------------------ pooling / upsampling
// 2x2x2 average pooling (bf16).
// One thread per output voxel and 8 consecutive channels; the eight children are
// summed in the same (d, h, w) order for every channel.
__global__ void k_avgpool(Vol vo, int C, const __bf16* __restrict__ X, int xs, int xo,
                          __bf16* __restrict__ Y, int row0) {
  const int C8 = C >> 3;
  const unsigned e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= (unsigned)vo.W * C8) return;
  const int w = (int)(e / C8), j = (int)(e - (unsigned)w * C8);
  unsigned row = row0 + blockIdx.y;  // (b, d, h) of the output
  const int h = (int)(row % vo.H);
  row /= vo.H;
  const int d = (int)(row % vo.D), b = (int)(row / vo.D);
  const Vol vi{vo.B, vo.D * 2, vo.H * 2, vo.W * 2};
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const bf16x8 x8 =
        *(const bf16x8*)(X + vox_id(vi, b, 2 * d + (k >> 2), 2 * h + ((k >> 1) & 1), 2 * w + (k & 1)) * xs + xo + 8 * j);
#pragma unroll
    for (int c = 0; c < 8; ++c) acc[c] += bf2f(x8[c]);
  }
  bf16x8 o8;
#pragma unroll
  for (int c = 0; c < 8; ++c) o8[c] = f2bf(acc[c] * 0.125f);
  *(bf16x8*)(Y + vox_id(vo, b, d, h, w) * C + 8 * j) = o8;
}
// Nearest 2x upsampling into a channel slice.
// One thread per output voxel and 8 consecutive channels (a 16-byte load and store).
__global__ void k_upsample(Vol vi, int C, const __bf16* __restrict__ X, __bf16* __restrict__ Y, int ys,
                           int yo, int row0) {
  const int C8 = C >> 3;
  const int Wo = vi.W * 2, Ho = vi.H * 2, Do = vi.D * 2;
  const unsigned e = blockIdx.x * blockDim.x + threadIdx.x;
  const unsigned nrow = (unsigned)Wo * C8;
  if (e >= nrow) return;
  const int w = (int)(e / C8), j = (int)(e - (unsigned)w * C8);
  unsigned row = row0 + blockIdx.y;  // (b, d, h) of the output
  const int h = (int)(row % Ho);
  row /= Ho;
  const int d = (int)(row % Do), b = (int)(row / Do);
  const long long o = (((long long)b * Do + d) * Ho + h) * Wo + w;
  const long long i = vox_id(vi, b, d >> 1, h >> 1, w >> 1);
  *(bf16x8*)(Y + o * ys + yo + 8 * j) = *(const bf16x8*)(X + i * C + 8 * j);
}
static inline int nb1(long long n) { return (int)((n + 255) / 256); }
void avgpool(const Vol& vo, int C, const __bf16* X, int xs, int xo, __bf16* Y, hipStream_t s) {
  const int rows = vo.B * vo.D * vo.H;
  for (int r0 = 0; r0 < rows; r0 += 65535) {  // grid.y limit
    const dim3 grid((unsigned)((vo.W * (C / 8) + 255) / 256), (unsigned)std::min(65535, rows - r0));
    hipLaunchKernelGGL(k_avgpool, grid, dim3(256), 0, s, vo, C, X, xs, xo, Y, r0);
  }
}
void upsample(const Vol& vi, int C, const __bf16* X, __bf16* Y, int ys, int yo, hipStream_t s) {
  const int rows = vi.B * vi.D * 2 * vi.H * 2;
  for (int r0 = 0; r0 < rows; r0 += 65535) {  // grid.y limit
    const dim3 grid((unsigned)((vi.W * 2 * (C / 8) + 255) / 256), (unsigned)std::min(65535, rows - r0));
    hipLaunchKernelGGL(k_upsample, grid, dim3(256), 0, s, vi, C, X, Y, ys, yo, r0);
  }
}

// ------------------------------------------------------------------ output head (1x1x1, C -> 1)
__global__ void k_head(long long V, int C, const __bf16* __restrict__ X, const float* __restrict__ w,
                       const float* __restrict__ b, float* __restrict__ y) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  float s = b[0];
  for (int c0 = 0; c0 < C; c0 += 8) {  // C is a multiple of 8: 16-byte loads
    const bf16x8 x8 = *(const bf16x8*)(X + i * C + c0);
#pragma unroll
    for (int c = 0; c < 8; ++c) s += w[c0 + c] * bf2f(x8[c]);
  }
  y[i] = s;
}
// Head backward: dYpre of the layer below, dy * w through its ReLU (outputs X) as bf16,
// and per-block partial sums of the head's own gradient: dy * X per channel and dy.
template <int C>
__global__ __launch_bounds__(256) void k_head_bwd(long long V, const __bf16* __restrict__ X,
                                                  const float* __restrict__ w, const float* __restrict__ dy,
                                                  __bf16* __restrict__ dYpre, float* __restrict__ part, int vpb) {
  constexpr int RS = 257;  // rows of one channel's partials, one bank apart
  __shared__ float red[(C + 1) * RS];
  float acc[C + 1], wc[C];
#pragma unroll
  for (int c = 0; c <= C; ++c) acc[c] = 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c) wc[c] = w[c];
  const long long v0 = (long long)blockIdx.x * vpb;
  for (int i = threadIdx.x; i < vpb; i += 256) {
    const long long vv = v0 + i;
    if (vv >= V) break;
    const float g = dy[vv];
#pragma unroll
    for (int c0 = 0; c0 < C; c0 += 8) {
      const bf16x8 x8 = *(const bf16x8*)(X + vv * C + c0);
      bf16x8 o;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float x = bf2f(x8[c]);
        o[c] = f2bf(x > 0.f ? g * wc[c0 + c] : 0.f);
        acc[c0 + c] += g * x;
      }
      *(bf16x8*)(dYpre + vv * C + c0) = o;
    }
    acc[C] += g;
  }
#pragma unroll
  for (int c = 0; c <= C; ++c) red[c * RS + threadIdx.x] = acc[c];
  __syncthreads();
  if ((int)threadIdx.x <= C) {
    float s = 0.f;
#pragma unroll 16
    for (int k = 0; k < 256; ++k) s += red[threadIdx.x * RS + k];
    part[(long long)blockIdx.x * (C + 1) + threadIdx.x] = s;
  }
}
void head_fwd(long long V, int C, const __bf16* X, const float* w, const float* b, float* y, hipStream_t s) {
  hipLaunchKernelGGL(k_head, dim3(nb1(V)), dim3(256), 0, s, V, C, X, w, b, y);
}
void head_bwd(long long V, const __bf16* X, const float* w, const float* dy, __bf16* dYpre, float* part,
              int nblk, float* dwb, hipStream_t s) {
  constexpr int C = 16;
  const int vpb = (int)((V + nblk - 1) / nblk);
  hipLaunchKernelGGL(k_head_bwd<C>, dim3(nblk), dim3(256), 0, s, V, X, w, dy, dYpre, part, vpb);
  hipLaunchKernelGGL(k_fold_rows, dim3(1), dim3(64), 0, s, part, nblk, C + 1, dwb);
}

// ------------------------------------------------------------------ loss
// Masked mean-squared error over fluid voxels: per-block partials of sum (y-t)^2*m
// and sum m, folded in order; the gradient dy = 2 (y - t) m / sum m needs the
// total, so it is a second pass.
__global__ void k_loss_partial(long long V, const float* __restrict__ y, const float* __restrict__ t,
                               const float* __restrict__ m, double* __restrict__ part, int vpb) {
  __shared__ double s1[256], s2[256];
  double a = 0, c = 0;
  const long long v0 = (long long)blockIdx.x * vpb;
  for (int i = threadIdx.x; i < vpb; i += 256) {
    const long long vv = v0 + i;
    if (vv >= V) break;
    const double d = (double)y[vv] - (double)t[vv];
    a += d * d * m[vv];
    c += m[vv];
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = c;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}
// The partials are staged in LDS by the whole block; one thread per column adds them in
// order (from memory, one dependent load per term took 36 us).
__global__ __launch_bounds__(256) void k_loss_fold(const double* __restrict__ part, int n, double* __restrict__ out) {
  __shared__ double sp[2048], tot[2];
  double s = 0;
  for (int i0 = 0; i0 < n; i0 += 1024) {
    const int m = min(1024, n - i0);
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * m; i += 256) sp[i] = part[2 * i0 + i];
    __syncthreads();
    if (threadIdx.x < 2)
#pragma unroll 8
      for (int i = 0; i < m; ++i) s += sp[2 * i + threadIdx.x];
  }
  if (threadIdx.x < 2) tot[threadIdx.x] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    out[0] = tot[1] > 0 ? tot[0] / tot[1] : 0.0;
    out[1] = tot[1];
  }
}
__global__ void k_loss_grad(long long V, const float* __restrict__ y, const float* __restrict__ t,
                            const float* __restrict__ m, const double* __restrict__ tot,
                            float* __restrict__ dy) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= V) return;
  const double c = tot[1];
  dy[i] = c > 0 ? (float)(2.0 * ((double)y[i] - (double)t[i]) * m[i] / c) : 0.f;
}
void masked_mse(long long V, const float* y, const float* t, const float* m, double* part, int nblk,
                double* out, float* dy, hipStream_t s) {
  const int vpb = (int)((V + nblk - 1) / nblk);
  hipLaunchKernelGGL(k_loss_partial, dim3(nblk), dim3(256), 0, s, V, y, t, m, part, vpb);
  hipLaunchKernelGGL(k_loss_fold, dim3(1), dim3(256), 0, s, part, nblk, out);
  if (dy) hipLaunchKernelGGL(k_loss_grad, dim3(nb1(V)), dim3(256), 0, s, V, y, t, m, out, dy);
}

// ------------------------------------------------------------------ parameters
// Adam on FP32 master weights (bias-corrected step sizes passed in), then the bf16
// copies the convolutions read.
__global__ void k_adam(long long n, float* __restrict__ w, const float* __restrict__ g,
                       float* __restrict__ m, float* __restrict__ vv, float lr_t, float b1, float b2,
                       float eps) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * vv[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  vv[i] = vi;
  w[i] -= lr_t * mi / (sqrtf(vi) + eps);
}
void adam(long long n, float* w, const float* g, float* m, float* v, float lr_t, float b1, float b2,
          float eps, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, dim3(nb1(n)), dim3(256), 0, s, n, w, g, m, v, lr_t, b1, b2, eps);
}

// Forward weights Wk[n][tap*cin + c] and flipped transposed input-gradient weights
// Wt[c][tap'*cout + n] = W[n][(26 - tap')*cin + c], both bf16.
__global__ void k_pack_weights(int cin, int cout, const float* __restrict__ W, __bf16* __restrict__ Wk,
                               __bf16* __restrict__ Wt) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  const int total = 27 * cin * cout;
  if (e >= total) return;
  const int c = e % cin;
  const int t2 = e / cin;
  const int tap = t2 % 27;
  const int n = t2 / 27;
  const __bf16 v = f2bf(W[e]);
  Wk[e] = v;
  if (Wt) Wt[(long long)c * 27 * cout + (26 - tap) * cout + n] = v;
}
void pack_weights(int cin, int cout, const float* W, __bf16* Wk, __bf16* Wt, hipStream_t s) {
  const int total = 27 * cin * cout;
  hipLaunchKernelGGL(k_pack_weights, dim3((total + 255) / 256), dim3(256), 0, s, cin, cout, W, Wk, Wt);
}

// ------------------------------------------------------------------ fills
__global__ void k_zero_f32(float* __restrict__ p, long long n) {
  long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long)gridDim.x * blockDim.x;
  for (; i < n; i += st) p[i] = 0.f;
}
void zero_f32(float* p, long long n, hipStream_t s) {
  int nb = (int)std::min<long long>((n + 255) / 256, 8192);
  if (nb < 1) nb = 1;
  hipLaunchKernelGGL(k_zero_f32, dim3(nb), dim3(256), 0, s, p, n);
}

// Probe of the MFMA lane layout assumed above: D = A (16x32) * B (32x16), A and B
// given row-major in FP32, D row-major.
__global__ void k_mfma_probe(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ D) {
  const int l = threadIdx.x;
  const int r = l & 15, q = l >> 4;
  bf16x8 a, b;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    a[j] = f2bf(A[r * 32 + q * 8 + j]);
    b[j] = f2bf(B[(q * 8 + j) * 16 + r]);
  }
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) D[(q * 4 + i) * 16 + r] = c[i];
}
void mfma_probe(const float* A, const float* B, float* D, hipStream_t s) {
  hipLaunchKernelGGL(k_mfma_probe, dim3(1), dim3(64), 0, s, A, B, D);
}

}  // namespace aqu

// ------------------------------------------------------------------ FLIP grid <-> network tensors
// The network sees the FLIP interior as one volume with (D, H, W) = (X, Y, Z), the
// same x-major, z-fastest order as the cell hash.
#include "aqflip_internal.h"

namespace aqu {

__device__ __forceinline__ void cell3(const aqf::Geom& G, long long n, int& x, int& y, int& z) {
  const uint32_t u = (uint32_t)n;  // n < X*Y*Z < 2^31
  x = (int)aqf::fast_div(u, G.divYZ);
  const uint32_t r = u - (uint32_t)x * (uint32_t)(G.Y * G.Z);
  y = (int)aqf::fast_div(r, G.divZ);
  z = (int)(r - (uint32_t)y * (uint32_t)G.Z);
}

// sigma = RMS of the right-hand side b over FLUID cells: sig[0] = sigma, sig[1] = 1/sigma
// (0 when there is no fluid or b vanishes).
__global__ void k_nn_sigma_part(aqf::Geom G, const uint8_t* __restrict__ content,
                                const float* __restrict__ rhs, double* __restrict__ part) {
  __shared__ double s1[256], s2[256];
  double a = 0, c = 0;
  const long long n0 = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long st = (long long)gridDim.x * blockDim.x;
  for (long long n = n0; n < G.ncells_hash; n += st) {
    int x, y, z;
    cell3(G, n, x, y, z);
    const long long gi = G.g(x, y, z);
    if (content[gi] != aqf::FLUID) continue;
    const double b = (double)rhs[gi];
    a += b * b;
    c += 1.0;
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = c;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}
// Sums of the two columns of n partial pairs, by one 256-thread block: thread t adds
// pairs t, t + 256, ... in order, then a fixed-shape tree (deterministic). The result
// is returned to thread 0.
__device__ void fold_pairs(const double* __restrict__ part, int n, double& a, double& c) {
  __shared__ double s1[256], s2[256];
  double x = 0, y = 0;
  for (int i = (int)threadIdx.x; i < n; i += 256) {
    x += part[2 * i];
    y += part[2 * i + 1];
  }
  s1[threadIdx.x] = x;
  s2[threadIdx.x] = y;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  a = s1[0];
  c = s2[0];
}
__global__ void k_nn_sigma_fold(const double* __restrict__ part, int n, double* __restrict__ sig) {
  double a, c;
  fold_pairs(part, n, a, c);
  if (threadIdx.x != 0) return;
  const double s = (c > 0) ? sqrt(a / c) : 0.0;
  sig[0] = s;
  sig[1] = s > 0 ? 1.0 / s : 0.0;
}
void nn_sigma(const aqf::Geom& G, const uint8_t* content, const float* rhs, double* part, int nparts,
              double* sig, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_sigma_part, dim3(nparts), dim3(256), 0, s, G, content, rhs, part);
  hipLaunchKernelGGL(k_nn_sigma_fold, dim3(1), dim3(256), 0, s, part, nparts, sig);
}

__global__ void k_nn_input(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ rhs,
                           const double* __restrict__ sig, __bf16* __restrict__ x0, float* __restrict__ mask) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  const bool fl = content[gi] == aqf::FLUID;
  const float b = fl ? (float)((double)rhs[gi] * sig[1]) : 0.f;
  __bf16* o = x0 + n * 8;
  o[0] = f2bf(b);
  o[1] = f2bf(fl ? 1.f : 0.f);
#pragma unroll
  for (int c = 2; c < 8; ++c) o[c] = f2bf(0.f);
  if (mask) mask[n] = fl ? 1.f : 0.f;
}
void nn_input(const aqf::Geom& G, const uint8_t* content, const float* rhs, const double* sig,
              __bf16* x0, float* mask, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_input, dim3((G.ncells_hash + 255) / 256), dim3(256), 0, s, G, content, rhs, sig,
                     x0, mask);
}

__global__ void k_nn_target(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ p,
                            const double* __restrict__ sig, float scale, float* __restrict__ t) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  const bool fl = content[gi] == aqf::FLUID;
  t[n] = (fl && sig[0] > 0) ? (float)((double)p[gi] / (sig[0] * (double)scale)) : 0.f;
}
void nn_target(const aqf::Geom& G, const uint8_t* content, const float* p, const double* sig, float scale,
               float* t, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_target, dim3((G.ncells_hash + 255) / 256), dim3(256), 0, s, G, content, p, sig,
                     scale, t);
}

__global__ void k_nn_output(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ y,
                            const double* __restrict__ sig, float scale, float* __restrict__ p) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, yy, z;
  cell3(G, n, x, yy, z);
  const long long gi = G.g(x, yy, z);
  const bool fl = content[gi] == aqf::FLUID;
  p[gi] = fl ? (float)((double)y[n] * sig[0] * (double)scale) : 0.f;
}
void nn_output(const aqf::Geom& G, const uint8_t* content, const float* y, const double* sig, float scale,
               float* p, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_output, dim3((G.ncells_hash + 255) / 256), dim3(256), 0, s, G, content, y, sig,
                     scale, p);
}

// ------------------------------------------------------------------ warm-start guess
// The guess runs on dense fields in hash order (x-major, z-fastest). On grids
// larger than the training resolution the right-hand side is restricted 2x per
// level (sum of the eight children; a coarse cell is FLUID when at least four of
// its children are), the network runs on the coarsest level, and its pressure is
// prolonged back with cell-centred trilinear weights (3/4, 1/4 per axis). The
// fine guess p is finally scaled by alpha = <p, b> / <p, A p> (A = the pressure
// operator of the FP64 residual, symmetric positive definite), the alpha that
// minimises the energy-norm error ||p* - alpha p||_A with A p* = b: whatever the
// network's scale error, the scaled guess is never further from the solution in
// that norm than a zero guess. (Minimising the residual norm instead would weigh
// the guess's high-frequency error, which the first sweeps remove anyway, and
// shrink its useful smooth part.)
__global__ void k_nn_gather(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ rhs,
                            float* __restrict__ b, float* __restrict__ m) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  const bool fl = content[gi] == aqf::FLUID;
  b[n] = fl ? rhs[gi] : 0.f;
  m[n] = fl ? 1.f : 0.f;
}
__global__ void k_nn_restrict(int Xc, int Yc, int Zc, const float* __restrict__ bf, const float* __restrict__ mf,
                              float* __restrict__ bc, float* __restrict__ mc) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (long long)Xc * Yc * Zc) return;
  const int z = (int)(n % Zc);
  const long long t = n / Zc;
  const int y = (int)(t % Yc), x = (int)(t / Yc);
  const int Yf = 2 * Yc, Zf = 2 * Zc;
  float sb = 0.f, sm = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const long long f = ((long long)(2 * x + (i >> 2)) * Yf + (2 * y + ((i >> 1) & 1))) * Zf + 2 * z + (i & 1);
    sb += bf[f];
    sm += mf[f];
  }
  const bool fl = sm >= 4.f;
  bc[n] = fl ? sb : 0.f;
  mc[n] = fl ? 1.f : 0.f;
}
__global__ void k_nn_sigma_dense(long long V, const float* __restrict__ b, const float* __restrict__ m,
                                 double* __restrict__ part) {
  __shared__ double s1[256], s2[256];
  double a = 0, c = 0;
  for (long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x; n < V;
       n += (long long)gridDim.x * blockDim.x) {
    if (m[n] == 0.f) continue;
    const double v = (double)b[n];
    a += v * v;
    c += 1.0;
  }
  s1[threadIdx.x] = a;
  s2[threadIdx.x] = c;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      s1[threadIdx.x] += s1[threadIdx.x + o];
      s2[threadIdx.x] += s2[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}
__global__ void k_nn_input_dense(long long V, const float* __restrict__ b, const float* __restrict__ m,
                                 const double* __restrict__ sig, __bf16* __restrict__ x0) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= V) return;
  __bf16* o = x0 + n * 8;
  o[0] = f2bf((float)((double)b[n] * sig[1]));
  o[1] = f2bf(m[n]);
#pragma unroll
  for (int c = 2; c < 8; ++c) o[c] = f2bf(0.f);
}
__global__ void k_nn_output_dense(long long V, const float* __restrict__ y, const float* __restrict__ m,
                                  const double* __restrict__ sig, float scale, float* __restrict__ p) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= V) return;
  p[n] = m[n] != 0.f ? (float)((double)y[n] * sig[0] * (double)scale) : 0.f;
}
__global__ void k_nn_prolong(int Xc, int Yc, int Zc, const float* __restrict__ pc, float* __restrict__ pf) {
  const int Xf = 2 * Xc, Yf = 2 * Yc, Zf = 2 * Zc;
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (long long)Xf * Yf * Zf) return;
  const int z = (int)(n % Zf);
  const long long t = n / Zf;
  const int y = (int)(t % Yf), x = (int)(t / Yf);
  // parent and the neighbouring parent on the child's side, weights 3/4 and 1/4
  const int px = x >> 1, py = y >> 1, pz = z >> 1;
  const int qx = min(max(px + ((x & 1) ? 1 : -1), 0), Xc - 1);
  const int qy = min(max(py + ((y & 1) ? 1 : -1), 0), Yc - 1);
  const int qz = min(max(pz + ((z & 1) ? 1 : -1), 0), Zc - 1);
  const int ix[2] = {px, qx}, iy[2] = {py, qy}, iz[2] = {pz, qz};
  const float w[2] = {0.75f, 0.25f};
  float s = 0.f;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        s += w[a] * w[b] * w[c] * pc[((long long)ix[a] * Yc + iy[b]) * Zc + iz[c]];
  pf[n] = s;
}
__global__ void k_nn_scatter(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ pf,
                             float* __restrict__ p) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  p[gi] = content[gi] == aqf::FLUID ? pf[n] : 0.f;
}
// <p, b> and <p, A p> over FLUID cells, A as in the FP64 residual.
// Per block: sum of p*b and p*(A p) over FLUID cells in a grid-stride loop, four
// cells per trip whose loads (content and p at the cell and its six neighbours, b)
// are all issued before any is used; each thread adds its cells in stride order.
__global__ void k_nn_alpha_part(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ rhs,
                                const float* __restrict__ p, double* __restrict__ part) {
  __shared__ double s1[256], s2[256];
  double qb = 0, qq = 0;
  const long long stride = (long long)gridDim.x * blockDim.x;
  const long long o[6] = {G.sx, -G.sx, (long long)G.EZ, -(long long)G.EZ, 1, -1};
  for (long long n0 = (long long)blockIdx.x * blockDim.x + threadIdx.x; n0 < G.ncells_hash; n0 += 4 * stride) {
    uint8_t cc[4], cn[4][6];
    float pc[4], pn[4][6], bc[4];
    bool ok[4], in[4][6];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const long long n = n0 + k * stride;
      ok[k] = n < G.ncells_hash;
      int x, y, z;
      cell3(G, ok[k] ? n : 0, x, y, z);
      const long long gi = G.g(x, y, z);
      in[k][0] = x + 1 < G.X, in[k][1] = x > 0, in[k][2] = y + 1 < G.Y;
      in[k][3] = y > 0, in[k][4] = z + 1 < G.Z, in[k][5] = z > 0;
      cc[k] = content[gi];
      pc[k] = p[gi];
      bc[k] = rhs[gi];
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        const long long gn = in[k][j] ? gi + o[j] : gi;
        cn[k][j] = content[gn];
        pn[k][j] = p[gn];
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (!ok[k] || cc[k] != aqf::FLUID) continue;
      const double q = (double)pc[k];
      double ap = 6.0 * q;
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        if (!in[k][j])
          ap -= q;
        else if (cn[k][j] == aqf::FLUID)
          ap -= (double)pn[k][j];
      }
      qb += q * (double)bc[k];
      qq += q * ap;
    }
  }
  s1[threadIdx.x] = qb;
  s2[threadIdx.x] = qq;
  __syncthreads();
  for (int r = 128; r > 0; r >>= 1) {
    if ((int)threadIdx.x < r) {
      s1[threadIdx.x] += s1[threadIdx.x + r];
      s2[threadIdx.x] += s2[threadIdx.x + r];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = s1[0];
    part[2 * blockIdx.x + 1] = s2[0];
  }
}
__global__ void k_nn_alpha_fold(const double* __restrict__ part, int n, double* __restrict__ alpha) {
  double qb, qq;
  fold_pairs(part, n, qb, qq);
  if (threadIdx.x != 0) return;
  alpha[0] = (qq > 0 && isfinite(qb / qq)) ? qb / qq : 0.0;
}
__global__ void k_nn_alpha_apply(aqf::Geom G, const double* __restrict__ alpha, float* __restrict__ p) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  p[gi] = (float)((double)p[gi] * alpha[0]);
}

// r = b - A p over FLUID cells (FP64 arithmetic, stored FP32), 0 elsewhere.
__global__ void k_nn_residual(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ rhs,
                              const float* __restrict__ p, float* __restrict__ r) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  if (content[gi] != aqf::FLUID) {
    r[gi] = 0.f;
    return;
  }
  const double pc = (double)p[gi];
  double ap = 6.0 * pc;
  const bool in[6] = {x + 1 < G.X, x > 0, y + 1 < G.Y, y > 0, z + 1 < G.Z, z > 0};
  const long long o[6] = {G.sx, -G.sx, (long long)G.EZ, -(long long)G.EZ, 1, -1};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    if (!in[k])
      ap -= pc;
    else if (content[gi + o[k]] == aqf::FLUID)
      ap -= (double)p[gi + o[k]];
  }
  r[gi] = (float)((double)rhs[gi] - ap);
}
// p += d on FLUID cells.
__global__ void k_nn_axpy(aqf::Geom G, const uint8_t* __restrict__ content, const float* __restrict__ d,
                          float* __restrict__ p) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= G.ncells_hash) return;
  int x, y, z;
  cell3(G, n, x, y, z);
  const long long gi = G.g(x, y, z);
  if (content[gi] == aqf::FLUID) p[gi] += d[gi];
}

static inline int nblk(long long n) { return (int)((n + 255) / 256); }

void nn_residual(const aqf::Geom& G, const uint8_t* content, const float* rhs, const float* p, float* r,
                 hipStream_t s) {
  hipLaunchKernelGGL(k_nn_residual, dim3(nblk(G.ncells_hash)), dim3(256), 0, s, G, content, rhs, p, r);
}
void nn_axpy(const aqf::Geom& G, const uint8_t* content, const float* d, float* p, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_axpy, dim3(nblk(G.ncells_hash)), dim3(256), 0, s, G, content, d, p);
}

void nn_guess_gather(const aqf::Geom& G, const uint8_t* content, const float* rhs, float* b, float* m,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_nn_gather, dim3(nblk(G.ncells_hash)), dim3(256), 0, s, G, content, rhs, b, m);
}
void nn_restrict(int Xc, int Yc, int Zc, const float* bf, const float* mf, float* bc, float* mc, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_restrict, dim3(nblk((long long)Xc * Yc * Zc)), dim3(256), 0, s, Xc, Yc, Zc, bf, mf,
                     bc, mc);
}
void nn_input_dense(long long V, const float* b, const float* m, double* part, int nparts, double* sig,
                    __bf16* x0, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_sigma_dense, dim3(nparts), dim3(256), 0, s, V, b, m, part);
  hipLaunchKernelGGL(k_nn_sigma_fold, dim3(1), dim3(256), 0, s, part, nparts, sig);
  hipLaunchKernelGGL(k_nn_input_dense, dim3(nblk(V)), dim3(256), 0, s, V, b, m, sig, x0);
}
void nn_output_dense(long long V, const float* y, const float* m, const double* sig, float scale, float* p,
                     hipStream_t s) {
  hipLaunchKernelGGL(k_nn_output_dense, dim3(nblk(V)), dim3(256), 0, s, V, y, m, sig, scale, p);
}
void nn_prolong(int Xc, int Yc, int Zc, const float* pc, float* pf, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_prolong, dim3(nblk(8LL * Xc * Yc * Zc)), dim3(256), 0, s, Xc, Yc, Zc, pc, pf);
}
void nn_scatter_scaled(const aqf::Geom& G, const uint8_t* content, const float* rhs, const float* pf, float* p,
                       double* part, int nparts, double* alpha, hipStream_t s) {
  hipLaunchKernelGGL(k_nn_scatter, dim3(nblk(G.ncells_hash)), dim3(256), 0, s, G, content, pf, p);
  hipLaunchKernelGGL(k_nn_alpha_part, dim3(nparts), dim3(256), 0, s, G, content, rhs, p, part);
  hipLaunchKernelGGL(k_nn_alpha_fold, dim3(1), dim3(256), 0, s, part, nparts, alpha);
  hipLaunchKernelGGL(k_nn_alpha_apply, dim3(nblk(G.ncells_hash)), dim3(256), 0, s, G, alpha, p);
}

// Host tensor (V x 2 floats) -> network input (V x 8 bf16).
__global__ void k_host_input(long long V, const float* __restrict__ x2, __bf16* __restrict__ x0) {
  const long long n = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= V) return;
  __bf16* o = x0 + n * 8;
  o[0] = f2bf(x2[2 * n]);
  o[1] = f2bf(x2[2 * n + 1]);
#pragma unroll
  for (int c = 2; c < 8; ++c) o[c] = f2bf(0.f);
}
void host_input(long long V, const float* x2, __bf16* x0, hipStream_t s) {
  hipLaunchKernelGGL(k_host_input, dim3((unsigned)((V + 255) / 256)), dim3(256), 0, s, V, x2, x0);
}

}  // namespace aqu
