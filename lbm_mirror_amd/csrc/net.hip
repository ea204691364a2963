// Learned warm start: a convolutional encoder-decoder trained and run with
// hand-written bf16 MFMA kernels (v_mfma_f32_16x16x32_bf16), FP32 accumulate.
//
// Layout: activations NHWC bf16 (pixel-major, channels contiguous), so that
// every 3x3 tap of 8 consecutive channels is one 16-byte load.  A 3x3 same
// convolution is the GEMM  out[p][co] = sum_{tap,ci} in[p+off(tap)][ci] *
// W[tap][ci][co]  with M = pixels, N = Cout, K = 9*Cin (implicit im2col: the
// loader gathers the A tile straight from the activation).  The data
// gradient is the same GEMM on the output gradient with the weights flipped
// and transposed (Wt[8-tap][co][ci] = W[tap][ci][co]); the weight gradient is
// the GEMM dW[(tap,ci)][co] = sum_p in[p+off(tap)][ci] * dOut[p][co], split
// over pixel ranges with a fixed-order reduction of the partial tiles, so
// training is deterministic run to run.
//
// A conv block takes 8 (or 4) x 16 pixels and 16*NC output channels, NC per
// layer so that the layer's channel count is a whole number of tiles: the
// pixels and their halo in LDS, the weights as ready MFMA fragments.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "../../include/lbm_mirror_amd/lbm.h"
#include "memory.hpp"
#include "net_init.hpp"
#include "readback.hpp"

namespace lbmnet {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Round-to-nearest-even FP32 -> bf16 bits (NaN kept quiet).
__host__ __device__ inline uint16_t f2bf(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return uint16_t((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return uint16_t(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t h) { return __builtin_bit_cast(float, uint32_t(h) << 16); }

// Two of f2bf in one instruction (v_cvt_pk_bf16_f32 rounds to nearest even).
__device__ inline uint32_t f2bf2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}

struct Act {  // element (pixel q, channel c) at p[q*ld + off + c]
  uint16_t* p;
  int ld, off;
};
// An activation lies kActPad elements into its allocation, behind zeros: what
// a kernel reads for a pixel outside the image, by an offset from the same
// base as the pixels (a 32-bit offset then serves both).
constexpr int kActPad = 128;
// Byte offsets from the allocation's start fit 32 bits.
inline bool act_small(const Act& a, size_t pixels) { return (pixels * a.ld + kActPad) * 2 < (size_t(1) << 32); }

constexpr int BM = 128, BK = 32, LK = BK + 8;


struct ConvArgs {
  int B, H, W;
  int cin, cout;  // GEMM K = 9*cin, N = cout; both multiples of 8
  Act in, out;
  const uint4* w;  // weight fragments (k_wconvert)
  const float* bias;
  int bias_n;
  float* outf;  // FP32 result (ld outf_n, columns < outf_n) instead of out
  int outf_n;
  int relu;
  Act mask;  // mask.p != null: result *= (mask > 0)
};

__device__ inline uint4 load_tap(const Act& s, int H, int W, int b, int y, int x, int tap, int c) {
  const int yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
  if (yy < 0 || yy >= H || xx < 0 || xx >= W) return make_uint4(0u, 0u, 0u, 0u);
  const size_t q = (size_t(b) * H + yy) * W + xx;
  return *reinterpret_cast<const uint4*>(s.p + q * s.ld + s.off + c);
}

// 16-channel tiles per conv block for N output channels: the widest block of
// at most 160 channels that divides N (N = 8, the output layer, takes 32).  160 in
// one block read the pixels once, not twice: 64 -> 160 channels at 128 x 128 106 ->
// 82 us.
__host__ __device__ inline int conv_nc(int N) {
  const int nc[6] = {10, 8, 6, 5, 4, 2};
  for (int k = 0; k < 6; ++k)
    if (N % (16 * nc[k]) == 0) return nc[k];
  return 2;
}
// Wavefronts of a conv block that share its pixels and split its tiles.  Two halve
// what the block reads of its weights, which comes through L1 at half LDS' rate
// (with one, twice the time of the MFMAs): at 256 x 256, 32 -> 96 channels 168 -> 138
// us, at 128 x 128 160 -> 64 77 -> 65 us, at 64 x 64 256 -> 96 65 -> 53 us.  Of two tiles
// each wavefront keeps both: its 16-byte stores are worth more (8 -> 32 channels 30
// us for 32).
__host__ __device__ constexpr int conv_wn(int nc) { return nc >= 4 && nc % 2 == 0 ? 2 : 1; }
// Weight fragments of a conv GEMM: per K step of 32 and 16-channel tile, the
// 64 lanes' 16-byte MFMA operands in lane order, so a wavefront loads one as
// 1 KiB in a row.  Lane l holds k = 8 (l / 16) .. + 7 of row l % 16.
__host__ __device__ inline int conv_steps(int cin) { return (9 * cin + 31) / 32; }
__host__ __device__ inline int conv_tiles(int N) {  // padded to whole blocks
  const int nc = conv_nc(N);
  return (N + 16 * nc - 1) / (16 * nc) * nc;
}
// The channel of row r of tile t.  Tiles go in pairs whose rows interleave by
// four: lane group g of the result then holds the 8 consecutive channels
// 8g .. 8g + 7 of the pair, one 16-byte store.
__host__ __device__ inline int conv_channel(int nc, int t, int r) {
  const int blk = t / nc, i = t - blk * nc, base = blk * nc * 16;
  if ((i | 1) >= nc) return base + 16 * i + r;  // the last tile of an odd block
  return base + 32 * (i / 2) + 8 * (r / 4) + 4 * (i & 1) + (r & 3);
}

constexpr int kPatchW = 18;  // 16 pixels and the halo


// Forward convolution and data gradient: the implicit GEMM over the 3x3 taps.
// A block takes 4*MT rows of 16 pixels of one image and 16*NC output
// channels; the pixels with their halo go to LDS once, all channels (one read
// of the activation instead of one per tap, one barrier instead of one per K
// step), and the nine taps read them there, each 16-pixel operand at its own
// shift.  Pixels lie 2*cin + 16 bytes apart.  The weights come as ready
// fragments from L1/L2, so they need no LDS either.  A wavefront has RT rows of
// pixels and NW tiles (conv_wn): per K step RT operands from LDS and NW from L1 for
// RT*NW MFMAs.  The weights are the first operand: a lane's results are then 8
// consecutive channels of one pixel, stored as they are.  Batch of 16 images of
// 256 x 256, per layer, against 128-pixel tiles gathered tap by tap through two
// LDS buffers: 96 -> 32 channels 237 -> 110 us, 32 -> 32 79 -> 42 us, at 32 x 32
// 96 -> 160 and 160 -> 160 channels 33 and 46 -> 16 and 21 us.  What bounds it
// then: the many-channel layers the MFMA issue (96 -> 32: 58 GFLOP, 42 us at the
// card's matrix-product rate) and LDS reads, the few-channel ones memory; the
// input gradient of 96 channels at 256 x 256 (178 -> 138 us) the 400 MB of
// its mask and result.
// MODE 0: cin a multiple of 32 (a K step lies in one tap); 1: any cin (each
// quarter of the lanes finds its own tap); 2: as 1, with the pixels read from
// the activation (their patch would not fit LDS, or their offsets 32 bits).
template <int NC, int MT, int MODE>
__global__ __launch_bounds__(256) void k_conv(ConvArgs a) {
  extern __shared__ u32x4 patch[];
  // wavefronts along the pixel rows and along the tiles, and what each has of both
  constexpr int WN = conv_wn(NC), NW = NC / WN, RT = MT * WN;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, px = lane & 15;
  const int tx = (a.W + 15) / 16, ty = (a.H + 4 * MT - 1) / (4 * MT);
  const int bx = blockIdx.x % tx, by = blockIdx.x / tx % ty, b = blockIdx.x / (tx * ty);
  const int x0 = bx * 16, y0 = by * 4 * MT;
  const int c8 = a.cin / 8, sp = c8 + 1;  // pixel pitch in 16-byte units
  const int wm = wave / WN, wn = wave % WN;
  const int nk = conv_steps(a.cin), nt = conv_tiles(a.cout), t0 = blockIdx.y * NC + wn * NW;
  const int zat = c8;  // MODE 1: a chunk of zeros (the first pixel's padding)
  if (MODE != 2) {
    // straight to LDS, 1 KiB a wavefront and instruction, so that the whole
    // patch is in flight at once and takes no registers; a wavefront loads
    // whole patch rows, whose lanes keep their column and chunk
    const int row = kPatchW * sp;
    for (int i0 = 0; i0 < row; i0 += 64) {
      const int i = i0 + lane, x = i / sp, c = i - x * sp;
      const bool in = c < c8 && unsigned(x0 - 1 + x) < unsigned(a.W) && i < row;
      const uint32_t o = uint32_t((x * a.in.ld + c * 8) * 2);
      for (int r = wave; r < 4 * MT + 2; r += 4) {
        u32x4* to = patch + r * row + i0;
        if (in && unsigned(y0 - 1 + r) < unsigned(a.H)) {
          const auto from = (const __attribute__((address_space(1))) char*)(
              a.in.p + ((size_t(b) * a.H + (y0 - 1 + r)) * a.W + x0) * a.in.ld + a.in.off - a.in.ld);
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(from + o),
                                           (__attribute__((address_space(3))) void*)to, 16, 0, 0);
        } else if (i < row) {
          to[lane] = u32x4{0u, 0u, 0u, 0u};
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  // what the results will need of the layer's input, in flight under the MFMAs
  constexpr int NP = (NW + 1) / 2;
  const int x = x0 + px;
  auto pixel = [&](int r) { return (size_t(b) * a.H + (y0 + wm * RT + r)) * a.W + x; };
  auto inside = [&](int r) { return y0 + wm * RT + r < a.H && x < a.W; };
  // a pair's first channel in this lane
  auto channel = [&](int p) { return 16 * (t0 + 2 * p) + (2 * p + 1 < NW ? 8 : 4) * g; };
  u32x4 mk[RT][NP];
  if (a.mask.p) {
    const auto mp = (const __attribute__((address_space(1))) uint16_t*)a.mask.p + a.mask.off;
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int p = 0; p < NP; ++p) {
        const auto at = mp + (inside(r) ? pixel(r) * a.mask.ld : size_t(0)) + (channel(p) < a.cout ? channel(p) : 0);
        if (2 * p + 1 < NW) {
          mk[r][p] = *(const __attribute__((address_space(1))) u32x4*)at;
        } else {
          const auto t = *(const __attribute__((address_space(1))) u32x2*)at;
          mk[r][p] = u32x4{t.x, t.y, 0u, 0u};
        }
      }
  }
  f32x4 acc[RT][NW];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < NW; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const auto wp = (const __attribute__((address_space(1))) u32x4*)a.w + size_t(t0) * 64 + lane;
  const int base = (wm * RT * kPatchW + px) * sp + (MODE == 0 ? g : 0);
  int tap = 0, c = 0;  // MODE 0: the K step's tap and first 8-channel chunk
  auto mma = [&](const u32x4 (&w)[NW], const u32x4 (&p)[RT]) {
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int n = 0; n < NW; ++n)
        acc[r][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w[n]),
                                                            __builtin_bit_cast(bf16x8, p[r]), acc[r][n], 0, 0, 0);
  };
  if constexpr (MODE == 0) {
    // nk = 9 * cin / 32 is a multiple of 3: three K steps per turn, the
    // weights of each loaded a whole turn ahead (the last turn's loads read
    // the fragments' padding)
    u32x4 wf[3][NW];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int n = 0; n < NW; ++n) wf[d][n] = wp[(d * nt + n) * 64];
    for (int k = 0; k < nk; k += 3) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        u32x4 pf[RT];
        const int off = base + (tap / 3 * kPatchW + tap % 3) * sp + c;
#pragma unroll
        for (int r = 0; r < RT; ++r) pf[r] = patch[off + r * kPatchW * sp];
        c += 4;
        if (c == c8) {
          c = 0;
          ++tap;
        }
        mma(wf[d], pf);
#pragma unroll
        for (int n = 0; n < NW; ++n) wf[d][n] = wp[size_t((k + 3 + d) * nt + n) * 64];
      }
    }
  } else {
    for (int k = 0; k < nk; ++k) {
      u32x4 wf[NW], pf[RT];
#pragma unroll
      for (int n = 0; n < NW; ++n) wf[n] = wp[size_t(k * nt + n) * 64];
      const int o = 4 * k + g, tp = o / c8, ch = o - tp * c8;  // this lane's tap and 8-channel chunk
      const bool in = tp < 9;
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        if (MODE == 1) {
          pf[r] = patch[in ? base + (r * kPatchW + tp / 3 * kPatchW + tp % 3) * sp + ch : zat];
        } else {
          const int y = y0 + wm * RT + r, x = x0 + px;
          const uint4 v = (in && y < a.H && x < a.W) ? load_tap(a.in, a.H, a.W, b, y, x, tp, ch * 8)
                                                     : make_uint4(0u, 0u, 0u, 0u);
          pf[r] = u32x4{v.x, v.y, v.z, v.w};
        }
      }
      mma(wf, pf);
    }
  }
  // 8 channels of a pixel per lane and store
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const bool pair = 2 * p + 1 < NW;
    const int ch = channel(p);
    if (ch >= a.cout) continue;
    float bias[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) bias[j] = (a.bias && ch + j < a.bias_n && (pair || j < 4)) ? a.bias[ch + j] : 0.f;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      if (!inside(r)) continue;
      const size_t m = pixel(r);
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[j] = j < 4 ? acc[r][2 * p][j] : (pair ? acc[r][pair ? 2 * p + 1 : 2 * p][j - 4] : 0.f);
        if (a.bias) v[j] = v[j] + bias[j];
        if (a.relu) v[j] = v[j] > 0.f ? v[j] : 0.f;
      }
      if (a.outf) {  // FP32 result (the output layer)
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (ch + j < a.outf_n && (pair || j < 4)) a.outf[m * a.outf_n + ch + j] = v[j];
        continue;
      }
      u32x4 w;
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = f2bf2(v[2 * j], v[2 * j + 1]);
      if (a.mask.p) {  // zero where the layer input was not positive
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (!(bf2f(uint16_t(mk[r][p][j] & 0xffffu)) > 0.f)) w[j] &= 0xffff0000u;
          if (!(bf2f(uint16_t(mk[r][p][j] >> 16)) > 0.f)) w[j] &= 0x0000ffffu;
        }
      }
      const auto op = (__attribute__((address_space(1))) uint16_t*)a.out.p + m * a.out.ld + a.out.off + ch;
      if (pair) *(__attribute__((address_space(1))) u32x4*)op = w;
      else *(__attribute__((address_space(1))) u32x2*)op = u32x2{w[0], w[1]};
    }
  }
}

template <int NC, int MT>
hipError_t launch_conv_t(const ConvArgs& a, size_t lds, hipStream_t s) {
  const dim3 grid(a.B * ((a.H + 4 * MT - 1) / (4 * MT)) * ((a.W + 15) / 16), conv_tiles(a.cout) / NC);
  if (lds > 160 * 1024 || !act_small(a.in, size_t(a.B) * a.H * a.W)) {
    hipLaunchKernelGGL((k_conv<NC, MT, 2>), grid, dim3(256), 0, s, a);
  } else if (a.cin % 32 == 0) {
    hipLaunchKernelGGL((k_conv<NC, MT, 0>), grid, dim3(256), lds, s, a);
  } else {
    hipLaunchKernelGGL((k_conv<NC, MT, 1>), grid, dim3(256), lds, s, a);
  }
  return hipGetLastError();
}

template <int NC>
hipError_t launch_conv_n(const ConvArgs& a, hipStream_t s) {
  // Blocks of 8 x 16 pixels, unless their patch exceeds LDS or the chip has
  // more CUs than there are such blocks: 4 x 16 there (64 x 64 images of a batch
  // of 16, 160 -> 96 channels: 22 us, 19 us with the lower block).  16 x 16 pixels
  // hold twice the accumulators and a patch that leaves fewer blocks on a CU:
  // 94 us for 75 us at 128 x 128, 160 -> 64 channels.
  auto lds = [&](int mt) { return size_t(((4 * mt + 2) * kPatchW) * (a.cin / 8 + 1) + 255) / 256 * 4096; };
  auto blocks = [&](int mt) {
    return size_t(a.B) * ((a.H + 4 * mt - 1) / (4 * mt)) * ((a.W + 15) / 16) * (conv_tiles(a.cout) / NC);
  };
  if (lds(2) <= 160 * 1024 && blocks(2) >= 256) return launch_conv_t<NC, 2>(a, lds(2), s);
  return launch_conv_t<NC, 1>(a, lds(1), s);
}

hipError_t launch_conv(const ConvArgs& a, hipStream_t s) {
  switch (conv_nc(a.cout)) {
    case 10: return launch_conv_n<10>(a, s);
    case 8: return launch_conv_n<8>(a, s);
    case 6: return launch_conv_n<6>(a, s);
    case 5: return launch_conv_n<5>(a, s);
    case 4: return launch_conv_n<4>(a, s);
    default: return launch_conv_n<2>(a, s);
  }
}

// A wavefront's 32 rows of the block tile against NC 16-column blocks of the
// B tile (2 x NC MFMA 16x16x32 per K step of 32).
template <int NC>
__device__ inline void mma_tile_n(const uint16_t* As, const uint16_t* Bs, int wave, int lane,
                                  f32x4 (&acc)[2][NC]) {
  bf16x8 af[2];
#pragma unroll
  for (int r = 0; r < 2; ++r)
    af[r] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(
                                           &As[(wave * 32 + r * 16 + (lane & 15)) * LK + (lane >> 4) * 8]));
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const bf16x8 bfr = __builtin_bit_cast(
        bf16x8, *reinterpret_cast<const uint4*>(&Bs[(c * 16 + (lane & 15)) * LK + (lane >> 4) * 8]));
#pragma unroll
    for (int r = 0; r < 2; ++r) acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[r], bfr, acc[r][c], 0, 0, 0);
  }
}

// 16-column blocks per weight-gradient tile for N output channels: the widest
// tile of at most 128 channels that divides N (N = 8 takes 32)
int wgrad_nc(int N) {
  for (int nc : {8, 6, 5, 4, 2})
    if (N % (16 * nc) == 0) return nc;
  return 2;
}

struct WgradArgs {
  int B, H, W, cin, cout;  // M' = 9*cin (+ the bias row), N' = cout, K' = pixels
  Act in, dpre;
  float* partial;  // [splits][9*cin + 8][cout]
  int chunk;       // pixels per split, multiple of BK
};

// Two 8-element chunks (pixels k and k+1 of the same 8 rows) into LDS rows
// base[e*stride], as one 32-bit write per row.
__device__ inline void scatter8x2(uint16_t* base, int stride, uint4 v0, uint4 v1) {
  const uint32_t w0[4] = {v0.x, v0.y, v0.z, v0.w}, w1[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    *reinterpret_cast<uint32_t*>(base + (2 * t) * stride) = (w1[t] << 16) | (w0[t] & 0xffffu);
    *reinterpret_cast<uint32_t*>(base + (2 * t + 1) * stride) = (w1[t] & 0xffff0000u) | (w0[t] >> 16);
  }
}

// Weight gradient: per split of the pixel range, one partial 128 x 16*NC tile
// of dW[(tap,ci)][co] = sum_p in[p+off(tap)][ci] * dpre[p][co].  Row 9*cin of
// the im2col operand is 1 on every pixel, so the same GEMM yields the bias
// gradient sum_p dpre[p][co] in that row (rows 9*cin+1 .. +7 are zero).  The
// K dimension is pixels: both operands arrive channel-contiguous and are
// transposed on their way into LDS, two pixels per 32-bit write; two LDS
// buffers, the next step's tiles loaded while the current one's MFMAs run.
template <int NC>
__global__ __launch_bounds__(256) void k_wgrad(WgradArgs a) {
  constexpr int BNc = 16 * NC;
  constexpr int BCH = BNc / 8;  // 8-channel chunks of a B row block per pixel
  __shared__ __align__(16) uint16_t As[2][BM * LK];
  __shared__ __align__(16) uint16_t Bs[2][BNc * LK];
  const int M = a.B * a.H * a.W, Mw = 9 * a.cin, Mx = Mw + 8, N = a.cout, HW = a.H * a.W;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BNc, s = blockIdx.z;
  const int p0 = s * a.chunk, p1 = min(p0 + a.chunk, M);
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  // The 16 lanes of a quarter-wavefront take 16 consecutive pixel pairs of
  // one 8-row group, so their transposing 32-bit LDS writes fall in 16
  // consecutive banks (row groups a multiple of 32 banks apart would
  // otherwise collide 8 ways)
  const int g = tid >> 4;
  const int m8 = m0 + g * 8;
  const bool mv = m8 < Mw, ones = m8 == Mw;
  const int tap = mv ? m8 / a.cin : 0;
  const int ci = mv ? m8 - tap * a.cin : 0;
  const int kq = 2 * (tid & 15);  // A: pixel pair (kq, kq+1) of the K step
  const bool bt = tid < 16 * BCH;  // B: 16 pixel pairs x BCH chunks
  const int kb = 2 * (tid & 15), nc = (tid >> 4) * 8;
  uint4 ra[2], rb[2];
  // (b, y, x) of this thread's first pixel kq of the current K step, advanced
  // by BK pixels per step without divisions
  int pb_ = p0 + kq;
  int cb = pb_ / HW, cy = (pb_ - cb * HW) / a.W, cx = pb_ - cb * HW - cy * a.W;
  auto gload = [&](int pb) {
    int b = cb, y = cy, x = cx;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int q = pb + kq + j;
      ra[j] = make_uint4(0u, 0u, 0u, 0u);
      if (q < p1) {
        if (mv) ra[j] = load_tap(a.in, a.H, a.W, b, y, x, tap, ci);
        else if (ones) ra[j].x = 0x3f80u;  // bf16 1.0 in row 9*cin
      }
      if (++x == a.W) {  // the pair's second pixel
        x = 0;
        if (++y == a.H) {
          y = 0;
          ++b;
        }
      }
    }
    cx += BK;
    while (cx >= a.W) {
      cx -= a.W;
      if (++cy == a.H) {
        cy = 0;
        ++cb;
      }
    }
    if (bt) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int q = pb + kb + j, n = n0 + nc;
        rb[j] = (q < p1 && n < N) ? *reinterpret_cast<const uint4*>(a.dpre.p + size_t(q) * a.dpre.ld + a.dpre.off + n)
                                  : make_uint4(0u, 0u, 0u, 0u);
      }
    }
  };
  auto sstore = [&](int buf) {
    scatter8x2(&As[buf][(g * 8) * LK + kq], LK, ra[0], ra[1]);
    if (bt) scatter8x2(&Bs[buf][nc * LK + kb], LK, rb[0], rb[1]);
  };
  f32x4 acc[2][NC];
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[r][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nk = p1 > p0 ? (p1 - p0 + BK - 1) / BK : 0;
  if (nk > 0) {
    gload(p0);
    sstore(0);
    __syncthreads();
  }
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) gload(p0 + (kt + 1) * BK);
    mma_tile_n<NC>(As[cur], Bs[cur], wave, lane, acc);
    if (kt + 1 < nk) sstore(cur ^ 1);  // read by no wave since the last barrier
    __syncthreads();
  }
  float* out = a.partial + size_t(s) * Mx * N;
#pragma unroll
  for (int r = 0; r < 2; ++r)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int m = m0 + wave * 32 + r * 16 + (lane >> 4) * 4 + j;
        const int n = n0 + c * 16 + (lane & 15);
        if (m <= Mw && n < N) out[size_t(m) * N + n] = acc[r][c][j];
      }
}

// The same partial tiles where image rows are a multiple of 32 pixels, so that a
// K step lies in one row.  A block takes one split, the three taps of one dy,
// 32 input channels and 16*NC output channels; per K step the input's 32
// pixels with one more on either side serve the three taps.  Both operands go
// to LDS as they lie in memory (pixel by pixel, straight from the loads) and are
// transposed on the way out (ds_read_b64_tr_b16: 16 lanes read 4 pixels x 16
// channels and each gets the 4 pixels of its channel), the tiles of a pixel
// exchanged by wg_swap against bank conflicts.
// Two buffers of kWgSteps K steps: the loads of one are in flight under the
// MFMAs of the other.  At 256 x 256, batch 16, 96 -> 32 channels: 300 us by k_wgrad,
// 167 us with the loads in flight waited for before the LDS reads (the compiler's
// wait, see tr_read2) and conflicts in half of LDS' cycles, 161 us without the
// conflicts, 134 us without the wait; 128 x 128, 160 -> 64: 174, 120, 114, 87 us.
// Three buffers, or four steps to a buffer, are no faster: what bounds it now is
// the pixels' way from L2 (each read for three dy and every 32 channels).  Where a K step lies is scalar arithmetic; a load costs
// its thread an add and a select (with addresses worked out per thread and
// load, their arithmetic bound the kernel).  Of the 6 x NC result tiles a
// wavefront has 3 x NC/2.  The K steps and their pixels are k_wgrad's, so the
// partial sums are its bits.
constexpr int kWgSteps = 2;
// Four transposing LDS reads of 8 bytes a lane (two operands of 8 pixels) at byte
// addresses `at` plus OFF, or two (one operand), waited for before their results
// are used.  In assembly because the compiler, which cannot tell the buffers apart,
// waits before any LDS read for all loads to LDS that are in flight, and those of
// the next K steps are meant to be.
template <int OFF>
__device__ __forceinline__ void tr_read2(const uint32_t (&p)[2], const uint32_t (&q)[2], bf16x8& a, bf16x8& b) {
  u32x2 r0, r1, r2, r3;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %4 offset:%8\n\t"
      "ds_read_b64_tr_b16 %1, %5 offset:%8\n\t"
      "ds_read_b64_tr_b16 %2, %6 offset:%8\n\t"
      "ds_read_b64_tr_b16 %3, %7 offset:%8\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r0), "=&v"(r1), "=&v"(r2), "=&v"(r3)
      : "v"(p[0]), "v"(p[1]), "v"(q[0]), "v"(q[1]), "n"(OFF)
      : "memory");
  a = __builtin_bit_cast(bf16x8, u32x4{r0.x, r0.y, r1.x, r1.y});
  b = __builtin_bit_cast(bf16x8, u32x4{r2.x, r2.y, r3.x, r3.y});
}
template <int OFF>
__device__ __forceinline__ void tr_read1(const uint32_t (&p)[2], bf16x8& a) {
  u32x2 r0, r1;
  asm volatile(
      "ds_read_b64_tr_b16 %0, %2 offset:%4\n\t"
      "ds_read_b64_tr_b16 %1, %3 offset:%4\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(r0), "=&v"(r1)
      : "v"(p[0]), "v"(p[1]), "n"(OFF)
      : "memory");
  a = __builtin_bit_cast(bf16x8, u32x4{r0.x, r0.y, r1.x, r1.y});
}
// Operands v[0 .. N) of one K step
template <int OFF, int N>
__device__ __forceinline__ void tr_read(const uint32_t (&at)[N][2], bf16x8 (&v)[N]) {
#pragma unroll
  for (int i = 0; i + 1 < N; i += 2) tr_read2<OFF>(at[i], at[i + 1], v[i], v[i + 1]);
  if constexpr (N % 2 == 1) tr_read1<OFF>(at[N - 1], v[N - 1]);
}
// Which 32-byte tile of a pixel (of PT) stands where: tile t at t ^ wg_swap(pixel).
// A transposing read takes 32 bytes of pixels r .. r + 3 and r + 8 .. r + 11 at a
// time (half a wavefront), which then lie in all 64 banks.
template <int PT>
__device__ inline int wg_swap(int px) {
  if (PT == 8) return (px & 3) | ((px >> 3 & 1) << 2);  // pixels 256 bytes apart
  if (PT == 4) return (px >> 1 & 1) | ((px >> 3 & 1) << 1);
  return px >> 3 & 1;
}
template <int NC>
__global__ __launch_bounds__(256) void k_wgrad32(WgradArgs a, int splits) {
  constexpr int PT = (NC + 1) / 2 * 2;           // 16-channel tiles (32 bytes) of a pixel in LDS
  constexpr int PA = 4, PB = 2 * PT;              // the same in 16-byte chunks
  constexpr int CA = 34 * PA, CS = CA + 32 * PB;  // chunks of a K step: of the input, of both
  constexpr int NT = (CS + 255) / 256, NH = (NC + 1) / 2;
  __shared__ u32x4 buf[2][kWgSteps][CS];
  const int M = a.B * a.H * a.W, N = a.cout, Mx = 9 * a.cin + 8;
  // the blocks of a split read the same pixels: all of them on one XCD (blocks
  // go round the 8 XCDs in turn), whose L2 then reads them once
  const int cblocks = (a.cin + 31) / 32, per = 3 * cblocks * ((N + 16 * NC - 1) / (16 * NC));
  const int turn = blockIdx.x / 8, s = turn / per * 8 + int(blockIdx.x) % 8, part = turn % per;
  if (s >= splits) return;  // (the splits rounded up to the XCDs)
  const int dy = part % 3, c0 = part / 3 % cblocks * 32, n0 = part / 3 / cblocks * 16 * NC;
  const int p0 = s * a.chunk, p1 = min(p0 + a.chunk, M), nk = p1 > p0 ? (p1 - p0 + 31) / 32 : 0;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, g = lane >> 4, j = lane & 15;
  // This thread's chunks of a K step: byte offset in the first step from the
  // allocation's start, and the cases in which there is nothing to load (a
  // zero is then read): never mind the step (channels beyond the layer's,
  // padding of the pitch), the row above or below the image, the pixel left or
  // right of it.
  constexpr uint32_t kNever = 1, kRow = 2, kLeft = 4, kRight = 8;
  using GC = const __attribute__((address_space(1))) char;
  uint32_t off[NT], gone[NT], adv[NT];
  bool is_a[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int i = tid + 256 * t;
    is_a[t] = i < CA;
    const int px = is_a[t] ? i / PA : (i - CA) / PB, at_ = is_a[t] ? i - px * PA : i - CA - px * PB;
    const int ch = at_ ^ (2 * (is_a[t] ? wg_swap<2>(px) : wg_swap<PT>(px)));  // (its tile, exchanged)
    const int c = (is_a[t] ? c0 : n0) + ch * 8;
    const bool ok = i < CS && ch < (is_a[t] ? 4 : 2 * NC) && c < (is_a[t] ? a.cin : N);
    gone[t] = !ok ? kNever : (!is_a[t] ? 0u : kRow | (px == 0 ? kLeft : 0u) | (px == 33 ? kRight : 0u));
    const int ld = is_a[t] ? a.in.ld : a.dpre.ld;
    const long long at = p0 + px + (is_a[t] ? (long long)(dy - 1) * a.W - 1 : 0ll);
    off[t] = uint32_t((at * ld + (is_a[t] ? a.in.off : a.dpre.off) + c + kActPad) * 2);
    adv[t] = 64u * uint32_t(ld);
  }
  GC* in0 = (GC*)(a.in.p - kActPad);
  GC* dp0 = (GC*)(a.dpre.p - kActPad);
  int x = p0 % a.W, y = p0 / a.W % a.H, left = nk;  // the next K step to load, and how many there are
  auto load = [&](int b) {
#pragma unroll
    for (int ks = 0; ks < kWgSteps; ++ks) {
      if (left-- <= 0) break;
      const uint32_t now = kNever | (unsigned(y + dy - 1) < unsigned(a.H) ? 0u : kRow) | (x == 0 ? kLeft : 0u) |
                           (x + 32 == a.W ? kRight : 0u);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t o = (gone[t] & now) ? 0u : off[t];
        if (256 * (t + 1) <= CS || tid + 256 * t < CS)
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)((is_a[t] ? in0 : dp0) + o),
                                           (__attribute__((address_space(3))) void*)(&buf[b][ks][256 * t + wave * 64]),
                                           16, 0, 0);
        off[t] += adv[t];
      }
      x += 32;
      if (x == a.W) {
        x = 0;
        if (++y == a.H) y = 0;
      }
    }
  };
  const int wm = wave & 1, wn = wave >> 1;
  // where the lane finds the first and the second four of an operand's 8 pixels:
  // byte addresses in the first buffer, of the input's tiles, then dpre's
  uint32_t at[3 + NH][2];
  const uint32_t lds0 = uint32_t(uintptr_t((__attribute__((address_space(3))) char*)&buf[0][0][0]));
#pragma unroll
  for (int e = 0; e < 2; ++e) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int tile = wm * 3 + i, r = 8 * g + (j >> 2) + tile / 2 + 4 * e;  // tap dx = tile / 2, channels 16 (tile % 2) ..
      at[i][e] = lds0 + r * PA * 16 + ((tile & 1) ^ wg_swap<2>(r)) * 32 + (j & 3) * 8;
    }
#pragma unroll
    for (int n = 0; n < NH; ++n) {
      const int r = 8 * g + (j >> 2) + 4 * e;
      at[3 + n][e] = lds0 + CA * 16 + r * PB * 16 + ((wn * NH + n) ^ wg_swap<PT>(r)) * 32 + (j & 3) * 8;
    }
  }
  const bool bias = dy == 1 && c0 == 0 && wm == 1;  // row 9*cin: ones against dpre
  f32x4 acc[3][NH], accb[NH];
#pragma unroll
  for (int n = 0; n < NH; ++n) {
    accb[n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 3; ++i) acc[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const uint32_t one = j == 0 ? 0x3f803f80u : 0u;
  const bf16x8 ones = __builtin_bit_cast(bf16x8, u32x4{one, one, one, one});
  if (nk > 0) load(0);
  for (int k0 = 0; k0 < nk; k0 += kWgSteps) {
    const int b = (k0 / kWgSteps) & 1;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // this buffer has arrived; no wave reads the other one any more
    if (k0 + kWgSteps < nk) load(b ^ 1);
    uint32_t now[3 + NH][2];
#pragma unroll
    for (int i = 0; i < 3 + NH; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) now[i][e] = at[i][e] + (b ? kWgSteps * CS * 16 : 0);
    auto k_step = [&](const bf16x8 (&v)[3 + NH]) {
#pragma unroll
      for (int n = 0; n < NH; ++n) {
        if (wn * NH + n >= NC) continue;
#pragma unroll
        for (int i = 0; i < 3; ++i) acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[3 + n], v[i], acc[i][n], 0, 0, 0);
        if (bias) accb[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[3 + n], ones, accb[n], 0, 0, 0);
      }
    };
    bf16x8 v[3 + NH];
    tr_read<0>(now, v);
    k_step(v);
    if (k0 + 1 < nk) {
      tr_read<CS * 16>(now, v);
      k_step(v);
    }
  }
  float* out = a.partial + size_t(s) * Mx * N;
#pragma unroll
  for (int n = 0; n < NH; ++n) {
    const int col = n0 + (wn * NH + n) * 16 + g * 4;
    if (wn * NH + n >= NC || col >= N) continue;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int tile = wm * 3 + i, c = c0 + (tile & 1) * 16 + j;
      if (c < a.cin)
        *reinterpret_cast<f32x4*>(out + size_t((dy * 3 + tile / 2) * a.cin + c) * N + col) = acc[i][n];
    }
    if (bias && j == 0) *reinterpret_cast<f32x4*>(out + size_t(9 * a.cin) * N + col) = accb[n];
  }
}

template <int NC>
hipError_t launch_wgrad_n(const WgradArgs& a, int splits, hipStream_t s) {
  const int cols = (a.cout + 16 * NC - 1) / (16 * NC);
  const size_t px = size_t(a.B) * a.H * a.W;
  // Fewer channels than its 32 leave k_wgrad32's tiles mostly empty: 49 us for 41
  // at 256 x 256 from 8 channels.  From 32 on it is the faster one there (96 -> 32
  // channels 300 -> 134 us, 32 -> 32 128 -> 63 us, 32 -> 3 110 -> 45 us) and down to
  // rows of one K step (160 channels at 32 x 32: 27 -> 19 us).
  if (a.cin > 16 && a.W % 32 == 0 && act_small(a.in, px) && act_small(a.dpre, px))
    hipLaunchKernelGGL(k_wgrad32<NC>, dim3((splits + 7) / 8 * 8 * 3 * ((a.cin + 31) / 32) * cols), dim3(256), 0, s, a,
                       splits);
  else
    hipLaunchKernelGGL(k_wgrad<NC>, dim3((9 * a.cin + 8 + BM - 1) / BM, cols, splits), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_wgrad(const WgradArgs& a, int splits, hipStream_t s) {
  switch (wgrad_nc(a.cout)) {
    case 8: return launch_wgrad_n<8>(a, splits, s);
    case 6: return launch_wgrad_n<6>(a, splits, s);
    case 5: return launch_wgrad_n<5>(a, splits, s);
    case 4: return launch_wgrad_n<4>(a, splits, s);
    default: return launch_wgrad_n<2>(a, splits, s);
  }
}

// grad[m*cr + n] = sum_s partial[s][m][n] for m <= 9*cin, n < cr (the
// unpadded Cout); row 9*cin is the bias, which follows the weights in the
// flat parameter layout.  A block takes 64 consecutive outputs: four groups
// of 64 threads add the splits k = g, g+4, ..., then the four sums are added
// in group order (a fixed order: training repeats bit for bit).  One launch for
// all layers, each with partial tiles of its own: a layer alone has 14 to 900
// blocks whose threads add up to 256 values one after the other, 113 us a step
// in twelve launches, 72 us in one.
struct WredLayer {
  const float* partial;
  float* grad;
  int splits, Mw, cpad, cr;
  unsigned end;  // of this layer's blocks
};
struct WredArgs {
  WredLayer layer[12];
};
__global__ __launch_bounds__(256) void k_wreduce(WredArgs a) {
  __shared__ float part[4][64];
  int q = 0;
  while (blockIdx.x >= a.layer[q].end) ++q;
  const WredLayer& L = a.layer[q];
  const int gq = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int i = int(blockIdx.x - (q > 0 ? a.layer[q - 1].end : 0u)) * 64 + l;
  const bool ok = i < (L.Mw + 1) * L.cr;
  const int m = ok ? i / L.cr : 0, n = ok ? i - m * L.cr : 0;
  // four running sums per thread (splits gq + 4(4i + u), u = 0..3) keep
  // four loads in flight; combined in a fixed order
  float su[4] = {0.f, 0.f, 0.f, 0.f};
  if (ok) {
    const size_t stride = size_t(L.Mw + 8) * L.cpad;
    const float* src = L.partial + size_t(m) * L.cpad + n;
    int k = gq;
    for (; k + 12 < L.splits; k += 16) {
#pragma unroll
      for (int u = 0; u < 4; ++u) su[u] += src[size_t(k + 4 * u) * stride];
    }
    for (int u = 0; k < L.splits; k += 4, ++u) su[u] += src[size_t(k) * stride];
  }
  part[gq][l] = (su[0] + su[1]) + (su[2] + su[3]);
  __syncthreads();
  if (gq == 0 && ok) L.grad[i] = ((part[0][l] + part[1][l]) + part[2][l]) + part[3][l];
}

// 8 channels (16 bytes, 16-byte aligned: channel offsets and row pitches are
// multiples of 8) as one vector access
__device__ inline void ld8(const uint16_t* p, float (&f)[8]) {
  const uint4 v = *reinterpret_cast<const uint4*>(p);
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    f[2 * t] = bf2f(uint16_t(w[t] & 0xffffu));
    f[2 * t + 1] = bf2f(uint16_t(w[t] >> 16));
  }
}
__device__ inline void st8(uint16_t* p, const float (&f)[8]) {
  uint32_t w[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) w[t] = f2bf2(f[2 * t], f[2 * t + 1]);
  *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

// 2x2 average pool of C channels: fine (H x W) -> coarse (H/2 x W/2).
__global__ void k_pool_fwd(Act src, Act dst, int B, int H, int W, int C) {
  const int C8 = C / 8, h = H / 2, w = W / 2;
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(B) * h * w * C8) return;
  const int c = int(i % C8) * 8;
  const size_t q = i / C8;
  const int x = int(q % w), y = int((q / w) % h), b = int(q / (size_t(w) * h));
  const size_t f00 = (size_t(b) * H + 2 * y) * W + 2 * x;
  const uint16_t* p00 = src.p + f00 * src.ld + src.off + c;
  const uint16_t* p01 = p00 + src.ld;
  const uint16_t* p10 = p00 + size_t(W) * src.ld;
  const uint16_t* p11 = p10 + src.ld;
  float a00[8], a01[8], a10[8], a11[8], o[8];
  ld8(p00, a00);
  ld8(p01, a01);
  ld8(p10, a10);
  ld8(p11, a11);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (((a00[e] + a01[e]) + a10[e]) + a11[e]) * 0.25f;
  st8(dst.p + q * dst.ld + dst.off + c, o);
}

// Pool backward into the skip gradient: g[p] = g[p] + (act[p] > 0 ? dpool[parent]/4 : 0).
__global__ void k_pool_bwd(Act dpool, Act gskip, Act act, int B, int H, int W, int C) {
  const int C8 = C / 8;
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(B) * H * W * C8) return;
  const int c = int(i % C8) * 8;
  const size_t p = i / C8;
  const int x = int(p % W), y = int((p / W) % H), b = int(p / (size_t(W) * H));
  const size_t par = (size_t(b) * (H / 2) + y / 2) * (W / 2) + x / 2;
  uint16_t* gp = gskip.p + p * gskip.ld + gskip.off + c;
  float g[8], v[8], d[8];
  ld8(gp, g);
  ld8(act.p + p * act.ld + act.off + c, v);
  ld8(dpool.p + par * dpool.ld + dpool.off + c, d);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float add = v[e] > 0.f ? d[e] * 0.25f : 0.f;
    g[e] = g[e] + add;
  }
  st8(gp, g);
}

// Nearest 2x upsample: dst fine pixel p = src coarse parent(p).
__global__ void k_up_fwd(Act src, Act dst, int B, int H, int W, int C) {
  const int C8 = C / 8;
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(B) * H * W * C8) return;
  const int c = int(i % C8) * 8;
  const size_t p = i / C8;
  const int x = int(p % W), y = int((p / W) % H), b = int(p / (size_t(W) * H));
  const size_t par = (size_t(b) * (H / 2) + y / 2) * (W / 2) + x / 2;
  *reinterpret_cast<uint4*>(dst.p + p * dst.ld + dst.off + c) =
      *reinterpret_cast<const uint4*>(src.p + par * src.ld + src.off + c);
}

// Upsample backward: coarse gradient = ((g00 + g01) + g10) + g11 of its four children.
__global__ void k_up_bwd(Act gfine, Act gcoarse, int B, int H, int W, int C) {
  const int C8 = C / 8, h = H / 2, w = W / 2;
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= size_t(B) * h * w * C8) return;
  const int c = int(i % C8) * 8;
  const size_t q = i / C8;
  const int x = int(q % w), y = int((q / w) % h), b = int(q / (size_t(w) * h));
  const size_t f00 = (size_t(b) * H + 2 * y) * W + 2 * x;
  const uint16_t* p00 = gfine.p + f00 * gfine.ld + gfine.off + c;
  const uint16_t* p01 = p00 + gfine.ld;
  const uint16_t* p10 = p00 + size_t(W) * gfine.ld;
  const uint16_t* p11 = p10 + gfine.ld;
  float a00[8], a01[8], a10[8], a11[8], o[8];
  ld8(p00, a00);
  ld8(p01, a01);
  ld8(p10, a10);
  ld8(p11, a11);
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = ((a00[e] + a01[e]) + a10[e]) + a11[e];
  st8(gcoarse.p + q * gcoarse.ld + gcoarse.off + c, o);
}

// Masked MSE over 3 output channels: gy[q][c] = bf16(2 (y - t) / (3 nf)) on
// counted pixels (channels 3..7 zero), per-block partial sums of (y - t)^2.
__global__ void k_loss(const float* y, const float* t, const uint8_t* m, int M, float inv3nf, uint16_t* gy,
                       double* partial) {
  __shared__ double red[256];
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (q < M) {
    uint16_t g[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (m[q]) {
      for (int c = 0; c < 3; ++c) {
        const float d = y[size_t(q) * 3 + c] - t[size_t(q) * 3 + c];
        s += double(d) * double(d);
        g[c] = f2bf(2.f * d * inv3nf);
      }
    }
    uint4 v;
    v.x = g[0] | (uint32_t(g[1]) << 16);
    v.y = g[2] | (uint32_t(g[3]) << 16);
    v.z = g[4] | (uint32_t(g[5]) << 16);
    v.w = g[6] | (uint32_t(g[7]) << 16);
    *reinterpret_cast<uint4*>(gy + size_t(q) * 8) = v;
  }
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (int(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_loss_reduce(const double* partial, int n, double scale, double* loss_out, float* loss_f) {
  __shared__ double red[256];
  double s = 0.0;
  for (int i = threadIdx.x; i < n; i += 256) s += partial[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int k = 128; k > 0; k >>= 1) {
    if (int(threadIdx.x) < k) red[threadIdx.x] += red[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (loss_out) *loss_out = red[0] * scale;
    if (loss_f) *loss_f = float(red[0] * scale);
  }
}

__global__ void k_adam(float* w, const float* g, float* m1, float* m2, size_t n, float lr, float b1, float b2,
                       float c1, float c2, float eps) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float a = b1 * m1[i] + (1.f - b1) * gi;
  const float b = b2 * m2[i] + (1.f - b2) * gi * gi;
  m1[i] = a;
  m2[i] = b;
  w[i] = w[i] - lr * (a / c1) / (sqrtf(b / c2) + eps);
}

// FP32 master [9][cin][cr] -> the bf16 weight fragments of the conv GEMMs:
// forward (K = taps x cin, N = cpad) and data gradient (taps flipped, K = taps
// x cpad, N = cin).  One launch for all layers.
struct WconvLayer {
  const float* wm;
  uint16_t *wb, *wt;
  int cin, cr, cpad;
  size_t end;  // in 16-byte units: of this layer's elements in the launch
};
struct WconvArgs {
  WconvLayer layer[12];
};
__host__ __device__ inline size_t conv_elements(int cin, int N) {
  return size_t(conv_steps(cin)) * conv_tiles(N) * 512;
}
__global__ void k_wconvert(WconvArgs a) {
  // a thread writes a lane's 16 bytes: one tap's 8 channels in a row, while 16
  // lanes read neighbouring floats (one element a thread: 18 us a step, not 9)
  const size_t step = size_t(gridDim.x) * 256;
  for (size_t i = size_t(blockIdx.x) * 256 + threadIdx.x; i < a.layer[11].end; i += step) {
    int k = 0;
    while (i >= a.layer[k].end) ++k;
    const WconvLayer& L = a.layer[k];
    size_t e = i - (k > 0 ? a.layer[k - 1].end : 0);
    const size_t nf = conv_elements(L.cin, L.cpad) / 8;
    const bool fwd = e < nf;
    if (!fwd) e -= nf;
    const int ci = fwd ? L.cin : L.cpad, N = fwd ? L.cpad : L.cin, nt = conv_tiles(N);
    const int lane = int(e & 63), frag = int(e >> 6), t = frag % nt;
    const int kk = frag / nt * 32 + (lane >> 4) * 8, tap = kk / ci, c = kk - tap * ci;
    const int n = conv_channel(conv_nc(N) / conv_wn(conv_nc(N)), t, lane & 15);
    uint32_t v[4] = {0u, 0u, 0u, 0u};
    if (tap < 9 && n < N) {
      const float* wm = L.wm + size_t(fwd ? tap : 8 - tap) * L.cin * L.cr;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int in = fwd ? c + j : n, out = fwd ? n : c + j;
        if (out < L.cr) v[j / 2] |= uint32_t(f2bf(wm[size_t(in) * L.cr + out])) << (j & 1 ? 16 : 0);
      }
    }
    reinterpret_cast<uint4*>(fwd ? L.wb : L.wt)[e] = make_uint4(v[0], v[1], v[2], v[3]);
  }
}

// In-place standardisation of stored targets: t = (t - mu) / sd.
__global__ void k_standardize(float* t, size_t n, float m0, float m1, float m2, float s0, float s1, float s2) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int c = int(i % 3);
  const float m = c == 0 ? m0 : (c == 1 ? m1 : m2);
  const float sd = c == 0 ? s0 : (c == 1 ? s1 : s2);
  t[i] = (t[i] - m) / sd;
}

// Network input from the lattices' flags and the words of upload_features: 16
// bytes a pixel.  (Laid out by the host this was 16 of the 20 ms of 16
// predictions of 256 x 256.)
__global__ void k_features(const uint8_t* flags, const uint32_t* tab, int B, int H, int W, uint16_t* x) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x, HW = uint32_t(H) * uint32_t(W);
  if (i >= B * HW) return;
  const uint32_t b = i / HW, r = i - b * HW, py = r / uint32_t(W), px = r - py * uint32_t(W);
  const uint32_t* per = tab + H + W + size_t(b) * (W + 1);
  const uint32_t row = tab[py], col = tab[H + px], own = per[0], at = per[1 + px];
  const uint32_t open = flags[i] >= 2 ? 0x3f80u : 0u;
  // channels 0 .. 7: open, speed | tau, profile | x, y | pressure, blockage
  reinterpret_cast<uint4*>(x)[i] =
      make_uint4(open | (own << 16), (own >> 16) | (row << 16), (col & 0xffffu) | (row & 0xffff0000u), at);
}

// Minibatch assembly from the on-device training set.
__global__ void k_gather(const uint16_t* xs, const float* ts, const uint8_t* ms, const uint32_t* idx, int B, int HW,
                         uint16_t* x, float* t, uint8_t* m) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;  // (the batch's pixels fit an int)
  if (i >= uint32_t(B) * uint32_t(HW)) return;
  const uint32_t b = i / uint32_t(HW), p = i - b * uint32_t(HW);
  const size_t src = size_t(idx[b]) * HW + p;
  *reinterpret_cast<uint4*>(x + size_t(i) * 8) = *reinterpret_cast<const uint4*>(xs + src * 8);
  t[size_t(i) * 3 + 0] = ts[src * 3 + 0];
  t[size_t(i) * 3 + 1] = ts[src * 3 + 1];
  t[size_t(i) * 3 + 2] = ts[src * 3 + 2];
  m[i] = ms[src];
}

}  // namespace lbmnet

using namespace lbmnet;

// defined with the rest of the C ABI (lbm_last_error reads it)
lbm_status lbmx_report(lbm_status s, const char* msg);

namespace {

lbm_status nfail(lbm_status s, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  return lbmx_report(s, buf);
}

#define NET_TRY(expr)                                                                  \
  do {                                                                                 \
    hipError_t e_ = (expr);                                                            \
    if (e_ != hipSuccess)                                                              \
      return nfail(e_ == hipErrorOutOfMemory ? LBM_ERR_OUT_OF_MEMORY : LBM_ERR_CRITICAL, \
                   "%s: %s", #expr, hipGetErrorString(e_));                            \
  } while (0)

// Density target: (rho - 1) / (3 u_max^2), the pressure p = (rho - 1)/3 in
// units of the inlet dynamic pressure u_max^2: O(1) from creeping to
// inertial flow.
double rho_unit(double u_max) { return 3.0 * u_max * u_max; }

struct Layer {
  int cin, cr, cpad;  // input channels, output channels (real / padded to 8)
  size_t w_off, b_off;
  uint16_t *wb = nullptr, *wt = nullptr;
  int relu;
  int level;
};

}  // namespace

struct lbm_net {
  lbm_net_config cfg;
  int device = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  bool timed = false;
  std::vector<Layer> layers;
  size_t nparam = 0;
  float *w = nullptr, *g = nullptr, *m1 = nullptr, *m2 = nullptr;
  uint64_t adam_t = 0;
  // activations (batch capacity B), level l has B*(H>>l)*(W>>l) pixels
  uint16_t* x = nullptr;
  uint16_t *a[4] = {}, *cat[3] = {}, *pool[4] = {}, *dec[3] = {}, *bott = nullptr;
  uint16_t *ga[4] = {}, *gcat[3] = {}, *gpool[4] = {}, *gdec[3] = {}, *gbott = nullptr, *gy = nullptr;
  float *y = nullptr, *t = nullptr;
  uint8_t* msk = nullptr;
  uint32_t* ftab = nullptr;  // upload_features' words
  // partial weight-gradient tiles: of all layers, or of as many at a time as the
  // memory there was holds; those that are not yet added up (reduce_gradients)
  float* partial = nullptr;
  size_t partial_n = 0, partial_used = 0;
  struct {
    int layer, splits;
    size_t at;
  } pending[12];
  int npending = 0;
  double* lpartial = nullptr;
  double* dloss = nullptr;
  float* dlosses = nullptr;
  uint32_t dlosses_n = 0;
  uint32_t* didx = nullptr;
  size_t didx_n = 0;
  // training set
  uint16_t* xs = nullptr;
  float* ts = nullptr;
  uint8_t* ms = nullptr;
  std::vector<double> nf;  // counted pixels per sample
  // output standardisation: the network predicts (target - mu) / sd per
  // channel; mu, sd come from the training set at the first training call
  double tsum[3] = {0, 0, 0}, tsq[3] = {0, 0, 0}, tcnt = 0;
  bool frozen = false;
  float mu[3] = {0.f, 0.f, 0.f}, sd[3] = {1.f, 1.f, 1.f};
};

namespace {

int W_(const lbm_net* n, int l) { return n->cfg.width >> l; }
int H_(const lbm_net* n, int l) { return n->cfg.height >> l; }

size_t level_pixels(const lbm_net* n, int l) { return size_t(n->cfg.batch) * H_(n, l) * W_(n, l); }

#define NS(expr)                  \
  do {                            \
    lbm_status s_ = (expr);       \
    if (s_ != LBM_OK) return s_;  \
  } while (0)

template <class T>
lbm_status dalloc(T** p, size_t count) {
  *p = nullptr;
  if (count == 0) return LBM_OK;
  NET_TRY(lbmx::device_alloc(p, count * sizeof(T)));
  // done when this returns: the network's stream does not wait for the null
  // stream's work, and a copy queued there could be cleared after it
  NET_TRY(hipMemset(*p, 0, count * sizeof(T)));
  NET_TRY(hipStreamSynchronize(nullptr));
  return LBM_OK;
}

lbm_status aalloc(uint16_t** p, size_t count) {
  const lbm_status s = dalloc(p, count + kActPad);
  if (s != LBM_OK) return s;
  *p += kActPad;
  return LBM_OK;
}
void afree(uint16_t* p) {
  if (p) (void)hipFree(p - kActPad);
}

void build_layers(lbm_net* n) {
  const int* w = n->cfg.widths;
  struct Spec {
    int cin, cout, relu, level;
  };
  const Spec spec[12] = {{8, w[0], 1, 0},        {w[0], w[0], 1, 0},        {w[0], w[1], 1, 1},
                         {w[1], w[1], 1, 1},     {w[1], w[2], 1, 2},        {w[2], w[2], 1, 2},
                         {w[2], w[3], 1, 3},     {w[3], w[3], 1, 3},        {w[3] + w[2], w[2], 1, 2},
                         {w[2] + w[1], w[1], 1, 1}, {w[1] + w[0], w[0], 1, 0}, {w[0], 3, 0, 0}};
  size_t off = 0;
  n->layers.clear();
  for (const Spec& s : spec) {
    Layer L;
    L.cin = s.cin;
    L.cr = s.cout;
    L.cpad = (s.cout + 7) / 8 * 8;
    L.relu = s.relu;
    L.level = s.level;
    L.w_off = off;
    off += size_t(9) * s.cin * s.cout;
    L.b_off = off;
    off += s.cout;
    n->layers.push_back(L);
  }
  n->nparam = off;
}

Act act(uint16_t* p, int ld, int off = 0) { return Act{p, ld, off}; }

// Splits of the pixel range for a weight-gradient launch of layer L: about
// kWgradBlocks blocks (tiles x splits), at least 256 pixels per split.
#ifndef LBMNET_WGRAD_BLOCKS
#define LBMNET_WGRAD_BLOCKS 1024
#endif
constexpr int kWgradBlocks = LBMNET_WGRAD_BLOCKS;
int wgrad_most_splits(const Layer& L, int M) {  // no fewer pixels have more
  const int bn = 16 * wgrad_nc(L.cpad);
  const int tiles = ((9 * L.cin + 8 + BM - 1) / BM) * ((L.cpad + bn - 1) / bn);
  return std::max(1, std::min(kWgradBlocks / std::max(1, tiles), (M + 255) / 256));
}
size_t wgrad_tile(const Layer& L) { return size_t(9 * L.cin + 8) * L.cpad; }  // floats of a split
void wgrad_shape(const lbm_net* n, const Layer& L, int B, int& splits, int& chunk) {
  const int M = B * H_(n, L.level) * W_(n, L.level);
  splits = wgrad_most_splits(L, M);
  chunk = ((M + splits - 1) / splits + BK - 1) / BK * BK;
  splits = (M + chunk - 1) / chunk;
}

lbm_status conv(lbm_net* n, int li, int B, Act in, Act out, float* outf) {
  const Layer& L = n->layers[li];
  ConvArgs a{};
  a.B = B;
  a.H = H_(n, L.level);
  a.W = W_(n, L.level);
  a.cin = L.cin;
  a.cout = L.cpad;
  a.in = in;
  a.out = out;
  a.w = reinterpret_cast<const uint4*>(L.wb);
  a.bias = n->w + L.b_off;
  a.bias_n = L.cr;
  a.outf = outf;
  a.outf_n = L.cr;
  a.relu = L.relu;
  a.mask = Act{nullptr, 0, 0};
  NET_TRY(launch_conv(a, n->stream));
  return LBM_OK;
}

// The weight and bias gradients of the layers whose partial tiles wait, into n->g.
lbm_status reduce_gradients(lbm_net* n) {
  if (n->npending == 0) return LBM_OK;
  WredArgs a{};
  unsigned end = 0;
  for (int k = 0; k < n->npending; ++k) {
    // the first layers first: their many splits take the longest to add up (12 us
    // a step less than with them last)
    const auto& p = n->pending[n->npending - 1 - k];
    const Layer& L = n->layers[p.layer];
    end += unsigned(((9 * L.cin + 1) * L.cr + 63) / 64);
    a.layer[k] = WredLayer{n->partial + p.at, n->g + L.w_off, p.splits, 9 * L.cin, L.cpad, L.cr, end};
  }
  n->npending = 0;
  n->partial_used = 0;
  hipLaunchKernelGGL(k_wreduce, dim3(end), dim3(256), 0, n->stream, a);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}

// Memory for the partial tiles: of every layer (256 x 256, batch 16, widths 32 to
// 160: 331 MiB), so that one launch adds them all up; where there is not that much,
// of the largest layer (47 MiB).  Every element that is read is written first.
lbm_status need_partial(lbm_net* n) {
  if (n->partial) return LBM_OK;
  size_t all = 0, most = 0;
  for (const Layer& L : n->layers) {
    const size_t k = size_t(wgrad_most_splits(L, int(level_pixels(n, L.level)))) * wgrad_tile(L);
    all += k;
    most = std::max(most, k);
  }
  n->partial_n = all;
  if (hipMalloc(reinterpret_cast<void**>(&n->partial), all * sizeof(float)) == hipSuccess) return LBM_OK;
  (void)hipGetLastError();
  n->partial = nullptr;
  n->partial_n = most;
  NET_TRY(lbmx::device_alloc(&n->partial, most * sizeof(float)));
  return LBM_OK;
}

// Backward of layer li given its pre-activation gradient dpre: the partial
// tiles of its weight and bias gradients, behind those that wait where they
// fit, and (if dx.p) the input gradient, masked by (in > 0) when mask_in.
lbm_status conv_bwd(lbm_net* n, int li, int B, Act in, Act dpre, Act dx, bool mask_in) {
  const Layer& L = n->layers[li];
  const int H = H_(n, L.level), W = W_(n, L.level);
  int splits, chunk;
  wgrad_shape(n, L, B, splits, chunk);
  const size_t size = size_t(splits) * wgrad_tile(L);
  if (n->partial_used + size > n->partial_n) NS(reduce_gradients(n));
  WgradArgs wa{B, H, W, L.cin, L.cpad, in, dpre, n->partial + n->partial_used, chunk};
  NET_TRY(launch_wgrad(wa, splits, n->stream));
  n->pending[n->npending++] = {li, splits, n->partial_used};
  n->partial_used += size;
  if (dx.p) {
    ConvArgs a{};
    a.B = B;
    a.H = H;
    a.W = W;
    a.cin = L.cpad;
    a.cout = L.cin;
    a.in = dpre;
    a.out = dx;
    a.w = reinterpret_cast<const uint4*>(L.wt);
    a.bias = nullptr;
    a.bias_n = 0;
    a.outf = nullptr;
    a.relu = 0;
    a.mask = mask_in ? in : Act{nullptr, 0, 0};
    NET_TRY(launch_conv(a, n->stream));
  }
  return LBM_OK;
}

unsigned blocks_for(size_t n, unsigned bs = 256) { return unsigned((n + bs - 1) / bs); }

lbm_status pool_fwd(lbm_net* n, int level, int B, Act src, Act dst, int C) {
  const int H = H_(n, level), W = W_(n, level);
  hipLaunchKernelGGL(k_pool_fwd, dim3(blocks_for(size_t(B) * (H / 2) * (W / 2) * (C / 8))), dim3(256), 0, n->stream,
                     src, dst, B, H, W, C);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}
lbm_status pool_bwd(lbm_net* n, int level, int B, Act dpool, Act gskip, Act actv, int C) {
  const int H = H_(n, level), W = W_(n, level);
  hipLaunchKernelGGL(k_pool_bwd, dim3(blocks_for(size_t(B) * H * W * (C / 8))), dim3(256), 0, n->stream, dpool, gskip,
                     actv, B, H, W, C);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}
lbm_status up_fwd(lbm_net* n, int level, int B, Act src, Act dst, int C) {
  const int H = H_(n, level), W = W_(n, level);
  hipLaunchKernelGGL(k_up_fwd, dim3(blocks_for(size_t(B) * H * W * (C / 8))), dim3(256), 0, n->stream, src, dst, B, H,
                     W, C);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}
lbm_status up_bwd(lbm_net* n, int level, int B, Act gfine, Act gcoarse, int C) {
  const int H = H_(n, level), W = W_(n, level);
  hipLaunchKernelGGL(k_up_bwd, dim3(blocks_for(size_t(B) * (H / 2) * (W / 2) * (C / 8))), dim3(256), 0, n->stream,
                     gfine, gcoarse, B, H, W, C);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}

lbm_status forward(lbm_net* n, int B) {
  const int* w = n->cfg.widths;
  const int cw[3] = {w[1] + w[0], w[2] + w[1], w[3] + w[2]};  // cat widths: [up | skip]
  // encoder
  NS(conv(n, 0, B, act(n->x, 8), act(n->a[0], w[0]), nullptr));
  NS(conv(n, 1, B, act(n->a[0], w[0]), act(n->cat[0], cw[0], w[1]), nullptr));
  NS(pool_fwd(n, 0, B, act(n->cat[0], cw[0], w[1]), act(n->pool[1], w[0]), w[0]));
  NS(conv(n, 2, B, act(n->pool[1], w[0]), act(n->a[1], w[1]), nullptr));
  NS(conv(n, 3, B, act(n->a[1], w[1]), act(n->cat[1], cw[1], w[2]), nullptr));
  NS(pool_fwd(n, 1, B, act(n->cat[1], cw[1], w[2]), act(n->pool[2], w[1]), w[1]));
  NS(conv(n, 4, B, act(n->pool[2], w[1]), act(n->a[2], w[2]), nullptr));
  NS(conv(n, 5, B, act(n->a[2], w[2]), act(n->cat[2], cw[2], w[3]), nullptr));
  NS(pool_fwd(n, 2, B, act(n->cat[2], cw[2], w[3]), act(n->pool[3], w[2]), w[2]));
  NS(conv(n, 6, B, act(n->pool[3], w[2]), act(n->a[3], w[3]), nullptr));
  NS(conv(n, 7, B, act(n->a[3], w[3]), act(n->bott, w[3]), nullptr));
  // decoder
  NS(up_fwd(n, 2, B, act(n->bott, w[3]), act(n->cat[2], cw[2], 0), w[3]));
  NS(conv(n, 8, B, act(n->cat[2], cw[2]), act(n->dec[2], w[2]), nullptr));
  NS(up_fwd(n, 1, B, act(n->dec[2], w[2]), act(n->cat[1], cw[1], 0), w[2]));
  NS(conv(n, 9, B, act(n->cat[1], cw[1]), act(n->dec[1], w[1]), nullptr));
  NS(up_fwd(n, 0, B, act(n->dec[1], w[1]), act(n->cat[0], cw[0], 0), w[1]));
  NS(conv(n, 10, B, act(n->cat[0], cw[0]), act(n->dec[0], w[0]), nullptr));
  NS(conv(n, 11, B, act(n->dec[0], w[0]), act(nullptr, 0), n->y));
  return LBM_OK;
}

lbm_status loss_fwd(lbm_net* n, int B, double nf, double* dloss, float* dlossf) {
  const int M = B * n->cfg.height * n->cfg.width;
  const float inv = float(1.0 / (3.0 * std::max(1.0, nf)));
  const unsigned nb = blocks_for(size_t(M));
  hipLaunchKernelGGL(k_loss, dim3(nb), dim3(256), 0, n->stream, n->y, n->t, n->msk, M, inv, n->gy, n->lpartial);
  NET_TRY(hipGetLastError());
  hipLaunchKernelGGL(k_loss_reduce, dim3(1), dim3(256), 0, n->stream, n->lpartial, int(nb),
                     1.0 / (3.0 * std::max(1.0, nf)), dloss, dlossf);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}

lbm_status backward(lbm_net* n, int B) {
  NS(need_partial(n));
  n->npending = 0;  // (of a backward pass that failed)
  n->partial_used = 0;
  const int* w = n->cfg.widths;
  const int cw[3] = {w[1] + w[0], w[2] + w[1], w[3] + w[2]};
  const Act none{nullptr, 0, 0};
  NS(conv_bwd(n, 11, B, act(n->dec[0], w[0]), act(n->gy, 8), act(n->gdec[0], w[0]), true));
  NS(conv_bwd(n, 10, B, act(n->cat[0], cw[0]), act(n->gdec[0], w[0]), act(n->gcat[0], cw[0]), true));
  NS(up_bwd(n, 0, B, act(n->gcat[0], cw[0], 0), act(n->gdec[1], w[1]), w[1]));
  NS(conv_bwd(n, 9, B, act(n->cat[1], cw[1]), act(n->gdec[1], w[1]), act(n->gcat[1], cw[1]), true));
  NS(up_bwd(n, 1, B, act(n->gcat[1], cw[1], 0), act(n->gdec[2], w[2]), w[2]));
  NS(conv_bwd(n, 8, B, act(n->cat[2], cw[2]), act(n->gdec[2], w[2]), act(n->gcat[2], cw[2]), true));
  NS(up_bwd(n, 2, B, act(n->gcat[2], cw[2], 0), act(n->gbott, w[3]), w[3]));
  NS(conv_bwd(n, 7, B, act(n->a[3], w[3]), act(n->gbott, w[3]), act(n->ga[3], w[3]), true));
  NS(conv_bwd(n, 6, B, act(n->pool[3], w[2]), act(n->ga[3], w[3]), act(n->gpool[3], w[2]), false));
  NS(pool_bwd(n, 2, B, act(n->gpool[3], w[2]), act(n->gcat[2], cw[2], w[3]), act(n->cat[2], cw[2], w[3]), w[2]));
  NS(conv_bwd(n, 5, B, act(n->a[2], w[2]), act(n->gcat[2], cw[2], w[3]), act(n->ga[2], w[2]), true));
  NS(conv_bwd(n, 4, B, act(n->pool[2], w[1]), act(n->ga[2], w[2]), act(n->gpool[2], w[1]), false));
  NS(pool_bwd(n, 1, B, act(n->gpool[2], w[1]), act(n->gcat[1], cw[1], w[2]), act(n->cat[1], cw[1], w[2]), w[1]));
  NS(conv_bwd(n, 3, B, act(n->a[1], w[1]), act(n->gcat[1], cw[1], w[2]), act(n->ga[1], w[1]), true));
  NS(conv_bwd(n, 2, B, act(n->pool[1], w[0]), act(n->ga[1], w[1]), act(n->gpool[1], w[0]), false));
  NS(pool_bwd(n, 0, B, act(n->gpool[1], w[0]), act(n->gcat[0], cw[0], w[1]), act(n->cat[0], cw[0], w[1]), w[0]));
  NS(conv_bwd(n, 1, B, act(n->a[0], w[0]), act(n->gcat[0], cw[0], w[1]), act(n->ga[0], w[0]), true));
  NS(conv_bwd(n, 0, B, act(n->x, 8), act(n->ga[0], w[0]), none, false));
  return reduce_gradients(n);
}

lbm_status refresh_weights(lbm_net* n) {
  WconvArgs a{};
  size_t end = 0;
  for (int k = 0; k < 12; ++k) {
    const Layer& L = n->layers[k];
    end += (conv_elements(L.cin, L.cpad) + conv_elements(L.cpad, L.cin)) / 8;
    a.layer[k] = WconvLayer{n->w + L.w_off, L.wb, L.wt, L.cin, L.cr, L.cpad, end};
  }
  hipLaunchKernelGGL(k_wconvert, dim3(unsigned(std::min<size_t>(blocks_for(end), 1 << 20))), dim3(256), 0, n->stream, a);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}

// Network input per cell (8 channels):
//   0 fluid indicator (flag >= 2), 1 u_max/0.08, 2 (tau-1/2)/0.7,
//   3 inlet profile shape 4(y-1/2)(ny-3/2-y)/(ny-2)^2, 4 x/(nx-1), 5 y/(ny-1),
//   6 log1p of a 1D hydraulic estimate of the pressure from column x to the
//     outlet in target units: sum over columns x' > x of the plane-Poiseuille
//     gradient 12 nu Q / h(x')^3 (h = open cells of the column, Q the inlet
//     flux), divided by u_max^2,
//   7 log((ny-2)/h(x)), the column's blockage.
// Channels 6-7 carry the domain-wide resistance a 3x3-convolution stack
// cannot integrate over its receptive field.
// Channels 6 and 7 of a lattice's columns.
void column_features(const lbm_net_config& cfg, const uint8_t* flags, double u_max, double tau, float* press,
                     float* block) {
  const int H = cfg.height, W = cfg.width;
  const double nu = (tau - 0.5) / 3.0;
  double S = 0.0;  // inlet flux / u_max
  for (int y = 1; y < H - 1; ++y) S += 4.0 * (y - 0.5) * (H - 1.5 - y) / ((H - 2.0) * (H - 2.0));
  std::vector<int> h(W, 0);
  for (int y = 0; y < H; ++y)
    for (int x = 0; x < W; ++x) h[x] += flags[size_t(y) * W + x] >= 2 ? 1 : 0;
  const double hfull = H > 2 ? double(H - 2) : 1.0;
  double acc = 0.0;
  for (int x = W - 1; x >= 0; --x) {
    const double hcol = h[x] > 0 ? double(h[x]) : 1.0;
    press[x] = float(std::log1p(12.0 * nu * S * acc / u_max));
    block[x] = float(std::log(hfull / hcol));
    acc += 1.0 / (hcol * hcol * hcol);
  }
}
float speed_feature(double u_max) { return float(u_max / 0.08); }
float tau_feature(double tau) { return float((tau - 0.5) / 0.7); }
float profile_feature(const lbm_net_config& cfg, int y) {
  const double H = cfg.height, yy = y;
  return float(4.0 * (yy - 0.5) * (H - 1.5 - yy) / ((H - 2.0) * (H - 2.0)));
}
float x_feature(const lbm_net_config& cfg, int x) { return float(double(x) / double(cfg.width - 1)); }
float y_feature(const lbm_net_config& cfg, int y) { return float(double(y) / double(cfg.height - 1)); }

void host_features(const lbm_net_config& cfg, const uint8_t* flags, double u_max, double tau, float* out) {
  const int H = cfg.height, W = cfg.width;
  std::vector<float> press(W), block(W);
  column_features(cfg, flags, u_max, tau, press.data(), block.data());
  for (int y = 0; y < H; ++y)
    for (int x = 0; x < W; ++x) {
      float* f = out + (size_t(y) * W + x) * 8;
      f[0] = flags[size_t(y) * W + x] >= 2 ? 1.f : 0.f;
      f[1] = speed_feature(u_max);
      f[2] = tau_feature(tau);
      f[3] = profile_feature(cfg, y);
      f[4] = x_feature(cfg, x);
      f[5] = y_feature(cfg, y);
      f[6] = press[x];
      f[7] = block[x];
    }
}

// The network input of B lattices of `flags`, as bf16(host_features): the flags
// and what the features depend on (row, column, lattice and its column, two
// channels to a word) go to the device, where k_features lays them out.
size_t feature_words(const lbm_net_config& cfg, int B) {
  return size_t(cfg.height) + cfg.width + size_t(B) * (cfg.width + 1);
}
lbm_status upload_features(lbm_net* n, int B, const uint8_t* flags, const double* u_max, const double* tau,
                           std::vector<uint32_t>& tab) {
  const int H = n->cfg.height, W = n->cfg.width;
  const size_t HW = size_t(H) * W;
  auto two = [](float lo, float hi) { return uint32_t(f2bf(lo)) | (uint32_t(f2bf(hi)) << 16); };
  tab.resize(feature_words(n->cfg, B));
  uint32_t* rows = tab.data();
  uint32_t* cols = rows + H;
  uint32_t* per = cols + W;
  for (int y = 0; y < H; ++y) rows[y] = two(profile_feature(n->cfg, y), y_feature(n->cfg, y));
  for (int x = 0; x < W; ++x) cols[x] = two(x_feature(n->cfg, x), 0.f);
  std::vector<float> press(W), block(W);
  for (int b = 0; b < B; ++b, per += W + 1) {
    column_features(n->cfg, flags + b * HW, u_max[b], tau[b], press.data(), block.data());
    per[0] = two(speed_feature(u_max[b]), tau_feature(tau[b]));
    for (int x = 0; x < W; ++x) per[1 + x] = two(press[x], block[x]);
  }
  NET_TRY(hipMemcpyAsync(n->msk, flags, B * HW, hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipMemcpyAsync(n->ftab, tab.data(), tab.size() * sizeof(uint32_t), hipMemcpyHostToDevice, n->stream));
  hipLaunchKernelGGL(k_features, dim3(blocks_for(B * HW)), dim3(256), 0, n->stream, n->msk, n->ftab, B, H, W, n->x);
  NET_TRY(hipGetLastError());
  return LBM_OK;
}

lbm_status upload_x(lbm_net* n, const float* x, size_t count) {
  std::vector<uint16_t> h(count);
  for (size_t i = 0; i < count; ++i) h[i] = f2bf(x[i]);
  NET_TRY(hipMemcpyAsync(n->x, h.data(), count * sizeof(uint16_t), hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipStreamSynchronize(n->stream));
  return LBM_OK;
}

void free_all(lbm_net* n) {
  for (Layer& L : n->layers) {
    (void)hipFree(L.wb);
    (void)hipFree(L.wt);
  }
  void* ps[] = {n->w,        n->g,     n->m1,      n->m2,   n->y,  n->t,  n->msk, n->ftab, n->partial,
                n->lpartial, n->dloss, n->dlosses, n->didx, n->xs, n->ts, n->ms};
  for (void* p : ps) (void)hipFree(p);
  for (uint16_t* p : {n->x, n->bott, n->gbott, n->gy}) afree(p);
  for (int l = 0; l < 4; ++l)
    for (uint16_t* p : {n->a[l], n->ga[l], n->pool[l], n->gpool[l]}) afree(p);
  for (int l = 0; l < 3; ++l)
    for (uint16_t* p : {n->cat[l], n->gcat[l], n->dec[l], n->gdec[l]}) afree(p);
  if (n->ev0) (void)hipEventDestroy(n->ev0);
  if (n->ev1) (void)hipEventDestroy(n->ev1);
  if (n->stream) (void)hipStreamDestroy(n->stream);
}

lbm_status create_impl(lbm_net* n) {
  const lbm_net_config& c = n->cfg;
  const int* w = c.widths;
  NET_TRY(hipSetDevice(n->device));
  NET_TRY(hipStreamCreateWithFlags(&n->stream, hipStreamNonBlocking));
  NET_TRY(hipEventCreate(&n->ev0));
  NET_TRY(hipEventCreate(&n->ev1));
  build_layers(n);
  NS(dalloc(&n->w, n->nparam));
  NS(dalloc(&n->g, n->nparam));
  NS(dalloc(&n->m1, n->nparam));
  NS(dalloc(&n->m2, n->nparam));
  for (Layer& L : n->layers) {
    // (three K steps of padding: the conv's last turn loads a turn ahead)
    NS(dalloc(&L.wb, conv_elements(L.cin, L.cpad) + 3 * 512 * size_t(conv_tiles(L.cpad))));
    NS(dalloc(&L.wt, conv_elements(L.cpad, L.cin) + 3 * 512 * size_t(conv_tiles(L.cin))));
  }
  const int cw[3] = {w[1] + w[0], w[2] + w[1], w[3] + w[2]};
  NS(aalloc(&n->x, level_pixels(n, 0) * 8));
  for (int l = 0; l < 4; ++l) {
    NS(aalloc(&n->a[l], level_pixels(n, l) * w[l]));
    NS(aalloc(&n->ga[l], level_pixels(n, l) * w[l]));
    if (l > 0) {
      NS(aalloc(&n->pool[l], level_pixels(n, l) * w[l - 1]));
      NS(aalloc(&n->gpool[l], level_pixels(n, l) * w[l - 1]));
    }
  }
  for (int l = 0; l < 3; ++l) {
    NS(aalloc(&n->cat[l], level_pixels(n, l) * cw[l]));
    NS(aalloc(&n->gcat[l], level_pixels(n, l) * cw[l]));
    NS(aalloc(&n->dec[l], level_pixels(n, l) * w[l]));
    NS(aalloc(&n->gdec[l], level_pixels(n, l) * w[l]));
  }
  NS(aalloc(&n->bott, level_pixels(n, 3) * w[3]));
  NS(aalloc(&n->gbott, level_pixels(n, 3) * w[3]));
  NS(aalloc(&n->gy, level_pixels(n, 0) * 8));
  NS(dalloc(&n->y, level_pixels(n, 0) * 3));
  NS(dalloc(&n->t, level_pixels(n, 0) * 3));
  NS(dalloc(&n->msk, level_pixels(n, 0)));
  NS(dalloc(&n->ftab, feature_words(n->cfg, c.batch)));
  if (c.capacity > 0) NS(need_partial(n));  // (a network that is to be trained)
  NS(dalloc(&n->lpartial, size_t(blocks_for(level_pixels(n, 0)))));
  NS(dalloc(&n->dloss, 1));
  const size_t HW = size_t(c.height) * c.width;
  if (c.capacity > 0) {
    NS(dalloc(&n->xs, size_t(c.capacity) * HW * 8));
    NS(dalloc(&n->ts, size_t(c.capacity) * HW * 3));
    NS(dalloc(&n->ms, size_t(c.capacity) * HW));
  }
  // He-normal initialisation, biases zero
  std::vector<float> hw(n->nparam, 0.f);
  HeLayer he[12];
  for (int k = 0; k < 12; ++k) {
    const Layer& L = n->layers[k];
    he[k] = {hw.data() + L.w_off, size_t(9) * L.cin * L.cr, L.cin};
  }
  he_normal(c.seed, he, 12);
  NET_TRY(hipMemcpy(n->w, hw.data(), n->nparam * sizeof(float), hipMemcpyHostToDevice));
  NS(refresh_weights(n));
  NET_TRY(hipStreamSynchronize(n->stream));
  return LBM_OK;
}

bool valid_config(const lbm_net_config* c) {
  if (c->height < 8 || c->width < 8 || c->height % 8 || c->width % 8) return false;
  for (int l = 0; l < 4; ++l)
    if (c->widths[l] <= 0 || c->widths[l] % 8) return false;
  if (c->batch < 1 || c->capacity < 0) return false;
  const size_t px = size_t(c->batch) * c->height * c->width;
  return px <= size_t(1) << 31;
}

}  // namespace

extern "C" {

lbm_status lbm_net_create(lbm_net** out, const lbm_net_config* cfg, int32_t device) {
  if (!out || !cfg) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  *out = nullptr;
  if (!valid_config(cfg))
    return nfail(LBM_ERR_INVALID_ARG, "net config: height/width must be multiples of 8 (>= 8), widths multiples of 8, batch >= 1");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || device < 0 || device >= ndev)
    return nfail(LBM_ERR_NOT_FOUND, "device %d not present", device);
  lbm_net* n = new lbm_net();
  n->cfg = *cfg;
  n->device = device;
  lbmx::read_back_user(1);
  lbm_status s = create_impl(n);
  if (s != LBM_OK) {
    free_all(n);
    delete n;
    lbmx::read_back_user(-1);
    return s;
  }
  *out = n;
  return LBM_OK;
}

lbm_status lbm_net_destroy(lbm_net* n) {
  if (!n) return LBM_OK;
  (void)hipSetDevice(n->device);
  if (n->stream) (void)hipStreamSynchronize(n->stream);
  free_all(n);
  delete n;
  lbmx::read_back_user(-1);
  return LBM_OK;
}

lbm_status lbm_net_param_count(lbm_net* n, uint64_t* count) {
  if (!n || !count) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  *count = n->nparam;
  return LBM_OK;
}

lbm_status lbm_net_get_params(lbm_net* n, float* p) {
  if (!n || !p) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  NET_TRY(hipSetDevice(n->device));
  NET_TRY(hipMemcpyAsync(p, n->w, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
  NET_TRY(hipStreamSynchronize(n->stream));
  return LBM_OK;
}

lbm_status lbm_net_set_params(lbm_net* n, const float* p) {
  if (!n || !p) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  NET_TRY(hipSetDevice(n->device));
  NET_TRY(hipMemcpyAsync(n->w, p, n->nparam * sizeof(float), hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipMemsetAsync(n->m1, 0, n->nparam * sizeof(float), n->stream));
  NET_TRY(hipMemsetAsync(n->m2, 0, n->nparam * sizeof(float), n->stream));
  n->adam_t = 0;
  NS(refresh_weights(n));
  NET_TRY(hipStreamSynchronize(n->stream));
  return LBM_OK;
}

lbm_status lbm_net_features(lbm_net* n, const uint8_t* flags, double u_max, double tau, float* features) {
  if (!n || !flags || !features) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  host_features(n->cfg, flags, u_max, tau, features);
  return LBM_OK;
}

lbm_status lbm_net_add_sample(lbm_net* n, const uint8_t* flags, double u_max, double tau, const double* rho,
                              const double* u) {
  if (!n || !flags || !rho || !u) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  if (int(n->nf.size()) >= n->cfg.capacity)
    return nfail(LBM_ERR_OVERFLOW, "training set full (capacity %d)", n->cfg.capacity);
  if (!(u_max > 0.0) || !(tau > 0.5)) return nfail(LBM_ERR_INVALID_ARG, "need u_max > 0 and tau > 1/2");
  const size_t HW = size_t(n->cfg.height) * n->cfg.width, k = n->nf.size();
  for (size_t i = 0; i < HW; ++i)
    if (!std::isfinite(rho[i]) || !std::isfinite(u[i]) || !std::isfinite(u[HW + i]))
      return nfail(LBM_ERR_INVALID_ARG, "sample has a non-finite value at cell %zu", i);
  std::vector<float> f(HW * 8);
  host_features(n->cfg, flags, u_max, tau, f.data());
  std::vector<uint16_t> xb(HW * 8);
  for (size_t i = 0; i < HW * 8; ++i) xb[i] = f2bf(f[i]);
  std::vector<float> t(HW * 3);
  std::vector<uint8_t> m(HW);
  double cnt = 0.0;
  const double ru = rho_unit(u_max);
  for (size_t i = 0; i < HW; ++i) {
    m[i] = flags[i] >= 2 ? 1 : 0;
    cnt += m[i];
    t[i * 3 + 0] = float(u[i] / u_max);
    t[i * 3 + 1] = float(u[HW + i] / u_max);
    t[i * 3 + 2] = float((rho[i] - 1.0) / ru);
    if (m[i])
      for (int c = 0; c < 3; ++c) {
        n->tsum[c] += t[i * 3 + c];
        n->tsq[c] += double(t[i * 3 + c]) * t[i * 3 + c];
      }
  }
  n->tcnt += cnt;
  if (n->frozen)
    for (size_t i = 0; i < HW * 3; ++i) t[i] = (t[i] - n->mu[i % 3]) / n->sd[i % 3];
  NET_TRY(hipSetDevice(n->device));
  NET_TRY(hipMemcpyAsync(n->xs + k * HW * 8, xb.data(), HW * 8 * sizeof(uint16_t), hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipMemcpyAsync(n->ts + k * HW * 3, t.data(), HW * 3 * sizeof(float), hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipMemcpyAsync(n->ms + k * HW, m.data(), HW, hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipStreamSynchronize(n->stream));
  n->nf.push_back(cnt);
  return LBM_OK;
}

lbm_status lbm_net_clear_samples(lbm_net* n) {
  if (!n) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  n->nf.clear();
  return LBM_OK;
}

lbm_status lbm_net_sample_count(lbm_net* n, uint32_t* count) {
  if (!n || !count) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  *count = uint32_t(n->nf.size());
  return LBM_OK;
}

lbm_status lbm_net_train(lbm_net* n, uint32_t steps, float lr, uint64_t seed, float* losses) {
  if (!n) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  const uint32_t S = uint32_t(n->nf.size());
  const int B = n->cfg.batch;
  if (S < uint32_t(B)) return nfail(LBM_ERR_INVALID_STATE, "training set holds %u samples, batch is %d", S, B);
  if (steps == 0) return LBM_OK;
  NET_TRY(hipSetDevice(n->device));
  if (!n->frozen && n->tcnt > 0) {
    for (int c = 0; c < 3; ++c) {
      const double m = n->tsum[c] / n->tcnt;
      const double v = std::max(n->tsq[c] / n->tcnt - m * m, 0.0);
      n->mu[c] = float(m);
      n->sd[c] = float(std::max(std::sqrt(v), 1e-6));
    }
    const size_t cnt = size_t(S) * n->cfg.height * n->cfg.width * 3;
    hipLaunchKernelGGL(k_standardize, dim3(blocks_for(cnt)), dim3(256), 0, n->stream, n->ts, cnt, n->mu[0], n->mu[1],
                       n->mu[2], n->sd[0], n->sd[1], n->sd[2]);
    NET_TRY(hipGetLastError());
    n->frozen = true;
  }
  // minibatch indices: a fresh seeded permutation per epoch
  std::vector<uint32_t> idx(size_t(steps) * B), perm(S);
  std::mt19937_64 rng(seed);
  size_t pos = S;
  std::vector<double> nfb(steps, 0.0);
  for (uint32_t k = 0; k < steps; ++k)
    for (int b = 0; b < B; ++b) {
      if (pos + 1 > S) {
        for (uint32_t i = 0; i < S; ++i) perm[i] = i;
        std::shuffle(perm.begin(), perm.end(), rng);
        pos = 0;
      }
      idx[size_t(k) * B + b] = perm[pos++];
      nfb[k] += n->nf[idx[size_t(k) * B + b]];
    }
  if (n->didx_n < idx.size()) {
    (void)hipFree(n->didx);
    n->didx = nullptr;
    NS(dalloc(&n->didx, idx.size()));
    n->didx_n = idx.size();
  }
  if (n->dlosses_n < steps) {
    (void)hipFree(n->dlosses);
    n->dlosses = nullptr;
    NS(dalloc(&n->dlosses, steps));
    n->dlosses_n = steps;
  }
  NET_TRY(hipMemcpyAsync(n->didx, idx.data(), idx.size() * sizeof(uint32_t), hipMemcpyHostToDevice, n->stream));
  const int HW = n->cfg.height * n->cfg.width;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  NET_TRY(hipEventRecord(n->ev0, n->stream));
  for (uint32_t k = 0; k < steps; ++k) {
    hipLaunchKernelGGL(k_gather, dim3(blocks_for(size_t(B) * HW)), dim3(256), 0, n->stream, n->xs, n->ts, n->ms,
                       n->didx + size_t(k) * B, B, HW, n->x, n->t, n->msk);
    NET_TRY(hipGetLastError());
    NS(forward(n, B));
    NS(loss_fwd(n, B, nfb[k], nullptr, n->dlosses + k));
    NS(backward(n, B));
    n->adam_t += 1;
    const float c1 = float(1.0 - std::pow(0.9, double(n->adam_t)));
    const float c2 = float(1.0 - std::pow(0.999, double(n->adam_t)));
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(n->nparam)), dim3(256), 0, n->stream, n->w, n->g, n->m1, n->m2,
                       n->nparam, lr, b1, b2, c1, c2, eps);
    NET_TRY(hipGetLastError());
    NS(refresh_weights(n));
  }
  NET_TRY(hipEventRecord(n->ev1, n->stream));
  if (losses)
    NET_TRY(hipMemcpyAsync(losses, n->dlosses, steps * sizeof(float), hipMemcpyDeviceToHost, n->stream));
  NET_TRY(hipStreamSynchronize(n->stream));
  n->timed = true;
  return LBM_OK;
}

lbm_status lbm_net_forward_raw(lbm_net* n, uint32_t count, const float* x, float* y) {
  if (!n || !x || !y) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  NET_TRY(hipSetDevice(n->device));
  const size_t HW = size_t(n->cfg.height) * n->cfg.width;
  for (uint32_t s = 0; s < count; s += n->cfg.batch) {
    const int B = int(std::min<uint32_t>(n->cfg.batch, count - s));
    NS(upload_x(n, x + size_t(s) * HW * 8, size_t(B) * HW * 8));
    NS(forward(n, B));
    NET_TRY(hipMemcpyAsync(y + size_t(s) * HW * 3, n->y, size_t(B) * HW * 3 * sizeof(float), hipMemcpyDeviceToHost,
                           n->stream));
    NET_TRY(hipStreamSynchronize(n->stream));
  }
  return LBM_OK;
}

lbm_status lbm_net_predict(lbm_net* n, uint32_t count, const uint8_t* flags, const double* u_max, const double* tau,
                           double* rho, double* u) {
  if (!n || !flags || !u_max || !tau || !rho || !u) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  NET_TRY(hipSetDevice(n->device));
  const size_t HW = size_t(n->cfg.height) * n->cfg.width;
  std::vector<uint32_t> tab;
  NET_TRY(hipEventRecord(n->ev0, n->stream));
  for (uint32_t s = 0; s < count; s += n->cfg.batch) {
    const int B = int(std::min<uint32_t>(n->cfg.batch, count - s));
    lbm_status st = upload_features(n, B, flags + s * HW, u_max + s, tau + s, tab);
    if (st == LBM_OK) st = forward(n, B);
    if (st != LBM_OK) {
      (void)hipStreamSynchronize(n->stream);  // `tab` may still be read
      return st;
    }
    auto denormalise = [&, s](const char* data, size_t offset, size_t bytes) {
      const float* o = reinterpret_cast<const float*>(data);
      const size_t p0 = offset / (3 * sizeof(float)), p1 = p0 + bytes / (3 * sizeof(float));
      for (size_t p = p0; p < p1;) {  // image by image
        const size_t k = s + p / HW, end = std::min(p1, (p / HW + 1) * HW);
        const uint8_t* fl = flags + k * HW;
        double* r = rho + k * HW;
        double* ux = u + k * 2 * HW;
        double* uy = ux + HW;
        const double um = u_max[k], ru = rho_unit(um);
        for (size_t i = p % HW; p < end; ++p, ++i, o += 3) {
          if (fl[i] >= 2) {
            ux[i] = (double(o[0]) * n->sd[0] + n->mu[0]) * um;
            uy[i] = (double(o[1]) * n->sd[1] + n->mu[1]) * um;
            r[i] = 1.0 + (double(o[2]) * n->sd[2] + n->mu[2]) * ru;
          } else {
            ux[i] = 0.0;
            uy[i] = 0.0;
            r[i] = 1.0;
          }
        }
      }
    };
    const lbmx::ReadBack r{n->y, size_t(B) * HW * 3 * sizeof(float), 3 * sizeof(float), denormalise};
    NET_TRY(lbmx::read_back(n->device, n->stream, &r, 1));
  }
  NET_TRY(hipEventRecord(n->ev1, n->stream));
  NET_TRY(hipEventSynchronize(n->ev1));
  n->timed = true;
  return LBM_OK;
}

lbm_status lbm_net_correct_flux(lbm_net* n, uint32_t count, const uint8_t* flags, const double* u_max, double* u) {
  if (!n || !flags || !u_max || !u) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  const int H = n->cfg.height, W = n->cfg.width;
  const size_t HW = size_t(H) * W;
  double S = 0.0;  // the inlet parabola's flux per unit u_max (the features' profile)
  for (int y = 1; y < H - 1; ++y) S += 4.0 * (y - 0.5) * (H - 1.5 - y) / ((H - 2.0) * (H - 2.0));
  std::vector<double> q(W);
  for (uint32_t k = 0; k < count; ++k) {
    const uint8_t* fl = flags + k * HW;
    double* ux = u + k * 2 * HW;
    double* uy = ux + HW;
    const double q_in = u_max[k] * S;
    std::fill(q.begin(), q.end(), 0.0);
    for (int y = 0; y < H; ++y)
      for (int x = 0; x < W; ++x)
        if (fl[size_t(y) * W + x] >= 2) q[x] += ux[size_t(y) * W + x];
    for (int y = 0; y < H; ++y)
      for (int x = 0; x < W; ++x) {
        const size_t i = size_t(y) * W + x;
        if (fl[i] < 2 || !(q[x] > 0.2 * q_in)) continue;
        const double s = q_in / q[x];
        ux[i] *= s;
        uy[i] *= s;
      }
  }
  return LBM_OK;
}

lbm_status lbm_net_loss_grad_raw(lbm_net* n, uint32_t count, const float* x, const float* t, const float* m,
                                 double* loss, float* grad) {
  if (!n || !x || !t || !m || !loss || !grad) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  if (count < 1 || int(count) > n->cfg.batch) return nfail(LBM_ERR_INVALID_ARG, "count must be 1..batch");
  NET_TRY(hipSetDevice(n->device));
  const int B = int(count);
  const size_t HW = size_t(n->cfg.height) * n->cfg.width, P = size_t(B) * HW;
  NS(upload_x(n, x, P * 8));
  std::vector<uint8_t> mb(P);
  double nf = 0.0;
  for (size_t i = 0; i < P; ++i) {
    mb[i] = m[i] > 0.f ? 1 : 0;
    nf += mb[i];
  }
  NET_TRY(hipMemcpyAsync(n->t, t, P * 3 * sizeof(float), hipMemcpyHostToDevice, n->stream));
  NET_TRY(hipMemcpyAsync(n->msk, mb.data(), P, hipMemcpyHostToDevice, n->stream));
  NS(forward(n, B));
  NS(loss_fwd(n, B, nf, n->dloss, nullptr));
  NS(backward(n, B));
  NET_TRY(hipMemcpyAsync(loss, n->dloss, sizeof(double), hipMemcpyDeviceToHost, n->stream));
  NET_TRY(hipMemcpyAsync(grad, n->g, n->nparam * sizeof(float), hipMemcpyDeviceToHost, n->stream));
  NET_TRY(hipStreamSynchronize(n->stream));
  return LBM_OK;
}

lbm_status lbm_net_get_output_scale(lbm_net* n, float mean[3], float stdev[3]) {
  if (!n || !mean || !stdev) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  for (int c = 0; c < 3; ++c) {
    mean[c] = n->mu[c];
    stdev[c] = n->sd[c];
  }
  return LBM_OK;
}

lbm_status lbm_net_set_output_scale(lbm_net* n, const float mean[3], const float stdev[3]) {
  if (!n || !mean || !stdev) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  if (n->frozen && !n->nf.empty())
    return nfail(LBM_ERR_INVALID_STATE, "training set already standardised with other statistics");
  for (int c = 0; c < 3; ++c) {
    if (!(stdev[c] > 0.f)) return nfail(LBM_ERR_INVALID_ARG, "stdev must be positive");
    n->mu[c] = mean[c];
    n->sd[c] = stdev[c];
  }
  n->frozen = true;
  return LBM_OK;
}

lbm_status lbm_net_last_ms(lbm_net* n, double* ms) {
  if (!n || !ms) return nfail(LBM_ERR_INVALID_ARG, "null argument");
  if (!n->timed) return nfail(LBM_ERR_INVALID_STATE, "no train or predict call yet");
  float f = 0.f;
  NET_TRY(hipEventElapsedTime(&f, n->ev0, n->ev1));
  *ms = f;
  return LBM_OK;
}

}  // extern "C"
