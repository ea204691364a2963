// Several D2Q9 steps per launch, between two population buffers.
//
// A one-step launch of a 2D lattice is bound by what happens around its
// arithmetic: up to some 10^5 cells by the launch itself (about 4 us from one
// dependent launch to the next), above that by reading and writing all
// populations for 200 instructions per cell.  Here a block takes a tile of
// cells with a margin of K cells on every side, reads its populations once,
// runs K steps on them in LDS, each on one margin cell less than the step
// before, and writes the tile: the margins are computed by several blocks,
// the populations move 1/K as often and one launch replaces K.
//
// In LDS the steps alternate as the launches of the one-step kernels do (the
// AA pattern): an even step leaves its results in the cell's own slots, an
// odd one pulls from and pushes to the neighbours' slots, and each slot is
// read and written by one thread per step, so a step needs one barrier and no
// second copy.  A cell outside the lattice is a cell whose results are zero,
// which is what the ghost ring of the one-step kernels amounts to.  The
// arithmetic of a cell is the one-step kernels' own: results are the same
// bits.
//
// Between blocks the two buffers alternate (a block's margin is read while
// its neighbours write), so launches come in pairs that end in the first
// buffer, in the natural layout.
//
// Measured against one-step launches in their tuned shape, us per step in F64,
// F32, F16, BF16: 256x64 3.67 -> 2.07, 3.56 -> 1.75, 3.17 -> 1.76, 3.19 -> 1.79;
// 512x256 5.32 -> 4.07, 4.66 -> 3.14, 4.26 -> 3.13, 4.25 -> 3.25; 1023x517 15.0 ->
// 11.4, 9.97 -> 6.85, 8.24 -> 6.33, 8.29 -> 6.54; 2048x2048 100 -> 56, 52 -> 28, 31.3 ->
// 24.5, 31.6 -> 25.8; 128 uneven lattices with 10.3 M cells 504 -> 174, 143 -> 84, 97 ->
// 75, 108 -> 79.  What bounds it, by counters: with many FP32 cells the issue of
// vector instructions (at four cycles each all of a launch's cycles: 128 lattices);
// in FP64, whose tile of shape A leaves room for one block per CU, half of that,
// the rest waits at the block's barriers; at 1023x517 half; at 256x64, 256 blocks of
// one pass each, a sixth: the chain of steps inside a launch and the launches.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"
#include "step_ops.hpp"

namespace lbmx {

namespace {

// populations in LDS, in the storage type (a 16-bit value is rounded every
// step, as it is between one-step launches)
template <class S, class T>
struct Lds {
  using E = S;
  __device__ static T ld(const E& p, T) { return p; }
  __device__ static void st(E& p, T v, T) { p = v; }
};
template <>
struct Lds<__half, float> {
  using E = uint16_t;
  __device__ static float ld(const E& p, float w) { return __half2float(__ushort_as_half(p)) + w; }
  __device__ static void st(E& p, float v, float w) { p = __half_as_ushort(__float2half(v - w)); }
};
template <>
struct Lds<__hip_bfloat16, float> {
  using E = uint16_t;
  __device__ static float ld(const E& p, float w) { return __bfloat162float(__ushort_as_bfloat16(p)) + w; }
  __device__ static void st(E& p, float v, float w) { p = __bfloat16_as_ushort(__float2bfloat16(v - w)); }
};

// The operator that most cells of the lattice carry (StepArgs::main), held in
// scalar registers for the whole launch.
template <class T>
struct MainOp {
  int flag;  // 0: none
  bool guo;
  uint32_t mask;
  T omega, F[3];
};

template <class L, class T, bool WB>
__device__ __forceinline__ void collide_main(T (&f)[L::Q], const MainOp<T>& m) {
  T rho, u[3];
  rho_u<L, T>(f, rho, u);
  if (m.guo) bgk_guo<L, T, WB>(f, rho, u, m.omega, m.F, m.mask);
  else bgk<L, T, WB>(f, rho, u, m.omega);
}

// K steps on the tile of (RW - 2K) x TY cells at (x0, y0).  A row of the tile
// with its margin is RW cells, so a wavefront takes 64 / RW whole rows at a time
// and a row's place, its flags and most branches are the same for all lanes;
// NW wavefronts share the rows, each keeping its own for the whole launch.
template <class L, class S, class T, bool WB, int K, int RW, int TY, int NW>
__device__ __forceinline__ void multi_tile(const StepArgs& args, const void* from, void* to, int x0, int y0) {
  static_assert(K % 2 == 0 && 64 % RW == 0 && RW > 2 * K, "tile shape");
  constexpr int Q = L::Q, RY = TY + 2 * K, R = RY * RW, RP = 64 / RW, J = (RY + RP * NW - 1) / (RP * NW);
  static_assert(R * (Q * sizeof(typename Lds<S, T>::E) + 1) <= 160 * 1024, "LDS of a CU");
  using M = Lds<S, T>;
  using E = typename M::E;
  using GS = __attribute__((address_space(1))) S;
  using GE = __attribute__((address_space(1))) E;
  using GB = const __attribute__((address_space(1))) uint8_t;
  __shared__ E lf[Q][R];
  __shared__ uint8_t lfl[R];
  StepArgs a = args;
  const int nx = a.nx, ny = a.ny;
  const size_t Np = a.Np;
  const int lane = int(threadIdx.x) & 63, wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  MainOp<T> m;
  {
    const auto op = (const __attribute__((address_space(4))) OpDev*)a.ops + a.main;
    m.flag = a.main;
    m.guo = op->coll == LBM_COLL_BGK_GUO;
    m.mask = op->force_mask;
    m.omega = T(op->omega);
    for (int d = 0; d < 3; ++d) m.F[d] = T(0) + T(op->vec[d]);
  }
  // this lane's column (wrapped into the lattice) and whether it is one
  const int lx = RW == 64 ? lane : lane % RW;
  int gx = x0 - K + lx;
  bool inx = gx >= 0 && gx < nx;
  if (!inx) {
    if (a.periodic & 1u) {
      gx %= nx;
      if (gx < 0) gx += nx;
      inx = true;
    } else {
      gx = 0;
    }
  }
  // the tile's row of this lane in turn j (RW = 64: one row per wavefront), and
  // the lattice's row behind it
  auto tile_row = [&](int j) { return RW == 64 ? wave + j * NW : (wave + j * NW) * RP + lane / RW; };
  auto row_of = [&](int r, int& gy) -> bool {
    gy = y0 - K + r;
    if (gy >= 0 && gy < ny) return true;
    if (!(a.periodic & 2u)) return false;
    gy %= ny;
    if (gy < 0) gy += ny;
    return true;
  };
  // One step of this lane's cell of a row.  In a row that is not plain the
  // walls turn round by selects and the faces apply their boundary; the
  // collision is then mostly the main one again, and runs once for all lanes
  // that share it.
  auto work = [&](T (&f)[Q], int flag, bool is_plain, int gy) {
    bool act = true;
    if (!is_plain) {
      using GOp = const __attribute__((address_space(4))) OpDev;
      GOp* ops = (GOp*)a.ops;
      const uint32_t cell = uint32_t(gy) * uint32_t(nx) + uint32_t(gx);
      const bool wall = (a.cls.bounce >> flag) & 1u;
      T g[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) g[q] = wall ? f[L::opp[q]] : f[q];
#pragma unroll
      for (int q = 0; q < Q; ++q) f[q] = flag == 0 ? T(0) : g[q];
      if ((a.cls.face >> flag) & 1u) {
        const int one = __builtin_amdgcn_readfirstlane(flag);
        if (__all(flag == one)) apply_boundary<L, T, WB>(f, ops + one, ops[one].bc, a, cell);
        else apply_boundary<L, T, WB>(f, ops + flag, ops[flag].bc, a, cell);
      }
      act = (a.cls.same >> flag) & 1u;
      if ((a.cls.other >> flag) & 1u) apply_collision<L, T, WB, true>(f, ops + flag, ops[flag].coll, a, cell, gx, gy, 0);
    }
    if (act) collide_main<L, T, WB>(f, m);
  };
  // turns of this wavefront whose 64 cells all carry the main operator: they
  // need neither flags nor tests
  uint32_t plain = 0;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r = tile_row(j);
    if (r >= RY) continue;
    int gy;
    const int i = r * RW + lx;
    T f[Q];
    if (!row_of(r, gy)) {
      lfl[i] = 0;
#pragma unroll
      for (int q = 0; q < Q; ++q) M::st(lf[q][i], T(0), T(L::w[q]));
      continue;
    }
    const uint32_t row = uint32_t(gy) * uint32_t(nx);
    const int fl = ((GB*)a.flags + row)[gx];
#pragma unroll
    for (int q = 0; q < Q; ++q) f[q] = Store<S, T>::ld((const GS*)from + (size_t(q) * Np + row) + gx, T(L::w[q]));
    const int flag = inx ? (fl < kMaxOps ? fl : kMaxOps) : 0;
    lfl[i] = uint8_t(flag);
    const bool all = __all(flag == m.flag);
    if (all) plain |= 1u << j;
    work(f, flag, all, gy);
#pragma unroll
    for (int q = 0; q < Q; ++q) M::st(lf[L::opp[q]][i], f[q], T(L::w[q]));
  }
  __syncthreads();
  // step s of the launch on the rows and columns that s steps have not used up;
  // ODD steps pull from and push to the neighbours, the others stay in the cell
  auto step = [&](auto odd, int s) {
    constexpr bool ODD = decltype(odd)::value;
    a.t = args.t + uint64_t(s);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int r = tile_row(j);
      if (r < s || r >= RY - s) continue;
      const int i = r * RW + lx;
      if (lx < s || lx >= RW - s) continue;
      const bool all = (plain >> j) & 1u;
      int flag = 0, gy = 0;
      if (!all) {
        flag = lfl[i];
        if (!row_of(r, gy)) gy = 0;
      }
      T f[Q];
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int up = ODD ? i - L::cx[q] - RW * L::cy[q] : i;
        const T v = M::ld(lf[ODD ? L::opp[q] : q][up], T(L::w[q]));
        f[q] = (ODD && sizeof(E) == 2 && lfl[up] == 0) ? T(0) : v;
      }
      work(f, flag, all, gy);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        if (ODD) M::st(lf[q][i + L::cx[q] + RW * L::cy[q]], f[q], T(L::w[q]));
        else M::st(lf[L::opp[q]][i], f[q], T(L::w[q]));
      }
    }
    __syncthreads();
  };
  for (int s = 1; s + 1 < K; s += 2) {
    step(std::integral_constant<bool, true>{}, s);
    step(std::integral_constant<bool, false>{}, s + 1);
  }
  step(std::integral_constant<bool, true>{}, K - 1);
  const int xo = x0 - K + lx;
  if (lx < K || lx >= RW - K || xo >= nx) return;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int r = tile_row(j), gy = y0 - K + r;
    if (r < K || r >= RY - K || gy >= ny) continue;
    const uint32_t row = uint32_t(gy) * uint32_t(nx);
#pragma unroll
    for (int q = 0; q < Q; ++q) ((GE*)to + (size_t(q) * Np + row))[xo] = lf[q][r * RW + lx];
  }
}

template <class L, class S, class T, bool WB, int K, int RW, int TY, int NW>
__global__ __launch_bounds__(64 * NW) void k_multi(StepArgs a, const void* from, void* to) {
  multi_tile<L, S, T, WB, K, RW, TY, NW>(a, from, to, int(blockIdx.x) * (RW - 2 * K), int(blockIdx.y) * TY);
}

template <class L, class S, class T, bool WB, int K, int RW, int TY, int NW>
__global__ __launch_bounds__(64 * NW) void k_multi_batch(BatchArgs b, int flip) {
  const Tile tl = b.tiles[blockIdx.x];
  StepArgs a = b.members[tl.member];
  a.t = *b.t0 + b.k;
  a.t_dev = nullptr;
  multi_tile<L, S, T, WB, K, RW, TY, NW>(a, flip ? a.f2 : a.f, flip ? a.f : a.f2, int(tl.c0 & 0xffffu) * (RW - 2 * K),
                                         int(tl.c0 >> 16) * TY);
}

// The shapes (K, RW, TY, wavefronts), and where each is the fastest of the
// twelve that were timed (us per step, F32 / F64):
//   A  4, 64, 24, 16  the least margin: 2048x1024 17.6 / 33.6 (D 18.8 / 36.5)
//   B  8, 32,  4, 10  the most blocks, the fewest launches: 256x64 1.82 / 2.14
//                     (C 2.14 / 2.68)
//   C  8, 32, 16, 16  300x200 2.56 / 3.20 (B 3.48 / 5.51, D 3.01 / 3.95)
//   D  4, 32, 24, 16  700x300 4.32 / 6.17 (C 4.69 / 7.42, A 4.88 / 6.40)
//   E  4, 32,  8,  8, F  2, 32, 8, 6, G  2, 64, 12, 8  for the steps that are
//                     left over from the longer launches
#define LBMX_MULTI_SHAPES(X) \
  X(A, 4, 64, 24, 16)        \
  X(B, 8, 32, 4, 10)         \
  X(C, 8, 32, 16, 16)        \
  X(D, 4, 32, 24, 16)        \
  X(E, 4, 32, 8, 8)          \
  X(F, 2, 32, 8, 6)          \
  X(G, 2, 64, 12, 8)

enum ShapeId {
#define LBMX_ENUM(ID, K, RW, TY, NW) kShape##ID,
  LBMX_MULTI_SHAPES(LBMX_ENUM)
#undef LBMX_ENUM
};

const MultiShape kShapes[] = {
#define LBMX_ENTRY(ID, K, RW, TY, NW) {kShape##ID, K, RW - 2 * K, TY},
    LBMX_MULTI_SHAPES(LBMX_ENTRY)
#undef LBMX_ENTRY
};

// one lattice (a; from and to), or a batch (b; flip: from f2 to f)
template <class S, class T, bool WB>
hipError_t launch_shape(const MultiShape& sh, const StepArgs* a, const void* from, void* to, const BatchArgs* b,
                        int flip, hipStream_t s) {
  switch (sh.id) {
#define LBMX_CASE(ID, K, RW, TY, NW)                                                                            \
  case kShape##ID:                                                                                              \
    if (a)                                                                                                      \
      hipLaunchKernelGGL((k_multi<D2Q9, S, T, WB, K, RW, TY, NW>),                                              \
                         dim3((a->nx + sh.tx - 1) / sh.tx, (a->ny + sh.ty - 1) / sh.ty), dim3(64 * NW), 0, s, *a, \
                         from, to);                                                                             \
    else                                                                                                        \
      hipLaunchKernelGGL((k_multi_batch<D2Q9, S, T, WB, K, RW, TY, NW>), dim3(b->ntiles), dim3(64 * NW), 0, s,  \
                         *b, flip);                                                                             \
    return hipGetLastError();
    LBMX_MULTI_SHAPES(LBMX_CASE)
#undef LBMX_CASE
  }
  return hipErrorInvalidValue;
}

hipError_t launch_storage(int storage, const MultiShape& sh, const StepArgs* a, const void* from, void* to,
                          const BatchArgs* b, int flip, hipStream_t s) {
  switch (storage) {
    case LBM_F64: return launch_shape<double, double, true>(sh, a, from, to, b, flip, s);
    case LBM_F32: return launch_shape<float, float, true>(sh, a, from, to, b, flip, s);
    case LBM_F16S: return launch_shape<__half, float, false>(sh, a, from, to, b, flip, s);
    case LBM_BF16S: return launch_shape<__hip_bfloat16, float, false>(sh, a, from, to, b, flip, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

// By the cells that one launch covers: few cells need many small blocks and
// long launches, many cells little margin.  F64 leaves C sooner (512x256: C
// 5.22, D 4.14; F32 C 3.24, D 3.63).  Both shapes on both sides of each line, us
// per step in F64 / F32 / F16 / BF16:
//   24000   150x150 B 3.20/2.23/2.15/2.19, C 2.83/2.18/2.15/2.19;
//           170x160 B 3.29/2.28/2.16/2.21, C 2.91/2.22/2.19/2.20 (256x64: B, see above)
//   100000  (F64) 300x300 C 4.40, D 4.22; 330x330 C 4.60, D 4.22
//   160000  400x380 C -/3.76/3.74/3.94, D -/3.70/3.61/3.70;
//           430x400 C -/3.92/3.81/3.99, D -/4.20/4.03/4.13
//   800000  900x850 D 14.5/8.22/7.79/8.13, A 14.3/8.44/7.96/8.37;
//           950x890 D 14.5/8.69/8.41/8.69, A 14.8/8.70/8.15/8.61
// At the lines the shapes differ by less than at a factor of two to either side:
// 13% at most (F64 at 22,500 cells).  A batch counts all its members' cells,
// whatever their widths.
MultiPlan multi_plan(int storage, uint64_t cells) {
  const uint64_t long_until = storage == LBM_F64 ? 100000 : 160000;
  if (cells <= 24000) return {3, {kShapes[kShapeB], kShapes[kShapeE], kShapes[kShapeF]}};
  if (cells <= long_until) return {3, {kShapes[kShapeC], kShapes[kShapeE], kShapes[kShapeF]}};
  if (cells <= 800000) return {2, {kShapes[kShapeD], kShapes[kShapeF]}};
  return {2, {kShapes[kShapeA], kShapes[kShapeG]}};
}

hipError_t launch_multi(int storage, const MultiShape& sh, const StepArgs& a, const void* from, void* to,
                        hipStream_t s) {
  return launch_storage(storage, sh, &a, from, to, nullptr, 0, s);
}

hipError_t launch_multi_batch(int storage, const MultiShape& sh, const BatchArgs& b, int flip, hipStream_t s) {
  if (b.ntiles == 0) return hipSuccess;
  return launch_storage(storage, sh, nullptr, nullptr, nullptr, &b, flip, s);
}

}  // namespace lbmx
