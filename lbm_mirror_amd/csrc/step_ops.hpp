// One cell's operators (the drivers' switch on the cell flag) and the storage
// types of the populations, shared by the fused stream+collide kernels.
#pragma once
#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "kernels.hpp"

namespace lbmx {

// ---- storage traits --------------------------------------------------------
template <class S, class T>
struct Store;
template <>
struct Store<double, double> {
  template <class P>
  __device__ static double ld(P p, double) { return *p; }
  template <class P>
  __device__ static void st(P p, double v, double) { *p = v; }
  __device__ static double zero(double) { return 0.0; }
};
#ifndef LBMX_NT
#define LBMX_NT 0
#endif
template <>
struct Store<float, float> {
  template <class P>
  __device__ static float ld(P p, float) {
    if (LBMX_NT & 1) return __builtin_nontemporal_load(p);
    return *p;
  }
  template <class P>
  __device__ static void st(P p, float v, float) {
    if (LBMX_NT & 2) __builtin_nontemporal_store(v, p);
    else *p = v;
  }
};
// Shifted 16-bit storage: the stored value is f_i − w_i.
template <>
struct Store<__half, float> {
  // as raw 16-bit words: the class type cannot be accessed through a
  // global-typed pointer
  template <class P>
  __device__ static float ld(P p, float w) {
    return __half2float(__ushort_as_half(*(const __attribute__((address_space(1))) unsigned short*)p)) + w;
  }
  template <class P>
  __device__ static void st(P p, float v, float w) {
    *(__attribute__((address_space(1))) unsigned short*)p = __half_as_ushort(__float2half(v - w));
  }
};
template <>
struct Store<__hip_bfloat16, float> {
  template <class P>
  __device__ static float ld(P p, float w) {
    return __bfloat162float(__ushort_as_bfloat16(*(const __attribute__((address_space(1))) unsigned short*)p)) + w;
  }
  template <class P>
  __device__ static void st(P p, float v, float w) {
    *(__attribute__((address_space(1))) unsigned short*)p = __bfloat16_as_ushort(__float2bfloat16(v - w));
  }
};

// A field of the lattice, typed as global memory: accesses through it are
// GLOBAL, not FLAT, also where the pointer was loaded from memory (batch
// members).
template <class T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gfield(const void* p) {
  return (__attribute__((address_space(1))) T*)(p);
}

// The boundary (kind bc) of one cell's operator (the drivers' switch(info)): f
// holds the pre-collision populations.
template <class L, class T, bool WB, class OpP>
__device__ __forceinline__ void apply_boundary(T (&f)[L::Q], OpP op, int bc, const StepArgs& a, uint32_t cell) {
  constexpr int Q = L::Q;
  switch (bc) {
    case LBM_BC_BOUNCE_BACK: {
      T g[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) g[i] = f[L::opp[i]];
#pragma unroll
      for (int i = 0; i < Q; ++i) f[i] = g[i];
      break;
    }
    case LBM_BC_ANTI_BOUNCE_BACK: {
      if constexpr (Q == 9) {
        const T f3 = f[3], f5 = f[5], f6 = f[6];
        f[3] = f[4];
        f[4] = f3;
        f[5] = f[7];
        f[6] = f[8];
        f[7] = f5;
        f[8] = f6;
      }
      break;
    }
    case LBM_BC_ZOUHE_PRESSURE_X: {
      const uint64_t t = a.t_dev ? *a.t_dev + a.t : a.t;
      const double rs = (op->ramp_steps > 0 && t < op->ramp_steps)
                            ? op->rho_start + op->rho_slope * double(t)
                            : op->rho_final;
      if constexpr (Q == 9) zouhe_p_d2q9<T>(f, op->east != 0, T(rs));
      if constexpr (Q == 27)
        zouhe_p_d3q27<T>(f, op->east != 0, T(rs), (op->flags & LBM_OPF_ZOUHE_NORMAL_ONLY) != 0);
      break;
    }
    case LBM_BC_ZOUHE_VELOCITY_X: {
      if constexpr (Q == 9) {
        const auto bv = gfield<const T>(a.bcvel);
        zouhe_u_d2q9<T>(f, op->east != 0, bv[cell], bv[a.N + cell]);
      }
      break;
    }
    case LBM_BC_EQUILIBRIUM: {
      const T u[3] = {T(op->vec[0]), T(op->vec[1]), T(op->vec[2])};
      equilibrium<L, T, WB>(T(op->rho_eq), u, f);
      break;
    }
    default:
      break;
  }
}

// Its collision (kind coll), writing the macros when asked; f holds the post-collision
// populations afterwards.
// LEAN: the lattice's operators are boundaries with BGK, BGKGuo or no collision
// (no particle field) and the step writes no macros: the rest is compiled out.
template <class L, class T, bool WB, bool LEAN, class OpP>
__device__ __forceinline__ void apply_collision(T (&f)[L::Q], OpP op, int coll, const StepArgs& a, uint32_t cell,
                                                int x, int y, int z) {
  constexpr int Q = L::Q;
  if (coll != LBM_COLL_NONE) {
    T rho, u[3];
    T B = T(1);
    auto por = gfield<T>(a.por);
    if (!LEAN && coll == LBM_COLL_PSM) {
      if (op->flags & LBM_OPF_PSM_STAMP_DISC) {
        const int xc[3] = {x, y, z};
        T rel[3];
#pragma unroll
        for (int d = 0; d < L::D; ++d) rel[d] = T(xc[d]) - T(op->disc[d]);
        B = disc_porosity<T, L::D>(rel, T(op->disc[3]), T(op->disc[4]));
        por[cell] = B;
      } else {
        B = por[cell];
      }
    }
    rho_u<L, T>(f, rho, u);
    if (!LEAN && a.write_macros) {
      gfield<T>(a.rho)[cell] = rho;
      auto um = gfield<T>(a.u);
      bool bad = !__builtin_isfinite(rho);
#pragma unroll
      for (int d = 0; d < L::D; ++d) {
        um[size_t(d) * a.N + cell] = u[d];
        bad = bad || !__builtin_isfinite(u[d]);
      }
      // one store per wavefront that meets a non-finite value
      const uint64_t m = __ballot(bad);
      if (m != 0 && a.status && __lane_id() == uint32_t(__ffsll((unsigned long long)m) - 1))
        __hip_atomic_store(a.status + kStatusNonFinite, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    const T om = T(op->omega);
    if (coll == LBM_COLL_BGK) {
      bgk<L, T, WB>(f, rho, u, om);
    } else if (coll == LBM_COLL_BGK_GUO) {
      T F[3];
      const auto cf = gfield<const T>(a.force);
      const bool use_cf = op->flags & LBM_OPF_GUO_CELL_FORCE;
#pragma unroll
      for (int d = 0; d < L::D; ++d) F[d] = (use_cf ? cf[size_t(d) * a.N + cell] : T(0)) + T(op->vec[d]);
      bgk_guo<L, T, WB>(f, rho, u, om, F, op->force_mask);
    } else if (LEAN) {
      // no other collision reaches a lean kernel
    } else if (coll == LBM_COLL_FPLBM) {
      // fplbm.hpp:60-133: BGKGuo's arithmetic with the cell force field and
      // u = m/rho; the macros hold rho and the momentum (FpLbmReset)
      T F[3] = {T(0), T(0), T(0)};
      const auto cf = gfield<const T>(a.force);
#pragma unroll
      for (int d = 0; d < L::D; ++d) F[d] = cf[size_t(d) * a.N + cell];
      if (a.write_macros) {
        T m[3] = {T(0), T(0), T(0)};
#pragma unroll
        for (int j = 1; j < Q; ++j)
#pragma unroll
          for (int d = 0; d < L::D; ++d)
            if (cdir<L>(j, d) != 0) m[d] = m[d] + T(cdir<L>(j, d)) * f[j];
        auto um = gfield<T>(a.u);
#pragma unroll
        for (int d = 0; d < L::D; ++d) um[size_t(d) * a.N + cell] = m[d];
      }
      bgk_guo<L, T, WB>(f, rho, u, om, F, 7u);
    } else if (coll == LBM_COLL_HLBM) {
      // hlbm.hpp:62-105: velocity u*B + N(1-B)/D (N when D = 0); the macros
      // receive that velocity, written here after the plain moments
      const T Bp = gfield<const T>(a.por)[cell];
      const T flip = T(1.0) - Bp;
      const T Dw = gfield<const T>(a.pd)[cell];
      const auto pn = gfield<const T>(a.pn);
#pragma unroll
      for (int d = 0; d < L::D; ++d) {
        const T Nd = pn[size_t(d) * a.N + cell];
        const T term = (Dw > T(0)) ? (Nd * flip) / Dw : Nd;
        u[d] = u[d] * Bp + term;
      }
      if (a.write_macros) {
        auto um = gfield<T>(a.u);
#pragma unroll
        for (int d = 0; d < L::D; ++d) um[size_t(d) * a.N + cell] = u[d];
      }
      bgk<L, T, WB>(f, rho, u, om);
    } else if (coll == LBM_COLL_PSM) {
      psm<L, T, WB>(f, rho, u, om, B);
      if (op->flags & (LBM_OPF_PSM_CELL_FORCE | LBM_OPF_PSM_FORCE_GATHER)) {
        T m[3];
        opp_momentum<L, T>(f, m);
        const T sc = (op->flags & LBM_OPF_PSM_CELL_FORCE) ? B : T(1.0) - B;
        auto fo = gfield<T>(a.force);
#pragma unroll
        for (int d = 0; d < L::D; ++d) fo[size_t(d) * a.N + cell] = m[d] * sc;
      }
    }
  }
}

template <class L, class T, bool WB, bool LEAN, class OpP>
__device__ __forceinline__ void apply_op(T (&f)[L::Q], OpP op, const StepArgs& a, uint32_t cell, int x, int y,
                                         int z) {
  // both kinds in one load
  const int bc = op->bc, coll = op->coll;
  apply_boundary<L, T, WB>(f, op, bc, a, cell);
  apply_collision<L, T, WB, LEAN>(f, op, coll, a, cell, x, y, z);
}

template <class L, class T, bool WB, bool LEAN = false>
__device__ __forceinline__ void collide_cell(T (&f)[L::Q], uint8_t fl, const StepArgs& a,
                                             uint32_t cell, int x, int y, int z) {
  // When every active lane of the wavefront carries the same flag (the bulk
  // of any lattice), the operator is read with scalar loads and its kind is
  // a scalar branch; mixed wavefronts take the per-lane path.
  // The operator table is written only by the host between launches: typed
  // as constant memory, a wavefront-uniform operator is read with scalar
  // loads whatever the kernel stores before its fields are used (as global
  // memory, the fault-word store of the macro-writing branch made the
  // compiler read every operator field with vector loads and wait for them:
  // the D3Q19 phase 1 205 -> 240 us); per-lane reads are vector loads either
  // way.
  using GOp = const __attribute__((address_space(4))) OpDev;
  GOp* ops = (GOp*)a.ops;
  const int fl0 = __builtin_amdgcn_readfirstlane(int(fl));
  if (__all(int(fl) == fl0)) {
    if (fl0 < kMaxOps) apply_op<L, T, WB, LEAN>(f, ops + fl0, a, cell, x, y, z);
  } else {
    if (fl < kMaxOps) apply_op<L, T, WB, LEAN>(f, ops + fl, a, cell, x, y, z);
  }
}

}  // namespace lbmx
