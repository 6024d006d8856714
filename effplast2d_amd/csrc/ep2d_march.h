// ep2d_march.h -- device code the row-marching kernels share: the arithmetic of
// one pseudo-time step on rows carried in registers (March, MarchStage), the
// split scheme's expressions, lane shifts and global access helpers.  The
// file is compiled with -ffp-contract=off (see ep2d_kernels.hip).
#pragma once

#include "ep2d_internal.h"

namespace ep2d {

namespace {

// ---------------------------------------------------------------------------
// Quotient by a uniform divisor d, given rd = RN(1/d): one product and one
// FMA correction (Markstein's method, the same correction step the AMDGPU and
// IA-64 division sequences end with).  For the operand ranges of this solver
// (no overflow, underflow or subnormal quotients) it returns the IEEE quotient
// a / d, so the fused FP64 kernel keeps the reference's arithmetic.
__device__ __forceinline__ double qdiv(double a, double d, double rd) {
  const double q = a * rd;
  return fma(fma(-q, d, a), rd, q);
}

// Global-memory access at a 32-bit element index: the base stays in SGPRs
// (uniform per wave) and the byte offset in one VGPR (saddr form).
template <typename T>
__device__ __forceinline__ T gld(const T* base, unsigned idx) {
  using GT = const __attribute__((address_space(1))) T;
  using GC = const __attribute__((address_space(1))) char;
  return *(GT*)((GC*)base + idx * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void gst(T* base, unsigned idx, T v) {
  using GT = __attribute__((address_space(1))) T;
  using GC = __attribute__((address_space(1))) char;
  *(GT*)((GC*)base + idx * (unsigned)sizeof(T)) = v;
}

// Block -> tile map.  Workgroups are dispatched round-robin over the 8 XCDs
// (block b to XCD b % 8), so XCD x receives its blocks as a contiguous run of
// the tile list: x*q + min(x, r) + b/8 with q = nb/8, r = nb%8 (the first r
// XCDs take one more).  A tile and its neighbours, which share halo rows,
// then mostly run on the same XCD and share its L2.
__device__ __forceinline__ int tile_of_block(int b, int nb) {
  const int x = b & 7, q = nb >> 3, r = nb & 7;
  return x * q + min(x, r) + (b >> 3);
}

// Raw buffer access for row marches: a resource (base in SGPRs; no range
// limit, every access is in bounds by construction), a per-lane byte offset
// fixed along the march and the row's byte offset, uniform, in an SGPR, so
// stepping to the next row costs no vector instruction.  readfirstlane states
// the row offset's uniformity (a value the compiler kept in a VGPR then costs
// one read, not a loop over lanes).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t brsrc(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, -1, 0x00020000);
}
// A resource bounded to the field's bytes (under 2 GiB): an access whose lane
// offset is kOob or more lies past the bound, so a load returns 0 and a store
// is dropped by the hardware.  A bound of 0 (bnull) does that for every lane.
constexpr unsigned kOob = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t brsrc_n(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes,
                                           0x00020000);
}
typedef unsigned int u32x2_t __attribute__((ext_vector_type(2)));
template <typename T>
__device__ __forceinline__ T bld(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff) {
  soff = __builtin_amdgcn_readfirstlane(soff);
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  else if constexpr (sizeof(T) == 4)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b8(r, voff, soff, 0));
}
template <typename T>
__device__ __forceinline__ void bst(__amdgpu_buffer_rsrc_t r, unsigned voff, unsigned soff, T v) {
  soff = __builtin_amdgcn_readfirstlane(soff);
  if constexpr (sizeof(T) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2_t, v), r, voff, soff, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
}

// Return-mapping scale (ComputeJ2 / ComputePlasticity, EffPlast2D.cu:109-176):
// a stress whose squared invariant s2 lies outside the yield radius coh is
// scaled by sc = coh / sqrt(s2); returns whether it is.  FP64 keeps the
// reference's test and quotient (sqrt, compare, divide), skipped when s2 <= c2
// = coh2lo, below which sqrt(s2) <= coh exactly.  The FP32 split scheme tests
// s2 against c2 = coh^2 (rounded to FP32) and scales by coh * rsq(s2), the
// hardware reciprocal square root (about one ulp): the scaled stress lies on
// the yield surface to FP32 accuracy either way.
template <typename CT>
__device__ __forceinline__ bool rm_scale(CT s2, CT coh, CT c2, CT& sc) {
  if constexpr (sizeof(CT) == 8) {
    if (s2 > c2) {
      const CT J = sqrt(s2);
      if (J > coh) {
        sc = coh / J;
        return true;
      }
    }
    return false;
  } else {
    if (s2 > c2) {
      sc = coh * __builtin_amdgcn_rsqf(s2);
      return true;
    }
    return false;
  }
}

// The same test and quotient for a vertex (v) and a cell (xx, yy) at once.  In
// FP64 the library's square root and division take 18 and 11 operations and two
// reciprocals, most of them to bring arguments into range and put back special
// results.  Where coh lies in rm_near's range no argument needs that: s2 > c2
// does not underflow, a finite root and quotient stay normal, and an infinite s2
// (root NaN) gets the factor 0 of coh / infinity.  Then Goldschmidt's iteration
// on the hardware's reciprocal root, with Markstein's final corrections (P.
// Markstein, IBM J. Res. Dev. 34, 1990), gives the root in 10 and the quotient in
// 6 operations, both correctly rounded like the library's (equal on 1.2e10
// arguments over the range), and the vertex's and the cell's chains overlap.
// FP64, every node yielding, us per iteration before and after: 64^2 4.4 -> 4.0,
// 512^2 6.9 -> 6.2 (resident), 1024^2 13.7 -> 12.0, 4096^2 115 -> 103 (chains).
__device__ __forceinline__ bool rm_near(double coh) {
  return coh >= 0x1p-300 && coh <= 0x1p300;
}
__device__ __forceinline__ bool rm_factor(double s2, double coh, double c2, double& sc) {
  const double y = __builtin_amdgcn_rsq(s2);
  double g = s2 * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(__builtin_fma(-g, g, s2), h, g);
  g = __builtin_fma(__builtin_fma(-g, g, s2), h, g);  // sqrt(s2)
  double w = h + h;
  w = __builtin_fma(__builtin_fma(-g, w, 1.0), w, w);  // its reciprocal
  const double q = coh * w;
  sc = __builtin_fmax(__builtin_fma(__builtin_fma(-g, q, coh), w, q), 0.0);
  return s2 > c2 && !(g <= coh);
}
// (SIDE: side by side; else one after the other, in the registers of one)
template <bool SIDE, typename CT>
__device__ __forceinline__ void rm_both(CT s2v, CT s2c, CT coh, CT c2, bool near, CT& v, CT& xx,
                                        CT& yy) {
  CT sc;
  if constexpr (sizeof(CT) == 8) {
    if (__builtin_expect(near, 1)) {
      CT sv;
      const bool yv = rm_factor(s2v, coh, c2, sv);
      v = yv ? v * sv : v;
      if constexpr (!SIDE) __builtin_amdgcn_sched_barrier(0);
      const bool yc = rm_factor(s2c, coh, c2, sc);
      xx = yc ? xx * sc : xx;
      yy = yc ? yy * sc : yy;
      return;
    }
  }
  if (rm_scale(s2v, coh, c2, sc)) v *= sc;
  if (rm_scale(s2c, coh, c2, sc)) {
    xx = xx * sc;
    yy = yy * sc;
  }
}

// The split scheme's FP32 arithmetic.  Every kernel computes these quantities
// through the functions below, so the split kernels agree with each other bit
// for bit.  The terms follow the reference's FP64 expressions
// (EffPlast2D.cu:16-33, 54-75, 109-176), which the FP64 scheme keeps as they
// are; here each product that ends in a sum is fused into it (one rounding
// instead of two, and one instruction fewer).  With residual checks every 500
// iterations, the 1024^2 RVE of three load steps stops at the same checks as
// the FP64 solve in every step, as it does with separate roundings.
//
// trial cell stress from the strain pair: P0 - K (exx + eyy) and
// 2G (e - (exx + eyy) / 3), with g2 = 2G
__device__ __forceinline__ void split_cell_trial(float exx, float eyy, float K, float g2, float P0,
                                                 float& pp, float& txx, float& tyy) {
  const float s = exx + eyy;
  pp = __builtin_fmaf(-K, s, P0);
  txx = g2 * __builtin_fmaf(s, -(1.0f / 3.0f), exx);
  tyy = g2 * __builtin_fmaf(s, -(1.0f / 3.0f), eyy);
}
// trial vertex shear: g (a / dY + b / dX) from the differences a of Ux in y
// and b of Uy in x
__device__ __forceinline__ float split_vertex_trial(float g, float a, float rdY, float b,
                                                   float rdX) {
  return g * __builtin_fmaf(a, rdY, b * rdX);
}
// squared invariants the return mapping tests: vertex, from the four-cell
// sums of the normal stresses; cell, from the four-vertex mean av
__device__ __forceinline__ float split_s2_vertex(float sxx, float syy, float txy) {
  return __builtin_fmaf(0.0625f * sxx, sxx, __builtin_fmaf(0.0625f * syy, syy, 2.0f * txy * txy));
}
__device__ __forceinline__ float split_s2_cell(float txx, float tyy, float av) {
  return __builtin_fmaf(txx, txx, __builtin_fmaf(tyy, tyy, 2.0f * av * av));
}
// damped velocity: v damp + dTrho (a ra + b rb), ra and rb the reciprocal
// grid steps of the two stress differences a and b
__device__ __forceinline__ float split_velocity(float v, float damp, float dTrho, float a,
                                               float ra, float b, float rb) {
  return __builtin_fmaf(v, damp, dTrho * __builtin_fmaf(a, ra, b * rb));
}
// displacement, FP64: u + v dT with one rounding (a fused multiply-add; the
// FP64 scheme keeps the reference's product and sum)
__device__ __forceinline__ double split_disp(double u, float v, double dT) {
  return __builtin_fma((double)v, dT, u);
}

// Workgroup barrier that waits for LDS traffic only: global loads issued
// before it (the next tile's prefetch) stay in flight.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ---------------------------------------------------------------------------
// Row-marching fused iteration.  One wave64 owns a strip of 64 columns
// (lane L <-> column i = s + L) and walks down rows j0-2 .. j1-1 of one RVE.
// Step j loads row j+1 of Ux and the mask, row j+2 of Uy and row j of V, and
// produces, all in registers:
//
//   trial cell row j+1 and trial vertex row j      (ComputeStress, :37-98)
//   return-mapped vertex row j and cell row j       (ComputeJ2 / Plasticity,
//                                                     :100-177)
//   V and U of row j, lanes 2..61                   (ComputeDisp, :3-35)
//
// Neighbours in x come from the adjacent lanes through DPP wave shifts;
// neighbours in y are the rows carried from the previous steps, so nothing
// is staged in LDS and no barrier is needed.  The loads of step j+1 are
// issued before step j computes.  Steps j0-2 and j0-1 only fill the carried
// rows (the halo of the segment); outputs start at row j0.
//
// Every expression is the fused tile kernel's (and so the reference's) in the
// same order: the two kernels give identical results.  EDGE segments (strips
// or rows touching the RVE boundary) keep the boundary conditions, zero the
// stress outside the grid and use the clamped vertex block of the reference's
// ComputeJ2 edge branches for cells on the boundary.

// value of lane L+1 (0 in lane 63) and of lane L-1 (0 in lane 0)
__device__ __forceinline__ int lane_next_i(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x130, 0xf, 0xf, true);  // wave_shl:1, bound_ctrl:0
}
__device__ __forceinline__ int lane_prev_i(int v) {
  return __builtin_amdgcn_mov_dpp(v, 0x138, 0xf, 0xf, true);  // wave_shr:1, bound_ctrl:0
}
__device__ __forceinline__ float lane_next(float v) {
  return __builtin_bit_cast(float, lane_next_i(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float lane_prev(float v) {
  return __builtin_bit_cast(float, lane_prev_i(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_next(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)lane_next_i((int)(unsigned)b);
  const unsigned hi = (unsigned)lane_next_i((int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double lane_prev(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)lane_prev_i((int)(unsigned)b);
  const unsigned hi = (unsigned)lane_prev_i((int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

template <typename CT, typename VT>
struct March {
  static __device__ __forceinline__ CT dx(double a, const RveDev& r) {
    if constexpr (sizeof(CT) == 8) return qdiv(a, r.dX, r.rdX);
    else return (CT)a * (CT)r.rdX;
  }
  static __device__ __forceinline__ CT dy(double a, const RveDev& r) {
    if constexpr (sizeof(CT) == 8) return qdiv(a, r.dY, r.rdY);
    else return (CT)a * (CT)r.rdY;
  }
  static __device__ __forceinline__ CT third(CT a) {
    if constexpr (sizeof(CT) == 8) return qdiv(a, 3.0, 1.0 / 3.0);
    else return a * (CT)(1.0 / 3.0);
  }

  struct Ld {
    double ux, uy;   // Ux row j+1, Uy row j+2
    unsigned m;      // mask row j+1
    VT vx, vy;       // V row j
  };

  template <bool EDGE>
  static __device__ __forceinline__ Ld load(const RveDev& r, const double* __restrict__ Ux,
                                            const double* __restrict__ Uy, const VT* Vx,
                                            const VT* Vy, int i, int j) {
    const int nX = r.nX, nY = r.nY, sx = nX + 1;
    Ld d;
    if (!EDGE) {
      // row bases are uniform (scalar arithmetic), the lane offset i is fixed
      d.ux = gld(Ux + (size_t)(j + 1) * sx, (unsigned)i);
      d.uy = gld(Uy + (size_t)(j + 2) * nX, (unsigned)i);
      d.m = gld(r.mask + (size_t)(j + 1) * nX, (unsigned)i);
      d.vx = gld(Vx + (size_t)j * sx, (unsigned)i);
      d.vy = gld(Vy + (size_t)j * nX, (unsigned)i);
    } else {
      const bool ci = i >= 0 && i < nX;
      d.ux = (i >= 0 && i <= nX && j + 1 >= 0 && j + 1 < nY) ? gld(Ux, (unsigned)((j + 1) * sx + i)) : 0.0;
      d.uy = (ci && j + 2 >= 0 && j + 2 <= nY) ? gld(Uy, (unsigned)((j + 2) * nX + i)) : 0.0;
      d.m = (ci && j + 1 >= 0 && j + 1 < nY) ? (unsigned)gld(r.mask, (unsigned)((j + 1) * nX + i)) : 0u;
      const bool vr = ci && j >= 0 && j < nY;
      d.vx = vr ? gld(Vx, (unsigned)(j * sx + i)) : (VT)0;
      d.vy = vr ? gld(Vy, (unsigned)(j * nX + i)) : (VT)0;
    }
    return d;
  }

  // Return mapping of a vertex from its trial shear stress and the four trial
  // cells around it, summed in the reference's order.
  static __device__ __forceinline__ CT vertex_rm(CT txy, CT sxx, CT syy, CT coh, CT c2lo) {
    CT s2;
    if constexpr (sizeof(CT) == 8)
      s2 = (CT)0.0625 * sxx * sxx + (CT)0.0625 * syy * syy + (CT)2.0 * txy * txy;
    else
      s2 = split_s2_vertex(sxx, syy, txy);
    CT sc;
    if (rm_scale(s2, coh, c2lo, sc)) txy *= sc;
    return txy;
  }
  static __device__ __forceinline__ void cell_rm(CT& txx, CT& tyy, CT av, CT coh, CT c2lo) {
    CT s2;
    if constexpr (sizeof(CT) == 8) s2 = txx * txx + tyy * tyy + (CT)2.0 * av * av;
    else s2 = split_s2_cell(txx, tyy, av);
    CT sc;
    if (rm_scale(s2, coh, c2lo, sc)) {
      txx = txx * sc;
      tyy = tyy * sc;
    }
  }

  template <bool EDGE>
  static __device__ void run(const RveDev& r, int cur, int vpar, int s, int j0, int j1,
                             const CT* gt) {
    const int nX = r.nX, nY = r.nY, sx = nX + 1;
    const int L = threadIdx.x & 63;
    const int i = s + L;
    const double* __restrict__ Uxi = r.Ux[cur];
    const double* __restrict__ Uyi = r.Uy[cur];
    double* __restrict__ Uxo = r.Ux[cur ^ 1];
    double* __restrict__ Uyo = r.Uy[cur ^ 1];
    // V updated in place in the current buffer (Vx2/Vy2 when vpar)
    VT* Vx = static_cast<VT*>(vpar ? r.Vx2 : r.Vx);
    VT* Vy = static_cast<VT*>(vpar ? r.Vy2 : r.Vy);
    const bool plastic = r.plastic != 0;
    const CT coh = (CT)r.coh;
    CT c2lo;
    if constexpr (sizeof(CT) == 8) c2lo = r.coh2lo;
    else c2lo = r.coh2lof;
    const CT K0 = (CT)r.K0, Kp = (CT)r.Kp, G0 = (CT)r.G0, Gp = (CT)r.Gp, P0 = (CT)r.P0;
    const CT vdampX = (CT)r.vdampX, vdampY = (CT)r.vdampY, dTrho = (CT)r.dTrho;
    const double dT = r.dT;
    const bool outLane = L >= 2 && L < 62 && (!EDGE || i < nX);
    const bool colC = !EDGE || (i >= 0 && i < nX);
    const bool colV = !EDGE || (i >= 0 && i < nX - 1);
    const bool leftEdge = EDGE && i == 0, rightEdge = EDGE && i == nX - 1;

    // carried rows (see the step comments below)
    const int jb = j0 - 2;
    double ux_c = 0.0, uy_c = 0.0, uy_n = 0.0;
    unsigned m_c = 0;
    if (!EDGE) {
      ux_c = gld(Uxi, (unsigned)(jb * sx + i));
      uy_n = gld(Uyi, (unsigned)((jb + 1) * nX + i));
      m_c = gld(r.mask, (unsigned)(jb * nX + i));
    } else {
      if (i >= 0 && i <= nX && jb >= 0 && jb < nY) ux_c = gld(Uxi, (unsigned)(jb * sx + i));
      if (colC && jb + 1 >= 0 && jb + 1 <= nY) uy_n = gld(Uyi, (unsigned)((jb + 1) * nX + i));
      if (colC && jb >= 0 && jb < nY) m_c = gld(r.mask, (unsigned)(jb * nX + i));
    }
    double uxs_c = lane_next(ux_c);
    CT tP_c = 0, tXX_c = 0, tYY_c = 0, sXX_c = 0, sYY_c = 0;   // trial cell row j
    CT tP_p = 0, tXX_p = 0, tYY_p = 0;                         // trial cell row j-1 (EDGE)
    CT tXY_p = 0, tXY_pp = 0;                                  // trial vertex rows j-1, j-2
    CT cP_p = 0, cYY_p = 0, cXY_p = 0;                         // corrected row j-1

    // the loads are unconditional (past the last step they re-read rows in
    // range: interior segments end at least one row above nY-1, edge loads
    // are guarded), so no branch joins in front of a wait
    auto fetch = [&](int j) {
      return load<EDGE>(r, Uxi, Uyi, Vx, Vy, i, EDGE ? j : min(j, j1 - 1));
    };
    auto step = [&](const int j, const Ld& ld) {

      // trial cell row j+1 (cell i, row j+1)
      const double ux_n = ld.ux, uy_nn = ld.uy;
      const unsigned m_n = ld.m;
      const double uxs_n = lane_next(ux_n);
      CT tP_n = 0, tXX_n = 0, tYY_n = 0;
      {
        const CT K = (m_n & M_CELL_MAT) ? Kp : K0;
        const CT G = (m_n & M_CELL_MAT) ? Gp : G0;
        const CT exx = dx(uxs_n - ux_n, r);
        const CT eyy = dy(uy_nn - uy_n, r);
        CT pp, txx, tyy;
        if constexpr (sizeof(CT) == 8) {
          pp = P0 - K * (exx + eyy);
          txx = (CT)2.0 * G * (exx - third(exx + eyy));
          tyy = (CT)2.0 * G * (eyy - third(exx + eyy));
        } else {
          split_cell_trial(exx, eyy, K, (CT)2.0 * G, P0, pp, txx, tyy);
        }
        const bool ok = !EDGE || (colC && j + 1 >= 0 && j + 1 < nY);
        if ((m_n & M_CELL_ZERO) || !ok) {
          pp = 0;
          txx = 0;
          tyy = 0;
        }
        tP_n = pp;
        tXX_n = txx;
        tYY_n = tyy;
      }
      const CT sXX_n = lane_next(tXX_n), sYY_n = lane_next(tYY_n);

      // trial vertex row j (vertex i, row j)
      const double uys_n = lane_next(uy_n);
      CT tXY_c;
      {
        const CT g = gt[(m_c >> M_VCLASS_SHIFT) & 15];
        CT txy;
        if constexpr (sizeof(CT) == 8) txy = g * (dy(uxs_n - uxs_c, r) + dx(uys_n - uy_n, r));
        else txy = split_vertex_trial(g, (CT)(uxs_n - uxs_c), (CT)r.rdY, (CT)(uys_n - uy_n),
                                      (CT)r.rdX);
        const bool ok = !EDGE || (colV && j >= 0 && j < nY - 1);
        if ((m_c & M_VERT_ZERO) || !ok) txy = 0;
        tXY_c = txy;
      }

      // return mapping: vertex row j, cell row j (and, on the top boundary,
      // cell row 0 once vertex row 1 exists)
      CT cXY_c = tXY_c, cP_c = tP_c, cXX_c = tXX_c, cYY_c = tYY_c;
      if (plastic) {
        const bool vok = !EDGE || (colV && j >= 0 && j < nY - 1);
        const CT sxx = tXX_c + sXX_c + tXX_n + sXX_n;
        const CT syy = tYY_c + sYY_c + tYY_n + sYY_n;
        if (vok) cXY_c = vertex_rm(tXY_c, sxx, syy, coh, c2lo);

        const CT pr_p = lane_prev(tXY_p), pr_c = lane_prev(tXY_c);
        if (!EDGE) {
          const CT av = (CT)0.25 * (pr_p + tXY_p + pr_c + tXY_c);
          cell_rm(cXX_c, cYY_c, av, coh, c2lo);
        } else {
          // vertex pair of this lane's cell in a vertex row: (first, second)
          const CT nx_p = lane_next(tXY_p), nx_c = lane_next(tXY_c), nx_pp = lane_next(tXY_pp);
          const CT pr_pp = lane_prev(tXY_pp);
          const CT pp_p = lane_prev(pr_p), pp_c = lane_prev(pr_c), pp_pp = lane_prev(pr_pp);
          auto first = [&](CT t, CT pr, CT pp) { return leftEdge ? t : (rightEdge ? pp : pr); };
          auto second = [&](CT t, CT pr, CT nxv) { return leftEdge ? nxv : (rightEdge ? pr : t); };
          if (colC && j >= 1 && j < nY - 1) {
            const CT av = (CT)0.25 * (first(tXY_p, pr_p, pp_p) + second(tXY_p, pr_p, nx_p) +
                                      first(tXY_c, pr_c, pp_c) + second(tXY_c, pr_c, nx_c));
            cell_rm(cXX_c, cYY_c, av, coh, c2lo);
          } else if (colC && j == nY - 1 && j >= 1) {  // rows nY-3, nY-2
            const CT av = (CT)0.25 * (first(tXY_pp, pr_pp, pp_pp) + second(tXY_pp, pr_pp, nx_pp) +
                                      first(tXY_p, pr_p, pp_p) + second(tXY_p, pr_p, nx_p));
            cell_rm(cXX_c, cYY_c, av, coh, c2lo);
          }
          if (j == 1) {  // cell row 0 from vertex rows 0 and 1
            CT xx = tXX_p, yy = tYY_p;
            if (colC) {
              const CT av = (CT)0.25 * (first(tXY_p, pr_p, pp_p) + second(tXY_p, pr_p, nx_p) +
                                        first(tXY_c, pr_c, pp_c) + second(tXY_c, pr_c, nx_c));
              cell_rm(xx, yy, av, coh, c2lo);
            }
            cP_p = tP_p;
            cYY_p = yy;
          }
        }
      }

      // velocity and displacement of row j
      const CT rP = lane_prev(cP_c), rXX = lane_prev(cXX_c);
      const CT rXY_c = lane_prev(cXY_c), rXY_p = lane_prev(cXY_p);
      if (j >= j0) {
        CT vx = (CT)ld.vx, vy = (CT)ld.vy;
        if (!EDGE || (i > 0 && j > 0 && j < nY - 1)) {
          if constexpr (sizeof(CT) == 8)
            vx = vx * vdampX + dTrho * (dx(-cP_c + rP + cXX_c - rXX, r) + dy(rXY_c - rXY_p, r));
          else
            vx = split_velocity(vx, vdampX, dTrho, -cP_c + rP + cXX_c - rXX, (CT)r.rdX,
                                rXY_c - rXY_p, (CT)r.rdY);
          if (outLane) gst(Vx + (size_t)j * sx, (unsigned)i, (VT)vx);
        }
        if (!EDGE || (i > 0 && i < nX - 1 && j > 0)) {
          if constexpr (sizeof(CT) == 8)
            vy = vy * vdampY + dTrho * (dy(-cP_c + cP_p + cYY_c - cYY_p, r) + dx(cXY_p - rXY_p, r));
          else
            vy = split_velocity(vy, vdampY, dTrho, -cP_c + cP_p + cYY_c - cYY_p, (CT)r.rdY,
                                cXY_p - rXY_p, (CT)r.rdX);
          if (outLane) gst(Vy + (size_t)j * nX, (unsigned)i, (VT)vy);
        }
        if (outLane && (!EDGE || j < nY)) {
          if constexpr (sizeof(CT) == 8) {
            gst(Uxo + (size_t)j * sx, (unsigned)i, ux_c + (double)vx * dT);
            gst(Uyo + (size_t)j * nX, (unsigned)i, uy_c + (double)vy * dT);
          } else {
            gst(Uxo + (size_t)j * sx, (unsigned)i, split_disp(ux_c, vx, dT));
            gst(Uyo + (size_t)j * nX, (unsigned)i, split_disp(uy_c, vy, dT));
          }
          if (EDGE) {
            if (i == nX - 1) gst(Uxo, (unsigned)(j * sx + i + 1), uxs_c);
            if (j == nY - 1) gst(Uyo, (unsigned)((j + 1) * nX + i), uy_n);
          }
        }
      }

      // rotate
      ux_c = ux_n;
      uxs_c = uxs_n;
      uy_c = uy_n;
      uy_n = uy_nn;
      m_c = m_n;
      tP_p = tP_c;
      tXX_p = tXX_c;
      tYY_p = tYY_c;
      tP_c = tP_n;
      tXX_c = tXX_n;
      tYY_c = tYY_n;
      sXX_c = sXX_n;
      sYY_c = sYY_n;
      tXY_pp = tXY_p;
      tXY_p = tXY_c;
      cP_p = cP_c;
      cYY_p = cYY_c;
      cXY_p = cXY_c;
    };
    // loads run one step ahead of the arithmetic: the wait for a step's rows
    // leaves the next step's loads in flight
    // (two steps per trip, each buffer refilled right after the step that
    // reads it, so no register copy has to wait for a load)
    Ld A = fetch(jb);
    for (int j = jb; j < j1; j += 2) {
      const Ld B = fetch(j + 1);
      step(j, A);
      if (j + 1 >= j1) break;
      A = fetch(j + 2);
      step(j + 1, B);
    }
  }
};

// ---------------------------------------------------------------------------
// Two iterations per launch (temporal blocking of the row-marching kernel).
// One iteration is written as a row stream (MarchStage): step j takes row j+1
// of Ux and the mask, row j+2 of Uy and row j of V of its input state and
// gives row j of its output state -- V, and U at every node of the row
// (updated where ComputeDisp updates it, unchanged where it does not, zero
// outside the grid) -- so a second stage can take it as input.  In k_march2
// stage A reads the state from HBM and stage B, two rows behind, reads A's
// rows from registers; only B's rows are written.  U and V are read from one
// buffer and written to the other (a neighbouring segment's halo needs the
// old velocities).  Valid outputs shrink by two lanes per stage: lanes 4..59,
// strips of 56 columns.  The arithmetic of each stage is the single-iteration
// kernels', so two stages give the same bits as two launches.
//
// EX stages run on strips that touch the left or right boundary (per-column
// tests), EY stages on segments whose rows reach the top or bottom boundary
// (per-row tests, uniform over the wave); EDGE is either.  CLEAN stages
// (segments whose mask bytes are all 0, chain kernels) read no mask: matrix
// K and G, no pore zeroing and the vertex modulus of four matrix cells, which
// is what the mask path computes from zero mask bytes.
//
// PL 1 or 0 fixes whether the RVE is plastic (interior segments: a step is one
// block of code up to the scaling); -1 reads it from the RVE.
// The vertex moduli by class in LDS, eight bytes apart: the class bits of a mask
// byte are the byte offset of its entry.
template <typename CT>
struct alignas(8) VertMod {
  CT g;
};
template <typename CT>
__device__ __forceinline__ CT vert_mod(const VertMod<CT>* gt, unsigned m) {
  static_assert(M_VCLASS_SHIFT == 3 && sizeof(VertMod<CT>) == 8, "class bits as a byte offset");
  return reinterpret_cast<const VertMod<CT>*>(reinterpret_cast<const char*>(gt) + (m & 0x78u))->g;
}

// Stages take the mask byte with its two zero bits inverted (1: the trial stress
// stays), so that each bit, widened to a word, selects with one instruction
// per 32 bits and without a compare.  (In assembly: the compiler would turn the
// widened bit back into arithmetic.)
__device__ __forceinline__ unsigned stage_mask(unsigned m) {
  return m ^ (unsigned)(M_CELL_ZERO | M_VERT_ZERO);
}
template <int BIT>
__device__ __forceinline__ unsigned mask_word(unsigned m) {
  unsigned w;
  asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(w) : "v"(m), "n"(__builtin_ctz(BIT)));
  return w;
}
template <typename CT>
__device__ __forceinline__ CT keep(unsigned w, CT a) {  // a, or 0 where w is 0
  if constexpr (sizeof(CT) == 4) {
    return __builtin_bit_cast(float, w & __builtin_bit_cast(unsigned, a));
  } else {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, a);
    return __builtin_bit_cast(double, (unsigned long long)(w & (unsigned)(b >> 32)) << 32 |
                                          (w & (unsigned)b));
  }
}
template <typename CT>
__device__ __forceinline__ CT pick(unsigned w, CT yes, CT no) {
  if constexpr (sizeof(CT) == 4) {
    const unsigned a = __builtin_bit_cast(unsigned, yes), b = __builtin_bit_cast(unsigned, no);
    return __builtin_bit_cast(float, (w & a) | (~w & b));
  } else {
    const unsigned long long a = __builtin_bit_cast(unsigned long long, yes),
                             b = __builtin_bit_cast(unsigned long long, no);
    const unsigned lo = (w & (unsigned)a) | (~w & (unsigned)b);
    const unsigned hi = (w & (unsigned)(a >> 32)) | (~w & (unsigned)(b >> 32));
    return __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
  }
}

template <typename CT, typename VT, bool EX, bool EY = EX, bool CLEAN = false, int PL = -1>
struct MarchStage {
  static constexpr bool EDGE = EX || EY;
  using M = March<CT, VT>;
  const RveDev* r;
  const VertMod<CT>* gt;
  int nX, nY, i;
  bool colC, colV, leftEdge, rightEdge, plastic, near;
  CT coh, c2lo, K0, Kp, G2_0, G2_p, P0, vdampX, vdampY, dTrho, g0;
  double dT;
  // grid steps held in registers: the stores of a step may alias the RVE
  // table, so values read from it would be read again after every store
  double dXd, dYd, rdXd, rdYd;
  CT rdXc, rdYc;
  // carried rows: U rows j and j+1, mask row j, trial cells j (and j-1) and
  // their sums with the right neighbours, the sums of vertex row j-1 and of its
  // 2x2 blocks, corrected row j-1 and the left neighbours of its shear.  The
  // sums stand where the invariants' expressions begin, so a neighbour's value
  // is needed in the step that computes it only (a lane shift there is an
  // operand of the addition) and the trial stresses end with their step (the
  // return mapping scales them in place).
  double ux_c, uxs_c, uy_c, uy_n;
  unsigned m_c;
  CT tP_c, tXX_c, tYY_c, hXX_c, hYY_c, tP_p, tXX_p, tYY_p, hXY_p, nXY_p, cP_p, cYY_p, cXY_p,
      rXY_p;

  struct Out {
    double ux, uy;   // output U of row j at this lane's column
    CT vx, vy;       // output V of row j (rounded to the storage type)
    bool updX, updY; // V was updated here (else it is the input)
  };

  // a coefficient in the arithmetic type.  Rounded to FP32 by the vector ALU,
  // it is moved back to a scalar register: the dozen of them would take a
  // vector register each
  static __device__ __forceinline__ CT uni(double a) {
    if constexpr (sizeof(CT) == 8) return a;
    else
      return __builtin_bit_cast(
          float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)a)));
  }

  __device__ __forceinline__ void setup(const RveDev& rr, const VertMod<CT>* g, int col) {
    r = &rr;
    gt = g;
    nX = rr.nX;
    nY = rr.nY;
    i = col;
    colC = !EX || (i >= 0 && i < nX);
    colV = !EX || (i >= 0 && i < nX - 1);
    leftEdge = EX && i == 0;
    rightEdge = EX && i == nX - 1;
    plastic = rr.plastic != 0;
    coh = uni(rr.coh);
    near = rm_near(rr.coh);
    if constexpr (sizeof(CT) == 8) c2lo = rr.coh2lo;
    else c2lo = rr.coh2lof;
    K0 = uni(rr.K0);
    Kp = uni(rr.Kp);
    G2_0 = uni(2.0 * rr.G0);  // 2G, exact
    g0 = uni(rr.gtab[0]);
    G2_p = uni(2.0 * rr.Gp);
    P0 = uni(rr.P0);
    dXd = rr.dX;
    dYd = rr.dY;
    rdXd = rr.rdX;
    rdYd = rr.rdY;
    rdXc = uni(rr.rdX);
    rdYc = uni(rr.rdY);
    vdampX = uni(rr.vdampX);
    vdampY = uni(rr.vdampY);
    dTrho = uni(rr.dTrho);
    dT = rr.dT;
  }

  // difference quotients: March::dx / March::dy with the steps in registers
  __device__ __forceinline__ CT dxs(double a) const {
    if constexpr (sizeof(CT) == 8) return qdiv(a, dXd, rdXd);
    else return (CT)a * rdXc;
  }
  __device__ __forceinline__ CT dys(double a) const {
    if constexpr (sizeof(CT) == 8) return qdiv(a, dYd, rdYd);
    else return (CT)a * rdYc;
  }

  // Ux row jb, Uy row jb+1, mask row jb (jb = first step)
  __device__ __forceinline__ void start(double ux, double uy1, unsigned m) {
    startS(ux, lane_next(ux), uy1, m);
  }
  // the same with Ux(i+1, jb) given (read from a ring row instead of shifted)
  __device__ __forceinline__ void startS(double ux, double uxs, double uy1, unsigned m) {
    ux_c = ux;
    uxs_c = uxs;
    uy_c = 0.0;
    uy_n = uy1;
    m_c = m;
    tP_c = tXX_c = tYY_c = hXX_c = hYY_c = 0;
    tP_p = tXX_p = tYY_p = 0;
    hXY_p = nXY_p = 0;
    cP_p = cYY_p = cXY_p = rXY_p = 0;
  }

  // FP32: the addition stays in the block of its shifted operand
  static __device__ __forceinline__ CT here(CT a) {
    if constexpr (sizeof(CT) == 4 && PL == 1) asm volatile("" : "+v"(a));
    return a;
  }

  __device__ __forceinline__ Out step(const int j, const double ux_n, const double uy_nn,
                                      const unsigned m_n, const CT vx_in, const CT vy_in) {
    return stepS(j, ux_n, lane_next(ux_n), lane_next(uy_n), uy_nn, m_n, vx_in, vy_in);
  }
  // the step with the right neighbours uxs_n = Ux(i+1, j+1) and uys_n =
  // Uy(i+1, j+1) given: a stage reading its rows from an LDS ring reads them
  // at the next position instead of shifting lanes (the same values in every
  // lane but the last, whose outputs no stage uses)
  __device__ __forceinline__ Out stepS(const int j, const double ux_n, const double uxs_n,
                                       const double uys_n, const double uy_nn,
                                       const unsigned m_n, const CT vx_in, const CT vy_in) {
    // trial cell row j+1
    CT tP_n, tXX_n, tYY_n;
    {
      CT K = K0, G2 = G2_0;
      if constexpr (!CLEAN) {
        const unsigned w = mask_word<M_CELL_MAT>(m_n);
        K = pick(w, Kp, K0);
        G2 = pick(w, G2_p, G2_0);
      }
      const CT exx = dxs(uxs_n - ux_n);
      const CT eyy = dys(uy_nn - uy_n);
      CT pp, txx, tyy;
      if constexpr (sizeof(CT) == 8) {
        pp = P0 - K * (exx + eyy);
        txx = G2 * (exx - M::third(exx + eyy));
        tyy = G2 * (eyy - M::third(exx + eyy));
      } else {
        split_cell_trial(exx, eyy, K, G2, P0, pp, txx, tyy);
      }
      if constexpr (!CLEAN) {
        const unsigned w = mask_word<M_CELL_ZERO>(m_n);
        pp = keep(w, pp);
        txx = keep(w, txx);
        tyy = keep(w, tyy);
      }
      tP_n = pp;
      tXX_n = txx;
      tYY_n = tyy;
    }
    const CT sXX_n = lane_next(tXX_n), sYY_n = lane_next(tYY_n);
    const CT hXX_n = here(tXX_n + sXX_n), hYY_n = here(tYY_n + sYY_n);
    const CT sxx = hXX_c + tXX_n + sXX_n, syy = hYY_c + tYY_n + sYY_n;  // vertex row j
    // trial vertex row j
    CT tXY_c;
    {
      const CT g = CLEAN ? g0 : vert_mod(gt, m_c);
      CT txy;
      if constexpr (sizeof(CT) == 8) txy = g * (dys(uxs_n - uxs_c) + dxs(uys_n - uy_n));
      else txy = split_vertex_trial(g, (CT)(uxs_n - uxs_c), rdYc, (CT)(uys_n - uy_n), rdXc);
      if constexpr (!CLEAN) txy = keep(mask_word<M_VERT_ZERO>(m_c), txy);
      tXY_c = txy;
    }
    // the vertex row's values in the block of this lane's cell (columns 0 and
    // nX-1: of the two columns next to the edge), and the block's sum
    const CT pr_c = lane_prev(tXY_c);
    CT f_c = pr_c, t_c = tXY_c;
    if constexpr (EX) {
      const CT nx = lane_next(tXY_c), pp = lane_prev(pr_c);
      f_c = leftEdge ? tXY_c : rightEdge ? pp : pr_c;
      t_c = leftEdge ? nx : rightEdge ? pr_c : tXY_c;
    }
    const CT hXY_c = here(f_c + t_c);
    const CT n_c = hXY_p + f_c + t_c;
    // return mapping
    CT cXY_c = tXY_c, cP_c = tP_c, cXX_c = tXX_c, cYY_c = tYY_c;
    const bool pl = PL < 0 ? plastic : PL != 0;
    if (pl) {
      // the squared invariants decide; the scaling is skipped where no lane of
      // the wave yields (stresses outside the grid do not count)
      CT s2v, s2c, n = n_c;
      if (EY && j == nY - 1) n = nXY_p;  // the two vertex rows above row nY-1
      const CT av = (CT)0.25 * n;
      if constexpr (sizeof(CT) == 8) {
        s2v = (CT)0.0625 * sxx * sxx + (CT)0.0625 * syy * syy + (CT)2.0 * tXY_c * tXY_c;
        s2c = cXX_c * cXX_c + cYY_c * cYY_c + (CT)2.0 * av * av;
      } else {
        s2v = split_s2_vertex(sxx, syy, tXY_c);
        s2c = split_s2_cell(cXX_c, cYY_c, av);
      }
      if (__any((s2v > c2lo && (!EX || colV)) || (s2c > c2lo && (!EX || colC)))) {
        rm_both<false>(s2v, s2c, coh, c2lo, near, cXY_c, cXX_c, cYY_c);
      }
      if (EY && j == 1) {
        // cell row 0, from vertex rows 0 and 1 (its own step did not have them)
        CT xx = tXX_p, yy = tYY_p;
        M::cell_rm(xx, yy, (CT)0.25 * n_c, coh, c2lo);
        cYY_p = yy;
      }
    }
    // velocity and displacement of row j
    const CT rP = lane_prev(cP_c), rXX = lane_prev(cXX_c);
    // FP32 takes the left neighbours' difference as the shifted difference (the
    // same value), the shift an operand of what follows; FP64, whose shifts
    // are two moves each, carries them to the next step
    CT dXY, rXY_c = 0;
    if constexpr (sizeof(CT) == 8) {
      rXY_c = lane_prev(cXY_c);
      dXY = rXY_c - rXY_p;
    } else {
      dXY = lane_prev(cXY_c - cXY_p);
      rXY_p = lane_prev(cXY_p);
    }
    Out o;
    CT vx = vx_in, vy = vy_in;
    o.updX = (!EX || (i > 0 && i < nX)) && (!EY || (j > 0 && j < nY - 1));
    o.updY = (!EX || (i > 0 && i < nX - 1)) && (!EY || (j > 0 && j < nY));
    if constexpr (sizeof(CT) == 8) {
      // U advances with the velocity before its rounding to the storage type
      // (as the tile and march kernels do); the next stage gets the stored value
      if (o.updX)
        vx = vx * vdampX + dTrho * (dxs(-cP_c + rP + cXX_c - rXX) + dys(dXY));
      if (o.updY)
        vy = vy * vdampY + dTrho * (dys(-cP_c + cP_p + cYY_c - cYY_p) + dxs(cXY_p - rXY_p));
    } else {
      if (o.updX)
        vx = (CT)(VT)split_velocity(vx, vdampX, dTrho, -cP_c + rP + cXX_c - rXX, rdXc,
                                    dXY, rdYc);
      if (o.updY)
        vy = (CT)(VT)split_velocity(vy, vdampY, dTrho, -cP_c + cP_p + cYY_c - cYY_p, rdYc,
                                    cXY_p - rXY_p, rdXc);
    }
    o.vx = (CT)(VT)vx;
    o.vy = (CT)(VT)vy;
    if constexpr (sizeof(CT) == 8) {
      o.ux = ux_c + (double)vx * dT;
      o.uy = uy_c + (double)vy * dT;
    } else {
      o.ux = split_disp(ux_c, vx, dT);
      o.uy = split_disp(uy_c, vy, dT);
    }
    // Ux column nX and Uy row nY are never updated
    if ((EX && i >= nX) || (EY && j >= nY)) o.ux = ux_c;
    if (EY && j >= nY) o.uy = uy_c;
    // rotate
    ux_c = ux_n;
    uxs_c = uxs_n;
    uy_c = uy_n;
    uy_n = uy_nn;
    m_c = m_n;
    tP_p = tP_c;
    tXX_p = tXX_c;
    tYY_p = tYY_c;
    tP_c = tP_n;
    tXX_c = tXX_n;
    tYY_c = tYY_n;
    hXX_c = hXX_n;
    hYY_c = hYY_n;
    hXY_p = hXY_c;
    nXY_p = n_c;
    cP_p = cP_c;
    cYY_p = cYY_c;
    cXY_p = cXY_c;
    rXY_p = rXY_c;
    return o;
  }
};

// Stage A's inputs in a two-iteration segment: the first rows (start) and,
// for step t, Ux row t+1, Uy row t+2, mask row t+1 and V row t of the state in
// HBM, through buffer resources (the lane's byte offset fixed, the row's in an
// SGPR).  Interior segments clamp rows to the segment's last step tEnd.  Edge
// segments bound each resource to its field: lanes outside the field's
// columns carry the offset kOob, and a row outside the field reads through a
// resource of bound 0, so every such load returns 0 without a branch.
template <typename CT, typename VT, bool EX, bool EY = EX, bool CLEAN = false>
struct StageInput {
  static constexpr bool EDGE = EX || EY;
  using Ld = typename March<CT, VT>::Ld;
  const double* Uxi;
  const double* Uyi;
  const VT* Vxi;
  const VT* Vyi;
  const unsigned char* mask;
  int nX, nY, sx, i, tEnd;
  unsigned o8, oV;
  __amdgpu_buffer_rsrc_t bUx, bUy, bVx, bVy, bM;
  // edge segments: lane offsets with the column test folded in (Ux columns
  // 0..nX, the others 0..nX-1; V is read for columns 0..nX-1 only)
  unsigned oUx, oC8, oM, oVc;

  __device__ __forceinline__ StageInput(const RveDev& r, int cur, int vpar, int col, int tEnd_)
      : Uxi(r.Ux[cur]), Uyi(r.Uy[cur]),
        Vxi(static_cast<const VT*>(vpar ? r.Vx2 : r.Vx)),
        Vyi(static_cast<const VT*>(vpar ? r.Vy2 : r.Vy)), mask(r.mask), nX(r.nX), nY(r.nY),
        sx(r.nX + 1), i(col), tEnd(tEnd_), o8((unsigned)col * 8u),
        oV((unsigned)col * (unsigned)sizeof(VT)) {
    if (!EDGE) {
      bUx = brsrc(Uxi);
      bUy = brsrc(Uyi);
      bVx = brsrc(Vxi);
      bVy = brsrc(Vyi);
      bM = brsrc(mask);
    } else {
      const unsigned ux = (unsigned)nY * (unsigned)sx, uy = (unsigned)(nY + 1) * (unsigned)nX;
      bUx = brsrc_n(Uxi, ux * 8u);
      bUy = brsrc_n(Uyi, uy * 8u);
      bVx = brsrc_n(Vxi, ux * (unsigned)sizeof(VT));
      bVy = brsrc_n(Vyi, uy * (unsigned)sizeof(VT));
      bM = brsrc_n(mask, (unsigned)nY * (unsigned)nX);
      const bool cx = col >= 0 && col <= nX, cc = col >= 0 && col < nX;
      oUx = cx ? o8 : kOob;
      oC8 = cc ? o8 : kOob;
      oM = cc ? (unsigned)col : kOob;
      oVc = cc ? oV : kOob;
    }
  }

  // Ux row jb, Uy row jb+1, mask row jb into the stage
  template <int PL>
  __device__ __forceinline__ void start(MarchStage<CT, VT, EX, EY, CLEAN, PL>& st, int jb) const {
    double ux = 0.0, uy = 0.0;
    unsigned m = 0;
    const bool colC = !EDGE || (i >= 0 && i < nX);
    if (!EDGE) {
      ux = gld(Uxi, (unsigned)(jb * sx + i));
      uy = gld(Uyi, (unsigned)((jb + 1) * nX + i));
      if (!CLEAN) m = gld(mask, (unsigned)(jb * nX + i));
    } else {
      if (i >= 0 && i <= nX && jb >= 0 && jb < nY) ux = gld(Uxi, (unsigned)(jb * sx + i));
      if (colC && jb + 1 >= 0 && jb + 1 <= nY) uy = gld(Uyi, (unsigned)((jb + 1) * nX + i));
      if (!CLEAN && colC && jb >= 0 && jb < nY) m = gld(mask, (unsigned)(jb * nX + i));
    }
    st.start(ux, uy, stage_mask(m));
  }

  __device__ __forceinline__ Ld fetch(int t0) const {
    const int t = EDGE ? t0 : min(t0, tEnd);
    Ld d;
    if (!EDGE) {
      d.ux = bld<double>(bUx, o8, (unsigned)(t + 1) * (unsigned)sx * 8u);
      d.uy = bld<double>(bUy, o8, (unsigned)(t + 2) * (unsigned)nX * 8u);
      d.m = CLEAN ? 0u : bld<unsigned char>(bM, (unsigned)i, (unsigned)(t + 1) * (unsigned)nX);
      d.vx = bld<VT>(bVx, oV, (unsigned)t * (unsigned)sx * (unsigned)sizeof(VT));
      d.vy = bld<VT>(bVy, oV, (unsigned)t * (unsigned)nX * (unsigned)sizeof(VT));
    } else {
      // rows outside a field read through a resource of bound 0 (the row
      // tests are uniform: scalar selects); the row offset is then 0
      const __amdgpu_buffer_rsrc_t none = brsrc_n(Uxi, 0u);
      const bool r1 = t + 1 >= 0 && t + 1 < nY, r2 = t + 2 >= 0 && t + 2 <= nY,
                 r0 = t >= 0 && t < nY;
      const unsigned s1 = r1 ? (unsigned)(t + 1) : 0u, s2 = r2 ? (unsigned)(t + 2) : 0u,
                     s0 = r0 ? (unsigned)t : 0u;
      d.ux = bld<double>(r1 ? bUx : none, oUx, s1 * (unsigned)sx * 8u);
      d.uy = bld<double>(r2 ? bUy : none, oC8, s2 * (unsigned)nX * 8u);
      d.m = CLEAN ? 0u : bld<unsigned char>(r1 ? bM : none, oM, s1 * (unsigned)nX);
      d.vx = bld<VT>(r0 ? bVx : none, oVc, s0 * (unsigned)sx * (unsigned)sizeof(VT));
      d.vy = bld<VT>(r0 ? bVy : none, oVc, s0 * (unsigned)nX * (unsigned)sizeof(VT));
    }
    return d;
  }
};

// Whether the mask is 0 over rows [jlo, jhi] and columns [ilo, ihi] (clipped
// to the grid), from the block map; the same answer in every lane.
__device__ __forceinline__ bool mask_clear(const RveDev& r, int ilo, int ihi, int jlo, int jhi) {
  ilo = max(ilo, 0);
  jlo = max(jlo, 0);
  ihi = min(ihi, r.nX - 1);
  jhi = min(jhi, r.nY - 1);
  if (ilo > ihi || jlo > jhi) return true;
  const int bx0 = ilo / kMapCols, bx1 = ihi / kMapCols;
  const int by0 = jlo / kMapRows, by1 = jhi / kMapRows;
  const int nbx = (r.nX + kMapCols - 1) / kMapCols;
  const int w = bx1 - bx0 + 1, n = w * (by1 - by0 + 1);
  unsigned any = 0;
  for (int q = (int)(threadIdx.x & 63); q < n; q += 64)
    any |= r.mmap[(by0 + q / w) * nbx + bx0 + q % w];
  return !__any(any != 0);
}

}  // namespace

}  // namespace ep2d
