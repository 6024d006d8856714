// ep2d_resident.hip -- a run of iterations with the RVE resident on the chip.
//
// The GPU's registers hold what the other kernels stream through HBM: each
// workgroup of up to eight waves keeps U and V of one tile of an RVE in
// registers for n iterations.  An iteration reads and writes no field and needs
// no launch.  What bounds it: the dependent chain of a wave's instructions at two
// waves to a SIMD, and the exchange between tiles -- a store reaches the
// memory both XCDs see in about 0.5 us and is read from there in about 1 us --
// which is why a tile computes T = 2 iterations between exchanges, on a halo
// of 2T nodes that it takes over from its neighbours.
//
// us per iteration, single RVE (tile kernel, one iteration a launch, before there
// were resident runs; chain kernels; here):
//            64^2             256^2            333^2            512^2
//   FP64     7.5 / 4.8 / 3.9  6.8 / 5.4 / 3.9  7.3 / 5.8 / 4.1  8.9 / 6.7 / 6.1
//   split    6.8 / 3.1 / 2.6  6.0 / 3.3 / 2.6  6.5 / 3.9 / 3.1  7.2 / 4.1 / 3.9
// One exchange an iteration (T = 1) on the same tiles: FP64 4.15, 4.5 and 4.6,
// split 3.25, 3.6 and 3.8 at 64^2, 256^2 and 333^2.
// The vector ALUs are busy 3% of the cycles at 64^2 (16 tiles), 33% at 333^2 in
// split, 43% (FP64) and 36% (split) at 512^2 with a tile on nearly every CU; waves
// wait half their life.
//
// Layout.  Lane L of every wave is column s+L of the tile's region, wave v
// holds rows jr + v R .. jr + v R + R - 1 of it: the tile's own nodes and 2T
// more on each side that has a neighbour.  Nodes of the halo are computed like
// own ones; after T iterations they are spoilt up to the own nodes and replaced.
// A wave works on its rows as arrays (ResRows): the chain kernels' expressions
// in their order, so the results are those kernels' bit for bit.  The rows
// above and below a wave's come from the neighbouring waves through LDS.
//
// Exchange.  A value travels in a 128-bit word of its two halves, each beside
// the exchange's tag, at agent scope: a half that carries the tag carries the
// value, so no flag, fence or order between words is needed.  Tags grow from
// launch to launch, so a word left over from an earlier one never matches.
// Words alternate between two halves of the buffer: a tile writes exchange
// k+1's words after every neighbour, the diagonal ones too, has published k,
// hence read k-1's (all its waves: a barrier stands between).
//
// Every wait ends.  A tile waits for its neighbours, so all tiles of a launch
// must run at once, and no tile starts before all have arrived.  The first
// workgroup of a launch to run counts its tiles among those in flight on the
// device and goes on only if all of them find their places together
// (resident_fits): tiles of the split two-row shape take half a CU's registers
// (118 a lane at eight waves), the others (146 to 204) a CU each.  The host does
// not launch what it knows to find no room (DeviceRoom).  Other work on the
// device gives its places up as it ends.  If there is no room, or the tiles have
// not all arrived within a quarter second (another process holds the GPU, or
// work this library does not know of), the launch ends without having changed
// anything and says so, those queued behind it do the same, and the caller takes
// the other kernels; until then the tiles that have arrived hold their places.
// Waits inside the run are bounded too.
#include "ep2d_internal.h"
#include "ep2d_march.h"

#include <hip/hip_ext.h>

namespace ep2d {

namespace {

// resident tiles in flight on this device: half-CU ones in the low 16 bits,
// whole ones above
__device__ unsigned g_resInUse;

__device__ __forceinline__ unsigned ald(unsigned* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned aadd(unsigned* p, unsigned v) {
  return __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned acas(unsigned* p, unsigned from, unsigned to) {
  __hip_atomic_compare_exchange_strong(p, &from, to, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                       __HIP_MEMORY_SCOPE_AGENT);
  return from;  // the value before
}

// Arrival of one workgroup (its first thread): the state all of them see.  The
// first to arrive decides: it counts the tiles in, waits for the others and
// lets the run go, or ends it.  (The others' bound is longer: it only serves
// if the first never decides.)
__device__ unsigned res_arrive(ResCtl* c, unsigned tiles, unsigned ticks, unsigned need,
                               unsigned cus) {
  const unsigned long long t0 = wall_clock64();
  if (aadd(&c->arrive, 1u) == 0) {
    const unsigned use = aadd(&g_resInUse, need) + need;
    unsigned how = ald(&c->failed) != 0u ? kResAfter
                   : !resident_fits(cus, use & 0xffffu, use >> 16) ? kResNoRoom
                   : ticks ? kResGo : kResLate;
    while (how == kResGo && ald(&c->arrive) < tiles) {
      if (wall_clock64() - t0 > ticks) how = kResLate;
      __builtin_amdgcn_s_sleep(1);
    }
    const unsigned was = acas(&c->state, 0u, how);
    return was != 0u ? was : how;
  }
  for (;;) {
    const unsigned s = ald(&c->state);
    if (s != 0u) return s;
    if (wall_clock64() - t0 > 4ull * ticks) {
      const unsigned was = acas(&c->state, 0u, kResLate);
      return was != 0u ? was : kResLate;
    }
    __builtin_amdgcn_s_sleep(1);
  }
}

// Departure: the last workgroup counts the tiles out (also those of a launch that
// did not run), clears the record for the next launch and tells the host how
// this one went.
__device__ void res_depart(ResCtl* c, unsigned tiles, unsigned need, unsigned run,
                           unsigned* told) {
  __builtin_amdgcn_s_waitcnt(0);
  if (aadd(&c->depart, 1u) + 1 != tiles) return;
  const unsigned s = ald(&c->state);
  aadd(&g_resInUse, 0u - need);
  __hip_atomic_store(&c->arrive, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&c->depart, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(&c->state, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (s == kResGo) {
    __hip_atomic_store(told, run, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  } else if (s != kResAfter) {
    __hip_atomic_store(&c->failed, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(told + 1, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// The exchange buffer is read and written through a buffer resource, past the
// L2 of one XCD (agent scope): two words of 64 bits at a time, an address of
// one vector register (the node's) and one scalar register (the value's).
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
constexpr int kAgent = 16;                       // sc1
constexpr int kAgentPoll = (int)0x80000010u;     // sc1, not to be moved out of a loop
// (stores take the whole offset in the vector register: with a scalar one the
// compiler lets the next instruction overwrite the data registers, and the
// 16-byte store then sent some of the next value's words)
__device__ __forceinline__ void xput(__amdgpu_buffer_rsrc_t x, unsigned off, unsigned a,
                                     unsigned b, unsigned tag) {
  const u32x4_t w = {a, tag, b, tag};
  __builtin_amdgcn_raw_buffer_store_b128(w, x, off, 0, kAgent);
}
__device__ __forceinline__ u32x4_t xget(__amdgpu_buffer_rsrc_t x, unsigned off, unsigned soff) {
  return __builtin_amdgcn_raw_buffer_load_b128(x, off, soff, kAgentPoll);
}

// The words of one node's values, in pairs: Ux, Uy and, when the neighbours'
// velocities are needed too (T > 1), V in one (FP32) or two.
template <typename VT, int T>
struct XNode {
  static constexpr int Q = T == 1 ? 2 : 2 + (int)sizeof(VT) / 4;
  static __device__ __forceinline__ void put(__amdgpu_buffer_rsrc_t x, unsigned off, unsigned soff,
                                             unsigned stride, unsigned tag, double ux, double uy,
                                             VT vx, VT vy) {
    auto two = [&](int k, double v) {
      const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
      xput(x, off + (soff + k * stride), (unsigned)b, (unsigned)(b >> 32), tag);
    };
    two(0, ux);
    two(1, uy);
    if constexpr (T > 1) {
      if constexpr (sizeof(VT) == 8) {
        two(2, vx);
        two(3, vy);
      } else {
        // (kept apart: read as one vector, the two rows' arrays would live in
        // memory)
        unsigned a = __builtin_bit_cast(unsigned, vx), b = __builtin_bit_cast(unsigned, vy);
        asm volatile("" : "+v"(a), "+v"(b));
        xput(x, off + (soff + 2 * stride), a, b, tag);
      }
    }
  }
  u32x4_t w[Q];
  __device__ __forceinline__ void get(__amdgpu_buffer_rsrc_t x, unsigned off, unsigned soff,
                                      unsigned stride) {
#pragma unroll
    for (int k = 0; k < Q; k++) w[k] = xget(x, off, soff + k * stride);
  }
  __device__ __forceinline__ bool is(unsigned tag) const {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < Q; k++) ok = ok && w[k].y == tag && w[k].w == tag;
    return ok;
  }
  __device__ __forceinline__ double two(int k) const {
    return __builtin_bit_cast(double, (unsigned long long)w[k].z << 32 | w[k].x);
  }
  __device__ __forceinline__ double ux() const { return two(0); }
  __device__ __forceinline__ double uy() const { return two(1); }
  __device__ __forceinline__ VT vx() const {
    if constexpr (T == 1) return (VT)0;
    else if constexpr (sizeof(VT) == 8) return two(2);
    else return __builtin_bit_cast(float, (unsigned)w[2].x);
  }
  __device__ __forceinline__ VT vy() const {
    if constexpr (T == 1) return (VT)0;
    else if constexpr (sizeof(VT) == 8) return two(3);
    else return __builtin_bit_cast(float, (unsigned)w[2].z);
  }
};

// LDS of a tile: the rows neighbouring waves read (two sets, alternating), and
// each wave's edge columns -- its own on the way out, the neighbours' on the
// way in; zeroes for the lanes past the tile.
template <typename CT, typename VT, int R, int T, int NW>
struct ResLds {
  static constexpr int RR = R == 2 ? 2 : 3;
  double ux[2][NW][RR][64];  // a wave's first, last but one and last row
  double uy[2][NW][RR][64];  // first, last, second
  double2 colU[NW][R][4 * T];
  VT colV[T > 1 ? NW : 1][R][4 * T][2];
  double rowU[4 * T][2][64];  // rows the neighbouring tiles hold
  VT rowV[T > 1 ? 4 * T : 1][2][64];
  double2 zeroU[R][4 * T];
  VT zeroV[T > 1 ? R : 1][4 * T][2];
  VertMod<CT> gt[16];
  unsigned state;
};

// Orders a wave's LDS accesses among its lanes (the LDS serves a wave's
// accesses in order; this keeps the compiler from moving them).
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// rows of a wave taken at a time (ResRows)
template <typename CT>
constexpr int res_chunk(int rows) {
  return rows > 3 ? 2 : rows;
}

// One iteration of a wave's R rows, C of them at a time: the marching stage's
// expressions (MarchStage) on rows held in arrays, so the C rows' independent
// operations fill each other's latency (a wave that marches row by row waits
// out most of it: four waves to a SIMD do not hide it) and one test per C rows
// skips the scaling where no lane yields.  Ux rows -2 and -1 and Uy row -1 lie
// above the wave's rows, Ux row R and Uy rows R and R+1 below them.
template <typename CT, typename VT, int R, int C, bool EX, bool EY, bool CLEAN>
struct ResRows {
  using M = March<CT, VT>;
  static constexpr bool F64 = sizeof(CT) == 8;
  const VertMod<CT>* gt;
  int nX, nY, i;
  bool colC, leftEdge, rightEdge, plastic, near;
  CT coh, c2lo, K0, Kp, G2_0, G2_p, P0, vdampX, vdampY, dTrho, g0;
  double dT, dXd, dYd, rdXd, rdYd;
  CT rdXc, rdYc;

  // lane_prev, but lane 0 gets its own value
  static __device__ __forceinline__ int prev_or(int v) {
    return __builtin_amdgcn_update_dpp(v, v, 0x138, 0xf, 0xf, false);
  }
  static __device__ __forceinline__ CT lane_prev_or(CT v) {
    if constexpr (!EX) {
      return lane_prev(v);
    } else if constexpr (F64) {
      const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
      const unsigned lo = (unsigned)prev_or((int)(unsigned)b);
      const unsigned hi = (unsigned)prev_or((int)(unsigned)(b >> 32));
      return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
    } else {
      return __builtin_bit_cast(float, prev_or(__builtin_bit_cast(int, v)));
    }
  }

  // a coefficient in the arithmetic type; rounded to FP32 by the vector ALU, it
  // is moved back to a scalar register
  static __device__ __forceinline__ CT uni(double a) {
    if constexpr (F64) return a;
    else
      return __builtin_bit_cast(
          float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, (float)a)));
  }
  __device__ __forceinline__ void setup(const RveDev& r, const VertMod<CT>* g, int col) {
    gt = g;
    nX = r.nX;
    nY = r.nY;
    i = col;
    colC = !EX || i < nX;
    leftEdge = EX && i == 0;
    rightEdge = EX && i == nX - 1;
    plastic = r.plastic != 0;
    near = rm_near(r.coh);
    coh = uni(r.coh);
    if constexpr (F64) c2lo = r.coh2lo;
    else c2lo = r.coh2lof;
    K0 = uni(r.K0);
    Kp = uni(r.Kp);
    G2_0 = uni(2.0 * r.G0);
    G2_p = uni(2.0 * r.Gp);
    g0 = uni(r.gtab[0]);
    P0 = uni(r.P0);
    dXd = r.dX;
    dYd = r.dY;
    rdXd = r.rdX;
    rdYd = r.rdY;
    rdXc = uni(r.rdX);
    rdYc = uni(r.rdY);
    vdampX = uni(r.vdampX);
    vdampY = uni(r.vdampY);
    dTrho = uni(r.dTrho);
    dT = r.dT;
  }
  __device__ __forceinline__ CT dxs(double a) const {
    if constexpr (F64) return qdiv(a, dXd, rdXd);
    else return (CT)a * rdXc;
  }
  __device__ __forceinline__ CT dys(double a) const {
    if constexpr (F64) return qdiv(a, dYd, rdYd);
    else return (CT)a * rdYc;
  }

  // rows -2 .. R of Ux and of the vertices at index k + 2, rows -1 .. R+1 of Uy
  // and rows -1 .. R of the cells at index k + 1; mask: the mask bytes of rows
  // k - 2
  template <typename Mask>
  __device__ __forceinline__ void iterate(int jw, double (&ux)[R], double (&uy)[R], VT (&vx)[R],
                                          VT (&vy)[R], double a0, double a1, double b1,
                                          double c0, double d0, double d1, const Mask& mask) const {
    double sx[R + 3];  // Ux of the next column
    CT tP[R + 2], tXX[R + 2], tYY[R + 2], tXY[R + 2];
    CT vXX[R + 1], vYY[R + 1], nXY[R + 1];  // sums of vertex row and cell row k at k + 1
    CT hXX = 0, hYY = 0, hXY = 0;
    CT cXX[R + 1], cYY[R + 1], cXY[R + 1];  // corrected rows -1 .. R-1 at k + 1
    // the rows before this iteration's updates reach them (row k is updated
    // after every use of its old value)
    double ox[R + 3], oy[R + 3];
    ox[0] = a0;
    ox[1] = a1;
    oy[0] = b1;
#pragma unroll
    for (int k = 0; k < R; k++) {
      ox[k + 2] = ux[k];
      oy[k + 1] = uy[k];
    }
    ox[R + 2] = c0;
    oy[R + 1] = d0;
    oy[R + 2] = d1;

    auto cell = [&](auto KK) {  // trial cell of row k
      constexpr int k = decltype(KK)::value;
      CT K = K0, G2 = G2_0;
      if constexpr (!CLEAN) {
        const unsigned w = mask.template word<M_CELL_MAT, k + 2>();
        K = pick(w, Kp, K0);
        G2 = pick(w, G2_p, G2_0);
      }
      const CT exx = dxs(sx[k + 2] - ox[k + 2]);
      const CT eyy = dys(oy[k + 2] - oy[k + 1]);
      CT pp, txx, tyy;
      if constexpr (F64) {
        pp = P0 - K * (exx + eyy);
        txx = G2 * (exx - M::third(exx + eyy));
        tyy = G2 * (eyy - M::third(exx + eyy));
      } else {
        split_cell_trial(exx, eyy, K, G2, P0, pp, txx, tyy);
      }
      if constexpr (!CLEAN) {
        const unsigned w = mask.template word<M_CELL_ZERO, k + 2>();
        pp = keep(w, pp);
        txx = keep(w, txx);
        tyy = keep(w, tyy);
      }
      tP[k + 1] = pp;
      tXX[k + 1] = txx;
      tYY[k + 1] = tyy;
      // the vertex row above's sums, and the start of this row's
      const CT x = lane_next(txx), y = lane_next(tyy);
      if constexpr (k >= 0) {
        vXX[k] = hXX + txx + x;
        vYY[k] = hYY + tyy + y;
      }
      hXX = txx + x;
      hYY = tyy + y;
    };
    auto vertex = [&](auto KK) {  // trial vertex of row k
      constexpr int k = decltype(KK)::value;
      const CT g = CLEAN ? g0 : vert_mod(gt, CLEAN ? 0u : mask.byte(k + 2));
      const double uyn = oy[k + 2], uys = lane_next(uyn);
      CT t;
      if constexpr (F64) t = g * (dys(sx[k + 3] - sx[k + 2]) + dxs(uys - uyn));
      else t = split_vertex_trial(g, (CT)(sx[k + 3] - sx[k + 2]), rdYc, (CT)(uys - uyn), rdXc);
      if constexpr (!CLEAN) t = keep(mask.template word<M_VERT_ZERO, k + 2>(), t);
      tXY[k + 2] = t;
    };
    // the vertex row in the blocks of this lane's cell, clamped to the grid in x
    // (EffPlast2D.cu:109-137), and the sum of the block of rows k-1 and k
    // (lane 0 of the first strip is column 0: it keeps its own value)
    auto block = [&](auto KK) {
      constexpr int k = decltype(KK)::value;
      const CT t = tXY[k + 2];
      CT f = lane_prev_or(t), c = t;
      if constexpr (EX) {
        const CT nx = lane_next(t), pp = lane_prev(f);
        c = leftEdge ? nx : rightEdge ? f : t;
        f = rightEdge ? pp : f;
      }
      if constexpr (k > -2) nXY[k + 1] = hXY + f + c;
      hXY = f + c;
    };
    // squared invariants of vertex and cell row k, and whether they may yield
    CT s2v[R + 1], s2c[R + 1];
    auto invariants = [&](auto KK) {
      constexpr int k = decltype(KK)::value;
      const int j = jw + k;
      const CT sxx = vXX[k + 1], syy = vYY[k + 1];
      const CT t = tXY[k + 2];
      if constexpr (F64)
        s2v[k + 1] = (CT)0.0625 * sxx * sxx + (CT)0.0625 * syy * syy + (CT)2.0 * t * t;
      else s2v[k + 1] = split_s2_vertex(sxx, syy, t);
      CT n = nXY[k + 1];
      if constexpr (EY) {
        // row 0, the first of its wave, takes vertex rows 0 and 1, row nY-1 the
        // two above it
        const CT below = nXY[k == 0 ? 2 : k + 1], above = nXY[k >= 0 ? k : 0];
        n = k >= 0 && j == nY - 1 ? above : n;
        n = k == 0 && j == 0 ? below : n;
      }
      const CT av = (CT)0.25 * n;
      const CT xx = tXX[k + 1], yy = tYY[k + 1];
      if constexpr (F64) s2c[k + 1] = xx * xx + yy * yy + (CT)2.0 * av * av;
      else s2c[k + 1] = split_s2_cell(xx, yy, av);
    };
    auto yields = [&](auto KK) {
      constexpr int k = decltype(KK)::value;
      return s2v[k + 1] > c2lo || s2c[k + 1] > c2lo;
    };
    auto scale = [&](auto KK) {
      constexpr int k = decltype(KK)::value;
      rm_both<true>(s2v[k + 1], s2c[k + 1], coh, c2lo, near, cXY[k + 1], cXX[k + 1], cYY[k + 1]);
    };
    CT rXY = 0;
    auto move = [&](auto KK) {  // velocity and displacement of row k
      constexpr int k = decltype(KK)::value;
      const int j = jw + k;
      const CT cP = tP[k + 1], pP = tP[k], xx = cXX[k + 1], yy = cYY[k + 1], pY = cYY[k];
      const CT xyc = cXY[k + 1], xyp = cXY[k];
      const CT rP = lane_prev(cP), rXX = lane_prev(xx);
      // the left neighbours' shear: FP32 shifts the difference (the same value)
      CT dXY, rXYp;
      if constexpr (F64) {
        if constexpr (k == 0) rXY = lane_prev(xyp);
        rXYp = rXY;
        rXY = lane_prev(xyc);
        dXY = rXY - rXYp;
      } else {
        rXYp = lane_prev(xyp);
        dXY = lane_prev(xyc - xyp);
      }
      CT wx = (CT)vx[k], wy = (CT)vy[k];
      // (V past the last column is nobody's)
      const bool updX = (!EX || !leftEdge) && (!EY || (j > 0 && j < nY - 1));
      const bool updY = (!EX || !(leftEdge || rightEdge)) && (!EY || (j > 0 && j < nY));
      if constexpr (F64) {
        if (updX) wx = wx * vdampX + dTrho * (dxs(-cP + rP + xx - rXX) + dys(dXY));
        if (updY) wy = wy * vdampY + dTrho * (dys(-cP + pP + yy - pY) + dxs(xyp - rXYp));
      } else {
        if (updX)
          wx = (CT)(VT)split_velocity(wx, vdampX, dTrho, -cP + rP + xx - rXX, rdXc, dXY,
                                      rdYc);
        if (updY)
          wy = (CT)(VT)split_velocity(wy, vdampY, dTrho, -cP + pP + yy - pY, rdYc, xyp - rXYp,
                                      rdXc);
      }
      const bool in = (!EX || colC) && (!EY || (j >= 0 && j < nY));
      if constexpr (F64) {
        ux[k] = in ? ox[k + 2] + (double)wx * dT : ox[k + 2];
        uy[k] = in ? oy[k + 1] + (double)wy * dT : oy[k + 1];
      } else {
        ux[k] = in ? split_disp(ox[k + 2], wx, dT) : ox[k + 2];
        uy[k] = in ? split_disp(oy[k + 1], wy, dT) : oy[k + 1];
      }
      vx[k] = (VT)wx;
      vy[k] = (VT)wy;
    };

    // rows above the first
    using N2 = std::integral_constant<int, -2>;
    using N1 = std::integral_constant<int, -1>;
    sx[0] = lane_next(ox[0]);
    sx[1] = lane_next(ox[1]);
    chunks<0>([&](auto K0_, auto N_) {
      constexpr int k0 = decltype(K0_)::value, cn = decltype(N_)::value;
      if constexpr (k0 == 0) {
        sx[2] = lane_next(ox[2]);
        vertex(N2{});
        block(N2{});
        vertex(N1{});
        block(N1{});
        cell(N1{});
        cell(std::integral_constant<int, 0>{});
      }
      each<k0, cn>([&](auto K) {
        constexpr int k = decltype(K)::value;
        sx[k + 3] = lane_next(ox[k + 3]);
        cell(std::integral_constant<int, k + 1>{});
        vertex(K);
        block(K);
      });
      constexpr int f = k0 == 0 ? -1 : k0, fn = cn + (k0 == 0 ? 1 : 0);
      each<f, fn>([&](auto K) {
        constexpr int k = decltype(K)::value;
        cXX[k + 1] = tXX[k + 1];
        cYY[k + 1] = tYY[k + 1];
        cXY[k + 1] = tXY[k + 2];
      });
      if (plastic) {
        bool any = false;
        each<f, fn>([&](auto K) {
          invariants(K);
          any = any || yields(K);
        });
        if (__any(any && (!EX || colC))) each<f, fn>([&](auto K) { scale(K); });
      }
      each<k0, cn>([&](auto K) { move(K); });
      // (the next rows' loads and shifts are not to be drawn up here: they
      // would take the registers of a row each)
      if constexpr (C < R) __builtin_amdgcn_sched_barrier(0);
    });
  }

  template <int K, int N, typename F>
  static __device__ __forceinline__ void each(F f) {
    if constexpr (N > 0) {
      f(std::integral_constant<int, K>{});
      each<K + 1, N - 1>(f);
    }
  }
  template <int K, typename F>
  static __device__ __forceinline__ void chunks(F f) {
    if constexpr (K < R) {
      constexpr int n = K + C <= R ? C : R - K;
      f(std::integral_constant<int, K>{}, std::integral_constant<int, n>{});
      chunks<K + n>(f);
    }
  }
};

template <typename CT, typename VT, int R, int T, int NW, bool EX, bool EY, bool CLEAN>
struct ResWave {
  using Rows = ResRows<CT, VT, R, res_chunk<CT>(R), EX, EY, CLEAN>;
  using Lds = ResLds<CT, VT, R, T, NW>;
  using Node = XNode<VT, T>;
  static constexpr int NM = (R + 6) / 4, C4 = 4 * T;

  double ux[R], uy[R];
  VT vx[R], vy[R];
  unsigned mk[NM];  // mask bytes of rows jw-2 .. jw+R, four to a word

  __device__ __forceinline__ unsigned byte(int k) const { return mk[k >> 2] >> (8 * (k & 3)); }
  template <int BIT, int k>
  __device__ __forceinline__ unsigned word() const {
    return mask_word<BIT << (8 * (k & 3))>(mk[k >> 2]);
  }

  __device__ __forceinline__ void run(const RveDev& r, const ResTile& q, int cur, VT* Vx, VT* Vy,
                                      int v, int nw, Lds& lds, int n, const char* xch,
                                      unsigned xpar, unsigned tag0, unsigned pollLimit,
                                      bool& lost) {
    const int nX = r.nX, nY = r.nY, sx = nX + 1;
    const int L = threadIdx.x & 63;
    const int i = q.s + L;
    int jw = q.jr + v * R;  // the wave's first row
    // lanes of the tile, its own columns, and the columns the neighbours own
    const int used = q.i1 - q.s + (q.xr >= 0 ? 2 * T : 1);
    const bool own = i >= q.i0 && i < q.i1;
    const bool inCol = i >= 0 && i < nX && L < used;
    const bool recv = L >= used || (L < 2 * T && q.xl >= 0) || (i >= q.i1 && q.xr >= 0);

    // the state: every row of the wave (0 outside the grid)
    {
      const double* Uxi = r.Ux[cur];
      const double* Uyi = r.Uy[cur];
      const bool cx = i >= 0 && i <= nX && L < used;
#pragma unroll
      for (int k = 0; k < R; k++) {
        const int j = jw + k;
        ux[k] = cx && j < nY ? gld(Uxi, (unsigned)(j * sx + i)) : 0.0;
        uy[k] = inCol && j <= nY ? gld(Uyi, (unsigned)(j * nX + i)) : 0.0;
        vx[k] = inCol && j < nY ? gld(Vx, (unsigned)(j * sx + i)) : (VT)0;
        vy[k] = inCol && j < nY ? gld(Vy, (unsigned)(j * nX + i)) : (VT)0;
      }
      if constexpr (!CLEAN) {
#pragma unroll
        for (int k = 0; k < NM; k++) mk[k] = 0u;
#pragma unroll
        for (int k = 0; k < R + 3; k++) {
          const int j = jw - 2 + k;
          if (inCol && j >= 0 && j < nY)
            mk[k >> 2] |= (unsigned)gld(r.mask, (unsigned)(j * nX + i)) << (8 * (k & 3));
        }
#pragma unroll
        for (int k = 0; k < NM; k++) mk[k] ^= 0x01010101u * (unsigned)(M_CELL_ZERO | M_VERT_ZERO);
      }
    }

    // the lane's entry of the wave's edge columns: row jw + er, column eq (of
    // the left edge below 2T, of the right edge from 2T on), and its place in
    // the exchange buffer going out and coming in
    const int er = L / C4, eq = L % C4;
    const int ej = jw + er;
    const bool left = eq < 2 * T;
    const bool act = er < R && ej >= q.j0 && ej < q.j1 && (left ? q.xl >= 0 : q.xr >= 0);
    // (byte offsets: side 0 of a boundary holds the left tile's columns)
    const unsigned xe = 16u * ((unsigned)(left ? q.xl : q.xr) + (unsigned)(ej * C4) +
                               (unsigned)(left ? eq : eq - 2 * T));
    unsigned xout = xe + (left ? 32u * T : 0u), xin = xe + (left ? 0u : 32u * T);
    unsigned xi = 16u * (unsigned)i;
    // where the lane's own columns go and the neighbours' come from
    const int fl = i - q.i0, ll = i - (q.i1 - 2 * T);
    const bool edgeL = fl >= 0 && fl < 2 * T, edgeR = ll >= 0 && ll < 2 * T && own;
    const int eout = edgeL ? fl : 2 * T + ll;
    const int ein = L < 2 * T ? L : 2 * T + (i - q.i1);
    const bool junk = L >= used;
    const double2* inU = junk ? &lds.zeroU[0][0] : &lds.colU[v][0][ein];
    const VT* inV = junk ? &lds.zeroV[0][0][0] : &lds.colV[T > 1 ? v : 0][0][T > 1 ? ein : 0][0];
    // rows the neighbours hold, and rows past the tile
    const int hiRow = q.j1 + (q.xd >= 0 ? 2 * T : 1);

    Rows st;
    st.setup(r, lds.gt, i);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    int ph = 0;          // iterations since the last exchange
    unsigned tag = tag0;
    for (int t = 0; t < n; t++) {
      const int p = t & 1;
      // the tests and coefficients that depend on a row's number and mask byte
      // are formed anew in each iteration: held through the loop, they would
      // take more registers than the state
      asm volatile("" : "+s"(jw));
      if constexpr (!CLEAN) {
#pragma unroll
        for (int k = 0; k < NM; k++) asm volatile("" : "+v"(mk[k]));
      }
      if (ph == T) {
        ph = 0;
        tag++;
        const __amdgpu_buffer_rsrc_t x = brsrc(xch + ((tag & 1) ? (size_t)xpar : 0));
        asm volatile("" : "+v"(xout), "+v"(xin), "+v"(xi));
        int nx = nX, ny = nY;
        asm volatile("" : "+s"(nx), "+s"(ny));
        const unsigned cs = 16u * C4 * (unsigned)ny, rs = 16u * (unsigned)nx;  // value strides
        const unsigned xu = 16u * (unsigned)q.xu, xd = 16u * (unsigned)q.xd;
        // out: edge columns (through LDS, one lane to a node), then edge rows
        if (edgeL || edgeR) {
#pragma unroll
          for (int k = 0; k < R; k++) {
            lds.colU[v][k][eout] = make_double2(ux[k], uy[k]);
            if constexpr (T > 1) {
              lds.colV[v][k][eout][0] = vx[k];
              lds.colV[v][k][eout][1] = vy[k];
            }
          }
        }
        lds_order();
        if (act) {
          const double2 c = lds.colU[v][er][eq];
          VT a = 0, b = 0;
          if constexpr (T > 1) {
            a = lds.colV[v][er][eq][0];
            b = lds.colV[v][er][eq][1];
          }
          Node::put(x, xout, 0u, cs, tag, c.x, c.y, a, b);
        }
        // the tile's first and last 2T own rows
        // (an arm for each row ends in a statement of its own: arms that end
        // alike would be merged into one with a computed row, and the rows
        // would live in memory)
        if (q.xu >= 0 && jw < q.j0 + 2 * T && jw + R > q.j0)
          Rows::template each<0, R>([&](auto KK) {
            constexpr int k = decltype(KK)::value;
            const int g = jw + k - q.j0;
            if (g >= 0 && g < 2 * T && own) {
              Node::put(x, xi, xu + (unsigned)((2 * T + g) * Node::Q) * rs, rs, tag, ux[k], uy[k],
                        vx[k], vy[k]);
              asm volatile("; row %0" ::"i"(k));
            }
          });
        if (q.xd >= 0 && jw < q.j1 && jw + R > q.j1 - 2 * T)
          Rows::template each<0, R>([&](auto KK) {
            constexpr int k = decltype(KK)::value;
            const int g = jw + k - (q.j1 - 2 * T);
            if (g >= 0 && g < 2 * T && own) {
              Node::put(x, xi, xd + (unsigned)(g * Node::Q) * rs, rs, tag, ux[k], uy[k], vx[k],
                        vy[k]);
              asm volatile("; row %0" ::"i"(k));
            }
          });
        // in: the wave's edge columns, and its share of the rows the
        // neighbours hold (row g of them: the 2T rows above the tile's own,
        // then the 2T below); polls until every word carries this exchange's
        // tag
        for (int g = v; g < 4 * T || g == v; g += nw) {
          const bool above = g < 2 * T;
          const bool cols = act && g == v;
          const bool rows = g < 4 * T && inCol && (above ? q.xu >= 0 : q.xd >= 0);
          const unsigned xg = (above ? xu : xd) + (unsigned)(g * Node::Q) * rs;
          Node c, w;
          for (unsigned polls = 0;; polls++) {
            if (cols) c.get(x, xin, 0u, cs);
            if (rows) w.get(x, xi, xg, rs);
            const bool late = (cols && !c.is(tag)) || (rows && !w.is(tag));
            if (!__any(late)) break;
            if (lost || polls >= pollLimit) {
              lost = true;
              break;
            }
          }
          if (cols) {
            lds.colU[v][er][eq] = make_double2(c.ux(), c.uy());
            if constexpr (T > 1) {
              lds.colV[v][er][eq][0] = c.vx();
              lds.colV[v][er][eq][1] = c.vy();
            }
          }
          if (rows) {
            lds.rowU[g][0][L] = w.ux();
            lds.rowU[g][1][L] = w.uy();
            if constexpr (T > 1) {
              lds.rowV[g][0][L] = w.vx();
              lds.rowV[g][1][L] = w.vy();
            }
          }
        }
        lds_barrier();
        auto fromCol = [&](auto KK) {
          constexpr int k = decltype(KK)::value;
          const double2 c = inU[k * C4];
          ux[k] = c.x;
          uy[k] = c.y;
          if constexpr (T > 1) {
            vx[k] = inV[2 * C4 * k];
            vy[k] = inV[2 * C4 * k + 1];
          }
        };
        if (jw >= q.j0 && jw + R <= q.j1) {
          if (recv) Rows::template each<0, R>(fromCol);
        } else {
          Rows::template each<0, R>([&](auto KK) {
            constexpr int k = decltype(KK)::value;
            const int j = jw + k;
            if (j >= q.j0 && j < q.j1) {
              if (recv) fromCol(KK);
            } else if (inCol && (j < q.j0 ? q.xu >= 0 : q.xd >= 0 && j < q.j1 + 2 * T)) {
              const int g = j < q.j0 ? j - q.jr : 2 * T + j - q.j1;
              ux[k] = lds.rowU[g][0][L];
              uy[k] = lds.rowU[g][1][L];
              if constexpr (T > 1) {
                vx[k] = lds.rowV[g][0][L];
                vy[k] = lds.rowV[g][1][L];
              }
            }
          });
        }
        // rows past the tile only feed rows nobody reads
        if (jw + R > hiRow && q.xd >= 0) {
#pragma unroll
          for (int k = 0; k < R; k++)
            if (jw + k >= hiRow) ux[k] = uy[k] = 0.0, vx[k] = vy[k] = (VT)0;
        }
      }
      ph++;
      // rows the neighbouring waves march over
      {
        auto& X = lds.ux[p][v];
        auto& Y = lds.uy[p][v];
        X[0][L] = ux[0];
        Y[0][L] = uy[0];
        X[1][L] = ux[R == 2 ? 1 : R - 2];
        Y[1][L] = uy[R - 1];
        if constexpr (R > 2) {
          X[2][L] = ux[R - 1];
          Y[2][L] = uy[1];
        }
      }
      lds_barrier();
      double a0 = 0.0, a1 = 0.0, b1 = 0.0, c0 = 0.0, d0 = 0.0, d1 = 0.0;
      if (v > 0) {
        auto& X = lds.ux[p][v - 1];
        a0 = X[R == 2 ? 0 : 1][L];
        a1 = X[R == 2 ? 1 : 2][L];
        b1 = lds.uy[p][v - 1][1][L];
      }
      if (v < nw - 1) {
        c0 = lds.ux[p][v + 1][0][L];
        d0 = lds.uy[p][v + 1][0][L];
        d1 = lds.uy[p][v + 1][R == 2 ? 1 : 2][L];
      }
      // U of the state before the last iteration: the stress fields of a load
      // step are recomputed from it (EffPlast2D.cu:428)
      if (t == n - 1) storeU(r, q, cur, i, jw, own);
      st.iterate(jw, ux, uy, vx, vy, a0, a1, b1, c0, d0, d1, *this);
    }
    storeU(r, q, cur ^ 1, i, jw, own);
#pragma unroll
    for (int k = 0; k < R; k++)
      if (own && jw + k >= q.j0 && jw + k < q.j1) {
        gst(Vx, (unsigned)((jw + k) * sx + i), vx[k]);
        gst(Vy, (unsigned)((jw + k) * nX + i), vy[k]);
      }
  }

  // this wave's own rows of U, and the nodes beside them that ComputeDisp
  // never updates (Ux column nX, by the last strip, and Uy row nY)
  __device__ __forceinline__ void storeU(const RveDev& r, const ResTile& q, int b, int i, int jw,
                                         bool own) const {
    const int nX = r.nX, nY = r.nY, sx = nX + 1;
    double* Uxo = r.Ux[b];
    double* Uyo = r.Uy[b];
#pragma unroll
    for (int k = 0; k < R; k++) {
      const int j = jw + k;
      if (j < q.j0) continue;
      if (j < q.j1 && (own || (q.xr < 0 && i == nX))) gst(Uxo, (unsigned)(j * sx + i), ux[k]);
      if ((j < q.j1 || j == nY) && own) gst(Uyo, (unsigned)(j * nX + i), uy[k]);
    }
  }
};

// waves of a SIMD the registers are held to: two tiles to a CU where they are
// given half of one (two split rows a wave), else one
template <typename CT, int R>
constexpr int res_waves() {
  return sizeof(CT) == 4 && R <= 2 ? 4 : 2;
}

template <typename CT, typename VT, int R, int T, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(res_waves<CT, R>()))) void k_resident(
    const RveDev* __restrict__ rves, const ResTile* __restrict__ tiles, int parity, int vpar,
    int n, const char* xch, unsigned xpar, unsigned tag0, ResCtl* ctl, ResLimits lim, unsigned need,
    unsigned cus, unsigned run, unsigned* told) {
  using Lds = ResLds<CT, VT, R, T, NW>;
  __shared__ Lds lds;
  const int v = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const ResTile q = tiles[blockIdx.x];
  const RveDev& r = rves[q.rve];
  if (threadIdx.x < 16) lds.gt[threadIdx.x].g = (CT)r.gtab[threadIdx.x];
  if (threadIdx.x < R * 4 * T) {
    (&lds.zeroU[0][0])[threadIdx.x] = make_double2(0.0, 0.0);
    if constexpr (T > 1) {
      (&lds.zeroV[0][0][0])[2 * threadIdx.x] = (VT)0;
      (&lds.zeroV[0][0][0])[2 * threadIdx.x + 1] = (VT)0;
    }
  }
  if (threadIdx.x == 0) lds.state = res_arrive(ctl, gridDim.x, lim.arriveTicks, need, cus);
  __syncthreads();
  if (lds.state == kResGo) {
    bool lost = false;
    const int cur = parity ^ r.cur;
    // waves with rows of the tile; the others only keep the barrier count
    const int rows = q.j1 - q.jr + (q.xd >= 0 ? 2 * T : 1);
    const int nw = min(NW, (rows + R - 1) / R);
    if (v < nw) {
      VT* Vx = static_cast<VT*>(vpar ? r.Vx2 : r.Vx);
      VT* Vy = static_cast<VT*>(vpar ? r.Vy2 : r.Vy);
      // the classes of the chain kernels, for this wave's rows and columns
      const int used = q.i1 - q.s + (q.xr >= 0 ? 2 * T : 1), jw = q.jr + v * R;
      const bool ex = !(q.s >= 1 && q.s + used - 1 <= r.nX - 2);
      const bool ey = !(jw >= 2 && jw + R <= r.nY - 1);
      const int L = threadIdx.x & 63, i = q.s + L;
      unsigned any = 0;
      if (i < r.nX && L < used)
        for (int j = max(jw - 2, 0); j <= min(jw + R, r.nY - 1); j++)
          any |= gld(r.mask, (unsigned)(j * r.nX + i));
      const bool clean = !__any(any != 0);
#define EP2D_RES(EX, EY, CLEAN)                                                     \
  {                                                                                 \
    ResWave<CT, VT, R, T, NW, EX, EY, CLEAN> wv;                                    \
    wv.run(r, q, cur, Vx, Vy, v, nw, lds, n, xch, xpar, tag0, lim.polls, lost);                \
  }
      if (ex && clean) EP2D_RES(true, true, true)
      else if (ex) EP2D_RES(true, true, false)
      else if (ey && clean) EP2D_RES(false, true, true)
      else if (ey) EP2D_RES(false, true, false)
      else if (clean) EP2D_RES(false, false, true)
      else EP2D_RES(false, false, false)
#undef EP2D_RES
    } else {
      // (one an iteration, and one an exchange)
      for (int t = 0; t < n + (n - 1) / T; t++) lds_barrier();
    }
    if (__any(lost) && (threadIdx.x & 63) == 0) acas(&ctl->state, kResGo, kResLost);
  }
  __syncthreads();
  if (threadIdx.x == 0) res_depart(ctl, gridDim.x, need, run, told);
}

// the kernel of a scheme and a tile shape
template <typename F>
auto res_dispatch(int mode, const ResShape& sh, F f) {
  auto is = [&](int R, int T, int NW) {
    return sh.rows == R && sh.every == T && sh.waves == NW;
  };
  if (mode == 2) {
    if (is(2, 2, 8)) return f(k_resident<float, float, 2, 2, 8>);
    if (is(4, 2, 8)) return f(k_resident<float, float, 4, 2, 8>);
  } else {
    if (is(2, 2, 8)) return f(k_resident<double, double, 2, 2, 8>);
    if (is(4, 2, 8)) return f(k_resident<double, double, 4, 2, 8>);
    if (is(6, 1, 8)) return f(k_resident<double, double, 6, 1, 8>);
  }
  throw std::invalid_argument("no resident kernel of this shape");
}

// parts of a side of n nodes whose tiles span `span` of them, 2T on each
// inner side a neighbour's and, on the last, one the node past the side
int res_parts(int n, int span, int T) {
  if (n + 1 <= span) return 1;
  if ((n + 1) / 2 <= span - 2 * T - 1) return 2;
  return (n + span - 4 * T - 1) / (span - 4 * T);
}

}  // namespace

// From runs of 500 iterations of one RVE whose nodes yield (us per iteration; in
// brackets the chains on the shortest segments of one round, at the same size
// in the same process):
//   split, two rows a wave:  64^2 2.6 (3.1), 256^2 2.6 (3.3), 336^2 3.1 (3.8),
//     with two tiles to a CU 352^2 3.4 (3.8), 392^2 3.5 (3.9); with eight strips
//     from 393^2 on 4.2 (3.9) and 447^2 4.7 (4.0): chains up to 447^2
//   split, four rows, one tile to a CU:  449^2 4.15 (4.12), 480^2 4.15 (4.04),
//     505^2 3.9 (4.1), 512^2 3.9 (4.1), 560^2 4.1 (4.3)
//   FP64, two rows:  64^2 4.0 (4.8), 256^2 4.1 (5.4), 336^2 4.2 (5.8); from 337^2
//     on the tiles find no room
//   FP64, four rows:  352^2 6.2 (5.9), 400^2 6.3 (6.3), 448^2 6.3 (6.6), 504^2
//     6.5 (6.5), 512^2 6.1 (6.7), 560^2 6.2 (7.2)
//   FP64, six rows, an exchange each iteration:  672^2 8.3 (8.3), 700^2 8.2 (8.4),
//     768^2 8.4 (9.1), 792^2 8.3 (9.4); from 793^2 on the tiles find no room.
//     600^2 and 640^2 lie past the four rows' room: chains, 7.5
std::vector<ResShape> resident_shapes(int mode) {
  if (mode == 2) return {{2, 2, 8, 1, 0, 392}, {4, 2, 8, 2, 448}};
  return {{2, 2, 8, 2, 0}, {4, 2, 8, 2, 448}, {6, 1, 8, 2, 672}};
}

int resident_tiles(const ResShape& sh, int mode, int n, int rve, size_t x0, ResTile* out,
                   size_t* pairs) {
  const int T = sh.every, H = sh.rows * sh.waves;
  if (H <= 4 * T || n < sh.from || (sh.to > 0 && n > sh.to)) return 0;
  const int strips = res_parts(n, 64, T), bands = res_parts(n, H, T);
  // a tile's own part is at least as wide as what its neighbours read of it
  if ((strips > 1 && n / strips < 4 * T) || (bands > 1 && n / bands < 2 * T)) return 0;
  const size_t Q = T == 1 ? 2 : mode == 2 ? 3 : 4;
  const size_t col = Q * 4 * (size_t)T * (size_t)n;  // pairs of one boundary, either way
  const size_t rows0 = x0 + col * (size_t)(strips - 1);
  if (pairs) *pairs = col * (size_t)(strips - 1 + bands - 1);
  if (!out) return strips * bands;
  int t = 0;
  for (int b = 0; b < bands; b++)
    for (int c = 0; c < strips; c++) {
      ResTile& q = out[t++];
      q = ResTile{};
      q.rve = rve;
      q.i0 = (int)((long)n * c / strips);
      q.i1 = (int)((long)n * (c + 1) / strips);
      q.j0 = (int)((long)n * b / bands);
      q.j1 = (int)((long)n * (b + 1) / bands);
      q.s = c > 0 ? q.i0 - 2 * T : 0;
      q.jr = b > 0 ? q.j0 - 2 * T : 0;
      q.xl = c > 0 ? (int)(x0 + col * (size_t)(c - 1)) : -1;
      q.xr = c < strips - 1 ? (int)(x0 + col * (size_t)c) : -1;
      q.xu = b > 0 ? (int)(rows0 + col * (size_t)(b - 1)) : -1;
      q.xd = b < bands - 1 ? (int)(rows0 + col * (size_t)b) : -1;
    }
  return t;
}

int device_cus(int device) {
  int cus = 0;
  EP2D_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device));
  return cus;
}

int resident_cost(const ResShape& sh, int mode) {
  int nb = 0;
  res_dispatch(mode, sh, [&](auto kern) {
    EP2D_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, (const void*)kern, 64 * sh.waves, 0));
    return 0;
  });
  return nb >= 2 ? sh.cost : nb == 1 ? 2 : 0;
}

void launch_resident(const ResLaunch& a, hipStream_t s, hipEvent_t e0, hipEvent_t e1) {
  const dim3 grid((unsigned)a.tiles), block(64 * a.shape.waves);
  res_dispatch(a.mode, a.shape, [&](auto kern) {
    const char* xch = a.xch;
    const unsigned need = a.half | a.whole << 16;
    if (e0)
      hipExtLaunchKernelGGL(kern, grid, block, 0, s, e0, e1, 0, a.rves, a.list, a.parity, a.vpar,
                            a.iters, xch, a.xpar, a.tag0, a.ctl, a.limits, need, a.cus, a.run,
                            a.told);
    else
      hipLaunchKernelGGL(kern, grid, block, 0, s, a.rves, a.list, a.parity, a.vpar, a.iters, xch,
                         a.xpar, a.tag0, a.ctl, a.limits, need, a.cus, a.run, a.told);
    return 0;
  });
  EP2D_HIP(hipGetLastError());
}

}  // namespace ep2d
