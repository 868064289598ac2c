// projection_device.hpp - device code of the tiled projections shared by the
// per-grid kernels (kernels_project.hip) and the batched step kernel
// (kernels_batch.hip).
#pragma once

#include <type_traits>

#include "fluid_device.hpp"
#include "kernels.hpp"
#include "step_device.hpp"

#pragma clang fp contract(off)

namespace osy {

// Per-cell gate byte of the tiled kernel, built in LDS from the flags.  The
// four face gates are set only for projected cells, so a cell that is not
// projected changes nothing when it runs the update.
enum : uint32_t {
  G_L = 1u << 0,     // u(i,j) moves   (left neighbour fluid)
  G_R = 1u << 1,     // u(i+1,j) moves (right neighbour fluid)
  G_B = 1u << 2,     // v(i,j) moves   (bottom neighbour fluid)
  G_T = 1u << 3,     // v(i,j+1) moves (top neighbour fluid)
  G_UPD = 1u << 4,   // cell is projected
  G_L2_SHIFT = 5,    // bits 5..6: log2(total_s) when total_s is 1, 2 or 4
  G_SLOW = 1u << 7,  // projected with total_s 0 or 3: divide
};

// d = o * (div / s) for the cell with gate byte g.  For s = 1, 2, 4 the
// quotient is div * 2^-log2(s), exact; for s = 0 or 3 (cells against a
// wall or the obstacle) the lanes that need it divide.  Exhaustively checked
// against IEEE division over all binary32 inputs (tests/test_quotient.py).
__device__ inline float relaxed_quotient(float div, uint32_t g, float o) {
  const float y = __uint_as_float(0x3F800000u - (((g >> G_L2_SHIFT) & 3u) << 23));
  float q = div * y;
  if (g & G_SLOW) q = div / (float)__builtin_popcount(g & 15u);
  return o * q;
}

// x + gate(d): d when the gate bit is set, else -0 (x + -0 == x for every x,
// signed zeros and NaN included), so the face keeps its bits when closed.
__device__ inline float gated_add(float x, float d, uint32_t g, int bit) {
  const uint32_t m = (uint32_t)((int32_t)(g << (31 - bit)) >> 31);
  return x + __uint_as_float((__float_as_uint(d) & m) | (~m & 0x80000000u));
}
// x - gate(d): d when set, else +0 (x - +0 == x for every x).
__device__ inline float gated_sub(float x, float d, uint32_t g, int bit) {
  const uint32_t m = (uint32_t)((int32_t)(g << (31 - bit)) >> 31);
  return x - __uint_as_float(__float_as_uint(d) & m);
}

// Two horizontally adjacent elements (cells 2q, 2q+1 of a row).
template <typename T> struct PairOf;
template <> struct PairOf<float> { using type = float2; };
template <> struct PairOf<__half> { using type = __half2; };
template <> struct PairOf<__hip_bfloat16> { using type = __hip_bfloat162; };

template <typename T>
__device__ inline void load_pair(const T* __restrict__ a, long k, bool in0, bool in1, float& x0,
                                 float& x1) {
  if (in0 && in1) {  // k is even and rows start on 64-element boundaries
    const typename PairOf<T>::type pr = *reinterpret_cast<const typename PairOf<T>::type*>(a + k);
    x0 = Store<T>::ld(pr.x);
    x1 = Store<T>::ld(pr.y);
  } else {
    x0 = in0 ? ldf(a, k) : 0.0f;
    x1 = in1 ? ldf(a, k + 1) : 0.0f;
  }
}

template <typename T>
__device__ inline void store_pair(T* __restrict__ a, long k, bool in0, bool in1, float x0,
                                  float x1) {
  if (in0 && in1) {
    typename PairOf<T>::type pr;
    pr.x = Store<T>::st(x0);
    pr.y = Store<T>::st(x1);
    *reinterpret_cast<typename PairOf<T>::type*>(a + k) = pr;
  } else {
    if (in0) stf(a, k, x0);
    if (in1) stf(a, k + 1, x1);
  }
}

// ---- register-resident kernels -----------------------------------------------
//
// NW wavefronts stacked vertically; wavefront w holds region rows
// [w*R, w*R + R), lane l holds cells 2l and 2l+1 of each of them: u, v and
// the face masks of both cells, all in VGPRs for the whole launch.  The
// region is 128 x NW*R cells.
//
// In a colour phase each row has one active cell per lane (parity b).  For
// b = 0 every face the cell touches is in the lane's own registers.  For
// b = 1 the right face u(2l+2) belongs to lane l+1: it is read and updated
// through DPP lane shifts.  The top face of a wavefront's last row belongs
// to the wavefront above and is exchanged through LDS (reg_phase).

__device__ inline float lane_from_right(float x) {  // lane l gets lane l+1's x (0 for lane 63)
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xf, 0xf, true));
}
__device__ inline float lane_from_left(float x) {  // lane l gets lane l-1's x (0 for lane 0)
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xf, 0xf, true));
}
__device__ inline uint32_t lane_from_left_u(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x138, 0xf, 0xf, true);
}

// A copy of x in a register of its own.  The values of a pair are loaded and
// stored as one 8-byte register; left to itself the compiler keeps them in
// such pairs through the sweeps, which it cannot colour without spilling.
__device__ inline float own_register(float x) {
  float y;
  asm("v_mov_b32 %0, %1" : "=v"(y) : "v"(x));
  return y;
}

// Gate byte of a cell from its flag f, the right neighbour's flag fr and
// the top neighbour's flag ft (same encoding as the LDS-tiled kernel).
__device__ inline uint32_t gate_byte(uint32_t f, uint32_t fr, uint32_t ft) {
  if (!(f & CF_UPD)) return 0;
  uint32_t g = G_UPD;
  if (f & CF_FU) g |= G_L;
  if (fr & CF_FU) g |= G_R;
  if (f & CF_FV) g |= G_B;
  if (ft & CF_FV) g |= G_T;
  const uint32_t s = (f >> CF_S_SHIFT) & 7u;
  if (s == 0 || s == 3)
    g |= G_SLOW;
  else
    g |= (s >> 1) << G_L2_SHIFT;
  return g;
}

struct RegArgs {
  int tw, th, k;  // tile pitch and sweeps per launch or stage (halo 2k)
  int ntx, nty;   // tiles per grid row and column
  int inset;      // 0, or 2k: how far the first region reaches out of the grid
  int sweeps;     // sweeps this launch (<= k)
  int forces;     // apply the velocity forces on load, pressure sums from 0
};

// Where a workgroup's tile lies.  Region (tx, ty) starts at grid cell
// (tx*tw, ty*th) - inset, all even, and is 128 x NW*R cells.  With inset 0 a
// tile owns the cells of its region at least 2k from the region's edges, and
// also those up to an edge that is the grid's own: nothing outside the grid
// reaches them, so the first and last tiles need no halo there, and
// (W - 4k) / tw tiles, rounded up, cover a row of W cells (one when
// W <= 128).  The batch's tiles keep the halo all round (inset 2k, W / tw
// tiles, rounded up).  Wavefront-uniform.
struct RegPlace {
  int K, gx0, gy0, w, rbase;
  int c0, c1, r0, r1;  // owned columns [c0, c1) and rows [r0, r1) of the region
  int rows;            // region rows inside the grid (inset 0)
  bool left, right, below, above;  // a neighbouring tile on that side
};

template <int R, int NW>
__device__ inline RegPlace reg_place(const RegArgs& a, int tile, int W, int H) {
  RegPlace pl;
  pl.K = a.k;
  const int tx = tile % a.ntx, ty = tile / a.ntx;
  pl.gx0 = tx * a.tw - a.inset;
  pl.gy0 = ty * a.th - a.inset;
  pl.w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  pl.rbase = pl.w * R;
  pl.left = tx > 0;
  pl.right = tx + 1 < a.ntx;
  pl.below = ty > 0;
  pl.above = ty + 1 < a.nty;
  pl.c0 = pl.left ? 2 * a.k : a.inset;
  pl.c1 = pl.right ? 2 * a.k + a.tw : W - pl.gx0;
  pl.r0 = pl.below ? 2 * a.k : a.inset;
  pl.r1 = pl.above ? 2 * a.k + a.th : H - pl.gy0;
  pl.rows = min(NW * R, H - pl.gy0);
  return pl;
}

// The divisor of update_pressure_at: d_t, and recip = 1.0 / (double)d_t
// (the double nearest 1/d_t) when 0 < |d_t| < 2, else 0.
struct PressureDivisor {
  float d_t;
  double recip;
};

// x / b for 0 < |b| < 2 with recip the double nearest 1 / b: the IEEE float
// quotient for every binary32 x.  The double is within 2^-52 of x / b; a
// quotient of two binary32 numbers lies at least 2^-49 of itself from every
// binary32 rounding midpoint in the normal range, and in the subnormal range
// it can only equal a midpoint if the divisor's lowest set bit weighs 2 or
// more, which |b| < 2 excludes.  (Exhaustive device check for b = 0.05 and
// 1/60: osy_arith_check, modes 5 and 6.)
__device__ inline float recip_quotient(float x, double recip) {
  return (float)((double)x * recip);
}

// How a kernel adds the pressure sums: not at all; through the double
// reciprocal with density = cell_size = 1, whose products are the identity;
// through it in general; by division.
enum PressureMode : int { PM_NONE = 0, PM_UNIT = 1, PM_RECIP = 2, PM_DIVIDE = 3 };

struct SweepParams {
  float o, density, csf;
  PressureDivisor pd;
  int drain;  // region column of the grid's last column (W - 1); past the
              // region (128 or more) in all but the last tiles of a row
};

// update_pressure_at (src/fluid.cu:221-227): p + ((d * density) * cell_size) / d_t.
template <int PM>
__device__ inline float pressure_add(float p, float d, const SweepParams& q) {
  if constexpr (PM == PM_UNIT) return p + recip_quotient(d, q.pd.recip);
  if constexpr (PM == PM_RECIP) return p + recip_quotient((d * q.density) * q.csf, q.pd.recip);
  if constexpr (PM == PM_DIVIDE) return p + ((d * q.density) * q.csf) / q.pd.d_t;
  return p;
}

// Register state of one lane.  The face masks (wavefronts of kind WK_ANY
// only, reg_masks) are one word per face, all
// ones where the projection may move the face, else 0: mu0, mu1 the left
// faces of cells 2l and 2l+1 (mu1 is also the right face of cell 2l, the
// next lane's mu0 that of cell 2l+1), mv0, mv1 their bottom faces (row r+1's
// are the top faces of row r), mt0, mt1 the top faces of row R-1.  A closed
// face then costs one bit operation in each update: x + d becomes
// x + (d or -0) and x - d becomes x - (d or +0), both of which leave every
// x's bits when closed.
//
// The last column of an open grid (the drain) is fluid but not projected:
// its left face moves with the cell to its left only, so the drain column's
// own d is forced to -0 (SweepParams::drain), which leaves that face as it
// is; its other faces are closed.
template <int R>
struct RegTile {
  float u0[R], u1[R], v0[R], v1[R];  // faces of cells 2l and 2l+1, rows 0..R-1
  float s0[R], s1[R];                // pressure sums (pressure runs only)
  uint32_t gw[R];                    // gate bytes: cell 2l in bits 0-7, 2l+1 in 8-15
  uint32_t mu0[R], mu1[R], mv0[R], mv1[R];
  uint32_t mt0, mt1;
  uint32_t cls[R];  // quotient_class of cell 2l, and of cell 2l+1 in the high half
  // wavefront-uniform
  bool enclosed;   // some projected cell has no open face (pressure runs)
  int kind;        // WaveKind, and the lanes of a wall or the drain
  unsigned long long lanes;
};

// What the cells of a wavefront's rows are.
enum WaveKind : int {
  WK_OPEN = 0,   // all open: no face mask, quotient div * 0.25
  WK_WALL = 1,   // open but for a wall, the same in every row: in some lanes
                 // the even cell is solid and the odd cell's left face closed
  WK_DRAIN = 2,  // open but for the drain column, an odd one, and the cells
                 // right of it (outside the grid)
  WK_DRAIN0 = 3,  // the same with an even drain column
  WK_ANY = 4,     // anything else: face masks, any quotient
};

// Every kind is straight-line code: a tile waits for its slowest neighbour,
// so the tiles at walls and obstacles set the pace of all, and a branch per
// row, which leaves nothing to overlap a row's latency with, made those 1.5
// times as slow.  A cell that moves nothing takes d = -0 where d is added
// and +0 where it is subtracted, which leaves every face's bits.
__device__ inline bool in_lanes(unsigned long long m) {
  return __builtin_amdgcn_inverse_ballot_w64(m);
}

// div / s with y = 1 / s rounded: third_quotient's correction, which for
// s = 1, 2, 4 adds the (exact) remainder of a quotient that is already
// rounded, so nothing.  With s = y = 0 it gives div * 0.  (Every s and binary32
// div against IEEE division: tests/test_any_quotient.py.)
__device__ inline float any_quotient(float div, float y, float s) {
  const float q0 = div * y;
  const float q1 = __builtin_fmaf(__builtin_fmaf(-q0, s, div), y, q0);
  return (q0 == 0.0f || __builtin_isinf(q0)) ? q0 : q1;
}

// The number s of a cell's open faces in the low byte and 12 / s (0 for
// s = 0) in the next: y = (12 / s) * RN(1 / 12) is 1 / s rounded for every s.
// (A table in a constant: with diverging branches here the compiler spilled a
// register at their join before it had widened the lane mask again.)
__device__ inline uint32_t quotient_class(int s) {
  return (uint32_t)s | ((0x346C0u >> (4 * s)) & 15u) << 8;
}

// The quotient of the active cell of row rho, parity B.  A projected cell
// without open faces adds div / 0 to its pressure (`enclosed`: the wavefront
// has such cells), which is div * infinity.
template <int R, int B, int PM, int KIND>
__device__ __attribute__((always_inline)) inline float kind_quotient(const RegTile<R>& t,
                                                                     const int rho, float div,
                                                                     int lane, int drain) {
  if constexpr (KIND == WK_WALL && B == 1) {
    const bool w = in_lanes(t.lanes);
    return any_quotient(div, w ? 1.0f / 3.0f : 0.25f, w ? 3.0f : 4.0f);
  }
  if constexpr (KIND == WK_ANY) {
    const uint32_t c = t.cls[rho] >> (16 * B);
    const float s = (float)(c & 255u), y = (float)((c >> 8) & 255u) * (1.0f / 12.0f);
    float q = any_quotient(div, y, s);
    if constexpr (PM != PM_NONE) {
      if (t.enclosed) q = (c & 255u) == 0 ? div * __builtin_inff() : q;
    }
    return 2 * lane + B == drain ? -0.0f : q;
  }
  return div * 0.25f;
}

// The changes of the active cell's faces: `l`, `b` are added to its left and
// bottom face, `r`, `t` subtracted from its right and top face.  For an odd
// cell the right face's is taken by the next lane, which masks it.
template <int B, int KIND>
__device__ __attribute__((always_inline)) inline void face_changes(float d, uint32_t ml,
                                                                   uint32_t mr, uint32_t mb,
                                                                   uint32_t mt,
                                                                   unsigned long long lanes,
                                                                   float& l, float& r, float& b,
                                                                   float& t) {
  l = r = b = t = d;
  if constexpr (KIND == WK_WALL) {
    if constexpr (B == 0) {
      l = b = in_lanes(lanes) ? -0.0f : d;
      r = t = in_lanes(lanes) ? 0.0f : d;
    } else {
      l = in_lanes(lanes) ? -0.0f : d;
    }
  } else if constexpr (KIND == WK_DRAIN0 || (KIND == WK_DRAIN && B == 1)) {
    l = b = in_lanes(lanes) ? -0.0f : d;
    r = t = in_lanes(lanes) ? 0.0f : d;
  } else if constexpr (KIND == WK_ANY) {
    l = __uint_as_float((__float_as_uint(d) & ml) | (~ml & 0x80000000u));
    b = __uint_as_float((__float_as_uint(d) & mb) | (~mb & 0x80000000u));
    if constexpr (B == 0) r = __uint_as_float(__float_as_uint(d) & mr);
    t = __uint_as_float(__float_as_uint(d) & mt);
  }
}

// apply_projection_at for the active cell of row rho (parity B) of every
// lane.  Cells near the region edge compute with stale neighbours; their
// wrong values move one cell per phase and never reach the tile within a
// launch, so no lane or row is masked.  Cells that are not projected gather
// a meaningless pressure sum, which reg_store leaves out.
template <typename T, int R, int B, int PM, int KIND>
__device__ __attribute__((always_inline)) inline void reg_row(RegTile<R>& t, const int rho,
                                                              float vt0, float vt1, float& dtop,
                                                              const SweepParams& sq, int lane) {
  const int up = rho + 1 < R ? rho + 1 : rho;  // row above (when inside the strip)
  const bool inside = rho + 1 < R;
  float cl, cr, cb, ct;
  if constexpr (B == 0) {
    const uint32_t mtop = inside ? t.mv0[up] : t.mt0;
    const float uu = t.u0[rho], ur = t.u1[rho], vv = t.v0[rho];
    const float vt = inside ? t.v0[up] : vt0;
    const float div = ((ur - uu) + vt) - vv;
    const float q = kind_quotient<R, 0, PM, KIND>(t, rho, div, lane, sq.drain);
    const float d = sq.o * q;
    if constexpr (PM != PM_NONE) t.s0[rho] = pressure_add<PM>(t.s0[rho], d, sq);
    face_changes<0, KIND>(d, t.mu0[rho], t.mu1[rho], t.mv0[rho], mtop, t.lanes, cl, cr, cb, ct);
    float nu0 = uu + cl, nu1 = ur - cr;
    rnd2<T>(nu0, nu1);
    t.u0[rho] = nu0;
    t.u1[rho] = nu1;
    if (inside) {
      float nv = vv + cb, nt = vt - ct;
      rnd2<T>(nv, nt);
      t.v0[rho] = nv;
      t.v0[up] = nt;
    } else {
      t.v0[rho] = rnd<T>(vv + cb);
      dtop = ct;
    }
  } else {
    const uint32_t mtop = inside ? t.mv1[up] : t.mt1;
    const float uu = t.u1[rho], ur = lane_from_right(t.u0[rho]), vv = t.v1[rho];
    const float vt = inside ? t.v1[up] : vt1;
    const float div = ((ur - uu) + vt) - vv;
    const float q = kind_quotient<R, 1, PM, KIND>(t, rho, div, lane, sq.drain);
    const float d = sq.o * q;
    if constexpr (PM != PM_NONE) t.s1[rho] = pressure_add<PM>(t.s1[rho], d, sq);
    face_changes<1, KIND>(d, t.mu1[rho], 0, t.mv1[rho], mtop, t.lanes, cl, cr, cb, ct);
    cr = lane_from_left(cr);
    if constexpr (KIND == WK_ANY) cr = __uint_as_float(__float_as_uint(cr) & t.mu0[rho]);
    float nu1 = uu + cl, nu0 = t.u0[rho] - cr;
    rnd2<T>(nu1, nu0);
    t.u1[rho] = nu1;
    t.u0[rho] = nu0;
    if (inside) {
      float nv = vv + cb, nt = vt - ct;
      rnd2<T>(nv, nt);
      t.v1[rho] = nv;
      t.v1[up] = nt;
    } else {
      t.v1[rho] = rnd<T>(vv + cb);
      dtop = ct;
    }
  }
}

// LDS the wavefronts exchange rows through, two slots of each (consecutive
// phases use different slots).
template <int NW>
struct RegShared {
  float2 vrow[2][NW][64];  // row 0 (v0, v1) of each wavefront
  float dsend[2][NW][64];  // top-row update for the wavefront above
};

// What a wavefront has read of its neighbours' rows after a phase and not
// yet used: the update from below of its row 0, and row 0 of the wavefront above.
struct RowExchange {
  float dd;
  float2 x;
};

// The update from below reaches row 0.  PB is the parity of row 0's active
// cell in the coming phase, the one whose face the wavefront below moved.
template <typename T, int R, int PB>
__device__ __attribute__((always_inline)) inline void reg_settle(RegTile<R>& t,
                                                                 const RowExchange& x) {
  if constexpr (PB == 1)
    t.v1[0] = rnd<T>(t.v1[0] - x.dd);
  else
    t.v0[0] = rnd<T>(t.v0[0] - x.dd);
}

// Rows RHO..LAST of one phase, unrolled at compile time.
template <typename T, int R, int PB, int PM, int KIND, int RHO, int LAST>
__device__ __attribute__((always_inline)) inline void reg_rows_from(RegTile<R>& t, float vt0,
                                                                    float vt1, float& dtop,
                                                                    const SweepParams& sq,
                                                                    int lane) {
  if constexpr (RHO <= LAST) {
    reg_row<T, R, ((PB + RHO) & 1), PM, KIND>(t, RHO, vt0, vt1, dtop, sq, lane);
    reg_rows_from<T, R, PB, PM, KIND, RHO + 1, LAST>(t, vt0, vt1, dtop, sq, lane);
  }
}

// The rows of a phase: those inside the strip first, then the first and the
// last, which need what the exchange of the previous phase brings, so its
// latency is hidden.  (Active cells of adjacent rows share no face, so the
// order of the rows does not matter.)
template <typename T, int R, int PB, int PM, int KIND>
__device__ __attribute__((always_inline)) inline void reg_rows(RegTile<R>& t, const RowExchange& x,
                                                               float& dtop, const SweepParams& sq,
                                                               int lane) {
  reg_rows_from<T, R, PB, PM, KIND, 1, R - 2>(t, 0.0f, 0.0f, dtop, sq, lane);
  reg_settle<T, R, PB>(t, x);
  reg_row<T, R, PB, PM, KIND>(t, 0, 0.0f, 0.0f, dtop, sq, lane);
  reg_row<T, R, ((PB + R - 1) & 1), PM, KIND>(t, R - 1, x.x.x, x.x.y, dtop, sq, lane);
}

// One colour phase.  PB is the parity of the active cell in row 0 of this
// wavefront (compile time: phases come in pairs with PB and 1 - PB); with
// ACTIVE false the wavefront's rows stay as they are.
//
// The top faces of a wavefront's last row are row 0's of the wavefront
// above.  One barrier per phase: each wavefront publishes its row 0 after
// computing (this phase's own updates, before the one from below) beside
// dtop, the update its last row makes to the row above; after the barrier it
// reads both its neighbours'.  In the next phase it applies the update from
// below to its row 0.  The row above as it has been read lacks that update too,
// but only in the cells that its own last row does not touch in that phase: those
// of the other parity.  The slots alternate between phases, so none is
// rewritten before every reader of its previous contents has passed the next
// barrier.  reg_begin publishes and reads the rows as loaded.
template <typename T, int R, int NW, int PB, int SLOT, int PM, int KIND, bool ACTIVE>
__device__ __attribute__((always_inline)) inline void reg_phase(RegTile<R>& t, RegShared<NW>& sh,
                                                                RowExchange& x, int lane, int w,
                                                                const SweepParams& sq) {
  float dtop = 0.0f;
  if constexpr (ACTIVE)
    reg_rows<T, R, PB, PM, KIND>(t, x, dtop, sq, lane);
  else
    reg_settle<T, R, PB>(t, x);
  if (w > 0) sh.vrow[SLOT][w][lane] = make_float2(t.v0[0], t.v1[0]);
  if (w < NW - 1) sh.dsend[SLOT][w][lane] = dtop;
  __syncthreads();
  x.dd = w > 0 ? sh.dsend[SLOT][w - 1][lane] : 0.0f;
  x.x = w < NW - 1 ? sh.vrow[SLOT][w + 1][lane] : make_float2(0.0f, 0.0f);
}

// `pairs` pairs of phases.  A loop of its own for each kind keeps the rows in
// the same registers throughout (a choice inside the loop made the compiler
// copy them at every phase).
template <typename T, int R, int NW, int PB, int PM, int KIND, bool ACTIVE>
__device__ __attribute__((always_inline)) inline void reg_pairs(RegTile<R>& t, RegShared<NW>& sh,
                                                                RowExchange& x, int lane, int w,
                                                                int pairs,
                                                                const SweepParams& sq) {
  for (int i = 0; i < pairs; i++) {
    if constexpr (ACTIVE && KIND == WK_ANY) {
      // the masks do not change during the launch; hiding that from the
      // compiler keeps it from hoisting what it derives from them out of the
      // phase loop into registers
#pragma unroll
      for (int rho = 0; rho < R; rho++) {
        asm volatile("" : "+v"(t.mu0[rho]), "+v"(t.mu1[rho]));
        asm volatile("" : "+v"(t.mv0[rho]), "+v"(t.mv1[rho]), "+v"(t.cls[rho]));
      }
      asm volatile("" : "+v"(t.mt0), "+v"(t.mt1));
    }
    reg_phase<T, R, NW, PB, 1, PM, KIND, ACTIVE>(t, sh, x, lane, w, sq);
    reg_phase<T, R, NW, 1 - PB, 0, PM, KIND, ACTIVE>(t, sh, x, lane, w, sq);
  }
}

// This lane's index, re-read from the thread index so that it is not kept
// live across the sweeps.
__device__ inline int reg_lane() {
  int tid = (int)threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid & 63;
}

// Loads the region of u, v (and the pressure sums) and the gate bytes of
// the tile into registers: every load first, from the even column clamped
// into the row (so a pair stays inside its row of P cells) and the row
// clamped into the grid, with no branch, so a wavefront waits for HBM once
// rather than once per row.  Cells outside the grid are then set to 0.
template <typename T, int PM, int R>
__device__ __attribute__((always_inline)) inline void reg_load(RegTile<R>& t, const StepParams& sp,
                                                               const uint8_t* __restrict__ gates,
                                                               const T* __restrict__ u_in,
                                                               const T* __restrict__ v_in,
                                                               const float* __restrict__ p,
                                                               const RegArgs& a,
                                                               const RegPlace& pl) {
  const int lane = reg_lane();
  const int W = sp.W, H = sp.H, P = sp.P;
  const int gi = pl.gx0 + 2 * lane;
  const bool col0 = (unsigned)gi < (unsigned)W, col1 = (unsigned)(gi + 1) < (unsigned)W;
  // a scalar row pointer and one column offset for every access
  const unsigned gic = (unsigned)min(max(gi, 0), P - 2);
  uint32_t graw[R];
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const long row = (long)min(max(pl.gy0 + pl.rbase + rho, 0), H - 1) * P;
    load_pair(u_in + row, gic, true, true, t.u0[rho], t.u1[rho]);
    load_pair(v_in + row, gic, true, true, t.v0[rho], t.v1[rho]);
    graw[rho] = *reinterpret_cast<const uint16_t*>(gates + row + gic);
    if constexpr (PM != PM_NONE) {
      // the sums of the owned cells only; they start at 0 with the forces
      const int r = pl.rbase + rho;
      t.s0[rho] = t.s1[rho] = 0.0f;
      if (!a.forces && r >= pl.r0 && r < pl.r1) {
        const float2 pp = *reinterpret_cast<const float2*>(p + row + gic);
        t.s0[rho] = pp.x;
        t.s1[rho] = pp.y;
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // a wavefront inside the grid whose cells are all open needs no more
  const bool inside = pl.gx0 >= 0 && pl.gx0 + 128 <= W && pl.gy0 + pl.rbase >= 0 &&
                      pl.gy0 + pl.rbase + R <= H;
  uint32_t open = 0x0F0Fu;
#pragma unroll
  for (int rho = 0; rho < R; rho++) open &= graw[rho];
  t.enclosed = false;
  t.lanes = 0;
  if (inside && __all(open == 0x0F0Fu)) {
    t.kind = WK_OPEN;
  } else {
    // cells outside the grid hold 0 and closed faces
    bool same = true;
    unsigned long long even = 0, odd = 0, wall1 = ~0ULL, none0 = ~0ULL, none1 = ~0ULL;
#pragma unroll
    for (int rho = 0; rho < R; rho++) {
      const bool row_in = (unsigned)(pl.gy0 + pl.rbase + rho) < (unsigned)H;
      const bool in0 = row_in && col0, in1 = row_in && col1;
      t.u0[rho] = in0 ? t.u0[rho] : 0.0f;
      t.v0[rho] = in0 ? t.v0[rho] : 0.0f;
      t.u1[rho] = in1 ? t.u1[rho] : 0.0f;
      t.v1[rho] = in1 ? t.v1[rho] : 0.0f;
      // the gate bytes of cells 2l and 2l+1 (static, built with the flags)
      const uint32_t g0 = in0 ? (graw[rho] & 0xFFu) : 0u, g1 = in1 ? (graw[rho] >> 8) : 0u;
      t.gw[rho] = g0 | g1 << 8;
      const int n0 = __builtin_popcount(g0 & 15u), n1 = __builtin_popcount(g1 & 15u);
      if constexpr (PM != PM_NONE)
        t.enclosed |= __any(((g0 & G_UPD) && n0 == 0) || ((g1 & G_UPD) && n1 == 0));
      const unsigned long long open0 = __ballot(n0 == 4), open1 = __ballot(n1 == 4);
      if (rho == 0) {
        even = open0;
        odd = open1;
      }
      wall1 &= __ballot(n1 == 3 && !(g1 & G_L));
      same = same && even == open0 && odd == open1 && (__ballot(n0 != 0) & ~open0) == 0;
      none0 &= __ballot(n0 == 0);
      none1 &= __ballot(n1 == 0);
    }
    // lanes from the drain column's on
    const int drain = W - 1 - pl.gx0;
    const unsigned long long past = drain < 128 ? ~0ULL << (drain >> 1) : 0ULL;
    // (an enclosed cell has to show in the pressure)
    same = same && !t.enclosed;
    t.kind = WK_ANY;
    if (same && (even & odd) == ~0ULL) {
      t.kind = WK_OPEN;
    } else if (same && even == odd && wall1 == ~odd && drain >= 128) {
      t.kind = WK_WALL;
      t.lanes = ~odd;
    } else if (same && odd == ~past && none1 == past) {
      t.lanes = past;
      if ((drain & 1) && even == ~(past << 1))
        t.kind = WK_DRAIN;
      else if (!(drain & 1) && even == ~past && none0 == past)
        t.kind = WK_DRAIN0;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    t.u0[rho] = own_register(t.u0[rho]);
    t.v0[rho] = own_register(t.v0[rho]);
    t.u1[rho] = own_register(t.u1[rho]);
    t.v1[rho] = own_register(t.v1[rho]);
    if (a.forces) {  // the forces' results as stored (rounded to T)
      const int gj = pl.gy0 + pl.rbase + rho;
      const bool row_in = (unsigned)gj < (unsigned)H;
      if (row_in && col0) {
        force_uv(sp, gi, gj, t.u0[rho], t.v0[rho]);
        t.u0[rho] = rnd<T>(t.u0[rho]);
        t.v0[rho] = rnd<T>(t.v0[rho]);
      }
      if (row_in && col1) {
        force_uv(sp, gi + 1, gj, t.u1[rho], t.v1[rho]);
        t.u1[rho] = rnd<T>(t.u1[rho]);
        t.v1[rho] = rnd<T>(t.v1[rho]);
      }
    }
    if constexpr (PM != PM_NONE) {
      t.s0[rho] = own_register(t.s0[rho]);
      t.s1[rho] = own_register(t.s1[rho]);
    } else {
      t.s0[rho] = t.s1[rho] = 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);  // row by row: mixed, they would spill
  }
}

// The face masks and quotient classes of a wavefront of kind WK_ANY, from
// its gate bytes.  A face's two cells agree about it except at the drain
// column, whose left face only the cell to its left names.
template <int R>
__device__ __attribute__((always_inline)) inline void reg_masks(RegTile<R>& t) {
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const uint32_t g0 = t.gw[rho] & 0xFFu, g1 = t.gw[rho] >> 8;
    t.mu0[rho] = 0u - ((g0 | (lane_from_left_u(g1) >> 1)) & 1u);
    t.mu1[rho] = 0u - ((g0 >> 1) & 1u);
    t.mv0[rho] = 0u - ((g0 >> 2) & 1u);
    t.mv1[rho] = 0u - ((g1 >> 2) & 1u);
    if (rho == R - 1) {
      t.mt0 = 0u - ((g0 >> 3) & 1u);
      t.mt1 = 0u - ((g1 >> 3) & 1u);
    }
    t.cls[rho] = quotient_class(__builtin_popcount(g0 & 15u)) |
                 quotient_class(__builtin_popcount(g1 & 15u)) << 16;
  }
}

// Before the first phase: row 0 of the wavefront above, as loaded (a zero
// update leaves every value's bits).
template <int R, int NW>
__device__ __attribute__((always_inline)) inline RowExchange reg_begin(const RegTile<R>& t,
                                                                       RegShared<NW>& sh, int w,
                                                                       int lane) {
  RowExchange x;
  x.dd = 0.0f;
  if (w > 0) sh.vrow[0][w][lane] = make_float2(t.v0[0], t.v1[0]);
  __syncthreads();
  x.x = w < NW - 1 ? sh.vrow[0][w + 1][lane] : make_float2(0.0f, 0.0f);
  return x;
}

// `sweeps` sweeps over the registers of a wavefront of kind KIND, after
// reg_begin.  A wavefront takes part in a phase while some of its rows can
// still reach the tile: rows [r0 - 1 - e, r1 + e) with e phases to come.  So
// it sits out the last phases (all but an odd one, which does no harm).
// Colour 0 (even cells) comes first; row 0's active parity in a colour-0
// phase, PB, is that of its grid row, gy0 + rbase (gy0 is even).
template <typename T, int R, int NW, int PB, int PM, int KIND>
__device__ __attribute__((always_inline)) inline void reg_sweeps_from(RegTile<R>& t,
                                                                      RegShared<NW>& sh,
                                                                      RowExchange x, int lane,
                                                                      const RegPlace& pl,
                                                                      int sweeps,
                                                                      const SweepParams& sq) {
  const int idle = max(max(pl.r0 - pl.rbase - R, pl.rbase - pl.r1 + 1), 0);
  const int pairs = max(2 * sweeps - idle + 1, 0) / 2;
  reg_pairs<T, R, NW, PB, PM, KIND, true>(t, sh, x, lane, pl.w, pairs, sq);
  reg_pairs<T, R, NW, PB, PM, KIND, false>(t, sh, x, lane, pl.w, sweeps - pairs, sq);
  reg_settle<T, R, PB>(t, x);
}

template <typename T, int PM, int R, int NW, int KIND>
__device__ __attribute__((always_inline)) inline void reg_sweeps(RegTile<R>& t, RegShared<NW>& sh,
                                                                 const RowExchange& x,
                                                                 const StepParams& sp,
                                                                 const RegPlace& pl, int sweeps) {
  const int lane = reg_lane();
  SweepParams sq;
  sq.o = sp.o;
  sq.density = sp.density;
  sq.csf = (float)sp.cs;
  sq.pd = PressureDivisor{sp.d_t, sp.pdt_recip};
  sq.drain = sp.W - 1 - pl.gx0;
  if (R % 2 == 0 || (pl.rbase & 1) == 0)
    reg_sweeps_from<T, R, NW, 0, PM, KIND>(t, sh, x, lane, pl, sweeps, sq);
  else
    reg_sweeps_from<T, R, NW, 1, PM, KIND>(t, sh, x, lane, pl, sweeps, sq);
}

// Writes back the owned tile, and the pressure sums of its projected cells
// (with `forces`, 0 for the others, as the forces leave them).
template <typename T, int PM, int R>
__device__ __attribute__((always_inline)) inline void reg_store(const RegTile<R>& t,
                                                                const uint8_t* __restrict__ gates,
                                                                T* __restrict__ u_out,
                                                                T* __restrict__ v_out,
                                                                float* __restrict__ p,
                                                                const StepParams& sp,
                                                                const RegArgs& a,
                                                                const RegPlace& pl) {
  const int lane = reg_lane();
  const int W = sp.W, P = sp.P;
  const int gi = pl.gx0 + 2 * lane;
  // the owned columns start and end at pairs, but for an odd W
  const bool own0 = 2 * lane >= pl.c0 && 2 * lane < pl.c1;
  const bool own1 = own0 && gi + 1 < W;
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const int r = pl.rbase + rho;
    if (r < pl.r0 || r >= pl.r1) continue;
    const long row = (long)(pl.gy0 + r) * P;
    const unsigned gk = (unsigned)gi;  // owned cells lie in the grid
    store_pair(u_out + row, gk, own0, own1, own_register(t.u0[rho]), own_register(t.u1[rho]));
    store_pair(v_out + row, gk, own0, own1, own_register(t.v0[rho]), own_register(t.v1[rho]));
    if constexpr (PM != PM_NONE) {
      if (own0) {
        const uint32_t g = *reinterpret_cast<const uint16_t*>(gates + row + gk);
        const bool upd0 = (g & G_UPD) != 0, upd1 = own1 && (g & (G_UPD << 8)) != 0;
        if (upd0 || a.forces) p[row + gk] = upd0 ? t.s0[rho] : 0.0f;
        if (upd1 || (own1 && a.forces)) p[row + gk + 1] = upd1 ? t.s1[rho] : 0.0f;
      }
    }
  }
}

// One launch of the register-resident projection for tile `tile` (row-major
// over the grid's ntx tiles per row), run by a workgroup of 64 * NW threads.
// From the load on each kind of wavefront runs code of its own, with the same
// barriers.
template <typename T, int PM, int R, int NW, int KIND>
__device__ __attribute__((always_inline)) inline void project_regs_kind(
    RegTile<R>& t, const StepParams& sp, const uint8_t* __restrict__ gates, T* __restrict__ u_out,
    T* __restrict__ v_out, float* __restrict__ p, const RegArgs& a, const RegPlace& pl,
    RegShared<NW>& sh) {
  if constexpr (KIND == WK_ANY) reg_masks<R>(t);
  const RowExchange x = reg_begin<R, NW>(t, sh, pl.w, reg_lane());
  reg_sweeps<T, PM, R, NW, KIND>(t, sh, x, sp, pl, a.sweeps);
  reg_store<T, PM, R>(t, gates, u_out, v_out, p, sp, a, pl);
}

template <typename T, int PM, int R, int NW>
__device__ __attribute__((always_inline)) inline void project_regs_tile(
    const StepParams& sp, const uint8_t* __restrict__ gates, const T* __restrict__ u_in,
    const T* __restrict__ v_in, T* __restrict__ u_out, T* __restrict__ v_out,
    float* __restrict__ p, const RegArgs& a, int tile, RegShared<NW>& sh) {
  const RegPlace pl = reg_place<R, NW>(a, tile, sp.W, sp.H);
  RegTile<R> t;
  reg_load<T, PM, R>(t, sp, gates, u_in, v_in, p, a, pl);
  if (t.kind == WK_OPEN)
    project_regs_kind<T, PM, R, NW, WK_OPEN>(t, sp, gates, u_out, v_out, p, a, pl, sh);
  else if (t.kind == WK_WALL)
    project_regs_kind<T, PM, R, NW, WK_WALL>(t, sp, gates, u_out, v_out, p, a, pl, sh);
  else if (t.kind == WK_DRAIN)
    project_regs_kind<T, PM, R, NW, WK_DRAIN>(t, sp, gates, u_out, v_out, p, a, pl, sh);
  else if (t.kind == WK_DRAIN0)
    project_regs_kind<T, PM, R, NW, WK_DRAIN0>(t, sp, gates, u_out, v_out, p, a, pl, sh);
  else
    project_regs_kind<T, PM, R, NW, WK_ANY>(t, sp, gates, u_out, v_out, p, a, pl, sh);
}

// ---- halo exchange of the resident kernel --------------------------------------
//
// Between stages a tile's halo comes from its neighbours through an exchange
// buffer of three slots of 8-byte words, each a cell pair's values: in
// binary32 one word (u0, u1) and one (v0, v1), in 16 bits one word for all
// four.  A word is its own flag: a slot's words hold kNoWord until the owner
// stores them and again once they have been read, so a reader polls the data
// itself and one store and one load carry a value between two CUs (a
// separate flag would add a wait for the stores, a barrier and a second
// round trip).  Words are written and read with relaxed agent-scope atomics,
// which bypass the caches that are not coherent between CUs and XCDs (a CU's
// L1, an XCD's L2); each word is single-copy atomic, and no order between
// words is needed.
//
// Ring t (the cells a tile's neighbours read before stage t) uses slot
// (base + t) % 3; base is kept in device memory and moved on at the end of a
// launch, so that the first rings of the next launch find clean slots.  A
// tile clears ring t-1 once it has read all its neighbours' ring t: a
// neighbour publishes ring t only after it has read ring t-1.  The clearing
// stores have completed before the tile publishes ring t+1, and a neighbour
// looks for ring t+2, the slot's next use, only after it has read ring t+1,
// so it never takes an old word for a new one.  The last ring of a launch is
// the one left to clear ("ring 0" of the next launch).
//
// A slot holds the region of every tile, a row of 64 words per region row
// and word kind, so that a wavefront's rows lie at constant offsets from one
// address (what bounds the exchange is instructions: the 16 wavefronts of a
// tile issue all of it between two sweeps).  A tile stores its ring at its
// own cells' places; a reader finds the cell that lies `d` tiles over in
// that tile's region, tw / 2 pairs or th rows back.
typedef unsigned long long XWord;
constexpr XWord kNoWord = ~0ULL;  // by its low half
constexpr int kXSlots = 3;

// Words per cell pair.
template <typename T> constexpr int xwords() { return sizeof(T) == 4 ? 2 : 1; }

__device__ inline XWord xload(const XWord* a) {
  return __hip_atomic_load(a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore(XWord* a, XWord w) {
  __hip_atomic_store(a, w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A pair's values as words.  A low half of all ones is a NaN with a full
// payload (two in 16 bits); such a value travels with one payload bit
// cleared.
template <typename T>
__device__ inline void pack_words(XWord* w, float u0, float u1, float v0, float v1) {
  if constexpr (sizeof(T) == 4) {
    w[0] = (XWord)__float_as_uint(u1) << 32 | min(__float_as_uint(u0), 0xFFFFFFFEu);
    w[1] = (XWord)__float_as_uint(v1) << 32 | min(__float_as_uint(v0), 0xFFFFFFFEu);
  } else {
    const T e[4] = {Store<T>::st(u0), Store<T>::st(u1), Store<T>::st(v0), Store<T>::st(v1)};
    uint32_t h[2];
    __builtin_memcpy(h, e, 8);
    w[0] = (XWord)h[1] << 32 | min(h[0], 0xFFFFFFFEu);
  }
}

template <typename T>
__device__ inline void unpack_words(const XWord* w, float& u0, float& u1, float& v0, float& v1) {
  if constexpr (sizeof(T) == 4) {
    u0 = __uint_as_float((uint32_t)w[0]);
    u1 = __uint_as_float((uint32_t)(w[0] >> 32));
    v0 = __uint_as_float((uint32_t)w[1]);
    v1 = __uint_as_float((uint32_t)(w[1] >> 32));
  } else {
    T e[4];
    __builtin_memcpy(e, w, 8);
    u0 = Store<T>::ld(e[0]);
    u1 = Store<T>::ld(e[1]);
    v0 = Store<T>::ld(e[2]);
    v1 = Store<T>::ld(e[3]);
  }
}

// A tile's place in a slot, and what of this wavefront's rows takes part:
// one bit per row, and the lanes of a row.  Worked out once; choosing a row's
// lanes then takes a bit test.
struct XPlace {
  int tile, half;   // half: tw / 2
  long tile_row;    // bytes from a word to that of the same cell seen from the
                    // tile row above
  unsigned own, ring;      // rows owned; rows of the ring, all owned lanes
  unsigned below, above;   // halo rows owned by the tiles below and above
  unsigned in;             // rows inside the grid
  unsigned long long own_m, ring_m;  // owned lanes; those of the ring's strips
  unsigned long long halo_m;         // lanes of the halo's strips
};

template <typename T, int R, int NW>
__device__ inline XPlace x_place(const RegArgs& a, const RegPlace& pl, int tile) {
  constexpr long kTile = (long)xwords<T>() * NW * R * 512;
  XPlace x;
  x.tile = tile;
  x.half = a.tw / 2;
  x.tile_row = a.ntx * kTile - (long)a.th * 512;
  x.own = x.ring = x.below = x.above = x.in = 0;
  const int K2 = 2 * pl.K;
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const int r = pl.rbase + rho;
    const bool own = r >= pl.r0 && r < pl.r1;
    x.own |= (own ? 1u : 0u) << rho;
    x.ring |= (own && ((pl.below && r < pl.r0 + K2) || (pl.above && r >= pl.r1 - K2)) ? 1u : 0u)
              << rho;
    x.below |= (pl.below && r < pl.r0 ? 1u : 0u) << rho;
    x.above |= (pl.above && r >= pl.r1 ? 1u : 0u) << rho;
    x.in |= (r < pl.rows ? 1u : 0u) << rho;
  }
  const int lane = reg_lane(), c = 2 * lane;
  const bool own = c >= pl.c0 && c < pl.c1;
  x.own_m = __ballot(own);
  x.ring_m = __ballot(own && ((pl.left && c < pl.c0 + K2) || (pl.right && c >= pl.c1 - K2)));
  x.halo_m = __ballot((pl.left && lane < pl.K) || (pl.right && lane >= 64 - pl.K));
  return x;
}

template <class Word>
__device__ inline Word* x_at(Word* slot, unsigned bytes) {
  return (Word*)((typename std::conditional<std::is_const<Word>::value, const char*, char*>::type)
                     slot + bytes);
}

// Stores the tile's ring in `slot`: the owned cells within 2k of a side that
// has a neighbour.  CLEAR stores kNoWord instead.
template <typename T, int R, int NW, bool CLEAR>
__device__ __attribute__((always_inline)) inline void ring_store(const RegTile<R>& t, XWord* slot,
                                                                 const XPlace& x,
                                                                 const RegPlace& pl) {
  constexpr int NWD = xwords<T>();
  constexpr unsigned kPlane = NW * R * 512u;  // bytes
  const unsigned at = (unsigned)x.tile * (NWD * kPlane) + (unsigned)(pl.rbase * 64 + reg_lane()) * 8u;
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    unsigned long long m = (x.ring >> rho) & 1u ? x.own_m : x.ring_m;
    if (!((x.own >> rho) & 1u)) m = 0;
    if (in_lanes(m)) {
      XWord w[NWD];
      if constexpr (!CLEAR)
        pack_words<T>(w, own_register(t.u0[rho]), own_register(t.u1[rho]),
                      own_register(t.v0[rho]), own_register(t.v1[rho]));
#pragma unroll
      for (int i = 0; i < NWD; i++)
        xstore(x_at(slot, at + i * kPlane) + rho * 64, CLEAR ? kNoWord : w[i]);
    }
  }
}

// Lanes of row rho that are halo, inside the grid.
__device__ inline unsigned long long halo_lanes(const XPlace& x, int rho) {
  const unsigned long long m =
      ((x.below | x.above) >> rho) & 1u ? x.own_m | x.halo_m : x.halo_m;
  return (x.in >> rho) & 1u ? m : 0ULL;
}

// Replaces u and v of the halo (the region's cells outside the owned ones,
// inside the grid) by the neighbours' rings in `slot`, waiting for them.
// Every load of a poll is issued before the first is looked at.  A wait ends
// with the words, after spin_ticks of wall clock (the error word is set), or
// as soon as another wait of the launch has timed out.
template <typename T, int R, int NW>
__device__ __attribute__((always_inline)) inline void ring_load(RegTile<R>& t, const XWord* slot,
                                                                const XPlace& x,
                                                                const RegPlace& pl, int* error,
                                                                long long spin_ticks) {
  constexpr int NWD = xwords<T>();
  constexpr unsigned kPlane = NW * R * 512u;  // bytes
  const int lane = reg_lane();
  const int dx = pl.left && lane < pl.K ? -1 : pl.right && lane >= 64 - pl.K ? 1 : 0;
  unsigned at = (unsigned)(x.tile + dx) * (NWD * kPlane) +
                (unsigned)(pl.rbase * 64 + lane - dx * x.half) * 8u;
  // where the tiles below and above have this wavefront's rows
  const XWord* lo = (const XWord*)((const char*)slot - x.tile_row);
  const XWord* hi = (const XWord*)((const char*)slot + x.tile_row);
  const long long t0 = wall_clock64();
  // at most six rows at a time, so that their words do not spill
  constexpr int kRows = R <= 6 ? R : (R + 1) / 2;
#pragma unroll
  for (int r0 = 0; r0 < R; r0 += kRows) {
    XWord w[kRows][NWD];
#pragma unroll
    for (int i = 0; i < kRows * NWD; i++) w[i / NWD][i % NWD] = 0;
    // poll one row until it is there, then all: the others mostly are, too
    for (int first = kRows - 1;;) {
      uint32_t most = 0;
      asm volatile("" : "+v"(at));  // no address per row kept across polls
#pragma unroll
      for (int q = 0; q < kRows; q++) {
        const int rho = r0 + q;
        if (q < first || rho >= R) continue;
        const XWord* from = (x.below >> rho) & 1u ? lo : (x.above >> rho) & 1u ? hi : slot;
        if (in_lanes(halo_lanes(x, rho)))
#pragma unroll
          for (int i = 0; i < NWD; i++) w[q][i] = xload(x_at(from, at + i * kPlane) + rho * 64);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kRows * NWD; i++) most = max(most, (uint32_t)w[i / NWD][i % NWD]);
      if (!__any(most == (uint32_t)kNoWord)) {
        if (first == 0) break;
        first = 0;
        continue;
      }
      if (__hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
      if (wall_clock64() - t0 > spin_ticks) {
        __hip_atomic_store(error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
#pragma unroll
    for (int q = 0; q < kRows; q++) {
      const int rho = r0 + q;
      if (rho >= R) continue;
      const bool halo = in_lanes(halo_lanes(x, rho));
      float u0, u1, v0, v1;
      unpack_words<T>(w[q], u0, u1, v0, v1);
      t.u0[rho] = halo ? u0 : t.u0[rho];
      t.u1[rho] = halo ? u1 : t.u1[rho];
      t.v0[rho] = halo ? v0 : t.v0[rho];
      t.v1[rho] = halo ? v1 : t.v1[rho];
    }
  }
}

}  // namespace osy
