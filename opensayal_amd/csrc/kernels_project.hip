// kernels_project.hip - over-relaxed red-black projection (src/fluid.cu:229-295).
//
// A sweep is the even colour phase ((i+j) even) then the odd one, over
// interior fluid cells.  Same-colour cells share no face, so every colour
// phase is a set of independent cell updates and any schedule that finishes
// one phase before the next starts reproduces the reference bit for bit.
//
// Four kernels.  A handle starts with k_project_regs (default_tuning); the
// autotuner times all four, and any of them can be set.
//  * k_project_regs: k sweeps per launch on a 128-cell wide region held in
//    registers (projection_device.hpp).
//  * k_project_resident: the same regions kept in registers for all n sweeps of
//    one launch, with halos exchanged between the tiles every k sweeps.
//  * k_project_colour: one launch per colour phase, in place (2n launches);
//    the plain restatement.
//  * k_project_tiled: temporal blocking in LDS.  A workgroup loads its tile plus a
//    halo of u, v and cell flags into LDS, runs up to k sweeps there, and
//    writes the tile to the other half of a ping-pong pair.  A colour phase
//    changes only faces of the cells it updates, so a value can be wrong
//    after phase s only within s cells of the region edge; a halo of 2k
//    cells keeps every face of the tile exact through 2k phases.  Each phase
//    updates only the cells whose results still reach the tile (a box that
//    shrinks by one cell per phase), so the redundant halo work falls off as
//    the sweeps proceed.
#include "projection.hpp"
#include "projection_device.hpp"

#pragma clang fp contract(off)

namespace osy {
namespace {

// apply_projection_at + update_pressure_at (src/fluid.cu:221-262) for the
// cell at k = j*P + i, given its flag byte.  Face gates: the reference checks
// !is_solid of the neighbour across each face; for a fluid cell that is the
// face's fluid-fluid flag (CF_FU of (i,j) and (i+1,j), CF_FV of (i,j) and
// (i,j+1)).
template <typename T>
__device__ inline void project_cell(const StepParams& sp, const uint8_t* flags, T* u, T* v,
                                    float* p, long k, uint8_t f) {
  const int P = sp.P;
  const float uu = ldf(u, k), ur = ldf(u, k + 1);
  const float vv = ldf(v, k), vt = ldf(v, k + P);
  const float div = ((ur - uu) + vt) - vv;
  const float vd = sp.o * (div / (float)cf_total_s(f));
  if (sp.pressure_on) p[k] = p[k] + (((vd * sp.density) * (float)sp.cs) / sp.d_t);
  if (f & CF_FU) stf(u, k, uu + vd);
  if (flags[k + 1] & CF_FU) stf(u, k + 1, ur - vd);
  if (f & CF_FV) stf(v, k, vv + vd);
  if (flags[k + P] & CF_FV) stf(v, k + P, vt - vd);
}

// One colour phase; thread (t, j) owns cell i = 2t + ((j + colour) & 1),
// the mapping of apply_projection_even/odd_kernel (src/fluid.cu:264-280).
template <typename T>
__global__ void __launch_bounds__(256) k_project_colour(StepParams sp, const uint8_t* flags, T* u,
                                                        T* v, float* p, int colour) {
  const int j = blockIdx.y * 4 + threadIdx.y;
  const int i = 2 * (int)(blockIdx.x * 64 + threadIdx.x) + ((j + colour) & 1);
  if (i < 1 || i > sp.W - 2 || j < 1 || j > sp.H - 2) return;
  const long k = (long)j * sp.P + i;
  const uint8_t f = flags[k];
  if (!(f & CF_UPD)) return;
  project_cell(sp, flags, u, v, p, k, f);
}

// ---- tiled kernel ----------------------------------------------------------

struct TiledArgs {
  int tw, th, k;  // owned tile, sweeps per launch (halo 2k)
  int pw, rh;     // region: pw cell pairs (2*pw cells) x rh rows
  int wpr;        // wavefronts per region row
  int ntx;        // tiles per grid row
  int sweeps;     // sweeps this launch (<= k)
  int forces;     // apply the velocity forces on load, pressure sums from 0
};

// LDS layout: U, V (and the pressure sums S) hold rh rows of two half-rows,
// the even columns of the region row then the odd ones, so the lanes that
// update one colour of a row touch consecutive words.  Lane l of column
// block cb handles cell pair q = 64*cb + l of every row its wavefront visits.
template <typename T, bool PRESSURE>
__global__ void __launch_bounds__(kTileThreads)
    k_project_tiled(StepParams sp, const uint8_t* __restrict__ flags, const T* __restrict__ u_in,
                    const T* __restrict__ v_in, T* __restrict__ u_out, T* __restrict__ v_out,
                    float* __restrict__ p, TiledArgs a) {
  extern __shared__ __align__(16) char smem[];
  const int pw = a.pw, rh = a.rh, K = a.k;
  const int pwp = pw + 1;
  const int rs = 2 * pwp;  // LDS row stride (elements)
  const int rw = 2 * pw;   // region width (cells)
  const int fs = rw + 1;   // flag row stride (bytes)
  const int ncell = rh * rs;
  float* U = (float*)smem;
  float* V = U + ncell;
  float* S = V + ncell;  // pressure sums (PRESSURE only)
  uint8_t* G = (uint8_t*)(PRESSURE ? S + ncell : V + ncell);
  uint8_t* F = G + ncell;

  const int lane = threadIdx.x & 63;
  // wavefront-uniform values live in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cb = wave % a.wpr;             // column block of this wavefront
  const int r0 = wave / a.wpr;             // its first row
  const int rstep = kTileWaves / a.wpr;    // its row stride
  const int q = cb * 64 + lane;            // this lane's cell pair
  const bool lane_on = q < pw;

  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int tx = tile % a.ntx, ty = tile / a.ntx;
  const int x0 = tx * a.tw, y0 = ty * a.th;
  const int gx0 = x0 - 2 * K, gy0 = y0 - 2 * K;  // region origin; gx0 is even
  const int W = sp.W, H = sp.H, P = sp.P;

  // flags of the region plus one column right and one row above
  for (int r = r0; r <= rh; r += rstep) {
    const int gj = gy0 + r;
    const bool row_in = (unsigned)gj < (unsigned)H;
    if (lane_on) {
#pragma unroll
      for (int b = 0; b < 2; b++) {
        const int gi = gx0 + 2 * q + b;
        F[r * fs + 2 * q + b] =
            (row_in && (unsigned)gi < (unsigned)W) ? flags[(long)gj * P + gi] : (uint8_t)0;
      }
    }
  }
  for (int r = threadIdx.x; r <= rh; r += kTileThreads) {
    const int gi = gx0 + rw, gj = gy0 + r;
    F[r * fs + rw] = ((unsigned)gi < (unsigned)W && (unsigned)gj < (unsigned)H)
                         ? flags[(long)gj * P + gi]
                         : (uint8_t)0;
  }
  // u, v (and pressure) of the region
  for (int r = r0; r < rh; r += rstep) {
    if (!lane_on) break;
    const int gj = gy0 + r;
    const int gi = gx0 + 2 * q;
    const bool row_in = (unsigned)gj < (unsigned)H;
    const bool in0 = row_in && (unsigned)gi < (unsigned)W;
    const bool in1 = row_in && (unsigned)(gi + 1) < (unsigned)W;
    const long gk = (long)gj * P + gi;
    float a0, a1, b0, b1;
    const int l0 = r * rs + q, l1 = l0 + pwp;
    load_pair(u_in, gk, in0, in1, a0, a1);
    load_pair(v_in, gk, in0, in1, b0, b1);
    if (a.forces) {  // the forces' results as stored (rounded to T)
      if (in0) force_uv(sp, gi, gj, a0, b0);
      if (in1) force_uv(sp, gi + 1, gj, a1, b1);
      a0 = rnd<T>(a0);
      a1 = rnd<T>(a1);
      b0 = rnd<T>(b0);
      b1 = rnd<T>(b1);
    }
    U[l0] = a0;
    U[l1] = a1;
    V[l0] = b0;
    V[l1] = b1;
    if constexpr (PRESSURE) {
      S[l0] = (in0 && !a.forces) ? p[gk] : 0.0f;
      S[l1] = (in1 && !a.forces) ? p[gk + 1] : 0.0f;
    }
  }
  __syncthreads();
  // gate bytes
  for (int r = r0; r < rh; r += rstep) {
    if (!lane_on) break;
#pragma unroll
    for (int b = 0; b < 2; b++) {
      const int lc = 2 * q + b;
      const uint8_t f = F[r * fs + lc];
      const uint8_t fr = F[r * fs + lc + 1];
      const uint8_t ft = F[(r + 1) * fs + lc];
      uint32_t g = 0;
      if (f & CF_UPD) {
        g = G_UPD;
        if (f & CF_FU) g |= G_L;
        if (fr & CF_FU) g |= G_R;
        if (f & CF_FV) g |= G_B;
        if (ft & CF_FV) g |= G_T;
        const int s = cf_total_s(f);
        if (s == 0 || s == 3)
          g |= G_SLOW;
        else
          g |= (uint32_t)(s >> 1) << G_L2_SHIFT;
      }
      G[r * rs + b * pwp + q] = (uint8_t)g;
    }
  }
  __syncthreads();

  const float o = sp.o;
  const int nphase = 2 * a.sweeps;
  for (int s = 0; s < nphase; s++) {
    const int c = s & 1;           // even cells first, as the reference
    const int e = nphase - 1 - s;  // phases still to come after this one
    const int lo = 2 * K - 1 - e;  // box of cells that still reach the tile
    const int chi = 2 * K + a.tw + e;
    const int rhi = 2 * K + a.th + e;
    int r = r0;
    if (lo > r0) r += ((lo - r0 + rstep - 1) / rstep) * rstep;
    // the pair's cell of colour c alternates with the row; b and the offset
    // of u(i+1) are the same for every lane of a row
    int b = (c + gy0 + r) & 1;
    const int bstep = rstep & 1;
    int own = r * rs + q + b * pwp;
    for (; r < rhi; r += rstep) {
      const int lc = 2 * q + b;
      if (lane_on && lc >= lo && lc < chi) {
        // every face a cell of this colour touches is touched by no other
        // cell of the phase, so the four writes are unconditional
        const int right = b ? own - pwp + 1 : own + pwp;  // u(i+1): next pair's even cell
        const int top = own + rs;
        const uint32_t g = G[own];
        const float uu = U[own], ur = U[right], vv = V[own], vt = V[top];
        const float div = ((ur - uu) + vt) - vv;
        const float d = relaxed_quotient(div, g, o);
        if constexpr (PRESSURE) {
          if (g & G_UPD) S[own] = S[own] + (((d * sp.density) * (float)sp.cs) / sp.d_t);
        }
        U[own] = rnd<T>(gated_add(uu, d, g, 0));
        U[right] = rnd<T>(gated_sub(ur, d, g, 1));
        V[own] = rnd<T>(gated_add(vv, d, g, 2));
        V[top] = rnd<T>(gated_sub(vt, d, g, 3));
      }
      own += bstep ? (b ? rstep * rs - pwp : rstep * rs + pwp) : rstep * rs;
      b ^= bstep;
    }
    __syncthreads();
  }

  // write back the owned tile
  for (int r = r0 + ((2 * K - r0 + rstep - 1) / rstep) * rstep; r < 2 * K + a.th; r += rstep) {
    if (!lane_on) break;
    const int gj = gy0 + r;
    if (gj >= H) break;
    const int lc = 2 * q;
    const int gi = gx0 + lc;
    const bool in0 = lc >= 2 * K && lc < 2 * K + a.tw && gi < W;
    const bool in1 = lc + 1 >= 2 * K && lc + 1 < 2 * K + a.tw && gi + 1 < W;
    if (!in0 && !in1) continue;
    const long gk = (long)gj * P + gi;
    const int l0 = r * rs + q, l1 = l0 + pwp;
    store_pair(u_out, gk, in0, in1, U[l0], U[l1]);
    store_pair(v_out, gk, in0, in1, V[l0], V[l1]);
    if constexpr (PRESSURE) {
      if (in0) p[gk] = S[l0];
      if (in1) p[gk + 1] = S[l1];
    }
  }
}

// Eight wavefronts hold 4, 8 or 10 rows each, sixteen hold taller regions
// (reg_waves): so a CU always has four wavefronts per SIMD to hide latency
// with (six at 4 rows), within 128 VGPRs (80 at 4 rows).  The compiler keeps to
// that by spilling: 8 rows without sums 6 to 8 values, 10 rows 39, with sums
// 8 rows 56 to 81 and 4 rows 13 to 17, nearly all of them at the load, the
// classification and the store, none in the phases of binary32; the resident
// kernels with sums 11 to 41, around the exchange of a stage as well.
template <int R, int NW> constexpr int reg_waves_per_simd() { return R == 4 && NW == 8 ? 6 : 4; }

template <typename T, int PM, int R, int NW>
__global__ void __launch_bounds__(64 * NW, (reg_waves_per_simd<R, NW>()))
    k_project_regs(StepParams sp, const uint8_t* __restrict__ gates, const T* __restrict__ u_in,
                   const T* __restrict__ v_in, T* __restrict__ u_out, T* __restrict__ v_out,
                   float* __restrict__ p, RegArgs a) {
  __shared__ RegShared<NW> sh;
  project_regs_tile<T, PM, R, NW>(sp, gates, u_in, v_in, u_out, v_out, p, a,
                                        xcd_tile(blockIdx.x, gridDim.x), sh);
}

template <typename T, bool PRESSURE>
void launch_tiled(const StepParams& sp, const GridView& g, const FieldPtrs& f, int* cur,
                  const ProjTuning& t, hipStream_t s) {
  TiledArgs a;
  a.tw = t.tw;
  a.th = t.th;
  a.k = t.k;
  a.pw = t.pw();
  a.rh = t.region_h();
  a.wpr = t.waves_per_row();
  a.ntx = (sp.W + a.tw - 1) / a.tw;
  const int nty = (sp.H + a.th - 1) / a.th;
  const size_t lds = t.lds_bytes(PRESSURE);
  for (int done = 0; done < sp.n; done += t.k) {
    a.sweeps = (sp.n - done < t.k) ? sp.n - done : t.k;
    a.forces = (done == 0 && sp.forces_in_projection) ? 1 : 0;
    const int nxt = 1 - *cur;
    hipLaunchKernelGGL((k_project_tiled<T, PRESSURE>), dim3(a.ntx * nty), dim3(kTileThreads), lds,
                       s, sp, g.flags, (const T*)f.u[*cur], (const T*)f.v[*cur], (T*)f.u[nxt],
                       (T*)f.v[nxt], f.p, a);
    *cur = nxt;
  }
}

// ---- resident kernel ---------------------------------------------------------
//
// All n sweeps in one launch: one workgroup per tile keeps its region in
// registers from the first sweep to the last.  The sweeps run in stages of
// k (the last stage takes the rest); after a stage the owned cells are
// exact and the halo is stale, so the workgroup stores the ring of owned
// cells its neighbours read as halo in the exchange buffer and takes its own
// halo from theirs (projection_device.hpp, "halo exchange").  The fields
// are read once, at the start, from buffer u_in, v_in and written once, at
// the end, to u_out, v_out.
//
// Every tile's workgroup must be resident at once (the host checks the
// tile count, ProjTuning::resident_plan); a wait is bounded by spin_ticks,
// after which the error word is set and the launch drains without waiting.
constexpr int kWaitVm = 0x0F70;  // s_waitcnt vmcnt(0)

struct ResidentArgs {
  int nstages;      // ceil(n / k)
  int last_sweeps;  // sweeps of the last stage
  XWord* slots;     // kXSlots slots of slot_words words
  long slot_words;
  unsigned* state;  // finished workgroups; slot of "ring 0"
  int* error;
  long long spin_ticks;
};

// All stages of a wavefront of kind KIND, and the store of its rows.
template <typename T, int PM, int R, int NW, int KIND>
__device__ __attribute__((always_inline)) inline void resident_kind(
    RegTile<R>& t, const StepParams& sp, const uint8_t* __restrict__ gates, T* __restrict__ u_out,
    T* __restrict__ v_out, float* __restrict__ p, const RegArgs& a, const ResidentArgs& ra,
    const RegPlace& pl, const XPlace& x, int base, RegShared<NW>& sh) {
  if constexpr (KIND == WK_ANY) reg_masks<R>(t);
  for (int s = 0; s < ra.nstages; s++) {
    if (s > 0) {
      XWord* ring = ra.slots + (long)((base + s) % kXSlots) * ra.slot_words;
      ring_store<T, R, NW, false>(t, ring, x, pl);
      ring_load<T, R, NW>(t, ring, x, pl, ra.error, ra.spin_ticks);
    }
    // the barrier in reg_begin: every wavefront has read its part of ring s
    const RowExchange rx = reg_begin<R, NW>(t, sh, pl.w, reg_lane());
    // no load is outstanding here; saying so keeps the compiler from waiting
    // for one, and so for the clearing stores below, in the sweeps
    __builtin_amdgcn_s_waitcnt(kWaitVm);
    if (s > 0)
      ring_store<T, R, NW, true>(t, ra.slots + (long)((base + s - 1) % kXSlots) * ra.slot_words,
                                 x, pl);
    reg_sweeps<T, PM, R, NW, KIND>(t, sh, rx, sp, pl,
                                         s + 1 == ra.nstages ? ra.last_sweeps : a.k);
    // this wavefront's clearing stores have completed before it publishes
    __builtin_amdgcn_s_waitcnt(kWaitVm);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
  }
  reg_store<T, PM, R>(t, gates, u_out, v_out, p, sp, a, pl);
}

template <typename T, int PM, int R, int NW>
__global__ void __launch_bounds__(64 * NW, (reg_waves_per_simd<R, NW>()))
    k_project_resident(StepParams sp, const uint8_t* __restrict__ gates,
                       const T* __restrict__ u_in, const T* __restrict__ v_in,
                       T* __restrict__ u_out, T* __restrict__ v_out, float* __restrict__ p,
                       RegArgs a, ResidentArgs ra) {
  __shared__ RegShared<NW> sh;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const RegPlace pl = reg_place<R, NW>(a, tile, sp.W, sp.H);
  const XPlace x = x_place<T, R, NW>(a, pl, tile);
  const int base = __builtin_amdgcn_readfirstlane((int)ra.state[1]);
  RegTile<R> t;
  reg_load<T, PM, R>(t, sp, gates, u_in, v_in, p, a, pl);
  if (t.kind == WK_OPEN)
    resident_kind<T, PM, R, NW, WK_OPEN>(t, sp, gates, u_out, v_out, p, a, ra, pl, x, base,
                                               sh);
  else if (t.kind == WK_WALL)
    resident_kind<T, PM, R, NW, WK_WALL>(t, sp, gates, u_out, v_out, p, a, ra, pl, x, base,
                                               sh);
  else if (t.kind == WK_DRAIN)
    resident_kind<T, PM, R, NW, WK_DRAIN>(t, sp, gates, u_out, v_out, p, a, ra, pl, x, base,
                                                sh);
  else if (t.kind == WK_DRAIN0)
    resident_kind<T, PM, R, NW, WK_DRAIN0>(t, sp, gates, u_out, v_out, p, a, ra, pl, x, base,
                                                 sh);
  else
    resident_kind<T, PM, R, NW, WK_ANY>(t, sp, gates, u_out, v_out, p, a, ra, pl, x, base,
                                              sh);
  // the last workgroup to finish moves "ring 0" to the ring left uncleared
  if (threadIdx.x == 0 && __hip_atomic_fetch_add(ra.state, 1u, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
    __hip_atomic_store(ra.state, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ra.state + 1, (unsigned)((base + ra.nstages - 1) % kXSlots),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The shapes' kernels, by region rows / 8 (resident ones:
// ProjTuning::resident_plan).
template <typename T, int PM>
const void* resident_kernel(int rows) {
  return rows == 4 ? (const void*)k_project_resident<T, PM, 4, 8>
                   : (const void*)k_project_resident<T, PM, 6, 16>;  // 12
}

template <typename T, int PM>
const void* regs_kernel(int rows) {
  if (rows == 4) return (const void*)k_project_regs<T, PM, 4, 8>;
  if (rows == 8) return (const void*)k_project_regs<T, PM, 8, 8>;
  switch (PM == PM_NONE ? rows : 0) {
    case 10: return (const void*)k_project_regs<T, PM_NONE, 10, 8>;
    case 12: return (const void*)k_project_regs<T, PM_NONE, 6, 16>;
    case 16: return (const void*)k_project_regs<T, PM_NONE, 8, 16>;
    default: return nullptr;
  }
}

RegArgs reg_args(const StepParams& sp, const ProjTuning& t) {
  RegArgs a;
  a.tw = t.tw;
  a.th = t.th;
  a.k = t.k;
  a.ntx = t.tiles_x(sp.W);
  a.nty = t.tiles_y(sp.H);
  a.inset = 0;
  a.sweeps = t.k;
  a.forces = sp.forces_in_projection ? 1 : 0;
  return a;
}

template <typename T, int PM>
void launch_resident(const StepParams& sp, const FieldPtrs& f, int* cur, const ProjTuning& t,
                     hipStream_t s) {
  if (sp.n <= 0) return;
  RegArgs a = reg_args(sp, t);
  ResidentArgs ra;
  ra.nstages = (sp.n + t.k - 1) / t.k;
  ra.last_sweeps = sp.n - (ra.nstages - 1) * t.k;
  ra.slots = (XWord*)f.exchange;
  ra.slot_words = t.exchange_words(sp.W, sp.H, sizeof(T));
  ra.state = f.rstate;
  ra.error = f.error;
  ra.spin_ticks = sp.spin_ticks;
  const int in = *cur, other = 1 - in;
  const T* u0 = (const T*)f.u[in];
  const T* v0 = (const T*)f.v[in];
  T* u1 = (T*)f.u[other];
  T* v1 = (T*)f.v[other];
  void* args[] = {(void*)&sp, (void*)&f.gates, (void*)&u0, (void*)&v0, (void*)&u1,
                  (void*)&v1, (void*)&f.p, (void*)&a, (void*)&ra};
  (void)hipLaunchKernel(resident_kernel<T, PM>(t.reg_rows()), dim3(a.ntx * a.nty),
                        dim3(64 * reg_waves(t.reg_rows())), args, 0, s);
  *cur = other;
}

template <typename T, int PM>
void launch_regs(const StepParams& sp, const FieldPtrs& f, int* cur, const ProjTuning& t,
                 hipStream_t s) {
  RegArgs a = reg_args(sp, t);
  for (int done = 0; done < sp.n; done += t.k) {
    a.sweeps = (sp.n - done < t.k) ? sp.n - done : t.k;
    if (done > 0) a.forces = 0;
    const int nxt = 1 - *cur;
    const T* u0 = (const T*)f.u[*cur];
    const T* v0 = (const T*)f.v[*cur];
    T* u1 = (T*)f.u[nxt];
    T* v1 = (T*)f.v[nxt];
    void* args[] = {(void*)&sp, (void*)&f.gates, (void*)&u0, (void*)&v0,
                    (void*)&u1, (void*)&v1,      (void*)&f.p, (void*)&a};
    (void)hipLaunchKernel(regs_kernel<T, PM>(t.reg_rows()), dim3(a.ntx * a.nty),
                          dim3(64 * reg_waves(t.reg_rows())), args, 0, s);
    *cur = nxt;
  }
}

}  // namespace

template <typename T>
hipError_t init_projection() {
  const int bytes = (int)kLdsLimit;
  hipError_t e = hipFuncSetAttribute((const void*)k_project_tiled<T, false>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess)
    e = hipFuncSetAttribute((const void*)k_project_tiled<T, true>,
                            hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return e;
}

template <typename T>
void enqueue_projection(const StepParams& sp, const GridView& g, const FieldPtrs& f, int* cur,
                        const ProjTuning& t, hipStream_t s) {
  if ((t.kernel == PROJ_RESIDENT || t.kernel == PROJ_REGS) && t.valid(sp.pressure_on)) {
    ProjTuning run;
    const bool resident = t.kernel == PROJ_RESIDENT && f.exchange &&
                          t.resident_plan(sp.W, sp.H, sp.cus, &run);
    if (!sp.pressure_on) {
      resident ? launch_resident<T, PM_NONE>(sp, f, cur, run, s)
               : launch_regs<T, PM_NONE>(sp, f, cur, t, s);
    } else if (sp.pdt_recip == 0.0) {
      resident ? launch_resident<T, PM_DIVIDE>(sp, f, cur, run, s)
               : launch_regs<T, PM_DIVIDE>(sp, f, cur, t, s);
    } else if (sp.density == 1.0f && sp.cs == 1) {
      resident ? launch_resident<T, PM_UNIT>(sp, f, cur, run, s)
               : launch_regs<T, PM_UNIT>(sp, f, cur, t, s);
    } else {
      resident ? launch_resident<T, PM_RECIP>(sp, f, cur, run, s)
               : launch_regs<T, PM_RECIP>(sp, f, cur, t, s);
    }
    return;
  }
  if (t.kernel == PROJ_TILED && t.valid(sp.pressure_on)) {
    if (sp.pressure_on)
      launch_tiled<T, true>(sp, g, f, cur, t, s);
    else
      launch_tiled<T, false>(sp, g, f, cur, t, s);
    return;
  }
  T* u = (T*)f.u[*cur];
  T* v = (T*)f.v[*cur];
  const dim3 grid((sp.W / 2 + 63) / 64 + 1, (sp.H + 3) / 4), block(64, 4);
  for (int sweep = 0; sweep < sp.n; sweep++) {
    hipLaunchKernelGGL(k_project_colour<T>, grid, block, 0, s, sp, g.flags, u, v, f.p, 0);
    hipLaunchKernelGGL(k_project_colour<T>, grid, block, 0, s, sp, g.flags, u, v, f.p, 1);
  }
}

#define OSY_PROJECTION(T)                                                                  \
  template hipError_t init_projection<T>();                                                \
  template void enqueue_projection<T>(const StepParams&, const GridView&, const FieldPtrs&, \
                                      int*, const ProjTuning&, hipStream_t);
// one storage type per object (OSY_ONLY_STORAGE), so that they build at once
#if !defined(OSY_ONLY_STORAGE) || OSY_ONLY_STORAGE == 0
OSY_PROJECTION(float)
#endif
#if !defined(OSY_ONLY_STORAGE) || OSY_ONLY_STORAGE == 1
OSY_PROJECTION(__half)
#endif
#if !defined(OSY_ONLY_STORAGE) || OSY_ONLY_STORAGE == 2
OSY_PROJECTION(__hip_bfloat16)
#endif

}  // namespace osy
