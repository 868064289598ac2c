// kernels_step.hip - the per-step phases of Fluid::update (src/fluid.cu:770-795)
// as HIP kernels for gfx950, plus mask build, reductions and layout copies.
//
// One step is: the projection launches (the first of which applies the
// external forces to every cell it loads), the velocity advection (which
// reads the projected field through the edge extrapolation, so the
// extrapolated field is never stored), and the smoke advection (which
// applies the smoke part of the forces as it loads and the decay as it
// stores).  Both advections write into the other half of a ping-pong pair
// instead of the reference's buffer-then-copy-back (src/fluid.cu:614-617,
// 569-571): same values, half the traffic.  The advections stage a tile of
// the fields plus a 4-cell halo in LDS with coalesced loads; a back-trace
// that leaves the staged region reads HBM directly.
#include "advect_device.hpp"
#include "fluid_device.hpp"
#include "kernels.hpp"
#include "batch.hpp"
#include "projection.hpp"
#include "projection_device.hpp"
#include "step_device.hpp"

#pragma clang fp contract(off)

namespace osy {
namespace {

constexpr int kBX = 64, kBY = 4;

inline dim3 cell_grid(int W, int H) {
  return dim3((W + kBX - 1) / kBX, (H + kBY - 1) / kBY);
}

// ---- mask build: Fluid::init_device_memory (src/fluid.cu:111-142) -------

// is_solid of the reference.  The obstacle test there is
// sqrt(pow(dx,2) + pow(dy,2)) < radius in double.  For an integer d2 and a
// radius that is a float widened to double, RN(sqrt(d2)) < r holds exactly
// when r > 0 and d2 < r*r, both sides exact in double (d2 < 2^51 and r*r
// has at most 48 significant bits); the test restates it that way so the
// result does not depend on the device's square root.
__device__ bool solid_at(const MaskParams& m, int i, int j) {
  const double dx = (double)i - m.cx, dy = (double)j - m.cy;
  const double d2 = dx * dx + dy * dy;
  const bool obstacle = m.obstacle_enable && m.radius > 0.0 && d2 < m.radius * m.radius;
  const bool pipe = i < m.pipe_length &&
                    (j == m.H / 2 - m.pipe_height / 2 - 1 || j == m.H / 2 + m.pipe_height / 2 + 1);
  return i == 0 || j == 0 || j == m.H - 1 || (!m.enable_drain && i == m.W - 1) || obstacle ||
         pipe;
}

__global__ void k_build_flags(MaskParams m, uint8_t* flags) {
  const int i = blockIdx.x * kBX + threadIdx.x;
  const int j = blockIdx.y * kBY + threadIdx.y;
  if (i >= m.P || j >= m.H) return;
  if (i >= m.W) {  // row padding: never read as fluid
    flags[(long)j * m.P + i] = 0;
    return;
  }
  const bool s = solid_at(m, i, j);
  const bool l = i > 0 && !solid_at(m, i - 1, j);
  const bool r = i + 1 < m.W && !solid_at(m, i + 1, j);
  const bool b = j > 0 && !solid_at(m, i, j - 1);
  const bool t = j + 1 < m.H && !solid_at(m, i, j + 1);
  const int total_s = (int)l + (int)r + (int)b + (int)t;
  uint8_t f = (uint8_t)(total_s << CF_S_SHIFT);
  if (!s) {
    f |= CF_FLUID;
    if (i >= 1 && i <= m.W - 2 && j >= 1 && j <= m.H - 2) f |= CF_UPD;
    if (l) f |= CF_FU;
    if (b) f |= CF_FV;
  }
  flags[(long)j * m.P + i] = f;
}

// The projection's gate byte of every cell (gate_byte: its face gates,
// projected bit and quotient class), from its flags and those of its right
// and top neighbours; 0 outside the grid and in the row padding.
__global__ void k_build_gates(MaskParams m, const uint8_t* flags, uint8_t* gates) {
  const int i = blockIdx.x * kBX + threadIdx.x;
  const int j = blockIdx.y * kBY + threadIdx.y;
  if (i >= m.P || j >= m.H) return;
  const long k = (long)j * m.P + i;
  if (i >= m.W) {
    gates[k] = 0;
    return;
  }
  const uint32_t f = flags[k];
  const uint32_t fr = i + 1 < m.W ? flags[k + 1] : 0u;
  const uint32_t ft = j + 1 < m.H ? flags[k + m.P] : 0u;
  gates[k] = (uint8_t)gate_byte(f, fr, ft);
}

// ---- P1: forces over 64 x 16 tiles (forces_tile), four rows per thread --
constexpr int kForcesTY = 16;
template <typename T>
__global__ void __launch_bounds__(kBX * kBY)
    k_forces(StepParams sp, int do_uv, int do_smoke, T* u, T* v, T* smoke, float* p) {
  static_assert(kBX == kAdvTX && kForcesTY % kBY == 0, "forces tile shape");
  forces_tile<T, kForcesTY, kBY>(sp, do_uv, do_smoke, u, v, smoke, p, blockIdx.x, blockIdx.y);
}

// ---- P5: thrust::reduce min/max of pressure (src/fluid.cu:778-787) -------

__device__ inline float wave_min(float x) {
  for (int o = 32; o > 0; o >>= 1) x = fminf(x, __shfl_xor(x, o));
  return x;
}
__device__ inline float wave_max(float x) {
  for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
  return x;
}

// One launch: every workgroup takes pieces of kMinmaxCells cells of a row, four
// pieces' loads in flight per thread, and the last to finish reduces the
// partial results (min and max in one word) of all; `done` counts the
// workgroups and is 0 between launches.  Bound by the loads' latency on
// small grids and by HBM on large ones.  Rows read a word at a time by 512
// workgroups of 4 wavefronts, and a second launch for the partial results,
// took 8.7 us at 397 x 223, 14.1 us at 1920 x 1080 and 27.7 us at 3840 x 2160; this
// takes 4.5, 7.1 and 12.9 us.
constexpr int kMinmaxThreads = 512, kMinmaxCells = 4 * kMinmaxThreads;

__device__ inline void block_minmax(float& lo, float& hi) {
  __shared__ float slo[kMinmaxThreads / 64], shi[kMinmaxThreads / 64];
  lo = wave_min(lo);
  hi = wave_max(hi);
  __syncthreads();  // of the reduction before
  if ((threadIdx.x & 63) == 0) {
    slo[threadIdx.x >> 6] = lo;
    shi[threadIdx.x >> 6] = hi;
  }
  __syncthreads();
  for (int w = 0; w < kMinmaxThreads / 64; w++) {
    lo = fminf(lo, slo[w]);
    hi = fmaxf(hi, shi[w]);
  }
}

__global__ void __launch_bounds__(kMinmaxThreads)
    k_minmax(int W, int H, int P, const float* __restrict__ p, unsigned long long* part,
             unsigned* done, float* out) {
  float lo = INFINITY, hi = -INFINITY;
  const int per_row = (W + kMinmaxCells - 1) / kMinmaxCells;
  const int pieces = per_row * H, step = gridDim.x;
  for (int t = blockIdx.x; t < pieces; t += 4 * step) {
    float4 x[4];
    int left[4];  // cells of the four that lie in the row
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int piece = min(t + q * step, pieces - 1);
      const int j = piece / per_row;
      const int i = (piece - j * per_row) * kMinmaxCells + 4 * (int)threadIdx.x;
      left[q] = W - i;
      // rows start on 64-element boundaries and are padded to 64 (P)
      x[q] = *reinterpret_cast<const float4*>(p + (long)j * P + min(i, P - 4));
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const float c[4] = {x[q].x, x[q].y, x[q].z, x[q].w};
#pragma unroll
      for (int e = 0; e < 4; e++) {
        lo = fminf(lo, e < left[q] ? c[e] : INFINITY);
        hi = fmaxf(hi, e < left[q] ? c[e] : -INFINITY);
      }
    }
  }
  block_minmax(lo, hi);
  __shared__ bool last;
  if (threadIdx.x == 0) {
    const unsigned long long both =
        (unsigned long long)__float_as_uint(hi) << 32 | __float_as_uint(lo);
    __hip_atomic_store(&part[blockIdx.x], both, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the word has reached the other XCDs before the count; an ordering atomic
    // would also write back and drop the whole L2.  (The fences on both sides
    // keep the compiler from moving either atomic past the wait, which is what
    // orders them on gfx950: tests/test_reduction_order.py.)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
           gridDim.x - 1;
  }
  __syncthreads();
  if (!last) return;
  lo = INFINITY;
  hi = -INFINITY;
  for (unsigned b = threadIdx.x; b < gridDim.x; b += kMinmaxThreads) {
    const unsigned long long both =
        __hip_atomic_load(&part[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    lo = fminf(lo, __uint_as_float((uint32_t)both));
    hi = fmaxf(hi, __uint_as_float((uint32_t)(both >> 32)));
  }
  block_minmax(lo, hi);
  if (threadIdx.x == 0) {
    out[0] = lo;
    out[1] = hi;
    __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

void launch_minmax(const StepParams& sp, const FieldPtrs& f, hipStream_t s) {
  const long pieces = (long)((sp.W + kMinmaxCells - 1) / kMinmaxCells) * sp.H;
  const unsigned blocks = (unsigned)min((pieces + 3) / 4, (long)kReduceBlocks);
  // after the range: the count of finished workgroups
  hipLaunchKernelGGL(k_minmax, dim3(blocks), dim3(kMinmaxThreads), 0, s, sp.W, sp.H, sp.P, f.p,
                     (unsigned long long*)f.scratch, (unsigned*)(f.prange + 2), f.prange);
}

// ---- P6-P8: the advections over 64 x 32 tiles, 512 threads ---------------
constexpr int kAdvTY = 32, kAdvNY = 8;

// 1-D grids of ntx x nty tiles in the XCD-aware order (xcd_tile).
template <typename T, bool CS1>
__global__ void __launch_bounds__(64 * kAdvNY)
    k_advect_velocity(StepParams sp, GridView g, const T* __restrict__ u,
                      const T* __restrict__ v, T* __restrict__ u_out, T* __restrict__ v_out,
                      int ntx) {
  __shared__ AdvShared<kAdvTY> sh;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  advect_velocity_tile<T, CS1, kAdvTY, kAdvNY>(sp, g, u, v, u_out, v_out, tile % ntx, tile / ntx,
                                               sh);
}

template <typename T, bool CS1>
__global__ void __launch_bounds__(64 * kAdvNY)
    k_advect_smoke(StepParams sp, GridView g, const T* __restrict__ u, const T* __restrict__ v,
                   const T* __restrict__ smoke, T* __restrict__ smoke_out, int ntx) {
  __shared__ AdvShared<kAdvTY> sh;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  advect_smoke_tile<T, CS1, kAdvTY, kAdvNY>(sp, g, u, v, smoke, smoke_out, tile % ntx,
                                            tile / ntx, sh);
}

// ---- P2b: apply_diffusion (src/fluid.cu:167-190) as Jacobi rounds -------
// Every interior cell (1 <= i <= W-2, 1 <= j <= H-2, solid or not) becomes
// (u + a*(((u(i-1,j) + u(i+1,j)) + u(i,j-1)) + u(i,j+1))) / (1 + 4a) of the
// previous round's u; borders keep theirs; v is not diffused.
//
// The tiles and registers are the register projection's (projection_device.hpp):
// NW wavefronts of R rows, lane l holds cells 2l and 2l+1 of each, and a
// launch runs up to 2k rounds on a tile with a halo of 2k cells, since a
// round moves a stale value one cell.  Left and right come from the lane's
// other cell and by a lane shift, below and above from the lane's other
// rows, and at the wavefront's first and last row through LDS, with one
// barrier per round; the rows inside are computed first, which hides that.
// What bounds it is the issue of vector instructions, so the quotient goes
// through the double reciprocal of the divisor where that is exact
// (recip_quotient), and only wavefronts that hold border cells select.
// 50 rounds of 1920 x 1080 take 78 us (5 launches of 15.6 us); with the region
// in LDS they took 175 us (9 launches of 19.4 us: six reads and writes of LDS
// and a division per cell and round).
template <int NW>
struct DiffShared {
  float2 first[2][NW][64], last[2][NW][64];  // rows 0 and R-1 of each wavefront
};

template <typename T, bool RECIP>
__device__ inline float diffused(float x, float sum, float a, float den, double recip) {
  const float y = x + a * sum;
  return rnd<T>(RECIP ? recip_quotient(y, recip) : y / den);
}

// One round of a wavefront's rows.  EDGE: cells outside `cols0`, `cols1`
// (even, odd cells) and rows outside [j_lo, j_hi) keep their values.
template <typename T, int R, bool RECIP, bool EDGE>
__device__ __attribute__((always_inline)) inline void diffuse_rows(
    float (&x0)[R], float (&x1)[R], const float2& below, const float2& above,
    const StepParams& sp, unsigned long long cols0, unsigned long long cols1, int j_lo, int j_hi) {
  float n0[R], n1[R];
#pragma unroll
  for (int q = 0; q < R; q++) {
    const int rho = q + 1 < R - 1 ? q + 1 : q + 1 == R - 1 ? 0 : R - 1;  // inner rows first
    const float b0 = rho > 0 ? x0[rho > 0 ? rho - 1 : 0] : below.x;
    const float b1 = rho > 0 ? x1[rho > 0 ? rho - 1 : 0] : below.y;
    const float t0 = rho + 1 < R ? x0[rho + 1 < R ? rho + 1 : rho] : above.x;
    const float t1 = rho + 1 < R ? x1[rho + 1 < R ? rho + 1 : rho] : above.y;
    const float s0 = ((lane_from_left(x1[rho]) + x1[rho]) + b0) + t0;
    const float s1 = ((x0[rho] + lane_from_right(x0[rho])) + b1) + t1;
    n0[rho] = diffused<T, RECIP>(x0[rho], s0, sp.visc_a, sp.visc_den, sp.visc_recip);
    n1[rho] = diffused<T, RECIP>(x1[rho], s1, sp.visc_a, sp.visc_den, sp.visc_recip);
    if constexpr (EDGE) {
      const bool row = rho >= j_lo && rho < j_hi;
      n0[rho] = in_lanes(row ? cols0 : 0ULL) ? n0[rho] : x0[rho];
      n1[rho] = in_lanes(row ? cols1 : 0ULL) ? n1[rho] : x1[rho];
    }
  }
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    x0[rho] = n0[rho];
    x1[rho] = n1[rho];
  }
}

template <typename T, int R, int NW, bool RECIP, bool EDGE>
__device__ __attribute__((always_inline)) inline void diffuse_rounds(
    float (&x0)[R], float (&x1)[R], DiffShared<NW>& sh, const StepParams& sp, int w, int rounds,
    int active, unsigned long long cols0, unsigned long long cols1, int j_lo, int j_hi) {
  const int lane = reg_lane();
  for (int it = 0; it < rounds; it++) {
    const int slot = it & 1;
    sh.first[slot][w][lane] = make_float2(x0[0], x1[0]);
    sh.last[slot][w][lane] = make_float2(x0[R - 1], x1[R - 1]);
    __syncthreads();
    // (a slot is written again two rounds on, after the barrier between)
    if (it < active) {
      const float2 below = sh.last[slot][max(w - 1, 0)][lane];
      const float2 above = sh.first[slot][min(w + 1, NW - 1)][lane];
      diffuse_rows<T, R, RECIP, EDGE>(x0, x1, below, above, sp, cols0, cols1, j_lo, j_hi);
    }
  }
}

// u goes from u_in to u_out; with copy_v the launch also moves v to v_out so
// that u and v stay in the same buffer of their pairs.
template <typename T, int R, int NW, bool RECIP>
__global__ void __launch_bounds__(64 * NW, NW / 2)
    k_diffuse(StepParams sp, const T* __restrict__ u_in, T* __restrict__ u_out,
              const T* __restrict__ v_in, T* __restrict__ v_out, int copy_v, RegArgs a) {
  __shared__ DiffShared<NW> sh;
  const RegPlace pl = reg_place<R, NW>(a, xcd_tile(blockIdx.x, gridDim.x), sp.W, sp.H);
  const int lane = reg_lane(), W = sp.W, H = sp.H, P = sp.P;
  const int gi = pl.gx0 + 2 * lane;
  // every load first, from the pair clamped into the row and the row clamped
  // into the grid
  const unsigned gic = (unsigned)min(gi, P - 2);
  float x0[R], x1[R];
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const long row = (long)min(pl.gy0 + pl.rbase + rho, H - 1) * P;
    load_pair(u_in + row, gic, true, true, x0[rho], x1[rho]);
  }
  const bool own0 = 2 * lane >= pl.c0 && 2 * lane < pl.c1;
  const bool own1 = own0 && gi + 1 < W;
  if (copy_v) {
#pragma unroll
    for (int rho = 0; rho < R; rho++) {
      const int r = pl.rbase + rho;
      if (r < pl.r0 || r >= pl.r1) continue;
      const long row = (long)(pl.gy0 + r) * P;
      float v0, v1;
      load_pair(v_in + row, gic, true, true, v0, v1);
      store_pair(v_out + row, (unsigned)gi, own0, own1, v0, v1);
    }
  }
  // cells that are updated: lanes, and rows [j_lo, j_hi) of the wavefront
  const unsigned long long cols0 = __ballot(gi >= 1 && gi <= W - 2);
  const unsigned long long cols1 = __ballot(gi + 1 <= W - 2);
  const int y = pl.gy0 + pl.rbase;
  const int j_lo = max(1 - y, 0), j_hi = min(H - 1 - y, R);
  // rounds in which some row can still reach the tile's own
  const int idle = max(max(pl.r0 - pl.rbase - R, pl.rbase - pl.r1) + 1, 0);
  const int active = a.sweeps - idle;
  if ((cols0 & cols1) == ~0ULL && j_lo == 0 && j_hi == R)
    diffuse_rounds<T, R, NW, RECIP, false>(x0, x1, sh, sp, pl.w, a.sweeps, active, cols0, cols1,
                                           j_lo, j_hi);
  else
    diffuse_rounds<T, R, NW, RECIP, true>(x0, x1, sh, sp, pl.w, a.sweeps, active, cols0, cols1,
                                          j_lo, j_hi);
#pragma unroll
  for (int rho = 0; rho < R; rho++) {
    const int r = pl.rbase + rho;
    if (r < pl.r0 || r >= pl.r1) continue;
    store_pair(u_out + (long)(pl.gy0 + r) * P, (unsigned)gi, own0, own1, x0[rho], x1[rho]);
  }
}

// `sp.n` rounds in launches of 2k; advances *uv by the launch count (v moves
// with u on the last launch when that count is odd).  Regions of 32 rows
// while their tiles fit the CUs once, else of 96 (kernel's figures above).
template <typename T>
void enqueue_diffusion(const StepParams& sp, const FieldPtrs& f, int* uv, hipStream_t s) {
  if (sp.n <= 0) return;
  ProjTuning t;
  bool low = false;
  auto fits = [&](int rows, int k_most, int k_least) {
    for (t.k = k_most; t.k >= k_least; t.k--) {
      t.tw = 128 - 4 * t.k;
      t.th = 8 * rows - 4 * t.k;
      if (t.tiles(sp.W, sp.H) <= sp.cus) return true;
    }
    return false;
  };
  low = fits(4, 6, 4);
  if (!low && !fits(12, 12, 5)) {
    t.k = 5;
    t.tw = 128 - 4 * t.k;
    t.th = 96 - 4 * t.k;
  }
  RegArgs a{};
  a.tw = t.tw;
  a.th = t.th;
  a.k = t.k;
  a.ntx = t.tiles_x(sp.W);
  a.nty = t.tiles_y(sp.H);
  const int launches = (sp.n + 2 * t.k - 1) / (2 * t.k);
  int cur = *uv;
  for (int q = 0; q < launches; q++) {
    a.sweeps = min(2 * t.k, sp.n - 2 * t.k * q);
    const int copy_v = (q + 1 == launches) && (launches & 1);
    const dim3 grid(a.ntx * a.nty), block(low ? 512 : 1024);
    auto* kernel = low ? (sp.visc_recip != 0.0 ? k_diffuse<T, 4, 8, true> : k_diffuse<T, 4, 8, false>)
                       : (sp.visc_recip != 0.0 ? k_diffuse<T, 6, 16, true>
                                               : k_diffuse<T, 6, 16, false>);
    hipLaunchKernelGGL(kernel, grid, block, 0, s, sp, (const T*)f.u[cur], (T*)f.u[1 - cur],
                       (const T*)f.v[cur], (T*)f.v[1 - cur], copy_v, a);
    cur = 1 - cur;
  }
  *uv = cur;
}

// ---- divergence norms (Fluid::get_divergence, src/fluid.cu:192-201) -------
__device__ inline double wave_sum_d(double x) {
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
  return x;
}
__device__ inline double wave_max_d(double x) {
  for (int o = 32; o > 0; o >>= 1) x = fmax(x, __shfl_xor(x, o));
  return x;
}

template <typename T>
__global__ void __launch_bounds__(256) k_div_partial(StepParams sp, GridView g, const T* u,
                                                     const T* v, double* part) {
  double ss = 0.0, mx = 0.0;
  for (int j = 1 + blockIdx.x; j <= sp.H - 2; j += gridDim.x)
    for (int i = 1 + threadIdx.x; i <= sp.W - 2; i += blockDim.x) {
      const long k = g.at(i, j);
      if (!(g.flags[k] & CF_FLUID)) continue;
      const double d = (((double)ldf(u, k + 1) - (double)ldf(u, k)) + (double)ldf(v, k + sp.P)) -
                       (double)ldf(v, k);
      ss += d * d;
      mx = fmax(mx, fabs(d));
    }
  __shared__ double sss[4], smx[4];
  ss = wave_sum_d(ss);
  mx = wave_max_d(mx);
  if ((threadIdx.x & 63) == 0) {
    sss[threadIdx.x >> 6] = ss;
    smx[threadIdx.x >> 6] = mx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; w++) {
      ss += sss[w];
      mx = fmax(mx, smx[w]);
    }
    part[2 * blockIdx.x] = ss;
    part[2 * blockIdx.x + 1] = mx;
  }
}

__global__ void __launch_bounds__(64) k_div_final(const double* part, int nparts, double* out) {
  double ss = 0.0, mx = 0.0;
  for (int b = threadIdx.x; b < nparts; b += 64) {
    ss += part[2 * b];
    mx = fmax(mx, part[2 * b + 1]);
  }
  ss = wave_sum_d(ss);
  mx = wave_max_d(mx);
  if (threadIdx.x == 0) {
    out[0] = sqrt(ss);
    out[1] = mx;
  }
}

// ---- layout copies --------------------------------------------------------
// mode 0: device field (T) -> reference float; 1: reference float -> device
// field; 2: flags -> is_solid; 3: flags -> total_s; 4: float device field
// (pressure) -> reference; 5: reference -> pressure.
template <typename T>
__global__ void k_layout(int mode, int W, int H, int P, T* dev, float* pdev, const uint8_t* flags,
                         void* ref) {
  const int i = blockIdx.x * kBX + threadIdx.x;
  const int j = blockIdx.y * kBY + threadIdx.y;
  if (i >= W || j >= H) return;
  const long k = (long)j * P + i;
  const long r = (long)(H - 1 - j) * W + i;  // Fluid::indx (src/fluid.cu:163-165)
  switch (mode) {
    case 0: ((float*)ref)[r] = ldf(dev, k); break;
    case 1: stf(dev, k, ((const float*)ref)[r]); break;
    case 2: ((int32_t*)ref)[r] = (flags[k] & CF_FLUID) ? 0 : 1; break;
    case 3: ((int32_t*)ref)[r] = cf_total_s(flags[k]); break;
    case 4: ((float*)ref)[r] = pdev[k]; break;
    case 5: pdev[k] = ((const float*)ref)[r]; break;
  }
}

template <typename T, bool CS1>
void advect_t(const StepParams& sp, const GridView& g, const FieldPtrs& f, int cur, int* uv,
              int* sm, hipStream_t s) {
  const int ntx = (sp.W + kAdvTX - 1) / kAdvTX, nty = (sp.H + kAdvTY - 1) / kAdvTY;
  const dim3 grid(ntx * nty), block(64 * kAdvNY);
  const int nxt = 1 - cur;
  T* u2 = (T*)f.u[nxt];
  T* v2 = (T*)f.v[nxt];
  hipLaunchKernelGGL((k_advect_velocity<T, CS1>), grid, block, 0, s, sp, g, (const T*)f.u[cur],
                     (const T*)f.v[cur], u2, v2, ntx);
  *uv = nxt;
  if (sp.smoke_on) {
    hipLaunchKernelGGL((k_advect_smoke<T, CS1>), grid, block, 0, s, sp, g, (const T*)u2,
                       (const T*)v2, (const T*)f.smoke[*sm], (T*)f.smoke[1 - *sm], ntx);
    *sm = 1 - *sm;
  }
}

template <typename T>
void step_t(const StepParams& sp_in, const FieldPtrs& f, int* uv, int* sm,
            const ProjTuning& tuning, hipStream_t s) {
  const GridView g{sp_in.W, sp_in.H, sp_in.P, sp_in.cs, f.flags};
  StepParams sp = sp_in;
  // the first tiled projection launch applies the velocity forces (and
  // starts the pressure sums at 0) as it loads; the smoke advection applies
  // the smoke forces as it loads
  // (with diffusion the forces come first as a pass of their own, then the
  // diffusion launches, src/fluid.cu:771-776)
  const bool diffuse = sp.visc_on && sp.n > 0;
  const bool fuse_uv =
      !diffuse && sp.n > 0 && tuning.kernel != PROJ_COLOUR && tuning.valid(sp.pressure_on);
  const bool fuse_smoke = sp.smoke_on;
  sp.forces_in_projection = fuse_uv ? 1 : 0;
  if (!fuse_uv || !fuse_smoke)
    hipLaunchKernelGGL(k_forces<T>,
                       dim3((sp.W + kBX - 1) / kBX, (sp.H + kForcesTY - 1) / kForcesTY),
                       dim3(kBX * kBY), 0, s, sp,
                       fuse_uv ? 0 : 1, fuse_smoke ? 0 : 1, (T*)f.u[*uv], (T*)f.v[*uv],
                       (T*)f.smoke[*sm], f.p);
  int cur = *uv;
  if (diffuse) enqueue_diffusion<T>(sp, f, &cur, s);
  enqueue_projection<T>(sp, g, f, &cur, tuning, s);
  if (sp.pressure_on) launch_minmax(sp, f, s);
  if (sp.cs == 1)
    advect_t<T, true>(sp, g, f, cur, uv, sm, s);
  else
    advect_t<T, false>(sp, g, f, cur, uv, sm, s);
}

template <typename T>
void divergence_t(const StepParams& sp, const FieldPtrs& f, int uv, hipStream_t s) {
  const GridView g{sp.W, sp.H, sp.P, sp.cs, f.flags};
  hipLaunchKernelGGL(k_div_partial<T>, dim3(kReduceBlocks), dim3(256), 0, s, sp, g,
                     (const T*)f.u[uv], (const T*)f.v[uv], f.dscratch);
  hipLaunchKernelGGL(k_div_final, dim3(1), dim3(64), 0, s, f.dscratch, kReduceBlocks,
                     f.dscratch + 2 * kReduceBlocks);
}

template <typename T>
void layout_t(int field, bool to_ref, const StepParams& sp, const FieldPtrs& f, int uv, int sm,
              void* ref, hipStream_t s) {
  T* dev = nullptr;
  int mode = to_ref ? 0 : 1;
  switch (field) {
    case OSY_FIELD_VEL_X: dev = (T*)f.u[uv]; break;
    case OSY_FIELD_VEL_Y: dev = (T*)f.v[uv]; break;
    case OSY_FIELD_SMOKE: dev = (T*)f.smoke[sm]; break;
    case OSY_FIELD_PRESSURE: mode = to_ref ? 4 : 5; break;
    case OSY_FIELD_IS_SOLID: mode = 2; break;
    case OSY_FIELD_TOTAL_S: mode = 3; break;
  }
  hipLaunchKernelGGL(k_layout<T>, cell_grid(sp.W, sp.H), dim3(kBX, kBY), 0, s, mode, sp.W, sp.H,
                     sp.P, dev, f.p, f.flags, ref);
}

}  // namespace

hipError_t init_projection_kernels() {
  hipError_t e = init_projection<float>();
  if (e == hipSuccess) e = init_projection<__half>();
  if (e == hipSuccess) e = init_projection<__hip_bfloat16>();
  return e;
}

void launch_build_flags(const MaskParams& m, uint8_t* flags, uint8_t* gates, hipStream_t s) {
  hipLaunchKernelGGL(k_build_flags, cell_grid(m.P, m.H), dim3(kBX, kBY), 0, s, m, flags);
  hipLaunchKernelGGL(k_build_gates, cell_grid(m.P, m.H), dim3(kBX, kBY), 0, s, m, flags, gates);
}

void enqueue_step(int storage, const StepParams& sp, const FieldPtrs& f, int* uv, int* sm,
                  const ProjTuning& tuning, hipStream_t s) {
  switch (storage) {
    case OSY_STORAGE_F16: step_t<__half>(sp, f, uv, sm, tuning, s); break;
    case OSY_STORAGE_BF16: step_t<__hip_bfloat16>(sp, f, uv, sm, tuning, s); break;
    default: step_t<float>(sp, f, uv, sm, tuning, s); break;
  }
}

void enqueue_projection_only(int storage, const StepParams& sp_in, const FieldPtrs& f, int* uv,
                             const ProjTuning& tuning, hipStream_t s) {
  const GridView g{sp_in.W, sp_in.H, sp_in.P, sp_in.cs, f.flags};
  StepParams sp = sp_in;
  sp.forces_in_projection = 0;
  switch (storage) {
    case OSY_STORAGE_F16: enqueue_projection<__half>(sp, g, f, uv, tuning, s); break;
    case OSY_STORAGE_BF16:
      enqueue_projection<__hip_bfloat16>(sp, g, f, uv, tuning, s);
      break;
    default: enqueue_projection<float>(sp, g, f, uv, tuning, s); break;
  }
}

namespace {
__global__ void __launch_bounds__(256) k_copy(uint4* __restrict__ dst,
                                              const uint4* __restrict__ src, size_t n) {
  for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (size_t)gridDim.x * 256)
    dst[k] = src[k];
}
__global__ void __launch_bounds__(256) k_clean_exchange(uint4* __restrict__ mem, size_t n) {
  for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (size_t)gridDim.x * 256) {
    const uint32_t w = k < 16 ? 0u : ~0u;
    mem[k] = make_uint4(w, w, w, w);
  }
}
}  // namespace

void enqueue_clean_exchange(void* mem, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  size_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_clean_exchange, dim3((unsigned)blocks), dim3(256), 0, s, (uint4*)mem, n);
}

void enqueue_copy(void* dst, const void* src, size_t bytes, hipStream_t s) {
  const size_t n = bytes / 16;
  size_t blocks = (n + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(k_copy, dim3((unsigned)blocks), dim3(256), 0, s, (uint4*)dst,
                     (const uint4*)src, n);
}

void enqueue_pressure_range(const StepParams& sp, const FieldPtrs& f, hipStream_t s) {
  launch_minmax(sp, f, s);
}

void enqueue_divergence(int storage, const StepParams& sp, const FieldPtrs& f, int uv,
                        hipStream_t s) {
  switch (storage) {
    case OSY_STORAGE_F16: divergence_t<__half>(sp, f, uv, s); break;
    case OSY_STORAGE_BF16: divergence_t<__hip_bfloat16>(sp, f, uv, s); break;
    default: divergence_t<float>(sp, f, uv, s); break;
  }
}

void enqueue_export(int field, int storage, const StepParams& sp, const FieldPtrs& f, int uv,
                    int sm, void* ref, hipStream_t s) {
  switch (storage) {
    case OSY_STORAGE_F16: layout_t<__half>(field, true, sp, f, uv, sm, ref, s); break;
    case OSY_STORAGE_BF16: layout_t<__hip_bfloat16>(field, true, sp, f, uv, sm, ref, s); break;
    default: layout_t<float>(field, true, sp, f, uv, sm, ref, s); break;
  }
}

void enqueue_import(int field, int storage, const StepParams& sp, const FieldPtrs& f, int uv,
                    int sm, const void* ref, hipStream_t s) {
  switch (storage) {
    case OSY_STORAGE_F16: layout_t<__half>(field, false, sp, f, uv, sm, (void*)ref, s); break;
    case OSY_STORAGE_BF16:
      layout_t<__hip_bfloat16>(field, false, sp, f, uv, sm, (void*)ref, s);
      break;
    default: layout_t<float>(field, false, sp, f, uv, sm, (void*)ref, s); break;
  }
}

}  // namespace osy
