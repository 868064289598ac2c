// kernels.hpp - launch interface of the solver's HIP kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

#include "../../include/opensayal.h"

namespace osy {

// Geometry of the solid mask (src/fluid.cu:111-126).
struct MaskParams {
  int W, H, P;
  int enable_drain;
  int obstacle_enable;
  double cx, cy, radius;  // radius as the float config value, widened
  int pipe_length, pipe_height;
};

// Everything a step needs besides the field pointers.
struct StepParams {
  int W, H, P, cs;
  int n;                 // projection sweeps
  float o, density, d_t;
  // apply_external_forces_at (src/fluid.cu:308-349)
  int smoke_length;
  int band_lo, band_hi;  // u = speed for band_lo <= j <= band_hi
  int smoke_count, smoke_height, smoke_mod, smoke_top;  // stripe rule
  int sband_lo, sband_hi;                                // single-band rule
  float speed, wind_smoke;
  int drag_on;
  float damping;          // expf(-drag_coeff * d_t), computed once on the host
  float gdt;              // g * d_t
  int src_active, src_x, src_y;
  float src_smoke, src_velocity;
  int pressure_on;
  int smoke_on;           // enable_smoke && wind_tunnel.smoke != 0
  int decay_on;
  float decay_rd;         // decay_rate * d_t
  // apply_diffusion_at (src/fluid.cu:176-183): a = viscosity * d_t / cs^2
  // and the divisor 1 + 4a, both in float as the reference computes them
  int visc_on;
  float visc_a, visc_den;
  double visc_recip;  // 1 / visc_den for 0 < |visc_den| < 2, else 0 (recip_quotient)
  // set by the step: the first projection launch applies the velocity
  // forces to what it loads and starts the pressure sums at 0
  int forces_in_projection;
  // 1.0 / (double)d_t when 0 < |d_t| < 2, else 0: the pressure sums'
  // division by d_t as a double multiply (recip_quotient)
  double pdt_recip;
  // bound of one neighbour wait of the resident projection (wall-clock ticks)
  long long spin_ticks;
  int cus;  // CUs of the device
};

// Device buffers of one simulation; T is the storage type of u, v, smoke.
struct FieldPtrs {
  void* u[2];
  void* v[2];
  void* smoke[2];
  float* p;
  uint8_t* flags;
  uint8_t* gates;   // projection gate byte per cell (static: built with the flags)
  float* scratch;   // reductions: partial results
  float* prange;    // [min, max] of pressure
  double* dscratch; // divergence reduction partials
  void* exchange;   // resident projection: halo exchange slots (null until needed)
  unsigned* rstate; // resident projection: finished workgroups, slot of ring 0
  int* error;       // set by a resident projection whose neighbour wait timed out
};

// Projection kernels selectable per handle.
enum ProjectionKernel : int {
  PROJ_COLOUR = 0,  // one launch per colour phase, 2n launches, in place
  PROJ_TILED = 1,   // LDS tiles, several sweeps per launch, ping-pong
  PROJ_REGS = 2,    // register-resident tiles, several sweeps per launch
  PROJ_RESIDENT = 3,  // register-resident tiles kept for all n sweeps, one launch
};

// Register-resident kernels: a region of 128 x 8*rows cells held in VGPRs,
// by 8 wavefronts of `rows` rows each up to 10 rows (two workgroups per CU),
// by 16 of rows / 2 above (one): four wavefronts per SIMD either way, and
// more at 4 rows.
constexpr int kRegWaves = 8;
inline bool reg_rows_supported(int rows) {
  return rows == 4 || rows == 8 || rows == 10 || rows == 12 || rows == 16;
}
inline int reg_waves(int rows) { return rows > 10 ? 2 * kRegWaves : kRegWaves; }

// Workgroup of the tiled kernel: 8 wavefronts of 64 lanes.
constexpr int kTileWaves = 8;
constexpr int kTileThreads = 64 * kTileWaves;
constexpr size_t kLdsLimit = 160 * 1024;

// Shape of the tiled projection.  A workgroup owns a tile of tw x th cells;
// it loads the tile plus a 2k-cell halo on every side (the region) into LDS,
// runs up to k sweeps there and writes the tile back.  A lane handles one
// pair of horizontally adjacent cells; a region row of pw pairs takes
// ceil(pw / 64) wavefronts.
struct ProjTuning {
  int kernel = PROJ_TILED;
  int tw = 240;  // tile width (even)
  int th = 32;   // tile height
  int k = 4;     // sweeps per launch
  int region_w() const { return tw + 4 * k; }
  int region_h() const { return th + 4 * k; }
  int pw() const { return region_w() / 2; }
  int waves_per_row() const {
    const int n = (pw() + 63) / 64;
    return n <= 1 ? 1 : n <= 2 ? 2 : n <= 4 ? 4 : 8;
  }
  // LDS: u and v (float), gate and flag bytes, and pressure sums (float)
  size_t lds_bytes(bool pressure) const {
    const size_t cells = (size_t)region_h() * 2 * (pw() + 1);
    const size_t flag_bytes = (size_t)(region_h() + 1) * (region_w() + 1);
    return cells * 4 * (pressure ? 3 : 2) + cells + flag_bytes;
  }
  // PROJ_REGS, PROJ_RESIDENT: region rows / 8
  int reg_rows() const { return (th + 4 * k) / kRegWaves; }
  bool valid(bool pressure) const {
    if (kernel == PROJ_COLOUR) return true;
    if (kernel == PROJ_REGS || kernel == PROJ_RESIDENT) {
      // with pressure sums (2 more VGPRs per row) only up to 64 rows are built; a
      // resident shape of 64 runs as one of 96 (resident_plan)
      const bool regs = k >= 1 && k <= 28 && tw == 128 - 4 * k && th >= 1 &&
                        (th + 4 * k) % kRegWaves == 0 && reg_rows_supported(reg_rows()) &&
                        !(pressure && reg_rows() > 8);
      // resident: a halo of 2k reaches only the adjacent tiles
      return regs && (kernel == PROJ_REGS || (tw >= 2 * k && th >= 2 * k));
    }
    return kernel == PROJ_TILED && k >= 1 && k <= 64 && tw >= 2 && th >= 1 && tw % 2 == 0 &&
           pw() <= 64 * kTileWaves && lds_bytes(pressure) <= kLdsLimit;
  }
  // register kernels: tiles over a W x H grid (the first and last of a row
  // or column own 2k cells more, RegPlace)
  int tiles_x(int W) const { return W <= 4 * k + tw ? 1 : (W - 4 * k + tw - 1) / tw; }
  int tiles_y(int H) const { return H <= 4 * k + th ? 1 : (H - 4 * k + th - 1) / th; }
  int tiles(int W, int H) const { return tiles_x(W) * tiles_y(H); }
  // What a resident projection of this shape runs on a device of `cus` CUs.
  // Every tile's workgroup must be on the GPU at once, and the fewer, larger
  // workgroups a CU holds, the less it computes and exchanges in its halos:
  // regions of 64 rows and more run as one of 96 (16 wavefronts of 6 rows, a
  // CU's registers; 50 sweeps of 1920 x 1080 at k = 5 take 120 us, in
  // regions of 64 rows, two per CU, 233 us).  False when those do not fit
  // either: then each stage is a launch of this shape's register kernel,
  // the same tiles and results.
  bool resident_plan(int W, int H, int cus, ProjTuning* run) const {
    *run = *this;
    if (reg_rows() > 4) run->th = kRegWaves * 12 - 4 * k;
    return run->th >= 2 * k && run->tiles(W, H) <= (reg_rows() == 4 ? 3 : 1) * cus;
  }
  // resident kernel: 8-byte words of one of its three exchange slots (every
  // tile's region, two words per cell pair in binary32, one in 16 bits)
  size_t exchange_words(int W, int H, size_t elem) const {
    return (size_t)tiles(W, H) * region_h() * 64 * (elem / 2);
  }
};

// Number of float slots `scratch` must hold, and doubles for `dscratch`.
constexpr int kReduceBlocks = 512;

// Tiles that a resident shape may be asked to have: as many as workgroups of
// its register kernel fit the device, from the launch bounds (which the
// compiler meets, by spilling where it has to): 8 wavefronts within 80 VGPRs at
// 4 rows (6 per SIMD: 3 workgroups per CU) and 128 at 8 and 10 rows (4: 2
// workgroups); 16 wavefronts above (1).  LDS (12 KiB per 8 wavefronts) and the wavefront
// slots allow more.  (The runtime's occupancy query was not used: it has
// returned 0 for a kernel that fits, depending on what ran before.)
inline int resident_slots(int rows, int cus) { return (rows == 4 ? 3 : rows <= 10 ? 2 : 1) * cus; }

// Lets the projection kernels use all of the LDS on the current device.
hipError_t init_projection_kernels();

// Cell flags, then the projection gate bytes derived from them.
void launch_build_flags(const MaskParams& m, uint8_t* flags, uint8_t* gates, hipStream_t s);

// One full step (src/fluid.cu:770-795).  `uv`/`sm` give the buffer index
// currently holding u,v / smoke and are advanced to the index holding the
// step's result.
void enqueue_step(int storage, const StepParams& sp, const FieldPtrs& f,
                  int* uv, int* sm, const ProjTuning& t, hipStream_t s);

// The projection alone (`sp.n` sweeps); advances *uv like enqueue_step.
void enqueue_projection_only(int storage, const StepParams& sp, const FieldPtrs& f, int* uv,
                             const ProjTuning& t, hipStream_t s);

// Divergence L2 / max-abs in FP64 over interior fluid cells; result in
// dscratch[0], dscratch[1] after the stream reaches this point.
void enqueue_divergence(int storage, const StepParams& sp, const FieldPtrs& f,
                        int uv, hipStream_t s);

// Layout conversion between the device layout and the reference's indx
// order, for a field of storage type `storage` (or float/int32 for the
// other fields).  `ref` is a device buffer of W*H 4-byte elements.
void enqueue_export(int field, int storage, const StepParams& sp,
                    const FieldPtrs& f, int uv, int sm, void* ref, hipStream_t s);
void enqueue_import(int field, int storage, const StepParams& sp,
                    const FieldPtrs& f, int uv, int sm, const void* ref, hipStream_t s);

// Frame export (update_fluid_pixels_kernel, src/graphics_handler.cu:258-285):
// W*H RGBA8888 pixels in the reference's indx order into the device buffer
// `out`, using the pressure range in f.prange.  pressure_on / smoke_on are the
// config's enable_pressure / enable_smoke.
void enqueue_render(int storage, const StepParams& sp, const FieldPtrs& f, int sm,
                    int pressure_on, int smoke_on, uint32_t* out, hipStream_t s);

// Path lines (update_traces_kernel, src/graphics_handler.cu:384-396) for the
// seed grid of spacing `distance`: (W/distance)*(H/distance)*length int32
// entries into each of the device buffers tx, ty.
void enqueue_traces(int storage, const StepParams& sp, const FieldPtrs& f, int uv, int distance,
                    int length, float d_t, int32_t* tx, int32_t* ty, hipStream_t s);

// Empties a resident projection's halo exchange buffer (`bytes` a multiple of
// 16): 256 bytes of state words, 0, and slots of words that hold nothing.  A
// kernel rather than a fill of the runtime's, so that it can be captured.
void enqueue_clean_exchange(void* mem, size_t bytes, hipStream_t s);

// Plain device-to-device copy of `bytes` (a multiple of 16) with 16-byte
// loads and stores, for calibrating hardware byte counters.
void enqueue_copy(void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace osy
