// Internal: the per-solve handle and helpers shared by the single-solve and
// batched entry points.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <vector>

#include "../../include/mcv_hip.h"
#include "mcv_device.hpp"
#include "mcv_fp32c.hpp"

namespace mcv {

// Records the message returned by mcv_hip_last_error() and returns code.
int fail(int code, const char *fmt, ...);
// A solve or a batch comes (1) or goes (-1): the read-backs' pinned memory is
// given back with the last of them (mcv_hip.hip).
void staging_user(int change);
// mcv_history_write that also checks the file's per-record sizes (mcv_netcdf.cpp)
int history_write_checked(const char *path, int32_t time_slot, const mcv_history_fields *rec,
                          long long npoint, long long ncell);

#define HIP_TRY(expr)                                                                   \
  do {                                                                                  \
    hipError_t e_ = (expr);                                                             \
    if (e_ != hipSuccess)                                                               \
      return ::mcv::fail(MCV_EDEVICE, "%s failed: %s (%s:%d)", #expr,                   \
                         hipGetErrorString(e_), __FILE__, __LINE__);                    \
  } while (0)

// Tile shapes (cells x cells per workgroup) the autotuner chooses from, FP64
// and FP32C.  Phase 2 of the stage kernel visits H*H*CX*CY interior slots plus
// H*(CX+CY)+1 far-end points; 6x4 (MCV4: 247) and 8x7 (MCV3: 255) fill 256
// threads in one pass, the larger shapes re-read less halo per cell.
constexpr int kTileVariants = 4;
template <int DOF> struct TileSet;
template <> struct TileSet<3> {
  static constexpr int cx[kTileVariants] = {8, 16, 10, 12};
  static constexpr int cy[kTileVariants] = {7, 4, 5, 6};
};
template <> struct TileSet<4> {
  static constexpr int cx[kTileVariants] = {6, 8, 5, 6};
  static constexpr int cy[kTileVariants] = {4, 4, 5, 6};
};

template <int DOF> struct TileSet32;
template <> struct TileSet32<3> {
  static constexpr int cx[kTileVariants] = {8, 16, 10, 16};
  static constexpr int cy[kTileVariants] = {7, 8, 5, 4};
};
template <> struct TileSet32<4> {
  static constexpr int cx[kTileVariants] = {6, 8, 8, 10};
  static constexpr int cy[kTileVariants] = {4, 4, 8, 6};
};

// Where the boundary pass runs: inside the next stage's kernel (its side tiles
// finish the points they stage) or in a launch of its own after each stage.
// The launch costs a dispatch and a drained chip, which dominates small work;
// inside, the side tiles live longer and drag on launches that fill the chip
// several times over.  The pass is built into the kernels of the two small tile
// shapes of each order, which small work takes.
// The limit, 18 tiles per CU, from both sides measured (us per step, launch of
// its own / inside): MCV3 6x32^2 FP64 RK4 38.4 / 29.1, 6x90^2 FP32C RK3 (972
// tiles) 30.2 / 26.9, MCV4 6x96^2 FP64 (2400) 91.7 / 88.0, MCV3 6x181^2 FP64 RK3
// (4218) 74.0 / 69.5, MCV4 6x160^2 FP64 (6144) 177.5 / 178.2, 6x384^2 FP32C
// 730 / 782; MCV3 6x90^2 FP32C ensembles per stage, 1 member 12.6 / 11.0, 4
// members (3888) 25.4 / 25.0, 6 members (5832) 32.0 / 32.8, 20 members 99.5 / 103.9.
constexpr int kFusedMaxTiles = 18 * 256;
inline bool sides_in_stage(int tile_variant, long long tiles) {
  return (tile_variant == 0 || tile_variant == 2) && tiles <= kFusedMaxTiles;
}

// Upper bound of the device bytes one solve of this configuration allocates
// (exact when the metric terms differ between panels).
size_t footprint_bytes(const mcv_config *c);

// The RK stages of a time step (time_scheme_mod.F90:13-69).  Levels: 0 = Yn
// (updated in place by the last stage), 1 and 2 = intermediate stage states.
// Each stage has a band of its own and reads that of the stage before it, which
// other workgroups of the same launch may still be reading; the last stage's
// keeps the raw lines of Y_n until the next step's last stage.
struct StageSpec {
  int kind, in, out;
  double c1;  // stage increment coefficient (x dt)
};
inline int stage_count(int scheme) { return scheme == MCV_RK4 ? 4 : 3; }
// The second stage is the one that the autotuners repeat: S1, S2, the
// accumulator and the first two bands, all it touches beside reading Y_n, are
// written anew by every step.
constexpr int kTuneStage = 1;
inline StageSpec stage_spec(const mcv_config &c, int s) {
  const double dt = c.dt;
  const StageSpec rk4[4] = {{kRK4S1, 0, 1, 0.5 * dt}, {kRK4S2, 1, 2, 0.5 * dt},
                            {kRK4S3, 2, 1, dt}, {kRK4S4, 1, 0, dt}};
  const StageSpec rk3[3] = {{kRK3S1, 0, 1, dt}, {kRK3S2, 1, 2, 0.25 * dt},
                            {kRK3S3, 2, 0, 2.0 / 3.0 * dt}};
  return c.scheme == MCV_RK4 ? rk4[s] : rk3[s];
}

// Arguments of stage s of a solve's time step, and of the boundary pass on the
// level it wrote.
StageArgs stage_args64(const mcv_handle *h, int s);
StageArgs32 stage_args32(const mcv_handle *h, int s);
BoundaryArgs boundary_args64(const mcv_handle *h, int s);
BoundaryArgs32 boundary_args32(const mcv_handle *h, int s);

// Milliseconds per stage of every tile shape: use(v) switches to shape v,
// stage() enqueues a stage as the steps would run it, boundary launch included
// where the shape needs one.  The shapes take turns, `reps` rounds, so that a
// drift meets them all; a turn is timed behind a stage that is not, over about
// kTuneMs (at most kTuneStages), and the best turn counts.  A shape that is a
// fifth behind after a round is not tried again.
constexpr float kTuneMs = 0.1f;
constexpr int kTuneStages = 8;
template <class Use, class Stage>
int time_shapes(hipStream_t stream, hipEvent_t *ev, int reps, const Use &use, const Stage &stage,
                double *ms) {
  int stages[kTileVariants] = {1, 1, 1, 1};
  static_assert(kTileVariants == 4, "one entry per shape");
  for (int r = -1; r < reps; ++r)  // the first round loads the code and sets the stretches
    for (int v = 0; v < kTileVariants; ++v) {
      if (r > 0 && ms[v] > 1.2 * *std::min_element(ms, ms + kTileVariants)) continue;
      int rc = use(v);
      for (int k = 0; k <= stages[v] && rc == MCV_OK; ++k) {
        if (k == 1) HIP_TRY(hipEventRecord(ev[0], stream));
        rc = stage();
      }
      if (rc) return rc;
      HIP_TRY(hipEventRecord(ev[1], stream));
      HIP_TRY(hipEventSynchronize(ev[1]));
      float t = 0.f;
      HIP_TRY(hipEventElapsedTime(&t, ev[0], ev[1]));
      t /= stages[v];
      ms[v] = r <= 0 ? t : std::min(ms[v], (double)t);
      if (r < 0) stages[v] = t * kTuneStages < kTuneMs ? kTuneStages : 1 + (int)(kTuneMs / t);
    }
  return MCV_OK;
}

}  // namespace mcv

// One solve on one device.
struct mcv_handle {
  mcv_config cfg{};
  int H = 0, npv = 0, nh = 0;
  long long np = 0;  // points per field
  hipStream_t stream = nullptr;
  mcv::MeshDev mesh{};
  std::vector<void *> allocs;  // every device allocation, freed together
  size_t device_bytes = 0;     // their sizes summed
  mcv::D2 *lpu[3] = {};        // levels (Yn, S1, S2): {phi, u} pairs
  double *lvv[3] = {};         //   and v
  double *phi_ref = nullptr;   // FP32C: the projected initial geopotential (FP64)
  double *acc[3] = {};         // RK4 accumulator: acc[0] {phiG, u} pairs, acc[2] v
  mcv::D3 *band_raw[4] = {};   // raw band lines written by the stage kernel, per stage
  double *cu0 = nullptr, *cv0 = nullptr;  // host contra winds until the first stage
  bool first_pending = true;
  double *partials = nullptr;
  int diag_blocks = 0;
  double *diag_out = nullptr;
  double *pack[6] = {};
  // history fields (allocated by the first mcv_hip_history_fields call):
  // u, v, contraU, contraV, phi, phi_t, zonal, meridional; uC, vC, phiC
  double *hist[8] = {};
  double *histc[3] = {};
  int64_t steps = 0;
  int tile = 0;  // index into the tile shapes of the solve's order
  // per-kernel timing (mcv_hip_step_timed)
  bool timing = false;
  hipEvent_t ev[3] = {};
  double stage_ms = 0.0, boundary_ms = 0.0;
  // FP32C form (precision == MCV_FP32C): FP32 levels of (phi - phi_ref, u, v),
  // compensation words of Y_n and FP32 accumulator; phi_ref is the projected
  // initial geopotential (FP64).
  bool fp32c = false;
  // levels, compensation words of Y_n and accumulator: {phi', u, v} records
  mcv::F3 *l32[3] = {};
  mcv::F3 *c32 = nullptr;
  mcv::F3 *a32 = nullptr;
  double *join[3] = {};  // FP64 reconstruction of Y_n for read-back and integrals
  mcv::MeshF32 mesh32{};
};
