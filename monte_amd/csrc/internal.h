// Internal declarations shared by the host C++ and the gfx950 kernels of
// libmonte.so.  Not part of the public ABI (include/monte.h is).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/monte.h"

namespace monte {

// IEEE FP64 add, subtract and multiply that the compiler never fuses into an
// FMA, for expressions that must round exactly as a CPU evaluates them (the
// pragma marks the operations themselves, so it holds after inlining; the
// __dadd_rn family alone does not stop that fusion).
__host__ __device__ inline double xadd(double a, double b) {
#pragma clang fp contract(off)
  return a + b;
}
__host__ __device__ inline double xsub(double a, double b) {
#pragma clang fp contract(off)
  return a - b;
}
__host__ __device__ inline double xmul(double a, double b) {
#pragma clang fp contract(off)
  return a * b;
}

constexpr int kRows = MONTE_TABLE_ROWS;
constexpr int kMaxLabels = MONTE_MAX_LABELS;
// MC detector tile: one birth of a wave (64 lanes) covers one tile of one cycle.
constexpr int kTileU = 8, kTileV = 8;
constexpr int kPadLo = 1;  // zero guard cells before u / v in padded filtered projections
constexpr int kPadHi = 3;  // and after (covers the +1 bilinear tap at the window edge)

// ------------------------------------------------------------------ FDK
// Per-view backprojection coefficients (computed on the host in FP64).  For a
// voxel centre (X,Y,Z):
//   U  = cx X + cy Y + c0                      distance along the central ray
//   su = su0 + suk (ax X + ay Y) / U           sample coordinate along u
//   sv = sv0 + svk Z / U                       sample coordinate along v
//   Dd = d0 + dx X + dy Y - sgn(gx X + gy Y) |hx X + hy Y|
//   w  = fac (wn / Dd)^2                       distance weight x angular step
// Standard preset: Dd = U, wn = sod, fac = dangle.  bp3d20 preset: Dd = 60 - d
// with d the signed point-line distance of recon/bp3d20_325.cpp:145-153.
// The sample coordinates are formed per voxel column in FP64 (U, 1/U, su and
// the first sv of the column's z-chunk), then split into an integer pixel
// index and an FP32 fraction, so the per-voxel FP32 work only moves a small
// fraction along v.  The bp3d20 sign test sgn(gx X + gy Y) is evaluated in
// unfused FP64 exactly as the reference evaluates it: at columns where it is
// zero in exact arithmetic (e.g. X = -Y at 135 degrees) the reference's
// rounding decides the sign of d, and with it the weight.
struct BpView {
  double cx, cy, c0;
  double ax, ay;
  double su0, suk;
  double sv0, svk;
  double gx, gy;
  float wn, d0, dx, dy;
  float hx, hy, fac, pad0;
};
static_assert(sizeof(BpView) == 120, "BpView layout");

// Geometry-wide constants of the backprojector.
struct BpGrid {
  int nx, ny, nz, nu, nv, n_views;
  int pitch;          // padded row pitch of filtered projections (nu + kPadLo + kPadHi)
  int rows;           // padded rows (nv + kPadLo + kPadHi)
  double gx0, gsx;    // X = gx0 + x * gsx (unfused, as recon/bp3d20_325.cpp:107)
  double gy0, gsy;
  double gz0, gsz;
  double lo_u, hi_u;  // valid sample window along u (inclusive)
  double lo_v, hi_v;
  int x0, x1;         // x range reconstructed (bp3d20 ROI)
  int mask;           // 1: sphere mask in voxel index space
  float mask_r2;
  int mcx, mcy, mcz;  // mask centre (voxel index)
};

// What the backprojector's tiling has to know of a scan: how far the volume
// reaches from the axis, the scale of the sample coordinates, and whether a
// quarter turn maps the scan onto itself.
struct BpReach {
  double sod, rad;  // source distance; largest in-plane distance of a voxel centre from the axis
  double suk, svk;  // |d(su)| per unit of y'/U, |d(sv)| per unit of Z/U
  bool zeros;       // the guard cells of the padded views hold zeros, and there is no mask
  bool half;        // view k + V/2 is view k turned by 180 degrees and so is the volume
  int turn;         // +-1: view k + V/4 is view k turned by +-90 degrees and so is the volume; 0: neither
};

// Filter constants: weight(r,c) = D / sqrt(D^2 + (a_u + b_u r)^2 + (a_v + b_v c)^2),
// out = cs * sum_r weight * p * h[r - b].
struct FilterParams {
  int nu, nv, n_views;
  int pitch, rows;    // padded output layout
  float D, a_u, b_u, a_v, b_v;
  float cs;
};

void compute_bp_views(const monte_geom& g, std::vector<BpView>& out);
BpGrid compute_bp_grid(const monte_geom& g);
BpReach compute_bp_reach(const monte_geom& g, const BpGrid& grid);
FilterParams compute_filter_params(const monte_geom& g);
void compute_filter_taps(const monte_geom& g, std::vector<float>& h);  // h[0..2nu-2], centre nu-1
// The factors cos(2 pi k / 64) of the filter's transforms
constexpr float kCos64[17] = {
    1.0f, 0.99518472667219693f, 0.98078528040323043f, 0.95694033573220882f, 0.92387953251128674f,
    0.88192126434835505f, 0.83146961230254524f, 0.77301045336273699f, 0.70710678118654757f,
    0.63439328416364549f, 0.55557023301960229f, 0.47139673682599781f, 0.38268343236508984f,
    0.29028467725446233f, 0.19509032201612833f, 0.09801714032956077f, 0.0f};
constexpr float cos64(int k) {
  k &= 63;
  return k <= 16 ? kCos64[k] : (k <= 32 ? -kCos64[32 - k] : (k <= 48 ? -kCos64[k - 32] : kCos64[64 - k]));
}
// Tables of the filter's row transforms: float2 twiddles [points], spectrum [points]
void compute_filter_spectrum(const monte_geom& g, int points, int lanes, std::vector<float>& out);

// ------------------------------------------------------------------- MC
// Device attenuation tables of one job, per label and keV row:
//   m[l][e] = (mu, photo/total, (photo+coherent)/total, 0), mu in cm^-1
//   mumax[e] = max_l mu  (the Woodcock majorant)
struct McTables {
  float4 m[kMaxLabels][kRows];
  float mumax[kRows];
  float pad[3];
};

// Device job descriptor of the persistent transport kernel.
struct McJob {
  const uint8_t* labels;
  const McTables* tables;
  const float* spectrum_cdf;     // [kRows] or null (mono)
  const float2* view_cs;         // cos, sin per view
  double* primary;
  double* scatter;
  int nx, ny, nz, nu, nv;
  int view_begin, n_views_sim;   // simulated views (indices into the tally arrays)
  float vx, vy, vz;
  float bx0, by0, bz0, bx1, by1, bz1;  // phantom box
  float inv_vx, inv_vy, inv_vz;
  float ix0, iy0, iz0;           // -b0 / v: voxel index = q inv_v + i0
  float sod, sdd;
  float un0, us, vn0, vs;        // u_idx = un0 + us * y', v_idx = vn0 + vs * z'
  float u_step, v_step;          // 1/us, 1/vs (signed pitch)
  float e_kev;
  int max_int, coherent;
  uint32_t key0, key1, job_id;
  uint32_t solid_set;            // label-set bits that attenuate at some energy (bit 4: any label does)
  uint32_t photons_per_view;
  // Photon n of a view aims at pixel j = n mod (nu nv) in aim order (iv nu + iu),
  // in cycle c = n / (nu nv).  A work unit is a group of `tile_group` detector
  // tiles of kTileU x kTileV pixels (tiles numbered u fastest, `tiles_u` per row,
  // `tiles` in all) over `cycle_block` consecutive cycles, and a birth takes one
  // tile of one cycle: so a unit's primary tallies fall on a few lines that it
  // hits once per cycle, and the units in flight share a narrow detector band.
  uint32_t tiles_u, tiles, tile_group;
  uint32_t cycles, cycle_block, cycle_blocks;  // ceil(photons / (nu nv)); per unit; blocks
  uint32_t batches_per_view;     // ceil(tiles / tile_group) * cycle_blocks
  uint64_t unit_begin;           // first global work unit of this job
  uint64_t unit_count;
  const uint8_t* ray_set;        // [n_views_sim][nu nv] first-flight label sets (aim order), or null
};

// FP64 geometry of the first-flight label sets (ray_sets_kernel).  A photon's
// first flight runs from the source towards the centre of its pixel, so the
// labels that segment crosses bound the attenuation it meets, and the largest
// mu among them is a valid Woodcock majorant for that flight.  Sets are bit
// masks: bit l for labels 0..3, bit 4 for any label >= 4 (then the flight
// takes the global majorant).
struct RayGrid {
  double un0, u_step, vn0, v_step;  // pixel centre: y' = (iu + 1/2 - un0) u_step, z' likewise
  double sod, xd;                   // source distance, detector plane x' = xd
  double org[3], bw[3];             // brick grid corner (the phantom's) and brick size
  int nb[3];                        // bricks per axis
  int nu, nv;
};

// What the launches before a transport need of one job: its flight box (the
// bounding box of its attenuating voxels, formed in `box`) and its first-flight
// label sets.  The jobs of a launch share the grids of these kernels; a job's
// blocks start at prep_begin and ray_begin.
struct McPrep {
  const uint8_t* labels;
  const double* cs64;            // FP64 (cos, sin) of every view, or null without sets
  uint8_t* bricks;               // brick sets [nb2][nb1][nb0]
  uint8_t* sets;                 // label sets [n_views][nu nv]
  RayGrid ray;
  double vox[3];                 // voxel size
  uint32_t solid;                // bit l: label l attenuates at some energy
  int nx, ny, nz;
  int box[6];                    // minima, maxima (voxels); {INT_MAX x 3, -1 x 3} before the launch
  int brick;                     // voxels a side, 0: no sets
  uint32_t box_blocks;           // the first of the job's prep blocks, for the box; the rest for bricks
  uint32_t prep_begin, ray_begin;
};
static_assert(sizeof(McPrep) <= 256, "the static scratch of the allocation-free projection counts 256 bytes for it");

// FP64 ray geometry of the exact primary estimator.
struct PrimaryGeom {
  double sod, sdd, un0, u_step, vn0, v_step;
  double b0[3], vox[3];
  int n[3];
  int nu, nv, n_views;
};

struct McCounters {  // device-side statistics
  unsigned long long histories, steps, interactions, photo, coherent, compton;
  unsigned long long tallied_primary, tallied_scatter, missed, capped;
};

// Where a launch's job descriptors, tables, CDFs, view tables, queue, counters
// and flight boxes sit in its device buffer.
struct McLayout {
  size_t jobs_off = 0, tab_off = 0, q_off = 0, cnt_off = 0, prep_off = 0, total = 0;
  std::vector<size_t> cdf_off, cs_off, cs64_off;
};

// A transport launch whose descriptors are in place in device memory;
// launching it is stream-ordered work only (capturable into a graph).
struct McPrepared {
  char* base = nullptr;
  McLayout L;
  int n = 0, slots = 1;
  uint64_t units = 0;
  uint32_t chunk = 1;  // units per queue chunk (the first job's simulated views; more with several jobs)
  std::vector<char> host;  // the uploaded descriptors, kept until the stream has passed the upload
  unsigned int* queue() const { return (unsigned int*)(base + L.q_off); }
  McCounters* counters() const { return (McCounters*)(base + L.cnt_off); }
};

}  // namespace monte

// ------------------------------------------------------------------ context
struct monte_ctx {
  int device = 0;
  hipStream_t own_stream = nullptr;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;  // times transport launches (created once, with the context)
  bool host_ptrs = false;
  std::string err;
  int n_cu = 256;

  // pinned host memory the transport's counters are copied to (as many jobs as fit)
  monte::McCounters* host_counters = nullptr;

  // attenuation tables (host copy, FP64): [n_tables][4][201]
  std::vector<double> tables;
  int n_tables = 0;

  monte_tuning tuning{};

  // growable device workspaces:
  //   0 forward filtered stack (padded)   1 adjoint filtered stack (padded)
  //   2 MC descriptors                    3 FDK constants (taps + per-view coefficients)
  //   4..7 staging for host-pointer mode and tuning scratch
  //   8 z-fastest copy of the volume for the matched projector
  //   9 column lists of the matched projector (per geometry)
  //  10 end-to-end step: MC descriptors and loss partial sums
  //  11 first-flight label sets of MC launches   12 those of the end-to-end step
  static constexpr int kSlots = 13;
  void* ws[kSlots] = {};
  size_t ws_size[kSlots] = {};

  // FDK constants cached by geometry
  std::vector<double> const_key;
  size_t taps_off = 0, views_off = 0, fft_off = 0;

  // projector column lists cached by geometry: offsets, then the lists
  std::vector<double> plan_key;
  size_t plan_list_off = 0;

  // hipGraph cache for monte_fdk_graph
  hipGraphExec_t graph_exec = nullptr;
  hipGraph_t graph = nullptr;
  std::vector<double> graph_key;

  // bumped by every monte_load_tables (keys of cached MC descriptors)
  uint64_t tables_gen = 0;

  // end-to-end step: prepared MC launch (keyed by job), and its graph
  monte::McPrepared e2e_mc;
  std::vector<double> e2e_mc_key;
  hipGraphExec_t e2e_exec = nullptr;
  hipGraph_t e2e_graph = nullptr;
  std::vector<double> e2e_graph_key;
};

namespace monte {

// error helpers
int fail(monte_ctx* c, int code, const std::string& msg);
#define MONTE_HIP(ctx, expr)                                                              \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess)                                                                 \
      return ::monte::fail((ctx), MONTE_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

// workspace slot i grown to at least bytes; returns nullptr on failure
void* workspace(monte_ctx* c, int slot, size_t bytes);

// Device scratch of the allocation-free entry points (a static device array,
// one per GPU; noalloc.hip): its address on `device` and its size, or nullptr
// before noalloc_setup has run on that device.
constexpr size_t kNoAllocScratchBytes = 128 * 1024;
int noalloc_setup(int device);  // with `device` current; 0 or a hipError_t
void* noalloc_scratch(int device);

// ---------------------------------------------------------- kernel launches
// Blocks of `threads` that one launch may have: HIP takes fewer than 2^32 threads along an axis.
constexpr uint64_t max_blocks(int threads) { return 0xffffffffull / (unsigned)threads; }

// FDK (fdk.hip)
// What a scan's backprojection and projection run, for tests: columns of an orbit (0: straight from
// memory, -1: refused), groups, voxels a thread, stack, tile_x, patch rows and columns, blocks (low
// 32 bits); the row projector's orbit (0: by voxels), blocks of rows, rows / 64 of a block, voxels a row.
constexpr int kRouteWords = 12;
void fdk_routes(const BpGrid& grid, const BpReach& reach, int nviews_chunk, int lds_r0, int lds_rows,
                const monte_tuning& t, int32_t out[kRouteWords]);
hipError_t launch_fill(float* p, float v, size_t n, hipStream_t s);
hipError_t launch_pad_copy(const float* filt, float* filt_pad, int n_views, int nu, int nv, int pitch, int rows,
                           hipStream_t s);
hipError_t launch_unpad_copy(const float* filt_pad, float* filt, int n_views, int nu, int nv, int pitch, int rows,
                             hipStream_t s);
hipError_t launch_fill_pads(float* buf, int n_views, int nu, int nv, int pitch, int rows, int wrap, hipStream_t s);
hipError_t launch_fold_pads(float* buf, int n_views, int nu, int nv, int pitch, int rows, hipStream_t s);
// filt_pad [n_views][rows][pitch] -> vol, views [view0, view0 + nviews_chunk)
hipError_t launch_backproject(const float* filt_pad, const BpView* views, int view0, int nviews_chunk,
                              const BpGrid& grid, const BpReach& reach, float* vol, int accumulate,
                              const monte_tuning& t, hipStream_t s);
// volT: the volume with z fastest ([y][x][z], see launch_transpose_zx); every
// cell of the padded views [view0, view0 + nviews_chunk) is written.  Padded
// rows [lds_r0, lds_r0 + lds_rows) must hold every row the views' voxels can
// reach (projector_rows); the others are written as zeros.
// Detector strips per view of the matched projector.
int project_strips(const BpGrid& grid);
// Column lists of the projector for views [0, n_views): with write false,
// offs[k * project_strips + st] receives each list's length; with write true,
// offs holds the exclusive prefix sums (plus the total at the end) and the
// lists are written to list.  orbit 2, 4: of the first columns of orbits only.
hipError_t launch_project_plan(const BpView* views, int n_views, const BpGrid& grid, int orbit, uint32_t* offs,
                               uint32_t* list, bool write, hipStream_t s);
// The projector by rows, where project_orbit is not 0 (its lists made for that
// orbit); launch_project elsewhere.
int project_orbit(const BpGrid& grid, const BpReach& reach, const monte_tuning& t);
hipError_t launch_project_rows(const float* volT, const BpView* views, int view0, int nviews_chunk, const BpGrid& grid,
                               const BpReach& reach, int orbit, float* filt_pad, int lds_r0, int lds_rows,
                               const uint32_t* plan_offs, const uint32_t* plan_list, hipStream_t s);
hipError_t launch_project(const float* volT, const BpView* views, int view0, int nviews_chunk, const BpGrid& grid,
                          float* filt_pad, int lds_r0, int lds_rows, const uint32_t* plan_offs,
                          const uint32_t* plan_list, const monte_tuning& t, hipStream_t s);
// Padded detector rows reachable by the voxels of views [view0, view0 + n).
void projector_rows(const std::vector<BpView>& views, int view0, int n, const BpGrid& grid, int& lds_r0,
                    int& lds_rows);
hipError_t launch_transpose_zx(const float* vol, float* volT, int nx, int ny, int nz, hipStream_t s);
// The filter with the guard cells (wrap: of the bp3d20 preset), and its transpose; tables of
// compute_filter_spectrum.
int filter_fft_points(int nu);
int filter_fft_lanes(int points);
hipError_t launch_fdk_filter(const float* proj, float* filt_pad, const float* taps, const float2* tables,
                             const FilterParams& fp, int wrap, hipStream_t s);
hipError_t launch_fdk_filter_T(const float* filt_pad, float* proj, const float* taps, const float2* tables,
                               const FilterParams& fp, hipStream_t s);

// MC (mc.hip)
// The work queue is kMcQueues counters kMcQueueStride words apart, each
// handing out one chunk (`chunk` consecutive work units) per round, and block
// b draws from queue b mod kMcQueues first.  Blocks are dealt to the 8 XCDs
// round robin, so an XCD draws from 3 of the queues and its L2 serves their
// chunks.  With units of detector tiles, 8, 16, 24, 32 and 64 queues took
// 84.5, 84.2, 83.4, 88.0 and 105.8 ms at 360 views x 1e7 photons, and 24 took
// 815.8 against 824.7 ms for 32 at 1e8 photons (fewer queues keep an XCD's
// units on fewer tiles; with units of consecutive photons 8, 16 and 32 had
// taken 164, 161 and 158 ms, the counters' contention then mattering more).
constexpr int kMcQueues = 24;
constexpr int kMcQueueStride = 16;
constexpr size_t kMcQueueBytes = sizeof(unsigned int) * kMcQueues * kMcQueueStride;
// Counter q starts past the units that the queue's waves take by rank, and a bit
// per spent queue sits in a word of the last counter's line.
constexpr int kMcSpentWord = (kMcQueues - 1) * kMcQueueStride + kMcQueueStride / 2;
static_assert(kMcQueues < 32, "one bit per queue");
__host__ __device__ inline unsigned int mc_queue_start(int q, int waves_per_block, int grid) {
  return (unsigned int)(waves_per_block * ((grid - q + kMcQueues - 1) / kMcQueues));
}
// Statistics: `slots` sets of counters per job, a block adding to set b mod slots
// (in one set, the adds of the 6144 waves of a short launch took 400 us); the
// host adds them up.
constexpr int kMcSlots = 32, kMcSlotsNoAlloc = 3;
hipError_t launch_mc_transport(const McJob* jobs_dev, int n_jobs, uint64_t total_units, uint32_t chunk,
                               unsigned int* queue, McCounters* counters, int slots, int block, int grid,
                               hipStream_t s);
hipError_t launch_mc_reset(unsigned int* queue, McCounters* counters, int n_counters, int block, int grid,
                           hipStream_t s);
// The flight boxes and brick sets of all jobs (prep_blocks in all), then their
// label sets (ray_blocks) and the boxes written into their descriptors.
// Brick sets: per brick of b^3 voxels widened by one voxel; label sets: per
// simulated view and pixel in aim order.  max_planes: the largest job's brick
// planes (nb0 + nb1 + nb2 + 3).  Without sets, launch_mc_boxes does the latter
// alone.
hipError_t launch_mc_prep(McPrep* preps, int n_jobs, uint32_t prep_blocks, hipStream_t s);
hipError_t launch_ray_sets(const McPrep* preps, McJob* jobs, int n_jobs, uint32_t ray_blocks, uint64_t max_planes,
                           hipStream_t s);
hipError_t launch_mc_boxes(const McPrep* preps, McJob* jobs, int n_jobs, hipStream_t s);
constexpr int kRayBlock = 256;  // pixels per block of the label sets
// prep: the phantom's flight box (launch_mc_prep without bricks).  bins:
// [n_bins][1 + n_labels] weight and attenuation of labels 0 .. n_labels - 1; weight
// is the sum of the weights, or 0 for one mono-energetic bin.
hipError_t launch_primary_exact(const PrimaryGeom& P, const McPrep* prep, const double* cs64, const uint8_t* labels,
                                const double* bins, int n_bins, int n_labels, double weight, float* out,
                                hipStream_t s);
// counts2 (nullable) is added to counts before the conversion
hipError_t launch_counts_to_lineint(const double* counts, const double* counts2, float* out, int n_views, int nu,
                                    int nv, uint64_t photons_per_view, hipStream_t s);
// out = a - b; partial[blk] = FP64 sum of out^2 over block blk's fixed share
// (grid-stride, reduced in a fixed order), then loss = 0.5 * sum(partial) in
// one more fixed-order pass: deterministic, so graph replays are bitwise equal.
constexpr int kLossBlocks = 1024;
hipError_t launch_residual_loss(const float* a, const float* b, float* out, size_t n, double* partial, double* loss,
                                hipStream_t s);
hipError_t launch_counts_to_lineint_flat(const double* counts, const double* flat, int flat_views, float* out,
                                         int n_views, int nu, int nv, hipStream_t s);

}  // namespace monte
