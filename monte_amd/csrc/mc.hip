// Monte Carlo photon transport for gfx950.
//
// Reference: the projection kernel of monte_cu/CBCT_real325.cu:419-846 and
// photon::delta_sampling :848-975 (voxel form: CBCT_real325im.cu:425-962).
// The reference gives each thread one detector pixel and loops serially over
// 360 views x 10^4 photons, so lanes idle whenever their photons' histories
// differ in length.  Here:
//   * one photon per lane, its random numbers drawn from a Philox4x32-10
//     stream keyed by (seed) with counter (block, photon, view, job), so any
//     history can be replayed and results do not depend on scheduling;
//   * the kernel is persistent: waves pull work units (a detector tile of 8 x 8
//     pixels over a block of photon cycles, in one view) from device work
//     queues shared by all jobs of a launch (24 counters, each block drawing
//     from its own first), so the units in flight share a thin slab of the
//     phantom and few tally lines;
//   * each loop iteration advances every flying lane by up to two Woodcock
//     steps (one Philox block).
//     Lanes that collide (real interaction pending), end their flight (tally
//     pending) or die (absorbed, capped) park; the wave runs the interaction
//     code, or tallies and refills (ballot + mbcnt prefix ranks), only once
//     enough lanes are parked or nothing else can run, so those branches
//     execute near full width instead of for one lane at a time;
//   * photons are born 64 at a time, one per lane with every lane active, into
//     a per-wave LDS buffer that dead lanes then take from;
//   * flights are clipped to the bounding box of the voxels that attenuate
//     (the reference clips to the phantom box, quirk Q9; mu is 0 in the
//     margin between the two, so no history changes) and the first step
//     starts at the box entry;
//   * primary and scatter counts are tallied with FP64 atomics.  Every tally
//     adds 1.0, so sums are exact integers and independent of order;
//   * statistics are counted per wave, from ballots of the lanes where events
//     happen, into 64-bit counters in LDS that go to the job's when it is
//     flushed.
#include <algorithm>
#include <climits>

#include "internal.h"

namespace monte {

// ------------------------------------------------------------------ RNG
// Philox4x32-10 (Salmon et al., SC'11).
__device__ inline void philox10(uint32_t& c0, uint32_t& c1, uint32_t& c2, uint32_t& c3, uint32_t k0,
                                uint32_t k1) {
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    // one 32 x 32 -> 64-bit multiply gives both halves (v_mad_u64_u32)
    const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
    const uint32_t lo0 = (uint32_t)p0, hi0 = (uint32_t)(p0 >> 32);
    const uint32_t lo1 = (uint32_t)p1, hi1 = (uint32_t)(p1 >> 32);
    // hi ^ c ^ k as one three-input XOR (truth table 0x96)
    uint32_t n0, n2;
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(n0) : "v"(hi1), "v"(c1), "s"(k0));
    asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(n2) : "v"(hi0), "v"(c3), "s"(k1));
    c0 = n0; c1 = lo1; c2 = n2; c3 = lo0;
    k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
  }
}

// A photon's stream: counter (ctr, photon, view, job); the four outputs of the
// last block are consumed in order.
struct Stream {
  uint32_t ctr, photon, view;
  uint32_t b0, b1, b2, b3;
  int left;
};

// ((x >> 8) + 1/2) 2^-24 in one rounding
__device__ inline float u01(uint32_t x) { return fmaf((float)(x >> 8), 5.9604644775390625e-08f, 2.98023223876953125e-08f); }

__device__ inline float next_u01(Stream& s, uint32_t job, uint32_t k0, uint32_t k1) {
  if (s.left == 0) {
    uint32_t c0 = s.ctr, c1 = s.photon, c2 = s.view, c3 = job;
    philox10(c0, c1, c2, c3, k0, k1);
    s.b0 = c0; s.b1 = c1; s.b2 = c2; s.b3 = c3;
    s.ctr += 1;
    s.left = 4;
  }
  const uint32_t x = s.b0;
  s.b0 = s.b1; s.b1 = s.b2; s.b2 = s.b3;
  s.left -= 1;
  return u01(x);
}

// The stream's next three uniforms, in order, with at most one new block: the
// same numbers as three next_u01 calls, but with one Philox call site, so a
// wave whose lanes sit at different offsets in their blocks runs the rounds
// once per trial of a rejection loop rather than once per draw.
__device__ inline void next3_u01(Stream& s, uint32_t job, uint32_t k0, uint32_t k1, float& r1, float& r2, float& r3) {
  uint32_t n0 = 0, n1 = 0, n2 = 0, n3 = 0;
  const int left = s.left;
  if (left < 3) {
    n0 = s.ctr; n1 = s.photon; n2 = s.view; n3 = job;
    philox10(n0, n1, n2, n3, k0, k1);
    s.ctr += 1;
  }
  // the unconsumed words in order are b0 .. b(left-1), then n0 .. n3
  const uint32_t x0 = left == 0 ? n0 : s.b0;
  const uint32_t x1 = left == 0 ? n1 : (left == 1 ? n0 : s.b1);
  const uint32_t x2 = left == 0 ? n2 : (left == 1 ? n1 : (left == 2 ? n0 : s.b2));
  // and what stays: left + 1 words after a new block, left - 3 otherwise
  const uint32_t w0 = left == 0 ? n3 : (left == 1 ? n2 : (left == 2 ? n1 : s.b3));
  const uint32_t w1 = left == 1 ? n3 : n2;
  s.b0 = w0; s.b1 = w1; s.b2 = n3;
  s.left = left < 3 ? left + 1 : left - 3;
  r1 = u01(x0); r2 = u01(x1); r3 = u01(x2);
}

// Reciprocal to 1 ulp (v_rcp_f32).  The physics below draws angles and
// energies whose parity with the FP64 oracle is statistical, so it takes the
// hardware reciprocal, square root and sine instead of correctly rounded
// sequences.
__device__ inline float rcp(float x) { return __builtin_amdgcn_rcpf(x); }

// --------------------------------------------------------------- physics
// Kahn's rejection sampling of the Klein-Nishina distribution as written in
// CBCT_real325.cu:687-722 (lambda = 511/E); returns rho = lambda'/lambda.
// Each trial takes the stream's next three uniforms (r1, r2, r3) whichever
// branch r1 picks, as the reference's trials do.
__device__ inline float kahn(float lambda, Stream& s, uint32_t job, uint32_t k0, uint32_t k1) {
  const float il2 = 2.0f * rcp(lambda);
  const float p1 = (lambda + 2.0f) * rcp(9.0f * lambda + 2.0f);
  for (int guard = 0; guard < 1000; ++guard) {
    float r1, r2, r3;
    next3_u01(s, job, k0, k1, r1, r2, r3);
    if (r1 < p1) {
      const float ro = 1.0f + il2 * r2;
      const float iro = rcp(ro);
      if (r3 <= 4.0f * (iro - iro * iro)) return ro;
    } else {
      const float ro = (lambda + 2.0f) * rcp(lambda + 2.0f * (1.0f - r2));
      const float q = lambda - ro * lambda + 1.0f;
      if (r3 <= 0.5f * (q * q + rcp(ro))) return ro;
    }
  }
  return 1.0f;  // unreachable in practice (acceptance > 1/2 per trial)
}

// Thomson angular distribution (1 + mu^2): closed-form inverse CDF
// mu = cbrt(A) - cbrt(1/A), A = |a| + sqrt(a^2 + 1) >= 1, a = 4u - 2, with
// cbrt(A) = 2^(log2(A) / 3) on the hardware log and exp.
__device__ inline float thomson_mu(float u) {
  const float a = 4.0f * u - 2.0f;
  const float A = fabsf(a) + __builtin_amdgcn_sqrtf(a * a + 1.0f);
  const float c = __builtin_amdgcn_exp2f(__builtin_amdgcn_logf(A) * 0.333333343f);
  const float m = c - rcp(c);
  return a < 0.f ? -m : m;
}

// Rotate unit direction d by polar cosine c and azimuth phi = 2 pi w (w in
// revolutions, as the hardware sine takes it): c d + s (cos(phi) e1 +
// sin(phi) e2) with e1 = (dx dz, dy dz, -r^2)/r, e2 = (-dy, dx, 0)/r and
// r = sqrt(dx^2 + dy^2), which stays accurate near the poles (1 - dz^2 would
// cancel); only for d on the z axis is the pair the x and y axes.
__device__ inline void rotate_dir(float& dx, float& dy, float& dz, float c, float w) {
  const float s = __builtin_amdgcn_sqrtf(fmaxf(0.f, 1.f - c * c));
  const float sp = __builtin_amdgcn_sinf(w), cp = __builtin_amdgcn_cosf(w);
  const float r = __builtin_amdgcn_sqrtf(dx * dx + dy * dy);
  float nx, ny, nz;
  if (r > 1e-15f) {  // r^2 stays a normal FP32 number
    const float ir = rcp(r);
    nx = c * dx + s * (dx * dz * cp - dy * sp) * ir;
    ny = c * dy + s * (dy * dz * cp + dx * sp) * ir;
    nz = c * dz - s * r * cp;
  } else {
    nx = s * cp;
    ny = s * sp;
    nz = dz >= 0.f ? c : -c;
  }
  const float nn = rsqrtf(nx * nx + ny * ny + nz * nz);
  dx = nx * nn; dy = ny * nn; dz = nz * nn;
}

__device__ inline int ebin_of(float e) {
  int b = (int)(e + 0.5f);  // CBCT_real325.cu:489: row (int)(Energy + 0.5)
  return b < 1 ? 1 : (b > kRows - 1 ? kRows - 1 : b);
}

// Slab test along one axis, folded into [lo, hi]; false if the ray misses.
__device__ inline bool slab(float p, float d, float b0, float b1, float& lo, float& hi) {
  if (d != 0.f) {
    const float inv = __builtin_amdgcn_rcpf(d);  // 1 ulp: the box clip has voxel-scale slack
    float ta = (b0 - p) * inv, tb = (b1 - p) * inv;
    lo = fmaxf(lo, fminf(ta, tb));
    hi = fminf(hi, fmaxf(ta, tb));
    return true;
  }
  return p >= b0 && p < b1;
}

// Parametric interval of p + t d inside the phantom box.
template <class JT>
__device__ inline bool ray_box(float px, float py, float pz, float dx, float dy, float dz, const JT& J,
                               float& t0, float& t1) {
  float lo = -INFINITY, hi = INFINITY;
  const bool ok = slab(px, dx, J.bx0, J.bx1, lo, hi) && slab(py, dy, J.by0, J.by1, lo, hi) &&
                  slab(pz, dz, J.bz0, J.bz1, lo, hi);
  if (!ok || !(hi > lo)) return false;
  t0 = lo; t1 = hi;
  return true;
}

using CJob = const __attribute__((address_space(4))) McJob;
using CU32 = const __attribute__((address_space(4))) uint32_t;

__device__ inline int job_of_unit(const CJob* jobs, int n_jobs, uint64_t u) {
  int lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (jobs[mid].unit_begin <= u) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Photon state of one lane.
struct Photon {
  float px, py, pz;    // position (world)
  float dx, dy, dz;    // unit direction (world)
  float e;             // energy (keV)
  float t, t1;         // flight parameter and box-exit parameter
  float mumax;         // Woodcock majorant of the current table row
  float lscale;        // ln 2 / mumax: a free path is -log2(u) * lscale
  float mu0, mu1, mu2, mu3;  // mu of labels 0..3 at the current table row
  int eb;              // table row
  int lab;             // label at the pending collision
  int nint;            // real interactions so far
  int view;            // tally view index (absolute)
  float cv, sv;        // cos, sin of the view angle
};

// Per-wave LDS copy of the current job's per-energy tables, read at every
// birth and flight start (the spectrum search alone is 8 dependent reads).
constexpr int kGuide = 256;  // spectrum guide cells

// Photons born 64 at a time, one per lane with every lane active, wait here
// until dead lanes take them; all are of one view and one cycle of one
// detector tile, and slots are the lanes that made them, i.e. the tile's
// pixels.  The rays of the tile's pixels in that view (direction, flight-box
// entry t0 (0 when the source is not clipped) and exit t1 (-1: no flight),
// label set) are formed once per tile and view and serve every cycle of it;
// per photon there is only the table row eb.  slot[k] is the slot of the k-th
// photon that entered the flight box.  A taker forms the rest as the birth
// did: the photon index from the slot, the position from the source and t0,
// the energy from the table row, the majorant from the label set.
struct BirthBuffer {
  float4 d0[64];  // direction and box entry t0 of a slot's ray
  float t1[64];
  uint8_t set[64], eb[64], slot[64];
};

constexpr int kWaveStats = 10;
struct WaveTables {
  unsigned long long stats[kWaveStats];  // the wave's event counts for the current job
  float cdf[kRows];      // spectrum CDF (unused for mono jobs)
  float mumax[kRows];    // Woodcock majorant
  float mu[4][kRows];    // mu of labels 0..3
  // guide[g] = the energy row drawn for u = g / kGuide (rows are <= 200): a
  // draw u in [g, g + 1) / kGuide lies between guide[g] and guide[g + 1]
  uint8_t guide[kGuide + 4];
  BirthBuffer bb;
};
// 6 waves per SIMD (24 per CU) fit in a CU's 160 KB of LDS
static_assert(24 * sizeof(WaveTables) <= 160 * 1024, "WaveTables too large for 6 waves per SIMD");

// Inverse CDF of the spectrum (CBCT_real325.cu:479-486): the first row e in
// [1, kRows - 1] with cdf[e] >= u, or the last row, searched within [lo, hi].
__device__ inline int spectrum_row(const float* cdf, float u, int lo, int hi) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (cdf[mid] < u) lo = mid + 1; else hi = mid;
  }
  return lo;
}

// kTally: the flight ended; the photon waits to be tallied with the next refill
// batch (its position and direction do not change meanwhile)
enum { kDead = 0, kTally = 1, kFly = 2, kCollide = 3 };  // dead or tally pending: state <= kTally
// Statistics are counted per wave, not per lane: where every lane of the wave
// is active, a ballot of the lanes where an event happened is added to the
// wave's 64-bit counter in LDS, and the counters go to the job's when it is
// flushed.  (Ten per-lane counters, incremented in the branches, took 56 of the
// kernel's 121 VGPRs.)
enum { kStatHistories, kStatSteps, kStatInteractions, kStatPhoto, kStatCoherent, kStatCompton, kStatTp, kStatTs,
       kStatMissed, kStatCapped, kStats };
static_assert(kStats == kWaveStats, "one LDS counter per statistic");

__device__ inline unsigned popc(uint64_t m) { return (unsigned)__popcll(m); }

// Adds the lanes where `pred` holds to the wave's counter k.  Called where
// every lane of the wave is active; lane 0 adds for the wave.
__device__ inline void count_lanes(WaveTables& wt, int k, bool pred) {
  const uint64_t m = __ballot(pred);
  if (__lane_id() == 0 && m != 0) atomicAdd(&wt.stats[k], (unsigned long long)popc(m));
}

// Straight line from the current position to the detector plane x' = sdd - sod.
enum { kTallyMiss = 0, kTallyPrimary = 1, kTallyScatter = 2 };

// Counts the tallies of a section from each lane's tally code (-1: none).
// Misses are not counted here: every history ends once, tallied, missed,
// absorbed or capped, so the flush derives them.
__device__ inline void count_tallies(WaveTables& wt, int code) {
  const uint64_t mp = __ballot(code == kTallyPrimary), ms = __ballot(code == kTallyScatter);
  if (__lane_id() == 0 && (mp | ms) != 0) {
    atomicAdd(&wt.stats[kStatTp], (unsigned long long)popc(mp));
    atomicAdd(&wt.stats[kStatTs], (unsigned long long)popc(ms));
  }
}

template <class JT>
__device__ inline int tally_cell(const Photon& p, const JT& J, size_t& idx) {
  const float cx = p.cv, cy = p.sv;
  const float xq = p.px * cx + p.py * cy, yq = -p.px * cy + p.py * cx;
  const float ddx = p.dx * cx + p.dy * cy, ddy = -p.dx * cy + p.dy * cx;
  if (!(ddx > 0.f)) {
    return kTallyMiss;
  }
  const float tt = ((J.sdd - J.sod) - xq) * __builtin_amdgcn_rcpf(ddx);
  const float yh = fmaf(tt, ddy, yq), zh = fmaf(tt, p.dz, p.pz);
  const float ui = fmaf(J.us, yh, J.un0), vi = fmaf(J.vs, zh, J.vn0);
  if (!(ui >= 0.f && ui < (float)J.nu && vi >= 0.f && vi < (float)J.nv)) {
    return kTallyMiss;
  }
  int iu = (int)floorf(ui), iv = (int)floorf(vi);
  iu = iu > J.nu - 1 ? J.nu - 1 : iu;
  iv = iv > J.nv - 1 ? J.nv - 1 : iv;
  idx = ((size_t)p.view * J.nu + iu) * J.nv + iv;
  return p.nint == 0 ? kTallyPrimary : kTallyScatter;
}

// Adds a photon that ends its flight here to its image; its tally code.
template <class JT>
__device__ inline int tally(const Photon& p, const JT& J) {
  size_t idx = 0;
  const int code = tally_cell(p, J, idx);
  if (code == kTallyPrimary) unsafeAtomicAdd(J.primary + idx, 1.0);
  if (code == kTallyScatter) unsafeAtomicAdd(J.scatter + idx, 1.0);
  return code;
}

// Label set meaning "any label": the flight takes the global majorant.
constexpr uint32_t kAnyLabel = 16u;

// The largest mu among the labels of `set` (bit l: label l in 0..3;
// kAnyLabel: every label) at the photon's table row, from its mu registers.
__device__ inline float set_majorant(const Photon& p, const WaveTables& wt, uint32_t set) {
  float mm;
  if (set & kAnyLabel) {
    mm = wt.mumax[p.eb];
  } else {
    mm = 0.f;
    if (set & 1u) mm = fmaxf(mm, p.mu0);
    if (set & 2u) mm = fmaxf(mm, p.mu1);
    if (set & 4u) mm = fmaxf(mm, p.mu2);
    if (set & 8u) mm = fmaxf(mm, p.mu3);
  }
  return mm;
}

// Starts a flight from the current position (after a scatter; a birth forms
// its tile's rays the same way, once per tile and view); returns false if the
// photon leaves without entering the flight box, or meets nothing that
// attenuates (the caller tallies it).  The Woodcock majorant is the largest mu
// among the labels of `set`.  t_in: the distance moved to the box entry, 0 if
// the photon starts inside.
template <class JT>
__device__ inline bool start_flight(Photon& p, const JT& J, const WaveTables& wt, uint32_t set, float& t_in) {
  p.mu0 = wt.mu[0][p.eb];
  p.mu1 = wt.mu[1][p.eb];
  p.mu2 = wt.mu[2][p.eb];
  p.mu3 = wt.mu[3][p.eb];
  const float mm = set_majorant(p, wt, set);
  if (!(mm > 0.f)) return false;
  float t0, t1;
  if (!ray_box(p.px, p.py, p.pz, p.dx, p.dy, p.dz, J, t0, t1) || !(t1 > 0.f)) return false;
  t_in = 0.f;
  if (t0 > 0.f) {
    p.px = fmaf(t0, p.dx, p.px); p.py = fmaf(t0, p.dy, p.py); p.pz = fmaf(t0, p.dz, p.pz);
    t1 -= t0;
    t_in = t0;
  }
  p.t = 0.f;
  p.t1 = t1;
  p.mumax = mm;
  p.lscale = 0.69314718055994531f * rcp(mm);
  return true;
}

// Copies a job's tables into the wave's LDS slot.
// The host builds the CDF from non-negative weights, so it is non-decreasing
// and the search within a guide cell returns the row a search over all rows
// would.
template <class JT>
__device__ inline void load_wave_tables(WaveTables& wt, const JT& J, int lane) {
  for (int e = lane; e < kRows; e += 64) {
    wt.cdf[e] = J.spectrum_cdf ? J.spectrum_cdf[e] : 0.f;
    wt.mumax[e] = J.tables->mumax[e];
#pragma unroll
    for (int l = 0; l < 4; ++l) wt.mu[l][e] = J.tables->m[l][e].x;
  }
  if (J.spectrum_cdf) {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the CDF in LDS is complete
    __builtin_amdgcn_wave_barrier();
    for (int g = lane; g <= kGuide; g += 64)
      wt.guide[g] = (uint8_t)spectrum_row(wt.cdf, (float)g * (1.0f / kGuide), 1, kRows - 1);
  }
}

// Attenuation at a label: labels 0..3 from registers, others from the table.
template <class JT>
__device__ inline float mu_at(const Photon& p, int lab, const JT& J) {
  const bool odd = (lab & 1) != 0;
  const float lo = odd ? p.mu1 : p.mu0, hi = odd ? p.mu3 : p.mu2;
  float mu = (lab & 2) ? hi : lo;
  if (lab > 3) mu = J.tables->m[lab][p.eb].x;
  return mu;
}

// a * b + c with 24-bit a, b, at full rate (the compiler otherwise picks the
// quarter-rate 64-bit multiply-add when it cannot prove the operand widths)
__device__ inline uint32_t mad_u24(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}

// min(max(x, 0), hi) for hi >= 0 as one median-of-three (the compiler forms
// it only when hi is a constant)
__device__ inline int clamp_index(int x, int hi) {
  int r;
  asm("v_med3_i32 %0, %1, 0, %2" : "=v"(r) : "v"(x), "s"(hi));
  return r;
}

// Position at flight parameter t and the index of its voxel.
template <class JT>
__device__ inline uint32_t voxel_at(const Photon& p, float t, const JT& J, float& qx, float& qy, float& qz) {
  qx = fmaf(t, p.dx, p.px); qy = fmaf(t, p.dy, p.py); qz = fmaf(t, p.dz, p.pz);
  // voxel index = (q - b0) / v as one FMA; truncation equals floor wherever
  // the clamp to [0, n - 1] does not already decide it
  const int ix = clamp_index((int)fmaf(qx, J.inv_vx, J.ix0), J.nx - 1);
  const int iy = clamp_index((int)fmaf(qy, J.inv_vy, J.iy0), J.ny - 1);
  const int iz = clamp_index((int)fmaf(qz, J.inv_vz, J.iz0), J.nz - 1);
  // 32-bit index from two 24-bit multiply-adds: the host checks
  // nz * ny < 2^24, nx < 2^24 and nx * ny * nz < 2^32
  return mad_u24(mad_u24((uint32_t)iz, (uint32_t)J.ny, (uint32_t)iy), (uint32_t)J.nx, (uint32_t)ix);
}

// Label byte of a voxel, by a global-address-space load; the caller clamps
// labels past the table (min(label, kMaxLabels - 1)) so no table read leaves it.
template <class JT>
__device__ inline uint32_t label_raw(uint32_t i, const JT& J) {
  return ((const __attribute__((address_space(1))) uint8_t*)J.labels)[i];
}

// A parked branch runs once at least this many lanes wait for it (or nothing
// else can run).  Interactions wait for 32 lanes: each batch costs a whole
// Klein-Nishina rejection loop and a flight set-up, so fuller batches pay
// (16, 24, 32, 40 and 48 lanes took 71.6, 69.4, 69.0, 70.9 and 88.0 ms on the full
// workload at 1e7 photons per view, the collided lanes idling longer past 32; 152.0,
// 151.4, 150.8, 149.7 and 148.9 on the end-to-end scan at 5e6).  Refills of 8 and 24
// lanes took 69.4 and 70.9 ms, 151.3 and 149.4.
constexpr unsigned kInteractBatch = 32;
constexpr unsigned kRefillBatch = 16;

__global__ __launch_bounds__(256) void mc_transport_kernel(const McJob* __restrict__ jobs, int n_jobs,
                                                           uint64_t total_units, uint32_t chunk,
                                                           unsigned int* __restrict__ queue,
                                                           McCounters* __restrict__ counters, int slots) {
  int job = -1;
  const int q_first = (int)(blockIdx.x % kMcQueues);
  int q_own = q_first;   // the queue the wave draws from
  bool q_begun = false;  // the wave has had its first unit
  // the current unit (wave-uniform): tiles [unit_t0, unit_t0 + unit_nt), each over
  // photon cycles [unit_cyc0, unit_cyc_end); the next birth takes tile unit_t0 +
  // unit_g of cycle unit_cyc
  uint32_t unit_t0 = 0, unit_nt = 0, unit_g = 0, unit_cyc0 = 0, unit_cyc = 0, unit_cyc_end = 0;
  uint64_t unit_act = 0;  // the tile's lanes (pixels) whose photons may collide
  int unit_view = 0;
  long long pending = -1;
  bool exhausted = false;
  uint32_t buf_head = 0, buf_n = 0;  // the birth buffer's next photon and photons left (wave-uniform)
  int buf_view = 0;                  // the view of the buffered photons, and its cos and sin
  float buf_cv = 0.f, buf_sv = 0.f;
  uint32_t buf_id0 = 0;              // photon index of the buffer's slot 0 (the tile's corner pixel)

  int state = kDead;
  Photon p{};
  Stream rs{};
  const int lane = __lane_id();
  // The job descriptors do not change during the launch: read them through the
  // constant address space, so wave-uniform fields come in by scalar loads.
  const CJob* cjobs = (const CJob*)jobs;
  extern __shared__ WaveTables wave_tables[];  // one slot per wave of the block
  WaveTables& wt = wave_tables[threadIdx.x >> 6];
  if (lane < kStats) wt.stats[lane] = 0;
  // adds the wave's counters to the job's and clears them; called once all the
  // histories the wave began for the job have ended, so the misses and the
  // interactions follow from the other counts
  auto flush = [&](McCounters* dst) {
    if (__lane_id() == 0) {
      unsigned long long v[kStats];
#pragma unroll
      for (int k = 0; k < kStats; ++k) {
        v[k] = wt.stats[k];
        wt.stats[k] = 0;
      }
      v[kStatMissed] = v[kStatHistories] - v[kStatTp] - v[kStatTs] - v[kStatPhoto] - v[kStatCapped];
      v[kStatInteractions] = v[kStatPhoto] + v[kStatCoherent] + v[kStatCompton];
      atomicAdd(&dst->histories, v[kStatHistories]); atomicAdd(&dst->steps, v[kStatSteps]);
      atomicAdd(&dst->interactions, v[kStatInteractions]); atomicAdd(&dst->photo, v[kStatPhoto]);
      atomicAdd(&dst->coherent, v[kStatCoherent]); atomicAdd(&dst->compton, v[kStatCompton]);
      atomicAdd(&dst->tallied_primary, v[kStatTp]); atomicAdd(&dst->tallied_scatter, v[kStatTs]);
      atomicAdd(&dst->missed, v[kStatMissed]); atomicAdd(&dst->capped, v[kStatCapped]);
    }
  };

  for (;;) {
    // fields are read where they are used, by scalar loads
    CJob* Jp = cjobs + __builtin_amdgcn_readfirstlane(job < 0 ? 0 : job);
    uint64_t dead = __ballot(state <= kTally);
    const uint64_t fly = __ballot(state == kFly);
    const uint64_t coll = __ballot(state == kCollide);
    const uint64_t pend = __ballot(state == kTally);
    const bool all_dead = (fly | coll) == 0;

    // 1) secure a work unit when lanes are idle and the current one is spent
    if (dead != 0 && unit_g >= unit_nt) {
      if (pending < 0 && !exhausted) {
        // in round r = k / chunk, queue q hands out chunk r kMcQueues + (q + r) mod kMcQueues,
        // unit k mod chunk of it: the chunks of a round are dealt to the queues rotated by
        // one per round, so no queue keeps the same detector rows when kMcQueues chunks
        // span a whole number of detector sweeps.  Units increase with k, so a queue is
        // spent once it hands out a unit past the end.
        // A wave's first unit is the one of its rank among the queue's waves (the
        // counters start past those), so a launch of few units per wave hardly
        // touches the counters.  A wave that finds its queue spent marks it, and
        // moves to the next one not marked: without the marks every wave of a
        // launch ended by drawing once from each of the 24.
        for (;;) {
          unsigned int k = 0;
          if (!q_begun) {
            q_begun = true;
            k = (blockIdx.x / kMcQueues) * (blockDim.x >> 6) + (threadIdx.x >> 6);
          } else if (lane == 0) {
            k = atomicAdd(queue + q_own * kMcQueueStride, 1u);
          }
          k = (unsigned int)__builtin_amdgcn_readfirstlane((int)k);
          const uint32_t r = k / chunk;
          const uint64_t u = ((uint64_t)r * kMcQueues + (uint64_t)((q_own + r) % kMcQueues)) * chunk + (k - r * chunk);
          if (u < total_units) {
            pending = (long long)u;
            break;
          }
          unsigned int spent = 0;
          if (lane == 0) spent = atomicOr(queue + kMcSpentWord, 1u << q_own) | (1u << q_own);
          spent = (unsigned int)__builtin_amdgcn_readfirstlane((int)spent);
          if (spent == (1u << kMcQueues) - 1u) break;
          do {
            q_own = q_own + 1 == kMcQueues ? 0 : q_own + 1;
          } while ((spent >> q_own) & 1u);
        }
        if (pending < 0) exhausted = true;
      }
      if (pending >= 0) {
        const int pj = __builtin_amdgcn_readfirstlane(job_of_unit(cjobs, n_jobs, (uint64_t)pending));
        if (pj == job || (all_dead && buf_n == 0 && pend == 0)) {  // buffered and ended photons are of the current job
          const bool switched = pj != job;
          if (switched) {
            if (job >= 0) flush(counters + job * slots + blockIdx.x % slots);
            job = pj;
          }
          // units run views fastest, then cycle blocks, then tile groups: the units in
          // flight share a few detector tiles, hence a thin z-slab of the phantom that
          // stays in L2, and each unit's primary tallies stay on a few lines
          const uint64_t local = (uint64_t)pending - cjobs[pj].unit_begin;
          const uint32_t nvs = (uint32_t)cjobs[pj].n_views_sim;
          const uint32_t bi = (uint32_t)(local / nvs);
          const uint32_t vl = (uint32_t)(local - (uint64_t)bi * nvs);
          unit_view = __builtin_amdgcn_readfirstlane(cjobs[pj].view_begin + (int)vl);
          {
            const uint32_t ncb = cjobs[pj].cycle_blocks, grp = cjobs[pj].tile_group;
            const uint32_t tg = bi / ncb, cb = bi - tg * ncb;
            unit_t0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tg * grp));
            unit_nt = (uint32_t)__builtin_amdgcn_readfirstlane((int)min(grp, cjobs[pj].tiles - tg * grp));
            unit_g = 0;
            unit_cyc0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(cb * cjobs[pj].cycle_block));
            unit_cyc = unit_cyc0;
            unit_cyc_end = (uint32_t)__builtin_amdgcn_readfirstlane(
                (int)min(unit_cyc0 + cjobs[pj].cycle_block, cjobs[pj].cycles));
          }
          pending = -1;
          if (switched) {  // J is re-read for the new job at the top of the loop
            load_wave_tables(wt, cjobs[pj], lane);
            __builtin_amdgcn_wave_barrier();
            continue;
          }
        }
      }
    }
    // 1b) tallies of the flights that ended, batched with the refills (all run when
    //     nothing flies, so none is left when the wave stops or changes job)
    if (pend != 0 && (popc(dead) >= kRefillBatch || fly == 0)) {
      int code = -1;
      if (state == kTally) {
        code = tally(p, *Jp);
        state = kDead;
      }
      count_tallies(wt, code);
    }
    if (all_dead && unit_g >= unit_nt && pending < 0 && exhausted && buf_n == 0) break;

    // 2) refill dead lanes from the birth buffer, after filling it when it is empty
    if (dead != 0 && (buf_n != 0 || unit_g < unit_nt) && (popc(dead) >= kRefillBatch || fly == 0)) {
      if (buf_n == 0) {
        // one tile of the unit in one cycle, one photon per lane with every lane
        // active: lane l aims at the centre of pixel (u_, v_) of the tile
        // (CBCT_real325.cu:464-466), and is photon n = cycle * nu nv + v_ nu + u_ of
        // the view, whose pixel in aim order is n mod (nu nv)
        const uint32_t t = unit_t0 + unit_g;
        const uint32_t tv = t / (uint32_t)Jp->tiles_u, tu = t - tv * (uint32_t)Jp->tiles_u;
        const uint32_t u_ = tu * kTileU + (uint32_t)lane % kTileU, v_ = tv * kTileV + (uint32_t)lane / kTileU;
        const uint32_t npix = (uint32_t)(Jp->nu * Jp->nv);
        const uint32_t pix = v_ * (uint32_t)Jp->nu + u_;
        const uint64_t n64 = (uint64_t)unit_cyc * npix + pix;
        const uint32_t id = (uint32_t)n64;
        CU32* vcs = (CU32*)Jp->view_cs + 2 * unit_view;  // read-only during the launch: scalar loads
        const float cv = __uint_as_float(vcs[0]), sv = __uint_as_float(vcs[1]);
        const bool on_det = u_ < (uint32_t)Jp->nu && v_ < (uint32_t)Jp->nv;
        if (unit_cyc == unit_cyc0) {
          // the tile's rays in this view, one per lane: the first flight runs from the
          // source towards the pixel centre, its majorant comes from the labels the
          // line crosses, and it starts at the flight box (start_flight's clip)
          const uint32_t set =
              on_det && Jp->ray_set ? (uint32_t)Jp->ray_set[(size_t)(unit_view - Jp->view_begin) * npix + pix]
                                    : kAnyLabel;
          const float yp = ((float)u_ + 0.5f - Jp->un0) * Jp->u_step;
          const float zp = ((float)v_ + 0.5f - Jp->vn0) * Jp->v_step;
          const float in = rsqrtf(fmaf(zp, zp, fmaf(Jp->sdd, Jp->sdd, yp * yp)));
          // the fused products are spelled out, so the direction's rounding does not
          // depend on which product the compiler would fuse here
          const float dx = fmaf(Jp->sdd, cv, -(yp * sv)) * in;
          const float dy = fmaf(cv, yp, Jp->sdd * sv) * in;
          const float dz = zp * in;
          float t0, t1;
          const bool hit = ray_box(-Jp->sod * cv, -Jp->sod * sv, 0.f, dx, dy, dz, *Jp, t0, t1) && t1 > 0.f;
          float tin = 0.f;
          if (t0 > 0.f) {
            t1 -= t0;
            tin = t0;
          }
          wt.bb.d0[lane] = make_float4(dx, dy, dz, tin);
          wt.bb.t1[lane] = hit ? t1 : -1.f;
          wt.bb.set[lane] = (uint8_t)set;
          // A ray that misses the flight box, or crosses only labels that never
          // attenuate, sends every photon straight to the detector, whatever its
          // energy: all of the unit's photons on it are tallied here with one add
          // (sums of ones are exact).  On the full workload (a 15 cm phantom before a
          // 61 cm detector) these are three photons in four.
          const bool may = on_det && hit && (set & Jp->solid_set) != 0;
          unit_act = __ballot(may);
          const bool inert = on_det && !may;
          if (unit_act != __ballot(on_det)) {
            const bool short_ = unit_cyc_end == Jp->cycles &&
                                (uint64_t)(Jp->cycles - 1) * npix + pix >= Jp->photons_per_view;
            const uint32_t full = unit_cyc_end - unit_cyc0;
            int code = -1;
            if (inert) {
              Photon q;
              q.view = unit_view;
              q.cv = cv; q.sv = sv;
              q.dx = dx; q.dy = dy; q.dz = dz;
              q.px = -Jp->sod * cv; q.py = -Jp->sod * sv; q.pz = 0.f;
              q.nint = 0;
              size_t idx = 0;
              code = tally_cell(q, *Jp, idx);
              const uint32_t n = full - (short_ ? 1u : 0u);
              if (code == kTallyPrimary && n != 0) unsafeAtomicAdd(Jp->primary + idx, (double)n);
            }
            const uint64_t mi = __ballot(inert), mp = __ballot(code == kTallyPrimary), ms = __ballot(short_);
            if (lane == 0) {
              atomicAdd(&wt.stats[kStatHistories], (unsigned long long)full * popc(mi) - popc(mi & ms));
              atomicAdd(&wt.stats[kStatTp], (unsigned long long)full * popc(mp) - popc(mp & ms));
            }
          }
        }
        bool born = false;
        int bcode = -1;  // tally code of a photon that misses the flight box
        const bool valid = ((unit_act >> lane) & 1u) != 0 && n64 < Jp->photons_per_view;
        if (valid) {
          Photon q;
          q.view = unit_view;
          q.cv = cv;
          q.sv = sv;
          {
            const float4 d0 = wt.bb.d0[lane];
            q.dx = d0.x; q.dy = d0.y; q.dz = d0.z;
          }
          q.px = -Jp->sod * cv; q.py = -Jp->sod * sv; q.pz = 0.f;
          float e = Jp->e_kev;
          if (Jp->spectrum_cdf) {
            Stream bs{};
            bs.photon = id; bs.view = (uint32_t)unit_view;
            const float u = next_u01(bs, Jp->job_id, Jp->key0, Jp->key1);
            const int g = (int)(u * (float)kGuide);  // exact: u < 1 and kGuide is a power of 2
            e = (float)spectrum_row(wt.cdf, u, wt.guide[g], wt.guide[g + 1]);
          }
          q.e = e;
          q.eb = ebin_of(e);
          q.nint = 0;
          // start_flight's tests: something attenuates, and the line meets the box
          q.mu0 = wt.mu[0][q.eb];
          q.mu1 = wt.mu[1][q.eb];
          q.mu2 = wt.mu[2][q.eb];
          q.mu3 = wt.mu[3][q.eb];
          born = set_majorant(q, wt, wt.bb.set[lane]) > 0.f && wt.bb.t1[lane] >= 0.f;
          if (born) {
            wt.bb.eb[lane] = (uint8_t)q.eb;
          } else {
            bcode = tally(q, *Jp);
          }
        }
        count_lanes(wt, kStatHistories, valid);
        count_tallies(wt, bcode);
        const uint64_t bm = __ballot(born);
        if (born)
          wt.bb.slot[__builtin_amdgcn_mbcnt_hi((uint32_t)(bm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bm, 0u))] =
              (uint8_t)lane;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // the buffer in LDS is complete
        __builtin_amdgcn_wave_barrier();
        buf_n = (uint32_t)popc(bm);
        buf_head = 0;
        buf_view = unit_view;
        buf_cv = cv;
        buf_sv = sv;
        buf_id0 = (uint32_t)((uint64_t)unit_cyc * npix + tv * kTileV * (uint32_t)Jp->nu + tu * kTileU);
        if (unit_act == 0 || ++unit_cyc == unit_cyc_end) {  // the tile is done
          ++unit_g;
          unit_cyc = unit_cyc0;
        }
      }
      const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(dead >> 32),
                                                      __builtin_amdgcn_mbcnt_lo((uint32_t)dead, 0u));
      if (state == kDead && rank < buf_n) {
        const int s = wt.bb.slot[buf_head + rank];
        // as the birth formed them (start_flight's box clip, majorant and scale)
        const float4 d0 = wt.bb.d0[s];
        p.dx = d0.x; p.dy = d0.y; p.dz = d0.z;
        const float tin = d0.w;
        p.px = fmaf(tin, p.dx, -Jp->sod * buf_cv);
        p.py = fmaf(tin, p.dy, -Jp->sod * buf_sv);
        p.pz = fmaf(tin, p.dz, 0.f);
        p.eb = wt.bb.eb[s];
        p.e = Jp->spectrum_cdf ? (float)p.eb : Jp->e_kev;  // a spectrum row is its energy in keV
        p.t = 0.f;
        p.t1 = wt.bb.t1[s];
        p.mu0 = wt.mu[0][p.eb];
        p.mu1 = wt.mu[1][p.eb];
        p.mu2 = wt.mu[2][p.eb];
        p.mu3 = wt.mu[3][p.eb];
        p.mumax = set_majorant(p, wt, wt.bb.set[s]);
        p.lscale = 0.69314718055994531f * rcp(p.mumax);
        p.nint = 0;
        p.view = buf_view;
        p.cv = buf_cv;
        p.sv = buf_sv;
        // the spectrum draw took block 0 of the photon's stream; flights take whole blocks
        rs.ctr = Jp->spectrum_cdf ? 1u : 0u;
        rs.photon = buf_id0 + (uint32_t)(s / kTileU) * (uint32_t)Jp->nu + (uint32_t)(s % kTileU);
        rs.view = (uint32_t)buf_view;
        rs.left = 0;
        state = kFly;
      }
      const uint32_t took = min((uint32_t)popc(dead), buf_n);
      buf_head += took;
      buf_n -= took;
    }
    // 3) interactions of the parked colliding lanes
    if (coll != 0 && (popc(coll) >= kInteractBatch || fly == 0)) {
      const bool cap = state == kCollide && p.nint >= Jp->max_int;
      count_lanes(wt, kStatCapped, cap);
      if (cap) state = kDead;
      int ev = 0;      // 1 photoelectric, 2 coherent, 3 Compton
      if (state == kCollide) {
        const float4 m = Jp->tables->m[p.lab][p.eb];
        rs.left = 0;  // interactions start on a fresh block
        const float u3 = next_u01(rs, Jp->job_id, Jp->key0, Jp->key1);
        asm volatile("" ::"v"(m.y), "v"(m.z));  // both cutoffs loaded and waited for together
        const bool photo = u3 <= m.y, coh = u3 <= m.z;
        if (photo) {
          ev = 1;
          state = kDead;
        } else {
          if (coh) {
            ev = 2;
            if (Jp->coherent) {
              const float cth = thomson_mu(next_u01(rs, Jp->job_id, Jp->key0, Jp->key1));
              const float w = next_u01(rs, Jp->job_id, Jp->key0, Jp->key1);  // azimuth / 2 pi
              rotate_dir(p.dx, p.dy, p.dz, cth, w);
            }
          } else {
            ev = 3;
            const float lam = 511.0f * rcp(p.e);
            const float ro = kahn(lam, rs, Jp->job_id, Jp->key0, Jp->key1);
            const float lamd = ro * lam;
            float cth = 1.0f - (lamd - lam);
            cth = cth < -1.f ? -1.f : cth;
            p.e = 511.0f * rcp(lamd);
            p.eb = ebin_of(p.e);
            const float w = next_u01(rs, Jp->job_id, Jp->key0, Jp->key1);  // azimuth / 2 pi
            rotate_dir(p.dx, p.dy, p.dz, cth, w);
          }
          p.nint += 1;
          float tin_;
          if (start_flight(p, *Jp, wt, kAnyLabel, tin_)) {
            state = kFly;
          } else {
            state = kTally;
          }
        }
      }
      count_lanes(wt, kStatPhoto, ev == 1);
      count_lanes(wt, kStatCoherent, ev == 2);
      count_lanes(wt, kStatCompton, ev == 3);
    }

    // 4) two Woodcock steps for every flying lane from one Philox block
    //    (distance, accept, distance, accept); both label loads are issued
    //    before either is used, and a flight ending on the first step leaves
    //    the block's other two uniforms unused.
    count_lanes(wt, kStatSteps, state == kFly);
    bool two = false;   // took the second step of the pair
    if (state == kFly) {
      uint32_t c0 = rs.ctr, c1 = rs.photon, c2 = rs.view, c3 = Jp->job_id;
      philox10(c0, c1, c2, c3, Jp->key0, Jp->key1);
      rs.ctr += 1;
      rs.left = 0;
      // u >= 2^-25, so the hardware log2 needs no denormal handling
      const float ta = fmaf(-__builtin_amdgcn_logf(u01(c0)), p.lscale, p.t);
      const float tb = fmaf(-__builtin_amdgcn_logf(u01(c2)), p.lscale, ta);
      float ax, ay, az, bx, by, bz;
      const uint32_t va = voxel_at(p, ta, *Jp, ax, ay, az);
      const uint32_t vb = voxel_at(p, tb, *Jp, bx, by, bz);
      // a step that leaves the flight box (most first flights end on their first
      // step) reads no label: its load would only add traffic to the line misses.
      // Both loads are issued before either value is used (the empty asm keeps
      // the clamps, and so the waits, after both).
      uint32_t ra = 0, rb = 0;
      if (ta < p.t1) ra = label_raw(va, *Jp);
      if (tb < p.t1) rb = label_raw(vb, *Jp);
      asm volatile("" : "+v"(ra), "+v"(rb));
      const int la = min((int)ra, kMaxLabels - 1), lb = min((int)rb, kMaxLabels - 1);
      const float mua = mu_at(p, la, *Jp), mub = mu_at(p, lb, *Jp);
      // Both attenuations are consumed here on every path (an empty asm taking
      // them as inputs): a table load for a label above 3 left pending on the
      // paths that end the flight made the compiler wait for every memory
      // operation, tally atomics included, at the start of the next step.
      asm volatile("" ::"v"(mua), "v"(mub));
      const bool real_a = u01(c1) * p.mumax < mua, real_b = u01(c3) * p.mumax < mub;
      if (ta >= p.t1) {
        state = kTally;
      } else if (real_a) {  // real collision: park until the wave runs interactions
        p.px = ax; p.py = ay; p.pz = az;
        p.lab = la;
        state = kCollide;
      } else {
        two = true;
        if (tb >= p.t1) {
          state = kTally;
        } else if (real_b) {
          p.px = bx; p.py = by; p.pz = bz;
          p.lab = lb;
          state = kCollide;
        } else {
          p.t = tb;
        }
      }
    }
    count_lanes(wt, kStatSteps, two);
  }
  if (job >= 0) flush(counters + job * slots + blockIdx.x % slots);
}

// --------------------------------------------- first-flight label sets
// (xadd, xsub and xmul are never fused into FMAs, so the label sets follow
// the oracle's operations bit for bit.)

__device__ inline uint32_t label_bit(int lab) { return lab < 4 ? 1u << lab : kAnyLabel; }

// The label sets of the bytes of w.
__device__ inline uint32_t label_bits(uint32_t w) {
  return label_bit((int)(w & 255u)) | label_bit((int)((w >> 8) & 255u)) | label_bit((int)((w >> 16) & 255u)) |
         label_bit((int)(w >> 24));
}

__device__ inline uint32_t load_u32(const uint8_t* p) {  // (any alignment)
  uint32_t w;
  __builtin_memcpy(&w, p, 4);
  return w;
}

// One thread per brick: the labels of the brick's voxels and of their
// neighbours one voxel outside it, so a sample point rounded across a brick
// face into a voxel of the next brick is still covered.  Bricks of 4^3 read
// their rows of up to 8 bytes as two words, the second overlapping the first,
// and look at the labels only once the words have differed (a phantom is mostly
// uniform): byte by byte, 216 loads a brick took 95 us at 325^3.
__device__ inline void brick_set(const McPrep& P, long i) {
  const int nx = P.nx, ny = P.ny, nz = P.nz, b = P.brick, nb0 = P.ray.nb[0], nb1 = P.ray.nb[1];
  const int bx = (int)(i % nb0), by = (int)((i / nb0) % nb1), bz = (int)(i / ((long)nb0 * nb1));
  const int x0 = max(bx * b - 1, 0), x1 = min(bx * b + b, nx - 1);
  const int y0 = max(by * b - 1, 0), y1 = min(by * b + b, ny - 1);
  const int z0 = max(bz * b - 1, 0), z1 = min(bz * b + b, nz - 1);
  uint32_t m = 0;
  if (x1 - x0 < 3 || x1 - x0 > 7) {
    for (int z = z0; z <= z1; ++z)
      for (int y = y0; y <= y1; ++y) {
        const uint8_t* row = P.labels + ((size_t)z * ny + y) * nx;
        int x = x0;
        for (; x + 3 <= x1; x += 4) m |= label_bits(load_u32(row + x));
        for (; x <= x1; ++x) m |= label_bit(row[x]);
      }
  } else {  // rows of two words, six rows (the last repeated past y1) in flight
    uint32_t any = 0, all = ~0u;
    for (int z = z0; z <= z1; ++z)
      for (int y = y0; y <= y1; y += 6) {
        uint32_t w[12];
#pragma unroll
        for (int r = 0; r < 6; ++r) {
          const uint8_t* row = P.labels + ((size_t)z * ny + min(y + r, y1)) * nx;
          w[2 * r] = load_u32(row + x0);
          w[2 * r + 1] = load_u32(row + x1 - 3);
        }
#pragma unroll
        for (int r = 0; r < 12; ++r) {
          any |= w[r];
          all &= w[r];
        }
        if (any != all) {  // not uniform so far: these words' own labels
#pragma unroll
          for (int r = 0; r < 12; ++r) m |= label_bits(w[r]);
        }
      }
    // the words before the first difference equal the first word
    m |= label_bits(load_u32(P.labels + ((size_t)z0 * ny + y0) * nx + x0));
  }
  P.bricks[i] = (uint8_t)m;
}

// Bounding box of the voxels whose label attenuates at some energy (labels are
// clamped as in transport), over 16-byte chunks of the label map taken as one
// array.  A chunk within a row costs two divisions; the box takes six atomics
// per block.  One block per slice reading bytes row after row took 232 us at
// 325^3.
__device__ inline void support_box(McPrep& P, uint32_t block) {
  __shared__ int red[4][6];
  const uint32_t n = (uint32_t)P.nx * (uint32_t)P.ny * (uint32_t)P.nz;  // (below 2^32)
  const uint32_t nx = (uint32_t)P.nx, ny = (uint32_t)P.ny, solid = P.solid;
  const uint32_t lead = (uint32_t)((uintptr_t)P.labels & 15u);  // bytes of the first chunk before the map
  const uint64_t chunks = ((uint64_t)lead + n + 15u) / 16u;
  int lo[3] = {INT_MAX, INT_MAX, INT_MAX}, hi[3] = {-1, -1, -1};
  auto add = [&](uint32_t first, uint32_t last) {  // voxels first .. last of one row
    const uint32_t r = first / nx, z = r / ny, y = r - z * ny;
    lo[0] = min(lo[0], (int)(first - r * nx)); hi[0] = max(hi[0], (int)(last - r * nx));
    lo[1] = min(lo[1], (int)y); hi[1] = max(hi[1], (int)y);
    lo[2] = min(lo[2], (int)z); hi[2] = max(hi[2], (int)z);
  };
  for (uint64_t c = (uint64_t)block * 256 + threadIdx.x; c < chunks; c += (uint64_t)P.box_blocks * 256) {
    const int64_t at = (int64_t)c * 16 - lead;  // voxel of the chunk's first byte
    uint32_t mask = 0;  // bit i: byte i attenuates
    if (at >= 0 && at + 16 <= (int64_t)n) {
      const uint4 w = *(const uint4*)(P.labels + at);
      if ((w.x | w.y | w.z | w.w) == 0u && !(solid & 1u)) continue;
      const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
      for (int i = 0; i < 16; ++i)
        mask |= ((solid >> min((ws[i / 4] >> (8 * (i % 4))) & 255u, (uint32_t)kMaxLabels - 1u)) & 1u) << i;
    } else {
      for (int i = 0; i < 16; ++i)
        if (at + i >= 0 && at + i < (int64_t)n)
          mask |= ((solid >> min((uint32_t)P.labels[at + i], (uint32_t)kMaxLabels - 1u)) & 1u) << i;
    }
    if (mask == 0) continue;
    const uint32_t first = (uint32_t)(at + __ffs((int)mask) - 1), last = (uint32_t)(at + 31 - __clz((int)mask));
    if (first / nx == last / nx) {
      add(first, last);
    } else {
      for (int i = 0; i < 16; ++i)
        if ((mask >> i) & 1u) add((uint32_t)(at + i), (uint32_t)(at + i));
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
    for (int a = 0; a < 3; ++a) {
      lo[a] = min(lo[a], __shfl_xor(lo[a], o, 64));
      hi[a] = max(hi[a], __shfl_xor(hi[a], o, 64));
    }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0)
    for (int a = 0; a < 3; ++a) {
      red[w][a] = lo[a];
      red[w][3 + a] = hi[a];
    }
  __syncthreads();
  if (threadIdx.x < 6) {
    const int a = threadIdx.x;
    int v = red[0][a];
    for (int i = 1; i < 4; ++i) v = a < 3 ? min(v, red[i][a]) : max(v, red[i][a]);
    if (a < 3 && v != INT_MAX) atomicMin(&P.box[a], v);
    if (a >= 3 && v >= 0) atomicMax(&P.box[a], v);
  }
}

// The job whose blocks of a shared grid include block b (begin: its first).
template <class F>
__device__ inline int job_of_block(int n_jobs, uint32_t b, F begin) {
  int lo = 0, hi = n_jobs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (begin(mid) <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Flight boxes and brick sets of all jobs in one launch: they read the same
// labels and do not depend on each other.  (A launch each per job, with the box
// read back by the host in between, took 4.3 of 10 ms of 24 uneven jobs.)
__global__ __launch_bounds__(256) void mc_prep_kernel(McPrep* __restrict__ preps, int n_jobs, uint32_t block0) {
  const uint32_t block = block0 + blockIdx.x;
  const int j = job_of_block(n_jobs, block, [&](int i) { return preps[i].prep_begin; });
  McPrep& P = preps[j];
  const uint32_t b = block - P.prep_begin;
  if (b < P.box_blocks) {
    support_box(P, b);
    return;
  }
  const long i = (long)(b - P.box_blocks) * 256 + threadIdx.x;
  if (i < (long)P.ray.nb[0] * P.ray.nb[1] * P.ray.nb[2]) brick_set(P, i);
}

// The flight box along axis a: [lo, hi) of the attenuating voxels, or of the
// phantom when nothing attenuates.
__device__ inline void flight_box(const McPrep& P, int a, double& lo, double& hi) {
  const double v = P.vox[a];
  const int dims[3] = {P.nx, P.ny, P.nz};
  const bool any = P.box[3] >= 0;
  lo = any ? xadd(P.ray.org[a], xmul((double)P.box[a], v)) : P.ray.org[a];
  hi = xadd(P.ray.org[a], xmul((double)(any ? P.box[3 + a] + 1 : dims[a]), v));
}

// Flights are clipped to that box: outside it mu is 0, so no history changes,
// and no Woodcock steps are spent crossing the empty margin of the phantom.
__device__ inline void set_job_box(const McPrep& P, McJob& J) {
  if (P.box[3] < 0) return;
  double lo[3], hi[3];
  for (int a = 0; a < 3; ++a) flight_box(P, a, lo[a], hi[a]);
  J.bx0 = (float)lo[0]; J.bx1 = (float)hi[0];
  J.by0 = (float)lo[1]; J.by1 = (float)hi[1];
  J.bz0 = (float)lo[2]; J.bz1 = (float)hi[2];
}

__global__ void mc_boxes_kernel(const McPrep* __restrict__ preps, McJob* __restrict__ jobs, int n_jobs) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n_jobs) set_job_box(preps[i], jobs[i]);
}

// One thread per (view, pixel): the union of the brick sets along the segment
// source -> pixel centre inside the flight box, by index-stepping traversal of
// the brick grid (every crossing recomputed from its plane index), or
// kAnyLabel if the segment misses the box.  A block's rays share a view, hence
// the source: with PLANES the distances of all brick planes from it are formed
// once per block in LDS, which leaves one FP64 multiply per axis and step (the
// walk of ~60 bricks a ray issues FP64 and integer VALU all the time: 5.2 ms at
// 325^3 / 512^2 / 360 views with the planes formed at every step, 3.2 ms so).
template <bool PLANES>
__global__ __launch_bounds__(kRayBlock) void ray_sets_kernel(const McPrep* __restrict__ preps, McJob* __restrict__ jobs,
                                                             int n_jobs, uint32_t block0) {
  extern __shared__ double planes[];
  const uint32_t block = block0 + blockIdx.x;
  const int j = job_of_block(n_jobs, block, [&](int i) { return preps[i].ray_begin; });
  const McPrep& P = preps[j];
  const RayGrid& R = P.ray;
  const int view_begin = jobs[j].view_begin;
  const int npix = R.nu * R.nv, per_view = (npix + kRayBlock - 1) / kRayBlock;
  const uint32_t b = block - P.ray_begin;
  const int kk = (int)(b / (uint32_t)per_view), pix = (int)(b - (uint32_t)kk * (uint32_t)per_view) * kRayBlock + (int)threadIdx.x;
  if (b == 0 && threadIdx.x == 0) set_job_box(P, jobs[j]);
  const double cb = P.cs64[2 * (view_begin + kk)], sb = P.cs64[2 * (view_begin + kk) + 1];
  const double S[3] = {xmul(-R.sod, cb), xmul(-R.sod, sb), 0.0};
  const int nb0 = R.nb[0], nb1 = R.nb[1], nb2 = R.nb[2];
  if (PLANES) {
    for (int i = threadIdx.x; i < nb0 + nb1 + nb2 + 3; i += kRayBlock) {
      const int a = i <= nb0 ? 0 : (i <= nb0 + 1 + nb1 ? 1 : 2);
      const int p = a == 0 ? i : (a == 1 ? i - nb0 - 1 : i - nb0 - nb1 - 2);
      const double org = a == 0 ? R.org[0] : (a == 1 ? R.org[1] : R.org[2]);
      const double bw = a == 0 ? R.bw[0] : (a == 1 ? R.bw[1] : R.bw[2]);
      planes[i] = xsub(xadd(org, xmul((double)p, bw)), a == 0 ? S[0] : (a == 1 ? S[1] : S[2]));
    }
    __syncthreads();
  }
  if (pix >= npix) return;
  uint8_t* out = P.sets + (size_t)kk * npix + pix;
  const int iv = pix / R.nu, iu = pix - iv * R.nu;
  const double yp = xmul(xsub(xadd((double)iu, 0.5), R.un0), R.u_step);
  const double zp = xmul(xsub(xadd((double)iv, 0.5), R.vn0), R.v_step);
  const double T[3] = {xsub(xmul(R.xd, cb), xmul(yp, sb)), xadd(xmul(R.xd, sb), xmul(yp, cb)), zp};
  double d[3], inv[3];
  double lo = 0.0, hi = 1.0;
  bool miss = false;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    double c0, c1;
    flight_box(P, a, c0, c1);
    d[a] = xsub(T[a], S[a]);
    if (d[a] != 0.0) {
      inv[a] = 1.0 / d[a];
      const double ta = xmul(xsub(c0, S[a]), inv[a]), tb = xmul(xsub(c1, S[a]), inv[a]);
      const double tl = ta < tb ? ta : tb, th = ta < tb ? tb : ta;
      if (tl > lo) lo = tl;
      if (th < hi) hi = th;
    } else {
      inv[a] = 0.0;
      if (S[a] < c0 || S[a] >= c1) miss = true;
    }
  }
  if (miss || !(hi > lo)) {
    *out = (uint8_t)kAnyLabel;
    return;
  }
  const double span = xsub(hi, lo);
  const double half = xmul(span, 0.5);
  const double tm = xadd(lo, half < 1e-9 ? half : 1e-9);  // a point just inside
  int idx[3];
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const double q = xadd(S[a], xmul(tm, d[a]));
    const int i = (int)floor(xsub(q, R.org[a]) / R.bw[a]);
    idx[a] = i < 0 ? 0 : (i > R.nb[a] - 1 ? R.nb[a] - 1 : i);
  }
  // per axis: index of the next plane, and the crossings left before the grid's end
  const int s0 = d[0] > 0.0 ? 1 : -1, s1 = d[1] > 0.0 ? 1 : -1, s2 = d[2] > 0.0 ? 1 : -1;
  int p0 = idx[0] + (s0 > 0), p1 = idx[1] + (s1 > 0), p2 = idx[2] + (s2 > 0);
  int left0 = s0 > 0 ? nb0 - 1 - idx[0] : idx[0], left1 = s1 > 0 ? nb1 - 1 - idx[1] : idx[1],
      left2 = s2 > 0 ? nb2 - 1 - idx[2] : idx[2];
  uint32_t at = ((uint32_t)idx[2] * (uint32_t)nb1 + (uint32_t)idx[1]) * (uint32_t)nb0 + (uint32_t)idx[0];
  auto crossing = [&](int a, int p) {
    if (d[a] == 0.0) return (double)INFINITY;
    const int first = a == 0 ? 0 : (a == 1 ? nb0 + 1 : nb0 + nb1 + 2);
    return xmul(PLANES ? planes[first + p] : xsub(xadd(R.org[a], xmul((double)p, R.bw[a])), S[a]), inv[a]);
  };
  uint32_t m = 0, cur = P.bricks[at];  // (a brick's set is waited for a step later)
  for (;;) {
    const double t0 = crossing(0, p0), t1 = crossing(1, p1), t2 = crossing(2, p2);
    const bool c1 = t1 < t0;
    const double t01 = c1 ? t1 : t0;
    const bool c2 = t2 < t01;
    if (!((c2 ? t2 : t01) < hi)) break;
    const bool y = c1 && !c2, x = !c1 && !c2;
    if ((c2 ? left2 : (c1 ? left1 : left0)) == 0) break;
    p0 += x ? s0 : 0;
    p1 += y ? s1 : 0;
    p2 += c2 ? s2 : 0;
    left0 -= x;
    left1 -= y;
    left2 -= c2;
    at += (uint32_t)(c2 ? s2 * nb0 * nb1 : (c1 ? s1 * nb0 : s0));
    const uint32_t next = P.bricks[at];
    m |= cur;
    cur = next;
  }
  *out = (uint8_t)(m | cur);
}

hipError_t launch_mc_prep(McPrep* preps, int n_jobs, uint32_t prep_blocks, hipStream_t s) {
  if (n_jobs < 1 || prep_blocks == 0) return hipErrorInvalidValue;
  for (uint64_t b = 0; b < prep_blocks; b += max_blocks(256))  // the jobs' blocks together may pass a launch's limit
    hipLaunchKernelGGL(mc_prep_kernel, dim3((unsigned)std::min(max_blocks(256), prep_blocks - b)), dim3(256), 0, s,
                       preps, n_jobs, (uint32_t)b);
  return hipGetLastError();
}

hipError_t launch_ray_sets(const McPrep* preps, McJob* jobs, int n_jobs, uint32_t ray_blocks, uint64_t max_planes,
                           hipStream_t s) {
  if (n_jobs < 1 || ray_blocks == 0) return hipErrorInvalidValue;
  for (uint64_t b = 0; b < ray_blocks; b += max_blocks(kRayBlock)) {
    const dim3 grid((unsigned)std::min(max_blocks(kRayBlock), ray_blocks - b));
    // the planes of grids up to 4096 bricks along the axes together fit in 32 KB of LDS
    if (max_planes <= 4096)
      hipLaunchKernelGGL(ray_sets_kernel<true>, grid, dim3(kRayBlock), sizeof(double) * max_planes, s, preps, jobs,
                         n_jobs, (uint32_t)b);
    else
      hipLaunchKernelGGL(ray_sets_kernel<false>, grid, dim3(kRayBlock), 0, s, preps, jobs, n_jobs, (uint32_t)b);
  }
  return hipGetLastError();
}

hipError_t launch_mc_boxes(const McPrep* preps, McJob* jobs, int n_jobs, hipStream_t s) {
  hipLaunchKernelGGL(mc_boxes_kernel, dim3((n_jobs + 63) / 64), dim3(64), 0, s, preps, jobs, n_jobs);
  return hipGetLastError();
}

__global__ void mc_reset_kernel(unsigned int* queue, McCounters* counters, int n_counters, int waves_per_block,
                                int grid) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < kMcQueues) queue[i * kMcQueueStride] = mc_queue_start(i, waves_per_block, grid);
  if (i == 0) queue[kMcSpentWord] = 0u;
  if (i < n_counters) counters[i] = McCounters{};
}

hipError_t launch_mc_reset(unsigned int* queue, McCounters* counters, int n_counters, int block, int grid,
                           hipStream_t s) {
  const int n = std::max(n_counters, (int)kMcQueues);
  hipLaunchKernelGGL(mc_reset_kernel, dim3((n + 255) / 256), dim3(256), 0, s, queue, counters, n_counters, block / 64,
                     grid);
  return hipGetLastError();
}

hipError_t launch_mc_transport(const McJob* jobs_dev, int n_jobs, uint64_t total_units, uint32_t chunk,
                               unsigned int* queue, McCounters* counters, int slots, int block, int grid,
                               hipStream_t s) {
  if (block % 64 || block > 256 || block <= 0 || grid <= 0 || chunk == 0 || slots < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(mc_transport_kernel, dim3(grid), dim3(block), sizeof(WaveTables) * (block / 64), s, jobs_dev,
                     n_jobs, total_units, chunk, queue, counters, slots);
  return hipGetLastError();
}

// ------------------------------------------------- exact primary (Siddon)
// One thread per (view, pixel): per-label path lengths along the source ->
// pixel-centre ray by index-stepping traversal (each crossing recomputed from
// its plane index, no running sums), kept in LDS, then combined with the
// attenuation of each spectral bin.  This is a deterministic integral, not MC
// tracking, and it runs in FP64 end to end: in FP32 the ray set-up from a
// source tens of cm away moves grazing rays by ~1e-6 cm, which changes short
// chords by ~1e-4 relative.
//
// What bounds it is the instructions of a step (about 30, and a label gather) on
// the rays that meet the phantom, so a step is kept short: the distances of all
// voxel planes from the source, which a block's rays share, are formed once per
// block in LDS (PLANES: grids of up to 4096 planes), a crossing is that times the
// ray's reciprocal, the traversal stays in the box of the attenuating voxels, and
// a label's length is added up only where the label changes.  A ray that meets no
// attenuating voxel skips the spectrum.  90 views of 512^2 of the 325^3 phantom at
// 120 kVp took 31.8 ms with three FP64 divisions, a read-add-write in LDS and an
// array access per step.
constexpr int kPrimU = 16, kPrimV = 16;  // pixels of a block: near rays share label lines, more so along u

template <bool PLANES>
__global__ __launch_bounds__(kPrimU * kPrimV) void primary_exact_kernel(PrimaryGeom P, const McPrep* __restrict__ prep,
                                                                        const double* __restrict__ cs64,
                                                                        const uint8_t* __restrict__ labels,
                                                                        const double* __restrict__ bins, int n_bins,
                                                                        int n_labels, double weight,
                                                                        float* __restrict__ out) {
  extern __shared__ double lds[];
  constexpr int kBlock = kPrimU * kPrimV;
  double* const lens = lds;                         // [n_labels][kBlock]
  double* const planes = lds + n_labels * kBlock;   // nx + ny + nz + 3
  const int tid = threadIdx.x;
  const int tiles_u = (P.nu + kPrimU - 1) / kPrimU, tiles_v = (P.nv + kPrimV - 1) / kPrimV;
  // Block b runs on XCD b mod 8, which takes the tile rows x, x + 8, ... of the
  // detector, each over all views: a row's rays share a thin slab of the phantom
  // that stays in its L2, and the rows that meet the phantom are spread evenly.
  const uint32_t xcd = blockIdx.x % 8u, j = blockIdx.x / 8u, row_blocks = (uint32_t)tiles_u * (uint32_t)P.n_views;
  const uint32_t row = j / row_blocks * 8u + xcd, jr = j % row_blocks;
  if (row >= (uint32_t)tiles_v) return;  // (the whole block)
  const int k = (int)(jr / (uint32_t)tiles_u), tu = (int)(jr % (uint32_t)tiles_u);
  const int iu = tu * kPrimU + tid % kPrimU, iv = (int)row * kPrimV + tid / kPrimU;
  const double cb = cs64[2 * k], sb = cs64[2 * k + 1];
  const double p0[3] = {-P.sod * cb, -P.sod * sb, 0.0};
  const int nx = P.n[0], ny = P.n[1], nz = P.n[2];
  for (int l = 0; l < n_labels; ++l) lens[l * kBlock + tid] = 0.0;
  if (PLANES) {
    for (int i = tid; i < nx + ny + nz + 3; i += kBlock) {
      const int a = i <= nx ? 0 : (i <= nx + 1 + ny ? 1 : 2);
      const int p = a == 0 ? i : (a == 1 ? i - nx - 1 : i - nx - ny - 2);
      planes[i] = (a == 0 ? P.b0[0] : (a == 1 ? P.b0[1] : P.b0[2])) + p * (a == 0 ? P.vox[0] : (a == 1 ? P.vox[1] : P.vox[2])) -
                  (a == 0 ? p0[0] : (a == 1 ? p0[1] : p0[2]));
    }
    __syncthreads();
  }
  if (iu >= P.nu || iv >= P.nv) return;
  const double yp = ((double)iu + 0.5 - P.un0) * P.u_step;
  const double zp = ((double)iv + 0.5 - P.vn0) * P.v_step;
  const double xd = P.sdd - P.sod;
  double d[3] = {xd * cb - yp * sb - p0[0], xd * sb + yp * cb - p0[1], zp};
  const double L = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
  double inv[3];
  double t0 = -INFINITY, t1 = INFINITY;
  bool hit = prep->box[3] >= 0;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    d[a] /= L;
    inv[a] = 1.0 / d[a];
    double c0, c1;
    flight_box(*prep, a, c0, c1);
    if (d[a] != 0.0) {
      const double ta = (c0 - p0[a]) * inv[a], tb = (c1 - p0[a]) * inv[a];
      t0 = fmax(t0, fmin(ta, tb));
      t1 = fmin(t1, fmax(ta, tb));
    } else if (p0[a] < c0 || p0[a] >= c1) {
      hit = false;
    }
  }
  t0 = fmax(t0, 0.0);
  t1 = fmin(t1, L);
  bool any = false;  // some length of a label that may attenuate
  if (hit && t1 > t0) {
    int idx[3];
    const double tm = t0 + fmin(0.5 * (t1 - t0), 1e-9);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int i = (int)floor((p0[a] + tm * d[a] - P.b0[a]) / P.vox[a]);
      idx[a] = min(max(i, 0), P.n[a] - 1);
    }
    const int s0 = d[0] > 0.0 ? 1 : -1, s1 = d[1] > 0.0 ? 1 : -1, s2 = d[2] > 0.0 ? 1 : -1;
    int q0 = idx[0] + (s0 > 0), q1 = idx[1] + (s1 > 0), q2 = idx[2] + (s2 > 0);
    int left0 = s0 > 0 ? nx - 1 - idx[0] : idx[0], left1 = s1 > 0 ? ny - 1 - idx[1] : idx[1],
        left2 = s2 > 0 ? nz - 1 - idx[2] : idx[2];
    uint32_t at = ((uint32_t)idx[2] * (uint32_t)ny + (uint32_t)idx[1]) * (uint32_t)nx + (uint32_t)idx[0];
    auto crossing = [&](int a, int p) {
      if (d[a] == 0.0) return (double)INFINITY;
      const int first = a == 0 ? 0 : (a == 1 ? nx + 1 : nx + ny + 2);
      return (PLANES ? planes[first + p] : P.b0[a] + p * P.vox[a] - p0[a]) * inv[a];
    };
    // the run of equal labels that began at t_run; `lab` is the label of the voxel
    // being crossed, loaded a step ahead
    double t = t0, t_run = t0;
    int run = 0x7fffffff;
    uint32_t lab = labels[at];
    auto end_run = [&](double te) {
      if (run < n_labels && te > t_run) {
        lens[run * kBlock + tid] += te - t_run;
        any = true;
      }
      t_run = te;
    };
    for (;;) {
      const double u0 = crossing(0, q0), u1 = crossing(1, q1), u2 = crossing(2, q2);
      const bool c1 = u1 < u0;
      const double u01 = c1 ? u1 : u0;
      const bool c2 = u2 < u01;
      const double un = c2 ? u2 : u01;
      const bool last = !(un < t1) || (c2 ? left2 : (c1 ? left1 : left0)) == 0;
      const uint32_t cur = lab;
      if (!last) {
        const bool y = c1 && !c2, x = !c1 && !c2;
        q0 += x ? s0 : 0;
        q1 += y ? s1 : 0;
        q2 += c2 ? s2 : 0;
        left0 -= x;
        left1 -= y;
        left2 -= c2;
        at += (uint32_t)(c2 ? s2 * nx * ny : (c1 ? s1 * nx : s0));
        lab = labels[at];
      }
      // labels past the table read as the last label, as in transport
      const int l = min((int)cur, kMaxLabels - 1);
      const double te = fmin(un, t1);
      if (l != run) {
        end_run(t);
        run = l;
      }
      t = fmax(t, te);
      if (last) break;
    }
    end_run(t);
  }
  double result = 0.0;
  if (any) {
    // bins: per spectral bin its weight and the attenuation of each label (one bin
    // of weight 1 when mono-energetic)
    auto combine = [&](bool opaque) {
      double num = 0.0, le = 0.0;
      for (int e = 0; e < n_bins; ++e) {
        const double* b = bins + (size_t)e * (n_labels + 1);
        le = 0.0;
        for (int l = 0; l < n_labels; ++l) {
          const double len = lens[l * kBlock + tid];
          if (!opaque || len != 0.0) le += len * b[1 + l];
        }
        if (weight > 0.0) num += b[0] * exp(-le);
      }
      return weight > 0.0 ? -log(num / weight) : le;
    };
    result = combine(false);
    if (result != result) result = combine(true);  // 0 of a label of infinite attenuation is nothing
  }
  out[((size_t)k * P.nu + iu) * P.nv + iv] = (float)result;
}

hipError_t launch_primary_exact(const PrimaryGeom& P, const McPrep* prep, const double* cs64, const uint8_t* labels,
                                const double* bins, int n_bins, int n_labels, double weight, float* out,
                                hipStream_t s) {
  const uint64_t rows8 = ((P.nv + kPrimV - 1) / kPrimV + 7) / 8;
  const uint64_t per_view = 8 * rows8 * ((P.nu + kPrimU - 1) / kPrimU);
  if (per_view == 0 || P.n_views <= 0) return hipSuccess;
  if (n_labels < 0 || n_labels > kMaxLabels) return hipErrorInvalidValue;
  const uint64_t np = (uint64_t)P.n[0] + P.n[1] + P.n[2] + 3;
  const size_t lens = sizeof(double) * n_labels * kPrimU * kPrimV;
  const int step = (int)std::min<uint64_t>(P.n_views, max_blocks(kPrimU * kPrimV) / per_view);  // views of a launch
  for (int k = 0; k < P.n_views; k += step) {
    PrimaryGeom Q = P;
    Q.n_views = std::min(step, P.n_views - k);
    const dim3 grid((unsigned)(per_view * Q.n_views));
    float* o = out + (size_t)k * P.nu * P.nv;
    if (np <= 3900)  // with 16 labels' lengths, 63 KB of LDS
      hipLaunchKernelGGL(primary_exact_kernel<true>, grid, dim3(kPrimU * kPrimV), lens + sizeof(double) * np, s, Q, prep,
                         cs64 + 2 * (size_t)k, labels, bins, n_bins, n_labels, weight, o);
    else
      hipLaunchKernelGGL(primary_exact_kernel<false>, grid, dim3(kPrimU * kPrimV), lens, s, Q, prep,
                         cs64 + 2 * (size_t)k, labels, bins, n_bins, n_labels, weight, o);
  }
  return hipGetLastError();
}

// ------------------------------------------------- counts -> line integrals
// CBCT_real325.cu:267-294: clamp N to [1, N0], L = ln N0 - ln N, with N0 the
// photons aimed at the pixel (FLAT 0): base + (a < rem), a = iv nu + iu the
// pixel's place in the aim order; or (an air scan) flat [1 or views][nu][nv],
// 0 where it is <= 0 (FLAT 1 and 2).
// `counts2`, when given, is added to `counts` first (primary + scatter tallies
// in one pass).
//
// A thread takes V pixels (V = 2 where rows of views stay 16-byte aligned) in
// kLineViews views, so N0 and its logarithm are formed once per pixel and no
// index needs a division per element.  The logarithm is table driven (P. T. P. Tang,
// ACM TOMS 16, 1990): of 2^e m, e ln 2 + ln c + ln(1 + r) with c near m from 128 values in
// LDS, r = m / c - 1 and 7 terms of the series, in FP64 to 3e-16 of the result from 1 up
// (exact at 1, where r = m - 1).  Bound by memory: 202 us for 360 views of 512^2, 12 bytes
// a pixel at 5.6 TB/s, with the library's logarithm 296, and with two of them and two
// 64-bit divisions a pixel 543.
constexpr int kLineViews = 12;
constexpr int kLogBits = 7;

__device__ inline void log_table(double2* tab) {  // {1 / c, ln c}; the block synchronises
  const int i = threadIdx.x;
  if (i < 1 << kLogBits) {
    const double inv = i == 0 ? 1.0 : (double)(float)((1 << kLogBits) / ((1 << kLogBits) + i + 0.5));
    tab[i] = make_double2(inv, -log(inv));
  }
}

__device__ inline double log_from(const double2* tab, double v) {
  const uint64_t bits = __double_as_longlong(v);
  const uint32_t hi = (uint32_t)(bits >> 32);
  if (hi - 0x00100000u >= 0x7fe00000u) return log(v);  // not a positive normal number
  const double2 t = tab[(hi >> (20 - kLogBits)) & ((1 << kLogBits) - 1)];
  const double m = __longlong_as_double((bits & 0xfffffffffffffull) | 0x3ff0000000000000ull);
  const double e = (double)((int)(hi >> 20) - 1023);
  const double r = fma(m, t.x, -1.0);
  double p = fma(r, 1.0 / 7.0, -1.0 / 6.0);
  p = fma(r, p, 1.0 / 5.0);
  p = fma(r, p, -1.0 / 4.0);
  p = fma(r, p, 1.0 / 3.0);
  p = fma(r, p, -0.5);
  return fma(e, 0.6931471805599453, t.y) + fma(r * r, p, r);
}

template <int FLAT, int V, bool TWO>
__global__ __launch_bounds__(256) void counts_to_lineint_kernel(const double* __restrict__ counts,
                                                                const double* __restrict__ counts2,
                                                                const double* __restrict__ flat, float* __restrict__ out,
                                                                int n_views, int nu, int nv, uint64_t base,
                                                                uint64_t rem) {
  using In = double __attribute__((ext_vector_type(V)));
  using Out = float __attribute__((ext_vector_type(V)));
  __shared__ double2 tab[1 << kLogBits];
  log_table(tab);
  __syncthreads();
  const int npix = nu * nv;
  const int pix = (int)(blockIdx.x * 256 + threadIdx.x) * V;  // iu nv + iv
  if (pix >= npix) return;
  double n0[V], ln0[V];
#pragma unroll
  for (int i = 0; i < V; ++i) {
    if (FLAT == 0) {
      const int iu = (pix + i) / nv, iv = pix + i - iu * nv;
      n0[i] = (double)(base + ((uint64_t)(iv * nu + iu) < rem ? 1 : 0));
    } else if (FLAT == 1) {
      n0[i] = flat[pix + i];
    }
    if (FLAT < 2) ln0[i] = log_from(tab, n0[i]);
  }
  const int k0 = (int)blockIdx.y * kLineViews, k1 = min(k0 + kLineViews, n_views);
#pragma unroll 4
  for (int k = k0; k < k1; ++k) {
    const size_t at = (size_t)k * npix + pix;
    In c = *(const In*)(counts + at);
    if (TWO) c += *(const In*)(counts2 + at);
    In f{};
    if (FLAT == 2) f = *(const In*)(flat + at);
    Out o;
#pragma unroll
    for (int i = 0; i < V; ++i) {
      const double top = FLAT == 2 ? f[i] : n0[i];
      double v = c[i];
      v = v > top ? top : v;
      v = v < 1.0 ? 1.0 : v;
      o[i] = top > 0.0 ? (float)((FLAT == 2 ? log_from(tab, top) : ln0[i]) - log_from(tab, v)) : 0.f;
    }
    *(Out*)(out + at) = o;
  }
}

template <int FLAT, bool TWO>
static hipError_t launch_lineint(const double* counts, const double* counts2, const double* flat, float* out,
                                 int n_views, int nu, int nv, uint64_t base, uint64_t rem, hipStream_t s) {
  if (n_views <= 0 || nu <= 0 || nv <= 0) return hipSuccess;
  const int npix = nu * nv;
  const uintptr_t all = (uintptr_t)counts | (TWO ? (uintptr_t)counts2 : 0) | (FLAT ? (uintptr_t)flat : 0);
  const bool pairs = npix % 2 == 0 && all % 16 == 0 && (uintptr_t)out % 8 == 0;
  // grid.y holds at most 65535 groups of views
  const size_t step = (size_t)65535 * kLineViews;
  for (size_t k = 0; k < (size_t)n_views; k += step) {
    const int n = (int)std::min(step, (size_t)n_views - k);
    const size_t off = k * npix;
    const dim3 grid((unsigned)((npix + (pairs ? 511 : 255)) / (pairs ? 512 : 256)),
                    (unsigned)((n + kLineViews - 1) / kLineViews));
    const double* f = FLAT == 2 ? flat + off : flat;
    if (pairs)
      hipLaunchKernelGGL((counts_to_lineint_kernel<FLAT, 2, TWO>), grid, dim3(256), 0, s, counts + off,
                         TWO ? counts2 + off : nullptr, f, out + off, n, nu, nv, base, rem);
    else
      hipLaunchKernelGGL((counts_to_lineint_kernel<FLAT, 1, TWO>), grid, dim3(256), 0, s, counts + off,
                         TWO ? counts2 + off : nullptr, f, out + off, n, nu, nv, base, rem);
  }
  return hipGetLastError();
}

hipError_t launch_counts_to_lineint_flat(const double* counts, const double* flat, int flat_views, float* out,
                                         int n_views, int nu, int nv, hipStream_t s) {
  if (flat_views == 1) return launch_lineint<1, false>(counts, nullptr, flat, out, n_views, nu, nv, 0, 0, s);
  return launch_lineint<2, false>(counts, nullptr, flat, out, n_views, nu, nv, 0, 0, s);
}

hipError_t launch_counts_to_lineint(const double* counts, const double* counts2, float* out, int n_views, int nu,
                                    int nv, uint64_t photons_per_view, hipStream_t s) {
  const uint64_t npix = (uint64_t)nu * (uint64_t)nv;
  if (npix == 0) return hipSuccess;
  const uint64_t base = photons_per_view / npix, rem = photons_per_view % npix;
  if (counts2) return launch_lineint<0, true>(counts, counts2, nullptr, out, n_views, nu, nv, base, rem, s);
  return launch_lineint<0, false>(counts, nullptr, nullptr, out, n_views, nu, nv, base, rem, s);
}

}  // namespace monte
