// ssolh -- wavefront flux integrator on one MI355X (gfx950).
//
// Replaces the reference's OpenMP realisation loop (src/ssol_solver.c:
// 1223-1248 running trace_radiative_path, :873-1127) by a wavefront: a lane
// per realisation, and per launch one ray of every path in flight.
//
//   k_start     draws the realisations' start points, sun directions and
//               wavelengths, traces their shadow rays and shades the start
//               points;
//   k_resume    takes the paths of a queue one ray further: two-level BVH
//               traversal in FP32 boxes with the reference's any-hit filter
//               inline (src/ssol_scene.c:438-536) and the FP64 quadric
//               refinement (src/ssol_shape.c:1449-1494), then the tail of the
//               reference loop iteration that traced the ray (miss, segment
//               extinction, Russian roulette, point update) and the head of
//               the next one (extinction, BSDF or virtual pass-through,
//               receiver weights). Both leave the paths that go on in the
//               next queue; finished realisations flush their tallies with
//               wave-aggregated FP64 atomics;
//   k_scan_chunks / k_scan_top / k_queue_list  list the queue's paths in the
//               order they started in (waves' counts, two-level scan, list).
//
// The host launches k_resume until no path goes on, or few enough do for one
// launch to run them through to their ends.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <float.h>
#include <math.h>
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <vector>

#include "ssolh.h"
#include "ssolh_device.hpp"
#include "ssolh_device32.hpp"

using namespace ssolh;

namespace {

constexpr int BLOCK = 128;           // threads per block (2 waves)
constexpr int MAX_STACK = 32;        // traversal stack entries per thread in LDS, largest kernel
constexpr int START_STACK = 20, RESUME_STACK = 32;  // LDS stack entries per lane of the path kernels
constexpr uint32_t SENTINEL = 0xFFFFFFFFu;
constexpr uint32_t LEAF = 0x80000000u;
constexpr uint32_t NONE = 0xFFFFFFFFu;
constexpr uint32_t TOP_REF = 0x40000000u;  // inner-node reference into the LDS copy
constexpr uint32_t EMPTY4 = 0xFFFFFFFEu;   // absent child of a 4-wide node
constexpr int TOP_NODES = 31;              // TLAS nodes staged in LDS (3.9 KB): 3 levels
constexpr float SLAB_SLACK = 0x1p-21f;     // box-test slack (FRay), per unit of max |o*|
constexpr int MAX_PEND = 8;          // compile-time bound of pending entries

// Per-thread message of the last failing call
thread_local char g_err[512] = "";

void set_err(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

#define HIP_TRY(expr)                                                        \
  do {                                                                       \
    hipError_t e__ = (expr);                                                 \
    if (e__ != hipSuccess) {                                                 \
      set_err("%s: %s (%s:%d)", #expr, hipGetErrorString(e__), __FILE__,     \
              __LINE__);                                                     \
      return -(int)e__;                                                      \
    }                                                                        \
  } while (0)

// -------------------------------------------------------------------------
// Device scene
// -------------------------------------------------------------------------
// IssInfo::obj_flags bit (beside the SSOLH_OBJECT_* ones): the object has
// one shaded shape
constexpr uint32_t OBJ_ONE_SHAPE = 1u << 31;

// What a hit on (instance, shaded shape) needs, gathered at upload so that a
// hit costs one lookup: global index = instance.isshape_first + sshape.
struct alignas(8) IssInfo {
  uint32_t inst;
  uint32_t shape;
  uint32_t mtl_front, mtl_back;
  int32_t receiver;        // receiver slot of the instance or -1
  uint32_t receiver_mask;  // ssol_side_flag bits
  uint32_t shape_type;     // enum ssolh_shape_type
  uint32_t obj_flags;      // SSOLH_OBJECT_* of the instance's object, OBJ_ONE_SHAPE
  int64_t prim_tally;      // first per-primitive slot or -1
};

// BVH node of the traversal: four child boxes as one 16-byte row per axis
// and side (box[axis][0] the four lower planes, box[axis][1] the upper
// ones; an absent child has lower planes +inf and upper planes -inf, which
// no ray crosses) and four child references in the form the traversal
// follows (inner node index, TOP_REF | index into the LDS copy,
// LEAF | (count - 1) << 28 | first item, or EMPTY4). Built at upload by
// collapsing the host's BVH2 (each node takes the children and grandchildren
// of a BVH2 node, opening the largest child boxes first), which halves the
// depth a ray descends.
struct alignas(16) Node4 {
  float box[3][2][4];
  uint32_t child[4];
  uint32_t pad[4];
};
static_assert(sizeof(Node4) == 128, "Node4 layout");

struct StartAlias {
  double prob;
  uint32_t inst, inst_alias;
};

struct DScene {
  Spectra spectra;
  const ssolh_medium* media;
  uint32_t air;
  const ssolh_material* mtls;
  const ssolh_shape* shapes;
  const ssolh_object* objects;
  const Node4* nodes;
  uint32_t tlas_root;
  // copies of the TLAS's top levels (breadth first, children in the set
  // referenced as TOP_REF | index), staged in LDS by the trace kernels
  const Node4* top;
  uint32_t ntop;
  uint32_t root_ref;         // first node reference of a traversal
  float slack_scale;         // box-test slack per unit of max |o*| (SLAB_SLACK)
  const ssolh_triangle* tris;
  const ssolh_instance* insts;
  const uint32_t* tlas_inst;
  const ssolh_inst_sshape* isshapes;
  const IssInfo* iss;
  const ssolh_sample_tri* stris;
  const ssolh_alias* alias;
  // per alias cell: its probability and the instances of its two sampled
  // triangles (the start instance in one load, for k_start_keys)
  const struct StartAlias* salias;
  const float* obj_box;  // [object][6]: object-space lo xyz, hi xyz
  uint32_t nstris;
  ssolh_sun sun;
  double S, S_proxy;
  uint32_t nrcv, nsamp;
};

// Ray and hit records, indexed by slot ------------------------------------
enum : uint32_t {
  RF_SIDE_SHIFT = 16,     // 2 bits: side of the origin point
  RF_DISCARD_VIRTUAL = 1u << 18,
  RF_REVERSED = 1u << 19,
  RF_ANY_HIT = 1u << 20
};

struct alignas(16) RayRec {
  double ox, oy, oz;
  double dx, dy, dz;
  float tmin;
  uint32_t iss_from;   // (instance, shaded shape) of the emitting point
  uint32_t prim_from;  // its triangle
  uint32_t flags;      // side << RF_SIDE_SHIFT | RF_*
};
static_assert(sizeof(RayRec) == 64, "RayRec layout");

struct alignas(16) HitRec {
  double t;             // distance of the nearest accepted triangle
  double qdst;          // nearest refined quadric distance (punched shapes)
  double nx, ny, nz;    // unnormalised world normal: triangle Ng, or quadric gradient
  uint32_t iss, prim;   // iss == NONE <=> miss
};
static_assert(sizeof(HitRec) == 48, "HitRec layout");

// Path state, indexed by slot ---------------------------------------------
enum : uint32_t {
  PF_STAGE_BOUNCE = 1u << 0,   // else: waiting for the shadow ray
  PF_HIT_VIRTUAL = 1u << 1,    // the point that emitted the ray is virtual
  PF_IN_ATM = 1u << 2,         // the incoming segment of that point was in air
  PF_ACTIVE = 1u << 3,
  PF_HIT_RECEIVER = 1u << 4    // the path reached a receiver (path tracking)
};

struct Counters {
  unsigned long long failed;
  unsigned long long spills;
  unsigned long long segments;      // traced rays (added by k_scan_top, one thread)
  unsigned int aborted;
  unsigned int stop;                // aborted as the current wavefront began
  unsigned int wavefronts;          // wavefronts begun
  unsigned int iterations, gens;    // generations of rays: of the passes so far, of this one
  unsigned int left;                // length of the list of paths that go on
  unsigned int log_flushes;         // reductions of the per-primitive log
  unsigned long long log_over;      // records that found the log full
};

// Segments of a large per-primitive log, and the distance between their
// counters (a cache line, in counters)
constexpr uint32_t LOG_SEGS = 16, LOG_LINE = 16;

// Tallies that every wave updates (global fields, counts) or that few keys
// share (receivers, sampled instances) are striped: block b adds into
// stripe b & mask, so concurrent atomics spread over many cache lines; the
// stripes are folded into stripe 0 after the solve. The stripe count of a
// tally shrinks with its size (2^21 doubles at most over all its stripes).
struct Tallies {
  double* global;   // [mask_g+1][njobs][16]: 6 fields x {w, w2}, then the
                    // realisation count (exact below 2^53); one 128-byte line
  double* rcv;      // [nrcv][2][10][2]: zero until folded (k_fold_rcv)
  double* samp;     // [mask_s+1][nsamp][2][2]
  unsigned long long* samp_count;    // [mask_s+1][nsamp]
  double* sxr;      // [mask_x+1][nsamp][nrcv][2][10][2]
  double* prim;     // [mask_p+1][nprim][2][10][2]
  uint32_t mask_g, mask_s, mask_x, mask_p;
  uint32_t nrcv, nsamp, njobs;
  uint64_t nprim;
  // Log of finished paths' per-primitive entries (prim_add), reduced into
  // `prim` by key (k_prim_reduce): record i is the key log_key[i] and the 10
  // fields' weights log_val[10 i ..]. Blocks log to the segment blockIdx &
  // log_mask, the log_seg records from segment * log_seg on; log_n[segment *
  // LOG_LINE] counts the records asked for, also past log_seg (those went to
  // atomics). log_cap: records of all segments, 0 without a log.
  uint32_t* log_key;
  double* log_val;
  unsigned long long* log_n;
  uint64_t log_cap;
  uint32_t log_seg, log_mask;
};

struct SolveParams {
  uint64_t N;
  uint64_t max_failed;
  uint64_t key;
  uint64_t counter;
  uint32_t slots;
  uint32_t npend;
  // several suns in one solve: realisations [job_first[j], job_first[j+1])
  // run under job_suns[j]; without job_suns the one job is the scene's sun
  const uint64_t* job_first;
  const ssolh_sun* job_suns;
  uint32_t njobs;
};

// Job of realisation id: the last j with job_first[j] <= id (empty jobs are
// skipped because their successor starts at the same id)
__device__ __forceinline__ uint32_t job_of(const SolveParams& prm, uint64_t id) {
  if (prm.njobs <= 1) return 0;
  uint32_t lo = 0, hi = prm.njobs;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (prm.job_first[mid] <= id) lo = mid; else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ const ssolh_sun& job_sun(const DScene& S, const SolveParams& prm,
                                                     uint32_t job) {
  return prm.job_suns ? prm.job_suns[job] : S.sun;
}

// Adjoint solve (score-function gradients, see shade_path): null grad <=> off.
struct AdjParams {
  double* grad;              // [nparams][3]: d/d aim angle 1, 2, d/d slope error
  const int32_t* inst_param; // [ninstances]: parameter slot of an instance or -1
  const double* axes;        // [nparams][2][3]: world rotation axes of the aim angles
  const double* gmap;        // [nprim_tallies][2]: upstream weight per unit absorbed flux
  double d_total;            // upstream weight of absorbed_by_receivers
  double4* s;                // [slots]: scores of the path (aim 1, aim 2, slope), q
  uint32_t* p;               // [slots]: parameter slot of the path or NONE
};

// Path recording (src/ssol_solver.c:898-1127): null vtx <=> off. Vertices
// are appended in arrival order, tagged with their realisation and index.
struct TrackParams {
  ssolh_track_vertex* vtx;
  unsigned long long* nvtx;  // vertices produced (may exceed cap)
  unsigned long long cap;
  uint8_t* type;             // [N] SSOLH_PATH_* of each realisation
  uint32_t* seq;             // [slots] vertices recorded by the slot's path
  double4* pos;              // [slots] the point the slot's ray leaves
  double sun_len, inf_len;
};

__device__ void track_vertex(const TrackParams& K, uint32_t slot, uint64_t path, d3 p, double w) {
  const uint32_t s = K.seq[slot];
  K.seq[slot] = s + 1;
  const unsigned long long i = atomicAdd(K.nvtx, 1ull);
  if (i < K.cap) {
    ssolh_track_vertex v;
    v.path = path;
    v.index = s;
    v.pad__ = 0;
    v.pos[0] = p.x; v.pos[1] = p.y; v.pos[2] = p.z;
    v.weight = w;
    K.vtx[i] = v;
  }
}

// Work list: slot of entry q (a null list is the identity)
__device__ __forceinline__ uint32_t slot_of(const uint32_t* list, uint32_t q) {
  return list ? list[q] : q;
}

// -------------------------------------------------------------------------
// Wave and block helpers (64-wide waves)
// -------------------------------------------------------------------------
// Value of lane (i ^ pattern) within DPP rows, both halves of a double
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((long long)(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo));
}

// Sums of N values (a multiple of 4) over the 64 lanes of a wave, every lane
// active: lane l returns the total of value (l / 16) * N / 4 + l % 16, where
// l % 16 < N / 4. Two swaps halve the values in hand instead of adding both
// halves of each: v_permlane32_swap leaves value i in the lower and value i +
// N/2 in the upper 32 lanes, v_permlane16_swap does the same for rows of 16;
// DPP moves then add up the row within quads (quad_perm [1,0,3,2], [2,3,0,1]),
// half rows (row_half_mirror) and the row (row_mirror). 20 values: 105
// instructions, where summing each over all lanes takes 540.
template <int N>
__device__ __forceinline__ double wave_totals(const double (&v)[N]) {
  static_assert(N % 4 == 0 && N / 4 <= 16, "values per row");
  auto swapped = [](double a, double b, auto swap) {
    const uint64_t x = (uint64_t)__double_as_longlong(a), y = (uint64_t)__double_as_longlong(b);
    const auto lo = swap((uint32_t)x, (uint32_t)y);
    const auto hi = swap((uint32_t)(x >> 32), (uint32_t)(y >> 32));
    return __longlong_as_double((long long)(((uint64_t)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((uint64_t)hi[1] << 32) | lo[1]));
  };
  double h[N / 2], r[N / 4];
#pragma unroll
  for (int i = 0; i < N / 2; ++i)
    h[i] = swapped(v[i], v[i + N / 2], [](uint32_t x, uint32_t y) {
      return __builtin_amdgcn_permlane32_swap(x, y, false, false);
    });
#pragma unroll
  for (int i = 0; i < N / 4; ++i)
    r[i] = swapped(h[i], h[i + N / 4], [](uint32_t x, uint32_t y) {
      return __builtin_amdgcn_permlane16_swap(x, y, false, false);
    });
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    r[i] += dpp_move<0xB1>(r[i]);
    r[i] += dpp_move<0x4E>(r[i]);
    r[i] += dpp_move<0x141>(r[i]);
    r[i] += dpp_move<0x140>(r[i]);
  }
  double s = r[0];
#pragma unroll
  for (int i = 1; i < N / 4; ++i) s = (__lane_id() & 15u) == (unsigned)i ? r[i] : s;
  return s;
}

__device__ __forceinline__ unsigned lane_id() { return __lane_id(); }

__device__ __forceinline__ void atomic_add(double* p, double v) {
  if (v != 0) unsafeAtomicAdd(p, v);
}

// Adds the wave's totals of v to base[i], i < NV, each by one lane. Every lane
// of the wave calls it.
template <int NV, int N>
__device__ __forceinline__ void add_totals(const double (&v)[N], double* base) {
  const double s = wave_totals<N>(v);
  const unsigned j = lane_id() & 15u, i = (lane_id() >> 4) * (N / 4) + j;
  if (j < N / 4 && i < NV) atomic_add(base + i, s);
}

// Adds the NV values of each participating lane at base[key*STRIDE + i]. The
// lanes of each key that several lanes hold are reduced across the wave and
// added by one atomic per value; a lane with a key of its own adds for
// itself. FP64 atomics issue at one rate for the whole device (about 88 of 20
// values per microsecond and CU), so a reduction pays from two lanes on.
// v is padded to N values, a multiple of 4. Must be called by the whole wave.
template <int NV, int STRIDE = NV, int N>
__device__ __forceinline__ void keyed_add(bool has, uint64_t key, const double (&v)[N],
                                          double* base) {
  bool todo = has, alone = false;
  for (uint64_t mask = __ballot(todo); mask; mask = __ballot(todo)) {
    const int leader = __ffsll((unsigned long long)mask) - 1;
    const uint64_t lkey = __shfl(key, leader, 64);
    const bool match = todo && key == lkey;
    if (__popcll(__ballot(match)) > 1) {
      double m[N];
#pragma unroll
      for (int i = 0; i < N; ++i) m[i] = match ? v[i] : 0.0;
      add_totals<NV, N>(m, base + lkey * STRIDE);
    } else {
      alone = alone || match;
    }
    todo = todo && !match;
  }
  if (alone) {
#pragma unroll
    for (int i = 0; i < NV; ++i) atomic_add(base + key * STRIDE + i, v[i]);
  }
}

__device__ __forceinline__ unsigned long long wave_count_add(bool pred, unsigned long long* ctr) {
  const uint64_t mask = __ballot(pred);
  if (!mask) return 0;
  const int leader = __ffsll((unsigned long long)mask) - 1;
  unsigned long long base = 0;
  if ((int)lane_id() == leader) base = atomicAdd(ctr, (unsigned long long)__popcll(mask));
  base = __shfl(base, leader, 64);
  const uint64_t below = mask & ((1ull << lane_id()) - 1ull);
  return base + (unsigned long long)__popcll(below);
}

// Record `pos` of the per-primitive log: the weights a[f] * factor of a key
template <typename R>
__device__ __forceinline__ void log_record(const Tallies& T, uint64_t pos, uint32_t key, const R* a,
                                           double factor) {
  T.log_key[pos] = key;
  double2* v = (double2*)(T.log_val + pos * 10u);
#pragma unroll
  for (int f = 0; f < 5; ++f)
    v[f] = make_double2((double)a[2 * f] * factor, (double)a[2 * f + 1] * factor);
}

// A finished path's per-primitive entry: the key and the 10 fields' weights
// a[f] * factor. FP64 atomics issue at one device-wide rate whatever their
// addresses, and the entries of a wave fall on as many primitives as it has
// lanes, so the 20 atomics of an entry (x and x^2 per field) would cost far
// more than the 84 bytes of a record in the log, which k_prim_reduce sums
// by key. A full log takes the atomics. Must be called by the
// whole wave.
template <typename R>
__device__ void prim_add(const Tallies& T, bool has, uint32_t key, const R* a, double factor) {
  const uint32_t s = blockIdx.x & T.log_mask;
  const unsigned long long pos = T.log_cap ? wave_count_add(has, T.log_n + s * LOG_LINE) : ~0ull;
  if (!has) return;
  if (pos < T.log_seg) {
    log_record(T, (uint64_t)s * T.log_seg + pos, key, a, factor);
    return;
  }
  double* pb = T.prim + (size_t)(blockIdx.x & T.mask_p) * T.nprim * 40u + (size_t)key * 20u;
#pragma unroll
  for (int f = 0; f < 10; ++f) {
    const double x = (double)a[f] * factor;
    atomic_add(pb + 2 * f, x);
    atomic_add(pb + 2 * f + 1, x * x);
  }
}

#include "ssolh_group.hpp"


// -------------------------------------------------------------------------
// Traversal with the reference hit filter
// -------------------------------------------------------------------------
// Ray of the box tests: the distance to the plane x = p is p * ix + ox (one
// FMA), and the rows of a node that hold the near planes of the ray's
// direction signs are read by offset, so a slab needs no min/max. The
// rounding of ox = -o * ix puts up to |ox| 2^-24 of error on every plane
// distance, which with km-scale origins is far more than the (p - o) * ix
// form's error near the origin (about 6e-5 m against 1e-6 m at 1.5 km):
// a box is crossed when tnear - slack <= tfar, slack = 2^-21 max |o*|
// (SLAB_SLACK), so the test culls no box the subtracting form keeps. ox, oy, oz are kept
// finite; a ray with a non-finite origin or direction gets
// ox = oy = oz = +inf, so tnear - slack is NaN and it crosses no box.
struct FRay {
  float ix, iy, iz;      // 1 / direction (components at least 1e-30 in magnitude)
  float ox, oy, oz;      // -origin / direction
  uint32_t nx, ny, nz;   // byte offset in a Node4 of each axis's near-plane row
};

__device__ __forceinline__ FRay make_fray32(float ox, float oy, float oz, float dx, float dy,
                                            float dz) {
  auto inv = [](float f) { return 1.0f / (fabsf(f) > 1e-30f ? f : copysignf(1e-30f, f)); };
  auto off = [](float o, float i) { return fminf(fmaxf(-o * i, -FLT_MAX), FLT_MAX); };
  FRay r;
  r.ix = inv(dx);
  r.iy = inv(dy);
  r.iz = inv(dz);
  r.ox = off(ox, r.ix);
  r.oy = off(oy, r.iy);
  r.oz = off(oz, r.iz);
  r.nx = r.ix < 0.f ? 16u : 0u;
  r.ny = r.iy < 0.f ? 48u : 32u;
  r.nz = r.iz < 0.f ? 80u : 64u;
  const bool finite = fabsf(ox) <= FLT_MAX && fabsf(oy) <= FLT_MAX && fabsf(oz) <= FLT_MAX &&
                      fabsf(dx) <= FLT_MAX && fabsf(dy) <= FLT_MAX && fabsf(dz) <= FLT_MAX;
  if (!finite) {
    r.ix = r.iy = r.iz = 1.f;
    r.ox = r.oy = r.oz = INFINITY;
  }
  return r;
}

__device__ __forceinline__ FRay make_fray(d3 o, d3 d) {
  return make_fray32((float)o.x, (float)o.y, (float)o.z, (float)d.x, (float)d.y, (float)d.z);
}

// Ray in the shear frame of the watertight ray/triangle test (Woop,
// Benthin, Wald, JCGT 2013): computed once per ray (and per instance).
struct Shear {
  int kx, ky, kz;
  double Sx, Sy, Sz;
};

__device__ __forceinline__ Shear make_shear(d3 d) {
  const double a[3] = {fabs(d.x), fabs(d.y), fabs(d.z)};
  const double v[3] = {d.x, d.y, d.z};
  Shear s;
  s.kz = a[0] > a[1] ? (a[0] > a[2] ? 0 : 2) : (a[1] > a[2] ? 1 : 2);
  s.kx = (s.kz + 1) % 3;
  s.ky = (s.kx + 1) % 3;
  if (v[s.kz] < 0) { const int t = s.kx; s.kx = s.ky; s.ky = t; }
  s.Sx = v[s.kx] / v[s.kz];
  s.Sy = v[s.ky] / v[s.kz];
  s.Sz = 1.0 / v[s.kz];
  return s;
}

__device__ __forceinline__ double comp(d3 p, int k) { return k == 0 ? p.x : (k == 1 ? p.y : p.z); }

// Watertight: a ray through a shared edge or vertex hits at least one of
// the triangles. The edge functions of a shared edge must come out as exact
// negations of each other in the two triangles, so no product here may be
// fused into an FMA. Returns the distance or -1.
__device__ __forceinline__ double ray_triangle(d3 o, const Shear& s, d3 v0, d3 v1, d3 v2) {
#pragma clang fp contract(off)
  const d3 A = v0 - o, B = v1 - o, C = v2 - o;
  const double Az = comp(A, s.kz), Bz = comp(B, s.kz), Cz = comp(C, s.kz);
  const double Ax = comp(A, s.kx) - s.Sx * Az, Ay = comp(A, s.ky) - s.Sy * Az;
  const double Bx = comp(B, s.kx) - s.Sx * Bz, By = comp(B, s.ky) - s.Sy * Bz;
  const double Cx = comp(C, s.kx) - s.Sx * Cz, Cy = comp(C, s.ky) - s.Sy * Cz;
  const double U = Cx * By - Cy * Bx;
  const double V = Ax * Cy - Ay * Cx;
  const double W = Bx * Ay - By * Ax;
  if ((U < 0 || V < 0 || W < 0) && (U > 0 || V > 0 || W > 0)) return -1;
  const double det = U + V + W;
  if (det == 0) return -1;
  const double T = U * s.Sz * Az + V * s.Sz * Bz + W * s.Sz * Cz;
  return T / det;
}

struct ShapeQ;

struct TraceState {
  double tbest;
  double qdst;     // nearest refined quadric distance
  uint32_t qiss;   // its (instance, shaded shape): the normal is rebuilt after the traversal
  uint32_t tri;  // the best triangle (its world normal is rebuilt after the traversal)
  uint32_t iss, prim;
  bool punched;  // the best triangle belongs to a punched surface
};

// World geometry normal (unnormalised) of mesh triangle `tri` of instance `inst`
__device__ __forceinline__ d3 mesh_ng(const DScene& S, uint32_t inst, const ssolh_triangle& tri) {
  const d3 v0 = ld3(tri.v0), v1 = ld3(tri.v1), v2 = ld3(tri.v2);
  return tmul(S.insts[inst].inv_linear, cross(v2 - v0, v1 - v0));
}

// Returns true if the candidate is accepted (src/ssol_scene.c:438-536).
__device__ bool filter(const DScene& S, const RayRec& r, d3 o, d3 d, uint32_t iss_id,
                       const ssolh_triangle& tri, double t, TraceState& ts, d3& ng_out,
                       bool& punched) {
  const uint32_t side_from = (r.flags >> RF_SIDE_SHIFT) & 3u;
  const IssInfo is = S.iss[iss_id];
  uint32_t side;
  double dst = 0;
  d3 qn = mk(0, 0, 0);
  if (t < r.tmin) return false;
  punched = is.shape_type != SSOLH_SHAPE_MESH;
  if (!punched) {
    if (t <= 1.e-6 || t <= r.tmin || (tri.prim == r.prim_from && iss_id == r.iss_from))
      return false;
    ng_out = mesh_ng(S, is.inst, tri);
    side = dot(ng_out, d) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
  } else {
    const ssolh_inst_sshape& q = S.isshapes[iss_id];
    const ssolh_shape& sh = S.shapes[is.shape];
    const d3 lo = mul(q.R_inv, o - ld3(q.T));
    const d3 ldir = mul(q.R_inv, d);
    d3 grad;
    if (!quadric_hit(sh.quadric, sh.qparam, lo, ldir, t, dst, grad)) return false;
    if (!(dst < (double)FLT_MAX)) return false;
    if ((double)(float)dst <= r.tmin) return false;
    qn = normalize(tmul(q.R_inv, grad));
    side = dot(d, qn) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
    if (iss_id == r.iss_from && side != side_from) return false;
  }
  if (r.flags & RF_REVERSED) side = side == SSOL_FRONT_ ? SSOL_BACK_ : SSOL_FRONT_;
  const ssolh_material& m = S.mtls[side == SSOL_FRONT_ ? is.mtl_front : is.mtl_back];
  if (m.type == SSOLH_MTL_VIRTUAL) {
    if (r.flags & RF_DISCARD_VIRTUAL) return false;
    if (!(is.receiver_mask & side)) return false;
  }
  if (punched && ts.qdst >= dst) {
    ts.qdst = dst;
    ts.qiss = iss_id;
  }
  return true;
}

// Distance at which the ray (o, d) leaves box b (lo xyz, hi xyz); an axis
// the ray runs parallel to bounds nothing.
__device__ double box_exit(const float* b, d3 o, d3 d) {
  const double oo[3] = {o.x, o.y, o.z}, dd[3] = {d.x, d.y, d.z};
  double t = INFINITY;
  for (int a = 0; a < 3; ++a) {
    if (dd[a] == 0) continue;
    const double t0 = ((double)b[a] - oo[a]) / dd[a], t1 = ((double)b[3 + a] - oo[a]) / dd[a];
    t = fmin(t, fmax(t0, t1));
  }
  return t;
}

// Distance at which the world ray (o, d) leaves the object box of instance
// inst_id (in the instance's object space, where the trace's triangle
// distances are taken)
__device__ double object_exit(const DScene& S, uint32_t inst_id, d3 o, d3 d) {
  const ssolh_instance& inst = S.insts[inst_id];
  const d3 T = mk(inst.transform[9], inst.transform[10], inst.transform[11]);
  return box_exit(S.obj_box + 6 * (size_t)inst.object, mul(inst.inv_linear, o - T),
                  mul(inst.inv_linear, d));
}

// Whether root k of the n roots t[] of a ray / quadric equation can be the
// one the filter's refinement takes for a candidate at a distance in
// [0, t_hi]: the root nearest the candidate's distance
__device__ bool root_choosable(const double t[2], int n, int k, double t_hi) {
  if (n == 1) return true;
  const double other = t[1 - k];
  if (!(fabs(other) < (double)FLT_MAX) || t[k] <= other) return true;
  return !(t_hi * 1.001 + 1e-3 < 0.5 * (t[k] + other));
}

// Whether the filter can accept a candidate on (instance, shaded shape)
// iss_id, a punched shape, for a ray that leaves it at tmin 0 (world ray o,
// d) and whose candidates on it lie within distance t_hi. The filter
// refines every candidate of the shape to the root of the same ray /
// quadric equation nearest the candidate's distance, and accepts it only
// past tmin and on the side the ray left. A root that passes these checks
// (computed here exactly as the filter computes them) can be chosen when it
// is the only root, when it is the nearer one, or when the candidates reach
// the midpoint between the roots; otherwise no candidate of the shape can be
// accepted.
__device__ bool punched_rehit_possible(const DScene& S, const RayRec& r, d3 o, d3 d,
                                       uint32_t iss_id, double t_hi) {
  const uint32_t side_from = (r.flags >> RF_SIDE_SHIFT) & 3u;
  const IssInfo is = S.iss[iss_id];
  const ssolh_inst_sshape& q = S.isshapes[iss_id];
  const ssolh_shape& sh = S.shapes[is.shape];
  const d3 lo = mul(q.R_inv, o - ld3(q.T));
  const d3 ldir = mul(q.R_inv, d);
  double a, b, c, t[2];
  if (!quadric_coeffs(sh.quadric, sh.qparam, lo, ldir, a, b, c)) return false;
  const int n = quadric_roots(a, b, c, t);
  for (int k = 0; k < n; ++k) {
    if (!(t[k] < (double)FLT_MAX)) continue;
    if ((double)(float)t[k] <= r.tmin) continue;
    const d3 grad = quadric_grad(sh.quadric, sh.qparam, lo + ldir * t[k]);
    const d3 qn = normalize(tmul(q.R_inv, grad));
    const uint32_t side = dot(d, qn) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
    if (side != side_from) continue;
    if (root_choosable(t, n, k, t_hi)) return true;
  }
  return false;
}

// Unit world normal of the quadric of (instance, shaded shape) `iss` where the
// world ray (o, d) meets it at distance dst: the gradient of quadric_hit's
// refinement at the same point, as the filter took it
__device__ d3 quadric_normal(const DScene& S, uint32_t iss, d3 o, d3 d, double dst) {
  const ssolh_inst_sshape& q = S.isshapes[iss];
  const ssolh_shape& sh = S.shapes[S.iss[iss].shape];
  const d3 lo = mul(q.R_inv, o - ld3(q.T));
  const d3 ldir = mul(q.R_inv, d);
  return normalize(tmul(q.R_inv, quadric_grad(sh.quadric, sh.qparam, lo + ldir * dst)));
}

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

// What a visit reads of a node: the near- and far-plane rows of the ray's
// direction signs and the child references
struct NodeRows {
  v4f n[3], f[3];
  v4u child;
};

// Rows of node `ref` of the device array (32-bit byte offsets from the
// array's base: the loads take the base in scalar registers)
__device__ __forceinline__ NodeRows node_rows(const Node4* __restrict__ nodes, uint32_t ref,
                                              const FRay& r) {
  const char* b = (const char*)nodes;
  const uint32_t base = ref * (uint32_t)sizeof(Node4);
  const uint32_t o[3] = {base + r.nx, base + r.ny, base + r.nz};
  NodeRows w;
  for (int a = 0; a < 3; ++a) {
    w.n[a] = *(const v4f*)(b + o[a]);
    w.f[a] = *(const v4f*)(b + (o[a] ^ 16u));
  }
  w.child = *(const v4u*)(b + base + 96u);
  return w;
}

// The same from the LDS copy of the top levels, through an LDS (address
// space 3) pointer: the loads are ds_reads, where a pointer that may address
// either LDS or global memory would make them flat accesses
__device__ __forceinline__ NodeRows lds_rows(const Node4* lds, uint32_t i, const FRay& r) {
  typedef const __attribute__((address_space(3))) char* lds_b;
  const lds_b b = (lds_b)lds;
  const uint32_t base = i * (uint32_t)sizeof(Node4);
  const uint32_t o[3] = {base + r.nx, base + r.ny, base + r.nz};
  typedef const __attribute__((address_space(3))) v4f* lf;
  typedef const __attribute__((address_space(3))) v4u* lu;
  NodeRows w;
  for (int a = 0; a < 3; ++a) {
    w.n[a] = *(lf)(b + o[a]);
    w.f[a] = *(lf)(b + (o[a] ^ 16u));
  }
  w.child = *(lu)(b + base + 96u);
  return w;
}

// Traversal stack of one lane: its first STACK entries in LDS (stride
// BLOCK), the rest, when the scene's bound exceeds STACK, in a global array
// of `extra` entries per work-list position (stride: the list's capacity)
struct TStack {
  uint32_t* lds;
  uint32_t* ovf;   // this lane's first overflow entry, or null
  uint32_t stride, extra;
  int sp;
};

template <int STACK>
__device__ __forceinline__ void tpush(TStack& s, uint32_t v) {
  if (s.sp < STACK) s.lds[s.sp * BLOCK] = v;
  else if ((uint32_t)(s.sp - STACK) < s.extra) s.ovf[(size_t)(s.sp - STACK) * s.stride] = v;
  ++s.sp;
}

// false: the stack is empty (or, never with the host's bound, past its end)
template <int STACK>
__device__ __forceinline__ bool tpop(TStack& s, uint32_t& ref) {
  if (s.sp == 0) return false;
  --s.sp;
  if (s.sp < STACK) {
    ref = s.lds[s.sp * BLOCK];
  } else {
    if ((uint32_t)(s.sp - STACK) >= s.extra) return false;
    ref = s.ovf[(size_t)(s.sp - STACK) * s.stride];
  }
  return true;
}

// One visit of a 4-wide inner node: the children whose boxes the ray
// crosses in [tmin, tmax], nearest first; the nearest becomes `ref`, the
// others are pushed farthest first (so the next nearest is on top). With no
// child crossed, `ref` is popped; false when the stack is empty.
template <int STACK>
__device__ __forceinline__ bool visit4(const NodeRows& w, const FRay& fr, float tmin, float tmax,
                                       float slack_scale, uint32_t& ref, TStack& st) {
  float k[4];
  uint32_t r[4];
  const float slack = slack_scale * fmaxf(fabsf(fr.ox), fmaxf(fabsf(fr.oy), fabsf(fr.oz)));
  for (int c = 0; c < 4; ++c) {
    const float tn = fmaxf(fmaxf(fmaf(w.n[0][c], fr.ix, fr.ox), fmaf(w.n[1][c], fr.iy, fr.oy)),
                           fmaxf(fmaf(w.n[2][c], fr.iz, fr.oz), tmin));
    const float tf = fminf(fminf(fmaf(w.f[0][c], fr.ix, fr.ox), fmaf(w.f[1][c], fr.iy, fr.oy)),
                           fminf(fmaf(w.f[2][c], fr.iz, fr.oz), tmax));
    k[c] = tn - slack <= tf ? tn : INFINITY;
    r[c] = w.child[c];
  }
  // sorting network (0,1)(2,3)(0,2)(1,3)(1,2)
  auto cs = [&](int a, int b) {
    const bool sw = k[b] < k[a];
    const float ka = k[a], kb = k[b];
    const uint32_t ra = r[a], rb = r[b];
    k[a] = sw ? kb : ka; k[b] = sw ? ka : kb;
    r[a] = sw ? rb : ra; r[b] = sw ? ra : rb;
  };
  cs(0, 1); cs(2, 3); cs(0, 2); cs(1, 3); cs(1, 2);
  const int cnt = (k[0] < INFINITY) + (k[1] < INFINITY) + (k[2] < INFINITY) + (k[3] < INFINITY);
  if (cnt == 0) return tpop<STACK>(st, ref);
  if (cnt >= 4) tpush<STACK>(st, r[3]);
  if (cnt >= 3) tpush<STACK>(st, r[2]);
  if (cnt >= 2) tpush<STACK>(st, r[1]);
  ref = r[0];
  return true;
}

// Overflow of the traversal stacks past their LDS part: `extra` entries per
// work-list position, `stride` = the list's capacity (null when the scene's
// stack bound fits in LDS)
struct TOvf {
  uint32_t* base;
  uint32_t stride, extra;
};

// What a traversal needs to know of one ray of the FP64 form: how it enters
// an instance, tests a triangle against the filter and what it hit.
struct Tracer64 {
  using Ray = RayRec;
  using Hit = HitRec;
  const DScene& S;
  const RayRec& r;
  TraceState ts;
  d3 o, d;   // the ray in the frame of the instance being traversed
  Shear sh;

  __device__ __forceinline__ Tracer64(const DScene& S_, const ShapeQ*, const RayRec& r_)
      : S(S_), r(r_) {
    ts.tbest = INFINITY;
    ts.qdst = INFINITY;
    ts.qiss = NONE;
    ts.tri = 0;
    ts.iss = NONE;
    ts.prim = 0;
    ts.punched = false;
  }
  __device__ __forceinline__ d3 ow() const { return mk(r.ox, r.oy, r.oz); }
  __device__ __forceinline__ d3 dw() const { return mk(r.dx, r.dy, r.dz); }
  __device__ __forceinline__ FRay world() const { return make_fray(ow(), dw()); }
  // A ray that leaves a point of a planar object can meet that object again
  // only at t ~ 0, which the filter rejects: its instance is not entered.
  // Nor is the instance of a one-shape object whose punched shape the ray
  // leaves when the filter could accept no candidate on it.
  __device__ __forceinline__ uint32_t skipped() const {
    if (r.tmin != 0.f) return NONE;
    const IssInfo e = S.iss[r.iss_from];
    if ((e.obj_flags & SSOLH_OBJECT_PLANAR) ||
        ((e.obj_flags & OBJ_ONE_SHAPE) && e.shape_type != SSOLH_SHAPE_MESH &&
         !punched_rehit_possible(S, r, ow(), dw(), r.iss_from, object_exit(S, e.inst, ow(), dw()))))
      return e.inst;
    return NONE;
  }
  template <class InstPtr>
  __device__ __forceinline__ FRay enter(InstPtr inst, uint32_t) {
    const d3 T = mk(inst->transform[9], inst->transform[10], inst->transform[11]);
    double m[9];
    for (int k = 0; k < 9; ++k) m[k] = inst->inv_linear[k];
    o = mul(m, ow() - T);
    d = mul(m, dw());
    sh = make_shear(d);
    return make_fray(o, d);
  }
  // Triangle `tri`, item `index`: true if it is the new nearest hit; tmax:
  // the box culling distance, the best hit so far widened by 2 ulp (FP32)
  __device__ __forceinline__ bool hit(const ssolh_triangle& tri, uint32_t index,
                                      uint32_t iss_first, float& tmax) {
    const double t = ray_triangle(o, sh, ld3(tri.v0), ld3(tri.v1), ld3(tri.v2));
    if (!(t >= r.tmin && t < ts.tbest)) return false;
    d3 ng;
    bool punched;
    const uint32_t iss = iss_first + tri.sshape;
    if (!filter(S, r, ow(), dw(), iss, tri, t, ts, ng, punched)) return false;
    ts.tbest = t;
    tmax = t < (double)FLT_MAX ? (float)t * 1.0000002f + 1e-30f : FLT_MAX;
    ts.iss = iss;
    ts.prim = tri.prim;
    ts.tri = index;
    ts.punched = punched;
    return true;
  }
  __device__ __forceinline__ HitRec result() const {
    HitRec h;
    h.t = ts.tbest;
    h.qdst = ts.qdst;
    d3 n = mk(0, 0, 0);
    if (ts.punched)
      n = quadric_normal(S, ts.qiss, ow(), dw(), ts.qdst);
    else if (ts.iss != NONE)
      n = mesh_ng(S, S.iss[ts.iss].inst, S.tris[ts.tri]);
    h.nx = n.x; h.ny = n.y; h.nz = n.z;
    h.iss = ts.iss;
    h.prim = ts.prim;
    return h;
  }
};

// One ray per lane, each on its own way through the tree. STACK: LDS stack
// entries per lane (the smaller the stack, the more blocks share a CU); the
// scene's bound beyond them goes to the overflow array, column q.
template <class Tracer, int STACK>
__device__ __forceinline__ typename Tracer::Hit
trace_lane(const DScene& S, const ShapeQ* SQ, const typename Tracer::Ray& r, uint32_t q,
           uint32_t* lds_stack, const Node4* lds_top, const TOvf& ovf) {
  Tracer tr(S, SQ, r);
  const bool any_hit = (r.flags & RF_ANY_HIT) != 0;
  TStack st{lds_stack + threadIdx.x, ovf.base ? ovf.base + q : nullptr, ovf.stride, ovf.extra, 0};
  FRay fr = tr.world();
  bool in_blas = false;
  uint32_t iss_first = 0;   // (instance, sshape) base of the BLAS being traversed
  const float ftmin = r.tmin;
  const uint32_t skip_inst = tr.skipped();

  // "while-while" traversal: the lanes of a wave first descend through inner
  // nodes together, then process their leaves together, which keeps the
  // node, instance and triangle code paths from interleaving per lane.
  // SENTINEL (all bits set) reads as a leaf reference and ends the descent.
  uint32_t ref = S.root_ref;
  bool alive = true;
  float tmax = FLT_MAX;
  while (alive) {
    while (!(ref & LEAF)) {
      // the whole node in one round of loads (LDS or global memory, each
      // through its own address space), then its four boxes
      const NodeRows n =
          (ref & TOP_REF) ? lds_rows(lds_top, ref & 0x0FFFFFFFu, fr) : node_rows(S.nodes, ref, fr);
      if (!visit4<STACK>(n, fr, ftmin, tmax, S.slack_scale, ref, st)) {
        alive = false;
        break;
      }
    }
    if (!alive) break;
    if (ref == SENTINEL) {
      // back to the TLAS
      in_blas = false;
      fr = tr.world();
      alive = tpop<STACK>(st, ref);
      continue;
    }
    const uint32_t first = ref & 0x0FFFFFFFu;
    if (!in_blas) {
      // TLAS leaf: one instance, enter its BLAS
      const uint32_t ii = S.tlas_inst[first];
      if (ii == skip_inst) {
        alive = tpop<STACK>(st, ref);
        continue;
      }
      const ssolh_instance* inst = S.insts + ii;
      fr = tr.enter(inst, ii);
      iss_first = inst->isshape_first;
      in_blas = true;
      tpush<STACK>(st, SENTINEL);
      ref = S.objects[inst->object].blas_root;
      continue;
    }
    const uint32_t cnt = ((ref >> 28) & 7u) + 1u;
    bool done = false;
    for (uint32_t k = 0; k < cnt && !done; ++k)
      done = tr.hit(S.tris[first + k], first + k, iss_first, tmax) && any_hit;
    if (done) break;
    alive = tpop<STACK>(st, ref);
  }
  return tr.result();
}

// Rays of a work list from memory (the renderer's)
template <int STACK>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_trace(DScene S, const uint32_t* __restrict__ list, const unsigned* __restrict__ count_ptr,
        const RayRec* __restrict__ rays, HitRec* __restrict__ hits, TOvf ovf) {
  __shared__ uint32_t lds_stack[STACK * BLOCK];
  __shared__ Node4 lds_top[TOP_NODES];
  const uint32_t count = *count_ptr;
  if (blockIdx.x * BLOCK >= count) return;  // whole blocks only: the staging syncs
  for (uint32_t i = threadIdx.x; i < S.ntop; i += BLOCK) lds_top[i] = S.top[i];
  __syncthreads();
  const uint32_t q = blockIdx.x * BLOCK + threadIdx.x;
  if (q >= count) return;
  const uint32_t slot = slot_of(list, q);
  const RayRec r = rays[slot];
  hits[slot] = trace_lane<Tracer64, STACK>(S, nullptr, r, q, lds_stack, lds_top, ovf);
}

// -------------------------------------------------------------------------
// TLAS refit for moved instances (the reference rebuilds its scene views on
// every solve, src/ssol_scene.c:346-433): the 4-wide TLAS keeps its
// topology and takes the world boxes of the instances' new frames, level by
// level from the deepest, in one workgroup; its LDS-staged copy of the top
// levels follows. *cost = sum over the TLAS's child boxes of their surface
// areas (x*y + y*z + z*x), the quality measure the host compares with the
// tree's at build time.
// -------------------------------------------------------------------------
constexpr int REFIT_THREADS = 1024;

// World box of instance ii: the 8 corners of its object's box under the
// instance transform, in FP64 and in the order of the host's TLAS build,
// rounded to FP32, widened by 2e-6 of its largest coordinate + 1e-6 (an
// empty object gets the degenerate box at the origin, widened alike)
__device__ void instance_world_box(const ssolh_instance& in, const float* ob, float lo[3],
                                   float hi[3]) {
  for (int k = 0; k < 3; ++k) { lo[k] = FLT_MAX; hi[k] = -FLT_MAX; }
  if (ob[0] > ob[3]) {
    for (int k = 0; k < 3; ++k) lo[k] = hi[k] = 0.f;
  } else {
    for (int c = 0; c < 8; ++c) {
      const double p[3] = {(double)((c & 1) ? ob[3] : ob[0]), (double)((c & 2) ? ob[4] : ob[1]),
                           (double)((c & 4) ? ob[5] : ob[2])};
      for (int k = 0; k < 3; ++k) {
        const double w = __dadd_rn(__dadd_rn(__dadd_rn(__dmul_rn(in.transform[k], p[0]),
                                                       __dmul_rn(in.transform[3 + k], p[1])),
                                             __dmul_rn(in.transform[6 + k], p[2])),
                                   in.transform[9 + k]);
        lo[k] = fminf(lo[k], (float)w);
        hi[k] = fmaxf(hi[k], (float)w);
      }
    }
  }
  float m = 0.f;
  for (int k = 0; k < 3; ++k) m = fmaxf(m, fmaxf(fabsf(lo[k]), fabsf(hi[k])));
  const float e = __fadd_rn(__fmul_rn(m, 2e-6f), 1e-6f);
  for (int k = 0; k < 3; ++k) { lo[k] = __fsub_rn(lo[k], e); hi[k] = __fadd_rn(hi[k], e); }
}

__global__ void __launch_bounds__(REFIT_THREADS)
k_tlas_refit(const ssolh_instance* __restrict__ insts, const uint32_t* __restrict__ tlas_inst,
             const float* __restrict__ obj_box, Node4* nodes, const uint32_t* __restrict__ order,
             const uint32_t* __restrict__ level_end, uint32_t nlevels, Node4* top,
             const uint32_t* __restrict__ top_src, uint32_t ntop, double* cost) {
  __shared__ double part[REFIT_THREADS];
  double acc = 0;
  uint32_t begin = 0;
  for (uint32_t l = 0; l < nlevels; ++l) {
    const uint32_t end = level_end[l];
    for (uint32_t i = begin + threadIdx.x; i < end; i += REFIT_THREADS) {
      Node4& n = nodes[order[i]];
      for (int c = 0; c < 4; ++c) {
        const uint32_t ref = n.child[c];
        if (ref == EMPTY4) continue;
        float lo[3], hi[3];
        if (ref & LEAF) {
          const ssolh_instance& in = insts[tlas_inst[ref & 0x0FFFFFFFu]];
          instance_world_box(in, obj_box + 6 * (size_t)in.object, lo, hi);
        } else {
          const Node4& m = nodes[ref];
          for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(fminf(m.box[a][0][0], m.box[a][0][1]), fminf(m.box[a][0][2], m.box[a][0][3]));
            hi[a] = fmaxf(fmaxf(m.box[a][1][0], m.box[a][1][1]), fmaxf(m.box[a][1][2], m.box[a][1][3]));
          }
        }
        for (int a = 0; a < 3; ++a) {
          n.box[a][0][c] = lo[a];
          n.box[a][1][c] = hi[a];
        }
        const double x = (double)hi[0] - lo[0], y = (double)hi[1] - lo[1],
                     z = (double)hi[2] - lo[2];
        acc += x * y + y * z + z * x;
      }
    }
    begin = end;
    __syncthreads();  // the next level reads this one's boxes
  }
  for (uint32_t i = threadIdx.x; i < ntop; i += REFIT_THREADS)
    for (int a = 0; a < 3; ++a)
      for (int sd = 0; sd < 2; ++sd)
        for (int c = 0; c < 4; ++c) top[i].box[a][sd][c] = nodes[top_src[i]].box[a][sd][c];
  part[threadIdx.x] = acc;
  __syncthreads();
  for (uint32_t w = REFIT_THREADS / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *cost = part[0];
}

// -------------------------------------------------------------------------
// TLAS build on the GPU (linear BVH, T. Karras, "Maximizing parallelism in
// the construction of BVHs, octrees, and k-d trees", HPG 2012): when moved
// instances have made a refit tree too loose, the TLAS is built anew over
// the instances' new world boxes without the host. Keys: 30-bit Morton codes
// of the box centres in the centres' bounds (ties broken by sorted position);
// a radix sort of (key, instance); the binary radix tree; boxes bottom-up;
// every BVH2 node at even depth becomes a 4-wide node over its children and
// grandchildren. Two single-workgroup kernels around the sort: the TLAS of a
// field holds tens of thousands of instances at most, which one workgroup
// handles in microseconds.
// -------------------------------------------------------------------------
constexpr int LBVH_THREADS = 1024;
constexpr int LBVH_MAX_LEVELS = 66;  // 4-wide levels of a tree of 30-bit keys + 32-bit ties

struct LbvhResult {
  uint32_t nodes4;  // 4-wide nodes written
  uint32_t depth4;  // deepest 4-wide level (root 0)
  uint32_t ntop;    // nodes of the LDS copy
  uint32_t pad;
  double cost;      // summed child-box surface area
};

__device__ __forceinline__ uint32_t spread10(uint32_t x) {
  x &= 0x3FFu;
  x = (x | (x << 16)) & 0x030000FFu;
  x = (x | (x << 8)) & 0x0300F00Fu;
  x = (x | (x << 4)) & 0x030C30C3u;
  x = (x | (x << 2)) & 0x09249249u;
  return x;
}

__global__ void __launch_bounds__(LBVH_THREADS)
k_lbvh_keys(const ssolh_instance* __restrict__ insts, const float* __restrict__ obj_box,
            uint32_t n, float* __restrict__ lbox, uint32_t* __restrict__ key,
            uint32_t* __restrict__ val) {
  __shared__ float red[6][LBVH_THREADS];
  float mn[3] = {FLT_MAX, FLT_MAX, FLT_MAX}, mx[3] = {-FLT_MAX, -FLT_MAX, -FLT_MAX};
  for (uint32_t i = threadIdx.x; i < n; i += LBVH_THREADS) {
    float lo[3], hi[3];
    instance_world_box(insts[i], obj_box + 6 * (size_t)insts[i].object, lo, hi);
    for (int a = 0; a < 3; ++a) {
      lbox[6 * (size_t)i + a] = lo[a];
      lbox[6 * (size_t)i + 3 + a] = hi[a];
      const float cen = 0.5f * (lo[a] + hi[a]);
      mn[a] = fminf(mn[a], cen);
      mx[a] = fmaxf(mx[a], cen);
    }
  }
  for (int a = 0; a < 3; ++a) { red[a][threadIdx.x] = mn[a]; red[3 + a][threadIdx.x] = mx[a]; }
  __syncthreads();
  for (uint32_t w = LBVH_THREADS / 2; w > 0; w >>= 1) {
    if (threadIdx.x < w)
      for (int a = 0; a < 3; ++a) {
        red[a][threadIdx.x] = fminf(red[a][threadIdx.x], red[a][threadIdx.x + w]);
        red[3 + a][threadIdx.x] = fmaxf(red[3 + a][threadIdx.x], red[3 + a][threadIdx.x + w]);
      }
    __syncthreads();
  }
  float lo[3], sc[3];
  for (int a = 0; a < 3; ++a) {
    lo[a] = red[a][0];
    const float ext = red[3 + a][0] - red[a][0];
    sc[a] = ext > 0.f ? 1023.f / ext : 0.f;
  }
  for (uint32_t i = threadIdx.x; i < n; i += LBVH_THREADS) {
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
      const float cen = 0.5f * (lbox[6 * (size_t)i + a] + lbox[6 * (size_t)i + 3 + a]);
      q[a] = (uint32_t)fminf(fmaxf((cen - lo[a]) * sc[a], 0.f), 1023.f);
    }
    key[i] = (spread10(q[0]) << 2) | (spread10(q[1]) << 1) | spread10(q[2]);
    val[i] = i;
  }
}

// Common-prefix length of sorted keys i and j (-1 out of range; equal keys
// compare their positions)
__device__ __forceinline__ int lbvh_delta(const uint32_t* k, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  const uint32_t a = k[i], b = k[j];
  return a == b ? 32 + __clz(i ^ j) : __clz(a ^ b);
}

// Work arrays of the build: child pairs and parents of the binary tree
// (internal nodes 0..n-2, leaf i as n-1+i), arrival counters, internal
// boxes, depths, 4-wide indices and levels
struct LbvhWork {
  int2* child;
  int* parent;
  unsigned* flag;
  float* ibox;
  uint32_t* depth;
  uint32_t* idx4;
  uint32_t* dep4;
};

__device__ __forceinline__ void lbvh_box(const LbvhWork& w, const float* lbox,
                                         const uint32_t* sval, int n, int x, float b[6]) {
  const float* src = x < n - 1 ? w.ibox + 6 * (size_t)x : lbox + 6 * (size_t)sval[x - (n - 1)];
  for (int k = 0; k < 6; ++k) b[k] = __hip_atomic_load(src + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void __launch_bounds__(LBVH_THREADS)
k_lbvh_finish(uint32_t n, const uint32_t* __restrict__ skey, const uint32_t* __restrict__ sval,
              const float* __restrict__ lbox, LbvhWork w, Node4* tlas, uint32_t tlas_base,
              uint32_t* tlas_inst, uint32_t* order, uint32_t* level_end, Node4* top,
              uint32_t* top_src, LbvhResult* res) {
  __shared__ uint32_t s_scan[LBVH_THREADS];
  __shared__ uint32_t s_lvl[LBVH_MAX_LEVELS];
  __shared__ uint32_t s_cur[LBVH_MAX_LEVELS];
  __shared__ double s_cost[LBVH_THREADS];
  __shared__ uint32_t s_max;
  const int N = (int)n;
  const uint32_t tid = threadIdx.x;
  for (uint32_t i = tid; i < n; i += LBVH_THREADS) tlas_inst[i] = sval[i];
  if (N == 1) {
    // one instance: a root with one leaf
    if (tid == 0) {
      float b[6];
      for (int k = 0; k < 6; ++k) b[k] = lbox[6 * (size_t)sval[0] + k];
      Node4 o;
      for (int a = 0; a < 3; ++a)
        for (int c = 0; c < 4; ++c) {
          o.box[a][0][c] = c == 0 ? b[a] : INFINITY;
          o.box[a][1][c] = c == 0 ? b[3 + a] : -INFINITY;
        }
      for (int c = 0; c < 4; ++c) { o.child[c] = c == 0 ? LEAF : EMPTY4; o.pad[c] = 0; }
      tlas[0] = o;
      top[0] = o;
      top_src[0] = tlas_base;
      order[0] = tlas_base;
      level_end[0] = 1;
      const double x = (double)b[3] - b[0], y = (double)b[4] - b[1], z = (double)b[5] - b[2];
      *res = LbvhResult{1u, 0u, 1u, 0u, x * y + y * z + z * x};
    }
    return;
  }
  // binary radix tree
  for (uint32_t t = tid; t < n - 1; t += LBVH_THREADS) {
    const int i = (int)t;
    w.flag[i] = 0;
    const int d = lbvh_delta(skey, N, i, i + 1) - lbvh_delta(skey, N, i, i - 1) >= 0 ? 1 : -1;
    const int dmin = lbvh_delta(skey, N, i, i - d);
    int lmax = 2;
    while (lbvh_delta(skey, N, i, i + lmax * d) > dmin) lmax *= 2;
    int l = 0;
    for (int s = lmax / 2; s >= 1; s /= 2)
      if (lbvh_delta(skey, N, i, i + (l + s) * d) > dmin) l += s;
    const int j = i + l * d;
    const int dnode = lbvh_delta(skey, N, i, j);
    int sp = 0;
    for (int s = (l + 1) / 2;; s = (s + 1) / 2) {
      if (lbvh_delta(skey, N, i, i + (sp + s) * d) > dnode) sp += s;
      if (s == 1) break;
    }
    const int g = i + sp * d + min(d, 0);
    const int left = min(i, j) == g ? N - 1 + g : g;
    const int right = max(i, j) == g + 1 ? N - 1 + g + 1 : g + 1;
    w.child[i] = make_int2(left, right);
    w.parent[left] = i;
    w.parent[right] = i;
  }
  if (tid == 0) w.parent[0] = -1;
  __threadfence();
  __syncthreads();
  // boxes bottom-up: the second of two children to arrive at a node forms it
  for (uint32_t t = tid; t < n; t += LBVH_THREADS) {
    int node = w.parent[N - 1 + (int)t];
    while (node >= 0) {
      const unsigned prev =
          __hip_atomic_fetch_add(w.flag + node, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
      if (prev == 0) break;
      float a[6], b[6];
      lbvh_box(w, lbox, sval, N, w.child[node].x, a);
      lbvh_box(w, lbox, sval, N, w.child[node].y, b);
      float* dst = w.ibox + 6 * (size_t)node;
      for (int k = 0; k < 3; ++k) {
        __hip_atomic_store(dst + k, fminf(a[k], b[k]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(dst + 3 + k, fmaxf(a[3 + k], b[3 + k]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
      }
      node = w.parent[node];
    }
  }
  __threadfence();
  __syncthreads();
  // depths, then the 4-wide index of every even-depth node (block scan)
  for (uint32_t t = tid; t < n - 1; t += LBVH_THREADS) {
    uint32_t dd = 0;
    for (int p = w.parent[t]; p >= 0; p = w.parent[p]) ++dd;
    w.depth[t] = dd;
  }
  if (tid == 0) s_max = 0;
  __threadfence();
  __syncthreads();
  uint32_t run = 0;
  for (uint32_t base = 0; base < n - 1; base += LBVH_THREADS) {
    const uint32_t t = base + tid;
    const uint32_t v = (t < n - 1 && !(w.depth[t] & 1u)) ? 1u : 0u;
    s_scan[tid] = v;
    __syncthreads();
    for (uint32_t off = 1; off < LBVH_THREADS; off <<= 1) {
      const uint32_t x = tid >= off ? s_scan[tid - off] : 0u;
      __syncthreads();
      s_scan[tid] += x;
      __syncthreads();
    }
    if (t < n - 1) w.idx4[t] = run + s_scan[tid] - v;
    run += s_scan[LBVH_THREADS - 1];
    __syncthreads();
  }
  __threadfence();
  __syncthreads();
  // the 4-wide nodes
  double acc = 0;
  for (uint32_t t = tid; t < n - 1; t += LBVH_THREADS) {
    if (w.depth[t] & 1u) continue;
    int ent[4], ne = 0;
    const int2 c2 = w.child[t];
    for (int side = 0; side < 2; ++side) {
      const int c = side ? c2.y : c2.x;
      if (c >= N - 1) {
        ent[ne++] = c;
      } else {
        ent[ne++] = w.child[c].x;
        ent[ne++] = w.child[c].y;
      }
    }
    Node4 o;
    for (int e = 0; e < 4; ++e) {
      if (e >= ne) {
        for (int a = 0; a < 3; ++a) { o.box[a][0][e] = INFINITY; o.box[a][1][e] = -INFINITY; }
        o.child[e] = EMPTY4;
        o.pad[e] = 0;
        continue;
      }
      float b[6];
      lbvh_box(w, lbox, sval, N, ent[e], b);
      for (int a = 0; a < 3; ++a) { o.box[a][0][e] = b[a]; o.box[a][1][e] = b[3 + a]; }
      o.child[e] = ent[e] >= N - 1 ? (LEAF | (uint32_t)(ent[e] - (N - 1)))
                                   : tlas_base + w.idx4[ent[e]];
      o.pad[e] = 0;
      const double x = (double)b[3] - b[0], y = (double)b[4] - b[1], z = (double)b[5] - b[2];
      acc += x * y + y * z + z * x;
    }
    const uint32_t k = w.idx4[t];
    tlas[k] = o;
    const uint32_t d4 = w.depth[t] / 2;
    w.dep4[k] = d4;
    atomicMax(&s_max, d4);
  }
  s_cost[tid] = acc;
  __threadfence();
  __syncthreads();
  for (uint32_t s = LBVH_THREADS / 2; s > 0; s >>= 1) {
    if (tid < s) s_cost[tid] += s_cost[tid + s];
    __syncthreads();
  }
  // levels for the refit, deepest first
  const uint32_t n4 = run, dmax = s_max;
  for (uint32_t l = tid; l < LBVH_MAX_LEVELS; l += LBVH_THREADS) s_lvl[l] = 0;
  __syncthreads();
  for (uint32_t k = tid; k < n4; k += LBVH_THREADS) atomicAdd(&s_lvl[w.dep4[k]], 1u);
  __syncthreads();
  if (tid == 0) {
    uint32_t acc_l = 0;
    for (int l = (int)dmax; l >= 0; --l) {
      s_cur[l] = acc_l;
      acc_l += s_lvl[l];
      level_end[dmax - l] = acc_l;
    }
  }
  __syncthreads();
  for (uint32_t k = tid; k < n4; k += LBVH_THREADS)
    order[atomicAdd(&s_cur[w.dep4[k]], 1u)] = tlas_base + k;
  __threadfence();
  __syncthreads();
  // the LDS copy of the top levels, breadth first
  if (tid == 0) {
    uint32_t q[TOP_NODES];
    uint32_t nq = 1;
    q[0] = tlas_base;
    for (uint32_t h = 0; h < nq && nq < (uint32_t)TOP_NODES; ++h)
      for (int c = 0; c < 4 && nq < (uint32_t)TOP_NODES; ++c) {
        const uint32_t ch = tlas[q[h] - tlas_base].child[c];
        if (!(ch & LEAF)) q[nq++] = ch;
      }
    for (uint32_t h = 0; h < nq; ++h) {
      Node4 o = tlas[q[h] - tlas_base];
      for (int c = 0; c < 4; ++c) {
        if (o.child[c] & LEAF) continue;
        for (uint32_t g = 0; g < nq; ++g)
          if (q[g] == o.child[c]) { o.child[c] = TOP_REF | g; break; }
      }
      top[h] = o;
      top_src[h] = q[h];
    }
    *res = LbvhResult{n4, dmax, nq, 0u, s_cost[0]};
  }
}

// -------------------------------------------------------------------------
// Paths
// -------------------------------------------------------------------------
__device__ uint32_t start_medium(const DScene& S, const ssolh_material& m, uint32_t side) {
  if (m.type == SSOLH_MTL_DIELECTRIC || m.type == SSOLH_MTL_THIN_DIELECTRIC)
    return (uint32_t)(side == SSOL_FRONT_ ? m.medium_in : m.medium_out);
  return S.air;
}

__device__ void flush_sampled_count(bool has, int samp_slot, const Tallies& T) {
  const uint64_t key = has ? (uint64_t)samp_slot : 0;
  const uint64_t mask = __ballot(has);
  if (!mask) return;
  unsigned long long* base = T.samp_count + (size_t)(blockIdx.x & T.mask_s) * T.nsamp;
  const int leader = __ffsll((unsigned long long)mask) - 1;
  const uint64_t lkey = __shfl(key, leader, 64);
  const bool match = has && key == lkey;
  const uint64_t mm = __ballot(match);
  if ((int)lane_id() == leader) atomicAdd(base + lkey, (unsigned long long)__popcll(mm));
  if (has && !match) atomicAdd(base + key, 1ull);
}

enum { FIN_NONE = 0, FIN_DONE = 1, FIN_KILLED = 2, FIN_FAILED = 3 };

#include "ssolh_fp32.hpp"
#include "ssolh_path.hpp"

#include "ssolh_render.hpp"

// Slot order of the first realisations by (sun, start instance). The
// realisations are drawn at random over the field, so in realisation order a
// wave's rays start on unrelated heliostats; placed by start instance, a
// wave's rays leave neighbouring points in like directions (coherent
// traversal) and its finished paths share tally keys (wave-reduced atomics).
// The sun (job) comes first so a batch keeps each wave on one sun, as the
// realisation order did. k_start_keys draws each realisation's start
// instance exactly as generate does; a stable radix sort of (key, index)
// pairs then gives the order, realisations of one key in index order.
template <bool FP32>
__device__ __forceinline__ uint32_t start_key(const DScene& S, const SolveParams& prm,
                                              uint64_t path, uint32_t ninst) {
  // S.stris[alias_pick(...)].instance (alias_pick32 for FP32) from one
  // StartAlias load
  uint32_t inst;
  if (FP32) {
    PathRng32 rng;
    rng.init(prm.key, prm.counter + path, 0);
    const float u0 = rng.next(), uc = rng.next();
    uint32_t i = (uint32_t)(u0 * (float)S.nstris);
    if (i >= S.nstris) i = S.nstris - 1;
    const StartAlias e = S.salias[i];
    inst = (double)uc < e.prob ? e.inst : e.inst_alias;
  } else {
    PathRng rng;
    rng.init(prm.key, prm.counter + path, 0);
    const double x = rng.next() * (double)S.nstris;
    uint32_t i = (uint32_t)x;
    if (i >= S.nstris) i = S.nstris - 1;
    const StartAlias e = S.salias[i];
    inst = (x - (double)i) < e.prob ? e.inst : e.inst_alias;
  }
  return job_of(prm, path) * ninst + inst;
}

// The start key of realisation first + i
template <bool FP32>
struct StartKeyOf {
  DScene S;
  SolveParams prm;
  uint64_t first;
  uint32_t ninst;
  __device__ uint32_t operator()(uint32_t i) const {
    return start_key<FP32>(S, prm, first + i, ninst);
  }
};

// The start keys of the wavefront's realisations and their indices, for the
// radix sort
template <bool FP32>
__global__ void __launch_bounds__(256)
k_start_keys(StartKeyOf<FP32> key_of, uint32_t count, uint32_t* __restrict__ key,
             uint32_t* __restrict__ idx) {
  const uint32_t q = blockIdx.x * 256 + threadIdx.x;
  if (q >= count) return;
  key[q] = key_of(q);
  idx[q] = q;
}

// Bits of the start keys (below nkeys) and the sort's work bytes for count
// realisations
uint32_t start_key_bits(uint64_t nkeys) {
  uint32_t bits = 1;
  while (bits < 32 && (uint64_t(1) << bits) < nkeys) ++bits;
  return bits;
}

hipError_t start_sort_bytes(uint32_t count, uint32_t bits, hipStream_t stream, size_t& bytes) {
  bytes = 0;
  return hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const uint32_t*)nullptr,
                                            (uint32_t*)nullptr, (const uint32_t*)nullptr,
                                            (uint32_t*)nullptr, (int)count, 0, (int)bits, stream);
}

// Sums of the stripes of every tally, in one launch, and the solve's
// counters beside them. A block takes a tile of 1024 / rows consecutive
// elements of one tally, its rows each every rows-th stripe, and adds the rows
// up in LDS: a tally of 40 elements in 256 stripes (one receiver) takes 16
// loads in a row instead of 256, and the launch as long as the largest tally
// takes to read (field of 100 paraboloids, 36 MB of stripes: six launches of
// together 507 us, one thread per element -> one of 25 us).
constexpr int FOLD_THREADS = 1024, FOLD_ROWS = 16;
struct FoldPart {
  const void* src;     // [stripes][n], doubles or (whole) 64-bit counts
  void* dst;           // [n], may be stripe 0 of src
  uint64_t n;
  uint32_t stripes;    // a power of two
  uint32_t first;      // first block of the part
  uint32_t whole;
};
constexpr int FOLD_PARTS = 6;
struct FoldArgs {
  FoldPart part[FOLD_PARTS];
  const Counters* C;
  Counters* C_out;
};

// Adds v to the sum s + e; e collects the rounding errors of s (Knuth's
// two-sum), so the fold adds none of its own to a tally: variances come from
// the difference of two of them
__device__ __forceinline__ void add_to(double& s, double& e, double v) {
  const double t = s + v, b = t - s;
  e += (s - (t - b)) + (v - b);
  s = t;
}

__device__ __forceinline__ void fold_tile(const FoldPart& p, uint64_t tile, double* lds) {
  const uint32_t rows = min(p.stripes, (uint32_t)FOLD_ROWS), cols = FOLD_THREADS / rows;
  const uint32_t row = threadIdx.x / cols, col = threadIdx.x % cols;
  const uint64_t i = tile * cols + col;
  double s = 0, e = 0;
  if (i < p.n)
    for (uint32_t k = row; k < p.stripes; k += rows) add_to(s, e, ((const double*)p.src)[k * p.n + i]);
  lds[threadIdx.x] = s;
  lds[FOLD_THREADS + threadIdx.x] = e;
  __syncthreads();
  if (row == 0 && i < p.n) {
    for (uint32_t k = 1; k < rows; ++k) {
      add_to(s, e, lds[k * cols + col]);
      e += lds[FOLD_THREADS + k * cols + col];
    }
    ((double*)p.dst)[i] = s + e;
  }
}

// The same for counts, which few tallies have: one thread per element
__device__ __forceinline__ void fold_counts(const FoldPart& p, uint64_t tile) {
  const uint64_t i = tile * FOLD_THREADS + threadIdx.x;
  if (i >= p.n) return;
  unsigned long long s = 0;
#pragma unroll 8
  for (uint32_t k = 0; k < p.stripes; ++k) s += ((const unsigned long long*)p.src)[k * p.n + i];
  ((unsigned long long*)p.dst)[i] = s;
}

// The receiver tally: a realisation starts on one sampled instance, so it is
// the folded sampled x receiver tally summed over the instances. n: doubles
// per instance, gridDim.y shares of the instances; rcv is zero before.
__global__ void __launch_bounds__(FOLD_THREADS)
k_fold_rcv(const double* __restrict__ sxr, uint64_t n, uint32_t nsamp, double* rcv) {
  __shared__ double lds[2 * FOLD_THREADS];
  constexpr uint32_t cols = FOLD_THREADS / FOLD_ROWS;
  const uint32_t row = threadIdx.x / cols, col = threadIdx.x % cols;
  const uint64_t i = (uint64_t)blockIdx.x * cols + col;
  double s = 0, e = 0;
  if (i < n)
    for (uint32_t k = blockIdx.y * FOLD_ROWS + row; k < nsamp; k += gridDim.y * FOLD_ROWS)
      add_to(s, e, sxr[k * n + i]);
  lds[threadIdx.x] = s;
  lds[FOLD_THREADS + threadIdx.x] = e;
  __syncthreads();
  if (row || i >= n) return;
  for (uint32_t k = 1; k < FOLD_ROWS; ++k) {
    add_to(s, e, lds[k * cols + col]);
    e += lds[FOLD_THREADS + k * cols + col];
  }
  atomic_add(rcv + i, s + e);
}

__global__ void __launch_bounds__(FOLD_THREADS) k_fold(FoldArgs a) {
  __shared__ double lds[2 * FOLD_THREADS];
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.C_out = *a.C;
  int k = FOLD_PARTS - 1;
  while (k > 0 && blockIdx.x < a.part[k].first) --k;
  const FoldPart& p = a.part[k];
  if (p.whole) fold_counts(p, blockIdx.x - p.first);
  else fold_tile(p, blockIdx.x - p.first, lds);
}

// -------------------------------------------------------------------------
// Deterministic test kernels
// -------------------------------------------------------------------------
__global__ void k_test_quadric(int quadric, double4 qp, uint32_t n, const double* org,
                               const double* dir, const double* hint, double* t, double* nrm) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double p[4] = {qp.x, qp.y, qp.z, qp.w};
  double tt;
  d3 g;
  if (quadric_hit(quadric, p, ld3(org + 3 * i), ld3(dir + 3 * i), hint[i], tt, g)) {
    t[i] = tt;
    nrm[3 * i] = g.x; nrm[3 * i + 1] = g.y; nrm[3 * i + 2] = g.z;
  } else {
    t[i] = INFINITY;
    nrm[3 * i] = nrm[3 * i + 1] = nrm[3 * i + 2] = 0;
  }
}

// wave_totals of four copies of a wave's 64 inputs: each row of 16 lanes
// returns the total of one (blocks of 64 threads: every lane active)
__global__ void __launch_bounds__(64) k_test_wave_sum(const double* in, double* out) {
  const double x = in[blockIdx.x * 64 + threadIdx.x];
  const double v[4] = {x, x, x, x};
  const double s = __shfl(wave_totals<4>(v), (int)(threadIdx.x & 48u), 64);
  out[blockIdx.x * 64 + threadIdx.x] = s;
}

// Uniforms from an array (0.5 once it is exhausted), for fixed-input tests
struct ArrayRng {
  const double* u;
  uint32_t n, i;
  __device__ double next() { return i < n ? u[i++] : 0.5; }
};

__global__ void k_test_sun(ssolh_sun sun, uint32_t n, const double* u, uint32_t nu,
                           double* out, uint32_t* used) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  ArrayRng rng{u + (size_t)i * nu, nu, 0};
  const d3 d = sample_sun(sun, rng);
  out[3 * i] = d.x; out[3 * i + 1] = d.y; out[3 * i + 2] = d.z;
  used[i] = rng.i;
}

__global__ void k_test_bsdf(ssolh_material m, double4 eta, uint32_t n, const double* wi,
                            const double* nrm, const double* u, uint32_t nu, double* wo,
                            double* w, int* lobe) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  ArrayRng rng{u + (size_t)i * nu, nu, 0};
  d3 o;
  int l;
  w[i] = bsdf_sample(m, eta.x, eta.y, eta.z, eta.w, ld3(wi + 3 * i), ld3(nrm + 3 * i), rng, o, l);
  wo[3 * i] = o.x; wo[3 * i + 1] = o.y; wo[3 * i + 2] = o.z;
  lobe[i] = l;
}

// Plain device-to-device copy: reads and writes exactly 16 B per element.
// Used to calibrate the HBM byte counters and as the achievable-bandwidth
// yardstick for the path-tracing kernels.
__global__ void __launch_bounds__(256) k_copy(const uint4* __restrict__ a, uint4* __restrict__ b,
                                             size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    b[i] = a[i];
}

__global__ void k_test_threefry(uint32_t n, const uint64_t* ctr, const uint64_t* key, uint64_t* out) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  threefry4x64_20(ctr + 4 * i, key + 4 * i, out + 4 * i);
}

}  // namespace

// -------------------------------------------------------------------------
// Host side
// -------------------------------------------------------------------------
struct DevBuf {
  void* p = nullptr;
  size_t n = 0;
};

// Device memory of ssolh_solve_noalloc: every buffer of its solve (path
// state, rays, hits, work lists, scan arrays, counters, tallies) is carved
// from this array, which each GPU holds from the library's load to the end
// of the process. Host code never names it as an address: each device's own
// copy is reached through the pointer hipGetSymbolAddress returns with that
// device current (kept per device by ssolh_create).
constexpr size_t SCRATCH_BYTES = size_t(64) << 20;
// folded tallies of up to so many bytes are kept in pinned host memory
constexpr size_t STAGE_MAX = size_t(64) << 20;
// records of the per-primitive log (84 B each plus 12 B of sort arrays)
constexpr uint64_t LOG_MAX_RECORDS = uint64_t(1) << 27;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mu;
void* g_scratch[MAX_DEVICES] = {};

struct ssolh_context {
  int device = 0;
  hipStream_t stream = nullptr;
  void* scratch = nullptr;  // this device's copy of the scratch array
  hipEvent_t ev[4] = {};
  // scene
  std::vector<DevBuf> scene_bufs;
  DScene scn{};
  bool has_scene = false;
  uint32_t nrcv = 0, nsamp = 0;
  uint64_t nprim = 0;
  uint32_t stack_depth = MAX_STACK;  // traversal stack bound of the scene's 4-wide nodes
  uint32_t lds_stack_cap = 0;        // 16, 24 or 32: LDS stack entries at most (0: MAX_STACK)
  bool may_pend = false;  // a receiver may let light pass: paths keep pending entries
  float slack_scale = SLAB_SLACK;     // box-test slack of the scenes uploaded next
  // TLAS refit of moved instances: per-object boxes, the TLAS nodes by level
  // (deepest first) and the top copy's sources, all in scene_bufs
  const float* obj_box = nullptr;
  const uint32_t* tlas_order = nullptr;
  const uint32_t* tlas_level_end = nullptr;
  uint32_t tlas_levels = 0;
  const uint32_t* top_src = nullptr;
  double* refit_cost = nullptr;
  double tlas_cost0 = 0;              // the TLAS's cost as built
  std::vector<uint32_t> inst_object;  // object of each instance as uploaded
  uint32_t ninst_sshapes = 0;
  uint32_t n_uploads = 0, n_refits = 0, n_builds = 0;
  // GPU TLAS builds: the TLAS's region of `nodes` (first index, capacity),
  // the BLASes' part of the stack bound, the build's work buffer
  uint32_t tlas_base = 0, tlas_cap = 0, blas_pb = 0;
  DevBuf lbvh;
  DevBuf render;  // renderer work buffer (ssolh_render)
  // solve buffers
  DevBuf start_sort;         // work bytes of the start-key sort
  DevBuf queue[2], list;     // paths in flight, their list
  DevBuf pend;               // pending entries
  DevBuf tallies;            // counters, group counts, striped tallies, group offsets
  DevBuf jobs, trace_ovf;
  // per-primitive log: keys, sorted keys, indices, sorted indices, values,
  // count, sort work (Tallies::log_*); log_sort, log_sidx, log_skey and
  // log_idx within it, log_sort_bytes of sort work
  DevBuf plog;
  void* log_sort = nullptr;
  size_t log_sort_bytes = 0;
  uint32_t *log_ckey = nullptr, *log_skey = nullptr, *log_idx = nullptr, *log_sidx = nullptr;
  uint32_t log_key_bits = 1;
  uint32_t log_cap_test = 0;          // ssolh_test_prim_log's cap (0: the default)
  uint32_t log_flushes = 0;           // the last solve's sorted reductions
  uint64_t log_overflowed = 0;        // and the entries it sent to the atomics
  DevBuf adj_state, adj_in, adj_grad;
  DevBuf trk_vtx, trk_type, trk_seq, trk_count, trk_pos;
  uint64_t trk_paths = 0;           // realisations of the last tracked solve
  unsigned long long trk_nvtx = 0;  // vertices it produced
  uint64_t trk_cap = 0;
  uint32_t ninstances = 0;
  uint32_t njobs = 1;
  const ShapeQ* shapeq = nullptr;  // per shape, in scene_bufs
  Tallies T{};
  // folded tallies: counters, then the tallies one after the other, copied to
  // `stage` (pinned) by each solve when they take at most STAGE_MAX bytes;
  // F: where the folded tallies are on the device
  DevBuf folded;
  Tallies F{};
  void* stage = nullptr;
  size_t stage_bytes = 0;
  bool staged = false;
  // last solve
  Counters last{};
  uint64_t segments = 0;
  double kernel_ms = 0, trace_ms = 0, shade_ms = 0;
  uint32_t iterations = 0;
  uint32_t wavefronts = 0;    // of the last solve
  uint32_t refilled = 0;
};

namespace {

int dev_alloc(DevBuf& b, size_t bytes) {
  if (b.n >= bytes && b.p) return 0;
  if (b.p) { (void)hipFree(b.p); b.p = nullptr; b.n = 0; }
  if (!bytes) bytes = 16;
  HIP_TRY(hipMalloc(&b.p, bytes));
  b.n = bytes;
  return 0;
}

// A solve's buffers carved from caller-independent device memory that is
// never freed (the library's static scratch array): each take advances a
// cursor, 256-byte aligned; nothing is allocated or released.
struct Arena {
  char* base;
  size_t size;
  size_t used;
};

int arena_take(Arena& a, DevBuf& b, size_t bytes) {
  if (!bytes) bytes = 16;
  // taken earlier in this solve and large enough (the start-instance
  // histogram of each chunk)
  if (b.p && b.n >= bytes && (char*)b.p >= a.base && (char*)b.p < a.base + a.size) return 0;
  const size_t off = (a.used + 255) & ~size_t(255);
  if (off > a.size || bytes > a.size - off) {
    set_err("ssolh_solve_noalloc: the solve needs more than the %zu bytes of the scratch array "
            "(%zu in use, %zu more asked)", a.size, off, bytes);
    return SSOLH_ERR_LIMIT;
  }
  b.p = a.base + off;
  b.n = bytes;
  a.used = off + bytes;
  return 0;
}

template <typename T>
int upload(ssolh_context* c, const T* src, size_t count, const T** dst) {
  DevBuf b;
  const size_t bytes = count * sizeof(T);
  int r = dev_alloc(b, bytes ? bytes : 16);
  if (r) return r;
  if (bytes) HIP_TRY(hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, c->stream));
  c->scene_bufs.push_back(b);
  *dst = (const T*)b.p;
  return 0;
}

void free_scene(ssolh_context* c) {
  for (auto& b : c->scene_bufs) if (b.p) (void)hipFree(b.p);
  c->scene_bufs.clear();
  c->has_scene = false;
}

// Inverse of a column-major 3x3 matrix; false when singular
bool inv3(const double* m, double* o) {
  const double a = m[0], b = m[3], cc = m[6], d = m[1], e = m[4], f = m[7], g = m[2], h = m[5],
               i = m[8];
  const double A = e * i - f * h, B = -(d * i - f * g), C = d * h - e * g;
  const double det = a * A + b * B + cc * C;
  if (det == 0 || !std::isfinite(det)) return false;
  const double r = 1.0 / det;
  // rows of the inverse (row-major r0..r2) stored column-major
  const double inv[3][3] = {{A * r, -(b * i - cc * h) * r, (b * f - cc * e) * r},
                            {B * r, (a * i - cc * g) * r, -(a * f - cc * d) * r},
                            {C * r, -(a * h - b * g) * r, (a * e - b * d) * r}};
  for (int row = 0; row < 3; ++row)
    for (int col = 0; col < 3; ++col) o[col * 3 + row] = inv[row][col];
  return true;
}

// Per (instance, shaded shape) records of the hit path, from the flat scene
int build_iss(const ssolh_scene* s, std::vector<IssInfo>& out) {
  out.assign(s->ninst_sshapes, IssInfo{});
  for (uint32_t i = 0; i < s->ninstances; ++i) {
    const ssolh_instance& in = s->instances[i];
    if (in.object >= s->nobjects) return -1;
    const ssolh_object& o = s->objects[in.object];
    for (uint32_t k = 0; k < o.sshape_count; ++k) {
      const uint64_t g = (uint64_t)in.isshape_first + k;
      const uint32_t ss = o.sshape_first + k;
      if (g >= s->ninst_sshapes || ss >= s->nsshapes) return -1;
      const ssolh_sshape& sh = s->sshapes[ss];
      if (sh.shape >= s->nshapes || sh.mtl_front >= s->nmaterials || sh.mtl_back >= s->nmaterials)
        return -1;
      IssInfo& d = out[g];
      d.inst = i;
      d.shape = sh.shape;
      d.mtl_front = sh.mtl_front;
      d.mtl_back = sh.mtl_back;
      d.receiver = in.receiver;
      d.receiver_mask = in.receiver_mask;
      d.shape_type = (uint32_t)s->shapes[sh.shape].type;
      d.obj_flags = o.flags | (o.sshape_count == 1 ? OBJ_ONE_SHAPE : 0u);
      d.prim_tally = s->inst_sshapes[g].prim_tally;
    }
  }
  return 0;
}

// LDS stack entries per lane of the trace kernel: the smallest of 16, 24, 32
// that holds the scene's bound (the more blocks then share a CU), within the
// context's cap; the rest of the bound goes to the overflow array
uint32_t trace_lds_stack(const ssolh_context* c) {
  uint32_t e = c->stack_depth <= 16 ? 16 : c->stack_depth <= 24 ? 24 : (uint32_t)MAX_STACK;
  if (c->lds_stack_cap && c->lds_stack_cap < e) e = c->lds_stack_cap;
  return e;
}

// BVH2 -> 4-wide nodes. A 4-wide node takes the children of a BVH2 node
// and, while it holds fewer than four and one of them is an inner node,
// replaces the inner child of largest box area by that child's children;
// each inner child left becomes a 4-wide node of its own. pb[i]: the most
// stack entries a descent from node i pushes (each visited node pushes all
// but one of the children a ray crosses).
struct Collapse4 {
  struct Ent {
    float lo[3], hi[3];
    uint32_t child, count;  // count 0: inner BVH2 node `child`
  };
  const ssolh_bvh_node* in;
  uint32_t nin;
  std::vector<Node4> out;
  std::vector<uint32_t> pb;
  int err = 0;
  char msg[160] = "";

  Collapse4(const ssolh_bvh_node* nodes, uint32_t n) : in(nodes), nin(n) {}

  static float area(const Ent& e) {
    const float x = e.hi[0] - e.lo[0], y = e.hi[1] - e.lo[1], z = e.hi[2] - e.lo[2];
    return x * y + y * z + z * x;
  }
  void fail(int code, const char* fmt, uint32_t a, uint32_t b) {
    if (!err) snprintf(msg, sizeof(msg), fmt, a, b);
    err = code;
  }
  // children of BVH2 node b appended to e[n..]
  void take(uint32_t b, Ent* e, int& n) {
    const ssolh_bvh_node& m = in[b];
    for (int k = 0; k < 2; ++k) {
      if (m.count[k] == SSOLH_BVH_EMPTY) continue;
      Ent& x = e[n++];
      for (int a = 0; a < 3; ++a) { x.lo[a] = m.lo[k][a]; x.hi[a] = m.hi[k][a]; }
      x.child = m.child[k];
      x.count = m.count[k];
    }
  }
  uint32_t root(uint32_t b) { return node(b, 0); }
  uint32_t node(uint32_t b, int depth) {
    if (b >= nin) { fail(SSOLH_ERR_ARG, "BVH node %u out of %u nodes", b, nin); return 0; }
    if (depth > 256) { fail(SSOLH_ERR_LIMIT, "BVH deeper than %u levels at node %u", 256, b); return 0; }
    Ent e[5];
    int n = 0;
    take(b, e, n);
    while (n < 4) {
      int best = -1;
      float ba = -1.f;
      for (int i = 0; i < n; ++i)
        if (e[i].count == 0 && area(e[i]) > ba) { ba = area(e[i]); best = i; }
      if (best < 0) break;
      const uint32_t b2 = e[best].child;
      if (b2 >= nin) { fail(SSOLH_ERR_ARG, "BVH child %u out of %u nodes", b2, nin); return 0; }
      e[best] = e[--n];
      take(b2, e, n);
    }
    const uint32_t me = (uint32_t)out.size();
    out.emplace_back();
    pb.push_back(0);
    uint32_t ref[4], deeper = 0;
    for (int i = 0; i < 4; ++i) {
      if (i >= n) { ref[i] = EMPTY4; continue; }
      if (e[i].count == 0) {
        ref[i] = node(e[i].child, depth + 1);
        if (err) return 0;
        deeper = std::max(deeper, pb[ref[i]]);
      } else {
        if (e[i].count > 8 || e[i].child >= (1u << 28)) {
          fail(SSOLH_ERR_LIMIT, "BVH leaf of %u items at %u (at most 8 below 2^28)", e[i].count,
               e[i].child);
          return 0;
        }
        ref[i] = LEAF | ((e[i].count - 1u) << 28) | e[i].child;
      }
    }
    Node4& o = out[me];
    for (int i = 0; i < 4; ++i) {
      for (int a = 0; a < 3; ++a) {
        o.box[a][0][i] = i < n ? e[i].lo[a] : INFINITY;
        o.box[a][1][i] = i < n ? e[i].hi[a] : -INFINITY;
      }
      o.child[i] = ref[i];
      o.pad[i] = 0;
    }
    pb[me] = (n > 1 ? (uint32_t)n - 1u : 0u) + deeper;
    return me;
  }
};

}  // namespace

extern "C" {

SSOLH_API const char* ssolh_last_error(void) { return g_err; }

SSOLH_API int ssolh_device_count(void) {
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess) return 0;
  return n;
}

SSOLH_API int ssolh_create(int device, ssolh_context** out) {
  if (!out) { set_err("ssolh_create: NULL output"); return SSOLH_ERR_ARG; }
  *out = nullptr;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= device) {
    set_err("ssolh_create: no HIP device %d (found %d)", device, n);
    return SSOLH_ERR_NO_DEVICE;
  }
  hipDeviceProp_t prop;
  HIP_TRY(hipGetDeviceProperties(&prop, device));
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    set_err("ssolh_create: device %d is %s, the kernels are built for gfx950", device,
            prop.gcnArchName);
    return SSOLH_ERR_NO_DEVICE;
  }
  if (device < 0 || device >= MAX_DEVICES) {
    set_err("ssolh_create: device %d beyond the %d this library serves", device, MAX_DEVICES);
    return SSOLH_ERR_NO_DEVICE;
  }
  HIP_TRY(hipSetDevice(device));
  void* scratch_ptr = nullptr;
  {
    // once per device, with the device current: the address of its copy of
    // the scratch array
    // (without it only ssolh_solve_noalloc is unavailable, and says so)
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[device]) {
      void* p = nullptr;
      const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e == hipSuccess && p) {
        g_scratch[device] = p;
      } else {
        (void)hipGetLastError();
        fprintf(stderr, "ssolh_create: hipGetSymbolAddress(scratch) on device %d: %s\n", device,
                hipGetErrorString(e));
      }
    }
    scratch_ptr = g_scratch[device];
  }
  ssolh_context* c = new ssolh_context();
  c->device = device;
  c->scratch = scratch_ptr;
  HIP_TRY(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  for (auto& e : c->ev) HIP_TRY(hipEventCreate(&e));
  *out = c;
  return 0;
}

SSOLH_API int ssolh_destroy(ssolh_context* c) {
  if (!c) return SSOLH_ERR_ARG;
  (void)hipSetDevice(c->device);
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  free_scene(c);
  for (DevBuf* b : {&c->start_sort, &c->queue[0], &c->queue[1], &c->list, &c->pend, &c->tallies,
                    &c->folded, &c->jobs, &c->trace_ovf, &c->lbvh, &c->render, &c->plog,
                    &c->adj_state, &c->adj_in, &c->adj_grad, &c->trk_vtx, &c->trk_type,
                    &c->trk_seq, &c->trk_count, &c->trk_pos})
    if (b->p) (void)hipFree(b->p);
  for (auto& e : c->ev) if (e) (void)hipEventDestroy(e);
  if (c->stage) (void)hipHostFree(c->stage);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
  return 0;
}

SSOLH_API int ssolh_scene_upload(ssolh_context* c, const struct ssolh_scene* s) {
  if (!c || !s) { set_err("ssolh_scene_upload: NULL argument"); return SSOLH_ERR_ARG; }
  if (!s->nsample_tris || !s->ninstances || !s->nnodes) {
    set_err("ssolh_scene_upload: empty scene (sampled triangles %u, instances %u)",
            s->nsample_tris, s->ninstances);
    return SSOLH_ERR_ARG;
  }
  std::vector<ShapeQ> shapeq(s->nshapes);
  for (uint32_t i = 0; i < s->nshapes; ++i) {
    const double* m = s->shapes[i].qtransform;
    ShapeQ& q = shapeq[i];
    if (!inv3(m, q.Rinv)) {
      set_err("ssolh_scene_upload: singular quadric transform of shape %u", i);
      return SSOLH_ERR_ARG;
    }
    for (int k = 0; k < 3; ++k) q.t[k] = m[9 + k];
  }
  std::vector<IssInfo> iss;
  if (build_iss(s, iss)) {
    set_err("ssolh_scene_upload: inconsistent instance / shaded-shape indices");
    return SSOLH_ERR_ARG;
  }
  HIP_TRY(hipSetDevice(c->device));
  HIP_TRY(hipStreamSynchronize(c->stream));
  free_scene(c);
  DScene& d = c->scn;
  int r = 0;
  const double* cdf = nullptr;
  r |= upload(c, s->spectra, s->nspectra, &d.spectra.sp);
  r |= upload(c, s->spectra_wl, s->spectra_len, &d.spectra.wl);
  r |= upload(c, s->spectra_val, s->spectra_len, &d.spectra.val);
  r |= upload(c, s->spectra_cdf, s->spectra_len, &cdf);
  d.spectra.cdf = cdf;
  r |= upload(c, s->media, s->nmedia, &d.media);
  r |= upload(c, s->materials, s->nmaterials, &d.mtls);
  r |= upload(c, s->shapes, s->nshapes, &d.shapes);
  // 4-wide traversal nodes from the host's BVH2: each object's BLAS (one
  // copy per distinct root) and the TLAS, with the objects' roots remapped
  Collapse4 col(s->nodes, s->nnodes);
  std::vector<ssolh_object> objects(s->objects, s->objects + s->nobjects);
  std::map<uint32_t, uint32_t> blas_of;  // BVH2 root -> 4-wide root
  uint32_t blas_pb = 0;
  for (ssolh_object& o : objects) {
    auto it = blas_of.find(o.blas_root);
    if (it == blas_of.end()) it = blas_of.emplace(o.blas_root, col.root(o.blas_root)).first;
    o.blas_root = it->second;
    blas_pb = std::max(blas_pb, col.pb[it->second]);
  }
  const uint32_t troot = col.root(s->tlas_root);
  if (col.err) { set_err("ssolh_scene_upload: %s", col.msg); return col.err; }
  if (col.out.size() >= (1u << 25)) {  // byte offsets of the nodes fit 32 bits
    set_err("ssolh_scene_upload: %zu BVH nodes", col.out.size());
    return SSOLH_ERR_LIMIT;
  }
  r |= upload(c, objects.data(), objects.size(), &d.objects);
  // the TLAS region holds any tree over the instances (a GPU build writes
  // at most ninstances 4-wide nodes)
  c->tlas_base = troot;
  c->tlas_cap = std::max<uint32_t>((uint32_t)col.out.size() - troot, s->ninstances);
  col.out.resize((size_t)troot + c->tlas_cap);
  r |= upload(c, col.out.data(), col.out.size(), &d.nodes);
  // host arrays of the uploads below, alive until the closing synchronize
  std::vector<Node4> top;
  std::vector<uint32_t> top_order{troot}, tlas_order, level_end;
  static const double zero = 0;
  {
    // the TLAS's first TOP_NODES nodes, breadth first, with the references
    // between them rewritten to TOP_REF | index
    std::vector<uint32_t>& order = top_order;
    for (size_t h = 0; h < order.size() && order.size() < (size_t)TOP_NODES; ++h)
      for (int k = 0; k < 4 && order.size() < (size_t)TOP_NODES; ++k) {
        const uint32_t ch = col.out[order[h]].child[k];
        if (!(ch & LEAF)) order.push_back(ch);
      }
    std::map<uint32_t, uint32_t> where;
    for (size_t i = 0; i < order.size(); ++i) where[order[i]] = (uint32_t)i;
    for (uint32_t g : order) {
      Node4 n = col.out[g];
      for (int k = 0; k < 4; ++k) {
        auto w = (n.child[k] & LEAF) ? where.end() : where.find(n.child[k]);
        if (w != where.end()) n.child[k] = TOP_REF | w->second;
      }
      top.push_back(n);
    }
    d.ntop = (uint32_t)top.size();
    d.root_ref = TOP_REF;
    d.slack_scale = c->slack_scale;
    top.resize(TOP_NODES);
    r |= upload(c, top.data(), top.size(), &d.top);
    order.resize(TOP_NODES);
    r |= upload(c, order.data(), order.size(), &c->top_src);
  }
  {
    // TLAS nodes by depth, deepest level first (the refit's order), and the
    // tree's cost as built
    std::vector<std::vector<uint32_t>> levels;
    std::vector<std::pair<uint32_t, uint32_t>> todo{{troot, 0u}};
    double cost = 0;
    while (!todo.empty()) {
      const auto [nd, depth] = todo.back();
      todo.pop_back();
      if (levels.size() <= depth) levels.resize(depth + 1);
      levels[depth].push_back(nd);
      const Node4& n = col.out[nd];
      for (int k = 0; k < 4; ++k) {
        if (n.child[k] == EMPTY4) continue;
        const double x = (double)n.box[0][1][k] - n.box[0][0][k];
        const double y = (double)n.box[1][1][k] - n.box[1][0][k];
        const double z = (double)n.box[2][1][k] - n.box[2][0][k];
        cost += x * y + y * z + z * x;
        if (!(n.child[k] & LEAF)) todo.push_back({n.child[k], depth + 1});
      }
    }
    for (size_t l = levels.size(); l-- > 0;) {
      tlas_order.insert(tlas_order.end(), levels[l].begin(), levels[l].end());
      level_end.push_back((uint32_t)tlas_order.size());
    }
    c->tlas_levels = (uint32_t)level_end.size();
    tlas_order.resize(std::max<size_t>(tlas_order.size(), s->ninstances));
    level_end.resize(std::max<size_t>(level_end.size(), LBVH_MAX_LEVELS));
    r |= upload(c, tlas_order.data(), tlas_order.size(), &c->tlas_order);
    r |= upload(c, level_end.data(), level_end.size(), &c->tlas_level_end);
    c->tlas_cost0 = cost;
    r |= upload(c, &zero, 1, (const double**)&c->refit_cost);
  }
  r |= upload(c, s->object_boxes, (size_t)s->nobjects * 6, &c->obj_box);
  d.obj_box = c->obj_box;
  // a lane's stack: the TLAS descent's pushes, the instance sentinel, the
  // deepest BLAS descent's pushes
  c->stack_depth = col.pb[troot] + 1 + blas_pb;
  c->blas_pb = blas_pb;
  r |= upload(c, s->triangles, s->ntriangles, &d.tris);
  r |= upload(c, s->instances, s->ninstances, &d.insts);
  r |= upload(c, s->tlas_instances, s->ninstances, &d.tlas_inst);
  r |= upload(c, s->inst_sshapes, s->ninst_sshapes, &d.isshapes);
  r |= upload(c, iss.data(), iss.size(), &d.iss);
  r |= upload(c, shapeq.data(), shapeq.size(), &c->shapeq);
  r |= upload(c, s->sample_tris, s->nsample_tris, &d.stris);
  r |= upload(c, s->sample_alias, s->nsample_tris, &d.alias);
  std::vector<StartAlias> salias(s->nsample_tris);
  for (uint32_t i = 0; i < s->nsample_tris; ++i)
    salias[i] = {s->sample_alias[i].prob, s->sample_tris[i].instance,
                 s->sample_tris[s->sample_alias[i].alias].instance};
  r |= upload(c, salias.data(), salias.size(), &d.salias);
  if (r) return r;
  d.air = s->air_medium;
  d.tlas_root = troot;
  d.nstris = s->nsample_tris;
  d.sun = s->sun;
  d.S = s->sampled_area;
  d.S_proxy = s->sampled_area_proxy;
  d.nrcv = s->nreceivers;
  d.nsamp = s->nsampled;
  c->nrcv = s->nreceivers;
  c->nsamp = s->nsampled;
  c->nprim = s->nprim_tallies;
  c->ninstances = s->ninstances;
  c->ninst_sshapes = s->ninst_sshapes;
  c->inst_object.resize(s->ninstances);
  for (uint32_t i = 0; i < s->ninstances; ++i) c->inst_object[i] = s->instances[i].object;
  HIP_TRY(hipStreamSynchronize(c->stream));  // the host arrays may go after return
  // pending entries are kept by paths that a receiver does not end: not
  // where every receiving side absorbs all light
  c->may_pend = false;
  for (const IssInfo& x : iss) {
    if (x.receiver < 0) continue;
    for (uint32_t side : {SSOL_FRONT_, SSOL_BACK_}) {
      const ssolh_material& m = s->materials[side == SSOL_FRONT_ ? x.mtl_front : x.mtl_back];
      const bool black = (m.type == SSOLH_MTL_MATTE || m.type == SSOLH_MTL_MIRROR) &&
                         m.reflectivity == 0;
      if ((x.receiver_mask & side) && !black) c->may_pend = true;
    }
  }
  c->has_scene = true;
  ++c->n_uploads;
  return 0;
}

SSOLH_API int ssolh_scene_move_instances(ssolh_context* c, uint32_t ninstances,
                                         const struct ssolh_instance* instances,
                                         uint32_t ninst_sshapes,
                                         const struct ssolh_inst_sshape* inst_sshapes,
                                         double* cost_ratio) {
  if (!c || !instances || (ninst_sshapes && !inst_sshapes)) {
    set_err("ssolh_scene_move_instances: NULL argument");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene || ninstances != c->ninstances || ninst_sshapes != c->ninst_sshapes) {
    set_err("ssolh_scene_move_instances: %u instances, %u (instance, shape) frames for a scene "
            "of %u and %u", ninstances, ninst_sshapes, c->ninstances, c->ninst_sshapes);
    return SSOLH_ERR_ARG;
  }
  for (uint32_t i = 0; i < ninstances; ++i)
    if (instances[i].object != c->inst_object[i]) {
      set_err("ssolh_scene_move_instances: instance %u changed object", i);
      return SSOLH_ERR_ARG;
    }
  HIP_TRY(hipSetDevice(c->device));
  DScene& d = c->scn;
  HIP_TRY(hipMemcpyAsync((void*)d.insts, instances, ninstances * sizeof(ssolh_instance),
                         hipMemcpyHostToDevice, c->stream));
  if (ninst_sshapes)
    HIP_TRY(hipMemcpyAsync((void*)d.isshapes, inst_sshapes,
                           ninst_sshapes * sizeof(ssolh_inst_sshape), hipMemcpyHostToDevice,
                           c->stream));
  k_tlas_refit<<<1, REFIT_THREADS, 0, c->stream>>>(
      d.insts, d.tlas_inst, c->obj_box, (Node4*)d.nodes, c->tlas_order, c->tlas_level_end,
      c->tlas_levels, (Node4*)d.top, c->top_src, d.ntop, c->refit_cost);
  HIP_TRY(hipGetLastError());
  double cost = 0;
  HIP_TRY(hipMemcpyAsync(&cost, c->refit_cost, sizeof(cost), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (cost_ratio) *cost_ratio = c->tlas_cost0 > 0 ? cost / c->tlas_cost0 : 1.0;
  ++c->n_refits;
  return 0;
}

SSOLH_API int ssolh_scene_build_tlas(ssolh_context* c) {
  if (!c || !c->has_scene) {
    set_err("ssolh_scene_build_tlas: no scene");
    return SSOLH_ERR_ARG;
  }
  const uint32_t n = c->ninstances;
  HIP_TRY(hipSetDevice(c->device));
  // work buffer: sort keys and values (twice), the radix sort's temporary,
  // instance boxes, the binary tree, results
  size_t sort_bytes = 0;
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (const uint32_t*)nullptr,
                                             (uint32_t*)nullptr, (const uint32_t*)nullptr,
                                             (uint32_t*)nullptr, (int)n, 0, 30, c->stream));
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t nn = n, ni = n > 1 ? n - 1 : 1;
  const size_t sizes[] = {nn * 4, nn * 4, nn * 4, nn * 4, sort_bytes, nn * 24, ni * 8,
                          (2 * nn) * 4, ni * 4, ni * 24, ni * 4, ni * 4, nn * 4,
                          sizeof(LbvhResult)};
  size_t total = 0;
  for (size_t b : sizes) total += al(b);
  if (int e = dev_alloc(c->lbvh, total)) return e;
  char* p = (char*)c->lbvh.p;
  void* part[14];
  for (int i = 0; i < 14; ++i) { part[i] = p; p += al(sizes[i]); }
  uint32_t *key = (uint32_t*)part[0], *skey = (uint32_t*)part[1], *val = (uint32_t*)part[2],
           *sval = (uint32_t*)part[3];
  LbvhWork w{(int2*)part[6], (int*)part[7], (unsigned*)part[8], (float*)part[9],
             (uint32_t*)part[10], (uint32_t*)part[11], (uint32_t*)part[12]};
  LbvhResult* res = (LbvhResult*)part[13];
  DScene& d = c->scn;
  k_lbvh_keys<<<1, LBVH_THREADS, 0, c->stream>>>(d.insts, c->obj_box, n, (float*)part[5], key,
                                                 val);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(part[4], sort_bytes, key, skey, val, sval, (int)n, 0,
                                             30, c->stream));
  k_lbvh_finish<<<1, LBVH_THREADS, 0, c->stream>>>(
      n, skey, sval, (const float*)part[5], w, (Node4*)d.nodes + c->tlas_base, c->tlas_base,
      (uint32_t*)d.tlas_inst, (uint32_t*)c->tlas_order, (uint32_t*)c->tlas_level_end,
      (Node4*)d.top, (uint32_t*)c->top_src, res);
  HIP_TRY(hipGetLastError());
  LbvhResult h{};
  HIP_TRY(hipMemcpyAsync(&h, res, sizeof(h), hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  if (h.nodes4 == 0 || h.nodes4 > c->tlas_cap || h.ntop == 0 || h.ntop > (uint32_t)TOP_NODES) {
    set_err("ssolh_scene_build_tlas: inconsistent build (%u nodes, %u top)", h.nodes4, h.ntop);
    return SSOLH_ERR_LIMIT;
  }
  d.ntop = h.ntop;
  d.root_ref = TOP_REF;
  c->tlas_levels = h.depth4 + 1;
  c->tlas_cost0 = h.cost;
  // a descent pushes at most 3 per 4-wide level above the leaves
  c->stack_depth = 3u * (h.depth4 + 1u) + 1u + c->blas_pb;
  ++c->n_builds;
  return 0;
}

SSOLH_API int ssolh_render(ssolh_context* c, const struct ssolh_render_args* a, double* pixels) {
  if (!c || !a || !pixels || !a->width || !a->height || !a->spp || a->mode > 1 ||
      (a->mode == 0 && !a->draft_samples)) {
    set_err("ssolh_render: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene) { set_err("ssolh_render: no scene"); return SSOLH_ERR_ARG; }
  const uint64_t npix = (uint64_t)a->width * a->height, total = npix * a->spp;
  if (npix > (1u << 28) || a->spp > (1u << 20)) {
    set_err("ssolh_render: %llu pixels x %u samples", (unsigned long long)npix, a->spp);
    return SSOLH_ERR_LIMIT;
  }
  HIP_TRY(hipSetDevice(c->device));
  const uint32_t batch = (uint32_t)std::min<uint64_t>(total, 1u << 21);
  const uint32_t nslot = 2 * batch;
  const uint32_t lds_stack = trace_lds_stack(c);
  const uint32_t extra = c->stack_depth > lds_stack ? c->stack_depth - lds_stack : 0;
  auto al = [](size_t b) { return (b + 255) / 256 * 256; };
  const size_t sizes[] = {(size_t)batch * sizeof(RenderState), (size_t)nslot * sizeof(RayRec),
                          (size_t)nslot * sizeof(HitRec), (size_t)nslot * 4, (size_t)nslot * 4,
                          npix * 8, (size_t)a->spp * 8, 16, (size_t)nslot * extra * 4 + 4};
  size_t bytes = 0;
  for (size_t b : sizes) bytes += al(b);
  if (int e = dev_alloc(c->render, bytes)) return e;
  char* p = (char*)c->render.p;
  void* part[9];
  for (int i = 0; i < 9; ++i) { part[i] = p; p += al(sizes[i]); }
  RenderState* st = (RenderState*)part[0];
  RayRec* rays = (RayRec*)part[1];
  HitRec* hits = (HitRec*)part[2];
  uint32_t* lists[2] = {(uint32_t*)part[3], (uint32_t*)part[4]};
  double* pix = (double*)part[5];
  float* draft = (float*)part[6];
  unsigned* cnt = (unsigned*)part[7];  // [0], [1]: list lengths, [2]: unused ticket
  const TOvf ovf{extra ? (uint32_t*)part[8] : nullptr, nslot, extra};
  HIP_TRY(hipMemsetAsync(pix, 0, npix * 8, c->stream));
  if (a->mode == 0)
    HIP_TRY(hipMemcpyAsync(draft, a->draft_samples, (size_t)a->spp * 8, hipMemcpyHostToDevice,
                           c->stream));
  RenderParams rp{};
  rp.width = a->width; rp.height = a->height; rp.spp = a->spp; rp.mode = a->mode;
  for (int k = 0; k < 3; ++k) {
    rp.pos[k] = a->position[k]; rp.ax[k] = a->axis_x[k]; rp.ay[k] = a->axis_y[k];
    rp.az[k] = a->axis_z[k]; rp.up[k] = a->up[k];
  }
  rp.key = a->rng_key;
  rp.draft = draft;
  for (uint64_t first = 0; first < total; first += batch) {
    rp.first = first;
    rp.count = (uint32_t)std::min<uint64_t>(total - first, batch);
    const uint32_t blocks = (rp.count + BLOCK - 1) / BLOCK;
    k_render_start<<<blocks, BLOCK, 0, c->stream>>>(c->scn, rp, st, rays, lists[0], cnt);
    HIP_TRY(hipGetLastError());
    int cur = 0;
    for (uint32_t iter = 0;; ++iter) {
      unsigned n = 0;
      HIP_TRY(hipMemcpyAsync(&n, cnt + cur, sizeof(n), hipMemcpyDeviceToHost, c->stream));
      HIP_TRY(hipStreamSynchronize(c->stream));
      if (!n) break;
      if (iter >= 100000) { set_err("ssolh_render: paths did not end"); return SSOLH_ERR_LIMIT; }
      const uint32_t tb = (n + BLOCK - 1) / BLOCK;
      if (lds_stack == 16)
        k_trace<16><<<tb, BLOCK, 0, c->stream>>>(c->scn, lists[cur], cnt + cur, rays, hits,
                                                ovf);
      else if (lds_stack == 24)
        k_trace<24><<<tb, BLOCK, 0, c->stream>>>(c->scn, lists[cur], cnt + cur, rays, hits,
                                                ovf);
      else
        k_trace<MAX_STACK><<<tb, BLOCK, 0, c->stream>>>(c->scn, lists[cur], cnt + cur,
                                                              rays, hits, ovf);
      HIP_TRY(hipGetLastError());
      HIP_TRY(hipMemsetAsync(cnt + (cur ^ 1), 0, sizeof(unsigned), c->stream));
      k_render_shade<<<blocks, BLOCK, 0, c->stream>>>(c->scn, rp, st, rays, hits, pix,
                                                      lists[cur ^ 1], cnt + (cur ^ 1));
      HIP_TRY(hipGetLastError());
      cur ^= 1;
    }
  }
  HIP_TRY(hipMemcpyAsync(pixels, pix, npix * 8, hipMemcpyDeviceToHost, c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  return 0;
}

SSOLH_API int ssolh_test_slab_slack(ssolh_context* c, float scale) {
  if (!c || !(scale >= 0.f && scale <= 1e-3f)) {
    set_err("ssolh_test_slab_slack: scale outside [0, 1e-3]");
    return SSOLH_ERR_ARG;
  }
  c->slack_scale = scale;
  c->scn.slack_scale = c->slack_scale;
  return 0;
}

SSOLH_API int ssolh_test_scene_counters(ssolh_context* c, uint32_t* uploads, uint32_t* refits,
                                        uint32_t* builds) {
  if (!c) return SSOLH_ERR_ARG;
  if (uploads) *uploads = c->n_uploads;
  if (refits) *refits = c->n_refits;
  if (builds) *builds = c->n_builds;
  return 0;
}

}  // extern "C"

namespace {

// Host description of a tracked and of an adjoint solve (host pointers)
struct TrackHost {
  double sun_len, inf_len;
  uint64_t cap;
};

struct AdjHost {
  uint32_t nparams;
  const int32_t* inst_param;  // [ninstances]
  const double* axes;         // [nparams][2][3]
  const double* gmap;         // [nprim_tallies][2] or null
  double d_total;
};

// One solve over `njobs` suns (njobs == 1: the scene's sun). Realisation
// ids [0, N) map to jobs through job_first.
int run_solve(ssolh_context* c, uint64_t N, uint64_t max_failed, uint64_t key, uint64_t counter,
              bool fp32, uint32_t path_slots, uint32_t npend, uint32_t njobs,
              const uint64_t* job_first_h, const ssolh_sun* job_suns_h,
              const AdjHost* adj = nullptr, const TrackHost* trk = nullptr,
              Arena* arena = nullptr) {
  // buffers come from the device allocator, or all from the arena
  auto alloc = [&](DevBuf& b, size_t bytes) -> int {
    return arena ? arena_take(*arena, b, bytes) : dev_alloc(b, bytes);
  };
  if (arena && (adj || trk || job_suns_h)) {
    set_err("ssolh_solve_noalloc: plain single-sun solves driven from the host only");
    return SSOLH_ERR_ARG;
  }
  if (adj && fp32) { set_err("ssolh_solve_adjoint: the adjoint runs in the FP64 form"); return SSOLH_ERR_ARG; }
  if (trk && (fp32 || adj || job_suns_h)) {
    set_err("ssolh_solve_tracked: paths are recorded by plain FP64 solves only");
    return SSOLH_ERR_ARG;
  }
  if (!trk) c->trk_paths = 0;  // the recorded paths belong to the last solve only
  if (npend > MAX_PEND) { set_err("ssolh_solve: at most %d pending entries", MAX_PEND); return SSOLH_ERR_LIMIT; }
  // Tally layout: each tally is striped over up to 256 copies while its
  // stripes hold at most 2^18 doubles (2^21 take 20 us more to clear and fold,
  // and no flush is faster for them); from the scratch array every stripe
  // count is halved until all tallies take at most half of it.
  uint32_t sg, sr, ss, sx, sp;
  size_t n_global, n_rcv, n_samp, n_sxr, n_prim, n_u64, tally_bytes;
  for (size_t cap = 256;; cap >>= 1) {
    auto pow2_stripes = [cap](size_t per_stripe_doubles) {
      size_t k = cap;
      while (k > 1 && k * per_stripe_doubles > (size_t(1) << 18)) k >>= 1;
      return (uint32_t)k;
    };
    sg = pow2_stripes((size_t)njobs * 16);
    sr = 1;  // zeros: the fold sums it from the sampled x receiver tally
    ss = pow2_stripes((size_t)c->nsamp * 5);
    sx = pow2_stripes((size_t)c->nsamp * c->nrcv * 40);
    sp = pow2_stripes((size_t)c->nprim * 40);
    n_global = (size_t)sg * njobs * 16;
    n_rcv = (size_t)sr * c->nrcv * 40;
    n_samp = (size_t)ss * c->nsamp * 4;
    n_sxr = (size_t)sx * c->nsamp * c->nrcv * 40;
    n_prim = (size_t)sp * c->nprim * 40;
    n_u64 = (size_t)ss * c->nsamp;
    tally_bytes = (n_global + n_rcv + n_samp + n_sxr + n_prim + n_u64) * 8 + 64;
    if (!arena || tally_bytes <= arena->size / 2 || cap == 1) break;
  }
  if (arena && tally_bytes > arena->size / 2) {
    set_err("ssolh_solve_noalloc: the scene's tallies take %zu bytes; at most %zu fit in the "
            "scratch array", tally_bytes, arena->size / 2);
    return SSOLH_ERR_LIMIT;
  }
  // Wavefront width. By default every realisation of the solve is in flight
  // at once, in start-instance order, when 2/5 of the device memory holds
  // what a realisation keeps there: its place in the order, its places in the
  // path queues and, in scenes whose receivers let light pass, its pending
  // entries. Larger solves run as many as fit at a time.
  const uint32_t npend_asked = npend;
  if (!c->may_pend) npend = 0;
  const size_t real = fp32 ? sizeof(float) : sizeof(double);
  const size_t planes = fp32 ? RAY_PLANES32 + STATE_PLANES32 : RAY_PLANES64 + STATE_PLANES64;
  TOvf ovf{nullptr, 0, c->stack_depth > START_STACK ? c->stack_depth - START_STACK : 0u};
  const size_t per_slot = 2 * sizeof(uint32_t) + 2 * planes * 16 + ovf.extra * sizeof(uint32_t) +
                          (size_t)npend * 2 * (sizeof(uint32_t) + 10 * real) +
                          (adj ? sizeof(double4) + sizeof(uint32_t) : 0) +
                          (trk ? sizeof(uint32_t) + sizeof(double4) : 0);
  uint64_t slots64 = path_slots;
  if (arena) {
    // An asked width is refused past what the array holds of slots with a
    // ray, a hit, a path record and pending entries each, whatever the scene
    // needs of these. The width taken is what is left beside the tallies, the
    // sort's work bytes and the alignment of the parts.
    const size_t most_slot = fp32 ? 233 + 88 * (size_t)npend_asked : 281 + 168 * (size_t)npend_asked;
    const uint64_t asked = std::min<uint64_t>(path_slots, N);
    if (asked > (arena->size - tally_bytes) / most_slot) {
      set_err("ssolh_solve_noalloc: %llu path slots do not fit beside the tallies in the scratch "
              "array", (unsigned long long)asked);
      return SSOLH_ERR_LIMIT;
    }
    size_t sort_bytes = 0;
    const uint64_t most = std::min<uint64_t>(std::min<uint64_t>(N, arena->size / per_slot), 1u << 28);
    HIP_TRY(start_sort_bytes((uint32_t)most, start_key_bits((uint64_t)njobs * c->ninstances),
                             c->stream, sort_bytes));
    const size_t fixed = tally_bytes + (sort_bytes + 255) / 256 * 256 + GROUP_BYTES + (64u << 10);
    const size_t rest = arena->size > fixed ? arena->size - fixed : 0;
    slots64 = rest / per_slot / BLOCK * BLOCK;
    if (slots64 < BLOCK) {
      set_err("ssolh_solve_noalloc: no path slot fits beside the tallies in the scratch array");
      return SSOLH_ERR_LIMIT;
    }
    if (path_slots) slots64 = std::min<uint64_t>(slots64, path_slots);
  }
  if (!slots64) {
    size_t free_b = 0, total_b = 0;
    HIP_TRY(hipMemGetInfo(&free_b, &total_b));
    const uint64_t fit = (uint64_t)(total_b / 5 * 2) / per_slot;
    slots64 = std::min<uint64_t>(std::max<uint64_t>(fit, 1u << 20), 1ull << 27);
    // and within what is free now (this context's own solve buffers count
    // as free: they are reallocated), when other work holds device memory
    size_t held = 0;
    for (const DevBuf* b : {&c->queue[0], &c->queue[1], &c->list, &c->pend, &c->trace_ovf,
                            &c->adj_state, &c->trk_seq})
      held += b->n;
    const uint64_t fit_free = (uint64_t)((free_b + held) / 10 * 9) / per_slot;
    slots64 = std::min<uint64_t>(slots64, std::max<uint64_t>(fit_free, 1u << 16));
  }
  if (slots64 > N) slots64 = N;
  slots64 = (slots64 + BLOCK - 1) / BLOCK * BLOCK;
  if (slots64 > (1ull << 28)) { set_err("ssolh_solve: at most 2^28 path slots"); return SSOLH_ERR_LIMIT; }
  const uint32_t slots = (uint32_t)slots64;
  const size_t n = slots;

  // With fewer slots than realisations the solve runs in chunks of `slots`
  // realisations, one after the other. Each is put in start-instance order
  // when there is something to order by (more than one sun or sampled
  // instance); otherwise realisation s of a chunk takes slot s, and the
  // chunks count as one wavefront whose slots take further realisations.
  const uint64_t nkeys = (uint64_t)njobs * c->ninstances;
  const bool orderable = (uint64_t)njobs * c->nsamp > 1 && nkeys <= (1u << 24);
  const bool refill = slots < N && !orderable;

  // start order: keys and indices before and after their sort, in the queue
  // that is not written before they have been read
  const uint32_t key_bits = start_key_bits(nkeys);
  const size_t part = (n + 63) / 64 * 64;  // 256-byte aligned parts
  size_t sort_bytes = 0;
  int r = 0;
  const bool group_starts = group_pays(slots, nkeys);
  if (orderable && !group_starts) {
    HIP_TRY(start_sort_bytes(slots, key_bits, c->stream, sort_bytes));
    if ((r = alloc(c->start_sort, sort_bytes))) return r;
  }
  // what a solve starts from zero, cleared at once: the counters, the record
  // count of the log, the counts of the groupings by start key and by
  // primitive (which each grouping leaves clear), the tallies (striped where
  // many waves meet, see Tallies); beside them the groupings' offsets
  // (the log's counts, which waves add to, on cache lines of their own; a
  // reduction's record counts)
  constexpr size_t log_n_at = 256, kept_at = log_n_at + LOG_SEGS * LOG_LINE * 8;
  constexpr size_t head_bytes = kept_at + 256;
  static_assert(sizeof(Counters) <= log_n_at && LOG_SEGS <= 64, "head of the cleared buffer");
  const size_t clear_bytes =
      head_bytes + 2 * GROUP_KEYS * sizeof(uint32_t) + (tally_bytes + 15) / 16 * 16;
  if ((r = alloc(c->tallies, clear_bytes + 2 * (GROUP_KEYS + 4) * sizeof(uint32_t)))) return r;
  HIP_TRY(hipMemsetAsync(c->tallies.p, 0, clear_bytes, c->stream));
  Counters* const ctr = (Counters*)c->tallies.p;
  unsigned long long* const log_n = (unsigned long long*)((char*)c->tallies.p + log_n_at);
  uint32_t* const log_kept = (uint32_t*)((char*)c->tallies.p + kept_at);
  uint32_t* const group = (uint32_t*)((char*)c->tallies.p + head_bytes);
  uint32_t* const offsets = (uint32_t*)((char*)c->tallies.p + clear_bytes);
  const GroupKeys start_keys{group, offsets, (uint32_t)std::min<uint64_t>(nkeys, UINT32_MAX)};
  const GroupKeys prim_keys{group + GROUP_KEYS, offsets + GROUP_KEYS + 4,
                            (uint32_t)std::min<uint64_t>((uint64_t)c->nprim * 2, UINT32_MAX)};
  // path queues, the list of places in the one being read, the waves' counts
  // of paths written and their scan
  for (int i = 0; i < 2; ++i)
    if ((r = alloc(c->queue[i], part * planes * 16))) return r;
  const uint32_t waves = slots / 64, chunks = (waves + SCAN_CHUNK - 1) / SCAN_CHUNK;
  if ((r = alloc(c->list, (n + 2 * waves + chunks) * sizeof(uint32_t)))) return r;
  uint32_t* const list = (uint32_t*)c->list.p;
  uint32_t *const wave_n = list + n, *const wave_off = wave_n + waves,
           *const wave_chunk = wave_off + waves;
  Pending W{};
  W.npend = npend;
  if (npend) {
    const size_t keys = npend * n * sizeof(uint32_t), vals = npend * n * 10 * real;
    if ((r = alloc(c->pend, 2 * keys + 2 * vals))) return r;
    char* p = (char*)c->pend.p;  // each part a multiple of 128 * 4 bytes
    W.pkey = (uint32_t*)p;
    W.qkey = (uint32_t*)(p + keys);
    W.pval = p + 2 * keys;
    W.qval = p + 2 * keys + vals;
  }
  // traversal stack entries past the LDS ones, per lane of a launch
  if (ovf.extra) {
    ovf.stride = slots;
    if ((r = alloc(c->trace_ovf, n * ovf.extra * sizeof(uint32_t)))) return r;
    ovf.base = (uint32_t*)c->trace_ovf.p;
  }
  // adjoint buffers
  AdjParams A{};
  if (adj) {
    const size_t ninst = c->ninstances, ngm = (size_t)c->nprim * 2;
    const size_t in_bytes = ninst * sizeof(int32_t) + 64 + (size_t)adj->nparams * 6 * sizeof(double) +
                            ngm * sizeof(double) + 64;
    if ((r = alloc(c->adj_state, n * (sizeof(double4) + sizeof(uint32_t)) + 256))) return r;
    if ((r = alloc(c->adj_in, in_bytes))) return r;
    if ((r = alloc(c->adj_grad, (size_t)adj->nparams * 3 * sizeof(double) + 8))) return r;
    char* ai = (char*)c->adj_in.p;
    int32_t* d_ip = (int32_t*)ai;
    double* d_axes = (double*)(ai + (ninst * sizeof(int32_t) + 63) / 64 * 64);
    double* d_gm = d_axes + (size_t)adj->nparams * 6;
    HIP_TRY(hipMemcpyAsync(d_ip, adj->inst_param, ninst * sizeof(int32_t), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipMemcpyAsync(d_axes, adj->axes, (size_t)adj->nparams * 6 * sizeof(double),
                           hipMemcpyHostToDevice, c->stream));
    if (adj->gmap && ngm)
      HIP_TRY(hipMemcpyAsync(d_gm, adj->gmap, ngm * sizeof(double), hipMemcpyHostToDevice, c->stream));
    else if (ngm)
      HIP_TRY(hipMemsetAsync(d_gm, 0, ngm * sizeof(double), c->stream));
    HIP_TRY(hipMemsetAsync(c->adj_grad.p, 0, (size_t)adj->nparams * 3 * sizeof(double), c->stream));
    A.grad = (double*)c->adj_grad.p;
    A.inst_param = d_ip;
    A.axes = d_axes;
    A.gmap = d_gm;
    A.d_total = adj->d_total;
    A.s = (double4*)c->adj_state.p;
    A.p = (uint32_t*)((char*)c->adj_state.p + (n * sizeof(double4) + 255) / 256 * 256);
  }
  // path recording buffers
  TrackParams K{};
  if (trk) {
    const uint64_t cap = std::max<uint64_t>(trk->cap, 1);
    if ((r = alloc(c->trk_vtx, cap * sizeof(ssolh_track_vertex)))) return r;
    if ((r = alloc(c->trk_type, N))) return r;
    if ((r = alloc(c->trk_seq, n * sizeof(uint32_t)))) return r;
    if ((r = alloc(c->trk_pos, n * sizeof(double4)))) return r;
    if ((r = alloc(c->trk_count, sizeof(unsigned long long)))) return r;
    HIP_TRY(hipMemsetAsync(c->trk_type.p, SSOLH_PATH_DROPPED, N, c->stream));
    HIP_TRY(hipMemsetAsync(c->trk_count.p, 0, sizeof(unsigned long long), c->stream));
    K.vtx = (ssolh_track_vertex*)c->trk_vtx.p;
    K.nvtx = (unsigned long long*)c->trk_count.p;
    K.cap = cap;
    K.type = (uint8_t*)c->trk_type.p;
    K.seq = (uint32_t*)c->trk_seq.p;
    K.pos = (double4*)c->trk_pos.p;
    K.sun_len = trk->sun_len;
    K.inf_len = trk->inf_len;
    c->trk_cap = cap;
    c->trk_paths = N;
  }
  // jobs
  if (job_suns_h) {
    if ((r = alloc(c->jobs, (njobs + 1) * sizeof(uint64_t) + njobs * sizeof(ssolh_sun)))) return r;
    HIP_TRY(hipMemcpyAsync(c->jobs.p, job_first_h, (njobs + 1) * sizeof(uint64_t),
                           hipMemcpyHostToDevice, c->stream));
    HIP_TRY(hipMemcpyAsync((char*)c->jobs.p + (njobs + 1) * sizeof(uint64_t), job_suns_h,
                           njobs * sizeof(ssolh_sun), hipMemcpyHostToDevice, c->stream));
  }

  double* tb = (double*)(group + 2 * GROUP_KEYS);
  c->T.global = tb;
  c->T.rcv = c->T.global + n_global;
  c->T.samp = c->T.rcv + n_rcv;
  c->T.sxr = c->T.samp + n_samp;
  c->T.prim = c->T.sxr + n_sxr;
  c->T.samp_count = (unsigned long long*)(c->T.prim + n_prim);
  c->T.mask_g = sg - 1;
  c->T.mask_s = ss - 1;
  c->T.mask_x = sx - 1;
  c->T.mask_p = sp - 1;
  c->T.nprim = c->nprim;
  c->T.nrcv = c->nrcv;
  c->T.nsamp = c->nsamp;
  c->T.njobs = njobs;
  c->njobs = njobs;
  // per-primitive log: room for one record per realisation, or four where
  // receivers pass light on and a path logs each primitive it met (a cavity
  // of ten bounces: 3.2), at most LOG_MAX_RECORDS; none from the scratch array
  bool group_log = false;
  c->T.log_key = nullptr;
  c->T.log_val = nullptr;
  c->T.log_n = nullptr;
  c->T.log_cap = 0;
  c->T.log_seg = c->T.log_mask = 0;
  uint32_t log_segs = 1;
  c->log_flushes = 0;
  c->log_overflowed = 0;
  if (!arena && c->nprim) {
    uint32_t cap = (uint32_t)std::min<uint64_t>(
        std::min<uint64_t>(N, LOG_MAX_RECORDS) * (c->may_pend ? 4 : 1), LOG_MAX_RECORDS);
    if (c->log_cap_test) cap = std::min(cap, c->log_cap_test);
    // One counter takes 1.6 ns per wave that logs, one wave after the other:
    // large logs have LOG_SEGS, whose segments (filled evenly, by block) hold
    // an eighth more than their share (4e6 paths: 1567 us of path kernels
    // with one counter, 1400 with 16)
    if (cap >= (1u << 18)) {
      log_segs = LOG_SEGS;
      cap = (cap / LOG_SEGS * 9 / 8 + 63) / 64 * 64 * LOG_SEGS;
    }
    uint32_t bits = 1;
    while (bits < 32 && (uint64_t(1) << bits) < (uint64_t)c->nprim * 2) ++bits;
    group_log = group_pays(cap, (uint64_t)c->nprim * 2);
    size_t sort_bytes = 0;
    if (!group_log)
      HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, sort_bytes, (const uint32_t*)nullptr,
                                                 (uint32_t*)nullptr, (const uint32_t*)nullptr,
                                                 (uint32_t*)nullptr, (int)cap, 0, (int)bits,
                                                 c->stream));
    auto up = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t k4 = up((size_t)cap * 4);
    const size_t bytes = 5 * k4 + up((size_t)cap * 80) + up(sort_bytes);
    if (alloc(c->plog, bytes)) {
      // no room left beside the path state: every entry takes the atomics
      (void)hipGetLastError();
      c->plog = DevBuf{};
      cap = 0;
    }
    if (cap) {
      char* q = (char*)c->plog.p;
      c->T.log_key = (uint32_t*)q;
      c->log_skey = (uint32_t*)(q + k4);
      c->log_idx = (uint32_t*)(q + 2 * k4);
      c->log_sidx = (uint32_t*)(q + 3 * k4);
      c->log_ckey = (uint32_t*)(q + 4 * k4);
      c->T.log_val = (double*)(q + 5 * k4);
      c->T.log_n = log_n;
      c->log_sort = q + 5 * k4 + up((size_t)cap * 80);
      c->log_sort_bytes = sort_bytes;
      c->log_key_bits = bits;
      c->T.log_cap = cap;
      c->T.log_seg = cap / log_segs;
      c->T.log_mask = log_segs - 1;
    }
  }
  // Sums the logged records into the per-primitive tally and empties the
  // log
  auto log_flush = [&]() -> int {
    if (!c->T.log_cap) return 0;
    const uint32_t cap = c->T.log_seg;  // of a segment
    // `shares` waves per key: one round of 64 records each for an even spread
    // of m records, 131,072 waves at most for that. A flux map's peak holds
    // several times the mean: with four rounds its waves run on alone (4e6
    // records of 4,096 keys: 253 us, with one 200).
    auto reduce = [&](uint32_t m, const uint32_t* skey) -> int {
      const uint32_t shares = (uint32_t)std::max<uint64_t>(
          1, std::min<uint64_t>(m / (64ull * prim_keys.keys), 131072u / prim_keys.keys));
      const uint32_t blocks = (uint32_t)(((uint64_t)prim_keys.keys * shares + 3) / 4);
      k_prim_reduce<<<blocks, 256, 0, c->stream>>>(prim_keys, skey, c->log_sidx, m, c->T.log_val,
                                                   shares, c->T.prim);
      HIP_TRY(hipGetLastError());
      return 0;
    };
    if (group_log) {
      const dim3 rank_grid((cap + GROUP_BLOCK - 1) / GROUP_BLOCK, log_segs);
      const dim3 place_grid((cap + 255) / 256, log_segs);
      k_group_rank<<<rank_grid, GROUP_THREADS, 0, c->stream>>>(
          LogKeyOf{c->T.log_key}, c->T.log_n, cap, prim_keys, nullptr, c->log_skey);
      HIP_TRY(hipGetLastError());
      k_group_scan<<<1, GROUP_THREADS, 0, c->stream>>>(prim_keys, c->T.log_n, log_segs, cap, log_kept,
                                                       ctr);
      HIP_TRY(hipGetLastError());
      k_group_place<<<place_grid, 256, 0, c->stream>>>(
          c->T.log_key, c->log_skey, log_kept, cap, prim_keys, c->log_sidx);
      HIP_TRY(hipGetLastError());
      return reduce((uint32_t)c->T.log_cap, nullptr);
    }
    unsigned long long asked[LOG_SEGS * LOG_LINE], n = 0;
    HIP_TRY(hipMemcpyAsync(asked, c->T.log_n, log_segs * LOG_LINE * sizeof(asked[0]),
                           hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(hipStreamSynchronize(c->stream));
    LogSegments parts{};
    uint32_t longest = 0;
    for (uint32_t s = 0; s < log_segs; ++s) {
      const uint32_t used = (uint32_t)std::min<unsigned long long>(asked[s * LOG_LINE], cap);
      n += asked[s * LOG_LINE];
      parts.first[s + 1] = parts.first[s] + used;
      longest = std::max(longest, used);
    }
    const uint32_t m = parts.first[log_segs];
    c->log_overflowed += n - m;
    if (m) {
      ++c->log_flushes;
      const dim3 list_grid((longest + 255) / 256, log_segs);
      k_log_list<<<list_grid, 256, 0, c->stream>>>(c->T.log_key, cap, parts, c->log_ckey, c->log_idx);
      HIP_TRY(hipGetLastError());
      size_t sb = c->log_sort_bytes;
      HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->log_sort, sb, c->log_ckey, c->log_skey,
                                                 c->log_idx, c->log_sidx, (int)m, 0,
                                                 (int)c->log_key_bits, c->stream));
      if (int e = reduce(m, c->log_skey)) return e;
    }
    if (n)
      HIP_TRY(hipMemsetAsync(c->T.log_n, 0, log_segs * LOG_LINE * sizeof(asked[0]), c->stream));
    return 0;
  };

  SolveParams prm;
  prm.N = N;
  prm.max_failed = max_failed;
  prm.key = key;
  prm.counter = counter;
  prm.slots = slots;
  prm.npend = npend;
  prm.njobs = njobs;
  prm.job_first = job_suns_h ? (const uint64_t*)c->jobs.p : nullptr;
  prm.job_suns = job_suns_h ? (const ssolh_sun*)((char*)c->jobs.p + (njobs + 1) * sizeof(uint64_t))
                            : nullptr;

  PathArgs args{};
  args.S = c->scn;
  args.SQ = c->shapeq;
  args.prm = prm;
  args.T = c->T;
  args.W = W;
  args.C = ctr;
  args.A = A;
  args.K = K;
  args.ovf = ovf;

  args.wave_in = args.wave_out = wave_n;
  args.in_n = &ctr->left;

  auto launch = [&](uint32_t blocks, auto k32, auto k64, auto kadj, auto ktrk) -> int {
    auto go = [&](auto kernel) { kernel<<<blocks, BLOCK, 0, c->stream>>>(args); };
    fp32 ? go(k32) : adj ? go(kadj) : trk ? go(ktrk) : go(k64);
    HIP_TRY(hipGetLastError());
    return 0;
  };
  auto start = [&](uint32_t count) {
    return launch((count + BLOCK - 1) / BLOCK, k_start<F32, false, false>,
                  k_start<F64, false, false>, k_start<F64, true, false>,
                  k_start<F64, false, true>);
  };
  // Paths that all fit on the chip at once (256 CUs of four SIMDs) run
  // through, unless their entries could fill the log. A further launch takes
  // 50 us beside its paths; one round and a third of waves leaves a last
  // round nearly empty (FP64 cavity of 5e5 paths: 4.75 ms at 2^18, 4.58 at
  // 3 * 2^16, 4.89 at 2^17).
  const uint32_t resident = (fp32 ? F32::WAVES : F64::WAVES) * 1024u * 64u;
  auto run_through = [&](uint32_t count) {
    return count <= resident && (!c->T.log_cap || count <= c->T.log_cap);
  };
  auto resume = [&](uint32_t count) {
    const uint32_t blocks = (count + BLOCK - 1) / BLOCK;
    return run_through(count)
               ? launch(blocks, k_resume<F32, false, false, true>,
                        k_resume<F64, false, false, true>, k_resume<F64, true, false, true>,
                        k_resume<F64, false, true, true>)
               : launch(blocks, k_resume<F32, false, false, false>,
                        k_resume<F64, false, false, false>, k_resume<F64, true, false, false>,
                        k_resume<F64, false, true, false>);
  };

  // The realisations first .. first + count - 1 in start-instance order:
  // drawn keys, grouped, or a stable radix sort of (key, index) (group_pays)
  auto order_starts = [&](uint64_t first, uint32_t count) -> int {
    uint32_t* key = (uint32_t*)c->queue[1].p;
    uint32_t *skey = key + part, *idx = skey + part, *order = idx + part;
    const uint32_t gg = (count + 255) / 256;
    const StartKeyOf<false> k64{c->scn, prm, first, c->ninstances};
    const StartKeyOf<true> k32{c->scn, prm, first, c->ninstances};
    if (group_starts) {
      const uint32_t gb = (count + GROUP_BLOCK - 1) / GROUP_BLOCK;
      if (fp32)
        k_group_rank<<<gb, GROUP_THREADS, 0, c->stream>>>(k32, nullptr, count, start_keys, key, skey);
      else
        k_group_rank<<<gb, GROUP_THREADS, 0, c->stream>>>(k64, nullptr, count, start_keys, key, skey);
      HIP_TRY(hipGetLastError());
      k_group_scan<<<1, GROUP_THREADS, 0, c->stream>>>(start_keys, nullptr, 0, 0, nullptr, nullptr);
      HIP_TRY(hipGetLastError());
      k_group_place<<<gg, 256, 0, c->stream>>>(key, skey, nullptr, count, start_keys, order);
      HIP_TRY(hipGetLastError());
      args.order = order;
      return 0;
    }
    if (fp32)
      k_start_keys<<<gg, 256, 0, c->stream>>>(k32, count, key, idx);
    else
      k_start_keys<<<gg, 256, 0, c->stream>>>(k64, count, key, idx);
    HIP_TRY(hipGetLastError());
    size_t sb = sort_bytes;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(c->start_sort.p, sb, key, skey, idx, order,
                                               (int)count, 0, (int)key_bits, c->stream));
    args.order = order;
    return 0;
  };

  float ms_path = 0;
  HIP_TRY(hipEventRecord(c->ev[0], c->stream));
  for (uint64_t first = 0; first < N; first += slots) {
    const uint32_t count = (uint32_t)std::min<uint64_t>(N - first, slots);
    args.first = first;
    args.count = count;
    args.order = nullptr;
    const bool wave = !refill || first == 0;
    k_path_begin<<<1, 1, 0, c->stream>>>(ctr, wave);
    HIP_TRY(hipGetLastError());
    if (orderable) if ((r = order_starts(first, count))) return r;
    HIP_TRY(hipEventRecord(c->ev[1], c->stream));
    PathQ from{(uint4*)c->queue[1].p, slots}, to{(uint4*)c->queue[0].p, slots};
    args.out = to;
    if ((r = start(count))) return r;
    // the paths that go on, from queue to queue, until a launch runs them
    // through; a few start in the places where k_start left them
    uint32_t going = count;
    args.list = nullptr;
    do {
      if (!run_through(going)) {
        const uint32_t w = (going + 63) / 64, ch = (w + SCAN_CHUNK - 1) / SCAN_CHUNK;
        k_scan_chunks<<<ch, SCAN_THREADS, 0, c->stream>>>(wave_n, w, wave_off, wave_chunk);
        HIP_TRY(hipGetLastError());
        k_scan_top<<<1, SCAN_THREADS, 0, c->stream>>>(ch, wave_chunk, &ctr->left, ctr);
        HIP_TRY(hipGetLastError());
        k_queue_list<<<(w + 3) / 4, 256, 0, c->stream>>>(wave_n, w, wave_off, wave_chunk, list);
        HIP_TRY(hipGetLastError());
        uint32_t left = 0;
        unsigned long long asked[LOG_SEGS * LOG_LINE], logged = 0;
        HIP_TRY(hipMemcpyAsync(&left, &ctr->left, sizeof(left), hipMemcpyDeviceToHost, c->stream));
        if (c->T.log_cap)
          HIP_TRY(hipMemcpyAsync(asked, c->T.log_n, log_segs * LOG_LINE * sizeof(asked[0]),
                                 hipMemcpyDeviceToHost, c->stream));
        HIP_TRY(hipStreamSynchronize(c->stream));
        if (left > going) {
          set_err("ssolh_solve: %u paths go on of %u", left, going);
          return SSOLH_ERR_LIMIT;
        }
        going = left;
        if (!going) break;
        args.list = list;
        // past half full, the log is summed before it overflows into atomics
        for (uint32_t s = 0; c->T.log_cap && s < log_segs; ++s)
          logged = std::max(logged, asked[s * LOG_LINE]);
        if (logged && logged >= c->T.log_seg / 2) if ((r = log_flush())) return r;
      }
      std::swap(from, to);
      args.in = from;
      args.out = to;
      if ((r = resume(going))) return r;
    } while (!run_through(going));
    HIP_TRY(hipEventRecord(c->ev[2], c->stream));
    if ((r = log_flush())) return r;
    if (first + slots < N) {  // the last chunk's events are read when the solve ends
      HIP_TRY(hipEventSynchronize(c->ev[2]));
      float t = 0;
      (void)hipEventElapsedTime(&t, c->ev[1], c->ev[2]);
      ms_path += t;
    }
  }
  // fold the stripes: into one buffer, copied whole to pinned host memory;
  // from the scratch array, in place
  const size_t parts[FOLD_PARTS] = {(size_t)njobs * 16, (size_t)c->nrcv * 40, (size_t)c->nsamp * 4,
                                    (size_t)c->nsamp * c->nrcv * 40, (size_t)c->nprim * 40,
                                    (size_t)c->nsamp};
  const uint32_t stripes[FOLD_PARTS] = {sg, sr, ss, sx, sp, ss};
  void* const src[FOLD_PARTS] = {c->T.global, c->T.rcv, c->T.samp, c->T.sxr, c->T.prim,
                                 c->T.samp_count};
  constexpr size_t head = (sizeof(Counters) + 63) / 64 * 64;
  size_t folded = head;
  for (size_t x : parts) folded += x * 8;
  FoldArgs fold{};
  fold.C = fold.C_out = ctr;
  c->F = c->T;
  c->staged = false;
  if (!arena) {
    if ((r = alloc(c->folded, folded))) return r;
    if (folded <= STAGE_MAX && c->stage_bytes < folded) {
      if (c->stage) (void)hipHostFree(c->stage);
      c->stage = nullptr;
      c->stage_bytes = 0;
      if (hipHostMalloc(&c->stage, folded, hipHostMallocDefault) == hipSuccess)
        c->stage_bytes = folded;
      else
        (void)hipGetLastError();  // then read from the device
    }
    c->staged = c->stage_bytes >= folded;
    fold.C_out = (Counters*)c->folded.p;
    double* d = (double*)((char*)c->folded.p + head);
    c->F.global = d; d += parts[0];
    c->F.rcv = d; d += parts[1];
    c->F.samp = d; d += parts[2];
    c->F.sxr = d; d += parts[3];
    c->F.prim = d; d += parts[4];
    c->F.samp_count = (unsigned long long*)d;
  }
  void* const dst[FOLD_PARTS] = {c->F.global, c->F.rcv, c->F.samp, c->F.sxr, c->F.prim,
                                 c->F.samp_count};
  uint32_t blocks = 0;
  for (int k = 0; k < FOLD_PARTS; ++k) {
    const bool whole = k == FOLD_PARTS - 1;
    const uint32_t cols = whole ? FOLD_THREADS
                                : FOLD_THREADS / std::min<uint32_t>(stripes[k], FOLD_ROWS);
    fold.part[k] = FoldPart{src[k], dst[k], parts[k], stripes[k], blocks, whole};
    blocks += (uint32_t)((parts[k] + cols - 1) / cols);
  }
  k_fold<<<blocks, FOLD_THREADS, 0, c->stream>>>(fold);
  HIP_TRY(hipGetLastError());
  if (c->nrcv && c->nsamp) {
    const dim3 grid((unsigned)((parts[1] + FOLD_THREADS / FOLD_ROWS - 1) / (FOLD_THREADS / FOLD_ROWS)),
                    std::min<uint32_t>((c->nsamp + 255) / 256, 64));
    k_fold_rcv<<<grid, FOLD_THREADS, 0, c->stream>>>(c->F.sxr, parts[1], c->nsamp, c->F.rcv);
    HIP_TRY(hipGetLastError());
  }
  if (c->staged)
    HIP_TRY(hipMemcpyAsync(c->stage, c->folded.p, folded, hipMemcpyDeviceToHost, c->stream));
  float total_ms = 0;
  HIP_TRY(hipEventRecord(c->ev[3], c->stream));
  HIP_TRY(hipStreamSynchronize(c->stream));
  (void)hipEventElapsedTime(&total_ms, c->ev[0], c->ev[3]);
  float last_ms = 0;
  (void)hipEventElapsedTime(&last_ms, c->ev[1], c->ev[2]);
  ms_path += last_ms;
  double rays = 0;  // counted beside job 0's global fields
  if (c->staged) {
    memcpy(&c->last, c->stage, sizeof(Counters));
    memcpy(&rays, (char*)c->stage + head + 13 * 8, sizeof(rays));
  } else {
    HIP_TRY(hipMemcpy(&c->last, fold.C_out, sizeof(Counters), hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(&rays, c->F.global + 13, sizeof(rays), hipMemcpyDeviceToHost));
  }
  c->segments = (uint64_t)rays;
  c->log_flushes += c->last.log_flushes;
  c->log_overflowed += c->last.log_over;
  if (trk) HIP_TRY(hipMemcpy(&c->trk_nvtx, c->trk_count.p, sizeof(c->trk_nvtx), hipMemcpyDeviceToHost));
  c->kernel_ms = total_ms;
  c->trace_ms = ms_path;  // tracing and shading are one kernel
  c->shade_ms = 0;
  c->iterations = c->last.iterations + c->last.gens;
  c->wavefronts = c->last.wavefronts;
  c->refilled = refill;
  return 0;
}

}  // namespace

extern "C" {

// `bytes` of the folded tallies at device address `src` (in c->F)
static int tallies_to(const ssolh_context* c, void* dst, const void* src, size_t bytes) {
  if (!bytes) return 0;
  if (c->staged) {
    memcpy(dst, (const char*)c->stage + ((const char*)src - (const char*)c->folded.p), bytes);
    return 0;
  }
  HIP_TRY(hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost));
  return 0;
}

SSOLH_API int ssolh_solve(ssolh_context* c, const struct ssolh_solve_args* a) {
  if (!c || !a || !a->realisations) { set_err("ssolh_solve: invalid arguments"); return SSOLH_ERR_ARG; }
  if (!c->has_scene) { set_err("ssolh_solve: no scene uploaded"); return SSOLH_ERR_ARG; }
  if (a->precision != SSOLH_FP64 && a->precision != SSOLH_FP32) {
    set_err("ssolh_solve: unknown precision %u", a->precision);
    return SSOLH_ERR_ARG;
  }
  HIP_TRY(hipSetDevice(c->device));
  const uint32_t npend = a->pending_entries ? a->pending_entries : 4;
  return run_solve(c, a->realisations, a->max_failed, a->rng_key, a->rng_counter,
                   a->precision == SSOLH_FP32, a->path_slots, npend, 1, nullptr, nullptr);
}

SSOLH_API int ssolh_solve_noalloc(ssolh_context* c, const struct ssolh_solve_args* a,
                                  struct ssolh_tallies* out) {
  if (!c || !a || !out || !a->realisations) {
    set_err("ssolh_solve_noalloc: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene) { set_err("ssolh_solve_noalloc: no scene uploaded"); return SSOLH_ERR_ARG; }
  if (a->precision != SSOLH_FP64 && a->precision != SSOLH_FP32) {
    set_err("ssolh_solve_noalloc: unknown precision %u", a->precision);
    return SSOLH_ERR_ARG;
  }
  if (a->graph_iterations) {
    set_err("ssolh_solve_noalloc: iterations are driven from the host (graph_iterations 0)");
    return SSOLH_ERR_ARG;
  }
  if (!c->scratch) { set_err("ssolh_solve_noalloc: no scratch array on this device"); return SSOLH_ERR_MEM; }
  HIP_TRY(hipSetDevice(c->device));
  // The solve's buffers come from the scratch array: the context's own
  // buffers are set aside for the call (nothing is freed or allocated) and
  // put back after it.
  DevBuf* bufs[] = {&c->start_sort, &c->queue[0], &c->queue[1], &c->list, &c->pend,
                    &c->tallies,    &c->trace_ovf};
  constexpr size_t NB = sizeof(bufs) / sizeof(bufs[0]);
  DevBuf saved[NB];
  for (size_t i = 0; i < NB; ++i) {
    saved[i] = *bufs[i];
    *bufs[i] = DevBuf{};
  }
  Arena arena{(char*)c->scratch, SCRATCH_BYTES, 0};
  const uint32_t npend = a->pending_entries ? a->pending_entries : 4;
  int r = run_solve(c, a->realisations, a->max_failed, a->rng_key, a->rng_counter,
                    a->precision == SSOLH_FP32, a->path_slots, npend, 1, nullptr, nullptr,
                    nullptr, nullptr, &arena);
  if (!r) r = ssolh_tallies_download(c, out);
  for (size_t i = 0; i < NB; ++i) *bufs[i] = saved[i];
  return r;
}

SSOLH_API int ssolh_solve_batch(ssolh_context* c, const struct ssolh_batch_args* a,
                                struct ssolh_batch_result* out) {
  if (!c || !a || !out || !a->nsuns || !a->suns || !a->realisations) {
    set_err("ssolh_solve_batch: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene) { set_err("ssolh_solve_batch: no scene uploaded"); return SSOLH_ERR_ARG; }
  if (a->precision != SSOLH_FP64 && a->precision != SSOLH_FP32) {
    set_err("ssolh_solve_batch: unknown precision %u", a->precision);
    return SSOLH_ERR_ARG;
  }
  if (a->nsuns > (1u << 24)) { set_err("ssolh_solve_batch: at most 2^24 suns"); return SSOLH_ERR_LIMIT; }
  std::vector<uint64_t> first(a->nsuns + 1, 0);
  for (uint32_t j = 0; j < a->nsuns; ++j) first[j + 1] = first[j] + a->realisations[j];
  if (!first[a->nsuns]) { set_err("ssolh_solve_batch: no realisation"); return SSOLH_ERR_ARG; }
  HIP_TRY(hipSetDevice(c->device));
  const uint32_t npend = a->pending_entries ? a->pending_entries : 4;
  const uint32_t njobs = a->nsuns;
  std::vector<ssolh_sun> suns(a->suns, a->suns + a->nsuns);
  int r = run_solve(c, first[a->nsuns], a->max_failed, a->rng_key, a->rng_counter,
                    a->precision == SSOLH_FP32, a->path_slots, npend, njobs, first.data(),
                    suns.data());
  if (r) return r;
  std::vector<double> g((size_t)njobs * 16);
  if ((r = tallies_to(c, g.data(), c->F.global, g.size() * sizeof(double)))) return r;
  for (uint32_t j = 0; j < njobs; ++j) {
    memcpy(out[j].global, &g[(size_t)j * 16], 12 * sizeof(double));
    out[j].realisation_count = (uint64_t)g[(size_t)j * 16 + 12];
  }
  return 0;
}

SSOLH_API int ssolh_solve_adjoint(ssolh_context* c, const struct ssolh_adjoint_args* a,
                                  double* grad) {
  if (!c || !a || !grad || !a->solve.realisations || !a->nparams || !a->inst_param || !a->axes) {
    set_err("ssolh_solve_adjoint: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene) { set_err("ssolh_solve_adjoint: no scene uploaded"); return SSOLH_ERR_ARG; }
  if (a->solve.precision != SSOLH_FP64) {
    set_err("ssolh_solve_adjoint: the adjoint runs in the FP64 form");
    return SSOLH_ERR_ARG;
  }
  for (uint32_t i = 0; i < c->ninstances; ++i) {
    if (a->inst_param[i] >= (int32_t)a->nparams) {
      set_err("ssolh_solve_adjoint: instance %u has parameter slot %d >= %u", i, a->inst_param[i],
              a->nparams);
      return SSOLH_ERR_ARG;
    }
  }
  HIP_TRY(hipSetDevice(c->device));
  AdjHost h{a->nparams, a->inst_param, a->axes, a->gmap, a->d_absorbed};
  const uint32_t npend = a->solve.pending_entries ? a->solve.pending_entries : 4;
  int r = run_solve(c, a->solve.realisations, a->solve.max_failed, a->solve.rng_key,
                    a->solve.rng_counter, false, a->solve.path_slots, npend, 1, nullptr, nullptr,
                    &h);
  if (r) return r;
  HIP_TRY(hipMemcpy(grad, c->adj_grad.p, (size_t)a->nparams * 3 * sizeof(double),
                    hipMemcpyDeviceToHost));
  double n = 0;
  if ((r = tallies_to(c, &n, c->F.global + 12, sizeof(double)))) return r;
  for (size_t i = 0; i < (size_t)a->nparams * 3; ++i) grad[i] = n > 0 ? grad[i] / n : 0.0;
  return 0;
}

SSOLH_API int ssolh_solve_tracked(ssolh_context* c, const struct ssolh_solve_args* a,
                                  const struct ssolh_track_args* t, uint64_t* nvertices) {
  if (!c || !a || !t || !nvertices || !a->realisations) {
    set_err("ssolh_solve_tracked: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->has_scene) { set_err("ssolh_solve_tracked: no scene uploaded"); return SSOLH_ERR_ARG; }
  if (a->precision != SSOLH_FP64) {
    set_err("ssolh_solve_tracked: paths are recorded by the FP64 form");
    return SSOLH_ERR_ARG;
  }
  if (!(t->sun_ray_length == t->sun_ray_length) || !(t->infinite_ray_length == t->infinite_ray_length)) {
    set_err("ssolh_solve_tracked: NaN ray length");
    return SSOLH_ERR_ARG;
  }
  HIP_TRY(hipSetDevice(c->device));
  TrackHost h{t->sun_ray_length, t->infinite_ray_length, t->max_vertices};
  const uint32_t npend = a->pending_entries ? a->pending_entries : 4;
  int r = run_solve(c, a->realisations, a->max_failed, a->rng_key, a->rng_counter, false,
                    a->path_slots, npend, 1, nullptr, nullptr, nullptr, &h);
  if (r) return r;
  *nvertices = c->trk_nvtx;
  return 0;
}

SSOLH_API int ssolh_track_download(ssolh_context* c, struct ssolh_track_vertex* v, uint64_t nv,
                                   uint8_t* types, uint64_t npaths) {
  if (!c || (nv && !v) || (npaths && !types)) {
    set_err("ssolh_track_download: invalid arguments");
    return SSOLH_ERR_ARG;
  }
  if (!c->trk_paths) { set_err("ssolh_track_download: no tracked solve"); return SSOLH_ERR_ARG; }
  if (nv > std::min<uint64_t>(c->trk_nvtx, c->trk_cap) || npaths > c->trk_paths) {
    set_err("ssolh_track_download: asked for %llu vertices and %llu paths, the solve holds %llu and %llu",
            (unsigned long long)nv, (unsigned long long)npaths,
            (unsigned long long)std::min<uint64_t>(c->trk_nvtx, c->trk_cap),
            (unsigned long long)c->trk_paths);
    return SSOLH_ERR_ARG;
  }
  HIP_TRY(hipSetDevice(c->device));
  if (nv) HIP_TRY(hipMemcpy(v, c->trk_vtx.p, nv * sizeof(ssolh_track_vertex), hipMemcpyDeviceToHost));
  if (npaths) HIP_TRY(hipMemcpy(types, c->trk_type.p, npaths, hipMemcpyDeviceToHost));
  return 0;
}

SSOLH_API int ssolh_tallies_download(ssolh_context* c, struct ssolh_tallies* o) {
  if (!c || !o) { set_err("ssolh_tallies_download: NULL argument"); return SSOLH_ERR_ARG; }
  HIP_TRY(hipSetDevice(c->device));
  const size_t n_rcv = (size_t)c->nrcv * 40, n_samp = (size_t)c->nsamp * 4;
  const size_t n_sxr = (size_t)c->nsamp * c->nrcv * 40, n_prim = (size_t)c->nprim * 40;
  double cnt0 = 0;
  int r = tallies_to(c, o->global, c->F.global, 12 * sizeof(double));
  if (!r) r = tallies_to(c, &cnt0, c->F.global + 12, sizeof(double));
  if (!r && o->receivers) r = tallies_to(c, o->receivers, c->F.rcv, n_rcv * 8);
  if (!r && o->sampled) r = tallies_to(c, o->sampled, c->F.samp, n_samp * 8);
  if (!r && o->sampled_count) r = tallies_to(c, o->sampled_count, c->F.samp_count, c->nsamp * 8);
  if (!r && o->sampled_x_receivers) r = tallies_to(c, o->sampled_x_receivers, c->F.sxr, n_sxr * 8);
  if (!r && o->primitives) r = tallies_to(c, o->primitives, c->F.prim, n_prim * 8);
  if (r) return r;
  o->realisation_count = (uint64_t)cnt0;
  o->failed_count = c->last.failed;
  o->segments = c->segments;
  o->pending_spills = c->last.spills;
  o->aborted = c->last.aborted;
  o->iterations = c->iterations;
  o->wavefronts = c->wavefronts;
  o->refilled = c->refilled;
  o->kernel_ms = c->kernel_ms;
  o->trace_ms = c->trace_ms;
  o->shade_ms = c->shade_ms;
  return 0;
}

SSOLH_API int ssolh_test_quadric_hits(ssolh_context* c, int quadric, const double qparam[4],
                                      uint32_t n, const double* org, const double* dir,
                                      const double* hint, double* t, double* normal) {
  if (!c || !n) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  double *d_o, *d_d, *d_h, *d_t, *d_n;
  HIP_TRY(hipMalloc(&d_o, n * 24)); HIP_TRY(hipMalloc(&d_d, n * 24));
  HIP_TRY(hipMalloc(&d_h, n * 8)); HIP_TRY(hipMalloc(&d_t, n * 8)); HIP_TRY(hipMalloc(&d_n, n * 24));
  HIP_TRY(hipMemcpy(d_o, org, n * 24, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_d, dir, n * 24, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_h, hint, n * 8, hipMemcpyHostToDevice));
  k_test_quadric<<<(n + 127) / 128, 128, 0, c->stream>>>(
      quadric, make_double4(qparam[0], qparam[1], qparam[2], qparam[3]), n, d_o, d_d, d_h, d_t, d_n);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipMemcpy(t, d_t, n * 8, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(normal, d_n, n * 24, hipMemcpyDeviceToHost));
  (void)hipFree(d_o); (void)hipFree(d_d); (void)hipFree(d_h); (void)hipFree(d_t); (void)hipFree(d_n);
  return 0;
}

SSOLH_API int ssolh_test_sun_dirs(ssolh_context* c, const struct ssolh_sun* sun, uint32_t n,
                                  const double* u, uint32_t nu, double* dir, uint32_t* used) {
  if (!c || !sun || !n || !nu || !u || !dir || !used) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  double *d_u, *d_o;
  uint32_t* d_used;
  HIP_TRY(hipMalloc(&d_u, (size_t)n * nu * 8)); HIP_TRY(hipMalloc(&d_o, n * 24));
  HIP_TRY(hipMalloc(&d_used, n * 4));
  HIP_TRY(hipMemcpy(d_u, u, (size_t)n * nu * 8, hipMemcpyHostToDevice));
  k_test_sun<<<(n + 127) / 128, 128, 0, c->stream>>>(*sun, n, d_u, nu, d_o, d_used);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipMemcpy(dir, d_o, n * 24, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(used, d_used, n * 4, hipMemcpyDeviceToHost));
  (void)hipFree(d_u); (void)hipFree(d_o); (void)hipFree(d_used);
  return 0;
}

SSOLH_API int ssolh_test_bsdf(ssolh_context* c, const struct ssolh_material* m, double eta_out,
                              double eta_in, double slab_eta, double slab_absorption, uint32_t n,
                              const double* wi, const double* normal, const double* u, uint32_t nu,
                              double* wo, double* weight, int* lobe) {
  if (!c || !m || !n || !nu || !wi || !normal || !u || !wo || !weight || !lobe) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  double *d_wi, *d_n, *d_u, *d_wo, *d_w;
  int* d_l;
  HIP_TRY(hipMalloc(&d_wi, n * 24)); HIP_TRY(hipMalloc(&d_n, n * 24));
  HIP_TRY(hipMalloc(&d_u, (size_t)n * nu * 8)); HIP_TRY(hipMalloc(&d_wo, n * 24));
  HIP_TRY(hipMalloc(&d_w, n * 8)); HIP_TRY(hipMalloc(&d_l, n * 4));
  HIP_TRY(hipMemcpy(d_wi, wi, n * 24, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_n, normal, n * 24, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_u, u, (size_t)n * nu * 8, hipMemcpyHostToDevice));
  k_test_bsdf<<<(n + 127) / 128, 128, 0, c->stream>>>(
      *m, make_double4(eta_out, eta_in, slab_eta, slab_absorption), n, d_wi, d_n, d_u, nu, d_wo,
      d_w, d_l);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipMemcpy(wo, d_wo, n * 24, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(weight, d_w, n * 8, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(lobe, d_l, n * 4, hipMemcpyDeviceToHost));
  (void)hipFree(d_wi); (void)hipFree(d_n); (void)hipFree(d_u); (void)hipFree(d_wo);
  (void)hipFree(d_w); (void)hipFree(d_l);
  return 0;
}

SSOLH_API int ssolh_test_threefry(ssolh_context* c, uint32_t n, const uint64_t* ctr,
                                  const uint64_t* key, uint64_t* out) {
  if (!c || !n) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  uint64_t *d_c, *d_k, *d_o;
  HIP_TRY(hipMalloc(&d_c, n * 32)); HIP_TRY(hipMalloc(&d_k, n * 32)); HIP_TRY(hipMalloc(&d_o, n * 32));
  HIP_TRY(hipMemcpy(d_c, ctr, n * 32, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(d_k, key, n * 32, hipMemcpyHostToDevice));
  k_test_threefry<<<(n + 127) / 128, 128, 0, c->stream>>>(n, d_c, d_k, d_o);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipMemcpy(out, d_o, n * 32, hipMemcpyDeviceToHost));
  (void)hipFree(d_c); (void)hipFree(d_k); (void)hipFree(d_o);
  return 0;
}

SSOLH_API int ssolh_test_group(ssolh_context* c, uint32_t n, uint32_t nkeys, const uint32_t* key,
                               uint32_t* order, uint32_t* offsets) {
  if (!c || !n || !nkeys || nkeys > GROUP_KEYS || !key || !order || !offsets) return SSOLH_ERR_ARG;
  for (uint32_t i = 0; i < n; ++i)
    if (key[i] >= nkeys) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  DevBuf keys, work;
  int r = dev_alloc(keys, 3 * (size_t)n * 4);
  if (!r) r = dev_alloc(work, GROUP_BYTES / 2);
  const auto run = [&]() -> int {
    uint32_t *d_key = (uint32_t*)keys.p, *d_rank = d_key + n, *d_order = d_rank + n;
    const GroupKeys g{(uint32_t*)work.p, (uint32_t*)work.p + GROUP_KEYS, nkeys};
    HIP_TRY(hipMemsetAsync(work.p, 0, GROUP_KEYS * 4, c->stream));
    HIP_TRY(hipMemcpyAsync(d_key, key, (size_t)n * 4, hipMemcpyHostToDevice, c->stream));
    k_group_rank<<<(n + GROUP_BLOCK - 1) / GROUP_BLOCK, GROUP_THREADS, 0, c->stream>>>(
        LogKeyOf{d_key}, nullptr, n, g, nullptr, d_rank);
    HIP_TRY(hipGetLastError());
    k_group_scan<<<1, GROUP_THREADS, 0, c->stream>>>(g, nullptr, 0, 0, nullptr, nullptr);
    HIP_TRY(hipGetLastError());
    k_group_place<<<(n + 255) / 256, 256, 0, c->stream>>>(d_key, d_rank, nullptr, n, g, d_order);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipStreamSynchronize(c->stream));
    HIP_TRY(hipMemcpy(order, d_order, (size_t)n * 4, hipMemcpyDeviceToHost));
    HIP_TRY(hipMemcpy(offsets, g.offsets, ((size_t)nkeys + 1) * 4, hipMemcpyDeviceToHost));
    return 0;
  };
  if (!r) r = run();
  (void)hipFree(keys.p);
  (void)hipFree(work.p);
  return r;
}

SSOLH_API int ssolh_test_wave_sum(ssolh_context* c, uint32_t nwaves, const double* in,
                                  double* out) {
  if (!c || !nwaves || !in || !out) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  double *d_in, *d_out;
  const size_t bytes = (size_t)nwaves * 64 * sizeof(double);
  HIP_TRY(hipMalloc(&d_in, bytes)); HIP_TRY(hipMalloc(&d_out, bytes));
  HIP_TRY(hipMemcpy(d_in, in, bytes, hipMemcpyHostToDevice));
  k_test_wave_sum<<<nwaves, 64, 0, c->stream>>>(d_in, d_out);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(c->stream));
  HIP_TRY(hipMemcpy(out, d_out, bytes, hipMemcpyDeviceToHost));
  (void)hipFree(d_in); (void)hipFree(d_out);
  return 0;
}

SSOLH_API int ssolh_test_trace_stack(ssolh_context* c, uint32_t lds_cap, uint32_t* bound) {
  if (!c || !(lds_cap == 0 || lds_cap == 16 || lds_cap == 24 || lds_cap == 32)) {
    set_err("ssolh_test_trace_stack: cap %u not 0, 16, 24 or 32", lds_cap);
    return SSOLH_ERR_ARG;
  }
  c->lds_stack_cap = lds_cap;
  if (bound) *bound = c->has_scene ? c->stack_depth : 0;
  return 0;
}

SSOLH_API int ssolh_test_prim_log(ssolh_context* c, uint32_t records, uint32_t* flushes,
                                  uint64_t* overflowed) {
  if (!c) return SSOLH_ERR_ARG;
  c->log_cap_test = records;
  if (flushes) *flushes = c->log_flushes;
  if (overflowed) *overflowed = c->log_overflowed;
  return 0;
}

SSOLH_API int ssolh_copy_bandwidth(ssolh_context* c, size_t bytes, int reps, double* gbs) {
  if (!c || bytes < 16 || reps < 1 || !gbs) return SSOLH_ERR_ARG;
  HIP_TRY(hipSetDevice(c->device));
  const size_t n = bytes / 16;
  uint4 *a, *b;
  HIP_TRY(hipMalloc(&a, n * 16));
  HIP_TRY(hipMalloc(&b, n * 16));
  HIP_TRY(hipMemsetAsync(a, 0x3c, n * 16, c->stream));
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0)); HIP_TRY(hipEventCreate(&e1));
  const unsigned grid = (unsigned)std::min<size_t>((n + 255) / 256, 8192);
  k_copy<<<grid, 256, 0, c->stream>>>(a, b, n);  // warm
  HIP_TRY(hipEventRecord(e0, c->stream));
  for (int r = 0; r < reps; ++r) k_copy<<<grid, 256, 0, c->stream>>>(a, b, n);
  HIP_TRY(hipEventRecord(e1, c->stream));
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipEventSynchronize(e1));
  float ms = 0;
  HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
  *gbs = 2.0 * (double)(n * 16) * reps / (ms * 1e-3) / 1e9;
  (void)hipEventDestroy(e0); (void)hipEventDestroy(e1);
  (void)hipFree(a); (void)hipFree(b);
  return 0;
}

}  // extern "C"
