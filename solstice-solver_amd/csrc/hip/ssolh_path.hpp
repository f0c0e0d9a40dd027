// Path kernels (included by ssolh.hip inside its anonymous namespace). One
// launch takes every path in flight one ray further: a lane traces its
// path's ray, shades the hit and, if the path goes on, appends it to the
// queue of the next launch, so the queue is dense, its records are read and
// written coalesced, and waves stay full. Only the ray is held in registers
// through the traversal; the rest of the path's state is read from the queue
// once the hit is known (k_resume) or waits in LDS (k_start, which draws the
// start point and traces the shadow ray). A launch of few paths keeps them in
// place and follows each to its end. Form: the FP64 form F64 or the FP32 form
// F32 (ssolh_fp32.hpp).

// What bounds them: vector issue and the traversal's node loads (rocprofv3,
// 1e8 FP64 paths: k_start 73 % VALU busy with 78 % of the lanes active, the
// passes after it 57-63 % with 45-65 %, texture addresser 47-61 %); HBM
// traffic is 1.7 TB/s. Waves per SIMD, measured on the 10k-heliostat field (3e7 FP64,
// 1e7 FP32 paths): FP64 16.3 ms at three (no spills), 18.0 at four (60 to 132
// bytes per lane spilled); FP32 5.3 ms at four, 5.7 at three. Separate
// generate, trace, shade and compaction launches, which the path kernels
// replace, took 21.2 and 6.8 ms there.
struct F64 {
  using real = double;
  using vec = d3;
  using Rng = PathRng;
  using Ray = RayRec;
  using Hit = HitRec;
  using Tracer = Tracer64;
  static constexpr int WAVES = 3;  // per SIMD
};
struct F32 {
  using real = float;
  using vec = f3;
  using Rng = PathRng32;
  using Ray = RayRec32;
  using Hit = HitRec32;
  using Tracer = Tracer32;
  static constexpr int WAVES = 4;
};

// A realisation in flight. The position and direction of the point a ray
// leaves are those of the ray (its origin is the last real point, also past
// a virtual one, whose ray keeps that origin).
template <class F>
struct Path {
  using real = typename F::real;
  typename F::Ray r;   // the ray to trace; (iss_from, prim_from) and the side bits: its point
  real pv[4];          // outgoing weights of the last real point (3); [3]: the initial flux
                       // until the first shading, then the incoming flux of the last virtual
                       // point crossed
  real pd[3];          // pending absorbed_by_receivers, extinguished, other
  typename F::vec n0;  // normal of the start point, until the first shading
  real wl, cosf;       // wavelength, cos factor
  uint32_t slot;       // place among the wavefront's realisations (pending entries, adjoint, track)
  uint32_t pid;        // realisation id - first
  uint32_t block;      // next block of its random stream
  uint32_t flags;      // PF_*
  uint32_t depth, media;         // in medium | out medium << 16
  uint32_t samp, job;            // sampled slot, sun
  uint32_t score, interval;      // roulette
  uint32_t npk, nqk;             // pending receiver and per-primitive entries held
  int fin;                       // FIN_*
  // of a finished path: dkey != NONE: its last hit absorbed it on receiver
  // key dkey, primitive key dpkey (or NONE), with pv = in0, in1, in2, kabs;
  // else pv[0] = missing, pv[1] = shadowed
  uint32_t dkey, dpkey;
};

// A queue of paths: planes of 16 bytes by place, cap places each. A launch
// writes the paths of its wave w that go on to places 64 w, 64 w + 1, ... and
// their number to n[w]; k_queue_list then lists the places in that order.
constexpr uint32_t RAY_PLANES64 = 4, STATE_PLANES64 = 7;
constexpr uint32_t RAY_PLANES32 = 3, STATE_PLANES32 = 4;
struct PathQ {
  uint4* p;
  uint32_t cap;
};

// Pending entries of the wavefront's realisations (receivers hit in
// passing): key and ten weights of entry k of a slot at slot * npend + k;
// Path::npk, nqk count the entries in use. The weights are of the form's
// type. Bound by the lines they touch: the paths of a wave hold ever sparser
// slots, so an entry's weights lie side by side (80 or 40 bytes, one or two
// lines) and not by weight, where each of the ten would be a line of its own.
struct Pending {
  uint32_t *pkey, *qkey;   // receiver, per-primitive keys: [slot][entry]
  void *pval, *qval;       // [slot][entry][10]
  uint32_t npend;
};
// Two neighbouring weights of an entry
template <typename R>
struct alignas(2 * sizeof(R)) WeightPair {
  R a, b;
};

struct PathArgs {
  DScene S;
  const ShapeQ* SQ;        // FP32 form
  SolveParams prm;
  Tallies T;
  Pending W;
  Counters* C;
  AdjParams A;
  TrackParams K;
  TOvf ovf;
  uint64_t first;          // first realisation of the wavefront
  const uint32_t* order;   // its realisations in slot order, or null (identity)
  uint32_t count;          // k_start: realisations to start
  PathQ in, out;           // k_resume: paths to take on; paths left for the next launch
  const uint32_t* list;    // places in `in`, in_n of them; null: the first count places, of
                           // which wave w takes the first wave_in[w] of its 64
  const unsigned* in_n;
  const uint32_t* wave_in;
  uint32_t* wave_out;      // paths each wave leaves for the next launch
};

// Sample triangle of a start point from the first uniform of its stream
// (alias table over the sampling proxy, by area)
__device__ __forceinline__ uint32_t alias_pick(const DScene& S, double u0) {
  const double x = u0 * (double)S.nstris;
  uint32_t i = (uint32_t)x;
  if (i >= S.nstris) i = S.nstris - 1;
  const ssolh_alias al = S.alias[i];
  return (x - (double)i) < al.prob ? i : al.alias;
}

// The form-independent state of a path at its start point
template <class F>
__device__ __forceinline__ void begin_path(Path<F>& p, typename F::real w0, uint32_t block,
                                           uint32_t med, uint32_t samp, uint32_t job) {
  p.pv[0] = p.pv[1] = p.pv[2] = p.pv[3] = w0;
  p.pd[0] = p.pd[1] = p.pd[2] = 0;
  p.block = block;
  p.flags = PF_ACTIVE;
  p.depth = 0;
  p.media = med | (med << 16);
  p.samp = samp;
  p.job = job;
  p.score = 0;
  p.interval = 64;
  p.npk = p.nqk = 0;
}

// Start of a realisation and its shadow ray (reference point_init,
// src/ssol_solver.c:207-358)
template <bool ADJ, bool TRACK>
__device__ __forceinline__ void start_path(const PathArgs& a, Path<F64>& p) {
  const DScene& S = a.S;
  const uint64_t path = a.first + p.pid;
  PathRng rng;
  rng.init(a.prm.key, a.prm.counter + path, 0);
  // area-weighted primitive through the alias table, uniform point
  const double u0 = rng.next(), u1 = rng.next(), u2 = rng.next();
  const uint32_t idx = alias_pick(S, u0);
  const ssolh_sample_tri st = S.stris[idx];
  const ssolh_instance& inst = S.insts[st.instance];
  const double sq = sqrt(u1);
  const double b0 = 1 - sq, b1 = sq * (1 - u2), b2 = sq * u2;
  const d3 v0 = ld3(st.v0), v1 = ld3(st.v1), v2 = ld3(st.v2);
  const d3 T = mk(inst.transform[9], inst.transform[10], inst.transform[11]);
  d3 pos = mul(inst.transform, v0 * b0 + v1 * b1 + v2 * b2) + T;
  const d3 ns = normalize(tmul(inst.inv_linear, cross(v2 - v0, v1 - v0)));

  const uint32_t job = job_of(a.prm, path);
  const ssolh_sun& sun = job_sun(S, a.prm, job);
  const d3 dir = sample_sun(sun, rng);
  p.wl = sample_wavelength(S.spectra, sun.wl_spectrum, rng.next());

  const uint32_t iss = inst.isshape_first + st.sshape;
  const IssInfo is = S.iss[iss];
  d3 N = ns;
  const bool punched = is.shape_type == SSOLH_SHAPE_PUNCHED;
  if (punched) {
    // lift onto the quadric (src/ssol_shape.c:1408-1447)
    const ssolh_shape& sh = S.shapes[is.shape];
    const ssolh_inst_sshape& q = S.isshapes[iss];
    d3 loc = mul(q.R_inv, pos - ld3(q.T));
    loc.z = quadric_z(sh.quadric, sh.qparam, loc.x, loc.y);
    N = normalize(tmul(q.R_inv, quadric_grad(sh.quadric, sh.qparam, loc)));
    pos = mul(q.R, loc) + ld3(q.T);
  }
  uint32_t side = SSOL_FRONT_;
  if (dot(N, dir) >= 0) { side = SSOL_BACK_; N = -N; }

  const d3 sun0 = ld3(sun.dir);
  const double surface_sun_cos = dot(N, dir);
  const double surface_sun0_cos = fabs(dot(sun0, N));
  const double sun0_sun_cos = dot(sun0, dir);
  const double proxy_cos = punched ? fabs(dot(ns, N)) : 1.0;
  const double w0 = sun.dni * S.S_proxy * fabs(surface_sun_cos / (proxy_cos * sun0_sun_cos));
  p.cosf = S.S_proxy / S.S * surface_sun0_cos / proxy_cos;

  const ssolh_material& m = S.mtls[side == SSOL_FRONT_ ? is.mtl_front : is.mtl_back];
  const uint32_t med = start_medium(S, m, side);

  if (TRACK) {
    // sun point and start point (src/ssol_solver.c:909-921)
    a.K.seq[p.slot] = 0;
    if (a.K.sun_len > 0) track_vertex(a.K, p.slot, path, pos - dir * a.K.sun_len, sun.dni);
    track_vertex(a.K, p.slot, path, pos, w0);
    a.K.pos[p.slot] = make_double4(pos.x, pos.y, pos.z, 0);
  }
  if (ADJ) {
    // w0 is proportional to |N.w|: d log w0 / d angle = ((a x N).w) / (N.w)
    const int32_t pp = a.A.inst_param[st.instance];
    double4 sc = make_double4(0, 0, 0, 0);
    if (pp >= 0) {
      const d3 a1 = ld3(a.A.axes + 6 * pp), a2 = ld3(a.A.axes + 6 * pp + 3);
      sc.x = dot(cross(a1, N), dir) / surface_sun_cos;
      sc.y = dot(cross(a2, N), dir) / surface_sun_cos;
    }
    a.A.s[p.slot] = sc;
    a.A.p[p.slot] = pp >= 0 ? (uint32_t)pp : NONE;
  }

  p.n0 = N;
  begin_path(p, w0, rng.block, med, (uint32_t)inst.sampled, job);

  // shadow ray toward the sun (src/ssol_solver.c:325-352)
  p.r.ox = pos.x; p.r.oy = pos.y; p.r.oz = pos.z;
  p.r.dx = -dir.x; p.r.dy = -dir.y; p.r.dz = -dir.z;
  p.r.tmin = 0;
  p.r.iss_from = iss;
  p.r.prim_from = st.prim;
  p.r.flags = (side << RF_SIDE_SHIFT) | RF_DISCARD_VIRTUAL | RF_REVERSED | RF_ANY_HIT;
}

// Sample triangle of a start point from the first two uniforms of its
// stream (FP32 form of alias_pick)
__device__ __forceinline__ uint32_t alias_pick32(const DScene& S, float u0, float uc) {
  uint32_t i = (uint32_t)(u0 * (float)S.nstris);
  if (i >= S.nstris) i = S.nstris - 1;
  const ssolh_alias al = S.alias[i];
  return (double)uc < al.prob ? i : al.alias;
}

// start_path in the FP32 form
__device__ __forceinline__ void start_path32(const PathArgs& a, Path<F32>& p) {
  const DScene& S = a.S;
  const ShapeQ* SQ = a.SQ;
  const uint64_t path = a.first + p.pid;
  PathRng32 rng;
  rng.init(a.prm.key, a.prm.counter + path, 0);
  const float u0 = rng.next(), uc = rng.next(), u1 = rng.next(), u2 = rng.next();
  const uint32_t idx = alias_pick32(S, u0, uc);
  const ssolh_sample_tri st = S.stris[idx];
  const ssolh_instance& inst = S.insts[st.instance];
  const float sq = sqrtf(u1);
  const float b0 = 1 - sq, b1 = sq * (1 - u2), b2 = sq * u2;
  const f3 v0 = ldf(st.v0), v1 = ldf(st.v1), v2 = ldf(st.v2);
  const f3 p_obj = v0 * b0 + v1 * b1 + v2 * b2;
  f3 off = mulf(inst.transform, p_obj);
  const f3 ns = normalize(tmulf(inst.inv_linear, cross(v2 - v0, v1 - v0)));

  const uint32_t job = job_of(a.prm, path);
  const ssolh_sun& sun = job_sun(S, a.prm, job);
  const f3 dir = sample_sun32(sun, rng);
  p.wl = (float)sample_wavelength(S.spectra, sun.wl_spectrum, (double)rng.next());

  const uint32_t iss = inst.isshape_first + st.sshape;
  const IssInfo is = S.iss[iss];
  f3 N = ns;
  const bool punched = is.shape_type == SSOLH_SHAPE_PUNCHED;
  if (punched) {
    // lift onto the quadric in FP64 (src/ssol_shape.c:1408-1447)
    const ssolh_shape& sh = S.shapes[is.shape];
    const ShapeQ& q = SQ[is.shape];
    d3 loc = mul(q.Rinv, tod(p_obj) - ld3(q.t));
    loc.z = quadric_z(sh.quadric, sh.qparam, loc.x, loc.y);
    N = tof(normalize(tmul(S.isshapes[iss].R_inv, quadric_grad(sh.quadric, sh.qparam, loc))));
    const ssolh_inst_sshape& qs = S.isshapes[iss];
    const d3 pw = mul(qs.R, loc) + ld3(qs.T) - inst_T(inst);
    off = tof(pw);
  }
  uint32_t side = SSOL_FRONT_;
  if (dot(N, dir) >= 0) { side = SSOL_BACK_; N = -N; }

  const f3 sun0 = mkf((float)sun.dir[0], (float)sun.dir[1], (float)sun.dir[2]);
  const float surface_sun_cos = dot(N, dir);
  const float surface_sun0_cos = fabsf(dot(sun0, N));
  const float sun0_sun_cos = dot(sun0, dir);
  const float proxy_cos = punched ? fabsf(dot(ns, N)) : 1.0f;
  const float w0 = (float)(sun.dni * S.S_proxy) * fabsf(surface_sun_cos / (proxy_cos * sun0_sun_cos));
  p.cosf = (float)(S.S_proxy / S.S) * surface_sun0_cos / proxy_cos;

  const ssolh_material& m = S.mtls[side == SSOL_FRONT_ ? is.mtl_front : is.mtl_back];
  const uint32_t med = start_medium(S, m, side);


  p.n0 = N;
  begin_path(p, w0, rng.block, med, (uint32_t)inst.sampled, job);
  p.r.ox = off.x; p.r.oy = off.y; p.r.oz = off.z;
  p.r.base = st.instance;
  p.r.dx = -dir.x; p.r.dy = -dir.y; p.r.dz = -dir.z;
  p.r.tmin = 0;
  p.r.iss_from = iss;
  p.r.prim_from = st.prim;
  p.r.flags = (side << RF_SIDE_SHIFT) | RF_DISCARD_VIRTUAL | RF_REVERSED | RF_ANY_HIT;
}

// The ten receiver weights of a hit (ssol_mc_receiver field order)
template <typename R>
__device__ __forceinline__ void receiver_weights(R in0, R in1, R in2, R kabs, R w[10]) {
  w[0] = in0; w[1] = in1; w[2] = in2;
  w[3] = in2 - in0; w[4] = in1 - in0;
  w[5] = in0 * kabs; w[6] = in1 * kabs; w[7] = in2 * kabs;
  w[8] = (in2 - in0) * kabs; w[9] = (in1 - in0) * kabs;
}

// Add the weights of a hit to the path's pending entries (n of the npend at
// keys, vals in use); false when npend entries hold other keys.
template <typename R>
__device__ bool pend_add(uint32_t* keys, R* vals, uint32_t npend, uint32_t& n, uint32_t key,
                         const R* w) {
  for (uint32_t k = 0; k < n; ++k) {
    if (keys[k] != key) continue;
    auto* v = (WeightPair<R>*)(vals + k * 10);
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      const WeightPair<R> x = v[f];
      v[f] = {x.a + w[2 * f], x.b + w[2 * f + 1]};
    }
    return true;
  }
  if (n >= npend) return false;
  keys[n] = key;
  auto* v = (WeightPair<R>*)(vals + n * 10);
#pragma unroll
  for (int f = 0; f < 5; ++f) v[f] = {w[2 * f], w[2 * f + 1]};
  ++n;
  return true;
}

// Weights that found no pending entry are flushed as a term of their own
template <typename R>
__device__ void spill(double* base, uint64_t key, const R* w, unsigned long long* spills) {
  atomicAdd(spills, 1ull);
  for (int f = 0; f < 10; ++f) {
    const double x = w[f];
    atomic_add(base + key * 20 + 2 * f, x);
    atomic_add(base + key * 20 + 2 * f + 1, x * x);
  }
}

// The same of a primitive, through the log (see prim_add; any lanes may call)
template <typename R>
__device__ void spill_prim(const Tallies& T, uint32_t key, const R* w, unsigned long long* spills) {
  if (T.log_cap) {
    const uint32_t s = blockIdx.x & T.log_mask;
    const unsigned long long pos = atomicAdd(T.log_n + s * LOG_LINE, 1ull);
    if (pos < T.log_seg) {
      atomicAdd(spills, 1ull);
      log_record(T, (uint64_t)s * T.log_seg + pos, key, w, 1.0);
      return;
    }
  }
  spill(T.prim + (size_t)(blockIdx.x & T.mask_p) * T.nprim * 40u, key, w, spills);
}

// The point a ray hit, relative to its origin's frame, and the unit normal
// there. The FP32 form rebases the position on the hit instance.
__device__ __forceinline__ void hit_point(const DScene& S, const RayRec& r, const HitRec& h,
                                          d3 dir, d3& pos, d3& N, uint32_t&) {
  N = normalize(mk(h.nx, h.ny, h.nz));
  const double t = S.iss[h.iss].shape_type == SSOLH_SHAPE_MESH ? h.t : h.qdst;
  pos = mk(r.ox, r.oy, r.oz) + dir * t;
}
__device__ __forceinline__ void hit_point(const DScene& S, const RayRec32&, const HitRec32& h,
                                          f3, f3& pos, f3& N, uint32_t& base) {
  pos = mkf(h.px, h.py, h.pz);
  N = mkf(h.nx, h.ny, h.nz);
  base = S.iss[h.iss].inst;
}
__device__ __forceinline__ d3 vec_of(double x, double y, double z) { return mk(x, y, z); }
__device__ __forceinline__ f3 vec_of(float x, float y, float z) { return mkf(x, y, z); }
__device__ __forceinline__ uint32_t base_of(const RayRec&) { return 0; }
__device__ __forceinline__ uint32_t base_of(const RayRec32& r) { return r.base; }
__device__ __forceinline__ void set_base(RayRec&, uint32_t) {}
__device__ __forceinline__ void set_base(RayRec32& r, uint32_t b) { r.base = b; }
__device__ __forceinline__ double exp_of(double x) { return exp(x); }
__device__ __forceinline__ float exp_of(float x) { return expf(x); }
template <class Rng>
__device__ __forceinline__ double bsdf_of(const ssolh_material& m, double eta_out, double eta_in,
                                          double slab_eta, double slab_abs, d3 wi, d3 N, Rng& rng,
                                          d3& wo, int& lobe, d3* hm) {
  return bsdf_sample(m, eta_out, eta_in, slab_eta, slab_abs, wi, N, rng, wo, lobe, hm);
}
template <class Rng>
__device__ __forceinline__ float bsdf_of(const ssolh_material& m, float eta_out, float eta_in,
                                         float slab_eta, float slab_abs, f3 wi, f3 N, Rng& rng,
                                         f3& wo, int& lobe, f3*) {
  return bsdf_sample32(m, eta_out, eta_in, slab_eta, slab_abs, wi, N, rng, wo, lobe);
}

// The reference loop body around one traced ray (trace_radiative_path,
// src/ssol_solver.c:939-1086): the tail of the iteration that traced it
// (miss, segment extinction, Russian roulette, point update) and the head of
// the next one (extinction, BSDF or virtual pass-through, receiver weights).
// True: p.r is the path's next ray; false: the path ended (p.fin, see Path).
template <class F, bool ADJ, bool TRACK>
__device__ __forceinline__ bool shade_path(const PathArgs& a, Path<F>& p,
                                           const typename F::Hit& h) {
  using real = typename F::real;
  using vec = typename F::vec;
  const DScene& S = a.S;
  const Tallies& T = a.T;
  const uint64_t path = a.first + p.pid;
  const uint32_t flags0 = p.flags;
  uint32_t in_med = p.media & 0xFFFFu, out_med = p.media >> 16;
  uint32_t iss = p.r.iss_from, prim = p.r.prim_from;
  uint32_t side = (p.r.flags >> RF_SIDE_SHIFT) & 3u;
  typename F::Rng rng;
  rng.init(a.prm.key, a.prm.counter + path, p.block);
  vec dir = vec_of(p.r.dx, p.r.dy, p.r.dz);
  if (!(flags0 & PF_STAGE_BOUNCE)) dir = -dir;  // the shadow ray points at the sun
  const vec rdir = dir;
  vec pos = vec_of(p.r.ox, p.r.oy, p.r.oz), N = p.n0;
  uint32_t base = base_of(p.r);
  real hit_t = 0;
  real missing = 0, shadowed = 0;
  p.fin = FIN_NONE;
  p.dkey = p.dpkey = NONE;
  bool direct = false;
  real din0 = 0, din1 = 0, din2 = 0, dabs = 0;

  if (!(flags0 & PF_STAGE_BOUNCE)) {
    // result of the shadow ray
    if (h.iss != NONE) {
      p.fin = FIN_DONE;
      shadowed = p.pv[3];  // the initial flux
    }
  } else {
    // tail of the iteration that traced this ray
    const bool hit_virtual = (flags0 & PF_HIT_VIRTUAL) != 0;
    const bool in_atm = (flags0 & PF_IN_ATM) != 0;
    // flux that left the emitting point
    const real left = hit_virtual ? p.pv[3] : p.pv[0];
    if (h.iss == NONE) {
      // escape point (src/ssol_solver.c:1012-1019)
      if constexpr (TRACK) if (a.K.inf_len > 0) {
        const double4 kp = a.K.pos[p.slot];
        track_vertex(a.K, p.slot, path, mk(kp.x, kp.y, kp.z) + dir * a.K.inf_len, left);
      }
      if (out_med != S.air) {
        p.fin = FIN_FAILED;  // ray lost outside air
      } else {
        // past a virtual point the segment from the last real point ends at
        // the virtual one (a real point's segment was counted at that point)
        if (hit_virtual) {
          const real absorbed = p.pv[0] - p.pv[3];
          if (in_atm) p.pd[1] += absorbed; else p.pd[2] += absorbed;
        }
        p.fin = FIN_DONE;
        missing = left;
      }
    } else {
      p.depth += hit_virtual ? 0u : 1u;
      if (p.depth > p.interval && p.depth % p.interval == 1) {
        if (rng.next() > real(0.5)) {
          p.score += 1;
          p.interval = 16;
        } else {
          p.fin = FIN_KILLED;
        }
      }
      if (p.fin == FIN_NONE) {
        // point_update_from_hit (src/ssol_solver.c:360-411)
        iss = h.iss;
        prim = h.prim;
        hit_point(S, p.r, h, dir, pos, N, base);
        if (dot(dir, N) < 0) side = SSOL_FRONT_;
        else { side = SSOL_BACK_; N = -N; }
        in_med = out_med;
        hit_t = h.t;
        if constexpr (TRACK) track_vertex(a.K, p.slot, path, pos, left);  // src/ssol_solver.c:1080-1083
      }
    }
  }

  if (p.fin == FIN_NONE) {
    const IssInfo is = S.iss[iss];
    const ssolh_material& m = S.mtls[side == SSOL_FRONT_ ? is.mtl_front : is.mtl_back];
    const bool in_atm = in_med == S.air;
    const bool receiver = (is.receiver_mask & side) != 0;
    const bool virt = m.type == SSOLH_MTL_VIRTUAL;
    if (receiver) p.flags |= PF_HIT_RECEIVER;
    real trans = 1;
    if (hit_t > 0) {
      const real k = (real)data_value(S.spectra, S.media[in_med].extinction, p.wl);
      if (k > 0) trans = exp_of(-k * hit_t);
    }
    const real in0 = p.pv[0] * trans;
    const real in1 = in_atm ? p.pv[1] : p.pv[1] * trans;
    const real in2 = !in_atm ? p.pv[2] : p.pv[2] * trans;
    real out0, out1, out2, kabs;
    uint32_t next_med = in_med;
    if (virt) {
      out0 = in0; out1 = in1; out2 = in2; kabs = 0;
    } else {
      real eta_out = 1, eta_in = 1, slab_eta = 1, slab_abs = 0;
      if (m.type == SSOLH_MTL_DIELECTRIC) {
        if ((uint32_t)m.medium_out != in_med) p.fin = FIN_FAILED;
        eta_out = (real)data_value(S.spectra, S.media[m.medium_out].refractive_index, p.wl);
        eta_in = (real)data_value(S.spectra, S.media[m.medium_in].refractive_index, p.wl);
      } else if (m.type == SSOLH_MTL_THIN_DIELECTRIC) {
        eta_out = (real)data_value(S.spectra, S.media[m.medium_out].refractive_index, p.wl);
        slab_eta = (real)data_value(S.spectra, m.slab_eta, p.wl);
        slab_abs = (real)data_value(S.spectra, m.slab_absorption, p.wl);
      }
      real w = 0;
      int lobe = LOBE_NONE;
      const vec wi = -dir;
      if (p.fin == FIN_NONE && dot(wi, N) > 0) {
        vec wo, hm = N;
        w = bsdf_of(m, eta_out, eta_in, slab_eta, slab_abs, wi, N, rng, wo, lobe, &hm);
        const real c = dot(N, wo);
        if ((c > 0 && lobe == LOBE_TRANSMIT) || (c < 0 && lobe == LOBE_REFLECT)) w = 0;
        dir = wo;
        if constexpr (ADJ) if (!(flags0 & PF_STAGE_BOUNCE) && w > 0 && m.type == SSOLH_MTL_MIRROR &&
            m.roughness > 0 && m.distribution == 0) {
          // first reflection of a path that starts on a parameterised
          // heliostat: score of the Beckmann microfacet density
          // p(h) = exp(-tan^2/m^2) / (pi m^2 cos^3) under a rotation of the
          // macro normal N about axis a (dN = a x N) and under m:
          //   dlog p/d angle = (2 sec^2/m^2 - 3) sec (h . (a x N))
          //   dlog p/dm      = 2 tan^2/m^3 - 2/m,  m = sqrt(2) slope error
          const uint32_t pp = a.A.p[p.slot];
          if (pp != NONE) {
            const double ct = fmin(dot(hm, N), 1.0);
            const double sec = 1.0 / ct, t2 = sec * sec - 1.0;
            const double mr = m.roughness;
            const double k = (2.0 * sec * sec / (mr * mr) - 3.0) * sec;
            const d3 a1 = ld3(a.A.axes + 6 * pp), a2 = ld3(a.A.axes + 6 * pp + 3);
            double4 sc = a.A.s[p.slot];
            sc.x += k * dot(hm, cross(a1, N));
            sc.y += k * dot(hm, cross(a2, N));
            sc.z += 1.4142135623730951 * (2.0 * t2 / (mr * mr * mr) - 2.0 / mr);
            a.A.s[p.slot] = sc;
          }
        }
      }
      kabs = 1 - w;
      out0 = in0 * w;
      out1 = in1 * w;
      out2 = receiver ? in2 * w : in2;
      if (lobe == LOBE_TRANSMIT && m.type == SSOLH_MTL_DIELECTRIC)
        next_med = (uint32_t)(m.medium_out == (int32_t)in_med ? m.medium_in : m.medium_out);
    }
    if (p.fin == FIN_NONE) {
      if (receiver) {
        p.pd[0] += in0 - out0;
        const uint32_t rkey = (uint32_t)is.receiver * 2u + (side == SSOL_FRONT_ ? 0u : 1u);
        const uint32_t pkey = is.prim_tally < 0 ? NONE
            : (uint32_t)(((uint64_t)is.prim_tally + prim) * 2u + (side == SSOL_FRONT_ ? 0u : 1u));
        // the path ends at this point (weight zero below): its weights join
        // the flush directly
        direct = out0 == 0;
        if (direct) {
          p.dkey = rkey;
          p.dpkey = pkey;
          din0 = in0; din1 = in1; din2 = in2; dabs = kabs;
        } else {
          real w10[10];
          receiver_weights(in0, in1, in2, kabs, w10);
          const size_t entry = (size_t)p.slot * a.W.npend;
          if (!pend_add(a.W.pkey + entry, (real*)a.W.pval + entry * 10, a.W.npend, p.npk, rkey,
                        w10)) {
            spill(T.sxr + (size_t)(blockIdx.x & T.mask_x) * T.nsamp * T.nrcv * 40u,
                  (uint64_t)p.samp * S.nrcv * 2u + rkey, w10, &a.C->spills);
          }
          if (pkey != NONE && !pend_add(a.W.qkey + entry, (real*)a.W.qval + entry * 10, a.W.npend,
                                        p.nqk, pkey, w10))
            spill_prim(T, pkey, w10, &a.C->spills);
        }
        if (ADJ && a.A.p[p.slot] != NONE) {
          if (pkey != NONE) a.A.s[p.slot].w += a.A.gmap[pkey] * (in0 * kabs);
          a.A.s[p.slot].w += a.A.d_total * (in0 - out0);
        }
      } else {
        p.pd[2] += in0 * kabs;
      }
      // extinction of the segment that reached this point, counted here at a
      // real point (past virtual points the segment runs from the last real
      // point); a virtual point counts it only if the path ends
      if (!virt || out0 == 0) {
        const real absorbed = p.pv[0] - in0;
        if (in_atm) p.pd[1] += absorbed; else p.pd[2] += absorbed;
      }
      if (out0 == 0) {
        p.fin = FIN_DONE;  // weight is zero: the segment ends here
      } else {
        if (virt) {
          // pass through: the same ray (the main direction where the path
          // starts on a virtual surface) beyond this hit
          p.r.dx = rdir.x; p.r.dy = rdir.y; p.r.dz = rdir.z;
          p.r.tmin = nextafterf((float)hit_t, FLT_MAX);
          p.pv[3] = in0;
        } else {
          p.r.ox = pos.x; p.r.oy = pos.y; p.r.oz = pos.z;
          p.r.dx = dir.x; p.r.dy = dir.y; p.r.dz = dir.z;
          p.r.tmin = 0;
          p.pv[0] = out0; p.pv[1] = out1; p.pv[2] = out2;
          set_base(p.r, base);
        }
        p.r.iss_from = iss;
        p.r.prim_from = prim;
        p.r.flags = side << RF_SIDE_SHIFT;
        p.flags = (p.flags & PF_HIT_RECEIVER) | PF_ACTIVE | PF_STAGE_BOUNCE |
                  (virt ? PF_HIT_VIRTUAL : 0u) | (in_atm ? PF_IN_ATM : 0u);
        p.media = in_med | (next_med << 16);
        p.block = rng.block;
        if constexpr (TRACK) a.K.pos[p.slot] = make_double4(pos.x, pos.y, pos.z, 0);
        return true;
      }
    }
  }
  if (TRACK) {
    // path type (src/ssol_solver.c:931, 1092-1094, 1111-1125)
    uint8_t ty;
    if (p.fin == FIN_KILLED) ty = SSOLH_PATH_DROPPED;
    else if (p.fin == FIN_FAILED) ty = SSOLH_PATH_ERROR;
    else if (!(flags0 & PF_STAGE_BOUNCE) && h.iss != NONE) ty = SSOLH_PATH_SHADOW;
    else ty = (p.flags & PF_HIT_RECEIVER) ? SSOLH_PATH_SUCCESS : SSOLH_PATH_MISSING;
    a.K.type[path] = ty;
  }
  p.pv[0] = direct ? din0 : missing;
  p.pv[1] = direct ? din1 : shadowed;
  p.pv[2] = din2;
  p.pv[3] = dabs;
  return false;
}

// Tallies of the wave's finished paths (p.fin != FIN_NONE); every lane of
// the wave calls it.
template <class F, bool ADJ>
__device__ __forceinline__ void flush_paths(const PathArgs& a, const Path<F>& p) {
  using real = typename F::real;
  const Tallies& T = a.T;
  const bool done = p.fin == FIN_DONE;
  const double factor = done ? (double)(1u << p.score) : 1.0;
  const bool last = done && p.dkey != NONE;
  {
    // global fields and the realisation count of the path's job (sun)
    const bool counted = done || p.fin == FIN_KILLED;
    const double g[6] = {p.cosf, p.pd[0], last ? real(0) : p.pv[1], last ? real(0) : p.pv[0],
                         p.pd[1], p.pd[2]};
    double g2[16];
    for (int i = 0; i < 6; ++i) {
      const double x = done ? g[i] * factor : 0.0;
      g2[2 * i] = x;
      g2[2 * i + 1] = x * x;
    }
    g2[12] = 1.0;
    g2[13] = g2[14] = g2[15] = 0.0;
    keyed_add<13, 16>(counted, counted ? p.job : 0, g2,
                      T.global + (size_t)(blockIdx.x & T.mask_g) * T.njobs * 16u);
    const double s4[4] = {g2[0], g2[1], g2[4], g2[5]};
    keyed_add<4>(done, done ? p.samp : 0, s4,
                 T.samp + (size_t)(blockIdx.x & T.mask_s) * T.nsamp * 4u);
    const unsigned long long nf = wave_count_add(p.fin == FIN_FAILED, &a.C->failed);
    if (p.fin == FIN_FAILED && nf + 1 >= a.prm.max_failed) atomicExch(&a.C->aborted, 1u);
  }
  // Receiver entries (sampled x receiver: the receiver tally is their sum,
  // k_fold_rcv), then per-primitive ones: the pending entries in turn,
  // then the last hit, which joins the pending entry of its key (before
  // squaring) if the path holds one
  real dw[10];
  receiver_weights(p.pv[0], p.pv[1], p.pv[2], p.pv[3], dw);
  double* sxr_base = T.sxr + (size_t)(blockIdx.x & T.mask_x) * T.nsamp * T.nrcv * 40u;
  for (int which = 0; which < 2; ++which) {
    const uint32_t n = !done ? 0u : which ? p.nqk : p.npk;
    const size_t entry = (size_t)p.slot * a.W.npend;
    const uint32_t* keys = (which ? a.W.qkey : a.W.pkey) + entry;
    const real* vals = (const real*)(which ? a.W.qval : a.W.pval) + entry * 10;
    const uint32_t lkey = !last ? NONE : which ? p.dpkey : p.dkey;
    bool lpend = lkey != NONE;
    for (uint32_t k = 0;; ++k) {
      uint32_t key = NONE;
      real v10[10];
      if (k < n) {
        key = keys[k];
        const bool merge = lpend && key == lkey;
        const auto* v = (const WeightPair<real>*)(vals + k * 10);
#pragma unroll
        for (int f = 0; f < 5; ++f) {
          const WeightPair<real> x = v[f];
          v10[2 * f] = x.a + (merge ? dw[2 * f] : real(0));
          v10[2 * f + 1] = x.b + (merge ? dw[2 * f + 1] : real(0));
        }
        if (merge) lpend = false;
      } else if (lpend) {
        key = lkey;
        for (int f = 0; f < 10; ++f) v10[f] = dw[f];
        lpend = false;
      }
      const bool has = key != NONE;
      if (!__ballot(has)) break;
      if (which) {
        prim_add(T, has, key, v10, factor);
        continue;
      }
      double v[20];
      for (int f = 0; f < 10; ++f) {
        const double x = has ? (double)v10[f] * factor : 0.0;
        v[2 * f] = x;
        v[2 * f + 1] = x * x;
      }
      keyed_add<20>(has, has ? (uint64_t)p.samp * (uint64_t)a.S.nrcv * 2u + key : 0, v, sxr_base);
    }
  }
  // adjoint: the path's weighted contribution times its scores, wave-reduced
  // (in start-instance order a wave's paths share a heliostat)
  if (ADJ) {
    const uint32_t pp = done ? a.A.p[p.slot] : NONE;
    const bool has = pp != NONE;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    if (has) {
      const double4 sc = a.A.s[p.slot];
      const double q = sc.w * factor;
      v[0] = q * sc.x;
      v[1] = q * sc.y;
      v[2] = q * sc.z;
    }
    keyed_add<3>(has, has ? pp : 0u, v, a.A.grad);
  }
}

__device__ __forceinline__ uint2 bits2(double v) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  return make_uint2((uint32_t)b, (uint32_t)(b >> 32));
}
__device__ __forceinline__ uint4 pack2(double x, double y) {
  const uint2 a = bits2(x), b = bits2(y);
  return make_uint4(a.x, a.y, b.x, b.y);
}
__device__ __forceinline__ double unpack_lo(uint4 v) {
  return __longlong_as_double((long long)(((uint64_t)v.y << 32) | v.x));
}
__device__ __forceinline__ double unpack_hi(uint4 v) {
  return __longlong_as_double((long long)(((uint64_t)v.w << 32) | v.z));
}

// A path past its first shading, to and from a place of a queue: its ray
// (which carries its side only), then the rest. An ended path keeps its place
// until the wave flushes it: fin and the keys take the ray's words.
template <class F>
__device__ __forceinline__ uint32_t flag_word(const Path<F>& p) {
  return (p.r.flags & (3u << RF_SIDE_SHIFT)) | (uint32_t)p.fin << 18 | p.flags << 8 |
         p.npk << 24 | p.nqk << 28;
}
template <class F>
__device__ __forceinline__ void set_flag_word(Path<F>& p, uint32_t w) {
  p.flags = (w >> 8) & 0xFFu;
  p.npk = (w >> 24) & 0xFu;
  p.nqk = w >> 28;
}
static_assert(RF_SIDE_SHIFT == 16 && MAX_PEND < 16 && FIN_FAILED < 4, "flag_word's fields");

__device__ __forceinline__ uint4* plane_at(const PathQ& Q, uint32_t plane, uint32_t i) {
  return Q.p + (size_t)plane * Q.cap + i;
}

__device__ __forceinline__ void store_ray(const PathQ& Q, uint32_t i, const Path<F64>& p) {
  *plane_at(Q, 0, i) = pack2(p.r.ox, p.r.oy);
  *plane_at(Q, 1, i) = pack2(p.r.oz, p.r.dx);
  *plane_at(Q, 2, i) = pack2(p.r.dy, p.r.dz);
}
__device__ __forceinline__ void store_state(const PathQ& Q, uint32_t i, const Path<F64>& p) {
  const bool ended = p.fin != FIN_NONE;
  const uint4 v[STATE_PLANES64 + 1] = {
      make_uint4(__float_as_uint(p.r.tmin), ended ? p.dkey : p.r.iss_from,
                 ended ? p.dpkey : p.r.prim_from, flag_word(p)),
      pack2(p.pv[0], p.pv[1]), pack2(p.pv[2], p.pv[3]), pack2(p.pd[0], p.pd[1]),
      pack2(p.pd[2], p.wl), make_uint4(p.slot, p.pid, bits2(p.cosf).x, bits2(p.cosf).y),
      make_uint4(p.block, p.depth, p.media, p.samp),
      make_uint4(p.job, p.score, p.interval, 0)};
#pragma unroll
  for (uint32_t k = 0; k <= STATE_PLANES64; ++k) *plane_at(Q, RAY_PLANES64 - 1 + k, i) = v[k];
}
__device__ __forceinline__ void load_ray(const PathQ& Q, uint32_t i, Path<F64>& p) {
  const uint4 a = *plane_at(Q, 0, i), b = *plane_at(Q, 1, i), c = *plane_at(Q, 2, i),
              m = *plane_at(Q, 3, i);
  p.r.ox = unpack_lo(a); p.r.oy = unpack_hi(a); p.r.oz = unpack_lo(b);
  p.r.dx = unpack_hi(b); p.r.dy = unpack_lo(c); p.r.dz = unpack_hi(c);
  p.r.tmin = __uint_as_float(m.x);
  p.r.iss_from = m.y;
  p.r.prim_from = m.z;
  p.r.flags = m.w & (3u << RF_SIDE_SHIFT);
}
__device__ __forceinline__ void load_state(const PathQ& Q, uint32_t i, Path<F64>& p) {
  uint4 v[STATE_PLANES64];
#pragma unroll
  for (uint32_t k = 0; k < STATE_PLANES64; ++k) v[k] = *plane_at(Q, RAY_PLANES64 + k, i);
  set_flag_word(p, plane_at(Q, 3, i)->w);
  p.pv[0] = unpack_lo(v[0]); p.pv[1] = unpack_hi(v[0]);
  p.pv[2] = unpack_lo(v[1]); p.pv[3] = unpack_hi(v[1]);
  p.pd[0] = unpack_lo(v[2]); p.pd[1] = unpack_hi(v[2]); p.pd[2] = unpack_lo(v[3]);
  p.wl = unpack_hi(v[3]);
  p.slot = v[4].x;
  p.pid = v[4].y;
  p.cosf = __longlong_as_double((long long)(((uint64_t)v[4].w << 32) | v[4].z));
  p.block = v[5].x;
  p.depth = v[5].y;
  p.media = v[5].z;
  p.samp = v[5].w;
  p.job = v[6].x;
  p.score = v[6].y;
  p.interval = v[6].z;
  p.n0 = mk(0, 0, 0);
}

__device__ __forceinline__ void store_ray(const PathQ& Q, uint32_t i, const Path<F32>& p) {
  auto f = [](float x) { return __float_as_uint(x); };
  *plane_at(Q, 0, i) = make_uint4(f(p.r.ox), f(p.r.oy), f(p.r.oz), p.r.base);
  *plane_at(Q, 1, i) = make_uint4(f(p.r.dx), f(p.r.dy), f(p.r.dz), f(p.r.tmin));
}
__device__ __forceinline__ void store_state(const PathQ& Q, uint32_t i, const Path<F32>& p) {
  auto f = [](float x) { return __float_as_uint(x); };
  const bool ended = p.fin != FIN_NONE;
  const uint4 v[STATE_PLANES32 + 1] = {
      make_uint4(ended ? p.dkey : p.r.iss_from, ended ? p.dpkey : p.r.prim_from, flag_word(p),
                 f(p.wl)),
      make_uint4(f(p.pv[0]), f(p.pv[1]), f(p.pv[2]), f(p.pv[3])),
      make_uint4(f(p.pd[0]), f(p.pd[1]), f(p.pd[2]), f(p.cosf)),
      make_uint4(p.slot, p.pid, p.block, p.depth),
      make_uint4(p.media, p.samp, p.job, p.score | p.interval << 16)};
#pragma unroll
  for (uint32_t k = 0; k <= STATE_PLANES32; ++k) *plane_at(Q, RAY_PLANES32 - 1 + k, i) = v[k];
}
__device__ __forceinline__ void load_ray(const PathQ& Q, uint32_t i, Path<F32>& p) {
  auto f = [](uint32_t x) { return __uint_as_float(x); };
  const uint4 a = *plane_at(Q, 0, i), b = *plane_at(Q, 1, i), m = *plane_at(Q, 2, i);
  p.r.ox = f(a.x); p.r.oy = f(a.y); p.r.oz = f(a.z); p.r.base = a.w;
  p.r.dx = f(b.x); p.r.dy = f(b.y); p.r.dz = f(b.z); p.r.tmin = f(b.w);
  p.r.iss_from = m.x;
  p.r.prim_from = m.y;
  p.r.flags = m.z & (3u << RF_SIDE_SHIFT);
}
__device__ __forceinline__ void load_state(const PathQ& Q, uint32_t i, Path<F32>& p) {
  auto f = [](uint32_t x) { return __uint_as_float(x); };
  uint4 v[STATE_PLANES32];
#pragma unroll
  for (uint32_t k = 0; k < STATE_PLANES32; ++k) v[k] = *plane_at(Q, RAY_PLANES32 + k, i);
  const uint4 m = *plane_at(Q, 2, i);
  set_flag_word(p, m.z);
  p.wl = f(m.w);
  p.pv[0] = f(v[0].x); p.pv[1] = f(v[0].y); p.pv[2] = f(v[0].z); p.pv[3] = f(v[0].w);
  p.pd[0] = f(v[1].x); p.pd[1] = f(v[1].y); p.pd[2] = f(v[1].z); p.cosf = f(v[1].w);
  p.slot = v[2].x;
  p.pid = v[2].y;
  p.block = v[2].z;
  p.depth = v[2].w;
  p.media = v[3].x;
  p.samp = v[3].y;
  p.job = v[3].z;
  p.score = v[3].w & 0xFFFFu;
  p.interval = v[3].w >> 16;
  p.n0 = mkf(0, 0, 0);
}
// fin and the keys of an ended path
template <class F>
__device__ __forceinline__ void load_end(const PathQ& Q, uint32_t i, Path<F>& p) {
  constexpr bool wide = sizeof(typename F::real) == 8;
  const uint4 m = *plane_at(Q, wide ? RAY_PLANES64 - 1 : RAY_PLANES32 - 1, i);
  p.fin = (int)(((wide ? m.w : m.z) >> 18) & 3u);
  p.dkey = wide ? m.y : m.x;
  p.dpkey = wide ? m.z : m.y;
}

// The form's start
template <bool ADJ, bool TRACK>
__device__ __forceinline__ void start_of(const PathArgs& a, Path<F64>& p) {
  start_path<ADJ, TRACK>(a, p);
}
template <bool ADJ, bool TRACK>
__device__ __forceinline__ void start_of(const PathArgs& a, Path<F32>& p) {
  start_path32(a, p);
}
template <class F>
__device__ __forceinline__ void blank_path(Path<F>& p) {
  p.r = typename F::Ray{};
  p.fin = FIN_NONE;
  p.dkey = p.dpkey = NONE;
  for (int i = 0; i < 4; ++i) p.pv[i] = 0;
  for (int i = 0; i < 3; ++i) p.pd[i] = 0;
  p.wl = p.cosf = 0;
  p.slot = p.pid = p.block = p.flags = p.depth = p.media = p.samp = p.job = 0;
  p.score = p.interval = p.npk = p.nqk = 0;
}

// The wave's paths that go on, to the next launch's queue (w: the wave of the
// launch), in lane order: the queue keeps the start-instance order
template <class F>
__device__ __forceinline__ void leave_paths(const PathArgs& a, bool alive, const Path<F>& p,
                                            uint32_t w) {
  const uint64_t m = __ballot(alive);
  const uint32_t i = w * 64u + (uint32_t)__popcll(m & ((1ull << lane_id()) - 1ull));
  if (alive) {
    store_ray(a.out, i, p);
    store_state(a.out, i, p);
  }
  if (lane_id() == 0) a.wave_out[w] = (uint32_t)__popcll(m);
}

// Rays the wave traced, beside the global fields of the block's stripe (job
// 0), and the generations of rays it went through
__device__ __forceinline__ void count_rays(const PathArgs& a, uint32_t rays, uint32_t gens) {
  if (lane_id() != 0 || !rays) return;
  unsafeAtomicAdd(a.T.global + (size_t)(blockIdx.x & a.T.mask_g) * a.T.njobs * 16u + 13,
                  (double)rays);
  if (gens > __hip_atomic_load(&a.C->gens, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
    atomicMax(&a.C->gens, gens);
}

template <class F, bool ADJ, bool TRACK>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(F::WAVES)))
k_start(PathArgs a) {
  using real = typename F::real;
  __shared__ uint32_t lds_stack[START_STACK * BLOCK];
  __shared__ real lds_state[6 * BLOCK];  // what the shading needs of the start point
  __shared__ Node4 lds_top[TOP_NODES];
  const uint32_t q = blockIdx.x * BLOCK + threadIdx.x;
  if (a.C->stop) {
    if (lane_id() == 0) a.wave_out[q / 64u] = 0;
    return;
  }
  for (uint32_t i = threadIdx.x; i < a.S.ntop; i += BLOCK) lds_top[i] = a.S.top[i];
  __syncthreads();
  bool alive = q < a.count;
  Path<F> p;
  blank_path(p);
  real* st = lds_state + threadIdx.x;
  if (alive) {
    p.slot = q;
    p.pid = a.order ? a.order[q] : q;
    start_of<ADJ, TRACK>(a, p);
    st[0] = p.n0.x; st[BLOCK] = p.n0.y; st[2 * BLOCK] = p.n0.z;
    st[3 * BLOCK] = p.wl; st[4 * BLOCK] = p.cosf; st[5 * BLOCK] = p.pv[0];
  }
  flush_sampled_count(alive, (int)p.samp, a.T);
  const uint64_t m = __ballot(alive);
  if (alive) {
    asm volatile("" ::: "memory");  // the values stay in LDS, not in registers
    const typename F::Hit h = trace_lane<typename F::Tracer, START_STACK>(
        a.S, a.SQ, p.r, q, lds_stack, lds_top, a.ovf);
    asm volatile("" ::: "memory");
    p.n0 = vec_of(st[0], st[BLOCK], st[2 * BLOCK]);
    p.wl = st[3 * BLOCK];
    p.cosf = st[4 * BLOCK];
    p.pv[0] = p.pv[1] = p.pv[2] = p.pv[3] = st[5 * BLOCK];
    alive = shade_path<F, ADJ, TRACK>(a, p, h);
  }
  leave_paths(a, alive, p, q / 64u);
  flush_paths<F, ADJ>(a, p);
  count_rays(a, (uint32_t)__popcll(m), 1);
}

// The queued paths, one ray further each; THROUGH: to their ends, each in
// its place of the queue (for launches of few paths)
template <class F, bool ADJ, bool TRACK, bool THROUGH>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(F::WAVES)))
k_resume(PathArgs a) {
  __shared__ uint32_t lds_stack[RESUME_STACK * BLOCK];
  __shared__ Node4 lds_top[TOP_NODES];
  const uint32_t count = a.list ? *a.in_n : a.count;
  if (blockIdx.x * BLOCK >= count) return;  // whole blocks only: the staging syncs
  for (uint32_t i = threadIdx.x; i < a.S.ntop; i += BLOCK) lds_top[i] = a.S.top[i];
  __syncthreads();
  const uint32_t q = blockIdx.x * BLOCK + threadIdx.x;
  const bool mine = a.list ? q < count : lane_id() < a.wave_in[q / 64u];
  const uint32_t at = a.list && mine ? a.list[q] : q;
  auto next_ray = [&](Path<F>& p) {
    load_ray(a.in, at, p);
    const typename F::Hit h = trace_lane<typename F::Tracer, RESUME_STACK>(
        a.S, a.SQ, p.r, q, lds_stack, lds_top, a.ovf);
    load_state(a.in, at, p);
    return shade_path<F, ADJ, TRACK>(a, p, h);
  };
  uint32_t rays = 0, gens = 0;
  Path<F> p;
  blank_path(p);
  if (THROUGH) {
    bool alive = mine;
    for (uint64_t m = __ballot(alive); m; m = __ballot(alive)) {
      rays += (uint32_t)__popcll(m);
      ++gens;
      if (alive) {
        Path<F> t;
        blank_path(t);
        alive = next_ray(t);
        store_ray(a.in, at, t);
        store_state(a.in, at, t);
      }
    }
    if (mine) {
      load_state(a.in, at, p);
      load_end(a.in, at, p);
    }
  } else {
    rays = (uint32_t)__popcll(__ballot(mine));
    gens = 1;
    bool alive = mine;
    if (mine) alive = next_ray(p);
    leave_paths(a, alive, p, q / 64u);
  }
  flush_paths<F, ADJ>(a, p);
  count_rays(a, rays, gens + (a.list ? 0u : 1u));  // right after k_start: with its generation
}

// The list of a queue's places from the waves' counts: exclusive scan of the
// counts in two levels (k_scan_chunks within chunks of SCAN_CHUNK counts,
// recording each chunk's total; k_scan_top over the totals, which gives the
// list's length), then k_queue_list writes wave w's places from offsets[w] +
// chunk[w / SCAN_CHUNK] on.
constexpr int SCAN_THREADS = 1024;
constexpr int SCAN_PER = 4;
constexpr int SCAN_CHUNK = SCAN_THREADS * SCAN_PER;
static_assert((1u << 28) / 64 / SCAN_CHUNK <= SCAN_THREADS, "one k_scan_top block scans every chunk");

__device__ void block_inclusive_scan(uint32_t* part) {
  const uint32_t tid = threadIdx.x;
  for (uint32_t off = 1; off < SCAN_THREADS; off <<= 1) {
    const uint32_t v = tid >= off ? part[tid - off] : 0u;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
}

__global__ void __launch_bounds__(SCAN_THREADS)
k_scan_chunks(const uint32_t* __restrict__ counts, uint32_t n, uint32_t* __restrict__ offsets,
              uint32_t* __restrict__ chunk) {
  __shared__ uint32_t part[SCAN_THREADS];
  const uint32_t tid = threadIdx.x;
  const uint32_t b0 = blockIdx.x * SCAN_CHUNK + tid * SCAN_PER;
  uint32_t v[SCAN_PER];
  uint32_t sum = 0;
#pragma unroll
  for (int k = 0; k < SCAN_PER; ++k) {
    v[k] = b0 + k < n ? counts[b0 + k] : 0u;
    sum += v[k];
  }
  part[tid] = sum;
  __syncthreads();
  block_inclusive_scan(part);
  uint32_t run = tid ? part[tid - 1] : 0u;
#pragma unroll
  for (int k = 0; k < SCAN_PER; ++k) {
    if (b0 + k < n) offsets[b0 + k] = run;
    run += v[k];
  }
  if (tid == SCAN_THREADS - 1) chunk[blockIdx.x] = part[SCAN_THREADS - 1];
}

// Also, between two launches of the path kernels: the generations of the one
// that ended join the solve's.
__global__ void __launch_bounds__(SCAN_THREADS)
k_scan_top(uint32_t nchunks, uint32_t* __restrict__ chunk, unsigned* total, Counters* C) {
  __shared__ uint32_t part[SCAN_THREADS];
  const uint32_t tid = threadIdx.x;
  const uint32_t v = tid < nchunks ? chunk[tid] : 0u;
  part[tid] = v;
  __syncthreads();
  block_inclusive_scan(part);
  if (tid < nchunks) chunk[tid] = part[tid] - v;
  if (tid == SCAN_THREADS - 1) *total = part[SCAN_THREADS - 1];
  if (tid == 0) {
    C->iterations += C->gens;
    C->gens = 0;
  }
}

__global__ void __launch_bounds__(256)
k_queue_list(const uint32_t* __restrict__ counts, uint32_t n, const uint32_t* __restrict__ offsets,
             const uint32_t* __restrict__ chunk, uint32_t* __restrict__ list) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x, w = i / 64u;
  if (w < n && lane_id() < counts[w]) list[offsets[w] + chunk[w / SCAN_CHUNK] + lane_id()] = i;
}

// A wavefront begins (wave; else the next realisations of its slots), unless
// too many paths have failed: then none of its realisations starts.
__global__ void k_path_begin(Counters* C, int wave) {
  C->iterations += C->gens;
  C->gens = 0;
  C->stop = C->aborted;
  if (wave && !C->stop) ++C->wavefronts;
}
