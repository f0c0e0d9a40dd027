// Single-precision form of the wavefront (included by ssolh.hip inside its
// anonymous namespace, after the shared records and helpers).
//
// Positions are rebased per instance: a point is (instance b, float offset
// from b's translation), so a float carries it with the precision of the
// instance's own size however far the instance sits from the origin. Rays
// are traversed in FP32 (TLAS in world space around the float origin, BLAS
// and watertight triangle test in the instance's frame), BSDFs and weights
// are FP32; the quadric root refinement (src/ssol_shape.c:864-1135) and the
// instance-entry transform run in FP64, and tallies accumulate in FP64.

struct alignas(16) RayRec32 {
  float ox, oy, oz;     // origin, offset from the translation of instance `base`
  uint32_t base;
  float dx, dy, dz;
  float tmin;
  uint32_t iss_from, prim_from, flags;
  uint32_t pad;
};
static_assert(sizeof(RayRec32) == 48, "RayRec32 layout");

struct alignas(16) HitRec32 {
  float px, py, pz;     // hit point, offset from the translation of the hit instance
  float t;              // distance of the nearest accepted triangle
  float nx, ny, nz;     // unit world normal (triangle Ng or quadric gradient)
  uint32_t iss, prim;   // iss == NONE <=> miss
  uint32_t pad[3];
};
static_assert(sizeof(HitRec32) == 48, "HitRec32 layout");

// Object -> quadric frame of each punched shape: p_q = Rinv (p_obj - t)
struct ShapeQ {
  double Rinv[9];
  double t[3];
};

__device__ __forceinline__ d3 inst_T(const ssolh_instance& in) {
  return mk(in.transform[9], in.transform[10], in.transform[11]);
}

// Ray origin and direction in the frame of instance i, FP64 (the
// translation difference is exact before the rotation)
__device__ __forceinline__ void to_instance(const DScene& S, uint32_t base, f3 off, f3 dir,
                                            uint32_t i, d3& o, d3& d) {
  const ssolh_instance& in = S.insts[i];
  const d3 rel = (inst_T(S.insts[base]) - inst_T(in)) + tod(off);
  o = mul(in.inv_linear, rel);
  d = mul(in.inv_linear, tod(dir));
}

struct FShear {
  int kx, ky, kz;
  float Sx, Sy, Sz;
};

__device__ __forceinline__ FShear make_shear32(f3 d) {
  const float a[3] = {fabsf(d.x), fabsf(d.y), fabsf(d.z)};
  const float v[3] = {d.x, d.y, d.z};
  FShear s;
  s.kz = a[0] > a[1] ? (a[0] > a[2] ? 0 : 2) : (a[1] > a[2] ? 1 : 2);
  s.kx = (s.kz + 1) % 3;
  s.ky = (s.kx + 1) % 3;
  if (v[s.kz] < 0) { const int t = s.kx; s.kx = s.ky; s.ky = t; }
  s.Sx = v[s.kx] / v[s.kz];
  s.Sy = v[s.ky] / v[s.kz];
  s.Sz = 1.0f / v[s.kz];
  return s;
}

__device__ __forceinline__ float compf(f3 p, int k) { return k == 0 ? p.x : (k == 1 ? p.y : p.z); }

// Watertight ray/triangle in FP32 (Woop, Benthin, Wald, JCGT 2013): an edge
// function that comes out exactly zero is recomputed in FP64, as the paper
// prescribes, so shared edges stay closed. No FMA contraction (exact
// negation of shared edges). Returns the distance or -1.
__device__ __forceinline__ float ray_triangle32(f3 o, const FShear& s, f3 v0, f3 v1, f3 v2) {
#pragma clang fp contract(off)
  const f3 A = v0 - o, B = v1 - o, C = v2 - o;
  const float Az = compf(A, s.kz), Bz = compf(B, s.kz), Cz = compf(C, s.kz);
  const float Ax = compf(A, s.kx) - s.Sx * Az, Ay = compf(A, s.ky) - s.Sy * Az;
  const float Bx = compf(B, s.kx) - s.Sx * Bz, By = compf(B, s.ky) - s.Sy * Bz;
  const float Cx = compf(C, s.kx) - s.Sx * Cz, Cy = compf(C, s.ky) - s.Sy * Cz;
  float U = Cx * By - Cy * Bx;
  float V = Ax * Cy - Ay * Cx;
  float W = Bx * Ay - By * Ax;
  if (U == 0.0f || V == 0.0f || W == 0.0f) {
    U = (float)((double)Cx * (double)By - (double)Cy * (double)Bx);
    V = (float)((double)Ax * (double)Cy - (double)Ay * (double)Cx);
    W = (float)((double)Bx * (double)Ay - (double)By * (double)Ax);
  }
  if ((U < 0 || V < 0 || W < 0) && (U > 0 || V > 0 || W > 0)) return -1;
  const float det = U + V + W;
  if (det == 0) return -1;
  const float T = U * s.Sz * Az + V * s.Sz * Bz + W * s.Sz * Cz;
  return T / det;
}

struct TraceState32 {
  float tbest;
  uint32_t iss, prim;
  bool punched;       // the best triangle belongs to a punched surface
  f3 nobj;            // object-space normal of the best (mesh) triangle
  double qdst;        // nearest refined quadric distance
  uint32_t qiss;      // its (instance, shaded shape)
};

// Reference any-hit filter (src/ssol_scene.c:438-536) in the frame of the
// instance being traversed (d: its FP32 ray direction); the quadric
// refinement rebuilds that ray in FP64 from the rebased origin.
__device__ bool filter32(const DScene& S, const ShapeQ* SQ, const RayRec32& r, f3 o, f3 d,
                         uint32_t iss_id, const ssolh_triangle& tri, float t,
                         TraceState32& ts, f3& nobj, bool& punched) {
  const uint32_t side_from = (r.flags >> RF_SIDE_SHIFT) & 3u;
  const IssInfo is = S.iss[iss_id];
  uint32_t side;
  double dst = 0;
  if (t < r.tmin) return false;
  punched = is.shape_type != SSOLH_SHAPE_MESH;
  if (!punched) {
    if (t <= 1.e-6f || t <= r.tmin || (tri.prim == r.prim_from && iss_id == r.iss_from))
      return false;
    const f3 v0 = ldf(tri.v0), v1 = ldf(tri.v1), v2 = ldf(tri.v2);
    nobj = cross(v2 - v0, v1 - v0);
    side = dot(nobj, d) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
  } else {
    const ssolh_shape& sh = S.shapes[is.shape];
    const ShapeQ& q = SQ[is.shape];
    d3 od, dd;
    to_instance(S, r.base, mkf(r.ox, r.oy, r.oz), mkf(r.dx, r.dy, r.dz), is.inst, od, dd);
    const d3 lo = mul(q.Rinv, od - ld3(q.t));
    const d3 ld = mul(q.Rinv, dd);
    d3 grad;
    if (!quadric_hit(sh.quadric, sh.qparam, lo, ld, (double)t, dst, grad)) return false;
    if (!(dst < (double)FLT_MAX)) return false;
    if ((float)dst <= r.tmin) return false;
    side = dot(ld, grad) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
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

// punched_rehit_possible for the FP32 form, with the FP32 filter's own
// quadric frame and side test (ray rebased at base, candidates within
// distance t_hi)
__device__ bool punched_rehit_possible32(const DScene& S, const ShapeQ* __restrict__ SQ,
                                         const RayRec32& r, uint32_t iss_id, double t_hi) {
  const uint32_t side_from = (r.flags >> RF_SIDE_SHIFT) & 3u;
  const IssInfo is = S.iss[iss_id];
  const ssolh_shape& sh = S.shapes[is.shape];
  const ShapeQ& q = SQ[is.shape];
  d3 od, dd;
  to_instance(S, r.base, mkf(r.ox, r.oy, r.oz), mkf(r.dx, r.dy, r.dz), is.inst, od, dd);
  const d3 lo = mul(q.Rinv, od - ld3(q.t));
  const d3 ld = mul(q.Rinv, dd);
  double a, b, c, t[2];
  if (!quadric_coeffs(sh.quadric, sh.qparam, lo, ld, a, b, c)) return false;
  const int n = quadric_roots(a, b, c, t);
  for (int k = 0; k < n; ++k) {
    if (!(t[k] < (double)FLT_MAX)) continue;
    if ((float)t[k] <= r.tmin) continue;
    const d3 grad = quadric_grad(sh.quadric, sh.qparam, lo + ld * t[k]);
    const uint32_t side = dot(ld, grad) < 0 ? SSOL_FRONT_ : SSOL_BACK_;
    if (side != side_from) continue;
    if (root_choosable(t, n, k, t_hi)) return true;
  }
  return false;
}

// Tracer64 in the FP32 form
struct Tracer32 {
  using Ray = RayRec32;
  using Hit = HitRec32;
  const DScene& S;
  const ShapeQ* SQ;
  const RayRec32& r;
  TraceState32 ts;
  f3 o, d;
  FShear sh;

  __device__ __forceinline__ Tracer32(const DScene& S_, const ShapeQ* SQ_, const RayRec32& r_)
      : S(S_), SQ(SQ_), r(r_) {
    ts.tbest = INFINITY;
    ts.iss = NONE;
    ts.prim = 0;
    ts.punched = false;
    ts.nobj = mkf(0, 0, 0);
    ts.qdst = INFINITY;
    ts.qiss = NONE;
  }
  __device__ __forceinline__ f3 off() const { return mkf(r.ox, r.oy, r.oz); }
  __device__ __forceinline__ f3 dw() const { return mkf(r.dx, r.dy, r.dz); }
  __device__ __forceinline__ FRay world() const {
    const f3 ow = tof(inst_T(S.insts[r.base]) + tod(off()));  // world origin, float
    return make_fray32(ow.x, ow.y, ow.z, r.dx, r.dy, r.dz);
  }
  // a ray leaving a planar object does not enter that object again, nor a
  // one-shape object's punched shape that no candidate could hit again (as
  // Tracer64)
  __device__ __forceinline__ uint32_t skipped() const {
    if (r.tmin != 0.f) return NONE;
    const IssInfo e = S.iss[r.iss_from];
    bool skip = (e.obj_flags & SSOLH_OBJECT_PLANAR) != 0;
    if (!skip && (e.obj_flags & OBJ_ONE_SHAPE) && e.shape_type != SSOLH_SHAPE_MESH) {
      d3 od, dd;
      to_instance(S, r.base, off(), dw(), e.inst, od, dd);
      const double t_hi = box_exit(S.obj_box + 6 * (size_t)S.insts[e.inst].object, od, dd);
      skip = !punched_rehit_possible32(S, SQ, r, r.iss_from, t_hi);
    }
    return skip ? e.inst : NONE;
  }
  template <class InstPtr>
  __device__ __forceinline__ FRay enter(InstPtr inst, uint32_t) {
    const d3 T = mk(inst->transform[9], inst->transform[10], inst->transform[11]);
    double m[9];
    for (int k = 0; k < 9; ++k) m[k] = inst->inv_linear[k];
    const d3 od = mul(m, (inst_T(S.insts[r.base]) - T) + tod(off())), dd = mul(m, tod(dw()));
    o = tof(od);
    d = tof(dd);
    sh = make_shear32(d);
    return make_fray(od, dd);
  }
  __device__ __forceinline__ bool hit(const ssolh_triangle& tri, uint32_t, uint32_t iss_first,
                                      float& tmax) {
    const float t = ray_triangle32(o, sh, ldf(tri.v0), ldf(tri.v1), ldf(tri.v2));
    if (!(t >= r.tmin && t < ts.tbest)) return false;
    f3 nobj;
    bool punched;
    const uint32_t iss = iss_first + tri.sshape;
    if (!filter32(S, SQ, r, o, d, iss, tri, t, ts, nobj, punched)) return false;
    ts.tbest = t;
    tmax = t < FLT_MAX ? t * 1.0000002f + 1e-30f : FLT_MAX;
    ts.iss = iss;
    ts.prim = tri.prim;
    ts.nobj = nobj;
    ts.punched = punched;
    return true;
  }
  __device__ __forceinline__ HitRec32 result() const {
    HitRec32 h;
    h.t = ts.tbest;
    h.iss = ts.iss;
    h.prim = ts.prim;
    h.pad[0] = h.pad[1] = h.pad[2] = 0;
    if (ts.iss != NONE) {
      // hit point relative to the hit instance, and the world normal, in FP64
      const uint32_t hiss = ts.punched ? ts.qiss : ts.iss;
      const IssInfo is = S.iss[hiss];
      const ssolh_instance& in = S.insts[is.inst];
      d3 od, dd;
      to_instance(S, r.base, off(), dw(), is.inst, od, dd);
      d3 p_obj, n_w;
      if (ts.punched) {
        const ssolh_shape& shp = S.shapes[is.shape];
        const ShapeQ& qq = SQ[is.shape];
        p_obj = od + dd * ts.qdst;
        const d3 pq = mul(qq.Rinv, p_obj - ld3(qq.t));
        n_w = tmul(S.isshapes[hiss].R_inv, quadric_grad(shp.quadric, shp.qparam, pq));
      } else {
        p_obj = od + dd * (double)ts.tbest;
        n_w = tmul(in.inv_linear, tod(ts.nobj));
      }
      const d3 p = mul(in.transform, p_obj);
      n_w = normalize(n_w);
      h.px = (float)p.x; h.py = (float)p.y; h.pz = (float)p.z;
      h.nx = (float)n_w.x; h.ny = (float)n_w.y; h.nz = (float)n_w.z;
    } else {
      h.px = h.py = h.pz = 0;
      h.nx = h.ny = h.nz = 0;
    }
    return h;
  }
};
