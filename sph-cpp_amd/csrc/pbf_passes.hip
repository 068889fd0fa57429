// pbf_passes.hip -- per-particle and neighbour-walk passes of the PBF step.
//
// Reference: Simulation/Source/particles.h:263-487 (one for_each_index lambda
// per pass) and Simulation/Source/main.cpp:71-124 (their order).
//
// Semantics on the device (the oracle's ORC_JACOBI mode): a pass reads the
// state as it was when the pass began and writes separate buffers, so the
// result does not depend on thread scheduling.  Where the reference writes
// in place while other particles read (the density fix at particles.h:303-305,
// XSPH at :439-446), this is the one place the device differs from the
// reference's serial CPU backend.
//
// Neighbour walks keep the list order and skip neighbours with r > h: every
// kernel term is exactly zero there (kernels.h:66,168) and adding a zero to a
// sum that started at +0 leaves it unchanged, so skipping is bit-exact for
// finite states.  Entries come in batches of eight, the next entries of a list
// loading under the current batch's arithmetic, by one lane or a quad per
// particle; while no particle has moved far from where its list was built,
// the walks go over the skin lists (pbf_walk.h).  One entry at a time over the
// full lists each pass waits on a chain of dependent loads.  Measured so, and
// as they are now, us a launch at 1,048,576 particles at rest: density 174 ->
// 62, multipliers 182 -> 63, updates 230 -> 88, XSPH 344 -> 143, vorticity 278
// -> 99, confinement 283 -> 102 (a step of all passes 4.8 -> 2.6 ms).
#include "pbf_walk.h"

namespace pbf {

constexpr int kBlock = 256;
static inline uint32_t nblocks(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

__device__ __forceinline__ bool in_span(uint32_t o, uint32_t b, uint32_t e) { return o >= b && o < e; }

// The lists a pass may walk: the full lists, and with `skin` the skin lists
// while the device's flags say that no particle has moved too far.
struct PassLists {
  const int32_t *nbr, *nbr_count, *snb, *snb_count;
  const unsigned long long* counters;
  int skin;
};
static PassLists pass_lists(const pbf_context* c, bool skin) {
  return PassLists{c->nbr, c->nbr_count, c->snb, c->snb_count, c->counters, skin ? 1 : 0};
}
struct Walk {
  const int32_t* list;
  int cnt;
};
__device__ __forceinline__ Walk walk_of(const PassLists& L, uint32_t p) {
  const bool skin = L.skin && skin_usable(L.counters, C_DISP_ALL);
  return Walk{skin ? L.snb : L.nbr, skin ? L.snb_count[p] : L.nbr_count[p]};
}
template <int LANES>
__device__ __forceinline__ bool pass_writes() {
  return lane_in_group<LANES>() == 0u;
}

// Quads below this many particles, single lanes above, for the reason given at
// density_lanes() in pbf_fused.hip: at 131,072 particles the two are within
// 10% of each other on these walks, at 32,768 quads take 60-70% of the time.
constexpr uint64_t kPassQuads = 131072;
#define PBF_PASS(c, name, kern, ...)                                                                             \
  do {                                                                                                           \
    const uint32_t n_ = (uint32_t)(c)->n;                                                                        \
    if (!n_) return;                                                                                             \
    KernelTimer* t_ = timer_begin((c), name);                                                                    \
    if (n_ <= kPassQuads)                                                                                        \
      hipLaunchKernelGGL(kern<4>, dim3(nblocks(4ull * n_)), dim3(kBlock), 0, (c)->stream, n_, __VA_ARGS__);   \
    else                                                                                                         \
      hipLaunchKernelGGL(kern<1>, dim3(nblocks(n_)), dim3(kBlock), 0, (c)->stream, n_, __VA_ARGS__);         \
    timer_end((c), t_);                                                                                          \
  } while (0)

// apply_external_forces (particles.h:263-270) and predict_positions (:275-287)
__global__ void __launch_bounds__(kBlock) k_forces_predict(uint32_t n, uint32_t b, uint32_t e, int flags, KParams K,
                                                           const uint32_t* __restrict__ oid,
                                                           const float4* __restrict__ x, float4* __restrict__ v,
                                                           float4* __restrict__ xs) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !in_span(oid[p], b, e)) return;
  f3 vp = ld3(v, p);
  if (flags & F_FORCES) {
    vp.y += K.g * K.dt;
    st3(v, p, vp);
  }
  if (flags & F_PREDICT) {
    f3 ps = add3(ld3(x, p), mul3(vp, K.dt));
    boundary(ps, K, p);
    st3(xs, p, ps);
  }
}

void launch_forces_predict(pbf_context* c, int flags, uint64_t b, uint64_t e) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "forces_predict");
  hipLaunchKernelGGL(k_forces_predict, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (uint32_t)b, (uint32_t)e,
                     flags, c->K, (const uint32_t*)c->oid, (const float4*)c->x, c->v, c->xs);
  timer_end(c, t);
}

// compute_densities (particles.h:292-313).  Reads xs, writes xt (the position
// star with the near-coincidence fix applied, particles.h:303-305) and rho;
// the API swaps xs and xt afterwards.
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_density(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                    const uint32_t* __restrict__ oid, const float4* __restrict__ xs,
                                                    const float4* __restrict__ v, float4* __restrict__ xt,
                                                    float* __restrict__ rho, PassLists L,
                                                    const float4* __restrict__ xs0,
                                                    unsigned long long* __restrict__ counters) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n) return;
  f3 xp = ld3(xs, p);
  if (!in_span(oid[p], b, e)) {
    if (pass_writes<LANES>()) st3(xt, p, xp);
    return;
  }
  Terms<1> sum{{K.mass_W0}};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, xp, K, xs, sum, near, [](uint32_t) { return NoData{}; },
      [&](f3, float d2, NoData, Terms<1>& t) { t.a[0] = K.mass * poly6_in(sqrt_cr(d2), K); });
  if (!pass_writes<LANES>()) return;
  uint32_t hacks = 0;
  if (near) {
    // magnitude(x*_p - x*_q) < 1e-8 (particles.h:304): the particle again, entry by entry
    float density = K.mass_W0;
    const int cnt = L.nbr_count[p];
    for (int k = 0; k < cnt; ++k) {
      const uint32_t q = (uint32_t)L.nbr[list_at(k, p, K.stride)];
      const f3 xq = ld3(xs, q);
      f3 d = sub3(xp, xq);
      float d2 = magsq3(d);
      if (!within_h(d2, K)) continue;
      if (d2 < K.T_hack) {
        const f3 vp = ld3(v, p);
        dec3(xp, div3(mul3(vp, K.dt), 50.0f));
        ++hacks;
        d = sub3(xp, xq);
        d2 = magsq3(d);
        if (!within_h(d2, K)) continue;
      }
      density += K.mass * poly6_in(sqrtf(d2), K);
    }
    sum.a[0] = density;
  }
  rho[p] = sum.a[0];
  st3(xt, p, xp);
  if (hacks) {
    atomicAdd(&counters[C_HACKS], (unsigned long long)hacks);
    // the fix's move counts against the skin lists
    if (K.skin_mode && !(move2(xp, xs0[p]) < K.disp_lim2)) atomicExch(&counters[C_DISP_ALL], 1ull);
  }
}

void launch_density(pbf_context* c, uint64_t b, uint64_t e) {
  PBF_PASS(c, "density", k_density, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->xs,
           (const float4*)c->v, c->xt, c->rho, pass_lists(c, c->pass_skin), (const float4*)c->xs0, c->counters);
}

// compute_pressure_lambdas (particles.h:318-342) from positions `pos`
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_lambda(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                   const uint32_t* __restrict__ oid, const float4* __restrict__ pos,
                                                   const float* __restrict__ rho, float* __restrict__ lam,
                                                   PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  // minus the sum of the gradients, and the sum of their squares
  Terms<4> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(pos, p), K, pos, sum, near, [](uint32_t) { return NoData{}; },
      [&](f3 d, float d2, NoData, Terms<4>& t) {
        const f3 grad = smul3(K.neg_inv_rho0, spiky_in(d, sqrt_cr(d2), K));
        t = Terms<4>{{-grad.x, -grad.y, -grad.z, magsq3(grad)}};
      });
  if (!pass_writes<LANES>()) return;
  const float sum_C = sum.a[3] + magsq3(f3{sum.a[0], sum.a[1], sum.a[2]});
  const float constraint = rho[p] / K.rho0 - 1.0f;
  const float C_p = ((double)constraint < 0.0) ? 0.0f : constraint;
  lam[p] = -C_p / (sum_C + K.eps);
}

void launch_lambda(pbf_context* c, const float4* pos, uint64_t b, uint64_t e) {
  PBF_PASS(c, "lambda", k_lambda, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid, pos,
           (const float*)c->rho, c->lam, pass_lists(c, c->pass_skin));
}

// compute_pressure_dps (particles.h:348-358): dp sum in list order
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_dp(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                               const uint32_t* __restrict__ oid, const float4* __restrict__ pos,
                                               const float* __restrict__ lam, float4* __restrict__ scr, PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  const float lp = lam[p];
  Terms<3> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(pos, p), K, pos, sum, near, [&](uint32_t q) { return lam[q]; },
      [&](f3 d, float d2, float lq, Terms<3>& t) {
        const f3 s = smul3(lp + lq, spiky_in(d, sqrt_cr(d2), K));
        t = Terms<3>{{s.x, s.y, s.z}};
      });
  if (pass_writes<LANES>()) st3(scr, p, smul3(K.inv_rho0, f3{sum.a[0], sum.a[1], sum.a[2]}));
}

void launch_dp(pbf_context* c, uint64_t b, uint64_t e) {
  PBF_PASS(c, "dp", k_dp, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->xs,
           (const float*)c->lam, c->scr, pass_lists(c, c->pass_skin));
}

// update_position_stars (particles.h:363-370): x* += scratch, boundary
__global__ void __launch_bounds__(kBlock) k_update_position_stars(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                                  const uint32_t* __restrict__ oid,
                                                                  const float4* __restrict__ scr,
                                                                  float4* __restrict__ xs,
                                                                  const float4* __restrict__ xs0,
                                                                  unsigned long long* __restrict__ counters) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  float mv = 0.0f;
  if (p < n && in_span(oid[p], b, e)) {
    f3 nw = add3(ld3(xs, p), ld3(scr, p));
    boundary(nw, K, p);
    st3(xs, p, nw);
    if (K.skin_mode) mv = move2(nw, xs0[p]);
  }
  if (K.skin_mode) record_move(mv, counters, C_DISP_ALL, K);
}

void launch_update_position_stars(pbf_context* c, uint64_t b, uint64_t e) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "update_position_stars");
  hipLaunchKernelGGL(k_update_position_stars, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (uint32_t)b,
                     (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->scr, c->xs,
                     (const float4*)c->xs0, c->counters);
  timer_end(c, t);
}

// update_velocities (particles.h:375-385)
// (the density rides in v.w, where the fused step's XSPH passes gather it)
__global__ void __launch_bounds__(kBlock) k_update_velocities(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                              const uint32_t* __restrict__ oid,
                                                              const float4* __restrict__ x,
                                                              const float4* __restrict__ xs,
                                                              const float* __restrict__ rho, float4* __restrict__ v) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !in_span(oid[p], b, e)) return;
  f3 vel = div3(sub3(ld3(xs, p), ld3(x, p)), K.dt);
  if ((double)magsq3(vel) < K.vthr) vel = {0.f, 0.f, 0.f};
  v[p] = make_float4(vel.x, vel.y, vel.z, rho[p]);
}

void launch_update_velocities(pbf_context* c, uint64_t b, uint64_t e) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "update_velocities");
  hipLaunchKernelGGL(k_update_velocities, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (uint32_t)b,
                     (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->x, (const float4*)c->xs,
                     (const float*)c->rho, c->v);
  timer_end(c, t);
}

// update_positions (particles.h:390-394)
__global__ void __launch_bounds__(kBlock) k_update_positions(uint32_t n, uint32_t b, uint32_t e,
                                                             const uint32_t* __restrict__ oid,
                                                             const float4* __restrict__ xs, float4* __restrict__ x) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n || !in_span(oid[p], b, e)) return;
  x[p] = xs[p];
}

void launch_update_positions(pbf_context* c, uint64_t b, uint64_t e) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "update_positions");
  hipLaunchKernelGGL(k_update_positions, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (uint32_t)b, (uint32_t)e,
                     (const uint32_t*)c->oid, (const float4*)c->xs, c->x);
  timer_end(c, t);
}

// apply_viscosity (particles.h:436-447), XSPH from vin into vout
struct VelocityDensity {
  float4 v;
  float rho;
};
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_viscosity(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                      const uint32_t* __restrict__ oid,
                                                      const float4* __restrict__ xs, const float* __restrict__ rho,
                                                      const float4* __restrict__ vin, float4* __restrict__ vout,
                                                      PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n) return;
  const f3 vp = ld3(vin, p);
  if (!in_span(oid[p], b, e)) {
    if (pass_writes<LANES>()) st3(vout, p, vp);
    return;
  }
  Terms<3> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(xs, p), K, xs, sum, near,
      [&](uint32_t q) { return VelocityDensity{gather4(vin, q), rho[q]}; },
      [&](f3, float d2, const VelocityDensity& q, Terms<3>& t) {
        const f3 s = div3_shared(mul3(sub3(xyz(q.v), vp), poly6_in(sqrt_cr(d2), K)), q.rho);
        t = Terms<3>{{s.x, s.y, s.z}};
      });
  if (!pass_writes<LANES>()) return;
  f3 nv = vp;
  acc3(nv, smul3(K.visc, f3{sum.a[0], sum.a[1], sum.a[2]}));
  st3(vout, p, nv);
}

void launch_viscosity(pbf_context* c, const float4* vin, float4* vout, uint64_t b, uint64_t e) {
  PBF_PASS(c, "viscosity", k_viscosity, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid,
           (const float4*)c->xs, (const float*)c->rho, vin, vout, pass_lists(c, c->pass_skin));
}

// compute_vorticity (particles.h:452-466): omega -> scr
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_vorticity(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                      const uint32_t* __restrict__ oid,
                                                      const float4* __restrict__ xs,
                                                      const float4* __restrict__ vin, float4* __restrict__ scr,
                                                      PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  const f3 vp = ld3(vin, p);
  Terms<3> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(xs, p), K, xs, sum, near, [&](uint32_t q) { return gather4(vin, q); },
      [&](f3 d, float d2, float4 vq, Terms<3>& t) {
        const f3 s = cross3(sub3(xyz(vq), vp), spiky_in(d, sqrt_cr(d2), K));
        t = Terms<3>{{s.x, s.y, s.z}};
      });
  if (pass_writes<LANES>()) st3(scr, p, f3{sum.a[0], sum.a[1], sum.a[2]});
}

void launch_vorticity(pbf_context* c, const float4* vin, uint64_t b, uint64_t e) {
  PBF_PASS(c, "vorticity", k_vorticity, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid,
           (const float4*)c->xs, vin, c->scr, pass_lists(c, c->pass_skin));
}

// apply_vorticity (particles.h:471-487): reads |omega_q| of neighbours, own v
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_apply_vorticity(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                            const uint32_t* __restrict__ oid,
                                                            const float4* __restrict__ xs,
                                                            const float4* __restrict__ scr, float4* __restrict__ v,
                                                            PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  Terms<3> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(xs, p), K, xs, sum, near, [&](uint32_t q) { return gather4(scr, q); },
      [&](f3 d, float d2, float4 wq, Terms<3>& t) {
        const f3 s = smul3(sqrt_cr(magsq3(xyz(wq))), spiky_in(d, sqrt_cr(d2), K));
        t = Terms<3>{{s.x, s.y, s.z}};
      });
  if (!pass_writes<LANES>()) return;
  const f3 eta = {sum.a[0], sum.a[1], sum.a[2]};
  const f3 N = div3(eta, sqrtf(magsq3(eta)) + K.r_eps);
  f3 vp = ld3(v, p);
  acc3(vp, mul3(mul3(cross3(N, ld3(scr, p)), K.vort), K.dt));
  st3(v, p, vp);
}

void launch_apply_vorticity(pbf_context* c, float4* vio, uint64_t b, uint64_t e) {
  PBF_PASS(c, "apply_vorticity", k_apply_vorticity, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid,
           (const float4*)c->xs, (const float4*)c->scr, vio, pass_lists(c, c->pass_skin));
}

// apply_surface_tension (particles.h:400-431).  Pass 1: colour field -> scr,
// with the density in w for pass 2's gathers.
template <int LANES>
__global__ void __launch_bounds__(kBlock) k_color(uint32_t n, uint32_t b, uint32_t e, KParams K,
                                                  const uint32_t* __restrict__ oid, const float4* __restrict__ xs,
                                                  const float* __restrict__ rho, float4* __restrict__ scr,
                                                  PassLists L) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  Terms<3> sum{};
  bool near = false;
  const Walk w = walk_of(L, p);
  walk_within<LANES>(
      w.list, w.cnt, p, ld3(xs, p), K, xs, sum, near, [&](uint32_t q) { return rho[q]; },
      [&](f3 d, float d2, float rq, Terms<3>& t) {
        const f3 s = div3_shared(spiky_in(d, sqrt_cr(d2), K), rq);
        t = Terms<3>{{s.x, s.y, s.z}};
      });
  const f3 color = smul3(K.h, f3{sum.a[0], sum.a[1], sum.a[2]});
  if (pass_writes<LANES>()) scr[p] = make_float4(color.x, color.y, color.z, rho[p]);
}

// One pair's cohesion and curvature force (particles.h:415-426).  The
// reference takes 2 rho0 / (rho_p + rho_q) in double and rounds it to float;
// the quotient of two floats rounded to double and then to float is the
// correctly rounded float quotient (53 >= 2 * 24 + 2, no subnormal result), so
// one float divide gives the same bits.
__device__ __forceinline__ f3 tension_term(f3 r, f3 sp, float4 sq, float rp, float rq, const KParams& K) {
  float r_mag = sqrt_cr(magsq3(r));
  if (r_mag < K.st_rmin_float) r_mag = (float)K.st_rmin;
  const f3 cohesion = div3_shared(smul3(-K.gamma * cspline(r_mag, K), r), r_mag);
  const f3 curvature = smul3(-K.gamma, sub3(sp, xyz(sq)));
  const float sum = rp + rq;
  float Kq = (2.0f * K.rho0) / sum;
  if (!(fabsf(Kq) >= 0x1p-100f && fabsf(Kq) <= 0x1p100f)) Kq = (float)(2.0 * (double)K.rho0 / (double)sum);
  return smul3(Kq, add3(cohesion, curvature));
}

// Pass 2: cohesion + curvature force into own v.  The r > h shortcut does
// not apply here: curvature (scratch_p - scratch_q) has no kernel factor, so
// the walk takes every entry of the full list.
//
// Bound by its gathers, two for each entry of the full list.  A neighbour's
// density comes with its colour when pass 1 ran over all particles (ALL: scr.w
// of every neighbour is its density), and by a gather of its own otherwise;
// measured at 262,144 and 1,048,576 particles, us: 77 and 325 with the third
// gather, 54 and 247 without.
template <int LANES, bool ALL>
__device__ __forceinline__ void tension_pass(uint32_t n, uint32_t b, uint32_t e, const KParams& K,
                                             const uint32_t* __restrict__ oid, const float4* __restrict__ xs,
                                             const float* __restrict__ rho, const float4* __restrict__ scr,
                                             float4* __restrict__ v, const int32_t* __restrict__ nbr,
                                             const int32_t* __restrict__ nbr_count) {
  const uint32_t p = particle_of<LANES>();
  if (p >= n || !in_span(oid[p], b, e)) return;
  const f3 xp = ld3(xs, p);
  const f3 sp = ld3(scr, p);
  const float rp = rho[p];
  f3 f = {0.f, 0.f, 0.f};
  const int cnt = nbr_count[p];
  auto color = [&](uint32_t q) {
    float4 s = gather4(scr, q);
    if (!ALL) s.w = rho[q];
    return s;
  };
  if constexpr (LANES != 1) {
    const uint32_t* __restrict__ row = quad_row(nbr, p, K.stride);
    const int u = (int)(threadIdx.x & 3u);
    for (int k0 = 0; k0 < cnt; k0 += kBatch) {
      float4 t[2], s[2];
      bool on[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        on[j] = k0 + 4 * j + u < cnt;
        const uint32_t q = on[j] ? row[(k0 + 4 * j) * 64] : p;
        t[j] = gather4(xs, q), s[j] = color(q);
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        f3 term = {0.f, 0.f, 0.f};
        if (on[j]) term = tension_term(sub3(xp, xyz(t[j])), sp, s[j], rp, s[j].w, K);
        quad_add3(f, term);
      }
    }
    if (u != 0) return;
  } else {
    constexpr int kHalf = 4;  // (four entries' data are 32 registers)
    const int4* __restrict__ row = list_row(nbr, p, K.stride);
    for (int k0 = 0; k0 < cnt; k0 += kHalf) {
      const int4 a = row[(k0 / 4) * 64];
      const uint32_t q4[kHalf] = {(uint32_t)a.x, (uint32_t)a.y, (uint32_t)a.z, (uint32_t)a.w};
      float4 t[kHalf], s[kHalf];
#pragma unroll
      for (int u = 0; u < kHalf; ++u) {
        const uint32_t q = k0 + u < cnt ? q4[u] : p;
        t[u] = gather4(xs, q), s[u] = color(q);
      }
#pragma unroll
      for (int u = 0; u < kHalf; ++u)
        if (k0 + u < cnt) acc3(f, tension_term(sub3(xp, xyz(t[u])), sp, s[u], rp, s[u].w, K));
    }
  }
  f3 vp = ld3(v, p);
  acc3(vp, mul3(div3(f, rp), K.dt));
  v[p] = make_float4(vp.x, vp.y, vp.z, rp);  // the density stays in v.w for the XSPH passes
}
#define PBF_TENSION_KERNEL(name, ALL)                                                                            \
  template <int LANES>                                                                                           \
  __global__ void __launch_bounds__(kBlock) name(uint32_t n, uint32_t b, uint32_t e, KParams K,                  \
                                                 const uint32_t* __restrict__ oid, const float4* __restrict__ xs, \
                                                 const float* __restrict__ rho, const float4* __restrict__ scr,  \
                                                 float4* __restrict__ v, const int32_t* __restrict__ nbr,        \
                                                 const int32_t* __restrict__ nbr_count) {                        \
    tension_pass<LANES, ALL>(n, b, e, K, oid, xs, rho, scr, v, nbr, nbr_count);                                  \
  }
PBF_TENSION_KERNEL(k_tension, true)
PBF_TENSION_KERNEL(k_tension_span, false)

static void launch_color(pbf_context* c, uint64_t b, uint64_t e, bool skin) {
  PBF_PASS(c, "color", k_color, (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->xs,
           (const float*)c->rho, c->scr, pass_lists(c, skin));
}
#define PBF_TENSION_ARGS                                                                             \
  (uint32_t)b, (uint32_t)e, c->K, (const uint32_t*)c->oid, (const float4*)c->xs, (const float*)c->rho, \
      (const float4*)c->scr, c->v, (const int32_t*)c->nbr, (const int32_t*)c->nbr_count
static void launch_tension(pbf_context* c, uint64_t b, uint64_t e) { PBF_PASS(c, "tension", k_tension, PBF_TENSION_ARGS); }
static void launch_tension_span(pbf_context* c, uint64_t b, uint64_t e) {
  PBF_PASS(c, "tension", k_tension_span, PBF_TENSION_ARGS);
}

void launch_surface_tension(pbf_context* c, uint64_t cb, uint64_t ce, uint64_t b, uint64_t e, bool skin) {
  KernelTimer* t = timer_begin(c, "surface_tension");
  launch_color(c, cb, ce, skin);
  if (cb == 0 && ce >= c->n)
    launch_tension(c, b, e);
  else  // (a neighbour outside the first span keeps its scratch)
    launch_tension_span(c, b, e);
  timer_end(c, t);
}

// ---- original-order transfers through the staging buffer ----
__global__ void k_gather_out_f4(uint32_t n, const uint32_t* __restrict__ oid, const float4* __restrict__ src,
                                float* __restrict__ dst, int comps) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint32_t o = oid[s];
  const float4 t = src[s];
  dst[(uint64_t)o * comps + 0] = t.x;
  if (comps > 1) dst[(uint64_t)o * comps + 1] = t.y;
  if (comps > 2) dst[(uint64_t)o * comps + 2] = t.z;
}
__global__ void k_gather_out_f1(uint32_t n, const uint32_t* __restrict__ oid, const float* __restrict__ src,
                                float* __restrict__ dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  dst[oid[s]] = src[s];
}
__global__ void k_scatter_in_f4(uint32_t n, const uint32_t* __restrict__ oid, const float* __restrict__ src3,
                                float4* __restrict__ dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint64_t o = oid[s];
  dst[s] = make_float4(src3[o * 3], src3[o * 3 + 1], src3[o * 3 + 2], 0.f);
}
__global__ void k_scatter_in_f1(uint32_t n, const uint32_t* __restrict__ oid, const float* __restrict__ src,
                                float* __restrict__ dst) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  dst[s] = src[oid[s]];
}

void launch_gather_out_f4(pbf_context* c, const float4* src, float* dst3, int comps) {
  const uint32_t n = (uint32_t)c->n;
  if (n) hipLaunchKernelGGL(k_gather_out_f4, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (const uint32_t*)c->oid,
                            src, dst3, comps);
}
__global__ void k_gather_out_rows(uint32_t n, const uint32_t* __restrict__ oid, const float* __restrict__ src,
                                  float* __restrict__ dst, int width) {
  const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint64_t o = oid[s];
  for (int k = 0; k < width; ++k) dst[o * width + k] = src[(uint64_t)s * width + k];
}
void launch_gather_out_rows(pbf_context* c, const float* src, float* dst, int width) {
  const uint32_t n = (uint32_t)c->n;
  if (n) hipLaunchKernelGGL(k_gather_out_rows, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n,
                            (const uint32_t*)c->oid, src, dst, width);
}
void launch_gather_out_f1(pbf_context* c, const float* src, float* dst) {
  const uint32_t n = (uint32_t)c->n;
  if (n) hipLaunchKernelGGL(k_gather_out_f1, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (const uint32_t*)c->oid,
                            src, dst);
}
void launch_scatter_in_f4(pbf_context* c, const float* src3, float4* dst) {
  const uint32_t n = (uint32_t)c->n;
  if (n) hipLaunchKernelGGL(k_scatter_in_f4, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (const uint32_t*)c->oid,
                            src3, dst);
}
void launch_scatter_in_f1(pbf_context* c, const float* src, float* dst) {
  const uint32_t n = (uint32_t)c->n;
  if (n) hipLaunchKernelGGL(k_scatter_in_f1, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, n, (const uint32_t*)c->oid,
                            src, dst);
}

}  // namespace pbf
