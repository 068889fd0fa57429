// pbf_fused.hip -- neighbour passes of the fused step (pbf_step).
//
// Same arithmetic, order and results as the per-pass kernels in
// pbf_passes.hip (particles.h:292-487), organised for a 64-wide wavefront:
//
//  * Latency: a neighbour walk is a chain of dependent loads (list entry, then
//    the neighbour's data).  Neighbours are taken in batches of kBatch: the
//    batch's list entries load first (two 16-byte loads of a lane), then all
//    gathers are issued, then the arithmetic runs in list order.  The density
//    and pressure passes load the next batch's entries while they work on the
//    current one.
//  * Only about half of a particle's listed neighbours lie within h (the list
//    radius is the 1.2 h bin spacing, neighbors.h:198); the others contribute
//    exact zeros, and a test of their squared distance leaves them out (the
//    single lanes' pressure update takes the density pass's verdicts from a
//    bit mask instead, and does not gather the others).  The first XSPH pass
//    appends the entries within h of the final positions to a compact row
//    (cnb); vorticity, vorticity-apply and the second XSPH pass walk only that
//    row, in the same order.
//  * A particle is walked by one lane, or in small scenes by four or sixteen
//    (pbf_walk.h).
//  * The density pass writes lambda into the w word of its x* output, so the
//    dp pass gathers a neighbour's x* and lambda in one 16-byte load.
//  * The near-coincidence fix of compute_densities (particles.h:303-305) moves
//    x*_p in the middle of the walk; when it fires, the density pass redoes
//    that particle with a plain walk from its first entry and raises the
//    iteration's flag, and the lambda and dp passes of that iteration fall
//    back to plain walks for the particles next to a moved one.
#include <hip/hip_cooperative_groups.h>

#include <algorithm>

#include "pbf_mlp_device.h"
#include "pbf_walk.h"

namespace pbf {

constexpr int kBlock = 256;
static inline uint32_t nblocks(uint64_t n) { return (uint32_t)((n + kBlock - 1) / kBlock); }

// x limited to [lo, hi] (NaN gives lo)
__device__ __forceinline__ float clampf(float x, float lo, float hi) { return x > lo ? (x < hi ? x : hi) : lo; }

// ---------------------------------------------------------------------------
// compute_densities (particles.h:292-313) + compute_pressure_lambdas (:318-342)
// xs -> xt (x* with lambda in w), rho, lam.  With FEAT, also the learned warm
// start's features of the particle (FeatCtl).
struct DensitySums {
  float density, sum_C;
  f3 sg;
  float dy, div;  // FEAT
  int within;     // FEAT
};
__device__ __forceinline__ DensitySums density_start(const KParams& K) {
  return DensitySums{K.mass_W0, 0.0f, {0.f, 0.f, 0.f}, 0.0f, 0.0f, 0};
}

// particles.h:304-305: a plain walk over the full list from its first entry,
// in list order, moves x*_p at each near-coincident entry
template <bool FEAT, bool FAST>
__device__ __forceinline__ DensitySums density_plain(uint32_t p, f3& xp, f3 vp, const KParams& K,
                                                     const float4* __restrict__ xs, const float4* __restrict__ v,
                                                     const int32_t* __restrict__ nbr,
                                                     const int32_t* __restrict__ nbr_count, uint32_t& hacks) {
  DensitySums s = density_start(K);
  const int full = nbr_count[p];
  for (int k0 = 0; k0 < full; k0 += kBatch) {
    // a batch's positions load together; the entries are taken in order
    uint32_t q[kBatch];
    load_batch(nbr, K.stride, k0, full, p, q);
    f3 t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = ld3(xs, q[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      f3 d = sub3(xp, t[u]);
      float d2 = magsq3(d);
      if (k0 + u >= full || !within_h(d2, K)) continue;
      if (d2 < K.T_hack) {
        dec3(xp, div3(mul3(ld3(v, p), K.dt), 50.0f));
        ++hacks;
        d = sub3(xp, t[u]);
        d2 = magsq3(d);
        if (!within_h(d2, K)) continue;
      }
      const float r = nb_sqrt<FAST>(d2);
      s.density += K.mass * poly6_in(r, K);
      const f3 grad = smul3(K.neg_inv_rho0, nb_spiky<FAST>(d, r, K));
      dec3(s.sg, grad);
      s.sum_C += magsq3(grad);
      if (FEAT) {
        ++s.within;
        s.dy -= d.y;
        const f3 dv = sub3(vp, ld3(v, q[u]));
        s.div -= (dv.x * grad.x + dv.y * grad.y) + dv.z * grad.z;
      }
    }
  }
  return s;
}

// rho, lambda and x* of the particle from its sums; returns the density error
// max(rho/rho0 - 1, 0).
__device__ __forceinline__ float density_finish(uint32_t p, const DensitySums& s, f3 xp, const KParams& K,
                                                float4* __restrict__ xt, float* __restrict__ rho,
                                                float* __restrict__ lam, float& sum_C, float& lp) {
  rho[p] = s.density;
  sum_C = s.sum_C + magsq3(s.sg);
  const float constraint = s.density / K.rho0 - 1.0f;
  const float C_p = ((double)constraint < 0.0) ? 0.0f : constraint;
  lp = -C_p / (sum_C + K.eps);
  lam[p] = lp;
  xt[p] = make_float4(xp.x, xp.y, xp.z, lp);  // the dp pass gathers x* and lambda in one load
  return constraint;
}

// By one lane; also the particle's within-h mask (bit k of wmask[p], of
// wmask[n + p] for k >= 64: entry k of the walked list lies within h; not
// read for a particle the density fix moved).
template <bool FEAT, bool FAST, bool SR>
__device__ __forceinline__ float density_lambda_one(uint32_t p, uint32_t n, const KParams& K, const float4* __restrict__ xs,
                                                    const float4* __restrict__ v, float4* __restrict__ xt,
                                                    float* __restrict__ rho, float* __restrict__ lam,
                                                    const int32_t* __restrict__ nbr,
                                                    const int32_t* __restrict__ nbr_count,
                                                    uint64_t* __restrict__ wmask, const FeatCtl& F,
                                                    uint32_t& hacks, float (&fo)[8], const int32_t* __restrict__ snb,
                                                    const int32_t* __restrict__ snb_count, bool skin) {
  f3 xp = ld3(xs, p);
  // the walk goes over the skin list when it may (skin lists, above); the
  // plain walk after a density fix always takes the full list
  const int32_t* __restrict__ walk = skin ? snb : nbr;
  const int cnt = skin ? snb_count[p] : nbr_count[p];
  DensitySums s = density_start(K);
  const bool plain = lost(xp);
  const f3 vp = FEAT ? ld3(v, p) : f3{0.f, 0.f, 0.f};
  // one walk over the list: the entries within h go into the sums, in list
  // order (padding entries read the far row and are never within h).  A
  // near-coincident entry (particles.h:304) ends the walk after its batch, and
  // the plain walk below redoes the particle with fresh sums; so it does a lost
  // particle.
  bool hack = plain;
  uint64_t m0 = 0, m1 = 0;
  const int4* __restrict__ row = list_row(walk, p, K.stride);
  uint32_t q[kBatch];
  load_row(row, 0, q);
  for (int k0 = 0; k0 < cnt && !hack; k0 += kBatch) {
    uint32_t bits = 0;
    float4 t[kBatch];
    f3 vq[FEAT ? kBatch : 1];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = gather4(xs, q[u]);
    if (FEAT) {
#pragma unroll
      for (int u = 0; u < kBatch; ++u) vq[u] = xyz(gather4(v, q[u]));
    }
    load_row(row, k0 + kBatch, q);  // the next batch's entries load under this one's work
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const f3 d = sub3(xp, xyz(t[u]));
      const float d2 = magsq3(d);
      const bool in = within_h(d2, K);
      hack |= d2 < K.T_hack;
      bits |= (uint32_t)in << u;
      if (in) {
        const float r = nb_sqrt<FAST, SR>(d2);
        s.density += K.mass * poly6_in(r, K);
        const f3 grad = smul3(K.neg_inv_rho0, nb_spiky<FAST, SR>(d, r, K));
        dec3(s.sg, grad);
        s.sum_C += magsq3(grad);
        if (FEAT) {  // (feature passes walk the full lists)
          ++s.within;
          s.dy -= d.y;
          const f3 dv = sub3(vp, vq[u]);
          s.div -= (dv.x * grad.x + dv.y * grad.y) + dv.z * grad.z;
        }
      }
    }
    // k0 is a multiple of kBatch = 8: a batch never straddles the two words
    if (k0 < 64)
      m0 |= (uint64_t)bits << k0;
    else
      m1 |= (uint64_t)bits << (k0 - 64);
  }
  if (!FEAT) {
    wmask[p] = m0;
    if (K.cap > 64) wmask[n + p] = m1;
  }
  if (hack) s = density_plain<FEAT, FAST>(p, xp, vp, K, xs, v, nbr, nbr_count, hacks);
  float sum_C, lp;
  const float constraint = density_finish(p, s, xp, K, xt, rho, lam, sum_C, lp);
  if (FEAT) {
    const float inv_s = 1.0f / kWarmLambdaScale;
    const float dyn = s.dy / (float)(s.within > 0 ? s.within : 1);
    fo[0] = clampf(constraint, -1.0f, 4.0f);
    fo[1] = clampf(lp * inv_s, -64.0f, 0.0f);
    fo[2] = clampf(F.lprev[p] * inv_s, -64.0f, 0.0f);
    fo[3] = clampf(sum_C * 1e-5f, 0.0f, 8.0f);
    fo[4] = clampf((float)s.within / 32.0f, 0.0f, 4.0f);
    fo[5] = clampf(vp.y * K.dt / K.h, -4.0f, 4.0f);
    fo[6] = clampf(dyn / K.h, -2.0f, 2.0f);
    fo[7] = clampf(s.div * K.mass * K.dt, -4.0f, 4.0f);
  }
  return constraint > 0.0f ? constraint : 0.0f;
}

// The same by L lanes (no features); lane 0 writes, counts the fixes and
// returns the error, the other lanes return 0.
template <bool FAST, bool SR, int L>
__device__ __forceinline__ float density_lambda_group(uint32_t p, const KParams& K, const float4* __restrict__ xs,
                                                     const float4* __restrict__ v, float4* __restrict__ xt,
                                                     float* __restrict__ rho, float* __restrict__ lam,
                                                     const int32_t* __restrict__ nbr,
                                                     const int32_t* __restrict__ nbr_count, uint32_t& hacks,
                                                     const int32_t* __restrict__ snb,
                                                     const int32_t* __restrict__ snb_count, bool skin) {
  f3 xp = ld3(xs, p);
  const int cnt = skin ? snb_count[p] : nbr_count[p];
  DensitySums s = density_start(K);
  bool hack = lost(xp);
  GroupRow<L> row(skin ? snb : nbr, p, K.stride);
  constexpr int kMine = GroupRow<L>::kMine;
  for (int k0 = 0; k0 < cnt && !hack; k0 += GroupRow<L>::kEntries) {
    uint32_t q[kMine];
    float4 t[kMine];
    row.template entries<true>(cnt - k0, K.pad, q);
#pragma unroll
    for (int j = 0; j < kMine; ++j) t[j] = gather4(xs, q[j]);
    row.advance();
    bool near = false;
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const f3 d = sub3(xp, xyz(t[j]));
      const float d2 = magsq3(d);
      near |= d2 < K.T_hack;
      float dens = 0.0f, c2 = 0.0f;
      f3 grad = {0.f, 0.f, 0.f};
      if (within_h(d2, K)) {
        const float r = nb_sqrt<FAST, SR>(d2);
        dens = K.mass * poly6_in(r, K);
        grad = smul3(K.neg_inv_rho0, nb_spiky<FAST, SR>(d, r, K));
        c2 = magsq3(grad);
      }
      group_sum<L, false>(s.density, dens);
      group_sum<L, true>(s.sg.x, grad.x);
      group_sum<L, true>(s.sg.y, grad.y);
      group_sum<L, true>(s.sg.z, grad.z);
      group_sum<L, false>(s.sum_C, c2);
    }
    hack = group_bits<L>(near) != 0u;
  }
  if (lane_in_group<L>() != 0u) return 0.0f;
  if (hack) s = density_plain<false, FAST>(p, xp, f3{0.f, 0.f, 0.f}, K, xs, v, nbr, nbr_count, hacks);
  float sum_C, lp;
  const float constraint = density_finish(p, s, xp, K, xt, rho, lam, sum_C, lp);
  return constraint > 0.0f ? constraint : 0.0f;
}

// Max and sum over the wavefront; every lane of the wavefront must call them.
__device__ __forceinline__ float wave_max(float e) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) e = fmaxf(e, __shfl_xor(e, d, 64));
  return e;
}
__device__ __forceinline__ unsigned long long wave_sum(unsigned long long e) {
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) e += __shfl_xor(e, d, 64);
  return e;
}
// a particle's error in 2^-32 units (errors above 2^31 saturate)
__device__ __forceinline__ unsigned long long fixed_error(float e) {
  return (unsigned long long)(fminf(e, 2147483648.0f) * 4294967296.0f);
}

// The learned warm start for one wavefront's 64 particles (every lane of the
// wavefront calls it; fo holds the lane's features, zero past n): the
// features go through LDS into the B operands of the network, which runs on
// four tiles of 16 particles, and wlam[q] = lprev[q] + scale * net(q).  The
// same operands and MFMA sequence as k_mlp_forward, so the same results.
__device__ __forceinline__ void warm_network(const FeatCtl& F, uint32_t wave_first, uint32_t n, const float (&fo)[8],
                                             float* __restrict__ s_feat) {
  const int l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  float4* row = reinterpret_cast<float4*>(s_feat + l * 8);
  row[0] = make_float4(fo[0], fo[1], fo[2], fo[3]);
  row[1] = make_float4(fo[4], fo[5], fo[6], fo[7]);
  __syncthreads();
  const MlpW W{F.w1, F.w2, nullptr, F.mp};
  v4s a1[4], a2[4][4];
  load_forward_operands(W, c, g, a1, a2);
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    v4s xb = {0, 0, 0, 0};
    if (g < 2) {
      const float4 f4 = *reinterpret_cast<const float4*>(s_feat + (16 * t + c) * 8 + 4 * g);
      xb = v4s{f2bf(f4.x), f2bf(f4.y), f2bf(f4.z), f2bf(f4.w)};
    }
    v4f z1[4], h1[4], z2[4], h2[4];
    const float y = mlp_forward(W, a1, a2, xb, g, z1, h1, z2, h2);
    const uint32_t q = wave_first + 16u * (uint32_t)t + (uint32_t)c;
    if (g == 0 && q < n) F.wlam[q] = F.lprev[q] + F.scale * y;
  }
}

// A particle is dirty when it or a particle in its list was moved by the
// density fix: its fused lambda and its within-h mask may be stale.  A list
// walk visits cells computed from floating-point coordinates (x + i*s,
// neighbors.h:177-179), which lie within two cells of the particle's own cell
// on every axis, so every particle that can list q sits within two cells of
// q's cell: the wavefront that moved q stamps those 5x5x5 cells, and
// lambda_repair looks through the lists of the particles in stamped cells for
// moved ones.  Past kMaxMovedMarked moved particles it looks through all of
// them (there the stamped cells would hold nearly everything).  (Stamping cells, two stores a lane,
// needs no launch of its own; stamping their particles took one, 4.5 us an
// iteration also when nothing had moved.)
constexpr uint32_t kMaxMovedMarked = 4096;
__device__ __forceinline__ void stamp_cells(uint64_t movers, uint32_t p, uint32_t stamp, const KParams& K,
                                            const uint32_t* __restrict__ key, uint32_t* __restrict__ cstamp) {
  const uint32_t lane = threadIdx.x & 63;
  while (movers != 0ull) {
    const uint32_t i = (uint32_t)__builtin_ctzll(movers);
    movers &= movers - 1ull;
    const uint32_t q = (uint32_t)__builtin_amdgcn_readlane((int)p, (int)i);
    const uint32_t kq = key[q];
    if (kq >= K.ncells) {  // outside the grid: nobody lists it
      if (lane == 0) cstamp[K.ncells] = stamp;
      continue;
    }
    // cell coordinates in the moved particle's own grid (its scene's); a grid
    // has fewer than 2^32 cells, so its layers do too
    const GridView G = grid_of(K, q);
    const uint32_t dxy = (uint32_t)G.dxy, lq = kq - G.off;
    const int cz = (int)(lq / dxy), rest = (int)(lq % dxy);
    const int cy = rest / (int)G.dimx, cx = rest % (int)G.dimx;
    for (int j = (int)lane; j < 125; j += 64) {
      const int z = cz - 2 + j / 25, y = cy - 2 + j / 5 % 5, x = cx - 2 + j % 5;
      if (z >= 0 && z < (int)G.dimz && y >= 0 && y < (int)G.dimy && x >= 0 && x < (int)G.dimx)
        cstamp[G.off + (uint32_t)z * dxy + (uint32_t)y * G.dimx + (uint32_t)x] = stamp;
    }
  }
}

// FM = 0: density and lambda only; 1: also the warm start's features (stored
// when F.feat is set); 2: also the network on them (F.wlam).  FAST: the
// PBF_OPT_FAST_MATH arithmetic.
// The pass bodies below take their block of particles (vb) and whether the
// calling thread is the one that clears the pass's flags (first): the same
// bodies run as their own kernels (vb from xcd_block()) and inside the
// persistent Jacobi kernel (vb from the calling block's share).
// With S.ehist, a wavefront's largest density error goes into a shard of row
// eslot (atomicMax on the bits of a non-negative float orders like the float)
// and its fixed-point sum into the same shard of S.esum.  With S.tol >= 0
// nothing runs once the solve is done.
// L: lanes per particle; a block of vb holds blockDim.x / L particles.
template <int FM, bool FAST, bool SR, int L>
__device__ __forceinline__ void density_pass(uint32_t vb, bool first, uint32_t n, int it, int eslot,
                                             const SolveCtl& S, const FeatCtl& F,
                                             const KParams& K, const float4* __restrict__ xs,
                                             const float4* __restrict__ v, float4* __restrict__ xt,
                                             float* __restrict__ rho, float* __restrict__ lam,
                                             const int32_t* __restrict__ nbr,
                                             const int32_t* __restrict__ nbr_count,
                                             uint64_t* __restrict__ wmask,
                                             const uint32_t* __restrict__ key,
                                             uint32_t* __restrict__ cstamp, uint32_t stamp,
                                             uint32_t* __restrict__ mflag,
                                             unsigned long long* __restrict__ counters,
                                             const int32_t* __restrict__ snb,
                                             const int32_t* __restrict__ snb_count) {
  if (S.tol >= 0.0f && counters[C_DONE] != 0ull) return;
  const uint32_t p = (vb * blockDim.x + threadIdx.x) / (uint32_t)L;
  // this iteration's pressure update records its moves in the other slot
  const bool skin = FM == 0 && skin_usable(counters, C_DISP + (it & 1));
  if (first) counters[C_DISP + ((it + 1) & 1)] = 0ull;
  float e = 0.0f;
  uint32_t hacks = 0;
  float fo[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (p < n) {
    if constexpr (L != 1)
      e = density_lambda_group<FAST, SR, L>(p, K, xs, v, xt, rho, lam, nbr, nbr_count, hacks, snb, snb_count, skin);
    else
      e = density_lambda_one<FM != 0, FAST, SR>(p, n, K, xs, v, xt, rho, lam, nbr, nbr_count, wmask, F, hacks, fo,
                                                snb, snb_count, skin);
  }
  if (FM != 0 && F.feat && p < n) {
    float4* o = reinterpret_cast<float4*>(F.feat + (uint64_t)p * 8);
    o[0] = make_float4(fo[0], fo[1], fo[2], fo[3]);
    o[1] = make_float4(fo[4], fo[5], fo[6], fo[7]);
  }
  if constexpr (FM == 2) {
    __shared__ __attribute__((aligned(16))) float s_feat[kBlock * 8];
    warm_network(F, p - (threadIdx.x & 63u), n, fo, s_feat + (threadIdx.x & ~63u) * 8);
  }
  // particles moved by the density fix: one set of counter updates per
  // wavefront (every lane of the wavefront is here)
  const uint64_t hm = __ballot(hacks != 0);
  if (hm) {
    const uint32_t wl = threadIdx.x & 63;
    const unsigned long long hsum = wave_sum((unsigned long long)hacks);
    unsigned long long base = 0;
    if (wl == 0) {
      base = atomicAdd(&counters[C_MOVED_N + (it & 1)], (unsigned long long)__popcll(hm));
      atomicAdd(&counters[C_HACKS], hsum);
      atomicExch(&counters[C_HACK_FLAG + (it & 1)], 1ull);
    }
    base = __shfl(base, 0, 64);
    if (hacks) mflag[p] = stamp;
    if (base < kMaxMovedMarked) stamp_cells(hm, p, stamp, K, key, cstamp);
  }
  if (S.ehist) {
    const unsigned long long es = wave_sum(fixed_error(e));
    e = wave_max(e);
    const uint32_t row = (uint32_t)eslot * kErrShards + ((vb * blockDim.x + threadIdx.x) >> 6) % kErrShards;
    if ((threadIdx.x & 63) == 0) {
      if (e > 0.0f) atomicMax(&S.ehist[row], __float_as_uint(e));
      if (es) atomicAdd(&S.esum[row], es);
    }
  }
}

// (the exact and fast instances of the plain pass fit 64 registers: 8 wavefronts per SIMD)
template <int FM, bool FAST, bool SR, int L>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu((FM == 0 && (SR || FAST)) ? 8 : 1)))
k_density_lambda_c(uint32_t n, int it, int eslot, SolveCtl S, FeatCtl F,
                   KParams K, const float4* __restrict__ xs,
                   const float4* __restrict__ v, float4* __restrict__ xt,
                   float* __restrict__ rho, float* __restrict__ lam,
                   const int32_t* __restrict__ nbr,
                   const int32_t* __restrict__ nbr_count,
                   uint64_t* __restrict__ wmask,
                   const uint32_t* __restrict__ key,
                   uint32_t* __restrict__ cstamp, uint32_t stamp,
                   uint32_t* __restrict__ mflag,
                   unsigned long long* __restrict__ counters,
                   const int32_t* __restrict__ snb,
                   const int32_t* __restrict__ snb_count) {
  density_pass<FM, FAST, SR, L>(xcd_block(), blockIdx.x == 0 && threadIdx.x == 0, n, it, eslot, S, F, K, xs, v, xt, rho,
                         lam, nbr, nbr_count, wmask, key, cstamp, stamp, mflag, counters, snb, snb_count);
}

// compute_pressure_lambdas (particles.h:318-342) from xt for the dirty
// particles of this iteration (plain walks).  The new lambda goes to lam and
// to the particle's xt.w; positions are read as three words, so no lane reads
// the w word that another lane writes.  Dirty are the particles that carry this
// iteration's moved stamp or list one that does; they are stamped in dirty for
// the dp pass.
__device__ __forceinline__ f3 ld3_words(const float4* a, uint32_t i) {
  const float* f = reinterpret_cast<const float*>(a + i);
  return {f[0], f[1], f[2]};
}

// the sums of one particle, by one lane
template <bool FAST>
__device__ __forceinline__ void repair_walk(uint32_t p, f3 xp, const KParams& K, const float4* __restrict__ xt,
                                            const int32_t* __restrict__ nbr, int cnt, f3& sg, float& sum_C) {
  for (int k0 = 0; k0 < cnt; k0 += kBatch) {
    uint32_t q[kBatch];
    load_batch(nbr, K.stride, k0, cnt, p, q);
    f3 t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = ld3_words(xt, q[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const f3 d = sub3(xp, t[u]);
      const float d2 = magsq3(d);
      if (k0 + u >= cnt || !within_h(d2, K)) continue;
      const float r = nb_sqrt<FAST>(d2);
      const f3 grad = smul3(K.neg_inv_rho0, nb_spiky<FAST>(d, r, K));
      dec3(sg, grad);
      sum_C += magsq3(grad);
    }
  }
}

// the same by L
template <bool FAST, int L>
__device__ __forceinline__ void repair_walk_group(uint32_t p, f3 xp, const KParams& K, const float4* __restrict__ xt,
                                                  const int32_t* __restrict__ nbr, int cnt, f3& sg, float& sum_C) {
  GroupRow<L> row(nbr, p, K.stride);
  constexpr int kMine = GroupRow<L>::kMine;
  for (int k0 = 0; k0 < cnt; k0 += GroupRow<L>::kEntries) {
    uint32_t q[kMine];
    f3 t[kMine];
    row.template entries<false>(cnt - k0, p, q);
#pragma unroll
    for (int j = 0; j < kMine; ++j) t[j] = ld3_words(xt, q[j]);
    row.advance();
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const f3 d = sub3(xp, t[j]);
      const float d2 = magsq3(d);
      float c2 = 0.0f;
      f3 grad = {0.f, 0.f, 0.f};
      if (k0 + (int)lane_in_group<L>() + L * j < cnt && within_h(d2, K)) {
        const float r = nb_sqrt<FAST>(d2);
        grad = smul3(K.neg_inv_rho0, nb_spiky<FAST>(d, r, K));
        c2 = magsq3(grad);
      }
      group_sum<L, true>(sg.x, grad.x);
      group_sum<L, true>(sg.y, grad.y);
      group_sum<L, true>(sg.z, grad.z);
      group_sum<L, false>(sum_C, c2);
    }
  }
}

// Whether an entry of p's list was moved (its stamp in mflag), 16 entries a step.
__device__ __forceinline__ bool lists_moved(uint32_t p, uint32_t stamp, const KParams& K,
                                            const int32_t* __restrict__ nbr, int cnt,
                                            const uint32_t* __restrict__ mflag) {
  bool hit = mflag[p] == stamp;
  for (int k0 = 0; k0 < cnt && !hit; k0 += 2 * kBatch) {
    uint32_t q[2][kBatch];
    load_batch(nbr, K.stride, k0, cnt, p, q[0]);
    if (k0 + kBatch < cnt) load_batch(nbr, K.stride, k0 + kBatch, cnt, p, q[1]);
    else
#pragma unroll
      for (int u = 0; u < kBatch; ++u) q[1][u] = p;
    uint32_t f[2][kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) f[0][u] = mflag[q[0][u]], f[1][u] = mflag[q[1][u]];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) hit |= (f[0][u] == stamp) | (f[1][u] == stamp);
  }
  return hit;
}

// The particles p of the block's threads with `take`, gathered in LDS; their
// count.  Every thread of the block calls it.
__device__ __forceinline__ uint32_t block_gather(bool take, uint32_t p, uint32_t* s_p, uint32_t* s_count) {
  const uint32_t wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const uint64_t m = __ballot(take);
  if ((threadIdx.x & 63u) == 0u) s_count[wave] = (uint32_t)__popcll(m);
  __syncthreads();
  uint32_t before = 0, total = 0;
  for (uint32_t w = 0; w < waves; ++w) {
    const uint32_t k = s_count[w];
    before += w < wave ? k : 0u;
    total += k;
  }
  if (take)
    s_p[before + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u))] = p;
  __syncthreads();
  return total;
}

template <bool FAST, int L>
__device__ __forceinline__ void repair_gathered(const uint32_t* s_p, uint32_t total, uint32_t stamp,
                                                const KParams& K, float4* __restrict__ xt,
                                                const float* __restrict__ rho, float* __restrict__ lam,
                                                const int32_t* __restrict__ nbr,
                                                const int32_t* __restrict__ nbr_count,
                                                uint32_t* __restrict__ dirty) {
  for (uint32_t i = threadIdx.x / (uint32_t)L; i < total; i += blockDim.x / (uint32_t)L) {
    const uint32_t p = s_p[i];
    const f3 xp = ld3_words(xt, p);
    const int cnt = nbr_count[p];
    float sum_C = 0.0f;
    f3 sg = {0.f, 0.f, 0.f};
    if constexpr (L == 1)
      repair_walk<FAST>(p, xp, K, xt, nbr, cnt, sg, sum_C);
    else
      repair_walk_group<FAST, L>(p, xp, K, xt, nbr, cnt, sg, sum_C);
    if (L != 1 && lane_in_group<L>() != 0u) continue;
    sum_C += magsq3(sg);
    const float constraint = rho[p] / K.rho0 - 1.0f;
    const float C_p = ((double)constraint < 0.0) ? 0.0f : constraint;
    const float lp = -C_p / (sum_C + K.eps);
    dirty[p] = stamp;
    lam[p] = lp;
    reinterpret_cast<float*>(xt + p)[3] = lp;
  }
}

// Every thread of the block calls it.  A block gathers its candidates in LDS,
// tests their lists and gathers the dirty ones, so that the walks fill their
// wavefronts.  With few moved particles the launch takes as long as one walk,
// so up to kQuadRepairs dirty particles in a block go four lanes a particle
// (sixteen lanes for the fewest were no faster).  Measured on the million
// particles of a dam break, us a launch timed with events (some 7 above the
// kernel's own time): 26.5 with 16 moved particles, 76 with 1,000 and 110 with
// 130,000 when every particle of a stamped cell was redone where it stood by
// one lane; 20, 57 and 105 so.  (Limits of 64 and 256 instead of 128, before
// the candidates were tested: 26.4 and 21.4 with 16 moved particles, 21.2 with
// 128, and 77.7 and 115 with 1,000, 77.6 with 128.)
constexpr uint32_t kQuadRepairs = 128;
template <bool FAST>
__device__ __forceinline__ void repair_pass(uint32_t vb, uint32_t n, int it, uint32_t stamp, const SolveCtl& S,
                                            const KParams& K, float4* __restrict__ xt,
                                            const float* __restrict__ rho, float* __restrict__ lam,
                                            const int32_t* __restrict__ nbr,
                                            const int32_t* __restrict__ nbr_count,
                                            const uint32_t* __restrict__ mflag,
                                            uint32_t* __restrict__ dirty, const uint32_t* __restrict__ key,
                                            const uint32_t* __restrict__ cstamp,
                                            const unsigned long long* __restrict__ counters) {
  if (S.tol >= 0.0f && counters[C_DONE] != 0ull) return;
  if (counters[C_HACK_FLAG + (it & 1)] == 0ull) return;
  const bool scan = counters[C_MOVED_N + (it & 1)] > kMaxMovedMarked;
  const uint32_t p0 = vb * blockDim.x + threadIdx.x;
  __shared__ uint32_t s_dirty[kBlock], s_count[kBlock / 64];
  uint32_t p = p0;
  uint32_t total = block_gather(p0 < n && (scan || cstamp[key[p0]] == stamp), p0, s_dirty, s_count);
  bool hit = threadIdx.x < total;
  if (hit) {
    p = s_dirty[threadIdx.x];
    hit = lists_moved(p, stamp, K, nbr, nbr_count[p], mflag);
  }
  __syncthreads();
  total = block_gather(hit, p, s_dirty, s_count);
  if (total <= kQuadRepairs)
    repair_gathered<FAST, 4>(s_dirty, total, stamp, K, xt, rho, lam, nbr, nbr_count, dirty);
  else
    repair_gathered<FAST, 1>(s_dirty, total, stamp, K, xt, rho, lam, nbr, nbr_count, dirty);
  __syncthreads();  // a block of the persistent kernel uses the rows again
}

template <bool FAST>
__global__ void __launch_bounds__(kBlock) k_lambda_repair(uint32_t n, int it, uint32_t stamp, SolveCtl S,
                                                          KParams K, float4* __restrict__ xt,
                                                          const float* __restrict__ rho, float* __restrict__ lam,
                                                          const int32_t* __restrict__ nbr,
                                                          const int32_t* __restrict__ nbr_count,
                                                          const uint32_t* __restrict__ mflag,
                                                          uint32_t* __restrict__ dirty,
                                                          const uint32_t* __restrict__ key,
                                                          const uint32_t* __restrict__ cstamp,
                                                          const unsigned long long* __restrict__ counters) {
  repair_pass<FAST>(xcd_block(), n, it, stamp, S, K, xt, rho, lam, nbr, nbr_count, mflag, dirty, key, cstamp,
                    counters);
}

__device__ __forceinline__ float mean_error(unsigned long long sum, uint32_t n) {
  return (float)((double)sum / 4294967296.0 / (double)n);
}

// A row's error, its shards combined (every lane of the wavefront calls them)
__device__ __forceinline__ float max_error_of(const SolveCtl& S, int row) {
  static_assert(kErrShards == 64, "one shard per lane");
  return wave_max(__uint_as_float(S.ehist[(uint32_t)row * kErrShards + (threadIdx.x & 63u)]));
}
__device__ __forceinline__ float mean_error_of(const SolveCtl& S, int row, uint32_t n) {
  return mean_error(wave_sum(S.esum[(uint32_t)row * kErrShards + (threadIdx.x & 63u)]), n);
}

// The pressure update's sum over the entries of one particle's list within h
// (particles.h:355-366), by one lane: under the density pass's mask (entries
// outside h then gather the particle itself), or with plain every entry of
// the list tested.
template <bool FAST, bool SR>
__device__ __forceinline__ f3 dp_walk(const int32_t* __restrict__ walk, int cnt, bool plain, uint64_t m0, uint64_t m1,
                                      uint32_t p, f3 xp, float lp, const KParams& K,
                                      const float4* __restrict__ xt) {
  f3 dp = {0.f, 0.f, 0.f};
  const int4* __restrict__ row = list_row(walk, p, K.stride);
  uint32_t q[kBatch];
  for (int k0 = 0; k0 < cnt; k0 += kBatch) {
    load_row(row, k0, q);
    const uint32_t bits = (uint32_t)((k0 < 64 ? m0 >> k0 : m1 >> (k0 - 64)) & 0xFFu);
    float4 t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = gather4(xt, (bits >> u) & 1u ? q[u] : p);
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const f3 d = sub3(xp, xyz(t[u]));
      const float d2 = magsq3(d);
      if (!((bits >> u) & 1u) || (plain && !within_h(d2, K))) continue;
      const float r = nb_sqrt<FAST, SR>(d2);
      acc3(dp, smul3(lp + t[u].w, nb_spiky<FAST, SR>(d, r, K)));
    }
  }
  return dp;
}

// The same for a lost particle, entry by entry up to the full list's count
// (every lane of its group takes all of them).  A walk of its own because a
// test for the count in dp_walk costs every wavefront with a dirty lane: an
// update of the collapsed 1M dam break 98 us with it, 92 so.
template <bool FAST>
__device__ __forceinline__ f3 lost_update(const int32_t* __restrict__ list, int cnt, uint32_t p, f3 xp, float lp,
                                          const KParams& K, const float4* __restrict__ xt) {
  f3 dp = {0.f, 0.f, 0.f};
  for (int k = 0; k < cnt; ++k) {
    const float4 t = gather4(xt, (uint32_t)list[list_at((uint32_t)k, p, K.stride)]);
    const f3 d = sub3(xp, xyz(t));
    const float d2 = magsq3(d);
    if (!within_h(d2, K)) continue;
    acc3(dp, smul3(lp + t.w, nb_spiky<FAST, false>(d, nb_sqrt<FAST, false>(d2), K)));
  }
  return dp;
}

// The same by L lanes.
template <bool FAST, bool SR, int L>
__device__ __forceinline__ f3 dp_walk_group(const int32_t* __restrict__ walk, int cnt, uint32_t p, f3 xp, float lp,
                                           const KParams& K, const float4* __restrict__ xt) {
  f3 dp = {0.f, 0.f, 0.f};
  GroupRow<L> row(walk, p, K.stride);
  constexpr int kMine = GroupRow<L>::kMine;
  for (int k0 = 0; k0 < cnt; k0 += GroupRow<L>::kEntries) {
    uint32_t q[kMine];
    float4 t[kMine];
    row.template entries<true>(cnt - k0, K.pad, q);
#pragma unroll
    for (int j = 0; j < kMine; ++j) t[j] = gather4(xt, q[j]);
    row.advance();
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const f3 d = sub3(xp, xyz(t[j]));
      const float d2 = magsq3(d);
      f3 term = {0.f, 0.f, 0.f};
      if (within_h(d2, K)) {
        const float r = nb_sqrt<FAST, SR>(d2);
        term = smul3(lp + t[j].w, nb_spiky<FAST, SR>(d, r, K));
      }
      group_add3<L>(dp, term);
    }
  }
  return dp;
}

// compute_pressure_dps (particles.h:348-358) + update_position_stars
// (:363-370); on the last iteration also update_velocities (:375-385).
// In an iterate-to-tolerance solve, slot `it` first checks the error its
// density pass measured: a rejected warm start (slot 0 error above the error
// before the warm start; with the retry, also slot 1's after the damped
// start) restores xsave; an error <= tol ends the solve with x* = xt.
// Neither applies an update.
template <bool FAST, bool SR, int L>
__device__ __forceinline__ void dp_pass(uint32_t vb, bool first, uint32_t n, int it, int last, uint32_t stamp,
                                        const SolveCtl& S,
                                        const KParams& K, const float4* __restrict__ xt,
                                        const float4* __restrict__ x, float4* __restrict__ xs,
                                        float4* __restrict__ v, const int32_t* __restrict__ nbr,
                                        const int32_t* __restrict__ nbr_count,
                                        const uint64_t* __restrict__ wmask,
                                        const uint32_t* __restrict__ dirty,
                                        unsigned long long* __restrict__ counters,
                                        const int32_t* __restrict__ snb,
                                        const int32_t* __restrict__ snb_count,
                                        const float4* __restrict__ xs0,
                                        const float* __restrict__ rho) {
  // C_DONE holds the slot that ended the solve, plus one.  Only a solve that
  // ended at an earlier slot skips this launch: blocks of the ending slot that
  // start after block 0 has written the flag must still copy xt to x*.
  if (S.tol >= 0.0f) {
    const unsigned long long done = counters[C_DONE];
    if (done != 0ull && done <= (unsigned long long)it) return;
  }
  // clear the next iteration's flags (nobody reads them until the next density pass)
  if (first) {
    counters[C_HACK_FLAG + ((it + 1) & 1)] = 0ull;
    counters[C_MOVED_N + ((it + 1) & 1)] = 0ull;
  }
  const uint32_t p = (vb * blockDim.x + threadIdx.x) / (uint32_t)L;
  // (every lane of a group computes the particle's new state; lane 0 writes it)
  const bool writes = lane_in_group<L>() == 0u;
  // what this slot does, the same for every thread: 0 the update, 1 the
  // rejected warm start's restore, 2 the end of the solve (x* = xt)
  int mode = 0;
  if (S.ehist) {
    const float e = S.mean ? mean_error_of(S, it + 1, n) : max_error_of(S, it + 1);
    bool grew = false;
    // slot 0 checks the warm start; with the retry, slot 1 checks the damped one
    if (S.warm && (it == 0 || (it == 1 && S.retry && counters[C_RETRY] != 0ull))) {
      grew = e > (S.mean ? mean_error_of(S, 0, n) : max_error_of(S, 0));
      if (S.strict) {  // the other error measure must not grow either
        const float o = S.mean ? max_error_of(S, 1) : mean_error_of(S, 1, n);
        const float o_pre = S.mean ? max_error_of(S, 0) : mean_error_of(S, 0, n);
        grew = grew || o > o_pre;
      }
    }
    if (grew) {
      mode = 1;
      if (first) {
        if (S.retry && it == 0) {  // x* goes back, and k_warm_retry applies the damped start
          counters[C_RETRY] = 1ull;
          counters[C_WARM_KEPT] = 2ull;
        } else {
          counters[C_WARM_KEPT] = 0ull;
        }
      }
    } else if (S.tol >= 0.0f && e <= S.tol) {
      mode = 2;
      if (first) {
        counters[C_DONE] = (unsigned long long)(it + 1);
        counters[C_ITERS] = (unsigned long long)(it + 1);
      }
    }
  }
  const bool track = K.skin_mode;  // x*_0 is kept: check the moves
  float mv = 0.0f;
  if (p < n && mode == 1) {
    const float4 sv = S.xsave[p];
    if (writes) xs[p] = sv;
    if (S.lsum && it == 0 && writes) S.lsum[p] = 0.0f;
    if (track) mv = move2(xyz(sv), xs0[p]);
  } else if (p < n && mode == 2) {
    const float4 t = xt[p];
    if (writes) xs[p] = t;
    if (S.lsum && it == 0 && writes) S.lsum[p] = 0.0f;
    if (track) mv = move2(xyz(t), xs0[p]);
  } else if (p < n) {
    // x* and lambda of a particle come in one load (xt.w holds lambda)
    const float4 xp4 = xt[p];
    const f3 xp = xyz(xp4);
    // a dirty particle (moved by the density fix, or next to one) walks its
    // whole list; the others walk the list the density pass walked (the skin
    // list when it could)
    const bool plain = counters[C_HACK_FLAG + (it & 1)] != 0ull && dirty[p] == stamp;
    const bool skin = !plain && skin_usable(counters, C_DISP + (it & 1));
    const int32_t* __restrict__ walk = skin ? snb : nbr;
    const float lp = xp4.w;
    const int cnt = skin ? snb_count[p] : nbr_count[p];
    // with no dirty lane in the wavefront every pair within h is one the
    // density pass accepted at the same positions (static ranges); the lanes
    // of a group find them by the same test, single lanes by the mask it left
    f3 dp;
    if (__builtin_expect(lost(xp), 0))
      dp = lost_update<FAST>(nbr, nbr_count[p], p, xp, lp, K, xt);
    else if constexpr (L != 1)
      dp = (SR && __ballot(plain) == 0ull) ? dp_walk_group<FAST, SR, L>(walk, cnt, p, xp, lp, K, xt)
                                           : dp_walk_group<FAST, false, L>(walk, cnt, p, xp, lp, K, xt);
    else {
      const uint64_t m0 = plain ? ~0ull : wmask[p];
      const uint64_t m1 = (plain || K.cap <= 64) ? ~0ull : wmask[n + p];
      dp = (SR && __ballot(plain) == 0ull) ? dp_walk<FAST, SR>(walk, cnt, false, m0, m1, p, xp, lp, K, xt)
                                           : dp_walk<FAST, false>(walk, cnt, plain, m0, m1, p, xp, lp, K, xt);
    }
    f3 nw = add3(xp, smul3(K.inv_rho0, dp));
    boundary(nw, K, p);
    if (writes) st3(xs, p, nw);
    if (track) mv = move2(nw, xs0[p]);
    if (S.lsum && writes) S.lsum[p] = (it == 0 ? 0.0f : S.lsum[p]) + lp;  // (slot 0 starts the sum)
    if (last && writes) {  // the density rides in v.w for the XSPH passes' gathers
      f3 vel = div3(sub3(nw, ld3(x, p)), K.dt);
      if ((double)magsq3(vel) < K.vthr) vel = {0.f, 0.f, 0.f};
      v[p] = make_float4(vel.x, vel.y, vel.z, rho[p]);
    }
  }
  if (track) record_move(mv, counters, C_DISP + ((it + 1) & 1), K);
}

template <bool FAST, bool SR, int L>
__global__ void __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(8))) k_dp_update_c(uint32_t n, int it, int last, uint32_t stamp, SolveCtl S,
                                                        KParams K, const float4* __restrict__ xt,
                                                        const float4* __restrict__ x, float4* __restrict__ xs,
                                                        float4* __restrict__ v, const int32_t* __restrict__ nbr,
                                                        const int32_t* __restrict__ nbr_count,
                                                        const uint64_t* __restrict__ wmask,
                                                                        const uint32_t* __restrict__ dirty,
                                                        unsigned long long* __restrict__ counters,
                                                        const int32_t* __restrict__ snb,
                                                        const int32_t* __restrict__ snb_count,
                                                        const float4* __restrict__ xs0,
                                                        const float* __restrict__ rho) {
  dp_pass<FAST, SR, L>(xcd_block(), blockIdx.x == 0 && threadIdx.x == 0, n, it, last, stamp, S, K, xt, x, xs, v, nbr,
                nbr_count, wmask, dirty, counters, snb, snb_count, xs0, rho);
}

// Warm start of an iterate-to-tolerance solve: one compute_pressure_dps +
// update_position_stars pass (particles.h:348-370) with the given
// multipliers in place of lambda, over the full lists with the within-h test.
// xt holds the position stars after the first density pass; they are kept in
// xsave for the fallback.
template <bool FAST>
__global__ void __launch_bounds__(kBlock) k_warm_dp(uint32_t n, KParams K, const float4* __restrict__ xt,
                                                    const float* __restrict__ wlam,
                                                    const int32_t* __restrict__ nbr,
                                                    const int32_t* __restrict__ nbr_count, float4* __restrict__ xs,
                                                    float4* __restrict__ xsave,
                                                    unsigned long long* __restrict__ counters,
                                                    const float4* __restrict__ xs0) {
  const uint32_t p = xcd_block() * blockDim.x + threadIdx.x;
  const bool track = K.skin_mode;
  float mv = 0.0f;
  if (p < n) {
    const float4 xp4 = xt[p];
    const f3 xp = xyz(xp4);
    const float lp = wlam[p];
    f3 dp = {0.f, 0.f, 0.f};
    const int cnt = nbr_count[p];
    for (int k0 = 0; k0 < cnt; k0 += kBatch) {
      uint32_t q[kBatch];
      load_batch(nbr, K.stride, k0, cnt, p, q);
      float4 t[kBatch];
      float lq[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        t[u] = xt[q[u]];
        lq[u] = wlam[q[u]];
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const f3 d = sub3(xp, xyz(t[u]));
        const float d2 = magsq3(d);
        if (k0 + u >= cnt || !within_h(d2, K)) continue;
        const float r = nb_sqrt<FAST>(d2);
        acc3(dp, smul3(lp + lq[u], nb_spiky<FAST>(d, r, K)));
      }
    }
    f3 nw = add3(xp, smul3(K.inv_rho0, dp));
    boundary(nw, K, p);
    st3(xs, p, nw);
    xsave[p] = xp4;
    // both x* (kept) and xt (restored on a rejection) count as moves (a NaN
    // among them too, which a maximum would drop)
    if (track) {
      mv = move2(nw, xs0[p]);
      if (mv < K.disp_lim2) mv = move2(xp, xs0[p]);
    }
  }
  // slot 0 reads parity 0
  if (track) record_move(mv, counters, C_DISP + 0, K);
}

// PBF_OPT_WARM_RETRY, after slot 0's pressure update: when that update put x*
// back because the warm start grew the error (C_RETRY), x* becomes the
// position stars before the warm start plus the update with the warm
// multipliers times kWarmRetryScale (k_warm_dp with scaled multipliers, from
// the saved positions); slot 1 then checks it against the same error.
template <bool FAST>
__global__ void __launch_bounds__(kBlock) k_warm_retry(uint32_t n, KParams K, const float4* __restrict__ xsave,
                                                       const float* __restrict__ wlam,
                                                       const int32_t* __restrict__ nbr,
                                                       const int32_t* __restrict__ nbr_count,
                                                       float4* __restrict__ xs,
                                                       unsigned long long* __restrict__ counters,
                                                       const float4* __restrict__ xs0) {
  if (counters[C_RETRY] == 0ull) return;
  const uint32_t p = xcd_block() * blockDim.x + threadIdx.x;
  const bool track = K.skin_mode;
  float mv = 0.0f;
  if (p < n) {
    const f3 xp = ld3(xsave, p);
    const float lp = kWarmRetryScale * wlam[p];
    f3 dp = {0.f, 0.f, 0.f};
    const int cnt = nbr_count[p];
    for (int k0 = 0; k0 < cnt; k0 += kBatch) {
      uint32_t q[kBatch];
      load_batch(nbr, K.stride, k0, cnt, p, q);
      float4 t[kBatch];
      float lq[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        t[u] = gather4(xsave, q[u]);
        lq[u] = kWarmRetryScale * wlam[q[u]];
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const f3 d = sub3(xp, xyz(t[u]));
        const float d2 = magsq3(d);
        if (k0 + u >= cnt || !within_h(d2, K)) continue;
        const float r = nb_sqrt<FAST>(d2);
        acc3(dp, smul3(lp + lq[u], nb_spiky<FAST>(d, r, K)));
      }
    }
    f3 nw = add3(xp, smul3(K.inv_rho0, dp));
    boundary(nw, K, p);
    st3(xs, p, nw);
    if (track) mv = move2(nw, xs0[p]);
  }
  // slot 1 reads parity 1
  if (track) record_move(mv, counters, C_DISP + 1, K);
}

// ---------------------------------------------------------------------------
// The passes after the pressure solve, by groups of lanes.  A compact row (cnb) holds
// the entries within h of the final positions as byte offsets into the
// particle arrays.
__device__ __forceinline__ float4 gather_at(const float4* __restrict__ a, uint32_t offset) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(a) + offset);
}

// the XSPH term of one pair within h (particles.h:441-444); vq.w: the
// neighbour's density
__device__ __forceinline__ f3 xsph_term(f3 xp, f3 vp, float4 t, float4 vq, const KParams& K) {
  const float r = sqrt_cr(magsq3(sub3(xp, xyz(t))));
  return div3_shared(mul3(sub3(xyz(vq), vp), poly6_in(r, K)), vq.w);
}

// The first XSPH pass of a lost particle (every lane of its group calls it):
// its entries within h into the compact row, their number, and their terms.
__device__ __forceinline__ uint32_t lost_viscosity(const int32_t* __restrict__ list, int cnt, uint32_t p, f3 xp, f3 vp,
                                                   bool writes, const KParams& K, const float4* __restrict__ xs,
                                                   const float4* __restrict__ vin, int32_t* __restrict__ out, f3& dv) {
  uint32_t nc = 0;
  for (int k = 0; k < cnt; ++k) {
    const uint32_t at = (uint32_t)list[list_at((uint32_t)k, p, K.stride)] << 4;
    const float4 t = gather_at(xs, at);
    if (!within_h(magsq3(sub3(xp, xyz(t))), K)) continue;
    if (writes) out[(nc & ~3u) * 64u + (nc & 3u)] = (int32_t)at;
    ++nc;
    acc3(dv, xsph_term(xp, vp, t, gather_at(vin, at), K));
  }
  return nc;
}

// apply_viscosity (particles.h:436-447), first call: walks the skin or full
// list and leaves the compact rows of the final positions for the passes that
// follow.  An accepted entry's place in the row is the number accepted before
// it: the group's verdicts come from one ballot.
template <int L>
__global__ void __launch_bounds__(kBlock) k_viscosity_first(uint32_t n, KParams K, const float4* __restrict__ xs,
                                                            const float4* __restrict__ vin,
                                                            float4* __restrict__ vout,
                                                            const int32_t* __restrict__ nbr,
                                                            const int32_t* __restrict__ nbr_count,
                                                            int32_t* __restrict__ cnb,
                                                            int32_t* __restrict__ cnb_count,
                                                            const unsigned long long* __restrict__ counters,
                                                            const int32_t* __restrict__ snb,
                                                            const int32_t* __restrict__ snb_count,
                                                            unsigned long long* __restrict__ skin_hint) {
  const uint32_t p = particle_of<L>();
  const uint32_t u = lane_in_group<L>();
  // the next step builds skin lists only if this one's moves kept them usable to the end
  if (K.skin_mode && blockIdx.x == 0 && threadIdx.x == 0) *skin_hint = counters[C_DISP_ALL] == 0ull ? 1ull : 0ull;
  if (p >= n) return;
  const f3 xp = ld3(xs, p);
  const float4 v4 = vin[p];
  const f3 vp = xyz(v4);
  // the skin list holds every entry within h while no particle has moved
  // 0.045 h over the step (skin lists, above)
  const bool skin = skin_usable(counters, C_DISP_ALL), alone = lost(xp);
  const int all = skin ? snb_count[p] : nbr_count[p], cnt = alone ? 0 : all;
  GroupRow<L> row(skin ? snb : nbr, p, K.stride);
  constexpr int kMine = GroupRow<L>::kMine;
  int32_t* __restrict__ out = cnb + list_at(0, p, K.stride);
  const uint32_t before = (1u << u) - 1u;
  f3 dv = {0.f, 0.f, 0.f};
  uint32_t nc = 0;
  for (int k0 = 0; k0 < cnt; k0 += GroupRow<L>::kEntries) {
    uint32_t at[kMine];
    float4 t[kMine], vq[kMine];
    row.template entries<true>(cnt - k0, K.pad, at);
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      at[j] <<= 4;
      t[j] = gather_at(xs, at[j]), vq[j] = gather_at(vin, at[j]);
    }
    row.advance();
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      const bool in = within_h(magsq3(sub3(xp, xyz(t[j]))), K);
      const uint32_t bits = group_bits<L>(in);
      f3 term = {0.f, 0.f, 0.f};
      if (in) {
        const uint32_t k = nc + (uint32_t)__popc(bits & before);
        out[(k & ~3u) * 64u + (k & 3u)] = (int32_t)at[j];
        term = xsph_term(xp, vp, t[j], vq[j], K);
      }
      nc += (uint32_t)__popc(bits);
      group_add3<L>(dv, term);
    }
  }
  if (__builtin_expect(alone, 0)) nc = lost_viscosity(skin ? snb : nbr, all, p, xp, vp, u == 0u, K, xs, vin, out, dv);
  if (u != 0u) return;
  cnb_count[p] = (int32_t)nc;
  f3 nv = vp;
  acc3(nv, smul3(K.visc, dv));
  vout[p] = make_float4(nv.x, nv.y, nv.z, v4.w);  // the density stays in w
}

// A group's walk over a compact row: TERM(load(offset)) gives the three terms
// of an entry, which enter `sum` in list order.  Lanes past the row's end
// gather the particle itself and add +0.
template <int L, class Load, class Term>
__device__ __forceinline__ void group_walk_compact(const int32_t* __restrict__ cnb, int cnt, uint32_t p,
                                                   const KParams& K, f3& sum, Load load, Term term) {
  GroupRow<L> row(cnb, p, K.stride);
  constexpr int kMine = GroupRow<L>::kMine;
  const int u = (int)lane_in_group<L>();
  for (int k0 = 0; k0 < cnt; k0 += GroupRow<L>::kEntries) {
    uint32_t at[kMine];
    decltype(load(0u)) a[kMine];
    row.template entries<false>(cnt - k0, p << 4, at);
#pragma unroll
    for (int j = 0; j < kMine; ++j) a[j] = load(at[j]);
    row.advance();
#pragma unroll
    for (int j = 0; j < kMine; ++j) {
      f3 t = {0.f, 0.f, 0.f};
      if (u + j * L < cnt - k0) t = term(a[j]);
      group_add3<L>(sum, t);
    }
  }
}
struct Pair2 {  // a neighbour's position and its velocity or vorticity
  float4 t, w;
};

// The same by one lane: entries k0 .. k0+7 of a compact row; entries at or past cnt are the
// particle itself.
__device__ __forceinline__ void load_compact(const int4* __restrict__ row, int k0, int cnt, uint32_t p,
                                             uint32_t (&at)[kBatch]) {
  load_row(row, k0, at);
#pragma unroll
  for (int u = 0; u < kBatch; ++u) at[u] = k0 + u < cnt ? at[u] : p << 4;
}
template <class Load, class Term>
__device__ __forceinline__ void lane_walk_compact(const int32_t* __restrict__ cnb, int cnt, uint32_t p,
                                                  const KParams& K, f3& sum, Load load, Term term) {
  const int4* __restrict__ row = list_row(cnb, p, K.stride);
  for (int k0 = 0; k0 < cnt; k0 += kBatch) {
    uint32_t at[kBatch];
    load_compact(row, k0, cnt, p, at);
    Pair2 q[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) q[u] = load(at[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (k0 + u < cnt) acc3(sum, term(q[u]));
  }
}

template <int L, class Load, class Term>
__device__ __forceinline__ void walk_compact(const int32_t* __restrict__ cnb, int cnt, uint32_t p, const KParams& K,
                                             f3& sum, Load load, Term term) {
  if constexpr (L != 1)
    group_walk_compact<L>(cnb, cnt, p, K, sum, load, term);
  else
    lane_walk_compact(cnb, cnt, p, K, sum, load, term);
}
// apply_viscosity, second call, fused with update_positions (particles.h:390-394)
template <int L>
__global__ void __launch_bounds__(kBlock) k_viscosity_last(uint32_t n, KParams K, const float4* __restrict__ xs,
                                                           const float4* __restrict__ vin, float4* __restrict__ vout,
                                                           float4* __restrict__ x, const int32_t* __restrict__ cnb,
                                                           const int32_t* __restrict__ cnb_count) {
  const uint32_t p = particle_of<L>();
  if (p >= n) return;
  const f3 xp = ld3(xs, p);
  const f3 vp = ld3(vin, p);
  f3 dv = {0.f, 0.f, 0.f};
  walk_compact<L>(
      cnb, cnb_count[p], p, K, dv, [&](uint32_t at) { return Pair2{gather_at(xs, at), gather_at(vin, at)}; },
      [&](const Pair2& q) { return xsph_term(xp, vp, q.t, q.w, K); });
  if (lane_in_group<L>() != 0u) return;
  f3 nv = vp;
  acc3(nv, smul3(K.visc, dv));
  st3(vout, p, nv);
  x[p] = make_float4(xp.x, xp.y, xp.z, 0.f);
}

// compute_vorticity (particles.h:452-466) -> scr (omega, and |omega| in w)
template <bool SR, int L>
__global__ void __launch_bounds__(kBlock) k_vorticity_c(uint32_t n, KParams K, const float4* __restrict__ xs,
                                                        const float4* __restrict__ vin, float4* __restrict__ scr,
                                                        const int32_t* __restrict__ cnb,
                                                        const int32_t* __restrict__ cnb_count) {
  const uint32_t p = particle_of<L>();
  if (p >= n) return;
  const f3 xp = ld3(xs, p);
  const f3 vp = ld3(vin, p);
  f3 w = {0.f, 0.f, 0.f};
  walk_compact<L>(
      cnb, cnb_count[p], p, K, w, [&](uint32_t at) { return Pair2{gather_at(xs, at), gather_at(vin, at)}; },
      [&](const Pair2& q) {
        const f3 d = sub3(xp, xyz(q.t));
        const float r = sqrt_cr(magsq3(d));
        return cross3(sub3(xyz(q.w), vp), nb_spiky<false, SR>(d, r, K));
      });
  if (lane_in_group<L>() != 0u) return;
  scr[p] = make_float4(w.x, w.y, w.z, sqrtf(magsq3(w)));  // |omega| for apply_vorticity's gathers
}

// apply_vorticity (particles.h:471-487), v in place (own particle only)
template <bool SR, int L>
__global__ void __launch_bounds__(kBlock) k_apply_vorticity_c(uint32_t n, KParams K, const float4* __restrict__ xs,
                                                              const float4* __restrict__ scr,
                                                              float4* __restrict__ v,
                                                              const int32_t* __restrict__ cnb,
                                                              const int32_t* __restrict__ cnb_count) {
  const uint32_t p = particle_of<L>();
  if (p >= n) return;
  const f3 xp = ld3(xs, p);
  f3 eta = {0.f, 0.f, 0.f};
  walk_compact<L>(
      cnb, cnb_count[p], p, K, eta, [&](uint32_t at) { return Pair2{gather_at(xs, at), gather_at(scr, at)}; },
      [&](const Pair2& q) {
        const f3 d = sub3(xp, xyz(q.t));
        const float r = sqrt_cr(magsq3(d));
        return smul3(q.w.w, nb_spiky<false, SR>(d, r, K));  // |omega_q|, computed by the vorticity pass
      });
  if (lane_in_group<L>() != 0u) return;
  const f3 N = div3(eta, sqrtf(magsq3(eta)) + K.r_eps);
  const float4 v4 = v[p];
  f3 vp = xyz(v4);
  acc3(vp, mul3(mul3(cross3(N, ld3(scr, p)), K.vort), K.dt));
  v[p] = make_float4(vp.x, vp.y, vp.z, v4.w);  // the density stays in w for the second XSPH pass
}

// The first XSPH pass by single lanes.  It runs one wavefront per block and stages each lane's
// compact row in its own LDS column (entry k of the 64 lanes contiguous): its
// second loop reads it there, and it goes to memory four entries at a time.
constexpr int kStageBlock = 64;
__global__ void __launch_bounds__(kStageBlock) k_viscosity_first_lane(
    uint32_t n, KParams K, const float4* __restrict__ xs, const float4* __restrict__ vin, float4* __restrict__ vout,
    const int32_t* __restrict__ nbr, const int32_t* __restrict__ nbr_count, int32_t* __restrict__ cnb,
    int32_t* __restrict__ cnb_count, const unsigned long long* __restrict__ counters,
    const int32_t* __restrict__ snb, const int32_t* __restrict__ snb_count,
    unsigned long long* __restrict__ skin_hint) {
  extern __shared__ uint32_t s_list[];  // [max(cap + 1, stride)][kStageBlock]
  const uint32_t lane = threadIdx.x;
  const uint32_t p = xcd_block() * blockDim.x + threadIdx.x;
  // the next step builds skin lists only if this one's moves kept them usable to the end
  if (K.skin_mode && blockIdx.x == 0 && lane == 0) *skin_hint = counters[C_DISP_ALL] == 0ull ? 1ull : 0ull;
  if (p >= n) return;
  const f3 xp = ld3(xs, p);
  const float4 v4 = vin[p];
  const f3 vp = xyz(v4);
  const bool skin = skin_usable(counters, C_DISP_ALL);
  const int cnt = skin ? snb_count[p] : nbr_count[p];
  const int4* __restrict__ row = list_row(skin ? snb : nbr, p, K.stride);
  int nc = 0;
  for (int k0 = 0; k0 < cnt; k0 += kBatch) {
    uint32_t q[kBatch];
    load_row(row, k0, q);
    float4 t[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) t[u] = gather4(xs, q[u]);
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      s_list[nc * kStageBlock + lane] = q[u] << 4;  // a rejected entry is overwritten by the next accepted one
      nc += within_h(magsq3(sub3(xp, xyz(t[u]))), K) ? 1 : 0;
    }
  }
  if (__builtin_expect(lost(xp), 0)) {  // again, up to the count
    nc = 0;
    for (int k = 0; k < cnt; ++k) {
      const uint32_t at = (uint32_t)(skin ? snb : nbr)[list_at((uint32_t)k, p, K.stride)] << 4;
      s_list[nc * kStageBlock + lane] = at;
      nc += within_h(magsq3(sub3(xp, xyz(gather_at(xs, at)))), K) ? 1 : 0;
    }
  }
  cnb_count[p] = nc;
  int4* out = reinterpret_cast<int4*>(cnb + list_at(0, p, K.stride));
  f3 dv = {0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < nc; k0 += kBatch) {
    uint32_t at[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) at[u] = k0 + u < nc ? s_list[(k0 + u) * kStageBlock + lane] : p << 4;
    out[(k0 / 4) * 64] = make_int4((int)at[0], (int)at[1], (int)at[2], (int)at[3]);
    out[(k0 / 4 + 1) * 64] = make_int4((int)at[4], (int)at[5], (int)at[6], (int)at[7]);
    Pair2 q[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) q[u] = Pair2{gather_at(xs, at[u]), gather_at(vin, at[u])};
#pragma unroll
    for (int u = 0; u < kBatch; ++u)
      if (k0 + u < nc) acc3(dv, xsph_term(xp, vp, q[u].t, q[u].w, K));
  }
  f3 nv = vp;
  acc3(nv, smul3(K.visc, dv));
  vout[p] = make_float4(nv.x, nv.y, nv.z, v4.w);  // the density stays in w
}

// ---- launchers ----
#define PBF_LAUNCH(c, name, kern, ...)                                                                    \
  do {                                                                                                    \
    const uint32_t n_ = (uint32_t)(c)->n;                                                                 \
    if (!n_) return;                                                                                      \
    KernelTimer* t_ = timer_begin((c), name);                                                             \
    const uint32_t b_ = (c)->tune.block_size;                                                             \
    hipLaunchKernelGGL(kern, dim3((n_ + b_ - 1) / b_), dim3(b_), 0, (c)->stream, n_, __VA_ARGS__);         \
    timer_end((c), t_);                                                                                   \
  } while (0)

// How many lanes of a pass share a particle (same results): sixteen, four or
// one.  More lanes take fewer steps with more wavefronts and pay for their
// ordered sums, a DPP addition for every entry and term in all lanes, so they
// win while fewer leave the chip short of wavefronts (524,288 single lanes
// fill it).  Measured, us per launch on a dam break at rest, timed with events
// (some 3 us above the kernels' own time); 16 lanes against 4:
//   particles            960          8,192        16,384       32,768
//   density              10.3 / 11.6  11.1 / 12.2  12.3 / 12.3  16.6 / 13.7
//   pressure update       8.1 /  9.8   8.9 /  9.8  10.3 / 10.1  13.6 / 11.0
//   first XSPH            8.5 / 10.6   8.7 / 11.1  10.2 / 11.2  12.9 / 12.3
//   vorticity             6.4 /  8.6   6.8 /  8.8   8.1 /  8.8   9.6 /  9.4
//   confinement           6.4 /  8.5   6.7 /  8.5   7.6 /  8.5   9.9 /  9.1
//   second XSPH           7.1 /  9.1   7.3 /  9.2   7.7 /  9.1   9.3 /  9.7
// and 4 against 1:
//   particles            32,768       131,072      262,144      1,048,576
//   density              10.7 / 14.3  19.8 / 18.0  30.8 / 25.8  95 / 80
//   pressure update       9.6 / 15.0  17.1 / 18.1  27.7 / 24.6  92 / 72
//   first XSPH           11.5 / 18.0  22.5 / 26.8  36.6 / 44.5  188 / 164
//   vorticity             8.8 / 13.1  15.9 / 17.8  25.8 / 27.1  111 / 96
//   confinement           8.6 / 13.1  15.3 / 16.3  26.8 / 27.6  87 / 84
//   second XSPH           9.1 / 15.0  15.3 / 17.1  26.0 / 27.4  86 / 83
// (single lanes overtake between 65,536 and 131,072 particles in the density
// pass, between 131,072, where the update takes 17.3 us by quads and 18.8 by
// lanes, and 196,608, 23.2 and 22.4, in the pressure update, and near 524,288
// in the passes after it)
constexpr uint64_t kRowsPressure = 12288, kQuadsDensity = 98304, kQuadsUpdate = 147456;
constexpr uint64_t kRowsTail = 24576, kQuadsTail = 524288;
static int density_lanes(const pbf_context* c) { return c->n <= kRowsPressure ? 16 : (c->n <= kQuadsDensity ? 4 : 1); }
static int update_lanes(const pbf_context* c) { return c->n <= kRowsPressure ? 16 : (c->n <= kQuadsUpdate ? 4 : 1); }
static int tail_lanes(const pbf_context* c) { return c->n <= kRowsTail ? 16 : (c->n <= kQuadsTail ? 4 : 1); }

// `lanes` lanes per particle
#define PBF_LAUNCH_LANES(c, name, lanes, kern, ...)                                                       \
  do {                                                                                                    \
    const uint64_t n_ = (c)->n;                                                                           \
    if (!n_) return;                                                                                      \
    KernelTimer* t_ = timer_begin((c), name);                                                             \
    const uint32_t b_ = (c)->tune.block_size;                                                             \
    hipLaunchKernelGGL(kern, dim3((uint32_t)((n_ * (lanes) + b_ - 1) / b_)), dim3(b_), 0, (c)->stream,    \
                       (uint32_t)n_, __VA_ARGS__);                                                        \
    timer_end((c), t_);                                                                                   \
  } while (0)

#define PBF_LAUNCH_STAGED(c, name, kern, ...)                                                              \
  do {                                                                                                      \
    const uint32_t n_ = (uint32_t)(c)->n;                                                                   \
    if (!n_) return;                                                                                        \
    KernelTimer* t_ = timer_begin((c), name);                                                               \
    hipLaunchKernelGGL(kern, dim3((n_ + kStageBlock - 1) / kStageBlock), dim3(kStageBlock),                 \
                       (uint32_t)(kStageBlock * std::max((c)->K.cap + 1, (c)->K.stride) * sizeof(uint32_t)), \
                       (c)->stream, n_, __VA_ARGS__);                                                       \
    timer_end((c), t_);                                                                                     \
  } while (0)

// the kernel template KT instantiated for the context's arithmetic (PBF_OPT_FAST_MATH)
#define PBF_LAUNCH_ARITH(launch, c, name, KT, ...)        \
  do {                                                    \
    if ((c)->K.fast)                                      \
      launch(c, name, (KT<true>), __VA_ARGS__);           \
    else                                                  \
      launch(c, name, (KT<false>), __VA_ARGS__);          \
  } while (0)

template <int FM, bool FAST, bool SR, int L>
static void launch_density_as(pbf_context* c, const char* name, int it, int eslot, const SolveCtl& S,
                              const FeatCtl& F) {
  PBF_LAUNCH_LANES(c, name, L, (k_density_lambda_c<FM, FAST, SR, L>), it, eslot, S, F, c->K, (const float4*)c->xs,
                   (const float4*)c->v, c->xt, c->rho, c->lam, (const int32_t*)c->nbr, (const int32_t*)c->nbr_count,
                   c->wmask, (const uint32_t*)c->key, c->cstamp, c->dirty_stamp, c->mflag, c->counters,
                   (const int32_t*)c->snb, (const int32_t*)c->snb_count);
}

template <int FM, int L>
static void launch_density_fm(pbf_context* c, const char* name, int it, int eslot, const SolveCtl& S,
                              const FeatCtl& F) {
  if (c->K.fast)
    launch_density_as<FM, true, false, L>(c, name, it, eslot, S, F);
  else if (c->K.static_ranges)
    launch_density_as<FM, false, true, L>(c, name, it, eslot, S, F);
  else
    launch_density_as<FM, false, false, L>(c, name, it, eslot, S, F);
}

void launch_density_lambda_masked(pbf_context* c, int it, int eslot, const SolveCtl& S, const FeatCtl& F) {
  if (F.wlam)
    launch_density_fm<2, 1>(c, "density_warm_network", it, eslot, S, F);
  else if (F.feat)
    launch_density_fm<1, 1>(c, "density_features", it, eslot, S, F);
  else
    switch (density_lanes(c)) {
      case 16: return launch_density_fm<0, 16>(c, "density_lambda", it, eslot, S, F);
      case 4: return launch_density_fm<0, 4>(c, "density_lambda", it, eslot, S, F);
      default: return launch_density_fm<0, 1>(c, "density_lambda", it, eslot, S, F);
    }
}

void launch_lambda_repair(pbf_context* c, int it, const SolveCtl& S) {
  PBF_LAUNCH_ARITH(PBF_LAUNCH, c, "lambda_repair", k_lambda_repair, it, c->dirty_stamp, S, c->K, c->xt,
             (const float*)c->rho, c->lam, (const int32_t*)c->nbr, (const int32_t*)c->nbr_count,
             (const uint32_t*)c->mflag, c->dirty, (const uint32_t*)c->key, (const uint32_t*)c->cstamp,
             (const unsigned long long*)c->counters);
}

#define PBF_DP_ARGS                                                                                              \
  it, last, c->dirty_stamp, S, c->K, (const float4*)c->xt, (const float4*)c->x, c->xs, c->v, (const int32_t*)c->nbr, \
      (const int32_t*)c->nbr_count, (const uint64_t*)c->wmask, (const uint32_t*)c->dirty, c->counters,             \
      (const int32_t*)c->snb, (const int32_t*)c->snb_count, (const float4*)c->xs0, (const float*)c->rho
template <bool FAST, bool SR>
static void launch_dp_as(pbf_context* c, int it, int last, const SolveCtl& S) {
  switch (update_lanes(c)) {
    case 16: PBF_LAUNCH_LANES(c, "dp_update", 16, (k_dp_update_c<FAST, SR, 16>), PBF_DP_ARGS); break;
    case 4: PBF_LAUNCH_LANES(c, "dp_update", 4, (k_dp_update_c<FAST, SR, 4>), PBF_DP_ARGS); break;
    default: PBF_LAUNCH_LANES(c, "dp_update", 1, (k_dp_update_c<FAST, SR, 1>), PBF_DP_ARGS);
  }
}

void launch_dp_update_masked(pbf_context* c, int it, int last, const SolveCtl& S) {
  if (c->K.fast)
    launch_dp_as<true, false>(c, it, last, S);
  else if (c->K.static_ranges)
    launch_dp_as<false, true>(c, it, last, S);
  else
    launch_dp_as<false, false>(c, it, last, S);
}

void launch_warm_retry(pbf_context* c, const float* warm) {
  PBF_LAUNCH_ARITH(PBF_LAUNCH, c, "warm_retry", k_warm_retry, c->K, (const float4*)c->xsave,
                   warm, (const int32_t*)c->nbr, (const int32_t*)c->nbr_count, c->xs, c->counters,
                   (const float4*)c->xs0);
}

void launch_warm_dp(pbf_context* c, const float* warm) {
  PBF_LAUNCH_ARITH(PBF_LAUNCH, c, "warm_dp", k_warm_dp, c->K, (const float4*)c->xt, warm, (const int32_t*)c->nbr,
             (const int32_t*)c->nbr_count, c->xs, c->xsave, c->counters, (const float4*)c->xs0);
}

// ---------------------------------------------------------------------------
// The Jacobi iterations of a step or the slots of a solve in one cooperative
// launch (PBF_OPT_PERSISTENT): each iteration runs the density, lambda-repair
// and pressure-update bodies above over the whole particle
// range, separated by grid-wide barriers instead of kernel boundaries, and a
// solve leaves the loop on the device once its slot met the tolerance (every
// block reads the done flag after the same barrier).  Each block takes a
// contiguous share of the 256-particle blocks, its share placed on its XCD
// (xcd_block()).  The host launches it with one 256-particle block per block
// and at most one block per CU (persistent_fits), far inside what the chip
// holds at once, so every block is resident whatever else the device runs.
struct JacobiArgs {
  uint32_t n, iters;
  int solve, last_vel;  // solve: slot it's errors go to slot it + 1; last_vel: velocities in the last iteration
  uint32_t stamp0;      // stamp of the first iteration (then one more per iteration)
  SolveCtl S;
  KParams K;
  float4 *xs, *v, *xt;
  const float4 *x, *xs0;
  float *rho, *lam;
  const int32_t *nbr, *nbr_count, *snb, *snb_count;
  uint64_t* wmask;
  uint32_t *cstamp, *mflag, *dirty;
  const uint32_t* key;
  unsigned long long* counters;
};

template <bool FAST, bool SR>
__global__ void __launch_bounds__(kBlock) k_jacobi_persistent(JacobiArgs A) {
  cooperative_groups::grid_group grid = cooperative_groups::this_grid();
  const uint32_t nvb = (A.n + blockDim.x - 1) / blockDim.x;
  const uint32_t per = (nvb + gridDim.x - 1) / gridDim.x;
  const uint32_t vb0 = xcd_block() * per, vb1 = min(nvb, vb0 + per);
  const FeatCtl F0{nullptr, nullptr, nullptr, nullptr, nullptr, 0.0f, nullptr};
  for (uint32_t it = 0; it < A.iters; ++it) {
    if (A.S.tol >= 0.0f && __atomic_load_n(&A.counters[C_DONE], __ATOMIC_RELAXED) != 0ull) break;
    const uint32_t stamp = A.stamp0 + it;
    const int eslot = A.solve ? (int)it + 1 : 0;
    for (uint32_t vb = vb0; vb < vb1; ++vb)
      density_pass<0, FAST, SR, 1>(vb, vb == 0 && threadIdx.x == 0, A.n, (int)it, eslot, A.S, F0, A.K, A.xs, A.v, A.xt,
                            A.rho, A.lam, A.nbr, A.nbr_count, A.wmask, A.key, A.cstamp, stamp, A.mflag, A.counters, A.snb,
                            A.snb_count);
    grid.sync();
    for (uint32_t vb = vb0; vb < vb1; ++vb)
      repair_pass<FAST>(vb, A.n, (int)it, stamp, A.S, A.K, A.xt, A.rho, A.lam, A.nbr, A.nbr_count, A.mflag,
                        A.dirty, A.key, A.cstamp, A.counters);
    grid.sync();
    const int last = A.last_vel && it + 1 == A.iters;
    for (uint32_t vb = vb0; vb < vb1; ++vb)
      dp_pass<FAST, SR, 1>(vb, vb == 0 && threadIdx.x == 0, A.n, (int)it, last, stamp, A.S, A.K, A.xt, A.x, A.xs, A.v,
                    A.nbr, A.nbr_count, A.wmask, A.dirty, A.counters, A.snb, A.snb_count, A.xs0, A.rho);
    grid.sync();
  }
}

// Blocks of one cooperative launch of the persistent kernel on the context's
// device (0: cooperative launches unavailable), found once per context.
// the persistent kernel's instance for the context's arithmetic
static const void* persistent_kernel(const pbf_context* c) {
  if (c->K.fast) return (const void*)k_jacobi_persistent<true, false>;
  if (c->K.static_ranges) return (const void*)k_jacobi_persistent<false, true>;
  return (const void*)k_jacobi_persistent<false, false>;
}

static uint32_t persistent_blocks(pbf_context* c) {
  int& blocks = c->coop_blocks[c->K.fast ? 1 : (c->K.static_ranges ? 2 : 0)];
  if (blocks >= 0) return (uint32_t)blocks;
  blocks = 0;
  int coop = 0, cus = 0, per_cu = 0;
  if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, c->device) != hipSuccess || !coop)
    return 0;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess) return 0;
  c->coop_cus = cus;
  const void* kern = persistent_kernel(c);
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, kBlock, 0) != hipSuccess) return 0;
  blocks = std::max(0, per_cu * cus);
  return (uint32_t)blocks;
}

uint32_t persistent_capacity(pbf_context* c) { return persistent_blocks(c); }

// The cooperative launch is used for at most one block per CU (particles up
// to 256 x CUs): a launch of the full co-resident capacity (5 blocks per CU at
// this kernel's registers) did not finish on the 1M-particle dam break.
bool persistent_fits(pbf_context* c) {
  const uint32_t cap = persistent_blocks(c);
  const uint64_t nvb = (c->n + kBlock - 1) / kBlock;
  return cap > 0 && nvb <= (uint64_t)std::min<uint32_t>((uint32_t)c->coop_cus, cap);
}

bool persistent_available(pbf_context* c) { return persistent_blocks(c) > 0; }

int launch_jacobi_persistent(pbf_context* c, uint32_t iters, bool solve, bool last_vel, const SolveCtl& S) {
  const uint32_t n = (uint32_t)c->n;
  if (!n || !iters) return PBF_OK;
  const uint32_t nvb = (n + kBlock - 1) / kBlock;
  const uint32_t blocks = std::min<uint32_t>(persistent_blocks(c), nvb);
  if (!blocks) return set_error(PBF_ERR_UNSUPPORTED, "cooperative launches are not available on this device");
  JacobiArgs A{n, iters, solve ? 1 : 0, last_vel ? 1 : 0, c->dirty_stamp + 1, S, c->K, c->xs, c->v, c->xt,
               (const float4*)c->x, (const float4*)c->xs0, c->rho, c->lam, (const int32_t*)c->nbr,
               (const int32_t*)c->nbr_count, (const int32_t*)c->snb, (const int32_t*)c->snb_count, c->wmask,
               c->cstamp, c->mflag, c->dirty, (const uint32_t*)c->key, c->counters};
  void* args[] = {&A};
  KernelTimer* t = timer_begin(c, "jacobi_persistent");
  const void* kern = persistent_kernel(c);
  c->coop_grid = blocks;
  const hipError_t e = hipLaunchCooperativeKernel(kern, dim3(blocks), dim3(kBlock), args, 0, c->stream);
  timer_end(c, t);
  c->dirty_stamp += iters;
  return check_hip(e, "jacobi_persistent");
}

// The record of the solve that just ran (pbf_get_solve_log): slots used,
// whether the warm start was kept, the last used slot's errors and the errors
// before the warm start.  One wavefront: the ring index advances on the
// device, so graph replays record every solve.
__device__ __forceinline__ void log_solve(uint32_t n, const SolveCtl& S,
                                          const unsigned long long* __restrict__ counters,
                                          pbf_solve_record* __restrict__ log,
                                          unsigned long long* __restrict__ count) {
  const unsigned long long idx = *count;
  const uint32_t k = (uint32_t)counters[C_ITERS];  // 1..kMaxSolveSlots
  const uint32_t nn = n ? n : 1u;
  pbf_solve_record r;
  r.index = idx;
  r.iterations = k;
  r.warm_start_kept = (int32_t)counters[C_WARM_KEPT];
  r.max_error = max_error_of(S, (int)k);
  r.mean_error = mean_error_of(S, (int)k, nn);
  r.max_error_before_warm_start = max_error_of(S, 0);
  r.mean_error_before_warm_start = mean_error_of(S, 0, nn);
  if ((threadIdx.x & 63u) != 0u) return;
  log[idx % PBF_SOLVE_LOG_SIZE] = r;
  *count = idx + 1;
}

// The end of a solve: update_velocities (particles.h:375-385; the density
// rides in v.w for the passes that follow), the kept warm multipliers (null:
// none) join the sum, and block 0's first wavefront writes the record.
__global__ void __launch_bounds__(kBlock) k_solve_end(uint32_t n, KParams K, SolveCtl S,
                                                      const float4* __restrict__ x, const float4* __restrict__ xs,
                                                      const float* __restrict__ rho, float4* __restrict__ v,
                                                      const float* __restrict__ warm, float* __restrict__ lsum,
                                                      const unsigned long long* __restrict__ counters,
                                                      pbf_solve_record* __restrict__ log,
                                                      unsigned long long* __restrict__ count) {
  if (blockIdx.x == 0 && threadIdx.x < 64u) log_solve(n, S, counters, log, count);
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  f3 vel = div3(sub3(ld3(xs, p), ld3(x, p)), K.dt);
  if ((double)magsq3(vel) < K.vthr) vel = {0.f, 0.f, 0.f};
  v[p] = make_float4(vel.x, vel.y, vel.z, rho[p]);
  if (warm) {
    const unsigned long long kept = counters[C_WARM_KEPT];
    if (kept != 0ull) lsum[p] += kept == 2ull ? kWarmRetryScale * warm[p] : warm[p];
  }
}

void launch_solve_end(pbf_context* c, const float* warm) {
  const SolveCtl S{-1.0f, 0, 0, c->ehist, c->esum, nullptr, nullptr, 0, 0};
  KernelTimer* t = timer_begin(c, "solve_end");
  hipLaunchKernelGGL(k_solve_end, dim3(std::max(1u, nblocks(c->n))), dim3(kBlock), 0, c->stream, (uint32_t)c->n,
                     c->K, S, (const float4*)c->x, (const float4*)c->xs, (const float*)c->rho, c->v, warm, c->lsum,
                     (const unsigned long long*)c->counters, c->slog, c->slog_count);
  timer_end(c, t);
}

// every row's shards combined, for the host
__global__ void __launch_bounds__(64) k_combine_errors(SolveCtl S, uint32_t* __restrict__ ehist_row,
                                                       unsigned long long* __restrict__ esum_row) {
  const float e = max_error_of(S, (int)blockIdx.x);
  const unsigned long long s = wave_sum(S.esum[blockIdx.x * kErrShards + threadIdx.x]);
  if (threadIdx.x == 0) {
    ehist_row[blockIdx.x] = __float_as_uint(e);
    esum_row[blockIdx.x] = s;
  }
}

void launch_combine_errors(pbf_context* c) {
  const SolveCtl S{-1.0f, 0, 0, c->ehist, c->esum, nullptr, nullptr, 0, 0};
  hipLaunchKernelGGL(k_combine_errors, dim3(kMaxSolveSlots + 1), dim3(64), 0, c->stream, S, c->ehist_row,
                     c->esum_row);
}

#define PBF_VISC_ARGS                                                                                          \
  c->K, (const float4*)c->xs, (const float4*)c->v, c->va, (const int32_t*)c->nbr, (const int32_t*)c->nbr_count, \
      c->cnb, c->cnb_count, (const unsigned long long*)c->counters, (const int32_t*)c->snb,                     \
      (const int32_t*)c->snb_count, c->skin_hint
void launch_viscosity_first(pbf_context* c) {
  switch (tail_lanes(c)) {
    case 16: PBF_LAUNCH_LANES(c, "viscosity", 16, k_viscosity_first<16>, PBF_VISC_ARGS); break;
    case 4: PBF_LAUNCH_LANES(c, "viscosity", 4, k_viscosity_first<4>, PBF_VISC_ARGS); break;
    default: PBF_LAUNCH_STAGED(c, "viscosity", k_viscosity_first_lane, PBF_VISC_ARGS);
  }
}

// the vorticity passes stay exact in both arithmetic modes; the static-range
// instance of the divide where KParams::static_ranges holds
#define PBF_LAUNCH_SR_AS(c, name, KT, L, ...)                         \
  do {                                                                \
    if ((c)->K.static_ranges)                                         \
      PBF_LAUNCH_LANES(c, name, L, (KT<true, L>), __VA_ARGS__);       \
    else                                                              \
      PBF_LAUNCH_LANES(c, name, L, (KT<false, L>), __VA_ARGS__);      \
  } while (0)
#define PBF_LAUNCH_SR(c, name, KT, ...)                               \
  switch (tail_lanes(c)) {                                            \
    case 16: PBF_LAUNCH_SR_AS(c, name, KT, 16, __VA_ARGS__); break;   \
    case 4: PBF_LAUNCH_SR_AS(c, name, KT, 4, __VA_ARGS__); break;     \
    default: PBF_LAUNCH_SR_AS(c, name, KT, 1, __VA_ARGS__);           \
  }

void launch_vorticity_masked(pbf_context* c) {
  PBF_LAUNCH_SR(c, "vorticity", k_vorticity_c, c->K, (const float4*)c->xs, (const float4*)c->va, c->scr,
                (const int32_t*)c->cnb, (const int32_t*)c->cnb_count);
}

void launch_apply_vorticity_masked(pbf_context* c) {
  PBF_LAUNCH_SR(c, "apply_vorticity", k_apply_vorticity_c, c->K, (const float4*)c->xs,
                (const float4*)c->scr, c->va, (const int32_t*)c->cnb, (const int32_t*)c->cnb_count);
}

#define PBF_LAST_ARGS \
  c->K, (const float4*)c->xs, (const float4*)c->va, c->v, c->x, (const int32_t*)c->cnb, (const int32_t*)c->cnb_count
void launch_viscosity_last(pbf_context* c) {
  switch (tail_lanes(c)) {
    case 16: PBF_LAUNCH_LANES(c, "viscosity_positions", 16, k_viscosity_last<16>, PBF_LAST_ARGS); break;
    case 4: PBF_LAUNCH_LANES(c, "viscosity_positions", 4, k_viscosity_last<4>, PBF_LAST_ARGS); break;
    default: PBF_LAUNCH_LANES(c, "viscosity_positions", 1, k_viscosity_last<1>, PBF_LAST_ARGS);
  }
}

}  // namespace pbf
