// pbf_walk.h -- neighbour walks shared by the fused step and the per-pass
// kernels: list rows, skin lists, quad walks.
#pragma once

#include "pbf_device.h"

namespace pbf {

constexpr int kBatch = 8;

__device__ __forceinline__ f3 xyz(float4 t) { return {t.x, t.y, t.z}; }

// Eight entries of a list from its row's address (row: entry 0 of the
// particle as four-entry groups, 64 groups apart; k0 a multiple of 8).
__device__ __forceinline__ const int4* list_row(const int32_t* __restrict__ list, uint32_t p, uint32_t stride) {
  return reinterpret_cast<const int4*>(list + list_at(0, p, stride));
}
// (loaded as compiler vectors, not as HIP's int4: with those the pressure
// update's single lanes took 78 us instead of 72 at 1,048,576 particles)
typedef int row4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void load_row(const int4* __restrict__ row, int k0, uint32_t (&q)[kBatch]) {
  const row4* r = reinterpret_cast<const row4*>(row) + (k0 / 4) * 64;
  const row4 a = r[0], b = r[64];
  q[0] = (uint32_t)a.x, q[1] = (uint32_t)a.y, q[2] = (uint32_t)a.z, q[3] = (uint32_t)a.w;
  q[4] = (uint32_t)b.x, q[5] = (uint32_t)b.y, q[6] = (uint32_t)b.z, q[7] = (uint32_t)b.w;
}
// Entries k0 .. k0+7 of particle p's list; entries at or past cnt are
// replaced by p (for the rows that are not padded, and for walks that gather
// from arrays without a far row).
__device__ __forceinline__ void load_batch(const int32_t* __restrict__ list, uint32_t stride, int k0, int cnt,
                                           uint32_t p, uint32_t (&q)[kBatch]) {
  load_row(list_row(list, p, stride), k0, q);
#pragma unroll
  for (int u = 0; u < kBatch; ++u) q[u] = k0 + u < cnt ? q[u] : p;
}

// Whether a position has a NaN or an infinity (or a square past the largest
// float).  The far row is not outside h of such a particle: the distance is a
// NaN, which within_h keeps.  So its list is taken entry by entry up to its
// count; the walks below pass over it and their callers do it on their own.
__device__ __forceinline__ bool lost(f3 x) { return !(magsq3(x) <= 3.402823466e38f); }

// Skin lists (built with the lists, pbf_grid.hip): the entries within
// 1.1 h of the positions the lists were built from (x*_0), in list order.  A
// pass may walk the skin list instead of the full one while no particle has
// moved 0.045 h or more from x*_0: an entry outside the skin list was at
// least 1.1 h away, so it is still farther than 1.01 h, well past h and any
// rounding of the within-h test, and adds nothing to any sum.  The entries
// within h come in the same order, so the sums are the same bit for bit.
// Every position a pressure update writes is checked against that move; a
// larger one (or a NaN position) sets a flag: C_DISP by iteration parity
// (read by the next iteration's passes) and C_DISP_ALL for the rest of the
// step.  The flags are written only when a move is too large, so a step at
// rest issues no atomics.
__device__ __forceinline__ bool skin_usable(const unsigned long long* __restrict__ counters, int flag) {
  return counters[C_SKIN] != 0ull && counters[flag] == 0ull;
}

// the squared move of a new position star from x*_0
__device__ __forceinline__ float move2(f3 nw, float4 x0) { return magsq3(sub3(nw, xyz(x0))); }

// Sets counters[a] and counters[C_DISP_ALL] when a lane's squared move m is
// not below the limit (NaN included); every lane of the wavefront calls it.
__device__ __forceinline__ void record_move(float m, unsigned long long* __restrict__ counters, int a,
                                            const KParams& K) {
  const uint64_t over = __ballot(!(m < K.disp_lim2));
  if (over != 0ull && (threadIdx.x & 63) == 0) {
    if (counters[a] == 0ull) atomicExch(&counters[a], 1ull);
    if (counters[C_DISP_ALL] == 0ull) atomicExch(&counters[C_DISP_ALL], 1ull);
  }
}

// ---------------------------------------------------------------------------
// Quad walks.  Four lanes share a particle: lane u of the quad takes entries
// u, 4 + u, 8 + u, ... of its list, evaluates its pairs, and the terms then
// enter the sums in list order: every lane adds the four lanes' terms one
// after the other (a DPP quad permute in the addition, no LDS), so that all
// four hold the particle's sum, the same bits as one lane's walk.  (A pair
// outside h contributes +0, which leaves a sum that began at +0 or above
// unchanged.)
//
// Why: a walk is a chain of loads and of about 80 operations a pair, which a
// scene too small to fill the chip waits out; a quad has a quarter of the
// steps.  Its gathers are cheaper too: four consecutive entries of one list
// are mostly consecutive slots of one cell (about 15 distinct lines of 128
// bytes a gather at rest, against 31 for 64 particles' k-th neighbours).  The
// price is the ordered sums (a DPP addition takes twice a plain one's time),
// so large scenes stay with single lanes (density_lanes, update_lanes, tail_lanes).
template <int CTRL>
__device__ __forceinline__ float quad_lane(float t) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ void quad_add(float& a, float t) {
  a += quad_lane<0x00>(t);
  a += quad_lane<0x55>(t);
  a += quad_lane<0xAA>(t);
  a += quad_lane<0xFF>(t);
}
__device__ __forceinline__ void quad_sub(float& a, float t) {
  a -= quad_lane<0x00>(t);
  a -= quad_lane<0x55>(t);
  a -= quad_lane<0xAA>(t);
  a -= quad_lane<0xFF>(t);
}
__device__ __forceinline__ void quad_add3(f3& a, f3 t) {
  quad_add(a.x, t.x);
  quad_add(a.y, t.y);
  quad_add(a.z, t.z);
}
// whether any lane of the quad says so
__device__ __forceinline__ bool quad_any(bool b) {
  int t = b ? 1 : 0;
  t |= __builtin_amdgcn_mov_dpp(t, 0xB1, 0xF, 0xF, true);  // lanes 1 0 3 2
  t |= __builtin_amdgcn_mov_dpp(t, 0x4E, 0xF, 0xF, true);  // lanes 2 3 0 1
  return t != 0;
}
// the quad lane's entries of particle p's list: entry k0 + u is row[k0 * 64]
__device__ __forceinline__ const uint32_t* quad_row(const int32_t* __restrict__ list, uint32_t p, uint32_t stride) {
  return reinterpret_cast<const uint32_t*>(list) + list_at(0, p, stride) + (threadIdx.x & 3u);
}

// L lanes share a particle: 1, 4 (a quad) or 16 (a row of the wavefront, whose
// walks take one entry a lane at a time, summed with row broadcasts)
template <int L>
__device__ __forceinline__ uint32_t particle_of() {
  return (xcd_block() * blockDim.x + threadIdx.x) / (uint32_t)L;
}
template <int L>
__device__ __forceinline__ uint32_t lane_in_group() {
  return threadIdx.x & (uint32_t)(L - 1);
}
template <int I>
__device__ __forceinline__ float row_lane(float t) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(t), 0x150 + I, 0xF, 0xF, true));
}
template <int L, bool SUB>
__device__ __forceinline__ void group_sum(float& a, float t) {
  if constexpr (L == 4) {
    SUB ? quad_sub(a, t) : quad_add(a, t);
  } else {
    static_assert(L == 16, "a row");
#define PBF_ROW_STEP(I) a = SUB ? a - row_lane<I>(t) : a + row_lane<I>(t);
    PBF_ROW_STEP(0) PBF_ROW_STEP(1) PBF_ROW_STEP(2) PBF_ROW_STEP(3) PBF_ROW_STEP(4) PBF_ROW_STEP(5)
    PBF_ROW_STEP(6) PBF_ROW_STEP(7) PBF_ROW_STEP(8) PBF_ROW_STEP(9) PBF_ROW_STEP(10) PBF_ROW_STEP(11)
    PBF_ROW_STEP(12) PBF_ROW_STEP(13) PBF_ROW_STEP(14) PBF_ROW_STEP(15)
#undef PBF_ROW_STEP
  }
}
template <int L>
__device__ __forceinline__ void group_add3(f3& a, f3 t) {
  group_sum<L, false>(a.x, t.x);
  group_sum<L, false>(a.y, t.y);
  group_sum<L, false>(a.z, t.z);
}
// the group's lanes of a ballot
template <int L>
__device__ __forceinline__ uint32_t group_bits(bool b) {
  return (uint32_t)(__ballot(b) >> (threadIdx.x & 63u & ~(uint32_t)(L - 1))) & ((1u << L) - 1u);
}
// A group's way along a list, kEntries entries a step, kMine of them the
// lane's own.  entries() gives the step's, those at or past `left` replaced by
// `past` (PADDED: the list's last eight are whole, and `past` is the far row);
// advance(), after the gathers, loads the next step's under them.
template <int L>
struct GroupRow {
  static constexpr int kEntries = L == 4 ? 8 : 16, kMine = kEntries / L;
  const uint32_t* __restrict__ row;
  uint32_t q[kMine];
  __device__ __forceinline__ GroupRow(const int32_t* __restrict__ list, uint32_t p, uint32_t stride)
      : row(reinterpret_cast<const uint32_t*>(list) + list_at(lane_in_group<L>(), p, stride)) {
    load();
  }
  template <bool PADDED>
  __device__ __forceinline__ void entries(int left, uint32_t past, uint32_t (&out)[kMine]) const {
#pragma unroll
    for (int j = 0; j < kMine; ++j)
      out[j] = (PADDED && L == 4) || (int)lane_in_group<L>() + j * L < left ? q[j] : past;
  }
  __device__ __forceinline__ void advance() {
    row += kEntries * 64;
    load();
  }

 private:
  __device__ __forceinline__ void load() {
#pragma unroll
    for (int j = 0; j < kMine; ++j) q[j] = row[j * L * 64];
  }
};

// Sums of N terms over the entries of a padded list within h of xp, in list
// order.  data(q) loads what the terms need of neighbour q beyond its
// position (entries outside h load the particle's own, which is at hand) and
// term(d, d2, data, t) sets the N terms; near becomes true when a pair lies
// within the near-coincidence distance.
template <int N>
struct Terms {
  float a[N];
};
template <int L, int N, class Data, class Term>
__device__ __forceinline__ void walk_within(const int32_t* __restrict__ list, int cnt, uint32_t p, f3 xp,
                                            const KParams& K, const float4* __restrict__ pos, Terms<N>& sum,
                                            bool& near, Data data, Term term) {
  if (__builtin_expect(lost(xp), 0)) {  // (the same for a quad's lanes, each of which takes the whole list)
    for (int k = 0; k < cnt; ++k) {
      const uint32_t q = (uint32_t)list[list_at((uint32_t)k, p, K.stride)];
      const f3 d = sub3(xp, xyz(gather4(pos, q)));
      const float d2 = magsq3(d);
      near |= d2 < K.T_hack;
      if (!within_h(d2, K)) continue;
      Terms<N> e{};
      term(d, d2, data(q), e);
#pragma unroll
      for (int i = 0; i < N; ++i) sum.a[i] += e.a[i];
    }
    return;
  }
  if constexpr (L != 1) {
    const uint32_t* __restrict__ row = quad_row(list, p, K.stride);
    uint32_t q[2] = {row[0], row[256]};
    for (int k0 = 0; k0 < cnt; k0 += kBatch) {
      const uint32_t qq[2] = {q[0], q[1]};
      const float4 t[2] = {gather4(pos, q[0]), gather4(pos, q[1])};
      row += kBatch * 64;
      q[0] = row[0], q[1] = row[256];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const f3 d = sub3(xp, xyz(t[j]));
        const float d2 = magsq3(d);
        near |= d2 < K.T_hack;
        Terms<N> e{};
        if (within_h(d2, K)) term(d, d2, data(qq[j]), e);
#pragma unroll
        for (int i = 0; i < N; ++i) quad_add(sum.a[i], e.a[i]);
      }
    }
    near = quad_any(near);
  } else {
    const int4* __restrict__ row = list_row(list, p, K.stride);
    uint32_t q[kBatch];
    for (int k0 = 0; k0 < cnt; k0 += kBatch) {
      load_row(row, k0, q);
      float4 t[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) t[u] = gather4(pos, q[u]);
      bool in[kBatch];
      decltype(data(0u)) more[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const float d2 = magsq3(sub3(xp, xyz(t[u])));
        in[u] = within_h(d2, K);
        more[u] = data(in[u] ? q[u] : p);
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) {
        const f3 d = sub3(xp, xyz(t[u]));
        const float d2 = magsq3(d);
        near |= d2 < K.T_hack;
        if (in[u]) {
          Terms<N> e{};
          term(d, d2, more[u], e);
#pragma unroll
          for (int i = 0; i < N; ++i) sum.a[i] += e.a[i];
        }
      }
    }
  }
}
struct NoData {};

}  // namespace pbf
