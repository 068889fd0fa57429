// pbf_grid.hip -- cell binning, stable radix sort, cell bounds, reorder,
// neighbour lists and the sort / bound primitives.
//
// Reference: Simulation/Source/neighbors.h:108-248 (calculate_bin_id,
// calculate_bins, sort_bins, find_bin_bounds, calculate_neighbor_indices,
// fill_neighbors) and Common/sim_algorithms.h:57-99 (sort_by_key,
// lower_bound, upper_bound).
//
// Sort.  The reference's sort_by_key is Thrust's stable sort of (cell key,
// particle index).  Particles here live in cell order from the previous
// step, so a stable sort of the current slots would order by
// (key, previous key, index).  Instead the (key, slot) pairs are listed in
// original-index order (written there by the binning pass) and sorted by a stable LSD radix sort on the key bits (up to 8
// a pass, per-tile histograms, wavefront ballot ranking): the result is
// exactly the (key, original index) order the reference produces.
//
// Lists.  Particles of one cell walk the same 27 cells: a wavefront takes
// them together, one candidate per lane, and appends every particle's accepted
// candidates in walk order through ballots (the cell walk, below), or, where
// few particles share a cell, a lane takes each (sparse_walk).  Particles
// with very many candidates go to a list that one wavefront each works off,
// skipping cells and runs of slots that are too far (k_fill_heavy).  With
// PBF_OPT_LANE_LISTS one lane per particle walks its cells by itself.
#include "pbf_device.h"

namespace pbf {

constexpr int kBlock = 256;

static inline uint32_t nblocks(uint64_t n, int per = kBlock) { return (uint32_t)((n + per - 1) / per); }

__global__ void k_fill_u32(uint32_t* p, uint32_t value, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}
__global__ void k_fill_u64(unsigned long long* p, unsigned long long value, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = value;
}

void launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_fill_u32, dim3(nblocks(n)), dim3(kBlock), 0, s, p, value, n);
}
void launch_fill_u64(unsigned long long* p, unsigned long long value, uint64_t n, hipStream_t s) {
  if (n) hipLaunchKernelGGL(k_fill_u64, dim3(nblocks(n)), dim3(kBlock), 0, s, p, value, n);
}

// ---------------------------------------------------------------------------
// Exclusive scan (three passes: tile sums, scan of tile sums, tile scans).
// A tile is 256 threads x 8 items.  64-wide wavefront scans with __shfl_up.
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t t = __shfl_up(v, d, 64);
    if (lane >= d) v += t;
  }
  return v;
}

// block-wide exclusive scan of one value per thread; returns the block total in *total
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* total) {
  __shared__ uint32_t wsum[kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == 63) wsum[w] = inc;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < kBlock / 64; ++i) {
    const uint32_t s = wsum[i];
    if (i < w) off += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

__global__ void __launch_bounds__(kBlock) k_scan_tiles(const uint32_t* in, uint64_t n, uint32_t* partials) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i)
    if (base + i < n) s += in[base + i];
  uint32_t tot;
  block_excl_scan(s, &tot);
  if (threadIdx.x == 0) partials[blockIdx.x] = tot;
}

// one block scans all tile sums in place (exclusive), looping with a carry
__global__ void __launch_bounds__(kBlock) k_scan_partials(uint32_t* partials, uint32_t np) {
  uint32_t carry = 0;
  for (uint32_t base = 0; base < np; base += kBlock) {
    const uint32_t i = base + threadIdx.x;
    const uint32_t v = i < np ? partials[i] : 0u;
    uint32_t tot;
    const uint32_t ex = block_excl_scan(v, &tot);
    if (i < np) partials[i] = carry + ex;
    carry += tot;
  }
}

__global__ void __launch_bounds__(kBlock) k_scan_apply(const uint32_t* in, uint32_t* out, uint64_t n,
                                                       const uint32_t* partials) {
  const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
  uint32_t vals[kScanItems];
  uint32_t s = 0;
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    vals[i] = (base + i < n) ? in[base + i] : 0u;
    s += vals[i];
  }
  uint32_t tot;
  uint32_t run = block_excl_scan(s, &tot) + partials[blockIdx.x];
#pragma unroll
  for (int i = 0; i < kScanItems; ++i) {
    if (base + i < n) out[base + i] = run;
    run += vals[i];
    if (base + i + 1 == n) out[n] = run;  // total
  }
}

uint64_t scan_partials_size(uint64_t n) { return (n + kScanTile - 1) / kScanTile + 1; }

void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* partials, hipStream_t s) {
  if (n == 0) {
    launch_fill_u32(out, 0u, 1, s);
    return;
  }
  const uint32_t nt = (uint32_t)((n + kScanTile - 1) / kScanTile);
  hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(kBlock), 0, s, in, n, partials);
  hipLaunchKernelGGL(k_scan_partials, dim3(1), dim3(kBlock), 0, s, partials, nt);
  hipLaunchKernelGGL(k_scan_apply, dim3(nt), dim3(kBlock), 0, s, in, out, n, (const uint32_t*)partials);
}

// ---------------------------------------------------------------------------
// calculate_bins (neighbors.h:120-125): the cell key of every slot, listed
// with the slot by original index: a stable sort of that sequence by key is
// the reference's stable sort of (key, index) pairs.
struct BinOut {
  uint32_t *sk, *sv;       // (key, slot) pairs by original index
  uint32_t* gsum;          // the sort's group sums, cleared for its counting passes
  uint32_t gsum_words;
  unsigned long long* counters;
};
__device__ __forceinline__ uint32_t bin_key(f3 ps, uint32_t p, const KParams& K) {
  return cell_key(bin_coord(ps.x, K.s), bin_coord(ps.y, K.s), bin_coord(ps.z, K.s), grid_of(K, p), K);
}

__global__ void __launch_bounds__(kBlock) k_bin(const float4* __restrict__ xs, uint32_t n, uint32_t bin_end,
                                                KParams K, const uint32_t* __restrict__ oid, BinOut B,
                                                unsigned long long* __restrict__ hint) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  for (uint32_t i = p; i < B.gsum_words; i += gridDim.x * blockDim.x) B.gsum[i] = 0u;
  if (p == 0) {  // counted by the list build that follows
    B.counters[C_HEAVY] = 0ull;
    B.counters[C_TILE] = 0ull;
    // skin lists if the moves since the last build kept them usable
    *hint = B.counters[C_DISP_ALL] == 0ull ? 1ull : 0ull;
    B.counters[C_DISP_ALL] = 0ull;
    B.counters[C_SKIN] = 0ull;
  }
  if (p >= n) return;
  const uint32_t o = oid[p];
  uint32_t k = K.ncells;  // particles past the bin span are placed in no cell
  if (o < bin_end) {
    k = bin_key(ld3(xs, p), p, K);
    if (k == K.ncells) atomicAdd(&B.counters[C_OUTSIDE], 1ull);
  }
  B.sk[o] = k;
  B.sv[o] = p;
}

// The start of a fused step in one pass over the particles: what it counts is
// cleared (StepInit), external forces (particles.h:263-270), prediction
// (:275-287) and the cell keys.  (As three launches the forces and the keys
// each read the particles again: 14.2 + 11.7 us at 1,048,576 particles against
// 18.0 so.)  Particles outside the grid are counted with the cell bounds.
__global__ void __launch_bounds__(kBlock) k_predict_bin(uint32_t n, KParams K, const uint32_t* __restrict__ oid,
                                                        const float4* __restrict__ x, float4* __restrict__ v,
                                                        float4* __restrict__ xs, BinOut B, StepInit I) {
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t all = gridDim.x * blockDim.x;
  for (uint32_t i = p; i < B.gsum_words; i += all) B.gsum[i] = 0u;
  for (uint32_t i = p; i < I.error_words; i += all) {
    I.ehist[i] = 0u;
    I.esum[i] = 0ull;
  }
  static_assert(C_NUM <= kBlock, "cleared by the first block");
  if (p < (uint32_t)C_NUM) B.counters[p] = p == C_ITERS ? I.iterations : (p == C_WARM_KEPT ? I.warm : 0ull);
  if (p >= n) return;
  const uint32_t o = oid[p];
  f3 vp = ld3(v, p);
  vp.y += K.g * K.dt;
  st3(v, p, vp);
  f3 ps = add3(ld3(x, p), mul3(vp, K.dt));
  boundary(ps, K, p);
  st3(xs, p, ps);
  B.sk[o] = bin_key(ps, p, K);
  B.sv[o] = p;
}

// the sort of a context's particles: keys go up to ncells (the outside bucket)
static RadixPlan cell_sort_plan(const pbf_context* c) {
  uint32_t bits = 1;
  while (bits < 32 && (c->K.ncells >> bits) != 0) ++bits;
  return radix_plan(c->n, bits);
}
static BinOut bin_out(pbf_context* c) {
  return BinOut{c->sk[0], c->sv[0], c->rsum, cell_sort_plan(c).sum_words(), c->counters};
}

void launch_bin(pbf_context* c, uint64_t bin_end) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "bin");
  hipLaunchKernelGGL(k_bin, dim3(nblocks(n)), dim3(kBlock), 0, c->stream, (const float4*)c->xs, n,
                     (uint32_t)bin_end, c->K, (const uint32_t*)c->oid, bin_out(c), c->skin_hint);
  timer_end(c, t);
}

void launch_predict_bin(pbf_context* c, const StepInit& I) {
  const uint32_t n = (uint32_t)c->n;
  KernelTimer* t = timer_begin(c, "predict_bin");
  hipLaunchKernelGGL(k_predict_bin, dim3(std::max(1u, nblocks(n))), dim3(kBlock), 0, c->stream, n, c->K,
                     (const uint32_t*)c->oid, (const float4*)c->x, c->v, c->xs, bin_out(c), I);
  timer_end(c, t);
}

void launch_sort(pbf_context* c) {
  if (!c->n) return;
  KernelTimer* t = timer_begin(c, "sort");
  c->sorted = radix_sort_pairs(c->sk[0], c->sv[0], c->sk[1], c->sv[1], cell_sort_plan(c), c->rhist, c->rsum,
                               c->stream);
  timer_end(c, t);
}

// find_bin_bounds (neighbors.h:137-148): begin[c] = lower_bound(keys, c);
// end[c] = upper_bound(keys, c) = lower_bound(keys, c + 1) = begin[c + 1].
// The stamps of the cells next to moved particles start every step at zero;
// in a fused step the particles of the outside bucket are counted here.
struct CellOut {
  const uint32_t* sorted;
  uint32_t n, ncells, count_outside;
  uint32_t *start, *cstamp;
  unsigned long long* counters;
};
__device__ __forceinline__ void cell_bounds(uint32_t c, const CellOut& C) {
  if (c > C.ncells + 1) return;
  C.cstamp[c] = 0u;
  uint32_t lo = 0, hi = C.n;
  while (lo < hi) {
    const uint32_t mid = (lo + hi) >> 1;
    if (C.sorted[mid] < c) lo = mid + 1;
    else hi = mid;
  }
  C.start[c] = lo;
  if (c == C.ncells && C.count_outside) C.counters[C_OUTSIDE] = C.n - lo;
}

// Gathers the persistent state into cell order; the first cell_blocks blocks
// find the cells' bounds meanwhile (chains of dependent loads, which the
// gather's traffic covers: 8 us at 1,048,576 particles as a launch of its
// own).
struct ReorderOut {
  float4 *x, *xs, *v, *scr;
  float *rho, *lam, *lsum;
  uint32_t *oid, *key, *sid;
  uint32_t *dirty, *mflag;  // cleared when set (a captured step's stamps repeat)
};
__global__ void __launch_bounds__(kBlock) k_reorder(uint32_t n, uint32_t cell_blocks, CellOut C,
                                                    const uint32_t* __restrict__ perm,
                                                    const float4* __restrict__ x, const float4* __restrict__ xs,
                                                    const float4* __restrict__ v, const float* __restrict__ rho,
                                                    const float* __restrict__ lam, const float4* __restrict__ scr,
                                                    const uint32_t* __restrict__ oid,
                                                    const float* __restrict__ lsum,
                                                    const uint32_t* __restrict__ sid, ReorderOut O) {
  if (blockIdx.x < cell_blocks) {
    cell_bounds(blockIdx.x * blockDim.x + threadIdx.x, C);
    return;
  }
  const uint32_t s = (blockIdx.x - cell_blocks) * blockDim.x + threadIdx.x;
  if (s >= n) return;
  const uint32_t p = perm[s];
  if (lsum) O.lsum[s] = lsum[p];
  if (sid) O.sid[s] = sid[p];
  O.x[s] = x[p];
  O.xs[s] = xs[p];
  O.v[s] = v[p];
  if (rho) {
    O.rho[s] = rho[p];
    O.lam[s] = lam[p];
    O.scr[s] = scr[p];
  }
  if (O.dirty) O.dirty[s] = O.mflag[s] = 0u;
  O.oid[s] = oid[p];
  if (O.key) O.key[s] = C.sorted[s];
}

// all_fields: densities, multipliers and the scratch vector move too; cells:
// after a sort by cell (keys and cell bounds follow), otherwise only by perm
static void reorder(pbf_context* c, const uint32_t* perm, bool all_fields, bool cells, bool fused) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  KernelTimer* t = timer_begin(c, "reorder");
  const CellOut C{cells ? c->sk[c->sorted] : nullptr, n, c->K.ncells, fused ? 1u : 0u, c->cell_start, c->cstamp,
                  c->counters};
  const uint32_t cell_blocks = cells ? nblocks((uint64_t)c->K.ncells + 2) : 0u;
  const bool clear = fused && c->capturing;
  const ReorderOut O{c->xa,   c->xsa,  c->va,  c->scra, c->rhoa, c->lama, c->lsuma,
                     c->oida, cells ? c->key : nullptr, c->sida, clear ? c->dirty : nullptr,
                     clear ? c->mflag : nullptr};
  hipLaunchKernelGGL(k_reorder, dim3(cell_blocks + nblocks(n)), dim3(kBlock), 0, c->stream, n, cell_blocks, C, perm,
                     (const float4*)c->x, (const float4*)c->xs, (const float4*)c->v,
                     all_fields ? (const float*)c->rho : nullptr, (const float*)c->lam, (const float4*)c->scr,
                     (const uint32_t*)c->oid, c->track_lsum ? (const float*)c->lsum : nullptr,
                     c->K.batched ? (const uint32_t*)c->sid : nullptr, O);
  timer_end(c, t);
  if (c->track_lsum) std::swap(c->lsum, c->lsuma);
  if (c->K.batched) {
    std::swap(c->sid, c->sida);
    c->K.sid = c->sid;
  }
  std::swap(c->x, c->xa);
  std::swap(c->xs, c->xsa);
  std::swap(c->v, c->va);
  if (all_fields) {
    std::swap(c->rho, c->rhoa);
    std::swap(c->lam, c->lama);
    std::swap(c->scr, c->scra);
  }
  std::swap(c->oid, c->oida);
}
void launch_reorder_cells(pbf_context* c, bool all_fields, bool fused) {
  reorder(c, c->sv[c->sorted], all_fields, true, fused);
}
void launch_reorder_by(pbf_context* c, const uint32_t* perm) { reorder(c, perm, true, false, false); }

// ---------------------------------------------------------------------------
// Bounding box of every cell's particles, 6 order-preserving integer
// encodings per cell (min x y z, max x y z).  A neighbour walk skips a cell
// whose box is at least s away from the walking particle: float subtraction,
// squaring and addition are monotone, so every candidate's d^2 (computed with
// the same operations) is at least the box bound and none could be accepted.
// The lists are unchanged.  Only the wavefront builder tests cells (of more
// than kBoxMin particles): in the one-lane walk a skip saves time only when
// all 64 lanes skip, which is rare.
//
// The same pass writes the box of every aligned run of 64 slots (a chunk).
// Slots inside a cell are in original-index order, not spatial order, so a
// crowded cell (thousands of particles after a collapse) can be near a
// particle while most of its chunks are not; the wavefront builder tests 64
// chunk boxes at once and gathers only the chunks that can hold a neighbour.
constexpr uint32_t kBoxMin = 32;
constexpr uint32_t kChunkMin = 128;  // cells above this size are walked chunk by chunk

__device__ __forceinline__ uint32_t ord_enc(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord_dec(uint32_t u) {
  return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// an empty box (word i of the boxes)
__device__ __forceinline__ uint32_t box_empty(uint64_t i) { return (i % 6 < 3) ? 0xFFFFFFFFu : 0u; }
__global__ void k_box_init(uint32_t* __restrict__ box, uint64_t count, const unsigned long long* __restrict__ counters) {
  if (counters[C_HEAVY] == 0ull) return;  // the boxes serve only the wavefront builder
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) box[i] = box_empty(i);
}

// Slots are in cell order: each wavefront reduces its runs of equal keys and
// the first lane of a run updates the cell's box.  A block whose slots all lie
// in one cell (a crowded cell holds thousands) updates it once: one update per
// wavefront on the same six words queued up in the cache.
constexpr int kBoxBlock = 1024;
__global__ void __launch_bounds__(kBoxBlock) k_cell_box(uint32_t n, uint32_t ncells, const uint32_t* __restrict__ key,
                                                     const float4* __restrict__ xs, uint32_t* __restrict__ box,
                                                     float4* __restrict__ chbox,
                                                     const unsigned long long* __restrict__ counters) {
  if (counters[C_HEAVY] == 0ull) return;
  const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const bool valid = p < n;
  const uint32_t k = valid ? key[p] : 0xFFFFFFFFu;
  const float4 t = valid ? xs[p] : make_float4(0.f, 0.f, 0.f, 0.f);
  uint32_t mn[3] = {ord_enc(t.x), ord_enc(t.y), ord_enc(t.z)};
  uint32_t mx[3] = {mn[0], mn[1], mn[2]};
  // chunk box over the wavefront's 64 slots (particles outside the grid are
  // never walked and left out)
  {
    const bool in = valid && k < ncells;
    uint32_t cmn[3], cmx[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      cmn[a] = in ? mn[a] : 0xFFFFFFFFu;
      cmx[a] = in ? mx[a] : 0u;
    }
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        cmn[a] = min(cmn[a], (uint32_t)__shfl_xor(cmn[a], d, 64));
        cmx[a] = max(cmx[a], (uint32_t)__shfl_xor(cmx[a], d, 64));
      }
    }
    if (lane == 0 && p < n) {
      const uint32_t ch = p >> 6;
      chbox[2 * ch] = make_float4(ord_dec(cmn[0]), ord_dec(cmn[1]), ord_dec(cmn[2]), 0.f);
      chbox[2 * ch + 1] = make_float4(ord_dec(cmx[0]), ord_dec(cmx[1]), ord_dec(cmx[2]), 0.f);
    }
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t kk = __shfl_down(k, d, 64);
    uint32_t omn[3], omx[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      omn[a] = __shfl_down(mn[a], d, 64);
      omx[a] = __shfl_down(mx[a], d, 64);
    }
    if (lane + d < 64 && kk == k) {
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        mn[a] = min(mn[a], omn[a]);
        mx[a] = max(mx[a], omx[a]);
      }
    }
  }
  const uint32_t first = blockIdx.x * blockDim.x, last = first + blockDim.x - 1;
  const uint32_t kf = key[first];
  if (last < n && key[last] == kf) {  // (the same for the whole block)
    __shared__ uint32_t s_box[6][kBoxBlock / 64];
    if (kf >= ncells) return;
    const uint32_t w = threadIdx.x >> 6;
    if (lane == 0)  // the wavefront is one run: its first lane holds the reduction
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        s_box[a][w] = mn[a];
        s_box[3 + a][w] = mx[a];
      }
    __syncthreads();
    if (threadIdx.x < 6) {
      uint32_t m = s_box[threadIdx.x][0];
      for (int i = 1; i < kBoxBlock / 64; ++i)
        m = threadIdx.x < 3 ? min(m, s_box[threadIdx.x][i]) : max(m, s_box[threadIdx.x][i]);
      if (threadIdx.x < 3)
        atomicMin(&box[6ull * kf + threadIdx.x], m);
      else
        atomicMax(&box[6ull * kf + threadIdx.x], m);
    }
    return;
  }
  const uint32_t prev = __shfl_up(k, 1, 64);
  if (valid && k < ncells && (lane == 0 || prev != k)) {
    uint32_t* b = box + 6ull * k;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      atomicMin(&b[a], mn[a]);
      atomicMax(&b[3 + a], mx[a]);
    }
  }
}

// Whether the list build clears the cell boxes on its way (a grid with few
// cells beside its particles: 8 MB at 1,048,576 particles under a kernel of
// 300 us); a sparse grid's are cleared only when they are needed.
static bool boxes_in_fill(const pbf_context* c) { return (uint64_t)c->K.ncells <= 2 * c->n; }

static void launch_cell_box(pbf_context* c) {
  const uint32_t n = (uint32_t)c->n;
  KernelTimer* t = timer_begin(c, "cell_box");
  const uint64_t count = 6ull * c->K.ncells;
  const unsigned long long* heavy = c->counters;
  if (!boxes_in_fill(c))
    hipLaunchKernelGGL(k_box_init, dim3(nblocks(count)), dim3(kBlock), 0, c->stream, c->cbox, count, heavy);
  hipLaunchKernelGGL(k_cell_box, dim3(nblocks(n, kBoxBlock)), dim3(kBoxBlock), 0, c->stream, n, c->K.ncells,
                     (const uint32_t*)c->key, (const float4*)c->xs, c->cbox, c->chbox, heavy);
  timer_end(c, t);
}

// true when no point of the box [l, h] can lie within s of ps (see above)
__device__ __forceinline__ bool box_far(float lx, float ly, float lz, float hx, float hy, float hz, f3 ps, float ss) {
  const float dx = ps.x < lx ? lx - ps.x : (ps.x > hx ? ps.x - hx : 0.0f);
  const float dy = ps.y < ly ? ly - ps.y : (ps.y > hy ? ps.y - hy : 0.0f);
  const float dz = ps.z < lz ? lz - ps.z : (ps.z > hz ? ps.z - hz : 0.0f);
  return (dx * dx + dy * dy) + dz * dz >= ss;
}
__device__ __forceinline__ bool cell_far(const uint32_t* __restrict__ box, uint32_t cell, f3 ps, float ss) {
  const uint32_t* b = box + 6ull * cell;
  return box_far(ord_dec(b[0]), ord_dec(b[1]), ord_dec(b[2]), ord_dec(b[3]), ord_dec(b[4]), ord_dec(b[5]), ps, ss);
}

// ---------------------------------------------------------------------------
// fill_neighbors (neighbors.h:197-230).  A particle walks its 27 cells in the
// reference's order (x offset outer, z inner; cell ids from the FP
// coordinates x + i*s, neighbors.h:171-185), skips itself and accepts
// d^2 < s^2 while the list has room.  Lists hold sorted slots (list_at).
//
// Tiers with identical results: the cell walk, with a lane per particle in
// sparse wavefronts, and k_fill_heavy (a wavefront per particle) for those that
// it hands on, in scenes of enough particles; with PBF_OPT_LANE_LISTS one lane per particle
// unless its cells hold more than twice K.heavy_budget candidates and its walk
// scans K.heavy_budget of them without filling the list (with the overflow
// count on: more than K.heavy_budget candidates).

struct WalkCells {
  float cx[3], cy[3], cz[3];
};

// a[i] for a loop index i without indexing the array at run time (which
// would put the array in scratch memory)
__device__ __forceinline__ float pick3(const float (&a)[3], int i) { return i == 0 ? a[0] : (i == 1 ? a[1] : a[2]); }

__device__ __forceinline__ WalkCells walk_cells(f3 ps, float s) {
  WalkCells w;
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const float off = (float)(i - 1) * s;
    w.cx[i] = bin_coord(ps.x + off, s);
    w.cy[i] = bin_coord(ps.y + off, s);
    w.cz[i] = bin_coord(ps.z + off, s);
  }
  return w;
}

// Skin lists (with `skin`): the entries within 1.1 h (K.skin2) of the
// positions the lists are built from, in list order; x*_0 = x*.
// The Jacobi passes walk them instead of the full lists while no particle has
// moved far enough for an entry outside them to come within h
// (pbf_fused.hip).
//
// The lane walk: one wavefront per block; each lane stages its entries in its
// own LDS column (entry k of the 64 lanes is contiguous) and writes them out
// at the end.  A staged entry is 16 bits: the slot's offset in its cell (10
// bits), the cell's place in the 27-cell walk (c, 5 bits) and whether the
// candidate lies within the skin radius (bit 15).  The offset stays below
// kMaxCellOffset because a lane walks a cell in full only when its 27 cells
// hold at most that many candidates, and otherwise stops after a budget below
// it.
constexpr int kFillBlock = 64;
constexpr uint32_t kMaxCellOffset = 1024u;

// Appends entries to particle p's list: four of them are one 16-byte store,
// and close() fills the last batch of eight with the far row, so that a walk
// loads whole batches without a test.
struct ListWriter {
  int4* row;
  uint32_t pad, count = 0;
  int4 e;
  __device__ __forceinline__ ListWriter(int32_t* __restrict__ list, uint32_t p, const KParams& K)
      : row(reinterpret_cast<int4*>(list + list_at(0, p, (uint32_t)K.stride))), pad(K.pad) {}
  __device__ __forceinline__ void add(uint32_t slot) {
    e = make_int4(e.y, e.z, e.w, (int)slot);
    if ((++count & 3u) == 0u) row[(count / 4u - 1u) * 64u] = e;
  }
  __device__ __forceinline__ void close() {
    uint32_t k = count;
    while (k & 7u) {
      e = make_int4(e.y, e.z, e.w, (int)pad);
      if ((++k & 3u) == 0u) row[(k / 4u - 1u) * 64u] = e;
    }
  }
};

// candidates a lane scans of a particle that may go to the wavefront builder
__host__ __device__ __forceinline__ uint32_t lane_budget(const KParams& K) {
  return K.heavy_budget < kMaxCellOffset - 8u ? K.heavy_budget : kMaxCellOffset - 8u;
}

// The lane walk of particle p: writes its list and count and returns true,
// or returns false when the particle goes to the wavefront builder (only with
// hand_on; without it there are at most kMaxCellOffset particles, so every
// offset fits).  ovf receives the candidates dropped by the cap.
template <bool SKIN>
__device__ __forceinline__ bool walk_list(uint32_t p, uint32_t n, bool hand_on, uint32_t lane,
                                          uint16_t* __restrict__ s_list,
                                          const float4* __restrict__ xs, const uint32_t* __restrict__ start,
                                          const KParams& K, int32_t* __restrict__ nbr,
                                          int32_t* __restrict__ nbr_count, uint32_t& ovf,
                                          int32_t* __restrict__ snb, int32_t* __restrict__ snb_count) {
  const f3 ps = ld3(xs, p);
  const WalkCells w = walk_cells(ps, K.s);
  const GridView G = grid_of(K, p);
  // the 27 cell ranges first, all loads in flight together (a cell outside
  // the grid is an empty range); the walk then waits only on candidates
  uint32_t cb[27], ce[27];
#pragma unroll
  for (int c = 0; c < 27; ++c) {
    const uint32_t cell = cell_key(pick3(w.cx, c / 9), pick3(w.cy, (c / 3) % 3), pick3(w.cz, c % 3), G, K);
    const bool in = cell < K.ncells;
    const uint32_t cc = in ? cell : 0u;
    const uint32_t b = start[cc], e = start[cc + 1];
    cb[c] = in ? b : 0u;
    ce[c] = in ? e : 0u;
  }
  uint32_t total = 0;
#pragma unroll
  for (int c = 0; c < 27; ++c) total += ce[c] - cb[c];
  // the lane's budget; below kMaxCellOffset - 8 so that a staged offset fits
  // in 10 bits (a batch of 8 may pass the budget before the test)
  const uint32_t hb = lane_budget(K);
  // every candidate must be seen to count the overflow: route by the total
  if (hand_on && K.count_overflow && total > hb) return false;
  // otherwise the walk ends when the list is full; a lane whose 27 cells hold
  // more than twice K.heavy_budget candidates and that has scanned
  // K.heavy_budget of them without filling its list hands the particle over
  // (the wavefront builder starts again and writes the same entries); lanes
  // with fewer candidates walk them all
  const uint32_t budget = hand_on && total > min(2u * hb, kMaxCellOffset) ? hb : 0xFFFFFFFFu;
  uint32_t scanned = 0;
  int count = 0;
  const int cap = K.cap;
#pragma unroll
  for (int c = 0; c < 27; ++c) {
    const uint32_t b = cb[c], e = ce[c];
    // staged form of slot q: (c << 10) + (q - b), computed as q + eb in 16 bits
    const uint32_t eb = ((uint32_t)c << 10) - b;
    // candidates of a cell are contiguous: load 8 at a time, test in order
    // (position buffers carry 8 rows of padding, so the loads need no clamp)
    for (uint32_t q0 = b; q0 < e; q0 += 8) {
      scanned += 8;
      if (scanned > budget && !K.count_overflow) return false;
      float4 t[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) t[u] = xs[q0 + (uint32_t)u];
      // branch-free acceptance: every candidate is stored in row
      // min(count, cap) and only an accepted one advances count, so a
      // rejected one is overwritten by the next accepted one (rows >= the
      // final count, and the spare row cap, are never read)
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const uint32_t q = q0 + (uint32_t)u;
        const float d2 = magsq3(sub3(ps, f3{t[u].x, t[u].y, t[u].z}));
        const bool acc = (q < e) & (q != p) & (d2 < K.ss);
        const uint32_t sb = SKIN ? (uint32_t)(d2 < K.skin2) << 15 : 0u;
        s_list[min(count, cap) * kFillBlock + lane] = (uint16_t)((q + eb) | sb);
        count += acc ? 1 : 0;
      }
      // a full list cannot change any more; only the overflow count could
      if (count >= cap && !K.count_overflow) goto done;
    }
  }
done:
  if (count > cap) {
    ovf = (uint32_t)(count - cap);
    count = cap;
  }
  nbr_count[p] = count;
  // staged entries come in walk order, so the cells' first slots are taken
  // from registers cell by cell
  ListWriter full(nbr, p, K), near(snb, p, K);
  int k = 0;
#pragma unroll
  for (int c = 0; c < 27; ++c) {
    const uint32_t b = cb[c];
    for (; k < count; ++k) {
      const uint32_t e16 = s_list[k * kFillBlock + lane];
      if (((e16 >> 10) & 31u) != (uint32_t)c) break;
      const uint32_t slot = b + (e16 & (kMaxCellOffset - 1u));
      full.add(slot);
      if (SKIN && (e16 >> 15)) near.add(slot);
    }
  }
  full.close();
  if (SKIN) {
    near.close();
    snb_count[p] = (int32_t)near.count;
  }
  return true;
}

// ---------------------------------------------------------------------------
// The cell walk.  A wavefront takes `width` consecutive slots.  Particles with
// the same walk cells (those of a cell, but for rounding in x + i*s) have the
// same candidates in the same order, the cells' slots one after the other: a
// stream.  Eight of them at a time have their positions broadcast into
// registers and go through the stream together, 64 candidates a round, one per
// lane: the ballot of a particle's accepted candidates gives each its place in
// the particle's row in LDS (the accepted before it: mbcnt).  A row takes the
// particle itself too, and the sign bit of an entry says whether it lies
// within the skin radius; one pass over the finished row, a lane per entry,
// takes the particle out and splits the skin list off, which costs less than
// either test in every round.  The eight particles' lists are then written out
// together, 16 bytes a lane.
//
// The slot of a stream position: each cell marks the position where its slots
// begin, and a running maximum over the lanes (DPP) carries the cell's number
// on to the positions that follow, so that a cell of any size takes the same
// time.
//
// Bound: vector instructions, 14 a particle and round out of 170 a particle
// (at rest 373 candidates in six rounds, 56 accepted; issue 98% busy), and in
// small scenes the chain cells -> bounds -> slots -> positions -> tests, which
// is why `width` falls with the scene.  Six wavefronts a SIMD: with the eight
// rounds of a stream in registers there are four, 358 us instead of 306.
// Measured, us a launch at rest, by width (in brackets one wavefront's 64
// particles with bits of acceptance in registers and a lane writing each
// list, which this replaces):
//   particles      4     8    16    32
//         960     14    16    23    38   (66)
//      32,768     28    25    32    47   (76)
//     131,072     68    56    58    65   (93)
//     524,288    229   180   172   173  (203)
//   1,048,576    445   341   314   306  (341)
constexpr uint32_t kRounds = 4;
constexpr uint32_t kChunk = 64u * kRounds;
constexpr uint32_t kMembers = 8;  // particles tested and written out together
constexpr uint32_t kUnit = 2;     // of these, without a branch between them

// The cell walk hands particles with more than crowded() candidates to
// k_fill_heavy, which skips whole cells and runs of slots that are too far: at
// once when the overflow is counted (every candidate must be seen), otherwise
// when it has tested walk_budget() of them and some list of the group is not
// full.  Measured on a collapsed scene of 1,048,576 particles (lists at their
// cap), us a step in both kernels: budget 768 556, 1,536 545, 2,304 567,
// 3,072 584; all candidates up to 3,072, none above 770.
__host__ __device__ __forceinline__ uint32_t crowded(const KParams& K) {
  return (K.count_overflow ? 2u : 4u) * K.heavy_budget;
}
__device__ __forceinline__ uint32_t walk_budget(const KParams& K, uint32_t total) {
  return total > crowded(K) ? (K.count_overflow ? 0u : 2u * K.heavy_budget) : 0xFFFFFFFFu;
}

// v with the lanes' values moved by a DPP control; lanes without a source, and
// rows outside the mask, get 0
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp0(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xF, false);
}
// inclusive sum over lanes 0..31
__device__ __forceinline__ uint32_t sum_scan32(uint32_t v) {
  v += dpp0<0x111, 0xF>(v);  // row_shr 1, 2, 4, 8
  v += dpp0<0x112, 0xF>(v);
  v += dpp0<0x114, 0xF>(v);
  v += dpp0<0x118, 0xF>(v);
  v += dpp0<0x142, 0xA>(v);  // row_bcast 15
  return v;
}
// inclusive maximum over the wavefront
__device__ __forceinline__ uint32_t max_scan64(uint32_t v) {
  v = max(v, dpp0<0x111, 0xF>(v));
  v = max(v, dpp0<0x112, 0xF>(v));
  v = max(v, dpp0<0x114, 0xF>(v));
  v = max(v, dpp0<0x118, 0xF>(v));
  v = max(v, dpp0<0x142, 0xA>(v));
  v = max(v, dpp0<0x143, 0xC>(v));  // row_bcast 31
  return v;
}
__device__ __forceinline__ float read_lane(float v, uint32_t lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), (int)lane));
}
// a lane's place among the lanes of mask m
__device__ __forceinline__ uint32_t rank_in(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
// a uniform value in a vector register: an operation on vector registers alone
// issues in half the time of one with a scalar operand
__device__ __forceinline__ float in_vgpr(float v) {
  float r;
  asm("v_mov_b32 %0, %1" : "=v"(r) : "s"(v));
  return r;
}

// CAP: the largest cap
template <uint32_t CAP>
struct CellWalkLds {
  // words of a row: the list's entries, the particle itself once for each of
  // its walk cells, and a round's past them; in the end the list and, from
  // kNear on, the skin list
  static constexpr uint32_t kPitch = CAP + 92u > 2u * CAP ? CAP + 92u : 2u * CAP, kNear = kPitch - CAP;
  uint32_t row[kMembers * kPitch];
  uint32_t mark[64];  // position j of a chunk: byte j / 64 of word j % 64
  uint32_t base[28];  // first slot of the cell minus its stream offset
};

// the candidates of stream positions [c0, c0 + kChunk): slots and positions
// (past the stream's end: the far row)
template <class Lds>
__device__ __forceinline__ void load_chunk(uint32_t c0, uint32_t total, uint32_t off, uint32_t cm, uint32_t lane, Lds& S, const float4* __restrict__ xs, uint32_t pad,
                                           uint32_t (&slot)[kRounds], f3 (&t)[kRounds]) {
  S.mark[lane] = 0u;
  __syncthreads();
  if (cm != 0u && off >= c0 && off < c0 + kChunk)
    reinterpret_cast<uint8_t*>(S.mark)[((off - c0) & 63u) * 4u + ((off - c0) >> 6)] = (uint8_t)(lane + 1u);
  // the cell that the chunk begins in: the last one that begins at or before c0
  const uint64_t begun = __builtin_amdgcn_ballot_w64(cm != 0u && off <= c0);
  uint32_t carry = 64u - (uint32_t)__builtin_clzll(begun | 1ull);
  __syncthreads();
  const uint32_t word = S.mark[lane];
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) {
    slot[r] = pad;
    if (c0 + r * 64u < total) {
      const uint32_t cell = max(max_scan64((word >> (8u * r)) & 255u), carry);
      carry = (uint32_t)__builtin_amdgcn_readlane((int)cell, 63);
      const uint32_t j = c0 + r * 64u + lane;
      if (j < total) slot[r] = S.base[cell - 1u] + j;
    }
  }
#pragma unroll
  for (uint32_t r = 0; r < kRounds; ++r) t[r] = ld3(xs, slot[r]);
}

// Where particles share their walk cells with few others, or with none (no
// cell at all for one that has left the grid), the cell walk sets up a stream
// for every one or two of them.  There each lane lists a particle: its cells go
// by three at a time, x and y the same, and their candidates four at a time as
// one stream, so that a lane waits for memory nine times twice and rarely
// oftener.  Returns false, with nothing listed, after kSparseMost candidates.
//
// A wavefront takes it when it would set up more streams than its particles
// times 8 / sparse_eighths(): one for three particles, for two, for each; with
// fewer slots a wavefront the streams stay the quicker ones for longer.
// Measured on random points, us a launch by particles a cell, all by streams /
// so (in brackets the tile walk that the cell walk replaced, which wrote no
// skin lists here):
//   particles           3                2               1               0.3             none in the grid
//      32,768      32 (54)         33 (49)         34 (46)         37 / 33 (45)
//     131,072      67 (67)         71 (61)         82 (60)         92 / 81 (58)      90 / 29 (11)
//     300,000     121 / 118 (112) 136 / 122 (104) 159 / 110 (99)  190 / 82 (97)
//   1,000,000     331 / 280 (258) 371 / 237 (245) 457 / 186 (237) 560 / 135 (232)   587 / 50 (35)
// (At 8,192 particles, four slots a wavefront, streams are the quicker ones
// always: 17 to 19, lanes 23 at 0.3 a cell and 42 at three.)
constexpr uint32_t kSparseMost = 256;
__device__ __forceinline__ uint32_t sparse_eighths(uint32_t width) {
  return width >= 32u ? 24u : (width >= 16u ? 16u : (width >= 8u ? 9u : 0u));
}
__device__ __forceinline__ bool sparse_walk(uint32_t p, f3 ps, const float4* __restrict__ xs,
                                            const uint32_t* __restrict__ start, const KParams& K,
                                            int32_t* __restrict__ nbr, int32_t* __restrict__ nbr_count,
                                            int32_t* __restrict__ snb, int32_t* __restrict__ snb_count, bool skin,
                                            uint32_t& ovf) {
  const WalkCells w = walk_cells(ps, K.s);
  const GridView G = grid_of(K, p);
  ListWriter full(nbr, p, K), near(snb, p, K);
  uint32_t dropped = 0, seen = 0;
#pragma unroll 1
  for (int xy = 0; xy < 9; ++xy) {
    uint32_t b[3], m[3];
#pragma unroll
    for (int z = 0; z < 3; ++z) {
      const uint32_t cell = cell_key(pick3(w.cx, xy / 3), pick3(w.cy, xy % 3), w.cz[z], G, K);
      const uint32_t c = cell < K.ncells ? cell : 0u;
      b[z] = start[c];
      m[z] = cell < K.ncells ? start[c + 1] - b[z] : 0u;
    }
    const uint32_t m1 = m[0], m2 = m1 + m[1], total = m2 + m[2];
    seen += total;
    if (seen > kSparseMost) return false;
#pragma unroll 1
    for (uint32_t j0 = 0; j0 < total; j0 += 4) {
      uint32_t q[4];
      f3 t[4];
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const uint32_t j = j0 + u;
        q[u] = j < m1 ? b[0] + j : (j < m2 ? b[1] + (j - m1) : (j < total ? b[2] + (j - m2) : K.pad));
        t[u] = ld3(xs, q[u]);
      }
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const float d2 = magsq3(sub3(ps, t[u]));
        if (!(d2 < K.ss) || q[u] == p) continue;
        if (full.count < (uint32_t)K.cap) {
          full.add(q[u]);
          if (skin && d2 < K.skin2) near.add(q[u]);
        } else {
          ++dropped;
        }
      }
    }
  }
  full.close();
  nbr_count[p] = (int32_t)full.count;
  if (skin) {
    near.close();
    snb_count[p] = (int32_t)near.count;
  }
  ovf += dropped;
  return true;
}

template <class Lds>
__device__ __forceinline__ void cell_walk(uint32_t tb, uint32_t width, uint32_t lane, uint64_t todo, f3 ps, uint32_t key,
                                          const float4* __restrict__ xs, const uint32_t* __restrict__ start,
                                          const KParams& K, int32_t* __restrict__ nbr,
                                          int32_t* __restrict__ nbr_count, int32_t* __restrict__ snb,
                                          int32_t* __restrict__ snb_count, bool skin, bool hand_on, Lds& S,
                                          uint64_t& heavy, uint32_t& ovf) {
  constexpr uint32_t kPitch = Lds::kPitch, kNear = Lds::kNear;
  f3 mid;
  uint64_t even;
  {
    const WalkCells w = walk_cells(ps, K.s);
    mid = {w.cx[1], w.cy[1], w.cz[1]};
    even = __builtin_amdgcn_ballot_w64(w.cx[0] == mid.x - 1.0f && w.cx[2] == mid.x + 1.0f && w.cy[0] == mid.y - 1.0f &&
                                       w.cy[2] == mid.y + 1.0f && w.cz[0] == mid.z - 1.0f && w.cz[2] == mid.z + 1.0f);
  }
  {
    // about as many streams as the cell walk would set up
    const uint32_t before = (uint32_t)__shfl_up((int)key, 1, 64);
    const uint64_t own = __builtin_amdgcn_ballot_w64(lane == 0u || key != before || key >= K.ncells) | ~even;
    if (sparse_eighths(width) * (uint32_t)__builtin_popcountll(own & todo) > 8u * (uint32_t)__builtin_popcountll(todo)) {
      bool listed = false;
      if ((todo >> lane) & 1ull)
        listed = sparse_walk(tb + lane, ps, xs, start, K, nbr, nbr_count, snb, snb_count, skin, ovf);
      todo &= ~__builtin_amdgcn_ballot_w64(listed);
    }
  }
  const uint32_t cap = (uint32_t)K.cap;
  const float ss = in_vgpr(K.ss), ks = in_vgpr(K.skin2);
  while (todo != 0ull) {
    // the particles that walk the same cells as the first one left
    const uint32_t i0 = (uint32_t)__builtin_ctzll(todo);
    const uint32_t key0 = (uint32_t)__builtin_amdgcn_readlane((int)key, (int)i0);
    const f3 mid0 = {read_lane(mid.x, i0), read_lane(mid.y, i0), read_lane(mid.z, i0)};
    uint64_t members = 1ull << i0;
    WalkCells w;
    if (even & members) {
      members = __builtin_amdgcn_ballot_w64(key == key0) & __builtin_amdgcn_ballot_w64(mid.x == mid0.x) &
                __builtin_amdgcn_ballot_w64(mid.y == mid0.y) & __builtin_amdgcn_ballot_w64(mid.z == mid0.z) & even & todo;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const float d = (float)(a - 1);
        w.cx[a] = mid0.x + d, w.cy[a] = mid0.y + d, w.cz[a] = mid0.z + d;
      }
    } else {
      // (x + i*s rounds into another cell, or a coordinate is not finite)
      w = walk_cells({read_lane(ps.x, i0), read_lane(ps.y, i0), read_lane(ps.z, i0)}, K.s);
    }
    todo &= ~members;
    // lanes 0..26: cell `lane` of the walk (x outer, z inner)
    const GridView G = grid_of(K, tb + i0);
    uint32_t cb = 0, cm = 0, cell = K.ncells;
    if (lane < 27u) {
      cell = cell_key(pick3(w.cx, (int)(lane / 9u)), pick3(w.cy, (int)((lane / 3u) % 3u)),
                      pick3(w.cz, (int)(lane % 3u)), G, K);
      if (cell < K.ncells) {
        cb = start[cell];
        cm = start[cell + 1] - cb;
      }
    }
    const uint32_t incl = sum_scan32(cm), off = incl - cm;
    const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 26);
    const uint32_t budget = hand_on ? walk_budget(K, total) : 0xFFFFFFFFu;
    if (budget == 0u) {
      heavy |= members;
      continue;
    }
    // how often a particle meets itself
    const uint32_t own = (uint32_t)__builtin_popcountll(
        __builtin_amdgcn_ballot_w64(lane < 27u && cell == key0 && cell < K.ncells));
    // bytes of a full row: the list's entries and the particle itself; what a
    // round adds past them is overwritten by the next
    const uint32_t room = 4u * (cap + own);
    __syncthreads();  // (the previous stream's reads are done)
    if (lane < 27u) S.base[lane] = cb - off;
    uint32_t idx[kMembers], at[kMembers], ne = 0;  // lanes; LDS bytes of the rows so far
    f3 pi[kMembers];
    uint32_t found = 0;
    auto next_group = [&]() {
      ne = 0;
#pragma unroll
      for (uint32_t e = 0; e < kMembers; ++e) {
        const bool on = members != 0ull;
        idx[e] = on ? (uint32_t)__builtin_ctzll(members) : 0u;
        // (places left over never accept)
        pi[e] = {in_vgpr(on ? read_lane(ps.x, idx[e]) : __builtin_inff()), in_vgpr(read_lane(ps.y, idx[e])),
                 in_vgpr(read_lane(ps.z, idx[e]))};
        at[e] = on ? 0u : room;
        members &= members - (on ? 1ull : 0ull);
        ne += on ? 1u : 0u;
      }
    };
    auto test = [&](uint32_t c, const uint32_t (&slot)[kRounds], const f3 (&t)[kRounds]) {
#pragma unroll
      for (uint32_t r = 0; r < kRounds; ++r) {
        if (c + r * 64u >= total) break;
#pragma unroll
        for (uint32_t e0 = 0; e0 < kMembers; e0 += kUnit) {
          if (e0 >= ne) break;
#pragma unroll
          for (uint32_t e = e0; e < e0 + kUnit; ++e) {
            const float d2 = magsq3(sub3(pi[e], t[r]));
            const uint64_t m = __builtin_amdgcn_ballot_w64(d2 < ss);
            // bit 31: within the skin radius (the sign of the difference)
            const uint32_t v = (__float_as_uint(d2 - ks) & 0x80000000u) | slot[r];
            if (__builtin_amdgcn_inverse_ballot_w64(m))
              *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(S.row + e * kPitch) + (at[e] + (rank_in(m) << 2))) = v;
            const uint32_t f = (uint32_t)__builtin_popcountll(m);
            found += f;
            at[e] = min(at[e] + 4u * f, room);
          }
        }
      }
    };
    // the lists of the group: the rows in order without the particle itself,
    // and their entries within the skin radius
    auto finish = [&]() {
      __syncthreads();
      const uint32_t mine = lane & (kMembers - 1u), q0 = lane / kMembers;
      uint32_t x[kMembers], p = 0, kept = 0, near = 0;
#pragma unroll
      for (uint32_t e = 0; e < kMembers; ++e) x[e] = S.row[e * kPitch + lane];
#pragma unroll
      for (uint32_t e = 0; e < kMembers; ++e) {
        if (e >= ne) break;
        const uint32_t pe = tb + idx[e], have = at[e] >> 2;
        uint32_t* __restrict__ row = S.row + e * kPitch;
        uint32_t k = 0, s = 0;
        auto compact = [&](uint32_t k0, uint32_t x) {
          const uint32_t q = x & 0x7FFFFFFFu;
          const uint64_t m = __builtin_amdgcn_ballot_w64(q != pe) & __builtin_amdgcn_ballot_w64(k0 + lane < have);
          const uint32_t to = k + rank_in(m);
          const uint64_t in = m & __builtin_amdgcn_ballot_w64(to < cap);
          if (__builtin_amdgcn_inverse_ballot_w64(in)) row[to] = q;
          k += (uint32_t)__builtin_popcountll(in);
          if (skin) {
            const uint64_t ms = in & __builtin_amdgcn_ballot_w64((int32_t)x < 0);
            if (__builtin_amdgcn_inverse_ballot_w64(ms)) (row + kNear + s)[rank_in(ms)] = q;
            s += (uint32_t)__builtin_popcountll(ms);
          }
        };
        if (have <= 64u) {
          compact(0u, x[e]);
        } else {  // (everything is read before the lists go over it)
          const uint32_t x1 = row[64u + lane], x2 = kPitch >= 192u ? row[128u + lane] : 0u;
          compact(0u, x[e]);
          compact(64u, x1);
          if (kPitch >= 192u) compact(128u, x2);
        }
        if (mine == e) p = pe, kept = k, near = s;
        found -= k;
      }
      __syncthreads();
      // out, padded to whole batches of eight
      if (mine < ne) {
        const uint64_t to = list_at(0, p, (uint32_t)K.stride);
        const int pad = (int)K.pad;
        auto write = [&](const uint32_t* from, int32_t* __restrict__ list, uint32_t n) {
          int4* out = reinterpret_cast<int4*>(list + to);
          for (uint32_t q = q0; 4u * q < ((n + 7u) & ~7u); q += 64u / kMembers) {
            const uint32_t k = 4u * q;
            const int4 x = *reinterpret_cast<const int4*>(from + k);
            out[q * 64u] = make_int4(k < n ? x.x : pad, k + 1u < n ? x.y : pad, k + 2u < n ? x.z : pad,
                                     k + 3u < n ? x.w : pad);
          }
        };
        write(S.row + mine * kPitch, nbr, kept);
        if (skin) write(S.row + mine * kPitch + kNear, snb, near);
        if (q0 == 0u) {
          nbr_count[p] = (int32_t)kept;
          if (skin) snb_count[p] = (int32_t)near;
        }
      }
      found -= ne * own;
      if (lane == 0u) ovf += found;
      found = 0u;
      __syncthreads();
    };
    uint32_t slot[kRounds];
    f3 t[kRounds];
    while (members != 0ull) {
      const uint64_t group = members;
      next_group();
      bool full = false;
      uint32_t c = 0;
      for (; c < total && c < budget && !full; c += kChunk) {
        load_chunk(c, total, off, cm, lane, S, xs, K.pad, slot, t);
        test(c, slot, t);
        uint32_t least = at[0];
#pragma unroll
        for (uint32_t e = 1; e < kMembers; ++e) least = min(least, at[e]);
        full = least >= room && !K.count_overflow;
      }
      if (c >= total || full) {
        finish();
      } else {
        heavy |= group & ~members;
        found = 0u;
      }
    }
  }
}

// Hand-offs and overflow counts go to the shared counters once per
// wavefront (a same-address atomic per lane serialises in L2 when many
// particles of a collapsed region hand off together).
__device__ __forceinline__ void count_fill(uint64_t hm, uint32_t p, uint32_t ovf, uint32_t lane,
                                           const KParams& K, uint32_t* __restrict__ heavy,
                                           unsigned long long* __restrict__ counters) {
  if (hm != 0ull) {
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(&counters[C_HEAVY], (unsigned long long)__popcll(hm));
    base = __shfl(base, 0, 64);
    if ((hm >> lane) & 1ull) heavy[base + (unsigned long long)__popcll(hm & ((1ull << lane) - 1ull))] = p;
  }
  if (K.count_overflow) {
    unsigned long long ov = ovf;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) ov += __shfl_xor(ov, d, 64);
    if (lane == 0 && ov) atomicAdd(&counters[C_OVERFLOW + blockIdx.x % kOverflowShards], ov);
  }
}

struct FillArgs {
  uint32_t n, fb, fe, width;
  int hand_on;  // k_fill_heavy follows and takes what the walks hand on
  const float4* xs;
  const uint32_t *oid, *key, *start;
  uint32_t* box;
  uint64_t box_words;
  int32_t *nbr, *nbr_count, *snb, *snb_count;
  uint32_t* heavy;
  unsigned long long* counters;
  int skin_mode;
  const unsigned long long* hint;
  float4* xs0;
};

// LANES: one lane per particle (PBF_OPT_LANE_LISTS); CAP: the longest list
template <bool LANES, uint32_t CAP>
__global__ void __launch_bounds__(kFillBlock, LANES ? 1 : (CAP <= 64 ? 6 : 5)) k_fill_neighbors(FillArgs A, KParams K) {
  extern __shared__ __attribute__((aligned(16))) unsigned char s_mem[];
  const uint32_t lane = threadIdx.x;
  const uint32_t tb = xcd_block() * A.width;
  const bool valid = lane < A.width && tb + lane < A.n;
  const uint32_t p = valid ? tb + lane : tb;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + lane; i < A.box_words; i += (uint64_t)gridDim.x * blockDim.x)
    A.box[i] = box_empty(i);
  // skin lists only when the previous step kept them usable to its end
  const int skin = A.skin_mode && *A.hint != 0ull;
  if (skin && blockIdx.x == 0 && lane == 0) A.counters[C_SKIN] = 1ull;
  const uint32_t o = A.oid[p];
  const bool query = valid && o >= A.fb && o < A.fe;
  const float4 ps4 = A.xs[p];
  if (valid) {
    if (A.skin_mode) A.xs0[p] = ps4;
    if (!query) {
      A.nbr_count[p] = 0;
      if (skin) A.snb_count[p] = 0;
    }
  }
  uint32_t ovf = 0;
  uint64_t hm = 0ull;
  if constexpr (LANES) {
    uint16_t* s_list = reinterpret_cast<uint16_t*>(s_mem);  // [cap + 1][kFillBlock]
    bool to_heavy = false;
    if (query)
      to_heavy = skin ? !walk_list<true>(p, A.n, A.hand_on != 0, lane, s_list, A.xs, A.start, K, A.nbr, A.nbr_count, ovf, A.snb, A.snb_count)
                      : !walk_list<false>(p, A.n, A.hand_on != 0, lane, s_list, A.xs, A.start, K, A.nbr, A.nbr_count, ovf, A.snb, A.snb_count);
    hm = __ballot(to_heavy);
  } else {
    __shared__ __attribute__((aligned(16))) CellWalkLds<CAP> S;
    const uint64_t todo = __builtin_amdgcn_ballot_w64(query);
    uint32_t key = A.key[p];
    if (K.batched && key == K.ncells) key += K.sid[p];  // (outside every cell, but in its own scene's grid)
    cell_walk(tb, A.width, lane, todo, xyz3(ps4), key, A.xs, A.start, K, A.nbr, A.nbr_count, A.snb, A.snb_count, skin != 0,
              A.hand_on != 0, S, hm, ovf);
    // (once for all: an atomic a wavefront took 0.5 ms at 8 million particles)
    if (K.count_overflow && blockIdx.x == 0 && lane == 0)
      atomicAdd(&A.counters[C_TILE], (unsigned long long)(min(A.fe, A.n) - min(A.fb, A.n)));
  }
  count_fill(hm, p, ovf, lane, K, A.heavy, A.counters);
}

// A group of 64 candidates of the wavefront builder, one per lane (valid:
// the lane holds a candidate other than p; t: its position): the accepted
// ones are appended in slot order through a ballot.  Returns true when the
// list is full and the walk may end.
__device__ __forceinline__ bool take_group(uint32_t q, bool valid, float4 t, f3 ps, const KParams& K, uint32_t n,
                                           uint32_t p, uint64_t below, uint32_t cap, int32_t* __restrict__ nbr,
                                           uint32_t& count, int skin, int32_t* __restrict__ snb, uint32_t& scount) {
  const float d2 = magsq3(sub3(ps, f3{t.x, t.y, t.z}));
  const bool acc = valid && d2 < K.ss;
  const uint64_t m = __ballot(acc);
  const uint32_t pos = count + (uint32_t)__popcll(m & below);
  if (acc && pos < cap) nbr[list_at(pos, p, K.stride)] = (int32_t)q;
  if (skin) {  // entries of the list (pos < cap) within the skin radius, in order
    const bool in = acc && pos < cap && d2 < K.skin2;
    const uint64_t ms = __ballot(in);
    if (in)
      snb[list_at(scount + (uint32_t)__popcll(ms & below), p, K.stride)] = (int32_t)q;
    scount += (uint32_t)__popcll(ms);
  }
  count += (uint32_t)__popcll(m);
  return count >= cap && !K.count_overflow;
}

// One wavefront per heavy particle; waves stride over the heavy list, whose
// length is read once per wave (every wave exits after the last entry).
__global__ void __launch_bounds__(kBlock) k_fill_heavy(uint32_t n, const float4* __restrict__ xs,
                                                       const uint32_t* __restrict__ start,
                                                       const uint32_t* __restrict__ box,
                                                       const float4* __restrict__ chbox, KParams K,
                                                       int32_t* __restrict__ nbr, int32_t* __restrict__ nbr_count,
                                                       const uint32_t* __restrict__ heavy,
                                                       unsigned long long* __restrict__ counters, int skin_mode,
                                                       const unsigned long long* __restrict__ hint,
                                                       int32_t* __restrict__ snb, int32_t* __restrict__ snb_count) {
  const int skin = skin_mode && *hint != 0ull;
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const uint32_t nwaves = (gridDim.x * blockDim.x) >> 6;
  const uint32_t nheavy = (uint32_t)counters[C_HEAVY];
  const uint64_t below = (1ull << lane) - 1ull;
  const uint32_t cap = (uint32_t)K.cap;
  for (uint32_t h = wave; h < nheavy; h += nwaves) {
    const uint32_t p = heavy[h];
    const f3 ps = ld3(xs, p);
    const WalkCells w = walk_cells(ps, K.s);
    const GridView G = grid_of(K, p);
    uint32_t count = 0;   // accepted so far, uncapped (uniform across the wave)
    uint32_t scount = 0;  // skin entries so far
    // lane c < 27 fetches cell c's range and box test, all in flight at once;
    // the wavefront then walks the cells in order from registers
    uint32_t lb = 0, le = 0;
    if (lane < 27) {
      const uint32_t cell =
          cell_key(pick3(w.cx, (int)lane / 9), pick3(w.cy, ((int)lane / 3) % 3), pick3(w.cz, (int)lane % 3), G, K);
      if (cell < K.ncells) {
        lb = start[cell];
        le = start[cell + 1];
        if (le - lb > kBoxMin && cell_far(box, cell, ps, K.ss)) le = lb;  // far: walk nothing
      }
    }
    for (int c = 0; c < 27; ++c) {
      const uint32_t b = (uint32_t)__shfl((int)lb, c, 64), e = (uint32_t)__shfl((int)le, c, 64);
      if (b == e) continue;
      // candidates come in groups of 64 (one per lane); two groups are
      // loaded before the first is tested, so that two loads of a
      // wavefront are in flight instead of one
      if (e - b <= kChunkMin) {
        for (uint32_t base = b; base < e; base += 128) {
          const uint32_t qa = base + lane, qb = base + 64 + lane;
          const bool va = qa < e && qa != p, vb = qb < e && qb != p;
          float4 ta = make_float4(0.f, 0.f, 0.f, 0.f), tb = ta;
          if (va) ta = xs[qa];
          if (vb) tb = xs[qb];
          if (take_group(qa, va, ta, ps, K, n, p, below, cap, nbr, count, skin, snb, scount)) goto done;
          if (base + 64 < e && take_group(qb, vb, tb, ps, K, n, p, below, cap, nbr, count, skin, snb, scount)) goto done;
        }
        continue;
      }
      // crowded cell: each lane tests one chunk box, then the wavefront
      // gathers the chunks that may hold a neighbour, in slot order
      const uint32_t c_last = (e - 1) >> 6;
      for (uint32_t c0 = b >> 6; c0 <= c_last; c0 += 64) {
        const uint32_t ch = c0 + lane;
        bool near = false;
        if (ch <= c_last) {
          const float4 lo = chbox[2 * ch], hi = chbox[2 * ch + 1];
          near = !box_far(lo.x, lo.y, lo.z, hi.x, hi.y, hi.z, ps, K.ss);
        }
        uint64_t todo = __ballot(near);
        while (todo) {
          const uint32_t ca = (uint32_t)__builtin_ctzll(todo);
          todo &= todo - 1ull;
          const bool two = todo != 0ull;
          const uint32_t cb = two ? (uint32_t)__builtin_ctzll(todo) : ca;
          if (two) todo &= todo - 1ull;
          const uint32_t qa = ((c0 + ca) << 6) + lane, qb = ((c0 + cb) << 6) + lane;
          const bool va = qa >= b && qa < e && qa != p, vb = two && qb >= b && qb < e && qb != p;
          float4 ta = make_float4(0.f, 0.f, 0.f, 0.f), tb = ta;
          if (va) ta = xs[qa];
          if (vb) tb = xs[qb];
          if (take_group(qa, va, ta, ps, K, n, p, below, cap, nbr, count, skin, snb, scount)) goto done;
          if (two && take_group(qb, vb, tb, ps, K, n, p, below, cap, nbr, count, skin, snb, scount)) goto done;
        }
      }
    }
  done:
    // the last batch of eight is filled with the far row
    const uint32_t kept = count < cap ? count : cap;
    if (lane < (8u - (kept & 7u)) % 8u) nbr[list_at(kept + lane, p, K.stride)] = (int32_t)K.pad;
    if (skin && lane < (8u - (scount & 7u)) % 8u) snb[list_at(scount + lane, p, K.stride)] = (int32_t)K.pad;
    if (lane == 0) {
      nbr_count[p] = (int32_t)kept;
      if (skin) snb_count[p] = (int32_t)scount;
      if (count > cap && K.count_overflow)
        atomicAdd(&counters[C_OVERFLOW + h % kOverflowShards], (unsigned long long)(count - cap));
    }
  }
}

// slots a wavefront of the cell walk takes (see there)
static uint32_t fill_width(uint64_t n) { return n <= 16384 ? 4u : (n <= 131072 ? 8u : (n <= 524288 ? 16u : 32u)); }

void launch_fill_neighbors(pbf_context* c, uint64_t fb, uint64_t fe) {
  const uint32_t n = (uint32_t)c->n;
  if (!n) return;
  // x*_0 is kept whenever skin lists may be used, the lists themselves when the
  // previous step's moves stayed below their limit (c->skin_hint)
  const int skin = c->K.skin_mode;
  KernelTimer* t = timer_begin(c, "fill_neighbors");
  const bool lanes = !c->K.tile_lists;
  const uint32_t width = lanes ? (uint32_t)kFillBlock : fill_width(n);
  // A small scene does without the wavefront builder (two launches, about 9 us
  // of a step of 960 particles): its walks hand no particle on, whatever its
  // candidates come to.  They come to more than n where walk cells repeat: x +
  // i*s can round into the cell of x + (i-1)*s (at x = 2.4 with s = 0.12 the
  // walk's x cells are 20, 20 and 21), up to twice an axis.
  const bool wide = c->K.batched || (c->K.dimx >= 3 && c->K.dimy >= 3 && c->K.dimz >= 3);
  const uint32_t hb = lane_budget(c->K);
  const uint32_t most = !lanes ? crowded(c->K)
                               : (c->K.count_overflow ? hb : std::min(2u * hb, kMaxCellOffset));
  const bool hand_on = !wide || n > most;
  const FillArgs A{n, (uint32_t)fb, (uint32_t)fe, width, hand_on ? 1 : 0, c->xs, c->oid, c->key, c->cell_start, c->cbox,
                   boxes_in_fill(c) ? 6ull * c->K.ncells : 0ull, c->nbr, c->nbr_count, c->snb, c->snb_count, c->heavy,
                   c->counters, skin, c->skin_hint, c->xs0};
  const dim3 grid(nblocks(n, (int)width)), block(kFillBlock);
  if (lanes)
    hipLaunchKernelGGL((k_fill_neighbors<true, 0>), grid, block, kFillBlock * (c->K.cap + 1) * sizeof(uint16_t), c->stream,
                       A, c->K);
  else
    // (rows for lists of up to 64 or 128 entries: the longer ones leave LDS for five wavefronts a SIMD instead of six)
    hipLaunchKernelGGL((c->K.cap <= 64 ? k_fill_neighbors<false, 64> : k_fill_neighbors<false, 128>), grid, block, 0,
                       c->stream, A, c->K);
  timer_end(c, t);
  if (!hand_on) return;
  // the cell and chunk boxes of the wavefront builder, built only when some particle went to it
  launch_cell_box(c);
  // enough waves to cover the chip; each loops over the heavy list (usually empty)
  t = timer_begin(c, "fill_heavy");
  const uint32_t blocks = std::min<uint32_t>(nblocks((uint64_t)n * 64), c->tune.heavy_blocks);
  hipLaunchKernelGGL(k_fill_heavy, dim3(blocks), dim3(kBlock), 0, c->stream, n, (const float4*)c->xs,
                     (const uint32_t*)c->cell_start, (const uint32_t*)c->cbox, (const float4*)c->chbox, c->K,
                     c->nbr, c->nbr_count, (const uint32_t*)c->heavy, c->counters, skin,
                     (const unsigned long long*)c->skin_hint, c->snb, c->snb_count);
  timer_end(c, t);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (u32 key, u32 value), up to 8 bits a pass, two
// launches a pass.
//
// Count: a tile's digit histogram, and its sum over groups of tiles (atomics
// of one group's few tiles).  Place: a block adds up what lies before its tile
// in its digits -- the groups before its own, then the tiles before it in the
// group, one coalesced kilobyte of counts each -- scans the digits, ranks its
// keys and stores them.  The counts of a million keys are 16 + 15 rows of that
// at most; the tile-by-tile scan between counting and placing that they
// replace took three launches of 4.5 us each.
//
// Ranks: a wavefront takes its keys of a tile 64 at a time, finds the lanes of
// equal digit with one ballot per digit bit and keeps its running counts in
// LDS, so that the block meets at a barrier twice a tile instead of four times
// every 256 keys.
//
// Tiles of 1,024 keys while there are few (a tile is a block: 32,768 keys give
// 32), of 4,096 above 262,144.  Past 2,048 tiles the rows before a tile are
// too many to add up in every block; k_radix_prefix then turns the groups'
// rows into prefixes first.
RadixPlan radix_plan(uint64_t n, uint32_t key_bits) {
  RadixPlan P{};
  P.n = n;
  P.items = n <= (1ull << 18) ? 4u : 16u;
  const uint64_t tile = (uint64_t)kBlock * P.items;
  P.ntiles = (uint32_t)((n + tile - 1) / tile);
  P.passes = (key_bits + 7) / 8;
  P.bits = (key_bits + P.passes - 1) / P.passes;
  P.key_bits = key_bits;
  P.prefixed = P.ntiles > 2048u;
  if (P.prefixed) {
    P.per_group = (P.ntiles + 63) / 64;
  } else {
    P.per_group = 1;
    while (P.per_group * P.per_group < P.ntiles) P.per_group *= 2;
  }
  // (at most 32 up to 2,048 tiles, 64 of the prefixed sort's)
  P.ngroups = P.ntiles ? (P.ntiles + P.per_group - 1) / P.per_group : 0u;
  return P;
}

template <int ITEMS>
__global__ void __launch_bounds__(kBlock) k_radix_count(const uint32_t* __restrict__ keys, uint64_t n, uint32_t shift,
                                                        uint32_t mask, uint32_t per_group,
                                                        uint32_t* __restrict__ hist, uint32_t* __restrict__ gsum) {
  __shared__ uint32_t h[256];
  h[threadIdx.x] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * ITEMS);
  uint32_t k[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint64_t idx = base + (uint64_t)i * kBlock + threadIdx.x;
    k[i] = idx < n ? keys[idx] : 0u;
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i)
    if (base + (uint64_t)i * kBlock + threadIdx.x < n) atomicAdd(&h[(k[i] >> shift) & mask], 1u);
  __syncthreads();
  const uint32_t c = h[threadIdx.x];
  hist[(uint64_t)blockIdx.x * 256u + threadIdx.x] = c;
  if (c) atomicAdd(&gsum[(uint64_t)(blockIdx.x / per_group) * 256u + threadIdx.x], c);
}

// a group's rows become the counts before each tile within the group
__global__ void __launch_bounds__(kBlock) k_radix_prefix(uint32_t ntiles, uint32_t per_group,
                                                         uint32_t* __restrict__ hist) {
  const uint32_t t0 = blockIdx.x * per_group, t1 = min(ntiles, t0 + per_group);
  uint32_t run = 0;
  for (uint32_t t = t0; t < t1; t += 16) {
    uint32_t c[16];
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) c[i] = t + i < t1 ? hist[(uint64_t)(t + i) * 256u + threadIdx.x] : 0u;
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) {
      if (t + i < t1) hist[(uint64_t)(t + i) * 256u + threadIdx.x] = run;
      run += c[i];
    }
  }
}

template <int ITEMS>
__global__ void __launch_bounds__(kBlock) k_radix_place(const uint32_t* __restrict__ keys,
                                                        const uint32_t* __restrict__ vals, RadixPlan P,
                                                        uint32_t shift, uint32_t bits,
                                                        const uint32_t* __restrict__ hist,
                                                        const uint32_t* __restrict__ gsum,
                                                        uint32_t* __restrict__ okeys, uint32_t* __restrict__ ovals) {
  constexpr int kWaves = kBlock / 64;
  // per wavefront: its running count of each digit, then its first output slot
  // (every access of a wavefront's row between the barriers is that
  // wavefront's own, in program order)
  __shared__ volatile uint32_t s_cnt[kWaves][256];
  const uint32_t d0 = threadIdx.x, lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint64_t base = (uint64_t)blockIdx.x * (kBlock * ITEMS) + w * (64u * ITEMS) + lane;
  uint32_t k[ITEMS], v[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint64_t idx = base + (uint64_t)i * 64u;
    k[i] = idx < P.n ? keys[idx] : 0u;
    v[i] = idx < P.n ? vals[idx] : 0u;
  }
#pragma unroll
  for (int i = 0; i < kWaves; ++i) s_cnt[i][threadIdx.x] = 0u;
  // digit d0: all of it, and what lies before this tile
  const uint32_t group = blockIdx.x / P.per_group;
  uint32_t total = 0, before = 0;
  for (uint32_t g0 = 0; g0 < P.ngroups; g0 += 8) {
    uint32_t c[8];
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) c[i] = g0 + i < P.ngroups ? gsum[(uint64_t)(g0 + i) * 256u + d0] : 0u;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      total += c[i];
      before += g0 + i < group ? c[i] : 0u;
    }
  }
  if (P.prefixed) {
    before += hist[(uint64_t)blockIdx.x * 256u + d0];
  } else {
    for (uint32_t t0 = group * P.per_group; t0 < blockIdx.x; t0 += 8) {
      uint32_t c[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) c[i] = t0 + i < blockIdx.x ? hist[(uint64_t)(t0 + i) * 256u + d0] : 0u;
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) before += c[i];
    }
  }
  uint32_t all;
  before += block_excl_scan(total, &all);  // (its barriers also cover the cleared counts)
  const uint32_t mask = (1u << bits) - 1u;
  const uint64_t lower = (1ull << lane) - 1ull;
  uint32_t rank[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const bool valid = base + (uint64_t)i * 64u < P.n;
    const uint32_t d = (k[i] >> shift) & mask;
    uint64_t peers = __ballot(valid);
    for (uint32_t b = 0; b < bits; ++b) {
      const uint64_t bal = __ballot(((d >> b) & 1u) != 0u);
      peers &= ((d >> b) & 1u) ? bal : ~bal;
    }
    const uint32_t done = s_cnt[w][d], mine = (uint32_t)__popcll(peers & lower);
    rank[i] = done + mine;
    if (valid && mine == 0u) s_cnt[w][d] = done + (uint32_t)__popcll(peers);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kWaves; ++i) {
    const uint32_t c = s_cnt[i][d0];
    s_cnt[i][d0] = before;
    before += c;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    if (base + (uint64_t)i * 64u >= P.n) continue;
    const uint32_t pos = s_cnt[w][(k[i] >> shift) & mask] + rank[i];
    okeys[pos] = k[i];
    ovals[pos] = v[i];
  }
}

// All passes of up to 4,096 keys in one block, in LDS: the launches of the
// passes above (two each) are most of their time then.  Measured on a step's
// sort of 960, 2,048 and 4,096 keys, us with the events that time it: 17, 19
// and 19 in four launches, 9, 12 and 13 in one (960 keys: 5.8 on the device).
constexpr int kSortBlock = 1024;
constexpr uint32_t kSortBlockKeys = 4096;
template <int ITEMS>
__global__ void __launch_bounds__(kSortBlock) k_sort_block(uint32_t* __restrict__ keys, uint32_t* __restrict__ vals,
                                                           uint32_t n, uint32_t key_bits, uint32_t pass_bits) {
  constexpr int kWaves = kSortBlock / 64;
  __shared__ uint32_t s_key[kSortBlock * ITEMS], s_val[kSortBlock * ITEMS];
  __shared__ volatile uint32_t s_cnt[kWaves][256];  // (as in k_radix_place)
  __shared__ uint32_t s_sum[4];
  const uint32_t lane = threadIdx.x & 63u, w = threadIdx.x >> 6;
  const uint32_t base = w * (64u * ITEMS) + lane;
  const uint64_t lower = (1ull << lane) - 1ull;
  uint32_t k[ITEMS], v[ITEMS], rank[ITEMS];
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t idx = base + (uint32_t)i * 64u;
    k[i] = idx < n ? keys[idx] : 0u;
    v[i] = idx < n ? vals[idx] : 0u;
  }
  for (uint32_t shift = 0; shift < key_bits; shift += pass_bits) {
    const uint32_t bits = min(pass_bits, key_bits - shift), mask = (1u << bits) - 1u;
    for (uint32_t d = lane; d < 256u; d += 64u) s_cnt[w][d] = 0u;
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const bool valid = base + (uint32_t)i * 64u < n;
      const uint32_t d = (k[i] >> shift) & mask;
      uint64_t peers = __ballot(valid);
      for (uint32_t b = 0; b < bits; ++b) {
        const uint64_t bal = __ballot(((d >> b) & 1u) != 0u);
        peers &= ((d >> b) & 1u) ? bal : ~bal;
      }
      const uint32_t done = s_cnt[w][d], mine = (uint32_t)__popcll(peers & lower);
      rank[i] = done + mine;
      if (valid && mine == 0u) s_cnt[w][d] = done + (uint32_t)__popcll(peers);
    }
    __syncthreads();
    // digit threadIdx.x: its keys in each wavefront, and all of them
    uint32_t c[kWaves], total = 0;
    if (threadIdx.x < 256u) {
#pragma unroll
      for (int i = 0; i < kWaves; ++i) {
        c[i] = s_cnt[i][threadIdx.x];
        total += c[i];
      }
    }
    const uint32_t incl = wave_incl_scan(total);
    if (threadIdx.x < 256u && lane == 63u) s_sum[w] = incl;
    __syncthreads();
    if (threadIdx.x < 256u) {
      uint32_t at = incl - total;
      for (uint32_t i = 0; i < w; ++i) at += s_sum[i];
#pragma unroll
      for (int i = 0; i < kWaves; ++i) {
        s_cnt[i][threadIdx.x] = at;
        at += c[i];
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      if (base + (uint32_t)i * 64u >= n) continue;
      const uint32_t pos = s_cnt[w][(k[i] >> shift) & mask] + rank[i];
      s_key[pos] = k[i];
      s_val[pos] = v[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
      const uint32_t idx = base + (uint32_t)i * 64u;
      if (idx < n) k[i] = s_key[idx], v[i] = s_val[idx];
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < ITEMS; ++i) {
    const uint32_t idx = base + (uint32_t)i * 64u;
    if (idx < n) keys[idx] = k[i], vals[idx] = v[i];
  }
}

uint64_t radix_hist_size(uint64_t n) { return 256ull * ((n + 1023) / 1024); }
template <int ITEMS>
static void radix_pass(const uint32_t* ki, const uint32_t* vi, uint32_t* ko, uint32_t* vo, const RadixPlan& P,
                       uint32_t shift, uint32_t bits, uint32_t* hist, uint32_t* gsum, hipStream_t s) {
  hipLaunchKernelGGL(k_radix_count<ITEMS>, dim3(P.ntiles), dim3(kBlock), 0, s, ki, P.n, shift, (1u << bits) - 1u,
                     P.per_group, hist, gsum);
  if (P.prefixed) hipLaunchKernelGGL(k_radix_prefix, dim3(P.ngroups), dim3(kBlock), 0, s, P.ntiles, P.per_group, hist);
  hipLaunchKernelGGL(k_radix_place<ITEMS>, dim3(P.ntiles), dim3(kBlock), 0, s, ki, vi, P, shift, bits,
                     (const uint32_t*)hist, (const uint32_t*)gsum, ko, vo);
}

// Stable LSD sort of (keys, vals) by P.key_bits bits, ping-ponging between
// (k0, v0) and (k1, v1); gsum starts at zero.  Returns 0 or 1: the buffer pair
// holding the result.
int radix_sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, const RadixPlan& P, uint32_t* hist,
                     uint32_t* gsum, hipStream_t s) {
  if (P.n <= 1) return 0;
  if (P.n <= kSortBlockKeys) {
    const auto kernel = P.n <= (uint64_t)kSortBlock ? k_sort_block<1> : k_sort_block<4>;
    hipLaunchKernelGGL(kernel, dim3(1), dim3(kSortBlock), 0, s, k0, v0, (uint32_t)P.n, P.key_bits, P.bits);
    return 0;
  }
  uint32_t *ki = k0, *vi = v0, *ko = k1, *vo = v1;
  int which = 0;
  for (uint32_t shift = 0; shift < P.key_bits; shift += P.bits, gsum += 256ull * P.ngroups) {
    const uint32_t bits = std::min(P.bits, P.key_bits - shift);
    if (P.items == 4)
      radix_pass<4>(ki, vi, ko, vo, P, shift, bits, hist, gsum, s);
    else
      radix_pass<16>(ki, vi, ko, vo, P, shift, bits, hist, gsum, s);
    std::swap(ki, ko);
    std::swap(vi, vo);
    which ^= 1;
  }
  return which;
}

// the sort_by_key primitive, the result back in keys and vals
int radix_sort_in_place(uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t key_bits, uint32_t* k2, uint32_t* v2,
                        uint32_t* hist, uint32_t* gsum, hipStream_t s) {
  const RadixPlan P = radix_plan(n, key_bits);
  launch_fill_u32(gsum, 0u, P.sum_words(), s);
  int rc = PBF_OK;
  if (radix_sort_pairs(keys, vals, k2, v2, P, hist, gsum, s)) {
    rc = check_hip(hipMemcpyAsync(keys, k2, n * 4, hipMemcpyDeviceToDevice, s), "sort_by_key copy");
    if (!rc) rc = check_hip(hipMemcpyAsync(vals, v2, n * 4, hipMemcpyDeviceToDevice, s), "sort_by_key copy");
  }
  if (!rc) rc = check_hip(hipGetLastError(), "radix sort launch");
  return rc;
}

int radix_sort_u32(uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t key_bits, hipStream_t s) {
  if (n <= 1) return PBF_OK;
  if (n > 0xFFFFFFFFull) return set_error(PBF_ERR_UNSUPPORTED, "sort_by_key: n must be < 2^32");
  if (key_bits == 0 || key_bits > 32) key_bits = 32;
  uint32_t* ws = nullptr;
  const uint64_t hist = radix_hist_size(n);
  int rc = check_hip(hipMallocAsync((void**)&ws, (2 * n + hist + kRadixSumWords) * 4, s), "hipMallocAsync");
  if (rc) return rc;
  rc = radix_sort_in_place(keys, vals, n, key_bits, ws, ws + n, ws + 2 * n, ws + 2 * n + hist, s);
  (void)hipFreeAsync(ws, s);
  return rc;
}

// lower_bound / upper_bound of every value of a counting range
__global__ void k_bounds(const uint32_t* __restrict__ sorted, uint64_t n, uint64_t b, uint64_t cnt,
                         uint32_t* __restrict__ out, int upper) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= cnt) return;
  const uint64_t val = b + i;
  uint64_t lo = 0, hi = n;
  while (lo < hi) {
    const uint64_t mid = (lo + hi) >> 1;
    const uint64_t k = sorted[mid];
    if (upper ? (k <= val) : (k < val)) lo = mid + 1;
    else hi = mid;
  }
  out[i] = (uint32_t)lo;
}

void launch_bounds_counting(const uint32_t* sorted, uint64_t n, uint64_t b, uint64_t e, uint32_t* out, int upper,
                            hipStream_t s) {
  const uint64_t cnt = e - b;
  if (!cnt) return;
  hipLaunchKernelGGL(k_bounds, dim3(nblocks(cnt)), dim3(kBlock), 0, s, sorted, n, b, cnt, out, upper);
}

}  // namespace pbf
