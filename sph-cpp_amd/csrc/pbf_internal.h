// pbf_internal.h -- shared declarations of the HIP PBF library (not part of the ABI).
//
// Device data layout (one context, n particles, C cells, K = list cap):
//   x, xs, v         float4[n]   position, position star, velocity, stored in cell order (sorted by
//                                (cell key, original index)); from the velocity update on, v.w holds the
//                                density of the last density pass (gathered by the XSPH passes)
//   xa, xsa, va      float4[n]   reorder targets, swapped with the above
//   xt               float4[n]   position stars after the density pass (hack applied)
//   scr              float4[n]   scratch vector: dp, vorticity or colour field (w: |omega|, or the
//                                density beside the colour)
//   rho, lam         float[n]
//   oid, oida        uint32[n]   original index of each sorted slot
//   key              uint32[n]   cell key of each slot
//   slot             uint32[n]   the kept slots of pbf_remove
//   sk[2], sv[2]     uint32[n]   radix-sort ping-pong buffers (cell key, slot)
//   rhist, rsum      uint32      radix digit histograms of the tiles, and their sums over groups
//   cell_start       uint32[C+2] first sorted slot of every cell (C = the outside bucket)
//   heavy            uint32[n]   particles that a whole wavefront lists (k_fill_heavy)
//   nbr              int32[n/64][K/4][64][4] neighbour lists tiled by groups of 64 particles:
//                                nbr[list_at(k, p, K)] (entries 4j .. 4j+3 of a particle are one
//                                16-byte load, a wavefront's one contiguous kilobyte, its whole
//                                list one block); padded with the far row to a multiple of 8
//   nbr_count        int32[n]
//   cnb, cnb_count   compact lists of the entries within h (same tiling; built by the first
//                                XSPH pass)
//   snb, snb_count   skin lists: the entries within 1.1 h of the positions the lists were built
//                                from (xs0), in list order (same tiling and padding)
//   far row          row `capacity` of the position stars (xs, xsa, xt) holds +inf: a padding
//                                entry of a list reads it and lies outside every radius
//   counters         u64[C_NUM]  overflow, outside, hacks, hack flags, solve state, ...
//   ehist, esum      uint32, u64[kMaxSolveSlots+1][kErrShards]  max (float bits) and sum of the
//                                density errors per solve slot, in shards that their readers combine
//   cstamp           uint32[C+2] == the iteration's stamp: a particle within two cells was moved
//                                by the density fix (cleared with cell_start)
//   lsum, lsuma      float[n]    multipliers summed over the updates of the last solve
//                                (carried through the reorder while a warm start may use them)
//   wlam, wgiven     float[n]    warm-start multipliers (slot order / original order)
//   xsave            float4[n]   position stars before a warm start (for its fallback)
#pragma once

#include <hip/hip_runtime.h>
#include <rocprofiler-sdk-roctx/roctx.h>
#include <stdint.h>

#include <string>
#include <vector>

#include "../../include/pbf.h"

namespace pbf {

// One scene of a batched context: its box (from the origin) and its grid,
// whose cells take the global keys [off, off + ncells).
struct SceneGeo {
  uint32_t dimx, dimy, dimz, off;
  uint32_t ncells, pad;
  uint64_t dxy;
  float bmax[3], pad2;
};

// Constants of one step, computed on the host exactly as the reference
// computes them (kernels.h norms in double, parameters.h derivations).
struct KParams {
  float h, hh, s, ss;            // smoothing radius, h*h, bin spacing, s*s
  float T_h;                     // smallest float d2 with sqrtf(d2) > h
  float T_hack;                  // smallest float d2 with (double)sqrtf(d2) >= 1e-8
  float poly6_norm, spiky_norm, cspline_norm, r_eps;
  float mass, mass_W0;           // rest mass, rest_mass * W(0)
  float rho0, neg_inv_rho0, inv_rho0;
  float g, dt, g_dt;
  float eps, visc, vort, gamma;
  double vthr;                   // 0.000001 * max_speed (particles.h:380), in double
  double st_rmin;                // h * 0.000001 (particles.h:420), in double
  float st_rmin_float;           // smallest float r with (double)r >= st_rmin
  float bmin[3], bmax[3], mover[3];
  uint32_t dimx, dimy, dimz;
  uint32_t ncells;
  uint64_t dxy;
  int cap;
  int stride;                    // list row length: cap rounded up to a multiple of 8
  int count_overflow;            // PBF_OPT_COUNT_OVERFLOW
  float skin2;                   // (1.1 h)^2: the radius of the skin lists
  float disp_lim2;               // (0.045 h)^2: squared moves below it keep the skin lists usable
  int skin_mode;                 // skin lists allowed (no PBF_OPT_FULL_LISTS)
  int tile_lists;                // the cell walk builds the lists (no PBF_OPT_LANE_LISTS)
  int fast;                      // PBF_OPT_FAST_MATH: hardware sqrt and reciprocal in the fused step
  int static_ranges;             // the exact sums' range tests hold for every accepted pair (nb_sqrt, nb_spiky)
  uint32_t pad;                  // the far row (the capacity): what the lists are padded with
  uint32_t heavy_budget;         // candidates before a particle gets a wavefront of its own (crowded, walk_budget, walk_list)
  // batched scenes: ncells is the total over the scenes, sid the scene of each slot
  int batched;
  const SceneGeo* scenes;
  const uint32_t* sid;
};

// The candidates that the cap drops are counted by atomics of every wavefront
// that drops some: on one address they queue up in the cache (500,000
// particles in clumps of 200: 410 us for the list build, 31,250 of them, and
// 150 without the count), so they are spread over this many, which the host
// adds up.
constexpr uint32_t kOverflowShards = 64;
enum Counter {
  C_OVERFLOW = 0,   // kOverflowShards counts
  C_FIRST = kOverflowShards,
  C_OUTSIDE = C_FIRST,
  C_HACKS,
  C_CLEARED,        // pbf_find_neighbors clears the counters before this one
  C_HACK_FLAG = C_CLEARED,     // two flags used on alternate Jacobi iterations
  C_HEAVY = C_HACK_FLAG + 2,   // number of entries in the heavy list
  C_MOVED_N,                   // two counts: particles moved by the density fix, per iteration parity
  C_DONE = C_MOVED_N + 2,      // iterate-to-tolerance: 0, or the slot whose error fell below the tolerance plus one
  C_ITERS,                     // iterate-to-tolerance: slots used
  C_WARM_KEPT,                 // the warm-start positions were kept (2: the damped retry's, PBF_OPT_WARM_RETRY)
  C_DISP,                      // two flags: some particle has moved too far for the skin lists by the
                               // end of the previous Jacobi iteration (parity of the iteration that reads it)
  // (a cache line of 128 bytes on: every wavefront reads C_SKIN, and behind the
  // atomics on C_HEAVY and C_DISP that waited: a pressure update of 256 late
  // scenes in a batch 485 us with the lines apart and 855 in one)
  C_SKIN = C_FIRST + 16,       // 1: this step's skin lists are built
  C_DISP_ALL,                  // the same over the whole step so far
  C_TILE,                      // particles that the cell walk set out to list (with PBF_OPT_COUNT_OVERFLOW;
                               // what it handed on is in C_HEAVY)
  C_RETRY,                     // the warm start grew the error at slot 0 and its damped retry was applied
  C_NUM
};
static_assert(C_DISP + 2 <= C_SKIN, "counters overlap");

constexpr uint32_t kMaxSolveSlots = PBF_MAX_SOLVE_ITERATIONS;
// The error of a slot is gathered by atomics of every wavefront: on one
// address they queue up in the cache (16,384 of them at 1,048,576 particles),
// so they are spread over this many, one per lane of the wavefront that reads
// them back.
constexpr uint32_t kErrShards = 64;
constexpr uint64_t kRowPad = 8;  // padding rows of the float4 particle buffers
constexpr float kWarmLambdaScale = PBF_WARM_LAMBDA_SCALE;

// Per-launch control of the Jacobi loop kernels.  A plain fixed-iteration
// step passes tol < 0 and null pointers.
struct SolveCtl {
  float tol;                   // >= 0: stop once the slot's density error is <= tol
  int warm;                    // a warm-start update was applied before slot 0
  int mean;                    // compare the mean error (else the maximum)
  uint32_t* ehist;             // max error as float bits: row 0 before the warm start, k+1 slot k
  unsigned long long* esum;    // sum of the errors in 2^-32 units, same rows (kErrShards each)
  float* lsum;                 // sum of the applied multipliers (null: not kept)
  const float4* xsave;         // position stars to restore when the warm start is rejected
  int strict;                  // reject the warm start when the max or the mean error grows
  int retry;                   // a rejected warm start is retried at kWarmRetryScale before the fallback to zero
};

// PBF_OPT_WARM_RETRY: the rejected warm start's multipliers are retried at this
// scale (exact in float) before the solve falls back to a zero warm start.
constexpr float kWarmRetryScale = 0.5f;

// The first density pass of a warm-started solve: the learned warm start's
// features, kept in device memory when feat is set, and with wlam set the
// network evaluated on them in the same pass:
// wlam[p] = lprev[p] + scale * net(features of p).
struct FeatCtl {
  float* feat;          // [n][8] (null: the features are not stored)
  const float* lprev;   // previous multiplier sums
  const short* w1;      // bf16 [64][16] first layer (features 8..15 zero)
  const short* w2;      // bf16 [64][64] second layer
  const float* mp;      // fp32 parameters (biases, output layer)
  float scale;
  float* wlam;          // null: no network in this pass
};

// Neighbour lists are tiled by groups of 64 particles, four entries of a
// particle together: entry k of particle p sits at
// ((p / 64) * stride + k - k % 4) * 64 + (p % 64) * 4 + k % 4.  Four entries
// are one 16-byte load, those of a wavefront's 64 particles one contiguous
// kilobyte, and a wavefront's whole list one contiguous block of stride * 256
// bytes.
__host__ __device__ __forceinline__ uint64_t list_at(uint32_t k, uint32_t p, uint32_t stride) {
  return ((uint64_t)(p >> 6) * stride + (k & ~3u)) * 64u + (p & 63u) * 4u + (k & 3u);
}
// entries of the lists of `capacity` particles, with the rows past the last
// list that a walk may load ahead (up to 31 past an entry)
inline uint64_t list_size(uint64_t capacity, uint64_t stride) { return ((capacity + 63) / 64 * stride + 32) * 64; }

// Pinned memory of one object (a context, a warm-start model) that its copies
// from and to ordinary memory go through (pbf_transfer.hip).  One transfer at
// a time: the caller synchronizes the stream before the next one (but see
// upload).
struct HostStage {
  static constexpr uint32_t kSlots = 8;
  static constexpr uint64_t kSlot = 2u << 20;    // bytes of a slot: 16 MB in all at most
  static constexpr uint64_t kTwo = 8u << 20, kFour = 32u << 20;  // from here on two and four threads copy
  static constexpr uint64_t kDirect = 1u << 16;  // up to here kernels read the pinned memory themselves
  unsigned char* pin = nullptr;
  uint64_t slot_bytes = 0;
  uint32_t nslots = 0;
  hipEvent_t done[kSlots] = {};
  // most: bytes of the transfers that it is made for (much larger ones go
  // through it where it has all its slots, and are the runtime's otherwise)
  int create(uint64_t most, uint64_t slot = kSlot);
  void destroy();
  bool fits(uint64_t bytes) const {
    return nslots == kSlots || bytes <= (nslots > 1 ? 2 : 1) * nslots * slot_bytes;
  }
  // whether the host's threads share a transfer
  bool threaded(uint64_t bytes) const { return nslots == kSlots && bytes >= kTwo; }
  // queues the copy on s; a caller reuses host when it has waited for s.  The
  // first chunk goes through slot `slot`: of two transfers with no wait
  // between them the second begins past the first one's.
  int upload(void* dev, const void* host, uint64_t bytes, hipStream_t s, uint32_t slot = 0);
  // waits for s and the copy
  int download(void* host, const void* dev, uint64_t bytes, hipStream_t s);

 private:
  int device = 0;
  hipError_t upload_part(unsigned char* dev, const unsigned char* host, uint64_t bytes, uint64_t chunk, uint32_t first,
                         uint32_t count, hipStream_t s);
  hipError_t download_part(unsigned char* host, const unsigned char* dev, uint64_t bytes, uint64_t chunk,
                           uint32_t first, uint32_t count, hipStream_t s);
  template <class Part>
  hipError_t in_parts(uint64_t bytes, Part part);
};

// What a caller's array lies in: ordinary memory, which copies go through the
// staging memory for, host memory that the runtime has pinned, or memory of
// the device (which callers may pass where an array is expected; managed
// memory counts as such).
enum class Memory { kPageable, kPinned, kDevice };
Memory memory_of(const void* p);

struct KernelTimer {
  std::string name;
  uint64_t launches = 0;
  double total_ms = 0.0;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> pending;
  std::vector<hipEvent_t> spare;  // events of folded launches, reused
};

}  // namespace pbf

struct pbf_context {
  pbf_params P;
  pbf::KParams K;
  hipStream_t stream = nullptr;
  int device = 0;
  uint64_t n = 0, capacity = 0;
  uint64_t dims[3] = {0, 0, 0};
  uint64_t ncells = 0;
  uint64_t grid_alloc = 0;  // cells allocated
  int cap = 60;
  int cap_alloc = 60;  // list rows allocated at pbf_create: the largest cap pbf_set_params accepts
  bool lists_valid = false;
  uint32_t last_iterations = 0;
  uint32_t dirty_stamp = 0;  // incremented per Jacobi iteration of the fused step
  bool last_was_solve = false;  // stats.iterations comes from the device counter
  bool track_lsum = false;      // lsum follows the particles through the reorder

  float4 *x = nullptr, *xs = nullptr, *v = nullptr;
  float4 *xa = nullptr, *xsa = nullptr, *va = nullptr;
  float4 *xt = nullptr, *scr = nullptr;
  float *rho = nullptr, *lam = nullptr, *rhoa = nullptr, *lama = nullptr;
  float4* scra = nullptr;
  uint32_t *oid = nullptr, *oida = nullptr, *key = nullptr;
  uint32_t *slot = nullptr, *tmp = nullptr, *tmpo = nullptr;
  uint32_t *sk[2] = {nullptr, nullptr}, *sv[2] = {nullptr, nullptr};
  uint32_t *rhist = nullptr, *rsum = nullptr;
  int sorted = 0;  // which of sk, sv the last sort left its result in
  uint32_t* heavy = nullptr;
  uint32_t* cstamp = nullptr;  // [cells + 2] == dirty_stamp: a particle within two cells was moved
  uint32_t* dirty = nullptr;  // == dirty_stamp: the particle or one of its neighbours moved
  uint32_t* mflag = nullptr;  // == dirty_stamp: the density fix moved the particle in that iteration
  uint32_t* cell_start = nullptr;
  uint32_t* cbox = nullptr;  // [6][cells] bounding box of each cell's particles (encoded)
  float4* chbox = nullptr;   // [2][n/64] bounding box (min, max) of each aligned run of 64 slots
  uint32_t* scan_partials = nullptr;
  int32_t *nbr = nullptr, *nbr_count = nullptr;
  int32_t *cnb = nullptr, *cnb_count = nullptr;
  int32_t *snb = nullptr, *snb_count = nullptr;  // skin lists (entries within 1.1 h when built)
  float4* xs0 = nullptr;                          // position stars the lists were built from
  // the per-pass entry points may walk the skin lists: pbf_find_neighbors built
  // them and only passes that check their moves have written x* since
  bool pass_skin = false;
  unsigned long long* skin_hint = nullptr;  // 1: the last step's moves kept the skin lists usable
  uint64_t* wmask = nullptr;  // [2][n] within-h masks of the last fused density pass by single lanes
  unsigned long long* counters = nullptr;
  uint32_t* ehist = nullptr;
  unsigned long long* esum = nullptr;
  uint32_t* ehist_row = nullptr;            // their shards combined, for the host
  unsigned long long* esum_row = nullptr;
  float* feat = nullptr;       // [n][8] features of the last warm-started solve
  bool feat_valid = false;
  short *mw1 = nullptr, *mw2 = nullptr;  // learned warm start: bf16 weights
  float* mp = nullptr;                   // and the fp32 parameters
  bool has_model = false;
  float warm_gain = 1.0f;  // learned warm start: Lambda_prev + warm_gain * S * net
  uint32_t nscenes = 1;
  std::vector<pbf::SceneGeo> scene_geo;   // host copy (batched contexts)
  pbf::SceneGeo* scenes = nullptr;        // device copy
  uint32_t *sid = nullptr, *sida = nullptr;  // scene of each slot (batched contexts)
  // captured pair of fused steps (pbf_step_graph)
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  uint64_t graph_n = 0, graph_version = 0;
  std::vector<void*> graph_sig;  // buffer pointers when the graph was captured
  uint64_t version = 0;  // bumped by anything that changes the launches of a step
  bool capturing = false;
  // captured pair of iterate-to-tolerance steps (pbf_solve_graph) and what it was captured for
  hipGraph_t sgraph = nullptr;
  hipGraphExec_t sgraph_exec = nullptr;
  uint64_t sgraph_n = 0, sgraph_version = 0;
  float sgraph_tol = 0.f, sgraph_gain = 0.f;
  uint32_t sgraph_max_it = 0;
  int sgraph_warm = -1;
  std::vector<void*> sgraph_sig;
  // per-solve records: a ring of PBF_SOLVE_LOG_SIZE and the number written so far
  pbf_solve_record* slog = nullptr;
  unsigned long long* slog_count = nullptr;
  pbf_tuning tune{256u, 768u, 8192u};
  int coop_blocks[3] = {-1, -1, -1};  // blocks of a cooperative launch of the persistent Jacobi kernel: exact,
                                      // fast and static-range exact arithmetic (-1: not yet found)
  int coop_cus = 0;               // compute units of the device (found with coop_blocks)
  uint32_t coop_grid = 0;         // blocks of the last step's cooperative launch (0: none)
  unsigned long long* done_host = nullptr;  // pinned copy of C_DONE, polled between slot chunks
  float *lsum = nullptr, *lsuma = nullptr, *wlam = nullptr, *wgiven = nullptr;
  float4* xsave = nullptr;
  bool has_given = false;
  float* stage = nullptr;  // device staging for original-order transfers (4 floats / particle)
  pbf::HostStage host;     // and host staging
  uint64_t* stage64 = nullptr;

  hipEvent_t region_a = nullptr, region_b = nullptr;
  std::vector<pbf::KernelTimer> timers;
};

namespace pbf {

// error plumbing (pbf_api.cpp)
int set_error(int code, const std::string& msg);

// A roctx range over the host side of one entry point (shown by
// rocprofv3 --marker-trace; a push and a pop that return at once when no
// profiler is attached).
struct TraceRange {
  explicit TraceRange(const char* name) { roctxRangePushA(name); }
  ~TraceRange() { roctxRangePop(); }
  TraceRange(const TraceRange&) = delete;
  TraceRange& operator=(const TraceRange&) = delete;
};
#define PBF_TRACE(name) ::pbf::TraceRange pbf_trace_range_(name)
int check_hip(hipError_t e, const char* what);

// timing hooks around launches (pbf_api.cpp)
KernelTimer* timer_begin(pbf_context* c, const char* name);
void timer_end(pbf_context* c, KernelTimer* t);

// ---- launchers (pbf_grid.hip) ----
void launch_fill_u32(uint32_t* p, uint32_t value, uint64_t n, hipStream_t s);
void launch_fill_u64(unsigned long long* p, unsigned long long value, uint64_t n, hipStream_t s);
// exclusive scan of in[0..n) into out[0..n]; out[n] = total.  partials needs scan_partials_size(n).
uint64_t scan_partials_size(uint64_t n);
void launch_exclusive_scan(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* partials, hipStream_t s);
void launch_bin(pbf_context* c, uint64_t bin_end);  // (key, slot) pairs by original index
// What a fused step starts from: iterations and warm for the solve's counters,
// and the first error_words words of its error history cleared.
struct StepInit {
  unsigned long long iterations, warm;
  uint32_t* ehist;
  unsigned long long* esum;
  uint32_t error_words;
};
void launch_predict_bin(pbf_context* c, const StepInit& I);  // forces, prediction and bins of a fused step
void launch_sort(pbf_context* c);                            // radix sort -> c->sorted
// gather the state into cell order, keys and cell bounds with it (without
// all_fields: densities, multipliers and the scratch vector stay where they
// are), or by a permutation of slots
void launch_reorder_cells(pbf_context* c, bool all_fields, bool fused);
void launch_reorder_by(pbf_context* c, const uint32_t* perm);
// How a sort of n keys is cut into tiles, groups of tiles and passes.
struct RadixPlan {
  uint64_t n;
  uint32_t items, ntiles, per_group, ngroups, passes, bits, key_bits;
  bool prefixed;
  uint32_t sum_words() const { return passes * ngroups * 256u; }
};
RadixPlan radix_plan(uint64_t n, uint32_t key_bits);
uint64_t radix_hist_size(uint64_t n);  // words, for any sort of up to n keys
// words of the group sums of any sort: four passes, at most 64 groups
constexpr uint64_t kRadixSumWords = 4ull * 64ull * 256ull;
int radix_sort_pairs(uint32_t* k0, uint32_t* v0, uint32_t* k1, uint32_t* v1, const RadixPlan& P, uint32_t* hist,
                     uint32_t* gsum, hipStream_t s);
int radix_sort_in_place(uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t key_bits, uint32_t* k2, uint32_t* v2,
                        uint32_t* hist, uint32_t* gsum, hipStream_t s);
void launch_fill_neighbors(pbf_context* c, uint64_t fb, uint64_t fe);
int radix_sort_u32(uint32_t* keys, uint32_t* vals, uint64_t n, uint32_t key_bits, hipStream_t s);
void launch_bounds_counting(const uint32_t* sorted, uint64_t n, uint64_t b, uint64_t e, uint32_t* out,
                            int upper, hipStream_t s);

// ---- launchers (pbf_passes.hip) ----
// flags for the particle-local kernel
enum { F_FORCES = 1, F_PREDICT = 2 };
void launch_forces_predict(pbf_context* c, int flags, uint64_t b, uint64_t e);
void launch_density(pbf_context* c, uint64_t b, uint64_t e);  // xs -> xt, rho
// ---- fused-step launchers (pbf_fused.hip): they build and use the compact lists ----
void launch_density_lambda_masked(pbf_context* c, int it, int eslot, const SolveCtl& S,
                                  const FeatCtl& F = FeatCtl{nullptr, nullptr});  // xs -> xt, rho, lam
void launch_combine_errors(pbf_context* c);                            // ehist, esum -> ehist_row, esum_row
void launch_lambda_repair(pbf_context* c, int it, const SolveCtl& S);  // lam from xt for dirty particles
void launch_dp_update_masked(pbf_context* c, int it, int last, const SolveCtl& S);
void launch_warm_dp(pbf_context* c, const float* warm);      // xt, multipliers -> xs (warm start), xsave = xt
// the end of a solve: velocities, the kept warm multipliers (null: none) into
// the sums, and its record
void launch_solve_end(pbf_context* c, const float* warm);
void launch_warm_retry(pbf_context* c, const float* warm);   // the damped warm start after a rejected one (a no-op otherwise)
// the Jacobi loop in one cooperative launch (PBF_OPT_PERSISTENT); advances dirty_stamp by iters
bool persistent_available(pbf_context* c);
uint32_t persistent_capacity(pbf_context* c);  // blocks of it the device holds at once (occupancy query)
bool persistent_fits(pbf_context* c);          // the particles fit one launch of it (one block per CU at most)
int launch_jacobi_persistent(pbf_context* c, uint32_t iters, bool solve, bool last_vel, const SolveCtl& S);
void launch_viscosity_first(pbf_context* c);                  // v -> va, compact lists of the final positions
void launch_vorticity_masked(pbf_context* c);                 // va -> scr
void launch_apply_vorticity_masked(pbf_context* c);           // va += ...
void launch_viscosity_last(pbf_context* c);                   // va -> v, x = x*
void launch_lambda(pbf_context* c, const float4* pos, uint64_t b, uint64_t e);
void launch_dp(pbf_context* c, uint64_t b, uint64_t e);                     // xs, lam -> scr
void launch_update_position_stars(pbf_context* c, uint64_t b, uint64_t e);
void launch_update_velocities(pbf_context* c, uint64_t b, uint64_t e);
void launch_update_positions(pbf_context* c, uint64_t b, uint64_t e);
void launch_viscosity(pbf_context* c, const float4* vin, float4* vout, uint64_t b, uint64_t e);
void launch_vorticity(pbf_context* c, const float4* vin, uint64_t b, uint64_t e);
void launch_apply_vorticity(pbf_context* c, float4* vio, uint64_t b, uint64_t e);
// skin: the colour field may walk the skin lists
void launch_surface_tension(pbf_context* c, uint64_t cb, uint64_t ce, uint64_t b, uint64_t e, bool skin);
// ---- learned warm start (pbf_mlp.hip) ----
// original-order transfer helpers
void launch_gather_out_f4(pbf_context* c, const float4* src, float* dst3, int comps);
void launch_gather_out_f1(pbf_context* c, const float* src, float* dst);
void launch_gather_out_rows(pbf_context* c, const float* src, float* dst, int width);  // [n][width] rows
void launch_scatter_in_f4(pbf_context* c, const float* src3, float4* dst);
void launch_scatter_in_f1(pbf_context* c, const float* src, float* dst);

}  // namespace pbf
