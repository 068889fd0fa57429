// pbf_mlp.hip -- learned warm start for the iterate-to-tolerance solve.
//
// No counterpart in the reference: its pressure solve starts every step's
// Jacobi iterations from lambda = 0 (Simulation/Source/particles.h:318-358).
// Here an 8-64-64-1 network with SiLU activations maps per-particle features
// of the first density pass to a correction of the previous solve's
// multiplier sums: the warm multiplier is Lambda_prev + S * net(features)
// (pbf_solve, PBF_WARM_LEARNED).
// It is evaluated and trained on the GPU: BF16 operands on MFMA
// (v_mfma_f32_16x16x16_bf16, FP32 accumulation), FP32 master weights, Adam.
//
// The network's layout and forward pass are in pbf_mlp_device.h.  Weight
// gradients contract over particles and go through LDS.
#include <algorithm>
#include <cstring>
#include <random>
#include <vector>

#include "pbf_mlp_device.h"

namespace pbf {

constexpr int kMaxTrainBlocks = 1024;

__device__ __forceinline__ v4s feature_operand(const float* __restrict__ f, bool valid, int g) {
  v4s xb = {0, 0, 0, 0};
  if (valid && g < 2) {
    const float4 t = *(const float4*)(f + 4 * g);
    xb = v4s{f2bf(t.x), f2bf(t.y), f2bf(t.z), f2bf(t.w)};
  }
  return xb;
}

// out[p] = base[p] + scale * net(feat[p]) (base may be null: 0); one
// wavefront per block, 16 particles per step.
__global__ void __launch_bounds__(64) k_mlp_forward(uint32_t n, const float* __restrict__ feat, MlpW W,
                                                    float scale, const float* __restrict__ base,
                                                    float* __restrict__ out) {
  const int l = threadIdx.x, c = l & 15, g = l >> 4;
  v4s a1[4], a2[4][4];
  load_forward_operands(W, c, g, a1, a2);
  const uint32_t groups = (n + 15) / 16;
  for (uint32_t gi = blockIdx.x; gi < groups; gi += gridDim.x) {
    const uint32_t p = gi * 16 + c;
    const bool valid = p < n;
    const v4s xb = feature_operand(feat + (uint64_t)(valid ? p : 0) * kFeat, valid, g);
    v4f z1[4], h1[4], z2[4], h2[4];
    const float y = mlp_forward(W, a1, a2, xb, g, z1, h1, z2, h2);
    if (valid && g == 0) out[p] = base ? base[p] + scale * y : scale * y;
  }
}

// Gradient of the mean squared error over `count` samples idx[0..count) for
// one batch.  Block b handles sample groups b, b + grid, ... of 16 and writes
// its partial gradient to part[b][kNPar] and its partial sum of squared errors
// to lpart[b].
//
// Bound by the chain of one group: operands, two layers and their derivatives
// with an exponential and a divide for every unit, then 19 KB of partials.  A
// block is four wavefronts, each with one of the four tiles of 16 units of
// either layer: a quarter of the operands, exponentials, MFMA and stores each.
// They exchange the activations and derivatives as B operands, and the
// outputs' products, which every wavefront adds up in the order of the units.
// Measured at 4,096 samples (256 blocks), us: 15.4 with one wavefront a block,
// 9.6 so.
__global__ void __launch_bounds__(256) k_mlp_train(uint32_t count, const uint32_t* __restrict__ idx,
                                                   const float* __restrict__ feat, const float* __restrict__ tgt,
                                                   MlpW W, float inv_batch, float* __restrict__ part,
                                                   float* __restrict__ lpart) {
  __shared__ __attribute__((aligned(16))) short sA[kHid * 16];   // [unit][particle]: dZ2
  __shared__ __attribute__((aligned(16))) short sA1[kHid * 16];  // [unit][particle]: dZ1
  __shared__ __attribute__((aligned(16))) short sH[kHid * 16];   // [unit][particle]: H1
  __shared__ __attribute__((aligned(16))) short sX[16 * 16];     // [particle][feature]
  __shared__ v4s sB[4][64], sD[4][64];                           // B operands: H1, dZ2
  __shared__ v4f sP[4][64];                                      // w3 * H2
  const int l = threadIdx.x & 63, t = threadIdx.x >> 6, c = l & 15, g = l >> 4;
  const int r0 = 16 * t + 4 * g;  // the lane's units: r0 .. r0 + 3
  // (the first of two dependent loads of a group goes out before the operands')
  auto sample_of = [&](uint32_t gi) { return gi * 16 + c < count ? idx[gi * 16 + c] : 0u; };
  uint32_t next = sample_of(blockIdx.x);
  const v4s a1 = *(const v4s*)(W.w1 + (16 * t + c) * 16 + 4 * g);
  v4s a2[4], a2t[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    a2[k] = *(const v4s*)(W.w2 + (16 * t + c) * kHid + 16 * k + 4 * g);
    a2t[k] = *(const v4s*)(W.w2t + (16 * t + c) * kHid + 16 * k + 4 * g);
  }
  const v4f b1 = *(const v4f*)(W.p + OFF_B1 + r0), b2 = *(const v4f*)(W.p + OFF_B2 + r0),
            w3 = *(const v4f*)(W.p + OFF_W3 + r0);
  const float b3 = W.p[OFF_B3];
  const v4f zero = {0.f, 0.f, 0.f, 0.f};
  v4f gW2[4] = {zero, zero, zero, zero}, gW1 = zero, db1 = zero, db2 = zero, dw3 = zero;
  float db3 = 0.f, loss = 0.f;
  const uint32_t groups = (count + 15) / 16;
  for (uint32_t gi = blockIdx.x; gi < groups; gi += gridDim.x) {
    const bool valid = gi * 16 + c < count;
    const uint32_t sample = next;
    const v4s xb = feature_operand(feat + (uint64_t)sample * kFeat, valid, g);
    next = gi + gridDim.x < groups ? sample_of(gi + gridDim.x) : 0u;
    const float target = valid ? tgt[sample] : 0.f;
    if (t == 0) *(v4s*)(sX + c * 16 + 4 * g) = xb;
    const v4f acc1 = mfma16(a1, xb, zero);
    v4f z1, z2, h2;
    v4s hb;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      z1[j] = acc1[j] + b1[j];
      hb[j] = f2bf(silu(z1[j]));
      sH[(r0 + j) * 16 + c] = hb[j];
    }
    sB[t][l] = hb;
    __syncthreads();
    v4f acc2 = zero, prod;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc2 = mfma16(a2[k], sB[k][l], acc2);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      z2[j] = acc2[j] + b2[j];
      h2[j] = silu(z2[j]);
      prod[j] = w3[j] * h2[j];
    }
    sP[t][l] = prod;
    __syncthreads();
    float y = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const v4f q = sP[k][l];
#pragma unroll
      for (int j = 0; j < 4; ++j) y += q[j];
    }
    y += __shfl_xor(y, 16, 64);
    y += __shfl_xor(y, 32, 64);
    const float diff = valid ? (y + b3) - target : 0.f;
    const float dout = 2.0f * diff * inv_batch;
    if (g == 0) {
      loss += diff * diff;
      db3 += dout;
    }
    v4s db;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      dw3[j] += dout * h2[j];
      const float d = dout * w3[j] * dsilu(z2[j]);
      db2[j] += d;
      db[j] = f2bf(d);
      sA[(r0 + j) * 16 + c] = db[j];
    }
    sD[t][l] = db;
    __syncthreads();
    // dW2 += dZ2 . H1^T (contraction over the 16 particles)
    const v4s A2 = *(const v4s*)(sA + (16 * t + c) * 16 + 4 * g);
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
      gW2[ti] = mfma16(A2, *(const v4s*)(sH + (16 * ti + c) * 16 + 4 * g), gW2[ti]);
    // dH1 = W2^T . dZ2, dZ1 = dH1 * silu'(Z1)
    v4f acc = zero;
#pragma unroll
    for (int k = 0; k < 4; ++k) acc = mfma16(a2t[k], sD[k][l], acc);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = acc[j] * dsilu(z1[j]);
      db1[j] += d;
      sA1[(r0 + j) * 16 + c] = f2bf(d);
    }
    __syncthreads();
    // dW1 += dZ1 . X^T
    const v4s B1 = {sX[(4 * g + 0) * 16 + c], sX[(4 * g + 1) * 16 + c], sX[(4 * g + 2) * 16 + c],
                    sX[(4 * g + 3) * 16 + c]};
    gW1 = mfma16(*(const v4s*)(sA1 + (16 * t + c) * 16 + 4 * g), B1, gW1);
    __syncthreads();
  }
  float* P = part + (uint64_t)blockIdx.x * kNPar;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = r0 + j;
    if (c < kFeat) P[OFF_W1 + r * kFeat + c] = gW1[j];
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) P[OFF_W2 + r * kHid + 16 * ti + c] = gW2[ti][j];
    const float b1s = red16(db1[j]), b2s = red16(db2[j]), w3s = red16(dw3[j]);
    if (c == 0) {
      P[OFF_B1 + r] = b1s;
      P[OFF_B2 + r] = b2s;
      P[OFF_W3 + r] = w3s;
    }
  }
  db3 = red16(db3);
  loss = red16(loss);
  if (threadIdx.x == 0) {
    P[OFF_B3] = db3;
    lpart[blockIdx.x] = loss;
  }
}

// Adam (Kingma & Ba 2015, algorithm 1) on one fp32 master weight.
struct AdamStep {
  float *p, *m, *v;
  float lr, b1, b2, eps, c1, c2;
};
__device__ __forceinline__ float adam_update(const AdamStep& A, uint32_t i, float gr) {
  const float mi = A.b1 * A.m[i] + (1.0f - A.b1) * gr;
  const float vi = A.b2 * A.v[i] + (1.0f - A.b2) * gr * gr;
  A.m[i] = mi;
  A.v[i] = vi;
  const float mh = mi / A.c1, vh = vi / A.c2;
  const float p = A.p[i] - A.lr * mh / (sqrtf(vh) + A.eps);
  A.p[i] = p;
  return p;
}

// the bf16 operand copies of parameter i, whose value is p
__device__ __forceinline__ void refresh_operand(uint32_t i, float p, short* __restrict__ w1, short* __restrict__ w2,
                                                short* __restrict__ w2t) {
  if (i < (uint32_t)OFF_B1) {
    w1[(i / kFeat) * 16 + i % kFeat] = f2bf(p);
  } else if (i >= (uint32_t)OFF_W2 && i < (uint32_t)OFF_B2) {
    const uint32_t j = i - OFF_W2;
    const short b = f2bf(p);
    w2[j] = b;
    w2t[(j % kHid) * kHid + j / kHid] = b;
  }
}

// The end of a batch: grad[i] = sum over the training blocks of part[b][i],
// in block order (deterministic), loss_out[0] = inv_batch * sum of lpart and
// loss_acc[0] += the same; with TRAIN the Adam update and the new bf16
// operands follow in the same launch and the gradient is not stored.
//
// Bound by the latency of the reads: the sum of a parameter is one chain of
// up to 1,024 additions that must stay in order, but its operands need not
// arrive in order.  A block takes 64 parameters; its eight wavefronts load
// kRows rows of the partials at a time (16 loads in flight per lane, the next
// rows under the current sums) into LDS, and one wavefront adds them up.
// Measured for a training epoch of 131,072 samples in batches of 4,096 (256
// rows) with the gradient over all of them: 3.58 ms with one lane per
// parameter reading row after row (72 us a batch, and 4.7 us each for Adam and
// the operands in kernels of their own), 1.23 ms so (1.01 with k_mlp_train's
// four wavefronts a block).
constexpr int kSumBlock = 512;
constexpr uint32_t kRows = 128;
template <bool TRAIN>
__global__ void __launch_bounds__(kSumBlock) k_mlp_finish(uint32_t nblk, const float* __restrict__ part,
                                                          const float* __restrict__ lpart, float inv_batch,
                                                          float* __restrict__ grad, float* __restrict__ loss_out,
                                                          float* __restrict__ loss_acc, AdamStep A,
                                                          short* __restrict__ w1, short* __restrict__ w2,
                                                          short* __restrict__ w2t) {
  constexpr int kWaves = kSumBlock / 64, kPer = kRows / kWaves;
  __shared__ float s_row[kRows][64];
  __shared__ float s_loss[kMaxTrainBlocks];
  const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint32_t i = blockIdx.x * 64 + lane;
  const uint32_t ic = min(i, (uint32_t)kNPar - 1u);
  float next[kPer];
#pragma unroll
  for (int r = 0; r < kPer; ++r) {
    const uint32_t b = w * kPer + (uint32_t)r;
    next[r] = b < nblk ? part[(uint64_t)b * kNPar + ic] : 0.f;
  }
  if (blockIdx.x == 0)
    for (uint32_t b = threadIdx.x; b < nblk; b += kSumBlock) s_loss[b] = lpart[b];
  float s = 0.f;
  for (uint32_t b0 = 0; b0 < nblk; b0 += kRows) {
    __syncthreads();  // the previous rows have been added up
#pragma unroll
    for (int r = 0; r < kPer; ++r) s_row[w * kPer + r][lane] = next[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kPer; ++r) {
      const uint32_t b = b0 + kRows + w * kPer + (uint32_t)r;
      next[r] = b < nblk ? part[(uint64_t)b * kNPar + ic] : 0.f;
    }
    if (w == 0) {
      const uint32_t rows = min(kRows, nblk - b0);
      if (rows == kRows) {
#pragma unroll 32
        for (uint32_t r = 0; r < kRows; ++r) s += s_row[r][lane];
      } else {
        for (uint32_t r = 0; r < rows; ++r) s += s_row[r][lane];
      }
    }
  }
  if (w == 0 && i < (uint32_t)kNPar) {
    if (TRAIN)
      refresh_operand(i, adam_update(A, i, s), w1, w2, w2t);
    else
      grad[i] = s;
  }
  if (blockIdx.x == 0 && w == 1 && lane == 0) {
    float l = 0.f;
#pragma unroll 16
    for (uint32_t b = 0; b < nblk; ++b) l += s_loss[b];
    loss_out[0] = l * inv_batch;
    if (loss_acc) loss_acc[0] += l * inv_batch;
  }
}

// one Adam update with a given gradient
__global__ void k_mlp_adam(const float* __restrict__ grad, AdamStep A, short* __restrict__ w1,
                           short* __restrict__ w2, short* __restrict__ w2t) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (uint32_t)kNPar) refresh_operand(i, adam_update(A, i, grad[i]), w1, w2, w2t);
}

// bf16 operand copies of the weights
__global__ void k_mlp_refresh(const float* __restrict__ p, short* __restrict__ w1, short* __restrict__ w2,
                              short* __restrict__ w2t) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (uint32_t)(kHid * 16)) {
    const int r = i / 16, f = i % 16;
    w1[i] = f < kFeat ? f2bf(p[OFF_W1 + r * kFeat + f]) : (short)0;
  }
  if (i < (uint32_t)(kHid * kHid)) {
    const int o = i / kHid, in = i % kHid;
    const short b = f2bf(p[OFF_W2 + i]);
    w2[i] = b;
    w2t[in * kHid + o] = b;
  }
}

// samples i = 0..n-1 from particle slot i * stride: the features and the
// target (lsum - lprev) / S limited to [-kTargetLimit, kTargetLimit]
constexpr float kTargetLimit = 64.0f;
__global__ void k_take_samples(uint64_t n, uint32_t stride, const float* __restrict__ feat,
                               const float* __restrict__ lsum, const float* __restrict__ lprev, float inv_scale,
                               float* __restrict__ fo, float* __restrict__ to) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const uint64_t p = i * stride;
  const float4* f = (const float4*)(feat + p * kFeat);
  float4* o = (float4*)(fo + i * kFeat);
  o[0] = f[0];
  o[1] = f[1];
  const float t = (lsum[p] - lprev[p]) * inv_scale;
  to[i] = t > -kTargetLimit ? (t < kTargetLimit ? t : kTargetLimit) : -kTargetLimit;
}

}  // namespace pbf

using namespace pbf;

struct pbf_warm_model {
  hipStream_t stream = nullptr;
  float* p = nullptr;  // fp32 master weights
  short *w1 = nullptr, *w2 = nullptr, *w2t = nullptr;
  float *m = nullptr, *v = nullptr, *grad = nullptr;
  float *part = nullptr, *lpart = nullptr, *loss = nullptr, *loss_acc = nullptr;
  float *feat = nullptr, *tgt = nullptr;
  uint32_t *perm = nullptr, *iota = nullptr;
  pbf::HostStage host;
  uint64_t count = 0, max_samples = 0;
  uint64_t adam_t = 0;
  bool has_params = false;
};

namespace pbf {

// Rows that predict has a workspace for (the training batches' partials, which
// nothing holds between calls), so that a call of as many allocates nothing
// (two allocations and their release are 10 of 32 us for 100 rows).
// Calls of more rows allocate theirs and take all rows in one upload, launch
// and download: in blocks of 32,768 with a wait between each, 131,072 and
// 1,000,000 rows took 320 and 2,800 us against 215 and 1,380 so.
constexpr uint64_t kPredictRows = 524288;
static_assert(kPredictRows * (kFeat + 1) <= (uint64_t)kMaxTrainBlocks * kNPar, "predict's rows in the partials");
// two slots of staging memory
constexpr uint64_t kStageSlot = 512u << 10, kStageBytes = 2 * kStageSlot;

static int upload(pbf_warm_model* M, void* dev, const void* host, uint64_t bytes, uint32_t slot = 0) {
  if (memory_of(host) == Memory::kPageable) return M->host.upload(dev, host, bytes, M->stream, slot);
  return check_hip(hipMemcpyAsync(dev, host, bytes, hipMemcpyDefault, M->stream), "upload");
}
static int download(pbf_warm_model* M, void* host, const void* dev, uint64_t bytes) {
  if (memory_of(host) == Memory::kPageable) return M->host.download(host, dev, bytes, M->stream);
  int rc = check_hip(hipMemcpyAsync(host, dev, bytes, hipMemcpyDefault, M->stream), "download");
  return rc ? rc : check_hip(hipStreamSynchronize(M->stream), "download");
}

static MlpW model_weights(const pbf_warm_model* M) { return MlpW{M->w1, M->w2, M->w2t, M->p}; }

static void refresh(pbf_warm_model* M) {
  hipLaunchKernelGGL(k_mlp_refresh, dim3((kHid * kHid + 255) / 256), dim3(256), 0, M->stream, (const float*)M->p,
                     M->w1, M->w2, M->w2t);
}

// the next Adam update (beta 0.9, 0.999, eps 1e-8)
static AdamStep next_adam(pbf_warm_model* M, float learning_rate) {
  const float b1 = 0.9f, b2 = 0.999f;
  ++M->adam_t;
  const float c1 = 1.0f - std::pow(b1, (float)M->adam_t), c2 = 1.0f - std::pow(b2, (float)M->adam_t);
  return AdamStep{M->p, M->m, M->v, learning_rate, b1, b2, 1e-8f, c1, c2};
}

// one batch of samples idx[0..count): its gradient and loss, or with `adam`
// its loss and the Adam update
static void run_batch(pbf_warm_model* M, const uint32_t* idx, uint32_t count, float* loss_acc, const AdamStep* adam) {
  const uint32_t groups = (count + 15) / 16;
  const uint32_t blocks = std::min<uint32_t>(groups, (uint32_t)kMaxTrainBlocks);
  const float inv = 1.0f / (float)count;
  hipLaunchKernelGGL(k_mlp_train, dim3(blocks), dim3(256), 0, M->stream, count, idx, (const float*)M->feat,
                     (const float*)M->tgt, model_weights(M), inv, M->part, M->lpart);
  const dim3 grid((kNPar + 63) / 64);
  if (adam)
    hipLaunchKernelGGL(k_mlp_finish<true>, grid, dim3(kSumBlock), 0, M->stream, blocks, (const float*)M->part,
                       (const float*)M->lpart, inv, (float*)nullptr, M->loss, loss_acc, *adam, M->w1, M->w2, M->w2t);
  else
    hipLaunchKernelGGL(k_mlp_finish<false>, grid, dim3(kSumBlock), 0, M->stream, blocks, (const float*)M->part,
                       (const float*)M->lpart, inv, M->grad, M->loss, loss_acc, AdamStep{}, (short*)nullptr,
                       (short*)nullptr, (short*)nullptr);
}

}  // namespace pbf

extern "C" {

int pbf_warm_model_create(uint64_t max_samples, pbf_warm_model** out) {
  PBF_TRACE("pbf_warm_model_create");
  if (!out) return set_error(PBF_ERR_ARG, "null argument");
  *out = nullptr;
  if (max_samples == 0 || max_samples >= (1ull << 32)) return set_error(PBF_ERR_ARG, "max_samples must be in [1, 2^32)");
  pbf_warm_model* M = new pbf_warm_model();
  M->max_samples = max_samples;
  auto A = [](void** ptr, uint64_t bytes) { return check_hip(hipMalloc(ptr, bytes), "hipMalloc"); };
  int rc;
  if ((rc = check_hip(hipStreamCreateWithFlags(&M->stream, hipStreamNonBlocking), "hipStreamCreate")) ||
      (rc = A((void**)&M->p, kNPar * 4)) || (rc = A((void**)&M->w1, kHid * 16 * 2)) ||
      (rc = A((void**)&M->w2, kHid * kHid * 2)) || (rc = A((void**)&M->w2t, kHid * kHid * 2)) ||
      (rc = A((void**)&M->m, kNPar * 4)) || (rc = A((void**)&M->v, kNPar * 4)) ||
      (rc = A((void**)&M->grad, kNPar * 4)) || (rc = A((void**)&M->part, (uint64_t)kMaxTrainBlocks * kNPar * 4)) ||
      (rc = A((void**)&M->lpart, kMaxTrainBlocks * 4)) || (rc = A((void**)&M->loss, 4)) ||
      (rc = A((void**)&M->loss_acc, 4)) || (rc = A((void**)&M->feat, max_samples * kFeat * 4)) ||
      (rc = A((void**)&M->tgt, max_samples * 4)) || (rc = A((void**)&M->perm, max_samples * 4)) ||
      (rc = A((void**)&M->iota, max_samples * 4)) || (rc = M->host.create(kStageBytes, kStageSlot))) {
    pbf_warm_model_destroy(M);
    return rc;
  }
  std::vector<uint32_t> io(max_samples);
  for (uint64_t i = 0; i < max_samples; ++i) io[i] = (uint32_t)i;
  if ((rc = check_hip(hipMemcpy(M->iota, io.data(), max_samples * 4, hipMemcpyHostToDevice), "upload"))) {
    pbf_warm_model_destroy(M);
    return rc;
  }
  *out = M;
  return PBF_OK;
}

int pbf_warm_model_destroy(pbf_warm_model* M) {
  if (!M) return PBF_OK;
  if (M->stream) hipStreamSynchronize(M->stream);
  void* ptrs[] = {M->p, M->w1, M->w2, M->w2t, M->m, M->v, M->grad, M->part, M->lpart, M->loss, M->loss_acc,
                  M->feat, M->tgt, M->perm, M->iota};
  for (void* q : ptrs)
    if (q) hipFree(q);
  M->host.destroy();
  if (M->stream) hipStreamDestroy(M->stream);
  delete M;
  return PBF_OK;
}

int pbf_warm_model_set_params(pbf_warm_model* M, const float* params) {
  if (!M || !params) return set_error(PBF_ERR_ARG, "null argument");
  int rc = upload(M, M->p, params, kNPar * 4);
  if (rc) return rc;
  refresh(M);
  launch_fill_u32((uint32_t*)M->m, 0u, kNPar, M->stream);
  launch_fill_u32((uint32_t*)M->v, 0u, kNPar, M->stream);
  M->adam_t = 0;
  M->has_params = true;
  return check_hip(hipStreamSynchronize(M->stream), "set_params");
}

int pbf_warm_model_get_params(pbf_warm_model* M, float* params) {
  if (!M || !params) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  return download(M, params, M->p, kNPar * 4);
}

// Uniform(-1/sqrt(fan_in), 1/sqrt(fan_in)) weights, zero biases.
int pbf_warm_model_init(pbf_warm_model* M, uint64_t seed) {
  if (!M) return set_error(PBF_ERR_ARG, "null argument");
  std::mt19937_64 rng(seed);
  std::vector<float> p(kNPar, 0.0f);
  auto fill = [&](int off, int count, float bound) {
    std::uniform_real_distribution<float> u(-bound, bound);
    for (int i = 0; i < count; ++i) p[off + i] = u(rng);
  };
  fill(OFF_W1, kHid * kFeat, 1.0f / std::sqrt((float)kFeat));
  fill(OFF_W2, kHid * kHid, 1.0f / std::sqrt((float)kHid));
  fill(OFF_W3, kHid, 1.0f / std::sqrt((float)kHid));
  return pbf_warm_model_set_params(M, p.data());
}

int pbf_warm_model_clear_samples(pbf_warm_model* M) {
  if (!M) return set_error(PBF_ERR_ARG, "null argument");
  M->count = 0;
  return PBF_OK;
}

int pbf_warm_model_add_samples(pbf_warm_model* M, const float* features, const float* targets, uint64_t count) {
  if (!M || (count && (!features || !targets))) return set_error(PBF_ERR_ARG, "null argument");
  if (M->count + count > M->max_samples) return set_error(PBF_ERR_CAPACITY, "sample store is full");
  float *f = M->feat + M->count * kFeat, *t = M->tgt + M->count;
  const uint64_t bytes = count * kFeat * 4;
  int rc;
  if (bytes > kStageBytes) {  // (the runtime's copies need no wait in between)
    if ((rc = check_hip(hipMemcpyAsync(f, features, bytes, hipMemcpyDefault, M->stream), "upload")) ||
        (rc = check_hip(hipMemcpyAsync(t, targets, count * 4, hipMemcpyDefault, M->stream), "upload")))
      return rc;
  } else {
    // the targets go through the second slot where the features take no more
    // than the first: 1 to 100 samples 21 us, 30 with a wait in between
    const bool apart = bytes <= kStageSlot;
    if ((rc = upload(M, f, features, bytes))) return rc;
    if (!apart && (rc = check_hip(hipStreamSynchronize(M->stream), "upload"))) return rc;
    if ((rc = upload(M, t, targets, count * 4, apart ? 1 : 0))) return rc;
  }
  if ((rc = check_hip(hipStreamSynchronize(M->stream), "upload"))) return rc;
  M->count += count;
  return PBF_OK;
}

// The features of the context's last warm-started solve and the multiplier
// sums that solve applied (scaled by 1/kWarmLambdaScale) of every stride-th
// particle, device to device.
int pbf_warm_model_add_from_context(pbf_warm_model* M, pbf_context* c, uint32_t stride) {
  PBF_TRACE("pbf_warm_model_add_from_context");
  if (!M || !c) return set_error(PBF_ERR_ARG, "null argument");
  if (stride == 0) return set_error(PBF_ERR_ARG, "stride must be >= 1");
  if (!c->feat_valid)
    return set_error(PBF_ERR_STATE,
                     "the context has no features (run a warm-started pbf_solve with PBF_OPT_KEEP_WARM_FEATURES)");
  const uint64_t n = (c->n + stride - 1) / stride;
  if (M->count + n > M->max_samples) return set_error(PBF_ERR_CAPACITY, "sample store is full");
  int rc = check_hip(hipStreamSynchronize(M->stream), "sync");
  if (rc) return rc;
  if (n) {
    const uint32_t blocks = (uint32_t)((n + 255) / 256);
    hipLaunchKernelGGL(k_take_samples, dim3(blocks), dim3(256), 0, c->stream, n, stride, (const float*)c->feat,
                       (const float*)c->lsum, (const float*)c->lsuma, 1.0f / kWarmLambdaScale,
                       M->feat + M->count * kFeat,
                       M->tgt + M->count);
  }
  if ((rc = check_hip(hipStreamSynchronize(c->stream), "add_from_context"))) return rc;
  M->count += n;
  return PBF_OK;
}

uint64_t pbf_warm_model_sample_count(const pbf_warm_model* M) { return M ? M->count : 0; }

int pbf_warm_model_gradient(pbf_warm_model* M, uint64_t first, uint32_t count, float* grad, float* loss) {
  PBF_TRACE("pbf_warm_model_gradient");
  if (!M || !grad) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  if (count == 0 || first + count > M->count) return set_error(PBF_ERR_ARG, "sample range out of bounds");
  run_batch(M, M->iota + first, count, nullptr, nullptr);
  int rc = download(M, grad, M->grad, kNPar * 4);
  if (!rc && loss) rc = download(M, loss, M->loss, 4);
  return rc;
}

int pbf_warm_model_adam_step(pbf_warm_model* M, const float* grad, float learning_rate) {
  PBF_TRACE("pbf_warm_model_adam_step");
  if (!M || !grad) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  int rc = upload(M, M->grad, grad, kNPar * 4);
  if (rc) return rc;
  hipLaunchKernelGGL(k_mlp_adam, dim3((kNPar + 255) / 256), dim3(256), 0, M->stream, (const float*)M->grad,
                     next_adam(M, learning_rate), M->w1, M->w2, M->w2t);
  return check_hip(hipStreamSynchronize(M->stream), "adam");
}

int pbf_warm_model_train(pbf_warm_model* M, uint32_t epochs, uint32_t batch, float learning_rate, uint64_t seed,
                         float* mean_loss) {
  PBF_TRACE("pbf_warm_model_train");
  if (!M) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  if (M->count == 0) return set_error(PBF_ERR_STATE, "no samples");
  if (batch == 0) return set_error(PBF_ERR_ARG, "batch must be positive");
  std::mt19937_64 rng(seed);
  std::vector<uint32_t> perms[2];
  uint64_t batches = 0;
  launch_fill_u32((uint32_t*)M->loss_acc, 0u, 1, M->stream);
  for (uint32_t e = 0; e < epochs; ++e) {
    // (drawn while the last epoch's may still be read, unless it was staged)
    std::vector<uint32_t>& perm = perms[M->host.fits(M->count * 4) ? 0u : e & 1u];
    perm.resize(M->count);
    for (uint64_t i = 0; i < M->count; ++i) perm[i] = (uint32_t)i;
    std::shuffle(perm.begin(), perm.end(), rng);
    // the permutation buffer is rewritten only after the previous epoch's batches ran
    int rc = check_hip(hipStreamSynchronize(M->stream), "train");
    if (rc) return rc;
    if ((rc = upload(M, M->perm, perm.data(), M->count * 4))) return rc;
    for (uint64_t s = 0; s < M->count; s += batch) {
      const uint32_t cnt = (uint32_t)std::min<uint64_t>(batch, M->count - s);
      const AdamStep adam = next_adam(M, learning_rate);
      run_batch(M, M->perm + s, cnt, M->loss_acc, &adam);
      ++batches;
    }
  }
  float acc = 0.f;
  if (int rc = download(M, &acc, M->loss_acc, 4)) return rc;  // (waits for everything)
  if (mean_loss) *mean_loss = batches ? acc / (float)batches : 0.f;
  return PBF_OK;
}

int pbf_warm_model_predict(pbf_warm_model* M, const float* features, uint64_t count, float* out) {
  PBF_TRACE("pbf_warm_model_predict");
  if (!M || (count && (!features || !out))) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  if (!count) return PBF_OK;
  if (count >= (1ull << 32)) return set_error(PBF_ERR_ARG, "count out of range");
  float *f = M->part, *o = M->part + kPredictRows * kFeat, *own = nullptr;
  uint64_t most = kPredictRows;
  if (count > kPredictRows) {
    if (hipMallocAsync((void**)&own, count * (kFeat + 1) * 4, M->stream) == hipSuccess) {
      f = own, o = own + count * kFeat, most = count;
    } else {  // (no room: block by block)
      (void)hipGetLastError();
      own = nullptr;
    }
  }
  int rc = PBF_OK;
  for (uint64_t first = 0; !rc && first < count; first += most) {
    const uint64_t rows = std::min<uint64_t>(most, count - first);
    if ((rc = upload(M, f, features + first * kFeat, rows * kFeat * 4))) break;
    const uint32_t groups = (uint32_t)((rows + 15) / 16);
    hipLaunchKernelGGL(k_mlp_forward, dim3(std::min<uint32_t>(groups, 4096u)), dim3(64), 0, M->stream, (uint32_t)rows,
                       (const float*)f, model_weights(M), 1.0f, nullptr, o);
    rc = download(M, out + first, o, rows * 4);
  }
  if (own) (void)hipFreeAsync(own, M->stream);
  return rc;
}

int pbf_set_warm_gain(pbf_context* c, float gain) {
  if (!c) return set_error(PBF_ERR_ARG, "null context");
  if (!(gain >= 0.0f && gain <= 4.0f)) return set_error(PBF_ERR_ARG, "gain must be in [0, 4]");
  c->warm_gain = gain;
  return PBF_OK;
}

int pbf_set_warm_model(pbf_context* c, pbf_warm_model* M) {
  PBF_TRACE("pbf_set_warm_model");
  if (!c || !M) return set_error(PBF_ERR_ARG, "null argument");
  if (!M->has_params) return set_error(PBF_ERR_STATE, "model has no parameters");
  int rc = check_hip(hipStreamSynchronize(M->stream), "sync");
  if (rc) return rc;
  if ((rc = check_hip(hipMemcpyAsync(c->mp, M->p, kNPar * 4, hipMemcpyDeviceToDevice, c->stream), "copy")) ||
      (rc = check_hip(hipMemcpyAsync(c->mw1, M->w1, kHid * 16 * 2, hipMemcpyDeviceToDevice, c->stream), "copy")) ||
      (rc = check_hip(hipMemcpyAsync(c->mw2, M->w2, kHid * kHid * 2, hipMemcpyDeviceToDevice, c->stream), "copy")))
    return rc;
  c->has_model = true;
  return check_hip(hipStreamSynchronize(c->stream), "set_warm_model");
}

}  // extern "C"
