// wf_mlp.hip — online training of the return-map surrogate (wf_mlp.hpp):
// deterministic FP32 forward/backward over logged samples and Adam
// (Kingma & Ba 2015), plus the inference test hook and sample collection.
//
// Gradients are summed in a fixed order (within a wavefront's samples, over a
// block's wavefronts, over the blocks), so the same inputs always give
// bit-identical weights.
#include "wf_mlp.hpp"

namespace wf {

// one wavefront takes 32 samples at a time; four wavefronts a block
constexpr int kGradWaves = 4;
constexpr int kGradThreads = 64 * kGradWaves;
constexpr int kGradChunk = 32 * kGradWaves;

// the per-lane operands of the 64 lanes of a wavefront (one wavefront)
__global__ __launch_bounds__(64) void k_mlp_pack(const float* __restrict__ w,
                                                 uint4* __restrict__ pack) {
  MlpWave mw;
  mlp_wave_load(w, mw);
  MlpLanePack lp;
  lp.a1 = mw.a1;
#pragma unroll
  for (int kb = 0; kb < 4; kb++) lp.a2[kb] = mw.a2[kb];
  lp.b3 = mw.b3;
  lp.pad = 0.f;
#pragma unroll
  for (int r = 0; r < 16; r++) {
    lp.b2r[r] = mw.b2r[r];
    lp.w3r[r] = mw.w3r[r];
  }
  uint4 q[kMlpPackWords];
  __builtin_memcpy(q, &lp, sizeof(lp));
  const int l = lane_id();
#pragma unroll
  for (int k = 0; k < kMlpPackWords; k++) pack[64 * k + l] = q[k];
}

// MFMA inference on explicit rows (n x 4): the test hook of mlp_wave_eval,
// loading the weights as the stress kernel does
__global__ __launch_bounds__(256) void k_mlp_infer(const uint4* __restrict__ pack,
                                                   const float* __restrict__ X, int n,
                                                   float* __restrict__ y) {
  MlpWave mw;
  mlp_wave_load_packed(pack, mw);
  const int lane = lane_id();
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int nwaves = (gridDim.x * blockDim.x) >> 6;
  for (int base = wave * 64; base < n; base += nwaves * 64) {
    const int r = base + lane;
    const bool valid = r < n;
    const float f0 = valid ? X[4 * r] : 0.f, f1 = valid ? X[4 * r + 1] : 0.f;
    const float f2 = valid ? X[4 * r + 2] : 0.f, f3 = valid ? X[4 * r + 3] : 0.f;
    const float out = mlp_wave_eval(mw, f0, f1, f2, f3);
    if (valid) y[r] = out;
  }
}

// FP32 matrix products of the training pass: v_mfma_f32_32x32x2_f32 takes A
// (32 x 2) as A[l % 32][l / 32] of lane l, B (2 x 32) as B[l / 32][l % 32],
// and holds D (32 x 32) as the BF16 form does (wf_mlp.hpp): register r of
// lane l is row mlp_row(r, l / 32), column l % 32.  Operands and sums are
// FP32.  A layer's output register r is therefore the B operand of the K-step
// that takes rows mlp_row(r, 0) and mlp_row(r, 1).
__device__ __forceinline__ int mlp_row(int r, int half) {
  return 8 * (r >> 2) + 4 * half + (r & 3);
}
__device__ __forceinline__ f32x16_t mfma_f32(float a, float b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// Orders this wavefront's LDS writes before its following LDS reads.
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  __builtin_amdgcn_wave_barrier();
}

// Gradient of L = 1/n sum (y_s - t_s)^2 over samples s*stride, s < n, as one
// partial (kMlpParams sums and the loss) per block.
//
// The pass is a chain of small matrix products over a batch of samples, so a
// wavefront runs 32 samples through FP32 MFMA, transposed like the inference:
// layer 1 (3 MFMAs, the bias as a fifth input), layer 2 (16), the error back
// through W2 (16).  The weight gradients contract over the samples, which
// lie along the lanes, so the activations and errors are turned in LDS (33
// floats a row: no bank conflicts); dW2 is 16 more MFMAs into registers that
// stay there over all of the wavefront's samples, while the short rows (dW1,
// the biases, dW3) are FP32 FMAs that run beside them.  A wavefront's chain
// (51 MFMAs of 64 cycles, 1.4 us) sets the time: 16,384 samples give 512
// wavefronts, one a SIMD on half of the chip, and the kernel takes 7.3 us.
// One thread a sample, with its 2,500 dependent FMAs and a parameter a thread
// for the sums, took 21.7 us.
// Sums run in sample order within a wavefront's accumulators, then over the
// wavefronts and blocks in order: the same inputs give the same bits.
constexpr int kTile = 32 * 33;
struct GradWaveLds {
  float h1[kTile], d1[kTile], h2[kTile], d2[kTile];  // [unit][sample]
  float4 x[32];
  float dy[32];
};
__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(const float* __restrict__ w,
                                                           const float* __restrict__ X,
                                                           const float* __restrict__ Y, int n,
                                                           int stride, int per_block,
                                                           float* __restrict__ part,
                                                           float* __restrict__ loss_part) {
  __shared__ float sw2[kTile];  // W2[in][out], 33 floats a row
  __shared__ GradWaveLds sl[kGradWaves];
  const int tid = threadIdx.x, wv = tid >> 6, lane = lane_id();
  const int half = lane >> 5, c = lane & 31;
  for (int k = tid; k < 1024; k += kGradThreads) sw2[(k >> 5) * 33 + (k & 31)] = w[kMlpOffW2 + k];
  // layer 1, W1^T and the bias: K-steps {x0, x1}, {x2, x3}, {1, 0}
  const float a10 = w[kMlpOffW1 + half * 32 + c], a11 = w[kMlpOffW1 + (2 + half) * 32 + c];
  const float a12 = half ? 0.f : w[kMlpOffB1 + c];
  float b2r[16], w3r[16];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    b2r[r] = w[kMlpOffB2 + mlp_row(r, half)];
    w3r[r] = w[kMlpOffW3 + mlp_row(r, half)];
  }
  const float b3 = w[kMlpOffB3];
  const float inv_n = 1.0f / (float)n;
  __syncthreads();
  float a2[16], a2t[16];  // W2^T and W2 at this lane's row, K-step by K-step
#pragma unroll
  for (int r = 0; r < 16; r++) {
    a2[r] = sw2[mlp_row(r, half) * 33 + c];
    a2t[r] = sw2[c * 33 + mlp_row(r, half)];
  }
  GradWaveLds& L = sl[wv];
  f32x16_t gw2;  // dW2[mlp_row(r, half)][c]
#pragma unroll
  for (int r = 0; r < 16; r++) gw2[r] = 0.f;
  float gw1[4] = {0.f, 0.f, 0.f, 0.f}, gb1 = 0.f, gb2 = 0.f, gw3 = 0.f;  // of unit c
  float gb3 = 0.f, loss = 0.f;
  const int s0 = blockIdx.x * per_block, s1 = min(n, s0 + per_block);
  for (int c0 = s0 + 32 * wv; c0 < s1; c0 += kGradChunk) {
    const bool valid = c0 + c < s1;  // rows past the end: x = 0 and no error
    const int64_t s = (int64_t)(c0 + c) * stride;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    float t = 0.f;
    if (valid) {
      x = make_float4(X[4 * s], X[4 * s + 1], X[4 * s + 2], X[4 * s + 3]);
      t = Y[s];
    }
    f32x16_t h1, h2, d1;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      h1[r] = d1[r] = 0.f;
      h2[r] = b2r[r];
    }
    h1 = mfma_f32(a12, 1.f, h1);
    h1 = mfma_f32(a10, half ? x.y : x.x, h1);
    h1 = mfma_f32(a11, half ? x.w : x.z, h1);
#pragma unroll
    for (int r = 0; r < 16; r++) h1[r] = fmaxf(h1[r], 0.f);
#pragma unroll
    for (int r = 0; r < 16; r++) h2 = mfma_f32(a2[r], h1[r], h2);
    float y = 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      h2[r] = fmaxf(h2[r], 0.f);
      y += w3r[r] * h2[r];
    }
    y = y + __shfl_xor(y, 32) + b3;
    const float e = y - t;
    const float dy = valid ? 2.f * e * inv_n : 0.f;
    f32x16_t d2;
#pragma unroll
    for (int r = 0; r < 16; r++) d2[r] = h2[r] > 0.f ? dy * w3r[r] : 0.f;
#pragma unroll
    for (int r = 0; r < 16; r++) d1 = mfma_f32(a2t[r], d2[r], d1);
    if (valid && half == 0) {
      gb3 += dy;
      loss += e * e * inv_n;
    }
    wave_lds_order();  // the previous samples have been read
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int at = mlp_row(r, half) * 33 + c;
      L.h1[at] = h1[r];
      L.h2[at] = h2[r];
      L.d2[at] = d2[r];
      L.d1[at] = h1[r] > 0.f ? d1[r] : 0.f;
    }
    if (half == 0) {
      L.x[c] = x;
      L.dy[c] = dy;
    }
    wave_lds_order();
    // unit c over the samples 2 j + half
#pragma unroll
    for (int j = 0; j < 16; j++) {
      const int sj = 2 * j + half, at = c * 33 + sj;
      const float d2v = L.d2[at], d1v = L.d1[at];
      gw2 = mfma_f32(L.h1[at], d2v, gw2);
      const float4 xs = L.x[sj];
      gw1[0] += d1v * xs.x;
      gw1[1] += d1v * xs.y;
      gw1[2] += d1v * xs.z;
      gw1[3] += d1v * xs.w;
      gb1 += d1v;
      gb2 += d2v;
      gw3 += L.dy[sj] * L.h2[at];
    }
  }
  // the two halves' sums, then the wavefronts' in order
#pragma unroll
  for (int k = 0; k < 4; k++) gw1[k] += __shfl_xor(gw1[k], 32);
  gb1 += __shfl_xor(gb1, 32);
  gb2 += __shfl_xor(gb2, 32);
  gw3 += __shfl_xor(gw3, 32);
  for (int o = 16; o > 0; o >>= 1) {
    gb3 += __shfl_xor(gb3, o);
    loss += __shfl_xor(loss, o);
  }
  wave_lds_order();
  static_assert(sizeof(GradWaveLds) >= sizeof(float) * (kMlpParams + 1), "a partial fits");
  float* mine = reinterpret_cast<float*>(&L);
#pragma unroll
  for (int r = 0; r < 16; r++) mine[kMlpOffW2 + mlp_row(r, half) * 32 + c] = gw2[r];
  if (half == 0) {
#pragma unroll
    for (int k = 0; k < 4; k++) mine[kMlpOffW1 + k * 32 + c] = gw1[k];
    mine[kMlpOffB1 + c] = gb1;
    mine[kMlpOffB2 + c] = gb2;
    mine[kMlpOffW3 + c] = gw3;
    if (c == 0) {
      mine[kMlpOffB3] = gb3;
      mine[kMlpParams] = loss;
    }
  }
  __syncthreads();
  for (int k = tid; k <= kMlpParams; k += kGradThreads) {
    float a = 0.f;
#pragma unroll
    for (int u = 0; u < kGradWaves; u++) a += reinterpret_cast<const float*>(&sl[u])[k];
    if (k < kMlpParams) part[(int64_t)blockIdx.x * kMlpParams + k] = a;
    else loss_part[blockIdx.x] = a;
  }
}

// The block partials summed, and with ADAM the Adam update of the parameter
// (Kingma & Ba 2015, Algorithm 1: beta1 0.9, beta2 0.999, eps 1e-8) instead
// of the gradient written out.  A block takes 64 consecutive parameters, so
// that its loads are coalesced, and sixteen wavefronts share the partials
// (wavefront g takes g, g + 16, ...), whose sums are added in order: a fixed
// order.  Bound by latency, so all of a wavefront's loads are in flight
// together: 3.5 us at 128 partials.  A thread per parameter walking 256
// partials took 66 us, a wavefront per parameter, one line a partial, 5.2 us,
// and this split with its loads one after another 5.8 us.
constexpr int kReduceWaves = 16;
template <bool ADAM>
__global__ __launch_bounds__(64 * kReduceWaves) void k_mlp_reduce(
    const float* __restrict__ part, const float* __restrict__ loss_part, int nblocks,
    float* __restrict__ grad, float* __restrict__ w, float* __restrict__ m, float* __restrict__ v,
    int t, float lr, float* __restrict__ loss) {
  __shared__ float sh[kReduceWaves][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int pidx = blockIdx.x * 64 + lane;
  // the Adam state is read and the bias corrections formed while the
  // partials are on their way
  float wp = 0.f, mp = 0.f, vp = 0.f, c1 = 1.f, c2 = 1.f;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  if (ADAM && g == 0 && pidx < kMlpParams) {
    wp = w[pidx];
    mp = m[pidx];
    vp = v[pidx];
    c1 = 1.f - powf(b1, (float)t);
    c2 = 1.f - powf(b2, (float)t);
  }
  // every partial of this wavefront in flight at once (nblocks is at most
  // kMlpMaxBlocks; a partial past it adds zero)
  constexpr int kEach = kMlpMaxBlocks / kReduceWaves;
  const float* src = pidx < kMlpParams ? part + pidx : loss_part;
  const int ld = pidx < kMlpParams ? kMlpParams : 1;
  float q[kEach], a = 0.f;
#pragma unroll
  for (int u = 0; u < kEach; u++) {
    const int b = g + u * kReduceWaves;
    q[u] = b < nblocks ? src[b * ld] : 0.f;
  }
#pragma unroll
  for (int u = 0; u < kEach; u++) a += q[u];
  sh[g][lane] = a;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int u = 1; u < kReduceWaves; u++) a += sh[u][lane];
  if (pidx == kMlpParams) *loss = a;
  if (pidx >= kMlpParams) return;
  if constexpr (ADAM) {
    const float mn = b1 * mp + (1.f - b1) * a;
    const float vn = b2 * vp + (1.f - b2) * a * a;
    m[pidx] = mn;
    v[pidx] = vn;
    w[pidx] = wp - lr * (mn / c1) / (sqrtf(vn / c2) + eps);
  } else {
    grad[pidx] = a;
  }
}

// sample collection: flags, exclusive scan (caller), scatter
__global__ void k_mlp_flags(const int* __restrict__ mlstep, int n, int* __restrict__ flags) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) flags[i] = mlstep[i] >= 0 ? 1 : 0;
}
__global__ void k_mlp_scatter(Fields f, int n, const int* __restrict__ pos, float* __restrict__ X,
                              float* __restrict__ Y) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n || f.mlstep[i] < 0) return;
  const int s = pos[i];
  for (int k = 0; k < 4; k++) X[4 * (int64_t)s + k] = f.mlx[k][i];
  Y[s] = f.mly[i];
}

void launch_mlp_pack(hipStream_t s, const float* w, void* pack) {
  hipLaunchKernelGGL(k_mlp_pack, dim3(1), dim3(64), 0, s, w, (uint4*)pack);
}

void launch_mlp_infer(hipStream_t s, const void* pack, const float* X, int n, float* y) {
  if (n <= 0) return;
  const int blocks = std::min(1024, (n + 255) / 256);
  hipLaunchKernelGGL(k_mlp_infer, dim3(blocks), dim3(256), 0, s, (const uint4*)pack, X, n, y);
}

// samples per block: whole chunks, so that only the last block has a rest
static int mlp_per_block(int n, int nblocks) {
  const int chunks = (n + kGradChunk - 1) / kGradChunk;
  return (chunks + nblocks - 1) / nblocks * kGradChunk;
}
static void launch_mlp_parts(hipStream_t s, const float* w, const float* X, const float* Y, int n,
                             int stride, float* part, float* loss_part, int nblocks) {
  hipLaunchKernelGGL(k_mlp_grad, dim3(nblocks), dim3(kGradThreads), 0, s, w, X, Y, n, stride,
                     mlp_per_block(n, nblocks), part, loss_part);
}
constexpr int kReduceBlocks = (kMlpParams + 1 + 63) / 64;  // the loss after the parameters

void launch_mlp_grad(hipStream_t s, const float* w, const float* X, const float* Y, int n,
                     int stride, float* part, float* loss_part, int nblocks, float* grad,
                     float* loss) {
  launch_mlp_parts(s, w, X, Y, n, stride, part, loss_part, nblocks);
  hipLaunchKernelGGL(k_mlp_reduce<false>, dim3(kReduceBlocks), dim3(64 * kReduceWaves), 0, s, part,
                     loss_part, nblocks, grad, (float*)nullptr, (float*)nullptr, (float*)nullptr, 0,
                     0.f, loss);
}

void launch_mlp_train_iter(hipStream_t s, float* w, float* m, float* v, const float* X,
                           const float* Y, int n, int stride, float* part, float* loss_part,
                           int nblocks, int t, float lr, float* loss) {
  launch_mlp_parts(s, w, X, Y, n, stride, part, loss_part, nblocks);
  hipLaunchKernelGGL(k_mlp_reduce<true>, dim3(kReduceBlocks), dim3(64 * kReduceWaves), 0, s, part,
                     loss_part, nblocks, (float*)nullptr, w, m, v, t, lr, loss);
}
int mlp_grad_blocks(int n) {
  return std::max(1, std::min(kMlpMaxBlocks, (n + kGradChunk - 1) / kGradChunk));
}


void launch_mlp_collect(hipStream_t s, const Fields& f, int n, float* X, float* Y, int* flags,
                        int* scan, int* scan_part, int* count) {
  const int g = (n + 255) / 256;
  hipLaunchKernelGGL(k_mlp_flags, dim3(g), dim3(256), 0, s, f.mlstep, n, flags);
  launch_scan_exclusive(s, flags, n, scan_part, scan);
  hipLaunchKernelGGL(k_mlp_scatter, dim3(g), dim3(256), 0, s, f, n, scan, X, Y);
  hipMemcpyAsync(count, scan + n, sizeof(int), hipMemcpyDeviceToDevice, s);
}

}  // namespace wf
