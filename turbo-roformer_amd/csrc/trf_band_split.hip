// Band split of BS-RoFormer on gfx950: per band f, the RMSNorm of the frame's din_f spectral features and
// a Linear din_f -> 256 (BandSplit, model.py:147-155; called at fast.py:377-380), written straight into the
// stack's token order.
//
// Arithmetic: fp32 throughout, on v_mfma_f32_32x32x2_f32 (fp32 products and sums, as the reference's fp32
// Linear).  The norm is linear in the output, so the kernel computes W' . x on the raw features, with
// W' = W * gamma * sqrt(din) folded at packing, and scales the accumulators by 1 / max(|x|, 1e-12).
//
// Shape: C^T = W' . x^T: MFMA rows are the 256 output features (8 tiles of 32, one per wave), columns are 32
// frames of one band, whose features the workgroup holds in LDS.  Four MFMAs share each 16-byte read of
// both operands: MFMA i of k-group q takes inputs 8q + 4hh + i of a lane (which inputs meet in an MFMA does
// not matter, as long as both operands agree), so a lane reads 4 consecutive features of its frame and 4
// consecutive packed weights, the weights from L2 two groups ahead.  A width that is 4 more than a multiple
// of 8 ends with a group of 4 inputs, two MFMAs.  The outputs leave through LDS as whole 1 KB rows.
// The workgroups of the widest bands go first.
// 17 s chunk (1701 frames, 62 bands of width 8 to 516; 136 MB, 27 us at the rate of a copy, 26 us of MFMA
// work at 2.1 GHz): 59 us a launch, of 86 for 4-wave workgroups that read frames and weights from global memory
// as they multiplied (the frames as 16 bytes of 32 rows) and stored 16 bytes a lane.
#include "trf_tiles.h"

namespace trf {

__device__ __forceinline__ f32x16 mfma32f(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

constexpr int kBandAhead = 2;      // k-groups the weights are loaded ahead
constexpr int kBandChunks = 32;    // feature chunks (4 inputs) of a frame held in LDS at a time
constexpr int kBandRow = kBandChunks + 1;  // the odd row length spreads a chunk of 16 frames over the banks

__global__ __launch_bounds__(64 * kTileWaves, 4) void k_band_split(const float* __restrict__ feats,
                                                                   const float* __restrict__ packed,
                                                                   float* __restrict__ X, const BandPlan p) {
  // the frames' features; at the end the 32 output rows (1 KB each)
  __shared__ u32x4 smem[kBandFrames * 64 + kBandFrames / 4];
  static_assert(kBandFrames == 32 && kBandFrames * kBandRow <= kBandFrames * 64, "features fit");
  float* const inv = reinterpret_cast<float*>(smem + kBandFrames * 64);
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5;
  const int band = p.order[blockIdx.x / p.ngroups];
  const int group = blockIdx.x - (blockIdx.x / p.ngroups) * p.ngroups;
  const int din = p.din[band], chunks = din >> 2, groups = din >> 3;
  const float* const W = packed + p.wofs[band];  // [groups][8 tiles][64 lanes][4], a tail of [8][64][2], bias [256]
  const int n0 = group * kBandFrames;
  const f32x4* const wq = reinterpret_cast<const f32x4*>(W) + wave * 64 + lane;
  f32x4 a[kBandAhead];
#pragma unroll
  for (int i = 0; i < kBandAhead; ++i)
    if (i < groups) a[i] = wq[i * 512];
  // Thread -> frame t and every 16th chunk of it: its share of the frame's squares.  Frames past the last
  // one repeat it (a column of the MFMAs of their own) and store nothing.
  const int t = threadIdx.x >> 4, c0 = threadIdx.x & 15;
  const float* const xr = feats + int64_t(min(n0 + t, p.n_frames - 1)) * p.width + p.col[band];
  float ss = 0.f;
  f32x16 acc = zero16();
#pragma unroll 1
  for (int part = 0; part < chunks; part += kBandChunks) {
    f32x4 x[kBandChunks / 16];
#pragma unroll
    for (int i = 0; i < kBandChunks / 16; ++i) {
      const int c = part + c0 + 16 * i;
      x[i] = c < chunks ? *reinterpret_cast<const f32x4*>(xr + 4 * c) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int e = 0; e < 4; ++e) ss = fmaf(x[i][e], x[i][e], ss);
    }
    if (part) lds_barrier();  // every wave has read the previous part
#pragma unroll
    for (int i = 0; i < kBandChunks / 16; ++i)
      smem[t * kBandRow + c0 + 16 * i] = __builtin_bit_cast(u32x4, x[i]);
    lds_barrier();
    const int g1 = min(groups, (part + kBandChunks) / 2);
#pragma unroll 1
    for (int g = part / 2; g < g1; g += kBandAhead) {
#pragma unroll
      for (int i = 0; i < kBandAhead; ++i) {
        if (g + i >= g1) break;
        const f32x4 b = __builtin_bit_cast(f32x4, smem[j * kBandRow + 2 * (g + i) - part + hh]);
        const f32x4 w = a[i];
        if (g + i + kBandAhead < groups) a[i] = wq[int64_t(g + i + kBandAhead) * 512];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = mfma32f(w[e], b[e], acc);
      }
    }
  }
  if (chunks & 1) {  // the last 4 inputs: 2hh + {0, 1}
    const float2 w = reinterpret_cast<const float2*>(W + int64_t(groups) * 2048)[wave * 64 + lane];
    const float2 b = reinterpret_cast<const float2*>(smem + j * kBandRow + (chunks - 1) % kBandChunks)[hh];
    acc = mfma32f(w.x, b.x, acc);
    acc = mfma32f(w.y, b.y, acc);
  }
#pragma unroll
  for (int m = 8; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
  if (c0 == 0) inv[t] = 1.0f / fmaxf(sqrtf(ss), 1e-12f);
  lds_barrier();  // the norms are there, every wave has read the features
  const float* const bias = W + int64_t(din) * 256;
  const float s = inv[j];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int o = 32 * wave + row_of_group(g, hh);
    const f32x4 b = *reinterpret_cast<const f32x4*>(bias + o);
    f32x4 v;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = fmaf(acc[4 * g + r], s, b[r]);
    smem[row_chunk(j, o >> 2)] = __builtin_bit_cast(u32x4, v);
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < kBandFrames / kTileWaves; ++i) {
    const int r = kBandFrames / kTileWaves * wave + i;
    if (n0 + r < p.n_frames)
      *reinterpret_cast<u32x4*>(X + (int64_t(n0 + r) * p.n_bands + band) * kDim + 4 * lane) = smem[row_chunk(r, lane)];
  }
}

// Packing of one band: W'[o][k] = w[o][k] * (gamma[k] * sqrt(din)) as A operands of v_mfma_f32_32x32x2_f32:
// dst[((q * 8 + t) * 64 + lane) * 4 + i] = W'[32t + lane%32][8q + 4(lane/32) + i], for the last 4 inputs of
// a width that is not a multiple of 8 dst[...][(t * 64 + lane) * 2 + i] = W'[32t + lane%32][din - 4 +
// 2(lane/32) + i], then the bias [256].
__global__ void k_pack_band_split(const float* __restrict__ w, const float* __restrict__ b,
                                  const float* __restrict__ gamma, int din, float sqrt_din, float* __restrict__ dst) {
  const int n_items = din * 256, full = (din & ~7) * 256;
  for (int it = blockIdx.x * blockDim.x + threadIdx.x; it < n_items + kDim; it += gridDim.x * blockDim.x) {
    if (it >= n_items) {
      dst[it] = b[it - n_items];
      continue;
    }
    const int per = it < full ? 4 : 2, u = it < full ? it : it - full;
    const int i = u % per, lane = u / per & 63, t = u / (per * 64) & 7, q = u / (per * 512);
    const int o = 32 * t + (lane & 31), k = (it < full ? 8 * q : din - 4) + per * (lane >> 5) + i;
    dst[it] = w[int64_t(o) * din + k] * (gamma[k] * sqrt_din);
  }
}

void launch_pack_band_split(const float* w, const float* b, const float* gamma, int din, float sqrt_din, float* dst,
                            hipStream_t st) {
  const int n = (din / 2) * 8 * 64 + kDim;
  hipLaunchKernelGGL(k_pack_band_split, dim3((n + 255) / 256), dim3(256), 0, st, w, b, gamma, din, sqrt_din, dst);
}

void launch_band_split(const float* feats, const float* packed, float* X, const BandPlan& plan, hipStream_t st) {
  hipLaunchKernelGGL(k_band_split, dim3(unsigned(plan.n_bands) * unsigned(plan.ngroups)), dim3(64 * kTileWaves), 0,
                     st, feats, packed, X, plan);
}

}  // namespace trf
