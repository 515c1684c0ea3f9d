// HIP kernels of the BS-RoFormer transformer stack for gfx950 (MI355X).
//
// All matrix products run on v_mfma_f32_32x32x16_bf16 (bf16 operands, fp32 accumulation).
// The kernels compute C^T = W . A^T, i.e. the 32 MFMA rows are output features and the 32
// MFMA columns are tokens.  With the 32x32 accumulator layout
//     lane l, register r  ->  row 8*(r/4) + 4*(l/32) + (r%4), column l%32
// every lane owns one token and runs of 4 consecutive features, so interleaved rotary pairs
// (2p, 2p+1), row norms and residual updates need no cross-lane exchange beyond one swap of
// the two half-waves.
//
// Numerics follow the reference kernels (src/turbo_roformer/csrc/kernels.cpp): fp32
// accumulators, fp32 residual stream, fp32 rotary/softmax/gate math, bf16 round-to-nearest-even
// for every GEMM/attention operand (kernels.cpp:30-33).
#include "trf_tiles.h"

#include <atomic>

#include <type_traits>

namespace trf {

// ============================================================ weight packing
// dst[t][ks][lane][e] = W[32t + lane%32][16ks + kperm(lane/32, e)] (kperm: natural 8hh + e, or register order
// 4hh + e / 8 + 4hh + e - 4).  Rows past `rows` are zero, and so is everything when W is null.  (See
// trf_internal.h.)
__global__ void k_pack(const uint16_t* __restrict__ W, int rows, int K, int layout, u32x4* __restrict__ dst) {
  const int ksteps = K / 16;
  const int64_t total = int64_t((rows + 31) / 32) * ksteps * 64;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int lane = int(i % 64);
  const int ks = int((i / 64) % ksteps);
  const int t = int(i / (64 * ksteps));
  const int row = 32 * t + (lane & 31), hh = lane >> 5;
  u32x4 v = zero4();
  if (W && row < rows) {
    const uint16_t* src = W + int64_t(row) * K + 16 * ks;
    if (layout == kPack32Natural) {
      v = *reinterpret_cast<const u32x4*>(src + 8 * hh);
    } else {
      const u32x2 lo = *reinterpret_cast<const u32x2*>(src + 4 * hh);
      const u32x2 hi = *reinterpret_cast<const u32x2*>(src + 8 + 4 * hh);
      v = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
  }
  dst[i] = v;
}

void launch_pack(const uint16_t* W, int rows, int K, int layout, uint8_t* dst, hipStream_t st) {
  const int64_t total = int64_t((rows + 31) / 32) * (K / 16) * 64;
  hipLaunchKernelGGL(k_pack, dim3(unsigned((total + 255) / 256)), dim3(256), 0, st, W, rows, K, layout,
                     reinterpret_cast<u32x4*>(dst));
}

// fp16 operand tiles, 32x32 register order, from hi + lo bf16 parts of the fp32 weights (lo optional):
// dst = fp16(hi + lo), round to nearest even.
__global__ void k_pack_f16(const uint16_t* __restrict__ hi, const uint16_t* __restrict__ lo, int rows, int K,
                           u32x4* __restrict__ dst) {
  const int ksteps = K / 16;
  const int64_t total = int64_t((rows + 31) / 32) * ksteps * 64;
  const int64_t i = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int lane = int(i % 64);
  const int ks = int((i / 64) % ksteps);
  const int t = int(i / (64 * ksteps));
  const int row = 32 * t + (lane & 31), hh = lane >> 5;
  u32x4 v = zero4();
  if (row < rows) {
    float f[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int k = 16 * ks + (e < 4 ? 4 * hh + e : 8 + 4 * hh + (e - 4));  // register order
      const int64_t idx = int64_t(row) * K + k;
      f[e] = bf16_to_f32(hi[idx]) + (lo ? bf16_to_f32(lo[idx]) : 0.0f);
    }
    v = u32x4{pk_f16(f[0], f[1]), pk_f16(f[2], f[3]), pk_f16(f[4], f[5]), pk_f16(f[6], f[7])};
  }
  dst[i] = v;
}

void launch_pack_f16(const uint16_t* hi, const uint16_t* lo, int rows, int K, uint8_t* dst, hipStream_t st) {
  const int64_t total = int64_t((rows + 31) / 32) * (K / 16) * 64;
  hipLaunchKernelGGL(k_pack_f16, dim3(unsigned((total + 255) / 256)), dim3(256), 0, st, hi, lo, rows, K,
                     reinterpret_cast<u32x4*>(dst));
}

__global__ void k_copy_f32(const float* __restrict__ src, int n, float* __restrict__ dst) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

void launch_copy_f32(const float* src, int n, float* dst, hipStream_t st) {
  hipLaunchKernelGGL(k_copy_f32, dim3((n + 255) / 256), dim3(256), 0, st, src, n, dst);
}

// ============================================================ add + L2 row norm
// One wave per row of 256: lane l holds columns 4l..4l+3.  (kernels.cpp:101-137)
__global__ __launch_bounds__(256) void k_add_rmsnorm(float* __restrict__ X, const void* __restrict__ Y,
                                                     int y_bf16, void* __restrict__ out, int out_bf16,
                                                     int64_t n, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = int64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (row >= n) return;
  float* xr = X + row * kDim + 4 * lane;
  f32x4 v = *reinterpret_cast<const f32x4*>(xr);
  if (Y) {
    if (y_bf16) {
      const u32x2 y = *reinterpret_cast<const u32x2*>(static_cast<const uint16_t*>(Y) + row * kDim + 4 * lane);
      v[0] += __uint_as_float(y[0] << 16);
      v[1] += __uint_as_float(y[0] & 0xFFFF0000u);
      v[2] += __uint_as_float(y[1] << 16);
      v[3] += __uint_as_float(y[1] & 0xFFFF0000u);
    } else {
      const f32x4 y = *reinterpret_cast<const f32x4*>(static_cast<const float*>(Y) + row * kDim + 4 * lane);
      v += y;
    }
    *reinterpret_cast<f32x4*>(xr) = v;
  }
  float ss = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m);
  const float inv = 1.0f / fmaxf(sqrtf(ss), eps);
  if (out_bf16) {
    u32x2 o = {pk_bf16(v[0] * inv, v[1] * inv), pk_bf16(v[2] * inv, v[3] * inv)};
    *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(out) + row * kDim + 4 * lane) = o;
  } else {
    *reinterpret_cast<f32x4*>(static_cast<float*>(out) + row * kDim + 4 * lane) = v * inv;
  }
}

void launch_add_rmsnorm(float* X, const void* Y, int y_bf16, void* out, int out_bf16, int64_t n, float eps,
                        hipStream_t st) {
  hipLaunchKernelGGL(k_add_rmsnorm, dim3(unsigned((n + 3) / 4)), dim3(256), 0, st, X, Y, y_bf16, out, out_bf16,
                     n, eps);
}

// ============================================================ fused QKV + gate GEMM, rotary epilogue
// A workgroup is 32 C consecutive padded positions of one sequence; wave h computes head h: its q, k and v
// weight tiles (two 32-row tiles each) one after the other, from L2 into registers, against the xn rows in
// LDS (see trf_tiles.h).  The accumulators of a tile leave at once:
//   q, k: rotated in fp32 (cos / sin rows of the tile's positions in LDS), packed; the half-waves trade
//     register groups so that a lane stores a whole 16-byte chunk (8 features) of its position and an
//     instruction writes two runs of 512 bytes (chunk-major rows, see token-order contract in trf_hip.h);
//   v: the operands of the product are swapped, so a lane holds one feature of 4 consecutive positions per
//     register group; V^T rows go through the wave's own 8 KB of LDS and leave as whole lines.
// The gate tile's 16 k-steps are split over the waves (two each) and summed through LDS.
// Bounded by the writes: 324 MB of Q, K, V^T at 105,462 tokens (68 us at the rate of 8-byte store streams).
// Workgroups of 256 rows that streamed the weights through LDS in 13 barrier-separated stages and stored
// 8 bytes a lane took 22.6 us at 101 frames x 62 bands (31 workgroups' rows on 256 CUs), 49 at 487 frames and
// 134 at 1701; these take 15, 34 and 129.  What is left at 1701 is the L2's: a tile's weights pass once per 64
// positions (the CUs' address units are 70% busy, waiting on it half of that time).  Staging the xn rows costs 4-way
// bank conflicts, 8% of the cycles.
// (kernels.cpp:439-540)
template <int C>
__global__ __launch_bounds__(64 * kTileWaves, 4) void k_qkv_rope(
    const uint16_t* __restrict__ xn, const uint8_t* __restrict__ layer, const float* __restrict__ rope, int mode,
    int L, int Lpad, int T, int F, uint16_t* __restrict__ Q, uint16_t* __restrict__ K, uint16_t* __restrict__ Vt,
    float* __restrict__ G) {
  constexpr int R = 32 * C;
  constexpr int kRope = R * 32, kGate = kRope + R * kRopeChunks;
  __shared__ u32x4 smem[kGate + kTileWaves * R * kHeads / 4];  // xn blocks, cos | sin rows, partial gates; then V^T
  static_assert(kGate + kTileWaves * R * kHeads / 4 >= kTileWaves * kHeadDim * R / 8, "V^T of the tile fits");
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5, h = wave;
  // From the last sequence to the first: beyond ~250 MB of Q, K and V^T the memory-side cache holds what was
  // written last, and the attention kernel starts at the first sequence (1701 frames x 62 bands: attention 375-378 us
  // after an ascending order, 360-369 after this one).
  const int nblk = Lpad / R, blk = int(gridDim.x - 1 - blockIdx.x), s = blk / nblk, p0 = (blk - s * nblk) * R;
  const TileWeights w{buffer_rsrc(layer, int(kLayerBytes)), lane * 16};
  auto tile = [&](int kind, int half) __attribute__((always_inline)) {  // kind 0 q, 1 k, 2 v
    return TileOff{{int(kOffQkvg) + (16 * kind + 2 * h + half) * 16 * kTileBytes, 0}};
  };
  u32x4 a[kWeightAhead][2], ag[2];
#pragma unroll
  for (int i = 0; i < kWeightAhead; ++i) a[i][0] = w.load(tile(0, 0).v[0] + i * kTileBytes);
#pragma unroll
  for (int i = 0; i < 2; ++i) ag[i] = w.load(int(kOffQkvg) + ((kQkvgTiles - 1) * 16 + 2 * wave + i) * kTileBytes);
  TilePositions<C> x;
  x.load(xn, mode, s, p0, L, T, F);
  stage_rope<C>(rope, p0, L, smem + kRope);
  x.put(smem);
  lds_barrier();
  gate_partials<C>(ag, smem, reinterpret_cast<float*>(smem + kGate), wave, lane);
  lds_barrier();
  {  // thread -> (position, head): 8 lanes write a token's 8 gates
    const int p = threadIdx.x >> 3, head = threadIdx.x & 7;
    if (p < R && p0 + p < L)
      G[token_of(mode, s, p0 + p, T, F) * kHeads + head] = gate_of<C>(
          reinterpret_cast<const float*>(smem + kGate), p, head,
          reinterpret_cast<const float*>(layer + kOffBgate));
  }
  auto xop = [&](int k, int, int ct) __attribute__((always_inline)) { return smem[(ct * 16 + k) * 64 + lane]; };
  auto none = [](int) __attribute__((always_inline)) {};
  const int64_t head0 = (int64_t(s) * kHeads + h) * kHeadDim * Lpad;  // first element of this (sequence, head)
#pragma unroll
  for (int kind = 0; kind < 2; ++kind) {
    const auto res = buffer_rsrc((kind ? K : Q) + head0, kHeadDim * Lpad * 2);
    const float sc = kind ? 1.0f : kLog2e;  // q leaves in units of log2(e): scores are base-2 exponents
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      f32x16 acc[C];
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = zero16();
      tile_gemm<16, C, kFfBf16, 1>(w, tile(kind, half).v, (half ? tile(kind + 1, 0) : tile(kind, 1)).v, a, acc, xop, none);
#pragma unroll
      for (int ct = 0; ct < C; ++ct) {
        const bool valid = p0 + 32 * ct + j < L;
        u32x2 o[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          o[g] = rotate_group(acc[ct], g, smem + kRope, 32 * ct + j, half, hh, sc);
          if (!valid) o[g] = u32x2{0u, 0u};
        }
#pragma unroll
        for (int q = 0; q < 2; ++q)
          __builtin_amdgcn_raw_buffer_store_b128(join_halves(o[2 * q], o[2 * q + 1]), res,
                                                 ((4 * half + 2 * q + hh) * Lpad + p0 + 32 * ct + j) * 16, 0, 0);
      }
    }
  }
  u32x2 vp[2][C][4];  // V^T: feature 32 half + j, positions 32 ct + 8g + 4hh + r
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    f32x16 acc[C];
#pragma unroll
    for (int ct = 0; ct < C; ++ct) acc[ct] = zero16();
    tile_gemm<16, C, kFfBf16, 1, true>(w, tile(2, half).v, tile(2, 1).v, a, acc, xop, none);
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = p0 + 32 * ct + row_of_group(g, hh) + r < L ? acc[ct][4 * g + r] : 0.f;
        vp[half][ct][g] = u32x2{pk_bf16(v[0], v[1]), pk_bf16(v[2], v[3])};
      }
  }
  lds_barrier();  // every wave has read the xn blocks and cos / sin rows
  constexpr int CH = 4 * C, RI = 64 / CH;  // 16-byte chunks of a V^T row, rows of one store instruction
  u32x4* const vs = smem + wave * (kHeadDim * CH);
#pragma unroll
  for (int half = 0; half < 2; ++half)
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * half + j;
        reinterpret_cast<u32x2*>(vs)[2 * (d * CH + ((4 * ct + g) ^ (d & (CH - 1)))) + hh] = vp[half][ct][g];
      }
  const auto vres = buffer_rsrc(Vt + head0, kHeadDim * Lpad * 2);
#pragma unroll
  for (int i = 0; i < kHeadDim / RI; ++i) {
    const int d = RI * i + lane / CH, c = lane & (CH - 1);
    __builtin_amdgcn_raw_buffer_store_b128(vs[d * CH + (c ^ (d & (CH - 1)))], vres, (d * Lpad + p0) * 2 + c * 16, 0, 0);
  }
}

int device_cu_count() {
  static std::atomic<int> cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n <= 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Token tiles of a launch over n rows: 32 rows while such tiles fit one per CU, 64 beyond.
static int token_tiles(int64_t n) { return n <= int64_t(32) * device_cu_count() ? 1 : 2; }

void launch_qkv(const uint16_t* xn, const uint8_t* layer, const float* rope, const SeqShape& sh, uint16_t* Q,
                uint16_t* K, uint16_t* Vt, float* G, hipStream_t st, const LaunchEvents& ev) {
  const int64_t rows = int64_t(sh.nseq) * sh.Lpad;
  if (rows <= 0) return;
  const int C = token_tiles(rows);
  const auto kernel = C == 1 ? k_qkv_rope<1> : k_qkv_rope<2>;
  hipExtLaunchKernelGGL(kernel, dim3(unsigned(rows / (32 * C))), dim3(64 * kTileWaves), 0, st, ev.start, ev.stop, 0,
                        xn, layer, rope, sh.mode, sh.L, sh.Lpad, sh.T, sh.F, Q, K, Vt, G);
}


// ============================================================ attention
// S^T = K . Q^T puts keys on MFMA rows and queries on columns.  Key rows are loaded in the
// order pi(i) (bits 2 and 3 of i swapped) so that register r of half-wave hh holds key
//     key_of(r, hh) = (r < 8 ? 8*hh + r : 16 + 8*hh + (r - 8))
// of its 32-key block: registers 0..7 / 8..15 are then exactly the 8 consecutive keys that
// lane supplies as the B operand (P^T) of the two 16-key PV instructions O^T += V^T . P^T.
__device__ __forceinline__ int key_perm(int i) { return (i & ~12) | ((i & 4) << 1) | ((i & 8) >> 1); }
__device__ __forceinline__ int key_of(int r, int hh) { return r < 8 ? 8 * hh + r : 8 + 8 * hh + r; }

// Exact softmax of one 32-query x 32-key score block held as S^T registers.
// Returns the unnormalised bf16 probabilities as two B operands and adds the fp32 sum.
// Scores are in units of log2(e) (q is pre-scaled), so e = 2^(s - m); with shift = 0 the caller has
// already subtracted the row max inside the MFMA accumulator.
__device__ __forceinline__ void softmax_block(const f32x16& sacc, int key0, int L, int hh, float shift, float& lsum,
                                              u32x4& p0, u32x4& p1) {
  float e[16];
  if (key0 + 32 <= L) {
#pragma unroll
    for (int r = 0; r < 16; ++r) e[r] = __builtin_amdgcn_exp2f(sacc[r] - shift);
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      e[r] = (key0 + key_of(r, hh) < L) ? __builtin_amdgcn_exp2f(sacc[r] - shift) : 0.f;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) lsum += e[r];
  p0[0] = pk_bf16(e[0], e[1]);
  p0[1] = pk_bf16(e[2], e[3]);
  p0[2] = pk_bf16(e[4], e[5]);
  p0[3] = pk_bf16(e[6], e[7]);
  p1[0] = pk_bf16(e[8], e[9]);
  p1[1] = pk_bf16(e[10], e[11]);
  p1[2] = pk_bf16(e[12], e[13]);
  p1[3] = pk_bf16(e[14], e[15]);
}

// The same probabilities for the single-sweep kernel, whose normaliser is the sum of the bf16-rounded P
// (the weights P.V actually applies), formed on the matrix pipe instead of by 16 VALU adds per block:
// v_mfma_f32_16x16x32_bf16 with A = `ones` and B = the P^T operand.  B lane l is column n = l % 16 and
// k-group l / 16; the P^T registers of lane l belong to query l % 32 = n + 16 ((l / 16) & 1), half
// (l / 32) of the keys.  A row 0 is 1 on k-groups 0 and 2 and row 1 on k-groups 1 and 3, so D row 0,
// column n (lane n, register 0) collects query n's 16 keys and row 1 (lane n, register 1) query n + 16's;
// the other rows stay 0.
__device__ __forceinline__ u32x4 rowsum_ones(int lane) {
  const int m = lane & 15, g = (lane >> 4) & 1;
  const uint32_t one = (m == 0 && g == 0) || (m == 1 && g == 1) ? 0x3f803f80u : 0u;
  return u32x4{one, one, one, one};
}

__device__ __forceinline__ f32x4 mfma16_rowsum(u32x4 ones, u32x4 p, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones), __builtin_bit_cast(bf16x8, p), c,
                                                 0, 0, 0);
}

__device__ __forceinline__ void softmax_block_psum(const f32x16& sacc, int key0, int L, int hh, const u32x4& ones,
                                                   f32x4& psum, u32x4& p0, u32x4& p1) {
  float e[16];
  if (key0 + 32 <= L) {
#pragma unroll
    for (int r = 0; r < 16; ++r) e[r] = __builtin_amdgcn_exp2f(sacc[r]);
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) e[r] = (key0 + key_of(r, hh) < L) ? __builtin_amdgcn_exp2f(sacc[r]) : 0.f;
  }
  p0 = u32x4{pk_bf16(e[0], e[1]), pk_bf16(e[2], e[3]), pk_bf16(e[4], e[5]), pk_bf16(e[6], e[7])};
  p1 = u32x4{pk_bf16(e[8], e[9]), pk_bf16(e[10], e[11]), pk_bf16(e[12], e[13]), pk_bf16(e[14], e[15])};
  psum = mfma16_rowsum(ones, p0, psum);
  psum = mfma16_rowsum(ones, p1, psum);
}

// Query j's sum from the row-sum accumulator (j = lane % 32; both half-waves get it).
__device__ __forceinline__ float psum_of_query(const f32x4& psum, int j) {
  const float a = __shfl(psum[0], j & 15), b = __shfl(psum[1], j & 15);
  return j < 16 ? a : b;
}

__device__ __forceinline__ float block_max(const f32x16& sacc, int key0, int L, int hh, float m) {
  if (key0 + 32 <= L) {
#pragma unroll
    for (int r = 0; r < 16; r += 2) m = fmaxf(fmaxf(m, sacc[r]), sacc[r + 1]);  // one v_max3_f32 per pair
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (key0 + key_of(r, hh) < L) m = fmaxf(m, sacc[r]);
  }
  return m;
}

// Epilogue: O[tok][h*64 + d] = bf16(acc * gate / sum), 4 consecutive features per store.
__device__ __forceinline__ void attn_store(const f32x16 (&o)[2], int q, int L, int s, int h, int hh, int mode, int T,
                                           int F, const float* __restrict__ G, float lsum,
                                           uint16_t* __restrict__ O) {
  if (q >= L) return;
  const int64_t tok = token_of(mode, s, q, T, F);
  const float sc = G[tok * kHeads + h] * (1.0f / lsum);
  uint16_t* dst = O + tok * (kHeads * kHeadDim) + h * kHeadDim;
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = 32 * dt + row_of_group(g, hh);
      u32x2 v = {pk_bf16(o[dt][4 * g] * sc, o[dt][4 * g + 1] * sc),
                 pk_bf16(o[dt][4 * g + 2] * sc, o[dt][4 * g + 3] * sc)};
      *reinterpret_cast<u32x2*>(dst + d0) = v;
    }
}

// Long sequences (time attention, L up to a few thousand).  The reference's exact, non-online softmax
// (kernels.cpp:286-384) first finds the row max m, then forms e = 2^(s - m) (q carries the factor
// log2(e), so scores are base-2 exponents), sums e in fp32, rounds P = e to bf16 unnormalised and
// accumulates P.V; the epilogue scales by gate/sum.  Here one sweep over the keys does the same with an
// integer shift c in place of m, fixed from the first 32 keys (see kAttHeadroomFast): a power-of-two
// shift changes neither the bf16 rounding of P nor the normalised result, QK^T is computed once instead of
// twice, and no max is taken after the first keys; a workgroup whose sums overflow redoes the sweep with
// a shift raised as scores exceed it.
// The normaliser is the fp32 sum of the rounded P (on the matrix pipe, softmax_block_psum) rather than
// of e.  With the row max the dominant key's P is exactly 1 and escapes bf16 rounding; with an integer
// shift it is rounded like the others, and dividing by the sum of the weights P.V actually applied makes
// up for that: against exact attention the result is within ~0.5 dB of the reference's arithmetic on
// peaked rows, where the sum of e leaves it 2-3 dB below.
// One workgroup = one (sequence, head) and 4 waves x 32 QT queries; with QT = 2 a wave holds two 32-query
// column tiles, so every K or V^T operand read from LDS feeds two MFMAs (QT = 1: see launch_attention).  Tiles of 64 keys of K and V^T stream
// through a ring of LDS buffers, loaded global->LDS directly (V^T with the XOR swizzle of its 16-byte
// chunks applied through each lane's source address, for bank-conflict-free operand reads).  Only the
// last key tile can hold keys >= L, so the masked code runs once.
constexpr int kAttWaves = 4;
constexpr int att_block_q(int QT) { return kAttWaves * 32 * QT; }  // queries per workgroup of QT column tiles a wave

// Physical 16-byte chunk of logical chunk c in LDS row R is c ^ chunk_swz(R).  Operand reads touch
// rows R0..R0+31 at one logical chunk; with 64 four-byte banks (two 128-byte rows per bank sweep) this
// pattern is conflict-free for every group of 16 lanes (and for groups of 8 with 32 banks).
__device__ __forceinline__ int chunk_swz(int R) { return (R & 7) ^ ((R >> 3) & 1); }

// This wave's share of staging one 8 KB K tile into LDS, chunk-major like K itself: LDS block c
// (64 rows x 16 B) holds features 8c..8c+7 of the tile's 64 keys, row R = key (R&32)|pi(R&31).  Wave w
// stages chunks 2w and 2w+1, one 1 KB instruction each (64 consecutive rows of one chunk plane).
__device__ __forceinline__ void stage_k_tile(__amdgpu_buffer_rsrc_t kres, int kt, int Lpad, u32x4* lds_tile,
                                             int wave, int lane) {
  const int key = (lane & 32) | key_perm(lane & 31);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = 2 * wave + i;
    buffer_load_lds16(kres, (c * Lpad + kt * 64 + key) * 16, lds_tile + c * 64);
  }
}

// This wave's share of staging one 8 KB V^T tile (64 rows x 8 chunks of 16 B) into LDS: rows
// 16w..16w+15 (two instructions of 8 rows).  Row R holds head feature R.
__device__ __forceinline__ void stage_v_tile(__amdgpu_buffer_rsrc_t vres, int kt, int Lpad, u32x4* lds_tile,
                                             int wave, int lane) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int R = 16 * wave + 8 * i + (lane >> 3), pc = lane & 7;
    buffer_load_lds16(vres, (R * Lpad + kt * 64 + 8 * (pc ^ chunk_swz(R))) * 2, lds_tile + (16 * wave + 8 * i) * 8);
  }
}

// K operands of one 32-key half of a tile (chunk 2ks+hh of rows 32kh..32kh+31: 16 lanes read 256
// consecutive bytes, so the chunk-major tile needs no swizzle).
__device__ __forceinline__ void load_k_half(const u32x4* __restrict__ Kl, int kh, int j, int hh, u32x4 (&ka)[4]) {
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) ka[ks] = Kl[(2 * ks + hh) * 64 + 32 * kh + j];
}

// Softmax shift of the single pass.  Scores are base-2 exponents and the shift c of a query is an
// integer.  With an integer shift, P = bf16(2^(s-c)) = 2^-c bf16(2^s), so the normalised result does not
// depend on which integer c is (up to the fp32 rounding of s - c), as long as nothing over- or
// underflows: it is the non-online softmax of the reference with the row max m replaced by an integer,
// which only moves P's bf16 rounding by a factor 2^(m - c) that is a power of two times 2^(m - ceil m).
//
// The sweep therefore takes c once, from the first 32 keys, kAttHeadroomFast above their max, and
// computes 2^(s - c) for every later key with no max at all.  Keys far below c underflow only past
// 2^-126, i.e. more than ~94 below the first keys' max, where their weight is below fp32 resolution
// anyway.  A key far above c (more than ~60 above the first keys' max) would overflow the sums: the
// sweep checks every row's sum against kAttSafeSum (and O for finiteness) at the end, and if any row of
// the workgroup fails, the workgroup redoes the sweep with the guarded shift: c raised (never lowered)
// whenever a score exceeds it, to kAttHeadroom above the running max, with the earlier probabilities,
// their sum and the P.V accumulators scaled by 2^-d (exact).
constexpr float kAttHeadroom = 8.0f;       // guarded sweep
constexpr float kAttHeadroomFast = 32.0f;  // fixed-shift sweep
constexpr float kAttSafeSum = 1099511627776.0f;  // 2^40: fixed-shift sums at most this leave O finite

// One 32-key half of a tile for one 32-query column tile: S^T = K.Q^T accumulated onto -c, then
// P = 2^(s - c) as two B operands and the fp32 sum.  FIRST (the first half of tile 0, 32 valid keys) sets c
// from its own row max; SAFE (the guarded sweep) raises c when a score exceeds it.
template <bool FIRST, bool MASK, bool SAFE>
__device__ __forceinline__ void attn_half(const u32x4 (&ka)[4], const u32x4 (&qb)[4], int key0, int L, int hh,
                                          const u32x4& ones, f32x16& negc, f32x4& psum, f32x16 (&o)[2], u32x4& p0,
                                          u32x4& p1) {
  f32x16 sacc = FIRST ? zero16() : negc;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) sacc = mfma32(ka[ks], qb[ks], sacc);
  float hm = 0.f;
  if (FIRST || SAFE) {
    hm = MASK ? block_max(sacc, key0, L, hh, -INFINITY) : block_max(sacc, 0, 32, hh, -INFINITY);
    hm = halfwave_max(hm);  // the query's 32 keys sit in lanes j and j + 32
  }
  if (FIRST) {
    const float c = ceilf(hm) + (SAFE ? kAttHeadroom : kAttHeadroomFast);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      negc[r] = -c;
      sacc[r] -= c;
    }
  } else if (SAFE && __any(hm > 0.f)) {  // a score above the shift somewhere in the wave (rare)
    const float d = hm > 0.f ? ceilf(hm) + kAttHeadroom : 0.f;
    const int di = int(d);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      negc[r] -= d;
      sacc[r] -= d;
    }
    // the row-sum accumulator of lane n < 16 holds queries n (register 0) and n + 16 (register 1)
    const int di16 = __shfl(di, (__lane_id() & 15) + 16);
    psum[0] = ldexpf(psum[0], -di);
    psum[1] = ldexpf(psum[1], -di16);
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[dt][r] = ldexpf(o[dt][r], -di);
  }
  softmax_block_psum(sacc, MASK ? key0 : 0, MASK ? L : 32, hh, ones, psum, p0, p1);
}

// One 64-key tile: per 32-key half, scores and probabilities for both query tiles, then P.V.
template <bool FIRST, bool MASK, bool SAFE, int QT>
__device__ __forceinline__ void attn_tile(const u32x4* __restrict__ Kl, const u32x4* __restrict__ Vl,
                                          const u32x4 (&qb)[QT][4], int key0, int L, int j, int hh,
                                          const u32x4& ones, f32x16 (&negc)[QT], f32x4 (&psum)[QT],
                                          f32x16 (&o)[QT][2]) {
#pragma unroll
  for (int kh = 0; kh < 2; ++kh) {
    u32x4 ka[4];
    load_k_half(Kl, kh, j, hh, ka);
    u32x4 p0[QT], p1[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (FIRST && kh == 0)
        attn_half<true, false, SAFE>(ka, qb[qt], 0, L, hh, ones, negc[qt], psum[qt], o[qt], p0[qt], p1[qt]);
      else
        attn_half<false, MASK, SAFE>(ka, qb[qt], key0 + 32 * kh, L, hh, ones, negc[qt], psum[qt], o[qt], p0[qt],
                                     p1[qt]);
    }
#pragma unroll
    for (int dt = 0; dt < 2; ++dt) {
      const int d = 32 * dt + j;
      const u32x4 v0 = Vl[d * 8 + ((4 * kh + hh) ^ chunk_swz(d))];
      const u32x4 v1 = Vl[d * 8 + ((4 * kh + 2 + hh) ^ chunk_swz(d))];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        o[qt][dt] = mfma32(v0, p0[qt], o[qt][dt]);
        o[qt][dt] = mfma32(v1, p1[qt], o[qt][dt]);
      }
    }
  }
}

// K/V tiles stream through a ring of kAttBufs LDS buffers, prefetched kAttBufs-1 tiles ahead.  Tile kt
// is ready once at most the loads of the tiles issued after it are outstanding (N per tile per wave:
// 2 for a K tile, 4 for K + V), and the barrier makes every wave's share visible.
constexpr int kAttBufs = 3;

template <int QT>
__global__ __launch_bounds__(256, 4 - QT) void k_attn_long(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
                                                   const uint16_t* __restrict__ Vt, const float* __restrict__ G,
                                                   uint16_t* __restrict__ O, int mode, int L, int Lpad, int T,
                                                   int F, int nqb) {
  __shared__ u32x4 lds[kAttBufs][2][64 * 8];  // [buffer][K, V^T][64 rows x 8 chunks]
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5;
  // XCD-aware order: workgroups are dealt round-robin to the 8 XCDs (8 L2 caches), so block b runs on
  // XCD b % 8.  Give all query blocks of one (sequence, head) consecutive slots of one XCD, so its K and
  // V^T are fetched from HBM once into that XCD's L2 (nseq * 8 heads is a multiple of 8).
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;  // grid = nseq * 8 * nqb blocks
  const int sh = xcd + 8 * (slot / nqb), qblk = slot % nqb;
  const int s = sh >> 3, h = sh & 7;
  const uint16_t* Qh = Q + int64_t(sh) * Lpad * kHeadDim;
  // K and V^T of this (sequence, head) as buffer resources for the direct-to-LDS tile loads.
  const __amdgpu_buffer_rsrc_t Kh = buffer_rsrc(K + int64_t(sh) * Lpad * kHeadDim, Lpad * kHeadDim * 2);
  const __amdgpu_buffer_rsrc_t Vh = buffer_rsrc(Vt + int64_t(sh) * kHeadDim * Lpad, Lpad * kHeadDim * 2);
  const int q0 = qblk * att_block_q(QT) + wave * 32 * QT;
  const bool active = q0 < L;  // idle waves still stage tiles and meet every barrier

  u32x4 qb[QT][4];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int q = q0 + 32 * qt + j;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      qb[qt][ks] = q < Lpad ? *reinterpret_cast<const u32x4*>(Qh + (int64_t(2 * ks + hh) * Lpad + q) * 8) : zero4();
  }

  const int nkt = Lpad / 64;  // >= 2: this kernel runs for L > 64
  const u32x4 ones = rowsum_ones(lane);
  f32x4 psum[QT];
  f32x16 negc[QT], o[QT][2];
  auto sweep = [&](auto safe_tag) {
    constexpr bool SAFE = decltype(safe_tag)::value;
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      psum[qt] = f32x4{0.f, 0.f, 0.f, 0.f};
      negc[qt] = o[qt][0] = o[qt][1] = zero16();
    }
#pragma unroll
    for (int i = 0; i < kAttBufs - 1; ++i)
      if (i < nkt) {
        stage_k_tile(Kh, i, Lpad, lds[i][0], wave, lane);
        stage_v_tile(Vh, i, Lpad, lds[i][1], wave, lane);
      }
    vmcnt_barrier<4 * (kAttBufs - 2)>();  // tile 0 (nkt >= 2 >= kAttBufs - 1)
    if (kAttBufs - 1 < nkt) {
      stage_k_tile(Kh, kAttBufs - 1, Lpad, lds[kAttBufs - 1][0], wave, lane);
      stage_v_tile(Vh, kAttBufs - 1, Lpad, lds[kAttBufs - 1][1], wave, lane);
    }
    if (active) attn_tile<true, false, SAFE, QT>(lds[0][0], lds[0][1], qb, 0, L, j, hh, ones, negc, psum, o);
    for (int kt = 1; kt < nkt - 1; ++kt) {
      if (kt + kAttBufs - 2 < nkt)  // K and V: 4 loads per younger tile in flight
        vmcnt_barrier<4 * (kAttBufs - 2)>();
      else
        vmcnt_barrier<0>();
      if (kt + kAttBufs - 1 < nkt) {
        const int b = (kt + kAttBufs - 1) % kAttBufs;
        stage_k_tile(Kh, kt + kAttBufs - 1, Lpad, lds[b][0], wave, lane);
        stage_v_tile(Vh, kt + kAttBufs - 1, Lpad, lds[b][1], wave, lane);
      }
      if (active)
        attn_tile<false, false, SAFE, QT>(lds[kt % kAttBufs][0], lds[kt % kAttBufs][1], qb, 0, L, j, hh, ones, negc,
                                      psum, o);
    }
    vmcnt_barrier<0>();
    if (active)
      attn_tile<false, true, SAFE, QT>(lds[(nkt - 1) % kAttBufs][0], lds[(nkt - 1) % kAttBufs][1], qb, (nkt - 1) * 64, L,
                                   j, hh, ones, negc, psum, o);
  };
  sweep(std::integral_constant<bool, false>{});
  // Overflow check of the fixed-shift sweep (a key far above the first ones): the guarded sweep again,
  // by the whole workgroup (it streams K/V through the shared LDS ring), if any of its rows failed.
  bool bad = false;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    bad |= !(psum_of_query(psum[qt], j) <= kAttSafeSum);
    float om = 0.f;
#pragma unroll
    for (int dt = 0; dt < 2; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) om = fmaxf(om, fabsf(o[qt][dt][r]));
    bad |= !(om <= 3.0e38f);
  }
  if (__syncthreads_or(active && bad)) sweep(std::integral_constant<bool, true>{});
  if (!active) return;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt)
    attn_store(o[qt], q0 + 32 * qt + j, L, s, h, hh, mode, T, F, G, psum_of_query(psum[qt], j), O);
}

// Short sequences (frequency attention, L <= 64).  One wave = one (sequence, head): all
// operands come straight from global memory into registers, the whole 64x64 score block is
// computed once, so the exact softmax needs a single pass.
__global__ __launch_bounds__(256) void k_attn_short(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
                                                    const uint16_t* __restrict__ Vt, const float* __restrict__ G,
                                                    uint16_t* __restrict__ O, int mode, int nsh, int L, int T,
                                                    int F) {
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5;
  const int sh = blockIdx.x * 4 + wave;
  if (sh >= nsh) return;
  const int s = sh >> 3, h = sh & 7;
  constexpr int Lp = 64;
  const uint16_t* Qh = Q + int64_t(sh) * Lp * kHeadDim;
  const uint16_t* Kh = K + int64_t(sh) * Lp * kHeadDim;
  const uint16_t* Vh = Vt + int64_t(sh) * kHeadDim * Lp;

  u32x4 ka[2][4], va[2][4];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
      ka[kh][ks] = *reinterpret_cast<const u32x4*>(Kh + (int64_t(2 * ks + hh) * Lp + 32 * kh + key_perm(j)) * 8);
#pragma unroll
  for (int dt = 0; dt < 2; ++dt)
#pragma unroll
    for (int kc = 0; kc < 4; ++kc)
      va[dt][kc] = reinterpret_cast<const u32x4*>(Vh + int64_t(32 * dt + j) * Lp)[2 * kc + hh];

#pragma unroll 1
  for (int qt = 0; qt < 2; ++qt) {
    const int q = 32 * qt + j;
    if (32 * qt >= L) break;
    u32x4 qb[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) qb[ks] = *reinterpret_cast<const u32x4*>(Qh + (int64_t(2 * ks + hh) * Lp + q) * 8);
    f32x16 sacc[2];
    float m = -INFINITY;
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      sacc[kh] = zero16();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) sacc[kh] = mfma32(ka[kh][ks], qb[ks], sacc[kh]);
      m = block_max(sacc[kh], 32 * kh, L, hh, m);
    }
    m = fmaxf(m, __shfl_xor(m, 32));
    const float ml = m;  // scores are already in units of log2(e)
    float lsum = 0.f;
    f32x16 o[2] = {zero16(), zero16()};
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
      u32x4 p0, p1;
      softmax_block(sacc[kh], 32 * kh, L, hh, ml, lsum, p0, p1);
#pragma unroll
      for (int dt = 0; dt < 2; ++dt) {
        o[dt] = mfma32(va[dt][2 * kh], p0, o[dt]);
        o[dt] = mfma32(va[dt][2 * kh + 1], p1, o[dt]);
      }
    }
    lsum += __shfl_xor(lsum, 32);
    attn_store(o, q, L, s, h, hh, mode, T, F, G, lsum, O);
  }
}

void launch_attention(const uint16_t* Q, const uint16_t* K, const uint16_t* Vt, const float* G, uint16_t* O,
                      const SeqShape& sh, hipStream_t st, const LaunchEvents& ev) {
  if (sh.L <= 64) {
    const int nsh = sh.nseq * kHeads;
    hipExtLaunchKernelGGL(k_attn_short, dim3((nsh + 3) / 4), dim3(256), 0, st, ev.start, ev.stop, 0, Q, K, Vt, G, O,
                          sh.mode, nsh, sh.L,
                       sh.T, sh.F);
  } else {
    // Two column tiles a wave share each operand read of a 256-query workgroup; one makes a 128-query
    // workgroup, for an odd number of 128-query blocks, whose last 256-query one would run half empty. us at
    // 62 bands, QT = 2 and 1: L = 101 11.2 and 9.6, 257 30.8 and 24.2, 384 35.3 and 30.3, 520 58.3 and 55.9,
    // 640 65.3 and 64.5, 896 114 and 114 (even numbers of blocks: 200 18.6 and 19.2, 800 102 and 101). With few and
    // with many sequences alike: L = 257 10.3 and 9.1 at 4, 216 and 173 at 496; 640 15.0 and 10.5 at 4, 213 and 192
    // at 186.
    const int blocks = (sh.L + att_block_q(1) - 1) / att_block_q(1);
    const int QT = blocks % 2 && blocks <= 5 ? 1 : 2;
    const int nqb = (sh.L + att_block_q(QT) - 1) / att_block_q(QT);
    const auto kernel = QT == 1 ? k_attn_long<1> : k_attn_long<2>;
    hipExtLaunchKernelGGL(kernel, dim3(sh.nseq * kHeads * nqb), dim3(64 * kAttWaves), 0, st, ev.start, ev.stop,
                          0, Q, K, Vt, G, O,
                       sh.mode, sh.L, sh.Lpad, sh.T, sh.F, nqb);
  }
}

// ============================================================ GELU
// erf-GELU x Phi(x) = max(x, 0) - 0.5|x| erfc(|x|/sqrt 2), with erfc from Abramowitz & Stegun 7.1.26
// (|error of erf| <= 1.5e-7): erfc(z) = t (a1 + t (a2 + t (a3 + t (a4 + t a5)))) e^(-z^2),
// t = 1/(1 + p z), p = 0.3275911.  Written in y = |x| sqrt(log2(e)/2) it is
//   0.5|x| erfc(|x|/sqrt 2) = y t P(t) 2^(-y^2),  t = 1/(1 + p' y),  p' = p / sqrt(log2 e),
//   P(t) = k (a1 + a2 t + a3 t^2 + a4 t^3 + a5 t^4),  k = 0.5 / sqrt(log2(e)/2),
// 11 VALU operations and two transcendentals; |GELU error| <= 2.2e-7 over the real line.  For x < 0 the
// result is the small erfc term itself (no cancellation).
constexpr float kGeluC = 0.84932180028801904f;   // sqrt(log2(e)/2)
constexpr float kGeluP = 0.27273748087922250f;   // 0.3275911 / sqrt(log2 e)
constexpr float kGeluA1 = 0.15001945782716460f;  // k * 0.254829592
constexpr float kGeluA2 = -0.16748465416966950f; // k * -0.284496736
constexpr float kGeluA3 = 0.83679339239730750f;  // k * 1.421413741
constexpr float kGeluA4 = -0.85547788041423880f; // k * -1.453152027
constexpr float kGeluA5 = 0.62485469502846850f;  // k * 1.061405429

__device__ __forceinline__ float gelu_erf(float x) {
  const float y = fabsf(x) * kGeluC;
  const float t = __builtin_amdgcn_rcpf(fmaf(kGeluP, y, 1.0f));
  float p = fmaf(kGeluA5, t, kGeluA4);
  p = fmaf(p, t, kGeluA3);
  p = fmaf(p, t, kGeluA2);
  p = fmaf(p, t, kGeluA1);
  const float e = __builtin_amdgcn_exp2f(-(y * y));
  return fmaf(-(y * t) * p, e, fmaxf(x, 0.0f));
}

// The same for the GELU op, which stands on its own and so has to be as close as 0.5 x (1 + erff(x / sqrt 2)) is:
// P one degree higher, with the smallest largest error (3.2e-9 in the GELU).  fp32 rms error over N(0, 1) inputs
// 2.2e-8 (that formula 2.4e-8, A&S 5.5e-8) and 1.4e-5 of the outputs rounded to the wrong bf16 (2.4e-5, 9.6e-5),
// for an FMA and a minimum more than A&S; erff itself made the op a third slower (98 and 131 us at 105,462 tokens,
// n_out = 1024).  The minimum keeps infinite x (y t = inf 0) at x and 0; it changes nothing else, since
// 2^(-y^2) is 0 long before.
constexpr float kOpGeluP = 0.33f;
constexpr float kOpGeluA0 = 0.13789169490337372f;
constexpr float kOpGeluA1 = 0.07618103176355362f;
constexpr float kOpGeluA2 = 0.32476791739463806f;
constexpr float kOpGeluA3 = -0.28829991817474365f;
constexpr float kOpGeluA4 = 0.4644383490085602f;
constexpr float kOpGeluA5 = -0.12627415359020233f;

__device__ __forceinline__ float gelu_op(float x) {
  const float y0 = fabsf(x) * kGeluC;
  const float y = fminf(y0, 64.0f);
  const float t = __builtin_amdgcn_rcpf(fmaf(kOpGeluP, y0, 1.0f));
  float p = fmaf(kOpGeluA5, t, kOpGeluA4);
  p = fmaf(p, t, kOpGeluA3);
  p = fmaf(p, t, kOpGeluA2);
  p = fmaf(p, t, kOpGeluA1);
  p = fmaf(p, t, kOpGeluA0);
  const float e = __builtin_amdgcn_exp2f(-(y * y));
  return fmaf(-(y * t) * p, e, fmaxf(x, 0.0f));
}

// erf-GELU of the fp16 and bf16 feed-forward, whose output is rounded to fp16 or bf16: x Phi(x) written as
// x sigmoid(z(x)), with z(x) = x P(min(x^2, 30)) and P a cubic, a minimax fit of logit Phi(x) weighted by
// how an error in z moves the GELU (x Phi (1 - Phi)).  In base 2 (the coefficients carry log2 e):
//   gelu(x) = x / (1 + 2^(-x P(x^2)))
// 8 VALU operations and two transcendentals (the A&S form above: 11 and two); |GELU error| <= 1.25e-5
// over the real line, against fp16 rounding steps of 1.2e-4 and more for |GELU| >= 0.25.  The clamp
// keeps z monotone past |x| = 5.5, where the sigmoid has saturated: large x give x, large -x give -0.
constexpr float kGeluClamp = 30.0f;
constexpr float kGeluL0 = 2.3016500915968159f;
constexpr float kGeluL1 = 0.10597803067691149f;
constexpr float kGeluL2 = -0.0007343367166309341f;
constexpr float kGeluL3 = -2.5004358251987334e-05f;

__device__ __forceinline__ float gelu_logistic(float x) {
  const float x2 = fminf(x * x, kGeluClamp);
  float p = fmaf(kGeluL3, x2, kGeluL2);
  p = fmaf(p, x2, kGeluL1);
  p = fmaf(p, x2, kGeluL0);
  const float e = __builtin_amdgcn_exp2f(-(x * p));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// ============================================================ token-tile GEMM kernels
// Workgroups of 8 waves on tiles of 32 C tokens, see trf_tiles.h.
constexpr int kDropOffset = 0x7ffffff0;  // a buffer offset past every resource: its loads give zeros

// The norms of a tile's tokens: wave w's partial sum of squares of token t is ssq[t * kTileWaves + w].
template <int C>
__device__ __forceinline__ void put_ssq(const f32x16 (&acc)[C], float* ssq, int wave, int j, int hh) {
#pragma unroll
  for (int ct = 0; ct < C; ++ct) {
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s = fmaf(acc[ct][r], acc[ct][r], s);
    s += __shfl_xor(s, 32);
    if (hh == 0) ssq[(32 * ct + j) * kTileWaves + wave] = s;
  }
}

__device__ __forceinline__ float inv_norm(const float* ssq, int t, float eps) {
  const f32x4 p = *reinterpret_cast<const f32x4*>(ssq + t * kTileWaves);
  const f32x4 q = *reinterpret_cast<const f32x4*>(ssq + t * kTileWaves + 4);
  return 1.0f / fmaxf(sqrtf(((p[0] + p[1]) + (p[2] + p[3])) + ((q[0] + q[1]) + (q[2] + q[3]))), eps);
}

// The end of a tile: acc (tile `wave` of every token's features) -> X rows and, normalised, xn rows (NORM).
// `rowbuf` holds the tile's fp32 rows; every wave has met since its last use, and since put_ssq (NORM).
template <int C, bool NORM>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[C], u32x4* rowbuf, const float* ssq, float eps,
                                           __amdgpu_buffer_rsrc_t xres, __amdgpu_buffer_rsrc_t nres, int wave,
                                           int lane) {
  constexpr int RW = 32 * C / kTileWaves;
  const int j = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int ct = 0; ct < C; ++ct)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 x = {acc[ct][4 * g], acc[ct][4 * g + 1], acc[ct][4 * g + 2], acc[ct][4 * g + 3]};
      rowbuf[row_chunk(32 * ct + j, 8 * wave + 2 * g + hh)] = __builtin_bit_cast(u32x4, x);
    }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const int t = wave * RW + i;
    const u32x4 v = rowbuf[row_chunk(t, lane)];
    const f32x4 x = __builtin_bit_cast(f32x4, v);
    __builtin_amdgcn_raw_buffer_store_b128(v, xres, lane * 16 + t * (kDim * 4), 0, 0);
    if (!NORM) continue;
    const float inv = inv_norm(ssq, t, eps);
    const u32x2 y = {pk_bf16(x[0] * inv, x[1] * inv), pk_bf16(x[2] * inv, x[3] * inv)};
    __builtin_amdgcn_raw_buffer_store_b64(y, nres, lane * 8 + t * (kDim * 2), 0, 0);
  }
}

// acc += x (or = x, INIT) for this wave's tile of features, from the tile's fp32 rows.
template <int C, bool INIT>
__device__ __forceinline__ void add_rows(const u32x4* rowbuf, f32x16 (&acc)[C], int wave, int j, int hh) {
#pragma unroll
  for (int ct = 0; ct < C; ++ct)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 x = __builtin_bit_cast(f32x4, rowbuf[row_chunk(32 * ct + j, 8 * wave + 2 * g + hh)]);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[ct][4 * g + r] = INIT ? x[r] : acc[ct][4 * g + r] + x[r];
    }
}

// ============================================================ GEMM + residual + next norm
// X[tok] += A[tok] . W^T (+ b); xn[tok] = X / max(|X|, eps), for any A width K (a multiple of 16) and a
// weight W [256][K] packed in natural k order (launch_pack, kPack32Natural); xn may be null (not written).
// A is staged in panels of 512 columns (a row's chunks past K are dropped).  HBM-bound (378 MB at
// 105,462 tokens and K = 512: 74 us at the rate of a copy; 486 MB and 95 us at K = 1024): 76 and 127 us, of
// 221 and 422 for waves that read A and W from global memory as they multiplied, with no LDS.
// (kernels.cpp:542-586)
template <int C>
__global__ __launch_bounds__(64 * kTileWaves, 4) void k_gemm_res_norm(const uint16_t* __restrict__ A, int K,
                                                                      const u32x4* __restrict__ wq,
                                                                      const float* __restrict__ bias,
                                                                      float* __restrict__ X,
                                                                      uint16_t* __restrict__ xn, int64_t n,
                                                                      float eps) {
  constexpr int R = 32 * C, RW = R / kTileWaves;  // tokens of the tile, rows a wave moves
  __shared__ u32x4 smem[R * 64 + R * kTileWaves / 4];
  float* const ssq = reinterpret_cast<float*>(smem + R * 64);
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5, t0 = wave * RW;
  const int64_t tok0 = int64_t(blockIdx.x) * R;
  const int rows = int(n - tok0 < R ? n - tok0 : R);
  const auto xres = buffer_rsrc(X + tok0 * kDim, rows * kDim * 4);
  const auto nres = buffer_rsrc(xn + tok0 * kDim, rows * kDim * 2);  // (no store without xn)
  const int KS = K / 16, chunks = K / 8, panels = (K + 511) / 512;
  const auto wres = buffer_rsrc(wq + int64_t(wave) * KS * 64, KS * kTileBytes);
  auto stage = [&](int panel) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int t = t0 + i, c = 64 * panel + (lane ^ (t & 15));
      const auto ares = buffer_rsrc(A + (tok0 + (t < rows ? t : 0)) * K, K * 2);  // one row
      buffer_load_lds16(ares, c < chunks ? c * 16 : kDropOffset, smem + t * 64);
    }
  };
  stage(0);
  u32x4 xr[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) xr[i] = buffer_load16(xres, lane * 16 + (t0 + i) * (kDim * 4), 0);
  auto weight = [&](int k) __attribute__((always_inline)) {  // k-step k (past the last one: the last, unused)
    return buffer_load16(wres, lane * 16, min(k, KS - 1) * kTileBytes);
  };
  u32x4 a[kWeightAhead];
#pragma unroll
  for (int i = 0; i < kWeightAhead; ++i) a[i] = weight(i);
  f32x16 acc[C];
#pragma unroll
  for (int ct = 0; ct < C; ++ct) acc[ct] = zero16();
  const int m = j & 15, base = j * 64 + (hh ^ (m & 1)), me = m & 14;  // chunk 2k + hh of token j
#pragma unroll 1
  for (int panel = 0; panel < panels; ++panel) {
    if (panel) {
      lds_barrier();  // every wave has read the previous panel
      stage(panel);
    }
    loads_barrier();
    const int steps = min(32, KS - 32 * panel);
#pragma unroll 1
    for (int g = 0; g < steps / 8; ++g) {
      const u32x4* p = smem + base + 16 * g;
      const int next = 32 * panel + 8 * g + kWeightAhead;
      u32x4 b[2][C];
#pragma unroll
      for (int ct = 0; ct < C; ++ct) b[0][ct] = p[me + ct * 32 * 64];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (k + 1 < 8) {
#pragma unroll
          for (int ct = 0; ct < C; ++ct) b[(k + 1) & 1][ct] = p[((2 * k + 2) ^ me) + ct * 32 * 64];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ct = 0; ct < C; ++ct) acc[ct] = mfma32(a[k % kWeightAhead], b[k & 1][ct], acc[ct]);
        a[k % kWeightAhead] = weight(next + k);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll 1
    for (int k = steps & ~7; k < steps; ++k) {  // K not a multiple of 128: only in the last panel
      const u32x4 w = weight(32 * panel + k);
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = mfma32(w, smem[base + ((2 * k) ^ me) + ct * 32 * 64], acc[ct]);
    }
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < RW; ++i) smem[row_chunk(t0 + i, lane)] = xr[i];
  lds_barrier();
  add_rows<C, false>(smem, acc, wave, j, hh);
  if (bias) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(bias + 32 * wave + row_of_group(g, hh));
#pragma unroll
      for (int ct = 0; ct < C; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[ct][4 * g + r] += b[r];
    }
  }
  if (xn) put_ssq(acc, ssq, wave, j, hh);
  lds_barrier();
  if (xn)
    store_tile<C, true>(acc, smem, ssq, eps, xres, nres, wave, lane);
  else
    store_tile<C, false>(acc, smem, ssq, eps, xres, nres, wave, lane);
}

void launch_gemm_res_norm(const uint16_t* A, int K, const uint8_t* w_packed, const float* bias, float* X,
                          uint16_t* xn, int64_t n, float eps, hipStream_t st, const LaunchEvents& ev) {
  // One panel of A: a tile's two memory phases leave little for the weights to bound, and 32-token tiles, whose
  // accumulators and X rows need no scratch, overlap them better.  us, 64- and 32-token tiles, K = 512: 22.1 and
  // 18.4 at 18,786 tokens, 23.2 and 24.5 at 24,800 (the one size where they lose: the 64-token tiles are one
  // round), 51.5 and 42.1 at 52,700, 91 and 76 at 105,462; K = 128: 60 and 52 there.  More panels: K = 768 57 and 54
  // at 52,700 but 27 and 29.6 at 24,800; K = 1024 63 and 68, 127 and 137 at 105,462.
  const int C = K <= 512 ? 1 : token_tiles(n);
  const auto kernel = C == 1 ? k_gemm_res_norm<1> : k_gemm_res_norm<2>;
  hipExtLaunchKernelGGL(kernel, dim3(unsigned((n + 32 * C - 1) / (32 * C))), dim3(64 * kTileWaves), 0, st, ev.start,
                        ev.stop, 0, A, K, reinterpret_cast<const u32x4*>(w_packed), bias, X, xn, n, eps);
}

// ============================================================ FF1 GEMM + GELU
// H = 0.5 x (1 + erf(x / sqrt 2)), x = xn . W^T + b  (nn.GELU() default, model.py:69), for a weight
// W [n_out][256] packed in natural k order (n_out a multiple of 32) and H [n][n_out].
// 256 outputs (one weight tile per wave) at a time, through LDS into H as 16-byte chunks of whole rows:
// position 32 t + (c ^ (t & 15)) for chunk c of token t, as for the tile's xn rows.
// Bounded by the H writes (270 MB at 105,462 tokens, n_out = 1024: 53 us at the rate of a copy): 109 us, of
// 267 for waves that read W from global memory one tile at a time and stored H in operand layout.
template <int C>
__global__ __launch_bounds__(64 * kTileWaves, 4) void k_gemm_gelu(const uint16_t* __restrict__ xn,
                                                                  const u32x4* __restrict__ wq,
                                                                  const float* __restrict__ b1, int n_out,
                                                                  uint16_t* __restrict__ H, int64_t n) {
  constexpr int R = 32 * C;
  __shared__ u32x4 smem[2 * R * 32];
  u32x4* const hs = smem + R * 32;  // the outputs on their way out
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5;
  const int64_t tok0 = int64_t(blockIdx.x) * R;
  const int rows = int(n - tok0 < R ? n - tok0 : R);
  const auto nres = buffer_rsrc(xn + tok0 * kDim, rows * kDim * 2);
  // 1 KB = two rows of 32 chunks per instruction; wave w moves instructions w, w + 8, ...
  const int rp = lane >> 5, rc = lane & 31;
#pragma unroll
  for (int i = 0; i < R / 2 / kTileWaves; ++i) {
    const int t = 2 * (kTileWaves * i + wave) + rp;
    buffer_load_lds16(nres, t * (kDim * 2) + 16 * (rc ^ (t & 15)), smem + 2 * (kTileWaves * i + wave) * 32);
  }
  const int tiles = n_out / 32;
  // weight tile t's blocks (past the last tile: the last one's, whose products are not stored)
  auto tile_res = [&](int t) { return buffer_rsrc(wq + int64_t(min(t, tiles - 1)) * 16 * 64, 16 * kTileBytes); };
  auto wr = tile_res(wave);
  u32x4 a[kWeightAhead];
#pragma unroll
  for (int i = 0; i < kWeightAhead; ++i) a[i] = buffer_load16(wr, lane * 16, i * kTileBytes);
  const int m = j & 15, base = j * 32 + (hh ^ (m & 1)), me = m & 14;  // chunk 2k + hh of token j
  loads_barrier();
#pragma unroll 1
  for (int t8 = 0; t8 < tiles; t8 += kTileWaves) {
    const int tile = t8 + wave;
    const auto next = tile_res(tile + kTileWaves);
    f32x16 acc[C];
    {
      f32x4 b[4];
#pragma unroll
      for (int g = 0; g < 4; ++g)
        b[g] = *reinterpret_cast<const f32x4*>(b1 + (tile < tiles ? 32 * tile : 0) + row_of_group(g, hh));
#pragma unroll
      for (int ct = 0; ct < C; ++ct)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[ct][r] = b[r >> 2][r & 3];
    }
    u32x4 b[2][C];
#pragma unroll
    for (int ct = 0; ct < C; ++ct) b[0][ct] = smem[base + me + ct * 32 * 32];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (k + 1 < 16) {
        const int c = ((2 * k + 2) & 16) + (((2 * k + 2) & 14) ^ me);
#pragma unroll
        for (int ct = 0; ct < C; ++ct) b[(k + 1) & 1][ct] = smem[base + c + ct * 32 * 32];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = mfma32(a[k % kWeightAhead], b[k & 1][ct], acc[ct]);
      if (k + kWeightAhead < 16)
        a[k % kWeightAhead] = buffer_load16(wr, lane * 16, (k + kWeightAhead) * kTileBytes);
      else
        a[k % kWeightAhead] = buffer_load16(next, lane * 16, (k + kWeightAhead - 16) * kTileBytes);
      __builtin_amdgcn_sched_barrier(0);
    }
    wr = next;
    if (t8) lds_barrier();  // the previous 256 outputs have left hs
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
#pragma unroll
      for (int g = 0; g < 4; ++g) {  // features 8g + 4hh .. +3 of this wave's tile: half hh of chunk 4 wave + g
        const int t = 32 * ct + j;
        const u32x2 v = {pk_bf16(gelu_op(acc[ct][4 * g]), gelu_op(acc[ct][4 * g + 1])),
                         pk_bf16(gelu_op(acc[ct][4 * g + 2]), gelu_op(acc[ct][4 * g + 3]))};
        reinterpret_cast<u32x2*>(hs)[2 * (t * 32 + ((4 * wave + g) ^ (t & 15))) + hh] = v;
      }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < R / 2 / kTileWaves; ++i) {
      const int t = 2 * (kTileWaves * i + wave) + rp;
      const u32x4 v = hs[t * 32 + (rc ^ (t & 15))];
      if (t < rows && 4 * t8 + rc < 4 * tiles)
        *reinterpret_cast<u32x4*>(H + (tok0 + t) * n_out + 32 * t8 + 8 * rc) = v;
    }
  }
}

// The same for a narrow output of many tokens: a wave is 32 tokens, from global memory to global memory, without
// LDS or barriers.  Above, one or two of the eight waves have a weight tile and the others only move rows; that
// costs when the rows no longer come and go under one round of workgroups.  us, above and here: n_out = 32 8.2 and
// 8.3 at 18,786 tokens, 14.4 and 8.1 at 52,700, 29.0 and 13.8 at 105,462; n_out = 64 9.3 and 10 at 32,674, 14.9 and
// 10.8 at 52,700, 29.6 and 19.9 at 105,462.  Same sums, so the same bits.
__global__ __launch_bounds__(256) void k_gemm_gelu_narrow(const uint16_t* __restrict__ xn, const u32x4* __restrict__ wq,
                                                          const float* __restrict__ b1, int n_out,
                                                          uint16_t* __restrict__ H, int64_t n) {
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5;
  const int64_t tok = (int64_t(blockIdx.x) * 4 + wave) * 32 + j;
  const bool valid = tok < n;
  const u32x4* const xr = reinterpret_cast<const u32x4*>(xn + (valid ? tok : n - 1) * kDim);
  u32x4 x[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) x[k] = xr[2 * k + hh];
  uint16_t* const hr = H + tok * n_out;
#pragma unroll 1
  for (int t = 0; t < n_out / 32; ++t) {
    const u32x4* const w = wq + t * 16 * 64 + lane;
    f32x16 acc;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(b1 + 32 * t + row_of_group(g, hh));
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[4 * g + r] = b[r];
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) acc = mfma32(w[k * 64], x[k], acc);
    if (!valid) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      *reinterpret_cast<u32x2*>(hr + 32 * t + row_of_group(g, hh)) =
          u32x2{pk_bf16(gelu_op(acc[4 * g]), gelu_op(acc[4 * g + 1])),
                pk_bf16(gelu_op(acc[4 * g + 2]), gelu_op(acc[4 * g + 3]))};
  }
}

void launch_gemm_gelu(const uint16_t* xn, const uint8_t* w_packed, const float* bias, int n_out, uint16_t* H,
                      int64_t n, hipStream_t st) {
  if (n_out <= 64 && n > 512 * int64_t(n_out)) {
    hipLaunchKernelGGL(k_gemm_gelu_narrow, dim3(unsigned((n + 127) / 128)), dim3(256), 0, st, xn,
                       reinterpret_cast<const u32x4*>(w_packed), bias, n_out, H, n);
    return;
  }
  const int C = token_tiles(n);
  const auto kernel = C == 1 ? k_gemm_gelu<1> : k_gemm_gelu<2>;
  hipLaunchKernelGGL(kernel, dim3(unsigned((n + 32 * C - 1) / (32 * C))), dim3(64 * kTileWaves), 0, st, xn,
                     reinterpret_cast<const u32x4*>(w_packed), bias, n_out, H, n);
}

// ============================================================ fused post-attention block
// out-projection + residual + norm, then FF1 + GELU + FF2 + residual + norm, for a tile of 32 C tokens:
//   acc  := O . Wout^T + X                      (wave w: features 32w..32w+31 of every token)
//   xn1  := acc / |acc|                         (FF1 B operands, in LDS)
//   for each of 4 blocks c of 256 hidden units (wave w: units 256c + 32w ..+31):
//     h   := b1 + xn1 . W1^T ;  gelu(h) -> LDS (FF2 B operands) ;  acc += gelu(h) . W2^T
//   acc  += b2 ; X := acc ; xn := acc / |acc|
// The accumulator registers of a 32-row tile are the B operand of two k-steps as they stand (W1, W2 are
// packed in register order), so xn1 and gelu(h) pass through LDS as whole operand blocks, and the
// 1024-wide hidden activation never leaves the chip.  FF1 of block c + 1 comes before FF2 of block c, whose
// MFMAs the GELU of block c + 1 is spread between.
// The feed-forward runs in bf16, fp16 or split-bf16 operands (PREC, FfPrecision); the out-projection stays
// bf16.  Split: both FF GEMMs take v = hi + lo (hi = bf16(v), lo = bf16(v - hi)) and form
// hi.hi + hi.lo + lo.hi with fp32 accumulation; the dropped lo.lo term is ~2^-16 relative.
// Without OUTPROJ the block starts at X and writes no xn (the feed-forward sub-layer alone).
//
// What it replaced: 256-token workgroups whose waves each held all 256 features of 32 tokens and took the
// weights from LDS in 41 barrier-separated stages (fp16, bf16), and the same with 16 tokens a wave on
// 16x16x32 MFMAs (split).  us per launch, then and now: 212 and 180 at 105,462 tokens in the stack (fp16),
// 80 and 21.5 at 6,262; the feed-forward alone 74 and 38 at 18,786 (fp16), 365 and 319 at 105,462 (split).
// At 105,462 tokens the parts are 74 us of HBM traffic (378 MB at the rate of a copy), 56 us of MFMA work
// and, without either, ~30 us for the weights' way from L2; the tiles of a round start together, so they
// overlap only in part (priorities for one of a CU's two workgroups change nothing). In cycles the fp16 block is 22%
// shorter there, 446k and 348k; the chip's power limit takes the clock from 2.27 to 1.95 GHz, also under the kernels
// beside it. The split block at C = 1 keeps 4 registers in scratch.
// (fast.py:311-331, kernels.cpp:542-642)

// FF operand packing of the one-part arithmetics.
template <int PREC>
__device__ __forceinline__ uint32_t pk_ff(float lo, float hi) {
  return PREC == kFfFp16 ? pk_f16(lo, hi) : pk_bf16(lo, hi);
}
// The bf16 hi and lo parts of a pair.
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = pk_bf16(a, b);
  lo = pk_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u));
}

// Operand pair (a, b) of an FF GEMM into word q of the part's operand registers.
template <int PREC>
__device__ __forceinline__ void pack_ff(float a, float b, u32x4 (&v)[ff_parts(PREC)], int q) {
  if constexpr (PREC == kFfSplit) {
    uint32_t h, l;
    split_pair(a, b, h, l);
    v[0][q] = h;
    v[1][q] = l;
  } else {
    v[0][q] = pk_ff<PREC>(a, b);
  }
}

// The split arithmetic at C = 2 holds 128 KB of operands: one workgroup per CU, 256 registers a wave.
constexpr int pa_waves_per_simd(int C, int prec) { return C == 2 && prec == kFfSplit ? 2 : 4; }

template <int C, bool OUTPROJ, int PREC>
__global__ __launch_bounds__(64 * kTileWaves, pa_waves_per_simd(C, PREC)) void k_post_attn(
    const uint16_t* __restrict__ O, const uint8_t* __restrict__ layer, float* __restrict__ X,
    uint16_t* __restrict__ xn, int64_t n, float eps) {
  constexpr int R = 32 * C, RW = R / kTileWaves;  // tokens of the tile, rows a wave moves
  constexpr int NP = ff_parts(PREC);
  constexpr int kPart = C * 16 * 64;  // one part of xn1 or of a hidden block as operand blocks [ct][k-step][lane]
  constexpr int kBias = 2 * NP * kPart, kSsq = kBias + (kHidden + kDim) / 4;
  __shared__ u32x4 smem[kSsq + R * kTileWaves / 4];
  u32x4* const xb = smem;               // xn1; with hb also the tile's O rows, X rows and output rows
  u32x4* const hb = smem + NP * kPart;  // gelu(h) of one block
  const u32x4* const bias = smem + kBias;  // b1, b2
  float* const ssq = reinterpret_cast<float*>(smem + kSsq);
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5, t0 = wave * RW;
  const int64_t tok0 = int64_t(blockIdx.x) * R;
  const int rows = int(n - tok0 < R ? n - tok0 : R);  // rows past the last token read as zeros, stores drop
  const auto xres = buffer_rsrc(X + tok0 * kDim, rows * kDim * 4);
  const auto nres = buffer_rsrc(xn + tok0 * kDim, rows * kDim * 2);  // (no store without OUTPROJ)
  const TileWeights w{buffer_rsrc(layer, int(kLayerBytes)), lane * 16};
  {
    static_assert(kDim * 4 == 512 * 2, "rows of O and X are 1 KB");
    const auto rres = OUTPROJ ? buffer_rsrc(O + tok0 * 512, rows * 1024) : xres;
#pragma unroll
    for (int i = 0; i < RW; ++i)
      buffer_load_lds16(rres, (t0 + i) * 1024 + 16 * (lane ^ ((t0 + i) & 15)), smem + (t0 + i) * 64);
    if (wave < 4) buffer_load_lds16(w.res, int(kOffBff1) + wave * 1024 + lane * 16, smem + kBias + wave * 64);
    if (wave == 4) buffer_load_lds16(w.res, int(kOffBff2) + lane * 16, smem + kBias + kHidden / 4);
  }
  u32x4 xr[RW];  // X rows, added after the out-projection
  if (OUTPROJ) {
#pragma unroll
    for (int i = 0; i < RW; ++i) xr[i] = buffer_load16(xres, lane * 16 + (t0 + i) * 1024, 0);
  }
  constexpr int w1[2] = {int(PREC == kFfFp16 ? kOffFf1F16 : kOffFf1), int(kOffFf1Lo)};
  constexpr int w2[2] = {int(PREC == kFfFp16 ? kOffFf2F16 : kOffFf2), int(kOffFf2Lo)};
  const TileOff out{{int(kOffOut) + wave * 32 * kTileBytes, 0}};
  auto ff1 = [&](int c) __attribute__((always_inline)) { return TileOff{{w1[0] + (8 * c + wave) * 16 * kTileBytes, w1[1] + (8 * c + wave) * 16 * kTileBytes}}; };
  auto ff2 = [&](int c) __attribute__((always_inline)) { return TileOff{{w2[0] + (64 * wave + 16 * c) * kTileBytes, w2[1] + (64 * wave + 16 * c) * kTileBytes}}; };
  u32x4 a[kWeightAhead][2];
  {
    const TileOff first = OUTPROJ ? out : ff1(0);
#pragma unroll
    for (int i = 0; i < kWeightAhead; ++i)
#pragma unroll
      for (int p = 0; p < (OUTPROJ ? 1 : NP); ++p) a[i][p] = w.load(first.v[p] + i * kTileBytes);
  }
  auto none = [](int) __attribute__((always_inline)) {};
  f32x16 acc[C];
  loads_barrier();
  if (OUTPROJ) {
#pragma unroll
    for (int ct = 0; ct < C; ++ct) acc[ct] = zero16();
    const int m = j & 15, base = j * 64 + (hh ^ (m & 1)), me = m & 14;  // chunk 2k + hh of token j
    tile_gemm<32, C, kFfBf16, NP>(w, out.v, ff1(0).v, a, acc,
                                [&](int k, int, int ct) __attribute__((always_inline)) {
                                  return smem[base + ((2 * k) ^ me) + ct * 32 * 64];
                                },
                                none);
    lds_barrier();
#pragma unroll
    for (int i = 0; i < RW; ++i) smem[row_chunk(t0 + i, lane)] = xr[i];
    lds_barrier();
  }
  add_rows<C, !OUTPROJ>(smem, acc, wave, j, hh);
  put_ssq(acc, ssq, wave, j, hh);
  lds_barrier();
#pragma unroll
  for (int ct = 0; ct < C; ++ct) {
    const float inv = inv_norm(ssq, 32 * ct + j, eps);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      u32x4 v[NP];
#pragma unroll
      for (int e = 0; e < 4; ++e) pack_ff<PREC>(acc[ct][8 * q + 2 * e] * inv, acc[ct][8 * q + 2 * e + 1] * inv, v, e);
#pragma unroll
      for (int p = 0; p < NP; ++p) xb[p * kPart + (ct * 16 + 2 * wave + q) * 64 + lane] = v[p];
    }
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 b = __builtin_bit_cast(f32x4, bias[kHidden / 4 + 8 * wave + 2 * g + hh]);
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[ct][4 * g + r] += b[r];
  }
  lds_barrier();

  f32x16 h[C];
  u32x4 hp[C][2][NP];  // gelu(h) as operands
  auto start_h = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4 b = __builtin_bit_cast(f32x4, bias[8 * (8 * c + wave) + 2 * g + hh]);
#pragma unroll
      for (int ct = 0; ct < C; ++ct)
#pragma unroll
        for (int r = 0; r < 4; ++r) h[ct][4 * g + r] = b[r];
    }
  };
  auto gelu_pair = [&](int v) __attribute__((always_inline)) {  // values 2v, 2v + 1 of the wave's 16 C per lane
    const int ct = v >> 3, p = v & 7;
    const float x = h[ct][2 * p], y = h[ct][2 * p + 1];
    if constexpr (PREC == kFfSplit)
      pack_ff<PREC>(gelu_erf(x), gelu_erf(y), hp[ct][p >> 2], p & 3);
    else
      pack_ff<PREC>(gelu_logistic(x), gelu_logistic(y), hp[ct][p >> 2], p & 3);
  };
  auto put_h = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
#pragma unroll
      for (int q = 0; q < 2; ++q)
#pragma unroll
        for (int p = 0; p < NP; ++p) hb[p * kPart + (ct * 16 + 2 * wave + q) * 64 + lane] = hp[ct][q][p];
    lds_barrier();
  };
  auto xop = [&](int k, int p, int ct) __attribute__((always_inline)) { return xb[p * kPart + (ct * 16 + k) * 64 + lane]; };
  auto hop = [&](int k, int p, int ct) __attribute__((always_inline)) { return hb[p * kPart + (ct * 16 + k) * 64 + lane]; };
  constexpr int kBlocks = kHidden / 256;
  start_h(0);
  tile_gemm<16, C, PREC, NP>(w, ff1(0).v, ff1(1).v, a, h, xop, none);
#pragma unroll
  for (int v = 0; v < 8 * C; ++v) gelu_pair(v);
  put_h();
#pragma unroll
  for (int c = 1; c < kBlocks; ++c) {
    start_h(c);
    tile_gemm<16, C, PREC, NP>(w, ff1(c).v, ff2(c - 1).v, a, h, xop, none);
    tile_gemm<16, C, PREC, NP>(w, ff2(c - 1).v, (c + 1 < kBlocks ? ff1(c + 1) : ff2(c)).v, a, acc, hop,
                             [&](int k) __attribute__((always_inline)) {
#pragma unroll
                               for (int v = k * C / 2; v < (k + 1) * C / 2; ++v) gelu_pair(v);
                             });
    lds_barrier();  // every wave has read block c - 1
    put_h();
  }
  tile_gemm<16, C, PREC, 0>(w, ff2(kBlocks - 1).v, out.v, a, acc, hop, none);
  if (OUTPROJ) put_ssq(acc, ssq, wave, j, hh);
  lds_barrier();
  store_tile<C, OUTPROJ>(acc, smem, ssq, eps, xres, nres, wave, lane);
}

namespace {
template <bool OUTPROJ>
void launch_block(const uint16_t* O, const uint8_t* layer, float* X, uint16_t* xn, int64_t n, int prec, float eps,
                  hipStream_t st, const LaunchEvents& ev) {
  const int C = token_tiles(n);
  const auto kernel =
      prec == kFfSplit  ? (C == 1 ? k_post_attn<1, OUTPROJ, kFfSplit> : k_post_attn<2, OUTPROJ, kFfSplit>)
      : prec == kFfFp16 ? (C == 1 ? k_post_attn<1, OUTPROJ, kFfFp16> : k_post_attn<2, OUTPROJ, kFfFp16>)
                        : (C == 1 ? k_post_attn<1, OUTPROJ, kFfBf16> : k_post_attn<2, OUTPROJ, kFfBf16>);
  hipExtLaunchKernelGGL(kernel, dim3(unsigned((n + 32 * C - 1) / (32 * C))), dim3(64 * kTileWaves), 0, st, ev.start,
                        ev.stop, 0, O, layer, X, xn, n, eps);
}
}  // namespace

void launch_post_attn(const uint16_t* O, const uint8_t* layer, float* X, uint16_t* xn, int64_t n, int ff_precision,
                      float eps, hipStream_t st, const LaunchEvents& ev) {
  launch_block<true>(O, layer, X, xn, n, ff_precision, eps, st, ev);
}

void launch_ff(const uint8_t* layer, float* X, int64_t n, int ff_precision, float eps, hipStream_t st) {
  launch_block<false>(nullptr, layer, X, nullptr, n, ff_precision, eps, st, LaunchEvents{});
}

}  // namespace trf
