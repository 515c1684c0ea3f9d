// Fused QKV GEMM + rotary + gates + exact softmax attention for sequences of at most 64 positions
// (frequency attention: the 62 bands of one frame), so that Q, K, V and the gates never leave the chip.
// It replaces the pair qkv_rope_gemm -> attention of the reference (kernels.cpp:439-540, 250-388) for
// short sequences, with the same arithmetic: fp32 accumulators, fp32 rotary, q times log2(e) before its
// bf16 rounding, bf16 q, k, v and unnormalised P, the exact row max over the valid keys, an fp32 sum of
// e = 2^(s - m), and O = (P.V) * gate / sum rounded to bf16 in token order.
//
// A workgroup is 4 heads of one sequence after another, padded to 32 C positions (C = 1 up to 32 positions,
// else 2), and a wave is one head from its projections to its output (trf_tiles.h has the staging and the
// weight streaming).  The waves meet twice per sequence, when its xn rows are in LDS and before the next
// one's replace them; in between each runs on its own, so that one wave's rotary, softmax and packing run
// under another's MFMAs.  The next sequence's xn is loaded during the attention.  At C = 2 a wave holds the q,
// k and v operands of 64 positions (96 registers): two workgroups a CU, two waves a SIMD.
//
// No data crosses lanes between the projection and the attention:
//   * q and k come out of C = W . xn^T with lane (j, hh) holding token j of the column tile and features
//     8g + 4hh + r.  Packed to bf16 in that "register order", q is the B operand (Q^T) and k the A
//     operand (K) of S^T = K . Q^T: both use the same permutation of the 16 head features of a k-step,
//     which leaves the dot products unchanged.
//   * v comes out of the swapped product C = xn . W_v^T (the xn rows are the A operand, the packed W_v
//     block the B operand), so lane (j, hh) holds feature j of tokens 8g + 4hh + r: exactly the A operand
//     (V^T) of O^T = V^T . P^T with the keys of a k-step in the register order in which the S^T accumulator
//     holds them, so P^T is the B operand straight from the accumulator.
// The row max and the row sum combine the two half-waves (the query's keys sit in lanes j and j + 32).
// O leaves through the wave's own LDS rows as whole 128-byte lines.
//
// Against workgroups of 4 sequences that streamed the weights through LDS and exchanged K and V^T between
// position halves (us): 62 positions, 251 sequences 35 and 23; 101 sequences 19.5 and 17; 1701 the same within 3%
// (264k cycles and 250k, at a lower clock).  At 1701 the MFMA pipe is busy 39%, the address units 50%, LDS 35% of the
// time, 11% of the cycles go to the bank conflicts of staging xn, and C = 2 keeps 12 registers in scratch; 8 weight
// k-steps ahead instead of 4, and 8 heads a workgroup instead of 4, changed nothing there.
#include "trf_tiles.h"

namespace trf {

constexpr int kFsDropped = kFusedShortDropped;  // buffer offset past any sequence's output: the store is dropped

// Key (or token) of register R of half-wave hh in a 32-row accumulator tile: row 8(R/4) + 4hh + R%4.
__device__ __forceinline__ int acc_row(int R, int hh) { return 8 * (R >> 2) + 4 * hh + (R & 3); }

// Two k-steps' operands from a tile's accumulators, in register order.
__device__ __forceinline__ void pack_tile(const f32x16& v, u32x4 (&out)[2]) {
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
    out[kk] = u32x4{pk_bf16(v[8 * kk], v[8 * kk + 1]), pk_bf16(v[8 * kk + 2], v[8 * kk + 3]),
                    pk_bf16(v[8 * kk + 4], v[8 * kk + 5]), pk_bf16(v[8 * kk + 6], v[8 * kk + 7])};
}

// The operands are formed here, before the next tile's products: left to itself the compiler forms them where
// they are read, and keeps the fp32 tiles until then.
__device__ __forceinline__ void pin(u32x4 (&v)[2]) { asm volatile("" : "+v"(v[0]), "+v"(v[1])::"memory"); }

constexpr int kFsWaves = 4;  // one head each

template <int C>
__global__ __launch_bounds__(64 * kFsWaves, 2) void k_qkv_attn_short(
    const uint16_t* __restrict__ xn, const uint8_t* __restrict__ layer, const float* __restrict__ rope, int mode,
    int nseq, int L, int T, int F, uint16_t* __restrict__ O) {
  constexpr int R = 32 * C;
  constexpr int kRope = R * 32, kGate = kRope + R * kRopeChunks, kOut = kGate + kFsWaves * R * kHeads / 4;
  __shared__ u32x4 smem[kOut + kFsWaves * 32 * 8];  // xn, cos | sin, partial gates, 32 output rows a wave
  float* const gates = reinterpret_cast<float*>(smem + kGate);
  const int lane = threadIdx.x & 63, wave = wave_id();
  const int j = lane & 31, hh = lane >> 5, h = kFsWaves * (blockIdx.x & 1) + wave;
  const TileWeights w{buffer_rsrc(layer, int(kLayerBytes)), lane * 16};
  auto tile = [&](int kind, int half) __attribute__((always_inline)) {  // kind 0 q, 1 k, 2 v
    return TileOff{{int(kOffQkvg) + (16 * kind + 2 * h + half) * 16 * kTileBytes, 0}};
  };
  auto xop = [&](int k, int, int ct) __attribute__((always_inline)) { return smem[(ct * 16 + k) * 64 + lane]; };
  auto none = [](int) __attribute__((always_inline)) {};
  const int stride = mode == 0 ? F : 1;  // tokens between positions
  u32x4* const os = smem + kOut + wave * 32 * 8;
  TilePositions<C, kFsWaves> x;
  x.load(xn, mode, blockIdx.x >> 1, 0, L, T, F);
  u32x4 a[kWeightAhead][2], ag[16 / kFsWaves];
#pragma unroll
  for (int i = 0; i < 16 / kFsWaves; ++i)
    ag[i] = w.load(int(kOffQkvg) + ((kQkvgTiles - 1) * 16 + 16 / kFsWaves * wave + i) * kTileBytes);
#pragma unroll
  for (int i = 0; i < kWeightAhead; ++i) a[i][0] = w.load(tile(2, 0).v[0] + i * kTileBytes);
  stage_rope<C, kFsWaves>(rope, 0, L, smem + kRope);
#pragma unroll 1
  for (int s = blockIdx.x >> 1; s < nseq; s += gridDim.x >> 1) {
    x.put(smem);
    lds_barrier();
    gate_partials<C, kFsWaves>(ag, smem, gates, wave, lane);
    u32x4 vb[2][C][2], kb[2][C][2], qb[2][C][2];  // [head half][position tile][k-step]
#pragma unroll
    for (int i = 0; i < 6; ++i) {  // the v, k and q tiles; the last one's next is the next sequence's first
      const int kind = 2 - i / 2, half = i & 1;
      const TileOff off = tile(kind, half), next = i == 5 ? tile(2, 0) : half ? tile(kind - 1, 0) : tile(kind, 1);
      f32x16 acc[C];
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = zero16();
      if (kind == 2)
        tile_gemm<16, C, kFfBf16, 1, true, 1>(w, off.v, next.v, a, acc, xop, none);
      else
        tile_gemm<16, C, kFfBf16, 1, false, 1>(w, off.v, next.v, a, acc, xop, none);
#pragma unroll
      for (int ct = 0; ct < C; ++ct) {
        if (kind == 2) {
          pack_tile(acc[ct], vb[half][ct]);
          pin(vb[half][ct]);
          continue;
        }
        u32x4 (&out)[2] = kind == 1 ? kb[half][ct] : qb[half][ct];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const u32x2 o = rotate_group(acc[ct], g, smem + kRope, 32 * ct + j, half, hh, kind == 1 ? 1.0f : kLog2e);
          out[g >> 1][2 * (g & 1)] = o[0];
          out[g >> 1][2 * (g & 1) + 1] = o[1];
        }
        pin(out);
      }
    }
    lds_barrier();  // the partial gates are there, and every wave has read xn
    if (s + int(gridDim.x >> 1) < nseq) x.load(xn, mode, s + (gridDim.x >> 1), 0, L, T, F);
    const auto ores = buffer_rsrc(O + token_of(mode, s, 0, T, F) * (kHeads * kHeadDim),
                                  ((L - 1) * stride + 1) * kHeads * kHeadDim * 2);
#pragma unroll
    for (int qt = 0; qt < C; ++qt) {
      f32x16 sacc[C];
#pragma unroll
      for (int kt = 0; kt < C; ++kt) {
        sacc[kt] = zero16();
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) sacc[kt] = mfma32(kb[half][kt][kk], qb[half][qt][kk], sacc[kt]);
      }
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < C; ++kt) {
        if (32 * kt + 32 <= L) {  // a key tile with no padded keys (uniform): no masking
#pragma unroll
          for (int r = 0; r < 16; r += 2) mx = fmaxf(fmaxf(mx, sacc[kt][r]), sacc[kt][r + 1]);
        } else {
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * kt + acc_row(r, hh) < L) mx = fmaxf(mx, sacc[kt][r]);
        }
      }
      const float m = halfwave_max(mx);
      float lsum = 0.f;
      f32x16 o[2] = {zero16(), zero16()};
#pragma unroll
      for (int kt = 0; kt < C; ++kt) {
        f32x16 e;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const bool in = 32 * kt + 32 <= L || 32 * kt + acc_row(r, hh) < L;
          e[r] = in ? __builtin_amdgcn_exp2f(sacc[kt][r] - m) : 0.f;
          lsum += e[r];
        }
        u32x4 pb[2];
        pack_tile(e, pb);
#pragma unroll
        for (int dt = 0; dt < 2; ++dt)
#pragma unroll
          for (int kk = 0; kk < 2; ++kk) o[dt] = mfma32(vb[dt][kt][kk], pb[kk], o[dt]);
      }
      const float sc = gate_of<C, kFsWaves>(gates, 32 * qt + j, h, reinterpret_cast<const float*>(layer + kOffBgate)) *
                       (1.0f / (lsum + __shfl_xor(lsum, 32)));
      // rows of 8 chunks (the head's 64 features), chunk c of row t at c ^ (t & 7)
#pragma unroll
      for (int dt = 0; dt < 2; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          reinterpret_cast<u32x2*>(os)[2 * (j * 8 + ((4 * dt + g) ^ (j & 7))) + hh] =
              u32x2{pk_bf16(o[dt][4 * g] * sc, o[dt][4 * g + 1] * sc),
                    pk_bf16(o[dt][4 * g + 2] * sc, o[dt][4 * g + 3] * sc)};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 8 * i + (lane >> 3), c = lane & 7, p = 32 * qt + t;
        const int off = p < L ? p * stride * (kHeads * kHeadDim * 2) + h * (kHeadDim * 2) + 16 * c : kFsDropped;
        __builtin_amdgcn_raw_buffer_store_b128(os[t * 8 + (c ^ (t & 7))], ores, off, 0, 0);
      }
    }
  }
}

void launch_qkv_attn_short(const uint16_t* xn, const uint8_t* layer, const float* rope, const SeqShape& sh,
                           uint16_t* O, hipStream_t st, const LaunchEvents& ev) {
  if (sh.nseq <= 0) return;
  const int C = sh.L <= 32 ? 1 : 2;
  const int slots = device_cu_count() * (C == 1 ? 2 : 1);  // sequences the device holds
  const auto kernel = C == 1 ? k_qkv_attn_short<1> : k_qkv_attn_short<2>;
  hipExtLaunchKernelGGL(kernel, dim3(2u * unsigned(sh.nseq < slots ? sh.nseq : slots)), dim3(64 * kFsWaves), 0, st,
                        ev.start, ev.stop, 0, xn, layer, rope, sh.mode, sh.nseq, sh.L, sh.T, sh.F, O);
}

}  // namespace trf
