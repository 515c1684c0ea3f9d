// Device code of the token-tile kernels (trf_kernels.hip, trf_qkv_attn_short.hip).
//
// A workgroup takes a tile of 32 C tokens (C = 1 or 2) and all output features: its 8 waves split the
// features (32-row weight tiles), and the tile's activations sit in LDS, where every wave reads them as MFMA
// operands.  A wave's weight tiles are its own, so they go from L2 straight into registers, kWeightAhead
// k-steps ahead of their MFMAs: nothing waits at a barrier for weights, and one 1 KB block feeds C MFMAs.
// What C and the register budget are chosen for: two workgroups of 8 waves per CU (at most 128 VGPRs and
// 80 KB of LDS each), so that one's memory phases and barriers run beside the other's matrix work.  The L2
// delivers ~50 bytes per cycle per CU, which bounds C = 1 (1.3 MB of weights per 32 tokens in the
// post-attention block); C = 4 fills a CU with one workgroup.  That block in us at C = 1 / 2 / 4: 18 / 24 /
// 45 at 6,262 tokens, 37 / 35 / 53 at 16,384, 223 / 172 / 225 at 105,462.  So a launch takes C = 1 while its
// 32-token tiles fit one per CU and C = 2 beyond (the residual GEMM's own rule is at its launch).  Between, us at
// C = 1 and 2, feed-forward in fp16: 23.1 and 19.8 at 8,246, 36.1 and 36.1 at 16,492, 54 and 44 at 30,194, 61 and 58
// at 32,984, 101 and 83 at 62,000; in split: 42 and 35 at 8,246, 70 and 77 at 16,492 (C = 2 has one workgroup a CU and
// starts its second round there), 102 and 90 at 30,194, 201 and 180 at 62,000; time QKV: 20 and 16 at 8,246, 31 and 27
// at 16,492, 45 and 33 at 30,194, 87 and 62 at 62,000.
//
// Rows of activations move in whole rows or half rows per wave instruction and are transposed through LDS.
// Loaded or stored in operand layout (32 rows x 16 bytes, the halves of a pair 32 lanes apart) an
// instruction occupies the CU's address path several times as long: the out-projection, residual and norm
// alone took 89 us at 105,462 tokens that way, 72 us through LDS (378 MB: the HBM rate of a copy).  Rows
// are held as 16-byte chunks, chunk c of token t at c ^ (t & 15): the 16 lanes of an LDS access then touch
// 16 different chunks of their 256 bytes.
#pragma once

#include "trf_device.h"

namespace trf {

constexpr int kTileWaves = 8;
constexpr int kWeightAhead = 4;  // k-steps a wave's weight blocks are loaded ahead (8 spills at C = 2)

__device__ __forceinline__ u32x4 buffer_load16(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// This wave's LDS operations have completed, then all waves meet; its global loads stay in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_waitcnt(0xC07F);  // vmcnt(63) expcnt(7) lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Everything this wave loads (direct-to-LDS loads too) has landed, then all waves meet.
__device__ __forceinline__ void loads_barrier() {
  __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) expcnt(7) lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Position of chunk c of token t in a tile of 1 KB rows.
__device__ __forceinline__ int row_chunk(int t, int c) { return t * 64 + (c ^ (t & 15)); }

// Operand products of the three feed-forward arithmetics (FfPrecision; split runs on bf16).
template <int PREC>
__device__ __forceinline__ f32x16 mfma_ff(u32x4 a, u32x4 b, f32x16 c) {
  return PREC == kFfFp16 ? mfma32h(a, b, c) : mfma32(a, b, c);
}
__host__ __device__ constexpr int ff_parts(int prec) { return prec == kFfSplit ? 2 : 1; }

// A wave's stream of weight blocks: k-step k of a GEMM is at offset off[part] + k KB of the layer.
struct TileWeights {
  __amdgpu_buffer_rsrc_t res;
  int lane16;
  __device__ __forceinline__ u32x4 load(int off) const { return buffer_load16(res, lane16, off); }
};
struct TileOff {
  int v[2];
};

// K-steps the activation operands are read ahead.
__host__ __device__ constexpr int tile_ahead(int C, int prec) { return C == 1 ? (prec == kFfSplit ? 2 : 4) : 1; }

// acc += W . B over KS k-steps (SWAP: B . W, tokens on the rows).  a holds the first kWeightAhead k-steps'
// blocks and is left with those of the next GEMM (at next[], NEXT parts; 0: there is none).  operand(k, part,
// ct) is the LDS operand.  side(k) is VALU work placed beside k-step k's MFMAs.
template <int KS, int C, int PREC, int NEXT, bool SWAP = false, int AHEAD = tile_ahead(C, PREC), typename Operand,
          typename Side>
__device__ __forceinline__ void tile_gemm(const TileWeights& w, const int (&off)[2], const int (&next)[2],
                                          u32x4 (&a)[kWeightAhead][2], f32x16 (&acc)[C], Operand&& operand,
                                          Side&& side) {
  constexpr int NP = ff_parts(PREC);
  u32x4 b[AHEAD + 1][NP][C];
  auto read = [&](int k) __attribute__((always_inline)) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int ct = 0; ct < C; ++ct) b[k % (AHEAD + 1)][p][ct] = operand(k, p, ct);
  };
#pragma unroll
  for (int k = 0; k < AHEAD; ++k) read(k);
#pragma unroll
  for (int k = 0; k < KS; ++k) {
    if (k + AHEAD < KS) read(k + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 (&ak)[2] = a[k % kWeightAhead];
    u32x4 (&bk)[NP][C] = b[k % (AHEAD + 1)];
#pragma unroll
    for (int ct = 0; ct < C; ++ct)
      acc[ct] = SWAP ? mfma_ff<PREC>(bk[0][ct], ak[0], acc[ct]) : mfma_ff<PREC>(ak[0], bk[0][ct], acc[ct]);
    if constexpr (NP == 2) {
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = mfma_ff<PREC>(ak[0], bk[1][ct], acc[ct]);
#pragma unroll
      for (int ct = 0; ct < C; ++ct) acc[ct] = mfma_ff<PREC>(ak[1], bk[0][ct], acc[ct]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      if (k + kWeightAhead < KS) {
        if (p < NP) ak[p] = w.load(off[p] + (k + kWeightAhead) * kTileBytes);
      } else if (p < NEXT) {
        ak[p] = w.load(next[p] + (k + kWeightAhead - KS) * kTileBytes);
      }
    }
    side(k);
    __builtin_amdgcn_sched_barrier(0);
  }
  // The products end here: without this the compiler may sink the whole MFMA chain, whose only readers come
  // later, past the next barrier, and keep every operand in scratch until then.
#pragma unroll
  for (int ct = 0; ct < C; ++ct) asm volatile("" : "+v"(acc[ct])::"memory");
}

// ---------------------------------------------------------------- projections of a tile of positions
constexpr int kRopeChunks = 16;  // 16-byte chunks of a position's [cos | sin] row (64 floats)

// xn of positions p0 .. p0 + 32C - 1 of sequence s, on its way to LDS as operand blocks [ct][k-step][lane]
// (lane (j, hh): features 16k + 8hh .. +7 of row 32 ct + j); positions past L take the last one's.  A wave
// instruction takes 4 chunks of 16 rows: 64-byte runs of global memory, 4-way conflicts in LDS.
template <int C, int NW = kTileWaves>
struct TilePositions {
  static constexpr int N = kTileWaves / NW;  // quads of chunks a wave takes: chunks 4 (w + NW i) .. +3
  u32x4 x[2 * C][N];
  __device__ __forceinline__ void load(const uint16_t* __restrict__ xn, int mode, int s, int p0, int L, int T, int F) {
    const int t4 = (threadIdx.x & 63) >> 2, c4 = 4 * (threadIdx.x >> 6) + (threadIdx.x & 3);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i) {
      const u32x4* const row =
          reinterpret_cast<const u32x4*>(xn + token_of(mode, s, min(p0 + 16 * i + t4, L - 1), T, F) * kDim);
#pragma unroll
      for (int k = 0; k < N; ++k) x[i][k] = row[c4 + 4 * NW * k];
    }
  }
  __device__ __forceinline__ void put(u32x4* xb) const {
    const int t4 = (threadIdx.x & 63) >> 2, c4 = 4 * (threadIdx.x >> 6) + (threadIdx.x & 3);
#pragma unroll
    for (int i = 0; i < 2 * C; ++i)
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int c = c4 + 4 * NW * k;
        xb[((i >> 1) * 16 + (c >> 1)) * 64 + 32 * (c & 1) + 16 * (i & 1) + t4] = x[i][k];
      }
  }
};

// [cos | sin] rows (chunk c of row t at c ^ (t & 15)) of positions p0 .. p0 + 32C - 1 into LDS.
template <int C, int NW = kTileWaves>
__device__ __forceinline__ void stage_rope(const float* __restrict__ rope, int p0, int L, u32x4* rrows) {
  constexpr int R = 32 * C, NT = 64 * NW;
  const u32x4* const rp = reinterpret_cast<const u32x4*>(rope);
#pragma unroll
  for (int i = 0; i < R * kRopeChunks / NT; ++i) {  // the table is [cos | sin][L][8 chunks]
    const int q = i * NT + threadIdx.x, t = q >> 4, c = q & 15;
    rrows[t * kRopeChunks + (c ^ (t & 15))] = rp[(int64_t(c >> 3) * L + min(p0 + t, L - 1)) * 8 + (c & 7)];
  }
}

// Register group g (features 8g + 4hh .. +3 of head half `half`) of position t, rotated in fp32, scaled and
// packed: the interleaved pairs are i = 16 half + 4g + 2hh + {0, 1}, in chunk 4 half + g of the cos and of
// the sin row.
__device__ __forceinline__ u32x2 rotate_group(const f32x16& a, int g, const u32x4* rrows, int t, int half, int hh,
                                              float scale) {
  const float2* const row = reinterpret_cast<const float2*>(rrows + t * kRopeChunks);
  const float2 c = row[2 * ((4 * half + g) ^ (t & 15)) + hh], sn = row[2 * ((8 + 4 * half + g) ^ (t & 15)) + hh];
  const float a0 = a[4 * g], a1 = a[4 * g + 1], a2 = a[4 * g + 2], a3 = a[4 * g + 3];
  return u32x2{pk_bf16(fmaf(a0, c.x, -(a1 * sn.x)) * scale, fmaf(a1, c.x, a0 * sn.x) * scale),
               pk_bf16(fmaf(a2, c.y, -(a3 * sn.y)) * scale, fmaf(a3, c.y, a2 * sn.y) * scale)};
}

// The half-waves' parts (features 8g + 4hh .. +3) of register groups 2q (lo) and 2q + 1 (hi) of a position
// joined into 16-byte chunks: lane (j, 0) gets chunk 2q, lane (j, 1) chunk 2q + 1.
__device__ __forceinline__ u32x4 join_halves(u32x2 lo, u32x2 hi) {
  const auto x = __builtin_amdgcn_permlane32_swap(lo[0], hi[0], false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(lo[1], hi[1], false, false);
  return u32x4{x[0], y[0], x[1], y[1]};
}

// This wave's share of the gate tile's 16 k-steps (operand blocks ag; rows 0..7 live in register group 0 of
// both half-waves) as partial sums [wave][position][head].
template <int C, int NW = kTileWaves>
__device__ __forceinline__ void gate_partials(const u32x4 (&ag)[16 / NW], const u32x4* xb, float* part, int wave,
                                              int lane) {
  const int j = lane & 31, hh = lane >> 5;
#pragma unroll
  for (int ct = 0; ct < C; ++ct) {
    f32x16 acc = zero16();
#pragma unroll
    for (int i = 0; i < 16 / NW; ++i) acc = mfma32(ag[i], xb[(ct * 16 + 16 / NW * wave + i) * 64 + lane], acc);
    *reinterpret_cast<f32x4*>(part + (wave * 32 * C + 32 * ct + j) * kHeads + 4 * hh) =
        f32x4{acc[0], acc[1], acc[2], acc[3]};
  }
}

// The sigmoid gate of a head and position, once every wave's partial sums are there.
template <int C, int NW = kTileWaves>
__device__ __forceinline__ float gate_of(const float* part, int p, int head, const float* __restrict__ bgate) {
  float g = part[p * kHeads + head];
#pragma unroll
  for (int w = 1; w < NW; ++w) g += part[(w * 32 * C + p) * kHeads + head];
  return 1.0f / (1.0f + expf(-(g + bgate[head])));
}

}  // namespace trf
