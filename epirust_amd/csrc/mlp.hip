// Surrogate MLP kernels for gfx950: bf16 operands on MFMA with FP32 accumulation.
//
// k_gemm: C[M x N] = A[M x K] * B[K x N] with arbitrary element strides (epi_gemm_bf16), a
// 64x64 block tile, BK = 32, four 64-lane waves each owning a 32x32 sub-tile computed with
// v_mfma_f32_32x32x16_bf16 (gfx950; A and B staged through LDS as 16-byte vectors, two
// buffers, the next tile prefetched into registers during the current one's MFMAs).
//
// k_mlp_stage: the network's products, whose operands the stages before wrote in the layout
// this one reads (every bf16 matrix by rows and transposed, k contiguous, zero-padded), with
// bias, GELU, loss, GELU' or the Adam step as epilogues. A forward pass is one stage per
// layer and a backward pass one stage per layer: the input gradient of layer l goes with the
// weight and bias gradients of layer l + 1. A training step of the 9 -> 4 x 512 -> 600
// network at 512 samples is 11 launches instead of 34.
//
// v_mfma_f32_32x32x16_bf16 lane layout (64 lanes, wave64):
//   A (32x16): lane l holds row l%32, k = 8*(l/32) .. +7 (eight bf16 in 128 bits)
//   B (16x32): lane l holds col l%32, k = 8*(l/32) .. +7
//   D (32x32, 16 floats / lane): lane l, element r -> row 8*(r/4) + 4*(l/32) + r%4, col l%32
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "mlp.hpp"

namespace epi {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kBM = 64, kBN = 64, kBK = 32;
constexpr int kLdsK = kBK + 8;  // LDS row: kBK k of one m (or n) plus 8 of padding
constexpr int kChunks = kBK / 8;  // 16-byte vectors per tile row along k
constexpr int kVecs = kBM * kBK / (256 * 8);  // 16-byte vectors per thread per operand tile

// How one 64 x kBK operand tile (rows r = m or n, columns k) is read from global memory.
enum : int { TILE_K_CONTIG = 0, TILE_R_CONTIG = 1, TILE_ELEMENT = 2 };

// Element (r, k) of an operand is X[r * ld_r + k * ld_k]. A whole tile inside the matrix
// whose contiguous dimension is 16-byte aligned is read as 16-byte vectors (kVecs of 8
// bf16 per thread, 256 threads): along k (ld_k == 1) or along r (ld_r == 1). Otherwise, at
// ragged edges or odd strides, element by element with bounds checks.
__device__ __forceinline__ int tile_mode(const uint16_t* X, int64_t ld_r, int64_t ld_k, int r0, int k0, int R,
                                         int K) {
  const bool full = r0 + 64 <= R && k0 + kBK <= K;
  const bool aligned = (reinterpret_cast<uintptr_t>(X) & 15u) == 0;
  if (full && aligned && ld_k == 1 && (ld_r & 7) == 0) return TILE_K_CONTIG;
  if (full && aligned && ld_r == 1 && (ld_k & 7) == 0) return TILE_R_CONTIG;
  return TILE_ELEMENT;
}

// Vector e (e = tid + 256 i, i < kVecs) of a tile: along k, row e / kChunks with k
// (e % kChunks) * 8 .. +7; along r, k e / 8 with rows (e % 8) * 8 .. +7.
struct TileRegs {
  u16x8 v[kVecs];
};

__device__ __forceinline__ void load_tile(TileRegs& t, const uint16_t* X, int64_t ld_r, int64_t ld_k, int r0,
                                          int k0, int R, int K, int mode, int tid) {
  if (mode == TILE_K_CONTIG) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int e = tid + 256 * i;
      t.v[i] = *reinterpret_cast<const u16x8*>(X + static_cast<int64_t>(r0 + e / kChunks) * ld_r + k0 + (e % kChunks) * 8);
    }
  } else if (mode == TILE_R_CONTIG) {
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      const int e = tid + 256 * i;
      t.v[i] = *reinterpret_cast<const u16x8*>(X + static_cast<int64_t>(k0 + (e >> 3)) * ld_k + r0 + (e & 7) * 8);
    }
  } else {  // ragged edges and odd strides: the along-k assignment, element by element
#pragma unroll 1
    for (int i = 0; i < kVecs; ++i) {
      const int e = tid + 256 * i;
      const int r = r0 + e / kChunks, kb = k0 + (e % kChunks) * 8;
      u16x8 v;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int k = kb + q;
        v[q] = (r < R && k < K) ? X[static_cast<int64_t>(r) * ld_r + static_cast<int64_t>(k) * ld_k] : 0;
      }
      t.v[i] = v;
    }
  }
}

// LDS tile s[r][k] (k contiguous): 16-byte stores, or 2-byte stores for a tile read
// along r.
__device__ __forceinline__ void store_tile(uint16_t (*s)[kLdsK], const TileRegs& t, int mode, int tid) {
#pragma unroll
  for (int i = 0; i < kVecs; ++i) {
    const int e = tid + 256 * i;
    if (mode == TILE_R_CONTIG) {
      const int k = e >> 3, rb = (e & 7) * 8;
#pragma unroll
      for (int q = 0; q < 8; ++q) s[rb + q][k] = t.v[i][q];
    } else {
      *reinterpret_cast<u16x8*>(&s[e / kChunks][(e % kChunks) * 8]) = t.v[i];
    }
  }
}

// fp32 -> bf16, round to nearest even (NaN kept quiet).
__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u && (u & 0x007FFFFFu)) return static_cast<uint16_t>((u >> 16) | 0x40u);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return static_cast<uint16_t>(u >> 16);
}

// GELU, tanh form: 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3)))
__device__ __forceinline__ float gelu(float x) {
  const float u = 0.7978845608028654f * (x + 0.044715f * x * x * x);
  return 0.5f * x * (1.0f + tanhf(u));
}
__device__ __forceinline__ float gelu_grad(float x) {
  const float x2 = x * x;
  const float u = 0.7978845608028654f * (x + 0.044715f * x2 * x);
  const float t = tanhf(u);
  const float du = 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x2);
  return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * du;
}

// C tile 64 x 64 per block of four wave64s (2 x 2), each a 32 x 32 sub-tile accumulated
// with v_mfma_f32_32x32x16_bf16 (gfx950): per kBK-wide k step, kBK / 16 MFMAs whose A operand is
// row (lane % 32) with k 8 * (lane / 32) .. +7, read from LDS as one 16-byte vector, and B
// likewise by column. The next k tile's global loads are issued before the current one's
// MFMAs (register prefetch), into the other of two LDS buffers, so each k step has one
// barrier.
__global__ __launch_bounds__(256) void k_gemm(GemmArgs g) {
  __shared__ __align__(16) uint16_t sA[2][kBM][kLdsK];
  __shared__ __align__(16) uint16_t sB[2][kBN][kLdsK];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.y * kBM, n0 = blockIdx.x * kBN;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  f32x16 acc = {0};

  int ma = tile_mode(g.A, g.lda_m, g.lda_k, m0, 0, g.M, g.K);
  int mb = tile_mode(g.B, g.ldb_n, g.ldb_k, n0, 0, g.N, g.K);
  TileRegs va, vb;
  load_tile(va, g.A, g.lda_m, g.lda_k, m0, 0, g.M, g.K, ma, tid);
  load_tile(vb, g.B, g.ldb_n, g.ldb_k, n0, 0, g.N, g.K, mb, tid);
  int buf = 0;
  for (int k0 = 0; k0 < g.K; k0 += kBK) {
    store_tile(sA[buf], va, ma, tid);
    store_tile(sB[buf], vb, mb, tid);
    __syncthreads();
    const int k1 = k0 + kBK;
    if (k1 < g.K) {  // uniform: prefetch the next tile while this one is multiplied
      ma = tile_mode(g.A, g.lda_m, g.lda_k, m0, k1, g.M, g.K);
      mb = tile_mode(g.B, g.ldb_n, g.ldb_k, n0, k1, g.N, g.K);
      load_tile(va, g.A, g.lda_m, g.lda_k, m0, k1, g.M, g.K, ma, tid);
      load_tile(vb, g.B, g.ldb_n, g.ldb_k, n0, k1, g.N, g.K, mb, tid);
    }
#pragma unroll
    for (int kk = 0; kk < kBK; kk += 16) {
      const int kq = kk + 8 * (lane >> 5);
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(&sA[buf][wm + (lane & 31)][kq]);
      const bf16x8 b = *reinterpret_cast<const bf16x8*>(&sB[buf][wn + (lane & 31)][kq]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
    }
    buf ^= 1;
  }
  const int col = n0 + wn + (lane & 31);
  if (col >= g.N) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int row = m0 + wm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    if (row < g.M) g.C[static_cast<int64_t>(row) * g.N + col] = acc[r];
  }
}

// ---- the network's stages

// A block's LDS: MFMA operand fragments of 16 k (one row or column per half wave, 1 KiB each),
// or a chunk of a bias gradient's rows. Four blocks' 38 KiB fit a CU's LDS.
constexpr int kFrag = 512;  // bf16 values of a fragment
constexpr int kArenaFrags = 38;

// Products of a TILES x TILES square of 32 x 32 tiles per block of four waves, each element's
// k added in order, 16 at a time. Both operands are stored with k contiguous, so a fragment
// is one 16-byte load per lane, straight into LDS in the order the MFMA reads it; all the
// loads of a pass (38 steps for one tile, 19 for four) are in flight before the one wait for
// them. One tile: its chain of MFMAs runs on the first wave, which is as fast as that chain
// can be, and the four waves share the loads and the epilogue. Four tiles: one per wave, each
// fragment read from memory once for two of them.
template <int TILES>
__device__ __forceinline__ f32x16 block_product(const MlpJob& g, int m0, int n0, uint16_t* arena) {
  constexpr int kPerStep = 2 * TILES;  // fragments: A's row tiles, then B's column tiles
  constexpr int kSteps = kArenaFrags / kPerStep;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 31, kq = 8 * (lane >> 5);
  const int wm = TILES == 1 ? 0 : wave >> 1, wn = TILES == 1 ? 0 : wave & 1;
  const int steps = (g.K + 15) >> 4;
  f32x16 acc = {};
  for (int s0 = 0; s0 < steps; s0 += kSteps) {
    const int n = min(kSteps, steps - s0);
    if (s0) __syncthreads();
    for (int f = wave; f < n * kPerStep; f += 4) {
      const int s = f / kPerStep, t = f % kPerStep;
      const uint16_t* p = t < TILES ? g.A + static_cast<int64_t>(m0 + 32 * t + r) * g.lda
                                    : g.Bt + static_cast<int64_t>(n0 + 32 * (t - TILES) + r) * g.ldb;
      p += 16 * (s0 + s) + kq;
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)p,
                                       (__attribute__((address_space(3))) void*)(arena + f * kFrag), 16, 0, 0);
    }
    __syncthreads();
    if (TILES > 1 || wave == 0) {
      for (int s = 0; s < n; ++s) {
        const uint16_t* f = arena + s * kPerStep * kFrag + lane * 8;
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(f + wm * kFrag);
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(f + (TILES + wn) * kFrag);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
      }
    }
  }
  return acc;
}

// Adam (Kingma & Ba) on one fp32 master parameter. The fused multiply-adds are written out:
// which product the compiler would fuse depends on the code around it.
__device__ __forceinline__ float adam_step(const AdamArgs& a, float g, float w, float& m, float& v) {
  const float mi = fmaf(1.0f - a.b1, g, a.b1 * m);
  const float vi = fmaf((1.0f - a.b2) * g, g, a.b2 * v);
  m = mi;
  v = vi;
  const float upd = a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  return w - upd;
}

// Four values of one column, rows row .. row + 3, to a transposed bf16 matrix.
__device__ __forceinline__ void store_col(uint16_t* t, int ld, int row, int col, const uint16_t (&h)[4]) {
  *reinterpret_cast<ushort4*>(t + static_cast<int64_t>(col) * ld + row) = make_ushort4(h[0], h[1], h[2], h[3]);
}

// What the job does with four products of one column, rows row0 .. row0 + 3 (a register quad
// of an MFMA tile), so the transpose is written 8 bytes at a time. Rows past M are zero in
// the transpose: it is a later product's k padding. Returns their part of the loss.
template <int KIND, bool WHOLE>
__device__ __forceinline__ float finish_rows(const MlpJob& g, const AdamArgs& ad, int row0, int col,
                                             const float (&acc)[4]) {
  const float bias = KIND == MLP_HIDDEN || KIND == MLP_OUTPUT || KIND == MLP_LOSS ? g.bias[col] : 0.0f;
  float in0[4], in1[4], in2[4];  // what the epilogue reads, all of it in flight together
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int64_t o = static_cast<int64_t>(WHOLE ? row0 + i : min(row0 + i, g.M - 1)) * g.N + col;
    if constexpr (KIND == MLP_LOSS) in0[i] = g.t[o];
    if constexpr (KIND == MLP_INPUT_GRAD) in0[i] = g.z[o];
    if constexpr (KIND == MLP_WEIGHT_GRAD)
      if (g.adam) {  // uniform
        in0[i] = g.w[o];
        in1[i] = g.m[o];
        in2[i] = g.v[o];
      }
  }
  float loss = 0.0f;
  uint16_t h[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = row0 + i;
    const int64_t o = static_cast<int64_t>(row) * g.N + col;
    h[i] = 0;
    if (!WHOLE && row >= g.M) continue;
    float out = acc[i];
    if constexpr (KIND == MLP_HIDDEN) {
      const float z = acc[i] + bias;
      if (g.c) g.c[o] = z;  // uniform
      out = gelu(z);
    } else if constexpr (KIND == MLP_OUTPUT) {
      g.c[o] = acc[i] + bias;
    } else if constexpr (KIND == MLP_LOSS) {
      const float d = (acc[i] + bias) - in0[i];
      loss += d * d;
      out = 2.0f * d * g.inv_count;
      g.c[o] = out;
    } else if constexpr (KIND == MLP_INPUT_GRAD) {
      out = acc[i] * gelu_grad(in0[i]);
      g.c[o] = out;
    } else if (g.adam) {
      out = adam_step(ad, acc[i], in0[i], in1[i], in2[i]);
      g.w[o] = out;
      g.m[o] = in1[i];
      g.v[o] = in2[i];
    } else {
      g.c[o] = out;
    }
    if (KIND != MLP_OUTPUT && g.row) {  // uniform
      h[i] = to_bf16(out);
      g.row[static_cast<int64_t>(row) * g.ld_row + col] = h[i];
    }
  }
  if (KIND != MLP_OUTPUT && g.col) store_col(g.col, g.ld_col, row0, col, h);  // uniform
  return loss;
}

template <int KIND>
__device__ __forceinline__ float finish_kind(const MlpJob& g, const AdamArgs& ad, int row0, int col,
                                             const float (&acc)[4]) {
  return row0 + 4 <= g.M ? finish_rows<KIND, true>(g, ad, row0, col, acc)
                         : finish_rows<KIND, false>(g, ad, row0, col, acc);
}

__device__ __forceinline__ float finish_quad(const MlpJob& g, const AdamArgs& ad, int row0, int col,
                                             const float (&acc)[4]) {
  switch (g.kind) {  // uniform
    case MLP_HIDDEN: return finish_kind<MLP_HIDDEN>(g, ad, row0, col, acc);
    case MLP_OUTPUT: return finish_kind<MLP_OUTPUT>(g, ad, row0, col, acc);
    case MLP_LOSS: return finish_kind<MLP_LOSS>(g, ad, row0, col, acc);
    case MLP_INPUT_GRAD: return finish_kind<MLP_INPUT_GRAD>(g, ad, row0, col, acc);
    default: return finish_kind<MLP_WEIGHT_GRAD>(g, ad, row0, col, acc);
  }
}

// Bias gradients of kSumCols columns: each column's rows added in order, as the block fetches
// kSumRows rows at a time into LDS, the next rows' loads in flight while lane c adds column
// c. What bounds it is that chain of dependent adds and a chunk's load latency.
constexpr int kSumCols = 8, kSumRows = 512, kSumStep = 256 / kSumCols, kSumLoads = kSumRows / kSumStep;
static_assert(kSumCols * kSumRows * 4 <= kArenaFrags * kFrag * 2, "a chunk of bias gradient rows fits the arena");
__device__ __forceinline__ void bias_grad(const MlpJob& g, const AdamArgs& ad, int n0, float* s) {
  const int c = threadIdx.x % kSumCols, r0 = threadIdx.x / kSumCols, n = n0 + c;
  float v[kSumLoads];
  const auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < kSumLoads; ++i) {
      const int k = k0 + r0 + i * kSumStep;
      v[i] = (n < g.N && k < g.K) ? g.z[static_cast<int64_t>(k) * g.N + n] : 0.0f;
    }
  };
  float sum = 0.0f;
  fetch(0);
  for (int k0 = 0; k0 < g.K; k0 += kSumRows) {
#pragma unroll
    for (int i = 0; i < kSumLoads; ++i) s[(r0 + i * kSumStep) * kSumCols + c] = v[i];
    __syncthreads();
    if (k0 + kSumRows < g.K) fetch(k0 + kSumRows);  // uniform
    if (threadIdx.x < kSumCols) {
      const int rows = min(kSumRows, g.K - k0);
#pragma unroll 16
      for (int r = 0; r < rows; ++r) sum += s[r * kSumCols + c];
    }
    __syncthreads();
  }
  if (threadIdx.x >= kSumCols || n >= g.N) return;
  if (g.adam) {
    float m = g.m[n], q = g.v[n];
    g.w[n] = adam_step(ad, sum, g.w[n], m, q);
    g.m[n] = m;
    g.v[n] = q;
  } else {
    g.c[n] = sum;
  }
}

// One block per TILES x TILES tiles (or per kSumCols bias columns); the stage's jobs follow
// one another in the grid. At the surrogate's shapes (512 x 512 outputs, 512 samples) a job is
// 256 blocks, one per CU, and the time is a launch plus a few memory latencies, so products
// are joined to what consumes them and to each other rather than tiled for reuse: 6.6 us a
// hidden layer forward (17 us and 64 blocks with an LDS-tiled product), 7.2 us an input
// gradient with its GELU' (17 + 4.7), 11 us with the next layer's weight and bias gradients
// and Adam (17 + 15 + 2 x 4.7 more).
template <int TILES>
__global__ __launch_bounds__(256) void k_mlp_stage(MlpStage st) {
  __shared__ __align__(16) uint16_t arena[kArenaFrags * kFrag];
  __shared__ float s_loss[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int j = 0;
  while (j + 1 < kMlpJobs && blockIdx.x >= st.begin[j + 1]) ++j;  // uniform
  const MlpJob& g = st.job[j];
  const int b = static_cast<int>(blockIdx.x - st.begin[j]);
  if (g.kind == MLP_BIAS_GRAD) {
    bias_grad(g, st.adam, b * kSumCols, reinterpret_cast<float*>(arena));
    return;
  }
  const int tiles_n = (g.N + 32 * TILES - 1) / (32 * TILES);
  const int m0 = b / tiles_n * (32 * TILES), n0 = b % tiles_n * (32 * TILES);
  const f32x16 acc = block_product<TILES>(g, m0, n0, arena);
  // a lane holds one column of a tile, rows 8 q + 4 (lane / 32) .. + 3 in register quad q
  const int row_at = m0 + 4 * (lane >> 5), col_at = n0 + (lane & 31);
  float loss = 0.0f;
  if constexpr (TILES == 1) {  // the first wave's tile, a quad per wave
    float* s_tile = reinterpret_cast<float*>(arena);
    if (wave == 0) {  // the only wave that read the fragments
#pragma unroll
      for (int r = 0; r < 16; ++r) s_tile[r * 64 + lane] = acc[r];
    }
    __syncthreads();
    float quad[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) quad[i] = s_tile[(4 * wave + i) * 64 + lane];
    if (col_at < g.N) loss = finish_quad(g, st.adam, row_at + 8 * wave, col_at, quad);
  } else {
    const int col = col_at + 32 * (wave & 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float quad[4] = {acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
      if (col < g.N) loss += finish_quad(g, st.adam, row_at + 32 * (wave >> 1) + 8 * q, col, quad);
    }
  }
  if (g.kind == MLP_LOSS) {
    for (int off = 32; off > 0; off >>= 1) loss += __shfl_xor(loss, off, 64);
    if (lane == 0) s_loss[wave] = loss;
    __syncthreads();
    if (threadIdx.x == 0) g.parts[b] = ((s_loss[0] + s_loss[1]) + (s_loss[2] + s_loss[3])) * g.inv_count;
  }
}

// bf16 copies of an fp32 matrix (R x C), by rows and transposed; the transpose's row padding
// up to a multiple of 64 is cleared.
__global__ void k_pack(const float* x, int R, int C, uint16_t* row, int ld_row, uint16_t* col, int ld_col) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= static_cast<int64_t>((R + 63) / 64 * 64) * C) return;
  const int64_t r = i / C, c = i % C;
  const uint16_t h = r < R ? to_bf16(x[i]) : static_cast<uint16_t>(0);
  row[r * ld_row + c] = h;
  col[c * ld_col + r] = h;
}

// Tiles per block: 2 x 2 halves the operand traffic and uses every SIMD's matrix core, and
// needs enough tiles to fill the chip even so; one tile per block shortens the stage where
// tiles are few. Training step at 1,024 samples, hidden layers of one width twice, one tile
// against four: 100 / 120 us at 512 (512 tiles), 135 / 145 at 1,024 (1,024 tiles), 192 / 180 at
// 1,536 (1,536 tiles), 262 / 228 at 2,048; 1,830 / 1,406 at 2,048 samples of 4,096.
constexpr int kManyTiles = 1280;
inline uint32_t blocks_of(const MlpJob& g, int t) {
  if (g.kind == MLP_BIAS_GRAD) return static_cast<uint32_t>((g.N + kSumCols - 1) / kSumCols);
  return static_cast<uint32_t>((g.M + 32 * t - 1) / (32 * t)) * static_cast<uint32_t>((g.N + 32 * t - 1) / (32 * t));
}
inline int tiles_of(int M, int N) {
  return static_cast<int64_t>((M + 31) / 32) * ((N + 31) / 32) >= kManyTiles ? 2 : 1;
}

}  // namespace

uint32_t mlp_loss_parts(int M, int N) {
  MlpJob g{};
  g.kind = MLP_LOSS;
  g.M = M;
  g.N = N;
  return blocks_of(g, tiles_of(M, N));
}

hipError_t mlp_stage(MlpStage& st, int n_jobs, hipStream_t s) {
  int t = 1;
  for (int j = 0; j < n_jobs; ++j)
    if (st.job[j].kind != MLP_BIAS_GRAD) t = std::max(t, tiles_of(st.job[j].M, st.job[j].N));
  uint32_t blocks = 0;
  for (int j = 0; j <= kMlpJobs; ++j) {
    st.begin[j] = j < n_jobs || j == kMlpJobs ? blocks : ~0u;
    if (j < n_jobs) blocks += blocks_of(st.job[j], t);
  }
  if (blocks == 0) return hipSuccess;
  if (t == 1) hipLaunchKernelGGL(k_mlp_stage<1>, dim3(blocks), dim3(256), 0, s, st);
  else hipLaunchKernelGGL(k_mlp_stage<2>, dim3(blocks), dim3(256), 0, s, st);
  return hipGetLastError();
}

hipError_t mlp_pack(const float* x, int R, int C, uint16_t* row, int ld_row, uint16_t* col, int ld_col,
                    hipStream_t s) {
  const int64_t n = static_cast<int64_t>(mlp_rows(R)) * C;
  hipLaunchKernelGGL(k_pack, dim3(static_cast<uint32_t>((n + 255) / 256)), dim3(256), 0, s, x, R, C, row, ld_row, col,
                     ld_col);
  return hipGetLastError();
}

hipError_t mlp_gemm(const GemmArgs& g, hipStream_t s) {
  if (g.M <= 0 || g.N <= 0 || g.K <= 0) return hipSuccess;
  dim3 grid((g.N + kBN - 1) / kBN, (g.M + kBM - 1) / kBM);
  hipLaunchKernelGGL(k_gemm, grid, dim3(256), 0, s, g);
  return hipGetLastError();
}

}  // namespace epi
