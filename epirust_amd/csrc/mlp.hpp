// Surrogate MLP: launch interface of the bf16-MFMA kernels (mlp.hip).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>

namespace epi {

// C[M x N] = A * B, fp32 row-major. A element (m, k) is A[m * lda_m + k * lda_k]; B element
// (k, n) is B[k * ldb_k + n * ldb_n].
struct GemmArgs {
  const uint16_t* A;
  const uint16_t* B;
  int64_t lda_m, lda_k, ldb_k, ldb_n;
  int M, N, K;
  float* C;
};

// bf16 matrices of the network: rows of mlp_pitch(columns) elements, mlp_rows(rows) of them,
// all zero at first. The padding columns stay zero (they are multiplied with); the padding
// rows are read, and what they give is dropped.
inline int mlp_rows(int rows) { return (rows + 63) / 64 * 64; }
inline int mlp_pitch(int cols) { return (cols + 63) / 64 * 64 + 16; }  // rows start on different channels

// What a stage does with the product of one tile (M rows, N columns).
enum : int {
  MLP_HIDDEN = 0,   // z = p + bias, kept in `c` if set; bf16 GELU(z) to `row` and `col`
  MLP_OUTPUT,       // z = p + bias to `c`
  MLP_LOSS,         // z = p + bias; its MSE against `t` to `parts`, the gradient to `c`, `row`, `col`
  MLP_INPUT_GRAD,   // p * GELU'(`z`) to `c`, `row`, `col`
  MLP_WEIGHT_GRAD,  // p to `c`, or an Adam step of `w` with it (bf16 copies to `row` and `col`)
  MLP_BIAS_GRAD,    // no product: column sums of `z` (K rows) to `c`, or an Adam step of `w` with them
};

struct AdamArgs {
  float lr, b1, b2, eps, c1, c2;
};

// One product A * Bt^T of a stage: A is M x K and Bt is N x K, both with k contiguous (pitch
// lda, ldb). Outputs that are null are not written. `row` is the bf16 result by rows, `col`
// its transpose, whose row padding is cleared.
struct MlpJob {
  int kind;
  int M, N, K;
  const uint16_t* A;
  int lda;
  const uint16_t* Bt;
  int ldb;
  const float* bias;
  const float* t;
  const float* z;
  float* c;
  uint16_t* row;
  uint16_t* col;
  int ld_row, ld_col;
  float* parts;
  float inv_count;
  int adam;  // apply the gradient to w, m, v instead of writing it
  float *w, *m, *v;
};

// Products that depend on nothing of each other, in one launch.
constexpr int kMlpJobs = 4;
struct MlpStage {
  MlpJob job[kMlpJobs];
  uint32_t begin[kMlpJobs + 1];  // first block of each job (filled by mlp_stage)
  AdamArgs adam;
};
// Loss parts that an MLP_LOSS job of this shape writes.
uint32_t mlp_loss_parts(int M, int N);

hipError_t mlp_gemm(const GemmArgs& g, hipStream_t s);
hipError_t mlp_stage(MlpStage& st, int n_jobs, hipStream_t s);
// bf16 copies of an fp32 matrix x (R x C, device or pinned host memory): by rows and
// transposed, the transpose's row padding cleared.
hipError_t mlp_pack(const float* x, int R, int C, uint16_t* row, int ld_row, uint16_t* col, int ld_col,
                    hipStream_t s);

}  // namespace epi
