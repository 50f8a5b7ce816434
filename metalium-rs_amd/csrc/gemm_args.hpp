// What the matrix-product kernels share (csrc/gemm.hip, csrc/gemm_f32.hip): a
// launch's arguments and its plan, the order of the output tiles, and the
// epilogue of a linear layer.
#pragma once

#include "common.hpp"
#include "tails.hpp"

namespace mi {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

struct GemmArgs {
  const void *a;
  const void *b;
  void *c;
  int64_t M, N, K;
  int64_t lda, ldb, ldc;
  int64_t sa, sb, sc;  // batch strides in elements (0 = broadcast)
  // Items come in groups: item z = (z / per_group, z % per_group) starts at
  // (z / per_group) * s?2 + (z % per_group) * s? (one group: per_group = batch).
  int64_t per_group;
  int64_t sa2, sb2, sc2;
  int tiles_m, tiles_n;
  int64_t kc;          // split-K: k per slice (blockIdx.z), 0 for none
  // Epilogue of a linear layer (batch 1): C = resid + (A B + bias), each sum
  // rounded in that order; null pointers skip the term.
  const float *bias;   // [N]
  const float *resid;  // [M, N], row pitch ldr
  int64_t ldr;
  // Direct BF16 kernel only: B's own k extent when A's k loop runs over
  // several copies of it (A = [hi | lo] parts of an F32 operand against one
  // B: B's k wraps modulo kb; 0 for none).
  int64_t kb = 0;
  // Direct BF16 kernel, EDGE 2 only: A's k steps back by ka from k = ka0 on
  // (0 for none).
  int64_t ka = 0, ka0 = 0;
  // Direct BF16 kernel only: B's rows are gate|up pairs (32 gate rows, then
  // the 32 up rows of the same outputs, ...), and C receives silu(gate) * up
  // for the N / 2 outputs -- SWIGLU_PARTS: as its BF16 parts ([M, N] BF16: a
  // row's heads, then its remainders); SWIGLU_BF16 / SWIGLU_F32: [M, N / 2]
  // rounded once to BF16, or F32; 0 for a plain product.
  int swiglu = 0;
  int out_bf16 = 0;  // gemm_f32.hip only: the result rounded to BF16
  QkvTail qkv;  // direct BF16 kernel only: the q|k|v tail instead of C
};

// The epilogue over one 32 x 32 accumulator fragment, whose lane holds column
// `col` at rows row0 + 8 (r / 4) + r % 4: the fragment's 16 residual values
// and its bias are all requested before any result is stored.  The result
// may be the residual itself (an in-place update), so a residual load issued
// after a store the compiler cannot prove disjoint waits for that store; per
// value, that chain made the write-out latency-bound.  Out-of-range values
// (GUARD) are not read.
template <bool GUARD>
__device__ __forceinline__ void fragment_epilogue(const GemmArgs &g, int64_t row0, int64_t col, float (&v)[16]) {
  float e[16];
  if (g.resid) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = row0 + 8 * (r >> 2) + (r & 3);
      e[r] = (!GUARD || (row < g.M && col < g.N)) ? g.resid[row * g.ldr + col] : 0.f;
    }
  }
  const float b = (g.bias && (!GUARD || col < g.N)) ? g.bias[col] : 0.f;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    float x = v[r];
    if (g.bias) x = __fadd_rn(x, b);
    if (g.resid) x = __fadd_rn(e[r], x);
    v[r] = x;
  }
}

// Map a linear workgroup id to an output tile (tm, tn), grouping the tiles
// each XCD receives.  Workgroup w runs on XCD w % 8.
__device__ __forceinline__ void tile_of(int w, int tiles_m, int tiles_n, int *tm, int *tn) {
  const int total = tiles_m * tiles_n;
  int t = w;
  if ((total & 7) == 0) t = (w & 7) * (total >> 3) + (w >> 3);
  // Within the XCD-ordered sequence, walk groups of GROUP_M tile rows.
  constexpr int GROUP_M = 4;
  const int group_size = GROUP_M * tiles_n;
  const int g = t / group_size;
  const int first_m = g * GROUP_M;
  const int gm = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const int in_g = t - g * group_size;
  *tm = first_m + in_g % gm;
  *tn = in_g / gm;
}

// `s_waitcnt vmcnt(N)`, the other counters left alone.
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}

struct Plan {
  int64_t M, N, K, batch;
  bool ta, tb;
  int ea, eb, eo;  // element kinds
  const void *a, *b;
  void *c;
  int64_t sa, sb, sc;
  int64_t lda, ldb;   // row pitch of each operand's storage
  int64_t kc = 0;     // split-K slice length (register kernel only)
  int splits = 1;
  bool fast = true;   // F32 operands split into BF16 parts (the fast matmul mode)
  const float *bias = nullptr;   // linear epilogue (batch 1): C = resid + (A B + bias)
  const float *resid = nullptr;
  int64_t ldr = 0;
  int64_t ldc = 0;                // result row pitch (0: N)
  int64_t per_group = 0;          // items per group (0: one group of `batch`)
  int64_t sa2 = 0, sb2 = 0, sc2 = 0;  // group strides
  int64_t kb = 0, ka = 0, ka0 = 0;  // direct BF16 kernel: operands whose k repeats (see GemmArgs)
  int swiglu = 0;  // direct BF16 kernel: gate|up pairs into silu(gate) * up (see GemmArgs)
  QkvTail qkv;     // direct BF16 kernel: the q|k|v tail (see QkvTail)
  // The RMSNorm of the F32 result's rows (mi_linear_add_rms_norm): taken by
  // the split-K reduce when the product splits over k (*norm_done set),
  // else run after the product by the caller.
  const float *norm_gamma = nullptr;
  float norm_eps = 0.0f;
  void *norm_out = nullptr;
  int norm_elem = MI_F32;
  bool *norm_done = nullptr;
};

// A product of F32 operands at F32 precision (csrc/gemm_f32.hip): batches, groups and split-K slices as the plan says.
hipError_t run_f32_pipe(const Plan &p, hipStream_t st);
// Whether run_f32_pipe takes the plan.
bool f32_pipe_fits(const Plan &p);
// The split-K slices it takes a product of one item in (1: none).
int f32_pipe_slices(const Plan &p);

}  // namespace mi
