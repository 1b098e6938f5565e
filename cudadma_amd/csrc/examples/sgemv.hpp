// sgemv ("n" form: y = alpha * A x, A column-major) with the vector, or the
// vector and the matrix panel, staged through LDS by DMA wavefronts.
//
// What the reference's example computes: src/examples/sgemv/sgemv_dma.cu
// (vector staged, one buffer :140-175; vector staged, two objects on the same
// DMA threads :262-325; vector and matrix staged :329-388 and :392-470).  Thread
// `row` owns one row: res = fma(A[row + j*lda], x[j], res) for ascending j from
// 0.0f, y[row] = alpha * res.  Written against the first-generation class names
// (cudaDMASequential, cudaDMAStrided of include/cudaDMA.h).
//
// The kernels need m to be a multiple of the columns staged per hand-off, except
// sgemvn_both_double, which takes multiples of 32 from the columns of one panel on.
// Where the matrix is staged, lda*4 has to be a multiple of 16 B and fit an int.
// Rows beyond n are neither read from global memory by compute threads nor written.
#pragma once

#include "../../../include/cudaDMA.h"

namespace examples {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Vector staged in one buffer; the matrix is read straight from global memory.
// Launch with COMPUTE_THREADS + DMA_THREADS_PER_LD threads.
template<int COMPUTE_THREADS, int DMA_THREADS_PER_LD, int VEC_ELMTS>
__global__ void sgemvn_vec_single(int n, int m, float alpha, const float* __restrict__ A, int lda,
                                  const float* __restrict__ x, float* __restrict__ y)
{
  __shared__ __attribute__((aligned(16))) float buff[VEC_ELMTS];
  cudaDMASequential<true, 16, 4 * VEC_ELMTS, DMA_THREADS_PER_LD>
    dma_ld_0(1, COMPUTE_THREADS, COMPUTE_THREADS);

  if (threadIdx.x < COMPUTE_THREADS) {
    dma_ld_0.start_async_dma();
    const int row = blockIdx.x * COMPUTE_THREADS + threadIdx.x;
    const bool live = row < n;
    const float* a_col = A + (live ? row : 0);
    float res = 0.0f;
    for (int i = 0; i < m; i += VEC_ELMTS) {
      dma_ld_0.wait_for_dma_finish();
#pragma unroll 8
      for (int j = 0; j < VEC_ELMTS; ++j) {
        res = __builtin_fmaf(*a_col, buff[j], res);
        a_col += lda;
      }
      if (i + VEC_ELMTS < m) dma_ld_0.start_async_dma();
    }
    if (live) y[row] = alpha * res;
  } else if (dma_ld_0.owns_this_thread()) {
    for (int i = 0; i < m; i += VEC_ELMTS)
      dma_ld_0.execute_dma(x + i, buff);
  }
}

// Vector staged through two buffers by two objects that share the same DMA
// threads ("manual" double buffering).  Launch with COMPUTE_THREADS + DMA_THREADS_PER_LD threads.
template<int COMPUTE_THREADS, int DMA_THREADS_PER_LD, int VEC_ELMTS>
__global__ void sgemvn_vec_manual(int n, int m, float alpha, const float* __restrict__ A, int lda,
                                  const float* __restrict__ x, float* __restrict__ y)
{
  __shared__ __attribute__((aligned(16))) float buff0[VEC_ELMTS];
  __shared__ __attribute__((aligned(16))) float buff1[VEC_ELMTS];
  typedef cudaDMASequential<true, 16, 4 * VEC_ELMTS, DMA_THREADS_PER_LD> dma_t;
  dma_t dma_ld_0(1, COMPUTE_THREADS, COMPUTE_THREADS);
  dma_t dma_ld_1(2, COMPUTE_THREADS, COMPUTE_THREADS);

  if (threadIdx.x < COMPUTE_THREADS) {
    dma_ld_0.start_async_dma();
    dma_ld_1.start_async_dma();
    const int row = blockIdx.x * COMPUTE_THREADS + threadIdx.x;
    const bool live = row < n;
    const float* a_col = A + (live ? row : 0);
    float res = 0.0f;
    for (int i = 0; i < m; i += 2 * VEC_ELMTS) {
      dma_ld_0.wait_for_dma_finish();
#pragma unroll 8
      for (int j = 0; j < VEC_ELMTS; ++j) {
        res = __builtin_fmaf(*a_col, buff0[j], res);
        a_col += lda;
      }
      if (i + 2 * VEC_ELMTS < m) dma_ld_0.start_async_dma();
      dma_ld_1.wait_for_dma_finish();
#pragma unroll 8
      for (int j = 0; j < VEC_ELMTS; ++j) {
        res = __builtin_fmaf(*a_col, buff1[j], res);
        a_col += lda;
      }
      if (i + 2 * VEC_ELMTS < m) dma_ld_1.start_async_dma();
    }
    if (live) y[row] = alpha * res;
  } else if (dma_ld_0.owns_this_thread()) {
    for (int i = 0; i < m; i += 2 * VEC_ELMTS) {
      dma_ld_0.execute_dma(x + i, buff0);
      dma_ld_1.execute_dma(x + i + VEC_ELMTS, buff1);
    }
  }
}

// Vector and a VEC_ELMTS-column panel of the matrix staged, one buffer each.
// The panel is VEC_ELMTS strided elements (columns) of COMPUTE_THREADS floats,
// packed in LDS by the one-stride constructor of the older interface.
// Launch with COMPUTE_THREADS + (1 + MAT_LDS) * DMA_THREADS_PER_LD threads.
template<int COMPUTE_THREADS, int DMA_THREADS_PER_LD, int VEC_ELMTS, int MAT_LDS>
__global__ void sgemvn_both_single(int n, int m, float alpha, const float* __restrict__ A, int lda,
                                   const float* __restrict__ x, float* __restrict__ y)
{
  __shared__ __attribute__((aligned(16))) float buff[VEC_ELMTS];
  __shared__ __attribute__((aligned(16))) float mat[VEC_ELMTS][COMPUTE_THREADS];

  cudaDMASequential<true, 16, 4 * VEC_ELMTS, DMA_THREADS_PER_LD>
    dma_ld_0(1, COMPUTE_THREADS, COMPUTE_THREADS);
  cudaDMAStrided<true, 16, 4 * COMPUTE_THREADS, MAT_LDS * DMA_THREADS_PER_LD, VEC_ELMTS>
    dma_ld_1(2, COMPUTE_THREADS, COMPUTE_THREADS + DMA_THREADS_PER_LD, 4 * lda);

  if (threadIdx.x < COMPUTE_THREADS) {
    dma_ld_0.start_async_dma();
    dma_ld_1.start_async_dma();
    float res = 0.0f;
    for (int i = 0; i < m; i += VEC_ELMTS) {
      dma_ld_0.wait_for_dma_finish();
      dma_ld_1.wait_for_dma_finish();
#pragma unroll
      for (int j = 0; j < VEC_ELMTS; ++j)
        res = __builtin_fmaf(mat[j][threadIdx.x], buff[j], res);
      if (i + VEC_ELMTS < m) {
        dma_ld_0.start_async_dma();
        dma_ld_1.start_async_dma();
      }
    }
    const int row = blockIdx.x * COMPUTE_THREADS + threadIdx.x;
    if (row < n) y[row] = alpha * res;
  } else if (dma_ld_0.owns_this_thread()) {
    for (int i = 0; i < m; i += VEC_ELMTS)
      dma_ld_0.execute_dma(x + i, buff);
  } else if (dma_ld_1.owns_this_thread()) {
    const float* panel = A + (long long)blockIdx.x * COMPUTE_THREADS;
    for (int i = 0; i < m; i += VEC_ELMTS) {
      dma_ld_1.execute_dma(panel, mat);
      panel += (long long)lda * VEC_ELMTS;
    }
  }
}

// Vector and matrix panel staged through two buffers each, four objects on
// disjoint DMA wavefronts.  A workgroup owns ROWS rows; the panels hold COLS columns,
// and the last one is moved back to end with column m - 1, its columns that were
// summed before are skipped (m >= COLS, m and COLS multiples of 32).
//
// What bounds it: a row's sum is one chain of multiply-adds in ascending column order, 8 cycles each (4096 columns:
// 14 us), and the wavefront that runs it also issues 12 LDS reads per 16 columns (160 cycles per 16 columns with the LDS to
// itself, 230 next to the DMA wavefronts).  4096 x 4096: 59 us with panels of 128 rows x 32 columns (32 workgroups,
// 128 hand-offs), 30 with 16 x 256.  Fewer DMA wavefronts leave too few bytes in flight (one per panel: 40 us).
// Launch with sgemv_both_double_threads<ROWS, VEC_DMA, MAT_DMA>() threads.
template<int ROWS, int VEC_DMA_THREADS, int MAT_DMA_THREADS>
constexpr int sgemv_both_double_threads() { return (ROWS < 64 ? 64 : ROWS) + 2 * (VEC_DMA_THREADS + MAT_DMA_THREADS); }

// 16 columns of a panel on their way from LDS to the chain of a compute thread.
template<int ROWS>
struct SgemvBlock {
  float a[16];
  f32x4_t x[4];
  __device__ __forceinline__ void load(const float* mat, const float* vec, const int row, const int col)
  {
    // one base address per group of columns that the offsets of ds_read2_b32 or ds_read2st64_b32 reach
    constexpr int kReach = ROWS == 32 ? 8 : 16;
#pragma unroll
    for (int g = 0; g < 16; g += kReach) {
      int base = (col + g) * ROWS + row;
      asm("" : "+v"(base));
#pragma unroll
      for (int j = 0; j < kReach; ++j) a[g + j] = mat[base + j * ROWS];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = *(const f32x4_t*)(vec + col + 4 * j);
  }
  __device__ __forceinline__ float chain(float res) const
  {
#pragma unroll
    for (int j = 0; j < 16; ++j) res = __builtin_fmaf(a[j], x[j / 4][j % 4], res);
    return res;
  }
};

// Sums the columns [first, COLS) of a panel; both are multiples of 32.
// The reads of one block go out back to back under the sums of the other: read and multiply-add in turn issue at
// half the speed (266 against 160 cycles per 16 columns), and left alone the scheduler reads a block right before it is needed.
template<int ROWS, int COLS>
__device__ __forceinline__ float sgemv_panel(const float* mat, const float* vec, const int row, const int first, float res)
{
  if constexpr (COLS == 32) {
    // two blocks are over before a pipeline has filled: the compiler's own order is 5 % faster (16384 x 224: 5.4 -> 5.1 us)
#pragma unroll
    for (int j = 0; j < COLS; ++j) res = __builtin_fmaf(mat[j * ROWS + row], vec[j], res);
    return res;
  }
  SgemvBlock<ROWS> even, odd;
  even.load(mat, vec, row, first);
  for (int c = first; c < COLS; c += 32) {
    odd.load(mat, vec, row, c + 16);
    __builtin_amdgcn_sched_barrier(0);
    res = even.chain(res);
    __builtin_amdgcn_sched_barrier(0);
    even.load(mat, vec, row, c + 32 < COLS ? c + 32 : 0);
    __builtin_amdgcn_sched_barrier(0);
    res = odd.chain(res);
    __builtin_amdgcn_sched_barrier(0);
  }
  return res;
}

template<int ROWS, int COLS, int VEC_DMA_THREADS, int MAT_DMA_THREADS, int MAT_BYTES = 4 * ROWS * COLS / MAT_DMA_THREADS>
__global__ __launch_bounds__((sgemv_both_double_threads<ROWS, VEC_DMA_THREADS, MAT_DMA_THREADS>()))
void sgemvn_both_double(int n, int m, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ x,
                        float* __restrict__ y)
{
  constexpr int kCompute = ROWS < 64 ? 64 : ROWS;       // with fewer rows the rest of the wavefront doubles them
  __shared__ __attribute__((aligned(16))) float buff0[COLS];
  __shared__ __attribute__((aligned(16))) float buff1[COLS];
  __shared__ __attribute__((aligned(16))) float mat0[COLS * ROWS];
  __shared__ __attribute__((aligned(16))) float mat1[COLS * ROWS];

  HIPDMA_ASSERT(m >= COLS && (m % 32) == 0);      // a shorter matrix would have the panel begin before its first column
  // a thread holds its share of a panel in registers, all of it unless MAT_BYTES says less: the next panel is on its way while this
  // one is read
  typedef cudaDMASequential<true, 16, 4 * COLS, VEC_DMA_THREADS> vec_dma_t;
  typedef CudaDMAStrided<true, 16, MAT_BYTES, 4 * ROWS, MAT_DMA_THREADS, COLS> mat_dma_t;
  vec_dma_t dma_vec_0(1, kCompute, kCompute);
  vec_dma_t dma_vec_1(2, kCompute, kCompute + VEC_DMA_THREADS);
  mat_dma_t dma_mat_0(3, kCompute, kCompute + 2 * VEC_DMA_THREADS, 4 * lda, 4 * ROWS);
  mat_dma_t dma_mat_1(4, kCompute, kCompute + 2 * VEC_DMA_THREADS + MAT_DMA_THREADS, 4 * lda, 4 * ROWS);

  const int panels = (m + COLS - 1) / COLS;
  const int row0 = blockIdx.x * ROWS;
  // first column of panel p
  auto begin = [&](const int p) { const int c = p * COLS; return c < m - COLS ? c : m - COLS; };

  if (threadIdx.x < kCompute) {
    dma_vec_0.start_async_dma();
    dma_mat_0.start_async_dma();
    if (panels > 1) { dma_vec_1.start_async_dma(); dma_mat_1.start_async_dma(); }
    const int row = threadIdx.x % ROWS;
    float res = 0.0f;
    for (int p = 0; p < panels; p += 2) {
      dma_vec_0.wait_for_dma_finish();
      dma_mat_0.wait_for_dma_finish();
      res = sgemv_panel<ROWS, COLS>(mat0, buff0, row, p * COLS - begin(p), res);
      if (p + 2 < panels) { dma_vec_0.start_async_dma(); dma_mat_0.start_async_dma(); }
      if (p + 1 < panels) {
        dma_vec_1.wait_for_dma_finish();
        dma_mat_1.wait_for_dma_finish();
        res = sgemv_panel<ROWS, COLS>(mat1, buff1, row, (p + 1) * COLS - begin(p + 1), res);
        if (p + 3 < panels) { dma_vec_1.start_async_dma(); dma_mat_1.start_async_dma(); }
      }
    }
    if (threadIdx.x < ROWS && row0 + row < n) y[row0 + row] = alpha * res;
  } else if (dma_vec_0.owns_this_thread()) {
    for (int p = 0; p < panels; p += 2) dma_vec_0.execute_dma(x + begin(p), buff0);
  } else if (dma_vec_1.owns_this_thread()) {
    for (int p = 1; p < panels; p += 2) dma_vec_1.execute_dma(x + begin(p), buff1);
  } else if (dma_mat_0.owns_this_thread()) {
    for (int p = 0; p < panels; p += 2) dma_mat_0.execute_dma(A + row0 + (long long)lda * begin(p), mat0);
  } else if (dma_mat_1.owns_this_thread()) {
    for (int p = 1; p < panels; p += 2) dma_mat_1.execute_dma(A + row0 + (long long)lda * begin(p), mat1);
  }
}

}  // namespace examples
