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
// sgemvn_ring, which takes multiples of 32 from 128 on.
// Where the matrix is staged, lda*4 has to be a multiple of 16 B and fit an int.
// Rows beyond n are neither read from global memory by compute threads nor written.
#pragma once

#include <utility>

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
// disjoint DMA wavefronts; a compute thread per row.  A workgroup owns ROWS rows, the panels hold COLS columns (m a multiple of
// COLS).  For narrow matrices and for many rows, where several workgroups share a compute unit and hide each other's hand-offs.
// Launch with sgemv_both_double_threads<ROWS, VEC_DMA, MAT_DMA>() threads.
template<int COMPUTE_THREADS, int VEC_DMA_THREADS, int MAT_DMA_THREADS>
constexpr int sgemv_both_double_threads() { return COMPUTE_THREADS + 2 * (VEC_DMA_THREADS + MAT_DMA_THREADS); }

template<int ROWS, int COLS, int VEC_DMA_THREADS, int MAT_DMA_THREADS, int MAT_BYTES = 4 * ROWS * COLS / MAT_DMA_THREADS>
__global__ __launch_bounds__((sgemv_both_double_threads<ROWS, VEC_DMA_THREADS, MAT_DMA_THREADS>()))
void sgemvn_both_double(int n, int m, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ x,
                        float* __restrict__ y)
{
  __shared__ __attribute__((aligned(16))) float buff0[COLS];
  __shared__ __attribute__((aligned(16))) float buff1[COLS];
  __shared__ __attribute__((aligned(16))) float mat0[COLS * ROWS];
  __shared__ __attribute__((aligned(16))) float mat1[COLS * ROWS];

  HIPDMA_ASSERT(m >= COLS && (m % COLS) == 0);
  // a thread holds its share of a panel in registers, all of it unless MAT_BYTES says less: the next panel is on its way while this
  // one is read
  typedef cudaDMASequential<true, 16, 4 * COLS, VEC_DMA_THREADS> vec_dma_t;
  typedef CudaDMAStrided<true, 16, MAT_BYTES, 4 * ROWS, MAT_DMA_THREADS, COLS> mat_dma_t;
  vec_dma_t dma_vec_0(1, ROWS, ROWS);
  vec_dma_t dma_vec_1(2, ROWS, ROWS + VEC_DMA_THREADS);
  mat_dma_t dma_mat_0(3, ROWS, ROWS + 2 * VEC_DMA_THREADS, 4 * lda, 4 * ROWS);
  mat_dma_t dma_mat_1(4, ROWS, ROWS + 2 * VEC_DMA_THREADS + MAT_DMA_THREADS, 4 * lda, 4 * ROWS);

  const int panels = m / COLS;
  const int row0 = blockIdx.x * ROWS;
  auto sum = [&](const float* mat, const float* vec, float res) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < COLS; ++j) res = __builtin_fmaf(mat[j * ROWS + threadIdx.x], vec[j], res);
    return res;
  };
  if (threadIdx.x < ROWS) {
    dma_vec_0.start_async_dma();
    dma_mat_0.start_async_dma();
    if (panels > 1) { dma_vec_1.start_async_dma(); dma_mat_1.start_async_dma(); }
    float res = 0.0f;
    for (int p = 0; p < panels; p += 2) {
      dma_vec_0.wait_for_dma_finish();
      dma_mat_0.wait_for_dma_finish();
      res = sum(mat0, buff0, res);
      if (p + 2 < panels) { dma_vec_0.start_async_dma(); dma_mat_0.start_async_dma(); }
      if (p + 1 < panels) {
        dma_vec_1.wait_for_dma_finish();
        dma_mat_1.wait_for_dma_finish();
        res = sum(mat1, buff1, res);
        if (p + 3 < panels) { dma_vec_1.start_async_dma(); dma_mat_1.start_async_dma(); }
      }
    }
    if (row0 + threadIdx.x < n) y[row0 + threadIdx.x] = alpha * res;
  } else if (dma_vec_0.owns_this_thread()) {
    for (int p = 0; p < panels; p += 2) dma_vec_0.execute_dma(x + p * COLS, buff0);
  } else if (dma_vec_1.owns_this_thread()) {
    for (int p = 1; p < panels; p += 2) dma_vec_1.execute_dma(x + p * COLS, buff1);
  } else if (dma_mat_0.owns_this_thread()) {
    for (int p = 0; p < panels; p += 2) dma_mat_0.execute_dma(A + row0 + (long long)lda * p * COLS, mat0);
  } else if (dma_mat_1.owns_this_thread()) {
    for (int p = 1; p < panels; p += 2) dma_mat_1.execute_dma(A + row0 + (long long)lda * p * COLS, mat1);
  }
}

// ---- sixteen rows per compute wavefront, a ring of stages of 128 columns ----
// A row's sum is one chain of multiply-adds in ascending column order, 4.6 cycles each with the operands in registers (4096 columns:
// 7.9 us), and every LDS request of the wavefront that runs the chain holds it up by about 7.  So the wavefront asks for four columns at a
// time: its four rows of sixteen lanes hold the same sixteen matrix rows, each a quarter of a stage's columns.  (With a lane per matrix
// row a request fetches one column, and the chain takes 17 cycles per column with the hand-offs; now 8.)  The quarters are summed
// one after the other: the lanes of one quarter run their 32 multiply-adds and hand the sums on to the lanes of the next one; what the
// other lanes compute meanwhile is not used.  The hand-over is one v_permlane16_swap or v_permlane32_swap, for which the quarters lie in the
// lane rows 0, 1, 3, 2.  The columns are swizzled in LDS: of four that follow each other, a wavefront's sixteen rows lie in four different
// quarters of the 64 banks.  Lane row h takes columns 4q .. 4q+3 of its quarter in the order that begins with 4q + h, so the four lane
// rows read four different ones.
//
// 4096 x 4096: 31.5 us with a lane per row and two register-staged panels of 256 columns, 17.2 now (19.5 from DRAM); 8192 x 8192 62 and 44;
// 512 x 16384, whose chain is all there is, 103 and 55.  Matrix instructions would run the same chain (v_mfma_f32_16x16x4_f32 adds its four
// products in order), at 8.1 cycles a column: no faster than this, hand-offs included.
constexpr int kSgemvRows = 16, kSgemvQuarter = 32, kSgemvCols = 4 * kSgemvQuarter;
constexpr int sgemv_lane_row(const int quarter) { return quarter < 2 ? quarter : 5 - quarter; }

template<int ROWS>
struct SgemvStage {
  float mat[kSgemvCols * ROWS];
  float vec[kSgemvCols];
};

// A stage on its way from LDS to the chain.
template<int ROWS>
struct SgemvBlock {
  float a[kSgemvQuarter];                   // a[4q + i]: column 4q + (i + lane row) % 4 of the quarter
  f32x4_t x[kSgemvQuarter / 4];

  // where a lane finds its row of column 4q + (i + lane row) % 4 of its quarter, q < 4; sixteen columns on the keys repeat
  struct Places {
    int at[4][4], vec;
    __device__ __forceinline__ Places(const int wave, const int lane)
    {
      const int h = lane >> 4, first = (h < 2 ? h : 5 - h) * kSgemvQuarter;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int col = 4 * q + ((i + h) & 3), chunk = (wave * kSgemvRows + (lane & 15)) / 4;
          at[q][i] = (first + col) * ROWS + hipdma::swizzled_chunk(col, chunk, ROWS / 4) * 4 + (lane & 3);
        }
      vec = first;
    }
  };
  __device__ __forceinline__ void load(const SgemvStage<ROWS>& stage, const Places& places)
  {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float* p = stage.mat + places.at[q][i];
        a[4 * q + i] = p[0];
        a[4 * (q + 4) + i] = p[16 * ROWS];
      }
#pragma unroll
    for (int q = 0; q < kSgemvQuarter / 4; ++q) x[q] = *(const f32x4_t*)(stage.vec + places.vec + 4 * q);
  }
  // The quarters from `first` on; on entry and exit the sums are in lane row 0.
  __device__ __forceinline__ float chain(float res, const int first) const
  {
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      if (p >= first) {
#pragma unroll
        for (int c = 0; c < kSgemvQuarter; ++c)
          res = __builtin_fmaf(a[(c & ~3) + ((c - sgemv_lane_row(p)) & 3)], x[c / 4][c % 4], res);
      }
      const unsigned bits = __float_as_uint(res);
      // first of the pair: odd lane rows (upper half) take the even ones' (lower half's) values; second: the other way round
      if (p == 0) res = __uint_as_float(__builtin_amdgcn_permlane16_swap(bits, bits, false, false)[0]);        // lane row 0 -> 1
      else if (p == 1) res = __uint_as_float(__builtin_amdgcn_permlane32_swap(bits, bits, false, false)[0]);   // 1 -> 3
      else if (p == 2) res = __uint_as_float(__builtin_amdgcn_permlane16_swap(bits, bits, false, false)[1]);   // 3 -> 2
      else res = __uint_as_float(__builtin_amdgcn_permlane32_swap(bits, bits, false, false)[1]);               // 2 -> 0
    }
    return res;
  }
};

template<typename IDS> struct SgemvGuards;
template<int... ID>
struct SgemvGuards<std::integer_sequence<int, ID...>> {
  cudaDMACustom of[sizeof...(ID)];
  __device__ __forceinline__ SgemvGuards(const int dma_threads, const int compute_threads)
    : of{cudaDMACustom(ID, dma_threads, compute_threads, compute_threads)...} {}
};

// ROWS rows per workgroup, one compute wavefront for sixteen of them; DMA wavefronts that share the columns of a stage.  Two of the four
// stages are on their way, by direct-to-LDS loads, which hold no registers; the third is read, the fourth waits to be: with three on their way a
// DMA wavefront waits for a stage to be given back before it reports the next one (2048 x 8192 30.0 -> 38 us), and more stages gain
// nothing (six, three on their way: 31).  A DMA wavefront gets rid of a 1 KB load every 50 ns, so one of them alone holds the chain up (32
// rows: 2048 x 8192 61 us, two 31).
// The last stage is moved back to end with column m - 1; its columns that were summed before are skipped (m >= 128, a multiple of 32).
template<int ROWS, int DMA_WAVES> constexpr int sgemv_ring_threads() { return 64 * (ROWS / kSgemvRows + DMA_WAVES); }
template<int ROWS, int DMA_WAVES>
__global__ __launch_bounds__((sgemv_ring_threads<ROWS, DMA_WAVES>()))
void sgemvn_ring(int n, int m, float alpha, const float* __restrict__ A, int lda, const float* __restrict__ x, float* __restrict__ y)
{
  constexpr int kStages = 4, kAhead = 2, kCompute = 64 * (ROWS / kSgemvRows), kCols = kSgemvCols / DMA_WAVES;
  static_assert(kAhead < kStages, "a stage is requested when the one before it in its place has long been read");
  __shared__ __attribute__((aligned(1024))) SgemvStage<ROWS> ring[kStages];
  typedef CudaDMAStrided<false, 16, 16, 4 * ROWS, 64, kCols> mat_dma_t;
  typedef CudaDMAStrided<false, 16, 16, 4 * kCols, 64, 1> vec_dma_t;
  constexpr int kLoads = mat_dma_t::loads_per_thread() + vec_dma_t::loads_per_thread();
  static_assert(kLoads * kAhead <= 63, "loads in flight that a wavefront can count");
  HIPDMA_ASSERT(m >= kSgemvCols && (m % kSgemvQuarter) == 0);      // a shorter matrix would have the stage begin before its first column
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int dma = wave < kCompute / 64 ? 0 : wave - kCompute / 64;           // number among the DMA wavefronts
  mat_dma_t dma_mat(4 * lda, 4 * ROWS, kCompute + 64 * dma);
  vec_dma_t dma_vec(4 * kCols, 4 * kCols, kCompute + 64 * dma);
  SgemvGuards<std::make_integer_sequence<int, kStages>> guards(64 * DMA_WAVES, kCompute);
  auto& guard = guards.of;

  const int blocks = (m + kSgemvCols - 1) / kSgemvCols;
  // workgroup b runs on XCD b % 8: every XCD gets a run of row tiles, whose pieces of a column share cache lines and pages with their
  // neighbours; pieces of 256 B are left dealt out (16384 x 16384 184 us, in runs 192)
  const int xcd = blockIdx.x & 7, each = gridDim.x >> 3, more = gridDim.x & 7;
  const int row0 = (ROWS >= 64 ? (int)blockIdx.x : xcd * each + (xcd < more ? xcd : more) + (int)(blockIdx.x >> 3)) * ROWS;
  auto begin = [&](const int b) { const int c = b * kSgemvCols; return c < m - kSgemvCols ? c : m - kSgemvCols; };

  if (wave >= kCompute / 64) {
    auto issue = [&](const int b, const int at) __attribute__((always_inline)) {
      const int col = begin(b) + dma * kCols;
      if (b >= kStages) guard[at].wait_for_dma_start_direct();       // the stages are empty to begin with
      dma_vec.template issue_direct_part<STORE_LDS_DIRECT, true>(x + col, ring[at].vec + dma * kCols, 0, 1);
      dma_mat.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(A + row0 + (long long)lda * col, ring[at].mat + dma * kCols * ROWS, 0, kLoads - 1);
    };
#pragma unroll
    for (int b = 0; b < kAhead; ++b)
      if (b < blocks) issue(b, b);
    auto land = [&](const int b, const int at) __attribute__((always_inline)) {
      if (b >= blocks) return;
      if (b + kAhead <= blocks) hipdma::wait_direct_loads<(kAhead - 1) * kLoads>();
      else hipdma::wait_direct_loads<0>();
      guard[at].finish_async_dma_direct();
      if (b + kAhead < blocks) issue(b + kAhead, (at + kAhead) % kStages);
    };
    for (int b = 0; b < blocks; b += kStages) {
#pragma unroll
      for (int i = 0; i < kStages; ++i) land(b + i, i);
    }
  } else {
    const typename SgemvBlock<ROWS>::Places places(wave, lane);
    SgemvBlock<ROWS> even, odd;
    float res = 0.0f;
    guard[0].wait_for_dma_finish();
    even.load(ring[0], places);
    unsigned seen = guard[1].peek_dma_finish();
    // Block b, in `cur`.  The requests of the next one go out back to back before the chain: in turn with its multiply-adds they
    // take half as long again.
    auto step = [&](const int b, const int at, SgemvBlock<ROWS>& cur, SgemvBlock<ROWS>& next) __attribute__((always_inline)) {
      if (b >= blocks) return;
      guard[at].start_async_dma();        // waits for the requests of `cur`: their stage may be filled again
      if (b + 1 < blocks) {
        guard[(at + 1) % kStages].wait_for_dma_finish(seen);
        next.load(ring[(at + 1) % kStages], places);
        seen = guard[(at + 2) % kStages].peek_dma_finish();
      }
      __builtin_amdgcn_sched_barrier(0);
      res = cur.chain(res, (b * kSgemvCols - begin(b)) / kSgemvQuarter);
      __builtin_amdgcn_sched_barrier(0);
    };
    for (int b = 0; b < blocks; b += kStages) {
#pragma unroll
      for (int i = 0; i < kStages; i += 2) {
        step(b + i, i, even, odd);
        step(b + i + 1, i + 1, odd, even);
      }
    }
    const int row = row0 + wave * kSgemvRows + lane;
    if (lane < kSgemvRows && row < n) y[row] = alpha * res;
  }
}

}  // namespace examples
