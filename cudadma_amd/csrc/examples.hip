// C-ABI launchers of the example consumers (saxpy, sgemv, 2-D stencil) that the
// reference ships under src/examples/; the kernels themselves live in
// examples/*.hpp and are written against the DMA classes only.
#include "common.hpp"
#include "workloads.hpp"
#include "examples/saxpy.hpp"
#include "examples/sgemv.hpp"
#include "examples/stencil2d.hpp"

namespace {

using namespace examples;

// ---- saxpy ----
constexpr int kSaxpyCompute = 256;          // four compute wavefronts
constexpr int kSaxpyDmaPerLd = 64;          // one wavefront per staged vector and buffer
const char* const kSaxpyNames[] = {
  "baseline: one element per thread, no LDS",
  "vec4: dwordx4 per thread, no LDS",
  "cudaDMASequential x2, one buffer per vector",
  "cudaDMASequential x4, two buffers per vector",
};

// ---- sgemv ----
constexpr int kGemvCompute = 128;
constexpr int kGemvDmaPerLd = 64;
constexpr int kGemvVecElmts = 256;          // columns per hand-off when only the vector is staged
constexpr int kGemvPanelCols = 32;          // columns per hand-off when the matrix panel is staged too (variant 3: the unit of m)
constexpr int kGemvMatLds = 2;              // DMA wavefronts on the matrix panel
const char* const kGemvNames[] = {
  "vector staged by cudaDMASequential, one buffer",
  "vector staged by two cudaDMASequential on shared DMA threads",
  "vector by cudaDMASequential + 32-column panel by cudaDMAStrided, one buffer each",
  "vector and matrix in a ring of four stages of 128 columns by direct-to-LDS CudaDMAStrided; 32-column panels, two buffers each, for narrow matrices and for many rows",
};

template<int ROWS, int MAT_DMA, int MAT_BYTES = 4 * ROWS * kGemvPanelCols / MAT_DMA>
void launch_sgemv_small_panels(hipStream_t s, int n, int m, float alpha, const float* a, int lda, const float* x, float* y)
{
  hipLaunchKernelGGL((sgemvn_both_double<ROWS, kGemvPanelCols, kGemvDmaPerLd, MAT_DMA, MAT_BYTES>), dim3((n + ROWS - 1) / ROWS),
                     dim3((sgemv_both_double_threads<ROWS, kGemvDmaPerLd, MAT_DMA>())), 0, s, n, m, alpha, a, lda, x, y);
}

template<int ROWS, int DMA_WAVES>
void launch_sgemv_ring(hipStream_t s, int n, int m, float alpha, const float* a, int lda, const float* x, float* y)
{
  hipLaunchKernelGGL((sgemvn_ring<ROWS, DMA_WAVES>), dim3((n + ROWS - 1) / ROWS), dim3((sgemv_ring_threads<ROWS, DMA_WAVES>())), 0, s,
                     n, m, alpha, a, lda, x, y);
}

// A row is one chain of multiply-adds whatever the tile, and sixteen rows per compute wavefront are what gives every chain a SIMD of its
// own; what the rows of a workgroup decide is how long the pieces of a column are that come from memory.  us, ring of 16 / 32 / 64 rows,
// from the caches and from DRAM:
//   4096 x 4096   17.2 / 18.4 / 22.5 and 19.5 / 19.9 / 26.9   (one workgroup of 16 rows per compute unit)
//   6000 x 2048   12.0 / 10.4 / 12.3 and 17.0 / 12.0 / 15.2   8192 x 8192   48 / 44 / 40 and 68 / 50 / 58
//   9000 x 512    5.4 / 6.0 / 5.8 and 8.5 / 7.8 / 7.1         16384 x 1024  15.3 / 14.7 / 13.7 and 19.3 / 16.4 / 14.3
// Two stages are over before a wide workgroup has started up: with fewer than 256 columns sixteen rows go further (8209 x 128 3.0 / 3.6 /
// 3.7 and 3.6 / 3.9 / 4.1).  The ring needs the columns of one stage, and its loads reach sixteen columns by 32-bit lane offsets.
// Narrower matrices and longer leading dimensions go through small panels, and so do those with more rows than 64 per compute
// unit: several workgroups then share a compute unit and hide each other's hand-offs (20480 x 4096 64 us, ring of 64 rows 72; 32768 x 4096 85 and
// 95), and narrow ones from 40 on (12288 x 224 from DRAM 5.7, ring of 16 rows 6.3).
// With 256 to about 300 columns and more than 32 rows per compute unit no shape is ahead in both states (10496 x 256: rings 3.8 / 4.6 / 4.5 and 6.4 / 6.2 /
// 5.7, panels of 32 columns 5.3 and 6.1; a lane per row with panels of 128 columns 4.3 and 5.9).
// From 112 rows on the longer pieces of 128 rows count, in bursts of 64 bytes a thread (64 / 128 rows: 32768 x 2048 42 / 39 us, 98304 x 1024
// 76 / 72).
void launch_sgemv_double(hipStream_t s, int n, int m, float alpha, const float* a, int lda, const float* x, float* y)
{
  const int cus = workloads::device_cus();
  const bool ring = m >= kSgemvCols && lda <= (0xffffffffLL - 4 * kSgemvRows) / (4 * kSgemvRows) && n <= (m < 2 * kSgemvCols ? 40 : 64) * cus;
  if (n > 112 * cus) launch_sgemv_small_panels<kGemvCompute, kGemvMatLds * kGemvDmaPerLd, 64>(s, n, m, alpha, a, lda, x, y);
  else if (!ring) launch_sgemv_small_panels<64, 64>(s, n, m, alpha, a, lda, x, y);
  else if (n <= 16 * cus || m < 2 * kSgemvCols) launch_sgemv_ring<16, 2>(s, n, m, alpha, a, lda, x, y);
  else if (n <= 32 * cus) launch_sgemv_ring<32, 2>(s, n, m, alpha, a, lda, x, y);
  else launch_sgemv_ring<64, 4>(s, n, m, alpha, a, lda, x, y);
}

// ---- 2-D stencil ----
constexpr int kUnitX = 32, kUnitY = 4, kRadius = 4;     // the dimensions are multiples of the reference's tile
const char* const kStencilNames[] = {
  "warp specialized, single buffer",
  "warp specialized, double buffer",
  "warp specialized, manual buffer",
  "non warp specialized, single buffer",
  "non warp specialized, double buffer",
};

template<typename TILE, int REACH>
void launch_stencil(int variant, hipStream_t s, const float2* src, float2* dst, examples::StencilGrid g, int dimz)
{
  g.tiles_x = (g.dimx + TILE::kX - 1) / TILE::kX;
  g.tiles_y = (g.dimy + TILE::kY - 1) / TILE::kY;
  g.items = g.tiles_x * g.tiles_y * dimz;
  // As many workgroups as share the pairs evenly, in whole rounds over the eight XCDs, up to `per_cu` per compute unit: one
  // 23 KiB tile of loads in flight is what volumes beyond the caches run best with (960 x 160 x 200: 95 us with one
  // workgroup per compute unit, 113 / 128 / 120 with two / three / four), and with the flat tile (9 KiB) four of them (133 / 98 /
  // 130 us with two / four / six).
  const int per_cu = TILE::kY >= 32 ? 1 : 4;
  const int most = workloads::persistent_grid(g.items, per_cu);
  const int rounds = (g.items + most - 1) / most;
  int grid = (g.items + rounds - 1) / rounds;
  if (grid > 8) grid = (grid + 7) / 8 * 8;
  const dim3 blocks((unsigned)grid);
  constexpr int kCompute = TILE::kComputeThreads, kDma = TILE::kDmaThreads;
  switch (variant) {
    case 0: hipLaunchKernelGGL((stencil_2D_warp_specialized_single_buffer<TILE, REACH>), blocks, dim3(kCompute + kDma), 0, s, src, dst, g); break;
    case 1: hipLaunchKernelGGL((stencil_2D_warp_specialized_double_buffer<TILE, REACH>), blocks, dim3(kCompute + 2 * kDma), 0, s, src, dst, g); break;
    case 2: hipLaunchKernelGGL((stencil_2D_warp_specialized_manual_buffer<TILE, REACH>), blocks, dim3(kCompute + kDma), 0, s, src, dst, g); break;
    case 3: hipLaunchKernelGGL((stencil_2D_non_warp_specialized_single_buffer<TILE, REACH>), blocks, dim3(kCompute), 0, s, src, dst, g); break;
    default: hipLaunchKernelGGL((stencil_2D_non_warp_specialized_double_buffer<TILE, REACH>), blocks, dim3(kCompute), 0, s, src, dst, g); break;
  }
}

typedef StencilTile<64, 32, 4, kRadius, 128> LargeTile;
typedef StencilTile<64, 8, 2, kRadius, 64> FlatTile;
typedef StencilTile<32, 4, 1, kRadius, 64> SmallTile;

template<int REACH>
void launch_stencil(int variant, hipStream_t s, const float2* src, float2* dst, const examples::StencilGrid& g, int dimz)
{
  // Tall tiles read 1.4 cells per cell computed, flat ones 2.25, most of them from the L2: worth 3 to 8 % once the volume
  // lies beyond the Infinity Cache (960 x 160 x 200: 95 against 98 us, 512 x 512 x 100: 80 against 85).  Where the caches hold
  // it the flat tiles spread the work better (128 x 512 x 58: 14.7 against 16.9 us), and where 32 does not divide the height the
  // rows computed twice cost more (960 x 164 x 100: 53 against 58 us).
  const bool beyond_caches = 16LL * g.dimx * g.dimy * dimz > (192LL << 20);
  const bool even = (g.dimy + 31) / 32 * 32 == (g.dimy + 7) / 8 * 8;
  if (g.dimx >= 64 && g.dimy >= 32 && beyond_caches && even) launch_stencil<LargeTile, REACH>(variant, s, src, dst, g, dimz);
  else if (g.dimx >= 64 && g.dimy >= 8) launch_stencil<FlatTile, REACH>(variant, s, src, dst, g, dimz);
  else launch_stencil<SmallTile, REACH>(variant, s, src, dst, g, dimz);
}

template<typename T, int N> constexpr int count_of(T (&)[N]) { return N; }

}  // namespace

extern "C" int cudadma_example_num_variants(int example)
{
  switch (example) {
    case CUDADMA_EXAMPLE_SAXPY: return count_of(kSaxpyNames);
    case CUDADMA_EXAMPLE_SGEMV: return count_of(kGemvNames);
    case CUDADMA_EXAMPLE_STENCIL2D: return count_of(kStencilNames);
    default: return 0;
  }
}

extern "C" const char* cudadma_example_variant_name(int example, int variant)
{
  if (variant < 0 || variant >= cudadma_example_num_variants(example)) return nullptr;
  switch (example) {
    case CUDADMA_EXAMPLE_SAXPY: return kSaxpyNames[variant];
    case CUDADMA_EXAMPLE_SGEMV: return kGemvNames[variant];
    default: return kStencilNames[variant];
  }
}

extern "C" int cudadma_example_saxpy(int variant, float a, const float* d_x, float* d_y, long long n, void* stream)
{
  if (variant < 0 || variant >= count_of(kSaxpyNames)) {
    cudadma_host::set_error("saxpy has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  constexpr int kChunk = SaxpyChunk<kSaxpyCompute>::kFloats;
  CUDADMA_REQUIRE(n >= 0, "n (%lld) is negative", n);
  CUDADMA_REQUIRE(variant == 0 || (n % kChunk) == 0, "n (%lld) must be a multiple of %d floats for this variant", n, kChunk);
  if (n == 0) return CUDADMA_OK;
  CUDADMA_REQUIRE(d_x != nullptr && d_y != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_x, 16) && cudadma_host::aligned_to(d_y, 16), "pointers must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const long long chunks = (n + kChunk - 1) / kChunk;
  const int grid = workloads::persistent_grid(chunks, 4);
  switch (variant) {
    case 0: hipLaunchKernelGGL(saxpy_baseline, dim3(grid), dim3(kSaxpyCompute), 0, s, d_y, d_x, a, n); break;
    case 1: hipLaunchKernelGGL(saxpy_vec4, dim3(grid), dim3(kSaxpyCompute), 0, s, d_y, d_x, a, n); break;
    case 2:
      hipLaunchKernelGGL((saxpy_dma_single<kSaxpyCompute, kSaxpyDmaPerLd>), dim3(grid), dim3(kSaxpyCompute + 2 * kSaxpyDmaPerLd),
                         0, s, d_y, d_x, a, chunks);
      break;
    default:
      hipLaunchKernelGGL((saxpy_dma_double<kSaxpyCompute, kSaxpyDmaPerLd>), dim3(grid), dim3(kSaxpyCompute + 4 * kSaxpyDmaPerLd),
                         0, s, d_y, d_x, a, chunks);
      break;
  }
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

extern "C" int cudadma_example_sgemv(int variant, int n, int m, float alpha, const float* d_a, int lda, const float* d_x,
                                     float* d_y, void* stream)
{
  if (variant < 0 || variant >= count_of(kGemvNames)) {
    cudadma_host::set_error("sgemv has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  CUDADMA_REQUIRE(n >= 0 && m >= 0, "negative dimension (n %d, m %d)", n, m);
  CUDADMA_REQUIRE(lda >= n, "lda (%d) is smaller than n (%d)", lda, n);
  if (n == 0) return CUDADMA_OK;
  CUDADMA_REQUIRE(d_a != nullptr && d_x != nullptr && d_y != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_x, 16), "x must be 16-byte aligned");
  // the objects that stage the matrix take the distance of two columns as an int
  CUDADMA_REQUIRE(variant < 2 || lda <= 0x7fffffff / 4, "lda (%d) must not exceed %d when the matrix is staged", lda, 0x7fffffff / 4);
  const int grid = (n + kGemvCompute - 1) / kGemvCompute;
  const int cols = variant == 0 ? kGemvVecElmts : variant == 1 ? 2 * kGemvVecElmts : kGemvPanelCols;
  CUDADMA_REQUIRE(m > 0 && (m % cols) == 0, "m (%d) must be a positive multiple of %d for this variant", m, cols);
  if (variant >= 2) {
    // the panel transfer reads whole groups of kGemvCompute rows with dwordx4 loads
    CUDADMA_REQUIRE(lda >= grid * kGemvCompute, "lda (%d) must cover %d rows (n rounded up to %d) when the matrix is staged",
                    lda, grid * kGemvCompute, kGemvCompute);
    CUDADMA_REQUIRE((lda % 4) == 0 && cudadma_host::aligned_to(d_a, 16), "A and lda*4 must be 16-byte aligned when the matrix is staged");
  }
  hipStream_t s = (hipStream_t)stream;
  switch (variant) {
    case 0:
      hipLaunchKernelGGL((sgemvn_vec_single<kGemvCompute, kGemvDmaPerLd, kGemvVecElmts>), dim3(grid),
                         dim3(kGemvCompute + kGemvDmaPerLd), 0, s, n, m, alpha, d_a, lda, d_x, d_y);
      break;
    case 1:
      hipLaunchKernelGGL((sgemvn_vec_manual<kGemvCompute, kGemvDmaPerLd, kGemvVecElmts>), dim3(grid),
                         dim3(kGemvCompute + kGemvDmaPerLd), 0, s, n, m, alpha, d_a, lda, d_x, d_y);
      break;
    case 2:
      hipLaunchKernelGGL((sgemvn_both_single<kGemvCompute, kGemvDmaPerLd, kGemvPanelCols, kGemvMatLds>), dim3(grid),
                         dim3(kGemvCompute + (1 + kGemvMatLds) * kGemvDmaPerLd), 0, s, n, m, alpha, d_a, lda, d_x, d_y);
      break;
    default: launch_sgemv_double(s, n, m, alpha, d_a, lda, d_x, d_y); break;
  }
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

extern "C" int cudadma_example_stencil2d(int variant, const float* d_src, float* d_dst, int dimx, int dimy, int dimz,
                                         int full_cross, void* stream)
{
  if (variant < 0 || variant >= count_of(kStencilNames)) {
    cudadma_host::set_error("stencil2d has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  CUDADMA_REQUIRE(dimx > 0 && dimy > 0 && dimz > 0, "dimensions must be positive (%d x %d x %d)", dimx, dimy, dimz);
  CUDADMA_REQUIRE((dimx % kUnitX) == 0 && (dimy % kUnitY) == 0, "dimx must be a multiple of %d and dimy of %d", kUnitX, kUnitY);
  CUDADMA_REQUIRE(variant == 0 || variant == 3 || (dimz % 2) == 0, "dimz (%d) must be even for the variants with two buffers", dimz);
  CUDADMA_REQUIRE(d_src != nullptr && d_dst != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_src, 16) && cudadma_host::aligned_to(d_dst, 8), "src must be 16-byte, dst 8-byte aligned");
  const long long row_stride = dimx + 2 * kRadius;
  const long long slice_stride = (dimy + 2 * kRadius) * row_stride;
  const long long offset = kRadius * slice_stride + kRadius * row_stride + kRadius;
  CUDADMA_REQUIRE(slice_stride * (dimz + 2 * kRadius) <= 0x7fffffffLL / 8, "volume too large for int element offsets");
  hipStream_t s = (hipStream_t)stream;
  const float2* src = reinterpret_cast<const float2*>(d_src);
  float2* dst = reinterpret_cast<float2*>(d_dst);
  const examples::StencilGrid g = {dimx, dimy, 0, 0, (int)offset, (int)row_stride, (int)slice_stride, 0, cudadma_host::aligned_to(d_dst, 16)};
  if (full_cross) launch_stencil<kRadius>(variant, s, src, dst, g, dimz);
  else launch_stencil<kRadius - 1>(variant, s, src, dst, g, dimz);
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}
