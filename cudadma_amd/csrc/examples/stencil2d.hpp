// The five buffering styles of the reference's 2-D stencil example on the wave64
// objects: every z slice of a padded float2 volume is cut into TILE_X x TILE_Y
// tiles, the tile plus its halo is brought into LDS by CudaDMAStrided (one
// strided element per tile row) and the compute threads average a cross of
// neighbours around every cell.
//
// What the reference's example does: src/examples/stencil/
//   warp_specialized_single_buffer.h:26-87, warp_specialized_double_buffer.h:26-107,
//   warp_specialized_manual_buffer.h:26-114, non_warp_specialized_single_buffer.h:26-61,
//   non_warp_specialized_double_buffer.h:24-91, arithmetic stencil_math.h:27-87,
//   launch geometry cudaDMA_stencil2D.cu:99-204.
// The reference gives every workgroup one 32 x 4 tile and lets it march through all
// slices.  Here the work is the list of (slice, tile) pairs, tiles of a slice first,
// and the workgroups of a persistent grid take every gridDim.x-th pair: a volume with
// few tiles per slice then still fills the chip, and the workgroups that run together
// hold neighbouring tiles of the same slices, so a halo row is found in the L2.
#pragma once

#include "../../../include/cudaDMAv2.h"

namespace examples {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// TILE_X x TILE_Y cells of float2 around which RADIUS cells of halo are staged.  A compute thread owns two
// neighbouring cells of ROWS consecutive rows (16 bytes a row): the neighbours above and below come out of LDS
// once per column (ROWS + 2 * reach rows for ROWS results), those to the left and right as two 16-byte reads
// per side.  DMA_THREADS fetch a tile in one step, so every load of a tile is in flight at once.
template<int TILE_X, int TILE_Y, int ROWS, int RADIUS, int DMA_THREADS>
struct StencilTile {
  static_assert(TILE_X % 2 == 0 && TILE_Y % ROWS == 0, "two cells by ROWS rows per compute thread");
  static constexpr int kX = TILE_X, kY = TILE_Y, kThreadRows = ROWS, kRadius = RADIUS;
  static constexpr int kPitch = TILE_X + 2 * RADIUS;
  static constexpr int kRows = TILE_Y + 2 * RADIUS;
  static constexpr int kRowBytes = kPitch * int(sizeof(float2));
  static constexpr int kElmts = kRows * kPitch;
  static constexpr int kComputeThreads = (TILE_X / 2) * (TILE_Y / ROWS);
  static constexpr int kDmaThreads = DMA_THREADS;
  static_assert(kComputeThreads % 64 == 0 && DMA_THREADS % 64 == 0, "groups are whole wavefronts");
  // bytes a thread holds when `threads` threads fetch the tile in one step
  static constexpr int bytes_per_thread(const int threads)
  { return 16 * ((kRows * hipdma::GridPlan::slots(kRowBytes / 16) + threads - 1) / threads); }
};

// The volume and the list of (slice, tile) pairs.  A dimension that the tile does not divide ends with a tile moved
// back to fit: its cells are computed twice, with the same result.
struct StencilGrid {
  int dimx, dimy;
  int tiles_x, tiles_y;
  int offset, row_stride, slice_stride;     // element index of interior point (0, 0, 0); strides in elements
  int items;                                // pairs in all
  int wide_stores;                          // the destination is 16-byte aligned
};

// The pairs of one workgroup: blockIdx.x-th first, then every gridDim.x-th, advanced by additions only.  Workgroup b
// runs on XCD b % 8: where the grid divides, each XCD gets an eighth of the pairs that are in work together, so
// that neighbouring tiles meet in its L2.
template<typename TILE>
struct StencilCursor {
  int item, tx, ty, z;
  __device__ __forceinline__ explicit StencilCursor(const StencilGrid& g)
  {
    int b = blockIdx.x;
    if ((gridDim.x % 8) == 0) b = (b % 8) * (int)(gridDim.x / 8) + b / 8;
    item = b;
    split(g, b, tx, ty, z);
    split(g, (int)gridDim.x, m_tx, m_ty, m_z);
  }
  __device__ __forceinline__ bool valid(const StencilGrid& g) const { return item < g.items; }
  __device__ __forceinline__ void next(const StencilGrid& g)
  {
    item += (int)gridDim.x;
    tx += m_tx;
    ty += m_ty;
    z += m_z;
    if (tx >= g.tiles_x) { tx -= g.tiles_x; ++ty; }
    if (ty >= g.tiles_y) { ty -= g.tiles_y; ++z; }
  }
  // element index of the tile's first cell
  __device__ __forceinline__ long long origin(const StencilGrid& g) const
  {
    const int x = min(tx * TILE::kX, g.dimx - TILE::kX), y = min(ty * TILE::kY, g.dimy - TILE::kY);
    return g.offset + (long long)z * g.slice_stride + (long long)y * g.row_stride + x;
  }
  __device__ __forceinline__ const float2* halo(const StencilGrid& g, const float2* src) const
  { return src + origin(g) - (TILE::kRadius * g.row_stride + TILE::kRadius); }
private:
  __device__ __forceinline__ static void split(const StencilGrid& g, const int i, int& x, int& y, int& s)
  {
    const int row = i / g.tiles_x;
    x = i - row * g.tiles_x;
    s = row / g.tiles_y;
    y = row - s * g.tiles_y;
  }
  int m_tx, m_ty, m_z;
};

// The cross sums of one thread's cells.  REACH neighbours are summed on each of the four arms and the
// sum is divided by 4*RADIUS+1.  The reference's loops stop one short of the radius
// (`d < RADIUS`, stencil_math.h:55-76) while dividing by 4*RADIUS+1 (:82-83); REACH
// = RADIUS-1 reproduces its numbers, REACH = RADIUS is the full cross.  Order of the sum, as there: centre, then the
// left, right, upper and lower arm, each from the inside out.
template<typename TILE, int REACH>
struct StencilSums {
  f32x4_t acc[TILE::kThreadRows];

  __device__ __forceinline__ static int column() { return 2 * (int)(threadIdx.x % (TILE::kX / 2)); }
  __device__ __forceinline__ static int first_row() { return TILE::kThreadRows * (int)(threadIdx.x / (TILE::kX / 2)); }

  __device__ __forceinline__ void sum(const float2* buffer)
  {
    constexpr int R = TILE::kRadius, N = TILE::kThreadRows, kPitch = TILE::kPitch;
    static_assert(R == 4, "the side arms are two 16-byte reads");
    const float2* centre = buffer + (first_row() + R) * kPitch + (column() + R);
    f32x4_t col[N + 2 * REACH];
#pragma unroll
    for (int i = 0; i < N + 2 * REACH; ++i) col[i] = *(const f32x4_t*)(centre + (i - REACH) * kPitch);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const float2* row = centre + i * kPitch;
      const f32x4_t l2 = *(const f32x4_t*)(row - 4), l1 = *(const f32x4_t*)(row - 2);
      const f32x4_t r1 = *(const f32x4_t*)(row + 2), r2 = *(const f32x4_t*)(row + 4);
      const f32x4_t c = col[i + REACH];
      // cells x-4 .. x+5 of the row, x and y components
      const float xs[10] = {l2[0], l2[2], l1[0], l1[2], c[0], c[2], r1[0], r1[2], r2[0], r2[2]};
      const float ys[10] = {l2[1], l2[3], l1[1], l1[3], c[1], c[3], r1[1], r1[3], r2[1], r2[3]};
      f32x4_t a = c;
#pragma unroll
      for (int d = 1; d <= REACH; ++d) a += f32x4_t{xs[4 - d], ys[4 - d], xs[5 - d], ys[5 - d]};
#pragma unroll
      for (int d = 1; d <= REACH; ++d) a += f32x4_t{xs[4 + d], ys[4 + d], xs[5 + d], ys[5 + d]};
#pragma unroll
      for (int d = 1; d <= REACH; ++d) a += col[i + REACH - d];
#pragma unroll
      for (int d = 1; d <= REACH; ++d) a += col[i + REACH + d];
      acc[i] = a;
    }
  }
  // dst: the tile's first cell
  __device__ __forceinline__ void store(const StencilGrid& g, float2* dst) const
  {
    float2* o = dst + (long long)first_row() * g.row_stride + column();
#pragma unroll
    for (int i = 0; i < TILE::kThreadRows; ++i) {
      const f32x4_t a = acc[i] / float(4 * TILE::kRadius + 1);
      if (g.wide_stores) {
        __builtin_nontemporal_store(a, (f32x4_t*)o);
      } else {
        o[0] = make_float2(a[0], a[1]);
        o[1] = make_float2(a[2], a[3]);
      }
      o += g.row_stride;
    }
  }
};

#define HIPDMA_STENCIL2D_ARGS \
  const float2* __restrict__ src_buffer, float2* __restrict__ dst_buffer, const StencilGrid g

// One buffer, one DMA group.  Launch kComputeThreads + kDmaThreads threads.
template<typename TILE, int REACH>
__global__ void __launch_bounds__(TILE::kComputeThreads + TILE::kDmaThreads)
stencil_2D_warp_specialized_single_buffer(HIPDMA_STENCIL2D_ARGS)
{
  __shared__ __attribute__((aligned(16))) float2 buffer[TILE::kElmts];
  CudaDMAStrided<true, 16, TILE::bytes_per_thread(TILE::kDmaThreads), TILE::kRowBytes, TILE::kDmaThreads, TILE::kRows>
    dma_ld(0, TILE::kComputeThreads, TILE::kComputeThreads, g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  StencilCursor<TILE> at(g);
  if (dma_ld.owns_this_thread()) {
    for (; at.valid(g); at.next(g))
      dma_ld.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(at.halo(g, src_buffer), buffer);
  } else {
    dma_ld.start_async_dma();
    while (at.valid(g)) {
      float2* dst = dst_buffer + at.origin(g);
      at.next(g);
      StencilSums<TILE, REACH> s;
      dma_ld.wait_for_dma_finish();
      s.sum(buffer);
      if (at.valid(g)) dma_ld.start_async_dma();
      s.store(g, dst);
    }
  }
}

// Two buffers, two DMA groups on disjoint wavefronts; a workgroup's pairs go through the buffers in turn.
// Launch kComputeThreads + 2*kDmaThreads threads.
template<typename TILE, int REACH>
__global__ void __launch_bounds__(TILE::kComputeThreads + 2 * TILE::kDmaThreads)
stencil_2D_warp_specialized_double_buffer(HIPDMA_STENCIL2D_ARGS)
{
  __shared__ __attribute__((aligned(16))) float2 buffer0[TILE::kElmts];
  __shared__ __attribute__((aligned(16))) float2 buffer1[TILE::kElmts];
  typedef CudaDMAStrided<true, 16, TILE::bytes_per_thread(TILE::kDmaThreads), TILE::kRowBytes, TILE::kDmaThreads, TILE::kRows> dma_t;
  dma_t dma_ld0(0, TILE::kComputeThreads, TILE::kComputeThreads, g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  dma_t dma_ld1(1, TILE::kComputeThreads, TILE::kComputeThreads + TILE::kDmaThreads, g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  StencilCursor<TILE> at(g);
  if (dma_ld0.owns_this_thread()) {
    for (; at.valid(g); at.next(g), at.next(g))
      dma_ld0.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(at.halo(g, src_buffer), buffer0);
  } else if (dma_ld1.owns_this_thread()) {
    for (at.next(g); at.valid(g); at.next(g), at.next(g))
      dma_ld1.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(at.halo(g, src_buffer), buffer1);
  } else {
    dma_ld0.start_async_dma();
    dma_ld1.start_async_dma();
    auto one = [&](const dma_t& dma, const float2* buffer) __attribute__((always_inline)) {
      float2* dst = dst_buffer + at.origin(g);
      at.next(g);
      StencilSums<TILE, REACH> s;
      dma.wait_for_dma_finish();
      s.sum(buffer);
      dma.start_async_dma();
      s.store(g, dst);
    };
    while (at.valid(g)) {
      one(dma_ld0, buffer0);
      if (at.valid(g)) one(dma_ld1, buffer1);
    }
  }
}

// Two buffers, two objects that share ONE DMA group; the group keeps the loads of
// both objects in flight through the two-phase calls.  Launch kComputeThreads + kDmaThreads threads.
template<typename TILE, int REACH>
__global__ void __launch_bounds__(TILE::kComputeThreads + TILE::kDmaThreads)
stencil_2D_warp_specialized_manual_buffer(HIPDMA_STENCIL2D_ARGS)
{
  __shared__ __attribute__((aligned(16))) float2 buffer0[TILE::kElmts];
  __shared__ __attribute__((aligned(16))) float2 buffer1[TILE::kElmts];
  typedef CudaDMAStrided<true, 16, TILE::bytes_per_thread(TILE::kDmaThreads), TILE::kRowBytes, TILE::kDmaThreads, TILE::kRows> dma_t;
  dma_t dma_ld0(0, TILE::kComputeThreads, TILE::kComputeThreads, g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  dma_t dma_ld1(1, TILE::kComputeThreads, TILE::kComputeThreads, g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  StencilCursor<TILE> at(g);
  if (dma_ld0.owns_this_thread()) {
    // `at` runs one pair ahead of the pair that lands
    auto request = [&](dma_t& dma) __attribute__((always_inline)) {
      const bool there = at.valid(g);
      if (there) dma.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(at.halo(g, src_buffer));
      at.next(g);
      return there;
    };
    bool first = request(dma_ld0), second = request(dma_ld1);
    while (first) {
      dma_ld0.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buffer0);
      first = request(dma_ld0);
      if (!second) break;
      dma_ld1.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buffer1);
      second = request(dma_ld1);
    }
  } else {
    dma_ld0.start_async_dma();
    dma_ld1.start_async_dma();
    auto one = [&](const dma_t& dma, const float2* buffer) __attribute__((always_inline)) {
      float2* dst = dst_buffer + at.origin(g);
      at.next(g);
      StencilSums<TILE, REACH> s;
      dma.wait_for_dma_finish();
      s.sum(buffer);
      dma.start_async_dma();
      s.store(g, dst);
    };
    while (at.valid(g)) {
      one(dma_ld0, buffer0);
      if (at.valid(g)) one(dma_ld1, buffer1);
    }
  }
}

// No specialisation: every thread transfers, then every thread computes; one buffer
// and two workgroup barriers per pair.  Launch kComputeThreads threads.
template<typename TILE, int REACH>
__global__ void __launch_bounds__(TILE::kComputeThreads)
stencil_2D_non_warp_specialized_single_buffer(HIPDMA_STENCIL2D_ARGS)
{
  __shared__ __attribute__((aligned(16))) float2 buffer[TILE::kElmts];
  CudaDMAStrided<false, 16, TILE::bytes_per_thread(TILE::kComputeThreads), TILE::kRowBytes, TILE::kComputeThreads, TILE::kRows>
    dma_ld(g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  for (StencilCursor<TILE> at(g); at.valid(g); at.next(g)) {
    dma_ld.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(at.halo(g, src_buffer), buffer);
    __syncthreads();                       // buffer full
    StencilSums<TILE, REACH> s;
    s.sum(buffer);
    __syncthreads();                       // buffer free again
    s.store(g, dst_buffer + at.origin(g));
  }
}

// No specialisation, two buffers and two objects: the loads of the pair after next
// are in flight (held in registers by the two-phase calls) while a pair is consumed,
// one barrier per pair.  Launch kComputeThreads threads.
template<typename TILE, int REACH>
__global__ void __launch_bounds__(TILE::kComputeThreads)
stencil_2D_non_warp_specialized_double_buffer(HIPDMA_STENCIL2D_ARGS)
{
  __shared__ __attribute__((aligned(16))) float2 buffer0[TILE::kElmts];
  __shared__ __attribute__((aligned(16))) float2 buffer1[TILE::kElmts];
  typedef CudaDMAStrided<false, 16, TILE::bytes_per_thread(TILE::kComputeThreads), TILE::kRowBytes, TILE::kComputeThreads, TILE::kRows> dma_t;
  dma_t dma_ld0(g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  dma_t dma_ld1(g.row_stride * int(sizeof(float2)), TILE::kRowBytes);
  StencilCursor<TILE> at(g), ahead(g);     // `ahead`: the next pair to request
  auto request = [&](dma_t& dma) __attribute__((always_inline)) {
    if (ahead.valid(g)) dma.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(ahead.halo(g, src_buffer));
    ahead.next(g);
  };
  auto one = [&](dma_t& dma, float2* buffer) __attribute__((always_inline)) {
    float2* dst = dst_buffer + at.origin(g);
    at.next(g);
    dma.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buffer);
    request(dma);
    __syncthreads();
    StencilSums<TILE, REACH> s;
    s.sum(buffer);
    s.store(g, dst);
  };
  request(dma_ld0);
  request(dma_ld1);
  while (at.valid(g)) {
    one(dma_ld0, buffer0);
    if (at.valid(g)) one(dma_ld1, buffer1);
  }
}

#undef HIPDMA_STENCIL2D_ARGS

}  // namespace examples
