// Config 4: 8th-order, 25-point star stencil over a 3-D grid, 32x32 tiles
// marched along z.  The buffering idioms are those of
// src/examples/stencil/warp_specialized_double_buffer.h:25-106 and
// src/examples/stencil/non_warp_specialized_single_buffer.h:34-58; the ring of
// ghost cells comes through CudaDMAHalo (include/cudaDMA.h:3653-4156), the
// stencil itself is the textbook one, not stencil_math.h.
//
// Per output plane z a compute thread owns four cells of the tile.  Their z
// neighbours live in a 9-deep register queue fed by one coalesced global load
// per cell and plane; the centre plane is shared through LDS: the interior is
// written by the compute threads themselves, the 4-wide ring around it by the
// DMA wavefront.  Two LDS planes alternate so the ring of plane z+1 lands
// while plane z is being computed.
#include "workloads.hpp"

namespace {

constexpr int kR = 4;
#ifndef STENCIL_TX
#define STENCIL_TX 32
#define STENCIL_TY 32
#endif
constexpr int kTX = STENCIL_TX, kTY = STENCIL_TY;    // 32 x 32, or 64 x 16 (rows of 256 B instead of 128 B)
static_assert((kTX == 32 && kTY == 32) || (kTX == 64 && kTY == 16), "tile_row_of_thread() knows these two shapes");
constexpr int kPitch = kTX + 2 * kR;                 // 40 (72) floats per LDS row
constexpr int kPlaneFloats = kPitch * (kTY + 2 * kR);
constexpr int kComputeThreads = 256;
constexpr int kDmaThreads = 64;
constexpr int kCells = kTX * kTY / kComputeThreads;   // 4 cells per compute thread
constexpr int kRowsPerPass = kComputeThreads / kTX;   // 8

// ring of a 32x32 float tile: 8 rows x 8 chunks + 64 strips x 1 chunk = 128 chunks of 16 B = 2 per DMA thread
constexpr int kRingChunks = (2 * kR * kTX + 2 * kR * kTY) * 4 / 16;                    // 128 (160) chunks of 16 B
constexpr int kRingBpt = 16 * ((kRingChunks + kDmaThreads - 1) / kDmaThreads);        // whole ring in one step
typedef CudaDMAHalo<true, 16, kRingBpt, 4, kDmaThreads, kR, false, kTX, kTY> halo_ws_t;
typedef CudaDMAHalo<false, 16, 16, 4, kComputeThreads, kR, false, kTX, kTY> halo_all_t;

struct Coeffs {
  float c0, c1, c2, c3, c4;
};

// One cell: same operations in the same order as the host statement.
__device__ __forceinline__ float stencil_cell(const float* __restrict__ plane, const int lx, const int ly,
                                              const float (&q)[2 * kR + 1], const Coeffs& k)
{
#pragma clang fp contract(off)
  const float* c = plane + (ly + kR) * kPitch + (lx + kR);
  const float cr[5] = {0.0f, k.c1, k.c2, k.c3, k.c4};
  float acc = k.c0 * q[kR];
#pragma unroll
  for (int r = 1; r <= kR; ++r) {
    const float sx = c[-r] + c[r];
    const float sy = c[-r * kPitch] + c[r * kPitch];
    const float sz = q[kR - r] + q[kR + r];
    acc = __builtin_fmaf(cr[r], (sx + sy) + sz, acc);
  }
  return acc;
}

struct TileWork {
  const float* in_origin;   // first interior cell of the tile in padded plane 0 of the z-chunk
  float* out_origin;        // first cell of the tile in output plane z0
  int planes;               // output planes in this chunk
};

// `zchunk` carries the chunk length in its low 24 bits; bit 24 asks for the
// XCD-aware numbering: workgroup b runs on XCD b % 8 (8 XCDs, round-robin
// dispatch), so giving XCD k the k-th eighth of the tile list keeps tiles that
// share ghost cells behind the same L2.  That eighth is a slab over the whole
// width of the grid (two tile rows at 512^3): the only ghost cells two XCDs both
// read from memory are the rows above and below a slab, 8 rows on 64 (reads
// 1.16 x the grid, reads + writes 1.08 x).  Bit 25 (one z-chunk, tile grid divisible
// by 2 x 4) makes it a compact block instead, half of the tiles in x by a quarter
// in y.  Its rim is shorter in cells, but not in cache lines: the 16 bytes of ghost
// cells on the inner side of a 1 KiB row piece cost a whole 128-byte line per row,
// and the measured traffic is higher (reads 1.21 x, total 1.11 x) at the same or a
// slightly shorter time; the slabs stay the default.
constexpr int kXcdFlag = 1 << 24;
constexpr int kXcdBlockFlag = 1 << 25;
constexpr int kXcds = 8;

__device__ __forceinline__ TileWork tile_work(const float* in, float* out, const int nx, const int ny, const int nz,
                                              const int zchunk_and_flags)
{
  const int zchunk = zchunk_and_flags & (kXcdFlag - 1);
  const int tiles_x = nx / kTX, tiles_y = ny / kTY;
  int b = blockIdx.x;
  int tx, ty;
  if (zchunk_and_flags & kXcdBlockFlag) {
    // XCD k = (kx, ky) of a 2 x 4 arrangement owns the block of tiles_x/2 x tiles_y/4 tiles at (kx, ky)
    const int xcd = b % kXcds, slot = b / kXcds;
    const int bw = tiles_x / 2, bh = tiles_y / 4;
    tx = (xcd % 2) * bw + slot % bw;
    ty = (xcd / 2) * bh + slot / bw;
    b = 0;
  } else {
    if (zchunk_and_flags & kXcdFlag) {
      // a contiguous run of tiles for each XCD; where eight does not divide the grid the first ones get a tile more
      // (224 x 416 x 300, 273 workgroups: 71 us without the renumbering, 48 with it)
      const int xcd = b % kXcds, each = (int)gridDim.x / kXcds, more = (int)gridDim.x % kXcds;
      b = xcd * each + (xcd < more ? xcd : more) + b / kXcds;
    }
    tx = b % tiles_x; b /= tiles_x;
    ty = b % tiles_y; b /= tiles_y;
  }
  const int z0 = b * zchunk;
  const size_t px = (size_t)nx + 2 * kR, py = (size_t)ny + 2 * kR;
  TileWork w;
  w.in_origin = in + ((size_t)z0 * py + (size_t)(ty * kTY + kR)) * px + (size_t)(tx * kTX + kR);
  w.out_origin = out + ((size_t)z0 * ny + (size_t)ty * kTY) * nx + (size_t)tx * kTX;
  w.planes = (nz - z0 < zchunk) ? (nz - z0) : zchunk;
  return w;
}

#ifdef HIPDMA_SWEEP_VARIANTS
__global__ void __launch_bounds__(kComputeThreads + kDmaThreads)
stencil_warp_specialized(const float* __restrict__ in, float* __restrict__ out, const int nx, const int ny,
                         const int nz, const int zchunk, const Coeffs k)
{
  __shared__ __attribute__((aligned(16))) float plane[2][kPlaneFloats];
  const int px = nx + 2 * kR;
  const size_t in_plane = (size_t)px * (size_t)(ny + 2 * kR);
  const size_t out_plane = (size_t)nx * ny;
  halo_ws_t halo0(0, kComputeThreads, kComputeThreads, px);
  halo_ws_t halo1(1, kComputeThreads, kComputeThreads, px);
  hipdma::GroupBarrier compute_barrier(2, kComputeThreads);
  const TileWork w = tile_work(in, out, nx, ny, nz, zchunk);
  float* lds_origin0 = &plane[0][kR * kPitch + kR];
  float* lds_origin1 = &plane[1][kR * kPitch + kR];

  if (halo0.owns_this_thread()) {
    // centre plane of output plane z is padded plane z + kR
    const float* src = w.in_origin + (size_t)kR * in_plane;
    for (int z = 0; z < w.planes; z += 2) {
      halo0.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(src, lds_origin0);
      src += in_plane;
      if (z + 1 < w.planes) halo1.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(src, lds_origin1);
      src += in_plane;
    }
  } else {
    const int lx = threadIdx.x % kTX;
    const int ly = threadIdx.x / kTX;
    float q[kCells][2 * kR + 1];
    const float* col = w.in_origin + (size_t)ly * px + lx;
#pragma unroll
    for (int i = 0; i < kCells; ++i)
#pragma unroll
      for (int p = 0; p < 2 * kR; ++p) q[i][p + 1] = col[(size_t)p * in_plane + (size_t)(i * kRowsPerPass) * px];
    halo0.start_async_dma();
    halo1.start_async_dma();
    // interior of the first centre plane
#pragma unroll
    for (int i = 0; i < kCells; ++i) lds_origin0[(ly + i * kRowsPerPass) * kPitch + lx] = q[i][kR + 1];
    const float* next = col + (size_t)(2 * kR) * in_plane;
    float* o = w.out_origin + (size_t)ly * nx + lx;

    auto one_plane = [&](const float* cur_plane, float* other_origin, const halo_ws_t& cur_halo, const bool last)
        __attribute__((always_inline)) {
      // slide the queue and fetch the newest plane
#pragma unroll
      for (int i = 0; i < kCells; ++i) {
#pragma unroll
        for (int p = 0; p < 2 * kR; ++p) q[i][p] = q[i][p + 1];
        q[i][2 * kR] = next[(size_t)(i * kRowsPerPass) * px];
      }
      next += in_plane;
      cur_halo.wait_for_dma_finish();
      compute_barrier.sync();
      float r[kCells];
#pragma unroll
      for (int i = 0; i < kCells; ++i) r[i] = stencil_cell(cur_plane, lx, ly + i * kRowsPerPass, q[i], k);
      cur_halo.start_async_dma();
      if (!last) {
#pragma unroll
        for (int i = 0; i < kCells; ++i) other_origin[(ly + i * kRowsPerPass) * kPitch + lx] = q[i][kR + 1];
      }
#pragma unroll
      for (int i = 0; i < kCells; ++i) o[(size_t)(i * kRowsPerPass) * nx] = r[i];
      o += out_plane;
    };
    for (int z = 0; z < w.planes; z += 2) {
      one_plane(plane[0], lds_origin1, halo0, z + 1 >= w.planes);
      if (z + 1 < w.planes) one_plane(plane[1], lds_origin0, halo1, z + 2 >= w.planes);
    }
  }
}
#endif  // HIPDMA_SWEEP_VARIANTS

#ifdef HIPDMA_SWEEP_VARIANTS
__global__ void __launch_bounds__(kComputeThreads)
stencil_not_specialized(const float* __restrict__ in, float* __restrict__ out, const int nx, const int ny,
                        const int nz, const int zchunk, const Coeffs k)
{
  __shared__ __attribute__((aligned(16))) float plane[kPlaneFloats];
  const int px = nx + 2 * kR;
  const size_t in_plane = (size_t)px * (size_t)(ny + 2 * kR);
  const size_t out_plane = (size_t)nx * ny;
  halo_all_t halo(px);
  const TileWork w = tile_work(in, out, nx, ny, nz, zchunk);
  float* lds_origin = &plane[kR * kPitch + kR];
  const int lx = threadIdx.x % kTX;
  const int ly = threadIdx.x / kTX;
  float q[kCells][2 * kR + 1];
  const float* col = w.in_origin + (size_t)ly * px + lx;
#pragma unroll
  for (int i = 0; i < kCells; ++i)
#pragma unroll
    for (int p = 0; p < 2 * kR; ++p) q[i][p + 1] = col[(size_t)p * in_plane + (size_t)(i * kRowsPerPass) * px];
  const float* next = col + (size_t)(2 * kR) * in_plane;
  const float* ring_src = w.in_origin + (size_t)kR * in_plane;
  float* o = w.out_origin + (size_t)ly * nx + lx;
  for (int z = 0; z < w.planes; ++z) {
#pragma unroll
    for (int i = 0; i < kCells; ++i) {
#pragma unroll
      for (int p = 0; p < 2 * kR; ++p) q[i][p] = q[i][p + 1];
      q[i][2 * kR] = next[(size_t)(i * kRowsPerPass) * px];
    }
    next += in_plane;
    halo.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(ring_src, lds_origin);
    ring_src += in_plane;
#pragma unroll
    for (int i = 0; i < kCells; ++i) lds_origin[(ly + i * kRowsPerPass) * kPitch + lx] = q[i][kR];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kCells; ++i)
      o[(size_t)(i * kRowsPerPass) * nx] = stencil_cell(plane, lx, ly + i * kRowsPerPass, q[i], k);
    o += out_plane;
    __syncthreads();
  }
}
#endif  // HIPDMA_SWEEP_VARIANTS

// ---------------------------------------------------------------------------
// dwordx4 version: a compute thread owns four consecutive cells of one tile row
// and moves them as one 16-byte access everywhere (global load of the newest
// plane, LDS write of the centre plane, LDS reads of the x/y neighbours, global
// store of the result).  PREFETCH planes beyond the nine of the stencil are
// kept in flight per thread so that a workgroup has (1 + PREFETCH) x 4 KiB of
// loads outstanding.
// ---------------------------------------------------------------------------
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kXQ = kTX / 4;                          // 8 threads per tile row
constexpr int kPrefetch = 3;
constexpr int kQueue = 2 * kR + 1 + kPrefetch;        // planes held in registers: 12 (the warp-specialised kernels take
                                                      // theirs, QUEUE, from the depth of the DMA wavefront's ring)
// The z column is a ring of registers: plane z + p of the chunk sits in slot
// (z + p) % kQueue, and the z loop is unrolled kQueue times so that every slot
// number is a compile-time constant and no plane is ever moved between registers.
#define HIPDMA_QSLOT(ROT, P) (((ROT) + (P)) % QUEUE)

enum SyncMode {
  kHandshakeAndBarrier = 0,   // empty/full handshake + one s_barrier per plane (DMA wavefront joins it)
  kHandshakeAndGroupBarrier,  // empty/full handshake + LDS-counter barrier of the compute wavefronts
  kBarrierOnly,               // execute_dma_no_sync + one s_barrier per plane
};

// Four cells of row ly starting at column lx; plane p of the z column is q[HIPDMA_QSLOT(ROT, p)].
// Same operations in the same order as the host statement: one multiply, then per
// radius five additions and one fused multiply-add.
// Tile row of a compute thread.  Eight consecutive lanes (an octet) share a row: 128 contiguous bytes.
// ds_read_b128 serves a wavefront in four passes of sixteen lanes, and a pass is not sixteen
// consecutive lanes: within each 32 lanes, pass 0 takes lanes 0-3, 12-15 and 20-27, pass 1 lanes 4-11,
// 16-19 and 28-31 (measured with SQ_LDS_BANK_CONFLICT on single-wavefront probes: 435 access patterns, all
// explained by this rule and 64 banks of 4 bytes).  A pass is free of conflicts when its sixteen lanes
// touch sixteen different 16-byte units modulo 256 bytes.  With octets o0..o3 of 32 lanes on rows whose
// first unit is a, b, c, d (mod 16) the two passes cover {a..a+3, b+4..b+7, c+4..c+7, d..d+3} and
// {a+4..a+7, b..b+3, c..c+3, d+4..d+7}: both tile the sixteen units when b = d = a + 8 and c = a.
// A row of the plane is 40 floats = 10 units, so rows four apart differ by 40 = 8 (mod 16) units and rows
// eight apart by 0: the four octets take rows y, y+4, y+8, y+12.  Every read of the stencil is this
// pattern shifted by a constant, so all of them are conflict-free; the ds_write_b128 of the interior is
// served eight consecutive lanes at a time (32 banks) and a contiguous row is conflict-free as it is.
__device__ __forceinline__ int tile_row_of_thread()
{
  if constexpr (kXQ == 8) {
    const int octet = threadIdx.x / kXQ;                // 0 .. 31
    const int wave = octet / 8, j = octet % 8;
    return 16 * (wave / 2) + 2 * (wave % 2) + (j / 4) + 4 * (j % 4);
  } else {
    // sixteen lanes per row of 72 floats = 18 units: a row covers all sixteen units modulo 16 once, a pass takes
    // lanes 0-3 and 12-15 of one row and lanes 4-11 of the next sixteen lanes' row, so those two rows must start at
    // the same unit modulo 16: eight rows apart (8 x 18 = 144 = 0 mod 16).  Wavefront w: rows 2w, 2w+8, 2w+1, 2w+9.
    const int wave = threadIdx.x / 64, g = (threadIdx.x / kXQ) % 4;
    return 2 * wave + (g / 2) + 8 * (g % 2);
  }
}

// The x and y neighbours of a thread's four cells, as they come out of the LDS plane: ten ds_read_b128.
// Named members, not arrays: the values have to live in registers across the hand-off that sits between
// the reads and the arithmetic, and an array inside a struct ends up in scratch memory here.
struct Neighbours {
  f32x4_t xl, xr, up1, up2, up3, up4, dn1, dn2, dn3, dn4;
  template<int R> __device__ __forceinline__ const f32x4_t& up() const
  { if constexpr (R == 1) return up1; else if constexpr (R == 2) return up2; else if constexpr (R == 3) return up3; else return up4; }
  template<int R> __device__ __forceinline__ const f32x4_t& dn() const
  { if constexpr (R == 1) return dn1; else if constexpr (R == 2) return dn2; else if constexpr (R == 3) return dn3; else return dn4; }
};
static_assert(kR == 4, "Neighbours names four rows above and four below");
__device__ __forceinline__ Neighbours stencil_fetch4(const float* __restrict__ plane, const int lx, const int ly)
{
  const float* c = plane + (ly + kR) * kPitch + (lx + kR);
  Neighbours n;
  n.xl = *(const f32x4_t*)(c - 4);
  n.xr = *(const f32x4_t*)(c + 4);
  n.up1 = *(const f32x4_t*)(c - 1 * kPitch);
  n.dn1 = *(const f32x4_t*)(c + 1 * kPitch);
  n.up2 = *(const f32x4_t*)(c - 2 * kPitch);
  n.dn2 = *(const f32x4_t*)(c + 2 * kPitch);
  n.up3 = *(const f32x4_t*)(c - 3 * kPitch);
  n.dn3 = *(const f32x4_t*)(c + 3 * kPitch);
  n.up4 = *(const f32x4_t*)(c - 4 * kPitch);
  n.dn4 = *(const f32x4_t*)(c + 4 * kPitch);
  return n;
}

// One radius of the sum for cell I: same operations in the same order as the host statement.
template<int ROT, int QUEUE, int I, int R>
__device__ __forceinline__ float stencil_term(const Neighbours& n, const float (&xs)[12], const f32x4_t (&q)[QUEUE],
                                              const float coeff, const float acc)
{
#pragma clang fp contract(off)
  const float sx = xs[4 + I - R] + xs[4 + I + R];
  const float sy = n.template up<R>()[I] + n.template dn<R>()[I];
  const float sz = q[HIPDMA_QSLOT(ROT, kR - R)][I] + q[HIPDMA_QSLOT(ROT, kR + R)][I];
  return __builtin_fmaf(coeff, (sx + sy) + sz, acc);
}
template<int ROT, int QUEUE, int I>
__device__ __forceinline__ float stencil_cell_i(const Neighbours& n, const float (&xs)[12], const f32x4_t (&q)[QUEUE],
                                                const Coeffs& k)
{
#pragma clang fp contract(off)
  float acc = k.c0 * xs[4 + I];
  acc = stencil_term<ROT, QUEUE, I, 1>(n, xs, q, k.c1, acc);
  acc = stencil_term<ROT, QUEUE, I, 2>(n, xs, q, k.c2, acc);
  acc = stencil_term<ROT, QUEUE, I, 3>(n, xs, q, k.c3, acc);
  acc = stencil_term<ROT, QUEUE, I, 4>(n, xs, q, k.c4, acc);
  return acc;
}

template<int ROT, int QUEUE>
__device__ __forceinline__ f32x4_t stencil_eval4(const Neighbours& n, const f32x4_t (&q)[QUEUE], const Coeffs& k)
{
  // x neighbourhood: 4 cells left, the centre cells, 4 cells right
  const f32x4_t xc = q[HIPDMA_QSLOT(ROT, kR)];
  const float xs[12] = {n.xl[0], n.xl[1], n.xl[2], n.xl[3], xc[0], xc[1], xc[2], xc[3], n.xr[0], n.xr[1], n.xr[2], n.xr[3]};
  f32x4_t out;
  out[0] = stencil_cell_i<ROT, QUEUE, 0>(n, xs, q, k);
  out[1] = stencil_cell_i<ROT, QUEUE, 1>(n, xs, q, k);
  out[2] = stencil_cell_i<ROT, QUEUE, 2>(n, xs, q, k);
  out[3] = stencil_cell_i<ROT, QUEUE, 3>(n, xs, q, k);
  return out;
}

template<int ROT, int QUEUE>
__device__ __forceinline__ f32x4_t stencil_cells4(const float* __restrict__ plane, const int lx, const int ly,
                                                  const f32x4_t (&q)[QUEUE], const Coeffs& k)
{
  return stencil_eval4<ROT, QUEUE>(stencil_fetch4(plane, lx, ly), q, k);
}

// Runs the body for z = 0 .. planes-1 with ROT = z % kQueue as a constant.  Whole
// groups of kQueue planes run without a single branch, so the compiler's
// s_waitcnt placement can count exactly how many younger loads and stores may
// stay in flight; only the last, partial group checks the plane count.
#define HIPDMA_Z_STEP(J, CHECK, ...) if constexpr ((J) < QUEUE) { if (!(CHECK) || z0 + (J) < planes) { constexpr int ROT = (J); const int z = z0 + (J); __VA_ARGS__ } }
#define HIPDMA_Z_GROUP(CHECK, ...)                                                                       \
  HIPDMA_Z_STEP(0, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(1, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(2, CHECK, __VA_ARGS__)   \
  HIPDMA_Z_STEP(3, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(4, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(5, CHECK, __VA_ARGS__)   \
  HIPDMA_Z_STEP(6, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(7, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(8, CHECK, __VA_ARGS__)   \
  HIPDMA_Z_STEP(9, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(10, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(11, CHECK, __VA_ARGS__) \
  HIPDMA_Z_STEP(12, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(13, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(14, CHECK, __VA_ARGS__) \
  HIPDMA_Z_STEP(15, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(16, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(17, CHECK, __VA_ARGS__) \
  HIPDMA_Z_STEP(18, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(19, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(20, CHECK, __VA_ARGS__) \
  HIPDMA_Z_STEP(21, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(22, CHECK, __VA_ARGS__) HIPDMA_Z_STEP(23, CHECK, __VA_ARGS__)
#define HIPDMA_FOR_Z(planes_expr, ...)                                       \
  {                                                                          \
    const int planes = (planes_expr);                                        \
    int z0 = 0;                                                              \
    for (; z0 + QUEUE <= planes; z0 += QUEUE) { HIPDMA_Z_GROUP(false, __VA_ARGS__) } \
    if (z0 < planes) { HIPDMA_Z_GROUP(true, __VA_ARGS__) }                   \
  }
// HIPDMA_FOR_Z unrolls QUEUE (at most 24) steps; the LDS planes rotate with period 4, so QUEUE is a multiple of 4
template<int QUEUE> struct queue_ok { static_assert(QUEUE >= 2 * kR + 2 && QUEUE <= 24 && QUEUE % 4 == 0, "QUEUE: 12, 16, 20 or 24"); };

// The DMA wavefront keeps the rings of the next RING - 1 planes in flight,
// each in the registers of its own CudaDMAHalo object (manual buffering with
// two-phase calls, as src/examples/stencil/warp_specialized_manual_buffer.h:54-71,
// eight or twelve objects deep), and lands them one per plane in one of four LDS planes.
// That distance matches the one at which the compute threads fetch the
// interior, so a ring is requested while the neighbouring tiles are pulling the
// same cache lines as their interior.  The objects that hold the registers
// carry no handshake; the four LDS planes are guarded by cudaDMACustom objects,
// the sync-only class of include/cudaDMA.h:4184-4208.
constexpr int kBufs = 4;
#ifndef STENCIL_RING_LOAD
#define STENCIL_RING_LOAD LOAD_CACHE_ALL
#endif
#ifndef STENCIL_INTERIOR_NT
#define STENCIL_INTERIOR_NT 0
#endif
constexpr int kRingLoad = STENCIL_RING_LOAD;
#ifndef STENCIL_RING_AHEAD
#define STENCIL_RING_AHEAD (RING - 1)
#endif
typedef CudaDMAHalo<false, 16, kRingBpt, 4, kDmaThreads, kR, false, kTX, kTY> halo_reg_t;

template<typename T>
struct Sixteen {
  T a0, a1, a2, a3, a4, a5, a6, a7, a8, a9, a10, a11, a12, a13, a14, a15;
  template<int I> __device__ __forceinline__ T& get()
  {
    if constexpr (I == 0) return a0; else if constexpr (I == 1) return a1; else if constexpr (I == 2) return a2;
    else if constexpr (I == 3) return a3; else if constexpr (I == 4) return a4; else if constexpr (I == 5) return a5;
    else if constexpr (I == 6) return a6; else if constexpr (I == 7) return a7; else if constexpr (I == 8) return a8;
    else if constexpr (I == 9) return a9; else if constexpr (I == 10) return a10; else if constexpr (I == 11) return a11;
    else if constexpr (I == 12) return a12; else if constexpr (I == 13) return a13; else if constexpr (I == 14) return a14;
    else return a15;
  }
};
template<typename T>
struct Four {
  T a0, a1, a2, a3;
  template<int I> __device__ __forceinline__ T& get()
  {
    if constexpr (I == 0) return a0; else if constexpr (I == 1) return a1; else if constexpr (I == 2) return a2;
    else return a3;
  }
};

#define HIPDMA_RING_STEP(J, CHECK, ...) \
  if constexpr ((J) < RING) { if (!(CHECK) || z0 + (J) < planes) { constexpr int S = (J); const int z = z0 + (J); __VA_ARGS__ } }
#define HIPDMA_RING_GROUP(CHECK, ...)                                                                            \
  HIPDMA_RING_STEP(0, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(1, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(2, CHECK, __VA_ARGS__) \
  HIPDMA_RING_STEP(3, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(4, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(5, CHECK, __VA_ARGS__) \
  HIPDMA_RING_STEP(6, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(7, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(8, CHECK, __VA_ARGS__) \
  HIPDMA_RING_STEP(9, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(10, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(11, CHECK, __VA_ARGS__) \
  HIPDMA_RING_STEP(12, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(13, CHECK, __VA_ARGS__) HIPDMA_RING_STEP(14, CHECK, __VA_ARGS__) \
  HIPDMA_RING_STEP(15, CHECK, __VA_ARGS__)
#define HIPDMA_FOR_RING(planes_expr, ...)                                        \
  {                                                                              \
    const int planes = (planes_expr);                                            \
    int z0 = 0;                                                                  \
    for (; z0 + RING <= planes; z0 += RING) { HIPDMA_RING_GROUP(false, __VA_ARGS__) } \
    if (z0 < planes) { HIPDMA_RING_GROUP(true, __VA_ARGS__) }                    \
  }

// One workgroup of five wavefronts per compute unit is the operating point: at most two wavefronts share a
// SIMD, so the register allocator may use 256 registers per lane instead of spilling to stay under 128.
// RING: halo objects of the DMA wavefront; the rings of RING - 1 planes are in flight, and the compute threads
// fetch the interior at the same distance (QUEUE = RING + 4 planes in registers).  Eight objects (seven planes,
// 2.8 us of look-ahead at 512^3) are the default; twelve (knob "stencil_ring") measured within +-2.5 % of eight
// from run to run, in both directions.
template<int SYNC, int RING = 8>
__global__ void __launch_bounds__(kComputeThreads + kDmaThreads) __attribute__((amdgpu_waves_per_eu(1, 2)))
stencil_ws_vec4(const float* __restrict__ in, float* __restrict__ out, const int nx, const int ny, const int nz,
                const int zchunk, const Coeffs k)
{
  __shared__ __attribute__((aligned(16))) float plane[kBufs][kPlaneFloats];
  const int px = nx + 2 * kR;
  const size_t in_plane = (size_t)px * (size_t)(ny + 2 * kR);
  const size_t out_plane = (size_t)nx * ny;
  // guards of the four LDS planes: empty/full handshake between the compute and the DMA wavefronts
  Four<cudaDMACustom> guard{cudaDMACustom(0, kDmaThreads, kComputeThreads, kComputeThreads),
                            cudaDMACustom(1, kDmaThreads, kComputeThreads, kComputeThreads),
                            cudaDMACustom(2, kDmaThreads, kComputeThreads, kComputeThreads),
                            cudaDMACustom(3, kDmaThreads, kComputeThreads, kComputeThreads)};
  hipdma::GroupBarrier compute_barrier(4, kComputeThreads);
  const TileWork w = tile_work(in, out, nx, ny, nz, zchunk);
  constexpr int kOrigin = kR * kPitch + kR;
  constexpr int QUEUE = RING + kR;
  constexpr int kRingAhead = STENCIL_RING_AHEAD;
  static_assert(RING >= 8 && RING <= 16 && RING % kBufs == 0, "HIPDMA_FOR_RING unrolls 8, 12 or 16 steps");
  static_assert(kRingAhead >= 2 && kRingAhead < RING, "a ring has to be requested before it lands and needs an object of its own");

  if (guard.a0.owns_this_thread()) {
    const halo_reg_t one(px, kComputeThreads);          // objects beyond RING are never used and cost nothing
    Sixteen<halo_reg_t> ring{one, one, one, one, one, one, one, one, one, one, one, one, one, one, one, one};
    // ring of the centre plane of output plane z: padded plane z + kR
    const float* ring0 = w.in_origin + (size_t)kR * in_plane;
    // a request past the last plane re-reads the last one: the loads stay unconditional, nothing lands from them
    const int last = w.planes - 1;
#define HIPDMA_ISSUE(I, ZP) \
    ring.get<(I)>().template start_xfer_async<true, kRingLoad, STORE_LDS>(ring0 + (size_t)((ZP) < last ? (ZP) : last) * in_plane);
#define HIPDMA_LAND(I, ZP)                                                                                   \
    if ((ZP) < w.planes) {                                                                                   \
      if constexpr (SYNC != kBarrierOnly) guard.get<(I) % kBufs>().wait_for_dma_start();                     \
      ring.get<(I)>().template wait_xfer_finish<true, kRingLoad, STORE_LDS>(&plane[(I) % kBufs][kOrigin]); \
      if constexpr (SYNC != kBarrierOnly) guard.get<(I) % kBufs>().finish_async_dma();                       \
    }
    // With the handshake the ring lands two planes ahead of its use instead of one: the compute
    // wavefronts then find the `full` word of a plane set when they first look, and never poll.
    constexpr int kLand = (SYNC == kBarrierOnly) ? 1 : 2;
    // planes 0 .. kRingAhead-1 are requested up front; planes 0 .. kLand-1 land before the first barrier
    if constexpr (kRingAhead > 0) { HIPDMA_ISSUE(0, 0) }
    if constexpr (kRingAhead > 1) { HIPDMA_ISSUE(1, 1) }
    if constexpr (kRingAhead > 2) { HIPDMA_ISSUE(2, 2) }
    if constexpr (kRingAhead > 3) { HIPDMA_ISSUE(3, 3) }
    if constexpr (kRingAhead > 4) { HIPDMA_ISSUE(4, 4) }
    if constexpr (kRingAhead > 5) { HIPDMA_ISSUE(5, 5) }
    if constexpr (kRingAhead > 6) { HIPDMA_ISSUE(6, 6) }
    if constexpr (kRingAhead > 7) { HIPDMA_ISSUE(7, 7) }
    if constexpr (kRingAhead > 8) { HIPDMA_ISSUE(8, 8) }
    if constexpr (kRingAhead > 9) { HIPDMA_ISSUE(9, 9) }
    if constexpr (kRingAhead > 10) { HIPDMA_ISSUE(10, 10) }
    if constexpr (kRingAhead > 11) { HIPDMA_ISSUE(11, 11) }
    if constexpr (kRingAhead > 12) { HIPDMA_ISSUE(12, 12) }
    if constexpr (kRingAhead > 13) { HIPDMA_ISSUE(13, 13) }
    if constexpr (kRingAhead > 14) { HIPDMA_ISSUE(14, 14) }
    HIPDMA_LAND(0, 0)
    if constexpr (kLand == 2) { HIPDMA_LAND(1, 1) }
    // iteration z: request plane z + kRingAhead, meet the compute wavefronts, land plane z + kLand
    HIPDMA_FOR_RING(w.planes, {
      HIPDMA_ISSUE((S + kRingAhead) % RING, z + kRingAhead)
      if constexpr (SYNC != kHandshakeAndGroupBarrier) __syncthreads();
      HIPDMA_LAND((S + kLand) % RING, z + kLand)
    })
#undef HIPDMA_ISSUE
#undef HIPDMA_LAND
  } else {
    const int lx = 4 * (threadIdx.x % kXQ);
    const int ly = tile_row_of_thread();
    (void)sizeof(queue_ok<QUEUE>);
    f32x4_t q[QUEUE];
    const float* col = w.in_origin + (size_t)ly * px + lx;
    // planes 0 .. QUEUE-2 of the chunk; every iteration fetches one more
    const int avail = w.planes + 2 * kR;                  // padded planes this chunk may touch
#pragma unroll
    for (int p = 0; p < QUEUE - 1; ++p)
      q[p] = (p < avail) ? *(const f32x4_t*)(col + (size_t)p * in_plane) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    if constexpr (SYNC != kBarrierOnly) {
      guard.a0.start_async_dma();
      guard.a1.start_async_dma();
      guard.a2.start_async_dma();
      guard.a3.start_async_dma();
    }
    *(f32x4_t*)(&plane[0][kOrigin] + ly * kPitch + lx) = q[kR];
    float* o = w.out_origin + (size_t)ly * nx + lx;
    // The wait for a plane's ring is split: its `full` word is read at the end of the plane before,
    // after that plane's arithmetic (by then the ring has landed), and looked at here.
    unsigned seen = 0;
    if constexpr (SYNC != kBarrierOnly) seen = guard.a0.peek_dma_finish();
    HIPDMA_FOR_Z(w.planes, {
      constexpr int B = ROT % kBufs;
      const cudaDMACustom& cur_halo = guard.get<B>();
      // past the end of the chunk the last plane is fetched again: unconditional loads keep the wait counts exact
      const int zf = (z + QUEUE - 1 < avail) ? (z + QUEUE - 1) : (avail - 1);
      if constexpr (STENCIL_INTERIOR_NT) q[HIPDMA_QSLOT(ROT, QUEUE - 1)] = __builtin_nontemporal_load((const f32x4_t*)(col + (size_t)zf * in_plane));
      else q[HIPDMA_QSLOT(ROT, QUEUE - 1)] = *(const f32x4_t*)(col + (size_t)zf * in_plane);
      if constexpr (SYNC != kBarrierOnly) cur_halo.wait_for_dma_finish(seen);
      if constexpr (SYNC == kHandshakeAndGroupBarrier) compute_barrier.sync();
      else __syncthreads();
      // With the handshake the plane is released as soon as its ten reads have returned (the release fence waits
      // for exactly those) and the `full` word of the next plane is requested right behind the signal: both LDS
      // round trips then run under the arithmetic of this plane instead of after it.
      const Neighbours nb = stencil_fetch4(plane[B], lx, ly);
      if constexpr (SYNC != kBarrierOnly) {
        cur_halo.start_async_dma();
        seen = guard.get<(B + 1) % kBufs>().peek_dma_finish();
      }
      *(f32x4_t*)(&plane[(B + 1) % kBufs][kOrigin] + ly * kPitch + lx) = q[HIPDMA_QSLOT(ROT, kR + 1)];
      const f32x4_t r = stencil_eval4<ROT, QUEUE>(nb, q, k);
      __builtin_nontemporal_store(r, (f32x4_t*)o);     // the output is not read again: 3 % faster than a plain store
      o += out_plane;
    })
  }
}

// The form that is not warp-specialised (src/examples/stencil/non_warp_specialized_single_buffer.h:34-58):
// every thread computes and every other thread also carries one chunk of the
// ring, requested one plane ahead; one LDS plane, two s_barriers per plane.
__global__ void __launch_bounds__(kComputeThreads)
stencil_all_vec4(const float* __restrict__ in, float* __restrict__ out, const int nx, const int ny, const int nz,
                 const int zchunk, const Coeffs k)
{
  __shared__ __attribute__((aligned(16))) float plane[kPlaneFloats];
  const int px = nx + 2 * kR;
  const size_t in_plane = (size_t)px * (size_t)(ny + 2 * kR);
  const size_t out_plane = (size_t)nx * ny;
  halo_all_t halo(px);
  const TileWork w = tile_work(in, out, nx, ny, nz, zchunk);
  float* lds_origin = &plane[kR * kPitch + kR];
  const int lx = 4 * (threadIdx.x % kXQ);
  const int ly = tile_row_of_thread();
  constexpr int QUEUE = kQueue;
  f32x4_t q[QUEUE];
  const float* col = w.in_origin + (size_t)ly * px + lx;
  const int avail = w.planes + 2 * kR;
#pragma unroll
  for (int p = 0; p < QUEUE - 1; ++p)
    q[p] = (p < avail) ? *(const f32x4_t*)(col + (size_t)p * in_plane) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  const float* ring0 = w.in_origin + (size_t)kR * in_plane;
  const int last = w.planes - 1;
  float* o = w.out_origin + (size_t)ly * nx + lx;
  halo.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(ring0);
  HIPDMA_FOR_Z(w.planes, {
    const int zf = (z + QUEUE - 1 < avail) ? (z + QUEUE - 1) : (avail - 1);
    q[HIPDMA_QSLOT(ROT, QUEUE - 1)] = *(const f32x4_t*)(col + (size_t)zf * in_plane);
    halo.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(lds_origin);
    *(f32x4_t*)(lds_origin + ly * kPitch + lx) = q[HIPDMA_QSLOT(ROT, kR)];
    __syncthreads();
    halo.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(ring0 + (size_t)(z < last ? z + 1 : last) * in_plane);
    *(f32x4_t*)o = stencil_cells4<ROT, QUEUE>(plane, lx, ly, q, k);
    o += out_plane;
    __syncthreads();
  })
}

}  // namespace

// The same kernels with tiles of 64 x 16 cells (rows of 256 B) are compiled from this file a second time
// (workloads_stencil_wide.hip) and reached through the variants from kWideTileVariants on: 2 to 8 % faster than the
// 32 x 32 tiles at 512^3 depending on the box (tiles of 128 x 8 cells were level with 32 x 32: their rings are twice
// as large).
constexpr int kWideTileVariants = 6;

// How many planes a workgroup takes.  Every workgroup pays for about twelve planes before its first output (2 * radius planes of
// the column plus the wait for them), whatever it then marches through.  A second workgroup on a compute unit slows both by 1.4
// where the caches hold the grids from one sweep to the next and up to twice where they come from DRAM; a third waits for its turn.
// Of the numbers of chunks that just fill the compute units once, twice or three times, the one with the least sum of these is taken
// (four were never the best).  Measured (us, resident / from DRAM, by workgroups; the first is one chunk per ceil(compute units / tiles)):
//   192 x 256 x 130  288: 16.4 / 23.5  480: 13.4 / 19.8  240: 14.6 / 16.4      480 x 384 x 142  360: 41 / 65  720: 41 / 56  180: 54 / 56
//   128^3            128:  9.9 / 10.8  256:  7.0 /  8.8                        384 x 320 x 200  360: 40 / 63  480: 36 / 53  240: 42 / 44
//   256^3            256: 30.3 / 33.8  512: 25.2 / 37.8                        512 x 512 x 64   256: 29 / 31  512: 26 / 38
// A shape is taken where it is faster both ways.  Where the chunks that it takes to occupy every compute unit, of 16 planes or more,
// still make one workgroup each (the last pair), a second one gains 10 to 17 % from the caches and loses 12 to 24 from DRAM: it is
// charged at the DRAM price there, as it is beyond what stays resident (448 x 512, 224 / 448 workgroups: 460 MiB 97 / 80 us, 500 MiB 112 / 125).
constexpr int kLeastZchunk = 4;
static int best_zchunk(const long long tiles_xy, const long long bytes, const int nz, const bool dwordx4)
{
  const long long cus = workloads::device_cus();
  const long long most = nz / kLeastZchunk > 1 ? nz / kLeastZchunk : 1;
  const long long cut = (cus + tiles_xy - 1) / tiles_xy, planes = (nz + cut - 1) / cut < 16 ? 16 : (nz + cut - 1) / cut;
  const bool one_fills = tiles_xy * ((nz + planes - 1) / planes) <= cus;
  // tenths of the time with one; the sweep kernels always want two
  const long long two = dwordx4 && (one_fills || bytes > (480LL << 20)) ? 20 : 14;
  int best = nz;
  long long least = -1;
  for (int k = 0; k <= 3; ++k) {
    long long chunks = k == 0 ? 1 : k * cus / tiles_xy;
    if (chunks < 1) continue;
    if (chunks > most) chunks = most;
    const int zchunk = (int)((nz + chunks - 1) / chunks);
    const long long grid = tiles_xy * ((nz + zchunk - 1) / zchunk);
    const long long rest = grid % (2 * cus);
    const long long last = rest == 0 ? 0 : rest > cus ? two : grid <= cus ? 10 : 12;     // a third shares the caches with what is left of the two
    const long long cost = (12 + zchunk) * (grid / (2 * cus) * two + last);
    if (least < 0 || cost < least) { least = cost; best = zchunk; }
  }
  return best;
}

#ifdef STENCIL_WIDE_TILES
extern "C" int cudadma_halo_stencil_wide_tiles(const float* d_in, float* d_out, int nx, int ny, int nz, int variant, void* stream)
{
  CUDADMA_REQUIRE(nx > 0 && ny > 0 && nz > 0, "grid dimensions must be positive");
  CUDADMA_REQUIRE((nx % kTX) == 0 && (ny % kTY) == 0, "the variants with wide tiles need nx a multiple of 64 and ny a multiple of 16");
  CUDADMA_REQUIRE(variant >= 0 && variant < 2, "the wide tiles are compiled for the two fastest kernel shapes");
#else
extern "C" int cudadma_halo_stencil_wide_tiles(const float* d_in, float* d_out, int nx, int ny, int nz, int variant, void* stream);

extern "C" int cudadma_halo_stencil(const float* d_in, float* d_out, int nx, int ny, int nz, int variant, void* stream)
{
  CUDADMA_REQUIRE(nx > 0 && ny > 0 && nz > 0, "grid dimensions must be positive");
  if (variant < 0 || variant >= cudadma_num_variants(CUDADMA_WORKLOAD_HALO)) {
    cudadma_host::set_error("halo stencil has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  if (variant >= kWideTileVariants) return cudadma_halo_stencil_wide_tiles(d_in, d_out, nx, ny, nz, variant - kWideTileVariants, stream);
  CUDADMA_REQUIRE((nx % kTX) == 0 && (ny % kTY) == 0, "nx and ny must be multiples of 32");
#endif
  CUDADMA_REQUIRE(d_in != nullptr && d_out != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_in, 16) && cudadma_host::aligned_to(d_out, 16), "pointers must be 16-byte aligned");
  const Coeffs k = {(float)(3.0 * (-205.0 / 72.0)), (float)(8.0 / 5.0), (float)(-1.0 / 5.0), (float)(8.0 / 315.0),
                    (float)(-1.0 / 560.0)};
  const long long tiles_xy = (long long)(nx / kTX) * (ny / kTY);
  int zchunk = workloads::tuning("stencil_zchunk", best_zchunk(tiles_xy, 4LL * (2LL * nx * ny) * nz, nz, variant <= 3));
  if (zchunk < kLeastZchunk) zchunk = kLeastZchunk;
  if (zchunk > nz) zchunk = nz;
  const int chunks = (nz + zchunk - 1) / zchunk;
  // knob "stencil_xcd_remap": 2 turns the XCD-aware numbering off, 4 asks for compact blocks instead of slabs
  const int remap = workloads::tuning("stencil_xcd_remap", 1);
  const long long grid = (long long)(nx / kTX) * (ny / kTY) * chunks;
  if (remap != 2) zchunk |= kXcdFlag;
  if (remap == 4 && chunks == 1 && ((nx / kTX) % 2) == 0 && ((ny / kTY) % 4) == 0) zchunk |= kXcdBlockFlag;
  CUDADMA_REQUIRE(grid <= 0x7fffffffLL, "grid too large");
  hipStream_t s = (hipStream_t)stream;
  const dim3 g((unsigned)grid), ws(kComputeThreads + kDmaThreads), all(kComputeThreads);
  switch (variant) {
    // knob "stencil_ring": 8 (default) or 12 halo objects on the DMA wavefront
    case 0:
      if (workloads::tuning("stencil_ring", 8) == 12) hipLaunchKernelGGL((stencil_ws_vec4<kBarrierOnly, 12>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      else hipLaunchKernelGGL((stencil_ws_vec4<kBarrierOnly, 8>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      break;
    case 1:
      if (workloads::tuning("stencil_ring", 8) == 12) hipLaunchKernelGGL((stencil_ws_vec4<kHandshakeAndBarrier, 12>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      else hipLaunchKernelGGL((stencil_ws_vec4<kHandshakeAndBarrier, 8>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      break;
    case 2:
      if (workloads::tuning("stencil_ring", 8) == 12) hipLaunchKernelGGL((stencil_ws_vec4<kHandshakeAndGroupBarrier, 12>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      else hipLaunchKernelGGL((stencil_ws_vec4<kHandshakeAndGroupBarrier, 8>), g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k);
      break;
    case 3: hipLaunchKernelGGL(stencil_all_vec4, g, all, 0, s, d_in, d_out, nx, ny, nz, zchunk, k); break;
#ifdef HIPDMA_SWEEP_VARIANTS
    case 4: hipLaunchKernelGGL(stencil_warp_specialized, g, ws, 0, s, d_in, d_out, nx, ny, nz, zchunk, k); break;
    default: hipLaunchKernelGGL(stencil_not_specialized, g, all, 0, s, d_in, d_out, nx, ny, nz, zchunk, k); break;
#else
    default: CUDADMA_REQUIRE(false, "halo stencil variant %d is a sweep kernel: build the library with make EXTRA=-DHIPDMA_SWEEP_VARIANTS", variant);
#endif
  }
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}
