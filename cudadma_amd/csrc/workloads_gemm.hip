// Config 5: C = A * B, bf16 inputs, fp32 accumulate, warp-specialised and
// double-buffered.  The reference has no GEMM; the nearest code is the SGEMV of
// src/examples/sgemv/sgemv_dma.cu:329-388 (Strided matrix tiles staged by DMA
// warps, FMA loop in the compute warps).  Here, for a workgroup tile BM x BN and K step 64:
//   * the first WM x WN wavefronts compute, each on WI x WJ blocks of
//     v_mfma_f32_32x32x16_bf16 (BM = 32*WI*WM, BN = 32*WJ*WN).  A fragments are
//     ds_read_b128 from rows padded to 144 B; B stays row-major [k][n] in LDS (rows
//     padded by 64 B) and is turned into k-major fragments on the way to the
//     registers by ds_read_b64_tr_b16;
//   * the next two wavefronts stage the A tiles (BM rows x 128 B, source stride K*2
//     bytes), the last two the B tiles (64 rows x 2*BN B, source stride N*2 bytes).
//     Each pair owns two CudaDMAStrided objects, one per LDS stage, and uses the
//     two-phase calls so that the tile two K steps ahead is already in flight (in the
//     object's registers) while the current one is consumed: a K step is shorter
//     than a trip to memory, one tile of look-ahead is not enough.
// Four compute wavefronts (2 x 2) share the SIMDs with the four DMA wavefronts one to
// one and get 256 registers each; eight (2 x 4, the 256 x 256 tile) make it three
// wavefronts per SIMD and 168 registers each, but two of them compute.
#include "dispatch.hpp"
#include "workloads.hpp"

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kBK = 64;
constexpr int kComputeThreads = 256;
constexpr int kDmaWave = 128;              // DMA threads per operand: two wavefronts

// Tile geometry for compute wavefronts that each own WI x WJ blocks of 32 x 32: the WM x WN
// wavefronts sit in a grid, so the workgroup tile is 32*WI*WM x 32*WJ*WN.
template<int WI, int WJ, int WM = 2, int WN = 2>
struct GemmShape {
  static constexpr int kCompute = 64 * WM * WN;     // compute threads; the DMA threads follow them
  static constexpr int kBM = 32 * WI * WM, kBN = 32 * WJ * WN;
  static constexpr int kAPitch = kBK * 2 + 16;      // 144 B per A row in LDS
  static constexpr int kBPitch = kBN * 2 + 64;      // B row in LDS: the four rows a transposing read touches land 64 B apart modulo 256
  static constexpr int kAStage = kBM * kAPitch;
  static constexpr int kBStage = kBK * kBPitch;
  static constexpr int kPerCu = 2 * (kAStage + kBStage) <= (80 << 10) ? 2 : 1;      // workgroups that share a compute unit's LDS
  typedef CudaDMAStrided<false, 16, kBM * kBK * 2 / kDmaWave, kBK * 2, kDmaWave, kBM> dma_a_t;   // kBM rows x 128 B
  typedef CudaDMAStrided<false, 16, kBK * kBN * 2 / kDmaWave, kBN * 2, kDmaWave, kBK> dma_b_t;   // 64 rows x 2*kBN B
};

using dispatch::tile_of_workgroup;
int tile_walk(const int m, const int n, const int k, const int tile_rows, const int tile_cols, const int per_cu)
{
  return dispatch::tile_walk(m, n, k, tile_rows, tile_cols, per_cu, workloads::device_cus());
}

// Order of one slice for the instruction scheduler: MFMAs matrix instructions with the READS
// LDS requests of the next slice issued two at a time behind the first of them; the last
// matrix instructions run with nothing behind them, so the data has landed when the next
// slice starts.
template<int G, int MFMAS, int READS>
__device__ __forceinline__ void pin_slice()
{
  if constexpr (G < MFMAS) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                    // one MFMA
    if constexpr (2 * G + 2 <= READS) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);   // two LDS reads
    else if constexpr (2 * G < READS) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    pin_slice<G + 1, MFMAS, READS>();
  }
}

template<int WI, int WJ, int WM = 2, int WN = 2>
__global__ void __launch_bounds__(64 * WM * WN + 2 * kDmaWave)
gemm_bf16_ws(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
             const int m, const int n, const int k, const int walk)
{
  typedef GemmShape<WI, WJ, WM, WN> shape;
  constexpr int kComputeThreads = shape::kCompute;
  typedef typename shape::dma_a_t dma_a_t;
  typedef typename shape::dma_b_t dma_b_t;
  constexpr int kAPitch = shape::kAPitch, kBPitch = shape::kBPitch;
  __shared__ __attribute__((aligned(16))) char lds_a[2][shape::kAStage];
  __shared__ __attribute__((aligned(16))) char lds_b[2][shape::kBStage];
  // The transfer objects carry no handshake of their own: a stage holds an A tile and a B tile,
  // and one sync object per stage covers the four DMA wavefronts of both operands, so the
  // compute wavefronts wait and signal once per stage instead of once per operand.
  dma_a_t dma_a0(k * 2, kAPitch, kComputeThreads);
  dma_a_t dma_a1(k * 2, kAPitch, kComputeThreads);
  dma_b_t dma_b0(n * 2, kBPitch, kComputeThreads + kDmaWave);
  dma_b_t dma_b1(n * 2, kBPitch, kComputeThreads + kDmaWave);
  cudaDMACustom stage0(0, 2 * kDmaWave, kComputeThreads, kComputeThreads);
  cudaDMACustom stage1(1, 2 * kDmaWave, kComputeThreads, kComputeThreads);
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / shape::kBM, n / shape::kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK;            // even: k is a multiple of 2 * kBK
  const int klast = ksteps - 1;

  // One DMA wavefront: tiles kt and kt+1 are requested up front, then every landed tile is
  // followed by the request for the tile two steps on (clamped past the end so that no load
  // sits behind a branch and s_waitcnt can leave the younger tile in flight).
  auto stage_tiles = [&](auto& d0, auto& d1, char* s0, char* s1, const unsigned short* src, const size_t step)
      __attribute__((always_inline)) {
    d0.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(src);
    d1.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(src + step);
    for (int kt = 0; kt < ksteps; kt += 2) {
      stage0.wait_for_dma_start();
      d0.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(s0);
      stage0.finish_async_dma();
      d0.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(src + (size_t)(kt + 2 < klast ? kt + 2 : klast) * step);
      stage1.wait_for_dma_start();
      d1.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(s1);
      stage1.finish_async_dma();
      d1.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(src + (size_t)(kt + 3 < klast ? kt + 3 : klast) * step);
    }
  };
  if (dma_a0.owns_this_thread()) {
    stage_tiles(dma_a0, dma_a1, lds_a[0], lds_a[1], a + (size_t)tile_m * shape::kBM * k, (size_t)kBK);
  } else if (dma_b0.owns_this_thread()) {
    stage_tiles(dma_b0, dma_b1, lds_b[0], lds_b[1], b + (size_t)tile_n * shape::kBN, (size_t)kBK * n);
  } else {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = (wave / WN) * 32 * WI, wn = (wave % WN) * 32 * WJ;     // this wavefront's corner in the workgroup tile
    f32x16_t acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    // both stages are free to begin with
    stage0.start_async_dma();
    stage1.start_async_dma();
    // A fragment: row wm + 32*i + lane%32, eight k starting at 16*ks + 8*(lane/32)
    const int a_off = (wm + (lane & 31)) * kAPitch + (lane >> 5) * 16;
    // B fragment through the transposing read: inside a group of 16 lanes, lane j points at
    // row (j/4) of a 4-row block and at column 4*(j%4); lane i then receives rows 0..3 of column i.
    const int j16 = lane & 15;
    const int b_off = ((lane >> 5) * 8 + (j16 >> 2)) * kBPitch + (wn + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
    // With 128 accumulator registers a SIMD holds one compute wavefront, which has to hide its
    // own LDS latency: the order "request the next slice, then multiply the current one" is
    // pinned against the instruction scheduler.  With the small tile two workgroups share a
    // compute unit and the scheduler's own order does better, and so it does with one (1408 x 2176 x 1920: 22 us against 24).
    constexpr bool kPinned = (WI * WJ >= 8) && (WM * WN == 4);
    // Fragments of one 16-deep slice of the K step: WI row blocks of A, WJ column blocks of B.
    auto load_frags = [&](bf16x8_t (&fa)[WI], bf16x8_t (&fb)[WJ], const char* sa, const char* sb, const int ks)
        __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
        fa[i] = *(const bf16x8_t*)(sa + i * 32 * kAPitch + ks * 32);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const char* p = sb + ks * 16 * kBPitch + j * 32 * 2;
        const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)p);
        const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) bf16x4_t*)(p + 4 * kBPitch));
        fb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    };
    auto multiply = [&](const bf16x8_t (&fa)[WI], const bf16x8_t (&fb)[WJ]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    };
    // One slice of the pinned schedule: the WI + 2*WJ LDS requests of the next slice are
    // issued one by one in the shadow of the WI*WJ matrix instructions of the current slice
    // (a matrix instruction holds its pipe for 32 cycles, the wavefront is free to issue an
    // LDS request meanwhile), and nothing moves across the ends of the slice.
    auto interleave = [&]() __attribute__((always_inline)) {
      if constexpr (kPinned) {
        pin_slice<0, WI * WJ, WI + 2 * WJ>();
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    // The one compute wavefront of a SIMD has to keep the matrix core fed by itself: the
    // fragments of the next slice are requested before the products of the current one are
    // issued, across the stage boundary too (the next stage is waited for, and its first slice
    // requested, ahead of the last products of the current stage).
    const char* sa0 = lds_a[0] + a_off; const char* sb0 = lds_b[0] + b_off;
    const char* sa1 = lds_a[1] + a_off; const char* sb1 = lds_b[1] + b_off;
    bf16x8_t fa0[WI], fb0[WJ], fa1[WI], fb1[WJ];
    static_assert(kBK / 16 == 4, "the slice schedule below is written for four slices per stage");
    if constexpr (!kPinned) {
      for (int kt = 0; kt < ksteps; kt += 2) {
        stage0.wait_for_dma_finish();
#pragma unroll
        for (int ks = 0; ks < kBK / 16; ++ks) { load_frags(fa0, fb0, sa0, sb0, ks); multiply(fa0, fb0); }
        stage0.start_async_dma();
        stage1.wait_for_dma_finish();
#pragma unroll
        for (int ks = 0; ks < kBK / 16; ++ks) { load_frags(fa0, fb0, sa1, sb1, ks); multiply(fa0, fb0); }
        stage1.start_async_dma();
      }
    } else {
      stage0.wait_for_dma_finish();
      load_frags(fa0, fb0, sa0, sb0, 0);
      for (int kt = 0; kt < ksteps; kt += 2) {
        load_frags(fa1, fb1, sa0, sb0, 1); multiply(fa0, fb0); interleave();
        load_frags(fa0, fb0, sa0, sb0, 2); multiply(fa1, fb1); interleave();
        // the `full` word of the next stage is read here and looked at one slice later
        const unsigned seen1 = stage1.peek_dma_finish();
        load_frags(fa1, fb1, sa0, sb0, 3); multiply(fa0, fb0); interleave();
        stage1.wait_for_dma_finish(seen1);
        load_frags(fa0, fb0, sa1, sb1, 0); multiply(fa1, fb1); interleave();
        stage0.start_async_dma();
        load_frags(fa1, fb1, sa1, sb1, 1); multiply(fa0, fb0); interleave();
        load_frags(fa0, fb0, sa1, sb1, 2); multiply(fa1, fb1); interleave();
        const unsigned seen0 = stage0.peek_dma_finish();
        load_frags(fa1, fb1, sa1, sb1, 3); multiply(fa0, fb0); interleave();
        if (kt + 2 < ksteps) {
          stage0.wait_for_dma_finish(seen0);
          load_frags(fa0, fb0, sa0, sb0, 0);
        }
        multiply(fa1, fb1); interleave();
        stage1.start_async_dma();
      }
    }
    // 32 x 32 block: register e of lane L holds row 8*(e/4) + 4*(L/32) + e%4, column L%32
    float* cbase = c + (size_t)(tile_m * shape::kBM + wm) * n + (size_t)tile_n * shape::kBN + wn;
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
          const int col = j * 32 + (lane & 31);
          __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
        }
  }
}

// ---- the same GEMM with the tiles brought in by global_load_lds_dwordx4 ----
// Why: a ds_write_b128 and a ds_read of another wavefront take turns on the LDS, a direct-to-LDS
// load does not hold up the reads (measured: readers + ds_write run as long as the sum of the
// two, readers + global_load_lds as long as the loads alone).  The tiles land unpadded, with the
// chunks of every row XOR-swizzled (STORE_LDS_DIRECT_SWIZZLE); without padding three stages fit
// in LDS (3 x 48 KB), and they are needed: a direct transfer cannot be requested before its stage
// is free, so the memory latency has to fit into two K steps instead of being bridged by
// registers.  Each DMA wavefront keeps two transfers in flight (issue_direct + wait_direct_loads).
template<typename T>
struct Three {
  T a0, a1, a2;
  template<int I> __device__ __forceinline__ T& get() { if constexpr (I == 0) return a0; else if constexpr (I == 1) return a1; else return a2; }
};

#ifdef HIPDMA_SWEEP_VARIANTS
__global__ void __launch_bounds__(kComputeThreads + 2 * kDmaWave)
gemm_bf16_ws_direct(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                    const int m, const int n, const int k, const int walk)
{
  constexpr int WI = 4, WJ = 2, kStages = 3;
  constexpr int kBM = 64 * WI, kBN = 64 * WJ;
  constexpr int kARow = kBK * 2, kBRow = kBN * 2;                 // 128 B and 256 B, unpadded
  constexpr int kAStage = kBM * kARow, kBStage = kBK * kBRow;     // 32 KB and 16 KB
  typedef CudaDMAStrided<false, 16, 16, kARow, kDmaWave, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, kDmaWave, kBK> dma_b_t;
  __shared__ __attribute__((aligned(1024))) char lds_a[kStages][kAStage];
  __shared__ __attribute__((aligned(1024))) char lds_b[kStages][kBStage];
  dma_a_t dma_a(k * 2, kARow, kComputeThreads);
  dma_b_t dma_b(n * 2, kBRow, kComputeThreads + kDmaWave);
  Three<cudaDMACustom> stage{cudaDMACustom(0, 2 * kDmaWave, kComputeThreads, kComputeThreads),
                             cudaDMACustom(1, 2 * kDmaWave, kComputeThreads, kComputeThreads),
                             cudaDMACustom(2, 2 * kDmaWave, kComputeThreads, kComputeThreads)};
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK;

  // One DMA wavefront: tile t lands in stage t % 3.  Tiles t+1 and t+2 are in flight while the
  // compute wavefronts work on tile t: the wavefront waits for tile t (leaving the younger
  // loads in flight), reports it, and then requests tile t+2 as soon as its stage is free.
  auto feed = [&](auto& dma, char* lds, auto stage_bytes, const unsigned short* src, const size_t step)
      __attribute__((always_inline)) {
    constexpr int kStageBytes = decltype(stage_bytes)::value;
    constexpr int kLoads = std::remove_reference<decltype(dma)>::type::loads_per_thread();
    stage.a0.wait_for_dma_start_direct();
    dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src, lds);
    stage.a1.wait_for_dma_start_direct();
    dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + step, lds + kStageBytes);
    auto land = [&](auto cur, auto nxt2, const int t) __attribute__((always_inline)) {
      if (t + 1 < ksteps) hipdma::wait_direct_loads<kLoads>(); else hipdma::wait_direct_loads<0>();
      stage.template get<decltype(cur)::value>().finish_async_dma_direct();
      if (t + 2 < ksteps) {
        stage.template get<decltype(nxt2)::value>().wait_for_dma_start_direct();
        dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + (size_t)(t + 2) * step, lds + decltype(nxt2)::value * kStageBytes);
      }
    };
    typedef std::integral_constant<int, 0> s0;
    typedef std::integral_constant<int, 1> s1;
    typedef std::integral_constant<int, 2> s2;
    for (int t = 0; t < ksteps; t += 3) {
      land(s0(), s2(), t);
      if (t + 1 < ksteps) land(s1(), s0(), t + 1);
      if (t + 2 < ksteps) land(s2(), s1(), t + 2);
    }
  };
  if (dma_a.owns_this_thread()) {
    feed(dma_a, &lds_a[0][0], std::integral_constant<int, kAStage>(), a + (size_t)tile_m * kBM * k, (size_t)kBK);
  } else if (dma_b.owns_this_thread()) {
    feed(dma_b, &lds_b[0][0], std::integral_constant<int, kBStage>(), b + (size_t)tile_n * kBN, (size_t)kBK * n);
  } else {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = (wave >> 1) * 32 * WI, wn = (wave & 1) * 32 * WJ;
    f32x16_t acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    stage.a0.start_async_dma();
    stage.a1.start_async_dma();
    stage.a2.start_async_dma();
    // A fragment of slice ks: row wm + 32*i + lane%32, chunk 2*ks + lane/32 of the 8 chunks of the row,
    // found at chunk position (2*ks + lane/32) ^ key(row); the key only depends on lane%32 here.
    int a_lane[kBK / 16];
    {
      const int row = wm + (lane & 31);
#pragma unroll
      for (int ks = 0; ks < kBK / 16; ++ks)
        a_lane[ks] = row * kARow + hipdma::swizzled_chunk(row, 2 * ks + (lane >> 5), kARow / 16) * 16;
    }
    // B fragment through the transposing read: inside a group of 16 lanes, lane j points at row (j/4) of a
    // 4-row block and at column 4*(j%4); the rows of the "lo" and "hi" reads are 4 apart.  Adding 16 rows
    // (the next slice) does not change a row's key.
    int b_lo[WJ], b_hi[WJ];
    {
      const int j16 = lane & 15;
      const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const int col_bytes = (wn + j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
        b_lo[j] = row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
        b_hi[j] = (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      }
    }
    auto load_frags = [&](bf16x8_t (&fa)[WI], bf16x8_t (&fb)[WJ], const char* sa, const char* sb, const int ks)
        __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
        fa[i] = *(const bf16x8_t*)(sa + i * 32 * kARow + a_lane[ks]);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_lo[j]));
        const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
            (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_hi[j]));
        fb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    };
    auto multiply = [&](const bf16x8_t (&fa)[WI], const bf16x8_t (&fb)[WJ]) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < WI; ++i)
#pragma unroll
        for (int j = 0; j < WJ; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      pin_slice<0, WI * WJ, WI + 2 * WJ>();
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8_t fa0[WI], fb0[WJ], fa1[WI], fb1[WJ];
    // One stage: on entry fa0/fb0 hold its slice 0; on exit they hold slice 0 of the next stage.
    auto k_stage = [&](const cudaDMACustom& cur, const cudaDMACustom& nxt, const int s, const int sn, const bool has_next)
        __attribute__((always_inline)) {
      const char* sa = lds_a[s]; const char* sb = lds_b[s];
      load_frags(fa1, fb1, sa, sb, 1); multiply(fa0, fb0);
      load_frags(fa0, fb0, sa, sb, 2); multiply(fa1, fb1);
      const unsigned seen = nxt.peek_dma_finish();
      load_frags(fa1, fb1, sa, sb, 3); multiply(fa0, fb0);
      if (has_next) {
        nxt.wait_for_dma_finish(seen);
        load_frags(fa0, fb0, lds_a[sn], lds_b[sn], 0);
      }
      multiply(fa1, fb1);
      cur.start_async_dma();
    };
    stage.a0.wait_for_dma_finish();
    load_frags(fa0, fb0, lds_a[0], lds_b[0], 0);
    for (int kt = 0; kt < ksteps; kt += 3) {
      k_stage(stage.a0, stage.a1, 0, 1, kt + 1 < ksteps);
      if (kt + 1 < ksteps) k_stage(stage.a1, stage.a2, 1, 2, kt + 2 < ksteps);
      if (kt + 2 < ksteps) k_stage(stage.a2, stage.a0, 2, 0, kt + 3 < ksteps);
    }
    float* cbase = c + (size_t)(tile_m * kBM + wm) * n + (size_t)tile_n * kBN + wn;
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
          const int col = j * 32 + (lane & 31);
          __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
        }
  }
}
#endif  // HIPDMA_SWEEP_VARIANTS

// ---- 256 x 256 tile, K step 32, four unpadded swizzled stages filled by global_load_lds_dwordx4 ----
// Eight compute wavefronts (2 x 4, 128 x 64 each, two per SIMD) and four DMA wavefronts.  A stage is
// 32 KB (A: 256 rows x 64 B, B: 32 rows x 512 B); each DMA wavefront keeps three transfers in flight.
template<typename T>
struct Four4 {
  T a0, a1, a2, a3;
  template<int I> __device__ __forceinline__ T& get() { if constexpr (I == 0) return a0; else if constexpr (I == 1) return a1; else if constexpr (I == 2) return a2; else return a3; }
};

constexpr int kDirect4DmaThreads = 128;    // DMA threads per operand
constexpr int kDirect4Ahead = 3;           // transfers in flight per DMA wavefront (2: 3 % slower; 4 stages allow no more)
#ifdef HIPDMA_SWEEP_VARIANTS
__global__ void __launch_bounds__(512 + 2 * kDirect4DmaThreads)
gemm_bf16_ws_direct4(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                     const int m, const int n, const int k, const int walk)
{
  constexpr int WI = 4, WJ = 2, WN = 4, kStages = 4, kBK4 = 32, kCompute = 512, kDmaWave = kDirect4DmaThreads;
  constexpr int kBM = 256, kBN = 256;
  constexpr int kARow = kBK4 * 2, kBRow = kBN * 2;                 // 64 B and 512 B, unpadded
  constexpr int kAStage = kBM * kARow, kBStage = kBK4 * kBRow;     // 16 KB and 16 KB
  typedef CudaDMAStrided<false, 16, 16, kARow, kDmaWave, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, kDmaWave, kBK4> dma_b_t;
  __shared__ __attribute__((aligned(1024))) char lds_a[kStages][kAStage];
  __shared__ __attribute__((aligned(1024))) char lds_b[kStages][kBStage];
  dma_a_t dma_a(k * 2, kARow, kCompute);
  dma_b_t dma_b(n * 2, kBRow, kCompute + kDmaWave);
  Four4<cudaDMACustom> stage{cudaDMACustom(0, 2 * kDmaWave, kCompute, kCompute), cudaDMACustom(1, 2 * kDmaWave, kCompute, kCompute),
                             cudaDMACustom(2, 2 * kDmaWave, kCompute, kCompute), cudaDMACustom(3, 2 * kDmaWave, kCompute, kCompute)};
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK4;            // a multiple of four: k is a multiple of 128

  // One DMA wavefront: tile t lands in stage t % 4; tiles t+1 .. t+3 are in flight while the compute
  // wavefronts work on tile t.
  auto feed = [&](auto& dma, char* lds, auto stage_bytes, const unsigned short* src, const size_t step)
      __attribute__((always_inline)) {
    constexpr int kStageBytes = decltype(stage_bytes)::value;
    constexpr int kLoads = std::remove_reference<decltype(dma)>::type::loads_per_thread();
    constexpr int kAhead = kDirect4Ahead;       // transfers in flight per DMA wavefront
    stage.a0.wait_for_dma_start_direct();
    dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src, lds);
    if constexpr (kAhead > 1) {
      stage.a1.wait_for_dma_start_direct();
      dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + step, lds + kStageBytes);
    }
    if constexpr (kAhead > 2) {
      stage.a2.wait_for_dma_start_direct();
      dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + 2 * step, lds + 2 * kStageBytes);
    }
    auto land = [&](auto cur, const int t) __attribute__((always_inline)) {
      constexpr int kCur = decltype(cur)::value, kNext = (kCur + kAhead) % kStages;
      // the younger transfers stay in flight (fewer at the end)
      if (t + kAhead - 1 < ksteps) hipdma::wait_direct_loads<(kAhead - 1) * kLoads>();
      else if (kAhead > 2 && t + 1 < ksteps) hipdma::wait_direct_loads<kLoads>();
      else hipdma::wait_direct_loads<0>();
      stage.template get<kCur>().finish_async_dma_direct();
      if (t + kAhead < ksteps) {
        stage.template get<kNext>().wait_for_dma_start_direct();
        dma.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + (size_t)(t + kAhead) * step, lds + kNext * kStageBytes);
      }
    };
    typedef std::integral_constant<int, 0> s0;
    typedef std::integral_constant<int, 1> s1;
    typedef std::integral_constant<int, 2> s2;
    typedef std::integral_constant<int, 3> s3;
    for (int t = 0; t < ksteps; t += 4) {
      land(s0(), t);
      land(s1(), t + 1);
      land(s2(), t + 2);
      land(s3(), t + 3);
    }
  };
  if (dma_a.owns_this_thread()) {
    feed(dma_a, &lds_a[0][0], std::integral_constant<int, kAStage>(), a + (size_t)tile_m * kBM * k, (size_t)kBK4);
  } else if (dma_b.owns_this_thread()) {
    feed(dma_b, &lds_b[0][0], std::integral_constant<int, kBStage>(), b + (size_t)tile_n * kBN, (size_t)kBK4 * n);
  } else {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = (wave / WN) * 32 * WI, wn = (wave % WN) * 32 * WJ;
    f32x16_t acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    stage.a0.start_async_dma();
    stage.a1.start_async_dma();
    stage.a2.start_async_dma();
    stage.a3.start_async_dma();
    // A fragment of slice ks: row wm + 32*i + lane%32, chunk 2*ks + lane/32 of the 4 chunks of the row, found at
    // chunk position (2*ks + lane/32) ^ key(row); the key only depends on lane%32 (wm and 32*i are multiples of 32).
    int a_lane[kBK4 / 16];
    {
      const int row = wm + (lane & 31);
#pragma unroll
      for (int ks = 0; ks < kBK4 / 16; ++ks)
        a_lane[ks] = row * kARow + hipdma::swizzled_chunk(row, 2 * ks + (lane >> 5), kARow / 16) * 16;
    }
    // B fragment through the transposing read; adding 16 rows (the next slice) does not change a row's key.
    int b_lo[WJ], b_hi[WJ];
    {
      const int j16 = lane & 15;
      const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const int col_bytes = (wn + j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
        b_lo[j] = row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
        b_hi[j] = (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      }
    }
    auto k_stage = [&](const cudaDMACustom& cur, const int s) __attribute__((always_inline)) {
      const char* sa = lds_a[s]; const char* sb = lds_b[s];
      cur.wait_for_dma_finish();
#pragma unroll
      for (int ks = 0; ks < kBK4 / 16; ++ks) {
        bf16x8_t fa[WI], fb[WJ];
#pragma unroll
        for (int i = 0; i < WI; ++i) fa[i] = *(const bf16x8_t*)(sa + i * 32 * kARow + a_lane[ks]);
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
          const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_lo[j]));
          const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_hi[j]));
          fb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
          for (int j = 0; j < WJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
      cur.start_async_dma();
    };
    for (int kt = 0; kt < ksteps; kt += 4) {
      k_stage(stage.a0, 0);
      k_stage(stage.a1, 1);
      k_stage(stage.a2, 2);
      k_stage(stage.a3, 3);
    }
    float* cbase = c + (size_t)(tile_m * kBM + wm) * n + (size_t)tile_n * kBN + wn;
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
          const int col = j * 32 + (lane & 31);
          __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
        }
  }
}
#endif  // HIPDMA_SWEEP_VARIANTS

// ---- the same kernel with A rows of 128 B: an A transfer covers two K steps ----
// A K step of 32 takes 64 B of every A row, half a cache line: the L1 fetches each line of the A
// panel twice, a step apart, and the compute wavefronts wait for the DMA wavefronts (measured with
// s_memtime stamps: 900 of 2350 cycles per step).  Here an A transfer brings 256 rows x 128 B
// (two K steps, whole lines) into one of two 32 KB buffers with its own guard; B keeps the four
// 16 KB stages of one K step each.  The compute wavefronts wait for a B stage every step and for
// an A buffer every other step.
__global__ void __launch_bounds__(512 + 2 * kDirect4DmaThreads)
gemm_bf16_ws_direct4_a64(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                         const int m, const int n, const int k, const int walk)
{
  constexpr int WI = 4, WJ = 2, WN = 4, kBStages = 4, kBK4 = 32, kCompute = 512, kDmaWave = kDirect4DmaThreads;
  constexpr int kBM = 256, kBN = 256;
  constexpr int kARow = 4 * kBK4, kBRow = kBN * 2;                 // 128 B (two K steps) and 512 B, unpadded
  constexpr int kABuf = kBM * kARow, kBStage = kBK4 * kBRow;       // 32 KB and 16 KB
  typedef CudaDMAStrided<false, 16, 16, kARow, kDmaWave, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, kDmaWave, kBK4> dma_b_t;
  __shared__ __attribute__((aligned(1024))) char lds_a[2][kABuf];
  __shared__ __attribute__((aligned(1024))) char lds_b[kBStages][kBStage];
  dma_a_t dma_a(k * 2, kARow, kCompute);
  dma_b_t dma_b(n * 2, kBRow, kCompute + kDmaWave);
  Four4<cudaDMACustom> gb{cudaDMACustom(0, kDmaWave, kCompute, kCompute + kDmaWave), cudaDMACustom(1, kDmaWave, kCompute, kCompute + kDmaWave),
                          cudaDMACustom(2, kDmaWave, kCompute, kCompute + kDmaWave), cudaDMACustom(3, kDmaWave, kCompute, kCompute + kDmaWave)};
  cudaDMACustom ga0(4, kDmaWave, kCompute, kCompute);
  cudaDMACustom ga1(5, kDmaWave, kCompute, kCompute);
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK4;            // a multiple of four: k is a multiple of 128

  if (dma_a.owns_this_thread()) {
    // Transfer p (K steps 2p and 2p+1) lands in buffer p % 2; transfer p+1 is requested as soon as
    // p has landed (its buffer was released when the compute wavefronts left transfer p-1).
    const unsigned short* src = a + (size_t)tile_m * kBM * k;
    const int transfers = ksteps / 2;     // even
    ga0.wait_for_dma_start_direct();
    dma_a.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src, lds_a[0]);
    for (int p = 0; p < transfers; p += 2) {
      hipdma::wait_direct_loads<0>();
      ga0.finish_async_dma_direct();
      ga1.wait_for_dma_start_direct();
      dma_a.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + (size_t)(p + 1) * (2 * kBK4), lds_a[1]);
      hipdma::wait_direct_loads<0>();
      ga1.finish_async_dma_direct();
      if (p + 2 < transfers) {
        ga0.wait_for_dma_start_direct();
        dma_a.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + (size_t)(p + 2) * (2 * kBK4), lds_a[0]);
      }
    }
  } else if (dma_b.owns_this_thread()) {
    // Tile t lands in stage t % 4; tiles t+1 .. t+3 are in flight while the compute wavefronts work on tile t.
    const unsigned short* src = b + (size_t)tile_n * kBN;
    const size_t step = (size_t)kBK4 * n;
    constexpr int kLoads = dma_b_t::loads_per_thread();
    constexpr int kAhead = kDirect4Ahead;
    gb.a0.wait_for_dma_start_direct();
    dma_b.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src, lds_b[0]);
    gb.a1.wait_for_dma_start_direct();
    dma_b.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + step, lds_b[1]);
    gb.a2.wait_for_dma_start_direct();
    dma_b.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + 2 * step, lds_b[2]);
    auto land = [&](auto cur, const int t) __attribute__((always_inline)) {
      constexpr int kCur = decltype(cur)::value, kNext = (kCur + kAhead) % kBStages;
      if (t + kAhead - 1 < ksteps) hipdma::wait_direct_loads<(kAhead - 1) * kLoads>();
      else if (t + 1 < ksteps) hipdma::wait_direct_loads<kLoads>();
      else hipdma::wait_direct_loads<0>();
      gb.template get<kCur>().finish_async_dma_direct();
      if (t + kAhead < ksteps) {
        gb.template get<kNext>().wait_for_dma_start_direct();
        dma_b.template issue_direct<STORE_LDS_DIRECT_SWIZZLE>(src + (size_t)(t + kAhead) * step, lds_b[kNext]);
      }
    };
    for (int t = 0; t < ksteps; t += 4) {
      land(std::integral_constant<int, 0>(), t);
      land(std::integral_constant<int, 1>(), t + 1);
      land(std::integral_constant<int, 2>(), t + 2);
      land(std::integral_constant<int, 3>(), t + 3);
    }
  } else {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int wm = (wave / WN) * 32 * WI, wn = (wave % WN) * 32 * WJ;
    f32x16_t acc[WI][WJ];
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
    gb.a0.start_async_dma();
    gb.a1.start_async_dma();
    gb.a2.start_async_dma();
    gb.a3.start_async_dma();
    ga0.start_async_dma();
    ga1.start_async_dma();
    // A fragment of slice ks (0..3 inside a buffer): row wm + 32*i + lane%32, chunk 2*ks + lane/32 of the 8 chunks
    // of the row, found at chunk position (2*ks + lane/32) ^ key(row); the key only depends on lane%32.
    int a_lane[4];
    {
      const int row = wm + (lane & 31);
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        a_lane[ks] = row * kARow + hipdma::swizzled_chunk(row, 2 * ks + (lane >> 5), kARow / 16) * 16;
    }
    // B fragment through the transposing read; adding 16 rows (the next slice) does not change a row's key.
    int b_lo[WJ], b_hi[WJ];
    {
      const int j16 = lane & 15;
      const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const int col_bytes = (wn + j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
        b_lo[j] = row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
        b_hi[j] = (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      }
    }
    // One K step: B stage s, slices 2*half and 2*half+1 of A buffer `abuf`.
    auto k_step = [&](const cudaDMACustom& gbs, const int s, const cudaDMACustom& gas, const int abuf, auto half)
        __attribute__((always_inline)) {
      constexpr int kHalf = decltype(half)::value;
      const char* sa = lds_a[abuf]; const char* sb = lds_b[s];
      if constexpr (kHalf == 0) gas.wait_for_dma_finish();
      gbs.wait_for_dma_finish();
#pragma unroll
      for (int ks = 0; ks < kBK4 / 16; ++ks) {
        bf16x8_t fa[WI], fb[WJ];
#pragma unroll
        for (int i = 0; i < WI; ++i) fa[i] = *(const bf16x8_t*)(sa + i * 32 * kARow + a_lane[2 * kHalf + ks]);
#pragma unroll
        for (int j = 0; j < WJ; ++j) {
          const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_lo[j]));
          const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_hi[j]));
          fb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
#pragma unroll
        for (int i = 0; i < WI; ++i)
#pragma unroll
          for (int j = 0; j < WJ; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
      gbs.start_async_dma();
      if constexpr (kHalf == 1) gas.start_async_dma();
    };
    typedef std::integral_constant<int, 0> h0;
    typedef std::integral_constant<int, 1> h1;
    for (int kt = 0; kt < ksteps; kt += 4) {
      k_step(gb.a0, 0, ga0, 0, h0());
      k_step(gb.a1, 1, ga0, 0, h1());
      k_step(gb.a2, 2, ga1, 1, h0());
      k_step(gb.a3, 3, ga1, 1, h1());
    }
    float* cbase = c + (size_t)(tile_m * kBM + wm) * n + (size_t)tile_n * kBN + wn;
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
          const int col = j * 32 + (lane & 31);
          __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
        }
  }
}

// ---- 256 x 256 tile without warp specialisation: four wavefronts that each fetch and multiply ----
// The objects are the form of CudaDMAStrided that is not warp-specialised (all 256 threads issue their
// share of a stage with issue_direct; src/examples/stencil/non_warp_specialized_single_buffer.h:47-57 is
// the reference's use of that form).  A wavefront owns a SIMD and a 128 x 128 block of C: 256 accumulator
// registers, 0.5 KB of fragments read per matrix instruction instead of 0.75, no DMA wavefronts to share the
// register file with.  Four stages of one K step (32); a K step starts with one s_barrier: by then every
// wavefront has waited for its own loads of the next stage, so that stage is complete, and every wavefront has
// left the previous stage, so that buffer takes the loads of the stage three steps on.  Those eight loads per
// thread are issued one at a time between groups of four products (issued back to back they hold the wavefront,
// and with it its matrix core, for 550 cycles: the address unit takes one 16-byte load of a wavefront per
// sixteen cycles); the fragments of the next slice, in the second half those of the next stage, are requested
// under the products of the current one.
#ifdef HIPDMA_SWEEP_VARIANTS
__global__ void __launch_bounds__(256)
gemm_bf16_all_direct(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                     const int m, const int n, const int k, const int walk)
{
  constexpr int WI = 4, WJ = 4, kStages = 4, kBK4 = 32, kThreads = 256;
  constexpr int kBM = 256, kBN = 256;
  constexpr int kARow = kBK4 * 2, kBRow = kBN * 2;                 // 64 B and 512 B, unpadded
  constexpr int kAStage = kBM * kARow, kBStage = kBK4 * kBRow;     // 16 KB and 16 KB
  typedef CudaDMAStrided<false, 16, 16, kARow, kThreads, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, kThreads, kBK4> dma_b_t;
  constexpr int kLoads = dma_a_t::loads_per_thread() + dma_b_t::loads_per_thread();     // per stage and thread
  __shared__ __attribute__((aligned(1024))) char lds_a[kStages][kAStage];
  __shared__ __attribute__((aligned(1024))) char lds_b[kStages][kBStage];
  dma_a_t dma_a(k * 2, kARow);
  dma_b_t dma_b(n * 2, kBRow);
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK4;            // a multiple of four
  const int klast = ksteps - 1;
  const unsigned short* const src_a = a + (size_t)tile_m * kBM * k;
  const unsigned short* const src_b = b + (size_t)tile_n * kBN;
  const size_t step_b = (size_t)kBK4 * n;
  // Stage t of the K loop into buffer t % 4: round g of the A loads (g < 4) or round g - 4 of the B loads.  Past
  // the end the last stage is requested again (into a buffer nobody reads any more): the loop keeps one shape and
  // one wait count.
  static_assert(dma_a_t::loads_per_thread() == 4 && dma_b_t::loads_per_thread() == 4, "eight loads per thread and stage");
  auto issue = [&](const int t, const int buf, const int g) __attribute__((always_inline)) {
    const int tt = t < klast ? t : klast;
    if (g < 4) dma_a.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(src_a + (size_t)tt * kBK4, lds_a[buf], g, 1);
    else dma_b.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(src_b + (size_t)tt * step_b, lds_b[buf], g - 4, 1);
  };
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32 * WI, wn = (wave & 1) * 32 * WJ;
  f32x16_t acc[WI][WJ];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  int a_lane[kBK4 / 16];
  {
    const int row = wm + (lane & 31);
#pragma unroll
    for (int ks = 0; ks < kBK4 / 16; ++ks)
      a_lane[ks] = row * kARow + hipdma::swizzled_chunk(row, 2 * ks + (lane >> 5), kARow / 16) * 16;
  }
  int b_lo[WJ], b_hi[WJ];
  {
    const int j16 = lane & 15;
    const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int col_bytes = (wn + j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
      b_lo[j] = row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      b_hi[j] = (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
    }
  }
  auto load_frags = [&](bf16x8_t (&fa)[WI], bf16x8_t (&fb)[WJ], const int buf, const int ks) __attribute__((always_inline)) {
    const char* sa = lds_a[buf]; const char* sb = lds_b[buf];
#pragma unroll
    for (int i = 0; i < WI; ++i) fa[i] = *(const bf16x8_t*)(sa + i * 32 * kARow + a_lane[ks]);
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_lo[j]));
      const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
          (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_hi[j]));
      fb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  };
  // Half a K step: the sixteen products of the slice in (fa, fb) in four groups of four.  Under the first three
  // groups the fragments of the slice (nbuf, nks) are requested into (na, nb): the four A blocks, then two B blocks
  // twice.  Behind every group goes one load of stage t + 3.  Nothing moves across the ends of a group.
  auto half_step = [&](const bf16x8_t (&fa)[WI], const bf16x8_t (&fb)[WJ], bf16x8_t (&na)[WI], bf16x8_t (&nb)[WJ],
                       const int nbuf, const int nks, const int t, const int buf, const int first_load)
      __attribute__((always_inline)) {
    const char* sa = lds_a[nbuf]; const char* sb = lds_b[nbuf];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      if (i == 0) {
#pragma unroll
        for (int q = 0; q < WI; ++q) na[q] = *(const bf16x8_t*)(sa + q * 32 * kARow + a_lane[nks]);
      } else if (i < 3) {
#pragma unroll
        for (int j = 2 * (i - 1); j < 2 * i; ++j) {
          const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + nks * 16 * kBRow + b_lo[j]));
          const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + nks * 16 * kBRow + b_hi[j]));
          nb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
#pragma unroll
      for (int j = 0; j < WJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
      // product, request, product, request, ...
#pragma unroll
      for (int q = 0; q < WJ; ++q) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i < 3) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      issue(t + 3, (buf + 3) % kStages, first_load + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  bf16x8_t fa0[WI], fb0[WJ], fa1[WI], fb1[WJ];
#pragma unroll
  for (int g = 0; g < 8; ++g) issue(0, 0, g);
#pragma unroll
  for (int g = 0; g < 8; ++g) issue(1, 1, g);
#pragma unroll
  for (int g = 0; g < 8; ++g) issue(2, 2, g);
  hipdma::wait_direct_loads<2 * kLoads>();
  __builtin_amdgcn_s_barrier();
  load_frags(fa0, fb0, 0, 0);
  // One K step on buffer `buf`: on entry fa0/fb0 hold its first slice and stages t + 1, t + 2 are in flight; on
  // exit fa0/fb0 hold the first slice of the next step.
  auto k_step = [&](const int t, const int buf) __attribute__((always_inline)) {
    hipdma::wait_direct_loads<kLoads>();          // this thread's part of stage t + 1 (stage t + 2 stays in flight)
    __builtin_amdgcn_s_barrier();
    half_step(fa0, fb0, fa1, fb1, buf, 1, t, buf, 0);
    half_step(fa1, fb1, fa0, fb0, (buf + 1) % kStages, 0, t, buf, 4);
  };
  for (int kt = 0; kt < ksteps; kt += 4) {
    k_step(kt, 0);
    k_step(kt + 1, 1);
    k_step(kt + 2, 2);
    k_step(kt + 3, 3);
  }
  hipdma::wait_direct_loads<0>();
  float* cbase = c + (size_t)(tile_m * kBM + wm) * n + (size_t)tile_n * kBN + wn;
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
        const int col = j * 32 + (lane & 31);
        __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
      }
}
#endif  // HIPDMA_SWEEP_VARIANTS

// ---- the same kernel with A transfers of two K steps (rows of 128 B) ----
// A K step of 32 takes 64 B of an A row, half a cache line, and the L1 asks the L2 for every line of the A panel
// twice (TCP_TCC_READ_REQ: 12.8 M requests per 4096^3 launch instead of 8.4 M).  Here an A transfer is 256 rows x
// 128 B for two K steps.  Three A buffers (96 KB) and the four B stages (64 KB) are all of the LDS: an A buffer is
// free two K steps after its last read and its next transfer has to be complete a step before its first, so two
// buffers would leave it one K step to land.  The A buffers form a ring indexed at run time (three does not divide the K steps of
// every problem); a K step issues 2 * WI loads, WI of B and half an A transfer.  <4, 4> is that kernel.  With WI = 2 the tile is
// 128 x 128; against the warp-specialised kernel of that tile it saves the ds_writes and the hand-offs (2560 x 2560 x 1024 21.5 -> 18 us,
// 1024^3 12.4 -> 10.3, both with the same order of tiles).
// STAGES is how far the loads run ahead: K step t requests B stage t + STAGES - 1, and A goes as far in STAGES / 2 + 1 buffers.  <2, 4>
// takes 80 KB of LDS and two workgroups share a compute unit.  Where the grid gives a compute unit one, its two K steps in flight
// do not cover the latency of DRAM: <2, 8>, 144 KB, has six (1408 x 1536 x 5248, 132 tiles: 44 us from the caches and 62 from DRAM with
// <2, 4>, 36 and 48 with <2, 8>; the warp-specialised kernel 44 and 47).
// With one wavefront per SIMD every instruction between two matrix instructions counts: the sources are pointers that move on with the
// requests, kept in scalar registers (left alone the compiler forms them by vector additions and v_readfirstlane in <2, 8>: 128 x 128 x 1536
// from the caches 13.5 us, 12.6 with the sources pinned, 12.2 with them moving; 4096^3 with <4, 4> 105.7 -> 104.7).
// Counters (2048 x 1024 x 4096, one workgroup per compute unit, <2, 4> / <2, 8>): matrix cores busy 43 / 53 %, LDS busy 21 / 27 %, no
// bank conflicts, wavefronts waiting for data 34 / 19 % of their cycles and for an issue slot 20 / 25 %; a K step takes a wavefront
// 600 / 480 cycles for 256 of matrix instructions and about 60 others.  Nothing is saturated: with nothing else resident the waits at
// the barrier of a K step and the issue of those 60 add up.
template<int WI, int STAGES>
__global__ void __launch_bounds__(256)
gemm_bf16_all_direct_a64(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                         const int m, const int n, const int k, const int walk)
{
  static_assert(STAGES == 4 || STAGES == 8, "the loop below takes four K steps at a time");
  constexpr int WJ = WI, kBStages = STAGES, kAAhead = STAGES / 2, kABufs = kAAhead + 1, kBK4 = 32, kThreads = 256;
  constexpr int kBM = 64 * WI, kBN = 64 * WJ;
  constexpr int kARow = 4 * kBK4, kBRow = kBN * 2;                 // 128 B (two K steps) and 128 * WI B, unpadded
  constexpr int kABuf = kBM * kARow, kBStage = kBK4 * kBRow;       // 8 * WI and 4 * WI KB
  typedef CudaDMAStrided<false, 16, 16, kARow, kThreads, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, kThreads, kBK4> dma_b_t;
  static_assert(dma_a_t::loads_per_thread() == 2 * WI && dma_b_t::loads_per_thread() == WI, "2 * WI loads per thread and K step");
  constexpr int kLoads = 2 * WI;
  __shared__ __attribute__((aligned(1024))) char lds_a[kABufs * kABuf];
  __shared__ __attribute__((aligned(1024))) char lds_b[kBStages][kBStage];
  dma_a_t dma_a(k * 2, kARow);
  dma_b_t dma_b(n * 2, kBRow);
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int ksteps = k / kBK4;            // a multiple of four
  const int klast = ksteps - 1, dlast = ksteps / 2 - 1;
  const unsigned short* next_a = a + (size_t)tile_m * kBM * k;      // A transfer and B stage to request next; both go up one by one
  const unsigned short* next_b = b + (size_t)tile_n * kBN;
  const size_t step_b = (size_t)kBK4 * n;
  // Round r of the B stage of K step t into B buffer `buf`; round r of A transfer d (K steps 2d, 2d+1) into A
  // buffer `buf`.  Past the end the last one is requested again, into a buffer nobody reads any more.  The source moves on with
  // the last round.
  auto issue_b = [&](const int t, const int buf, const int r) __attribute__((always_inline)) {
    dma_b.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(next_b, lds_b[buf], r, 1);
    if (r == WI - 1) { next_b += t < klast ? step_b : 0; asm("" : "+s"(next_b)); }
  };
  auto issue_a = [&](const int d, const int buf, const int r) __attribute__((always_inline)) {
    dma_a.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(next_a, lds_a + buf * kABuf, r, 1);
    if (r == 2 * WI - 1) { next_a += d < dlast ? 2 * kBK4 : 0; asm("" : "+s"(next_a)); }
  };
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * 32 * WI, wn = (wave & 1) * 32 * WJ;
  f32x16_t acc[WI][WJ];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  // A fragment of slice q (0..3 inside a buffer): row wm + 32*i + lane%32, chunk 2*q + lane/32 of the 8 chunks of the row
  int a_lane[4];
  {
    const int row = wm + (lane & 31);
#pragma unroll
    for (int q = 0; q < 4; ++q)
      a_lane[q] = row * kARow + hipdma::swizzled_chunk(row, 2 * q + (lane >> 5), kARow / 16) * 16;
  }
  int b_lo[WJ], b_hi[WJ];
  {
    const int j16 = lane & 15;
    const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int col_bytes = (wn + j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
      b_lo[j] = row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      b_hi[j] = (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
    }
  }
  // The group of products under which the B fragments are first requested, and reads behind each product: with four groups A, B and
  // B take one each, with two everything goes under the first, to have landed after the second.
  constexpr int kBFrom = WI == 4 ? 1 : 0, kReads = WI == 4 ? 1 : 3;
  // Half a K step: WI * WI products in WI groups; under the first three (one) the fragments of slice q of A buffer
  // `abuf` and of slice ks of B stage `bbuf` are requested into (na, nb); `after_group(i)` places the loads.
  auto half_step = [&](const bf16x8_t (&fa)[WI], const bf16x8_t (&fb)[WJ], bf16x8_t (&na)[WI], bf16x8_t (&nb)[WJ],
                       const int abuf, const int q, const int bbuf, const int ks, auto after_group)
      __attribute__((always_inline)) {
    const char* sa = lds_a + abuf * kABuf; const char* sb = lds_b[bbuf];
#pragma unroll
    for (int i = 0; i < WI; ++i) {
      if (i == 0) {
#pragma unroll
        for (int r = 0; r < WI; ++r) na[r] = *(const bf16x8_t*)(sa + r * 32 * kARow + a_lane[q]);
      }
      if (i >= kBFrom && i < kBFrom + WJ / 2) {
#pragma unroll
        for (int j = 2 * (i - kBFrom); j < 2 * (i - kBFrom) + 2; ++j) {
          const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_lo[j]));
          const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
              (__attribute__((address_space(3))) bf16x4_t*)(sb + ks * 16 * kBRow + b_hi[j]));
          nb[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
      }
#pragma unroll
      for (int j = 0; j < WJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i], fb[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int r = 0; r < WJ; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        if (i < kBFrom + WJ / 2) __builtin_amdgcn_sched_group_barrier(0x100, kReads, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      after_group(i);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  bf16x8_t fa0[WI], fb0[WJ], fa1[WI], fb1[WJ];
  // Group g of the requests, in the order that all wait counts assume: B stage g and the half of A transfer (g + 1) / 2 that goes with it
  // (the first half with odd g); group 0 is B stage 0 and all of A transfer 0.  K step t reads groups up to t + 1 and issues group
  // t + STAGES - 1.
  auto issue_of_group = [&](const int g, const int i) __attribute__((always_inline)) {
    issue_b(g, g % kBStages, i);
    issue_a((g + 1) / 2, (g + 1) / 2 % kABufs, (g % 2 == 1 ? 0 : WI) + i);
  };
  constexpr int kFirstGroups = 2;             // behind group 0, before the first product
#pragma unroll
  for (int r = 0; r < 2 * WI; ++r) issue_a(0, 0, r);
#pragma unroll
  for (int r = 0; r < WI; ++r) issue_b(0, 0, r);
#pragma unroll
  for (int g = 1; g <= kFirstGroups; ++g) {
#pragma unroll
    for (int r = 0; r < WI; ++r) issue_of_group(g, r);
  }
  hipdma::wait_direct_loads<kFirstGroups * kLoads>();
  __builtin_amdgcn_s_barrier();
  // first slice of K step 0
  {
#pragma unroll
    for (int r = 0; r < WI; ++r) fa0[r] = *(const bf16x8_t*)(lds_a + r * 32 * kARow + a_lane[0]);
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)(lds_b[0] + b_lo[j]));
      const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)(lds_b[0] + b_hi[j]));
      fb0[j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  }
  // One K step t on B buffer bbuf and slices (2*h, 2*h+1) of A buffer abuf; the next step starts in A buffer nabuf at slice nq.  It
  // issues B stage t + STAGES - 1 into the buffer that step t - 1 has left and rounds [ar, ar + WI) of A transfer ad into A buffer aibuf.
  auto k_step = [&](const int t, const int bbuf, const int abuf, const int h, const int nabuf, const int nq,
                    const int ad, const int aibuf, const int ar) __attribute__((always_inline)) {
    // everything up to K step t + 2 - STAGES, which issued what step t + 1 reads; what the steps since then issued stays in flight
    hipdma::wait_direct_loads<(kBStages - 3) * kLoads>();
    __builtin_amdgcn_s_barrier();
    half_step(fa0, fb0, fa1, fb1, abuf, 2 * h + 1, bbuf, 1, [&](const int i) __attribute__((always_inline)) {
      issue_b(t + kBStages - 1, (bbuf + kBStages - 1) % kBStages, i);
    });
    half_step(fa1, fb1, fa0, fb0, nabuf, nq, (bbuf + 1) % kBStages, 0, [&](const int i) __attribute__((always_inline)) {
      issue_a(ad, aibuf, ar + i);
    });
  };
  auto ring = [](const int i) __attribute__((always_inline)) { return i < kABufs ? i : i - kABufs; };
  int ab0 = 0;                                // A buffer of transfer kt / 2
  // K steps kt to kt + 3, the first in B buffer B0
  auto four_steps = [&](const int kt, auto first) __attribute__((always_inline)) {
    constexpr int B0 = decltype(first)::value;
    const int ab1 = ring(ab0 + 1), ab2 = ring(ab0 + 2);       // transfers kt / 2 + 1 and kt / 2 + 2
    const int abn = ring(ab0 + kAAhead);      // transfer kt / 2 + kAAhead, requested during K steps kt and kt + 1
    const int d = (kt >> 1) + kAAhead;
    k_step(kt, B0, ab0, 0, ab0, 2, d, abn, 0);
    k_step(kt + 1, B0 + 1, ab0, 1, ab1, 0, d, abn, WI);
    k_step(kt + 2, B0 + 2, ab1, 0, ab1, 2, d + 1, ab0, 0);    // the next transfer takes the buffer transfer kt / 2 has left
    k_step(kt + 3, B0 + 3, ab1, 1, ab2, 0, d + 1, ab0, WI);
    ab0 = ab2;
  };
  // With eight stages the first four K steps issue two groups each, 3 to 10, and so reach the distance that the others keep.  (All six
  // groups before the first product held it up: 128 x 128 x 768 from the caches 7.9 us, 7.6 so, 7.4 with <2, 4>.)  Groups 8 to 10 go where K steps 0 to 2 have been.
  auto ramp_step = [&](auto step) __attribute__((always_inline)) {
    constexpr int t = decltype(step)::value, issued = kFirstGroups + 2 * t;
    hipdma::wait_direct_loads<(issued - (t + 1)) * kLoads>();
    __builtin_amdgcn_s_barrier();
    half_step(fa0, fb0, fa1, fb1, t / 2, 2 * (t % 2) + 1, t, 1, [&](const int i) __attribute__((always_inline)) { issue_of_group(issued + 1, i); });
    half_step(fa1, fb1, fa0, fb0, (t + 1) / 2, t % 2 == 0 ? 2 : 0, t + 1, 0, [&](const int i) __attribute__((always_inline)) { issue_of_group(issued + 2, i); });
  };
  // the B buffers are named by constants: one turn of the loop goes through all of them
  if constexpr (kBStages == 8) {
    ramp_step(std::integral_constant<int, 0>());
    ramp_step(std::integral_constant<int, 1>());
    ramp_step(std::integral_constant<int, 2>());
    ramp_step(std::integral_constant<int, 3>());
    ab0 = 2;
    for (int kt = 4; kt < ksteps; kt += 8) {
      four_steps(kt, std::integral_constant<int, 4>());
      if (kt + 4 < ksteps) four_steps(kt + 4, std::integral_constant<int, 0>());
    }
  } else {
    for (int kt = 0; kt < ksteps; kt += 4) four_steps(kt, std::integral_constant<int, 0>());
  }
  hipdma::wait_direct_loads<0>();
  float* cbase = c + (size_t)(tile_m * kBM + wm) * n + (size_t)tile_n * kBN + wn;
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int row = i * 32 + 8 * (e / 4) + 4 * (lane >> 5) + (e % 4);
        const int col = j * 32 + (lane & 31);
        __builtin_nontemporal_store(acc[i][j][e], &cbase[(size_t)row * n + col]);
      }
}

// ---- small grids: the K steps dealt out to the wavefronts of a workgroup ----
// A grid of few tiles leaves compute units idle, and a product of few rows and columns is one long chain of K steps per tile.  Here the tile
// is 32 * WI x 32 * WJ, every one of the WAVES wavefronts holds all of it, and wavefront w takes the K steps (of 64) w, w + WAVES, ...  A
// wavefront brings its own operands with direct-to-LDS loads into a stage of its own and is the only one to read them, so nothing in the loop
// waits for another wavefront: no barrier, no hand-off, s_waitcnt alone.  It takes a whole stage into registers, and while it multiplies
// it the next one is on its way into the same place.  At the end the partial tiles are added through LDS.
// What bounds the loop is the way into the LDS: direct loads land at 64 B a cycle of a compute unit, however many wavefronts issue them (16 cycles
// per KB; fragment reads take 4).  32 x 32 brings 4 KB per K = 32, 64 cycles, and takes 70; 64 x 64 brings 8 KB, 128 cycles, and takes 126 to
// 144, against 417 to 434 of a 128 x 128 tile with four wavefronts, which is 4 to 16 times the work.
// Measured (us, former choice -> this, from the caches and from DRAM): 512^3 6.0 -> 3.5 and 7.2 -> 4.0; 128 x 128 x 8192 48.7 -> 9.9 and 48.9 ->
// 16.6; 1024^3 9.2 -> 6.2 and 10.1 -> 7.3; 2560 x 384 x 6528 40.7 -> 22.4 and 60 -> 28.
// Stages of K = 32, two per wavefront, read A in pieces of 64 B, half a cache line: 1024 x 1024 x 4096 18.5 us, 16.4 so.  Four wavefronts with four
// such stages 18.9.  Tiles of 64 x 128 the same way start and end too slowly (1408^3 11.8 against 11.3 with 64 x 64).
template<int WI, int WJ, int WAVES>
__global__ void __launch_bounds__(64 * WAVES)
gemm_bf16_dealt_steps(const unsigned short* __restrict__ a, const unsigned short* __restrict__ b, float* __restrict__ c,
                      const int m, const int n, const int k, const int walk)
{
  constexpr int kSlices = 4, kStepK = 16 * kSlices, kBM = 32 * WI, kBN = 32 * WJ;
  constexpr int kARow = 2 * kStepK, kBRow = 2 * kBN;
  constexpr int kAStage = kBM * kARow, kStage = kAStage + kStepK * kBRow;
  typedef CudaDMAStrided<false, 16, 16, kARow, 64, kBM> dma_a_t;
  typedef CudaDMAStrided<false, 16, 16, kBRow, 64, kStepK> dma_b_t;
  constexpr int kALoads = dma_a_t::loads_per_thread(), kLoads = kALoads + dma_b_t::loads_per_thread();
  constexpr int kProducts = WI * WJ;                               // per slice of 16
  constexpr int kShare = 16 * kProducts / WAVES;                   // accumulators that a wavefront adds up and stores in the end
  __shared__ __attribute__((aligned(1024))) char lds[WAVES * kStage];
  static_assert(kProducts * 4096 <= kStage, "a partial tile takes the place of a stage");
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  dma_a_t dma_a(k * 2, kARow, 64 * wave);
  dma_b_t dma_b(n * 2, kBRow, 64 * wave);
  int tile_m, tile_n;
  tile_of_workgroup(blockIdx.x, m / kBM, n / kBN, walk, tile_m, tile_n);
  const int all_steps = k / kStepK;
  const int steps = (all_steps - wave + WAVES - 1) / WAVES;        // of this wavefront
  const unsigned short* next_a = a + (size_t)tile_m * kBM * k + wave * kStepK;      // the stage to request next
  const unsigned short* next_b = b + (size_t)tile_n * kBN + (size_t)wave * kStepK * n;
  const size_t step_b = (size_t)WAVES * kStepK * n;
  // as an LDS address: a generic one would be compared with null at every load
  char* const stage = (char*)((HIPDMA_LDS_AS char*)lds + wave * kStage);
  auto issue = [&](const int g) __attribute__((always_inline)) {
    if (g < kALoads) dma_a.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(next_a, stage, g, 1);
    else dma_b.template issue_direct_part<STORE_LDS_DIRECT_SWIZZLE, true>(next_b, stage + kAStage, g - kALoads, 1);
    if (g == kLoads - 1) {
      next_a += WAVES * kStepK; next_b += step_b;
      asm("" : "+s"(next_a));               // kept in scalar registers
      asm("" : "+s"(next_b));
    }
  };
  f32x16_t acc[WI][WJ];
#pragma unroll
  for (int i = 0; i < WI; ++i)
#pragma unroll
    for (int j = 0; j < WJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  int a_lane[kSlices], b_lo[WJ], b_hi[WJ];
  {
    const int row = lane & 31;
#pragma unroll
    for (int ks = 0; ks < kSlices; ++ks) a_lane[ks] = row * kARow + hipdma::swizzled_chunk(row, 2 * ks + (lane >> 5), kARow / 16) * 16;
  }
  {
    const int j16 = lane & 15;
    const int row = (lane >> 5) * 8 + (j16 >> 2);
#pragma unroll
    for (int j = 0; j < WJ; ++j) {
      const int col_bytes = (j * 32 + ((lane >> 4) & 1) * 16 + (j16 & 3) * 4) * 2;
      b_lo[j] = kAStage + row * kBRow + hipdma::swizzled_chunk(row, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
      b_hi[j] = kAStage + (row + 4) * kBRow + hipdma::swizzled_chunk(row + 4, col_bytes >> 4, kBRow / 16) * 16 + (col_bytes & 15);
    }
  }
  bf16x8_t fa[kSlices][WI], fb[kSlices][WJ];
  auto load_frags = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < kSlices; ++ks) {
#pragma unroll
      for (int i = 0; i < WI; ++i) fa[ks][i] = *(const bf16x8_t*)(stage + i * 32 * kARow + a_lane[ks]);
#pragma unroll
      for (int j = 0; j < WJ; ++j) {
        const bf16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)(stage + ks * 16 * kBRow + b_lo[j]));
        const bf16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((__attribute__((address_space(3))) bf16x4_t*)(stage + ks * 16 * kBRow + b_hi[j]));
        fb[ks][j] = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    }
  };
  // The products of a stage, with `more` the loads of the next one spread behind them.
  auto multiply = [&](auto more) __attribute__((always_inline)) {
    constexpr int kAll = kSlices * kProducts, kEach = (kLoads + kAll - 1) / kAll;      // loads behind a product
#pragma unroll
    for (int p = 0; p < kAll; ++p) {
      const int ks = p / kProducts, i = p % kProducts / WJ, j = p % WJ;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[ks][i], fb[ks][j], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int g = p * kEach; g < (p + 1) * kEach && g < kLoads; ++g) issue(g);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (steps > 0) {
#pragma unroll
    for (int g = 0; g < kLoads; ++g) issue(g);
    hipdma::wait_direct_loads<0>();
    load_frags();
    for (int t = 1; t < steps; ++t) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");           // the stage has been read: the next one may land
      multiply(std::true_type());
      hipdma::wait_direct_loads<0>();
      load_frags();
    }
    multiply(std::false_type());
  }
  // The accumulators go to LDS as they lie in the registers; every wavefront then adds up kShare of them, in the order of the wavefronts,
  // and stores those.  Wavefronts beyond the K steps have nothing to add.
  const int active = all_steps < WAVES ? all_steps : WAVES;
  constexpr int kPiece = kShare % 4 == 0 ? 4 : 2;                  // accumulators of one LDS access
  typedef float piece_t __attribute__((ext_vector_type(kPiece)));
  constexpr int kPieces = 16 * kProducts / kPiece;
  auto piece_of = [&](const int partial, const int q) __attribute__((always_inline)) {
    return (piece_t*)(lds + ((partial * kPieces + q) * 64 + lane) * sizeof(piece_t));
  };
  __syncthreads();                          // the stages are no longer read
  if (wave < active) {
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      piece_t v;
#pragma unroll
      for (int e = 0; e < kPiece; ++e) v[e] = acc[q * kPiece / 16 / WJ][q * kPiece / 16 % WJ][q * kPiece % 16 + e];
      *piece_of(wave, q) = v;
    }
  }
  __syncthreads();
  piece_t sum[kShare / kPiece];
#pragma unroll
  for (int q = 0; q < kShare / kPiece; ++q) sum[q] = *piece_of(0, wave * (kShare / kPiece) + q);
#pragma unroll
  for (int w = 1; w < WAVES; ++w)
    if (w < active) {
#pragma unroll
      for (int q = 0; q < kShare / kPiece; ++q) sum[q] += *piece_of(w, wave * (kShare / kPiece) + q);
    }
  float* const cbase = c + (size_t)tile_m * kBM * n + (size_t)tile_n * kBN;
#pragma unroll
  for (int q = 0; q < kShare / kPiece; ++q)
#pragma unroll
    for (int e = 0; e < kPiece; ++e) {
      const int at = wave * kShare + q * kPiece + e, block = at / 16, reg = at % 16;
      const int row = block / WJ * 32 + 8 * (reg / 4) + 4 * (lane >> 5) + reg % 4, col = block % WJ * 32 + (lane & 31);
      __builtin_nontemporal_store(sum[q][e], &cbase[(size_t)row * n + col]);
    }
}

template<int WI, int WJ, int WAVES>
int launch_dealt_steps(const uint16_t* d_a, const uint16_t* d_b, float* d_c, int m, int n, int k, hipStream_t stream)
{
  constexpr int kPerCu = 2 * WAVES * (WI + WJ) * 4096 <= (160 << 10) ? 2 : 1;
  hipLaunchKernelGGL((gemm_bf16_dealt_steps<WI, WJ, WAVES>), dim3((unsigned)((m / (32 * WI)) * (n / (32 * WJ)))), dim3(64 * WAVES), 0, stream,
                     d_a, d_b, d_c, m, n, k, tile_walk(m, n, k, 32 * WI, 32 * WJ, kPerCu));
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

template<int WI, int WJ, int WM = 2, int WN = 2>
int launch_gemm(const uint16_t* d_a, const uint16_t* d_b, float* d_c, int m, int n, int k, hipStream_t stream)
{
  typedef GemmShape<WI, WJ, WM, WN> shape;
  CUDADMA_REQUIRE((m % shape::kBM) == 0 && (n % shape::kBN) == 0,
                  "this variant needs m a multiple of %d and n of %d (got %d x %d)", shape::kBM, shape::kBN, m, n);
  const long long grid = (long long)(m / shape::kBM) * (n / shape::kBN);
  CUDADMA_REQUIRE(grid <= 0x7fffffffLL, "grid too large");
  hipLaunchKernelGGL((gemm_bf16_ws<WI, WJ, WM, WN>), dim3((unsigned)grid), dim3(shape::kCompute + 2 * kDmaWave), 0, stream,
                     d_a, d_b, d_c, m, n, k, tile_walk(m, n, k, shape::kBM, shape::kBN, shape::kPerCu));
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

template<int B_STAGES>
int launch_all_direct_128(const uint16_t* d_a, const uint16_t* d_b, float* d_c, int m, int n, int k, hipStream_t stream)
{
  const long long grid = (long long)(m / 128) * (n / 128);
  CUDADMA_REQUIRE(grid <= 0x7fffffffLL, "grid too large");
  hipLaunchKernelGGL((gemm_bf16_all_direct_a64<2, B_STAGES>), dim3((unsigned)grid), dim3(256), 0, stream, d_a, d_b, d_c, m, n, k,
                     tile_walk(m, n, k, 128, 128, B_STAGES == 8 ? 1 : 2));
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

}  // namespace

extern "C" int cudadma_gemm_bf16(const uint16_t* d_a, const uint16_t* d_b, float* d_c, int m, int n, int k,
                                 int variant, void* stream)
{
  CUDADMA_REQUIRE(m > 0 && n > 0 && k > 0, "dimensions must be positive");
  CUDADMA_REQUIRE((m % 128) == 0 && (n % 128) == 0 && (k % (2 * kBK)) == 0,
                  "m, n and k must be multiples of 128 (got %d x %d x %d)", m, n, k);
  if (variant < 0 || variant >= cudadma_num_variants(CUDADMA_WORKLOAD_GEMM)) {
    cudadma_host::set_error("gemm has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  CUDADMA_REQUIRE(d_a != nullptr && d_b != nullptr && d_c != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_a, 16) && cudadma_host::aligned_to(d_b, 16) && cudadma_host::aligned_to(d_c, 16),
                  "pointers must be 16-byte aligned");
  CUDADMA_REQUIRE((long long)k * 2 <= 0x7fffffffLL && (long long)n * 2 <= 0x7fffffffLL, "row pitch must fit an int");
  hipStream_t s = (hipStream_t)stream;
  if (variant == 0) {
    using dispatch::GemmForm;
    switch (dispatch::gemm_form(m, n, k, workloads::device_cus())) {
      case GemmForm::kDealt32x32: return launch_dealt_steps<1, 1, 8>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::kDealt32x64: return launch_dealt_steps<1, 2, 8>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::kDealt64x64: return launch_dealt_steps<2, 2, 8>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::kDealt64x64Two: return launch_dealt_steps<2, 2, 4>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::k128Far: return launch_all_direct_128<8>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::k128: return launch_all_direct_128<4>(d_a, d_b, d_c, m, n, k, s);
      case GemmForm::k256: variant = 9; break;
      case GemmForm::kLongRows: variant = 1; break;
    }
  }
  switch (variant) {
    case 1: return launch_gemm<2, 2>(d_a, d_b, d_c, m, n, k, s);
    case 2: return launch_gemm<2, 4>(d_a, d_b, d_c, m, n, k, s);
    case 3: return launch_gemm<4, 2>(d_a, d_b, d_c, m, n, k, s);
#ifdef HIPDMA_SWEEP_VARIANTS
    case 5: return launch_gemm<4, 2, 2, 4>(d_a, d_b, d_c, m, n, k, s);
#endif
    case 6: case 7: case 8: case 9: {
      CUDADMA_REQUIRE((m % 256) == 0 && (n % 256) == 0, "this variant needs m and n multiples of 256 (got %d x %d)", m, n);
      // 6 and 7 go over to 64-bit row offsets by themselves (issue_direct), 8 and 9 are compiled for lane offsets alone
      CUDADMA_REQUIRE(variant <= 7 || dispatch::direct_rows_fit(n, k), "rows of %d x %d are too long for the lane offsets of this variant (0, 1 and 7 take them)", k, n);
      const long long grid = (long long)(m / 256) * (n / 256);
      CUDADMA_REQUIRE(grid <= 0x7fffffffLL, "grid too large");
      const int walk = tile_walk(m, n, k, 256, 256, 1);
      if (variant == 7) hipLaunchKernelGGL(gemm_bf16_ws_direct4_a64, dim3((unsigned)grid), dim3(512 + 2 * kDirect4DmaThreads), 0, s, d_a, d_b, d_c, m, n, k, walk);
      else if (variant == 9) hipLaunchKernelGGL((gemm_bf16_all_direct_a64<4, 4>), dim3((unsigned)grid), dim3(256), 0, s, d_a, d_b, d_c, m, n, k, walk);
#ifdef HIPDMA_SWEEP_VARIANTS
      else if (variant == 6) hipLaunchKernelGGL(gemm_bf16_ws_direct4, dim3((unsigned)grid), dim3(512 + 2 * kDirect4DmaThreads), 0, s, d_a, d_b, d_c, m, n, k, walk);
      else hipLaunchKernelGGL(gemm_bf16_all_direct, dim3((unsigned)grid), dim3(256), 0, s, d_a, d_b, d_c, m, n, k, walk);
#else
      else CUDADMA_REQUIRE(false, "gemm variant %d is a sweep kernel: build the library with make EXTRA=-DHIPDMA_SWEEP_VARIANTS", variant);
#endif
      CUDADMA_HIP_CHECK(hipGetLastError());
      return CUDADMA_OK;
    }
    default: {
#ifdef HIPDMA_SWEEP_VARIANTS
      CUDADMA_REQUIRE((m % 256) == 0, "this variant needs m a multiple of 256 (got %d)", m);
      const long long grid = (long long)(m / 256) * (n / 128);
      CUDADMA_REQUIRE(grid <= 0x7fffffffLL, "grid too large");
      hipLaunchKernelGGL(gemm_bf16_ws_direct, dim3((unsigned)grid), dim3(kComputeThreads + 2 * kDmaWave), 0, s, d_a, d_b, d_c, m, n, k, tile_walk(m, n, k, 256, 128, 1));
      CUDADMA_HIP_CHECK(hipGetLastError());
      return CUDADMA_OK;
#else
      CUDADMA_REQUIRE(false, "gemm variant %d is a sweep kernel: build the library with make EXTRA=-DHIPDMA_SWEEP_VARIANTS", variant);
#endif
    }
  }
}
