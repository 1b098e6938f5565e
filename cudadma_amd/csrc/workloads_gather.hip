// Config 3: indirect gather of 128-byte records with CudaDMAIndirect, 32 records
// per LDS tile.  Shapes follow the warp-specialised kernels of
// src/tests/test_indirect/cudaDMA_test_indirect_v2.cu:52-120, made persistent
// and multi-buffered as src/examples/stencil/warp_specialized_manual_buffer.h:54-71.
// Two consumers:
//   copy   out[i] = table[idx[i]]                       (checks every moved byte)
//   rowsum out[t][j] = sum_r tile[r][j], r ascending     (the reported workload)
#include "dispatch.hpp"
#include "workloads.hpp"

namespace {
using workloads::vec4_t;

constexpr int kRecBytes = 128;
constexpr int kRecFloats = kRecBytes / 4;
constexpr int kRecsPerTile = 32;
constexpr int kTileBytes = kRecBytes * kRecsPerTile;     // 4 KiB
constexpr int kDmaThreads = 128;
constexpr int kComputeThreads = 128;

// TILES tiles in one transfer: 32 B per DMA thread for each, all in one step
template<int TILES>
using dma_of = CudaDMAIndirect<true, true, 16, TILES * kTileBytes / kDmaThreads, kRecBytes, kDmaThreads, TILES * kRecsPerTile>;
typedef dma_of<1> dma_t;

struct CopyConsumer {
  static constexpr bool kWritesEveryRecord = true;
  template<int TILES>
  static __device__ __forceinline__ void run(const char* lds_tile, float* __restrict__ out, const long long tile, const dma_of<TILES>& dma)
  {
    static_assert(TILES == 1 && kTileBytes == 2 * 16 * kComputeThreads, "two vectors per compute thread");
    vec4_t v[2];
    const vec4_t* src = (const vec4_t*)lds_tile;
    v[0] = src[threadIdx.x];
    v[1] = src[threadIdx.x + kComputeThreads];
    dma.start_async_dma();
    // Non-temporal: the records written are not read again, and lines of them would push those of the table out of the L2 (us, plain /
    // non-temporal: 6 Mi records from a table of 24000 248 / 136, 24000 x 512 Ki from DRAM 23 / 15; 8 Mi from one of 4 Mi 367 / 319).
    vec4_t* dst = (vec4_t*)(out + tile * (kTileBytes / 4));
    __builtin_nontemporal_store(v[0], &dst[threadIdx.x]);
    __builtin_nontemporal_store(v[1], &dst[threadIdx.x + kComputeThreads]);
  }
};

struct RowsumConsumer {
  static constexpr bool kWritesEveryRecord = false;
  template<int TILES>
  static __device__ __forceinline__ void run(const char* lds_tiles, float* __restrict__ out, const long long tile, const dma_of<TILES>& dma)
  {
    static_assert(TILES * kRecFloats <= kComputeThreads, "a sum per compute thread");
    // 32 sums per tile: the first 32 compute threads each add one word of every record, record 0 first; the next 32 those of the next tile
    const float* t = (const float*)lds_tiles + threadIdx.x / kRecFloats * (kTileBytes / 4) + threadIdx.x % kRecFloats;
    float acc = 0.0f;
    if (threadIdx.x < TILES * kRecFloats) {
      acc = t[0];
#pragma unroll
      for (int r = 1; r < kRecsPerTile; ++r) acc = acc + t[r * kRecFloats];
    }
    dma.start_async_dma();
    if (threadIdx.x < TILES * kRecFloats) out[tile * kRecFloats + threadIdx.x] = acc;
  }
};

// STAGES objects share the DMA threads; each has its own buffer of TILES tiles.  With PREFETCH the index words of an
// object's next tile are requested right after its current tile (prefetch_index), one turn of the ring before
// they are used: the transfer that uses them then waits only for loads older than they are, and the elements of
// the other STAGES - 1 objects stay in flight across it.  Without it every start_xfer_async fetches its own index
// words and, a wavefront's loads returning in order, waits until nothing of the thread is in flight any more.
template<typename Consumer, int STAGES, bool PREFETCH = false, int TILES = 1>
__global__ void __launch_bounds__(kDmaThreads + kComputeThreads)
gather_manual(const float* __restrict__ table, const int* __restrict__ idx, float* __restrict__ out,
              const long long all_tiles)
{
  typedef dma_of<TILES> dma_t;
  // transfers, the last of them moved back to end with the last tile
  const long long num_tiles = (all_tiles + TILES - 1) / TILES;
  auto tile_of = [&](const long long t) __attribute__((always_inline)) { return TILES == 1 || t * TILES < all_tiles - TILES ? t * TILES : all_tiles - TILES; };
  auto words = [&](const long long t) __attribute__((always_inline)) { return idx + tile_of(t) * kRecsPerTile; };
  __shared__ __attribute__((aligned(16))) char buf[STAGES][TILES * kTileBytes];
  dma_t dma0(0, kComputeThreads, kComputeThreads);
  dma_t dma1(1, kComputeThreads, kComputeThreads);
  dma_t dma2(2, kComputeThreads, kComputeThreads);
  dma_t dma3(3, kComputeThreads, kComputeThreads);
  const long long stride = gridDim.x;
  const long long first = blockIdx.x;
#define HIPDMA_FOR_STAGES(...)                                                    \
  { constexpr int s = 0; dma_t& d = dma0; __VA_ARGS__ }                           \
  if constexpr (STAGES > 1) { constexpr int s = 1; dma_t& d = dma1; __VA_ARGS__ } \
  if constexpr (STAGES > 2) { constexpr int s = 2; dma_t& d = dma2; __VA_ARGS__ } \
  if constexpr (STAGES > 3) { constexpr int s = 3; dma_t& d = dma3; __VA_ARGS__ }
  if (dma0.owns_this_thread()) {
    long long t = first;
    if (t + (2 * STAGES - 1) * stride < num_tiles) {
      // Steady state with no branch around any load, entered from a prologue that has none either:
      // waiting for one stage then leaves the loads of the other stages in flight.
      if constexpr (PREFETCH) {
        // a prefetch beyond the last tile reads the last tile's words instead (never used): no branch
        const long long last = num_tiles - 1;
        HIPDMA_FOR_STAGES({ d.template prefetch_index<true>(words(t + s * stride)); })
        HIPDMA_FOR_STAGES({
          d.template start_xfer_async_prefetched<true, LOAD_CACHE_ALL, STORE_LDS>(words(t + s * stride), table);
          d.template prefetch_index<true>(words(t + (s + STAGES) * stride));
        })
        do {
          HIPDMA_FOR_STAGES({
            d.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buf[s]);
            d.template start_xfer_async_prefetched<true, LOAD_CACHE_ALL, STORE_LDS>(words(t + (s + STAGES) * stride), table);
            const long long ahead = t + (s + 2 * STAGES) * stride;
            d.template prefetch_index<true>(words(ahead < last ? ahead : last));
          })
          t += STAGES * stride;
        } while (t + (2 * STAGES - 1) * stride < num_tiles);
      } else {
        HIPDMA_FOR_STAGES({
          d.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(words(t + s * stride), table);
        })
        do {
          HIPDMA_FOR_STAGES({
            d.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buf[s]);
            d.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(words(t + (s + STAGES) * stride), table);
          })
          t += STAGES * stride;
        } while (t + (2 * STAGES - 1) * stride < num_tiles);
      }
    } else {
      HIPDMA_FOR_STAGES({
        const long long tt = t + s * stride;
        if (tt < num_tiles) d.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(words(tt), table);
      })
    }
    // the last tiles of this workgroup
    for (; t < num_tiles; t += STAGES * stride) {
      HIPDMA_FOR_STAGES({
        const long long tt = t + s * stride;
        if (tt < num_tiles) {
          d.template wait_xfer_finish<true, LOAD_CACHE_ALL, STORE_LDS>(buf[s]);
          const long long nx = tt + STAGES * stride;
          if (nx < num_tiles) d.template start_xfer_async<true, LOAD_CACHE_ALL, STORE_LDS>(words(nx), table);
        }
      })
    }
  } else {
    HIPDMA_FOR_STAGES({ d.start_async_dma(); })
    for (long long t = first; t < num_tiles; t += STAGES * stride) {
      HIPDMA_FOR_STAGES({
        const long long tt = t + s * stride;
        if (tt < num_tiles) {
          d.wait_for_dma_finish();
          Consumer::template run<TILES>(buf[s], out, tile_of(tt), d);
        }
      })
    }
  }
#undef HIPDMA_FOR_STAGES
}

template<typename Consumer>
__global__ void __launch_bounds__(kDmaThreads + kComputeThreads)
gather_single(const float* __restrict__ table, const int* __restrict__ idx, float* __restrict__ out,
              const long long num_tiles)
{
  __shared__ __attribute__((aligned(16))) char buf[kTileBytes];
  dma_t dma(0, kComputeThreads, kComputeThreads);
  if (dma.owns_this_thread()) {
    for (long long t = blockIdx.x; t < num_tiles; t += gridDim.x)
      dma.template execute_dma<true, LOAD_CACHE_ALL, STORE_LDS>(idx + t * kRecsPerTile, table, buf);
  } else {
    dma.start_async_dma();
    for (long long t = blockIdx.x; t < num_tiles; t += gridDim.x) {
      dma.wait_for_dma_finish();
      Consumer::template run<1>(buf, out, t, dma);
    }
  }
}

template<typename Consumer>
int launch_gather(const float* d_table, const int32_t* d_idx, float* d_out, size_t n_records, size_t n_idx,
                  int variant, void* stream)
{
  CUDADMA_REQUIRE((n_idx % kRecsPerTile) == 0, "n_idx (%zu) must be a multiple of %d", n_idx, kRecsPerTile);
  CUDADMA_REQUIRE(n_records > 0 && n_records <= 0x7fffffffull, "the table (%zu records) is indexed with int record numbers", n_records);
  if (variant < 0 || variant >= cudadma_num_variants(CUDADMA_WORKLOAD_GATHER)) {
    cudadma_host::set_error("gather has no variant %d", variant);
    return CUDADMA_ERANGE;
  }
  if (n_idx == 0) return CUDADMA_OK;
  CUDADMA_REQUIRE(d_table != nullptr && d_idx != nullptr && d_out != nullptr, "NULL pointer");
  CUDADMA_REQUIRE(cudadma_host::aligned_to(d_table, 16) && cudadma_host::aligned_to(d_out, 16), "pointers must be 16-byte aligned");
  const long long tiles = (long long)(n_idx / kRecsPerTile);
  hipStream_t s = (hipStream_t)stream;
  const dim3 block(kDmaThreads + kComputeThreads);
  // Workgroups per compute unit of the numbered variants.  Objects that fetch their own index words drain the DMA wavefronts at every
  // transfer and need many workgroups to cover that (six with several objects, eight with one).  With the index
  // words requested ahead two objects and three workgroups are enough (0.634 ms on the configuration's 512 MiB
  // table, which the caches help to serve); a table several times the Infinity Cache wants four (0.724 ms against
  // 0.775 ms without the prefetch on 1.875 GiB).
  // The copy consumer writes as much as it reads and wants a shorter queue still: two (74.6 % on the 512 MiB table,
  // 69.5 % on 1.875 GiB, against 74.0 / 68.2 with three).
  const int ahead_wgs = Consumer::kWritesEveryRecord ? 2 : n_records * (size_t)kRecBytes <= (1ull << 30) ? 3 : 4;
  auto grid = [&](const int per_cu, const long long n) { return dim3((unsigned)workloads::persistent_grid(n, per_cu)); };
  if constexpr (Consumer::kWritesEveryRecord) {
    // The library's choice: a short list is over before two workgroups per compute unit with two tiles each have filled their queues; eight
    // with one tile start sooner (copies of 32 Ki records from the caches 3.6 us against 4.0).
    if (variant == 0) variant = n_idx * (size_t)kRecBytes <= (32ull << 20) ? 1 : 6;
  } else if (variant == 0) {
    // The library's choice: short lists as above.  Longer ones take four tiles in one transfer, whose sums occupy all compute threads (with one
    // tile in turn a quarter of one of the two wavefronts adds while the DMA wavefronts wait for the buffer): 16 KiB in flight per
    // workgroup instead of 8, a quarter of the hand-offs.  It counts where an L2 holds the table (us, variant 6 / this: 6 Mi indices of 24000
    // records 104 / 51, of 60000 106 / 66, 1 Mi of 24000 21 / 13); elsewhere what is in flight does.
    // Between 64 and 112 Ki indices the short form is 0.3 us ahead from the caches, beyond
    // the long one (2 Mi records, 176 Ki indices 4.6 / 4.6 and from DRAM 7.8 / 7.4; 24000, 256 Ki 5.2 / 4.6 and 6.3 / 6.0).
    if (n_idx <= (112u << 10)) variant = 1;
    else {
      const int wgs = dispatch::rowsum_workgroups(n_records * (unsigned long long)kRecBytes, n_idx);
      hipLaunchKernelGGL((gather_manual<Consumer, 1, true, 4>), grid(wgs, (tiles + 3) / 4), block, 0, s, d_table, d_idx, d_out, tiles);
      CUDADMA_HIP_CHECK(hipGetLastError());
      return CUDADMA_OK;
    }
  }
  switch (variant) {
    case 6: hipLaunchKernelGGL((gather_manual<Consumer, 2, true>), grid(ahead_wgs, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
    case 1: hipLaunchKernelGGL(gather_single<Consumer>, grid(8, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
    case 2: hipLaunchKernelGGL((gather_manual<Consumer, 2>), grid(6, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
    case 3: hipLaunchKernelGGL((gather_manual<Consumer, 4>), grid(6, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
    case 4: hipLaunchKernelGGL((gather_manual<Consumer, 4, true>), grid(ahead_wgs, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
    default: hipLaunchKernelGGL((gather_manual<Consumer, 3, true>), grid(ahead_wgs, tiles), block, 0, s, d_table, d_idx, d_out, tiles); break;
  }
  CUDADMA_HIP_CHECK(hipGetLastError());
  return CUDADMA_OK;
}

}  // namespace

extern "C" int cudadma_gather_copy(const float* d_table, const int32_t* d_idx, float* d_out, size_t n_records,
                                   size_t n_idx, int variant, void* stream)
{ return launch_gather<CopyConsumer>(d_table, d_idx, d_out, n_records, n_idx, variant, stream); }

extern "C" int cudadma_gather_rowsum(const float* d_table, const int32_t* d_idx, float* d_out, size_t n_records,
                                     size_t n_idx, int variant, void* stream)
{ return launch_gather<RowsumConsumer>(d_table, d_idx, d_out, n_records, n_idx, variant, stream); }
