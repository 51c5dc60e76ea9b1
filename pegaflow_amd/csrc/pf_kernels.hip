// pf_kernels.hip — gfx950 gather/scatter kernels of the KV-block transfer
// path, plus the synthetic-data, verification and spin kernels used by the
// benchmark and the parity tests.
//
// The transfer is pure data movement (no contraction, so no MFMA).  A launch
// moves `n_chunks` chunks of `chunk_bytes` each, described by (src, dst)
// address pairs in device memory.  Addresses may be HBM (the paged layer
// tensor, a staging buffer) or host-mapped pinned memory (zero-copy over the
// host link).  The same kernel therefore serves:
//   * save:    paged layer tensor -> pinned host (or HBM staging), a gather;
//   * restore: pinned host (or HBM staging) -> paged layer tensor, a scatter.
//
// Work decomposition: copies between device buffers split a chunk into units
// of 64 * UNROLL 16-byte elements, one wave each; copies over the host link
// into tiles of blockDim.x * UNROLL elements, one workgroup each.  Every lane
// issues UNROLL independent 16-byte loads (global_load_dwordx4) before its
// UNROLL stores, so each wave keeps UNROLL * 1 KiB in flight — enough to cover
// HBM latency and, for zero-copy, the much longer host-link read latency.  Consecutive
// lanes touch consecutive 16-byte words, so every wave instruction covers one
// contiguous 1 KiB span (fully coalesced).  No LDS: source and destination
// share the same byte order within a chunk.
#include <hip/hip_runtime.h>

#include "pf_common.h"

namespace pf {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
// Global-address-space views: the addresses arrive as integers, and without
// the address space the compiler would emit generic (flat) accesses.
typedef __attribute__((address_space(1))) u32x4 g_u32x4;
typedef u32x4 u32x4_any __attribute__((aligned(1)));  // at any address
typedef __attribute__((address_space(1))) u32x4_any g_u32x4_any;
typedef __attribute__((address_space(1))) uint8_t g_u8;
typedef __attribute__((address_space(1))) uint64_t g_u64;

template <bool NT>
__device__ __forceinline__ u32x4 load16(const g_u32x4* p) {
  if constexpr (NT)
    return __builtin_nontemporal_load(p);
  else
    return *p;
}

template <bool NT>
__device__ __forceinline__ void store16(g_u32x4* p, u32x4 v) {
  if constexpr (NT)
    __builtin_nontemporal_store(v, p);
  else
    *p = v;
}

// NTL / NTS select non-temporal (streaming) loads / stores: every byte is
// touched exactly once, so there is nothing to gain from keeping it in L2 or
// the MALL, and streaming accesses leave those caches to other traffic.
// Workgroup -> tile order.  Workgroups are dealt round-robin to the 8 XCDs
// (workgroup b runs on XCD b % 8).  With xcd_major set (and one workgroup
// per tile), XCD x instead takes one contiguous range of tiles:
//   n = 8q + r tiles; XCD x owns q + (x < r) tiles starting at x*q + min(x, r);
//   workgroup b = 8i + x handles the i-th of them.
// The workgroups with b % 8 == x number exactly q + (x < r), so this is a
// bijection of [0, n).
__device__ __forceinline__ uint32_t tile_of(uint32_t b, uint32_t n, bool xcd_major) {
  if (!xcd_major) return b;
  const uint32_t x = b & 7u, i = b >> 3, q = n >> 3, r = n & 7u;
  return x * q + (x < r ? x : r) + i;
}

// ---------------------------------------------------------------------------
// Layer completion marks.  A load that covers several layers in one launch
// can still report each layer as soon as its bytes are in place: every
// workgroup, after its stores, bumps its layer's tile counter, and the
// workgroup that brings the counter to the layer's tile count writes the
// call's value into word[layer] of each signal target (host-mapped pinned
// memory, device memory, or another process's IPC-mapped device memory).
//
// Visibility.  Each XCD has its own L2, so a byte stored by one workgroup is
// visible to readers on other XCDs only once it has left that L2.  A
// release fence at agent scope per workgroup would write the whole L2 back
// every time (measured: 2.2x slower from pinned memory, 40x from HBM).
// Instead the marking kernels store their bytes through the L2 to the device's
// coherence point (store16_through: the sc1 policy that agent-scope stores
// have) and wait for every store's acknowledgement (s_waitcnt 0) before the
// workgroup barrier; only then does one lane bump the counter (an agent-scope
// atomic).  The lane whose add completes the layer therefore knows that every
// byte of it has reached the coherence point: it puts the counter back to 0
// (ready for the next launch on the stream) and writes the marks, at system
// scope for host memory, with nothing left to flush or to read again.  A
// release would write back the L2 of its own XCD, which holds none of the
// layer's bytes, under every other workgroup's copy: with a release and an
// acquire per layer, 61 layers of 4.7 MB took 120 us, without 94, and 32 of
// 5.2 MB 66 and 54 (unmarked 93 and 53).  A reader that sees word[layer] ==
// value and then acquires, or starts a kernel afterwards, sees every byte of
// that layer.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void layer_done(const SignalTargets& t, uint32_t* counter,
                                           uint32_t layer) {
  // Orders the compiler and this wave's accesses; touches no cache.
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (uint32_t i = 0; i < t.count; ++i) {
    uint64_t* w = reinterpret_cast<uint64_t*>(t.words[i]) + layer;
    if ((t.host_mask >> i) & 1u)
      __hip_atomic_store(w, t.value[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    else
      __hip_atomic_store(w, t.value[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// The marks of layers that earlier kernels or copies put in place.
__device__ __forceinline__ void write_marks(const SignalTargets& t, uint32_t layer) {
  for (uint32_t i = 0; i < t.count; ++i) {
    uint64_t* w = reinterpret_cast<uint64_t*>(t.words[i]) + layer;
    if ((t.host_mask >> i) & 1u)
      __hip_atomic_store(w, t.value[i], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    else
      __hip_atomic_store(w, t.value[i], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Called by one lane per workgroup once the workgroup's stores of chunk c are
// acknowledged.  start[0..n] are the launch-relative first chunks of its
// layers (increasing, start[0] == 0 <= c < start[n]; m's own table or a copy
// of it in LDS, as layer[]); the search keeps start[lo] <= c < start[hi].
template <class Table>
__device__ __forceinline__ void tile_done(const LayerMarks& m, Table start, Table layers,
                                          uint32_t c, uint32_t tiles_per_chunk) {
  uint32_t lo = 0, hi = m.n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (start[mid] <= c) lo = mid;
    else hi = mid;
  }
  const uint32_t layer = layers[lo];
  const uint32_t tiles = (start[lo + 1] - start[lo]) * tiles_per_chunk;
  uint32_t* cnt = m.counters + layer * kCounterStride;
  const uint32_t prev = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
  if (prev + 1 == tiles) {
    layer_done(m.targets, cnt, layer);
  }
}

// The layer that workgroup `wg` of a marked copy belongs to: its first
// workgroup and chunk, its chunks in this launch, its units over all launches
// (0: not counted) and its index in the call.
struct MarkGroup {
  uint32_t wg_start, chunk_start, chunks, units, layer;
};

// wg < wg_start[n]; the search keeps wg_start[lo] <= wg < wg_start[hi].
__device__ __forceinline__ MarkGroup mark_group(const MarkTable& m, uint32_t wg,
                                                uint32_t units_per_chunk) {
  uint32_t lo = 0, hi = m.n;
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (m.wg_start[mid] <= wg) lo = mid;
    else hi = mid;
  }
  const uint32_t chunks = m.chunk_start[lo + 1] - m.chunk_start[lo];
  return {m.wg_start[lo], m.chunk_start[lo], chunks, chunks * units_per_chunk, m.layer[lo]};
}

// The table lives in the kernel's arguments: read with constant indices only,
// so it stays in scalar registers.
__device__ __forceinline__ MarkGroup mark_group(const SliceMarks& m, uint32_t wg, uint32_t) {
  MarkGroup g{m.wg_start[0], m.chunk_start[0], m.chunk_start[1] - m.chunk_start[0], m.units[0],
              m.layer[0]};
#pragma unroll
  for (uint32_t i = 1; i < kSliceMarkLayers; ++i)
    if (i < m.n && m.wg_start[i] <= wg)
      g = {m.wg_start[i], m.chunk_start[i], m.chunk_start[i + 1] - m.chunk_start[i], m.units[i],
           m.layer[i]};
  return g;
}

// A value that every lane of the wave holds, in scalar registers.
__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

// 16 bytes at base + 16 * lane, written through the XCD's L2 to the device's
// coherence point (the sc1 policy of an agent-scope store, which the language
// offers for at most 8 bytes at a time).  `base` is the same for the whole
// wave; `bytes` bounds the store: lanes past it write nothing.
__device__ __forceinline__ void store16_through(uint64_t base, uint32_t bytes, uint32_t lane,
                                                u32x4 v) {
  constexpr int kSc1 = 16;
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
      reinterpret_cast<void*>(base), 0, static_cast<int>(bytes), 0x00027000);
  __builtin_amdgcn_raw_buffer_store_b128(v, r, static_cast<int>(lane * 16), 0, kSc1);
}

// Unit u of a chunk whose addresses or size are not 16-byte aligned.  A chunk's
// stores are 16-byte words at aligned addresses, its loads the 16 bytes that go
// there, at whatever address they have; up to 15 bytes in front of the first
// word go with the chunk's first unit and those behind the last word with its
// last (THROUGH: written through the L2, as the words are).
template <bool THROUGH>
__device__ __forceinline__ void copy_unaligned_unit(const ChunkDesc& d, uint32_t u,
                                                    uint32_t units_per_chunk, uint64_t chunk_bytes,
                                                    uint32_t lane) {
  const uint64_t to_word = (16u - (d.dst & 15u)) & 15u;
  const uint64_t head = to_word < chunk_bytes ? to_word : chunk_bytes;
  const uint64_t words = (chunk_bytes - head) >> 4;  // <= 64 * units_per_chunk
  const uint32_t tail = static_cast<uint32_t>(chunk_bytes - head) & 15u;
  const uint64_t src = d.src + head, dst = d.dst + head;
  const uint64_t e0 = static_cast<uint64_t>(u) * 64u;
  auto byte = [&](uint64_t to, uint64_t from) {
    const uint8_t v = *reinterpret_cast<const g_u8*>(from);
    if constexpr (THROUGH)
      __hip_atomic_store(reinterpret_cast<g_u8*>(to), v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    else
      *reinterpret_cast<g_u8*>(to) = v;
  };
  if (e0 + lane < words)
    store16_through(dst + e0 * 16u, 1024u, lane,
                    __builtin_nontemporal_load(reinterpret_cast<const g_u32x4_any*>(src) + e0 +
                                               lane));
  if (u == 0 && lane < head) byte(d.dst + lane, d.src + lane);
  if (u == units_per_chunk - 1 && lane < tail)
    byte(dst + words * 16u + lane, src + words * 16u + lane);
}

// A marked copy between device buffers: the device-sourced marked load (one
// launch over its layers, table in device memory) and the staged load's
// scatter of a slice whose layers it reports itself (table in the arguments).
//
// Bound by HBM and by the reports.  A unit is 64 lanes x UNROLL words of one
// chunk and belongs to one wave, so a chunk of any size wastes at most part of
// its last unit.  Workgroup w copies the consecutive units of one layer that
// its index gives it (see marked_shape) and then adds their number to the layer's
// counter, once: adds to one counter run one after another (about 20 ns).
// Workgroups start in index order, so the layers land in order.
//
// Visibility: as in the marking protocol above, with 16-byte write-through
// stores.  They run at the rate of ordinary ones (288 MB of 36 KiB chunks 93
// us, ordinary 97, non-temporal 105-115), so no L2 has to be written back
// before a report.  The per-workgroup release fence that this replaces allowed
// only 128 workgroups.  61 layers of 4.7 MB, one launch and one marking kernel
// each before, took 450 us, here 94 in one launch; a single 40 MiB layer (a staged
// slice, under the next slice's copy) takes 21.8, with the fences 24.0.
//
// Chunks that are not aligned (ALIGNED false) go by units of 64 words, their odd
// bytes written through as well: 61 layers of 4.7 MB in 36,865-byte chunks land
// one by one in 163 us a call (one unmarked launch, every layer marked behind it,
// 155; a byte-wise launch a layer 2,123).
template <int UNROLL, bool ALIGNED, class Marks>
__global__ void __launch_bounds__(kMarkedThreads)
copy_chunks_marked_kernel(const ChunkDesc* __restrict__ descs, MarkedShape shape,
                          uint64_t chunk_bytes, uint32_t n_wg, Marks marks) {
  const uint32_t chunk16 = static_cast<uint32_t>(chunk_bytes / 16);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  constexpr uint32_t kWaves = kMarkedThreads / 64;
  for (uint32_t wg = blockIdx.x; wg < n_wg; wg += gridDim.x) {
    const MarkGroup g = mark_group(marks, wg, shape.units_per_chunk);
    const uint32_t group_units = g.chunks * shape.units_per_chunk;
    const uint32_t first = (wg - g.wg_start) * shape.wg_units;
    const uint32_t left = group_units - first;
    const uint32_t mine = left < shape.wg_units ? left : shape.wg_units;
    for (uint32_t i = wave; i < mine; i += kWaves) {
      const uint32_t unit = first + i;
      const uint32_t c = unit / shape.units_per_chunk;
      const uint32_t in_chunk = unit - c * shape.units_per_chunk;
      const ChunkDesc d = descs[g.chunk_start + c];
      if constexpr (!ALIGNED) {
        copy_unaligned_unit<true>(d, in_chunk, shape.units_per_chunk, chunk_bytes, lane);
      } else {
        const uint32_t e0 = in_chunk * (64u * UNROLL);
        const g_u32x4* __restrict__ src = reinterpret_cast<const g_u32x4*>(d.src) + e0;
        const uint32_t words = chunk16 - e0;  // of this unit and what follows it
        u32x4 v[UNROLL];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
          if (u * 64u + lane < words) v[u] = load16<true>(src + u * 64u + lane);
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
          if (u * 64u >= words) break;
          const uint32_t n = words - u * 64u;
          store16_through(d.dst + (static_cast<uint64_t>(e0) + u * 64u) * 16u,
                          (n < 64u ? n : 64u) * 16u, lane, v[u]);
        }
      }
    }
    if (g.units == 0) continue;  // marked by another kernel (uniform: no barrier is missed)
    __builtin_amdgcn_s_waitcnt(0);  // every store of this wave acknowledged
    __syncthreads();
    if (threadIdx.x == 0) {
      uint32_t* cnt = marks.counters + g.layer * kCounterStride;
      const uint32_t prev = __hip_atomic_fetch_add(cnt, mine, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
      if (prev + mine == g.units) layer_done(marks.targets, cnt, g.layer);
    }
  }
}

// The fixed-map copy: between device buffers, and the descriptor uploads.
//
// Bound by HBM.  A unit is 64 lanes x UNROLL words of one chunk and belongs to
// one wave: wave w of the launch copies unit w, so chunks of any size keep
// every lane busy but for part of a chunk's last unit.  (A workgroup per tile
// of 512 threads left lanes idle on every chunk that 8 KiB do not divide:
// 1.34 GB of 10 KiB chunks gathered at 5.1 TB/s, with units 6.1; 168 MB of 2
// KiB chunks 5.1 and 5.8.)  Workgroups have at most 4 waves: with 8 the 32 KiB
// chunks of the Llama prefix gather at 5.95 TB/s and scatter at 5.44, with 4
// at 6.10 and 5.61.  Streaming stores (THROUGH) are written through the L2 and
// may stay in the memory-side cache: non-temporal ones, which bypass it, were
// as fast on 1.34 GB and 11-25% slower on 67-288 MB.
constexpr uint32_t kFixedThreads = 256;

template <int UNROLL, bool NTL, bool THROUGH>
__global__ void __launch_bounds__(kFixedThreads)
copy_chunks_v16_kernel(const ChunkDesc* __restrict__ descs, uint32_t units_per_chunk,
                       uint32_t n_units, uint32_t chunk16, uint32_t xcd_major) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t waves = blockDim.x >> 6;
  const uint32_t n_wg = (n_units + waves - 1) / waves;
  const bool remap = xcd_major && gridDim.x == n_wg;
  for (uint32_t b = blockIdx.x; b < n_wg; b += gridDim.x) {
    const uint32_t unit = __builtin_amdgcn_readfirstlane(tile_of(b, n_wg, remap) * waves +
                                                         (threadIdx.x >> 6));
    if (unit >= n_units) continue;
    const uint32_t c = unit / units_per_chunk;
    const uint32_t e0 = (unit - c * units_per_chunk) * (64u * UNROLL);
    const ChunkDesc d = descs[c];
    const g_u32x4* __restrict__ src = reinterpret_cast<const g_u32x4*>(d.src) + e0;
    g_u32x4* __restrict__ dst = reinterpret_cast<g_u32x4*>(d.dst) + e0;
    const uint32_t words = chunk16 - e0;  // of this unit and what follows it
    u32x4 v[UNROLL];
    if (words >= 64u * UNROLL) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) v[u] = load16<NTL>(src + u * 64u + lane);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        if constexpr (THROUGH)
          store16_through(d.dst + (static_cast<uint64_t>(e0) + u * 64u) * 16u, 1024u, lane, v[u]);
        else
          dst[u * 64u + lane] = v[u];
      }
    } else {
      // Partial last unit of a chunk: guarded per word.
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
        if (u * 64u + lane < words) v[u] = load16<NTL>(src + u * 64u + lane);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u)
        if (u * 64u + lane < words) {
          if constexpr (THROUGH)
            store16_through(d.dst + (static_cast<uint64_t>(e0) + u * 64u) * 16u, 1024u, lane,
                            v[u]);
          else
            dst[u * 64u + lane] = v[u];
        }
    }
  }
}

// Copies over the host link take their tiles from a work queue instead of a
// fixed workgroup -> tile map.  Workgroups are dealt to the 8 XCDs
// statically, and when the copy reads or writes host memory the XCDs
// progress at very different rates (the link is not shared fairly between
// them): with a fixed map the copy ends when the slowest XCD does, and a
// marked load's layers land only when the slowest XCD gets to them
// (measured: the first of 32 Llama layers after half the load).  Here a
// small persistent grid pulls tile indices from one counter, so the fast
// XCDs take more tiles and tiles, hence layers, finish in order; with few
// requests in flight the link also runs closer to its peak (Llama restore
// 24.1 -> 23.3 ms of kernel time with 64 workgroups).
//
// The queue is two words, queue[0] the next tile and queue[1] the
// workgroups that have left, both 0 when a launch starts.  A workgroup
// leaves after a pull past the last tile, and counts itself out with an
// acquire-release add; the last one out has seen every workgroup's final
// pull, so it puts both words back to 0.  The launch therefore leaves the
// queue as it found it, whatever the host knows of earlier launches: a
// replayed graph or a launch on another stream after this one finds 0.
// Launches that run at the same time need queues of their own.
//
// A small call's descriptors lie in pinned host memory: reading one in front of
// each tile put a host-link round trip there, 2 us idle and as long as the
// posted writes ahead of it take in a save.  With TABLE each workgroup takes all
// of them (at most kQueueTableMax, and the layers' table of a marking launch)
// into LDS first: 64 chunks of 32 KiB load in 73 -> 62 us and save in 71 -> 64,
// 320 load in 225 -> 208 and save in 251 -> 227 (call and wait; the link takes
// 36.6 and 183, an empty kernel and its wait 9.5).
// Fetching the next tile and its descriptor during the copy of this one, by a
// wave of its own, made large copies 1-8% slower: the link runs best with few
// requests.
//
// MARK adds the per-layer completion marks, with write-through stores (see
// layer_done).
template <int UNROLL, bool NTL, bool NTS, bool MARK, bool TABLE>
__global__ void __launch_bounds__(1024)
copy_chunks_queue_kernel(const ChunkDesc* __restrict__ descs, uint32_t n_chunks,
                         uint32_t tiles_per_chunk, uint32_t n_tiles, uint32_t chunk16,
                         LayerMarks marks, uint32_t* queue) {
  __shared__ uint32_t s_tile;
  __shared__ ChunkDesc s_desc[TABLE ? kQueueTableMax : 1];
  __shared__ uint32_t s_start[TABLE && MARK ? kQueueTableMax + 1 : 1];
  __shared__ uint32_t s_layer[TABLE && MARK ? kQueueTableMax : 1];
  const uint32_t stride = blockDim.x;
  const uint32_t tile_elems = stride * UNROLL;
  const uint32_t lane = threadIdx.x & 63u;
  if constexpr (TABLE) {
    // Read by every lane after the next barrier.
    for (uint32_t i = threadIdx.x; i < n_chunks; i += stride) s_desc[i] = descs[i];
    if constexpr (MARK) {
      for (uint32_t i = threadIdx.x; i <= marks.n; i += stride) s_start[i] = marks.chunk_start[i];
      for (uint32_t i = threadIdx.x; i < marks.n; i += stride) s_layer[i] = marks.layer[i];
    }
  }
  for (;;) {
    if (threadIdx.x == 0)
      s_tile = __hip_atomic_fetch_add(queue, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const uint32_t t = s_tile;
    __syncthreads();  // every lane has read s_tile before it is written again
    if (t >= n_tiles) {  // uniform: the queue is empty for every later pull too
      if (threadIdx.x == 0) {
        const uint32_t out = __hip_atomic_fetch_add(queue + 1, 1u, __ATOMIC_ACQ_REL,
                                                    __HIP_MEMORY_SCOPE_AGENT);
        if (out + 1 == gridDim.x) {
          __hip_atomic_store(queue, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(queue + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      break;
    }
    const uint32_t c = t / tiles_per_chunk;
    const uint32_t tile = t - c * tiles_per_chunk;
    const ChunkDesc d = TABLE ? s_desc[c] : descs[c];
    const g_u32x4* __restrict__ src = reinterpret_cast<const g_u32x4*>(d.src);
    g_u32x4* __restrict__ dst = reinterpret_cast<g_u32x4*>(d.dst);
    const uint32_t tile_base = tile * tile_elems;
    const uint32_t base_e = tile_base + threadIdx.x;
    auto put = [&](uint32_t e, u32x4 v) {  // word e, of this lane
      if constexpr (MARK)
        store16_through(uniform64(d.dst) +
                            static_cast<uint64_t>(__builtin_amdgcn_readfirstlane(e - lane)) * 16u,
                        1024u, lane, v);
      else
        store16<NTS>(dst + e, v);
    };
    u32x4 v[UNROLL];
    if (tile_base + tile_elems <= chunk16) {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) v[u] = load16<NTL>(src + base_e + u * stride);
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) put(base_e + u * stride, v[u]);
    } else {
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint32_t e = base_e + u * stride;
        if (e < chunk16) v[u] = load16<NTL>(src + e);
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const uint32_t e = base_e + u * stride;
        if (e < chunk16) put(e, v[u]);
      }
    }
    if constexpr (MARK) {
      __builtin_amdgcn_s_waitcnt(0);  // every store of this wave acknowledged
      __syncthreads();
      if (threadIdx.x == 0) {
        if constexpr (TABLE)
          tile_done(marks, s_start, s_layer, c, tiles_per_chunk);
        else
          tile_done(marks, marks.chunk_start, marks.layer, c, tiles_per_chunk);
      }
    }
  }
}

// Marks the listed layers (layers with nothing to copy, and layers copied by
// DMA earlier on the same stream).
__global__ void mark_layers_kernel(LayerList list, SignalTargets t) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < list.n) write_marks(t, list.ids[i]);
}

// Bounded device-side wait: lane 0 polls *word until it reaches `value` or
// `max_ticks` of the device wall clock have passed, so the wave always ends.
// On a timeout *timed_out (if given) is set to 1.
__global__ void wait_word_kernel(const uint64_t* word, uint64_t value, uint64_t max_ticks,
                                 uint32_t* timed_out) {
  if (threadIdx.x != 0) return;
  const uint64_t start = static_cast<uint64_t>(wall_clock64());
  while (__hip_atomic_load(word, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM) < value) {
    if (static_cast<uint64_t>(wall_clock64()) - start >= max_ticks) {
      if (timed_out)
        __hip_atomic_store(timed_out, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
    __builtin_amdgcn_s_sleep(2);
  }
}

// Chunks whose addresses or size are not 16-byte aligned, over the host link: a
// byte per lane.  The link is the bound: 59 MB in 12,300-byte chunks load in
// 1,095-1,186 us and save in 1,100, where the link takes 1,032 (by 16-byte words,
// as below, 1,072 and 1,108-1,145).
__global__ void __launch_bounds__(1024)
copy_chunks_b1_kernel(const ChunkDesc* __restrict__ descs, uint32_t n_chunks,
                      uint64_t chunk_bytes) {
  for (uint32_t c = blockIdx.x; c < n_chunks; c += gridDim.x) {
    const ChunkDesc d = descs[c];
    const g_u8* __restrict__ src = reinterpret_cast<const g_u8*>(d.src);
    g_u8* __restrict__ dst = reinterpret_cast<g_u8*>(d.dst);
    for (uint64_t i = threadIdx.x; i < chunk_bytes; i += blockDim.x) dst[i] = src[i];
  }
}

// The same between device buffers, by units as in the fixed map.  Bound by HBM:
// 59 MB in 12,300-byte chunks take 27 us, byte by byte 61; 200-byte chunks 66 and
// 115.  (Aligned loads shifted between the lanes were no faster.)
__global__ void __launch_bounds__(kFixedThreads)
copy_chunks_unaligned_kernel(const ChunkDesc* __restrict__ descs, uint32_t units_per_chunk,
                             uint32_t n_units, uint64_t chunk_bytes) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t waves = blockDim.x >> 6;
  const uint32_t n_wg = (n_units + waves - 1) / waves;
  for (uint32_t b = blockIdx.x; b < n_wg; b += gridDim.x) {
    const uint32_t unit =
        __builtin_amdgcn_readfirstlane(b * waves + (threadIdx.x >> 6));
    if (unit >= n_units) continue;
    const uint32_t c = unit / units_per_chunk;
    copy_unaligned_unit<false>(descs[c], unit - c * units_per_chunk, units_per_chunk, chunk_bytes,
                               lane);
  }
}

// Upper bound on workgroups per launch; larger tile counts loop.
static constexpr uint32_t kMaxGrid = 1u << 20;

template <int UNROLL, bool NTL, bool THROUGH>
static void launch_v16_nt(dim3 grid, dim3 block, hipStream_t stream, const ChunkDesc* d,
                          uint32_t upc, uint32_t n_units, uint32_t c16, uint32_t xcd) {
  hipLaunchKernelGGL((copy_chunks_v16_kernel<UNROLL, NTL, THROUGH>), grid, block, 0, stream, d,
                     upc, n_units, c16, xcd);
}

template <int UNROLL>
static hipError_t launch_v16(const ChunkDesc* d_descs, uint32_t units_per_chunk,
                             uint32_t n_units, uint32_t chunk16, uint32_t threads,
                             uint32_t flags, uint32_t max_grid, hipStream_t stream) {
  const uint32_t cap = max_grid ? max_grid : kMaxGrid;
  const uint32_t waves = threads / 64;
  const uint32_t n_wg = (n_units + waves - 1) / waves;
  const dim3 grid(n_wg < cap ? n_wg : cap), block(threads);
  const uint32_t xcd = (flags & PF_KERNEL_XCD_MAJOR) ? 1u : 0u;
  switch (flags & PF_KERNEL_NONTEMPORAL) {
    case 0:
      launch_v16_nt<UNROLL, false, false>(grid, block, stream, d_descs, units_per_chunk, n_units,
                                          chunk16, xcd);
      break;
    case PF_KERNEL_NT_LOADS:
      launch_v16_nt<UNROLL, true, false>(grid, block, stream, d_descs, units_per_chunk, n_units,
                                         chunk16, xcd);
      break;
    case PF_KERNEL_NT_STORES:
      launch_v16_nt<UNROLL, false, true>(grid, block, stream, d_descs, units_per_chunk, n_units,
                                         chunk16, xcd);
      break;
    default:
      launch_v16_nt<UNROLL, true, true>(grid, block, stream, d_descs, units_per_chunk, n_units,
                                        chunk16, xcd);
      break;
  }
  return hipGetLastError();
}

// One queued launch.
struct QueueLaunch {
  dim3 grid, block;
  hipStream_t stream;
  const ChunkDesc* descs;
  uint32_t n_chunks, tiles_per_chunk, n_tiles, chunk16;
  const LayerMarks* marks;
  uint32_t* queue;
  bool table;
};

template <int UNROLL, bool NTL, bool NTS, bool MARK, bool TABLE>
static void launch_queue_as(const QueueLaunch& q) {
  hipLaunchKernelGGL((copy_chunks_queue_kernel<UNROLL, NTL, NTS, MARK, TABLE>), q.grid, q.block,
                     0, q.stream, q.descs, q.n_chunks, q.tiles_per_chunk, q.n_tiles, q.chunk16,
                     q.marks ? *q.marks : LayerMarks{}, q.queue);
}

// A marking launch's stores are written through, whatever the flags.
template <int UNROLL, bool NTL, bool NTS>
static void launch_queue_nt(const QueueLaunch& q) {
  if (q.marks && !q.table) launch_queue_as<UNROLL, NTL, false, true, false>(q);
  else if (q.marks) launch_queue_as<UNROLL, NTL, false, true, true>(q);
  else if (!q.table) launch_queue_as<UNROLL, NTL, NTS, false, false>(q);
  else launch_queue_as<UNROLL, NTL, NTS, false, true>(q);
}

template <int UNROLL>
static void launch_queue(const QueueLaunch& q, uint32_t flags) {
  switch (flags & PF_KERNEL_NONTEMPORAL) {
    case 0: launch_queue_nt<UNROLL, false, false>(q); break;
    case PF_KERNEL_NT_LOADS: launch_queue_nt<UNROLL, true, false>(q); break;
    case PF_KERNEL_NT_STORES: launch_queue_nt<UNROLL, false, true>(q); break;
    default: launch_queue_nt<UNROLL, true, true>(q); break;
  }
}

// Tiles of a launch: every tile index < n_tiles maps to chunk < n_chunks and
// element offsets < tiles_per_chunk * tile_elems; elements >= chunk16 are
// masked, and the full-tile path is taken only when the whole tile lies
// below chunk16.  chunk16 < 2^31 and tile_elems <= 16384 keep
// tile_base + tile_elems in 32 bits.
static bool tile_geometry(uint32_t n_chunks, uint64_t chunk_bytes, uint32_t threads,
                          uint32_t unroll, uint32_t* tpc, uint32_t* n_tiles, uint32_t* c16) {
  const uint64_t chunk16 = chunk_bytes / 16;
  if (chunk16 >= (1ull << 31)) return false;
  const uint64_t tile_elems = static_cast<uint64_t>(threads) * unroll;
  if (tile_elems == 0) return false;
  const uint64_t tiles_per_chunk = (chunk16 + tile_elems - 1) / tile_elems;
  const uint64_t tiles = tiles_per_chunk * n_chunks;
  if (tiles > 0xffffffffull) return false;
  *tpc = static_cast<uint32_t>(tiles_per_chunk);
  *n_tiles = static_cast<uint32_t>(tiles);
  *c16 = static_cast<uint32_t>(chunk16);
  return true;
}

// `unroll` carries the loads in flight per lane (low byte) and the
// PF_KERNEL_NT_LOADS / PF_KERNEL_NT_STORES / PF_KERNEL_XCD_MAJOR flags.
hipError_t launch_copy_chunks(const ChunkDesc* d_descs, uint32_t n_chunks,
                              uint64_t chunk_bytes, bool aligned16, bool host_side,
                              uint32_t threads, uint32_t unroll,
                              uint32_t max_grid, hipStream_t stream) {
  if (n_chunks == 0 || chunk_bytes == 0) return hipSuccess;
  if (threads == 0 || threads > 1024 || threads % 64 != 0) return hipErrorInvalidValue;
  const uint32_t flags = unroll & (PF_KERNEL_NONTEMPORAL | PF_KERNEL_XCD_MAJOR);
  unroll &= 0xffu;
  if (max_grid > kMaxGrid) max_grid = kMaxGrid;
  if (!aligned16 && !host_side) {
    uint64_t upc = (chunk_bytes / 16 + 63) / 64;
    if (upc == 0) upc = 1;
    const uint64_t units = upc * n_chunks;
    if (units > 0xffffffffu - 16u) return hipErrorInvalidValue;
    const uint32_t waves = kFixedThreads / 64;
    const uint32_t n_wg = static_cast<uint32_t>((units + waves - 1) / waves);
    const uint32_t cap = max_grid ? max_grid : kMaxGrid;
    hipLaunchKernelGGL(copy_chunks_unaligned_kernel, dim3(n_wg < cap ? n_wg : cap),
                       dim3(kFixedThreads), 0, stream, d_descs, static_cast<uint32_t>(upc),
                       static_cast<uint32_t>(units), chunk_bytes);
    return hipGetLastError();
  }
  if (!aligned16) {
    const uint32_t grid = n_chunks < kMaxGrid ? n_chunks : kMaxGrid;
    hipLaunchKernelGGL(copy_chunks_b1_kernel, dim3(grid), dim3(threads), 0,
                       stream, d_descs, n_chunks, chunk_bytes);
    return hipGetLastError();
  }
  // The waves' units are the launch's tiles; workgroups of at most kFixedThreads.
  if (threads > kFixedThreads) threads = kFixedThreads;
  uint32_t upc = 0, units = 0, c16 = 0;
  if (!tile_geometry(n_chunks, chunk_bytes, 64, unroll, &upc, &units, &c16) ||
      units > 0xffffffffu - 16u)
    return hipErrorInvalidValue;
  switch (unroll) {
    case 1: return launch_v16<1>(d_descs, upc, units, c16, threads, flags, max_grid, stream);
    case 2: return launch_v16<2>(d_descs, upc, units, c16, threads, flags, max_grid, stream);
    case 4: return launch_v16<4>(d_descs, upc, units, c16, threads, flags, max_grid, stream);
    case 8: return launch_v16<8>(d_descs, upc, units, c16, threads, flags, max_grid, stream);
    case 16: return launch_v16<16>(d_descs, upc, units, c16, threads, flags, max_grid, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_copy_chunks_queue(const ChunkDesc* d_descs, uint32_t n_chunks,
                                    uint64_t chunk_bytes, uint32_t threads, uint32_t unroll,
                                    uint32_t grid, bool table, const LayerMarks* marks,
                                    uint32_t* queue, hipStream_t stream) {
  if (n_chunks == 0 || chunk_bytes == 0) return hipSuccess;
  if (threads == 0 || threads > 1024 || threads % 64 != 0 || grid == 0 || !queue)
    return hipErrorInvalidValue;
  // Every layer of a marking launch has a chunk, so its table fits too.
  if (table && (n_chunks > kQueueTableMax || (marks && marks->n > n_chunks)))
    return hipErrorInvalidValue;
  if (marks && (marks->n == 0 || !marks->chunk_start || !marks->layer || !marks->counters ||
                marks->targets.count == 0 || marks->targets.count > kMaxSignalTargets))
    return hipErrorInvalidValue;
  const uint32_t flags = unroll & PF_KERNEL_NONTEMPORAL;
  unroll &= 0xffu;
  QueueLaunch q{dim3(grid), dim3(threads), stream, d_descs, n_chunks, 0, 0, 0, marks, queue,
                table};
  if (!tile_geometry(n_chunks, chunk_bytes, threads, unroll, &q.tiles_per_chunk, &q.n_tiles,
                     &q.chunk16))
    return hipErrorInvalidValue;
  if (static_cast<uint64_t>(q.n_tiles) + grid > 0xffffffffull) return hipErrorInvalidValue;
  if (grid > kMaxGrid) return hipErrorInvalidValue;
  switch (unroll) {
    case 1: launch_queue<1>(q, flags); break;
    case 2: launch_queue<2>(q, flags); break;
    case 4: launch_queue<4>(q, flags); break;
    case 8: launch_queue<8>(q, flags); break;
    case 16: launch_queue<16>(q, flags); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// Every unit of a marked launch lies in its chunk: chunk16 < 2^31, and the
// units of a launch are counted in 32 bits.
static bool marked_fits(const MarkedShape& s, uint32_t n_chunks, uint64_t chunk_bytes,
                        bool aligned16, uint64_t n_wg) {
  return !(aligned16 && chunk_bytes % 16) && chunk_bytes / 16 < (1ull << 31) &&
         static_cast<uint64_t>(n_chunks) * s.units_per_chunk + s.wg_units <= 0xffffffffull &&
         n_wg > 0 && n_wg + kMaxGrid <= 0xffffffffull;
}

template <bool ALIGNED, class Marks>
static hipError_t launch_marked(const ChunkDesc* d_descs, uint64_t chunk_bytes,
                                const MarkedShape& s, uint32_t n_wg, uint32_t max_grid,
                                const Marks& marks, hipStream_t stream) {
  uint32_t cap = max_grid ? max_grid : kMaxGrid;
  if (cap > kMaxGrid) cap = kMaxGrid;
  hipLaunchKernelGGL((copy_chunks_marked_kernel<kMarkedUnroll, ALIGNED, Marks>),
                     dim3(n_wg < cap ? n_wg : cap), dim3(kMarkedThreads), 0, stream, d_descs, s,
                     chunk_bytes, n_wg, marks);
  return hipGetLastError();
}

hipError_t launch_copy_chunks_marked(const ChunkDesc* d_descs, uint32_t n_chunks,
                                     uint64_t chunk_bytes, uint32_t max_grid, SliceMarks marks,
                                     hipStream_t stream) {
  if (n_chunks == 0 || chunk_bytes == 0) return hipSuccess;
  if (marks.n == 0 || marks.n > kSliceMarkLayers || !marks.counters ||
      marks.targets.count == 0 || marks.targets.count > kMaxSignalTargets ||
      marks.chunk_start[0] != 0 || marks.chunk_start[marks.n] != n_chunks)
    return hipErrorInvalidValue;
  const MarkedShape s = marked_shape(chunk_bytes, n_chunks, marks.n, true);
  // Groups in chunk order, each counting at least its own units.
  uint64_t wg = 0;
  for (uint32_t g = 0; g < marks.n; ++g) {
    if (marks.chunk_start[g + 1] <= marks.chunk_start[g]) return hipErrorInvalidValue;
    const uint64_t chunks = marks.chunk_start[g + 1] - marks.chunk_start[g];
    if (marks.units[g] != 0 && marks.units[g] < chunks * s.units_per_chunk)
      return hipErrorInvalidValue;
    marks.wg_start[g] = static_cast<uint32_t>(wg);
    wg += marked_workgroups(s, chunks);
  }
  if (!marked_fits(s, n_chunks, chunk_bytes, true, wg)) return hipErrorInvalidValue;
  marks.wg_start[marks.n] = static_cast<uint32_t>(wg);
  return launch_marked<true>(d_descs, chunk_bytes, s, static_cast<uint32_t>(wg), max_grid, marks,
                             stream);
}

hipError_t launch_copy_chunks_mark_table(const ChunkDesc* d_descs, uint32_t n_chunks,
                                         uint64_t chunk_bytes, bool aligned16, uint32_t n_wg,
                                         uint32_t max_grid, const MarkTable& marks,
                                         hipStream_t stream) {
  if (n_chunks == 0 || chunk_bytes == 0) return hipSuccess;
  if (marks.n == 0 || !marks.wg_start || !marks.chunk_start || !marks.layer || !marks.counters ||
      marks.targets.count == 0 || marks.targets.count > kMaxSignalTargets)
    return hipErrorInvalidValue;
  const MarkedShape s = marked_shape(chunk_bytes, n_chunks, marks.n, aligned16);
  if (!marked_fits(s, n_chunks, chunk_bytes, aligned16, n_wg)) return hipErrorInvalidValue;
  return aligned16 ? launch_marked<true>(d_descs, chunk_bytes, s, n_wg, max_grid, marks, stream)
                   : launch_marked<false>(d_descs, chunk_bytes, s, n_wg, max_grid, marks, stream);
}

hipError_t launch_mark_layers(const LayerList& list, const SignalTargets& t,
                              hipStream_t stream) {
  if (list.n == 0) return hipSuccess;
  if (list.n > kLayerListMax || t.count == 0 || t.count > kMaxSignalTargets)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(mark_layers_kernel, dim3(1), dim3(kLayerListMax), 0, stream, list, t);
  return hipGetLastError();
}

hipError_t launch_wait_word(uint64_t word, uint64_t value, uint64_t max_ticks,
                            uint64_t timed_out, hipStream_t stream) {
  hipLaunchKernelGGL(wait_word_kernel, dim3(1), dim3(64), 0, stream,
                     reinterpret_cast<const uint64_t*>(word), value, max_ticks,
                     reinterpret_cast<uint32_t*>(timed_out));
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Synthetic data: splitmix64 words, word[i] = mix64(seed + (off+i+1)*GAMMA).
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

static constexpr uint64_t kGamma = 0x9E3779B97F4A7C15ull;

__global__ void __launch_bounds__(256)
fill_random_kernel(uint64_t* __restrict__ dst, uint64_t n_words, uint64_t seed,
                   uint64_t word_offset) {
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
       i < n_words; i += step)
    dst[i] = mix64(seed + (word_offset + i + 1) * kGamma);
}

__global__ void __launch_bounds__(256)
verify_random_kernel(const uint64_t* __restrict__ src, uint64_t n_words,
                     uint64_t seed, uint64_t word_offset,
                     unsigned long long* count) {
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  unsigned long long bad = 0;
  for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
       i < n_words; i += step)
    bad += src[i] != mix64(seed + (word_offset + i + 1) * kGamma);
  if (bad) atomicAdd(count, bad);
}

// One workgroup per chunk (grid-stride over chunks).
__global__ void __launch_bounds__(256)
verify_random_chunks_kernel(const uint64_t* __restrict__ addrs,
                            const uint64_t* __restrict__ word_offsets, uint64_t n,
                            uint64_t chunk_words, uint64_t seed,
                            unsigned long long* count) {
  unsigned long long bad = 0;
  for (uint64_t c = blockIdx.x; c < n; c += gridDim.x) {
    const g_u64* src = reinterpret_cast<const g_u64*>(addrs[c]);
    const uint64_t off = word_offsets[c];
    for (uint64_t i = threadIdx.x; i < chunk_words; i += blockDim.x)
      bad += src[i] != mix64(seed + (off + i + 1) * kGamma);
  }
  if (bad) atomicAdd(count, bad);
}

__global__ void __launch_bounds__(256)
compare_kernel(const uint8_t* __restrict__ a, const uint8_t* __restrict__ b,
               uint64_t n, unsigned long long* count) {
  const uint64_t step = static_cast<uint64_t>(gridDim.x) * blockDim.x;
  const uint64_t tid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  unsigned long long bad = 0;
  const bool aligned = ((reinterpret_cast<uint64_t>(a) | reinterpret_cast<uint64_t>(b)) & 7) == 0;
  uint64_t tail_start = 0;
  if (aligned) {
    const uint64_t* wa = reinterpret_cast<const uint64_t*>(a);
    const uint64_t* wb = reinterpret_cast<const uint64_t*>(b);
    const uint64_t nw = n / 8;
    for (uint64_t i = tid; i < nw; i += step) {
      uint64_t x = wa[i] ^ wb[i];
      for (int k = 0; k < 8; ++k) bad += ((x >> (8 * k)) & 0xff) != 0;
    }
    tail_start = nw * 8;
  }
  for (uint64_t i = tail_start + tid; i < n; i += step) bad += a[i] != b[i];
  if (bad) atomicAdd(count, bad);
}

__global__ void spin_kernel(uint64_t ticks) {
  if (threadIdx.x == 0) {
    const uint64_t start = static_cast<uint64_t>(wall_clock64());
    while (static_cast<uint64_t>(wall_clock64()) - start < ticks)
      __builtin_amdgcn_s_sleep(4);
  }
}

static uint32_t grid_for(uint64_t items, uint32_t threads) {
  uint64_t g = (items + threads - 1) / threads;
  if (g > 65536) g = 65536;
  if (g == 0) g = 1;
  return static_cast<uint32_t>(g);
}

hipError_t launch_fill_random(uint64_t dst, uint64_t size_bytes, uint64_t seed,
                              uint64_t word_offset, hipStream_t stream) {
  const uint64_t n = size_bytes / 8;
  hipLaunchKernelGGL(fill_random_kernel, dim3(grid_for(n, 256)), dim3(256), 0,
                     stream, reinterpret_cast<uint64_t*>(dst), n, seed,
                     word_offset);
  return hipGetLastError();
}

hipError_t launch_verify_random(uint64_t addr, uint64_t size_bytes,
                                uint64_t seed, uint64_t word_offset,
                                unsigned long long* d_count,
                                hipStream_t stream) {
  const uint64_t n = size_bytes / 8;
  hipLaunchKernelGGL(verify_random_kernel, dim3(grid_for(n, 256)), dim3(256), 0,
                     stream, reinterpret_cast<const uint64_t*>(addr), n, seed,
                     word_offset, d_count);
  return hipGetLastError();
}

hipError_t launch_verify_random_chunks(const uint64_t* d_addrs,
                                       const uint64_t* d_word_offsets,
                                       uint64_t n, uint64_t chunk_bytes,
                                       uint64_t seed,
                                       unsigned long long* d_count,
                                       hipStream_t stream) {
  const uint32_t grid = n < 65536 ? static_cast<uint32_t>(n) : 65536u;
  hipLaunchKernelGGL(verify_random_chunks_kernel, dim3(grid), dim3(256), 0, stream,
                     d_addrs, d_word_offsets, n, chunk_bytes / 8, seed, d_count);
  return hipGetLastError();
}

hipError_t launch_compare(uint64_t a, uint64_t b, uint64_t size_bytes,
                          unsigned long long* d_count, hipStream_t stream) {
  hipLaunchKernelGGL(compare_kernel, dim3(grid_for(size_bytes / 8 + 1, 256)),
                     dim3(256), 0, stream, reinterpret_cast<const uint8_t*>(a),
                     reinterpret_cast<const uint8_t*>(b), size_bytes, d_count);
  return hipGetLastError();
}

hipError_t launch_spin(uint64_t ticks, hipStream_t stream) {
  hipLaunchKernelGGL(spin_kernel, dim3(1), dim3(64), 0, stream, ticks);
  return hipGetLastError();
}

}  // namespace pf
