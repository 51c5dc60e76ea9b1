// pf_launch.h — how the transfer code (pf_transfer.cpp) shapes its launches,
// as plain functions of sizes and settings, in a header of their own so the
// rules are tested on the host (tests/native/launch_rules_test.cpp).
#pragma once

#include <algorithm>
#include <cstdint>

#include "pf_common.h"

namespace pf {

// A queued launch: threads per workgroup, loads in flight per lane with their
// flags, and persistent workgroups.
struct QueueShape {
  uint32_t threads, unroll, grid;
};

// Whether a call of n descriptors with a launch over the host link, in chunks of
// chunk_bytes, leaves them in host memory for its workgroups to take into LDS.
// Every workgroup reads them all, and a save of short chunks has many workgroups
// for few bytes: 1,024 chunks of 256 B to 2 KiB save in 62-94 us in place and
// 51-83 uploaded, of 4 KiB in 120 and 124, 256 chunks of 1 KiB in 38.6 and 39.5.
inline bool table_in_place(size_t n, uint64_t chunk_bytes, bool is_save) {
  return n <= kQueueTableMax && !(is_save && n > 512 && chunk_bytes < 4096);
}

// Whether a call of n descriptors leaves them in host memory for the waves of a
// copy between device buffers, which read their own: `narrow` bytes of its copies
// go by waves of 1 KiB, a read each.  In place less uploaded, us a call: 1,024
// chunks of 32 KiB gather -3.5, of 64 KiB -1.3, of 128 KiB +1.4, of 256 KiB +7.1,
// of 512 KiB +13.4 (and scattered by waves of 2 KiB, or marked, -3 to -10 all the
// way); of 64 KiB and 3 bytes -0.3, of 128 KiB and 3 bytes +6.  The waves of one
// chunk share its read, so few chunks cost little: 32 of 8 MiB -5.5.
inline bool waves_in_place(size_t n, uint64_t narrow) { return n <= 64 || narrow <= 64ull << 20; }

// A marked load's layers from device memory share one launch that marks each as it
// lands, but for layers of this size: those have a fixed-map launch each, and their
// marks behind it.  The marked kernel falls behind that by a fifth once a call
// exceeds the memory-side cache (256 MiB), and the launches cost about 8 us a layer.
// One launch and one a layer, us a call: 8 layers of 32 MiB 105 and 146, of 64 MiB
// 238 and 228 (by 32 KiB chunks 252 and 256), of 96 MiB 347 and 316 (362 and 351), of
// 128 MiB 461 and 402 (469 and 453), of 256 MiB 874 and 725.
constexpr uint64_t kOwnLaunchBytes = 96ull << 20;

// Workgroups of a load of n chunks in place on a route at its default grid.  Each
// reads the whole table first, and a load of few bytes has no work for many:
// with 16 and 64 workgroups, 2 MiB (64 chunks of 32 KiB) load in 61.7 and 65.3 us,
// marked 67.4 and 70.1, 10 MiB in 208.3 and 211.3, 32 MiB in 611 and 614.  Beside
// a save the many get more of the link, from about 8 MiB on: with 16 and 64, 2 MiB
// take 2.5 and 2.7 ms, 10 MiB 4.3 and 2.1, 32 MiB 5.7 and 1.8, 128 MiB 12.2 and
// 4.7.  So one a 128 KiB, at least 16.
inline uint32_t small_load_grid(uint32_t grid, uint64_t n, uint64_t chunk_bytes) {
  const uint64_t want = n * chunk_bytes / (128u << 10);
  return static_cast<uint32_t>(std::min<uint64_t>(grid, std::max<uint64_t>(16, want)));
}

// The queued launch of a route set to s for chunks of chunk_bytes.  max_grid caps
// the workgroups (0: no cap).
//
// The route's setting holds, however few the chunks of a save.  A shape of their own
// for small ones (8 workgroups, tiles by a fixed map, streaming stores) was as
// fast alone (64, 320 and 1,024 chunks of 32 KiB in 62, 217-240 and 624 us, so
// 64, 227 and 646) but ran at the pace of the XCD that a restore beside it left
// the least of the link: 1.4, 4.4 and 12.1 ms beside one, so 0.35, 0.98 and 2.0.
inline QueueShape queue_shape(QueueShape s, uint64_t chunk_bytes, uint32_t max_grid) {
  if (max_grid && s.grid > max_grid) s.grid = max_grid;
  // Chunks smaller than a tile (e.g. 4 KiB segments of one tensor-parallel
  // rank) get workgroups sized to the chunk, and proportionally more of
  // them, so each pull moves a whole chunk with every lane busy and the
  // bytes in flight stay the same (measured: 4 KiB-segment save 53.9 ->
  // 55.6 GB/s).
  const uint64_t u = s.unroll & 0xffu;
  const uint64_t want = u ? ((chunk_bytes / 16 + u - 1) / u + 63) / 64 * 64 : s.threads;
  if (want < s.threads) {
    const uint32_t threads = static_cast<uint32_t>(want < 64 ? 64 : want);
    const uint64_t grid = static_cast<uint64_t>(s.grid) * s.threads / threads;
    s.grid = static_cast<uint32_t>(std::min<uint64_t>(grid, 1u << 16));
    if (max_grid && s.grid > max_grid) s.grid = max_grid;
    s.threads = threads;
  }
  return s;
}

}  // namespace pf
