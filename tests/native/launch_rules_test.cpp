// launch_rules_test.cpp — the launch shapes' rules (pf_launch.h) on the host
// (no GPU), built by tests/test_native.py from the library's own sources:
//   * a queued launch keeps its route's workgroups, loads in flight and flags;
//   * a small load at the default grid: workgroups by its bytes;
//   * the calls over the host link, and between device buffers, whose
//     descriptors are read in place;
//   * a marked copy's workgroups a layer, by the layer's and the launch's bytes;
//   * chunks smaller than a tile: workgroups of the chunk's size, as many
//     lanes in all, within the caps.
// Exit status 0 and "ok" on success; the first failed checks are printed.
#include <cstdio>
#include <string>

#include "pf_launch.h"

using namespace pf;

namespace {

int failures = 0;

void expect(bool cond, const std::string& what) {
  if (!cond && ++failures <= 20) std::printf("FAILED: %s\n", what.c_str());
}

std::string text(const QueueShape& s) {
  return std::to_string(s.threads) + " threads, unroll " + std::to_string(s.unroll) + ", grid " +
         std::to_string(s.grid);
}

void same(const QueueShape& got, const QueueShape& want, const std::string& what) {
  expect(got.threads == want.threads && got.unroll == want.unroll && got.grid == want.grid,
         what + ": " + text(got) + ", not " + text(want));
}

}  // namespace

int main() {
  const QueueShape save{PF_SAVE_HOST_DEFAULT_THREADS, PF_SAVE_HOST_DEFAULT_UNROLL,
                        PF_SAVE_HOST_DEFAULT_GRID};
  same(queue_shape(save, 32768, 0), save, "default save");
  for (uint32_t grid : {1u, 3u, 32u, 64u, 5000u}) {
    const QueueShape s{256, 4u | PF_KERNEL_NT_LOADS, grid};
    const std::string what = std::to_string(grid) + " workgroups";
    same(queue_shape(s, 131072, 0), s, what);
    same(queue_shape(s, 131072, 7), {256, s.unroll, grid < 7 ? grid : 7}, what + ", capped");
  }
  // A 4 KiB chunk is 128 lanes of two words, a 16-byte one a wave.
  same(queue_shape(save, 4096, 0), {128, save.unroll, 128}, "4 KiB chunks");
  same(queue_shape(save, 4096, 100), {128, save.unroll, 100}, "4 KiB chunks, capped");
  same(queue_shape({512, 2, 1u << 20}, 16, 0), {64, 2, 1u << 16}, "16-byte chunks");
  // A small load's workgroups: 16 up to 2 MiB, the route's 64 from 8 MiB on.
  const uint64_t loads[][3] = {{1, 16, 16}, {64, 32768, 16}, {64, 36864, 18}, {128, 32768, 32},
                               {255, 32768, 63}, {256, 32768, 64}, {1024, 131072, 64},
                               {1, 1ull << 34, 64}};
  for (const auto& t : loads)
    expect(small_load_grid(PF_LOAD_HOST_DEFAULT_GRID, t[0], t[1]) == t[2],
           "load of " + std::to_string(t[0]) + " chunks of " + std::to_string(t[1]));
  expect(small_load_grid(3, 64, 32768) == 3, "no more workgroups than the route's");
  for (bool is_save : {false, true}) {
    const std::string what = is_save ? "save in place" : "load in place";
    expect(table_in_place(1, 16, is_save) && table_in_place(512, 16, is_save), what);
    expect(table_in_place(513, 4096, is_save) && table_in_place(1024, 1 << 20, is_save), what);
    expect(table_in_place(513, 4080, is_save) == !is_save, what + ", short chunks");
    expect(!table_in_place(1025, 4096, is_save), what + ", many chunks");
  }
  // Between device buffers: by the bytes that waves of 1 KiB move, but for few chunks.
  const uint64_t MiB = 1ull << 20;
  expect(waves_in_place(2048, 64 * MiB) && waves_in_place(65, 0), "narrow waves in place");
  expect(!waves_in_place(2048, 64 * MiB + 1) && !waves_in_place(65, 512 * MiB),
         "narrow waves uploaded");
  expect(waves_in_place(64, 512 * MiB) && waves_in_place(1, 1ull << 40), "few chunks in place");
  // Workgroups that report a layer of a marked copy, one after another: few enough
  // for large layers, and enough of them in launches of small ones.
  const uint64_t marked[][4] = {{1280, 32768, 1, 640},  {640, 32768, 1, 320},
                                {128, 32768, 1, 128},   {32, 32768, 1, 128},
                                {10240, 32768, 8, 640}, {7808, 36864, 61, 144},
                                {64, 32768, 32, 8}};
  for (const auto& t : marked) {
    const MarkedShape s = marked_shape(t[1], t[0], t[2], true);
    expect(marked_workgroups(s, t[0] / t[2]) == t[3],
           "marked copy of " + std::to_string(t[0]) + " chunks in " + std::to_string(t[2]) +
               " layers: " + std::to_string(marked_workgroups(s, t[0] / t[2])));
    // The units of a chunk do not depend on the launch that copies it.
    expect(s.units_per_chunk == marked_shape(t[1], 1, 1, true).units_per_chunk, "units");
  }
  const uint64_t odd[][2] = {{1, 1}, {15, 1}, {1024, 1}, {1039, 1}, {1040, 2}, {12301, 12}};
  for (const auto& t : odd)
    expect(marked_shape(t[0], 100, 1, false).units_per_chunk == t[1], "unaligned units");
  if (failures) {
    std::printf("%d checks failed\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
