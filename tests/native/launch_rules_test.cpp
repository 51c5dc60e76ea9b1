// launch_rules_test.cpp — the launch shapes' rules (pf_launch.h) on the host
// (no GPU), built by tests/test_native.py from the library's own sources:
//   * a queued save keeps its route's workgroups, loads in flight and flags,
//     with its descriptors in place or not;
//   * the calls over the host link whose descriptors are read in place;
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
  for (bool table : {false, true}) {
    const std::string where = table ? " in place" : " uploaded";
    same(queue_shape(save, 32768, true, table, false, 0), save, "default save" + where);
    for (uint32_t grid : {1u, 3u, 32u, 64u, 5000u}) {
      const QueueShape s{256, 4u | PF_KERNEL_NT_LOADS, grid};
      same(queue_shape(s, 131072, true, table, false, 0), s,
           "save of " + std::to_string(grid) + " workgroups" + where);
      same(queue_shape(s, 131072, true, table, false, 7), {256, s.unroll, grid < 7 ? grid : 7},
           "capped save of " + std::to_string(grid) + " workgroups" + where);
    }
    // A 4 KiB chunk is 128 lanes of two words, a 16-byte one a wave.
    same(queue_shape(save, 4096, true, table, false, 0), {128, save.unroll, 128},
         "save of 4 KiB chunks" + where);
    same(queue_shape(save, 4096, true, table, false, 100), {128, save.unroll, 100},
         "capped save of 4 KiB chunks" + where);
    same(queue_shape({512, 2, 1u << 20}, 16, true, table, false, 0), {64, 2, 1u << 16},
         "save of 16-byte chunks" + where);
  }
  for (bool is_save : {false, true}) {
    const std::string what = is_save ? "save in place" : "load in place";
    expect(table_in_place(1, 16, is_save) && table_in_place(512, 16, is_save), what);
    expect(table_in_place(513, 4096, is_save) && table_in_place(1024, 1 << 20, is_save), what);
    expect(table_in_place(513, 4080, is_save) == !is_save, what + ", short chunks");
    expect(!table_in_place(1025, 4096, is_save), what + ", many chunks");
  }
  if (failures) {
    std::printf("%d checks failed\n", failures);
    return 1;
  }
  std::printf("ok\n");
  return 0;
}
