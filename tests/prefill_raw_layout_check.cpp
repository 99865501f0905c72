// Host-side walk over what the prefill kernel does on raw weights (the mx_raw_* functions of
// vkernels_amd/csrc/moe_prefill_layout.hpp, compiled for the CPU):
//   - every load of codes and scale bytes lies inside the tensors, steps past the end included,
//     and the 16 bytes a lane takes as its operand are K block 2 half + hh of its weight row;
//   - the K loop's schedule of a wavefront, restated with the schedule functions of the same header:
//     no operand of rows is read before every wavefront's copies of it have landed, no copy
//     overwrites a ring slot that may still be read, no weight register is read before its load has
//     landed or loaded again before it is read, no scale bytes are read before their copies have
//     landed or replaced before they are read, nothing is in flight when the epilogue begins.
// Usage: prefill_raw_layout_check stage K ncols experts ; exit status 0 = all hold.
// With -DVK_LAYOUT_BREAK_WAIT=n wait n (0, 1) lets one operation too many stay outstanding.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "moe_prefill_layout.hpp"

using namespace vk;

#define CHECK(cond, ...)                          \
  do {                                            \
    if (!(cond)) {                                \
      std::fprintf(stderr, "FAILED %s: ", #cond); \
      std::fprintf(stderr, __VA_ARGS__);          \
      std::fprintf(stderr, "\n");                 \
      return 1;                                   \
    }                                             \
  } while (0)

#ifndef VK_LAYOUT_BREAK_WAIT
#define VK_LAYOUT_BREAK_WAIT -1
#endif

namespace {

constexpr int kTerms = 3;

enum Kind { kCopy, kLoad, kScales };

struct Model {
  struct Op { Kind kind; int id; };  // K step of a copy, half step of a load, group of four steps of scale bytes
  std::vector<Op> ops;
  size_t landed = 0;
  std::vector<int> count[3], done[3];
  std::vector<int> copies_seen, reads, reads_done, reads_seen, moved;
  int group_in_lds = -1;
  explicit Model(int nsteps) {
    const size_t n = 2 * (size_t)nsteps + 16;
    for (int k = 0; k < 3; ++k) count[k].assign(n, 0), done[k].assign(n, 0);
    for (auto* v : {&copies_seen, &reads, &reads_done, &reads_seen, &moved}) v->assign(n, 0);
  }
  void issue(Kind k, int id) {
    ops.push_back({k, id});
    ++count[k][id];
  }
  void wait(int n) {
    for (; landed + (size_t)n < ops.size(); ++landed) ++done[ops[landed].kind][ops[landed].id];
  }
  void barrier() {
    copies_seen = done[kCopy];
    reads_seen = reads_done;
  }
};

int walk(int live, int nsteps) {
  Model m(nsteps);
  const int G = mx_raw_groups(live, kTerms), Q = 2 * G, ops = mx_raw_ops(kTerms), step_copies = mx_row_ops(kTerms);
  auto issue = [&](int step, int half, int k) {
    if (k < 4) {
      const int s = 2 * step + half;
      if (s >= 4) CHECK(m.moved[s - 4] == 16, "live %d: half step %d is loaded over codes that are still to be moved", live, s);
      CHECK(mx_raw_weight_set(s) == mx_raw_weight_set(s + 4), "sets");
      m.issue(kLoad, s);
    } else {
      const int old = step - kMxRing;
      if (old >= 0) CHECK(m.reads_seen[old] == m.reads[old] && m.reads[old] > 0, "live %d: a copy of step %d overwrites one that is read", live, step);
      m.issue(kCopy, step);
    }
    return 0;
  };
  auto move = [&](int s, int words) {
    CHECK(m.done[kLoad][s] == 4, "live %d: codes of half step %d are moved before they have landed", live, s);
    m.moved[s] += words;
    return 0;
  };
  auto read_scales = [&](int step) {
    CHECK(m.done[kScales][step >> 2] == 2 && m.group_in_lds == step >> 2, "live %d: scale bytes of step %d", live, step);
    return 0;
  };
  auto read = [&](int step) {
    CHECK(m.copies_seen[step] == step_copies, "live %d: an operand of step %d is read before its copies have landed", live, step);
    ++m.reads[step];
    return 0;
  };
  m.issue(kScales, 0);
  m.issue(kScales, 0);
  m.group_in_lds = 0;
  for (int s = 0; s < 4; ++s)
    for (int k = 0; k < ops; ++k)
      if (issue(s >> 1, s & 1, k)) return 1;
  m.wait(2 * ops);
  m.barrier();
  if (read_scales(0) || move(0, 16) || read(0) || read(0)) return 1;
  for (int c = 0; c < nsteps; ++c) {
    for (int q = 0; q < Q; ++q) {
      const int half = q / G;
      CHECK(m.moved[2 * c + half] == 16, "live %d: half step %d is multiplied before all its codes are moved", live, 2 * c + half);
      if (read(q + 2 < Q ? c : c + 1)) return 1;
      for (int t = 0; t < 4; ++t) {
        for (int k = 0; k < ops; ++k)
          if (mx_raw_op_slot(live, kTerms, k) == 4 * (q - half * G) + t && issue(c + 2, half, k)) return 1;
        for (int x = 0; x < 16; ++x)
          if (mx_raw_fix_slot(live, kTerms, x) == 4 * (q - half * G) + t && move(2 * c + half + 1, 1)) return 1;
      }
      if (q == G - 1) {
        m.wait(mx_raw_middle_wait(live, kTerms) + (VK_LAYOUT_BREAK_WAIT == 0 ? 1 : 0));
        if (c + 1 < nsteps && read_scales(c + 1)) return 1;
      }
      if (q == G && (c & 3) == 2 && c + 2 < nsteps) {
        m.group_in_lds = (c + 2) >> 2;
        m.issue(kScales, (c + 2) >> 2);
        m.issue(kScales, (c + 2) >> 2);
      }
      if (q == Q - 3) {
        m.wait(mx_raw_row_wait(live, kTerms) + (VK_LAYOUT_BREAK_WAIT == 1 ? 1 : 0));
        m.reads_done = m.reads;
        m.barrier();
      }
    }
  }
  m.wait(0);
  CHECK(m.landed == m.ops.size(), "operations in flight when the epilogue starts");
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const int stage = std::atoi(argv[1]), K = std::atoi(argv[2]), ncols = std::atoi(argv[3]), E = std::atoi(argv[4]);
  const int nsteps = K / 128, rows = stage == 0 ? 2 * ncols : ncols;
  CHECK(K % kMxRawK == 0 && nsteps % 4 == 0, "K");
  const size_t code_bytes = (size_t)E * rows * (K / 2), scale_bytes = (size_t)E * rows * (K / 32);
  for (int unit = 0; unit < mx_units(stage, ncols); ++unit)
    for (int t = 0; t < 4; ++t)
      for (int n = 0; n < 32; ++n) {
        const int row = mx_raw_row(stage, ncols, unit, t, n);
        CHECK(row >= 0 && row < rows, "row");
        const int want = mx_weight_row(stage, ncols, unit, t, n);
        CHECK(row == want || want >= rows, "row");
        for (int step = 0; step < nsteps + 2; ++step) {
          const int at = step < nsteps ? step : nsteps - 1;
          for (int half = 0; half < 2; ++half)
            for (int hh = 0; hh < 2; ++hh) {
              const size_t off = (size_t)(E - 1) * rows * (K / 2) + mx_raw_lane_offset(row, K, hh) + mx_raw_load_offset(step, nsteps, half);
              CHECK(off + 16 <= code_bytes, "codes");
              CHECK(mx_raw_lane_offset(row, K, hh) + mx_raw_load_offset(step, nsteps, half) ==
                        (size_t)row * (K / 2) + (size_t)at * 64 + (2 * half + hh) * 16, "K block");
            }
          const int start = step < nsteps - 4 ? step : nsteps - 4;
          CHECK((size_t)(E - 1) * rows * (K / 32) + (size_t)row * (K / 32) + 4 * start + 16 <= scale_bytes, "scale bytes");
        }
      }
  CHECK(kMxRing * mx_slot_bytes(kTerms) + kMxWaves * kMxRawScaleBytes <= 160 * 1024 - 2048, "LDS");
  for (int live = 2; live <= 4; ++live)
    if (walk(live, nsteps)) return 1;
  return 0;
}
