// Host check of the phases of the BFS and SSSP kernels
// (tpds22-artifact_amd/csrc/team_rounds.hpp), built with g++ by
// tests/test_team_rounds.py.  A launch is played on a host copy of the counters:
// rounds of given widths, those up to a bound by the team, the others by the grid,
// stretches of at most 5 rounds, some of a round's vertices in the segments and some
// in the queue.  In every phase the writes are put in order, each workgroup outside
// the team reads its input at random moments between them (the first, the last and
// all moments in between, so after any number of team rounds), and a workgroup of
// the team reads first.  Everyone has to see the same input: the width that the
// round before made.
// Every third launch has bucket steps between its rounds, with the SSSP's far counts.
// "plant shared": the team counts in the grid's counters, by level.
// "plant report": every stretch leaves its report in the same place.
// "plant far": a stretch goes on over any number of bucket steps.
// All must be caught.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <functional>
#include <random>
#include <vector>

#include "team_rounds.hpp"

using namespace hs_rounds;

namespace {
bool plant_shared, plant_report, plant_far;

struct Launch {
  uint64_t word[kSlots][64] = {};
  std::mt19937_64 rng;
  long reads = 0, wrong = 0;

  uint32_t report_at(uint32_t k) const { return plant_report ? kReport : report(k); }
  Side team() const { return plant_shared ? kGrid : kTeam; }

  // One phase: the writes in order, `readers` reads of each word at random moments.
  void phase(const std::vector<std::function<void()>> &writes, const std::vector<std::pair<const uint64_t *, uint64_t>> &input) {
    std::vector<std::vector<const std::pair<const uint64_t *, uint64_t> *>> at(writes.size() + 1);
    for (const auto &in : input)
      for (int r = 0; r < 6; ++r) at[r == 0 ? 0 : r == 1 ? writes.size() : rng() % (writes.size() + 1)].push_back(&in);
    for (size_t t = 0; t <= writes.size(); ++t) {
      for (const auto *in : at[t]) {
        ++reads;
        wrong += *in->first != in->second;
      }
      if (t < writes.size()) writes[t]();
    }
  }

  // widths[r] = 0 inside a launch of `buckets`: round r is a bucket step.  A round adds
  // its number to the far list of its bucket, a bucket step of e to that of e + 1.
  void run(const std::vector<uint64_t> &widths, uint64_t bound, bool buckets) {
    word[slot(kGrid, kLight, 0)][0] = widths[0];
    uint32_t j = 0, e = 0;
    uint64_t far = 0;  // of bucket e
    bool reported = false;
    auto last = [&](uint32_t r) { return r >= widths.size() || (widths[r] == 0 && !buckets); };
    // the far list's part of round r
    auto step = [&](std::vector<std::function<void()>> &w, uint32_t r) {
      if (!buckets) return;
      if (widths[r] == 0) {
        const uint32_t gone = other(e + 2);
        w.push_back([this, gone] { word[gone][0] = 0; });
        far = 0;
        ++e;
      }
      far += r + 1;
      const uint32_t at = other(e);
      const uint64_t n = r + 1;
      w.push_back([this, at, n] { word[at][0] += n; });
    };
    for (uint32_t r = 0, k = 0; !last(r); ++k) {
      std::vector<std::function<void()>> w;
      std::vector<std::pair<const uint64_t *, uint64_t>> input;
      if (reported) {
        input.push_back({&word[report_at(k - 1)][0], r});
        input.push_back({&word[report_at(k - 1)][1], widths[r]});
        if (widths[r] == 0) input.push_back({&word[report_at(k - 1)][2], far});
      } else {
        input.push_back({&word[slot(kGrid, kLight, plant_shared ? r : k)][0], widths[r]});
        input.push_back({&word[slot(kGrid, kChunks, plant_shared ? r : k)][0], r ? widths[r] / 7 : 0});
        if (widths[r] == 0) input.push_back({&word[other(e)][0], far});
      }
      const bool one_bucket = !reported && widths[r] == 0;
      auto clear = [&](uint32_t s) { w.push_back([this, s] { word[s][0] = 0; }); };
      auto add = [&](Side side, Counter c, uint32_t i, uint64_t n) {
        w.push_back([this, side, c, i, n] { word[slot(side, c, i)][0] += n; });
      };
      const bool by_team = widths[r] <= bound;
      open_round(kGrid, plant_shared ? r : k, clear);
      if (!by_team) {
        add(kGrid, kGrab, plant_shared ? r : k, 1);
        if (r + 1 < widths.size()) {
          add(kGrid, kLight, plant_shared ? r + 1 : k + 1, widths[r + 1]);
          add(kGrid, kChunks, plant_shared ? r + 1 : k + 1, widths[r + 1] / 7);
        }
        step(w, r);
        ++r;
      } else {
        for (int q = 0; q < 5; ++q) {
          open_round(team(), plant_shared ? r : j, clear);
          add(team(), kGrab, plant_shared ? r : j, 1);
          if (r + 1 < widths.size()) {
            add(team(), kLight, plant_shared ? r + 1 : j + 1, widths[r + 1]);
            add(team(), kChunks, plant_shared ? r + 1 : j + 1, widths[r + 1] / 7);
          }
          step(w, r);
          ++r;
          ++j;
          if (last(r) || widths[r] > bound) break;
          if (widths[r] == 0 && one_bucket && !plant_far) break;
        }
        const uint64_t next = r < widths.size() ? widths[r] : 0;
        const uint32_t at = report_at(k);
        w.push_back([this, at, r] { word[at][0] = r; });
        w.push_back([this, at, next] { word[at][1] = next; });
        w.push_back([this, at, n = far] { word[at][2] = n; });
      }
      reported = by_team;
      phase(w, input);
      if (wrong) return;  // what follows would read a launch that has gone wrong
    }
  }
};
}  // namespace

int main(int argc, char **argv) {
  plant_shared = argc > 2 && !strcmp(argv[2], "shared");
  plant_far = argc > 2 && !strcmp(argv[2], "far");
  plant_report = argc > 2 && !strcmp(argv[2], "report");
  long reads = 0, launches = 0, bad = 0;
  for (int trial = 0; trial < 3000; ++trial) {
    Launch l;
    l.rng.seed(9100 + trial);
    std::vector<uint64_t> widths{1};
    const size_t rounds = 1 + l.rng() % 60;
    for (size_t i = 1; i < rounds; ++i) widths.push_back(1 + (l.rng() % 3 ? l.rng() % 100 : l.rng() % 2000));
    if (trial % 3 == 0)
      for (size_t i = 1; i < rounds; ++i) widths[i] = l.rng() % 3 ? widths[i] : 0;
    l.run(widths, 100, trial % 3 == 0);
    reads += l.reads;
    bad += l.wrong != 0;
    ++launches;
  }
  // a team leaves the kernel when a wait fails: not beside a barrier that never does
  for (uint32_t grid = 1; grid < 300; ++grid)
    for (uint32_t size = 1; size <= grid; ++size) {
      bad += team_usable(size, grid, false);
      bad += team_usable(size, grid, true) != (size < grid && size <= 32);
      bad += team_edges(size) != size * team_edges(32) / 32;  // a small team takes its share
    }
  // a stretch is shorter than the limit of the others' polls, one in 1.4 us, for rounds
  // of a team of up to 500 us, and never empty
  for (uint64_t limit = 1; limit < 1ull << 32; limit = limit * 3 / 2 + 1) {
    const uint32_t rounds = team_rounds((uint32_t)limit);
    bad += rounds < 1 || rounds > 256 || (rounds > 1 && rounds * 512ull > limit + 512);
  }
  // a mesh of mean degree 3.4, counted as 4, 1000 levels of 1000 vertices: never pulled;
  // a power-law graph's wide levels: pulled, its first and last: not
  for (uint64_t level = 0; level < 1000; ++level) bad += pull_pays(4000, 4000 * level, 3400000, 1000000);
  const uint64_t n = 1 << 22, m = 16 * n;
  bad += pull_pays(16, 0, m, n) || pull_pays(16 * 20000, 16, m, n) || pull_pays(16 * 400, m, m, n);
  bad += !pull_pays(m / 6, m / 100, m, n) || !pull_pays(m / 2, m / 5, m, n) || !pull_pays(n, m, m, n);
  printf("launches %ld reads %ld failures %ld\n", launches, reads, bad);
  return bad ? 1 : 0;
}
