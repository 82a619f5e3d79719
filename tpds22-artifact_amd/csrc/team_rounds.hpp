// team_rounds.hpp -- where the BFS and SSSP kernels keep their counters, shared by
// the kernels (graph.hip) and a host check (tests/test_team_rounds.py builds
// tests/team_rounds_check.cpp with g++).
//
// The launch is a sequence of phases with a grid barrier after each: phase k is one
// round of the whole grid, or a stretch of rounds by a team while the other
// workgroups wait in the barrier.  At the start of a phase EVERY workgroup reads the
// phase's input and decides from it what the phase is, and nothing makes the team
// wait until the others have read: a workgroup may read at any time up to its
// arrival at the phase's barrier, when the team has done any number of rounds.  So
// no word that is read there may be written in the same phase:
//  - the input a grid phase left is read from the grid's counters.  They are
//    indexed by the phase, a round of the grid adds to those of k + 1 and clears
//    those of k + 2, and a stretch only clears k + 2; the counters of phase k are
//    next written in phase k + 1 (cleared) or k + 2 (added to), behind a barrier
//    that every workgroup reaches only after it has read them;
//  - the team's rounds count in counters of their own, indexed by the number of
//    team rounds so far (`j`), which nobody else reads;
//  - what a stretch left is read from its report, in one of two places by the
//    phase's parity, next written in phase k + 2;
//  - the words of the team's own barrier are read by the team alone.
// The SSSP's far counters, one per bucket and three in turn, are added to by both
// sides.  Bucket e's is read where the next step is a bucket step, which adds to
// e + 1's and clears e + 2's; the bucket step after it would clear e's, so a stretch
// that begins with a bucket step whose count was read from the counter ends before
// the second one, and the next stretch has the count from the report.
#pragma once

#include <stdint.h>

#if defined(__HIPCC__)
#define HS_ROUND_FN __host__ __device__ inline
#else
#define HS_ROUND_FN inline
#endif

namespace hs_rounds {

enum Side : uint32_t { kGrid = 0, kTeam = 12 };                // first slot of each side's counters
enum Counter : uint32_t { kLight = 0, kGrab = 3, kChunks = 6 };  // three of each
constexpr uint32_t kOther = 9;       // three more: the BFS's pull chunks by phase, the SSSP's far lists by bucket
constexpr uint32_t kReport = 21;     // two reports
constexpr uint32_t kTeamWords = 23;  // the words of the team's barrier, two slots
constexpr uint32_t kSlots = 25;

// counter of round i (a phase of the grid, or a team round j)
HS_ROUND_FN uint32_t slot(Side side, Counter c, uint32_t i) { return side + c + i % 3; }
HS_ROUND_FN uint32_t other(uint32_t i) { return kOther + i % 3; }
HS_ROUND_FN uint32_t report(uint32_t k) { return kReport + (k & 1); }

// Whether a launch has a team: some workgroups, at most kTeamMax, of a grid that has
// others, whose barrier gives up like the team's own waits do (an abort, the spin
// limit).  A cooperative grid sync does not: a team whose wait failed would leave the
// others in it for good.
constexpr uint32_t kTeamMax = 32;
HS_ROUND_FN bool team_usable(uint32_t size, uint32_t grid, bool bounded) {
  return bounded && size < grid && size <= kTeamMax;
}

// Edges of a round up to which a team of `size` workgroups runs it: 4096 for each, as
// the others stand still meanwhile.  A bound for the full team alone (2^17) left rounds
// of 8000 edges to 2 of 16 workgroups (mesh of 1.1M vertices, SSSP with 16: 51
// ms, 24 so, 37 without a team).
HS_ROUND_FN uint64_t team_edges(uint32_t size) { return 4096ull * size; }

// Whether a BFS pulls a level whose frontier has `ahead` of the graph's m edges, when
// `behind` were those of the levels before (both by the mean degree, which a frontier of
// hubs exceeds).  It has to be 1/8 of the edges left: any factor from 4 to 64 gives the
// same times at R-MAT 12..22; 2 costs 45% at R-MAT 22.  And as a pull looks at every
// vertex, whatever the frontier is, 1/16 of the vertices: the rounded-up mean degree
// runs out of edges before a mesh or a road network ends, and with the first rule alone
// a grid without a team then pulled every narrow level that was left.
HS_ROUND_FN bool pull_pays(uint64_t ahead, uint64_t behind, uint64_t m, uint64_t n) {
  return ahead * 8 > (m > behind ? m - behind : 0) && ahead * 16 > n;
}

// Rounds of a stretch, at most: the others poll once in 1.4 us meanwhile, and as many
// times as the arena's spin limit allows, so that small limits, under which every round
// of the grid succeeds, get short stretches (a round of a team takes 2-6 us on meshes
// and up to some 50).
HS_ROUND_FN uint32_t team_rounds(uint32_t spin_limit) {
  return spin_limit / 512 < 255 ? spin_limit / 512 + 1 : 256;
}

// the counters that round i of a side clears for the rounds after it
template <class Clear>
HS_ROUND_FN void open_round(Side side, uint32_t i, Clear clear) {
  clear(slot(side, kLight, i + 2));
  clear(slot(side, kChunks, i + 2));
  clear(slot(side, kGrab, i + 1));
}

}  // namespace hs_rounds
