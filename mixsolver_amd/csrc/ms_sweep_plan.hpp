// ms_sweep_plan.hpp -- the steps of a level-scheduled sweep and the places of
// its packed entries (ms_levels.hip).  Host code without a device, so that it
// can be checked without one.
#pragma once
#include <algorithm>
#include <vector>

namespace ms {

constexpr int kSlice = 64;    // SELL slice height = one wavefront
constexpr int kSegThreads = 1024;   // workgroup of a run of narrow levels
constexpr int kNarrowRows = 2048;   // widest level such a run takes
constexpr int kPre = 4;        // most entries per row that a sweep fetches ahead (hexahedra 3, prisms 2-3)
constexpr int kTailSteps = 6;  // empty steps after a run's last, so that fetching ahead needs no bound

// One step of the workgroup that walks a run of narrow levels, or a wide
// level: rows [t0, t0 + n) of the level order, entry k of its lane t at
// base + k * stride + t, w entries at most; near: all neighbours of its rows
// are in the workgroup's ring (1), or not (0).  32 bytes, one scalar load.
struct alignas(32) SweepStep {
  int t0, n, w, near;
  long long base;
  int stride;
};

// Places between the entries k and k + 1 of a row: whole wavefronts, or the
// step's own rows where they are fewer (a chain's steps have one row, and
// rounding them up would take 64 times its entries).  Lanes beyond a step's
// rows load its last row's entries, so nothing past them is read.
constexpr int sweep_stride(int n) { return n < kSlice ? n : (n + kSlice - 1) & ~(kSlice - 1); }

// levels [l0, l1) of a sweep: a run of narrow ones, walked by one workgroup of
// `block` threads in steps [s0, s1) from position t0 on, or one wide level
struct LevSeg {
  int l0, l1;
  bool narrow;
  int s0 = 0, s1 = 0, t0 = 0, block = kSegThreads;
  SweepStep step{};   // a wide level's
};

struct SweepSteps {
  std::vector<SweepStep> st;
  int width = 0;       // entries per row of every step of a run (more: rows beyond the width fetched ahead exist)
  bool more = false;
  long long nent = 0;
};

// Steps of the levels lev (CSR over the level order's positions); width_of(t):
// entries of the row at position t.
template <class Width>
SweepSteps sweep_steps(const std::vector<int> &lev, std::vector<LevSeg> &segs, Width width_of) {
  SweepSteps S;
  int widest_row = 1;
  for (int t = 0; t < lev.back(); t++) widest_row = std::max(widest_row, width_of(t));
  S.width = std::min(widest_row, kPre);
  S.more = widest_row > kPre;
  auto add = [&](int t, int n, int least) {
    if (n >= kSlice) S.nent = (S.nent + kSlice - 1) / kSlice * kSlice;   // whole wavefronts load aligned
    SweepStep d{t, n, least, 0, S.nent, sweep_stride(n)};
    for (int i = 0; (S.more || least < S.width) && i < n; i++) d.w = std::max(d.w, width_of(t + i));
    S.nent += (long long)d.w * d.stride;
    S.st.push_back(d);
  };
  for (auto &g : segs) {
    g.s0 = (int)S.st.size();
    g.t0 = lev[g.l0];
    if (!g.narrow) {
      add(g.t0, lev[g.l1] - g.t0, 1);   // a launch of its own, as wide as its own rows
      g.s1 = (int)S.st.size();
      g.step = S.st.back();
      continue;
    }
    int widest = 1;
    for (int l = g.l0; l < g.l1; l++) widest = std::max(widest, lev[l + 1] - lev[l]);
    g.block = std::min(kSegThreads, (widest + kSlice - 1) / kSlice * kSlice);
    for (int l = g.l0; l < g.l1; l++)
      for (int t = lev[l]; t < lev[l + 1]; t += g.block) add(t, std::min(g.block, lev[l + 1] - t), S.width);
    g.s1 = (int)S.st.size();
    for (int i = 0; i < kTailSteps; i++) S.st.push_back(SweepStep{});
  }
  return S;
}

// Whether both directions' entries are worth their padding: a step is as wide
// as its longest row, so a few long rows among many short ones would take many
// times the matrix (nstore stored entries); such a pattern is swept from the
// matrix itself.  A million entries (12 MB) are always packed.
constexpr bool sweep_packs(long long nent, long long nstore) { return nent <= 3 * nstore + (1 << 20); }

}  // namespace ms
