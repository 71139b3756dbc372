// resplan_checks.cpp -- how the on-chip solvers deal rows to blocks
// (fortranfvcell_amd/csrc/fvc_resplan.h) under AddressSanitizer and
// UndefinedBehaviorSanitizer, against what the scheme promises: every row is
// held by one block, a window slot found for a column holds that column, and
// every halo row is one that its owner publishes.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../../fortranfvcell_amd/csrc/fvc_resplan.h"

using namespace fvc;

static int failures = 0, plans = 0;
#define CHECK(cond, ...)                                          \
  do {                                                            \
    if (!(cond)) {                                                \
      std::fprintf(stderr, "FAIL %s:%d: ", __FILE__, __LINE__);   \
      std::fprintf(stderr, __VA_ARGS__);                          \
      std::fprintf(stderr, "\n");                                 \
      if (++failures > 20) std::exit(1);                          \
    }                                                             \
  } while (0)

static void check_plan(const ResPlan &p, int n, int rmax, int bmax, int hmax) {
  ++plans;
  CHECK(p.nb >= 1 && p.nb <= bmax && p.R >= 1 && p.R <= rmax && p.nh >= 0 && p.nh <= hmax, "limits n=%d", n);
  std::vector<int> owner(n, -1), local(n, -1);
  std::vector<char> edge(n, 0);
  std::vector<ResMap> maps(p.nb);
  for (int c = 0; c < p.nb; ++c) {
    maps[c].init(p, n, c);
    for (int l = 0; l < rmax; ++l) {
      const int i = maps[c].own(l);
      if (i < 0) continue;
      CHECK(i < n && owner[i] < 0, "row %d held twice or out of range", i);
      owner[i] = c;
      local[i] = l;
      edge[i] = maps[c].edge(l);
    }
  }
  for (int i = 0; i < n; ++i) CHECK(owner[i] >= 0, "row %d of %d held by no block", i, n);
  for (int c = 0; c < p.nb; ++c) {
    const ResMap &m = maps[c];
    for (int h = 0; h < p.nh; ++h) {
      const int j = m.halo(h);
      if (j < 0) continue;
      CHECK(j < n && owner[j] != c, "halo %d of block %d is row %d, its own or none", h, c, j);
      CHECK(edge[j], "halo row %d is not published", j);
      CHECK(m.slot(j, rmax) == rmax + h, "halo row %d: slot %d, entry %d", j, m.slot(j, rmax), h);
    }
    // columns around the block's rows, and far ones
    for (int l = 0; l < rmax; l += 1 + l % 7) {
      const int i = m.own(l);
      if (i < 0) continue;
      CHECK(m.slot(i, rmax) == l, "own row %d", i);
      const int d[] = {1, 2, 3, 4, p.H, p.H - 1, p.H + 1, p.S, p.S + 1, p.S - 1, p.S + 3, p.S - 3, 2 * p.S, n / 2};
      for (int q : d)
        for (int s = -1; s <= 1; s += 2) {
          const long j = (long)i + s * (long)q;
          if (j < 0 || j >= n) continue;
          const int at = m.slot((int)j, rmax);
          if (at < 0) {
            if (!p.tile) CHECK(std::labs(s * (long)q) > p.H, "strip: column %ld of row %d lost", j, i);
            continue;
          }
          if (at < rmax) CHECK(m.own(at) == j, "slot %d is not column %ld", at, j);
          else CHECK(at - rmax < p.nh && m.halo(at - rmax) == j, "halo slot %d is not column %ld", at - rmax, j);
        }
    }
  }
}

// Every system that takes part has its team of blocks, the blocks' lists hold
// it once per block of the team, and going through the lists never waits in a
// ring.
static void check_batch(const std::vector<int> &neq, int cap) {
  const ResBatchPlan p = plan_resident_batch(neq, 1.5, cap);
  if (p.rpt == 0) return;
  ++plans;
  const int n = (int)neq.size();
  CHECK(p.blocks <= cap && p.blocks % 8 == 0 && (int)p.ptr.size() == p.blocks + 1, "%d blocks of %d", p.blocks, cap);
  std::vector<int> seen(n, 0), at(p.blocks);
  for (int b = 0; b < p.blocks; ++b) {
    at[b] = p.ptr[b];
    for (int k = p.ptr[b]; k < p.ptr[b + 1]; ++k) {
      const int i = p.list[k];
      CHECK(p.on[i] && b >= p.first[i] && b < p.first[i] + p.count[i], "block %d runs system %d of others", b, i);
      ++seen[i];
    }
  }
  int left = 0;
  for (int i = 0; i < n; ++i) {
    if (!p.on[i]) { CHECK(seen[i] == 0, "system %d", i); continue; }
    ++left;
    CHECK(seen[i] == p.count[i] && p.first[i] + p.count[i] <= p.blocks, "system %d: %d of %d blocks", i, seen[i], p.count[i]);
    CHECK((long)p.count[i] * p.rpt * kResThreads >= neq[i], "system %d does not fit its team", i);
  }
  for (bool moved = true; moved;) {
    moved = false;
    for (int b = 0; b < p.blocks; ++b) {
      if (at[b] >= p.ptr[b + 1]) continue;
      const int i = p.list[at[b]];
      if (p.first[i] != b) continue;
      bool ready = true;
      for (int k = b; k < b + p.count[i]; ++k) ready = ready && at[k] < p.ptr[k + 1] && p.list[at[k]] == i;
      if (!ready) continue;
      for (int k = b; k < b + p.count[i]; ++k) ++at[k];
      --left;
      moved = true;
    }
  }
  CHECK(left == 0, "%d systems wait for each other", left);
}

int main() {
  unsigned seed = 1;
  const auto rnd = [&] { return (seed = seed * 1664525u + 1013904223u) >> 8; };
  for (int t = 0; t < 60; ++t) {
    std::vector<int> neq(1 + rnd() % (t < 30 ? 40 : 400));
    for (int &v : neq) v = 1 + (int)std::pow(10.0, (rnd() % 1000) / 1000.0 * (t % 3 == 0 ? 3.0 : 5.7));
    for (int cap : {256, 304, 64, 8}) check_batch(neq, cap);
  }
  const int sizes[] = {9, 64, 513, 2047, 4096, 5003, 12707, 40000};
  for (int n : sizes)
    for (int rmax : {512, 1024, 4096})
      for (int bmax : {8, 40, 256}) {
        const int hmax = 1500;
        for (int H : {1, 2, 7, 30, 64, 131, 256, 700}) {
          ResPlan p{};
          p.H = H;
          if (H < n && res_strips(n, H, rmax, bmax, hmax, p)) check_plan(p, n, rmax, bmax, hmax);
          for (int ntx = 1; ntx <= 12; ntx += 1 + ntx / 4)
            for (int hx : {1, 3, 4}) {
              ResPlan q{};
              q.H = H;
              if (H < n && res_tiles(n, H, hx, ntx, rmax, bmax, hmax, q)) check_plan(q, n, rmax, bmax, hmax);
            }
        }
      }
  // the launch shape: enough room, and within the chip
  for (int cus : {4, 8, 64, 104, 256, 304})
    for (long n = 1; n < 3000000; n += 1 + n / 3) {
      const ResShape s = resident_shape((int)n, cus);
      if (s.rpt == 0) continue;
      CHECK(s.blocks >= 1 && s.blocks <= kResMaxBlocks && s.blocks <= cus + 0, "%ld rows: %d blocks", n, s.blocks);
      CHECK((long)s.blocks * s.rpt * kResThreads >= n, "%ld rows do not fit %d blocks of %d", n, s.blocks, s.rpt);
      CHECK(s.blocks == 1 || s.blocks % 8 == 0, "%d blocks", s.blocks);
    }
  for (int code = 1; code <= 2; ++code)
    for (int rpt = 1; rpt <= 8; rpt *= 2) {
      const int h = res_max_halo(code, rpt);
      CHECK(h >= 0 && h <= kResMaxHalo && res_lds_bytes(code, rpt, h) <= kResLds, "LDS of code %d rpt %d", code, rpt);
    }
  std::printf("%d plans, %d failures\n", plans, failures);
  return failures != 0;
}
