// resplan_kinds.cpp -- launch shapes, shared memory and plans of the on-chip
// solvers (fortranfvcell_amd/csrc/fvc_resplan.h) for each of the four methods,
// under AddressSanitizer and UndefinedBehaviorSanitizer: what a shape promises
// fits a CU, and meshes numbered row by row have a plan up to 1,020,000 rows.
#include <cstdio>
#include <cstdlib>

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

// The plan that resident_prep's last block takes for rows of length S whose
// columns reach hx aside and H away; nb 0: none.
static ResPlan choose(int n, int H, int S, int hx, int kind, const ResShape &s) {
  const int rmax = kResThreads * s.rpt, hmax = res_max_halo(kind, s.rpt);
  const bool one_step = kind != kResBicgstab;
  ResPlan best{};
  bool any = res_strips(n, H, rmax, s.blocks, hmax, best), one = any && best.nb <= kResOneStep;
  for (int ntx = 1; ntx <= s.blocks; ++ntx) {
    ResPlan p{};
    if (!res_tiles(n, S, hx, ntx, rmax, s.blocks, hmax, p)) continue;
    one = one || p.nb <= kResOneStep;
    if (any && res_cost(best, one_step) <= res_cost(p, one_step)) continue;
    best = p;
    any = true;
  }
  if (any) {
    ++plans;
    CHECK(best.nb >= 1 && best.nb <= s.blocks && best.R <= rmax && best.nh <= hmax, "%d rows, method %d: limits", n, kind);
    CHECK(!one_step || !one || best.nb <= kResOneStep, "%d rows, method %d: %d blocks, 64 would do", n, kind, best.nb);
  }
  return best;
}

int main() {
  const int kinds[] = {kResPcg, kResBicgstab, kResMixedPcg, kResGmres};
  for (int kind : kinds) {
    for (int rpt = 1; rpt <= 8; rpt *= 2) {
      const int h = res_max_halo(kind, rpt);
      // static: GMRES' Hessenberg matrix, rotations and sums; all: 1 KB of reductions and state
      const size_t fixed = kind == kResGmres ? ((kResGmresK + 1) * kResGmresK + 5 * (kResGmresK + 3)) * sizeof(double) : 0;
      CHECK(h > 0 && h <= kResMaxHalo && res_lds_bytes(kind, rpt, h) + fixed <= kResLds, "LDS of method %d, %d rows", kind, rpt);
      CHECK(kResThreads * rpt + h <= 65536, "window slots of method %d, %d rows, are 16 bits", kind, rpt);
    }
    for (int cus : {8, 64, 104, 256, 304})
      for (long n = 1; n < 1200000; n += 1 + n / 50) {
        const ResShape s = resident_shape((int)n, cus, kind);
        if (s.rpt == 0) continue;
        CHECK(s.rpt == 1 || s.rpt == 2 || s.rpt == 4 || s.rpt == 8, "%ld rows: %d a thread", n, s.rpt);
        CHECK(s.blocks >= 1 && s.blocks <= kResMaxBlocks && s.blocks <= cus, "%ld rows: %d blocks", n, s.blocks);
        CHECK((long)s.blocks * s.rpt * kResThreads >= n, "%ld rows do not fit %d blocks of %d", n, s.blocks, s.rpt);
      }
    CHECK(resident_shape(1048576, 256, kind).rpt == 8 && resident_shape(1048577, 256, kind).rpt == 0, "the chip's limit");
    // quads of any aspect between 1/2 and 2, and squares cut into triangles
    for (int nx = 40; nx <= 1428; nx += 1 + nx / 23)
      for (int ny = nx / 2; ny <= 2 * nx; ny += 1 + ny / 17) {
        const int n = nx * ny;
        if (n > 1020000) continue;
        const ResShape s = resident_shape(n, 256, kind);
        CHECK(s.blocks == 1 || choose(n, nx, nx, 1, kind, s).nb > 0, "%d x %d quads, method %d: no plan", nx, ny, kind);
      }
    for (int m = 24; 2 * m * m <= 1020000; ++m) {
      const ResShape s = resident_shape(2 * m * m, 256, kind);
      CHECK(s.blocks == 1 || choose(2 * m * m, 2 * m - 1, 2 * m, 3, kind, s).nb > 0, "%d^2 triangles, method %d: no plan", m, kind);
    }
    CHECK(choose(1048576, 1024, 1024, 1, kind, resident_shape(1048576, 256, kind)).nb > 0, "1024^2 quads, method %d", kind);
  }
  std::printf("%d plans, %d failures\n", plans, failures);
  return failures != 0;
}
