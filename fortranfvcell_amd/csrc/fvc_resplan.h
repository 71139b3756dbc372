// fvc_resplan.h -- how a system's rows are dealt to the blocks of the on-chip
// solvers (fvc_resident.h): which rows a block holds, which rows of others it
// needs, and where in its window a column is found.  Free of HIP, so that it
// also builds with the CPU sanitizers (tests/sanitize).
#pragma once
#include <stddef.h>

#include <algorithm>
#include <cmath>
#include <vector>

#if defined(__HIPCC__)
#define FVC_HD __host__ __device__ __forceinline__
#else
#define FVC_HD inline
#endif

namespace fvc {

constexpr int kResThreads = 512;     // two waves per SIMD: 256 registers a thread
constexpr int kResMaxBlocks = 256;   // partial sums: up to four blocks per lane of a wave
constexpr int kResMaxHalo = 2048;    // halo rows of a block
constexpr int kResGroups = 16;       // groups of 16 blocks whose sums are added first
// The words of one buffer for the partial sums of nb blocks: a pair per
// (value, block) up to 64 blocks, beyond that one per (group, value, block of
// the group) and one per (receiving group, value, group).
constexpr int kResSums = 5, kResGroupSums = 16 * kResSums;
constexpr int res_part_half(int nb) { return nb <= 64 ? 2 * kResSums * 64 : 2 * 2 * kResGroups * kResGroupSums; }
constexpr int kResPartWords = 2 * res_part_half(kResMaxBlocks);

// How rows are dealt to blocks, decided on the device by resident_prep_kernel
// (the host never sees the columns of a resident system).
// Strips: block c owns rows [c R, (c+1) R); its halo is the H rows on either
// side.  Tiles: the rows seen as a grid of S columns (row = y S + x), block
// (tx, ty) owns W x T of it; its halo is the frame around the tile, one row
// above and below, hx columns left and right.
struct ResPlan {
  int nb;                  // blocks that take part; 0: not solvable this way
  int tile;                // 1 tiles, 0 strips
  int R;                   // rows per block
  int H;                   // largest |column - row|
  int S, W, T, hx, ntx;    // tiles
  int nh;                  // halo entries per block
  int ticket;              // prep: blocks that are done
  int pad[5];
};

// Where a block's rows and halo rows are.
struct ResMap {
  ResPlan p;
  int neq, c, x0, y0, ny;
  FVC_HD void init(const ResPlan &plan, int n, int block) {
    p = plan;
    neq = n;
    c = block;
    x0 = y0 = 0;
    ny = 1;
    if (p.tile) {
      ny = (neq + p.S - 1) / p.S;
      x0 = (c % p.ntx) * p.W;
      y0 = (c / p.ntx) * p.T;
    }
  }
  FVC_HD int at(int x, int y) const {
    if (x < 0 || x >= p.S || y < 0 || y >= ny) return -1;
    const long r = (long)y * p.S + x;
    return r < neq ? (int)r : -1;
  }
  // the global row of local row l, or -1
  FVC_HD int own(int l) const {
    if (l >= p.R) return -1;
    if (!p.tile) {
      const long r = (long)c * p.R + l;
      return r < neq ? (int)r : -1;
    }
    return at(x0 + l % p.W, y0 + l / p.W);
  }
  // does another block's halo hold local row l?
  FVC_HD bool edge(int l) const {
    if (!p.tile) return l < p.H || l >= p.R - p.H;
    const int lx = l % p.W, ly = l / p.W;
    return lx < p.hx || lx >= p.W - p.hx || ly == 0 || ly == p.T - 1;
  }
  // the global row of halo entry h, or -1
  FVC_HD int halo(int h) const {
    if (!p.tile) {
      const long r = h < p.H ? (long)c * p.R - p.H + h : (long)(c + 1) * p.R + (h - p.H);
      return r >= 0 && r < neq ? (int)r : -1;
    }
    const int wide = p.W + 2 * p.hx;
    if (h < wide) return at(x0 - p.hx + h, y0 - 1);
    h -= wide;
    if (h < wide) return at(x0 - p.hx + h, y0 + p.T);
    h -= wide;
    if (h < p.T * p.hx) return at(x0 - p.hx + h % p.hx, y0 + h / p.hx);
    h -= p.T * p.hx;
    return at(x0 + p.W + h % p.hx, y0 + h / p.hx);
  }
  // the window slot of column j: local rows first, halo entries from `base`
  // on; -1 where neither holds it
  FVC_HD int slot(int j, int base) const {
    if (!p.tile) {
      const long d = (long)j - (long)c * p.R;
      if (d >= 0 && d < p.R) return (int)d;
      if (d < 0 && d >= -p.H) return base + (int)(d + p.H);
      if (d >= p.R && d < p.R + p.H) return base + p.H + (int)(d - p.R);
      return -1;
    }
    const int y = j / p.S, lx = j - y * p.S - x0, ly = y - y0;
    const int wide = p.W + 2 * p.hx;
    if (lx >= -p.hx && lx < p.W + p.hx) {
      if (ly == -1) return base + lx + p.hx;
      if (ly == p.T) return base + wide + lx + p.hx;
      if (ly >= 0 && ly < p.T) {
        if (lx < 0) return base + 2 * wide + ly * p.hx + lx + p.hx;
        if (lx >= p.W) return base + 2 * wide + p.T * p.hx + ly * p.hx + lx - p.W;
        return ly * p.W + lx;
      }
    }
    return -1;
  }
};

// Tiles of ntx columns for rows of length S whose columns reach hx aside:
// false where they do not fit rmax rows a block, bmax blocks or hmax halo
// entries.
FVC_HD bool res_tiles(int n, int S, int hx, int ntx, int rmax, int bmax, int hmax, ResPlan &p) {
  if (hx > 4 || S < 8 || ntx < 1 || ntx > S / 8 || ntx > bmax) return false;
  const int ny = (n + S - 1) / S, W = (S + ntx - 1) / ntx;
  if (W > rmax) return false;
  const int t0 = rmax / W, nty = (ny + t0 - 1) / t0;
  if ((long)ntx * nty > bmax) return false;
  const int T = (ny + nty - 1) / nty;
  p.nb = ntx * nty;
  p.tile = 1;
  p.R = W * T;
  p.S = S;
  p.W = W;
  p.T = T;
  p.hx = hx;
  p.ntx = ntx;
  p.nh = 2 * (W + 2 * hx) + 2 * hx * T;
  return p.nh <= hmax;
}

// Which of two plans is taken: where one_step is asked for, the one of at most
// kResOneStep blocks, then the one of fewer halo entries (253 x 257 rows: 2.6 us
// per PCG iteration in 64 strips of 514 halo entries, 3.1 in 72 tiles of 134).
constexpr int kResOneStep = 64;   // blocks up to which the sums are added in one step
FVC_HD int res_cost(const ResPlan &p, bool one_step) {
  return (one_step && p.nb > kResOneStep ? 2 * kResMaxHalo : 0) + p.nh;
}

// Strips of rmax rows for columns up to H rows away.
FVC_HD bool res_strips(int n, int H, int rmax, int bmax, int hmax, ResPlan &p) {
  const int nb = (int)(((long)n + rmax - 1) / rmax);
  if (nb > bmax || 2L * H > hmax) return false;
  p.nb = nb;
  p.tile = 0;
  p.R = rmax;
  p.nh = 2 * H;
  return true;
}

// The solvers held on chip.
constexpr int kResPcg = 1, kResBicgstab = 2, kResMixedPcg = 3, kResGmres = 4;

// The blocks' shared memory: the operand window (own rows, then halo
// entries), x and the shadow residual (read once per iteration; the other
// vectors are in registers, which these two would overflow at eight rows a
// thread), the halo rows' vectors, and both kinds' global row numbers.
// Mixed precision: the window (doubles at the FP64 updates), three floats a
// halo row; x stays in memory.  GMRES: the window, x, and the Hessenberg
// matrix of up to kResGmresK columns, static.
constexpr int kResGmresK = 32;
constexpr int res_halo_vecs(int code) { return code == kResBicgstab ? 5 : 4; }
constexpr int res_own_vecs(int code) { return code == kResBicgstab ? 2 : 1; }
constexpr size_t res_own_bytes(int code) {
  return code == kResMixedPcg ? sizeof(double) + sizeof(int) : (1 + res_own_vecs(code)) * sizeof(double) + sizeof(int);
}
constexpr size_t res_halo_bytes(int code) {
  return code == kResGmres      ? sizeof(double) + sizeof(int)
         : code == kResMixedPcg ? sizeof(double) + 3 * sizeof(float) + sizeof(int)
                                : (1 + res_halo_vecs(code)) * sizeof(double) + sizeof(int);
}
constexpr size_t res_lds_bytes(int code, int rpt, int nh) {
  return (size_t)kResThreads * rpt * res_own_bytes(code) + (size_t)nh * res_halo_bytes(code);
}
constexpr size_t kResLds = 156 * 1024;   // of a CU's 160 KB, less the reductions' static part
// the halo entries that fit beside rpt rows per thread
constexpr int res_max_halo(int code, int rpt) {
  const size_t fixed = code == kResGmres ? ((kResGmresK + 1) * kResGmresK + 5 * (kResGmresK + 3)) * sizeof(double) : 0;
  const size_t left = kResLds - fixed - res_lds_bytes(code, rpt, 0);
  const size_t nh = left / res_halo_bytes(code);
  return nh < (size_t)kResMaxHalo ? (int)nh : kResMaxHalo;
}

// Rows per thread and blocks at most for neq rows on `cus` compute units;
// rpt 0: the system does not fit the chip.  Measured on MI355X (us per
// iteration, PCG / BiCGSTAB):
//   * one block needs no exchange: 2,025 rows 1.7 / 3.1 against 2.2 / 4.2 on
//     8 blocks; 4,096 rows 2.5 / 5.4 against 2.1 / 4.2, so one block up to
//     2,048 rows;
//   * then one row a thread while 52 blocks hold them (64 with the sixth more
//     that tiles need): 12,707 rows 2.1 / 4.2 against 2.3 / 4.7 at two, but
//     32,300 rows 2.4 / 5.0 either way, and GMRES on 26,895 rows 2.59 ms a solve
//     on 64 blocks against 2.50 on 32;
//   * up to 64 blocks the sums need one step instead of two: 59,713 rows 2.5 /
//     5.2 on 64 blocks of 1,024 against 3.1 / 6.1 on 72, 65,160 rows 2.6 / 5.4
//     against 3.1 / 6.1 on 80 (GMRES 3.73 -> 2.83 ms a solve, mixed PCG 8.4 ->
//     7.5), so two rows a thread as long as 64 blocks hold them, and for PCG
//     four: 81,200 rows 2.8 against 3.1 at two, 127,800 rows 2.9 against 3.1
//     (BiCGSTAB 6.1 against 6.0, 6.5 against 6.1).  More blocks than 64 are
//     launched for plans that need them; res_cost prefers the others.
//     BiCGSTAB stays with the plan of least halo from 53,248 rows on, at a price
//     (59,713 rows 0.33 ms a solve against 0.29 on 64 blocks).  Its count of
//     iterations moves with the order of the sums, and on the one system where
//     it is held to the reference's, 65,536 rows of steady transport, 5,096
//     iterations within 3 %, it is 5,143 with this plan and 5,445 on 64 blocks.
//     One system does not show that either plan needs fewer in general;
//   * beyond, the fewest rows per thread: 160,860 rows 3.1 / 6.1 at 2, 3.5 / 7.0
//     at 4, 3.9 / 8.5 at 8 -- as long as a twentieth of the rows stays free for
//     tiles that the mesh's edge cuts (524,176 rows in strips at 4 took half as
//     long again as in tiles at 8).
struct ResShape {
  int rpt, blocks;
};
inline ResShape resident_shape(int neq, int cus, int kind = kResPcg) {
  const long n = neq, most = (cus < kResMaxBlocks ? cus : kResMaxBlocks) & ~7;
  for (int rpt = 1; rpt <= 4; rpt *= 2)
    if (n <= (long)kResThreads * rpt) return {rpt, 1};
  if (most < 8) return {0, 0};
  auto blocks = [&](int rpt) {   // a sixth more than full ones
    const long nb = (n + (long)kResThreads * rpt - 1) / ((long)kResThreads * rpt);
    const long want = (nb + nb / 6 + 8) & ~7L;
    return (int)(want < most ? want : most);
  };
  for (int rpt = 1; rpt <= (kind == kResPcg ? 4 : 2); rpt *= 2) {
    const long few = rpt == 1 || kind == kResBicgstab ? 52 : kResOneStep;
    if (n <= (long)kResThreads * rpt * (most < few ? most : few)) return {rpt, blocks(rpt)};
  }
  for (int rpt = 2; rpt <= 8; rpt *= 2) {
    const long room = (long)kResThreads * rpt * most;
    if (n <= (rpt < 8 ? room - room / 20 : room)) return {rpt, blocks(rpt)};
  }
  return {0, 0};
}

// ---------------------------------------------------------------- batches --
//
// Teams of blocks for a batch: how many rows a thread holds (one choice for
// the launch), each system's team, and each block's systems in turn.
struct ResBatchPlan {
  int rpt = 0, blocks = 0;             // rpt 0: nothing to gain
  std::vector<char> on;                // per system: solved by this launch
  std::vector<int> first, count;       // its team
  std::vector<int> ptr, list;          // block b runs list[ptr[b]] .. list[ptr[b + 1] - 1] in this order
  double load = 0.0;                   // the most loaded block, us per unit of iterations
};

// us per PCG iteration at 1, 2, 4, 8 rows a thread, one full block and a team
// (MI355X)
constexpr double kResIterAlone[4] = {1.3, 1.3, 1.7, 2.5}, kResIterTeam[4] = {2.1, 2.3, 2.7, 3.8};

// blocks: co-resident ones.  A system's iterations are taken as
// neq^(expo - 1) (PCG on these meshes: expo 1.5), its time as iterations
// times the time of one, which hardly falls with more blocks: so a team is
// as small as holds the system, and the rows per thread are those whose most
// loaded block ends first: few systems want few rows a thread (short
// iterations), many want eight (a third of the block time of one row).
// Systems go longest first onto the run of blocks that is free first; runs
// may start anywhere (256 systems of side 32 .. 512: 1.15 times the mean
// load against 1.41 with runs at multiples of the team).
inline ResBatchPlan plan_resident_batch(const std::vector<int> &neq, double expo, int blocks) {
  const int n = (int)neq.size();
  ResBatchPlan best;
  blocks = (blocks < kResMaxBlocks ? blocks : kResMaxBlocks) & ~7;
  if (blocks < 8) return best;
  std::vector<double> its(n), cost(n), load;
  std::vector<int> order, count(n), first(n), run;
  for (int i = 0; i < n; ++i) its[i] = std::pow((double)neq[i], expo - 1.0);
  for (int q = 0; q < 4; ++q) {
    double total = 0.0;
    bool all = true;
    order.clear();
    for (int i = 0; i < n; ++i) {
      const long g = ((long)neq[i] + (kResThreads << q) - 1) / (kResThreads << q);
      count[i] = g <= blocks ? (int)g : 0;
      all = all && count[i] > 0;
      if (!count[i]) continue;
      cost[i] = its[i] * (g > 1 ? kResIterTeam[q] : kResIterAlone[q]);
      total += g * cost[i];
      order.push_back(i);
    }
    // (at eight rows a thread, systems that do not fit are left out)
    if (order.empty() || (!all && q < 3) || (best.rpt && total / blocks >= best.load)) continue;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return cost[a] > cost[b]; });
    load.assign(blocks, 0.0);
    double longest = 0.0;
    for (int i : order) {
      // the run of count[i] blocks whose largest load is least: the largest
      // load of every run by a queue of candidates
      const int g = count[i];
      int at = 0;
      double when = -1.0;
      run.clear();
      size_t head = 0;
      for (int k = 0; k < blocks; ++k) {
        while (run.size() > head && load[run.back()] <= load[k]) run.pop_back();
        run.push_back(k);
        if (run[head] <= k - g) ++head;
        if (k + 1 >= g && (when < 0.0 || load[run[head]] < when)) {
          when = load[run[head]];
          at = k + 1 - g;
        }
      }
      first[i] = at;
      for (int k = at; k < at + g; ++k) load[k] = when + cost[i];
      longest = longest < when + cost[i] ? when + cost[i] : longest;
    }
    if (best.rpt && longest >= best.load) continue;
    best.rpt = 1 << q;
    best.load = longest;
    best.first = first;
    best.count = count;
    best.list = order;
  }
  if (!best.rpt) return best;
  best.on.assign(n, 0);
  std::vector<std::vector<int>> lists(blocks);
  int used = 0;
  for (int i : best.list) {
    best.on[i] = 1;
    used = used < best.first[i] + best.count[i] ? best.first[i] + best.count[i] : used;
    for (int k = best.first[i]; k < best.first[i] + best.count[i]; ++k) lists[k].push_back(i);
  }
  best.blocks = (used + 7) & ~7;
  best.list.clear();
  best.ptr.assign(1, 0);
  for (int k = 0; k < best.blocks; ++k) {
    best.list.insert(best.list.end(), lists[k].begin(), lists[k].end());
    best.ptr.push_back((int)best.list.size());
  }
  return best;
}

}  // namespace fvc
