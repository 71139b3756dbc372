// fvc_resplan.h -- how a system's rows are dealt to the blocks of the on-chip
// solvers (fvc_resident.h): which rows a block holds, which rows of others it
// needs, and where in its window a column is found.  Free of HIP, so that it
// also builds with the CPU sanitizers (tests/sanitize).
#pragma once
#include <stddef.h>

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
// two buffers of either a word pair per (value, block), or one per (group,
// value, block of the group) and one per (receiving group, value, group)
constexpr int kResPartWords = 2 * 2 * 2 * kResGroups * 64;

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

// The blocks' shared memory: the operand window (own rows, then halo
// entries), x and the shadow residual (read once per iteration; the other
// vectors are in registers, which these two would overflow at eight rows a
// thread), the halo rows' vectors, and both kinds' global row numbers.
constexpr int res_halo_vecs(int code) { return code == 1 ? 4 : 5; }
constexpr int res_own_vecs(int code) { return code == 1 ? 1 : 2; }
constexpr size_t res_lds_bytes(int code, int rpt, int nh) {
  return (size_t)kResThreads * rpt * ((1 + res_own_vecs(code)) * sizeof(double) + sizeof(int)) +
         (size_t)nh * ((1 + res_halo_vecs(code)) * sizeof(double) + sizeof(int));
}
constexpr size_t kResLds = 156 * 1024;   // of a CU's 160 KB, less the reductions' static part
// the halo entries that fit beside rpt rows per thread
constexpr int res_max_halo(int code, int rpt) {
  const size_t left = kResLds - res_lds_bytes(code, rpt, 0);
  const size_t nh = left / ((1 + res_halo_vecs(code)) * sizeof(double) + sizeof(int));
  return nh < (size_t)kResMaxHalo ? (int)nh : kResMaxHalo;
}

// Rows per thread and blocks at most for neq rows on `cus` compute units;
// rpt 0: the system does not fit the chip.  Measured on MI355X (us per
// iteration, PCG / BiCGSTAB):
//   * one block needs no exchange: 2,025 rows 1.9 / 4.0 against 2.6 / 5.1 on
//     8 blocks; 4,095 rows 2.8 / 5.9 against 2.6 / 5.2, so one block up to
//     2,048 rows;
//   * up to 64 blocks the sums need one step instead of two: 32,300 rows 3.2
//     on 40 blocks of 1,024 against 3.7 on 80 of 512, but 65,536 rows 3.6
//     either on 80 of 1,024 or 40 of 2,048, so two rows a thread at most for
//     that;
//   * beyond, the fewest rows per thread: 262,144 rows 4.6 at 2, 4.8 at 4,
//     5.5 at 8 -- as long as a twentieth of the rows stays free for tiles that
//     the mesh's edge cuts (524,176 rows 8.1 in strips at 4, 5.6 in tiles at 8).
struct ResShape {
  int rpt, blocks;
};
inline ResShape resident_shape(int neq, int cus) {
  const long n = neq, most = (cus < kResMaxBlocks ? cus : kResMaxBlocks) & ~7;
  for (int rpt = 1; rpt <= 4; rpt *= 2)
    if (n <= (long)kResThreads * rpt) return {rpt, 1};
  if (most < 8) return {0, 0};
  auto blocks = [&](int rpt) {   // a sixth more than full ones
    const long nb = (n + (long)kResThreads * rpt - 1) / ((long)kResThreads * rpt);
    const long want = (nb + nb / 6 + 8) & ~7L;
    return (int)(want < most ? want : most);
  };
  for (int rpt = 1; rpt <= 2; rpt *= 2)
    if (n <= (long)kResThreads * rpt * (most < 52 ? most : 52) && blocks(rpt) <= 64) return {rpt, blocks(rpt)};
  for (int rpt = 2; rpt <= 8; rpt *= 2) {
    const long room = (long)kResThreads * rpt * most;
    if (n <= (rpt < 8 ? room - room / 20 : room)) return {rpt, blocks(rpt)};
  }
  return {0, 0};
}

}  // namespace fvc
