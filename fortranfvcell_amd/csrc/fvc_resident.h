// fvc_resident.h -- PCG, BiCGSTAB, mixed PCG and GMRES with the whole system
// held on chip (of GMRES, all but the basis).
//
// One launch solves the system: every block loads its rows' matrix entries
// once into registers and keeps its rows of every Krylov vector there too
// (256 CUs hold 128 MB of registers; a row of a 4-neighbour system with its
// six vectors takes about 100 bytes), so that an iteration reads neither the
// matrix nor a vector from memory.  (At eight rows a thread the 256 registers of
// a lane do not hold everything: up to 204 bytes of scratch a lane, BiCGSTAB at
// width 4.  With the exchanges' words it moves 15 MB an iteration past L2 at
// 1,048,576 rows, streamed 243; PCG on 160,000 rows, two a thread and no scratch,
// 1.8 MB, streamed 22.)  What an iteration waits for is the exchange between
// blocks, once per grid reduction:
//   * the SpMV reads its operand from an LDS window of the block's own rows
//     and of the halo rows its columns reach.  A halo row's operand is not
//     sent: its r, s, p ... follow the same recurrences as the owner's, on
//     the same values, so only the result of the previous SpMV at that row
//     has to arrive, and it travels together with the reduction;
//   * a block's partial sums go to all blocks, and every block adds all of
//     them in the same order and runs the scalar recurrence itself.
// Both travel as 8-byte words that carry half a double and the number of the
// exchange, stored and loaded at agent scope (past the caches that are not
// coherent between XCDs): a reader polls the data itself, so an exchange is
// one store and one load away, with no fence, no flag and no cache
// write-back.  Two buffers alternate; a block can run at most one exchange
// ahead of any other (it needs every block's partial sums), so a word is
// never overwritten before it was read.
//
// Measured on MI355X (us per PCG iteration, one exchange each): 1.1 in one
// block of 400 rows, 2.1 at 5,120 rows (10 blocks), 2.4 at 32,300 (40), 3.1 at
// 160,860 (168), 4.9 at 1,048,576 (256); a launch per phase costs 9 us at 4,096
// rows and 26-30 us at a million.  An iteration of one block is a chain of
// latencies (LDS, barriers, quotients), one of many adds the flight of its words,
// twice beyond 64 blocks; with 1,024 halo rows a side instead of 256 the flight
// was twice as long.  The halo volume is
// what makes the difference at 256 blocks, so rows are dealt in tiles of the
// mesh where the columns show one (ResPlan), else in contiguous strips.
#pragma once
#include <limits.h>
#include <stddef.h>

#include <type_traits>

#include "fvc_batch.h"
#include "fvc_krylov.h"
#include "fvc_resplan.h"

namespace fvc {

// Polls of a bounded wait: about 0.4 s.  The first exchange of a solve is also
// where its blocks wait until all of them have a CU, and some may not get one
// for as long as another stream's kernel runs; the engine that streams needs no
// such thing, so that wait is given up after about 3 ms, what that engine takes
// for BiCGSTAB on 1,048,576 rows.  Beside a kernel of one wave that runs 0.8 s, such a
// solve takes 6.4 ms (394 with the full wait), 3.2 if it streams at once.
constexpr unsigned kResSpin = 1u << 20, kResFirst = 1u << 13;

typedef unsigned long long res_word;

// KState::pad6 after a launch: solved, or the system does not fit this scheme
// (solve it another way).  Anything else, or the err word set: a wait expired.
constexpr int kResSolved = 1, kResDeclined = 2;

// ------------------------------------------------------------------- prep --

struct ResPrepArgs {
  Mat A;
  ResPlan *plan;           // zeroed
  res_word *part, *rows;   // cleared here: nparts and 4 neq words
  int nparts;
  int rmax, bmax, hmax;    // rows per block, blocks and halo entries at most
  int one_step;            // prefer plans of at most kResOneStep blocks
  const double *x;         // copied to keep (neq), the start vector of a solve that
  double *keep;            // must be done again; null: not asked for
};

// The columns of row i that count: off-diagonal entries other than
// ELLPACK's padding (column 1 with value 0).
template <int F, class Fn>
__device__ __forceinline__ void res_columns(const Mat &A, int i, Fn &&fn) {
  if constexpr (F == F_CSRD) {
    for (int k = A.ia[i] - 1; k < A.ia[i + 1] - 1; ++k) fn(A.ja[k] - 1);
  } else {
    constexpr int w = F == F_ELL3 ? 3 : 4;
#pragma unroll
    for (int k = 0; k < w; ++k) {
      const int j = A.ja[(size_t)w * i + k] - 1;
      if (j != 0 || A.av[(size_t)w * i + k] != 0.0) fn(j);
    }
  }
}

// Clears the exchange words, finds the largest |column - row|, and (its last
// block) decides how the rows are dealt.  One pass over the columns by
// gridDim.x blocks.
template <int F>
__device__ __forceinline__ void resident_prep(const ResPrepArgs &a) {
  __shared__ int s_h, s_last, s_best, s_hx[2];
  const int n = a.A.neq, step = (int)(gridDim.x * blockDim.x);
  if (threadIdx.x == 0) s_h = 0;
  __syncthreads();
  const int first = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  for (size_t k = first; k < (size_t)4 * n; k += (size_t)step) a.rows[k] = 0ull;
  for (int k = first; k < a.nparts; k += step) a.part[k] = 0ull;
  if (a.keep)
    for (long i = first; i < n; i += step) a.keep[i] = a.x[i];
  int h = 0;
  for (long i = first; i < n; i += step) {
    res_columns<F>(a.A, (int)i, [&](int j) { h = max(h, abs(j - (int)i)); });
    if (F == F_CSRD && a.A.ia[i + 1] - a.A.ia[i] > 4) h = n;   // longer rows do not fit the registers
  }
  atomicMax(&s_h, h);
  __syncthreads();
  if (threadIdx.x == 0) {
    atomicMax(&a.plan->H, s_h);
    fence_release();
    s_last = __hip_atomic_fetch_add(&a.plan->ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
             (int)gridDim.x;
    fence_acquire();
    s_hx[0] = s_hx[1] = 0;
    s_best = INT_MAX;
  }
  __syncthreads();
  if (!s_last) return;
  const int H = __hip_atomic_load(&a.plan->H, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (H >= n) return;   // a row too long, or nothing to gain: nb stays 0
  // A structured numbering shows a row length S of H (quads: the north and
  // south neighbours) or H + 1 (triangles split from quads): every offset is
  // then a row up or down and a few columns aside, and none wraps around an
  // end of the row.  Looked for on 512 rows spread over the system and, for
  // each S, on the four rows at either end of 32 of its rows, where the wrong S
  // wraps (1,024 rows spread out missed that on one in twenty of the meshes of
  // 2 n^2 triangles, n = 24 .. 700: 307,328 rows solved by BiCGSTAB one kernel per
  // phase, 1.62 ms, instead of on chip); the solve checks every column
  // against its window and declines otherwise.
  const int ns = min(n, 512);
  int worst[2] = {0, 0};
  auto look = [&](int i, int s) {
    const int S = max(H + s, 1), yi = i / S;
    res_columns<F>(a.A, i, [&](int j) {
      const int yj = j / S;
      const int dy = yj - yi, dx = abs((j - yj * S) - (i - yi * S));
      worst[s] = max(worst[s], abs(dy) > 1 ? n : dx);
    });
  };
  for (int q = threadIdx.x; q < ns; q += blockDim.x) {
    const int i = (int)((long)q * n / ns);
    look(i, 0);
    look(i, 1);
  }
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int S = max(H + s, 1);
    for (int q = threadIdx.x; q < 256; q += blockDim.x) {
      const int e = q & 7;
      const long i = (long)(q >> 3) * (n / S) / 32 * S + (e < 4 ? e : S - 8 + e);
      if (i >= 0 && i < n) look((int)i, s);
    }
  }
#pragma unroll
  for (int s = 0; s < 2; ++s)
    if (worst[s] > 0) atomicMax(&s_hx[s], worst[s]);
  __syncthreads();
  // thread t tries t / 2 + 1 columns of tiles over the row lengths H and
  // H + 1 in turn; the least cost wins
  auto tiles = [&](int q, ResPlan &p) {
    return res_tiles(n, H + (q & 1), max(s_hx[q & 1], 1), (q >> 1) + 1, a.rmax, a.bmax, a.hmax, p);
  };
  for (int q = threadIdx.x; q < 2 * min(a.bmax, kResMaxBlocks); q += blockDim.x) {
    ResPlan p{};
    if (tiles(q, p)) atomicMin(&s_best, (res_cost(p, a.one_step) << 10) | q);
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  ResPlan p{};
  const bool strips = res_strips(n, H, a.rmax, a.bmax, a.hmax, p);
  if (s_best < INT_MAX && !(strips && res_cost(p, a.one_step) <= (s_best >> 10))) tiles(s_best & 1023, p);
  p.H = H;
  p.ticket = (int)gridDim.x;
  *a.plan = p;
}

template <int F>
__global__ __launch_bounds__(256) void resident_prep_kernel(ResPrepArgs a) {
  resident_prep<F>(a);
}

// --------------------------------------------------------------- exchange --

__device__ __forceinline__ res_word res_load(const res_word *p) {
  return __hip_atomic_load(const_cast<res_word *>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_store(res_word *p, res_word v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A double as two words, `apart` from each other: the exchange's number in the
// low half, half of the double in the high one.  Sums keep their low halves
// together and their high halves together, so that a wave's load of either is
// of whole lines (half as many lines to a look: 4 % of a PCG iteration at 160
// blocks and above); a row's two words are neighbours, for a tile's columns are
// published row by row.
__device__ __forceinline__ void res_put(res_word *p, size_t apart, double v, unsigned ep) {
  const res_word u = __builtin_bit_cast(res_word, v);
  res_store(p, (u << 32) | ep);
  res_store(p + apart, (u & 0xffffffff00000000ull) | ep);
}
__device__ __forceinline__ double res_get(res_word lo, res_word hi) {
  return __builtin_bit_cast(double, (hi & 0xffffffff00000000ull) | (lo >> 32));
}

// Sums over a wavefront in the ALU's data path (row shifts by DPP, swaps of
// halves and of rows) instead of the shuffles' trips through LDS.  Two waves
// share a SIMD, so the sums of every wave at once are bound by instructions: K
// values one by one take 6 K steps of three, while a swap halves the lanes of
// two values at the price of one, and up to four values are one after two
// swaps: 7 steps instead of 18 or 24.
template <int Ctrl>
__device__ __forceinline__ double res_dpp_add(double v) {
  const res_word u = __builtin_bit_cast(res_word, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, Ctrl, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), Ctrl, 0xF, 0xF, true);
  return v + __builtin_bit_cast(double, ((res_word)(unsigned)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double res_row_sum(double v) {   // of each 16 lanes, in the last
  v = res_dpp_add<0x111>(v);   // row_shr:1
  v = res_dpp_add<0x112>(v);   // row_shr:2
  v = res_dpp_add<0x114>(v);   // row_shr:4
  return res_dpp_add<0x118>(v);   // row_shr:8
}
// a's halves (rows) added in the lower half (even rows), b's in the other
template <bool Halves>
__device__ __forceinline__ double res_fold(double a, double b) {
  const res_word u = __builtin_bit_cast(res_word, a), w = __builtin_bit_cast(res_word, b);
  const auto swap = [](unsigned x, unsigned y) {
    if constexpr (Halves) return __builtin_amdgcn_permlane32_swap(x, y, false, false);
    else return __builtin_amdgcn_permlane16_swap(x, y, false, false);
  };
  const auto lo = swap((unsigned)u, (unsigned)w), hi = swap((unsigned)(u >> 32), (unsigned)(w >> 32));
  return __builtin_bit_cast(double, ((res_word)hi[0] << 32) | lo[0]) +
         __builtin_bit_cast(double, ((res_word)hi[1] << 32) | lo[1]);
}
// The sums of K <= 4 values: value k in the last lane of row res_sum_row<K>(k).
template <int K>
__device__ __forceinline__ constexpr int res_sum_row(int k) { return K == 1 ? 3 - k : ((k & 1) << 1) | (k >> 1); }
template <int K>
__device__ __forceinline__ double res_wave_sums(const double *v) {
  if constexpr (K == 1) {
    const double r = res_dpp_add<0x142>(res_row_sum(v[0]));   // row_bcast:15: two rows in the last lane of row 3, and of row 1,
    return res_dpp_add<0x143>(r);                             // which row_bcast:31 takes there
  }
  const double a = res_fold<true>(v[0], K > 1 ? v[K > 1 ? 1 : 0] : 0.0);
  const double b = K > 2 ? res_fold<true>(v[K > 2 ? 2 : 0], K > 3 ? v[K > 3 ? 3 : 0] : 0.0) : 0.0;
  return res_row_sum(res_fold<false>(a, b));
}
__device__ __forceinline__ double res_lane(double v, int lane) {
  const res_word u = __builtin_bit_cast(res_word, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, lane);
  const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), lane);
  return __builtin_bit_cast(double, ((res_word)hi << 32) | lo);
}

// How long a wave sleeps, in units of 64 cycles, before it looks for the first
// time: a look takes about as long as a word takes to arrive, so one that comes
// too early costs a second one and slows the words of others.  The sums of a
// flat exchange or of a group and the halo's rows are one word's flight away,
// the group totals two.  PCG, us per iteration, without any and with these:
// 32,300 rows (40 blocks) 2.73 / 2.41, 160,860 (168) 3.44 / 3.07, 429,713 (224)
// 4.21 / 3.69, 1,048,576 (256) 5.39 / 4.97; four units more or less at any of
// them changes that by up to 3 %.
constexpr int kResNapSums = 10, kResNapGroup = 8, kResNapRows = 14, kResNapTotals = 46;

// Waits for up to E doubles (or floats, a word each), at(q) being the address
// of the q-th's low half or null, the other half `apart` words on; all loads of
// a poll are issued together.  False if the wait expired, after `limit` polls
// or when another wait did (*err).
template <int Nap, int E, class T, class At>
__device__ __forceinline__ bool res_wait(unsigned ep, T *v, size_t apart, unsigned limit, const unsigned *err, At &&at) {
  res_word lo[E], hi[E];
  __builtin_amdgcn_s_sleep(Nap);
  for (unsigned spins = 0;;) {
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const res_word *p = at(q);
      lo[q] = hi[q] = ep;
      if (p) {
        lo[q] = res_load(p);
        if constexpr (sizeof(T) == 8) hi[q] = res_load(p + apart);
      }
    }
    bool ok = true;
#pragma unroll
    for (int q = 0; q < E; ++q) ok = ok && (unsigned)lo[q] == ep && (unsigned)hi[q] == ep;
    if (ok) break;
    if (++spins > limit) return false;
    if (spins >= 1024u) {   // somebody is late: leave the memory to them
      __builtin_amdgcn_s_sleep(8);
      if ((spins & 1023u) == 0u && ld_relaxed(const_cast<unsigned *>(err)) != 0u) return false;
    }
  }
#pragma unroll
  for (int q = 0; q < E; ++q) {
    if constexpr (sizeof(T) == 8) v[q] = res_get(lo[q], hi[q]);
    else v[q] = __builtin_bit_cast(float, (unsigned)(lo[q] >> 32));
  }
  return true;
}

struct ResArgs {
  Mat A;
  const ResPlan *plan;     // null: one block holds the system
  KState *st;              // written by block 0 at the end: pad6 is a kRes* outcome
  const double *m;         // Jacobi diagonal
  double *x;
  const double *b;
  res_word *rows;          // 2 buffers of 2 neq words
  res_word *part;          // two buffers of part_half words
  unsigned *err;           // set when a wait expired; the waits of others end too
  int part_half;
  unsigned first;          // polls that the first exchange may take
  unsigned strict;         // from this exchange on a wait ends after one look (tests)
  double tol;
  double delta;            // mixed: residual drop that triggers an FP64 update
  int max_inner;           // mixed: FP32 iterations between updates, at most
  double *gv;              // GMRES: basis columns 1 .. k, own rows only, ld apart
  size_t ld;
  int k;
  int maxit, x0_zero, stop_rule;
};

// A block's place among the others and its exchanges with them.
struct ResNet {
  static constexpr int NT = kResThreads;
  static constexpr int HE = 3;   // halo entries a thread waits for at once

  const ResArgs &a;
  ResMap map;
  int *row;                // LDS: global row of each own row, or -1
  int *hrow;               // LDS: global row of each halo entry, or -1
  double *red;             // LDS: kMaxK * kMaxWaves
  KState *S;               // LDS
  int *bad;                // LDS
  int nh, nb;
  unsigned ep = 0;
  unsigned pub = 0;        // bit k: another block reads the thread's row k
  double sc[3];            // alpha, beta, omega of the last exchange that read them
  int done = 0;

  __device__ __forceinline__ ResNet(const ResArgs &args) : a(args) {}

  // The words of the rows in one buffer: a pair per double, one per float.
  template <class T>
  __device__ __forceinline__ res_word *row_words(unsigned e, int j) const {
    return a.rows + (size_t)(e & 1) * 2 * a.A.neq + (sizeof(T) / 4) * (size_t)j;
  }
  template <class T>
  __device__ __forceinline__ void publish(int k, T v) const {
    if (!(pub >> k & 1u)) return;
    res_word *to = row_words<T>(ep + 1, row[threadIdx.x + k * NT]);
    if constexpr (sizeof(T) == 8) res_put(to, 1, v, ep + 1);
    else res_store(to, ((res_word)__builtin_bit_cast(unsigned, v) << 32) | (ep + 1));
  }

  // The K sums of up to 16 members, 16 lanes to a value.
  template <int Nap, int K, int E>
  __device__ __forceinline__ void group_sums(const res_word *from, int members, unsigned limit, double *tot) {
    const int lane = (int)threadIdx.x & (kWave - 1);
    double g[E];
    const bool in = (lane & 15) < members;
    if (!res_wait<Nap, E>(ep, g, kResGroupSums, limit, a.err, [&](int q) -> const res_word * {
          const int e = lane + q * kWave;
          return in && e < 16 * K ? from + e : nullptr;
        }))
      *bad = 1;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const double s = res_row_sum(in && lane + q * kWave < 16 * K ? g[q] : 0.0);
#pragma unroll
      for (int k = 4 * q; k < (K < 4 * q + 4 ? K : 4 * q + 4); ++k) tot[k] = res_lane(s, 16 * (k & 3) + 15);
    }
  }

  // One exchange: the block's K sums to every block and theirs here, added in
  // the order of the blocks; the published rows of the halo into hdst (LDS,
  // nh entries; null: none); then epi()(totals) on thread 0, epi() itself
  // while the totals are on their way.  publish() goes before; work() is what
  // no other block waits for and is done meanwhile.  The first N scalars of
  // the new state are read on the way out (sc, done).  Some waves wait for the
  // sums and the others for the halo.  False if a wait expired.
  template <int K, int N, class T, class Epi, class Work>
  __device__ __forceinline__ bool exchange(const double *v, T *hdst, Epi &&epi, Work &&work) {
    ++ep;
    const int t = (int)threadIdx.x, lane = t & (kWave - 1), wid = t / kWave;
    {
      const double s = res_wave_sums<(K < 4 ? K : 4)>(v);
      const int k = res_sum_row<(K < 4 ? K : 4)>(lane >> 4);
      if ((lane & 15) == 15 && k < K) red[k * kMaxWaves + wid] = s;
      if constexpr (K > 4) {
        const double s4 = res_wave_sums<1>(v + 4);
        if (lane == kWave - 1) red[4 * kMaxWaves + wid] = s4;
      }
    }
    lds_barrier();
    static_assert(K <= kResSums, "a lane adds at most two of the groups' sums");
    constexpr int E = K > 4 ? 2 : 1;   // the fifth value goes with the first 16 lanes
    res_word *part = a.part + (size_t)(ep & 1) * (size_t)a.part_half;
    const unsigned limit = ep >= a.strict ? 0u : ep == 1 ? a.first : kResSpin;
    // Up to 64 blocks a lane per block adds all sums.  Beyond, so many
    // readers of so many words hold each other up (256 blocks: 7 us), and
    // the sums go in two steps: the first block of 16 adds its group's and
    // passes the totals to every group, 16 lanes to a value in both steps.
    const bool wide = nb > kWave, leads = wide && (map.c & 15) == 0;
    const int waiting = leads ? 2 : 1;   // waves that wait for sums
    if (wid == 0) {
      double own = 0.0;
      if (lane < K) {
        double q[NT / kWave];
#pragma unroll
        for (int w = 0; w < NT / kWave; ++w) q[w] = red[lane * kMaxWaves + w];
        own = q[0];
#pragma unroll
        for (int w = 1; w < NT / kWave; ++w) own += q[w];
        const int to = wide ? (map.c >> 4) * 2 * kResGroupSums + lane * 16 + (map.c & 15) : lane * 2 * kWave + map.c;
        if (nb > 1) res_put(part + to, wide ? kResGroupSums : kWave, own, ep);
      }
      auto close = epi();
      work();
      double tot[K];
      if (nb == 1) {
#pragma unroll
        for (int k = 0; k < K; ++k) tot[k] = res_lane(own, k);
      } else if (!wide) {
        double pv[K];
        if (!res_wait<kResNapSums, K>(ep, pv, kWave, limit, a.err, [&](int q) -> const res_word * {
              return lane < nb ? part + (q * 2 * kWave + lane) : nullptr;
            }))
          *bad = 1;
#pragma unroll
        for (int k = 0; k < K; ++k) pv[k] = lane < nb ? pv[k] : 0.0;
        const double s = res_wave_sums<(K < 4 ? K : 4)>(pv);
#pragma unroll
        for (int k = 0; k < (K < 4 ? K : 4); ++k) tot[k] = res_lane(s, 16 * res_sum_row<(K < 4 ? K : 4)>(k) + 15);
        if constexpr (K > 4) tot[4] = res_lane(res_wave_sums<1>(pv + 4), kWave - 1);
      } else {
        group_sums<kResNapTotals, K, E>(part + 2 * (size_t)(kResGroups + (map.c >> 4)) * kResGroupSums, (nb + 15) / 16, limit, tot);
      }
      if (lane == 0) close(tot);
    } else if (leads && wid == 1) {
      work();
      const int grp = map.c >> 4;
      double tot[K];
      group_sums<kResNapGroup, K, E>(part + 2 * (size_t)grp * kResGroupSums, nb - 16 * grp, limit, tot);
      // lane (value, group): that group's copy, all in one store (everyone waits
      // for this wave: a store per value was 1.3 us slower at 256 blocks)
      double mine = 0.0;
#pragma unroll
      for (int k = 0; k < (K < 4 ? K : 4); ++k)
        if (lane >> 4 == k) mine = tot[k];
      res_word *to = part + 2 * (size_t)((kResGroups + (lane & 15)) * kResGroupSums) + grp;
      if (lane < 16 * K && (lane & 15) < (nb + 15) / 16) res_put(to + (lane & 48), kResGroupSums, mine, ep);
      if (K > 4 && lane < (nb + 15) / 16) res_put(to + 64, kResGroupSums, tot[K - 1], ep);
    } else {
      work();
    }
    if (nb > 1 && hdst && wid >= waiting) {
      const int ht = NT - waiting * kWave, h0 = t - waiting * kWave;
      auto from = [&](int h) -> const res_word * {
        const int j = h < nh ? hrow[h] : -1;
        return j >= 0 ? row_words<T>(ep, j) : nullptr;
      };
      for (int base = 0; base < nh; base += ht * HE) {
        T hv[HE];
        const bool few = nh - base <= ht;
        const bool ok = few ? res_wait<kResNapRows, 1>(ep, hv, 1, limit, a.err, [&](int) { return from(base + h0); })
                            : res_wait<kResNapRows, HE>(ep, hv, 1, limit, a.err, [&](int q) { return from(base + h0 + q * ht); });
        if (!ok) {
          *bad = 1;
          break;
        }
#pragma unroll
        for (int q = 0; q < HE; ++q) {
          const int h = base + h0 + q * ht;
          if ((q == 0 || !few) && h < nh && hrow[h] >= 0) hdst[h] = hv[q];
        }
      }
    }
    lds_barrier();
    // all at once: each read is a trip to LDS
    int lost = nb > 1 ? *bad : 0;
    if constexpr (N > 0) {
      done = S->done;
      sc[0] = S->alpha;
      sc[1] = N > 1 ? S->beta : 0.0;
      sc[2] = N > 2 ? S->omega : 0.0;
      asm volatile("" : "+v"(lost), "+v"(done), "+v"(sc[0]), "+v"(sc[1]), "+v"(sc[2]));
    }
    if (!lost) return true;
    if (t == 0) st_relaxed(a.err, 1u);
    return false;
  }
  template <int K, int N = 0, class T, class Epi>
  __device__ __forceinline__ bool exchange(const double *v, T *hdst, Epi &&epi) {
    return exchange<K, N>(v, hdst, epi, [] {});
  }

  // Block 0 writes the state, all of it but `next`, which is a solve's err
  // word (cleared before the launch; one block alone never waits).
  __device__ __forceinline__ void outcome(int how) {
    if (map.c != 0) return;
    if (threadIdx.x == 0) {
      S->pad6 = how;
      S->next = 0;
    }
    lds_barrier();
    constexpr int skip = offsetof(KState, next) / sizeof(unsigned);
    for (int q = (int)threadIdx.x; q < (int)(sizeof(KState) / sizeof(unsigned)); q += NT)
      if (q != skip || nb == 1)
        reinterpret_cast<unsigned *>(a.st)[q] = reinterpret_cast<const unsigned *>(S)[q];
  }
};

// Row i's off-diagonal values and columns (0-based; -1: none there, and the
// value 0, which then multiplies the row's own operand); i < 0: no row.
// False if the row has more than fit.
template <int F>
__device__ __forceinline__ bool res_row(const Mat &A, int i, double *v, int *j) {
  constexpr int NW = F == F_ELL3 ? 3 : 4;
#pragma unroll
  for (int e = 0; e < 4; ++e) j[e] = -1;
#pragma unroll
  for (int e = 0; e < NW; ++e) v[e] = 0.0;
  if (i < 0) return true;
  if constexpr (F == F_CSRD) {
    const int k1 = A.ia[i] - 1, cnt = A.ia[i + 1] - 1 - k1;
#pragma unroll
    for (int e = 0; e < NW; ++e)
      if (e < cnt) {
        v[e] = A.av[k1 + e];
        j[e] = A.ja[k1 + e] - 1;
      }
    return cnt <= NW;
  } else {
#pragma unroll
    for (int e = 0; e < NW; ++e) {
      v[e] = A.av[(size_t)NW * i + e];
      if (v[e] != 0.0) j[e] = A.ja[(size_t)NW * i + e] - 1;
    }
    return true;
  }
}
// The window slots of those columns, two to a word, for local row l.
__device__ __forceinline__ bool res_slots(const ResMap &map, int l, int base, const int *j, unsigned *idx) {
  bool ok = true;
  int s[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    s[e] = j[e] < 0 ? l : map.slot(j[e], base);
    if (s[e] < 0) {
      ok = false;
      s[e] = l;
    }
  }
  idx[0] = (unsigned)s[0] | ((unsigned)s[1] << 16);
  idx[1] = (unsigned)s[2] | ((unsigned)s[3] << 16);
  return ok;
}

// The matrix rows of a block's threads in registers and the FP64 window.
template <int F, int RPT>
struct Resident : ResNet {
  static constexpr int NW = F == F_ELL3 ? 3 : 4, RB = NT * RPT;

  double *win;             // LDS: RB + nh
  double *own;             // LDS: x, then the shadow residual (RB each)
  double *hs;              // LDS: the halo rows' vectors, nh each
  double av[RPT][NW], dm[RPT];
  unsigned idx[RPT][2];

  __device__ __forceinline__ Resident(const ResArgs &args) : ResNet(args) {}

  __device__ __forceinline__ double *state(int q) const { return hs + (size_t)q * nh; }

  // Loads the matrix rows.  False where a column is outside the window.
  __device__ __forceinline__ bool load_rows() {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int l = (int)threadIdx.x + k * NT;
      const int i = map.own(l);
      row[l] = i;
      dm[k] = i >= 0 ? a.A.ad[i] : 1.0;
      if (i >= 0 && nb > 1 && map.edge(l)) pub |= 1u << k;
      int j[4];
      ok = res_row<F>(a.A, i, av[k], j) && ok;
      ok = res_slots(map, l, RB, j, idx[k]) && ok;
    }
    return ok;
  }

  // (A u)_k from the window; own = the row's own operand.  The reference's
  // order of the products, as RowRegs / row_apply.
  __device__ __forceinline__ double apply(int k, double own) const {
    const double x0 = win[idx[k][0] & 0xffffu], x1 = win[idx[k][0] >> 16], x2 = win[idx[k][1] & 0xffffu];
    const double t5 = dm[k] * own;
    if constexpr (F == F_ELL3) {
      return ((av[k][0] * x0 + av[k][1] * x1) + av[k][2] * x2) + t5;
    } else {
      const double x3 = win[idx[k][1] >> 16];
      if constexpr (F == F_CSRD) return (((t5 + av[k][0] * x0) + av[k][1] * x1) + av[k][2] * x2) + av[k][3] * x3;
      else return (((av[k][0] * x0 + av[k][1] * x1) + av[k][2] * x2) + av[k][3] * x3) + t5;
    }
  }

  // r = b - A x0 on the block's rows, x0 read from memory.
  __device__ __forceinline__ void residual(double *r, double *bb) {
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int l = (int)threadIdx.x + k * NT, i = row[l];
      double xi = 0.0, ax = 0.0;
      bb[k] = 0.0;
      if (i >= 0) {
        bb[k] = a.b[i];
        if (!a.x0_zero) {
          xi = a.x[i];
          ax = row_apply<F>(a.A, i, XVec{a.x});
        }
      }
      own[l] = xi;
      r[k] = bb[k] - ax;
    }
  }

  // Energy x.Ax (GMRES: x.b) and ||b - Ax||^2 (src/Iterativos.f:82-83,204-205,
  // 412), then x and the state are written.
  // A breakdown or an overflow depends on the roundings on the way there, so
  // such a solve is declined, with x as it came: it is solved again in the
  // other engine's order of sums, whose outcome the caller gets.
  __device__ __forceinline__ void finish(bool energy_xb = false) {
    if (S->status == S_BREAKDOWN || S->status == S_NONFINITE) return outcome(kResDeclined);
    const int t = (int)threadIdx.x;
    const double *x = own + t;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      win[t + k * NT] = x[k * NT];
      publish(k, x[k * NT]);
    }
    double none[1] = {0.0};
    // the halo's x must be here before the product: an exchange of its own
    if (!exchange<1>(none, win + RB, [] { return [](const double *) {}; })) return;
    double v[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const double xi = x[k * NT], ax = apply(k, xi);
      const int i = row[t + k * NT];
      const double bi = i >= 0 ? a.b[i] : 0.0;
      const double ri = bi - ax;
      v[0] += xi * (energy_xb ? bi : ax);
      v[1] += ri * ri;
    }
    KState *s = S;
    if (!exchange<2, 0, double>(v, nullptr, [s] {
          return [s](const double *tot) {
            s->energy = tot[0];
            s->res2 = tot[1];
          };
        }))
      return;
#pragma unroll
    for (int k = 0; k < RPT; ++k)
      if (row[t + k * NT] >= 0) a.x[row[t + k * NT]] = x[k * NT];
    outcome(kResSolved);
  }

  __device__ __forceinline__ void pcg();
  __device__ __forceinline__ void bicgstab();
  __device__ __forceinline__ void gmres();
};

// The fused PCG (cg1_*, fvc_krylov.h), one exchange per iteration.
template <int F, int RPT>
__device__ __forceinline__ void Resident<F, RPT>::pcg() {
  const int t = (int)threadIdx.x;
  Cg1Args e{};
  e.tol = a.tol;
  e.maxit = a.maxit;
  e.stop_rule = a.stop_rule;
  KState *s_ = S;
  double r[RPT], w[RPT], s[RPT], p[RPT];
  double *x = own + t;
  double *hr = state(0), *hw = state(1), *hsv = state(2), *hm = state(3);
  const bool ok = load_rows();
  residual(r, w);   // w = b for the moment
  for (int h = t; h < nh; h += NT) {
    const int j = hrow[h];
    hm[h] = j >= 0 ? a.m[j] : 1.0;
    hr[h] = hw[h] = hsv[h] = 0.0;
    win[RB + h] = 0.0;
  }
  double v[4] = {0.0, 0.0, 0.0, ok ? 0.0 : 1.0};
#pragma unroll
  for (int k = 0; k < RPT; ++k) {
    s[k] = p[k] = 0.0;
    publish(k, r[k]);
    v[0] += r[k] * (r[k] / dm[k]);
    v[1] += w[k] * w[k];
    v[2] += r[k] * r[k];
  }
  if (!exchange<4, 1>(v, hr, [&] {
        return [&](const double *tot) {
          cg1_epi(e, CG1_SETUP, s_, tot);
          if (tot[3] != 0.0) s_->pend = 1;
        };
      }))
    return;
  if (S->pend) return outcome(kResDeclined);   // a block's columns do not fit its window
  // round 0 is W0 (w = A u), the following ones CG1_ITER
  for (int it = 0; !done; ++it) {
    const double al = sc[0], be = sc[1];
    if (it > 0) {
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        const double u = win[t + k * NT];   // r / m, of the previous iteration
        p[k] = it == 1 ? u : u + be * p[k];
        s[k] = it == 1 ? w[k] : w[k] + be * s[k];
        r[k] = r[k] - al * s[k];
      }
      for (int h = t; h < nh; h += NT) {
        const double sj = it == 1 ? hw[h] : hw[h] + be * hsv[h];
        hsv[h] = sj;
        hr[h] = hr[h] - al * sj;
      }
    }
    double u[RPT], v3[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      u[k] = r[k] / dm[k];
      win[t + k * NT] = u[k];
      v3[0] += r[k] * u[k];
      v3[2] += r[k] * r[k];
    }
    for (int h = t; h < nh; h += NT) win[RB + h] = hr[h] / hm[h];
    lds_barrier();
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      w[k] = apply(k, u[k]);
      publish(k, w[k]);
      v3[1] += w[k] * u[k];
    }
    const bool go = exchange<3, 2>(
        v3, hw,
        [&] {
          const Cg1Scalars c = cg1_scalars(s_);
          return [&, c](const double *tot) {
            if (it == 0) cg1_epi(e, CG1_W0, s_, tot + 1);
            else cg1_iter_epi(e, c, s_, tot);
          };
        },
        [&] {
          if (it > 0) {
#pragma unroll
            for (int k = 0; k < RPT; ++k) x[k * NT] = x[k * NT] + al * p[k];
          }
        });
    if (!go) return;
  }
  finish();
}

// The two-phase BiCGSTAB (bicg2_*, fvc_krylov.h), one exchange per phase.
template <int F, int RPT>
__device__ __forceinline__ void Resident<F, RPT>::bicgstab() {
  const int t = (int)threadIdx.x;
  Bicg2Args e{};
  e.tol = a.tol;
  e.maxit = a.maxit;
  e.stop_rule = a.stop_rule;
  KState *s_ = S;
  double s[RPT], q_[RPT], p[RPT], v[RPT];   // s holds b between P and Q; q_ is t
  double *x = own + t, *rh = own + RB + t;
  double *hsb = state(0), *ht = state(1), *hp = state(2), *hv = state(3), *hm = state(4);
  const bool ok = load_rows();
  residual(s, q_);
  for (int h = t; h < nh; h += NT) {
    const int j = hrow[h];
    hm[h] = j >= 0 ? a.m[j] : 1.0;
    hsb[h] = ht[h] = hp[h] = hv[h] = 0.0;
    win[RB + h] = 0.0;
  }
  double v0[4] = {0.0, 0.0, 0.0, ok ? 0.0 : 1.0};
#pragma unroll
  for (int k = 0; k < RPT; ++k) {
    const double ri = s[k];
    rh[k * NT] = p[k] = ri;
    v[k] = 0.0;
    publish(k, ri);
    v0[0] += ri * (ri / dm[k]);
    v0[1] += ri * ri;
    v0[2] += q_[k] * q_[k];
    q_[k] = 0.0;
  }
  if (!exchange<4, 1>(v0, hp, [&] {
        return [&](const double *tot) {
          bicg2_epi(e, B2_SETUP, s_, tot);
          if (tot[3] != 0.0) s_->pend = 1;
        };
      }))
    return;
  if (S->pend) return outcome(kResDeclined);
  for (int h = t; h < nh; h += NT) hsb[h] = hp[h];
  for (int it = 1; !done; ++it) {
    // P: completes iteration it - 1, p, v = A (p/m)
    double v3[3] = {0.0, 0.0, 0.0};
    if (it > 1) {
      const double be = sc[1], om = sc[2];
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        const double z2 = win[t + k * NT];   // s / m, of Q
        const double bi = s[k] - om * q_[k];
        x[k * NT] = x[k * NT] + om * z2;
        s[k] = bi;
        p[k] = bi + be * (p[k] - om * v[k]);
        v3[1] += bi * z2;
        v3[2] += bi * bi;
      }
      for (int h = t; h < nh; h += NT) {
        const double bi = hsb[h] - om * ht[h];
        hsb[h] = bi;
        hp[h] = bi + be * (hp[h] - om * hv[h]);
      }
    }
#pragma unroll
    for (int k = 0; k < RPT; ++k) win[t + k * NT] = p[k] / dm[k];
    for (int h = t; h < nh; h += NT) win[RB + h] = hp[h] / hm[h];
    lds_barrier();
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      v[k] = apply(k, win[t + k * NT]);
      publish(k, v[k]);
      v3[0] += v[k] * rh[k * NT];
    }
    if (!exchange<3, 1>(v3, hv, [&] {
          const Bicg2Scalars c = bicg2_scalars(s_);
          return [&, c](const double *tot) { bicg2_p_epi(e, c, s_, tot); };
        }))
      return;
    if (done) break;
    // Q: s = b - alpha v, t = A (s/m)
    const double al = sc[0];
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      s[k] = s[k] - al * v[k];
      x[k * NT] = x[k * NT] + al * win[t + k * NT];   // p / m, of P
      win[t + k * NT] = s[k] / dm[k];
    }
    for (int h = t; h < nh; h += NT) {
      hsb[h] = hsb[h] - al * hv[h];
      win[RB + h] = hsb[h] / hm[h];
    }
    double v4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) v4[2] += rh[k * NT] * s[k];
    lds_barrier();
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      q_[k] = apply(k, win[t + k * NT]);
      publish(k, q_[k]);
      v4[0] += q_[k] * s[k];
      v4[1] += q_[k] * q_[k];
      v4[3] += rh[k * NT] * q_[k];
    }
    if (!exchange<4, 3>(v4, ht, [&] {
          const Bicg2Scalars c = bicg2_scalars(s_);
          return [&, c](const double *tot) { bicg2_q_epi(c, s_, tot); };
        }))
      return;
  }
  finish();
}

// GMRES(k) with modified Gram-Schmidt in the reference's order (gmres_phase,
// fvc_krylov.h), an exchange for each of the i + 1 reductions of Arnoldi step
// i.  The vector being orthogonalised stays in registers; the basis columns,
// k times too large for them, are in memory, where only their own block reads
// them: the next column is on its way while the block waits for a sum, so
// that a projection costs little more than its exchange.  The Hessenberg
// matrix, the rotations and the back substitution are in every block's LDS.
template <int F, int RPT>
__device__ __forceinline__ void Resident<F, RPT>::gmres() {
  __shared__ double hbuf[(kResGmresK + 1) * kResGmresK + 5 * (kResGmresK + 3)];
  const int t = (int)threadIdx.x;
  KState *st = S;
  GmresArgs e{};
  e.tol = a.tol;
  e.k = a.k;
  e.maxit = a.maxit;
  e.stop_rule = a.stop_rule;
  e.h = hbuf;
  e.cs = hbuf + (kResGmresK + 1) * kResGmresK;
  e.sn = e.cs + kResGmresK + 3;
  e.e = e.sn + kResGmresK + 3;
  e.y = e.e + kResGmresK + 3;
  e.nrm = e.y + kResGmresK + 3;
  double *x = own + t;
  double w[RPT], gj[RPT], gn[RPT];
  const double none[1] = {0.0};
  const bool ok = load_rows();
#pragma unroll
  for (int k = 0; k < RPT; ++k) x[k * NT] = 0.0;
  for (int h = t; h < nh; h += NT) win[RB + h] = 0.0;
  const auto column = [&](int c, int i) -> double & { return a.gv[(size_t)(c - 1) * a.ld + i]; };
  const auto load_column = [&](int c, double *g) {
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int i = row[t + k * NT];
      g[k] = i >= 0 ? column(c, i) : 0.0;
    }
  };
  for (bool first = true; !st->done; first = false) {
    // g1 = (b - A x) / m
    if (!first) {
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        win[t + k * NT] = x[k * NT];
        publish(k, x[k * NT]);
      }
      if (!exchange<1>(none, win + RB, [] { return [](const double *) {}; })) return;
    }
    double v[4] = {0.0, 0.0, 0.0, ok ? 0.0 : 1.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int i = row[t + k * NT];
      const double bi = i >= 0 ? a.b[i] : 0.0;
      const double ri = first ? bi : bi - apply(k, x[k * NT]);
      w[k] = ri / dm[k];
      v[0] += w[k] * w[k];
      if (first) v[1] += bi * bi;
      v[2] += ri * ri;
      publish(k, w[k]);
    }
    if (!exchange<4>(v, win + RB, [&] {
          return [&](const double *tot) {
            gmres_start_epi(e, st, first, tot);
            if (tot[3] != 0.0) st->pend = 1;
          };
        }))
      return;
    if (st->pend) return outcome(kResDeclined);
    if (st->done) break;
    for (int i = 1; i <= a.k; ++i) {
      // column i = w / ||w||, w = A g_i / m (the halo holds w of its rows)
      const double ni = e.nrm[i];
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        const double g = w[k] / ni;
        const int r = row[t + k * NT];
        win[t + k * NT] = g;
        if (r >= 0) column(i, r) = g;
        if (i == 1) gj[k] = g;
      }
      for (int h = t; h < nh; h += NT) win[RB + h] = win[RB + h] / ni;
      if (i > 1) load_column(1, gj);
      lds_barrier();
      double d[1] = {0.0};
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        w[k] = apply(k, win[t + k * NT]) / dm[k];
        d[0] += w[k] * gj[k];
      }
      if (i > 2) load_column(2, gn);
      if (!exchange<1, 1, double>(d, nullptr, [&] {
            return [&](const double *tot) {
              e.h[(size_t)(i - 1) * (a.k + 1)] = tot[0];
              st->alpha = tot[0];
            };
          }))
        return;
      for (int j = 1; j <= i; ++j) {
        const double hj = sc[0];
        d[0] = 0.0;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
          w[k] = w[k] - hj * gj[k];
          if (j == i) {
            d[0] += w[k] * w[k];
            publish(k, w[k]);
          } else {
            gj[k] = j + 1 == i ? win[t + k * NT] : gn[k];   // column i is still in the window
            d[0] += w[k] * gj[k];
          }
        }
        if (j + 2 < i) load_column(j + 2, gn);
        if (!exchange<1, 1>(d, j == i ? win + RB : nullptr, [&] {
              return [&](const double *tot) {
                double *hi = e.h + (size_t)(i - 1) * (a.k + 1);
                if (j < i) {
                  hi[j] = tot[0];
                  st->alpha = tot[0];
                  return;
                }
                const double norm = sqrt(tot[0]);
                hi[i] = norm;
                e.nrm[i + 1] = norm;
                gmres_close_step(e, st, i);
              };
            }))
          return;
      }
      if (st->inner_done) break;
    }
    // x += sum_j y(j) g(j), in order
    const int nI = st->ni;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int r = row[t + k * NT];
      double xr = x[k * NT];
      if (r >= 0)
        for (int j = 1; j <= nI; ++j) xr = xr + e.y[j] * column(j, r);
      x[k * NT] = xr;
    }
    lds_barrier();
    if (t == 0) gmres_xupd_epi(e, st, nI);
    lds_barrier();
  }
  finish(true);
}

// Mixed precision (fvc_mixed.h): the scaled FP32 rows and the four FP32
// vectors {r~, q, p, y} in registers; x stays in memory, where only a block's
// own threads read it, and the FP64 matrix is read again at the reliable
// updates, whose window of x takes the place of the FP32 one.
template <int F, int RPT>
struct ResidentMixed : ResNet {
  static constexpr int NW = F == F_ELL3 ? 3 : 4, RB = NT * RPT;

  double *win;             // LDS: RB + nh, as floats between the updates
  float *hs;               // LDS: the halo rows' r~, q, p, nh each
  float av[RPT][NW], dsq[RPT];
  unsigned idx[RPT][2];

  __device__ __forceinline__ ResidentMixed(const ResArgs &args) : ResNet(args) {}

  __device__ __forceinline__ bool load_rows() {
    bool ok = true;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int l = (int)threadIdx.x + k * NT, i = map.own(l);
      row[l] = i;
      if (i >= 0 && nb > 1 && map.edge(l)) pub |= 1u << k;
      const double m = i >= 0 ? a.m[i] : 1.0;
      const double si = 1.0 / sqrt(m);
      dsq[k] = (float)sqrt(m);
      double v[NW];
      int j[4];
      ok = res_row<F>(a.A, i, v, j) && ok;
#pragma unroll
      for (int e = 0; e < NW; ++e) {
        av[k][e] = j[e] >= 0 ? (float)(v[e] * si * (1.0 / sqrt(a.m[j[e]]))) : 0.0f;
      }
      ok = res_slots(map, l, RB, j, idx[k]) && ok;
    }
    return ok;
  }

  // (S A S p)_k, unit diagonal (as RowRegs32 / row_apply32)
  __device__ __forceinline__ float apply32(int k, float own) const {
    const float *w = reinterpret_cast<const float *>(win);
    const float x0 = w[idx[k][0] & 0xffffu], x1 = w[idx[k][0] >> 16], x2 = w[idx[k][1] & 0xffffu];
    if constexpr (F == F_ELL3) {
      return ((av[k][0] * x0 + av[k][1] * x1) + av[k][2] * x2) + own;
    } else {
      const float x3 = w[idx[k][1] >> 16];
      if constexpr (F == F_CSRD) return (((own + av[k][0] * x0) + av[k][1] * x1) + av[k][2] * x2) + av[k][3] * x3;
      else return (((av[k][0] * x0 + av[k][1] * x1) + av[k][2] * x2) + av[k][3] * x3) + own;
    }
  }
  // (A x)_k in FP64: the row from memory, x from the window.
  __device__ __forceinline__ double apply64(int k, int i, double own) const {
    double v[NW];
    int j[4];
    res_row<F>(a.A, i, v, j);
    const double x0 = win[idx[k][0] & 0xffffu], x1 = win[idx[k][0] >> 16], x2 = win[idx[k][1] & 0xffffu];
    const double t5 = a.A.ad[i] * own;
    if constexpr (F == F_ELL3) {
      return ((v[0] * x0 + v[1] * x1) + v[2] * x2) + t5;
    } else {
      const double x3 = win[idx[k][1] >> 16];
      if constexpr (F == F_CSRD) return (((t5 + v[0] * x0) + v[1] * x1) + v[2] * x2) + v[3] * x3;
      else return (((v[0] * x0 + v[1] * x1) + v[2] * x2) + v[3] * x3) + t5;
    }
  }

  // x of own and halo rows into the window
  __device__ __forceinline__ bool window_x() {
    const int t = (int)threadIdx.x;
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int i = row[t + k * NT];
      const double xi = i >= 0 ? a.x[i] : 0.0;
      win[t + k * NT] = xi;
      publish(k, xi);
    }
    const double none[1] = {0.0};
    return exchange<1>(none, win + RB, [] { return [](const double *) {}; });
  }

  __device__ __forceinline__ void pcg() {
    const int t = (int)threadIdx.x;
    MixedArgs e{};
    e.tol = a.tol;
    e.delta = a.delta;
    e.maxit = a.maxit;
    e.max_inner = a.max_inner;
    KState *st = S;
    float *w32 = reinterpret_cast<float *>(win);
    float *hr = hs, *hq = hs + nh, *hp = hs + 2 * nh;
    float r[RPT], q[RPT], p[RPT], y[RPT];
    const bool ok = load_rows();
    for (int h = t; h < nh; h += NT) hr[h] = hq[h] = hp[h] = 0.0f;
    double v[4] = {0.0, 0.0, 0.0, ok ? 0.0 : 1.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int i = row[t + k * NT];
      r[k] = q[k] = p[k] = y[k] = 0.0f;
      double bi = 0.0, ri = 0.0;
      if (i >= 0) {
        // (x as given is whole in memory until the first exchange is over)
        bi = a.b[i];
        if (a.x0_zero) {
          a.x[i] = 0.0;
          ri = bi;
        } else {
          ri = bi - row_apply<F>(a.A, i, XVec{a.x});
        }
        r[k] = (float)(ri * (1.0 / sqrt(a.m[i])));
      }
      publish(k, r[k]);
      v[0] += (double)r[k] * (double)r[k];
      v[1] += ri * ri;
      v[2] += bi * bi;
    }
    if (!exchange<4>(v, hr, [&] {
          return [&](const double *tot) {
            mixed_epi(e, MX_SETUP, st, tot);
            if (tot[3] != 0.0) st->pend = 1;
          };
        }))
      return;
    if (S->pend) return outcome(kResDeclined);
    while (!S->done) {
      if (S->next == MX_A) {
        const float al = S->step_i ? 0.0f : (float)S->alpha, be = S->ni ? 0.0f : (float)S->beta;
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
          y[k] = y[k] + al * p[k];
          r[k] = r[k] - al * q[k];
          p[k] = r[k] + be * p[k];
          w32[t + k * NT] = p[k];
        }
        for (int h = t; h < nh; h += NT) {
          const float rh = hr[h] - al * hq[h], ph = rh + be * hp[h];
          hr[h] = rh;
          hp[h] = ph;
          w32[RB + h] = ph;
        }
        lds_barrier();
        double v5[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < RPT; ++k) {
          q[k] = apply32(k, p[k]);
          publish(k, q[k]);
          const double rd = r[k], qd = q[k];
          v5[0] += (double)p[k] * qd;
          v5[1] += rd * qd;
          v5[2] += qd * qd;
          v5[3] += rd * rd;
          const double ru = rd * (double)dsq[k];
          v5[4] += ru * ru;
        }
        if (!exchange<5>(v5, hq, [&] {
              const MixedScalars c = mixed_scalars(e, st);
              return [&, c](const double *tot) { mixed_a_epi(e, c, st, tot); };
            }))
          return;
        continue;
      }
      // a reliable update: x += S (y + alpha p), r~ = S (b - A x) in FP64
      const float al = (float)S->alpha;
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        const int i = row[t + k * NT];
        const float yi = y[k] + al * p[k];
        if (i >= 0) a.x[i] = a.x[i] + (1.0 / sqrt(a.m[i])) * (double)yi;
        y[k] = 0.0f;
        }
      if (!window_x()) return;
      double v3[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int k = 0; k < RPT; ++k) {
        const int i = row[t + k * NT];
        if (i >= 0) {
          const double bi = a.b[i], ri = bi - apply64(k, i, win[t + k * NT]);
          r[k] = (float)(ri * (1.0 / sqrt(a.m[i])));
          v3[1] += ri * ri;
          v3[2] += bi * bi;
        }
        publish(k, r[k]);
        v3[0] += (double)r[k] * (double)r[k];
        }
      if (!exchange<3>(v3, hr, [&] { return [&](const double *tot) { mixed_epi(e, MX_R, st, tot); }; })) return;
    }
    if (S->status == S_NONFINITE) return outcome(kResDeclined);
    if (!window_x()) return;
    double v2[2] = {0.0, 0.0};
#pragma unroll
    for (int k = 0; k < RPT; ++k) {
      const int i = row[t + k * NT];
      if (i >= 0) {
        const double xi = win[t + k * NT], ax = apply64(k, i, xi), ri = a.b[i] - ax;
        v2[0] += xi * ax;
        v2[1] += ri * ri;
      }
    }
    if (!exchange<2, 0, double>(v2, nullptr, [st] {
          return [st](const double *tot) {
            st->energy = tot[0];
            st->res2 = tot[1];
          };
        }))
      return;
    if (t == 0) S->mgs_j = map.p.H;   // whether every column is an int16 offset away
    outcome(kResSolved);
  }
};

// Sets a block up as part c of a system and solves it.  dyn: the block's
// dynamic shared memory (res_lds_bytes).
template <int F, int RPT, int Code>
__device__ __forceinline__ void resident_solve(const ResArgs &a, const ResPlan &p, int c, double *dyn) {
  __shared__ double red[kMaxK * kMaxWaves];
  __shared__ KState S;
  __shared__ int bad;
  const int t = (int)threadIdx.x;
  for (int k = t; k < (int)(sizeof(KState) / sizeof(unsigned)); k += kResThreads)
    reinterpret_cast<unsigned *>(&S)[k] = 0u;
  if (t == 0) bad = 0;
  using Sys = std::conditional_t<Code == kResMixedPcg, ResidentMixed<F, RPT>, Resident<F, RPT>>;
  Sys w(a);
  w.map.init(p, a.A.neq, c);
  w.nh = p.nb > 1 ? p.nh : 0;
  w.nb = p.nb;
  w.win = dyn;
  if constexpr (Code == kResMixedPcg) {
    w.hs = reinterpret_cast<float *>(dyn + kResThreads * RPT + w.nh);
    w.row = reinterpret_cast<int *>(w.hs + 3 * (size_t)w.nh);
  } else {
    w.own = dyn + kResThreads * RPT + w.nh;
    w.hs = w.own + (size_t)res_own_vecs(Code) * kResThreads * RPT;
    w.row = reinterpret_cast<int *>(w.hs + (Code == kResGmres ? 0 : (size_t)res_halo_vecs(Code) * w.nh));
  }
  w.hrow = w.row + kResThreads * RPT;
  w.red = red;
  w.S = &S;
  w.bad = &bad;
  for (int h = t; h < w.nh; h += kResThreads) w.hrow[h] = w.map.halo(h);
  __syncthreads();
  if constexpr (Code == kResBicgstab) w.bicgstab();
  else if constexpr (Code == kResGmres) w.gmres();
  else w.pcg();
}

// Does block c take part in plan p?
template <int RPT, int Code>
__device__ __forceinline__ bool resident_part(const ResPlan &p, int c) {
  return c < p.nb && p.nb <= kResMaxBlocks && p.nh <= res_max_halo(Code, RPT) && p.R <= kResThreads * RPT;
}

// One system on the whole grid, one block per CU, all co-resident (the host
// checks that the grid fits).
template <int F, int RPT, int Code>
__global__ __launch_bounds__(kResThreads) void resident_kernel(ResArgs a) {
  extern __shared__ double dyn[];
  ResPlan p{};
  if (a.plan) {
    p = *a.plan;
  } else {
    p.nb = 1;
    p.R = a.A.neq;
  }
  const int g = (int)gridDim.x, b = (int)blockIdx.x;
  // consecutive parts of the system on one XCD (blocks b = x mod 8)
  const int c = (g & 7) == 0 ? (b & 7) * (g >> 3) + (b >> 3) : b;
  if (p.nb == 0 && b == 0 && threadIdx.x == 0) a.st->pad6 = kResDeclined;
  if (!resident_part<RPT, Code>(p, c)) return;
  resident_solve<F, RPT, Code>(a, p, c, dyn);
}

// ---------------------------------------------------------------- batches --
//
// Many systems in one launch: a system gets a team of consecutive blocks just
// large enough to hold it, and a block's systems follow each other in the
// order of one list, the same for all blocks, so teams never wait in a ring.
// All blocks are co-resident.
struct ResBatchArgs {
  int w;
  const double *ad, *av, *b;
  const int *ia, *ja;
  double *x;
  const SysDesc *desc;       // g_first, g_count: the team
  const int *part_off;       // where a system's words for partial sums start
  const int *block_ptr, *block_list;
  KState *st;                // per system, cleared
  ResPlan *plans;            // per system, cleared
  res_word *rows, *part;
  unsigned *err;
  unsigned strict;           // as ResArgs'
  double tol, delta;
  int maxit, x0_zero, stop_rule, max_inner, rmax, hmax;
};

// An int / a struct of ints that is the same for the whole wavefront, in
// scalar registers (the compiler cannot tell: the kernel also stores).
__device__ __forceinline__ int res_uniform(const int *p) { return __builtin_amdgcn_readfirstlane(*p); }
template <class T>
__device__ __forceinline__ T res_uniform_ints(const T *p) {
  static_assert(sizeof(T) % sizeof(int) == 0, "a struct of ints");
  T v;
  int w[sizeof(T) / sizeof(int)];
#pragma unroll
  for (size_t k = 0; k < sizeof(T) / sizeof(int); ++k) w[k] = res_uniform(reinterpret_cast<const int *>(p) + k);
  __builtin_memcpy(&v, w, sizeof(T));
  return v;
}

// A team's first exchange waits for its members' earlier systems (up to 12 s).
constexpr unsigned kResFirstTeam = 32 * kResSpin;

template <int F>
__device__ __forceinline__ void resident_batch_mat(const ResBatchArgs &B, const SysDesc &D, Mat &A) {
  A.neq = D.neq;
  A.w = B.w;
  A.ad = B.ad + D.row_off;
  A.av = B.av + D.val_off;
  A.au = nullptr;
  A.ia = F == F_CSRD ? B.ia + D.ia_off : nullptr;
  A.ja = B.ja + D.val_off;
  A.tptr = A.tsrc = A.tpos = nullptr;
}

// blockIdx.y: the systems of `multi` (those of more than one block)
template <int F>
__global__ __launch_bounds__(256) void resident_batch_prep_kernel(ResBatchArgs B, const int *multi) {
  const int sys = multi[blockIdx.y];
  const SysDesc D = B.desc[sys];
  ResPrepArgs a{};
  resident_batch_mat<F>(B, D, a.A);
  a.plan = B.plans + sys;
  a.part = B.part + B.part_off[sys];
  a.rows = B.rows + (size_t)4 * D.row_off;
  a.nparts = 2 * res_part_half(D.g_count);
  a.rmax = B.rmax;
  a.bmax = D.g_count;
  a.hmax = B.hmax;
  resident_prep<F>(a);
}

template <int F, int RPT, int Code>
__global__ __launch_bounds__(kResThreads) void resident_batch_kernel(ResBatchArgs B) {
  extern __shared__ double dyn[];
  __shared__ unsigned stop;
  const int g = (int)gridDim.x, b0 = (int)blockIdx.x;
  const int b = (g & 7) == 0 ? (b0 & 7) * (g >> 3) + (b0 >> 3) : b0;
  const int k1 = res_uniform(B.block_ptr + b + 1);
  for (int k = res_uniform(B.block_ptr + b); k < k1; ++k) {
    const int sys = res_uniform(B.block_list + k);
    const SysDesc D = res_uniform_ints(B.desc + sys);
    const int c = b - D.g_first;
    ResPlan p{};
    if (D.g_count > 1) {
      p = res_uniform_ints(B.plans + sys);
    } else {
      p.nb = 1;
      p.R = D.neq;
    }
    if (p.nb == 0 && c == 0 && threadIdx.x == 0) B.st[sys].pad6 = kResDeclined;
    if (!resident_part<RPT, Code>(p, c)) continue;
    ResArgs a{};
    resident_batch_mat<F>(B, D, a.A);
    a.st = B.st + sys;
    a.m = a.A.ad;
    a.x = B.x + D.row_off;
    a.b = B.b + D.row_off;
    a.rows = B.rows + (size_t)4 * D.row_off;
    a.part = B.part + res_uniform(B.part_off + sys);
    a.part_half = res_part_half(D.g_count);
    a.err = B.err;
    a.first = kResFirstTeam;
    a.strict = B.strict;
    a.tol = B.tol;
    a.maxit = B.maxit;
    a.x0_zero = B.x0_zero;
    a.stop_rule = B.stop_rule;
    a.delta = B.delta;
    a.max_inner = B.max_inner;
    resident_solve<F, RPT, Code>(a, p, c, dyn);
    // Once a wait expired, every block leaves, all of its waves or none: the
    // word is set while others look at it, and a block whose wave 0 alone had
    // left would go on to its next system with nobody to run the scalar part, a
    // loop without an end where one block holds that system and waits for no one.
    if (threadIdx.x == 0) stop = ld_relaxed(B.err);
    __syncthreads();   // (also: LDS is reused)
    if (stop != 0u) return;
  }
}

}  // namespace fvc
