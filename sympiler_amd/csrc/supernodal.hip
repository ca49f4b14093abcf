// supernodal.hip -- solves on a supernodal (BCSC) lower triangle for gfx950,
// the forward one bit-identical to the reference's blocked solve.
//
// Reference: sparse_blas/sptrsv.cpp:176-199 (sptrsv_csc_block) with the dense
// kernels of sparse_blas/dense_blas/BLAS.cpp: lsolve_BLAS (:3-96) and
// matvec_BLAS (:286-349); sparse_blas/sptrsv.cpp:239-279
// (sptrsv_csc_levelset_block) is the same per-supernode routine under a level
// schedule, scattering with atomics.
//
// Layout (the reference's): supernode i owns columns s_i .. s_i + w_i - 1 and
// nrows_i block rows; its values are a column-major nrows_i x w_i block at
// Lx[Lp[i]] whose first w_i rows are its own columns and whose row r is row
// Li[Lp[i] + r] of L.  Per supernode the reference solves the dense top
// (every row subtracts its products column by column, left to right, then
// divides), multiplies the rows below by the solved part (column blocks of 8,
// then 4, then 1; each block's products summed left to right and added to a
// zeroed temporary), and subtracts the temporary from x at those rows,
// supernode after supernode.
//
// Executor: one persistent launch of four-wave workgroups that take tickets
// level by level of the tree.  A ticket is up to four narrow supernodes (at
// most 64 columns: one wavefront solves the top and multiplies the first
// SN_NARROW_ROWS rows below), the top of one wide supernode (the workgroup),
// or 64 rows below a top (the workgroup, its column blocks dealt over the
// waves).  Every wait is for an earlier ticket, which a running workgroup
// holds.  The subtraction into x is pulled instead of pushed: each supernode
// writes its temporaries to T where the rows that subtract them read their
// lists (ascending supernode order, the order of the reference's serial
// loop): entry j of the 64 rows of a wave lies side by side, so a load of T
// is one contiguous run.
//
// What bounds it: the chain of tree levels -- for each, the widest top's
// columns (a division, a broadcast and a multiply-subtract each, about 75 ns)
// plus the hand-offs -- for one right-hand side and the last levels of a
// block.  A top's rows lie one per lane, 64 to a wave, and each wave streams
// its rows' entries with SN_AHEAD column blocks in flight; the wave whose
// rows are next solves its 64 columns with lane broadcasts and hands x on
// through LDS, block of 8 by block of 8, while the other waves subtract.
// Measured on the 13-level nested-dissection-shaped factor (8,191 supernodes
// up to 512 wide, 36 M values), forward and transposed: one right-hand side
// 4.35 ms with one wavefront per top -> 1.07 ms, 32 right-hand sides 11.6 ->
// 3.22 ms.
#include <algorithm>
#include <vector>

#include "device.h"

namespace symamd {

namespace {

constexpr int SN_AHEAD = 4;  // column blocks of 8 whose entries are in flight

struct SnArgs {
  const int *sup, *nrows, *Lp;  // the reference's supernode arrays
  const double *Lx;
  double *x;                    // right-hand side in, solution out
  double *T;                    // temporaries, placed where the rows' lists are read
  const int *tb;                // supernode i's rows below start at tb[i]
  const int *tdst;              // place in T of each row below
  const int4 *list;             // row r subtracts T[x + j*z], j < y
  const int2 *unit;             // unit u: (supernode, 0 = top or c = chunk c - 1 below)
  const int *tick;              // ticket t runs units tick[t] .. tick[t+1]
  const int *dptr, *dlist;      // units that unit u waits for
  int *flags, *state;           // one tag per (column tile, unit)
  int nunits, ntick, total_waves;
  const int *rowb;              // transposed: rows below (at tb)
  const int *tbelow;            // transposed: first column-group unit of a supernode, or -1
  int k, tiles;                 // right-hand sides: column c at x + c*ldx; tiles of KT
  int64_t ldx, tcount;          // column c's temporaries at T + c*tcount
  uint64_t timeout;
};

// v on lane j (j uniform), for every lane
__device__ __forceinline__ double lane_value(double v, int j) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, j);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), j);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The right-hand side columns of one tile; columns past k repeat the last
// one (solved again, not stored).
template <int KT>
struct Cols {
  double *x[KT];
  bool live[KT];
  __device__ __forceinline__ Cols(const SnArgs &a, int tile) {
#pragma unroll
    for (int c = 0; c < KT; ++c) {
      const int col = tile * KT + c;
      live[c] = col < a.k;
      x[c] = a.x + (int64_t)min(col, a.k - 1) * a.ldx;
    }
  }
};

// The values are computed here: without it the compiler moves a block's
// subtractions past the wait for the next block, and keeps their operands in
// registers (and then in scratch memory) until there.
template <int KT>
__device__ __forceinline__ void hold(double (&v)[KT]) {
#pragma unroll
  for (int c = 0; c < KT; ++c) asm volatile("" : "+v"(v[c]));
}

// Columns solved so far of the workgroup's top, kept in LDS: the wave that
// solved a block of eight stores their x, then the count; LDS operations of a
// wave complete in order, so a wave that reads the count reads those x.
__device__ __forceinline__ void lds_publish(int *prog, int v, int lane) {
  asm volatile("" ::: "memory");
  if (lane == 0) __hip_atomic_store(prog, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
// Waits until the count reaches `need`; the waves solve their rows in
// ascending count order and wait for nothing else, so it always does.
__device__ __forceinline__ void lds_wait(const int *prog, int need, int &seen) {
  while (seen < need)
    seen = __builtin_amdgcn_readfirstlane(
        __hip_atomic_load(prog, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
  asm volatile("" ::: "memory");
}

// Waits for one tag (every lane reads it); bounded by the watchdog as
// wait_list is.
__device__ __forceinline__ void wait_flag(const int *f, int target, int *state,
                                          uint64_t timeout) {
  if (ld_dev(f) == target) return;
  const uint64_t t0 = wall_ticks();
  for (int rounds = 1; ld_dev(f) != target; ++rounds) {
    __builtin_amdgcn_s_sleep(1);
    if ((rounds & 63) == 0 && wall_ticks() - t0 > timeout) {
      if ((threadIdx.x & 63) == 0) atomicOr(&state[ST_ERROR], 1);
      break;
    }
  }
  asm volatile("" ::: "memory");
}

// One lane per row: v minus the row's temporaries, in list order, GB entries
// per round with the next round's loads in flight.  Entries past the row's
// list are its last one (or T's first), not used.
template <int KT>
__device__ __forceinline__ void gather_list(double (&v)[KT], const double *T, int64_t tcount,
                                            const int4 &l) {
  constexpr int GB = 16 / KT;
  double ta[GB][KT], tb[GB][KT];
  auto load = [&](double (&t)[GB][KT], int j) {
#pragma unroll
    for (int u = 0; u < GB; ++u) {
      const double *p = T + (l.x + (int64_t)max(min(j + u, l.y - 1), 0) * l.z);
#pragma unroll
      for (int q = 0; q < KT; ++q) t[u][q] = ld_dev(p + q * tcount);
    }
  };
  auto subtract = [&](const double (&t)[GB][KT], int j) {
#pragma unroll
    for (int u = 0; u < GB; ++u)
#pragma unroll
      for (int q = 0; q < KT; ++q) v[q] = j + u < l.y ? v[q] - t[u][q] : v[q];
  };
  if (!__any(l.y > 0)) return;
  load(ta, 0);
  for (int j = 0;;) {
    load(tb, j + GB);
    subtract(ta, j);
    j += GB;
    if (!__any(j < l.y)) break;
    load(ta, j + GB);
    subtract(tb, j);
    j += GB;
    if (!__any(j < l.y)) break;
  }
}

// p[i] for a uniform p: a scalar base and a 32-bit lane offset, so a load
// needs no per-lane 64-bit address.
__device__ __forceinline__ double at(const double *p, int i) {
  return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(p) + (unsigned)i * 8u);
}

// Eight columns from c0 of one row's entries (lane = row), loads clamped to
// the top's last column.
__device__ __forceinline__ void load_cols(double (&m)[8], const double *M, int row, int c0,
                                          int w, int nr) {
#pragma unroll
  for (int j = 0; j < 8; ++j) m[j] = at(M + (int64_t)min(c0 + j, w - 1) * nr, row);
}

// A row's diagonal and its correctly rounded reciprocal, for quotients off
// the IEEE division's long chain: with y = RN(1/d), one Newton step on a * y
// gives a quotient within one unit in the last place, and a second with its
// exact remainder the correctly rounded one (Markstein, IBM J. Res. Dev. 34,
// 1990), as long as no step leaves the normal range.  `usable` says so for
// the diagonal, in_range() for a dividend; otherwise the division is done.
struct Diag {
  double d, y;
  bool usable;
  __device__ __forceinline__ explicit Diag(double v) : d(v), y(1.0 / v), usable(in_range(v, 100)) {}
  // 2^-e <= |v| < 2^e
  static __device__ __forceinline__ bool in_range(double v, int e) {
    const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu;
    return hi - ((unsigned)(1023 - e) << 20) < ((unsigned)(2 * e) << 20);
  }
  __device__ __forceinline__ double divide(double a) const {
    const double q0 = a * y;
    const double q1 = __builtin_fma(__builtin_fma(-d, q0, a), y, q0);
    return __builtin_fma(__builtin_fma(-d, q1, a), y, q1);
  }
};

// Eight columns of a wave's own diagonal, lanes lb .. lb + B - 1 their rows
// (B < 8 in the last block only): at step j lane lb + j divides, the quotient
// is broadcast, and every later row subtracts its product; TRANS takes the
// columns from the last one.  res keeps a lane's quotient.  Lanes already
// solved, and lanes past the last column, go on computing values that nothing
// reads.  entry(j) loads m[j] again, for the block whose quotients need the
// division.
template <int KT, bool TRANS, typename Entry>
__device__ __forceinline__ void solve_block(double (&acc)[KT], double (&res)[KT],
                                            const double (&m)[8], const Diag &dg, int lb, int B,
                                            int lane, Entry entry) {
  double start[KT], num[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) {
    start[c] = acc[c];
    num[c] = 1.0;
  }
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int j = TRANS ? 7 - t : t;
    if (TRANS && j >= B) continue;
    double q[KT];
#pragma unroll
    for (int c = 0; c < KT; ++c) {
      num[c] = lane == lb + j ? acc[c] : num[c];
      q[c] = dg.divide(acc[c]);
      res[c] = lane == lb + j ? q[c] : res[c];
    }
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = acc[c] - lane_value(q[c], lb + j) * m[j];
  }
  bool ok = dg.usable;
#pragma unroll
  for (int c = 0; c < KT; ++c) ok = ok && Diag::in_range(num[c], 900);
  if (__any(lane >= lb && lane < lb + min(B, 8) && !ok)) {
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = start[c];
#pragma unroll 1
    for (int t = 0; t < min(B, 8); ++t) {
      const int j = TRANS ? min(B, 8) - 1 - t : t;
      const double mj = entry(j);
#pragma unroll
      for (int c = 0; c < KT; ++c) {
        const double q = acc[c] / dg.d;
        res[c] = lane == lb + j ? q : res[c];
        acc[c] = acc[c] - lane_value(q, lb + j) * mj;
      }
    }
  }
}

// A wave's own n <= 64 columns from column c0, the first SN_AHEAD blocks in
// buf; done(lb, B) after each block.  Rounds of SN_AHEAD full blocks take no
// branch, so the waits for their loads stay exact.
template <int KT, typename Done>
__device__ __forceinline__ void own_columns(double (&acc)[KT], double (&res)[KT],
                                            double (&buf)[SN_AHEAD][8], const Diag &dg, int c0,
                                            int n, const double *M, int row, int w, int nr,
                                            int lane, Done done) {
  auto block = [&](int b, const double (&m)[8]) {
    const int B = min(8, n - 8 * b);
    solve_block<KT, false>(acc, res, m, dg, 8 * b, B, lane, [&](int j) {
      return at(M + (int64_t)(c0 + 8 * b + j) * nr, row);
    });
    done(8 * b, B);
  };
  int b = 0;
  for (; 8 * (b + SN_AHEAD) <= n; b += SN_AHEAD) {
#pragma unroll
    for (int q = 0; q < SN_AHEAD; ++q) {
      block(b + q, buf[q]);
      load_cols(buf[q], M, row, c0 + 8 * (b + q + SN_AHEAD), w, nr);
    }
  }
#pragma unroll
  for (int q = 0; q < SN_AHEAD; ++q)
    if (8 * (b + q) < n) block(b + q, buf[q]);
}

// Rows 64g .. 64g+63 of a wide top, by one wave.  `buf` holds the first
// SN_AHEAD column blocks of the wave's rows.
template <int KT>
__device__ __forceinline__ void top_group(const SnArgs &a, const Cols<KT> &col, const double *T,
                                          double (&buf)[SN_AHEAD][8], const Diag &dg, int g,
                                          int s, int w, int nr, const double *M, double *xs,
                                          int *prog, int &seen, int lane) {
  const int row = min(64 * g + lane, w - 1);
  double acc[KT], res[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) {
    acc[c] = col.x[c][s + row];
    res[c] = 0.0;
  }
  gather_list<KT>(acc, T, a.tcount, a.list[s + row]);
  // columns of earlier groups: x from LDS as it is solved
  for (int b0 = 0; b0 < 8 * g; b0 += SN_AHEAD) {
#pragma unroll
    for (int q = 0; q < SN_AHEAD; ++q) {
      const int c0 = 8 * (b0 + q);
      lds_wait(prog, c0 + 8, seen);
      double xv[8][KT];
#pragma unroll
      for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int c = 0; c < KT; ++c) xv[j][c] = xs[(c0 + j) * KT + c];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
#pragma unroll
        for (int c = 0; c < KT; ++c) acc[c] = acc[c] - xv[j][c] * buf[q][j];
      }
      hold<KT>(acc);
      load_cols(buf[q], M, row, c0 + 8 * SN_AHEAD, w, nr);
    }
  }
  // the group's own columns
  own_columns<KT>(acc, res, buf, dg, 64 * g, min(64, w - 64 * g), M, row, w, nr, lane,
                  [&](int lb, int B) {
                    if (lane >= lb && lane < lb + B) {
#pragma unroll
                      for (int c = 0; c < KT; ++c) xs[(64 * g + lane) * KT + c] = res[c];
                    }
                    lds_publish(prog, 64 * g + lb + B, lane);
                  });
#pragma unroll
  for (int c = 0; c < KT; ++c)
    if (64 * g + lane < w && col.live[c]) st_dev(&col.x[c][s + row], res[c]);
}

// A narrow supernode (w <= SN_NARROW) by one wave: the top, then the first
// SN_NARROW_ROWS rows below, two per lane; xs is the wave's LDS.
template <int KT>
__device__ __forceinline__ void narrow_unit(const SnArgs &a, const Cols<KT> &col, double *T,
                                            int u, int tile, int i, int target, double *xs,
                                            int lane) {
  const int s = a.sup[i], w = a.sup[i + 1] - s, nr = a.nrows[i];
  const double *M = a.Lx + a.Lp[i];
  const int row = min(lane, w - 1);
  double buf[SN_AHEAD][8];
#pragma unroll
  for (int q = 0; q < SN_AHEAD; ++q) load_cols(buf[q], M, row, 8 * q, w, nr);
  const Diag dg(M[row + (int64_t)row * nr]);
  double acc[KT], res[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) {
    acc[c] = col.x[c][s + row];
    res[c] = 0.0;
  }
  const int4 list = a.list[s + row];
  int *const flags = a.flags + (int64_t)tile * a.nunits;
  wait_units(a.dptr, a.dlist, u, flags, target, a.state, a.timeout);
  gather_list<KT>(acc, T, a.tcount, list);
  own_columns<KT>(acc, res, buf, dg, 0, w, M, row, w, nr, lane, [](int, int) {});
  if (lane < w) {
#pragma unroll
    for (int c = 0; c < KT; ++c) {
      xs[lane * KT + c] = res[c];
      if (col.live[c]) st_dev(&col.x[c][s + lane], res[c]);
    }
  }
  wave_lds_sync();
  const int below = min(nr - w, SN_NARROW_ROWS);
  for (int r0 = 0; r0 < below; r0 += 64) {
    const int k = w + min(r0 + lane, below - 1);
    double t[KT];
#pragma unroll
    for (int c = 0; c < KT; ++c) t[c] = 0.0;
    int cb = 0;
    // two blocks' entries in flight, one where their x fill the registers
    constexpr int NB = KT < 4 ? 2 : 1;
    for (; w - cb >= 8 * NB; cb += 8 * NB) {
      double m[NB][8];
#pragma unroll
      for (int h = 0; h < NB; ++h) load_cols(m[h], M, k, cb + 8 * h, w, nr);
#pragma unroll
      for (int h = 0; h < NB; ++h)
#pragma unroll
        for (int c = 0; c < KT; ++c) {
          double sum = xs[(cb + 8 * h) * KT + c] * m[h][0];
#pragma unroll
          for (int j = 1; j < 8; ++j) sum = sum + xs[(cb + 8 * h + j) * KT + c] * m[h][j];
          t[c] = t[c] + sum;
        }
    }
    for (int B; cb < w; cb += B) {
      B = w - cb >= 8 ? 8 : w - cb >= 4 ? 4 : 1;
      double m[8];
      load_cols(m, M, k, cb, w, nr);
#pragma unroll
      for (int c = 0; c < KT; ++c) {
        double sum = xs[cb * KT + c] * m[0];
#pragma unroll
        for (int j = 1; j < 8; ++j)
          if (j < B) sum = sum + xs[(cb + j) * KT + c] * m[j];
        t[c] = t[c] + sum;
      }
    }
    if (r0 + lane < below) {
      const int64_t p = a.tdst[a.tb[i] + r0 + lane];
#pragma unroll
      for (int c = 0; c < KT; ++c) st_dev(&T[p + c * a.tcount], t[c]);
    }
  }
  publish_fence();
  if (lane == 0) st_dev(&flags[u], target);
  wave_lds_sync();
}

// 64 rows below a top by the workgroup: the column blocks of eight are dealt
// over the waves, NBW consecutive blocks each per pass; the block sums go to
// LDS and wave c adds column c's in block order.  The entries are loaded
// before the wait for the top.
template <int KT>
__device__ __forceinline__ void below_unit(const SnArgs &a, const Cols<KT> &col, double *T,
                                           int u, int tile, int i, int first, int target,
                                           double *xs, double *sums) {
  constexpr int NBW = 8 / KT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = a.sup[i], w = a.sup[i + 1] - s, nr = a.nrows[i];
  const double *M = a.Lx + a.Lp[i];
  const int k = min(w + first + lane, nr - 1);
  int *const flags = a.flags + (int64_t)tile * a.nunits;
  const int nb = w / 8;  // full blocks; then one of 4 where 4 are left, then single columns
  double m[NBW][8], tail[8];
#pragma unroll
  for (int h = 0; h < NBW; ++h) load_cols(m[h], M, k, 8 * (wave * NBW + h), w, nr);
  load_cols(tail, M, k, 8 * nb, w, nr);
  const int64_t place = a.tdst[a.tb[i] + k - w];
  if (wave == 0) wait_units(a.dptr, a.dlist, u, flags, target, a.state, a.timeout);
  __syncthreads();
#pragma unroll
  for (int c = 0; c < KT; ++c)
    for (int r = threadIdx.x; r < w; r += 256) xs[r * KT + c] = ld_dev(&col.x[c][s + r]);
  __syncthreads();
  double t = 0.0;  // waves 0 .. KT-1: this row's temporary of column `wave`
  int half = 0;
  for (int p = 0; p < nb; p += 4 * NBW) {
    double *const out = sums + half * (4 * NBW * KT * 64);
#pragma unroll
    for (int h = 0; h < NBW; ++h) {
      const int b = p + wave * NBW + h;
      if (b < nb) {
#pragma unroll
        for (int c = 0; c < KT; ++c) {
          double sum = xs[8 * b * KT + c] * m[h][0];
#pragma unroll
          for (int j = 1; j < 8; ++j) sum = sum + xs[(8 * b + j) * KT + c] * m[h][j];
          out[((wave * NBW + h) * KT + c) * 64 + lane] = sum;
        }
      }
    }
    if (p + 4 * NBW < nb) {
#pragma unroll
      for (int h = 0; h < NBW; ++h)
        load_cols(m[h], M, k, 8 * (p + (4 + wave) * NBW + h), w, nr);
    }
    __syncthreads();
    if (wave < KT) {
      const int cnt = min(4 * NBW, nb - p);
      for (int b = 0; b < cnt; ++b) t = t + out[(b * KT + wave) * 64 + lane];
    }
    half ^= 1;
  }
  if (wave < KT) {
    int cb = 8 * nb, q = 0;
    if (w - cb >= 4) {
      double sum = xs[cb * KT + wave] * tail[0];
#pragma unroll
      for (int j = 1; j < 4; ++j) sum = sum + xs[(cb + j) * KT + wave] * tail[j];
      t = t + sum;
      q = 4;
    }
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (j >= q && cb + j < w) t = t + xs[(cb + j) * KT + wave] * tail[j];
    if (w + first + lane < nr) st_dev(&T[place + wave * a.tcount], t);
    publish_fence();
  }
  __syncthreads();
  if (threadIdx.x == 0) st_dev(&flags[u], target);
}

// Workgroup's next (ticket, column tile), ticket-major; -1 past the last.
__device__ __forceinline__ int next_ticket(const SnArgs &a, int *slot) {
  __syncthreads();
  if (threadIdx.x == 0) {
    slot[0] = atomicAdd(&a.state[ST_TICKET], 1);
    slot[1] = 0;
  }
  __syncthreads();
  const int tt = __builtin_amdgcn_readfirstlane(slot[0]);
  return tt < a.ntick * a.tiles ? tt : -1;
}

template <int KT>
__global__ __launch_bounds__(256, 2) void k_supernodal(SnArgs a) {
  __shared__ double xs[SN_WMAX * KT];
  __shared__ double sums[2 * 4 * 8 * 64];
  __shared__ int slot[2];  // the ticket; columns solved of the current top
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int target = ld_dev(&a.state[ST_EPOCH]) + 1;
  for (;;) {
    const int tt = next_ticket(a, slot);
    if (tt < 0) break;
    const int tk = tt / a.tiles, tile = tt - tk * a.tiles;
    const Cols<KT> col(a, tile);
    double *const T = a.T + (int64_t)tile * a.tcount * KT;
    const int u0 = a.tick[tk], u1 = a.tick[tk + 1];
    const int2 un = a.unit[u0];
    const int i = __builtin_amdgcn_readfirstlane(un.x);
    const int chunk = __builtin_amdgcn_readfirstlane(un.y);
    const int w = a.sup[i + 1] - a.sup[i];
    if (chunk > 0) {
      const int first = (w <= SN_NARROW ? SN_NARROW_ROWS : 0) + (chunk - 1) * 64;
      below_unit<KT>(a, col, T, u0, tile, i, first, target, xs, sums);
    } else if (w <= SN_NARROW) {
      if (u0 + wave < u1) {
        const int node = __builtin_amdgcn_readfirstlane(a.unit[u0 + wave].x);
        narrow_unit<KT>(a, col, T, u0 + wave, tile, node, target, xs + wave * 64 * KT, lane);
      }
    } else {
      const int s = a.sup[i], nr = a.nrows[i];
      const double *M = a.Lx + a.Lp[i];
      int *const flags = a.flags + (int64_t)tile * a.nunits;
      int seen = 0;
      for (int g = wave; g < 4 || 64 * g < w; g += 4) {
        const int row = min(64 * g + lane, w - 1);
        double buf[SN_AHEAD][8];
#pragma unroll
        for (int q = 0; q < SN_AHEAD; ++q) load_cols(buf[q], M, row, 8 * q, w, nr);
        const Diag dg(M[row + (int64_t)row * nr]);
        if (g < 4) {  // each wave's first group: the entries are on their way
          if (wave == 0) wait_units(a.dptr, a.dlist, u0, flags, target, a.state, a.timeout);
          __syncthreads();
        }
        if (64 * g < w) top_group<KT>(a, col, T, buf, dg, g, s, w, nr, M, xs, &slot[1], seen, lane);
      }
      publish_fence();
      __syncthreads();
      if (threadIdx.x == 0) st_dev(&flags[u0], target);
    }
  }
  persistent_finish(a.state, a.total_waves);
}

// ---------------------------------------------------- transposed solve
// L^T x = b on the same storage (the semantics of parsy's blockedLTsolve,
// sparse_blas/parsy/triangularSolve/Triangular_BCSC.cpp:125-186), tickets
// level by level from the root.  Per supernode: for each top column c, t =
// sum over the rows below, ascending, of M[r, c] times x at that row, and
// x[s+c] -= t; then the top's transposed solve from its last column: x_c /=
// M[c, c] and every x_r, r < c, loses M[c, r] * x_c.  The order is the
// oracle's (orc_sptrsv_csc_block_t).
//
// A narrow supernode with at most SN_NARROW_ROWS rows below is one wave's
// work, four to a ticket.  Otherwise 64 of its columns' sums over the rows
// below are a ticket (the workgroup: tiles of 64 x 64 entries are loaded
// along the rows, coalesced, and turned in LDS so that a lane then owns a
// column), and its top another (waves take groups of 64 columns from the
// last one, hand x on through LDS as in the forward solve, and wait for
// their own group's sums only).

// Rows r0 .. r0+7 of one column's entries (lane = column; the pointer is at
// its row 0); rows past `last` repeat it.
__device__ __forceinline__ void load_rows(double (&m)[8], const double *C, int r0, int last) {
  if (r0 + 7 <= last) {
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = C[r0 + j];
  } else {
#pragma unroll
    for (int j = 0; j < 8; ++j) m[j] = C[max(min(r0 + j, last), 0)];
  }
}

// Columns 64g .. 64g+63 of a top, by one wave: x from LDS for the columns of
// later groups (xs and the count are not used by a narrow supernode, whose
// only group is the last).
template <int KT>
__device__ __forceinline__ void top_group_t(double (&acc)[KT], double (&res)[KT],
                                            double (&buf)[SN_AHEAD][8], const Diag &dg, int g,
                                            int w, int nr, const double *M, double *xs,
                                            int *prog, int &seen, int lane) {
  const double *C = M + (int64_t)min(64 * g + lane, w - 1) * nr;
  const int top = (w - 1) / 8;  // last block of eight rows
#pragma unroll
  for (int c = 0; c < KT; ++c) res[c] = 0.0;
  int b = top;
  auto later = [&](double (&m)[8]) {
    const int c0 = 8 * b, B = min(8, w - c0);
    lds_wait(prog, w - c0, seen);
    double xv[8][KT];
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int c = 0; c < KT; ++c) xv[j][c] = xs[min(c0 + j, w - 1) * KT + c];
#pragma unroll
    for (int j = 7; j >= 0; --j)
      if (j < B) {
#pragma unroll
        for (int c = 0; c < KT; ++c) acc[c] = acc[c] - m[j] * xv[j][c];
      }
    hold<KT>(acc);
  };
  auto own = [&](double (&m)[8]) {
    const int c0 = 8 * b, lb = c0 - 64 * g;
    solve_block<KT, true>(acc, res, m, dg, lb, w - c0, lane,
                          [&](int j) { return C[c0 + j]; });
    if (xs) {
      if (lane >= lb && lane < lb + 8 && 64 * g + lane < w) {
#pragma unroll
        for (int c = 0; c < KT; ++c) xs[(64 * g + lane) * KT + c] = res[c];
      }
      lds_publish(prog, w - c0, lane);
    }
  };
  // SN_AHEAD blocks per round, slot q of round n holding block top - 4n - q
  for (int b0 = top; b0 >= 8 * g; b0 -= SN_AHEAD) {
#pragma unroll
    for (int q = 0; q < SN_AHEAD; ++q) {
      b = b0 - q;
      if (b >= 8 * g) {
        if (b >= 8 * g + 8)
          later(buf[q]);
        else
          own(buf[q]);
      }
      load_rows(buf[q], C, max(8 * (b - SN_AHEAD), 0), nr - 1);
    }
  }
}

__device__ __forceinline__ void preload_t(double (&buf)[SN_AHEAD][8], const double *M, int g,
                                          int w, int nr, int lane) {
  const double *C = M + (int64_t)min(64 * g + lane, w - 1) * nr;
  const int top = (w - 1) / 8;
#pragma unroll
  for (int q = 0; q < SN_AHEAD; ++q) load_rows(buf[q], C, max(8 * (top - q), 0), nr - 1);
}

template <int KT>
__device__ __forceinline__ void narrow_unit_t(const SnArgs &a, const Cols<KT> &col, int u,
                                              int tile, int i, int target, int lane) {
  const int s = a.sup[i], w = a.sup[i + 1] - s, nr = a.nrows[i], below = nr - w;
  const double *M = a.Lx + a.Lp[i];
  const int *rows = a.rowb + a.tb[i];
  const int c = min(lane, w - 1);
  double buf[SN_AHEAD][8];
  preload_t(buf, M, 0, w, nr, lane);
  const Diag dg(M[c + (int64_t)c * nr]);
  double acc[KT], res[KT], t[KT];
#pragma unroll
  for (int q = 0; q < KT; ++q) {
    acc[q] = col.x[q][s + c];
    t[q] = 0.0;
  }
  const double *C = M + (int64_t)c * nr + w;
  int *const flags = a.flags + (int64_t)tile * a.nunits;
  double ma[8], mb[8];
  if (below > 0) {
    load_rows(ma, C, 0, below - 1);
    wait_units(a.dptr, a.dlist, u, flags, target, a.state, a.timeout);
    for (int r0 = 0; r0 < below; r0 += 64) {
      double xr[KT];
      const int row = rows[min(r0 + lane, below - 1)];
#pragma unroll
      for (int q = 0; q < KT; ++q) xr[q] = ld_dev(&col.x[q][row]);
      auto add = [&](const double (&m)[8], int r) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (r + j < below) {
#pragma unroll
            for (int q = 0; q < KT; ++q) {
              const double p = m[j] * lane_value(xr[q], (r + j) & 63);
              t[q] = r + j == 0 ? p : t[q] + p;
            }
          }
      };
      const int end = min(r0 + 64, below);
      for (int r = r0; r < end; r += 16) {
        load_rows(mb, C, min(r + 8, below - 1), below - 1);
        add(ma, r);
        load_rows(ma, C, min(r + 16, below - 1), below - 1);
        if (r + 8 < end) add(mb, r + 8);
      }
    }
#pragma unroll
    for (int q = 0; q < KT; ++q) acc[q] = acc[q] - t[q];
  }
  int seen = 0;
  top_group_t<KT>(acc, res, buf, dg, 0, w, nr, M, nullptr, nullptr, seen, lane);
#pragma unroll
  for (int q = 0; q < KT; ++q)
    if (lane < w && col.live[q]) st_dev(&col.x[q][s + lane], res[q]);
  publish_fence();
  if (lane == 0) st_dev(&flags[u], target);
}

constexpr int SN_PITCH = 65;  // doubles per column of a turned tile (no bank conflicts)

// The sums over the rows below of columns 64g .. 64g+63, by the workgroup.
// Tiles of 64 rows; wave v loads 16 columns of a tile along its rows, the
// next tile's entries and x in flight while this one is summed; wave c then
// adds right-hand side c's products, a lane per column.
template <int KT>
__device__ __forceinline__ void below_unit_t(const SnArgs &a, int u, int tile, int i, int g,
                                             int target, double *turn, double *xrow) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = a.sup[i], w = a.sup[i + 1] - s, nr = a.nrows[i], below = nr - w;
  const double *M = a.Lx + a.Lp[i] + w;
  const int *rows = a.rowb + a.tb[i];
  int *const flags = a.flags + (int64_t)tile * a.nunits;
  double m[16];
  auto load = [&](int r0) {
    const int r = min(r0 + lane, below - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      m[j] = at(M + (int64_t)min(64 * g + 16 * wave + j, w - 1) * nr, r);
  };
  load(0);
  int row = rows[min(lane, below - 1)];
  if (wave == 0) wait_units(a.dptr, a.dlist, u, flags, target, a.state, a.timeout);
  __syncthreads();
  // wave c of the first KT holds x of right-hand side c at the tile's rows
  const int cw = tile * KT + wave;
  double *const xc = a.x + (int64_t)min(cw, a.k - 1) * a.ldx;
  const bool mine = cw < a.k;
  double xr = wave < KT ? ld_dev(&xc[row]) : 0.0;
  double t = 0.0;
  int half = 0;
  for (int r0 = 0; r0 < below; r0 += 64) {
    double *const tl = turn + half * 64 * SN_PITCH;
    double *const xl = xrow + (half * KT + min(wave, KT - 1)) * 64;
#pragma unroll
    for (int j = 0; j < 16; ++j) tl[(16 * wave + j) * SN_PITCH + lane] = m[j];
    if (wave < KT) xl[lane] = xr;
    if (r0 + 64 < below) {
      load(r0 + 64);
      row = rows[min(r0 + 64 + lane, below - 1)];
      if (wave < KT) xr = ld_dev(&xc[row]);
    }
    __syncthreads();
    if (wave < KT) {
      const int cnt = min(64, below - r0);
      int r = 0;
      if (r0 == 0) {
        t = tl[lane * SN_PITCH] * xl[0];
        r = 1;
      }
      for (; r + 8 <= cnt; r += 8) {
        double p[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) p[j] = tl[lane * SN_PITCH + r + j] * xl[r + j];
#pragma unroll
        for (int j = 0; j < 8; ++j) t = t + p[j];
      }
      for (; r < cnt; ++r) t = t + tl[lane * SN_PITCH + r] * xl[r];
    }
    half ^= 1;
  }
  if (wave < KT) {
    const int c = 64 * g + lane;
    if (c < w && mine) st_dev(&xc[s + c], xc[s + c] - t);
    publish_fence();
  }
  __syncthreads();
  if (threadIdx.x == 0) st_dev(&flags[u], target);
}

template <int KT>
__global__ __launch_bounds__(256, 2) void k_supernodal_t(SnArgs a) {
  // a top's x, or two turned tiles and the x at their rows
  constexpr int TILES = 2 * 64 * SN_PITCH + 2 * KT * 64;
  __shared__ double mem[SN_WMAX * KT > TILES ? SN_WMAX * KT : TILES];
  __shared__ int slot[2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int target = ld_dev(&a.state[ST_EPOCH]) + 1;
  for (;;) {
    const int tt = next_ticket(a, slot);
    if (tt < 0) break;
    const int tk = tt / a.tiles, tile = tt - tk * a.tiles;
    const Cols<KT> col(a, tile);
    const int u0 = a.tick[tk], u1 = a.tick[tk + 1];
    const int2 un = a.unit[u0];
    const int i = __builtin_amdgcn_readfirstlane(un.x);
    const int chunk = __builtin_amdgcn_readfirstlane(un.y);
    const int s = a.sup[i], w = a.sup[i + 1] - s, nr = a.nrows[i];
    int *const flags = a.flags + (int64_t)tile * a.nunits;
    if (chunk > 0) {
      below_unit_t<KT>(a, u0, tile, i, chunk - 1, target, mem, mem + 2 * 64 * SN_PITCH);
    } else if (w <= SN_NARROW && nr - w <= SN_NARROW_ROWS) {
      if (u0 + wave < u1) {
        const int node = __builtin_amdgcn_readfirstlane(a.unit[u0 + wave].x);
        narrow_unit_t<KT>(a, col, u0 + wave, tile, node, target, lane);
      }
    } else {
      const double *M = a.Lx + a.Lp[i];
      const int G = (w + 63) / 64, ub = a.tbelow[i];
      int seen = 0;
      for (int g = G - 1 - wave; g >= 0; g -= 4) {
        double buf[SN_AHEAD][8];
        preload_t(buf, M, g, w, nr, lane);
        const int c = min(64 * g + lane, w - 1);
        const Diag dg(M[c + (int64_t)c * nr]);
        if (ub >= 0)
          wait_flag(&flags[ub + g], target, a.state, a.timeout);
        double acc[KT], res[KT];
#pragma unroll
        for (int q = 0; q < KT; ++q) acc[q] = ld_dev(&col.x[q][s + c]);
        top_group_t<KT>(acc, res, buf, dg, g, w, nr, M, mem, &slot[1], seen, lane);
#pragma unroll
        for (int q = 0; q < KT; ++q)
          if (64 * g + lane < w && col.live[q]) st_dev(&col.x[q][s + c], res[q]);
      }
      publish_fence();
      __syncthreads();
      if (threadIdx.x == 0) st_dev(&flags[u0], target);
    }
  }
  persistent_finish(a.state, a.total_waves);
}

}  // namespace

namespace {

// Units and tickets of one direction, level by level.  Per level: the column
// groups of the wide supernodes (transposed only; they come before the top
// that uses them), the wide tops, the narrow supernodes four to a ticket, and
// the further rows below (forward only, 64 per unit).
struct SnSchedule {
  std::vector<int2> unit;  // (supernode, 0 or 1 + chunk)
  std::vector<int> tick;   // unit bounds per ticket
  std::vector<int> top;    // per supernode: the unit that solves its top
  std::vector<int> first;  // per supernode: its first chunk unit, or -1
};

void sn_schedule(int m, const int *h_sup, const std::vector<int> &lev,
                 const std::vector<int> &tb, bool transposed, SnSchedule &s) {
  std::vector<int> order(m);
  for (int i = 0; i < m; ++i) order[i] = transposed ? m - 1 - i : i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return lev[x] < lev[y]; });
  s.tick.assign(1, 0);
  s.top.assign(m, -1);
  s.first.assign(m > 0 ? m : 1, -1);
  auto width = [&](int i) { return h_sup[i + 1] - h_sup[i]; };
  auto below = [&](int i) { return tb[i + 1] - tb[i]; };
  auto narrow = [&](int i) {
    return width(i) <= SN_NARROW && (!transposed || below(i) <= SN_NARROW_ROWS);
  };
  auto close = [&] { s.tick.push_back((int)s.unit.size()); };
  auto chunks = [&](int i, int count) {
    for (int c = 0; c < count; ++c) {
      if (c == 0) s.first[i] = (int)s.unit.size();
      s.unit.push_back(make_int2(i, c + 1));
      close();
    }
  };
  for (int a = 0, b = 0; a < m; a = b) {
    while (b < m && lev[order[b]] == lev[order[a]]) ++b;
    if (transposed)
      for (int j = a; j < b; ++j)
        if (!narrow(order[j]) && below(order[j]) > 0) chunks(order[j], (width(order[j]) + 63) / 64);
    for (int j = a; j < b; ++j)
      if (!narrow(order[j])) {
        s.top[order[j]] = (int)s.unit.size();
        s.unit.push_back(make_int2(order[j], 0));
        close();
      }
    int open = 0;
    for (int j = a; j < b; ++j)
      if (narrow(order[j])) {
        s.top[order[j]] = (int)s.unit.size();
        s.unit.push_back(make_int2(order[j], 0));
        if (++open == 4) {
          close();
          open = 0;
        }
      }
    if (open) close();
    if (!transposed)
      for (int j = a; j < b; ++j) {
        const int i = order[j], rest = below(i) - (narrow(i) ? SN_NARROW_ROWS : 0);
        if (rest > 0) chunks(i, (rest + 63) / 64);
      }
  }
}

void flatten_deps(std::vector<std::vector<int>> &deps, std::vector<int> &ptr,
                  std::vector<int> &list) {
  ptr.assign(1, 0);
  list.clear();
  for (std::vector<int> &d : deps) {
    std::sort(d.begin(), d.end());
    d.erase(std::unique(d.begin(), d.end()), d.end());
    list.insert(list.end(), d.begin(), d.end());
    ptr.push_back((int)list.size());
  }
}

}  // namespace

int sn_analyze(symamd_handle h, int n, int m, const int *h_sup, const int *h_nrows,
               const int *h_Lp, const int *h_Li, symamd_snplan_s **out) {
  if (n < 0 || m < 0 || (m > 0 && (!h_sup || !h_nrows || !h_Lp || !h_Li)))
    return fail(SYMAMD_ERR_INVALID_ARG, "supernodal analyze: bad arguments");
  if (m == 0 && n > 0)
    return fail(SYMAMD_ERR_STRUCTURE, "supernodal analyze: no supernodes for %d columns", n);
  if (m > 0 && (h_sup[0] != 0 || h_sup[m] != n))
    return fail(SYMAMD_ERR_STRUCTURE, "supernodes must cover columns 0 .. n-1");
  std::vector<int> tb(m + 1, 0), cnt(n + 1, 0);
  for (int i = 0; i < m; ++i) {
    const int s = h_sup[i], w = h_sup[i + 1] - s, nr = h_nrows[i];
    if (w < 1 || nr < w)
      return fail(SYMAMD_ERR_STRUCTURE, "supernode %d: width %d, %d rows", i, w, nr);
    if (w > SN_WMAX)
      return fail(SYMAMD_ERR_NOT_SUPPORTED, "supernode %d is %d columns wide (at most %d)", i,
                  w, SN_WMAX);
    if (i > 0 && h_Lp[i] < h_Lp[i - 1] + (int64_t)h_nrows[i - 1] * (h_sup[i] - h_sup[i - 1]))
      return fail(SYMAMD_ERR_STRUCTURE, "supernode %d's values overlap the previous block", i);
    // the rows below the top must lie below the supernode (the top's own
    // row ids are not read, as in the reference)
    for (int r = w; r < nr; ++r) {
      const int row = h_Li[h_Lp[i] + r];
      if (row < s + w || row >= n)
        return fail(SYMAMD_ERR_STRUCTURE, "supernode %d: block row %d is row %d", i, r, row);
      cnt[row + 1]++;
    }
    tb[i + 1] = tb[i] + (nr - w);
  }
  for (int r = 0; r < n; ++r) cnt[r + 1] += cnt[r];
  // the rows' lists, in ascending supernode order, and the place in T of each
  // row below: entry j of the rows one wave gathers (64 consecutive ones of a
  // supernode) lies side by side, lists padded to the longest; rows of very
  // uneven lists (padding past three entries in four) keep theirs contiguous
  std::vector<int> tdst(tb[m] > 0 ? tb[m] : 1), rowb(tb[m] > 0 ? tb[m] : 1);
  std::vector<int4> list(n > 0 ? n : 1, make_int4(0, 0, 0, 0));
  int64_t tcount = 0;
  for (int i = 0; i < m; ++i)
    for (int r0 = h_sup[i]; r0 < h_sup[i + 1]; r0 += 64) {
      const int r1 = std::min(r0 + 64, h_sup[i + 1]);
      const int64_t total = cnt[r1] - cnt[r0];
      int64_t longest = 0;
      for (int r = r0; r < r1; ++r) longest = std::max<int64_t>(longest, cnt[r + 1] - cnt[r]);
      const bool side = longest * (r1 - r0) <= 4 * total;
      for (int r = r0; r < r1; ++r)
        if (cnt[r + 1] > cnt[r])
          list[r] = make_int4((int)(tcount + (side ? r - r0 : cnt[r] - cnt[r0])), 0,
                              side ? r1 - r0 : 1, 0);
      tcount += side ? longest * (r1 - r0) : total;
      if (tcount > INT_MAX)
        return fail(SYMAMD_ERR_NOT_SUPPORTED, "supernodal analyze: over 2^31 temporaries");
    }
  std::vector<int> owner(n);
  for (int i = 0; i < m; ++i)
    for (int c = h_sup[i]; c < h_sup[i + 1]; ++c) owner[c] = i;
  // levels (a supernode is one above the highest of the supernodes writing
  // to its rows; transposed: one below the deepest of the supernodes owning
  // its rows below): tickets are dealt level by level, so every leaf is taken
  // before any supernode that waits, and every unit waits only for units
  // dealt before it
  std::vector<int> lev(m, 0), tlev(m, 0);
  int old_tasks = 0;
  for (int i = 0; i < m; ++i) {
    const int w = h_sup[i + 1] - h_sup[i];
    for (int k = 0; k < h_nrows[i] - w; ++k) {
      const int row = h_Li[h_Lp[i] + w + k];
      rowb[tb[i] + k] = row;
      tdst[tb[i] + k] = list[row].x + list[row].y++ * list[row].z;
      lev[owner[row]] = std::max(lev[owner[row]], lev[i] + 1);
    }
    old_tasks += std::max(1, (h_nrows[i] - w + 127) / 128);
  }
  for (int i = m - 1; i >= 0; --i)
    for (int k = tb[i]; k < tb[i + 1]; ++k) tlev[i] = std::max(tlev[i], tlev[owner[rowb[k]]] + 1);
  SnSchedule fwd, bwd;
  sn_schedule(m, h_sup, lev, tb, false, fwd);
  sn_schedule(m, h_sup, tlev, tb, true, bwd);
  // forward: a top waits for the units that write its rows' temporaries, a
  // chunk of the rows below for its top
  std::vector<std::vector<int>> deps(fwd.unit.size());
  for (int i = 0; i < m; ++i) {
    const int head = h_sup[i + 1] - h_sup[i] <= SN_NARROW ? SN_NARROW_ROWS : 0;
    for (int k = 0; k < tb[i + 1] - tb[i]; ++k) {
      const int producer = k < head ? fwd.top[i] : fwd.first[i] + (k - head) / 64;
      std::vector<int> &d = deps[fwd.top[owner[rowb[tb[i] + k]]]];
      if (d.empty() || d.back() != producer) d.push_back(producer);
    }
  }
  for (size_t u = 0; u < fwd.unit.size(); ++u)
    if (fwd.unit[u].y > 0) deps[u].push_back(fwd.top[fwd.unit[u].x]);
  std::vector<int> dptr, dlist, tdptr, tdlist;
  flatten_deps(deps, dptr, dlist);
  // transposed: the units that read x at the rows below (a narrow supernode,
  // the column groups of a wide one) wait for the tops of their owners; a
  // wide top waits for its own groups by tag
  deps.assign(bwd.unit.size(), {});
  for (size_t u = 0; u < bwd.unit.size(); ++u) {
    const int i = bwd.unit[u].x;
    if (bwd.unit[u].y == 0 && bwd.first[i] >= 0) continue;
    std::vector<int> &d = deps[u];
    for (int k = tb[i]; k < tb[i + 1]; ++k) {
      const int o = bwd.top[owner[rowb[k]]];
      if (d.empty() || d.back() != o) d.push_back(o);
    }
  }
  flatten_deps(deps, tdptr, tdlist);
  auto *q = new symamd_snplan_s();
  q->n = n;
  q->m = m;
  q->tcount = tcount;
  q->ntasks = old_tasks;
  q->units = (int)fwd.unit.size();
  q->tickets = (int)fwd.tick.size() - 1;
  q->tunits = (int)bwd.unit.size();
  q->ttickets = (int)bwd.tick.size() - 1;
  const int64_t flags = std::max(1, std::max(q->units, q->tunits));
  int rc = SYMAMD_OK;
  auto up = [&](int **dst, const int *src, size_t count) {
    if (rc != SYMAMD_OK) return;
    if (hipMalloc(dst, sizeof(int) * (count ? count : 1)) != hipSuccess ||
        (count && hipMemcpy(*dst, src, sizeof(int) * count, hipMemcpyHostToDevice) != hipSuccess))
      rc = fail(SYMAMD_ERR_ALLOC, "supernodal plan upload failed");
  };
  up(&q->d_sup, h_sup, m + 1);
  up(&q->d_nrows, h_nrows, m);
  up(&q->d_Lp, h_Lp, m + 1);
  up(&q->d_tb, tb.data(), m + 1);
  up(&q->d_list, reinterpret_cast<const int *>(list.data()), 4 * (size_t)n);
  up(&q->d_tdst, tdst.data(), tb[m]);
  up(&q->d_rowb, rowb.data(), tb[m]);
  up(&q->d_unit, reinterpret_cast<const int *>(fwd.unit.data()), 2 * fwd.unit.size());
  up(&q->d_tick, fwd.tick.data(), fwd.tick.size());
  up(&q->d_dptr, dptr.data(), dptr.size());
  up(&q->d_dlist, dlist.data(), dlist.size());
  up(&q->d_tunit, reinterpret_cast<const int *>(bwd.unit.data()), 2 * bwd.unit.size());
  up(&q->d_ttick, bwd.tick.data(), bwd.tick.size());
  up(&q->d_tdptr, tdptr.data(), tdptr.size());
  up(&q->d_tdlist, tdlist.data(), tdlist.size());
  up(&q->d_tbelow, bwd.first.data(), m);
  if (rc == SYMAMD_OK &&
      (hipMalloc(&q->d_T, sizeof(double) * (q->tcount > 0 ? q->tcount : 1)) != hipSuccess ||
       hipMalloc(&q->d_flags, sizeof(int) * flags) != hipSuccess ||
       hipMalloc(&q->d_state, sizeof(int) * ST_WORDS) != hipSuccess ||
       hipMemset(q->d_flags, 0, sizeof(int) * flags) != hipSuccess ||
       hipMemset(q->d_state, 0, sizeof(int) * ST_WORDS) != hipSuccess))
    rc = fail(SYMAMD_ERR_ALLOC, "supernodal plan allocation failed");
  if (rc != SYMAMD_OK) {
    sn_destroy(q);
    return rc;
  }
  (void)h;
  *out = q;
  return SYMAMD_OK;
}

int sn_solve(symamd_handle h, symamd_snplan_s *q, const double *d_Lx, double *d_x, int k,
             int64_t ldx, bool transposed) {
  if (q->m == 0 || k == 0) return SYMAMD_OK;
  // tickets run over (task, column) pairs in 32-bit counters
  if ((int64_t)q->ntasks * k >= (int64_t)INT_MAX)
    return fail(SYMAMD_ERR_NOT_SUPPORTED,
                "supernodal solve: %d tasks x %d columns exceed the 32-bit ticket range; "
                "solve the columns in smaller batches", q->ntasks, k);
  // columns per tile: a row's entries are loaded once for the columns of a
  // tile, but each step of a top's chain then divides for all of them.  On
  // the 13-level factor, forward + transposed with tiles of 1 / 2 / 4: k = 2
  // 1.19 / 1.29 / - ms, k = 4 1.46 / 1.38 / 1.73 ms, k = 32 5.86 / 3.57 /
  // 3.21 ms.
  const int kt = k < 4 ? 1 : k < 16 ? 2 : 4;
  const int tiles = (k + kt - 1) / kt;
  // temporaries and tags for the tiles' columns
  if (tiles * kt > q->kcap) {
    double *T = nullptr;
    int *flags = nullptr;
    const int64_t cols = (int64_t)tiles * kt;
    const int64_t tc = q->tcount > 0 ? q->tcount : 1;
    const int64_t nt = std::max(1, std::max(q->units, q->tunits));
    if (hipMalloc(&T, sizeof(double) * tc * cols) != hipSuccess ||
        hipMalloc(&flags, sizeof(int) * nt * cols) != hipSuccess) {
      if (T) (void)hipFree(T);
      return fail(SYMAMD_ERR_ALLOC, "supernodal temporaries for %d columns", k);
    }
    // cleared tags read as "not ready" in every epoch
    SYMAMD_HIP(hipMemsetAsync(flags, 0, sizeof(int) * nt * cols, h->stream));
    SYMAMD_HIP(hipStreamSynchronize(h->stream));
    if (q->d_T) (void)hipFree(q->d_T);
    if (q->d_flags) (void)hipFree(q->d_flags);
    q->d_T = T;
    q->d_flags = flags;
    q->kcap = (int)cols;
  }
  SnArgs a;
  a.sup = q->d_sup;
  a.nrows = q->d_nrows;
  a.Lp = q->d_Lp;
  a.Lx = d_Lx;
  a.x = d_x;
  a.T = q->d_T;
  a.tb = q->d_tb;
  a.tdst = q->d_tdst;
  a.list = reinterpret_cast<const int4 *>(q->d_list);
  a.unit = reinterpret_cast<const int2 *>(transposed ? q->d_tunit : q->d_unit);
  a.tick = transposed ? q->d_ttick : q->d_tick;
  a.dptr = transposed ? q->d_tdptr : q->d_dptr;
  a.dlist = transposed ? q->d_tdlist : q->d_dlist;
  a.nunits = transposed ? q->tunits : q->units;
  a.ntick = transposed ? q->ttickets : q->tickets;
  a.rowb = q->d_rowb;
  a.tbelow = q->d_tbelow;
  a.flags = q->d_flags;
  a.state = q->d_state;
  a.k = k;
  a.tiles = tiles;
  a.ldx = ldx;
  a.tcount = q->tcount > 0 ? q->tcount : 1;
  a.timeout = h->timeout_ticks();
  void (*const kfn)(SnArgs) =
      transposed ? (kt == 1 ? k_supernodal_t<1> : kt == 2 ? k_supernodal_t<2> : k_supernodal_t<4>)
                 : (kt == 1 ? k_supernodal<1> : kt == 2 ? k_supernodal<2> : k_supernodal<4>);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)kfn, 256, 0) !=
          hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  // tickets are dealt in order, so any grid size is safe
  const int64_t grid = std::min((int64_t)per_cu * h->num_cus, (int64_t)a.ntick * tiles);
  a.total_waves = (int)grid * 4;
  kfn<<<(unsigned)grid, 256, 0, h->stream>>>(a);
  SYMAMD_HIP(hipGetLastError());
  return SYMAMD_OK;
}

int sn_check(symamd_handle h, symamd_snplan_s *q) {
  int st[ST_WORDS];
  SYMAMD_HIP(hipStreamSynchronize(h->stream));
  SYMAMD_HIP(hipMemcpy(st, q->d_state, sizeof(st), hipMemcpyDeviceToHost));
  if (st[ST_ERROR]) return fail(SYMAMD_ERR_TIMEOUT, "a supernodal wait exceeded the watchdog");
  return SYMAMD_OK;
}

void sn_destroy(symamd_snplan_s *q) {
  if (!q) return;
  void *ptrs[] = {q->d_sup,  q->d_nrows, q->d_Lp,    q->d_tb,     q->d_list,  q->d_tdst,
                  q->d_rowb, q->d_unit,  q->d_tick,  q->d_dptr,   q->d_dlist, q->d_tunit,
                  q->d_ttick, q->d_tdptr, q->d_tdlist, q->d_tbelow, q->d_T,   q->d_flags,
                  q->d_state};
  for (void *x : ptrs)
    if (x) (void)hipFree(x);
  delete q;
}

}  // namespace symamd
