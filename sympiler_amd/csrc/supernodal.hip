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
// What bounds it: the chain of tree levels, for one right-hand side and the
// last levels of a block: for each, the hand-offs between its units (gather,
// top, rows below) and the widest top's columns (about 70 clocks, 29 ns, each:
// two Newton steps for the quotient, a broadcast, a multiply and a subtract;
// the 2,734 columns on the 13-level factor's longest path are a quarter of its
// forward solve).  A top's rows lie one per
// lane, 64 to a wave, and each wave streams its rows' entries with SN_AHEAD
// column blocks in flight; the wave whose rows are next solves its 64 columns
// with lane broadcasts and hands x on through LDS, block of 8 by block of 8,
// while the other waves subtract.  Long lists of temporaries are gathered by
// workgroups of their own ahead of the top.
// Measured on the 13-level nested-dissection-shaped factor (8,191 supernodes
// up to 512 wide, 36 M values), forward + transposed, in ms: one right-hand
// side 1.36 + 3.06 with one wavefront per top, 0.45 + 0.65 with a workgroup,
// 0.32 + 0.43 with the quotients from reciprocals, the whole diagonal block
// in flight, gathered lists and turned tiles; 32 right-hand sides 4.6 + 6.9,
// 1.71 + 1.50, 1.34 + 1.27.
#include <algorithm>
#include <map>
#include <vector>

#include "device.h"

namespace symamd {

namespace {

// Column blocks of 8 whose entries are in flight: a wave's own 64 columns,
// whose chain (about 29 ns a column) runs ahead of any load issued during it.
constexpr int SN_AHEAD = 8;

// One unit, read in one scalar load: the supernode's first column, width and
// block rows, its values at Lx[p], its rows below at tdst / rowb[tb], and the
// slots it waits for, dlist[d0 .. d0 + dn).  kind: SN_NARROW_UNIT, SN_TOP, or
// first row below / column group of a chunk, or SN_GATHER_UNIT - row group.  A
// top whose row groups are gathered, and a transposed top, waits for the slots
// d0 + 4g of its groups (dn < 0).  w = 0: no unit.
struct SnUnit {
  int s, w, nr, kind, p, tb, d0, dn;
};
constexpr int SN_GATHER_UNIT = -3, SN_NARROW_UNIT = -2, SN_TOP = -1;

struct SnArgs {
  const SnUnit *unit;           // slots 4t .. 4t+3: the units of ticket t
  const double *Lx;
  double *x;                    // right-hand side in, solution out
  double *T;                    // temporaries, placed where the rows' lists are read
  const int *tdst;              // place in T of each row below
  const int4 *list;             // row r subtracts T[x + j*z], j < y
  const int *dlist;             // slots that a unit waits for
  int *flags, *state;           // one tag per (column tile, slot)
  int ntick, total_waves;
  const int *rowb;              // transposed: rows below
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

// The values are computed (and loads they come from waited for) here.  After
// a block's subtractions: the compiler would move them past the wait for the
// next block and keep their operands in registers until there.  Before a loop
// that loads ahead: a load that may still be pending on its entry makes every
// round wait for all of its loads.
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
template <int KT, int GB>
__device__ __forceinline__ void gather_list(double (&v)[KT], const double *T, int64_t tcount,
                                            const int4 &l) {
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
// the IEEE division's longer chain: with y = RN(1/d), one Newton step on a * y
// gives a quotient within one unit in the last place, and a second with its
// exact remainder the correctly rounded one (Markstein, IBM J. Res. Dev. 34,
// 1990), as long as no step leaves the normal range.  usable says so for the
// diagonal, in_range() of the quotient for the rest (a zero, infinite, tiny or
// huge dividend leaves a quotient out of its range); otherwise the division
// is done.
struct Diag {
  double d, y;
  bool usable;
  __device__ __forceinline__ explicit Diag(double v) : d(v), y(1.0 / v), usable(in_range(v, 100)) {
    asm volatile("" : "+v"(d), "+v"(y));
  }
  // 2^-e <= |v| < 2^e
  static __device__ __forceinline__ bool in_range(double v, int e) {
    const unsigned hi = (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu;
    return hi - ((unsigned)(1023 - e) << 20) < ((unsigned)(2 * e) << 20);
  }
  __device__ __forceinline__ double step(double a, double q) const {
    return __builtin_fma(__builtin_fma(-d, q, a), y, q);
  }
  __device__ __forceinline__ double divide(double a) const { return step(a, step(a, a * y)); }
};

// Eight columns of a wave's own diagonal, lanes lb .. lb + B - 1 their rows
// (B < 8 in the last block only): at step j lane lb + j divides, the quotient
// is broadcast, and every later row subtracts its product; TRANS takes the
// columns from the last one.  res keeps a lane's quotient.  Lanes already
// solved, and lanes past the last column, go on computing values that nothing
// reads.  A block whose quotients need the division (zeros of the right-hand
// side do) is done again step by step, with entries picked from m: loading them
// once more put a memory round trip on each step.
template <int KT, bool TRANS>
__device__ __forceinline__ void solve_block(double (&acc)[KT], double (&res)[KT],
                                            const double (&m)[8], const Diag &dg, int lb, int B,
                                            int lane) {
  double start[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) start[c] = acc[c];
#pragma unroll
  for (int t = 0; t < 8; ++t) {
    const int j = TRANS ? 7 - t : t;
    if (TRANS && j >= B) continue;
    double q[KT];
#pragma unroll
    for (int c = 0; c < KT; ++c) {
      q[c] = dg.divide(acc[c]);
      res[c] = lane == lb + j ? q[c] : res[c];
    }
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = acc[c] - lane_value(q[c], lb + j) * m[j];
  }
  bool ok = dg.usable;
#pragma unroll
  for (int c = 0; c < KT; ++c) ok = ok && Diag::in_range(res[c], 790);
  if (__any(lane >= lb && lane < lb + min(B, 8) && !ok)) {
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = start[c];
#pragma unroll 1
    for (int t = 0; t < min(B, 8); ++t) {
      const int j = TRANS ? min(B, 8) - 1 - t : t;
      double mj = 0.0;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        double e = m[u];
        asm volatile("" : "+v"(e));  // a value, not a place to be loaded from
        mj = j == u ? e : mj;
      }
#pragma unroll
      for (int c = 0; c < KT; ++c) {
        const double q = acc[c] / dg.d;
        res[c] = lane == lb + j ? q : res[c];
        acc[c] = acc[c] - lane_value(q, lb + j) * mj;
      }
    }
  }
}

// The last B < 8 columns of a row below: a block of four where four are left,
// then single columns.
template <int KT>
__device__ __forceinline__ void last_columns(double &t, const double *x, const double (&m)[8],
                                             int B) {
  if (B >= 4) {
    double sum = x[0] * m[0];
#pragma unroll
    for (int j = 1; j < 4; ++j) sum = sum + x[j * KT] * m[j];
    t = t + sum;
  }
#pragma unroll
  for (int j = 0; j < 7; ++j)
    if (j >= (B & 4) && j < B) t = t + x[j * KT] * m[j];
}

// A wave's own n <= 64 columns, in buf; done(lb, B) after each block.
template <int KT, typename Done>
__device__ __forceinline__ void own_columns(double (&acc)[KT], double (&res)[KT],
                                            const double (&buf)[SN_AHEAD][8], const Diag &dg,
                                            int n, int lane, Done done) {
#pragma unroll
  for (int b = 0; b < 8; ++b) {
    const int B = min(8, n - 8 * b);
    if (B > 0) {
      solve_block<KT, false>(acc, res, buf[b], dg, 8 * b, B, lane);
      done(8 * b, B);
    }
  }
}

// Rows 64g .. 64g+63 of a wide top, by one wave.  `buf` holds the first
// SN_AHEAD column blocks of the wave's rows.
template <int KT>
__device__ __forceinline__ void top_group(const SnArgs &a, const Cols<KT> &col, const double *T,
                                          double (&buf)[SN_AHEAD][8], const Diag &dg,
                                          const int4 &list, const int *gathered, int target,
                                          int g, int s, int w, int nr, const double *M, double *xs,
                                          int *prog, int &seen, int lane) {
  const int row = min(64 * g + lane, w - 1);
  double acc[KT], res[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) res[c] = 0.0;
  if (gathered) {
    wait_flag(gathered, target, a.state, a.timeout);
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = ld_dev(&col.x[c][s + row]);
  } else {
#pragma unroll
    for (int c = 0; c < KT; ++c) acc[c] = col.x[c][s + row];
    gather_list<KT, 16 / KT>(acc, T, a.tcount, list);
  }
  hold<KT>(acc);
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
  own_columns<KT>(acc, res, buf, dg, min(64, w - 64 * g), lane,
                  [&](int lb, int B) {
                    // every lane stores: solved rows their x again, the
                    // others what no wave reads before their own block's count
#pragma unroll
                    for (int c = 0; c < KT; ++c) xs[(64 * g + lane) * KT + c] = res[c];
                    lds_publish(prog, 64 * g + lb + B, lane);
                  });
#pragma unroll
  for (int c = 0; c < KT; ++c)
    if (64 * g + lane < w && col.live[c]) st_dev(&col.x[c][s + row], res[c]);
}

// A narrow supernode (w <= SN_NARROW) by one wave: the top, then the first
// SN_NARROW_ROWS rows below, a lane per row; xs is the wave's LDS.  The first
// blocks of the rows below are loaded before the wait too.
template <int KT>
__device__ __forceinline__ void narrow_unit(const SnArgs &a, const Cols<KT> &col, double *T,
                                            const SnUnit &n, int *flags, int slot, int target,
                                            double *xs, int lane) {
  constexpr int LA = 2;  // blocks of the rows below in flight
  const int s = n.s, w = n.w, nr = n.nr;
  const double *M = a.Lx + n.p;
  const int row = min(lane, w - 1);
  double buf[SN_AHEAD][8];
#pragma unroll
  for (int q = 0; q < SN_AHEAD; ++q) load_cols(buf[q], M, row, 8 * q, w, nr);
  const int4 list = a.list[s + row];
  // the rows below: item it is block it % nb of the lane's row of half it / nb
  const int below = min(nr - w, SN_NARROW_ROWS), nb = (w + 7) >> 3;
  const int items = ((below + 63) >> 6) * nb;
  double low[LA][8];
  auto load_item = [&](double (&m)[8], int it) {
    const int h = it >= nb ? 1 : 0;
    load_cols(m, M, w + max(min(64 * h + lane, below - 1), -1), 8 * (it - h * nb), w, nr);
  };
#pragma unroll
  for (int q = 0; q < LA; ++q) load_item(low[q], q);
  int place[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    place[h] = below > 0 ? a.tdst[n.tb + min(64 * h + lane, below - 1)] : 0;
  double acc[KT], res[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) {
    acc[c] = col.x[c][s + row];
    res[c] = 0.0;
  }
  const Diag dg(at(M + (int64_t)row * nr, row));
  wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
  gather_list<KT, 8 / KT>(acc, T, a.tcount, list);
  hold<KT>(acc);
  own_columns<KT>(acc, res, buf, dg, w, lane, [](int, int) {});
  if (lane < w) {
#pragma unroll
    for (int c = 0; c < KT; ++c) {
      xs[lane * KT + c] = res[c];
      if (col.live[c]) st_dev(&col.x[c][s + lane], res[c]);
    }
  }
  wave_lds_sync();
  double t[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) t[c] = 0.0;
  for (int i0 = 0; i0 < items; i0 += LA) {
#pragma unroll
    for (int q = 0; q < LA; ++q) {
      const int it = i0 + q;
      if (it < items) {
        const int h = it >= nb ? 1 : 0, cb = 8 * (it - h * nb);
        if (w - cb >= 8) {
#pragma unroll
          for (int c = 0; c < KT; ++c) {
            double sum = xs[cb * KT + c] * low[q][0];
#pragma unroll
            for (int j = 1; j < 8; ++j) sum = sum + xs[(cb + j) * KT + c] * low[q][j];
            t[c] = t[c] + sum;
          }
        } else {
#pragma unroll
          for (int c = 0; c < KT; ++c) last_columns<KT>(t[c], xs + cb * KT + c, low[q], w - cb);
        }
        if (cb + 8 >= w) {
#pragma unroll
          for (int c = 0; c < KT; ++c) {
            if (64 * h + lane < below) st_dev(&T[place[h] + c * a.tcount], t[c]);
            t[c] = 0.0;
          }
        }
      }
      load_item(low[q], min(it + LA, 2 * nb - 1));
    }
  }
  publish_fence();
  if (lane == 0) st_dev(&flags[slot], target);
  wave_lds_sync();
}

// 64 rows below a top by the workgroup: the column blocks of eight are dealt
// over the waves, NBW consecutive blocks each per pass; the block sums go to
// LDS and wave c adds column c's in block order.  The entries are loaded
// before the wait for the top.
template <int KT>
__device__ __forceinline__ void below_unit(const SnArgs &a, const Cols<KT> &col, double *T,
                                           const SnUnit &n, int *flags, int slot, int target,
                                           double *xs, double *sums) {
  constexpr int NBW = 8 / KT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = n.s, w = n.w, nr = n.nr, first = n.kind;
  const double *M = a.Lx + n.p;
  const int k = min(w + first + lane, nr - 1);
  const int nb = w / 8;  // full blocks; then one of 4 where 4 are left, then single columns
  double m[NBW][8], tail[8];
#pragma unroll
  for (int h = 0; h < NBW; ++h) load_cols(m[h], M, k, 8 * (wave * NBW + h), w, nr);
  load_cols(tail, M, k, 8 * nb, w, nr);
  const int64_t place = a.tdst[n.tb + k - w];
  if (wave == 0) wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
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
    const int cb = 8 * nb;
    last_columns<KT>(t, xs + cb * KT + wave, tail, w - cb);
    if (w + first + lane < nr) st_dev(&T[place + wave * a.tcount], t);
    publish_fence();
  }
  __syncthreads();
  if (threadIdx.x == 0) st_dev(&flags[slot], target);
}

// x of rows 64g .. 64g+63 of a wide top minus their temporaries, by the
// workgroup: rounds of 64 / KT list entries, a quarter of them loaded by each
// wave with the next round's in flight, turned over in LDS to wave c, which
// subtracts right-hand side c's in list order.  For tops of long lists: one
// wave per 64 rows took 19 us for the 512 rows of about 200 entries at the
// root of the 13-level factor, twice, before and during the solve.
template <int KT>
__device__ __forceinline__ void gather_unit(const SnArgs &a, const double *T, const SnUnit &n,
                                            int tile, int *flags, int slot, int target,
                                            double *stage) {
  constexpr int EW = 16 / KT, E = 4 * EW;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = 64 * (SN_GATHER_UNIT - n.kind) + lane;
  const int row = n.s + min(r, n.w - 1);
  const int4 l = a.list[row];
  const int cw = tile * KT + wave;
  double *const xc = a.x + (int64_t)min(cw, a.k - 1) * a.ldx;
  double v = xc[row];
  int longest = l.y;
  for (int off = 32; off > 0; off >>= 1) longest = max(longest, __shfl_xor(longest, off));
  longest = __builtin_amdgcn_readfirstlane(longest);
  if (wave == 0) wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
  __syncthreads();
  double ta[EW][KT], tb[EW][KT];
  auto load = [&](double (&t)[EW][KT], int j0) {
#pragma unroll
    for (int u = 0; u < EW; ++u) {
      const double *p = T + (l.x + (int64_t)max(min(j0 + wave * EW + u, l.y - 1), 0) * l.z);
#pragma unroll
      for (int q = 0; q < KT; ++q) t[u][q] = ld_dev(p + q * a.tcount);
    }
  };
  auto round = [&](double (&t)[EW][KT], int j0) {
    __syncthreads();  // the round before is read
#pragma unroll
    for (int u = 0; u < EW; ++u)
#pragma unroll
      for (int q = 0; q < KT; ++q) stage[((wave * EW + u) * KT + q) * 64 + lane] = t[u][q];
    load(t, j0 + 2 * E);
    __syncthreads();
    if (wave < KT) {
      const int cnt = min(E, longest - j0);
      for (int e = 0; e < cnt; e += 8) {
        double p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) p[u] = stage[(min(e + u, E - 1) * KT + wave) * 64 + lane];
#pragma unroll
        for (int u = 0; u < 8; ++u) v = j0 + e + u < min(l.y, j0 + E) ? v - p[u] : v;
      }
    }
  };
  load(ta, 0);
  load(tb, E);
  for (int j0 = 0; j0 < longest; j0 += 2 * E) {
    round(ta, j0);
    if (j0 + E < longest) round(tb, j0 + E);
  }
  if (wave < KT) {
    if (r < n.w && cw < a.k) st_dev(&xc[row], v);
    publish_fence();
  }
  __syncthreads();
  if (threadIdx.x == 0) st_dev(&flags[slot], target);
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
    int *const flags = a.flags + (int64_t)tile * a.ntick * 4;
    const SnUnit n = a.unit[4 * tk];
    if (n.kind >= 0) {
      below_unit<KT>(a, col, T, n, flags, 4 * tk, target, xs, sums);
    } else if (n.kind <= SN_GATHER_UNIT) {
      gather_unit<KT>(a, T, n, tile, flags, 4 * tk, target, sums);
    } else if (n.kind == SN_NARROW_UNIT) {
      const SnUnit m = a.unit[4 * tk + wave];
      if (m.w > 0)
        narrow_unit<KT>(a, col, T, m, flags, 4 * tk + wave, target, xs + wave * 64 * KT, lane);
    } else {
      const int w = n.w, nr = n.nr;
      const double *M = a.Lx + n.p;
      int seen = 0;
      for (int g = wave; g < 4 || 64 * g < w; g += 4) {
        const int row = min(64 * g + lane, w - 1);
        double buf[SN_AHEAD][8];
#pragma unroll
        for (int q = 0; q < SN_AHEAD; ++q) load_cols(buf[q], M, row, 8 * q, w, nr);
        const int4 list = a.list[n.s + row];
        const Diag dg(at(M + (int64_t)row * nr, row));
        if (g < 4) {  // each wave's first group: the entries are on their way
          if (wave == 0 && n.dn > 0)
            wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
          __syncthreads();
        }
        if (64 * g < w)
          top_group<KT>(a, col, T, buf, dg, list, n.dn < 0 ? &flags[n.d0 + 4 * g] : nullptr,
                        target, g, n.s, w, nr, M, xs, &slot[1], seen, lane);
      }
      publish_fence();
      __syncthreads();
      if (threadIdx.x == 0) st_dev(&flags[4 * tk], target);
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
// below are a ticket (the workgroup), and its top another: waves take groups
// of 64 columns from the last one, hand x on through LDS as in the forward
// solve, and wait for their own group's sums only.
//
// A lane owns a column, and a column's entries are contiguous: reading them
// lane by lane touches 64 cache lines per load.  So entries are loaded along
// the rows and turned in LDS.

constexpr int SN_ROWS_T = 16;            // rows of a turned block
constexpr int SN_PITCH_T = SN_ROWS_T + 1;

// Rows r0 .. r0+15 of columns c0 .. c0+63: four columns per load, lane l row
// l & 15 of column 4j + l / 16.  Clamped to the block's last row and the
// top's last column.
__device__ __forceinline__ void load_turn(double (&m)[16], const double *M, int r0, int c0,
                                          int w, int nr, int lane) {
  const double *R = M + min(r0 + (lane & 15), nr - 1);
#pragma unroll
  for (int j = 0; j < 16; ++j) m[j] = R[(int64_t)min(c0 + 4 * j + (lane >> 4), w - 1) * nr];
}

// The block turned: v[r] = row r of the lane's column.  tile: the wave's LDS,
// whose operations complete in the order a wave issues them.
__device__ __forceinline__ void turn_in(const double (&m)[16], double *tile, int lane) {
  asm volatile("" ::: "memory");
#pragma unroll
  for (int j = 0; j < 16; ++j) tile[(4 * j + (lane >> 4)) * SN_PITCH_T + (lane & 15)] = m[j];
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void turn_out(double (&v)[16], const double *tile, int lane) {
  asm volatile("" ::: "memory");
#pragma unroll
  for (int r = 0; r < 16; ++r) v[r] = tile[lane * SN_PITCH_T + r];
  asm volatile("" ::: "memory");
}
__device__ __forceinline__ void turn(double (&v)[16], const double (&m)[16], double *tile,
                                     int lane) {
  turn_in(m, tile, lane);
  turn_out(v, tile, lane);
}

// Eight rows c0 .. c0+7 of a wave's own columns (lanes lb .. lb+7).
template <int KT, typename Done>
__device__ __forceinline__ void own_rows(double (&acc)[KT], double (&res)[KT],
                                         const double (&m)[8], const Diag &dg, int c0, int lb,
                                         int w, int lane, Done done) {
  if (c0 < w) {
    solve_block<KT, true>(acc, res, m, dg, lb, w - c0, lane);
    done();
  }
}

// Columns 64g .. 64g+63 of a top, by one wave, from its last row: x from LDS
// for the columns of later groups (a narrow supernode, with one group, passes
// no xs).  m: the first two blocks of 16 rows, from the last.
template <int KT>
__device__ __forceinline__ void top_group_t(double (&acc)[KT], double (&res)[KT],
                                            double (&m)[2][16], const Diag &dg, int g, int w,
                                            int nr, const double *M, double *tile, double *xs,
                                            int *prog, int &seen, int lane) {
#pragma unroll
  for (int c = 0; c < KT; ++c) res[c] = 0.0;
  hold<KT>(acc);
  const int last = (w - 1) >> 4;
  auto eight = [&](const double (&v)[16], int b, int h) {
    const int c0 = 16 * b + 8 * h;
    double v8[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v8[j] = v[8 * h + j];
    if (b >= 4 * g + 4) {
      if (c0 < w) {
        lds_wait(prog, w - c0, seen);
        double xv[8][KT];
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
          for (int c = 0; c < KT; ++c) xv[j][c] = xs[min(c0 + j, w - 1) * KT + c];
#pragma unroll
        for (int j = 7; j >= 0; --j)
          if (c0 + j < w) {
#pragma unroll
            for (int c = 0; c < KT; ++c) acc[c] = acc[c] - v8[j] * xv[j][c];
          }
        hold<KT>(acc);
      }
    } else {
      const int lb = c0 - 64 * g;
      own_rows<KT>(acc, res, v8, dg, c0, lb, w, lane, [&] {
        if (xs) {
#pragma unroll
          for (int c = 0; c < KT; ++c) xs[(64 * g + lane) * KT + c] = res[c];
          lds_publish(prog, w - c0, lane);
        }
      });
    }
  };
  if constexpr (KT < 4) {
    // the next block is turned while this one is worked on (13-level factor:
    // 442 -> 433 us; with four columns the registers run out, 1.30 -> 1.42 ms)
    double va[16], vb[16];
    turn(va, m[0], tile, lane);
    load_turn(m[0], M, max(16 * (last - 2), 0), 64 * g, w, nr, lane);
    auto block = [&](const double (&v)[16], double (&vn)[16], double (&mn)[16], int b) {
      turn_in(mn, tile, lane);
      load_turn(mn, M, max(16 * (b - 3), 0), 64 * g, w, nr, lane);
      eight(v, b, 1);
      turn_out(vn, tile, lane);
      eight(v, b, 0);
    };
    for (int b = last; b >= 4 * g; b -= 2) {
      block(va, vb, m[1], b);
      if (b - 1 >= 4 * g) block(vb, va, m[0], b - 1);
    }
  } else {
    for (int b0 = last; b0 >= 4 * g; b0 -= 2) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const int b = b0 - q;
        if (b >= 4 * g) {
          double v[16];
          turn(v, m[q], tile, lane);
          load_turn(m[q], M, max(16 * (b - 2), 0), 64 * g, w, nr, lane);
          eight(v, b, 1);
          eight(v, b, 0);
        }
      }
    }
  }
}

template <int KT>
__device__ __forceinline__ void narrow_unit_t(const SnArgs &a, const Cols<KT> &col,
                                              const SnUnit &n, int *flags, int slot, int target,
                                              double *tile, int lane) {
  const int s = n.s, w = n.w, nr = n.nr, below = nr - w;
  const double *M = a.Lx + n.p;
  const int *rows = a.rowb + n.tb;
  const int c = min(lane, w - 1);
  // blocks of 16 rows below, ascending, then the top's from its last
  const int nb = (below + 15) >> 4, last = (w - 1) >> 4;
  auto first_row = [&](int it) { return it < nb ? w + 16 * it : max(16 * (last - (it - nb)), 0); };
  double m[2][16];
  load_turn(m[0], M, first_row(0), 0, w, nr, lane);
  load_turn(m[1], M, first_row(1), 0, w, nr, lane);
  double acc[KT], res[KT];
#pragma unroll
  for (int q = 0; q < KT; ++q) acc[q] = col.x[q][s + c];
  const Diag dg(M[c + (int64_t)c * nr]);
  if (below > 0) {
    const int r0 = rows[min(lane, below - 1)], r1 = rows[min(64 + lane, below - 1)];
    wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
    double x0[KT], x1[KT], t[KT];
#pragma unroll
    for (int q = 0; q < KT; ++q) {
      x0[q] = ld_dev(&col.x[q][r0]);
      x1[q] = ld_dev(&col.x[q][r1]);
      t[q] = 0.0;
    }
    hold<KT>(x0);
    hold<KT>(x1);
    for (int i0 = 0; i0 < nb; i0 += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int it = i0 + u;
        if (it < nb) {
          double v[16];
          turn(v, m[u], tile, lane);
          load_turn(m[u], M, first_row(it + 2), 0, w, nr, lane);
          if (it == 4) {
#pragma unroll
            for (int q = 0; q < KT; ++q) x0[q] = x1[q];
          }
          const int cnt = below - 16 * it;
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (j < cnt) {
#pragma unroll
              for (int q = 0; q < KT; ++q) {
                const double p = v[j] * lane_value(x0[q], (16 * it + j) & 63);
                t[q] = 16 * it + j == 0 ? p : t[q] + p;
              }
            }
        }
      }
    }
#pragma unroll
    for (int q = 0; q < KT; ++q) acc[q] = acc[q] - t[q];
    if (nb & 1) {  // the top's first block is in m[1]
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const double d = m[0][j];
        m[0][j] = m[1][j];
        m[1][j] = d;
      }
    }
  }
  int seen = 0;
  top_group_t<KT>(acc, res, m, dg, 0, w, nr, M, tile, nullptr, nullptr, seen, lane);
#pragma unroll
  for (int q = 0; q < KT; ++q)
    if (lane < w && col.live[q]) st_dev(&col.x[q][s + lane], res[q]);
  publish_fence();
  if (lane == 0) st_dev(&flags[slot], target);
}

constexpr int SN_PITCH = 65;   // doubles per column of a turned 64 x 64 tile
constexpr int SN_TILES = 4;    // tiles of 64 rows below in flight

// The sums over the rows below of columns 64g .. 64g+63, by the workgroup.
// Tiles of 64 rows; wave v loads 16 columns of a tile along its rows, four
// tiles in flight, x at the rows of 256 at a time in LDS; wave c then adds
// right-hand side c's products, a lane per column.
template <int KT>
__device__ __forceinline__ void below_unit_t(const SnArgs &a, const Cols<KT> &col,
                                             const SnUnit &n, int tile, int *flags, int slot,
                                             int target, double *turned, double *xrow) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int s = n.s, w = n.w, nr = n.nr, below = nr - w, g = n.kind;
  const double *M = a.Lx + n.p + w;
  const int *rows = a.rowb + n.tb;
  double m[SN_TILES][16];
  auto load = [&](double (&d)[16], int r0) {
    const int r = min(r0 + lane, below - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      d[j] = at(M + (int64_t)min(64 * g + 16 * wave + j, w - 1) * nr, r);
  };
#pragma unroll
  for (int q = 0; q < SN_TILES; ++q) load(m[q], 64 * q);
  int row = rows[min((int)threadIdx.x, below - 1)];
  if (wave == 0) wait_list(a.dlist + n.d0, n.dn, flags, target, a.state, a.timeout);
  __syncthreads();
  double xn[KT];
#pragma unroll
  for (int c = 0; c < KT; ++c) xn[c] = ld_dev(&col.x[c][row]);
  row = rows[min(256 + (int)threadIdx.x, below - 1)];
  double t = 0.0;
  int half = 0;
  for (int r0 = 0; r0 < below; r0 += 64 * SN_TILES) {
    __syncthreads();  // the x of the rows before are read
#pragma unroll
    for (int c = 0; c < KT; ++c) xrow[c * 256 + threadIdx.x] = xn[c];
    if (r0 + 256 < below) {
#pragma unroll
      for (int c = 0; c < KT; ++c) xn[c] = ld_dev(&col.x[c][row]);
      row = rows[min(r0 + 512 + (int)threadIdx.x, below - 1)];
    }
#pragma unroll
    for (int q = 0; q < SN_TILES; ++q) {
      const int r = r0 + 64 * q;
      if (r < below) {
        double *const tl = turned + half * 64 * SN_PITCH;
#pragma unroll
        for (int j = 0; j < 16; ++j) tl[(16 * wave + j) * SN_PITCH + lane] = m[q][j];
        load(m[q], r + 64 * SN_TILES);
        __syncthreads();
        if (wave < KT) {
          const double *const xl = xrow + wave * 256 + 64 * q, *const ml = tl + lane * SN_PITCH;
          const int cnt = min(64, below - r);
          int i = 0;
          if (r == 0) {
            t = ml[0] * xl[0];
            i = 1;
          }
          for (; i + 8 <= cnt; i += 8) {
            double p[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) p[j] = ml[i + j] * xl[i + j];
#pragma unroll
            for (int j = 0; j < 8; ++j) t = t + p[j];
          }
          for (; i < cnt; ++i) t = t + ml[i] * xl[i];
        }
        half ^= 1;
      }
    }
  }
  if (wave < KT) {
    const int c = 64 * g + lane, cw = tile * KT + wave;
    double *const xc = a.x + (int64_t)min(cw, a.k - 1) * a.ldx;
    if (c < w && cw < a.k) st_dev(&xc[s + c], xc[s + c] - t);
    publish_fence();
  }
  __syncthreads();
  if (threadIdx.x == 0) st_dev(&flags[slot], target);
}

template <int KT>
__global__ __launch_bounds__(256, 2) void k_supernodal_t(SnArgs a) {
  // a top's x and the waves' turned blocks, or two turned tiles and the x at
  // their rows
  constexpr int TOP = SN_WMAX * KT + 4 * 64 * SN_PITCH_T;
  constexpr int TILES = 2 * 64 * SN_PITCH + 256 * KT;
  __shared__ double mem[TOP > TILES ? TOP : TILES];
  __shared__ int slot[2];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int target = ld_dev(&a.state[ST_EPOCH]) + 1;
  double *const mine = mem + SN_WMAX * KT + wave * 64 * SN_PITCH_T;
  for (;;) {
    const int tt = next_ticket(a, slot);
    if (tt < 0) break;
    const int tk = tt / a.tiles, tile = tt - tk * a.tiles;
    const Cols<KT> col(a, tile);
    int *const flags = a.flags + (int64_t)tile * a.ntick * 4;
    const SnUnit n = a.unit[4 * tk];
    if (n.kind >= 0) {
      below_unit_t<KT>(a, col, n, tile, flags, 4 * tk, target, mem, mem + 2 * 64 * SN_PITCH);
    } else if (n.kind == SN_NARROW_UNIT) {
      const SnUnit u = a.unit[4 * tk + wave];
      if (u.w > 0) narrow_unit_t<KT>(a, col, u, flags, 4 * tk + wave, target, mine, lane);
    } else {
      const int w = n.w, nr = n.nr;
      const double *M = a.Lx + n.p;
      int seen = 0;
      for (int g = (w + 63) / 64 - 1 - wave; g >= 0; g -= 4) {
        const int last = (w - 1) >> 4, c = min(64 * g + lane, w - 1);
        double m[2][16];
        load_turn(m[0], M, 16 * last, 64 * g, w, nr, lane);
        load_turn(m[1], M, max(16 * (last - 1), 0), 64 * g, w, nr, lane);
        const Diag dg(M[c + (int64_t)c * nr]);
        if (n.dn < 0) wait_flag(&flags[n.d0 + 4 * g], target, a.state, a.timeout);
        double acc[KT], res[KT];
#pragma unroll
        for (int q = 0; q < KT; ++q) acc[q] = ld_dev(&col.x[q][n.s + c]);
        top_group_t<KT>(acc, res, m, dg, g, w, nr, M, mine, mem, &slot[1], seen, lane);
#pragma unroll
        for (int q = 0; q < KT; ++q)
          if (64 * g + lane < w && col.live[q]) st_dev(&col.x[q][n.s + c], res[q]);
      }
      publish_fence();
      __syncthreads();
      if (threadIdx.x == 0) st_dev(&flags[4 * tk], target);
    }
  }
  persistent_finish(a.state, a.total_waves);
}

}  // namespace

namespace {

// Tickets of one direction, level by level, in slots of four units.  Per
// level: the groups of 64 rows or columns that are gathered or summed ahead of
// a wide top (forward: where a row's list is longer than SN_GATHER_LONG;
// transposed: where there are rows below), the wide tops, the narrow
// supernodes four to a ticket, and the further rows below (forward only, 64
// per unit).
struct SnSchedule {
  std::vector<SnUnit> unit;           // four slots per ticket
  std::vector<int> top;               // per supernode: the slot that solves its top
  std::vector<int> group;             // per supernode: the slot of its first group, or -1
  std::vector<int> first;             // per supernode: the slot of its first chunk, or -1
  std::map<int, int> widths;          // tickets of a level -> levels
  std::vector<int> dlist;
};

void sn_schedule(int m, const int *h_sup, const int *h_nrows, const int *h_Lp,
                 const std::vector<int> &lev, const std::vector<int> &tb,
                 const std::vector<int> &longest, bool transposed, SnSchedule &s) {
  std::vector<int> order(m);
  for (int i = 0; i < m; ++i) order[i] = transposed ? m - 1 - i : i;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return lev[x] < lev[y]; });
  s.top.assign(m, -1);
  s.group.assign(m, -1);
  s.first.assign(m, -1);
  auto width = [&](int i) { return h_sup[i + 1] - h_sup[i]; };
  auto below = [&](int i) { return tb[i + 1] - tb[i]; };
  auto narrow = [&](int i) {
    return width(i) <= SN_NARROW && (!transposed || below(i) <= SN_NARROW_ROWS);
  };
  auto put = [&](int i, int kind) {
    s.unit.push_back({h_sup[i], width(i), h_nrows[i], kind, h_Lp[i], tb[i], 0, 0});
    return (int)s.unit.size() - 1;
  };
  auto close = [&] {
    while (s.unit.size() % 4) s.unit.push_back({0, 0, 0, SN_NARROW_UNIT, 0, 0, 0, 0});
  };
  for (int a = 0, b = 0; a < m; a = b) {
    const size_t before = s.unit.size();
    while (b < m && lev[order[b]] == lev[order[a]]) ++b;
    for (int j = a; j < b; ++j)
      if (!narrow(order[j]) &&
          (transposed ? below(order[j]) > 0 : longest[order[j]] > SN_GATHER_LONG))
        for (int g = 0; 64 * g < width(order[j]); ++g) {
          const int u = put(order[j], transposed ? g : SN_GATHER_UNIT - g);
          if (g == 0) s.group[order[j]] = u;
          close();
        }
    for (int j = a; j < b; ++j)
      if (!narrow(order[j])) {
        s.top[order[j]] = put(order[j], SN_TOP);
        close();
      }
    for (int j = a; j < b; ++j)
      if (narrow(order[j])) s.top[order[j]] = put(order[j], SN_NARROW_UNIT);
    close();
    if (!transposed)
      for (int j = a; j < b; ++j) {
        const int i = order[j];
        for (int r = narrow(i) ? SN_NARROW_ROWS : 0; r < below(i); r += 64) {
          const int u = put(i, r);
          if (s.first[i] < 0) s.first[i] = u;
          close();
        }
      }
    ++s.widths[(int)((s.unit.size() - before) / 4)];
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
  // uneven lists (padding past three entries in four), and all rows where that
  // padding could pass 32-bit places, keep theirs contiguous
  std::vector<int> tdst(tb[m] > 0 ? tb[m] : 1), rowb(tb[m] > 0 ? tb[m] : 1);
  std::vector<int4> list(n > 0 ? n : 1, make_int4(0, 0, 0, 0));
  const bool pad = 4 * (int64_t)cnt[n] <= INT_MAX;
  int64_t tcount = 0;
  for (int i = 0; i < m; ++i)
    for (int r0 = h_sup[i]; r0 < h_sup[i + 1]; r0 += 64) {
      const int r1 = std::min(r0 + 64, h_sup[i + 1]);
      const int64_t total = cnt[r1] - cnt[r0];
      int64_t longest = 0;
      for (int r = r0; r < r1; ++r) longest = std::max<int64_t>(longest, cnt[r + 1] - cnt[r]);
      const bool side = pad && longest * (r1 - r0) <= 4 * total;
      for (int r = r0; r < r1; ++r)
        if (cnt[r + 1] > cnt[r])
          list[r] = make_int4((int)(tcount + (side ? r - r0 : cnt[r] - cnt[r0])), 0,
                              side ? r1 - r0 : 1, 0);
      tcount += side ? longest * (r1 - r0) : total;
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
  std::vector<int> own, optr(m + 1, 0);  // owners of a supernode's rows below, in row order
  int old_tasks = 0;
  for (int i = 0; i < m; ++i) {
    const int w = h_sup[i + 1] - h_sup[i];
    int last = -1;
    for (int k = 0; k < h_nrows[i] - w; ++k) {
      const int row = h_Li[h_Lp[i] + w + k], o = owner[row];
      int4 &l = list[row];
      rowb[tb[i] + k] = row;
      tdst[tb[i] + k] = l.x + l.y++ * l.z;
      if (o != last) {
        own.push_back(o);
        lev[o] = std::max(lev[o], lev[i] + 1);
        last = o;
      }
    }
    optr[i + 1] = (int)own.size();
    old_tasks += std::max(1, (h_nrows[i] - w + 127) / 128);
  }
  for (int i = m - 1; i >= 0; --i)
    for (int k = optr[i]; k < optr[i + 1]; ++k) tlev[i] = std::max(tlev[i], tlev[own[k]] + 1);
  std::vector<int> longest(m, 0);  // longest list of a supernode's rows
  for (int i = 0; i < m; ++i)
    for (int r = h_sup[i]; r < h_sup[i + 1]; ++r) longest[i] = std::max(longest[i], cnt[r + 1] - cnt[r]);
  SnSchedule fwd, bwd;
  sn_schedule(m, h_sup, h_nrows, h_Lp, lev, tb, longest, false, fwd);
  sn_schedule(m, h_sup, h_nrows, h_Lp, tlev, tb, longest, true, bwd);
  // forward: a top, or the row groups of one that has them, waits for the
  // units that write its rows' temporaries, a chunk of the rows below for its
  // top.  transposed: the units that read x at the rows below (a narrow
  // supernode, the column groups of a wide one, which share a list) wait for the
  // tops of their owners.  A top with groups waits for those.  A unit's rows
  // meet another's in ascending order, so a pair met again follows itself.
  std::vector<std::pair<int, int>> pairs;  // (waiting slot, slot waited for)
  std::vector<int> last(fwd.unit.size(), -1);
  for (int i = 0; i < m; ++i) {
    const int w = h_sup[i + 1] - h_sup[i], below = tb[i + 1] - tb[i];
    const int head = w <= SN_NARROW ? SN_NARROW_ROWS : 0, d0 = (int)bwd.dlist.size();
    for (int k = 0; k < below; ++k) {
      const int row = rowb[tb[i] + k], o = owner[row];
      const int producer = k < head ? fwd.top[i] : fwd.first[i] + 4 * ((k - head) / 64);
      const int u = fwd.group[o] < 0 ? fwd.top[o] : fwd.group[o] + 4 * ((row - h_sup[o]) / 64);
      if (last[u] != producer) pairs.emplace_back(u, producer);
      last[u] = producer;
    }
    for (int r = head, u = fwd.first[i]; u >= 0 && r < below; r += 64, u += 4)
      pairs.emplace_back(u, fwd.top[i]);
    for (int k = optr[i]; k < optr[i + 1]; ++k) bwd.dlist.push_back(bwd.top[own[k]]);
    std::sort(bwd.dlist.begin() + d0, bwd.dlist.end());
    bwd.dlist.erase(std::unique(bwd.dlist.begin() + d0, bwd.dlist.end()), bwd.dlist.end());
    const int dn = (int)bwd.dlist.size() - d0;
    for (int g = 0; dn > 0 && (bwd.group[i] < 0 ? g == 0 : 64 * g < w); ++g) {
      SnUnit &u = bwd.unit[bwd.group[i] < 0 ? bwd.top[i] : bwd.group[i] + 4 * g];
      u.d0 = d0;
      u.dn = dn;
    }
  }
  std::vector<int> dptr(fwd.unit.size() + 1, 0);
  for (const auto &d : pairs) ++dptr[d.first + 1];
  for (size_t u = 0; u + 1 < dptr.size(); ++u) dptr[u + 1] += dptr[u];
  fwd.dlist.resize(pairs.size());
  std::vector<int> at(dptr.begin(), dptr.end() - 1);
  for (const auto &d : pairs) fwd.dlist[at[d.first]++] = d.second;
  for (size_t u = 0; u < fwd.unit.size(); ++u)
    if (dptr[u + 1] > dptr[u]) {
      std::sort(fwd.dlist.begin() + dptr[u], fwd.dlist.begin() + dptr[u + 1]);
      fwd.unit[u].d0 = dptr[u];
      fwd.unit[u].dn = dptr[u + 1] - dptr[u];
    }
  for (SnSchedule *s : {&fwd, &bwd})
    for (int i = 0; i < m; ++i)
      if (s->group[i] >= 0) {
        s->unit[s->top[i]].d0 = s->group[i];
        s->unit[s->top[i]].dn = -1;
      }
  auto *q = new symamd_snplan_s();
  q->n = n;
  q->m = m;
  q->tcount = tcount;
  q->ntasks = old_tasks;
  q->tickets = (int)(fwd.unit.size() / 4);
  q->ttickets = (int)(bwd.unit.size() / 4);
  q->widths[0].assign(fwd.widths.begin(), fwd.widths.end());
  q->widths[1].assign(bwd.widths.begin(), bwd.widths.end());
  const int64_t flags = 4 * (int64_t)std::max(1, std::max(q->tickets, q->ttickets));
  int rc = SYMAMD_OK;
  auto up = [&](int **dst, const int *src, size_t count) {
    if (rc != SYMAMD_OK) return;
    if (hipMalloc(dst, sizeof(int) * (count ? count : 1)) != hipSuccess ||
        (count && hipMemcpy(*dst, src, sizeof(int) * count, hipMemcpyHostToDevice) != hipSuccess))
      rc = fail(SYMAMD_ERR_ALLOC, "supernodal plan upload failed");
  };
  up(&q->d_tdst, tdst.data(), tb[m]);
  up(&q->d_rowb, rowb.data(), tb[m]);
  up(&q->d_list, reinterpret_cast<const int *>(list.data()), 4 * (size_t)n);
  up(&q->d_unit, reinterpret_cast<const int *>(fwd.unit.data()), 8 * fwd.unit.size());
  up(&q->d_dlist, fwd.dlist.data(), fwd.dlist.size());
  up(&q->d_tunit, reinterpret_cast<const int *>(bwd.unit.data()), 8 * bwd.unit.size());
  up(&q->d_tdlist, bwd.dlist.data(), bwd.dlist.size());
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

// Columns per tile: a row's entries are loaded once for the columns of a tile,
// but each step of a top's chain then divides for all of them.  On the 13-level
// factor, forward + transposed with tiles of 1 / 2 / 4: k = 2 0.86 / 0.93 / - ms,
// k = 4 1.11 / 1.02 / 1.32 ms, k = 13 2.30 / 1.76 / 1.83 ms, k = 32 4.94 / 3.17 /
// 2.61 ms.  Where the levels hold few tickets the chain is all there is, and
// narrower tiles run side by side: a level takes 1 / 1.27 / 1.9 times as long
// with tiles of 1 / 2 / 4 columns (about 5 us with one), once per SN_BUSY
// tickets, and each ticket 12.5 ns of the counter.  Forward, k = 32, in ms with
// tiles of 1 / 2 / 4: 600 supernodes of 64 columns in 364 levels 3.23 / 4.01 /
// 5.98, 20,000 of 4 columns in 635 levels 3.27 / 3.08 / 4.01, of 1 column in 157
// 2.78 / 1.68 / 1.25, the 13-level factor 2.47 / 1.60 / 1.37.
static int sn_widest_tile(int k) { return k < 4 ? 1 : k < 16 ? 2 : 4; }
static int sn_tile(const std::vector<std::pair<int, int>> &widths, int64_t tickets, int k) {
  constexpr double SN_BUSY = 128.0, CHAIN[3] = {1.0, 1.27, 1.9};
  const int widest = sn_widest_tile(k);
  int best = widest;
  double least = 0.0;
  for (int kt = widest, i = widest / 2; kt >= 1; kt /= 2, i = kt / 2) {
    const double tiles = (k + kt - 1) / kt;
    if (kt < widest && tickets * tiles >= INT_MAX) break;
    double us = 0.0;
    for (const auto &w : widths)
      us += w.second * (5.0 * CHAIN[i] * std::max(1.0, w.first * tiles / SN_BUSY) +
                        0.0125 * w.first * tiles);
    if (kt == widest || us < 0.92 * least) {
      least = us;
      best = kt;
    }
  }
  return best;
}

int sn_solve(symamd_handle h, symamd_snplan_s *q, const double *d_Lx, double *d_x, int k,
             int64_t ldx, bool transposed) {
  if (q->m == 0 || k == 0) return SYMAMD_OK;
  // tickets run over (task, column) pairs in 32-bit counters
  if ((int64_t)q->ntasks * k >= (int64_t)INT_MAX)
    return fail(SYMAMD_ERR_NOT_SUPPORTED,
                "supernodal solve: %d tasks x %d columns exceed the 32-bit ticket range; "
                "solve the columns in smaller batches", q->ntasks, k);
  const int kt = sn_tile(q->widths[transposed], transposed ? q->ttickets : q->tickets, k);
  const int tiles = (k + kt - 1) / kt;
  // temporaries and tags for the columns of whole tiles; those that a caller's
  // graph reads stay until the plan is destroyed
  const bool cap = capturing(h->stream);
  const int widest = sn_widest_tile(k);
  const int64_t cols = ((int64_t)k + widest - 1) / widest * widest;
  if (cols > q->kcap) {
    if (cap)
      return fail(SYMAMD_ERR_NOT_SUPPORTED,
                  "supernodal temporaries for %d columns not prepared before capture", k);
    double *T = nullptr;
    int *flags = nullptr;
    const int64_t tc = q->tcount > 0 ? q->tcount : 1;
    const int64_t nt = 4 * (int64_t)std::max(1, std::max(q->tickets, q->ttickets));
    if (hipMalloc(&T, sizeof(double) * tc * cols) != hipSuccess ||
        hipMalloc(&flags, sizeof(int) * nt * cols) != hipSuccess) {
      (void)hipGetLastError();
      if (T) (void)hipFree(T);
      return fail(SYMAMD_ERR_ALLOC, "supernodal temporaries for %d columns", k);
    }
    // cleared tags read as "not ready" in every epoch
    SYMAMD_HIP(hipMemsetAsync(flags, 0, sizeof(int) * nt * cols, h->stream));
    SYMAMD_HIP(hipStreamSynchronize(h->stream));
    for (void *old : {(void *)q->d_T, (void *)q->d_flags}) {
      if (q->captured)
        q->retired.push_back(old);
      else
        (void)hipFree(old);
    }
    q->captured = false;
    q->d_T = T;
    q->d_flags = flags;
    q->kcap = (int)cols;
  }
  if (cap) q->captured = true;
  SnArgs a;
  a.unit = reinterpret_cast<const SnUnit *>(transposed ? q->d_tunit : q->d_unit);
  a.Lx = d_Lx;
  a.x = d_x;
  a.T = q->d_T;
  a.tdst = q->d_tdst;
  a.list = reinterpret_cast<const int4 *>(q->d_list);
  a.dlist = transposed ? q->d_tdlist : q->d_dlist;
  a.ntick = transposed ? q->ttickets : q->tickets;
  a.rowb = q->d_rowb;
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
  void *ptrs[] = {q->d_tdst,  q->d_rowb,   q->d_list, q->d_unit, q->d_dlist,
                  q->d_tunit, q->d_tdlist, q->d_T,    q->d_flags, q->d_state};
  for (void *x : ptrs)
    if (x) (void)hipFree(x);
  for (void *x : q->retired) (void)hipFree(x);
  delete q;
}

}  // namespace symamd
