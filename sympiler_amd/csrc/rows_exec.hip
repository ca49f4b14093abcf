// rows_exec.hip -- forward solve of matrices with long, uneven rows for
// gfx950: one persistent launch, rows shared by as many lanes as they have
// entries, values passed from row to row by themselves.
//
// It runs sync-free solves with several lanes per row (the unit executor of
// executors.hip cuts levels into units and waits for whole units; with rows
// of 1 to 256 entries a unit waits for hundreds of others, about 7 us per
// level).  Here every row is its own item:
//   - before the solve the right-hand sides are copied aside and X is filled
//     with the mark (a signalling NaN that no arithmetic produces), so a value
//     read from X is either the mark or the solution: readers poll the values
//     they need, and no tag or store acknowledgement lies on the chain;
//   - a row's entries lie one or a few per lane, all their loads in flight at
//     once; only the values not there yet are read again;
//   - rows are scheduled level by level, in each level by the lanes they
//     take, so that one wavefront solves 1 to 64 rows of similar length; with
//     several right-hand sides a row too long for one wavefront is a
//     workgroup's (its waves' sums meet in LDS).
// What bounds it is the chain of levels for one right-hand side (a store on
// one XCD reaching a poll on another, the lanes' reduction, the division:
// 1.4 us per level) and, for several and where levels are wide, the tickets
// (one counter, 13 ns each; few wide levels stay on the units, see
// tickets_win).  Zipf(1.8) matrix, n = 1e6, 459 levels, in ms with the unit
// executor and here: one right-hand side 3.38 / 0.65, 4 columns 5.1 / 0.79, 13
// columns 10 / 1.06, 32 columns 18.0 / 1.38 (0.22 of it the turns of a
// column-major block).
// Workgroups take tickets in schedule order, so every value waited for is
// held by a running workgroup; waits are bounded by the watchdog.
//
// Arithmetic: x = (b - sum) / L[i,i], the sum over a lane's entries pairwise,
// then across lanes and waves in a fixed order; results do not depend on
// timing.  (Subtracting the products of short rows from b one by one, in the
// reference's order, leaves an error against 64 bits 1.6 times the unit
// executor's, whose lanes sum first too.)
#include <algorithm>
#include <new>
#include <vector>

#include "device.h"

namespace symamd {

namespace {

// Entries per lane in flight: one right-hand side, several, and the rows a
// workgroup shares.  Lanes per row are chosen so that a row takes one round
// where its wavefront is wide enough.
constexpr int rows_epl(int c) { return c == 1 ? 4 : 8; }
constexpr int ROWS_EPL_GROUP = 16;
// Waves per workgroup.
constexpr int rows_waves(int c) { return c == 1 ? 2 : 8; }
// 32 column lanes: rows of at most ROWS_SHORT entries (two in three of the Zipf
// matrix) are solved ROWS_PER_LANE to a lane, all their loads in flight, which
// takes a quarter of their tickets (1.60 -> 1.35 ms; with 8 and 16 column
// lanes, whose wavefronts hold more rows, it measured slower).
constexpr int ROWS_SHORT = 2, ROWS_PER_LANE = 4;
constexpr bool rows_short(int c) { return c == 32; }
// Item kinds: log2 of the slices per row, or
constexpr int ROWS_KIND_SHORT = 16, ROWS_KIND_GROUP = 17;

template <typename T>
struct RowArgs {
  const int4 *rec;    // per scheduled row: first entry, diagonal entry, row
  const int4 *item;   // per wave of a ticket: first record, rows, kind; a workgroup's row:
                      // its record, kind
  const int *ci;
  const T *val;
  const T *b;         // right-hand sides, row-major, k per row
  T *x;               // marks, then the solution: row i, column c at i*rs + c*cs
  int64_t rs, cs;
  int k, tiles, ntick, total_waves;
  int *state;
  uint64_t timeout;
};

// Values of up to N entries of one lane: loads them all, then again those
// that still read as the mark.
template <typename T, int N>
__device__ __forceinline__ void wait_values(T (&x)[N], const T *const (&p)[N],
                                            const bool (&use)[N], int *state, uint64_t timeout) {
#pragma unroll
  for (int j = 0; j < N; ++j) x[j] = ld_dev(p[j]);
  bool pend = false;
#pragma unroll
  for (int j = 0; j < N; ++j) pend = pend || (use[j] && is_mark(x[j]));
  if (!__any(pend)) return;
  const uint64_t t0 = wall_ticks();
  for (int rounds = 1; __any(pend); ++rounds) {
    __builtin_amdgcn_s_sleep(1);
    if (pend) {
#pragma unroll
      for (int j = 0; j < N; ++j)
        if (use[j] && is_mark(x[j])) x[j] = ld_dev(p[j]);
      pend = false;
#pragma unroll
      for (int j = 0; j < N; ++j) pend = pend || (use[j] && is_mark(x[j]));
    }
    if ((rounds & 63) == 0 && wall_ticks() - t0 > timeout) {
      if (pend) atomicOr(&state[ST_ERROR], 1);
      break;
    }
  }
}

// Sum over entries e0 + first, + step, ... below e1 of value times x: rounds
// of N entries, added pairwise, the rounds in order.
template <typename T, int N>
__device__ __forceinline__ T row_sum(const RowArgs<T> &a, int e0, int e1, int first, int step,
                                     int64_t co, bool act) {
  T acc = T(0);
  for (int base = first; __any(act && e0 + base < e1); base += N * step) {
    T v[N], x[N];
    const T *p[N];
    bool use[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const int e = e0 + base + j * step;
      use[j] = act && e < e1;
      const int q = min(e, e1);
      v[j] = a.val[q];
      p[j] = a.x + ((int64_t)a.ci[q] * a.rs + co);
    }
    wait_values<T, N>(x, p, use, a.state, a.timeout);
#pragma unroll
    for (int j = 0; j < N; ++j) v[j] = use[j] ? v[j] * x[j] : T(0);
#pragma unroll
    for (int h = N / 2; h >= 1; h >>= 1)
#pragma unroll
      for (int j = 0; j < h; ++j) v[j] = v[j] + v[j + h];
    acc = acc + v[0];
  }
  return acc;
}

template <typename T, int C>
__global__ __launch_bounds__(64 * rows_waves(C), 4) void k_rows(RowArgs<T> a) {
  constexpr int W = rows_waves(C), SMAX = 64 / C;
  __shared__ int slot;
  __shared__ T part[W][C];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane % C, sub = lane / C;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) slot = atomicAdd(&a.state[ST_TICKET], 1);
    __syncthreads();
    const int tt = __builtin_amdgcn_readfirstlane(slot);
    if (tt >= a.ntick * a.tiles) break;
    const int tk = tt / a.tiles, tile = tt - tk * a.tiles;
    const int col = tile * C + c;
    const bool live = col < a.k;
    const int cc = min(col, a.k - 1);
    const int64_t co = cc * a.cs;
    const int4 it = a.item[tk * W + wave];
    if (it.w == ROWS_KIND_GROUP) {
      // one row for the workgroup: wave and slice take every (W * SMAX)-th
      // entry, slices are added by lane, waves in order
      const int4 r = it;
      const T b = a.b[(int64_t)r.z * a.k + cc], d = a.val[r.y];
      T s = row_sum<T, ROWS_EPL_GROUP>(a, r.x, r.y, wave * SMAX + sub, W * SMAX, co, true);
#pragma unroll
      for (int off = C; off < 64; off <<= 1) s += __shfl_xor(s, off);
      if (sub == 0) part[wave][c] = s;
      __syncthreads();
      if (wave == 0 && sub == 0) {
        T sum = part[0][c];
#pragma unroll
        for (int w = 1; w < W; ++w) sum += part[w][c];
        if (live) st_dev(&a.x[r.z * a.rs + co], (b - sum) / d);
      }
      continue;
    }
    const int cnt = it.y;
    if (cnt == 0) continue;
    if (rows_short(C) && it.w == ROWS_KIND_SHORT) {
      constexpr int M = ROWS_PER_LANE, N = ROWS_SHORT;
      T v[M * N], x[M * N], b[M], d[M];
      const T *p[M * N];
      bool use[M * N];
      int row[M];
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const int i = sub + SMAX * m;
        const int4 r = a.rec[it.x + min(i, cnt - 1)];
        row[m] = i < cnt ? r.z : -1;
        b[m] = a.b[(int64_t)r.z * a.k + cc];
        d[m] = a.val[r.y];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const int q = min(r.x + j, r.y);
          use[m * N + j] = i < cnt && r.x + j < r.y;
          v[m * N + j] = a.val[q];
          p[m * N + j] = a.x + ((int64_t)a.ci[q] * a.rs + co);
        }
      }
      wait_values<T, M * N>(x, p, use, a.state, a.timeout);
#pragma unroll
      for (int m = 0; m < M; ++m) {
        T s = T(0);
#pragma unroll
        for (int j = 0; j < N; ++j)
          if (use[m * N + j]) s = s + v[m * N + j] * x[m * N + j];
        if (row[m] >= 0 && live) st_dev(&a.x[row[m] * a.rs + co], (b[m] - s) / d[m]);
      }
      continue;
    }
    const int lg = it.w, slice = sub & ((1 << lg) - 1), i = sub >> lg;
    const bool act = i < cnt;
    const int4 r = a.rec[it.x + min(i, cnt - 1)];
    const T b = a.b[(int64_t)r.z * a.k + cc], d = a.val[r.y];
    T s = row_sum<T, rows_epl(C)>(a, r.x, r.y, slice, 1 << lg, co, act);
    for (int off = C; off < (C << lg); off <<= 1) s += __shfl_xor(s, off);
    const T x = (b - s) / d;
    if (act && slice == 0 && live) st_dev(&a.x[r.z * a.rs + co], x);
  }
  persistent_finish(a.state, a.total_waves);
}

// b[i*k + c] = X[i*rs + c*cs], X's place marked.
template <typename T>
__global__ __launch_bounds__(256) void k_rows_begin(int64_t count, int k, int64_t rs, int64_t cs,
                                                    T *X, T *b) {
  for (int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x; t < count;
       t += (int64_t)gridDim.x * 256) {
    const int64_t i = k == 1 ? t : t / k, c = t - i * k;
    T *p = X + i * rs + c * cs;
    b[t] = *p;
    *p = mark_value<T>();
  }
}

// Column-major block B (row i, column c at i + c*ld) through LDS tiles of 64
// rows x 32 columns: begin copies it row-major to b and marks x; end copies x
// back.
template <typename T, bool BEGIN>
__global__ __launch_bounds__(256) void k_rows_turn(int n, int k, int64_t ld, T *B, T *b, T *x) {
  __shared__ T tile[64][33];
  const int i0 = blockIdx.x * 64, c0 = blockIdx.y * 32;
  const int tr = threadIdx.x % 64, tc = threadIdx.x / 64;
  const int wc = threadIdx.x % 32, wr = threadIdx.x / 32;
  if (BEGIN) {
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int c = tc + 4 * m, i = i0 + tr;
      if (i < n && c0 + c < k) tile[tr][c] = B[i + (int64_t)(c0 + c) * ld];
    }
  } else {
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = wr + 8 * m, i = i0 + r;
      if (i < n && c0 + wc < k) tile[r][wc] = x[(int64_t)i * k + c0 + wc];
    }
  }
  __syncthreads();
  if (BEGIN) {
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int r = wr + 8 * m, i = i0 + r;
      if (i < n && c0 + wc < k) {
        b[(int64_t)i * k + c0 + wc] = tile[r][wc];
        x[(int64_t)i * k + c0 + wc] = mark_value<T>();
      }
    }
  } else {
#pragma unroll
    for (int m = 0; m < 8; ++m) {
      const int c = tc + 4 * m, i = i0 + tr;
      if (i < n && c0 + c < k) B[i + (int64_t)(c0 + c) * ld] = tile[tr][c];
    }
  }
}

// Workgroups per CU: enough to have the rows of the next levels loaded ahead;
// more only poll and slow the chain (n = 1e6, in ms: one right-hand side with
// 512 / 1024 / 2048 waves 0.65 / 0.72 / 0.98; 4 columns with 1024 / 2048 /
// 4096 1.11 / 0.79 / 0.91; 32 columns 2.69 / 1.55 / 1.35).  Where levels are
// wide more do not help either, as the ticket counter is the limit: 27-point
// grid of 96^3 in eight colours, one right-hand side, 512 / 1024 / 2048 / 4096
// waves 0.40 / 0.42 / 0.43 / 0.47.
constexpr int ROWS_PER_CU(int c) { return c == 1 ? 1 : c == 8 ? 1 : 2; }

int rows_cols(int k) { return k == 1 ? 1 : k <= 8 ? 8 : k <= 16 ? 16 : 32; }

// The schedule's shape for C column lanes.  Classes of rows, in solving order:
// those a workgroup shares (0), those of lgmax .. 0 slices (1 .. lgmax + 1),
// short ones (lgmax + 2); up to ROWS_CLASSES.
constexpr int ROWS_CLASSES = 9;
struct RowShape {
  int waves, smax, epl, lgmax;
  bool group, shorts;
  explicit RowShape(int C)
      : waves(rows_waves(C)), smax(64 / C), epl(rows_epl(C)), lgmax(0), group(C > 1),
        shorts(rows_short(C)) {
    while ((1 << lgmax) < smax) ++lgmax;
  }
  __host__ __device__ int classes() const { return lgmax + 3; }
  __device__ int cls(int len) const {
    if (group && len > 2 * epl * smax) return 0;
    if (shorts && len <= ROWS_SHORT) return lgmax + 2;
    int lg = 0;
    while (lg < lgmax && (epl << lg) < len) ++lg;
    return lgmax + 1 - lg;
  }
  // rows of one wave's item, and the item's kind
  __host__ __device__ int rows(int c) const {
    return c == 0 ? 1 : c == lgmax + 2 ? smax * ROWS_PER_LANE : smax >> (lgmax + 1 - c);
  }
  // tickets of a level with these counts
  int64_t tickets(const int *count) const {
    int64_t items = (int64_t)count[0] * waves;
    for (int c = 1; c < classes(); ++c) items += (count[c] + rows(c) - 1) / rows(c);
    return (items + waves - 1) / waves;
  }
  __device__ int kind(int c) const { return c == lgmax + 2 ? ROWS_KIND_SHORT : lgmax + 1 - c; }
};

// Rows of each class, a workgroup per level.
constexpr int ROWS_BUILD = 512;
__global__ __launch_bounds__(ROWS_BUILD) void k_rows_count(RowShape sh,
                                                           const int *__restrict__ lvl,
                                                           const int *__restrict__ rp,
                                                           int *count) {
  __shared__ int cnt[ROWS_CLASSES];
  const int l = blockIdx.x, t = threadIdx.x;
  if (t < ROWS_CLASSES) cnt[t] = 0;
  __syncthreads();
  for (int q = lvl[l] + t; q < lvl[l + 1]; q += ROWS_BUILD)
    atomicAdd(&cnt[sh.cls(rp[q + 1] - 1 - rp[q])], 1);
  __syncthreads();
  if (t < ROWS_CLASSES) count[l * ROWS_CLASSES + t] = cnt[t];
}

// Records and items of a level, a workgroup per level: per level the rows a
// workgroup shares, then the others by descending slices, each class in level
// order; waves of a ticket filled from one level, the last ones left empty.
// first[l] .. first[l + 1]: the level's items.
__global__ __launch_bounds__(ROWS_BUILD) void k_rows_fill(RowShape sh,
                                                          const int *__restrict__ lvl,
                                                          const int *__restrict__ rp,
                                                          const int *__restrict__ perm,
                                                          const int *__restrict__ count,
                                                          const int64_t *__restrict__ first,
                                                          int4 *rec, int4 *item) {
  __shared__ int next[ROWS_CLASSES], base[ROWS_CLASSES + 1];
  __shared__ int in_wave[ROWS_BUILD / 64][ROWS_CLASSES];
  const int l = blockIdx.x, t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int q0 = lvl[l], q1 = lvl[l + 1], nc = sh.classes();
  if (t == 0) {
    base[0] = 0;
    for (int c = 0; c < ROWS_CLASSES; ++c) {
      next[c] = base[c];
      base[c + 1] = base[c] + count[l * ROWS_CLASSES + c];
    }
  }
  __syncthreads();
  int4 *const it = item + first[l];
  for (int qb = q0; qb < q1; qb += ROWS_BUILD) {
    const int q = qb + t;
    const int c = q < q1 ? sh.cls(rp[q + 1] - 1 - rp[q]) : -1;
    int rank = 0;
    for (int k = 0; k < nc; ++k) {
      const unsigned long long m = __ballot(c == k);
      if (c == k) rank = __popcll(m & ((1ull << lane) - 1));
      if (lane == 0) in_wave[wave][k] = __popcll(m);
    }
    __syncthreads();
    if (c >= 0) {
      int at = next[c] + rank;
      for (int w = 0; w < wave; ++w) at += in_wave[w][c];
      int4 r = make_int4(rp[q], rp[q + 1] - 1, perm[q], 0);
      rec[q0 + at] = r;
      if (c == 0) {
        r.w = ROWS_KIND_GROUP;
        for (int w = 0; w < sh.waves; ++w) it[(int64_t)at * sh.waves + w] = r;
      }
    }
    __syncthreads();
    if (t < nc)
      for (int w = 0; w < ROWS_BUILD / 64; ++w) next[t] += in_wave[w][t];
    __syncthreads();
  }
  int64_t at = (int64_t)base[1] * sh.waves;
  for (int c = 1; c < nc; ++c) {
    const int R = sh.rows(c), n = base[c + 1] - base[c], items = (n + R - 1) / R;
    for (int i = t; i < items; i += ROWS_BUILD)
      it[at + i] = make_int4(q0 + base[c] + i * R, min(R, n - i * R), 0, sh.kind(c));
    at += items;
  }
  for (int64_t i = at + t; i < first[l + 1] - first[l]; i += ROWS_BUILD)
    it[i] = make_int4(0, 0, 0, 0);
}

// Device scratch given back to the stream.
struct RowScratch {
  hipStream_t stream;
  std::vector<void *> ptrs;
  explicit RowScratch(hipStream_t s) : stream(s) {}
  ~RowScratch() {
    for (void *q : ptrs) (void)hipFreeAsync(q, stream);
  }
  template <typename T>
  bool get(T **q, size_t count) {
    if (hipMallocAsync((void **)q, sizeof(T) * count, stream) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    ptrs.push_back(*q);
    return true;
  }
};

// The schedule for C column lanes is made on the device (a host pass over the
// rows and the copies of their arrays took 6 ms of the first solve of the Zipf
// matrix); the host only adds up the levels' items.
int count_rows(symamd_plan p, int C, hipStream_t stream, RowSchedule &s) {
  const RowShape sh(C);
  const int L = p->levels;
  RowScratch scratch(stream);
  int *d_count = nullptr;
  s.count.resize((size_t)L * ROWS_CLASSES);
  if (!scratch.get(&d_count, s.count.size()))
    return fail(SYMAMD_ERR_ALLOC, "row schedule for %d rows", p->n);
  k_rows_count<<<L, ROWS_BUILD, 0, stream>>>(sh, p->d_lvl_ptr, p->d_rp, d_count);
  SYMAMD_HIP(hipGetLastError());
  SYMAMD_HIP(hipMemcpyAsync(s.count.data(), d_count, sizeof(int) * s.count.size(),
                            hipMemcpyDeviceToHost, stream));
  SYMAMD_HIP(hipStreamSynchronize(stream));
  int64_t tickets = 0;
  for (int l = 0; l < L; ++l) tickets += sh.tickets(&s.count[(size_t)l * ROWS_CLASSES]);
  s.tickets = (int)tickets;
  return SYMAMD_OK;
}

int build_rows(symamd_plan p, int C, hipStream_t stream, RowSchedule &s) {
  const RowShape sh(C);
  const int L = p->levels;
  RowScratch scratch(stream);
  int *d_count = nullptr;
  int64_t *d_first = nullptr;
  std::vector<int64_t> first(L + 1, 0);
  for (int l = 0; l < L; ++l)
    first[l + 1] = first[l] + sh.waves * (int64_t)sh.tickets(&s.count[(size_t)l * ROWS_CLASSES]);
  if (!scratch.get(&d_count, s.count.size()) || !scratch.get(&d_first, first.size()) ||
      hipMalloc(&s.d_rec, sizeof(int4) * std::max(p->n, 1)) != hipSuccess ||
      hipMalloc(&s.d_item, sizeof(int4) * std::max<int64_t>(first[L], 1)) != hipSuccess) {
    (void)hipGetLastError();
    return fail(SYMAMD_ERR_ALLOC, "row schedule for %d rows", p->n);
  }
  SYMAMD_HIP(hipMemcpyAsync(d_count, s.count.data(), sizeof(int) * s.count.size(),
                            hipMemcpyHostToDevice, stream));
  SYMAMD_HIP(hipMemcpyAsync(d_first, first.data(), sizeof(int64_t) * first.size(),
                            hipMemcpyHostToDevice, stream));
  k_rows_fill<<<L, ROWS_BUILD, 0, stream>>>(sh, p->d_lvl_ptr, p->d_rp, p->d_perm, d_count, d_first,
                                            s.d_rec, s.d_item);
  SYMAMD_HIP(hipGetLastError());
  // what was built serves solves on any stream from here on
  SYMAMD_HIP(hipStreamSynchronize(stream));
  std::vector<int>().swap(s.count);
  return SYMAMD_OK;
}

// The schedule, counted or built on first use.  While a caller records the
// handle's stream that is done on a stream of its own (rows_path has seen that
// one was counted before, so the plan's arrays are in place).  Without the
// memory the plan remembers so, for this number of column lanes.
int rows_schedule(symamd_handle h, symamd_plan p, int C, bool build, RowSchedule **out) {
  auto found = p->rows.find(C);
  if (found == p->rows.end() || (build && !found->second.d_rec && !found->second.failed)) {
    const bool cap = capturing(h->stream);
    RelaxedCapture relaxed;
    hipStream_t own = nullptr;
    if (cap) SYMAMD_HIP(hipStreamCreateWithFlags(&own, hipStreamNonBlocking));
    const hipStream_t stream = cap ? own : h->stream;
    RowSchedule s;
    int rc = SYMAMD_OK;
    try {
      if (found != p->rows.end())
        s = found->second;
      else
        rc = count_rows(p, C, stream, s);
      if (rc == SYMAMD_OK && build) rc = build_rows(p, C, stream, s);
    } catch (const std::bad_alloc &) {
      rc = fail(SYMAMD_ERR_ALLOC, "row schedule for %d rows", p->n);
    }
    if (own) (void)hipStreamDestroy(own);
    if (rc != SYMAMD_OK) {
      if (s.d_rec) (void)hipFree(s.d_rec);
      if (s.d_item) (void)hipFree(s.d_item);
      if (rc != SYMAMD_ERR_ALLOC) return rc;
      s = RowSchedule();
      s.failed = true;
    }
    found = p->rows.insert_or_assign(C, std::move(s)).first;
  }
  *out = &found->second;
  return found->second.failed ? fail(SYMAMD_ERR_ALLOC, "row schedule for %d rows", p->n)
                              : SYMAMD_OK;
}

// Whether the tickets take no longer than the units would.  The unit executor
// spends its time on levels (6.6 us each, and 0.25 us for every entry that a
// lane of the longest row adds) and, where those are wide, on entries (15.5 ps
// each) and on the values of wide blocks (2.2 ps each); this one on tickets,
// which workgroups take from one counter (13 ns each for one right-hand side,
// 12.2 with 8 column lanes, or 24 ps an entry where rows take several rounds;
// 9.6 and 10 with 16 and 32, against which the units start 15 and 20 us ahead).  So long chains of narrow levels run here and
// few wide levels on the units.  The constants are fitted to which of the two
// was faster on 46 patterns in FP64 and FP32; near the line the side taken is up
// to a fifth slower than the other.  In ms, units / here, the side taken after it: 27-point
// grid of 96^3 in natural order (666 levels) k = 1 2.90 / 1.03, k = 32 4.40 /
// 1.78, here; in eight colours 0.16 / 0.40, 0.82 / 1.15, units, of 64^3 0.11 /
// 0.14, 0.26 / 0.38, units; 20 levels of 20,000 rows of 12 entries k = 1 0.22 /
// 0.17, here, k = 32 0.54 / 0.71, units; 100 levels of 4,000 k = 32 1.14 / 0.76,
// here; 40 of 8,000 rows of 40 entries k = 1 0.49 / 0.49, k = 32 0.91 / 3.78,
// units; two levels, 300,000 rows of 64 entries, 0.36 / 0.42, 0.62 / 3.29, units;
// 64 levels of 1,500 rows of up to 63 entries k = 32 0.64 / 0.70, here.
bool tickets_win(symamd_plan p, int k, int lanes, int tile, int tickets) {
  const int C = rows_cols(k), eff = std::max(1, std::min(lanes, 64 / tile_cols(k, tile)));
  const double units = p->levels * (6600.0 + 250.0 * p->max_row_nnz / eff) + 0.0155 * p->nnz +
                       (k <= 8 ? 0.0 : 0.0022) * p->n * k;
  const double rows = C == 1 ? 13.0 * tickets : C == 8 ? std::max(12.2 * tickets, 0.024 * p->nnz)
                      : C == 16 ? 15000.0 + 9.6 * tickets : 20000.0 + 10.0 * tickets;
  return rows <= units;
}

template <typename T, int C>
int launch_rows_c(symamd_handle h, RowArgs<T> a) {
  constexpr int W = rows_waves(C);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_rows<T, C>, 64 * W,
                                                   0) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  int64_t grid = (int64_t)std::min(per_cu, ROWS_PER_CU(C)) * h->num_cus;
  if (h->max_waves > 0) grid = std::min<int64_t>(grid, (h->max_waves + W - 1) / W);
  grid = std::max<int64_t>(1, std::min<int64_t>(grid, (int64_t)a.ntick * a.tiles));
  a.total_waves = (int)grid * W;
  k_rows<T, C><<<(unsigned)grid, 64 * W, 0, h->stream>>>(a);
  SYMAMD_HIP(hipGetLastError());
  return SYMAMD_OK;
}

template <typename T>
int launch_rows_t(symamd_handle h, symamd_plan p, void *d_B, int k, int64_t ld, int64_t rs,
                  int64_t cs, bool turn) {
  RowSchedule *s = nullptr;
  const int C = rows_cols(k);
  SYMAMD_TRY(rows_schedule(h, p, C, true, &s));
  const int64_t count = (int64_t)p->n * k;
  RowArgs<T> a{};
  a.rec = s->d_rec;
  a.item = s->d_item;
  a.ntick = s->tickets;
  a.tiles = (k + C - 1) / C;
  a.ci = p->d_ci;
  a.val = (const T *)p->d_val;
  T *const b = (T *)p->d_ws;
  a.b = b;
  a.k = k;
  a.state = p->d_state;
  a.timeout = h->timeout_ticks();
  const dim3 tg((unsigned)((p->n + 63) / 64), (unsigned)((k + 31) / 32));
  if (turn) {
    a.x = b + count;
    a.rs = k;
    a.cs = 1;
    k_rows_turn<T, true><<<tg, 256, 0, h->stream>>>(p->n, k, ld, (T *)d_B, b, a.x);
  } else {
    a.x = (T *)d_B;
    a.rs = rs;
    a.cs = cs;
    const unsigned grid = (unsigned)std::min<int64_t>((count + 255) / 256, 8192);
    k_rows_begin<T><<<grid, 256, 0, h->stream>>>(count, k, rs, cs, a.x, b);
  }
  SYMAMD_HIP(hipGetLastError());
  switch (C) {
    case 1: SYMAMD_TRY((launch_rows_c<T, 1>(h, a))); break;
    case 8: SYMAMD_TRY((launch_rows_c<T, 8>(h, a))); break;
    case 16: SYMAMD_TRY((launch_rows_c<T, 16>(h, a))); break;
    default: SYMAMD_TRY((launch_rows_c<T, 32>(h, a)));
  }
  if (turn) {
    k_rows_turn<T, false><<<tg, 256, 0, h->stream>>>(p->n, k, ld, (T *)d_B, b, a.x);
    SYMAMD_HIP(hipGetLastError());
  }
  return SYMAMD_OK;
}

}  // namespace

// Bytes of the workspace: the right-hand sides, and for turned blocks the
// solution.
static size_t rows_bytes(symamd_plan p, int k, bool turn) {
  return (size_t)p->n * k * (turn ? 2 : 1) * (p->dtype == SYMAMD_F64 ? 8 : 4);
}

// Whether a solve of k right-hand sides runs here: sync-free, the marked
// protocol on, no unit trace, memory for the schedule and the workspace, and
// either the tuner timed it so or, untuned, several lanes per row fit beside
// the unit executor's column tile (one lane per row keeps the reference's
// order in every row, which that one does; so it also solves untuned blocks of
// more than 32 columns) and the tickets take no longer.  A solve being recorded
// by the caller needs an earlier one, as the unit executor does; it runs here
// where the units it would need were not built by that one.
bool rows_path(symamd_handle h, symamd_plan p, int k, bool turn, int exec, const Choice &c) {
  if (exec != SYMAMD_EXEC_SYNCFREE || c.rows == 0 || h->unmarked || h->trace ||
      rows_bytes(p, k, turn) >= p->rows_limit || p->n == 0)
    return false;
  if (c.rows < 0 && (c.lanes < 2 || 2 * tile_cols(k, c.tile) > 64)) return false;
  const bool cap = capturing(h->stream);
  if (cap && p->rows.empty()) return false;
  RowSchedule *s = nullptr;
  if (rows_schedule(h, p, rows_cols(k), false, &s) != SYMAMD_OK) return false;
  if (c.rows > 0 || tickets_win(p, k, c.lanes, c.tile, s->tickets)) return true;
  return cap && !p->units.count(2 * forward_rows_per_unit(k, c.lanes, c.tile));
}

// The schedule and the workspace, before any launch or capture.  A workspace
// that did not fit is not asked for again, nor is a larger one.
int prepare_rows(symamd_handle h, symamd_plan p, int k, bool turn) {
  RowSchedule *s = nullptr;
  SYMAMD_TRY(rows_schedule(h, p, rows_cols(k), true, &s));
  const size_t bytes = rows_bytes(p, k, turn);
  const int rc = plan_workspace(h, p, bytes);
  if (rc == SYMAMD_ERR_ALLOC) p->rows_limit = bytes;
  return rc;
}

// B in place; turn: a column-major block of leading dimension ld through the
// row-major workspace.  prepare_rows must have run.
int launch_rows(symamd_handle h, symamd_plan p, void *d_B, int k, int64_t ld, int64_t rs,
                int64_t cs, bool turn) {
  if (p->n == 0 || k == 0) return SYMAMD_OK;
  return p->dtype == SYMAMD_F64 ? launch_rows_t<double>(h, p, d_B, k, ld, rs, cs, turn)
                                : launch_rows_t<float>(h, p, d_B, k, ld, rs, cs, turn);
}

}  // namespace symamd
