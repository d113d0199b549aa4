// query.hip -- radius queries over a diagram's grid (celery.rs:700-855,
// :1023-1075; interface.rs:348-365).
//
// Two passes over the same walk: the first counts each query's results, a
// u64 scan turns the counts into CSR offsets, the second writes the ids in
// the reference's order.
//
// Box queries walk the index box of the query in (i, j, k) loop order.  The
// cells of a row (i, j) that the radius reaches are one interval of k (the
// gap distance only grows away from the query's cell), and consecutive cells
// are consecutive in the grid order, so a row is one run of points (or cell
// ids) found from two delimiters.  A query has 16 lanes, a row each, and long
// rows are walked by the whole wavefront; the fill pass of a few thousand
// queries and fewer gives each a wavefront.  The neighbour cloud walks the
// shell table in canonical order, 64 entries per step, until the first key
// above the radius.
//
// The points of a step's runs are walked one per lane, so loads and stores of
// neighbouring lanes are neighbouring addresses.  Large query sets are taken
// in grid order of their positions, so the wavefronts running together read
// the same grid cells.  The walk is bound by the instructions around each 64
// points and by the reads of delimiters, sorted indices and point records:
// integer and byte work.
#include "launch.h"
#include "tess_internal.h"

namespace tess {

namespace {

__device__ __forceinline__ int q_axis_index(double v, double vmin, double vmax, double inv, int cpd) {
  if (v >= vmax) return cpd - 1;  // celery.rs:269-282
  double t = (v - vmin) * inv;
  if (!(t > 0.0)) return 0;       // saturating cast, NaN -> 0
  if (t >= 2147483647.0) return cpd - 1;
  int i = (int)t;
  return i < cpd - 1 ? i : cpd - 1;
}

// celery.rs:682-697: the first argument only when strictly smaller / larger.
__device__ __forceinline__ double min_float(double a, double b) { return a < b ? a : b; }
__device__ __forceinline__ double max_float(double a, double b) { return a > b ? a : b; }

__device__ __forceinline__ int cell_gap(int a, int b) {
  const int d = (a > b ? a - b : b - a) - 1;
  return d > 0 ? d : 0;
}

// Within one wavefront LDS operations execute in issue order: a phase
// boundary only has to keep the compiler from moving LDS accesses across it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Lane l's value as a scalar.
__device__ __forceinline__ uint32_t lane_u(uint32_t v, int l) {
  return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ double lane_d(double v, int l) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  return __longlong_as_double(
      (long long)(((unsigned long long)lane_u((uint32_t)(u >> 32), l) << 32) | lane_u((uint32_t)u, l)));
}

// Running maximum over the lanes (inclusive), values >= -1: DPP row shifts
// inside the rows of 16, then row broadcasts (lanes without a source: -1).
__device__ __forceinline__ int wave_max_scan(int v) {
  int t;
  t = __builtin_amdgcn_update_dpp(-1, v, 0x111, 0xf, 0xf, false); v = t > v ? t : v;  // row_shr:1
  t = __builtin_amdgcn_update_dpp(-1, v, 0x112, 0xf, 0xf, false); v = t > v ? t : v;  // row_shr:2
  t = __builtin_amdgcn_update_dpp(-1, v, 0x114, 0xf, 0xf, false); v = t > v ? t : v;  // row_shr:4
  t = __builtin_amdgcn_update_dpp(-1, v, 0x118, 0xf, 0xf, false); v = t > v ? t : v;  // row_shr:8
  t = __builtin_amdgcn_update_dpp(-1, v, 0x142, 0xa, 0xf, false); v = t > v ? t : v;  // row_bcast:15
  t = __builtin_amdgcn_update_dpp(-1, v, 0x143, 0xc, 0xf, false); v = t > v ? t : v;  // row_bcast:31
  return v;
}

// Exclusive prefix of v over the wavefront; *total = the sum.  DPP row
// shifts inside each row of 16 lanes, then the row totals broadcast by
// row_bcast:15 / :31 (lanes without a source add 0).
__device__ __forceinline__ uint32_t wave_excl(uint32_t v, int lane, uint32_t* total) {
  (void)lane;
  int x = (int)v;
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xa, 0xf, false);  // row_bcast:15 -> rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xc, 0xf, false);  // row_bcast:31 -> rows 2, 3
  *total = (uint32_t)__builtin_amdgcn_readlane(x, 63);
  return (uint32_t)x - v;
}

// Runs of at least this many points (on average over a step's runs) are
// walked one by one by the whole wavefront: no search for a position's run
// (or, with 16 lanes a query, four times the lanes), but the last 64 of every
// run are part empty.  At 1M clustered points (290 a run) the fill pass of 1M
// real-radius queries took 1.92 ms with a wavefront per query so and 2.45 ms
// with the runs' concatenation searched; between 15 and 35 points a run the
// two forms are within 5 %.
constexpr uint32_t kRunWalkMin = 48;

// The points of the step's 64 runs, in lane order: lane l's run holds len
// points from grid position s0 on (len 0: none).  MODE 0 keeps every point
// (only the count is needed in the count pass), MODE 1 the points within the
// radius (celery.rs:700-702, :843-851), MODE 2 the points of the target group
// (interface.rs:358-361), MODE 3 lists the positions themselves (cell ids);
// kept points are written in walk order (ballot rank).  Long runs are walked
// one after another; short ones as their concatenation, 64 positions at a
// time, a lane finding its run from heads marked in LDS.
template <int MODE>
__device__ __forceinline__ bool keep_point(const QueryArgs& a, uint32_t s, double qx, double qy, double qz, double r2,
                                           uint32_t& id) {
  if (MODE == 3) {
    id = s;
    return true;
  }
  if (MODE == 1) {
    const PointRec pr = a.pts[s];
    id = pr.id;
    const double dx = qx - pr.x, dy = qy - pr.y, dz = qz - pr.z;
    return (dx * dx + dy * dy) + dz * dz <= r2;
  }
  id = a.sorted[s];
  return MODE == 0 || a.groups[s] == a.target_group;
}

template <int MODE, bool FILL>
__device__ __forceinline__ void emit_points(const QueryArgs& a, uint32_t s0, uint32_t len, int lane, double qx,
                                            double qy, double qz, double r2, uint64_t& cursor, uint64_t end,
                                            uint8_t* head) {
  constexpr bool ALL = MODE == 0 || MODE == 3;
  uint32_t total;
  const uint32_t start = wave_excl(len, lane, &total);
  if (ALL && !FILL) {
    cursor += total;
    return;
  }
  const uint64_t below = (1ull << lane) - 1ull;
  const uint64_t runs = __ballot(len > 0);
  if (total >= kRunWalkMin * (uint32_t)__popcll(runs)) {
    for (uint64_t m = runs; m;) {
      const int l = __builtin_ctzll(m);
      m &= m - 1ull;
      const uint32_t b = (uint32_t)__builtin_amdgcn_readlane((int)s0, l);
      const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)len, l);
      for (uint32_t p = (uint32_t)lane; p < n + (uint32_t)lane; p += 64) {  // whole wavefronts
        uint32_t id = 0;
        const bool keep = p < n && keep_point<MODE>(a, b + p, qx, qy, qz, r2, id);
        if (ALL) {
          if (keep && cursor + p < end) a.ids[cursor + p] = id;
        } else {
          const uint64_t km = __ballot(keep);
          if (FILL && keep) {
            const uint64_t pos = cursor + (uint64_t)__popcll(km & below);
            if (pos < end) a.ids[pos] = id;
          }
          cursor += (uint64_t)__popcll(km);
        }
      }
      if (ALL) cursor += n;
    }
    return;
  }
  int carry = 0;  // the run holding the last position of the previous window
  for (uint32_t base = 0; base < total; base += 64) {
    const uint32_t p = base + (uint32_t)lane;
    // the run of position p: the last non-empty one starting at or before p
    // (each writes its lane at its start in this window, then a running
    // maximum; before the window's first start, the carried run)
    head[lane] = 0xff;
    wave_sync();
    if (len > 0 && start >= base && start - base < 64u) head[start - base] = (uint8_t)lane;
    wave_sync();
    const int h = head[lane];
    int c = wave_max_scan(h == 0xff ? -1 : h);
    c = c > carry ? c : carry;
    carry = __builtin_amdgcn_readlane(c, 63);
    wave_sync();
    const uint32_t cs0 = __shfl(s0, c, 64), cstart = __shfl(start, c, 64);
    uint32_t id = 0;
    const bool keep = p < total && keep_point<MODE>(a, cs0 + (p - cstart), qx, qy, qz, r2, id);
    if (ALL) {
      if (keep && cursor + p < end) a.ids[cursor + p] = id;
    } else {
      const uint64_t m = __ballot(keep);
      if (FILL && keep) {
        const uint64_t pos = cursor + (uint64_t)__popcll(m & below);
        if (pos < end) a.ids[pos] = id;
      }
      cursor += (uint64_t)__popcll(m);
    }
  }
  if (ALL) cursor += total;
}

// The index box of a query and its rows.
struct QueryBox {
  int i0, j0, k0, k1, hx, hy, hz;
  uint32_t nj, rows;  // rows 0: nothing in reach
  double r2;
};

// A z extent past the largest double has cells of infinite size: a gap of 0
// cells is then no number (0 x inf) and out of reach, a gap of 1 and more in
// reach of an infinite radius^2, and a row's cells in reach are no interval.
// Its rows are taken cell by cell.  (Infinite or no number, by the exponent:
// on the scalar unit.)
__device__ __forceinline__ bool cell_by_cell(const GridDev& G) {
  return ((uint32_t)((unsigned long long)__double_as_longlong(G.sz) >> 52) & 0x7ffu) == 0x7ffu;
}

__device__ __forceinline__ QueryBox query_box(const GridDev& G, double qx, double qy, double qz, double r) {
  QueryBox q;
  const int cpd = G.cpd;
  q.i0 = q_axis_index(max_float(qx - r, G.xmin), G.xmin, G.xmax, G.ix, cpd);
  q.j0 = q_axis_index(max_float(qy - r, G.ymin), G.ymin, G.ymax, G.iy, cpd);
  q.k0 = q_axis_index(max_float(qz - r, G.zmin), G.zmin, G.zmax, G.iz, cpd);
  const int i1 = q_axis_index(min_float(qx + r, G.xmax), G.xmin, G.xmax, G.ix, cpd);
  const int j1 = q_axis_index(min_float(qy + r, G.ymax), G.ymin, G.ymax, G.iy, cpd);
  q.k1 = q_axis_index(min_float(qz + r, G.zmax), G.zmin, G.zmax, G.iz, cpd);
  q.hx = q_axis_index(qx, G.xmin, G.xmax, G.ix, cpd);
  q.hy = q_axis_index(qy, G.ymin, G.ymax, G.iy, cpd);
  q.hz = q_axis_index(qz, G.zmin, G.zmax, G.iz, cpd);
  q.r2 = r * r;
  const int ni = i1 - q.i0 + 1, nj = j1 - q.j0 + 1;
  q.nj = nj > 0 ? (uint32_t)nj : 0u;
  // a NaN radius admits no cell (ds <= NaN is false): skip the walk
  q.rows = ni > 0 && nj > 0 && q.k1 >= q.k0 && r == r ? (uint32_t)ni * (uint32_t)nj : 0u;
  if (cell_by_cell(G)) q.rows *= (uint32_t)(q.k1 - q.k0 + 1);  // (at most cpd^3, 10^9)
  return q;
}

// Row t of the box: its cells in reach are first .. first + count - 1.
// celery.rs:708-743: the gap distance of the query's cell to (i, j, k) is
// compared with the radius; along k it falls to the query's cell and rises
// after it, so the reached cells are an interval, whose ends a bisection of
// k0 .. hz and of hz .. k1 finds (the query's own k is reached if any is).
// With a negative radius hz may lie outside k0 .. k1: then the interval is
// bounded on the other side by the box.
__device__ __forceinline__ uint32_t query_row(const GridDev& G, const QueryBox& q, uint32_t t, uint32_t& first) {
  const int cpd = G.cpd;
  int ka = q.k0, kb = q.k1;
  if (cell_by_cell(G)) {
    const uint32_t nk = (uint32_t)(q.k1 - q.k0 + 1);
    ka = kb = q.k0 + (int)(t % nk);
    t /= nk;
  }
  const int i = q.i0 + (int)(t / q.nj), j = q.j0 + (int)(t % q.nj);
  const double gx = (double)cell_gap(q.hx, i) * G.sx, gy = (double)cell_gap(q.hy, j) * G.sy;
  const double g2 = gx * gx + gy * gy;
  auto in = [&](int k) {
    const double gz = (double)cell_gap(q.hz, k) * G.sz;
    return g2 + gz * gz <= q.r2;
  };
  first = ((uint32_t)i * (uint32_t)cpd + (uint32_t)j) * (uint32_t)cpd;  // celery.rs:317-325
  // the box's k nearest the query's
  const int near = q.hz < ka ? ka : (q.hz > kb ? kb : q.hz);
  if (!in(near)) return 0;
  for (int hi = near; ka < hi;) {  // the smallest k in reach is in ka .. hi
    const int mid = (ka + hi) >> 1;
    if (in(mid))
      hi = mid;
    else
      ka = mid + 1;
  }
  for (int lo = near; lo < kb;) {  // the largest is in lo .. kb
    const int mid = (lo + kb + 1) >> 1;
    if (in(mid))
      lo = mid;
    else
      kb = mid - 1;
  }
  first += (uint32_t)ka;
  return (uint32_t)(kb - ka + 1);
}

// find_cells_in_radius (KIND 0) and the two neighbour searches built on it
// (KIND 1 cell radius, KIND 2 real radius): celery.rs:753-855.

// Cells or points of every query's rows (unfiltered: an upper bound for KIND
// 2), 16 lanes (a DPP row) per query, a row of the box each.  1M queries of
// 10 cells: 120 us (one wavefront per query, a lane per cell: 450 us).
template <int KIND>
__global__ __launch_bounds__(256) void k_query_box_count(QueryArgs a) {
  const int sub = threadIdx.x & 15;
  const uint32_t w = blockIdx.x * 16u + (threadIdx.x >> 4);
  const bool live = w < (uint32_t)a.nq;
  const uint32_t qi = live ? (a.order ? a.order[w] : w) : 0u;
  const double* p = a.q + 3 * (size_t)qi;
  QueryBox q = query_box(a.g, p[0], p[1], p[2], a.radius[(size_t)qi * a.rstride]);
  uint32_t sum = 0;
  if (live)
    for (uint32_t t = (uint32_t)sub; t < q.rows; t += 16) {
      uint32_t first;
      const uint32_t n = query_row(a.g, q, t, first);
      if (n) sum += KIND == 0 ? n : a.delim[first + n] - a.delim[first];
    }
  int v = (int)sum;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  if (live && sub == 15) a.count[qi] = (uint32_t)v;
}

// The ids (without FILL their exact number): 16 lanes per query, 16 rows of
// the box per step, so that four queries share the instructions of the walk's
// set-up.  Short rows are walked by the query's 16 lanes; when the step's rows
// hold kRunWalkMin points or more on average, the whole wavefront takes them,
// one query after the other, and reads 64 neighbouring points at a time.
// a.count (nullable): ids per query.  Fill pass of 1M queries, one wavefront
// per query over 64 cells a step before: real radius at clustered points (124
// ids) 2.89 -> 1.63 ms, at uniform points (5 ids) 0.65 -> 0.29 ms; cell radius
// at clustered points (1,183 ids) 2.49 -> 1.96 ms.
template <int KIND, bool FILL>
__global__ __launch_bounds__(256) void k_query_box(QueryArgs a) {
  constexpr int MODE = KIND == 0 ? 3 : (KIND == 1 ? 0 : 1);
  constexpr bool ALL = MODE != 1;
  constexpr int kAhead = 2;  // points of every lane in flight
  const int lane = threadIdx.x & 63, sub = lane & 15, group = lane & 48;
  const uint32_t w = blockIdx.x * 16u + (threadIdx.x >> 4);
  const bool live = w < (uint32_t)a.nq;
  const uint32_t qi = live ? (a.order ? a.order[w] : w) : 0u;
  const double qx = a.q[3 * (size_t)qi], qy = a.q[3 * (size_t)qi + 1], qz = a.q[3 * (size_t)qi + 2];
  QueryBox q = query_box(a.g, qx, qy, qz, a.radius[(size_t)qi * a.rstride]);
  if (!live) q.rows = 0;
  const uint64_t begin = FILL ? a.offsets[qi] : 0;
  const uint32_t room = FILL ? (uint32_t)(a.offsets[qi + 1] - begin) : 0u;
  uint32_t cursor = 0;  // ids listed so far
  for (uint32_t base = 0; __ballot(base < q.rows); base += 16) {
    uint32_t s0 = 0, len = 0;
    if (base < q.rows && (uint32_t)sub < q.rows - base) {
      uint32_t first;
      const uint32_t n = query_row(a.g, q, base + (uint32_t)sub, first);
      if (KIND == 0) {
        s0 = first;
        len = n;
      } else if (n) {
        s0 = a.delim[first];
        len = a.delim[first + n] - s0;
      }
    }
    const uint64_t all = __ballot(len > 0);
    uint32_t total;
    (void)wave_excl(len, lane, &total);
    if (total >= kRunWalkMin * (uint32_t)__popcll(all)) {
      for (int g = 0; g < 64; g += 16) {
        uint32_t runs = (uint32_t)(all >> g) & 0xffffu;
        if (!runs) continue;
        const double gx = lane_d(qx, g), gy = lane_d(qy, g), gz = lane_d(qz, g), g2 = lane_d(q.r2, g);
        const uint64_t gbegin = ((uint64_t)lane_u((uint32_t)(begin >> 32), g) << 32) | lane_u((uint32_t)begin, g);
        const uint32_t groom = lane_u(room, g);
        uint32_t at = lane_u(cursor, g);
        uint32_t* ids = a.ids + gbegin;
        for (; runs; runs &= runs - 1u) {
          const int l = g + __builtin_ctz(runs);
          const uint32_t b = lane_u(s0, l), n = lane_u(len, l);
          for (uint32_t p0 = 0; p0 < n; p0 += 64) {
            const uint32_t p = p0 + (uint32_t)lane;
            uint32_t id = 0;
            const bool keep = p < n && keep_point<MODE>(a, b + p, gx, gy, gz, g2, id);
            if (ALL) {
              if (keep && at + p < groom) ids[at + p] = id;
            } else {
              const uint64_t m = __ballot(keep);
              const uint32_t pos = at + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
              if (FILL && keep && pos < groom) ids[pos] = id;
              at += (uint32_t)__popcll(m);
            }
          }
          if (ALL) at += n;
        }
        if (group == g) cursor = at;
      }
      continue;
    }
    uint32_t* ids = a.ids + begin;
    for (uint32_t runs = (uint32_t)(all >> group) & 0xffffu; runs; runs &= runs - 1u) {
      const int l = group + __builtin_ctz(runs);
      const uint32_t b = (uint32_t)__shfl((int)s0, l, 64), n = (uint32_t)__shfl((int)len, l, 64);
      for (uint32_t p0 = 0; p0 < n; p0 += 16 * kAhead) {
        uint32_t id[kAhead];
        bool keep[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          const uint32_t p = p0 + 16u * u + (uint32_t)sub;
          id[u] = 0;
          keep[u] = p < n && keep_point<MODE>(a, b + p, qx, qy, qz, q.r2, id[u]);
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
          if (ALL) {
            const uint32_t pos = cursor + p0 + 16u * u + (uint32_t)sub;
            if (keep[u] && pos < room) ids[pos] = id[u];
          } else {
            const uint32_t m = (uint32_t)(__ballot(keep[u]) >> group) & 0xffffu;
            const uint32_t pos = cursor + (uint32_t)__popc(m & ((1u << sub) - 1u));
            if (FILL && keep[u] && pos < room) ids[pos] = id[u];
            cursor += (uint32_t)__popc(m);
          }
        }
      }
      if (ALL) cursor += n;
    }
  }
  if (live && sub == 0 && a.count) a.count[qi] = cursor;
}

// The same by a wavefront per query, 64 rows a step, for query sets too small
// to fill the chip with four queries a wavefront, whose long rows are walked
// one after the other for all four (kBoxWaveMax).
template <int KIND, bool FILL>
__global__ __launch_bounds__(256) void k_query_box_wave(QueryArgs a) {
  constexpr int MODE = KIND == 0 ? 3 : (KIND == 1 ? 0 : 1);
  __shared__ uint8_t heads[4][64];
  uint8_t* head = heads[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  const uint32_t w = blockIdx.x * 4u + (threadIdx.x >> 6);
  if (w >= (uint32_t)a.nq) return;
  const uint32_t qi = a.order ? a.order[w] : w;
  const double qx = a.q[3 * (size_t)qi], qy = a.q[3 * (size_t)qi + 1], qz = a.q[3 * (size_t)qi + 2];
  const QueryBox q = query_box(a.g, qx, qy, qz, a.radius[(size_t)qi * a.rstride]);
  uint64_t cursor = FILL ? a.offsets[qi] : 0;
  const uint64_t begin = cursor, end = FILL ? a.offsets[qi + 1] : 0;
  for (uint32_t base = 0; base < q.rows; base += 64) {
    uint32_t s0 = 0, len = 0;
    if ((uint32_t)lane < q.rows - base) {
      uint32_t first;
      const uint32_t n = query_row(a.g, q, base + (uint32_t)lane, first);
      if (KIND == 0) {
        s0 = first;
        len = n;
      } else if (n) {
        s0 = a.delim[first];
        len = a.delim[first + n] - s0;
      }
    }
    emit_points<MODE, FILL>(a, s0, len, lane, qx, qy, qz, q.r2, cursor, end, head);
  }
  if (lane == 0 && a.count) a.count[qi] = (uint32_t)(cursor - begin);
}

// Cell::compute_neighbor_cloud: expand_all_in_radius from the query's grid
// cell (celery.rs:1023-1075) + the group filter (interface.rs:358-361).  The
// table covers every key <= the largest radius (or is the full order).
template <bool FILL>
__global__ __launch_bounds__(256) void k_query_cloud(QueryArgs a) {
  __shared__ uint8_t heads[4][64];
  uint8_t* head = heads[threadIdx.x >> 6];
  const int lane = threadIdx.x & 63;
  const int w = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= a.nq) return;
  const int qi = a.order ? (int)a.order[w] : w;
  const GridDev& G = a.g;
  const int cpd = G.cpd;
  const double qx = a.q[3 * (size_t)qi], qy = a.q[3 * (size_t)qi + 1], qz = a.q[3 * (size_t)qi + 2];
  const double r = a.radius[(size_t)qi * a.rstride];
  const int hx = q_axis_index(qx, G.xmin, G.xmax, G.ix, cpd);
  const int hy = q_axis_index(qy, G.ymin, G.ymax, G.iy, cpd);
  const int hz = q_axis_index(qz, G.zmin, G.zmax, G.iz, cpd);
  uint64_t cursor = FILL ? a.offsets[qi] : 0;
  const uint64_t end = FILL ? a.offsets[qi + 1] : 0;
  for (int base = 0; base < a.tlen; base += 64) {
    const int t = base + lane;
    const bool have = t < a.tlen;
    const double key = have ? a.key[t] : 0.0;
    const bool beyond = have && key > r;  // celery.rs:1036: the loop ends here
    const bool take = have && !beyond;    // keys ascend: the taken lanes are a prefix
    uint32_t s0 = 0, len = 0;
    if (take) {
      int ox, oy, oz;
      unpack_off(a.off[t], ox, oy, oz);
      const int bx = hx + ox, by = hy + oy, bz = hz + oz;
      if (bx >= 0 && bx < cpd && by >= 0 && by < cpd && bz >= 0 && bz < cpd) {
        const uint32_t b = ((uint32_t)bx * (uint32_t)cpd + (uint32_t)by) * (uint32_t)cpd + (uint32_t)bz;
        s0 = a.delim[b];
        len = a.delim[b + 1] - s0;
      }
    }
    if (a.groups)
      emit_points<2, FILL>(a, s0, len, lane, qx, qy, qz, 0.0, cursor, end, head);
    else
      emit_points<0, FILL>(a, s0, len, lane, qx, qy, qz, 0.0, cursor, end, head);
    if (__ballot(beyond)) break;
  }
  if (lane == 0 && a.count) a.count[qi] = (uint32_t)(FILL ? cursor - a.offsets[qi] : cursor);
}

// Points of every cloud's grid cells (no group filter): 16 lanes (a DPP row)
// per query, 16 table entries a step, so four queries share a wavefront's
// instructions.  From kCloudCountMin queries on, which then fill the chip:
// 200k queries 80 -> 51 us, 1M 330 -> 140.  Fewer keep a wavefront each, whose chain of
// steps is a quarter as long.
constexpr int kCloudCountMin = 16384;
__global__ __launch_bounds__(256) void k_query_cloud_count(QueryArgs a) {
  const int lane = threadIdx.x & 63, sub = lane & 15, group = lane & 48;
  const uint32_t w = blockIdx.x * 16u + (threadIdx.x >> 4);
  const bool live = w < (uint32_t)a.nq;
  const uint32_t qi = live ? (a.order ? a.order[w] : w) : 0u;
  const GridDev& G = a.g;
  const int cpd = G.cpd;
  const double r = a.radius[(size_t)qi * a.rstride];
  const int hx = q_axis_index(a.q[3 * (size_t)qi], G.xmin, G.xmax, G.ix, cpd);
  const int hy = q_axis_index(a.q[3 * (size_t)qi + 1], G.ymin, G.ymax, G.iy, cpd);
  const int hz = q_axis_index(a.q[3 * (size_t)qi + 2], G.zmin, G.zmax, G.iz, cpd);
  uint32_t sum = 0;
  bool done = !live;
  for (int base = 0; base < a.tlen; base += 16) {
    const int t = base + sub;
    const bool have = !done && t < a.tlen;
    const bool beyond = have && a.key[t] > r;  // celery.rs:1036: the loop ends here
    if (have && !beyond) {
      int ox, oy, oz;
      unpack_off(a.off[t], ox, oy, oz);
      const int bx = hx + ox, by = hy + oy, bz = hz + oz;
      if (bx >= 0 && bx < cpd && by >= 0 && by < cpd && bz >= 0 && bz < cpd) {
        const uint32_t b = ((uint32_t)bx * (uint32_t)cpd + (uint32_t)by) * (uint32_t)cpd + (uint32_t)bz;
        sum += a.delim[b + 1] - a.delim[b];
      }
    }
    done = done || ((__ballot(beyond) >> group) & 0xffffull) != 0;
    if (!__ballot(!done)) break;
  }
  int v = (int)sum;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);  // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);  // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);  // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);  // row_shr:8
  if (live && sub == 15) a.count[qi] = (uint32_t)v;
}

// Queries up to which a box fill gets a wavefront each.  Real-radius calls over
// 200k points, four queries a wavefront and one: 64 queries with 26,000 points
// in their boxes 1,062 and 280 us, 4,096 of them 1,019 and 405, 8,192 1,089
// and 543, 16,384 1,363 and 780; with 6 points in their boxes 72 and 69, 105
// and 111, 104 and 113, 119 and 126, and falling behind from there (65,536:
// 140 and 158).
constexpr int kBoxWaveMax = 8192;

template <int KIND, bool FILL>
void launch_box(const QueryArgs& a, hipStream_t s) {
  if (a.nq <= kBoxWaveMax)
    hipLaunchKernelGGL((k_query_box_wave<KIND, FILL>), dim3((unsigned)((a.nq + 3) / 4)), dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_query_box<KIND, FILL>), dim3((unsigned)((a.nq + 15) / 16)), dim3(256), 0, s, a);
}

template <bool FILL>
hipError_t launch_query_pass(const QueryArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)((a.nq + 3) / 4)), block(256);
  const dim3 grid16((unsigned)((a.nq + 15) / 16));
  switch (a.kind) {
    case 0:
      if (FILL)
        launch_box<0, true>(a, s);
      else
        hipLaunchKernelGGL((k_query_box_count<0>), grid16, block, 0, s, a);
      break;
    case 1:
      if (FILL)
        launch_box<1, true>(a, s);
      else
        hipLaunchKernelGGL((k_query_box_count<1>), grid16, block, 0, s, a);
      break;
    case 2:
      launch_box<2, FILL>(a, s);
      break;
    default:
      if (!FILL && !a.groups && a.nq >= kCloudCountMin)
        hipLaunchKernelGGL(k_query_cloud_count, grid16, block, 0, s, a);
      else
        hipLaunchKernelGGL((k_query_cloud<FILL>), grid, block, 0, s, a);
      break;
  }
  return hipGetLastError();
}

}  // namespace

// Ids of query q from src[from[q] ..] to dst[to[q] .. to[q + 1]): 16 lanes per
// query, eight ids of every lane in flight.  124 ids for each of 1M queries:
// 500 -> 259 us (one wavefront per query, one id of a lane at a time).
__global__ __launch_bounds__(256) void k_query_compact(int nq, const uint64_t* __restrict__ from,
                                                       const uint64_t* __restrict__ to,
                                                       const uint32_t* __restrict__ src,
                                                       uint32_t* __restrict__ dst) {
  constexpr int kAhead = 8;
  const int sub = threadIdx.x & 15;
  const uint32_t q = blockIdx.x * 16u + (threadIdx.x >> 4);
  if (q >= (uint32_t)nq) return;
  const uint64_t t = to[q], m = to[q + 1] - t;
  src += from[q];
  dst += t;
  for (uint64_t k0 = (uint64_t)sub; k0 < m; k0 += 16 * kAhead) {
    uint32_t v[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (k0 + 16 * u < m) v[u] = src[k0 + 16 * u];
#pragma unroll
    for (int u = 0; u < kAhead; ++u)
      if (k0 + 16 * u < m) dst[k0 + 16 * u] = v[u];
  }
}

namespace {

// Largest radius, every workgroup's by one atomic on the order-keeping
// integer.  A cloud query needs it on the host for its shell table; the radii
// themselves took 200 us to come down and be looked through (200k of them).
__global__ __launch_bounds__(256) void k_radius_max(const double* __restrict__ radius, size_t m,
                                                    unsigned long long* __restrict__ key) {
  __shared__ unsigned long long best[4];
  unsigned long long b = 0;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < m; i += (size_t)gridDim.x * 256) {
    const double r = radius[i];
    const unsigned long long u = (unsigned long long)__double_as_longlong(r == r ? r : (double)INFINITY);
    const unsigned long long k = u >> 63 ? ~u : u | 1ull << 63;
    b = k > b ? k : b;
  }
#pragma unroll
  for (int o = 1; o < 64; o *= 2) {
    const unsigned long long v = __shfl_xor(b, o);
    b = v > b ? v : b;
  }
  if ((threadIdx.x & 63) == 0) best[threadIdx.x >> 6] = b;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) b = best[w] > b ? best[w] : b;
    atomicMax(key, b);
  }
}

}  // namespace

hipError_t launch_radius_max(const double* radius, size_t m, uint64_t* key, hipStream_t s) {
  hipError_t e = launch_fill_u32(reinterpret_cast<uint32_t*>(key), 2, 0u, s);
  if (e != hipSuccess || m == 0) return e;
  const size_t blocks = (m + 1023) / 1024;
  hipLaunchKernelGGL(k_radius_max, dim3((unsigned)(blocks < 256 ? blocks : 256)), dim3(256), 0, s, radius, m,
                     reinterpret_cast<unsigned long long*>(key));
  return hipGetLastError();
}

hipError_t launch_query_count(const QueryArgs& a, hipStream_t s) { return launch_query_pass<false>(a, s); }
hipError_t launch_query_fill(const QueryArgs& a, hipStream_t s) { return launch_query_pass<true>(a, s); }
hipError_t launch_query_compact(int nq, const uint64_t* from, const uint64_t* to, const uint32_t* src, uint32_t* dst,
                                hipStream_t s) {
  if (nq <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_query_compact, dim3((unsigned)((nq + 15) / 16)), dim3(256), 0, s, nq, from, to, src, dst);
  return hipGetLastError();
}

}  // namespace tess
