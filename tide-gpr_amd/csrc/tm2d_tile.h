// Workgroup tiles of the 2-D TM propagator and its exact adjoint: one
// launch advances a tile of 64 columns x W*R rows of one shot by several time
// steps.
//
// A workgroup of W wavefronts holds the whole tile in registers: lane = column,
// and each wavefront R consecutive rows.  The tile is loaded once with a halo
// of `halo` cells on every side, advanced step by step, and its inner cells
// stored once.  x-neighbours come from cross-lane moves; of the y-neighbours
// only the first and last rows of a wavefront are exchanged, through LDS, with
// one barrier before each half-step.  Cells near the rim of the tile go stale
// by 2P-1 cells per step and side (P = half the stencil order), so `steps`
// steps need a halo of steps * (2P-1); wavefronts that hold only stale rows
// skip the step.
//
// Why this shape.  A tile of one wavefront recomputes and re-reads a halo of
// K rows on each side of 4 rows; a tile of 32 or 64 rows re-reads a few
// percent, so the state crosses HBM once per 4 to 8 steps and each step costs
// one short pass over registers.  Where a launch has few tiles, its duration
// is that of one wavefront's instruction stream, and a loop over steps of one
// to four rows is many times shorter than a fully unrolled tile.
//
// Every cell update is the single-step expression in the same operation order
// (no FMA contraction), so results do not depend on the tile or the number
// of steps per launch.
#pragma once

#include "tm2d_device.h"
#include "tm2d_stencil.h"

namespace tide_hip {
namespace tm2d {

constexpr int kTileSteps = 8;   // most steps per launch
constexpr int kTileWaves = 16;  // most wavefronts per workgroup

// Order of a problem's tiles in a launch: the tiles that meet a grid edge or a
// CPML strip first, then the rectangle [xa, xb) x [ya, yb) of the others.  Edge
// tiles take longer, so they neither leave a tail nor, dealt by dealt_index,
// load one XCD more than another.  Rows of tiles in one contiguous run per XCD
// gave the first and the last XCD the top and bottom rows; fp32, us per step,
// before and after: 400 x 901 cells and 12 shots forward 18.3 -> 14.0, adjoint
// 49 -> 42; 1024 x 1024 and 4 shots 15.0 -> 11.9 and 32.7 -> 29.7.
struct TileOrder {
  int32_t n_yt, xa, xb, ya, yb;
  __host__ __device__ __forceinline__ int edges(int n_xt) const {
    return n_xt * n_yt - (xb - xa) * (yb - ya);
  }
  // Column and row of the o-th tile.
  __device__ __forceinline__ void at(int o, int n_xt, int &xt, int &yt) const {
    const int wide = xb - xa, top = ya * n_xt, side = (yb - ya) * (n_xt - wide);
    int first = 0, width = n_xt, skip_from = n_xt, skip = 0;  // columns from skip_from on move by skip
    if (o >= edges(n_xt)) {
      o -= edges(n_xt);
      first = ya;
      width = wide;
      skip_from = 0;
      skip = xa;
    } else if (o >= top + side) {
      o -= top + side;
      first = yb;
    } else if (o >= top) {
      o -= top;
      first = ya;
      width = n_xt - wide;
      skip_from = xa;
      skip = wide;
    }
    yt = o / width;
    xt = o - yt * width;
    yt += first;
    if (xt >= skip_from) xt += skip;
  }
};

// Index of workgroup b among n: runs of 16 tiles go to the XCDs in turn.  Each
// XCD gets its share of the edge tiles, and neighbours mostly share an L2.
__device__ __forceinline__ int dealt_index(int b, int n) {
  constexpr int kRun = 16, kAll = 8 * kRun;
  const int first = b & ~(kAll - 1);
  return first + kAll > n ? b : first + (b & 7) * kRun + ((b >> 3) & (kRun - 1));
}

template <typename T> struct TileFwdArgs {
  Geom<T> g;
  Points pts;  // built with build_point_table_lanes(64 - 2 halo, halo)
  const T *ca, *cb, *cq;
  const T *in[7];  // ey hx hz m_ey_x m_ey_z m_hx_z m_hz_x, before the first step
  T *out[7];       // the same after the last step
  const T *f;      // source terms of the first step (null: none) and the
  T *r;            // receiver row of the first step (null: none); the next
  int64_t f_stride, r_stride;  // step's are one stride further
  void *ey_store[kTileSteps], *curl_store[kTileSteps];  // null: no snapshot
  int32_t n_shots, steps, halo, own_rows;
  TileOrder order;
  int32_t tile0;  // first workgroup of the problem in a launch of several
};

template <typename T> struct TileAdjArgs {
  Geom<T> g;
  Points pts;
  const T *ca, *cb, *cq;
  const T *in[7];  // lambda ey hx hz, then the memories of hz_x hx_z ey_x ey_z
  T *out[7];
  const T *grad_r;  // receiver cotangents of the first (latest) step
  T *grad_f;        // source-term gradients of that step (null: not wanted)
  int64_t r_stride, f_stride;
  const void *ey_store[kTileSteps], *curl_store[kTileSteps];  // null: no term
  double *gca, *gcb;  // FP64 accumulators, one plane per shot; null: not wanted
  double step_scale;
  int32_t n_shots, steps, halo, own_rows, tile0;
  TileOrder order;
};

// A kernel's arguments, read anew at each call: the compiler loads every
// kernel argument it can at the kernel's start and keeps it for its last use,
// which overflows the scalar registers; values read through this reference are
// loaded where they are used.  The arguments are those of the kernel itself, or
// an entry of a table that was complete before the launch.
template <typename A> struct ArgRef {
  using P = const A __attribute__((address_space(4))) *;
  P p;
  __device__ __forceinline__ const A &operator()() const {
    P q = p;
    asm volatile("" : "+s"(q));
    return *(const A *)q;
  }
};
template <typename A> __device__ __forceinline__ ArgRef<A> kernel_args() {
  return {(typename ArgRef<A>::P)__builtin_amdgcn_kernarg_segment_ptr()};
}

// A pointer read through an ArgRef, which the compiler does not know to
// point to global memory (it would use flat accesses, whose waits include LDS).
template <typename U> __device__ __forceinline__ U *as_global(U *p) {
  using G = U __attribute__((address_space(1))) *;
  return (U *)(G)p;
}

// Place of this wavefront's rows and lanes in the grid.
struct TilePlace {
  int lane, w, waves, xt, x, y;  // column of this lane, first row of the wave
  int row0;                      // first row of the wave within the tile
  int rows;                      // rows of the tile
  bool edge;                     // the tile meets a grid edge or a CPML strip
};

template <typename T, int P, int R>
__device__ __forceinline__ TilePlace tile_place(const Geom<T> &g, const TileOrder &order, int n_xt,
                                                int tile, int halo, int own_rows) {
  TilePlace c;
  c.lane = threadIdx.x;
  c.w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  c.waves = (int)blockDim.y;
  c.rows = c.waves * R;
  int yt;
  order.at(tile, n_xt, c.xt, yt);
  const int x0 = c.xt * (64 - 2 * halo) - halo, y0 = yt * own_rows - halo;
  c.x = x0 + c.lane;
  c.row0 = c.w * R;
  c.y = y0 + c.row0;
  c.edge = x0 < P || x0 + 63 > g.nx - P - 1 || x0 < g.pml_x0 || x0 + 63 >= g.pml_x1h ||
           y0 < P || y0 + c.rows - 1 > g.ny - P - 1 || y0 < g.pml_y0 ||
           y0 + c.rows - 1 >= g.pml_y1h;
  return c;
}

// LDS rows through which neighbouring wavefronts exchange: of the field read
// ahead (offsets -(P-1) .. P), the first P and last P-1 rows of each
// wavefront; of the field read behind (-P .. P-1), the last P and first P-1.
template <typename T, int P> struct TileRows {
  static constexpr int kRows = 4 * P - 2;  // per wavefront
  T *a_first, *b_last, *a_last, *b_first;  // this lane's column of wavefront 0
  T *amp;        // [waves][steps][64]: see TilePoints
  int *entries;  // [waves][3][64] point-table scratch

  __host__ __device__ static size_t bytes(int waves, int steps) {
    return (size_t)waves * 64 * ((kRows + steps) * sizeof(T) + 3 * sizeof(int));
  }
  __device__ __forceinline__ TileRows(void *mem, int waves, int steps, int lane) {
    T *const p = (T *)mem + lane;
    a_first = p;
    b_last = p + waves * P * 64;
    a_last = p + waves * 2 * P * 64;
    b_first = p + waves * (3 * P - 1) * 64;
    amp = p + waves * kRows * 64;
    entries = (int *)((T *)mem + waves * (kRows + steps) * 64);
  }
  // This lane's amplitude of step j.
  __device__ __forceinline__ const T *amp_at(const TilePlace &c, int steps, int j) const {
    return amp + (c.w * steps + j) * 64;
  }
};

// Publishes the rim rows of `v`, to be read by get_a() / get_b() after the
// next barrier.
template <typename T, int P, int R>
__device__ __forceinline__ void put_a(const TileRows<T, P> &l, const TilePlace &c, const T (&v)[R]) {
#pragma unroll
  for (int k = 0; k < P; ++k) l.a_first[(c.w * P + k) * 64] = v[k];
#pragma unroll
  for (int k = 0; k + 1 < P; ++k) l.a_last[(c.w * (P - 1) + k) * 64] = v[R - (P - 1) + k];
}
template <typename T, int P, int R>
__device__ __forceinline__ void put_b(const TileRows<T, P> &l, const TilePlace &c, const T (&v)[R]) {
#pragma unroll
  for (int k = 0; k < P; ++k) l.b_last[(c.w * P + k) * 64] = v[R - P + k];
#pragma unroll
  for (int k = 0; k + 1 < P; ++k) l.b_first[(c.w * (P - 1) + k) * 64] = v[k];
}
// Rows -(P-1) .. R-1+P of a wavefront's neighbourhood (index 0 = row -(P-1)).
// The outermost wavefronts read their own rows there: stale rim cells.
template <typename T, int P, int R>
__device__ __forceinline__ void get_a(const TileRows<T, P> &l, const TilePlace &c, const T (&v)[R],
                                      T (&out)[R + 2 * P - 1]) {
  const int up = max(c.w - 1, 0), dn = min(c.w + 1, c.waves - 1);
#pragma unroll
  for (int k = 0; k + 1 < P; ++k) out[k] = l.a_last[(up * (P - 1) + k) * 64];
#pragma unroll
  for (int k = 0; k < R; ++k) out[P - 1 + k] = v[k];
#pragma unroll
  for (int k = 0; k < P; ++k) out[P - 1 + R + k] = l.a_first[(dn * P + k) * 64];
}
// Rows -P .. R-1+P-1 (index 0 = row -P).
template <typename T, int P, int R>
__device__ __forceinline__ void get_b(const TileRows<T, P> &l, const TilePlace &c, const T (&v)[R],
                                      T (&out)[R + 2 * P - 1]) {
  const int up = max(c.w - 1, 0), dn = min(c.w + 1, c.waves - 1);
#pragma unroll
  for (int k = 0; k < P; ++k) out[k] = l.b_last[(up * P + k) * 64];
#pragma unroll
  for (int k = 0; k < R; ++k) out[P + k] = v[k];
#pragma unroll
  for (int k = 0; k + 1 < P; ++k) out[P + R + k] = l.b_first[(dn * (P - 1) + k) * 64];
}

// Values of v at lanes -N .. N around each lane (index N = this lane).
template <typename T, int N>
__device__ __forceinline__ void lane_window(T v, T (&s)[2 * N + 1]) {
  s[N] = v;
#pragma unroll
  for (int k = 1; k <= N; ++k) {
    s[N + k] = shfl_dn1(s[N + k - 1]);
    s[N - k] = shfl_up1(s[N - k + 1]);
  }
}

// What holds of each row of a wavefront, one bit per row (wave-uniform).
struct RowBits {
  int e, h;    // in the update domain of Ey and Hz, of Hx
  int pe, ph;  // in a y strip at whole points, at half points
  int own;     // owned by the tile and inside the grid

  template <typename T, int P, int R>
  __device__ __forceinline__ void set(const Geom<T> &g, const TilePlace &c, int halo) {
    e = h = pe = ph = own = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int y = c.y + r;
      e |= (y >= P && y < g.ny - P + 1) << r;
      h |= (y >= P && y < g.ny - P) << r;
      pe |= (y < g.pml_y0 || y >= g.pml_y1) << r;
      ph |= (y < g.pml_y0 || y >= g.pml_y1h) << r;
      own |= (c.row0 + r >= halo && c.row0 + r < c.rows - halo && y < g.ny) << r;
    }
    e = __builtin_amdgcn_readfirstlane(e);
    h = __builtin_amdgcn_readfirstlane(h);
    pe = __builtin_amdgcn_readfirstlane(pe);
    ph = __builtin_amdgcn_readfirstlane(ph);
    own = __builtin_amdgcn_readfirstlane(own);
  }
  // A copy whose tests are made anew wherever it is used: the compiler may not
  // assume it unchanged, and so does not keep a lane mask per row and test
  // across the time loop, which overflows the scalar registers.
  __device__ __forceinline__ RowBits again() const {
    RowBits b = *this;
    asm volatile("" : "+s"(b.e), "+s"(b.h), "+s"(b.pe), "+s"(b.ph), "+s"(b.own));
    return b;
  }
};

// Waits for every load in flight.  Without it the waits for the loads before
// a time loop stand inside the loop, where they also wait for the snapshot
// stores of the previous step (loads and stores share one counter).
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), the other counters free
}

// d / k for the CPML stretch k, rounded exactly as the IEEE division.  For
// floats the quotient is formed in 64 bits from the reciprocal of k, held
// once per launch: d (1/k) in 64 bits is within 2^-52 of the quotient, and a
// quotient of two 24-bit numbers is never closer than 2^-49 to the midpoint
// of two neighbouring floats, so rounding it to 32 bits gives the quotient's
// own rounding (zeros, infinities and NaN included).  Three instructions
// instead of the eleven dependent ones of a 32-bit division.
template <typename T> struct Stretch;
template <> struct Stretch<float> {
  using Held = double;
  __host__ __device__ static __forceinline__ double hold(float k) { return 1.0 / (double)k; }
  __host__ __device__ static __forceinline__ float apply(float d, double r) {
    return (float)((double)d * r);
  }
};
template <> struct Stretch<double> {
  using Held = double;
  __host__ __device__ static __forceinline__ double hold(double k) { return k; }
  __host__ __device__ static __forceinline__ double apply(double d, double k) { return d / k; }
};

// CPML profiles of one axis at a column (per lane) or a row.
template <typename T> struct Prof {
  T a, b;
  double k;  // Stretch<T>::hold
  __device__ __forceinline__ T over(T d) const { return Stretch<T>::apply(d, k); }
};

// Entry i of an axis of n points; `first` is kA (whole points) or kAh (half
// points), the first of three consecutive profiles a, b, k.
template <typename T>
__device__ __forceinline__ Prof<T> prof_at(const T *prof, int n, int i, int first) {
  const T *const p = as_global(prof) + first * n + i;
  return {p[0], p[n], Stretch<T>::hold(p[2 * n])};
}

// The y profiles of a wavefront's rows, one row per lane; read back with
// cross-lane reads, which need every lane active (see LaneRows).
template <typename T> struct RowProfs {
  Prof<T> e, h;  // of the E phase (whole points) and the H phase (half points)
  __device__ __forceinline__ void load(const Geom<T> &g, int y_first, int lane) {
    const int y = min(max(y_first + lane, 0), g.ny - 1);
    e = prof_at<T>(g.py, g.ny, y, kA);
    h = prof_at<T>(g.py, g.ny, y, kAh);
  }
  // Entry of row r when `on` (uniform).
  static __device__ __forceinline__ Prof<T> at(const Prof<T> &p, int r, bool on) {
    Prof<T> q = {(T)0, (T)0, 1.0};
    if (on) q = {lane_read(p.a, r), lane_read(p.b, r), lane_read(p.k, r)};
    return q;
  }
};

// Sources and receivers of a wavefront's rows.  The entries of a (row, shot,
// tile) segment are sorted by lane, so each lane's are a run that starts at
// its kPointFirst and ends at its kPointLast entry.  Surveys put their points
// on one row: the first row of the wavefront that has any keeps each lane's
// first entry in registers and that entry's amplitudes of all steps of the
// launch in LDS, so a step waits for no global load there; other rows walk
// their segment.
template <typename T, int R> struct TilePoints {
  int mask;        // rows that have points
  int fast;        // row whose first entries are held (-1: no points at all)
  int first;       // this lane's first entry in that row (-1: none)
  int2 en;

  __device__ __forceinline__ void segment(const Points &pts, int y, int n_shots, int s, int xt,
                                          int &b, int &e) const {
    const int64_t si = ((int64_t)as_global(pts.row_slot)[y] * n_shots + s) * pts.n_xt + xt;
    b = as_global(pts.seg)[si];
    e = as_global(pts.seg)[si + 1];
  }
  __device__ __forceinline__ void load(const Points &pts, const TilePlace &c, int ny, int n_shots,
                                       int s, int *entries) {
    mask = 0;
    fast = -1;
    first = -1;
    en = make_int2(0, 0);
#pragma unroll
    for (int r = R - 1; r >= 0; --r) {
      const int y = c.y + r;
      if (y < 0 || y >= ny || as_global(pts.row_slot)[y] < 0) continue;
      int b, e;
      segment(pts, y, n_shots, s, c.xt, b, e);
      if (b >= e) continue;
      mask |= 1 << r;
      fast = r;
    }
    if (fast < 0) return;  // uniform over the wavefront
    int b, e1;
    segment(pts, c.y + fast, n_shots, s, c.xt, b, e1);
    int *const mine = entries + c.w * 3 * 64;
    mine[c.lane] = -1;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int e = b + c.lane; e < e1; e += 64) {
      const int2 q = as_global(pts.ent)[e];
      if (q.x & kPointFirst) {
        mine[q.x & 63] = e;
        mine[64 + (q.x & 63)] = q.x;
        mine[128 + (q.x & 63)] = q.y;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    first = mine[c.lane];
    if (first < 0) return;
    en = make_int2(mine[64 + c.lane], mine[128 + c.lane]);
  }
  // Keeps the amplitudes of this lane's first entry, when it is of kind
  // `kind` (0 source, 1 receiver), in LDS: v holds those of the first step, the
  // next step's are `stride` on.
  __device__ __forceinline__ void amplitudes(T *amp, const TilePlace &c, int steps, int kind,
                                             const T *v, int64_t stride) const {
    if (first < 0 || v == nullptr || ((en.x >> 8) & 1) != kind) return;
    amp += c.w * steps * 64;
    for (int j = 0; j < steps; ++j) amp[j * 64] = as_global(v)[j * stride + en.y];
  }
  // Calls row(r, v) for each row with points, v this lane's value of the row
  // (one copy of the code for all rows).
  template <typename F> __device__ __forceinline__ void each(T (&v)[R], F row) const {
    for (int m = mask; m != 0; m &= m - 1) {  // uniform
      const int r = __builtin_ctz(m);
      T x = v[0];
#pragma unroll
      for (int k = 1; k < R; ++k) x = r == k ? v[k] : x;
      row(r, x);
#pragma unroll
      for (int k = 0; k < R; ++k) v[k] = r == k ? x : v[k];
    }
  }
  // Forward: sources (halo copies too; `amp` the held amplitude), then
  // receivers (owned cells only: lanes `own`, rows of the bits `own_rows`).
  __device__ __forceinline__ void forward(const Points &pts, const TilePlace &c, int n_shots, int s,
                                          const T *amp, const T *f, T *rec, bool own,
                                          int own_rows, T (&ey)[R]) const {
    each(ey, [&](int r, T &v) {
      const bool mine = own && (own_rows >> r & 1);
      auto one = [&](int2 q, bool held) {
        if (((q.x >> 8) & 1) == 0) {
          if (f != nullptr) v += held ? *amp : as_global(f)[q.y];
        } else if (mine && (q.x & kPointCopy) == 0 && rec != nullptr) {
          as_global(rec)[q.y] = v;
        }
      };
      if (r == fast) {
        if (first >= 0) {
          one(en, true);
          int2 q = en;
          for (int e = first; (q.x & kPointLast) == 0;) {
            q = as_global(pts.ent)[++e];
            one(q, false);
          }
        }
        return;
      }
      int b, e;
      segment(pts, c.y + r, n_shots, s, c.xt, b, e);
      for (; b < e; ++b) {
        const int2 q = as_global(pts.ent)[b];
        if ((q.x & 63) == c.lane) one(q, false);
      }
    });
  }
  // Adjoint: receivers inject (halo copies too), then sources (owned
  // cells only) read.
  __device__ __forceinline__ void adjoint(const Points &pts, const TilePlace &c, int n_shots, int s,
                                          const T *amp, const T *gr, T *gf, bool own,
                                          int own_rows, T (&ley)[R]) const {
    each(ley, [&](int r, T &v) {
      const bool mine = own && (own_rows >> r & 1) && gf != nullptr;
      auto add = [&](int2 q, bool held) {
        if (((q.x >> 8) & 1) == 1 && gr != nullptr) v += held ? *amp : as_global(gr)[q.y];
      };
      auto read = [&](int2 q) {
        if (mine && ((q.x >> 8) & 1) == 0 && (q.x & kPointCopy) == 0) as_global(gf)[q.y] = v;
      };
      if (r == fast) {
        if (first >= 0) {
          add(en, true);
          int2 q = en;
          for (int e = first; (q.x & kPointLast) == 0;) {
            q = as_global(pts.ent)[++e];
            add(q, false);
          }
          read(en);
          q = en;
          for (int e = first; (q.x & kPointLast) == 0;) {
            q = as_global(pts.ent)[++e];
            read(q);
          }
        }
        return;
      }
      int b, e;
      segment(pts, c.y + r, n_shots, s, c.xt, b, e);
      for (int k = b; k < e; ++k) {
        const int2 q = as_global(pts.ent)[k];
        if ((q.x & 63) == c.lane) add(q, false);
      }
      for (int k = b; k < e; ++k) {
        const int2 q = as_global(pts.ent)[k];
        if ((q.x & 63) == c.lane) read(q);
      }
    });
  }
};

// Loads R rows of one plane at clamped rows and columns: a cell outside the
// grid gets a copy of an edge cell, which no cell of the update domain reads.
template <typename T, int R>
__device__ __forceinline__ void load_rows(T (&v)[R], const T *__restrict__ p, const uint32_t (&at)[R]) {
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = *elem32(p, at[r]);
}

template <typename T, int R>
__device__ __forceinline__ void tile_offsets(const Geom<T> &g, const TilePlace &c, uint32_t (&at)[R]) {
  const int xc = min(max(c.x, 0), g.nx - 1);
#pragma unroll
  for (int r = 0; r < R; ++r) at[r] = (uint32_t)(min(max(c.y + r, 0), g.ny - 1) * g.nx + xc);
}

// ----------------------------------------------------------------- forward
// What a forward tile holds beside its fields: lane masks, profiles and the
// coefficients of its cells.
template <typename T, int P, int R, bool EDGE> struct TileCells {
  bool own;                       // this lane's column is owned and inside the grid
  bool e_col, hz_col;             // in the update domain of Ey and Hx, of Hz
  bool pml_xe, pml_xh, any_x;     // in an x strip; some lane of the wavefront is
  RowBits rows;
  uint32_t at[R];
  Prof<T> px, pxh;
  RowProfs<T> yp;
  T rdy, rdx;
  T ca[R], cb[R], cq[R];

  __device__ __forceinline__ void set(const Geom<T> &g, const TilePlace &c, int halo) {
    const int nx = g.nx, x = c.x, x0 = c.x - c.lane;
    own = c.lane >= halo && c.lane < 64 - halo && x < nx;
    e_col = !EDGE || (x >= P && x < nx - P + 1);
    hz_col = !EDGE || (x >= P && x < nx - P);
    pml_xe = EDGE && (x < g.pml_x0 || x >= g.pml_x1);
    pml_xh = EDGE && (x < g.pml_x0 || x >= g.pml_x1h);
    any_x = EDGE && (x0 < g.pml_x0 || x0 + 63 >= g.pml_x1h);
    rows.set<T, P, R>(g, c, halo);
    tile_offsets<T, R>(g, c, at);
    rdy = g.rdy;
    rdx = g.rdx;
  }
  __device__ __forceinline__ void profiles(const Geom<T> &g, const TilePlace &c) {
    px = pxh = {(T)0, (T)0, 1.0};
    if constexpr (EDGE) {
      if (any_x) {
        const int xc = min(max(c.x, 0), g.nx - 1);
        px = prof_at<T>(g.px, g.nx, xc, kA);
        pxh = prof_at<T>(g.px, g.nx, xc, kAh);
      }
      yp.load(g, c.y, c.lane);
    }
  }
};

// The fields of a forward tile and the phases of one step, each followed by a
// barrier: hz() publishes Ey and updates Hz, hx() updates Hx, publishes it and
// differences Hz, curl() leaves curl H in `d`.
template <typename T, int P, int R, bool EDGE> struct TileFields {
  T ey[R], hx[R], hz[R];
  T mex[R], mez[R], mhxz[R], mhzx[R];
  T d[R];
  using Cells = TileCells<T, P, R, EDGE>;

  __device__ __forceinline__ void load(const Cells &k, const T *const *in, int64_t base) {
    load_rows<T, R>(ey, as_global(in[0]) + base, k.at);
    load_rows<T, R>(hx, as_global(in[1]) + base, k.at);
    load_rows<T, R>(hz, as_global(in[2]) + base, k.at);
  }
  __device__ __forceinline__ void load_memories(const Cells &k, const T *const *in, int64_t base) {
    if constexpr (EDGE) {
#pragma unroll
      for (int r = 0; r < R; ++r) mex[r] = mez[r] = mhxz[r] = mhzx[r] = (T)0;
      if (k.any_x) {
        load_rows<T, R>(mex, as_global(in[3]) + base, k.at);
        load_rows<T, R>(mhzx, as_global(in[6]) + base, k.at);
      }
      if ((k.rows.pe | k.rows.ph) != 0) {
        load_rows<T, R>(mez, as_global(in[4]) + base, k.at);
        load_rows<T, R>(mhxz, as_global(in[5]) + base, k.at);
      }
    }
  }
  __device__ __forceinline__ void update_hz(const Cells &k, const RowBits &b) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T e[2 * P + 1];
      lane_window<T, P>(ey[r], e);
      T v = d_half<T, P>([&](int o) { return e[P + o]; }, k.rdx);
      if (k.hz_col && (!EDGE || (b.e >> r & 1))) {
        if (k.pml_xh) {
          const T m = k.pxh.b * mex[r] + k.pxh.a * v;
          mex[r] = m;
          v = k.pxh.over(v) + m;
        }
        hz[r] = hz[r] + k.cq[r] * v;
      }
    }
  }
  __device__ __forceinline__ void update_hx(const Cells &k, const RowBits &b,
                                            const TileRows<T, P> &lds, const TilePlace &c) {
    T e[R + 2 * P - 1];
    get_a<T, P, R>(lds, c, ey, e);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool pyh = EDGE && (b.ph >> r & 1);
      Prof<T> py = {(T)0, (T)0, 1.0};  // read with every lane active
      if constexpr (EDGE) py = RowProfs<T>::at(k.yp.h, r, pyh);
      T v = d_half<T, P>([&](int o) { return e[P - 1 + r + o]; }, k.rdy);
      if (k.e_col && (!EDGE || (b.h >> r & 1))) {
        if (pyh) {
          const T m = py.b * mez[r] + py.a * v;
          mez[r] = m;
          v = py.over(v) + m;
        }
        hx[r] = hx[r] - k.cq[r] * v;
      }
    }
  }
  __device__ __forceinline__ void difference_hz(const Cells &k) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      T h[2 * P + 1];
      lane_window<T, P>(hz[r], h);
      d[r] = d_int<T, P>([&](int o) { return h[P + o]; }, k.rdx);
    }
  }
  __device__ __forceinline__ void curl(const Cells &k, const RowBits &b, const TileRows<T, P> &lds,
                                       const TilePlace &c) {
    T h[R + 2 * P - 1];
    get_b<T, P, R>(lds, c, hx, h);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool pye = EDGE && (b.pe >> r & 1);
      Prof<T> py = {(T)0, (T)0, 1.0};  // read with every lane active
      if constexpr (EDGE) py = RowProfs<T>::at(k.yp.e, r, pye);
      T v = d_int<T, P>([&](int o) { return h[P + r + o]; }, k.rdy);
      if (k.e_col && (!EDGE || (b.e >> r & 1))) {
        if (k.pml_xe) {
          const T m = k.px.b * mhzx[r] + k.px.a * d[r];
          mhzx[r] = m;
          d[r] = k.px.over(d[r]) + m;
        }
        if (pye) {
          const T m = py.b * mhxz[r] + py.a * v;
          mhxz[r] = m;
          v = py.over(v) + m;
        }
      }
      d[r] = d[r] - v;
    }
  }
  // Snapshots of the owned cells of the update domain: Ey before the update
  // and curl H (either buffer may be absent).
  template <int FMT>
  __device__ __forceinline__ void snapshot(const Cells &k, const RowBits &b, void *ey_buf,
                                           void *curl_buf, int64_t base) const {
    const int put_rows = EDGE ? b.own & b.e : b.own;
    auto put = [&](char *buf, const T (&v)[R]) {
      if (buf == nullptr) return;  // uniform
      void *const plane = buf + base * (FMT == 2 ? 2 : (int64_t)sizeof(T));
      if (!(k.own && k.e_col)) return;
      if (put_rows == (1 << R) - 1) {
#pragma unroll
        for (int r = 0; r < R; ++r) put_store32<T, FMT>(plane, k.at[r], v[r]);
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (put_rows >> r & 1) put_store32<T, FMT>(plane, k.at[r], v[r]);
      }
    };
    put(as_global((char *)ey_buf), ey);
    put(as_global((char *)curl_buf), d);
  }
  __device__ __forceinline__ void update_ey(const Cells &k, const RowBits &b) {
#pragma unroll
    for (int r = 0; r < R; ++r)
      if (k.e_col && (!EDGE || (b.e >> r & 1))) ey[r] = k.ca[r] * ey[r] + k.cb[r] * d[r];
  }
  __device__ __forceinline__ void store(const Cells &k, T *const *out, int64_t base) const {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      if (!(k.rows.own >> r & 1) || !k.own) continue;
      const uint32_t o = k.at[r];
      *elem32(as_global(out[0]) + base, o) = ey[r];
      *elem32(as_global(out[1]) + base, o) = hx[r];
      *elem32(as_global(out[2]) + base, o) = hz[r];
      if constexpr (EDGE) {
        if (k.pml_xh) *elem32(as_global(out[3]) + base, o) = mex[r];
        if (k.rows.ph >> r & 1) *elem32(as_global(out[4]) + base, o) = mez[r];
        if (k.rows.pe >> r & 1) *elem32(as_global(out[5]) + base, o) = mhxz[r];
        if (k.pml_xe) *elem32(as_global(out[6]) + base, o) = mhzx[r];
      }
    }
  }
};

template <typename T, int P, int R, int FMT, bool EDGE>
__device__ __forceinline__ void tile_forward(ArgRef<TileFwdArgs<T>> args, const TilePlace &c, int s,
                                             const TileRows<T, P> &lds) {
  using Args = TileFwdArgs<T>;
  constexpr int HS = 2 * P - 1;  // rim cells that go stale per step
  const Args &a = args();
  const Geom<T> &g = a.g;
  const int steps = a.steps, halo = a.halo;
  const int64_t base = (int64_t)s * g.numel;
  TileCells<T, P, R, EDGE> k;
  TileFields<T, P, R, EDGE> u;
  k.set(g, c, halo);
  u.load(k, a.in, base);
  load_rows<T, R>(k.cq, as_global(a.cq) + (g.cq_b ? base : 0), k.at);
  load_rows<T, R>(k.ca, as_global(a.ca) + (g.ca_b ? base : 0), k.at);
  load_rows<T, R>(k.cb, as_global(a.cb) + (g.cb_b ? base : 0), k.at);
  k.profiles(g, c);
  u.load_memories(k, a.in, base);
  TilePoints<T, R> points;
  points.load(a.pts, c, g.ny, a.n_shots, s, lds.entries);
  points.amplitudes(lds.amp, c, steps, 0, a.f, a.f_stride);
  wait_loads();

  for (int j = 0; j < steps; ++j) {
    // rows whose new values are still needed; the rest of the tile is stale
    const int lo = halo - (steps - 1 - j) * HS, hi = c.rows - lo;
    const bool active = c.row0 < hi + P - 1 && c.row0 + R > lo - P;  // uniform
    const RowBits b = k.rows.again();
    put_a<T, P, R>(lds, c, u.ey);
    if (active) u.update_hz(k, b);
    __syncthreads();
    if (active) u.update_hx(k, b, lds, c);
    put_b<T, P, R>(lds, c, u.hx);
    if (active) u.difference_hz(k);
    __syncthreads();
    if (active) {
      u.curl(k, b, lds, c);
      if constexpr (FMT != 0) {
        if (b.own != 0) {  // uniform
          const Args &q = args();
          u.template snapshot<FMT>(k, b, q.ey_store[j], q.curl_store[j], base);
        }
      }
      u.update_ey(k, b);
      if (points.fast >= 0) {  // uniform
        const Args &q = args();
        const T *const f = q.f != nullptr ? q.f + j * q.f_stride : nullptr;
        T *const rec = q.r != nullptr ? q.r + j * q.r_stride : nullptr;
        points.forward(q.pts, c, q.n_shots, s, lds.amp_at(c, steps, j), f, rec, k.own, b.own, u.ey);
      }
    }
  }
  const Args &z = args();
  u.store(k, z.out, base);
}

// Workgroup `flat` of a problem.
template <typename T, int P, int R, int FMT>
__device__ __forceinline__ void tile_fwd_group(ArgRef<TileFwdArgs<T>> args, int flat) {
  extern __shared__ double tile_lds[];
  const TileFwdArgs<T> &a = args();
  const TileRows<T, P> lds(tile_lds, (int)blockDim.y, a.steps, (int)threadIdx.x);
  const int tile = flat / a.n_shots, s = flat - tile * a.n_shots;
  const TilePlace c = tile_place<T, P, R>(a.g, a.order, a.pts.n_xt, tile, a.halo, a.own_rows);
  if (c.edge)  // uniform over the workgroup
    tile_forward<T, P, R, FMT, true>(args, c, s, lds);
  else
    tile_forward<T, P, R, FMT, false>(args, c, s, lds);
}

template <typename T, int P, int R, int W, int FMT>
__global__ __launch_bounds__(64 * W) void tile_fwd(TileFwdArgs<T>) {
  tile_fwd_group<T, P, R, FMT>(kernel_args<TileFwdArgs<T>>(),
                               dealt_index((int)blockIdx.x, (int)gridDim.x));
}

// Several problems in one launch: workgroup b of the launch belongs to problem
// tile_item[b], whose arguments for this launch are table[tile_item[b]].
template <typename T, int P, int R, int W, int FMT>
__global__ __launch_bounds__(64 * W) void tile_fwd_items(const TileFwdArgs<T> *__restrict__ table,
                                                         const int32_t *__restrict__ tile_item) {
  const int flat = dealt_index((int)blockIdx.x, (int)gridDim.x);
  const ArgRef<TileFwdArgs<T>> args{(typename ArgRef<TileFwdArgs<T>>::P)(table + tile_item[flat])};
  tile_fwd_group<T, P, R, FMT>(args, flat - args().tile0);
}

// ------------------------------------------------------------ Born forward
// The background and the Born-scattered field of a tile together: the
// scattered Ey update adds dca Ey^n + dcb curl H^n of the background (its values
// before this step's update, still in registers).
template <typename T> struct TileBornArgs {
  Geom<T> g;
  Points pts;
  const T *ca, *cb, *cq, *dca, *dcb;  // dca, dcb null: no scattering term
  const T *in[14];                    // the background's seven arrays, then the scattered field's
  T *out[14];
  const T *f0, *df;                   // source terms of the first step
  T *bg_r, *r;                        // receiver rows of the first step
  int64_t f_stride, r_stride;
  void *hist[4];  // Ey^n, curl^n of the background, of the scattered field; first
  int64_t hist_stride;  // step's planes, the next step's hist_stride bytes on
  int32_t n_shots, steps, halo, own_rows;
  TileOrder order;
};

template <typename T, int P, int R, bool STORE, bool EDGE>
__device__ __forceinline__ void tile_born_step(ArgRef<TileBornArgs<T>> args, const TilePlace &c, int s,
                                               const TileRows<T, P> &lds,
                                               const TileRows<T, P> &lds2) {
  using Args = TileBornArgs<T>;
  constexpr int HS = 2 * P - 1;
  const Args &a = args();
  const Geom<T> &g = a.g;
  const int steps = a.steps, halo = a.halo;
  const int64_t base = (int64_t)s * g.numel;
  TileCells<T, P, R, EDGE> k;
  TileFields<T, P, R, EDGE> u, v;  // background, scattered
  T da[R], db[R];
  k.set(g, c, halo);
  u.load(k, a.in, base);
  v.load(k, a.in + 7, base);
  load_rows<T, R>(k.cq, as_global(a.cq) + (g.cq_b ? base : 0), k.at);
  load_rows<T, R>(k.ca, as_global(a.ca) + (g.ca_b ? base : 0), k.at);
  load_rows<T, R>(k.cb, as_global(a.cb) + (g.cb_b ? base : 0), k.at);
  const bool scatter = a.dca != nullptr;
  if (scatter) {
    load_rows<T, R>(da, as_global(a.dca) + (g.ca_b ? base : 0), k.at);
    load_rows<T, R>(db, as_global(a.dcb) + (g.cb_b ? base : 0), k.at);
  }
  k.profiles(g, c);
  u.load_memories(k, a.in, base);
  v.load_memories(k, a.in + 7, base);
  TilePoints<T, R> points;
  points.load(a.pts, c, g.ny, a.n_shots, s, lds.entries);
  points.amplitudes(lds.amp, c, steps, 0, a.f0, a.f_stride);
  points.amplitudes(lds2.amp, c, steps, 0, a.df, a.f_stride);
  wait_loads();

  for (int j = 0; j < steps; ++j) {
    const int lo = halo - (steps - 1 - j) * HS, hi = c.rows - lo;
    const bool active = c.row0 < hi + P - 1 && c.row0 + R > lo - P;  // uniform
    const RowBits b = k.rows.again();
    put_a<T, P, R>(lds, c, u.ey);
    put_a<T, P, R>(lds2, c, v.ey);
    if (active) {
      u.update_hz(k, b);
      v.update_hz(k, b);
    }
    __syncthreads();
    if (active) {
      u.update_hx(k, b, lds, c);
      v.update_hx(k, b, lds2, c);
    }
    put_b<T, P, R>(lds, c, u.hx);
    put_b<T, P, R>(lds2, c, v.hx);
    if (active) {
      u.difference_hz(k);
      v.difference_hz(k);
    }
    __syncthreads();
    if (active) {
      u.curl(k, b, lds, c);
      v.curl(k, b, lds2, c);
      if constexpr (STORE) {
        if (b.own != 0) {  // uniform
          const Args &q = args();
          const int64_t at = j * q.hist_stride;
          u.template snapshot<1>(k, b, (char *)q.hist[0] + at, (char *)q.hist[1] + at, base);
          v.template snapshot<1>(k, b, (char *)q.hist[2] + at, (char *)q.hist[3] + at, base);
        }
      }
      v.update_ey(k, b);
      if (scatter) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (k.e_col && (!EDGE || (b.e >> r & 1)))
            v.ey[r] = v.ey[r] + (da[r] * u.ey[r] + db[r] * u.d[r]);
      }
      u.update_ey(k, b);
      if (points.fast >= 0) {  // uniform
        const Args &q = args();
        const int64_t fo = j * q.f_stride, ro = j * q.r_stride;
        points.forward(q.pts, c, q.n_shots, s, lds.amp_at(c, steps, j),
                       q.f0 != nullptr ? q.f0 + fo : nullptr,
                       q.bg_r != nullptr ? q.bg_r + ro : nullptr, k.own, b.own, u.ey);
        points.forward(q.pts, c, q.n_shots, s, lds2.amp_at(c, steps, j),
                       q.df != nullptr ? q.df + fo : nullptr,
                       q.r != nullptr ? q.r + ro : nullptr, k.own, b.own, v.ey);
      }
    }
  }
  const Args &z = args();
  u.store(k, z.out, base);
  v.store(k, z.out + 7, base);
}

template <typename T, int P, int R, int W, bool STORE>
__global__ __launch_bounds__(64 * W) void tile_born(TileBornArgs<T>) {
  const ArgRef<TileBornArgs<T>> args = kernel_args<TileBornArgs<T>>();
  const TileBornArgs<T> &a = args();
  extern __shared__ double tile_lds[];
  const int waves = (int)blockDim.y;
  const TileRows<T, P> lds(tile_lds, waves, a.steps, (int)threadIdx.x);
  const TileRows<T, P> lds2((char *)tile_lds + TileRows<T, P>::bytes(waves, a.steps), waves, a.steps,
                            (int)threadIdx.x);
  const int flat = dealt_index((int)blockIdx.x, (int)gridDim.x);
  const int tile = flat / a.n_shots, s = flat - tile * a.n_shots;
  const TilePlace c = tile_place<T, P, R>(a.g, a.order, a.pts.n_xt, tile, a.halo, a.own_rows);
  if (c.edge)  // uniform over the workgroup
    tile_born_step<T, P, R, STORE, true>(args, c, s, lds, lds2);
  else
    tile_born_step<T, P, R, STORE, false>(args, c, s, lds, lds2);
}

// ----------------------------------------------------------------- adjoint
// The transposes of the E step and of the H half-step, each with its CPML
// memories; dHx/dz carries the negated term, so that its differences swap
// their operands instead of negating (bit-identical).
template <typename T, int P, int R, int FMT, bool EDGE>
__device__ __forceinline__ void tile_adjoint(ArgRef<TileAdjArgs<T>> args, const TilePlace &c, int s,
                                             const TileRows<T, P> &lds) {
  using Args = TileAdjArgs<T>;
  constexpr int HS = 2 * P - 1;
  const Args &a = args();
  const Geom<T> &g = a.g;
  const T rdy = g.rdy, rdx = g.rdx;
  const int steps = a.steps;
  const int64_t base = (int64_t)s * g.numel;
  const int ny = g.ny, nx = g.nx, x = c.x;
  const int halo = a.halo;
  const bool own = c.lane >= halo && c.lane < 64 - halo && x < nx;
  const bool e_col = !EDGE || (x >= P && x < nx - P + 1);
  const bool hz_col = !EDGE || (x >= P && x < nx - P);
  const bool pml_xe = EDGE && (x < g.pml_x0 || x >= g.pml_x1);
  const bool pml_xh = EDGE && (x < g.pml_x0 || x >= g.pml_x1h);
  const int x0 = x - c.lane;
  const bool any_x = EDGE && (x0 < g.pml_x0 || x0 + 63 >= g.pml_x1h);
  const bool want = FMT != 0 && (a.gca != nullptr || a.gcb != nullptr);

  RowBits rows;
  rows.set<T, P, R>(g, c, halo);
  uint32_t at[R];
  tile_offsets<T, R>(g, c, at);
  Prof<T> px = {(T)0, (T)0, 1.0}, pxh = px;
  RowProfs<T> yp;
  if constexpr (EDGE) {
    if (any_x) {
      const int xc = min(max(x, 0), nx - 1);
      px = prof_at<T>(g.px, g.nx, xc, kA);
      pxh = prof_at<T>(g.px, g.nx, xc, kAh);
    }
    yp.load(g, c.y, c.lane);
  }
  double ga[R], gb[R];
#pragma unroll
  for (int r = 0; r < R; ++r) ga[r] = gb[r] = 0.0;

  T ley[R], lhx[R], lhz[R], ca[R], cb[R], cq[R];
  load_rows<T, R>(ley, as_global(a.in[0]) + base, at);
  load_rows<T, R>(cb, as_global(a.cb) + (g.cb_b ? base : 0), at);
  load_rows<T, R>(lhx, as_global(a.in[1]) + base, at);
  load_rows<T, R>(lhz, as_global(a.in[2]) + base, at);
  load_rows<T, R>(cq, as_global(a.cq) + (g.cq_b ? base : 0), at);
  load_rows<T, R>(ca, as_global(a.ca) + (g.ca_b ? base : 0), at);
  T mx[R], my[R], nxm[R], nz[R];
  if constexpr (EDGE) {
#pragma unroll
    for (int r = 0; r < R; ++r) mx[r] = my[r] = nxm[r] = nz[r] = (T)0;
    if (any_x) {
      load_rows<T, R>(mx, as_global(a.in[3]) + base, at);
      load_rows<T, R>(nxm, as_global(a.in[5]) + base, at);
    }
    if ((rows.pe | rows.ph) != 0) {
      load_rows<T, R>(my, as_global(a.in[4]) + base, at);
      load_rows<T, R>(nz, as_global(a.in[6]) + base, at);
    }
  }
  TilePoints<T, R> points;
  points.load(a.pts, c, g.ny, a.n_shots, s, lds.entries);
  points.amplitudes(lds.amp, c, steps, 1, a.grad_r, -a.r_stride);
  wait_loads();

  for (int j = 0; j < steps; ++j) {
    const int lo = halo - (steps - 1 - j) * HS, hi = c.rows - lo;
    const bool active = c.row0 < hi + P - 1 && c.row0 + R > lo - P;  // uniform
    const RowBits b = rows.again();
    // this step's snapshots, read well before the gradient needs them
    const Args &a = args();
    const bool have = want && (a.ey_store[j] != nullptr || a.curl_store[j] != nullptr);
    T se[R], sc[R];
    if constexpr (FMT != 0) {
      if (have && b.own != 0) {  // uniform
        // an absent stream reads the other one; its sum is never stored
        const void *const e = a.ey_store[j], *const q = a.curl_store[j];
        const int64_t off = base * (FMT == 2 ? 2 : (int64_t)sizeof(T));
        const char *const pe = as_global((const char *)(e ? e : q)) + off;
        const char *const pq = as_global((const char *)(q ? q : e)) + off;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          se[r] = (T)get_store32<T, FMT>(pe, at[r]);
          sc[r] = (T)get_store32<T, FMT>(pq, at[r]);
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) se[r] = sc[r] = (T)0;
      }
    }
    T nr[R];  // negated adjoint of dHx/dz
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bool pye = EDGE && (b.pe >> r & 1);
      Prof<T> py = {(T)0, (T)0, 1.0};  // read with every lane active
      if constexpr (EDGE) py = RowProfs<T>::at(yp.e, r, pye);
      nr[r] = (T)0;
      if (e_col && (!EDGE || (b.e >> r & 1))) {
        const T q = cb[r] * ley[r];
        nr[r] = q;
        if (pye) {
          const T mn = py.b * my[r] - q;
          my[r] = mn;
          nr[r] = py.over(q) - py.a * mn;
        }
      }
    }
    put_a<T, P, R>(lds, c, nr);
    if (active) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool in = e_col && (!EDGE || (b.e >> r & 1));
        T rx = (T)0;  // adjoint of dHz/dx
        if (in) {
          const T q = cb[r] * ley[r];
          rx = q;
          if (pml_xe) {
            const T mn = px.b * mx[r] + q;
            mx[r] = mn;
            rx = px.a * mn + px.over(q);
          }
        }
        T h[2 * P + 1];
        lane_window<T, P>(rx, h);
        const T d = d_int_adj<T, P>([&](int o) { return h[P + o]; }, rdx);
        if (in) lhz[r] = lhz[r] + d;
      }
    }
    __syncthreads();
    T rz[R];
    if (active) {
      T n[R + 2 * P - 1];
      get_a<T, P, R>(lds, c, nr, n);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool pyh = EDGE && (b.ph >> r & 1);
        Prof<T> py = {(T)0, (T)0, 1.0};  // read with every lane active
        if constexpr (EDGE) py = RowProfs<T>::at(yp.h, r, pyh);
        // n holds the negated terms: the transposed difference of the terms
        // is the plain half-point difference of their negatives
        const T d = d_half<T, P>([&](int o) { return n[P - 1 + r + o]; }, rdy);
        if (e_col && (!EDGE || (b.e >> r & 1))) lhx[r] = lhx[r] + d;
        rz[r] = (T)0;  // adjoint of dEy/dz
        if (e_col && (!EDGE || (b.h >> r & 1))) {
          const T q = -cq[r] * lhx[r];
          rz[r] = q;
          if (pyh) {
            const T mn = py.b * nz[r] + q;
            nz[r] = mn;
            rz[r] = py.a * mn + py.over(q);
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < R; ++r) rz[r] = (T)0;
    }
    put_b<T, P, R>(lds, c, rz);
    T dx[R];
    if (active) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        T rxh = (T)0;  // adjoint of dEy/dx
        if (hz_col && (!EDGE || (b.e >> r & 1))) {
          const T q = cq[r] * lhz[r];
          rxh = q;
          if (pml_xh) {
            const T mn = pxh.b * nxm[r] + q;
            nxm[r] = mn;
            rxh = pxh.a * mn + pxh.over(q);
          }
        }
        T h[2 * P + 1];
        lane_window<T, P>(rxh, h);
        dx[r] = d_half_adj<T, P>([&](int o) { return h[P + o]; }, rdx);
      }
    }
    __syncthreads();
    if (active) {
      T z[R + 2 * P - 1];
      get_b<T, P, R>(lds, c, rz, z);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bool in = e_col && (!EDGE || (b.e >> r & 1));
        const T dz = d_half_adj<T, P>([&](int o) { return z[P + r + o]; }, rdy);
        if (in) ley[r] = ca[r] * ley[r] + (dz + dx[r]);
      }
      if (points.fast >= 0) {  // uniform
        const Args &q = args();
        const T *const gr = q.grad_r != nullptr ? q.grad_r - j * q.r_stride : nullptr;
        T *const gf = q.grad_f != nullptr ? q.grad_f - j * q.f_stride : nullptr;
        points.adjoint(q.pts, c, q.n_shots, s, lds.amp_at(c, steps, j), gr, gf, own, b.own, ley);
      }
      if constexpr (FMT != 0) {
        if (have) {  // uniform; rim cells hold snapshots of 0 or are never added
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const double lm = (double)ley[r];
            ga[r] = fma(lm, (double)se[r], ga[r]);
            gb[r] = fma(lm, (double)sc[r], gb[r]);
          }
        }
      }
    }
  }

  const Args &z = args();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (!(rows.own >> r & 1) || !own) continue;
    const uint32_t o = at[r];
    *elem32(as_global(z.out[0]) + base, o) = ley[r];
    *elem32(as_global(z.out[1]) + base, o) = lhx[r];
    *elem32(as_global(z.out[2]) + base, o) = lhz[r];
    if constexpr (EDGE) {
      if (e_col && (rows.e >> r & 1)) {
        if (pml_xe) *elem32(as_global(z.out[3]) + base, o) = mx[r];
        if (rows.pe >> r & 1) *elem32(as_global(z.out[4]) + base, o) = my[r];
        if (x < nx - P && pml_xh) *elem32(as_global(z.out[5]) + base, o) = nxm[r];
        if (rows.h & rows.ph & (1 << r)) *elem32(as_global(z.out[6]) + base, o) = nz[r];
      }
    }
    if constexpr (FMT != 0) {
      if (want && e_col && (!EDGE || (rows.e >> r & 1))) {
        if (z.gca) *elem32(as_global(z.gca) + base, o) += ga[r] * z.step_scale;
        if (z.gcb) *elem32(as_global(z.gcb) + base, o) += gb[r] * z.step_scale;
      }
    }
  }
}

template <typename T, int P, int R, int FMT>
__device__ __forceinline__ void tile_adj_group(ArgRef<TileAdjArgs<T>> args, int flat) {
  extern __shared__ double tile_lds[];
  const TileAdjArgs<T> &a = args();
  const TileRows<T, P> lds(tile_lds, (int)blockDim.y, a.steps, (int)threadIdx.x);
  const int tile = flat / a.n_shots, s = flat - tile * a.n_shots;
  const TilePlace c = tile_place<T, P, R>(a.g, a.order, a.pts.n_xt, tile, a.halo, a.own_rows);
  if (c.edge)  // uniform over the workgroup
    tile_adjoint<T, P, R, FMT, true>(args, c, s, lds);
  else
    tile_adjoint<T, P, R, FMT, false>(args, c, s, lds);
}

template <typename T, int P, int R, int W, int FMT>
__global__ __launch_bounds__(64 * W) void tile_adj(TileAdjArgs<T>) {
  tile_adj_group<T, P, R, FMT>(kernel_args<TileAdjArgs<T>>(),
                               dealt_index((int)blockIdx.x, (int)gridDim.x));
}

// Several problems in one launch, as tile_fwd_items.
template <typename T, int P, int R, int W, int FMT>
__global__ __launch_bounds__(64 * W) void tile_adj_items(const TileAdjArgs<T> *__restrict__ table,
                                                         const int32_t *__restrict__ tile_item) {
  const int flat = dealt_index((int)blockIdx.x, (int)gridDim.x);
  const ArgRef<TileAdjArgs<T>> args{(typename ArgRef<TileAdjArgs<T>>::P)(table + tile_item[flat])};
  tile_adj_group<T, P, R, FMT>(args, flat - args().tile0);
}

}  // namespace tm2d
}  // namespace tide_hip
