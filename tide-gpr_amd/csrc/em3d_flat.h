// Step kernels of the 3-D propagator: forward H and E updates and their
// transposes.
//
// They are bound by memory: a step reads and writes whole volumes (forward
// fp32: H phase 10, E phase 11 values per cell, the adjoint 10 and 11, plus
// 6 snapshot values and two FP64 gradient sums).  A wavefront therefore takes
// kChunk consecutive cells of the volume, across row and plane ends, 16
// bytes per lane: no lane is left over whatever the row length, every access
// of the cell itself is full cache lines, and about ten 1 KB loads are in
// flight per wavefront.  The neighbours one row or plane away are the same
// kind of load at another offset and come from the L2, the x-neighbour is the
// next element of the same vector.  Cells at the faces, and CPML strips, are
// masks per cell.  The vectors need element alignment only.
//
// Against tiles of 62 columns by one row marching through 4 to 16 planes, one
// value per lane (fp32, 2 shots, us per launch): 281^3 padded cells, H 475 ->
// 398, E 507 -> 421 (4.2 TB/s of the counted bytes, copies reach 4.6); 217^3
// cells, E with snapshots 482 -> 301, the transposes 304 -> 287 and 588 -> 408;
// 57 x 69 x 78 cells, 17 -> 9, 25 -> 12, 19 -> 14 and 42 -> 24.
#pragma once

namespace tide_hip {
namespace em3d {

template <typename T> constexpr int kVec = 16 / (int)sizeof(T);
template <typename T> constexpr int kChunk = 64 * kVec<T>;
template <typename T> using Vec = T __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));

// The kernel's arguments, read where they are used: a reference to the
// by-value parameter would be loaded whole at kernel start and spill.
template <typename A> __device__ __forceinline__ const A &flat_args() {
  uint64_t p = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  using C = const __attribute__((address_space(4))) A;
  return *(const A *)(C *)p;
}
// A pointer read that way is not known to be global memory.
template <typename T> __device__ __forceinline__ T *as_global(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)p;
}

// The cells of one wavefront.
template <typename T> struct Chunk {
  static constexpr int V = kVec<T>;
  int lane, group, shot, index;  // index: chunk of the volume
  int wave0, numel;              // first cell (uniform), cells of a volume
  int64_t base;                  // first cell of the shot's volume
  int x[V], y[V], z[V];
  int dom;                       // bit k: cell k is updated

  __device__ __forceinline__ Chunk(const Args3<T> &a) {
    const Geom3<T> &g = a.g;
    const int G = (int)blockDim.y;
    const uint32_t n_chunks = (uint32_t)a.n_chunks;
    const uint32_t n_groups = ((uint32_t)a.n_shots + G - 1) / G;
    const uint32_t flat = (uint32_t)xcd_remap((int64_t)blockIdx.x, (int64_t)n_chunks * n_groups);
    uint32_t c = flat, q = 0;
    if (n_groups > 1) {
      if (a.shot_fast) {
        c = flat / n_groups;
        q = flat - c * n_groups;
      } else {
        q = flat / n_chunks;
        c = flat - q * n_chunks;
      }
    }
    lane = (int)threadIdx.x;
    group = (int)q;
    // threadIdx.y is one value per wavefront: made explicit so the shot's
    // volume pointers stay scalar
    shot = group * G + __builtin_amdgcn_readfirstlane((int)threadIdx.y);
    index = (int)c;
    wave0 = (int)c * kChunk<T>;
    numel = g.numel;
    base = (int64_t)shot * numel;
    const uint32_t i = (uint32_t)wave0 + (uint32_t)(lane * V);
    const uint32_t plane = (uint32_t)(g.ny * g.nx);
    const uint32_t zz = __umulhi(i, g.mul_plane) >> g.shift_plane;
    const uint32_t in_plane = i - zz * plane;
    const uint32_t yy = __umulhi(in_plane, g.mul_row) >> g.shift_row;
    int xk = (int)(in_plane - yy * (uint32_t)g.nx), yk = (int)yy, zk = (int)zz;
    dom = 0;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      x[k] = xk;
      y[k] = yk;
      z[k] = zk;
      if (xk >= 1 && yk >= 1 && zk >= 1 && zk < g.nz) dom |= 1 << k;
      if (++xk == g.nx) {
        xk = 0;
        if (++yk == g.ny) {
          yk = 0;
          ++zk;
        }
      }
    }
    const int left = numel - wave0 - lane * V;  // cells of the volume here
    if (left < V) dom &= (1 << max(left, 0)) - 1;
  }
  // All cells, shifted by `lo` .. `hi`, lie in the volume (uniform).
  __device__ __forceinline__ bool inside(int lo, int hi) const {
    return wave0 + lo >= 0 && hi <= numel - wave0 - kChunk<T>;
  }
};

// Loads of a chunk at an offset; p points at the shot's volume.  FAST: the
// chunk at that offset is inside the volume; else indices are clamped to it.
template <typename T, bool FAST> struct Ld {
  static constexpr int V = kVec<T>;
  const Chunk<T> &c;
  __device__ __forceinline__ void operator()(const T *p, int off, T (&out)[V]) const {
    if constexpr (FAST) {
      const T *const q = as_global(p) + (c.wave0 + off);
      const Vec<T> v = *reinterpret_cast<const Vec<T> *>(elem32(q, (uint32_t)(c.lane * V)));
#pragma unroll
      for (int k = 0; k < V; ++k) out[k] = v[k];
    } else {
#pragma unroll
      for (int k = 0; k < V; ++k) out[k] = one(p, off + k);
    }
  }
  __device__ __forceinline__ T one(const T *p, int off) const {
    if constexpr (FAST) return *elem32(as_global(p) + (c.wave0 + off), (uint32_t)(c.lane * V));
    // 64 bits: cells past the end of the largest volumes
    const int64_t i = (int64_t)c.wave0 + c.lane * V + off;
    return as_global(p)[min(max(i, (int64_t)0), (int64_t)c.numel - 1)];
  }
  // The elements one further on (step +1) or back (-1) of the vector `v` at
  // offset 0 of p.
  __device__ __forceinline__ void next(const T *p, const T (&v)[V], T (&out)[V]) const {
#pragma unroll
    for (int k = 0; k + 1 < V; ++k) out[k] = v[k + 1];
    out[V - 1] = one(p, V);
  }
  __device__ __forceinline__ void prev(const T *p, const T (&v)[V], T (&out)[V]) const {
    out[0] = one(p, -1);
#pragma unroll
    for (int k = 1; k < V; ++k) out[k] = v[k - 1];
  }
};

// Stores a chunk (its cells past the end of the volume excepted).
template <typename T, typename U = T>
__device__ __forceinline__ void put(const Chunk<T> &c, U *p, const U (&v)[kVec<T>]) {
  constexpr int V = kVec<T>;
  using W = U __attribute__((ext_vector_type(V), aligned(sizeof(U))));
  U *const q = elem32(as_global(p) + c.wave0, (uint32_t)(c.lane * V));
  if (c.inside(0, 0)) {
    W w;
#pragma unroll
    for (int k = 0; k < V; ++k) w[k] = v[k];
    *reinterpret_cast<W *>(q) = w;
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (c.lane * V + k < c.numel - c.wave0) q[k] = v[k];
  }
}

// Snapshots: written once and read once, much later, so non-temporal; cells
// outside the update domain are left alone.
template <typename T, int FMT>
__device__ __forceinline__ void put_snapshot(const Chunk<T> &c, void *p, const T (&v)[kVec<T>]) {
  constexpr int V = kVec<T>;
  using U = typename std::conditional<FMT == 2, uint16_t, T>::type;
  using W = U __attribute__((ext_vector_type(V), aligned(sizeof(U))));
  U *const q = elem32(as_global((U *)p) + c.base + c.wave0, (uint32_t)(c.lane * V));
  W w;
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if constexpr (FMT == 2) w[k] = f32_to_bf16((float)v[k]);
    else w[k] = v[k];
  }
  if (c.dom == (1 << V) - 1) {
    __builtin_nontemporal_store(w, reinterpret_cast<W *>(q));
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (c.dom >> k & 1) __builtin_nontemporal_store((U)w[k], q + k);
  }
}
template <typename T, int FMT>
__device__ __forceinline__ void get_snapshot(const Chunk<T> &c, const void *p, T (&v)[kVec<T>]) {
  constexpr int V = kVec<T>;
  using U = typename std::conditional<FMT == 2, uint16_t, T>::type;
  using W = U __attribute__((ext_vector_type(V), aligned(sizeof(U))));
  const U *const q = elem32(as_global((const U *)p) + c.base + c.wave0, (uint32_t)(c.lane * V));
  if (c.inside(0, 0)) {
    const W w = __builtin_nontemporal_load(reinterpret_cast<const W *>(q));
#pragma unroll
    for (int k = 0; k < V; ++k) {
      if constexpr (FMT == 2) v[k] = bf16_to_f32(w[k]);
      else v[k] = w[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      v[k] = (T)0;
      if (c.dom >> k & 1) {
        if constexpr (FMT == 2) v[k] = bf16_to_f32(__builtin_nontemporal_load(q + k));
        else v[k] = __builtin_nontemporal_load(q + k);
      }
    }
  }
}

// Profile records of an axis: {a, b, kappa, 0} per coordinate.
template <typename T> struct Prof3 {
  T a, b, k;
  static __device__ __forceinline__ Prof3 at(const T *table, int i) {
    using Q = T __attribute__((ext_vector_type(4)));
    const Q v = *reinterpret_cast<const Q *>(as_global(table) + 4 * (int64_t)i);
    return {v[0], v[1], v[2]};
  }
};

// Cells of the mask `among` whose coordinate lies in a strip [.., lo) or
// [hi, ..).
template <int V>
__device__ __forceinline__ int in_strip(int among, const int (&x)[V], int lo, int hi, int shift = 0) {
  int m = 0;
#pragma unroll
  for (int k = 0; k < V; ++k)
    if (x[k] + shift < lo || x[k] + shift >= hi) m |= 1 << k;
  return m & among;
}
template <int V>
__device__ __forceinline__ int below(int among, const int (&x)[V], int hi) {
  int m = 0;
#pragma unroll
  for (int k = 0; k < V; ++k)
    if (x[k] < hi) m |= 1 << k;
  return m & among;
}

// Two CPML-corrected differences along one axis and their memories.  load()
// is called early, so that its latency is that of the other loads; the cells of
// a lane that are not in the strip keep their memory.
template <typename T, bool FAST> struct StripFwd {
  static constexpr int V = kVec<T>;
  int cells;  // in the strip
  T m1[V], m2[V];
  Prof3<T> p[V];
  __device__ __forceinline__ void load(const Chunk<T> &c, int cells_, const T *prof,
                                       const int (&x)[V], const T *mem1, const T *mem2) {
    cells = cells_;
    if (cells == 0) return;
    const Ld<T, FAST> ld{c};
    ld(mem1 + c.base, 0, m1);
    ld(mem2 + c.base, 0, m2);
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (cells >> k & 1) p[k] = Prof3<T>::at(prof, x[k]);
  }
  __device__ __forceinline__ void apply(const Chunk<T> &c, T *mem1, T *mem2, T (&d1)[V], T (&d2)[V]) {
    if (cells == 0) return;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      if (cells >> k & 1) {
        m1[k] = p[k].b * m1[k] + p[k].a * d1[k];
        m2[k] = p[k].b * m2[k] + p[k].a * d2[k];
        d1[k] = d1[k] / p[k].k + m1[k];
        d2[k] = d2[k] / p[k].k + m2[k];
      }
    }
    put<T>(c, mem1 + c.base, m1);
    put<T>(c, mem2 + c.base, m2);
  }
};

// The transpose: q1, q2 are the adjoints of two CPML-corrected differences at
// these cells, n1, n2 those at the neighbours `off` cells away (coordinate
// x + step); on return those of the raw differences.  own / nb: cells whose
// own / neighbour's coordinate is in a strip.  The cells' next memories go to
// next1, next2.
template <typename T, bool FAST>
__device__ __forceinline__ void strip_adjoint(const Chunk<T> &c, int own, int nb, const T *prof,
                                              const int (&x)[kVec<T>], int step, int off,
                                              const T *mem1, const T *mem2, T *next1, T *next2,
                                              T (&q1)[kVec<T>], T (&q2)[kVec<T>], T (&n1)[kVec<T>],
                                              T (&n2)[kVec<T>]) {
  constexpr int V = kVec<T>;
  if ((own | nb) == 0) return;
  const Ld<T, FAST> ld{c};
  T m1[V], m2[V], e1[V], e2[V];
  ld(mem1 + c.base, 0, m1);
  ld(mem2 + c.base, 0, m2);
  ld(mem1 + c.base, off, e1);
  ld(mem2 + c.base, off, e2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (own >> k & 1) {
      const Prof3<T> p = Prof3<T>::at(prof, x[k]);
      m1[k] = p.b * m1[k] + q1[k];
      m2[k] = p.b * m2[k] + q2[k];
      q1[k] = p.a * m1[k] + q1[k] / p.k;
      q2[k] = p.a * m2[k] + q2[k] / p.k;
    }
    if (nb >> k & 1) {
      const Prof3<T> p = Prof3<T>::at(prof, x[k] + step);
      n1[k] = p.a * (p.b * e1[k] + n1[k]) + n1[k] / p.k;
      n2[k] = p.a * (p.b * e2[k] + n2[k]) + n2[k] / p.k;
    }
  }
  if (own != 0) {
    put<T>(c, next1 + c.base, m1);
    put<T>(c, next2 + c.base, m2);
  }
}

// ------------------------------------------------------------------ points
// The table has one row per chunk; a chunk's entries of one shot are sorted by
// kind (0 source, 1 receiver), then by point.  Sources and receivers outside
// the update domain do nothing.

// Adds amp[entry] to the entries' cells of kind `kind`, in table order.
template <typename T>
__device__ __forceinline__ void add_points3(const Chunk<T> &c, const Points &pts, int b, int e,
                                            int kind, const T *amp, T (&v)[kVec<T>]) {
  constexpr int V = kVec<T>;
  for (; b < e; b += 64) {  // uniform
    const bool on = b + c.lane < e;
    const int2 en = on ? as_global(pts.ent)[b + c.lane] : make_int2(0, 0);
    const bool mine = on && (en.x >> 8) == kind;
    const T a = mine ? as_global(amp)[en.y] : (T)0;
    for (uint64_t m = __ballot(mine); m != 0; m &= m - 1) {
      const int from = __builtin_ctzll(m);
      const int cell = __builtin_amdgcn_readlane(en.x, from) & 0xff;
      const T s = lane_read(a, from);
#pragma unroll
      for (int k = 0; k < V; ++k)
        if (c.lane == cell / V && cell % V == k && (c.dom >> k & 1)) v[k] += s;
    }
  }
}
__device__ __forceinline__ float from_lane(float v, int lane) {
  return __builtin_bit_cast(float,
                            __builtin_amdgcn_ds_bpermute(lane * 4, __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double from_lane(double v, int lane) {
  const long long u = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_ds_bpermute(lane * 4, (int)u);
  const int hi = __builtin_amdgcn_ds_bpermute(lane * 4, (int)(u >> 32));
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
// out[entry] = value of the entry's cell, for the entries of kind `kind`.
template <typename T>
__device__ __forceinline__ void read_points3(const Chunk<T> &c, const Points &pts, int b, int e,
                                             int kind, T *out, const T (&v)[kVec<T>]) {
  constexpr int V = kVec<T>;
  for (; b < e; b += 64) {  // uniform: every lane takes part in the exchange
    const bool on = b + c.lane < e;
    const int2 en = on ? as_global(pts.ent)[b + c.lane] : make_int2(0, 0);
    const int cell = en.x & 0xff;
    const int dom = __builtin_amdgcn_ds_bpermute(cell / V * 4, c.dom);
    T r = (T)0;
#pragma unroll
    for (int k = 0; k < V; ++k) {
      const T w = from_lane(v[k], cell / V);
      r = cell % V == k ? w : r;
    }
    if (on && (en.x >> 8) == kind && (dom >> (cell % V) & 1)) as_global(out)[en.y] = r;
  }
}
// Calls f(v) with the component `comp` (uniform) of a cell's three.
template <typename T, typename F>
__device__ __forceinline__ void with_component(int comp, T (&v0)[kVec<T>], T (&v1)[kVec<T>],
                                               T (&v2)[kVec<T>], F f) {
  constexpr int V = kVec<T>;
  T v[V];
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const T a0 = v0[k], a1 = v1[k], a2 = v2[k];
    v[k] = comp == 0 ? a0 : (comp == 1 ? a1 : a2);
  }
  f(v);
#pragma unroll
  for (int k = 0; k < V; ++k) {  // selects: a choice of arrays would put them in memory
    const T a0 = v0[k], a1 = v1[k], a2 = v2[k];
    v0[k] = comp == 0 ? v[k] : a0;
    v1[k] = comp == 1 ? v[k] : a1;
    v2[k] = comp == 2 ? v[k] : a2;
  }
}

// ----------------------------------------------------------- forward: H
template <typename T, bool FAST>
__device__ __forceinline__ void h3_cells(const Chunk<T> &c) {
  constexpr int V = kVec<T>;
  const Args3<T> &a = flat_args<Args3<T>>();
  const Geom3<T> &g = a.g;
  const Ld<T, FAST> ld{c};
  const int nx = g.nx, plane = g.ny * g.nx;
  T *const *f = a.f;
  const int64_t base = c.base;
  const int has_x = below<V>(c.dom, c.x, nx - 1);
  T ex[V], ey[V], ez[V], ex_y[V], ez_y[V], ex_z[V], ey_z[V], ey_x[V], ez_x[V];
  T cq[V], hx[V], hy[V], hz[V];
  ld(f[EX] + base, 0, ex);
  ld(f[EY] + base, 0, ey);
  ld(f[EZ] + base, 0, ez);
  ld(f[EX] + base, nx, ex_y);
  ld(f[EZ] + base, nx, ez_y);
  ld(f[EX] + base, plane, ex_z);
  ld(f[EY] + base, plane, ey_z);
  ld.next(f[EY] + base, ey, ey_x);
  ld.next(f[EZ] + base, ez, ez_x);
  ld(a.cq + (g.cq_b ? base : 0), 0, cq);
  ld(f[HX] + base, 0, hx);
  ld(f[HY] + base, 0, hy);
  ld(f[HZ] + base, 0, hz);
  StripFwd<T, FAST> sx;
  sx.load(c, in_strip<V>(has_x, c.x, g.x0, g.x1h), g.qx + 4 * nx, c.x, f[M_EZ_X], f[M_EY_X]);

  const Args3<T> &q = flat_args<Args3<T>>();
  const Geom3<T> &h = q.g;
  T d1[V], d2[V];
  T u0[V], u1[V], u2[V];  // curl, first terms
  // d/dx: Ez into Hy, Ey into Hz
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const bool on = has_x >> k & 1;
    d1[k] = on ? (ez_x[k] - ez[k]) * h.rdx : (T)0;
    d2[k] = on ? (ey_x[k] - ey[k]) * h.rdx : (T)0;
  }
  sx.apply(c, q.f[M_EZ_X], q.f[M_EY_X], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    u1[k] = d1[k];
    u2[k] = d2[k];
  }
  // d/dz: Ey into Hx, Ex into Hy
  const int has_z = below<V>(c.dom, c.z, h.nz - 1);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const bool on = has_z >> k & 1;
    d1[k] = on ? (ey_z[k] - ey[k]) * h.rdz : (T)0;
    d2[k] = on ? (ex_z[k] - ex[k]) * h.rdz : (T)0;
  }
  StripFwd<T, FAST> s;
  s.load(c, in_strip<V>(has_z, c.z, h.z0, h.z1h), h.qz + 4 * h.nz, c.z, q.f[M_EY_Z], q.f[M_EX_Z]);
  s.apply(c, q.f[M_EY_Z], q.f[M_EX_Z], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    u0[k] = d1[k];
    u1[k] = u1[k] - d2[k];
  }
  // d/dy: Ez into Hx, Ex into Hz
  const int has_y = below<V>(c.dom, c.y, h.ny - 1);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    const bool on = has_y >> k & 1;
    d1[k] = on ? (ez_y[k] - ez[k]) * h.rdy : (T)0;
    d2[k] = on ? (ex_y[k] - ex[k]) * h.rdy : (T)0;
  }
  s.load(c, in_strip<V>(has_y, c.y, h.y0, h.y1h), h.qy + 4 * h.ny, c.y, q.f[M_EZ_Y], q.f[M_EX_Y]);
  s.apply(c, q.f[M_EZ_Y], q.f[M_EX_Y], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (c.dom >> k & 1) {
      hx[k] = hx[k] - cq[k] * (u0[k] - d1[k]);
      hy[k] = hy[k] - cq[k] * u1[k];
      hz[k] = hz[k] - cq[k] * (d2[k] - u2[k]);
    }
  }
  put<T>(c, q.f[HX] + base, hx);
  put<T>(c, q.f[HY] + base, hy);
  put<T>(c, q.f[HZ] + base, hz);
}

template <typename T>
__global__ __launch_bounds__(512) void h3_flat(Args3<T>) {
  const Args3<T> &a = flat_args<Args3<T>>();
  const Chunk<T> c(a);
  if (c.shot >= a.n_shots) return;
  if (c.inside(0, max(a.g.ny * a.g.nx, kVec<T>))) h3_cells<T, true>(c);
  else h3_cells<T, false>(c);
}

// ----------------------------------------------------------- forward: E
// BORN: the scattered field of the Born forward, updated as
// ca E + cb curl + dca E_bg + dcb curl_bg in that order (reference
// maxwell_3d_inst.cpp:1444-1456).
template <typename T, int FMT, bool BORN, bool FAST>
__device__ __forceinline__ void e3_cells(const Chunk<T> &c) {
  constexpr int V = kVec<T>;
  const Args3<T> &a = flat_args<Args3<T>>();
  const Geom3<T> &g = a.g;
  const Ld<T, FAST> ld{c};
  const int nx = g.nx, plane = g.ny * g.nx;
  T *const *f = a.f;
  const int64_t base = c.base;
  T hx[V], hy[V], hz[V], hx_z[V], hy_z[V], hx_y[V], hz_y[V], hy_x[V], hz_x[V];
  T ca[V], cb[V], e0[V], e1[V], e2[V];
  ld(f[HX] + base, 0, hx);
  ld(f[HY] + base, 0, hy);
  ld(f[HZ] + base, 0, hz);
  ld(f[HX] + base, -nx, hx_y);
  ld(f[HZ] + base, -nx, hz_y);
  ld(f[HX] + base, -plane, hx_z);
  ld(f[HY] + base, -plane, hy_z);
  ld.prev(f[HY] + base, hy, hy_x);
  ld.prev(f[HZ] + base, hz, hz_x);
  ld(a.ca + (g.ca_b ? base : 0), 0, ca);
  ld(a.cb + (g.cb_b ? base : 0), 0, cb);
  ld(f[EX] + base, 0, e0);
  ld(f[EY] + base, 0, e1);
  ld(f[EZ] + base, 0, e2);
  StripFwd<T, FAST> sx;
  sx.load(c, in_strip<V>(c.dom, c.x, g.x0, g.x1), g.qx, c.x, f[M_HZ_X], f[M_HY_X]);

  const Args3<T> &q = flat_args<Args3<T>>();
  const Geom3<T> &h = q.g;
  T d1[V], d2[V];
  T u0[V], u1[V], u2[V];
  // d/dx: Hz into Ey, Hy into Ez
#pragma unroll
  for (int k = 0; k < V; ++k) {
    d1[k] = (hz[k] - hz_x[k]) * h.rdx;
    d2[k] = (hy[k] - hy_x[k]) * h.rdx;
  }
  sx.apply(c, q.f[M_HZ_X], q.f[M_HY_X], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    u1[k] = d1[k];
    u2[k] = d2[k];
  }
  // d/dz: Hy into Ex, Hx into Ey
#pragma unroll
  for (int k = 0; k < V; ++k) {
    d1[k] = (hy[k] - hy_z[k]) * h.rdz;
    d2[k] = (hx[k] - hx_z[k]) * h.rdz;
  }
  StripFwd<T, FAST> s;
  s.load(c, in_strip<V>(c.dom, c.z, h.z0, h.z1), h.qz, c.z, q.f[M_HY_Z], q.f[M_HX_Z]);
  s.apply(c, q.f[M_HY_Z], q.f[M_HX_Z], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    u0[k] = d1[k];
    u1[k] = u1[k] - d2[k];
  }
  // d/dy: Hz into Ex, Hx into Ez
#pragma unroll
  for (int k = 0; k < V; ++k) {
    d1[k] = (hz[k] - hz_y[k]) * h.rdy;
    d2[k] = (hx[k] - hx_y[k]) * h.rdy;
  }
  s.load(c, in_strip<V>(c.dom, c.y, h.y0, h.y1), h.qy, c.y, q.f[M_HZ_Y], q.f[M_HX_Y]);
  s.apply(c, q.f[M_HZ_Y], q.f[M_HX_Y], d1, d2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    u0[k] = u0[k] - d1[k];
    u2[k] = d2[k] - u2[k];
  }
  if constexpr (FMT != 0) {
    if (q.st[0] != nullptr) {
      put_snapshot<T, FMT>(c, q.st[0], e0);
      put_snapshot<T, FMT>(c, q.st[1], e1);
      put_snapshot<T, FMT>(c, q.st[2], e2);
    }
    if (q.st[3] != nullptr) {
      put_snapshot<T, FMT>(c, q.st[3], u0);
      put_snapshot<T, FMT>(c, q.st[4], u1);
      put_snapshot<T, FMT>(c, q.st[5], u2);
    }
  }
  if constexpr (BORN) {
    const Ld<T, FAST> ld2{c};
    T da[V], db[V], b0[V], b1[V], b2[V], r0[V], r1[V], r2[V];
    ld2(q.dca, 0, da);
    ld2(q.dcb, 0, db);
    ld2(q.bg[0] + base, 0, b0);
    ld2(q.bg[1] + base, 0, b1);
    ld2(q.bg[2] + base, 0, b2);
    ld2(q.bg[3] + base, 0, r0);
    ld2(q.bg[4] + base, 0, r1);
    ld2(q.bg[5] + base, 0, r2);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      if (c.dom >> k & 1) {
        e0[k] = ca[k] * e0[k] + cb[k] * u0[k] + da[k] * b0[k] + db[k] * r0[k];
        e1[k] = ca[k] * e1[k] + cb[k] * u1[k] + da[k] * b1[k] + db[k] * r1[k];
        e2[k] = ca[k] * e2[k] + cb[k] * u2[k] + da[k] * b2[k] + db[k] * r2[k];
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k) {
      if (c.dom >> k & 1) {
        e0[k] = ca[k] * e0[k] + cb[k] * u0[k];
        e1[k] = ca[k] * e1[k] + cb[k] * u1[k];
        e2[k] = ca[k] * e2[k] + cb[k] * u2[k];
      }
    }
  }
  // Sources of this shot, then receivers.
  const int slot = as_global(q.pts.row_slot)[c.index];
  if (slot >= 0) {  // uniform
    const int64_t si = (int64_t)slot * q.n_shots + c.shot;
    const int b = as_global(q.pts.seg)[si], e = as_global(q.pts.seg)[si + 1];
    if (q.src_amp != nullptr)
      with_component<T>(q.src_comp, e0, e1, e2,
                        [&](T (&v)[V]) { add_points3<T>(c, q.pts, b, e, 0, q.src_amp, v); });
    if (q.rec_out != nullptr)
      with_component<T>(q.rec_comp, e0, e1, e2,
                        [&](T (&v)[V]) { read_points3<T>(c, q.pts, b, e, 1, q.rec_out, v); });
  }
  put<T>(c, q.f[EX] + base, e0);
  put<T>(c, q.f[EY] + base, e1);
  put<T>(c, q.f[EZ] + base, e2);
}

template <typename T, int FMT, bool BORN = false>
__global__ __launch_bounds__(512) void e3_flat(Args3<T>) {
  const Args3<T> &a = flat_args<Args3<T>>();
  const Chunk<T> c(a);
  if (c.shot >= a.n_shots) return;
  if (c.inside(-(a.g.ny * a.g.nx), 0)) e3_cells<T, FMT, BORN, true>(c);
  else e3_cells<T, FMT, BORN, false>(c);
}

// ------------------------------------------------------------- adjoint
// Transpose of the E update: lambda_H += D^T (raw E-curl adjoints); the
// E-phase adjoint memories advance into a.mn.
template <typename T, bool FAST>
__device__ __forceinline__ void adj_e3_cells(const Chunk<T> &c) {
  constexpr int V = kVec<T>;
  const Args3<T> &a = flat_args<Args3<T>>();
  const Geom3<T> &g = a.g;
  const Ld<T, FAST> ld{c};
  const int nx = g.nx, plane = g.ny * g.nx;
  T *const *f = a.f;
  const int64_t base = c.base;
  const T *const cb = a.cb + (g.cb_b ? base : 0);
  T b[V], l0[V], l1[V], l2[V], bz[V], l0z[V], l1z[V], by[V], l0y[V], l2y[V], bx[V], l1x[V], l2x[V];
  T h0[V], h1[V], h2[V];
  ld(cb, 0, b);
  ld(f[EX] + base, 0, l0);
  ld(f[EY] + base, 0, l1);
  ld(f[EZ] + base, 0, l2);
  ld.next(cb, b, bx);
  ld.next(f[EY] + base, l1, l1x);
  ld.next(f[EZ] + base, l2, l2x);
  ld(cb, plane, bz);
  ld(f[EX] + base, plane, l0z);
  ld(f[EY] + base, plane, l1z);
  ld(cb, nx, by);
  ld(f[EX] + base, nx, l0y);
  ld(f[EZ] + base, nx, l2y);
  ld(f[HX] + base, 0, h0);
  ld(f[HY] + base, 0, h1);
  ld(f[HZ] + base, 0, h2);
  const Args3<T> &q = flat_args<Args3<T>>();
  const Geom3<T> &h = q.g;
  T r1[V], r2[V], n1[V], n2[V];
  // z: dHy/dz of Ex (+) and dHx/dz of Ey (-)
  const int has_z = below<V>(c.dom, c.z, h.nz - 1);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = b[k] * l0[k];
    r2[k] = -(b[k] * l1[k]);
    n1[k] = (has_z >> k & 1) ? bz[k] * l0z[k] : (T)0;
    n2[k] = (has_z >> k & 1) ? -(bz[k] * l1z[k]) : (T)0;
  }
  strip_adjoint<T, FAST>(c, in_strip<V>(c.dom, c.z, h.z0, h.z1),
                         in_strip<V>(has_z, c.z, h.z0, h.z1, 1), h.qz, c.z, 1, plane, q.f[M_HY_Z],
                         q.f[M_HX_Z], q.mn[M_HY_Z], q.mn[M_HX_Z], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (c.dom >> k & 1) {
      h0[k] = h0[k] + (r2[k] - n2[k]) * h.rdz;
      h1[k] = h1[k] + (r1[k] - n1[k]) * h.rdz;
    }
  }
  // y: dHz/dy of Ex (-) and dHx/dy of Ez (+)
  const int has_y = below<V>(c.dom, c.y, h.ny - 1);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = -(b[k] * l0[k]);
    r2[k] = b[k] * l2[k];
    n1[k] = (has_y >> k & 1) ? -(by[k] * l0y[k]) : (T)0;
    n2[k] = (has_y >> k & 1) ? by[k] * l2y[k] : (T)0;
  }
  strip_adjoint<T, FAST>(c, in_strip<V>(c.dom, c.y, h.y0, h.y1),
                         in_strip<V>(has_y, c.y, h.y0, h.y1, 1), h.qy, c.y, 1, nx, q.f[M_HZ_Y],
                         q.f[M_HX_Y], q.mn[M_HZ_Y], q.mn[M_HX_Y], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (c.dom >> k & 1) {
      h0[k] = h0[k] + (r2[k] - n2[k]) * h.rdy;
      h2[k] = h2[k] + (r1[k] - n1[k]) * h.rdy;
    }
  }
  // x: dHz/dx of Ey (+) and dHy/dx of Ez (-)
  const int has_x = below<V>(c.dom, c.x, nx - 1);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = b[k] * l1[k];
    r2[k] = -(b[k] * l2[k]);
    n1[k] = (has_x >> k & 1) ? bx[k] * l1x[k] : (T)0;
    n2[k] = (has_x >> k & 1) ? -(bx[k] * l2x[k]) : (T)0;
  }
  strip_adjoint<T, FAST>(c, in_strip<V>(c.dom, c.x, h.x0, h.x1),
                         in_strip<V>(has_x, c.x, h.x0, h.x1, 1), h.qx, c.x, 1, 1, q.f[M_HZ_X],
                         q.f[M_HY_X], q.mn[M_HZ_X], q.mn[M_HY_X], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    if (c.dom >> k & 1) {
      h1[k] = h1[k] + (r2[k] - n2[k]) * h.rdx;
      h2[k] = h2[k] + (r1[k] - n1[k]) * h.rdx;
    }
  }
  put<T>(c, q.f[HX] + base, h0);
  put<T>(c, q.f[HY] + base, h1);
  put<T>(c, q.f[HZ] + base, h2);
}

template <typename T>
__global__ __launch_bounds__(512) void adj_e3_flat(Args3<T>) {
  const Args3<T> &a = flat_args<Args3<T>>();
  const Chunk<T> c(a);
  if (c.shot >= a.n_shots) return;
  if (c.inside(0, max(a.g.ny * a.g.nx, kVec<T>))) adj_e3_cells<T, true>(c);
  else adj_e3_cells<T, false>(c);
}

// Transpose of the H update: lambda_E = ca lambda_E + D^T (raw H-term
// adjoints); H-phase adjoint memories advance into a.mn; then receivers
// inject grad_r[t], sources read grad_f[t], and this shot's terms of the
// coefficient gradient, against the stored forward state, go to pa and pb.
template <typename T, int FMT, bool FAST>
__device__ __forceinline__ void adj_h3_cells(const Chunk<T> &c, double (&pa)[kVec<T>],
                                             double (&pb)[kVec<T>]) {
  constexpr int V = kVec<T>;
  const Args3<T> &a = flat_args<Args3<T>>();
  const Geom3<T> &g = a.g;
  const Ld<T, FAST> ld{c};
  const int nx = g.nx, plane = g.ny * g.nx;
  T *const *f = a.f;
  const int64_t base = c.base;
  const T *const cq = a.cq + (g.cq_b ? base : 0);
  T w[V], h0[V], h1[V], h2[V], wz[V], h0z[V], h1z[V], wy[V], h0y[V], h2y[V], wx[V], h1x[V], h2x[V];
  T ca[V], e0[V], e1[V], e2[V];
  ld(cq, 0, w);
  ld(f[HX] + base, 0, h0);
  ld(f[HY] + base, 0, h1);
  ld(f[HZ] + base, 0, h2);
  ld.prev(cq, w, wx);
  ld.prev(f[HY] + base, h1, h1x);
  ld.prev(f[HZ] + base, h2, h2x);
  ld(cq, -plane, wz);
  ld(f[HX] + base, -plane, h0z);
  ld(f[HY] + base, -plane, h1z);
  ld(cq, -nx, wy);
  ld(f[HX] + base, -nx, h0y);
  ld(f[HZ] + base, -nx, h2y);
  ld(a.ca + (g.ca_b ? base : 0), 0, ca);
  ld(f[EX] + base, 0, e0);
  ld(f[EY] + base, 0, e1);
  ld(f[EZ] + base, 0, e2);
  const Args3<T> &q = flat_args<Args3<T>>();
  const Geom3<T> &h = q.g;
  const int nz = h.nz, ny = h.ny;
  T r1[V], r2[V], n1[V], n2[V], t0[V], t1[V], t2[V];
  auto keep = [](int cells, T (&v)[V], T (&u)[V]) {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (!(cells >> k & 1)) v[k] = u[k] = (T)0;
  };
  auto from2 = [](int among, const int (&x)[V]) {  // the lower neighbour is updated too
    int m = 0;
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (x[k] >= 2) m |= 1 << k;
    return m & among;
  };
  // z: Hx term dEy/dz (-cq lHx) and Hy term dEx/dz (+cq lHy)
  int own = below<V>(c.dom, c.z, nz - 1), nb = from2(c.dom, c.z);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = -w[k] * h0[k];
    r2[k] = w[k] * h1[k];
    n1[k] = -wz[k] * h0z[k];
    n2[k] = wz[k] * h1z[k];
  }
  keep(own, r1, r2);
  keep(nb, n1, n2);
  strip_adjoint<T, FAST>(c, in_strip<V>(own, c.z, h.z0, h.z1h),
                         in_strip<V>(nb, c.z, h.z0, h.z1h, -1), h.qz + 4 * nz, c.z, -1, -plane,
                         q.f[M_EY_Z], q.f[M_EX_Z], q.mn[M_EY_Z], q.mn[M_EX_Z], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    t0[k] = (n2[k] - r2[k]) * h.rdz;
    t1[k] = (n1[k] - r1[k]) * h.rdz;
  }
  // y: Hx term dEz/dy (+cq lHx) and Hz term dEx/dy (-cq lHz)
  own = below<V>(c.dom, c.y, ny - 1);
  nb = from2(c.dom, c.y);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = w[k] * h0[k];
    r2[k] = -w[k] * h2[k];
    n1[k] = wy[k] * h0y[k];
    n2[k] = -wy[k] * h2y[k];
  }
  keep(own, r1, r2);
  keep(nb, n1, n2);
  strip_adjoint<T, FAST>(c, in_strip<V>(own, c.y, h.y0, h.y1h),
                         in_strip<V>(nb, c.y, h.y0, h.y1h, -1), h.qy + 4 * ny, c.y, -1, -nx,
                         q.f[M_EZ_Y], q.f[M_EX_Y], q.mn[M_EZ_Y], q.mn[M_EX_Y], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    t0[k] = t0[k] + (n2[k] - r2[k]) * h.rdy;
    t2[k] = (n1[k] - r1[k]) * h.rdy;
  }
  // x: Hy term dEz/dx (-cq lHy) and Hz term dEy/dx (+cq lHz)
  own = below<V>(c.dom, c.x, nx - 1);
  nb = from2(c.dom, c.x);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    r1[k] = -w[k] * h1[k];
    r2[k] = w[k] * h2[k];
    n1[k] = -wx[k] * h1x[k];
    n2[k] = wx[k] * h2x[k];
  }
  keep(own, r1, r2);
  keep(nb, n1, n2);
  strip_adjoint<T, FAST>(c, in_strip<V>(own, c.x, h.x0, h.x1h),
                         in_strip<V>(nb, c.x, h.x0, h.x1h, -1), h.qx + 4 * nx, c.x, -1, -1,
                         q.f[M_EZ_X], q.f[M_EY_X], q.mn[M_EZ_X], q.mn[M_EY_X], r1, r2, n1, n2);
#pragma unroll
  for (int k = 0; k < V; ++k) {
    t1[k] = t1[k] + (n2[k] - r2[k]) * h.rdx;
    t2[k] = t2[k] + (n1[k] - r1[k]) * h.rdx;
    if (c.dom >> k & 1) {
      e0[k] = ca[k] * e0[k] + t0[k];
      e1[k] = ca[k] * e1[k] + t1[k];
      e2[k] = ca[k] * e2[k] + t2[k];
    }
  }
  // receivers inject grad_r[t]; sources read grad_f[t]
  const int slot = as_global(q.pts.row_slot)[c.index];
  if (slot >= 0) {  // uniform
    const int64_t si = (int64_t)slot * q.n_shots + c.shot;
    const int b = as_global(q.pts.seg)[si], e = as_global(q.pts.seg)[si + 1];
    if (q.src_amp != nullptr)
      with_component<T>(q.rec_comp, e0, e1, e2,
                        [&](T (&v)[V]) { add_points3<T>(c, q.pts, b, e, 1, q.src_amp, v); });
    if (q.rec_out != nullptr)
      with_component<T>(q.src_comp, e0, e1, e2,
                        [&](T (&v)[V]) { read_points3<T>(c, q.pts, b, e, 0, q.rec_out, v); });
  }
  put<T>(c, q.f[EX] + base, e0);
  put<T>(c, q.f[EY] + base, e1);
  put<T>(c, q.f[EZ] + base, e2);
  if constexpr (FMT != 0) {
    const Args3<T> &y = flat_args<Args3<T>>();
    auto product = [&](void *const *st, double (&p)[V]) {
      T s0[V], s1[V], s2[V];
      get_snapshot<T, FMT>(c, st[0], s0);
      get_snapshot<T, FMT>(c, st[1], s1);
      get_snapshot<T, FMT>(c, st[2], s2);
#pragma unroll
      for (int k = 0; k < V; ++k)
        p[k] = ((double)e0[k] * (double)s0[k] + (double)e1[k] * (double)s1[k] +
                (double)e2[k] * (double)s2[k]) * y.step_scale;
    };
    if (y.gca != nullptr) product(y.st, pa);
    if (y.gcb != nullptr) product(y.st + 3, pb);
  }
}

// acc[cell] += p of the update domain's cells.
template <typename T>
__device__ __forceinline__ void add_gradient(const Chunk<T> &c, double *acc,
                                             const double (&p)[kVec<T>]) {
  constexpr int V = kVec<T>;
  using D = double __attribute__((ext_vector_type(V), aligned(8)));
  double *const q = elem32(as_global(acc) + c.wave0, (uint32_t)(c.lane * V));
  if (c.dom == (1 << V) - 1) {
    D d = *reinterpret_cast<D *>(q);
#pragma unroll
    for (int k = 0; k < V; ++k) d[k] += p[k];
    *reinterpret_cast<D *>(q) = d;
  } else {
#pragma unroll
    for (int k = 0; k < V; ++k)
      if (c.dom >> k & 1) q[k] += p[k];
  }
}

// A workgroup holds the shots of a group, one wavefront each; their gradient
// terms are summed in LDS in shot order.
template <typename T, int FMT>
__global__ __launch_bounds__(512) void adj_h3_flat(Args3<T>) {
  constexpr int V = kVec<T>;
  extern __shared__ double red[];  // [2][G][V][64] when several shots reduce
  const Args3<T> &a = flat_args<Args3<T>>();
  const Chunk<T> c(a);
  const bool active = c.shot < a.n_shots;  // idle wavefronts join the barrier
  double pa[V], pb[V];
#pragma unroll
  for (int k = 0; k < V; ++k) pa[k] = pb[k] = 0.0;
  if (active) {
    if (c.inside(-(a.g.ny * a.g.nx), 0)) adj_h3_cells<T, FMT, true>(c, pa, pb);
    else adj_h3_cells<T, FMT, false>(c, pa, pb);
  }
  if constexpr (FMT != 0) {
    const Args3<T> &q = flat_args<Args3<T>>();
    const int G = (int)blockDim.y;
    const int64_t at = q.per_shot_grad ? c.base : c.group * q.group_stride;
    if (q.per_shot_grad || G == 1) {  // uniform
      if (!active) return;
      if (q.gca != nullptr) add_gradient<T>(c, q.gca + at, pa);
      if (q.gcb != nullptr) add_gradient<T>(c, q.gcb + at, pb);
      return;
    }
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
#pragma unroll
    for (int k = 0; k < V; ++k) {
      red[(w * V + k) * 64 + c.lane] = pa[k];
      red[((G + w) * V + k) * 64 + c.lane] = pb[k];
    }
    __syncthreads();
    for (int pass = w; pass < 2; pass += G) {
      double *const out = pass == 0 ? q.gca : q.gcb;
      if (out == nullptr) continue;
      double sum[V];
#pragma unroll
      for (int k = 0; k < V; ++k) {
        sum[k] = 0.0;
        for (int s = 0; s < G; ++s) sum[k] += red[((pass * G + s) * V + k) * 64 + c.lane];
      }
      add_gradient<T>(c, out + at, sum);
    }
  }
}

}  // namespace em3d
}  // namespace tide_hip
