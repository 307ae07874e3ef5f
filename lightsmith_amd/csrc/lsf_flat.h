// The bulk Yee update of engines with a periodic axis: H and E kernels whose lanes take the cells of a plane end to
// end, V = 2 consecutive x cells each, instead of a wavefront per row. Same arithmetic per cell as lsf_step.h (the
// fields are bit-identical); what differs is how cells map to lanes and how ghosts and addresses are formed.
//
// What bounds it: unit cells are narrow (tens of cells) and of any width, so a 64-cell row wavefront leaves a third
// or more of its lanes idle, and every load of the row kernels remaps its three indices through the ghosts and the
// Bloch phases. Here `lpr` = ceil(nx / V) lanes per row are laid end to end and a wavefront takes 64 of them, whatever
// rows they fall in; a neighbour is wrapped once per tile (the row above or below and the cell past a row's end are
// lane offsets fixed over the march) and only the lanes at a face apply a phase. Every address is a wave-uniform
// 64-bit base of the plane plus a fixed 32-bit lane offset: no address arithmetic in the loop. A row's last lane
// starts at nx - V when V does not divide nx: it overlaps its neighbour, computes the shared cells again and stores
// only its own, so every load is in bounds and V wide.
// What is left: waits for memory (57-72 % of the wavefronts' time, 3.4 of them per SIMD for the registers of complex cells),
// the vector units busy for 23-36 % of the cycles; 4.6-4.9 TB/s on one 76 x 61 x 256 complex cell, 5.4 (E) and 6.2 (H) on the
// complex members of 12 as a batch.
// Measured (complex64), row kernels -> these: one 76 x 61 x 256 cell 114 -> 63 us per step, its 3 x 3 column's launches
// included; 12 cells of 50-98 x 50-98 x 256 as one batch 847 -> 520 us per step. One cell per lane: 60 against 55 us on
// the first, 521 against 515 us on the second.
#pragma once

#include "lsf_step.h"

namespace lsf {

// Source corrections of the cells a lane has just stored: V cells from (i, j) of the planes [z0, z1), element e on only
// if e >= sh. The launch this replaces costs 4.5-4.9 us a step whatever its size; here a tile outside the boxes' planes
// pays a compare. It runs after the tile's march, on the lane's own stored values: inside the march it cost the loops
// registers (25 more scalar spills, 5 % of a Bloch cell's step). The row kernels leave their corrections to launches: even
// at their end this slows the E kernel of 4-pole nodes from 143 to 204 us (4 boxes of 96^3). Rows are added in launch
// order, each sum from zero, as the launches add them: the fields are the same bits.
template <class T, int V>
__device__ __forceinline__ void correct(const Corrs& s, const long long* step_at, long long ahead, T* F, const Grid& g,
                                        bool own, int i, int j, int sh, int z0, int z1) {
  z0 = max(z0, s.z[0]);
  z1 = min(z1, s.z[1]);
  if (s.n == 0 || z0 >= z1) return;
  const long long step = *(const long long*)as_global(step_at) + ahead;
  for (int q = 0; q < s.n; ++q) {
    const Corr& o = s.c[q];
    if (!o.gather && (step < 0 || step >= o.table_len)) continue;
    const int n0 = o.n[0], n1 = o.n[1], n2 = o.n[2], dj = j - o.lo[1];
    if (!own || dj < 0 || dj >= n1) continue;
    for (int k = max(z0, o.lo[2]); k < min(z1, o.lo[2] + n2); ++k)
      for (int e = sh; e < V; ++e) {
        const int di = i + e - o.lo[0];
        if (di < 0 || di >= n0) continue;
        for (int c = 0; c < 3; ++c) {
          const int r = ((const int*)as_global(o.row))[((c * n2 + k - o.lo[2]) * n1 + dj) * n0 + di];
          if (r < 0) continue;
          const T* w = (const T*)as_global((const T*)o.w) + (long long)r * o.width;
          T acc = zero<T>();
          if (o.gather) {
            const long long* sidx = (const long long*)as_global(o.sidx) + (long long)r * o.width;
            for (int p = 0; p < o.width; ++p) acc = add(acc, mul(w[p], ((const T*)as_global((const T*)o.src))[sidx[p]]));
          } else {
            const float* tab = (const float*)as_global(o.table) + step * o.width;
            for (int p = 0; p < o.width; ++p) acc = add(acc, scl(tab[p], w[p]));
          }
          T* f = (T*)as_global(F) + (long long)c * g.N + cidx(g, i + e, j, k);
          *f = add(*f, o.scale ? scl(((const float*)as_global(o.scale))[r], acc) : acc);
        }
      }
  }
}

// The step's index where the E kernel may read it: the counter advances while that kernel runs.
__device__ __forceinline__ void note_step(const StepArgs& a, int lt) {
  if (lt == 0 && threadIdx.x == 0 && a.corr.step) *(long long*)as_global(a.corr.step) = *(const long long*)as_global(a.counter);
}

namespace flat {

// V values of the field type from base + a 32-bit byte offset (global memory, 4-byte aligned)
typedef float f1u __attribute__((ext_vector_type(1), aligned(4)));
template <int W> struct Words;
template <> struct Words<1> { typedef float type; };
template <> struct Words<2> { typedef f2u type; };
template <> struct Words<4> { typedef f4u type; };

typedef gptr<const char> cbytes;
typedef gptr<char> bytes;

__device__ __forceinline__ void unpack(float w, float (&o)[1]) { o[0] = w; }
__device__ __forceinline__ void unpack(f2u w, float (&o)[2]) { o[0] = w.x; o[1] = w.y; }
__device__ __forceinline__ void unpack(f2u w, c32 (&o)[1]) { o[0] = mk(w.x, w.y); }
__device__ __forceinline__ void unpack(f4u w, c32 (&o)[2]) { o[0] = mk(w.x, w.y); o[1] = mk(w.z, w.w); }
__device__ __forceinline__ float pack(const float (&o)[1]) { return o[0]; }
__device__ __forceinline__ f2u pack(const float (&o)[2]) { return f2u{o[0], o[1]}; }
__device__ __forceinline__ f2u pack(const c32 (&o)[1]) { return f2u{o[0].x, o[0].y}; }
__device__ __forceinline__ f4u pack(const c32 (&o)[2]) { return f4u{o[0].x, o[0].y, o[1].x, o[1].y}; }

// A wave-uniform base held in scalar registers: without this the loop's addresses are rewritten into per-lane 64-bit
// pointers advanced every plane (two vector registers and an addition for each of some 20 arrays).
template <class P>
__device__ __forceinline__ P uni(P p) {
  unsigned long long u = (unsigned long long)p;
  asm("" : "+s"(u));
  return (P)u;
}

template <class T, int V>
__device__ __forceinline__ void ldv(cbytes b, unsigned off, T (&o)[V]) {
  typedef typename Words<V * (int)sizeof(T) / 4>::type W;
  unpack(*(gptr<const W>)(b + off), o);
}
template <class T, int V>
__device__ __forceinline__ void stv(bytes b, unsigned off, const T (&o)[V]) {
  typedef typename Words<V * (int)sizeof(T) / 4>::type W;
  *(gptr<W>)(b + off) = pack(o);
}
template <class T>
__device__ __forceinline__ T ld1(cbytes b, unsigned off) {
  T o[1];
  ldv<T, 1>(b, off, o);
  return o[0];
}
template <class T>
__device__ __forceinline__ void st1(bytes b, unsigned off, T v) {
  const T o[1] = {v};
  stv<T, 1>(b, off, o);
}

template <class T, int V>
__device__ __forceinline__ void fill0(T (&o)[V]) {
#pragma unroll
  for (int e = 0; e < V; ++e) o[e] = zero<T>();
}

// Where a lane sits: its row, its cells and what it owns of them.
template <int V>
struct Lane {
  int j, i0;          // row, first cell it loads
  int sh;             // cells it loads but does not own (its row neighbour's), at its low end
  bool act;           // owns some cells
  bool first, last;   // holds the row's cell 0 / cell nx - 1 (its last element)
  bool x_next;        // cell i0 + V exists
};

template <int V>
__device__ __forceinline__ Lane<V> lane_of(const StepArgs& a, unsigned w0, int lane) {
  Lane<V> q;
  const unsigned lp = (unsigned)a.lpr * (unsigned)a.g.n[1];
  const unsigned l = min(w0 + (unsigned)lane, lp - 1u);
  q.j = (int)(l / (unsigned)a.lpr);
  const int in = (int)(l - (unsigned)q.j * (unsigned)a.lpr) * V;
  q.i0 = min(in, a.g.n[0] - V);
  q.sh = in - q.i0;
  q.act = w0 + (unsigned)lane < lp && in < a.g.n[0];
  q.first = q.i0 == 0;
  q.last = q.i0 + V == a.g.n[0];
  q.x_next = q.i0 + V < a.g.n[0];
  return q;
}

// Store a lane's values: V wide, or only its own cells in a row's overlapping last lane.
template <class T, int V>
__device__ __forceinline__ void put(bytes b, unsigned off, const T (&o)[V], int sh) {
  if (V == 1 || sh == 0) {
    stv(b, off, o);
  } else {
#pragma unroll
    for (int e = 1; e < V; ++e)
      if (e >= sh) st1(b, off + (unsigned)(e * (int)sizeof(T)), o[e]);
  }
}

// CPML along x: the profile of a lane's cells and their psi index (-1 outside the slab). A slab's psi index need not
// run with the cells, so x psi moves cell by cell; only the slab's own lanes do it.
template <int V>
struct XSlab {
  float4 pr[V];
  int p[V];
  bool any;
};

template <int V>
__device__ __forceinline__ XSlab<V> xslab(const float4* prof, int i0) {
  XSlab<V> s;
  s.any = false;
#pragma unroll
  for (int e = 0; e < V; ++e) {
    s.pr[e] = prof ? ((const float4*)as_global(prof))[i0 + e] : no_pml();
    s.p[e] = (int)s.pr[e].w;
    s.any = s.any || s.p[e] >= 0;
  }
  return s;
}

template <class T, int V>
__device__ __forceinline__ void ld_xpsi(cbytes b, unsigned row, const XSlab<V>& s, T (&o)[V]) {
#pragma unroll
  for (int e = 0; e < V; ++e) o[e] = s.p[e] >= 0 ? ld1<T>(b, (row + (unsigned)s.p[e]) * (unsigned)sizeof(T)) : zero<T>();
}
template <class T, int V>
__device__ __forceinline__ void st_xpsi(bytes b, unsigned row, const XSlab<V>& s, int sh, const T (&o)[V]) {
#pragma unroll
  for (int e = 0; e < V; ++e)
    if (s.p[e] >= 0 && e >= sh) st1<T>(b, (row + (unsigned)s.p[e]) * (unsigned)sizeof(T), o[e]);
}

// acc += the CPML term of one axis, per cell in its slab (pml_apply's arithmetic); keep: psi keeps its old value there
template <class T, int V>
__device__ __forceinline__ void xterm(T (&acc)[V], const XSlab<V>& s, int has_k, float coef, const T (&der)[V],
                                      T (&psi)[V], bool keep0, bool keepl) {
#pragma unroll
  for (int e = 0; e < V; ++e) {
    T pn = psi[e];
    const T v = add(acc[e], pml_apply(s.pr[e], has_k, coef, der[e], pn));
    acc[e] = s.p[e] >= 0 ? v : acc[e];
    const bool keep = (e == 0 && keep0) || (e == V - 1 && keepl);
    psi[e] = keep ? psi[e] : pn;
  }
}
template <class T, int V>
__device__ __forceinline__ void term(T (&acc)[V], const float4 pr, int has_k, float coef, const T (&der)[V],
                                     T (&psi)[V], bool keep0, bool keepl) {
#pragma unroll
  for (int e = 0; e < V; ++e) {
    T pn = psi[e];
    acc[e] = add(acc[e], pml_apply(pr, has_k, coef, der[e], pn));
    const bool keep = (e == 0 && keep0) || (e == V - 1 && keepl);
    psi[e] = keep ? psi[e] : pn;
  }
}

template <class T, int V>
__device__ __forceinline__ void diff(const T (&a)[V], const T (&b)[V], T (&o)[V]) {
#pragma unroll
  for (int e = 0; e < V; ++e) o[e] = sub(a[e], b[e]);
}

template <class T, int V>
__device__ __forceinline__ void rot_if(bool w, c32 ph, T (&o)[V]) {
#pragma unroll
  for (int e = 0; e < V; ++e) o[e] = w ? rot(o[e], ph) : o[e];
}

// the value a lane's lower neighbour reads as its next cell: the first cell the lane owns
template <class T, int V>
__device__ __forceinline__ T own_first(const T (&o)[V], int sh) {
  return sh ? o[V - 1] : o[0];
}

// ---------------------------------------------------------------------------------------------
// H update: lsf_step.h h_tile, V cells per lane
// ---------------------------------------------------------------------------------------------
template <class T, int V, int WAVES>
__device__ __forceinline__ void h_tile(const StepArgs& a, int t) {
  const Grid& g = a.g;
  constexpr unsigned S = sizeof(T);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tz = t / a.tiles_x, tp = t - tz * a.tiles_x;
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const unsigned w0 = (unsigned)(tp * WAVES + wv) * 64u;
  if (w0 >= (unsigned)a.lpr * (unsigned)ny) return;
  const Lane<V> q = lane_of<V>(a, w0, lane);
  const int z0 = tz * a.zc, z1 = min(z0 + a.zc, nz);
  const size_t plane = (size_t)nx * (size_t)ny * S, comp = (size_t)g.N * S;
  const cbytes Eg = (cbytes)as_global((const char*)a.E);
  const bytes Hg = (bytes)as_global((char*)a.H);
  const bool perx = g.per[0], pery = g.per[1], perz = g.per[2];

  const unsigned ol = ((unsigned)q.j * (unsigned)nx + (unsigned)q.i0) * S;
  const bool wy = pery && q.j + 1 == ny - 1;  // the row above is the high ghost: row 1 times the phase
  const int ju = wy ? 1 : min(q.j + 1, ny - 1);
  const unsigned ou = ((unsigned)ju * (unsigned)nx + (unsigned)q.i0) * S;
  const bool halo = lane == 63 && q.x_next;
  // a ghost cell nx - 1 as the next cell is cell 1 times the phase
  const bool gl = perx && q.last, gh = perx && halo && q.i0 + V == nx - 1;
  const unsigned og = ((unsigned)q.j * (unsigned)nx + 1u) * S;
  const unsigned oh = gh ? og : ol + V * S;

  // stepped box: the row's part per lane; cell 0 and cell nx - 1 may be left out (kf, kl)
  const bool yin = q.j < ny - 1 && (!pery || q.j >= 1);
  const bool oky[3] = {q.act && yin, q.act && (pery ? yin : true), q.act && yin};
  const bool kf = perx && q.first;
  const bool kl[3] = {perx && q.last, q.last, q.last};

  const XSlab<V> xs = xslab<V>(a.pml[0].prof, q.i0);
  const bool has_x = __ballot(xs.any) != 0ull;
  const float4 py = a.pml[1].prof ? ((const float4*)as_global(a.pml[1].prof))[q.j] : no_pml();
  const int pyi = (int)py.w;
  const bool has_y = __ballot(pyi >= 0) != 0ull;
  const unsigned oy = ((unsigned)max(pyi, 0) * (unsigned)nx + (unsigned)q.i0) * S;
  const unsigned rx = (unsigned)q.j * (unsigned)a.pml[0].ns;
  const size_t px_plane = (size_t)ny * (size_t)a.pml[0].ns * S, py_plane = (size_t)nx * (size_t)a.pml[1].ns * S;
  const bytes psx1 = (bytes)as_global((char*)a.pml[0].psi[1]), psx2 = (bytes)as_global((char*)a.pml[0].psi[2]);
  const bytes psy0 = (bytes)as_global((char*)a.pml[1].psi[0]), psy2 = (bytes)as_global((char*)a.pml[1].psi[2]);
  const bytes psz0 = (bytes)as_global((char*)a.pml[2].psi[0]), psz1 = (bytes)as_global((char*)a.pml[2].psi[1]);

  T cx[V], cy[V], cz[V];  // E of the row on the current plane
  auto load_row = [&](int k, T (&x)[V], T (&y)[V], T (&z)[V]) {
    const bool wz = perz && k == nz - 1;
    const cbytes b = uni(Eg + (size_t)(wz ? 1 : min(k, nz - 1)) * plane);
    ldv<T, V>(b, ol, x);
    ldv<T, V>(uni(b + comp), ol, y);
    ldv<T, V>(uni(b + 2 * comp), ol, z);
    if (gl) {  // (only y and z components are read as a next cell)
      y[V - 1] = rot(ld1<T>(b + comp, og), g.ph[0]);
      z[V - 1] = rot(ld1<T>(b + 2 * comp, og), g.ph[0]);
    }
    if (wz) {
      rot_if(true, g.ph[2], x);
      rot_if(true, g.ph[2], y);
      rot_if(true, g.ph[2], z);
    }
  };
  load_row(z0, cx, cy, cz);

  for (int k = z0; k < z1; ++k) {
    const float4 pz = a.pml[2].prof ? ld_uniform(a.pml[2].prof, k) : no_pml();
    const int pzi = (int)pz.w;
    const cbytes Ek = uni(Eg + (size_t)k * plane), Ek1 = uni(Ek + comp), Ek2 = uni(Ek + 2 * comp);
    const bytes Hk = uni(Hg + (size_t)k * plane), Hk1 = uni(Hk + comp), Hk2 = uni(Hk + 2 * comp);
    const bytes x1 = uni(psx1 + (size_t)k * px_plane), x2 = uni(psx2 + (size_t)k * px_plane);
    const bytes y0 = uni(psy0 + (size_t)k * py_plane), y2 = uni(psy2 + (size_t)k * py_plane);
    const bytes zz0 = uni(psz0 + (size_t)max(pzi, 0) * plane), zz1 = uni(psz1 + (size_t)max(pzi, 0) * plane);
    // ---- loads
    T nx_[V], ny_[V], nz_[V], ux[V], uz[V], hx[V], hy[V], hz[V];
    load_row(k + 1, nx_, ny_, nz_);
    ldv<T, V>(Ek, ou, ux);
    ldv<T, V>(Ek2, ou, uz);
    ldv<T, V>(Hk, ol, hx);
    ldv<T, V>(Hk1, ol, hy);
    ldv<T, V>(Hk2, ol, hz);
    T hly = zero<T>(), hlz = zero<T>();
    if (halo) {
      hly = ld1<T>(Ek1, oh);
      hlz = ld1<T>(Ek2, oh);
    }
    T qx1[V], qx2[V], qy0[V], qy2[V], qz0[V], qz1[V];
    if (has_x) {
      ld_xpsi<T, V>(x1, rx, xs, qx1);
      ld_xpsi<T, V>(x2, rx, xs, qx2);
    }
    if (has_y) {
      fill0(qy0);
      fill0(qy2);
      if (pyi >= 0) {
        ldv<T, V>(y0, oy, qy0);
        ldv<T, V>(y2, oy, qy2);
      }
    }
    if (pzi >= 0) {
      ldv<T, V>(zz0, ol, qz0);
      ldv<T, V>(zz1, ol, qz1);
    }
    // ---- compute
    rot_if(wy, g.ph[1], ux);
    rot_if(wy, g.ph[1], uz);
    if (gh) {
      hly = rot(hly, g.ph[0]);
      hlz = rot(hlz, g.ph[0]);
    }
    T ynext = shfl_dn(own_first(cy, q.sh)), znext = shfl_dn(own_first(cz, q.sh));
    if (lane == 63) {
      ynext = hly;
      znext = hlz;
    }
    const bool zin = k < nz - 1 && (!perz || k >= 1);
    const bool okz[3] = {zin, zin, perz ? zin : true};
    T da[V], db[V], acc[V];
    auto curl = [&](int d1, int d2) {
#pragma unroll
      for (int e = 0; e < V; ++e) acc[e] = scl(-g.cH, fmad(g.s[d1], da[e], scl(-g.s[d2], db[e])));
    };
    auto finish = [&](int c, T (&h)[V]) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const bool keep = (e == 0 && kf) || (e == V - 1 && kl[c]);
        h[e] = keep ? h[e] : add(h[e], acc[e]);
      }
    };
    // H_x: y difference of E_z, z difference of E_y
    if (okz[0]) {
      diff(uz, cz, da);
      diff(ny_, cy, db);
      curl(1, 2);
      if (has_y && pyi >= 0) term(acc, py, a.pml[1].has_k, -g.cH * g.s[1], da, qy0, kf, kl[0]);
      if (pzi >= 0) term(acc, pz, a.pml[2].has_k, g.cH * g.s[2], db, qz0, kf, kl[0]);
      finish(0, hx);
      if (oky[0]) {
        put<T, V>(Hk, ol, hx, q.sh);
        if (has_y && pyi >= 0) put<T, V>(y0, oy, qy0, q.sh);
        if (pzi >= 0) put<T, V>(zz0, ol, qz0, q.sh);
      }
    }
    // H_y: z difference of E_x, x difference of E_z
    if (okz[1]) {
      diff(nx_, cx, da);
#pragma unroll
      for (int e = 0; e < V; ++e) db[e] = sub(e + 1 < V ? cz[e + 1 < V ? e + 1 : 0] : znext, cz[e]);
      curl(2, 0);
      if (has_x) xterm(acc, xs, a.pml[0].has_k, g.cH * g.s[0], db, qx1, kf, kl[1]);
      if (pzi >= 0) term(acc, pz, a.pml[2].has_k, -g.cH * g.s[2], da, qz1, kf, kl[1]);
      finish(1, hy);
      if (oky[1]) {
        put<T, V>(Hk1, ol, hy, q.sh);
        if (has_x) st_xpsi<T, V>(x1, rx, xs, q.sh, qx1);
        if (pzi >= 0) put<T, V>(zz1, ol, qz1, q.sh);
      }
    }
    // H_z: x difference of E_y, y difference of E_x
    if (okz[2]) {
#pragma unroll
      for (int e = 0; e < V; ++e) da[e] = sub(e + 1 < V ? cy[e + 1 < V ? e + 1 : 0] : ynext, cy[e]);
      diff(ux, cx, db);
      curl(0, 1);
      if (has_x) xterm(acc, xs, a.pml[0].has_k, -g.cH * g.s[0], da, qx2, kf, kl[2]);
      if (has_y && pyi >= 0) term(acc, py, a.pml[1].has_k, g.cH * g.s[1], db, qy2, kf, kl[2]);
      finish(2, hz);
      if (oky[2]) {
        put<T, V>(Hk2, ol, hz, q.sh);
        if (has_x) st_xpsi<T, V>(x2, rx, xs, q.sh, qx2);
        if (has_y && pyi >= 0) put<T, V>(y2, oy, qy2, q.sh);
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      cx[e] = nx_[e];
      cy[e] = ny_[e];
      cz[e] = nz_[e];
    }
  }
  correct<T, V>(a.corr, a.counter, 0, (T*)a.H, g, q.act, q.i0, q.j, q.sh, z0, z1);
}

// ---------------------------------------------------------------------------------------------
// E update: lsf_step.h e_tile without D-form poles, V cells per lane
// ---------------------------------------------------------------------------------------------
template <class T, int MAT, int V, int WAVES>
__device__ __forceinline__ void e_tile(const StepArgs& a, int t, const float* tab) {
  const Grid& g = a.g;
  constexpr unsigned S = sizeof(T);
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tz = t / a.tiles_x, tp = t - tz * a.tiles_x;
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const unsigned w0 = (unsigned)(tp * WAVES + wv) * 64u;
  if (w0 >= (unsigned)a.lpr * (unsigned)ny) return;
  const Lane<V> q = lane_of<V>(a, w0, lane);
  const int z0 = tz * a.zc, z1 = min(z0 + a.zc, nz);
  const size_t plane = (size_t)nx * (size_t)ny * S, comp = (size_t)g.N * S;
  const cbytes Hg = (cbytes)as_global((const char*)a.H);
  const bytes Eg = (bytes)as_global((char*)a.E);
  const bool perx = g.per[0], pery = g.per[1], perz = g.per[2];

  const unsigned oc = (unsigned)q.j * (unsigned)nx + (unsigned)q.i0;  // cell offset in the plane
  const unsigned ol = oc * S;
  const bool wy = pery && q.j - 1 == 0;  // the row below is the low ghost: row ny - 2 times the conjugate phase
  const int jd = wy ? ny - 2 : max(q.j - 1, 0);
  const unsigned od = ((unsigned)jd * (unsigned)nx + (unsigned)q.i0) * S;
  const bool halo = lane == 0 && q.i0 > 0 && q.sh == 0;
  // a ghost cell 0 as the previous cell is cell nx - 2 times the conjugate phase
  const bool gf = perx && q.first, gh = perx && halo && q.i0 == 1;
  const unsigned og = ((unsigned)q.j * (unsigned)nx + (unsigned)(nx - 2)) * S;
  const unsigned oh = gh ? og : ol - S;

  const bool yin = q.j >= 1 && q.j < ny - 1;
  const bool oky[3] = {q.act && yin, q.act && (pery ? yin : q.j < ny - 1), q.act && yin};
  const bool kf[3] = {perx && q.first, q.first, q.first};
  const bool kl = q.last;

  const XSlab<V> xs = xslab<V>(a.pml[0].prof, q.i0);
  const bool has_x = __ballot(xs.any) != 0ull;
  const float4 py = a.pml[1].prof ? ((const float4*)as_global(a.pml[1].prof))[q.j] : no_pml();
  const int pyi = (int)py.w;
  const bool has_y = __ballot(pyi >= 0) != 0ull;
  const unsigned oy = ((unsigned)max(pyi, 0) * (unsigned)nx + (unsigned)q.i0) * S;
  const unsigned rx = (unsigned)q.j * (unsigned)a.pml[0].ns;
  const size_t px_plane = (size_t)ny * (size_t)a.pml[0].ns * S, py_plane = (size_t)nx * (size_t)a.pml[1].ns * S;
  const bytes psx1 = (bytes)as_global((char*)a.pml[0].psi[1]), psx2 = (bytes)as_global((char*)a.pml[0].psi[2]);
  const bytes psy0 = (bytes)as_global((char*)a.pml[1].psi[0]), psy2 = (bytes)as_global((char*)a.pml[1].psi[2]);
  const bytes psz0 = (bytes)as_global((char*)a.pml[2].psi[0]), psz1 = (bytes)as_global((char*)a.pml[2].psi[1]);

  const cbytes midg = (cbytes)as_global((const char*)a.mid), cbdg = (cbytes)as_global((const char*)a.cbd);
  const size_t plane4 = (size_t)nx * (size_t)ny * 4, comp4 = (size_t)g.N * 4;

  T px[V], py_[V];  // H_x, H_y of the previous plane
  auto plane_of = [&](int k) { return perz && k == 0 ? nz - 2 : k; };
  {
    const int k = z0 - 1;
    if (k >= 0) {
      const cbytes b = Hg + (size_t)plane_of(k) * plane;
      ldv<T, V>(b, ol, px);
      ldv<T, V>(b + comp, ol, py_);
      if (perz && k == 0) {
        rot_if(true, conjg(g.ph[2]), px);
        rot_if(true, conjg(g.ph[2]), py_);
      }
    } else {
      fill0(px);
      fill0(py_);
    }
  }
  for (int k = z0; k < z1; ++k) {
    const float4 pz = a.pml[2].prof ? ld_uniform(a.pml[2].prof, k) : no_pml();
    const int pzi = (int)pz.w;
    const cbytes Hk = uni(Hg + (size_t)plane_of(k) * plane), Hk1 = uni(Hk + comp), Hk2 = uni(Hk + 2 * comp);
    const bytes Ek = uni(Eg + (size_t)k * plane), Ek1 = uni(Ek + comp), Ek2 = uni(Ek + 2 * comp);
    const bytes x1 = uni(psx1 + (size_t)k * px_plane), x2 = uni(psx2 + (size_t)k * px_plane);
    const bytes y0 = uni(psy0 + (size_t)k * py_plane), y2 = uni(psy2 + (size_t)k * py_plane);
    const bytes zz0 = uni(psz0 + (size_t)max(pzi, 0) * plane), zz1 = uni(psz1 + (size_t)max(pzi, 0) * plane);
    // ---- loads
    float cb[MAT == 0 ? 3 : 1][V];
    float ids[V];  // packed ids, moved as words
    if (MAT == 1) ldv<float, V>(uni(midg + (size_t)k * plane4), oc * 4u, ids);
    if (MAT == 0) {
#pragma unroll
      for (int c = 0; c < (MAT == 0 ? 3 : 1); ++c) ldv<float, V>(uni(cbdg + (size_t)c * comp4 + (size_t)k * plane4), oc * 4u, cb[c]);
    }
    T ev[3][V];
#pragma unroll
    for (int c = 0; c < 3; ++c) ldv<T, V>(c == 0 ? Ek : (c == 1 ? Ek1 : Ek2), ol, ev[c]);
    T hx[V], hy[V], hz[V], dx_[V], dz_[V];
    ldv<T, V>(Hk, ol, hx);
    ldv<T, V>(Hk1, ol, hy);
    ldv<T, V>(Hk2, ol, hz);
    ldv<T, V>(Hk, od, dx_);
    ldv<T, V>(Hk2, od, dz_);
    T hly = zero<T>(), hlz = zero<T>();
    if (halo) {
      hly = ld1<T>(Hk1, oh);
      hlz = ld1<T>(Hk2, oh);
    }
    if (gf) {  // (only y and z components are read as a previous cell)
      hy[0] = rot(ld1<T>(Hk1, og), conjg(g.ph[0]));
      hz[0] = rot(ld1<T>(Hk2, og), conjg(g.ph[0]));
    }
    T qx1[V], qx2[V], qy0[V], qy2[V], qz0[V], qz1[V];
    if (has_x) {
      ld_xpsi<T, V>(x1, rx, xs, qx1);
      ld_xpsi<T, V>(x2, rx, xs, qx2);
    }
    if (has_y) {
      fill0(qy0);
      fill0(qy2);
      if (pyi >= 0) {
        ldv<T, V>(y0, oy, qy0);
        ldv<T, V>(y2, oy, qy2);
      }
    }
    if (pzi >= 0) {
      ldv<T, V>(zz0, ol, qz0);
      ldv<T, V>(zz1, ol, qz1);
    }
    // ---- compute
    const bool zin = k >= 1 && k < nz - 1;
    const bool okz[3] = {zin, zin, perz ? zin : k < nz - 1};
    if (perz && k == 0) {
      rot_if(true, conjg(g.ph[2]), hx);
      rot_if(true, conjg(g.ph[2]), hy);
      rot_if(true, conjg(g.ph[2]), hz);
    }
    rot_if(wy, conjg(g.ph[1]), dx_);
    rot_if(wy, conjg(g.ph[1]), dz_);
    if (gh) {
      hly = rot(hly, conjg(g.ph[0]));
      hlz = rot(hlz, conjg(g.ph[0]));
    }
    T yprev = shfl_up(hy[V - 1]), zprev = shfl_up(hz[V - 1]);
    if (lane == 0) {
      yprev = hly;
      zprev = hlz;
    }
    auto coef = [&](int c, int e) -> float {
      if (MAT == 1) return tab[(__float_as_uint(ids[e]) >> (8 * c)) & 255u];
      return cb[MAT == 0 ? c : 0][e];
    };
    T da[V], db[V], acc[V];
    float cbe[V];
    auto curl = [&](int c, int d1, int d2) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        cbe[e] = coef(c, e);
        acc[e] = scl(cbe[e], fmad(g.s[d1], da[e], scl(-g.s[d2], db[e])));
      }
    };
    // a CPML term with the cells' own coefficients
    auto yz = [&](const float4 pr, int has_k, float s, const T (&der)[V], T (&psi)[V], int c) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        T pn = psi[e];
        acc[e] = add(acc[e], pml_apply(pr, has_k, cbe[e] * s, der[e], pn));
        const bool keep = (e == 0 && kf[c]) || (e == V - 1 && kl);
        psi[e] = keep ? psi[e] : pn;
      }
    };
    auto xx = [&](float s, const T (&der)[V], T (&psi)[V], int c) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        T pn = psi[e];
        const T v = add(acc[e], pml_apply(xs.pr[e], a.pml[0].has_k, cbe[e] * s, der[e], pn));
        acc[e] = xs.p[e] >= 0 ? v : acc[e];
        const bool keep = (e == 0 && kf[c]) || (e == V - 1 && kl);
        psi[e] = keep ? psi[e] : pn;
      }
    };
    auto finish = [&](int c) {
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const bool keep = (e == 0 && kf[c]) || (e == V - 1 && kl);
        ev[c][e] = keep ? ev[c][e] : add(ev[c][e], acc[e]);
      }
    };
    // E_x: y difference of H_z, z difference of H_y
    if (okz[0]) {
      diff(hz, dz_, da);
      diff(hy, py_, db);
      curl(0, 1, 2);
      if (has_y && pyi >= 0) yz(py, a.pml[1].has_k, g.s[1], da, qy0, 0);
      if (pzi >= 0) yz(pz, a.pml[2].has_k, -g.s[2], db, qz0, 0);
      finish(0);
      if (oky[0]) {
        put<T, V>(Ek, ol, ev[0], q.sh);
        if (has_y && pyi >= 0) put<T, V>(y0, oy, qy0, q.sh);
        if (pzi >= 0) put<T, V>(zz0, ol, qz0, q.sh);
      }
    }
    // E_y: z difference of H_x, x difference of H_z
    if (okz[1]) {
      diff(hx, px, da);
#pragma unroll
      for (int e = 0; e < V; ++e) db[e] = sub(hz[e], e > 0 ? hz[e > 0 ? e - 1 : 0] : zprev);
      curl(1, 2, 0);
      if (has_x) xx(-g.s[0], db, qx1, 1);
      if (pzi >= 0) yz(pz, a.pml[2].has_k, g.s[2], da, qz1, 1);
      finish(1);
      if (oky[1]) {
        put<T, V>(Ek1, ol, ev[1], q.sh);
        if (has_x) st_xpsi<T, V>(x1, rx, xs, q.sh, qx1);
        if (pzi >= 0) put<T, V>(zz1, ol, qz1, q.sh);
      }
    }
    // E_z: x difference of H_y, y difference of H_x
    if (okz[2]) {
#pragma unroll
      for (int e = 0; e < V; ++e) da[e] = sub(hy[e], e > 0 ? hy[e > 0 ? e - 1 : 0] : yprev);
      diff(hx, dx_, db);
      curl(2, 0, 1);
      if (has_x) xx(g.s[0], da, qx2, 2);
      if (has_y && pyi >= 0) yz(py, a.pml[1].has_k, -g.s[1], db, qy2, 2);
      finish(2);
      if (oky[2]) {
        put<T, V>(Ek2, ol, ev[2], q.sh);
        if (has_x) st_xpsi<T, V>(x2, rx, xs, q.sh, qx2);
        if (has_y && pyi >= 0) put<T, V>(y2, oy, qy2, q.sh);
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      px[e] = hx[e];
      py_[e] = hy[e];
    }
  }
  correct<T, V>(a.corr, a.corr.step, 0, (T*)a.E, g, q.act, q.i0, q.j, q.sh, z0, z1);
}

}  // namespace flat

template <class T, int V, int WAVES, bool LOOP>
__global__ void __launch_bounds__(64 * WAVES) k_flat_h(const StepArgs* __restrict__ args, Sched sc) {
  for (int b = blockIdx.x; b < sc.n_pad; b += gridDim.x) {
    const int t = tile_of(b, sc);
    if (t < sc.n_tiles) {
      int m, lt;
      member_of(sc, t, m, lt);
      note_step(args[m], lt);
      flat::h_tile<T, V, WAVES>(args[m], lt);
    }
    if (!LOOP) break;
  }
}

// Each member's tile 0 advances its step counter: counter[1] = n, counter[0] = n + 1 (engine.py:678).
template <class T, int MAT, int V, int WAVES, bool LOOP>
__global__ void __launch_bounds__(64 * WAVES) k_flat_e(const StepArgs* __restrict__ args, Sched sc) {
  __shared__ float tab[MAT == 1 ? 256 : 1];
  int cur = -1;
  for (int b = blockIdx.x; b < sc.n_pad; b += gridDim.x) {
    const int t = tile_of(b, sc);
    if (t >= sc.n_tiles) {
      if (!LOOP) break;
      continue;
    }
    int m, lt;
    member_of(sc, t, m, lt);
    const StepArgs& a = args[m];
    tick_counter(a, lt);
    if (MAT == 1 && m != cur) {
      load_tables<MAT, WAVES, 0>(a, cur >= 0, tab, nullptr);
      cur = m;
    }
    flat::e_tile<T, MAT, V, WAVES>(a, lt, tab);
    if (!LOOP) break;
  }
}

}  // namespace lsf
