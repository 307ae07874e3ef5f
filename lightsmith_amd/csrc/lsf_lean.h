// Bulk H and E half-steps of real engines without periodic axes, forward (without D-form poles in the E update) and
// adjoint. Same arithmetic per cell as the row kernels (lsf_step.h, lsf_adjoint.h): the fields are bit-identical.
//
// Mapping. The rows of a plane are laid end to end, one x cell per lane. A wavefront takes 64 lanes and owns 63 of them:
// the last (H) or the first (E) only supplies its value to the x difference of its neighbour, so no cell needs a halo
// load. A lane marches the z planes of its tile with what the z difference needs in registers.
//
// What bounds it. The half-steps move 36 (H) and 40-48 (E) bytes a cell, at 5 TB/s from HBM and up to 7 from the memory-side
// cache; the row kernels reached 4 to 4.9 TB/s on boxes that fit there, held by their instructions (110-160 a cell: 64-bit
// addresses, three index tests a component, a third of the lanes past a row's end on ragged rows) and, in the adjoint
// ones, by a chain of dependent loads in branches. So, as in the single pass (lsf_pass.h): every address is a scalar
// base and a 32-bit lane offset that advances by a plane, cells that do not step keep their value by a select, whole
// wavefronts outside a CPML slab skip its terms and the lanes outside it read a psi that they do not use. What is left are the
// bytes and the waits for them: 5.5 (H) and 6.1 TB/s (E) on a 514 x 96 x 80 box with half of its cells in slabs, 6.35-6.6 on a
// 256 x 192 x 96 one, of the 7.1 that a copy reaches there; the wavefronts wait for memory 48-63 % of their time, the vector
// units are busy for 40-44 % of the cycles (forward, 114-143 instructions a cell) and 59-67 % (adjoint, 210).
// Measured, row -> lean kernels: at flat_kernel (lsf.hip), which picks between them.
#pragma once

#include "lsf_adjoint.h"
#include "lsf_flat.h"

namespace lsf {

constexpr int LEAN_WAVES = 4, LEAN_OWN = 63;

namespace lean {

using flat::bytes;
using flat::cbytes;
using flat::ld1;
using flat::st1;

// A lane offset the compiler does not look into: a load then takes it as the 32-bit offset from a scalar base.
__device__ __forceinline__ unsigned lane_off(unsigned o) {
  asm("" : "+v"(o));
  return o;
}
__device__ __forceinline__ cbytes in_bytes(const void* p) { return (cbytes)as_global((const char*)p); }
__device__ __forceinline__ bytes out_bytes(void* p) { return (bytes)as_global((char*)p); }

// A lane's cell, its tile's planes and the byte offsets of the cell and its y neighbours (clamped to the grid) on plane z0.
struct Cell {
  int lane, i, j;
  bool on, own;
  int z0, z1;
  unsigned o0, o1, o2, plane;
};

// UP: the wavefront's last lane is its neighbour's x + 1; else its first is its neighbour's x - 1.
template <bool UP>
__device__ __forceinline__ Cell cell_of(const StepArgs& a, int t) {
  Cell q;
  const int nx = a.g.n[0], ny = a.g.n[1], total = nx * ny;
  q.lane = threadIdx.x & 63;
  const int tz = t / a.tiles_x, tp = t - tz * a.tiles_x;
  const int l0 = (tp * LEAN_WAVES + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * LEAN_OWN;
  q.on = l0 < total;
  const int lr = l0 + q.lane - (UP ? 0 : 1), l = min(max(lr, 0), total - 1);
  q.j = l / nx;
  q.i = l - q.j * nx;
  q.own = (UP ? q.lane < 63 : q.lane > 0) && lr < total;
  q.z0 = tz * a.zc;
  q.z1 = min(q.z0 + a.zc, a.g.n[2]);
  q.plane = (unsigned)total * 4u;
  const unsigned row = (unsigned)nx * 4u;
  q.o1 = lane_off((unsigned)l * 4u + (unsigned)q.z0 * q.plane);
  q.o0 = lane_off(q.o1 - (q.j > 0 ? row : 0u));
  q.o2 = lane_off(q.o1 + (q.j < ny - 1 ? row : 0u));
  return q;
}

__device__ __forceinline__ float4 prof_at(const PmlAx& p, int at) {
  return p.prof ? ((const float4*)as_global(p.prof))[at] : no_pml();
}
__device__ __forceinline__ bool in_slab(const float4 pr) { return pr.w >= 0.f; }

// The z profile of a plane, from scalar loads near the slabs only.
__device__ __forceinline__ float4 z_prof(const StepArgs& a, const PmlAx& p, int k) {
  return p.prof && (k < a.zlo || k >= a.zhi) ? ld_uniform(p.prof, k) : no_pml();
}

// psi offsets of the cell: x slabs [k][j][p], y slabs [k][p][i], z slabs [p][j][i]; lanes outside a slab take its first entry
__device__ __forceinline__ unsigned x_off(const StepArgs& a, const PmlAx& p, const float4 pr, int k, int j) {
  return lane_off((unsigned)((k * a.g.n[1] + j) * p.ns + max((int)pr.w, 0)) * 4u);
}
__device__ __forceinline__ unsigned y_off(const StepArgs& a, const PmlAx& p, const float4 pr, int k, int i) {
  return lane_off((unsigned)((k * p.ns + max((int)pr.w, 0)) * a.g.n[0] + i) * 4u);
}
__device__ __forceinline__ unsigned z_off(const Cell& q, unsigned o, int k, int p) {
  return lane_off(o + (unsigned)(p - k) * q.plane);
}

// acc + the CPML term of an axis for the lanes in its slab; psi advances there where the cell steps
__device__ __forceinline__ float term(float acc, const float4 pr, int has_k, float coef, float der, bool st, float& psi) {
  float n = psi;
  const float v = acc + pml_apply(pr, has_k, coef, der, n);
  const bool in = in_slab(pr);
  psi = st && in ? n : psi;
  return in ? v : acc;
}

// ---------------------------------------------------------------------------------------------
// H half-step (lsf_step.h h_tile)
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void h_tile(const StepArgs& a, int t) {
  const Grid& g = a.g;
  Cell q = cell_of<true>(a, t);
  if (!q.on) return;
  const int nz = g.n[2];
  const bool xh = q.i < g.n[0] - 1, yh = q.j < g.n[1] - 1;
  const PmlAx *px = &a.pml[0], *py = &a.pml[1], *pz = &a.pml[2];
  const float4 prx = prof_at(*px, q.i), pry = prof_at(*py, q.j);
  const bool has_x = __ballot(in_slab(prx)) != 0ull, has_y = __ballot(in_slab(pry)) != 0ull;
  const size_t comp = (size_t)g.N * 4;
  const cbytes E0 = in_bytes(a.E), E1 = E0 + comp, E2 = E1 + comp;
  const bytes H0 = out_bytes(a.H), H1 = H0 + comp, H2 = H1 + comp;
  const float cH = g.cH;

  float x1 = ld1<float>(E0, q.o1), y1 = ld1<float>(E1, q.o1);
  for (int k = q.z0; k < q.z1; ++k) {
    const unsigned dk = k + 1 < nz ? q.plane : 0u;
    const cbytes U0 = flat::uni(E0 + dk), U1 = flat::uni(E1 + dk);
    const float nx1 = ld1<float>(U0, q.o1), ny1 = ld1<float>(U1, q.o1);
    const float w1 = ld1<float>(E2, q.o1), w2 = ld1<float>(E2, q.o2), x2 = ld1<float>(E0, q.o2);
    float hx = ld1<float>(H0, q.o1), hy = ld1<float>(H1, q.o1), hz = ld1<float>(H2, q.o1);
    float qxy = 0.f, qzy = 0.f, qyx = 0.f, qzx = 0.f, qxz = 0.f, qyz = 0.f;
    unsigned ox = 0u, oy = 0u, oz = 0u;
    if (has_x) {
      ox = x_off(a, *px, prx, k, q.j);
      qyx = ld1<float>(in_bytes(px->psi[1]), ox);
      qzx = ld1<float>(in_bytes(px->psi[2]), ox);
    }
    if (has_y) {
      oy = y_off(a, *py, pry, k, q.i);
      qxy = ld1<float>(in_bytes(py->psi[0]), oy);
      qzy = ld1<float>(in_bytes(py->psi[2]), oy);
    }
    const float4 prz = z_prof(a, *pz, k);
    const int iz = (int)prz.w;
    if (iz >= 0) {
      oz = z_off(q, q.o1, k, iz);
      qxz = ld1<float>(in_bytes(pz->psi[0]), oz);
      qyz = ld1<float>(in_bytes(pz->psi[1]), oz);
    }
    const bool zh = k < nz - 1;
    {  // H_x: y difference of E_z, z difference of E_y
      const bool st = yh && zh;
      const float da = w2 - w1, db = ny1 - y1;
      float acc = scl(-cH, fmad(g.s[1], da, scl(-g.s[2], db)));
      if (has_y) acc = term(acc, pry, py->has_k, -cH * g.s[1], da, st, qxy);
      if (iz >= 0) acc = term(acc, prz, pz->has_k, cH * g.s[2], db, st, qxz);
      hx = st ? hx + acc : hx;
    }
    {  // H_y: z difference of E_x, x difference of E_z
      const bool st = xh && zh;
      const float da = nx1 - x1, db = shfl_dn(w1) - w1;
      float acc = scl(-cH, fmad(g.s[2], da, scl(-g.s[0], db)));
      if (has_x) acc = term(acc, prx, px->has_k, cH * g.s[0], db, st, qyx);
      if (iz >= 0) acc = term(acc, prz, pz->has_k, -cH * g.s[2], da, st, qyz);
      hy = st ? hy + acc : hy;
    }
    {  // H_z: x difference of E_y, y difference of E_x
      const bool st = xh && yh;
      const float da = shfl_dn(y1) - y1, db = x2 - x1;
      float acc = scl(-cH, fmad(g.s[0], da, scl(-g.s[1], db)));
      if (has_x) acc = term(acc, prx, px->has_k, -cH * g.s[0], da, st, qzx);
      if (has_y) acc = term(acc, pry, py->has_k, cH * g.s[1], db, st, qzy);
      hz = st ? hz + acc : hz;
    }
    if (q.own) {
      st1<float>(H0, q.o1, hx);
      st1<float>(H1, q.o1, hy);
      st1<float>(H2, q.o1, hz);
      if (has_x && in_slab(prx)) {
        st1<float>(out_bytes(px->psi[1]), ox, qyx);
        st1<float>(out_bytes(px->psi[2]), ox, qzx);
      }
      if (has_y && in_slab(pry)) {
        st1<float>(out_bytes(py->psi[0]), oy, qxy);
        st1<float>(out_bytes(py->psi[2]), oy, qzy);
      }
      if (iz >= 0) {
        st1<float>(out_bytes(pz->psi[0]), oz, qxz);
        st1<float>(out_bytes(pz->psi[1]), oz, qyz);
      }
    }
    x1 = nx1;
    y1 = ny1;
    q.o1 += q.plane;
    q.o2 += q.plane;
  }
  correct<float, 1>(a.corr, a.counter, 0, (float*)a.H, g, q.own, q.i, q.j, 0, q.z0, q.z1);
}

// The E coefficients of a cell: packed ids (MAT 1, through the block's table) or the three values (MAT 0)
template <int MAT>
struct Coef {
  uint32_t id;
  float v[MAT == 0 ? 3 : 1];
  __device__ __forceinline__ void load(const StepArgs& a, unsigned o) {
    if (MAT == 1) {
      id = __float_as_uint(ld1<float>(in_bytes(a.mid), o));
    } else {
      const cbytes m = in_bytes(a.cbd);
      const size_t comp = (size_t)a.g.N * 4;
#pragma unroll
      for (int c = 0; c < (MAT == 0 ? 3 : 1); ++c) v[c] = ld1<float>(m + (size_t)c * comp, o);
    }
  }
  __device__ __forceinline__ float of(int c, const float* tab) const {
    return MAT == 1 ? tab[(id >> (8 * c)) & 255u] : v[MAT == 0 ? c : 0];
  }
};

// ---------------------------------------------------------------------------------------------
// E half-step (lsf_step.h e_tile without poles)
// ---------------------------------------------------------------------------------------------
template <int MAT>
__device__ __forceinline__ void e_tile(const StepArgs& a, int t, const float* tab) {
  const Grid& g = a.g;
  Cell q = cell_of<false>(a, t);
  if (!q.on) return;
  const int nz = g.n[2];
  const bool xh = q.i < g.n[0] - 1, xe = xh && q.i >= 1, yh = q.j < g.n[1] - 1, ye = yh && q.j >= 1;
  const PmlAx *px = &a.pml[0], *py = &a.pml[1], *pz = &a.pml[2];
  const float4 prx = prof_at(*px, q.i), pry = prof_at(*py, q.j);
  const bool has_x = __ballot(in_slab(prx)) != 0ull, has_y = __ballot(in_slab(pry)) != 0ull;
  const size_t comp = (size_t)g.N * 4;
  const cbytes H0 = in_bytes(a.H), H1 = H0 + comp, H2 = H1 + comp;
  const bytes E0 = out_bytes(a.E), E1 = E0 + comp, E2 = E1 + comp;

  float pxv = 0.f, pyv = 0.f;  // H_x, H_y of the plane below
  if (q.z0 > 0) {
    pxv = ld1<float>(H0, lane_off(q.o1 - q.plane));
    pyv = ld1<float>(H1, lane_off(q.o1 - q.plane));
  }
  for (int k = q.z0; k < q.z1; ++k) {
    Coef<MAT> m;
    m.load(a, q.o1);
    const float hx = ld1<float>(H0, q.o1), hy = ld1<float>(H1, q.o1), hz = ld1<float>(H2, q.o1);
    const float hx0 = ld1<float>(H0, q.o0), hz0 = ld1<float>(H2, q.o0);
    float ex = ld1<float>(E0, q.o1), ey = ld1<float>(E1, q.o1), ez = ld1<float>(E2, q.o1);
    float sxy = 0.f, szy = 0.f, syx = 0.f, szx = 0.f, sxz = 0.f, syz = 0.f;
    unsigned ox = 0u, oy = 0u, oz = 0u;
    if (has_x) {
      ox = x_off(a, *px, prx, k, q.j);
      syx = ld1<float>(in_bytes(px->psi[1]), ox);
      szx = ld1<float>(in_bytes(px->psi[2]), ox);
    }
    if (has_y) {
      oy = y_off(a, *py, pry, k, q.i);
      sxy = ld1<float>(in_bytes(py->psi[0]), oy);
      szy = ld1<float>(in_bytes(py->psi[2]), oy);
    }
    const float4 prz = z_prof(a, *pz, k);
    const int iz = (int)prz.w;
    if (iz >= 0) {
      oz = z_off(q, q.o1, k, iz);
      sxz = ld1<float>(in_bytes(pz->psi[0]), oz);
      syz = ld1<float>(in_bytes(pz->psi[1]), oz);
    }
    auto cb = [&](int c) {
      const float v = m.of(c, tab);
      return v < 0.f ? g.cdx : v;
    };
    const bool zh = k < nz - 1, ze = zh && k >= 1;
    {  // E_x: y difference of H_z, z difference of H_y
      const bool st = xh && ye && ze;
      const float da = hz - hz0, db = hy - pyv, c = cb(0);
      float acc = scl(c, fmad(g.s[1], da, scl(-g.s[2], db)));
      if (has_y) acc = term(acc, pry, py->has_k, c * g.s[1], da, st, sxy);
      if (iz >= 0) acc = term(acc, prz, pz->has_k, -c * g.s[2], db, st, sxz);
      ex = st ? ex + acc : ex;
    }
    {  // E_y: z difference of H_x, x difference of H_z
      const bool st = xe && yh && ze;
      const float da = hx - pxv, db = hz - shfl_up(hz), c = cb(1);
      float acc = scl(c, fmad(g.s[2], da, scl(-g.s[0], db)));
      if (has_x) acc = term(acc, prx, px->has_k, -c * g.s[0], db, st, syx);
      if (iz >= 0) acc = term(acc, prz, pz->has_k, c * g.s[2], da, st, syz);
      ey = st ? ey + acc : ey;
    }
    {  // E_z: x difference of H_y, y difference of H_x
      const bool st = xe && ye && zh;
      const float da = hy - shfl_up(hy), db = hx - hx0, c = cb(2);
      float acc = scl(c, fmad(g.s[0], da, scl(-g.s[1], db)));
      if (has_x) acc = term(acc, prx, px->has_k, c * g.s[0], da, st, szx);
      if (has_y) acc = term(acc, pry, py->has_k, -c * g.s[1], db, st, szy);
      ez = st ? ez + acc : ez;
    }
    if (q.own) {
      st1<float>(E0, q.o1, ex);
      st1<float>(E1, q.o1, ey);
      st1<float>(E2, q.o1, ez);
      if (has_x && in_slab(prx)) {
        st1<float>(out_bytes(px->psi[1]), ox, syx);
        st1<float>(out_bytes(px->psi[2]), ox, szx);
      }
      if (has_y && in_slab(pry)) {
        st1<float>(out_bytes(py->psi[0]), oy, sxy);
        st1<float>(out_bytes(py->psi[2]), oy, szy);
      }
      if (iz >= 0) {
        st1<float>(out_bytes(pz->psi[0]), oz, sxz);
        st1<float>(out_bytes(pz->psi[1]), oz, syz);
      }
    }
    pxv = hx;
    pyv = hy;
    q.o0 += q.plane;
    q.o1 += q.plane;
  }
  correct<float, 1>(a.corr, a.corr.step, 0, (float*)a.E, g, q.own, q.i, q.j, 0, q.z0, q.z1);
}

// ---------------------------------------------------------------------------------------------
// adjoint half-steps (lsf_adjoint.h): the differenced values are (k + c) F + c chi inside a slab, F outside
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ float mix(float f, const float4 pr, int has_k, float chi) {
  const float2 fc = adj_fc(pr, has_k);
  return in_slab(pr) ? fc.x * f + fc.y * chi : f;
}

// chi <- b (F_old + chi) where the cell steps and lies in the slab
__device__ __forceinline__ float advance(float chi, const float4 pr, float old, bool st) {
  return st && in_slab(pr) ? pr.x * (old + chi) : chi;
}

__device__ __forceinline__ void ah_tile(const StepArgs& a, int t) {
  const Grid& g = a.g;
  Cell q = cell_of<true>(a, t);
  if (!q.on) return;
  const int nz = g.n[2];
  const bool xh = q.i < g.n[0] - 1, yh = q.j < g.n[1] - 1;
  const PmlAx *ex_ = &a.xpml[0], *ey_ = &a.xpml[1], *ez_ = &a.xpml[2];  // E side: read
  const PmlAx *hx_ = &a.pml[0], *hy_ = &a.pml[1], *hz_ = &a.pml[2];     // H side: advanced
  const int ju = min(q.j + 1, g.n[1] - 1);
  const float4 pex = prof_at(*ex_, q.i), pey = prof_at(*ey_, q.j), peu = prof_at(*ey_, ju);
  const float4 phx = prof_at(*hx_, q.i), phy = prof_at(*hy_, q.j);
  const bool e_x = __ballot(in_slab(pex)) != 0ull, e_y = __ballot(in_slab(pey) || in_slab(peu)) != 0ull;
  const bool h_x = __ballot(in_slab(phx)) != 0ull, h_y = __ballot(in_slab(phy)) != 0ull;
  const size_t comp = (size_t)g.N * 4;
  const cbytes E0 = in_bytes(a.E), E1 = E0 + comp, E2 = E1 + comp;
  const bytes H0 = out_bytes(a.H), H1 = H0 + comp, H2 = H1 + comp;

  // E_x, E_y of the plane and their values differenced along z, carried from the plane below
  float x1 = ld1<float>(E0, q.o1), y1 = ld1<float>(E1, q.o1);
  float zx = x1, zy = y1;
  {
    const float4 pr = z_prof(a, *ez_, q.z0);
    const int p = (int)pr.w;
    if (p >= 0) {
      const unsigned o = z_off(q, q.o1, q.z0, p);
      zx = mix(x1, pr, ez_->has_k, ld1<float>(in_bytes(ez_->psi[0]), o));
      zy = mix(y1, pr, ez_->has_k, ld1<float>(in_bytes(ez_->psi[1]), o));
    }
  }
  for (int k = q.z0; k < q.z1; ++k) {
    const int ku = min(k + 1, nz - 1);
    const unsigned dk = k + 1 < nz ? q.plane : 0u;
    const cbytes U0 = flat::uni(E0 + dk), U1 = flat::uni(E1 + dk);
    const float nx1 = ld1<float>(U0, q.o1), ny1 = ld1<float>(U1, q.o1);
    const float w1 = ld1<float>(E2, q.o1), w2 = ld1<float>(E2, q.o2), x2 = ld1<float>(E0, q.o2);
    float hx = ld1<float>(H0, q.o1), hy = ld1<float>(H1, q.o1), hz = ld1<float>(H2, q.o1);
    // chi of the E side: along y of the row and the row above, x, and z of the plane above
    float cxy = 0.f, czy = 0.f, cxyu = 0.f, czyu = 0.f, cyx = 0.f, czx = 0.f, cxz = 0.f, cyz = 0.f;
    if (e_y) {
      const unsigned o = y_off(a, *ey_, pey, k, q.i), u = y_off(a, *ey_, peu, k, q.i);
      cxy = ld1<float>(in_bytes(ey_->psi[0]), o);
      czy = ld1<float>(in_bytes(ey_->psi[2]), o);
      cxyu = ld1<float>(in_bytes(ey_->psi[0]), u);
      czyu = ld1<float>(in_bytes(ey_->psi[2]), u);
    }
    if (e_x) {
      const unsigned o = x_off(a, *ex_, pex, k, q.j);
      cyx = ld1<float>(in_bytes(ex_->psi[1]), o);
      czx = ld1<float>(in_bytes(ex_->psi[2]), o);
    }
    const float4 pzu = z_prof(a, *ez_, ku);
    const int izu = (int)pzu.w;
    if (izu >= 0) {
      const unsigned o = lane_off(q.o1 + dk + (unsigned)(izu - ku) * q.plane);
      cxz = ld1<float>(in_bytes(ez_->psi[0]), o);
      cyz = ld1<float>(in_bytes(ez_->psi[1]), o);
    }
    // chi of the H side
    float qxy = 0.f, qzy = 0.f, qyx = 0.f, qzx = 0.f, qxz = 0.f, qyz = 0.f;
    unsigned ox = 0u, oy = 0u, oz = 0u;
    if (h_x) {
      ox = x_off(a, *hx_, phx, k, q.j);
      qyx = ld1<float>(in_bytes(hx_->psi[1]), ox);
      qzx = ld1<float>(in_bytes(hx_->psi[2]), ox);
    }
    if (h_y) {
      oy = y_off(a, *hy_, phy, k, q.i);
      qxy = ld1<float>(in_bytes(hy_->psi[0]), oy);
      qzy = ld1<float>(in_bytes(hy_->psi[2]), oy);
    }
    const float4 phz = z_prof(a, *hz_, k);
    const int iz = (int)phz.w;
    if (iz >= 0) {
      oz = z_off(q, q.o1, k, iz);
      qxz = ld1<float>(in_bytes(hz_->psi[0]), oz);
      qyz = ld1<float>(in_bytes(hz_->psi[1]), oz);
    }
    const float yw1 = e_y ? mix(w1, pey, ey_->has_k, czy) : w1, yw2 = e_y ? mix(w2, peu, ey_->has_k, czyu) : w2;
    const float yx1 = e_y ? mix(x1, pey, ey_->has_k, cxy) : x1, yx2 = e_y ? mix(x2, peu, ey_->has_k, cxyu) : x2;
    const float xw1 = e_x ? mix(w1, pex, ex_->has_k, czx) : w1, xy1 = e_x ? mix(y1, pex, ex_->has_k, cyx) : y1;
    const float zxu = izu >= 0 ? mix(nx1, pzu, ez_->has_k, cxz) : nx1, zyu = izu >= 0 ? mix(ny1, pzu, ez_->has_k, cyz) : ny1;
    const bool zh = k < nz - 1;
    {  // H_x
      const bool st = yh && zh;
      const float da = yw2 - yw1, db = zyu - zy;
      if (h_y) qxy = advance(qxy, phy, hx, st);
      if (iz >= 0) qxz = advance(qxz, phz, hx, st);
      hx = st ? hx - g.cH * (g.s[1] * da - g.s[2] * db) : hx;
    }
    {  // H_y
      const bool st = xh && zh;
      const float da = zxu - zx, db = shfl_dn(xw1) - xw1;
      if (h_x) qyx = advance(qyx, phx, hy, st);
      if (iz >= 0) qyz = advance(qyz, phz, hy, st);
      hy = st ? hy - g.cH * (g.s[2] * da - g.s[0] * db) : hy;
    }
    {  // H_z
      const bool st = xh && yh;
      const float da = shfl_dn(xy1) - xy1, db = yx2 - yx1;
      if (h_x) qzx = advance(qzx, phx, hz, st);
      if (h_y) qzy = advance(qzy, phy, hz, st);
      hz = st ? hz - g.cH * (g.s[0] * da - g.s[1] * db) : hz;
    }
    if (q.own) {
      st1<float>(H0, q.o1, hx);
      st1<float>(H1, q.o1, hy);
      st1<float>(H2, q.o1, hz);
      if (h_x && in_slab(phx)) {
        st1<float>(out_bytes(hx_->psi[1]), ox, qyx);
        st1<float>(out_bytes(hx_->psi[2]), ox, qzx);
      }
      if (h_y && in_slab(phy)) {
        st1<float>(out_bytes(hy_->psi[0]), oy, qxy);
        st1<float>(out_bytes(hy_->psi[2]), oy, qzy);
      }
      if (iz >= 0) {
        st1<float>(out_bytes(hz_->psi[0]), oz, qxz);
        st1<float>(out_bytes(hz_->psi[1]), oz, qyz);
      }
    }
    x1 = nx1;
    y1 = ny1;
    zx = zxu;
    zy = zyu;
    q.o1 += q.plane;
    q.o2 += q.plane;
  }
}

template <int MAT>
__device__ __forceinline__ void ae_tile(const StepArgs& a, int t, const float* tab) {
  const Grid& g = a.g;
  Cell q = cell_of<false>(a, t);
  if (!q.on) return;
  const int nz = g.n[2];
  const bool xh = q.i < g.n[0] - 1, xe = xh && q.i >= 1, yh = q.j < g.n[1] - 1, ye = yh && q.j >= 1;
  const PmlAx *ex_ = &a.pml[0], *ey_ = &a.pml[1], *ez_ = &a.pml[2];      // E side: advanced
  const PmlAx *hx_ = &a.xpml[0], *hy_ = &a.xpml[1], *hz_ = &a.xpml[2];   // H side: read
  const int jd = max(q.j - 1, 0);
  const float4 pex = prof_at(*ex_, q.i), pey = prof_at(*ey_, q.j);
  const float4 phx = prof_at(*hx_, q.i), phy = prof_at(*hy_, q.j), phd = prof_at(*hy_, jd);
  const bool e_x = __ballot(in_slab(pex)) != 0ull, e_y = __ballot(in_slab(pey)) != 0ull;
  const bool h_x = __ballot(in_slab(phx)) != 0ull, h_y = __ballot(in_slab(phy) || in_slab(phd)) != 0ull;
  const size_t comp = (size_t)g.N * 4;
  const cbytes H0 = in_bytes(a.H), H1 = H0 + comp, H2 = H1 + comp;
  const bytes E0 = out_bytes(a.E), E1 = E0 + comp, E2 = E1 + comp;

  float zxd = 0.f, zyd = 0.f;  // H_x, H_y of the plane below as differenced along z
  if (q.z0 > 0) {
    const unsigned o = lane_off(q.o1 - q.plane);
    zxd = ld1<float>(H0, o);
    zyd = ld1<float>(H1, o);
    const float4 pr = z_prof(a, *hz_, q.z0 - 1);
    const int p = (int)pr.w;
    if (p >= 0) {
      const unsigned oc = z_off(q, q.o1, q.z0, p);
      zxd = mix(zxd, pr, hz_->has_k, ld1<float>(in_bytes(hz_->psi[0]), oc));
      zyd = mix(zyd, pr, hz_->has_k, ld1<float>(in_bytes(hz_->psi[1]), oc));
    }
  }
  for (int k = q.z0; k < q.z1; ++k) {
    Coef<MAT> m;
    m.load(a, q.o1);
    const float hx = ld1<float>(H0, q.o1), hy = ld1<float>(H1, q.o1), hz = ld1<float>(H2, q.o1);
    const float hx0 = ld1<float>(H0, q.o0), hz0 = ld1<float>(H2, q.o0);
    float ex = ld1<float>(E0, q.o1), ey = ld1<float>(E1, q.o1), ez = ld1<float>(E2, q.o1);
    // chi of the H side: along y of the row and the row below, x and z
    float cxy = 0.f, czy = 0.f, cxyd = 0.f, czyd = 0.f, cyx = 0.f, czx = 0.f, cxz = 0.f, cyz = 0.f;
    if (h_y) {
      const unsigned o = y_off(a, *hy_, phy, k, q.i), d = y_off(a, *hy_, phd, k, q.i);
      cxy = ld1<float>(in_bytes(hy_->psi[0]), o);
      czy = ld1<float>(in_bytes(hy_->psi[2]), o);
      cxyd = ld1<float>(in_bytes(hy_->psi[0]), d);
      czyd = ld1<float>(in_bytes(hy_->psi[2]), d);
    }
    if (h_x) {
      const unsigned o = x_off(a, *hx_, phx, k, q.j);
      cyx = ld1<float>(in_bytes(hx_->psi[1]), o);
      czx = ld1<float>(in_bytes(hx_->psi[2]), o);
    }
    const float4 phz = z_prof(a, *hz_, k);
    const int izh = (int)phz.w;
    if (izh >= 0) {
      const unsigned o = z_off(q, q.o1, k, izh);
      cxz = ld1<float>(in_bytes(hz_->psi[0]), o);
      cyz = ld1<float>(in_bytes(hz_->psi[1]), o);
    }
    // chi of the E side
    float sxy = 0.f, szy = 0.f, syx = 0.f, szx = 0.f, sxz = 0.f, syz = 0.f;
    unsigned ox = 0u, oy = 0u, oz = 0u;
    if (e_x) {
      ox = x_off(a, *ex_, pex, k, q.j);
      syx = ld1<float>(in_bytes(ex_->psi[1]), ox);
      szx = ld1<float>(in_bytes(ex_->psi[2]), ox);
    }
    if (e_y) {
      oy = y_off(a, *ey_, pey, k, q.i);
      sxy = ld1<float>(in_bytes(ey_->psi[0]), oy);
      szy = ld1<float>(in_bytes(ey_->psi[2]), oy);
    }
    const float4 pez = z_prof(a, *ez_, k);
    const int iz = (int)pez.w;
    if (iz >= 0) {
      oz = z_off(q, q.o1, k, iz);
      sxz = ld1<float>(in_bytes(ez_->psi[0]), oz);
      syz = ld1<float>(in_bytes(ez_->psi[1]), oz);
    }
    const float yz1 = h_y ? mix(hz, phy, hy_->has_k, czy) : hz, yz0 = h_y ? mix(hz0, phd, hy_->has_k, czyd) : hz0;
    const float yx1 = h_y ? mix(hx, phy, hy_->has_k, cxy) : hx, yx0 = h_y ? mix(hx0, phd, hy_->has_k, cxyd) : hx0;
    const float xz1 = h_x ? mix(hz, phx, hx_->has_k, czx) : hz, xy1 = h_x ? mix(hy, phx, hx_->has_k, cyx) : hy;
    const float zx = izh >= 0 ? mix(hx, phz, hz_->has_k, cxz) : hx, zy = izh >= 0 ? mix(hy, phz, hz_->has_k, cyz) : hy;
    const bool zh = k < nz - 1, ze = zh && k >= 1;
    {  // E_x
      const bool st = xh && ye && ze;
      const float da = yz1 - yz0, db = zy - zyd;
      if (e_y) sxy = advance(sxy, pey, ex, st);
      if (iz >= 0) sxz = advance(sxz, pez, ex, st);
      ex = st ? ex + m.of(0, tab) * (g.s[1] * da - g.s[2] * db) : ex;
    }
    {  // E_y
      const bool st = xe && yh && ze;
      const float da = zx - zxd, db = xz1 - shfl_up(xz1);
      if (e_x) syx = advance(syx, pex, ey, st);
      if (iz >= 0) syz = advance(syz, pez, ey, st);
      ey = st ? ey + m.of(1, tab) * (g.s[2] * da - g.s[0] * db) : ey;
    }
    {  // E_z
      const bool st = xe && ye && zh;
      const float da = xy1 - shfl_up(xy1), db = yx1 - yx0;
      if (e_x) szx = advance(szx, pex, ez, st);
      if (e_y) szy = advance(szy, pey, ez, st);
      ez = st ? ez + m.of(2, tab) * (g.s[0] * da - g.s[1] * db) : ez;
    }
    if (q.own) {
      st1<float>(E0, q.o1, ex);
      st1<float>(E1, q.o1, ey);
      st1<float>(E2, q.o1, ez);
      if (e_x && in_slab(pex)) {
        st1<float>(out_bytes(ex_->psi[1]), ox, syx);
        st1<float>(out_bytes(ex_->psi[2]), ox, szx);
      }
      if (e_y && in_slab(pey)) {
        st1<float>(out_bytes(ey_->psi[0]), oy, sxy);
        st1<float>(out_bytes(ey_->psi[2]), oy, szy);
      }
      if (iz >= 0) {
        st1<float>(out_bytes(ez_->psi[0]), oz, sxz);
        st1<float>(out_bytes(ez_->psi[1]), oz, syz);
      }
    }
    zxd = zx;
    zyd = zy;
    q.o0 += q.plane;
    q.o1 += q.plane;
  }
}

}  // namespace lean

template <bool ADJ, bool LOOP>
__global__ void __launch_bounds__(64 * LEAN_WAVES) k_lean_h(const StepArgs* __restrict__ args, Sched sc) {
  for (int b = blockIdx.x; b < sc.n_pad; b += gridDim.x) {
    const int t = tile_of(b, sc);
    if (t < sc.n_tiles) {
      int m, lt;
      member_of(sc, t, m, lt);
      if (ADJ) {
        lean::ah_tile(args[m], lt);
      } else {
        note_step(args[m], lt);
        lean::h_tile(args[m], lt);
      }
    }
    if (!LOOP) break;
  }
}

template <bool ADJ, int MAT, bool LOOP>
__global__ void __launch_bounds__(64 * LEAN_WAVES) k_lean_e(const StepArgs* __restrict__ args, Sched sc) {
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
      load_tables<MAT, LEAN_WAVES, 0>(a, cur >= 0, tab, nullptr);
      cur = m;
    }
    if (ADJ) lean::ae_tile<MAT>(a, lt, tab);
    else lean::e_tile<MAT>(a, lt, tab);
    if (!LOOP) break;
  }
}

}  // namespace lsf
