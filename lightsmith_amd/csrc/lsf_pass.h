// One time step in a single pass over the grid: H^{n+1/2} and E^{n+1} from E^n and H^{n-1/2}, for real fields on cubic
// cells without periodic axes (engine.py:630-663 with the pure-ADE update of engine.py:769-793). Same arithmetic per
// cell as the row kernels (lsf_step.h): the fields equal those of an H launch followed by an E launch.
//
// The pass reads one buffer set (E, H, H-side psi) and writes the other, so no wavefront reads another's new values;
// steps go in pairs (set 0 to 1 and back), so that the caller's buffers hold the state whenever the host has it.
// E-side psi and the pole state are updated in place: one owner each.
//
// Mapping. The rows of a plane are laid end to end, one x cell per lane; a wavefront takes 64 lanes and owns the middle
// 62. Its first lane computes H only (the x - 1 neighbour of the second), its last supplies E at x + 1, so no cell
// needs a halo load of its own. Per plane of the z march a lane computes H of its cell and, once more, H_x and H_z of
// the cell below it in y (from the same inputs as their owner), then E; H of the plane below is carried in registers
// (a tile begins with H_x, H_y of the plane below it).
//
// What bounds it. Two launches move E and H three times between them (72 B per cell and step and the coefficients), the
// pass moves each once in and once out (48 B); its re-reads of neighbouring rows and planes are served by the caches.
// Past the memory-side cache that is HBM (320^3, 3 poles: 2.73 GB a step at 4.4 TB/s, the vector units busy for 37 % of the
// cycles, 270 instructions a cell); within it the step's bytes move at 5.1-5.4 TB/s and instructions weigh as much: the
// vector units are busy for 70 % of a 131 x 117 x 150 box's cycles (dense coefficients, kappa, 45 % of the cells in slabs:
// 355 a cell) and for 54 % of a 192 x 160 x 128 one's with one-pole nodes (276 a cell). So:
// - every address is a wave-uniform base and a 32-bit lane offset; the three row offsets advance by a plane per
//   iteration (a component is below 4 GB), nothing else is recomputed;
// - lanes outside a CPML slab read a psi that they do not use, whole wavefronts outside one skip its terms;
// - D-form nodes are advanced by node, not by cell: the owners of a plane's nodes list them in LDS, the lanes take 64
//   at a time.
// Two cells per lane halve the instructions but take 150-200 registers (320^3, 3 poles: 742 us against 667), two rows
// per lane gain nothing over one, and an occupancy forced by launch bounds spills (up to 4 times slower).
//
// Measured, us per step, two kernels -> pass, at pass_pays (lsf.hip), which picks between them.
#pragma once

#include "lsf_flat.h"

namespace lsf {

// D-form nodes of a 32-cell x chunk and component: first pole slot, and which cells hold a node
struct DChunk {
  int base;
  unsigned mask;
};

struct PassArgs {
  Grid g;
  const float* E_in;
  const float* H_in;
  float* E_out;
  float* H_out;
  const float* cbd;
  const uint32_t* mid;
  const float* mtab;
  const float4* prof[2][3];   // [E side, H side][axis], null without CPML on the axis
  float* psiE[3][3];          // [axis][component]
  const float* psiHi[3][3];
  float* psiHo[3][3];
  int ns[2][3];
  int has_k[2][3];            // the axis has the kappa term
  int zlo, zhi;               // planes [zlo, zhi) lie in no z slab
  const DChunk* dform;        // [N2][N1][nchunk][3]
  void* P;
  int nchunk, media_stride, n_media_floats;
  const float* media;
  long long* counter;
  int tiles_p, zc;            // tiles per plane, planes per tile
  int second;                 // the second pass of a pair
  Corrs corr;                 // source corrections of E
};

constexpr int PASS_WAVES = 4, PASS_OWN = 62;

namespace pass {

using flat::bytes;
using flat::cbytes;
using flat::ld1;
using flat::st1;

// The D-form nodes a wavefront owns on one plane, packed: E^n of each, then its sum of pole increments; its slot and
// medium.
struct Nodes {
  float e[192];
  int slot[192];
  unsigned char m[192];
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A lane offset the compiler does not look into: a load then takes it as the 32-bit offset from a scalar base (seen as
// a shifted index it becomes a 64-bit addition per load).
__device__ __forceinline__ unsigned lane_off(unsigned o) {
  asm("" : "+v"(o));
  return o;
}

__device__ __forceinline__ float hide(float x) {
  asm("" : "+v"(x));
  return x;
}

__device__ __forceinline__ cbytes in_bytes(const void* p) { return (cbytes)as_global((const char*)p); }
__device__ __forceinline__ bytes out_bytes(void* p) { return (bytes)as_global((char*)p); }

template <int MAT, int NP, int KAP>
__device__ __forceinline__ void tile(const PassArgs& a, int t, const float* tab, const float4* med, Nodes* nodes) {
  const Grid& g = a.g;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tz = t / a.tiles_p, tp = t - tz * a.tiles_p;
  const int nx = g.n[0], ny = g.n[1], nz = g.n[2];
  const int total = nx * ny;
  const int l0 = (tp * PASS_WAVES + wv) * PASS_OWN;
  if (l0 >= total) return;
  const int lr = l0 + lane - 1;
  const int l = min(max(lr, 0), total - 1);
  const int j = l / nx, i = l - j * nx;
  const bool own = lane >= 1 && lane <= PASS_OWN && lr < total;
  const int z0 = tz * a.zc, z1 = min(z0 + a.zc, nz);
  const unsigned plane = (unsigned)total * 4u, row = (unsigned)nx * 4u;

  // the cell and its y neighbours (clamped to the grid), as byte offsets in a component
  const unsigned in_plane = (unsigned)l * 4u;
  const unsigned kb = (unsigned)(z0 > 0 ? z0 - 1 : 0) * plane;
  unsigned o1 = lane_off(in_plane + kb);
  unsigned o0 = lane_off(o1 - (j > 0 ? row : 0u)), o2 = lane_off(o1 + (j < ny - 1 ? row : 0u));

  // which cells step (engine.py:47-66); what a cell that steps reads of its neighbours' new H always steps itself
  const bool xh = i < nx - 1, xe = xh && i >= 1, yh = j < ny - 1, ye = yh && j >= 1;
  const float cH = g.cH;

  // CPML of the lane: x, and y of its row and the row below
  const float4* q;
  q = a.prof[0][0];
  const float4 pex = q ? ((const float4*)as_global(q))[i] : no_pml();
  q = a.prof[1][0];
  const float4 phx = q ? ((const float4*)as_global(q))[i] : no_pml();
  q = a.prof[0][1];
  const float4 pey = q ? ((const float4*)as_global(q))[j] : no_pml();
  q = a.prof[1][1];
  const float4 phy = q ? ((const float4*)as_global(q))[j] : no_pml();
  const float4 phy0 = q ? ((const float4*)as_global(q))[max(j - 1, 0)] : no_pml();
  const bool has_xh = __ballot(phx.w >= 0.f) != 0ull, has_xe = __ballot(pex.w >= 0.f) != 0ull;
  const bool has_yh = __ballot(phy.w >= 0.f || phy0.w >= 0.f) != 0ull, has_ye = __ballot(pey.w >= 0.f) != 0ull;

  const size_t comp = (size_t)g.N * 4;
  const cbytes E0 = in_bytes(a.E_in), E1 = E0 + comp, E2 = E1 + comp;
  const cbytes H0 = in_bytes(a.H_in), H1 = H0 + comp, H2 = H1 + comp;
  const bytes F0 = out_bytes(a.E_out), F1 = F0 + comp, F2 = F1 + comp;
  const bytes G0 = out_bytes(a.H_out), G1 = G0 + comp, G2 = G1 + comp;
  const cbytes M0 = in_bytes(MAT == 1 ? (const void*)a.mid : (const void*)a.cbd), M1 = M0 + comp, M2 = M1 + comp;

  // acc + the CPML term of one axis; psi advances. KAP: no axis has the kappa term (0), every one with CPML (1) or some (2:
  // asked for each, 1 % of a 131 x 117 x 150 box's step). (The profile's c is hidden from the loop: its products with the
  // coefficients would be kept in a register each.)
  auto pml = [](float acc, const float4 pr, int has_k, float coef, float der, float& psi) {
    return acc + pml_apply(make_float4(pr.x, hide(pr.y), KAP ? hide(pr.z) : pr.z, pr.w), KAP == 1 || (KAP == 2 && has_k), coef, der, psi);
  };
  // the same along x or y, for the lanes in the slab
  auto pml_in = [&](float acc, const float4 pr, int has_k, float coef, float der, float& psi) {
    const float v = pml(acc, pr, has_k, coef, der, psi);
    return pr.w >= 0.f ? v : acc;
  };
  // psi offsets: x slabs [k][j][p], y slabs [k][p][i], z slabs [p][j][i] (o: the cell's offset on plane k)
  auto xoff = [&](int f, const float4 pr, int k, int jj) {
    return lane_off((unsigned)((k * ny + jj) * a.ns[f][0] + max((int)pr.w, 0)) * 4u);
  };
  auto yoff = [&](int f, const float4 pr, int k) {
    return lane_off((unsigned)((k * a.ns[f][1] + max((int)pr.w, 0)) * nx + i) * 4u);
  };
  auto zoff = [&](unsigned o, int k, int p) { return lane_off(o + (unsigned)(p - k) * plane); };

  // --- D-form nodes: the next plane's list in LDS, its first round of pole pairs in registers
  constexpr int NPR = NP > 0 ? NP : 1;
  Pair<float> pp[NPR];
  int slot = 0;
  int pos[3] = {-1, -1, -1};
  int cnt = 0;
  const gptr<Pair<float>> Pg = as_global((Pair<float>*)a.P);
  const unsigned below_bit = (1u << (i & 31)) - 1u;
  unsigned oc = 0u;  // the lane's D-form chunk of the next plane to list
  const unsigned oc_plane = (unsigned)ny * (unsigned)a.nchunk * 24u;
  if (NP > 0) oc = lane_off((((unsigned)z0 * (unsigned)ny + (unsigned)j) * (unsigned)a.nchunk + (unsigned)(i >> 5)) * 24u);
  auto load_chunks = [&](DChunk (&dc)[3]) {
    const cbytes b = in_bytes(a.dform);
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const f2u v = *(gptr<const f2u>)(b + oc + (unsigned)c * 8u);
      dc[c].base = __float_as_int(v.x);
      dc[c].mask = __float_as_uint(v.y);
    }
    oc += oc_plane;
  };
  auto list_nodes = [&](const DChunk (&dc)[3]) {
    cnt = 0;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const bool d = own && ((dc[c].mask >> (i & 31)) & 1u);
      const unsigned long long m = __ballot(d);
      const int at = cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      pos[c] = d ? at : -1;
      if (d) nodes->slot[at] = dc[c].base + __popc(dc[c].mask & below_bit);
      cnt += __popcll(m);
    }
    if (cnt > 0) {
      wave_sync();
      if (lane < cnt) {
        slot = nodes->slot[lane];
        load_slot((const Pair<float>*)Pg + (size_t)(unsigned)slot * NPR, pp);
      }
    }
  };

  float x1, y0, y1;            // E_x of the cell, E_y of the cell and the row below, on plane k
  float hxq = 0.f, hyq = 0.f;  // H_x, H_y of the cell on plane k - 1
  if (NP > 0) {
    DChunk dc[3];
    load_chunks(dc);
    list_nodes(dc);
  }
  if (z0 > 0) {  // H_x, H_y of the plane below the tile
    const int k = z0 - 1;
    const float ax = ld1<float>(E0, o1), ay = ld1<float>(E1, o1), az = ld1<float>(E2, o1), azu = ld1<float>(E2, o2);
    float hx = ld1<float>(H0, o1), hy = ld1<float>(H1, o1);
    const unsigned u1 = lane_off(o1 + plane);
    x1 = ld1<float>(E0, u1);
    y1 = ld1<float>(E1, u1);
    float qy = 0.f, qx = 0.f, qz0 = 0.f, qz1 = 0.f;
    float4 pz = no_pml();
    if (has_yh) qy = ld1<float>(in_bytes(a.psiHi[1][0]), yoff(1, phy, k));
    if (has_xh) qx = ld1<float>(in_bytes(a.psiHi[0][1]), xoff(1, phx, k, j));
    if (k < a.zlo || k >= a.zhi) pz = a.prof[1][2] ? ld_uniform(a.prof[1][2], k) : no_pml();
    const int iz = (int)pz.w;
    if (iz >= 0) {
      const unsigned o = zoff(o1, k, iz);
      qz0 = ld1<float>(in_bytes(a.psiHi[2][0]), o);
      qz1 = ld1<float>(in_bytes(a.psiHi[2][1]), o);
    }
    {
      const float da = azu - az, db = y1 - ay;
      float acc = -cH * (da - db);
      if (has_yh) acc = pml_in(acc, phy, a.has_k[1][1], -cH, da, qy);
      if (iz >= 0) acc = pml(acc, pz, a.has_k[1][2], cH, db, qz0);
      hxq = hx + acc;
    }
    {
      const float azr = shfl_dn(az), da = x1 - ax, db = azr - az;
      float acc = -cH * (da - db);
      if (has_xh) acc = pml_in(acc, phx, a.has_k[1][0], cH, db, qx);
      if (iz >= 0) acc = pml(acc, pz, a.has_k[1][2], -cH, da, qz1);
      hyq = hy + acc;
    }
    o0 += plane;
    o1 += plane;
    o2 += plane;
  } else {
    x1 = ld1<float>(E0, o1);
    y1 = ld1<float>(E1, o1);
  }
  y0 = ld1<float>(E1, o0);

  for (int k = z0; k < z1; ++k) {
    const unsigned dk = k + 1 < nz ? plane : 0u;  // (E of the plane above: scalar bases a plane up)
    const cbytes U0 = flat::uni(E0 + dk), U1 = flat::uni(E1 + dk);
    // ---- loads: E of plane k (E_z of the three rows, E_x of the outer two) and, of the plane above, E_x, E_y
    const float w0 = ld1<float>(E2, o0), w1 = ld1<float>(E2, o1), w2 = ld1<float>(E2, o2);
    const float x0 = ld1<float>(E0, o0), x2 = ld1<float>(E0, o2);
    const float nx1 = ld1<float>(U0, o1), ny0 = ld1<float>(U1, o0), ny1 = ld1<float>(U1, o1);
    float hx0 = ld1<float>(H0, o0), hx1 = ld1<float>(H0, o1), hy1 = ld1<float>(H1, o1);
    float hz0 = ld1<float>(H2, o0), hz1 = ld1<float>(H2, o1);
    uint32_t id = 0u;
    float cb[3] = {};
    if (MAT == 1) {
      id = __float_as_uint(ld1<float>(M0, o1));
    } else {
      cb[0] = ld1<float>(M0, o1);
      cb[1] = ld1<float>(M1, o1);
      cb[2] = ld1<float>(M2, o1);
    }
    DChunk dc[3];
    if (NP > 0 && k + 1 < z1) load_chunks(dc);
    // psi: q of H (row below: suffix 0), s of E; names: component, axis
    float qxy = 0.f, qxy0 = 0.f, qzy = 0.f, qzy0 = 0.f, qyx = 0.f, qzx = 0.f, qzx0 = 0.f, qxz = 0.f, qxz0 = 0.f, qyz = 0.f;
    float sxy = 0.f, szy = 0.f, syx = 0.f, szx = 0.f, sxz = 0.f, syz = 0.f;
    unsigned oxh = 0u, oxe = 0u, oyh = 0u, oye = 0u, ozh = 0u, oze = 0u;
    if (has_xh) {
      oxh = xoff(1, phx, k, j);
      const unsigned o = xoff(1, phx, k, max(j - 1, 0));
      qyx = ld1<float>(in_bytes(a.psiHi[0][1]), oxh);
      qzx = ld1<float>(in_bytes(a.psiHi[0][2]), oxh);
      qzx0 = ld1<float>(in_bytes(a.psiHi[0][2]), o);
    }
    if (has_yh) {
      oyh = yoff(1, phy, k);
      const unsigned o = yoff(1, phy0, k);
      qxy = ld1<float>(in_bytes(a.psiHi[1][0]), oyh);
      qzy = ld1<float>(in_bytes(a.psiHi[1][2]), oyh);
      qxy0 = ld1<float>(in_bytes(a.psiHi[1][0]), o);
      qzy0 = ld1<float>(in_bytes(a.psiHi[1][2]), o);
    }
    float4 pzh = no_pml(), pze = no_pml();
    if (k < a.zlo || k >= a.zhi) {
      if (a.prof[1][2]) pzh = ld_uniform(a.prof[1][2], k);
      if (a.prof[0][2]) pze = ld_uniform(a.prof[0][2], k);
    }
    const int izh = (int)pzh.w, ize = (int)pze.w;
    if (izh >= 0) {
      ozh = zoff(o1, k, izh);
      qxz = ld1<float>(in_bytes(a.psiHi[2][0]), ozh);
      qyz = ld1<float>(in_bytes(a.psiHi[2][1]), ozh);
      qxz0 = ld1<float>(in_bytes(a.psiHi[2][0]), zoff(o0, k, izh));
    }
    if (has_xe) {
      oxe = xoff(0, pex, k, j);
      syx = ld1<float>(in_bytes(a.psiE[0][1]), oxe);
      szx = ld1<float>(in_bytes(a.psiE[0][2]), oxe);
    }
    if (has_ye) {
      oye = yoff(0, pey, k);
      sxy = ld1<float>(in_bytes(a.psiE[1][0]), oye);
      szy = ld1<float>(in_bytes(a.psiE[1][2]), oye);
    }
    if (ize >= 0) {
      oze = zoff(o1, k, ize);
      sxz = ld1<float>(in_bytes(a.psiE[2][0]), oze);
      syz = ld1<float>(in_bytes(a.psiE[2][1]), oze);
    }

    // ---- H^{n+1/2}: CPML terms in ascending axis order; a cell that does not step keeps its H and psi
    const bool zh = k < nz - 1;
    {  // H_x: y difference of E_z, z difference of E_y
      const bool st = yh && zh;
      const float da = w2 - w1, db = ny1 - y1, da0 = w1 - w0, db0 = ny0 - y0;
      float acc = -cH * (da - db), acc0 = -cH * (da0 - db0);
      if (has_yh) {
        float n = qxy, n0 = qxy0;
        acc = pml_in(acc, phy, a.has_k[1][1], -cH, da, n);
        acc0 = pml_in(acc0, phy0, a.has_k[1][1], -cH, da0, n0);
        qxy = st ? n : qxy;
      }
      if (izh >= 0) {
        float n = qxz, n0 = qxz0;
        acc = pml(acc, pzh, a.has_k[1][2], cH, db, n);
        acc0 = pml(acc0, pzh, a.has_k[1][2], cH, db0, n0);
        qxz = st ? n : qxz;
      }
      hx1 = st ? hx1 + acc : hx1;
      hx0 += acc0;
    }
    {  // H_y: z difference of E_x, x difference of E_z
      const bool st = xh && zh;
      const float da = nx1 - x1, db = shfl_dn(w1) - w1;
      float acc = -cH * (da - db);
      if (has_xh) {
        float n = qyx;
        acc = pml_in(acc, phx, a.has_k[1][0], cH, db, n);
        qyx = st ? n : qyx;
      }
      if (izh >= 0) {
        float n = qyz;
        acc = pml(acc, pzh, a.has_k[1][2], -cH, da, n);
        qyz = st ? n : qyz;
      }
      hy1 = st ? hy1 + acc : hy1;
    }
    {  // H_z: x difference of E_y, y difference of E_x
      const bool st = xh && yh;
      const float da = shfl_dn(y1) - y1, db = x2 - x1, da0 = shfl_dn(y0) - y0, db0 = x1 - x0;
      float acc = -cH * (da - db), acc0 = -cH * (da0 - db0);
      if (has_xh) {
        float n = qzx, n0 = qzx0;
        acc = pml_in(acc, phx, a.has_k[1][0], -cH, da, n);
        acc0 = pml_in(acc0, phx, a.has_k[1][0], -cH, da0, n0);
        qzx = st ? n : qzx;
      }
      if (has_yh) {
        float n = qzy, n0 = qzy0;
        acc = pml_in(acc, phy, a.has_k[1][1], cH, db, n);
        acc0 = pml_in(acc0, phy0, a.has_k[1][1], cH, db0, n0);
        qzy = st ? n : qzy;
      }
      hz1 = st ? hz1 + acc : hz1;
      hz0 += acc0;
    }

    // ---- poles
    auto coef = [&](int c) -> float {
      if (MAT == 1) return tab[(id >> (8 * c)) & 255u];
      return cb[c];
    };
    const float cv[3] = {coef(0), coef(1), coef(2)};
    if (NP > 0 && cnt > 0) {
      const bool multi = a.n_media_floats > a.media_stride;
      const float eo[3] = {x1, y1, w1};
#pragma unroll
      for (int c = 0; c < 3; ++c)
        if (pos[c] >= 0) {
          nodes->e[pos[c]] = eo[c];
          if (multi) nodes->m[pos[c]] = (unsigned char)((int)(-cv[c]) - 1);
        }
      wave_sync();
      auto advance = [&](int r, int sl, Pair<float> (&p)[NPR]) {
        const float eold = nodes->e[r];
        const float4* mp = med + (multi ? (int)nodes->m[r] * (NP + 1) : 0);
        float dp = 0.f;
#pragma unroll
        for (int n = 0; n < NPR; ++n) {
          const float4 cf = mp[1 + n];
          const float pn = fmad(cf.x, p[n].p, fmad(cf.y, p[n].q, scl(cf.z, eold)));
          dp = add(dp, sub(pn, p[n].p));
          p[n].q = p[n].p;
          p[n].p = pn;
        }
        nodes->e[r] = dp;
        store_slot((Pair<float>*)Pg + (size_t)(unsigned)sl * NPR, p);
      };
      if (lane < cnt) advance(lane, slot, pp);
      constexpr int MORE = NP <= 2 ? 2 : 1;  // further rounds loaded together (at most 186 nodes: three in all)
      for (int r0 = 64; r0 < cnt; r0 += 64 * MORE) {
        Pair<float> pq[MORE][NPR];
        int sq[MORE];
#pragma unroll
        for (int b = 0; b < MORE; ++b)
          if (r0 + 64 * b + lane < cnt) {
            sq[b] = nodes->slot[r0 + 64 * b + lane];
            load_slot((const Pair<float>*)Pg + (size_t)(unsigned)sq[b] * NPR, pq[b]);
          }
#pragma unroll
        for (int b = 0; b < MORE; ++b)
          if (r0 + 64 * b + lane < cnt) advance(r0 + 64 * b + lane, sq[b], pq[b]);
      }
      wave_sync();
    }

    // ---- E^{n+1}
    const bool ze = k >= 1 && zh;
    auto finish = [&](int c, bool st, float eold, float dE) {
      float enew = eold + dE;
      if (NP > 0 && pos[c] >= 0) {
        const float inv = med[((int)(-cv[c]) - 1) * (NP + 1)].x;
        enew = fmad(inv, dE - nodes->e[pos[c]], eold);
      }
      return st ? enew : eold;
    };
    auto cbe = [&](int c) { return NP > 0 && cv[c] < 0.f ? g.cdx : cv[c]; };
    float ex, ey, ew;
    {  // E_x: y difference of H_z, z difference of H_y
      const bool st = xh && ye && ze;
      const float da = hz1 - hz0, db = hy1 - hyq, c = cbe(0);
      float acc = c * (da - db);
      if (has_ye) {
        float n = sxy;
        acc = pml_in(acc, pey, a.has_k[0][1], c, da, n);
        sxy = st ? n : sxy;
      }
      if (ize >= 0) {
        float n = sxz;
        acc = pml(acc, pze, a.has_k[0][2], -c, db, n);
        sxz = st ? n : sxz;
      }
      ex = finish(0, st, x1, acc);
    }
    {  // E_y: z difference of H_x, x difference of H_z
      const bool st = xe && yh && ze;
      const float da = hx1 - hxq, db = hz1 - shfl_up(hz1), c = cbe(1);
      float acc = c * (da - db);
      if (has_xe) {
        float n = syx;
        acc = pml_in(acc, pex, a.has_k[0][0], -c, db, n);
        syx = st ? n : syx;
      }
      if (ize >= 0) {
        float n = syz;
        acc = pml(acc, pze, a.has_k[0][2], c, da, n);
        syz = st ? n : syz;
      }
      ey = finish(1, st, y1, acc);
    }
    {  // E_z: x difference of H_y, y difference of H_x
      const bool st = xe && ye && zh;
      const float da = hy1 - shfl_up(hy1), db = hx1 - hx0, c = cbe(2);
      float acc = c * (da - db);
      if (has_xe) {
        float n = szx;
        acc = pml_in(acc, pex, a.has_k[0][0], c, da, n);
        szx = st ? n : szx;
      }
      if (has_ye) {
        float n = szy;
        acc = pml_in(acc, pey, a.has_k[0][1], -c, db, n);
        szy = st ? n : szy;
      }
      ew = finish(2, st, w1, acc);
    }
    // ---- stores: every owned cell (what does not step keeps its value in the other set)
    if (own) {
      st1<float>(F0, o1, ex);
      st1<float>(F1, o1, ey);
      st1<float>(F2, o1, ew);
      st1<float>(G0, o1, hx1);
      st1<float>(G1, o1, hy1);
      st1<float>(G2, o1, hz1);
      if (has_xh && phx.w >= 0.f) {
        st1<float>(out_bytes(a.psiHo[0][1]), oxh, qyx);
        st1<float>(out_bytes(a.psiHo[0][2]), oxh, qzx);
      }
      if (has_xe && pex.w >= 0.f) {
        st1<float>(out_bytes(a.psiE[0][1]), oxe, syx);
        st1<float>(out_bytes(a.psiE[0][2]), oxe, szx);
      }
      if (has_yh && phy.w >= 0.f) {
        st1<float>(out_bytes(a.psiHo[1][0]), oyh, qxy);
        st1<float>(out_bytes(a.psiHo[1][2]), oyh, qzy);
      }
      if (has_ye && pey.w >= 0.f) {
        st1<float>(out_bytes(a.psiE[1][0]), oye, sxy);
        st1<float>(out_bytes(a.psiE[1][2]), oye, szy);
      }
      if (izh >= 0) {
        st1<float>(out_bytes(a.psiHo[2][0]), ozh, qxz);
        st1<float>(out_bytes(a.psiHo[2][1]), ozh, qyz);
      }
      if (ize >= 0) {
        st1<float>(out_bytes(a.psiE[2][0]), oze, sxz);
        st1<float>(out_bytes(a.psiE[2][1]), oze, syz);
      }
    }
    if (NP > 0 && k + 1 < z1) {
      wave_sync();  // the list's readers are done
      list_nodes(dc);
    }
    x1 = nx1;
    y0 = ny0;
    y1 = ny1;
    hxq = hx1;
    hyq = hy1;
    o0 += plane;
    o1 += plane;
    o2 += plane;
  }
  correct<float, 1>(a.corr, a.second ? a.corr.step : a.counter, a.second, a.E_out, g, own, i, j, 0, z0, z1);
}

// The pair's passes advance the step counter: counter[1] = n after each, counter[0] = n + 1 after the second only (the
// operations that follow a pass read counter[1]). No pass writes a word that its blocks may still read: the first reads
// counter[0] and writes counter[1] and its copy of n, the second reads the copy.
__device__ __forceinline__ void tick_pair(const PassArgs& a, int lt) {
  if (lt != 0 || threadIdx.x != 0) return;
  long long* cnt = (long long*)as_global(a.counter);
  long long* step = (long long*)as_global(a.corr.step);
  if (a.second) {
    const long long n = *step + 1;
    cnt[1] = n;
    cnt[0] = n + 1;
  } else {
    cnt[1] = *step = cnt[0];
  }
}

}  // namespace pass

template <int MAT, int NP, int KAP>
__global__ void __launch_bounds__(64 * PASS_WAVES) k_pass(const PassArgs* __restrict__ args, Sched sc) {
  __shared__ float tab[MAT == 1 ? 256 : 1];
  __shared__ float4 med_tab[NP > 0 ? MAX_MEDIA_VEC4 : 1];
  __shared__ pass::Nodes nodes[NP > 0 ? PASS_WAVES : 1];
  const int t = tile_of(blockIdx.x, sc);
  if (t >= sc.n_tiles) return;  // whole block
  int m, lt;
  member_of(sc, t, m, lt);
  const PassArgs& a = args[m];
  pass::tick_pair(a, lt);
  if (MAT == 1 || NP > 0) load_tables<MAT, PASS_WAVES, NP>(a, false, tab, med_tab);
  pass::tile<MAT, NP, KAP>(a, lt, tab, med_tab, nodes + (NP > 0 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0));
}

}  // namespace lsf
