// fdtd_quad.h -- the fused Yee + CPML face passes, four x cells per lane.
//
// What bounds them: on grids past the caches HBM, a half step reads three
// components, updates three more and reads their media, 36-42 bytes a cell, at
// half a flop per byte; on small grids the chain of dependent accesses from
// launch to last store.  A lane that owns one cell asks for 4 bytes a load and
// cannot keep enough of them in flight; a lane here owns the 16-byte vector of
// cells i0 .. i0 + 3 (8 bytes of binary16), a quarter of the memory
// instructions and four times the bytes in flight per wave.
//
// The x-y plane holds nx / 4 + 1 vectors a row.  The grid is cut along y and z
// into boxes (QuadPlan): the interior, whose cells lie in no y or z slab, and
// up to four slabs around it.  A tile is a run of 64 * rows consecutive vectors
// of a box's plane in x-fastest order (it may wrap from one row to the next, so
// no width leaves lanes idle) and marches kc planes, the z neighbours carried
// in registers; one launch runs all boxes, an interior tile in code without y
// and z slabs.  (The x slabs stay in the interior's rows: as boxes of their own
// they share no line with it, 256^3 with 10 layers: 107 + 144 us per pass
// against 141 + 44.  Two launches, each with its own registers, 6 and 3 waves a
// SIMD, lose to one: 256^3 386 against 369 us per step, 64^3 27.4 against 18.6.)
//
// The y neighbours come from memory (the row was loaded by a nearby lane: L1
// or L2), the x neighbours inside a vector from the lane itself, across vectors
// by a DPP wave shift, and by one extra load at a wave's edge and at the edge
// of a row.  The last vector of a row ends past the sweep: its cells there go
// back as they were read.  Every load of a plane is issued before its
// arithmetic, the psi values and the first TF/SF term among them; along x and
// y a slab is a matter of the lane, along z of the plane.
//
// Per cell the arithmetic and its order are the one-cell passes', so the
// results are the same bits.
#pragma once
#include "fdtd_device.h"

namespace sfd {
namespace SFD_NS {

// a 16-byte vector at any 4-byte boundary (psi rows)
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// the field vector of a lane: raw bits, conversion, and the write-back of the
// first n cells (the others keep the bits of old)
template <class T> struct Quad;
template <> struct Quad<float> {
  typedef f32x4 raw;
  static __device__ __forceinline__ void cvt(raw r, float, float (&v)[4]) {
    v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w;
  }
  static __device__ __forceinline__ raw pack(const float (&v)[4], float, raw old, int n) {
    raw r;
    r.x = n > 0 ? v[0] : old.x;
    r.y = n > 1 ? v[1] : old.y;
    r.z = n > 2 ? v[2] : old.z;
    r.w = n > 3 ? v[3] : old.w;
    return r;
  }
};
template <> struct Quad<__half> {
  typedef u32x2 raw;
  static __device__ __forceinline__ void cvt(raw r, float s, float (&v)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      v[c] = Store<__half>::cvt((unsigned short)((c < 2 ? r.x : r.y) >> (16 * (c & 1))), s);
  }
  static __device__ __forceinline__ raw pack(const float (&v)[4], float is, raw old, int n) {
    unsigned h[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const unsigned o = ((c < 2 ? old.x : old.y) >> (16 * (c & 1))) & 0xffffu;
      const unsigned w = __half_as_ushort(__float2half_rn(rounded(v[c] * is)));
      h[c] = c < n ? w : o;
    }
    raw r;
    r.x = h[0] | (h[1] << 16);
    r.y = h[2] | (h[3] << 16);
    return r;
  }
};
template <class T>
__device__ __forceinline__ typename Quad<T>::raw ldq(const SFD_GLOBAL char *b, unsigned ob) {
  return ld_at((const SFD_GLOBAL typename Quad<T>::raw *)b, ob);
}

// four psi values of a slab row, and the write-back of cells a .. n - 1
__device__ __forceinline__ void ld_psi(const SFD_GLOBAL float *b, unsigned ob, float (&v)[4]) {
  const f32x4u t = *(const SFD_GLOBAL f32x4u *)((const SFD_GLOBAL char *)b + ob);
  v[0] = t.x; v[1] = t.y; v[2] = t.z; v[3] = t.w;
}
__device__ __forceinline__ void st_psi(SFD_GLOBAL float *b, unsigned ob, const float (&v)[4],
                                       int a, int n) {
  if (a <= 0 && n >= 4) {
    f32x4u t;
    t.x = v[0]; t.y = v[1]; t.z = v[2]; t.w = v[3];
    *(SFD_GLOBAL f32x4u *)((SFD_GLOBAL char *)b + ob) = t;
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (c >= a && c < n) st_at(b, ob + 4u * c, v[c]);
  }
}

// the x slab cells of a vector: cells a .. n - 1 (n <= a: none), the first
// cell's slab index q (cells below a shift it below the slab: the caller's
// psi bases allow for -3).  An interior at least four cells wide keeps a
// vector from meeting both slabs.  last: the last swept index, hs: the first
// high-slab index.
struct XSlab {
  int a, n, q;
};
__device__ __forceinline__ XSlab x_slab(int i0, int L0, int L1, int hs, int last) {
  XSlab s{0, 0, 0};
  if (i0 < L0) {
    s.n = min(L0 - i0, 4);
    s.q = i0;
  } else if (L1 && i0 + 3 >= hs) {
    s.a = max(hs - i0, 0);
    s.n = min(last + 1 - i0, 4);
    s.q = L0 + i0 - hs;
  }
  return s;
}

// G2 (or GM2) per cell and the Yee update of one component's four cells
template <bool UNI>
__device__ __forceinline__ void yee4(const MedTab &t, float2 cu, u32x2 m, const float (&f)[4],
                                     const float (&a)[4], const float (&ia)[4],
                                     const float (&b)[4], const float (&ib)[4], float (&r)[4],
                                     float (&g2)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float2 co = UNI ? cu : t.gg[((c < 2 ? m.x : m.y) >> (16 * (c & 1))) & 0xffffu];
    g2[c] = co.y;
    r[c] = yee_upd(co.x, f[c], co.y, curl2(a[c], ia[c], b[c], ib[c]));
  }
}

// psi <- b psi + d c in cells a .. n - 1, F += sgn G2 psi there, psi stored.
// ALL: the slab holds every cell of the vector (y and z slabs; the cells past
// the sweep are dropped at the stores)
template <bool ALL, bool NEG>
__device__ __forceinline__ void psi4(SFD_GLOBAL float *s, unsigned ob, float (&psi)[4],
                                     const float (&d)[4], const float (&cc)[4],
                                     const float (&bb)[4], const float (&g2)[4], int a, int n,
                                     float (&r)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float v = madd(d[c] * cc[c], bb[c], psi[c]);
    psi[c] = v;
    const float x = madd(r[c], NEG ? -g2[c] : g2[c], v);
    r[c] = ALL || (c >= a && c < n) ? x : r[c];
  }
  st_psi(s, ob, psi, a, n);
}

// Waits for the plane's loads in one place.  Left to the compiler, each psi
// value is waited for where it is used, and as the slab branches leave it no
// count of what was issued since, each of those waits takes in the stores
// before it: four to six store round trips a plane.
__device__ __forceinline__ void plane_wait() {
  __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0)
}

#define SFD_ALL4(x) {(x), (x), (x), (x)}

// the lane's vector in tile t of box x: its row j and first cell i0, the
// tile's planes k0 .. k1 - 1, and whether the vector is the first or the last
// of its box's row; false for a lane past the box (these are the last lanes
// of the tile: no other lane's wave shift needs them)
struct QuadPos {
  int i0, j, k0, k1;
  bool first, last;
};
__device__ __forceinline__ bool quad_pos(const QuadBox &x, int t, QuadPos &o) {
  const int bz = t / x.tx, run = t - bz * x.tx;
  const int f = (run * (int)blockDim.y + (int)threadIdx.y) * kWave + (int)threadIdx.x;
  const int r = f / x.nq, q = f - r * x.nq;
  o.i0 = 4 * (x.q0 + q);
  o.j = x.j0 + r;
  o.k0 = x.k0 + bz * x.kc;
  o.k1 = min(o.k0 + x.kc, x.k0 + x.nk);
  o.first = q == 0;
  o.last = q == x.nq - 1;
  return r < x.nj;
}
// a box read through whatever address space holds it
template <class B>
__device__ __forceinline__ QuadBox load_box(const B &b) {
  return QuadBox{b.q0, b.nq, b.j0, b.nj, b.k0, b.nk, b.tx, b.kc};
}
// tile t of a plan
template <class P>
__device__ __forceinline__ bool quad_pos(const P &p, int t, QuadPos &o) {
  int b = 0, start = 0;
#pragma unroll
  for (int i = 1; i < kQuadBoxes; ++i)
    if (t >= p.start[i]) { b = i; start = p.start[i]; }
  return quad_pos(load_box(p.box[b]), t - start, o);
}

// a descriptor whose members are read anew where this is called: held across
// the march, the bases of fields, media and psi fill the scalar registers and
// spill (130 of them)
template <class G>
__device__ __forceinline__ const G &reread(const G &g) {
  const G *p = &g;
  asm volatile("" : "+s"(p));
  return *p;
}

// The TF/SF faces crossing the vector's cells on one plane (tile_nodal's
// header comment says how faces are held): the plane's mask, and the first
// face's term of each cell and component, loaded with the plane.
struct QuadFaces {
  unsigned mz;
  float t[3][4];
};
template <class PS>
__device__ __forceinline__ bool quad_faces(const PS &x, const FaceAddr *fal, const unsigned (&col)[4],
                                           int i0, int j, int k, QuadFaces &o) {
  o.mz = ro_uniform_u(x.mz, k);
  if (!((col[0] | col[1] | col[2] | col[3]) & o.mz)) return false;
  const float *terms = x.terms;
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const unsigned b = col[c] & o.mz & x.cm[q];
      if (b) o.t[q][c] = terms[term_index(fal, __builtin_ctz(b), i0 + c, j, k)];
    }
  return true;
}
// component q's faces onto the four cells, in the reference's order
template <class S, class PS>
__device__ __forceinline__ void quad_add(const PS &x, const FaceAddr *fal, const QuadFaces &o,
                                         const unsigned (&col)[4], int q, int i0, int j, int k, float s,
                                         float is, float (&r)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const unsigned b = col[c] & o.mz & x.cm[q];
    if (b) r[c] = add_faces<S>(b, o.t[q][c], fal, x.terms, i0 + c, j, k, r[c], s, is);
  }
}
// the faces of the vector's column, per cell (none past the sweep)
template <class PS>
__device__ __forceinline__ void quad_col(const PS &x, int i0, int j, int nx, unsigned (&col)[4]) {
  const unsigned my = ((const SFD_GLOBAL unsigned *)x.my)[j];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const unsigned m = ((const SFD_GLOBAL unsigned *)x.mx)[min(i0 + c, nx)];
    col[c] = i0 + c <= nx ? m & my : 0u;
  }
}

// one tile of the E face pass.  CPML: the slabs it may meet.  UNI: every cell of the tile holds the medium
// whose coefficients are cu (else tab's).
// X: the TF/SF faces of xs are applied before each store (fal: their
// addresses in LDS).
template <int CPML, bool UNI, bool X, class T, class G, class PS>
__device__ __forceinline__ void equad_tile(const G &g, const MedTab &tab, float2 cu,
                                           const QuadPos &at, const PS &xs_,
                                           const FaceAddr *fal) {
  typedef Quad<T> V;
  typedef Store<T> S;
  typedef typename V::raw raw;
  typedef const SFD_GLOBAL float *cgf;
  constexpr unsigned ES = sizeof(T);
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int i0 = at.i0, j = at.j, k0 = at.k0, k1 = at.k1;
  const long long fpb = g.pxy * ES, mpb = g.pxy * 2;   // plane strides, bytes
  const unsigned lo = (unsigned)((j + 1) * (int)g.px + g.xoff + i0);
  const unsigned of = lo * ES, om = lo * 2u, fy = (unsigned)g.px * ES;
  // the x - 1 neighbours that no lane to the left holds
  const bool edge = threadIdx.x == 0 || at.first;
  const bool cy = j < ny;
  const int nxc = nx - i0, nxn = nx + 1 - i0;   // cells inside i < nx, i <= nx
  const float idyh_ = ((cgf)g.id[4])[j + 1];
  float idxh[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) idxh[c] = ((cgf)g.id[3])[min(i0 + c, nx) + 1];
  XSlab xs{0, 0, 0};
  int qyn = 0;
  bool syn = false;
  float by = 0.0f, ccy = 0.0f, bx[4] = {}, ccx[4] = {};
  const int Lx = g.L[0][0] + g.L[0][1], Ly = g.L[1][0] + g.L[1][1];
  if (CPML & kSlabX) {
    xs = x_slab(i0, g.L[0][0], g.L[0][1], nx - g.L[0][1] + 1, nx);
    if (xs.n > xs.a) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        bx[c] = ((cgf)g.pbe[0])[min(i0 + c, nx) + 1];
        ccx[c] = ((cgf)g.pce[0])[min(i0 + c, nx) + 1];
      }
    }
  }
  if (CPML & kSlabY) {
    syn = slab_node(j, ny, g.L[1][0], g.L[1][1], qyn);
    if (syn) { by = ((cgf)g.pbe[1])[j + 1]; ccy = ((cgf)g.pce[1])[j + 1]; }
  }
  const bool sxn = (CPML & kSlabX) && xs.n > xs.a;
  // byte offsets of the vector in the slab planes (see epass_tile); the x
  // slabs' bases lie four values early
  const unsigned oA = (unsigned)(qyn * nx + i0) * 4u;         // psi_Exy
  const unsigned oB = (unsigned)(j * nx + i0) * 4u;           // psi_Exz
  const unsigned oC = (unsigned)(j * (nx + 1) + i0) * 4u;     // psi_Eyz
  const unsigned oD = (unsigned)(j * Lx + xs.q + 4) * 4u;     // psi_Eyx, psi_Ezx
  const unsigned oE = (unsigned)(qyn * (nx + 1) + i0) * 4u;   // psi_Ezy
  float hxk[4], hyk[4];   // plane k - 1 of Hx, Hy
  {
    const long long kb = (long long)k0 * fpb;
    const raw rx = ldq<T>(plane_base((char *)g.f[3], kb), of), ry = ldq<T>(plane_base((char *)g.f[4], kb), of);
    V::cvt(rx, g.fs[3], hxk);
    V::cvt(ry, g.fs[4], hyk);
  }
  unsigned col[4] = {};
  if (X) quad_col(xs_, i0, j, nx, col);
  for (int k = k0; k < k1; ++k) {
    const G &p = CPML == kSlabAll || X ? reread(g) : g;
    const bool cz = k < nz;
    const long long kb = (long long)(k + 1) * fpb, kmb = (long long)(k + 1) * mpb;
    // ---- issue every load of this plane
    const float idzh_ = ro_uniform(p.id[5], k + 1);
    const SFD_GLOBAL char *hxp = plane_base((char *)p.f[3], kb), *hyp = plane_base((char *)p.f[4], kb),
                          *hzp = plane_base((char *)p.f[5], kb);
    SFD_GLOBAL char *const exp = plane_base((char *)p.f[0], kb), *const eyp = plane_base((char *)p.f[1], kb),
                         *const ezp = plane_base((char *)p.f[2], kb);
    const raw rhx = ldq<T>(hxp, of), rhy = ldq<T>(hyp, of), rhz = ldq<T>(hzp, of);
    const raw rhzj = ldq<T>(hzp, of - fy), rhxj = ldq<T>(hxp, of - fy);
    const raw rex = ldq<T>(exp, of), rey = ldq<T>(eyp, of), rez = ldq<T>(ezp, of);
    u32x2 mx{}, my{}, mz{};
    if (!UNI) {
      mx = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[0], kmb), om);
      my = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[1], kmb), om);
      mz = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[2], kmb), om);
    }
    typename S::raw_t rhze = 0, rhye = 0;
    if (edge) { rhze = S::ldr(hzp, of - ES); rhye = S::ldr(hyp, of - ES); }
    int qzn = 0;
    const bool szn = (CPML & kSlabZ) && slab_node(k, nz, p.L[2][0], p.L[2][1], qzn);
    float bzp = 0.0f, ccz = 0.0f;
    float vxy[4], vxz[4], vyz[4], vyx[4], vzy[4], vzx[4];   // (used where loaded)
    SFD_GLOBAL float *sExy = nullptr, *sExz = nullptr, *sEyz = nullptr, *sEyx = nullptr,
                     *sEzy = nullptr, *sEzx = nullptr;
    if (CPML) {
      if (szn) {
        bzp = ro_uniform(p.pbe[2], k + 1);
        ccz = ro_uniform(p.pce[2], k + 1);
        sExz = plane_base((float *)p.psi[PSI_EXZ], (long long)qzn * (ny + 1) * nx);
        sEyz = plane_base((float *)p.psi[PSI_EYZ], (long long)qzn * ny * (nx + 1));
        ld_psi(sExz, oB, vxz);
        if (cy) ld_psi(sEyz, oC, vyz);
      }
      if ((CPML & kSlabY) && Ly) {
        sExy = plane_base((float *)p.psi[PSI_EXY], (long long)k * Ly * nx);
        sEzy = plane_base((float *)p.psi[PSI_EZY], (long long)k * Ly * (nx + 1));
        if (syn) {
          ld_psi(sExy, oA, vxy);
          if (cz) ld_psi(sEzy, oE, vzy);
        }
      }
      if ((CPML & kSlabX) && Lx) {
        sEyx = plane_base((float *)p.psi[PSI_EYX], (long long)k * ny * Lx - 4);
        sEzx = plane_base((float *)p.psi[PSI_EZX], (long long)k * (ny + 1) * Lx - 4);
        if (sxn) {
          if (cy) ld_psi(sEyx, oD, vyx);
          if (cz) ld_psi(sEzx, oD, vzx);
        }
      }
    }
    QuadFaces fc;
    const bool fx = X && quad_faces(xs_, fal, col, i0, j, k, fc);
    // ---- compute
    if (CPML || X) plane_wait();
    float hx[4], hy[4], hz[4], d0[4], d1[4], f[4], r[4], g2[4];
    V::cvt(rhx, p.fs[3], hx);
    V::cvt(rhy, p.fs[4], hy);
    V::cvt(rhz, p.fs[5], hz);
    const float hzl = from_left(hz[3], 0.0f), hyl = from_left(hy[3], 0.0f);
    const float hze = edge ? S::cvt(rhze, p.fs[5]) : hzl, hye = edge ? S::cvt(rhye, p.fs[4]) : hyl;
    const float dzx[4] = {hz[0] - hze, hz[1] - hz[0], hz[2] - hz[1], hz[3] - hz[2]};
    const float dyx[4] = {hy[0] - hye, hy[1] - hy[0], hy[2] - hy[1], hy[3] - hy[2]};
    const float idyh[4] = SFD_ALL4(idyh_), idzh[4] = SFD_ALL4(idzh_);
    const float by4[4] = SFD_ALL4(by), ccy4[4] = SFD_ALL4(ccy);
    const float bz4[4] = SFD_ALL4(bzp), ccz4[4] = SFD_ALL4(ccz);
    {  // Ex: x[0,nx-1] y[0,ny] z[0,nz]
      V::cvt(rhzj, p.fs[5], d0);
#pragma unroll
      for (int c = 0; c < 4; ++c) { d0[c] = hz[c] - d0[c]; d1[c] = hy[c] - hyk[c]; }
      V::cvt(rex, p.fs[0], f);
      yee4<UNI>(tab, cu, mx, f, d0, idyh, d1, idzh, r, g2);
      if (CPML) {
        if (syn) psi4<true, false>(sExy, oA, vxy, d0, ccy4, by4, g2, 0, nxc, r);
        if (szn) psi4<true, true>(sExz, oB, vxz, d1, ccz4, bz4, g2, 0, nxc, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 0, i0, j, k, p.fs[0], p.fi[0], r);
      st_at((SFD_GLOBAL raw *)exp, of, V::pack(r, p.fi[0], rex, nxc));
    }
    {  // Ey: x[0,nx] y[0,ny-1] z[0,nz]
#pragma unroll
      for (int c = 0; c < 4; ++c) d0[c] = hx[c] - hxk[c];
      V::cvt(rey, p.fs[1], f);
      yee4<UNI>(tab, cu, my, f, d0, idzh, dzx, idxh, r, g2);
      if (CPML && cy) {
        if (szn) psi4<true, false>(sEyz, oC, vyz, d0, ccz4, bz4, g2, 0, nxn, r);
        if (sxn) psi4<false, true>(sEyx, oD, vyx, dzx, ccx, bx, g2, xs.a, xs.n, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 1, i0, j, k, p.fs[1], p.fi[1], r);
      if (cy) st_at((SFD_GLOBAL raw *)eyp, of, V::pack(r, p.fi[1], rey, nxn));
    }
    {  // Ez: x[0,nx] y[0,ny] z[0,nz-1]
      V::cvt(rhxj, p.fs[3], d1);
#pragma unroll
      for (int c = 0; c < 4; ++c) d1[c] = hx[c] - d1[c];
      V::cvt(rez, p.fs[2], f);
      yee4<UNI>(tab, cu, mz, f, dyx, idxh, d1, idyh, r, g2);
      if (CPML && cz) {
        if (syn) psi4<true, true>(sEzy, oE, vzy, d1, ccy4, by4, g2, 0, nxn, r);
        if (sxn) psi4<false, false>(sEzx, oD, vzx, dyx, ccx, bx, g2, xs.a, xs.n, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 2, i0, j, k, p.fs[2], p.fi[2], r);
      if (cz) st_at((SFD_GLOBAL raw *)ezp, of, V::pack(r, p.fi[2], rez, nxn));
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) { hxk[c] = hx[c]; hyk[c] = hy[c]; }
  }
}

// one tile of the H face pass
template <int CPML, bool UNI, bool X, class T, class G, class PS>
__device__ __forceinline__ void hquad_tile(const G &g, const MedTab &tab, float2 cu,
                                           const QuadPos &at, const PS &xs_,
                                           const FaceAddr *fal) {
  typedef Quad<T> V;
  typedef Store<T> S;
  typedef typename V::raw raw;
  typedef const SFD_GLOBAL float *cgf;
  constexpr unsigned ES = sizeof(T);
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const int i0 = at.i0, j = at.j, k0 = at.k0, k1 = at.k1;
  const long long fpb = g.pxy * ES, mpb = g.pxy * 2;
  const unsigned lo = (unsigned)((j + 1) * (int)g.px + g.xoff + i0);
  const unsigned of = lo * ES, om = lo * 2u, fy = (unsigned)g.px * ES;
  // the x + 1 neighbours that no lane to the right holds (the last vector of
  // a grid's row needs none: its cells with i < nx have theirs in the vector)
  const bool edge = threadIdx.x == kWave - 1 || at.last;
  const bool cy = j < ny;
  const int nxc = nx - i0, nxn = nx + 1 - i0;
  const float idye_ = ((cgf)g.id[1])[j + 1];
  float idxe[4];
#pragma unroll
  for (int c = 0; c < 4; ++c) idxe[c] = ((cgf)g.id[0])[min(i0 + c, nx) + 1];
  XSlab xs{0, 0, 0};
  int qyc = 0;
  bool syc = false;
  float by = 0.0f, ccy = 0.0f, bx[4] = {}, ccx[4] = {};
  const int Lx = g.L[0][0] + g.L[0][1], Ly = g.L[1][0] + g.L[1][1];
  if (CPML & kSlabX) {
    xs = x_slab(i0, g.L[0][0], g.L[0][1], nx - g.L[0][1], nx - 1);
    if (xs.n > xs.a) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        bx[c] = ((cgf)g.pbm[0])[min(i0 + c, nx) + 1];
        ccx[c] = ((cgf)g.pcm[0])[min(i0 + c, nx) + 1];
      }
    }
  }
  if (CPML & kSlabY) {
    syc = cy && slab_cell(j, ny, g.L[1][0], g.L[1][1], qyc);
    if (syc) { by = ((cgf)g.pbm[1])[j + 1]; ccy = ((cgf)g.pcm[1])[j + 1]; }
  }
  const bool sxc = (CPML & kSlabX) && xs.n > xs.a;
  const unsigned oA = (unsigned)(qyc * (nx + 1) + i0) * 4u;   // psi_Hxy
  const unsigned oB = (unsigned)(j * (nx + 1) + i0) * 4u;     // psi_Hxz
  const unsigned oC = (unsigned)(j * nx + i0) * 4u;           // psi_Hyz
  const unsigned oD = (unsigned)(j * Lx + xs.q + 4) * 4u;     // psi_Hyx, psi_Hzx
  const unsigned oE = (unsigned)(qyc * nx + i0) * 4u;         // psi_Hzy
  float ex[4], ey[4];   // plane k of Ex, Ey
  {
    const long long kb = (long long)(k0 + 1) * fpb;
    const raw rx = ldq<T>(plane_base((char *)g.f[0], kb), of), ry = ldq<T>(plane_base((char *)g.f[1], kb), of);
    V::cvt(rx, g.fs[0], ex);
    V::cvt(ry, g.fs[1], ey);
  }
  unsigned col[4] = {};
  if (X) quad_col(xs_, i0, j, nx, col);
  for (int k = k0; k < k1; ++k) {
    const G &p = CPML == kSlabAll || X ? reread(g) : g;
    const bool cz = k < nz;
    const long long kb = (long long)(k + 1) * fpb, kmb = (long long)(k + 1) * mpb;
    const float idze_ = ro_uniform(p.id[2], k + 1);
    const SFD_GLOBAL char *exn = plane_base((char *)p.f[0], kb + fpb), *eyn = plane_base((char *)p.f[1], kb + fpb);
    const SFD_GLOBAL char *exp = plane_base((char *)p.f[0], kb), *eyp = plane_base((char *)p.f[1], kb),
                          *ezp = plane_base((char *)p.f[2], kb);
    SFD_GLOBAL char *const hxp = plane_base((char *)p.f[3], kb), *const hyp = plane_base((char *)p.f[4], kb),
                         *const hzp = plane_base((char *)p.f[5], kb);
    const raw rexk = ldq<T>(exn, of), reyk = ldq<T>(eyn, of), rez = ldq<T>(ezp, of);
    const raw rezj = ldq<T>(ezp, of + fy), rexj = ldq<T>(exp, of + fy);
    const raw rhx = ldq<T>(hxp, of), rhy = ldq<T>(hyp, of), rhz = ldq<T>(hzp, of);
    u32x2 mx{}, my{}, mz{};
    if (!UNI) {
      mx = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[3], kmb), om);
      my = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[4], kmb), om);
      mz = ld_at((const SFD_GLOBAL u32x2 *)plane_base((const char *)p.mi[5], kmb), om);
    }
    typename S::raw_t reze = 0, reye = 0;
    if (edge) { reze = S::ldr(ezp, of + 4 * ES); reye = S::ldr(eyp, of + 4 * ES); }
    int qzc = 0;
    const bool szc = (CPML & kSlabZ) && cz && slab_cell(k, nz, p.L[2][0], p.L[2][1], qzc);
    float bzp = 0.0f, ccz = 0.0f;
    float vxy[4], vxz[4], vyz[4], vyx[4], vzy[4], vzx[4];   // (used where loaded)
    SFD_GLOBAL float *sHxy = nullptr, *sHxz = nullptr, *sHyz = nullptr, *sHyx = nullptr,
                     *sHzy = nullptr, *sHzx = nullptr;
    if (CPML) {
      if (szc) {
        bzp = ro_uniform(p.pbm[2], k + 1);
        ccz = ro_uniform(p.pcm[2], k + 1);
        sHxz = plane_base((float *)p.psi[PSI_HXZ], (long long)qzc * ny * (nx + 1));
        sHyz = plane_base((float *)p.psi[PSI_HYZ], (long long)qzc * (ny + 1) * nx);
        if (cy) ld_psi(sHxz, oB, vxz);
        ld_psi(sHyz, oC, vyz);
      }
      if ((CPML & kSlabY) && Ly) {
        sHxy = plane_base((float *)p.psi[PSI_HXY], (long long)k * Ly * (nx + 1));
        sHzy = plane_base((float *)p.psi[PSI_HZY], (long long)k * Ly * nx);
        if (syc) {
          if (cz) ld_psi(sHxy, oA, vxy);
          ld_psi(sHzy, oE, vzy);
        }
      }
      if ((CPML & kSlabX) && Lx) {
        sHyx = plane_base((float *)p.psi[PSI_HYX], (long long)k * (ny + 1) * Lx - 4);
        sHzx = plane_base((float *)p.psi[PSI_HZX], (long long)k * ny * Lx - 4);
        if (sxc) {
          if (cz) ld_psi(sHyx, oD, vyx);
          if (cy) ld_psi(sHzx, oD, vzx);
        }
      }
    }
    QuadFaces fc;
    const bool fx = X && quad_faces(xs_, fal, col, i0, j, k, fc);
    // ---- compute
    if (CPML || X) plane_wait();
    float exk[4], eyk[4], ez[4], d0[4], d1[4], f[4], r[4], g2[4];
    V::cvt(rexk, p.fs[0], exk);
    V::cvt(reyk, p.fs[1], eyk);
    V::cvt(rez, p.fs[2], ez);
    const float ezr = from_right(ez[0]), eyr = from_right(ey[0]);
    const float eze = edge ? S::cvt(reze, p.fs[2]) : ezr, eye = edge ? S::cvt(reye, p.fs[1]) : eyr;
    const float dzx[4] = {ez[1] - ez[0], ez[2] - ez[1], ez[3] - ez[2], eze - ez[3]};
    const float dyx[4] = {ey[1] - ey[0], ey[2] - ey[1], ey[3] - ey[2], eye - ey[3]};
    const float idye[4] = SFD_ALL4(idye_), idze[4] = SFD_ALL4(idze_);
    const float by4[4] = SFD_ALL4(by), ccy4[4] = SFD_ALL4(ccy);
    const float bz4[4] = SFD_ALL4(bzp), ccz4[4] = SFD_ALL4(ccz);
    {  // Hx: x[0,nx] y[0,ny-1] z[0,nz-1]
      V::cvt(rezj, p.fs[2], d1);
#pragma unroll
      for (int c = 0; c < 4; ++c) { d0[c] = eyk[c] - ey[c]; d1[c] = d1[c] - ez[c]; }
      V::cvt(rhx, p.fs[3], f);
      yee4<UNI>(tab, cu, mx, f, d0, idze, d1, idye, r, g2);
      if (CPML && cy && cz) {
        if (syc) psi4<true, true>(sHxy, oA, vxy, d1, ccy4, by4, g2, 0, nxn, r);
        if (szc) psi4<true, false>(sHxz, oB, vxz, d0, ccz4, bz4, g2, 0, nxn, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 0, i0, j, k, p.fs[3], p.fi[3], r);
      if (cy && cz) st_at((SFD_GLOBAL raw *)hxp, of, V::pack(r, p.fi[3], rhx, nxn));
    }
    {  // Hy: x[0,nx-1] y[0,ny] z[0,nz-1]
#pragma unroll
      for (int c = 0; c < 4; ++c) d1[c] = exk[c] - ex[c];
      V::cvt(rhy, p.fs[4], f);
      yee4<UNI>(tab, cu, my, f, dzx, idxe, d1, idze, r, g2);
      if (CPML && cz) {
        if (szc) psi4<true, true>(sHyz, oC, vyz, d1, ccz4, bz4, g2, 0, nxc, r);
        if (sxc) psi4<false, false>(sHyx, oD, vyx, dzx, ccx, bx, g2, xs.a, xs.n, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 1, i0, j, k, p.fs[4], p.fi[4], r);
      if (cz) st_at((SFD_GLOBAL raw *)hyp, of, V::pack(r, p.fi[4], rhy, nxc));
    }
    {  // Hz: x[0,nx-1] y[0,ny-1] z[0,nz]
      V::cvt(rexj, p.fs[0], d0);
#pragma unroll
      for (int c = 0; c < 4; ++c) d0[c] = d0[c] - ex[c];
      V::cvt(rhz, p.fs[5], f);
      yee4<UNI>(tab, cu, mz, f, d0, idye, dyx, idxe, r, g2);
      if (CPML && cy) {
        if (syc) psi4<true, false>(sHzy, oE, vzy, d0, ccy4, by4, g2, 0, nxc, r);
        if (sxc) psi4<false, true>(sHzx, oD, vzx, dyx, ccx, bx, g2, xs.a, xs.n, r);
      }
      if (X && fx) quad_add<S>(xs_, fal, fc, col, 2, i0, j, k, p.fs[5], p.fi[5], r);
      if (cy) st_at((SFD_GLOBAL raw *)hzp, of, V::pack(r, p.fi[5], rhz, nxc));
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) { ex[c] = exk[c]; ey[c] = eyk[c]; }
  }
}
#undef SFD_ALL4

}  // namespace SFD_NS
}  // namespace sfd
