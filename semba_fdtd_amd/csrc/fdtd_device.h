// fdtd_device.h -- device code the kernel files share: tile decoding, the
// update arithmetic, the media tables in LDS, plane addressing, field storage,
// and the sources a face pass applies inline.  Compiled once per arithmetic
// mode (SFD_NS = fast or exact, see fdtd_kernels.hip).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include "fdtd_internal.h"

#ifndef SFD_NS
#error "compile with -DSFD_NS=fast or -DSFD_NS=exact"
#endif
#ifndef SFD_EXACT
#define SFD_EXACT 0
#endif

namespace sfd {
namespace SFD_NS {


// pole states prefetched into registers per edge: one Lorentz pair is two
// complex(8) states in EXACT and one folded complex64 state in FAST
#if SFD_EXACT
typedef double2 jstate_t;  // complex(8) pole state, reference layout
typedef double coef_t;
constexpr int kPre = 2;
#else
typedef float2 jstate_t;   // complex64 state, conjugate pairs folded
typedef float coef_t;
#ifndef SFD_PREFETCH_POLES
#define SFD_PREFETCH_POLES 1
#endif
constexpr int kPre = SFD_PREFETCH_POLES;
#endif

// global memory, spelled out for the pointers the compiler cannot infer it
// for (those read out of memory rather than passed as kernel arguments)
#define SFD_GLOBAL __attribute__((address_space(1)))

// hardware dispatches block b to XCD b % 8; give each XCD one contiguous
// range of tiles so that x/y neighbours share that XCD's L2
__device__ __forceinline__ int xcd_remap(int b, int nblk) {
  const int q = nblk >> 3, r = nblk & 7;
  const int xcd = b & 7, loc = b >> 3;
  return (xcd < r) ? xcd * (q + 1) + loc : r * (q + 1) + (xcd - r) * q + loc;
}

__device__ __forceinline__ void decode_tile(const TileMap &tm, int b, int &bx, int &by,
                                            int &bz) {
  if (tm.remap) b = xcd_remap(b, tm.nblk);
  bx = b % tm.tx;
  b /= tm.tx;
  by = b % tm.ty;
  bz = b / tm.ty;
}

// slab coordinate along a stretched axis.  "node" axes hold n+1 positions
// (tangential E, normal H), "cell" axes n.  High slabs start after the
// interior: node n-Lhi+1, cell n-Lhi (borderscpml.F90:149-193).
__device__ __forceinline__ bool slab_node(int c, int n, int L0, int L1, int &q) {
  if (c < L0) { q = c; return true; }
  const int hs = n - L1 + 1;
  if (c >= hs) { q = L0 + (c - hs); return true; }
  return false;
}
__device__ __forceinline__ bool slab_cell(int c, int n, int L0, int L1, int &q) {
  if (c < L0) { q = c; return true; }
  const int hs = n - L1;
  if (c >= hs) { q = L0 + (c - hs); return true; }
  return false;
}

// The update arithmetic.  EXACT: plain products and sums (the file is built
// without contraction), the reference's order.  FAST: explicit fused
// multiply-adds, so that every variant of a pass (one or four cells per lane,
// one grid or a batch) rounds the same way and gives the same bits.
// a*ia - b*ib
__device__ __forceinline__ float curl2(float a, float ia, float b, float ib) {
#if SFD_EXACT
  return a * ia - b * ib;
#else
  return __builtin_fmaf(a, ia, -(b * ib));
#endif
}
// g1*f + g2*cu
__device__ __forceinline__ float yee_upd(float g1, float f, float g2, float cu) {
#if SFD_EXACT
  return g1 * f + g2 * cu;
#else
  return __builtin_fmaf(g1, f, g2 * cu);
#endif
}
// x + g*v
__device__ __forceinline__ float madd(float x, float g, float v) {
#if SFD_EXACT
  return x + g * v;
#else
  return __builtin_fmaf(g, v, x);
#endif
}

// per-medium tables staged in LDS (TBL) or read from global memory
struct MedTab {
  const float2 *gg;     // {G1,G2} or {GM1,GM2}
  const int *slot;      // dispersive slot per medium (-1: not dispersive)
  const int *anp;       // stored poles per slot
  const coef_t *acf;    // per slot per pole {kr,ki,br,bi,g3r,g3i}
};

__device__ __forceinline__ const coef_t *ade_coefs(const AdeSet &ad) {
#if SFD_EXACT
  return ad.aded;
#else
  return ad.adef;
#endif
}

// LDS layout: gg[nm+1] | slot[nm+1] | anp[ndisp] | (8-byte aligned) acf.
// ad: the pole state whose tables are staged (ADE only).
template <bool TBL, bool ADE>
__device__ __forceinline__ MedTab stage_tables(const DevGrid &g, const float *a,
                                               const float *b, float2 *lds,
                                               const AdeSet *ad = nullptr) {
  MedTab t;
  const int nm = g.nmedia;
  if (TBL) {
    int *ls = reinterpret_cast<int *>(lds + (nm + 1));
    int *lnp = ls + (nm + 1);
    const int nd = ADE ? ad->ndisp : 0;
    const size_t off = ((size_t)(nm + 1) * 12 + (size_t)nd * 4 + 7) & ~(size_t)7;
    coef_t *lcf = reinterpret_cast<coef_t *>(reinterpret_cast<char *>(lds) + off);
    const int tid = threadIdx.y * blockDim.x + threadIdx.x;
    const int nt = blockDim.x * blockDim.y;
    for (int m = tid; m <= nm; m += nt) {
      lds[m] = make_float2(a[m], b[m]);
      if (ADE) ls[m] = nd ? ad->dslot[m] : -1;
    }
    if (ADE) {
      const coef_t *cf = ade_coefs(*ad);
      for (int d = tid; d < nd; d += nt) lnp[d] = ad->anp[d];
      for (int q = tid; q < nd * kPMax * 6; q += nt) lcf[q] = cf[q];
    }
    __syncthreads();
    t.gg = lds;
    t.slot = ls;
    t.anp = lnp;
    t.acf = lcf;
  } else {
    t.gg = nullptr;
    t.slot = ADE ? ad->dslot : nullptr;
    t.anp = ADE ? ad->anp : nullptr;
    t.acf = ADE ? ade_coefs(*ad) : nullptr;
  }
  return t;
}

// the coefficient pairs of one field alone
__device__ __forceinline__ MedTab stage_pair(int nmedia, const float *a, const float *b,
                                             float2 *lds) {
  const int tid = threadIdx.y * blockDim.x + threadIdx.x, nt = blockDim.x * blockDim.y;
  for (int m = tid; m <= nmedia; m += nt) lds[m] = make_float2(a[m], b[m]);
  __syncthreads();
  return MedTab{lds, nullptr, nullptr, nullptr};
}

template <bool TBL>
__device__ __forceinline__ float2 coef(const MedTab &t, const float *a, const float *b, int m) {
  if (TBL) return t.gg[m];
  return make_float2(a[m], b[m]);
}

// Loads and stores of the march address a plane through a base pointer that
// is the same for every lane (scalar registers) plus the lane's byte offset
// inside the plane (one 32-bit register).  The plane base is made opaque to
// the compiler, which otherwise hoists a 64-bit (array base + offset) pair per
// array and lane out of the march; it stays in the global address space so
// that the accesses are global, not flat, loads and stores.
template <class T>
__device__ __forceinline__ SFD_GLOBAL T *plane_base(T *base, long long P) {
  SFD_GLOBAL T *q = (SFD_GLOBAL T *)(base + P);
  asm volatile("" : "+s"(q));
  return q;
}
template <class T>
__device__ __forceinline__ T ld_at(const SFD_GLOBAL T *base, unsigned ob) {
  return *reinterpret_cast<const SFD_GLOBAL T *>(reinterpret_cast<const SFD_GLOBAL char *>(base) +
                                                 ob);
}
template <class T>
__device__ __forceinline__ void st_at(SFD_GLOBAL T *base, unsigned ob, T v) {
  *reinterpret_cast<SFD_GLOBAL T *>(reinterpret_cast<SFD_GLOBAL char *>(base) + ob) = v;
}

// an element of a table the kernel never writes, at an index the same for
// every lane: read through the constant address space, i.e. by a scalar load
// that does not join the vector-memory counter shared with the stores
__device__ __forceinline__ float ro_uniform(const float *t, int idx) {
  return ((const __attribute__((address_space(4))) float *)t)[idx];
}
__device__ __forceinline__ int ro_uniform_i(const int *t, int idx) {
  return ((const __attribute__((address_space(4))) int *)t)[idx];
}
__device__ __forceinline__ unsigned ro_uniform_u(const unsigned *t, int idx) {
  return ((const __attribute__((address_space(4))) unsigned *)t)[idx];
}

// Field storage of the face passes: each field array holds fp32 values, or
// binary16 values with a per-array scale.
template <class T> struct Store;
// fp32 fields: plain 16-byte vectors (the scale arguments are unused)
template <> struct Store<float> {
  static __device__ __forceinline__ float ld1(const float *b, long long p, float) { return b[p]; }
  static __device__ __forceinline__ void st1(float *b, long long p, float, float v) { b[p] = v; }
  static __device__ __forceinline__ float ld1(const SFD_GLOBAL float *b, long long p, float) {
    return b[p];
  }
  static __device__ __forceinline__ void st1(SFD_GLOBAL float *b, long long p, float, float v) {
    b[p] = v;
  }
  // a plane base and the lane's byte offset in the plane; ldr/cvt split the
  // load from the conversion so that a plane's loads all issue first
  typedef float raw_t;
  static __device__ __forceinline__ raw_t ldr(const SFD_GLOBAL char *b, unsigned ob) {
    return ld_at((const SFD_GLOBAL float *)b, ob);
  }
  static __device__ __forceinline__ float cvt(raw_t r, float) { return r; }
  static __device__ __forceinline__ float ldo(const SFD_GLOBAL char *b, unsigned ob, float) {
    return ld_at((const SFD_GLOBAL float *)b, ob);
  }
  static __device__ __forceinline__ void sto(SFD_GLOBAL char *b, unsigned ob, float, float v) {
    st_at((SFD_GLOBAL float *)b, ob, v);
  }
  // a value as it reads back after being stored by a pass, and by a source
  static __device__ __forceinline__ float trip(float v, float, float) { return v; }
  static __device__ __forceinline__ float trip_src(float v, float, float) { return v; }
  static __device__ __forceinline__ void st_src(float *b, long long p, float, float v) { b[p] = v; }
};
// binary16 fields with a per-array scale: value = half * s, stored as
// round(value / s); 8-byte vectors, fp32 arithmetic.  Every scale product is
// rounded to fp32 on its own (an empty asm barrier keeps the compiler from
// fusing it into the arithmetic that uses it, or into the conversion to
// binary16 as a mixed-precision FMA, which would round once instead of
// twice), so every kernel shape rounds alike.
__device__ __forceinline__ float rounded(float x) {
  asm("" : "+v"(x));
  return x;
}
// A source launch of its own (fdtd_aux.hip) stores half(value / s) through the
// mixed-precision FMA, one rounding; a source inside a pass stores the same.
// (The result is read two cycles later: a partial register write.)
__device__ __forceinline__ unsigned short half_src(float v, float is) {
  unsigned r;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0\n\ts_nop 1" : "=v"(r) : "v"(is), "v"(v));
  return (unsigned short)r;
}
template <> struct Store<__half> {
  static __device__ __forceinline__ float ld1(const float *b, long long p, float s) {
    return rounded(__half2float(reinterpret_cast<const __half *>(b)[p]) * s);
  }
  static __device__ __forceinline__ void st1(float *b, long long p, float is, float v) {
    reinterpret_cast<__half *>(b)[p] = __float2half_rn(rounded(v * is));
  }
  static __device__ __forceinline__ float ld1(const SFD_GLOBAL float *b, long long p, float s) {
    const unsigned short h = ((const SFD_GLOBAL unsigned short *)b)[p];
    return rounded(__half2float(__ushort_as_half(h)) * s);
  }
  static __device__ __forceinline__ void st1(SFD_GLOBAL float *b, long long p, float is, float v) {
    ((SFD_GLOBAL unsigned short *)b)[p] = __half_as_ushort(__float2half_rn(rounded(v * is)));
  }
  typedef unsigned short raw_t;
  static __device__ __forceinline__ raw_t ldr(const SFD_GLOBAL char *b, unsigned ob) {
    return ld_at((const SFD_GLOBAL unsigned short *)b, ob);
  }
  static __device__ __forceinline__ float cvt(raw_t h, float s) {
    return rounded(__half2float(__ushort_as_half(h)) * s);
  }
  static __device__ __forceinline__ float ldo(const SFD_GLOBAL char *b, unsigned ob, float s) {
    return cvt(ldr(b, ob), s);
  }
  static __device__ __forceinline__ void sto(SFD_GLOBAL char *b, unsigned ob, float is, float v) {
    st_at((SFD_GLOBAL unsigned short *)b, ob, __half_as_ushort(__float2half_rn(rounded(v * is))));
  }
  static __device__ __forceinline__ float trip(float v, float s, float is) {
    return cvt(__half_as_ushort(__float2half_rn(rounded(v * is))), s);
  }
  static __device__ __forceinline__ float trip_src(float v, float s, float is) {
    return cvt(half_src(v, is), s);
  }
  static __device__ __forceinline__ void st_src(float *b, long long p, float is, float v) {
    reinterpret_cast<unsigned short *>(b)[p] = half_src(v, is);
  }
};

// 16-byte and 8-byte vectors as the compiler's own vector types (these load
// and store through global-address-space pointers)
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x4 v4(float a, float b, float c, float d) {
  f32x4 r;
  r.x = a; r.y = b; r.z = c; r.w = d;
  return r;
}

// lane l receives lane l - 1's v (wave_shr:1); lane 0 receives first
__device__ __forceinline__ float from_left(float v, float first) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, first),
                                                               __builtin_bit_cast(int, v), 0x138,
                                                               0xf, 0xf, false));
}
// lane l receives lane l + 1's v (wave_shl:1); lane 63 receives 0
__device__ __forceinline__ float from_right(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                               0x130, 0xf, 0xf, false));
}

// ---- batches of independent grids
// a tile map read word by word through the constant address space (scalar
// loads; the maps never change during a launch)
__device__ __forceinline__ TileMap const_tilemap(const TileMap *t) {
  static_assert(sizeof(TileMap) % sizeof(int) == 0, "TileMap holds ints only");
  typedef const __attribute__((address_space(4))) int CInt;
  TileMap m;
  int *o = reinterpret_cast<int *>(&m);
  for (int q = 0; q < (int)(sizeof(TileMap) / sizeof(int)); ++q) o[q] = ((CInt *)t)[q];
  return m;
}

__device__ __forceinline__ int batch_grid(const int *start, int ngrid, int t) {
  int lo = 0, hi = ngrid - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= t) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The column (i, j) of the tile's lane and the tile's z chunk bz.  Tiles are
// 64-wide x segments of blockDim.y rows, or, in flat tile maps, runs of
// 64 * blockDim.y consecutive columns of the x-y plane in x-fastest order
// (grids whose nx + 1 is far from a multiple of 64 then leave no lane idle;
// every neighbour of the face passes comes from memory, so a run may wrap
// from one row to the next).  j > ny marks a lane past the plane.
__device__ __forceinline__ void tile_column(const TileMap &tm, int blk, int nx, int &i, int &j,
                                            int &bz) {
  int bx, by;
  decode_tile(tm, blk, bx, by, bz);
  if (tm.flat) {
    const int f = bx * kWave * (int)blockDim.y + (int)threadIdx.y * kWave + (int)threadIdx.x;
    i = f % (nx + 1);
    j = f / (nx + 1);
  } else {
    i = bx * kWave + threadIdx.x;
    j = by * blockDim.y + threadIdx.y;
  }
}

// The sources a pass applies inline (PassSrc; CPassSrc read through the
// constant address space).  They cost a pass two loads per lane and tile and
// one scalar load, one AND and one branch per plane; as kernels of their own
// (three per half for a plane wave's face axes, one for nodal cells) they cost
// a launch each, 4.4-9 us, and a second trip to memory for every face cell.
typedef __attribute__((address_space(4))) PassSrc CPassSrc;

// the address of face q's term at cell (i, j, k); fal: the faces in LDS
__device__ __forceinline__ int term_index(const FaceAddr *fal, int q, int i, int j, int k) {
  const FaceAddr a = fal[q];
  return a.base + i * a.sx + j * a.sy + k * a.sz;
}
// the faces in bits applied to v in the reference's order; first: the first
// face's term, loaded with the plane.  Binary16 storage rounds before and
// after each face, as a launch of its own on the stored value would; what
// comes back is a stored value, which the pass's store leaves as it is.
template <class S>
__device__ __forceinline__ float add_faces(unsigned bits, float first, const FaceAddr *fal,
                                           const float *terms, int i, int j, int k, float v,
                                           float s, float is) {
  v = S::trip_src(S::trip(v, s, is) + first, s, is);
  bits &= bits - 1;
  while (bits) {
    const int q = __builtin_ctz(bits);
    bits &= bits - 1;
    v = S::trip_src(v + terms[term_index(fal, q, i, j, k)], s, is);
  }
  return v;
}
// the first face's term of component bits (loaded ahead of its use)
__device__ __forceinline__ float first_term(unsigned bits, const FaceAddr *fal,
                                            const float *terms, int i, int j, int k) {
  return bits ? terms[term_index(fal, __builtin_ctz(bits), i, j, k)] : 0.0f;
}

// LDS of the face addresses, behind the media table of tab bytes
static __host__ __device__ __forceinline__ size_t face_lds_offset(size_t tab) {
  return (tab + 15) & ~(size_t)15;
}
template <class PS>
__device__ __forceinline__ const FaceAddr *stage_faces(const PS &x, float2 *lds, size_t tab) {
  FaceAddr *f = reinterpret_cast<FaceAddr *>(reinterpret_cast<char *>(lds) + face_lds_offset(tab));
  const int t = threadIdx.y * blockDim.x + threadIdx.x;
  const FaceAddr *src = x.fa;
  if (t < x.nface) f[t] = src[t];
  return f;
}

// AdvanceNodalE/H on the cells of one tile, after its march: the block's own
// stores are visible to it behind the barrier, and no other block writes the
// tile's cells.  Every thread of the block calls this.
template <class T, class G, class PS>
__device__ __forceinline__ void nodal_cells(const G &g, const PS &x, int c0, int c1, int off = 0) {
  __syncthreads();
  const int t = threadIdx.y * blockDim.x + threadIdx.x, nt = blockDim.x * blockDim.y;
  const int n = x.n + off + (x.dn ? *x.dn : 0);
  // cells that share a field value run in order, on one thread
  const int step = x.serial ? 1 : nt;
  for (int c = x.serial ? (t == 0 ? c0 : c1) : c0 + t; c < c1; c += step) {
    const NodalCell &cell = x.cells[c];
    if (cell.skip) continue;
    const float v = x.values[(long long)n * x.nsrc + cell.src];
    float *f = g.f[cell.comp];
    const float old = cell.hard ? 0.0f : Store<T>::ld1(f, cell.p, g.fs[cell.comp]);
    Store<T>::st_src(f, cell.p, g.fi[cell.comp], nodal_apply(old, cell, v));
  }
}
template <class T, class PS>
__device__ __forceinline__ void tile_nodal(const DevGrid &g, const TileMap &tm, const PS &x,
                                           int blk, int off = 0) {
  if (!x.nstart) return;
  const int tile = tm.remap ? xcd_remap(blk, tm.nblk) : blk;
  const int c0 = x.nstart[tile], c1 = x.nstart[tile + 1];
  if (c0 < c1) nodal_cells<T>(g, x, c0, c1, off);
}

// the tile's word (see kTileFaces) and its medium or -1
__device__ __forceinline__ int tile_info(const int *tmed) {
  return tmed ? __builtin_amdgcn_readfirstlane(tmed[blockIdx.x]) : 0;
}
__device__ __forceinline__ int tile_medium(int info) { return (info & 0xffff) - 1; }

}  // namespace SFD_NS
}  // namespace sfd
