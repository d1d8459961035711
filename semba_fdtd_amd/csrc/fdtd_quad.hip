// fdtd_quad.hip -- kernels of the four-cell face passes of one grid (fdtd_quad.h).
#include "fdtd_observe.h"
#include "fdtd_quad.h"

namespace sfd {
namespace SFD_NS {

// one launch; the kernels read the descriptor where the launch
// left it, in the constant kernel-argument segment
struct QuadArgs {
  DevGrid g;
  QuadPlan p;
  const int *tmed;
  PassSrc x;      // the half's sources
  int nobs;       // blocks ahead of the tiles' that observe (a multiple of 8:
                  // the tiles keep their XCDs)
  ObservePart obs;
};
typedef __attribute__((address_space(4))) QuadArgs CQuadArgs;

// One tile.  info: its word (kTileFaces).  A tile whose cells hold one medium
// reads no media and takes its coefficients by scalar loads: no table, no
// barrier before its first loads.  X: some tiles meet TF/SF faces (none of
// those in y or z slabs).  Every thread of the block calls this.
template <bool H, int CPML, bool X, class T, class G, class PS>
__device__ __forceinline__ void run_quad(const G &g, float2 *lds, int info, const QuadPos &at,
                                         bool live, const PS &x) {
  const float *const t1 = H ? g.gm1 : g.g1, *const t2 = H ? g.gm2 : g.g2;
  const int m0 = tile_medium(info);
  const bool faces = X && (info & kTileFaces[H ? 1 : 0]);
  const FaceAddr *fal = nullptr;
  MedTab tab{};
  float2 cu = make_float2(0.f, 0.f);
  if (faces) fal = stage_faces(x, lds, (size_t)(g.nmedia + 1) * sizeof(float2));
  if (m0 >= 0) {
    cu = make_float2(ro_uniform(t1, m0), ro_uniform(t2, m0));
    if (faces) __syncthreads();
  } else {
    tab = stage_pair(g.nmedia, t1, t2, lds);
  }
  if (!live) return;
#define SFD_RUN(U, F)                                                     \
  do {                                                                    \
    if (H) hquad_tile<CPML, U, F, T>(g, tab, cu, at, x, fal);             \
    else equad_tile<CPML, U, F, T>(g, tab, cu, at, x, fal);               \
  } while (0)
  if (faces) {
    if (m0 >= 0) SFD_RUN(true, X);
    else SFD_RUN(false, X);
  } else {
    if (m0 >= 0) SFD_RUN(true, false);
    else SFD_RUN(false, false);
  }
#undef SFD_RUN
}

// SLABS, X: what the launch's tiles may meet
template <bool H, int SLABS, bool X, class T>
__global__ void __launch_bounds__(256, SLABS == 0 && !X ? 6 : 1) k_quad(QuadArgs) {
  extern __shared__ float2 lds_tab[];
  const CQuadArgs &a = *(const CQuadArgs *)__builtin_amdgcn_kernarg_segment_ptr();
  if ((int)blockIdx.x < a.nobs) {
    observe_block(a.g, a.obs, a.obs.n, (int)blockIdx.x, (int)(blockDim.x * blockDim.y));
    return;
  }
  const int t = xcd_remap((int)blockIdx.x - a.nobs, a.p.nblk);
  const int info = ro_uniform_i(a.tmed, t);
  QuadPos at;
  const bool live = quad_pos(a.p, t, at);
  int c0 = 0, c1 = 0;   // the tile's nodal cells
  if (a.x.nstart) {
    c0 = ro_uniform_i(a.x.nstart, t);
    c1 = ro_uniform_i(a.x.nstart, t + 1);
  }
  if (SLABS == kSlabMix && t >= a.p.start[1]) run_quad<H, kSlabAll, false, T>(a.g, lds_tab, info, at, live, a.x);
  else run_quad<H, SLABS == kSlabMix ? kSlabX : SLABS, X, T>(a.g, lds_tab, info, at, live, a.x);
  if (c0 < c1) nodal_cells<T>(a.g, a.x, c0, c1);
}

// The tiles of every grid of a batch, one block each, descriptors read through
// the constant address space.  X: some grid's passes apply sources inline.
template <bool H, bool X, class T>
__global__ void __launch_bounds__(256) k_quad_batch(BatchDev bd) {
  extern __shared__ float2 lds_tab[];
  typedef __attribute__((address_space(4))) DevGrid CDevGrid;
  typedef __attribute__((address_space(4))) QuadTile CQuadTile;
  typedef __attribute__((address_space(4))) QuadBox CQuadBox;
  const CQuadTile &qt = ((const CQuadTile *)bd.qtiles)[blockIdx.x];
  const int b = qt.grid, info = qt.info;
  const CDevGrid &g = *(const CDevGrid *)(bd.grids + b);
  const CPassSrc &x = *((const CPassSrc *)bd.src[H ? 1 : 0] + (X ? b : 0));
  QuadPos at;
  const bool live = quad_pos(load_box(((const CQuadBox *)bd.qboxes)[qt.box]), qt.t, at);
  if (info & kTileSlabs) run_quad<H, kSlabAll, false, T>(g, lds_tab, info, at, live, x);
  else run_quad<H, kSlabX, X, T>(g, lds_tab, info, at, live, x);
  if (X && (info & kTileNodal[H ? 1 : 0]))
    nodal_cells<T>(g, x, ro_uniform_i(x.nstart, qt.tg), ro_uniform_i(x.nstart, qt.tg + 1),
                   bd.n);
}

int launch_quad_batch(const BatchDev &bd, int half, int rows, size_t lds, int fp16, void *stream) {
  const dim3 grid((unsigned)bd.total), blk(kWave, (unsigned)rows);
  hipStream_t s = (hipStream_t)stream;
  const bool x = bd.src[half ? 1 : 0];
  if (x) lds = face_lds_offset(lds) + kPassFaces * sizeof(FaceAddr);
#define SFD_QB(X, T)                                                                        \
  do {                                                                                      \
    if (half) hipLaunchKernelGGL((k_quad_batch<true, X, T>), grid, blk, lds, s, bd);        \
    else hipLaunchKernelGGL((k_quad_batch<false, X, T>), grid, blk, lds, s, bd);            \
  } while (0)
  if (fp16 && x) SFD_QB(true, __half);
  else if (fp16) SFD_QB(false, __half);
  else if (x) SFD_QB(true, float);
  else SFD_QB(false, float);
#undef SFD_QB
  return (int)hipGetLastError();
}

// The medium that all six media arrays hold on every swept cell of a tile plus
// one, or 0 (they hold several), from every thread of its block.
__device__ __forceinline__ int tile_one_medium(const DevGrid &g, const QuadPos &at, bool live) {
  __shared__ int lo, hi;
  if (threadIdx.x == 0 && threadIdx.y == 0) { lo = 0x7fffffff; hi = -0x7fffffff; }
  __syncthreads();
  int a = 0x7fffffff, b = -0x7fffffff;
  const int n = g.nx + 1 - at.i0;   // cells inside the sweeps
  if (live)
    for (int k = at.k0; k < at.k1; ++k) {
      const long long q = (long long)(k + 1) * g.pxy + (long long)(at.j + 1) * g.px + g.xoff + at.i0;
#pragma unroll
      for (int c = 0; c < 6; ++c) {
        const u32x2 v = *reinterpret_cast<const u32x2 *>(g.mi[c] + q);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          const int m = (int)(((x < 2 ? v.x : v.y) >> (16 * (x & 1))) & 0xffffu);
          if (x < n) { a = min(a, m); b = max(b, m); }
        }
      }
    }
  atomicMin(&lo, a);
  atomicMax(&hi, b);
  __syncthreads();
  return lo == hi ? lo + 1 : 0;
}

// the word of each tile: out[t] = flags[t] plus it, or added to the batch's
// qtiles[t].info
__global__ void __launch_bounds__(256) k_quad_media(DevGrid g, QuadPlan p, const int *flags, int *out) {
  QuadPos at;
  const bool live = quad_pos(p, (int)blockIdx.x, at);
  const int m = tile_one_medium(g, at, live);
  if (threadIdx.x == 0 && threadIdx.y == 0) out[blockIdx.x] = flags[blockIdx.x] + m;
}
__global__ void __launch_bounds__(256) k_quad_media_batch(BatchDev bd) {
  QuadTile &qt = bd.qtiles[blockIdx.x];
  QuadPos at;
  const bool live = quad_pos(bd.qboxes[qt.box], qt.t, at);
  const int m = tile_one_medium(bd.grids[qt.grid], at, live);
  if (threadIdx.x == 0 && threadIdx.y == 0) qt.info += m;
}

int launch_quad_media(const DevGrid &g, const QuadPlan &p, int rows, const int *flags, int *out,
                      void *stream) {
  if (p.nblk <= 0) return 0;
  hipLaunchKernelGGL(k_quad_media, dim3((unsigned)p.nblk), dim3(kWave, (unsigned)rows), 0,
                     (hipStream_t)stream, g, p, flags, out);
  return (int)hipGetLastError();
}

int launch_quad_media_batch(const BatchDev &bd, int rows, void *stream) {
  if (bd.total <= 0) return 0;
  hipLaunchKernelGGL(k_quad_media_batch, dim3((unsigned)bd.total), dim3(kWave, (unsigned)rows), 0,
                     (hipStream_t)stream, bd);
  return (int)hipGetLastError();
}

int launch_quad(const DevGrid &g, const QuadPlan &p, int slabs, int rows, const int *tmed,
                int half, const PassSrc &src, const ObservePart *obs, void *stream) {
  if (p.nblk <= 0) return 0;
  QuadArgs a{g, p, tmed, src, 0, {}};
  if (obs) {
    a.obs = *obs;
    a.nobs = (observe_blocks(*obs, kWave * rows) + 7) & ~7;
  }
  const dim3 grid((unsigned)(p.nblk + a.nobs)), blk(kWave, (unsigned)rows);
  const size_t tab = (size_t)(g.nmedia + 1) * sizeof(float2);
  const size_t lds = src.nface ? face_lds_offset(tab) + kPassFaces * sizeof(FaceAddr) : tab;
  hipStream_t s = (hipStream_t)stream;
#define SFD_Q(C, X, T)                                                               \
  do {                                                                               \
    if (half) hipLaunchKernelGGL((k_quad<true, C, X, T>), grid, blk, lds, s, a);     \
    else hipLaunchKernelGGL((k_quad<false, C, X, T>), grid, blk, lds, s, a);         \
  } while (0)
#define SFD_QC(C, X)                 \
  do {                               \
    if (g.fp16) SFD_Q(C, X, __half); \
    else SFD_Q(C, X, float);         \
  } while (0)
  const bool x = src.nface > 0;
  if (slabs == kSlabAll) SFD_QC(kSlabAll, false);
  else if (slabs == kSlabMix && x) SFD_QC(kSlabMix, true);
  else if (slabs == kSlabMix) SFD_QC(kSlabMix, false);
  else if (slabs == kSlabX && x) SFD_QC(kSlabX, true);
  else if (slabs == kSlabX) SFD_QC(kSlabX, false);
  else if (x) SFD_QC(0, true);
  else SFD_QC(0, false);
#undef SFD_QC
#undef SFD_Q
  return (int)hipGetLastError();
}

}  // namespace SFD_NS
}  // namespace sfd
