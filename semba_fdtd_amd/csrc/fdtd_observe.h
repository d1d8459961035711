// fdtd_observe.h -- the observation of a grid after a step, as a launch of its
// own (fdtd_aux.hip) and as blocks of a face pass (fdtd_quad.hip).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "fdtd_internal.h"

namespace sfd {

// The TF/SF term +-G * Incid * id (AdvancePlaneWaveE/H, planewaves.F90:878-1475)
// of cell w of the faces' cells at step n: what pw_apply adds to the field,
// with the same roundings.
template <class P>
__device__ __forceinline__ void pw_term_cell(const P &t, long long w, int n) {
#pragma clang fp contract(off)
  int lo = 0, hi = t.nf - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (t.start[mid] <= w) lo = mid; else hi = mid - 1;
  }
  const PwFace &f = t.faces[lo];
  const int half = lo >= t.nf0 ? 1 : 0;
  const int ua = f.axis == 0 ? 1 : 0, va = f.axis == 2 ? 1 : 2;
  const int c = (int)(w - t.start[lo]), nu = f.hi[ua] - f.lo[ua] + 1;
  int cc[3];
  cc[f.axis] = f.fixed;
  cc[ua] = f.lo[ua] + c % nu;
  cc[va] = f.lo[va] + c / nu;
  const float tm = half ? (float)(t.tiempo[n] + (double)0.5f * t.dt) : (float)t.tiempo[n];
  const float x = t.G[half] * pw_incid(f, t.waves, t.phys, t.pstride, tm, cc) * f.id;
  t.out[w] = f.sign > 0.0f ? x : -x;
}

// Blocks of nt threads that sample a part's probes, at least one.  A part that
// moves the sample count has one block, which reads it before it moves it; the
// others, of as few as 64 threads inside a face pass, take one probe a thread:
// 10000 probes of a 64^3 cavity 162 us a step with one block, 11.2 so.
template <class P>
__host__ __device__ __forceinline__ int probe_blocks(const P &x, int nt) {
  return x.sample && !x.advance && x.o.np > nt ? (x.o.np + nt - 1) / nt : 1;
}

// UpdateObservation (observation.F90:2620-2672 point probes, :3553-3600
// frequency-domain sums), block blk of nt threads.  The first blocks sample the
// probes: row *count + row of their buffer, *count moving where the part says
// so, on the device so that a recorded step can be replayed.  The blocks after
// them take one (point, frequency) pair of a frequency-domain box per thread:
// the three components of the point are read once and multiplied by the
// complex(8) phase factor of the step (each part scaled by the real sample).
// The last blocks write the TF/SF terms of the next step, one cell per thread,
// for the passes that apply them inline.  All only read the fields, and no
// block reads what another writes.
template <class G, class P>
__device__ __forceinline__ void observe_block(const G &g, const P &x, int n, int blk, int nt) {
#pragma clang fp contract(off)
  const auto &o = x.o;
  const int t = (int)threadIdx.y * (int)blockDim.x + (int)threadIdx.x;
  auto field = [&](int c, long long p) {
    return g.fp16 ? __half2float(reinterpret_cast<const __half *>(g.f[c])[p]) * g.fs[c] : g.f[c][p];
  };
  const int bp = probe_blocks(x, nt);
  if (blk < bp) {
    if (!x.sample || o.np <= 0) return;
    __shared__ int first;
    if (t == 0) first = *o.count;
    __syncthreads();
    const int row = first + x.row;
    if (row < o.cap)
      for (int q = blk * nt + t; q < o.np; q += bp * nt) {
        const ProbeDev &pr = o.pr[q];
        if (x.half == 2 || pr.comp / 3 == x.half)
          o.buf[(long long)row * o.np + q] = field(pr.comp, pr.p);
      }
    __syncthreads();
    if (t == 0 && x.advance) *o.count = min(first + x.advance, o.cap);
    return;
  }
  const int dn = o.dn ? *o.dn : 0;
  const int bd = bp + (int)((x.d1 - x.d0 + nt - 1) / nt);
  if (blk >= bd) {
    const long long w = x.w0 + (long long)(blk - bd) * nt + t;
    if (w < x.w1 && n + 1 + dn < o.pw.ntime) pw_term_cell(o.pw, w, n + 1 + dn);
    return;
  }
  // A box starts at a multiple of every block's size: the block's threads share
  // it, and its descriptor comes by scalar loads.  (Read by each lane it was most
  // of the work: E and H boxes of 1.8 M pairs on 64^3 45.8 against 37.4 us a
  // step, of 6.6 M on 96^3 216 against 157.)
  const long long w = x.d0 + (long long)(blk - bp) * nt;
  typedef __attribute__((address_space(4))) DftDev CDft;
  const CDft *box = (const CDft *)o.dft;
  int q = 0;
  while (q + 1 < o.ndft && box[q + 1].start <= w) ++q;
  const CDft &d = box[q];
  const long long u = w + t - d.start;
  if (u >= (long long)d.cnt[0] * d.cnt[1] * d.cnt[2] * d.nfreq) return;
  const long long pt = u / d.nfreq;
  const int f = (int)(u - pt * d.nfreq);
  const int it = (int)(pt % d.cnt[0]);
  const int jt = (int)((pt / d.cnt[0]) % d.cnt[1]);
  const int kt = (int)(pt / ((long long)d.cnt[0] * d.cnt[1]));
  const long long p = (long long)(d.first[2] + kt * d.stride[2] + 1) * g.pxy +
                      (long long)(d.first[1] + jt * d.stride[1] + 1) * g.px + g.xoff +
                      d.first[0] + it * d.stride[0];
  const double2 a = d.aux[(long long)(n + dn) * d.nfreq + f];
  for (int c = 0; c < 3; ++c) {
    const double v = (double)field(3 * d.kind + c, p);
    double2 *acc = d.acc + (pt * 3 + c) * d.nfreq + f;
    const double2 o2 = *acc;
    *acc = make_double2(o2.x + a.x * v, o2.y + a.y * v);
  }
}

}  // namespace sfd
