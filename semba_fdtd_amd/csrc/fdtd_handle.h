// fdtd_handle.h -- host-side state of one grid (the opaque fdtd_handle of
// the C ABI) and the helpers the host translation units share.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <unordered_map>
#include <vector>

#include "fdtd_internal.h"
#include "sembafdtd.h"

namespace sfd_host {
using namespace sfd;
struct Source {
  int comp, hard;
  int box[6];
  float amp, deltaevol;
  int numus;
  std::vector<float> evol;
};

struct AdeIn {           // the dispersive media of one field, as set by the caller
  int ndisp = 0;
  std::vector<int32_t> dmed, dnp;
  std::vector<double> dk, db, dg3;
  long long nedges[3] = {0, 0, 0};  // dispersive edges per component
  size_t jbytes[3] = {0, 0, 0};      // pole-current bytes per component
};

struct DftIn {           // one frequency-domain observation box
  int kind;
  int box[6], stride[3];
  std::vector<float> freq;
};

// one launch of TF/SF faces: the faces of one wave and one face axis
struct PwGroup {
  int half;                       // 0: E faces, 1: H faces
  std::vector<PwRun> runs;        // step from the launch (dn = null)
  std::vector<long long> start;   // prefix of face areas, runs.size()+1 entries
  PwRun *druns[2] = {};           // device copies: [0] launch step, [1] device counter
  long long *dstart = nullptr;
};

// Has a device table been built: by launches that ran, or by launches that a
// caller is recording, for the other calls of that recording alone (rec: the
// recording's id plus one, 0: none).
struct BuiltIn {
  bool now = false;
  unsigned long long rec = 0;
  bool ok(unsigned long long id) const { return now || (id && id == rec); }
  void set(unsigned long long id) { if (id) rec = id; else now = true; }
  void drop() { now = false; rec = 0; }
};

// a media table past this many entries is shared by four rows of the four-cell
// passes (quad_default)
constexpr int kManyMedia = 256;

// the tiles of the four-cell passes: boxes, the slabs they meet (launch_quad),
// rows per block, planes per tile
struct QuadLayout {
  QuadPlan p = {};
  int slabs = 0, rows = 1, kc = 1;
};

// the sources of a half that a pass applies inline, and its nodal cells' tables
// (src.nstart and src.cells: their device copies, once placed)
struct SrcTables {
  bool on = false;
  PassSrc src = {};
  std::vector<int> nstart;
  std::vector<NodalCell> cells;
};

struct PlaneWaveIn {     // sgg%PlaneWave(j) (planeonde_t, fdetypes.F90:458-465)
  int esq[6];            // esqx1, esqx2, esqy1, esqy2, esqz1, esqz2
  int nmodes;
  float p[kPwModes][3], e[kPwModes][3], incert[kPwModes];
  float deltaevol;
  std::vector<float> evol;
  float eps0, mu0;
};
}  // namespace sfd_host

struct fdtd_handle {
  std::string err;
  int device = 0;
  hipStream_t stream = nullptr;       // the stream every launch goes to
  hipStream_t solo_stream = nullptr;  // its own stream while lent to a batch
  bool own_stream = false;
  int mode = FDTD_MODE_FAST;
  int storage = FDTD_STORE_FP32;
  sfd::DevGrid g{};
  // 64-cell x tiles of the one-cell passes: as set, and the default by depth,
  // which the granular calls keep where the fused passes run four cells per lane
  sfd::TileMap tm{}, tm_default{};
  int xcells = 1;              // 4: the fused passes run four cells per lane
  bool tile_set = false;       // fdtd_set_tiling was called
  int tile_zchunk = 32;        // planes per z chunk as set (tm.kc: clipped to the grid)
  std::vector<void *> allocs;
  std::unordered_map<void *, size_t> sizes;   // of each allocation
  int64_t bytes = 0;
  float *fld[6] = {};
  int16_t *mi[6] = {};
  // media
  int nmedia = -1;
  int media_max = 0;  // largest media index written so far
  std::vector<float> g2h, gm2h;
  std::vector<int32_t> kindh;
  float *dg[4] = {};
  // spacing
  std::vector<float> idh_[6];
  float *did[6] = {};
  // cpml
  float *dprof[12] = {};
  long long psilen[12] = {};       // psi values per slab array
  // dispersive media: [0] electric (on E), [1] magnetic (on H)
  sfd_host::AdeIn adein[2];
  // first-order Mur faces
  int mur_faces[6] = {0, 0, 0, 0, 0, 0};
  std::vector<float> cab1h;            // [6][nmedia+1]
  bool mur_ready = false;
  std::vector<void *> mur_allocs;
  std::vector<sfd::MurRun> mur_runs;   // host copy (past pointers on the device)
  sfd::MurRun *dmur = nullptr;
  long long mur_total = 0;
  bool ade_ready = false;
  std::vector<void *> ade_allocs;
  // time
  double dt = 0.0;
  std::vector<double> tiempo;
  // nodal
  std::vector<sfd_host::Source> srcs;
  bool nodal_ready = false;
  std::vector<void *> nodal_allocs;
  sfd::NodalCell *dcells[2] = {};
  int ncells[2] = {0, 0};
  int serial[2] = {0, 0};
  float *dvalues = nullptr;
  int nvalues_steps = 0;
  // TF/SF plane waves
  std::vector<sfd_host::PlaneWaveIn> pwin;
  std::vector<float> line[3];           // LineX/Y/Z over [-1, n+1]
  bool pw_ready = false;
  std::vector<void *> pw_allocs;
  std::vector<sfd::PwFace> pw_faces[2];      // E faces, H faces, in reference order
  std::vector<sfd_host::PwGroup> pw_groups;  // launch groups, in reference order
  sfd::PwWave *dwaves = nullptr;
  float *dphys = nullptr;
  int pstride = 0;
  double *dtiempo = nullptr;
  // some face has cells outside its component's sweep (a box on the grid's edge):
  // the two passes' own launches reach them, the one-launch step does not
  bool pw_edge = false;
  // the faces of each half as the face passes apply them inline (pw_masks:
  // at most kPassFaces, all inside their components' sweeps), and the buffer
  // of both halves' terms, which holds those of step pw_terms_n (-1: none) until
  // a caller has recorded a step that writes it (pw_recorded)
  bool pw_masks[2] = {false, false};
  sfd::PassSrc pw_src[2] = {};
  std::vector<unsigned> pw_bits[2][3];  // host copy of the faces' index masks
  sfd::PwTerms pw_terms{};
  int pw_terms_n = -1;
  bool pw_recorded = false;
  long long pw_split = 0;          // terms of the E faces
  // per half: the sources the pass applies inline under the tiling (valid while
  // psrc_gen == src_gen).  src_gen counts the changes of the tiling, the sources
  // and the pole-state boxes.
  unsigned src_gen = 1, psrc_gen = 0;
  bool inline_ok = true;           // (sfd_set_inline_sources)
  bool psrc_on[2] = {false, false};
  sfd::PassSrc psrc[2] = {};
  std::vector<void *> psrc_allocs;
  // frequency-domain observation
  std::vector<sfd_host::DftIn> dftin;
  std::vector<sfd::DftDev> dfts;
  sfd::DftDev *ddfts = nullptr;       // device copy of dfts, the boxes of E first
  long long dft_end[2] = {0, 0};      // pairs of E's boxes, of all boxes
  bool dft_ready = false;
  std::vector<void *> dft_allocs;     // phase tables (rebuilt with the time vector)
  std::vector<void *> dft_sums;       // running sums (kept across rebuilds)
  // probes
  sfd::ProbeDev *dprobes = nullptr;
  int nprobe = 0;
  float *dpbuf = nullptr;
  int *dpcount = nullptr;
  int pcap = 0;
  // graph
  int *dstep = nullptr;           // device step counter of the captured step
  hipGraphExec_t gexec = nullptr;
  hipGraph_t graph = nullptr;
  bool graph_ok = false;
  // the same two-pass step recorded graph_steps times in one graph
  int graph_steps = 16;
  hipGraphExec_t mexec = nullptr;
  hipGraph_t mgraph = nullptr;
  // one-launch steps (k_step): a second copy of the time-stepping state (B),
  // the A->B and B->A descriptors and a captured pair of steps
  int step_rows = 0;              // 0: two passes per step; else rows per block (4, 8, 16)
  int step_kc = 32;
  int step_creq[17] = {};  // rows per block asked for each
                                  // tile class (0: the default); a class on fewer
                                  // rows than step_rows runs the step's tiles cut
                                  // into row bands
  bool step_vec = true;           // plain tiles run four x cells per lane (k_step4)
  int step_merge = -1, step_fork = -1;   // (sfd_set_step_plan)
  // the branches of a recorded one-launch step
  hipStream_t side[2] = {};
  hipEvent_t forked = nullptr, joined[2] = {};
  int cus = 256;                  // compute units of the device
  int lds_max = 65536;            // LDS bytes a block may use on the device
  bool step_ready = false;
  bool step_stale = true;         // B's fields must be refreshed from A
  std::vector<void *> step_allocs;       // the second state
  std::vector<void *> step_small;        // descriptors' tables
  std::vector<size_t> step_sizes;        // layout of the second state
  sfd::DevGrid gB;
  sfd::StepDev sd[2];             // [0] A -> B, [1] B -> A
  // tiles grouped by class (bit 0 CPML, 1 poles, 2 sources; 8 plain tiles
  // four cells per lane): one launch per class with tiles, each over its
  // slice of the device tile list
  std::vector<int> step_cls, step_cnt, step_off;
  std::vector<int> step_crows;           // rows per block of each class launch
  std::vector<int> step_uni;             // leading single-medium tiles of each class launch
  // the words of the tiles of the one-cell pass map tm (while tmed_on; tiling and
  // media changes drop it), tmed_cap of them, then their flags
  int *tmed = nullptr;
  int tmed_cap = 0;
  sfd_host::BuiltIn tmed_on;
  sfd_host::BuiltIn gmed_on;   // tmed holds the granular calls' (tm_default) instead
  // the four-cell passes' tiles and their words and flags (while tmed_on and the
  // grid runs these passes)
  sfd_host::QuadLayout quad;
  int *qmed = nullptr;
  int qmed_cap = 0;
  std::vector<double> step_cells;        // Yee cells owned per class
  std::vector<double> step_bytes;        // compulsory HBM bytes of one launch per class
  uint8_t *mi8[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};  // step mode
  void *stage = nullptr;                 // packed staging buffer of host transfers
  size_t stage_bytes = 0;
  // the stored previous field of the pole updates may differ from the field
  // (fields set from outside, granular calls): the next pair reads it
  bool prev_exact = true;
  bool prev_lazy = false;      // the stored previous fields await settle_prev
  sfd::StepTile *dtiles = nullptr;
  std::vector<sfd::StepTile> step_tiles;  // host copy of the tile list (batches)
  // TF/SF faces of both halves for the step kernels and the buffer of their
  // incident field, refreshed before every step
  sfd::PwFace *dsfaces = nullptr;
  int step_nf0 = 0, step_nf = 0;
  long long step_maxcells = 0;
  float *dinc = nullptr;
  sfd::StepSrc *dstepsrc = nullptr;
  hipGraphExec_t pexec = nullptr;
  hipGraph_t pgraph = nullptr;
  std::vector<sfd::NodalCell> hcells[2];   // host copies of the nodal cells
  unsigned version = 0;           // bumped by every change that drops the graph
  // the batch the grid is admitted to (null: none).  While it is set the
  // batch's captured step replays over the grid's buffers and shares its step
  // counter, so the grid's own stepping calls and fdtd_destroy are refused.
  fdtd_batch *batch = nullptr;
  // probe samples taken since the last fdtd_read_probes (or fdtd_set_probes):
  // a call that would take more than the buffer holds is refused
  long long pbuffered = 0;
};


// helpers shared by the host translation units (fdtd_host.cpp)
namespace sfd_host {
int fail(fdtd_handle *h, int code, const char *fmt, ...) __attribute__((format(printf, 3, 4)));
int dalloc(fdtd_handle *h, void **p, size_t bytes, std::vector<void *> *list = nullptr);
int refuse_batched(fdtd_handle *h);
// extents of component comp's Alloc box per axis
void alloc_extent(const fdtd_handle *h, int comp, long long ext[3]);
int probe_room(fdtd_handle *h, long long more);
bool quads_fit(const fdtd_handle *h);
QuadLayout plan_quads(const fdtd_handle *h, int rows, int kc);
int prepare(fdtd_handle *h);
int build_tile_media(fdtd_handle *h);
int build_granular_media(fdtd_handle *h);
int run_pw(fdtd_handle *h, int half, int n, const int *dn);
int run_nodal(fdtd_handle *h, int half, int n, const int *dn);
// the sources of a half as a one-cell pass over tile map tm applies them, on
// only where it can (else run_pw and run_nodal follow the pass); flags (null:
// not wanted): per block of tm, what its tile meets is added
void make_pass_src(const fdtd_handle *h, const sfd::TileMap &tm, int half, SrcTables *out,
                   std::vector<int> *flags);
// the same for the four-cell passes (flags: the words of the layout's tiles)
void make_quad_src(const fdtd_handle *h, const QuadLayout &l, int half, SrcTables *out, int *flags);
// UpdateObservation at step n (or *dn + n): point probes, frequency-domain
// sums, and (pw) the TF/SF terms of the next step; half 0, 1: the E, the H
// quantities alone (the H part moves the sample count), 2: all.  run_observe
// launches it on grid g (h->g or the written copy of a one-launch step).
sfd::ObservePart observe_part(const fdtd_handle *h, int half, int n, const int *dn, bool probes,
                              bool dft, bool pw);
int run_observe(fdtd_handle *h, const sfd::DevGrid &g, const sfd::ObservePart &p);
int run_mur(fdtd_handle *h);
int run_ade(fdtd_handle *h, int side);
void invalidate_graph(fdtd_handle *h);
// the one-launch step: its descriptors and tile plan (step_rows > 0), the
// second state refreshed from the first when stale, a class's rows per block
int build_step(fdtd_handle *h);
int sync_b(fdtd_handle *h);
int class_rows(const fdtd_handle *h, int c);
bool step_supported(const fdtd_handle *h, int rows);
}  // namespace sfd_host

// a failed HIP call on grid h: its message, and FDTD_ERR_HIP from the caller
#define HIPCHK(h, call)                                                        \
  do {                                                                         \
    hipError_t e_ = (call);                                                    \
    if (e_ != hipSuccess)                                                      \
      return sfd_host::fail(h, FDTD_ERR_HIP, "%s: %s (%s:%d)", #call,          \
                            hipGetErrorString(e_), __FILE__, __LINE__);        \
  } while (0)
