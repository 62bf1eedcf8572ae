// C-ABI layer: argument checks, plans (block table, halo gather table, BC
// tables, tile table, stage workspace), launches, hipGraph capture and
// error reporting.  Declarations: include/famrdp_capi.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <string>
#include <vector>

#include "famrdp_kernels.hip"
#include "famrdp_adjoint.hip"
#include "famrdp_reverse.h"
#include "famrdp_tune.h"
#include "../../include/famrdp_capi.h"

using namespace famrdp;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

#define HIP_TRY(expr)                                                                          \
  do {                                                                                         \
    hipError_t e_ = (expr);                                                                    \
    if (e_ != hipSuccess) return fail(FAMRDP_E_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define LAUNCH_CHECK()                                                                         \
  do {                                                                                         \
    hipError_t e_ = hipGetLastError();                                                         \
    if (e_ != hipSuccess) return fail(FAMRDP_E_HIP, std::string("kernel launch: ") + hipGetErrorString(e_)); \
  } while (0)

inline hipStream_t S(void* s) { return reinterpret_cast<hipStream_t>(s); }
inline unsigned nblk(int64_t n, int t = 256) { return (unsigned)((n + t - 1) / t); }

Gas to_gas(const famrdp_gas* g) { return Gas{g->gamma, g->R, g->mu0, g->T0, g->Ts, g->Pr_lam}; }

bool bad_lim(int32_t lim) { return lim != FAMRDP_LIMITER_MINMOD && lim != FAMRDP_LIMITER_VANLEER; }

// Per-workgroup partial results of the CFL reduction (k_cfl_partial), for
// the entry point that allocates nothing (famrdp_cfl_dt_noalloc): a
// library-owned array of 2 x CFL_PARTS doubles (16 KiB) on each GPU, held
// until the process ends and shared by every call on that GPU.  Its address
// is taken once per device (hipGetSymbolAddress, with that device current)
// and only that address is handed to kernels and copies.
constexpr int CFL_PARTS = 1024;

}  // namespace

static __device__ __align__(256) double scratch[2 * CFL_PARTS];

namespace {

int cfl_scratch(double** ptr) {
  static std::mutex mu;
  static std::vector<double*> per_dev;
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  if ((int)per_dev.size() <= dev) per_dev.resize(dev + 1, nullptr);
  if (!per_dev[dev]) {
    void* a = nullptr;
    const hipError_t e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !a)
      return fail(FAMRDP_E_HIP, std::string("cfl_dt_noalloc: hipGetSymbolAddress: ") + hipGetErrorString(e));
    per_dev[dev] = static_cast<double*>(a);
  }
  *ptr = per_dev[dev];
  return FAMRDP_OK;
}

}  // namespace

// The small device arrays of a plan, gathered so that one allocation and one
// copy make them all: an allocation or a synchronous copy costs 10-30 us
// whatever its size, and a plan has about forty such arrays.
class TableSet {
 public:
  TableSet() = default;
  TableSet(const TableSet&) = delete;
  TableSet& operator=(const TableSet&) = delete;
  ~TableSet() { std::free(bytes_); }
  template <class T>
  void table(T** dst, const std::vector<T>& src) {   // a device copy of src (none of an empty one)
    if (src.empty()) return;
    const size_t at = up(len_), end = at + sizeof(T) * src.size();
    if (end > cap_) {                                // (realloc moves large buffers without a copy)
      cap_ = std::max(end, 2 * cap_);
      char* p = static_cast<char*>(std::realloc(bytes_, cap_));
      if (!p) throw std::bad_alloc();
      bytes_ = p;
    }
    std::memcpy(bytes_ + at, src.data(), sizeof(T) * src.size());
    len_ = end;
    slots_.push_back({reinterpret_cast<void**>(dst), at, false});
  }
  template <class T>
  void scratch(T** dst, size_t count) {              // not initialised
    if (count == 0) return;
    slots_.push_back({reinterpret_cast<void**>(dst), scratch_, true});
    scratch_ += up(sizeof(T) * count);
  }
  bool make(char** mem) {
    const size_t tables = up(len_);
    if (tables + scratch_ == 0) return true;
    if (hipMalloc(mem, tables + scratch_) != hipSuccess) return false;
    if (len_ > 0 && hipMemcpy(*mem, bytes_, len_, hipMemcpyHostToDevice) != hipSuccess)
      return false;
    for (const Slot& s : slots_) *s.dst = *mem + (s.scratch ? tables : 0) + s.at;
    return true;
  }

 private:
  static constexpr size_t ALIGN = 256;
  struct Slot { void** dst; size_t at; bool scratch; };
  static size_t up(size_t n) { return (n + ALIGN - 1) / ALIGN * ALIGN; }
  char* bytes_ = nullptr;
  size_t len_ = 0, cap_ = 0, scratch_ = 0;
  std::vector<Slot> slots_;
};

struct famrdp_plan {
  int nblocks = 0, ghost = 2, limiter = 0;
  Gas gas{};
  std::vector<int32_t> dims;             // 3 per block
  std::vector<int64_t> N;
  char* d_tables = nullptr;              // holds every d_ array below
  BlockDesc* d_blocks = nullptr;
  // staging ring for block-table uploads: a slot is reused only after the
  // copy that last read it has completed (its event), so uploads do not
  // drain the stream
  static constexpr int NSTAGE = 8;
  BlockDesc* h_stage[NSTAGE] = {};
  hipEvent_t stage_ev[NSTAGE] = {};
  bool stage_used[NSTAGE] = {};
  int stage_next = 0;
  std::vector<BlockDesc> h_blocks;
  bool blocks_uploaded = false;
  bool table_in_graph = false;    // a captured launch writes the device table whenever its graph is replayed
  HaloEntry* d_halo = nullptr;
  int nhalo = 0;
  double* d_halo_stage = nullptr;
  // ghost cells of a step (famrdp_ghost.h)
  GhostEntry* d_ghost = nullptr;
  GhostChain* d_chains = nullptr;
  BcEntry* d_ops = nullptr;
  GhostSnap* d_snaps = nullptr;
  double* d_ghost_stage = nullptr;
  int nghost_direct = 0, nghost_staged = 0, nghost_late = 0, nghost_kept = 0, nsnaps = 0;
  BcEntry* d_bc[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  int nbc[6] = {0, 0, 0, 0, 0, 0};
  int64_t bc_maxcells[6] = {0, 0, 0, 0, 0, 0};
  Tile* d_tiles = nullptr;
  int ntiles = 0;
  double* d_monitor = nullptr;    // per-workgroup partial counts of the state monitor (persistent_grid)
  Tile3* d_tiles3[NUM_TILE_VARIANTS] = {};
  int ntiles3[NUM_TILE_VARIANTS] = {};
  int len3[NUM_TILE_VARIANTS] = {};   // variant_len of all blocks
  int tile_variant = -1;          // -1: by the blocks' sizes (default_variant)
  int auto_all = 0;               // then: the variant of launches over all blocks
  std::vector<int> auto_block;    // and of a block's own launches
  int persistent_grid = 0;
  int ncu = 256;                  // compute units of the device the plan was made on
  // workspace
  std::vector<double*> q1, q2, G;
  // graph cache
  hipStream_t cap_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t graph_exec = nullptr;
  std::vector<const void*> graph_key;
  double graph_dt = 0.0;
  int graph_flags = -1;
  bool has_workspace = true;
  // adjoint workspace
  bool has_adjoint = false;
  BlockDesc* d_blocks_adj = nullptr;         // same blocks with q -> qh (recompute buffer)
  std::vector<BlockDesc> h_blocks_adj;
  std::vector<double*> adj_bufs;
  SweepTile* d_sweep_ik = nullptr;           // reverse sweeps along i (with k), along j and of the viscous part
  SweepTile* d_sweep_j = nullptr;
  SweepTile* d_sweep_v = nullptr;
  int nsweep_ik = 0, nsweep_j = 0, nsweep_v = 0;
  HaloEntry* d_halo_sorted = nullptr;        // halo entries sorted by source cell
  HaloSrc* d_halo_src = nullptr;
  int nhalo_src = 0;
  double* d_halo_S = nullptr;
  double* d_bc_snap[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  double* d_bc_part[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
  double* d_bc_red[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};   // per-chunk sums of d_bc_part
  // stage timing (HIP events on the launch stream, eager launches only)
  bool timing = false;
  bool capturing = false;
  std::vector<hipEvent_t> ev_pool;
  size_t ev_used = 0;
};

namespace {

// Face geometry: axis (0..2) and low/high side.
inline int face_axis(int f) { return f / 2; }
inline bool face_lo(int f) { return f % 2 == 0; }

// The copies of the exchange, in the order given (a later one wins).
int add_cuts(const famrdp_plan* p, int ncut, const famrdp_cut* cuts, GhostTable& table) {
  const int g = p->ghost;
  for (int c = 0; c < ncut; ++c) {
    const famrdp_cut& ct = cuts[c];
    if (ct.tgt_block < 0 || ct.tgt_block >= p->nblocks || ct.src_block < 0 || ct.src_block >= p->nblocks ||
        ct.tgt_face < 0 || ct.tgt_face > 5 || ct.src_face < 0 || ct.src_face > 5)
      return fail(FAMRDP_E_INVALID, "cut " + std::to_string(c) + ": block or face out of range");
    if (ct.orient != 0)
      return fail(FAMRDP_E_UNSUPPORTED, "orient=" + std::to_string(ct.orient) + " not supported in stage 1");
    const int32_t* dt = &p->dims[3 * ct.tgt_block];
    const int32_t* ds = &p->dims[3 * ct.src_block];
    int lo_t[3] = {0, 0, 0}, ext_t[3] = {dt[0], dt[1], dt[2]};
    int lo_s[3] = {0, 0, 0}, ext_s[3] = {ds[0], ds[1], ds[2]};
    const int at = face_axis(ct.tgt_face), as = face_axis(ct.src_face);
    lo_t[at] = face_lo(ct.tgt_face) ? 0 : dt[at] - g;  // halo.py:19-23
    ext_t[at] = g;
    lo_s[as] = face_lo(ct.src_face) ? g : ds[as] - 2 * g;  // halo.py:26-33
    ext_s[as] = g;
    if (ext_t[0] != ext_s[0] || ext_t[1] != ext_s[1] || ext_t[2] != ext_s[2])
      return fail(FAMRDP_E_INVALID, "cut " + std::to_string(c) + ": ghost slab and source slab shapes differ");
    for (int a = 0; a < ext_t[0]; ++a)
      for (int b = 0; b < ext_t[1]; ++b)
        for (int k = 0; k < ext_t[2]; ++k) {
          const int64_t sc = ((int64_t)(lo_s[0] + a) * ds[1] + (lo_s[1] + b)) * ds[2] + (lo_s[2] + k);
          table.copy(ct.tgt_block, lo_t[0] + a, lo_t[1] + b, lo_t[2] + k, ct.src_block, (int32_t)sc);
        }
  }
  return FAMRDP_OK;
}

// Stream-ordered upload of a block table through the staging ring.
int upload_table(famrdp_plan* p, BlockDesc* dst, const std::vector<BlockDesc>& src, hipStream_t st) {
  const int s = p->stage_next;
  p->stage_next = (s + 1) % famrdp_plan::NSTAGE;
  if (p->stage_used[s]) HIP_TRY(hipEventSynchronize(p->stage_ev[s]));   // that slot's last copy is done
  std::memcpy(p->h_stage[s], src.data(), sizeof(BlockDesc) * p->nblocks);
  HIP_TRY(hipMemcpyAsync(dst, p->h_stage[s], sizeof(BlockDesc) * p->nblocks, hipMemcpyHostToDevice, st));
  HIP_TRY(hipEventRecord(p->stage_ev[s], st));
  p->stage_used[s] = true;
  return FAMRDP_OK;
}

// Puts the caller's arrays into the host copy of the block table and says
// whether the plan's table and the reverse sweep's have changed by it.  q ==
// nullptr leaves the state pointers as they are (the reverse sweep reads its own
// copy, qh); kxyz / vol == nullptr keep the bound metrics.  q1t / q2t: where the
// step's stage-1/2 results go (caller arrays), or NULL for the plan's workspace.
// Arguments that are refused leave the table as it is.
int bind_host(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol, bool need_q,
              double* const* q1t, double* const* q2t, bool& changed, bool& changed_adj) {
  if (need_q && !q) return fail(FAMRDP_E_INVALID, "q pointer array is NULL");
  for (int b = 0; q && b < p->nblocks; ++b)
    if (!q[b]) return fail(FAMRDP_E_INVALID, "q[" + std::to_string(b) + "] is NULL");
  changed = changed_adj = !p->blocks_uploaded || p->table_in_graph;
  for (int b = 0; b < p->nblocks; ++b) {
    BlockDesc& d = p->h_blocks[b];
    const double* kx = kxyz ? kxyz[b] : d.kxyz;
    const double* vo = vol ? vol[b] : d.vol;
    double* s1 = q1t ? q1t[b] : p->q1[b];
    double* s2 = q2t ? q2t[b] : p->q2[b];
    if ((q && d.q != q[b]) || d.kxyz != kx || d.vol != vo || d.q1 != s1 || d.q2 != s2) changed = true;
    if (d.kxyz != kx || d.vol != vo) changed_adj = true;
    if (q) d.q = q[b];
    d.kxyz = kx;
    d.vol = vo;
    d.q1 = s1;
    d.q2 = s2;
  }
  return FAMRDP_OK;
}

// Whether an array of `in` and one of `out` (one per block, 5 N doubles each)
// share memory: q_in and q of a step from one into the other.
bool states_overlap(const famrdp_plan* p, const double* const* in, double* const* out) {
  struct Range { uintptr_t lo, hi; bool out; };
  std::vector<Range> v;
  v.reserve(2 * (size_t)p->nblocks);
  for (int b = 0; b < p->nblocks; ++b) {
    const uintptr_t n = sizeof(double) * 5 * (uintptr_t)p->N[b], i = (uintptr_t)in[b], o = (uintptr_t)out[b];
    v.push_back({i, i + n, false});
    v.push_back({o, o + n, true});
  }
  std::sort(v.begin(), v.end(), [](const Range& a, const Range& b) { return a.lo < b.lo; });
  uintptr_t end[2] = {0, 0};               // how far the arrays so far reach, of in and of out
  for (const Range& x : v) {
    if (x.lo < end[x.out ? 0 : 1]) return true;
    end[x.out] = std::max(end[x.out], x.hi);
  }
  return false;
}

int upload_adj(famrdp_plan* p, hipStream_t st) {
  for (int b = 0; b < p->nblocks; ++b) {
    BlockDesc a = p->h_blocks[b];
    a.q = p->h_blocks_adj[b].qh;
    p->h_blocks_adj[b] = a;
  }
  return upload_table(p, p->d_blocks_adj, p->h_blocks_adj, st);
}

// bind_host, and the tables uploaded where a pointer changed.
int bind(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol, hipStream_t st,
         bool need_q = true, double* const* q1t = nullptr, double* const* q2t = nullptr) {
  bool changed, changed_adj;
  int rc = bind_host(p, q, kxyz, vol, need_q, q1t, q2t, changed, changed_adj);
  if (rc) return rc;
  p->blocks_uploaded = false;   // until all of it is
  if (changed) {
    rc = upload_table(p, p->d_blocks, p->h_blocks, st);
    if (rc) return rc;
  }
  if (p->has_adjoint && changed_adj) {
    rc = upload_adj(p, st);
    if (rc) return rc;
  }
  p->blocks_uploaded = true;
  return FAMRDP_OK;
}

// Copies of one 5*N array per block (dst[b] <- src[b]) in as few launches
// as the job table allows (COPY_JOBS blocks per launch).
template <class Dst, class Src>
int copy_blocks(famrdp_plan* p, hipStream_t st, Dst dst_of, Src src_of) {
  for (int b0 = 0; b0 < p->nblocks; b0 += COPY_JOBS) {
    const int nj = std::min(COPY_JOBS, p->nblocks - b0);
    CopyJobs jobs{};
    int64_t nmax = 0;
    for (int j = 0; j < nj; ++j) {
      jobs.dst[j] = dst_of(b0 + j);
      jobs.src[j] = src_of(b0 + j);
      jobs.n[j] = 5 * p->N[b0 + j];
      nmax = std::max(nmax, jobs.n[j]);
    }
    const int64_t gx = std::min<int64_t>((nmax + 1023) / 1024, 65535);
    k_copy_jobs<<<dim3((unsigned)gx, (unsigned)nj), 256, 0, st>>>(jobs);
    LAUNCH_CHECK();
  }
  return FAMRDP_OK;
}

// The halo exchange on its own.
int launch_halo(famrdp_plan* p, hipStream_t st) {
  if (p->nhalo == 0) return FAMRDP_OK;
  const BlockDesc* tb = p->d_blocks;
  k_halo_gather<<<nblk(p->nhalo), 256, 0, st>>>(tb, p->d_halo, p->nhalo, p->d_halo_stage);
  LAUNCH_CHECK();
  k_halo_scatter<<<nblk(p->nhalo), 256, 0, st>>>(tb, p->d_halo, p->nhalo, p->d_halo_stage);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

// The BC faces in Face order, on their own.
int launch_bc(famrdp_plan* p, hipStream_t st) {
  for (int f = 0; f < 6; ++f) {
    if (p->nbc[f] == 0) continue;
    dim3 grid(nblk(p->bc_maxcells[f]), (unsigned)p->nbc[f]);
    k_bc_face<<<grid, 256, 0, st>>>(p->d_blocks, p->d_bc[f], p->ghost, p->gas.gamma, p->gas.R);
    LAUNCH_CHECK();
  }
  return FAMRDP_OK;
}

// Halo exchange and BCs of a step (workspace plans); with `snapshot`, the
// inner layers of isothermal faces are recorded as each face finds them (for
// the reverse sweep).
int launch_ghosts(famrdp_plan* p, hipStream_t st, const BlockDesc* tb, bool snapshot = false) {
  const int nsnap = snapshot ? p->nsnaps : 0;
  const int n1 = p->nghost_direct + p->nghost_staged + nsnap, n2 = p->nghost_staged + p->nghost_late;
  SnapPtrs snap{};
  for (int f = 0; f < 6; ++f) snap.face[f] = p->d_bc_snap[f];
  if (n1 > 0) {
    k_ghost_first<<<nblk(n1), 256, 0, st>>>(tb, p->d_ghost, p->nghost_direct, p->nghost_staged, p->d_chains, p->d_ops,
                                            p->gas.gamma, p->gas.R, p->d_ghost_stage, p->d_snaps, nsnap, snap);
    LAUNCH_CHECK();
  }
  if (n2 > 0) {
    k_ghost_second<<<nblk(n2), 256, 0, st>>>(tb, p->d_ghost + p->nghost_direct, p->nghost_staged, p->nghost_late,
                                             p->d_chains, p->d_ops, p->gas.gamma, p->gas.R, p->d_ghost_stage);
    LAUNCH_CHECK();
  }
  return FAMRDP_OK;
}

hipEvent_t next_event(famrdp_plan* p) {
  if (p->ev_used == p->ev_pool.size()) {
    hipEvent_t e = nullptr;
    if (hipEventCreate(&e) != hipSuccess) return nullptr;
    p->ev_pool.push_back(e);
  }
  return p->ev_pool[p->ev_used++];
}

// the i-marching and wide variants address a block's arrays with 32-bit byte offsets
bool variant_fits(const famrdp_plan* p, int v) {
  if (!is_march_variant(v) && !is_wide_variant(v)) return true;
  for (int b = 0; b < p->nblocks; ++b)
    if (!march_fits(p->N[b])) return false;
  return true;
}

int batched_variant(const famrdp_plan* p) { return p->tile_variant < 0 ? p->auto_all : p->tile_variant; }

int launch_stages(famrdp_plan* p, double dt, int flags, hipStream_t st, bool adj = false, int nstages = 3) {
  const bool direct = (flags & FAMRDP_STEP_DIRECT) != 0;
  const BlockDesc* dtab = adj ? p->d_blocks_adj : p->d_blocks;
  const std::vector<BlockDesc>& htab = adj ? p->h_blocks_adj : p->h_blocks;
  const int vb = batched_variant(p);
  if (flags & FAMRDP_STEP_BATCHED) {
    // every batched launch indexes a device tile table: refuse to launch without one
    if (!p->d_blocks || (direct ? (!p->d_tiles || p->ntiles < 1)
                                : (!p->d_tiles3[vb] || p->ntiles3[vb] < 1)))
      return fail(FAMRDP_E_INVALID, "batched step: tile table missing");
  }
  for (int stage = 1; stage <= nstages; ++stage) {
    const bool tm = p->timing && !p->capturing;
    hipEvent_t e0 = tm ? next_event(p) : nullptr, e1 = tm ? next_event(p) : nullptr;
    if (tm && (!e0 || !e1)) return fail(FAMRDP_E_HIP, "hipEventCreate failed");
    if (tm) HIP_TRY(hipEventRecord(e0, st));
    if (!direct && (flags & FAMRDP_STEP_BATCHED)) {
      launch_fused_batched(vb, dtab, p->d_tiles3[vb], p->ntiles3[vb], stage, p->gas, p->limiter, dt, p->len3[vb], st);
      LAUNCH_CHECK();
    } else if (!direct) {
      for (int b = 0; b < p->nblocks; ++b) {
        launch_fused(p->tile_variant < 0 ? p->auto_block[b] : p->tile_variant, htab[b], stage, p->gas, p->limiter, dt, p->ncu, st);
        LAUNCH_CHECK();
      }
    } else if (flags & FAMRDP_STEP_BATCHED) {
      k_viscous_flux_batched<<<p->persistent_grid, 256, 0, st>>>(dtab, p->d_tiles, p->ntiles, stage, p->gas);
      LAUNCH_CHECK();
      k_stage_batched<<<p->persistent_grid, 256, 0, st>>>(dtab, p->d_tiles, p->ntiles, p->gas.gamma,
                                                          p->limiter, dt, stage);
      LAUNCH_CHECK();
    } else {
      for (int b = 0; b < p->nblocks; ++b) {
        const BlockDesc& d = htab[b];
        const double* qin = stage == 1 ? d.q : (stage == 2 ? d.q1 : d.q2);
        double* qout = stage == 1 ? d.q1 : (stage == 2 ? d.q2 : d.q);
        Gas gb = p->gas;
        gb.mu0 = d.mu0;
        k_viscous_flux<<<nblk(d.N), 256, 0, st>>>(qin, d.kxyz, d.G, d.ni, d.nj, d.nk, gb);
        LAUNCH_CHECK();
        k_stage<<<nblk(d.N), 256, 0, st>>>(qin, d.q, qout, d.kxyz, d.vol, d.G, d.ni, d.nj, d.nk, p->gas.gamma,
                                           p->limiter, dt * d.dt_scale, stage);
        LAUNCH_CHECK();
      }
    }
    if (tm) HIP_TRY(hipEventRecord(e1, st));
  }
  return FAMRDP_OK;
}

int run_step(famrdp_plan* p, double dt, int flags, hipStream_t st) {
  const int rc = launch_ghosts(p, st, p->d_blocks);
  if (rc) return rc;
  return launch_stages(p, dt, flags, st);
}

}  // namespace

extern "C" {

const char* famrdp_last_error(void) { return g_last_error.c_str(); }

const char* famrdp_version(void) { return "famrdp-mi355x 0.18 (gfx950, fp64, fused, split, i-marching and wide stage kernels, chosen by size or autotuned)"; }

int famrdp_cons_to_prim(const double* q, double* pv, int64_t n, double gamma, void* stream) {
  if (n < 0 || (n > 0 && (!q || !pv))) return fail(FAMRDP_E_INVALID, "cons_to_prim: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_cons_to_prim<<<nblk(n), 256, 0, S(stream)>>>(q, pv, n, gamma);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_prim_to_cons(const double* pv, double* q, int64_t n, double gamma, void* stream) {
  if (n < 0 || (n > 0 && (!q || !pv))) return fail(FAMRDP_E_INVALID, "prim_to_cons: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_prim_to_cons<<<nblk(n), 256, 0, S(stream)>>>(pv, q, n, gamma);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_sutherland(const double* T, double* mu, int64_t n, double mu0, double T0, double Ts, void* stream) {
  if (n < 0 || (n > 0 && (!T || !mu))) return fail(FAMRDP_E_INVALID, "sutherland: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_sutherland<<<nblk(n), 256, 0, S(stream)>>>(T, mu, n, mu0, T0, Ts);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_speed_of_sound(const double* rho, const double* p, double* c, int64_t n, double gamma, void* stream) {
  if (n < 0 || (n > 0 && (!rho || !p || !c))) return fail(FAMRDP_E_INVALID, "speed_of_sound: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_speed_of_sound<<<nblk(n), 256, 0, S(stream)>>>(rho, p, c, n, gamma);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_limiter(const double* a, const double* b, double* out, int64_t n, int32_t limiter, void* stream) {
  if (bad_lim(limiter)) return fail(FAMRDP_E_KEY, "unknown limiter code " + std::to_string(limiter));
  if (n < 0 || (n > 0 && (!a || !b || !out))) return fail(FAMRDP_E_INVALID, "limiter: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_limiter<<<nblk(n), 256, 0, S(stream)>>>(a, b, out, n, limiter);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_fastmath_probe(const double* x, double* out_rcp, double* out_sqrt, double* out_rsqrt, int64_t n,
                          void* stream) {
  if (n < 0 || (n > 0 && (!x || !out_rcp || !out_sqrt))) return fail(FAMRDP_E_INVALID, "fastmath_probe: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_fastmath_probe<<<nblk(n), 256, 0, S(stream)>>>(x, out_rcp, out_sqrt, out_rsqrt, n);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_fastmath_probe1(const double* x, double* out_rcp, double* out_rsqrt, int64_t n, void* stream) {
  if (n < 0 || (n > 0 && (!x || !out_rcp || !out_rsqrt))) return fail(FAMRDP_E_INVALID, "fastmath_probe1: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_fastmath_probe1<<<nblk(n), 256, 0, S(stream)>>>(x, out_rcp, out_rsqrt, n);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_muscl2(const double* pv, double* pv_L, double* pv_R, int32_t nvar, int32_t n0, int32_t n1, int32_t n2,
                  int32_t axis, int32_t limiter, void* stream) {
  if (bad_lim(limiter)) return fail(FAMRDP_E_KEY, "unknown limiter code " + std::to_string(limiter));
  if (axis < 1 || axis > 3 || nvar < 1 || n0 < 1 || n1 < 1 || n2 < 1)
    return fail(FAMRDP_E_INVALID, "muscl2: bad shape or axis");
  const int na = axis == 1 ? n0 : (axis == 2 ? n1 : n2);
  if (na < 4) return fail(FAMRDP_E_INVALID, "muscl2: need at least 4 cells along the axis");
  const int64_t nf = (int64_t)(axis == 1 ? n0 - 3 : n0) * (axis == 2 ? n1 - 3 : n1) * (axis == 3 ? n2 - 3 : n2);
  k_muscl2<<<nblk(nf), 256, 0, S(stream)>>>(pv, pv_L, pv_R, nvar, n0, n1, n2, axis, limiter);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_roe_flux(const double* UL, const double* UR, const double* nxyz, double* F, int64_t n, double gamma,
                    double eps_entropy, void* stream) {
  if (n < 0 || (n > 0 && (!UL || !UR || !nxyz || !F))) return fail(FAMRDP_E_INVALID, "roe_flux: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_roe_flux<<<nblk(n), 256, 0, S(stream)>>>(UL, UR, nxyz, F, n, gamma, eps_entropy);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_invscd_rhs(const double* q, const double* kxyz, const double* vol, double* rhs, int32_t ni, int32_t nj,
                      int32_t nk, double gamma, int32_t limiter, void* stream) {
  if (bad_lim(limiter)) return fail(FAMRDP_E_KEY, "unknown limiter code " + std::to_string(limiter));
  if (ni < 1 || nj < 1 || nk < 1 || !q || !kxyz || !vol || !rhs) return fail(FAMRDP_E_INVALID, "invscd_rhs: bad arguments");
  Gas g{};
  g.gamma = gamma;
  g.R = g.Pr_lam = g.T0 = 1.0;
  const unsigned grid = rhs_grid<4, 4, 4>(ni, nj, nk);
  constexpr int nth = CrossGeom<4, 4, 4>::NTH;
  if (limiter == LIM_VANLEER)
    k_invscd_rhs<4, 4, 4, LIM_VANLEER><<<grid, nth, 0, S(stream)>>>(q, kxyz, vol, rhs, ni, nj, nk, stage_gas(g), gamma);
  else
    k_invscd_rhs<4, 4, 4, LIM_MINMOD><<<grid, nth, 0, S(stream)>>>(q, kxyz, vol, rhs, ni, nj, nk, stage_gas(g), gamma);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_viscous_rhs(const double* q, const double* kxyz, double* rhs, int32_t ni, int32_t nj, int32_t nk,
                       const famrdp_gas* gas, double* work, void* stream) {
  if (ni < 1 || nj < 1 || nk < 1 || !q || !kxyz || !rhs || !gas || !work)
    return fail(FAMRDP_E_INVALID, "viscous_rhs: bad arguments");
  k_viscous_rhs<4, 8, 8><<<rhs_grid<4, 8, 8>(ni, nj, nk), WideGeom<4, 8, 8>::NGW, 0, S(stream)>>>(q, kxyz, rhs, ni, nj, nk,
                                                                                    to_gas(gas));
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_axpby(double* out, double a, const double* x, double b, const double* y, double c, const double* z,
                 int64_t n, int32_t mode, void* stream) {
  if (n < 0 || (n > 0 && (!out || !y || !z || (mode != 1 && !x)))) return fail(FAMRDP_E_INVALID, "axpby: bad arguments");
  if (n == 0) return FAMRDP_OK;
  k_axpby<<<nblk(n), 256, 0, S(stream)>>>(out, a, x, b, y, c, z, n, mode);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_compute_metrics(const double* xyz, double* jac, double* kxyz, double* vol, int32_t ni, int32_t nj,
                           int32_t nk, void* stream) {
  if (ni < 1 || nj < 1 || nk < 1 || !xyz || !jac || !kxyz || !vol) return fail(FAMRDP_E_INVALID, "compute_metrics: bad arguments");
  if (!metrics_marched(ni, nj, nk)) {
    k_metrics_cell<<<nblk((int64_t)ni * nj * nk), 256, 0, S(stream)>>>(xyz, jac, kxyz, vol, ni, nj, nk);
    LAUNCH_CHECK();
    return FAMRDP_OK;
  }
  // segments as long as leaves four workgroups per CU, 8 planes at most (a
  // segment starts with four planes that it does not work on): 20^3 takes 7.1
  // us with 1 plane and 17.2 with 8, 204^3 403 with 1, 308 with 8, 315 with 16
  const int64_t tiles = (int64_t)((nj + METRIC_TJ - 1) / METRIC_TJ) * ((nk + METRIC_TK - 1) / METRIC_TK);
  const int len = (int)std::clamp<int64_t>((ni * tiles + 1023) / 1024, 1, 8);
  k_metrics<<<(unsigned)(tiles * ((ni + len - 1) / len)), METRIC_TJ * METRIC_TK, 0, S(stream)>>>(xyz, jac, kxyz, vol,
                                                                                                ni, nj, nk, len);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_cfl_dt(const double* q, const double* kxyz, const double* vol, int32_t ni, int32_t nj, int32_t nk,
                  int32_t ghost, const famrdp_gas* gas, double cfl, double* out, double* work, void* stream) {
  if (!q || !kxyz || !vol || !gas || !out || !work || ghost < 0 || ni <= 2 * ghost || nj <= 2 * ghost ||
      nk <= 2 * ghost)
    return fail(FAMRDP_E_INVALID, "cfl_dt: bad arguments");
  const int parts = CFL_PARTS;
  k_cfl_partial<<<parts, 256, 0, S(stream)>>>(q, kxyz, vol, ni, nj, nk, ghost, to_gas(gas), work, work + parts);
  LAUNCH_CHECK();
  k_cfl_final<<<1, 256, 0, S(stream)>>>(work, work + parts, parts, cfl, out);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_cfl_dt_noalloc(const double* q, const double* kxyz, const double* vol, int32_t ni, int32_t nj,
                          int32_t nk, int32_t ghost, const famrdp_gas* gas, double cfl, double* out, void* stream) {
  if (!q || !kxyz || !vol || !gas || !out || ghost < 0 || ni <= 2 * ghost || nj <= 2 * ghost || nk <= 2 * ghost)
    return fail(FAMRDP_E_INVALID, "cfl_dt_noalloc: bad arguments");
  double* work = nullptr;
  const int rc = cfl_scratch(&work);
  if (rc) return rc;
  // the partials of every workgroup are written before k_cfl_final reads
  // them: nothing left in the array by an earlier call is read
  k_cfl_partial<<<CFL_PARTS, 256, 0, S(stream)>>>(q, kxyz, vol, ni, nj, nk, ghost, to_gas(gas), work,
                                                  work + CFL_PARTS);
  LAUNCH_CHECK();
  k_cfl_final<<<1, 256, 0, S(stream)>>>(work, work + CFL_PARTS, CFL_PARTS, cfl, out);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_plan_timing(famrdp_plan* p, int32_t enable, double* stage_ms, int64_t* stage_count) {
  if (!p) return fail(FAMRDP_E_INVALID, "plan is NULL");
  if (enable) {
    p->timing = true;
    p->ev_used = 0;
    return FAMRDP_OK;
  }
  double total = 0.0;
  int64_t n = 0;
  for (size_t i = 0; i + 1 < p->ev_used; i += 2) {
    HIP_TRY(hipEventSynchronize(p->ev_pool[i + 1]));
    float ms = 0.f;
    HIP_TRY(hipEventElapsedTime(&ms, p->ev_pool[i], p->ev_pool[i + 1]));
    total += ms;
    ++n;
  }
  p->timing = false;
  p->ev_used = 0;
  if (stage_ms) *stage_ms = total;
  if (stage_count) *stage_count = n;
  return FAMRDP_OK;
}

int famrdp_plan_destroy(famrdp_plan* p) {
  if (!p) return FAMRDP_OK;
  for (auto e : p->ev_pool) (void)hipEventDestroy(e);
  if (p->graph_exec) (void)hipGraphExecDestroy(p->graph_exec);
  if (p->graph) (void)hipGraphDestroy(p->graph);
  if (p->cap_stream) (void)hipStreamDestroy(p->cap_stream);
  for (auto* x : p->adj_bufs) (void)hipFree(x);
  for (auto* x : p->q1) (void)hipFree(x);
  for (auto* x : p->q2) (void)hipFree(x);
  for (auto* x : p->G) (void)hipFree(x);
  if (p->d_tables) (void)hipFree(p->d_tables);
  for (int s = 0; s < famrdp_plan::NSTAGE; ++s) {
    if (p->stage_ev[s]) {
      if (p->stage_used[s]) (void)hipEventSynchronize(p->stage_ev[s]);
      (void)hipEventDestroy(p->stage_ev[s]);
    }
  }
  if (p->h_stage[0]) (void)hipHostFree(p->h_stage[0]);   // one allocation for the ring
  delete p;
  return FAMRDP_OK;
}

}  // extern "C"

namespace {

// A plan in the making, destroyed unless it is given away.
struct PlanOwner {
  famrdp_plan* p;
  ~PlanOwner() { (void)famrdp_plan_destroy(p); }
};

int plan_create_impl(famrdp_plan** out, int32_t nblocks, const int32_t* dims, int32_t ncut, const famrdp_cut* cuts,
                     int32_t nbc, const famrdp_bc* bcs, const famrdp_gas* gas, int32_t limiter, int32_t ghost,
                     int32_t plan_flags) {
  if (nblocks < 1 || !dims || !gas || ncut < 0 || nbc < 0 || (ncut > 0 && !cuts) || (nbc > 0 && !bcs))
    return fail(FAMRDP_E_INVALID, "plan_create: bad arguments");
  if (bad_lim(limiter)) return fail(FAMRDP_E_KEY, "unknown limiter code " + std::to_string(limiter));
  if (ghost < 1) return fail(FAMRDP_E_INVALID, "ghost must be >= 1");
  if (ghost != 2 && !(plan_flags & FAMRDP_PLAN_NO_WORKSPACE))
    return fail(FAMRDP_E_UNSUPPORTED, "the step needs ghost=2 (the MUSCL-2 stencil width)");
  PlanOwner owner{new famrdp_plan()};
  famrdp_plan* p = owner.p;
  p->nblocks = nblocks;
  p->ghost = ghost;
  p->limiter = limiter;
  p->gas = to_gas(gas);
  p->dims.assign(dims, dims + 3 * nblocks);
  p->has_workspace = !(plan_flags & FAMRDP_PLAN_NO_WORKSPACE);
  int rc = FAMRDP_OK;
  for (int b = 0; b < nblocks; ++b) {
    const int32_t* d = &dims[3 * b];
    if (d[0] < 2 * ghost || d[1] < 2 * ghost || d[2] < 2 * ghost)
      return fail(FAMRDP_E_INVALID, "block " + std::to_string(b) + ": each padded size must be >= 2*ghost");
    if ((int64_t)d[0] * d[1] * d[2] > INT32_MAX)   // tile kernels index cells in 32 bits
      return fail(FAMRDP_E_INVALID, "block " + std::to_string(b) + ": 2^31 or more cells");
    // the reverse kernels address cells with 32-bit byte offsets
    if ((plan_flags & FAMRDP_PLAN_ADJOINT) && (int64_t)d[0] * d[1] * d[2] >= (int64_t(1) << 29))
      return fail(FAMRDP_E_INVALID, "block " + std::to_string(b) + ": 2^29 or more cells in an adjoint plan");
    p->N.push_back((int64_t)d[0] * d[1] * d[2]);
  }
  TableSet tables;
  // workspace and block table
  p->h_blocks.resize(nblocks);
  for (int b = 0; b < nblocks; ++b) {
    double *q1 = nullptr, *q2 = nullptr, *G = nullptr;
    if (p->has_workspace && (hipMalloc(&q1, sizeof(double) * 5 * p->N[b]) != hipSuccess ||
        hipMalloc(&q2, sizeof(double) * 5 * p->N[b]) != hipSuccess ||
        hipMalloc(&G, sizeof(double) * 9 * p->N[b]) != hipSuccess)) {
      if (q1) (void)hipFree(q1);
      if (q2) (void)hipFree(q2);
      if (G) (void)hipFree(G);
      return fail(FAMRDP_E_HIP, "plan_create: workspace allocation failed");
    }
    p->q1.push_back(q1);
    p->q2.push_back(q2);
    p->G.push_back(G);
    BlockDesc& bd = p->h_blocks[b];
    bd = BlockDesc{};
    bd.q1 = q1; bd.q2 = q2; bd.G = G;
    bd.ni = dims[3 * b]; bd.nj = dims[3 * b + 1]; bd.nk = dims[3 * b + 2];
    bd.N = p->N[b];
    bd.wrap_mod = tile_wrap_mod(bd.ni, bd.nj, bd.nk);
    bd.mu0 = p->gas.mu0;
    bd.dt_scale = 1.0;
  }
  p->has_adjoint = (plan_flags & FAMRDP_PLAN_ADJOINT) != 0 && p->has_workspace;
  if (p->has_adjoint) {
    p->h_blocks_adj = p->h_blocks;
    for (int b = 0; b < nblocks; ++b) {
      const int64_t n = p->N[b];
      // qh, la, lb, (l0: the caller's cotangent array, bound by each
      // famrdp_step_vjp), fs, vs
      const int64_t sizes[6] = {5 * n, 5 * n, 5 * n, 0, 5 * n, 8 * n};
      double* bufs[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
      for (int i = 0; i < 6; ++i) {
        if (sizes[i] == 0) {
          p->adj_bufs.push_back(nullptr);
          continue;
        }
        if (hipMalloc(&bufs[i], sizeof(double) * sizes[i]) != hipSuccess)
          return fail(FAMRDP_E_HIP, "plan_create: adjoint workspace allocation failed");
        p->adj_bufs.push_back(bufs[i]);
        if (hipMemset(bufs[i], 0, sizeof(double) * sizes[i]) != hipSuccess)
          return fail(FAMRDP_E_HIP, "plan_create: adjoint workspace clear failed");
      }
      BlockDesc& a = p->h_blocks_adj[b];
      a.qh = bufs[0]; a.la = bufs[1]; a.lb = bufs[2]; a.l0 = bufs[3]; a.fs = bufs[4]; a.vs = bufs[5];
      a.q = a.qh;
      p->h_blocks[b].qh = a.qh; p->h_blocks[b].la = a.la; p->h_blocks[b].lb = a.lb;
      p->h_blocks[b].l0 = a.l0; p->h_blocks[b].fs = a.fs; p->h_blocks[b].vs = a.vs;
    }
    tables.scratch(&p->d_blocks_adj, nblocks);
  }
  tables.scratch(&p->d_blocks, nblocks);
  if (hipHostMalloc(&p->h_stage[0], sizeof(BlockDesc) * nblocks * famrdp_plan::NSTAGE) != hipSuccess)
    return fail(FAMRDP_E_HIP, "plan_create: block table staging allocation failed");
  for (int s = 0; s < famrdp_plan::NSTAGE; ++s) {
    p->h_stage[s] = p->h_stage[0] + (size_t)s * nblocks;
    if (hipEventCreateWithFlags(&p->stage_ev[s], hipEventDisableTiming) != hipSuccess)
      return fail(FAMRDP_E_HIP, "plan_create: block table staging allocation failed");
  }
  // halo gather table
  GhostTable ghosts(ghost, nblocks, dims);
  rc = add_cuts(p, ncut, cuts, ghosts);
  if (rc) return rc;
  std::vector<HaloEntry> halo;
  ghosts.halo(halo);
  p->nhalo = (int)halo.size();
  tables.table(&p->d_halo, halo);
  tables.scratch(&p->d_halo_stage, 5 * halo.size());
  // BC tables grouped by face (Face order, dispatch.py:15)
  std::vector<BcEntry> byface[6];
  for (int i = 0; i < nbc; ++i) {
    const famrdp_bc& c = bcs[i];
    if (c.block < 0 || c.block >= nblocks || c.face < 0 || c.face > 5 || c.kind < 0 || c.kind > 4)
      return fail(FAMRDP_E_INVALID, "bc " + std::to_string(i) + ": block, face or kind out of range");
    BcEntry e{};
    e.block = c.block; e.face = c.face; e.kind = c.kind; e.T_wall = c.T_wall;
    for (int v = 0; v < 5; ++v) e.q_inf[v] = c.q_inf[v];
    byface[c.face].push_back(e);
    const int32_t* d = &dims[3 * c.block];
    const int ax = c.face / 2;
    const int64_t cells = (int64_t)d[(ax + 1) % 3] * d[(ax + 2) % 3];
    p->bc_maxcells[c.face] = std::max(p->bc_maxcells[c.face], cells);
  }
  for (int f = 0; f < 6; ++f) {
    // a block with two BCs on one face keeps the last (dict semantics)
    std::vector<BcEntry> uniq;
    for (auto& e : byface[f]) {
      bool replaced = false;
      for (auto& u : uniq) if (u.block == e.block) { u = e; replaced = true; }
      if (!replaced) uniq.push_back(e);
    }
    p->nbc[f] = (int)uniq.size();
    byface[f] = uniq;
    tables.table(&p->d_bc[f], uniq);
  }
  if (p->has_workspace) {   // exchange and BCs of a step in one table
    ghosts.boundary(byface, p->bc_maxcells, p->has_adjoint);
    ghosts.finish();
    p->nghost_direct = ghosts.ndirect;
    p->nghost_staged = ghosts.nstaged;
    p->nghost_late = ghosts.nlate;
    p->nghost_kept = ghosts.nkept;
    p->nsnaps = (int)ghosts.snaps.size();
    tables.table(&p->d_ghost, ghosts.entries);
    tables.table(&p->d_chains, ghosts.chains);
    tables.table(&p->d_ops, ghosts.ops);
    tables.table(&p->d_snaps, ghosts.snaps);
    tables.scratch(&p->d_ghost_stage, 5 * (size_t)ghosts.nstaged);
  }
  if (p->has_adjoint) {
    if (p->nhalo > 0) {
      std::vector<HaloEntry> sorted = halo;
      std::stable_sort(sorted.begin(), sorted.end(), [](const HaloEntry& a, const HaloEntry& b) {
        return a.sb != b.sb ? a.sb < b.sb : a.sc < b.sc;
      });
      std::vector<HaloSrc> us;
      for (int e = 0; e < (int)sorted.size(); ++e) {
        if (us.empty() || us.back().sb != sorted[e].sb || us.back().sc != sorted[e].sc)
          us.push_back(HaloSrc{sorted[e].sb, sorted[e].sc, e, 0});
        us.back().count++;
      }
      p->nhalo_src = (int)us.size();
      tables.table(&p->d_halo_sorted, sorted);
      tables.table(&p->d_halo_src, us);
      tables.scratch(&p->d_halo_S, 5 * us.size());
    }
    for (int f = 0; f < 6; ++f) {
      if (p->nbc[f] == 0) continue;
      const size_t n = (size_t)p->nbc[f] * 5 * (size_t)p->bc_maxcells[f];
      tables.scratch(&p->d_bc_snap[f], n * p->ghost);
      tables.scratch(&p->d_bc_part[f], n);
      tables.scratch(&p->d_bc_red[f], (size_t)p->nbc[f] * 5 * BC_RED_PARTS);
    }
  }
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    ncu = 256;
  // tile table for the batched launches
  std::vector<Tile> tiles;
  for (int b = 0; b < nblocks; ++b)
    for (int64_t s = 0; s < p->N[b]; s += 256) tiles.push_back(Tile{b, (int32_t)s});
  p->ntiles = (int)tiles.size();
  tables.table(&p->d_tiles, tiles);
  for (int v = 0; v < NUM_TILE_VARIANTS; ++v) {
    int TI, TJ, TK;
    tile_dims(v, TI, TJ, TK);
    p->len3[v] = variant_len(v, nblocks, dims, ncu);
    std::vector<Tile3> tiles3;
    for (int b = 0; b < nblocks; ++b) {
      const int32_t* d = &dims[3 * b];
      if (is_march_variant(v)) {   // i0 = 2 x segment index + strip bit
        const MarchTiling mt = march_tiling(TJ, TK, d[1], d[2]);
        for (int sg = 0; sg < march_nseg(d[0], p->len3[v]); ++sg)
          for (int t = 0; t < mt.count(); ++t) {
            int j0, k0, tr;
            march_tile_of(mt, TJ, TK, t, j0, k0, tr);
            tiles3.push_back(Tile3{b, 2 * sg + tr, j0, k0});
          }
        continue;
      }
      for (int i = 0; i < d[0]; i += TI)
        for (int j = 0; j < d[1]; j += TJ)
          for (int k = 0; k < d[2]; k += TK) tiles3.push_back(Tile3{b, i, j, k});
    }
    p->ntiles3[v] = (int)tiles3.size();
    tables.table(&p->d_tiles3[v], tiles3);
  }
  p->persistent_grid = std::min(p->ntiles, ncu * 8);
  p->ncu = ncu;
  p->auto_all = default_variant(nblocks, dims, ncu, variant_fits(p, 18));
  for (int b = 0; b < nblocks; ++b)
    p->auto_block.push_back(default_variant(1, &dims[3 * b], ncu, march_fits(p->N[b])));
  if (p->has_adjoint) {
    SweepSet ik{{}, {}, SWEEP_IK}, jj{{}, {}, SWEEP_J}, vv{{}, {}, SWEEP_V};
    for (int b = 0; b < nblocks; ++b) {
      const int32_t* d = &dims[3 * b];
      ik.along.push_back(d[0]);
      ik.across.push_back(d[1] * d[2]);
      vv.along.push_back(d[0]);
      vv.across.push_back(d[1] * (d[2] + 4));
      jj.along.push_back(d[1]);
      jj.across.push_back(d[0] * d[2]);
    }
    const int64_t slots = SWEEP_WAVES * 4 * (int64_t)ncu;   // four SIMDs per CU
    const int li = sweep_len({&ik, &vv}, slots), lj = sweep_len({&jj}, slots);
    const std::vector<SweepTile> tabs[3] = {sweep_tiles(ik, li), sweep_tiles(jj, lj), sweep_tiles(vv, li)};
    SweepTile** dst[3] = {&p->d_sweep_ik, &p->d_sweep_j, &p->d_sweep_v};
    int* cnt[3] = {&p->nsweep_ik, &p->nsweep_j, &p->nsweep_v};
    for (int t = 0; t < 3; ++t) {
      *cnt[t] = (int)tabs[t].size();
      tables.table(dst[t], tabs[t]);
    }
  }
  tables.scratch(&p->d_monitor, p->persistent_grid);
  if (!tables.make(&p->d_tables)) return fail(FAMRDP_E_HIP, "plan_create: table upload failed");
  *out = p;
  owner.p = nullptr;
  return FAMRDP_OK;
}

}  // namespace

extern "C" {

int famrdp_plan_create(famrdp_plan** out, int32_t nblocks, const int32_t* dims, int32_t ncut, const famrdp_cut* cuts,
                       int32_t nbc, const famrdp_bc* bcs, const famrdp_gas* gas, int32_t limiter, int32_t ghost,
                       int32_t plan_flags) {
  if (!out) return fail(FAMRDP_E_INVALID, "plan_create: out is NULL");
  *out = nullptr;
  try {   // its tables grow with the blocks: nothing may leave a C entry
    return plan_create_impl(out, nblocks, dims, ncut, cuts, nbc, bcs, gas, limiter, ghost, plan_flags);
  } catch (const std::exception&) {
    return fail(FAMRDP_E_HIP, "plan_create: out of host memory for the plan's tables");
  }
}

int famrdp_plan_set_tile(famrdp_plan* p, int32_t variant) {
  if (!p || variant < 0 || variant >= NUM_TILE_VARIANTS) return fail(FAMRDP_E_INVALID, "set_tile: bad plan or variant");
  if (!variant_fits(p, variant))
    return fail(FAMRDP_E_INVALID, "set_tile: variant " + std::to_string(variant) +
                                      " addresses a block's kxyz with 32-bit offsets (blocks under 59,652,323 cells)");
  p->tile_variant = variant;
  if (p->graph_exec) { (void)hipGraphExecDestroy(p->graph_exec); p->graph_exec = nullptr; }
  if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
  return FAMRDP_OK;
}

int famrdp_plan_get_tile(const famrdp_plan* p, int32_t* variant, int32_t* dims3) {
  if (!p) return fail(FAMRDP_E_INVALID, "get_tile: plan is NULL");
  if (variant) *variant = batched_variant(p);
  if (dims3) {
    tile_dims(batched_variant(p), dims3[0], dims3[1], dims3[2]);
    dims3[0] = p->len3[batched_variant(p)];
  }
  return FAMRDP_OK;
}

int famrdp_plan_autotune(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol,
                         double dt, int32_t flags, int32_t reps, double* ms_out, void* stream) {
  if (!p || !kxyz || !vol || reps < 1) return fail(FAMRDP_E_INVALID, "autotune: bad arguments");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "autotune: plan was created without stage workspace");
  int rc = bind(p, q, kxyz, vol, S(stream));
  if (rc) return rc;
  hipStream_t st = S(stream);
  struct Events {   // given back however the tuning ends
    hipEvent_t e[3] = {nullptr, nullptr, nullptr};
    ~Events() {
      for (hipEvent_t x : e)
        if (x) (void)hipEventDestroy(x);
    }
  } ev;
  for (hipEvent_t& e : ev.e) HIP_TRY(hipEventCreate(&e));
  // stages 1 and 2 of variant v n times.  They read q (and q1) and write the
  // q1, q2 workspace only: the state is untouched; stage 2 also reads q0, as
  // stage 3 does.
  auto pairs = [&](int v, int n) -> int {
    for (int stage = 0; stage < 2 * n; ++stage) {
      if (flags & FAMRDP_STEP_BATCHED) {
        launch_fused_batched(v, p->d_blocks, p->d_tiles3[v], p->ntiles3[v], 1 + stage % 2, p->gas, p->limiter, dt,
                             p->len3[v], st);
      } else {
        for (int b = 0; b < p->nblocks; ++b)
          launch_fused(v, p->h_blocks[b], 1 + stage % 2, p->gas, p->limiter, dt, p->ncu, st);
      }
      LAUNCH_CHECK();
    }
    return FAMRDP_OK;
  };
  auto first = [&](int v, float& cold, float& warm) -> int {
    for (int i = 0; i < 3; ++i) {
      HIP_TRY(hipEventRecord(ev.e[i], st));
      if (i < 2 && (rc = pairs(v, 1))) return rc;
    }
    HIP_TRY(hipEventSynchronize(ev.e[2]));
    HIP_TRY(hipEventElapsedTime(&cold, ev.e[0], ev.e[1]));
    HIP_TRY(hipEventElapsedTime(&warm, ev.e[1], ev.e[2]));
    return FAMRDP_OK;
  };
  auto rest = [&](int v, int n, float& t) -> int {
    HIP_TRY(hipEventRecord(ev.e[0], st));
    if ((rc = pairs(v, n))) return rc;
    HIP_TRY(hipEventRecord(ev.e[1], st));
    HIP_TRY(hipEventSynchronize(ev.e[1]));
    HIP_TRY(hipEventElapsedTime(&t, ev.e[0], ev.e[1]));
    t /= n;
    return FAMRDP_OK;
  };
  bool fits[NUM_TILE_VARIANTS];
  float ms[NUM_TILE_VARIANTS];
  for (int v = 0; v < NUM_TILE_VARIANTS; ++v) fits[v] = variant_fits(p, v);
  int best = 0;
  rc = tune_variants(NUM_TILE_VARIANTS, fits, reps, first, rest, ms, best);
  if (rc) return rc;
  for (int v = 0; ms_out && v < NUM_TILE_VARIANTS; ++v) ms_out[v] = fits[v] ? ms[v] : 1e30;
  return famrdp_plan_set_tile(p, best);
}

int famrdp_plan_set_block_params(famrdp_plan* p, const double* mu0, const double* dt_scale) {
  if (!p) return fail(FAMRDP_E_INVALID, "set_block_params: plan is NULL");
  for (int b = 0; b < p->nblocks; ++b) {
    if (mu0) p->h_blocks[b].mu0 = mu0[b];
    if (dt_scale) p->h_blocks[b].dt_scale = dt_scale[b];
    if (p->has_adjoint) {
      p->h_blocks_adj[b].mu0 = p->h_blocks[b].mu0;
      p->h_blocks_adj[b].dt_scale = p->h_blocks[b].dt_scale;
    }
  }
  p->blocks_uploaded = false;   // re-uploaded by the next bind
  if (p->graph_exec) { (void)hipGraphExecDestroy(p->graph_exec); p->graph_exec = nullptr; }
  if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
  return FAMRDP_OK;
}

}  // extern "C"

namespace {

// Reverse of one step; the stage-1/2 states are recomputed from q_start, or
// copied from q1s/q2s when the caller kept them from the forward step.
int step_vjp_impl(famrdp_plan* p, double* const* q_start, const double* const* q1s, const double* const* q2s,
                  const double* const* kxyz, const double* const* vol, double* const* lam, double dt, double* dqinf,
                  int32_t flags, void* stream) {
  if (!p || !q_start || !kxyz || !vol || !lam) return fail(FAMRDP_E_INVALID, "step_vjp: bad arguments");
  if (!p->has_adjoint) return fail(FAMRDP_E_INVALID, "step_vjp: plan was created without FAMRDP_PLAN_ADJOINT");
  for (int b = 0; b < p->nblocks; ++b)
    if (!kxyz[b] || !vol[b] || !lam[b] || !q_start[b] || (q1s && (!q1s[b] || !q2s[b])))
      return fail(FAMRDP_E_INVALID, "step_vjp: NULL pointer for block " + std::to_string(b));
  hipStream_t st = S(stream);
  // metrics only: every reverse kernel reads the adjoint table (state qh),
  // and q_start is read by the copy below
  int rc = bind(p, nullptr, kxyz, vol, st, false);
  if (rc) return rc;
  // The adjoint table reads the caller's arrays where it can instead of
  // copies of them: the stage states when supplied (read only), lam as the
  // cotangent of the post-halo/BC state l0 -- it enters stage 3 there, which
  // scales it in place (each cell reads and then writes its own), stages 2
  // and 1 add to it and the BC and halo reverses finish the result in it --
  // and q_start itself as the state the halo and BCs are applied to when the
  // caller gives it up.
  const bool consume = (flags & FAMRDP_VJP_CONSUME_START) != 0;
  bool rebind = false;
  for (int b = 0; b < p->nblocks; ++b) {
    BlockDesc& a = p->h_blocks_adj[b];
    double* qh = consume ? q_start[b] : p->adj_bufs[6 * b];   // adj_bufs: qh, la, lb, (l0), fs, vs per block
    double* q1 = q1s ? const_cast<double*>(q1s[b]) : p->q1[b];
    double* q2 = q1s ? const_cast<double*>(q2s[b]) : p->q2[b];
    double* la = p->adj_bufs[6 * b + 1];
    if (a.qh != qh || a.q != qh || a.q1 != q1 || a.q2 != q2 || a.la != la || a.l0 != lam[b]) rebind = true;
    a.qh = qh;
    a.q = qh;
    a.q1 = q1;
    a.q2 = q2;
    a.la = la;
    a.l0 = lam[b];
  }
  if (rebind) {
    rc = upload_table(p, p->d_blocks_adj, p->h_blocks_adj, st);
    if (rc) return rc;
  }
  // ---- q0' = BC(halo(q_start)) into qh (BC snapshots kept), then stages 1-2
  if (!consume) {
    rc = copy_blocks(p, st, [&](int b) { return p->h_blocks_adj[b].qh; }, [&](int b) { return q_start[b]; });
    if (rc) return rc;
  }
  rc = launch_ghosts(p, st, p->d_blocks_adj, true);
  if (rc) return rc;
  if (!q1s) {
    rc = launch_stages(p, dt, flags & ~FAMRDP_VJP_CONSUME_START, st, true, 2);
    if (rc) return rc;
  }
  // ---- reverse the three stages
  for (int stage = 3; stage >= 1; --stage) {
    launch_stage_vjp(p->d_blocks_adj, p->d_sweep_v, p->nsweep_v, p->d_sweep_ik, p->nsweep_ik, p->d_sweep_j, p->nsweep_j,
                     stage, p->gas, dt, p->limiter, st);
    LAUNCH_CHECK();
  }
  // ---- BCs reversed (Face order backwards), then the halo copy
  for (int f = 5; f >= 0; --f) {
    if (p->nbc[f] == 0) continue;
    dim3 grid(nblk(p->bc_maxcells[f]), (unsigned)p->nbc[f]);
    k_bc_face_vjp<<<grid, 256, 0, st>>>(p->d_blocks_adj, p->d_bc[f], p->ghost, p->gas.gamma, p->gas.R,
                                        p->d_bc_snap[f], p->d_bc_part[f], p->bc_maxcells[f]);
    LAUNCH_CHECK();
    k_bc_reduce<<<dim3(BC_RED_PARTS, (unsigned)p->nbc[f]), 256, 0, st>>>(p->d_blocks_adj, p->d_bc[f],
                                                                        p->d_bc_part[f], p->bc_maxcells[f],
                                                                        p->d_bc_red[f]);
    LAUNCH_CHECK();
    k_bc_reduce_final<<<p->nbc[f], 64, 0, st>>>(p->d_bc[f], p->d_bc_red[f], dqinf);
    LAUNCH_CHECK();
  }
  if (p->nhalo > 0) {
    k_halo_vjp_gather<<<nblk(p->nhalo_src), 256, 0, st>>>(p->d_blocks_adj, p->d_halo_src, p->nhalo_src,
                                                          p->d_halo_sorted, p->d_halo_S);
    LAUNCH_CHECK();
    k_halo_vjp_clear<<<nblk(p->nhalo), 256, 0, st>>>(p->d_blocks_adj, p->d_halo, p->nhalo);
    LAUNCH_CHECK();
    k_halo_vjp_apply<<<nblk(p->nhalo_src), 256, 0, st>>>(p->d_blocks_adj, p->d_halo_src, p->nhalo_src, p->d_halo_S);
    LAUNCH_CHECK();
  }
  return FAMRDP_OK;
}

}  // namespace

extern "C" {

int famrdp_step_vjp(famrdp_plan* p, double* const* q_start, const double* const* kxyz, const double* const* vol,
                    double* const* lam, double dt, double* dqinf, int32_t flags, void* stream) {
  return step_vjp_impl(p, q_start, nullptr, nullptr, kxyz, vol, lam, dt, dqinf, flags, stream);
}

int famrdp_step_vjp_stages(famrdp_plan* p, double* const* q_start, const double* const* q1, const double* const* q2,
                           const double* const* kxyz, const double* const* vol, double* const* lam, double dt,
                           double* dqinf, int32_t flags, void* stream) {
  if (!q1 || !q2) return fail(FAMRDP_E_INVALID, "step_vjp_stages: stage-state arrays are NULL");
  return step_vjp_impl(p, q_start, q1, q2, kxyz, vol, lam, dt, dqinf, flags, stream);
}

int famrdp_plan_stage_states(famrdp_plan* p, double* const* q1_out, double* const* q2_out, void* stream) {
  if (!p || !q1_out || !q2_out) return fail(FAMRDP_E_INVALID, "stage_states: bad arguments");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "stage_states: plan has no stage workspace");
  hipStream_t st = S(stream);
  for (int b = 0; b < p->nblocks; ++b)
    if (!q1_out[b] || !q2_out[b]) return fail(FAMRDP_E_INVALID, "stage_states: NULL pointer for block " + std::to_string(b));
  int rc = copy_blocks(p, st, [&](int b) { return q1_out[b]; },
                       [&](int b) { return static_cast<const double*>(p->q1[b]); });
  if (rc) return rc;
  return copy_blocks(p, st, [&](int b) { return q2_out[b]; },
                     [&](int b) { return static_cast<const double*>(p->q2[b]); });
}

int famrdp_objective(int32_t kind, const double* q, const double* kxyz, const double* vol, int32_t ni, int32_t nj,
                     int32_t nk, int32_t ghost, double gamma, double* J, double* grad, double* work, void* stream) {
  if ((kind != 0 && kind != 1) || !q || !kxyz || !vol || !J || !grad || !work || ni < 1 || nj < 1 || nk < 1)
    return fail(FAMRDP_E_INVALID, "objective: bad arguments");
  const int parts = 1024;
  k_objective<<<parts, 256, 0, S(stream)>>>(kind, q, kxyz, vol, ni, nj, nk, ghost, gamma, grad, work);
  LAUNCH_CHECK();
  k_sum_final<<<1, 256, 0, S(stream)>>>(work, parts, J);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_plan_check_state(famrdp_plan* p, double* const* q, double* out, void* stream) {
  if (!p || !out) return fail(FAMRDP_E_INVALID, "check_state: NULL plan or output");
  int rc = bind(p, q, nullptr, nullptr, S(stream));
  if (rc) return rc;
  k_monitor_partial<<<p->persistent_grid, 256, 0, S(stream)>>>(p->d_blocks, p->d_tiles, p->ntiles, p->ghost,
                                                               p->gas.gamma, p->d_monitor);
  LAUNCH_CHECK();
  k_sum_parts<<<1, 256, 0, S(stream)>>>(p->d_monitor, p->persistent_grid, out);
  LAUNCH_CHECK();
  return FAMRDP_OK;
}

int famrdp_halo_exchange(famrdp_plan* p, double* const* q, void* stream) {
  if (!p) return fail(FAMRDP_E_INVALID, "plan is NULL");
  int rc = bind(p, q, nullptr, nullptr, S(stream));
  if (rc) return rc;
  return launch_halo(p, S(stream));
}

int famrdp_apply_bc(famrdp_plan* p, double* const* q, void* stream) {
  if (!p) return fail(FAMRDP_E_INVALID, "plan is NULL");
  int rc = bind(p, q, nullptr, nullptr, S(stream));
  if (rc) return rc;
  return launch_bc(p, S(stream));
}

int famrdp_step(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol, double dt,
                int32_t flags, void* stream) {
  if (!p || !kxyz || !vol) return fail(FAMRDP_E_INVALID, "step: NULL plan or metric pointer arrays");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "step: plan was created without stage workspace");
  for (int b = 0; b < p->nblocks; ++b)
    if (!kxyz[b] || !vol[b]) return fail(FAMRDP_E_INVALID, "step: NULL kxyz/vol for block " + std::to_string(b));
  int rc = bind(p, q, kxyz, vol, S(stream));
  if (rc) return rc;
  return run_step(p, dt, flags, S(stream));
}

int famrdp_step_from(famrdp_plan* p, const double* const* q_in, double* const* q, const double* const* kxyz,
                     const double* const* vol, double dt, int32_t flags, void* stream) {
  if (!p || !q_in || !kxyz || !vol) return fail(FAMRDP_E_INVALID, "step_from: NULL plan or pointer arrays");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "step_from: plan was created without stage workspace");
  for (int b = 0; b < p->nblocks; ++b)
    if (!q_in[b] || !kxyz[b] || !vol[b])
      return fail(FAMRDP_E_INVALID, "step_from: NULL q_in/kxyz/vol for block " + std::to_string(b));
  // the launch that copies fills ghost cells from other blocks' q_in meanwhile
  if (q && states_overlap(p, q_in, q)) return fail(FAMRDP_E_INVALID, "step_from: an array of q_in shares memory with one of q");
  hipStream_t st = S(stream);
  hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &capture) != hipSuccess) (void)hipGetLastError();   // (the launch will say)
  p->table_in_graph |= capture != hipStreamCaptureStatusNone;
  bool changed, changed_adj;
  int rc = bind_host(p, q, kxyz, vol, true, nullptr, nullptr, changed, changed_adj);
  if (rc) return rc;
  p->blocks_uploaded = false;
  if (p->has_adjoint && changed_adj && (rc = upload_adj(p, st))) return rc;
  if (p->nblocks <= STEP_START_BLOCKS) {
    StepStart ss{};
    for (int b = 0; b < p->nblocks; ++b) {
      ss.block[b] = p->h_blocks[b];
      ss.src[b] = q_in[b];
    }
    const int n = p->nghost_direct + p->nghost_staged + p->nghost_late + p->nghost_kept;
    k_step_start<<<p->ntiles + nblk(n), 256, 0, st>>>(ss, p->d_blocks, p->nblocks, p->d_tiles, p->ntiles, p->ghost,
                                                      p->d_ghost, n, p->d_chains, p->d_ops, p->gas.gamma, p->gas.R);
    LAUNCH_CHECK();
    p->blocks_uploaded = true;
    return launch_stages(p, dt, flags, st);
  }
  for (int b0 = 0; b0 < p->nblocks; b0 += STEP_START_BLOCKS) {
    const int n = std::min(STEP_START_BLOCKS, p->nblocks - b0);
    StepStart ss{};
    int64_t most = 0;
    for (int b = 0; b < n; ++b) {
      ss.block[b] = p->h_blocks[b0 + b];
      ss.src[b] = q_in[b0 + b];
      most = std::max(most, p->N[b0 + b]);
    }
    // four 16-byte accesses per thread, until the chip is full
    const int gx = (int)std::min<int64_t>((5 * most + 2047) / 2048, 4096);
    k_step_copy<<<dim3(gx, n), 256, 0, st>>>(ss, p->d_blocks + b0);
    LAUNCH_CHECK();
  }
  p->blocks_uploaded = true;
  return run_step(p, dt, flags, st);
}
int famrdp_step_stages(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol,
                       double dt, int32_t flags, double* const* q1_out, double* const* q2_out, void* stream) {
  if (!p || !kxyz || !vol || !q1_out || !q2_out) return fail(FAMRDP_E_INVALID, "step_stages: NULL plan or pointer arrays");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "step_stages: plan was created without stage workspace");
  for (int b = 0; b < p->nblocks; ++b) {
    if (!kxyz[b] || !vol[b] || !q1_out[b] || !q2_out[b])
      return fail(FAMRDP_E_INVALID, "step_stages: NULL kxyz/vol/q1/q2 for block " + std::to_string(b));
    if (q && (q1_out[b] == q[b] || q2_out[b] == q[b] || q1_out[b] == q2_out[b]))
      return fail(FAMRDP_E_INVALID, "step_stages: q, q1 and q2 of block " + std::to_string(b) + " must be distinct");
  }
  int rc = bind(p, q, kxyz, vol, S(stream), true, q1_out, q2_out);
  if (rc) return rc;
  return run_step(p, dt, flags, S(stream));
}

int famrdp_step_graph(famrdp_plan* p, double* const* q, const double* const* kxyz, const double* const* vol,
                      double dt, int32_t flags, int32_t nsteps, void* stream) {
  if (!p || !kxyz || !vol || nsteps < 0) return fail(FAMRDP_E_INVALID, "step_graph: bad arguments");
  if (!p->has_workspace) return fail(FAMRDP_E_INVALID, "step_graph: plan was created without stage workspace");
  for (int b = 0; b < p->nblocks; ++b)
    if (!kxyz[b] || !vol[b]) return fail(FAMRDP_E_INVALID, "step_graph: NULL kxyz/vol for block " + std::to_string(b));
  int rc = bind(p, q, kxyz, vol, S(stream));
  if (rc) return rc;
  std::vector<const void*> key;
  for (int b = 0; b < p->nblocks; ++b) {
    key.push_back(q[b]);
    key.push_back(kxyz[b]);
    key.push_back(vol[b]);
  }
  if (!p->graph_exec || key != p->graph_key || dt != p->graph_dt || flags != p->graph_flags) {
    if (p->graph_exec) { (void)hipGraphExecDestroy(p->graph_exec); p->graph_exec = nullptr; }
    if (p->graph) { (void)hipGraphDestroy(p->graph); p->graph = nullptr; }
    if (!p->cap_stream) HIP_TRY(hipStreamCreateWithFlags(&p->cap_stream, hipStreamNonBlocking));
    HIP_TRY(hipStreamSynchronize(S(stream)));
    HIP_TRY(hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal));
    p->capturing = true;
    rc = run_step(p, dt, flags, p->cap_stream);
    p->capturing = false;
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(p->cap_stream, &g);
    if (rc) { if (g) (void)hipGraphDestroy(g); return rc; }
    if (e != hipSuccess) return fail(FAMRDP_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    p->graph = g;
    HIP_TRY(hipGraphInstantiate(&p->graph_exec, p->graph, nullptr, nullptr, 0));
    p->graph_key = key;
    p->graph_dt = dt;
    p->graph_flags = flags;
  }
  for (int s = 0; s < nsteps; ++s) HIP_TRY(hipGraphLaunch(p->graph_exec, S(stream)));
  return FAMRDP_OK;
}

}  // extern "C"
