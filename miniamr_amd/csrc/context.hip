// context.hip -- context lifetime, host<->device copies, mesh plan upload,
// checksum table, fused stage entry point and timing for libminiamr_dev.so.
#include <stdarg.h>
#include <stdlib.h>
#include <stdio.h>
#include <string.h>
#include <algorithm>
#include <thread>
#include <type_traits>

#include "amr_adjoint.h"
#include "amr_internal.h"

int amr_set_error(amr_dev *d, int rc, const char *fmt, ...)
{
   if (d) {
      va_list ap;
      va_start(ap, fmt);
      vsnprintf(d->err, sizeof(d->err), fmt, ap);
      va_end(ap);
   }
   return rc;
}

int amr_hip_check(amr_dev *d, hipError_t e, const char *what)
{
   return amr_set_error(d, e == hipErrorOutOfMemory ? AMR_ERR_NOMEM : AMR_ERR_HIP,
                        "%s: %s", what, hipGetErrorString(e));
}

static hipEvent_t get_event(amr_dev *d)
{
   if (!d->ev_free.empty()) {
      hipEvent_t e = d->ev_free.back();
      d->ev_free.pop_back();
      return e;
   }
   hipEvent_t e = nullptr;
   if (hipEventCreate(&e) != hipSuccess)
      return nullptr;
   return e;
}

void amr_span_begin(amr_dev *d, int cat)
{
   d->span_skipped = !d->timing || (d->timing_stencil_only && cat != 1);
   if (d->span_skipped)
      return;
   amr_dev::Span s;
   s.a = get_event(d);
   s.b = nullptr;
   s.cat = cat;
   if (s.a)
      hipEventRecord(s.a, d->stream);
   d->spans.push_back(s);
}

void amr_span_end(amr_dev *d)
{
   if (d->span_skipped || d->spans.empty())
      return;
   amr_dev::Span &s = d->spans.back();
   s.b = get_event(d);
   if (s.b)
      hipEventRecord(s.b, d->stream);
}

// The device's address of `bytes` bytes of page-locked host memory at p, or
// null (pageable memory, device memory, or a range that one allocation does
// not hold).  A download writes there with its own kernel: staging the block
// on the device and copying it cost a second launch and pass (3-32 us of a
// block's 20-50).  The runtime reports a range's size in 32 bits, so inside an
// allocation of 4 GiB or more the answer can be null too; the download is then
// a staged one.
static double *device_view(void *p, size_t bytes)
{
   hipPointerAttribute_t a;
   if (hipPointerGetAttributes(&a, p) != hipSuccess) {
      (void) hipGetLastError();   // pageable memory: not an error of ours
      return nullptr;
   }
   if (a.type != hipMemoryTypeHost || !a.devicePointer)
      return nullptr;
   void *start = nullptr;
   size_t size = 0;
   if (hipPointerGetAttribute(&start, HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR,
                              (hipDeviceptr_t) p) != hipSuccess ||
       hipPointerGetAttribute(&size, HIP_POINTER_ATTRIBUTE_RANGE_SIZE, (hipDeviceptr_t) p) !=
          hipSuccess) {
      (void) hipGetLastError();
      return nullptr;
   }
   // the range may be given by the host's or the device's address
   const char *q = (const char *) p, *s = (const char *) start;
   if (q < s || q >= s + size) {
      q = (const char *) a.devicePointer;
      if (q < s || q >= s + size)
         return nullptr;
   }
   return bytes <= size - (size_t) (q - s) ? (double *) a.devicePointer : nullptr;
}

extern "C" {

int amr_dev_create(const amr_dev_config *cfg, amr_dev **out)
{
   if (!out)
      return AMR_ERR_ARG;
   *out = nullptr;
   if (!cfg)
      return AMR_ERR_ARG;
   amr_dev *d = new amr_dev();
   *out = d;
   d->c = *cfg;
   if (cfg->nx < 2 || cfg->ny < 2 || cfg->nz < 2 || (cfg->nx | cfg->ny | cfg->nz) & 1)
      return amr_set_error(d, AMR_ERR_ARG, "block sizes must be even and >= 2");
   if (cfg->num_vars < 1 || cfg->max_blocks < 1)
      return amr_set_error(d, AMR_ERR_ARG, "num_vars and max_blocks must be positive");
   if (cfg->stencil != 0 && cfg->stencil != 7 && cfg->stencil != 27)
      return amr_set_error(d, AMR_ERR_ARG, "stencil must be 0, 7 or 27");
   if (cfg->precision < AMR_PREC_F64 || cfg->precision > AMR_PREC_BF16)
      return amr_set_error(d, AMR_ERR_ARG, "unknown precision %d", cfg->precision);

   int ndev = 0;
   if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
      return amr_set_error(d, AMR_ERR_NODEV, "no HIP device available");
   if (cfg->device < 0 || cfg->device >= ndev)
      return amr_set_error(d, AMR_ERR_NODEV, "device %d out of range (%d devices)",
                           cfg->device, ndev);
   HIP_TRY(d, hipSetDevice(cfg->device));
   hipDeviceProp_t prop;
   HIP_TRY(d, hipGetDeviceProperties(&prop, cfg->device));
   if (strncmp(prop.gcnArchName, "gfx950", 6) != 0)
      return amr_set_error(d, AMR_ERR_NODEV, "device %d is %s, this library is built for gfx950",
                           cfg->device, prop.gcnArchName);
   if (int rc = amr_noalloc_init(d))   // static scratch of amr_dev_split_noalloc
      return rc;

   d->elem_bytes = cfg->precision == AMR_PREC_F64 ? 8 : cfg->precision == AMR_PREC_F32 ? 4 : 2;
   const char *fz = getenv("MINIAMR_FUSED");
   d->fused_mode = fz ? atoi(fz) : 1;
   if (cfg->stencil == 0)
      d->fused_mode = 0;   // the variable-work stencils read other variables' faces
   d->two_interiors = d->fused_mode != 0;   // second I and ZI
   const RecordLayout rl = make_record_layout(cfg->nx, cfg->ny, cfg->nz, cfg->stencil,
                                              d->elem_bytes, d->two_interiors);
   Lay &g = d->g;
   g = rl.g;
   for (int p = 0; p < 2; p++) {
      d->oI_par[p] = rl.oI_par[p];
      d->oZI_par[p] = rl.oZI_par[p];
   }
   d->par.assign(cfg->num_vars, 0);
   d->stale.assign(cfg->num_vars, 0);
   if (d->two_interiors) {
      d->slot_par.assign((size_t) cfg->num_vars * cfg->max_blocks, 0);
      d->active.assign(cfg->max_blocks, 0);
   }
   int64_t cells = (int64_t) g.gx * g.gy * g.gz;
   g.var_stride = g.rec * cfg->max_blocks;
   size_t pool_bytes = (size_t) g.var_stride * cfg->num_vars * d->elem_bytes;

   HIP_TRY(d, hipStreamCreateWithFlags(&d->stream, hipStreamNonBlocking));
   HIP_TRY(d, hipMalloc(&d->pool, pool_bytes));
   HIP_TRY(d, hipMemsetAsync(d->pool, 0, pool_bytes, d->stream));
   HIP_TRY(d, hipMalloc(&d->d_sorted, sizeof(int32_t) * cfg->max_blocks));
   HIP_TRY(d, hipMalloc(&d->d_partials, sizeof(double) * (size_t) cfg->num_vars * cfg->max_blocks));
   HIP_TRY(d, hipMalloc(&d->d_stage, sizeof(double) * (size_t) cells * cfg->num_vars));
   d->h_pinned_bytes = sizeof(double) * std::max<size_t>(4096, (size_t) cfg->num_vars * 64);
   HIP_TRY(d, hipHostMalloc((void **) &d->h_pinned, d->h_pinned_bytes, hipHostMallocDefault));
   if (cfg->stencil == 0) {
      const size_t bytes = sizeof(unsigned long long) * kCountSlots * kCountStride;
      HIP_TRY(d, hipMalloc(&d->d_check_counts, bytes));
      HIP_TRY(d, hipMemsetAsync(d->d_check_counts, 0, bytes, d->stream));
   }
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   return AMR_OK;
}

int amr_dev_destroy(amr_dev *d)
{
   if (!d)
      return AMR_OK;
   if (d->stream)
      hipStreamSynchronize(d->stream);
   for (auto &s : d->spans) {
      if (s.a) hipEventDestroy(s.a);
      if (s.b) hipEventDestroy(s.b);
   }
   for (auto e : d->ev_free)
      hipEventDestroy(e);
   hipFree(d->pool);
   hipFree(d->d_sorted);
   hipFree(d->d_jobs);
   hipFree(d->d_partials);
   hipFree(d->d_sums);
   hipFree(d->d_stage);
   hipFree(d->d_scratch);
   hipFree(d->d_jobbuf);
   hipFree(d->d_codec);
   hipFree(d->d_msgs);
   hipFree(d->d_cmp);
   hipFree(d->d_fjobs);
   hipFree(d->d_redir);
   hipFree(d->d_faces);
   hipFree(d->d_edges);
   hipFree(d->d_mjobs);
   hipFree(d->d_a0);
   hipFree(d->d_check_counts);
   hipFree(d->d_matwork);
   hipFree(d->mk_blocks);
   hipFree(d->mk_parents);
   hipFree(d->mk_objects);
   hipFree(d->mk_levels);
   hipFree(d->mk_out);
   if (d->h_pinned)
      hipHostFree(d->h_pinned);
   if (d->h_plan)
      hipHostFree(d->h_plan);
   if (d->stream && d->owns_stream)
      hipStreamDestroy(d->stream);
   if (d->mark_stream && d->mark_stream != d->stream)
      hipStreamDestroy(d->mark_stream);
   if (d->h_jobstage)
      hipHostFree(d->h_jobstage);
   amr_tape_free(d);
   delete d;
   return AMR_OK;
}

const char *amr_dev_last_error(const amr_dev *d)
{
   return d ? d->err : "no context";
}

int amr_dev_upload_block(amr_dev *d, int slot, const double *cells)
{
   if (!d || !cells || slot < 0 || slot >= d->c.max_blocks)
      return amr_set_error(d, AMR_ERR_ARG, "upload: slot %d out of range", slot);
   if (amr_require_fresh(d, 0, d->c.num_vars, "upload_block"))   // or later: over these cells
      return AMR_ERR_STATE;
   if (int rc = amr_unify(d, 0, d->c.num_vars))
      return rc;
   size_t bytes = sizeof(double) * (size_t) d->g.gx * d->g.gy * d->g.gz * d->c.num_vars;
   HIP_TRY(d, hipMemcpyAsync(d->d_stage, cells, bytes, hipMemcpyHostToDevice, d->stream));
   int rc = amr_launch_convert_in(d, slot);
   if (rc)
      return rc;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   amr_slot_written(d, slot);
   amr_tape_record(d, AMR_OP_UPLOAD, slot);
   return AMR_OK;
}

int amr_dev_download_block(amr_dev *d, int slot, double *cells)
{
   if (d && amr_require_fresh(d, 0, d->c.num_vars, "download_block"))
      return AMR_ERR_STATE;
   if (!d || !cells || slot < 0 || slot >= d->c.max_blocks)
      return amr_set_error(d, AMR_ERR_ARG, "download: slot %d out of range", slot);
   if (int rc = amr_unify(d, 0, d->c.num_vars))
      return rc;
   if (int rc = amr_slots_current(d, &slot, 1))
      return rc;
   size_t bytes = sizeof(double) * (size_t) d->g.gx * d->g.gy * d->g.gz * d->c.num_vars;
   if (double *direct = device_view(cells, bytes)) {
      int rc = amr_launch_convert_out(d, slot, direct);
      if (rc)
         return rc;
      HIP_TRY(d, hipStreamSynchronize(d->stream));
      return AMR_OK;
   }
   int rc = amr_launch_convert_out(d, slot, d->d_stage);
   if (rc)
      return rc;
   HIP_TRY(d, hipMemcpyAsync(cells, d->d_stage, bytes, hipMemcpyDeviceToHost, d->stream));
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   return AMR_OK;
}

}  // extern "C"

int amr_lay(amr_dev *d, int start, int num, Lay *out)
{
   *out = d->g;
   if (num <= 0)
      return AMR_OK;
   const int p = d->par[start];
   for (int v = start + 1; v < start + num; v++)
      if (d->par[v] != p)
         return amr_set_error(d, AMR_ERR_STATE,
                              "variables %d and %d hold their cells in different copies",
                              start, v);
   out->oI = d->oI_par[p];
   out->oZI = d->oZI_par[p];
   return AMR_OK;
}

Lay amr_lay_other(const amr_dev *d, const Lay &L)
{
   Lay o = L;
   const int p = L.oI == d->oI_par[1] && d->two_interiors ? 1 : 0;
   o.oI = d->oI_par[1 - p];
   o.oZI = d->oZI_par[1 - p];
   return o;
}

// ---- inactive slots and the two interior copies
// A fused stage moves the cells of the active blocks from one interior copy
// to the other; a slot outside the active list keeps its cells where they
// were written.  slot_par remembers that copy, and whatever looks at such a
// slot (a download, the codec, a split or consolidation, a mesh that makes
// it active or reads it) first has its interior and z-plane copies moved.
// The moves travel as kernel arguments: no allocation, nothing to wait for.
struct CopyMove {
   int32_t slot, var, num, from;   // variables [var, var+num), from copy `from`
};
constexpr int kMoves = 64;
struct CopyMoves {
   CopyMove m[kMoves];
};

template <typename T>
static __global__ void k_move_copies(T *__restrict__ pool, CopyMoves mv, Lay L, int4 off, int nI,
                                     int nZ)
{
   const CopyMove m = mv.m[blockIdx.x];
   if ((int) blockIdx.y >= m.num)
      return;
   T *rec = pool + (int64_t) (m.var + blockIdx.y) * L.var_stride + (int64_t) m.slot * L.rec;
   const int sI = m.from ? off.y : off.x, dI = m.from ? off.x : off.y;
   const int sZ = m.from ? off.w : off.z, dZ = m.from ? off.z : off.w;
   for (int t = threadIdx.x; t < nI; t += blockDim.x)
      rec[dI + t] = rec[sI + t];
   for (int t = threadIdx.x; t < nZ; t += blockDim.x)
      rec[dZ + t] = rec[sZ + t];
}

static int move_copies(amr_dev *d, const std::vector<CopyMove> &mv)
{
   const int4 off = make_int4(d->oI_par[0], d->oI_par[1], d->oZI_par[0], d->oZI_par[1]);
   const int nI = d->g.nx * d->g.ny * d->g.nz, nZ = 2 * d->g.nx * d->g.ny;
   for (size_t t = 0; t < mv.size(); t += kMoves) {
      CopyMoves a;
      const int n = (int) std::min<size_t>(kMoves, mv.size() - t);
      memset(&a, 0, sizeof(a));
      memcpy(a.m, &mv[t], sizeof(CopyMove) * n);
      const dim3 grid(n, d->c.num_vars);
      if (d->elem_bytes == 8)
         hipLaunchKernelGGL(k_move_copies<uint64_t>, grid, dim3(256), 0, d->stream,
                            (uint64_t *) d->pool, a, d->g, off, nI, nZ);
      else if (d->elem_bytes == 4)
         hipLaunchKernelGGL(k_move_copies<uint32_t>, grid, dim3(256), 0, d->stream,
                            (uint32_t *) d->pool, a, d->g, off, nI, nZ);
      else
         hipLaunchKernelGGL(k_move_copies<uint16_t>, grid, dim3(256), 0, d->stream,
                            (uint16_t *) d->pool, a, d->g, off, nI, nZ);
      HIP_TRY(d, hipGetLastError());
   }
   return AMR_OK;
}

// The moves that bring slot `slot`, held as `is` says, to the copies `want`.
static void add_moves(std::vector<CopyMove> &mv, int slot, const uint8_t *is, const uint8_t *want,
                      int nv)
{
   for (int v = 0; v < nv;) {
      int e = v + 1;
      while (e < nv && is[e] == is[v] && want[e] == want[v])
         e++;
      if (is[v] != want[v])
         mv.push_back({slot, v, e - v, is[v]});
      v = e;
   }
}

// The cells of variables [start, start+num) go to the first variable's copy:
// fused stages of single variables leave them in different ones, and a launch
// works on one.  A variable's stale ghost planes are filled first, from the
// copy that the move then overwrites.  The inactive slots that the plan's jobs
// read were brought to the copies par named when the plan came, and move along.
int amr_unify(amr_dev *d, int start, int num)
{
   std::vector<CopyMove> mv;
   for (int v = start + 1; v < start + num; v++) {
      if (d->par[v] == d->par[start])
         continue;
      if (int rc = amr_require_fresh(d, v, 1, "variables in different copies"))
         return rc;
      for (int s : d->h_sorted)
         mv.push_back({s, v, 1, d->par[v]});
      for (int s : d->inactive_src) {
         uint8_t &is = d->slot_par[(size_t) s * d->c.num_vars + v];
         if (is == d->par[v])
            mv.push_back({s, v, 1, d->par[v]});
         is = d->par[start];
      }
      d->par[v] = d->par[start];
   }
   return move_copies(d, mv);
}

void amr_slot_written(amr_dev *d, int slot)
{
   if (d->two_interiors)
      memcpy(&d->slot_par[(size_t) slot * d->c.num_vars], d->par.data(), d->c.num_vars);
}

bool amr_slot_current(const amr_dev *d, int slot)
{
   return !d->two_interiors || d->active[slot] ||
          !memcmp(&d->slot_par[(size_t) slot * d->c.num_vars], d->par.data(), d->c.num_vars);
}

int amr_slots_current(amr_dev *d, const int32_t *slots, int n)
{
   std::vector<CopyMove> mv;
   for (int t = 0; t < n; t++)
      if (!amr_slot_current(d, slots[t])) {
         add_moves(mv, slots[t], &d->slot_par[(size_t) slots[t] * d->c.num_vars], d->par.data(),
                   d->c.num_vars);
         amr_slot_written(d, slots[t]);
      }
   return move_copies(d, mv);
}

int amr_home_copies(amr_dev *d)
{
   if (!d->two_interiors)
      return AMR_OK;
   for (int s : d->h_sorted)
      amr_slot_written(d, s);
   const std::vector<uint8_t> home(d->c.num_vars, 0);
   std::vector<CopyMove> mv;
   for (int s = 0; s < d->c.max_blocks; s++)
      add_moves(mv, s, &d->slot_par[(size_t) s * d->c.num_vars], home.data(), d->c.num_vars);
   if (int rc = move_copies(d, mv))
      return rc;
   std::fill(d->slot_par.begin(), d->slot_par.end(), 0);
   std::fill(d->par.begin(), d->par.end(), 0);
   return AMR_OK;
}

// MINIAMR_HOIST=0 keeps every fused job in its own direction's launch (the
// default moves the y and z coarse/fine jobs -- with the edges not folded those
// of blocks without a boundary face -- into the first launch, below).
static bool hoist_on()
{
   static int v = -1;
   if (v < 0) {
      const char *e = getenv("MINIAMR_HOIST");
      v = e ? atoi(e) != 0 : 1;
   }
   return v != 0;
}

// MINIAMR_FOLD_EDGES=0 keeps the 27-point edge extensions of in-place faces
// as exchange jobs (the default folds them into the reads, below).
static bool fold_edges_on()
{
   static int v = -1;
   if (v < 0) {
      const char *e = getenv("MINIAMR_FOLD_EDGES");
      v = e ? atoi(e) != 0 : 1;
   }
   return v != 0;
}

// Edge sources of a fused stage (EdgeSrc).  In the reference a ghost edge
// cell of a block gets its value from the last fill that writes it in a
// stage (27-point stencil, --code 0; ref/comm.c:1597-1688, 1911-1965): a
// same-level y fill copies its source's x-extended rows, a same-level z fill
// the whole ring of its source's z plane, a boundary fill the block's own
// whole plane next to the face; a prolongation or restriction writes no edge
// cell, which then keeps what the slot held (stale).  Following these copies
// back to a cell that is an interior cell, a coarse/fine ghost cell or a
// stale one gives the value the stage's stencil sees.
namespace {

struct Cell { int slot, i, j, k; };

// How a face's ghost plane is filled, when not from a same-level block:
// no job or a coarse/fine one (neither writes ring cells), or the boundary.
enum { FK_NONE = -1, FK_BC = -2, FK_CF = -3 };

struct EdgeResolver {
   const Lay &g;
   const std::vector<int32_t> &kind;   // per slot and face: FK_*, or the same-level source
   Lay L0;   // g with the interior copies at offset 0 (ES_I / ES_ZI offsets)

   EdgeResolver(const Lay &g_, const std::vector<int32_t> &kind_) : g(g_), kind(kind_), L0(g_)
   {
      L0.oI = 0;
      L0.oZI = 0;
   }

   // The cell whose value block b's cell (i, j, k) holds when the stencil
   // runs: follow the last fill that wrote it, then the fill that had written
   // the cell this one read by then (phases x, y, z: `p` is the last phase
   // that counts), and so on.  A cell that no fill of those phases writes
   // holds what the slot held before, except a coarse/fine ghost cell that a
   // boundary fill of an earlier phase read: that is the previous stage's
   // value, which the coarse/fine job copies to the cell of the boundary's
   // edge line before it writes the new one (FusedJob::ring) -- so the chain
   // ends at that edge cell.
   Cell resolve(int b, int i, int j, int k) const
   {
      int p = 2;
      Cell last{b, i, j, k};
      for (int hop = 0; hop < 12; hop++) {
         const bool g3[3] = {i == 0 || i == g.nx + 1, j == 0 || j == g.ny + 1,
                             k == 0 || k == g.nz + 1};
         const int ng = g3[0] + g3[1] + g3[2];
         if (!ng)
            return {b, i, j, k};
         int d = p, src = FK_NONE;
         for (; d >= 0; d--) {
            if (!g3[d])
               continue;
            const int f = d == 0 ? (i != 0) : d == 1 ? 2 + (j != 0) : 4 + (k != 0);
            src = kind[6 * (size_t) b + f];
            // a same-level fill covers the ghosts of earlier directions only
            const bool later = (d < 1 && g3[1]) || (d < 2 && g3[2]);
            if (src == FK_BC || (src >= 0 && !later))
               break;
         }
         if (d < 0) {
            const int e = g3[0] ? 0 : g3[1] ? 1 : 2;
            const int f = 2 * e + (e == 0 ? i != 0 : e == 1 ? j != 0 : k != 0);
            return ng == 1 && e > p && kind[6 * (size_t) b + f] == FK_CF ? last : Cell{b, i, j, k};
         }
         last = {b, i, j, k};
         const bool hi = d == 0 ? i != 0 : d == 1 ? j != 0 : k != 0;
         const int n = d == 0 ? g.nx : d == 1 ? g.ny : g.nz;
         int &c = d == 0 ? i : d == 1 ? j : k;
         if (src == FK_BC) {
            c = hi ? n : 1;
         } else {
            b = src;
            c = hi ? 1 : n;
         }
         p = d - 1;
      }
      return {-1, 0, 0, 0};
   }

   // a cell as an entry: axis is the direction of the line (-1 for a corner);
   // cells at z = 1 / z = nz of lines across z are read from the z-plane copies
   bool entry(const Cell &c, int axis, EdgeSrc &e) const
   {
      if (c.slot < 0)
         return false;
      const bool ghost = c.i == 0 || c.i == g.nx + 1 || c.j == 0 || c.j == g.ny + 1 ||
                         c.k == 0 || c.k == g.nz + 1;
      const bool zc = axis != 2 && (c.k == 1 || c.k == g.nz);
      e.slot = c.slot;
      e.stride = 0;
      if (!ghost) {
         e.kind = zc ? ES_ZI : ES_I;
         e.off = zc ? zcopy(L0, c.i, c.j, c.k) : home(L0, c.i, c.j, c.k);
      } else {
         e.kind = ES_ABS;
         e.off = zc ? zcopy(g, c.i, c.j, c.k) : home(g, c.i, c.j, c.k);
      }
      return true;
   }

   // entry of a line of n cells along `axis` from block b's cell c; false if
   // they are not one affine run.  No copy on the way changes the coordinate
   // along the line, and every cell of the line follows the same fills, so the
   // first cell's source gives the others'.
   bool line(const Cell &c, int axis, int n, bool fold, EdgeSrc &e) const
   {
      const Cell c0 = fold ? resolve(c.slot, c.i, c.j, c.k) : c;
      if (!entry(c0, axis, e))
         return false;
      auto at = [&](int t) {
         Cell x = c0;
         (axis == 0 ? x.i : axis == 1 ? x.j : x.k) += t;
         EdgeSrc y;
         entry(x, axis, y);
         return y;
      };
      if (n > 1) {
         const EdgeSrc e1 = at(1), el = at(n - 1);
         e.stride = e1.off - e.off;
         return e1.kind == e.kind && el.kind == e.kind && el.off == e.off + (n - 1) * e.stride;
      }
      return true;
   }

   // the kEdgeSrcs entries of block b
   bool block(int b, bool fold, EdgeSrc *out) const
   {
      const int X[2] = {0, g.nx + 1}, Y[2] = {0, g.ny + 1}, Z[2] = {0, g.nz + 1};
      bool ok = true;
      for (int xs = 0; xs < 2; xs++)
         for (int ys = 0; ys < 2; ys++)
            ok &= line(Cell{b, X[xs], Y[ys], 1}, 2, g.nz, fold, out[xs * 2 + ys]);
      for (int xs = 0; xs < 2; xs++)
         for (int zs = 0; zs < 2; zs++)
            ok &= line(Cell{b, X[xs], 1, Z[zs]}, 1, g.ny, fold, out[4 + xs * 2 + zs]);
      for (int ys = 0; ys < 2; ys++)
         for (int zs = 0; zs < 2; zs++)
            ok &= line(Cell{b, 1, Y[ys], Z[zs]}, 0, g.nx, fold, out[8 + ys * 2 + zs]);
      for (int xs = 0; xs < 2; xs++)
         for (int ys = 0; ys < 2; ys++)
            for (int zs = 0; zs < 2; zs++)
               ok &= line(Cell{b, X[xs], Y[ys], Z[zs]}, -1, 1, fold, out[12 + xs * 4 + ys * 2 + zs]);
      return ok;
   }
};

}  // namespace

// The plan of amr_dev_stage_fused.  Edges folded (27-point): same-level and
// boundary faces are read in place, edges through the entries above, and only
// coarse/fine jobs remain.  Otherwise a face is read in place when its job is
// a same-level copy and the block has no boundary face (a boundary fill with
// the 27-point extension reads the block's own ghost planes as they were
// before the later phases of the stage); such a face's job is dropped (x, and
// y/z for the 7-point stencil) or reduced to its edge extension (y/z for the
// 27-point stencil), and every job that reads a source's ghost row that is
// read in place is redirected to the block that row would be copied from.
// It is computed on the host only; set_mesh uploads it.
struct FusedPlan {
   std::vector<FusedJob> fj;
   int32_t fc[3] = {0, 0, 0};
   std::vector<EdgeSrc> edges;
   std::vector<int32_t> redir;
   std::vector<FaceSrc> faces;
   bool all_faces = false;
   std::vector<amr_face_job> mj;
   int32_t mc[3] = {0, 0, 0};
   bool fold = false;
};

// The plan's FaceSrc table.  27-point stencil: the faces read in place (same
// level) and the block's own planes.  7-point stencil: every face in place
// when that is possible (all_faces): its jobs read interiors only, at every
// kind, so no ghost plane is needed as long as each has at most one source
// (four quarters for a restriction) and all blocks named are active.  Empty
// where the plane-by-plane kernels serve.
static void face_sources(const amr_dev *d, const int32_t *sorted, int n_active,
                         const amr_face_job *jobs, int nj, FusedPlan &P)
{
   P.all_faces = false;
   P.faces.clear();
   if (!amr_uses_box(d))
      return;
   if (d->g.stencil != 7) {
      P.faces.assign(6 * (size_t) n_active, FaceSrc{FS_OWN, {-1, -1, -1, -1}});
      for (size_t i = 0; i < 6 * (size_t) n_active; i++)
         if (P.redir[i] >= 0)
            P.faces[i] = FaceSrc{FS_SAME, {P.redir[i], -1, -1, -1}};
         else if (P.redir[i] == kRedirBc)
            P.faces[i].kind = FS_BC;
      return;
   }
   std::vector<int32_t> at(d->c.max_blocks, -1);   // slot -> place in sorted
   bool ok = true;
   for (int in = 0; in < n_active; in++) {
      ok &= at[sorted[in]] < 0;
      at[sorted[in]] = in;
   }
   std::vector<FaceSrc> F(6 * (size_t) std::max(n_active, 1), FaceSrc{FS_OWN, {-1, -1, -1, -1}});
   for (int t = 0; t < nj && ok; t++) {
      const amr_face_job &j = jobs[t];
      ok = at[j.dst] >= 0 && at[j.src] >= 0 && !(j.kind & AMR_FACE_GHOSTS);
      if (!ok)
         break;
      FaceSrc &f = F[6 * (size_t) at[j.dst] + j.face];
      if (j.kind == AMR_FACE_RESTRICT) {
         int32_t &q = f.s[j.iq + 2 * j.jq];
         ok = (f.kind == FS_OWN || f.kind == FS_RESTRICT) && q < 0;
         f.kind = FS_RESTRICT;
         q = j.src;
      } else {
         ok = f.kind == FS_OWN;
         if (j.kind == AMR_FACE_SAME) f = FaceSrc{FS_SAME, {j.src, -1, -1, -1}};
         else if (j.kind == AMR_FACE_BC) f = FaceSrc{FS_BC, {-1, -1, -1, -1}};
         else f = FaceSrc{FS_PROLONG, {j.src, j.iq, j.jq, -1}};
      }
   }
   P.all_faces = ok;
   if (!ok)   // the other fused stage: same-level faces in place
      for (size_t i = 0; i < 6 * (size_t) n_active; i++)
         F[i] = P.redir[i] >= 0 ? FaceSrc{FS_SAME, {P.redir[i], -1, -1, -1}}
                                : FaceSrc{FS_OWN, {-1, -1, -1, -1}};
   P.faces.swap(F);
}

static void compute_fused_plan(const amr_dev *d, const int32_t *sorted, int n_active,
                               const amr_face_job *jobs, const int32_t count[3], FusedPlan &P)
{
   const int M = d->c.max_blocks;
   std::vector<int32_t> kind(6 * (size_t) M, FK_NONE);
   std::vector<uint8_t> bc(M, 0), quarters(6 * (size_t) M, 0);
   const int nj = count[0] + count[1] + count[2];
   bool fold = d->g.stencil == 27 && fold_edges_on();
   for (int t = 0; t < nj; t++) {
      const amr_face_job &j = jobs[t];
      const size_t at = 6 * (size_t) j.dst + j.face;
      if (j.kind == AMR_FACE_BC) {
         bc[j.dst] = 1;
         kind[at] = FK_BC;
      } else if (j.kind == AMR_FACE_SAME) {
         kind[at] = j.src;
      } else {
         kind[at] = FK_CF;
         quarters[at] |= j.kind == AMR_FACE_PROLONG ? 15 : 1 << (j.iq + 2 * j.jq);
         fold &= !(j.kind & AMR_FACE_GHOSTS);
      }
   }
   // folding expects whole coarse/fine planes
   for (size_t at = 0; at < kind.size() && fold; at++)
      fold = kind[at] != FK_CF || quarters[at] == 15;
   // Faces read in place: same-level ones and, when edges are folded, the
   // boundary's.  Without folding the jobs of a boundary block all run: a
   // boundary fill with the 27-point extension reads the block's own ghost
   // planes as they were before the later phases of the stage.
   auto inplace = [&](int slot, int f) {
      const int k = kind[6 * (size_t) slot + f];
      return fold ? (k == FK_CF ? FK_NONE : k) : (bc[slot] || k < 0) ? -1 : k;
   };
   // edge sources of every active block: folded (27-point stencil) unless a
   // line is not one affine run, in which case the plan keeps the extensions
   std::vector<EdgeSrc> &edges = P.edges;
   edges.assign(kEdgeSrcs * (size_t) M, EdgeSrc{0, 0, 0, ES_ABS});
   {
      // the blocks are independent: spread them over a few host threads
      // (the resolution takes ~2 ms for 5,500 blocks on one)
      const EdgeResolver R(d->g, kind);
      auto resolve_range = [&](int i0, int i1, bool f) {
         bool ok = true;
         for (int in = i0; in < i1; in++)
            ok &= R.block(sorted[in], f, &edges[kEdgeSrcs * (size_t) sorted[in]]);
         return ok;
      };
      const int nt = n_active >= 2048 ? 8 : 1;
      auto run_all = [&](bool f) {
         if (nt == 1)
            return resolve_range(0, n_active, f);
         std::vector<std::thread> th;
         std::vector<char> ok(nt, 1);
         for (int t = 0; t < nt; t++)
            th.emplace_back([&, t] {
               ok[t] = resolve_range((int) ((int64_t) n_active * t / nt),
                                     (int) ((int64_t) n_active * (t + 1) / nt), f);
            });
         for (auto &x : th)
            x.join();
         return std::all_of(ok.begin(), ok.end(), [](char c) { return c != 0; });
      };
      if (fold)
         fold = run_all(true);
      if (!fold)
         run_all(false);
   }
   P.fold = fold;
   // Jobs by launch.  The y and z prolongations and restrictions of blocks
   // without a boundary face go with the x phase: they read only interior
   // cells, which no job writes, and write ghost cells that only later
   // phases' jobs (27-point rings) and the stencil read -- an x job reads
   // ghost cells only in a boundary fill of its own block.  The y and z
   // launches keep the jobs that read rings -- none when edges are folded:
   // then only coarse/fine jobs are left and one launch holds them all.
   std::vector<FusedJob> ph[3];
   const bool hoist = hoist_on();
   for (int t = 0, dir = 0; dir < 3; dir++)
      for (int e = 0; e < count[dir]; e++, t++) {
         const amr_face_job &j = jobs[t];
         FusedJob f;
         f.jb = j;
         f.mode = FJ_FULL;
         f.alt[0] = f.alt[1] = f.alt[2] = f.alt[3] = -1;
         f.ring = 0;
         if (fold && (j.kind == AMR_FACE_SAME || j.kind == AMR_FACE_BC))
            continue;                       // read where it is, edges included
         if (fold && dir > 0) {
            // boundary faces of earlier phases beside this coarse/fine plane
            for (int f2 = 0; f2 < 2 * dir; f2++)
               f.ring |= (kind[6 * (size_t) j.dst + f2] == FK_BC) << f2;
         }
         if (j.kind == AMR_FACE_SAME && inplace(j.dst, j.face) >= 0) {
            if (dir == 0 || d->g.stencil == 7)
               continue;                    // nothing outside the face interior
            f.mode = FJ_EXT_ONLY;
         }
         if (d->g.stencil == 27 && dir > 0 &&
             (j.kind == AMR_FACE_SAME || j.kind == AMR_FACE_BC)) {
            f.alt[0] = inplace(j.src, 0);
            f.alt[1] = inplace(j.src, 1);
            if (dir == 2) {
               f.alt[2] = inplace(j.src, 2);
               f.alt[3] = inplace(j.src, 3);
            }
         }
         const bool cf = j.kind == AMR_FACE_PROLONG || j.kind == AMR_FACE_RESTRICT;
         ph[hoist && dir > 0 && cf && (fold || !bc[j.dst]) ? 0 : dir].push_back(f);
      }
   // the jobs that bring stale ghost planes up to date (amr_require_fresh)
   std::vector<amr_face_job> &mj = P.mj;
   int32_t *mc = P.mc;
   for (int t = 0, dir = 0; dir < 3; dir++)
      for (int e = 0; e < count[dir]; e++, t++)
         if (!fold && jobs[t].kind == AMR_FACE_SAME && inplace(jobs[t].dst, jobs[t].face) >= 0) {
            mj.push_back(jobs[t]);
            mc[dir]++;
         }
   std::vector<FusedJob> &fj = P.fj;
   fj.reserve(nj);
   for (int p = 0; p < 3; p++) {
      fj.insert(fj.end(), ph[p].begin(), ph[p].end());
      P.fc[p] = (int32_t) ph[p].size();
   }
   P.redir.assign(6 * (size_t) std::max(n_active, 1), -1);
   for (int in = 0; in < n_active; in++)
      for (int f = 0; f < 6; f++)
         P.redir[6 * (size_t) in + f] = inplace(sorted[in], f);   // FK_BC: kRedirBc
   face_sources(d, sorted, n_active, jobs, nj, P);
}

// A fused stage leaves unwritten the ghost cells its stencil reads where
// they are.  The interiors it read them from are still in the record's other
// copy, until the next stage writes it.
//   Edges folded: every such cell is in the tables -- the planes of the faces
// read in place (redir) and the edge entries -- and their sources are
// interior cells, coarse/fine ghost cells and stale edge cells, none of which
// is filled here, so one launch copies them all (k_fill_in_place).
//   Otherwise they are what the same-level jobs of blocks without a boundary
// face write (7-point stages that read every face in place: all jobs).  A
// job's reads of other ghost cells find them as the plain stage's earlier
// phases left them, so rerunning those jobs, in direction order, on the other
// copy gives every ghost cell the plain stage's value.
template <typename T>
static __global__ __launch_bounds__(256) void k_fill_in_place(
   T *__restrict__ pool, const int32_t *__restrict__ sorted, const int32_t *__restrict__ redir,
   const EdgeSrc *__restrict__ edges, Lay L, int var0)
{
   const int slot = sorted[blockIdx.x];
   T *const var = pool + (int64_t) (var0 + blockIdx.y) * L.var_stride;
   T *const rec = var + (int64_t) slot * L.rec;
   auto fill = [&](int i, int j, int k, T v) {
      rec[home(L, i, j, k)] = v;
      if (k == 1 || k == L.nz)
         rec[zcopy(L, i, j, k)] = v;
   };
   for (int f = 0; f < 6; f++) {
      const int from = redir[6 * (int64_t) blockIdx.x + f];
      if (from == -1)
         continue;
      const int dir = f >> 1, hi = f & 1, n = dir == 0 ? L.nx : dir == 1 ? L.ny : L.nz;
      const int na = dir == 0 ? L.ny : L.nx, nb = dir == 2 ? L.ny : L.nz;
      const bool own = from == kRedirBc;   // the block's own plane next to the face
      const T *const src = own ? rec : var + (int64_t) from * L.rec;
      const int ghost = hi ? n + 1 : 0, plane = own == (hi != 0) ? n : 1;
      for (int t = threadIdx.x; t < na * nb; t += blockDim.x) {
         const int a = 1 + t / nb, b = 1 + t % nb;
         const int i = dir == 0 ? ghost : a, j = dir == 0 ? a : dir == 1 ? ghost : b,
                   k = dir == 2 ? ghost : b;
         const int si = dir == 0 ? plane : i, sj = dir == 1 ? plane : j, sk = dir == 2 ? plane : k;
         fill(i, j, k, src[dir == 2 ? zcopy(L, si, sj, sk) : home(L, si, sj, sk)]);
      }
   }
   const EdgeSrc *const es = edges + (int64_t) kEdgeSrcs * slot;
   const int nz4 = 4 * L.nz, ny4 = 4 * L.ny, nx4 = 4 * L.nx;
   for (int e = threadIdx.x; e < nz4 + ny4 + nx4 + 8; e += blockDim.x) {
      int i, j, k, line, t;
      if (e < nz4) {
         line = e / L.nz; t = e - line * L.nz;
         i = (line & 2) ? L.nx + 1 : 0; j = (line & 1) ? L.ny + 1 : 0; k = t + 1;
      } else if (e < nz4 + ny4) {
         const int h = e - nz4;
         line = h / L.ny; t = h - line * L.ny;
         i = (line & 2) ? L.nx + 1 : 0; k = (line & 1) ? L.nz + 1 : 0; j = t + 1;
         line += 4;
      } else if (e < nz4 + ny4 + nx4) {
         const int h = e - nz4 - ny4;
         line = h / L.nx; t = h - line * L.nx;
         j = (line & 2) ? L.ny + 1 : 0; k = (line & 1) ? L.nz + 1 : 0; i = t + 1;
         line += 8;
      } else {
         const int h = e - nz4 - ny4 - nx4;
         line = 12 + h; t = 0;
         i = (h & 4) ? L.nx + 1 : 0; j = (h & 2) ? L.ny + 1 : 0; k = (h & 1) ? L.nz + 1 : 0;
      }
      const int64_t from = edge_at(es[line], L, t);
      if (from != (int64_t) slot * L.rec + home(L, i, j, k))
         fill(i, j, k, var[from]);
   }
}

static int launch_fill_in_place(amr_dev *d, const Lay &L, int start, int num)
{
   if (!d->n_active)
      return AMR_OK;
   const dim3 grid(d->n_active, num);
   if (d->elem_bytes == 8)
      hipLaunchKernelGGL(k_fill_in_place<uint64_t>, grid, dim3(256), 0, d->stream,
                         (uint64_t *) d->pool, d->d_sorted, d->d_redir, d->d_edges, L, start);
   else if (d->elem_bytes == 4)
      hipLaunchKernelGGL(k_fill_in_place<uint32_t>, grid, dim3(256), 0, d->stream,
                         (uint32_t *) d->pool, d->d_sorted, d->d_redir, d->d_edges, L, start);
   else
      hipLaunchKernelGGL(k_fill_in_place<uint16_t>, grid, dim3(256), 0, d->stream,
                         (uint16_t *) d->pool, d->d_sorted, d->d_redir, d->d_edges, L, start);
   HIP_TRY(d, hipGetLastError());
   return AMR_OK;
}

int amr_require_fresh(amr_dev *d, int start, int num, const char *what)
{
   const int end = std::min(start + num, (int) d->stale.size());
   for (int a = start; a < end;) {
      if (!d->stale[a]) {
         a++;
         continue;
      }
      int b = a + 1;   // a run of stale variables whose cells are in one copy
      while (b < end && d->stale[b] && d->par[b] == d->par[a])
         b++;
      Lay L;
      if (int rc = amr_lay(d, a, b - a, &L))
         return rc;
      const Lay Lr = amr_lay_other(d, L);
      if (d->fold_edges) {
         if (int rc = launch_fill_in_place(d, Lr, a, b - a))
            return rc;
         for (int v = a; v < b; v++)
            d->stale[v] = 0;
         a = b;
         continue;
      }
      const amr_face_job *jobs = d->all_faces ? d->d_jobs : d->d_mjobs;
      const int32_t *cnt = d->all_faces ? d->count : d->mcount;
      for (int dir = 0, off = 0; dir < 3; off += cnt[dir], dir++)
         if (int rc = amr_launch_exchange_jobs(d, jobs + off, cnt[dir], Lr, a, b - a))
            return amr_set_error(d, rc, "%s: bringing ghost planes up to date: %s", what,
                                 d->err);
      for (int v = a; v < b; v++)
         d->stale[v] = 0;
      a = b;
   }
   return AMR_OK;
}

int amr_set_mesh_impl(amr_dev *d, const int32_t *sorted, int n_active,
                      const amr_face_job *jobs, const int32_t count[3])
{
   if (!d || n_active < 0 || n_active > d->c.max_blocks || (n_active && !sorted) || !count)
      return amr_set_error(d, AMR_ERR_ARG, "set_mesh: bad arguments");
   int nj = 0;
   for (int i = 0; i < 3; i++) {
      if (count[i] < 0)
         return amr_set_error(d, AMR_ERR_ARG, "set_mesh: negative job count");
      nj += count[i];
   }
   if (nj && !jobs)
      return amr_set_error(d, AMR_ERR_ARG, "set_mesh: jobs missing");
   if (int rc = amr_require_fresh(d, 0, d->c.num_vars, "set_mesh"))
      return rc;
   // Validate every job on the host: slots in range and faces/quarters legal,
   // so no kernel can address outside the pool.
   for (int i = 0; i < n_active; i++)
      if (sorted[i] < 0 || sorted[i] >= d->c.max_blocks)
         return amr_set_error(d, AMR_ERR_ARG, "set_mesh: slot %d out of range", sorted[i]);
   for (int t = 0; t < nj; t++) {
      const amr_face_job &j = jobs[t];
      int dir = t < count[0] ? 0 : t < count[0] + count[1] ? 1 : 2;
      if (j.kind < AMR_FACE_SAME || j.kind > AMR_FACE_BC_GHOSTS || j.face / 2 != dir ||
          j.face < 0 || j.face > 5 || j.dst < 0 || j.dst >= d->c.max_blocks ||
          j.src < 0 || j.src >= d->c.max_blocks || (j.iq & ~1) || (j.jq & ~1))
         return amr_set_error(d, AMR_ERR_ARG, "set_mesh: bad face job %d", t);
   }
   if (d->two_interiors) {
      for (int x : d->h_sorted) {   // slots that leave the list stay where they are
         amr_slot_written(d, x);
         d->active[x] = 0;
      }
      std::vector<int32_t> used(sorted, sorted + n_active);
      std::vector<uint8_t> act(d->c.max_blocks, 0);
      for (int i = 0; i < n_active; i++)
         act[sorted[i]] = 1;
      d->closed = true;
      std::vector<int32_t> outside;   // inactive slots the jobs read, each once
      std::vector<uint8_t> seen(d->c.max_blocks, 0);
      for (int t = 0; t < nj; t++) {
         const int s = jobs[t].src;
         if (!act[s] && !seen[s])
            outside.push_back(s);
         seen[s] = 1;
         d->closed &= act[s] && act[jobs[t].dst];
      }
      used.insert(used.end(), outside.begin(), outside.end());
      if (int rc = amr_slots_current(d, used.data(), (int) used.size()))
         return rc;
      d->active.swap(act);
      d->inactive_src.swap(outside);
   }
   // The fused plan is host work; it runs before the wait below, so it
   // overlaps the device work still queued (split and consolidate data).
   FusedPlan fp;
   if (d->two_interiors)
      compute_fused_plan(d, sorted, n_active, jobs, count, fp);
   // Queued work may still read the old plan and the staging buffer may
   // still feed the last set_mesh's copies: wait, then replace.
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   auto grow = [&](void **buf, int *cap, int need, size_t elem) -> int {
      if (need <= *cap)
         return AMR_OK;
      const int c = std::max(need, 2 * *cap);
      hipFree(*buf);
      *buf = nullptr;
      *cap = 0;
      HIP_TRY(d, hipMalloc(buf, elem * (size_t) c));
      *cap = c;
      return AMR_OK;
   };
   if (int rc = grow((void **) &d->d_jobs, &d->jobs_cap, nj, sizeof(amr_face_job)))
      return rc;
   if (d->two_interiors) {
      if (int rc = grow((void **) &d->d_fjobs, &d->fjobs_cap, (int) fp.fj.size(), sizeof(FusedJob)))
         return rc;
      if (int rc = grow((void **) &d->d_mjobs, &d->mjobs_cap, (int) fp.mj.size(),
                        sizeof(amr_face_job)))
         return rc;
      if (!d->d_edges)
         HIP_TRY(d, hipMalloc(&d->d_edges, sizeof(EdgeSrc) * fp.edges.size()));
      if (!d->d_redir)
         HIP_TRY(d, hipMalloc(&d->d_redir, sizeof(int32_t) * 6 * (size_t) d->c.max_blocks));
      if (!d->d_faces && !fp.faces.empty())
         HIP_TRY(d, hipMalloc(&d->d_faces, sizeof(FaceSrc) * 6 * (size_t) d->c.max_blocks));
   }
   // One pinned staging buffer, then copies ordered on the stream before
   // any later launch (pageable hipMemcpy of the ~3 MB plan took 0.5-2 ms).
   struct Piece {
      void *dst;
      const void *src;
      size_t bytes;
   };
   std::vector<Piece> pieces;
   pieces.push_back({d->d_sorted, sorted, sizeof(int32_t) * (size_t) n_active});
   pieces.push_back({d->d_jobs, jobs, sizeof(amr_face_job) * (size_t) nj});
   if (d->two_interiors) {
      pieces.push_back({d->d_fjobs, fp.fj.data(), sizeof(FusedJob) * fp.fj.size()});
      pieces.push_back({d->d_edges, fp.edges.data(), sizeof(EdgeSrc) * fp.edges.size()});
      pieces.push_back({d->d_redir, fp.redir.data(), sizeof(int32_t) * fp.redir.size()});
      pieces.push_back({d->d_faces, fp.faces.data(), sizeof(FaceSrc) * fp.faces.size()});
      pieces.push_back({d->d_mjobs, fp.mj.data(), sizeof(amr_face_job) * fp.mj.size()});
   }
   size_t total = 0;
   for (const Piece &q : pieces)
      total += (q.bytes + 255) / 256 * 256;
   if (total > d->h_plan_bytes) {
      if (d->h_plan)
         hipHostFree(d->h_plan);
      d->h_plan = nullptr;
      d->h_plan_bytes = 0;
      HIP_TRY(d, hipHostMalloc(&d->h_plan, total, hipHostMallocDefault));
      d->h_plan_bytes = total;
   }
   size_t at = 0;
   for (const Piece &q : pieces) {
      if (!q.bytes)
         continue;
      char *h = (char *) d->h_plan + at;
      memcpy(h, q.src, q.bytes);
      HIP_TRY(d, hipMemcpyAsync(q.dst, h, q.bytes, hipMemcpyHostToDevice, d->stream));
      at += (q.bytes + 255) / 256 * 256;
   }
   d->h_sorted.assign(sorted, sorted + n_active);
   d->n_active = n_active;
   for (int i = 0; i < 3; i++)
      d->count[i] = count[i];
   d->whole_ghosts = false;
   for (int t = 0; t < nj; t++)
      d->whole_ghosts |= (jobs[t].kind & AMR_FACE_GHOSTS) != 0;
   d->plan_version++;
   if (d->two_interiors) {
      d->fold_edges = fp.fold;
      d->all_faces = fp.all_faces;
      for (int i = 0; i < 3; i++) {
         d->fcount[i] = fp.fc[i];
         d->mcount[i] = fp.mc[i];
      }
   }
   return AMR_OK;
}

int amr_comm_impl(amr_dev *d, int start, int num, int stage, int permute)
{
   static const int perm[6][3] = { {0, 1, 2}, {1, 2, 0}, {2, 0, 1},
                                   {0, 2, 1}, {1, 0, 2}, {2, 1, 0} };
   if (!d || start < 0 || num < 0 || start + num > d->c.num_vars || stage < 0)
      return amr_set_error(d, AMR_ERR_ARG, "comm: variables [%d, %d) out of range", start,
                           start + num);
   if (!num)
      return AMR_OK;
   if (amr_order_reads_ghosts(d->g.stencil, stage, permute))
      if (int rc = amr_require_fresh(d, start, num, "comm"))
         return rc;
   if (int rc = amr_unify(d, start, num))
      return rc;
   // one span per direction when timing per direction, else one in all
   if (!d->timing_dirs)
      amr_span_begin(d, 0);
   for (int o = 0; o < 3; o++) {
      int dir = permute ? perm[stage % 6][o] : o;
      if (d->timing_dirs)
         amr_span_begin(d, kSpanExchangeX + dir);
      int rc = amr_launch_exchange_dir(d, dir, start, num);
      if (d->timing_dirs)
         amr_span_end(d);
      if (rc)
         return rc;
   }
   if (!d->timing_dirs)
      amr_span_end(d);
   // every ghost cell of these variables is written again
   for (int v = start; v < start + num; v++)
      d->stale[v] = 0;
   return AMR_OK;
}

int amr_stencil_impl(amr_dev *d, int var, int calc_stage)
{
   if (!d || var < 0 || var >= d->c.num_vars || calc_stage < 0)
      return amr_set_error(d, AMR_ERR_ARG, "stencil: variable %d out of range", var);
   if (int rc = amr_require_fresh(d, var, 1, "stencil"))
      return rc;
   amr_span_begin(d, 1);
   int rc = amr_launch_stencil(d, var, 1, false, calc_stage);
   amr_span_end(d);
   return rc;
}

extern "C" {

int amr_dev_set_mesh(amr_dev *d, const int32_t *sorted, int n_active,
                     const amr_face_job *jobs, const int32_t count[3])
{
   int rc = amr_set_mesh_impl(d, sorted, n_active, jobs, count);
   if (rc || !d->tape || !d->tape->on || d->replaying)
      return rc;
   TapePlan pl;
   pl.sorted.assign(sorted, sorted + n_active);
   pl.jobs.assign(jobs, jobs + (count[0] + count[1] + count[2]));
   for (int i = 0; i < 3; i++)
      pl.count[i] = count[i];
   d->tape->plans.push_back(std::move(pl));
   d->tape->cur_plan = (int) d->tape->plans.size() - 1;
   amr_tape_record(d, AMR_OP_SET_MESH, d->tape->cur_plan);
   return AMR_OK;
}

int amr_dev_comm(amr_dev *d, int start, int num, int stage, int permute)
{
   int rc = amr_comm_impl(d, start, num, stage, permute);
   if (!rc)
      amr_tape_record(d, AMR_OP_COMM, start, num, stage, permute);
   return rc;
}

int amr_dev_stencil(amr_dev *d, int var)
{
   int rc = amr_stencil_impl(d, var, 0);
   if (!rc)
      amr_tape_record(d, AMR_OP_STENCIL, var);
   return rc;
}

int amr_dev_stencil_stage(amr_dev *d, int var, int calc_stage)
{
   int rc = amr_stencil_impl(d, var, calc_stage);
   if (!rc)
      amr_tape_record(d, AMR_OP_STENCIL, var);
   return rc;
}

int amr_dev_set_materials(amr_dev *d, double a1, const double *a0, int n)
{
   if (!d || d->g.stencil != 0)
      return amr_set_error(d, AMR_ERR_ARG, "set_materials: the context is not a --stencil 0 one");
   if (!a0 || n != d->c.num_vars / 4 || n < 1)
      return amr_set_error(d, AMR_ERR_ARG, "set_materials: %d coefficients, need num_vars/4 = %d",
                           n, d->c.num_vars / 4);
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   if (!d->d_a0)
      HIP_TRY(d, hipMalloc(&d->d_a0, sizeof(double) * n));
   HIP_TRY(d, hipMemcpy(d->d_a0, a0, sizeof(double) * n, hipMemcpyHostToDevice));
   d->mat = n;
   d->a1 = a1;
   return AMR_OK;
}

int amr_dev_read_check_counts(amr_dev *d, int64_t counts[2])
{
   if (!d || !counts)
      return AMR_ERR_ARG;
   counts[0] = counts[1] = 0;
   if (!d->d_check_counts)
      return AMR_OK;
   unsigned long long h[kCountSlots * kCountStride];
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   HIP_TRY(d, hipMemcpy(h, d->d_check_counts, sizeof(h), hipMemcpyDeviceToHost));
   for (int t = 0; t < kCountSlots; t++)
      for (int i = 0; i < 2; i++)
         counts[i] += (int64_t) h[t * kCountStride + i];
   return AMR_OK;
}

int amr_dev_check_sum(amr_dev *d, int var, double *sum)
{
   if (!d || !sum || var < 0 || var >= d->c.num_vars)
      return amr_set_error(d, AMR_ERR_ARG, "check_sum: variable %d out of range", var);
   amr_span_begin(d, 2);
   int rc = amr_launch_block_sums(d, var, 1);
   if (!rc)
      rc = amr_launch_reduce_sums(d, var, 1, (double *) d->d_stage);
   amr_span_end(d);
   if (rc)
      return rc;
   HIP_TRY(d, hipMemcpyAsync(d->h_pinned, d->d_stage, sizeof(double), hipMemcpyDeviceToHost,
                             d->stream));
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   *sum = d->h_pinned[0];
   return AMR_OK;
}

}  // extern "C"

// Snapshot scratch for split/merge: every job needs num_vars * (n/2)^3
// values; batches larger than the cap are processed in order in chunks
// (safe: a chunk can only overwrite slots freed by itself or earlier
// chunks, never a slot a later chunk still reads).
static const size_t kScratchCap = (size_t) 512 << 20;

static int ensure_scratch(amr_dev *d, size_t bytes)
{
   if (bytes <= d->scratch_bytes)
      return AMR_OK;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   hipFree(d->d_scratch);
   d->d_scratch = nullptr;
   d->scratch_bytes = 0;
   HIP_TRY(d, hipMalloc(&d->d_scratch, bytes));
   d->scratch_bytes = bytes;
   return AMR_OK;
}

static int ensure_jobbuf(amr_dev *d, size_t bytes)
{
   if (bytes <= d->jobbuf_bytes)
      return AMR_OK;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   hipFree(d->d_jobbuf);
   d->d_jobbuf = nullptr;
   d->jobbuf_bytes = 0;
   HIP_TRY(d, hipMalloc(&d->d_jobbuf, bytes));
   d->jobbuf_bytes = bytes;
   return AMR_OK;
}

// Jobs read slots where they are and write them where par says.  A slot that
// is written whole (a child; a merged block by its eight octants) needs no
// move of what it held.
template <typename J>
static int refine_slots_current(amr_dev *d, const J *jobs, int n)
{
   if (!d->two_interiors)
      return AMR_OK;
   if (int rc = amr_unify(d, 0, d->c.num_vars))
      return rc;
   std::vector<uint8_t> octants;   // of each merged block, when first needed
   for (int t = 0; t < n; t++) {
      int32_t rd, wr;
      if constexpr (std::is_same<J, amr_split_job>::value) {
         rd = jobs[t].parent;
         wr = jobs[t].child;
      } else {
         rd = jobs[t].child;
         wr = jobs[t].dst;
      }
      if (int rc = amr_slots_current(d, &rd, 1))
         return rc;
      if (amr_slot_current(d, wr))
         continue;
      if constexpr (!std::is_same<J, amr_split_job>::value) {
         if (octants.empty()) {
            octants.assign(d->c.max_blocks, 0);
            for (int q = t; q < n; q++)
               octants[jobs[q].dst] |= 1 << jobs[q].octant;
         }
         if (octants[wr] != 0xff) {
            if (int rc = amr_slots_current(d, &wr, 1))
               return rc;
            continue;
         }
      }
      amr_slot_written(d, wr);
   }
   return AMR_OK;
}

int amr_split_slots_current(amr_dev *d, const amr_split_job *jobs, int n)
{
   return refine_slots_current(d, jobs, n);
}

template <typename J>
static int refine_data(amr_dev *d, const J *jobs, int n, bool split)
{
   if (!d || n < 0 || (n && !jobs))
      return amr_set_error(d, AMR_ERR_ARG, "split/consolidate: bad arguments");
   if (!n)
      return AMR_OK;
   for (int t = 0; t < n; t++) {
      int a = split ? ((const amr_split_job *) (const void *) &jobs[t])->parent
                    : ((const amr_merge_job *) (const void *) &jobs[t])->dst;
      int b = split ? ((const amr_split_job *) (const void *) &jobs[t])->child
                    : ((const amr_merge_job *) (const void *) &jobs[t])->child;
      int o = split ? ((const amr_split_job *) (const void *) &jobs[t])->octant
                    : ((const amr_merge_job *) (const void *) &jobs[t])->octant;
      if (a < 0 || a >= d->c.max_blocks || b < 0 || b >= d->c.max_blocks || o < 0 || o > 7)
         return amr_set_error(d, AMR_ERR_ARG, "split/consolidate: bad job %d", t);
   }
   if (int rc = refine_slots_current(d, jobs, n))
      return rc;
   size_t per_job = (size_t) d->c.num_vars * (d->g.nx / 2) * (d->g.ny / 2) * (d->g.nz / 2) *
                    d->elem_bytes;
   int chunk = (int) std::max<size_t>(1, std::min<size_t>(n, kScratchCap / per_job));
   // A context of its own sizes both buffers once for the largest batch of
   // jobs a refinement step can have (8 per slot): growing one waits for the
   // device, stages still queued included.  Batch members, which share one
   // stream and would each hold the scratch, size them as needed.
   const size_t most = 8 * (size_t) d->c.max_blocks;
   const size_t scratch_want =
      d->owns_stream ? per_job * std::max<size_t>(chunk, std::min(most, kScratchCap / per_job))
                     : per_job * chunk;
   int rc = ensure_scratch(d, scratch_want);
   if (!rc)
      rc = ensure_jobbuf(d, sizeof(J) * (d->owns_stream ? std::max<size_t>(n, most) : (size_t) n));
   if (rc)
      return rc;
   // The job list goes through pinned staging with a copy ordered on the
   // stream, so the host does not wait here for the stages still queued
   // (the refinement's host work then overlaps them).  A stream that has
   // drained frees the whole staging buffer; else the list is appended, and
   // only when it does not fit does the host wait.
   const size_t jb = (sizeof(J) * (size_t) n + 255) / 256 * 256;
   if (d->jobstage_used && hipStreamQuery(d->stream) == hipSuccess)
      d->jobstage_used = 0;
   if (d->jobstage_used + jb > d->jobstage_bytes) {
      HIP_TRY(d, hipStreamSynchronize(d->stream));
      d->jobstage_used = 0;
      if (jb > d->jobstage_bytes) {
         if (d->h_jobstage)
            hipHostFree(d->h_jobstage);
         d->h_jobstage = nullptr;
         d->jobstage_bytes = 0;
         const size_t cap = std::max<size_t>(jb, 4 << 20);
         HIP_TRY(d, hipHostMalloc(&d->h_jobstage, cap, hipHostMallocDefault));
         d->jobstage_bytes = cap;
      }
   }
   char *stage = (char *) d->h_jobstage + d->jobstage_used;
   memcpy(stage, jobs, sizeof(J) * n);
   d->jobstage_used += jb;
   HIP_TRY(d, hipMemcpyAsync(d->d_jobbuf, stage, sizeof(J) * n, hipMemcpyHostToDevice,
                             d->stream));
   amr_span_begin(d, 3);
   for (int t0 = 0; t0 < n && !rc; t0 += chunk) {
      int m = std::min(chunk, n - t0);
      const J *dj = (const J *) d->d_jobbuf + t0;
      rc = split ? amr_launch_split(d, (const amr_split_job *) dj, m, d->d_scratch)
                 : amr_launch_merge(d, (const amr_merge_job *) dj, m, d->d_scratch);
   }
   amr_span_end(d);
   return rc;
}

int amr_split_impl(amr_dev *d, const amr_split_job *jobs, int n)
{
   if (d && amr_require_fresh(d, 0, d->c.num_vars, "split"))
      return AMR_ERR_STATE;
   return refine_data(d, jobs, n, true);
}

int amr_merge_impl(amr_dev *d, const amr_merge_job *jobs, int n)
{
   if (d && amr_require_fresh(d, 0, d->c.num_vars, "consolidate"))
      return AMR_ERR_STATE;
   return refine_data(d, jobs, n, false);
}

extern "C" {

int amr_dev_split(amr_dev *d, const amr_split_job *jobs, int n)
{
   int rc = amr_split_impl(d, jobs, n);
   if (!rc && n && d->tape && d->tape->on && !d->replaying) {
      const int first = (int) d->tape->splits.size();
      d->tape->splits.insert(d->tape->splits.end(), jobs, jobs + n);
      amr_tape_record(d, AMR_OP_SPLIT, first, n);
   }
   return rc;
}

int amr_dev_consolidate(amr_dev *d, const amr_merge_job *jobs, int n)
{
   int rc = amr_merge_impl(d, jobs, n);
   if (!rc && n && d->tape && d->tape->on && !d->replaying) {
      const int first = (int) d->tape->merges.size();
      d->tape->merges.insert(d->tape->merges.end(), jobs, jobs + n);
      amr_tape_record(d, AMR_OP_MERGE, first, n);
   }
   return rc;
}

int amr_dev_reserve_sums(amr_dev *d, int n_rows)
{
   if (!d || n_rows < 1)
      return amr_set_error(d, AMR_ERR_ARG, "reserve_sums: n_rows must be positive");
   if (n_rows <= d->sum_rows)
      return AMR_OK;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   hipFree(d->d_sums);
   d->d_sums = nullptr;
   d->sum_rows = 0;
   HIP_TRY(d, hipMalloc(&d->d_sums, sizeof(double) * (size_t) n_rows * d->c.num_vars));
   HIP_TRY(d, hipMemset(d->d_sums, 0, sizeof(double) * (size_t) n_rows * d->c.num_vars));
   d->sum_rows = n_rows;
   d->plan_version++;
   size_t need = sizeof(double) * (size_t) n_rows * d->c.num_vars;
   if (need > d->h_pinned_bytes) {
      hipHostFree(d->h_pinned);
      d->h_pinned = nullptr;
      HIP_TRY(d, hipHostMalloc((void **) &d->h_pinned, need, hipHostMallocDefault));
      d->h_pinned_bytes = need;
   }
   return AMR_OK;
}

int amr_dev_read_sums(amr_dev *d, int row0, int n_rows, double *out)
{
   if (!d || !out || row0 < 0 || n_rows < 0 || row0 + n_rows > d->sum_rows)
      return amr_set_error(d, AMR_ERR_ARG, "read_sums: rows [%d, %d) out of range", row0,
                           row0 + n_rows);
   size_t bytes = sizeof(double) * (size_t) n_rows * d->c.num_vars;
   HIP_TRY(d, hipMemcpyAsync(d->h_pinned, d->d_sums + (size_t) row0 * d->c.num_vars, bytes,
                             hipMemcpyDeviceToHost, d->stream));
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   memcpy(out, d->h_pinned, bytes);
   return AMR_OK;
}

}  // extern "C"

int amr_stage_impl(amr_dev *d, int start, int num, int stage, int permute, int sum_row)
{
   if (!d || start < 0 || num < 0 || start + num > d->c.num_vars)
      return amr_set_error(d, AMR_ERR_ARG, "stage: variables out of range");
   if (sum_row >= d->sum_rows)
      return amr_set_error(d, AMR_ERR_ARG, "stage: checksum row %d not reserved", sum_row);
   int rc = amr_comm_impl(d, start, num, stage, permute);
   if (rc)
      return rc;
   amr_span_begin(d, 1);
   rc = amr_launch_stencil(d, start, num, sum_row >= 0, stage);
   amr_span_end(d);
   if (rc || sum_row < 0)
      return rc;
   amr_span_begin(d, 2);
   rc = amr_launch_reduce_sums(d, start, num,
                               d->d_sums + (size_t) sum_row * d->c.num_vars + start);
   amr_span_end(d);
   return rc;
}

extern "C" {

int amr_dev_stage(amr_dev *d, int start, int num, int stage, int permute, int sum_row)
{
   int rc = amr_stage_impl(d, start, num, stage, permute, sum_row);
   if (!rc)
      amr_tape_record(d, AMR_OP_STAGE, start, num, stage, permute);
   return rc;
}

int amr_dev_stage_fused(amr_dev *d, int start, int num, int stage, int permute, int sum_row)
{
   if (!d)
      return AMR_ERR_ARG;
   // The plain stage where in-place reads cannot stand in for it (permuted
   // phases, --code 1/2 planes, taping and replay, jobs on inactive blocks),
   // and below ~1e8 cell updates where the fused stage still needs the three
   // ordered exchange launches (edges not folded): such stages are bound by
   // launch latency, where the fused kernels' longer set-up costs more than
   // the ghost planes they save (1-7% slower).  With folded edges a stage is
   // one coarse/fine launch and the stencil at most: 60 blocks of 6x10x14 in
   // FP32 take 2.6 ms for 200 stages against 5.6 ms plain, the moving-object
   // run (16^3, 12 variables) 32.5 ms against 35.4.
   const double cells = (double) d->n_active * num * d->g.nx * d->g.ny * d->g.nz;
   // a 7-point stage that reads every face in place is one launch at any size,
   // and the order of the phases does not matter to it
   if (!d->two_interiors || !d->closed || (permute && !d->all_faces) || d->whole_ghosts ||
       (d->tape && d->tape->on) || d->replaying ||
       (d->fused_mode == 1 && cells < 1.0e8 && !d->all_faces && !d->fold_edges))
      return amr_dev_stage(d, start, num, stage, permute, sum_row);
   if (start < 0 || num < 0 || start + num > d->c.num_vars)
      return amr_set_error(d, AMR_ERR_ARG, "stage: variables out of range");
   if (sum_row >= d->sum_rows)
      return amr_set_error(d, AMR_ERR_ARG, "stage: checksum row %d not reserved", sum_row);
   if (!num)
      return AMR_OK;
   if (int rc = amr_unify(d, start, num))
      return rc;
   if (!d->timing_dirs && !d->all_faces)
      amr_span_begin(d, 0);
   for (int dir = 0; dir < 3 && !d->all_faces; dir++) {
      if (d->timing_dirs)
         amr_span_begin(d, kSpanExchangeX + dir);
      int rc = amr_launch_exchange_fused_dir(d, dir, start, num);
      if (d->timing_dirs)
         amr_span_end(d);
      if (rc)
         return rc;
   }
   if (!d->timing_dirs && !d->all_faces)
      amr_span_end(d);
   amr_span_begin(d, 1);
   int rc = amr_launch_stencil_fused(d, start, num, sum_row >= 0);
   amr_span_end(d);
   if (rc)
      return rc;
   for (int v = start; v < start + num; v++)
      d->stale[v] = 1;
   if (sum_row < 0)
      return AMR_OK;
   amr_span_begin(d, 2);
   rc = amr_launch_reduce_sums(d, start, num,
                               d->d_sums + (size_t) sum_row * d->c.num_vars + start);
   amr_span_end(d);
   return rc;
}

int amr_dev_sync(amr_dev *d)
{
   if (!d)
      return AMR_ERR_ARG;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   return AMR_OK;
}

int amr_dev_set_timing(amr_dev *d, int on)
{
   if (!d)
      return AMR_ERR_ARG;
   d->timing = on != 0;
   d->timing_dirs = on == 2;
   d->timing_stencil_only = on == 3;
   return AMR_OK;
}

int amr_dev_read_timing(amr_dev *d, double ms[4])
{
   if (!d || !ms)
      return AMR_ERR_ARG;
   ms[0] = ms[1] = ms[2] = ms[3] = 0.0;
   HIP_TRY(d, hipStreamSynchronize(d->stream));
   for (auto &s : d->spans) {
      float t = 0.0f;
      if (s.a && s.b && hipEventElapsedTime(&t, s.a, s.b) == hipSuccess) {
         if (s.cat >= kSpanExchangeX) {
            ms[0] += t;                                   // exchange, by direction
            d->exchange_ms[s.cat - kSpanExchangeX] += t;
         } else {
            ms[s.cat] += t;
         }
      }
      if (s.a) d->ev_free.push_back(s.a);
      if (s.b) d->ev_free.push_back(s.b);
   }
   d->spans.clear();
   return AMR_OK;
}

int amr_dev_read_exchange_timing(amr_dev *d, double ms[3])
{
   if (!d || !ms)
      return AMR_ERR_ARG;
   for (int i = 0; i < 3; i++) {
      ms[i] = d->exchange_ms[i];
      d->exchange_ms[i] = 0.0;
   }
   return AMR_OK;
}

int amr_dev_memory(const amr_dev *d, size_t *bytes, int *buffers)
{
   if (!d || !bytes)
      return AMR_ERR_ARG;
   const size_t b[] = {
      d->pool ? (size_t) d->g.var_stride * d->c.num_vars * d->elem_bytes : 0,
      d->d_sorted ? sizeof(int32_t) * d->c.max_blocks : 0,
      sizeof(amr_face_job) * (size_t) d->jobs_cap,
      d->d_partials ? sizeof(double) * (size_t) d->c.num_vars * d->c.max_blocks : 0,
      sizeof(double) * (size_t) d->sum_rows * d->c.num_vars,
      d->d_stage ? sizeof(double) * (size_t) d->g.gx * d->g.gy * d->g.gz * d->c.num_vars : 0,
      d->scratch_bytes, d->jobbuf_bytes, d->h_pinned ? d->h_pinned_bytes : 0 };
   size_t tot = 0;
   int n = 0;
   for (size_t x : b) {
      tot += x;
      n += x > 0;
   }
   *bytes = tot;
   if (buffers)
      *buffers = n;
   return AMR_OK;
}

}  // extern "C"
