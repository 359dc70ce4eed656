// matstencil.hip -- the variable-work stencils of --stencil 0
// (ref/stencil.c:43-73 stencil_driver, :147-981).
//
// With --stencil 0 the variables form mat = num_vars/4 "materials" in four
// classes: class c holds variables [c*mat, (c+1)*mat).  Variable 0 and the
// variables from 4*mat on take the plain 7-point average (k_stencil).  Every
// other variable takes, by calculation stage % 6, one of six updates coupled
// to other variables, followed by the clamp of stencil_check:
//   0    a pointwise update from variables 0, 1 and class partners;
//   1-3  a sweep along x, y or z that updates in place: each cell reads its
//        predecessor's new value, so one thread owns a line and walks it in
//        order (variable 1 and class 0 are pointwise here);
//   4    a 7-point product stencil with the class partners;
//   5    a 27-point sum of the class partners.
// 4 and 5 read the old values of the whole block (a Jacobi update): they
// write a work buffer that a second kernel commits (clamping as it goes).
// Every expression keeps the reference's evaluation order (left to right,
// no contraction), so the FP64 path is bit-identical; the clamp's
// data-dependent operation counts are summed on the device for the report.
//
// One workgroup per active block; cells are addressed through home(), so
// face, edge and z-copy parts of the record stay consistent.
#include "kern_exchange.h"
#include "kern_stencil.h"

namespace {

using namespace amrk;

// Class partners (offsets in units of mat) of the 7-point update -- x, y, z
// neighbours -- and of the 27-point update -- neighbours with 1, 2 and 3
// non-zero offsets (ref/stencil.c:661-845).
__constant__ int kPartner[4][3] = {{1, 2, 3}, {1, 2, -1}, {1, -2, -1}, {-3, -2, -1}};

struct MatArgs {
   int var, mat;
   double a1;
   const double *a0;          // mat values (device)
   unsigned long long *counts;  // slot pairs: [0] clamps that divide, [1] that scale
};

// One block's cells of every variable.
template <typename T>
struct BlockView {
   T *pool;
   int64_t vs, base;   // variable stride, slot offset
   typedef typename Acc<T>::type A;
   __device__ A get(const Lay &L, int u, int i, int j, int k) const
   {
      return to_acc(pool[u * vs + base + home(L, i, j, k)]);
   }
   // store a new value of variable u; returns the value as stored
   __device__ A put(const Lay &L, int u, int i, int j, int k, A v) const
   {
      const T t = from_acc<T>(v);
      T *rec = pool + u * vs + base;
      rec[home(L, i, j, k)] = t;
      if (k == 1 || k == L.nz)
         rec[zcopy(L, i, j, k)] = t;
      return to_acc(t);
   }
};

template <typename T>
__device__ __forceinline__ BlockView<T> view(T *pool, const int32_t *sorted, const Lay &L)
{
   BlockView<T> b;
   b.pool = pool;
   b.vs = L.var_stride;
   b.base = (int64_t) sorted[blockIdx.x] * L.rec;
   return b;
}

// stencil_check (ref/stencil.c:966-981): |v|, then v / (a1 + a0[0] + v) for
// v >= 1 or v * (10 - a1) for v < 0.1.
template <typename A>
__device__ __forceinline__ A clamp(A v, const MatArgs &m, unsigned &ndiv, unsigned &nmul)
{
   v = fabs(v);
   if (v >= A(1.0)) {
      v = v / ((A(m.a1) + A(m.a0[0])) + v);
      ndiv++;
   } else if (v < A(0.1)) {
      v = v * (A(10.0) - A(m.a1));
      nmul++;
   }
   return v;
}

// The clamps of a wavefront, added to one of kCountSlots counter pairs, each on
// a line of its own: with one pair for all, the whole-stage launch (7,000
// wavefronts) spent 150 of its 200 us on those two addresses.
__device__ __forceinline__ void add_counts(const MatArgs &m, unsigned ndiv, unsigned nmul)
{
   for (int o = 32; o > 0; o >>= 1) {
      ndiv += __shfl_down(ndiv, o, 64);
      nmul += __shfl_down(nmul, o, 64);
   }
   if ((threadIdx.x & 63) == 0 && (ndiv | nmul)) {
      unsigned long long *const c =
         m.counts + ((blockIdx.x + 5 * blockIdx.y + 11 * (threadIdx.x >> 6)) & (kCountSlots - 1)) *
                       kCountStride;
      atomicAdd(&c[0], (unsigned long long) ndiv);
      atomicAdd(&c[1], (unsigned long long) nmul);
   }
}

// Pointwise updates: stage 0 (stencil_0, ref/stencil.c:147-225) and, for
// stages 1-3, variable 1 and class 0 (ref/stencil.c:233-262 and twins).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_mat_point(T *pool, const int32_t *sorted, Lay L,
                                                        MatArgs m, int op)
{
   typedef typename Acc<T>::type A;
   const BlockView<T> b = view(pool, sorted, L);
   const int var = m.var, mat = m.mat, ncell = L.nx * L.ny * L.nz;
   const A a1 = A(m.a1), one = A(1.0);
   unsigned ndiv = 0, nmul = 0;
   for (int t = threadIdx.x; t < ncell; t += kThreads) {
      const int i = 1 + t / (L.ny * L.nz), j = 1 + (t / L.nz) % L.ny, k = 1 + t % L.nz;
      const A v = b.get(L, var, i, j, k), p0 = b.get(L, 0, i, j, k), p1 = b.get(L, 1, i, j, k);
      A r;
      if (op == 0) {
         if (var == 1) {
            r = p1;
            for (int u = mat; u < 2 * mat; u++)
               r = r + b.get(L, u, i, j, k) * p0;
         } else if (var < mat) {
            r = v + v * ((p0 + p1) - a1 * v);
         } else if (var < 2 * mat) {
            r = v * (((p0 + v) + a1 * b.get(L, var + mat, i, j, k)) +
                     (one - a1) * b.get(L, var + 2 * mat, i, j, k)) / p1;
         } else if (var < 3 * mat) {
            r = v + b.get(L, var - mat, i, j, k) *
                       ((a1 * p0 + A(m.a0[var - 2 * mat]) * v) +
                        (one - a1) * b.get(L, var + mat, i, j, k)) / p1;
         } else {
            const A a0 = A(m.a0[var - 3 * mat]), q = b.get(L, var - 2 * mat, i, j, k);
            r = v + q * (((a1 * p0 + a0 * v) + (one - a0) * b.get(L, var - mat, i, j, k)) +
                         (one - a1) * q) / (p1 * p1);
         }
      } else if (var == 1) {
         r = p1;
         for (int u = 2; u < mat + 2; u++)
            r = r + b.get(L, u, i, j, k) * p0;
         r = r / (a1 + r);
      } else {   // class 0 of a sweep stage
         r = v + v * ((p0 + p1) - a1 * v) / (A(m.a0[var]) + p1);
      }
      b.put(L, var, i, j, k, clamp(r, m, ndiv, nmul));
   }
   add_counts(m, ndiv, nmul);
}

// In-place sweeps of classes 1-3 along axis ax (stages 1-3: stencil_x,
// stencil_y, stencil_z, ref/stencil.c:263-660).  Thread = line; the
// predecessor's value is the new one, the successor's the old one.  The
// gate variable g (the variable itself for class 1, var - mat for class 2,
// var - 2*mat for class 3) picks the weights.  After the line is done the
// thread clamps it (only its own line's cells are read by the sweep).
template <typename T>
__global__ __launch_bounds__(kThreads) void k_mat_sweep(T *pool, const int32_t *sorted, Lay L,
                                                        MatArgs m, int ax)
{
   typedef typename Acc<T>::type A;
   const BlockView<T> b = view(pool, sorted, L);
   const int var = m.var, mat = m.mat, cls = var / mat;
   const int n = ax == 0 ? L.nx : ax == 1 ? L.ny : L.nz;
   const int n1 = ax == 0 ? L.ny : L.nx;   // slower in-plane axis
   const int n2 = ax == 2 ? L.ny : L.nz;   // faster in-plane axis
   const A a1 = A(m.a1), a0 = A(m.a0[var - cls * mat]);
   const int g = cls == 1 ? var : var - (cls - 1) * mat;
   unsigned ndiv = 0, nmul = 0;
   for (int t = threadIdx.x; t < n1 * n2; t += kThreads) {
      const int c1 = 1 + t / n2, c2 = 1 + t % n2;
      auto at = [&](int u, int p) {
         int i, j, k;
         canon(ax, p, c1, c2, i, j, k);
         return b.get(L, u, i, j, k);
      };
      A prev = at(var, 0);
      for (int p = 1; p <= n; p++) {
         const A v = at(var, p), vn = at(var, p + 1), q1 = at(1, p);
         const A gv = cls == 1 ? v : at(g, p);
         const A gm = cls == 1 ? prev : at(g, p - 1);
         const A gp = cls == 1 ? vn : at(g, p + 1);
         const A tmp1 = fabs(gv - gm), tmp2 = fabs(gv - gp);
         const A w = tmp1 > tmp2 ? tmp1 - tmp2 : tmp2 - tmp1;
         const A num = ((tmp1 * prev) + (w * (v + q1))) + (tmp2 * vn);
         A den;
         if (cls == 1) {
            den = ((((a1 + a0) + prev) + v) + vn) + at(0, p);
            den = den + q1;
         } else {
            den = ((a1 + a0) + at(var - mat, p)) + at(cls == 2 ? var + mat : var - 2 * mat, p);
            den = ((den + prev) + v) + vn;
         }
         int i, j, k;
         canon(ax, p, c1, c2, i, j, k);
         prev = b.put(L, var, i, j, k, num / den);
      }
      for (int p = 1; p <= n; p++) {
         int i, j, k;
         canon(ax, p, c1, c2, i, j, k);
         b.put(L, var, i, j, k, clamp(b.get(L, var, i, j, k), m, ndiv, nmul));
      }
   }
   add_counts(m, ndiv, nmul);
}

// Jacobi updates, stages 4 and 5 (stencil_7 / stencil_27, ref/stencil.c:661-958):
// new values into work[in][cell] (accumulator type), old values everywhere.
template <typename T>
__global__ __launch_bounds__(kThreads) void k_mat_jacobi(T *pool, const int32_t *sorted, Lay L,
                                                         MatArgs m, int op,
                                                         typename Acc<T>::type *work)
{
   typedef typename Acc<T>::type A;
   const BlockView<T> b = view(pool, sorted, L);
   const int var = m.var, mat = m.mat, cls = var / mat, ncell = L.nx * L.ny * L.nz;
   const int qx = var + kPartner[cls][0] * mat, qy = var + kPartner[cls][1] * mat,
             qz = var + kPartner[cls][2] * mat;
   const A a1 = A(m.a1);
   A *out = work + (int64_t) blockIdx.x * ncell;
   for (int t = threadIdx.x; t < ncell; t += kThreads) {
      const int i = 1 + t / (L.ny * L.nz), j = 1 + (t / L.nz) % L.ny, k = 1 + t % L.nz;
      const A v = b.get(L, var, i, j, k);
      A r;
      if (op == 4) {
         A s = b.get(L, var, i - 1, j, k) * b.get(L, qx, i - 1, j, k);
         s = s + b.get(L, var, i, j - 1, k) * b.get(L, qy, i, j - 1, k);
         s = s + b.get(L, var, i, j, k - 1) * b.get(L, qz, i, j, k - 1);
         s = s + v * v;
         s = s + b.get(L, var, i, j, k + 1) * b.get(L, qz, i, j, k + 1);
         s = s + b.get(L, var, i, j + 1, k) * b.get(L, qy, i, j + 1, k);
         s = s + b.get(L, var, i + 1, j, k) * b.get(L, qx, i + 1, j, k);
         r = s / A(7.0) * (a1 + v);
      } else {
         const int q[4] = {var, qx, qy, qz};   // by number of non-zero offsets
         A s = A(0);
         for (int d = 0; d < 27; d++) {
            const int di = d / 9 - 1, dj = (d / 3) % 3 - 1, dk = d % 3 - 1;
            const A e = b.get(L, q[(di != 0) + (dj != 0) + (dk != 0)], i + di, j + dj, k + dk);
            s = d ? s + e : e;
         }
         r = s / (a1 + A(27.0));
      }
      out[t] = r;
   }
}

template <typename T>
__global__ __launch_bounds__(kThreads) void k_mat_commit(T *pool, const int32_t *sorted, Lay L,
                                                         MatArgs m,
                                                         const typename Acc<T>::type *work)
{
   const BlockView<T> b = view(pool, sorted, L);
   const int ncell = L.nx * L.ny * L.nz;
   const typename Acc<T>::type *in = work + (int64_t) blockIdx.x * ncell;
   unsigned ndiv = 0, nmul = 0;
   for (int t = threadIdx.x; t < ncell; t += kThreads) {
      const int i = 1 + t / (L.ny * L.nz), j = 1 + (t / L.nz) % L.ny, k = 1 + t % L.nz;
      b.put(L, m.var, i, j, k, clamp(in[t], m, ndiv, nmul));
   }
   add_counts(m, ndiv, nmul);
}

// ---- a whole stage
// The variables (u, mat+u, 2*mat+u, 3*mat+u) form a group: apart from
// variables 0 and 1, an update reads no variable outside its group.  So once
// variable 0 and, in calculation stages 0-3, variable 1 are done, the groups
// are independent: one launch, one workgroup per (block, group), the four
// variables in class order.  One launch per variable left the device with one
// workgroup per block at a time (176 blocks: 19 x 59 us for stage 5).  The
// group's boxes stay in LDS throughout: each cell is read once and written
// once, and no neighbour read computes a record offset.  Measured there (20
// variables, FP64): a stage 930 -> 145 us, the group launch 32 / 66 / 66 / 66
// / 89 / 96 us for calculation stages 0-5; bound by the sweeps' serial lines
// and, in stages 4 and 5, by one workgroup per CU fitting its LDS.
constexpr int kGroupThreads = 512;
constexpr size_t kGroupLds = 156 * 1024;

template <typename T>
size_t group_lds(const Lay &L)
{
   return sizeof(typename Acc<T>::type) *
          (4 * (size_t) L.gx * L.gy * L.gz + (size_t) L.nx * L.ny * L.nz);
}

template <typename T>
__global__ __launch_bounds__(kGroupThreads) void k_mat_group(T *pool, const int32_t *sorted,
                                                             Lay L, MatArgs m, int op)
{
   typedef typename Acc<T>::type A;
   extern __shared__ __align__(16) unsigned char smem[];
   const int u = blockIdx.y, mat = m.mat;
   const int nbox = L.gx * L.gy * L.gz, ncell = L.nx * L.ny * L.nz, sy = L.gz, sx = L.gy * L.gz;
   A *const box = (A *) smem, *const tmp = box + 4 * nbox;
   T *const rec = pool + (int64_t) sorted[blockIdx.x] * L.rec;
   const T *const i0 = rec + L.oI, *const i1 = rec + L.var_stride + L.oI;   // variables 0 and 1
   const A a1 = A(m.a1), one = A(1.0);
   const int first = op < 4 ? 2 : 1;   // variables below are done
   const int tid = threadIdx.x;
   auto stored = [](A v) { return to_acc(from_acc<T>(v)); };
   unsigned ndiv = 0, nmul = 0;
   // cell t of the record's order of variable var (and its z-plane copy)
   auto put = [&](int var, int t, A v) {
      const int i = t / (L.ny * L.nz), r = t - i * L.ny * L.nz, j = r / L.nz, k = r - j * L.nz;
      T *const out = rec + (int64_t) var * L.var_stride;
      const T x = from_acc<T>(v);
      out[L.oI + t] = x;
      if (k == 0) out[L.oZI + i * L.ny + j] = x;
      if (k == L.nz - 1) out[L.oZI + (L.nx + i) * L.ny + j] = x;
   };
   if (op <= 3) {
      // pointwise updates: class 0, and in stage 0 all classes, which read
      // each other at one cell only -- no box needed
      for (int t = tid; t < ncell; t += kGroupThreads) {
         const A p0 = to_acc(i0[t]), p1 = to_acc(i1[t]);
         A v[4];
#pragma unroll
         for (int c = 0; c < 4; c++)
            if (c == 0 || op == 0)
               v[c] = to_acc(rec[(int64_t) (c * mat + u) * L.var_stride + L.oI + t]);
         if (u >= first) {
            A r;
            if (op != 0) r = v[0] + v[0] * ((p0 + p1) - a1 * v[0]) / (A(m.a0[u]) + p1);
            else r = v[0] + v[0] * ((p0 + p1) - a1 * v[0]);
            put(u, t, clamp(r, m, ndiv, nmul));
         }
         if (op != 0)
            continue;
         if (mat + u >= first) {
            v[1] = v[1] * (((p0 + v[1]) + a1 * v[2]) + (one - a1) * v[3]) / p1;
            v[1] = stored(clamp(v[1], m, ndiv, nmul));
            put(mat + u, t, v[1]);
         }
         const A a0 = A(m.a0[u]);
         v[2] = v[2] + v[1] * ((a1 * p0 + a0 * v[2]) + (one - a1) * v[3]) / p1;
         v[2] = stored(clamp(v[2], m, ndiv, nmul));
         put(2 * mat + u, t, v[2]);
         v[3] = v[3] + v[1] * (((a1 * p0 + a0 * v[3]) + (one - a0) * v[2]) + (one - a1) * v[1]) /
                          (p1 * p1);
         put(3 * mat + u, t, clamp(v[3], m, ndiv, nmul));
      }
      if (op == 0) {
         add_counts(m, ndiv, nmul);
         return;
      }
   }
   // boxes of classes lo..3
   const int lo = op <= 3 ? 1 : 0;
   for (int e = tid; e < nbox; e += kGroupThreads) {
      const int i = e / sx, r = e - i * sx, j = r / sy, k = r - j * sy, h = home(L, i, j, k);
#pragma unroll
      for (int c = 0; c < 4; c++)
         if (c >= lo)
            box[(c - lo) * nbox + e] = to_acc(rec[(int64_t) (c * mat + u) * L.var_stride + h]);
   }
   __syncthreads();
   // LDS place of interior cell t of the record's order
   auto at = [&](int t) {
      const int i = t / (L.ny * L.nz), r = t - i * L.ny * L.nz, j = r / L.nz, k = r - j * L.nz;
      return (i + 1) * sx + (j + 1) * sy + k + 1;
   };
   const A *const c1 = box + (1 - lo) * nbox, *const c2 = c1 + nbox, *const c3 = c2 + nbox;
   for (int cls = lo; cls < 4; cls++) {
      const int var = cls * mat + u;
      if (var < first)
         continue;
      A *const me = box + (cls - lo) * nbox;
      if (op <= 3) {
         // in-place sweep, a thread per line (k_mat_sweep's expressions)
         const int ax = op - 1;
         const int n = ax == 0 ? L.nx : ax == 1 ? L.ny : L.nz;
         const int n1 = ax == 0 ? L.ny : L.nx, n2 = ax == 2 ? L.ny : L.nz;
         const int s = ax == 0 ? sx : ax == 1 ? sy : 1;
         const int s1 = ax == 0 ? sy : sx, s2 = ax == 2 ? sy : 1;
         const int r0 = ax == 0 ? L.ny * L.nz : ax == 1 ? L.nz : 1;   // step in record order
         const int r1 = ax == 0 ? L.nz : L.ny * L.nz, r2 = ax == 2 ? L.nz : 1;
         const A a0 = A(m.a0[u]);
         for (int t = tid; t < n1 * n2; t += kGroupThreads) {
            const int l1 = t / n2, l2 = t - l1 * n2;
            const int b0 = (l1 + 1) * s1 + (l2 + 1) * s2, g0 = l1 * r1 + l2 * r2;
            A prev = me[b0];
            for (int p = 1; p <= n; p++) {
               const int q = b0 + p * s, g = g0 + (p - 1) * r0;
               const A v = me[q], vn = me[q + s], q1 = to_acc(i1[g]);
               const A gv = cls == 1 ? v : c1[q];
               const A gm = cls == 1 ? prev : c1[q - s];
               const A gp = cls == 1 ? vn : c1[q + s];
               const A tmp1 = fabs(gv - gm), tmp2 = fabs(gv - gp);
               const A w = tmp1 > tmp2 ? tmp1 - tmp2 : tmp2 - tmp1;
               const A num = ((tmp1 * prev) + (w * (v + q1))) + (tmp2 * vn);
               A den;
               if (cls == 1) {
                  den = ((((a1 + a0) + prev) + v) + vn) + to_acc(i0[g]);
                  den = den + q1;
               } else {
                  den = cls == 2 ? ((a1 + a0) + c1[q]) + c3[q] : ((a1 + a0) + c2[q]) + c1[q];
                  den = ((den + prev) + v) + vn;
               }
               prev = stored(num / den);
               me[q] = prev;
            }
         }
         __syncthreads();
         for (int t = tid; t < ncell; t += kGroupThreads) {
            const int q = at(t);
            me[q] = stored(clamp(me[q], m, ndiv, nmul));
         }
      } else {
         const A *const qx = box + (cls + kPartner[cls][0]) * nbox,
                 *const qy = box + (cls + kPartner[cls][1]) * nbox,
                 *const qz = box + (cls + kPartner[cls][2]) * nbox;
         for (int t = tid; t < ncell; t += kGroupThreads) {
            const int q = at(t);
            const A v = me[q];
            A r;
            if (op == 4) {
               A s = me[q - sx] * qx[q - sx];
               s = s + me[q - sy] * qy[q - sy];
               s = s + me[q - 1] * qz[q - 1];
               s = s + v * v;
               s = s + me[q + 1] * qz[q + 1];
               s = s + me[q + sy] * qy[q + sy];
               s = s + me[q + sx] * qx[q + sx];
               r = s / A(7.0) * (a1 + v);
            } else {
               A s = A(0);
#pragma unroll
               for (int d = 0; d < 27; d++) {
                  const int di = d / 9 - 1, dj = (d / 3) % 3 - 1, dk = d % 3 - 1;
                  const int nz = (di != 0) + (dj != 0) + (dk != 0);   // non-zero offsets
                  const A *const src = nz == 0 ? me : nz == 1 ? qx : nz == 2 ? qy : qz;
                  const A e = src[q + di * sx + dj * sy + dk];
                  s = d ? s + e : e;
               }
               r = s / (a1 + A(27.0));
            }
            tmp[t] = r;
         }
         __syncthreads();
         for (int t = tid; t < ncell; t += kGroupThreads)
            me[at(t)] = stored(clamp(tmp[t], m, ndiv, nmul));
      }
      __syncthreads();
   }
   for (int t = tid; t < ncell; t += kGroupThreads) {
      const int q = at(t);
      for (int cls = lo; cls < 4; cls++)
         if (cls * mat + u >= first)
            put(cls * mat + u, t, box[(cls - lo) * nbox + q]);
   }
   add_counts(m, ndiv, nmul);
}

template <typename T>
int launch_mat(amr_dev *d, int var, int calc_stage)
{
   typedef typename Acc<T>::type A;
   Lay L;
   if (int rc = amr_lay(d, 0, d->c.num_vars, &L))
      return rc;
   MatArgs m;
   m.var = var;
   m.mat = d->mat;
   m.a1 = d->a1;
   m.a0 = d->d_a0;
   m.counts = d->d_check_counts;
   const dim3 grid(d->n_active), blk(kThreads);
   const int op = calc_stage % 6, cls = var / d->mat;
   if (op == 0 || (op <= 3 && (var == 1 || cls == 0))) {
      hipLaunchKernelGGL(k_mat_point<T>, grid, blk, 0, d->stream, (T *) d->pool, d->d_sorted, L,
                         m, op);
   } else if (op <= 3) {
      hipLaunchKernelGGL(k_mat_sweep<T>, grid, blk, 0, d->stream, (T *) d->pool, d->d_sorted, L,
                         m, op - 1);
   } else {
      const size_t need = (size_t) d->n_active * d->g.nx * d->g.ny * d->g.nz * sizeof(A);
      if (need > d->matwork_bytes) {
         HIP_TRY(d, hipStreamSynchronize(d->stream));
         hipFree(d->d_matwork);
         d->d_matwork = nullptr;
         d->matwork_bytes = 0;
         HIP_TRY(d, hipMalloc(&d->d_matwork, need));
         d->matwork_bytes = need;
      }
      hipLaunchKernelGGL(k_mat_jacobi<T>, grid, blk, 0, d->stream, (T *) d->pool, d->d_sorted, L,
                         m, op, (A *) d->d_matwork);
      hipLaunchKernelGGL(k_mat_commit<T>, grid, blk, 0, d->stream, (T *) d->pool, d->d_sorted, L,
                         m, (const A *) d->d_matwork);
   }
   HIP_TRY(d, hipGetLastError());
   return AMR_OK;
}

template <typename T>
int launch_group(amr_dev *d, int calc_stage)
{
   Lay L;
   if (int rc = amr_lay(d, 0, d->c.num_vars, &L))
      return rc;
   MatArgs m;
   m.var = 0;
   m.mat = d->mat;
   m.a1 = d->a1;
   m.a0 = d->d_a0;
   m.counts = d->d_check_counts;
   // stage 0 needs no box, the sweeps those of classes 1-3 (two workgroups
   // per CU at 12^3 FP64), the Jacobi updates four and the new values
   const int op = calc_stage % 6;
   const size_t lds = op == 0 ? 0
                    : op <= 3 ? sizeof(typename Acc<T>::type) * 3 * (size_t) L.gx * L.gy * L.gz
                              : group_lds<T>(L);
   if (!d->group_lds_set) {   // more than the default limit of a launch
      HIP_TRY(d, hipFuncSetAttribute((const void *) &k_mat_group<T>,
                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int) kGroupLds));
      d->group_lds_set = true;
   }
   hipLaunchKernelGGL(k_mat_group<T>, dim3(d->n_active, d->mat), dim3(kGroupThreads), lds,
                      d->stream, (T *) d->pool, d->d_sorted, L, m, op);
   HIP_TRY(d, hipGetLastError());
   return AMR_OK;
}

}  // namespace

bool amr_mat_groups_fit(const amr_dev *d)
{
   return (d->c.precision == AMR_PREC_F64 ? group_lds<double>(d->g) : group_lds<float>(d->g)) <=
          kGroupLds;
}

int amr_launch_mat_groups(amr_dev *d, int calc_stage)
{
   if (!d->n_active)
      return AMR_OK;
   if (!d->d_a0)
      return amr_set_error(d, AMR_ERR_STATE, "stencil 0: amr_dev_set_materials not called");
   switch (d->c.precision) {
   case AMR_PREC_F64: return launch_group<double>(d, calc_stage);
   case AMR_PREC_F32: return launch_group<float>(d, calc_stage);
   default: return launch_group<uint16_t>(d, calc_stage);
   }
}

// One variable's update of a --stencil 0 stage other than the plain 7-point
// ones (variable 0 and variables >= 4*mat are left to the caller).
int amr_launch_mat_stencil(amr_dev *d, int var, int calc_stage)
{
   if (!d->n_active)
      return AMR_OK;
   if (!d->d_a0)
      return amr_set_error(d, AMR_ERR_STATE, "stencil 0: amr_dev_set_materials not called");
   switch (d->c.precision) {
   case AMR_PREC_F64: return launch_mat<double>(d, var, calc_stage);
   case AMR_PREC_F32: return launch_mat<float>(d, var, calc_stage);
   default: return launch_mat<uint16_t>(d, var, calc_stage);
   }
}
