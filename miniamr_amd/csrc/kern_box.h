// kern_box.h -- the 7- and 27-point stencil on a block's whole ghost box held
// in LDS.  A workgroup owns one block and sweeps over its variables: each
// variable's interior and ghost planes are loaded as vectors of C cells in
// record order, whatever the block's shape, parked in LDS, and every thread
// computes its outputs from there.  What hides the loads is the other
// workgroups of the CU: the next variable's loads, held in registers during
// the sums, took 120-176 registers and cost more waves than they gained (10^3
// FP64 98.5-103.7 ms a run against 94.8).
//
// What bounded the plane-by-plane form (kern_stencil.h) off the 16 x 16 faces
// it was shaped for: one thread per (j, k) column and a barrier per x plane,
// so an 8^3 block keeps 64 of 256 threads at work and a 10^3 block 100, with
// one scalar load per ghost cell.  Here the index arithmetic is done once per
// block: a variable costs a thread its loads (one scalar base per variable and
// 32-bit offsets that do not change), the LDS traffic and the sums.
//
// Measured: 890 blocks of 10^3 x 40 variables, FP64, a 7-point stage 365 us
// (three exchange launches and the stencil) -> 152 us, bound by its traffic
// (22.7 KB per block-variable of 16 KB algorithmic: ghost planes, z-plane
// copies, 80-byte rows in 128-byte lines; 5.3 TB/s, 0.82 of a copy's rate) and
// the workgroups in flight; 64 blocks of 8^3 x 4 variables 23 -> 5 us, bound by
// the launch.
//
// Faces.  A ghost plane is read from where its values come from (FaceSrc): the
// block's own plane, a same-level neighbour's interior, the block's own
// boundary plane, a coarse neighbour's cells / 4 or sums of four fine cells,
// rounded to the storage type as the ghost plane would hold them.
#pragma once

#include <type_traits>

#include "kern_stencil.h"

namespace amrk {

// Division of n < 2^13 by d: (n * ceil(2^19 / d)) >> 19 in one full-rate
// 24-bit multiplication; exact for the ranges the host has checked.
__device__ __forceinline__ uint32_t div19(uint32_t n, uint32_t m)
{
   return __umul24(n, m) >> 19;
}

// Sizes of a launch, computed on the host (box_dims).
struct BoxDims {
   int V;                   // variables a workgroup sweeps over
   int nt;                  // threads per workgroup
   int R;                   // LDS elements per row: nz cells, k = nz+1, .., k = 0 of the next row
   int nvec;                // vectors of a variable's interior
   int nface;               // vectors of its six faces
   int box;                 // LDS elements per variable
   int dbl;                 // two boxes in LDS: one barrier per variable
   int seg, cols;           // 27-point: x segments, vector columns
   uint32_t m_nvz, m_nvy, m_ny, m_cols;   // div19 multipliers
};

template <typename T, int C>
__device__ __forceinline__ typename VecN<T, C>::type ld_bytes(gptr<T> b, uint32_t byte)
{
   typedef typename VecN<T, C>::type VT;
   return *(gptr<const VT>) ((gptr<const char>) b + byte);
}

template <typename T>
__device__ __forceinline__ T ld_byte1(gptr<T> b, uint32_t byte)
{
   return *(gptr<const T>) ((gptr<const char>) b + byte);
}

template <typename T, int C>
__device__ __forceinline__ void st_bytes(gptr<T> b, uint32_t byte, typename VecN<T, C>::type v)
{
   typedef typename VecN<T, C>::type VT;
   const gptr<VT> p = (gptr<VT>) ((gptr<char>) b + byte);
   if constexpr (sizeof(T) == 8)
      __builtin_nontemporal_store(v, p);
   else
      *p = v;
}

// Where cell (i, j, k) of the box sits in LDS.  The row of (i, j) holds
// k = 1..nz from a vector-aligned start; k = nz+1 follows, and k = 0 is the
// element before (the end of the previous row's padding).
__device__ __forceinline__ int box_pos(const Lay &L, const BoxDims &B, int C, int i, int j, int k)
{
   return C + (i * L.gy + j) * B.R + k - 1;
}

// Offset in a neighbour's record of the cell (a, b) (1-based in-plane
// coordinates) next to the shared face, f being the face of the block that
// reads it; z faces from the z-plane copies.
__device__ __forceinline__ int facing(const Lay &L, int f, int a, int b)
{
   if (f < 2)
      return L.oI + ((f ? 0 : L.nx - 1) * L.ny + a - 1) * L.nz + b - 1;
   if (f < 4)
      return L.oI + ((a - 1) * L.ny + (f == 3 ? 0 : L.ny - 1)) * L.nz + b - 1;
   return L.oZI + ((f == 5 ? 0 : L.nx) + a - 1) * L.ny + b - 1;
}

// One block's variables v0 .. v0+nv-1.  QV interior vectors, QF face vectors
// and QE edge cells per thread.  faces: the block's six FaceSrc (null: its
// own ghost planes); es: where its edges are (27-point; null: its own).
// 32-bit byte offsets: a variable's slab must be smaller than 4 GiB.
template <typename T, int ST, int C, int QV, int QF, int QE>
__device__ __forceinline__ void box_sweep(T *__restrict__ pool, int slot, const Lay &L,
                                          const Lay &Lo, const BoxDims &B,
                                          const FaceSrc *__restrict__ faces,
                                          const EdgeSrc *__restrict__ es, int v0, int nv,
                                          typename Acc<T>::type *lds, double *red,
                                          double *__restrict__ partials, int part_stride)
{
   typedef typename Acc<T>::type A;
   typedef typename VecN<T, C>::type VT;
   typedef typename VecN<A, C>::type AT;
   typedef typename VecN<T, 2>::type V2;
   constexpr uint32_t EB = sizeof(T);
   const int tid = threadIdx.x, nt = B.nt;
   const uint32_t own = (uint32_t) slot * (uint32_t) L.rec;
   const int nvz = L.nz / C, nvy = L.ny / C;
   gptr<T> vb = uniform_base(global_view(pool) + (int64_t) v0 * L.var_stride);

   // interior vectors t = tid + q*nt, record order
   int pi[QV];
#pragma unroll
   for (int q = 0; q < QV; q++) {
      const int t = tid + q * nt;
      const int r = div19(t, B.m_nvz), kv = t - r * nvz;   // r = i*ny + j
      const int i = div19(r, B.m_ny), j = r - i * L.ny;
      const bool on = t < B.nvec;
      pi[q] = on ? box_pos(L, B, C, i + 1, j + 1, kv * C + 1) : -1;
   }
   const uint32_t oi = (own + L.oI + tid * C) * EB, oo = (own + Lo.oI + tid * C) * EB;
   const uint32_t step = (uint32_t) (nt * C) * EB;
   // face vectors e = tid + q*nt over W, E, S, N, D, U
   enum { NONE = 0, VEC = 1, PRO = 2, RES = 3 };
   constexpr int NR = ST == 7 ? C : 1;       // cells per vector that a restriction fills
   int fk[QF], pf[QF], keep[QF];
   bool zf[QF];
   uint32_t of[QF][NR], rd[QF];
#pragma unroll
   for (int q = 0; q < QF; q++) {
      int e = tid + q * nt;
      const int nx_ = L.ny * nvz, ny_ = L.nx * nvz, nz_ = L.nx * nvy;
      int f;
      if (e < 2 * nx_) { f = e >= nx_; e -= f * nx_; }
      else if (e < 2 * (nx_ + ny_)) { e -= 2 * nx_; f = e >= ny_; e -= f * ny_; f += 2; }
      else { e -= 2 * (nx_ + ny_); f = e >= nz_; e -= f * nz_; f += 4; }
      const bool on = tid + q * nt < B.nface;
      if (!on) { e = 0; f = 0; }
      const int dir = f >> 1, hi = f & 1;
      const int na = dir == 0 ? L.ny : L.nx, nb = dir == 2 ? L.ny : L.nz;
      const int nvb = dir == 2 ? nvy : nvz;
      const int a = div19(e, dir == 2 ? B.m_nvy : B.m_nvz) + 1, b = (e - (a - 1) * nvb) * C + 1;
      pf[q] = dir == 0 ? box_pos(L, B, C, hi ? L.nx + 1 : 0, a, b)
            : dir == 1 ? box_pos(L, B, C, a, hi ? L.ny + 1 : 0, b)
                       : box_pos(L, B, C, a, b, hi ? L.nz + 1 : 0);
      zf[q] = dir == 2;
      keep[q] = 0;
      rd[q] = 0;
      const FaceSrc F = faces ? faces[f] : FaceSrc{FS_OWN, {-1, -1, -1, -1}};
      const uint32_t ghost = own + L.oF[f] + (a - 1) * nb + b - 1;
      fk[q] = on ? VEC : NONE;
      if (F.kind == FS_OWN) {
         of[q][0] = ghost * EB;
      } else if (F.kind == FS_SAME) {
         of[q][0] = ((uint32_t) F.s[0] * (uint32_t) L.rec + facing(L, f, a, b)) * EB;
      } else if (F.kind == FS_BC) {
         of[q][0] = (own + facing(L, f ^ 1, a, b)) * EB;
      }
      if constexpr (ST == 7) {
         if (F.kind == FS_PROLONG) {
            // fine cells (a, 2m+1), (a, 2m+2) take the coarse cell / 4
            fk[q] = on ? PRO : NONE;
            of[q][0] = ((uint32_t) F.s[0] * (uint32_t) L.rec +
                        facing(L, f, ((a + 1) >> 1) + F.s[2] * (na / 2),
                               ((b + 1) >> 1) + F.s[1] * (nb / 2))) * EB;
         } else if (F.kind == FS_RESTRICT) {
            // coarse cell <- its four fine cells: (fa, fb), (fa, fb+1) and
            // the row after; a quarter without a job keeps the plane's cell
            fk[q] = on ? RES : NONE;
            const int ja = a > na / 2, fa = 2 * (a - ja * (na / 2)) - 1;
            rd[q] = (uint32_t) (facing(L, f, 2, 1) - facing(L, f, 1, 1)) * EB;
#pragma unroll
            for (int m = 0; m < C; m++) {
               const int bm = b + m, ib = bm > nb / 2, fb = 2 * (bm - ib * (nb / 2)) - 1;
               const int src = ib ? (ja ? F.s[3] : F.s[1]) : (ja ? F.s[2] : F.s[0]);
               // an even element, so that the pair load below is aligned
               of[q][m] = src < 0 ? ((ghost + m) & ~1u) * EB
                                  : ((uint32_t) src * (uint32_t) L.rec + facing(L, f, fa, fb)) * EB;
               keep[q] |= (src < 0) << m;
            }
         }
      }
   }
   // edge cells: four lines each along z, y and x, then the corners
   constexpr int QE1 = QE ? QE : 1;
   uint32_t oe[QE1];
   int pe[QE1];
   if constexpr (QE > 0) {
      const int nz4 = 4 * L.nz, ny4 = 4 * L.ny, nx4 = 4 * L.nx, ne = nz4 + ny4 + nx4 + 8;
#pragma unroll
      for (int q = 0; q < QE; q++) {
         const int e = tid + q * nt;
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
            const int h = e < ne ? e - nz4 - ny4 - nx4 : 0;
            line = 12 + h; t = 0;
            i = (h & 4) ? L.nx + 1 : 0; j = (h & 2) ? L.ny + 1 : 0; k = (h & 1) ? L.nz + 1 : 0;
         }
         pe[q] = e < ne ? box_pos(L, B, C, i, j, k) : -1;
         oe[q] = (es ? (uint32_t) edge_at(es[line], L, t) : own + home(L, i, j, k)) * EB;
      }
   }

   VT ri[QV], rf[QF];
   T re[QE1];
   auto load = [&]() {
#pragma unroll
      for (int q = 0; q < QV; q++)
         if (pi[q] >= 0)
            ri[q] = ld_bytes<T, C>(vb, oi + q * step);
#pragma unroll
      for (int q = 0; q < QF; q++)
         if (fk[q] == VEC)
            rf[q] = ld_bytes<T, C>(vb, of[q][0]);
      if constexpr (QE > 0) {
#pragma unroll
         for (int q = 0; q < QE; q++)
            if (pe[q] >= 0)
               re[q] = ld_byte1(vb, oe[q]);
      }
   };

   // 27-point: this thread's first column task (segment, column)
   const int ntask = B.seg * B.cols, len = ST == 27 ? (L.nx + B.seg - 1) / B.seg : 0;
   const int sx = L.gy * B.R;
   for (int u = 0; u < nv; u++) {
      load();
      A *const bx = lds + (B.dbl && (u & 1) ? B.box : 0);
      AT ci[QV];
#pragma unroll
      for (int q = 0; q < QV; q++)
         if (pi[q] >= 0) {
#pragma unroll
            for (int m = 0; m < C; m++)
               ci[q][m] = to_acc((T) ri[q][m]);
            *(AT *) (bx + pi[q]) = ci[q];
         }
#pragma unroll
      for (int q = 0; q < QF; q++)
         if (fk[q] != NONE) {
            AT x;
            if constexpr (ST == 7) {
               if (fk[q] == PRO) {
                  T v[C / 2];
#pragma unroll
                  for (int m = 0; m < C / 2; m++)
                     v[m] = ld_byte1(vb, of[q][0] + m * EB);
#pragma unroll
                  for (int m = 0; m < C; m++)
                     rf[q][m] = from_acc<T>(to_acc(v[m / 2]) / A(4));
               } else if (fk[q] == RES) {
                  V2 v[2 * C];
#pragma unroll
                  for (int m = 0; m < C; m++) {
                     v[2 * m] = ld_bytes<T, 2>(vb, of[q][m]);
                     v[2 * m + 1] = ld_bytes<T, 2>(vb, of[q][m] + rd[q]);
                  }
#pragma unroll
                  for (int m = 0; m < C; m++) {
                     A w = to_acc((T) v[2 * m][0]);
                     w = w + to_acc((T) v[2 * m][1]);
                     w = w + to_acc((T) v[2 * m + 1][0]);
                     w = w + to_acc((T) v[2 * m + 1][1]);
                     rf[q][m] = keep[q] >> m & 1 ? (T) v[2 * m][m & 1] : from_acc<T>(w);
                  }
               }
            }
#pragma unroll
            for (int m = 0; m < C; m++)
               x[m] = to_acc((T) rf[q][m]);
            if (!zf[q]) {
               *(AT *) (bx + pf[q]) = x;
            } else {
#pragma unroll
               for (int m = 0; m < C; m++)
                  bx[pf[q] + m * B.R] = x[m];
            }
         }
      if constexpr (QE > 0) {
#pragma unroll
         for (int q = 0; q < QE; q++)
            if (pe[q] >= 0)
               bx[pe[q]] = to_acc(re[q]);
      }
      const gptr<T> cb = vb;
      vb += L.var_stride;
      __syncthreads();
      double bsum = 0.0;
      if constexpr (ST == 7) {
#pragma unroll
         for (int q = 0; q < QV; q++)
            if (pi[q] >= 0) {
               const A *p = bx + pi[q];
               const AT w = *(const AT *) (p - sx), e = *(const AT *) (p + sx),
                        n0 = *(const AT *) (p - B.R), n1 = *(const AT *) (p + B.R);
               A c[C + 2];
               c[0] = p[-1];
               c[C + 1] = p[C];
#pragma unroll
               for (int m = 0; m < C; m++)
                  c[m + 1] = ci[q][m];
               VT o;
#pragma unroll
               for (int m = 0; m < C; m++) {
                  A x = w[m] + n0[m];     // ref/stencil.c:82-101's order
                  x = x + c[m];
                  x = x + c[m + 1];
                  x = x + c[m + 2];
                  x = x + n1[m];
                  x = x + e[m];
                  o[m] = from_acc<T>(divide<A, 7>(x));
               }
               st_bytes<T, C>(cb, oo + q * step, o);
               const int t = tid + q * nt, r = div19(t, B.m_nvz), kv = t - r * nvz;
               if (kv == 0) st(cb, own + Lo.oZI + r, (T) o[0]);
               if (kv == nvz - 1) st(cb, own + Lo.oZI + L.nx * L.ny + r, (T) o[C - 1]);
               if (partials) {
#pragma unroll
                  for (int m = 0; m < C; m++)
                     bsum += (double) to_acc((T) o[m]);
               }
            }
      } else {
         // A task is an x segment of one vector column: it walks its planes
         // with the 9-term sums of the last two in registers, each row read
         // as one vector and its two neighbours.  Segments recompute the sums
         // of the planes they share; they keep the threads busy where a face
         // has few columns.
         for (int x = tid; x < ntask; x += nt) {
            const int sg = div19(x, B.m_cols), col = x - sg * B.cols;
            const int j = div19(col, B.m_nvz), kv = col - j * nvz;
            const int i0 = sg * len + 1, i1 = min(i0 + len - 1, L.nx);   // output planes
            const A *p = bx + box_pos(L, B, C, i0 - 1, j, kv * C + 1);
            A s_prev[C] = {}, s_cur[C] = {};
            uint32_t o = (own + Lo.oI + ((uint32_t) (i0 - 1) * L.ny + j) * L.nz + kv * C) * EB;
            uint32_t zo = own + Lo.oZI + (i0 - 1) * L.ny + j;
            for (int i = i0 - 1; i <= i1 + 1; i++) {   // plane i's sums; output i - 1
               A s[C];
#pragma unroll
               for (int row = 0; row < 3; row++) {
                  const A *pr = p + row * B.R;
                  const AT c = *(const AT *) pr;
                  A v[C + 2];
                  v[0] = pr[-1];
                  v[C + 1] = pr[C];
#pragma unroll
                  for (int m = 0; m < C; m++)
                     v[m + 1] = c[m];
#pragma unroll
                  for (int m = 0; m < C; m++) {
                     s[m] = row ? s[m] + v[m] : v[m];
                     s[m] = s[m] + v[m + 1];
                     s[m] = s[m] + v[m + 2];
                  }
               }
               p += sx;
               if (i > i0) {
                  VT ov;
#pragma unroll
                  for (int m = 0; m < C; m++) {
                     const A w = (s_prev[m] + s_cur[m]) + s[m];
                     ov[m] = from_acc<T>(divide<A, 27>(w));
                     if (partials)
                        bsum += (double) to_acc((T) ov[m]);
                  }
                  st_bytes<T, C>(cb, o, ov);
                  if (kv == 0) st(cb, zo, (T) ov[0]);
                  if (kv == nvz - 1) st(cb, zo + (uint32_t) (L.nx * L.ny), (T) ov[C - 1]);
                  o += (uint32_t) (L.ny * L.nz) * EB;
                  zo += L.ny;
               }
#pragma unroll
               for (int m = 0; m < C; m++) {
                  s_prev[m] = s_cur[m];
                  s_cur[m] = s[m];
               }
            }
         }
      }
      if (partials) {
         bsum = wave_reduce(bsum);
         if ((tid & 63) == 0)
            red[tid >> 6] = bsum;
      }
      if (partials || !B.dbl)
         __syncthreads();
      if (partials && tid == 0) {
         double s = 0.0;
         for (int w = 0; w < nt / 64; w++)
            s += red[w];
         global_view(partials)[(int64_t) (v0 + u) * part_stride] = s;
      }
   }
}

}  // namespace amrk
