// box.hip -- launches of the whole-box stencil kernels (kern_box.h).
#include <stdlib.h>
#include <algorithm>

#include "kern_box.h"

namespace {

using namespace amrk;

template <typename T, int ST, int C, int QV, int QF>
__global__ __launch_bounds__(512) void k_box(T *__restrict__ pool,
                                             const int32_t *__restrict__ sorted,
                                             const FaceSrc *__restrict__ faces,
                                             const EdgeSrc *__restrict__ edges, Lay L, Lay Lo,
                                             BoxDims B, int var0, int var_end,
                                             double *__restrict__ partials, int part_stride)
{
   extern __shared__ __align__(16) unsigned char smem[];
   __shared__ double red[8];
   const int in = blockIdx.x, slot = sorted[in];
   const int v0 = var0 + blockIdx.y * B.V;
   box_sweep<T, ST, C, QV, QF, ST == 27 ? 2 : 0>(
      pool, slot, L, Lo, B, faces ? faces + 6 * (int64_t) in : nullptr,
      edges ? edges + (int64_t) kEdgeSrcs * slot : nullptr, v0, min(B.V, var_end - v0),
      (typename Acc<T>::type *) smem, red, partials ? partials + in : nullptr, part_stride);
}

// div19's multiplier for divisor d and dividends up to nmax; clears ok when
// the quotient would not be exact for all of them.
uint32_t mul19(int d, int nmax, bool &ok)
{
   const uint32_t m = ((1u << 19) + d - 1) / d, e = m * d - (1u << 19);
   ok = ok && nmax < (1 << 13) && (uint64_t) nmax * e < (1u << 19);
   return m;
}

// Vector width and sizes of a launch over n_active blocks and num variables;
// false when a box does not fit (then the plane-by-plane kernels serve).
template <typename T>
bool box_dims(const Lay &g, int st, int n_active, int num, BoxDims &B, int &C, int &QV,
              size_t &lds)
{
   typedef typename Acc<T>::type A;
   C = sizeof(T) < 8 && g.ny % 4 == 0 && g.nz % 4 == 0 ? 4 : 2;
   if (g.ny > 64 || g.nz > 64 || g.nx > 64 ||
       (uint64_t) g.var_stride * sizeof(T) >= ((uint64_t) 1 << 32))
      return false;
   const int nvz = g.nz / C;
   B.R = g.nz + C;
   B.box = (g.gx * g.gy * B.R + C + C - 1) / C * C;
   B.nvec = g.nx * g.ny * nvz;
   B.nface = 2 * (g.ny * g.nz + g.nx * g.nz + g.nx * g.ny) / C;
   const int ne = 4 * (g.nx + g.ny + g.nz) + 8;
   const size_t bytes = (size_t) B.box * sizeof(A);
   // Threads: the fewest with at most two interior vectors each, else the
   // widest workgroup with up to eight (QF = 2 up to four vectors, then 4).
   // Widest 512 for the 7-point stencil (16^3 FP32, 40 variables: 126.6 ms a
   // run of 400 stages against 129.0 at 256 and 152.5 at 128), 128 for the
   // 27-point one, whose columns are fewer than its vectors (6x10x14 FP64:
   // 45.4 ms against 45.5 at 64 and 256).
   const int most = st == 7 ? 512 : 128;
   QV = 0;
   for (int pass = 0; pass < 2 && !QV; pass++)
      for (int nt = pass ? most : 64; nt <= (pass ? 512 : most) && !QV; nt *= 2) {
         const int need = (B.nvec + nt - 1) / nt, nf = (B.nface + nt - 1) / nt;
         const int q = need <= 1 ? 1 : need <= 2 ? 2 : need <= 4 ? 4 : 8;
         if (need > (pass ? 8 : 2) || nf > (q == 8 ? 4 : 2) || (st == 27 && ne > 2 * nt))
            continue;
         B.nt = nt;
         QV = q;
      }
   if (!QV || bytes > 56 * 1024)
      return false;
   // Variables per workgroup: sweeps as long as 4096 workgroups remain (10^3
   // FP64, 890 blocks x 40 variables: 94.8 ms a run, 93.8 with 8192, 106.2
   // with one variable each; 16^3 FP32: 129.0 / 130.8 / 147.0).
   const int64_t items = (int64_t) n_active * num;
   int V = (int) std::max<int64_t>(1, std::min<int64_t>(num, items / 4096));
   B.V = (num + (num + V - 1) / V - 1) / ((num + V - 1) / V);
   B.dbl = B.V > 1 && 2 * bytes <= 32 * 1024;
   B.cols = g.ny * nvz;
   B.seg = std::max(1, std::min(B.nt / B.cols, g.nx / 2));
   bool ok = true;
   B.m_nvz = mul19(nvz, std::max(B.nvec + B.nt, std::max(B.nface, B.cols)), ok);
   B.m_nvy = mul19(std::max(1, g.ny / C), B.nface, ok);
   B.m_ny = mul19(g.ny, (B.nvec + B.nt) / nvz + 1, ok);
   B.m_cols = mul19(B.cols, std::max(B.nt, B.seg * B.cols), ok);
   lds = bytes * (B.dbl ? 2 : 1);
   return ok;
}

template <typename T, int ST, int C>
int go(amr_dev *d, int QV, size_t lds, const FaceSrc *faces, const EdgeSrc *edges, const Lay &L,
       const Lay &Lo, const BoxDims &B, int start, int num, double *parts)
{
   const dim3 grid(d->n_active, (num + B.V - 1) / B.V);
#define GO(qv, qf)                                                                             \
   hipLaunchKernelGGL((k_box<T, ST, C, qv, qf>), grid, dim3(B.nt), lds, d->stream,              \
                      (T *) d->pool, d->d_sorted, faces, edges, L, Lo, B, start, start + num,   \
                      parts, d->c.max_blocks)
   switch (QV) {
   case 1: GO(1, 2); break;
   case 2: GO(2, 2); break;
   case 4: GO(4, 2); break;
   default: GO(8, 4); break;
   }
#undef GO
   HIP_TRY(d, hipGetLastError());
   return AMR_OK;
}

template <typename T, int ST>
int launch(amr_dev *d, const FaceSrc *faces, const EdgeSrc *edges, const Lay &L, const Lay &Lo,
           int start, int num, double *parts)
{
   BoxDims B;
   int C, QV;
   size_t lds;
   if (!box_dims<T>(d->g, ST, d->n_active, num, B, C, QV, lds))
      return amr_set_error(d, AMR_ERR_ARG, "block %dx%dx%d too large for the box stencil", L.nx,
                           L.ny, L.nz);
   if constexpr (sizeof(T) < 8)
      if (C == 4)
         return go<T, ST, 4>(d, QV, lds, faces, edges, L, Lo, B, start, num, parts);
   return go<T, ST, 2>(d, QV, lds, faces, edges, L, Lo, B, start, num, parts);
}

template <typename F>
auto by_type(int prec, F f)
{
   switch (prec) {
   case AMR_PREC_F64: return f((double) 0);
   case AMR_PREC_F32: return f((float) 0);
   default: return f((uint16_t) 0);
   }
}

}  // namespace

// MINIAMR_STENCIL_BOX=0 leaves every stencil to the plane-by-plane kernels.
// (One variable per workgroup is the tightest case: wider ones are only
// chosen for boxes far below the limits.)
bool amr_box_fits(const amr_dev *d, int st)
{
   static const bool on = [] {
      const char *e = getenv("MINIAMR_STENCIL_BOX");
      return !e || atoi(e) != 0;
   }();
   return on && by_type(d->c.precision, [&](auto z) {
             BoxDims B;
             int C, QV;
             size_t lds;
             return box_dims<decltype(z)>(d->g, st, 1, 1, B, C, QV, lds);
          });
}

int amr_launch_box(amr_dev *d, int st, const FaceSrc *faces, const EdgeSrc *edges, const Lay &L,
                   const Lay &Lo, int start, int num, double *parts)
{
   return by_type(d->c.precision, [&](auto z) {
      typedef decltype(z) T;
      return st == 7 ? launch<T, 7>(d, faces, edges, L, Lo, start, num, parts)
                     : launch<T, 27>(d, faces, edges, L, Lo, start, num, parts);
   });
}
