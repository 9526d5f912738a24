// Batched `unsplit` (hydro/umuscl.f90:22-171) for gfx950.
//
// Input and output keep the reference's Fortran layouts so that the kernel
// sits behind the reference's own call boundary:
//   uin   (nv,-1:4,-1:4,-1:4,5)   gravin (nv,-1:4,-1:4,-1:4,3)
//   flux  (nv,1:3,1:3,1:3,5,3)    tmp    (nv,1:3,1:3,1:3,2,3)
// repeated `ngroups` times back to back (one array set per oct batch).
//
// Work decomposition.  The 7-point slopes run on tiles of 16 octs
// (oct_tile.hpp): every primitive, traced cell and face once, exchanged
// through LDS.  2^20 octs: 1.40 ms in FP64 (hllc, minmod; 5.5 GB that it
// cannot do without, 3.9 TB/s) and 1.07 ms in FP32-mixed (5.1 TB/s, the rate
// of a copy); with a gravity array 1.60 ms in FP64.  One thread per row of
// three faces, as below, took 1.54, 1.20 (staged primitives) and 2.03 ms.
//
// The 27-point slopes (slope_type 3) read the whole 6^3 stencil and keep one
// row of faces per thread: per oct the reference computes fluxes on 36
// faces, 12 per direction, arranged as 4 rows of 3 faces (x rows at j,k in
// {1,2}, faces i=1..3; likewise y and z).  The octs of a batch are
// consecutive lanes, so every global load of a (cell, variable) pair is a
// coalesced segment.  A row needs the traced states of its 4 cells (s = 0..3
// along the row).  Because every value is a deterministic function of its
// inputs, both decompositions give the reference's values bit for bit.
#include <type_traits>

#include "hydro_device.hpp"
#include "unsplit_args.hpp"
#include "unsplit_device.hpp"
#include "oct_tile.hpp"

namespace ramses {

// UnsplitArgs is declared in unsplit_args.hpp

namespace {

using unsplit_dev::unsplit_task;

// One thread per (group, row, lane) task of the 27-point slopes; G: a.grav is
// non-null.
template <typename R, int RS, bool G>
__global__ __launch_bounds__(768) void unsplit_rows(UnsplitArgs a) {
  const long t = (long)xcd_contiguous(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (t >= a.ngroups * 12L * a.nv) return;
  unsplit_task<R, RS, true, false, -1, G>(a, t, a.ngroups, a.ngrid_last);
}

// One tile of 16 octs per workgroup (oct_tile.hpp); G: a.grav is non-null.
// Octs are counted through the batches, lane fastest; octs past the last
// read the last one's stencil and store nothing.
template <typename R, int RS, int ST, bool G>
__global__ __launch_bounds__(oct_tile::kThreads)
__attribute__((amdgpu_waves_per_eu(4, 8))) void unsplit_tile(UnsplitArgs a, long nocts) {
  using namespace oct_tile;
  __shared__ R s[kLds];
  const int t = threadIdx.x, l = t % kOcts;
  const int nv = a.nv;
  const long o0 = (long)xcd_contiguous(blockIdx.x, gridDim.x) * kOcts;
  long g;   // this thread's oct: lane of batch g
  int lane;
  {
    long o = o0 + l;
    if (o >= nocts) o = nocts - 1;
    if (nocts <= 0x7fffffffL) {
      g = (unsigned)o / (unsigned)nv;
      lane = (int)((unsigned)o - (unsigned)g * (unsigned)nv);
    } else {
      g = o / nv;
      lane = (int)(o - g * nv);
    }
  }
  const HydroParams hp = a.hp;
  const double dt = a.dt;
  const SolverConsts<R> sc = scalar(make_consts<R>(hp));
  const double dtxhalf = scalar(dt * 0.5);
  const double smalle = scalar(hp.smallc * hp.smallc / hp.gamma / (hp.gamma - 1.0));  // hydro/umuscl.f90:884
  // strides between cells and between variables
  const size_t cs = a.compact ? (size_t)nv * 5 : (size_t)nv, vs = a.compact ? (size_t)nv : (size_t)nv * 216;
  const size_t gcs = a.compact ? (size_t)nv * 3 : (size_t)nv;
  const double* u = a.uin + g * ((size_t)nv * 216 * 5) + lane;
  const double* gr = G ? a.grav + g * ((size_t)nv * 216 * 3) + lane : nullptr;
  double w[kLoads][5], acc[kLoads][3];
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    const int e = t + k * kThreads;
    if (e < kPairs) {
      const size_t cell = a.compact ? (size_t)(e / kOcts) : (size_t)kTab.cell[e / kOcts];
#pragma unroll
      for (int v = 0; v < 5; ++v) w[k][v] = u[cell * cs + v * vs];
#pragma unroll
      for (int v = 0; v < 3; ++v) acc[k][v] = G ? gr[cell * gcs + v * vs] : 0.0;
    }
  }
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    const int e = t + k * kThreads;
    if (e < kPairs)
      put_prim(s, e, ctoprim_cell<R>(w[k][0], w[k][1], w[k][2], w[k][3], w[k][4], acc[k][0], acc[k][1], acc[k][2],
                                     dtxhalf, smalle, hp));
  }
  __syncthreads();
  // the scaling of a direction is formed again only where its dx differs from
  // the last one's (two divisions each)
  FluxScale fs = scalar(make_scale(dt, a.dx[0]));
  R dtdx[3] = {(R)fs.dtdx, (R)fs.dtdx, (R)fs.dtdx};
  if (a.dx[1] != a.dx[0]) dtdx[1] = scalar((R)(dt / a.dx[1]));
  if (a.dx[2] != a.dx[0]) dtdx[2] = scalar((R)(dt / a.dx[2]));
  trace_tile<R, ST>(s, t, sc, dtdx);
  const size_t fvs = (size_t)nv * 27;
  for (int k = 0; k < 2; ++k) {
    const int f = tile_face(t, k);
    if (f < 0) return;
    const int d = __builtin_amdgcn_readfirstlane(f) / 12;  // the four faces of a wavefront share their direction
    const Face<R> fl = get_side(s, f, 0, l), fr = get_side(s, f, 1, l);
    const Flux6<R> fg = riemann_fixed<R, RS>(fl, fr, sc);
    const double dxd = d == 0 ? a.dx[0] : (d == 1 ? a.dx[1] : a.dx[2]);
    if (dxd != fs.dx) fs = scalar(make_scale(dt, dxd));
    const R val[7] = {fg.f[0], fg.f[1], fg.f[3], fg.f[4], fg.f[2], (R)0.5 * (fl.un + fr.un), fg.f[5]};  // :845
    double out[7];
    scale_flux<7>(val, fs, out);  // :106,111,129,153
    if (o0 + l < nocts) {
      double *flux, *tmp;
      size_t st;
      if (a.compact) {
        st = (size_t)nv;
        flux = a.flux + (size_t)(7 * f) * nv + lane;
        tmp = flux + 5 * st;
      } else {
        st = fvs;
        flux = a.flux + g * fvs * 15 + (size_t)(kTab.out[f] + 27 * 5 * d) * nv + lane;
        tmp = a.tmp + g * fvs * 6 + (size_t)(kTab.out[f] + 27 * 2 * d) * nv + lane;
      }
      flux[0] = out[0];
      flux[(size_t)(1 + d) * st] = out[1];  // the momenta in their own order (:809-842)
      flux[(size_t)(d == 0 ? 2 : 1) * st] = out[2];
      flux[(size_t)(d == 2 ? 2 : 3) * st] = out[3];
      flux[4 * st] = out[4];
      tmp[0] = out[5];
      tmp[st] = out[6];
    }
  }
}

}  // namespace

// Minmod, the reference's default slope (hydro/hydro_parameters.f90:76),
// has kernels with the limiter fixed at compile time (ST = 1); the other
// 7-point types take it at run time (ST = -1).  The 27-point slopes read the
// whole 6^3 stencil and take the row kernel.  Kernels without a gravity
// array (G = false) read none and test no pointer; the reference always
// passes one (zeros without Poisson).
template <typename R, int RS, bool S27>
static void launch_t(const UnsplitArgs& a, long grid, int block, hipStream_t stream) {
  if constexpr (S27) {
    const dim3 g((unsigned)grid), b(block);
    if (a.grav)
      hipLaunchKernelGGL((unsplit_rows<R, RS, true>), g, b, 0, stream, a);
    else
      hipLaunchKernelGGL((unsplit_rows<R, RS, false>), g, b, 0, stream, a);
  } else {
    const long nocts = (a.ngroups - 1) * a.nv + a.ngrid_last;
    if (nocts <= 0) return;
    const dim3 g((unsigned)((nocts + oct_tile::kOcts - 1) / oct_tile::kOcts)), b(oct_tile::kThreads);
    const bool st1 = a.hp.slope_type == 1;
    if (a.grav) {
      if (st1)
        hipLaunchKernelGGL((unsplit_tile<R, RS, 1, true>), g, b, 0, stream, a, nocts);
      else
        hipLaunchKernelGGL((unsplit_tile<R, RS, -1, true>), g, b, 0, stream, a, nocts);
    } else {
      if (st1)
        hipLaunchKernelGGL((unsplit_tile<R, RS, 1, false>), g, b, 0, stream, a, nocts);
      else
        hipLaunchKernelGGL((unsplit_tile<R, RS, -1, false>), g, b, 0, stream, a, nocts);
    }
  }
}

template <typename R>
static void launch_r(const UnsplitArgs& a, long grid, int block, hipStream_t stream) {
  const bool s27 = a.hp.slope_type == 3;
  switch (a.hp.riemann) {
    case kHLLC: s27 ? launch_t<R, kHLLC, true>(a, grid, block, stream) : launch_t<R, kHLLC, false>(a, grid, block, stream); break;
    case kHLL: s27 ? launch_t<R, kHLL, true>(a, grid, block, stream) : launch_t<R, kHLL, false>(a, grid, block, stream); break;
    case kACOUSTIC:
    case kEXACT:
      s27 ? launch_t<R, kDynamicRiemann, true>(a, grid, block, stream)
          : launch_t<R, kDynamicRiemann, false>(a, grid, block, stream);
      break;
    default: s27 ? launch_t<R, kLLF, true>(a, grid, block, stream) : launch_t<R, kLLF, false>(a, grid, block, stream); break;
  }
}

const oct_tile::Tables& tile_tables() {
  static constexpr oct_tile::Tables t = oct_tile::make_tables();
  return t;
}

hipError_t launch_unsplit(const UnsplitArgs& a, bool fp32, hipStream_t stream) {
  const long threads = a.ngroups * 12L * a.nv;
  if (threads <= 0) return hipSuccess;
  // Rows (27-point slopes): any multiple of 64 works with the flat (batch,
  // row, lane) mapping.  The autotuner picks per device.
  const int block = tuning().unsplit_block ? tuning().unsplit_block : 256;
  const long grid = (threads + block - 1) / block;
  if (fp32)
    launch_r<float>(a, grid, block, stream);
  else
    launch_r<double>(a, grid, block, stream);
  return hipGetLastError();
}

}  // namespace ramses
