// One level of an oct-tree (AMR) godunov sweep on the GPU:
// godfine1 (hydro/godunov_fine.f90:486-911) over the level's active octs, all
// reading the tree (son / father / nbor) and the state (uold / unew) resident
// in HBM in the reference's memory model:
//   amr_tile     16 octs per workgroup: their 80-cell stencils gathered into
//                LDS (get3cubefather/get3cubepos, amr/nbors_utils.f90:5-300; a
//                missing neighbour oct is a buffer oct interpolated from its
//                father's 7-point neighbourhood: getnborfather :404-525 and
//                interpol_hydro, hydro/interpol_hydro.f90:268-637), unsplit
//                with a zero flux at faces next to a refined cell (:720-749),
//                and the level update unew += F(i) - F(i+1) (:751-792);
//   amr_reflux   the conservative correction of coarser leaf neighbours
//                (:798-908), gathered per coarse cell and summed in the
//                reference's order (batch, dimension, side, face) so the
//                result is bitwise and deterministic without atomics.
// The 27-point slopes and the prolongations of interpol_var 1 and 2 take the
// staged form of amr_tile: amr_gather (6x6x6 stencils in nvector-strided
// batches), amr_unsplit (the rows or faces of unsplit_device.hpp) and
// amr_update.
// Index conventions are the reference's (1-based cells and grids; arrays
// are passed so that element i of the reference is p[i]).
#include <type_traits>

#include "hydro_device.hpp"
#include "unsplit_args.hpp"
#include "amr_args.hpp"
#include "amr_device.hpp"
#include "unsplit_device.hpp"
#include "oct_tile.hpp"

namespace ramses {
hipError_t launch_cons_finish(const double* partials, long nblocks, double* out, int accumulate, hipStream_t s);


namespace {

// One (batch b, father neighbour j in 0..26, lane) task.
__device__ __forceinline__ void gather_task(const AmrLevelArgs& a, int noct, int b, int j, int lane) {
  const int nv = a.nv;
  const int oct = b * nv + lane;
  if (oct >= noct) return;
  const AmrTreeView& t = a.t;
  const int igrid = a.active[oct];
  const long f = t.father[igrid];
  const int i1 = j % 3, j1 = (j / 3) % 3, k1 = j / 9;
  const long nf = nbor_father_cell(t, f, i1, j1, k1, a.ilevel);
  if (nf <= 0) {
    atomicOr(a.error, 1);
    return;
  }
  const int igrid_n = t.son[nf];
  const size_t us = (size_t)nv * 216;               // variable stride in uin
  double* uin = a.uin + (size_t)b * us * 5 + lane;
  unsigned char* ok = a.ok + (size_t)b * us + lane;
  // Every load of a branch is issued before its first store: the stores into
  // uin could alias uold as far as the compiler knows, so interleaving them
  // would serialise the 40 loads into a chain of memory latencies.
  if (igrid_n > 0) {
    double val[8][5];
    unsigned char okv[8];
#pragma unroll
    for (int ind = 1; ind <= 8; ++ind) {
      const long c = cell_of(t, ind, igrid_n);
#pragma unroll
      for (int v = 0; v < 5; ++v) val[ind - 1][v] = a.uold[(long)v * a.ustride + c];
      okv[ind - 1] = t.son[c] > 0 ? 1 : 0;
    }
#pragma unroll
    for (int ind = 1; ind <= 8; ++ind) {
      const int i2 = (ind - 1) & 1, j2 = ((ind - 1) >> 1) & 1, k2 = (ind - 1) >> 2;
      const int i3 = 1 + 2 * (i1 - 1) + i2, j3 = 1 + 2 * (j1 - 1) + j2, k3 = 1 + 2 * (k1 - 1) + k2;
      const size_t s = (size_t)((i3 + 1) + 6 * ((j3 + 1) + 6 * (k3 + 1))) * nv;
#pragma unroll
      for (int v = 0; v < 5; ++v) uin[s + (size_t)v * us] = val[ind - 1][v];
      ok[s] = okv[ind - 1];
    }
  } else {
    long nb7[7];
    nbor_father7(t, nf, a.ilevel, nb7);
    double u1[7][5], u2[8][5];
#pragma unroll
    for (int q = 0; q < 7; ++q)
#pragma unroll
      for (int v = 0; v < 5; ++v) u1[q][v] = a.uold[(long)v * a.ustride + nb7[q]];
    interpol_oct(u1, u2, a.interpol_type, a.interpol_var, a.hp.smallr);
#pragma unroll
    for (int ind = 1; ind <= 8; ++ind) {
      const int i2 = (ind - 1) & 1, j2 = ((ind - 1) >> 1) & 1, k2 = (ind - 1) >> 2;
      const int i3 = 1 + 2 * (i1 - 1) + i2, j3 = 1 + 2 * (j1 - 1) + j2, k3 = 1 + 2 * (k1 - 1) + k2;
      const size_t s = (size_t)((i3 + 1) + 6 * ((j3 + 1) + 6 * (k3 + 1))) * nv;
#pragma unroll
      for (int v = 0; v < 5; ++v) uin[s + (size_t)v * us] = u2[ind - 1][v];
      ok[s] = 0;
    }
  }
}

// Flat grid-stride over the 27*nv tasks of every batch, lane fastest, so a
// wavefront covers two neighbours j of 32 octs and every (cell, variable)
// store is one coalesced segment.  A level of a few thousand octs spreads
// over all CUs instead of one workgroup per batch: each task is a chain of
// dependent tree loads, and the chains of one CU share its memory pipeline.
__global__ __launch_bounds__(256) void amr_gather(AmrLevelArgs a) {
  const int noct = level_count(a.noct, a.dnoct);
  const int nv = a.nv;
  const long per_batch = 27L * nv;
  const long ntask = (long)((noct + nv - 1) / nv) * per_batch;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < ntask; t += (long)gridDim.x * blockDim.x) {
    const int b = (int)(t / per_batch);
    const int rem = (int)(t - b * per_batch);
    gather_task(a, noct, b, rem / nv, rem % nv);
  }
}

__device__ __forceinline__ size_t fslot(int i3, int j3, int k3) { return (size_t)((i3 - 1) + 3 * ((j3 - 1) + 3 * (k3 - 1))); }

// Level update of one (cell ind, variable v) of lane `lane` of batch b, q =
// (ind-1)*5 + v: unew += flux(i3) - flux(i3+1) for idim = 1, 2, 3 in order
// (hydro/godunov_fine.f90:751-792).
__device__ __forceinline__ void update_cell(const AmrLevelArgs& a, int b, int q, int lane) {
  const int nv = a.nv;
  const size_t fvs = (size_t)nv * 27;
  const double* flux = a.flux + (size_t)b * fvs * 15;
  const int ind = q / 5 + 1, v = q % 5;
  const int i2 = (ind - 1) & 1, j2 = ((ind - 1) >> 1) & 1, k2 = (ind - 1) >> 2;
  const int i3 = 1 + i2, j3 = 1 + j2, k3 = 1 + k2;
  const long c = (long)v * a.ustride + cell_of(a.t, ind, a.active[b * nv + lane]);
  double acc = a.unew[c];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int i0 = d == 0, j0 = d == 1, k0 = d == 2;
    const size_t base = (size_t)27 * (v + 5 * d);
    const double fl = flux[(fslot(i3, j3, k3) + base) * nv + lane];
    const double fr = flux[(fslot(i3 + i0, j3 + j0, k3 + k0) + base) * nv + lane];
    acc = acc + (fl - fr);
  }
  a.unew[c] = acc;
}

// The level's unsplit over all batches (workgroups of 128), the flux reset
// at faces next to a refined cell folded into the face stores: one (batch,
// face, lane) task per thread on levels of at most u.face_octs octs, where
// the chain of dependent steps matters more than the arithmetic, else one
// (batch, row, lane) task per thread.  Small levels spread over every CU.
// The levels carry no gravity array (u.grav is null), so the tasks are the
// gravity-free ones.
template <typename R, int RS, bool S27, int ST>
__global__ __launch_bounds__(768) void amr_unsplit(AmrLevelArgs a, UnsplitArgs u) {
  const int noct = level_count(a.noct, a.dnoct);
  const int nv = a.nv;
  const int nb = (noct + nv - 1) / nv;
  const int ngrid_last = noct - (nb - 1) * nv;
  const long stride = (long)gridDim.x * blockDim.x;
  if (noct <= u.face_octs) {
    const long ntask = (long)nb * 36 * nv;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < ntask; t += stride)
      unsplit_dev::face_task<R, RS, S27, true, ST, false>(u, t, nb, ngrid_last);
  } else {
    const long ntask = (long)nb * 12 * nv;
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < ntask; t += stride)
      unsplit_dev::unsplit_task<R, RS, S27, true, ST, false>(u, t, nb, ngrid_last);
  }
}

// The level update, one (batch, cell, variable, lane) task per thread.
__global__ __launch_bounds__(256) void amr_update(AmrLevelArgs a) {
  const int noct = level_count(a.noct, a.dnoct);
  const int nv = a.nv;
  const long per_batch = 40L * nv;
  const long ntask = (long)((noct + nv - 1) / nv) * per_batch;
  for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < ntask; t += (long)gridDim.x * blockDim.x) {
    const int b = (int)(t / per_batch);
    const int rem = (int)(t - b * per_batch);
    const int lane = rem % nv;
    if (b * nv + lane < noct) update_cell(a, b, rem / nv, lane);
  }
}

// godfine1 of one level without its reflux, 16 octs per workgroup
// (oct_tile.hpp): the stencil gather, the unsplit chain and the level update
// in one kernel, the stencil and the fluxes in LDS.  Global memory sees the
// tree, the state, the update, and the fluxes through the sides where the
// neighbour oct is missing, which are all that amr_reflux reads.
//
// The separate kernels stage 13.4 KB per oct through memory: on a level of
// 2^17 octs the gather took 0.40 ms, the solve 0.20 and the update 0.05; and
// a level of a thousand octs paid three launches of 5 to 17 us.
//
// Gather: one (father neighbour, oct) task per thread, 27 x 16 of the 512.
// The neighbours are ordered by how many of their cells a face depends on
// (centre and sides 8, edges 2, corners none, which are only checked to
// exist), so a wavefront loads alike.  The conserved state goes to LDS one
// variable at a time, which keeps a task's prolongation in registers.
// interpol_var 0 only: the other modes mix the variables.
//
// What bounds it is the gather: on 10^5 octs in FP64 17,000 of a tile's
// 30,000 cycles (FP32-mixed 16,300 of 26,400), which the other workgroup of
// the CU fills in part (vector issue is busy half the time).  The wavefronts
// of the corner neighbours, which only walk the tree, take 4,400 of them, the
// edges' 7,500 and the two of centre and sides, eight cells of five variables
// and their sons, 15,000 and 17,000.  Tiles next to each other in the level's
// list run on one XCD, whose L2 then holds the cells that their stencils share
// (on 10^5 octs 262 -> 250 us, on 3 10^4 98 -> 90), and the state to update
// is loaded while the faces are solved (another 1%).
template <typename R, int RS, int ST>
__global__ __launch_bounds__(oct_tile::kThreads)
__attribute__((amdgpu_waves_per_eu(4, 8))) void amr_tile(AmrLevelArgs a, double dx, const double* d_dt) {
  using namespace oct_tile;
  // the conserved state of the 80 cells, then their primitives, then the
  // traced states (R), then the fluxes
  __shared__ double sd[kLds];
  __shared__ unsigned char refined[kPairs];   // by slot and oct
  __shared__ unsigned char missing[6][kOcts]; // by side
  constexpr int kOwn = (40 * kOcts + kThreads - 1) / kThreads;
  R* s = reinterpret_cast<R*>(sd);
  const int noct = level_count(a.noct, a.dnoct);
  const int ntiles = (noct + kOcts - 1) / kOcts;
  const AmrTreeView& t = a.t;
  const HydroParams hp = a.hp;
  const double dt = *d_dt;
  const SolverConsts<R> sc = scalar(make_consts<R>(hp));
  const FluxScale fs = scalar(make_scale(dt, dx));
  const double dtxhalf = scalar(dt * 0.5);
  const double smalle = scalar(hp.smallc * hp.smallc / hp.gamma / (hp.gamma - 1.0));  // hydro/umuscl.f90:884
  const R h = scalar((R)(dt / dx));
  const R dtdx[3] = {h, h, h};
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    // opaque to the compiler, which would otherwise carry the addresses of
    // every step across the loop and spill them
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int l = tid % kOcts;
    const int o = (int)xcd_contiguous(tile, ntiles) * kOcts + l;
    const bool valid = o < noct;
    const int igrid = a.active[valid ? o : noct - 1];
    const int k27 = tid / kOcts;
    if (k27 < 27) {
      const int j = kTab.order[k27];
      const int i1 = j % 3, j1 = (j / 3) % 3, k1 = j / 9;
      const long nf = nbor_father_cell(t, t.father[igrid], i1, j1, k1, a.ilevel);
      if (nf <= 0) atomicOr(a.error, 1);
      if (nf > 0 && k27 < 19) {
        const int gn = t.son[nf];
        unsigned long long sub = kTab.sub[j];
        if (k27 >= 1 && k27 < 7) {  // side 2*d + (plus side)
          const int side = i1 != 1 ? (i1 >> 1) : (j1 != 1 ? 2 + (j1 >> 1) : 4 + (k1 >> 1));
          missing[side][l] = gn <= 0;
        }
        if (gn > 0) {
          if (k27 < 7) {
#pragma unroll
            for (int i = 0; i < 8; ++i) refined[(int)(sub >> 8 * i & 255) * kOcts + l] = t.son[cell_of(t, i + 1, gn)] > 0;
#pragma unroll
            for (int v = 0; v < 5; ++v) {
              double w[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) w[i] = a.uold[(long)v * a.ustride + cell_of(t, i + 1, gn)];
#pragma unroll
              for (int i = 0; i < 8; ++i) sd[(int)(sub >> 8 * i & 255) * kCellStride + v * kOcts + l] = w[i];
            }
          } else {
            // an edge neighbour's two cells on the oct's side of it
            const int free_bit = i1 == 1 ? 1 : (j1 == 1 ? 2 : 4);
            const int i0 = (i1 == 0 ? 1 : 0) + (j1 == 0 ? 2 : 0) + (k1 == 0 ? 4 : 0);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
              const int i = i0 + (q ? free_bit : 0);
              const long c = cell_of(t, i + 1, gn);
              double* p = sd + (int)(sub >> 8 * i & 255) * kCellStride + l;
              double w[5];
#pragma unroll
              for (int v = 0; v < 5; ++v) w[v] = a.uold[(long)v * a.ustride + c];
#pragma unroll
              for (int v = 0; v < 5; ++v) p[v * kOcts] = w[v];
            }
          }
        } else {
          long nb7[7];
          nbor_father7(t, nf, a.ilevel, nb7);
#pragma unroll 1
          for (int v = 0; v < 5; ++v) {
            double u7[7], u8[8];
#pragma unroll
            for (int q = 0; q < 7; ++q) u7[q] = a.uold[(long)v * a.ustride + nb7[q]];
            interpol_cons(u7, u8, a.interpol_type);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const int slot = (int)(sub >> 8 * i & 255);
              if (slot != 255) sd[slot * kCellStride + v * kOcts + l] = u8[i];
            }
          }
          if (k27 < 7) {
#pragma unroll
            for (int i = 0; i < 8; ++i) refined[(int)(sub >> 8 * i & 255) * kOcts + l] = 0;
          }
        }
      }
    }
    __syncthreads();
    // In FP64 a cell's primitives go over its conserved state; FP32's
    // packed ones go over other cells' state, after a barrier.
    Prim<R> q[kLoads];
#pragma unroll
    for (int k = 0; k < kLoads; ++k) {
      const int e = tid + k * kThreads;
      if (e < kPairs) {
        const double* p = sd + (e / kOcts) * kCellStride + e % kOcts;
        q[k] = ctoprim_cell<R>(p[0], p[kOcts], p[2 * kOcts], p[3 * kOcts], p[4 * kOcts], 0.0, 0.0, 0.0, dtxhalf,
                               smalle, hp);
        if constexpr (sizeof(R) == 8) put_prim(s, e, q[k]);
      }
    }
    __syncthreads();
    if constexpr (sizeof(R) == 4) {
#pragma unroll
      for (int k = 0; k < kLoads; ++k) {
        const int e = tid + k * kThreads;
        if (e < kPairs) put_prim(s, e, q[k]);
      }
      __syncthreads();
    }
    // the update's own state, in flight while the faces are solved
    double own[kOwn];
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int e = tid + k * kThreads;
      own[k] = valid && e < 40 * kOcts ? a.unew[(long)(e / kOcts % 5) * a.ustride + cell_of(t, e / (5 * kOcts) + 1, igrid)] : 0.0;
    }
    trace_tile<R, ST>(s, tid, sc, dtdx);
    // fluxes, (f*dt)/dx in conserved order, zero next to a refined cell
    // (hydro/godunov_fine.f90:720-749); each face's go over its own traced
    // states, which only its wavefront reads
    for (int k = 0; k < 2; ++k) {
      const int f = tile_face(tid, k);
      if (f < 0) continue;
      const Face<R> fl = get_side(s, f, 0, l), fr = get_side(s, f, 1, l);
      const Flux6<R> fg = riemann_fixed<R, RS>(fl, fr, sc);
      const R val[5] = {fg.f[0], fg.f[1], fg.f[3], fg.f[4], fg.f[2]};
      double out[5];
      scale_flux<5>(val, fs, out);
      if (refined[kTab.side[f][0] * kOcts + l] | refined[kTab.side[f][1] * kOcts + l]) {
#pragma unroll
        for (int v = 0; v < 5; ++v) out[v] = 0.0;
      }
      const int d = __builtin_amdgcn_readfirstlane(f) / 12, x = __builtin_amdgcn_readfirstlane(f) / 4 % 3;
      const int m1 = 1 + d, m2 = d == 0 ? 2 : 1, m3 = d == 2 ? 2 : 3;  // the momenta in their own order
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // the reads above stay above
      double* p = reinterpret_cast<double*>(s + f * kFaceStride) + l;
      p[0] = out[0];
      p[m1 * kOcts] = out[1];
      p[m2 * kOcts] = out[2];
      p[m3 * kOcts] = out[3];
      p[4 * kOcts] = out[4];
      if (x != 1 && valid && missing[2 * d + (x >> 1)][l]) {
        const size_t fvs = (size_t)a.nv * 27;
        double* flux = a.flux + (size_t)(o / a.nv) * fvs * 15 + (size_t)(kTab.out[f] + 27 * 5 * d) * a.nv + o % a.nv;
        flux[0] = out[0];
        flux[m1 * fvs] = out[1];
        flux[m2 * fvs] = out[2];
        flux[m3 * fvs] = out[3];
        flux[4 * fvs] = out[4];
      }
    }
    __syncthreads();
    // unew += flux(i) - flux(i+1) for x, y, z in order (:751-792): 8 cells x
    // 5 variables x 16 octs
#pragma unroll
    for (int k = 0; k < kOwn; ++k) {
      const int e = tid + k * kThreads;
      if (e >= 40 * kOcts) continue;
      const int ind = e / (5 * kOcts), v = e / kOcts % 5;
      const int x[3] = {ind & 1, (ind >> 1) & 1, ind >> 2};
      if (valid) {
        const long c = (long)v * a.ustride + cell_of(t, ind + 1, igrid);
        double acc = own[k];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int T = d == 0 ? x[1] + 2 * x[2] : (d == 1 ? x[0] + 2 * x[2] : x[0] + 2 * x[1]);
          const R* p = s + (12 * d + 4 * x[d] + T) * kFaceStride;
          acc = acc + (reinterpret_cast<const double*>(p)[v * kOcts + l] -
                       reinterpret_cast<const double*>(p + 4 * kFaceStride)[v * kOcts + l]);
        }
        a.unew[c] = acc;
      }
    }
    __syncthreads();
  }
}

// The solve of the staged path: the 27-point slopes, whose faces depend on
// the whole 6^3 stencil, and prolongations that mix the variables (minmod
// there too with the limiter fixed at compile time).
template <typename R, int RS>
void launch_solve(const AmrLevelArgs& a, const UnsplitArgs& u, unsigned grid, unsigned block, hipStream_t s) {
  if (a.hp.slope_type == 3)
    hipLaunchKernelGGL((amr_unsplit<R, RS, true, -1>), dim3(grid), dim3(block), 0, s, a, u);
  else if (a.hp.slope_type == 1)
    hipLaunchKernelGGL((amr_unsplit<R, RS, false, 1>), dim3(grid), dim3(block), 0, s, a, u);
  else
    hipLaunchKernelGGL((amr_unsplit<R, RS, false, -1>), dim3(grid), dim3(block), 0, s, a, u);
}

// Minmod (the reference's default slope) has the limiter fixed at compile
// time; other slope types take it at run time.
template <typename R, int RS>
void launch_tile(const AmrLevelArgs& a, double dx, const double* d_dt, unsigned grid, hipStream_t s) {
  if (a.hp.slope_type == 1)
    hipLaunchKernelGGL((amr_tile<R, RS, 1>), dim3(grid), dim3(oct_tile::kThreads), 0, s, a, dx, d_dt);
  else
    hipLaunchKernelGGL((amr_tile<R, RS, -1>), dim3(grid), dim3(oct_tile::kThreads), 0, s, a, dx, d_dt);
}

// f(std::integral_constant<int, RS>) for the configured solver.
template <typename F>
void with_solver(int riemann, F f) {
  switch (riemann) {
    case kHLLC: f(std::integral_constant<int, kHLLC>{}); break;
    case kHLL: f(std::integral_constant<int, kHLL>{}); break;
    case kACOUSTIC:
    case kEXACT: f(std::integral_constant<int, kDynamicRiemann>{}); break;
    default: f(std::integral_constant<int, kLLF>{}); break;
  }
}

constexpr unsigned kRefluxSplit = 1u << 16;  // (see reflux_tasks)
constexpr unsigned kRefluxFew = 1u << 12;
__host__ __device__ inline bool reflux_from_coarse(unsigned nf, unsigned nc) {
  return nc <= kRefluxFew || 8ULL * nc <= 6ULL * nf;
}

// Conservative correction of the coarser leaf cells next to the level's
// octs.  A coarse leaf c receives from each fine oct o that sits across one
// of its faces the four (reset) fluxes of o's boundary faces on c's side,
// times -1/8 (c left of o) or +1/8 (c right of o).  The reference adds them
// in loop order: batch of o, then dimension, then side, then face (k3, j3,
// i3); the same order is rebuilt here from the position of o in the level's
// active list.  Variables [v0, v1); first: the key of the contributor through
// which c was found, or -1 where c is visited once.
__device__ __forceinline__ void reflux_cell(const AmrLevelArgs& a, int g, int ind, long c, int v0, int v1, int first) {
  const AmrTreeView& t = a.t;
  const int p[3] = {(ind - 1) & 1, ((ind - 1) >> 1) & 1, (ind - 1) >> 2};
  // the six neighbour cells first (independent loads), then their sons
  long nc[6];
#pragma unroll
  for (int in = 1; in <= 6; ++in) {
    const int ax = (in - 1) >> 1, plus = (in - 1) & 1;
    const bool inside = plus ? (p[ax] == 0) : (p[ax] == 1);
    int q[3] = {p[0], p[1], p[2]};
    q[ax] = 1 - p[ax];
    const int gn = inside ? g : t.son[nbor_of(t, g, in)];
    nc[in - 1] = gn > 0 ? cell_of(t, 1 + q[0] + 2 * q[1] + 4 * q[2], gn) : 0;
  }
  int so[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) so[k] = nc[k] > 0 ? t.son[nc[k]] : 0;
  int pz[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) pz[k] = so[k] > 0 ? a.pos[so[k]] : 0;
  // up to 6 contributing octs: key = batch*6 + 2*d + side in the upper half,
  // the oct's position below; a fixed network sorts them (as an array indexed
  // by their number they would live in scratch memory)
  constexpr long long kNone = 0x7fffffffffffffffLL;
  long long kp[6];
#pragma unroll
  for (int in = 1; in <= 6; ++in) {
    const int ax = (in - 1) >> 1, plus = (in - 1) & 1;
    kp[in - 1] = kNone;
    if (any_lane(so[in - 1] > 0)) {
      // c is on o's minus side when n is c's plus neighbour
      const long long key = (long long)(pz[in - 1] / a.nv) * 6 + 2 * ax + (plus ? 0 : 1);
      if (so[in - 1] > 0) kp[in - 1] = key << 32 | (long long)pz[in - 1];
    }
  }
  auto order = [&](int i, int k) {
    const long long lo = kp[i] < kp[k] ? kp[i] : kp[k], hi = kp[i] < kp[k] ? kp[k] : kp[i];
    kp[i] = lo;
    kp[k] = hi;
  };
  order(1, 2); order(4, 5); order(0, 2); order(3, 5); order(0, 1); order(3, 4);
  order(2, 5); order(0, 3); order(1, 4); order(2, 4); order(1, 3); order(2, 3);
  if (kp[0] == kNone) return;
  if (first >= 0 && (int)(kp[0] >> 32) != first) return;  // the first contributor takes the cell
  const int nv = a.nv;
  const size_t fvs = (size_t)nv * 27;
  const double oneontwotondim = 1.0 / 8.0;
  // The oct side's 2x2 faces: the transverse coordinates run over {1,2} and
  // the normal one is 1 (side 0, the oct's minus face) or 3 (side 1).  Formed
  // only for as many contributors as some lane has.
  const double* fe[6];
  int f1[6], f2[6];  // steps along the lower and the upper transverse axis
#pragma unroll
  for (int e = 0; e < 6; ++e) {
    fe[e] = nullptr;
    f1[e] = f2[e] = 0;
    if (any_lane(kp[e] != kNone)) {
      const int key = (int)(kp[e] >> 32), pos = (int)kp[e];
      const int b = key / 6, d = (key - 6 * b) >> 1, side = key & 1;
      f1[e] = d == 0 ? 3 * nv : nv;
      f2[e] = d == 2 ? 3 * nv : 9 * nv;
      fe[e] = a.flux + (size_t)b * fvs * 15 + (pos - b * nv) + (27 * 5 * d + side * (d == 0 ? 2 : (d == 1 ? 6 : 18))) * nv;
    }
  }
  // All contributions are loaded first (independent loads, issued together),
  // then summed in the reference's order: contributor e by key, and within
  // it the 4 faces of the oct side in (k3, j3, i3) loop order.
  for (int v = v0; v < v1; ++v) {
    double fv[6][4];
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      if (kp[e] == kNone) break;
      const double* flux = fe[e] + (size_t)v * fvs;
#pragma unroll
      for (int q = 0; q < 4; ++q) fv[e][q] = flux[(q & 1) * f1[e] + (q >> 1) * f2[e]];
    }
    double s = a.unew[(long)v * a.ustride + c];
#pragma unroll
    for (int e = 0; e < 6; ++e) {
      if (kp[e] == kNone) break;
      const int side = (int)(kp[e] >> 32) & 1;
#pragma unroll
      for (int q = 0; q < 4; ++q) s = side ? s + fv[e][q] * oneontwotondim : s - fv[e][q] * oneontwotondim;
    }
    a.unew[(long)v * a.ustride + c] = s;
  }
}

// The leaves are found from the side with fewer tasks: every cell of the
// coarser level, or every side of the level's own octs where the neighbour
// oct is missing (its cell is the leaf), of which the first in the
// reference's order takes the cell.  Behind 2,000 octs on a level of 32,768
// the first way takes 8.1 us, the second 6.8; behind 95,000 14.3 and 21.7.
// The first walk is two dependent loads shorter, so coarser levels of few
// octs, where latency is all there is, always take it (4,096 octs: 5.3
// against 6.8 us behind 2,000 and 5.6 against 7.7 behind 400).  Where that is
// few tasks, each variable is a task of its own: the walk is repeated, but
// the kernel is bound by latency then.  blk of nblk workgroups.
__device__ __forceinline__ void reflux_tasks(const AmrLevelArgs& a, unsigned blk, unsigned nblk) {
  const AmrTreeView& t = a.t;
  const unsigned nf = (unsigned)level_count(a.noct, a.dnoct), nc = (unsigned)level_count(a.noct_coarse, a.dnoct_coarse);
  if (nf == 0 || nc == 0) return;
  const unsigned stride = nblk * blockDim.x, id = blk * blockDim.x + threadIdx.x;
  const bool coarse = reflux_from_coarse(nf, nc);
  const unsigned per = coarse ? 8 * nc : 6 * nf;  // below 2^31, as cell indices are
  const unsigned split = per < kRefluxSplit ? 5 : 1;
  const unsigned octs = coarse ? nc : nf;
  for (unsigned i = id; i < per * split; i += stride) {
    const unsigned v0 = split == 1 ? 0 : i / per, r = split == 1 ? i : i - v0 * per;
    const int v1 = split == 1 ? 5 : (int)v0 + 1;
    const unsigned k = r / octs, o = r - k * octs;  // (cell or side, oct), the oct fastest
    int g, ind, first;
    long c;
    if (coarse) {
      g = a.active_coarse[o];
      ind = (int)k + 1;
      c = cell_of(t, ind, g);
      first = -1;
    } else {
      c = nbor_of(t, a.active[o], (int)k + 1);
      if (c <= t.ncoarse) continue;
      const unsigned q = (unsigned)(c - t.ncoarse - 1), m = q / (unsigned)t.ngridmax;
      g = (int)(q - m * (unsigned)t.ngridmax) + 1;
      ind = (int)m + 1;
      first = (int)(o / a.nv) * 6 + (int)k;  // c lies on the oct's side k: the same key as reflux_cell's
    }
    if (t.son[c] == 0) reflux_cell(a, g, ind, c, (int)v0, v1, first);  // only leaves (:811,863)
  }
}

__global__ __launch_bounds__(256) void amr_reflux(AmrLevelArgs a) { reflux_tasks(a, blockIdx.x, gridDim.x); }

// The cells of a level, 32 octs x 8 cells per 256 threads and turn: 32
// consecutive octs per cell, so that a variable is read in runs of 256 bytes
// where the octs are (cell by cell of each oct it is runs of 64), and no
// division finds the cell.  The oct count is the host value or, with dn set,
// the one in device memory; f(igrid, ind); blk of nblk workgroups of a
// multiple of 256 threads.
template <typename F>
__device__ __forceinline__ void for_level_cells(const int* active, int noct, int blk, int nblk, F f) {
  const int ind = (int)(threadIdx.x >> 5 & 7) + 1, per = (int)(blockDim.x >> 8);
  const int first = (blk * per + (int)(threadIdx.x >> 8)) * 32 + (int)(threadIdx.x & 31);
  for (int o = first; o < noct; o += nblk * per * 32) f(active[o], ind);
}
template <typename F>
__device__ __forceinline__ void for_level_cells(const int* active, int noct, F f) {
  for_level_cells(active, noct, (int)blockIdx.x, (int)gridDim.x, f);
}

// set_unew / set_uold over the level's active cells (hydro/godunov_fine.f90:58-65, 193-197).
__global__ __launch_bounds__(256) void amr_copy_level(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                     const double* src, double* dst, long ustride) {
  for_level_cells(active, level_count(noct_h, dn), [&](int g, int ind) {
    const long c = cell_of(t, ind, g);
    double q[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = src[(long)v * ustride + c];
#pragma unroll
    for (int v = 0; v < 5; ++v) dst[(long)v * ustride + c] = q[v];
  });
}

// upl for one refined cell c with son oct s: the average of its children
// (hydro/interpol_hydro.f90:72-263). Density with the smallr floor, then
// momenta and total energy, each summed over the children in order and /8;
// with interpol_var 1 or 2 the energy is instead rebuilt from the children's
// average internal energy plus the kinetic energy of the averaged state.
__device__ inline void upl_cell(const AmrTreeView& t, double* u, long ustride, long c, int s, double smallr,
                                int ivar_mode) {
  double getx = 0.0;
  for (int ind = 1; ind <= 8; ++ind) getx = getx + fmax_f(u[cell_of(t, ind, s)], smallr);
  double out[5];
  out[0] = getx / 8.0;
  for (int v = 1; v < 5; ++v) {
    getx = 0.0;
    for (int ind = 1; ind <= 8; ++ind) getx = getx + u[(long)v * ustride + cell_of(t, ind, s)];
    out[v] = getx / 8.0;
  }
  if (ivar_mode == 1 || ivar_mode == 2) {
    getx = 0.0;
    for (int ind = 1; ind <= 8; ++ind) {
      const long cs = cell_of(t, ind, s);
      const double rho = fmax_f(u[cs], smallr);
      double ekin = 0.0;
      for (int d = 1; d <= 3; ++d) {
        const double m = u[(long)d * ustride + cs];
        ekin = ekin + 0.5 * (m * m) / rho;
      }
      getx = getx + u[4 * ustride + cs] - ekin;
    }
    const double rho = fmax_f(out[0], smallr);
    double ekin = 0.0;
    for (int d = 1; d <= 3; ++d) ekin = ekin + 0.5 * (out[d] * out[d]) / rho;
    out[4] = getx / 8.0 + ekin;
  }
  for (int v = 0; v < 5; ++v) u[(long)v * ustride + c] = out[v];
}

// upload_fine: refined cells of the level get the average of their children
// (hydro/interpol_hydro.f90:5-67).  flag1 (or null): flag every cell too, all
// that flag_fine does below levelmin (init_flag, amr/flag_utils.f90:150-157).
__global__ __launch_bounds__(256) void amr_upload(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                 double* u, long ustride, double smallr, int ivar_mode, int* flag1) {
  for_level_cells(active, level_count(noct_h, dn), [&](int g, int ind) {
    const long c = cell_of(t, ind, g);
    const int s = t.son[c];
    if (flag1) flag1[c] = 1;
    if (s > 0) upl_cell(t, u, ustride, c, s, smallr, ivar_mode);
  });
}

// set_uold followed by upload_fine of the level in one pass
// (hydro/godunov_fine.f90:135-232, hydro/interpol_hydro.f90:5-263): a leaf
// takes unew, a refined cell the average of its children's uold (set_uold
// writes every cell and upload_fine then rewrites the refined ones, so the
// result is the same).  The first thread also ends the level step's time
// bookkeeping: dtnew(l-1) = dtnew(l) if nsubcycle(l-1) == 1, or dtold(l) +
// dtnew(l) after the second substep (amr/amr_step.f90:573-576); nsub_coarser
// 0: level l is levelmin.  The first `refluxers` workgroups do the level's
// reflux instead (reflux_tasks), which reads its fluxes and adds to the
// coarser level's unew: neither touches what the other reads.
__global__ __launch_bounds__(256) void amr_finish(AmrLevelArgs a, double* u, int ivar_mode, double* dt,
                                                 const double* dtold, int nsub_coarser, int icount, int refluxers) {
  if ((int)blockIdx.x < refluxers) {
    reflux_tasks(a, blockIdx.x, (unsigned)refluxers);
    return;
  }
  const AmrTreeView& t = a.t;
  const double* unew = a.unew;
  const long ustride = a.ustride;
  const double smallr = a.hp.smallr;
  const int l = a.ilevel;
  const int noct = level_count(a.noct, a.dnoct);
  if ((int)blockIdx.x == refluxers && threadIdx.x == 0 && noct > 0 && nsub_coarser > 0) {
    if (nsub_coarser == 1) dt[l - 1] = dt[l];
    if (icount == 2) dt[l - 1] = dtold[l] + dt[l];
  }
  for_level_cells(a.active, noct, (int)blockIdx.x - refluxers, (int)gridDim.x - refluxers, [&](int g, int ind) {
    const long c = cell_of(t, ind, g);
    const int s = t.son[c];
    if (s <= 0) {
      double q[5];
#pragma unroll
      for (int v = 0; v < 5; ++v) q[v] = unew[(long)v * ustride + c];
#pragma unroll
      for (int v = 0; v < 5; ++v) u[(long)v * ustride + c] = q[v];
    } else {
      upl_cell(t, u, ustride, c, s, smallr, ivar_mode);
    }
  });
}

// The workgroup's largest w, in thread 0.
__device__ __forceinline__ double block_max(double w) {
  __shared__ double red[16];
  for (int off = 32; off > 0; off >>= 1) w = fmax_f(w, __shfl_xor(w, off, 64));
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = w;
  __syncthreads();
  if (threadIdx.x == 0)
    for (int k = 1; k < (int)(blockDim.x >> 6); ++k) w = fmax_f(w, red[k]);
  return w;
}

// courant_fine over the level's leaf cells (hydro/courant_fine.f90:44-131):
// block max of the cmpdt wave speed, block dt limit min-combined (exact,
// see cmpdt_w).
__global__ __launch_bounds__(256) void amr_courant(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                  const double* u, long ustride, double dx, HydroParams hp,
                                                  double* d_dt) {
  double w = 0.0;
  for_level_cells(active, level_count(noct_h, dn), [&](int g, int ind) {
    const long c = cell_of(t, ind, g);
    if (t.son[c] == 0)
      w = fmax_f(w, cmpdt_w(u[c], u[ustride + c], u[2 * ustride + c], u[3 * ustride + c], u[4 * ustride + c], hp));
  });
  w = block_max(w);
  if (threadIdx.x == 0 && w > 0.0)
    atomicMin(reinterpret_cast<unsigned long long*>(d_dt), dt_bits(cmpdt_from_w(w, dx, hp)));
}

// set_unew, newdt_fine and courant_fine of a level in one pass over its
// cells (hydro/godunov_fine.f90:40-130, pm/newdt_fine.f90:51,177,
// hydro/courant_fine.f90:44-131): every cell copies uold to unew and every
// leaf joins the max of the cmpdt wave speed in d.wmax.  The workgroup that
// finishes last does the level's time-step bookkeeping (amr/amr_step.f90):
//   dtold(l) = dtnew(l); dtnew(l) = min(start, dtnew(l-1)/nsubcycle(l-1)
//   below levelmin, the limit of the largest wave speed) (:327-330; the dt
//   limit is non-increasing in the wave speed and min is exact, so the order
//   of the minima does not matter), and where no finer level has octs
//   dtold(l+1) = dtnew(l+1) = dtnew(l)/nsubcycle(l), t += dtnew(l) (:353-362,
//   amr/update_time.f90:217,331); cnt counts update_time calls (nstep) and
//   cell updates.
// As kernels of one thread before and after the pass these took 2.6 us each,
// twice a level step.  At most 256 workgroups of 1024: their two atomics meet
// at one address each (3,600 workgroups of 256 took 78 us for a level of
// 115k octs, 36 of them for these).
constexpr int kBeginThreads = 1024;
__global__ __launch_bounds__(kBeginThreads) void amr_begin(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                const double* u, double* unew, long ustride, double dx,
                                                HydroParams hp, AmrStepDt d, double* partials) {
  const int noct = level_count(noct_h, dn);
  double w = 0.0;
  ConsSums cs{0.0, 0.0, 0.0};  // courant_fine's sums over the leaves (partials set)
  const double vol = dx * dx * dx;
  for_level_cells(active, noct, [&](int g, int ind) {
    const long c = cell_of(t, ind, g);
    const int s = t.son[c];
    double q[5];
#pragma unroll
    for (int v = 0; v < 5; ++v) q[v] = u[(long)v * ustride + c];
#pragma unroll
    for (int v = 0; v < 5; ++v) unew[(long)v * ustride + c] = q[v];
    if (s == 0) {
      w = fmax_f(w, cmpdt_w(q[0], q[1], q[2], q[3], q[4], hp));
      if (partials) cons_add(cs, q[0], q[1], q[2], q[3], q[4], vol, hp.smallr);
    }
  });
  if (partials) {
    __shared__ double cred[3 * (kBeginThreads / 64)];
    cons_block_store(cs, partials, blockIdx.x, cred);
  }
  const unsigned working = min((unsigned)((noct + kBeginThreads / 8 - 1) / (kBeginThreads / 8)), gridDim.x);
  if (blockIdx.x >= working) return;
  w = block_max(w);
  if (threadIdx.x != 0) return;
  // The count depends on what the maximum returned, so it cannot be seen
  // before the maximum; a fence in its place would write back and drop the
  // XCD's whole L2 for every workgroup (0.13 ms of a level of 10^5 octs).
  unsigned dep = (unsigned)atomicMax(d.wmax, w > 0.0 ? dt_bits(w) : 0ULL);
  asm volatile("v_and_b32 %0, 0, %0" : "+v"(dep));
  if (atomicAdd(d.done, 1u + dep) != working - 1) return;
  const double wm = __longlong_as_double((long long)atomicExch(d.wmax, 0ULL));
  *d.done = 0;
  const int l = d.l;
  double v = d.start;
  if (d.nsub_coarser > 0) v = fmin_f(d.dt[l - 1] / (double)d.nsub_coarser, v);
  if (wm > 0.0) v = fmin_f(v, cmpdt_from_w(wm, dx, hp));
  d.dtold[l] = d.dt[l];
  d.dt[l] = v;
  if (d.cnt) d.cnt[1] += 8LL * noct;
  if (d.has_finer && (dn ? dn[1] > 0 : d.finer_octs > 0)) return;
  if (d.has_finer) {
    d.dtold[l + 1] = v / (double)d.nsub;
    d.dt[l + 1] = v / (double)d.nsub;
  }
  d.time[0] = d.time[0] + v;
  if (d.cnt) d.cnt[0] += 1;
}

// update_time's conservation baselines (amr/update_time.f90:229-246) at
// the first update_time of a coarse step: mass_tot_0 = mass_tot and einit =
// epot_tot + ekin_tot (epot_tot = 0 without gravity), each only while still
// zero.  mass_tot and ekin_tot are then the courant_fine sums of the levels
// the step's first descent has visited (amr/amr_step.f90:327-352): levelmin
// down to the first level with no finer octs, each level's sum added as one
// term (hydro/courant_fine.f90:152-153).  A level's sum runs in the
// reference's serial order -- batches of nvector grids, cell position ind,
// grid in the batch (:44-102) -- so the values have its rounding.  The
// workgroup gathers chunks of kConsChunk terms of that order into LDS, many
// threads loading in parallel, so the tree walks and loads of a chunk
// overlap.  Threads 0 and 64 add a chunk's mass and energy terms in order
// while the wavefronts after the first two gather the next chunk into the
// second buffer.  A cell
// that is not a leaf adds +0.0, which leaves the positive running sum
// unchanged.  With dn the level counts are read from device memory and
// `armed` (nonzero: nstep_coarse changed since the last update_time)
// decides at run time.
constexpr int kConsChunk = 2048;
constexpr int kConsThreads = 1024;


// Terms [q0, q0 + kConsChunk) of a level's serial order into tp (mass,
// energy), loaded by threads [first, kConsThreads); past the level's end,
// zeros.
__device__ __forceinline__ void cons_gather(const int* active, int n, int nv, AmrTreeView t, const double* u,
                                            long ustride, double vol, long q0, int first, double2* tp) {
  // term q: batch b0 = q / (8 nv) * nv (only the last batch is short, so
  // 8 b0 terms precede it), then slot s = q - 8 b0 = (ind - 1) * ng + grid
  const long nterm = 8L * n;
  for (int k = (int)threadIdx.x - first; k < kConsChunk; k += kConsThreads - first) {
    double vm = 0.0, ve = 0.0;
    if (q0 + k < nterm) {
      const int q = (int)(q0 + k);  // 8 n <= 8 ngridmax fits the reference's 32-bit cell indices
      const int b0 = q / (8 * nv) * nv;
      const int ng = min(nv, n - b0);
      const int sl = q - 8 * b0;
      const long c = cell_of(t, sl / ng + 1, active[b0 + sl % ng]);
      if (t.son[c] == 0) {
        vm = u[c] * vol;                 // hydro/courant_fine.f90:95-97
        ve = u[4 * ustride + c] * vol;   // :100-102
      }
    }
    tp[k] = make_double2(vm, ve);
  }
}

// Adds component `which` (0: mass, 1: energy) of the first cnt terms of tp
// to acc, in order, by one thread.  The LDS loads run ahead of the chain of
// additions.  Mass and energy are summed by threads of two different
// wavefronts: an FP64 addition occupies its SIMD for 8 cycles whatever the
// number of active lanes, so the two chains in one wavefront shared one
// SIMD (2.5 ms for the adaptive Sedov run's baselines, 2.0 ms split).
__device__ __forceinline__ void cons_add(const double2* tp, int cnt, int which, double& acc) {
  int k0 = 0;
  for (; k0 + 16 <= cnt; k0 += 16) {
    double v[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = which == 0 ? tp[k0 + j].x : tp[k0 + j].y;
#pragma unroll
    for (int j = 0; j < 16; ++j) acc = acc + v[j];
  }
  for (; k0 < cnt; ++k0) acc = acc + (which == 0 ? tp[k0].x : tp[k0].y);
}

__global__ __launch_bounds__(kConsThreads) void amr_cons0_kernel(ConsLevels lv, const int* dn, AmrTreeView t,
                                                                const double* u, long ustride, int levelmin,
                                                                int nlevelmax, double boxlen, int nv, const int* armed,
                                                                double* cons0) {
  __shared__ double2 tp[2][kConsChunk];  // double-buffered chunks of (mass, energy) terms
  if (armed && *armed == 0) return;
  if (cons0[0] != 0.0 && cons0[1] != 0.0) return;
  const bool adder_waves = threadIdx.x < 128;
  const int which = threadIdx.x == 0 ? 0 : 1;  // thread 0 sums the mass, thread 64 the energy
  double tot = 0.0;                            // threads 0 and 64: mass_tot, ekin_tot
  for (int l = levelmin; l <= nlevelmax; ++l) {
    const int n = dn ? dn[l] : lv.noct[l];
    if (n <= 0) break;
    const int* active = lv.active[l];
    const double dx = __builtin_ldexp(1.0, -l) * boxlen;
    const double vol = dx * dx * dx;
    const long nterm = 8L * n;
    const long nchunk = (nterm + kConsChunk - 1) / kConsChunk;
    double acc = 0.0;
    cons_gather(active, n, nv, t, u, ustride, vol, 0, 0, tp[0]);
    __syncthreads();
    // threads 0 and 64 add chunk c while the wavefronts after the first two
    // gather c + 1
    for (long c = 0; c < nchunk; ++c) {
      const int b = (int)(c & 1);
      if (threadIdx.x == 0 || threadIdx.x == 64)
        cons_add(tp[b], (int)min((long)kConsChunk, nterm - c * kConsChunk), which, acc);
      else if (!adder_waves && c + 1 < nchunk)
        cons_gather(active, n, nv, t, u, ustride, vol, (c + 1) * kConsChunk, 128, tp[b ^ 1]);
      __syncthreads();
    }
    tot = tot + acc;
    if (l == nlevelmax || (dn ? dn[l + 1] : lv.noct[l + 1]) == 0) break;
  }
  if (threadIdx.x == 0 && cons0[1] == 0.0) cons0[1] = tot;        // mass_tot_0
  if (threadIdx.x == 64 && cons0[0] == 0.0) cons0[0] = 0.0 + tot;  // einit = epot_tot + ekin_tot
}

__global__ void clear_bits(int* p, int mask) { p[0] &= ~mask; }

__global__ void set_ints(int* p, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

// Grid of a launch over the cells of noct octs (for_level_cells): sized to a
// host count, a fixed persistent grid for a count read from device memory.
inline unsigned cell_grid(int noct, const int* dn) {
  return dn ? persist_blocks() : (unsigned)((noct + 31) / 32);
}

// Workgroups of a level's reflux, 0 without a coarser level.
static unsigned reflux_grid(const AmrLevelArgs& a) {
  if (!a.active_coarse || (!a.dnoct_coarse && a.noct_coarse <= 0)) return 0;
  if (a.dnoct) return persist_blocks();
  const unsigned nf = (unsigned)a.noct, nc = (unsigned)a.noct_coarse;
  const long per = reflux_from_coarse(nf, nc) ? 8L * nc : 6L * nf;
  return (unsigned)(((per < (long)kRefluxSplit ? 5 * per : per) + 255) / 256);
}

// gather + unsplit + update of one level (godunov_fine without its reflux);
// dt is read from d_dt.  With a.dnoct / a.dnoct_coarse the counts are read
// from device memory and the grids are persistent (batch loops), so the
// launches can be captured.
hipError_t launch_amr_sweep(const AmrLevelArgs& a, double dx, const double* d_dt, double* tmp, bool fp32,
                              hipStream_t s) {
  const bool dev = a.dnoct != nullptr;
  if (!dev && a.noct <= 0) return hipSuccess;
  hipError_t e;
  if (a.hp.slope_type != 3 && a.interpol_var == 0) {
    const unsigned grid = dev ? persist_blocks() : (unsigned)((a.noct + oct_tile::kOcts - 1) / oct_tile::kOcts);
    with_solver(a.hp.riemann, [&](auto rs) {
      if (fp32)
        launch_tile<float, decltype(rs)::value>(a, dx, d_dt, grid, s);
      else
        launch_tile<double, decltype(rs)::value>(a, dx, d_dt, grid, s);
    });
    if ((e = hipGetLastError()) != hipSuccess) return e;
  } else {
    const int nbatch = (a.noct + a.nv - 1) / a.nv;
    const unsigned gblocks = (unsigned)(((long)nbatch * 27 * a.nv + 255) / 256);
    hipLaunchKernelGGL(amr_gather, dim3(dev ? persist_blocks() : gblocks), dim3(256), 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    UnsplitArgs u;
    u.uin = a.uin;
    u.grav = nullptr;
    u.flux = a.flux;
    u.tmp = tmp;
    u.dx[0] = u.dx[1] = u.dx[2] = dx;
    u.dt = 0.0;
    u.d_dt = d_dt;
    u.ngroups = nbatch;
    u.ngrid_last = a.noct - (nbatch - 1) * a.nv;
    u.nv = a.nv;
    u.hp = a.hp;
    u.ok = a.ok;
    u.face_octs = amr_face_octs();
    const unsigned block = 128;
    const long tasks = (long)nbatch * (a.noct <= u.face_octs ? 36 : 12) * a.nv;
    // the fixed grids of the captured mode keep the 384 x persist_blocks()
    // threads of one batch per 384-thread workgroup
    const unsigned grid = dev ? 3 * persist_blocks() : (unsigned)((tasks + block - 1) / block);
    with_solver(a.hp.riemann, [&](auto rs) {
      if (fp32)
        launch_solve<float, decltype(rs)::value>(a, u, grid, block, s);
      else
        launch_solve<double, decltype(rs)::value>(a, u, grid, block, s);
    });
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const unsigned ugrid = dev ? 2 * persist_blocks() : (unsigned)(((long)nbatch * 40 * a.nv + 255) / 256);
    hipLaunchKernelGGL(amr_update, dim3(ugrid), dim3(256), 0, s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  return hipGetLastError();
}

hipError_t launch_amr_reflux(const AmrLevelArgs& a, hipStream_t s) {
  const unsigned grid = reflux_grid(a);
  if (grid == 0 || (!a.dnoct && a.noct <= 0)) return hipSuccess;
  hipLaunchKernelGGL(amr_reflux, dim3(grid), dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_amr_copy(const int* active, int noct, const AmrTreeView& t, const double* src, double* dst,
                           long ustride, hipStream_t s, const int* dn) {
  if (!dn && noct <= 0) return hipSuccess;
  hipLaunchKernelGGL(amr_copy_level, dim3(cell_grid(noct, dn)), dim3(256), 0, s, active, noct, dn, t, src, dst,
                     ustride);
  return hipGetLastError();
}

hipError_t launch_amr_upload(const int* active, int noct, const AmrTreeView& t, double* u, long ustride,
                             double smallr, int ivar_mode, hipStream_t s, const int* dn, int* flag1) {
  if (!dn && noct <= 0) return hipSuccess;
  hipLaunchKernelGGL(amr_upload, dim3(cell_grid(noct, dn)), dim3(256), 0, s, active, noct, dn, t, u, ustride,
                     smallr, ivar_mode, flag1);
  return hipGetLastError();
}

hipError_t launch_amr_courant(const int* active, int noct, const AmrTreeView& t, const double* u, long ustride,
                              double dx, const HydroParams& hp, double* d_dt, hipStream_t s, const int* dn) {
  if (!dn && noct <= 0) return hipSuccess;
  hipLaunchKernelGGL(amr_courant, dim3(cell_grid(noct, dn)), dim3(256), 0, s, active, noct, dn, t, u, ustride,
                     dx, hp, d_dt);
  return hipGetLastError();
}

static unsigned begin_grid(int noct, bool persistent) {
  const unsigned nb = (unsigned)((noct + kBeginThreads / 8 - 1) / (kBeginThreads / 8));
  return persistent || nb > 256 ? 256 : nb;
}

// With partials (amr_begin_partials_bytes) the level's conservation sums are
// added into sums[0..2] after the pass.
hipError_t launch_amr_begin(const int* active, int noct, const AmrTreeView& t, const double* u, double* unew,
                            long ustride, double dx, const HydroParams& hp, const AmrStepDt& d, hipStream_t s,
                            const int* dn, double* partials, double* sums) {
  if (!dn && noct <= 0) return hipSuccess;
  const unsigned nb = begin_grid(noct, dn != nullptr);
  hipLaunchKernelGGL(amr_begin, dim3(nb), dim3(kBeginThreads), 0, s, active, noct, dn, t, u, unew, ustride, dx, hp, d, partials);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !partials) return e;
  return launch_cons_finish(partials, nb, sums, 1, s);
}

size_t amr_begin_partials_bytes(int noct, bool persistent) {
  const size_t nb = begin_grid(noct, persistent);
  return (nb > 0 ? nb : 1) * 3 * sizeof(double);
}

// set_uold, upload_fine, the reflux into the coarser level and the end of the
// level step's time bookkeeping, in one launch.
hipError_t launch_amr_finish(const AmrLevelArgs& a, double* u, double* dt, const double* dtold, int nsub_coarser,
                             int icount, hipStream_t s) {
  if (!a.dnoct && a.noct <= 0) return hipSuccess;
  const unsigned refluxers = reflux_grid(a);
  hipLaunchKernelGGL(amr_finish, dim3(refluxers + cell_grid(a.noct, a.dnoct)), dim3(256), 0, s, a, u, a.interpol_var, dt,
                     dtold, nsub_coarser, icount, (int)refluxers);
  return hipGetLastError();
}

hipError_t launch_amr_cons0(const ConsLevels& lv, const int* dn, const AmrTreeView& t, const double* u, long ustride,
                            int levelmin, int nlevelmax, double boxlen, int nv, const int* armed, double* cons0,
                            hipStream_t s) {
  hipLaunchKernelGGL(amr_cons0_kernel, dim3(1), dim3(kConsThreads), 0, s, lv, dn, t, u, ustride, levelmin, nlevelmax,
                     boxlen, nv, armed, cons0);
  return hipGetLastError();
}

hipError_t launch_clear_bits(int* p, int mask, hipStream_t s) {
  hipLaunchKernelGGL(clear_bits, dim3(1), dim3(1), 0, s, p, mask);
  return hipGetLastError();
}

hipError_t launch_set_ints(int* p, int n, int v, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(set_ints, dim3((n + 255) / 256), dim3(256), 0, s, p, n, v);
  return hipGetLastError();
}

}  // namespace ramses
