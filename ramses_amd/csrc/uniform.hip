// Resident uniform periodic level: the godunov_fine -> godfine1 sweep
// (hydro/godunov_fine.f90:5-35, 486-911) with set_unew/set_uold replaced by
// ping-pong buffers, and the courant_fine dt reduction
// (hydro/courant_fine.f90:1-159) fused into the update epilogue.
//
// State: u[var][z][y][x], n^3 doubles per variable (SoA, x fastest).
//
// Kernel structure (2.5D blocking).  A workgroup owns an interior tile of
// TX x TY columns and marches along z through a chunk of TZ planes.  Its
// threads cover the tile and the ring of cells next to its four sides (the
// corners excluded), so the traced states of the halo cells that face the
// tile are computed by a thread like any other.  Per plane:
//   1. each thread computes slopes and traced states of its own cell from
//      its column (registers) and its x/y neighbours (LDS), and leaves the
//      left states in LDS,
//   2. the z face below the cell is solved from the previous plane's traced
//      state kept in registers; with the x/y fluxes of that plane (LDS) it
//      completes the plane below, whose new state is written and its cmpdt
//      limit min-reduced (wavefront shuffles, then LDS across waves, then one
//      64-bit atomic min on the bit pattern of the positive double),
//   3. x/y faces are solved from the exchanged left states, their fluxes and
//      the next plane's primitives (own cell and the tile's surroundings)
//      left in LDS.
// Two barriers a plane part these (the fluxes have LDS of their own, which
// still lets three FP64 or four FP32-mixed workgroups share a CU); with the
// primitives of two planes and one area for states and fluxes there were
// five in FP64 and seven in FP32-mixed.
//
// What bounds it: vector issue (75% of the cycles, at the 2.0 GHz that this
// load leaves of 2.4).  At 256^3 a pass takes 816 us in FP64 and 520 us in
// FP32-mixed (918 and 578 with five and seven barriers, energies of both
// sides of a face and two roots a face), at 512^3 6.4 ms.  Four FP64 waves a
// SIMD (128 VGPRs, one LDS area more shared and a third barrier) ran 3%
// slower.
// Each primitive is computed by one ctoprim per cell per workgroup, each
// face flux once, and every value keeps the reference's operation order, so
// the FP64 path reproduces godfine1+unsplit on a uniform grid bit for bit.
#include <type_traits>

#include "hydro_device.hpp"

namespace ramses {

namespace {

struct UniformArgs {
  const double* u;
  double* unew;
  const double* d_dt;     // time step (device)
  double* d_dt_next;      // fused courant output or null
  double* partials;       // courant_fine sums per workgroup (3 doubles each) or null
  int n;
  double dx;
  HydroParams hp;
};

// Slot state layout (device doubles, see ramses_level_slot in the header).
enum SlotField : int { kTime = 0, kTend = 1, kDtUse = 2, kDtNext = 3, kDone = 4, kSteps = 5, kParity = 6, kStepped = 7 };

constexpr int kMaxSlots = 32;

struct BatchSlot {
  double* buf[2];
  double* state;
  int n;
  int tz;
  double dx;
};

struct BatchArgs {
  BatchSlot slot[kMaxSlots];
  int blk0[kMaxSlots + 1];
  int nslots;
  HydroParams hp;
};

__device__ __forceinline__ int wrapi(int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); }

// Threads of a TX x TY tile: one per interior cell plus one per halo cell
// whose traced state a tile face needs (the 2*(TX+TY) non-corner cells of
// the one-cell ring), rounded up to whole wavefronts.
template <int TX, int TY>
constexpr int tile_threads() { return (TX * TY + 2 * (TX + TY) + 63) / 64 * 64; }

// One workgroup's tile of a level: columns [x0, x0+TX) x [y0, y0+TY),
// planes [z0, z0+TZ).  Shared by the single-level and the batched kernels.
// A tile may reach past the level's last column or row (n >= TX, TY): the
// periodic wrap makes the threads there repeat cells of the other side, and
// they store nothing.  ST: the slope type fixed at compile time, or -1 (see
// slope1).
template <typename R, int TX, int TY, int RS, bool SUMS = false, int ST = -1>
__device__ __forceinline__ void level_tile(const double* __restrict__ u, double* __restrict__ unew, int n, double dx,
                                           double dt, double* d_dt_next, const HydroParams& hp, int x0, int y0,
                                           int z0, int TZ, double* partials = nullptr, long block = 0) {
  constexpr int EX = TX + 2, EY = TY + 2;      // tile with its one-cell ring
  constexpr int QX = TX + 4, QY = TY + 4;      // primitive plane with 2-cell halo
  constexpr int NQ = QX * QY;
  constexpr int NE = EX * EY;
  constexpr int NI = TX * TY;
  constexpr int NT = tile_threads<TX, TY>();
  static_assert(NI % 64 == 0, "interior cells fill whole wavefronts");

  __shared__ R qs[5][NQ];                   // primitives of the plane whose states are traced
  __shared__ __align__(16) R qm[10][NE];    // its traced left states: x, then y
  __shared__ __align__(16) double fl[10][NE];  // fluxes (scaled): x, then y
  __shared__ double red[NT / 64];

  const long plane = (long)n * n;
  const long vstride = plane * n;
  const int t = threadIdx.x;
  // Threads [0, NI) own the interior cells, x fastest.  Threads [NI, NI +
  // 2*(TX+TY)) own the ring cells a tile face needs: the left column (its
  // qm_x), the right column (its qp_x and the face x = TX+1/2), the bottom
  // row (qm_y) and the top row (qp_y and the face y = TY+1/2).  Corner cells
  // feed no face and get no thread.  Since NI is a multiple of 64, the ring
  // cells fill waves of their own, which skip the z face, the update and the
  // courant epilogue.
  // (ex, ey) are coordinates in the tile with its ring, interior 1..TX, 1..TY.
  enum { kNone = -1, kInterior = 0, kLeft, kRight, kBottom, kTop };
  int ex = 1, ey = 1, kind = kNone;
  if (t < NI) {
    ex = 1 + t % TX;
    ey = 1 + t / TX;
    kind = kInterior;
  } else if (t < NI + 2 * (TX + TY)) {
    int h = t - NI;
    if (h < 2 * TY) {
      ex = h < TY ? 0 : TX + 1;
      ey = 1 + h % TY;
      kind = h < TY ? kLeft : kRight;
    } else {
      h -= 2 * TY;
      ex = 1 + h % TX;
      ey = h < TX ? 0 : TY + 1;
      kind = h < TX ? kBottom : kTop;
    }
  }
  const int e = ey * EX + ex;  // own slot in the exchange areas
  const int qo = (ey + 1) * QX + (ex + 1);  // own cell in the primitive plane
  const bool inside = x0 + ex <= n && y0 + ey <= n;  // (interior threads) the cell is not a repeated one

  // The ring's waves also convert the cells around the ring that its slopes
  // read: a column or row outside each side and the ring's four corners.
  constexpr int kOuter = 2 * (TX + TY) + 4;
  static_assert(kOuter <= NT - NI, "one outer cell per thread of the ring's waves");
  int ox = 1, oy = 1;
  const bool outer = t >= NI && t < NI + kOuter;
  if (outer) {
    int h = t - NI;
    if (h < 2 * TY) {
      ox = h < TY ? -1 : TX + 2;
      oy = 1 + h % TY;
    } else if (h < 2 * (TX + TY)) {
      h -= 2 * TY;
      ox = 1 + h % TX;
      oy = h < TX ? -1 : TY + 2;
    } else {
      h -= 2 * (TX + TY);
      ox = h % 2 ? TX + 1 : 0;
      oy = h / 2 ? TY + 1 : 0;
    }
  }
  const int qx = (oy + 1) * QX + (ox + 1);

  // A plane of one variable is addressed from a scalar base by a 32-bit byte
  // offset that a thread keeps for the whole march (its own cell, and the
  // outer cell it converts), so that a load or store takes no vector
  // instruction for its address.
  auto at = [&](const double* base, unsigned off) {
    return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(base) + off);
  };
  auto offset = [&](int cx, int cy) { return 8u * (unsigned)(wrapi(y0 - 1 + cy, n) * n + wrapi(x0 - 1 + cx, n)); };
  const unsigned own = offset(ex, ey), own2 = offset(ox, oy);

  const SolverConsts<R> sc = scalar(make_consts<R>(hp));
  const double dtxhalf = scalar(dt * 0.5);
  const double smalle = scalar(hp.smallc * hp.smallc / hp.gamma / (hp.gamma - 1.0));
  const R dtdx = scalar((R)(dt / dx));
  const FluxScale fs = scalar(make_scale(dt, dx));

  struct Raw {
    double v[5];
  };
  // keeps the compiler from forming 64-bit vector addresses ahead of the march
  auto fixed = [](unsigned off) {
    asm("" : "+v"(off));
    return off;
  };
  auto load = [&](int zp, unsigned off) {
    const double* up = u + (long)wrapi(zp, n) * plane;
    Raw r;
#pragma unroll
    for (int v = 0; v < 5; ++v) r.v[v] = at(up + v * vstride, fixed(off));
    return r;
  };
  auto prim = [&](const Raw& r) {
    return ctoprim_cell<R>(r.v[0], r.v[1], r.v[2], r.v[3], r.v[4], 0.0, 0.0, 0.0, dtxhalf, smalle, hp);
  };
  auto put_q = [&](const Prim<R>& q, int c) {
    qs[0][c] = q.r;
    qs[1][c] = q.u;
    qs[2][c] = q.v;
    qs[3][c] = q.w;
    qs[4][c] = q.p;
  };
  auto read_q = [&](int c) { return Prim<R>{qs[0][c], qs[1][c], qs[2][c], qs[3][c], qs[4][c]}; };
  auto put_qm = [&](const Prim<R>& q, int row) {
    qm[row][e] = q.r;
    qm[row + 1][e] = q.u;
    qm[row + 2][e] = q.v;
    qm[row + 3][e] = q.w;
    qm[row + 4][e] = q.p;
  };
  auto read_qm = [&](int row, int c) {
    return Prim<R>{qm[row][c], qm[row + 1][c], qm[row + 2][c], qm[row + 3][c], qm[row + 4][c]};
  };

  // own-column primitives at p-1 and p; for minmod their difference in place
  // of those at p-1 (every difference along z serves two planes)
  Prim<R> qprev = prim(load(z0 - 2, own)), qcur = prim(load(z0 - 1, own));
  if constexpr (ST == 1) qprev = qcur - qprev;
  // values carried from the previous plane
  Face<R> fz_left{};          // rotated qm_z of plane p-1
  double fz_prev[5] = {0, 0, 0, 0, 0};  // flux through the z face below plane p-1 (scaled)
  double wmax = 0.0;  // largest cmpdt wave speed of the new state
  ConsSums cs{0.0, 0.0, 0.0};  // courant_fine's sums of the new state (SUMS)
  const double vol = dx * dx * dx;

  // The march over the planes z0-1 .. z0+TZ.  kWaves: 0 for a wave of
  // interior cells, 1 for the ring's waves; the cell kinds of a wave are then
  // known at compile time (the cells of a wave are all interior or all ring,
  // NI being a multiple of 64).  A plane takes two barriers:
  //   A: the primitives of plane p and the x and y fluxes of plane p-1 are
  //      there.  Trace plane p, leave the left states; solve the z face
  //      between p-1 and p and finish plane p-1.
  //   B: the left states of plane p are there, and every reader of the
  //      primitives and of the fluxes of p-1 is done.  Solve the x and y
  //      faces of plane p, leave their fluxes and the primitives of p+1.
  auto march = [&](auto waves_tag) {
    constexpr bool interior = decltype(waves_tag)::value == 0;
    // FP32-mixed has the registers to keep the own column's conserved state
    // for its update two planes later (541 us at 256^3, 590 with it loaded
    // again); in FP64 it is loaded again, and where the solvers that are not
    // fixed at compile time spill with it: with minmod (acoustic, 288^3: 897
    // us, 960 with it kept) and with sums
    constexpr bool kKeep = interior && sizeof(R) == 4 && !(RS == kDynamicRiemann && (ST == 1 || SUMS));
    const bool ring = kind > kInterior;
    const bool xdir = kind == kLeft || kind == kRight;
    if (interior || ring) put_q(qcur, qo);
    if (!interior && outer) put_q(prim(load(z0 - 1, own2)), qx);
    Raw next = load(z0, own);
    Raw u0{}, uc{};
    for (int p = z0 - 1;; ++p) {
      const bool faces_xy = p >= z0 && p < z0 + TZ;
      __syncthreads();  // A
      const Prim<R> qnext = prim(next);
      const Raw u1 = u0;  // conserved state of plane p-1 (kKeep)
      if constexpr (kKeep) {
        u0 = uc;
        uc = next;
      }
      Prim<R> qp_x{}, qp_y{};
      {
        const Prim<R> xm = read_q(qo - 1), xp = read_q(qo + 1);
        const Prim<R> ym = read_q(qo - QX), yp = read_q(qo + QX);
        const Prim<R> dqx = slope_prim<R, ST>(xm, qcur, xp, sc.slope_type, sc.theta);
        const Prim<R> dqy = slope_prim<R, ST>(ym, qcur, yp, sc.slope_type, sc.theta);
        Prim<R> dqz;
        if constexpr (ST == 1) {
          const Prim<R> drgt = qnext - qcur;
          dqz = minmod(qprev, drgt);
          qprev = drgt;
        } else {
          dqz = slope_prim<R, ST>(qprev, qcur, qnext, sc.slope_type, sc.theta);
          qprev = qcur;
        }
        const Source<R> src = trace_sources<R, ST>(qcur, dqx, dqy, dqz, sc.gamma, sc.div_hi);
        if constexpr (interior) {
          Prim<R> q_x, q_y, qp_z, qm_z;
          trace_dir(qcur, dqx, src, dtdx, sc.smallr, qp_x, q_x);
          trace_dir(qcur, dqy, src, dtdx, sc.smallr, qp_y, q_y);
          trace_dir(qcur, dqz, src, dtdx, sc.smallr, qp_z, qm_z);
          if (faces_xy) {
            put_qm(q_x, 0);
            put_qm(q_y, 5);
          }
          // z face below plane p (between p-1 and p)
          double fz[5] = {0, 0, 0, 0, 0};
          if (p >= z0) {
            const Flux6<R> g = riemann_fixed<R, RS>(fz_left, rotate(qp_z, 2), sc);
            R fc[5];
            unrotate(g, 2, fc);
            scale_flux<5>(fc, fs, fz);  // hydro/umuscl.f90:153
          }
          // plane p-1 is complete: hydro/godunov_fine.f90:751-792 in idim
          // order, unew = ((uold + dFx) + dFy) + dFz
          if (p >= z0 + 1) {
            const Raw old = kKeep ? u1 : load(p - 1, own);
            double un[5];
#pragma unroll
            for (int v = 0; v < 5; ++v) {
              const double ux = old.v[v] + (fl[v][e] - fl[v][e + 1]);
              const double uy = ux + (fl[5 + v][e] - fl[5 + v][e + EX]);
              un[v] = uy + (fz_prev[v] - fz[v]);
            }
            if (inside) {
              double* np = unew + (long)(p - 1) * plane;
#pragma unroll
              for (int v = 0; v < 5; ++v)
                *reinterpret_cast<double*>(reinterpret_cast<char*>(np + v * vstride) + fixed(own)) = un[v];
            }
            if (d_dt_next) {
              if constexpr (sizeof(R) == 8) wmax = fmax_f(wmax, cmpdt_w(un[0], un[1], un[2], un[3], un[4], hp, sc.smallp));
              else wmax = fmax_f(wmax, cmpdt_w_fast(un[0], un[1], un[2], un[3], un[4], hp));
            }
            if (SUMS && inside) cons_add(cs, un[0], un[1], un[2], un[3], un[4], vol, hp.smallr);
          }
          fz_left = rotate(qm_z, 2);
#pragma unroll
          for (int v = 0; v < 5; ++v) fz_prev[v] = fz[v];
        } else {
          // a left or right ring cell feeds only an x face, a bottom or top
          // one only a y face, and none a z face
          Prim<R> q;
          trace_dir(qcur, xdir ? dqx : dqy, src, dtdx, sc.smallr, qp_x, q);
          if (ring && faces_xy) put_qm(q, xdir ? 0 : 5);
        }
      }
      qcur = qnext;
      if (p == z0 + TZ) break;
      __syncthreads();  // B
      if (faces_xy) {
        if constexpr (interior) {
          R fc[5];
          double f[5];
          unrotate(riemann_fixed<R, RS>(rotate(read_qm(0, e - 1), 0), rotate(qp_x, 0), sc), 0, fc);  // x-1/2
          scale_flux<5>(fc, fs, f);  // hydro/umuscl.f90:106
#pragma unroll
          for (int v = 0; v < 5; ++v) fl[v][e] = f[v];
          unrotate(riemann_fixed<R, RS>(rotate(read_qm(5, e - EX), 1), rotate(qp_y, 1), sc), 1, fc);  // y-1/2
          scale_flux<5>(fc, fs, f);  // :129
#pragma unroll
          for (int v = 0; v < 5; ++v) fl[5 + v][e] = f[v];
        } else if (kind == kRight || kind == kTop) {
          // the right column's x faces and the top row's y faces in one pass
          const Prim<R> l = read_qm(xdir ? 0 : 5, xdir ? e - 1 : e - EX);
          auto face = [&](const Prim<R>& q) {
            const Face<R> fx = rotate(q, 0), fy = rotate(q, 1);
            return xdir ? fx : fy;
          };
          const Flux6<R> g = riemann_fixed<R, RS>(face(l), face(qp_x), sc);
          R fcx[5], fcy[5], fc[5];
          double f[5];
          unrotate(g, 0, fcx);
          unrotate(g, 1, fcy);
#pragma unroll
          for (int v = 0; v < 5; ++v) fc[v] = xdir ? fcx[v] : fcy[v];
          scale_flux<5>(fc, fs, f);
#pragma unroll
          for (int v = 0; v < 5; ++v) fl[(xdir ? 0 : 5) + v][e] = f[v];
        }
      }
      next = load(p + 2, own);
      if (interior || ring) put_q(qcur, qo);
      if (!interior && outer) put_q(prim(load(p + 1, own2)), qx);
    }
  };
  // The interior waves and the ring's waves run copies of the march with
  // their cell kinds fixed, both meeting the same barriers in the same order
  // (at 512^3: FP64 5.5% faster, FP32-mixed 3.5% once held to 128 VGPRs).
  if (t >= NI) march(std::integral_constant<int, 1>{});
  else march(std::integral_constant<int, 0>{});

  if (d_dt_next) {
    // wavefront max of w with shuffles, then across the block's waves; the
    // block's dt limit is cmpdt_from_w(max w), min-combined across blocks
    for (int off = 32; off > 0; off >>= 1) wmax = fmax_f(wmax, __shfl_xor(wmax, off, 64));
    const int wave = t >> 6, lane = t & 63;
    if (lane == 0) red[wave] = wmax;
    __syncthreads();
    if (t == 0) {
      double m = red[0];
      for (int w = 1; w < NT / 64; ++w) m = fmax_f(m, red[w]);
      if (m > 0.0) atomicMin(reinterpret_cast<unsigned long long*>(d_dt_next), dt_bits(cmpdt_from_w(m, dx, hp)));
    }
  }
  if constexpr (SUMS) {
    __shared__ double cred[3 * (NT / 64)];
    cons_block_store(cs, partials, block, cred);
  }
}


template <typename R, int TX, int TY, int RS, bool SUMS, int ST>
// The register budget: 3 waves per SIMD in FP64 (162 VGPRs), 4 in FP32-mixed
// (at most 128).
__global__ __launch_bounds__((tile_threads<TX, TY>()))
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 3, 8))) void uniform_godunov_kernel(UniformArgs a, int ntx,
                                                                                           int nty, int TZ) {
  // Workgroup b runs on XCD b % 8 (the hardware deals them out in turn).
  // Giving each XCD a contiguous range of tiles (x fastest, then y, then z
  // chunk; xcd_contiguous) keeps the tiles that run side by side on one XCD
  // spatial neighbours, and their shared halo columns are served by that
  // XCD's L2 instead of HBM.  The last chunk may be shorter.
  const int logical = (int)xcd_contiguous(blockIdx.x, gridDim.x);
  const int tx = logical % ntx, ty = (logical / ntx) % nty, z0 = logical / (ntx * nty) * TZ;
  level_tile<R, TX, TY, RS, SUMS, ST>(a.u, a.unew, a.n, a.dx, *a.d_dt, a.d_dt_next, a.hp, tx * TX, ty * TY, z0,
                                     min(TZ, a.n - z0), a.partials, blockIdx.x);
}

// Many independent levels advanced by one launch (continuous batching).
// Workgroups [blk0[s], blk0[s+1]) belong to slot s; a slot whose state says
// `done` is skipped.  The slot's buffer parity selects input and output.
template <typename R, int TX, int TY, int RS, int ST>
__global__ __launch_bounds__((tile_threads<TX, TY>()))
__attribute__((amdgpu_waves_per_eu(sizeof(R) == 4 ? 4 : 3, 8))) void batch_godunov_kernel(BatchArgs a) {
  const int b = blockIdx.x;
  int s = 0;
  while (s + 1 < a.nslots && b >= a.blk0[s + 1]) ++s;
  const BatchSlot& sl = a.slot[s];
  double* st = sl.state;
  if (st[kDone] != 0.0) return;
  const int par = (int)st[kParity];
  const double* u = sl.buf[par];
  double* unew = sl.buf[par ^ 1];
  const int n = sl.n;
  const int ntx = (n + TX - 1) / TX, nty = (n + TY - 1) / TY;
  // neighbouring tiles of a slot on one XCD (see uniform_godunov_kernel)
  const int local = (int)xcd_contiguous(b - a.blk0[s], a.blk0[s + 1] - a.blk0[s]);
  const int tx = local % ntx, ty = (local / ntx) % nty, z0 = local / (ntx * nty) * sl.tz;
  level_tile<R, TX, TY, RS, false, ST>(u, unew, n, sl.dx, st[kDtUse], st + kDtNext, a.hp, tx * TX, ty * TY, z0,
                                      min(sl.tz, n - z0));
}

// Per-slot bookkeeping before each batched step (one thread per slot):
// finish the previous step (t += dt, flip the buffer parity), stop at t_end,
// and choose this step's dt = min(courant dt, t_end - t); then reset the
// fused courant accumulator to newdt_fine's start value
// (pm/newdt_fine.f90:51) capped by cmpdt's C*dx/smallc
// (hydro/godunov_utils.f90:114).  The end-time cap is this server's own
// contract (a request asks for the state at t_end) and has no counterpart in
// the reference: newdt_fine (pm/newdt_fine.f90:51-173) never looks at the
// output times, and amr_step writes an output once t >= tout
// (amr/amr_step.f90:151), after the step that crossed it.  Every other step
// uses the reference's courant dt unchanged.
__global__ void batch_advance_kernel(BatchArgs a) {
  const int s = threadIdx.x;
  if (s >= a.nslots) return;
  const BatchSlot& sl = a.slot[s];
  double* st = sl.state;
  if (st[kDone] != 0.0) return;
  if (st[kStepped] != 0.0) {
    st[kTime] = st[kTime] + st[kDtUse];
    st[kSteps] = st[kSteps] + 1.0;
    st[kParity] = 1.0 - st[kParity];
    st[kStepped] = 0.0;
  }
  if (st[kTime] >= st[kTend]) {
    st[kDone] = 1.0;
    return;
  }
  st[kDtUse] = fmin_f(st[kDtNext], st[kTend] - st[kTime]);
  const double boxlen = sl.n * sl.dx;
  st[kDtNext] = fmin_f(boxlen / a.hp.smallc, a.hp.courant_factor * sl.dx / a.hp.smallc);
  st[kStepped] = 1.0;
}

// courant_fine over a uniform level without gravity: max of the cmpdt wave
// speed per block, then the block's dt limit min-combined across blocks
// (exactly min over cells of cmpdt, see cmpdt_w).
__global__ void courant_kernel(const double* u, long ncell, double dx, HydroParams hp, double* d_dt,
                               double* partials) {
  double wmax = 0.0;
  ConsSums cs{0.0, 0.0, 0.0};
  const double vol = dx * dx * dx;
  for (long c = (long)blockIdx.x * blockDim.x + threadIdx.x; c < ncell; c += (long)gridDim.x * blockDim.x) {
    wmax = fmax_f(wmax, cmpdt_w(u[c], u[c + ncell], u[c + 2 * ncell], u[c + 3 * ncell], u[c + 4 * ncell], hp));
    if (partials) cons_add(cs, u[c], u[c + ncell], u[c + 2 * ncell], u[c + 3 * ncell], u[c + 4 * ncell], vol, hp.smallr);
  }
  if (partials) {
    __shared__ double cred[3 * 4];
    cons_block_store(cs, partials, blockIdx.x, cred);
  }
  for (int off = 32; off > 0; off >>= 1) wmax = fmax_f(wmax, __shfl_xor(wmax, off, 64));
  __shared__ double red[4];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) red[wave] = wmax;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = fmax_f(m, red[w]);
    if (m > 0.0) atomicMin(reinterpret_cast<unsigned long long*>(d_dt), dt_bits(cmpdt_from_w(m, dx, hp)));
  }
}

__global__ void set_double(double* p, double v) { *p = v; }

__global__ void set_doubles(double* p, int n, double v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// Sum of the per-workgroup conservation sums in block order: thread t adds
// blocks t, t+256, ... in order, then a fixed pairwise tree; out[0..2] is
// overwritten, or incremented when `accumulate` (courant_fine's
// mass_tot = mass_tot + mass_all, hydro/courant_fine.f90:152-154).
__global__ __launch_bounds__(256) void cons_finish(const double* partials, long nblocks, double* out,
                                                  int accumulate) {
  __shared__ double sh[3][256];
  const int t = threadIdx.x;
  double m = 0.0, e = 0.0, ei = 0.0;
  for (long b = t; b < nblocks; b += 256) {
    m = m + partials[3 * b];
    e = e + partials[3 * b + 1];
    ei = ei + partials[3 * b + 2];
  }
  sh[0][t] = m;
  sh[1][t] = e;
  sh[2][t] = ei;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (t < h) {
      sh[0][t] = sh[0][t] + sh[0][t + h];
      sh[1][t] = sh[1][t] + sh[1][t + h];
      sh[2][t] = sh[2][t] + sh[2][t + h];
    }
    __syncthreads();
  }
  if (t == 0) {
    for (int k = 0; k < 3; ++k) out[k] = accumulate ? out[k] + sh[k][0] : sh[k][0];
  }
}

__global__ void init_slot_kernel(double* st, double t_end, double start) {
  st[kTime] = 0.0;
  st[kTend] = t_end;
  st[kDtUse] = 0.0;
  st[kDtNext] = start;
  st[kDone] = 0.0;
  st[kSteps] = 0.0;
  st[kParity] = 0.0;
  st[kStepped] = 0.0;
}

__global__ void cmpdt_group(const double* uu, const double* gg, int nv, int ncell, double dx, HydroParams hp,
                            double* d_dt) {
  // hydro/godunov_utils.f90:114-118: dt = min(C*dx/smallc, min over cells)
  double dt = hp.courant_factor * dx / hp.smallc;
  for (int k = threadIdx.x; k < ncell; k += blockDim.x) {
    const double gx = gg ? gg[k] : 0.0, gy = gg ? gg[k + nv] : 0.0, gz = gg ? gg[k + 2 * nv] : 0.0;
    dt = fmin_f(dt, cmpdt_cell(uu[k], uu[k + nv], uu[k + 2 * nv], uu[k + 3 * nv], uu[k + 4 * nv], gx, gy, gz, dx, hp));
  }
  for (int off = 32; off > 0; off >>= 1) dt = fmin_f(dt, __shfl_xor(dt, off, 64));
  __shared__ double red[4];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = dt;
  __syncthreads();
  if (threadIdx.x == 0) {
    double m = red[0];
    for (int w = 1; w < (int)(blockDim.x >> 6); ++w) m = fmin_f(m, red[w]);
    *d_dt = m;
  }
}

template <typename R, int TX, int TY, bool SUMS, int ST>
void launch_tile_st(const UniformArgs& a, int ntx, int nty, int TZ, dim3 grid, hipStream_t s) {
  const dim3 block(tile_threads<TX, TY>());
  switch (a.hp.riemann) {
    case kHLLC:
      hipLaunchKernelGGL((uniform_godunov_kernel<R, TX, TY, kHLLC, SUMS, ST>), grid, block, 0, s, a, ntx, nty, TZ);
      break;
    case kHLL:
      hipLaunchKernelGGL((uniform_godunov_kernel<R, TX, TY, kHLL, SUMS, ST>), grid, block, 0, s, a, ntx, nty, TZ);
      break;
    case kACOUSTIC:
    case kEXACT:
      hipLaunchKernelGGL((uniform_godunov_kernel<R, TX, TY, kDynamicRiemann, SUMS, ST>), grid, block, 0, s, a, ntx, nty,
                         TZ);
      break;
    default:
      hipLaunchKernelGGL((uniform_godunov_kernel<R, TX, TY, kLLF, SUMS, ST>), grid, block, 0, s, a, ntx, nty, TZ);
      break;
  }
}

// Launch the level kernel; with sums, then add the workgroups' conservation
// sums into d_sums[0..2] in block order.  Minmod, the reference's default
// slope (hydro/hydro_parameters.f90:76), has kernels of its own with the
// limiter fixed at compile time; other slope types take it at run time.
template <typename R, int TX, int TY>
hipError_t launch_tile(const UniformArgs& a, int TZ, double* d_sums, hipStream_t s) {
  const int ntx = (a.n + TX - 1) / TX, nty = (a.n + TY - 1) / TY;
  const dim3 grid((unsigned)(ntx * nty * ((a.n + TZ - 1) / TZ)));
  const bool st1 = a.hp.slope_type == 1;
  if (a.partials) {
    st1 ? launch_tile_st<R, TX, TY, true, 1>(a, ntx, nty, TZ, grid, s)
        : launch_tile_st<R, TX, TY, true, -1>(a, ntx, nty, TZ, grid, s);
    hipLaunchKernelGGL(cons_finish, dim3(1), dim3(256), 0, s, (const double*)a.partials, (long)grid.x, d_sums, 0);
  } else {
    st1 ? launch_tile_st<R, TX, TY, false, 1>(a, ntx, nty, TZ, grid, s)
        : launch_tile_st<R, TX, TY, false, -1>(a, ntx, nty, TZ, grid, s);
  }
  return hipGetLastError();
}

// Time estimate of W workgroups of TZ planes on the 256 CUs, in us: m of
// them on the fullest CU, TZ + 2 planes each (two are marched for their
// traced states only).  A CU takes its m workgroups' planes side by side
// while they fit, then one after the other at full throughput.  The plane
// times are those measured with 16x12 tiles (hllc, minmod): one workgroup
// alone 3.4 us a plane in FP64 and 2.4 in FP32-mixed, three FP64 ones 6.6,
// four FP32-mixed ones 4.9.  The estimate is within 10% of the measured time
// for n = 16..256 and z chunks of 2..128 planes (larger levels: see
// launch_uniform_godunov).
inline double level_estimate(long W, int TZ, bool fp32) {
  const double m = (double)((W + 255) / 256);
  const double plane = fp32 ? (m <= 4 ? 1.5 + 0.85 * m : 1.4 * m) : (m <= 3 ? 1.75 + 1.65 * m : 2.2 * m);
  return (TZ + 2) * plane;
}

// The same for 32x16 tiles, of which a CU holds one: 6.2 us a plane in FP64,
// 3.6 in FP32-mixed.
inline double wide_estimate(long W, int TZ, bool fp32) { return (TZ + 2) * (fp32 ? 3.6 : 6.2) * (double)((W + 255) / 256); }

// The z chunk with the least estimate, at least 2 planes and at most
// max_blocks workgroups.  Long chunks repeat fewer planes, short ones fill
// the chip: 2 planes at n <= 64, 6 at 96, 16 at 128, 32 at 256 and 64 at 512
// in FP64 (with max_blocks out of the way), the fastest or within 3% of it
// among those measured.  No chunk is longer than `longest`.
inline int best_tz(int n, long tiles, bool fp32, long max_blocks, int longest,
                   double (*estimate)(long, int, bool) = level_estimate, double* time = nullptr) {
  const int last = longest < n ? longest : n;
  int best = last;
  double least = 1e300;
  for (int tz = n < 2 ? n : 2; tz <= last; ++tz) {
    const long W = tiles * ((n + tz - 1) / tz);
    if (W > max_blocks && tz < last) continue;
    const double t = estimate(W, tz, fp32);
    if (t < least) {
      least = t;
      best = tz;
    }
  }
  if (time) *time = least;
  return best;
}

constexpr int kBatchTX = 16, kBatchTY = 12;
inline long batch_tiles(int n) { return (long)((n + kBatchTX - 1) / kBatchTX) * ((n + kBatchTY - 1) / kBatchTY); }

template <typename R, int RS>
void launch_batch_t(const BatchArgs& a, int nblocks, hipStream_t s) {
  constexpr int TX = kBatchTX, TY = kBatchTY, NT = tile_threads<TX, TY>();
  if (a.hp.slope_type == 1)  // minmod: see launch_tile
    hipLaunchKernelGGL((batch_godunov_kernel<R, TX, TY, RS, 1>), dim3(nblocks), dim3(NT), 0, s, a);
  else
    hipLaunchKernelGGL((batch_godunov_kernel<R, TX, TY, RS, -1>), dim3(nblocks), dim3(NT), 0, s, a);
}

}  // namespace

// One z chunk for every slot of a batch: the least estimate for all their
// workgroups together (a slot that is done exits at once and is not known
// here).
static int batch_tz(const int* n, int nslots, bool fp32) {
  int best = 32;
  double least = 1e300;
  for (int tz : {2, 4, 6, 8, 12, 16, 24, 32}) {
    long W = 0;
    for (int i = 0; i < nslots; ++i) W += batch_tiles(n[i]) * ((n[i] + tz - 1) / tz);
    const double t = level_estimate(W, tz, fp32);
    if (t < least) {
      least = t;
      best = tz;
    }
  }
  return best;
}

// The workgroups of a batch at its shortest z chunk.
long level_batch_blocks(const int* n, int nslots) {
  long W = 0;
  for (int i = 0; i < nslots; ++i) W += batch_tiles(n[i]) * ((n[i] + 1) / 2);
  return W;
}

// Continuous batching: one bookkeeping launch and one update launch advance
// every slot of `slots` by one step of its own dt.
hipError_t launch_level_batch(double* const* buf0, double* const* buf1, double* const* state, const int* n,
                              const double* dx, int nslots, const HydroParams& hp, bool fp32, hipStream_t s) {
  BatchArgs a{};
  a.nslots = nslots;
  a.hp = hp;
  const int tz = batch_tz(n, nslots, fp32);
  int blocks = 0;
  for (int i = 0; i < nslots; ++i) {
    BatchSlot& sl = a.slot[i];
    sl.buf[0] = buf0[i];
    sl.buf[1] = buf1[i];
    sl.state = state[i];
    sl.n = n[i];
    sl.dx = dx[i];
    sl.tz = tz;
    a.blk0[i] = blocks;
    blocks += (int)(batch_tiles(n[i]) * ((n[i] + tz - 1) / tz));
  }
  a.blk0[nslots] = blocks;
  hipLaunchKernelGGL(batch_advance_kernel, dim3(1), dim3(64), 0, s, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || blocks == 0) return e;
  if (fp32) {
    if (hp.riemann == kHLLC) launch_batch_t<float, kHLLC>(a, blocks, s);
    else if (hp.riemann == kHLL) launch_batch_t<float, kHLL>(a, blocks, s);
    else if (hp.riemann == kACOUSTIC || hp.riemann == kEXACT) launch_batch_t<float, kDynamicRiemann>(a, blocks, s);
    else launch_batch_t<float, kLLF>(a, blocks, s);
  } else {
    if (hp.riemann == kHLLC) launch_batch_t<double, kHLLC>(a, blocks, s);
    else if (hp.riemann == kHLL) launch_batch_t<double, kHLL>(a, blocks, s);
    else if (hp.riemann == kACOUSTIC || hp.riemann == kEXACT) launch_batch_t<double, kDynamicRiemann>(a, blocks, s);
    else launch_batch_t<double, kLLF>(a, blocks, s);
  }
  return hipGetLastError();
}

hipError_t launch_init_slot(double* state, double t_end, double start, hipStream_t s) {
  hipLaunchKernelGGL(init_slot_kernel, dim3(1), dim3(1), 0, s, state, t_end, start);
  return hipGetLastError();
}

hipError_t launch_cmpdt(const double* uu, const double* gg, int nv, int ncell, double dx, const HydroParams& hp,
                        double* d_dt, hipStream_t stream) {
  hipLaunchKernelGGL(cmpdt_group, dim3(1), dim3(256), 0, stream, uu, gg, nv, ncell, dx, hp, d_dt);
  return hipGetLastError();
}

hipError_t launch_cons_finish(const double* partials, long nblocks, double* out, int accumulate, hipStream_t s) {
  hipLaunchKernelGGL(cons_finish, dim3(1), dim3(256), 0, s, partials, nblocks, out, accumulate);
  return hipGetLastError();
}

hipError_t launch_set_doubles(double* p, int n, double v, hipStream_t s) {
  hipLaunchKernelGGL(set_doubles, dim3((n + 63) / 64), dim3(64), 0, s, p, n, v);
  return hipGetLastError();
}

hipError_t launch_set_double(double* p, double v, hipStream_t s) {
  hipLaunchKernelGGL(set_double, dim3(1), dim3(1), 0, s, p, v);
  return hipGetLastError();
}

// The workgroups that a launch with sums may have, 3 doubles each in the
// caller's buffer (the level launch: 8x8 tiles of 4 planes).
static long sums_blocks(int n) {
  const long blocks = (long)n * n * n / 256;
  return blocks > 1 ? blocks : 1;
}
size_t uniform_sums_work_bytes(int n) { return (size_t)sums_blocks(n) * 3 * sizeof(double); }

hipError_t launch_courant(const double* u, int n, double dx, const HydroParams& hp, double* d_dt, hipStream_t s,
                          double* partials, double* d_sums) {
  const long ncell = (long)n * n * n;
  long blocks = (ncell + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  // n^3 need not be a multiple of 256: the kernel strides over the cells, so
  // the workgroups that the buffer has room for take the rest
  if (partials && blocks > sums_blocks(n)) blocks = sums_blocks(n);
  hipLaunchKernelGGL(courant_kernel, dim3((unsigned)blocks), dim3(256), 0, s, u, ncell, dx, hp, d_dt, partials);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !partials) return e;
  hipLaunchKernelGGL(cons_finish, dim3(1), dim3(256), 0, s, (const double*)partials, blocks, d_sums, 0);
  return hipGetLastError();
}

// Tile choice: the launch-shape knob when it divides n, else 16x12 (three
// interior waves and one ring wave: the ring's work is a third of a tile's,
// against a half for 16x8), whose last tiles may reach past the level, or
// 16x8 for n <= 24, where a third of a 16x12 tile's rows would.  Where the
// estimates say so by a margin, 32x16, one workgroup of 10 waves on each CU,
// whose ring is a fifth of the tile.  Of the sides up to 160 that is 64 and
// 128 in FP64 and 56 and 64 in FP32-mixed, where its workgroups just fill the
// CUs.  The estimates were measured with hllc and minmod; the choice holds for
// every solver with minmod, moncen and its generalised form, 32x16's time in
// 16x12's: 64^3 0.87 to 0.95 in FP64 and 0.81 to 0.90 in FP32-mixed, 128^3
// 0.80 to 0.90, 56^3 0.83 to 0.97.  What the margin leaves out would gain with
// some and lose with others (96^3 0.95 to 1.02 and 0.90 to 1.09, 128^3 in
// FP32-mixed 0.86 to 1.09, 160^3 0.83 to 1.01 and 0.94 to 1.22), and 32^3
// loses (1.13 to 1.51).  Larger levels take longer for a plane than the
// estimate says (512^3 FP32-mixed 4.4 against 3.8 ms): 16x12 above 160.
hipError_t launch_uniform_godunov(const double* u, double* unew, int n, double dx, const double* d_dt,
                                  double* d_dt_next, const HydroParams& hp, bool fp32, hipStream_t s,
                                  double* partials, double* d_sums) {
  UniformArgs a{u, unew, d_dt, d_dt_next, partials, n, dx, hp};
  int TX = 16, TY = 12;
  const int tile = tuning().level_tile;
  if (tile == 1 && n % 32 == 0) { TX = 32; TY = 8; }
  else if (tile == 3 || n < 16) { TX = 8; TY = 8; }
  else if (tile == 4 && n % 32 == 0) { TX = 32; TY = 16; }
  else if ((tile == 2 && n % 16 == 0) || (tile == 0 && n <= 24)) { TX = 16; TY = 8; }
  const auto tiles_of = [n](int tx, int ty) { return (long)((n + tx - 1) / tx) * ((n + ty - 1) / ty); };
  // with sums, three doubles per workgroup have to fit the caller's buffer
  const long max_blocks = partials ? sums_blocks(n) : 0x7fffffffL;
  // The estimates were measured with hllc up to 256^3.  On larger levels they
  // ask for chunks of up to all n planes, whose workgroups end too far apart:
  // 64 planes at most there (384^3 in FP32-mixed 1696 us in chunks of 64
  // planes, 1805 in one of 384, llf and moncen with sums 2044 and 2313; FP64
  // 2832 and, of 192, 2965).  In FP32-mixed workgroups of the exact solver,
  // whose faces iterate for as long as their states need, end farther apart
  // still: 192^3 takes 507 us in chunks of 16 planes and 568 in those of 39,
  // 288^3 1595 and 2012 (of 144).  acoustic: 192^3 the same, 288^3 818 in
  // chunks of 36 and 897.  Up to 160^3 the estimated chunks are the better
  // ones (160^3, exact: 349 us in chunks of 23 planes, 364 of 16).
  int longest = n > 256 ? 64 : n;
  if (fp32 && n > 160 && hp.riemann == kEXACT) longest = 16;
  if (fp32 && n > 160 && hp.riemann == kACOUSTIC) longest = 40;
  int TZ = tuning().level_tz;
  if (tile == 0 && TZ == 0 && TY == 12 && n >= 32 && n <= 160) {
    double narrow, wide;
    best_tz(n, tiles_of(16, 12), fp32, max_blocks, longest, level_estimate, &narrow);
    best_tz(n, tiles_of(32, 16), fp32, max_blocks, longest, wide_estimate, &wide);
    if (wide < 0.93 * narrow) { TX = 32; TY = 16; }
  }
  const long tiles = tiles_of(TX, TY);
  if (TZ < 4 || TZ > n || n % TZ != 0 || tiles * (n / TZ) > max_blocks) 
    TZ = best_tz(n, tiles, fp32, max_blocks, longest, TX == 32 && TY == 16 ? wide_estimate : level_estimate);
  if (fp32) {
    if (TY == 12) return launch_tile<float, 16, 12>(a, TZ, d_sums, s);
    if (TX == 32 && TY == 16) return launch_tile<float, 32, 16>(a, TZ, d_sums, s);
    if (TX == 32) return launch_tile<float, 32, 8>(a, TZ, d_sums, s);
    if (TX == 16) return launch_tile<float, 16, 8>(a, TZ, d_sums, s);
    return launch_tile<float, 8, 8>(a, TZ, d_sums, s);
  }
  if (TY == 12) return launch_tile<double, 16, 12>(a, TZ, d_sums, s);
  if (TX == 32 && TY == 16) return launch_tile<double, 32, 16>(a, TZ, d_sums, s);
  if (TX == 32) return launch_tile<double, 32, 8>(a, TZ, d_sums, s);
  if (TX == 16) return launch_tile<double, 16, 8>(a, TZ, d_sums, s);
  return launch_tile<double, 8, 8>(a, TZ, d_sums, s);
}

}  // namespace ramses
