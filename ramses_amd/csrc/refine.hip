// Mesh refinement on the GPU: the refinement map of a level (flag_fine,
// amr/flag_utils.f90:57-106) and the creation / destruction of the octs of
// the next level (refine_fine, amr/refine_utils.f90:332-585), with the tree
// (son / father / nbor), the flags and the free-grid list resident in HBM.
//
// flag_fine      flag_mark   test_flag: a refined cell stays flagged while a
//                            child is refined or flagged (:168-208), and
//                            beside it the hydro_flag / hydro_refine gradient
//                            criteria (hydro/hydro_flag.f90:1-180,
//                            hydro/godunov_utils.f90:125-263), one word per oct
//                flag_smooth smooth_fine (:555-677), its three passes in one,
//                            and at the end ensure_ref_rules (:213-276)
// refine_fine    refine_scan what is made, killed and kept, each with its rank
//                            in the order in which the reference visits cells,
//                            and the decision
//                refine_apply make_grid_fine (:590-948): the k-th new oct takes
//                            the k-th free grid from the head of the free
//                            list, links to its father and neighbour cells,
//                            and its cells are prolongated (interpol_hydro);
//                            kill_grid (:953-1158): the k-th killed oct is
//                            cleared and appended to the tail of the free list;
//                            the next level's grid list rebuilt as build_comm
//                            does from the linked list
//                            (amr/virtual_boundaries.f90:1286-1420): survivors
//                            in order, then new octs in creation order.
//                            Ten launches of 3 to 10 us, 150 in an adaptive
//                            coarse step, when the marks, each scan's tiles,
//                            totals and offsets, the decision, the makes, the
//                            kills and the list were kernels of their own.
// The free list of the reference is a FIFO (taken at headf, returned at
// tailf); here it is a ring of ngridmax grid indices.
#include "hydro_device.hpp"
#include "amr_args.hpp"
#include "amr_device.hpp"

namespace ramses {

hipError_t launch_set_ints(int* p, int n, int v, hipStream_t s);

struct RefineParams {
  double err_grad_d, err_grad_u, err_grad_p;
  double floor_d, floor_u, floor_p;
  int nexpand;
};

struct TreeMut {
  int* son;
  int* father;
  int* nbor;
};

namespace {

// --- flag_fine ----------------------------------------------------------

// Cells of the level in cell-major order: i -> (ind = i / noct + 1, a = i %
// noct).  The flag kernels loop over them grid-stride; the oct count is the
// host value or, with dn set, the one in device memory.
__device__ __forceinline__ void level_cell(const int* active, int noct, const AmrTreeView& t, long i, int& g,
                                           int& ind, long& c) {
  ind = (int)(i / noct) + 1;
  g = active[i % noct];
  c = cell_of(t, ind, g);
}

#define FOR_LEVEL_CELLS(noct_h, dn)                                                             \
  const int noct = level_count(noct_h, dn);                                                     \
  const long ncells_ = 8L * noct, stride_ = (long)gridDim.x * blockDim.x;                       \
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < ncells_; i += stride_)

// Below levelmin every cell is flagged (init_flag :150-157).
__global__ void flag_all(const int* active, int noct_h, const int* dn, AmrTreeView t, int* flag1) {
  FOR_LEVEL_CELLS(noct_h, dn) {
    int g, ind;
    long c;
    level_cell(active, noct, t, i, g, ind, c);
    flag1[c] = 1;
  }
}

struct Prim3 {
  double d, v[3], p;
};

// hydro_refine's conversion to primitives (godunov_utils.f90:149-180).
__device__ __forceinline__ Prim3 refine_prim(const double* u, long us, long c, const HydroParams& hp) {
  Prim3 q;
  q.d = fmax_f(u[c], hp.smallr);
  for (int d = 0; d < 3; ++d) q.v[d] = u[(long)(d + 1) * us + c] / q.d;
  double ek = 0.0;
  for (int d = 0; d < 3; ++d) ek = ek + (0.5 * q.d) * (q.v[d] * q.v[d]);
  q.p = (hp.gamma - 1.0) * (u[4 * us + c] - ek);
  return q;
}

__device__ __forceinline__ double grad_err(double g, double m, double d, double floor_x) {
  return 2.0 * fmax_f(__builtin_fabs((d - m) / ((d + m) + floor_x)), __builtin_fabs((m - g) / ((m + g) + floor_x)));
}

// Whether cell ind of grid g meets a gradient criterion.
__device__ __forceinline__ bool hydro_flagged(const AmrTreeView& t, const double* u, long us, const RefineParams& rp,
                                              const HydroParams& hp, int g, int ind) {
  const long c = cell_of(t, ind, g);
  // The six neighbours' states are loaded before any test (independent
  // loads, issued together); the tests have no side effects, so OR-ing all
  // of them gives the flag of the reference's short-circuit order.
  const Prim3 m = refine_prim(u, us, c, hp);
  long cn[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const long cc = nbor_cell(t, g, ind, k + 1);
    cn[k] = cc != 0 ? cc : nbor_of(t, g, k + 1);  // missing neighbour: the father's neighbour
  }
  Prim3 nq[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) nq[k] = refine_prim(u, us, cn[k], hp);
  bool ok = false;
#pragma unroll
  for (int idim = 0; idim < 3; ++idim) {
    const Prim3& l = nq[2 * idim];
    const Prim3& r = nq[2 * idim + 1];
    if (rp.err_grad_d >= 0.0) ok = ok | (grad_err(l.d, m.d, r.d, rp.floor_d) > rp.err_grad_d);
    if (rp.err_grad_p >= 0.0) ok = ok | (grad_err(l.p, m.p, r.p, rp.floor_p) > rp.err_grad_p);
    if (rp.err_grad_u >= 0.0) {
      const double fu2 = rp.floor_u * rp.floor_u;
      const double cg = __builtin_sqrt(fmax_f(hp.gamma * l.p / l.d, fu2));
      const double cm = __builtin_sqrt(fmax_f(hp.gamma * m.p / m.d, fu2));
      const double cd = __builtin_sqrt(fmax_f(hp.gamma * r.p / r.d, fu2));
      for (int d = 0; d < 3; ++d) {
        const double vg = l.v[d], vm = m.v[d], vd = r.v[d];
        const double e1 = __builtin_fabs((vd - vm) / ((((cd + cm) + __builtin_fabs(vd)) + __builtin_fabs(vm)) + rp.floor_u));
        const double e2 = __builtin_fabs((vm - vg) / ((((cm + cg) + __builtin_fabs(vm)) + __builtin_fabs(vg)) + rp.floor_u));
        ok = ok | (2.0 * fmax_f(e1, e2) > rp.err_grad_u);
      }
    }
  }
  return ok;
}

// A level's flags between flag_mark and the last flag_smooth are one word per
// oct: bit ind-1 the flag of cell ind, bit 8+ind-1 its gradient criterion.
// The words alternate between two cells of each oct in flag2.
__device__ __forceinline__ long flag_word(const AmrTreeView& t, int which, int g) { return cell_of(t, 1 + which, g); }

// 32 octs a workgroup, eight cells each: 32 consecutive octs per cell, so the
// level's cells are read in runs of 256 bytes.
__global__ __launch_bounds__(256) void flag_mark(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                const double* u, long us, const int* flag1, int* flag2,
                                                RefineParams rp, HydroParams hp, int hydro) {
  __shared__ int word[32];
  const int noct = level_count(noct_h, dn);
  const int lane = threadIdx.x & 31, ind = (threadIdx.x >> 5) + 1;
  for (int base = blockIdx.x * 32; base < noct; base += gridDim.x * 32) {
    const int a = base + lane;
    if (threadIdx.x < 32) word[threadIdx.x] = 0;
    __syncthreads();
    if (a < noct) {
      const int g = active[a];
      const int s = t.son[cell_of(t, ind, g)];
      int f = 0;
      if (s > 0)
        for (int k = 1; k <= 8; ++k) {
          const long cc = cell_of(t, k, s);
          if (t.son[cc] > 0 || flag1[cc] == 1) f = 1;
        }
      if (hydro && hydro_flagged(t, u, us, rp, hp, g, ind)) f |= 256;
      if (f) atomicOr(&word[lane], f << (ind - 1));
    }
    __syncthreads();
    if (threadIdx.x < 32 && a < noct) flag2[flag_word(t, 0, active[a])] = word[lane];
    __syncthreads();
  }
}

// smooth_fine (amr/flag_utils.f90:555-677): three Jacobi passes, a cell being
// flagged when it was, or when at least 1, 2, 2 of its six neighbours at the
// level were; cells whose oct does not exist stay unflagged.  One launch does
// all three: three passes reach three cells, so an oct's own flags follow
// from an 8^3 block of flags around it, its 26 neighbour octs and the next
// one along each axis.  Eight lanes hold the block as bits, a z plane each: a
// pass is a few shifts and a carry-save count of six planes.  Bits that wrap
// from row to row start at the block's faces and stay off the centre's two
// columns for three passes.
//
// A launch per pass took 4.8 us on levels of a thousand octs, 121 of them in
// an adaptive coarse step; this form is 11 us for all three.
//
// 32 lanes find the neighbours of an oct, 8 octs a workgroup.  merge: the
// gradient criteria join after the passes; last: ensure_ref_rules (an oct
// with a missing or unrefined neighbour is unflagged) if asked, and the flags
// go to flag1.
__global__ __launch_bounds__(256) void flag_smooth(const int* active, int noct_h, const int* dn, AmrTreeView t,
                                                  int ilevel, int from, int* flag2, int* flag1, int merge, int last,
                                                  int ensure) {
  __shared__ unsigned long long flags[8][8], exist[8][8];
  __shared__ int own[8], bad[8];
  const int noct = level_count(noct_h, dn);
  const int o = threadIdx.x >> 5, j = threadIdx.x & 31;
  for (int base = blockIdx.x * 8; base < noct; base += gridDim.x * 8) {
    if (j < 8) {
      flags[o][j] = 0;
      exist[o][j] = 0;
    }
    if (j == 8) bad[o] = 0;
    __syncthreads();
    const int a = base + o;
    if (a < noct && j < 27) {
      const int x = j % 3, y = (j / 3) % 3, z = j / 9;
      const int g = active[a];
      const long nf = nbor_father_cell(t, t.father[g], x, y, z, ilevel);
      const int gn = nf > 0 ? t.son[nf] : 0;
      // the oct's cells 2x+1.. of the block (its own at 3, 4)
      auto put = [&](unsigned w, int bx, int by, int bz, int nz) {
        for (int k = 0; k < nz; ++k) {
          const unsigned q = w >> 4 * k & 15;
          const unsigned long long m = (unsigned long long)((q & 3) | (q & 12) << 6) << (bx + 8 * by);
          if (m) atomicOr(&flags[o][bz + k], m);
        }
      };
      auto mark = [&](unsigned e, int bx, int by, int bz, int nz) {
        for (int k = 0; k < nz; ++k)
          atomicOr(&exist[o][bz + k], (unsigned long long)((e & 3) | (e & 12) << 6) << (bx + 8 * by));
      };
      if (gn > 0) {
        const int w = flag2[flag_word(t, from, gn)];
        put((unsigned)w & 255, 2 * x + 1, 2 * y + 1, 2 * z + 1, 2);
        mark(15, 2 * x + 1, 2 * y + 1, 2 * z + 1, 2);
        if (j == 13) own[o] = w;
        if ((x != 1) + (y != 1) + (z != 1) == 1) {
          // the next oct along the axis: its layer of four cells at 0 or 7
          const int ax = x != 1 ? 0 : (y != 1 ? 1 : 2), plus = (ax == 0 ? x : (ax == 1 ? y : z)) == 2;
          const int gf = t.son[nbor_of(t, gn, 1 + 2 * ax + plus)];
          if (gf > 0) {
            const unsigned b = (unsigned)flag2[flag_word(t, from, gf)] & 255;
            if (ax == 0) {
              const unsigned q = plus ? b : b >> 1;  // cells of x bit 0, or 1
              const unsigned c = (q & 1) | (q >> 2 & 1) << 2 | (q >> 4 & 1) << 4 | (q >> 6 & 1) << 6;
              put(c, plus ? 7 : 0, 3, 3, 2);
              mark(5, plus ? 7 : 0, 3, 3, 2);
            } else if (ax == 1) {
              const unsigned q = plus ? b : b >> 2;
              put((q & 3) | (q >> 4 & 3) << 4, 3, plus ? 7 : 0, 3, 2);
              mark(3, 3, plus ? 7 : 0, 3, 2);
            } else {
              put(plus ? b & 15 : b >> 4, 3, 3, plus ? 7 : 0, 1);
              mark(15, 3, 3, plus ? 7 : 0, 1);
            }
          }
        }
      } else {
        atomicOr(&bad[o], 1);
      }
    }
    __syncthreads();
    if (threadIdx.x < 64) {
      const int q = threadIdx.x >> 3, z = threadIdx.x & 7;  // one wavefront: oct q, plane z
      unsigned long long S = flags[q][z];
      const unsigned long long E = exist[q][z];
#pragma unroll
      for (int pass = 0; pass < 3; ++pass) {
        const unsigned long long up = __shfl_down(S, 1, 8), dn_ = __shfl_up(S, 1, 8);
        const unsigned long long nb[6] = {S << 1, S >> 1, S << 8, S >> 8, z < 7 ? up : 0, z > 0 ? dn_ : 0};
        unsigned long long one = 0, two = 0;
#pragma unroll
        for (int k = 0; k < 6; ++k) {
          two |= one & nb[k];
          one |= nb[k];
        }
        S = (S | (pass == 0 ? one : two)) & E;
      }
      const unsigned long long r = S >> 27;  // x = 3, y = 3
      const int nib = (int)(r & 3) | (int)(r >> 8 & 3) << 2;
      int f = __shfl(nib, 3, 8) | __shfl(nib, 4, 8) << 4;
      const int a2 = base + q;
      if (a2 < noct) {
        const int w = own[q], g = active[a2];
        if (merge) f |= w >> 8 & 255;
        if (last)
          flag1[cell_of(t, z + 1, g)] = ensure && bad[q] ? 0 : f >> z & 1;
        else if (z == 0)
          flag2[flag_word(t, from ^ 1, g)] = f | (w & ~255);
      }
    }
    __syncthreads();
  }
}

// --- exclusive scan of 64-bit counters ----------------------------------

constexpr int kScanThreads = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ long long block_excl_scan(long long x, long long* sh, long long& total) {
  // wave-level inclusive scan, then across the block's waves
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  long long v = x;
  for (int o = 1; o < 64; o <<= 1) {
    const long long y = __shfl_up(v, o, 64);
    if (lane >= o) v += y;
  }
  if (lane == 63) sh[wid] = v;
  __syncthreads();
  long long base = 0, tot = 0;
  const int nw = blockDim.x >> 6;
  for (int w = 0; w < nw; ++w) {
    if (w < wid) base += sh[w];
    tot += sh[w];
  }
  __syncthreads();
  total = tot;
  return base + v - x;
}

// Values that the last workgroup of a launch reads from the others.  A device
// -scope exchange that returns has reached the point where all XCDs meet, so
// the count that depends on its return value cannot be seen before it; a
// fence instead would write back and drop the whole L2 of the XCD, for every
// workgroup.
__device__ __forceinline__ unsigned publish(long long* p, long long v) {
  unsigned r = (unsigned)atomicExch(reinterpret_cast<unsigned long long*>(p), (unsigned long long)v);
  asm volatile("v_and_b32 %0, 0, %0" : "+v"(r));
  return r;  // 0, after the exchange
}
__device__ __forceinline__ long long published(const long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One block: exclusive scan of published tile totals; sums[ntiles] = grand
// total, returned to every thread.
__device__ long long scan_totals(long long* sums, long ntiles, long long* sh) {
  long long carry = 0;
  for (long b0 = 0; b0 < ntiles; b0 += blockDim.x) {
    const long i = b0 + threadIdx.x;
    const long long x = i < ntiles ? published(sums + i) : 0;
    long long total;
    const long long e = block_excl_scan(x, sh, total);
    if (i < ntiles) sums[i] = carry + e;
    carry += total;
  }
  if (threadIdx.x == 0) sums[ntiles] = carry;
  return carry;
}

__device__ __forceinline__ long long scan_offset(const long long* out, const long long* sums, long i) {
  return out[i] + sums[i / kScanTile];
}

// --- refine_fine ----------------------------------------------------------

// The decision of a refinement, in device memory: octs created and killed,
// whether it is carried out, and the next level's octs and the free list's
// head and length before it.
enum Ctrl : int { kCreate = 0, kKill, kOk, kFine, kHead, kNumbf, kCtrlInts };

// Workspace of a refinement of nslot slots whose next level has nf octs.
// Slot p = batch*256 + (ind-1)*32 + lane over the level's active list in
// nvector=32 batches, the order in which the reference visits cells.
struct RefineWork {
  long long* mark;   // per slot: create (low 32 bits) | kill << 32
  long long* off;    // exclusive scan of mark within its tile
  long long* sums;   // the tiles' offsets, and the grand total
  long long* fsums;  // the same of the surviving octs
  int* rank;         // per oct of the next level: its place among the survivors of its tile, or -1
  int* copy;         // the next level's list before
  int* ctrl;
  unsigned* done;    // workgroups that have finished; zero between launches
};

inline long refine_slots(int noct) { return (long)((noct + 31) / 32) * 256; }
inline size_t scan_tiles(long n) { return (size_t)((n + kScanTile - 1) / kScanTile) + 1; }

RefineWork refine_work(void* work, long nslot, int nf) {
  RefineWork w;
  w.mark = (long long*)(((uintptr_t)work + 255) & ~(uintptr_t)255);
  w.off = w.mark + nslot;
  w.sums = w.off + nslot;
  w.fsums = w.sums + scan_tiles(nslot);
  w.rank = (int*)(w.fsums + scan_tiles(nf));
  w.copy = w.rank + nf;
  w.ctrl = w.copy + nf;
  w.done = (unsigned*)(w.ctrl + kCtrlInts);
  return w;
}

// What a refinement is decided from.  With dn, dnf and dfree the level's and
// the next level's oct counts and the free list {head, numbf, used_mem} are
// read from device memory; else they are the host's.
struct RefineScan {
  AmrTreeView t;
  const int* active;
  const int* fine;  // the next level's list
  const int* flag1;
  const int* dn;
  const int* dnf;
  const int* dfree;
  int noct, nfine, head, numbf, capacity;
  int* error;  // or null
  RefineWork w;
};

// One mark per slot, and for every oct of the next level whether it survives:
// a refined cell whose flag is 0 loses its oct, a flagged leaf gets one, and
// the exclusive scans of both give every new, killed or surviving oct its
// rank in the reference's order.  The workgroup that finishes last turns the
// tiles' totals into offsets and decides: ok is 0 when there is nothing to do
// or when the free list cannot hold the new octs ("No more free memory",
// amr/refine_utils.f90:415-423: error bit 4, nothing is modified).  A
// refinement that would take the next level beyond `capacity` octs (the
// workspace of a captured step) is refused the same way (error bit 8).
//
// A workgroup knows from the counts whether it works, and only the working
// ones are waited for: one that starts after the decision has to read the
// same counts, so nothing here writes them (refine_apply does).
__global__ __launch_bounds__(kScanThreads) void refine_scan(RefineScan r) {
  __shared__ long long sh[kScanThreads / 64];
  __shared__ int last;
  const int noct = r.dn ? *r.dn : r.noct, nf = r.dnf ? *r.dnf : r.nfine;
  const long nslot = (long)((noct + 31) / 32) * 256;
  const int nt = (int)((nslot + kScanTile - 1) / kScanTile), ntf = (nf + kScanTile - 1) / kScanTile;
  const unsigned working = min((unsigned)max(nt + ntf, 1), gridDim.x);
  if (blockIdx.x >= working) return;
  unsigned dep = 0;
  for (int tile = blockIdx.x; tile < nt + ntf; tile += gridDim.x) {
    long long v[kScanItems], s = 0, total;
    if (tile < nt) {
      const long base = (long)tile * kScanTile + (long)threadIdx.x * kScanItems;
      for (int k = 0; k < kScanItems; ++k) {
        const long p = base + k;
        v[k] = 0;
        if (p < nslot) {
          const int q = (int)(p & 255), a = (int)(p >> 8) * 32 + (q & 31);
          if (a < noct) {
            const long c = cell_of(r.t, (q >> 5) + 1, r.active[a]);
            const int son = r.t.son[c], f = r.flag1[c];
            if (f == 1 && son == 0) v[k] = 1;
            if (f == 0 && son > 0) v[k] = 1LL << 32;
          }
          r.w.mark[p] = v[k];
        }
        s += v[k];
      }
      long long run = block_excl_scan(s, sh, total);
      for (int k = 0; k < kScanItems; ++k) {
        if (base + k < nslot) r.w.off[base + k] = run;
        run += v[k];
      }
      if (threadIdx.x == 0) dep |= publish(r.w.sums + tile, total);
    } else {
      const int base = (tile - nt) * kScanTile + (int)threadIdx.x * kScanItems;
      for (int k = 0; k < kScanItems; ++k) {
        v[k] = 0;
        if (base + k < nf) {
          const int g = r.fine[base + k];
          r.w.copy[base + k] = g;
          v[k] = r.flag1[r.t.father[g]] != 0 ? 1 : 0;  // its father cell is refined
        }
        s += v[k];
      }
      int run = (int)block_excl_scan(s, sh, total);
      for (int k = 0; k < kScanItems; ++k) {
        if (base + k < nf) r.w.rank[base + k] = v[k] ? run : -1;
        run += (int)v[k];
      }
      if (threadIdx.x == 0) dep |= publish(r.w.fsums + (tile - nt), total);
    }
  }
  if (threadIdx.x == 0) last = atomicAdd(r.w.done, 1u + dep) == working - 1;
  __syncthreads();
  if (!last) return;
  const long long tot = scan_totals(r.w.sums, nt, sh);
  scan_totals(r.w.fsums, ntf, sh);
  if (threadIdx.x != 0) return;
  *r.w.done = 0;
  const int head = r.dfree ? r.dfree[0] : r.head, numbf = r.dfree ? r.dfree[1] : r.numbf;
  const int nc = (int)(tot & 0xffffffffLL), nk = (int)(tot >> 32);
  int ok = (nc > 0 || nk > 0) ? 1 : 0;
  if (ok && nc >= numbf) {
    ok = 0;
    if (r.error) atomicOr(r.error, 4);
  }
  if (ok && (long)nf - nk + nc > r.capacity) {
    ok = 0;
    if (r.error) atomicOr(r.error, 8);
  }
  r.w.ctrl[kCreate] = nc;
  r.w.ctrl[kKill] = nk;
  r.w.ctrl[kOk] = ok;
  r.w.ctrl[kFine] = nf;
  r.w.ctrl[kHead] = head;
  r.w.ctrl[kNumbf] = numbf;
}

struct RefineRun {
  AmrTreeView t;      // read view of the same arrays as m
  TreeMut m;
  const int* active;  // level ilevel
  const int* dn;      // its oct count in device memory, or null
  int noct;
  int* dnf;           // the next level's count and the free list in device memory, or null
  int* dfree;
  int* fine;          // the next level's list
  int* pos;
  int* ring;
  int cap;          // ngridmax
  double* uold;
  double* unew;
  long us;
  int* flag1;
  int* flag2;
  double* xg;       // grid centres xg[3*igrid + d], or null
  double dx;        // cell size of the level being refined (0.5^ilevel)
  int interpol_type, interpol_var;
  double smallr;
  int* error;
  RefineWork w;
};

// The k-th new oct takes the k-th free grid.
__device__ __forceinline__ int new_grid(const RefineRun& r, int k) {
  return r.ring[(int)(((long)r.w.ctrl[kHead] + k) % r.cap)];
}

__device__ void make_slot(const RefineRun& r, long p) {
  if ((r.w.mark[p] & 0xffffffffLL) == 0) return;
  const int b = (int)(p >> 8), q = (int)(p & 255);
  const int ind = (q >> 5) + 1, lane = q & 31;
  const int igrid = r.active[b * 32 + lane];
  const long c = cell_of(r.t, ind, igrid);
  const int k = (int)(scan_offset(r.w.off, r.w.sums, p) & 0xffffffffLL);
  const int g = new_grid(r, k);
  r.m.son[c] = g;
  r.m.father[g] = (int)c;
  if (r.xg) {  // centre of the new oct = centre of its father cell (make_grid_fine :663-673)
    const int p[3] = {(ind - 1) & 1, ((ind - 1) >> 1) & 1, (ind - 1) >> 2};
    for (int d = 0; d < 3; ++d) r.xg[3L * g + d] = r.xg[3L * igrid + d] + ((double)p[d] - 0.5) * r.dx;
  }
  long nb[7];
  nb[0] = c;
  for (int in = 1; in <= 6; ++in) {
    const long n = nbor_cell(r.t, igrid, ind, in);
    if (n == 0) atomicOr(r.error, 2);  // "Fatal error in make_grid_fine"
    nb[in] = n;
    r.m.nbor[(long)(in - 1) * r.cap + g] = (int)n;
  }
  double u1[7][5], u2[8][5];
  for (int j = 0; j < 7; ++j)
    for (int v = 0; v < 5; ++v) u1[j][v] = r.uold[(long)v * r.us + nb[j]];
  interpol_oct(u1, u2, r.interpol_type, r.interpol_var, r.smallr);
  for (int j = 1; j <= 8; ++j) {
    const long cc = cell_of(r.t, j, g);
    for (int v = 0; v < 5; ++v) r.uold[(long)v * r.us + cc] = u2[j - 1][v];
    r.m.son[cc] = 0;
    r.flag1[cc] = 0;
  }
}

__device__ void kill_slot(const RefineRun& r, long p) {
  if ((r.w.mark[p] >> 32) == 0) return;
  const int b = (int)(p >> 8), q = (int)(p & 255);
  const int ind = (q >> 5) + 1, lane = q & 31;
  const long c = cell_of(r.t, ind, r.active[b * 32 + lane]);
  const int k = (int)(scan_offset(r.w.off, r.w.sums, p) >> 32);
  const int g = r.m.son[c];
  r.m.son[c] = 0;
  r.m.father[g] = 0;
  if (r.xg)
    for (int d = 0; d < 3; ++d) r.xg[3L * g + d] = 0.0;
  for (int in = 1; in <= 6; ++in) r.m.nbor[(long)(in - 1) * r.cap + g] = 0;
  for (int j = 1; j <= 8; ++j) {
    const long cc = cell_of(r.t, j, g);
    r.m.son[cc] = 0;
    r.flag1[cc] = 0;
    r.flag2[cc] = 0;
    for (int v = 0; v < 5; ++v) {
      r.uold[(long)v * r.us + cc] = 0.0;
      r.unew[(long)v * r.us + cc] = 0.0;
    }
  }
  r.ring[(int)(((long)r.w.ctrl[kHead] + r.w.ctrl[kNumbf] + k) % r.cap)] = g;
}

// The decided refinement: the new octs read the level's own cells and take
// grids that were free before, the killed ones clear the next level's and go
// behind the free list's tail, and the next level's list is rebuilt:
// survivors in order (from its copy; nothing moves when nothing is killed),
// then the new octs; pos follows.  One thread brings counts in device memory
// up to date, which this kernel takes from ctrl.  No part reads what another
// writes.
__global__ __launch_bounds__(128) void refine_apply(RefineRun r) {
  const int* ctrl = r.w.ctrl;
  if (!ctrl[kOk]) return;
  const long n = (long)((level_count(r.noct, r.dn) + 31) / 32) * 256;
  const long stride = (long)gridDim.x * blockDim.x, id = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nc = ctrl[kCreate], nk = ctrl[kKill], nf = ctrl[kFine];
  if (id == 0 && r.dnf) {
    const int numbf = ctrl[kNumbf];
    *r.dnf = nf - nk + nc;
    r.dfree[0] = (int)(((long)ctrl[kHead] + nc) % r.cap);
    if (nc > 0) r.dfree[2] = r.cap - (numbf - nc);  // make_grid_fine's last used_mem
    r.dfree[1] = numbf - nc + nk;
  }
  for (long i = (nk > 0 ? 0 : nf) + id; i < (long)nf + nc; i += stride) {
    int g, at;
    if (i < nf) {
      const int k = r.w.rank[i];
      if (k < 0) continue;
      g = r.w.copy[i];
      at = k + (int)r.w.fsums[i / kScanTile];
    } else {
      g = new_grid(r, (int)(i - nf));
      at = (int)i - nk;
    }
    r.fine[at] = g;
    r.pos[g] = at;
  }
  for (long p = id; p < n; p += stride) {
    make_slot(r, p);
    kill_slot(r, p);
  }
}

inline unsigned nblk(long n, int b) { return (unsigned)((n + b - 1) / b); }

}  // namespace

// flag_fine(ilevel, icount) for one level (amr/flag_utils.f90:57-106).  With
// dn the oct count is read from device memory (persistent grids).
hipError_t launch_flag_fine(const int* active, int noct, const AmrTreeView& t, int ilevel, int icount, int levelmin,
                            int nlevelmax, const double* u, long us, int* flag1, int* flag2, const RefineParams& rp,
                            const HydroParams& hp, hipStream_t s, const int* dn) {
  if (ilevel == nlevelmax || (!dn && noct <= 0)) return hipSuccess;
  if (ilevel < levelmin) {
    hipLaunchKernelGGL(flag_all, dim3(dn ? persist_blocks() : nblk(8L * noct, 256)), dim3(256), 0, s, active, noct, dn, t,
                       flag1);
    return hipGetLastError();
  }
  const int hydro = rp.err_grad_d >= 0.0 || rp.err_grad_p >= 0.0 || rp.err_grad_u >= 0.0;
  hipLaunchKernelGGL(flag_mark, dim3(dn ? persist_blocks() : nblk(noct, 32)), dim3(256), 0, s, active, noct, dn, t, u, us,
                     (const int*)flag1, flag2, rp, hp, hydro);
  // smooth, join the criteria, then nexpand times more
  for (int e = 0; e <= rp.nexpand; ++e)
    hipLaunchKernelGGL(flag_smooth, dim3(dn ? persist_blocks() : nblk(noct, 8)), dim3(256), 0, s, active, noct, dn, t,
                       ilevel, e & 1, flag2, flag1, e == 0 ? 1 : 0, e == rp.nexpand ? 1 : 0,
                       ilevel > levelmin && icount < 2 ? 1 : 0);
  return hipGetLastError();
}

// Workspace of refine_fine for a level of noct octs whose next level has
// noct_fine octs.
size_t refine_work_bytes(int noct, int noct_fine) {
  const long nslot = refine_slots(noct);
  return (2 * (size_t)nslot + scan_tiles(nslot) + scan_tiles(noct_fine)) * sizeof(long long) +
         (2 * (size_t)noct_fine + kCtrlInts + 1) * sizeof(int) + 256;
}

// refine_fine(ilevel) (amr/refine_utils.f90:332-585).  The one host
// synchronisation reads the number of octs to create and to kill.
// On return *noct_fine, *head, *numbf describe the rebuilt next level and
// the free list.  *nofree = 1 (and nothing is modified) when the free list
// cannot hold the new octs.
hipError_t launch_refine_fine(const int* active, int noct, int ilevel, const AmrTreeView& t, const TreeMut& m,
                              int* active_fine, int* noct_fine, int* pos, int* ring, int* head, int* numbf,
                              int* used_mem, int* flag1, int* flag2, double* xg, double* uold, double* unew,
                              int interpol_type, int interpol_var, double smallr, void* work, int* d_error,
                              int* nofree, hipStream_t s) {
  *nofree = 0;
  if (noct <= 0) return hipSuccess;
  const long nslot = refine_slots(noct);
  const int nf = *noct_fine;
  const RefineWork w = refine_work(work, nslot, nf);
  hipError_t e = launch_set_ints((int*)w.done, 1, 0, s);
  if (e != hipSuccess) return e;
  const RefineScan scan{t, active, active_fine, flag1, nullptr, nullptr, nullptr, noct, nf, *head, *numbf,
                        0x7fffffff, nullptr, w};
  const unsigned tiles = nblk(nslot, kScanTile) + nblk(nf, kScanTile);
  hipLaunchKernelGGL(refine_scan, dim3(tiles), dim3(kScanThreads), 0, s, scan);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  int ctrl[kCtrlInts];
  if ((e = hipMemcpyAsync(ctrl, w.ctrl, sizeof(ctrl), hipMemcpyDeviceToHost, s)) != hipSuccess) return e;
  if ((e = hipStreamSynchronize(s)) != hipSuccess) return e;
  const int ncreate = ctrl[kCreate], nkill = ctrl[kKill];
  if (ncreate == 0 && nkill == 0) return hipSuccess;
  if (!ctrl[kOk]) {  // "No more free memory" (:415-423)
    *nofree = 1;
    return hipSuccess;
  }
  const RefineRun r{t, m, active, nullptr, noct, nullptr, nullptr, active_fine, pos, ring, t.ngridmax, uold, unew, t.ncell + 1, flag1,
                    flag2, xg, __builtin_ldexp(1.0, -ilevel), interpol_type, interpol_var, smallr, d_error, w};
  hipLaunchKernelGGL(refine_apply, dim3(nblk(nslot, 128)), dim3(128), 0, s, r);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  *noct_fine = nf - nkill + ncreate;
  *head = (int)(((long)*head + ncreate) % t.ngridmax);
  if (ncreate > 0) *used_mem = t.ngridmax - (*numbf - ncreate);  // make_grid_fine's last value
  *numbf = *numbf - ncreate + nkill;
  return hipSuccess;
}

// refine_fine(ilevel) with no host synchronisation, for a captured launch
// sequence: the level counts dn_l (level ilevel) and dn_f (level ilevel+1)
// and the free list dfree = {head, numbf, used_mem} live in device memory;
// work holds refine_work_bytes(capacity, capacity), every level holding at
// most `capacity` octs.  A refinement that would exhaust the free list sets
// error bit 4, one that would exceed the capacity error bit 8; either changes
// nothing.  done: a counter in device memory, zero between launches.
hipError_t launch_refine_fine_dev(const int* active, const int* dn_l, int ilevel, const AmrTreeView& t,
                                  const TreeMut& m, int* active_fine, int* dn_f, int* pos, int* ring, int* dfree,
                                  unsigned* done, int* flag1, int* flag2, double* xg, double* uold, double* unew,
                                  int interpol_type, int interpol_var, double smallr, void* work, int* d_error,
                                  int capacity, hipStream_t s) {
  RefineWork w = refine_work(work, refine_slots(capacity), capacity);
  w.done = done;
  const RefineScan scan{t, active, active_fine, flag1, dn_l, dn_f, dfree, 0, 0, 0, 0, capacity, d_error, w};
  hipLaunchKernelGGL(refine_scan, dim3(persist_blocks() / 2), dim3(kScanThreads), 0, s, scan);
  const RefineRun r{t, m, active, dn_l, 0, dn_f, dfree, active_fine, pos, ring, t.ngridmax, uold, unew, t.ncell + 1, flag1,
                    flag2, xg, __builtin_ldexp(1.0, -ilevel), interpol_type, interpol_var, smallr, d_error, w};
  hipLaunchKernelGGL(refine_apply, dim3(persist_blocks()), dim3(128), 0, s, r);
  return hipGetLastError();
}

}  // namespace ramses
