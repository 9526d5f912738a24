// The unsplit chain on tiles of 16 octs, shared by unsplit.hip (octs gathered
// by the caller) and amr.hip (octs gathered from the tree).
//
// An oct's 36 faces need 32 traced cells, its 8 own ones and the 24 next to
// its sides, and these the primitives of 80 cells.  A workgroup of eight
// wavefronts computes each of them once:
//   1. the primitives of the 80 cells of its 16 octs, into LDS;
//   2. one traced cell per thread, its six neighbours read from LDS, the
//      traced states written over the primitives by face and side;
//   3. one face per thread, the last 64 of the 576 by the last wavefront.
// The 16 octs are the fast index, so a wavefront holds four cells or four
// faces of one kind and direction and takes no divergent branch on them, and
// every access to an oct batch is a run of 128 bytes.
//
// Eight wavefronts are two per SIMD, so that two workgroups fill the four
// per SIMD that 128 VGPRs allow (nine wavefronts, one face each, left the
// second workgroup out: 1.97 ms against 1.44 ms for 2^20 octs in FP64; held
// to five per SIMD it spills: 1.94 ms).  8 octs and four wavefronts measured
// the same in FP64 and 9% slower in FP32-mixed, where runs of 64 bytes cost
// more than the finer grain gives.
#pragma once

#include <type_traits>

#include "hydro_device.hpp"

namespace ramses {
namespace oct_tile {

constexpr int kOcts = 16;
constexpr int kCells = 80;
constexpr int kTraced = 32;
constexpr int kFaces = 36;
constexpr int kThreads = kTraced * kOcts;
constexpr int kWaves = kThreads / 64;
constexpr int kOwnWaves = 8 * kOcts / 64;              // wavefronts of the octs' own cells; as many per direction beyond
constexpr int kRest = kFaces * kOcts - kThreads;       // face tasks beyond one per thread
constexpr int kPairs = kCells * kOcts;                 // (cell, oct) pairs
constexpr int kLoads = (kPairs + kThreads - 1) / kThreads;
constexpr int kCellStride = 5 * kOcts;                 // [cell][variable][oct]
constexpr int kFaceStride = 10 * kOcts;                // [face][left 5, right 5][oct]

// Stencil cell (i,j,k), each in -1..4, as an index.
constexpr int cell6(int i, int j, int k) { return (i + 1) + 6 * ((j + 1) + 6 * (k + 1)); }

// Traced cell c: 0..7 the oct's own, x fastest; then 8 + 8*d + 4*side + T the
// cells beyond its sides, T the position in the side, lower axis fastest.
// Face 12*d + 4*x + T: direction d, between the cells x and x+1 along it.
struct Tables {
  signed char slot[216];          // stencil cell -> 0..79, or -1 where no face needs it
  unsigned char cell[kCells];     // and back
  unsigned long long nbr[kTraced];  // slots of a traced cell and of its -x,+x,-y,+y,-z,+z neighbours, a byte each
  unsigned char side[kFaces][2];  // slots of a face's left and right cell
  unsigned char out[kFaces];      // a face's place in flux(1:3,1:3,1:3), (i-1)+3*((j-1)+3*(k-1))
  unsigned char order[27];        // neighbour octs i1+3*(j1+3*k1): centre and sides, then edges, then corners
  unsigned long long sub[27];     // slots of a neighbour oct's eight cells, a byte each, 255 for the unneeded
};

constexpr Tables make_tables() {
  Tables t{};
  int n = 0;
  for (int c = 0; c < 216; ++c) {
    const int x[3] = {c % 6 - 1, (c / 6) % 6 - 1, c / 36 - 1};
    int out = 0, edge = 0;
    for (int a = 0; a < 3; ++a) {
      if (x[a] < 1 || x[a] > 2) ++out;
      if (x[a] == 0 || x[a] == 3) ++edge;
    }
    const bool read = out <= 1 || (out == 2 && edge == 2);
    t.slot[c] = read ? (signed char)n : (signed char)-1;
    if (read) t.cell[n++] = (unsigned char)c;
  }
  for (int c = 0; c < kTraced; ++c) {
    int x[3] = {1 + (c & 1), 1 + ((c >> 1) & 1), 1 + (c >> 2)};
    if (c >= 8) {
      const int d = (c - 8) / 8, side = ((c - 8) / 4) % 2, T = c % 4;
      const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
      x[d] = side ? 3 : 0;
      x[t1] = 1 + (T & 1);
      x[t2] = 1 + (T >> 1);
    }
    t.nbr[c] = (unsigned long long)t.slot[cell6(x[0], x[1], x[2])];
    for (int a = 0; a < 3; ++a)
      for (int s = 0; s < 2; ++s) {
        int y[3] = {x[0], x[1], x[2]};
        y[a] += s ? 1 : -1;
        t.nbr[c] |= (unsigned long long)t.slot[cell6(y[0], y[1], y[2])] << 8 * (1 + 2 * a + s);
      }
  }
  for (int f = 0; f < kFaces; ++f) {
    const int d = f / 12, xf = (f / 4) % 3, T = f % 4;
    const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
    int x[3] = {0, 0, 0};
    x[t1] = 1 + (T & 1);
    x[t2] = 1 + (T >> 1);
    x[d] = xf;
    t.side[f][0] = (unsigned char)t.slot[cell6(x[0], x[1], x[2])];
    x[d] = xf + 1;
    t.side[f][1] = (unsigned char)t.slot[cell6(x[0], x[1], x[2])];
    t.out[f] = (unsigned char)((x[0] - 1) + 3 * ((x[1] - 1) + 3 * (x[2] - 1)));
  }
  int m = 0;
  for (int kind = 0; kind < 4; ++kind)  // neighbours off the centre along `kind` axes
    for (int j = 0; j < 27; ++j) {
      const int y[3] = {j % 3, (j / 3) % 3, j / 9};
      if ((y[0] != 1) + (y[1] != 1) + (y[2] != 1) == kind) t.order[m++] = (unsigned char)j;
      for (int s = 0; s < 8; ++s)
        t.sub[j] |= (unsigned long long)(unsigned char)t.slot[cell6(2 * y[0] - 1 + (s & 1), 2 * y[1] - 1 + ((s >> 1) & 1),
                                                                    2 * y[2] - 1 + (s >> 2))] << 8 * s;
    }
  return t;
}

constexpr Tables kHost = make_tables();
static_assert(kHost.slot[215] == -1 && kHost.cell[79] == 201, "80 stencil cells");
__constant__ Tables kTab = make_tables();

// The LDS of a workgroup: the primitives [cell][variable][oct], later the
// traced states [face][side][oct] (rotated: rho, normal velocity, pressure,
// two tangential velocities).
constexpr int kLds = kCells * kCellStride;
static_assert(kFaces * kFaceStride <= kLds, "the traced states fit over the primitives");

template <typename R>
__device__ __forceinline__ void put_prim(R* s, int e, const Prim<R>& q) {
  R* p = s + (e / kOcts) * kCellStride + e % kOcts;
  p[0] = q.r;
  p[kOcts] = q.u;
  p[2 * kOcts] = q.v;
  p[3 * kOcts] = q.w;
  p[4 * kOcts] = q.p;
}

template <typename R>
__device__ __forceinline__ Prim<R> get_prim(const R* s, int slot, int l) {
  const R* p = s + slot * kCellStride + l;
  return Prim<R>{p[0], p[kOcts], p[2 * kOcts], p[3 * kOcts], p[4 * kOcts]};
}

template <typename R>
__device__ __forceinline__ void put_side(R* s, int face, int side, int l, const Face<R>& f) {
  R* p = s + face * kFaceStride + side * 5 * kOcts + l;
  p[0] = f.r;
  p[kOcts] = f.un;
  p[2 * kOcts] = f.p;
  p[3 * kOcts] = f.ut1;
  p[4 * kOcts] = f.ut2;
}

template <typename R>
__device__ __forceinline__ Face<R> get_side(const R* s, int face, int side, int l) {
  const R* p = s + face * kFaceStride + side * 5 * kOcts + l;
  return Face<R>{p[0], p[kOcts], p[2 * kOcts], p[3 * kOcts], p[4 * kOcts]};
}

// Step 2: every thread t calls it, after the barrier that completes the
// primitives in s; returns after the barrier that completes the traced
// states.  dtdx: per direction.
template <typename R, int ST>
__device__ __forceinline__ void trace_tile(R* s, int t, const SolverConsts<R>& sc, const R dtdx[3]) {
  const int l = t % kOcts, c = t / kOcts;
  const int wave = __builtin_amdgcn_readfirstlane(t / 64);
  Prim<R> q, D[3];
  const unsigned long long nb = kTab.nbr[c];
  auto at = [&](int k) { return get_prim(s, (int)(nb >> 8 * k) & 255, l); };
  q = at(0);
#pragma unroll
  for (int a = 0; a < 3; ++a)
    D[a] = slope_prim<R, ST>(at(1 + 2 * a), q, at(2 + 2 * a), sc.slope_type, sc.theta);
  const Source<R> src = trace_sources<R, ST>(q, D[0], D[1], D[2], sc.gamma, sc.div_hi);
  if (wave < kOwnWaves) {  // own cells: every direction, both sides
    Prim<R> qp[3], qm[3];
#pragma unroll
    for (int d = 0; d < 3; ++d) trace_dir(q, D[d], src, dtdx[d], sc.smallr, qp[d], qm[d]);
    __syncthreads();
    const int x[3] = {c & 1, (c >> 1) & 1, c >> 2};
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int T = d == 0 ? x[1] + 2 * x[2] : (d == 1 ? x[0] + 2 * x[2] : x[0] + 2 * x[1]);
      put_side(s, 12 * d + 4 * x[d] + T, 1, l, rotate(qp[d], d));
      put_side(s, 12 * d + 4 * (x[d] + 1) + T, 0, l, rotate(qm[d], d));
    }
  } else {  // beyond a side: the state that faces the oct
    const int d = wave / kOwnWaves - 1, T = c % 4;
    const bool side = (c / 4) & 1;
    Face<R> f;
    auto toward = [&](auto dir) {
      constexpr int dd = decltype(dir)::value;
      Prim<R> qp, qm;
      trace_dir(q, D[dd], src, dtdx[dd], sc.smallr, qp, qm);
      const Face<R> fp = rotate(qp, dd), fm = rotate(qm, dd);
      f.r = side ? fp.r : fm.r;
      f.un = side ? fp.un : fm.un;
      f.p = side ? fp.p : fm.p;
      f.ut1 = side ? fp.ut1 : fm.ut1;
      f.ut2 = side ? fp.ut2 : fm.ut2;
    };
    if (d == 0) toward(std::integral_constant<int, 0>{});
    else if (d == 1) toward(std::integral_constant<int, 1>{});
    else toward(std::integral_constant<int, 2>{});
    __syncthreads();
    put_side(s, 12 * d + (side ? 8 : 0) + T, side, l, f);
  }
  __syncthreads();
}

// Step 3's tasks: the face of thread t's k-th task (k = 0, 1), or -1.
__device__ __forceinline__ int tile_face(int t, int k) {
  if (k == 0) return t / kOcts;
  return t >= kThreads - kRest ? (t + kRest) / kOcts : -1;
}
static_assert(kThreads % 64 == 0 && kRest % 64 == 0 && kRest > 0 && kRest <= kThreads, "whole wavefronts of faces");

}  // namespace oct_tile
}  // namespace ramses
