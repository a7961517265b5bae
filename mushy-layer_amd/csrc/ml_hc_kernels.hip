// ml_hc_kernels.hip — HIP kernels for gfx950 of the nonlinear (H, Theta)
// operator of AMRNonLinearMultiCompOp: fused closure + red/black smoothing,
// residual with max-norm, FAS restriction, operator application, and a
// single-workgroup kernel that runs the coarse part of a FAS V-cycle.
// Every kernel recomputes the phase-diagram closure from (H, Theta) staged
// in LDS, so theta/Theta_l are never written to HBM.
//
// Arithmetic follows the reference's evaluation order with contraction off
// (-ffp-contract=off), so the FP64 instantiation reproduces the CPU oracle
// bit for bit.
#include <hip/hip_ext.h>

#include <type_traits>

#include "ml_common.h"
#include "ml_kernels.h"
#include "ml_tile.h"

namespace ml {

namespace {

constexpr int kThreads = 256;
constexpr int kWGCells = 1024;   // largest level of the single-workgroup kernel

enum : int { kResid = 1, kApply = 2, kRestrict = 3 };

// Closure of every in-domain position within ext, then the derived-variable
// BC at wall ghosts within ext (computeDiffusedVar,
// src/AMRNonLinearMultiCompOp.cpp:57-98).
template <typename T, int DIM, int TX, int TY, int TZ>
__device__ inline void tile_diffused_var(const HCArgs<T>& A, const Tile<DIM, TX, TY, TZ>& t,
                                         const T* sphi, T* sphl, int ext, int homog) {
  const Geom& g = A.g;
  const int E = t.E;
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int ex, ey, ez;
    t.coords(e, ex, ey, ez);
    if (!t.within(ex, ey, ez, ext)) continue;
    const Pos P = t.pos(g, ex, ey, ez);
    if (P.kind != 1) continue;
    T th, cl;
    closure<T>(sphi[e], sphi[E + e], A.cp, th, cl);
    sphl[e] = th;
    sphl[E + e] = cl;
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int ex, ey, ez;
    t.coords(e, ex, ey, ez);
    if (!t.within(ex, ey, ez, ext)) continue;
    const Pos P = t.pos(g, ex, ey, ez);
    if (P.kind != 2) continue;
    const int stride = P.gd == 0 ? 1 : (P.gd == 1 ? t.EX : t.EXY);
    const int eint = P.gs == 0 ? e + stride : e - stride;
    const int isign = P.gs == 0 ? -1 : 1;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const T x1 = sphl[n * E + eint];
      T gv = x1;
      if (A.bc.apply) {
        const T v = homog ? T(0) : T(A.bc.val[P.gd][P.gs][n]);
        gv = bc_ghost<T>(A.bc.type[P.gd][P.gs][n], v, x1, isign, T(g.dx));
      }
      sphl[n * E + e] = gv;
    }
  }
  __syncthreads();
}

// ---------------------------------------------------------------------------
// 2D red/black relaxation over regions of 32 x 32 positions: the core of
// 32 - 2H cells a side that the workgroup owns and a halo of H cells (H = the
// colour passes, one more where a result of the relaxed state follows).  A
// pass updates one colour from the closure as of its start, frozen within it
// (levelGSRB, src/AMRNonLinearMultiCompOp.cpp:815-949, and NONLINEARSMOOTHING,
// src/AMRNonLinearMultiCompOpF.ChF:125-195).
//
// A pass is bound by its chain of some 170 FP64 instructions (stencil and
// closure), so no lane may idle in it: each of the 512 threads holds the two
// cells of an x pair, one of each colour (slot m: the cell of parity m), and
// a pass runs one slot with every lane at work, where one cell per lane
// leaves half of them waiting.  State, closure, right-hand side, lambda and
// faces of both cells stay in registers; LDS holds only the closure, which
// the neighbours read (16 KB).  Rows are 256 B apart and a row's active cells
// alternate with the next row's, so the 32 lanes of an 8-byte LDS access
// cover every bank once.
//
// What a launch costs besides its passes is fetching its code and arguments,
// both cold: so the arguments are one small struct (not the operator's
// geometry), the tile is the 2D workgroup index (no divisions), the faces,
// right-hand side and state of a pair come as 16-byte loads with 32-bit
// offsets, and the closure of the incoming state is one loop for both cells.
//
//   RB_PLAIN     the relaxed state
//   RB_RESTRICT  ... and the FAS restriction of its residual and itself
//   RB_NORM      ... and the max-norm of its residual with the stopping rule
// With rhs_out the right-hand side first receives L(phi) of the incoming
// state.  Measured (events around the launch, 256^2 mushy state): 8 passes
// 14.4 us, 21.2 us with one cell per lane (32x8 tiles, 512 threads); at 512^2
// 34.7 against 74.3 us; on the way down one launch of 10.5 us replaces
// relaxation, restriction and operator (9.0 + 7.3 + 8.4 us).
//
// GEN: any grid -- a periodic length below 32 or odd, arrays beyond 32-bit
// byte offsets.  Equal colours meet at the seam of an odd length.  A region
// that holds it reads a pass's neighbours as of its start (the new closures
// are stored after a barrier), and along x it starts one cell earlier where
// that keeps the seam from falling inside a pair, whose cells would share a
// slot's turn; its core is narrower for that (pair_core_x).  Only on very short
// rows, where a region holds several seams, a pass looks at both slots.  One
// sweep of 129 x 128 8.1 us, of 257 x 256 8.3 (11.4 and 11.3 with both slots
// everywhere; 7.5 and 7.9 with even lengths), of 23 x 500 8.6 (11.1), of
// 17 x 500, with both, 12; four sweeps of 385 x 384 28.7 us (34.7; even 24.3).
enum : int { RB_PLAIN = 0, RB_RESTRICT = 1, RB_NORM = 2 };
constexpr int kRB = 32;            // positions per side
constexpr int kRBThreads = kRB * kRB / 2;
// Core cells along x.  With an odd periodic length the core and its halo are no
// wider than the row, so that they hold one seam at most, and leave a column for
// the shift off it; where that would more than halve the core (rows below 18
// cells in a sweep, 24 in four) the core stays whole and `both` is set.
__host__ __device__ inline int pair_core_x(int nx, int per0, int H, bool* both) {
  const int whole = kRB - 2 * H;
  *both = false;
  if (!per0 || !(nx & 1)) return whole;
  const int w = (nx < kRB - 2 ? nx : kRB - 2) - 2 * H;
  *both = 2 * w < whole;
  return *both ? whole : w & ~1;
}

template <typename T>
struct PairArgs {
  const int* skip;
  const T *phi, *rhs, *b0, *b1, *a;    // a nullable
  int nx, ny, sy, npass, first, per0, per1, ntx;
  unsigned ncell;
  long long nf0, nf1;
  T alpha, beta, dxinv;
  T *phi_out, *rhs_out;
  const T *pc, *pc0;                   // prolongation source (nullable)
  T *out, *phic, *phic0;
  int cnx, cny, csy;                   // the coarse level of pc or of out
  unsigned cncell;
  unsigned long long* norm;
  CtlFuse fuse;
  ClosureP<T> cp;
  T gs[2][2][2], gb[2][2][2];          // GhostForm
};

// linear prolongation (prolong_value) of the correction pc - pc0 to fine cell
// (i, j); the outer coarse neighbour is at most one cell beyond the coarse
// level, so it wraps or clamps without a division
template <typename T, typename Off>
__device__ __forceinline__ void prolong_pair2(const PairArgs<T>& A, int i, int j, T* p) {
  constexpr T fx1 = T(3) / T(16), fx2 = T(9) / T(16), f0 = T(1) / T(16);
  const int ic = i >> 1, jc = j >> 1;
  int X1 = ic + ((i & 1) ? 1 : -1), Y1 = jc + ((j & 1) ? 1 : -1);
  if (X1 < 0) X1 = A.per0 ? A.cnx - 1 : 0;
  if (X1 >= A.cnx) X1 = A.per0 ? 0 : A.cnx - 1;
  if (Y1 < 0) Y1 = A.per1 ? A.cny - 1 : 0;
  if (Y1 >= A.cny) Y1 = A.per1 ? 0 : A.cny - 1;
  const Off r0 = Off(1) + Off(A.csy) * Off(jc + 1), r1 = Off(1) + Off(A.csy) * Off(Y1 + 1);
  const Off q[4] = {(r0 + Off(ic)) * Off(sizeof(T)), (r1 + Off(X1)) * Off(sizeof(T)), (r0 + Off(X1)) * Off(sizeof(T)),
                    (r1 + Off(ic)) * Off(sizeof(T))};
  auto ld = [](const T* b, Off o) { return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(b) + o); };
  T v[2][4];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int c = 0; c < 4; ++c) v[n][c] = ld(A.pc + (n ? A.cncell : 0u), q[c]);
  if (A.pc0) {
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int c = 0; c < 4; ++c) v[n][c] = v[n][c] - ld(A.pc0 + (n ? A.cncell : 0u), q[c]);
  }
#pragma unroll
  for (int n = 0; n < 2; ++n) {
    p[n] = p[n] + fx2 * v[n][0] + f0 * v[n][1];
    p[n] = p[n] + fx1 * (v[n][2] + v[n][3]);
  }
}

// two values at any 8-byte alignment in one load
typedef double dbl2u __attribute__((ext_vector_type(2), aligned(8)));

template <typename T, int MODE, bool GEN>
__global__ __launch_bounds__(kRBThreads, 4) void hc_relax_pair_kernel(PairArgs<T> A) {
  using Off = typename std::conditional<GEN, unsigned long long, unsigned>::type;
  constexpr int NP = kRB * kRB;
  constexpr Off W = sizeof(T);
  __shared__ T sl[2 * NP];                                  // closure
  __shared__ T sr[MODE == RB_RESTRICT ? 2 * NP : 1];        // restriction scratch
  const int nx = A.nx, ny = A.ny, npass = A.npass;
  const int H = npass + (MODE == RB_PLAIN ? 0 : 1);
  const int core = kRB - 2 * H;
  // GEN: both slots in every pass
  bool both = false;
  const int corex = GEN ? pair_core_x(nx, A.per0, H, &both) : core;
  // GEN: the workgroups of all tiles in one dimension
  const int by = GEN ? int(blockIdx.x / unsigned(A.ntx)) : int(blockIdx.y);
  const int bx = GEN ? int(blockIdx.x) - by * A.ntx : int(blockIdx.x);
  const int x0 = bx * corex, y0 = by * core;
  const int ey = threadIdx.x >> 4, ex0 = 2 * (threadIdx.x & 15);
  const bool per0 = A.per0 != 0, per1 = A.per1 != 0;
  // GEN: the core and its halo hold the seam of an odd length (careful); the
  // pairs' shift against it
  bool careful = false;
  int sh = 0;
  if constexpr (GEN) {
    if (per0 && (nx & 1)) {
      const int at = x0 < H ? H - x0 : nx - (x0 - H);   // the seam, from the halo's first cell
      careful = both || at < corex + 2 * H;
      sh = !both && careful ? at & 1 : 0;
    }
    if (per1 && (ny & 1)) careful = careful || ny < kRB || y0 < H || ny - (y0 - H) < kRB;
  }
  const int Hx = H + sh;   // the core's first column in the region
  const int ux0 = x0 - Hx + ex0, uy = y0 - H + ey;
  auto wrap = [](int v, int n) {
    if (GEN) {
      v %= n;
      return v < 0 ? v + n : v;
    }
    return v < 0 ? v + n : (v >= n ? v - n : v);   // n >= 32: at most one length away
  };
  const bool iny = uy >= 0 && uy < ny;
  const bool oky = iny || per1;
  const int gj = oky ? wrap(uy, ny) : 0;
  // distance from the core
  auto beyond = [&](int e, int lo0, int n) {
    const int lo = lo0 - e, hi = e - (lo0 + n) + 1;
    const int d = lo > hi ? lo : hi;
    return d > 0 ? d : 0;
  };
  const int dy = beyond(ey, H, core);
  const int wy = per1 ? 0 : ((gj == 0 ? 4 : 0) | (gj == ny - 1 ? 8 : 0));
  // cells of the pair in x order: c = 0, 1; slot m holds cell m ^ swap
  const bool in0 = ux0 >= 0 && ux0 < nx, in1 = ux0 >= -1 && ux0 + 1 < nx;
  const bool near = !GEN || ex0 < Hx + corex + H;   // (columns beyond the halo: a narrow core leaves some)
  const bool ok0 = near && oky && (in0 || per0), ok1 = near && oky && (in1 || per0);
  const int gx0 = ok0 ? wrap(ux0, nx) : 0, gx1 = ok1 ? wrap(ux0 + 1, nx) : 0;
  // parity of the pair's first cell
  const int swap = (GEN ? (per0 ? gx0 : ux0) + gj : ux0 + uy) & 1;
  const Off row = Off(A.sy) * Off(gj + 1) + Off(1);
  const Off q0 = (row + Off(gx0)) * W, q1 = (row + Off(gx1)) * W;   // byte offsets

  auto ld = [](const T* b, Off o) { return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(b) + o); };
  T ph[2][2], rr[2][2], aa[2][2], lam[2][2], pl[2][2];
  CellFaces<T, 2> F[2];
  const Off fx0 = (Off(gx0) + Off(nx + 1) * Off(gj)) * W, fx1 = (Off(gx1) + Off(nx + 1) * Off(gj)) * W;
  const Off fy0 = (Off(gx0) + Off(nx) * Off(gj)) * W, fy1 = (Off(gx1) + Off(nx) * Off(gj)) * W;
  if (ok0 && ok1 && gx1 == gx0 + 1) {
    auto ld2 = [](const T* b, Off o) { return *reinterpret_cast<const dbl2u*>(reinterpret_cast<const char*>(b) + o); };
    dbl2u vp[2], vr[2], vx[2], vl[2], vh[2];
    T vz[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) vp[n] = ld2(A.phi + (n ? A.ncell : 0u), q0);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      vr[n] = ld2(A.rhs + (n ? A.ncell : 0u), q0);
      const T *bx = A.b0 + (n ? A.nf0 : 0), *by = A.b1 + (n ? A.nf1 : 0);
      vx[n] = ld2(bx, fx0);
      vz[n] = ld(bx + 2, fx0);
      vl[n] = ld2(by, fy0);
      vh[n] = ld2(by + nx, fy0);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const bool second = (m ^ swap) != 0;
        ph[m][n] = second ? vp[n].y : vp[n].x;
        rr[m][n] = second ? vr[n].y : vr[n].x;
        F[m].v[n][0] = second ? vx[n].y : vx[n].x;
        F[m].v[n][1] = second ? vz[n] : vx[n].y;
        F[m].v[n][2] = second ? vl[n].y : vl[n].x;
        F[m].v[n][3] = second ? vh[n].y : vh[n].x;
      }
  } else {
    // a pair across the periodic seam or beside a wall
#pragma unroll 1
    for (int m = 0; m < 2; ++m) {
      const bool second = (m ^ swap) != 0;
      if (!(second ? ok1 : ok0)) continue;
      const Off qm = second ? q1 : q0, fx = second ? fx1 : fx0, fy = second ? fy1 : fy0;
      T v[2][6];
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const T *bx = A.b0 + (n ? A.nf0 : 0), *by = A.b1 + (n ? A.nf1 : 0);
        v[n][0] = ld(A.phi + (n ? A.ncell : 0u), qm);
        v[n][1] = ld(A.rhs + (n ? A.ncell : 0u), qm);
        v[n][2] = ld(bx, fx);
        v[n][3] = ld(bx + 1, fx);
        v[n][4] = ld(by, fy);
        v[n][5] = ld(by + nx, fy);
      }
      auto take = [&](int k) __attribute__((always_inline)) {
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          ph[k][n] = v[n][0];
          rr[k][n] = v[n][1];
#pragma unroll
          for (int f = 0; f < 4; ++f) F[k].v[n][f] = v[n][2 + f];
        }
      };
      if (m == 0)
        take(0);
      else
        take(1);
    }
  }
  // (the loads above are in bounds in any case)
  if (A.skip && *A.skip) return;
  int e[2], lim[2], gi[2], wall[2];
  Off q[2];
  bool cell[2], owner[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const bool second = (m ^ swap) != 0;
    const int ex = ex0 + (second ? 1 : 0);
    e[m] = ey * kRB + ex;
    cell[m] = second ? ok1 : ok0;
    gi[m] = second ? gx1 : gx0;
    q[m] = second ? q1 : q0;
    const int dx = beyond(ex, Hx, corex);
    const int dist = dx > dy ? dx : dy;
    owner[m] = (second ? in1 : in0) && iny && dist == 0;
    lim[m] = cell[m] ? H - 1 - dist : -1;   // last pass that updates the cell
    wall[m] = wy | (per0 ? 0 : ((gi[m] == 0 ? 1 : 0) | (gi[m] == nx - 1 ? 2 : 0)));
    aa[m][0] = aa[m][1] = T(1);
    if (A.a && cell[m]) {
      aa[m][0] = ld(A.a, q[m]);
      aa[m][1] = ld(A.a + A.ncell, q[m]);
    }
  }
  if (A.pc) {
#pragma unroll 1
    for (int m = 0; m < 2; ++m) {
      if (!(m ? cell[1] : cell[0])) continue;
      T v[2] = {m ? ph[1][0] : ph[0][0], m ? ph[1][1] : ph[0][1]};
      prolong_pair2<T, Off>(A, m ? gi[1] : gi[0], gj, v);
      if (m == 0) {
        ph[0][0] = v[0];
        ph[0][1] = v[1];
      } else {
        ph[1][0] = v[0];
        ph[1][1] = v[1];
      }
    }
  }
  // one copy of the closure for both cells
#pragma unroll 1
  for (int m = 0; m < 2; ++m) {
    T th, cl;
    closure<T>(m ? ph[1][0] : ph[0][0], m ? ph[1][1] : ph[0][1], A.cp, th, cl);
    if (m ? cell[1] : cell[0]) {
      sl[m ? e[1] : e[0]] = th;
      sl[NP + (m ? e[1] : e[0])] = cl;
    }
    if (m == 0) {
      pl[0][0] = th;
      pl[0][1] = cl;
    } else {
      pl[1][0] = th;
      pl[1][1] = cl;
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    lam[m][0] = lambda_of<T, 2>(F[m], 0, aa[m][0], A.alpha, A.beta, A.dxinv);
    lam[m][1] = lambda_of<T, 2>(F[m], 1, aa[m][1], A.alpha, A.beta, A.dxinv);
  }
  __syncthreads();
  // L(phi) of slot m; a neighbour beyond a wall is the ghost of the cell's
  // own closure (computeDiffusedVar's BC)
  auto lof = [&](auto M, T(&out)[2]) __attribute__((always_inline)) {
    constexpr int m = decltype(M)::value;
    T st[2][5];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const T* s = sl + n * NP + e[m];
      st[n][0] = pl[m][n];
      st[n][1] = s[1];
      st[n][2] = s[-1];
      st[n][3] = s[kRB];
      st[n][4] = s[-kRB];
    }
    if (wall[m]) {
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const int k = 1 + 2 * (f >> 1) + (1 - (f & 1));
          const T gh = fma(A.gs[f >> 1][f & 1][n], st[n][0], A.gb[f >> 1][f & 1][n]);
          st[n][k] = ((wall[m] >> f) & 1) ? gh : st[n][k];
        }
    }
#pragma unroll
    for (int n = 0; n < 2; ++n)
      out[n] = lof_of<T, 2>(F[m], n, st[n], aa[m][n], ph[m][n], A.alpha, A.beta, A.dxinv);
  };
  auto st = [](T* b, Off o, T v) { *reinterpret_cast<T*>(reinterpret_cast<char*>(b) + o) = v; };
  if (A.rhs_out) {
    auto add = [&](auto M) __attribute__((always_inline)) {
      constexpr int m = decltype(M)::value;
      if (lim[m] < 0) return;
      T lf[2];
      lof(M, lf);
      rr[m][0] = rr[m][0] + lf[0];
      rr[m][1] = rr[m][1] + lf[1];
      if (owner[m]) {
        st(A.rhs_out, q[m], rr[m][0]);
        st(A.rhs_out + A.ncell, q[m], rr[m][1]);
      }
    };
    add(IC<0>{});
    add(IC<1>{});
    __syncthreads();   // the passes below overwrite the closure just read
  }
  auto runs = [&](int m, int p, int colour) {
    return p <= lim[m] && (!GEN || ((gi[m] + gj) & 1) == colour);
  };
  auto put = [&](int m) __attribute__((always_inline)) {
    sl[e[m]] = pl[m][0];
    sl[NP + e[m]] = pl[m][1];
  };
  auto update = [&](auto M, int p, int colour) __attribute__((always_inline)) {
    constexpr int m = decltype(M)::value;
    if (!runs(m, p, colour)) return;
    T lf[2];
    lof(M, lf);
#pragma unroll
    for (int n = 0; n < 2; ++n) ph[m][n] = ph[m][n] - lam[m][n] * (lf[n] - rr[m][n]);
    closure<T>(ph[m][0], ph[m][1], A.cp, pl[m][0], pl[m][1]);
    if (!GEN || !careful) put(m);
  };
#pragma unroll 1
  for (int p = 0; p < npass; ++p) {
    const int colour = (A.first + p) & 1;
    if (both || colour == 0) update(IC<0>{}, p, colour);
    if (both || colour == 1) update(IC<1>{}, p, colour);
    if (careful) {
      __syncthreads();
      if ((both || colour == 0) && runs(0, p, colour)) put(0);
      if ((both || colour == 1) && runs(1, p, colour)) put(1);
    }
    __syncthreads();
  }
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    if (!owner[m]) continue;
    st(A.phi_out, q[m], ph[m][0]);
    st(A.phi_out + A.ncell, q[m], ph[m][1]);
  }
  if constexpr (MODE == RB_NORM) {
    T mx = T(0);
    int nan = 0;
    auto res = [&](auto M) __attribute__((always_inline)) {
      constexpr int m = decltype(M)::value;
      if (!owner[m]) return;
      T lf[2];
      lof(M, lf);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const T ar = fabs(rr[m][n] - lf[n]);
        if (ar != ar) nan = 1;
        else if (ar > mx) mx = ar;
      }
    };
    res(IC<0>{});
    res(IC<1>{});
    block_max_atomic<T>(mx, nan, A.norm, A.fuse);
  }
  if constexpr (MODE == RB_RESTRICT) {
    // RESTRICTRESNLVC / RESTRICT (src/AMRNonLinearMultiCompOpF.ChF:452-585):
    // (rhs - L phi)/4 and phi/4 per fine cell, child sums in Fortran order
    T tr[2][2];
    auto res = [&](auto M) __attribute__((always_inline)) {
      constexpr int m = decltype(M)::value;
      if (!owner[m]) return;
      T lf[2];
      lof(M, lf);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        tr[m][n] = (rr[m][n] - lf[n]) / T(4);
        sr[n * NP + e[m]] = ph[m][n] / T(4);
      }
    };
    res(IC<0>{});
    res(IC<1>{});
    __syncthreads();   // every closure has been read
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      if (!owner[m]) continue;
      sl[e[m]] = tr[m][0];
      sl[NP + e[m]] = tr[m][1];
    }
    __syncthreads();
    // coarse cells of the core (at most 13 a side), 16 threads a row
    const int cy = threadIdx.x >> 4, cx = threadIdx.x & 15;
    const int I = x0 / 2 + cx, J = y0 / 2 + cy;
    if (cx >= corex / 2 || cy >= core / 2 || I >= A.cnx || J >= A.cny) return;
    const Off qc = (Off(I + 1) + Off(A.csy) * Off(J + 1)) * W;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      T s = T(0), sp = T(0);
#pragma unroll
      for (int jj = 0; jj < 2; ++jj)
#pragma unroll
        for (int ii = 0; ii < 2; ++ii) {
          const int f = n * NP + (2 * cy + jj + H) * kRB + 2 * cx + ii + Hx;
          s = s + sl[f];
          sp = sp + sr[f];
        }
      st(A.out + (n ? A.cncell : 0u), qc, s);
      st(A.phic + (n ? A.cncell : 0u), qc, sp);
      st(A.phic0 + (n ? A.cncell : 0u), qc, sp);
    }
  }
}

// Residual (with max-norm), operator application, and FAS restriction of
// one tile with a one-cell halo.
template <typename T, int DIM, int TX, int TY, int TZ, int MODE>
__device__ __forceinline__ void hc_tile_body(const HCArgs<T>& A, const TileIO<T>& io, int tile) {
  if (A.skip && *A.skip) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const Geom& g = A.g;
  Tile<DIM, TX, TY, TZ> t;
  t.init_at(1, io.ntx, io.nty, tile);
  const int E = t.E;
  T* sphi = reinterpret_cast<T*>(smem_raw);
  T* sphl = sphi + 2 * E;
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));

  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    int ex, ey, ez;
    t.coords(e, ex, ey, ez);
    const Pos P = t.pos(g, ex, ey, ez);
    if (P.kind == 1) {
      const long long q = g.ci(P.i, P.j, P.k);
      sphi[e] = io.phi[q];
      sphi[E + e] = io.phi[q + g.ncell];
    }
  }
  __syncthreads();
  tile_diffused_var<T, DIM, TX, TY, TZ>(A, t, sphi, sphl, 1, io.homog);

  if (MODE == kResid || MODE == kApply) {
    T mx = T(0);
    int nan = 0;
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
      int ex, ey, ez;
      t.coords(e, ex, ey, ez);
      if (!t.within(ex, ey, ez, 0)) continue;
      const int gi = t.x0 - t.H + ex, gj = t.y0 - t.H + ey, gk = DIM == 3 ? t.z0 - t.H + ez : 0;
      if (gi >= g.n[0] || gj >= g.n[1] || (DIM == 3 && gk >= g.n[2])) continue;
      const long long q0 = g.ci(gi, gj, gk);
      CellFaces<T, DIM> F;
      load_faces<T, DIM>(A, gi, gj, gk, F);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const long long q = q0 + n * g.ncell;
        T st[7];
        gather_lds<T, DIM>(sphl + n * E, e, t.EX, t.EXY, st);
        const T aq = A.a ? A.a[q] : T(1);
        const T lof = lof_of<T, DIM>(F, n, st, aq, sphi[n * E + e], A.alpha, A.beta, dxinv);
        if (MODE == kResid) {
          const T r = io.rhs[q] - lof;
          if (io.out) io.out[q] = r;
          const T ar = fabs(r);
          if (ar != ar) nan = 1;
          else if (ar > mx) mx = ar;
        } else {
          io.out[q] = io.add ? io.add[q] + lof : lof;
        }
      }
    }
    if (MODE == kResid && io.norm) block_max_atomic<T>(mx, nan, io.norm, io.fuse);
    return;
  }

  if (MODE == kRestrict) {
    // RESTRICTRESNLVC (src/AMRNonLinearMultiCompOpF.ChF:452-542):
    // res_c(i/2) = 0 + sum over children in Fortran order of (rhs - L phi)/2^d;
    // with io.phic also RESTRICT (:555-585) of the state into phic/phic0.
    T* sres = sphl + 2 * E;
    constexpr int NC = TX * TY * (DIM == 3 ? TZ : 1);
    const T denom = DIM == 3 ? T(8) : T(4);
    const Geom gc = io.gc;
    for (int c = threadIdx.x; c < NC; c += blockDim.x) {
      const int cx = c % TX, cr = c / TX, cy = cr % TY, cz = cr / TY;
      const int gi = t.x0 + cx, gj = t.y0 + cy, gk = DIM == 3 ? t.z0 + cz : 0;
      if (gi >= g.n[0] || gj >= g.n[1] || (DIM == 3 && gk >= g.n[2])) continue;
      const int e = (cx + t.H) + t.EX * (cy + t.H) + t.EXY * (DIM == 3 ? cz + t.H : 0);
      const long long q0 = g.ci(gi, gj, gk);
      CellFaces<T, DIM> F;
      load_faces<T, DIM>(A, gi, gj, gk, F);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        const long long q = q0 + n * g.ncell;
        T st[7];
        gather_lds<T, DIM>(sphl + n * E, e, t.EX, t.EXY, st);
        const T aq = A.a ? A.a[q] : T(1);
        const T lof = lof_of<T, DIM>(F, n, st, aq, sphi[n * E + e], A.alpha, A.beta, dxinv);
        sres[n * NC + c] = (io.rhs[q] - lof) / denom;
      }
    }
    __syncthreads();
    constexpr int CX = TX / 2, CY = TY / 2, CZ = DIM == 3 ? TZ / 2 : 1;
    constexpr int NCC = CX * CY * CZ;
    for (int c = threadIdx.x; c < NCC; c += blockDim.x) {
      const int cx = c % CX, cr = c / CX, cy = cr % CY, cz = cr / CY;
      const int I = t.x0 / 2 + cx, J = t.y0 / 2 + cy, K = DIM == 3 ? t.z0 / 2 + cz : 0;
      if (I >= gc.n[0] || J >= gc.n[1] || (DIM == 3 && K >= gc.n[2])) continue;
      const long long qc = gc.ci(I, J, K);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        T s = T(0), sp = T(0);
        for (int kk = 0; kk < (DIM == 3 ? 2 : 1); ++kk)
          for (int jj = 0; jj < 2; ++jj)
            for (int ii = 0; ii < 2; ++ii) {
              const int f = (2 * cx + ii) + TX * ((2 * cy + jj) + TY * (DIM == 3 ? 2 * cz + kk : 0));
              s = s + sres[n * NC + f];
              const int e = (2 * cx + ii + t.H) + t.EX * (2 * cy + jj + t.H) +
                            t.EXY * (DIM == 3 ? 2 * cz + kk + t.H : 0);
              sp = sp + sphi[n * E + e] / denom;
            }
        io.out[qc + n * gc.ncell] = s;
        if (io.phic) {
          io.phic[qc + n * gc.ncell] = sp;
          io.phic0[qc + n * gc.ncell] = sp;
        }
      }
    }
  }
}

template <typename T, int DIM, int TX, int TY, int TZ, int MODE>
__global__ __launch_bounds__(kThreads) void hc_tile_kernel(HCArgs<T> A, TileIO<T> io) {
  hc_tile_body<T, DIM, TX, TY, TZ, MODE>(A, io, int(blockIdx.x));
}

// batched operator applications: workgroup w applies tile map[w] & mask of job map[w] >> bits
template <typename T, int DIM, int TX, int TY, int TZ>
__global__ __launch_bounds__(kThreads) void hc_apply_batch_kernel(const HCApplyJob<T>* __restrict__ jobs,
                                                                  const unsigned* __restrict__ map) {
  const unsigned w = map[blockIdx.x];
  const HCApplyJob<T>& J = jobs[w >> kBatchTileBits];
  hc_tile_body<T, DIM, TX, TY, TZ, kApply>(J.A, J.io, int(w & kBatchTileMask));
}

// ---------------------------------------------------------------------------
// Single-workgroup FAS V-cycle over the small levels (at most kWGCells cells
// and everything below).  All levels' state, right-hand side, initial state,
// lambda and faces live in LDS for the whole cycle (hc_coarse_lds_bytes; the
// faces come as one contiguous block), so a level visit waits for no global
// memory.
//
// A wavefront alone on its SIMD issues an operation every 8 cycles whether it
// depends on the last one or not, and a branch costs four of them: the count
// of instructions along a visit is what bounds it.  So each thread owns one
// cell of each colour (an x pair; cells t and t + 512 where rows are odd)
// with its faces, lambda, state and closure in registers; a wall's ghost is
// written by its cell's owner with each update, into a slot that the stencil
// reads like any neighbour; offsets come from the host; nothing is divided.
// Levels whose pairs fit one wavefront are visited by wave 0 alone with
// wavefront-scope syncs.  The visits are one runtime loop: every launch
// fetches the code it runs.  Measured at 256^2 (levels 32^2 to 2^2): 65 us a
// launch, 84 us with one cell per lane and the levels' data in global memory;
// 3D (12x8x6 down) 87 against 180 us.
//
// A pass updates one colour and recomputes the closure of exactly the cells
// it updated (the other colour's is unchanged since its own update).  The
// bottom relaxation ends after the first red/black iteration that leaves
// every cell's state unchanged to the bit: each later one would repeat it.
constexpr int kHCWG = 512;

// linear prolongation from LDS: e(x, y, z) the coarse correction
template <typename T, int DIM, class E>
__device__ __forceinline__ T prolong_lds(const int* nc, const int* per, int i, int j, int k, E e, T p) {
  const T den = T(1) / (DIM == 3 ? T(64) : T(16));
  const T fx1 = T(3) * den, fx2 = T(9) * den, fx3 = T(27) * den, f0 = T(1) * den;
  auto outer = [&](int v, int d) {
    const int c = v >> 1, o = c + ((v & 1) ? 1 : -1), n = nc[d];
    return o < 0 ? (per[d] ? n - 1 : 0) : (o >= n ? (per[d] ? 0 : n - 1) : o);
  };
  const int X0 = i >> 1, Y0 = j >> 1, Z0 = DIM == 3 ? k >> 1 : 0;
  const int X1 = outer(i, 0), Y1 = outer(j, 1), Z1 = DIM == 3 ? outer(k, 2) : 0;
  if (DIM == 2) {
    p = p + fx2 * e(X0, Y0, 0) + f0 * e(X1, Y1, 0);
    p = p + fx1 * (e(X1, Y0, 0) + e(X0, Y1, 0));
  } else {
    p = p + fx3 * e(X0, Y0, Z0) + f0 * e(X1, Y1, Z1);
    p = p + fx2 * (e(X1, Y0, Z0) + e(X0, Y1, Z0) + e(X0, Y0, Z1));
    p = p + fx1 * (e(X1, Y1, Z0) + e(X0, Y1, Z1) + e(X1, Y0, Z1));
  }
  return p;
}

template <typename T, int DIM>
__global__ __launch_bounds__(kHCWG) void hc_coarse_vcycle_kernel(HCCoarse<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  typedef T vec2 __attribute__((ext_vector_type(2)));
  const int tid = threadIdx.x;
  const int nl = A.nl, tot = A.tot, N0 = A.off[1], tot1 = tot - N0;
  T* P = reinterpret_cast<T*>(smem_raw);   // state [2][tot]
  T* R = P + 2 * tot;                       // right-hand side [2][tot]
  T* P0 = R + 2 * tot;                      // initial state of the levels below the first [2][tot1]
  T* SL = P0 + 2 * tot1;                    // closure of the level [2][kWGCells], then ...
  constexpr int CS = kWGCells;              // (component stride of both)
  T* SX = SL + 2 * CS;                      // ... wall ghosts of the owners' cells, or the restriction terms
  T* FC = SX + 2 * CS;                      // faces, as the block holds them
  T* LM = FC + A.nfaces;                    // lambda [2][tot], kept for the way up (nl > 1)
  // ghost rule of every wall face f = 2d + s on the first level: s, b per
  // component; one more entry of zeros for cells without a wall
  __shared__ T GT[2 * DIM + 1][4];
  // first level's state and right-hand side, and the faces: loads first
  const long long sy = A.n[0] + 2, sz = sy * (A.n[1] + 2), nc0 = sz * (DIM == 3 ? A.n[2] + 2 : 1);
  auto level_of = [&](int l) __attribute__((always_inline)) {
    CLev L;
    for (int d = 0; d < 3; ++d) L.n[d] = d < DIM ? A.n[d] >> l : 1;
    L.nx = L.n[0];
    L.nxy = L.n[0] * L.n[1];
    L.off = A.off[l];
    L.N = A.off[l + 1] - L.off;
    return L;
  };
  const CLev L0 = level_of(0);
#pragma unroll
  for (int f = 0; f <= 2 * DIM; ++f)
    if (tid == f) {
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        GT[f][2 * n] = f < 2 * DIM ? A.gs[f >> 1][f & 1][n] : T(0);
        GT[f][2 * n + 1] = f < 2 * DIM ? A.gb[f >> 1][f & 1][n] : T(0);
      }
    }
  long long q0[2];
  T h0[2][2], r0[2][2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int c = tid + m * kHCWG;
    if (c >= N0) continue;
    int i, j, k;
    clev_coords(L0, c, i, j, k);
    q0[m] = (i + 1) + sy * (j + 1) + (DIM == 3 ? sz * (k + 1) : 0);
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      h0[m][n] = A.phi[q0[m] + n * nc0];
      r0[m][n] = A.rhs[q0[m] + n * nc0];
    }
  }
  {
    constexpr int KF = 6;
    const vec2* src = reinterpret_cast<const vec2*>(A.faces);
    vec2* dst = reinterpret_cast<vec2*>(FC);
    const int n2 = A.nfaces >> 1;
#pragma unroll 1
    for (int base = tid; base < n2; base += KF * kHCWG) {
      vec2 v[KF];
#pragma unroll
      for (int k = 0; k < KF; ++k)
        if (base + k * kHCWG < n2) v[k] = src[base + k * kHCWG];
#pragma unroll
      for (int k = 0; k < KF; ++k)
        if (base + k * kHCWG < n2) dst[base + k * kHCWG] = v[k];
    }
  }
  if (A.skip && *A.skip) return;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int c = tid + m * kHCWG;
    if (c >= N0) continue;
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      P[n * tot + c] = h0[m][n];
      R[n * tot + c] = r0[m][n];
    }
  }
  __syncthreads();
  const T rdenom = DIM == 3 ? T(0.125) : T(0.25);   // (a division by 2^d is this product)

#pragma unroll 1
  for (int v = 0; v < 2 * nl - 1; ++v) {
    const bool up = v >= nl, bot = v == nl - 1, down = v < nl - 1;
    const int l = up ? 2 * nl - 2 - v : v;
    const CLev L = level_of(l);
    const int off = L.off, offc = off + L.N;
    const bool even = (L.nx & 1) == 0;
    const bool small = cown_active<kHCWG>(L) <= 64;
    const int step = small ? 64 : kHCWG;   // threads of this visit
    const T lsc = T(1 << l);
    const T dx = A.dx * lsc;
    const T dxinv = T(1) / (dx * dx);
    auto sync = [&]() __attribute__((always_inline)) {
      if (small)
        wave_sync();
      else
        __syncthreads();
    };
    int fo[DIM], nf[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      fo[d] = A.fo[l][d];
      nf[d] = A.nf[l][d];
    }
    if (!small || tid < 64) {
      // state (on the way up with the prolonged correction) and closure, one
      // cell per thread
#pragma unroll 1
      for (int c = tid; c < L.N; c += step) {
        T ph[2] = {P[off + c], P[tot + off + c]};
        if (up) {
          int i, j, k;
          clev_coords(L, c, i, j, k);
          const int nc[3] = {L.n[0] >> 1, L.n[1] >> 1, L.n[2] >> 1};
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const T* pc = P + n * tot + offc;
            const T* p0 = P0 + n * tot1 + (offc - N0);
            auto e = [&](int x, int y, int z) -> T {
              const int q = x + nc[0] * (y + nc[1] * z);
              return pc[q] - p0[q];
            };
            ph[n] = prolong_lds<T, DIM>(nc, A.per, i, j, k, e, ph[n]);
            P[n * tot + off + c] = ph[n];
          }
        }
        T th, cl;
        closure<T>(ph[0], ph[1], A.cp, th, cl);
        SL[c] = th;
        SL[CS + c] = cl;
      }
      sync();
      // the thread's cell of each colour: neighbours, faces, lambda, right-
      // hand side, state, closure
      COwn o;
      cown_set<kHCWG>(L, o);
      int c[2], nb[2][2 * DIM], col[2], wall[2];
      bool multi[2] = {false, false};
      CellFaces<T, DIM> F[2];
      T ph[2][2], pl[2][2], rr[2][2], aa[2][2], lam[2][2], ws[2][2], wb[2][2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        c[m] = 0;
        if (o.p[m] < 0) continue;
        int i, j, k;
        cunpack(o.p[m], i, j, k);
        c[m] = i + L.nx * j + L.nxy * k;
        col[m] = (i + j + k) & 1;
        // the first wall's ghost lives in the owner's slot of SX, rewritten
        // with each update; further walls of the cell are formed on reading
        const int slot = 2 * CS + m * kHCWG + tid;
        const int iv[3] = {i, j, k};
        int first = 2 * DIM;
        wall[m] = 0;
#pragma unroll
        for (int d = DIM - 1; d >= 0; --d) {
          const int st = d == 0 ? 1 : (d == 1 ? L.nx : L.nxy);
          const int nd = L.n[d];
          const int w = A.per[d] ? 0 : 1;
          const bool lo = iv[d] == 0, hi = iv[d] == nd - 1;
          nb[m][2 * d] = lo ? (w ? slot : c[m] + (nd - 1) * st) : c[m] - st;
          nb[m][2 * d + 1] = hi ? (w ? slot : c[m] - (nd - 1) * st) : c[m] + st;
          if (w && (lo || hi)) {
            wall[m] |= (lo ? 1 << (2 * d) : 0) | (hi ? 2 << (2 * d) : 0);
            first = lo ? 2 * d : 2 * d + 1;
          }
        }
        wall[m] &= wall[m] - 1;   // (first is the lowest)
        multi[m] = wall[m] != 0;
        const T lsw = lsc;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          ws[m][n] = GT[first][2 * n];
          const T b = GT[first][2 * n + 1];
          wb[m][n] = ws[m][n] < T(0) ? b : b * lsw;   // a Neumann constant scales with dx
        }
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const int fx = L.n[0] + (d == 0), fy = L.n[1] + (d == 1);
          const int at = fo[d] + i + fx * (j + (DIM == 3 ? fy * k : 0));
          const int st = d == 0 ? 1 : (d == 1 ? fx : fx * fy);
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            F[m].v[n][2 * d] = FC[at + n * nf[d]];
            F[m].v[n][2 * d + 1] = FC[at + n * nf[d] + st];
          }
        }
        aa[m][0] = aa[m][1] = T(1);
        if (A.a[l]) {
          const long long lsy = L.n[0] + 2, lsz = lsy * (L.n[1] + 2);
          const long long q = (i + 1) + lsy * (j + 1) + (DIM == 3 ? lsz * (k + 1) : 0);
          aa[m][0] = A.a[l][q];
          aa[m][1] = A.a[l][q + lsz * (DIM == 3 ? L.n[2] + 2 : 1)];
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          if (up) {
            lam[m][n] = LM[n * tot + off + c[m]];
          } else {
            lam[m][n] = lambda_of<T, DIM>(F[m], n, aa[m][n], A.alpha, A.beta, dxinv);
            if (nl > 1) LM[n * tot + off + c[m]] = lam[m][n];
          }
          rr[m][n] = R[n * tot + off + c[m]];
          ph[m][n] = P[n * tot + off + c[m]];
          pl[m][n] = SL[n * CS + c[m]];
          SX[n * CS + m * kHCWG + tid] = fma(ws[m][n], pl[m][n], wb[m][n]);
        }
      }
      // L(phi) of slot m
      auto lof = [&](auto M, T(&out)[2]) __attribute__((always_inline)) {
        constexpr int m = decltype(M)::value;
        T st[2][7];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          st[n][0] = pl[m][n];
#pragma unroll
          for (int f = 0; f < 2 * DIM; ++f) st[n][1 + 2 * (f >> 1) + (1 - (f & 1))] = SL[n * CS + nb[m][f]];
        }
        if (multi[m]) {
#pragma unroll
          for (int f = 1; f < 2 * DIM; ++f)
#pragma unroll
            for (int n = 0; n < 2; ++n)
              if ((wall[m] >> f) & 1) {
                const T s = GT[f][2 * n], b = GT[f][2 * n + 1];
                st[n][1 + 2 * (f >> 1) + (1 - (f & 1))] = fma(s, pl[m][n], s < T(0) ? b : b * lsc);
              }
        }
#pragma unroll
        for (int n = 0; n < 2; ++n)
          out[n] = lof_of<T, DIM>(F[m], n, st[n], aa[m][n], ph[m][n], A.alpha, A.beta, dxinv);
      };
      if (!up && (v > 0 || A.add_first)) {
        // FAS right-hand side: rhs += L(phi)
        auto add = [&](auto M) __attribute__((always_inline)) {
          constexpr int m = decltype(M)::value;
          if (o.p[m] < 0) return;
          T lf[2];
          lof(M, lf);
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            rr[m][n] = rr[m][n] + lf[n];
            R[n * tot + off + c[m]] = rr[m][n];
          }
        };
        add(IC<0>{});
        add(IC<1>{});
        sync();   // the passes overwrite the closures just read
      }
      bool changed = false;
      auto update = [&](auto M) __attribute__((always_inline)) {
        constexpr int m = decltype(M)::value;
        if (o.p[m] < 0) return;
        T lf[2];
        lof(M, lf);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const T nv = ph[m][n] - lam[m][n] * (lf[n] - rr[m][n]);
          changed = changed || bits_of(nv) != bits_of(ph[m][n]);
          ph[m][n] = nv;
        }
        closure<T>(ph[m][0], ph[m][1], A.cp, pl[m][0], pl[m][1]);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          SL[n * CS + c[m]] = pl[m][n];
          SX[n * CS + m * kHCWG + tid] = fma(ws[m][n], pl[m][n], wb[m][n]);
        }
      };
      // the bottom ends at its fixed point
      auto fixed = [&]() __attribute__((always_inline)) {
        const bool go = small ? __any(changed) : __syncthreads_or(changed);
        changed = false;
        return !go;
      };
      const int its = bot ? A.bottom : (up ? A.nu2 : A.nu1);
      if (even) {
#pragma unroll 1
        for (int it = 0; it < its; ++it) {
          update(IC<0>{});
          sync();
          update(IC<1>{});
          sync();
          if (bot && fixed()) break;
        }
      } else {
#pragma unroll 1
        for (int p = 0; p < 2 * its; ++p) {
          if (o.p[0] >= 0 && col[0] == (p & 1)) update(IC<0>{});
          if (o.p[1] >= 0 && col[1] == (p & 1)) update(IC<1>{});
          sync();
          if (bot && (p & 1) && fixed()) break;
        }
      }
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (o.p[m] >= 0) {
          P[off + c[m]] = ph[m][0];
          P[tot + off + c[m]] = ph[m][1];
        }
      if (down) {
        // restriction (RESTRICTRESNLVC / RESTRICT): (rhs - L phi)/2^d per
        // cell, then child sums in Fortran order
        auto res = [&](auto M) __attribute__((always_inline)) {
          constexpr int m = decltype(M)::value;
          if (o.p[m] < 0) return;
          T lf[2];
          lof(M, lf);
          rr[m][0] = (rr[m][0] - lf[0]) * rdenom;
          rr[m][1] = (rr[m][1] - lf[1]) * rdenom;
        };
        res(IC<0>{});
        res(IC<1>{});
        sync();   // the ghosts in SX have been read
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (o.p[m] >= 0) {
            SX[c[m]] = rr[m][0];
            SX[CS + c[m]] = rr[m][1];
          }
        sync();
        const CLev C = level_of(l + 1);
#pragma unroll 1
        for (int cc = tid; cc < C.N; cc += step) {
          int I, J, K;
          clev_coords(C, cc, I, J, K);
          const int f0 = 2 * I + L.nx * (2 * J) + (DIM == 3 ? L.nxy * (2 * K) : 0);
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            T s = T(0), sp = T(0);
#pragma unroll
            for (int kk = 0; kk < (DIM == 3 ? 2 : 1); ++kk)
#pragma unroll
              for (int jj = 0; jj < 2; ++jj)
#pragma unroll
                for (int ii = 0; ii < 2; ++ii) {
                  const int f = f0 + ii + L.nx * jj + L.nxy * kk;
                  s = s + SX[n * CS + f];
                  sp = sp + P[n * tot + off + f] * rdenom;
                }
            R[n * tot + offc + cc] = s;
            P[n * tot + offc + cc] = sp;
            P0[n * tot1 + (offc - N0) + cc] = sp;
          }
        }
      }
    }
    // the next visit reads what this one wrote: wave 0 alone where both are
    // small, else the workgroup
    bool next_small = false;
    if (small && v + 1 < 2 * nl - 1) next_small = cown_active<kHCWG>(level_of(v + 1 >= nl ? 2 * nl - 3 - v : v + 1)) <= 64;
    if (!next_small)
      __syncthreads();
    else if (tid < 64)
      wave_sync();
  }
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int c = tid + m * kHCWG;
    if (c >= N0) continue;
#pragma unroll
    for (int n = 0; n < 2; ++n) A.phi[q0[m] + n * nc0] = P[n * tot + c];
  }
}

// closure of valid cells and wall ghosts (computeDiffusedVar, LevelData form)
template <typename T, int DIM>
__global__ void hc_diffused_var_kernel(HCArgs<T> A, const T* __restrict__ phi, T* __restrict__ out,
                                       int homog) {
  const Geom& g = A.g;
  const int gx = g.n[0] + 2, gy = g.n[1] + 2, gz = DIM == 3 ? g.n[2] + 2 : 1;
  const long long total = (long long)gx * gy * gz;
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < total;
       c += (long long)gridDim.x * blockDim.x) {
    const int i = int(c % gx) - 1;
    const long long r = c / gx;
    const int j = int(r % gy) - 1;
    const int k = DIM == 3 ? int(r / gy) - 1 : 0;
    const Pos P = classify<DIM>(g, i, j, k);
    const long long q = g.ci(i, j, k);
    if (P.kind == 0) continue;
    const long long qs = g.ci(P.i, P.j, P.k);
    T th, cl;
    closure<T>(phi[qs], phi[qs + g.ncell], A.cp, th, cl);
    if (P.kind == 2 && A.bc.apply) {
      const int isign = P.gs ? 1 : -1;
      const T v0 = homog ? T(0) : T(A.bc.val[P.gd][P.gs][0]);
      const T v1 = homog ? T(0) : T(A.bc.val[P.gd][P.gs][1]);
      th = bc_ghost<T>(A.bc.type[P.gd][P.gs][0], v0, th, isign, T(g.dx));
      cl = bc_ghost<T>(A.bc.type[P.gd][P.gs][1], v1, cl, isign, T(g.dx));
    }
    out[q] = th;
    out[q + g.ncell] = cl;
  }
}

// ---- streaming relaxation for large 2D levels ----------------------------
// The (H, Theta) counterpart of the linear operator's streaming kernel: a
// workgroup owns a block of columns and a segment of rows ("planes" below)
// and marches through them with a window of 4 planes in LDS
// holding (H, Theta) and their closure (theta, Theta_l).  With plane R just
// loaded (and its closure taken), colour pass p runs on plane R-1-p, so
// plane R-P is final and is written.  A cell's pass reads its own state and
// the closure of its other-colour neighbours, all as of the start of that
// pass, exactly as in the tiled kernel; an updated cell's closure (and its
// wall ghosts') is refreshed at once, which its same-colour cells never read
// (after the launch's last pass nothing reads it, so it is skipped there).
// Per plane and position the face coefficients, rhs (and aCoef) stay in
// registers in compile-time-indexed sets, loaded two planes ahead; lambda is
// formed where it is used.  Every input is read once per launch.  SEAM: the
// rows are periodic with an odd length, so the two cells at their seam share a
// colour and read each other as of the start of a pass.
template <typename T>
struct HCoef {
  CellFaces<T, 2> F;
  T rr[2], aq[2], v[2];   // rhs, aCoef, state as loaded
};

template <typename T, int TX, int P, int NT, bool HASA, bool SEAM>
__global__ __launch_bounds__(NT) void hc_relax_stream_kernel(HCArgs<T> A, const T* __restrict__ in,
                                                             T* __restrict__ out, const T* __restrict__ rhs,
                                                             int first, int nbx, int seg) {
  if (A.skip && *A.skip) return;
  constexpr int EX = TX + 2 * P;
  constexpr int EL = EX;
  constexpr int K = (EL + NT - 1) / NT;   // 1; without the loops over it a sweep of 2048^2 measured 3 % slower
  static_assert(P >= 1 && P <= 2, "one or two colour passes per launch");
  constexpr int W = 4;   // planes in the window
  constexpr int MD = 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* su = reinterpret_cast<T*>(smem_raw);
  const Geom& g = A.g;
  const int nz = g.n[MD];
  const bool zper = g.periodic[MD] != 0;
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));
  const T dxg = T(g.dx);
  const int bx = int(blockIdx.x) % nbx, bz = int(blockIdx.x) / nbx;
  const int x0 = bx * TX;
  const int z0 = bz * seg;
  const int z1 = z0 + seg < nz ? z0 + seg : nz;
  SPos S[K];
  int gt[K][2];   // a lateral ghost's BC type and value per component
  T gval[K][2];
#pragma unroll
  for (int kk = 0; kk < K; ++kk) {
    const int e = threadIdx.x + kk * NT;
    gt[kk][0] = gt[kk][1] = 0;
    gval[kk][0] = gval[kk][1] = T(0);
    if (e < EL) {
      spos_init<TX, P>(g, x0, e, S[kk]);
      for (int sd = 0; sd < 2; ++sd)
        if (S[kk].kind == 2 && S[kk].gs == sd)
          for (int n = 0; n < 2; ++n) {
            gt[kk][n] = A.bc.type[0][sd][n];
            gval[kk][n] = T(A.bc.val[0][sd][n]);
          }
    } else {
      S[kk].kind = 0;
      S[kk].dist = P;
      S[kk].owner = 0;
    }
  }
  // derived-variable ghost beyond wall (d, sd) of component n from the
  // interior closure value x (computeDiffusedVar's BC)
  auto ghost = [&](int d, int sd, int n, T x) {
    return A.bc.apply ? bc_ghost<T>(A.bc.type[d][sd][n], T(A.bc.val[d][sd][n]), x, sd ? 1 : -1, dxg) : x;
  };
  auto zwrap = [&](int z) { return z < 0 ? z + nz : (z >= nz ? z - nz : z); };
  auto real_plane = [&](int z) { return zper || (z >= 0 && z < nz); };
  // 32-bit element offsets (levels below 2^28 cells per component)
  const unsigned csz = unsigned(g.sy);
  const unsigned cn = unsigned(g.ncell);
  unsigned fpl[2], fup[2], fn[2];
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    fpl[d] = unsigned(g.fn[d][0]);
    fn[d] = unsigned(g.nface[d]);
  }
  fup[0] = 1;
  fup[MD] = fpl[MD];
  unsigned cl[K], fl[K][2];
#pragma unroll
  for (int kk = 0; kk < K; ++kk) {
    const SPos& s = S[kk];
    cl[kk] = unsigned(s.gx + 1);
#pragma unroll
    for (int d = 0; d < 2; ++d)
      fl[kk][d] = unsigned(s.gx);
  }
  auto ld = [](const T* p, unsigned i) -> T {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + (i * unsigned(sizeof(T))));
  };
  constexpr int NS = P + 3;
  HCoef<T> cs[NS][K];
  auto prefetch = [&](int R, HCoef<T>(&pf)[K]) {
    const int zw = zper ? zwrap(R) : (R < 0 ? 0 : (R >= nz ? nz - 1 : R));
    const unsigned qz = unsigned(zw + 1) * csz;
#pragma unroll
    for (int kk = 0; kk < K; ++kk) {
      const unsigned q = cl[kk] + qz;   // a ghost reads its interior neighbour
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        pf[kk].v[n] = ld(in, q + unsigned(n) * cn);
        pf[kk].rr[n] = ld(rhs, q + unsigned(n) * cn);
        if (HASA) pf[kk].aq[n] = ld(A.a, q + unsigned(n) * cn);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          const unsigned f = fl[kk][d] + unsigned(zw) * fpl[d] + unsigned(n) * fn[d];
          pf[kk].F.v[n][2 * d] = ld(A.b[d], f);
          pf[kk].F.v[n][2 * d + 1] = ld(A.b[d], f + fup[d]);
        }
      }
    }
  };
  const int zl = (!zper && z0 - P < 0) ? 0 : z0 - P;
  const int zend = z1 - 1 + P;
  // window slot of plane R: (H, Theta, theta, Theta_l) of EL positions each
  // (the bottom wall's ghost plane -1 is slot 3)
  auto slot = [&](int R) { return su + ((R - zl) & (W - 1)) * (4 * EL); };
  auto step = [&](auto J, int R) {
    constexpr int j = decltype(J)::value;
    // A. commit plane R: state, closure, lateral ghosts (or the top wall's
    // ghost plane)
    T* pl = slot(R);
    if (real_plane(R)) {
#pragma unroll
      for (int kk = 0; kk < K; ++kk) {
        const SPos& s = S[kk];
        const int e = threadIdx.x + kk * NT;
        if (s.kind == 0) continue;
        const T h = cs[j][kk].v[0], c = cs[j][kk].v[1];
        T th, clv;
        closure<T>(h, c, A.cp, th, clv);
        if (s.kind == 1) {
          pl[e] = h;
          pl[EL + e] = c;
          pl[2 * EL + e] = th;
          pl[3 * EL + e] = clv;
          if (!zper && R == 0) {
            T* gp = slot(-1);
            gp[2 * EL + e] = ghost(MD, 0, 0, th);
            gp[3 * EL + e] = ghost(MD, 0, 1, clv);
          }
        } else {
          const int isign = s.gs == 0 ? -1 : 1;
          pl[2 * EL + e] = A.bc.apply ? bc_ghost<T>(gt[kk][0], gval[kk][0], th, isign, dxg) : th;
          pl[3 * EL + e] = A.bc.apply ? bc_ghost<T>(gt[kk][1], gval[kk][1], clv, isign, dxg) : clv;
        }
      }
    } else if (!zper && R == nz) {
      const T* below = slot(nz - 1);
#pragma unroll
      for (int kk = 0; kk < K; ++kk) {
        const int e = threadIdx.x + kk * NT;
        if (S[kk].kind != 1) continue;
        pl[2 * EL + e] = ghost(MD, 1, 0, below[2 * EL + e]);
        pl[3 * EL + e] = ghost(MD, 1, 1, below[3 * EL + e]);
      }
    }
    // B. loads of plane R+2 into the set of plane R+2-NS, no longer in use
    constexpr int jn = (j + 2) % NS;
    prefetch(R + 2, cs[jn]);
    __syncthreads();
    // C. the colour passes; pass p on plane R-1-p uses set (j-1-p) mod NS
    auto pass = [&](auto PP) {
      constexpr int p = decltype(PP)::value;
      constexpr int jp = (j - 1 - p + 2 * NS) % NS;
      const int z = R - 1 - p;
      const int reach = P - 1 - p;
      const bool run = z >= z0 - reach && z < z1 + reach && real_plane(z);
      if (run) {
        const int zw = zwrap(z);
        const int colour = (first + p) & 1;
        T* pz = slot(z);
        const T* pm = slot(z - 1);
        const T* pp = slot(z + 1);
        auto mine = [&](const SPos& s) __attribute__((always_inline)) {
          return s.kind == 1 && s.dist <= reach && !((s.gx + zw + colour) & 1);
        };
        // an updated cell's closure and its wall ghosts: lateral, then along
        // the march
        auto refresh = [&](const SPos& s, int e, T h, T c) __attribute__((always_inline)) {
          T th, clv;
          closure<T>(h, c, A.cp, th, clv);
          pz[2 * EL + e] = th;
          pz[3 * EL + e] = clv;
          if (!g.periodic[0]) {
            if (s.gx == 0) {
              pz[2 * EL + e - 1] = ghost(0, 0, 0, th);
              pz[3 * EL + e - 1] = ghost(0, 0, 1, clv);
            }
            if (s.gx == g.n[0] - 1) {
              pz[2 * EL + e + 1] = ghost(0, 1, 0, th);
              pz[3 * EL + e + 1] = ghost(0, 1, 1, clv);
            }
          }
          if (!zper) {
            if (zw == 0) {
              T* gp = slot(-1);
              gp[2 * EL + e] = ghost(MD, 0, 0, th);
              gp[3 * EL + e] = ghost(MD, 0, 1, clv);
            }
            if (zw == nz - 1) {
              T* gp = slot(nz);
              gp[2 * EL + e] = ghost(MD, 1, 0, th);
              gp[3 * EL + e] = ghost(MD, 1, 1, clv);
            }
          }
        };
#pragma unroll
        for (int kk = 0; kk < K; ++kk) {
          const SPos& s = S[kk];
          if (!mine(s)) continue;
          const int e = threadIdx.x + kk * NT;
          const HCoef<T>& C = cs[jp][kk];
          T nv[2];
#pragma unroll
          for (int n = 0; n < 2; ++n) {
            const T* lz = pz + (2 + n) * EL;
            T st[7];
            st[0] = lz[e];
            st[1] = lz[e + 1];
            st[2] = lz[e - 1];
            st[3] = pp[(2 + n) * EL + e];
            st[4] = pm[(2 + n) * EL + e];
            const T ph = pz[n * EL + e];
            const T aq = HASA ? C.aq[n] : T(1);
            const T lam = lambda_of<T, 2>(C.F, n, aq, A.alpha, A.beta, dxinv);
            const T lof = lof_of<T, 2>(C.F, n, st, aq, ph, A.alpha, A.beta, dxinv);
            nv[n] = ph - lam * (lof - C.rr[n]);
          }
          pz[e] = nv[0];
          pz[EL + e] = nv[1];
          // the last pass's closure is never read: its cells' neighbours
          // (the other colour) are not updated again in this launch
          if constexpr (p < P - 1 && !SEAM) refresh(s, e, nv[0], nv[1]);
        }
        if constexpr (p < P - 1 && SEAM) {
          __syncthreads();   // the two cells at the seam read each other's closure
#pragma unroll
          for (int kk = 0; kk < K; ++kk) {
            const int e = threadIdx.x + kk * NT;
            if (mine(S[kk])) refresh(S[kk], e, pz[e], pz[EL + e]);
          }
        }
      }
      __syncthreads();
    };
    pass(IC<0>{});
    if constexpr (P > 1) pass(IC<1>{});
    // D. plane R-P is final
    const int zs = R - P;
    if (zs >= z0 && zs < z1) {
      const T* ps = slot(zs);
#pragma unroll
      for (int kk = 0; kk < K; ++kk) {
        if (!S[kk].owner) continue;
        const unsigned q = cl[kk] + unsigned(zs + 1) * csz;
        const int e = threadIdx.x + kk * NT;
        *reinterpret_cast<T*>(reinterpret_cast<char*>(out) + q * unsigned(sizeof(T))) = ps[e];
        *reinterpret_cast<T*>(reinterpret_cast<char*>(out) + (q + cn) * unsigned(sizeof(T))) = ps[EL + e];
      }
    }
  };
  prefetch(zl, cs[0]);
  prefetch(zl + 1, cs[1]);
  for (int R = zl; R <= zend; R += NS) {
    step(IC<0>{}, R);
    if (R + 1 <= zend) step(IC<1>{}, R + 1);
    if (R + 2 <= zend) step(IC<2>{}, R + 2);
    if constexpr (NS > 3) {
      if (R + 3 <= zend) step(IC<3 % NS>{}, R + 3);
    }
    if constexpr (NS > 4) {
      if (R + 4 <= zend) step(IC<4 % NS>{}, R + 4);
    }
  }
}

}  // namespace

// ---------------------------------------------------------------- launchers

template <typename T, int DIM>
struct TileDims;
template <typename T>
struct TileDims<T, 2> {
  static constexpr int TX = 32, TY = 8, TZ = 1;
};
template <typename T>
struct TileDims<T, 3> {
  static constexpr int TX = 16, TY = 8, TZ = 4;
};

template <typename T, int DIM>
static int tiles_of(const Geom& g, int& ntx, int& nty) {
  using D = TileDims<T, DIM>;
  ntx = (g.n[0] + D::TX - 1) / D::TX;
  nty = (g.n[1] + D::TY - 1) / D::TY;
  const int ntz = DIM == 3 ? (g.n[2] + D::TZ - 1) / D::TZ : 1;
  return ntx * nty * ntz;
}

template <typename T, int DIM>
static size_t tile_lds(int halo, bool restrict_mode) {
  using D = TileDims<T, DIM>;
  const size_t E = size_t(D::TX + 2 * halo) * (D::TY + 2 * halo) * (DIM == 3 ? D::TZ + 2 * halo : 1);
  size_t n = 4 * E;
  if (restrict_mode) n += 2 * size_t(D::TX) * D::TY * (DIM == 3 ? D::TZ : 1);
  return n * sizeof(T);
}

template <typename T, int DIM, int MODE>
static hipError_t launch_tile(const HCArgs<T>& A, TileIO<T> io, hipStream_t s) {
  using D = TileDims<T, DIM>;
  const int nt = tiles_of<T, DIM>(A.g, io.ntx, io.nty);
  const size_t lds = tile_lds<T, DIM>(1, MODE == kRestrict);
  if (lds > kMaxLds) return hipErrorInvalidValue;
  hipLaunchKernelGGL((hc_tile_kernel<T, DIM, D::TX, D::TY, D::TZ, MODE>), dim3(nt), dim3(kThreads), lds, s, A, io);
  return hipGetLastError();
}

// Colour passes of one 2D relaxation launch: up to 512^2 cells the launches
// are latency-bound and four sweeps share one (core 16^2 of the 32^2 region;
// at 512^2 34.7 us against four launches of 13.9 us); larger levels, where
// the halo's work counts, take one sweep (core 28^2).
constexpr long long kDeepHaloCells = 512 * 512;

static int relax_passes_per_launch(const Geom& g) { return g.nvalid() <= kDeepHaloCells ? 8 : 2; }

// algorithmic bytes of a relaxation launch: state (2 comps) in and out, rhs,
// a, faces (2 comps) once each; the coarse state (and its initial copy) when
// prolonged on load
template <typename T>
static double relax_bytes(const HCArgs<T>& A, const TileIO<T>& io) {
  const double cells = double(A.g.nvalid());
  double faces = 0;
  for (int d = 0; d < A.g.dim; ++d) faces += double(A.g.nface[d]);
  double b = 2 * cells + 2 * cells + (A.a ? 2 * cells : 0) + 2 * faces + 2 * cells;
  if (io.pc) b += 2 * io.gc.nvalid() * (io.pc0 ? 2 : 1);
  return b * sizeof(T);
}

template <typename T, int MODE>
static hipError_t launch_relax_pair(const HCArgs<T>& A, const TileIO<T>& io, hipStream_t s, const LaunchTimer* tm) {
  const int H = io.npass + (MODE == RB_PLAIN ? 0 : 1);
  if (io.npass < 1 || H > 9) return hipErrorInvalidValue;
  const Geom& g = A.g;
  PairArgs<T> P{};
  P.skip = A.skip;
  P.phi = io.phi;
  P.rhs = io.rhs;
  P.b0 = A.b[0];
  P.b1 = A.b[1];
  P.a = A.a;
  P.nx = g.n[0];
  P.ny = g.n[1];
  P.sy = int(g.sy);
  P.npass = io.npass;
  P.first = io.first;
  P.per0 = g.periodic[0];
  P.per1 = g.periodic[1];
  P.ncell = unsigned(g.ncell);
  P.nf0 = g.nface[0];
  P.nf1 = g.nface[1];
  P.alpha = A.alpha;
  P.beta = A.beta;
  P.dxinv = T(1) / (T(g.dx) * T(g.dx));
  P.phi_out = io.phi_out;
  P.rhs_out = io.rhs_out;
  P.pc = io.pc;
  P.pc0 = io.pc0;
  P.out = io.out;
  P.phic = io.phic;
  P.phic0 = io.phic0;
  P.cnx = io.gc.n[0];
  P.cny = io.gc.n[1];
  P.csy = int(io.gc.sy);
  P.cncell = unsigned(io.gc.ncell);
  P.norm = io.norm;
  P.fuse = io.fuse;
  P.cp = A.cp;
  const GhostForm<T> gf = ghost_form<T>(A.bc, T(g.dx));
  for (int d = 0; d < 2; ++d)
    for (int sd = 0; sd < 2; ++sd)
      for (int n = 0; n < 2; ++n) {
        P.gs[d][sd][n] = gf.s[d][sd][n];
        P.gb[d][sd][n] = gf.b[d][sd][n];
      }
  bool both = false;
  const int core = kRB - 2 * H, corex = pair_core_x(g.n[0], g.periodic[0], H, &both);
  const int ntx = (g.n[0] + corex - 1) / corex, nty = (g.n[1] + core - 1) / core;
  if (g.ncell >= (1LL << 32)) return hipErrorInvalidValue;   // (32-bit component stride)
  P.ntx = ntx;
  // GEN where a grid needs it: more than 2^16 - 1 tiles along y included
  bool gen = nty > 65535 || 8 * (g.ncell > g.nface[0] + g.nface[1] ? g.ncell : g.nface[0] + g.nface[1]) >= (1LL << 32);
  for (int d = 0; d < 2; ++d) gen = gen || (g.periodic[d] && (g.n[d] < kRB || (g.n[d] & 1)));
  const bool timed = tm && *tm->n < tm->cap;
  if (tm && !timed) ++*tm->missed;
  auto kern = gen ? hc_relax_pair_kernel<T, MODE, true> : hc_relax_pair_kernel<T, MODE, false>;
  hipExtLaunchKernelGGL(kern, gen ? dim3(unsigned(ntx) * unsigned(nty)) : dim3(ntx, nty), dim3(kRBThreads), 0, s, timed ? tm->start[*tm->n] : nullptr,
                        timed ? tm->stop[*tm->n] : nullptr, 0, P);
  const hipError_t err = hipGetLastError();
  if (err == hipSuccess && timed) {
    *tm->bytes += relax_bytes(A, io);
    ++*tm->n;
  }
  return err;
}

// One colour pass of a 3D level straight from memory (Sweep3).  The closure
// of the neighbours is worked out again by every cell that reads it: 3.5 of
// them per cell and pass, some 3 us of the chip's FP64 units at 96 x 64 x 48,
// against tiles that stage 3.75 positions per cell and leave half their lanes
// idle in a pass.  MODE 0: in place on `out`; 1: from `in`, every cell written
// to `out` (every pass of the GEN form); 2: no pass, `out` = `in` + prolonged
// pc - pc0.  Two passes: 69 us at 128^3 (a march along z with planes in LDS:
// 161), 17.6 at 96 x 64 x 48 (tiles: 50.9), 12 from 48 x 32 x 24 down to 16^3
// (tiles: 17); GEN 89 us at 129 x 128 x 128, 20 at 97 x 64 x 48.
template <typename T, bool GEN>
struct HCSweep {
  Sweep3<GEN> S;
  const int* skip;
  const T* in;
  T* out;
  const T* rhs;
  const T* a;
  const T* b[3];
  const T* pc;
  const T* pc0;
  long long ncell, nface[3];
  T alpha, beta, dxinv, gs[3][2][2], gb[3][2][2];
  ClosureP<T> cp;
};
template <typename T, int MODE, bool GEN>
__global__ __launch_bounds__(256) void hc_sweep3_kernel(HCSweep<T, GEN> A, Geom gc) {
  if (A.skip && *A.skip) return;
  Sweep3Pos<GEN> P;
  if (!sweep3_pos(A.S, P)) return;
  if constexpr (MODE == 2) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      if (!(m ? P.oth : P.act)) continue;
      const auto q = m ? P.qo : P.q;
      const int i = m ? P.i + 1 - 2 * P.par : P.i;
#pragma unroll
      for (int n = 0; n < 2; ++n)
        put_at(A.out + n * A.ncell, q,
              prolong_value<T, 3>(gc, i, P.j, P.k, A.pc + n * gc.ncell, A.pc0 ? A.pc0 + n * gc.ncell : nullptr,
                                  get_at(A.in + n * A.ncell, q)));
    }
  } else {
    const T* in = MODE == 1 ? A.in : A.out;
    if (MODE == 1 && P.oth) {
      put_at(A.out, P.qo, get_at(in, P.qo));
      put_at(A.out + A.ncell, P.qo, get_at(in + A.ncell, P.qo));
    }
    if (!P.act) return;
    T h[7], c[7];
    h[0] = get_at(in, P.q);
    c[0] = get_at(in + A.ncell, P.q);
#pragma unroll
    for (int f = 0; f < 6; ++f) {
      h[1 + (f ^ 1)] = get_at(in, P.nb[f]);
      c[1 + (f ^ 1)] = get_at(in + A.ncell, P.nb[f]);
    }
    CellFaces<T, 3> F;
    T aq[2], rr[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
#pragma unroll
      for (int d = 0; d < 3; ++d)
        sweep3_faces(A.S, P, d, A.b[d] + n * A.nface[d], F.v[n][2 * d], F.v[n][2 * d + 1]);
      rr[n] = get_at(A.rhs + n * A.ncell, P.q);
      aq[n] = A.a ? get_at(A.a + n * A.ncell, P.q) : T(1);
    }
    T st[2][7];
#pragma unroll
    for (int m = 0; m < 7; ++m) closure<T>(h[m], c[m], A.cp, st[0][m], st[1][m]);
    if (P.wall) {
#pragma unroll
      for (int f = 0; f < 6; ++f)
        if ((P.wall >> f) & 1)
#pragma unroll
          for (int n = 0; n < 2; ++n)
            st[n][1 + (f ^ 1)] = fma(A.gs[f >> 1][f & 1][n], st[n][0], A.gb[f >> 1][f & 1][n]);
    }
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const T ph = n ? c[0] : h[0];
      const T lam = lambda_of<T, 3>(F, n, aq[n], A.alpha, A.beta, A.dxinv);
      const T lof = lof_of<T, 3>(F, n, st[n], aq[n], ph, A.alpha, A.beta, A.dxinv);
      put_at(A.out + n * A.ncell, P.q, ph - lam * (lof - rr[n]));
    }
  }
}

// npass >= 1 colour passes of a 3D level: the prolongation, or the first
// pass, from buf[*cur] to the other buffer, the others in place there (GEN:
// each on to the other buffer)
template <typename T, bool GEN>
hipError_t hc_relax_sweeps(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, int first,
                           const Geom* gc, const T* pc, const T* pc0, hipStream_t s, const LaunchTimer* tm) {
  const Geom& g = A.g;
  HCSweep<T, GEN> V{};
  V.S = sweep3_make<GEN>(g);
  V.skip = A.skip;
  V.rhs = rhs;
  V.a = A.a;
  V.pc = pc;
  V.pc0 = pc0;
  V.ncell = g.ncell;
  V.alpha = A.alpha;
  V.beta = A.beta;
  V.dxinv = T(1) / (T(g.dx) * T(g.dx));
  V.cp = A.cp;
  const GhostForm<T> gf = ghost_form<T>(A.bc, T(g.dx));
  double faces = 0;
  for (int d = 0; d < 3; ++d) {
    V.b[d] = A.b[d];
    V.nface[d] = g.nface[d];
    faces += double(g.nface[d]);
    for (int sd = 0; sd < 2; ++sd)
      for (int n = 0; n < 2; ++n) {
        V.gs[d][sd][n] = gf.s[d][sd][n];
        V.gb[d][sd][n] = gf.b[d][sd][n];
      }
  }
  const Geom gcc = gc ? *gc : g;
  for (int p = pc ? -1 : 0; p < npass; ++p) {
    V.S.colour = (first + p) & 1;
    const bool timed = p >= 0 && tm && *tm->n < tm->cap;
    if (p >= 0 && tm && !timed) ++*tm->missed;
    const bool moves = GEN || p < 0 || (p == 0 && !pc);
    V.in = buf[*cur];
    V.out = buf[moves ? 1 - *cur : *cur];
    auto kern = p < 0 ? hc_sweep3_kernel<T, 2, GEN> : (moves ? hc_sweep3_kernel<T, 1, GEN> : hc_sweep3_kernel<T, GEN ? 1 : 0, GEN>);
    hipExtLaunchKernelGGL(kern, dim3(8 * V.S.chunk), dim3(256), 0, s, timed ? tm->start[*tm->n] : nullptr,
                          timed ? tm->stop[*tm->n] : nullptr, 0, V, gcc);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (timed) {
      // both components: every state read, rhs and a of the colour, every
      // face; the colour written (a first pass: every cell)
      const double cells = double(g.nvalid());
      *tm->bytes += (2 * cells + cells * (1 + (A.a ? 1 : 0)) + 2 * faces + (moves ? 2 : 1) * cells) * sizeof(T);
      ++*tm->n;
    }
    if (moves) *cur = 1 - *cur;
  }
  return hipSuccess;
}

// streaming launch shape: columns of 252 cells (256 threads)
struct HCStream {
  static constexpr int NT = 256, SEGMIN = 8;
};

// 2D levels whose plain relaxations stream (above 512^2 cells), with 32-bit
// offsets for both components of every array.  Not with an odd periodic
// length along the march: the rows at its seam share colours, and a pass
// reaches one of them before the other.
constexpr long long kHCStreamCells2 = 512 * 512;
inline bool hc_streams(const Geom& g) {
  long long nf = 0;
  for (int d = 0; d < g.dim; ++d) nf = nf > g.nface[d] ? nf : g.nface[d];
  const long long most = 2 * (g.ncell > nf ? g.ncell : nf);
  return g.dim == 2 && g.nvalid() > kHCStreamCells2 && g.n[1] >= 8 && !(g.periodic[1] && (g.n[1] & 1)) &&
         most < (1LL << 29);
}

template <typename T, int P, bool HASA, bool SEAM>
hipError_t hc_stream_launch(const HCArgs<T>& A, const T* in, T* out, const T* rhs, int first, hipStream_t s,
                            const LaunchTimer* tm) {
  using D = HCStream;
  constexpr int TX = D::NT - 2 * P, EL = D::NT;
  const Geom& g = A.g;
  const int nbx = (g.n[0] + TX - 1) / TX;
  const size_t lds = size_t(4) * 4 * EL * sizeof(T);
  auto kern = hc_relax_stream_kernel<T, TX, P, D::NT, HASA, SEAM>;
  // segments sized so that the whole grid is resident at once
  static int resident = 0;
  if (!resident) {
    int dev = 0, cus = 0, per = 0;
    if (hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) ==
                                                 hipSuccess &&
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void*>(kern), D::NT, lds) ==
            hipSuccess &&
        cus > 0 && per > 0)
      resident = cus * per;
    else
      resident = 768;
  }
  const int nz = g.n[1];
  const int per_column = resident / nbx > 1 ? resident / nbx : 1;
  int seg = (nz + per_column - 1) / per_column;
  if (seg < D::SEGMIN) seg = D::SEGMIN;
  const int nbz = (nz + seg - 1) / seg;
  const bool timed = tm && *tm->n < tm->cap;
  if (tm && !timed) ++*tm->missed;
  hipExtLaunchKernelGGL(kern, dim3(nbx * nbz), dim3(D::NT), lds, s, timed ? tm->start[*tm->n] : nullptr,
                        timed ? tm->stop[*tm->n] : nullptr, 0, A, in, out, rhs, first, nbx, seg);
  const hipError_t e = hipGetLastError();
  if (e == hipSuccess && timed) {
    const double cells = double(g.nvalid());
    double faces = 0;
    for (int d = 0; d < 2; ++d) faces += double(g.nface[d]);
    const double by = 2 * cells + 2 * cells + (HASA ? 2 * cells : 0) + 2 * faces + 2 * cells;
    *tm->bytes += by * sizeof(T);
    ++*tm->n;
  }
  return e;
}

template <typename T>
hipError_t hc_relax_stream(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, int first,
                           hipStream_t s, const LaunchTimer* tm) {
  const bool seam = A.g.periodic[0] && (A.g.n[0] & 1);
  int done = 0;
  while (done < npass) {
    const int p = (npass - done) >= 2 ? 2 : 1;
    const int f = (first + done) & 1;
    // (a single pass refreshes no closure, so it has no use for SEAM)
    auto launch = A.a ? (p == 1 ? hc_stream_launch<T, 1, true, false>
                                : (seam ? hc_stream_launch<T, 2, true, true> : hc_stream_launch<T, 2, true, false>))
                      : (p == 1 ? hc_stream_launch<T, 1, false, false>
                                : (seam ? hc_stream_launch<T, 2, false, true> : hc_stream_launch<T, 2, false, false>));
    const hipError_t e = launch(A, buf[*cur], buf[1 - *cur], rhs, f, s, tm);
    if (e != hipSuccess) return e;
    *cur = 1 - *cur;
    done += p;
  }
  return hipSuccess;
}

template <typename T>
hipError_t hc_relax_tiles(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, int first,
                          const Geom* gc, const T* pc, const T* pc0, hipStream_t s, const LaunchTimer* tm) {
  if (npass > 0 && A.g.dim == 3)
    return sweep3_plain(A.g) ? hc_relax_sweeps<T, false>(A, buf, cur, rhs, npass, first, gc, pc, pc0, s, tm)
                             : hc_relax_sweeps<T, true>(A, buf, cur, rhs, npass, first, gc, pc, pc0, s, tm);
  // plain relaxations of large levels stream along the last direction
  if (!pc && npass > 0 && hc_streams(A.g)) return hc_relax_stream<T>(A, buf, cur, rhs, npass, first, s, tm);
  const int pmax = relax_passes_per_launch(A.g);
  int done = 0;
  while (done < npass) {
    TileIO<T> io{};
    io.phi = buf[*cur];
    io.phi_out = buf[1 - *cur];
    io.rhs = rhs;
    io.npass = (npass - done) < pmax ? (npass - done) : pmax;
    io.first = (first + done) & 1;
    if (done == 0 && pc) {
      io.gc = *gc;
      io.pc = pc;
      io.pc0 = pc0;
    }
    const hipError_t e = launch_relax_pair<T, RB_PLAIN>(A, io, s, tm);
    if (e != hipSuccess) return e;
    *cur = 1 - *cur;
    done += io.npass;
  }
  if (npass == 0 && pc) {
    // a prolongation with no smoothing after it (per cell, in place)
    return prolong_linear<T>(A.g, 2, buf[*cur], pc, pc0, s);
  }
  return hipSuccess;
}

template <typename T>
hipError_t hc_relax(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, int first,
                    hipStream_t s, const LaunchTimer* tm) {
  if (npass <= 0) return hipSuccess;
  return hc_relax_tiles<T>(A, buf, cur, rhs, npass, first, nullptr, nullptr, nullptr, s, tm);
}

bool hc_fuses(const Geom& g) { return g.dim == 2 && !hc_streams(g); }

template <typename T>
hipError_t hc_relax_restrict(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, T* rhs_out, int npass,
                             const Geom& gc, T* resc, T* phic, T* phic0, hipStream_t s) {
  if (npass < 1 || rhs_out == rhs) return hipErrorInvalidValue;
  const int pmax = relax_passes_per_launch(A.g);
  for (int done = 0; done < npass;) {
    TileIO<T> io{};
    io.phi = buf[*cur];
    io.phi_out = buf[1 - *cur];
    io.rhs = done && rhs_out ? rhs_out : rhs;
    io.rhs_out = done ? nullptr : rhs_out;
    io.npass = (npass - done) < pmax ? (npass - done) : pmax;
    io.first = done & 1;
    const bool end = done + io.npass == npass;
    if (end) {
      io.gc = gc;
      io.out = resc;
      io.phic = phic;
      io.phic0 = phic0;
    }
    const hipError_t e = end ? launch_relax_pair<T, RB_RESTRICT>(A, io, s, nullptr)
                             : launch_relax_pair<T, RB_PLAIN>(A, io, s, nullptr);
    if (e != hipSuccess) return e;
    *cur = 1 - *cur;
    done += io.npass;
  }
  return hipSuccess;
}

template <typename T>
hipError_t hc_relax_final(const HCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, const Geom* gc,
                          const T* pc, const T* pc0, unsigned long long* norm, const CtlFuse& fuse, hipStream_t s) {
  if (npass < 1) return hipErrorInvalidValue;
  const int pmax = relax_passes_per_launch(A.g);
  for (int done = 0; done < npass;) {
    TileIO<T> io{};
    io.phi = buf[*cur];
    io.phi_out = buf[1 - *cur];
    io.rhs = rhs;
    io.npass = (npass - done) < pmax ? (npass - done) : pmax;
    io.first = done & 1;
    if (done == 0 && pc) {
      io.gc = *gc;
      io.pc = pc;
      io.pc0 = pc0;
    }
    const bool end = done + io.npass == npass;
    if (end) {
      io.norm = norm;
      io.fuse = fuse;
    }
    const hipError_t e =
        end ? launch_relax_pair<T, RB_NORM>(A, io, s, nullptr) : launch_relax_pair<T, RB_PLAIN>(A, io, s, nullptr);
    if (e != hipSuccess) return e;
    *cur = 1 - *cur;
    done += io.npass;
  }
  return hipSuccess;
}

int hc_coarse_cells() { return kWGCells; }

// state, right-hand side and (nl > 1) lambda of every level, the initial state
// below the first, closure and ghosts of one level, the faces; and the ghost
// rules (static).  At most 156,192 bytes over all shapes of up to 1024 cells
// (4 x 4 x 64; in 2D 149,504 at 64 x 16).
static size_t hc_coarse_lds_dyn(int nl, int tot, int n0, size_t nfaces) {
  return sizeof(double) * ((nl > 1 ? 6 : 4) * size_t(tot) + 2 * size_t(tot - n0) + 4 * kWGCells + nfaces);
}
size_t hc_coarse_lds_bytes(const Geom& g, int nl, size_t nfaces) {
  int tot = 0;
  for (int l = 0; l < nl; ++l) tot += int(coarsen_geom(g, 1 << l).nvalid());
  return hc_coarse_lds_dyn(nl, tot, int(g.nvalid()), nfaces) + sizeof(double) * 4 * (2 * g.dim + 1);
}

template <typename T>
hipError_t hc_coarse_vcycle(const Geom& g, const BCDesc& bc, HCCoarse<T> A, hipStream_t s) {
  if (g.nvalid() > kWGCells || A.nl < 1 || A.nl > kHCCoarseLevels) return hipErrorInvalidValue;
  for (int d = 0; d < 3; ++d) {
    A.n[d] = g.n[d];
    A.per[d] = g.periodic[d];
  }
  int fo = 0;
  for (int l = 0; l < A.nl; ++l) {
    const Geom gl = l == 0 ? g : coarsen_geom(g, 1 << l);
    A.off[l + 1] = A.off[l] + int(gl.nvalid());
    for (int d = 0; d < g.dim; ++d) {
      A.fo[l][d] = fo;
      A.nf[l][d] = int(gl.nface[d]);
      fo += 2 * A.nf[l][d];
    }
  }
  A.tot = A.off[A.nl];
  A.dx = T(g.dx);
  const GhostForm<T> gf = ghost_form<T>(bc, T(g.dx));
  for (int d = 0; d < 3; ++d)
    for (int sd = 0; sd < 2; ++sd)
      for (int n = 0; n < 2; ++n) {
        A.gs[d][sd][n] = gf.s[d][sd][n];
        A.gb[d][sd][n] = gf.b[d][sd][n];
      }
  static_assert(sizeof(T) == sizeof(double), "the LDS map's element");
  const size_t lds = hc_coarse_lds_dyn(A.nl, A.tot, A.off[1], size_t(A.nfaces));
  if (g.dim == 2)
    hipLaunchKernelGGL((hc_coarse_vcycle_kernel<T, 2>), dim3(1), dim3(kHCWG), lds, s, A);
  else
    hipLaunchKernelGGL((hc_coarse_vcycle_kernel<T, 3>), dim3(1), dim3(kHCWG), lds, s, A);
  return hipGetLastError();
}

template <typename T>
hipError_t hc_residual(const HCArgs<T>& A, T* phi, const T* rhs, T* res, unsigned long long* norm,
                       int homog, hipStream_t s, const CtlFuse& fuse) {
  if (fuse.ctl && !norm) return hipErrorInvalidValue;
  TileIO<T> io{};
  io.fuse = fuse;
  io.phi = phi;
  io.rhs = rhs;
  io.out = res;
  io.norm = norm;
  io.homog = homog;
  return A.g.dim == 2 ? launch_tile<T, 2, kResid>(A, io, s) : launch_tile<T, 3, kResid>(A, io, s);
}

template <typename T>
hipError_t hc_apply_op(const HCArgs<T>& A, T* phi, T* lhs, const T* add, int homog, hipStream_t s) {
  TileIO<T> io{};
  io.phi = phi;
  io.out = lhs;
  io.add = add;
  io.homog = homog;
  return A.g.dim == 2 ? launch_tile<T, 2, kApply>(A, io, s) : launch_tile<T, 3, kApply>(A, io, s);
}

int hc_apply_tiles(const Geom& g, int* ntx, int* nty) {
  return g.dim == 2 ? tiles_of<double, 2>(g, *ntx, *nty) : tiles_of<double, 3>(g, *ntx, *nty);
}

template <typename T>
hipError_t hc_apply_batch(int dim, const HCApplyJob<T>* jobs, const unsigned* map, int nblocks, hipStream_t s) {
  if (nblocks <= 0) return hipSuccess;
  if (dim == 2) {
    using D = TileDims<T, 2>;
    const size_t lds = tile_lds<T, 2>(1, false);
    hipLaunchKernelGGL((hc_apply_batch_kernel<T, 2, D::TX, D::TY, D::TZ>), dim3(nblocks), dim3(kThreads), lds, s,
                       jobs, map);
  } else {
    using D = TileDims<T, 3>;
    const size_t lds = tile_lds<T, 3>(1, false);
    hipLaunchKernelGGL((hc_apply_batch_kernel<T, 3, D::TX, D::TY, D::TZ>), dim3(nblocks), dim3(kThreads), lds, s,
                       jobs, map);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t hc_restrict_residual(const HCArgs<T>& A, const Geom& gc, T* phi, const T* rhs, T* resc,
                                int homog, hipStream_t s) {
  return hc_restrict_all<T>(A, gc, phi, rhs, resc, nullptr, nullptr, homog, s);
}

template <typename T>
hipError_t hc_restrict_all(const HCArgs<T>& A, const Geom& gc, T* phi, const T* rhs, T* resc, T* phic, T* phic0,
                           int homog, hipStream_t s) {
  TileIO<T> io{};
  io.phi = phi;
  io.rhs = rhs;
  io.out = resc;
  io.gc = gc;
  io.phic = phic;
  io.phic0 = phic0;
  io.homog = homog;
  return A.g.dim == 2 ? launch_tile<T, 2, kRestrict>(A, io, s) : launch_tile<T, 3, kRestrict>(A, io, s);
}

template <typename T>
hipError_t hc_diffused_var(const HCArgs<T>& A, const T* phi, T* out, int homog, hipStream_t s) {
  const long long total = A.g.ncell;
  const int blocks = int((total + 255) / 256);
  if (A.g.dim == 2)
    hipLaunchKernelGGL((hc_diffused_var_kernel<T, 2>), dim3(blocks), dim3(256), 0, s, A, phi, out, homog);
  else
    hipLaunchKernelGGL((hc_diffused_var_kernel<T, 3>), dim3(blocks), dim3(256), 0, s, A, phi, out, homog);
  return hipGetLastError();
}

template hipError_t hc_relax<double>(const HCArgs<double>&, double* const[2], int*, const double*, int, int,
                                     hipStream_t, const LaunchTimer*);
template hipError_t hc_relax_tiles<double>(const HCArgs<double>&, double* const[2], int*, const double*, int, int,
                                           const Geom*, const double*, const double*, hipStream_t,
                                           const LaunchTimer*);
template hipError_t hc_relax_restrict<double>(const HCArgs<double>&, double* const[2], int*, const double*, double*,
                                              int, const Geom&, double*, double*, double*, hipStream_t);
template hipError_t hc_relax_final<double>(const HCArgs<double>&, double* const[2], int*, const double*, int,
                                           const Geom*, const double*, const double*, unsigned long long*,
                                           const CtlFuse&, hipStream_t);
template hipError_t hc_coarse_vcycle<double>(const Geom&, const BCDesc&, HCCoarse<double>, hipStream_t);
template hipError_t hc_residual<double>(const HCArgs<double>&, double*, const double*, double*,
                                        unsigned long long*, int, hipStream_t, const CtlFuse&);
template hipError_t hc_apply_op<double>(const HCArgs<double>&, double*, double*, const double*, int, hipStream_t);
template hipError_t hc_apply_batch<double>(int, const HCApplyJob<double>*, const unsigned*, int, hipStream_t);
template hipError_t hc_restrict_residual<double>(const HCArgs<double>&, const Geom&, double*, const double*,
                                                 double*, int, hipStream_t);
template hipError_t hc_restrict_all<double>(const HCArgs<double>&, const Geom&, double*, const double*, double*,
                                            double*, double*, int, hipStream_t);
template hipError_t hc_diffused_var<double>(const HCArgs<double>&, const double*, double*, int, hipStream_t);

}  // namespace ml
