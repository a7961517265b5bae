// ml_vc_kernels.hip — kernels of the linear variable-coefficient operator
//
//   L u = alpha*a*u - beta*c*u - beta*div(b grad u)      (one component)
//
// behind DarcyBrinkmanOp (src/DarcyBrinkmanOp.cpp, src/DarcyBrinkmanOpF.ChF;
// a = 1, b = -Pr, c = (Pr/Da) chi/Pi) and AMRProjectionOp (c absent,
// alpha = 0, beta = 1, b = -S_face).  The arithmetic of each cell follows
// GSRBHELMHOLTZDB / DBCOMPUTERES / DBCOMPUTEOP / RESTRICTRESDB term by term
// (compiled with -ffp-contract=off), so the FP64 results are those of the
// CPU restatement bit for bit.
//
//   vc_relax_tile_kernel   red/black Gauss-Seidel, homogeneous BCs (the
//                          residual-correction smoother), npass colour
//                          passes per launch over a tile grown by npass
//                          cells, input and output arrays distinct;
//                          optional zero start and piecewise-constant
//                          prolongation of a coarse correction on load
//   vc_tile_kernel         residual (+ max-norm, + fused phi += e),
//                          operator application, restricted residual
//   vc_coarse_vcycle_kernel  the V-cycle below the tiled levels in one
//                          workgroup (levels of at most 1024 cells)
#include <hip/hip_ext.h>

#include "ml_common.h"
#include <algorithm>

#include "ml_kernels.h"
#include "ml_tile.h"

namespace ml {

namespace {

constexpr int kVCThreads = 256;   // halo-1 tile kernels
constexpr int kVCWG = 512;        // single-workgroup kernel threads
constexpr int kVCWGCells = 1024;  // largest level it holds
constexpr int kVCM = kVCWGCells / kVCWG;

enum { kVCResid = 0, kVCApply = 1, kVCRestrict = 2 };

// Face coefficients of one component around a cell: v[2d] lo, v[2d+1] hi.
template <typename T, int DIM>
struct Faces1 {
  T v[2 * DIM];
};

template <typename T, int DIM>
__device__ inline void load_faces1(const VCArgs<T>& A, int i, int j, int k, Faces1<T, DIM>& F) {
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    F.v[2 * d] = A.b[d][A.g.fi(d, i, j, k)];
    F.v[2 * d + 1] = A.b[d][A.g.fi(d, i + (d == 0), j + (d == 1), k + (d == 2))];
  }
}

// lambda = 1/(alpha*a - beta*c + sum_d scale*beta*(b_hi + b_lo))
// (DarcyBrinkmanOp::resetLambda, src/DarcyBrinkmanOp.cpp:265-296, SUMFACES3
// src/DarcyBrinkmanOpF.ChF:511-545).
template <typename T, int DIM>
__device__ inline T vc_lambda(const Faces1<T, DIM>& F, T aq, bool hasc, T cq, T alpha, T beta, T scale) {
  T lam = aq * alpha;
  if (hasc) lam = lam + (-beta) * cq;
#pragma unroll
  for (int d = 0; d < DIM; ++d) lam = lam + scale * beta * (F.v[2 * d + 1] + F.v[2 * d]);
  return T(1) / lam;
}

// lofphi (src/DarcyBrinkmanOpF.ChF:125-147): alpha*a*u - beta*c*u - beta*S*dxinv
// from p[0] centre, p[2d+1] = +e_d, p[2d+2] = -e_d.
template <typename T, int DIM>
__device__ inline T vc_lof(const Faces1<T, DIM>& F, const T* p, T aq, bool hasc, T cq, T alpha, T beta, T dxinv) {
  const T p0 = p[0];
  T s = F.v[1] * (p[1] - p0) - F.v[0] * (p0 - p[2]) + F.v[3] * (p[3] - p0) - F.v[2] * (p0 - p[4]);
  if (DIM == 3) s = s + F.v[5] * (p[5] - p0) - F.v[4] * (p0 - p[6]);
  T lof = alpha * aq * p0;
  if (hasc) lof = lof - beta * cq * p0;
  return lof - beta * s * dxinv;
}

// Relaxation of L e = r on one tile with a halo of npass cells.  The
// coefficients, lambda and rhs of every position a thread may update are
// loaded once into registers; a pass updates one colour and refreshes the
// homogeneous wall ghosts of the cells it updated, so one barrier per pass.
// The body works on tile `tile` of the level (a batched launch maps its
// workgroups to (instance, tile) pairs).
// ODD: a periodic length is odd, so the two cells at its seam share a colour
// and read each other: a pass forms its values, then writes them.  (2D and
// plain relaxation only: a level that coarsens has even lengths.)
// In 3D for the fused forms and batches only.
template <typename T, int DIM, int TX, int TY, int TZ, int HMAX, int NT, bool ODD>
__device__ __forceinline__ void vc_relax_tile_body(const VCArgs<T>& A, const T* __restrict__ in, T* __restrict__ out,
                                                   const T* __restrict__ rhs, int npass, int first, int zero_init,
                                                   const Geom& gc, const T* __restrict__ pc, int ntx, int nty,
                                                   const Geom& gr, T* __restrict__ resc, const VCFinal<T>& fin,
                                                   int tile) {
  if (A.skip && *A.skip) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int EMAX = (TX + 2 * HMAX) * (TY + 2 * HMAX) * (DIM == 3 ? TZ + 2 * HMAX : 1);
  constexpr int KMAX = (EMAX + NT - 1) / NT;
  const Geom& g = A.g;
  Tile<DIM, TX, TY, TZ> t;
  // with a restriction or a residual to produce, one more halo cell keeps
  // the core's neighbours exact after the last pass
  const bool final = fin.phi != nullptr;
  t.init_at(npass + ((resc || final) ? 1 : 0), ntx, nty, tile);
  T* su = reinterpret_cast<T*>(smem_raw);
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));
  PosRec R[KMAX];
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) pos_record<DIM, TX, TY, TZ>(g, t, threadIdx.x + kk * NT, R[kk]);
  Faces1<T, DIM> F[KMAX];
  T aq[KMAX], cv[KMAX], lam[KMAX], rr[KMAX], v[KMAX], pv[KMAX], fv[KMAX], frhs[KMAX];
  // every global load of the tile is issued before the first use
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    v[kk] = T(0);
    pv[kk] = T(0);
    // phi near the core (for a wall ghost: of its interior neighbour)
    if (final && r.kind != 0 && r.dist <= 1) fv[kk] = fin.phi[r.q];
    if (r.kind != 1) continue;
    if (!zero_init) v[kk] = in[r.q];
    if (pc) pv[kk] = pc[gc.ci(r.i / 2, r.j / 2, DIM == 3 ? r.k / 2 : 0)];
    if (final && r.owner) frhs[kk] = fin.rhs[r.q];
  }
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.kind != 1 || r.dist > t.H - 1) continue;
    load_faces1<T, DIM>(A, r.i, r.j, r.k, F[kk]);
    aq[kk] = A.a ? A.a[r.q] : T(1);
    cv[kk] = A.c ? A.c[r.q] : T(0);
    rr[kk] = rhs[r.q];
  }
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.kind != 1) continue;
    T val = v[kk];
    if (pc) val = val + pv[kk];
    su[r.e] = val;
    if (r.dist > t.H - 1) continue;
    lam[kk] = vc_lambda<T, DIM>(F[kk], aq[kk], A.c != nullptr, cv[kk], A.alpha, A.beta, dxinv);
  }
  __syncthreads();
  // homogeneous wall ghosts of the staged state
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.kind != 2) continue;
    su[r.e] = bc_ghost<T>(A.bc.type[r.gd][r.gs][0], T(0), su[r.eint], r.gs == 0 ? -1 : 1, T(g.dx));
  }
  __syncthreads();
  for (int p = 0; p < npass; ++p) {
    const int gext = t.H - p;
    const int colour = (first + p) & 1;
    auto mine = [&](const PosRec& r) {
      return r.kind == 1 && r.dist <= gext - 1 && !((r.i + r.j + r.k + colour) & 1);
    };
    auto value = [&](int kk) __attribute__((always_inline)) {
      T st[7];
      gather_lds<T, DIM>(su, R[kk].e, t.EX, t.EXY, st);
      const T lof = vc_lof<T, DIM>(F[kk], st, aq[kk], A.c != nullptr, cv[kk], A.alpha, A.beta, dxinv);
      return st[0] - lam[kk] * (lof - rr[kk]);
    };
    if constexpr (ODD) {
#pragma unroll
      for (int kk = 0; kk < KMAX; ++kk)
        if (mine(R[kk])) v[kk] = value(kk);
      __syncthreads();
    }
#pragma unroll
    for (int kk = 0; kk < KMAX; ++kk) {
      const PosRec& r = R[kk];
      if (!mine(r)) continue;
      const T nv = ODD ? v[kk] : value(kk);
      su[r.e] = nv;
      // wall ghosts of this cell (it is their interior neighbour)
      const int iv[3] = {r.i, r.j, r.k};
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        if (g.periodic[d]) continue;
        const int stride = d == 0 ? 1 : (d == 1 ? t.EX : t.EXY);
#pragma unroll
        for (int sd = 0; sd < 2; ++sd) {
          if (iv[d] != (sd ? g.n[d] - 1 : 0)) continue;
          su[sd ? r.e + stride : r.e - stride] = bc_ghost<T>(A.bc.type[d][sd][0], T(0), nv, sd ? 1 : -1, T(g.dx));
        }
      }
    }
    __syncthreads();
  }
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.owner) out[r.q] = su[r.e];
  }
  if (final) {
    // u = phi + e near the core, its inhomogeneous wall ghosts, then the
    // residual of the full equation at the owned cells (DBCOMPUTERES order,
    // as vc_tile_kernel<kVCResid> with e)
    T* sv = su + t.E;
#pragma unroll
    for (int kk = 0; kk < KMAX; ++kk) {
      const PosRec& r = R[kk];
      if (r.dist > 1) continue;
      if (r.kind == 1) {
        sv[r.e] = fv[kk] + su[r.e];
      } else if (r.kind == 2) {
        // the interior value u = phi + e of the ghost's neighbour
        const T ui = fv[kk] + su[r.eint];
        sv[r.e] = bc_ghost<T>(A.bc.type[r.gd][r.gs][0], T(A.bc.val[r.gd][r.gs][0]), ui, r.gs == 0 ? -1 : 1,
                              T(g.dx));
      }
    }
    __syncthreads();
    T mx = T(0);
    int nan = 0;
#pragma unroll
    for (int kk = 0; kk < KMAX; ++kk) {
      const PosRec& r = R[kk];
      if (!r.owner) continue;
      fin.phi_out[r.q] = sv[r.e];
      T st[7];
      gather_lds<T, DIM>(sv, r.e, t.EX, t.EXY, st);
      const T lof = vc_lof<T, DIM>(F[kk], st, aq[kk], A.c != nullptr, cv[kk], A.alpha, A.beta, dxinv);
      const T res = frhs[kk] - lof;
      fin.res[r.q] = res;
      const T ar = fabs(res);
      if (ar != ar) nan = 1;
      else if (ar > mx) mx = ar;
    }
    block_max_atomic<T>(mx, nan, ctl_slot(nullptr, fin.fuse), fin.fuse);
    return;
  }
  if (!resc) return;
  // restricted residual of the relaxed correction (RESTRICTRESDB,
  // src/DarcyBrinkmanOpF.ChF:402-509, homogeneous BCs): (r - L e)/2^d per
  // fine cell, child sums in Fortran order
  T* sres = su + t.E;
  const T denom = DIM == 3 ? T(8) : T(4);
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (!r.owner) continue;
    int ex, ey, ez;
    t.coords(r.e, ex, ey, ez);
    const int c = (ex - t.H) + TX * ((ey - t.H) + TY * (DIM == 3 ? ez - t.H : 0));
    T st[7];
    gather_lds<T, DIM>(su, r.e, t.EX, t.EXY, st);
    const T lof = vc_lof<T, DIM>(F[kk], st, aq[kk], A.c != nullptr, cv[kk], A.alpha, A.beta, dxinv);
    sres[c] = (rr[kk] - lof) / denom;
  }
  __syncthreads();
  constexpr int CX = TX / 2, CY = TY / 2, CZ = DIM == 3 ? TZ / 2 : 1;
  for (int c = threadIdx.x; c < CX * CY * CZ; c += NT) {
    const int cx = c % CX, cr = c / CX, cy = cr % CY, cz = cr / CY;
    const int I = t.x0 / 2 + cx, J = t.y0 / 2 + cy, K = DIM == 3 ? t.z0 / 2 + cz : 0;
    if (I >= gr.n[0] || J >= gr.n[1] || (DIM == 3 && K >= gr.n[2])) continue;
    T sum = T(0);
    for (int kk = 0; kk < (DIM == 3 ? 2 : 1); ++kk)
      for (int jj = 0; jj < 2; ++jj)
        for (int ii = 0; ii < 2; ++ii)
          sum = sum + sres[(2 * cx + ii) + TX * ((2 * cy + jj) + TY * (DIM == 3 ? 2 * cz + kk : 0))];
    resc[gr.ci(I, J, K)] = sum;
  }
}

template <typename T, int DIM, int TX, int TY, int TZ, int HMAX, int NT, bool ODD>
__global__ __launch_bounds__(NT) void vc_relax_tile_kernel(VCArgs<T> A, const T* __restrict__ in,
                                                           T* __restrict__ out, const T* __restrict__ rhs, int npass,
                                                           int first, int zero_init, Geom gc,
                                                           const T* __restrict__ pc, int ntx, int nty, Geom gr,
                                                           T* __restrict__ resc, VCFinal<T> fin) {
  vc_relax_tile_body<T, DIM, TX, TY, TZ, HMAX, NT, ODD>(A, in, out, rhs, npass, first, zero_init, gc, pc, ntx, nty,
                                                        gr, resc, fin, int(blockIdx.x));
}

// batched form: workgroup w relaxes tile map[w] & mask of job map[w] >> bits
template <typename T, int DIM, int TX, int TY, int TZ, int HMAX, int NT>
__global__ __launch_bounds__(NT) void vc_relax_batch_kernel(const VCRelaxJob<T>* __restrict__ jobs,
                                                            const unsigned* __restrict__ map) {
  const unsigned w = map[blockIdx.x];
  const VCRelaxJob<T>& J = jobs[w >> kBatchTileBits];
  vc_relax_tile_body<T, DIM, TX, TY, TZ, HMAX, NT, false>(J.A, J.in, J.out, J.rhs, J.npass, J.first, J.zero_init, J.gc,
                                                          J.pc, J.ntx, J.nty, J.gr, J.resc, J.fin,
                                                          int(w & kBatchTileMask));
}

// Residual / operator / restricted residual over a tile with a one-cell halo.
// kVCResid: u = phi (+ e when e != nullptr, written to phi_out), res = rhs - L u
//           (res optional), max-norm into *norm (optional);
// kVCApply: out = L u;  kVCRestrict: out (coarse) = child sums of (rhs - L u)/2^d.
template <typename T, int DIM, int TX, int TY, int TZ, int MODE>
__device__ __forceinline__ void vc_tile_body(const VCArgs<T>& A, const VCTileIO<T>& io, int tile) {
  if (A.skip && *A.skip) return;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int EMAX = (TX + 2) * (TY + 2) * (DIM == 3 ? TZ + 2 : 1);
  constexpr int KMAX = (EMAX + kVCThreads - 1) / kVCThreads;
  const Geom& g = A.g;
  Tile<DIM, TX, TY, TZ> t;
  t.init_at(1, io.ntx, io.nty, tile);
  T* su = reinterpret_cast<T*>(smem_raw);
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));
  PosRec R[KMAX];
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) pos_record<DIM, TX, TY, TZ>(g, t, threadIdx.x + kk * kVCThreads, R[kk]);
  // owner data of the residual / operator modes, loaded with the state
  Faces1<T, DIM> OF[KMAX];
  T oaq[KMAX], ocv[KMAX], orhs[KMAX], v[KMAX], ev[KMAX];
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    v[kk] = T(0);
    ev[kk] = T(0);
    if (r.kind != 1) continue;
    v[kk] = io.phi[r.q];
    if (io.e) ev[kk] = io.e[r.q];
  }
  if (MODE == kVCResid || MODE == kVCApply) {
#pragma unroll
    for (int kk = 0; kk < KMAX; ++kk) {
      const PosRec& r = R[kk];
      if (!r.owner) continue;
      load_faces1<T, DIM>(A, r.i, r.j, r.k, OF[kk]);
      oaq[kk] = A.a ? A.a[r.q] : T(1);
      ocv[kk] = A.c ? A.c[r.q] : T(0);
      if (MODE == kVCResid) orhs[kk] = io.rhs[r.q];
    }
  }
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.kind != 1) continue;
    T val = v[kk];
    if (io.e) val = val + ev[kk];
    su[r.e] = val;
  }
  __syncthreads();
#pragma unroll
  for (int kk = 0; kk < KMAX; ++kk) {
    const PosRec& r = R[kk];
    if (r.kind != 2) continue;
    const T v = io.homog ? T(0) : T(A.bc.val[r.gd][r.gs][0]);
    su[r.e] = bc_ghost<T>(A.bc.type[r.gd][r.gs][0], v, su[r.eint], r.gs == 0 ? -1 : 1, T(g.dx));
  }
  __syncthreads();
  if (MODE == kVCResid || MODE == kVCApply) {
    T mx = T(0);
    int nan = 0;
#pragma unroll
    for (int kk = 0; kk < KMAX; ++kk) {
      const PosRec& r = R[kk];
      if (!r.owner) continue;
      if (MODE == kVCResid && io.e) io.phi_out[r.q] = su[r.e];
      T st[7];
      gather_lds<T, DIM>(su, r.e, t.EX, t.EXY, st);
      const T lof = vc_lof<T, DIM>(OF[kk], st, oaq[kk], A.c != nullptr, ocv[kk], A.alpha, A.beta, dxinv);
      if (MODE == kVCResid) {
        const T res = orhs[kk] - lof;
        if (io.out) io.out[r.q] = res;
        const T ar = fabs(res);
        if (ar != ar) nan = 1;
        else if (ar > mx) mx = ar;
      } else {
        io.out[r.q] = lof;
      }
    }
    if (MODE == kVCResid && (io.norm || io.fuse.ctl))
      block_max_atomic<T>(mx, nan, ctl_slot(io.norm, io.fuse), io.fuse);
    return;
  }
  // kVCRestrict (RESTRICTRESDB, src/DarcyBrinkmanOpF.ChF:402-509)
  constexpr int NC = TX * TY * (DIM == 3 ? TZ : 1);
  T* sres = su + t.E;
  const T denom = DIM == 3 ? T(8) : T(4);
  for (int c = threadIdx.x; c < NC; c += blockDim.x) {
    const int cx = c % TX, cr = c / TX, cy = cr % TY, cz = cr / TY;
    const int gi = t.x0 + cx, gj = t.y0 + cy, gk = DIM == 3 ? t.z0 + cz : 0;
    if (gi >= g.n[0] || gj >= g.n[1] || (DIM == 3 && gk >= g.n[2])) continue;
    const int e = (cx + 1) + t.EX * (cy + 1) + t.EXY * (DIM == 3 ? cz + 1 : 0);
    const long long q = g.ci(gi, gj, gk);
    Faces1<T, DIM> F;
    load_faces1<T, DIM>(A, gi, gj, gk, F);
    const T aq = A.a ? A.a[q] : T(1);
    const T cv = A.c ? A.c[q] : T(0);
    T st[7];
    gather_lds<T, DIM>(su, e, t.EX, t.EXY, st);
    const T lof = vc_lof<T, DIM>(F, st, aq, A.c != nullptr, cv, A.alpha, A.beta, dxinv);
    sres[c] = (io.rhs[q] - lof) / denom;
  }
  __syncthreads();
  constexpr int CX = TX / 2, CY = TY / 2, CZ = DIM == 3 ? TZ / 2 : 1;
  constexpr int NCC = CX * CY * CZ;
  const Geom gcc = io.gc;
  for (int c = threadIdx.x; c < NCC; c += blockDim.x) {
    const int cx = c % CX, cr = c / CX, cy = cr % CY, cz = cr / CY;
    const int I = t.x0 / 2 + cx, J = t.y0 / 2 + cy, K = DIM == 3 ? t.z0 / 2 + cz : 0;
    if (I >= gcc.n[0] || J >= gcc.n[1] || (DIM == 3 && K >= gcc.n[2])) continue;
    T s = T(0);
    for (int kk = 0; kk < (DIM == 3 ? 2 : 1); ++kk)
      for (int jj = 0; jj < 2; ++jj)
        for (int ii = 0; ii < 2; ++ii)
          s = s + sres[(2 * cx + ii) + TX * ((2 * cy + jj) + TY * (DIM == 3 ? 2 * cz + kk : 0))];
    io.out[gcc.ci(I, J, K)] = s;
  }
}

template <typename T, int DIM, int TX, int TY, int TZ, int MODE>
__global__ __launch_bounds__(kVCThreads) void vc_tile_kernel(VCArgs<T> A, VCTileIO<T> io) {
  vc_tile_body<T, DIM, TX, TY, TZ, MODE>(A, io, int(blockIdx.x));
}

// batched residuals: workgroup w computes tile map[w] & mask of job map[w] >> bits
template <typename T, int DIM, int TX, int TY, int TZ>
__global__ __launch_bounds__(kVCThreads) void vc_resid_batch_kernel(const VCResidJob<T>* __restrict__ jobs,
                                                                    const unsigned* __restrict__ map) {
  const unsigned w = map[blockIdx.x];
  const VCResidJob<T>& J = jobs[w >> kBatchTileBits];
  vc_tile_body<T, DIM, TX, TY, TZ, kVCResid>(J.A, J.io, int(w & kBatchTileMask));
}

// batched 8-byte copies and zero fills: workgroup w handles chunk map[w] &
// mask of job map[w] >> bits
__global__ __launch_bounds__(256) void words_batch_kernel(const WordsJob* __restrict__ jobs,
                                                          const unsigned* __restrict__ map) {
  const unsigned w = map[blockIdx.x];
  const WordsJob& J = jobs[w >> kBatchTileBits];
  const long long c0 = (long long)(w & kBatchTileMask) * kWordsChunk;
  const long long c1 = c0 + kWordsChunk < J.n ? c0 + kWordsChunk : J.n;
  for (long long i = c0 + threadIdx.x; i < c1; i += 256) J.dst[i] = J.src ? J.src[i] : 0ull;
}

// ---------------------------------------------------------------------------
// Single-workgroup V-cycle over the small levels of a device descriptor.  The
// correction, right-hand side, lambda, faces, a and c of every level live in
// LDS for the whole cycle (compact, x fastest, levels one after another;
// faces as one block, read once).
//
// A wavefront alone on its SIMD issues an operation every 8 cycles whether it
// depends on the last one or not, and a branch costs four of them: the count
// of instructions along a visit bounds it.  Each thread owns one cell of each
// colour of a level (even row length) or the cells t and t + 512, with their
// data in registers; a wall's ghost is written by its cell's owner with each
// update, into a slot that the stencil reads like any neighbour; offsets come
// from the host.  Levels whose owners fit one wavefront are visited by wave 0
// alone.  The visits are one runtime loop: every launch fetches the code it
// runs.  Measured with BiCGStab bottoms, against per-visit geometry and
// shuffled dot products: five 2D levels from 32x32 63 -> 46 us a launch, two
// levels from 44x20 (bottom 22x10) 165 -> 115; a visit is now some 6.5K
// cycles, half of them its set-up.

// levels one launch may hold; 1024 cells make at most 5 (2D) or 3 (3D): no side falls below 2
constexpr int kVCL = kVCCoarseLevels;
template <int DIM>
struct VCLevels {
  static constexpr int n = DIM == 3 ? 4 : kVCL;
};

// x of lane ^ 2^k, k < 5 (DPP within rows of 16, a row swap)
template <int K>
__device__ __forceinline__ int lane_xor32(int x) {
  if constexpr (K == 0) return __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, true);    // quad_perm 1,0,3,2
  if constexpr (K == 1) return __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, true);    // quad_perm 2,3,0,1
  if constexpr (K == 2)   // half mirror (^7), then reversed quads (^3)
    return __builtin_amdgcn_update_dpp(0, __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, true), 0x1B, 0xF, 0xF, true);
  if constexpr (K == 3) return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, true);   // row rotated by 8
  return x;
}
template <int K>
__device__ __forceinline__ double lane_add(double s) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(s);
  const int lo = int(u), hi = int(u >> 32);
  if constexpr (K < 4) {
    const unsigned long long o =
        (unsigned long long)unsigned(lane_xor32<K>(lo)) | ((unsigned long long)unsigned(lane_xor32<K>(hi)) << 32);
    return s + __longlong_as_double((long long)o);
  } else {
    // both halves of each swapped pair in every lane: the same sum everywhere
    auto swap = [](int x) {
      if constexpr (K == 4) return __builtin_amdgcn_permlane16_swap(x, x, false, false);
      else return __builtin_amdgcn_permlane32_swap(x, x, false, false);
    };
    const auto a = swap(lo), b = swap(hi);
    const double p = __longlong_as_double((long long)((unsigned long long)unsigned(a[0]) | ((unsigned long long)unsigned(b[0]) << 32)));
    const double q = __longlong_as_double((long long)((unsigned long long)unsigned(a[1]) | ((unsigned long long)unsigned(b[1]) << 32)));
    return p + q;
  }
}
// the pairwise tree s_t + s_{t+h}, h = P/2 .. 1, over the first P lanes (P a
// power of two); the value of lane 0, uniform.  (Each node adds the same two
// values in either order.)
__device__ __forceinline__ double lane_tree(double s, int P) {
  if (P > 32) s = lane_add<5>(s);
  if (P > 16) s = lane_add<4>(s);
  if (P > 8) s = lane_add<3>(s);
  if (P > 4) s = lane_add<2>(s);
  if (P > 2) s = lane_add<1>(s);
  if (P > 1) s = lane_add<0>(s);
  const unsigned long long u = (unsigned long long)__double_as_longlong(s);
  const unsigned lo = __builtin_amdgcn_readfirstlane(int(u)), hi = __builtin_amdgcn_readfirstlane(int(u >> 32));
  return __longlong_as_double((long long)((unsigned long long)lo | ((unsigned long long)hi << 32)));
}

// LDS of the coarse V-cycle in elements: corrections, right-hand sides and
// lambda of every level, a and c, ghost slots (or restriction terms), faces
struct VCLdsMap {
  int e, r, lm, a, c, x, f, end;
};
__host__ __device__ inline VCLdsMap vc_lds_map(int tot, int nfaces, bool hasa, bool hasc) {
  VCLdsMap M;
  M.e = 0;
  M.r = tot;
  M.lm = 2 * tot;
  M.a = 3 * tot;
  M.c = M.a + (hasa ? tot : 0);
  M.x = M.c + (hasc ? tot : 0);
  M.f = M.x + kVCWGCells;
  M.end = M.f + nfaces;
  return M;
}

// One cell's data of a level: neighbours as LDS indices (a wall's ghost in
// the owner's slot), faces, alpha*a, beta*c, lambda.
template <typename T, int DIM>
struct VCCell {
  int nb[2 * DIM], wall;   // wall: faces beyond the first wall
  T ws, wb;                // the first wall's ghost: ws*u + wb
  Faces1<T, DIM> F;
  T al, bc, lam;
};

// lof (vc_lof) of the cell whose value is u, neighbours from sm
template <typename T, int DIM>
__device__ __forceinline__ T vccell_lof(const VCCell<T, DIM>& X, const T* sm, T u, bool hasc, const VCDesc<T>& D, T beta,
                                        T dxinv) {
  T p[2 * DIM];
#pragma unroll
  for (int f = 0; f < 2 * DIM; ++f) p[f] = sm[X.nb[f]];
  if (X.wall) {
#pragma unroll
    for (int f = 1; f < 2 * DIM; ++f)
      if ((X.wall >> f) & 1) p[f] = fma(D.gs[f >> 1][f & 1], u, D.gb[f >> 1][f & 1]);
  }
  T s = X.F.v[1] * (p[1] - u) - X.F.v[0] * (u - p[0]) + X.F.v[3] * (p[3] - u) - X.F.v[2] * (u - p[2]);
  if (DIM == 3) s = s + X.F.v[5] * (p[5] - u) - X.F.v[4] * (u - p[4]);
  T lof = X.al * u;
  if (hasc) lof = lof - X.bc * u;
  return lof - beta * s * dxinv;
}

template <typename T, int DIM>
__device__ __forceinline__ void vccell_build(VCCell<T, DIM>& X, const VCDesc<T>& D, const VCLdsMap& M, const T* sm,
                                             const CLev& L, const int* fo, int i, int j, int k, int slot, bool hasa,
                                             bool hasc, T alpha, T beta, T dxinv, bool up, T* LM) {
  const int c = L.off + i + L.nx * j + L.nxy * k;
  const int iv[3] = {i, j, k};
  X.wall = 0;
  X.ws = X.wb = T(0);
#pragma unroll
  for (int d = DIM - 1; d >= 0; --d) {
    const int st = d == 0 ? 1 : (d == 1 ? L.nx : L.nxy);
    const int nd = L.n[d];
    const bool w = D.per[d] == 0;
    const bool lo = iv[d] == 0, hi = iv[d] == nd - 1;
    X.nb[2 * d] = M.e + (lo ? c + (nd - 1) * st : c - st);
    X.nb[2 * d + 1] = M.e + (hi ? c - (nd - 1) * st : c + st);
    if (w) {
      if (lo) X.nb[2 * d] = M.x + slot;
      if (hi) X.nb[2 * d + 1] = M.x + slot;
      if (lo || hi) {
        X.ws = lo ? D.gs[d][0] : D.gs[d][1];
        X.wb = lo ? D.gb[d][0] : D.gb[d][1];
        X.wall |= (lo ? 1 << (2 * d) : 0) | (hi ? 2 << (2 * d) : 0);
      }
    }
  }
  X.wall &= X.wall - 1;   // (the first wall is the lowest bit)
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int fx = L.n[0] + (d == 0), fy = L.n[1] + (d == 1);
    const int at = M.f + fo[d] + i + fx * (j + (DIM == 3 ? fy * k : 0));
    X.F.v[2 * d] = sm[at];
    X.F.v[2 * d + 1] = sm[at + (d == 0 ? 1 : (d == 1 ? fx : fx * fy))];
  }
  const T aq = hasa ? sm[M.a + c] : T(1), cq = hasc ? sm[M.c + c] : T(0);
  X.al = alpha * aq;
  X.bc = beta * cq;
  if (up) {
    X.lam = LM[c];
  } else {
    X.lam = vc_lambda<T, DIM>(X.F, aq, hasc, cq, alpha, beta, dxinv);
    LM[c] = X.lam;
  }
}

// BiCGStab on the coarsest level L from its relaxed correction: L e = r with
// homogeneous BCs, preconditioner preCond (e = lambda*r, then two red/black
// iterations).  Preconditioned BiCGStab with restarts; eps 1e-6, reps 1e-12,
// hang 1e-8, small 1e-30, 5 restarts, L2 norms.  Dot products in a fixed
// order: 64 interleaved lane sums over the compact cell index, then the tree
// of lane_tree over the smallest power of two of lanes >= min(N, 64).
//
// Thread t holds cell t (and t + 512) of every vector in registers; only the
// vector under the operator passes through LDS, with its ghosts.  Up to 64
// cells wave 0 works alone and a dot product needs no LDS at all (the tree is
// lane swaps: 18 operations, where six 64-bit shuffles were some 700 cycles);
// beyond, the products pass through LDS, two buffers used in turn, one
// barrier each.  One copy of preconditioner and operator serves both halves
// of an iteration.  sm[z..]: the operator's vector (the level's corrections),
// sm[dot..]: 2*N values.
template <typename T, int DIM>
__device__ __forceinline__ void vcx_bicgstab(const VCDesc<T>& D, const VCLdsMap& M, T* sm, const CLev& L, const int* fo,
                                             bool hasa, bool hasc, T alpha, T beta, int imax, int dot0) {
  const int N = L.N;
  const bool small = N <= 64, two = N > kVCWG;
  if (small && threadIdx.x >= 64) return;   // (the caller syncs the workgroup)
  const int tid = threadIdx.x, lane = tid & 63;
  auto sync = [&]() __attribute__((always_inline)) {
    if (small)
      wave_sync();
    else
      __syncthreads();
  };
  const T dx = T(L.dx);
  const T dxinv = T(1) / (dx * dx);
  T* Z = sm + M.e + L.off;
  const T* rhs = sm + M.r + L.off;
  VCCell<T, DIM> X[2];
  bool own[2];
  int col[2];
  T ph[2], r[2], rt[2], e[2], p[2], pt[2], vv[2], f[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int c = tid + m * kVCWG;
    own[m] = c < N && (m == 0 || two);
    ph[m] = r[m] = rt[m] = e[m] = p[m] = pt[m] = vv[m] = f[m] = T(0);
    col[m] = 0;
    if (!own[m]) continue;
    int i, j, k;
    clev_coords(L, c, i, j, k);
    col[m] = (i + j + k) & 1;
    vccell_build<T, DIM>(X[m], D, M, sm, L, fo, i, j, k, c, hasa, hasc, alpha, beta, dxinv, true, sm + M.lm);
    ph[m] = Z[c];
    f[m] = rhs[c];
  }
  auto put = [&](int m, T v) __attribute__((always_inline)) {
    Z[tid + m * kVCWG] = v;
    sm[M.x + tid + m * kVCWG] = fma(X[m].ws, v, X[m].wb);
  };
  int P2 = 1;
  while (P2 < 64 && P2 < N) P2 <<= 1;
  int buf = 0;
  auto dot = [&](const T* x, const T* y) __attribute__((always_inline)) {
    T s = T(0);
    if (small) {
      if (own[0]) s = s + x[0] * y[0];
    } else {
      T* q = sm + dot0 + buf * N;
      buf ^= 1;
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (own[m]) q[tid + m * kVCWG] = x[m] * y[m];
      __syncthreads();
      for (int c = lane; c < N; c += 64) s = s + q[c];
    }
    return lane_tree(s, P2);
  };
  const T eps = T(1e-6), reps = T(1e-12), hang = T(1e-8), tiny = T(1e-30);
  T norm0 = T(0), norm1 = T(0), r0 = T(0);
  T rho0 = 0, rho1 = 0, alpha0 = 0, alpha1 = 0, omega0 = 0, omega1 = 0;
  bool init = true, fresh = true, begin = true;
  int restarts = 0, recount = 0, it = 0;
  for (;;) {
    if (fresh) {
      // residual of phi (at the start, and after a restart)
      fresh = false;
      sync();
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (own[m]) put(m, ph[m]);
      sync();
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        if (!own[m]) continue;
        r[m] = f[m] - vccell_lof<T, DIM>(X[m], sm, ph[m], hasc, D, beta, dxinv);
        rt[m] = r[m];
        e[m] = T(0);
      }
      norm0 = sqrt(dot(r, r));
      if (begin) {
        begin = false;
        norm1 = norm0;
        r0 = norm0;
      } else {
        rho0 = alpha0 = omega0 = T(0);
        ++restarts;
        init = true;
      }
    }
    if (!(it < imax && norm0 > eps * norm1 && norm1 > T(0))) break;
    ++it;
    norm1 = norm0;
    alpha1 = alpha0;
    omega1 = omega0;
    rho1 = rho0;
    rho0 = dot(rt, r);
    if (rho0 == T(0)) break;
    if (init) {
      p[0] = r[0];
      p[1] = r[1];
      init = false;
    } else {
      const T bt = (rho0 / rho1) * (alpha1 / omega1);
      const T sv = -bt * omega1;
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        T q = bt * p[m];
        q = q + sv * vv[m];
        p[m] = q + T(1) * r[m];
      }
    }
    // half 0: pt = preCond(p), v = L pt; half 1: st = preCond(r), t = L st
#pragma unroll 1
    for (int half = 0; half < 2; ++half) {
      T g[2], z[2], w[2] = {T(0), T(0)};
      sync();   // the last operator's reads are done
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        g[m] = half ? r[m] : p[m];
        z[m] = T(0);
        if (!own[m]) continue;
        z[m] = g[m] * X[m].lam;
        put(m, z[m]);
      }
      sync();
#pragma unroll 1
      for (int pass = 0; pass < 5; ++pass) {
        // four colour passes, then the operator at every cell
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          if (!own[m] || (pass < 4 && col[m] != (pass & 1))) continue;
          const T lof = vccell_lof<T, DIM>(X[m], sm, z[m], hasc, D, beta, dxinv);
          if (pass < 4) {
            z[m] = z[m] - X[m].lam * (lof - g[m]);
            put(m, z[m]);
          } else {
            w[m] = lof;
          }
        }
        if (pass < 4) sync();
      }
      if (half == 0) {
        pt[0] = z[0];
        pt[1] = z[1];
        vv[0] = w[0];
        vv[1] = w[1];
        const T mm = dot(rt, vv);
        alpha0 = rho0 / mm;
        if (fabs(mm) > tiny * fabs(rho0)) {
          const T na = -alpha0;
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            r[m] = r[m] + na * vv[m];
            e[m] = e[m] + alpha0 * pt[m];
          }
          norm0 = sqrt(dot(r, r));
        } else {
          r[0] = r[1] = T(0);
          norm0 = T(0);
        }
        if (!(norm0 > eps * r0 && norm0 > reps * r0)) break;
      } else {
        const T tr = dot(w, r), tt = dot(w, w);
        omega0 = tr / tt;
        const T nw = -omega0;
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          e[m] = e[m] + omega0 * z[m];
          r[m] = r[m] + nw * w[m];
        }
        norm0 = sqrt(dot(r, r));
      }
    }
    if (norm0 <= eps * r0 || norm0 <= reps * r0) break;
    if (omega0 == T(0) || norm0 > (T(1) - hang) * norm1) {
      if (recount == 0) {
        recount = 1;
      } else {
        recount = 0;
        ph[0] = ph[0] + T(1) * e[0];
        ph[1] = ph[1] + T(1) * e[1];
        if (restarts == 5) {
          e[0] = e[1] = T(0);
          break;
        }
        fresh = true;
      }
    }
  }
  sync();
#pragma unroll
  for (int m = 0; m < 2; ++m)
    if (own[m]) Z[tid + m * kVCWG] = ph[m] + T(1) * e[m];
}

template <typename T, int DIM>
__device__ __forceinline__ void vc_coarse_vcycle_body(const VCDesc<T>* __restrict__ Dp) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  constexpr int LL = VCLevels<DIM>::n;
  typedef T vec2 __attribute__((ext_vector_type(2)));
  const VCDesc<T>& D = *Dp;
  if (D.skip && *D.skip) return;
  const int tid = threadIdx.x;
  const int nl = D.nl, tot = D.tot, N0 = D.off[1];
  const bool hasc = D.c[0] != nullptr, hasa = D.a[0] != nullptr;
  const T alpha = D.alpha, beta = D.beta;
  const VCLdsMap M = vc_lds_map(tot, D.nfaces, hasa, hasc);
  T* sm = reinterpret_cast<T*>(smem_raw);
  T *E = sm + M.e, *R = sm + M.r, *LM = sm + M.lm, *SX = sm + M.x;
  auto level_of = [&](int l) __attribute__((always_inline)) {
    CLev L;
    for (int d = 0; d < 3; ++d) L.n[d] = d < DIM ? D.n[d] >> l : 1;
    L.nx = L.n[0];
    L.nxy = L.n[0] * L.n[1];
    L.off = D.off[l];
    L.N = D.off[l + 1] - L.off;
    L.dx = D.dx * double(1 << l);
    return L;
  };
  const CLev L0 = level_of(0);
  // right-hand side of the first level, a and c of all levels, the faces: all
  // global loads first
  auto fab = [&](const CLev& L, int c) __attribute__((always_inline)) {
    int i, j, k;
    clev_coords(L, c, i, j, k);
    const int sy = L.n[0] + 2, sz = sy * (L.n[1] + 2);
    return (i + 1) + sy * (j + 1) + (DIM == 3 ? sz * (k + 1) : 0);
  };
  T r0[2];
  int q0[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int c = tid + m * kVCWG;
    if (c >= N0) continue;
    q0[m] = fab(L0, c);
    r0[m] = D.r[q0[m]];
  }
  if (hasc || hasa) {
    // level 0: cells t and t + 512; coarser levels: cell t
    T cv[LL + 1], av[LL + 1];
#pragma unroll
    for (int l = 0; l < LL; ++l) {
      if (l >= nl) continue;
      const CLev L = level_of(l);
#pragma unroll
      for (int m = 0; m < (l ? 1 : 2); ++m) {
        const int c = tid + m * kVCWG;
        if (c >= L.N) continue;
        const int q = l ? fab(L, c) : q0[m];
        if (hasc) cv[l + (l ? 1 : m)] = D.c[l][q];
        if (hasa) av[l + (l ? 1 : m)] = D.a[l][q];
      }
    }
#pragma unroll
    for (int l = 0; l < LL; ++l) {
      if (l >= nl) continue;
#pragma unroll
      for (int m = 0; m < (l ? 1 : 2); ++m) {
        const int c = tid + m * kVCWG;
        if (c >= D.off[l + 1] - D.off[l]) continue;
        if (hasc) sm[M.c + D.off[l] + c] = cv[l + (l ? 1 : m)];
        if (hasa) sm[M.a + D.off[l] + c] = av[l + (l ? 1 : m)];
      }
    }
  }
  {
    constexpr int KF = 4;
    const vec2* src = reinterpret_cast<const vec2*>(D.faces);
    T* dst = sm + M.f;
    const int n2 = D.nfaces >> 1;
#pragma unroll 1
    for (int base = tid; base < n2; base += KF * kVCWG) {
      vec2 v[KF];
#pragma unroll
      for (int k = 0; k < KF; ++k)
        if (base + k * kVCWG < n2) v[k] = src[base + k * kVCWG];
#pragma unroll
      for (int k = 0; k < KF; ++k)
        if (base + k * kVCWG < n2) {
          dst[2 * (base + k * kVCWG)] = v[k].x;
          dst[2 * (base + k * kVCWG) + 1] = v[k].y;
        }
    }
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
    if (tid + m * kVCWG < N0) R[tid + m * kVCWG] = r0[m];
  __syncthreads();

#pragma unroll 1
  for (int v = 0; v < 2 * nl - 1; ++v) {
    const bool up = v >= nl, bot = v == nl - 1, down = v < nl - 1;
    const int l = up ? 2 * nl - 2 - v : v;
    const CLev L = level_of(l);
    const int off = L.off, offc = off + L.N;
    const bool even = (L.nx & 1) == 0;
    const bool small = cown_active<kVCWG>(L) <= 64;
    const int step = small ? 64 : kVCWG;   // threads of this visit
    const T dx = T(L.dx);
    const T dxinv = T(1) / (dx * dx);
    auto sync = [&]() __attribute__((always_inline)) {
      if (small)
        wave_sync();
      else
        __syncthreads();
    };
    int fo[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) fo[d] = D.fo[l][d];
    if (!small || tid < 64) {
      COwn o;
      cown_set<kVCWG>(L, o);
      VCCell<T, DIM> X[2];
      int c[2], col[2];
      T u[2], rr[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        c[m] = 0;
        if (o.p[m] < 0) continue;
        int i, j, k;
        cunpack(o.p[m], i, j, k);
        c[m] = i + L.nx * j + L.nxy * k;
        col[m] = (i + j + k) & 1;
        vccell_build<T, DIM>(X[m], D, M, sm, L, fo, i, j, k, m * kVCWG + tid, hasa, hasc, alpha, beta, dxinv, up, LM);
        rr[m] = R[off + c[m]];
        // from zero on the way down, e_f + e_c(parent) on the way up
        u[m] = T(0);
        if (up)
          u[m] = E[off + c[m]] +
                 E[offc + (i >> 1) + (L.nx >> 1) * ((j >> 1) + (DIM == 3 ? (L.n[1] >> 1) * (k >> 1) : 0))];
      }
      auto put = [&](int m) __attribute__((always_inline)) {
        E[off + c[m]] = u[m];
        SX[m * kVCWG + tid] = fma(X[m].ws, u[m], X[m].wb);
      };
#pragma unroll
      for (int m = 0; m < 2; ++m)
        if (o.p[m] >= 0) put(m);
      sync();
      auto update = [&](auto MM) __attribute__((always_inline)) {
        constexpr int m = decltype(MM)::value;
        if (o.p[m] < 0) return;
        const T lof = vccell_lof<T, DIM>(X[m], sm, u[m], hasc, D, beta, dxinv);
        u[m] = u[m] - X[m].lam * (lof - rr[m]);
        put(m);
      };
      const int its = bot ? D.bottom : (up ? D.nu2 : D.nu1);
      if (even) {
#pragma unroll 1
        for (int it = 0; it < its; ++it) {
          update(IC<0>{});
          sync();
          update(IC<1>{});
          sync();
        }
      } else {
#pragma unroll 1
        for (int p = 0; p < 2 * its; ++p) {
          if (o.p[0] >= 0 && col[0] == (p & 1)) update(IC<0>{});
          if (o.p[1] >= 0 && col[1] == (p & 1)) update(IC<1>{});
          sync();
        }
      }
      if (down) {
        // restricted residual (homogeneous BCs, RESTRICTRESDB order)
        const T rdenom = DIM == 3 ? T(0.125) : T(0.25);
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (o.p[m] >= 0) rr[m] = (rr[m] - vccell_lof<T, DIM>(X[m], sm, u[m], hasc, D, beta, dxinv)) * rdenom;
        sync();   // the ghosts in SX have been read
#pragma unroll
        for (int m = 0; m < 2; ++m)
          if (o.p[m] >= 0) SX[c[m]] = rr[m];
        sync();
        const CLev C = level_of(l + 1);
#pragma unroll 1
        for (int cc = tid; cc < C.N; cc += step) {
          int I, J, K;
          clev_coords(C, cc, I, J, K);
          const int f0 = 2 * I + L.nx * (2 * J) + (DIM == 3 ? L.nxy * (2 * K) : 0);
          T s = T(0);
#pragma unroll
          for (int kk = 0; kk < (DIM == 3 ? 2 : 1); ++kk)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj)
#pragma unroll
              for (int ii = 0; ii < 2; ++ii) s = s + SX[f0 + ii + L.nx * jj + L.nxy * kk];
          R[offc + cc] = s;
        }
      }
    }
    if (bot && D.bottom_solver == 1) {
      if (!small) __syncthreads();
      if (small && L.N > 64) __syncthreads();   // all waves join the solver
      vcx_bicgstab<T, DIM>(D, M, sm, L, fo, hasa, hasc, alpha, beta, D.bottom_imax, M.end);
    }
    // the next visit reads what this one wrote: wave 0 alone where both are
    // small, else the workgroup
    bool next_small = false;
    if (small && !(bot && D.bottom_solver == 1 && L.N > 64) && v + 1 < 2 * nl - 1)
      next_small = cown_active<kVCWG>(level_of(v + 1 >= nl ? 2 * nl - 3 - v : v + 1)) <= 64;
    if (!next_small)
      __syncthreads();
    else if (tid < 64)
      wave_sync();
  }
#pragma unroll
  for (int m = 0; m < 2; ++m)
    if (tid + m * kVCWG < N0) D.e[q0[m]] = E[tid + m * kVCWG];
}

template <typename T, int DIM>
__global__ __launch_bounds__(kVCWG) void vc_coarse_vcycle_kernel(const VCDesc<T>* __restrict__ Dp) {
  vc_coarse_vcycle_body<T, DIM>(Dp);
}

// batched form: workgroup w runs the coarse V-cycle of descriptor descs[w]
template <typename T, int DIM>
__global__ __launch_bounds__(kVCWG) void vc_coarse_batch_kernel(const VCDesc<T>* const* __restrict__ descs) {
  // the descriptor address is uniform over the workgroup: keep it scalar
  const unsigned long long a = reinterpret_cast<unsigned long long>(descs[blockIdx.x]);
  const unsigned lo = __builtin_amdgcn_readfirstlane(unsigned(a)), hi = __builtin_amdgcn_readfirstlane(unsigned(a >> 32));
  vc_coarse_vcycle_body<T, DIM>(reinterpret_cast<const VCDesc<T>*>((static_cast<unsigned long long>(hi) << 32) | lo));
}

template <int DIM>
struct VCRelaxTile;
template <>
struct VCRelaxTile<2> {
  static constexpr int TX = 16, TY = 16, TZ = 1, HMAX = 9, NT = 1024;   // measured best of 11 shapes at 256^2
};
template <>
struct VCRelaxTile<3> {
  // 1024 threads: two staged positions per thread, no register spill (19 %
  // faster at 128^3 than 512 threads)
  static constexpr int TX = 16, TY = 8, TZ = 4, HMAX = 2, NT = 1024;
};
// batches with many cells are bandwidth-bound: a 32x32 core restages fewer
// halo cells per owned cell (2.4x at the 9-cell halo, 4.5x for 16x16)
struct VCRelaxBatchWide2 {
  static constexpr int TX = 32, TY = 32, TZ = 1, HMAX = 9, NT = 1024;
};
template <int DIM>
struct VCTile;
template <>
struct VCTile<2> {
  static constexpr int TX = 32, TY = 8, TZ = 1;
};
template <>
struct VCTile<3> {
  static constexpr int TX = 16, TY = 8, TZ = 4;
};

template <int TX, int TY, int TZ>
int vc_tiles(const Geom& g, int& ntx, int& nty) {
  ntx = (g.n[0] + TX - 1) / TX;
  nty = (g.n[1] + TY - 1) / TY;
  const int ntz = g.dim == 3 ? (g.n[2] + TZ - 1) / TZ : 1;
  return ntx * nty * ntz;
}

template <typename T, int DIM, typename D>
hipError_t vc_relax_cfg(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                        const Geom* gc, const T* pc, hipStream_t s, const Geom* gr, T* resc, const LaunchTimer* tm,
                        const VCFinal<T>* fin) {
  int ntx, nty;
  const int nt = vc_tiles<D::TX, D::TY, D::TZ>(A.g, ntx, nty);
  const Geom gcc = gc ? *gc : A.g;
  const Geom grr = gr ? *gr : A.g;
  if ((resc || fin) && npass + 1 > D::HMAX) return hipErrorInvalidValue;
  bool odd = false;
  for (int d = 0; d < DIM; ++d) odd = odd || (A.g.periodic[d] && (A.g.n[d] & 1));
  odd = odd && npass > 0;
  if (odd && (DIM != 2 || resc || fin)) return hipErrorInvalidValue;   // (such a level does not coarsen)
  const VCFinal<T> none{};
  int done = 0;
  bool first_launch = true;
  while (done < npass || (first_launch && npass == 0 && (zero_init || pc || resc))) {
    first_launch = false;
    const int p = (npass - done) < D::HMAX ? (npass - done) : D::HMAX;
    const int h = p + ((resc || fin) ? 1 : 0);
    size_t lds = size_t(D::TX + 2 * h) * (D::TY + 2 * h) * (DIM == 3 ? D::TZ + 2 * h : 1);
    if (resc) lds += size_t(D::TX) * D::TY * D::TZ;
    if (fin) lds *= 2;   // e and u = phi + e
    const bool timed = tm && *tm->n < tm->cap;
    if (tm && !timed) ++*tm->missed;
    const bool zi = done == 0 && zero_init;
    const T* pcl = done == 0 ? pc : nullptr;
    // a timed launch carries its start and stop events in the dispatch
    auto kern = odd ? vc_relax_tile_kernel<T, DIM, D::TX, D::TY, D::TZ, D::HMAX, D::NT, DIM == 2>
                    : vc_relax_tile_kernel<T, DIM, D::TX, D::TY, D::TZ, D::HMAX, D::NT, false>;
    hipExtLaunchKernelGGL(kern, dim3(nt), dim3(D::NT), lds * sizeof(T), s, timed ? tm->start[*tm->n] : nullptr,
                          timed ? tm->stop[*tm->n] : nullptr, 0, A, buf[*cur], buf[1 - *cur], rhs, p, done & 1,
                          zi ? 1 : 0, gcc, pcl, ntx, nty, grr, resc, fin ? *fin : none);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (timed) {
      // algorithmic bytes: state in (unless zero start), coarse correction,
      // rhs, a, c, faces once each; state out and restricted residual once
      const double cells = double(A.g.nvalid());
      const double coarse = cells / double(DIM == 3 ? 8 : 4);
      double faces = 0;
      for (int d = 0; d < DIM; ++d) faces += double(A.g.nface[d]);
      double b = cells * (zi ? 0 : 1) + (pcl ? coarse : 0) + cells + (A.a ? cells : 0) + (A.c ? cells : 0) + faces;
      b += cells + (resc ? coarse : 0);
      if (fin) b += 2 * cells + 2 * cells;   // phi and the full rhs in; phi + e and the residual out
      *tm->bytes += b * sizeof(T);
      ++*tm->n;
    }
    *cur = 1 - *cur;
    done += p;
  }
  return hipSuccess;
}

// ---- streaming relaxation for large 2D levels ----------------------------
// A workgroup owns TX columns and a segment of rows ("planes" below), and
// marches through them with a window of P+2 planes in LDS.  With plane R just
// loaded, colour pass p runs on plane R-1-p (p = 0..P-1), so plane R-P is
// final and is written: the passes form a pipeline along the march instead
// of a halo in that direction.  Pass p covers the lateral positions within
// P-1-p of the block and the planes within P-1-p of the segment, so the
// core ends exact after P passes, as in the tiled kernel.  Every input value
// of the extended block is read once per launch; a plane's coefficients
// stay in registers for the P steps that use them and are loaded one plane
// ahead of their first use, so their loads overlap the previous plane's
// passes.  Stencil, lambda and update are the tiled kernel's, so results
// are identical bit for bit.  SEAM: the rows are periodic with an odd length,
// so the two cells at their seam share a colour and read each other as of the
// start of a pass.
template <typename T>
struct SCoef {
  Faces1<T, 2> F;
  T aq, cq, rr, lam;
};

template <typename T, int TX, int P, int NT, bool SEAM>
__global__ __launch_bounds__(NT) void vc_relax_stream_kernel(VCArgs<T> A, const T* __restrict__ in,
                                                             T* __restrict__ out, const T* __restrict__ rhs,
                                                             int first, int zero_init, Geom gc,
                                                             const T* __restrict__ pc, int nbx, int seg) {
  if (A.skip && *A.skip) return;
  constexpr int EL = NT;   // positions of a plane: one a thread
  static_assert(TX + 2 * P == NT, "one position a thread");
  static_assert(P >= 1 && P <= 2, "one or two colour passes per launch");
  constexpr int W = 4;   // planes in the window (P+2 <= 4; a power of two)
  constexpr int MD = 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* su = reinterpret_cast<T*>(smem_raw);
  const Geom& g = A.g;
  const int nz = g.n[MD];
  const bool zper = g.periodic[MD] != 0;
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));
  const bool hasc = A.c != nullptr;
  const int bx = int(blockIdx.x) % nbx, bz = int(blockIdx.x) / nbx;
  const int x0 = bx * TX;
  const int z0 = bz * seg;
  const int z1 = z0 + seg < nz ? z0 + seg : nz;
  const int e = int(threadIdx.x);
  SPos s;
  spos_init<TX, P>(g, x0, e, s);
  s.gtype = 0;
  for (int sd = 0; sd < 2; ++sd)
    if (s.kind == 2 && s.gs == sd) s.gtype = A.bc.type[0][sd][0];
  auto zwrap = [&](int z) { return z < 0 ? z + nz : (z >= nz ? z - nz : z); };
  auto real_plane = [&](int z) { return zper || (z >= 0 && z < nz); };
  // 32-bit element offsets: a position's lateral part, computed once, plus a
  // plane part common to the workgroup (levels below 2^29 cells per array)
  const unsigned csz = unsigned(g.sy);   // cell stride between planes
  unsigned fpl[2], fup[2];                              // face plane stride, offset to the upper face
#pragma unroll
  for (int d = 0; d < 2; ++d) fpl[d] = unsigned(g.fn[d][0]);
  fup[0] = 1;
  fup[MD] = fpl[MD];
  const unsigned cgsz = unsigned(gc.sy);
  const unsigned cl = unsigned(s.gx + 1), fl = unsigned(s.gx), ccl = unsigned(s.gx / 2 + 1);
  auto ld = [](const T* p, unsigned i) -> T {
    return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + (i * unsigned(sizeof(T))));
  };
  // register sets of P+3 planes (R-P .. R+2 at step R), addressed by
  // compile-time indices: plane zl+m lives in set m % NS.  Loads go straight
  // into their set and are used only at that plane's commit two steps later,
  // so no instruction touches a load in flight.
  constexpr int NS = P + 3;
  SCoef<T> cs[NS];
  T sv[NS], scv[NS];   // state and coarse correction as loaded
  // the same loads for every position and plane (in-domain addresses; an
  // absent array is replaced by a duplicate read of rhs), so that the waits
  // for a set's loads can count the loads issued after it exactly
  const T* vin = zero_init ? rhs : in;
  const T* ain = A.a ? A.a : rhs;
  const T* cin = hasc ? A.c : rhs;
  const T* cvp = pc ? pc : rhs;
  auto prefetch = [&](int R, SCoef<T>& pf, T& v, T& cv) {
    const int zw = zper ? zwrap(R) : (R < 0 ? 0 : (R >= nz ? nz - 1 : R));
    const unsigned qz = unsigned(zw + 1) * csz, cz = unsigned(zw / 2 + 1) * cgsz;
    const unsigned q = cl + qz;   // a ghost reads its interior neighbour
    v = ld(vin, q);
    cv = ld(cvp, pc ? ccl + cz : q);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const unsigned f = fl + unsigned(zw) * fpl[d];
      pf.F.v[2 * d] = ld(A.b[d], f);
      pf.F.v[2 * d + 1] = ld(A.b[d], f + fup[d]);
    }
    pf.aq = ld(ain, q);
    pf.cq = ld(cin, q);
    pf.rr = ld(rhs, q);
  };
  const int zl = (!zper && z0 - P < 0) ? 0 : z0 - P;
  const int zend = z1 - 1 + P;   // last step: plane z1 - 1 is final
  // window slot of plane R (the bottom wall's ghost plane -1 is slot 3)
  auto slot = [&](int R) { return su + ((R - zl) & (W - 1)) * EL; };
  auto step = [&](auto J, int R) {
    constexpr int j = decltype(J)::value;
    // A. commit plane R (or the top wall's ghost plane)
    T* pl = slot(R);
    if (real_plane(R) && s.kind != 0) {
      T val = zero_init ? T(0) : sv[j];
      if (pc) val = val + scv[j];
      if (s.kind == 1) {
        pl[e] = val;
        if (!zper && R == 0) slot(-1)[e] = bc_ghost<T>(A.bc.type[MD][0][0], T(0), val, -1, T(g.dx));
        if (!A.a) cs[j].aq = T(1);
        if (!hasc) cs[j].cq = T(0);
        if (s.dist <= P - 1)
          cs[j].lam = vc_lambda<T, 2>(cs[j].F, cs[j].aq, hasc, cs[j].cq, A.alpha, A.beta, dxinv);
      } else {
        pl[e] = bc_ghost<T>(s.gtype, T(0), val, s.gs == 0 ? -1 : 1, T(g.dx));
      }
    } else if (!zper && R == nz && s.kind == 1) {
      const T* below = slot(nz - 1);
      pl[e] = bc_ghost<T>(A.bc.type[MD][1][0], T(0), below[e], 1, T(g.dx));
    }
    // B. loads of plane R+2 into the set of plane R+2-NS, no longer in use
    constexpr int jn = (j + 2) % NS;
    prefetch(R + 2, cs[jn], sv[jn], scv[jn]);   // beyond the segment: a clamped plane, unused
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
        const bool mine = s.kind == 1 && s.dist <= reach && !((s.gx + zw + first + p) & 1);
        T* pz = slot(z);
        const T* pm = slot(z - 1);
        const T* pp = slot(z + 1);
        auto value = [&]() __attribute__((always_inline)) {
          T st[7];
          st[0] = pz[e];
          st[1] = pz[e + 1];
          st[2] = pz[e - 1];
          st[3] = pp[e];
          st[4] = pm[e];
          const SCoef<T>& C = cs[jp];
          const T lof = vc_lof<T, 2>(C.F, st, C.aq, hasc, C.cq, A.alpha, A.beta, dxinv);
          return st[0] - C.lam * (lof - C.rr);
        };
        T nv;
        if constexpr (SEAM) {
          if (mine) nv = value();
          __syncthreads();   // the two cells at the seam read each other
        }
        if (mine) {
          if constexpr (!SEAM) nv = value();
          pz[e] = nv;
          // wall ghosts of this cell: lateral, then along the march
          if (!g.periodic[0]) {
            if (s.gx == 0) pz[e - 1] = bc_ghost<T>(A.bc.type[0][0][0], T(0), nv, -1, T(g.dx));
            if (s.gx == g.n[0] - 1) pz[e + 1] = bc_ghost<T>(A.bc.type[0][1][0], T(0), nv, 1, T(g.dx));
          }
          if (!zper) {
            if (zw == 0) slot(-1)[e] = bc_ghost<T>(A.bc.type[MD][0][0], T(0), nv, -1, T(g.dx));
            if (zw == nz - 1) slot(nz)[e] = bc_ghost<T>(A.bc.type[MD][1][0], T(0), nv, 1, T(g.dx));
          }
        }
      }
      __syncthreads();
    };
    pass(IC<0>{});
    if constexpr (P > 1) pass(IC<1>{});
    // D. plane R-P is final
    const int zs = R - P;
    if (zs >= z0 && zs < z1 && s.owner)
      *reinterpret_cast<T*>(reinterpret_cast<char*>(out) + ((cl + unsigned(zs + 1) * csz) * unsigned(sizeof(T)))) =
          slot(zs)[e];
  };
  prefetch(zl, cs[0], sv[0], scv[0]);
  prefetch(zl + 1, cs[1], sv[1], scv[1]);
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

struct VCStream {
  static constexpr int NT = 256, SEGMIN = 8;
};

// 2D levels on which plain relaxation launches stream (above 512^2); the
// tiled kernel keeps the fused restriction / residual.  Not with an odd
// periodic length along the march: the rows at its seam share colours, and a
// pass reaches one of them before the other.
constexpr long long kStreamCells2 = 512 * 512;
inline bool vc_streams(const Geom& g) {
  long long nf = 0;
  for (int d = 0; d < g.dim; ++d) nf = nf > g.nface[d] ? nf : g.nface[d];
  const long long most = g.ncell > nf ? g.ncell : nf;
  return g.dim == 2 && g.nvalid() > kStreamCells2 && g.n[1] >= 8 && !(g.periodic[1] && (g.n[1] & 1)) &&
         most < (1LL << 29);   // byte offsets of every array within 32 bits
}

template <typename T, int P, bool SEAM>
hipError_t vc_stream_launch(const VCArgs<T>& A, const T* in, T* out, const T* rhs, int first, bool zero_init,
                            const Geom& gc, const T* pc, hipStream_t s, const LaunchTimer* tm) {
  using D = VCStream;
  constexpr int TX = D::NT - 2 * P, EL = D::NT;
  const Geom& g = A.g;
  const int nbx = (g.n[0] + TX - 1) / TX;
  const size_t lds = size_t(4) * EL * sizeof(T);
  auto kern = vc_relax_stream_kernel<T, TX, P, D::NT, SEAM>;
  // segments sized so that the whole grid is resident at once (one round of
  // workgroups; measured best at 2048^2: a grid that fills every CU's
  // workgroup slots beats both fewer, longer segments and a second round)
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
                        timed ? tm->stop[*tm->n] : nullptr, 0, A, in, out, rhs, first, zero_init ? 1 : 0, gc, pc, nbx,
                        seg);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (timed) {
    const double cells = double(g.nvalid());
    double faces = 0;
    for (int d = 0; d < 2; ++d) faces += double(g.nface[d]);
    double by = cells * (zero_init ? 0 : 1) + (pc ? cells / 4 : 0) + cells +
                (A.a ? cells : 0) + (A.c ? cells : 0) + faces + cells;
    *tm->bytes += by * sizeof(T);
    ++*tm->n;
  }
  return hipSuccess;
}

// npass colour passes by streaming launches of up to 2 passes each
template <typename T>
hipError_t vc_relax_stream(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                           const Geom* gc, const T* pc, hipStream_t s, const LaunchTimer* tm) {
  const Geom gcc = gc ? *gc : A.g;
  const bool seam = A.g.periodic[0] && (A.g.n[0] & 1);
  int done = 0;
  while (done < npass) {
    const int p = (npass - done) >= 2 ? 2 : (npass - done);
    const bool zi = done == 0 && zero_init;
    const T* pcl = done == 0 ? pc : nullptr;
    auto launch = p == 2 ? (seam ? vc_stream_launch<T, 2, true> : vc_stream_launch<T, 2, false>)
                         : (seam ? vc_stream_launch<T, 1, true> : vc_stream_launch<T, 1, false>);
    const hipError_t e = launch(A, buf[*cur], buf[1 - *cur], rhs, done & 1, zi, gcc, pcl, s, tm);
    if (e != hipSuccess) return e;
    *cur = 1 - *cur;
    done += p;
  }
  return hipSuccess;
}

// the homogeneous wall ghosts of a correction
template <typename T>
GhostForm<T> vc_ghost_form(BCDesc bc, T dx) {
  bc.apply = 1;
  for (auto& d : bc.val)
    for (auto& s : d)
      for (auto& v : s) v = 0.0;
  return ghost_form<T>(bc, dx);
}

// One colour pass of a 3D level straight from memory (Sweep3).  MOVE: from
// `in`, or zero, plus the coarse correction pc, every cell written to `out`
// (the first pass, and every pass of the GEN form); otherwise in place on
// `out`.  Two passes with c: 37 us at 128^3 (92 bytes a cell needed, 102
// counted beyond the L2s: 5.8 TB/s; a march along z with a window of planes in
// LDS was 71), 8.5 at 64^3 and 7.5 at 16^3 (16 x 8 x 4 tiles with the halo of
// both passes: 15.1 and 8.0); GEN 50 at 129 x 128 x 128.
template <typename T, bool GEN>
struct VCSweep {
  Sweep3<GEN> S;
  const int* skip;
  const T* in;
  T* out;
  const T* rhs;
  const T* a;
  const T* c;
  const T* b[3];
  const T* pc;
  typename Sweep3<GEN>::Off csy, csz;   // coarse cell strides
  T alpha, beta, dxinv, gs[3][2], gb[3][2];
  int zero;
};
template <typename T, bool MOVE, bool GEN>
__global__ __launch_bounds__(256) void vc_sweep3_kernel(VCSweep<T, GEN> A) {
  using Off = typename Sweep3<GEN>::Off;
  if (A.skip && *A.skip) return;
  Sweep3Pos<GEN> P;
  if (!sweep3_pos(A.S, P)) return;
  auto val = [&](Off q, int i, int j, int k) __attribute__((always_inline)) {
    if (!MOVE) return get_at(A.out, q);
    T v = A.zero ? T(0) : get_at(A.in, q);
    if (A.pc) v = v + get_at(A.pc, Off((i >> 1) + 1) + A.csy * Off((j >> 1) + 1) + A.csz * Off((k >> 1) + 1));
    return v;
  };
  if (MOVE && P.oth) put_at(A.out, P.qo, val(P.qo, P.i, P.j, P.k));   // (both cells of a pair have one coarse cell)
  if (!P.act) return;
  T st[7];
  st[0] = val(P.q, P.i, P.j, P.k);
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    int iv[3] = {P.i, P.j, P.k};
    if (MOVE) {
      const int d = f >> 1, n = A.S.n[d];
      iv[d] = f & 1 ? (iv[d] == n - 1 ? (A.S.per[d] ? 0 : iv[d]) : iv[d] + 1)
                    : (iv[d] == 0 ? (A.S.per[d] ? n - 1 : 0) : iv[d] - 1);
    }
    st[1 + (f ^ 1)] = val(P.nb[f], iv[0], iv[1], iv[2]);
  }
  Faces1<T, 3> F;
#pragma unroll
  for (int d = 0; d < 3; ++d) sweep3_faces(A.S, P, d, A.b[d], F.v[2 * d], F.v[2 * d + 1]);
  const bool hasc = A.c != nullptr;
  const T aq = A.a ? get_at(A.a, P.q) : T(1), cq = hasc ? get_at(A.c, P.q) : T(0), rr = get_at(A.rhs, P.q);
  if (P.wall) {
#pragma unroll
    for (int f = 0; f < 6; ++f)
      if ((P.wall >> f) & 1) st[1 + (f ^ 1)] = fma(A.gs[f >> 1][f & 1], st[0], A.gb[f >> 1][f & 1]);
  }
  const T lam = vc_lambda<T, 3>(F, aq, hasc, cq, A.alpha, A.beta, A.dxinv);
  const T lof = vc_lof<T, 3>(F, st, aq, hasc, cq, A.alpha, A.beta, A.dxinv);
  put_at(A.out, P.q, st[0] - lam * (lof - rr));
}

// npass >= 1 colour passes: the first from buf[*cur] to the other buffer,
// the others in place there (GEN: each on to the other buffer)
template <typename T, bool GEN>
hipError_t vc_relax_sweeps(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                           const Geom* gc, const T* pc, hipStream_t s, const LaunchTimer* tm) {
  const Geom& g = A.g;
  using Off = typename Sweep3<GEN>::Off;
  VCSweep<T, GEN> V{};
  V.S = sweep3_make<GEN>(g);
  V.skip = A.skip;
  V.rhs = rhs;
  V.a = A.a;
  V.c = A.c;
  for (int d = 0; d < 3; ++d) V.b[d] = A.b[d];
  if (gc) {
    V.csy = Off(gc->sy);
    V.csz = Off(gc->sz);
  }
  V.alpha = A.alpha;
  V.beta = A.beta;
  V.dxinv = T(1) / (T(g.dx) * T(g.dx));
  const GhostForm<T> gf = vc_ghost_form<T>(A.bc, T(g.dx));
  for (int d = 0; d < 3; ++d)
    for (int sd = 0; sd < 2; ++sd) {
      V.gs[d][sd] = gf.s[d][sd][0];
      V.gb[d][sd] = gf.b[d][sd][0];
    }
  double faces = 0;
  for (int d = 0; d < 3; ++d) faces += double(g.nface[d]);
  for (int p = 0; p < npass; ++p) {
    V.S.colour = p & 1;
    const bool timed = tm && *tm->n < tm->cap;
    if (tm && !timed) ++*tm->missed;
    const bool moves = GEN || p == 0;
    V.in = buf[*cur];
    V.out = buf[moves ? 1 - *cur : *cur];
    V.zero = p == 0 && zero_init ? 1 : 0;
    V.pc = p == 0 ? pc : nullptr;
    auto kern = moves ? vc_sweep3_kernel<T, true, GEN> : vc_sweep3_kernel<T, GEN, GEN>;
    hipExtLaunchKernelGGL(kern, dim3(8 * V.S.chunk), dim3(256), 0, s, timed ? tm->start[*tm->n] : nullptr,
                          timed ? tm->stop[*tm->n] : nullptr, 0, V);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (timed) {
      // state, rhs, a and c of the colour and the other colour's state once;
      // every face; the colour written (a pass that moves: every cell)
      const double cells = double(g.nvalid());
      const double b = cells * (p == 0 && zero_init ? 0 : 1) + (p == 0 && pc ? cells / 8 : 0) +
                       0.5 * cells * (1 + (A.a ? 1 : 0) + (A.c ? 1 : 0)) + faces + (moves ? 1.0 : 0.5) * cells;
      *tm->bytes += b * sizeof(T);
      ++*tm->n;
    }
    if (moves) *cur = 1 - *cur;
  }
  return hipSuccess;
}

// tiles of the 2D relaxation on large levels (short halo, wide rows;
// measured best of 6 shapes at 2048^2)
struct VCRelaxWide2 {
  static constexpr int TX = 64, TY = 8, TZ = 1, HMAX = 2, NT = 256;
};
constexpr long long kWideCells = 512 * 512;   // levels above this use the wide tiles

inline bool vc_wide(const Geom& g) { return g.dim == 2 && g.nvalid() > kWideCells; }

// passes one relaxation launch can do on level g
inline int vc_hmax(const Geom& g) {
  return vc_wide(g) ? VCRelaxWide2::HMAX : (g.dim == 2 ? VCRelaxTile<2>::HMAX : VCRelaxTile<3>::HMAX);
}

template <typename T, int DIM>
hipError_t vc_relax_dim(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                        const Geom* gc, const T* pc, hipStream_t s, const Geom* gr = nullptr, T* resc = nullptr,
                        const LaunchTimer* tm = nullptr, const VCFinal<T>* fin = nullptr) {
  if (DIM == 3 && !resc && !fin && npass > 0)
    return sweep3_plain(A.g) ? vc_relax_sweeps<T, false>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, tm)
                             : vc_relax_sweeps<T, true>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, tm);
  if constexpr (DIM == 2) {
    if (!resc && !fin && npass > 0 && vc_streams(A.g))
      return vc_relax_stream<T>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, tm);
    if (vc_wide(A.g))
      return vc_relax_cfg<T, 2, VCRelaxWide2>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, gr, resc, tm, fin);
  }
  return vc_relax_cfg<T, DIM, VCRelaxTile<DIM>>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, gr, resc, tm, fin);
}

template <typename T, int DIM, int MODE>
hipError_t vc_tile_dim(const VCArgs<T>& A, VCTileIO<T> io, hipStream_t s) {
  using D = VCTile<DIM>;
  const int nt = vc_tiles<D::TX, D::TY, D::TZ>(A.g, io.ntx, io.nty);
  size_t lds = size_t(D::TX + 2) * (D::TY + 2) * (DIM == 3 ? D::TZ + 2 : 1);
  if (MODE == kVCRestrict) lds += size_t(D::TX) * D::TY * D::TZ;
  hipLaunchKernelGGL((vc_tile_kernel<T, DIM, D::TX, D::TY, D::TZ, MODE>), dim3(nt), dim3(kVCThreads),
                     lds * sizeof(T), s, A, io);
  return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t vc_relax(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                    const Geom* gc, const T* pc, hipStream_t s, const LaunchTimer* tm) {
  return A.g.dim == 2 ? vc_relax_dim<T, 2>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, nullptr, nullptr, tm)
                      : vc_relax_dim<T, 3>(A, buf, cur, rhs, npass, zero_init, gc, pc, s, nullptr, nullptr, tm);
}

template <typename T>
hipError_t vc_relax_restrict(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, bool zero_init,
                             const Geom& gr, T* resc, hipStream_t s, const LaunchTimer* tm) {
  const int hmax = vc_hmax(A.g);
  if (npass + 1 <= hmax)
    return A.g.dim == 2 ? vc_relax_dim<T, 2>(A, buf, cur, rhs, npass, zero_init, nullptr, nullptr, s, &gr, resc, tm)
                        : vc_relax_dim<T, 3>(A, buf, cur, rhs, npass, zero_init, nullptr, nullptr, s, &gr, resc, tm);
  hipError_t e = vc_relax<T>(A, buf, cur, rhs, npass, zero_init, nullptr, nullptr, s, tm);
  if (e != hipSuccess) return e;
  return vc_restrict_residual<T>(A, gr, buf[*cur], rhs, resc, s);
}

template <typename T>
hipError_t vc_relax_final(const VCArgs<T>& A, T* const buf[2], int* cur, const T* rhs, int npass, const Geom* gc,
                          const T* pc, const VCFinal<T>& fin, bool* fused, hipStream_t s, const LaunchTimer* tm) {
  const int hmax = vc_hmax(A.g);
  *fused = npass >= 1 && npass + 1 <= hmax && fin.phi && fin.phi_out != fin.phi;
  if (!*fused) return hipSuccess;
  return A.g.dim == 2 ? vc_relax_dim<T, 2>(A, buf, cur, rhs, npass, false, gc, pc, s, nullptr, nullptr, tm, &fin)
                      : vc_relax_dim<T, 3>(A, buf, cur, rhs, npass, false, gc, pc, s, nullptr, nullptr, tm, &fin);
}

template <typename T>
hipError_t vc_residual(const VCArgs<T>& A, const T* phi, const T* e, T* phi_out, const T* rhs, T* res,
                       unsigned long long* norm, int homog, hipStream_t s, const CtlFuse& fuse) {
  if (e && (!phi_out || phi_out == phi)) return hipErrorInvalidValue;
  VCTileIO<T> io{};
  io.phi = phi;
  io.e = e;
  io.phi_out = phi_out;
  io.rhs = rhs;
  io.out = res;
  io.norm = norm;
  io.fuse = fuse;
  io.homog = homog;
  return A.g.dim == 2 ? vc_tile_dim<T, 2, kVCResid>(A, io, s) : vc_tile_dim<T, 3, kVCResid>(A, io, s);
}

int vc_resid_tiles(const Geom& g, int* ntx, int* nty) {
  return g.dim == 2 ? vc_tiles<VCTile<2>::TX, VCTile<2>::TY, VCTile<2>::TZ>(g, *ntx, *nty)
                    : vc_tiles<VCTile<3>::TX, VCTile<3>::TY, VCTile<3>::TZ>(g, *ntx, *nty);
}

template <typename T>
hipError_t vc_resid_batch(int dim, const VCResidJob<T>* jobs, const unsigned* map, int nblocks, hipStream_t s) {
  if (nblocks <= 0) return hipSuccess;
  if (dim == 2) {
    using D = VCTile<2>;
    const size_t lds = size_t(D::TX + 2) * (D::TY + 2) * sizeof(T);
    hipLaunchKernelGGL((vc_resid_batch_kernel<T, 2, D::TX, D::TY, D::TZ>), dim3(nblocks), dim3(kVCThreads), lds, s,
                       jobs, map);
  } else {
    using D = VCTile<3>;
    const size_t lds = size_t(D::TX + 2) * (D::TY + 2) * (D::TZ + 2) * sizeof(T);
    hipLaunchKernelGGL((vc_resid_batch_kernel<T, 3, D::TX, D::TY, D::TZ>), dim3(nblocks), dim3(kVCThreads), lds, s,
                       jobs, map);
  }
  return hipGetLastError();
}

hipError_t words_batch(const WordsJob* jobs, const unsigned* map, int nblocks, hipStream_t s) {
  if (nblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(words_batch_kernel, dim3(nblocks), dim3(256), 0, s, jobs, map);
  return hipGetLastError();
}

template <typename T>
hipError_t vc_apply_op(const VCArgs<T>& A, const T* phi, T* lhs, int homog, hipStream_t s) {
  VCTileIO<T> io{};
  io.phi = phi;
  io.out = lhs;
  io.homog = homog;
  return A.g.dim == 2 ? vc_tile_dim<T, 2, kVCApply>(A, io, s) : vc_tile_dim<T, 3, kVCApply>(A, io, s);
}

template <typename T>
hipError_t vc_restrict_residual(const VCArgs<T>& A, const Geom& gc, const T* phi, const T* rhs, T* resc,
                                hipStream_t s) {
  VCTileIO<T> io{};
  io.phi = phi;
  io.rhs = rhs;
  io.out = resc;
  io.gc = gc;
  io.homog = 1;
  return A.g.dim == 2 ? vc_tile_dim<T, 2, kVCRestrict>(A, io, s) : vc_tile_dim<T, 3, kVCRestrict>(A, io, s);
}

// phi = rhs * lambda on the valid cells (the first step of preCond)
template <typename T, int DIM>
__global__ __launch_bounds__(256) void vc_lambda_mult_kernel(VCArgs<T> A, const T* __restrict__ rhs,
                                                             T* __restrict__ phi) {
  const Geom& g = A.g;
  const long long n = g.nvalid();
  const T dxinv = T(1) / (T(g.dx) * T(g.dx));
  for (long long c = blockIdx.x * (long long)blockDim.x + threadIdx.x; c < n; c += (long long)gridDim.x * blockDim.x) {
    const int i = int(c % g.n[0]);
    const long long r = c / g.n[0];
    const int j = int(r % g.n[1]);
    const int k = int(r / g.n[1]);
    Faces1<T, DIM> F;
    load_faces1<T, DIM>(A, i, j, k, F);
    const long long q = g.ci(i, j, k);
    const T aq = A.a ? A.a[q] : T(1);
    const T cv = A.c ? A.c[q] : T(0);
    phi[q] = rhs[q] * vc_lambda<T, DIM>(F, aq, A.c != nullptr, cv, A.alpha, A.beta, dxinv);
  }
}

// (x, y) over the valid cells in the order of the coarse V-cycle's BiCGStab:
// one wavefront, 64 interleaved lane sums over the compact cell index, then
// the pairwise tree s_t + s_{t+h}, h = P/2 .. 1 (P the smallest power of two
// >= min(cells, 64))
template <typename T>
__global__ __launch_bounds__(64) void vc_dot_kernel(Geom g, const T* __restrict__ x, const T* __restrict__ y,
                                                    T* __restrict__ out) {
  const long long n = g.nvalid();
  T s = T(0);
  for (long long c = threadIdx.x; c < n; c += 64) {
    const int i = int(c % g.n[0]);
    const long long r = c / g.n[0];
    const long long q = g.ci(i, int(r % g.n[1]), int(r / g.n[1]));
    s = s + x[q] * y[q];
  }
  int P2 = 1;
  while (P2 < 64 && P2 < n) P2 <<= 1;
  for (int h = P2 >> 1; h >= 1; h >>= 1) s = s + __shfl_down(s, h, 64);
  if (threadIdx.x == 0) *out = s;
}

template <typename T>
hipError_t vc_lambda_mult(const VCArgs<T>& A, const T* rhs, T* phi, hipStream_t s) {
  const long long n = A.g.nvalid();
  const int blocks = int(std::min<long long>((n + 255) / 256, 4096));
  if (A.g.dim == 2)
    hipLaunchKernelGGL((vc_lambda_mult_kernel<T, 2>), dim3(blocks), dim3(256), 0, s, A, rhs, phi);
  else
    hipLaunchKernelGGL((vc_lambda_mult_kernel<T, 3>), dim3(blocks), dim3(256), 0, s, A, rhs, phi);
  return hipGetLastError();
}

template <typename T>
hipError_t vc_dot(const Geom& g, const T* x, const T* y, T* out, hipStream_t s) {
  hipLaunchKernelGGL((vc_dot_kernel<T>), dim3(1), dim3(64), 0, s, g, x, y, out);
  return hipGetLastError();
}

// ---- batched form --------------------------------------------------------
bool vc_batch_level_ok(const Geom& g) { return !vc_wide(g); }

int vc_batch_hmax(int dim) { return dim == 2 ? VCRelaxTile<2>::HMAX : VCRelaxTile<3>::HMAX; }

int vc_batch_tiles(const Geom& g, int shape, int* ntx, int* nty) {
  if (g.dim == 3) return vc_tiles<VCRelaxTile<3>::TX, VCRelaxTile<3>::TY, VCRelaxTile<3>::TZ>(g, *ntx, *nty);
  return shape == 1 ? vc_tiles<VCRelaxBatchWide2::TX, VCRelaxBatchWide2::TY, 1>(g, *ntx, *nty)
                    : vc_tiles<VCRelaxTile<2>::TX, VCRelaxTile<2>::TY, VCRelaxTile<2>::TZ>(g, *ntx, *nty);
}

template <class D, int DIM>
static size_t vc_batch_lds_dim(int npass, bool resc, bool fin) {
  const int h = npass + ((resc || fin) ? 1 : 0);
  size_t lds = size_t(D::TX + 2 * h) * (D::TY + 2 * h) * (DIM == 3 ? D::TZ + 2 * h : 1);
  if (resc) lds += size_t(D::TX) * D::TY * D::TZ;
  if (fin) lds *= 2;
  return lds;
}

size_t vc_batch_lds(int dim, int shape, int npass, bool resc, bool fin) {
  const size_t e = dim == 3 ? vc_batch_lds_dim<VCRelaxTile<3>, 3>(npass, resc, fin)
                            : (shape == 1 ? vc_batch_lds_dim<VCRelaxBatchWide2, 2>(npass, resc, fin)
                                          : vc_batch_lds_dim<VCRelaxTile<2>, 2>(npass, resc, fin));
  return e * sizeof(double);
}

template <typename T>
hipError_t vc_relax_batch(int dim, int shape, const VCRelaxJob<T>* jobs, const unsigned* map, int nblocks, size_t lds,
                          hipStream_t s, const LaunchTimer* tm) {
  if (nblocks <= 0) return hipSuccess;
  const bool timed = tm && *tm->n < tm->cap;
  if (tm && !timed) ++*tm->missed;
  hipEvent_t e0 = timed ? tm->start[*tm->n] : nullptr, e1 = timed ? tm->stop[*tm->n] : nullptr;
  if (dim == 2 && shape == 1) {
    using D = VCRelaxBatchWide2;
    hipExtLaunchKernelGGL((vc_relax_batch_kernel<T, 2, D::TX, D::TY, D::TZ, D::HMAX, D::NT>), dim3(nblocks),
                          dim3(D::NT), lds, s, e0, e1, 0, jobs, map);
  } else if (dim == 2) {
    using D = VCRelaxTile<2>;
    hipExtLaunchKernelGGL((vc_relax_batch_kernel<T, 2, D::TX, D::TY, D::TZ, D::HMAX, D::NT>), dim3(nblocks),
                          dim3(D::NT), lds, s, e0, e1, 0, jobs, map);
  } else {
    using D = VCRelaxTile<3>;
    hipExtLaunchKernelGGL((vc_relax_batch_kernel<T, 3, D::TX, D::TY, D::TZ, D::HMAX, D::NT>), dim3(nblocks),
                          dim3(D::NT), lds, s, e0, e1, 0, jobs, map);
  }
  if (timed) ++*tm->n;
  return hipGetLastError();
}

__global__ void ctl_gather_kernel(SolveCtl* const* __restrict__ ctls, SolveCtl* __restrict__ out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = *ctls[i];
}

hipError_t ctl_gather(SolveCtl* const* ctls, SolveCtl* out, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(ctl_gather_kernel, dim3((n + 255) / 256), dim3(256), 0, s, ctls, out, n);
  return hipGetLastError();
}

template <typename T>
hipError_t vc_coarse_batch(int dim, const VCDesc<T>* const* descs, int n, size_t lds, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  if (dim == 2)
    hipLaunchKernelGGL((vc_coarse_batch_kernel<T, 2>), dim3(n), dim3(kVCWG), lds, s, descs);
  else
    hipLaunchKernelGGL((vc_coarse_batch_kernel<T, 3>), dim3(n), dim3(kVCWG), lds, s, descs);
  return hipGetLastError();
}

template <typename T>
size_t vc_coarse_lds_bytes(const Geom* g, int l0, int nlev, bool bicgstab) {
  long long tot = 0, nf = 0;
  for (int l = l0; l < nlev; ++l) {
    tot += g[l].nvalid();
    for (int d = 0; d < g[l].dim; ++d) nf += g[l].nface[d];
  }
  // with a and c; BiCGStab above 64 cells: two buffers of products
  const long long N = g[nlev - 1].nvalid();
  const size_t extra = bicgstab && N > 64 ? size_t(2 * N) : 0;
  return (size_t(vc_lds_map(int(tot), int(nf + (nf & 1)), true, true).end) + extra) * sizeof(T);
}

template <typename T>
void vc_desc_geometry(VCDesc<T>& D, const Geom& g, const BCDesc& bc, int nl) {
  D.nl = nl;
  for (int d = 0; d < 3; ++d) {
    D.n[d] = g.n[d];
    D.per[d] = g.periodic[d];
  }
  D.dx = T(g.dx);
  int fo = 0;
  for (int l = 0; l < nl; ++l) {
    const Geom gl = l == 0 ? g : coarsen_geom(g, 1 << l);
    D.off[l + 1] = D.off[l] + int(gl.nvalid());
    for (int d = 0; d < g.dim; ++d) {
      D.fo[l][d] = fo;
      fo += int(gl.nface[d]);
    }
  }
  D.tot = D.off[nl];
  const GhostForm<T> gf = vc_ghost_form<T>(bc, T(g.dx));
  for (int d = 0; d < 3; ++d)
    for (int s = 0; s < 2; ++s) {
      D.gs[d][s] = gf.s[d][s][0];
      D.gb[d][s] = gf.b[d][s][0];
    }
}

template <typename T>
hipError_t vc_coarse_vcycle(const VCDesc<T>* dev_desc, int dim, size_t lds, hipStream_t s) {
  if (dim == 2)
    hipLaunchKernelGGL((vc_coarse_vcycle_kernel<T, 2>), dim3(1), dim3(kVCWG), lds, s, dev_desc);
  else
    hipLaunchKernelGGL((vc_coarse_vcycle_kernel<T, 3>), dim3(1), dim3(kVCWG), lds, s, dev_desc);
  return hipGetLastError();
}

bool vc_small_level(const Geom& g) { return g.nvalid() <= kVCWGCells; }
int vc_coarse_levels_max(int dim) { return dim == 3 ? VCLevels<3>::n : VCLevels<2>::n; }

template hipError_t vc_relax<double>(const VCArgs<double>&, double* const[2], int*, const double*, int, bool,
                                     const Geom*, const double*, hipStream_t, const LaunchTimer*);
template hipError_t vc_relax_restrict<double>(const VCArgs<double>&, double* const[2], int*, const double*, int, bool,
                                              const Geom&, double*, hipStream_t, const LaunchTimer*);
template hipError_t vc_relax_final<double>(const VCArgs<double>&, double* const[2], int*, const double*, int,
                                           const Geom*, const double*, const VCFinal<double>&, bool*, hipStream_t,
                                           const LaunchTimer*);
template hipError_t vc_residual<double>(const VCArgs<double>&, const double*, const double*, double*,
                                        const double*, double*, unsigned long long*, int, hipStream_t,
                                        const CtlFuse&);
template hipError_t vc_apply_op<double>(const VCArgs<double>&, const double*, double*, int, hipStream_t);
template hipError_t vc_lambda_mult<double>(const VCArgs<double>&, const double*, double*, hipStream_t);
template hipError_t vc_dot<double>(const Geom&, const double*, const double*, double*, hipStream_t);
template hipError_t vc_restrict_residual<double>(const VCArgs<double>&, const Geom&, const double*, const double*,
                                                 double*, hipStream_t);
template void vc_desc_geometry<double>(VCDesc<double>&, const Geom&, const BCDesc&, int);
template hipError_t vc_coarse_vcycle<double>(const VCDesc<double>*, int, size_t, hipStream_t);
template size_t vc_coarse_lds_bytes<double>(const Geom*, int, int, bool);
template hipError_t vc_relax_batch<double>(int, int, const VCRelaxJob<double>*, const unsigned*, int, size_t,
                                           hipStream_t, const LaunchTimer*);
template hipError_t vc_coarse_batch<double>(int, const VCDesc<double>* const*, int, size_t, hipStream_t);
template hipError_t vc_resid_batch<double>(int, const VCResidJob<double>*, const unsigned*, int, hipStream_t);

}  // namespace ml
