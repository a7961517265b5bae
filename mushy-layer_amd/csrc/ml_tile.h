// ml_tile.h — device helpers shared by the tiled stencil kernels: position
// classification against periodic / wall boundaries, per-thread position
// records of a tile's extended region, face-coefficient gathers and the
// L(phi) bracket of the reference's Fortran stencils.
#pragma once

#include <type_traits>

#include "ml_common.h"
#include "ml_kernels.h"

namespace ml {

// Position classification of an (unwrapped) index vector of a tile's
// extended region: in-domain (after periodic wrap), one-cell ghost of a
// non-periodic wall (exactly one direction outside), or invalid.
struct Pos {
  int i, j, k;   // wrapped coordinates; for a ghost: the interior neighbour
  int kind;      // 0 invalid, 1 in-domain, 2 wall ghost
  int gd, gs;    // ghost direction and side (0 lo, 1 hi)
};

template <int DIM>
__device__ inline Pos classify(const Geom& g, int ci, int cj, int ck) {
  int c[3] = {ci, cj, ck};
  Pos P;
  P.gd = 0;
  P.gs = 0;
  int nout = 0, far = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int n = g.n[d];
    if (c[d] < 0 || c[d] >= n) {
      if (g.periodic[d]) {
        c[d] = ((c[d] % n) + n) % n;
      } else if (c[d] == -1) {
        P.gd = d; P.gs = 0; c[d] = 0; ++nout;
      } else if (c[d] == n) {
        P.gd = d; P.gs = 1; c[d] = n - 1; ++nout;
      } else {
        far = 1;
      }
    }
  }
  if (DIM == 2) c[2] = 0;
  P.i = c[0];
  P.j = c[1];
  P.k = c[2];
  P.kind = (far || nout > 1) ? 0 : (nout == 1 ? 2 : 1);
  return P;
}

// Face coefficients around a cell, both components: bf[n][2d+s] is the
// lo (s = 0) / hi (s = 1) face of direction d.
template <typename T, int DIM>
struct CellFaces {
  T v[2][2 * DIM];
};

template <typename T, int DIM>
__device__ inline void load_faces(const Geom& g, const T* const* b, int i, int j, int k, CellFaces<T, DIM>& F) {
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const T* bd = b[d] + (long long)n * g.nface[d];
      F.v[n][2 * d] = bd[g.fi(d, i, j, k)];
      F.v[n][2 * d + 1] = bd[g.fi(d, i + (d == 0), j + (d == 1), k + (d == 2))];
    }
}

template <typename T, int DIM>
__device__ inline void load_faces(const HCArgs<T>& A, int i, int j, int k, CellFaces<T, DIM>& F) {
  load_faces<T, DIM>(A.g, A.b, i, j, k, F);
}

// lambda = 1/(alpha*a + sum_d scale*beta*(b_hi + b_lo))
// (src/AMRNonLinearMultiCompOp.cpp:540-573, SUMFACESNLVC).
template <typename T, int DIM>
__device__ inline T lambda_of(const CellFaces<T, DIM>& F, int n, T aq, T alpha, T beta, T scale) {
  T lam = aq * alpha;
#pragma unroll
  for (int d = 0; d < DIM; ++d) lam = lam + scale * beta * (F.v[n][2 * d + 1] + F.v[n][2 * d]);
  return T(1) / lam;
}

// The L(phi) bracket (src/AMRNonLinearMultiCompOpF.ChF:125-160) from the
// seven stencil values p[0] = centre, p[2d+1] = +e_d, p[2d+2] = -e_d.
template <typename T, int DIM>
__device__ inline T lof_of(const CellFaces<T, DIM>& F, int n, const T* p, T aq, T phic, T alpha, T beta,
                           T dxinv) {
  const T p0 = p[0];
  T s = F.v[n][1] * (p[1] - p0) - F.v[n][0] * (p0 - p[2]) + F.v[n][3] * (p[3] - p0) - F.v[n][2] * (p0 - p[4]);
  if (DIM == 3) s = s + F.v[n][5] * (p[5] - p0) - F.v[n][4] * (p0 - p[6]);
  return alpha * aq * phic - beta * s * dxinv;
}

// Extended-region bookkeeping of one tile.
template <int DIM, int TX, int TY, int TZ>
struct Tile {
  int H, EX, EY, EZ, EXY, E;
  int x0, y0, z0;
  __device__ inline void init(int halo, int ntx, int nty) { init_at(halo, ntx, nty, blockIdx.x); }
  // tile b of the level (b != blockIdx.x when several grids share a launch)
  __device__ inline void init_at(int halo, int ntx, int nty, int b) {
    H = halo;
    EX = TX + 2 * H;
    EY = TY + 2 * H;
    EZ = DIM == 3 ? TZ + 2 * H : 1;
    EXY = EX * EY;
    E = EXY * EZ;
    const int tx = b % ntx, r = b / ntx, ty = r % nty, tz = r / nty;
    x0 = tx * TX;
    y0 = ty * TY;
    z0 = DIM == 3 ? tz * TZ : 0;
  }
  __device__ inline void coords(int e, int& ex, int& ey, int& ez) const {
    ex = e % EX;
    const int r = e / EX;
    ey = r % EY;
    ez = r / EY;
  }
  // within the core grown by `ext` cells
  __device__ inline bool within(int ex, int ey, int ez, int ext) const {
    const int ox = ex - H, oy = ey - H, oz = ez - (DIM == 3 ? H : 0);
    bool ok = ox >= -ext && ox < TX + ext && oy >= -ext && oy < TY + ext;
    if (DIM == 3) ok = ok && oz >= -ext && oz < TZ + ext;
    return ok;
  }
  __device__ inline Pos pos(const Geom& g, int ex, int ey, int ez) const {
    return classify<DIM>(g, x0 - H + ex, y0 - H + ey, DIM == 3 ? z0 - H + ez : 0);
  }
};

// Gather the 2*DIM+1 phi_l stencil values of LDS position e.
template <typename T, int DIM>
__device__ inline void gather_lds(const T* pl, int e, int EX, int EXY, T* p) {
  p[0] = pl[e];
  p[1] = pl[e + 1];
  p[2] = pl[e - 1];
  p[3] = pl[e + EX];
  p[4] = pl[e - EX];
  if (DIM == 3) {
    p[5] = pl[e + EXY];
    p[6] = pl[e - EXY];
  }
}

// Per-thread record of one LDS position of a tile's extended region.
struct PosRec {
  long long q;   // global cell index (in-domain) or of the interior neighbour (ghost)
  int e;         // LDS position
  int kind;      // 0 unused/invalid, 1 in-domain, 2 wall ghost
  int dist;      // distance outside the core (0 inside)
  int eint;      // ghost: LDS position of the interior neighbour
  int gd, gs;    // ghost direction / side
  int i, j, k;   // wrapped coordinates
  bool owner;    // core cell inside the domain: written back by this tile
};


// Fill the record of LDS position e of tile t.
template <int DIM, int TX, int TY, int TZ>
__device__ inline void pos_record(const Geom& g, const Tile<DIM, TX, TY, TZ>& t, int e, PosRec& r) {
  r.e = e;
  r.kind = 0;
  r.owner = false;
  r.dist = 1 << 20;
  if (e >= t.E) return;
  int ex, ey, ez;
  t.coords(e, ex, ey, ez);
  const int ox = ex - t.H, oy = ey - t.H, oz = DIM == 3 ? ez - t.H : 0;
  const int dxo = ox < 0 ? -ox : (ox >= TX ? ox - TX + 1 : 0);
  const int dyo = oy < 0 ? -oy : (oy >= TY ? oy - TY + 1 : 0);
  const int dzo = DIM == 3 ? (oz < 0 ? -oz : (oz >= TZ ? oz - TZ + 1 : 0)) : 0;
  r.dist = dxo > dyo ? (dxo > dzo ? dxo : dzo) : (dyo > dzo ? dyo : dzo);
  const int gi = t.x0 + ox, gj = t.y0 + oy, gk = DIM == 3 ? t.z0 + oz : 0;
  const Pos P = classify<DIM>(g, gi, gj, gk);
  r.kind = P.kind;
  r.i = P.i;
  r.j = P.j;
  r.k = P.k;
  r.gd = P.gd;
  r.gs = P.gs;
  r.q = g.ci(P.i, P.j, P.k);
  const int stride = P.gd == 0 ? 1 : (P.gd == 1 ? t.EX : t.EXY);
  r.eint = P.gs == 0 ? e + stride : e - stride;
  r.owner = r.dist == 0 && P.kind == 1 && gi < g.n[0] && gj < g.n[1] && (DIM == 2 || gk < g.n[2]);
}

// ---- single-workgroup kernels: one level held compactly in LDS (x fastest)
struct CLev {
  int n[3];
  int nx, nxy, N, off;   // off: the level's offset in the workgroup's LDS arrays
  double dx;
};

// q = x / d, r = x % d for x >= 0, d > 0: a shift and a mask when d is a
// power of two (every level of a power-of-two grid), integer division
// otherwise.  d is uniform across the workgroup, so the branch is too.
__device__ __forceinline__ void divmod_pos(int x, int d, int& q, int& r) {
  if ((d & (d - 1)) == 0) {
    const int s = __builtin_ctz(d);
    q = x >> s;
    r = x & (d - 1);
  } else {
    q = x / d;
    r = x - q * d;
  }
}

__device__ inline void clev_coords(const CLev& L, int c, int& i, int& j, int& k) {
  int r;
  divmod_pos(c, L.nx, r, i);
  divmod_pos(r, L.n[1], k, j);
}

__device__ inline void clev_set(CLev& L, const Geom& g, int off) {
  for (int d = 0; d < 3; ++d) L.n[d] = g.n[d];
  L.nx = g.n[0];
  L.nxy = g.n[0] * g.n[1];
  L.N = L.nxy * g.n[2];
  L.off = off;
  L.dx = g.dx;
}

// wavefront-scope barrier: orders the LDS accesses of the lanes of one wave
__device__ inline void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// cells of a level owned by this thread: packed (i | j << 10 | k << 20), -1
// when none.  Even row length: the pair (2s + par, j, k), (2s + 1 - par, j, k)
// of opposite colours; otherwise cells t and t + NT.
struct COwn {
  int p[2];
};

__device__ inline int cpack(int i, int j, int k) { return i | (j << 10) | (k << 20); }
__device__ inline void cunpack(int v, int& i, int& j, int& k) {
  i = v & 1023;
  j = (v >> 10) & 1023;
  k = v >> 20;
}

// threads owning cells of level L
template <int NT>
__device__ inline int cown_active(const CLev& L) {
  return (L.nx & 1) == 0 ? (L.N >> 1) : (L.N < NT ? L.N : NT);
}

template <int NT>
__device__ inline void cown_set(const CLev& L, COwn& o) {
  const int t = threadIdx.x;
  o.p[0] = o.p[1] = -1;
  if ((L.nx & 1) == 0) {
    const int h = L.nx >> 1;
    if (t < (L.N >> 1)) {
      int s, r, j, k;
      divmod_pos(t, h, r, s);
      divmod_pos(r, L.n[1], k, j);
      const int par = (j + k) & 1;
      o.p[0] = cpack(2 * s + par, j, k);
      o.p[1] = cpack(2 * s + 1 - par, j, k);
    }
  } else {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int c = t + m * NT;
      if (c >= L.N) continue;
      int i, j, k;
      clev_coords(L, c, i, j, k);
      o.p[m] = cpack(i, j, k);
    }
  }
}


// neighbour compact indices of cell (i,j,k) of level L, face f = 2d + s
// (s = 1: +e_d): periodic images wrap; across a wall the cell itself, with
// bit f of `wall` set
template <int DIM>
__device__ __forceinline__ void clev_nbrs(const CLev& L, const int* per, int i, int j, int k, int* nb, int& wall) {
  const int iv[3] = {i, j, k};
  const int c = i + L.nx * j + L.nxy * k;
  wall = 0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const int nd = L.n[d];
    const int st = d == 0 ? 1 : (d == 1 ? L.nx : L.nxy);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int v = iv[d] + (s ? 1 : -1);
      if (v >= 0 && v < nd) {
        nb[2 * d + s] = c + (s ? st : -st);
      } else if (per[d]) {
        nb[2 * d + s] = c + (s ? -(nd - 1) * st : (nd - 1) * st);
      } else {
        nb[2 * d + s] = c;
        wall |= 1 << (2 * d + s);
      }
    }
  }
}

// ---- streaming (plane-marching) kernels ----------------------------------
// A workgroup owns a block of columns (2D: TX cells in x; 3D: TX x TY cells
// in (x, y)) extended by a lateral halo of P cells, and marches along the
// last direction.  IC<N> passes a compile-time index to a generic lambda.
template <int N>
struct IC {
  static constexpr int value = N;
};

// lateral position of the extended column block: global coordinate (wrapped
// when periodic), kind 1 cell / 2 wall ghost / 0 unused, distance to the core,
// owner flag, and for a ghost its side (gx: its interior neighbour)
struct SPos {
  int gx;
  int kind, dist, owner;
  int gs;
  int gtype;   // a ghost's boundary type (resolved once: a per-thread index
               // into the kernel arguments would be a memory load)
};

template <int TX, int P>
__device__ inline void spos_init(const Geom& g, int x0, int e, SPos& s) {
  const int l = e - P, n = g.n[0];
  int v = x0 + l;
  s.dist = l < 0 ? -l : (l >= TX ? l - TX + 1 : 0);
  s.owner = s.dist == 0 && v >= 0 && v < n;
  s.kind = 1;
  s.gs = 0;
  if (v < 0 || v >= n) {
    if (g.periodic[0]) {
      v = v < 0 ? v + n : v - n;
    } else {
      s.kind = v == -1 || v == n ? 2 : 0;
      s.gs = v >= n;
    }
  }
  // every position gets an in-domain coordinate (unused ones clamped), so the
  // prefetch can load unconditionally
  s.gx = v < 0 ? 0 : (v >= n ? n - 1 : v);
}

// ---- 3D colour passes straight from memory --------------------------------
// One launch updates the cells of one colour: they read the other colour and
// themselves only, so a pass can work in place, without tiles and halos.  (A
// 16 x 8 x 4 tile with the halo of two passes stages 3.75 positions per cell
// it keeps.)  A thread handles a pair of cells (2s, 2s+1) of a row, one of
// which has the colour: every lane works, and rows are read and written
// whole.  Blocks of 2^lpx pairs by 256 >> lpx rows; the blocks of one L2
// (workgroups go round the 8 of them) are neighbours in the level.
// Byte offsets within one component are 32-bit.
//
// GEN: any 3D level.  At the seam of an odd periodic length two cells of a
// colour are neighbours, and each has to see the other as of the start of the
// pass: so every pass goes from one buffer to the other (a row's pairs still
// hold one cell of each colour).  Offsets are 64-bit.
template <bool GEN>
struct Sweep3 {
  using Off = typename std::conditional<GEN, unsigned long long, unsigned>::type;
  int n[3], per[3];
  Off sy, sz, fx[3], fxy[3];   // cell and face strides (row, plane)
  int lpx, nbx, nby, nblocks, chunk, colour;
};

// whether level g needs no GEN
inline bool sweep3_plain(const Geom& g) {
  long long most = g.ncell;
  for (int d = 0; d < 3; ++d) {
    if (g.periodic[d] && (g.n[d] & 1)) return false;
    most = most > g.nface[d] ? most : g.nface[d];
  }
  return g.dim == 3 && most < (1LL << 29);
}

template <bool GEN>
inline Sweep3<GEN> sweep3_make(const Geom& g) {
  using Off = typename Sweep3<GEN>::Off;
  Sweep3<GEN> S{};
  for (int d = 0; d < 3; ++d) {
    S.n[d] = g.n[d];
    S.per[d] = g.periodic[d];
    S.fx[d] = Off(g.fn[d][0]);
    S.fxy[d] = Off(g.fn[d][0] * g.fn[d][1]);
  }
  S.sy = Off(g.sy);
  S.sz = Off(g.sz);
  const int pairs = (g.n[0] + 1) / 2;
  // the widest row of a block, up to 64 pairs, that leaves the fewest lanes idle
  auto blocks = [&](int l) { return ((pairs + (1 << l) - 1) >> l) * ((g.n[1] + (256 >> l) - 1) / (256 >> l)); };
  S.lpx = 6;
  for (int l = 5; l >= 3; --l)
    if (blocks(l) < blocks(S.lpx)) S.lpx = l;
  S.nbx = (pairs + (1 << S.lpx) - 1) >> S.lpx;
  S.nby = (g.n[1] + (256 >> S.lpx) - 1) / (256 >> S.lpx);
  S.nblocks = S.nbx * S.nby * g.n[2];
  S.chunk = (S.nblocks + 7) / 8;
  return S;
}

template <bool GEN>
struct Sweep3Pos {
  using Off = typename Sweep3<GEN>::Off;
  int i, j, k, par;
  bool act, oth;       // the pair's cell of the colour, its other cell: in the level
  Off q, qo;           // ... their indices
  Off nb[6];           // neighbours of the cell of the colour (-x, +x, ...), itself beyond a wall
  unsigned wall;       // bit f: neighbour f is a wall's ghost
};

template <bool GEN>
__device__ __forceinline__ bool sweep3_pos(const Sweep3<GEN>& S, Sweep3Pos<GEN>& P) {
  using Off = typename Sweep3<GEN>::Off;
  const int l = int(blockIdx.x & 7u) * S.chunk + int(blockIdx.x >> 3);
  if (l >= S.nblocks || int(blockIdx.x >> 3) >= S.chunk) return false;
  const int bx = l % S.nbx, r = l / S.nbx, by = r % S.nby;
  P.k = r / S.nby;
  const int s = (bx << S.lpx) + (int(threadIdx.x) & ((1 << S.lpx) - 1));
  P.j = by * (256 >> S.lpx) + (int(threadIdx.x) >> S.lpx);
  if (2 * s >= S.n[0] || P.j >= S.n[1]) return false;
  P.par = (P.j + P.k + S.colour) & 1;
  P.i = 2 * s + P.par;
  P.act = P.i < S.n[0];
  P.oth = 2 * s + 1 - P.par < S.n[0];
  const Off row = S.sy * Off(P.j + 1) + S.sz * Off(P.k + 1);
  P.q = row + Off(P.i + 1);
  P.qo = row + Off(2 * s + 2 - P.par);
  P.wall = 0;
  const int iv[3] = {P.i, P.j, P.k};
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const Off st = d == 0 ? Off(1) : (d == 1 ? S.sy : S.sz);
    const Off span = st * Off(S.n[d] - 1);
    const bool lo = iv[d] == 0, hi = iv[d] == S.n[d] - 1;
    P.nb[2 * d] = lo ? (S.per[d] ? P.q + span : P.q) : P.q - st;
    P.nb[2 * d + 1] = hi ? (S.per[d] ? P.q - span : P.q) : P.q + st;
    if (!S.per[d]) P.wall |= (lo ? 1u << (2 * d) : 0u) | (hi ? 2u << (2 * d) : 0u);
  }
  return true;
}

// element i of p
template <typename T, typename Off>
__device__ __forceinline__ T get_at(const T* p, Off i) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(p) + i * Off(sizeof(T)));
}
template <typename T, typename Off>
__device__ __forceinline__ void put_at(T* p, Off i, T v) {
  *reinterpret_cast<T*>(reinterpret_cast<char*>(p) + i * Off(sizeof(T))) = v;
}
// the six faces of the cell, component array b
template <typename T, bool GEN>
__device__ __forceinline__ void sweep3_faces(const Sweep3<GEN>& S, const Sweep3Pos<GEN>& P, int d, const T* b, T& lo,
                                             T& hi) {
  using Off = typename Sweep3<GEN>::Off;
  const Off f = Off(P.i) + S.fx[d] * Off(P.j) + S.fxy[d] * Off(P.k);
  lo = get_at(b, f);
  hi = get_at(b, f + (d == 0 ? Off(1) : (d == 1 ? S.fx[1] : S.fxy[2])));
}

}  // namespace ml
