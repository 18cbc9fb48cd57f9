// wx_kernels.hip -- gfx950 kernels of the Walicxe-2D hot path.
//
// Data layout in HBM: one padded 20x20 tile per variable per block,
// [id][var][cell], id = the reference's block ID, the cells in the order of
// tile_cell (interior, ghost layer 1, ghost layer 2, corners).  Every kernel
// below assigns one workgroup to one leaf block and stages the tile in LDS,
// there as padded rows (IDX).
//
// One step (src/tstep.f90:4-126) is three launches over the leaf list:
//   k_stageA      Uⁿ -> U^{n+1/2} interior (first-order fluxes, dt/2)
//   k_stageB      pulls the 2-layer ghost ring of U^{n+1/2} from the
//                 neighbours (boundaryII semantics), limited fluxes, update,
//                 viscosity; writes U^{n+1} interior and the U^{n+1/2} ring
//                 in place over Uⁿ (tstep.f90:85 copies the whole padded block)
//   k_fillI_cool  pulls ghost layer 1 (boundaryI), imposes the jet, applies
//                 cooling on cells 0..17, writes the final tile to the other
//                 buffer, and emits the next CFL partials and the refinement
//                 flag of the block (fused timestep/criteria epilogue).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "wx_device.h"
#include "wx_mlp.h"
#include "wx_physics.h"

namespace wx {

__device__ __forceinline__ int IDX(int i, int j) { return (j + 1) * NP + (i + 1); }
__device__ __forceinline__ int INT(int i, int j) { return (j - 1) * NX + (i - 1); }   // tile_cell of an interior cell

// threadIdx.x computed again from the wave's number (in a scalar register) and
// the lane: two instructions each time instead of a vector register held, or
// spilled, across a kernel whose budget is 64 of them.
__device__ __forceinline__ int wave_of() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6); }
__device__ __forceinline__ int tid_again(int wave) {
  int lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=&v"(lane));
  return wave * 64 + lane;
}

// Queue entry of workgroup b in a one-entry-per-workgroup launch of G
// workgroups.  The hardware deals workgroups to the 8 XCDs round robin
// (b % 8); within each run of 64 workgroups this hands XCD x the 8
// consecutive entries 8x..8x+7, so that neighbouring blocks, which share
// ghost data, are computed behind the same L2.  The last partial run keeps
// the identity, so the map is a bijection of [0, G).
__device__ __forceinline__ int xcd_entry(int b, int G) {
  if (b >= (G & ~63)) return b;
  return (b & ~63) | ((b & 7) << 3) | ((b >> 3) & 7);
}

// ---------------------------------------------------------------------
// Ghost gather: value of one non-corner ghost cell of block `dst` at
// (side, layer, pos) from the op that last wrote its segment.
//   side 0 left (i = 1-layer), 1 right (i = 16+layer), 2 bottom (j = 1-layer),
//   3 top (j = 16+layer); layer 1 is adjacent to the interior, 2 outer;
//   pos 1..16 runs along the side.
// Formulas: src/boundaryII.f90:143-500 and src/boundaryI.f90:109-382.
template <int NEQ>
__device__ __forceinline__ void src_cell(const wx_params *__restrict__ p, const double *__restrict__ A,
                                         const BlockRec *__restrict__ binfo, int b, int i, int j,
                                         bool imposed, double vjet, double *v) {
  const double *t = A + (size_t)b * NEQ * NC + INT(i, j);   // gathers read interiors
#pragma unroll
  for (int k = 0; k < NEQ; ++k) v[k] = t[k * NC];
  if (imposed) {
    BlockRec r = binfo[b];
    if (in_jet(p, r.level, r.icx, r.icy, i, j)) jet_state<NEQ>(p, vjet, v);
  }
}

template <int NEQ>
__device__ __forceinline__ void ghost_gather(const wx_params *__restrict__ p, const double *__restrict__ A,
                             const BlockRec *__restrict__ binfo, int2 op, int dst, int dlev,
                             int dicx, int dicy, int side, int layer, int pos, double vjet,
                             double *g) {
  const int kind = op.y & 15;
  const int src = op.x;
  const bool simp = (op.y & GF_SRC_IMPOSED) != 0;
  const bool dimp = (op.y & GF_DST_IMPOSED) != 0;
  const int off = (op.y >> GF_OFF_SHIFT) & 15;
  const bool xside = side < 2;
  // destination cell
  int di, dj;
  if (side == 0) { di = 1 - layer; dj = pos; }
  else if (side == 1) { di = NX + layer; dj = pos; }
  else if (side == 2) { dj = 1 - layer; di = pos; }
  else { dj = NY + layer; di = pos; }
  if (kind == GK_COPY) {
    int si = di, sj = dj;
    if (side == 0) si = di + NX;
    else if (side == 1) si = di - NX;
    else if (side == 2) sj = dj + NY;
    else sj = dj - NY;
    src_cell<NEQ>(p, A, binfo, src, si, sj, simp, vjet, g);
  } else if (kind == GK_RESTRICT) {
    const int half = (pos - 1) >> 3;
    int i1, j1;
    if (xside) {
      int jj = pos - 8 * half;
      i1 = (side == 0) ? (2 * di - 1 + NX) : (2 * (di - NX) - 1);
      j1 = 2 * jj - 1;
    } else {
      int ii = pos - 8 * half;
      i1 = 2 * ii - 1;
      j1 = (side == 2) ? (2 * dj - 1 + NY) : (2 * (dj - NY) - 1);
    }
    double a[NEQ], b2[NEQ], c[NEQ], d[NEQ];
    src_cell<NEQ>(p, A, binfo, src, i1, j1, simp, vjet, a);
    src_cell<NEQ>(p, A, binfo, src, i1 + 1, j1, simp, vjet, b2);
    src_cell<NEQ>(p, A, binfo, src, i1, j1 + 1, simp, vjet, c);
    src_cell<NEQ>(p, A, binfo, src, i1 + 1, j1 + 1, simp, vjet, d);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) g[k] = 0.25 * (((a[k] + b2[k]) + c[k]) + d[k]);
  } else if (kind == GK_PROLONG) {
    int si, sj;
    if (xside) {
      si = (side == 0) ? NX : 1;
      sj = (dj + 1) / 2 + off;
    } else {
      sj = (side == 2) ? NY : 1;
      si = (di + 1) / 2 + off;
    }
    src_cell<NEQ>(p, A, binfo, src, si, sj, simp, vjet, g);
  } else {  // GK_BOXOUT / GK_BOXREF : mirror own interior
    int si = di, sj = dj;
    if (side == 0) si = 1 - di;
    else if (side == 1) si = 2 * NX + 1 - di;
    else if (side == 2) sj = 1 - dj;
    else sj = 2 * NY + 1 - dj;
    src_cell<NEQ>(p, A, binfo, dst, si, sj, simp, vjet, g);
    if (kind == GK_BOXREF) {
      if (xside) g[1] = -g[1];
      else g[2] = -g[2];
    }
  }
  if (dimp && in_jet(p, dlev, dicx, dicy, di, dj)) jet_state<NEQ>(p, vjet, g);
}

// (Selects rather than branches: branches that assign i or j make the
// compiler keep the pair in scratch memory.)
__device__ __forceinline__ void ghost_coords(int side, int layer, int pos, int &i, int &j) {
  static_assert(NX == NY, "one edge index for both directions");
  const int edge = (side & 1) ? NX + layer : 1 - layer;
  const bool xside = side < 2;
  i = xside ? edge : pos;
  j = xside ? pos : edge;
}

// (i, j) of cell c < 320 of a tile's device order: the interior, then ghost
// layer 1.
__device__ __forceinline__ void tile_ij(int c, int &i, int &j) {
  if (c < 256) {
    i = c % 16 + 1;
    j = c / 16 + 1;
  } else {
    const int g = c - 256;
    ghost_coords(g >> 4, 1, (g & 15) + 1, i, j);
  }
}

// The states on the two sides of a face: the cells c0 and c0 + stride of the
// tile (and the next ones for choice 2's reconstruction).  A y-face's states
// are swapped into the x frame (swapy, src/swapy.f90:4-13), so one solver call
// serves both.
template <int NEQ>
__device__ __forceinline__ void face_state(const double *prim, int c, bool yf, double *q) {
#pragma unroll
  for (int k = 0; k < NEQ; ++k) q[k] = prim[((k == 1 || k == 2) && yf ? 3 - k : k) * NC + c];
}

// A block's faces, shared out over the workgroup; face(yf, c0, stride, ff)
// gives the flux.  LDSX: x-face fi = 0..16 of row j goes to F at
// [k][(j-1)*17+fi], y-face fj = 0..16 of column i to G at [k][fj*16+(i-1)].
// Otherwise a cell's left x-face stays with the cell's thread (fx, threads
// below 256) and F is not used: the waves take the 288 other faces first (the
// y-faces, then the right x-faces of row j to G at [k][272+(j-1)]; the lanes
// past the last repeat it) and the cells' own last, so that these take
// registers only after the sweep.
constexpr int NG = 288;   // fluxes per variable in G
template <int NEQ, int BS, bool LDSX, class Face>
__device__ __forceinline__ void sweep_faces(int wave, double *F, double *G, double *fx, Face face) {
  if constexpr (LDSX) {
    for (int f = tid_again(wave); f < 544; f += BS) {
      const bool yf = f >= 272;
      const int g = yf ? f - 272 : f;
      const int c0 = yf ? IDX(g % 16 + 1, g / 16) : IDX(g % 17, g / 17 + 1);
      double ff[NEQ];
      face(yf, c0, yf ? NP : 1, ff);
      double *o = yf ? G : F;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) o[((k == 1 || k == 2) && yf ? 3 - k : k) * 272 + g] = ff[k];
    }
  } else {
    for (int r = wave < 4 ? wave * 64 + BS - 256 : wave * 64 - 256; r < NG || wave < 4; r += BS) {
      const int tid = tid_again(wave);
      const bool own = r >= NG;
      const int g = own ? tid : min(r + (tid & 63), NG - 1);   // cell, or place in G
      const bool yf = !own && g < 272;
      const int c0 = yf ? IDX(g % 16 + 1, g / 16) : (own ? IDX(g % 16, g / 16 + 1) : IDX(16, g - 271));
      double ff[NEQ];
      face(yf, c0, yf ? NP : 1, ff);
      if (own) {
#pragma unroll
        for (int k = 0; k < NEQ; ++k) fx[k] = ff[k];
        break;
      }
#pragma unroll
      for (int k = 0; k < NEQ; ++k) G[((k == 1 || k == 2) && yf ? 3 - k : k) * NG + g] = ff[k];
    }
  }
}

// Flux sweep shared by both stages.  prim: LDS tile [NEQ][NC].  Choice 1
// (stage A) takes the fluxes through LDS; choice 2 (stage B) reconstructs with
// the limiter and keeps the cells' left ones.  SOLVER / LIM fix the solver and
// limiter at compile time (-1 / -99: read from p); the arithmetic is the same
// either way.
template <int NEQ, int CHOICE, int BS, int SOLVER = -1, int LIM = -99>
__device__ __forceinline__ int flux_sweep_t(const wx_params *__restrict__ p, int wave, const double *prim, double *F,
                                            double *G, double *fx) {
  int err = 0;
  const int lim = LIM != -99 ? LIM : p->limiter;
  sweep_faces<NEQ, BS, CHOICE == 1>(wave, F, G, fx, [&](bool yf, int c0, int stride, double *ff) __attribute__((always_inline)) {
    double ql[NEQ], qr[NEQ];
    face_state<NEQ>(prim, c0, yf, ql);
    face_state<NEQ>(prim, c0 + stride, yf, qr);
    if constexpr (CHOICE == 2) {
      double qll[NEQ], qrr[NEQ];
      face_state<NEQ>(prim, c0 - stride, yf, qll);
      face_state<NEQ>(prim, c0 + 2 * stride, yf, qrr);
      limiter<NEQ>(lim, qll, ql, qr, qrr);
    }
    err |= riemann<NEQ, SOLVER>(p, ql, qr, ff);
  });
  return err;
}

// The sweep with the common configurations compiled in: HLLC, and in
// stage B the minmod or van Leer limiter; anything else reads p.
template <int NEQ, int CHOICE, int BS>
__device__ __forceinline__ int flux_sweep(const wx_params *__restrict__ p, int wave, const double *prim, double *F,
                                          double *G, double *fx) {
  if (p->solver == 0) {
    if (CHOICE == 1) return flux_sweep_t<NEQ, CHOICE, BS, 0>(p, wave, prim, F, G, fx);
    if (p->limiter == 1) return flux_sweep_t<NEQ, CHOICE, BS, 0, 1>(p, wave, prim, F, G, fx);
    if (p->limiter == 2) return flux_sweep_t<NEQ, CHOICE, BS, 0, 2>(p, wave, prim, F, G, fx);
  }
  return flux_sweep_t<NEQ, CHOICE, BS>(p, wave, prim, F, G, fx);
}

// The sweep of a block of mild primitives (wx_physics.h).  cs: the cells'
// sound speeds in the tile's layout (choice 1, whose face states are cells).
// Returns whether every face of this thread was served.
template <int NEQ, int CHOICE, int BS, int SOLVER, int LIM>
__device__ __forceinline__ bool flux_sweep_short(const wx_params *__restrict__ p, int wave, const double *prim,
                                                 const double *cs, double *F, double *G, double *fx) {
  bool ok = true;
  sweep_faces<NEQ, BS, CHOICE == 1>(wave, F, G, fx, [&](bool yf, int c0, int stride, double *ff) __attribute__((always_inline)) {
    double ql[NEQ], qr[NEQ];
    face_state<NEQ>(prim, c0, yf, ql);
    face_state<NEQ>(prim, c0 + stride, yf, qr);
    if constexpr (CHOICE == 2) {
      double qll[NEQ], qrr[NEQ];
      face_state<NEQ>(prim, c0 - stride, yf, qll);
      face_state<NEQ>(prim, c0 + 2 * stride, yf, qrr);
      limiter_mild<NEQ, LIM>(qll, ql, qr, qrr);
      const Rcp rl = rdiv(ql[0]), rr = rdiv(qr[0]);
      const double csl = fsqrt(quot(p->gamma * ql[3], rl)), csr = fsqrt(quot(p->gamma * qr[3], rr));
      ok = riemann_mild<NEQ, SOLVER, true>(p, ql, qr, csl, csr, rl, rr, ff) & ok;
    } else {
      const Rcp none{0.0, 0.0};
      ok = riemann_mild<NEQ, SOLVER, false>(p, ql, qr, cs[c0], cs[c0 + stride], none, none, ff) & ok;
    }
  });
  return ok;
}

// The short form where it holds (every primitive the faces read is mild; the
// limiter minmod or van Leer), redone in the general form by the waves that
// meet a face it does not serve.
template <int NEQ, int CHOICE, int BS>
__device__ __forceinline__ int flux_sweep_mild(const wx_params *__restrict__ p, int wave, bool mild, const double *prim,
                                               const double *cs, double *F, double *G, double *fx) {
  bool ok = false;
  const int solver = p->solver, lim = CHOICE == 1 ? 1 : p->limiter;
  if (!WX_RARE(!mild) && lim == 1) {
    if (solver == 0) ok = flux_sweep_short<NEQ, CHOICE, BS, 0, 1>(p, wave, prim, cs, F, G, fx);
    else if (solver == 1) ok = flux_sweep_short<NEQ, CHOICE, BS, 1, 1>(p, wave, prim, cs, F, G, fx);
    else ok = flux_sweep_short<NEQ, CHOICE, BS, 2, 1>(p, wave, prim, cs, F, G, fx);
  } else if (CHOICE == 2 && !WX_RARE(!mild) && lim == 2) {
    if (solver == 0) ok = flux_sweep_short<NEQ, CHOICE, BS, 0, 2>(p, wave, prim, cs, F, G, fx);
    else if (solver == 1) ok = flux_sweep_short<NEQ, CHOICE, BS, 1, 2>(p, wave, prim, cs, F, G, fx);
    else ok = flux_sweep_short<NEQ, CHOICE, BS, 2, 2>(p, wave, prim, cs, F, G, fx);
  }
  if (!WX_RARE(!__all(ok))) return 0;
  // (with the solver and limiter compiled in here as well, stage B spills: 81
  // registers with five variables, a wave per SIMD less with six)
  return flux_sweep_t<NEQ, CHOICE, BS>(p, wave, prim, F, G, fx);
}

// The right x-face's flux of cell tid's thread: its right neighbour's left
// one (the lane above, within the row of 16), or for the last cell of row j
// the one in G.  Whole waves.
__device__ __forceinline__ double flux_right(double left, const double *G, int j) {
  const double edge = G[272 + j - 1];
  const uint64_t l = (uint64_t)__double_as_longlong(left), e = (uint64_t)__double_as_longlong(edge);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)e, (int)(uint32_t)l, 0x101, 0xf, 0xf, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp((int)(uint32_t)(e >> 32), (int)(uint32_t)(l >> 32), 0x101, 0xf,
                                                            0xf, false);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Whether every wave of the workgroup found its cells mild: each wave's
// verdict goes to its word of w before a barrier, and is read after it.
__device__ __forceinline__ void mild_vote(uint32_t *w, int wave, bool ok) {
  w[wave] = __all(ok) ? 0u : 1u;   // the same word from every lane
}
template <int BS>
__device__ __forceinline__ bool mild_result(const uint32_t *w) {
  uint32_t bad = 0;
#pragma unroll
  for (int k = 0; k < BS / 64; ++k) bad |= w[k];
  return __builtin_amdgcn_readfirstlane(bad) == 0;
}

// dt/dx and dt/dy of a block's update (uniform).
__device__ __forceinline__ void dt_over_dx(const wx_params *__restrict__ p, bool pok, double dt, int level,
                                           double &dtdx, double &dtdy) {
  const double dx = p->dx[level - 1], dy = p->dy[level - 1];
  if (pok && unit_range(dt)) {
    dtdx = fdiv(dt, dx);
    dtdy = __double_as_longlong(dx) == __double_as_longlong(dy) ? dtdx : fdiv(dt, dy);
  } else {
    dtdx = dt / dx;
    dtdy = dt / dy;
  }
}

// Cylindrical source terms, src/step.f90:49-76 (prims of the stage).
template <int NEQ, bool MILD>
__device__ __forceinline__ void cyl_source(const wx_params *__restrict__ p, const double *prim, int i,
                                           int j, int icy, int lev, double *S) {
  double radius = ((double)(j + icy) - 0.5) * p->dy[lev - 1];
  double rho = prim[0 * NC + IDX(i, j)];
  double v1 = prim[1 * NC + IDX(i, j)], v2 = prim[2 * NC + IDX(i, j)], pr = prim[3 * NC + IDX(i, j)];
  double H = 0.5 * rho * (v1 * v1 + v2 * v2) + (p->cv + 1.) * pr;
  const Rcp rr = rdiv_<MILD>(radius);
  S[0] = -quot_<MILD>(rho * v2, rr);
  S[1] = -quot_<MILD>(rho * v1 * v2, rr);
  S[2] = -quot_<MILD>(rho * v2 * v2, rr);
  S[3] = -quot_<MILD>(H * v2, rr);
#pragma unroll
  for (int k = 4; k < NEQ; ++k) S[k] = -quot_<MILD>(prim[k * NC + IDX(i, j)] * v2, rr);
}

// ---------------------------------------------------------------------
// Stage A: src/tstep.f90:22-46 (hllcfluxes choice 1 + step with dt/2).
// MILD: the short divisions where they hold (wx_physics.h), and the cells'
// sound speeds taken once per cell instead of once per face and side.
// DT: the step's dt too (k_dtreduce with advance), at most BS blocks of one
// instance: every workgroup takes it from all blocks' partials, in the order
// k_dtreduce takes, and workgroup 0 writes it.
template <int NEQ, int BS, bool PERSIST, bool MILD, bool DT = false>
__device__ __forceinline__ void stageA_body(const wx_params *__restrict__ P, QueueRef q, const double *__restrict__ U,
                                            double *__restrict__ Q, const double *__restrict__ Pc,
                                            DevScalars *__restrict__ Sa) {
  __shared__ double prim[NEQ * NC];
  __shared__ double F[NEQ * 272];
  __shared__ double G[NEQ * 272];
  __shared__ double cst[MILD ? 18 * NP : 1];   // sound speeds of rows 0..17
  __shared__ uint32_t votes[BS / 64];
  __shared__ double dtw[2][BS / 64];   // DT: the waves' minima
  const int wave = wave_of();
  // the first entry's record is read together with the queue length
  const int b0 = PERSIST ? (int)blockIdx.x : xcd_entry(blockIdx.x, gridDim.x);
  LeafRec Lnext = q.rec[min(b0, q.cap - 1)];
  const int nleaf = q.hdr->nleaf;
  // one queue entry per workgroup, or (PERSIST) entries blockIdx.x +
  // k * gridDim.x; the loop form costs registers, so each is its own kernel
  for (int l = b0; l < nleaf; l += gridDim.x) {
  const LeafRec L = Lnext;
  if (PERSIST && l + (int)gridDim.x < nleaf) Lnext = q.rec[l + gridDim.x];
  const wx_params *__restrict__ p = P + L.inst;
  DevScalars *__restrict__ S = Sa + L.inst;
  const double *ub = U + (size_t)L.id * NEQ * NC;
  // the interior and ghost layer 1 are one contiguous range of every
  // variable.  Under DMC the pressure of cells 0..17 is the one the last
  // cooling left (the reference's primit, src/coolingdmc.f90:27-38 and
  // src/tstep.f90:27-36), not the one u gives back.
  const bool carried = Pc && p->cooling == 2;
  if constexpr (DT) {
    const int tid = tid_again(wave);
    double a = 1.e30, c = 1e30;
    if (tid < nleaf) {
      const int id = q.rec[tid].id;
      a = dmin(a, q.stat[2 * id]);
      c = dmin(c, q.stat[2 * id + 1]);
    }
    for (int o = 32; o > 0; o >>= 1) {
      a = dmin(a, __shfl_xor(a, o));
      c = dmin(c, __shfl_xor(c, o));
    }
    if ((tid & 63) == 0) { dtw[0][wave] = a; dtw[1][wave] = c; }
  }
  const double *pcb = carried ? Pc + (size_t)L.id * NC : nullptr;
  const bool pok = MILD && mild_params(p, L.level);
  bool ok = pok;
  if constexpr (MILD) {
    const RecipP rp = recip_params(p);
    const double tiny = mild_tiny(p);
#pragma unroll
    for (int n = 0; n < (320 + BS - 1) / BS; ++n) {
      const int c = tid_again(wave) + n * BS;
      if (c >= 320) break;
      double uu[NEQ], q[NEQ], T;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) uu[k] = ub[k * NC + c];
      bool okc = uprim_mild<NEQ>(p, rp, tiny, q, uu, T) & pok;
      if (carried) {
        q[3] = pcb[c];
        okc &= (q[3] >= 0x1p-64) & (q[3] <= kHuge);
      }
      int i, j;
      tile_ij(c, i, j);
      cst[IDX(i, j) - NP] = fsqrt(fdiv(p->gamma * q[3], q[0]));
      if (WX_RARE(!okc)) {
        const double pc = q[3];
        uprim<NEQ>(p, q, uu, T);
        if (carried) q[3] = pc;
      }
      ok &= okc;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(i, j)] = q[k];
    }
    mild_vote(votes, wave, ok);
  } else {
    for (int c = tid_again(wave); c < 320; c += BS) {
      double uu[NEQ], q[NEQ], T;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) uu[k] = ub[k * NC + c];
      uprim<NEQ>(p, q, uu, T);
      if (carried) q[3] = pcb[c];
      int i, j;
      tile_ij(c, i, j);
#pragma unroll
      for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(i, j)] = q[k];
    }
  }
  __syncthreads();
  const bool mild = MILD && mild_result<BS>(votes);
  int err;
  if constexpr (MILD) err = flux_sweep_mild<NEQ, 1, BS>(p, wave, mild, prim, cst - NP, F, G, nullptr);
  else err = flux_sweep<NEQ, 1, BS>(p, wave, prim, F, G, nullptr);
  __syncthreads();
  const int tid = tid_again(wave);
  double dt;
  if constexpr (DT) {
    double a = dtw[0][0], c = dtw[1][0];
#pragma unroll
    for (int k = 1; k < BS / 64; ++k) { a = dmin(a, dtw[0][k]); c = dmin(c, dtw[1][k]); }
    if (BS < 1024) { a = dmin(a, 1.e30); c = dmin(c, 1e30); }   // k_dtreduce's waves without a block
    dt = dmin(p->cfl * a, 0.4 * c * p->Psc / p->tsc);
    // written by a thread past the cells'
    if (blockIdx.x == 0 && tid == BS - 1) {
      S->dtp_min = a;
      S->dtcool_min = c;
      S->dt = dt;
      const double t = S->time + dt;
      S->time = t;
      if (p->otherb) {
        S->vjet = jet_velocity(p, t);
        S->vjet_time = t;
        S->vjet_ok = 1;
      }
    }
  } else {
    dt = S->dt;
  }
  if (tid < 256) {   // one thread per interior cell
    const double dtm = dt / 2.;
    double dtdx, dtdy;
    dt_over_dx(p, pok, dtm, L.level, dtdx, dtdy);
    const int i = tid % 16 + 1, j = tid / 16 + 1;
    double Sc[NEQ];
    if (p->cylindrical) {
      if (mild) cyl_source<NEQ, true>(p, prim, i, j, L.icy, L.level, Sc);
      else cyl_source<NEQ, false>(p, prim, i, j, L.icy, L.level, Sc);
    }
    double *qb = Q + (size_t)L.id * NEQ * NC;
#pragma unroll
    for (int k = 0; k < NEQ; ++k) {
      double v = ub[k * NC + tid] - dtdx * (F[k * 272 + (j - 1) * 17 + i] - F[k * 272 + (j - 1) * 17 + i - 1])
                 - dtdy * (G[k * 272 + j * 16 + (i - 1)] - G[k * 272 + (j - 1) * 16 + (i - 1)]);
      if (p->cylindrical) v = v + dtm * Sc[k];
      qb[k * NC + tid] = v;
    }
  }
  if (err) atomicOr(&S->err, WX_EHLLC);
  __syncthreads();   // the next queue entry reuses the LDS tiles
   if (!PERSIST) break;   // one entry per workgroup: no loop
  }
}

// The one-entry-per-workgroup form is compiled for 8 waves per SIMD (at 512
// threads that caps it at 64 VGPRs, with a few spills: 8.5 vs 9.2 ns per
// block at 74 VGPRs and 6 waves on the 16-variant cooling jet; the smaller
// workgroups are held to fewer waves by their LDS anyway).
template <int NEQ, int BS, bool PERSIST>
__global__ __launch_bounds__(BS, PERSIST ? 1 : 8) void k_stageA(const wx_params *__restrict__ P, QueueRef q,
                                                const double *__restrict__ U, double *__restrict__ Q,
                                                const double *__restrict__ Pc, DevScalars *__restrict__ Sa) {
  stageA_body<NEQ, BS, PERSIST, false>(P, q, U, Q, Pc, Sa);
}
// For the few blocks it serves (wx_host.cpp) two workgroups a compute unit are enough.
template <int NEQ>
__global__ __launch_bounds__(512, 4) void k_stageA_dt(const wx_params *__restrict__ P, QueueRef q,
                                                const double *__restrict__ U, double *__restrict__ Q,
                                                const double *__restrict__ Pc, DevScalars *__restrict__ Sa) {
  stageA_body<NEQ, 512, false, false, true>(P, q, U, Q, Pc, Sa);
}
template <int NEQ, int BS>
__global__ __launch_bounds__(BS, 8) void k_stageA_mild(const wx_params *__restrict__ P, QueueRef q,
                                                const double *__restrict__ U, double *__restrict__ Q,
                                                const double *__restrict__ Pc, DevScalars *__restrict__ Sa) {
  stageA_body<NEQ, BS, false, true>(P, q, U, Q, Pc, Sa);
}

// ---------------------------------------------------------------------
// Stage B: src/tstep.f90:53-88 with boundaryII pulled from the neighbours.
// Bound by memory latency at the occupancy its registers allow (without the
// fluxes it takes three quarters of the time).  MILD: the short divisions where they hold (wx_physics.h).
template <int NEQ, int BS, bool PERSIST, bool MILD>
__device__ __forceinline__ void stageB_body(const wx_params *__restrict__ P, QueueRef q, const int2 *__restrict__ ops,
                                            const BlockRec *__restrict__ binfo, double *__restrict__ U,
                                            const double *__restrict__ Q, double *__restrict__ Qring,
                                            DevScalars *__restrict__ Sa) {
  __shared__ double prim[NEQ * NC];
  __shared__ double G[NEQ * NG];
  __shared__ uint32_t votes[BS / 64];
  const int wave = wave_of();
  const int b0 = PERSIST ? (int)blockIdx.x : xcd_entry(blockIdx.x, gridDim.x);
  LeafRec Lnext = q.rec[min(b0, q.cap - 1)];
  const int nleaf = q.hdr->nleaf;
  for (int l = b0; l < nleaf; l += gridDim.x) {
  const int r = l;
  const LeafRec L = Lnext;
  if (PERSIST && l + (int)gridDim.x < nleaf) Lnext = q.rec[l + gridDim.x];
  const wx_params *__restrict__ p = P + L.inst;
  DevScalars *__restrict__ S = Sa + L.inst;
  const int b = L.id;
  const double time = S->time;
  const bool imp = (L.flags & 1) != 0;
  const double vjet = p->otherb ? jet_velocity_at(p, S, time) : 0.0;
  const double *qb = Q + (size_t)b * NEQ * NC;
  double *ub = U + (size_t)b * NEQ * NC;
  const int tid0 = tid_again(wave);
  // two-layer ghost ring: 4 sides x 2 layers x 16 positions = 128 cells,
  // gathered by waves of their own when the workgroup has them.  The op of
  // the ghost's segment is read first, so that its latency overlaps the
  // interior's primitive recovery.
  const int gt = BS >= 384 ? tid0 - 256 : tid0;
  const bool ghost = gt >= 0 && gt < 128;
  const int side = gt >> 5, layer = ((gt >> 4) & 1) + 1, pos = (gt & 15) + 1;
  const bool keep1 = (p->compat & 2) && p->bc[2] == 0;   // lb_outfyb
  int2 op = make_int2(0, 0);
  if (ghost) op = ops[r * 8 + side * 2 + ((pos - 1) >> 3)];
  const bool pok = MILD && mild_params(p, L.level);
  RecipP rp{};
  double tiny = 0.0;
  if constexpr (MILD) {
    rp = recip_params(p);
    tiny = mild_tiny(p);
  }
  bool ok = true;
  auto recover = [&](double *q, const double *uu) __attribute__((always_inline)) {
    double T;
    if constexpr (MILD) ok &= uprim_any<NEQ>(p, rp, pok, tiny, q, uu, T);
    else uprim<NEQ>(p, q, uu, T);
  };
  // interior of U^{n+1/2} (imposed when the block is in the source list)
  if (tid0 < 256) {
    const int i = tid0 % 16 + 1, j = tid0 / 16 + 1;
    double uu[NEQ], q[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = qb[k * NC + tid0];
    if (imp && in_jet(p, L.level, L.icx, L.icy, i, j)) jet_state<NEQ>(p, vjet, uu);
    recover(q, uu);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(i, j)] = q[k];
  }
  if (ghost) {
    double gh[NEQ];
    int gi, gj;
    ghost_gather<NEQ>(p, Q, binfo, op, b, L.level, L.icx, L.icy, side, layer, pos, vjet, gh);
    ghost_coords(side, layer, pos, gi, gj);
    // the ring of U^{n+1/2} goes to its own tile's ring in the U^{n+1/2}
    // buffer (Qring is Q: this launch reads only interiors of Q), where the
    // fill leaves layer 2 as the step's final value (src/tstep.f90:85 copies
    // up's ring into u; boundaryI rewrites layer 1, except the segments that
    // the OUTFYB mode's list leaves to the carried values)
    if (layer == 2 || keep1) {
      double *rb = Qring + (size_t)b * NEQ * NC + 256 + (layer - 1) * 64 + side * 16 + pos - 1;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) rb[k * NC] = gh[k];
    }
    double q[NEQ];
    recover(q, gh);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(gi, gj)] = q[k];
  }
  if constexpr (MILD) mild_vote(votes, wave, ok);
  __syncthreads();
  const bool mild = MILD && mild_result<BS>(votes);
  int err;
  double fx[NEQ];
  if constexpr (MILD) err = flux_sweep_mild<NEQ, 2, BS>(p, wave, mild, prim, nullptr, nullptr, G, fx);
  else err = flux_sweep<NEQ, 2, BS>(p, wave, prim, nullptr, G, fx);
  const int tid = tid_again(wave);
  double u0[NEQ];
  if (tid < 256) {
#pragma unroll
    for (int k = 0; k < NEQ; ++k) u0[k] = ub[k * NC + tid];
  }
  __syncthreads();
  const int i = tid % 16 + 1, j = tid / 16 + 1;
  double Sc[NEQ];
  if (tid < 256 && p->cylindrical) {
    if (mild) cyl_source<NEQ, true>(p, prim, i, j, L.icy, L.level, Sc);
    else cyl_source<NEQ, false>(p, prim, i, j, L.icy, L.level, Sc);
  }
  // the viscosity's stencil (src/viscosity.f90:6-25, on the finest two
  // levels, src/tstep.f90:82) reads Uⁿ of the interior and of ghost layer 1
  // from the primitive tile, which is free after the sweep
  const bool visc = L.level >= p->nlevs - 1;
  if (visc) {
    __syncthreads();   // the sweep's and the sources' reads of the primitives are done
    if (tid < 256)
#pragma unroll
      for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(i, j)] = u0[k];
    for (int g = tid; g < 64; g += blockDim.x) {
      int ri, rj;
      ghost_coords(g >> 4, 1, (g & 15) + 1, ri, rj);
#pragma unroll
      for (int k = 0; k < NEQ; ++k) prim[k * NC + IDX(ri, rj)] = ub[k * NC + 256 + g];
    }
    __syncthreads();
  }
  double un[NEQ];
  if (tid < 256) {   // one thread per interior cell
    const double dt = S->dt;
    double dtdx, dtdy;
    dt_over_dx(p, pok, dt, L.level, dtdx, dtdy);
    const double eta = p->eta;
#pragma unroll
    for (int k = 0; k < NEQ; ++k) {
      const double *uk = prim + k * NC;
      double v = u0[k] - dtdx * (flux_right(fx[k], G + k * NG, j) - fx[k])
                 - dtdy * (G[k * NG + j * 16 + (i - 1)] - G[k * NG + (j - 1) * 16 + (i - 1)]);
      if (p->cylindrical) v = v + dt * Sc[k];
      if (visc)   // no dt factor
        v = v + eta * (uk[IDX(i + 1, j)] + uk[IDX(i - 1, j)] + uk[IDX(i, j + 1)] + uk[IDX(i, j - 1)] - 4. * u0[k]);
      un[k] = v;
    }
  }
  // each thread writes the one interior cell of Uⁿ it read (the stencil's
  // reads of other cells were from the tile in LDS)
  if (tid < 256)
#pragma unroll
    for (int k = 0; k < NEQ; ++k) ub[k * NC + tid] = un[k];
  if (err) atomicOr(&S->err, WX_EHLLC);
  __syncthreads();   // the next queue entry reuses the LDS tiles
   if (!PERSIST) break;   // one entry per workgroup: no loop
  }
}

// Five workgroups on a compute unit: 27.5 KB of LDS (the cells' left x-fluxes
// stay in registers and cross to the left neighbour between lanes; with all of
// them in LDS it was 37.8 KB) and 96 VGPRs (the ghosts are written out when
// gathered, U^n is read after the sweep).  us per launch at four / five:
// 1 174 blocks, of which four hold 1 024 at a time, 21.6 / 19.6; 5 319
// 58.5 / 54.3; 19 250 203 / 191.  Six variables need more registers.
constexpr int kStageBWaves = 5;
template <int NEQ, int BS, bool PERSIST>
__global__ __launch_bounds__(BS, PERSIST || NEQ > 5 ? 1 : kStageBWaves) void k_stageB(const wx_params *__restrict__ P, QueueRef q,
                                                const int2 *__restrict__ ops,
                                                const BlockRec *__restrict__ binfo,
                                                double *__restrict__ U, const double *__restrict__ Q,
                                                double *__restrict__ Qring, DevScalars *__restrict__ Sa) {
  stageB_body<NEQ, BS, PERSIST, false>(P, q, ops, binfo, U, Q, Qring, Sa);
}
template <int NEQ, int BS>
__global__ __launch_bounds__(BS, NEQ > 5 ? 1 : kStageBWaves) void k_stageB_mild(const wx_params *__restrict__ P, QueueRef q,
                                                const int2 *__restrict__ ops,
                                                const BlockRec *__restrict__ binfo,
                                                double *__restrict__ U, const double *__restrict__ Q,
                                                double *__restrict__ Qring, DevScalars *__restrict__ Sa) {
  stageB_body<NEQ, BS, false, true>(P, q, ops, binfo, U, Q, Qring, Sa);
}

// ---------------------------------------------------------------------
// Block statistics: CFL partials (src/timestep.f90:29-41) and the
// refinement flag (src/criteria.f90:16-50) from a tile of primitives.
// Indexed by block ID: stat[2id] = min dx/(|u|+cs), dy/(|v|+cs);
// stat[2id+1] = DMC t_cool min; flag[id]: 1 refine, 2 coarsen, 0 neither.
// BS below 256: each wave takes several groups of 64 cells, one after the
// other, and the groups are folded in the same order.
template <int NEQ, int BS = 256>
__device__ __forceinline__ void block_stats(const wx_params *__restrict__ p, bool pok, const double *prim, int id, int lev,
                                            double *stat, int8_t *flag, int8_t *flagq) {
  __shared__ double red[3][16];
  const int tid = threadIdx.x;
  double dtp, dtc, grad;
#pragma unroll 1
  for (int n = 0; n < (BS < 256 ? 256 / BS : 1); ++n) {
  const int cell_id = tid + n * BS;
  const int i = cell_id % 16 + 1, j = cell_id / 16 + 1;
  dtp = 1.e30;
  dtc = 1e30;
  grad = 0.;
  if (cell_id < 256) {   // one thread per interior cell
    const double rho = prim[0 * NC + IDX(i, j)], vx = prim[1 * NC + IDX(i, j)];
    const double vy = prim[2 * NC + IDX(i, j)], pr = prim[3 * NC + IDX(i, j)];
    const double *P4 = prim + 3 * NC, *P1 = prim;
    // the reference's max of the four quotients |dP|/am is the quotient of
    // the largest |dP| (a correctly rounded division by am > 0 is monotonic),
    // bit for bit, at one division instead of four
    const double dp = dmax(dmax(dmax(fabs(P4[IDX(i + 1, j)] - pr), fabs(P4[IDX(i - 1, j)] - pr)),
                                fabs(P4[IDX(i, j + 1)] - pr)), fabs(P4[IDX(i, j - 1)] - pr));
    const double dr = dmax(dmax(dmax(fabs(P1[IDX(i + 1, j)] - rho), fabs(P1[IDX(i - 1, j)] - rho)),
                                fabs(P1[IDX(i, j + 1)] - rho)), fabs(P1[IDX(i, j - 1)] - rho));
    // the short divisions where the cell is in their range (the primitives
    // are floored; a difference is zero or at least an ulp of them)
    const bool mild = pok & (rho >= 1e-15) & (rho <= kHuge) & (pr >= 0x1p-64) & (pr <= kHuge) & (fabs(vx) <= kHuge) &
                      (fabs(vy) <= kHuge) & (dp <= 0x1p200) & (dr <= 0x1p200);
    auto cell = [&](auto short_form) __attribute__((always_inline)) {
      constexpr bool M = decltype(short_form)::value;
      const double cs = sqrt_<M>(div_<M>(p->gamma * pr, rho));
      dtp = dmin(dtp, div_<M>(p->dx[lev - 1], fabs(vx) + cs));
      dtp = dmin(dtp, div_<M>(p->dy[lev - 1], fabs(vy) + cs));
      const double am = dmax(1e-15, fabs(pr));
      const double am2 = dmax(1e-15, fabs(rho));
      grad = dmax(div_<M>(dp, am), div_<M>(dr, am2));
    };
    if (!WX_RARE(!mild)) cell(std::true_type{});
    else cell(std::false_type{});
    if (p->cooling == 2) {
      double T = (pr / rho) * p->Tempsc;
      if (T > 1e4) {
        double al = cooldmc(p, T) * (rho * rho);
        dtc = dmin(dtc, p->cv * pr / al);
      }
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    dtp = dmin(dtp, __shfl_xor(dtp, o));
    dtc = dmin(dtc, __shfl_xor(dtc, o));
    grad = dmax(grad, __shfl_xor(grad, o));
  }
  const int w = cell_id >> 6;
  if ((tid & 63) == 0) { red[0][w] = dtp; red[1][w] = dtc; red[2][w] = grad; }
  }
  __syncthreads();
  if (tid == 0) {
    if (BS < 256) {
      dtp = red[0][0];
      dtc = red[1][0];
      grad = red[2][0];
    }
    for (int k = 1; k < (BS < 256 ? 4 : (int)(blockDim.x >> 6)); ++k) {
      dtp = dmin(dtp, red[0][k]);
      dtc = dmin(dtc, red[1][k]);
      grad = dmax(grad, red[2][k]);
    }
    stat[2 * id] = dtp;
    stat[2 * id + 1] = dtc;
    int8_t fl = 0;
    if (grad >= p->tol) fl = (lev < p->nlevs) ? 1 : 0;
    else if (grad <= p->tol2) fl = 2;
    flag[id] = fl;
    if (flagq) *flagq = fl;
  }
}

// ---------------------------------------------------------------------
// boundaryI + cooling (+ CFL / criteria epilogue): src/tstep.f90:92-122.
// Cooling surrogate on the 18x18 cells of a tile (coolingh instances only):
// features per cell, the network per wave on groups of 16 cells (matrix
// cores), then per cell either the network's update or -- outside the
// training hull or when the energy residual exceeds the tolerance -- the
// exact routine.  The network's temperature output is a correction to the
// routine's relaxation law T1 = 10 + (T - 10) exp(-ce dt)
// (src/coolingh.f90:249-250) evaluated with the tabulated loss; the energy
// residual is the change of thermal energy (2 - y1) T1 that correction
// makes, relative to the old thermal energy (2 - y0) T.
// A cell outside takes the exact routine in a pass of its own, over a list
// of such cells: a wave that held one of them used to run it for all its cells.
// Each cell is worked on by the thread that loaded it into the tile (cell
// tid, then tid + BS), which also writes its cooled state to ob and its
// primitives to the tile.  The inference reads every cell's features.
template <int NEQ, int BS>
__device__ __forceinline__ void cool_surrogate(const wx_params *__restrict__ p, SurDev *__restrict__ M, double dts,
                                               double *tile, double *__restrict__ ob) {
  constexpr int NWAVE = BS / 64, G = (20 + NWAVE - 1) / NWAVE;   // 20 groups of 16 cells
  __shared__ bf16x4 sx[320];
  __shared__ float sy[320 * 2];
  __shared__ float scedt[320];      // ce dt of the tabulated relaxation; negative outside the hull
  __shared__ double sT[320], sK[320];   // temperature, kinetic energy
  __shared__ uint16_t list[320];
  __shared__ uint32_t nfb;
  const int tid = threadIdx.x;
  if (tid == 0) nfb = 0u;
#pragma unroll
  for (int n = 0; n < (320 + BS - 1) / BS; ++n) {
    const int c = tid + n * BS;
    if (c >= 320) break;
    int i, j;
    tile_ij(c, i, j);
    double uu[NEQ], q[NEQ], T;
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = tile[k * NC + IDX(i, j)];
    uprim<NEQ>(p, q, uu, T);
    float f[4], cedt;
    const bool in = sur_features(M, uu[0], T, uu[4] / uu[0], dts, f, cedt);
#pragma unroll
    for (int k = 0; k < 4; ++k) f[k] = (f[k] - M->in_mu[k]) / M->in_sig[k];
    sx[c] = pack4(f[0], f[1], f[2], f[3]);
    scedt[c] = in ? cedt : -1.f;
    sT[c] = T;
    sK[c] = 0.5 * q[0] * (q[1] * q[1] + q[2] * q[2]);
  }
  __syncthreads();
  {
    const int l = tid & 63, r = l & 15, qq = l >> 4, w = tid >> 6;
    bf16x4 xb[G];
    f32x4 y[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int c = 16 * (w + NWAVE * g) + r;
      xb[g] = bf16x4{0, 0, 0, 0};
      if (qq == 0 && c < 320) xb[g] = sx[c];
    }
    mlp_fwd16<G>(M, xb, y);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int c = 16 * (w + NWAVE * g) + r;
      if (qq == 0 && c < 320) {
        sy[2 * c] = y[g][0];
        sy[2 * c + 1] = y[g][1];
      }
    }
  }
  __syncthreads();
  auto put = [&](int c, int i, int j, const double *uu) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NEQ; ++k) ob[k * NC + c] = uu[k];
    double q[NEQ], T;
    uprim<NEQ>(p, q, uu, T);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) tile[k * NC + IDX(i, j)] = q[k];
  };
#pragma unroll
  for (int n = 0; n < (320 + BS - 1) / BS; ++n) {
    const int c = tid + n * BS;
    if (c >= 320) break;
    int i, j;
    tile_ij(c, i, j);
    double uu[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = tile[k * NC + IDX(i, j)];
    const double T = sT[c];
    const double y0 = uu[4] / uu[0];
    const float corr = sy[2 * c] * M->out_sig[0] + M->out_mu[0];
    const float dx = sy[2 * c + 1] * M->out_sig[1] + M->out_mu[1];
    double y1 = y0 - (double)dx;
    y1 = dmin(y1, 1.);
    y1 = dmax(y1, 0.0001);
    // the relaxation law with the tabulated loss, then the network's
    // correction log10(T1 / T1_table)
    const float cedt = scedt[c];
    double tt = 10. + (T - 10.) * (double)__expf(-cedt);
    tt = dmax(tt, 0.1 * T);
    tt = dmin(tt, 10. * T);
    tt = dmax(tt, 10.);
    double t1 = tt * (double)exp10f(corr);
    t1 = dmax(t1, 0.1 * T);
    t1 = dmin(t1, 10. * T);
    t1 = dmax(t1, 10.);
    const double resid = (2. - y1) * fabs(t1 - tt) / ((2. - y0) * T);
    if (!(cedt >= 0.f) || !(resid <= (double)M->tol)) {
      list[atomicAdd(&nfb, 1u)] = (uint16_t)c;
    } else {
      uu[4] = y1 * uu[0];
      uu[3] = p->cv * (2. * uu[0] - uu[4]) * t1 / p->Tempsc + sK[c];
      put(c, i, j, uu);
    }
  }
  __syncthreads();
  const uint32_t n = nfb;
  for (uint32_t k = tid; k < n; k += BS) {
    const int c = list[k];
    int i, j;
    tile_ij(c, i, j);
    double uu[NEQ];
#pragma unroll
    for (int v = 0; v < NEQ; ++v) uu[v] = tile[v * NC + IDX(i, j)];
    atomic_h<NEQ>(p, dts, uu);
    put(c, i, j, uu);
  }
  if (tid == 0) {
    if (n) atomicAdd(&M->fallbacks, (unsigned long long)n);
    atomicAdd(&M->cells, 320ull);
  }
}

// Waves per SIMD the plain one-entry-per-workgroup fill is compiled for: 5
// caps it at 96 VGPRs (nothing spilled on its hot path), which measured
// faster than 4 waves at 109 VGPRs (16.8 vs 17.8 ns per block on the
// 16-variant cooling jet; 6 waves spill).  The persistent form carries the
// next record as well and keeps 1024 / BS.
constexpr int kFillWaves = 5;

template <int NEQ, bool SUR, int BS, bool PERSIST>
__global__ __launch_bounds__(BS, (SUR ? (PERSIST ? 2 : 1024 / BS) : (PERSIST ? 1024 / BS : kFillWaves))) void k_fillI_cool(const wx_params *__restrict__ P, QueueRef q,
                                                    const int2 *__restrict__ ops,
                                                    const BlockRec *__restrict__ binfo,
                                                    const double *__restrict__ Uin,
                                                    double *__restrict__ Uout,
                                                    double *__restrict__ stat,
                                                    int8_t *__restrict__ flag,
                                                    DevScalars *__restrict__ Sa,
                                                    FlagOut fo,
                                                    SurDev *__restrict__ M,
                                                    double *__restrict__ Pc) {
  __shared__ double tile[NEQ * NC];
  const int b0 = PERSIST ? (int)blockIdx.x : xcd_entry(blockIdx.x, gridDim.x);
  LeafRec Lnext = q.rec[min(b0, q.cap - 1)];
  const int nleaf = q.hdr->nleaf;
  // the scalars are final for the step (dt reduction and stages A and B
  // are done; this kernel does not write them)
  if (fo.flagq && blockIdx.x == 0)
    for (int t = threadIdx.x; t < fo.ninst; t += blockDim.x) fo.Sout[t] = Sa[t];
  for (int l = b0; l < nleaf; l += gridDim.x) {
  const int r = l;
  const LeafRec L = Lnext;
  if (PERSIST && l + (int)gridDim.x < nleaf) Lnext = q.rec[l + gridDim.x];
  const wx_params *__restrict__ p = P + L.inst;
  DevScalars *__restrict__ S = Sa + L.inst;
  const int b = L.id, level = L.level, icx = L.icx, icy = L.icy, inst = L.inst, lidx = L.lidx;
  const int tid = threadIdx.x;
  const double time = S->time;
  const bool imp = (L.flags & 1) != 0;
  const double vjet = p->otherb ? jet_velocity_at(p, S, time) : 0.0;
  const double *ib = Uin + (size_t)b * NEQ * NC;
  double *ob = Uout + (size_t)b * NEQ * NC;
  // interior U^{n+1}; imposed where listed
  for (int c = tid; c < 256; c += blockDim.x) {
    const int i = c % 16 + 1, j = c / 16 + 1;
    double uu[NEQ];
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = ib[k * NC + c];
    if (imp && in_jet(p, level, icx, icy, i, j)) jet_state<NEQ>(p, vjet, uu);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) tile[k * NC + IDX(i, j)] = uu[k];
  }
  // ghost layer 1 (64 cells) from the list; a cell no entry writes keeps the
  // U^{n+1/2} ring that stage B left in this tile's ring of Uout, imposed
  // where listed.  Ghost g is gathered by the thread that cools it below:
  // thread g with 256 threads, thread 256 + g with more.
  const int gt = BS > 256 ? tid - 256 : tid;
  if (gt >= 0 && gt < 64) {
    const int side = gt >> 4, pos = (gt & 15) + 1;
    const int2 op = ops[r * 8 + side * 2 + ((pos - 1) >> 3)];
    int gi, gj;
    ghost_coords(side, 1, pos, gi, gj);
    double g[NEQ];
    if ((op.y & 15) != GK_NONE) {
      ghost_gather<NEQ>(p, Uin, binfo, op, b, level, icx, icy, side, 1, pos, vjet, g);
    } else {
#pragma unroll
      for (int k = 0; k < NEQ; ++k) g[k] = ob[k * NC + 256 + gt];
      if (imp && in_jet(p, level, icx, icy, gi, gj)) jet_state<NEQ>(p, vjet, g);
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k) tile[k * NC + IDX(gi, gj)] = g[k];
  }
  // ghost layer 2 keeps stage B's U^{n+1/2} ring (already in Uout); the
  // source is imposed on its cells where listed (before the cooling, which
  // writes other cells, so that the source speed is not held across it)
  if (imp)
    for (int g = tid; g < 64; g += blockDim.x) {
      int gi, gj;
      ghost_coords(g >> 4, 2, (g & 15) + 1, gi, gj);
      if (in_jet(p, level, icx, icy, gi, gj)) {
        double v[NEQ];
        jet_state<NEQ>(p, vjet, v);
#pragma unroll
        for (int k = 0; k < NEQ; ++k) ob[k * NC + 320 + g] = v[k];
      }
    }
  // cooling over cells 0..n+1 (src/coolingh.f90:19-20, src/coolingdmc.f90:23-24)
  // except the four corner cells, which nothing reads: the interior (cell
  // c < 256) and the non-corner ghosts of layer 1 (c = 256 + the gather's
  // index).  Every cell is cooled by the thread that loaded it, so no wave
  // waits for another's loads.
  // Each cooled cell goes to Uout, and its primitives to the LDS tile for
  // the epilogue's 5-point stencils.
  const int mode = p->cooling;
  bool done = false;
  if constexpr (SUR && NEQ >= 5) {
    if (mode == 1) {
      cool_surrogate<NEQ, BS>(p, M, S->dt * p->tsc, tile, ob);
      done = true;
    }
  }
  const double dts = S->dt * p->tsc;
  // the short divisions (wx_physics.h) pay where coolingh runs; without n_HI
  // they gained nothing (DMC ensemble 44.7 against 45.1 us, 16 blocks of the
  // adiabatic explosion 5.8 against 6.1)
  constexpr bool SHORT = NEQ >= 5;
  const bool pok = SHORT && mild_params(p, level);
  RecipP rp{};
  if constexpr (SHORT) rp = recip_params(p);
  double *pcb = Pc ? Pc + (size_t)b * NC : nullptr;
  // cell c of this thread: cooled state to Uout, its primitives to the tile
  // (under DMC with the cooled pressure, carried into the next step,
  // src/coolingdmc.f90:27-38; the primitives' velocities serve the epilogue's
  // signal speeds only).  cool returns false, the cell unchanged, where its
  // short form does not hold; those cells take the general one afterwards.
  // Neither pass is a loop: the compiler moves the constants of the loop's
  // exponentials and powers out of it, more than the registers hold (115
  // scalar-register spills and scratch traffic in every wave).
  auto cool_pass = [&](auto cool, auto cool_any) __attribute__((always_inline)) {
    auto put = [&](int c, int i, int j, const double *uu, double pcool) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < NEQ; ++k) ob[k * NC + c] = uu[k];
      double q[NEQ], T;
      if constexpr (SHORT) uprim_any<NEQ>(p, rp, pok, 0.0, q, uu, T);
      else uprim<NEQ>(p, q, uu, T);
      if (mode == 2) {
        q[3] = pcool;
        if (pcb) pcb[c] = pcool;
      }
#pragma unroll
      for (int k = 0; k < NEQ; ++k) tile[k * NC + IDX(i, j)] = q[k];
    };
    uint32_t left = 0;   // bit n: cell tid + n * BS
#pragma unroll
    for (int n = 0; n < (320 + BS - 1) / BS; ++n) {
      const int c = tid + n * BS;
      if (c >= 320) break;
      int i, j;
      tile_ij(c, i, j);
      double uu[NEQ], pcool = 0.0;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) uu[k] = tile[k * NC + IDX(i, j)];
      if (cool(uu, pcool)) put(c, i, j, uu, pcool);
      else left |= 1u << n;
    }
    if (!WX_RARE(__any(left != 0))) return;
#pragma unroll
    for (int n = 0; n < (320 + BS - 1) / BS; ++n) {
      const int c = tid + n * BS;
      if (!(left >> n & 1)) continue;
      int i, j;
      tile_ij(c, i, j);
      double uu[NEQ], pcool = 0.0;
#pragma unroll
      for (int k = 0; k < NEQ; ++k) uu[k] = tile[k * NC + IDX(i, j)];
      cool_any(uu, pcool);
      put(c, i, j, uu, pcool);
    }
  };
  if (!done && mode == 1) {
    cool_pass(
        [&](double *uu, double &) {
          if constexpr (NEQ >= 5) {
            double q[NEQ], T;
            const bool ok = uprim_mild<NEQ>(p, rp, 0.0, q, uu, T) & pok & (uu[0] >= 1e-15);
            return ok && atomic_mild<NEQ>(p, rp, dts, q, T, uu);
          }
          return true;
        },
        [&](double *uu, double &) { atomic_h<NEQ>(p, dts, uu); });
  } else if (!done && mode == 2) {
    cool_pass(
        [&](double *uu, double &pcool) {
          double q[NEQ], T;
          if constexpr (SHORT) {
            if (!(uprim_mild<NEQ>(p, rp, 0.0, q, uu, T) & pok)) return false;
          } else {
            uprim<NEQ>(p, q, uu, T);
          }
          cool_dmc<NEQ>(p, dts, q, T, uu, pcool);
          return true;
        },
        [&](double *uu, double &pcool) {
          double q[NEQ], T;
          uprim<NEQ>(p, q, uu, T);
          cool_dmc<NEQ>(p, dts, q, T, uu, pcool);
        });
  } else if (!done) {
    cool_pass([](double *, double &) { return true; }, [](double *, double &) {});
  }
  __syncthreads();
  block_stats<NEQ, BS>(p, pok, tile, b, level, stat, flag, fo.flagq ? fo.flagq + fo.inst_off[inst] + lidx : nullptr);
  __syncthreads();   // the next queue entry reuses the LDS tile
   if (!PERSIST) break;   // one entry per workgroup: no loop
  }
}

// Statistics only (after upload or a mesh change).
template <int NEQ>
// Under DMC (Pc != nullptr, the instance cooling with DMC) the pressure is
// the carried one, or (pc_init 1, or 2 and the record's pad bit 0) the
// block's state came from outside and the carried pressure starts as the
// one u gives (the reference's calcprim after basegrid or a warm start).
__global__ __launch_bounds__(256) void k_blockstat(const wx_params *__restrict__ P,
                                                   const LeafRec *__restrict__ leaves,
                                                   const double *__restrict__ U,
                                                   double *__restrict__ stat,
                                                   int8_t *__restrict__ flag,
                                                   double *__restrict__ Pc, int pc_init) {
  __shared__ double tile[NEQ * NC];
  const int l = blockIdx.x;
  const LeafRec L = leaves[l];
  const wx_params *__restrict__ p = P + L.inst;
  const double *ub = U + (size_t)L.id * NEQ * NC;
  const bool carried = Pc && p->cooling == 2;
  const bool init = pc_init == 1 || (pc_init == 2 && (L.pad & 1));
  double *pcb = carried ? Pc + (size_t)L.id * NC : nullptr;
  for (int c = threadIdx.x; c < 18 * 18; c += blockDim.x) {
    const int i = c % 18, j = c / 18;
    double uu[NEQ], q[NEQ], T;
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = ub[k * NC + tile_cell(i, j)];
    uprim<NEQ>(p, q, uu, T);
    if (carried) {
      if (init) pcb[tile_cell(i, j)] = q[3];
      else q[3] = pcb[tile_cell(i, j)];
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k) tile[k * NC + IDX(i, j)] = q[k];
  }
  __syncthreads();
  block_stats<NEQ>(p, mild_params(p, L.level), tile, L.id, L.level, stat, flag, nullptr);
}

// dt = min(cfl*dtp, 0.4*dtcool*Psc/tsc) (src/timestep.f90:50); optionally
// time += dt (src/main.f90:88).  Workgroup i reduces instance i's records.
__global__ __launch_bounds__(1024) void k_dtreduce(const wx_params *__restrict__ P,
                                                   const LeafRec *__restrict__ rec,
                                                   const double *__restrict__ stat,
                                                   const int32_t *__restrict__ inst_off,
                                                   DevScalars *__restrict__ Sa, int advance) {
  __shared__ double r0[16], r1[16];
  const int inst = blockIdx.x;
  const wx_params *__restrict__ p = P + inst;
  DevScalars *__restrict__ S = Sa + inst;
  const int n = inst_off[inst + 1] - inst_off[inst];
  const LeafRec *__restrict__ mine = rec + inst_off[inst];
  // what the last thread needs is read with the first loads of the chain
  // inst_off -> rec -> stat, not after it
  const double cfl = p->cfl, Psc = p->Psc, tsc = p->tsc, time = S->time;
  const bool jet = p->otherb != 0;
  double a = 1.e30, c = 1e30;
  // four records a round: a record's ID and then its partials are two trips to
  // memory, and one workgroup makes them all (5 319 leaves: 9.5 us one record
  // at a time, 7.9 now)
  for (int k = threadIdx.x; k < n; k += 4 * blockDim.x) {
    int id[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) id[u] = mine[min(k + u * (int)blockDim.x, n - 1)].id;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      // no record twice: a minimum with a NaN takes its other operand or not by
      // their order
      const double sa = stat[2 * id[u]], sc = stat[2 * id[u] + 1];
      const bool in = k + u * (int)blockDim.x < n;
      a = in ? dmin(a, sa) : a;
      c = in ? dmin(c, sc) : c;
    }
  }
  for (int o = 32; o > 0; o >>= 1) {
    a = dmin(a, __shfl_xor(a, o));
    c = dmin(c, __shfl_xor(c, o));
  }
  if ((threadIdx.x & 63) == 0) { r0[threadIdx.x >> 6] = a; r1[threadIdx.x >> 6] = c; }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int nw = (blockDim.x + 63) >> 6;
    for (int k = 1; k < nw; ++k) { a = dmin(a, r0[k]); c = dmin(c, r1[k]); }
    S->dtp_min = a;
    S->dtcool_min = c;
    double dt = dmin(cfl * a, 0.4 * c * Psc / tsc);
    S->dt = dt;
    const double t = advance ? time + dt : time;
    if (advance) S->time = t;
    if (jet) {   // the jet source speed of the step, once instead of per wave of the stages
      S->vjet = jet_velocity(p, t);
      S->vjet_time = t;
      S->vjet_ok = 1;
    }
  }
}

// Compacted queue entry l = record leafbase[i] + l - inst_off[i] of the
// per-instance regions, i the instance with inst_off[i] <= l < inst_off[i+1]
// (binary search); copies the record and its 8 + 8 ghost ops.
__global__ __launch_bounds__(256) void k_build_queue(const QueueHdr *__restrict__ hdr,
                                                     const int32_t *__restrict__ inst_off,
                                                     const int32_t *__restrict__ leafbase,
                                                     const int32_t *__restrict__ slotbase,
                                                     const int32_t *__restrict__ reg_ids,
                                                     const BlockRec *__restrict__ binfo,
                                                     const int32_t *__restrict__ slot_flag,
                                                     const int2 *__restrict__ slot_ops2,
                                                     const int2 *__restrict__ slot_ops1,
                                                     LeafRec *__restrict__ rec, int2 *__restrict__ ops2,
                                                     int2 *__restrict__ ops1) {
  const int n = hdr->nleaf, ni = hdr->ninst;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 8 * n; t += gridDim.x * blockDim.x) {
    const int l = t >> 3, k = t & 7;
    int lo = 0, hi = ni - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (inst_off[mid] <= l) lo = mid;
      else hi = mid - 1;
    }
    const int lp = l - inst_off[lo];
    const size_t slot = (size_t)slotbase[lo] + (size_t)reg_ids[(size_t)leafbase[lo] + lp];
    if (k == 0) {
      const BlockRec b = binfo[slot];
      rec[l] = LeafRec{(int32_t)slot, b.level, b.icx, b.icy, slot_flag[slot], lp, lo, 0};
    }
    ops2[(size_t)l * 8 + k] = slot_ops2[slot * 8 + k];
    if (ops1) ops1[(size_t)l * 8 + k] = slot_ops1[slot * 8 + k];
  }
}

// The changed per-slot ops (and, with flag != nullptr, leaf flags) of an
// upload, read in place from the pinned staging.
__global__ __launch_bounds__(256) void k_slot_scatter(const SlotOps *__restrict__ src, int n,
                                                      int2 *__restrict__ ops, int32_t *__restrict__ flag) {
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < 8 * n; t += gridDim.x * blockDim.x) {
    const int r = t >> 3, k = t & 7;
    const size_t slot = (size_t)src[r].slot;
    ops[slot * 8 + k] = src[r].ops[k];
    if (flag && k == 0) flag[slot] = src[r].flag;
  }
}

// Refinement flags in queue order for the host's admesh, and the instances'
// scalars; both outputs may be pinned host memory (mapped), so that the host
// reads them after the stream synchronises with no copy launched.
__global__ __launch_bounds__(256) void k_gather_flags(QueueRef q, const int32_t *__restrict__ inst_off,
                                                      const int8_t *__restrict__ flag,
                                                      int8_t *__restrict__ flagq, const DevScalars *__restrict__ S,
                                                      DevScalars *__restrict__ Sout, int ninst) {
  const int n = q.hdr->nleaf;
  for (int l = blockIdx.x * blockDim.x + threadIdx.x; l < n; l += gridDim.x * blockDim.x) {
    const LeafRec r = q.rec[l];
    flagq[inst_off[r.inst] + r.lidx] = flag[r.id];   // by leaf position, whatever the queue order
  }
  if (Sout && blockIdx.x == 0)
    for (int i = threadIdx.x; i < ninst; i += blockDim.x) Sout[i] = S[i];
}

// ---------------------------------------------------------------------
// admesh data ops: src/refine.f90:30-42 (injection over the padded block)
// and src/coarse.f90:182-366 (MPIP branch: 2x2 means incl. ghosts, then
// outer ghost copies), and the statistics of the new leaf.  One workgroup per
// new leaf, one thread per cell of its padded tile: a mesh change has a few
// ops, so the launch is a chain of latencies (the op from host memory, the
// source cells, the tile) and takes each once; with 256 threads, the copies
// and the statistics reading the source separately and the outer ghosts
// copied by one thread per variable it took 10.6 us against 7.5 for the few
// ops of a step of the 64x16-root jet.
template <int NEQ>
__global__ __launch_bounds__(512) void k_meshops(const wx_params *__restrict__ P, const MeshOp *__restrict__ ops,
                                                 double *__restrict__ U, double *__restrict__ stat,
                                                 int8_t *__restrict__ flag, double *__restrict__ Pc) {
  // workgroup 4 * o + s: son s of a refine op o; a coarse op's dad is done
  // by its first workgroup
  const MeshOp op = ops[blockIdx.x >> 2];
  const int s = blockIdx.x & 3;
  const bool refine = op.kind == 0;
  if (!refine && s != 0) return;
  const int son = s == 0 ? op.s1 : s == 1 ? op.s2 : s == 2 ? op.s3 : op.s4;
  const int dst = refine ? son : op.a;
  const wx_params *__restrict__ p = P + op.inst;
  double *pcb = (Pc && p->cooling == 2) ? Pc + (size_t)dst * NC : nullptr;
  __shared__ double d[NEQ * NC];   // the new leaf's primitives, for its statistics
  const int tid = threadIdx.x;
  if (tid < NC) {
    const int i = tid % NP - 1, j = tid / NP - 1;
    double uu[NEQ];
    if (refine) {
      const double *pb = U + (size_t)op.a * NEQ * NC +
                         tile_cell((i + 1) / 2 + ((s & 1) ? NX / 2 : 0), (j + 1) / 2 + ((s & 2) ? NY / 2 : 0));
#pragma unroll
      for (int k = 0; k < NEQ; ++k) uu[k] = pb[k * NC];
    } else {
      // dad cells 0..17 from the four sons (son covers half of either
      // direction); the outermost cells take their neighbour's value: the
      // copies of src/coarse.f90:349-358, applied in order, leave every one
      // of them with the nearest cell of 0..17
      const int ci = min(max(i, 0), NX + 1), cj = min(max(j, 0), NY + 1);
      const int sx = (ci <= NX / 2) ? 0 : 1, sy = (cj <= NY / 2) ? 0 : 1;
      const int from = sy ? (sx ? op.s4 : op.s3) : (sx ? op.s2 : op.s1);
      const int i1 = 2 * (ci - sx * (NX / 2)) - 1, j1 = 2 * (cj - sy * (NY / 2)) - 1;
      const double *sb = U + (size_t)from * NEQ * NC;
      const int c00 = tile_cell(i1, j1), c10 = tile_cell(i1 + 1, j1), c01 = tile_cell(i1, j1 + 1),
                c11 = tile_cell(i1 + 1, j1 + 1);
#pragma unroll
      for (int k = 0; k < NEQ; ++k)
        uu[k] = 0.25 * (((sb[k * NC + c00] + sb[k * NC + c10]) + sb[k * NC + c01]) + sb[k * NC + c11]);
    }
    double *db = U + (size_t)dst * NEQ * NC + tile_cell(i, j);
#pragma unroll
    for (int k = 0; k < NEQ; ++k) db[k * NC] = uu[k];
    // primitives of cells 0..17; under DMC the carried pressure starts from
    // them (src/refine.f90:231-258, src/coarse.f90:178, 360 recompute primit)
    if ((stat || pcb) && i >= 0 && i <= NX + 1 && j >= 0 && j <= NY + 1) {
      double q[NEQ], T;
      uprim<NEQ>(p, q, uu, T);
      if (pcb) pcb[tile_cell(i, j)] = q[3];
#pragma unroll
      for (int k = 0; k < NEQ; ++k) d[k * NC + IDX(i, j)] = q[k];
    }
  }
  if (!stat) return;
  __syncthreads();
  block_stats<NEQ>(p, mild_params(p, op.level), d, dst, op.level, stat, flag, nullptr);
}

// Layout transposes between the device's tiles and the reference's
// u(nb, ieq, i, j) with nb fastest (ld = number of block rows).
template <int NEQ>
__global__ void k_transpose(int cap, const double *__restrict__ src, double *__restrict__ dst,
                            int to_fortran, int ld) {
  const size_t n = (size_t)cap * NEQ * NC;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    if (to_fortran) {
      // t enumerates the Fortran array: nb fastest
      const size_t nb = t % cap, r = t / cap;
      const size_t k = r % NEQ, cell = r / NEQ;     // cell = (i+1) + 20*(j+1)
      dst[t] = src[((nb + 1) * NEQ + k) * NC + tile_cell((int)(cell % NP) - 1, (int)(cell / NP) - 1)];
    } else {
      const size_t cell = t % NC, r = t / NC;
      const size_t k = r % NEQ, id = r / NEQ;       // id 0..cap-1 -> block id+1
      dst[((id + 1) * NEQ + k) * NC + tile_cell((int)(cell % NP) - 1, (int)(cell / NP) - 1)] =
          src[(cell * NEQ + k) * (size_t)ld + id];
    }
  }
}

// The cells of one tile variable per 128 threads reordered, between padded
// host rows and the device's order; src may be dst.  Both are read and written
// in the order of memory, the tile turned over in LDS.
__global__ __launch_bounds__(256) void k_reorder(size_t ntile, const double *src, double *dst, int to_rows) {
  __shared__ double t[2][NC];
  const int h = threadIdx.x >> 7, l = threadIdx.x & 127;
  const size_t v = (size_t)blockIdx.x * 2 + h;
  if (v < ntile)
    for (int c = l; c < NC; c += 128) {
      const int d = to_rows ? c : tile_cell(c % NP - 1, c / NP - 1);
      t[h][d] = src[v * NC + c];
    }
  __syncthreads();
  if (v < ntile)
    for (int c = l; c < NC; c += 128) {
      const int d = to_rows ? tile_cell(c % NP - 1, c / NP - 1) : c;
      dst[v * NC + c] = t[h][d];
    }
}

template <int NEQ>
__global__ void k_calcprim(const wx_params *__restrict__ p, int cap, const double *__restrict__ U,
                           double *__restrict__ prim) {
  const size_t n = (size_t)(cap + 1) * NC;
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x) {
    const size_t id = t / NC, c = t % NC;
    double uu[NEQ], q[NEQ], T;
#pragma unroll
    for (int k = 0; k < NEQ; ++k) uu[k] = U[(id * NEQ + k) * NC + c];
    if (uu[0] == 0.0 && uu[3] == 0.0) {
#pragma unroll
      for (int k = 0; k < NEQ; ++k) q[k] = 0.0;
    } else {
      uprim<NEQ>(p, q, uu, T);
    }
#pragma unroll
    for (int k = 0; k < NEQ; ++k) prim[(id * NEQ + k) * NC + c] = q[k];
  }
}

// ---------------------------------------------------------------------
// launch wrappers
#define WX_DISPATCH(NEQV, CALL)                  \
  switch (NEQV) {                                \
    case 4: { constexpr int N = 4; CALL; } break; \
    case 5: { constexpr int N = 5; CALL; } break; \
    case 6: { constexpr int N = 6; CALL; } break; \
    default: return WX_EARG;                     \
  }

static inline int hip_status() { return hipGetLastError() == hipSuccess ? WX_OK : WX_EHIP; }

int launch_build_queue(const QueueHdr *hdr, const int32_t *inst_off, const int32_t *leafbase,
                       const int32_t *slotbase, const int32_t *reg_ids, const BlockRec *binfo,
                       const int32_t *slot_flag, const int2 *slot_ops2, const int2 *slot_ops1, LeafRec *rec,
                       int2 *ops2, int2 *ops1, int grid, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  hipLaunchKernelGGL(k_build_queue, dim3(grid), dim3(256), 0, stream, hdr, inst_off, leafbase, slotbase, reg_ids,
                     binfo, slot_flag, slot_ops2, slot_ops1, rec, ops2, ops1);
  return hip_status();
}

int launch_slot_scatter(const SlotOps *src, int n, int2 *ops, int32_t *flag, hipStream_t stream) {
  if (n <= 0) return WX_OK;
  const int grid = min(max(1, (8 * n + 255) / 256), 1024);
  hipLaunchKernelGGL(k_slot_scatter, dim3(grid), dim3(256), 0, stream, src, n, ops, flag);
  return hip_status();
}

// Workgroup sizes the stage kernels are built for (4, 6 or 8 waves), and
// the one-entry-per-workgroup / persistent forms.
#define WX_BS_DISPATCH(BSV, CALL)                    \
  switch (BSV) {                                     \
    case 256: { constexpr int B = 256; CALL; } break; \
    case 384: { constexpr int B = 384; CALL; } break; \
    case 512: { constexpr int B = 512; CALL; } break; \
    default: return WX_EARG;                         \
  }
#define WX_PERSIST_DISPATCH(PV, CALL)                     \
  if (PV) { constexpr bool PS = true; CALL; }             \
  else { constexpr bool PS = false; CALL; }

// Launches from which stages A and B use the short divisions.  They take a
// quarter of the instructions out (stage B 1 167 -> 866 per wave), but a block
// that holds a velocity below the bound (mild_tiny) pays for both forms, and a
// small launch lasts as long as its slowest block.  us per launch, general /
// short: stage A at 1 174 blocks 13.9 / 13.0, at 532 7.8 / 8.2, on 19 250
// 138 / 122; stage B at 520 11.9 / 13.1, at 1 177 19.6 / 20.2, at 5 319
// 58.4 / 54.2, at 19 250 206 / 191.
// Where the run's constants lie outside the short forms' range no block is
// served by them (QueueRef::general): stages A and B of 6 144 blocks took 58 and
// 81 us so, 46 and 65 in the general form.
constexpr int kMildA = 1024, kMildB = 3000;

int launch_stageA(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const double *U,
                  double *Q, const double *Pc, DevScalars *S, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  if (q.stat) {   // with the dt reduction
    if (persist || bs != 512 || grid > 512) return WX_EARG;
    WX_DISPATCH(neq, hipLaunchKernelGGL((k_stageA_dt<N>), dim3(grid), dim3(512), 0, stream, P, q, U, Q, Pc, S));
    return hip_status();
  }
  if (!persist && !q.general && grid >= kMildA) {
    WX_BS_DISPATCH(bs, WX_DISPATCH(neq, hipLaunchKernelGGL((k_stageA_mild<N, B>), dim3(grid), dim3(B), 0, stream, P, q, U, Q, Pc, S)));
    return hip_status();
  }
  WX_PERSIST_DISPATCH(persist, WX_BS_DISPATCH(bs, WX_DISPATCH(neq, hipLaunchKernelGGL((k_stageA<N, B, PS>), dim3(grid), dim3(B), 0, stream, P, q, U, Q, Pc, S))));
  return hip_status();
}

int launch_stageB(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const int2 *ops,
                  const BlockRec *binfo, double *U, double *Q, DevScalars *S, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  if (!persist && !q.general && grid >= kMildB) {
    WX_BS_DISPATCH(bs, WX_DISPATCH(neq, hipLaunchKernelGGL((k_stageB_mild<N, B>), dim3(grid), dim3(B), 0, stream, P, q, ops, binfo, U, Q, Q, S)));
    return hip_status();
  }
  WX_PERSIST_DISPATCH(persist, WX_BS_DISPATCH(bs, WX_DISPATCH(neq, hipLaunchKernelGGL((k_stageB<N, B, PS>), dim3(grid), dim3(B), 0, stream, P, q, ops, binfo, U, Q, Q, S))));
  return hip_status();
}

// Launches of tiles of five variables from which the fill takes two waves per
// block instead of four.  Its 320 cells are five passes of a wave: four waves take
// two rounds, three of them idle in the second (five of eight slots used), two
// take three rounds (five of six), and ten such workgroups fill a compute unit
// to the byte of LDS and at the same five waves per SIMD.  A block takes longer,
// so it needs many rounds of blocks: passes of 5 322 blocks 80.3 -> 81.6 ms, of
// ensembles without n_HI 125.5 -> 127.1, of two groups of 9 600 blocks
// 297.4 -> 293.4.  With six variables a tile is 19.6 KB, eight such workgroups
// fit, and four waves per SIMD: 146 us against 143 on 10 930 blocks.
constexpr int kFill128 = 8192;

int launch_fillI_cool(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const int2 *ops,
                      const BlockRec *binfo, const double *Uin, double *Uout, double *stat, int8_t *flag,
                      DevScalars *S, FlagOut fo, double *Pc, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  if (!persist && bs == 256 && neq == 5 && grid >= kFill128) {
    hipLaunchKernelGGL((k_fillI_cool<5, false, 128, false>), dim3(grid), dim3(128), 0, stream, P, q, ops, binfo, Uin, Uout, stat, flag, S, fo, nullptr, Pc);
    return hip_status();
  }
  WX_PERSIST_DISPATCH(persist, WX_BS_DISPATCH(bs, WX_DISPATCH(neq, hipLaunchKernelGGL((k_fillI_cool<N, false, B, PS>), dim3(grid), dim3(B), 0, stream, P, q, ops, binfo, Uin, Uout, stat, flag, S, fo, nullptr, Pc))));
  return hip_status();
}

int launch_fillI_cool_sur(const wx_params *P, int neq, QueueRef q, int grid, int bs, int persist, const int2 *ops,
                          const BlockRec *binfo, const double *Uin, double *Uout, double *stat, int8_t *flag,
                          DevScalars *S, SurDev *M, FlagOut fo, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  switch (neq) {   // coolingh needs u(5) = n_HI
    case 5: WX_PERSIST_DISPATCH(persist, WX_BS_DISPATCH(bs, hipLaunchKernelGGL((k_fillI_cool<5, true, B, PS>), dim3(grid), dim3(B), 0, stream, P, q, ops, binfo, Uin, Uout, stat, flag, S, fo, M, nullptr))); break;
    case 6: WX_PERSIST_DISPATCH(persist, WX_BS_DISPATCH(bs, hipLaunchKernelGGL((k_fillI_cool<6, true, B, PS>), dim3(grid), dim3(B), 0, stream, P, q, ops, binfo, Uin, Uout, stat, flag, S, fo, M, nullptr))); break;
    default: return WX_EARG;
  }
  return hip_status();
}

int launch_blockstat(const wx_params *P, int neq, const LeafRec *leaves, int nleaf, const double *U,
                     double *stat, int8_t *flag, double *Pc, int pc_init, hipStream_t stream) {
  if (nleaf <= 0) return WX_OK;
  WX_DISPATCH(neq, hipLaunchKernelGGL(k_blockstat<N>, dim3(nleaf), dim3(256), 0, stream, P, leaves, U, stat, flag, Pc,
                                      pc_init));
  return hip_status();
}

int launch_dtreduce(const wx_params *P, const LeafRec *rec, const double *stat, const int32_t *inst_off,
                    int ninst, DevScalars *S, int advance, hipStream_t stream) {
  if (ninst <= 0 || advance == kDtInStageA) return WX_OK;
  hipLaunchKernelGGL(k_dtreduce, dim3(ninst), dim3(1024), 0, stream, P, rec, stat, inst_off, S, advance);
  return hip_status();
}

int launch_gather_flags(QueueRef q, const int32_t *inst_off, int grid, const int8_t *flag, int8_t *flagq,
                        const DevScalars *S,
                        DevScalars *Sout, int ninst, hipStream_t stream) {
  if (grid <= 0) return WX_OK;
  hipLaunchKernelGGL(k_gather_flags, dim3(grid), dim3(256), 0, stream, q, inst_off, flag, flagq, S, Sout, ninst);
  return hip_status();
}

int launch_meshops(const wx_params *P, int neq, const MeshOp *ops, int nops, double *U, double *stat, int8_t *flag,
                   double *Pc, hipStream_t stream) {
  if (nops <= 0) return WX_OK;
  WX_DISPATCH(neq, hipLaunchKernelGGL(k_meshops<N>, dim3(4 * nops), dim3(512), 0, stream, P, ops, U, stat, flag, Pc));
  return hip_status();
}

// Upload copies: workgroups (x, y) copy part x of copy y, in 16-byte words
// when both ends and the size allow, else 4-byte words, else bytes.
__global__ __launch_bounds__(256) void k_h2d(const CopyDesc *__restrict__ d, int base) {
  const CopyDesc c = d[base + blockIdx.y];
  const uint64_t al = (uint64_t)c.dst | (uint64_t)c.src | c.bytes;
  const size_t t0 = (size_t)blockIdx.x * blockDim.x + threadIdx.x, st = (size_t)gridDim.x * blockDim.x;
  if ((al & 15) == 0) {
    const uint4 *s = (const uint4 *)c.src;
    uint4 *o = (uint4 *)c.dst;
    const size_t n = c.bytes / 16;
    for (size_t i = t0; i < n; i += 2 * st) {   // two words in flight: a read crosses the host link
      const uint4 v = s[i], w = s[i + st < n ? i + st : i];
      o[i] = v;
      if (i + st < n) o[i + st] = w;
    }
  } else if ((al & 3) == 0) {
    const uint32_t *s = (const uint32_t *)c.src;
    uint32_t *o = (uint32_t *)c.dst;
    for (size_t i = t0; i < c.bytes / 4; i += st) o[i] = s[i];
  } else {
    const uint8_t *s = (const uint8_t *)c.src;
    uint8_t *o = (uint8_t *)c.dst;
    for (size_t i = t0; i < c.bytes; i += st) o[i] = s[i];
  }
}

int launch_h2d(const CopyDesc *d, int n, hipStream_t stream) {
  for (int base = 0; base < n; base += 65535) {
    const int m = n - base < 65535 ? n - base : 65535;
    hipLaunchKernelGGL(k_h2d, dim3(16, m), dim3(256), 0, stream, d, base);
  }
  return hip_status();
}

int launch_transpose(int neq, int cap, const double *src, double *dst, int mode, int ld, hipStream_t stream) {
  if (mode >= 2) {   // cap tiles, one by one
    const size_t ntile = (size_t)cap * neq;
    if (ntile == 0) return WX_OK;
    hipLaunchKernelGGL(k_reorder, dim3((unsigned)((ntile + 1) / 2)), dim3(256), 0, stream, ntile, src, dst, mode == 3);
    return hip_status();
  }
  WX_DISPATCH(neq, hipLaunchKernelGGL(k_transpose<N>, dim3(1024), dim3(256), 0, stream, cap, src, dst, mode, ld));
  return hip_status();
}

int launch_calcprim(const wx_params *P, int neq, int cap, const double *U, double *prim, hipStream_t stream) {
  WX_DISPATCH(neq, hipLaunchKernelGGL(k_calcprim<N>, dim3(1024), dim3(256), 0, stream, P, cap, U, prim));
  return hip_status();
}

}  // namespace wx
