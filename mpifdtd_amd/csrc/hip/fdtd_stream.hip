// fdtd_stream.hip -- FP64 UPML step, temporally blocked, for gfx950.
//
// One launch advances the whole grid by up to T = K x S steps (K wavefronts of S
// stages each).  A workgroup walks a strip of columns row by row: each lane
// holds C adjacent columns, and a row passes through the stages one after the
// other, stage s working on the row s behind the newest one, so that the rows
// in flight stay in registers (a slot per row, updated in place; the row loop
// is unrolled by the number of slots, so no value moves) and each is read from
// memory once and written once per launch.  The wavefronts of a workgroup hand
// finished rows on through LDS.  Neighbours along a row come from the adjacent
// lane by DPP, neighbours across rows are the other slots: no halo is
// recomputed in the marching direction except where a strip begins, and 2 T of
// a strip's 64 C columns across it.
//
// The interior cells (every UPML coefficient 1) run
//   E += curl(H)/eps + (s_n - s_{n-1}),   H += c0^2 curl(E)
// on the three fields alone; there the reference's auxiliaries follow from the
// fields (J = D = eps (E - s), M = B = mu0 H) and are formed when they are asked
// for (stream_fill_aux).  Strips of the frame run the full recurrences; in their
// cells without UPML the auxiliaries are formed from the fields as a row is
// loaded.  What bounds it: the chain of a row's dependent FP64 operations, LDS
// hand-ons and one barrier per row (counters of MPI TM on 1056 x 1056: a busy compute
// unit's VALU works 47 % of the time, its waves wait 39 % of theirs, HBM traffic
// 3.3 TB/s), at 6.7 us a step on 1056 x 1056 where the two-launch step that reads and
// writes every array took 57 (8-step launches of 53 us, TM).
// Physics per step as in the reference (mpiTM_UPML.c:196-217,
// mpiTE_UPML.c:290-304, fdtdTM_upml.c:54-66, fdtdTE_upml.c:168-192).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "fdtd_hip.h"
#include "fdtd_internal.h"
#include "fdtd_stream_dev.h"

#define HIPCHK(x)                                                                                    \
  do {                                                                                               \
    hipError_t e_ = (x);                                                                             \
    if (e_ != hipSuccess) return fdtd_fail(FDTD_EHIP, "%s failed: %s", #x, hipGetErrorString(e_)); \
  } while (0)

// A strip: core rows [r0, r1) x columns [j0, j1) written; lane 0's first column
// bj, first input row b0, last input row bl (array coordinates, ring included).
struct StreamStrip {
  int j0, j1, bj, r0, r1, b0, bl, kind;
  int smp, s0, s1, pad[5];  // contour sides through the strip (a bit each), rows with their samples
};

struct StreamSide {
  int horiz, fi, lo, n, off, ef, hf, pad;
  double es;
};

struct StreamArgs {
  const D2 *src;  // the nine arrays of the state, `stride` bytes apart
  D2 *dst;
  size_t stride;
  const double *ie0, *ie1;  // 1/eps of the E components, 0 on the ring
  const double *xt;         // [NPXa][8] row coefficients
  const double *yt;         // [6][NPYa] column coefficients
  const D2 *ex, *ey;        // e^{i kx x}, e^{i ky y} (plain: of the pulse's carrier)
  const StreamStrip *strips;
  int ns, NPXa, NPYa, T;
  int xlo, xhi;             // rows without UPML
  double c2, mu0;
  // sources: entry 0 the step before the launch's first, then its steps
  double c[2][STREAM_T + 1][2];  // MPI: c[0] = ray_coef e^{-i w t}; plain: dot e^{i w off} per component
  double po[2][STREAM_T + 1];    // plain: the pulse's offset (gap - (time - t0)) per component
  double ps[STREAM_T + 1][2];    // point source
  int on[2], ps_on, ps_i, ps_j, hasprev;
  double cpc, spc;
  // contour samples [step][3][total] (es E, H, H one cell back), or null
  D2 *csamp;
  int ctot;
  StreamSide side[4];
};

// The kernel's arguments read where they are used: rows with a source, contour
// samples.  Read through the plain argument they are all loaded ahead of the row
// loop, and the scalar registers spill (270 lane reads an iteration).
__device__ __forceinline__ CAS(StreamArgs) rare_args()
{
#ifdef __HIP_DEVICE_COMPILE__
  CAS(StreamArgs) p = (CAS(StreamArgs))__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
#else
  return nullptr;
#endif
}

// values per cell a row hands on: complex and real (1/eps)
__host__ __device__ constexpr int stream_nv(int mode, int pml) { return pml ? (mode == FDTD_MODE_TM ? 7 : 8) : 3; }
__host__ __device__ constexpr int stream_ni(int mode) { return mode == FDTD_MODE_TM ? 1 : 2; }
__host__ __device__ constexpr int stream_cols(int mode, int flav) { return mode == FDTD_MODE_TE && flav == FDTD_FLAVOUR_PLAIN ? 1 : 2; }
__host__ __device__ constexpr int stream_pf(int mode, int flav) { return mode == FDTD_MODE_TM && flav == FDTD_FLAVOUR_MPI ? 2 : 1; }
#define STREAM_IPF 2
// Smallest 1/eps of the blocked steps: where 1/eps is smaller (or zero: a perfect
// conductor), E is the source alone to all but its last bits, and J = D = eps (E - s)
// cannot be formed from it; grids with such a cell step by the kernels that keep J and D.
// At 2^-20 the difference keeps 32 bits.
#define STREAM_IE_MIN 0x1p-20
// LDS of the rows handed on: K - 1 pairs of wavefronts, two rows each
__host__ __device__ constexpr int stream_lds_v(int mode, int pml, int C, int S) { return (STREAM_T / S - 1) * 2 * stream_nv(mode, pml) * C * 64; }
__host__ __device__ constexpr int stream_lds_i(int mode, int C, int S) { return (STREAM_T / S - 1) * 2 * stream_ni(mode) * C * 64; }

// PF: rows fetched ahead of the one that enters the first stage (a row's turn is
// shorter than a load's latency)
template <int MODE, int FLAV, int PML, int C, int S, int PF>
__device__ __forceinline__ void strip_body(const StreamArgs &a, const StreamStrip t, D2 *lv, double *li, D2 *ls)
{
  constexpr bool TM = MODE == FDTD_MODE_TM, MPI = FLAV == FDTD_FLAVOUR_MPI;
  static_assert(S == 2 && STREAM_T / S > 2, "the sampling of the first wavefront's steps");
  constexpr int K = STREAM_T / S, NS = (MPI ? S + 1 : S + 2) + PF;
  // values of a cell.  Interior TM: E Hx Hy, TE: Ex Ey Hz.
  // Frame TM: E J D Mx Bx My By, TE: Ex Ey Bz Mz Jx Dx Jy Dy
  constexpr int NV = stream_nv(MODE, PML), NI = stream_ni(MODE);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int NPX = a.NPXa, NPY = a.NPYa;
  const int col = t.bj + lane * C;
  const double c2 = a.c2, mu0 = a.mu0;
  D2 V[NS][NV][C];
  double I[NS][NI][C];
  // interior MPI rows with a scatterer: the wave's factor e^{i k.r} (1/eps - 1) (the
  // others have no registers left and form it where it is used)
  constexpr bool WK = !PML && MPI;
  D2 W[WK ? NS : 1][NI][C];
  // interior plain rows with a scatterer: the pulse's change in the wavefront's second
  // step, formed with the first's; one row's is wanted while the next row's is formed
  constexpr bool PK = !PML && !MPI;
  static_assert(!PK || (S == 2 && NS % 2 == 0), "two rows' pulses by the slot's parity");
  D2 P1[PK ? 2 : 1][NI][C];
  bool fl[NS];
  // frame: the row's coefficients, scalar registers loaded an iteration ahead
  double X[PML ? NS : 1][8];
  auto src = [&](int f) { return (const D2 *)((const char *)a.src + f * a.stride); };
  auto dst = [&](int f) { return (D2 *)((char *)a.dst + f * a.stride); };
#pragma unroll
  for (int q = 0; q < NS; q++) {
    fl[q] = false;
    if (PML)
#pragma unroll
      for (int x = 0; x < 8; x++) X[q][x] = 0;
#pragma unroll
    for (int c = 0; c < C; c++) {
#pragma unroll
      for (int v = 0; v < NV; v++) V[q][v][c] = d2(0, 0);
#pragma unroll
      for (int v = 0; v < NI; v++) {
        I[q][v][c] = 0;
        if (WK || q == 0) W[q][v][c] = d2(0, 0);
        if (q < (PK ? 2 : 1)) P1[q][v][c] = d2(0, 0);
      }
    }
  }
  // the hand-on rows start as zeros (rows before the strip's first)
  for (int q = threadIdx.x; q < stream_lds_v(MODE, PML, C, S); q += 64 * K) lv[q] = d2(0, 0);
  for (int q = threadIdx.x; q < stream_lds_i(MODE, C, S); q += 64 * K) li[q] = 0;
  __syncthreads();
  // column values
  D2 ey[C];
#pragma unroll
  for (int c = 0; c < C; c++) ey[c] = a.ey[min(col + c, NPY - 1)];
  const bool lin = col < NPY;             // frame: lanes past the grid hold zeros
  // Clamped column of the loads: lanes past the core's halo, which a narrow frame strip has
  // many of, take its last column, or rows whose scatterer only they see would form its
  // wave (80 x 80 with a cylinder in the middle, us per 8 steps: plain TE 76 -> 39, MPI TM
  // 42 -> 29).
  const int lc = min(col, min(NPY - C, t.j1 + STREAM_T - 1));
  double y0 = 1, y1 = 1, y2 = 1, y3 = 1, s2p = 2, s2m = 2;
  bool ypml = false;
  if (PML) {
    y0 = a.yt[lc];
    y1 = a.yt[NPY + lc];
    y2 = a.yt[2 * NPY + lc];
    y3 = a.yt[3 * NPY + lc];
    const double sy = a.yt[4 * NPY + lc];
    s2p = 2.0 + sy;
    s2m = 2.0 - sy;
    ypml = a.yt[5 * NPY + lc] != 0;
  }
  const int ps_row = TM && MPI && a.ps_on ? a.ps_i : -1000000;
  auto rowc = [&](int r) { return min(max(r, 0), NPX - 1); };

  // MPI: the factors of this wavefront's steps (interior: their change)
  double cs[MPI ? S : 1][2];
  if (MPI) {
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
      for (int x = 0; x < 2; x++) cs[s][x] = a.c[0][w * S + s + 1][x] - (PML ? 0.0 : a.c[0][w * S + s][x]);
  }
  // interior MPI: e^{i kx x} of the newest row, loaded an iteration ahead (loaded where a
  // row meets a scatterer, it was a wait for two loads in turn: 1056 x 1056 with a
  // cylinder 59.9 -> 52.2 us per 8 steps, 44 without the cylinder)
  D2 exr = d2(0, 0), exn = d2(0, 0);
  auto ahead = [&](int r) {
    if (!WK) return;
    exr = exn;
    exn = cload2(a.ex + __builtin_amdgcn_readfirstlane(rowc(r)));
  };
  auto wave = [&](int v, int r, int c, double ie) -> D2 {
    if (WK) return mul(ie == 0.0 ? 0.0 : ie - 1.0, cmulp(exr, ey[c]));
    CAS(StreamArgs) R = rare_args();
    const double f = ie == 0.0 || !R->on[v] ? 0.0 : ie - 1.0;
    return mul(f, cmulp(cload2(R->ex + __builtin_amdgcn_readfirstlane(rowc(r))), ey[c]));
  };
  // the pulse on component q at a cell and step entry st: e^{-(d/50)^2}, times the wave's factor and the step's
  auto pulse = [&](CAS(StreamArgs) R, D2 g, int q, int r, int c, int st) -> D2 {
    const double d = (double)r * R->cpc + (double)(col + c) * R->spc + R->po[q][st];
    const double z = d / 50.0;
    return mul(exp(-(z * z)), cmulp(g, d2(R->c[q][st][0], R->c[q][st][1])));
  };
  // both steps' changes of the pulse on the row in slot q: the first's goes to E, the
  // second's to P1.  One block for the pulse at three step entries, so that its argument
  // loads and exponentials are waited for once a row instead of in each stage (531 x 402
  // TE with a cylinder 94.6 -> 66.9 us per 8 steps, 53.1 without the cylinder).
  // The argument's product with 0.02 in place of a quotient by 50 (six of them a row and
  // component) took plain TE on 1056 x 1056 from 120 to 104 us per 8 steps, plain TM from 93
  // to 82; the argument's own rounding, 1e-13 of a distance near 1000, stays the larger.
  auto pulses = [&](int q, int r) {
    CAS(StreamArgs) R = rare_args();
    const D2 x = cload2(R->ex + __builtin_amdgcn_readfirstlane(rowc(r)));
    const double along = (double)r * R->cpc, across = R->spc;
    const int st = w * S;
#pragma unroll
    for (int v = 0; v < NI; v++)
#pragma unroll
      for (int c = 0; c < C; c++) {
        const double ie = I[q][v][c], f = ie == 0.0 || !R->on[v] ? 0.0 : ie - 1.0;
        const D2 g = mul(f, cmulp(x, ey[c]));
        const double d = along + (double)(col + c) * across;
        D2 p[3];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          const double z = (d + R->po[v][st + k]) * 0.02;
          p[k] = mul(exp(-(z * z)), cmulp(g, d2(R->c[v][st + k][0], R->c[v][st + k][1])));
        }
        V[q][v][c] = add(V[q][v][c], sub(p[1], p[0]));
        P1[PK ? q & 1 : 0][v][c] = sub(p[2], p[1]);
      }
  };
  // the source of component v at stage s: its value (frame) or its change since the step before (interior, MPI)
  auto source = [&](int v, int s, int r, int c, D2 g) -> D2 {
    if (MPI) return cmulp(g, d2(cs[s][0], cs[s][1]));
    CAS(StreamArgs) R = rare_args();
    const int st = w * S + s + 1;
    return pulse(R, g, v, r, c, st);
  };
  constexpr int Q0 = TM ? 0 : (MPI ? 1 : 0);  // components with a source: [Q0, NI)

  // a slot whose values are in place: does its row hold a scatterer cell, and the wave's factor there
  auto flag = [&](int q, int r) {
    bool any = false;
#pragma unroll
    for (int v = 0; v < NI; v++)
#pragma unroll
      for (int c = 0; c < C; c++) any = any || (I[q][v][c] != 1.0 && I[q][v][c] != 0.0);
    fl[q] = __ballot(any) != 0;
    if (WK && RARE(fl[q])) {
#pragma unroll
      for (int v = Q0; v < NI; v++)
#pragma unroll
        for (int c = 0; c < C; c++) W[WK ? q : 0][v][c] = wave(v, r, c, I[q][v][c]);
    }
  };
  auto table = [&](int q, int r0) {
    if (!PML) return;
    const double *x = a.xt + (size_t)__builtin_amdgcn_readfirstlane(rowc(r0)) * 8;
#pragma unroll
    for (int v = 0; v < 8; v++) X[PML ? q : 0][v] = cload(x + v);
  };
  auto load = [&](int q, int r0) {
    const int r = min(rowc(r0), t.bl);
    const unsigned k = (unsigned)(r * NPY + lc);
#pragma unroll
    for (int c = 0; c < C; c++) {
      I[q][0][c] = a.ie0[k + c];
      if (!TM) I[q][1][c] = a.ie1[k + c];
    }
    if (!PML) {
#pragma unroll
      for (int v = 0; v < 3; v++)
#pragma unroll
        for (int c = 0; c < C; c++) V[q][v][c] = src(3 * v)[k + c];
    } else {
      const bool p = ypml || (r < a.xlo || r >= a.xhi);
      if (TM) {
        V[q][0][0] = src(0)[k];
        V[q][1][0] = (p ? src(1) : src(0))[k];
        V[q][2][0] = (p ? src(2) : src(0))[k];
        V[q][3][0] = (p ? src(4) : src(3))[k];
        V[q][4][0] = (p ? src(5) : src(3))[k];
        V[q][5][0] = (p ? src(7) : src(6))[k];
        V[q][6][0] = (p ? src(8) : src(6))[k];
      } else {
        V[q][0][0] = src(0)[k];
        V[q][1][0] = src(3)[k];
        V[q][2][0] = (p ? src(8) : src(6))[k];
        V[q][3][0] = (p ? src(7) : src(6))[k];
        V[q][4][0] = (p ? src(1) : src(0))[k];
        V[q][5][0] = (p ? src(2) : src(0))[k];
        V[q][6][0] = (p ? src(4) : src(3))[k];
        V[q][7][0] = (p ? src(5) : src(3))[k];
      }
    }
  };
  // what a loaded row still needs before its first stage (after the wait for its loads)
  auto settle = [&](int q, int r0) {
    const int r = min(rowc(r0), t.bl);
    flag(q, r);
    if (PML) {
      const bool p = ypml || X[PML ? q : 0][7] != 0;
      // M = B = mu0 H where the cell keeps no auxiliaries
      const double f = p ? 1.0 : mu0;
      if (TM) {
#pragma unroll
        for (int v = 3; v < 7; v++) V[q][v][0] = mul(f, V[q][v][0]);
      } else {
        V[q][2][0] = mul(f, V[q][2][0]);
        V[q][3][0] = mul(f, V[q][3][0]);
      }
      // J = D = eps (E - s) there, s the source of the step before
      const bool ps = TM && MPI && r == ps_row;
      if (RARE(fl[q] || ps)) {
        CAS(StreamArgs) R = rare_args();
#pragma unroll
        for (int v = 0; v < NI; v++) {
          const double ie = I[q][v][0];
          D2 d = V[q][v][0];
          if (v >= Q0 && R->hasprev) {
            const D2 g = wave(v, r, 0, ie);
            d = sub(d, MPI ? cmulp(g, d2(R->c[0][0][0], R->c[0][0][1])) : pulse(R, g, v, r, 0, 0));
          }
          if (ps && col == R->ps_j) d = sub(d, d2(R->ps[0][0], R->ps[0][1]));
          const double e = ie == 0.0 ? 0.0 : 1.0 / ie;
          d = mul(e, d);
          const int vj = TM ? 1 : 4 + 2 * v;
          if (!p) V[q][vj][0] = V[q][vj + 1][0] = d;
        }
      }
      if (!lin) {
#pragma unroll
        for (int v = 0; v < NV; v++) V[q][v][0] = d2(0, 0);
#pragma unroll
        for (int v = 0; v < NI; v++) I[q][v][0] = 0;
      }
    }
  };

  // E half of the row in slot q (row r) at stage s, the H of the row before it in slot qb
  auto ehalf = [&](int q, int qb, int r, int s) {
    const int st = w * S + s + 1;
    if (!PML) {
      if (TM) {
#pragma unroll
        for (int c = 0; c < C; c++) {
          const D2 hl = c ? V[q][1][c - 1] : below(V[q][1][C - 1]);
          const D2 curl = sub(sub(V[q][2][c], V[qb][2][c]), sub(V[q][1][c], hl));
          V[q][0][c] = mad(I[q][0][c], curl, V[q][0][c]);
        }
      } else {
#pragma unroll
        for (int c = 0; c < C; c++) {
          const D2 hl = c ? V[q][2][c - 1] : below(V[q][2][C - 1]);
          V[q][0][c] = mad(I[q][0][c], sub(V[q][2][c], hl), V[q][0][c]);
          V[q][1][c] = mad(I[q][1][c], sub(V[qb][2][c], V[q][2][c]), V[q][1][c]);
        }
      }
      if (RARE(fl[q])) {
        if (PK) {
          if (s == 0) {
            pulses(q, r);
          } else {
#pragma unroll
            for (int v = 0; v < NI; v++)
#pragma unroll
              for (int c = 0; c < C; c++) V[q][v][c] = add(V[q][v][c], P1[PK ? q & 1 : 0][v][c]);
          }
        } else {
#pragma unroll
          for (int v = Q0; v < NI; v++)
#pragma unroll
            for (int c = 0; c < C; c++) V[q][v][c] = add(V[q][v][c], source(v, s, r, c, WK ? W[WK ? q : 0][v][c] : wave(v, r, c, I[q][v][c])));
        }
      }
      if (TM && MPI && RARE(r == ps_row)) {
        CAS(StreamArgs) R = rare_args();
#pragma unroll
        for (int c = 0; c < C; c++)
          if (col + c == R->ps_j) V[q][0][c] = add(V[q][0][c], d2(R->ps[st][0] - R->ps[st - 1][0], R->ps[st][1] - R->ps[st - 1][1]));
      }
    } else {
      if (TM) {
        const D2 cr = sub(sub(V[q][6][0], V[qb][6][0]), sub(V[q][4][0], below(V[q][4][0])));
        const D2 nj = mad(X[PML ? q : 0][0], V[q][1][0], mul(X[PML ? q : 0][1], cr));
        V[q][2][0] = mad(y0, V[q][2][0], mul(y1, sub(nj, V[q][1][0])));
        V[q][1][0] = nj;
        V[q][0][0] = mul(I[q][0][0], V[q][2][0]);
      } else {
        const D2 njx = mad(y0, V[q][4][0], mul(y1, sub(V[q][2][0], below(V[q][2][0]))));
        V[q][5][0] = add(V[q][5][0], sub(mul(X[PML ? q : 0][0], njx), mul(X[PML ? q : 0][1], V[q][4][0])));
        V[q][4][0] = njx;
        const D2 njy = mad(c2, sub(V[qb][2][0], V[q][2][0]), V[q][6][0]);
        const double rs = X[PML ? q : 0][5];
        V[q][7][0] = mad(X[PML ? q : 0][2], V[q][7][0], sub(mul(s2p * rs, njy), mul(s2m * rs, V[q][6][0])));
        V[q][6][0] = njy;
        V[q][0][0] = mul(I[q][0][0], V[q][5][0]);
        V[q][1][0] = mul(I[q][1][0], V[q][7][0]);
      }
      if (RARE(fl[q])) {
#pragma unroll
        for (int v = Q0; v < NI; v++) V[q][v][0] = add(V[q][v][0], source(v, s, r, 0, wave(v, r, 0, I[q][v][0])));
      }
      if (TM && MPI && RARE(r == ps_row)) {
        CAS(StreamArgs) R = rare_args();
        if (col == R->ps_j) V[q][0][0] = add(V[q][0][0], d2(R->ps[st][0], R->ps[st][1]));
      }
    }
  };
  // TM: Hx of the row in slot q
  auto hxhalf = [&](int q, int r) {
    if (!PML) {
#pragma unroll
      for (int c = 0; c < C; c++) {
        const D2 er = c < C - 1 ? V[q][0][c + 1] : above(V[q][0][0]);
        V[q][1][c] = mad(-c2, sub(er, V[q][0][c]), V[q][1][c]);
      }
    } else {
      const D2 dE = sub(above(V[q][0][0]), V[q][0][0]);
      const D2 nm = sub(mul(y2, V[q][3][0]), mul(y3, dE));
      V[q][4][0] = add(V[q][4][0], sub(mul(X[PML ? q : 0][2], nm), mul(X[PML ? q : 0][3], V[q][3][0])));
      V[q][3][0] = nm;
    }
  };
  // TM: Hy of the row in slot qb (row r), TE: Hz; the next row's E in slot q
  auto hrow = [&](int q, int qb, int r) {
    if (!PML) {
      if (TM) {
#pragma unroll
        for (int c = 0; c < C; c++) V[qb][2][c] = mad(c2, sub(V[q][0][c], V[qb][0][c]), V[qb][2][c]);
      } else {
#pragma unroll
        for (int c = 0; c < C; c++) {
          const D2 er = c < C - 1 ? V[qb][0][c + 1] : above(V[qb][0][0]);
          const D2 ce = sub(sub(V[q][1][c], V[qb][1][c]), sub(er, V[qb][0][c]));
          V[qb][2][c] = mad(-c2, ce, V[qb][2][c]);
        }
      }
    } else {
      if (TM) {
        const D2 nm = mad(X[PML ? qb : 0][6], sub(V[q][0][0], V[qb][0][0]), V[qb][5][0]);
        const double rs = X[PML ? qb : 0][5];
        V[qb][6][0] = mad(X[PML ? qb : 0][4], V[qb][6][0], sub(mul(s2p * rs, nm), mul(s2m * rs, V[qb][5][0])));
        V[qb][5][0] = nm;
      } else {
        const D2 ce = sub(sub(V[q][1][0], V[qb][1][0]), sub(above(V[qb][0][0]), V[qb][0][0]));
        const D2 nm = sub(mul(X[PML ? qb : 0][3], V[qb][3][0]), mul(X[PML ? qb : 0][4], ce));
        V[qb][2][0] = mad(y2, V[qb][2][0], mul(y3, sub(nm, V[qb][3][0])));
        V[qb][3][0] = nm;
      }
    }
  };
  // the H values of a cell as fields (TM v 1 Hx, 2 Hy; TE 2 Hz)
  auto hval = [&](int q, int v, int c) -> D2 {
    if (!PML) return V[q][v][c];
    return mul(c2, V[q][TM ? (v == 1 ? 4 : 6) : 2][0]);
  };
  // Contour samples of row r after step entry st, its values from val(v, c): TM E Hx Hy,
  // TE Ex Ey Hz.  The first wavefront stores none itself: it waits for its loads, and a
  // store among them would be waited for as well (rows of 2.1 us instead of 0.8).  It
  // leaves the row of its first step in ls for the second wavefront, and every wavefront
  // samples its predecessor's last step from the row it takes.
  auto sample = [&](int r, int st, auto val) {
    CAS(StreamArgs) R = rare_args();
    const int tot = R->ctot;
    D2 *base = R->csamp + (size_t)(st - 1) * 3 * tot;
#pragma unroll 1
    for (int m = t.smp; m; m &= m - 1) {
      const CAS_(StreamSide) &g = R->side[__builtin_ctz(m)];
      const int lo = g.lo, fi = g.fi, off = g.off;
      if (g.horiz ? r < lo || r >= lo + g.n : r != fi && r != fi - 1) continue;
#pragma unroll
      for (int c = 0; c < C; c++) {
        const int j = col + c;
        if (j < t.j0 || j >= t.j1) continue;
        const int x = g.horiz ? j : r, y = g.horiz ? r : j;  // across, along the side
        if (y < lo || y >= lo + g.n) continue;
        const D2 h = TM && g.hf == 1 ? val(1, c) : val(2, c);
        const int p = off + (y - lo);
        if (x == fi) {
          base[p] = mul(g.es, TM || !g.ef ? val(0, c) : val(1, c));
          base[tot + p] = h;
        } else if (x == fi - 1) {
          base[2 * tot + p] = h;
        }
      }
    }
  };
  const int s1 = a.csamp ? t.s1 : t.s0;
  auto sampled = [&](int r) { return r >= t.s0 && r < s1; };
  // values of the row in slot q as sample takes them
  auto field = [&](int q) {
    return [&, q](int v, int c) -> D2 { return TM ? (v ? hval(q, v, c) : V[q][0][c]) : (v < 2 ? V[q][v][c] : hval(q, 2, c)); };
  };
  auto leave = [&](int q, int p) {
    D2 *o = ls + p * (3 * C * 64) + lane;
    auto val = field(q);
#pragma unroll
    for (int c = 0; c < C; c++)
#pragma unroll
      for (int v = 0; v < 3; v++) o[(v * C + c) * 64] = val(v, c);
  };
  auto left = [&](int p) {
    return [&, p](int v, int c) -> D2 { return ls[p * (3 * C * 64) + (v * C + c) * 64 + lane]; };
  };
  auto store = [&](int q, int r) {
    if (r < t.r0 || r >= t.r1) return;
#pragma unroll
    for (int c = 0; c < C; c++) {
      const int j = col + c;
      if (j < t.j0 || j >= t.j1) continue;
      const unsigned k = (unsigned)(r * NPY + j);
      dst(0)[k] = V[q][0][c];
      dst(3)[k] = TM ? hval(q, 1, c) : V[q][1][c];
      dst(6)[k] = hval(q, 2, c);
      if (PML) {
        const bool p = ypml || X[PML ? q : 0][7] != 0;
        if (p) {
          if (TM) {
            dst(1)[k] = V[q][1][0];
            dst(2)[k] = V[q][2][0];
            dst(4)[k] = V[q][3][0];
            dst(5)[k] = V[q][4][0];
            dst(7)[k] = V[q][5][0];
            dst(8)[k] = V[q][6][0];
          } else {
            dst(1)[k] = V[q][4][0];
            dst(2)[k] = V[q][5][0];
            dst(4)[k] = V[q][6][0];
            dst(5)[k] = V[q][7][0];
            dst(7)[k] = V[q][3][0];
            dst(8)[k] = V[q][2][0];
          }
        }
      }
    }
  };
  // rows handed from wavefront w to w + 1: buffer parity p
  auto put = [&](int q, int p) {
    D2 *o = lv + (2 * w + p) * (NV * C * 64) + lane;
    double *oi = li + (2 * w + p) * (NI * C * 64) + lane;
#pragma unroll
    for (int c = 0; c < C; c++) {
#pragma unroll
      for (int v = 0; v < NV; v++) o[(v * C + c) * 64] = V[q][v][c];
#pragma unroll
      for (int v = 0; v < NI; v++) oi[(v * C + c) * 64] = I[q][v][c];
    }
  };
  auto take = [&](int q, int p) {
    const D2 *o = lv + (2 * (w - 1) + p) * (NV * C * 64) + lane;
    const double *oi = li + (2 * (w - 1) + p) * (NI * C * 64) + lane;
#pragma unroll
    for (int c = 0; c < C; c++) {
#pragma unroll
      for (int v = 0; v < NV; v++) V[q][v][c] = o[(v * C + c) * 64];
#pragma unroll
      for (int v = 0; v < NI; v++) I[q][v][c] = oi[(v * C + c) * 64];
    }
  };

  // Iteration `it`: wavefront w's newest row is b0 + it - w (S + 2) (the row its
  // predecessor finished two iterations before), in slot it mod NS; the next one is
  // fetched meanwhile.  The last core row leaves the last wavefront in iteration nit - 1.
  const int row0 = t.b0 - w * (S + 2);
  const int nit = (t.r1 - t.b0) + S + (K - 1) * (S + 2);
  const int st0 = w * S;
  // A copy of the row loop for the first, the last and the other wavefronts: with
  // the loads, the stores and the LDS reads of a row in one copy, the compiler waits
  // for every outstanding load wherever the branches join.
  auto march = [&](auto FIRST, auto LAST) {
    constexpr bool first = decltype(FIRST)::value, last = decltype(LAST)::value;
    if (first) {
#pragma unroll
      for (int q = 0; q < PF; q++) {
        load(q, t.b0 + q);
        __builtin_amdgcn_sched_barrier(0);  // in the order the loop waits for them
      }
    }
    table(0, row0);
    ahead(row0);
    for (int it0 = 0; it0 < nit; it0 += NS) {
#pragma unroll
      for (int u = 0; u < NS; u++) {
        const int it = it0 + u;
        // (left by return, not skipped: a join with the skipping path would again wait for every load)
        if (RARE(it >= nit)) return;
        const int n = row0 + it;
        ahead(n + 1);
        if (first) settle(u, n);
        else flag(u, n);
        if (first) load((u + PF) % NS, n + PF);
        else {
          take((u + 1) % NS, (it + 1) & 1);
          if (RARE(sampled(n + 1)) && st0 <= a.T) sample(n + 1, st0, field((u + 1) % NS));
          if (w == 1 && RARE(sampled(n + S))) sample(n + S, 1, left((it + 1) & 1));
        }
        table((u + 1) % NS, n + 1);
#pragma unroll
        for (int s = 0; s < S; s++) {
          const int A = (u - s + 2 * NS) % NS, B = (u - s - 1 + 2 * NS) % NS, Z = (u - s - 2 + 2 * NS) % NS;
          const int st = st0 + s + 1, r = n - s;
          if (!RARE(st > a.T)) {
            if (MPI) {
              ehalf(A, B, r, s);
              if (TM) hxhalf(A, r);
              hrow(A, B, r - 1);
            } else {
              if (TM) hxhalf(A, r);
              hrow(A, B, r - 1);
              ehalf(B, Z, r - 1, s);
            }
            if (RARE(sampled(r - 1)) && (last || s < S - 1)) {
              if (first) leave(B, it & 1);
              else sample(r - 1, st, field(B));
            }
          }
        }
        const int O = (u - S + 2 * NS) % NS;
        if (last) store(O, n - S);
        else put(O, it & 1);
        lds_barrier();
      }
    }
  };
  if (w == 0) march(std::true_type(), std::false_type());
  else if (w == K - 1) march(std::false_type(), std::true_type());
  else march(std::false_type(), std::false_type());
}

template <int MODE, int FLAV, int PML, int C, int S, int PF>
__global__ __launch_bounds__(64 * (STREAM_T / S)) __attribute__((amdgpu_waves_per_eu(2))) void k_stream(StreamArgs a)
{
  __shared__ D2 lv[stream_lds_v(MODE, PML, C, S)];
  __shared__ double li[stream_lds_i(MODE, C, S)];
  __shared__ D2 ls[2 * 3 * C * 64];
  // workgroup b runs on XCD b % 8: each XCD takes a contiguous eighth of the strips
  const int per = (a.ns + 7) / 8;
  const int id = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (id >= a.ns) return;
  const StreamStrip t = cload(a.strips + id);
  strip_body<MODE, FLAV, PML, C, S, PF>(a, t, lv, li, ls);
}

// Both kinds of strips in one launch (kind 0 interior, 1 frame): small grids, whose
// two launches would each leave most of the chip idle.
template <int MODE, int FLAV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void k_stream_both(StreamArgs a)
{
  constexpr int C = stream_cols(MODE, FLAV), nv0 = stream_lds_v(MODE, 0, C, 2), nv1 = stream_lds_v(MODE, 1, 1, 2);
  __shared__ D2 lv[nv0 > nv1 ? nv0 : nv1];
  __shared__ double li[stream_lds_i(MODE, C, 2)];
  __shared__ D2 ls[2 * 3 * C * 64];
  const int per = (a.ns + 7) / 8;
  const int id = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (id >= a.ns) return;
  const StreamStrip t = cload(a.strips + id);
  if (t.kind == 0) strip_body<MODE, FLAV, 0, stream_cols(MODE, FLAV), 2, STREAM_IPF>(a, t, lv, li, ls);
  else strip_body<MODE, FLAV, 1, 1, 2, stream_pf(MODE, FLAV)>(a, t, lv, li, ls);
}

// The auxiliaries of the cells without UPML from the fields (the steps do not keep
// them there): J = D = eps (E - s), M = B = mu0 H, s the source of the last step
// (entry 0 of the source arrays).
template <int MODE, int FLAV>
__global__ __launch_bounds__(256) void k_stream_aux(StreamArgs a)
{
  constexpr bool TM = MODE == FDTD_MODE_TM, MPI = FLAV == FDTD_FLAVOUR_MPI;
  const int j = 1 + blockIdx.x * 64 + threadIdx.x, i = 1 + blockIdx.y * 4 + threadIdx.y;
  const int NPY = a.NPYa;
  if (i > a.NPXa - 2 || j > NPY - 2) return;
  if (a.xt[(size_t)i * 8 + 7] != 0 || a.yt[5 * NPY + j] != 0) return;
  const size_t k = (size_t)i * NPY + j;
  auto src = [&](int f) { return (const D2 *)((const char *)a.src + f * a.stride); };
  auto dst = [&](int f) { return (D2 *)((char *)a.dst + f * a.stride); };
  auto dval = [&](int v, double ie, D2 e) -> D2 {
    if (a.on[v] && ie != 1.0 && a.hasprev && (TM || !MPI || v == 1)) {
      D2 g = cmulp(mul(ie - 1.0, cmulp(a.ex[i], a.ey[j])), d2(a.c[MPI ? 0 : v][0][0], a.c[MPI ? 0 : v][0][1]));
      if (!MPI) {
        const double z = ((double)i * a.cpc + (double)j * a.spc + a.po[v][0]) / 50.0;
        g = mul(exp(-(z * z)), g);
      }
      e = sub(e, g);
    }
    if (TM && MPI && a.ps_on && i == a.ps_i && j == a.ps_j) e = sub(e, d2(a.ps[0][0], a.ps[0][1]));
    return d2(e.x / ie, e.y / ie);
  };
  if (TM) {
    dst(1)[k] = dst(2)[k] = dval(0, a.ie0[k], src(0)[k]);
    dst(4)[k] = dst(5)[k] = mul(a.mu0, src(3)[k]);
    dst(7)[k] = dst(8)[k] = mul(a.mu0, src(6)[k]);
  } else {
    dst(1)[k] = dst(2)[k] = dval(0, a.ie0[k], src(0)[k]);
    dst(4)[k] = dst(5)[k] = dval(1, a.ie1[k], src(3)[k]);
    dst(7)[k] = dst(8)[k] = mul(a.mu0, src(6)[k]);
  }
}

// What the host asks of a permittivity map: whether a cell's 1/eps lies outside
// [STREAM_IE_MIN, 1 / STREAM_IE_MIN], NaN included, and the box of the scatterer's cells.
struct StreamMap {
  int odd, i0, i1, j0, j1;  // rows [NPXa - i0, i1), columns [NPYa - j0, j1): all zero without a scatterer
};

// 1/eps, 0 on the ring of cells that are never updated.  A workgroup takes 64 columns of
// STREAM_IE_ROWS rows, so that few wavefronts widen the map's box: with one row each, their
// accesses to it were most of the time (2000 x 1500 with a cylinder 77 -> 23 us).
#define STREAM_IE_ROWS 32
__global__ __launch_bounds__(256) void k_stream_ie(const double *eps, int NPXa, int NPYa, double *ie, StreamMap *m)
{
  const int j = blockIdx.x * 64 + threadIdx.x, r0 = blockIdx.y * STREAM_IE_ROWS + threadIdx.y;
  unsigned long long cols = 0;  // of the scatterer's cells, and their rows
  int lo = INT_MAX, hi = -1;
  bool odd = false;
#pragma unroll
  for (int r = 0; r < STREAM_IE_ROWS; r += 4) {
    const int i = r0 + r;
    const bool in = i < NPXa && j < NPYa, ring = i == 0 || j == 0 || i >= NPXa - 1 || j >= NPYa - 1;
    const size_t k = (size_t)i * NPYa + j;
    const double v = in ? 1.0 / eps[k] : 1.0;
    if (in) ie[k] = ring ? 0.0 : v;
    odd = odd || (!ring && !(fabs(v) >= STREAM_IE_MIN && fabs(v) <= 1.0 / STREAM_IE_MIN));
    const unsigned long long b = __ballot(!ring && v != 1.0);
    cols |= b;
    if (b) {
      lo = min(lo, i);
      hi = i;
    }
  }
  if (odd) m->odd = 1;
  if (!cols || threadIdx.x) return;
  atomicMax(&m->i0, NPXa - lo);
  atomicMax(&m->i1, hi + 1);
  atomicMax(&m->j0, NPYa - (j + __builtin_ctzll(cols)));
  atomicMax(&m->j1, j + 64 - __builtin_clzll(cols));
}

// The ring of cells that no step writes, zero in all nine arrays of a new second state (the
// auxiliaries of its cells without UPML are formed before they are read).
__global__ __launch_bounds__(256) void k_stream_ring(D2 *G, size_t stride, int NPXa, int NPYa)
{
  const int q = blockIdx.x * 256 + threadIdx.x, side = blockIdx.y, n = side < 2 ? NPYa : NPXa;
  if (q >= n) return;
  const size_t k = side < 2 ? (size_t)(side ? NPXa - 1 : 0) * NPYa + q : (size_t)q * NPYa + (side == 3 ? NPYa - 1 : 0);
  for (int f = 0; f < 9; f++) ((D2 *)((char *)G + f * stride))[k] = d2(0, 0);
}

// ---------------------------------------------------------------- host

// most strips of a launch of both kinds: two workgroups on each of the 256 compute units
#define STREAM_BOTH_MAX 512

struct StreamState {
  fdtd_grid_desc d;
  int NPXa, NPYa, off;
  size_t ncell;
  D2 *G;  // the nine arrays a launch writes, swapped with the grid's after it; made by the first launch
  size_t stride;
  double *ie[2];  // in one block
  double *xt, *yt;
  D2 *exy;
  StreamMap *map;  // device, per 1/eps map; in one block with xt, yt and exy
  StreamMap seen;  // of all maps together
  StreamStrip *strips;  // interior, then frame
  int nint, nfrm;
  int xlo, xhi, ylo, yhi;  // the box without UPML
  StreamSide side[4];
  int ctot;
  D2 *csamp;
  // the wave of the last step, and its source terms
  bool wave, coefs;
  double angle, k, omega, time, dot[2];
  int use[2];
  D2 c[2], ps;
  double po[2];
  double cpc, spc;
  long steps;
};

int stream_create(const fdtd_grid_desc &d, int off, const Contour &ct, StreamState **out)
{
  StreamState *s = new StreamState();
  *out = s;
  memset((void *)s, 0, sizeof *s);
  s->d = d;
  s->off = off;
  s->NPXa = d.N_PX + 2 * off;
  s->NPYa = d.N_PY + 2 * off;
  s->ncell = (size_t)s->NPXa * s->NPYa;
  s->stride = stream_stride(s->ncell);
  // a grid without room for these, or past 32-bit cell indexes, steps in place
  if (s->ncell >= (size_t)1 << 31) return FDTD_ENOMEM;
  const size_t X = s->NPXa, Y = s->NPYa, maps = d.mode == FDTD_MODE_TM ? 1 : 2;
  char *b = nullptr;
  const size_t tables = (X * 8 + Y * 6) * sizeof(double) + (X + Y) * sizeof(D2);
  if (dev_malloc(&s->ie[0], maps * s->ncell * sizeof(double)) != hipSuccess ||
      dev_malloc(&b, tables + 2 * sizeof(StreamMap)) != hipSuccess) {
    (void)hipGetLastError();
    return FDTD_ENOMEM;
  }
  if (maps > 1) s->ie[1] = s->ie[0] + s->ncell;
  s->exy = (D2 *)b;
  s->xt = (double *)(s->exy + X + Y);
  s->yt = s->xt + X * 8;
  s->map = (StreamMap *)(s->yt + Y * 6);
  s->ctot = ct.total;
  for (int q = 0; q < 4; q++) {
    const Seg &g = ct.s[q];
    StreamSide &x = s->side[q];
    const int i0 = (int)(g.k0 / s->NPYa), j0 = (int)(g.k0 % s->NPYa);
    x.horiz = g.dk != 1;  // the column is fixed, the row varies
    x.fi = x.horiz ? j0 : i0;
    x.lo = x.horiz ? i0 : j0;
    x.n = g.n;
    x.off = g.off;
    x.ef = g.ef == 0 ? 0 : 1;
    x.hf = g.hf == 3 ? 1 : 2;
    x.es = g.es;
  }
  return FDTD_OK;
}

void stream_destroy(StreamState *s)
{
  if (!s) return;
  (void)dev_free(s->G);
  (void)dev_free(s->ie[0]);
  (void)dev_free(s->exy);
  (void)dev_free(s->strips);
  (void)dev_free(s->csamp);
  delete s;
}


int stream_set_coefs(StreamState *s, const fdtd_coef_tables *t)
{
  const int X = s->NPXa, Y = s->NPYa, off = s->off, T = STREAM_T;
  const bool tm = s->d.mode == FDTD_MODE_TM;
  const double c2 = 1.0 / s->d.mu0;
  std::vector<double> tab((size_t)X * 8 + (size_t)Y * 6);
  double *const xt = tab.data(), *const yt = xt + (size_t)X * 8;
  std::vector<char> px(X, 0), py(Y, 0);
  for (int i = 0; i < X; i++) {
    const bool ring = i == 0 || i == X - 1;
    const int x = std::min(std::max(i - off, 0), s->d.N_PX - 1);
    double *r = &xt[(size_t)i * 8];
    bool p = t->sx[x] != 0.0;
    for (int q = 0; q < 5; q++) {
      r[q] = t->x[q][x];
      p = p || r[q] != 1.0;
    }
    if (tm) r[1] *= c2;            // the curl is taken of B
    if (!tm && ring) r[4] = 0.0;   // keeps the ring's H zero
    r[5] = 1.0 / (2.0 + t->sx[x]);
    r[6] = ring ? 0.0 : 1.0;
    px[i] = p && !ring;
  }
  for (int j = 0; j < Y; j++) {
    const bool ring = j == 0 || j == Y - 1;
    const int y = std::min(std::max(j - off, 0), s->d.N_PY - 1);
    bool p = t->sy[y] != 0.0;
    for (int q = 0; q < 4; q++) {
      yt[(size_t)q * Y + j] = t->y[q][y];
      p = p || t->y[q][y] != 1.0;
    }
    if (!tm) yt[(size_t)Y + j] *= c2;
    if (ring) yt[3 * (size_t)Y + j] = 0.0;  // keeps the ring's H zero
    yt[4 * (size_t)Y + j] = t->sy[y];
    py[j] = p && !ring;
  }
  // the box of updated cells without UPML (none if UPML rows or columns lie inside it)
  auto box = [](const std::vector<char> &p, int &lo, int &hi) {
    lo = 1;
    hi = (int)p.size() - 1;
    while (lo < hi && p[lo]) lo++;
    while (hi > lo && p[hi - 1]) hi--;
    for (int i = lo; i < hi; i++)
      if (p[i]) hi = lo;
  };
  int xlo, xhi, ylo, yhi;
  box(px, xlo, xhi);
  box(py, ylo, yhi);
  s->xlo = xlo;
  s->xhi = xhi;
  s->ylo = ylo;
  s->yhi = yhi;
  // the cells that keep auxiliaries: every updated one outside the box's rows or columns
  for (int i = 0; i < X; i++) xt[(size_t)i * 8 + 7] = i > 0 && i < X - 1 && (i < xlo || i >= xhi) ? 1.0 : 0.0;
  for (int j = 0; j < Y; j++) yt[5 * (size_t)Y + j] = j > 0 && j < Y - 1 && (j < ylo || j >= yhi) ? 1.0 : 0.0;
  HIPCHK(hipMemcpy(s->xt, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
  // interior strips: every cell of their blocks lies in the box
  const int I0 = xlo + T, I1 = xhi - T, J0 = ylo + T, J1 = yhi - T;
  const bool inner = I0 < I1 && J0 < J1;
  struct Band {
    int kind, r0, r1;
    std::vector<Span> cols;
  };
  std::vector<Band> bands;
  auto band = [&](int kind, int r0, int r1, int c0, int c1) {
    if (r0 < r1 && c0 < c1)
      bands.push_back({kind, r0, r1, cover_cols(c0, c1, Y, kind ? 64 : 64 * stream_cols(s->d.mode, s->d.flavour), T, T)});
  };
  if (inner) {  // the longer strips first
    band(1, 1, I0, 1, Y - 1);
    band(1, I1, X - 1, 1, Y - 1);
    band(1, I0, I1, 1, J0);
    band(1, I0, I1, J1, Y - 1);
    band(0, I0, I1, J0, J1);
  } else {
    band(1, 1, X - 1, 1, Y - 1);
  }
  // rows of a band's strips of at most L, and how many of them
  auto split = [](const Band &b, int L, int &nch) {
    nch = std::max(1, (b.r1 - b.r0 + L - 1) / L);
    const int rows = (b.r1 - b.r0 + nch - 1) / nch;
    nch = (b.r1 - b.r0 + rows - 1) / rows;
    return rows;
  };
  std::vector<StreamStrip> v;
  auto fill = [&](const Band &b, int L) {
    int nch;
    const int rows = split(b, L, nch);
    for (int r = b.r0; r < b.r1; r += rows)
      for (const Span &c : b.cols) {
        StreamStrip t;
        memset(&t, 0, sizeof t);
        t.kind = b.kind;
        t.j0 = c.c0;
        t.j1 = c.c1;
        t.bj = c.b0;
        t.r0 = r;
        t.r1 = std::min(b.r1, r + rows);
        t.b0 = r == 1 ? 0 : r - T;
        t.bl = std::min(X - 1, t.r1 - 1 + T);
        t.s0 = t.r1;
        for (int q = 0; q < 4; q++) {
          // the sides that pass through the strip and the rows they take
          const StreamSide &g = s->side[q];
          const int ra = std::max(t.r0, g.horiz ? g.lo : g.fi - 1), rb = std::min(t.r1, g.horiz ? g.lo + g.n : g.fi + 1);
          const int ca = std::max(t.j0, g.horiz ? g.fi - 1 : g.lo), cb = std::min(t.j1, g.horiz ? g.fi + 1 : g.lo + g.n);
          if (g.n <= 0 || ra >= rb || ca >= cb) continue;
          t.smp |= 1 << q;
          t.s0 = std::min(t.s0, ra);
          t.s1 = std::max(t.s1, rb);
        }
        v.push_back(t);
      }
  };
  // Rows per strip {frame, interior}.  A strip's T + lag rows of run-in favour long
  // strips, a chip with idle compute units short ones: the shortest pair whose strips
  // all run at once, both kinds in one launch (two workgroups of these registers fit a
  // compute unit).  8-step launches of the TM grids: 276 x 276 {8, 12} 31.9 us,
  // {16, 24} 39.1; 1056 x 1056 {16, 32} 58.5 us (one generation), {16, 24} 79.2 (two),
  // {24, 48} 71.1, apart 38.0 + 45.4 (since then 29.9 and 52.2 with the
  // chosen pairs).  Larger grids run the two kinds apart.
  static const int rows[][2] = {{8, 12}, {8, 16}, {16, 24}, {16, 32}, {24, 48}, {32, 64}, {64, 128}};
  size_t q = 0;
  for (; q + 1 < sizeof rows / sizeof rows[0]; q++) {
    size_t all = 0;
    for (const Band &b : bands) {
      int nch;
      split(b, rows[q][b.kind ? 0 : 1], nch);
      all += nch * b.cols.size();
    }
    if (all <= STREAM_BOTH_MAX) break;
  }
  for (const Band &b : bands) {
    if (!b.kind) s->nfrm = (int)v.size();
    fill(b, rows[q][b.kind ? 0 : 1]);
  }
  if (!inner) s->nfrm = (int)v.size();
  s->nint = (int)v.size() - s->nfrm;
  (void)dev_free(s->strips);
  s->strips = nullptr;
  s->coefs = false;
  if (dev_malloc(&s->strips, v.size() * sizeof(StreamStrip)) != hipSuccess) {  // the grid steps in place
    (void)hipGetLastError();
    return FDTD_OK;
  }
  HIPCHK(hipMemcpy(s->strips, v.data(), v.size() * sizeof(StreamStrip), hipMemcpyHostToDevice));
  s->coefs = true;
  s->wave = false;
  return FDTD_OK;
}

int stream_set_eps(StreamState *s, double *const *eps)
{
  const dim3 blk(64, 4), grd((s->NPYa + 63) / 64, (s->NPXa + STREAM_IE_ROWS - 1) / STREAM_IE_ROWS);
  StreamMap m[2];
  HIPCHK(hipMemsetAsync(s->map, 0, sizeof m, 0));
  for (int e = 0; e < 2; e++)
    if (s->ie[e]) hipLaunchKernelGGL(k_stream_ie, grd, blk, 0, 0, eps[e], s->NPXa, s->NPYa, s->ie[e], s->map + e);
  HIPCHK(hipGetLastError());
  HIPCHK(hipMemcpy(m, s->map, sizeof m, hipMemcpyDeviceToHost));
  s->seen = StreamMap{m[0].odd | m[1].odd, std::max(m[0].i0, m[1].i0), std::max(m[0].i1, m[1].i1),
                      std::max(m[0].j0, m[1].j0), std::max(m[0].j1, m[1].j1)};
  return FDTD_OK;
}

void stream_reset(StreamState *s) { s->steps = 0; }
long stream_steps_done(const StreamState *s) { return s->steps; }

// whether a step with these parameters continues the steps taken so far
bool stream_follows(const StreamState *s, const fdtd_step_params *p)
{
  if (!s->coefs || s->seen.odd) return false;
  if (!s->steps) return true;
  return p->angle_deg == s->angle && p->k == s->k && p->omega == s->omega && p->time == s->time + 1 &&
         (s->d.flavour == FDTD_FLAVOUR_MPI || s->d.mode == FDTD_MODE_TM ||
          (p->dot_x == s->dot[0] && p->dot_y == s->dot[1] && p->use_x == s->use[0] && p->use_y == s->use[1]));
}

// the wave of a step (its tables, s->wave, are made when a launch needs them)
static void take_wave(StreamState *s, const fdtd_step_params *p)
{
  if (s->wave && p->angle_deg == s->angle && p->k == s->k && p->omega == s->omega) return;
  const double rad = p->angle_deg * M_PI / 180.0;
  s->cpc = cos(rad) / s->d.c0;
  s->spc = sin(rad) / s->d.c0;
  s->wave = false;
  s->angle = p->angle_deg;
  s->k = p->k;
  s->omega = p->omega;
}

static int set_wave(StreamState *s, const fdtd_step_params *p)
{
  take_wave(s, p);
  if (s->wave) return FDTD_OK;
  const bool mpi = s->d.flavour == FDTD_FLAVOUR_MPI;
  const double rad = p->angle_deg * M_PI / 180.0;
  const double kx = mpi ? cos(rad) * p->k : s->cpc * p->omega, ky = mpi ? sin(rad) * p->k : s->spc * p->omega;
  std::vector<D2> t(s->NPXa + s->NPYa);
  for (int i = 0; i < s->NPXa; i++) t[i] = make_double2(cos((i - s->off) * kx), sin((i - s->off) * kx));
  for (int j = 0; j < s->NPYa; j++) t[s->NPXa + j] = make_double2(cos((j - s->off) * ky), sin((j - s->off) * ky));
  HIPCHK(hipMemcpy(s->exy, t.data(), t.size() * sizeof(D2), hipMemcpyHostToDevice));
  s->wave = true;
  return FDTD_OK;
}

// the components that carry the pulse, and its projection on them
static void take_dot(StreamState *s, const fdtd_step_params *p)
{
  if (s->d.flavour == FDTD_FLAVOUR_MPI) return;
  const bool tm = s->d.mode == FDTD_MODE_TM;
  s->dot[0] = tm ? 1.0 : p->dot_x;
  s->dot[1] = tm ? 0.0 : p->dot_y;
  s->use[0] = tm ? 1 : p->use_x;
  s->use[1] = tm ? 0 : p->use_y;
}

// the source terms of step e
static void take_source(StreamState *s, const fdtd_step_params &e)
{
  const fdtd_grid_desc &d = s->d;
  const bool tm = d.mode == FDTD_MODE_TM;
  if (d.flavour == FDTD_FLAVOUR_MPI) {
    const double wt = e.omega * e.time;
    s->c[0] = make_double2(e.ray_coef * cos(wt), -e.ray_coef * sin(wt));
  } else {
    // field_scatteredPulse constants (field.c:226-241)
    const double gx[2] = {tm ? 0.0 : 0.5, 0.0}, gy[2] = {0.0, tm ? 0.0 : 0.5};
    for (int v = 0; v < 2; v++) {
      const double t0 = -((d.N_PX / 2.0 + gx[v]) * s->cpc + (d.N_PY / 2 + gy[v]) * s->spc) + 500;
      s->po[v] = gx[v] * s->cpc + gy[v] * s->spc - (e.time - t0);
      const double ph = s->po[v] * e.omega;
      s->c[v] = make_double2(s->dot[v] * cos(ph), s->dot[v] * sin(ph));
    }
  }
  s->ps = make_double2(e.ps_re, e.ps_im);
}

int stream_note(StreamState *s, const fdtd_step_params *p)
{
  take_wave(s, p);
  take_dot(s, p);
  take_source(s, *p);
  s->steps++;
  s->time = p->time;
  return FDTD_OK;
}

// A block takes nearly the same time for any number of steps (its rows pass through every
// wavefront), the kernels of a step, two launches and with the per-step NTFF two more, as
// many times as there are steps.  Both in us, fitted to calls of 1 to 9 steps on 40 x 40 to
// 3200 x 3200 cells.  One step / a block of four: 80 x 80 MPI TM 6.6 / 30, plain TM 6.9 / 35,
// plain TE 7.3 / 32; 276 x 276 8.6 / 30, 8.5 / 41, 9.0 / 39; 700 x 700 26 / 36, 26 / 52,
// 26 / 72; 1056 x 1056 53 / 62, 53 / 107, 54 / 97; 2000 x 2000 258 / 153, 268 / 221, 267 / 276;
// with the per-step NTFF, MPI TM: 80 x 80 16 / 48, 276 x 276 21 / 49, 700 x 700 48 / 75.
// Calls of three steps so, against a block each: 80 x 80 plain TE 20 / 31, 531 x 402 plain
// TM 42 / 44, MPI TM 276 x 276 25 / 30.  Frame strips with a scatterer, which form its wave
// without room to keep it, make a small grid's launch longer: 80 x 80 and 276 x 276 with a
// cylinder up to the UPML, 8 steps: MPI TM 45, plain TM 56, plain TE 84.
int stream_few(const StreamState *s, int binned)
{
  const bool mpi = s->d.flavour == FDTD_FLAVOUR_MPI, tm = s->d.mode == FDTD_MODE_TM;
  const double n = (double)s->ncell;
  const double step = 6.5 + 36e-6 * n + 34e-6 * std::max(0.0, n - 9e5) + (binned ? 8 + 5.5e-3 * binned : 0);
  double launch = (mpi ? 29 + 18e-6 * n : tm ? 40 + 16e-6 * n : 35 + 52e-6 * n) + (binned ? 13 : 0);
  const StreamMap &m = s->seen;
  const int h = 2 * STREAM_T;  // a frame strip reaches that far into the box
  const bool frame = s->NPXa - m.i0 < s->xlo + h || m.i1 > s->xhi - h || s->NPYa - m.j0 < s->ylo + h || m.j1 > s->yhi - h;
  if (m.i1 && frame && n < 262144) launch += mpi ? 16 : tm ? 14 : 45;
  return std::min(STREAM_T, (int)(launch / step));
}

static void fill_args(const StreamState *s, StreamArgs &a, const D2 *src, D2 *dst)
{
  const fdtd_grid_desc &d = s->d;
  memset((void *)&a, 0, sizeof a);
  a.src = src;
  a.dst = dst;
  a.stride = s->stride;
  a.ie0 = s->ie[0];
  a.ie1 = s->ie[1];
  a.xt = s->xt;
  a.yt = s->yt;
  a.ex = s->exy;
  a.ey = s->exy + s->NPXa;
  a.NPXa = s->NPXa;
  a.NPYa = s->NPYa;
  a.xlo = s->xlo;
  a.xhi = s->xhi;
  a.c2 = 1.0 / d.mu0;
  a.mu0 = d.mu0;
  const bool mpi = d.flavour == FDTD_FLAVOUR_MPI, tm = d.mode == FDTD_MODE_TM;
  a.on[0] = mpi || tm ? tm : s->use[0];
  a.on[1] = tm ? 0 : (mpi ? 1 : s->use[1]);
  a.ps_on = d.point_source && tm && mpi;
  a.ps_i = d.N_PX / 2 + s->off;
  a.ps_j = d.N_PY / 2 + s->off;
  a.cpc = s->cpc;
  a.spc = s->spc;
  a.hasprev = s->steps > 0;
  for (int q = 0; q < 2; q++) {
    a.c[q][0][0] = s->steps ? s->c[q].x : 0;
    a.c[q][0][1] = s->steps ? s->c[q].y : 0;
    a.po[q][0] = s->po[q];
  }
  a.ps[0][0] = s->steps ? s->ps.x : 0;
  a.ps[0][1] = s->steps ? s->ps.y : 0;
}

template <int MODE, int FLAV>
static void launch(const StreamState *s, StreamArgs a)
{
  if (s->nint + s->nfrm <= STREAM_BOTH_MAX) {
    a.ns = s->nint + s->nfrm;
    a.strips = s->strips;
    hipLaunchKernelGGL((k_stream_both<MODE, FLAV>), dim3(8 * ((a.ns + 7) / 8)), dim3(256), 0, 0, a);
    return;
  }
  a.ns = s->nfrm;
  a.strips = s->strips;
  hipLaunchKernelGGL((k_stream<MODE, FLAV, 1, 1, 2, stream_pf(MODE, FLAV)>), dim3(8 * ((a.ns + 7) / 8)), dim3(256), 0, 0, a);
  a.ns = s->nint;
  a.strips = s->strips + s->nfrm;
  if (a.ns) hipLaunchKernelGGL((k_stream<MODE, FLAV, 0, stream_cols(MODE, FLAV), 2, STREAM_IPF>), dim3(8 * ((a.ns + 7) / 8)), dim3(256), 0, 0, a);
}

// n <= STREAM_T steps from the arrays *F, which then hold the new state (the
// buffer is swapped with the state's own); with at >= 0, the contour's samples
// after every step in the entries [at, at + n) of the state's STREAM_SAMPLES, from
// *smp on ([n][3][total]).  FDTD_ENOMEM, with nothing changed, if there is no room for these
// or for the second state
int stream_steps(StreamState *s, D2 **F, const fdtd_step_params *p, int n, int at, D2 **smp)
{
  if (n < 1 || n > STREAM_T) return fdtd_fail(FDTD_EINVAL, "bad number of steps %d", n);
  const bool mpi = s->d.flavour == FDTD_FLAVOUR_MPI, tm = s->d.mode == FDTD_MODE_TM;
  const size_t entry = 3 * (size_t)s->ctot;
  if (!s->G) {
    if (dev_malloc(&s->G, 9 * s->stride) != hipSuccess) {
      (void)hipGetLastError();
      return FDTD_ENOMEM;
    }
    hipLaunchKernelGGL(k_stream_ring, dim3((std::max(s->NPXa, s->NPYa) + 255) / 256, 4), dim3(256), 0, 0, s->G, s->stride,
                       s->NPXa, s->NPYa);
  }
  if (at >= 0) {
    if (at + n > STREAM_SAMPLES) return fdtd_fail(FDTD_EINVAL, "bad sample entry %d", at);
    if (!s->csamp) {
      if (dev_malloc(&s->csamp, STREAM_SAMPLES * entry * sizeof(D2)) != hipSuccess) {
        (void)hipGetLastError();
        return FDTD_ENOMEM;
      }
      HIPCHK(hipMemset(s->csamp, 0, STREAM_SAMPLES * entry * sizeof(D2)));
    }
  }
  int rc = set_wave(s, p);
  if (rc) return rc;
  take_dot(s, p);
  StreamArgs a;
  fill_args(s, a, *F, s->G);
  a.T = n;
  for (int q = 0; q < n; q++) {
    take_source(s, p[q]);
    for (int v = 0; v < 2; v++) {
      a.c[v][q + 1][0] = s->c[v].x;
      a.c[v][q + 1][1] = s->c[v].y;
      a.po[v][q + 1] = s->po[v];
    }
    a.ps[q + 1][0] = s->ps.x;
    a.ps[q + 1][1] = s->ps.y;
  }
  if (at >= 0) {
    a.csamp = s->csamp + at * entry;
    a.ctot = s->ctot;
    memcpy(a.side, s->side, sizeof a.side);
    if (smp) *smp = a.csamp;
  }
  if (tm && mpi) launch<FDTD_MODE_TM, FDTD_FLAVOUR_MPI>(s, a);
  else if (tm) launch<FDTD_MODE_TM, FDTD_FLAVOUR_PLAIN>(s, a);
  else if (mpi) launch<FDTD_MODE_TE, FDTD_FLAVOUR_MPI>(s, a);
  else launch<FDTD_MODE_TE, FDTD_FLAVOUR_PLAIN>(s, a);
  HIPCHK(hipGetLastError());
  std::swap(*F, s->G);
  s->steps += n;
  s->time = p[n - 1].time;
  return FDTD_OK;
}

// the auxiliaries of the cells without UPML, formed in F
int stream_fill_aux(StreamState *s, D2 *F)
{
  StreamArgs a;
  fill_args(s, a, F, F);
  const dim3 blk(64, 4), grd((s->NPYa - 2 + 63) / 64, (s->NPXa - 2 + 3) / 4);
  const bool mpi = s->d.flavour == FDTD_FLAVOUR_MPI, tm = s->d.mode == FDTD_MODE_TM;
  if (tm && mpi) hipLaunchKernelGGL((k_stream_aux<FDTD_MODE_TM, FDTD_FLAVOUR_MPI>), grd, blk, 0, 0, a);
  else if (tm) hipLaunchKernelGGL((k_stream_aux<FDTD_MODE_TM, FDTD_FLAVOUR_PLAIN>), grd, blk, 0, 0, a);
  else if (mpi) hipLaunchKernelGGL((k_stream_aux<FDTD_MODE_TE, FDTD_FLAVOUR_MPI>), grd, blk, 0, 0, a);
  else hipLaunchKernelGGL((k_stream_aux<FDTD_MODE_TE, FDTD_FLAVOUR_PLAIN>), grd, blk, 0, 0, a);
  HIPCHK(hipGetLastError());
  return FDTD_OK;
}
