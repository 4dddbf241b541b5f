// fdtd_stream_split.hip -- FP64 split-field PML (fdtdTM.c, fdtdTE.c) and
// non-standard FDTD (nsFdtdTM.c, nsFdtdTE.c) steps, temporally blocked, for gfx950.
//
// The scheme of fdtd_stream.hip: a workgroup of SP_K wavefronts walks a strip of 64
// columns row by row, each wavefront takes a row through S steps, the rows in flight
// stay in register slots, and a finished row goes on to the next wavefront through
// LDS.  One body serves the whole grid: the absorbing layer differs from the interior
// by its coefficients only.  A cell's state is its two split components and the two
// fields of the other kind; the sum the split solvers also keep (Ez, Hz) is formed
// where it is used, and written at the end.
//
//   split TM   2 sigma rx, rx = 1/(eps + sigma_x) give both coefficients of
//              field_pmlCoef: (eps - sigma)/(eps + sigma) = 1 - 2 sigma rx; likewise ry
//   split TE   the same of eps_x with sigma_y and of eps_y with sigma_x
//   NS         the per-cell coefficient maps of fdtd_hip_grid_set_ns_coefs
//
// Bound as fdtd_stream.hip is (latency of a row's turn); the two launches per step
// that this replaces read and wrote every array (216 to 272 B per cell and step).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>
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

enum { SPLIT_TM = 0, SPLIT_TE = 1, NS_TM = 2, NS_TE = 3 };
#define SP_K 4
#define SP_PF 2  // rows fetched ahead of the first stage
// stages per wavefront, cell coefficients, rows a stage lags behind the one before it
__host__ __device__ constexpr int sp_s(int ph) { return ph == NS_TE ? 1 : 2; }
__host__ __device__ constexpr int sp_ni(int ph) { return ph == NS_TE ? 10 : ph == NS_TM ? 4 : 3; }
__host__ __device__ constexpr int sp_lag(int ph) { return ph == NS_TE ? 2 : 1; }
__host__ __device__ constexpr int sp_t(int ph) { return SP_K * sp_s(ph); }

struct SplitStrip {
  int j0, j1, bj, r0, r1, b0, bl, pad;
};

struct SplitArgs {
  const D2 *src;  // the nine arrays of the state, `stride` bytes apart
  D2 *dst;
  size_t stride;
  const double *cm;  // [NI][ncell] cell coefficients, 0 on the ring
  size_t cstride;    // bytes between them
  const double *xt;  // [NPXa][4] row coefficients
  const double *yt;  // [3][NPYa] column coefficients
  const D2 *ex, *ey; // e^{i kx x}, e^{i ky y}
  const SplitStrip *strips;
  int ns, NPXa, NPYa, T;
  double r2;         // NS: r / 2
  double c[2][STREAM_T + 1][2];  // the source's factor of each component at steps 1..T
};

__device__ __forceinline__ CAS(SplitArgs) rare_args()
{
#ifdef __HIP_DEVICE_COMPILE__
  CAS(SplitArgs) p = (CAS(SplitArgs))__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
#else
  return nullptr;
#endif
}

template <int PH>
__global__ __launch_bounds__(64 * SP_K) __attribute__((amdgpu_waves_per_eu(2))) void k_stream_split(SplitArgs a)
{
  constexpr bool TM = PH == SPLIT_TM || PH == NS_TM, NS = PH == NS_TM || PH == NS_TE;
  constexpr int S = sp_s(PH), K = SP_K, LG = sp_lag(PH), NI = sp_ni(PH), NV = 4, PF = SP_PF;
  // slots: the rows of the stages, the one behind the last stage where it is read
  // (TM: Hy; NS TE: Hz), the rows fetched ahead
  constexpr int NSL = LG * S + (PH == SPLIT_TE ? 1 : 2) + PF;
  __shared__ D2 lv[(K - 1) * 2 * NV * 64];
  __shared__ double li[(K - 1) * 2 * NI * 64];
  const int per = (a.ns + 7) / 8;
  const int id = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  if (id >= a.ns) return;
  const SplitStrip t = cload(a.strips + id);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int NPX = a.NPXa, NPY = a.NPYa;
  const int col = t.bj + lane;
  const int lc = min(col, min(NPY - 1, t.j1 + sp_t(PH)));  // lanes past the halo take its last column
  const bool lin = col < NPY;  // lanes past the grid hold zeros
  D2 V[NSL][NV];
  double I[NSL][NI];
  double X[NSL][4];  // the row's coefficients, scalar registers loaded an iteration ahead
  // e^{i kx x} of the row, likewise, and the source's factors at the wavefront's steps: loaded
  // where a row meets a scatterer, they were waits for two loads in turn in every stage (split
  // TM 901 x 653 with a cylinder 42.8 -> 41.1 us per 8 steps, 34 without).  NS TE, which
  // waits for its twelve arrays, does not gain: it loads the row's where it is used.
  D2 EX[NSL];
  double cs[S][2][2];
#pragma unroll
  for (int s = 0; s < S; s++)
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int x = 0; x < 2; x++) cs[s][c][x] = a.c[c][w * S + s + 1][x];
  bool fl[NSL];
  D2 PE[S];  // NS TM: Ez of the row behind a stage's two, before the stage updated it
#pragma unroll
  for (int q = 0; q < NSL; q++) {
    fl[q] = false;
#pragma unroll
    for (int v = 0; v < NV; v++) V[q][v] = d2(0, 0);
#pragma unroll
    for (int v = 0; v < NI; v++) I[q][v] = 0;
#pragma unroll
    for (int x = 0; x < 4; x++) X[q][x] = 0;
    EX[q] = d2(0, 0);
  }
#pragma unroll
  for (int s = 0; s < S; s++) PE[s] = d2(0, 0);
  for (int q = threadIdx.x; q < (K - 1) * 2 * NV * 64; q += 64 * K) lv[q] = d2(0, 0);
  for (int q = threadIdx.x; q < (K - 1) * 2 * NI * 64; q += 64 * K) li[q] = 0;
  __syncthreads();
  const D2 ey = a.ey[lc];
  const double y0 = a.yt[lc], y1 = a.yt[NPY + lc], y2 = a.yt[2 * NPY + lc];
  const double r2 = a.r2;
  auto rowc = [&](int r) { return min(max(r, 0), NPX - 1); };
  auto src = [&](int f) { return (const D2 *)((const char *)a.src + f * a.stride); };
  auto dst = [&](int f) { return (D2 *)((char *)a.dst + f * a.stride); };
  // the arrays of the four values
  constexpr int F[4] = {TM ? 1 : 0, TM ? 2 : 3, TM ? 3 : 7, TM ? 6 : 8};

  auto table = [&](int q, int r) {
    const double *x = a.xt + (size_t)__builtin_amdgcn_readfirstlane(rowc(r)) * 4;
#pragma unroll
    for (int v = 0; v < 3; v++) X[q][v] = cload(x + v);
    if (PH != NS_TE) EX[q] = cload2(a.ex + __builtin_amdgcn_readfirstlane(rowc(r)));
  };
  auto load = [&](int q, int r0) {
    const int r = min(rowc(r0), t.bl);
    const unsigned k = (unsigned)(r * NPY + lc);
#pragma unroll
    for (int v = 0; v < NI; v++) I[q][v] = ((const double *)((const char *)a.cm + v * a.cstride))[k];
#pragma unroll
    for (int v = 0; v < NV; v++) V[q][v] = src(F[v])[k];
  };
  auto flag = [&](int q) {
    const bool any = PH == NS_TE ? (I[q][NI - 2] != 0.0 || I[q][NI - 1] != 0.0) : I[q][NI - 1] != 0.0;
    fl[q] = __ballot(any) != 0;
  };
  auto settle = [&](int q) {
    if (!lin) {
#pragma unroll
      for (int v = 0; v < NV; v++) V[q][v] = d2(0, 0);
#pragma unroll
      for (int v = 0; v < NI; v++) I[q][v] = 0;
    }
    flag(q);
  };
  // the source on component c (factor map f) of row r in slot q, its factor at the step k
  auto source = [&](int q, int f, int r, D2 k) -> D2 {
    const D2 x = PH == NS_TE ? cload2(rare_args()->ex + __builtin_amdgcn_readfirstlane(rowc(r))) : EX[q];
    return cmulp(mul(I[q][f], cmulp(x, ey)), k);
  };

  // one stage: the rows in slots A (newest, row r), B, Z, Y behind it, at step st
  auto stage = [&](int s, int A, int B, int Z, int Y, int r, int st) {
    if (PH == SPLIT_TM) {  // calcH, calcE, the wave on Ezx (fdtdTM.c:283-327)
      const D2 eA = add(V[A][0], V[A][1]), eB = add(V[B][0], V[B][1]);
      V[A][2] = sub(mul(y1, V[A][2]), mul(y2, sub(above(eA), eA)));
      V[B][3] = mad(X[B][1], V[B][3], mul(X[B][2], sub(eA, eB)));
      const double rx = I[B][0], ry = I[B][1];
      V[B][0] = mad(fma(-X[B][0], rx, 1.0), V[B][0], mul(rx, sub(V[B][3], V[Z][3])));
      V[B][1] = mad(fma(-y0, ry, 1.0), V[B][1], mul(-ry, sub(V[B][2], below(V[B][2]))));
      if (RARE(fl[B])) V[B][0] = add(V[B][0], source(B, 2, r - 1, d2(cs[s][0][0], cs[s][0][1])));
    } else if (PH == SPLIT_TE) {  // calcE, the wave on Ey, calcH (fdtdTE.c:283-321)
      const D2 hA = add(V[A][2], V[A][3]), hB = add(V[B][2], V[B][3]);
      const double ry = I[A][0], rx = I[A][1];
      V[A][0] = mad(fma(-y0, ry, 1.0), V[A][0], mul(ry, sub(hA, below(hA))));
      V[A][1] = mad(fma(-X[A][0], rx, 1.0), V[A][1], mul(-rx, sub(hA, hB)));
      if (RARE(fl[A])) V[A][1] = add(V[A][1], source(A, 2, r, d2(cs[s][1][0], cs[s][1][1])));
      V[B][2] = sub(mul(X[B][1], V[B][2]), mul(X[B][2], sub(V[A][1], V[B][1])));
      V[B][3] = mad(y1, V[B][3], mul(y2, sub(above(V[B][0]), V[B][0])));
    } else if (PH == NS_TM) {  // calcH, calcE, the NS wave on Ezy (nsFdtdTM.c:68-151)
      const D2 eA = add(V[A][0], V[A][1]), c = add(V[B][0], V[B][1]), l = PE[s];
      const D2 u = above(c), d = below(c), ur = above(eA), dr = below(eA), ul = above(l);
      // second differences across the rows at j + 1 and j, across the columns at i + 1 and i
      const D2 nx = sub(mad(-2.0, u, add(ur, ul)), mad(-2.0, c, add(eA, l)));
      const D2 ny = sub(mad(-2.0, eA, add(ur, dr)), mad(-2.0, c, add(u, d)));
      V[B][2] = sub(mul(y1, V[B][2]), mul(I[B][1], mad(r2, nx, sub(u, c))));
      V[B][3] = mad(X[B][1], V[B][3], mul(I[B][2], mad(r2, ny, sub(eA, c))));
      V[B][0] = mad(X[B][0], V[B][0], mul(I[B][0], sub(V[B][3], V[Z][3])));
      V[B][1] = mad(y0, V[B][1], mul(-I[B][0], sub(V[B][2], below(V[B][2]))));
      if (RARE(fl[B])) V[B][1] = add(V[B][1], source(B, 3, r - 1, d2(cs[s][0][0], cs[s][0][1])));
      PE[s] = c;
    } else {  // calcH, then calcE a row behind it, the NS waves (nsFdtdTE.c:242-308)
      V[B][2] = sub(mul(I[B][4 % NI], V[B][2]), mul(I[B][5 % NI], sub(V[A][1], V[B][1])));
      V[B][3] = mad(I[B][6 % NI], V[B][3], mul(I[B][7 % NI], sub(above(V[B][0]), V[B][0])));
      const D2 rr = add(V[B][2], V[B][3]), c = add(V[Z][2], V[Z][3]), l = add(V[Y][2], V[Y][3]);
      const D2 u = above(c), d = below(c), dr = below(rr), dl = below(l), ul = above(l);
      const D2 nx = sub(mad(-2.0, c, add(rr, l)), mad(-2.0, d, add(dr, dl)));
      const D2 ny = sub(mad(-2.0, c, add(u, d)), mad(-2.0, l, add(ul, dl)));
      V[Z][0] = mad(I[Z][0], V[Z][0], mul(I[Z][1], mad(r2, nx, sub(c, d))));
      V[Z][1] = mad(I[Z][2 % NI], V[Z][1], mul(-I[Z][3 % NI], mad(r2, ny, sub(c, l))));
      if (RARE(fl[Z])) {
        V[Z][0] = add(V[Z][0], source(Z, 8 % NI, r - 2, d2(cs[s][0][0], cs[s][0][1])));
        V[Z][1] = add(V[Z][1], source(Z, 9 % NI, r - 2, d2(cs[s][1][0], cs[s][1][1])));
      }
    }
  };
  auto store = [&](int q, int r) {
    if (r < t.r0 || r >= t.r1 || col < t.j0 || col >= t.j1) return;
    const unsigned k = (unsigned)(r * NPY + col);
#pragma unroll
    for (int v = 0; v < NV; v++) dst(F[v])[k] = V[q][v];
    D2 sum = TM ? add(V[q][0], V[q][1]) : add(V[q][2], V[q][3]);
    // the split TM solver forms Ez before the wave is added to Ezx (fdtdTM.c:283-288)
    if (PH == SPLIT_TM && I[q][2] != 0.0) {
      CAS(SplitArgs) R = rare_args();
      sum = sub(sum, source(q, 2, r, d2(R->c[0][a.T][0], R->c[0][a.T][1])));
    }
    dst(TM ? 0 : 6)[k] = sum;
  };
  auto put = [&](int q, int p) {
    D2 *o = lv + (2 * w + p) * (NV * 64) + lane;
    double *oi = li + (2 * w + p) * (NI * 64) + lane;
#pragma unroll
    for (int v = 0; v < NV; v++) o[v * 64] = V[q][v];
#pragma unroll
    for (int v = 0; v < NI; v++) oi[v * 64] = I[q][v];
  };
  auto take = [&](int q, int p) {
    const D2 *o = lv + (2 * (w - 1) + p) * (NV * 64) + lane;
    const double *oi = li + (2 * (w - 1) + p) * (NI * 64) + lane;
#pragma unroll
    for (int v = 0; v < NV; v++) V[q][v] = o[v * 64];
#pragma unroll
    for (int v = 0; v < NI; v++) I[q][v] = oi[v * 64];
  };

  // Iteration `it`: wavefront w's newest row is b0 + it - w (LG S + 2), in slot it mod
  // NSL; the last core row leaves the last wavefront in iteration nit - 1.
  const int row0 = t.b0 - w * (LG * S + 2);
  const int nit = (t.r1 - t.b0) + LG * S + (K - 1) * (LG * S + 2);
  auto march = [&](auto FIRST, auto LAST) {  // a copy per kind of wavefront (see fdtd_stream.hip)
    constexpr bool first = decltype(FIRST)::value, last = decltype(LAST)::value;
    if (first) {
#pragma unroll
      for (int q = 0; q < PF; q++) {
        load(q, t.b0 + q);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    table(0, row0);
    for (int it0 = 0; it0 < nit; it0 += NSL) {
#pragma unroll
      for (int u = 0; u < NSL; u++) {
        const int it = it0 + u;
        if (RARE(it >= nit)) return;
        const int n = row0 + it;
        if (first) settle(u);
        else flag(u);
        if (first) load((u + PF) % NSL, n + PF);
        else take((u + 1) % NSL, (it + 1) & 1);
        table((u + 1) % NSL, n + 1);
#pragma unroll
        for (int s = 0; s < S; s++) {
          const int st = w * S + s + 1, q = u - LG * s + 4 * NSL;
          if (!RARE(st > a.T)) stage(s, q % NSL, (q - 1) % NSL, (q - 2) % NSL, (q - 3) % NSL, n - LG * s, st);
        }
        const int O = (u - LG * S + 4 * NSL) % NSL;
        if (last) store(O, n - LG * S);
        else put(O, it & 1);
        lds_barrier();
      }
    }
  };
  if (w == 0) march(std::true_type(), std::false_type());
  else if (w == K - 1) march(std::false_type(), std::true_type());
  else march(std::false_type(), std::false_type());
}

// Split-field solvers' cell coefficients from the eps maps: {rx, ry, 1/eps - 1} (TM of
// EPS_EZ; TE ry of EPS_EX, rx of EPS_EY, the factor of EPS_EY), 0 on the ring
template <int PH>
__global__ __launch_bounds__(256) void k_split_cells(const double *e0, const double *e1, const double *sx, const double *sy,
                                                     int NPXa, int NPYa, double *cm, size_t n)
{
  const int j = blockIdx.x * 64 + threadIdx.x, i = blockIdx.y * 4 + threadIdx.y;
  if (i >= NPXa || j >= NPYa) return;
  const size_t k = (size_t)i * NPYa + j;
  const bool ring = i == 0 || j == 0 || i == NPXa - 1 || j == NPYa - 1;
  const double ex = e0[k], ey = PH == SPLIT_TM ? e0[k] : e1[k];
  const double rx = 1.0 / (ey + sx[i]), ry = 1.0 / (ex + sy[j]);
  cm[k] = ring ? 0.0 : (PH == SPLIT_TM ? rx : ry);
  cm[n + k] = ring ? 0.0 : (PH == SPLIT_TM ? ry : rx);
  cm[2 * n + k] = ring ? 0.0 : 1.0 / ey - 1.0;
}

// NS TM: {C_EZXLX (= C_EZYLY), C_HXLY, C_HYLX, wave factor} of the five maps; NS TE: the
// ten maps; 0 on the ring
__global__ __launch_bounds__(256) void k_ns_cells(const double *nsc, int tm, int NPXa, int NPYa, double *cm, size_t n)
{
  const int j = blockIdx.x * 64 + threadIdx.x, i = blockIdx.y * 4 + threadIdx.y;
  if (i >= NPXa || j >= NPYa) return;
  const size_t k = (size_t)i * NPYa + j;
  const bool ring = i == 0 || j == 0 || i == NPXa - 1 || j == NPYa - 1;
  for (int v = 0; v < (tm ? 4 : 10); v++) cm[v * n + k] = ring ? 0.0 : nsc[(tm && v ? v + 1 : v) * n + k];
}

// ---------------------------------------------------------------- host

struct SplitState {
  fdtd_grid_desc d;
  int ph, NPXa, NPYa;
  size_t ncell, stride;
  D2 *G;  // the nine arrays a launch writes, swapped with the grid's after it; made by the first launch
  double *cm, *xt, *yt;
  D2 *exy;  // in one block with xt, yt
  SplitStrip *strips;
  int ns;
  bool coefs, cells, wave;
  double angle, k, r2;
};

int split_create(const fdtd_grid_desc &d, SplitState **out)
{
  SplitState *s = new SplitState();
  *out = s;
  memset((void *)s, 0, sizeof *s);
  s->d = d;
  const bool tm = d.mode == FDTD_MODE_TM;
  s->ph = d.flavour == FDTD_FLAVOUR_NS ? (tm ? NS_TM : NS_TE) : (tm ? SPLIT_TM : SPLIT_TE);
  s->NPXa = d.N_PX;
  s->NPYa = d.N_PY;
  s->ncell = (size_t)s->NPXa * s->NPYa;
  s->stride = stream_stride(s->ncell);
  // a grid without room for these, or past 32-bit cell indexes, steps in place
  if (s->ncell >= (size_t)1 << 31) return FDTD_ENOMEM;
  const size_t nx = s->NPXa, ny = s->NPYa;
  if (dev_malloc(&s->cm, sp_ni(s->ph) * s->ncell * sizeof(double)) != hipSuccess ||
      dev_malloc(&s->exy, (nx + ny) * sizeof(D2) + (nx * 4 + ny * 3) * sizeof(double)) != hipSuccess) {
    (void)hipGetLastError();
    return FDTD_ENOMEM;
  }
  s->xt = (double *)(s->exy + nx + ny);
  s->yt = s->xt + nx * 4;
  // Strips: a halo of T cells below and left, T + 1 above and right (the non-standard TE
  // half reaches one cell further there).  Rows per strip as in fdtd_stream.hip: the
  // shortest strips that all run at once, two workgroups on each of 256 compute units.
  const int T = sp_t(s->ph), X = s->NPXa, Y = s->NPYa;
  const std::vector<Span> cols = cover_cols(1, Y - 1, Y, 64, T, T + 1);
  int rows = 0;
  for (int L : {8, 12, 16, 24, 32, 48, 64, 96, 128}) {
    const int nch = (X - 2 + L - 1) / L;
    rows = (X - 2 + nch - 1) / nch;
    if ((X - 2 + rows - 1) / rows * cols.size() <= 512) break;
  }
  std::vector<SplitStrip> v;
  for (int r = 1; r < X - 1; r += rows)
    for (const Span &c : cols) {
      SplitStrip q;
      q.j0 = c.c0;
      q.j1 = c.c1;
      q.bj = c.b0;
      q.r0 = r;
      q.r1 = std::min(X - 1, r + rows);
      q.b0 = r == 1 ? 0 : r - T;
      q.bl = std::min(X - 1, q.r1 + T);
      q.pad = 0;
      v.push_back(q);
    }
  s->ns = (int)v.size();
  if (dev_malloc(&s->strips, v.size() * sizeof(SplitStrip)) != hipSuccess) {
    (void)hipGetLastError();
    return FDTD_ENOMEM;
  }
  HIPCHK(hipMemcpy(s->strips, v.data(), v.size() * sizeof(SplitStrip), hipMemcpyHostToDevice));
  return FDTD_OK;
}

void split_destroy(SplitState *s)
{
  if (!s) return;
  (void)dev_free(s->G);
  (void)dev_free(s->cm);
  (void)dev_free(s->exy);
  (void)dev_free(s->strips);
  delete s;
}

int split_set_coefs(SplitState *s, const fdtd_coef_tables *t)
{
  const int X = s->NPXa, Y = s->NPYa;
  std::vector<double> tab((size_t)X * 4 + (size_t)Y * 3, 0.0);
  double *const xt = tab.data(), *const yt = xt + (size_t)X * 4;
  const double mu = s->d.mu0;
  auto coef = [&](double sig) { return (1.0 - sig / mu) / (1.0 + sig / mu); };
  const bool ns = s->ph == NS_TM || s->ph == NS_TE;
  for (int i = 0; i < X; i++) {
    double *r = &xt[(size_t)i * 4];
    const bool ring = i == 0 || i == X - 1;
    r[0] = ns ? t->x[0][i] : 2.0 * t->x[0][i];
    r[1] = ns ? t->x[1][i] : coef(t->x[1][i]);
    r[2] = ns || ring ? 0.0 : 1.0 / (mu + t->x[1][i]);  // 0 keeps the ring's H zero
  }
  for (int j = 0; j < Y; j++) {
    const bool ring = j == 0 || j == Y - 1;
    yt[j] = ns ? t->y[0][j] : 2.0 * t->y[0][j];
    yt[(size_t)Y + j] = ns ? t->y[1][j] : coef(t->y[1][j]);
    yt[2 * (size_t)Y + j] = ns || ring ? 0.0 : 1.0 / (mu + t->y[1][j]);
  }
  HIPCHK(hipMemcpy(s->xt, tab.data(), tab.size() * sizeof(double), hipMemcpyHostToDevice));
  s->coefs = true;
  return FDTD_OK;
}

int split_set_eps(SplitState *s, double *const *eps, const double *sx, const double *sy)
{
  const dim3 blk(64, 4), grd((s->NPYa + 63) / 64, (s->NPXa + 3) / 4);
  if (s->ph == SPLIT_TM)
    hipLaunchKernelGGL(k_split_cells<SPLIT_TM>, grd, blk, 0, 0, eps[0], eps[1], sx, sy, s->NPXa, s->NPYa, s->cm, s->ncell);
  else if (s->ph == SPLIT_TE)
    hipLaunchKernelGGL(k_split_cells<SPLIT_TE>, grd, blk, 0, 0, eps[0], eps[1], sx, sy, s->NPXa, s->NPYa, s->cm, s->ncell);
  else
    return FDTD_OK;
  HIPCHK(hipGetLastError());
  s->cells = true;
  return FDTD_OK;
}

int split_set_ns(SplitState *s, const double *nsc, double r2)
{
  const dim3 blk(64, 4), grd((s->NPYa + 63) / 64, (s->NPXa + 3) / 4);
  hipLaunchKernelGGL(k_ns_cells, grd, blk, 0, 0, nsc, s->ph == NS_TM ? 1 : 0, s->NPXa, s->NPYa, s->cm, s->ncell);
  HIPCHK(hipGetLastError());
  s->r2 = r2;
  s->cells = true;
  return FDTD_OK;
}

int split_depth(const SplitState *s) { return s->coefs && s->cells ? sp_t(s->ph) : 0; }

// Steps that take no more time one by one: a launch of blocks costs nearly the same for
// any number of them, the kernels of a step, two launches, once a step.  Calls of 1, 2 and
// 3 steps, one by one / in a block, us: 80 x 80 NS TM 6.1, 12, 19 / 17, 22, 22; 276 x 276
// split TM 7.5, 15, 22 / 16, 18, 18, NS TE 7.8, 16, 23 / 18, 18, 18; 700 x 700 split TM 18,
// 36 / 24, 29; 2000 x 2000 split TM 144, 289 / 187, 189, NS TE 220, 439 / 251, 247;
// 3200 x 3200 split TM 431 / 417, NS TE 529 / 521.
int split_few(const SplitState *s)
{
  const size_t n = s->ncell;
  return n < (size_t)1 << 16 && s->ph == NS_TM ? 3 : n < (size_t)1 << 18 ? 2 : n < (size_t)8 << 20 ? 1 : 0;
}

// n <= split_depth() steps of one wave direction from *F, which then holds the new state;
// FDTD_ENOMEM, with nothing changed, if there is no room for the second state
int split_steps(SplitState *s, D2 **F, const fdtd_step_params *p, int n)
{
  if (!s->G) {
    if (dev_malloc(&s->G, 9 * s->stride) != hipSuccess) {
      (void)hipGetLastError();
      return FDTD_ENOMEM;
    }
    // (the ring and the arrays these solvers do not use stay zero)
    HIPCHK(hipMemsetAsync(s->G, 0, 9 * s->stride, 0));
  }
  const double rad = p->angle_deg * M_PI / 180.0, kx = cos(rad) * p->k, ky = sin(rad) * p->k;
  if (!s->wave || p->angle_deg != s->angle || p->k != s->k) {
    std::vector<D2> t(s->NPXa + s->NPYa);
    for (int i = 0; i < s->NPXa; i++) t[i] = make_double2(cos(i * kx), sin(i * kx));
    for (int j = 0; j < s->NPYa; j++) t[s->NPXa + j] = make_double2(cos(j * ky), sin(j * ky));
    HIPCHK(hipMemcpy(s->exy, t.data(), t.size() * sizeof(D2), hipMemcpyHostToDevice));
    s->wave = true;
    s->angle = p->angle_deg;
    s->k = p->k;
  }
  SplitArgs a;
  memset((void *)&a, 0, sizeof a);
  a.src = *F;
  a.dst = s->G;
  a.stride = s->stride;
  a.cm = s->cm;
  a.cstride = s->ncell * sizeof(double);
  a.xt = s->xt;
  a.yt = s->yt;
  a.ex = s->exy;
  a.ey = s->exy + s->NPXa;
  a.strips = s->strips;
  a.ns = s->ns;
  a.NPXa = s->NPXa;
  a.NPYa = s->NPYa;
  a.T = n;
  a.r2 = s->r2;
  const bool ns = s->ph == NS_TM || s->ph == NS_TE, te = s->ph == SPLIT_TE || s->ph == NS_TE;
  for (int q = 0; q < n; q++) {
    const fdtd_step_params &e = p[q];
    // e^{i (k.r - w t1)} - e^{i (k.r - w t0)} (field.c:155-199), TE at gap (0, 1/2)
    const double t1 = ns ? e.time + 1.0 : e.time + 0.5, t0 = ns ? e.time : e.time - 0.5, g = te ? 0.5 * ky : 0.0;
    const double re = e.ray_coef * (cos(g - e.omega * t1) - cos(g - e.omega * t0));
    const double im = e.ray_coef * (sin(g - e.omega * t1) - sin(g - e.omega * t0));
    for (int c = 0; c < 2; c++) {
      double f = 1.0;
      if (s->ph == NS_TE) f = c == 0 ? (e.use_x ? e.dot_x : 0.0) : (e.use_y ? e.dot_y : 0.0);
      a.c[c][q + 1][0] = f * re;
      a.c[c][q + 1][1] = f * im;
    }
  }
  const dim3 grid(8 * ((s->ns + 7) / 8)), blk(64 * SP_K);
  switch (s->ph) {
    case SPLIT_TM: hipLaunchKernelGGL(k_stream_split<SPLIT_TM>, grid, blk, 0, 0, a); break;
    case SPLIT_TE: hipLaunchKernelGGL(k_stream_split<SPLIT_TE>, grid, blk, 0, 0, a); break;
    case NS_TM: hipLaunchKernelGGL(k_stream_split<NS_TM>, grid, blk, 0, 0, a); break;
    default: hipLaunchKernelGGL(k_stream_split<NS_TE>, grid, blk, 0, 0, a); break;
  }
  HIPCHK(hipGetLastError());
  std::swap(*F, s->G);
  return FDTD_OK;
}
