// Device kernels of the acoustic RK4 hot path for gfx950 (MI355X).
//
// State layout in HBM: q(n,n,nr,5,6), i fastest, one n*n*nr block per field
// per panel, stored as S = double (FP64 path) or float (FP32-state variant:
// storage only -- every kernel computes in FP64 with FP64 tables and ghosts).  All arithmetic follows the reference's expression order and is
// compiled with -ffp-contract=off, so results match the CPU restatement of
// the reference bit for bit (tables are built on the host, see
// solar_tables.cpp).
//
//   k_gather  : the panel exchange (derivative.f90:55-133,374-452) as an
//               on-device gather: 9-tap Lagrange interpolation along the
//               sender's edge rows (interpolation.f90:140-378), for vectors
//               with the basis conversion at the source points
//               (transform.f90:8-59) and the receiver-basis transform
//               (transform.f90:114-276).
//   k_stage   : one RK stage fused in a single pass over HBM: DDX/DDY/DDR
//               (derivative.f90), COMPUTE_DIVERGENCE / COMPUTE_GRADIENT
//               (grad.f90:13-136), the RHS (compute_rhs_acoustic.f90:38-149),
//               BC_RHS, SPONGE and the 2N update (timestep.f90:64-69).
//   k_filter  : FILTER_EXP (filter.f90:9-781): xi then eta filter through an
//               LDS plane tile, then the 11-tap radial filter from a
//               register window.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "solar_device.hpp"
#include "solar_kernels.hpp"
#include "solar_tiles.hpp"

namespace solar {

__device__ __forceinline__ int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// a / b rounded to nearest -- the IEEE quotient, bit for bit -- from
// y = RN(1/b), precomputed where b is fixed: q = RN(a y), then two
// corrections q <- RN(q - r y) with the negated remainder r = b q - a, exact
// by FMA once q is within an ulp of a/b (Markstein: with y within half an ulp
// of 1/b and q within an ulp of a/b, the correction rounds to RN(a/b)).  The
// negated remainder keeps the sign of a zero quotient (-0 / b = -0).  The
// remainders and quotients must stay normal: with the divisors in
// [2^-60, 2^60] (fast, checked on the host) a numerator whose exponent lies
// in [-900, 900], or zero, may take this path; others (subnormal field
// values occur in the tails of Gaussian pulses) take the hardware division
// (div_group), as do all when fast is false.  An infinite numerator gives
// NaN here where the division gives an infinity (both non-finite).  Five
// FP64 operations and an exponent test, against about a dozen with a
// quarter-rate reciprocal.
__device__ __forceinline__ double quot_rcp(double a, double b, double y) {
  const double q0 = a * y;
  const double r0 = __builtin_fma(b, q0, -a);
  const double q1 = __builtin_fma(-r0, y, q0);
  const double r1 = __builtin_fma(b, q1, -a);
  return __builtin_fma(-r1, y, q1);
}
// The numerator test: above 1800 when the exponent lies outside [-900, 900].
__device__ __forceinline__ unsigned quot_exp(double a) { return (unsigned)(__builtin_amdgcn_frexp_exp(a) + 900); }
// A group of quotients with one test (RCP): every lane takes the reciprocal
// sequence; in a wave where some lane's numerators fail the test (or fast
// is false) those lanes redo the group by hardware division.  The common
// path then has no branch per quotient.  Without RCP, hardware division.
// live: the lane's quotients are used (lanes of a partial tile without a point
// of their own divide what their cells happen to hold).
// Measured in one call: the FP32-state step at c3 16.23 -> 16.03 ms against
// a guard per quotient; the FP64 stages were 0 to 6% slower with it than
// with hardware division, and keep that (a guard per quotient had been slower
// there too: it drained the prefetch at the loop's back edge).
template <bool RCP, int N>
__device__ __forceinline__ void div_group(const double (&a)[N], const double (&b)[N], const double (&y)[N], bool fast,
                                          bool live, double (&q)[N]) {
  if constexpr (!RCP) {
#pragma unroll
    for (int t = 0; t < N; ++t) q[t] = a[t] / b[t];
    return;
  }
  unsigned m = 0;
#pragma unroll
  for (int t = 0; t < N; ++t) {
    q[t] = quot_rcp(a[t], b[t], y[t]);
    m = max(m, quot_exp(a[t]));
  }
  const bool slow = live && (!fast || m > 1800u);
  if (__builtin_expect(__ballot(slow) != 0, 0)) {
    if (slow) {
#pragma unroll
      for (int t = 0; t < N; ++t) q[t] = a[t] / b[t];
    }
  }
}

// Source point (i,j) of along-edge index a on the strip of edge e at layer l
// (1..3): S rows l, N rows n-1-l, W columns l, E columns n-1-l (0-based),
// i.e. rows/columns 2..4 and N-1..N-3 of grad.f90:28-31.
__device__ __forceinline__ int strip_index(int e, int l, int a, int n) {
  switch (e) {
    case kS: return l * n + a;
    case kN: return (n - 1 - l) * n + a;
    case kW: return a * n + l;
    default: return a * n + (n - 1 - l);
  }
}

// Ghost strips of one receiver edge (receiver panel P, edge e) over the
// planes [k0, k1), all three layers.  Per plane the sender's three source
// lines (rows/columns 2..4 or N-1..N-3 of grad.f90:28-31) are staged in LDS
// -- for vectors already converted to (theta, phi) with the sender's metric
// (transform.f90:19-56); threads walk the layer index fastest so the three
// adjacent columns of a W/E strip share cache lines.  Each thread then
// interpolates ghost values along the edge with the 9-point Lagrange weights
// (interpolation.f90:140-378; unit weights encode the end-point copies) and,
// for vectors, applies the receiver-basis transform (transform.f90:161-274).
// The conversion, weight and transform tables do not depend on the plane:
// each thread loads its own once into registers.  The next plane's source
// values load while this plane is interpolated, and the staged lines are
// double-buffered in LDS, so one barrier per plane suffices.
//   gx*: [P][side W/E][k][m][l],  gy*: [P][side S/N][k][l][m]
//   ecols: when not null, the compact copies of the sender's edge columns
//     (edge_cols layout, written by the stage that produced q); W/E strips
//     are then read from there, one contiguous run per field and plane,
//     instead of three values from every row of the field.
//   NI: strip points per thread (3n <= NI * blockDim.x)
//   sline: 2 buffers x 3 layers x (3 quantities for vectors, else 1) x n
//   qwr (not null, row strips only): the source is q + betar * qwr, the
//     input of a stage that is rebuilt from q and qw (the edge columns hold
//     it as computed).
template <bool VEC, typename S, int NI>
__device__ __forceinline__ void gather_edge(const DevTables& T, int P, int e, int k0, int k1, int fld,
                                            const S* __restrict__ q, const S* __restrict__ ecols, int sfield,
                                            double* __restrict__ gxs, double* __restrict__ gys,
                                            double* __restrict__ gxv, double* __restrict__ gyv,
                                            long long field_stride_out, double* sline, const S* __restrict__ qwr,
                                            double betar) {
  constexpr int NQ = VEC ? 3 : 1;
  const int n = T.n, nr = T.nr;
  const Route rt = T.route[P * 4 + e];
  const int s = rt.sender, se = rt.sender_edge;
  const size_t plane = (size_t)n * n, nf = plane * nr;
  const int colstrip = (se == kW || se == kE);  // column strips: layer index is the fast memory index
  const bool from_cols = colstrip && ecols != nullptr;
  // source of field f at plane k, strip offset x: src[f * fstr + k * kstr + x]
  const S* src = from_cols ? ecols + (size_t)(s * 2 + (se == kE)) * nr * edge_cols_plane(n) : q + (size_t)s * 5 * nf;
  const size_t fstr = from_cols ? (size_t)3 * n : nf, kstr = from_cols ? edge_cols_plane(n) : plane;
  const auto sp = to_global(src + (size_t)(sfield + fld) * fstr);
  const auto vx = to_global(src + fstr);
  const auto ve = vx + fstr;
  const bool rec = qwr != nullptr && !from_cols;  // block-uniform
  const auto wsrc = to_global((rec ? qwr : q) + (size_t)s * 5 * nf);
  const auto wsp = wsrc + (size_t)(sfield + fld) * nf;
  const auto wvx = wsrc + nf;
  const auto wve = wvx + nf;
  const int ctype = s < 4 ? 0 : s - 3;
  const double* cv = T.conv + (size_t)ctype * plane * 6;
  const int lstride = NQ * n, bstride = 3 * lstride;
  const size_t fo = (size_t)fld * field_stride_out;

  // This thread's staged points (l, a) and its outputs (l, m), with their
  // plane-independent tables.
  int sidx[NI], sslot[NI];
  bool sval[NI], oval[NI];
  double c[NI][6];
  int obase_l[NI], omp[NI];
  size_t obase[NI];
  double w[NI][9], ab[NI][2];
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int t = threadIdx.x + it * blockDim.x;
    sval[it] = t < 3 * n;
    oval[it] = sval[it];
    const int tt = sval[it] ? t : 0;
    const int l = colstrip ? tt % 3 + 1 : tt / n + 1;
    const int a = colstrip ? tt / 3 : tt % n;
    const int pidx = strip_index(se, l, a, n);  // point in the sender's plane
    sidx[it] = from_cols ? tt : pidx;            // edge_cols: (a, l) at a * 3 + l - 1
    sslot[it] = (l - 1) * lstride + a;
    if (VEC) {
#pragma unroll
      for (int x = 0; x < 6; ++x) c[it][x] = cv[(size_t)pidx * 6 + x];
    }
    const int lo = (e < 2) ? tt % 3 + 1 : tt / n + 1;  // output layout: l fastest for x ghosts
    const int m = (e < 2) ? tt / 3 : tt % n;
    const int mp = rt.reverse ? n - 1 - m : m;
    obase_l[it] = (lo - 1) * lstride;
    omp[it] = mp;
#pragma unroll
    for (int tp = 0; tp < 9; ++tp) w[it][tp] = T.gw[((size_t)(lo - 1) * n + mp) * 9 + tp];
    if (VEC) {
      const double* abp = T.trans + ((((size_t)s * 4 + se) * 3 + (lo - 1)) * n + mp) * 2;
      ab[it][0] = abp[0];
      ab[it][1] = abp[1];
    }
    obase[it] = (e < 2) ? fo + ((size_t)(P * 2 + e) * nr * n + m) * 3 + (lo - 1)
                        : fo + ((size_t)(P * 2 + (e - 2)) * nr * 3 + (lo - 1)) * n + m;
  }
  const auto gs = to_global(e < 2 ? gxs : gys);
  const auto gv = to_global(e < 2 ? gxv : gyv);

  // source values of one plane, in the storage type until staged
  S pv[NI], xv[NI], yv[NI], pw[NI], xw[NI], yw[NI];
  auto load = [&](int k) {
    const size_t kp = (size_t)k * kstr;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      pv[it] = sp[kp + sidx[it]];
      if (VEC) {
        xv[it] = vx[kp + sidx[it]];
        yv[it] = ve[kp + sidx[it]];
      }
      if (rec) {
        pw[it] = wsp[kp + sidx[it]];
        if (VEC) {
          xw[it] = wvx[kp + sidx[it]];
          yw[it] = wve[kp + sidx[it]];
        }
      }
    }
  };
  load(k0);
  for (int k = k0; k < k1; ++k) {
    double* buf = sline + ((k - k0) & 1) * bstride;
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      if (!sval[it]) continue;
      double* ln = buf + sslot[it];
      double pvd = static_cast<double>(pv[it]);
      if (rec) pvd = pvd + betar * static_cast<double>(pw[it]);
      ln[0] = pvd;
      if (VEC) {
        double x = static_cast<double>(xv[it]), y = static_cast<double>(yv[it]);
        if (rec) {
          x = x + betar * static_cast<double>(xw[it]);
          y = y + betar * static_cast<double>(yw[it]);
        }
        ln[n] = c[it][0] * (c[it][1] * x + c[it][2] * y);
        ln[2 * n] = c[it][3] * (c[it][4] * x + c[it][5] * y);
      }
    }
    load(min(k + 1, k1 - 1));  // past the last plane: loaded and not used
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      if (!oval[it]) continue;
      const double* ln = buf + obase_l[it];
      double ps = 0.0, ths = 0.0, phs = 0.0;
#pragma unroll
      for (int tp = 0; tp < 9; ++tp) {
        const int a = clampi(omp[it] - 4 + tp, 0, n - 1);
        const double wt = w[it][tp];
        ps = ps + ln[a] * wt;
        if (VEC) {
          ths = ths + ln[n + a] * wt;
          phs = phs + ln[2 * n + a] * wt;
        }
      }
      const size_t o = obase[it] + (size_t)k * 3 * n;
      gs[o] = ps;
      if (VEC) gv[o] = ab[it][0] * ths + ab[it][1] * phs;
    }
  }
}

// Planes whose source strips a tile has in LDS at a time (6x32^2x64 step: 114 us
// with two, 116 with one).
constexpr int kGatherPlanes = 2;

// The ghost cells of one stage tile (columns i0.. of wi, rows j0.. of wj) of
// panel P over planes [k0, k1), p' and the velocity across the edge, by
// k_gather's expressions in its order: the same bits.  The tile's threads
// stage the source points of every panel edge the tile's halo crosses -- per
// edge three lines, as far as the nine-point sums reach -- converted to
// (p', theta, phi), for NP planes at a time, and each thread whose halo cell (hi, hj)
// is a ghost (ghost, on edge e) sums its own: ghosts[plane][p', v][thread].
// What bounds it is latency, so the block's weights load before its strips,
// and its radial windows after them (held meanwhile they made the rebuilding
// stage spill: 8.8 -> 13.1 us at 6x16^2x24).  Stage with its ghosts against
// gather and stage, us: 6x16^2x24 7.2 to 8.8 against 4.4 + 5.5 to 7.4;
// 6x32^2x64 14 to 20 against 5.3 + 12 to 18; and a launch less.
//   q, w: the stage's input and, REC, the accumulator it is rebuilt from.
//   strips: NP x 3 x (staged points) doubles.
template <typename S, bool REC, int NP>
__device__ __forceinline__ void gather_tile(const DevTables& T, int P, int i0, int j0, int wi, int wj, int k0, int k1,
                                            const S* __restrict__ q, const S* w, double betar, int tid, int nth,
                                            bool ghost, int e, int hi, int hj, double* ghosts, double* strips) {
  const int n = T.n, nr = T.nr;
  const size_t plane = (size_t)n * n, nf = plane * nr;
  // Per edge the tile's ghosts reach (W, E, S, N): the first along-edge index
  // of its ghosts in the sender's order, and the strip's first point and end
  // in the list of staged points (empty for the others).
  const int routes = T.route_bits[P];
  const bool on[4] = {i0 == 0, i0 + wi + 3 > n, j0 == 0, j0 + wj + 3 > n};
  int first[4], from[4], start[4], D = 0;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const int m0 = x < 2 ? j0 : i0, len = x < 2 ? wj : wi;
    first[x] = routes >> (6 * x) & 32 ? n - m0 - len : m0;
    from[x] = max(first[x] - 4, 0);
    start[x] = D;
    D += on[x] ? 3 * (min(first[x] + len + 4, n) - from[x]) : 0;
  }
  if (D == 0) return;  // block-uniform
  const auto pick = [](const int (&v)[4], int x) { return x == 0 ? v[0] : x == 1 ? v[1] : x == 2 ? v[2] : v[3]; };
  // this thread's ghost cell: its weights, the staged points they apply to, its transform
  double wt[9], ab0 = 0.0, ab1 = 0.0;
  int base = 0, mp = 0;
  if (ghost) {
    const int r = routes >> (6 * e);
    const int lo = e == kW ? -hi - 1 : e == kE ? hi - n : e == kS ? -hj - 1 : hj - n;
    const int m = e < 2 ? hj : hi;
    mp = r & 32 ? n - 1 - m : m;
    base = pick(start, e) + lo - 3 * pick(from, e);
    const double* g = T.gw + ((size_t)lo * n + mp) * 9;
#pragma unroll
    for (int tp = 0; tp < 9; ++tp) wt[tp] = g[tp];
    const double* abp = T.trans + (((size_t)(r & 31) * 3 + lo) * n + mp) * 2;  // [sender][sender edge][l][m]
    ab0 = abp[0];
    ab1 = abp[1];
  }
  for (int kg = k0; kg < k1; kg += NP) {
    if (kg != k0) __syncthreads();  // the strips are read
    for (int t = tid; t < D; t += nth) {
      const int x = (t >= start[1]) + (t >= start[2]) + (t >= start[3]);
      const int u = t - pick(start, x), r = routes >> (6 * x) & 31, sender = r >> 2;
      const int pidx = strip_index(r & 3, u % 3 + 1, pick(from, x) + u / 3, n);
      const double* cv = T.conv + ((size_t)(sender < 4 ? 0 : sender - 3) * plane + pidx) * 6;
      const size_t o = (size_t)sender * 5 * nf + pidx;
      double c[6];
#pragma unroll
      for (int y = 0; y < 6; ++y) c[y] = cv[y];
      S v[NP][3], vw[NP][3];
#pragma unroll
      for (int kk = 0; kk < NP; ++kk) {
        if (kg + kk >= k1) break;
        const size_t ok = o + (size_t)(kg + kk) * plane;
        v[kk][0] = q[ok + 4 * nf];
        v[kk][1] = q[ok + nf];
        v[kk][2] = q[ok + 2 * nf];
        if constexpr (REC) {
          vw[kk][0] = w[ok + 4 * nf];
          vw[kk][1] = w[ok + nf];
          vw[kk][2] = w[ok + 2 * nf];
        }
      }
#pragma unroll
      for (int kk = 0; kk < NP; ++kk) {
        if (kg + kk >= k1) break;
        double d[3];
#pragma unroll
        for (int y = 0; y < 3; ++y) {
          d[y] = static_cast<double>(v[kk][y]);
          if constexpr (REC) d[y] = d[y] + betar * static_cast<double>(vw[kk][y]);
        }
        double* ln = strips + kk * 3 * D + t;
        ln[0] = d[0];
        ln[D] = c[0] * (c[1] * d[1] + c[2] * d[2]);
        ln[2 * D] = c[3] * (c[4] * d[1] + c[5] * d[2]);
      }
    }
    __syncthreads();
    if (ghost) {
#pragma unroll
      for (int kk = 0; kk < NP; ++kk) {
        if (kg + kk >= k1) break;
        const double* ln = strips + kk * 3 * D + base;
        double ps = 0.0, ths = 0.0, phs = 0.0;
#pragma unroll
        for (int tp = 0; tp < 9; ++tp) {
          const int a = 3 * clampi(mp - 4 + tp, 0, n - 1);
          ps = ps + ln[a] * wt[tp];
          ths = ths + ln[D + a] * wt[tp];
          phs = phs + ln[2 * D + a] * wt[tp];
        }
        double* g = ghosts + (kg + kk - k0) * 2 * nth + tid;
        g[0] = ps;
        g[nth] = ab0 * ths + ab1 * phs;
      }
    }
  }
}

// blockIdx.x = (chunk of planes)*24 + (receiver panel P)*4 + (receiver edge e);
// blockIdx.y selects a field offset (the filter's five scalars).
// The FP32-state vector gather at six waves per SIMD (80 registers, a 12-byte
// spill): c3 80 against 97 us.  The FP64 one gained nothing at c3 and lost
// at 6x96^2x192 (28 against 23 us) and keeps the compiler's choice.
template <bool VEC, typename S, int NI>
__global__ __launch_bounds__(gather_threads_max(NI))
__attribute__((amdgpu_waves_per_eu(VEC && NI == 1 && sizeof(S) == 4 ? 6 : 1)))
void k_gather(DevTables T, const S* __restrict__ q,
                                                 const S* __restrict__ ecols, int sfield,
                                                 double* __restrict__ gxs, double* __restrict__ gys,
                                                 double* __restrict__ gxv, double* __restrict__ gyv,
                                                 long long field_stride_out, const S* __restrict__ qwr,
                                                 double betar) {
  extern __shared__ double sline[];
  const int kc = gather_kc(T.nr);
  const int k0 = (blockIdx.x / 24) * kc, edge = blockIdx.x % 24;
  gather_edge<VEC, S, NI>(T, edge / 4, edge % 4, k0, min(k0 + kc, T.nr), blockIdx.y, q, ecols, sfield, gxs, gys,
                          gxv, gyv, field_stride_out, sline, qwr, betar);
}

// Arguments of one stage launch (single grid; an ensemble launch takes the
// tables, buffers and dt from the members M).
template <typename S>
struct StageArgs {
  DevTables T;
  const S* qin;
  S *qout, *qw, *qwo;  // qwo: kStageRecon's qw output
  const double *gxp, *gyp, *gxv, *gyv;
  double alpha, beta, beta_r, dt;
  int kchunk, nkch, rhs_mode;
  int tile_w;  // PART only
  const double* c2f;
  double* divout;
  int div32;
  const double *tl_dc2, *tl_div;
  S* ecols;
  const EnsMember* M;
  const int4* items;
  int nitems, cur, wcur;
  bool gather;    // host only: the stage is to compute its ghost cells if it can,
  bool* gathers;  // or (not null): only say whether it can
};

// Flags of a stage instantiation beyond kStoreNoQ and kStageRecon.
constexpr int kStageRhs = 4;  // evaluates the RHS alone (rhs_mode holds its flags), KIND 0
constexpr int kStageAux = 8;  // c2f or divout is given
// The streams that no other block reads (q and qw stores; rho' and qw loads)
// are non-temporal; kStagePlain: they are not (launch_stage_t; single grids, and
// with a c^2 field or kept divergences only the stored-q variants).  Partial
// tiles load plainly either way: they share 128-byte lines with their neighbours.
constexpr int kStagePlain = 16;
// The stage computes its tiles' ghost cells itself (gather_tile): no gather
// launch before it.  Short chunks of planes only (launch_stage_t).
constexpr int kStageGather = 32;
// One shell (nr == 1), with kStageGather: the radial windows hold one plane
// and the LDS tiles one buffer, so 96 registers and 20 KB where there were 130
// and 40, and the grid is resident at once (us per launch, 6x204^2: first 14.1
// -> 10.1, rebuilding 19.3 -> 12.8; step 104 -> 77).
constexpr int kStageShell = 64;

// Reciprocal-based quotients (div_group) in the FP32-state stages only.
template <typename S>
constexpr bool kStageRcp = sizeof(S) == 4;

// Occupancy floor of the stage kernel in waves per SIMD.  Every variant takes
// 96 to 167 registers and none spills at three; floors of two and four
// measured within 1% of three in every case but one (four, where the divergences
// are kept, makes the rebuilding stage spill: gradient 218 -> 229 ms).  The
// partial tiles' own-ghost stages run at four (below).
constexpr int kStageWaves = 3;
// Four where a partial tile's stage computes its ghost cells (the rebuilding one
// aside): left alone it takes 130 registers, and of blocks of five waves only one
// fits a CU (6x40^2x30: 19 us a stage against 13, which a spill of 12 to 16 bytes
// a lane is in).
constexpr int kGatherWaves = 4;

// One RK stage (or one RHS evaluation, kStageRhs), one pass over HBM.  A
// block owns a TI x TJ column tile of one panel and marches through a chunk
// of radial planes; p' and v_r sit in 7-plane register windows for the radial
// stencils, and the i/j neighbours of plane k come from a double-buffered LDS
// tile, one barrier per plane.
//   KIND 0: first stage (qw taken as 0, written), 1: middle stage (qw read and
//   written), 2: last stage (qw read, not written back).
//   FL: kStoreNoQ (FP64): the stage stores qw (in place) and the
//   edge columns of q, but not q itself.  kStageRecon (KIND 1): the stage
//   input is qin + beta_r * qw, rebuilt wherever it is read (own point, halo
//   cells, radial window) with the expression the previous stage rounded when
//   it computed it, so the same bits; q goes to qout and qw to qwo, a buffer
//   other than qw (other blocks still read qw's halo cells).  kStageRhs,
//   kStageAux: above.
//   MODE 1: ensemble launch.  The block walks a list of work items (member,
//   tile, panel, plane range) with a grid-sized stride; q is read from
//   M.q[cur] and stored to M.q[1-cur], qw is read from M.qw[wcur] and stored
//   there or (kStageRecon) to M.qw[1-wcur].  MODE 2: tangent-linear stage (tl_dc2,
//   tl_div used).
//   ecols (optional; in an ensemble the member's): the stage also stores its
//   output at the edge columns i = 1..3 and n-4..n-2 in the edge_cols layout,
//   for the next gather -- p', v_xi, v_eta after stages 1-4 (the vector
//   gather), all five fields after the last stage (the filter gather).
//   PART: the tiles are tile_w <= TI wide, any width, and need not divide n;
//   the block is one-dimensional.  In the last tile of a row or column the E
//   (N) halo cells begin at the panel edge, inside the tile; threads without a
//   point of their own (beyond the panel, or surplus in the block, part_point)
//   load through an in-panel point, read cells of the LDS tiles and write
//   nothing.
//
// What bounds it.  Memory on large grids: at 6x256^2x384 the five FP64 stages
// move their 640 bytes a point at 4.96 TB/s (first 4.76, rebuilding 4.88, third
// 5.24, last 5.05; 6x128^2x256 4.64, 4.62, 5.11, 5.03).  A march of 10, 15 or 20
// streams with no arithmetic, plane by plane in the same tiles, moves 4.8 (4.9 at
// 6x128^2x256) whatever their number, and one shot over the streams 5.5: the
// march is no ceiling, and what keeps either from 5.5 is not known.  On small
// grids it is the instructions issued per point and plane.  So
//   - every access is a wave-uniform base plus a 32-bit lane offset;
//   - a halo cell is loaded by one thread (y halos by the first waves, x
//     halos by the next, so which of v_xi and v_eta a wave needs is uniform);
//     ghost-strip values load under a wave-uniform branch that only waves at
//     a panel edge take;
//   - a plane's loads come in two groups.  What the plane's start needs (halo
//     cells, v_xi, v_eta, the plane entering the radial windows) is consumed
//     there, and the next plane's values load into the freed registers before
//     the barrier.  What the update at its end needs (rho', qw) loads at the
//     end of the plane before.  Either group is in flight for a whole plane,
//     no register holds a value twice, and none is copied between planes.
// Against six halo loads a thread, a second copy of the plane's registers and
// results held over to the next plane: vector instructions per plane 390 ->
// 298 (first stage), 475 -> 348 (rebuilding), 425 -> 339 (FP32 state);
// registers 234 -> 131 (rebuilding), so three waves per SIMD where there were
// two; us per launch in 32x8 tiles, 6x128^2x256: first 558 -> 462, rebuilding
// 978 -> 902; 6x256^2x384 FP32 state, middle 2866 -> 2661, last 2494 -> 2002.
template <int TI, int TJ, int KIND, typename S, int MODE = 0, bool PART = false, int FL = 0>
__global__ __launch_bounds__(TI* TJ) __attribute__((amdgpu_waves_per_eu(PART && (FL & kStageGather) && !(FL & kStageRecon) ? kGatherWaves : kStageWaves)))
void k_stage(StageArgs<S> A) {
  constexpr bool NOQ = (FL & kStoreNoQ) != 0, RECON = (FL & kStageRecon) != 0;
  constexpr bool STREAM = (FL & kStagePlain) == 0, GATH = (FL & kStageGather) != 0;
  constexpr bool SHELL = (FL & kStageShell) != 0;
  constexpr bool RHS = (FL & kStageRhs) != 0, AUX = (FL & (kStageRhs | kStageAux)) != 0;
  constexpr bool ENS = MODE == 1, TL = MODE == 2, WIDE = sizeof(S) == 8;
  static_assert(!(NOQ || RECON) || (MODE != 2 && WIDE), "the stored-q schedule variants are FP64, not tangent-linear");
  static_assert(!RECON || (KIND == 1 && !NOQ), "a rebuilt input is a middle stage's");
  static_assert(!NOQ || KIND != 2, "the last stage stores q");
  static_assert(!SHELL || GATH, "a shell's chunk is short");
  static_assert(!GATH || (MODE == 0 && !AUX && !STREAM), "own ghost cells: plain stages of one grid");
  static_assert(!RHS || (KIND == 0 && MODE == 0 && !NOQ), "an RHS evaluation is of kind 0");
  // halo cells: 6 rows of TI (y), then TJ rows of 6 (x) from a wave boundary on
  constexpr int NT = TI * TJ, NHC = PART ? 1 : ((6 * TI + 63) / 64 * 64 + 6 * TJ + NT - 1) / NT;
  constexpr int NB = SHELL ? 1 : 2;
  __shared__ double sp[NB][TJ + 6][TI + 6];
  __shared__ double svx[NB][TJ][TI + 6];
  __shared__ double sve[NB][TJ + 6][TI + 6];

  const int W = PART ? A.tile_w : TI, HY = (6 * W + 63) / 64 * 64;
  const int tid = PART ? threadIdx.x : threadIdx.y * TI + threadIdx.x;
  const PartPoint pt = PART ? part_point(tid, W, TJ) : PartPoint{(int)threadIdx.x, (int)threadIdx.y, true};
  const int tx = pt.tx, ty = pt.ty;
  const int wave0 = __builtin_amdgcn_readfirstlane(tid & ~63);  // this wave's first thread

  const int n_items = ENS ? A.nitems : 1;
  for (int item = ENS ? (int)blockIdx.x : 0; item < n_items; item += ENS ? (int)gridDim.x : 1) {
  int bi, bj, P, k0, k1, mem = 0;
  if constexpr (ENS) {
    const auto w = (const __attribute__((address_space(4))) int*)(A.items + item);
    mem = w[0];
    bi = w[1] & 0xffff;
    bj = w[1] >> 16;
    P = w[2] & 0xff;
    k0 = w[2] >> 8;
    k1 = w[3];
  } else {
    const int nti = (A.T.n + W - 1) / W, ntj = (A.T.n + TJ - 1) / TJ;
    int b = xcd_remap(blockIdx.x, nti * ntj * 6 * A.nkch);
    bi = b % nti;
    b /= nti;
    bj = b % ntj;
    b /= ntj;
    P = b % 6;
    k0 = b / 6 * A.kchunk;
    k1 = min(k0 + A.kchunk, A.T.nr);
    if (k0 >= A.T.nr) return;
  }
  // the member's record through the constant address space: scalar loads
  const auto& E = ((const __attribute__((address_space(4))) EnsMember*)A.M)[mem];
  const int n = ENS ? E.T.n : A.T.n, nr = ENS ? E.T.nr : A.T.nr;
  const double dt = ENS ? E.dt : A.dt;
  const CRadialRows rows = const_rows(ENS ? E.T.rad : A.T.rad);
  // antisymmetric taps (checked when the tables are uploaded)
  const double c4 = ENS ? E.T.fcx[4] : A.T.fcx[4], c5 = ENS ? E.T.fcx[5] : A.T.fcx[5],
               c6 = ENS ? E.T.fcx[6] : A.T.fcx[6];
  const int i0 = bi * W, j0 = bj * TJ, i = i0 + tx, j = j0 + ty;
  const int wi = PART ? min(W, n - i0) : TI, wj = PART ? min(TJ, n - j0) : TJ;  // the tile inside the panel
  const bool own_in = !PART || (pt.own && tx < wi && ty < wj);
  const int ic = PART ? min(i, n - 1) : i, jc = PART ? min(j, n - 1) : j;
  const size_t plane = (size_t)n * n, nf = plane * nr;
  const unsigned cell = (unsigned)(jc * n + ic), off = cell * (unsigned)sizeof(S);
  // byte bases of this panel's field 0 and byte strides of fields and planes
  const size_t ps = plane * sizeof(S), fs = nf * sizeof(S), pbase = (size_t)P * 5 * nf;
  const auto bytes = [](const void* p) { return (GlobalBytes)p; };
  const GlobalBytes qb = bytes((ENS ? reinterpret_cast<const S*>(E.q[A.cur]) : A.qin) + pbase);
  const GlobalBytes wb = bytes((ENS ? reinterpret_cast<const S*>(E.qw[A.wcur]) : A.qw) + pbase);
  const GlobalBytes ob = bytes((ENS ? reinterpret_cast<const S*>(E.q[1 - A.cur]) : A.qout) + pbase);
  const GlobalBytes wob = RECON ? bytes((ENS ? reinterpret_cast<const S*>(E.qw[1 - A.wcur]) : A.qwo) + pbase) : wb;
  // edge-column copy: layer l = i (W) or n-1-i (E); the others store none
  const int ecl = i <= 3 ? i : n - 1 - i;
  const S* const ecols = RHS ? nullptr : ENS ? reinterpret_cast<const S*>(E.ecols) : A.ecols;
  const bool ec_on = !RHS && ecols != nullptr && ecl >= 1 && ecl <= 3 && own_in;
  const GlobalBytes ecb = bytes(ecols + (size_t)(P * 2) * nr * edge_cols_plane(n));
  const unsigned ec_off =
      (unsigned)(((i > 3 ? (size_t)nr * edge_cols_plane(n) : 0) + (size_t)j * 3 + (ecl - 1)) * sizeof(S));

  // This thread's halo cells: the offset in a field plane (0, any valid cell,
  // for a ghost or an unused slot), the offset in a plane of the ghost strips,
  // and the LDS cells.
  const size_t gx_side = (size_t)nr * n * 3, gs = (size_t)3 * n * sizeof(double);
  const GlobalBytes gxp = bytes((ENS ? E.gxp : A.gxp) + (size_t)(P * 2) * gx_side);
  const GlobalBytes gyp = bytes((ENS ? E.gyp : A.gyp) + (size_t)(P * 2) * gx_side);
  const GlobalBytes gxv = bytes((ENS ? E.gxv : A.gxv) + (size_t)(P * 2) * gx_side);
  const GlobalBytes gyv = bytes((ENS ? E.gyv : A.gyv) + (size_t)(P * 2) * gx_side);
  unsigned hoff[NHC], goff[NHC];
  int hrow[NHC], hcol[NHC];
  bool hin[NHC], hg[NHC], wave_g[NHC], xh[NHC];
#pragma unroll
  for (int c = 0; c < NHC; ++c) {
    const int h = tid + c * NT;
    xh[c] = wave0 + c * NT >= HY;  // wave-uniform
    int hi, hj;
    if (xh[c]) {
      const int h6 = (h - HY) % 6;
      hrow[c] = (h - HY) / 6 + 3;
      hcol[c] = h6 < 3 ? h6 : wi + h6;
      hin[c] = hrow[c] < wj + 3;
    } else {
      const int r = h / W;
      hrow[c] = r < 3 ? r : wj + r;
      hcol[c] = h % W + 3;
      hin[c] = r < 6 && hcol[c] < wi + 3;
    }
    hi = i0 - 3 + hcol[c];
    hj = j0 - 3 + hrow[c];
    hoff[c] = goff[c] = 0;
    hg[c] = false;
    if (!hin[c]) {
      hrow[c] = hcol[c] = 0;
    } else if (hi < 0 || hi >= n) {
      hg[c] = true;
      goff[c] = (unsigned)((hi < 0 ? hj * 3 - hi - 1 : gx_side + hj * 3 + hi - n) * sizeof(double));
    } else if (hj < 0 || hj >= n) {
      hg[c] = true;
      goff[c] = (unsigned)((hj < 0 ? (-hj - 1) * n + hi : gx_side + (hj - n) * n + hi) * sizeof(double));
    } else {
      hoff[c] = (unsigned)((hj * n + hi) * sizeof(S));
    }
    wave_g[c] = __ballot(hg[c]) != 0;
  }

  // what plane k's start needs, loaded a plane ahead; in the storage type
  // (a conversion at the load would wait for it there)
  S vx_n, ve_n, pn = 0, rn = 0, hp[NHC], hv[NHC];
  double gp[NHC] = {}, gv[NHC] = {};
  S w1_n = 0, w2_n = 0, wpn = 0, wrn = 0, rp[NHC] = {}, rv[NHC] = {};  // RECON: qw at the same points
  auto load_start = [&](int k) {
    const GlobalBytes q = qb + (size_t)k * ps, w = wb + (size_t)k * ps;
    const size_t kn = (size_t)min(k + 3, nr - 1) * ps;  // the plane entering the windows before plane k
#pragma unroll
    for (int c = 0; c < NHC; ++c)
      if (!GATH && wave_g[c]) {
        const size_t kg = (size_t)k * gs;
        const unsigned g = lane_offset(goff[c]);
        gp[c] = load_at<double>((xh[c] ? gxp : gyp) + kg, g);
        gv[c] = load_at<double>((xh[c] ? gxv : gyv) + kg, g);
      }
    const unsigned o = lane_offset(off);
    if constexpr (!SHELL) {
      pn = load_at<S>(qb + kn + 4 * fs, o);
      rn = load_at<S>(qb + kn + 3 * fs, o);
    }
    if constexpr (RECON && !SHELL) {
      wpn = load_at<S>(wb + kn + 4 * fs, o);
      wrn = load_at<S>(wb + kn + 3 * fs, o);
    }
    vx_n = load_at<S>(q + fs, o);
    ve_n = load_at<S>(q + 2 * fs, o);
    if constexpr (RECON) {
      w1_n = load_at<S>(w + fs, o);
      w2_n = load_at<S>(w + 2 * fs, o);
    }
#pragma unroll
    for (int c = 0; c < NHC; ++c) {
      const size_t fv = xh[c] ? fs : 2 * fs;
      const unsigned h = lane_offset(hoff[c]);
      hp[c] = load_at<S>(q + 4 * fs, h);
      hv[c] = load_at<S>(q + fv, h);
      if constexpr (RECON) {
        rp[c] = load_at<S>(w + 4 * fs, h);
        rv[c] = load_at<S>(w + fv, h);
      }
    }
  };
  // what its update needs
  S q1_n, w_n[5] = {};
  double c2_n = 0.0, tdc2 = 0.0, tdiv = 0.0;
  auto load_update = [&](int k) {
    const unsigned o = lane_offset(off);
    const auto get = [&](GlobalBytes p) { return STREAM && !PART ? load_at_nt<S>(p, o) : load_at<S>(p, o); };
    q1_n = get(qb + (size_t)k * ps);
#pragma unroll
    for (int f = 0; f < 5; ++f)
      if (KIND != 0 && !(RECON && (f == 1 || f == 2))) w_n[f] = get(wb + (size_t)k * ps + f * fs);
    const size_t dk = ((size_t)P * nf + (size_t)k * plane) * sizeof(double);
    const unsigned o8 = lane_offset(cell * 8u);
    if (AUX || TL) {
      if (A.c2f) c2_n = load_at<double>(bytes(A.c2f) + dk, o8);
    }
    if constexpr (TL) {
      tdc2 = load_at<double>(bytes(A.tl_dc2) + dk, o8);
      tdiv = load_at<double>(bytes(A.tl_div) + dk, o8);
    }
  };

  load_start(k0);
  double Ci = to_global(ENS ? E.T.ci : A.T.ci)[ic], Dj = to_global(ENS ? E.T.dj : A.T.dj)[jc];
  double dc = to_global(ENS ? E.T.dc : A.T.dc)[cell], tdx = to_global(ENS ? E.T.tdx : A.T.tdx)[cell],
         tde = to_global(ENS ? E.T.tde : A.T.tde)[cell], xy = to_global(ENS ? E.T.xy : A.T.xy)[cell];
  // GATH: the tile's ghost cells first.
  extern __shared__ double ghost_lds[];  // ghost values [plane][p', v][thread], then source strips
  const int nth = PART ? (int)blockDim.x : NT;
  if constexpr (GATH) {
    static_assert(NHC == 1, "one halo cell per thread");
    const int hi = i0 - 3 + hcol[0], hj = j0 - 3 + hrow[0];
    gather_tile<S, RECON, SHELL ? 1 : kGatherPlanes>(A.T, P, i0, j0, wi, wj, k0, k1, A.qin, A.qw, A.beta_r, tid, nth, hg[0],
                          hi < 0 ? kW : hi >= n ? kE : hj < 0 ? kS : kN, hi, hj, ghost_lds,
                          ghost_lds + (size_t)A.kchunk * 2 * nth);
  }
  // Radial windows of p' and v_r over planes kb..kb+6.
  double pw[7], rw[7];
  int kb = clampi(k0 - 3, 0, nr - 7);
  const int q0 = SHELL ? 3 : 0, q1 = SHELL ? 4 : 7;  // a shell: slot 3 holds its plane
#pragma unroll
  for (int q = q0; q < q1; ++q) {  // (nr == 1 otherwise: every slot holds plane 0, with DDR weights 0)
    const size_t kq = (size_t)min(kb + q, nr - 1) * ps;
    pw[q] = load_at<S>(qb + kq + 4 * fs, off);
    rw[q] = load_at<S>(qb + kq + 3 * fs, off);
    if constexpr (RECON) {
      pw[q] = pw[q] + A.beta_r * load_at<S>(wb + kq + 4 * fs, off);
      rw[q] = rw[q] + A.beta_r * load_at<S>(wb + kq + 3 * fs, off);
    }
  }
  const double yCi = 1.0 / Ci, yDj = 1.0 / Dj;  // the divisors fixed for this thread's column
  const bool fdiv = (ENS ? E.T.fast_div : A.T.fast_div) != 0;
  // Everything loaded so far arrives before the loop, so that the waits inside
  // it are those of its own loads.
  asm volatile("" : "+v"(dc), "+v"(tdx), "+v"(tde), "+v"(xy), "+v"(Ci), "+v"(Dj));
#pragma unroll
  for (int q = q0; q < q1; ++q) asm volatile("" : "+v"(pw[q]), "+v"(rw[q]));
  asm volatile("" : "+v"(vx_n), "+v"(ve_n));
  if constexpr (!SHELL) asm volatile("" : "+v"(pn), "+v"(rn));
  if constexpr (RECON) asm volatile("" : "+v"(w1_n), "+v"(w2_n));
  if constexpr (RECON && !SHELL) asm volatile("" : "+v"(wpn), "+v"(wrn));
#pragma unroll
  for (int c = 0; c < NHC; ++c) {
    asm volatile("" : "+v"(hp[c]), "+v"(hv[c]), "+v"(gp[c]), "+v"(gv[c]));
    if constexpr (RECON) asm volatile("" : "+v"(rp[c]), "+v"(rv[c]));
  }
  load_update(k0);

  for (int k = k0; k < k1; ++k) {
    const int want = clampi(k - 3, 0, nr - 7);
    if (!SHELL && want != kb) {  // slides by exactly one plane: plane k+3 enters
#pragma unroll
      for (int q = 0; q < 6; ++q) {
        pw[q] = pw[q + 1];
        rw[q] = rw[q + 1];
      }
      pw[6] = RECON ? pn + A.beta_r * wpn : pn;
      rw[6] = RECON ? rn + A.beta_r * wrn : rn;
      kb = want;
    }
    // p', v_r at plane k: window slot k - kb, 3 on interior planes
    const int wk = k - kb;
    double pc = pw[3], rc = rw[3];
    if (!SHELL && wk != 3) {
      asm volatile("");  // stays a branch
#pragma unroll
      for (int q = 0; q < 7; ++q) {
        pc = wk == q ? pw[q] : pc;
        rc = wk == q ? rw[q] : rc;
      }
    }
    const int bf = SHELL ? 0 : k & 1;
    const double vx = RECON ? vx_n + A.beta_r * w1_n : vx_n;
    const double ve = RECON ? ve_n + A.beta_r * w2_n : ve_n;
    const S w1 = w1_n, w2 = w2_n;  // RECON: used by the update as well
    if (own_in) {
      sp[bf][ty + 3][tx + 3] = pc;
      svx[bf][ty][tx + 3] = vx;
      sve[bf][ty + 3][tx + 3] = ve;
    }
#pragma unroll
    for (int c = 0; c < NHC; ++c) {
      // field halo cells (rebuilt); ghost cells are the gathered stage input
      double p = RECON ? hp[c] + A.beta_r * rp[c] : hp[c];
      double v = RECON ? hv[c] + A.beta_r * rv[c] : hv[c];
      if (wave_g[c]) {
        if constexpr (GATH) {
          gp[c] = ghost_lds[(k - k0) * 2 * nth + tid];
          gv[c] = ghost_lds[((k - k0) * 2 + 1) * nth + tid];
        }
        p = hg[c] ? gp[c] : p;
        v = hg[c] ? gv[c] : v;
      }
      if (hin[c]) {
        sp[bf][hrow[c]][hcol[c]] = p;
        if (xh[c])
          svx[bf][hrow[c] - 3][hcol[c]] = v;
        else
          sve[bf][hrow[c]][hcol[c]] = v;
      }
    }
    if constexpr (!SHELL) load_start(min(k + 1, k1 - 1));  // the last plane's is loaded and not used
    __syncthreads();

    // 7-point DRP stencils, ascending taps from 0 (derivative.f90:137-148,
    // 456-467, 656-668, 704-754).  In xi and eta the coefficients are the
    // same (d_eta = d_xi), antisymmetric, and the centre tap is 0 (checked
    // when the tables are uploaded): its product, +-0 for a finite value,
    // leaves the sum unchanged, so it is not formed.
    const double tap[7] = {-c6, -c5, -c4, 0.0, c4, c5, c6};
    double dvx = 0.0, dve = 0.0, dpx = 0.0, dpe = 0.0, dvr = 0.0, dpr = 0.0;
    // the radial row is block-uniform and read-only: through the constant
    // address space it comes in with scalar loads, which the vector-load
    // waits do not count
    const auto& row = rows[k];
#pragma unroll
    for (int q = 0; q < 7; ++q) {
      if (q != 3) {
        dvx = dvx + tap[q] * svx[bf][ty][tx + q];
        dve = dve + tap[q] * sve[bf][ty + q][tx + 3];
        dpx = dpx + tap[q] * sp[bf][ty + 3][tx + q];
        dpe = dpe + tap[q] * sp[bf][ty + q][tx + 3];
      }
      if (!SHELL || q == 3) {  // (a shell's weights are 0: one product has the value of the seven's sum)
        dvr = dvr + row.w[q] * rw[q];
        dpr = dpr + row.w[q] * pw[q];
      }
    }

    // grad.f90:125-133 and :49-57.
    // quotients by C, D, r and rho0 (grad.f90:52-53, 128-130;
    // compute_rhs_acoustic.f90:88-146), in two groups: the second divides
    // the first's results
    const double q1 = RECON ? q1_n + A.beta_r * w_n[0] : q1_n;
    double qa[7];
    {
      const double na[7] = {dvx, dve, 2.0 * rc, xy * dpe, xy * dpx, dpr, q1 * row.g0};
      const double ba[7] = {Ci, Dj, row.r, Dj, Ci, row.rho0, row.rho0};
      const double ya[7] = {yCi, yDj, row.inv_r, yDj, yCi, row.inv_rho0, row.inv_rho0};
      div_group<kStageRcp<S>>(na, ba, ya, fdiv, own_in, qa);
    }
    const double div = (row.inv_r * ((dc * (qa[0] + qa[1]) - tdx * vx) - tde * ve) + dvr) + qa[2];
    const double gxi = row.inv_r * (Dj * dpx + qa[3]);
    const double get = row.inv_r * (Ci * dpe + qa[4]);

    // compute_rhs_acoustic.f90:38-149 (forcing omitted).
    double r1 = -(row.rho0 * div);
    r1 = r1 - rc * row.drho0dr;
    double qc[2];
    {
      const double nb[2] = {gxi, get};
      const double bb[2] = {row.rho0, row.rho0};
      const double yb[2] = {row.inv_rho0, row.inv_rho0};
      div_group<kStageRcp<S>>(nb, bb, yb, fdiv, own_in, qc);
    }
    double r2 = -qc[0];
    double r3 = -qc[1];
    double r4 = -qa[5];
    r4 = r4 - qa[6];
    // c2f: optional 3-D c^2 (n,n,nr,6); the radial profile otherwise
    double c2rho0 = row.c2rho0;
    if (AUX || TL) {
      if (A.c2f) c2rho0 = c2_n * row.rho0;
    }
    if constexpr (AUX) {
      if (A.divout && own_in) {  // div(v) of the stage input, kept for the adjoint (FP64, or FP32 when div32)
        const size_t dk = (size_t)P * nf + (size_t)k * plane;
        if (A.div32)
          store_at(bytes(A.divout) + dk * 4, cell * 4u, static_cast<float>(div));
        else
          store_at(bytes(A.divout) + dk * 8, cell * 8u, div);
      }
    }
    double r5 = -(c2rho0 * div);
    // tangent-linear run: d r5 / d c^2 = -rho0 div of the primal stage input
    if constexpr (TL) r5 = r5 - (tdc2 * row.rho0) * tdiv;
    r5 = r5 + row.rho0g0 * rc;

    // no BC_RHS and no SPONGE in 2-D (bc_acoustic_wave.f90:11, sponge.f90:18)
    const bool do_bc = (RHS ? (A.rhs_mode & 1) : true) && nr > 1;
    const bool do_sp = (RHS ? (A.rhs_mode & 2) : true) && nr > 1;
    if (do_bc && (k == 0 || k == nr - 1)) {  // bc_acoustic_wave.f90:14-34
      asm volatile("");  // stays a branch
      r1 = 0.0; r2 = 0.0; r3 = 0.0; r4 = 0.0; r5 = 0.0;
    }
    if (do_sp) {  // sponge.f90:48-50, after BC_RHS (timestep.f90:65-66)
      asm volatile("");
      const double sg = row.sigma;
      r1 = r1 - sg * (q1 - 0.0);
      r4 = r4 - sg * (rc - 0.0);
      r5 = r5 - sg * (pc - 0.0);
    }

    const size_t kp = (size_t)k * ps;
    const unsigned o = lane_offset(off);
    if constexpr (RHS) {
      const double r[5] = {r1, r2, r3, r4, r5};
      load_update(min(k + 1, k1 - 1));
      if (own_in) {
#pragma unroll
        for (int f = 0; f < 5; ++f) store_at(ob + kp + f * fs, o, static_cast<S>(r[f]));
      }
    } else {
      // timestep.f90:68-69: qw = alpha*qw + dt*rhs ; q = q + beta*qw
      const double r[5] = {r1, r2, r3, r4, r5}, x[5] = {q1, vx, ve, rc, pc};
      S wn[5], qn[5];
#pragma unroll
      for (int f = 0; f < 5; ++f) {
        const S w = RECON && f == 1 ? w1 : RECON && f == 2 ? w2 : w_n[f];
        const double wd = (KIND == 0 ? 0.0 : A.alpha * w) + dt * r[f];
        qn[f] = static_cast<S>(x[f] + A.beta * wd);
        wn[f] = static_cast<S>(wd);
      }
      if constexpr (!SHELL) load_update(min(k + 1, k1 - 1));
      if (own_in) {
        const auto put = [&](GlobalBytes p, S v) {
          if constexpr (STREAM)
            store_at_nt(p, o, v);
          else
            store_at(p, o, v);
        };
#pragma unroll
        for (int f = 0; f < 5; ++f) {
          if (!NOQ) put(ob + kp + f * fs, qn[f]);
          if (KIND != 2) put(wob + kp + f * fs, wn[f]);
        }
      }
      if (ec_on) {
        const GlobalBytes e = ecb + (size_t)k * edge_cols_plane(n) * sizeof(S);
        const unsigned eo = lane_offset(ec_off);
#pragma unroll
        for (int f = 0; f < 5; ++f)
          if (KIND == 2 || f == 1 || f == 2 || f == 4) store_at(e + (size_t)f * 3 * n * sizeof(S), eo, qn[f]);
      }
    }
    if constexpr (SHELL) break;
  }
  if constexpr (ENS) __syncthreads();  // the next item rewrites the LDS tiles
  }
}

// FILTER_EXP for one field of one panel over a chunk of radial planes.
//   fgx/fgy: ghosts of the unfiltered field (filter.f90:25-28), layouts as in
//   k_gather, 12 sides (6 panels x 2) per field.
// Per plane: the (TJ+6) x (TI+6) tile of the unfiltered field goes to LDS
// (prefetched into registers two planes ahead), FILTER_XI runs on the
// in-panel rows, FILTER_ETA on the result, and FILTER_R accumulates the
// plane's terms into the eleven pending outputs in registers.
template <int TI, int TJ>
struct FilterLds {
  alignas(16) double sq[TJ + 6][TI + 6];  // rows of TI + 6 doubles: 16-byte aligned pairs
  alignas(16) double sx[TJ + 6][TI];
};

// The tile (bi, bj) of field F of panel P (PF = 5P + F) over planes [k0, k1).
// PART: the tile may reach past the panel edge; threads past it store nothing,
// and tile cells beyond the panel's three ghost layers stay 0.
// PAIR: FILTER_XI tasks of two adjacent outputs (below).  R: adjacent rows
// per thread (blocks of TI x TJ / R), whose FILTER_ETA sums share R + 6 reads
// where single rows take 7 each.  SHELL: nr == 1, the 2-D case.
template <int TI, int TJ, typename S, bool PART = false, bool PAIR = (sizeof(S) == 4), int R = 1, bool SHELL = false>
__device__ __forceinline__ void filter_tile(const DevTables& T, int bi, int bj, int PF, int k0, int k1,
                                            const S* __restrict__ qin, S* __restrict__ qout,
                                            const double* __restrict__ fgx, const double* __restrict__ fgy,
                                            FilterLds<TI, TJ>& lds) {
  constexpr int NT = TI * TJ / R;
  constexpr int NCELL = (TJ + 6) * (TI + 6);
  constexpr int NC = (NCELL + NT - 1) / NT;
  static_assert(R == 1 || PAIR, "several rows per thread: paired FILTER_XI tasks");
  auto& sq = lds.sq;
  auto& sx = lds.sx;
  const int n = T.n, nr = T.nr;
  const int P = PF / 5, F = PF % 5;
  const int tx = threadIdx.x, ty = threadIdx.y * R;  // this thread's first row
  const int i0 = bi * TI, j0 = bj * TJ;
  const int i = i0 + tx, j = j0 + ty;
  bool own_in[R];
#pragma unroll
  for (int r = 0; r < R; ++r) own_in[r] = !PART || (i < n && j + r < n);

  const size_t plane = (size_t)n * n, nf = plane * nr;
  const S* g = qin + (size_t)PF * nf;
  S* o = qout + (size_t)PF * nf;
  const size_t gx_side = (size_t)nr * n * 3, gy_side = (size_t)nr * 3 * n;
  const size_t fstride = (size_t)12 * gx_side;
  const double* gxW = fgx + F * fstride + (size_t)(P * 2) * gx_side;
  const double* gyS = fgy + F * fstride + (size_t)(P * 2) * gy_side;
  const size_t ij = own_in[0] ? (size_t)j * n + i : 0;

  // filter.f90:652,726-777: the five planes at each end are zero; in the 2-D
  // case FILTER_R returns its input (filter.f90:647-650).
  if constexpr (!SHELL)
    for (int k = k0; k < k1; ++k)
      if (k < kNstr || k >= nr - kNstr)
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (own_in[r]) o[(size_t)k * plane + ij + (size_t)r * n] = static_cast<S>(0.0);
  const int a = SHELL ? 0 : max(k0, kNstr), bnd = SHELL ? 1 : min(k1, nr - kNstr);
  if (a >= bnd) return;

  // Tile cells this thread fills: kind 1 a field cell, 2 a ghost-strip cell,
  // 0 none.  Field cells load from the plane base (a wave-uniform address)
  // plus a per-lane 32-bit byte offset, so advancing a plane costs no vector
  // instruction; ghost cells (plane stride 3n, uniform too) have per-lane
  // pointers.  Every load is issued unconditionally from a valid address:
  // lanes without a field cell read the plane's first element, lanes without
  // a ghost cell the strip's first element.  Kind-0 cells (the corners beyond
  // the panel in both directions, cells past a partial tile's ghost layers)
  // feed only outputs that are not stored, so they keep whatever was loaded.
  const int tid = threadIdx.y * TI + tx;
  unsigned foff[NC];
  const double* gp[NC];
  int kind[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int e = tid + c * NT;
    kind[c] = 0;
    foff[c] = 0;
    gp[c] = gxW;
    if (e < NCELL) {
      const int rr = e / (TI + 6), cc = e % (TI + 6);
      const int gj = j0 - 3 + rr, gi = i0 - 3 + cc;
      const bool jin = gj >= 0 && gj < n, iin = gi >= 0 && gi < n;
      if (jin && iin) {
        foff[c] = (unsigned)(((size_t)gj * n + gi) * sizeof(S));  // < n*n*sizeof(S)
        kind[c] = 1;
      } else if (jin && gi < n + 3) {  // gi >= -3 always; beyond the E ghosts: none
        gp[c] = (gi < 0) ? gxW + (size_t)gj * 3 + (-gi - 1) : gxW + gx_side + (size_t)gj * 3 + (gi - n);
        kind[c] = 2;
      } else if (iin && gj < n + 3) {
        gp[c] = (gj < 0) ? gyS + (size_t)(-gj - 1) * n + gi : gyS + gy_side + (size_t)(gj - n) * n + gi;
        kind[c] = 2;
      }
    }
  }
  // Two planes in flight in alternating buffers pa / pb: a plane is consumed
  // whole by the LDS write that starts its step, and its buffer is refilled
  // with the plane two ahead right there, so a load has the rest of its step
  // and the whole next step to arrive (no register copies between
  // iterations, which would wait on the loads).  Field cells stay in the
  // storage type in flight (.f) and are widened when they go to LDS, next to
  // the FP64 ghost-strip cells (.g): a conversion at the load would also wait
  // on every load in flight.
  // FP64 state: one value per cell, from the field or (in a wave with ghost
  // cells, by a per-lane address select) from the strip.
  constexpr bool kWide = sizeof(S) == sizeof(double);
  struct FPlaneN {
    double g[NC];
    S f[NC];
  };
  struct FPlaneW {
    double g[NC];
  };
  using FPlane = std::conditional_t<kWide, FPlaneW, FPlaneN>;
  // the ghost-strip load and the select only in waves that hold a ghost cell
  // (a wave-uniform branch; tiles off the panel edges have none)
  bool wave_g[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) wave_g[c] = __ballot(kind[c] == 2) != 0;
  const size_t gstride = (size_t)3 * n;
  // the loads name global memory explicitly (the pointers come from kernel
  // arguments through a select the compiler cannot see through)
  using GD = const __attribute__((address_space(1))) double*;
  using GS = const __attribute__((address_space(1))) S*;
  auto load_plane = [&](int kk, FPlane& dst) {
    const char* fb = reinterpret_cast<const char*>(g + (size_t)kk * plane);  // wave-uniform
    const size_t goff = (size_t)kk * gstride;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if constexpr (kWide) {
        if (wave_g[c]) {
          const double* p = kind[c] == 2 ? gp[c] + goff : reinterpret_cast<const double*>(fb + foff[c]);
          dst.g[c] = *(GD)p;
        } else {
          dst.g[c] = *(GD)(fb + foff[c]);
        }
      } else {
        dst.f[c] = *(GS)(fb + foff[c]);
        dst.g[c] = wave_g[c] ? *(GD)(gp[c] + goff) : 0.0;
      }
    }
  };
  auto widen = [&](const FPlane& L, int c) -> double {
    if constexpr (kWide) {
      return L.g[c];
    } else {
      const double fv = static_cast<double>(L.f[c]);
      if (wave_g[c]) return kind[c] == 2 ? L.g[c] : fv;
      return fv;
    }
  };

  // FILTER_XI on in-panel rows (filter.f90:176-315); rows beyond the panel
  // edge keep the unfiltered ghost, which FILTER_ETA uses (filter.f90:43).
  // The sums start from the first product, not from the reference's 0.0: the
  // two differ only in the sign of a zero result.  A sum's value does not
  // depend on the signs of zero terms, so FILTER_ETA's outputs keep the
  // reference's values (possibly with another zero sign), and the stored
  // sum -- FILTER_R's, or FILTER_ETA's in 2-D, both from 0.0, which never
  // gives -0 -- has the reference's bits.
  // PAIR: a task is two adjacent outputs of one row, read as four aligned
  // 16-byte pairs (eight values for two 7-tap sums), 22 x 16 tasks for a
  // 32 x 16 tile: half the LDS reads of one output per thread (FP32 filter
  // at c3 2.79 -> 2.61 ms).  With one row per thread the FP64 filter takes
  // pairs on panels up to 128 (filter 6x128^2x256 -3%, 6x96^2x192 -7%, the
  // ensemble step -0.8%) and one output per thread on larger ones
  // (6x256^2x384: 2.93 -> 3.14 ms with pairs).
  typedef double dpair __attribute__((ext_vector_type(2)));  // one 16-byte LDS access
  auto xi_pass = [&]() {
    if constexpr (!PAIR) {
      for (int rr = ty; rr < TJ + 6; rr += TJ) {
        const int gj = j0 - 3 + rr;
        double xv;
        if (gj >= 0 && gj < n) {
          xv = T.filt[0] * sq[rr][tx];
#pragma unroll
          for (int q = 1; q < 7; ++q) xv = xv + T.filt[q] * sq[rr][tx + q];
        } else {
          xv = sq[rr][tx + 3];
        }
        sx[rr][tx] = xv;
      }
      return;
    }
    constexpr int NTASK = (TJ + 6) * (TI / 2);
    for (int t = tid; t < NTASK; t += NT) {
      const int rr = t / (TI / 2), c0 = 2 * (t % (TI / 2));
      const dpair* src = reinterpret_cast<const dpair*>(&sq[rr][c0]);
      double v[8];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const dpair d = src[h];
        v[2 * h] = d.x;
        v[2 * h + 1] = d.y;
      }
      const int gj = j0 - 3 + rr;
      double x0, x1;
      if (gj >= 0 && gj < n) {
        x0 = T.filt[0] * v[0];
        x1 = T.filt[0] * v[1];
#pragma unroll
        for (int q = 1; q < 7; ++q) {
          x0 = x0 + T.filt[q] * v[q];
          x1 = x1 + T.filt[q] * v[q + 1];
        }
      } else {
        x0 = v[3];
        x1 = v[4];
      }
      dpair out;
      out.x = x0;
      out.y = x1;
      *reinterpret_cast<dpair*>(&sx[rr][c0]) = out;
    }
  };

  if constexpr (SHELL) {  // the one plane: FILTER_XI, FILTER_ETA, stored as they come
    FPlane p0;
    load_plane(0, p0);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = tid + c * NT;
      if (e < NCELL) (&sq[0][0])[e] = widen(p0, c);
    }
    __syncthreads();
    xi_pass();
    __syncthreads();
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double v = 0.0;  // stored: the reference's sum from 0.0
#pragma unroll
      for (int q = 0; q < 7; ++q) v = v + T.filt[q] * sx[ty + r + q][tx];
      if (own_in[r]) o[ij + (size_t)r * n] = static_cast<S>(v);
    }
    return;
  }

  // FILTER_R (filter.f90:682-693), output plane k = sum over q of
  // filtr[q] * eta(k - 5 + q), summed from 0.0 in q order.  The taps are
  // symmetric (filtr[q] == filtr[10 - q], checked when the tables are
  // uploaded), so each arriving plane's six distinct products feed the eleven
  // pending outputs: acc[d] is output plane kk - 5 + d, which takes the term
  // q = 10 - d of plane kk, the same order and the same products as the
  // sum over a window of the last eleven planes with 6 multiplies instead of 11.
  double acc[R][11];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int q = 0; q < 11; ++q) acc[r][q] = 0.0;

  const int kbeg = a - kNstr, kend = bnd + kNstr;  // kend - kbeg >= 11
  // store: the step completes an output plane (every step from the 11th on)
  auto step = [&](int kk, FPlane& cur, auto store) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int e = tid + c * NT;
      if (e < NCELL) (&sq[0][0])[e] = widen(cur, c);
    }
    load_plane(min(kk + 2, kend - 1), cur);  // past the end: a plane that is loaded and not used
    __syncthreads();
    xi_pass();
    __syncthreads();
    // FILTER_ETA (filter.f90:448-629), from the first product, as FILTER_XI:
    // FILTER_R's sum from 0.0 does not see the sign of a zero input.
    double e[R + 6];  // the column's R + 6 rows
#pragma unroll
    for (int q = 0; q < R + 6; ++q) e[q] = sx[ty + q][tx];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      double v = T.filt[0] * e[r];
#pragma unroll
      for (int q = 1; q < 7; ++q) v = v + T.filt[q] * e[r + q];
      double pr[6];
#pragma unroll
      for (int m = 0; m < 6; ++m) pr[m] = T.filtr[m] * v;
#pragma unroll
      for (int d = 0; d < 10; ++d) acc[r][d] = acc[r][d] + pr[d < 6 ? d : 10 - d];
      acc[r][10] = 0.0 + pr[0];
      if constexpr (decltype(store)::value) {
        if (own_in[r]) o[(size_t)(kk - kNstr) * plane + ij + (size_t)r * n] = static_cast<S>(acc[r][0]);
      }
#pragma unroll
      for (int d = 0; d < 10; ++d) acc[r][d] = acc[r][d + 1];
    }
  };
  // Branch-free memory traffic per iteration (a fixed warm-up, then pairs of
  // storing steps, then at most one more), so the waits before each LDS
  // write leave the other buffer's loads in flight.
  using NoStore = std::integral_constant<bool, false>;
  using Store = std::integral_constant<bool, true>;
  FPlane pa, pb;
  load_plane(kbeg, pa);
  load_plane(kbeg + 1, pb);
  int kk = kbeg;
  for (; kk < kbeg + 2 * kNstr; kk += 2) {  // fill the radial window: planes a-5 .. a+4
    step(kk, pa, NoStore());
    step(kk + 1, pb, NoStore());
  }
  for (; kk + 1 < kend; kk += 2) {
    step(kk, pa, Store());
    step(kk + 1, pb, Store());
  }
  if (kk < kend) step(kk, pa, Store());
}

// Occupancy floor: six waves per SIMD (80 registers), three 512-thread
// blocks per CU.  Left alone, the FP32-state filter takes 84 registers and
// runs five waves, two blocks per CU, which leaves the barriers of each
// plane less to overlap with; at 80 it does not spill (the 32x16 and 16x16
// tiles; the other shapes spill 36 bytes and keep no floor).
// Two rows per thread take 118 registers: four waves (five spill and take
// three times as long).
template <int TI, int TJ, typename S, int R>
constexpr int filter_waves() { return R > 1 ? 4 : (sizeof(S) == 4 && TI * TJ >= 256 && !(TI == 64 && TJ == 4) && !(TI == 32 && TJ == 8)) ? 6 : 1; }

template <int TI, int TJ, typename S, bool PART = false, bool PAIR = (sizeof(S) == 4), int R = 1, bool SHELL = false>
__global__ __launch_bounds__(TI* TJ / R) __attribute__((amdgpu_waves_per_eu(SHELL ? 1 : filter_waves<TI, TJ, S, R>())))
void k_filter(DevTables T, const S* __restrict__ qin,
                                                    S* __restrict__ qout, const double* __restrict__ fgx,
                                                    const double* __restrict__ fgy, int kchunk, int nkch) {
  __shared__ FilterLds<TI, TJ> lds;
  const int n = T.n, nr = T.nr;
  const int nti = (n + TI - 1) / TI, ntj = (n + TJ - 1) / TJ;
  const int nb = nti * ntj * 30 * nkch;
  int b = xcd_remap(blockIdx.x, nb);
  const int bi = b % nti;
  b /= nti;
  const int bj = b % ntj;
  b /= ntj;
  const int PF = b % 30;  // panel*5 + field
  const int ch = b / 30;
  const int k0 = ch * kchunk;
  const int k1 = min(k0 + kchunk, nr);
  if (k0 >= nr) return;
  filter_tile<TI, TJ, S, PART, PAIR, R, SHELL>(T, bi, bj, PF, k0, k1, qin, qout, fgx, fgy, lds);
}

// Ensemble FILTER_EXP: work items (member, tile, 5P+F, plane range), q[cur] -> q[1-cur].
// FILTER_XI in paired tasks (the members are small panels).  Six waves per
// SIMD (80 registers, a 32-byte spill at 32x16): faster than five waves
// without the spill (37.22 against 37.64 ms per 48-member step).
template <int TI, int TJ>
__global__ __launch_bounds__(TI* TJ) __attribute__((amdgpu_waves_per_eu(6))) void k_filter_ens(const EnsMember* __restrict__ M, const int4* __restrict__ items,
                                                        int nitems, int cur) {
  __shared__ FilterLds<TI, TJ> lds;
  for (int item = blockIdx.x; item < nitems; item += gridDim.x) {
    const int4 w = items[item];
    const EnsMember& E = M[w.x];
    filter_tile<TI, TJ, double, false, true>(E.T, w.y & 0xffff, w.y >> 16, w.z & 0xff, w.z >> 8, w.w, E.q[cur], E.q[1 - cur],
                                E.fgx, E.fgy, lds);
    __syncthreads();  // the next item rewrites the LDS tiles
  }
}

// Ensemble gather over a group of members: their blocks laid end to end
// (table[x] = first block of the group's member x, 24 *
// gather_blocks_per_edge(nr, chunks) blocks each; table[nmem + x] = its index
// in M); blockIdx.y selects the field.
template <bool VEC, int NI>
__global__ __launch_bounds__(gather_threads_max(NI)) void k_gather_ens(const EnsMember* __restrict__ M, const int* __restrict__ table,
                                                     int nmem, int cur, int cols, int chunks, int wcur,
                                                     double betar) {
  extern __shared__ double sline[];
  const int b = blockIdx.x;
  int lo = 0, hi = nmem - 1;  // last member whose first block is <= b
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (table[mid] <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  const EnsMember& E = M[table[nmem + lo]];
  const int li = b - table[lo], nr = E.T.nr, kc = gather_kc(nr, chunks);
  const int k0 = (li / 24) * kc, edge = li % 24, k1 = min(k0 + kc, nr);
  const long long fs = 12LL * nr * E.T.n * 3;
  const double* ec = cols ? E.ecols : nullptr;
  const double* qwr = VEC && wcur >= 0 ? E.qw[wcur] : nullptr;
  if (VEC)
    gather_edge<true, double, NI>(E.T, edge / 4, edge % 4, k0, k1, blockIdx.y, E.q[cur], ec, 4, E.gxp, E.gyp,
                                  E.gxv, E.gyv, fs, sline, qwr, betar);
  else
    gather_edge<false, double, NI>(E.T, edge / 4, edge % 4, k0, k1, blockIdx.y, E.q[cur], ec, 0, E.fgx, E.fgy,
                                   nullptr, nullptr, fs, sline, nullptr, 0.0);
}

// Non-finite scan and v_r sum of squares; acc[0] counts non-finite values,
// acc[1] accumulates squares.
template <typename S>
__global__ void k_scan(const S* __restrict__ q, size_t total, size_t nf, double* acc, int mode, int field) {
  double s = 0.0;
  for (size_t x = (size_t)blockIdx.x * blockDim.x + threadIdx.x; x < total; x += (size_t)gridDim.x * blockDim.x) {
    if (mode == 0) {
      const double v = static_cast<double>(q[x]);
      s += (isfinite(v) ? 0.0 : 1.0);
    } else {
      // `field` of panel p
      const size_t p = x / nf, r = x % nf;
      const double v = static_cast<double>(q[(p * 5 + field) * nf + r]);
      s += v * v;
    }
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) atomicAdd(&acc[mode], s);
}

__global__ void k_zero(double* p, int count) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < count) p[t] = 0.0;
}

// Gathers field slots of a staging state buffer into place: dst[(p*5+dfield)]
// <- src[p] for the ghost test entry points.
template <typename S>
__global__ void k_place(const double* __restrict__ src, S* __restrict__ dst, size_t nf, int dfield) {
  const size_t total = nf * 6;
  for (size_t x = (size_t)blockIdx.x * blockDim.x + threadIdx.x; x < total; x += (size_t)gridDim.x * blockDim.x) {
    const size_t p = x / nf, r = x % nf;
    dst[(p * 5 + dfield) * nf + r] = static_cast<S>(src[x]);
  }
}

// ---------------------------------------------------------------- launchers


int chunks_for(int tiles, int nr, int target_blocks, int min_chunk) {
  int nk = (target_blocks + tiles - 1) / tiles;
  const int maxk = nr / min_chunk > 0 ? nr / min_chunk : 1;
  if (nk > maxk) nk = maxk;
  if (nk < 1) nk = 1;
  return nk;
}

// Radial chunks of a march of `tiles` column tiles that does not fill the
// chip: of every split of the nr planes, the one with the least estimated
// time, (rounds of blocks) x (planes per block + warm).  The first rule,
// chunks_for, keeps chunks long, for the bytes that a chunk's window re-reads;
// a small grid lies in the caches and is bound by the serial chain of its
// planes instead (about 1.8 us a plane in the stage kernels, 0.5 in the filter).
//   warm: planes' worth of work before a block's first output;
//   resident: blocks a CU holds; one block alone runs `alone` times as long
//   per plane as its share of a full CU.
int small_grid_chunks(int tiles, int nr, double warm, int resident, double alone) {
  constexpr int kCus = 256;
  int best = 1;
  double least = 0.0;
  for (int nk = 1; nk <= nr; ++nk) {
    const int planes = (nr + nk - 1) / nk;
    if (nk > 1 && planes == (nr + nk - 2) / (nk - 1)) continue;  // the same chunk length in more blocks
    const int blocks = tiles * ((nr + planes - 1) / planes);
    const int slots = kCus * resident, rest = blocks % slots;
    const double rounds =
        blocks / slots * resident + (rest == 0 ? 0.0 : rest <= kCus ? alone : (rest + kCus - 1) / kCus);
    const double t = rounds * (planes + warm);
    if (nk == 1 || t < least) {
      least = t;
      best = nk;
    }
  }
  return best;
}

// Dynamic LDS of one gather launch; above 64 KiB the kernel is allowed it once.
template <typename K>
static hipError_t gather_lds(K kernel, size_t lds) {
  if (lds <= 64 * 1024) return hipSuccess;
  return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(lds));
}

template <bool VEC, typename S, int NI>
static hipError_t launch_gather_v(const DevTables& T, const S* q, const S* ecols, int sfield, int nfields,
                                  double* gxs, double* gys, double* gxv, double* gyv, hipStream_t st, const S* qwr,
                                  double betar) {
  const long long field_stride = 12LL * T.nr * T.n * 3;
  const int kc = gather_kc(T.nr);
  dim3 grid((unsigned)(24 * ((T.nr + kc - 1) / kc)), (unsigned)nfields);
  const int nt = gather_threads(T.n, NI);
  const size_t lds = sizeof(double) * 2 * 3 * (VEC ? 3 : 1) * (size_t)T.n;  // n <= 512: at most 72 KiB
  hipError_t e = gather_lds(&k_gather<VEC, S, NI>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_gather<VEC, S, NI>), grid, dim3(nt), lds, st, T, q, ecols, sfield, gxs, gys, gxv, gyv,
                     field_stride, qwr, betar);
  return hipGetLastError();
}

template <typename S>
static hipError_t launch_gather_t(const DevTables& T, const S* q, const S* ecols, bool vec, int sfield, int nfields,
                                  double* gxs, double* gys, double* gxv, double* gyv, hipStream_t st, const S* qwr,
                                  double betar) {
  const bool two = 3 * T.n > 1024;  // n > 341: two strip points per thread
  if (vec)
    return two ? launch_gather_v<true, S, 2>(T, q, ecols, sfield, nfields, gxs, gys, gxv, gyv, st, qwr, betar)
               : launch_gather_v<true, S, 1>(T, q, ecols, sfield, nfields, gxs, gys, gxv, gyv, st, qwr, betar);
  return two ? launch_gather_v<false, S, 2>(T, q, ecols, sfield, nfields, gxs, gys, gxv, gyv, st, qwr, betar)
             : launch_gather_v<false, S, 1>(T, q, ecols, sfield, nfields, gxs, gys, gxv, gyv, st, qwr, betar);
}

hipError_t launch_gather(const DevTables& T, const void* q, bool f32, bool vec, int sfield, int nfields, double* gxs,
                         double* gys, double* gxv, double* gyv, hipStream_t st, const void* ecols, const void* qwr,
                         double betar) {
  if (f32) {
    if (qwr) return hipErrorInvalidValue;  // rebuilt stage inputs: FP64 storage only
    return launch_gather_t(T, static_cast<const float*>(q), static_cast<const float*>(ecols), vec, sfield, nfields,
                           gxs, gys, gxv, gyv, st, static_cast<const float*>(nullptr), 0.0);
  }
  return launch_gather_t(T, static_cast<const double*>(q), static_cast<const double*>(ecols), vec, sfield, nfields,
                         gxs, gys, gxv, gyv, st, static_cast<const double*>(qwr), betar);
}

// The longest chunk of planes whose ghost cells a stage computes itself: the
// LDS that holds them, and the planes in front of which the block stands
// still, grow with it (us a step, gather launches -> own ghosts: chunks of 1,
// 6x16^2x24 64 -> 54; 4, 6x32^2x64 129 -> 114; 5, 6x32^2x100 173 -> 160; 8,
// FP32 state 6x96^2x16 168 -> 174).
constexpr int kGatherChunk = 6;
// PART: a.tile_w is the tile width (at most TI).
template <int TI, int TJ, typename S, bool PART = false>
static hipError_t launch_stage_t(StageArgs<S> a, int stage, int xf, hipStream_t st, const LaunchShape& ls) {
  const DevTables& T = a.T;
  const int W = PART ? a.tile_w : TI;
  const int tiles = ((T.n + W - 1) / W) * ((T.n + TJ - 1) / TJ) * 6;
  // radial chunks of >= 24 planes, ~12k blocks, at most 8 chunks: 8 chunks measured best at
  // 6x96^2x192 (0.342 ms per stage against 0.375 with 6), 6x128^2x256 and 6x256^2x384
  int nkch = std::min(8, chunks_for(tiles, T.nr, 12288, 24));
  // below two rounds of three blocks a CU the split with the shortest chain
  // (us per stage, before -> after: 6x16^2x24 49 -> 9, 6x32^2x64 71 -> 21,
  // 6x64^2x64 78 -> 51, FP32 state 6x64^2x128 75 -> 58, 6x128^2x128 345 -> 336;
  // at 1728 blocks, 6x96^2x192, 24-plane chunks are still the best: 294
  // against 318 at 20 planes, 308 at 16)
  if (tiles * nkch < 1536) nkch = small_grid_chunks(tiles, T.nr, 1.0, 3, 1.25);
  if (ls.stage_chunks > 0) nkch = ls.stage_chunks;
  // Non-temporal streams, but not where the step's buffers stay in the 256 MB
  // last-level cache between launches (stream_past_cache; the stages without a
  // plain form stay non-temporal there: the last of a step that keeps
  // divergences or has a c^2 field, every FP32-state one with a field), and in partial
  // tiles only where rows and tiles are of whole 64-byte segments: else a
  // neighbouring tile completes the segment in L2 (stage, 6x204^2x100: 1.03 ->
  // 0.95 ms; with whole segments, 6x200^2x150, plain stores are slower: 1.17 ->
  // 1.24 ms; plain loads there: step 7.41 -> 7.18 ms).  A template flag: chosen
  // by a branch in the plane loop it cost the large grids 1 to 2%.
  const bool plain = !stream_past_cache((size_t)30 * T.n * T.n * T.nr * sizeof(S)) ||
                     (PART && (T.n * sizeof(S) % 64 != 0 || W * sizeof(S) % 64 != 0));
  a.nkch = nkch;
  a.kchunk = (T.nr + nkch - 1) / nkch;
  const dim3 grid(tiles * nkch), block = PART ? dim3(part_threads(W, TJ)) : dim3(TI, TJ);
  a.alpha = kAlphaRk4[stage < 0 ? 0 : stage];
  a.beta = kBetaRk4[stage < 0 ? 0 : stage];
  const int kind = stage <= 0 ? 0 : (stage < 4 ? 1 : 2);
#define SOLAR_STAGE_LAUNCH(K, M, FL) hipLaunchKernelGGL((k_stage<TI, TJ, K, S, M, PART, FL>), grid, block, lds, st, a)
  // the variants beyond the plain stages: 64x8, 32x8 and 16x16 tiles
  constexpr bool kMain = (TI == 64 && TJ == 8) || (TI == 32 && TJ == 8) || (TI == 16 && TJ == 16);
  const bool aux = a.c2f || a.divout;
  // Stages with their own ghost cells: short chunks on grids whose streams are
  // plain (there the launch of a gather, 4 to 6 us, is worth more than the
  // edge blocks' extra work), as long as the LDS leaves as many blocks on a CU
  // as registers allow and the grid has (6x64^2x48 FP32 state with one block
  // less: 183 -> 225 us a step).
  const int nti = (T.n + W - 1) / W, ntj = (T.n + TJ - 1) / TJ;
  // (a partial tile one short of the last can reach the last's edge too)
  const size_t strip_points = (nti <= (PART ? 2 : 1) ? 2 : 1) * 3 * (TJ + 8) + (ntj <= (PART ? 2 : 1) ? 2 : 1) * 3 * (W + 8);
  const size_t tile_lds = sizeof(double) * (T.nr == 1 ? 1 : 2) * (2 * (TJ + 6) + TJ) * (TI + 6);
  size_t lds = sizeof(double) * ((size_t)a.kchunk * 2 * block.x * block.y +
                                 (size_t)std::min(a.kchunk, kGatherPlanes) * 3 * strip_points);
  const int waves = (int)(block.x * block.y + 63) / 64;
  const int per_cu = std::max(1, std::min(4 * kStageWaves / waves, (tiles * nkch + 255) / 256));
  const bool gather = kMain && plain && !aux && !a.rhs_mode && !a.tl_dc2 && a.kchunk <= kGatherChunk &&
                      tile_lds + lds <= 64 * 1024 && (tile_lds + lds + 2048) * per_cu <= 160 * 1024;
  if (a.gathers) {
    *a.gathers = gather;
    return hipSuccess;
  }
  if (a.gather && !gather) return hipErrorInvalidValue;
  if (!a.gather) lds = 0;
  if (a.rhs_mode) {
    if (xf || a.tl_dc2 || a.divout) return hipErrorInvalidValue;
    SOLAR_STAGE_LAUNCH(0, 0, kStageRhs);
    return hipGetLastError();
  }
  if constexpr (kMain && sizeof(S) == 8) {
    if (xf) {
      if (a.tl_dc2) return hipErrorInvalidValue;
#define SOLAR_STAGE_XF(FL)                          \
  if (xf == kStoreNoQ && kind == 0)                 \
    SOLAR_STAGE_LAUNCH(0, 0, kStoreNoQ | (FL));     \
  else if (xf == kStoreNoQ && kind == 1)            \
    SOLAR_STAGE_LAUNCH(1, 0, kStoreNoQ | (FL));     \
  else if (xf == kStageRecon && kind == 1 && a.qwo) \
    SOLAR_STAGE_LAUNCH(1, 0, kStageRecon | (FL));   \
  else                                              \
    return hipErrorInvalidValue;
      if (a.gather && T.nr == 1) {
        SOLAR_STAGE_XF(kStageGather | kStagePlain | kStageShell)
      } else if (a.gather) {
        SOLAR_STAGE_XF(kStageGather | kStagePlain)
      } else if (aux && plain) {
        SOLAR_STAGE_XF(kStageAux | kStagePlain)
      } else if (aux) {
        SOLAR_STAGE_XF(kStageAux)
      } else if (plain) {
        SOLAR_STAGE_XF(kStagePlain)
      } else {
        SOLAR_STAGE_XF(0)
      }
#undef SOLAR_STAGE_XF
      return hipGetLastError();
    }
    if constexpr (!PART) {  // the tangent-linear stage: FP64, tiles that divide n
      if (a.tl_dc2) {
        if (kind == 0)
          SOLAR_STAGE_LAUNCH(0, 2, 0);
        else if (kind == 1)
          SOLAR_STAGE_LAUNCH(1, 2, 0);
        else
          SOLAR_STAGE_LAUNCH(2, 2, 0);
        return hipGetLastError();
      }
    }
  }
  if (xf || a.tl_dc2) return hipErrorInvalidValue;
#define SOLAR_STAGE_KIND(FL)      \
  if (kind == 0)                  \
    SOLAR_STAGE_LAUNCH(0, 0, FL); \
  else if (kind == 1)             \
    SOLAR_STAGE_LAUNCH(1, 0, FL); \
  else                            \
    SOLAR_STAGE_LAUNCH(2, 0, FL);
  if constexpr (kMain) {
    if (a.gather && T.nr == 1) {
      SOLAR_STAGE_KIND(kStageGather | kStagePlain | kStageShell)
      return hipGetLastError();
    }
    if (a.gather) {
      SOLAR_STAGE_KIND(kStageGather | kStagePlain)
      return hipGetLastError();
    }
    if (aux) {
      SOLAR_STAGE_KIND(kStageAux)
      return hipGetLastError();
    }
    if (plain) {
      SOLAR_STAGE_KIND(kStagePlain)
      return hipGetLastError();
    }
  }
  if (aux) return hipErrorInvalidValue;
  SOLAR_STAGE_KIND(0)
#undef SOLAR_STAGE_KIND
#undef SOLAR_STAGE_LAUNCH
  return hipGetLastError();
}

// Tile shapes (TI x TJ) compiled for the stage and filter kernels; the
// default is the measured best for the widest TI dividing n.  A requested
// shape that does not divide n falls back to the default.  When no compiled
// shape divides n (n not a multiple of 16), the partial-tile kernels run with
// 32-wide or 16-wide tiles, whichever pads n less (ties to 32).
static bool fits(int n, int ti, int tj) { return ti > 0 && tj > 0 && n % ti == 0 && n % tj == 0; }
static int pad_pick_ti(int n) { return ((n + 31) / 32) * 32 <= ((n + 15) / 16) * 16 ? 32 : 16; }

template <typename S>
static hipError_t launch_stage_s(StageArgs<S> a, int stage, int xf, hipStream_t st, const LaunchShape& ls) {
  const int n = a.T.n;
  if (n % 16 != 0) {
    a.tile_w = part_width(n, a.T.nr);
    return launch_stage_t<64, 8, S, true>(a, stage, xf, st, ls);
  }
  int ti = ls.stage_ti, tj = ls.stage_tj;
  // Measured best (us per stage): 64x8 on panels from 128 (32x8 there:
  // 6x128^2x256 660 -> 705, and the 6x256^2x384 step 24.9 -> 23.7 ms: fewer
  // halo cells), 32x8 on smaller ones that 32 divides (6x64^2x64 52 against 58
  // for 64x8), else 16x16.  The variants of the stored-q schedule, of a c^2
  // field, kept divergences or a tangent-linear run exist for these three.
  const bool plain = !xf && !a.c2f && !a.divout && !a.tl_dc2;
  if (!fits(n, ti, tj) || (!plain && !((ti == 64 && tj == 8) || (ti == 32 && tj == 8) || (ti == 16 && tj == 16)))) {
    ti = n % 64 == 0 && n >= 128 ? 64 : n % 32 == 0 ? 32 : 16;
    tj = ti == 16 ? 16 : 8;
  }
#define SOLAR_STAGE_CASE(X, Y) \
  if (ti == X && tj == Y) return launch_stage_t<X, Y, S>(a, stage, xf, st, ls);
  SOLAR_STAGE_CASE(64, 8)
  SOLAR_STAGE_CASE(64, 4)
  SOLAR_STAGE_CASE(32, 16)
  SOLAR_STAGE_CASE(32, 4)
  SOLAR_STAGE_CASE(32, 8)
#undef SOLAR_STAGE_CASE
  return launch_stage_t<16, 16, S>(a, stage, xf, st, ls);
}

template <typename S>
static StageArgs<S> stage_args(const DevTables& T, const void* qin, void* qout, void* qw, void* qwo, void* ecols) {
  StageArgs<S> a{};
  a.T = T;
  a.qin = static_cast<const S*>(qin);
  a.qout = static_cast<S*>(qout);
  a.qw = static_cast<S*>(qw);
  a.qwo = static_cast<S*>(qwo);
  a.ecols = static_cast<S*>(ecols);
  return a;
}

bool stage_gathers(const DevTables& T, bool f32, int stage, int xf, const LaunchShape& ls, const double* c2f,
                   const double* divout, const double* tl_dc2) {
  bool yes = false;
  auto ask = [&](auto a) {
    a.c2f = c2f;
    a.divout = const_cast<double*>(divout);
    a.tl_dc2 = tl_dc2;
    a.gathers = &yes;
    (void)launch_stage_s(a, stage, xf, nullptr, ls);
  };
  if (f32)
    ask(stage_args<float>(T, nullptr, nullptr, nullptr, nullptr, nullptr));
  else
    ask(stage_args<double>(T, nullptr, nullptr, nullptr, nullptr, nullptr));
  return yes;
}

hipError_t launch_stage(const DevTables& T, const void* qin, void* qout, void* qw, bool f32, const double* gxp,
                        const double* gyp, const double* gxv, const double* gyv, int stage, double dt, int rhs_mode,
                        hipStream_t st, const LaunchShape& ls, const double* c2f, double* divout, int div32,
                        const double* tl_dc2, const double* tl_div, void* ecols, int xf, void* qwo, double beta_r,
                        bool gather) {
  auto go = [&](auto a) {
    a.gxp = gxp;
    a.gyp = gyp;
    a.gxv = gxv;
    a.gyv = gyv;
    a.beta_r = beta_r;
    a.dt = dt;
    a.rhs_mode = rhs_mode;
    a.c2f = c2f;
    a.divout = divout;
    a.div32 = div32;
    a.tl_dc2 = tl_dc2;
    a.tl_div = tl_div;
    a.gather = gather;
    return launch_stage_s(a, stage, xf, st, ls);
  };
  // (the stored-q schedule variants and the tangent-linear stage are FP64: launch_stage_t refuses others)
  return f32 ? go(stage_args<float>(T, qin, qout, qw, qwo, ecols)) : go(stage_args<double>(T, qin, qout, qw, qwo, ecols));
}

template <int TI, int TJ, typename S, bool PART = false, bool PAIR = (sizeof(S) == 4), int R = 1, bool SHELL = false>
static hipError_t launch_filter_t(const DevTables& T, const S* qin, S* qout, const double* fgx, const double* fgy,
                                  hipStream_t st, const LaunchShape& ls) {
  const int tiles = ((T.n + TI - 1) / TI) * ((T.n + TJ - 1) / TJ) * 30;
  // radial chunks of >= 64 planes (each re-reads 10 halo planes), ~4k blocks: a single chunk per
  // column at 6x256^2x384 leaves a long tail (3.45 ms against 2.96 ms with two)
  int nkch = R > 1 ? small_grid_chunks(tiles, T.nr, 2.0 * kNstr, 2, 1.5) : chunks_for(tiles, T.nr, 4096, 64);
  // a chunk re-reads ten planes, so a small grid is split less far than the
  // stages (us, before -> after: 6x16^2x96 55 -> 16, 6x32^2x64 48 -> 25,
  // 6x48^2x100 66 -> 44; from 1620 blocks on, 6x96^2x192, all splits into
  // 32 to 96 planes measured within 2%)
  if (R == 1 && tiles * nkch < 1536) nkch = small_grid_chunks(tiles, T.nr, 2.0 * kNstr, 1, 1.5);
  if (ls.filter_chunks > 0) nkch = ls.filter_chunks;
  const int kchunk = (T.nr + nkch - 1) / nkch;
  dim3 grid(tiles * nkch), block(TI, TJ / R);
  hipLaunchKernelGGL((k_filter<TI, TJ, S, PART, PAIR, R, SHELL>), grid, block, 0, st, T, qin, qout, fgx, fgy, kchunk, nkch);
  return hipGetLastError();
}

template <typename S>
static hipError_t launch_filter_s(const DevTables& T, const S* qin, S* qout, const double* fgx, const double* fgy,
                                  hipStream_t st, const LaunchShape& ls) {
  // FILTER_XI in paired tasks: always for an FP32 state, for FP64 on panels up to 128
  const bool pair = sizeof(S) == 4 || T.n <= 128;
  // One shell: no radial sums, so 28 registers instead of 76 and eight waves
  // per SIMD; the smallest tiles fill the chip best (us, 6x204^2: 15.8 -> 13.6,
  // 32 wide 14.9, 64 wide 17.9; 6x300^2 26.2 -> 21.5; 6x512^2 52.3 -> 48.3).
  if (T.nr == 1)
    return T.n % 16 ? launch_filter_t<16, 16, S, true, true, 1, true>(T, qin, qout, fgx, fgy, st, ls)
                    : launch_filter_t<16, 16, S, false, true, 1, true>(T, qin, qout, fgx, fgy, st, ls);
  if (T.n % 16 != 0) {  // partial tiles
    if (pad_pick_ti(T.n) == 32)
      return pair ? launch_filter_t<32, 16, S, true, true>(T, qin, qout, fgx, fgy, st, ls)
                  : launch_filter_t<32, 16, S, true, false>(T, qin, qout, fgx, fgy, st, ls);
    return pair ? launch_filter_t<16, 16, S, true, true>(T, qin, qout, fgx, fgy, st, ls)
                : launch_filter_t<16, 16, S, true, false>(T, qin, qout, fgx, fgy, st, ls);
  }
  int ti = ls.filter_ti, tj = ls.filter_tj;
  // FP64 on panels from 128: 64x16 tiles with two rows a thread.  Fewer halo
  // cells (1.50 tile cells a point against 1.63, and whole lines of them) and
  // LDS reads: 6x256^2x384 2.94 -> 2.58 ms, 6x128^2x256 489 -> 456 us.  The
  // FP32-state filter is bound by its FP64 arithmetic instead and keeps one
  // row (6x256^2x384 2.28 against 2.40 ms); so do smaller panels (6x64^2x128
  // 73.2 against 72.2 us).
  if constexpr (sizeof(S) == 8) {
    if (T.n % 64 == 0 && T.n >= 128 && !fits(T.n, ti, tj))
      return launch_filter_t<64, 16, S, false, true, 2>(T, qin, qout, fgx, fgy, st, ls);
  }
  if (!fits(T.n, ti, tj)) {  // measured best: 32x16 (n%32==0), 16x16
    ti = T.n % 32 == 0 ? 32 : 16;
    tj = 16;
  }
  if (pair && ti == 32 && tj == 16) return launch_filter_t<32, 16, S, false, true>(T, qin, qout, fgx, fgy, st, ls);
  if (pair && ti == 16 && tj == 16) return launch_filter_t<16, 16, S, false, true>(T, qin, qout, fgx, fgy, st, ls);
#define SOLAR_FILTER_CASE(A, B) \
  if (ti == A && tj == B) return launch_filter_t<A, B, S>(T, qin, qout, fgx, fgy, st, ls);
  SOLAR_FILTER_CASE(32, 16)
  SOLAR_FILTER_CASE(16, 16)
  SOLAR_FILTER_CASE(64, 4)
  SOLAR_FILTER_CASE(32, 8)
  SOLAR_FILTER_CASE(64, 8)
  SOLAR_FILTER_CASE(64, 16)
#undef SOLAR_FILTER_CASE
  if (T.n % 32 == 0)
    return pair ? launch_filter_t<32, 16, S, false, true>(T, qin, qout, fgx, fgy, st, ls)
                : launch_filter_t<32, 16, S>(T, qin, qout, fgx, fgy, st, ls);
  return pair ? launch_filter_t<16, 16, S, false, true>(T, qin, qout, fgx, fgy, st, ls)
              : launch_filter_t<16, 16, S>(T, qin, qout, fgx, fgy, st, ls);
}

hipError_t launch_filter(const DevTables& T, const void* qin, void* qout, bool f32, const double* fgx,
                         const double* fgy, hipStream_t st, const LaunchShape& ls) {
  if (f32)
    return launch_filter_s(T, static_cast<const float*>(qin), static_cast<float*>(qout), fgx, fgy, st, ls);
  return launch_filter_s(T, static_cast<const double*>(qin), static_cast<double*>(qout), fgx, fgy, st, ls);
}

hipError_t launch_scan(const void* q, bool f32, size_t nf, double* acc, int mode, hipStream_t st, int field) {
  if (field < 0 || field > 4) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_zero, dim3(1), dim3(64), 0, st, acc, 2);
  const size_t total = mode == 0 ? nf * 30 : nf * 6;
  if (f32)
    hipLaunchKernelGGL(k_scan<float>, dim3(1024), dim3(256), 0, st, static_cast<const float*>(q), total, nf, acc, mode,
                       field);
  else
    hipLaunchKernelGGL(k_scan<double>, dim3(1024), dim3(256), 0, st, static_cast<const double*>(q), total, nf, acc,
                       mode, field);
  return hipGetLastError();
}

hipError_t launch_place(const double* src, void* dst, bool f32, size_t nf, int dfield, hipStream_t st) {
  if (f32)
    hipLaunchKernelGGL(k_place<float>, dim3(1024), dim3(256), 0, st, src, static_cast<float*>(dst), nf, dfield);
  else
    hipLaunchKernelGGL(k_place<double>, dim3(1024), dim3(256), 0, st, src, static_cast<double*>(dst), nf, dfield);
  return hipGetLastError();
}

// ---------------------------------------------------------------- ensembles

template <int TI, int TJ>
static hipError_t launch_stage_ens_t(const EnsMember* M, const int4* items, int nitems, int grid, int stage, int cur,
                                     int wcur, bool stored_q, hipStream_t st) {
  StageArgs<double> a{};
  a.alpha = kAlphaRk4[stage];
  a.beta = kBetaRk4[stage];
  a.beta_r = stage > 0 ? kBetaRk4[stage - 1] : 0.0;
  a.M = M;
  a.items = items;
  a.nitems = nitems;
  a.cur = cur;
  a.wcur = wcur;
  const dim3 g(grid), block(TI, TJ);
  if (!stored_q && stage == 0)
    hipLaunchKernelGGL((k_stage<TI, TJ, 0, double, 1>), g, block, 0, st, a);
  else if (!stored_q && stage < 4)
    hipLaunchKernelGGL((k_stage<TI, TJ, 1, double, 1>), g, block, 0, st, a);
  else if (stage == 0)
    hipLaunchKernelGGL((k_stage<TI, TJ, 0, double, 1, false, kStoreNoQ>), g, block, 0, st, a);
  else if (stage == 2)
    hipLaunchKernelGGL((k_stage<TI, TJ, 1, double, 1, false, kStoreNoQ>), g, block, 0, st, a);
  else if (stage < 4)
    hipLaunchKernelGGL((k_stage<TI, TJ, 1, double, 1, false, kStageRecon>), g, block, 0, st, a);
  else
    hipLaunchKernelGGL((k_stage<TI, TJ, 2, double, 1>), g, block, 0, st, a);
  return hipGetLastError();
}

hipError_t launch_stage_ens(const EnsMember* M, const int* items, int nitems, int grid, int ti, int tj, int stage,
                            int cur, int wcur, bool stored_q, hipStream_t st) {
  const int4* it = reinterpret_cast<const int4*>(items);
  if (nitems <= 0) return hipSuccess;
  if (stage < 0 || stage > 4) return hipErrorInvalidValue;
  if (ti == 64 && tj == 8) return launch_stage_ens_t<64, 8>(M, it, nitems, grid, stage, cur, wcur, stored_q, st);
  if (ti == 32 && tj == 8) return launch_stage_ens_t<32, 8>(M, it, nitems, grid, stage, cur, wcur, stored_q, st);
  if (ti == 16 && tj == 16) return launch_stage_ens_t<16, 16>(M, it, nitems, grid, stage, cur, wcur, stored_q, st);
  return hipErrorInvalidValue;
}

hipError_t launch_filter_ens(const EnsMember* M, const int* items, int nitems, int grid, int ti, int tj, int cur,
                             hipStream_t st) {
  const int4* it = reinterpret_cast<const int4*>(items);
  if (nitems <= 0) return hipSuccess;
  if (ti == 32 && tj == 16)
    hipLaunchKernelGGL((k_filter_ens<32, 16>), dim3(grid), dim3(32, 16), 0, st, M, it, nitems, cur);
  else if (ti == 16 && tj == 16)
    hipLaunchKernelGGL((k_filter_ens<16, 16>), dim3(grid), dim3(16, 16), 0, st, M, it, nitems, cur);
  else if (ti == 32 && tj == 8)
    hipLaunchKernelGGL((k_filter_ens<32, 8>), dim3(grid), dim3(32, 8), 0, st, M, it, nitems, cur);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

template <bool VEC, int NI>
static hipError_t launch_gather_ens_v(const EnsMember* M, const int* table, int nmem, int nblocks, int maxn, int cur,
                                      int cols, int chunks, hipStream_t st, int wcur, double betar) {
  const int nt = gather_threads(maxn, NI);
  const size_t lds = sizeof(double) * 2 * 3 * (VEC ? 3 : 1) * (size_t)maxn;
  hipError_t e = gather_lds(&k_gather_ens<VEC, NI>, lds);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((k_gather_ens<VEC, NI>), dim3(nblocks, VEC ? 1 : 5), dim3(nt), lds, st, M, table, nmem, cur,
                     cols, chunks, wcur, betar);
  return hipGetLastError();
}

hipError_t launch_gather_ens(const EnsMember* M, const int* table, int nmem, int nblocks, int maxn, bool vec, int cur,
                             bool cols, int chunks, hipStream_t st, int wcur, double betar) {
  const bool two = 3 * maxn > 1024;  // n > 341: two strip points per thread
  const int c = cols ? 1 : 0;
  if (chunks < 1) return hipErrorInvalidValue;
  if (vec)
    return two ? launch_gather_ens_v<true, 2>(M, table, nmem, nblocks, maxn, cur, c, chunks, st, wcur, betar)
               : launch_gather_ens_v<true, 1>(M, table, nmem, nblocks, maxn, cur, c, chunks, st, wcur, betar);
  return two ? launch_gather_ens_v<false, 2>(M, table, nmem, nblocks, maxn, cur, c, chunks, st, wcur, betar)
             : launch_gather_ens_v<false, 1>(M, table, nmem, nblocks, maxn, cur, c, chunks, st, wcur, betar);
}

}  // namespace solar
