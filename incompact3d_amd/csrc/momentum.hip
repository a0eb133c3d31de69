// Fused momentum right-hand side of transeq.f90:73-470 along periodic
// directions (bounded.hip holds the sweeps along bounded ones).
//
// One launch per sweep direction d computes for each velocity component c
// the three compact solves the reference does for that pair
//     D1_d(u_d u_c)   (transeq.f90:125/198/259)
//     D1_d(u_c)       (transeq.f90:128/201/262)
//     D2_d(u_c)       (transeq.f90:301/336/442)
// and accumulates  -1/2 D1_d(u_d u_c) - 1/2 u_d D1_d(u_c) + nu D2_d(u_c)
// into the running right-hand side, so each (d, c) pair moves four fields
// through HBM (u_d, u_c, the accumulator in, the accumulator out) instead of
// ten.  Each input window is read once; the three solves (two on the
// first-derivative matrix, one on the second-derivative matrix) run between
// one set of block barriers.  The x sweep, the last one in the
// reference's order, also applies AB3 (time_integrators.f90:85-100): the new
// velocity goes to a second buffer, because the other components still read
// the old one.  With FP32 compute the FP64 velocity is not touched here: the
// sweep writes the step's increment in FP32 and the new FP32 velocity, and the
// gradient correction adds the increment to the FP64 velocity, so that the
// FP64 state is read and written once per step.
#include <algorithm>
#include <cmath>
#include <vector>

#include "bounded_impl.h"

namespace x3d {

template <typename T>
struct MomArgs {
  // the component of blockIdx.z: the velocity along the sweep, and per
  // component u_c, the running right-hand side in (null: none) and out
  const T *ud;
  const T *uc[3], *acc[3];
  T *out[3];
  const T *pk1, *pk2;           // packed first/second-derivative sets
  T alfa1, den1, alfa2, den2;
  T rden1, rden2;               // 1 / den
  Sten<T> s;
  T xnu;
  int n, na, nb;
  long long sa, sb, se;         // line strides (y/z sweeps)
  int kdepth;                   // carry-chain depth in segments (y/z sweeps)
  // AB3 epilogue (x sweep only), du = ca*f1 + cb*f2 + cc*f3 in FP64:
  //   FP64: u_new = du + u_c
  //   FP32: delta = du, shadow = du + u_c (the FP64 velocity adds delta later)
  const T *f2[3], *f3[3];
  double *u_new[3];
  float *delta[3];
  float *shadow[3];
  double ca, cb, cc;
  int nterms;                   // 0: no AB3
  MomUpdate<T> up;              // x sweep of the general step
};

// ---------------------------------------------------------------- y / z sweeps
// Three components to a launch.  256^3 FP64: 292 (y) and 278 us (z), 5.1 and 3.9
// TB/s of the fields it moves; with the fields end to end (solver.hip) 312 and
// 282, without the solves then 315 and 260, loads alone 135 and 165, stores
// alone 75: bound by strided reads and writes in turn.  FP32 150 and 128 us, the
// vector ALU busy for 69 and 83 % of them.
template <typename T, int L>
__global__ void __launch_bounds__(1024) mom_yz_kernel(const MomArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = blockDim.y;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int n = A.n;
  // LDS: two coefficient tables, carries of three right-hand sides
  T *cs1 = smem, *cs2 = cs1 + 4 * n, *cf = cs2 + 4 * n, *cb = cf + 3 * P * TL;
  T *gf = cb + 3 * P * TL, *gb = gf + 2 * P, *x0s = gb + 2 * P, *xns = x0s + 3 * TL;
  int bx, b;
  block_coords<sizeof(T) == 4>(bx, b);
  const int comp = (int)blockIdx.z;
  const T *const uc = A.uc[comp];
  const T *const acc = A.acc[comp];
  T *const out = A.out[comp];
  const int a = bx * TL + line;
  const bool active = a < A.na;
  // lines past the end compute on a copy of the last line (no load branches)
  const int al = active ? a : A.na - 1;
  const int e0 = seg * L;        // n = P*L: every segment is full
  // byte offsets in 32 bits (the host checks the field size), so each load is
  // a uniform base plus one VGPR offset
  const unsigned base = ((unsigned)al * (unsigned)A.sa + (unsigned)b * (unsigned)A.sb) * (unsigned)sizeof(T);
  const unsigned step = (unsigned)A.se * (unsigned)sizeof(T);
  // windows reach at most 4 points past either end of the line (n >= 8)
  auto wrap = [&](int j) { return (unsigned)(j < 0 ? j + n : (j >= n ? j - n : j)); };
  // right-hand sides: w[0] of D1(u_d u_c), w[1] of D1(u_c) (first-derivative
  // matrix), w[2] of D2(u_c) (second-derivative matrix); u_c is read over
  // [e0-4, e0+L+4), u_d over [e0-2, e0+L+2), each once, before the
  // coefficient copy and its barrier
  __builtin_amdgcn_s_setprio(3);   // issue this block's loads ahead of other blocks' arithmetic
  TableCopy<T, 2> tc;
  tc.load(A.pk1, A.pk2, tid, nthr, 4 * n);
  T w[3][L], ud[L];
  {
    T wc[L + 8];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) wc[k] = at(uc, base + wrap(e0 - 4 + k) * step);
    {
      T p[L + 4];
#pragma unroll
      for (int k = 0; k < L + 4; ++k) {
        const T d = at(A.ud, base + wrap(e0 - 2 + k) * step);
        p[k] = d * wc[k + 2];
        if (k >= 2 && k < L + 2) ud[k - 2] = d;
      }
#pragma unroll
      for (int m = 0; m < L; ++m) w[0][m] = interior_row<OP_DER1, T, L + 4>(p, m + 2, A.s);
    }
#pragma unroll
    for (int m = 0; m < L; ++m) {
      w[1][m] = interior_row<OP_DER1, T, L + 8>(wc, m + 4, A.s);
      w[2][m] = interior_row<OP_DER2, T, L + 8>(wc, m + 4, A.s);
    }
  }
  __builtin_amdgcn_s_setprio(0);   // back to normal priority once the loads are out
  tc.store(cs1, cs2, A.pk1, A.pk2, tid, nthr, 4 * n);
  __syncthreads();
  seg_solve<T, L, 3, 2>(w, e0, cs1, A.alfa1, A.rden1, cs2, A.alfa2, A.rden2, cf, cb, gf, gb, x0s, xns, line, seg,
                        TL, P, A.kdepth);
  if (!active) return;
  // -1/2 D1(u_d u_c) - 1/2 u_d D1(u_c) + nu D2(u_c)
#pragma unroll
  for (int m = 0; m < L; ++m) w[0][m] = T(-0.5) * w[0][m] + T(-0.5) * (ud[m] * w[1][m]) + A.xnu * w[2][m];
  if (acc) {
    // acc may be out (in-place accumulation): all of this thread's acc
    // points are read before any is written
    T ac[L];
#pragma unroll
    for (int m = 0; m < L; ++m) ac[m] = at(acc, base + (unsigned)(e0 + m) * step);
#pragma unroll
    for (int m = 0; m < L; ++m) at(out, base + (unsigned)(e0 + m) * step) = ac[m] + w[0][m];
  } else {
#pragma unroll
    for (int m = 0; m < L; ++m) at(out, base + (unsigned)(e0 + m) * step) = w[0][m];
  }
}

// ---------------------------------------------------------------- one line on one wavefront
// The two coefficient sets of a line, V points per lane (lane k owns points
// kV .. kV+V-1), held in registers.
template <typename T, int V>
struct LineCoef {
  T fs1[V], fw1[V], ffw1[V], sm1[V], fs2[V], fw2[V], ffw2[V], sm2[V];
  __device__ __forceinline__ void load(const MomArgs<T> &A, const int lane) {
#pragma unroll
    for (int m = 0; m < V; ++m) {
      const int e = lane * V + m;
      fs1[m] = A.pk1[4 * e]; fw1[m] = A.pk1[4 * e + 1]; ffw1[m] = A.pk1[4 * e + 2]; sm1[m] = A.pk1[4 * e + 3];
      fs2[m] = A.pk2[4 * e]; fw2[m] = A.pk2[4 * e + 1]; ffw2[m] = A.pk2[4 * e + 2]; sm2[m] = A.pk2[4 * e + 3];
    }
  }
};

// -1/2 D1(u_d u_c) - 1/2 u_d D1(u_c) + nu D2(u_c) of one periodic line held
// by a wavefront: the halos come from the neighbour lanes (DPP), the three
// solves are wave_solve's lane-parallel Thomas sweeps.
template <typename T, int V>
__device__ __forceinline__ void mom_line(const MomArgs<T> &A, const LineCoef<T, V> &C, const T (&ud)[V],
                                         const T (&uc)[V], T (&r)[V], const int lane) {
  {
    T p[V];
#pragma unroll
    for (int m = 0; m < V; ++m) p[m] = ud[m] * uc[m];
    T v[V + 4];
    halo_window<T, V, 2, 2>(p, v, lane);
    T w[V];
#pragma unroll
    for (int m = 0; m < V; ++m) w[m] = A.s.afi * (v[m + 3] - v[m + 1]) + A.s.bfi * (v[m + 4] - v[m]);
    wave_solve<T, V>(w, C.fs1, C.fw1, C.ffw1, C.sm1, A.alfa1, A.rden1, lane);
#pragma unroll
    for (int m = 0; m < V; ++m) r[m] = T(-0.5) * w[m];
  }
  {
    T v[V + 4];
    halo_window<T, V, 2, 2>(uc, v, lane);
    T w[V];
#pragma unroll
    for (int m = 0; m < V; ++m) w[m] = A.s.afi * (v[m + 3] - v[m + 1]) + A.s.bfi * (v[m + 4] - v[m]);
    wave_solve<T, V>(w, C.fs1, C.fw1, C.ffw1, C.sm1, A.alfa1, A.rden1, lane);
#pragma unroll
    for (int m = 0; m < V; ++m) r[m] += T(-0.5) * (ud[m] * w[m]);
  }
  {
    T v[V + 8];
    halo_window<T, V, 4, 4>(uc, v, lane);
    T w[V];
#pragma unroll
    for (int m = 0; m < V; ++m) w[m] = interior_row<OP_DER2, T, V + 8>(v, m + 4, A.s);
    wave_solve<T, V>(w, C.fs2, C.fw2, C.ffw2, C.sm2, A.alfa2, A.rden2, lane);
#pragma unroll
    for (int m = 0; m < V; ++m) r[m] += A.xnu * w[m];
  }
}

// ---------------------------------------------------------------- x sweep (one wavefront per line)
// GEN: the general velocity update (RK3, bounded y or z) in place of plain AB3.
// ALL: a wavefront takes the three components of a line one after another, else
// that of blockIdx.z.  Bound by memory, 18 fields in all (20 with u_x read for
// each component): 256^3 FP64 494 -> 441 us (5.5 TB/s), FP32 283 -> 251, the
// channel's 256x129x128 FP64 133 -> 110.
template <typename T, int V, bool GEN, bool ALL>
__global__ void __launch_bounds__(256) mom_x_kernel(const MomArgs<T> A, int nlines) {
  const int lane = threadIdx.x & 63;
  const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
  const int nwaves = (gridDim.x * blockDim.x) >> 6;
  const int n = A.n;
  LineCoef<T, V> C;
  C.load(A, lane);
  // the next velocities (u_x of the next line last) are loaded before this
  // component is solved, so that their latency overlaps the solves (each wave
  // loops over several lines)
  // memory order in 16 bytes of the widest type; FP32 keeps run order, 16 or 32
  // bytes a lane (512^3: 2050 us against 2300)
  constexpr int PER = sizeof(T) == 4 && !GEN ? V : (V == 1 ? 1 : 2);
  using Tile = LineTile<T, V, PER>;
  __shared__ __align__(16) T lines[4 * Tile::WORDS];
  const Tile tile(lines);
  T ud[V], uc[V], um[V], nx[V], nd[V];   // run order; um (u_c), nx, nd: memory order
  const int c0 = ALL ? 0 : (int)blockIdx.z, c1 = ALL ? 3 : c0 + 1;
  if (wave < nlines) {
    tile.load(A.ud + (long long)wave * n, nd);
    if constexpr (!ALL) tile.load(A.uc[c0] + (long long)wave * n, nx);
  }
  for (int ln = wave; ln < nlines; ln += nwaves) {
    const long long base = (long long)ln * n;
    tile.to_run(nd, ud);
#pragma unroll 1
    for (int comp = c0; comp < c1; ++comp) {
      const T *const acc_in = A.acc[comp], *const f2_in = A.f2[comp], *const f3_in = A.f3[comp];
      const bool more = ln + nwaves < nlines;
      if constexpr (ALL) {
#pragma unroll
        for (int m = 0; m < V; ++m) um[m] = comp == 0 ? nd[m] : nx[m];
        if (comp < 2) tile.load(A.uc[comp + 1] + base, nx);
        else if (more) tile.load(A.ud + base + (long long)nwaves * n, nd);
      } else {
#pragma unroll
        for (int m = 0; m < V; ++m) um[m] = nx[m];
        if (more) {
          tile.load(A.ud + base + (long long)nwaves * n, nd);
          tile.load(A.uc[comp] + base + (long long)nwaves * n, nx);
        }
      }
      tile.to_run(um, uc);
      // every epilogue input is read before the first store (the compiler
      // cannot move loads above stores to possibly aliasing arrays), and ahead
      // of the solves where there are registers for it
      constexpr bool EARLY = V * sizeof(T) <= 32;
      T r[V], acc[V], f2[V], f3[V], rot[V];
      double un[V];
      auto inputs = [&] {
        if constexpr (GEN) {
          const MomUpdate<T> &U = A.up;
          tile.load(acc_in + base, acc);
          if (U.nterms >= 2) tile.load(U.f2[comp] + base, f2);
          if (U.nterms >= 3) tile.load(U.f3[comp] + base, f3);
          if (U.rot[comp]) tile.load(U.rot[comp] + base, rot);
          if constexpr (sizeof(T) == 4) tile.load(U.u64[comp] + base, un);
        } else {
          if (acc_in) tile.load(acc_in + base, acc);
          if (A.nterms >= 2) tile.load(f2_in + base, f2);
          if (A.nterms >= 3) tile.load(f3_in + base, f3);
        }
      };
      if constexpr (EARLY) inputs();
      T run[V];
      mom_line<T, V>(A, C, ud, uc, run, lane);
      tile.to_memory(run, r);
      if constexpr (!EARLY) inputs();
      if constexpr (GEN) {
        const MomUpdate<T> &U = A.up;
        const int lu = __builtin_amdgcn_readfirstlane(ln), k = lu / U.ny, j = lu - k * U.ny;
#pragma unroll
        for (int m = 0; m < V; ++m) {
          r[m] = mom_forced(U, comp, acc[m] + r[m], rot[m]);
          const double uo = sizeof(T) == 8 ? (double)um[m] : un[m];
          un[m] = pre_correc_point(U, comp, tile.point(m), j, k, mom_increment(U, r[m], f2[m], f3[m]) + uo);
        }
        tile.store(A.out[comp] + base, r);
        tile.store(U.u64[comp] + base, un);
        if constexpr (sizeof(T) == 4) {
          float sh[V];
#pragma unroll
          for (int m = 0; m < V; ++m) sh[m] = (float)un[m];
          tile.store(U.u32[comp] + base, sh);
        }
        continue;
      }
      if (acc_in) {
#pragma unroll
        for (int m = 0; m < V; ++m) r[m] = acc[m] + r[m];
      }
      tile.store(A.out[comp] + base, r);
      if (A.nterms) {
        // AB3 with FP64 accumulation: du = a f1 + b f2 + c f3, u_new = du + u_old
        double du[V];
#pragma unroll
        for (int m = 0; m < V; ++m) {
          if (A.nterms == 1) du[m] = A.ca * (double)r[m];
          else if (A.nterms == 2) du[m] = A.ca * (double)r[m] + A.cb * (double)f2[m];
          else du[m] = A.ca * (double)r[m] + A.cb * (double)f2[m] + A.cc * (double)f3[m];
        }
        if constexpr (sizeof(T) == 8) {
          // u_c is the FP64 velocity itself
          double un[V];
#pragma unroll
          for (int m = 0; m < V; ++m) un[m] = du[m] + (double)um[m];
          tile.store(A.u_new[comp] + base, un);
        } else {
          float d[V], sh[V];
#pragma unroll
          for (int m = 0; m < V; ++m) {
            d[m] = (float)du[m];
            sh[m] = (float)(du[m] + (double)um[m]);
          }
          tile.store(A.delta[comp] + base, d);
          tile.store(A.shadow[comp] + base, sh);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- host side

// The fused sweeps of precision T cover bounded lines that have a plan in that
// precision (bounded.hip; up to 1024 points, where the operators that the
// solver's other calls use end) and periodic lines with nx = 64, 128, 256 or
// 512 (one wavefront per x line, 1..8 points per lane) and ny, nz that YzShape
// can plan (a multiple of 16 whose block fits; 16..512 for both precisions).
// An FP32 solver does not ask for the FP64 plan, whose tables are twice the
// size in LDS: on free-slip lines of 257 points in x or 513 in y or z and on
// stretched walls of 513 points only FP32 fits (RK3 step, per operator and
// fused: 257^3 10727 and 7598, 256x513x128 stretched 8967 and 4759 us), on 17
// points only FP64 has its two segments (17^3 901 and 249 us).
// The product derivative uses the set of parity d==c (transeq.f90:125) and the
// velocity derivative the opposite one; one set serves both on periodic lines,
// so they must hold the same coefficients, which is the case there
// (schemes.f90:583-596 builds ffp from ff and prepares both from the same
// diagonals when ncl1 = ncln = 0).
template <typename T>
bool momentum_fusable(const Context &c) {
  for (int d = 0; d < 3; ++d) {
    const DirCoef &D = c.dir[d];
    if (D.bc1 != 0 && D.bcn != 0) {
      if (D.n > 1024 || !bounded_momentum_ok<T>(c, d)) return false;
      continue;
    }
    if (D.bc1 != 0 || D.bcn != 0) return false;
    if (!same_set(c.sets[D.set_d1_even], c.sets[D.set_d1_odd])) return false;
    if (!same_set(c.sets[D.set_d2_even], c.sets[D.set_d2_odd])) return false;
    if (d == 0) {
      const int V = D.n / 64;
      if (D.n % 64 != 0 || !(V == 1 || V == 2 || V == 4 || V == 8)) return false;
    } else if (!YzShape<double>().plan(D.n, 2, 3) || !YzShape<float>().plan(D.n, 2, 3)) {
      return false;
    }
  }
  return true;
}
template bool momentum_fusable<double>(const Context &);
template bool momentum_fusable<float>(const Context &);

template <typename T, bool GEN, bool ALL>
static void launch_mom_x(const MomArgs<T> &A, int V, int nlines, dim3 grid, dim3 block, hipStream_t st) {
  switch (V) {
    case 1: hipLaunchKernelGGL((mom_x_kernel<T, 1, GEN, ALL>), grid, block, 0, st, A, nlines); break;
    case 2: hipLaunchKernelGGL((mom_x_kernel<T, 2, GEN, ALL>), grid, block, 0, st, A, nlines); break;
    case 4: hipLaunchKernelGGL((mom_x_kernel<T, 4, GEN, ALL>), grid, block, 0, st, A, nlines); break;
    default: hipLaunchKernelGGL((mom_x_kernel<T, 8, GEN, ALL>), grid, block, 0, st, A, nlines); break;
  }
}

// One sweep of all three components (blockIdx.z): 3 launches a step instead
// of 9.  Small grids gain: a one-component sweep of 64^3 leaves most of the
// chip idle (128 to 256 blocks), three at once fill it (ten 64^3 FP32 steps
// with the learned closure 2.53 -> 2.19 ms); at 256^3 the time is the same
// (five steps 11.41 -> 11.40 ms FP64, 6.62 -> 6.64 ms FP32).
template <typename T>
int launch_momentum(const Context &c, int dir, const MomIO<T> &io, int nx, int ny, int nz, hipStream_t st) {
  const DirCoef &D = c.dir[dir];
  if (D.bc1 != 0) return launch_bounded_momentum<T>(c, dir, io, st);
  if (!same_set(c.sets[D.set_d1_even], c.sets[D.set_d1_odd]) || !same_set(c.sets[D.set_d2_even], c.sets[D.set_d2_odd]))
    return fail(X3D_ERR_UNSUPPORTED, "fused momentum sweep: product and velocity sets differ");
  const TriSet &s1 = c.sets[D.set_d1_even];
  const TriSet &s2 = c.sets[D.set_d2_even];
  MomArgs<T> A{};
  A.ud = io.u[dir];
  for (int i = 0; i < 3; ++i) {
    A.uc[i] = io.u[i];
    A.acc[i] = io.acc[i];
    A.out[i] = io.out[i];
    A.f2[i] = io.f2[i];
    A.f3[i] = io.f3[i];
    A.u_new[i] = io.u_new[i];
    A.delta[i] = io.delta[i];
    A.shadow[i] = io.shadow[i];
  }
  TriDev<T> t1, t2;
  if constexpr (sizeof(T) == 8) { t1 = s1.dev64(); t2 = s2.dev64(); }
  else { t1 = s1.dev32(); t2 = s2.dev32(); }
  A.pk1 = t1.pk; A.pk2 = t2.pk;
  A.alfa1 = t1.alfa; A.den1 = t1.sm_den; A.alfa2 = t2.alfa; A.den2 = t2.sm_den;
  A.rden1 = t1.rden; A.rden2 = t2.rden;
  A.s = cast_sten<T>(D.s);
  A.xnu = (T)c.xnu;
  A.n = D.n;
  A.ca = io.ca; A.cb = io.cb; A.cc = io.cc; A.nterms = io.nterms;
  const int n = D.n;
  if (dir == 0) {
    const int V = n / 64;
    if (n % 64 != 0 || !(V == 1 || V == 2 || V == 4 || V == 8))
      return fail(X3D_ERR_UNSUPPORTED, "fused x sweep needs nx = 64, 128, 256 or 512");
    for (int i = 0; i < 3 && !io.general; ++i)
      if (io.nterms && (sizeof(T) == 8 ? !io.u_new[i] : (!io.delta[i] || !io.shadow[i])))
        return fail(X3D_ERR_ARG, "momentum: AB3 output buffers missing");
    const int nlines = ny * nz;
    // Up to 8192 lines there are too few wavefronts to put a line's components
    // into one (128 x 64^2: 1715 us a step against 1740; 128^3 with 16384 lines:
    // 1532 against 1510).  The wavefronts' lines are of one number each; FP64
    // has two wavefronts a SIMD and gains from the loads ahead (256^3: 441 us
    // with 8192, 475 with 65536), FP32 from more of them (267 and 251).
    const bool all = nlines > 8192;
    const int most = sizeof(T) == 8 ? 8192 : 65536, per = (nlines + most - 1) / most;
    const int waves = (nlines + per - 1) / per;
    const dim3 grid((waves + 3) / 4, 1, all ? 1 : 3), block(256);
    if (io.general) {
      X3D_TRY(fill_update<T>(c, io, &A.up));
      for (int i = 0; i < 3; ++i)
        if (!io.acc[i]) return fail(X3D_ERR_ARG, "momentum: the x sweep comes last");
      if (all) launch_mom_x<T, true, true>(A, V, nlines, grid, block, st);
      else launch_mom_x<T, true, false>(A, V, nlines, grid, block, st);
    } else {
      if (all) launch_mom_x<T, false, true>(A, V, nlines, grid, block, st);
      else launch_mom_x<T, false, false>(A, V, nlines, grid, block, st);
    }
  } else {
    if (io.nterms) return fail(X3D_ERR_ARG, "AB3 is fused into the x sweep only");
    if (dir == 1) {
      A.na = nx; A.nb = nz; A.sa = 1; A.sb = (long long)nx * ny; A.se = nx;
    } else {
      A.na = nx; A.nb = ny; A.sa = 1; A.sb = nx; A.se = (long long)nx * ny;
    }
    constexpr int L = YzShape<T>::L;
    YzShape<T> Y;
    if (!Y.plan(n, 2, 3)) return fail(X3D_ERR_UNSUPPORTED, "fused y/z sweep: line length not supported");
    if ((size_t)nx * ny * nz * sizeof(T) >= ((size_t)1 << 32))
      return fail(X3D_ERR_UNSUPPORTED, "fused y/z sweep: field larger than 4 GiB");
    A.kdepth = std::max(t1.kdepth, t2.kdepth);
    const dim3 grid((A.na + Y.TL - 1) / Y.TL, A.nb, 3), block(Y.TL, Y.P);
    const size_t shmem = Y.shmem;
    hipLaunchKernelGGL((mom_yz_kernel<T, L>), grid, block, shmem, st, A);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(X3D_ERR_HIP, std::string("momentum launch: ") + hipGetErrorString(e));
  return X3D_OK;
}

template int launch_momentum<double>(const Context &, int, const MomIO<double> &, int, int, int, hipStream_t);
template int launch_momentum<float>(const Context &, int, const MomIO<float> &, int, int, int, hipStream_t);

}  // namespace x3d
