#pragma once
// Segmented solves of lines with free-slip or no-slip ends, and of periodic
// lines that are no whole number of segments.
//
// The n_out rows of a line are cut into P segments of L, one thread each, as
// in seg_solve, but anchored at both ends: segments 0 .. P-3 start at s L, the
// last one covers the last L rows, and the one before it takes the r <= L rows
// left between them, filled up with rows that pass both recurrences through
// unchanged (fs = -1; fw = 0, ff fw = -1; right-hand side 0).  The boundary
// closures, at most four rows at each end (derive.f90), then always sit at
// the same registers of the first and of the last thread of a line, and their
// points are in that thread's window: they cost no loads and no barrier of
// their own.  A closure row is a weighted sum of the end's first eight points
// with weights worked out at initialisation, in one form for every boundary
// kind, parity and operator: first differences for the derivatives, second
// differences for the second derivative, so that a row of small differences
// keeps the rounding error of the interior form; the points themselves for
// the interpolations.
#include "lines_impl.h"

namespace x3d {

// Words of one table on the device: P*L packed rows, then the closure weights
// [end][row from the end][8].
constexpr int EDGE_WORDS = 2 * 4 * 8;

// Closure rows at each end (NR), the points row q reads (its first NE(q)), and
// what its weights multiply (KIND): 0 the points, 1 U0 and first differences,
// 2 U0, U1 - U0 and second differences.
template <int OP>
struct EdgeForm {
  static constexpr int NR = OP == OP_DER1 || OP == OP_DERPV ? 2 : (OP == OP_DERVP ? 1 : (OP == OP_INTERVP ? 3 : 4));
  static constexpr int KIND = OP == OP_DER2 ? 2 : (OP == OP_INTERVP || OP == OP_INTERPV ? 0 : 1);
  static constexpr int NE(int q) {
    return OP == OP_DER1 ? 4 : (OP == OP_DER2 ? q + 5 : (OP == OP_INTERVP ? q + 5 : (OP == OP_INTERPV ? q + 4 : 3)));
  }
};

// Constant memory as the scalar unit reads it: the weights are the same for
// every lane, and as ordinary loads they cost each end's thread a chain of
// vector-memory latencies (the channel's y momentum sweep took 183 us with
// those; the weights now come in through scalar loads).
template <typename T>
using CPtr = const __attribute__((address_space(4))) T *;
template <typename T>
__device__ __forceinline__ CPtr<T> uniform_ptr(const T *p) {
  return (CPtr<T>)p;
}

template <int OP, typename T>
__device__ __forceinline__ void edge_rows(const T (&U)[8], CPtr<T> W, T (&r)[4]) {
  using F = EdgeForm<OP>;
  constexpr int NB = F::NE(F::NR - 1);
  T b[8];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if constexpr (F::KIND == 0) b[j] = U[j];
    else if (j == 0) b[j] = U[0];
    else if (F::KIND == 1 || j == 1) b[j] = U[j] - U[j - 1];
    else b[j] = (U[j] - U[j - 1]) - (U[j - 1] - U[j - 2]);
  }
#pragma unroll
  for (int q = 0; q < F::NR; ++q) {
    T a = W[8 * q] * b[0];
#pragma unroll
    for (int j = 1; j < NB; ++j)
      if (j < F::NE(q)) a += W[8 * q + j] * b[j];
    r[q] = a;
  }
}

// First output row of a segment, and how many rows it has.
template <int L>
__device__ __forceinline__ int bound_first(int seg, int P, int n_out) {
  return seg == P - 1 ? n_out - L : seg * L;
}
template <int L>
__device__ __forceinline__ int bound_rows(int seg, int P, int n_out) {
  return seg == P - 2 ? n_out - (P - 1) * L : L;
}

// Right-hand sides of a segment from its window U(e0-HW .. e0+L+HW-1), e0 its
// first row; edge the closure weights, rows how many rows the segment has.
template <int OP, typename T, int L, int HW>
__device__ __forceinline__ void bound_rhs(const T (&win)[L + 2 * HW], T (&w)[L], const Sten<T> &s,
                                          const T *edge, const int seg, const int P, const int rows) {
  using F = EdgeForm<OP>;
  const CPtr<T> W = uniform_ptr(edge);
  // window index of the line's last point, seen from the last segment
  constexpr int FAR = L + HW - 1 + (OP == OP_DERVP || OP == OP_INTERVP) - (OP == OP_DERPV || OP == OP_INTERPV);
#pragma unroll
  for (int m = 0; m < L; ++m) w[m] = interior_row<OP, T, L + 2 * HW>(win, m + HW, s);
  if (seg == 0) {
    T U[8], r[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) U[j] = win[HW + j];
    edge_rows<OP, T>(U, W, r);
#pragma unroll
    for (int q = 0; q < F::NR; ++q) w[q] = r[q];
  } else if (seg == P - 1) {
    T U[8], r[4];
#pragma unroll
    for (int j = 0; j < 8; ++j) U[j] = win[FAR - j];
    edge_rows<OP, T>(U, W + 32, r);
#pragma unroll
    for (int q = 0; q < F::NR; ++q) w[L - 1 - q] = r[q];
  }
  if (rows < L) {
#pragma unroll
    for (int m = 1; m < L; ++m)
      if (m >= rows) w[m] = T(0);
  }
}

// The rows of a segment to memory; NT: streaming stores.
template <typename T, int L, bool NT>
__device__ __forceinline__ void store_rows(T *p, const unsigned off, const unsigned step, const T (&v)[L],
                                           const int rows) {
  if (rows == L) {
#pragma unroll
    for (int m = 0; m < L; ++m) {
      if constexpr (NT) st_nt(p, off + (unsigned)m * step, v[m]);
      else at(p, off + (unsigned)m * step) = v[m];
    }
  } else {
#pragma unroll
    for (int m = 0; m < L; ++m)
      if (m < rows) at(p, off + (unsigned)m * step) = v[m];
  }
}

// Table of right-hand side q of N on NT tables: the first N-NT+1 share table
// 0, the others have one each.
template <int N, int NT>
constexpr int table_of(int q) { return q <= N - NT ? 0 : q - (N - NT); }

// seg_solve without a periodic closure, on NT tables cs[t] (P*L packed rows
// each, in LDS; the caller's barrier after filling them precedes the call).
// cf, cb: N*P*TL words, gf, gb: NT*P.
template <typename T, int L, int N, int NT>
__device__ __forceinline__ void bound_solve(T (&v)[N][L], const T *cs, T *cf, T *cb, T *gf, T *gb, const int line,
                                            const int seg, const int TL, const int P, const int K) {
  const int PT = P * TL, CW = 4 * P * L;
  const T *c0 = cs + 4 * (seg * L);
  T prev[N], g[NT];
#pragma unroll
  for (int q = 0; q < N; ++q) prev[q] = T(0);
#pragma unroll
  for (int t = 0; t < NT; ++t) g[t] = T(1);
#pragma unroll
  for (int m = 0; m < L; ++m) {
    T f[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f[t] = c0[t * CW + 4 * m];
      g[t] = -f[t] * g[t];
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
      prev[q] = v[q][m] - prev[q] * f[table_of<N, NT>(q)];
      v[q][m] = prev[q];
    }
  }
#pragma unroll
  for (int q = 0; q < N; ++q) cf[q * PT + seg * TL + line] = prev[q];
  if (line == 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t) gf[t * P + seg] = g[t];
  }
  __syncthreads();
  if (seg > 0) {
    T cin[N];
#pragma unroll
    for (int q = 0; q < N; ++q) cin[q] = T(0);
    for (int s0 = seg - K > 0 ? seg - K : 0; s0 < seg; s0 += 4) {
      T gs[4][NT], cv[4][N];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = s0 + j < seg ? s0 + j : seg - 1;
#pragma unroll
        for (int t = 0; t < NT; ++t) gs[j][t] = gf[t * P + s];
#pragma unroll
        for (int q = 0; q < N; ++q) cv[j][q] = cf[q * PT + s * TL + line];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (s0 + j < seg) {
#pragma unroll
          for (int q = 0; q < N; ++q) cin[q] = cv[j][q] + gs[j][table_of<N, NT>(q)] * cin[q];
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) g[t] = T(1);
#pragma unroll
    for (int m = 0; m < L; ++m) {
#pragma unroll
      for (int t = 0; t < NT; ++t) g[t] = -c0[t * CW + 4 * m] * g[t];
#pragma unroll
      for (int q = 0; q < N; ++q) v[q][m] += g[table_of<N, NT>(q)] * cin[q];
    }
  }
  T nxt[N];
#pragma unroll
  for (int q = 0; q < N; ++q) nxt[q] = T(0);
#pragma unroll
  for (int t = 0; t < NT; ++t) g[t] = T(1);
#pragma unroll
  for (int m = L - 1; m >= 0; --m) {
    T fw[NT], ffw[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      fw[t] = c0[t * CW + 4 * m + 1];
      ffw[t] = c0[t * CW + 4 * m + 2];
      g[t] = -ffw[t] * g[t];
    }
#pragma unroll
    for (int q = 0; q < N; ++q) {
      nxt[q] = fw[table_of<N, NT>(q)] * v[q][m] - ffw[table_of<N, NT>(q)] * nxt[q];
      v[q][m] = nxt[q];
    }
  }
#pragma unroll
  for (int q = 0; q < N; ++q) cb[q * PT + seg * TL + line] = nxt[q];
  if (line == 0) {
#pragma unroll
    for (int t = 0; t < NT; ++t) gb[t * P + seg] = g[t];
  }
  __syncthreads();
  if (seg < P - 1) {
    T c[N];
#pragma unroll
    for (int q = 0; q < N; ++q) c[q] = T(0);
    const int last = seg + K < P - 1 ? seg + K : P - 1;
    for (int s0 = last; s0 > seg; s0 -= 4) {
      T gs[4][NT], cv[4][N];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int s = s0 - j > seg ? s0 - j : seg + 1;
#pragma unroll
        for (int t = 0; t < NT; ++t) gs[j][t] = gb[t * P + s];
#pragma unroll
        for (int q = 0; q < N; ++q) cv[j][q] = cb[q * PT + s * TL + line];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (s0 - j > seg) {
#pragma unroll
          for (int q = 0; q < N; ++q) c[q] = cv[j][q] + gs[j][table_of<N, NT>(q)] * c[q];
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) g[t] = T(1);
#pragma unroll
    for (int m = L - 1; m >= 0; --m) {
#pragma unroll
      for (int t = 0; t < NT; ++t) g[t] = -c0[t * CW + 4 * m + 2] * g[t];
#pragma unroll
      for (int q = 0; q < N; ++q) v[q][m] += g[table_of<N, NT>(q)] * c[q];
    }
  }
}

// Copy of NT device tables of cnt words into LDS split around the caller's
// window loads, as TableCopy does for two: R words a thread through registers,
// what is left of larger tables (a block may have fewer threads than words)
// straight in store().
template <typename T, int NT, int R = 2>
struct BoundCopy {
  T v[NT][R];
  __host__ __device__ __forceinline__ void load(const T *const (&src)[NT], int tid, int nthr, int cnt) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (tid + r * nthr < cnt) v[t][r] = src[t][tid + r * nthr];
  }
  __host__ __device__ __forceinline__ void store(T *cs, const T *const (&src)[NT], int tid, int nthr,
                                                 int cnt) const {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (tid + r * nthr < cnt) cs[t * cnt + tid + r * nthr] = v[t][r];
      for (int i = tid + R * nthr; i < cnt; i += nthr) cs[t * cnt + i] = src[t][i];
    }
  }
};

// Table of one operator of a direction at precision T (null: none): segments
// of the precision's length, or (longer) one row longer.
template <typename T>
struct BoundDev {
  const T *pk = nullptr, *edge = nullptr;
  int P = 0, K = 0;
};
template <typename T>
BoundDev<T> bound_dev(const Context &c, int dir, int op, int par, bool longer = false) {
  const BoundTab &b = c.btab[dir][op][par];
  const AnchorTab<T> *t;
  if constexpr (sizeof(T) == 8) t = &b.t64[longer ? 1 : 0];
  else t = &b.t32[longer ? 1 : 0];
  BoundDev<T> d;
  if (!t->pk) return d;
  const int L = (sizeof(T) == 8 ? SEG_L64 : SEG_L32) + (longer ? 1 : 0);
  d.P = t->P;
  d.K = t->K;
  d.pk = t->pk;
  d.edge = t->pk + 4 * (size_t)d.P * L;
  return d;
}

// Launch shape: TL lines of 128 bytes a row (fewer where the block or its LDS
// would not fit) x P segments; extra(TL) words of LDS beside the solve's.
template <typename T, int LEN = sizeof(T) == 8 ? SEG_L64 : SEG_L32>
struct BoundShape {
  static constexpr int L = LEN;
  int P = 0, TL = 0;
  size_t shmem = 0;
  template <typename F>
  bool plan(int n_out, int nt, int nrhs, F extra) {
    if (n_out < 2 * L) return false;
    P = (n_out + L - 1) / L;
    for (TL = 128 / (int)sizeof(T); TL >= 8; TL >>= 1) {
      shmem = sizeof(T) * ((size_t)nt * 4 * P * L + 2 * (size_t)nrhs * P * TL + 2 * (size_t)nt * P + extra(TL));
      if (TL * P <= 1024 && shmem <= 65536) return true;
    }
    return false;
  }
  bool plan(int n_out, int nt, int nrhs) {
    return plan(n_out, nt, nrhs, [](int) { return (size_t)0; });
  }
};

// Segment length of a sweep: one row longer where a block's lines then need
// fewer wavefronts on the fullest of a compute unit's four SIMDs.  Bounded
// lines have 2^k + 1 points: in segments of 8 rows 129 points take 17 x 16
// threads, a fifth wavefront for the last segment, and 6.8 wavefronts a
// compute unit were resident on average; in segments of 9 rows they take
// 15 x 16, four wavefronts.  256 x 129 x 128: y momentum sweep FP64 124 -> 84,
// FP32 64 -> 44 us, y gradient sweep 54 -> 45 and 31 -> 21 us.  Where the count
// a SIMD stays (65 points: 3 wavefronts or 2) the shorter segments are as fast
// (momentum) or faster (gradient 8.9 against 9.8, 6.6 against 8.0 us at 65^3).
template <typename T>
struct BoundPick {
  bool longer = false;
  int P = 0, TL = 0;
  size_t shmem = 0;
  template <typename F>
  bool plan(int n_out, int nt, int nrhs, F extra) {
    BoundShape<T> Y;
    BoundShape<T, BoundShape<T>::L + 1> Z;
    if (!Y.plan(n_out, nt, nrhs, extra)) return false;
    P = Y.P; TL = Y.TL; shmem = Y.shmem;
    // (a block has a thread for each row of a line)
    if (Z.plan(n_out, nt, nrhs, extra) && Z.TL * Z.P >= n_out &&
        (Z.TL * Z.P + 255) / 256 * Y.TL < (Y.TL * Y.P + 255) / 256 * Z.TL) {
      longer = true;
      P = Z.P; TL = Z.TL; shmem = Z.shmem;
    }
    return true;
  }
  bool plan(int n_out, int nt, int nrhs) {
    return plan(n_out, nt, nrhs, [](int) { return (size_t)0; });
  }
};

// ---------------------------------------------------------------- velocity update
// What the x momentum sweep does with a finished right-hand side besides
// storing it, on boxes with bounded directions and in RK3: the channel's
// forcing (momentum_forcing_channel, Case-Channel.f90:396-420), the AB3 or RK3
// combination with FP64 accumulation (time_integrators.f90:85-157) and
// pre_correc (navier.f90:502-789): zero normal velocity on free-slip faces,
// the wall velocity from the stored wall pressure gradient on no-slip walls.
template <typename T>
struct MomUpdate {
  const T *f2[3], *f3[3];
  double *u64[3];               // FP64: the new velocity; FP32: the FP64 velocity, updated in place
  float *u32[3];                // FP32: the new velocity's rounding
  double ca, cb, cc;
  int nterms;
  double addc;                  // constant pressure gradient (x component)
  const T *rot[3];              // spin-up rotation: velocity and factor (null: none)
  T rotc[3];
  int face[3];                  // free-slip faces of each direction: bit 0 low, bit 1 high
  int wall;                     // no-slip y walls: bit 0 low, bit 1 high
  const double *wallg;          // dpdx, dpdz of the low wall, then of the high one, [k*nx + i] each
  double gdt;
  int nx, ny, nz;
};

// The right-hand side of a point with the forcing on it.
template <typename T>
__device__ __forceinline__ T mom_forced(const MomUpdate<T> &A, const int comp, T r, const T rot) {
  if (comp == 0 && A.addc != 0.0) r = (T)((double)r + A.addc);
  if (A.rot[comp]) r = r + A.rotc[comp] * rot;
  return r;
}

template <typename T>
__device__ __forceinline__ double mom_increment(const MomUpdate<T> &A, const T f1, const T f2, const T f3) {
  if (A.nterms == 1) return A.ca * (double)f1;
  if (A.nterms == 2) return A.ca * (double)f1 + A.cb * (double)f2;
  return A.ca * (double)f1 + A.cb * (double)f2 + A.cc * (double)f3;
}

// pre_correc of one point of component comp.
template <typename T>
__device__ __forceinline__ double pre_correc_point(const MomUpdate<T> &A, const int comp, const int i, const int j,
                                                   const int k, double v) {
  const int f = A.face[comp];
  if (f) {
    const int e = comp == 0 ? i : (comp == 1 ? j : k);
    const int last = (comp == 0 ? A.nx : (comp == 1 ? A.ny : A.nz)) - 1;
    if (((f & 1) && e == 0) || ((f & 2) && e == last)) v = 0.0;
  }
  if (A.wall) {
    const bool lo = (A.wall & 1) && j == 0, hi = (A.wall & 2) && j == A.ny - 1;
    if (lo || hi) {
      const size_t np = (size_t)A.nx * A.nz, q = (size_t)k * A.nx + i;
      if (comp == 1) v = 0.0;
      else v = 0.0 + A.wallg[((hi ? 2 : 0) + (comp == 0 ? 0 : 1)) * np + q] * A.gdt;
    }
  }
  return v;
}

template <typename T>
int fill_update(const Context &c, const MomIO<T> &io, MomUpdate<T> *U) {
  for (int i = 0; i < 3; ++i) {
    U->f2[i] = io.f2[i];
    U->f3[i] = io.f3[i];
    U->u64[i] = io.u_new[i];
    U->u32[i] = io.shadow[i];
    U->rot[i] = io.rot[i];
    U->rotc[i] = io.rotc[i];
    U->face[i] = (c.dir[i].bc1 == 1 ? 1 : 0) | (c.dir[i].bcn == 1 ? 2 : 0);
    if (!io.u_new[i] || (sizeof(T) == 4 && !io.shadow[i]) || (io.nterms >= 2 && !io.f2[i]) ||
        (io.nterms >= 3 && !io.f3[i]))
      return fail(X3D_ERR_ARG, "momentum: velocity update buffers missing");
  }
  if (io.nterms < 1) return fail(X3D_ERR_ARG, "momentum: no terms to update the velocity with");
  U->ca = io.ca; U->cb = io.cb; U->cc = io.cc; U->nterms = io.nterms;
  U->addc = io.addc;
  U->wall = (io.wall1 ? 1 : 0) | (io.walln ? 2 : 0);
  U->wallg = io.wallg;
  if (U->wall && !U->wallg) return fail(X3D_ERR_ARG, "momentum: wall planes missing");
  U->gdt = io.gdt;
  U->nx = c.p.nx; U->ny = c.p.ny; U->nz = c.p.nz;
  return X3D_OK;
}

// ---------------------------------------------------------------- projection
// Inputs of each sweep and the solve they feed: I0/I1 interpolations, D0 the
// derivative (-1: absent).
//   DIV_X   out0 = Dvp(u), out1 = Ivp(v), out2 = Ivp(w)        navier.f90:297,313-314
//   DIV_Y   out0 = Ivp(in0) + Dvp(in1), out1 = Ivp(in2)         navier.f90:321-327
//   DIV_Z   out0 = Ivp(in0) + Dvp(in1)                          navier.f90:333-339
//   GRAD_Z  out0 = Ipv(in0), out1 = Dpv(in0)                    navier.f90:400-403
//   GRAD_Y  out0 = Ipv(in0), out1 = Dpv(in0), out2 = Ipv(in1)   navier.f90:414-419
//   GRAD_X  u -= Dpv(in0), v -= Ipv(in1), w -= Ipv(in2)         navier.f90:426-431, cor_vel 206-249
template <int SW>
struct Recipe;
template <>
struct Recipe<SW_DIV_X> {
  static constexpr bool PV = false;
  static constexpr int NIN = 3, NI = 2, I0 = 1, I1 = 2, D0 = 0;
};
template <>
struct Recipe<SW_DIV_Y> {
  static constexpr bool PV = false;
  static constexpr int NIN = 3, NI = 2, I0 = 0, I1 = 2, D0 = 1;
};
template <>
struct Recipe<SW_DIV_Z> {
  static constexpr bool PV = false;
  static constexpr int NIN = 2, NI = 1, I0 = 0, I1 = -1, D0 = 1;
};
template <>
struct Recipe<SW_GRAD_Z> {
  static constexpr bool PV = true;
  static constexpr int NIN = 1, NI = 1, I0 = 0, I1 = -1, D0 = 0;
};
template <>
struct Recipe<SW_GRAD_Y> {
  static constexpr bool PV = true;
  static constexpr int NIN = 2, NI = 2, I0 = 0, I1 = 1, D0 = 0;
};
template <>
struct Recipe<SW_GRAD_X> {
  static constexpr bool PV = true;
  static constexpr int NIN = 3, NI = 2, I0 = 1, I1 = 2, D0 = 0;
};

// cor_vel of the general step (navier.f90:206-249) and the wall planes of the
// pressure gradient over gdt that gradp keeps (navier.f90:456-479).
struct CorVel {
  double *u64[3];
  float *u32[3];                // FP32 compute: the velocity's rounding (else null)
  int apply;
  int wall;                     // bit 0 low, bit 1 high
  double *wallg;                // dpdx, dpdz of the low wall, then of the high one
  double gdt;
  int nx, ny, nz;
};

template <typename T>
__device__ __forceinline__ void store_wall(const CorVel &A, const int comp, const int i, const int j, const int k,
                                           const T g) {
  if (!A.wall || comp == 1) return;
  const bool lo = (A.wall & 1) && j == 0, hi = (A.wall & 2) && j == A.ny - 1;
  if (!lo && !hi) return;
  const size_t np = (size_t)A.nx * A.nz;
  A.wallg[((hi ? 2 : 0) + (comp == 0 ? 0 : 1)) * np + (size_t)k * A.nx + i] = (double)g / A.gdt;
}

template <typename T>
int fill_corvel(const Context &c, const ProjIO<T> &io, CorVel *A) {
  for (int i = 0; i < 3; ++i) {
    A->u64[i] = io.u64[i];
    A->u32[i] = io.u32[i];
    if (io.apply && (!io.u64[i] || (sizeof(T) == 4 && !io.u32[i])))
      return fail(X3D_ERR_ARG, "projection: GRAD_X needs the FP64 velocity");
  }
  A->apply = io.apply ? 1 : 0;
  A->wall = (io.wall1 ? 1 : 0) | (io.walln ? 2 : 0);
  A->wallg = io.wallg;
  if (A->wall && !A->wallg) return fail(X3D_ERR_ARG, "projection: wall planes missing");
  A->gdt = io.gdt;
  A->nx = c.p.nx; A->ny = c.p.ny; A->nz = c.p.nz;
  return X3D_OK;
}

// Block maximum and sum into divp[block] and divp[blocks + block]
// (navier.f90:348-361), every thread of the block taking part.
__device__ __forceinline__ void block_max_sum(double mx, double sm, const int tid, const int nthr,
                                              double *__restrict__ divp) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double om = __shfl_xor(mx, off), os = __shfl_xor(sm, off);
    if ((tid ^ off) >= nthr) continue;   // a lane that the last wavefront does not have
    mx = om > mx ? om : mx;
    sm += os;
  }
  __shared__ double rmx[16], rsm[16];
  if ((tid & 63) == 0) {
    rmx[tid >> 6] = mx;
    rsm[tid >> 6] = sm;
  }
  __syncthreads();
  if (tid == 0) {
    double bm = rmx[0], bs = rsm[0];
    for (int i = 1; i < (nthr + 63) / 64; ++i) {
      bm = rmx[i] > bm ? rmx[i] : bm;
      bs += rsm[i];
    }
    const unsigned nblk = gridDim.x * gridDim.y, blk = blockIdx.y * gridDim.x + blockIdx.x;
    divp[blk] = bm;
    divp[nblk + blk] = bs;
  }
}

// quotient of small positive integers (idx < 2^22) by a uniform divisor
__device__ __forceinline__ int small_div(int idx, int n, float rn) {
  int q = (int)((float)idx * rn);
  const int rem = idx - q * n;
  if (rem < 0) --q;
  else if (rem >= n) ++q;
  return q;
}

}  // namespace x3d
