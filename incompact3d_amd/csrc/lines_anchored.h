#pragma once
// One line operator on anchored segments (bounded_impl.h): free-slip and
// no-slip ends of any length, and periodic lines that are no whole number of
// segments.  They replace, for the library's own coefficient sets,
// seg_wall_kernel, whose boundary threads read their closure rows from memory
// in a pass of their own before the windows were loaded, and line_kernel's
// 16- to 64-point segments with their chain through every segment.
#include "bounded_impl.h"

namespace x3d {

template <typename T>
struct AnchorArgs {
  const T *u[3], *acc[3];       // batch of up to three (blockIdx.z)
  T *t[3];
  const T *pk[3], *edge[3];
  const T *u2, *mul;            // single operators: product input, epilogue factor
  T ac, rc;                     // t = ac*acc + rc*(mul*result)
  const T *pp;                  // post-multiplier along the line
  T alfa, rden;                 // periodic closure
  Sten<T> s;
  int n_in, n_out, P, K;
  int na, nb;
  long long sb_in, sb_out, se;  // y/z: strides of b in and out, and of a line's points
  int row;                      // x: LDS words of a line
};

// Right-hand side of a segment from its window.
template <typename T, int OP, int L, bool PER>
__device__ __forceinline__ void anchor_rhs(const AnchorArgs<T> &A, const int q, const T (&win)[L + 8], T (&w)[L],
                                           const int seg, const int rows) {
  if constexpr (!PER) {
    bound_rhs<OP, T, L, 4>(win, w, A.s, A.edge[q], seg, A.P, rows);
  } else {
#pragma unroll
    for (int m = 0; m < L; ++m) {
      w[m] = interior_row<OP, T, L + 8>(win, m + 4, A.s);
      if (m >= rows) w[m] = T(0);
    }
  }
}

// Sherman-Morrison closure of periodic lines (derive.f90:55-59); ends: 2*TL
// words of LDS.
template <typename T, int L>
__device__ __forceinline__ void anchor_close(const AnchorArgs<T> &A, T (&w)[L], const T *cs, T *ends, const int line,
                                             const int seg, const int TL) {
  if (seg == 0) ends[line] = w[0];
  if (seg == A.P - 1) ends[TL + line] = w[L - 1];
  __syncthreads();
  const T sx = (ends[line] - A.alfa * ends[TL + line]) * A.rden;
#pragma unroll
  for (int m = 0; m < L; ++m) w[m] = w[m] - sx * cs[4 * (seg * L + m) + 3];
}

template <typename T, int OP, int L, bool PER, bool EPI>
__global__ void __launch_bounds__(1024) anchor_yz_kernel(const AnchorArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n_in = A.n_in, n_out = A.n_out;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + CW, *cb = cf + P * TL, *gf = cb + P * TL, *gb = gf + P, *ends = gb + P;
  const int q = (int)blockIdx.z;
  const T *const u = A.u[q];
  const int a = (int)blockIdx.x * TL + line, b = (int)blockIdx.y;
  const bool active = a < A.na;
  const int al = active ? a : A.na - 1;
  const int e0 = bound_first<L>(seg, P, n_out), rows = bound_rows<L>(seg, P, n_out);
  const unsigned ib = ((unsigned)al + (unsigned)b * (unsigned)A.sb_in) * (unsigned)sizeof(T);
  const unsigned step = (unsigned)A.se * (unsigned)sizeof(T);
  auto place = [&](int j) {
    if constexpr (PER) return (unsigned)(j < 0 ? j + n_in : (j >= n_in ? j - n_in : j));
    else return (unsigned)(j < 0 ? 0 : (j >= n_in ? n_in - 1 : j));
  };
  const T *const src[1] = {A.pk[q]};
  if constexpr (sizeof(T) == 4) __builtin_amdgcn_s_setprio(3);
  T w[1][L];
  BoundCopy<T, 1> tc;
  {
    T win[L + 8];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) {
      const unsigned o = ib + place(e0 - 4 + k) * step;
      T x = at(u, o);
      if (EPI && A.u2) x *= at(A.u2, o);
      win[k] = x;
    }
    tc.load(src, tid, nthr, CW);
    if constexpr (sizeof(T) == 4) __builtin_amdgcn_s_setprio(0);
    anchor_rhs<T, OP, L, PER>(A, q, win, w[0], seg, rows);
  }
  tc.store(cs, src, tid, nthr, CW);
  __syncthreads();
  bound_solve<T, L, 1, 1>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
  if constexpr (PER) anchor_close<T, L>(A, w[0], cs, ends, line, seg, TL);
  if (!active) return;
  int e1 = e0;
  asm volatile("" : "+v"(e1));   // offsets worked out again rather than held through the solve
  if (A.pp) {
#pragma unroll
    for (int m = 0; m < L; ++m) w[0][m] *= A.pp[m < rows ? e1 + m : e1];
  }
  const unsigned ob = ((unsigned)al + (unsigned)b * (unsigned)A.sb_out) * (unsigned)sizeof(T) + (unsigned)e1 * step;
  if constexpr (EPI) {
    if (A.mul) {
#pragma unroll
      for (int m = 0; m < L; ++m) w[0][m] *= at(A.mul, ob + (unsigned)(m < rows ? m : 0) * step);
    }
#pragma unroll
    for (int m = 0; m < L; ++m) w[0][m] = A.rc * w[0][m];
    if (const T *acc = A.acc[q]) {
      T aa[L];
#pragma unroll
      for (int m = 0; m < L; ++m) aa[m] = at(acc, ob + (unsigned)(m < rows ? m : 0) * step);
#pragma unroll
      for (int m = 0; m < L; ++m) w[0][m] = A.ac * aa[m] + w[0][m];
    }
  }
  store_rows<T, L, true>(A.t[q], ob, step, w[0], rows);
}

// x lines: TL whole lines, one contiguous piece of memory, through LDS.
template <typename T, int OP, int L, bool PER, bool EPI>
__global__ void __launch_bounds__(1024) anchor_x_kernel(const AnchorArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n_in = A.n_in, n_out = A.n_out, row = A.row;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + CW, *cb = cf + P * TL, *gf = cb + P * TL, *gb = gf + P, *ends = gb + P,
    *tile = ends + 2 * TL;
  const int q = (int)blockIdx.z;
  const T *const u = A.u[q], *const pk = A.pk[q];
  const int l0 = (int)blockIdx.x * TL;
  const int nl = min(TL, A.na - l0);
  const long long bi = (long long)l0 * n_in, bo = (long long)l0 * n_out;
  const float rni = 1.0f / (float)n_in, rno = 1.0f / (float)n_out;
  for (int idx = tid; idx < nl * n_in; idx += nthr) {
    const int l = small_div(idx, n_in, rni);
    T x = u[bi + idx];
    if (EPI && A.u2) x *= A.u2[bi + idx];
    tile[l * row + idx - l * n_in] = x;
  }
  for (int i = tid; i < CW; i += nthr) cs[i] = pk[i];
  __syncthreads();
  const int e0 = bound_first<L>(seg, P, n_out), rows = bound_rows<L>(seg, P, n_out);
  const T *const pl = tile + line * row;
  T w[1][L];
  {
    T win[L + 8];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) {
      const int j = e0 - 4 + k;
      if constexpr (PER) win[k] = pl[j < 0 ? j + n_in : (j >= n_in ? j - n_in : j)];
      else win[k] = pl[j < 0 ? 0 : (j >= n_in ? n_in - 1 : j)];
    }
    anchor_rhs<T, OP, L, PER>(A, q, win, w[0], seg, rows);
  }
  bound_solve<T, L, 1, 1>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
  if constexpr (PER) anchor_close<T, L>(A, w[0], cs, ends, line, seg, TL);
#pragma unroll
  for (int m = 0; m < L; ++m)
    if (m < rows) tile[line * row + e0 + m] = w[0][m];
  __syncthreads();
  T *const t = A.t[q];
  for (int idx = tid; idx < nl * n_out; idx += nthr) {
    const int l = small_div(idx, n_out, rno);
    T r = tile[l * row + idx - l * n_out];
    if constexpr (EPI) {
      if (A.mul) r *= A.mul[bo + idx];
      r = A.rc * r;
      if (A.acc[q]) r = A.ac * A.acc[q][bo + idx] + r;
    }
    t[bo + idx] = r;
  }
}

template <typename T, int OP, int L>
static void launch_anchor_yz(const AnchorArgs<T> &A, bool per, bool epi, dim3 grid, dim3 block, size_t sh,
                             hipStream_t st) {
  if constexpr (L == BoundShape<T>::L) {
    if (per) {
      if (epi) hipLaunchKernelGGL((anchor_yz_kernel<T, OP, L, true, true>), grid, block, sh, st, A);
      else hipLaunchKernelGGL((anchor_yz_kernel<T, OP, L, true, false>), grid, block, sh, st, A);
      return;
    }
    if (epi) {
      hipLaunchKernelGGL((anchor_yz_kernel<T, OP, L, false, true>), grid, block, sh, st, A);
      return;
    }
  }
  hipLaunchKernelGGL((anchor_yz_kernel<T, OP, L, false, false>), grid, block, sh, st, A);
}

template <typename T, int OP>
static void launch_anchor_x(const AnchorArgs<T> &A, bool per, bool epi, dim3 grid, dim3 block, size_t sh,
                            hipStream_t st) {
  constexpr int L = BoundShape<T>::L;
  if (per) {
    if (epi) hipLaunchKernelGGL((anchor_x_kernel<T, OP, L, true, true>), grid, block, sh, st, A);
    else hipLaunchKernelGGL((anchor_x_kernel<T, OP, L, true, false>), grid, block, sh, st, A);
  } else {
    if (epi) hipLaunchKernelGGL((anchor_x_kernel<T, OP, L, false, true>), grid, block, sh, st, A);
    else hipLaunchKernelGGL((anchor_x_kernel<T, OP, L, false, false>), grid, block, sh, st, A);
  }
}

// Covers a call whose coefficients are the library's own set of the
// direction, operator and parity, with the direction's own ends, and whose
// lines have a table (bounded_setup).  y and z lines run with full 128-byte
// rows: segments of the precision's length, or one row longer where those
// would need more than 1024 threads (plain bounded operators).
template <typename T>
int launch_anchored(const LineCall<T> &c, const LineTriple<T> *triple, bool *done, hipStream_t st) {
  *done = false;
  const Context *g = ctx();
  if (!g) return X3D_OK;
  const DirCoef &D = g->dir[c.dir];
  const bool per = c.tri.periodic != 0;
  const bool pv = c.op == OP_DERPV || c.op == OP_INTERPV, vp = c.op == OP_DERVP || c.op == OP_INTERVP;
  const int n_in = c.dir == 0 ? c.nx : (c.dir == 1 ? c.ny : c.nz);
  if (n_in != (pv ? D.nm : D.n) || c.n_out != (vp ? D.nm : D.n)) return X3D_OK;
  if (per != (D.bc1 == 0) || per != (D.bcn == 0)) return X3D_OK;
  if (!per && (c.bc1 != D.bc1 || c.bcn != D.bcn)) return X3D_OK;
  const int batch = triple ? 3 : 1;
  const bool epi = triple ? triple->acc[0] || triple->acc[1] || triple->acc[2]
                          : c.u2 || c.acc || c.mul || c.rc != T(1);
  auto own = [&](int par) -> bool {
    const BoundTab &b = g->btab[c.dir][c.op][par];
    if constexpr (sizeof(T) == 8) return b.set64[0] && (b.set64[0] == c.tri.pk || b.set64[1] == c.tri.pk);
    else return b.set32[0] && (b.set32[0] == c.tri.pk || b.set32[1] == c.tri.pk);
  };
  if (!triple && (c.npaire < 0 || c.npaire > 1 || !own(c.npaire))) return X3D_OK;
  bool longer = false;
  BoundShape<T> Y;
  BoundShape<T, BoundShape<T>::L + 1> Z;
  AnchorArgs<T> A{};
  A.row = (n_in > c.n_out ? n_in : c.n_out) | 1;
  dim3 block;
  size_t sh;
  if (c.dir == 0) {
    if (!Y.plan(c.n_out, 1, 1, [&](int TL) { return (size_t)TL * (A.row + 2); })) return X3D_OK;
  } else {
    auto ends = [](int TL) { return 2 * (size_t)TL; };
    if (!Y.plan(c.n_out, 1, 1, ends) || Y.TL * (int)sizeof(T) < 128) {
      if (per || epi || !Z.plan(c.n_out, 1, 1, ends) || Z.TL * (int)sizeof(T) < 128) return X3D_OK;
      longer = true;
    }
  }
  block = longer ? dim3(Z.TL, Z.P) : dim3(Y.TL, Y.P);
  sh = longer ? Z.shmem : Y.shmem;
  for (int i = 0; i < batch; ++i) {
    const BoundDev<T> t = bound_dev<T>(*g, c.dir, c.op, triple ? triple->par[i] : c.npaire, longer);
    if (!t.pk) return X3D_OK;
    A.pk[i] = t.pk;
    A.edge[i] = t.edge;
    A.P = t.P;
    A.K = std::max(A.K, t.K);
    A.u[i] = triple ? triple->u[i] : c.u;
    A.t[i] = triple ? triple->t[i] : c.t;
    A.acc[i] = triple ? triple->acc[i] : c.acc;
  }
  const size_t nout = (size_t)c.nx * c.ny * c.nz / n_in * c.n_out;
  const size_t nmax = std::max((size_t)c.nx * c.ny * c.nz, nout);
  if (nmax * sizeof(T) >= ((size_t)1 << 32)) return X3D_OK;
  A.u2 = c.u2; A.mul = c.mul; A.ac = c.ac; A.rc = c.rc; A.pp = c.pp;
  A.alfa = c.tri.alfa; A.rden = c.tri.rden;
  A.s = c.s;
  A.n_in = n_in;
  A.n_out = c.n_out;
  int TL = (int)block.x;
  if (c.dir == 0) {
    if (c.pp) return X3D_OK;
    A.na = c.ny * c.nz;
    const dim3 grid((A.na + TL - 1) / TL, 1, batch);
    switch (c.op) {
      case OP_DER1: launch_anchor_x<T, OP_DER1>(A, per, epi, grid, block, sh, st); break;
      case OP_DER2: launch_anchor_x<T, OP_DER2>(A, per, epi, grid, block, sh, st); break;
      case OP_DERVP: launch_anchor_x<T, OP_DERVP>(A, per, epi, grid, block, sh, st); break;
      case OP_INTERVP: launch_anchor_x<T, OP_INTERVP>(A, per, epi, grid, block, sh, st); break;
      case OP_DERPV: launch_anchor_x<T, OP_DERPV>(A, per, epi, grid, block, sh, st); break;
      default: launch_anchor_x<T, OP_INTERPV>(A, per, epi, grid, block, sh, st); break;
    }
  } else {
    if (c.dir == 1) {
      A.na = c.nx; A.nb = c.nz; A.se = c.nx;
      A.sb_in = (long long)c.nx * n_in;
      A.sb_out = (long long)c.nx * c.n_out;
    } else {
      A.na = c.nx * c.ny; A.nb = 1; A.se = A.na;
    }
    const dim3 grid((A.na + TL - 1) / TL, A.nb, batch);
    constexpr int L = BoundShape<T>::L;
#define X3D_ANCHOR(OP)                                                              \
  case OP:                                                                          \
    if (longer) launch_anchor_yz<T, OP, L + 1>(A, per, epi, grid, block, sh, st);   \
    else launch_anchor_yz<T, OP, L>(A, per, epi, grid, block, sh, st);              \
    break;
    switch (c.op) {
      X3D_ANCHOR(OP_DER1)
      X3D_ANCHOR(OP_DER2)
      X3D_ANCHOR(OP_DERVP)
      X3D_ANCHOR(OP_INTERVP)
      X3D_ANCHOR(OP_DERPV)
      X3D_ANCHOR(OP_INTERPV)
    }
#undef X3D_ANCHOR
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(X3D_ERR_HIP, std::string("anchored line launch: ") + hipGetErrorString(e));
  *done = true;
  return X3D_OK;
}

}  // namespace x3d
