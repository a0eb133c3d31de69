// Fused momentum and projection sweeps along bounded directions (free-slip and
// no-slip ends), the counterparts of momentum.hip and projection.hip for
// periodic ones, on the anchored segments of bounded_impl.h.
//
// Before, every derivative of such a direction was a launch of its own that
// read its operand, its epilogue's fields and wrote its result: ten fields
// moved per direction and component where these sweeps move four, and on a
// 65^3 box some 57 launches of 5-19 us per sub-step whose time was launch and
// load latency.  A sweep takes the three components in one launch
// (blockIdx.z).
#include <algorithm>
#include <cmath>
#include <vector>

#include "bounded_impl.h"

namespace x3d {

// ---------------------------------------------------------------- tables
namespace {

// One closure row applied to a function of the point index.
template <int OP, typename F>
double row_of(int i, int n_in, int n_out, const Sten<double> &s, int bc1, int bcn, int par, F U) {
  if (is_boundary_row<OP>(i, n_out)) return boundary_row<OP, double>(i, n_in, n_out, s, bc1, bcn, par, U);
  double v[9];
  for (int k = 0; k < 9; ++k) v[k] = U(i - 4 + k);
  return interior_row<OP, double, 9>(v, 4, s);
}

template <int OP>
void edge_weights(int n_in, int n_out, const Sten<double> &s, int bc1, int bcn, int par, double *W) {
  using F = EdgeForm<OP>;
  std::fill(W, W + EDGE_WORDS, 0.0);
  for (int end = 0; end < 2; ++end)
    for (int q = 0; q < F::NR; ++q) {
      const int i = end == 0 ? q : n_out - 1 - q;
      double w[8] = {};
      // the row's value on the function of the distance from this end that
      // the weight multiplies: a point, or the sums of differences
      auto on = [&](auto f) {
        return row_of<OP>(i, n_in, n_out, s, bc1, bcn, par, [&](int j) { return f(end == 0 ? j : n_in - 1 - j); });
      };
      for (int j = 0; j < F::NE(q); ++j) {
        if (F::KIND == 0) w[j] = on([&](int d) { return d == j ? 1.0 : 0.0; });
        else if (j == 0) w[j] = on([](int) { return 1.0; });
        else if (F::KIND == 1) w[j] = on([&](int d) { return d >= j ? 1.0 : 0.0; });
        else if (j == 1) w[j] = on([](int d) { return (double)d; });
        else w[j] = on([&](int d) { return d > j - 1 ? (double)(d - j + 1) : 0.0; });
      }
      // weights that vanish for the row's form and come out as rounding
      double top = 0.0;
      for (int j = 0; j < 8; ++j) {
        const double p = on([&](int d) { return d == j ? 1.0 : 0.0; });
        top = std::max(top, std::fabs(p));
      }
      for (int j = 0; j < 8; ++j) W[(end * 4 + q) * 8 + j] = std::fabs(w[j]) < 1e-13 * top ? 0.0 : w[j];
    }
}

void edge_table(int op, int n_in, int n_out, const Sten<double> &s, int bc1, int bcn, int par, double *W) {
  switch (op) {
    case OP_DER1: edge_weights<OP_DER1>(n_in, n_out, s, bc1, bcn, par, W); break;
    case OP_DER2: edge_weights<OP_DER2>(n_in, n_out, s, bc1, bcn, par, W); break;
    case OP_DERVP: edge_weights<OP_DERVP>(n_in, n_out, s, bc1, bcn, par, W); break;
    case OP_INTERVP: edge_weights<OP_INTERVP>(n_in, n_out, s, bc1, bcn, par, W); break;
    case OP_DERPV: edge_weights<OP_DERPV>(n_in, n_out, s, bc1, bcn, par, W); break;
    default: edge_weights<OP_INTERPV>(n_in, n_out, s, bc1, bcn, par, W); break;
  }
}

// The packed factors of a set on anchored segments of L rows (their
// Sherman-Morrison word too, zero in the rows between), and the chain depth of
// those segments.
std::vector<double> padded_rows(const TriSet &t, int n, int L, double tol, int *P, int *K) {
  *P = (n + L - 1) / L;
  std::vector<double> pk(4 * (size_t)*P * L), gf(*P, 1.0), gb(*P, 1.0);
  for (int s = 0; s < *P; ++s) {
    const int first = s == *P - 1 ? n - L : s * L, rows = s == *P - 2 ? n - (*P - 1) * L : L;
    for (int m = 0; m < L; ++m) {
      double *q = &pk[4 * ((size_t)s * L + m)];
      if (m < rows) {
        const int e = first + m;
        q[0] = t.fs[e];
        q[1] = t.fw[e];
        q[2] = t.ff[e] * t.fw[e];
        q[3] = t.sm[e];
      } else {
        q[0] = -1.0;
        q[2] = -1.0;
      }
      gf[s] *= std::fabs(q[0]);
      gb[s] *= std::fabs(q[2]);
    }
  }
  *K = chain_depth(gf, gb, tol);
  return pk;
}

// One precision's table of segments of L rows, packed rows, then the weights,
// appended to those of the other operators.
template <typename T>
void append_table(const TriSet &t, int n, int L, double tol, const double *W, std::vector<unsigned char> &all,
                  AnchorTab<T> *out) {
  std::vector<double> p = padded_rows(t, n, L, tol, &out->P, &out->K);
  p.insert(p.end(), W, W + EDGE_WORDS);
  const std::vector<T> h(p.begin(), p.end());
  all.resize((all.size() + 15) / 16 * 16);
  out->off = all.size();
  const auto *b = reinterpret_cast<const unsigned char *>(h.data());
  all.insert(all.end(), b, b + h.size() * sizeof(T));
}

template <typename T>
void append_tables(const TriSet &t, int n, const double *W, std::vector<unsigned char> &all, AnchorTab<T> (&out)[2]) {
  constexpr int L = sizeof(T) == 8 ? SEG_L64 : SEG_L32;
  const double tol = sizeof(T) == 8 ? 1e-18 : 1e-9;
  if (n < 2 * L) return;
  append_table<T>(t, n, L, tol, W, all, &out[0]);
  if (n >= 2 * (L + 1)) append_table<T>(t, n, L + 1, tol, W, all, &out[1]);
}

template <typename T>
void place_tables(unsigned char *dev, AnchorTab<T> (&t)[2]) {
  for (auto &q : t)
    if (q.P) q.pk = reinterpret_cast<T *>(dev + q.off);
}

}  // namespace

// Lines of two segments or more get tables, periodic ones only where neither
// the wavefront kernels (x) nor whole segments (y, z) cover them.  One
// allocation and one copy for all: with two of each a table, up to 144 tables,
// x3d_init took 2.4 ms on a 65^3 free-slip box, 0.86 without any, and takes 1.0.
int bounded_setup(Context &c) {
  std::vector<unsigned char> all;
  for (int d = 0; d < 3; ++d) {
    const DirCoef &D = c.dir[d];
    const bool per = D.bc1 == 0;
    if (per != (D.bcn == 0)) continue;
    if (per) {
      const int V = D.n / 64;
      if (d == 0 ? (D.n % 64 == 0 && (V == 1 || V == 2 || V == 4 || V == 8)) : D.n % SEG_L32 == 0) continue;
    }
    for (int op = 0; op < 6; ++op)
      for (int par = 0; par < 2; ++par) {
        // parities the reference has: both for the derivatives on the
        // velocity points, odd (0) and even (1) operands alike; the even one
        // for the other staggered operators
        if (!per && par == 0 && (op == OP_INTERVP || op == OP_DERPV || op == OP_INTERPV)) continue;
        LineCall<double> call;
        X3D_TRY(make_line_call<double>(c, d, op, par, &call));
        int set = -1;
        for (size_t q = 0; q < c.sets.size(); ++q)
          if (c.sets[q].d64 == call.tri.pk) set = (int)q;
        if (set < 0) return fail(X3D_ERR_STATE, "bounded tables: unknown coefficient set");
        const TriSet &t = c.sets[set];
        const int n_out = call.n_out, n_in = op == OP_DERPV || op == OP_INTERPV ? D.nm : D.n;
        if (n_in < 8 || n_out < 8) continue;
        BoundTab &b = c.btab[d][op][par];
        double W[EDGE_WORDS] = {};
        if (!per) edge_table(op, n_in, n_out, D.s, D.bc1, D.bcn, par, W);
        b.set64[0] = t.d64;
        b.set32[0] = t.d32;
        for (const TriSet &f : c.sets)
          if (f.name[0] == t.name[0] && same_set(f, t)) {
            b.set64[1] = f.d64;
            b.set32[1] = f.d32;
            break;
          }
        append_tables<double>(t, n_out, W, all, b.t64);
        append_tables<float>(t, n_out, W, all, b.t32);
      }
  }
  if (all.empty()) return X3D_OK;
  X3D_HIP(hipMalloc(&c.btab_mem, all.size()));
  X3D_HIP(hipMemcpy(c.btab_mem, all.data(), all.size(), hipMemcpyHostToDevice));
  for (auto &d : c.btab)
    for (auto &o : d)
      for (BoundTab &b : o) {
        place_tables<double>(static_cast<unsigned char *>(c.btab_mem), b.t64);
        place_tables<float>(static_cast<unsigned char *>(c.btab_mem), b.t32);
      }
  return X3D_OK;
}

void bounded_free(Context &c) {
  if (c.btab_mem) (void)hipFree(c.btab_mem);
  c.btab_mem = nullptr;
  for (auto &d : c.btab)
    for (auto &o : d)
      for (BoundTab &b : o) b = BoundTab();
}

// ---------------------------------------------------------------- momentum
template <typename T>
struct BMomArgs {
  const T *u[3], *acc[3];
  T *out[3];
  // tables of D1(u_d u_c), D1(u_c), D2(u_c): [0] for components across the
  // sweep, [1] for the component along it (the parities swap)
  const T *pk[2][3], *edge[2][3];
  Sten<T> s;
  T xnu;
  int dir, n, P, K;
  int na, nb;                   // lines (a fastest) of a y or z sweep; x: na lines in all
  long long sb, se;             // strides of b and of a line's points (a has stride 1)
  int row;                      // x: LDS words of a line
  const T *m1, *m2, *m4;        // stretched y: ppy, pp2y, pp4y*ppy (null: uniform)
  MomUpdate<T> up;              // x sweep
};

// Blocks up to this many threads run a kernel whose register budget is theirs:
// the budget of 1024 threads, 128 registers, spilled 10 (L = 9, NT = 2) to 14
// (L = 8, NT = 3, x) of them: 65^3 FP64 16.6 -> 14.4 us a y or z sweep, the
// channel's y sweep 96 -> 84.  (Blocks of x lines are smaller: their LDS.)
constexpr int BMOM_FEW = 512;
// Larger blocks of y and z lines.  A solver's bounded lines have 2^k + 1 points
// (the pressure solve's sizes), and only 513 of them need such blocks: in FP64
// 65 x 8 threads with segments of 8 rows and two tables (three do not fit in
// LDS), in FP32 31 x 32 with segments of 17.  Others are not compiled.
template <typename T>
constexpr bool bmom_many(bool longer, int nt) {
  return sizeof(T) == 8 ? !longer && nt == 2 : longer;
}

// -1/2 D1(u_d u_c) - 1/2 u_d D1(u_c) + nu D2(u_c) of the rows of a segment:
// the right-hand sides from the windows.
template <typename T, int L>
__device__ __forceinline__ void bmom_rhs(const BMomArgs<T> &A, const T (&wc)[L + 8], const T (&wd)[L + 4],
                                         T (&w)[3][L], const bool along, const int seg, const int rows) {
  T p[L + 4];
#pragma unroll
  for (int k = 0; k < L + 4; ++k) p[k] = wd[k] * wc[k + 2];
  T c2[L + 4];
#pragma unroll
  for (int k = 0; k < L + 4; ++k) c2[k] = wc[k + 2];
  bound_rhs<OP_DER1, T, L, 2>(p, w[0], A.s, A.edge[along][0], seg, A.P, rows);
  bound_rhs<OP_DER1, T, L, 2>(c2, w[1], A.s, A.edge[along][1], seg, A.P, rows);
  bound_rhs<OP_DER2, T, L, 4>(wc, w[2], A.s, A.edge[along][2], seg, A.P, rows);
}

// y and z lines, straight from memory: a block's rows are TL consecutive
// points (128 bytes), each input is read once.  NT: 2 where the two first
// derivatives have the same factors (no-slip ends), else 3.  Bound by the
// latency of its loads and of the two carry chains, like mom_yz_kernel.
template <typename T, int L, int NT, int MAXT>
__global__ void __launch_bounds__(MAXT) bmom_yz_kernel(const BMomArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n = A.n;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + NT * CW, *cb = cf + 3 * P * TL, *gf = cb + 3 * P * TL, *gb = gf + NT * P;
  T *met = gb + NT * P;         // 3n words with a stretched mesh
  const int comp = (int)blockIdx.z;
  const bool along = comp == A.dir;
  const T *const uc = A.u[comp], *const ud = A.u[A.dir], *const acc = A.acc[comp];
  T *const out = A.out[comp];
  const int a = (int)blockIdx.x * TL + line, b = (int)blockIdx.y;
  const bool active = a < A.na;
  const int al = active ? a : A.na - 1;
  const int e0 = bound_first<L>(seg, P, n), rows = bound_rows<L>(seg, P, n);
  const unsigned base = ((unsigned)al + (unsigned)b * (unsigned)A.sb) * (unsigned)sizeof(T);
  const unsigned step = (unsigned)A.se * (unsigned)sizeof(T);
  auto clamp = [&](int j) { return (unsigned)(j < 0 ? 0 : (j >= n ? n - 1 : j)); };
  const T *src[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) src[t] = A.pk[along][NT == 2 ? t + 1 : t];
  __builtin_amdgcn_s_setprio(3);
  BoundCopy<T, NT> tc;
  tc.load(src, tid, nthr, CW);
  T w[3][L], dd[L];
  {
    T wc[L + 8], wd[L + 4];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) wc[k] = at(uc, base + clamp(e0 - 4 + k) * step);
#pragma unroll
    for (int k = 0; k < L + 4; ++k) wd[k] = at(ud, base + clamp(e0 - 2 + k) * step);
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int m = 0; m < L; ++m) dd[m] = wd[m + 2];
    bmom_rhs<T, L>(A, wc, wd, w, along, seg, rows);
  }
  const T *const msrc[3] = {A.m1, A.m2, A.m4};
  BoundCopy<T, 3, 1> mc;
  if (A.m1) mc.load(msrc, tid, nthr, n);
  tc.store(cs, src, tid, nthr, CW);
  if (A.m1) mc.store(met, msrc, tid, nthr, n);
  __syncthreads();
  bound_solve<T, L, 3, NT>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
  if (!active) return;
  // the row offsets are worked out again rather than held through the solve
  // (they spilled)
  int e1 = e0;
  asm volatile("" : "+v"(e1));
  if (A.m1) {
#pragma unroll
    for (int m = 0; m < L; ++m) {
      const int e = e1 + m < n ? e1 + m : n - 1;
      const T p1 = met[e], p2 = met[n + e], p4 = met[2 * n + e];
      w[0][m] = T(-0.5) * (p1 * w[0][m]) + T(-0.5) * (dd[m] * (p1 * w[1][m])) +
                A.xnu * (p2 * w[2][m]) - A.xnu * (p4 * w[1][m]);
    }
  } else {
#pragma unroll
    for (int m = 0; m < L; ++m) w[0][m] = T(-0.5) * w[0][m] + T(-0.5) * (dd[m] * w[1][m]) + A.xnu * w[2][m];
  }
  // loads of rows past the segment's repeat its last one, without branches
  const unsigned ob = base + (unsigned)e1 * step;
  if (acc) {
    // acc may be out: this thread's points are all read before any is written
    T ac[L];
#pragma unroll
    for (int m = 0; m < L; ++m) ac[m] = at(acc, ob + (unsigned)(m < rows ? m : rows - 1) * step);
#pragma unroll
    for (int m = 0; m < L; ++m) w[0][m] = ac[m] + w[0][m];
  }
  store_rows<T, L, false>(out, ob, step, w[0], rows);
}

// x lines: TL whole lines are one contiguous piece of memory, staged in LDS
// (odd line stride: the threads of a wave fall into different banks), solved
// as above and written back in order with the velocity update.  A thread has
// all its loads of a stage in flight together: one after another they were a
// chain of memory latencies (65^3 FP64: 20.8 -> 18.2 us; bproj_x_kernel 13.4
// -> 10.1).
template <typename T, int L, int NT>
__global__ void __launch_bounds__(BMOM_FEW) bmom_x_kernel(const BMomArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n = A.n, row = A.row;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + NT * CW, *cb = cf + 3 * P * TL, *gf = cb + 3 * P * TL, *gb = gf + NT * P;
  T *td = gb + NT * P, *tt = td + TL * row;   // u_d; u_c (along the sweep: free)
  const int comp = (int)blockIdx.z;
  const bool along = comp == 0;
  const int l0 = (int)blockIdx.x * TL;
  const int tot = min(TL, A.na - l0) * n;
  const unsigned base = (unsigned)l0 * (unsigned)n;   // (a field is under 4 GiB)
  const float rn = 1.0f / (float)n;
  const T *src[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) src[t] = A.pk[along][NT == 2 ? t + 1 : t];
  BoundCopy<T, NT> cp;
  cp.load(src, tid, nthr, CW);
  {
    // n <= P L: at most L points a thread
    T r0[L], r1[L];
#pragma unroll
    for (int m = 0; m < L; ++m) {
      const unsigned o = (base + (unsigned)min(tid + m * nthr, tot - 1)) * (unsigned)sizeof(T);
      r0[m] = at(A.u[0], o);
      if (!along) r1[m] = at(A.u[comp], o);
    }
#pragma unroll
    for (int m = 0; m < L; ++m) {
      const int idx = tid + m * nthr;
      if (idx >= tot) continue;
      const int l = small_div(idx, n, rn), q = l * row + idx - l * n;
      td[q] = r0[m];
      if (!along) tt[q] = r1[m];
    }
  }
  cp.store(cs, src, tid, nthr, CW);
  __syncthreads();
  const int e0 = bound_first<L>(seg, P, n), rows = bound_rows<L>(seg, P, n);
  auto clamp = [&](int j) { return j < 0 ? 0 : (j >= n ? n - 1 : j); };
  const T *const pc = (along ? td : tt) + line * row, *const pd = td + line * row;
  T w[3][L], dd[L];
  {
    T wc[L + 8], wd[L + 4];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) wc[k] = pc[clamp(e0 - 4 + k)];
#pragma unroll
    for (int k = 0; k < L + 4; ++k) wd[k] = pd[clamp(e0 - 2 + k)];
#pragma unroll
    for (int m = 0; m < L; ++m) dd[m] = wd[m + 2];
    bmom_rhs<T, L>(A, wc, wd, w, along, seg, rows);
  }
  bound_solve<T, L, 3, NT>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
  // the tile of the other field takes the result: u_c stays for the update
  T *const tr = along ? tt : td;
#pragma unroll
  for (int m = 0; m < L; ++m)
    if (m < rows)
      tr[line * row + e0 + m] = T(-0.5) * w[0][m] + T(-0.5) * (dd[m] * w[1][m]) + A.xnu * w[2][m];
  __syncthreads();
  const T *const tc = along ? td : tt;
  const MomUpdate<T> &U = A.up;
  // the points' indices are worked out again rather than held through the solve
  int t1 = tid;
  asm volatile("" : "+v"(t1));
  constexpr int H = 4;
#pragma unroll
  for (int m0 = 0; m0 < L; m0 += H) {
    T ac[H], f2[H], f3[H], rot[H];
    double uo[H];
#pragma unroll
    for (int h = 0; h < H; ++h) {
      if (m0 + h >= L) continue;
      const unsigned e = base + (unsigned)min(t1 + (m0 + h) * nthr, tot - 1), o = e * (unsigned)sizeof(T);
      ac[h] = A.acc[comp] ? at(A.acc[comp], o) : T(0);
      f2[h] = U.nterms >= 2 ? at(U.f2[comp], o) : T(0);
      f3[h] = U.nterms >= 3 ? at(U.f3[comp], o) : T(0);
      rot[h] = U.rot[comp] ? at(U.rot[comp], o) : T(0);
      if constexpr (sizeof(T) == 4) uo[h] = U.u64[comp][e];
    }
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const int idx = t1 + (m0 + h) * nthr;
      if (m0 + h >= L || idx >= tot) continue;
      const int l = small_div(idx, n, rn), i = idx - l * n;
      const unsigned e = base + (unsigned)idx;
      if constexpr (sizeof(T) == 8) uo[h] = (double)tc[l * row + i];
      const T f1 = mom_forced(U, comp, ac[h] + tr[l * row + i], rot[h]);
      at(A.out[comp], e * (unsigned)sizeof(T)) = f1;
      const int ln = l0 + l, k = ln / U.ny, j = ln - k * U.ny;
      const double un = pre_correc_point(U, comp, i, j, k, mom_increment(U, f1, f2[h], f3[h]) + uo[h]);
      U.u64[comp][e] = un;
      if constexpr (sizeof(T) == 4) at(U.u32[comp], e * (unsigned)sizeof(T)) = (float)un;
    }
  }
}

template <typename T>
static bool bmom_plan(const Context &c, int dir, BoundPick<T> *Y, int *nt) {
  const DirCoef &D = c.dir[dir];
  const bool same = same_set(c.sets[D.set_d1_even], c.sets[D.set_d1_odd]);
  *nt = same ? 2 : 3;
  for (int op : {OP_DER1, OP_DER2})
    for (int par = 0; par < 2; ++par)
      if (!bound_dev<T>(c, dir, op, par).pk) return false;
  const int row = D.n | 1, n = D.n;
  const bool stretched = dir == 1 && c.p.istret != 0;
  return Y->plan(n, *nt, 3, [&](int TL) {
    return dir == 0 ? 2 * (size_t)TL * row : (stretched ? 3 * (size_t)n : (size_t)0);
  }) && (Y->TL * Y->P <= BMOM_FEW || (dir != 0 && bmom_many<T>(Y->longer, *nt)));
}

template <typename T>
bool bounded_momentum_ok(const Context &c, int dir) {
  BoundPick<T> Y;
  int nt;
  return bmom_plan<T>(c, dir, &Y, &nt);
}
template bool bounded_momentum_ok<double>(const Context &, int);
template bool bounded_momentum_ok<float>(const Context &, int);

template <typename T, int L>
static void launch_bmom_x(const BMomArgs<T> &A, int nt, dim3 grid, dim3 block, size_t sh, hipStream_t st) {
  if (nt == 2) hipLaunchKernelGGL((bmom_x_kernel<T, L, 2>), grid, block, sh, st, A);
  else hipLaunchKernelGGL((bmom_x_kernel<T, L, 3>), grid, block, sh, st, A);
}

template <typename T, int L, int NT>
static void launch_bmom_nt(const BMomArgs<T> &A, dim3 grid, dim3 block, size_t sh, hipStream_t st) {
  if constexpr (bmom_many<T>(L != BoundShape<T>::L, NT)) {
    if (block.x * block.y > BMOM_FEW) {
      hipLaunchKernelGGL((bmom_yz_kernel<T, L, NT, 1024>), grid, block, sh, st, A);
      return;
    }
  }
  hipLaunchKernelGGL((bmom_yz_kernel<T, L, NT, BMOM_FEW>), grid, block, sh, st, A);
}

template <typename T, int L>
static void launch_bmom_yz(const BMomArgs<T> &A, int nt, dim3 grid, dim3 block, size_t sh, hipStream_t st) {
  if (nt == 2) launch_bmom_nt<T, L, 2>(A, grid, block, sh, st);
  else launch_bmom_nt<T, L, 3>(A, grid, block, sh, st);
}

template <typename T>
int launch_bounded_momentum(const Context &c, int dir, const MomIO<T> &io, hipStream_t st) {
  const int nx = c.p.nx, ny = c.p.ny, nz = c.p.nz;
  BoundPick<T> Y;
  int nt = 0;
  if (!bmom_plan<T>(c, dir, &Y, &nt)) return fail(X3D_ERR_UNSUPPORTED, "bounded momentum sweep: line not covered");
  if ((size_t)nx * ny * nz * sizeof(T) >= ((size_t)1 << 32))
    return fail(X3D_ERR_UNSUPPORTED, "bounded momentum sweep: field larger than 4 GiB");
  const DirCoef &D = c.dir[dir];
  constexpr int L = BoundShape<T>::L;
  BMomArgs<T> A{};
  for (int i = 0; i < 3; ++i) {
    A.u[i] = io.u[i];
    A.acc[i] = io.acc[i];
    A.out[i] = io.out[i];
  }
  for (int along = 0; along < 2; ++along) {
    // the product u_d u_c is even along d for the component along it, odd
    // otherwise; u_c the other way round (transeq.f90:125-146)
    const BoundDev<T> t[3] = {bound_dev<T>(c, dir, OP_DER1, along, Y.longer),
                              bound_dev<T>(c, dir, OP_DER1, 1 - along, Y.longer),
                              bound_dev<T>(c, dir, OP_DER2, 1 - along, Y.longer)};
    for (int q = 0; q < 3; ++q) {
      A.pk[along][q] = t[q].pk;
      A.edge[along][q] = t[q].edge;
      A.K = std::max(A.K, t[q].K);
    }
  }
  A.s = cast_sten<T>(D.s);
  A.xnu = (T)c.xnu;
  A.dir = dir;
  A.n = D.n;
  A.P = Y.P;
  const dim3 block(Y.TL, Y.P);
  if (dir == 0) {
    A.na = ny * nz;
    A.row = D.n | 1;
    X3D_TRY(fill_update<T>(c, io, &A.up));
    const dim3 grid((A.na + Y.TL - 1) / Y.TL, 1, 3);
    if (Y.longer) launch_bmom_x<T, L + 1>(A, nt, grid, block, Y.shmem, st);
    else launch_bmom_x<T, L>(A, nt, grid, block, Y.shmem, st);
  } else {
    if (io.nterms) return fail(X3D_ERR_ARG, "the velocity update belongs to the x sweep");
    if (dir == 1) {
      A.na = nx; A.nb = nz; A.sb = (long long)nx * ny; A.se = nx;
      if (c.p.istret != 0) {
        A.m1 = sizeof(T) == 8 ? (const T *)c.ppy64 : (const T *)c.ppy32;
        A.m2 = sizeof(T) == 8 ? (const T *)c.pp2y64 : (const T *)c.pp2y32;
        A.m4 = sizeof(T) == 8 ? (const T *)c.pp4yy64 : (const T *)c.pp4yy32;
      }
    } else {
      // every z line starts in the first plane: one run of nx*ny lines
      A.na = nx * ny; A.nb = 1; A.sb = 0; A.se = (long long)nx * ny;
    }
    const dim3 grid((A.na + Y.TL - 1) / Y.TL, A.nb, 3);
    if (Y.longer) launch_bmom_yz<T, L + 1>(A, nt, grid, block, Y.shmem, st);
    else launch_bmom_yz<T, L>(A, nt, grid, block, Y.shmem, st);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(X3D_ERR_HIP, std::string("bounded momentum launch: ") + hipGetErrorString(e));
  return X3D_OK;
}
template int launch_bounded_momentum<double>(const Context &, int, const MomIO<double> &, hipStream_t);
template int launch_bounded_momentum<float>(const Context &, int, const MomIO<float> &, hipStream_t);

// ---------------------------------------------------------------- projection
template <typename T>
struct BProjArgs {
  const T *in[3];
  T *out[3];
  const T *pkI, *pkD, *edgeI, *edgeD;
  Sten<T> s;
  int n_in, n_out, P, K;
  int na, nb;
  long long sb_in, sb_out, se;  // y/z: strides of b in and out, and of a line's points
  int row;                      // x: LDS words of a line
  const T *met;                 // stretched y: the derivative's metric (null: none)
  double *divp;                 // DIV_Z: per-block max and sum of |div u*|
  CorVel cv;                    // GRAD_X
};

// y and z sweeps of the divergence and of the gradient (the recipes of
// projection.hip).  Input and output lines differ in length, so outputs never
// overwrite inputs.
template <typename T, int L, int SW>
__global__ void __launch_bounds__(1024) bproj_yz_kernel(const BProjArgs<T> A) {
  using R = Recipe<SW>;
  constexpr int OPI = R::PV ? OP_INTERPV : OP_INTERVP;
  constexpr int OPD = R::PV ? OP_DERPV : OP_DERVP;
  constexpr int N = R::NI + 1;
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n_in = A.n_in, n_out = A.n_out;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + 2 * CW, *cb = cf + N * P * TL, *gf = cb + N * P * TL, *gb = gf + 2 * P;
  const int a = (int)blockIdx.x * TL + line, b = (int)blockIdx.y;
  const bool active = a < A.na;
  const int al = active ? a : A.na - 1;
  const int e0 = bound_first<L>(seg, P, n_out), rows = bound_rows<L>(seg, P, n_out);
  const unsigned ib = ((unsigned)al + (unsigned)b * (unsigned)A.sb_in) * (unsigned)sizeof(T);
  const unsigned step = (unsigned)A.se * (unsigned)sizeof(T);
  auto clamp = [&](int j) { return (unsigned)(j < 0 ? 0 : (j >= n_in ? n_in - 1 : j)); };
  const T *const src[2] = {A.pkI, A.pkD};
  __builtin_amdgcn_s_setprio(3);
  BoundCopy<T, 2> tc;
  tc.load(src, tid, nthr, CW);
  T w[N][L];
#pragma unroll
  for (int i = 0; i < R::NIN; ++i) {
    T win[L + 8];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) win[k] = at(A.in[i], ib + clamp(e0 - 4 + k) * step);
    if (i == R::I0) bound_rhs<OPI, T, L, 4>(win, w[0], A.s, A.edgeI, seg, P, rows);
    if constexpr (R::NI == 2) {
      if (i == R::I1) bound_rhs<OPI, T, L, 4>(win, w[1], A.s, A.edgeI, seg, P, rows);
    }
    if (i == R::D0) bound_rhs<OPD, T, L, 4>(win, w[N - 1], A.s, A.edgeD, seg, P, rows);
  }
  __builtin_amdgcn_s_setprio(0);
  tc.store(cs, src, tid, nthr, CW);
  __syncthreads();
  bound_solve<T, L, N, 2>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
  if (A.met) {
#pragma unroll
    for (int m = 0; m < L; ++m) w[N - 1][m] *= A.met[e0 + m < n_out ? e0 + m : n_out - 1];
  }
  const unsigned ob = ((unsigned)al + (unsigned)b * (unsigned)A.sb_out) * (unsigned)sizeof(T) + (unsigned)e0 * step;
  if constexpr (SW == SW_DIV_Y || SW == SW_DIV_Z) {
#pragma unroll
    for (int m = 0; m < L; ++m) w[0][m] += w[N - 1][m];
  }
  if (active) {
    store_rows<T, L, R::PV>(A.out[0], ob, step, w[0], rows);
    if constexpr (SW == SW_DIV_Y) store_rows<T, L, false>(A.out[1], ob, step, w[1], rows);
    if constexpr (R::PV) store_rows<T, L, true>(A.out[1], ob, step, w[N - 1], rows);
    if constexpr (SW == SW_GRAD_Y) store_rows<T, L, true>(A.out[2], ob, step, w[1], rows);
  }
  if constexpr (SW == SW_DIV_Z) {
    if (A.divp) {
      double mx = -1.0e300, sm = 0.0;
      if (active) {
#pragma unroll
        for (int m = 0; m < L; ++m) {
          if (m >= rows) continue;
          const double v = (double)w[0][m];
          mx = v > mx ? v : mx;
          sm += fabs(v);
        }
      }
      block_max_sum(mx, sm, tid, nthr, A.divp);
    }
  }
}

// x sweeps: the three fields are independent (blockIdx.z): the derivative of
// the x component, the interpolations of the other two; the gradient sweep
// subtracts its result from the velocity (cor_vel, navier.f90:206-249).
template <typename T, int L, bool PV>
__global__ void __launch_bounds__(1024) bproj_x_kernel(const BProjArgs<T> A) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);
  const int TL = blockDim.x, P = A.P, n_in = A.n_in, n_out = A.n_out, row = A.row;
  const int line = threadIdx.x, seg = threadIdx.y;
  const int tid = seg * TL + line, nthr = TL * P;
  const int CW = 4 * P * L;
  T *cs = smem, *cf = cs + CW, *cb = cf + P * TL, *gf = cb + P * TL, *gb = gf + P, *tile = gb + P;
  const int comp = (int)blockIdx.z;
  const int l0 = (int)blockIdx.x * TL;
  const int nl = min(TL, A.na - l0);
  const T *const in = A.in[comp], *const pk = comp == 0 ? A.pkD : A.pkI;
  const long long bi = (long long)l0 * n_in, bo = (long long)l0 * n_out;
  const float rni = 1.0f / (float)n_in, rno = 1.0f / (float)n_out;
  const T *const src[1] = {pk};
  BoundCopy<T, 1> cp;
  cp.load(src, tid, nthr, CW);
  {
    // n_in <= P L + 1: at most L + 1 points a thread (L where n_in < n_out)
    constexpr int R = PV ? L : L + 1;
    const int tot = nl * n_in;
    T r[R];
#pragma unroll
    for (int m = 0; m < R; ++m) r[m] = in[bi + min(tid + m * nthr, tot - 1)];
#pragma unroll
    for (int m = 0; m < R; ++m) {
      const int idx = tid + m * nthr;
      if (idx >= tot) continue;
      const int l = small_div(idx, n_in, rni);
      tile[l * row + idx - l * n_in] = r[m];
    }
  }
  cp.store(cs, src, tid, nthr, CW);
  __syncthreads();
  const int e0 = bound_first<L>(seg, P, n_out), rows = bound_rows<L>(seg, P, n_out);
  const T *const pl = tile + line * row;
  T w[1][L];
  {
    T win[L + 8];
#pragma unroll
    for (int k = 0; k < L + 8; ++k) {
      const int j = e0 - 4 + k;
      win[k] = pl[j < 0 ? 0 : (j >= n_in ? n_in - 1 : j)];
    }
    if (comp == 0) bound_rhs<PV ? OP_DERPV : OP_DERVP, T, L, 4>(win, w[0], A.s, A.edgeD, seg, P, rows);
    else bound_rhs<PV ? OP_INTERPV : OP_INTERVP, T, L, 4>(win, w[0], A.s, A.edgeI, seg, P, rows);
  }
  bound_solve<T, L, 1, 1>(w, cs, cf, cb, gf, gb, line, seg, TL, P, A.K);
#pragma unroll
  for (int m = 0; m < L; ++m)
    if (m < rows) tile[line * row + e0 + m] = w[0][m];
  __syncthreads();
  int t1 = tid;   // as in bmom_x_kernel
  asm volatile("" : "+v"(t1));
  const int tot = nl * n_out;
  T *const out = A.out[comp];
  double *const u64 = A.cv.u64[comp];
  double uo[L];
  if (PV && A.cv.apply) {
#pragma unroll
    for (int m = 0; m < L; ++m) uo[m] = u64[bo + min(t1 + m * nthr, tot - 1)];
  }
#pragma unroll
  for (int m = 0; m < L; ++m) {
    const int idx = t1 + m * nthr;
    if (idx >= tot) continue;
    const int l = small_div(idx, n_out, rno), i = idx - l * n_out;
    const T g = tile[l * row + i];
    if constexpr (!PV) {
      out[bo + idx] = g;
    } else {
      const int ln = l0 + l, k = ln / A.cv.ny, j = ln - k * A.cv.ny;
      store_wall(A.cv, comp, i, j, k, g);
      if (A.cv.apply) {
        const double u = uo[m] - (double)g;
        u64[bo + idx] = u;
        if (A.cv.u32[comp]) A.cv.u32[comp][bo + idx] = (float)u;
      }
    }
  }
}

// Rows of the two projection passes along a direction.
static int proj_out(const DirCoef &D, bool pv) { return pv ? D.n : D.nm; }
static int proj_in(const DirCoef &D, bool pv) { return pv ? D.nm : D.n; }

template <typename T>
static bool bproj_plan(const Context &c, int dir, bool pv, BoundPick<T> *Y) {
  const DirCoef &D = c.dir[dir];
  const int row = D.n | 1;
  if (dir == 0) return Y->plan(proj_out(D, pv), 1, 1, [&](int TL) { return (size_t)TL * row; });
  return Y->plan(proj_out(D, pv), 2, 3);
}

template <typename T>
bool bounded_projection_ok(const Context &c, int dir) {
  BoundPick<T> Y;
  if (!bound_dev<T>(c, dir, OP_DERVP, 0).pk) return false;
  for (int op : {OP_INTERVP, OP_DERPV, OP_INTERPV})
    if (!bound_dev<T>(c, dir, op, 1).pk) return false;
  return bproj_plan<T>(c, dir, false, &Y) && bproj_plan<T>(c, dir, true, &Y);
}
template bool bounded_projection_ok<double>(const Context &, int);
template bool bounded_projection_ok<float>(const Context &, int);

template <typename T, int L>
static void launch_bproj_x(const BProjArgs<T> &A, bool pv, dim3 grid, dim3 block, size_t sh, hipStream_t st) {
  if (pv) hipLaunchKernelGGL((bproj_x_kernel<T, L, true>), grid, block, sh, st, A);
  else hipLaunchKernelGGL((bproj_x_kernel<T, L, false>), grid, block, sh, st, A);
}

template <typename T, int L>
static void launch_bproj_yz(const BProjArgs<T> &A, int sw, dim3 grid, dim3 block, size_t sh, hipStream_t st) {
  switch (sw) {
    case SW_DIV_Y: hipLaunchKernelGGL((bproj_yz_kernel<T, L, SW_DIV_Y>), grid, block, sh, st, A); break;
    case SW_DIV_Z: hipLaunchKernelGGL((bproj_yz_kernel<T, L, SW_DIV_Z>), grid, block, sh, st, A); break;
    case SW_GRAD_Z: hipLaunchKernelGGL((bproj_yz_kernel<T, L, SW_GRAD_Z>), grid, block, sh, st, A); break;
    default: hipLaunchKernelGGL((bproj_yz_kernel<T, L, SW_GRAD_Y>), grid, block, sh, st, A); break;
  }
}

template <typename T>
int launch_bounded_projection(const Context &c, int sw, const ProjIO<T> &io, hipStream_t st) {
  const int dir = (sw == SW_DIV_X || sw == SW_GRAD_X) ? 0 : (sw == SW_DIV_Y || sw == SW_GRAD_Y) ? 1 : 2;
  const bool pv = sw >= SW_GRAD_Z;
  const DirCoef &D = c.dir[dir];
  BoundPick<T> Y;
  if (!bproj_plan<T>(c, dir, pv, &Y)) return fail(X3D_ERR_UNSUPPORTED, "bounded projection sweep: line not covered");
  if ((size_t)c.p.nx * c.p.ny * c.p.nz * sizeof(T) >= ((size_t)1 << 32))
    return fail(X3D_ERR_UNSUPPORTED, "bounded projection sweep: field larger than 4 GiB");
  const BoundDev<T> tI = bound_dev<T>(c, dir, pv ? OP_INTERPV : OP_INTERVP, 1, Y.longer);
  const BoundDev<T> tD = bound_dev<T>(c, dir, pv ? OP_DERPV : OP_DERVP, pv ? 1 : 0, Y.longer);
  BProjArgs<T> A{};
  for (int i = 0; i < 3; ++i) {
    A.in[i] = io.in[i];
    A.out[i] = io.out[i];
  }
  A.pkI = tI.pk; A.pkD = tD.pk; A.edgeI = tI.edge; A.edgeD = tD.edge;
  A.K = std::max(tI.K, tD.K);
  A.s = cast_sten<T>(D.s);
  A.n_in = proj_in(D, pv);
  A.n_out = proj_out(D, pv);
  A.P = Y.P;
  if (dir == 1 && c.p.istret != 0) {
    if constexpr (sizeof(T) == 8) A.met = pv ? c.ppy64 : c.ppyi64;
    else A.met = pv ? c.ppy32 : c.ppyi32;
  }
  const int nx = c.p.nx, ny = c.p.ny, nz = c.p.nz;
  constexpr int L = BoundShape<T>::L;
  const dim3 block(Y.TL, Y.P);
  if (dir == 0) {
    A.na = ny * nz;
    A.row = D.n | 1;
    if (pv) X3D_TRY(fill_corvel<T>(c, io, &A.cv));
    const dim3 grid((A.na + Y.TL - 1) / Y.TL, 1, 3);
    if (Y.longer) launch_bproj_x<T, L + 1>(A, pv, grid, block, Y.shmem, st);
    else launch_bproj_x<T, L>(A, pv, grid, block, Y.shmem, st);
  } else {
    if (dir == 1) {
      // x is on the pressure grid; z on the velocity grid in both passes
      A.na = c.nxm; A.nb = nz; A.se = c.nxm;
      A.sb_in = (long long)c.nxm * A.n_in;
      A.sb_out = (long long)c.nxm * A.n_out;
    } else {
      A.na = c.nxm * c.nym; A.nb = 1; A.se = A.na;
    }
    const dim3 grid((A.na + Y.TL - 1) / Y.TL, A.nb);
    if (sw == SW_DIV_Z) {
      A.divp = io.divp;
      if (io.divp_blocks) *io.divp_blocks = (int)(grid.x * grid.y);
    }
    if (Y.longer) launch_bproj_yz<T, L + 1>(A, sw, grid, block, Y.shmem, st);
    else launch_bproj_yz<T, L>(A, sw, grid, block, Y.shmem, st);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(X3D_ERR_HIP, std::string("bounded projection launch: ") + hipGetErrorString(e));
  return X3D_OK;
}
template int launch_bounded_projection<double>(const Context &, int, const ProjIO<double> &, hipStream_t);
template int launch_bounded_projection<float>(const Context &, int, const ProjIO<float> &, hipStream_t);

}  // namespace x3d
