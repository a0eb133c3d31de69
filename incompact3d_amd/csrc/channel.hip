// Wall-bounded (channel) pieces of the device time step:
//   init_channel        Case-Channel.f90:96-128  (laminar profile + noise)
//   channel_cfr         Case-Channel.f90:220-261 (constant flow rate)
//   momentum_forcing    Case-Channel.f90:396-410 (constant pressure gradient)
//   pre_correc, ncly=2  navier.f90:616-690       (wall velocity)
//   gradp, ncly=2       navier.f90:456-479       (wall pressure gradient / gdt)
// The fields are the reference's (nx,ny,nz) arrays, i fastest; the FP64
// velocity and, in the FP32-bulk step, its FP32 copy are updated together.
#include <cmath>

#include "x3d_internal.h"

namespace x3d {

namespace {

constexpr int CH_THREADS = 256;
constexpr int CH_RED_BLOCKS = 1024;

unsigned ch_blocks(size_t n) {
  size_t b = (n + CH_THREADS * 4 - 1) / (CH_THREADS * 4);
  if (b < 1) b = 1;
  if (b > 65535u * 8u) b = 65535u * 8u;
  return (unsigned)b;
}

// Uniform [0,1) of the counter seed*2^40 + comp*2^36 + idx: the SplitMix64
// output function (Steele, Lea & Flood, 2014) applied to counter * golden
// gamma, top 53 bits.  A counter-based stream gives every point its own
// number independently of the launch shape, on the host and the device.
__device__ __forceinline__ double hash_uniform(unsigned long long seed, int comp, unsigned long long idx) {
  unsigned long long z = ((seed << 40) + ((unsigned long long)comp << 36) + idx) * 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  z = z ^ (z >> 31);
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

// init_channel, iin=1 with idir_stream=1 (Case-Channel.f90:96-128):
// u = init_noise um (2 r - 1) + 1 - y^2, v and w = init_noise um (2 r - 1),
// um = exp(-0.2 y^2), y = yc[j] (the wall-normal coordinate minus yly/2).
__global__ void __launch_bounds__(CH_THREADS)
    channel_init_kernel(double *__restrict__ ux, double *__restrict__ uy, double *__restrict__ uz,
                        const double *__restrict__ yc, int nx, int ny, size_t n, double noise,
                        unsigned long long seed) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) {
    const int j = (int)((q / (size_t)nx) % (size_t)ny);
    const double y = yc[j];
    const double um = exp(-0.2 * y * y);
    const double r0 = hash_uniform(seed, 0, q), r1 = hash_uniform(seed, 1, q), r2 = hash_uniform(seed, 2, q);
    ux[q] = noise * um * (2.0 * r0 - 1.0) + 1.0 - y * y;
    uy[q] = noise * um * (2.0 * r1 - 1.0);
    uz[q] = noise * um * (2.0 * r2 - 1.0);
  }
}

// Sum over the block; every thread gets it.
__device__ __forceinline__ double block_sum(double sm) {
  __shared__ double r[CH_THREADS / 64];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sm += __shfl_xor(sm, off);
  if ((threadIdx.x & 63) == 0) r[threadIdx.x >> 6] = sm;
  __syncthreads();
  double t = r[0];
#pragma unroll
  for (int i = 1; i < CH_THREADS / 64; ++i) t += r[i];
  return t;
}

// Partial sums of u / ppy(j) (channel_cfr's ub before its coefficient), a
// wavefront per x line at a time: one division a line and lane, and no index
// arithmetic a point (256x129x128: 14.4 -> 8.9 us).  ppy == nullptr stands for
// the uniform mesh's ppy = 1.
__global__ void __launch_bounds__(CH_THREADS)
    bulk_partials(const double *__restrict__ u, const double *__restrict__ ppy, int nx, int ny, int nlines,
                  double *__restrict__ partial) {
  constexpr int W = CH_THREADS / 64;
  const int lane = threadIdx.x & 63;
  double sm = 0.0;
  for (int l = blockIdx.x * W + (int)(threadIdx.x >> 6); l < nlines; l += (int)gridDim.x * W) {
    const double *const p = u + (size_t)l * nx;
    double a = 0.0;
#pragma unroll 4
    for (int i = lane; i < nx; i += 64) a += p[i];
    sm += ppy ? a / ppy[l % ny] : a;
  }
  sm = block_sum(sm);
  if (threadIdx.x == 0) partial[blockIdx.x] = sm;
}

// the partial sums of bulk_partials added up, the same way in every block
__device__ __forceinline__ double bulk_total(const double *__restrict__ partial) {
  double sm = 0.0;
#pragma unroll
  for (int i = 0; i < CH_RED_BLOCKS / CH_THREADS; ++i) sm += partial[i * CH_THREADS + threadIdx.x];
  return block_sum(sm);
}

// out = ub = coeff * sum
__global__ void __launch_bounds__(CH_THREADS)
    bulk_finish(const double *__restrict__ partial, double coeff, double *__restrict__ out) {
  const double t = bulk_total(partial);
  if (threadIdx.x == 0) out[0] = t * coeff;
}

// u <- u - can, can = -(constant - ub) (Case-Channel.f90:250-256).  Each block
// adds up the partial sums for itself while its points are on the way, instead
// of a launch of one block in front (4.6 us).
constexpr int SHIFT_PT = 8;   // points a thread
__global__ void __launch_bounds__(CH_THREADS)
    cfr_shift_kernel(double *__restrict__ u, float *__restrict__ u32, const double *__restrict__ partial,
                     double coeff, double constant, size_t n) {
  const size_t q0 = (size_t)blockIdx.x * (CH_THREADS * SHIFT_PT) + threadIdx.x;
  double v[SHIFT_PT];
#pragma unroll
  for (int i = 0; i < SHIFT_PT; ++i) {
    const size_t q = q0 + (size_t)i * CH_THREADS;
    v[i] = u[q < n ? q : n - 1];
  }
  const double can = -(constant - bulk_total(partial) * coeff);
#pragma unroll
  for (int i = 0; i < SHIFT_PT; ++i) {
    const size_t q = q0 + (size_t)i * CH_THREADS;
    if (q >= n) break;
    const double r = v[i] - can;
    u[q] = r;
    if (u32) u32[q] = (float)r;
  }
}

// f += c (momentum_forcing_channel with cpg, Case-Channel.f90:403-410)
template <typename T>
__global__ void __launch_bounds__(CH_THREADS) add_const_kernel(T *__restrict__ f, double c, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) f[q] = (T)((double)f[q] + c);
}

// the spin-up rotation of momentum_forcing_channel (Case-Channel.f90:413-418):
// f += a v, with a = -wrotation for dux (v = uy) and +wrotation for duy (v = ux)
template <typename T>
__global__ void __launch_bounds__(CH_THREADS) axpy_kernel(T *__restrict__ f, const T *__restrict__ v, T a, size_t n) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += stride) f[q] = f[q] + a * v[q];
}

// pre_correc on the y walls (navier.f90:616-690, no MHD, byx = byy = byz = 0):
// ux = 0 + dpdx gdt, uy = 0, uz = 0 + dpdz gdt on plane j of each wall; the
// stored planes are dpdx(i,k), dpdz(i,k) at [k*nx + i].
__global__ void __launch_bounds__(CH_THREADS)
    wall_velocity_kernel(double *__restrict__ ux, double *__restrict__ uy, double *__restrict__ uz,
                         float *__restrict__ vx, float *__restrict__ vy, float *__restrict__ vz,
                         const double *__restrict__ dpdx, const double *__restrict__ dpdz, double gdt, int nx,
                         int ny, int nz, int j) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nx * nz) return;
  const int i = q % nx, k = q / nx;
  const size_t o = (size_t)i + (size_t)nx * ((size_t)j + (size_t)ny * k);
  const double a = 0.0 + dpdx[q] * gdt, b = 0.0, c = 0.0 + dpdz[q] * gdt;
  ux[o] = a;
  uy[o] = b;
  uz[o] = c;
  if (vx) {
    vx[o] = (float)a;
    vy[o] = (float)b;
    vz[o] = (float)c;
  }
}

// gradp on the y walls (navier.f90:456-479): plane j of a gradient component
// over gdt into the stored plane dst[k*nx + i]
template <typename T>
__global__ void __launch_bounds__(CH_THREADS)
    wall_store_kernel(const T *__restrict__ g, double *__restrict__ dst, double gdt, int nx, int ny, int nz, int j) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nx * nz) return;
  const int i = q % nx, k = q / nx;
  dst[q] = (double)g[(size_t)i + (size_t)nx * ((size_t)j + (size_t)ny * k)] / gdt;
}

}  // namespace

int launch_channel_init(double *ux, double *uy, double *uz, const double *yc, int nx, int ny, int nz, double noise,
                        unsigned long long seed, hipStream_t st) {
  const size_t n = (size_t)nx * ny * nz;
  if (n >= ((size_t)1 << 36)) return fail(X3D_ERR_UNSUPPORTED, "channel noise: more than 2^36 points");
  hipLaunchKernelGGL(channel_init_kernel, dim3(ch_blocks(n)), dim3(CH_THREADS), 0, st, ux, uy, uz, yc, nx, ny, n,
                     noise, seed);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}

// out = ub = coeff * sum u / ppy; partial holds CH_RED_BLOCKS doubles
static void launch_partials(const double *u, const double *ppy, int nx, int ny, int nz, double *partial,
                            hipStream_t st) {
  hipLaunchKernelGGL(bulk_partials, dim3(CH_RED_BLOCKS), dim3(CH_THREADS), 0, st, u, ppy, nx, ny, ny * nz, partial);
}

int launch_bulk(const double *u, const double *ppy, int nx, int ny, int nz, double coeff, double *partial,
                double *out, hipStream_t st) {
  launch_partials(u, ppy, nx, ny, nz, partial, st);
  hipLaunchKernelGGL(bulk_finish, dim3(1), dim3(CH_THREADS), 0, st, partial, coeff, out);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}

// u <- u + (constant - ub), and its FP32 rounding (u32, or null)
int launch_cfr(double *u, float *u32, const double *ppy, int nx, int ny, int nz, double coeff, double constant,
               double *partial, hipStream_t st) {
  launch_partials(u, ppy, nx, ny, nz, partial, st);
  const size_t n = (size_t)nx * ny * nz, per = CH_THREADS * SHIFT_PT;
  hipLaunchKernelGGL(cfr_shift_kernel, dim3((unsigned)((n + per - 1) / per)), dim3(CH_THREADS), 0, st, u, u32, partial,
                     coeff, constant, n);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}

template <typename T>
int launch_add_const(T *f, double c, size_t n, hipStream_t st) {
  hipLaunchKernelGGL((add_const_kernel<T>), dim3(ch_blocks(n)), dim3(CH_THREADS), 0, st, f, c, n);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}
template int launch_add_const<double>(double *, double, size_t, hipStream_t);
template int launch_add_const<float>(float *, double, size_t, hipStream_t);

template <typename T>
int launch_axpy(T *f, const T *v, double a, size_t n, hipStream_t st) {
  hipLaunchKernelGGL((axpy_kernel<T>), dim3(ch_blocks(n)), dim3(CH_THREADS), 0, st, f, v, (T)a, n);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}
template int launch_axpy<double>(double *, const double *, double, size_t, hipStream_t);
template int launch_axpy<float>(float *, const float *, double, size_t, hipStream_t);

int launch_wall_velocity(double *const u[3], float *const v[3], const double *dpdx, const double *dpdz, double gdt,
                         int nx, int ny, int nz, int j, hipStream_t st) {
  const int cnt = nx * nz;
  hipLaunchKernelGGL(wall_velocity_kernel, dim3((cnt + CH_THREADS - 1) / CH_THREADS), dim3(CH_THREADS), 0, st, u[0],
                     u[1], u[2], v[0], v[1], v[2], dpdx, dpdz, gdt, nx, ny, nz, j);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}

template <typename T>
int launch_wall_store(const T *g, double *dst, double gdt, int nx, int ny, int nz, int j, hipStream_t st) {
  const int cnt = nx * nz;
  hipLaunchKernelGGL((wall_store_kernel<T>), dim3((cnt + CH_THREADS - 1) / CH_THREADS), dim3(CH_THREADS), 0, st, g,
                     dst, gdt, nx, ny, nz, j);
  X3D_HIP(hipGetLastError());
  return X3D_OK;
}
template int launch_wall_store<double>(const double *, double *, double, int, int, int, int, hipStream_t);
template int launch_wall_store<float>(const float *, double *, double, int, int, int, int, hipStream_t);

}  // namespace x3d
