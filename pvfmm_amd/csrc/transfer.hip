// Device construction of the V-list transfer blocks: the kernel of every child offset on the
// lattice, its DFT, and the blocks of the 26 parent offsets in the forms of the Hadamard kernels.
// Runs once per operator set and device, not per tree: assembled on the host for each tree, these
// blocks were most of a setup (a context call on 100k moved points, Stokes, m = 6, FP32: 151 ms
// with the host assembly in every call, 11.7 ms without).  Bound by the gathers of G, which stay
// in the caches; 5-15 ms at m = 6 to 10.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "common.hpp"
#include "device_fmm.hpp"
#include "kernels.hpp"
#include "transfer.hpp"

namespace pvfmm_amd {

VGrid v_grid(int m) {
  VGrid g;
  g.n = 2 * m - 1;
  g.nh = m;
  g.M = g.n * g.n * g.nh;
  return g;
}

namespace {

#define TR_LAUNCH_CHECK() HIP_CHECK(hipGetLastError())

constexpr int kRz = 49;  // child offsets of one rz plane, transformed together

struct Scratch {
  double* p = nullptr;
  explicit Scratch(size_t n) { HIP_CHECK(hipMalloc(&p, sizeof(double) * n)); }
  ~Scratch() { (void)hipFree(p); }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
};

unsigned grid_of(int64_t n) { return (unsigned)((n + 255) / 256); }

__device__ __forceinline__ bool near_box(int rx, int ry, int rz) {
  return max(abs(rx), max(abs(ry), abs(rz))) < 2;
}

// g[(r * ne + q) * n^3 + (z n + y) n + x] = K_q(w h - r), w the displacement stored at w mod n
// (|w_d| <= m - 1; zero elsewhere), r the kRz offsets of plane rz
template <int KIND>
__global__ __launch_bounds__(256) void k_lattice_kernel(int m, int n, double h, int rz, double* __restrict__ g) {
  constexpr int NE = KIND == 2 ? 9 : 1;
  const int64_t n3 = (int64_t)n * n * n, idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= kRz * n3) return;
  const int r = (int)(idx / n3), p = (int)(idx % n3);
  const int x = p % n, y = (p / n) % n, z = p / (n * n);
  const int wx = x < m ? x : x - n, wy = y < m ? y : y - n, wz = z < m ? z : z - n;
  const int rx = r % 7 - 3, ry = r / 7 - 3;
  double v[NE];
#pragma unroll
  for (int q = 0; q < NE; q++) v[q] = 0.0;
  if (!near_box(rx, ry, rz) && -wx < m && -wy < m && -wz < m) {
    const double d[3] = {wx * h - rx, wy * h - ry, wz * h - rz};
    const double rinv = 1.0 / sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
    constexpr double pi = 3.14159265358979323846;
    if constexpr (KIND == 0) {
      v[0] = rinv / (4 * pi);
    } else {
#pragma unroll
      for (int i = 0; i < 3; i++)
#pragma unroll
        for (int j = 0; j < 3; j++) v[3 * i + j] = rinv * ((i == j) + d[i] * d[j] * rinv * rinv) / (8 * pi);
    }
  }
#pragma unroll
  for (int q = 0; q < NE; q++) g[((int64_t)r * NE + q) * n3 + p] = v[q];
}

// Twiddles exp(-2 pi i k / n) of the block
// points per axis: every m whose spectra fit the card, more than the transforms of an evaluation take
// (k_fft_up holds m^3 values in LDS)
constexpr int kMaxN = 1024;
__device__ __forceinline__ void load_twiddles(double2* tw, int n) {
  for (int k = threadIdx.x; k < n; k += 256) {
    double s, c;
    sincospi(2.0 * k / n, &s, &c);
    tw[k] = double2{c, -s};
  }
  __syncthreads();
}

// One DFT axis of `count` grids: out[o] = sum_x in[...] w^{k x}.  The line of output o = (b, k)
// starts at in + base(o) with stride `stride`.
__global__ __launch_bounds__(256) void k_dft_x(int n, int nh, int64_t rows, const double* __restrict__ in,
                                               double2* __restrict__ out) {
  __shared__ double2 tw[kMaxN];
  load_twiddles(tw, n);
  const int64_t o = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (o >= rows * nh) return;
  const int k = (int)(o % nh);
  const double* line = in + (o / nh) * n;
  double re = 0, im = 0;
  for (int x = 0, e = 0; x < n; x++, e = (e + k >= n) ? e + k - n : e + k) {
    re = fma(line[x], tw[e].x, re);
    im = fma(line[x], tw[e].y, im);
  }
  out[o] = double2{re, im};
}
// along an axis of length n whose elements are `stride` apart (stride = nh for y, nh n for z):
// in and out [b][axis][stride]
__global__ __launch_bounds__(256) void k_dft_c(int n, int64_t stride, int64_t total, double scale, const double2* __restrict__ in,
                                               double2* __restrict__ out) {
  __shared__ double2 tw[kMaxN];
  load_twiddles(tw, n);
  const int64_t o = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (o >= total) return;
  const int64_t c = o % stride, q = o / stride;
  const int k = (int)(q % n);
  const double2* line = in + (q / n) * n * stride + c;
  double re = 0, im = 0;
  for (int x = 0, e = 0; x < n; x++, e = (e + k >= n) ? e + k - n : e + k) {
    const double2 v = line[x * stride], w = tw[e];
    re += v.x * w.x - v.y * w.y;
    im += v.x * w.y + v.y * w.x;
  }
  out[o] = double2{re * scale, im * scale};
}

// Entry (k, n) of the real-form block of parent offset R at frequency f
struct Blocks {
  const double2* G;
  int M, e0, e1;
  __device__ __forceinline__ double entry(int R, int f, int k, int n) const {
    const int s = (k & 15) >> 1, t = (n & 15) >> 1, i = k >> 4, j = n >> 4;
    const int rx = 2 * (R % 3 - 1) + (s & 1) - (t & 1), ry = 2 * ((R / 3) % 3 - 1) + ((s >> 1) & 1) - ((t >> 1) & 1),
              rz = 2 * (R / 9 - 1) + ((s >> 2) & 1) - ((t >> 2) & 1);
    if (near_box(rx, ry, rz)) return 0.0;
    const int ri = (rx + 3) + 7 * (ry + 3) + 49 * (rz + 3);
    const double2 v = G[((int64_t)ri * e0 * e1 + i * e1 + j) * M + f];
    return ((k & 1) == 0) ? ((n & 1) == 0 ? v.x : v.y) : ((n & 1) == 0 ? -v.y : v.x);
  }
};
__device__ __forceinline__ int offset_of(int o) { return o < 13 ? o : o + 1; }  // the 26 offsets, without 13

__global__ __launch_bounds__(256) void k_transfer_real(Blocks B, double* __restrict__ Vp) {
  const int NB = B.e0 * B.e1;
  const int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= (int64_t)27 * B.M * NB * 256) return;
  const int q = (int)(idx & 3), l = (int)(idx >> 2) & 63;
  const int64_t u = idx >> 8;
  const int nb = (int)(u % B.e1), kb = (int)(u / B.e1 % B.e0);
  const int64_t rf = u / NB;
  const int R = (int)(rf / B.M), f = (int)(rf % B.M);
  Vp[idx] = R == 13 ? 0.0 : B.entry(R, f, 16 * kb + 4 * (l >> 4) + q, 16 * nb + (l & 15));
}

// tau_f = 2^(14 - e) with every entry of frequency f's blocks below 2^e
__global__ __launch_bounds__(256) void k_transfer_tau(Blocks B, double* __restrict__ tau, float* __restrict__ tinv) {
  const int f = blockIdx.x * 256 + threadIdx.x;
  if (f >= B.M) return;
  double mx = 0;
  for (int64_t r = 0; r < (int64_t)343 * B.e0 * B.e1; r++) {
    const double2 v = B.G[r * B.M + f];
    mx = fmax(mx, fmax(fabs(v.x), fabs(v.y)));
  }
  int e = 0;
  if (mx > 0) (void)frexp(mx, &e);
  const double t = mx > 0 ? ldexp(1.0, min(100, max(-100, 14 - e))) : 1.0;
  tau[f] = t;
  tinv[f] = (float)(1.0 / t);
}

__device__ __forceinline__ uint16_t half_bits(_Float16 h) { return __builtin_bit_cast(uint16_t, h); }

// scalar kernels: [pair j][part p][f][lane][i], part 1 times kSplitLow
__global__ __launch_bounds__(256) void k_transfer_fp16_scalar(Blocks B, const double* __restrict__ tau, uint16_t* __restrict__ Vh) {
  const int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= (int64_t)13 * B.M * 512) return;
  const int i = (int)(idx & 7), l = (int)(idx >> 3) & 63;
  const int64_t jf = idx >> 9;
  const int j = (int)(jf / B.M), f = (int)(jf % B.M);
  const double x = B.entry(offset_of(2 * j + (l >> 5)), f, 8 * ((l >> 4) & 1) + i, l & 15) * tau[f];
  const _Float16 h0 = (_Float16)x, h1 = (_Float16)((x - (double)h0) * (double)kSplitLow);
  Vh[((((int64_t)j * 2 + 0) * B.M + f) * 64 + l) * 8 + i] = half_bits(h0);
  Vh[((((int64_t)j * 2 + 1) * B.M + f) * 64 + l) * 8 + i] = half_bits(h1);
}

// Stokes: [f][pair j][chunk c][tile nb][part p][lane][i]
__global__ __launch_bounds__(256) void k_transfer_fp16_stokes(Blocks B, const double* __restrict__ tau, uint16_t* __restrict__ Vh) {
  const int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= (int64_t)B.M * 13 * 9 * 512) return;
  const int i = (int)(idx & 7), l = (int)(idx >> 3) & 63;
  const int64_t u = idx >> 9;  // ((f * 13 + j) * 3 + c) * 3 + nb
  const int nb = (int)(u % 3), c = (int)(u / 3 % 3), j = (int)(u / 9 % 13), f = (int)(u / 117);
  const int q = 4 * c + (l >> 4), a = q / 6, b = q % 6;
  const double x = B.entry(offset_of(2 * j + a), f, 8 * b + i, 16 * nb + (l & 15)) * tau[f];
  const _Float16 h0 = (_Float16)x, h1 = (_Float16)(x - (double)h0);
  Vh[((u * 2 + 0) * 64 + l) * 8 + i] = half_bits(h0);
  Vh[((u * 2 + 1) * 64 + l) * 8 + i] = half_bits(h1);
}

template <typename Real>
__global__ __launch_bounds__(256) void k_convert(const double* __restrict__ in, int rows_in, int cols_in, Real* __restrict__ out,
                                                 int rows, int ld_out, bool transposed) {
  const int64_t idx = blockIdx.x * (int64_t)256 + threadIdx.x;
  if (idx >= (int64_t)rows * ld_out) return;
  int i = (int)(idx / ld_out), j = (int)(idx % ld_out);
  if (transposed) {
    const int t = i;
    i = j;
    j = t;
  }
  out[idx] = (i < rows_in && j < cols_in) ? (Real)in[(int64_t)i * cols_in + j] : Real(0);
}

template <typename Real>
__global__ __launch_bounds__(256) void k_transpose(const Real* __restrict__ in, int rows, int cols, Real* __restrict__ out) {
  __shared__ Real tile[16][17];
  const int r0 = blockIdx.x * 16, c0 = blockIdx.y * 16, x = threadIdx.x & 15, y = threadIdx.x >> 4;
  if (r0 + y < rows && c0 + x < cols) tile[y][x] = in[(int64_t)(r0 + y) * cols + c0 + x];
  __syncthreads();
  if (c0 + y < cols && r0 + x < rows) out[(int64_t)(c0 + y) * rows + r0 + x] = tile[x][y];
}

}  // namespace

void transfer_spectra(hipStream_t s, int kind, int m, double* G) {
  const VGrid g = v_grid(m);
  if (g.n > kMaxN || (kind != 0 && kind != 2)) throw Error(kErrUnsupported, "multipole order too large for the V-list transform");
  const int ne = kind == 2 ? 9 : 1;
  const double h = kRad0 / (m - 1);
  const int64_t grids = (int64_t)kRz * ne, n3 = (int64_t)g.n * g.n * g.n, nx = (int64_t)g.n * g.n * g.nh;
  Scratch lat(grids * n3), a(2 * grids * nx), b(2 * grids * nx);
  for (int rz = -3; rz <= 3; rz++) {
    if (kind == 0)
      hipLaunchKernelGGL(k_lattice_kernel<0>, dim3(grid_of(kRz * n3)), dim3(256), 0, s, m, g.n, h, rz, lat.p);
    else
      hipLaunchKernelGGL(k_lattice_kernel<2>, dim3(grid_of(kRz * n3)), dim3(256), 0, s, m, g.n, h, rz, lat.p);
    TR_LAUNCH_CHECK();
    double2 *pa = reinterpret_cast<double2*>(a.p), *pb = reinterpret_cast<double2*>(b.p);
    hipLaunchKernelGGL(k_dft_x, dim3(grid_of(grids * nx)), dim3(256), 0, s, g.n, g.nh, grids * g.n * g.n, (const double*)lat.p, pa);
    TR_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_dft_c, dim3(grid_of(grids * nx)), dim3(256), 0, s, g.n, (int64_t)g.nh, grids * nx, 1.0,
                       (const double2*)pa, pb);
    TR_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_dft_c, dim3(grid_of(grids * nx)), dim3(256), 0, s, g.n, (int64_t)g.nh * g.n, grids * nx, 1.0 / (double)n3,
                       (const double2*)pb, reinterpret_cast<double2*>(G) + (int64_t)(rz + 3) * grids * nx);
    TR_LAUNCH_CHECK();
  }
  HIP_CHECK(hipStreamSynchronize(s));
}

void transfer_real(hipStream_t s, int e0, int e1, int M, const double* G, double* Vp) {
  const Blocks B{reinterpret_cast<const double2*>(G), M, e0, e1};
  hipLaunchKernelGGL(k_transfer_real, dim3(grid_of((int64_t)27 * M * e0 * e1 * 256)), dim3(256), 0, s, B, Vp);
  TR_LAUNCH_CHECK();
}

void transfer_fp16(hipStream_t s, int e0, int e1, int M, const double* G, uint16_t* Vh, float* tinv) {
  const Blocks B{reinterpret_cast<const double2*>(G), M, e0, e1};
  Scratch tau(M);
  hipLaunchKernelGGL(k_transfer_tau, dim3(grid_of(M)), dim3(256), 0, s, B, tau.p, tinv);
  TR_LAUNCH_CHECK();
  if (e0 == 1 && e1 == 1)
    hipLaunchKernelGGL(k_transfer_fp16_scalar, dim3(grid_of((int64_t)13 * M * 512)), dim3(256), 0, s, B, (const double*)tau.p, Vh);
  else if (e0 == 3 && e1 == 3)
    hipLaunchKernelGGL(k_transfer_fp16_stokes, dim3(grid_of((int64_t)13 * M * 9 * 512)), dim3(256), 0, s, B,
                       (const double*)tau.p, Vh);
  else
    throw Error(kErrInternal, "no fp16 transfer form for this kernel");
  TR_LAUNCH_CHECK();
  HIP_CHECK(hipStreamSynchronize(s));  // tau
}

template <typename Real>
void convert_matrix(hipStream_t s, const double* in, int rows_in, int cols_in, Real* out, int rows, int ld_out, bool transposed) {
  if (rows <= 0 || ld_out <= 0) return;
  hipLaunchKernelGGL(k_convert<Real>, dim3(grid_of((int64_t)rows * ld_out)), dim3(256), 0, s, in, rows_in, cols_in, out, rows,
                     ld_out, transposed);
  TR_LAUNCH_CHECK();
}
template void convert_matrix<float>(hipStream_t, const double*, int, int, float*, int, int, bool);
template void convert_matrix<double>(hipStream_t, const double*, int, int, double*, int, int, bool);

template <typename Real>
void transpose_matrix(hipStream_t s, const Real* in, int rows, int cols, Real* out) {
  if (rows <= 0 || cols <= 0) return;
  hipLaunchKernelGGL(k_transpose<Real>, dim3((rows + 15) / 16, (cols + 15) / 16), dim3(256), 0, s, in, rows, cols, out);
  TR_LAUNCH_CHECK();
}
template void transpose_matrix<float>(hipStream_t, const float*, int, int, float*);
template void transpose_matrix<double>(hipStream_t, const double*, int, int, double*);

}  // namespace pvfmm_amd
