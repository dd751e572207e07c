// Local gauge alignment of neighbouring images (no reference function: the
// reference measures image distances with the gauge-invariant metric s_jb,
// mepgl.cu:31-32, and interpolates the raw fields).
//
// For image n >= 1, xi_n minimises |A_n + D xi - A_{n-1}|^2 over the grid,
// D being the forward difference (zero in the last column for x and the last
// row for y).  The normal equations L xi = dx^2 D^T (A_{n-1} - A_n), with L
// the Neumann graph Laplacian of the grid, are solved exactly in its
// eigenbasis, the orthonormal DCT-II C[i][k] = w_k cos(pi k (i + 1/2) / N)
// with eigenvalues lam_k = 2 - 2 cos(pi k / N):
//   xi = C ((C^T b C) / (lam_l + lam_k)) C^T,  the constant mode set to zero,
// as four dense products per image (k_dct_gemm).  The transform accumulates
// along the string, chi_n = chi_{n-1} + xi_n, and is applied as
// A_n += D chi_n and psi_a,n *= exp(i q_a chi_n) (fields, direction and both
// gradient buffers; the A parts of the direction and gradients do not
// change).  The forward curl of every plaquette is unchanged, and no
// neighbour A distance grows.  Strings with a fixed A (no self field) are
// left as they are.
//
// Work buffers: planes 0 and 1 of the string's double scratch in the fields'
// layout (cubic_rhs): b and the stage products, then xi and chi in plane 0.
#include "gauge_local.hpp"
#include "kernels_common.hpp"

namespace mepgl {

// Right-hand side b = dx^2 D^T (A_{n-1} - A_n) of image n (zero for image 0):
// a site's x-bond to its left and y-bond below enter with +R, its own bonds
// with -R (R = A_{n-1} - A_n, times dx for the dx^2 / dx scaling).  Four rows in
// flight: 64 images of 256^2 in FP64 53 -> 36 us.
template <class T>
__global__ __launch_bounds__(kBlock) void k_glocal_rhs(AuxArgs a) {
  const WorkItem it = load_item(a.items, xcd_item(blockIdx.x, a.nitems));
  const DevString& s = a.strings[it.string];
  if (s.nsf) return;
  const Strip t = strip_of(s, it);
  if (t.i >= s.N) return;
  const int N = s.N, i = t.i;
  const long long IS = s.image_stride, PS = s.plane_stride, P = s.pitch;
  double* W = (double*)s.cubic_rhs + (long long)t.n * IS;
  const T* X1 = (const T*)s.x[a.xin] + (long long)t.n * IS;
  const T* X0 = X1 - IS;
  if (t.n == 0) {
    for (int j = t.j0; j < t.j1; ++j) W[(long long)j * P + i] = 0;
    return;
  }
  // R on a row's y-bond below is the row before's own.
  const int left = i >= 1 ? 1 : 0;
  auto R = [&](int plane, long long off) {
    return (double)X0[plane * PS + off] - (double)X1[plane * PS + off];
  };
  double below = t.j0 >= 1 ? R(PAY, (long long)(t.j0 - 1) * P + i) : 0.0;
  constexpr int B = 4;  // rows in flight
  for (int j0 = t.j0; j0 < t.j1; j0 += B) {
    double rl[B], rx[B], ry[B];
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const long long o = (long long)min(j0 + r, t.j1 - 1) * P + i;
      rl[r] = R(PAX, o - left), rx[r] = R(PAX, o), ry[r] = R(PAY, o);
    }
#pragma unroll
    for (int r = 0; r < B; ++r) {
      const int j = j0 + r;
      if (j >= t.j1) break;
      double v = 0;
      if (left) v += rl[r];
      if (i <= N - 2) v -= rx[r];
      if (j >= 1) v += below;
      if (j <= N - 2) v -= ry[r];
      below = ry[r];
      W[(long long)j * P + i] = s.dx * v;
    }
  }
}

// out(m, n) = sum_k A(m, k) B(k, n) for every image of one string,
// A(m, k) = A[m ar + k ac], B(k, n) = B[k br + n bc].  With lam, the output is
// divided by lam[m] + lam[n] and its (0, 0) element set to zero.
//
// FP64 matrix cores: a wavefront computes 32 x 32 outputs by 16 x 16 x 4
// products, W x W wavefronts share the operands' 16-deep k tiles in LDS, and
// the next tiles are loaded into registers meanwhile.  AK / BK: the operand is
// contiguous along k; its tile is then kept with k innermost, so that both its
// loads and the LDS accesses run along memory.  Workgroups of one image stay
// on one XCD, whose L2 then holds its 8 N^2 bytes.  64 products of 256^2 take 58
// us (27 at the matrix units' 78.6 TFLOP/s), 97 on the vector units with 4 x 4
// outputs per thread; 32 of 160^2 take 19 and 45.
constexpr int kGemmK = 16;
using double4 = double __attribute__((ext_vector_type(4)));

template <int TS, bool KIN>
struct GemmTile {
  static constexpr int pitch = KIN ? kGemmK + 2 : TS + 16;  // in LDS without bank conflicts
  static constexpr int size = KIN ? TS * pitch : kGemmK * pitch;
  static __device__ __forceinline__ int at(int x, int k) {
    return KIN ? x * pitch + k : k * pitch + x;
  }
  // Element e of the tile in memory order.
  static __device__ __forceinline__ int x_of(int e) { return KIN ? e / kGemmK : e % TS; }
  static __device__ __forceinline__ int k_of(int e) { return KIN ? e % kGemmK : e / TS; }
};

template <int W, bool AK, bool BK>
__global__ __launch_bounds__(W * W * kWave) void k_dct_gemm(GemmArgs g) {
  constexpr int TS = 32 * W, T = W * W * kWave, PER = TS * kGemmK / T;
  using TA = GemmTile<TS, AK>;
  using TB = GemmTile<TS, BK>;
  __shared__ double As[TA::size];
  __shared__ double Bs[TB::size];
  const int N = g.n, tiles = (N + TS - 1) / TS;
  const int id = xcd_item(blockIdx.x, gridDim.x);
  const int z = id / (tiles * tiles), tile = id % (tiles * tiles);
  const int m0 = tile / tiles * TS, n0 = tile % tiles * TS;
  const double* A = g.A + z * g.abatch;
  const double* B = g.B + z * g.bbatch;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int wm = wave / W * 32, wn = wave % W * 32, x = lane % 16, kq = lane / 16;
  double ra[PER], rb[PER];
  // Rows and columns past the matrix repeat its last (their outputs are not
  // stored); steps of k past it are zero in both operands.
  auto load = [&](int k0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + i * T;
      const int ka = k0 + TA::k_of(e), kb = k0 + TB::k_of(e);
      const int m = min(m0 + TA::x_of(e), N - 1), n = min(n0 + TB::x_of(e), N - 1);
      const double va = A[m * g.ar + min(ka, N - 1) * g.ac];
      const double vb = B[min(kb, N - 1) * g.br + n * g.bc];
      ra[i] = ka < N ? va : 0.0;
      rb[i] = kb < N ? vb : 0.0;
    }
  };
  double4 acc[2][2] = {};
  load(0);
  for (int k0 = 0; k0 < N; k0 += kGemmK) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = threadIdx.x + i * T;
      As[TA::at(TA::x_of(e), TA::k_of(e))] = ra[i];
      Bs[TB::at(TB::x_of(e), TB::k_of(e))] = rb[i];
    }
    __syncthreads();
    if (k0 + kGemmK < N) load(k0 + kGemmK);
#pragma unroll
    for (int k = 0; k < kGemmK; k += 4) {
      double a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        a[i] = As[TA::at(wm + 16 * i + x, k + kq)];
        b[i] = Bs[TB::at(wn + 16 * i + x, k + kq)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
  double* O = g.O + z * g.obatch;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * r + kq, n = n0 + wn + 16 * j + x;
        if (m >= N || n >= N) continue;
        double v = acc[i][j][r];
        if (g.lam) v = (m == 0 && n == 0) ? 0.0 : v / (g.lam[m] + g.lam[n]);
        O[m * g.orow + n] = v;
      }
}

// chi_n = chi_{n-1} + xi_n in image order, one thread per site of one string;
// eight images are read before the first of them is written (64 of 256^2: 23 ->
// 11 us).
__global__ __launch_bounds__(256) void k_glocal_prefix(double* W, int N, int F, long long pitch,
                                                      long long IS) {
  const long long e = blockIdx.x * (long long)blockDim.x + threadIdx.x;
  if (e >= (long long)N * N) return;
  double* const w = W + (e / N) * pitch + e % N;
  double acc = w[0];  // image 0: zero
  int n = 1;
  constexpr int B = 8;
  for (; n + B <= F; n += B) {
    double v[B];
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = w[(n + k) * IS];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      acc = acc + v[k];
      w[(n + k) * IS] = acc;
    }
  }
  for (; n < F; ++n) {
    acc = acc + w[n * IS];
    w[n * IS] = acc;
  }
}

// A_n += D chi_n; psi_a,n *= exp(i q_a chi_n) in the fields, the direction
// and both gradient buffers, four rows at a time: a group's loads are in
// flight together before its first store.
template <class T>
__global__ __launch_bounds__(kBlock) void k_glocal_apply(AuxArgs a) {
  const WorkItem it = load_item(a.items, xcd_item(blockIdx.x, a.nitems));
  const DevString& s = a.strings[it.string];
  if (s.nsf) return;
  const Strip t = strip_of(s, it);
  if (t.n == 0 || t.i >= s.N) return;
  const int N = s.N, i = t.i;
  const long long IS = s.image_stride, PS = s.plane_stride, P = s.pitch;
  const double* X = (const double*)s.cubic_rhs + (long long)t.n * IS + i;
  const long long first = (long long)t.n * IS + i;
  T* const XA = (T*)s.x[a.xin] + first;
  T* const bufs[4] = {XA, (T*)s.d[a.dcur] + first, (T*)s.g[0] + first, (T*)s.g[1] + first};
  const int right = i <= N - 2 ? 1 : 0;  // the last column has no x-bond
  constexpr int R = 4;
  for (int j0 = t.j0; j0 < t.j1; j0 += R) {
    double chi[R + 1], dx[R];
    T ax[R], ay[R];
#pragma unroll
    for (int r = 0; r <= R; ++r) chi[r] = X[min(j0 + r, N - 1) * P];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const long long o = min(j0 + r, t.j1 - 1) * P;
      dx[r] = X[min(j0 + r, N - 1) * P + right];
      ax[r] = XA[PAX * PS + o];
      ay[r] = XA[PAY * PS + o];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int j = j0 + r;
      if (j >= t.j1) break;
      if (right) XA[PAX * PS + j * P] = (T)((double)ax[r] + (dx[r] - chi[r]) / s.dx);
      if (j <= N - 2) XA[PAY * PS + j * P] = (T)((double)ay[r] + (chi[r + 1] - chi[r]) / s.dx);
    }
    for (int c = 0; c < s.nc; ++c) {
      double cs[R], sn[R];
#pragma unroll
      for (int r = 0; r < R; ++r) sincos(s.q[c] * chi[r], &sn[r], &cs[r]);
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        T* const U = bufs[b] + (PU1 + 2 * c) * PS;
        T* const V = bufs[b] + (PV1 + 2 * c) * PS;
        T u[R], v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const long long o = min(j0 + r, t.j1 - 1) * P;
          u[r] = U[o], v[r] = V[o];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
          if (j0 + r >= t.j1) break;
          const long long o = (j0 + r) * P;
          const double ur = u[r], vr = v[r];
          U[o] = (T)(ur * cs[r] - vr * sn[r]);
          V[o] = (T)(ur * sn[r] + vr * cs[r]);
        }
      }
    }
  }
}

hipError_t launch_glocal(const AuxArgs& a, int which, bool fp32, hipStream_t st) {
  if (a.nitems <= 0) return hipSuccess;
  const dim3 g((unsigned)a.nitems), b(kBlock);
  if (which == 0) {
    if (fp32)
      hipLaunchKernelGGL(k_glocal_rhs<float>, g, b, 0, st, a);
    else
      hipLaunchKernelGGL(k_glocal_rhs<double>, g, b, 0, st, a);
  } else {
    if (fp32)
      hipLaunchKernelGGL(k_glocal_apply<float>, g, b, 0, st, a);
    else
      hipLaunchKernelGGL(k_glocal_apply<double>, g, b, 0, st, a);
  }
  return hipGetLastError();
}

template <int W>
void dct_gemm(const GemmArgs& g, int F, hipStream_t st) {
  const unsigned t = (unsigned)((g.n + 32 * W - 1) / (32 * W));
  const dim3 grid(t * t * (unsigned)F), block(W * W * kWave);
  if (g.ac != 1)
    hipLaunchKernelGGL((k_dct_gemm<W, false, false>), grid, block, 0, st, g);
  else if (g.bc == 1)
    hipLaunchKernelGGL((k_dct_gemm<W, true, false>), grid, block, 0, st, g);
  else
    hipLaunchKernelGGL((k_dct_gemm<W, true, true>), grid, block, 0, st, g);
}

// 64 x 64 tiles of four wavefronts read their operands half as often as 32 x 32
// tiles of one (64 products of 256^2: 58 us against 75), which pad less: they
// are taken where they save more than a fifth of the padded outputs (32 products
// of 160^2: 19 us against 21; 65 of 200^2 the same either way).
hipError_t launch_dct_gemm(const GemmArgs& g, int F, hipStream_t st) {
  const long long p2 = (g.n + 63) / 64 * 64, p1 = (g.n + 31) / 32 * 32;
  if (4 * p2 * p2 <= 5 * p1 * p1)
    dct_gemm<2>(g, F, st);
  else
    dct_gemm<1>(g, F, st);
  return hipGetLastError();
}

hipError_t launch_glocal_prefix(double* W, int N, int F, long long pitch, long long IS,
                                hipStream_t st) {
  const long long sites = (long long)N * N;
  hipLaunchKernelGGL(k_glocal_prefix, dim3((unsigned)((sites + 255) / 256)), dim3(256), 0, st, W,
                     N, F, pitch, IS);
  return hipGetLastError();
}

}  // namespace mepgl
