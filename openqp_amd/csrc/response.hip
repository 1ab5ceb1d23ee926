// response.hip -- dense contraction of the MRSF response pass.
//
// The quartet kernels store the pass's integrals, T[tri(x, y)][z][w] = (xy|zw)
// (JKParams::T); with nd non-symmetric densities M_q the pass is then two matrix
// products over T,
//   K_q[x][z] = sum_{y, w} T[tri(x, y)][z][w] M_q[y][w]   (all q),
//   J_q[x][y] = sum_{z, w} T[tri(x, y)][z][w] M_q[z][w]   (the Coulomb q),
// on the FP64 matrix units.  What bounds it: nd is 7 per trial vector, so an
// element of T read (twice for K, once for J) meets nd columns and the reads of T
// bound the kernel, not the matrix units.  Adding every quartet into nd matrices
// instead costs 12 nd atomics and as many gathers per s quartet.  (H2O)8/6-31G, 28
// densities: 50.9 ms per pass then, now 0.31 + 0.12 ms for the two products (T, 0.51 GB,
// read twice for K and once for J: 3.3 and 4.4 TB/s) and 1.75 ms in all; other sizes at
// response_elems() in session.hip.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "response.h"

namespace oqph {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

// raw[y][w][c][v] (v fastest) -> M[q = v nmat + c][y][w], rows of ld doubles, the tail cleared
__global__ void k_rsp_pack(const double* __restrict__ raw, int n, int ld, int nmat, int nf, double* __restrict__ M) {
  const int nd = nmat * nf;
  const long long m = (long long)n * ld * nd, step = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += step) {
    const int k = (int)(i % nd);  // c nf + v
    const long long yw = i / nd;
    const int w = (int)(yw % ld), y = (int)(yw / ld);
    const int q = (k % nf) * nmat + k / nf;
    M[((size_t)q * n + y) * ld + w] = w < n ? raw[((size_t)y * n + w) * nd + k] : 0.0;
  }
}

// F[q][y][w] -> raw[y][w][c][v]
__global__ void k_rsp_unpack(const double* __restrict__ F, int n, int nmat, int nf, double* __restrict__ raw) {
  const int nd = nmat * nf;
  const long long m = (long long)n * n * nd, step = (long long)gridDim.x * blockDim.x;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += step) {
    const int k = (int)(i % nd), q = (k % nf) * nmat + k / nf;
    raw[i] = F[(size_t)q * n * n + i / nd];
  }
}

// A block takes 16 CT rows and 16 NV densities; its eight wavefronts take every
// eighth y (K) or z (J) of the block's share and meet in LDS.  K: the rows are
// z0 .. of one x; J: pairs (x, y).  A lane reads 4 consecutive w of its row and of
// its density (a row's four lane groups: 128 bytes); which w of a 16-wide step is
// the k-th of a matrix instruction does not matter as long as both sides agree.
template <int CT, int NV, bool COUL>
__global__ __launch_bounds__(512) void k_response(ResponseParams r) {
  __shared__ double s_out[16 * NV][16 * CT + 1];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, row = lane & 15, g = lane >> 4;
  const int n = r.n, ld = r.ld;
  const long long nld = (long long)n * ld;
  for (int i = threadIdx.x; i < 16 * NV * (16 * CT + 1); i += 512) (&s_out[0][0])[i] = 0.0;
  const int nt = (n + 16 * CT - 1) / (16 * CT);
  const int x = COUL ? 0 : (int)blockIdx.x / nt;
  const long long row0 = COUL ? (long long)blockIdx.x * 16 * CT : ((int)blockIdx.x - x * nt) * 16 * CT;
  const long long nrow = COUL ? r.npair : n;
  const double* A[CT];  // rows past the end read the last row and are dropped
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    const long long i = row0 + 16 * t + row < nrow ? row0 + 16 * t + row : nrow - 1;
    A[t] = r.T + i * (COUL ? nld : ld) + 4 * g;
  }
  const int j0 = (int)blockIdx.y * 16 * NV;
  const double* B[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int c = j0 + 16 * j + row < r.ncol ? j0 + 16 * j + row : r.ncol - 1;
    B[j] = r.M + (size_t)r.col[c] * nld + 4 * g;
  }
  v4d acc[CT][NV];
#pragma unroll
  for (int t = 0; t < CT; ++t)
#pragma unroll
    for (int j = 0; j < NV; ++j) acc[t][j] = v4d{0.0, 0.0, 0.0, 0.0};
  for (int o = (int)blockIdx.z * 8 + wave; o < n; o += 8 * (int)gridDim.z) {
    const long long p = x >= o ? (long long)x * (x + 1) / 2 + o : (long long)o * (o + 1) / 2 + x;
    const long long ao = COUL ? (long long)o * ld : p * nld, bo = (long long)o * ld;
#pragma unroll 2
    for (int d = 0; d < ld; d += 16) {
      v2d a[CT][2], b[NV][2];
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        a[t][0] = *(const v2d*)(A[t] + ao + d);
        a[t][1] = *(const v2d*)(A[t] + ao + d + 2);
      }
#pragma unroll
      for (int j = 0; j < NV; ++j) {
        b[j][0] = *(const v2d*)(B[j] + bo + d);
        b[j][1] = *(const v2d*)(B[j] + bo + d + 2);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
          for (int j = 0; j < NV; ++j)
            acc[t][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][k / 2][k % 2], b[j][k / 2][k % 2], acc[t][j], 0, 0, 0);
    }
  }
  __syncthreads();
  // element i of a lane's result: row 4 i + lane / 16, column lane % 16
#pragma unroll
  for (int t = 0; t < CT; ++t)
#pragma unroll
    for (int j = 0; j < NV; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) unsafeAtomicAdd(&s_out[16 * j + row][16 * t + 4 * i + g], acc[t][j][i]);
  __syncthreads();
  for (int i = threadIdx.x; i < 256 * CT * NV; i += 512) {
    const int c = i / (16 * CT), z = i - c * (16 * CT);
    if (j0 + c >= r.ncol || row0 + z >= nrow) continue;
    const double v = r.scale * s_out[c][z];
    if (v == 0.0) continue;
    double* F = r.F + (size_t)r.col[j0 + c] * n * n;
    if constexpr (COUL) {
      const long long p = row0 + z;
      int px = (int)((sqrt(8.0 * (double)p + 1.0) - 1.0) * 0.5);
      while ((long long)px * (px + 1) / 2 > p) --px;
      while ((long long)(px + 1) * (px + 2) / 2 <= p) ++px;
      const int py = (int)(p - (long long)px * (px + 1) / 2);
      unsafeAtomicAdd(F + (size_t)px * n + py, v);
      if (px != py) unsafeAtomicAdd(F + (size_t)py * n + px, v);
    } else {
      unsafeAtomicAdd(F + (size_t)x * n + row0 + z, v);
    }
  }
}

// blocks of 256 for m elements, at most 64 per CU: one thread per element would end at 2^32
static unsigned rsp_blocks(long long m) { return (unsigned)std::min<long long>((m + 255) / 256, 16384); }

void launch_rsp_pack(const double* raw, int n, int ld, int nmat, int nf, double* M, hipStream_t s) {
  const long long m = (long long)n * ld * nmat * nf;
  hipLaunchKernelGGL(k_rsp_pack, dim3(rsp_blocks(m)), dim3(256), 0, s, raw, n, ld, nmat, nf, M);
}

void launch_rsp_unpack(const double* F, int n, int nmat, int nf, double* raw, hipStream_t s) {
  const long long m = (long long)n * n * nmat * nf;
  hipLaunchKernelGGL(k_rsp_unpack, dim3(rsp_blocks(m)), dim3(256), 0, s, F, n, nmat, nf, raw);
}

template <int NV, bool COUL>
static void response_t(const ResponseParams& r, hipStream_t s) {
  constexpr int CT = 2, R = 16 * CT;
  const long long rows = COUL ? (r.npair + R - 1) / R : (long long)r.n * ((r.n + R - 1) / R);
  const int groups = (r.ncol + 16 * NV - 1) / (16 * NV);
  // four blocks per CU, but a wavefront keeps at least one o of its own
  const long long want = (4ll * r.ncu + rows * groups - 1) / (rows * groups);
  const int split = (int)std::max<long long>(1, std::min<long long>(want, (r.n + 7) / 8));
  hipLaunchKernelGGL((k_response<CT, NV, COUL>), dim3((unsigned)rows, (unsigned)groups, (unsigned)split), dim3(512), 0,
                     s, r);
}

// 16, 32 or 64 densities per read of T
template <bool COUL>
static void response_n(const ResponseParams& r, hipStream_t s) {
  if (r.ncol <= 0) return;
  if (r.ncol <= 16) response_t<1, COUL>(r, s);
  else if (r.ncol <= 32) response_t<2, COUL>(r, s);
  else response_t<4, COUL>(r, s);
}

void launch_response(bool coulomb, const ResponseParams& r, hipStream_t s) {
  if (coulomb) response_n<true>(r, s);
  else response_n<false>(r, s);
}

}  // namespace oqph
