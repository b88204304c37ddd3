// spectral.h -- the pieces of the eigenbasis solve that the single domain
// (spectral.hip) and the ensemble (ensemble.hip) share: the real orthogonal
// eigenbasis of one axis of the seven-point operator, its Jacobi eigenvalues,
// and the FP64 matrix-core tile that applies a basis along one axis.
//
// One axis of n cells: between flow guards (fixed values) the eigenvectors are
// the sines Q(x, k) = sqrt(2/(n+1)) sin(pi (x+1)(k+1)/(n+1)); on a periodic axis
// the constant, the cosine and sine pairs and, for even n, the alternating
// vector.  The Jacobi iteration matrix J has eigenvalues lambda = 2 (ax cos tx +
// ay cos ty + az cos tz); with 2 (ax + ay + az) = 1, lambda - 1 = -sum 4 a
// sin^2(t/2) and lambda + 1 = sum 4 a cos^2(t/2), which keep their digits at
// both ends of the spectrum.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace picard {

// Any axis up to this many cells is transformed by a dense product (2 n FP64
// operations per cell and axis).
constexpr int kSpecMaxAxis = 1024;

// Stored basis: rows and columns padded with zeros, rows (the summed index) to
// a multiple of 16, columns (the output index) to a multiple of 64.
__host__ __device__ inline int spec_rows(int n) { return (n + 15) & ~15; }
__host__ __device__ inline int spec_cols(int n) { return (n + 63) & ~63; }
__host__ __device__ inline int64_t spec_mat_len(int n) {
  return (int64_t)spec_rows(n) * spec_cols(n);
}

// Q(x, k), 0 <= x, k < n.
__device__ inline double spec_basis(int n, bool flow, int x, int k) {
  if (flow) {
    const int64_t q = (int64_t)(x + 1) * (k + 1) % (2 * (int64_t)(n + 1));
    return sqrt(2.0 / (double)(n + 1)) * sinpi((double)q / (double)(n + 1));
  }
  if (k == 0) return sqrt(1.0 / (double)n);
  if ((n & 1) == 0 && k == n - 1) return (x & 1) ? -sqrt(1.0 / (double)n) : sqrt(1.0 / (double)n);
  const int m = (k + 1) >> 1;                       // wave number of the pair (2m - 1, 2m)
  const int64_t q = (int64_t)m * x % n;
  const double a = 2.0 * (double)q / (double)n;
  return sqrt(2.0 / (double)n) * ((k & 1) ? cospi(a) : sinpi(a));
}

// t/2 of eigenvector k in units of pi: lambda's cos t, t = 2 pi h.
__device__ inline double spec_half_angle(int n, bool flow, int k) {
  if (flow) return 0.5 * (double)(k + 1) / (double)(n + 1);
  if ((n & 1) == 0 && k == n - 1) return 0.5;
  return (double)((k + 1) >> 1) / (double)n;
}

// ln|lambda| and the sign of lambda from s = 1 - lambda and c = 1 + lambda.
__device__ __forceinline__ double spec_ln(double s, double c, bool *neg) {
  *neg = s > c;
  return log1p(-fmin(*neg ? c : s, 1.0));
}

// Host: spectral.hip.
int spec_axis_tables(hipStream_t s, int n, bool flow, double a, double *fwd, double *inv, double *eig);
struct SpecTile;
int spec_product(hipStream_t s, const SpecTile &t, bool xaxis);
double spec_slowest(const int n[3], const int flow[3], const double a[3]);

typedef double d4v __attribute__((ext_vector_type(4)));

// One output tile of a basis applied along one axis.  The tile holds 32 AT
// axis outputs by 64 columns of the other two axes; four waves of 16 AT x 32.
// FP64 matrix instructions (16x16x4: lane l gives A(l % 16, l / 16) and
// B(l / 16, l % 16) and holds rows l / 16 + 4 v, column l % 16 of the result).
// Bound: the FP64 matrix rate (2 n operations per element against 16 bytes);
// a step of 16 summed indices costs a wave 4 * 2 AT instructions of 64 cycles
// and 2 + AT eight-byte LDS reads per four of them, so LDS and the loads, one step
// ahead in registers, stay behind the matrix cores.
//
// XAXIS: columns are rows of x (data element (col, k) at col * ld + k);
// otherwise a column group of 16 consecutive doubles sits at (g / gpr) gs +
// (g % gpr) 16, and element k of a column at + k ld.  `total` columns in all.  The
// outputs lie by ldo and gso, where a product changes the axis' length.
struct SpecTile {
  const double *M;       // basis, [summed index][output index], pitch np
  const double *in;
  double *out;
  int n, np;             // axis cells, basis pitch
  int nout;              // outputs stored per column (x: the padded row, so that padding stays 0)
  int64_t ld, gs, ldo, gso;
  int64_t total;
  uint32_t gpr;
};

constexpr int kSpecT = 256;
constexpr int kSpecK = 16;                          // summed indices per step
constexpr int kSpecCols = 64;
constexpr int kSpecQs = 80;                         // LDS pitch of a 64-wide row: 128 B past a
                                                    // multiple of 256 B, so the four rows a
                                                    // fragment reads do not meet in a bank
constexpr int kSpecXs = 18;                         // LDS pitch of an x row of 16
constexpr int kSpecLds = 2 * kSpecK * kSpecQs;      // doubles of one buffer (basis + data)

template <int AT, bool XAXIS>
__device__ __forceinline__ void spec_tile(const SpecTile &t, int axis0, int64_t col0, double *lds) {
  static_assert(kSpecCols * kSpecXs <= kSpecK * kSpecQs, "x rows fit the data half");
  const int tid = (int)threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wa = (wave & 1) * 16 * AT, wc = (wave >> 1) * 32;
  const int li = lane & 15, lk = lane >> 4;
  constexpr int QW = 32 * AT;                       // axis outputs of the tile
  constexpr int QN = kSpecK * QW / 2 / kSpecT;      // 16-byte basis loads per thread
  d4v acc[AT][2];
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c) acc[a][c] = d4v{0.0, 0.0, 0.0, 0.0};

  // data: two 16-byte loads per thread and step
  const double *dp[2];
  bool dok[2];
  int dk[2], dl[2];                                 // first summed index, LDS offset
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int e = tid + q * kSpecT;
    if (XAXIS) {
      const int r = e >> 3, kp = (e & 7) * 2;
      dok[q] = col0 + r < t.total;
      dk[q] = kp;
      dl[q] = r * kSpecXs + kp;
      dp[q] = t.in + (dok[q] ? (col0 + r) * t.ld : 0) + kp;
    } else {
      const int k = e >> 5, c = (e & 31) * 2;
      const uint32_t g = (uint32_t)((col0 + c) >> 4);   // fewer than 2^32 groups of 16
      dok[q] = col0 + c < t.total;
      dk[q] = k;
      dl[q] = k * kSpecQs + c;
      dp[q] = t.in + (dok[q] ? (int64_t)(g / t.gpr) * t.gs + (int64_t)(g % t.gpr) * 16 + (c & 15) : 0) + (int64_t)k * t.ld;
    }
  }
  double2 rq[QN], rd[2];
  auto load = [&](int k0) {
#pragma unroll
    for (int q = 0; q < QN; ++q) {
      const int e = tid + q * kSpecT, k = e / (QW / 2), c = (e % (QW / 2)) * 2;
      rq[q] = *reinterpret_cast<const double2 *>(t.M + (int64_t)(k0 + k) * t.np + axis0 + c);
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      rd[q] = make_double2(0.0, 0.0);
      // an x row is padded with zeros to a multiple of 16; other axes end at n
      if (dok[q] && (XAXIS || k0 + dk[q] < t.n))
        rd[q] = *reinterpret_cast<const double2 *>(dp[q] + (XAXIS ? (int64_t)k0 : (int64_t)k0 * t.ld));
    }
  };
  auto put = [&](int b) {
    double *Q = lds + b * kSpecLds, *D = Q + kSpecK * kSpecQs;
#pragma unroll
    for (int q = 0; q < QN; ++q) {
      const int e = tid + q * kSpecT, k = e / (QW / 2), c = (e % (QW / 2)) * 2;
      *reinterpret_cast<double2 *>(Q + k * kSpecQs + c) = rq[q];
    }
#pragma unroll
    for (int q = 0; q < 2; ++q) *reinterpret_cast<double2 *>(D + dl[q]) = rd[q];
  };
  load(0);
  put(0);
  __syncthreads();
  int b = 0;
  for (int k0 = 0; k0 < t.n; k0 += kSpecK, b ^= 1) {
    const bool more = k0 + kSpecK < t.n;            // block-uniform
    if (more) load(k0 + kSpecK);
    const double *Q = lds + b * kSpecLds, *D = Q + kSpecK * kSpecQs;
#pragma unroll
    for (int ks = 0; ks < kSpecK; ks += 4) {
      double fq[AT], fd[2];
#pragma unroll
      for (int a = 0; a < AT; ++a) fq[a] = Q[(ks + lk) * kSpecQs + wa + 16 * a + li];
#pragma unroll
      for (int c = 0; c < 2; ++c)
        fd[c] = XAXIS ? D[(wc + 16 * c + li) * kSpecXs + ks + lk] : D[(ks + lk) * kSpecQs + wc + 16 * c + li];
#pragma unroll
      for (int a = 0; a < AT; ++a)
#pragma unroll
        for (int c = 0; c < 2; ++c)
          acc[a][c] = XAXIS ? __builtin_amdgcn_mfma_f64_16x16x4f64(fd[c], fq[a], acc[a][c], 0, 0, 0)
                            : __builtin_amdgcn_mfma_f64_16x16x4f64(fq[a], fd[c], acc[a][c], 0, 0, 0);
    }
    if (more) put(b ^ 1);                           // last read two steps ago, a barrier between
    __syncthreads();
  }
#pragma unroll
  for (int a = 0; a < AT; ++a)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int row = lk + 4 * v;
        const int ax = axis0 + wa + 16 * a + (XAXIS ? li : row);
        const int64_t col = col0 + wc + 16 * c + (XAXIS ? row : li);
        if (ax >= t.nout || col >= t.total) continue;
        if (XAXIS) {
          t.out[col * t.ldo + ax] = acc[a][c][v];
        } else {
          const uint32_t g = (uint32_t)(col >> 4);
          t.out[(int64_t)(g / t.gpr) * t.gso + (int64_t)(g % t.gpr) * 16 + (col & 15) + (int64_t)ax * t.ldo] =
              acc[a][c][v];
        }
      }
}

}  // namespace picard
