// bcpot_modes.hip -- BCpotentials (BCpotentials.f90:51-141) for the FP32-split and
// the order-free FP64 form: the open-boundary face sums in FP64, mode by mode.
//
// For a flow dimension d and a plane of cells, the offset across the plane is (t1 -
// tt1, t2 - tt2): a 2D convolution with the distance table's plane at that normal
// offset, which is even in every offset (CalcDistance.f90:25-91).  Over 2 N cells of a
// transverse axis, the charge in the first N, it is a circular convolution with an
// even real kernel, so the real Fourier basis diagonalises it, a cosine and its sine
// with one eigenvalue:
//     U_f = Q1 Q2 ( sum_n lambda_n . Q1^T Q2^T C_n ),
// lambda_n = the cosine sums of plane n, formed once.  Both faces read the same
// lambda, n cells from the one and nd + 1 - n from the other.
//
// The basis goes along an axis as a dense product on the FP64 matrix cores (spectral.h),
// 12 n^4 operations a flow dimension.  Bound: those, about 50 TF/s, and writing 4 n^3
// modes.  FFTs in LDS of the zero-padded complex planes moved 16 n^3 doubles
// a pass, columns at a stride of a row.  Against those: a step of 160^3, x open, 36.7 ->
// 34.6 ms; a solve of 128^3, all open, 3.70 -> 2.72; a step of 53 x 38 x 45, all open, 1.41 ->
// 1.27; 16^3 the same, 0.57.
#include <algorithm>

#include "picard_internal.h"
#include "spectral.h"

namespace picard {
namespace {

constexpr int kT = 256;

// One flow dimension: normal d, transverse t1 < t2; the modes [k2][k1] of the charge lie at
// k1 m1 + k2 m2 + n md, the table's eigenvalues at w1 l1 + w2 l2 + (n - 1) ld, w = (k + 1) / 2.
struct ModeGeo {
  int nd, n1, n2;
  int64_t m1, m2, md;
  int64_t l1, l2, ld;
  int64_t s1, s2, sd;        // node strides
  int64_t D0, d1, d2, dd;    // distance table: the centre and the strides
};

ModeGeo mode_geo(const GridDims &g, int d) {
  const int n[3] = {g.nx, g.ny, g.nz};
  const int64_t node[3] = {1, g.X, (int64_t)g.X * g.Y};
  const int64_t DX = 2 * (int64_t)g.nx + 1, DY = 2 * (int64_t)g.ny + 1;
  const int64_t dist[3] = {1, DX, DX * DY};
  const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
  const int64_t px = (g.nx + 15) & ~15, lx = (2 * g.nx + 15) & ~15;
  ModeGeo m;
  m.nd = n[d];
  m.n1 = n[t1];
  m.n2 = n[t2];
  if (d == 0) m.md = 1, m.m1 = px, m.m2 = px * 2 * g.ny;            // [kz][ky][x]
  if (d == 1) m.m1 = 1, m.md = lx, m.m2 = lx * g.ny;                // [kz][y][kx]
  if (d == 2) m.m1 = 1, m.m2 = lx, m.md = lx * 2 * g.ny;            // [z][ky][kx]
  // along the lanes of k_modes: the normal for x faces, else k1
  if (d == 0) m.ld = 1, m.l1 = m.nd, m.l2 = (int64_t)m.nd * (m.n1 + 1);
  else m.l1 = 1, m.ld = m.n1 + 1, m.l2 = (int64_t)m.nd * (m.n1 + 1);
  m.s1 = node[t1];
  m.s2 = node[t2];
  m.sd = node[d];
  m.D0 = n[0] * dist[0] + n[1] * dist[1] + n[2] * dist[2];
  m.d1 = dist[t1];
  m.d2 = dist[t2];
  m.dd = dist[d];
  return m;
}

// *odd set where a table entry differs from its mirror image at positive offsets.
__global__ void __launch_bounds__(kT) k_modes_even(GridDims g, const double *__restrict__ D,
                                                    int32_t *__restrict__ odd) {
  const int64_t DX = 2 * (int64_t)g.nx + 1, DY = 2 * (int64_t)g.ny + 1, DZ = 2 * (int64_t)g.nz + 1;
  bool bad = false;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < DX * DY * DZ;
       t += (int64_t)gridDim.x * kT) {
    const int i = abs((int)(t % DX) - g.nx), j = abs((int)(t / DX % DY) - g.ny),
              k = abs((int)(t / (DX * DY)) - g.nz);
    bad |= !(D[t] == D[g.nx + i + DX * (g.ny + j + DY * (g.nz + k))]);
  }
  if (bad) *odd = 1;
}

// One transverse axis of the table's cosine sums, n offsets to n + 1 wave numbers: FIRST from the
// table along t1 to A [a][o2][w1], then along t2 to the eigenvalues.
template <bool FIRST>
__global__ void __launch_bounds__(kT) k_modes_eig(ModeGeo m, const double *__restrict__ M,
                                                   const double *__restrict__ D,
                                                   double *__restrict__ A,
                                                   double *__restrict__ lam) {
  const int W1 = m.n1 + 1;
  const int n = FIRST ? m.n1 : m.n2;
  const int64_t total = (int64_t)m.nd * W1 * (FIRST ? m.n2 : m.n2 + 1);
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < total; t += (int64_t)gridDim.x * kT) {
    const int w1 = (int)(t % W1);
    const int64_t r = t / W1;
    const int x2 = (int)(r % (FIRST ? m.n2 : m.n2 + 1)), a = (int)(r / (FIRST ? m.n2 : m.n2 + 1));
    const int w = FIRST ? w1 : x2;
    const double *in = FIRST ? D + m.D0 + (a + 1) * m.dd + x2 * m.d2 : A + (int64_t)a * m.n2 * W1 + w1;
    const int64_t st = FIRST ? m.d1 : W1;
    // the basis' cosine of w, over its value at 0
    const int np = spec_cols(2 * n);
    const double *q = M + (w ? 2 * w - 1 : 0);
    double v = 0.0;
    for (int o = 1; o < n; ++o) v += q[(int64_t)o * np] * in[o * st];
    v = in[0] + 2.0 * (v / q[0]);
    if (FIRST) A[t] = v;
    else lam[w1 * m.l1 + x2 * m.l2 + a * m.ld] = v;
  }
}

// Interior charge into rows of px, padded with zeros.
__global__ void __launch_bounds__(kT) k_modes_pack(GridDims g, int px, const double *__restrict__ C,
                                                    double *__restrict__ out) {
  const int64_t len = (int64_t)px * g.ny * g.nz;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < len; t += (int64_t)gridDim.x * kT) {
    const uint32_t row = (uint32_t)(t / px), x = (uint32_t)(t % px);
    const uint32_t y = row % (uint32_t)g.ny, z = row / (uint32_t)g.ny;
    out[t] = x < (uint32_t)g.nx
                 ? C[(x + 1) + (int64_t)g.X * (y + 1) + (int64_t)g.X * g.Y * (z + 1)]
                 : 0.0;
  }
}

// Both faces' modes [face][k2][k1].  XF (x faces, the sum over contiguous x): 16 lanes
// share a mode; otherwise a thread has one, its neighbours the next k1.
template <bool XF>
__global__ void __launch_bounds__(kT) k_modes(ModeGeo m, const double *__restrict__ ch,
                                               const double *__restrict__ lam,
                                               double *__restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x;
  const int64_t mode = XF ? t >> 4 : t;
  const int64_t L1 = 2 * m.n1, modes = L1 * 2 * m.n2;
  if (mode >= modes) return;             // whole groups of 16
  const int k1 = (int)(mode % L1), k2 = (int)(mode / L1);
  const double *c = ch + k1 * m.m1 + k2 * m.m2;
  const double *l = lam + ((k1 + 1) >> 1) * m.l1 + ((k2 + 1) >> 1) * m.l2;
  double f0 = 0.0, f1 = 0.0;
  if (XF) {
    for (int n = (int)(t & 15); n < m.nd; n += 16) {
      const double v = c[n];
      f0 += v * l[n];
      f1 += v * l[m.nd - 1 - n];
    }
    for (int o = 8; o; o >>= 1) {
      f0 += __shfl_xor(f0, o, 16);
      f1 += __shfl_xor(f1, o, 16);
    }
    if (t & 15) return;
  } else {
#pragma unroll 4
    for (int n = 0; n < m.nd; ++n) {
      const double v = c[n * m.md];
      f0 += v * l[n * m.ld];
      f1 += v * l[(m.nd - 1 - n) * m.ld];
    }
  }
  out[mode] = f0;
  out[modes + mode] = f1;
}

// The faces back along t1, [face][k2][j1], and along t2 into the guard planes.
template <bool FIRST>
__global__ void __launch_bounds__(kT) k_modes_back(ModeGeo m, const double *__restrict__ M,
                                                    const double *__restrict__ in,
                                                    double *__restrict__ out, double scale) {
  const int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x;
  const int n2 = FIRST ? 2 * m.n2 : m.n2;
  if (t >= (int64_t)m.n1 * n2 * 2) return;
  const int j1 = (int)(t % m.n1), x2 = (int)(t / m.n1 % n2), f = (int)(t / ((int64_t)m.n1 * n2));
  const int L = 2 * (FIRST ? m.n1 : m.n2), np = spec_cols(L);
  const double *src = FIRST ? in + ((int64_t)f * 2 * m.n2 + x2) * 2 * m.n1
                            : in + (int64_t)f * 2 * m.n2 * m.n1 + j1;
  const int64_t st = FIRST ? 1 : m.n1;
  const double *q = M + (FIRST ? j1 : x2);
  double v = 0.0;
#pragma unroll 8
  for (int k = 0; k < L; ++k) v += q[(int64_t)k * np] * src[k * st];
  if (FIRST) out[t] = v;
  else out[(j1 + 1) * m.s1 + (x2 + 1) * m.s2 + (f ? (m.nd + 1) * m.sd : 0)] = v * scale;
}

// Packed charge; one axis transformed, twice as long; both, four times; both faces' modes
// (8 n1 n2) and their first way back (4 n1 n2).
int64_t work_len(const GridDims &g) {
  const int64_t rows = (int64_t)g.ny * g.nz, px = (g.nx + 15) & ~15;
  const int64_t big = std::max<int64_t>(rows, (int64_t)g.nx * std::max(g.ny, g.nz));
  return 7 * px * rows + 12 * big;
}

unsigned blocks_of(int64_t n) {
  const int64_t b = (n + kT - 1) / kT;
  return (unsigned)(b < 1 ? 1 : (b > 16384 ? 16384 : b));
}

}  // namespace

void bcpot_modes_release(picard_ctx *c) {
  for (int d = 0; d < 3; ++d)
    for (double **p : {&c->face_fwd[d], &c->face_inv[d], &c->face_lam[d]})
      if (*p) (void)hipFree(*p), *p = nullptr;
  if (c->face_work) (void)hipFree(c->face_work), c->face_work = nullptr;
}

// Bases and eigenvalues from the current distance table; *even = false if that
// has not the symmetry.  The caller has checked the faces' lengths.
int bcpot_modes_prepare(picard_ctx *c, bool *even) {
  const GridDims &g = c->gd;
  const int n[3] = {g.nx, g.ny, g.nz};
  hipStream_t s = c->stream;
  PICARD_HIP(hipMemsetAsync(c->s.counters, 0, sizeof(int32_t), s));
  k_modes_even<<<2048, kT, 0, s>>>(g, c->D, c->s.counters);
  PICARD_HIP(hipGetLastError());
  PICARD_HIP(hipMemcpyAsync(c->host_counters, c->s.counters, sizeof(int32_t), hipMemcpyDeviceToHost, s));
  PICARD_HIP(hipStreamSynchronize(s));
  *even = c->host_counters[0] == 0;
  if (!*even) return PICARD_OK;
  auto later = [&](double **p, int64_t doubles) {
    return *p ? PICARD_OK : alloc_later(c, reinterpret_cast<void **>(p), (int64_t)sizeof(double) * doubles);
  };
  PICARD_TRY(later(&c->face_work, work_len(g)));
  for (int d = 0; d < 3; ++d) {
    if (!(g.flow[(d + 1) % 3] || g.flow[(d + 2) % 3]) || (c->face_fwd[d] && c->face_inv[d])) continue;
    PICARD_TRY(later(&c->face_fwd[d], spec_mat_len(2 * n[d])));
    PICARD_TRY(later(&c->face_inv[d], spec_mat_len(2 * n[d])));
    PICARD_TRY(spec_axis_tables(s, 2 * n[d], false, 0.0, c->face_fwd[d], c->face_inv[d], nullptr));
  }
  for (int d = 0; d < 3; ++d) {
    if (!g.flow[d]) continue;
    const ModeGeo m = mode_geo(g, d);
    PICARD_TRY(later(&c->face_lam[d], (int64_t)m.nd * (m.n1 + 1) * (m.n2 + 1)));
    // A: nd n2 (n1 + 1) values of the work array's 7 nd n1 n2
    k_modes_eig<true><<<blocks_of((int64_t)m.nd * m.n2 * (m.n1 + 1)), kT, 0, s>>>(
        m, c->face_fwd[d == 0 ? 1 : 0], c->D, c->face_work, nullptr);
    k_modes_eig<false><<<blocks_of((int64_t)m.nd * (m.n2 + 1) * (m.n1 + 1)), kT, 0, s>>>(
        m, c->face_fwd[d == 2 ? 1 : 2], nullptr, c->face_work, c->face_lam[d]);
    PICARD_HIP(hipGetLastError());
  }
  return PICARD_OK;
}

int launch_bcpot_modes(picard_ctx *c, double kfac) {
  const GridDims &g = c->gd;
  if (!g.flow[0] && !g.flow[1] && !g.flow[2]) return PICARD_OK;      // no faces
  hipStream_t s = c->stream;
  const int px = (g.nx + 15) & ~15, lx = (2 * g.nx + 15) & ~15;
  const int64_t rows = (int64_t)g.ny * g.nz;
  double *B0 = c->face_work, *B1 = B0 + px * rows, *B2 = B1 + 2 * px * rows;   // lx <= 2 px
  k_modes_pack<<<blocks_of(px * rows), kT, 0, s>>>(g, px, c->C, B0);
  PICARD_HIP(hipGetLastError());
  bool x_done = false;                   // B1 = the charge's modes along x [z][y][kx]
  for (int d = 0; d < 3; ++d) {
    if (!g.flow[d]) continue;
    const ModeGeo m = mode_geo(g, d);
    const int t1 = d == 0 ? 1 : 0, t2 = d == 2 ? 1 : 2;
    SpecTile t;
    t.M = c->face_fwd[t1];
    t.np = spec_cols(2 * m.n1);
    t.in = B0;
    t.out = B1;
    t.n = m.n1;
    if (d == 0) {                        // y: [z][y][px] to [z][ky][px]
      t.nout = 2 * g.ny;
      t.ld = t.ldo = px;
      t.gs = (int64_t)px * g.ny;
      t.gso = 2 * t.gs;
      t.total = (int64_t)px * g.nz;
      t.gpr = (uint32_t)(px / 16);
      PICARD_TRY(spec_product(s, t, false));
    } else if (!x_done) {                // x: rows of px to rows of lx
      t.nout = lx;
      t.ld = px;
      t.ldo = lx;
      t.gs = t.gso = 0;
      t.total = rows;
      t.gpr = 1;
      PICARD_TRY(spec_product(s, t, true));
      x_done = true;
    }
    t.M = c->face_fwd[t2];
    t.np = spec_cols(2 * m.n2);
    t.in = B1;
    t.out = B2;
    t.n = m.n2;
    t.nout = 2 * m.n2;
    if (d == 2) {                        // y: [z][y][lx] to [z][ky][lx]
      t.ld = t.ldo = lx;
      t.gs = (int64_t)lx * g.ny;
      t.gso = 2 * t.gs;
      t.total = (int64_t)lx * g.nz;
      t.gpr = (uint32_t)(lx / 16);
    } else {                             // z: the whole planes
      t.total = d == 0 ? (int64_t)px * 2 * g.ny : (int64_t)lx * g.ny;
      t.ld = t.ldo = t.total;
      t.gs = t.gso = 0;
      t.gpr = (uint32_t)(t.total / 16);
    }
    PICARD_TRY(spec_product(s, t, false));
    const int64_t modes = (int64_t)4 * m.n1 * m.n2;
    double *F = B2 + 4 * px * rows, *T = F + 2 * modes;
    if (d == 0)
      k_modes<true><<<(unsigned)((modes * 16 + kT - 1) / kT), kT, 0, s>>>(m, B2, c->face_lam[d], F);
    else
      k_modes<false><<<(unsigned)((modes + kT - 1) / kT), kT, 0, s>>>(m, B2, c->face_lam[d], F);
    k_modes_back<true><<<(unsigned)(((int64_t)m.n1 * 2 * m.n2 * 2 + kT - 1) / kT), kT, 0, s>>>(
        m, c->face_inv[t1], F, T, 1.0);
    k_modes_back<false><<<(unsigned)(((int64_t)m.n1 * m.n2 * 2 + kT - 1) / kT), kT, 0, s>>>(
        m, c->face_inv[t2], T, c->U, kfac);
    PICARD_HIP(hipGetLastError());
  }
  return PICARD_OK;
}

}  // namespace picard
