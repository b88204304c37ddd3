// spectral.hip -- the Jacobi solve's long middle in closed form, for the forms
// that are not held to the reference's rounding (FP32-split, and FP64 with the
// order-free deposit).
//
// CalcEpotential.f90:58-92 is a linear iteration: with r_b the residual of
// iterate b, U_p = U_b - af sum_{i < p-b} J^i r_b and r_p = J^{p-b} r_b.  J is
// diagonal in the product of the axes' eigenbases (spectral.h), so one transform of r_b gives
// every later iterate and the norm of its residual.  The solve transforms r_b,
// finds the iterate the stop rule will pick, goes to a few iterates before it
// in one step and leaves the rest, with the stop test itself, to the sweeps
// (grid.hip): the iterate returned and its count are those of sweeping all the way, to FP64
// rounding.
//
// The stop rule's residual takes the previous iterate's values across periodic
// boundaries (CalcEpotential.f90:83-92), which makes it J0 r_{p-1}: one Jacobi
// step of the plain residual with zeros beyond every boundary.  Without a periodic axis its norm is
// the plain one's, which falls from iterate to iterate.  With one it is not a sum over eigenvectors,
// and it may pass the threshold, rise again, and stay below while modes that never decay (the mean of
// a box without an open axis, the checkerboard of even edges) hold the plain norm above.  So the
// step goes no further than the iterates that provably do not pass:
//     |J0 r_{p-1}|^2 >= f(p) - B(p),   f(p) = |r_p|^2,
// B the part across the boundaries, 2 a (u_0 . v_n-1 + u_n-1 . v_0) of the first and last planes of
// u = r_p and v = r_{p-1} for each periodic axis.  For the first iterates B is
// formed as it stands; for the others every mode of a plane's sum enters with its modulus, which
// falls with p, as f does, so that f(q) - B(p) > threshold^2 clears all iterates p to q.  What that
// leaves open before the stop is looked at one by one again (k_spec_clear).
//
// Cost: six axis transforms of 2 n operations a cell, whatever the number of
// sweeps (about 3 n^2 to 1e-6).  Measured, whole solve with its last sweeps
// against sweeping: 16^3 0.19 ms (FP32 sweeps 7.3), 64^3 0.38 ms (FP64 sweeps 280),
// 128^3 all open to 1e-10 0.60 ms (FP32 sweeps 620), 160^3 1.3 ms (FP32 sweeps 880), 256^3 4.3 ms (3900).
// Against the FP64 form that sweeps all the way U differs by 2e-15 to 3e-13
// (the FP32 sweeps differed by 5e-7 to 5e-6) and the sweep counts are equal.
#include <algorithm>
#include <cmath>

#include "picard_internal.h"
#include "reduce.h"
#include "spectral.h"

namespace picard {

constexpr int kSpecCand = 8;        // candidates per pass over the spectrum
constexpr int kSpecPasses = 3;
// iterates that are looked at for the rule's norm: the first kSpecFirst one by one, then kSpecLater
// in growing and again falling distances up to the plain norm's crossing
constexpr int kSpecFirst = 16;
constexpr int kSpecLater = 40;
constexpr int kSpecLook = kSpecFirst + kSpecLater;
constexpr int kSpecEach = 4;        // of them in one block
constexpr int kSpecNear = 32;       // and one by one again after the last of them that is clear

// Device state of one search.  `skip`: no step is taken (0: go on).
struct SpecState {
  double q[kSpecCand];              // candidates, in sweeps after the base iterate
  double lo, hi, flo, fhi;          // bracket of the plain norm's crossing, and the norms^2 there
  double T, f0;                     // threshold^2, the base residual's norm^2
  double look[kSpecLater];          // the later iterates that are looked at, ascending
  double end;                       // the last of them: the crossing, or the last that is tested
  double clear, above, left;        // iterates up to here do not pass, the bound there less B, sweeps left
  double slope;                     // d ln f there
  int32_t near;                     // more iterates are looked at one by one
  double steps;                     // sweeps the step covers
  int64_t to;                       // iterate the step ends on
  int64_t ahead;                    // sweeps from there to about the stop
  int32_t skip;
  uint32_t arrive;
};

namespace {

constexpr int kT = 256;
enum { kSpecGo = 0, kSpecFew = 1, kSpecBad = 2, kSpecUnclear = 3 };
// fewer sweeps than this are not worth the step (about 30 launches)
constexpr int kSpecFewest = 32;

// Compact padded FP64 layout of the transforms: x fastest, rows of PX.
struct SpecGeo {
  int nx, ny, nz, PX;
  int64_t X, XY;                    // node strides of the guard layout
  int px, py, pz;
  int64_t len;                      // PX ny nz
  double ax, ay, az, af, dx2, dy2, dz2;
  const double *eig[3];             // per axis: 4 a sin^2 (n values), then 4 a cos^2
};

// A basis, its transpose and, unless eig is null, the axis' eigenvalue rows.
__global__ void __launch_bounds__(kT) k_spec_basis(int n, int flow, double a, double *fwd, double *inv,
                                                   double *eig) {
  const int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x;
  const int np = spec_cols(n);
  if (t >= spec_mat_len(n)) return;
  const int r = (int)(t / np), c = (int)(t % np);
  const bool in = r < n && c < n;
  fwd[t] = in ? spec_basis(n, flow != 0, r, c) : 0.0;
  inv[t] = in ? spec_basis(n, flow != 0, c, r) : 0.0;
  if (eig && r == 0 && c < n) {
    const double h = spec_half_angle(n, flow != 0, c);
    const double s = sinpi(h), q = cospi(h);
    eig[c] = 4.0 * a * s * s;
    eig[n + c] = 4.0 * a * q * q;
  }
}

// Ends a reduction: true in the block that finishes last, after every
// block's partials are visible.
__device__ __forceinline__ bool last_block(uint32_t *arrive) {
  __shared__ bool last;
  if (threadIdx.x == 0) {
    __threadfence();
    last = atomicAdd(arrive, 1u) == n_blocks() - 1;
  }
  __syncthreads();
  if (last) __threadfence();
  return last;
}

// r = b - A u of the base iterate with periodic images of u itself, into the
// compact layout (padding zero), and its norm; the last block sets up the search.  `old`: the iterate
// before, whose halo the rule's residual of this one takes; its norm is looked at as well.
__global__ void __launch_bounds__(kT) k_spec_residual(SpecGeo g, const double *__restrict__ u,
                                                      const double *__restrict__ old,
                                                      const double *__restrict__ b,
                                                      double *__restrict__ out,
                                                      double *__restrict__ partials,
                                                      const JacobiState *js, SpecState *st,
                                                      int64_t base, double lnmax) {
  __shared__ double sh[kT / 64];
  double acc = 0.0, acc_rule = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < g.len; t += (int64_t)gridDim.x * kT) {
    const uint32_t row = (uint32_t)(t / g.PX), x = (uint32_t)(t % g.PX);
    const uint32_t y = row % (uint32_t)g.ny, z = row / (uint32_t)g.ny;
    double r = 0.0, rule = 0.0;
    if ((int)x < g.nx) {
      const int64_t c = (x + 1) + g.X * (int64_t)(y + 1) + g.XY * (int64_t)(z + 1);
      const int64_t e = g.px && (int)x == g.nx - 1 ? c - (g.nx - 1) : c + 1;
      const int64_t w = g.px && x == 0 ? c + (g.nx - 1) : c - 1;
      const int64_t n = g.py && (int)y == g.ny - 1 ? c - (g.ny - 1) * g.X : c + g.X;
      const int64_t s = g.py && y == 0 ? c + (g.ny - 1) * g.X : c - g.X;
      const int64_t tp = g.pz && (int)z == g.nz - 1 ? c - (g.nz - 1) * g.XY : c + g.XY;
      const int64_t bt = g.pz && z == 0 ? c + (g.nz - 1) * g.XY : c - g.XY;
      const double u2 = 2.0 * u[c];
      r = b[c] - ((u[e] + u[w] - u2) / g.dx2 + (u[n] + u[s] - u2) / g.dy2 +
                  (u[tp] + u[bt] - u2) / g.dz2);
      rule = r;
      if (old) {
        const int64_t XY = g.XY;
        if (e != c + 1) rule += (u[e] - old[c + 1]) / g.dx2;
        if (w != c - 1) rule += (u[w] - old[c - 1]) / g.dx2;
        if (n != c + g.X) rule += (u[n] - old[c + g.X]) / g.dy2;
        if (s != c - g.X) rule += (u[s] - old[c - g.X]) / g.dy2;
        if (tp != c + XY) rule += (u[tp] - old[c + XY]) / g.dz2;
        if (bt != c - XY) rule += (u[bt] - old[c - XY]) / g.dz2;
      }
    }
    out[t] = r;
    acc += r * r;
    acc_rule += rule * rule;
  }
  const double s = block_sum(acc, sh);
  if (threadIdx.x == 0) partials[blockIdx.x] = s;
  if (old) {
    __syncthreads();
    const double s_rule = block_sum(acc_rule, sh);
    if (threadIdx.x == 0) partials[gridDim.x + blockIdx.x] = s_rule;
  }
  if (!last_block(&st->arrive)) return;
  const double f0 = final_sum(partials, gridDim.x, sh);
  double f0_rule = f0;
  if (old) {
    __syncthreads();
    f0_rule = final_sum(partials + gridDim.x, gridDim.x, sh);
  }
  if (threadIdx.x) return;
  st->arrive = 0;
  st->f0 = f0;
  const double T = js->thresh * js->thresh;
  st->T = T;
  st->to = -1;
  const double span = (double)(js->last - base);
  // an infinite or NaN residual is left to the sweeps, as is a solve that has stopped
  st->skip = !(f0 < 1.0e300) || !(T < 1.0e300) ? kSpecBad : (js->slot[base & 1].done || f0 <= T || !(f0_rule > 1.000001 * T) ? kSpecFew : kSpecGo);
  // no mode decays slower than the slowest one
  double hi = span;
  if (T > 0.0 && lnmax < 0.0) hi = fmin(span, ceil(log(T / f0) / (2.0 * lnmax)) + 1.0);
  st->lo = 0.0;
  st->flo = f0;
  st->hi = hi;
  st->fhi = -1.0;
  for (int i = 0; i < kSpecCand; ++i) st->q[i] = fmax(1.0, floor(ldexp(hi, -i)));
}

// The iterate the step ends on: `margin` before the last that is known not to pass, or before the end
// of the solve when that is the last one tested, by more than rounding moves the norm.
__device__ __forceinline__ void spec_finish(const JacobiState *js, SpecState *st, int64_t base, int margin,
                                            double clear, double above, double left) {
  const bool all = clear >= (double)((int64_t)js->maxit - 1 - base) && above > 1.02 * st->T;
  // of `left` sweeps that are expected after the last clear iterate, three are kept for the estimate
  const int64_t on = all ? 1 : (int64_t)fmax(1.0, fmin(left, 1024.0));
  const int64_t in = on > 3 ? (on - 3 < 3 ? on - 3 : 3) : 0;
  const int64_t to = (all ? js->last : base + (int64_t)clear) - margin + in;
  if (to - base < kSpecFewest || to > 0x7fffff00) {
    st->skip = st->end > 4.0 * kSpecFewest ? kSpecUnclear : kSpecFew;
    return;
  }
  st->to = to;
  st->ahead = margin - in + on;
  st->steps = (double)(to - base);
}

// sum w lambda^(2 q) over the spectrum for the pass's candidates, descending
// (pass 0: halvings of the bound) or ascending in q (later passes: a division
// of the bracket); the last block narrows the bracket and, after the last pass,
// interpolates ln(norm^2) in it.  Bound: one read of the spectrum and the
// exponentials (eight per mode that has not decayed away); on small grids the chain of the
// block's and the last block's sums: the candidates' together, 28 -> 10 us at 16^3.
__global__ void __launch_bounds__(kT) k_spec_search(SpecGeo g, const double *__restrict__ R,
                                                    double *__restrict__ partials, const JacobiState *js,
                                                    SpecState *st, int64_t base, int margin, int seams,
                                                    int pass) {
  __shared__ double sh[kT / 64][kSpecCand];
  __shared__ double tot[kSpecCand];
  if (st->skip) return;
  double q2[kSpecCand], qmin = 1.0e300;
#pragma unroll
  for (int i = 0; i < kSpecCand; ++i) {
    q2[i] = 2.0 * st->q[i];
    qmin = fmin(qmin, q2[i]);
  }
  double acc[kSpecCand];
#pragma unroll
  for (int i = 0; i < kSpecCand; ++i) acc[i] = 0.0;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < g.len; t += (int64_t)gridDim.x * kT) {
    const uint32_t row = (uint32_t)(t / g.PX), x = (uint32_t)(t % g.PX);
    if ((int)x >= g.nx) continue;
    const uint32_t y = row % (uint32_t)g.ny, z = row / (uint32_t)g.ny;
    bool neg;
    const double ln = spec_ln(g.eig[0][x] + g.eig[1][y] + g.eig[2][z],
                              g.eig[0][g.nx + x] + g.eig[1][g.ny + y] + g.eig[2][g.nz + z], &neg);
    if (qmin * ln < -700.0) continue;                // below the smallest double at every candidate
    const double w = R[t] * R[t];
#pragma unroll
    for (int i = 0; i < kSpecCand; ++i) acc[i] += w * exp(q2[i] * ln);
  }
  // the candidates' block sums together, then their totals, 32 lanes each
#pragma unroll
  for (int i = 0; i < kSpecCand; ++i) {
    for (int off = 32; off > 0; off >>= 1) acc[i] += __shfl_down(acc[i], off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][i] = acc[i];
  }
  __syncthreads();
  if (threadIdx.x < kSpecCand) {
    double s = 0.0;
    for (int w = 0; w < kT / 64; ++w) s += sh[w][threadIdx.x];
    partials[(int64_t)threadIdx.x * gridDim.x + blockIdx.x] = s;
  }
  __syncthreads();                       // before the fence of thread 0
  if (!last_block(&st->arrive)) return;
  static_assert(kT == 32 * kSpecCand, "32 lanes to a candidate");
  {
    const int i = threadIdx.x >> 5;
    double s = 0.0;
    for (unsigned q = threadIdx.x & 31; q < gridDim.x; q += 32) s += partials[(int64_t)i * gridDim.x + q];
    for (int off = 16; off > 0; off >>= 1) s += __shfl_down(s, off, 32);
    if ((threadIdx.x & 31) == 0) tot[i] = s;
  }
  __syncthreads();
  if (threadIdx.x) return;
  st->arrive = 0;
  double lo = st->lo, hi = st->hi, flo = st->flo, fhi = st->fhi;
  for (int i = 0; i < kSpecCand; ++i) {
    const double q = st->q[i];
    if (tot[i] > st->T) {
      if (q > lo) lo = q, flo = tot[i];
    } else if (q < hi || fhi < 0.0) {
      hi = q, fhi = tot[i];
    }
  }
  st->lo = lo;
  st->hi = hi;
  st->flo = flo;
  st->fhi = fhi;
  if (pass + 1 < kSpecPasses) {
    for (int i = 0; i < kSpecCand; ++i)
      st->q[i] = fmax(1.0, floor(lo + (hi - lo) * (double)(i + 1) / (double)(kSpecCand + 1)));
    return;
  }
  // the crossing; nothing is tested past maxit
  double end = hi;
  if (fhi < 0.0) {
    end = 1.0e300;
  } else if (hi > lo) {
    const double a = log(flo), c = log(fmax(fhi, 1.0e-300));
    if (st->T > 0.0 && c < a) end = fmin(hi, fmax(lo, lo + (log(st->T) - a) * (hi - lo) / (c - a)));
  }
  end = fmax(0.0, fmin(ceil(end), (double)((int64_t)js->maxit - 1 - base)));
  st->end = end;
  if (end < (double)kSpecFewest) {
    st->skip = kSpecFew;
    return;
  }
  // 20 in a geometric progression to half way, 12 evenly on, 8 closing in on the end
  const double half = fmax((double)kSpecFirst, 0.5 * end), step = (end - half) / 13.0;
  const double ratio = exp(log(half / kSpecFirst) / 20.0);
  double q = kSpecFirst, near = step;
  for (int i = 0; i < kSpecLater; ++i) {
    if (i >= 32) q = i == kSpecLater - 1 ? end : end - (near *= 0.5);
    st->look[i] = fmin(end, floor(q));
    q = i < 19 ? q * ratio : half + step * (double)(i - 19);
  }
  // without a periodic axis the plain norm is the rule's
  if (!seams) spec_finish(js, st, base, margin, end <= lo ? end : end - 1.0, end <= lo ? flo : 0.0, 0.0);
}

// Sum of w_i over the block for N values a thread, in thread 0 .. N - 1 of the block.
template <int N>
__device__ __forceinline__ double sum_each(double (&v)[N], double (*sh)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    for (int off = 32; off > 0; off >>= 1) v[i] += __shfl_down(v[i], off, 64);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][i] = v[i];
  }
  __syncthreads();
  double s = 0.0;
  if (threadIdx.x < N)
    for (int w = 0; w < kT / 64; ++w) s += sh[w][threadIdx.x];
  __syncthreads();
  return s;
}

// The periodic axes of a box: cells, stride of the axis and of the columns across it in the
// spectrum, the columns' counts, weight, and the basis.
struct SpecSeam {
  int n, ca, cb;
  int64_t s, sa, sb;
  int axis, ax_a, ax_b;
  double a;
  const double *Q;
};
struct SpecSeams {
  int count;
  SpecSeam s[3];
};

// How far no iterate passes the rule (see above).  blockIdx.y: four iterates, the first ones'
// boundary part signed, the later ones' of moduli; blockIdx.z: a periodic axis, a thread taking columns
// of modes along it.  The plain norms come with the first axis.  A mode that has decayed by e^60 is left
// out, in f to the safe side, in B by less than 1e-24 of the base norm, which the test adds.
// The last block sums and decides.  NEAR, the second launch: the iterates that follow, one by one and signed
// again, unless the first was sharp: 16 to 20 sweeps less for a solve to 1e-2 or 1e-3 (16^3 0.35 -> 0.26 ms,
// 32^3 0.43 -> 0.29), where it is not needed one or two for 12 to 150 us.
// Bound: the exponentials of every mode and iterate, 250 us at 160^3 with
// two periodic axes (393 with the logarithm of the decayed modes too); on small grids the
// chain of one column and the decision, 18 us at 16^3 (eight iterates a block and the decision in one
// thread: 39).
template <bool NEAR>
__global__ void __launch_bounds__(kT) k_spec_clear(SpecGeo g, SpecSeams ss, const double *__restrict__ R,
                                                   double *__restrict__ partials, const JacobiState *js,
                                                   SpecState *st, int64_t base, int margin) {
  constexpr int N = kSpecEach;
  constexpr int kLook = NEAR ? kSpecNear : kSpecLook, kFirst = NEAR ? kSpecNear : kSpecFirst;
  __shared__ double sh[kT / 64][2 * N];
  __shared__ double sums[kLook][4];                  // f, then an axis each
  if (st->skip || (NEAR && !st->near)) return;
  const SpecSeam m = ss.s[blockIdx.z];
  const int first = (int)blockIdx.y * N;             // the block's iterates
  const double past = NEAR ? st->clear + (double)first : 0.0;
  const int nx[3] = {g.nx, g.ny, g.nz};
  double q[N], acc[2 * N];                           // f, then B
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int j = first + i - kFirst;
    q[i] = j >= 0 ? st->look[j] - 1.0 : 0.0;
    acc[i] = acc[N + i] = 0.0;
  }
  const double *es = g.eig[m.axis], *ea = g.eig[m.ax_a], *eb = g.eig[m.ax_b];
  const int np = spec_cols(m.n);
  const int64_t columns = (int64_t)m.ca * m.cb;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < columns; t += (int64_t)gridDim.x * kT) {
    const int ia = (int)(t % m.ca), ib = (int)(t / m.ca);
    const double *r = R + ia * m.sa + ib * m.sb;
    const double sab = ea[ia] + eb[ib], cab = ea[nx[m.ax_a] + ia] + eb[nx[m.ax_b] + ib];
    if (NEAR || first < kFirst) {
      // the two planes' sums of iterates first .. first + N, the rule's being one later
      double v0[N + 1], vn[N + 1];
#pragma unroll
      for (int i = 0; i <= N; ++i) v0[i] = vn[i] = 0.0;
      double next = r[0];
      for (int k = 0; k < m.n; ++k) {
        const double lam = 1.0 - (sab + es[k]);
        double w = next;
        if (k + 1 < m.n) next = r[(k + 1) * m.s];
        if (NEAR) {
          bool neg;
          const double s = sab + es[k], c = cab + es[m.n + k];
          if (past * fmin(s, c) > 60.0) continue;
          const double e = exp(past * spec_ln(s, c, &neg));
          w = neg && fmod(past, 2.0) != 0.0 ? -w * e : w * e;
        } else {
          for (int i = 0; i < first; ++i) w *= lam;
        }
        const double Q0 = m.Q[k], Qn = m.Q[(int64_t)(m.n - 1) * np + k];
#pragma unroll
        for (int i = 0; i <= N; ++i) {
          v0[i] += Q0 * w;
          vn[i] += Qn * w;
          if (i) acc[i - 1] += w * w;
          w *= lam;
        }
      }
#pragma unroll
      for (int i = 0; i < N; ++i)
        acc[N + i] += 2.0 * m.a * (v0[i + 1] * vn[i] + vn[i + 1] * v0[i]);
    } else {
      double S[N];
#pragma unroll
      for (int i = 0; i < N; ++i) S[i] = 0.0;
      // a cosine and its sine (the same eigenvalue) together: their largest value on any plane
      double r0 = r[0], r1 = 0.0;
      for (int k = 0; k < m.n;) {
        const bool pair = k > 0 && k + 1 < m.n;
        const double p2 = r0 * r0 + r1 * r1;
        const int up = k + (pair ? 2 : 1);
        if (up < m.n) r0 = r[up * m.s];
        r1 = up + 1 < m.n ? r[(up + 1) * m.s] : 0.0;
        const double s = sab + es[k], c = cab + es[m.n + k];
        k = up;
        if (q[0] * fmin(s, c) > 60.0) continue;      // ln(1 - x) <= -x, at every iterate of the block
        bool neg;
        const double ln = spec_ln(s, c, &neg), lam = fabs(1.0 - s);
        const double amp = sqrt(p2 * (pair ? 2.0 : 1.0) / (double)m.n);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          if (q[i] * ln < -60.0) continue;
          const double e = exp(q[i] * ln);
          S[i] += amp * e;
          acc[i] += p2 * ((e * lam) * (e * lam));
        }
      }
#pragma unroll
      for (int i = 0; i < N; ++i) acc[N + i] += 4.0 * m.a * S[i] * S[i];
    }
  }
  const double s = sum_each<2 * N>(acc, sh);
  // entry: iterate, then f or the axis; the blocks of a group side by side
  const unsigned nb = gridDim.x;
  if (threadIdx.x < 2 * N) {
    const int i = first + (int)(threadIdx.x % N);
    const bool plain = threadIdx.x < N;
    if (!plain || blockIdx.z == 0)
      partials[((int64_t)i * 4 + (plain ? 0 : 1 + blockIdx.z)) * nb + blockIdx.x] = s;
  }
  __syncthreads();                       // before the fence of thread 0
  if (!last_block(&st->arrive)) return;
  static_assert(kSpecLook * 4 <= kT && kSpecLook < 64 && kSpecFirst % kSpecEach == 0, "one thread a sum, one lane an iterate");
  if ((int)threadIdx.x < kLook * 4) {
    const int i = (int)threadIdx.x >> 2, w = (int)threadIdx.x & 3;
    double v = 0.0;
    if (w <= ss.count)
      for (unsigned b = 0; b < nb; ++b) v += partials[((int64_t)i * 4 + w) * nb + b];
    sums[i][w] = v;
  }
  __syncthreads();
  if (threadIdx.x >= 64) return;
  // a lane an iterate: is it, or the stretch up to it from the one before, clear?
  const int l = (int)threadIdx.x;
  const double T = st->T + 1.0e-24 * st->f0;
  const int from = l <= kFirst ? l : l - 1;          // whose B
  const bool ok = l < kLook && ((!NEAR && l == kFirst) ||
                                sums[l][0] - (sums[from][1] + sums[from][2] + sums[from][3]) > T);
  const int cleared = (int)__builtin_ctzll(~__ballot(ok));     // lane 63 is none
  if (l) return;
  st->arrive = 0;
  double f = 0.0, B = 0.0;
  if (cleared) {
    const double *v = sums[cleared - 1];
    f = v[0];
    B = v[1] + v[2] + v[3];
  }
  // sweeps until the rule's norm meets the threshold, about: where one mode is left B falls as f does, and
  // the square of the part across the boundaries, which B leaves out, is a / 2 of it, 1 / 12
  auto until = [&](double slope) {
    return slope < 0.0 && B < f ? fmax(0.0, log(T / (f - 0.917 * B)) / slope) : 0.0;
  };
  if (NEAR) {
    const double clear = fmin(st->end, st->clear + (double)cleared);
    double left = st->left;
    if (cleared) {
      if (clear > st->clear) st->above = f - B;
      left = 1.0 + ceil(until(st->slope));
    }
    spec_finish(js, st, base, margin, clear, st->above, left);
    return;
  }
  double clear = (double)cleared, left = 0.0;
  if (cleared > kFirst) {
    const double at = st->look[cleared - 1 - kFirst];
    clear = at;
    // ln f is convex: the chord from the nearest one before, continued, lies below it
    int was = cleared - 2 - kFirst;
    while (was >= 0 && st->look[was] >= at) --was;
    const double slope = was >= 0 ? log(f / sums[kFirst + was][0]) / (at - st->look[was]) : 0.0;
    if (slope < 0.0 && clear < st->end) {
      if (f - B > T) clear = fmin(st->end, clear + floor(log((T + B) / f) / slope));
      left = fmax(0.0, 1.0 + ceil(at + until(slope) - clear));
    }
    st->slope = slope;
  } else {
    st->slope = 0.0;
  }
  // Where the mode left is constant across the boundaries B is sharp, a few sweeps short of the stop;
  // where more are left it is several times that.
  double sharp = 0.0;
  for (int d = 0; d < ss.count; ++d) sharp += 4.0 * ss.s[d].a / (double)ss.s[d].n;
  st->near = B > 1.1 * sharp * f && clear < st->end ? 1 : 0;
  if (!st->near) {
    spec_finish(js, st, base, margin, clear, f - B, left);
    return;
  }
  st->clear = clear;
  st->above = f - B;
  st->left = left;
}

// The spectrum of the step's change of U, -af times the sum of its sweeps' residuals.
__global__ void __launch_bounds__(kT) k_spec_scale(SpecGeo g, const double *__restrict__ R,
                                                   double *__restrict__ out, const SpecState *st) {
  if (st->skip) return;
  const double q = st->steps;
  const bool odd = fmod(q, 2.0) != 0.0;
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < g.len; t += (int64_t)gridDim.x * kT) {
    const uint32_t row = (uint32_t)(t / g.PX), x = (uint32_t)(t % g.PX);
    const uint32_t y = row % (uint32_t)g.ny, z = row / (uint32_t)g.ny;
    double v = 0.0;
    if ((int)x < g.nx) {
      const double s = g.eig[0][x] + g.eig[1][y] + g.eig[2][z];
      const double c = g.eig[0][g.nx + x] + g.eig[1][g.ny + y] + g.eig[2][g.nz + z];
      bool neg;
      const double ln = spec_ln(s, c, &neg);
      const double sg = neg && odd ? -1.0 : 1.0;
      // (1 - lambda^q) / (1 - lambda)
      v = s == 0.0 ? q : (neg ? 1.0 - sg * exp(q * ln) : -expm1(q * ln)) / s;
      v = -g.af * v * R[t];
    }
    out[t] = v;
  }
}

// U_to = U_base + its change on interior nodes, into the sweeps' buffer of iterate `to`.
__global__ void __launch_bounds__(kT) k_spec_apply(SpecGeo g, const double *__restrict__ du,
                                                   const double *u, double *b0, double *b1,
                                                   double *b2, const SpecState *st) {
  if (st->skip) return;
  const int r = (int)(st->to % 3);
  double *out = r == 0 ? b0 : (r == 1 ? b1 : b2);
  for (int64_t t = (int64_t)blockIdx.x * kT + threadIdx.x; t < g.len; t += (int64_t)gridDim.x * kT) {
    const uint32_t row = (uint32_t)(t / g.PX), x = (uint32_t)(t % g.PX);
    if ((int)x >= g.nx) continue;
    const uint32_t y = row % (uint32_t)g.ny, z = row / (uint32_t)g.ny;
    const int64_t c = (x + 1) + g.X * (int64_t)(y + 1) + g.XY * (int64_t)(z + 1);
    out[c] = u[c] + du[t];
  }
}

// One axis of the transform over the whole array: 36 TFLOP/s FP64 at 160^3
// (37 us), 43 at 128^3 (20 us), where a large library product reaches 73.  Axis tiles of a column tile
// next to each other on one XCD (block b runs on XCD b % 8), so that the
// columns are read from its L2 after the first.
template <int AT, bool XAXIS>
__global__ void __launch_bounds__(kSpecT) k_spec_axis(SpecTile t, int nat, int64_t nct,
                                                      const SpecState *st) {
  __shared__ double lds[2 * kSpecLds];
  if (st && st->skip) return;
  const int64_t i = blockIdx.x >> 3;
  const int at = (int)(i % nat);
  const int64_t ct = (i / nat) * 8 + (blockIdx.x & 7);
  if (ct >= nct) return;
  spec_tile<AT, XAXIS>(t, at * 32 * AT, ct * kSpecCols, lds);
}

template <bool XAXIS>
void launch_axis(hipStream_t s, const SpecTile &t, const SpecState *st) {
  const int64_t nct = (t.total + kSpecCols - 1) / kSpecCols;
  // outputs in tiles of 64, or of 32 where that pads less
  const bool wide = ((t.nout + 63) & ~63) == ((t.nout + 31) & ~31);
  const int nat = wide ? (t.nout + 63) / 64 : (t.nout + 31) / 32;
  const unsigned blocks = (unsigned)(((nct + 7) & ~int64_t(7)) * nat);
  if (wide) k_spec_axis<2, XAXIS><<<blocks, kSpecT, 0, s>>>(t, nat, nct, st);
  else k_spec_axis<1, XAXIS><<<blocks, kSpecT, 0, s>>>(t, nat, nct, st);
}

}  // namespace

// The forms that are held to the reference's rounding use it to find their
// stop, where the sweeps up to it can do without the stop test.
bool spec_eligible(const picard_ctx *c) { return c->spec_mem && !(c->split && c->mx_forced); }

// The split form's FP64 iterates go with them: its own sweeps do without.
void spec_release(picard_ctx *c) {
  if (c->spec_mem) (void)hipFree(c->spec_mem);
  c->spec_mem = nullptr;
  for (int q = 0; q < 3 && c->split; ++q) {
    if (c->jb_mem[q]) (void)hipFree(c->jb_mem[q]);
    c->jb_mem[q] = c->jb[q] = nullptr;
  }
}

// Basis, transpose and eigenvalue parts of one axis; `a` is the Jacobi weight of its neighbours.
int spec_axis_tables(hipStream_t s, int n, bool flow, double a, double *fwd, double *inv, double *eig) {
  k_spec_basis<<<grid_blocks(spec_mat_len(n), kT), kT, 0, s>>>(n, flow, a, fwd, inv, eig);
  PICARD_HIP(hipGetLastError());
  return PICARD_OK;
}

// One basis applied along one axis of one array (bcpot_modes.hip).
int spec_product(hipStream_t s, const SpecTile &t, bool xaxis) {
  if (xaxis) launch_axis<true>(s, t, nullptr);
  else launch_axis<false>(s, t, nullptr);
  PICARD_HIP(hipGetLastError());
  return PICARD_OK;
}

// Largest ln|lambda| of a box from the axes' smallest 4 a sin^2 and 4 a cos^2.
double spec_slowest(const int n[3], const int flow[3], const double a[3]) {
  double smin = 0.0, cmin = 0.0;
  const double pi = 3.14159265358979323846;
  for (int d = 0; d < 3; ++d) {
    const double h = flow[d] ? 0.5 / (n[d] + 1) : 0.0;
    const double k = flow[d] ? 0.5 / (n[d] + 1) : (n[d] % 2 ? 0.5 / n[d] : 0.0);
    smin += 4.0 * a[d] * std::sin(pi * h) * std::sin(pi * h);
    cmin += 4.0 * a[d] * std::sin(pi * k) * std::sin(pi * k);
  }
  return std::log1p(-std::fmin(smin, cmin));
}

// The axes' bases and eigenvalues, and the transforms' buffers.
int spec_create(picard_ctx *c) {
  const GridDims &g = c->gd;
  const int n[3] = {g.nx, g.ny, g.nz};
  if (!(c->split || c->order_free || jacobi_block_eligible(g)) || n[0] > kSpecMaxAxis ||
      n[1] > kSpecMaxAxis || n[2] > kSpecMaxAxis)
    return PICARD_OK;
  const double d2[3] = {g.dxyz[0] * g.dxyz[0], g.dxyz[1] * g.dxyz[1], g.dxyz[2] * g.dxyz[2]};
  const double sum = 1.0 / d2[0] + 1.0 / d2[1] + 1.0 / d2[2];
  // one allocation, its parts at multiples of 256 bytes
  auto part = [](int64_t doubles) { return (doubles + 31) & ~int64_t(31); };
  const int64_t len = part((int64_t)((g.nx + 15) & ~15) * g.ny * g.nz);
  const int64_t state = part((int64_t)(sizeof(SpecState) + sizeof(double) - 1) / (int64_t)sizeof(double));
  int64_t total = 3 * len + state;
  for (int d = 0; d < 3; ++d) total += 2 * spec_mat_len(n[d]) + part(2 * n[d]);
  hipError_t rc = hipMalloc(&c->spec_mem, sizeof(double) * total);
  for (int q = 0; q < 3 && c->split && rc == hipSuccess; ++q) {
    rc = hipMalloc(&c->jb_mem[q], sizeof(double) * (g.G + 2));
    c->jb[q] = c->jb_mem[q] + 1;
  }
  if (rc != hipSuccess) {
    (void)hipGetLastError();
    spec_release(c);
    if (rc == hipErrorOutOfMemory) return PICARD_OK;
    PICARD_HIP(rc);
  }
  double *p = c->spec_mem;
  auto take = [&](int64_t doubles) {
    double *q = p;
    p += doubles;
    return q;
  };
  for (double *&b : c->spec_buf) b = take(len);
  double w[3];
  for (int d = 0; d < 3; ++d) {
    c->spec_fwd[d] = take(spec_mat_len(n[d]));     // a multiple of 16 x 64 doubles
    c->spec_inv[d] = take(spec_mat_len(n[d]));
    c->spec_eig[d] = take(part(2 * n[d]));
    w[d] = 0.5 / (d2[d] * sum);                       // ax, ay, az of CalcEpotential.f90:44-47
    PICARD_TRY(spec_axis_tables(c->stream, n[d], g.flow[d], w[d], c->spec_fwd[d], c->spec_inv[d],
                                c->spec_eig[d]));
  }
  c->spec_lnmax = spec_slowest(n, g.flow, w);
  c->spec_st = reinterpret_cast<SpecState *>(take(state));
  PICARD_HIP(hipMemsetAsync(c->spec_st, 0, sizeof(SpecState), c->stream));
  static_assert(sizeof(JacobiState) <= kHostState / 2 && sizeof(SpecState) <= kHostState / 2, "pinned mirrors");
  c->spec_host = reinterpret_cast<SpecState *>(reinterpret_cast<char *>(c->js_host) + kHostState / 2);
  return PICARD_OK;
}

// From iterate `base` (in `u`, guard layout; `old`: the one before, if there is one) to an iterate at
// least `margin` before the one the stop rule will pick, left in the sweeps' buffers jb.  *to: that
// iterate, *ahead: sweeps to about the stop; or, with nothing done, kSpecFewLeft: too few sweeps are
// left for a step, kSpecNoNorm: the residual has no finite norm, kSpecNotClear: early iterates may
// pass the rule (few cells between periodic boundaries).
int spec_step(picard_ctx *c, const double *u, const double *old, int64_t base, int margin, bool apply, int64_t *to,
              int64_t *ahead) {
  const GridDims &g = c->gd;
  hipStream_t s = c->stream;
  SpecGeo sg;
  sg.nx = g.nx; sg.ny = g.ny; sg.nz = g.nz;
  sg.PX = (g.nx + 15) & ~15;
  sg.X = g.X; sg.XY = (int64_t)g.X * g.Y;
  sg.px = !g.flow[0]; sg.py = !g.flow[1]; sg.pz = !g.flow[2];
  sg.len = (int64_t)sg.PX * g.ny * g.nz;
  const double dx = g.dxyz[0], dy = g.dxyz[1], dz = g.dxyz[2];
  const double den = 1.0 / ((dx * dy) * (dx * dy) + (dx * dz) * (dx * dz) + (dy * dz) * (dy * dz));
  sg.ax = 0.5 * den * ((dy * dz) * (dy * dz));            // CalcEpotential.f90:44-47
  sg.ay = 0.5 * den * ((dx * dz) * (dx * dz));
  sg.az = 0.5 * den * ((dx * dy) * (dx * dy));
  sg.af = 0.5 * den * ((dx * dy * dz) * (dx * dy * dz));
  sg.dx2 = dx * dx; sg.dy2 = dy * dy; sg.dz2 = dz * dz;
  for (int d = 0; d < 3; ++d) sg.eig[d] = c->spec_eig[d];
  SpecState *st = c->spec_st;
  double *B0 = c->spec_buf[0], *B1 = c->spec_buf[1], *B2 = c->spec_buf[2];
  const int64_t P = (int64_t)sg.PX * g.ny;
  auto axis = [&](int d, double *const *mat, const double *in, double *out) {
    SpecTile t;
    t.M = mat[d];
    t.in = in;
    t.out = out;
    t.n = d == 0 ? g.nx : (d == 1 ? g.ny : g.nz);
    t.np = spec_cols(t.n);
    t.nout = d == 0 ? sg.PX : t.n;
    t.ld = d == 2 ? P : sg.PX;
    t.gs = d == 1 ? P : 0;
    t.ldo = t.ld;
    t.gso = t.gs;
    t.total = d == 0 ? (int64_t)g.ny * g.nz : (d == 1 ? (int64_t)sg.PX * g.nz : P);
    t.gpr = (uint32_t)((d == 1 ? sg.PX : t.total) / 16);
    if (d == 0) launch_axis<true>(s, t, st);
    else launch_axis<false>(s, t, st);
  };
  // blocks of the passes over the array: one per CU while they have work, then eight
  // elements a thread, four per CU at most; their partials fit the context's array (the search keeps
  // eight sums per block)
  int64_t nb = std::max((sg.len + 8 * kT - 1) / (8 * kT), std::min<int64_t>((sg.len + kT - 1) / kT, 256));
  if (nb > 1024) nb = 1024;
  const int64_t cap = 4 * c->s.partials_len / kSpecCand;
  if (nb > cap) nb = cap;
  const unsigned B = (unsigned)(nb < 1 ? 1 : nb);
  double *part = c->s.partials;
  k_spec_residual<<<B, kT, 0, s>>>(sg, u, old, c->b, B0, part, c->js, st, base, c->spec_lnmax);
  axis(0, c->spec_fwd, B0, B1);
  axis(1, c->spec_fwd, B1, B2);
  axis(2, c->spec_fwd, B2, B0);
  SpecSeams ss;
  ss.count = 0;
  const int n[3] = {g.nx, g.ny, g.nz};
  const int64_t stride[3] = {1, sg.PX, P};
  const double weight[3] = {sg.ax, sg.ay, sg.az};
  int64_t columns = 0;
  for (int d = 0; d < 3; ++d) {
    if (g.flow[d]) continue;
    const int a = d == 0 ? 1 : 0, b = d == 2 ? 1 : 2;
    ss.s[ss.count++] = SpecSeam{n[d], n[a], n[b], stride[d], stride[a], stride[b], d, a, b, weight[d],
                                c->spec_fwd[d]};
    columns = std::max(columns, (int64_t)n[a] * n[b]);
  }
  for (int p = 0; p < kSpecPasses; ++p)
    k_spec_search<<<B, kT, 0, s>>>(sg, B0, part, c->js, st, base, margin, ss.count, p);
  if (ss.count) {
    const int64_t room = 4 * c->s.partials_len / (4 * kSpecLook);
    const int64_t nb = std::max<int64_t>(1, std::min((columns + kT - 1) / kT, room));
    k_spec_clear<false><<<dim3((unsigned)nb, kSpecLook / kSpecEach, ss.count), kT, 0, s>>>(
        sg, ss, B0, part, c->js, st, base, margin);
    k_spec_clear<true><<<dim3((unsigned)nb, kSpecNear / kSpecEach, ss.count), kT, 0, s>>>(
        sg, ss, B0, part, c->js, st, base, margin);
  }
  if (apply) {
    k_spec_scale<<<B, kT, 0, s>>>(sg, B0, B1, st);
    axis(0, c->spec_inv, B1, B2);
    axis(1, c->spec_inv, B2, B1);
    axis(2, c->spec_inv, B1, B2);
    k_spec_apply<<<B, kT, 0, s>>>(sg, B2, u, c->jb[0], c->jb[1], c->jb[2], st);
  }
  PICARD_HIP(hipGetLastError());
  PICARD_HIP(hipMemcpyAsync(c->spec_host, st, sizeof(SpecState), hipMemcpyDeviceToHost, s));
  PICARD_HIP(hipStreamSynchronize(s));
  const SpecState *h = c->spec_host;
  *to = h->skip ? (h->skip == kSpecBad ? kSpecNoNorm : (h->skip == kSpecUnclear ? kSpecNotClear : kSpecFewLeft))
                : h->to;
  *ahead = h->skip ? 0 : h->ahead;
  return PICARD_OK;
}

}  // namespace picard
