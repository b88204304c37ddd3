// bcpot_seq.hip -- BCpotentials (BCpotentials.f90:51-141) in the reference's
// order: every face node's value is one chain of N_x N_y N_z additions, k, then
// j, then i fastest, of C(interior) * D(window).
//
// Bound: the chain.  A lane owns one face node, so the time is the number of
// cells times what a product and a dependent addition take (12.5 cycles of
// 2.4 GHz, measured), if the operands keep up: the lanes of a wave need the
// same charge and neighbouring distances.  Charge and distances are staged in
// LDS kRB rows at a time, the next kRB rows on their way from memory meanwhile
// (a trip takes longer than a short row's sums); the charge comes out as
// one LDS read per 16 terms, spread by row broadcasts (read per term it and the
// distances would take 27 cycles a term, the LDS rate of one wave).
// Face nodes of all open dimensions go out in one launch of one-wave blocks: few
// chains are there to fill the chip (2 N^2 / 64 waves per dimension), so none waits
// for another's face.
//  - x faces, lanes along y: the distances of a charge row j are D(., j - jj), one
//    column of N_x values per lane offset; a ring in LDS holds the columns that
//    the lanes use and takes one new column per row.
//  - y and z faces, lanes along x: one row of N_x + 63 distances per charge row.
#include <type_traits>

#include "picard_internal.h"

namespace picard {
namespace {

constexpr int kU = 16;              // terms per group
constexpr int kRB = 4;              // rows staged at a time
constexpr int kRing = 64 + kRB;     // x faces: columns held
constexpr int kPitch = kRing + 1;   // odd, so that a column's values spread over the banks
constexpr int kMaxNC = 3;           // 64-cell chunks of a charge row

struct FaceTask {
  int nx, ny, nz;
  int64_t X, XY, DX, DXY;
  int tasks[3];                     // blocks of the x, y and z faces
  double kfac;
};

// lane q of the lane's row of 16, in every lane of the row
template <int Q>
__device__ __forceinline__ double row_bcast(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x150 + Q, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x150 + Q, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

template <int A, int B, typename F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

// Between lanes' stores to LDS and other lanes' reads of them, and between those reads and the next
// stores there.  A block is one wave, whose LDS accesses the hardware keeps in order: this holds
// the compiler to it and costs no instruction.
__device__ __forceinline__ void staged() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// LDS of one block, in doubles: charge rows, then the ring or the rows of distances.
template <int NC>
constexpr int kFaceLds = kRB * 64 * NC + (64 * NC * kPitch > kRB * 64 * (NC + 1) ? 64 * NC * kPitch
                                                                               : kRB * 64 * (NC + 1));

// The sum of one task's lanes, N_x <= 64 NC.  XF: element i of a charge row's
// distances is at base + i kPitch in LDS, otherwise at base + i.  Rows and
// columns are staged whole chunks at a time: lanes past the end repeat the last
// value, which no sum takes, so that nothing in the staging is conditional.
template <bool XF, int NC>
__device__ __forceinline__ double face_chain(const FaceTask &t, const double *__restrict__ C,
                                             const double *__restrict__ D, double *lds, int a0,
                                             int bb, int dim, int face) {
  const int lane = (int)threadIdx.x;
  const int nx = t.nx, ny = t.ny, nz = t.nz;
  constexpr int ST = XF ? kPitch : 1;
  constexpr int ND = XF ? NC : NC + 1;                 // chunks of a staged row of distances
  constexpr int NP = 64 * NC, SEG = 64 * ND;
  double *const crow = lds;                            // kRB charge rows
  double *const dist = lds + kRB * NP;                 // ring, or kRB rows of distances
  // distances of row (k, j): x faces the column of lane 0 (y offset j - a0), y/z
  // faces the row; both advance by one y index with j and one z index with k
  int64_t yi, zi;                                      // 0-based D indices of row (1, 1)
  if (dim == 1) {                                      // BCpotentials.f90:91/94
    yi = face == 0 ? ny + 1 : 0;
    zi = nz + 1 - bb;
  } else if (dim == 2) {                               // :122/125
    yi = ny + 1 - bb;
    zi = face == 0 ? nz + 1 : 0;
  } else {                                             // :60/63
    yi = ny + 1 - a0;
    zi = nz + 1 - bb;
  }
  // staged value m of a row: x faces cell m; y/z faces x index nx - a0 - 62 + m
  // (lane l, cell i, 0-based: nx + 1 + i - a0 - l, that is m = i + 63 - l)
  const int x0 = XF ? (face == 0 ? nx + 1 : 0) : nx - a0 - 62;
  uint32_t xo[ND], co[NC];                             // the lane's values, inside the rows
#pragma unroll
  for (int q = 0; q < ND; ++q) {
    const int x = x0 + lane + 64 * q;
    xo[q] = (uint32_t)(x < 0 ? 0 : (x > 2 * nx ? 2 * nx : x));
  }
#pragma unroll
  for (int q = 0; q < NC; ++q) co[q] = (uint32_t)(lane + 64 * q < nx ? lane + 64 * q : nx - 1);
  auto store = [&](const double (&r)[ND], int slot) {
#pragma unroll
    for (int q = 0; q < ND; ++q) {
      const int m = lane + 64 * q;
      dist[XF ? m * kPitch + slot : slot * SEG + m] = r[q];
    }
  };
  // the batch of rows on its way: rows (fk, fj) ... of one plane, past the last
  // plane the last one's again
  double rd[kRB][ND], rc[kRB][NC];
  const double *fd = D + t.DX * yi + t.DXY * zi, *fc = C + 1 + t.X + t.XY;
  int fj = 1, fk = 1;
  auto fetch = [&]() {
    const int left = ny - fj;                          // rows after the first
#pragma unroll
    for (int b = 0; b < kRB; ++b) {
      const int h = b < left ? b : left;
      const double *dp = fd + t.DX * h, *cp = fc + t.X * h;
#pragma unroll
      for (int q = 0; q < ND; ++q) rd[b][q] = dp[xo[q]];
#pragma unroll
      for (int q = 0; q < NC; ++q) rc[b][q] = cp[co[q]];
    }
    if (left >= kRB) {
      fj += kRB;
      fd += t.DX * kRB;
      fc += t.X * kRB;
    } else {
      const int64_t up = fk < nz ? 1 : 0;
      fd += t.DXY * up - t.DX * (fj - 1);
      fc += t.XY * up - t.X * (fj - 1);
      fj = 1;
      ++fk;
    }
  };
  double s = 0.0;
  auto read = [&](double &c, double (&d)[kU], const double *cp, const double *dp) {
    c = cp[lane & 15];
#pragma unroll
    for (int q = 0; q < kU; ++q) d[q] = dp[q * ST];
  };
  // all products, then the chain: issued in turn, each addition would wait for
  // its product and that for its broadcast
  auto products = [&](double (&p)[kU], double c, const double (&d)[kU]) {
    static_for<0, kU>([&](auto q) { p[q.value] = row_bcast<q.value>(c) * d[q.value]; });
    __builtin_amdgcn_sched_barrier(0);
  };
  auto sum = [&](double c, const double (&d)[kU]) {
    double p[kU];
    products(p, c, d);
#pragma unroll
    for (int q = 0; q < kU; ++q) s = s + p[q];
  };
  const int full = nx / kU, part = nx - full * kU;
  int slot = 0;                                        // x faces: the row's newest column
  fetch();
  for (int k = 1; k <= nz; ++k) {
    staged();                                          // the last plane's reads
    if (XF) {                                          // a new plane: the 63 older columns
      slot = 63;
      // below y = 0 there is no column, and no lane with a node uses one
      const double *dp = D + t.DXY * (int64_t)(nz + k - bb);
#pragma unroll 1
      for (int l = 63; l >= 1; l -= 9) {
        double w[9][ND];
#pragma unroll
        for (int h = 0; h < 9; ++h) {
          const int y = ny + 1 - a0 - (l - h);
          const double *p = dp + t.DX * (int64_t)(y < 0 ? 0 : y);
#pragma unroll
          for (int q = 0; q < ND; ++q) w[h][q] = p[xo[q]];
        }
#pragma unroll
        for (int h = 0; h < 9; ++h) store(w[h], 63 - (l - h));
      }
    }
    for (int j = 1; j <= ny; j += kRB) {
      staged();                                        // the last rows' reads
#pragma unroll
      for (int b = 0; b < kRB; ++b) {
        const int sl = XF ? (slot + b >= kRing ? slot + b - kRing : slot + b) : b;
        store(rd[b], sl);
#pragma unroll
        for (int q = 0; q < NC; ++q) crow[b * NP + lane + 64 * q] = rc[b][q];
      }
      staged();
      fetch();
      const int rows = ny + 1 - j < kRB ? ny + 1 - j : kRB;
      for (int b = 0; b < rows; ++b) {
        const int base = XF ? (slot - lane < 0 ? slot - lane + kRing : slot - lane) : b * SEG + 63 - lane;
        const double *cp = crow + b * NP, *dp = dist + base;
        double ca, cb, da[kU], db[kU];
        // pairs of groups without a branch inside, each reading one group ahead
        // (after the last the row's first again)
        read(ca, da, cp, dp);
        int g = 0;
        for (; g + 2 <= full; g += 2) {
          read(cb, db, cp + kU, dp + kU * ST);
          sum(ca, da);
          const int step = g + 2 < full || part ? 2 * kU : -g * kU;
          cp += step;
          dp += step * ST;
          read(ca, da, cp, dp);
          sum(cb, db);
        }
        if (g < full) {
          if (part) read(cb, db, cp + kU, dp + kU * ST);
          sum(ca, da);
          ca = cb;
#pragma unroll
          for (int q = 0; q < kU; ++q) da[q] = db[q];
        }
        if (part) {
          double p[kU];
          products(p, ca, da);
#pragma unroll
          for (int q = 0; q < kU; ++q)
            if (q < part) s = s + p[q];
        }
        if (++slot == kRing) slot = 0;
      }
    }
  }
  return s;
}

template <int NC>
__global__ void __launch_bounds__(64) k_bcpot_seq(FaceTask t, const double *__restrict__ C,
                                                  const double *__restrict__ D,
                                                  double *__restrict__ U) {
  __shared__ double lds[kFaceLds<NC>];
  int b = (int)blockIdx.x, dim = 0;
  while (dim < 2 && b >= t.tasks[dim]) b -= t.tasks[dim++];
  const int na = dim == 0 ? t.ny : t.nx;               // face nodes along the lanes
  const int nb = dim == 2 ? t.ny : t.nz;
  const int tiles = (na + 63) / 64;
  const int a0 = (b % tiles) * 64 + 1;
  b /= tiles;
  const int bb = b % nb + 1, face = b / nb;
  const double s = dim == 0 ? face_chain<true, NC>(t, C, D, lds, a0, bb, dim, face)
                            : face_chain<false, NC>(t, C, D, lds, a0, bb, dim, face);
  const int a = a0 + (int)threadIdx.x;
  if (a > na) return;
  const int64_t g1 = face == 0 ? 0 : (dim == 0 ? t.nx : (dim == 1 ? t.ny : t.nz)) + 1;
  const int64_t at = dim == 0   ? g1 + t.X * a + t.XY * bb
                     : dim == 1 ? a + t.X * g1 + t.XY * bb
                                : a + t.X * bb + t.XY * g1;
  U[at] = s * t.kfac;
}

}  // namespace

// At most 192 cells a row.  Measured against the kernels that share charge or
// distances between the chains of a block (grid.hip): 32^3 x faces 2.43 -> 0.63 ms,
// 64^3 23.2 -> 3.9, 128^3 154 -> 27.5, 190x190x160 404 -> 291, all faces of
// 49x72x60 182 -> 4.4.  Beyond, the ring leaves room for one wave a CU, and the
// 131072 chains of 256^3 would take eight rounds.
bool bcpot_seq_eligible(const GridDims &g) { return g.nx <= 64 * kMaxNC; }

int launch_bcpot_seq(picard_ctx *c, double kfac) {
  const GridDims &g = c->gd;
  FaceTask t;
  t.nx = g.nx; t.ny = g.ny; t.nz = g.nz;
  t.X = g.X; t.XY = (int64_t)g.X * g.Y;
  t.DX = 2 * (int64_t)g.nx + 1;
  t.DXY = t.DX * (2 * (int64_t)g.ny + 1);
  t.kfac = kfac;
  int total = 0;
  for (int d = 0; d < 3; ++d) {
    const int na = d == 0 ? g.ny : g.nx, nb = d == 2 ? g.ny : g.nz;
    t.tasks[d] = g.flow[d] ? 2 * nb * ((na + 63) / 64) : 0;
    total += t.tasks[d];
  }
  if (!total) return PICARD_OK;
  if (g.nx <= 64) k_bcpot_seq<1><<<total, 64, 0, c->stream>>>(t, c->C, c->D, c->U);
  else if (g.nx <= 128) k_bcpot_seq<2><<<total, 64, 0, c->stream>>>(t, c->C, c->D, c->U);
  else k_bcpot_seq<3><<<total, 64, 0, c->stream>>>(t, c->C, c->D, c->U);
  PICARD_HIP(hipGetLastError());
  return PICARD_OK;
}

}  // namespace picard
