// jacobi_block.hip -- several FP64 Jacobi sweeps per launch with the
// reference's rounding, for the stretch of a solve in which no stop test is
// due (CalcEpotential.f90:74-80 and :100-239 without :83-96).
//
// Bound on small and middle grids: a pass of one sweep costs its launch, one
// trip to memory and the reduction of its residual, 10 us at 16^3 and 16 at 64^3,
// hardly any of it arithmetic.  Here a block keeps a tile of TY x TZ rows (y, z) of the whole x
// extent with a halo of T rows on every side, takes T sweeps on chip, each
// valid on one row less all around, and stores the tile: one launch and one
// trip to memory per T sweeps, for (TY + 2T)(TZ + 2T) / (TY TZ) times the loads
// (from L2: an XCD's blocks own neighbouring tiles).  A wave owns one y row and all the tile's z planes
// in registers, so z-neighbours are its own and x-neighbours come by wave
// shifts; only the y-neighbours go through LDS, one write and two reads a row.
// Every cell's arithmetic is k_jacobi_pass's, in its operand order; a periodic
// neighbour is an image that the tile computes for itself from the same values.
#include "picard_internal.h"

namespace picard {
namespace {

struct BlockGeo {
  int nx, ny, nz;
  int64_t X, XY;                 // node strides
  int px, py, pz;
  int nyt, nzt;                  // tiles
  double ax, ay, az, af;
};

// value of the next lower / higher lane (0 past the wave's ends)
__device__ __forceinline__ double lane_below(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_above(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double at_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

// CX cells a lane (x = lane + 64 c), nx <= 64 CX.
template <int CX, int T, int TY, int TZ, bool PX>
__global__ void __launch_bounds__(64 * (TY + 2 * T)) k_jacobi_block(BlockGeo g,
                                                                     const double *__restrict__ in,
                                                                     double *__restrict__ out,
                                                                     const double *__restrict__ b) {
  constexpr int NY = TY + 2 * T, NZ = TZ + 2 * T;
  // two copies where they fit: then one barrier a sweep
  constexpr int NB = T > 2 && 2 * NY * NZ * CX * 512 <= 150 * 1024 ? 2 : 1;
  __shared__ double rows[NB][NY][NZ][64 * CX];
  const int lane = (int)threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.y);
  // tile: an eighth of them, y fastest, to XCD blockIdx.x % 8 (whole z slabs gave
  // some XCDs more tiles than CUs: 4.2 us a sweep at 40x60x70, now 2.4)
  const int tile = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
  if (tile >= g.nyt * g.nzt) return;           // the whole block
  const int tz = tile / g.nyt, ty = tile % g.nyt;
  const int y0 = ty * TY, z0 = tz * TZ;
  // the wave's row: interior (or an image of one), a flow guard, or nothing
  int y = y0 - T + w;
  bool inner = y >= 0 && y < g.ny;
  if (g.py && !inner) {
    y %= g.ny;
    if (y < 0) y += g.ny;
    inner = true;
  }
  // Every load is unconditional, so that a wave waits for memory once: rows and
  // planes beyond the guards, and lanes past the row's end, take the nearest
  // ones' values, which nothing that is kept reads.
  y = y < -1 ? -1 : (y > g.ny ? g.ny : y);
  double u[NZ][CX], bf[NZ][CX];
  double end[NZ];                              // flow x: the row's guards, east in lane xl, west elsewhere
  uint32_t zin = 0;                            // planes that the sweeps update
  const int xl = g.nx - 1 - 64 * (CX - 1);     // lane of the row's last cell
  uint32_t xo[CX];
  const uint32_t eo = lane == xl ? (uint32_t)g.nx + 1 : 0;
#pragma unroll
  for (int c = 0; c < CX; ++c) xo[c] = (uint32_t)(lane + 64 * c < g.nx ? lane + 64 * c : g.nx - 1) + 1;
#pragma unroll
  for (int zi = 0; zi < NZ; ++zi) {
    int z = z0 - T + zi;
    bool in_z = z >= 0 && z < g.nz;
    if (g.pz && !in_z) {
      z %= g.nz;
      if (z < 0) z += g.nz;
      in_z = true;
    }
    if (in_z) zin |= 1u << zi;
    z = z < -1 ? -1 : (z > g.nz ? g.nz : z);
    const int64_t row = g.X * (int64_t)(y + 1) + g.XY * (int64_t)(z + 1);
    const double *ur = in + row, *br = b + row;
#pragma unroll
    for (int c = 0; c < CX; ++c) {
      u[zi][c] = ur[xo[c]];
      if (zi > 0 && zi < NZ - 1) bf[zi][c] = br[xo[c]];
    }
    if (!PX && zi > 0 && zi < NZ - 1) end[zi] = ur[eo];
  }
#pragma unroll
  for (int zi = 1; zi < NZ - 1; ++zi) {
#pragma unroll
    for (int c = 0; c < CX; ++c) bf[zi][c] = g.af * bf[zi][c];
  }
#pragma unroll
  for (int s = 1; s <= T; ++s) {
    auto &buf = rows[NB == 2 ? s & 1 : 0];
    if (NB == 1 && s > 1) __syncthreads();     // the last sweep's reads
    if (w >= s - 1 && w <= NY - s) {           // those that a row of this sweep reads
#pragma unroll
      for (int zi = s; zi < NZ - s; ++zi)
#pragma unroll
        for (int c = 0; c < CX; ++c) buf[w][zi][lane + 64 * c] = u[zi][c];
    }
    __syncthreads();
    if (!inner || w < s || w >= NY - s) continue;   // the whole wave
    // the y-neighbours of every plane first: one wait for LDS a sweep
    double un[NZ][CX], us[NZ][CX];
#pragma unroll
    for (int zi = s; zi < NZ - s; ++zi)
#pragma unroll
      for (int c = 0; c < CX; ++c) {
        un[zi][c] = buf[w + 1][zi][lane + 64 * c];
        us[zi][c] = buf[w - 1][zi][lane + 64 * c];
      }
    // planes that all are swept, away from flow guards, without the selects
    const bool every = T > 2 && (zin & (((1u << (NZ - 2 * s)) - 1) << s)) == (((1u << (NZ - 2 * s)) - 1) << s);
#pragma unroll
    for (int way = T > 2 ? 0 : 1; way < 2; ++way) {
      const bool all = way == 0;
      if (all != every) continue;
      double below[CX];
#pragma unroll
      for (int c = 0; c < CX; ++c) below[c] = u[s - 1][c];
#pragma unroll
      for (int zi = s; zi < NZ - s; ++zi) {
        double cur[CX];
#pragma unroll
        for (int c = 0; c < CX; ++c) cur[c] = u[zi][c];
        // a plane that is not swept (a flow guard, or beyond one) keeps its
        // value by a select: a branch per row left each row's LDS reads and its
        // chain of ten operations unoverlapped (64^3: 3.4 us a sweep)
        const bool swept = all || (zin >> zi & 1);
#pragma unroll
        for (int c = 0; c < CX; ++c) {
          double uw = lane_below(cur[c]), ue = lane_above(cur[c]);
          const double w0 = c > 0 ? at_lane(cur[c > 0 ? c - 1 : 0], 63)
                                  : (PX ? at_lane(cur[CX - 1], xl)
                                        : (CX == 1 ? end[zi] : at_lane(end[zi], xl == 0 ? 1 : 0)));
          const double e0 = c + 1 < CX ? at_lane(cur[c + 1 < CX ? c + 1 : c], 0)
                                       : (PX ? at_lane(cur[0], 0)
                                             : (CX == 1 ? end[zi] : at_lane(end[zi], xl)));
          uw = lane == 0 ? w0 : uw;
          ue = lane == (c == CX - 1 ? xl : 63) ? e0 : ue;
          // CalcEpotential.f90:74-80
          const double v = g.ax * (ue + uw) + g.ay * (un[zi][c] + us[zi][c]) +
                           g.az * (u[zi + 1][c] + below[c]) - bf[zi][c];
          u[zi][c] = swept ? v : cur[c];
        }
#pragma unroll
        for (int c = 0; c < CX; ++c) below[c] = cur[c];
      }
    }
  }
  if (w < T || w >= T + TY || y0 - T + w >= g.ny) return;
#pragma unroll
  for (int zi = T; zi < T + TZ; ++zi) {
    const int z = z0 - T + zi;
    if (z >= g.nz) break;
    const int64_t row = g.X * (int64_t)(y + 1) + g.XY * (int64_t)(z + 1);
#pragma unroll
    for (int c = 0; c < CX; ++c)
      if (lane + 64 * c < g.nx) out[row + lane + 64 * c + 1] = u[zi][c];
  }
}

template <int CX, int T, int TY, int TZ>
void launch(hipStream_t s, BlockGeo g, const double *in, double *out, const double *b) {
  g.nyt = (g.ny + TY - 1) / TY;
  g.nzt = (g.nz + TZ - 1) / TZ;
  const int blocks = (g.nyt * g.nzt + 7) / 8 * 8;
  const dim3 block(64, TY + 2 * T);
  if (g.px) k_jacobi_block<CX, T, TY, TZ, true><<<blocks, block, 0, s>>>(g, in, out, b);
  else k_jacobi_block<CX, T, TY, TZ, false><<<blocks, block, 0, s>>>(g, in, out, b);
}

}  // namespace

// Rows of at most 128 cells: two cells a lane fill the registers and LDS.
// Wider grids are bound by memory and take the passes of one sweep.
bool jacobi_block_eligible(const GridDims &g) { return g.nx <= 128; }

// Tile and sweeps per launch, by what is resident at once on 256 CUs: beyond
// that a launch runs in rounds and every round pays the trip to memory. Measured,
// us per sweep (a pass of one sweep: 11.1 at 32^3, 17 at 49x72x60, 15.9 at 64^3), 4.4 us of
// a launch being its start, loads and stores:
//   rows to 64, the smallest tile that has at most 256, x 4 sweeps: 2x2 1.59 at 32^3 (4x4: 2.2);
//   3x3 1.83 at 48^3 (4x4: 2.05); 4x4 2.19 at 64^3 (x 2 sweeps: 2.4, 2x2 x 4: 5.1); 5x4
//   2.40 at 49x72x60 and 6x4 2.71 at 64x96x64 (4x4 x 2: 2.92 and 3.16);
//   beyond, 4x4 x 2 3.68 at 64x96x96 (576 tiles; 6x6 x 4: 4.04, registers spilled);
//   rows to 128: 4x4 x 2 4.75 at 72^3 (324 tiles, two resident a CU; 6x6: 5.02)
//   and 6.45 at 128x100x96 (600; 6x6, 272: 8.56); 6x6 x 2 5.21 at 96^3 (256,
//   one a CU; 4x4, 576: 6.63).
// Before the planes that a sweep needs alone were loaded and stored in LDS, the rows kept
// twice there (one barrier a sweep) and the selects left out away from flow guards: 1.69
// at 32^3, 2.39 at 64^3.
enum BlockPlan { kRows22x4, kRows33x4, kRows44x4, kRows54x4, kRows64x4, kRows44x2, kWide44x2, kWide66x2 };

static BlockPlan block_plan(const GridDims &g) {
  auto tiles = [&](int ty, int tz) {
    return (int64_t)((g.ny + ty - 1) / ty) * ((g.nz + tz - 1) / tz);
  };
  if (g.nx <= 64) {
    if (tiles(2, 2) <= 256) return kRows22x4;
    if (tiles(3, 3) <= 256) return kRows33x4;
    if (tiles(4, 4) <= 256) return kRows44x4;
    if (tiles(5, 4) <= 256) return kRows54x4;
    return tiles(6, 4) <= 256 ? kRows64x4 : kRows44x2;
  }
  return tiles(6, 6) <= 256 && tiles(4, 4) > 512 ? kWide66x2 : kWide44x2;
}

int jacobi_block_sweeps(const GridDims &g) {
  const BlockPlan p = block_plan(g);
  return p <= kRows64x4 ? 4 : 2;
}

// Iterates from -> from + jacobi_block_sweeps * launches in the rotating
// buffers jb[q % 3] (a launch's two buffers differ: its sweeps are no multiple
// of 3), 1 <= from (periodic neighbours are images of the interior).
int launch_jacobi_block(picard_ctx *c, int64_t from, int64_t launches) {
  const GridDims &g = c->gd;
  const double dx = g.dxyz[0], dy = g.dxyz[1], dz = g.dxyz[2];
  const double den = 1.0 / ((dx * dy) * (dx * dy) + (dx * dz) * (dx * dz) + (dy * dz) * (dy * dz));
  BlockGeo bg;
  bg.nx = g.nx; bg.ny = g.ny; bg.nz = g.nz;
  bg.X = g.X; bg.XY = (int64_t)g.X * g.Y;
  bg.px = !g.flow[0]; bg.py = !g.flow[1]; bg.pz = !g.flow[2];
  bg.nyt = bg.nzt = 0;
  bg.ax = 0.5 * den * ((dy * dz) * (dy * dz));            // CalcEpotential.f90:44-47
  bg.ay = 0.5 * den * ((dx * dz) * (dx * dz));
  bg.az = 0.5 * den * ((dx * dy) * (dx * dy));
  bg.af = 0.5 * den * ((dx * dy * dz) * (dx * dy * dz));
  const BlockPlan plan = block_plan(g);
  const int T = jacobi_block_sweeps(g);
  for (int64_t q = 0; q < launches; ++q, from += T) {
    const double *in = c->jb[from % 3];
    double *out = c->jb[(from + T) % 3];
    switch (plan) {
      case kRows22x4: launch<1, 4, 2, 2>(c->stream, bg, in, out, c->b); break;
      case kRows33x4: launch<1, 4, 3, 3>(c->stream, bg, in, out, c->b); break;
      case kRows44x4: launch<1, 4, 4, 4>(c->stream, bg, in, out, c->b); break;
      case kRows54x4: launch<1, 4, 5, 4>(c->stream, bg, in, out, c->b); break;
      case kRows64x4: launch<1, 4, 6, 4>(c->stream, bg, in, out, c->b); break;
      case kRows44x2: launch<1, 2, 4, 4>(c->stream, bg, in, out, c->b); break;
      case kWide44x2: launch<2, 2, 4, 4>(c->stream, bg, in, out, c->b); break;
      case kWide66x2: launch<2, 2, 6, 6>(c->stream, bg, in, out, c->b); break;
    }
  }
  PICARD_HIP(hipGetLastError());
  return PICARD_OK;
}

}  // namespace picard
