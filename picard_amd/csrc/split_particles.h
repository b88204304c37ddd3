// split_particles.h -- what the single domain's split form (split.hip) and the ensemble
// (ensemble.hip) share of the particles held as a lower node and an FP32 offset:
// the push, the box tests, the counting pass of the sort and the deposit's loads.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace picard {

constexpr double kFix = 1099511627776.0;       // 2^40
constexpr double kFixInv = 1.0 / 1099511627776.0;

// Carry a coordinate offset into [0, 1): returns the integer carry.
__device__ __forceinline__ int carry(float &f) {
  const float fl = floorf(f);
  f = f - fl;
  int c = (int)fl;
  if (f >= 1.0f) {           // f - floor(f) rounded up to 1
    f = 0.0f;
    c += 1;
  }
  return c;
}

// AdvancePosition in the split form: xi += v dt/dx.
__device__ __forceinline__ void push_one(int (&c)[3], float (&f)[3], const float (&v)[3], float3 dtdx) {
  f[0] = f[0] + v[0] * dtdx.x;
  f[1] = f[1] + v[1] * dtdx.y;
  f[2] = f[2] + v[2] * dtdx.z;
#pragma unroll
  for (int d = 0; d < 3; ++d) c[d] = (int16_t)(c[d] + carry(f[d]));
}

// xi < 1/2 is x < Lmin; xi > n + 1/2 is x > Lmax.
__device__ __forceinline__ bool below(int c, float f) { return c < 0 || (c == 0 && f < 0.5f); }
__device__ __forceinline__ bool above(int c, float f, int n) {
  return c > n || (c == n && f > 0.5f);
}

// counter[k] += 1 for every lane of the wave with k >= 0, one atomic per
// distinct key: the lanes sharing the leader's key (the lowest pending lane)
// take ranks by lane order after the value the leader's add of their count
// returned.  Returns what the lane's own add of 1 would have returned in one
// order of the adds (-1 for k < 0).  Particles arrive nearly sorted by key,
// so a wave holds two or three keys and the adds do not meet on one address
// lane after lane.  Every lane stays in the loop (its condition is the
// wave-uniform mask of pending lanes) and values cross lanes only through
// readlane, which reads the lane whatever the exec mask; the leader's bit
// leaves the mask every pass, so the loop ends within 64 passes.
__device__ __forceinline__ int32_t wave_add1(int32_t *counter, int32_t k) {
  const int lane = (int)(threadIdx.x & 63);
  bool pending = k >= 0;
  int32_t ret = -1;
  uint64_t todo = __ballot(pending);
  while (todo) {
    const int leader = (int)__builtin_ctzll(todo);
    const int32_t kl = __builtin_amdgcn_readlane(k, leader);
    const bool mine = pending && k == kl;
    const uint64_t m = __ballot(mine) | (1ull << leader);
    int32_t base = 0;
    if (lane == leader) base = atomicAdd(&counter[kl], (int32_t)__popcll(m));
    base = __builtin_amdgcn_readlane(base, leader);
    if (mine) {
      ret = base + (int32_t)__popcll(m & ((1ull << lane) - 1ull));
      pending = false;
    }
    todo &= ~m;
  }
  return ret;
}

// Places of a block's keys in a counting sort: hist[k] gains each key's count, r[h] is
// the particle's rank among all of its key (-1 for k[h] < 0).  A block takes PER x
// 256 consecutive particles; they arrive nearly sorted and move a cell or so, so most
// keys lie in a short stretch from the first one's, or in the same stretch a row
// (`row` keys) or a plane (`plane`) before or after.  Those five are counted in LDS
// (the count before is the rank within the block), each key then takes one atomic on
// its histogram entry, whose return places the block's particles of that key.  The
// other keys are added a wave at a time.  With the ranks known the scatter adds
// nothing: at 128^3 with 64 particles a cell (1.4e8) flag and scatter take 0.94 + 3.04 ms,
// where one stretch of 1024 keys took 1.17 + 3.04, and a wave's adds in both passes
// 1.09 + 4.02; the step's push, 1.14 ms as a pass of its own, costs them 0.1.
// The stretch: 512 / 640 / 768 / 1024 keys take 0.92 / 0.94 / 0.96 / 1.08 ms there (more
// to clear, fewer blocks to a CU), 207 / 175 / 162 / 126 us with two particles a cell, whose
// 1024 spread over as many keys (one stretch of 1024: 185).
// PER: four particles a thread, or one where that leaves CUs idle (with one stretch, a
// sort of 6.6e4 particles 37 and 34 us, of 1.0e6 49 both ways, of 1.7e7 355 and 390).
constexpr int kFlagPer = 4;
constexpr int kFlagWin = 640;            // keys of a stretch
constexpr int kFlagBack = 128;           // of them below the first particle's
struct KeyWindow {
  int32_t cnt[5 * kFlagWin];
  int32_t first;
};

// Every thread of a block of 256 takes part, `row` and `plane` are the block's; returns after a barrier.
template <int PER>
__device__ __forceinline__ void count_keys(const int32_t (&k)[PER], int32_t (&r)[PER],
                                           int32_t *__restrict__ hist, KeyWindow &w, int32_t row,
                                           int32_t plane) {
  for (int e = threadIdx.x; e < 5 * kFlagWin; e += 256) w.cnt[e] = 0;
  const uint64_t kept = __ballot(k[0] >= 0);
  if (threadIdx.x < 64) {                // the first wave's first kept particle
    const int32_t kf = kept ? __builtin_amdgcn_readlane(k[0], (int)__builtin_ctzll(kept)) : 0;
    if (threadIdx.x == 0) w.first = kf - kFlagBack;
  }
  __syncthreads();
  const int32_t k0 = w.first;
  const int32_t on[5] = {0, row, -row, plane, -plane};
  int at[PER];                           // the count's place: by the key alone; -1: elsewhere
#pragma unroll
  for (int h = 0; h < PER; ++h) {
    at[h] = -1;
#pragma unroll
    for (int m = 4; m >= 0; --m) {
      const uint32_t d = (uint32_t)k[h] - (uint32_t)k0 - (uint32_t)on[m];
      if (d < (uint32_t)kFlagWin) at[h] = m * kFlagWin + (int)d;
    }
    if (k[h] < 0) at[h] = -1;
    r[h] = -1;
    if (at[h] >= 0) r[h] = atomicAdd(&w.cnt[at[h]], 1);
    const int32_t far = wave_add1(hist, at[h] >= 0 ? -1 : k[h]);
    if (at[h] < 0) r[h] = far;
  }
  __syncthreads();
  // each counted key's place in the histogram, over its count
#pragma unroll
  for (int m = 0; m < 5; ++m)
    for (int e = threadIdx.x; e < kFlagWin; e += 256) {
      const int32_t c = w.cnt[m * kFlagWin + e];
      if (c) w.cnt[m * kFlagWin + e] = atomicAdd(&hist[(uint32_t)k0 + (uint32_t)on[m] + e], c);
    }
  __syncthreads();
#pragma unroll
  for (int h = 0; h < PER; ++h)
    if (at[h] >= 0) r[h] += w.cnt[at[h]];
  __syncthreads();
}

// a[q0 .. q0 + N) (N 4 or 8, q0 a multiple of N, a 16-byte aligned), those from n on as zero
template <int N>
__device__ __forceinline__ void load_chunk(const float *a, int64_t q0, int64_t n, float (&o)[N]) {
  if (q0 + N <= n) {
#pragma unroll
    for (int h = 0; h < N; h += 4)
      *reinterpret_cast<float4 *>(&o[h]) = *reinterpret_cast<const float4 *>(a + q0 + h);
  } else {
#pragma unroll
    for (int h = 0; h < N; ++h) o[h] = q0 + h < n ? a[q0 + h] : 0.0f;
  }
}
template <int N, typename I16>           // int16_t or uint16_t
__device__ __forceinline__ void load_chunk(const I16 *a, int64_t q0, int64_t n, int (&o)[N]) {
  static_assert(sizeof(I16) == 2, "16-bit integers");
  if (q0 + N <= n) {
    int p[N / 2];
    if constexpr (N == 8) {
      const int4 w = *reinterpret_cast<const int4 *>(a + q0);
      p[0] = w.x, p[1] = w.y, p[2] = w.z, p[3] = w.w;
    } else {
      const int2 w = *reinterpret_cast<const int2 *>(a + q0);
      p[0] = w.x, p[1] = w.y;
    }
#pragma unroll
    for (int h = 0; h < N; ++h) o[h] = (I16)(h & 1 ? p[h >> 1] >> 16 : p[h >> 1] & 0xffff);
  } else {
#pragma unroll
    for (int h = 0; h < N; ++h) o[h] = q0 + h < n ? a[q0 + h] : 0;
  }
}
template <int N>
__device__ __forceinline__ void load_chunk(const uint8_t *a, int64_t q0, int64_t n, int (&o)[N]) {
  if (q0 + N <= n) {
    uint32_t p[N / 4];
    if constexpr (N == 8) {
      const uint2 w = *reinterpret_cast<const uint2 *>(a + q0);
      p[0] = w.x, p[1] = w.y;
    } else {
      p[0] = *reinterpret_cast<const uint32_t *>(a + q0);
    }
#pragma unroll
    for (int h = 0; h < N; ++h) o[h] = (int)(p[h >> 2] >> (8 * (h & 3)) & 0xffu);
  } else {
#pragma unroll
    for (int h = 0; h < N; ++h) o[h] = q0 + h < n ? a[q0 + h] : 0;
  }
}

// (unsigned long long)(w 2^40) for a weight, 0 <= w <= 1 (NaN: 0): below 2^52 the
// integer is in the low mantissa bits of trunc + 2^52, two adds in place of the
// conversion's seven operations.
__device__ __forceinline__ unsigned long long weight_units(float w) {
  const float w1 = fminf(fmaxf(w, 0.0f), 1.0f);
  const double v = __builtin_trunc(double(w1) * kFix) + 4503599627370496.0;
  return (unsigned long long)__double_as_longlong(v) - 0x4330000000000000ull;
}

}  // namespace picard
