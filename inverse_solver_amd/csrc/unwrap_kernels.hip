// Phase unwrapping on the device: the residue map of 2x2 loops and the raster
// integration of wrapped differences with 2 pi step maps, in single precision
// as the reference's goldstein_GPU kernels compute them
// (Codes/sub_code/goldstein_GPU/get_residue_cuda.cu:35-66,
//  unwrapp_phase_goldstein_cuda.cu:60-113).  Arrays are column-major
// (n1 fastest, then n2, then the angle index n3).
#include <hip/hip_runtime.h>
#include <cstdint>

#include "goldstein.hpp"
#include "unwrap_kernels.hpp"

namespace cbs {

constexpr float kPiF = 3.141592654f;
constexpr float kTwoPiF = 2.0f * kPiF;

// fmodf(fmodf(a, b) + b, b) for b = 2 pi, bit for bit, without fmodf's loop.
// fmodf(a, b): with q = trunc(|a| / b) from the rounded product with 1 / b, |a| - q b is one fused
// multiply-add.  q is off by one only where |a| / b is within 2^-10 of a whole number (|a| / b < 4096),
// so the difference lies in (-0.01, b + 0.01), below 8, and is a whole multiple of 2^-21, the last
// place of b (of |a| where that is below 4, and then q = 0): it is exact, and so is the correction by b.
// The second fmodf has an argument in [0, 2 b]: up to two exact subtractions.
// NaN, infinities and larger arguments take fmodf.
__device__ __forceinline__ float wrap_two_pi(float a) {
  constexpr float b = kTwoPiF;
  const float m = fabsf(a);
  if (!(m < 4096.0f * b)) return fmodf(fmodf(a, b) + b, b);
  float r = fmaf(-truncf(m * (1.0f / b)), b, m);
  r = r < 0.0f ? r + b : r;
  r = r >= b ? r - b : r;
  float x = copysignf(r, a) + b;
  x = x >= b ? x - b : x;
  return x >= b ? x - b : x;
}

// residue[d1, d2, z] over the (n1 - 1) x (n2 - 1) loops of each angle
__global__ void phase_residues(const float* __restrict__ p, float* __restrict__ out, int n1, int n2, int n3) {
  const long long m1 = n1 - 1, m2 = n2 - 1;
  const long long total = m1 * m2 * n3;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (long long)gridDim.x * blockDim.x) {
    const long long d12 = i % (m1 * m2);
    const int z = (int)(i / (m1 * m2));
    const int d2 = (int)(d12 / m1), d1 = (int)(d12 % m1);
    const long long b = (long long)z * n1 * n2;
    const float v11 = p[b + (long long)d2 * n1 + d1];
    const float v21 = p[b + (long long)d2 * n1 + d1 + 1];
    const float v12 = p[b + (long long)(d2 + 1) * n1 + d1];
    const float v22 = p[b + (long long)(d2 + 1) * n1 + d1 + 1];
    const float a = wrap_two_pi(v11 - v12 + kPiF);   // along n2 at row d1
    const float c = wrap_two_pi(v21 - v22 + kPiF);   // along n2 at row d1 + 1
    const float e = wrap_two_pi(v11 - v21 + kPiF);   // along n1 at column d2
    const float f = wrap_two_pi(v12 - v22 + kPiF);   // along n1 at column d2 + 1
    out[i] = roundf((a + f - c - e) / kTwoPiF);
  }
}

// The reference's update last + d - step * 2 * pi is one fused multiply-add under nvcc's
// default contraction (--fmad=true); it is written as fmaf here so that the rounding does
// not depend on the compiler's choice.

// One step of the integration: the wrapped difference of cur to the unwrapped last value.
__device__ __forceinline__ float unwrap_step(float cur, float last, float step) {
  const float d = wrap_two_pi(cur - last + kPiF) - kPiF;
  return fmaf(-step, kTwoPiF, last + d);
}

// The integration is a chain of dependent steps down a line, so its time is the steps' latency:
// the lines are staged through LDS (a step that waited for its own strided load took 0.54 us,
// with fmodf's loop a good part of it), one lane walks each, and eight steps' values are read
// ahead of their chain (one at a time: 19 us).  24 maps of 96^2: column 53 -> 15 us, rows 51 -> 14 us.
__device__ __forceinline__ float unwrap_line(float* p, const float* st, int cnt, float last) {
  int i = 0;
  for (; i + 8 <= cnt; i += 8) {
    float v[8], s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { v[j] = p[i + j]; s[j] = st[i + j]; }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      last = unwrap_step(v[j], last, s[j]);
      p[i + j] = last;
    }
  }
  for (; i < cnt; ++i) {
    last = unwrap_step(p[i], last, st[i]);
    p[i] = last;
  }
  return last;
}

// first column (d1 = 0) of every angle, integrated along n2; one wave an angle
__global__ __launch_bounds__(64) void phase_integrate_column(float* __restrict__ p, const int32_t* __restrict__ step2,
                                                             int n1, int n2, int n3) {
  constexpr int C = 512;
  __shared__ float s_p[C], s_s[C];
  const int z = blockIdx.x;
  float* __restrict__ col = p + (long long)z * n1 * n2;
  const int32_t* __restrict__ st = step2 + (long long)z * n2;
  float last = col[0];
  for (int c0 = 1; c0 < n2; c0 += C) {
    const int cnt = min(C, n2 - c0);
    for (int i = threadIdx.x; i < cnt; i += 64) {
      s_p[i] = col[(long long)(c0 + i) * n1];
      s_s[i] = (float)st[c0 + i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      last = unwrap_line(s_p, s_s, cnt, last);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < cnt; i += 64) col[(long long)(c0 + i) * n1] = s_p[i];
    __syncthreads();
  }
}

// every row (fixed d2, angle), integrated along n1 from its already unwrapped first element: 16
// rows a wave (a lane each), 64 columns at a time, the next columns requested meanwhile
__global__ __launch_bounds__(64) void phase_integrate_rows(float* __restrict__ p, const int32_t* __restrict__ step1,
                                                           int n1, int n2, int n3) {
  constexpr int R = 16, C = 64, PC = C + 1;
  __shared__ float s_p[R * PC], s_s[R * PC];
  const int lane = threadIdx.x;
  const long long rows = (long long)n2 * n3, r0 = (long long)blockIdx.x * R;
  const int nr = rows - r0 < R ? (int)(rows - r0) : R;
  float* __restrict__ base = p + r0 * n1;
  const int32_t* __restrict__ sb = step1 + r0 * n1;
  float last = lane < nr ? base[(long long)lane * n1] : 0.0f;
  float vp[R];
  int32_t vs[R];
  auto request = [&](int c0) {
    const int c = min(c0 + lane, n1 - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const long long i = (long long)min(r, nr - 1) * n1 + c;
      vp[r] = base[i];
      vs[r] = sb[i];
    }
  };
  if (n1 > 1) request(1);
  for (int c0 = 1; c0 < n1; c0 += C) {
    const int cnt = min(C, n1 - c0);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      s_p[r * PC + lane] = vp[r];
      s_s[r * PC + lane] = (float)vs[r];
    }
    __syncthreads();
    if (c0 + C < n1) request(c0 + C);
    if (lane < nr) {
      last = unwrap_line(s_p + lane * PC, s_s + lane * PC, cnt, last);
    }
    __syncthreads();
    if (lane < cnt)
      for (int r = 0; r < nr; ++r) base[(long long)r * n1 + c0 + lane] = s_p[r * PC + lane];
    __syncthreads();
  }
}

// Step maps and the residue count (list[0]) cleared before a placement.
__global__ void phase_clear(int32_t* __restrict__ step1, long long n1, int32_t* __restrict__ step2, long long n2,
                            PhaseResidue* __restrict__ list) {
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n1 + n2; i += (long long)gridDim.x * blockDim.x) {
    if (i < n1) step1[i] = 0;
    else step2[i - n1] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) list[0] = PhaseResidue{0, 0.0f};
}

// The non-zero residues as (flat index, value) pairs from list[1] on, in no order, the first cap of
// them; list[0].index counts them all.  One atomic a wave.
__global__ void phase_collect(const float* __restrict__ res, long long m, PhaseResidue* __restrict__ list, int cap) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const float v = i < m ? res[i] : 0.0f;
  const bool hit = v != 0.0f;
  const unsigned long long hits = __ballot(hit);
  if (!hits) return;
  const int lane = threadIdx.x & 63;
  const int first = __ffsll((unsigned long long)hits) - 1;
  int at = 0;
  if (lane == first) at = atomicAdd(&list[0].index, __popcll(hits));
  at = __shfl(at, first, 64);
  at += __popcll(hits & ((1ull << lane) - 1));
  if (hit && at < cap) list[1 + at] = PhaseResidue{(int32_t)i, v};
}

// remove_dipoles_cuda.cu:50-106, one launch per direction (0..3 = d1 - 1, d2 - 1, d1 + 1,
// d2 + 1), a thread an element: the positive residues act (one that is cancelled is zero in the
// later directions).  Within one direction every negative neighbour belongs to one positive
// residue, so no element is touched by two threads; an element another thread writes is negative
// before and not positive after.  A dipole along d2 writes +-1 (directions 1 / 3) into step1 at
// (d1 + 1, min(d2, d2') + 1).
__global__ void phase_dipoles(float* __restrict__ res, int32_t* __restrict__ step1, int m1, int m2, int n3,
                              int direction) {
  const long long rid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (rid >= (long long)m1 * m2 * n3 || !(res[rid] > 0.0f)) return;
  const long long plane = (long long)m1 * m2;
  const int z = (int)(rid / plane);
  const int d12 = (int)(rid % plane);
  const int d2 = d12 / m1, d1 = d12 % m1;
  const int p1 = d1 - (direction == 0 ? 1 : 0) + (direction == 2 ? 1 : 0);
  const int p2 = d2 - (direction == 1 ? 1 : 0) + (direction == 3 ? 1 : 0);
  if (p1 < 0 || p2 < 0 || p1 >= m1 || p2 >= m2) return;
  const long long pid = (long long)z * plane + (long long)p2 * m1 + p1;
  float pv = res[pid];
  if (!(pv < 0.0f)) return;
  float v = res[rid];
  const float rem = fminf(v, -pv);
  v = roundf(v - rem);
  pv = roundf(pv + rem);
  res[rid] = v;
  res[pid] = pv;
  if (direction == 1 || direction == 3) {
    const long long n1 = m1 + 1, n2 = m2 + 1;
    const long long c1 = p1 + 1, c2 = min(d2, p2) + 1;
    step1[(long long)z * n1 * n2 + c2 * n1 + c1] = (int32_t)rintf(direction == 1 ? rem : -rem);
  }
}

// get_shortest_sort_cuda.cu:64-87: the gs::kNearest nearest residues of every listed
// residue, out[(i * kNearest + k) * 2 + {0, 1}] = {id, distance}.
__global__ void phase_nearest(const int32_t* __restrict__ rows, int n, const int32_t* __restrict__ table,
                              int table_size, const int32_t* __restrict__ zstart, const int32_t* __restrict__ square,
                              int s1, int s2, int32_t* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int cur[2 * gs::kNearest];
  gs::nearest<gs::kNearest>(nullptr, rows, n, table, table_size, zstart, square, s1, s2, i, cur);
  for (int k = 0; k < 2 * gs::kNearest; ++k) out[(long long)i * 2 * gs::kNearest + k] = cur[k];
}

// raster_branches_cuda.cu:65-135: add each branch's jump to the step maps.  A branch to
// the border (p1 = -1) ends at the nearer border of the (n1, n2) map; on the d1 = -1
// side it adds to step2 of column p2 d2 + 1.  Otherwise each row path between the two
// ends is crossed at d1 = p2 d1 + trunc(i / steps * (p1 d1 - p2 d1)) + 1, taken as a flat
// index of step1 (so a crossing one past the last row wraps to the next column, as there);
// a flat index outside the map is dropped.
__global__ void phase_raster(const int32_t* __restrict__ br, int nb, int32_t* __restrict__ step1,
                             int32_t* __restrict__ step2, int n1, int n2, int n3) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nb) return;
  const int32_t* r = br + 6 * (long long)b;
  int p1x = r[0], p1y = r[1], p2x = r[2], p2y = r[3];
  const int z = r[4];
  int jump = r[5];
  if (p1x == -1) {
    const bool xs = p2x < n1 - p2x;
    const bool ys = p2y < n2 - p2y;
    const int mdx = xs ? p2x : n1 - p2x;
    const int mdy = ys ? p2y : n2 - p2y;
    p1x = mdx > mdy ? p2x : (xs ? -1 : n1 - 1);
    p1y = mdx < mdy ? p2y : (ys ? -1 : n2 - 1);
    if (p1x == -1) {
      const long long k = (long long)n2 * z + p2y + 1;
      if (k >= 0 && k < (long long)n2 * n3) atomicAdd(&step2[k], jump);
      return;
    }
  }
  if (p1y == p2y) return;
  if (p2y > p1y) {
    int t = p1y;
    p1y = p2y;
    p2y = t;
    t = p1x;
    p1x = p2x;
    p2x = t;
    jump = -jump;
  }
  const int steps = p1y - p2y;
  const long long total = (long long)n1 * n2 * n3;
  const float dxf = (float)(p1x - p2x);
  for (int i = 0; i < steps; ++i) {
    const int cy = p2y + i + 1;
    const float frac = (float)((double)i / (double)steps);   // the single-precision quotient
    const int cx = p2x + (int)(frac * dxf) + 1;
    const long long k = (long long)n1 * n2 * z + (long long)n1 * cy + cx;
    if (k >= 0 && k < total) atomicAdd(&step1[k], jump);
  }
}

}  // namespace cbs

