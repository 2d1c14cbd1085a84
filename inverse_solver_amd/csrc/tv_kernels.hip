// Isotropic 3D TV proximal step (FISTA on the dual) on the device, FP32, for a
// real potential (kappamax = 0) or a complex one.
// Codes/sub_code/TV_FISTA_inner_v2.m:1-123 for 3D input:
//   y   = project(in - lam * div(R))                   (:38, project_non_neg + TV_L)
//   P'  = R + grad(y) / (12 lam);  P' /= max(|P'|, 1)  (:38-42, TV_L_trans, project_TV)
//   R   = P' + (t - 1)/t' (P' - P)                     (:44-47)
//   out = project(in - lam * div(P))                   (:51)
// with periodic forward differences grad_k(y) = y - y(+e_k) and
// div(P) = sum_k P_k - P_k(-e_k).  |P'| is the isotropic norm over the three
// components, each |.|^2 of a complex value for complex input (project_TV :79-91).
// project (project_non_neg :57-75): with non_neg, real part clamped to [vmin, vmax];
// for complex input a negative imaginary part is set to 0 and, when vimag_max > 0,
// the imaginary part is capped at vimag_max; dirichlet zeroes the six faces.
#include <algorithm>

#include "fft_core.hpp"
#include "tv_kernels.hpp"

namespace cbs {

#define GRID_STRIDE_TV(i, total) \
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < (total); i += (long long)gridDim.x * blockDim.x)

__device__ __forceinline__ float tv_abs2(float v) { return v * v; }
__device__ __forceinline__ float tv_abs2(float2 v) { return v.x * v.x + v.y * v.y; }
__device__ __forceinline__ float2 operator+(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 operator-(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 operator*(float s, float2 a) { return make_float2(s * a.x, s * a.y); }
__device__ __forceinline__ float2 operator/(float2 a, float s) { return make_float2(a.x / s, a.y / s); }
__device__ __forceinline__ void tv_zero_val(float& v) { v = 0.f; }
__device__ __forceinline__ void tv_zero_val(float2& v) { v = make_float2(0.f, 0.f); }

__device__ __forceinline__ float tv_bounds(float v, const TvArgs& a) {
  if (a.non_neg) v = fminf(fmaxf(v, a.vmin), a.vmax);
  return v;
}
__device__ __forceinline__ float2 tv_bounds(float2 v, const TvArgs& a) {
  if (a.non_neg) v.x = fminf(fmaxf(v.x, a.vmin), a.vmax);
  if (v.y < 0.f) v.y = 0.f;
  if (a.vimag_max > 0.f && v.y > a.vimag_max) v.y = a.vimag_max;
  return v;
}

template <class T>
__device__ __forceinline__ void tv_div_project_body(const T* __restrict__ in, const T* __restrict__ Q,
                                                    T* __restrict__ y, const TvArgs& a) {
  const long long n = (long long)a.nx * a.ny * a.nz;
  GRID_STRIDE_TV(i, n) {
    const int x = (int)(i % a.nx);
    const long long yz = i / a.nx;
    const int yy = (int)(yz % a.ny), z = (int)(yz / a.ny);
    const long long ix = x == 0 ? i + (a.nx - 1) : i - 1;
    const long long iy = yy == 0 ? i + (long long)(a.ny - 1) * a.nx : i - a.nx;
    const long long iz = z == 0 ? i + (long long)(a.nz - 1) * a.nx * a.ny : i - (long long)a.nx * a.ny;
    const T div = ((Q[i] + Q[n + i]) + Q[2 * n + i]) - Q[ix] - Q[n + iy] - Q[2 * n + iz];
    T v = tv_bounds(in[i] - a.lam * div, a);
    if (a.dirichlet && (x == 0 || yy == 0 || z == 0 || x == a.nx - 1 || yy == a.ny - 1 || z == a.nz - 1))
      tv_zero_val(v);
    y[i] = v;
  }
}

// One inner iteration in one launch.  The dual iterates are kept as P_k alone: with
// R = P_k + theta (P_k - P_{k-1}) formed on the fly (the expression, and so the rounding,
// that a stored R would hold), the iteration reads P_k, P_{k-1} and in and writes P_{k+1},
// 10 values a voxel, where separate kernels for y and the dual update moved 18 (R read
// twice and written, y written and read).
//
// A block takes a tile of (x, y) columns, 62 x 6 or another shape of its 512 threads on grids that one covers
// with fewer blocks (tv_columns), one thread a column and one more each side, and ZC = 3 planes of z.  It
// requests every operand of its planes before the first is used
// (with one plane requested ahead of the other the launch waited for memory once a plane), then
// walks up z: the R_x and R_y of the lower neighbours and then the y of the upper ones pass
// through LDS; R_z and y of the plane below stay in registers.
// The buffers of a reconstruction grid fit the 256 MB Infinity Cache, which bounds the launch.
// Neighbouring tiles write parts of the same 128-byte lines, so the blocks are numbered with a
// contiguous run for every XCD (xcd_position): with neighbours on different XCDs an iteration
// took 19.1 us instead of 10.9 (real, 96 x 96 x 97, 30 x 14 tiles) and 38 instead of 29
// (complex, 161 x 161 x 61).  Per iteration, launch gaps included: real 14.3 -> 10.2 us, complex
// 46 -> 26.6 us (126 MB of the 10 values: 4.7 TB/s; 18 values at 5.0 TB/s before).  Other tiles
// and plane counts (32 x 16, 32 x 8, 64 x 4; 2 to 6 planes) are within 5 %, 8 planes 25 % slower.
// FIRST: P_k = P_{k-1} = 0 (no buffer is read, so none has to be cleared).
// Off: type of a byte offset inside one z plane (32 bits but for planes of 4 GiB and more); the
// plane's base is uniform, so every access is a scalar base and this offset.
constexpr int kTvT = 512;       // threads: 2^lg columns in x, the rest in y

// 1 / sqrt(s) for s >= 1: the hardware's (1 ulp) and one Newton step; infinity gives 0 and NaN NaN.
__device__ __forceinline__ float tv_rsqrt(float s) {
  const float r = __builtin_amdgcn_rsqf(s);
  const float e = fmaf(-s * r, r, 1.0f);
  return s < 3.0e38f ? fmaf(0.5f * r, e, r) : r;
}

// LG: 2^LG threads in x; 0: lg_ at run time (the shifts cost 2 to 12 % of a launch, so the usual shape is compiled).
template <class T, int ZC, bool FIRST, class Off, int LG>
__global__ __launch_bounds__(kTvT) void tv_inner(const T* __restrict__ in, const T* __restrict__ Pc,
                                                 const T* __restrict__ Pp, T* __restrict__ Pn, TvArgs a,
                                                 float theta, int lg_) {
  __shared__ T sx[kTvT], sz[kTvT], sy[kTvT];   // R_x, R_y and y of a plane
  const int lg = LG > 0 ? LG : lg_, nt = 1 << lg, mt = kTvT >> lg;
  const int tx = threadIdx.x, ty = threadIdx.y, me = ty * nt + tx;
  const unsigned gx = (a.nx + nt - 3) / (nt - 2), gy = (a.ny + mt - 3) / (mt - 2);
  const unsigned pos = xcd_position(blockIdx.x, gridDim.x), bx = pos % gx, byz = pos / gx;
  const int x = (int)bx * (nt - 2) + tx - 1, y = (int)(byz % gy) * (mt - 2) + ty - 1;
  const int z0 = (int)(byz / gy) * ZC, z1 = min(z0 + ZC, a.nz);
  const bool mine = tx > 0 && tx < nt - 1 && ty > 0 && ty < mt - 1 && x < a.nx && y < a.ny;
  // periodic column of this thread (columns past the upper neighbour of the last one are not
  // used: they take the last column)
  const int xw = x < 0 ? a.nx - 1 : x < a.nx ? x : x == a.nx ? 0 : a.nx - 1;
  const int yw = y < 0 ? a.ny - 1 : y < a.ny ? y : y == a.ny ? 0 : a.ny - 1;
  const Off col = ((Off)yw * (Off)a.nx + (Off)xw) * (Off)sizeof(T);
  const long long nxy = (long long)a.nx * a.ny, n = nxy * a.nz;
  const int lx = me - (tx > 0), ly = ty > 0 ? me - nt : me;                    // lower neighbours
  const int ux = me + (tx < nt - 1), uy = ty < mt - 1 ? me + nt : me;          // upper neighbours
  const float c = 1.0f / (12.0f * a.lam);
  const bool edge = a.dirichlet && (xw == 0 || yw == 0 || xw == a.nx - 1 || yw == a.ny - 1);
  auto ld = [&](const T* plane) { return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(plane) + col); };
  auto st = [&](T* plane, T v) { *reinterpret_cast<T*>(reinterpret_cast<char*>(plane) + col) = v; };
  auto momentum = [&](T p, T o) { return p + theta * (p - o); };

  // the operands of planes z0 .. z1 (plane nz is plane 0), all requested here
  T vi[ZC + 1], p[ZC + 1][3], o[ZC + 1][3];
#pragma unroll
  for (int q = 0; q <= ZC; ++q) {
    if (z0 + q > z1) break;
    const long long i = (z0 + q < a.nz ? (long long)(z0 + q) : 0) * nxy;
    if constexpr (!FIRST) {
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        p[q][k] = ld(Pc + k * n + i);
        o[q][k] = ld(Pp + k * n + i);
      }
    }
    vi[q] = ld(in + i);
  }
  T rz_below{};                 // R_z one plane down
  if constexpr (!FIRST) {
    const long long i = 2 * n + (long long)(z0 > 0 ? z0 - 1 : a.nz - 1) * nxy;
    rz_below = momentum(ld(Pc + i), ld(Pp + i));
  }
  T q0{}, q1{}, q2{}, y_below{};   // plane below: R_x + c grad_x, R_y + c grad_y, R_z and y
#pragma unroll
  for (int q = 0; q <= ZC; ++q) {
    const int z = z0 + q;
    if (z > z1) break;
    T v = vi[q];
    T r0{}, r1{}, r2{};
    if constexpr (!FIRST) {
      r0 = momentum(p[q][0], o[q][0]);
      r1 = momentum(p[q][1], o[q][1]);
      r2 = momentum(p[q][2], o[q][2]);
      sx[me] = r0;
      sz[me] = r1;
    }
    if constexpr (!FIRST) {
      lds_barrier();
      const T div = ((r0 + r1) + r2) - sx[lx] - sz[ly] - rz_below;
      v = v - a.lam * div;
    }
    v = tv_bounds(v, a);
    const int zw = z < a.nz ? z : 0;
    if (edge || (a.dirichlet && (zw == 0 || zw == a.nz - 1))) tv_zero_val(v);
    sy[me] = v;
    lds_barrier();
    if (q > 0 && mine) {        // the plane below has all it needs
      const T p2 = q2 + c * (y_below - v);
      const float inv = tv_rsqrt(fmaxf(tv_abs2(q0) + tv_abs2(q1) + tv_abs2(p2), 1.0f));
      const long long i = (long long)(z - 1) * nxy;
      st(Pn + i, inv * q0);
      st(Pn + n + i, inv * q1);
      st(Pn + 2 * n + i, inv * p2);
    }
    q0 = r0 + c * (v - sy[ux]);
    q1 = r1 + c * (v - sy[uy]);
    q2 = rz_below = r2;
    y_below = v;
    if constexpr (FIRST) lds_barrier();   // sy is written again before the next barrier
  }
}

// Two inner iterations in one launch: reads P_k, P_{k-1} and in, writes P1 = P_{k+1} and P2 = P_{k+2},
// 13 values a voxel where two launches of tv_inner move 20, with one start and drain of the chip for two.
//
// P_{k+2} of a voxel needs P_{k+1} of its neighbours and that their y, so a block of TX x TY threads, a
// thread a column, holds two more columns on each side than it writes and walks up z through its planes,
// two planes more below and two steps more above.  In the step that takes plane a, the first iteration's y
// of plane a and the second one's y of plane b = a - 2 share the LDS passes and their two barriers; P1 of
// plane a - 1 and P2 of plane b - 1 leave it.  Every value is the expression of tv_inner.
// theta: the momentum between P_k and P_{k-1}; theta1: between P1 and P_k.
// A step is bound by the latency of its barriers and of the operands, requested D planes ahead: two for real
// input (78 registers, two blocks a CU), one for complex (105, one block a CU; two ahead: 18.6 for 18.0 us).
// An iteration, us: real 96 x 96 x 97 10.4 (tv_inner) -> 8.6, 200 x 190 x 110 35.5 -> 24.6; complex
// 161 x 161 x 61 26.7 -> 18.0, 200 x 190 x 110 85.5 -> 55.7, 100 x 110 x 100 20.9 -> 14.6.  With 1024 and
// 512 threads the 161 x 161 x 61 and 200 x 190 x 110 complex take 19.9 and 19.7, 59.5 and 61.9.
constexpr int kTvT2 = 768;
template <class T, class Off>
__global__ __launch_bounds__(kTvT2) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 3)))
void tv_inner2(const T* __restrict__ in, const T* __restrict__ Pc,
                                                   const T* __restrict__ Pp, T* __restrict__ P1, T* __restrict__ P2,
                                                   TvArgs a, TvTiles g, float theta, float theta1) {
  __shared__ T sx[kTvT2], sz[kTvT2], sy[kTvT2];   // R_x, R_y and y of the first iteration, plane a
  __shared__ T tx1[kTvT2], tz1[kTvT2], ty1[kTvT2];   // the same of the second, plane b
  const int me = threadIdx.x, tx = me % g.tx, ty = me / g.tx;
  const unsigned pos = xcd_position(blockIdx.x, gridDim.x), bx = pos % g.gx, byz = pos / g.gx;
  const int x = (int)bx * (g.tx - 4) + tx - 2, y = (int)(byz % g.gy) * (g.ty - 4) + ty - 2;
  const int z0 = (int)(byz / g.gy) * g.zc, z1 = min(z0 + g.zc, a.nz);
  const bool mine = tx >= 2 && tx < g.tx - 2 && ty >= 2 && ty < g.ty - 2 && x < a.nx && y < a.ny;
  auto wrap = [](int i, int n) {
    i %= n;
    return i < 0 ? i + n : i;
  };
  const int xw = wrap(x, a.nx), yw = wrap(y, a.ny);
  const Off col = ((Off)yw * (Off)a.nx + (Off)xw) * (Off)sizeof(T);
  const long long nxy = (long long)a.nx * a.ny, n = nxy * a.nz;
  const int lx = me - (tx > 0), ly = ty > 0 ? me - g.tx : me;                          // lower neighbours
  const int ux = me + (tx < g.tx - 1), uy = ty < g.ty - 1 ? me + g.tx : me;            // upper neighbours
  const float c = 1.0f / (12.0f * a.lam);
  const bool edge = a.dirichlet && (xw == 0 || yw == 0 || xw == a.nx - 1 || yw == a.ny - 1);
  auto ld = [&](const T* plane) { return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(plane) + col); };
  auto st = [&](T* plane, T v) { *reinterpret_cast<T*>(reinterpret_cast<char*>(plane) + col) = v; };
  auto on_face = [&](int zw) { return edge || (a.dirichlet && (zw == 0 || zw == a.nz - 1)); };

  int za = wrap(z0 - 2, a.nz), za1 = 0, zb = 0;    // planes a, a - 1 and b, wrapped
  T p[3], o[3], vi;                                // P_k, P_{k-1} and in of plane a
  T pn[3]{}, on[3]{}, vn{};                        // and of plane a + 1
  constexpr int D = sizeof(T) == 4 ? 2 : 1;
  int zn = za + 1 < a.nz ? za + 1 : 0;
  auto request = [&](int z, T (&pz)[3], T (&oz)[3], T& vz) {
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      pz[k] = ld(Pc + k * n + z * nxy);
      oz[k] = ld(Pp + k * n + z * nxy);
    }
    vz = ld(in + z * nxy);
  };
  request(za, p, o, vi);
  if constexpr (D == 2) request(zn, pn, on, vn);
  T pk[3]{}, vi_a1{}, vi_b{};                      // P_k and in of plane a - 1, in of plane b
  T q0{}, q1{}, rz{}, y_a1{};                      // plane a - 1: R_x + c grad_x, R_y + c grad_y, R_z and y
  T t[3]{}, u0{}, u1{}, tz{}, y_b1{};              // R of the second iteration, plane b; as above, plane b - 1
  const int last = z1 - z0 + 4;
  for (int s = 0; s <= last; ++s) {
    // the first iteration is through a step before the last, the second one starts at s = 3
    const bool one = s < last, two = s >= 3;
    const int zm = zn + 1 < a.nz ? zn + 1 : 0;     // plane a + 2
    T pm[3]{}, om[3]{}, vm{}, r[3]{}, v{}, w{};
    if constexpr (D == 2) {
      if (s + 2 < last) request(zm, pm, om, vm);
    } else {
      if (s + 1 < last) request(zn, pn, on, vn);
    }
    if (one) {
#pragma unroll
      for (int k = 0; k < 3; ++k) r[k] = p[k] + theta * (p[k] - o[k]);
      sx[me] = r[0];
      sz[me] = r[1];
    }
    if (two) {
      tx1[me] = t[0];
      tz1[me] = t[1];
    }
    lds_barrier();
    if (one) {
      v = tv_bounds(vi - a.lam * (((r[0] + r[1]) + r[2]) - sx[lx] - sz[ly] - rz), a);
      if (on_face(za)) tv_zero_val(v);
      sy[me] = v;
    }
    if (two) {
      w = tv_bounds(vi_b - a.lam * (((t[0] + t[1]) + t[2]) - tx1[lx] - tz1[ly] - tz), a);
      if (on_face(zb)) tv_zero_val(w);
      ty1[me] = w;
    }
    lds_barrier();
    const int a1 = z0 - 3 + s, b1 = z0 - 5 + s;    // planes a - 1 and b - 1
    if (two) {
      if (mine && b1 >= z0) {
        const T m2 = tz + c * (y_b1 - w);
        const float inv1 = tv_rsqrt(fmaxf(tv_abs2(u0) + tv_abs2(u1) + tv_abs2(m2), 1.0f));
        st(P2 + b1 * nxy, inv1 * u0);
        st(P2 + n + b1 * nxy, inv1 * u1);
        st(P2 + 2 * n + b1 * nxy, inv1 * m2);
      }
      u0 = t[0] + c * (w - ty1[ux]);
      u1 = t[1] + c * (w - ty1[uy]);
      tz = t[2];
      y_b1 = w;
    }
    if (one) {
      if (s >= 2) {
        const T p2 = rz + c * (y_a1 - v);
        const float inv = tv_rsqrt(fmaxf(tv_abs2(q0) + tv_abs2(q1) + tv_abs2(p2), 1.0f));
        const T n0 = inv * q0, n1 = inv * q1, n2 = inv * p2;
        if (mine && a1 >= z0 && a1 < z1) {
          st(P1 + a1 * nxy, n0);
          st(P1 + n + a1 * nxy, n1);
          st(P1 + 2 * n + a1 * nxy, n2);
        }
        t[0] = n0 + theta1 * (n0 - pk[0]);
        t[1] = n1 + theta1 * (n1 - pk[1]);
        t[2] = n2 + theta1 * (n2 - pk[2]);
      }
      q0 = r[0] + c * (v - sy[ux]);
      q1 = r[1] + c * (v - sy[uy]);
      rz = r[2];
      y_a1 = v;
    }
    vi_b = vi_a1;
    vi_a1 = vi;
    vi = vn;
    if constexpr (D == 2) vn = vm;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      pk[k] = p[k];
      p[k] = pn[k];
      o[k] = on[k];
      if constexpr (D == 2) {
        pn[k] = pm[k];
        on[k] = om[k];
      }
    }
    zb = za1;
    za1 = za;
    za = zn;
    zn = zm;
  }
}

__global__ void tv_div_project(const float* __restrict__ in, const float* __restrict__ Q, float* __restrict__ y,
                               TvArgs a) {
  tv_div_project_body(in, Q, y, a);
}
__global__ void tv_div_project_c(const float2* __restrict__ in, const float2* __restrict__ Q, float2* __restrict__ y,
                                 TvArgs a) {
  tv_div_project_body(in, Q, y, a);
}

// Columns of a tv_inner block and the blocks of one layer: 64 x 8 threads, or the shape that needs the fewest blocks
// where that is a third less, counting what short rows cost in memory access (an iteration of 26 x 148 x 44 6.4 -> 5.4
// us real, 8.4 -> 6.1 complex; 1 x 500 x 500 59 -> 7 us; but 64 x 64 x 65 real with 32 threads in x, 15 for 22 blocks,
// 5.9 -> 6.4, and 83 x 62 x 45 with 8 6.0 -> 7.4).
struct TvColumns {
  int lg;                   // 2^lg threads in x
  unsigned gx, gy;
};
static TvColumns tv_columns(const TvArgs& a) {
  auto of = [&](int lg) {
    const unsigned nt = 1u << lg, mt = (unsigned)kTvT >> lg;
    return TvColumns{lg, (a.nx + nt - 3) / (nt - 2), (a.ny + mt - 3) / (mt - 2)};
  };
  auto cost = [](const TvColumns& c) {
    const double row[] = {0, 0, 2.0, 1.5, 1.15, 1.0, 1.0, 1.0};
    return (double)c.gx * c.gy * row[c.lg];
  };
  TvColumns best = of(6);
  const double limit = 0.65 * cost(best);
  for (int lg : {7, 5, 4, 3, 2}) {
    const TvColumns c = of(lg);
    if (cost(c) <= limit && cost(c) < cost(best)) best = c;
  }
  return best;
}
constexpr int kTvZ = 3;

template <class T, class Off>
static void launch_inner(hipStream_t st, const T* in, const T* Pc, const T* Pp, T* Pn, const TvArgs& a, float theta,
                         bool first) {
  const TvColumns c = tv_columns(a);
  const dim3 grid(c.gx * c.gy * (unsigned)((a.nz + kTvZ - 1) / kTvZ)), block(1u << c.lg, (unsigned)kTvT >> c.lg);
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, 0, st, in, Pc, Pp, Pn, a, theta, c.lg); };
  if (c.lg == 6 && first) launch(tv_inner<T, kTvZ, true, Off, 6>);
  else if (c.lg == 6) launch(tv_inner<T, kTvZ, false, Off, 6>);
  else if (first) launch(tv_inner<T, kTvZ, true, Off, 0>);
  else launch(tv_inner<T, kTvZ, false, Off, 0>);
}
template <class T>
static void launch_inner(hipStream_t st, const T* in, const T* Pc, const T* Pp, T* Pn, const TvArgs& a, float theta,
                         bool first) {
  if ((unsigned long long)a.nx * a.ny * sizeof(T) < (1ull << 32))
    launch_inner<T, unsigned>(st, in, Pc, Pp, Pn, a, theta, first);
  else
    launch_inner<T, unsigned long long>(st, in, Pc, Pp, Pn, a, theta, first);
}
void tv_inner_real(hipStream_t st, const float* in, const float* Pc, const float* Pp, float* Pn, const TvArgs& a,
                   float theta, bool first) {
  launch_inner<float>(st, in, Pc, Pp, Pn, a, theta, first);
}
void tv_inner_complex(hipStream_t st, const float2* in, const float2* Pc, const float2* Pp, float2* Pn,
                      const TvArgs& a, float theta, bool first) {
  launch_inner<float2>(st, in, Pc, Pp, Pn, a, theta, first);
}

// Tiles of tv_inner2 and whether it pays (gz > 0): columns of up to 60 in x and what the threads of a block
// hold in y, shared out evenly, and the planes a block that take the least time.  Times in us, fitted to 100 grids from
// 8^3 to 200 x 190 x 110: a launch of tv_inner2 3 and, a step, what grows with the waves w of a CU, 0.65 + 0.046 w real
// (24 waves at most: two full blocks) or 0.7 + 0.079 w complex (12); an iteration of tv_inner 3.3 and its bytes at 5.2 TB/s
// or 3.2 for every three or four blocks of a CU, 5.2 (real) and 6.5 (complex) at least.
// Small complex grids gain as real ones do (8^3 6.0 -> 3.3 us, 30 x 58 x 119 8.4 -> 6.1); flat ones keep tv_inner
// (500 x 500 x 1 real 5.5, 7.0; complex 7.0, 12.6).
TvTiles tv_tiles(const TvArgs& a, bool cplx) {
  TvTiles g;
  g.gx = (a.nx + 59) / 60;
  g.tx = (a.nx + g.gx - 1) / g.gx + 4;
  const int uy = kTvT2 / g.tx - 4;
  g.gy = (a.ny + uy - 1) / uy;
  g.ty = (a.ny + g.gy - 1) / g.gy + 4;
  const long long cols = (long long)g.gx * g.gy, cus = 256;
  const int waves = (g.tx * g.ty + 63) / 64;       // of a block
  // blocks on a CU: by registers, and by the 18 and 36 KB of LDS
  const long long held = std::max(1, std::min((cplx ? 12 : 24) / waves, cplx ? 4 : 8));
  double best = 0.0;
  for (int zc = 1; zc <= a.nz; ++zc) {
    const long long nb = cols * ((a.nz + zc - 1) / zc);
    const long long rounds = (nb + held * cus - 1) / (held * cus);
    const double w = (double)waves * std::min(held, (nb + cus - 1) / cus);
    const double t = 3.0 + (double)rounds * (zc + 4) * (cplx ? 0.7 + 0.079 * w : 0.65 + 0.046 * w);
    if (best == 0.0 || t < best) {
      best = t;
      g.zc = zc;
    }
    if (nb <= cus) break;                          // one block a CU: more planes a block only take longer
  }
  g.gz = (a.nz + g.zc - 1) / g.zc;
  const double bytes = 10.0 * (cplx ? 8.0 : 4.0) * a.nx * a.ny * a.nz;
  const TvColumns c = tv_columns(a);
  const double rounds1 = (double)c.gx * c.gy * ((a.nz + kTvZ - 1) / kTvZ) / (cplx ? 768 : 1024);
  if (best >= 2.0 * std::max(cplx ? 6.5 : 5.2, 3.3 + std::max(bytes / 5.2e6, 3.2 * rounds1)) || cols * g.gz >= (1ll << 31)) g.gz = 0;
  return g;
}
template <class T>
static void launch_inner2(hipStream_t st, const T* in, const T* Pc, const T* Pp, T* P1, T* P2, const TvArgs& a,
                          const TvTiles& g, float theta, float theta1) {
  const dim3 grid((unsigned)((long long)g.gx * g.gy * g.gz)), block((unsigned)(g.tx * g.ty));
  if ((unsigned long long)a.nx * a.ny * sizeof(T) < (1ull << 32))
    hipLaunchKernelGGL((tv_inner2<T, unsigned>), grid, block, 0, st, in, Pc, Pp, P1, P2, a, g, theta, theta1);
  else
    hipLaunchKernelGGL((tv_inner2<T, unsigned long long>), grid, block, 0, st, in, Pc, Pp, P1, P2, a, g, theta, theta1);
}
void tv_inner2_real(hipStream_t st, const float* in, const float* Pc, const float* Pp, float* P1, float* P2,
                    const TvArgs& a, const TvTiles& g, float theta, float theta1) {
  launch_inner2<float>(st, in, Pc, Pp, P1, P2, a, g, theta, theta1);
}
void tv_inner2_complex(hipStream_t st, const float2* in, const float2* Pc, const float2* Pp, float2* P1, float2* P2,
                       const TvArgs& a, const TvTiles& g, float theta, float theta1) {
  launch_inner2<float2>(st, in, Pc, Pp, P1, P2, a, g, theta, theta1);
}

__global__ void tv_zero(float* __restrict__ buf, long long n) {
  GRID_STRIDE_TV(i, n) buf[i] = 0.f;
}

// grad[i] = -(i / n_rhs) * sum_r conj(u_r[i]) * conj(w_r[flip_z(i)]), FP64 sums.
// Codes/BACKWARD_SOLVER_MULTI.m:50-53 with w = flip(conj(w_adjoint), 3).
__global__ void field_gradient(const float2* __restrict__ u, const float2* __restrict__ w, int nx, int ny, int nz,
                               int n_rhs, double2* __restrict__ grad) {
  const long long nxy = (long long)nx * ny;
  const long long n = nxy * nz;
  GRID_STRIDE_TV(i, n) {
    const long long z = i / nxy;
    const long long j = i + (nz - 1 - 2 * z) * nxy;   // same (x, y), z -> nz - 1 - z
    double sr = 0.0, si = 0.0;
    for (int r = 0; r < n_rhs; ++r) {
      const float2 a = u[(long long)r * n + i];
      const float2 b = w[(long long)r * n + j];
      // conj(a) * conj(b) = (a.x b.x - a.y b.y) - i (a.x b.y + a.y b.x)
      sr += (double)a.x * b.x - (double)a.y * b.y;
      si -= (double)a.x * b.y + (double)a.y * b.x;
    }
    const double inv = 1.0 / n_rhs;
    grad[i] = make_double2(si * inv, -sr * inv);   // -i (sr + i si) / n_rhs
  }
}

// FISTA of BACKWARD_SOLVER_MULTI (Codes/BACKWARD_SOLVER_MULTI.m:152-160) on the device,
// the iterates complex128 and x fastest.  Proximal input u - inv_alpha grad, rounded to
// complex64 (cplx) or its real part to float32, as the host loop forms it before the TV
// prox of that type.
__global__ void fista_prox_input(const double2* __restrict__ u, const double2* __restrict__ grad, double inv_alpha,
                                 long long n, int cplx, void* __restrict__ out) {
  GRID_STRIDE_TV(i, n) {
    const double2 g = grad[i], v = u[i];
    const double re = v.x - inv_alpha * g.x, im = v.y - inv_alpha * g.y;
    if (cplx) static_cast<float2*>(out)[i] = make_float2((float)re, (float)im);
    else static_cast<float*>(out)[i] = (float)re;
  }
}

// Principal square root of a + ib (a branch cut on the negative real axis, the sign of
// b kept for a <= 0): t = sqrt((|z| + |a|) / 2), then (t, b / 2t) for a >= 0 and
// (|b| / 2t, copysign(t, b)) for a < 0, so that neither part suffers cancellation.
__device__ __forceinline__ double2 csqrt_principal(double a, double b) {
  if (a == 0.0 && b == 0.0) return make_double2(0.0, b);
  const double t = sqrt(0.5 * (hypot(a, b) + fabs(a)));
  if (a >= 0.0) return make_double2(t, b / (2.0 * t));
  return make_double2(fabs(b) / (2.0 * t), copysign(t, b));
}

// After the proximal step s (complex64 when cplx, else float32, widened to FP64):
// u = s + c (s - x), x = s, ri = n_m sqrt(u + 1).
__global__ void fista_momentum(const void* __restrict__ s, int cplx, double2* __restrict__ x, double2* __restrict__ u,
                               double2* __restrict__ ri, long long n, double c, double n_m) {
  GRID_STRIDE_TV(i, n) {
    double2 sv;
    if (cplx) {
      const float2 f = static_cast<const float2*>(s)[i];
      sv = make_double2((double)f.x, (double)f.y);
    } else {
      sv = make_double2((double)static_cast<const float*>(s)[i], 0.0);
    }
    const double2 xv = x[i];
    const double2 un = make_double2(sv.x + c * (sv.x - xv.x), sv.y + c * (sv.y - xv.y));
    u[i] = un;
    x[i] = sv;
    const double2 r = csqrt_principal(un.x + 1.0, un.y);
    ri[i] = make_double2(n_m * r.x, n_m * r.y);
  }
}

}  // namespace cbs
