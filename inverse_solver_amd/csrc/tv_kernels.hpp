#pragma once
#include <hip/hip_runtime.h>

namespace cbs {

struct TvArgs {
  int nx, ny, nz;
  float lam, vmin, vmax, vimag_max;
  int non_neg, dirichlet;
};

// Blocks of tv_inner2: gx x gy x gz of them, each of tx x ty threads and zc planes; gz = 0: tv_inner is faster.
struct TvTiles {
  int gx, gy, gz, tx, ty, zc;
};

// y = project(in - lam div(Q)) of a real potential (one float per voxel, the dual Q three) or a
// complex one (complex64 per voxel).
__global__ void tv_div_project(const float* __restrict__ in, const float* __restrict__ Q, float* __restrict__ y,
                               TvArgs a);
__global__ void tv_div_project_c(const float2* __restrict__ in, const float2* __restrict__ Q, float2* __restrict__ y,
                                 TvArgs a);
// One inner iteration: Pn = P_{k+1} from Pc = P_k and Pp = P_{k-1} (three volumes each, Pn apart
// from both) and the momentum theta between them; first: P_0 = 0, Pc and Pp are not read.
void tv_inner_real(hipStream_t st, const float* in, const float* Pc, const float* Pp, float* Pn, const TvArgs& a,
                   float theta, bool first);
void tv_inner_complex(hipStream_t st, const float2* in, const float2* Pc, const float2* Pp, float2* Pn,
                      const TvArgs& a, float theta, bool first);
// Two of them: P1 = P_{k+1} and P2 = P_{k+2} (apart from Pc, Pp and each other), with the momentum theta
// between P_k and P_{k-1} and theta1 between P_{k+1} and P_k.
void tv_inner2_real(hipStream_t st, const float* in, const float* Pc, const float* Pp, float* P1, float* P2,
                    const TvArgs& a, const TvTiles& g, float theta, float theta1);
void tv_inner2_complex(hipStream_t st, const float2* in, const float2* Pc, const float2* Pp, float2* P1, float2* P2,
                       const TvArgs& a, const TvTiles& g, float theta, float theta1);
TvTiles tv_tiles(const TvArgs& a, bool cplx);
__global__ void tv_zero(float* __restrict__ buf, long long n);

// Misfit gradient from the forward and adjoint 3D fields (n_rhs blocks of nx*ny*nz complex64).
__global__ void field_gradient(const float2* __restrict__ u, const float2* __restrict__ w, int nx, int ny, int nz,
                               int n_rhs, double2* __restrict__ grad);

// FISTA iterates on the device (complex128, x fastest): the proximal input and the
// momentum / RI update of BACKWARD_SOLVER_MULTI.m:152-160.
__global__ void fista_prox_input(const double2* __restrict__ u, const double2* __restrict__ grad, double inv_alpha,
                                 long long n, int cplx, void* __restrict__ out);
__global__ void fista_momentum(const void* __restrict__ s, int cplx, double2* __restrict__ x, double2* __restrict__ u,
                               double2* __restrict__ ri, long long n, double c, double n_m);

}  // namespace cbs
