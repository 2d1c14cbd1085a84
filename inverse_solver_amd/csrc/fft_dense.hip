// Line transforms of any length on the matrix cores (see fft_rt.hpp).
//
// A line of n = F m elements is F interleaved lines of m, each transformed as a product with
// the m x m DFT matrix, then F-point butterflies:
//   Z_r[k] = sum_j x[F j + r] W_m^{jk},   X[k + m q] = sum_r W_F^{rq} (W_n^{rk} Z_r[k]).
// The products run on the FP32 matrix instructions.  With a_j = x_j + x_{m-j}, b_j = x_j - x_{m-j}
// and h = floor(m / 2),
//   C_k = sum_{j<=h} cos(2 pi jk / m) a_j,   S_k = sum_{j<=h} sin(2 pi jk / m) b_j,
//   Z[k] = C_k - i S_k,   Z[m - k] = C_k + i S_k       (signs swapped for the inverse),
// so a line costs 2 m operations an element, half of the plain product, and an output row k <= h
// gives two elements.  A 16 x 16 x 4 instruction holds 16 rows k, 16 lines and 4 elements j; the
// real and imaginary parts of the lines are separate right operands of the same left one, and
// the left operands are picked from a table of the m roots in LDS.
//
// A block holds a tile of 16 lines in LDS, element e of line l at e P + l.  Every wave takes
// (r, 16 rows) tasks, keeps their results in registers until all have read the tile, and writes
// them over it.  Against Bluestein's transform on a compiled length (two transforms of 2 n points
// and more, ten LDS round trips) this is two or three round trips.
#include "fft_rt.hpp"

namespace cbs {

constexpr int kL = 16;          // lines of a tile

typedef float v4f __attribute__((ext_vector_type(4)));

// F-point butterflies over r (element r m + k of every line), in place.
template <int F, bool INV, int P, int NT>
__device__ __forceinline__ void dense_butterfly(float2* __restrict__ lds, int m, int tid) {
  for (int i = tid; i < m * kL; i += NT) {
    float2* x = lds + (i >> 4) * P + (i & 15);
    float2 v[F];
#pragma unroll
    for (int r = 0; r < F; ++r) v[r] = x[r * m * P];
    Dft<F, INV>::run(v);
#pragma unroll
    for (int q = 0; q < F; ++q) x[q * m * P] = v[q];
  }
  lds_barrier();
}

// x mod m for 0 <= x < 2^20 (the float quotient is off by one at most)
__device__ __forceinline__ int mod_small(int x, int m, float inv_m) {
  int r = x - (int)((float)x * inv_m) * m;
  r = r < 0 ? r + m : r;
  return r >= m ? r - m : r;
}

// The tables, requested (load) ahead of the tile and put into LDS with it: the m roots
// (cos, sin)(2 pi e / m), then, for F > 1, exp(-2 pi i e / n): at most 2 n <= TK NT values.
template <int NT, int TK>
struct DenseTables {
  float2 v[TK];
  int cnt;
  __device__ __forceinline__ void load(const DenseArgs& p, int tid) {
    cnt = dense_tables(p);
#pragma unroll
    for (int k = 0; k < TK; ++k) v[k] = p.tab[min(tid + k * NT, cnt - 1)];
  }
  __device__ __forceinline__ void store(float2* __restrict__ s_tw, int tid) const {
#pragma unroll
    for (int k = 0; k < TK; ++k)
      if (tid + k * NT < cnt) s_tw[tid + k * NT] = v[k];
  }
};

// Transform of the 16 lines of the tile (natural order in and out, unnormalised).  s_tw: the
// tables of DenseTables.  Called by every thread after a barrier; ends with one.
template <int P, int NT, int TPW, bool INV>
__device__ void dense_lines(float2* __restrict__ lds, const float2* __restrict__ s_tw, const DenseArgs& p, int tid) {
  constexpr int NW = NT / 64;
  const int lane = tid & 63, c = lane & 15, g = lane >> 4;
  // the waves of a block sit on the four SIMDs in turn; where the tasks are fewer than the waves, the
  // first wave to take one moves on from block to block, so that no SIMD is left without
  const int w = __builtin_amdgcn_readfirstlane(((tid >> 6) + blockIdx.x) & (NW - 1));
  const int F = p.F, m = p.m, h = m >> 1;
  float2 lo[TPW][4], hi[TPW][4];      // Z_r[k] and Z_r[m - k], twiddled, of rows k = 16 t + 4 g + i
#pragma unroll
  for (int q = 0; q < TPW; ++q) {
    const int task = w + q * NW;
    if (task < p.ntask) {
      const int t = (task * p.inv_F) >> 16, r = task - t * F;
      const int row = 16 * t + c;                          // left operand: row of this lane
      // byte offset of the root of element j = 4 s + g, stepped by 4 rows' worth
      const unsigned m8 = 8u * (unsigned)m;
      unsigned e = 8u * (unsigned)mod_small(g * row, m, p.inv_m);
      const unsigned de = 8u * (unsigned)mod_small(4 * row, m, p.inv_m);
      v4f cr = {0.f, 0.f, 0.f, 0.f}, ci = cr, sr = cr, si = cr;
      auto next_root = [&] {
        const float2 wt = *byte_at<const float2>(s_tw, e);
        e += de;
        e = min(e, e - m8);        // e - m8 wraps above e where e < m8
        return wt;
      };
      auto product = [&](float2 wt, float2 x, float2 y, float2 ya) {
        const float2 a = cadd(x, ya), b = csub(x, y);
        cr = __builtin_amdgcn_mfma_f32_16x16x4f32(wt.x, a.x, cr, 0, 0, 0);
        ci = __builtin_amdgcn_mfma_f32_16x16x4f32(wt.x, a.y, ci, 0, 0, 0);
        sr = __builtin_amdgcn_mfma_f32_16x16x4f32(wt.y, b.x, sr, 0, 0, 0);
        si = __builtin_amdgcn_mfma_f32_16x16x4f32(wt.y, b.y, si, 0, 0, 0);
      };
      const float2* base = lds + r * P + c;
      // the first and the last step hold the elements that are their own mirror (0 and m / 2)
      // and the ones past h, which are zero
      auto edge = [&](int j) {
        const int jc = j < h ? j : h;
        const int mj = jc ? m - jc : 0;
        float2 x = base[F * jc * P], y = base[F * mj * P];
        const float2 wt = next_root();
        if (j > h) x = y = make_float2(0.f, 0.f);
        product(wt, x, y, mj == jc ? make_float2(0.f, 0.f) : y);
      };
      edge(g);
      // two steps at a time: their six operands are read before the first product
      const float2* xa = base + F * (4 + g) * P;
      const float2* xb = base + F * (m - 4 - g) * P;
      const int dx = 4 * F * P;
      int s = 1;
      for (; s + 1 < p.ks - 1; s += 2) {
        const float2 x0 = xa[0], y0 = xb[0], x1 = xa[dx], y1 = xb[-dx];
        const float2 w0 = next_root(), w1 = next_root();
        xa += 2 * dx;
        xb -= 2 * dx;
        product(w0, x0, y0, y0);
        product(w1, x1, y1, y1);
      }
      if (s < p.ks - 1) {
        const float2 x0 = xa[0], y0 = xb[0], w0 = next_root();
        product(w0, x0, y0, y0);
      }
      if (p.ks > 1) edge(4 * (p.ks - 1) + g);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float2 u = make_float2(cr[i] + si[i], ci[i] - sr[i]);   // C - i S
        const float2 v = make_float2(cr[i] - si[i], ci[i] + sr[i]);   // C + i S
        lo[q][i] = INV ? v : u;
        hi[q][i] = INV ? u : v;
        if (r > 0) {
          const int k = min(16 * t + 4 * g + i, h);
          const float2 wl = s_tw[m + r * k], wh = s_tw[m + r * (m - k)];
          lo[q][i] = INV ? cmulc(lo[q][i], wl) : cmul(lo[q][i], wl);
          hi[q][i] = INV ? cmulc(hi[q][i], wh) : cmul(hi[q][i], wh);
        }
      }
    }
  }
  lds_barrier();
#pragma unroll
  for (int q = 0; q < TPW; ++q) {
    const int task = w + q * NW;
    if (task < p.ntask) {
      const int t = (task * p.inv_F) >> 16, r = task - t * F;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = 16 * t + 4 * g + i;
        if (k > h) continue;
        lds[(r * m + k) * P + c] = lo[q][i];
        if (k > 0) lds[(r * m + m - k) * P + c] = hi[q][i];
      }
    }
  }
  lds_barrier();
  switch (F) {
    case 1: break;
    case 2: dense_butterfly<2, INV, P, NT>(lds, m, tid); break;
    case 3: dense_butterfly<3, INV, P, NT>(lds, m, tid); break;
    case 4: dense_butterfly<4, INV, P, NT>(lds, m, tid); break;
    case 5: dense_butterfly<5, INV, P, NT>(lds, m, tid); break;
    case 6: dense_butterfly<6, INV, P, NT>(lds, m, tid); break;
    case 7: dense_butterfly<7, INV, P, NT>(lds, m, tid); break;
    default: dense_butterfly<8, INV, P, NT>(lds, m, tid); break;
  }
}

// ------------------------------------------------------------------ contiguous lines
// 16 rows of n <= 64 EC contiguous elements per block, two rows a wave: element (k, ch) of a
// thread is position lane + 64 ch of row 2 w + k.  Loads are clamped to the tile instead of
// predicated (rows past the last one repeat it and are not stored), so that they leave in one go.
constexpr int kNT = 512;
constexpr int kRW = kL * 64 / kNT;
constexpr int kPR = kL + 1;        // lanes walking a row spread over the banks
constexpr int tables_k(int n, int nt) { return (2 * n + nt - 1) / nt; }

template <int EC, class T>
__device__ __forceinline__ void load_rows(const T* __restrict__ base, int n, int nr, int w, int lane,
                                          T (&v)[kRW * EC]) {
#pragma unroll
  for (int k = 0; k < kRW; ++k) {
    const T* __restrict__ row = base + min(w * kRW + k, nr - 1) * n;
#pragma unroll
    for (int ch = 0; ch < EC; ++ch)
      v[k * EC + ch] = *byte_at<const T>(row, (unsigned)sizeof(T) * (unsigned)min(lane + 64 * ch, n - 1));
  }
}
// The potential of the rows: re and im of every element, the imaginary part in memory only where st.Vr is null.
template <int EC>
__device__ __forceinline__ void load_potential(const StateArgs& st, const Consts& c, int r0, int n, int nr, int w, int lane,
                                               float2 (&v)[kRW * EC]) {
  const bool real = st.Vr != nullptr;
  const unsigned sz = real ? 4u : 8u;
  const char* __restrict__ base = (real ? reinterpret_cast<const char*>(st.Vr) : reinterpret_cast<const char*>(st.V)) +
                                  (long long)r0 * n * sz;
#pragma unroll
  for (int k = 0; k < kRW; ++k) {
    const char* __restrict__ row = base + (long long)(min(w * kRW + k, nr - 1) * n) * sz;
#pragma unroll
    for (int ch = 0; ch < EC; ++ch) {
      const unsigned o = sz * (unsigned)min(lane + 64 * ch, n - 1);
      v[k * EC + ch].x = *byte_at<const float>(row, o);
      v[k * EC + ch].y = -c.eps;
      if (!real) v[k * EC + ch].y = *byte_at<const float>(row, o + 4u);
    }
  }
}
template <int EC>
__device__ __forceinline__ void put_rows(float2* __restrict__ lds, int n, int w, int lane, const float2 (&v)[kRW * EC]) {
#pragma unroll
  for (int k = 0; k < kRW; ++k)
#pragma unroll
    for (int ch = 0; ch < EC; ++ch)
      if (lane + 64 * ch < n) lds[(lane + 64 * ch) * kPR + w * kRW + k] = v[k * EC + ch];
}
template <int EC>
__device__ __forceinline__ void store_rows(float2* __restrict__ base, int n, int nr, int w, int lane,
                                           const float2* __restrict__ lds) {
#pragma unroll
  for (int k = 0; k < kRW; ++k) {
    const int l = w * kRW + k;
    if (l >= nr) break;
    float2* __restrict__ row = base + l * n;
#pragma unroll
    for (int ch = 0; ch < EC; ++ch)
      if (lane + 64 * ch < n) *byte_at<float2>(row, 8u * (unsigned)(lane + 64 * ch)) = lds[(lane + 64 * ch) * kPR + l];
  }
}

template <int EC, int TPW>
__global__ __launch_bounds__(kNT) void dense_rows(float2* data, long long nrows, DenseArgs p, int inverse) {
  extern __shared__ float2 s_tw[];             // the tables, then n x 17 of the tile
  float2* lds = s_tw + dense_tables(p);
  const int n = p.n, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long r0 = (long long)blockIdx.x * kL;
  const int nr = nrows - r0 < kL ? (int)(nrows - r0) : kL;
  float2* __restrict__ base = data + r0 * n;
  DenseTables<kNT, tables_k(64 * EC, kNT)> tabs;
  tabs.load(p, tid);
  float2 v[kRW * EC];
  load_rows<EC>(base, n, nr, w, lane, v);
  tabs.store(s_tw, tid);
  put_rows<EC>(lds, n, w, lane, v);
  lds_barrier();
  if (inverse) dense_lines<kPR, kNT, TPW, true>(lds, s_tw, p, tid);
  else dense_lines<kPR, kNT, TPW, false>(lds, s_tw, p, tid);
  store_rows<EC>(base, n, nr, w, lane, lds);
}

// Per-axis form: the inverse x transform of the spectrum rows, the pointwise update of
// update_plain (born_step) and the forward x transform of the next p in one launch, as
// line_rows_update.  The operands of the update are requested once the tile is in LDS and stay in
// flight through the inverse transform (lds_barrier; nothing else is read from memory until then).
// UPD = UPD_DEFER or UPD_PAIR: the launch is a steady one (that update, next p = gamma x), its
// pointwise step straight-line code; UPD = UPD_NONE takes every kind at run time.
template <int EC, int TPW, int UPD>
__global__ __launch_bounds__(kNT) __attribute__((amdgpu_waves_per_eu(EC <= 3 ? 4 : 1)))
void dense_rows_update(StateArgs st, Tables tb, Consts c, DenseArgs p, int upd_,
                                                         int fwd_, int jj_inv, int jj_fwd, ConvArgs cv) {
  constexpr int K = kRW * EC;
  const int upd = UPD == UPD_NONE ? upd_ : UPD;
  const int fwd = UPD == UPD_NONE ? fwd_ : FWD_GAMMA;
  extern __shared__ float2 s_tw[];
  float2* lds = s_tw + dense_tables(p);
  const int n = p.n, tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int slot = blockIdx.y;
  const int rows = c.ny * c.nz;                          // < 2^31: a slot's voxels fit a launch
  const int r0 = blockIdx.x * kL;
  const int nr = rows - r0 < kL ? rows - r0 : kL;
  const long long ro = (long long)slot * st.rhs_stride + (long long)r0 * n;
  float2* __restrict__ spec = st.spec + ro;
  float2* __restrict__ F = st.field + ro;
  float2* __restrict__ f = st.fstate + ro;
  if (cv.norms && jj_inv > 0) {
    const int rr = slot / cv.P;
    if (conv_stopped(cv, jj_inv - 1, rr)) {
      if (!conv_stopped(cv, jj_inv - 2, rr) && upd_kind(jj_inv - 1, cv.M) == UPD_DEFER)
        for (int i = tid; i < nr * n; i += kNT) F[i] = cadd(F[i], f[i]);
      return;
    }
  }
  const bool rq = upd != UPD_NONE;
  const bool rf = reads_f(upd, fwd), rF = reads_F(upd);
  const int par = st.parity[slot];
  DenseTables<kNT, tables_k(64 * EC, kNT)> tabs;
  tabs.load(p, tid);
  float2 xq[K], vv[K], xo[K], Fo[K];
  if (rq) load_rows<EC>(spec, n, nr, w, lane, xq);
  float2 rx[EC];                 // x ramp and mask of the thread's positions
  float mx[EC];
#pragma unroll
  for (int ch = 0; ch < EC; ++ch) {
    const int e = min(lane + 64 * ch, n - 1);
    rx[ch] = *byte_at<const float2>(tb.ramp_x, 8u * (unsigned)e);
    mx[ch] = *byte_at<const float>(tb.mask_x, 4u * (unsigned)e);
  }
  float2 ryz[kRW];               // y and z factors of the wave's rows
  float myz[kRW];
#pragma unroll
  for (int k = 0; k < kRW; ++k) {
    const int row = r0 + min(w * kRW + k, nr - 1);
    const int z = __builtin_amdgcn_readfirstlane(row / c.ny), y = row - z * c.ny;
    ryz[k] = cmul(tb.ramp_y[y], tb.ramp_z[z]);
    myz[k] = tb.mask_y[y] * tb.mask_z[z];
  }
  tabs.store(s_tw, tid);
  if (rq) put_rows<EC>(lds, n, w, lane, xq);
  load_potential<EC>(st, c, r0, n, nr, w, lane, vv);
  if (rf) load_rows<EC>(f, n, nr, w, lane, xo);
  if (rF) load_rows<EC>(F, n, nr, w, lane, Fo);
  lds_barrier();
  if (rq) dense_lines<kPR, kNT, TPW, true>(lds, s_tw, p, tid);
  const bool wF = writes_F(upd), wf = fwd == FWD_GAMMA;
  const bool want_norm = st.norms != nullptr;
  const bool want_fref = st.fref != nullptr && upd == UPD_VQ_ADD;
  const float sg_inv = sign_inv(jj_inv ? (jj_inv + par) & 1 : 0);
  const float sg_fwd = sign_fwd(jj_fwd ? (jj_fwd + par) & 1 : 0);
  double nrm = 0.0, nrmF = 0.0;
#pragma unroll
  for (int k = 0; k < kRW; ++k) {
    const int l = w * kRW + k;
    const bool mine = l < nr;
    float2* __restrict__ Frow = F + l * n;
    float2* __restrict__ frow = f + l * n;
#pragma unroll
    for (int ch = 0; ch < EC; ++ch) {
      const int i = k * EC + ch, e = lane + 64 * ch;
      if (e >= n) continue;
      const float2 q = rq ? lds[e * kPR + l] : make_float2(0.f, 0.f);
      const float2 xi = rf ? xo[i] : make_float2(0.f, 0.f), Fi = rF ? Fo[i] : make_float2(0.f, 0.f);
      float2 Fn = make_float2(0.f, 0.f), xn;
      double nq = 0.0;
      const float2 pn = born_step(upd, fwd, q, cmul(rx[ch], ryz[k]), mx[ch] * myz[k], vv[i], xi, Fi, c.inv_eps, sg_inv,
                                  sg_fwd, Fn, xn, want_norm, nq);
      if (mine) {
        nrm += nq;
        if (want_fref) nrmF += (double)Fn.x * Fn.x + (double)Fn.y * Fn.y;
        if (wF) *byte_at<float2>(Frow, 8u * (unsigned)e) = Fn;
        if (wf) *byte_at<float2>(frow, 8u * (unsigned)e) = xn;
      }
      lds[e * kPR + l] = pn;
    }
  }
  if (want_norm) flush_norm(nrm, st.norms, slot);
  if (want_fref) flush_norm(nrmF, st.fref, slot);
  if (fwd == FWD_NONE) return;
  lds_barrier();
  dense_lines<kPR, kNT, TPW, false>(lds, s_tw, p, tid);
  store_rows<EC>(spec, n, nr, w, lane, lds);
}

// ------------------------------------------------------------------ strided lines
// Tiles as fft_strided: 16 consecutive x positions of n <= KC NT / 16 elements.
// fn(k, i, in): element k of a thread is at i of the LDS tile and i / 16 of the line; column tid % 16.
template <int KC, int NT, class Fn>
__device__ __forceinline__ void each_strided(int n, int tid, const Fn& fn) {
#pragma unroll
  for (int k = 0; k < KC; ++k) {
    const int i = tid + k * NT;
    if (i < n * kL) fn(k, i);
  }
}
// The tile between memory (line element e at base + e es) and v; columns past tv repeat the last one
// and are not stored.
template <int KC, int NT>
__device__ __forceinline__ void load_strided(const float2* __restrict__ base, long long es, int n, int tv, int tid,
                                             float2 (&v)[KC]) {
  const float2* __restrict__ q = base + min(tid & 15, tv - 1);
#pragma unroll
  for (int k = 0; k < KC; ++k) v[k] = q[min((tid >> 4) + k * (NT / kL), n - 1) * es];
}
template <int KC, int NT>
__device__ __forceinline__ void store_strided(float2* __restrict__ base, long long es, int n, int tv, int tid,
                                              const float2* __restrict__ lds) {
  if ((tid & 15) >= tv) return;
  float2* __restrict__ q = base + (long long)(tid >> 4) * es + (tid & 15);
  const long long step = (NT / kL) * es;
  each_strided<KC, NT>(n, tid, [&](int k, int i) { q[k * step] = lds[i]; });
}

template <int KC, int NT, int TPW>
__global__ __launch_bounds__(NT) void dense_strided(float2* data, int nx, long long es, long long os, int nouter,
                                                     DenseArgs p, int inverse, int inner, long long os2, unsigned grouped) {
  extern __shared__ float2 s_tw[];
  float2* lds = s_tw + dense_tables(p);
  const int n = p.n, tid = threadIdx.x;
  const int ntile = (nx + kL - 1) / kL;
  const unsigned bid = tile_position(grouped);
  const int xt = bid % ntile;
  const int o = bid / ntile;
  const int tv = nx - xt * kL < kL ? nx - xt * kL : kL;
  float2* __restrict__ base = data + (long long)(o / inner) * os2 + (long long)(o % inner) * os + (long long)xt * kL;
  DenseTables<NT, tables_k(KC * NT / kL, NT)> tabs;
  tabs.load(p, tid);
  float2 v[KC];
  load_strided<KC, NT>(base, es, n, tv, tid, v);
  tabs.store(s_tw, tid);
  each_strided<KC, NT>(n, tid, [&](int k, int i) { lds[i] = v[k]; });
  lds_barrier();
  if (inverse) dense_lines<kL, NT, TPW, true>(lds, s_tw, p, tid);
  else dense_lines<kL, NT, TPW, false>(lds, s_tw, p, tid);
  store_strided<KC, NT>(base, es, n, tv, tid, lds);
}

// Per-axis form, one field component: the forward z transform, the Green's multiply of
// green_plain and the inverse z transform in one launch.
template <int KC, int NT, int TPW>
__global__ __launch_bounds__(NT) void dense_strided_green(float2* data, Tables tb, Consts c, DenseArgs p,
                                                           const uint8_t* __restrict__ parity, int jj, ConvArgs cv,
                                                           unsigned grouped) {
  extern __shared__ float2 s_tw[];
  float2* lds = s_tw + dense_tables(p);
  const int n = p.n, tid = threadIdx.x;
  const int ntile = (c.nx + kL - 1) / kL;
  const unsigned bid = tile_position(grouped);
  const int xt = bid % ntile;
  const int o = bid / ntile;
  const int y = o % c.ny, slot = o / c.ny;      // the grid holds ceil(nx / 16) ny slots blocks
  if (cv.norms && conv_stopped(cv, jj - 1, slot)) return;
  const int flip = flip_of(jj, parity, slot);
  const int x0 = xt * kL;
  const int tv = c.nx - x0 < kL ? c.nx - x0 : kL;
  const long long es = (long long)c.nx * c.ny;
  float2* __restrict__ base = data + (long long)slot * c.nvox + (long long)y * c.nx + x0;
  DenseTables<NT, tables_k(KC * NT / kL, NT)> tabs;
  tabs.load(p, tid);
  float2 v[KC];
  load_strided<KC, NT>(base, es, n, tv, tid, v);
  const int tx = tid & 15;                       // every element of a thread is in one column
  const float gxy = tb.green_x[flip * c.nx + x0 + (tx < tv ? tx : 0)] + (tb.green_y[flip * c.ny + y] - c.km2);
  const float* __restrict__ gz = tb.green_z + flip * c.nz;
  float gzv[KC];
#pragma unroll
  for (int k = 0; k < KC; ++k) gzv[k] = gz[min((tid >> 4) + k * (NT / kL), n - 1)];
  tabs.store(s_tw, tid);
  each_strided<KC, NT>(n, tid, [&](int k, int i) { lds[i] = v[k]; });
  lds_barrier();
  dense_lines<kL, NT, TPW, false>(lds, s_tw, p, tid);
  const float eps2 = c.eps * c.eps;
  each_strided<KC, NT>(n, tid, [&](int k, int i) {
    const float d = gxy + gzv[k];
    const float s = c.inv_n * __builtin_amdgcn_rcpf(fmaf(d, d, eps2));   // hardware reciprocal (1 ulp)
    lds[i] = cmul(lds[i], make_float2(d * s, c.eps * s));
  });
  lds_barrier();
  dense_lines<kL, NT, TPW, true>(lds, s_tw, p, tid);
  store_strided<KC, NT>(base, es, n, tv, tid, lds);
}

// The same for vector runs: the three components' tiles in LDS, the dyadic factor of green_plain_vec between
// the transforms.  68 x 98 x 58 x 4 rhs of three components, with the x passes fused as well: 263 -> 145 us an
// iteration (Bluestein's transforms and separate passes before).
template <int KC, int NT, int TPW>
__global__ __launch_bounds__(NT) void dense_strided_green3(float2* data, Tables tb, Consts c, DenseArgs p,
                                                            const uint8_t* __restrict__ parity, int jj, ConvArgs cv,
                                                           unsigned grouped) {
  extern __shared__ float2 s_tw[];
  float2* lds = s_tw + dense_tables(p);
  const int n = p.n, tid = threadIdx.x, tile = n * kL;
  const int ntile = (c.nx + kL - 1) / kL;
  const unsigned bid = tile_position(grouped);
  const int xt = bid % ntile;
  const int o = bid / ntile;
  const int y = o % c.ny, r = o / c.ny;         // the grid holds ceil(nx / 16) ny rhs blocks
  if (cv.norms && conv_stopped(cv, jj - 1, r)) return;
  const int flip = flip_of(jj, parity, 3 * r);
  const int x0 = xt * kL;
  const int tv = c.nx - x0 < kL ? c.nx - x0 : kL;
  const long long es = (long long)c.nx * c.ny;
  float2* __restrict__ base = data + (long long)(3 * r) * c.nvox + (long long)y * c.nx + x0;
  DenseTables<NT, tables_k(KC * NT / kL, NT)> tabs;
  tabs.load(p, tid);
  float2 va[KC], vb[KC];                         // two components are in flight
  load_strided<KC, NT>(base, es, n, tv, tid, va);
  load_strided<KC, NT>(base + c.nvox, es, n, tv, tid, vb);
  tabs.store(s_tw, tid);
  each_strided<KC, NT>(n, tid, [&](int k, int i) { lds[i] = va[k]; });
  load_strided<KC, NT>(base + 2 * c.nvox, es, n, tv, tid, va);
  each_strided<KC, NT>(n, tid, [&](int k, int i) { lds[tile + i] = vb[k]; });
  each_strided<KC, NT>(n, tid, [&](int k, int i) { lds[2 * tile + i] = va[k]; });
  lds_barrier();
#pragma unroll 1
  for (int q = 0; q < 3; ++q) dense_lines<kL, NT, TPW, false>(lds + q * tile, s_tw, p, tid);
  const int tx = flip * c.nx + x0 + min(tid & 15, tv - 1);   // every element of a thread is in one column
  const float gx = tb.green_x[tx], gy = tb.green_y[flip * c.ny + y], rx = tb.rad_x[tx], ry = tb.rad_y[flip * c.ny + y];
  const float* __restrict__ gz = tb.green_z + flip * n;
  const float* __restrict__ rz = tb.rad_z + flip * n;
  each_strided<KC, NT>(n, tid, [&](int, int i) {
    const int z = i >> 4;
    dyadic_mul(c, gx + gy + gz[z] - c.km2, rx, ry, rz[z], lds[i], lds[tile + i], lds[2 * tile + i]);
  });
  lds_barrier();
#pragma unroll 1
  for (int q = 0; q < 3; ++q) dense_lines<kL, NT, TPW, true>(lds + q * tile, s_tw, p, tid);
#pragma unroll 1
  for (int q = 0; q < 3; ++q) store_strided<KC, NT>(base + q * c.nvox, es, n, tv, tid, lds + q * tile);
}

// (longest line, threads of the strided kernels, most tasks of a tile).  The strided kernels
// take 256 threads where four waves hold the tasks: a CU then keeps twice the blocks, and with
// them twice the waves that have work in the products.  Lines of up to 64 points have at most 4 tasks, of up
// to 128 at most 8; only 170, 185 and 190 points take (192, 512, 16) and six lengths from 396 on (448, 512, 32).
#define DENSE_LIST(X) X(64, 256, 4) X(128, 256, 4) X(128, 512, 8) X(192, 512, 8) X(192, 512, 16) X(256, 512, 16) \
  X(320, 512, 16) X(384, 512, 16) X(448, 512, 16) X(448, 512, 32)
constexpr int tasks_a_wave(int tasks, int nt) { return (tasks + nt / 64 - 1) / (nt / 64); }
#define DENSE_ENTRY(N, NT, TASKS)                                                                                  \
  {&dense_rows<N / 64, tasks_a_wave(TASKS, kNT)>, &dense_strided<N * kL / NT, NT, tasks_a_wave(TASKS, NT)>,        \
   {&dense_rows_update<N / 64, tasks_a_wave(TASKS, kNT), UPD_NONE>,                                                \
    &dense_rows_update<N / 64, tasks_a_wave(TASKS, kNT), UPD_DEFER>,                                               \
    &dense_rows_update<N / 64, tasks_a_wave(TASKS, kNT), UPD_PAIR>},                                               \
   &dense_strided_green<N * kL / NT, NT, tasks_a_wave(TASKS, NT)>,                                                 \
   &dense_strided_green3<N * kL / NT, NT, tasks_a_wave(TASKS, NT)>, N, TASKS, kNT, NT, kL},
static const DenseInfo kDense[] = {DENSE_LIST(DENSE_ENTRY)};

const DenseInfo* find_dense(int n, int ntask) {
  for (const auto& e : kDense)
    if (n <= e.nmax && ntask <= e.tasks) return &e;
  return nullptr;
}

}  // namespace cbs
