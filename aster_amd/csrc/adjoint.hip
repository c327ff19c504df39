// Hand-written adjoint of the leapfrog (kick-drift-kick) step for trajectory
// gradients with respect to initial positions, velocities and masses.
//
// Forward step s (h = dt/2, a_s = a(x_s), Plummer-softened Newton):
//   vh = v_s + h a_s ;  x_{s+1} = x_s + dt vh ;  v_{s+1} = vh + h a_{s+1}
// (update_leapfrog, src/physics/tool_chain_impl.cpp:169-185, in the same
// expression order as aster_step). With lx, lv the adjoints of x, v:
//   lvh = lv_{s+1} + dt lx_{s+1}
//   lx_s = lx_{s+1} + J(x_s)^T (c_s lvh) [+ dL/dx_s at snapshots],  lv_s = lvh
//   lm  += M(x_s)^T (c_s lvh)
// where J = da/dx, M = da/dm and c_s = dt for s > 0 (the first half-kick of
// step s and the second half-kick of step s-1 act at the same x_s with the
// same weight, so their vector-Jacobian products merge) and c_0 = h. The last
// step's second half-kick has weight h lv_N = 0 because the loss depends on
// positions only.
//
// Time reversal: the state is recovered backwards from (x_{s+1}, v_{s+1},
// a_{s+1}) as vh = v_{s+1} - h a_{s+1}, x_s = x_{s+1} - dt vh, and
// v_s = vh - h a(x_s); every ckpt_every steps the state is re-anchored to the
// checkpoint written by the forward pass, so reconstruction error cannot grow
// over more than one segment. a(x_s) comes out of the same fused kernel as the
// vector-Jacobian products:
//   a_k   = G sum_j m_j d / s^3
//   gx_k  = G sum_j [u / s^3 - 3 d (d . u) / s^5],  u = m_k w_j - m_j w_k
//   gm_k  = -G sum_j (w_j . d) / s^3
// with d = x_j - x_k, s^2 = |d|^2 + eps^2, FP32 pair arithmetic on separations
// formed in FP64 (as ASTER_ALLPAIRS_FP32_KAHAN), Kahan-compensated FP32 sums
// over 64-source tiles and an FP64 combine over source slices.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "device.hpp"

namespace aster {

__device__ __forceinline__ float unpack_mass_adj(double w) {
  return __uint_as_float((unsigned)(unsigned long long)__double_as_longlong(w));
}

// Sources of the fused kernel, padded to npad with zero-mass bodies: positions
// (FP64, FP32 mass in the low word of w) and {w, m} in FP32. Masses are scaled
// by msc (Fp32Scales), so a and J^T w come out scaled by 2^-k.

// One target and its seven sums over a tile: a (3), J^T w (3), M^T w.
template <bool MASK>
struct AdjTarget {
  double px, py, pz;
  float wx, wy, wz, mk;
  __device__ __forceinline__ AdjTarget(const double4& q, const float4& w)
      : px(q.x), py(q.y), pz(q.z), wx(w.x), wy(w.y), wz(w.z), mk(w.w) {}

  // Adds source (q, p) to s. skip: the target's own pair, whose d = 0, but u =
  // m_k w_k - m_k w_k comes out of the FMA as the rounding error of m_k w_k,
  // which eps^-3 would amplify.
  __device__ __forceinline__ void pair(const double4& q, const float4& p, bool skip, float eps2,
                                       float* __restrict__ s) const {
    const float dx = (float)(q.x - px), dy = (float)(q.y - py), dz = (float)(q.z - pz);
    float r2 = fmaf(dx, dx, eps2);
    r2 = fmaf(dy, dy, r2);
    r2 = fmaf(dz, dz, r2);
    float inv = __builtin_amdgcn_rsqf(r2);
    if (MASK) inv = (r2 > 0.f) ? inv : 0.f;
    inv = skip ? 0.f : inv;
    const float inv2 = inv * inv;
    const float inv3 = inv2 * inv;
    const float mj = unpack_mass_adj(q.w);
    const float f = mj * inv3;
    s[0] = fmaf(f, dx, s[0]);
    s[1] = fmaf(f, dy, s[1]);
    s[2] = fmaf(f, dz, s[2]);
    const float ux = fmaf(mk, p.x, -(mj * wx));
    const float uy = fmaf(mk, p.y, -(mj * wy));
    const float uz = fmaf(mk, p.z, -(mj * wz));
    const float du = fmaf(dx, ux, fmaf(dy, uy, dz * uz));
    // J^T w: inv3 u - 3 (d.u) inv5 d = inv3 (u - s d), s = 3 (d.u) inv^2
    const float s3 = (du * inv2) * 3.f;
    s[3] = fmaf(fmaf(-s3, dx, ux), inv3, s[3]);
    s[4] = fmaf(fmaf(-s3, dy, uy), inv3, s[4]);
    s[5] = fmaf(fmaf(-s3, dz, uz), inv3, s[5]);
    const float dw = fmaf(dx, p.x, fmaf(dy, p.y, dz * p.z));
    s[6] = fmaf(-dw, inv3, s[6]);
  }

  // The sums of one 64-source tile; SELF: source `self` of it is the target.
  // AHEAD: the next source is read before the sums over the present one, and
  // kept there (k_adj_tiles with one tile per wave: 247 -> 235 us a step at n =
  // 16384; with four tiles per wave it costs 1 us at n = 1000).
  template <bool SELF, bool AHEAD>
  __device__ __forceinline__ void tile(const double4* __restrict__ src, const float4* __restrict__ wsrc, int self,
                                       float eps2, float* __restrict__ s) const {
#pragma unroll
    for (int c = 0; c < 7; ++c) s[c] = 0.f;
    if constexpr (AHEAD) {
      double4 q = src[0];
      float4 p = wsrc[0];
#pragma unroll 8
      for (int k = 0; k < kApTile; ++k) {
        const int j = min(k + 1, kApTile - 1);
        const double4 nq = src[j];
        const float4 np = wsrc[j];
        __builtin_amdgcn_sched_barrier(0);
        pair(q, p, SELF && k == self, eps2, s);
        hold_pad(q);
        q = nq;
        p = np;
      }
    } else {
#pragma unroll 8
      for (int k = 0; k < kApTile; ++k) pair(src[k], wsrc[k], SELF && k == self, eps2, s);
    }
  }
};

// One target per lane, one slice of the sources per block row: out [S][7][n].
// Sources are read with wave-uniform addresses, through the scalar cache.
template <bool MASK>
__global__ __launch_bounds__(256) void k_adj_fused(const double4* __restrict__ src, const float4* __restrict__ wsrc,
                                                   int n, int npad, int slice_len, float eps2,
                                                   double* __restrict__ out) {
  const int i = blockIdx.x * kApBlock + threadIdx.x;
  const int ii = i < n ? i : n - 1;
  const int sl = blockIdx.y;
  const int jb = sl * slice_len;
  const int je = min(jb + slice_len, npad);
  const AdjTarget<MASK> me(src[ii], wsrc[ii]);
  const int lane = threadIdx.x & 63;
  // the wavefront's targets i0 .. i0 + 63 are sources of tile i0 (tiles are
  // 64-aligned, as are the slices)
  const int self_tile = __builtin_amdgcn_readfirstlane(i - lane);
  float S[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  float C[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  for (int t = jb; t < je; t += kApTile) {
    float s[7];
    if (t == self_tile)
      me.template tile<true, false>(src + t, wsrc + t, lane, eps2, s);
    else
      me.template tile<false, false>(src + t, wsrc + t, 0, eps2, s);
#pragma unroll
    for (int q = 0; q < 7; ++q) kahan_add32(S[q], C[q], s[q]);
  }
  if (i < n) {
    double* o = out + (size_t)sl * 7 * n;
#pragma unroll
    for (int q = 0; q < 7; ++q) o[(size_t)q * n + i] = (double)S[q] - (double)C[q];
  }
}

// What a backward step does with the sums of x_s. For coordinate c of body i
// (k = c n + i): v_s = vh - h a(x_s), or the checkpoint velocity; lx += gx (+
// the snapshot's gradient). Then the reverse half of step s - 1 (not for s =
// 0): lvh = lv + dt lx; vh = v_s - h a; x -= dt vh, or the checkpoint's
// position; v = vh; lv = lvh; w = c lvh.
struct AdjStep {
  double gsc, G;  // scales of the sums: a and gx by G 2^k, gm by G
  double dt;
  double cw;      // weight of the next w
  int last;       // s = 0: no step before it; a goes to acc
  double *x, *v, *lx, *lv, *lm, *acc;
  const double* ckv;    // checkpoint velocities of s, may be null
  const double* gsnap;  // snapshot gradients of s, may be null
  const double* ckx;    // checkpoint positions of s - 1, may be null
  double4* src;         // sources of s - 1
  float4* wsrc;
};

// The reverse half of a step: x and w of the step before.
__device__ __forceinline__ void adj_reverse(const AdjStep& A, size_t k, double vs, double a, double lx, double* xn,
                                            double* wn) {
#pragma clang fp contract(off)
  const double h = 0.5 * A.dt;
  const double lvh = A.lv[k] + A.dt * lx;
  const double vh = vs - h * a;
  *xn = A.ckx ? A.ckx[k] : A.x[k] - A.dt * vh;
  A.x[k] = *xn;
  A.v[k] = vh;
  A.lv[k] = lvh;
  *wn = A.cw * lvh;
}

__device__ __forceinline__ void adj_update(const AdjStep& A, size_t k, double a, double gx, double* xn, double* wn) {
#pragma clang fp contract(off)
  const double h = 0.5 * A.dt;
  const double vs = A.ckv ? A.ckv[k] : A.v[k] - h * a;
  double g = A.lx[k] + gx;
  if (A.gsnap) g += A.gsnap[k];
  A.lx[k] = g;
  if (A.last) {
    A.v[k] = vs;
    A.acc[k] = a;
    *xn = *wn = 0.0;
  } else {
    adj_reverse(A, k, vs, a, g, xn, wn);
  }
}

__device__ __forceinline__ double adj_mass_slot(float mf) {
  return __longlong_as_double((long long)(unsigned long long)__float_as_uint(mf));
}

// The first reverse half (step N - 1, accelerations of the forward pass), with
// the sources and padding of both source buffers.
__global__ __launch_bounds__(256) void k_adj_first(int n, int npad, float msc, AdjStep A,
                                                   const double* __restrict__ m, double4* __restrict__ src2,
                                                   float4* __restrict__ wsrc2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npad) return;
  double4 q = make_double4(0.0, 0.0, 0.0, adj_mass_slot(0.f));
  float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
  if (i < n) {
    double xn[3], wn[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t k = (size_t)c * n + i;
      adj_reverse(A, k, A.v[k], A.acc[k], A.lx[k], &xn[c], &wn[c]);
    }
    const float mf = (float)m[i] * msc;
    q = make_double4(xn[0], xn[1], xn[2], adj_mass_slot(mf));
    w = make_float4((float)wn[0], (float)wn[1], (float)wn[2], mf);
  }
  A.src[i] = q;
  A.wsrc[i] = w;
  src2[i] = q;  // the masses and padding stay, the rest is rewritten
  wsrc2[i] = w;
}

// Sums the slice partials in slice order, scales them, and applies the step's
// update with the sums in registers: with the pair kernel two launches a step
// (four small ones of about 4.7 us each before).
__global__ __launch_bounds__(256) void k_adj_step(int n, int S, const double* __restrict__ part, AdjStep A) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  // 4 slices per round, their 28 loads issued before the first add (clamped
  // slice index); the adds stay in slice order
  double s[7] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < S; k0 += 4) {
    double v[4][7];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int k = min(k0 + u, S - 1);
#pragma unroll
      for (int q = 0; q < 7; ++q) v[u][q] = part[((size_t)k * 7 + q) * n + i];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (k0 + u < S)
#pragma unroll
        for (int q = 0; q < 7; ++q) s[q] += v[u][q];
  }
  double xn[3], wn[3];
#pragma unroll
  for (int c = 0; c < 3; ++c)
    adj_update(A, (size_t)c * n + i, s[c] * A.gsc, s[3 + c] * A.gsc, &xn[c], &wn[c]);
  A.lm[i] += s[6] * A.G;
  if (!A.last) {
    const float mf = A.wsrc[i].w;
    A.src[i] = make_double4(xn[0], xn[1], xn[2], adj_mass_slot(mf));
    A.wsrc[i] = make_float4((float)wn[0], (float)wn[1], (float)wn[2], mf);
  }
}

// Small and middle-sized problems: the tiles of a slice spread over the waves
// of a block, sources in LDS, as k_allpairs_tiles: W worker waves sum GR tiles
// each per round for the block's 64 / GR targets, one more wave takes the tile
// sums in tile order, Kahan-compensated within each slice, the slices in FP64:
// the bits of k_adj_fused and k_adj_step. With GR = 4 a block takes every
// source and its last wave applies the step's update, so a backward step is
// one launch (the sources then alternate between two buffers); with `part`
// block row y takes slice y and writes its sums for k_adj_step.
template <int W, int GR, bool MASK>
__global__ __launch_bounds__(64 * (W + 1)) void k_adj_tiles(const double4* __restrict__ src,
                                                            const float4* __restrict__ wsrc, int n, int tiles,
                                                            int slice_tiles, float eps2, double* __restrict__ part,
                                                            AdjStep A) {
  constexpr int TG = 64 / GR;      // targets of the block, lanes of a group
  constexpr int R = GR * W;        // tiles per round
  constexpr int NC = GR == 1 ? 7 : 2;  // sums per lane of the last wave
  static_assert(GR == 1 || GR == 4, "the last wave's lanes are laid out for 64 or 16 targets");
  __shared__ double4 tq[W][GR][kApTile + 1];
  __shared__ float4 tp[W][GR][kApTile + 1];
  __shared__ float sums[2][R][7][TG];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * TG;
  int t0 = 0;
  if (part) {  // this block's slice
    t0 = blockIdx.y * slice_tiles;
    tiles = min(slice_tiles, tiles - t0);
  }
  const int rounds = (tiles + R - 1) / R;
  if (w < W) {
    const int ti = lane % TG, g = lane / TG;
    const int i = min(i0 + ti, n - 1);
    double4 q[GR];
    float4 p[GR];
    auto fetch = [&](int rd) {
#pragma unroll
      for (int u = 0; u < GR; ++u) {
        const int j = (t0 + min(rd * R + GR * w + u, tiles - 1)) * kApTile + lane;
        q[u] = src[j];
        p[u] = wsrc[j];
      }
    };
    fetch(0);
    const AdjTarget<MASK> me(src[i], wsrc[i]);
    for (int rd = 0; rd < rounds; ++rd) {
      const int first = rd * R + GR * w;
      if (first < tiles) {  // wave-uniform
        wave_sync();        // the wave is done with its previous tiles
#pragma unroll
        for (int u = 0; u < GR; ++u) {
          tq[w][u][lane] = q[u];
          tp[w][u][lane] = p[u];
        }
        wave_sync();
        if (rd + 1 < rounds) fetch(rd + 1);
        float s[7];
        // the block's targets all lie in one tile
        const int st = i0 / kApTile - (t0 + first);
        const int self = st == g ? (i & (kApTile - 1)) : -1;
        if (st >= 0 && st < GR)
          me.template tile<true, GR == 1>(tq[w][g], tp[w][g], self, eps2, s);
        else
          me.template tile<false, GR == 1>(tq[w][g], tp[w][g], self, eps2, s);
#pragma unroll
        for (int c = 0; c < 7; ++c) sums[rd & 1][GR * w + g][c][ti] = s[c];
      }
      __syncthreads();  // the sums of this round are there, those of the round before are taken
    }
    return;
  }
  // Sum h of a lane. GR = 1: quantity h of target `lane`. GR = 4: lanes 0..47
  // coordinate lane / 16 of a and of J^T w of target lane % 16, lanes 48..63
  // M^T w (h = 0; h = 1 repeats it).
  const int ti = lane % TG, cl = lane / TG;
  float S[NC], C[NC];
  double tot[NC];
#pragma unroll
  for (int h = 0; h < NC; ++h) {
    S[h] = C[h] = 0.f;
    tot[h] = 0.0;
  }
  int left = slice_tiles;  // tiles to the end of the slice
  for (int rd = 0; rd < rounds; ++rd) {
    __syncthreads();
    const int cnt = min(R, tiles - rd * R);
    for (int k = 0; k < cnt; ++k) {
      const bool end = --left == 0 || (rd + 1 == rounds && k + 1 == cnt);
#pragma unroll
      for (int h = 0; h < NC; ++h) {
        const int c = GR == 1 ? h : cl == 3 ? 6 : 3 * h + cl;
        kahan_add32(S[h], C[h], sums[rd & 1][k][c][ti]);
        if (end) {
          tot[h] += (double)S[h] - (double)C[h];
          S[h] = C[h] = 0.f;
        }
      }
      if (end) left = slice_tiles;
    }
  }
  const int i = i0 + ti;
  if (i >= n) return;
  if constexpr (GR == 1) {
#pragma unroll
    for (int h = 0; h < NC; ++h) part[((size_t)blockIdx.y * 7 + h) * n + i] = tot[h];
  } else if (cl == 3) {
    A.lm[i] += tot[0] * A.G;
  } else {
    double xn, wn;
    adj_update(A, (size_t)cl * n + i, tot[0] * A.gsc, tot[1] * A.gsc, &xn, &wn);
    if (!A.last) {
      reinterpret_cast<double*>(A.src + i)[cl] = xn;
      reinterpret_cast<float*>(A.wsrc + i)[cl] = (float)wn;
    }
  }
}

__global__ void k_copy(size_t cnt, const double* __restrict__ s, double* __restrict__ d) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cnt) d[i] = s[i];
}

// ----------------------------------------------------------------- host ----

static int dcopy(aster_ctx* c, const double* s, double* d, size_t cnt) {
  hipLaunchKernelGGL(k_copy, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, c->stream, cnt, s, d);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

// Which kernels take a backward step of n bodies. Step in us, before (k_adj_fused
// and four small launches) / one launch, GR = 4 / k_adj_tiles by slices, GR = 1
// / k_adj_fused, two launches: n = 256 40 / 10.7 / 14 / 37, 1000 200 / 13.6 / 36
// / 213, 4096 208 / 33 / 36 / 225, 8192 210 / 116 / 70 / 223, 16384 290 / 425 /
// 235 / 274, 32768 891 / 1638 / 857 / 831, 65536 3277 / 6439 / 3431 / 3031.
// One launch fills the 256 CUs once up to 4096 bodies (16 targets a block).
static bool adj_one_launch(int64_t n) { return n <= 4096; }
static bool adj_in_tiles(int64_t n) { return n <= 20480; }

static void launch_adj_pairs(hipStream_t st, bool one, bool mask, const double4* src, const float4* wsrc, int n,
                             int npad, int S, int slice, float eps2, double* part, const AdjStep& A) {
  const int tiles = npad / kApTile, st_tiles = slice / kApTile;
  if (one) {
    // W = 4 waves hold 16 tiles (1024 sources) in one round
    const int W = tiles <= 16 ? 4 : 8;
    auto k = W == 4 ? (mask ? k_adj_tiles<4, 4, true> : k_adj_tiles<4, 4, false>)
                    : (mask ? k_adj_tiles<8, 4, true> : k_adj_tiles<8, 4, false>);
    hipLaunchKernelGGL(k, dim3((n + 15) / 16), dim3(64 * (W + 1)), 0, st, src, wsrc, n, tiles, st_tiles, eps2, nullptr,
                       A);
  } else if (adj_in_tiles(n)) {
    auto k = mask ? k_adj_tiles<4, 1, true> : k_adj_tiles<4, 1, false>;
    hipLaunchKernelGGL(k, dim3((n + 63) / 64, S), dim3(64 * 5), 0, st, src, wsrc, n, tiles, st_tiles, eps2, part, A);
  } else {
    auto k = mask ? k_adj_fused<true> : k_adj_fused<false>;
    hipLaunchKernelGGL(k, dim3(npad / kApBlock, S), dim3(kApBlock), 0, st, src, wsrc, n, npad, slice, eps2, part);
  }
}

int traj_forward(aster_ctx* c, double dt, int64_t nsteps, int64_t ckpt, int32_t nsnap, const int64_t* snaps,
                 double* snap_pos) {
  AdjointState& S = c->adj;
  S.ready = false;
  if (!std::isfinite(dt) || nsteps < 1 || ckpt < 1 || nsnap < 0 || (nsnap > 0 && !snaps))
    return fail(c, ASTER_ERR_INVALID, "need dt finite, nsteps >= 1, ckpt_every >= 1, snapshot steps");
  for (int q = 0; q < nsnap; ++q)
    if (snaps[q] < 1 || snaps[q] > nsteps || (q > 0 && snaps[q] <= snaps[q - 1]))
      return fail(c, ASTER_ERR_INVALID, "snapshot steps must be ascending within [1, nsteps]");
  if (c->P.pn_flags & ASTER_PN_TERMS) return fail(c, ASTER_ERR_INVALID, "the adjoint covers Newtonian forces");
  if (c->P.lower > 0 || (c->P.upper >= 0 && c->P.upper < c->n))
    return fail(c, ASTER_ERR_INVALID, "the adjoint evaluates the full body range only");
  const int64_t n = c->n;
  const size_t n3 = (size_t)3 * n;
  const int64_t nck = nsteps / ckpt + 1;
  if ((double)nck * 2.0 * n3 * 8.0 > 64e9) return fail(c, ASTER_ERR_CAPACITY, "checkpoints would exceed 64 GB");
  ASTER_HIP(c, S.ckpt_x.reserve(nck * n3));
  ASTER_HIP(c, S.ckpt_v.reserve(nck * n3));
  ASTER_HIP(c, S.snapg.reserve(std::max<size_t>(1, (size_t)nsnap * n3)));
  S.nsteps = nsteps;
  S.ckpt_every = ckpt;
  S.nsnap = nsnap;
  S.dt = dt;
  S.P = c->P;
  S.snap_steps.assign(snaps, snaps + nsnap);
  int rc;
  const int method = ASTER_ALLPAIRS_FP32_KAHAN;
  if ((rc = compute_forces(c, method))) return rc;
  int q = 0;
  for (int64_t s = 0; s < nsteps; ++s) {
    if (s % ckpt == 0) {  // the evaluation before applied the closing kick
      const size_t o = (size_t)(s / ckpt) * n3;
      if ((rc = dcopy(c, c->x.p, S.ckpt_x.p + o, n3)) || (rc = dcopy(c, c->v.p, S.ckpt_v.p + o, n3))) return rc;
      if ((rc = launch_kick_drift(c, 0.0, dt))) return rc;
    }
    if (q < nsnap && snaps[q] == s + 1) {
      if ((rc = dcopy(c, c->x.p, S.snapg.p + (size_t)q * n3, n3))) return rc;
      ++q;
    }
    const bool close = s + 1 == nsteps || (s + 1) % ckpt == 0;
    if ((rc = compute_forces(c, method, close ? StepPost{POST_KICK, 0.0, dt} : StepPost{POST_KICK_DRIFT, dt, dt})))
      return rc;
  }
  if (snap_pos && nsnap > 0) {
    std::vector<double> h((size_t)nsnap * n3);
    ASTER_HIP(c, hipMemcpyAsync(h.data(), S.snapg.p, h.size() * 8, hipMemcpyDeviceToHost, c->stream));
    ASTER_HIP(c, hipStreamSynchronize(c->stream));
    for (int k = 0; k < nsnap; ++k)
      for (int64_t i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d)
          snap_pos[(size_t)k * n3 + 3 * i + d] = h[(size_t)k * n3 + (size_t)d * n + i];
  }
  S.own_acc = true;
  S.ready = true;
  return ASTER_OK;
}

static int backward_passes(aster_ctx* c, const double* gsnap, double* gx, double* gv, double* gm) {
  AdjointState& S = c->adj;
  if (!S.ready) return fail(c, ASTER_ERR_STATE, "call aster_traj_forward first (and do not step in between)");
  if (S.nsnap > 0 && !gsnap) return fail(c, ASTER_ERR_INVALID, "snapshot gradients required");
  const int n = (int)c->n;
  const int npad = (int)c->npad;
  const size_t n3 = (size_t)3 * n;
  const double dt = S.dt, h = 0.5 * dt;
  ASTER_HIP(c, S.lx.reserve(n3));
  ASTER_HIP(c, S.lv.reserve(n3));
  ASTER_HIP(c, S.lm.reserve(n));
  for (int b = 0; b < 2; ++b) {
    ASTER_HIP(c, S.src[b].reserve(npad));
    ASTER_HIP(c, S.wsrc[b].reserve(npad));
  }
  // Snapshot gradients to device planes (reusing the snapshot buffer).
  if (S.nsnap > 0) {
    std::vector<double> hbuf((size_t)S.nsnap * n3);
    for (int k = 0; k < S.nsnap; ++k)
      for (int i = 0; i < n; ++i)
        for (int d = 0; d < 3; ++d) hbuf[(size_t)k * n3 + (size_t)d * n + i] = gsnap[(size_t)k * n3 + 3 * i + d];
    ASTER_HIP(c, hipMemcpyAsync(S.snapg.p, hbuf.data(), hbuf.size() * 8, hipMemcpyHostToDevice, c->stream));
    ASTER_HIP(c, hipStreamSynchronize(c->stream));
  }
  ASTER_HIP(c, hipMemsetAsync(S.lx.p, 0, n3 * 8, c->stream));
  ASTER_HIP(c, hipMemsetAsync(S.lv.p, 0, n3 * 8, c->stream));
  ASTER_HIP(c, hipMemsetAsync(S.lm.p, 0, n * 8, c->stream));
  int q = S.nsnap - 1;
  if (q >= 0 && S.snap_steps[q] == S.nsteps) {
    int rc = dcopy(c, S.snapg.p + (size_t)q * n3, S.lx.p, n3);
    if (rc) return rc;
    --q;
  }
  c->src_ready = SrcReady{};  // the passes below move the state
  int Sl = choose_split(c);
  int64_t slice = round_up((npad + Sl - 1) / Sl, kApTile);
  Sl = (int)((npad + slice - 1) / slice);
  const bool one = adj_one_launch(n);
  if (!one) ASTER_HIP(c, S.part.reserve((size_t)Sl * 7 * n));
  Fp32Scales sc;
  int rc0 = fp32_scales(c, &sc);
  if (rc0) return rc0;
  AdjStep A{};
  A.gsc = sc.gsc;
  A.G = c->P.G;
  A.dt = dt;
  A.x = c->x.p;
  A.v = c->v.p;
  A.lx = S.lx.p;
  A.lv = S.lv.p;
  A.lm = S.lm.p;
  A.acc = c->a.p;
  // weight and checkpoint of the reverse half of step s, to source buffer b
  auto aim = [&](int64_t s, int b) {
    A.cw = s > 0 ? dt : h;
    A.ckx = s % S.ckpt_every == 0 ? S.ckpt_x.p + (size_t)(s / S.ckpt_every) * n3 : nullptr;
    A.src = S.src[b].p;
    A.wsrc = S.wsrc[b].p;
  };
  int b = 0;
  aim(S.nsteps - 1, b);
  phase_begin(c, ASTER_PHASE_KICKDRIFT);
  hipLaunchKernelGGL(k_adj_first, dim3(npad / 256), dim3(256), 0, c->stream, n, npad, sc.msc, A, c->m.p, S.src[1].p,
                     S.wsrc[1].p);
  phase_end(c, ASTER_PHASE_KICKDRIFT);
  for (int64_t s = S.nsteps - 1; s >= 0; --s) {
    const double4* src = S.src[b].p;
    const float4* wsrc = S.wsrc[b].p;
    if (one) b ^= 1;  // other blocks still read this step's sources
    A.last = s == 0;
    A.ckv = s % S.ckpt_every == 0 ? S.ckpt_v.p + (size_t)(s / S.ckpt_every) * n3 : nullptr;
    A.gsnap = nullptr;
    if (q >= 0 && S.snap_steps[q] == s) {
      A.gsnap = S.snapg.p + (size_t)q * n3;
      --q;
    }
    if (s > 0) aim(s - 1, b);
    phase_begin(c, ASTER_PHASE_ADJOINT);
    launch_adj_pairs(c->stream, one, sc.mask, src, wsrc, n, npad, Sl, (int)slice, sc.eps2, S.part.p, A);
    phase_end(c, ASTER_PHASE_ADJOINT);
    if (!one) {
      phase_begin(c, ASTER_PHASE_COMBINE);
      hipLaunchKernelGGL(k_adj_step, dim3((n + 255) / 256), dim3(256), 0, c->stream, n, Sl, (const double*)S.part.p, A);
      phase_end(c, ASTER_PHASE_COMBINE);
    }
    ASTER_HIP(c, hipGetLastError());
  }
  // The state is back at step 0 (re-anchored to the first checkpoint) with
  // a = a(x_0) from the mixed-precision kernel.
  c->acc_valid = true;
  c->acc_stale = false;
  c->acc_method = ASTER_ALLPAIRS_FP32_KAHAN;
  S.ready = false;
  auto down = [&](const double* dev, double* host) -> int {
    std::vector<double> t(n3);
    ASTER_HIP(c, hipMemcpyAsync(t.data(), dev, n3 * 8, hipMemcpyDeviceToHost, c->stream));
    ASTER_HIP(c, hipStreamSynchronize(c->stream));
    for (int i = 0; i < n; ++i)
      for (int d = 0; d < 3; ++d) host[3 * (size_t)i + d] = t[(size_t)d * n + i];
    return ASTER_OK;
  };
  int rc;
  if (gx && (rc = down(S.lx.p, gx))) return rc;
  if (gv && (rc = down(S.lv.p, gv))) return rc;
  if (gm) {
    ASTER_HIP(c, hipMemcpyAsync(gm, S.lm.p, n * 8, hipMemcpyDeviceToHost, c->stream));
    ASTER_HIP(c, hipStreamSynchronize(c->stream));
  }
  return ASTER_OK;
}

// The gradient of the trajectory as it was run: with the forward pass's
// parameters and last accelerations, whatever was set or evaluated since.
int traj_backward(aster_ctx* c, const double* gsnap, double* gx, double* gv, double* gm) {
  AdjointState& S = c->adj;
  const aster_params now = c->P;
  int rc = ASTER_OK;
  if (S.ready) {
    c->P = S.P;
    if (!S.own_acc) rc = compute_forces(c, ASTER_ALLPAIRS_FP32_KAHAN);
  }
  if (!rc) rc = backward_passes(c, gsnap, gx, gv, gm);
  c->P = now;
  if (now.G != S.P.G || now.softening != S.P.softening || now.pn_flags != S.P.pn_flags || now.lower != S.P.lower ||
      now.upper != S.P.upper)
    c->acc_valid = false;
  return rc;
}

}  // namespace aster
