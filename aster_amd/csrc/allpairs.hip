// All-pairs gravitational accelerations on CDNA4.
//
// FP32 paths: one target body per lane; source bodies are read with
// wave-uniform addresses, so they arrive through the scalar cache into SGPRs
// and feed VALU instructions directly (no LDS staging, no barriers). The
// source range is split into slices (grid.y) so that a 64K-body problem puts
// several waves on every SIMD; slice partials are combined in FP64 in a fixed
// order, so results are deterministic. Up to some tens of thousands of bodies
// one launch does the whole evaluation and the integrator's update instead,
// with the sources in LDS (k_allpairs_tiles). Per interaction the plain FP32 loop
// issues 3 sub + 3 fma (r^2) + 1 rsq + 3 mul + 3 fma = 12 VALU + 1
// transcendental; the mixed method forms the separation in FP64 and rounds it
// (3 add_f64 + 3 cvt instead of 3 sub: 15 VALU + 1 transcendental) and
// accumulates with Kahan compensation across 64-source tiles.
//
// FP64 path: the reference's operation order (Parallelized::compute_forces,
// src/utils/builder_endpoint.cpp:729-757, with compute_gravitational,
// src/physics/tool_chain_impl.cpp:120-137), each target's sources summed in j
// order, IEEE division and square root, no contraction: bit-identical to the
// CPU path. The pair contributions of a chunk of sources are formed by a whole
// block and summed per target afterwards.
#include <algorithm>
#include <cfloat>
#include <cmath>
#include <mutex>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "device.hpp"

namespace aster {

// ---------------------------------------------------------------- FP32 ----

enum { ACC_PLAIN = 0, ACC_TILE_KAHAN = 1 };

// Sources, padded to npad with zero-mass bodies at the origin. Bodies outside
// the source range [lower, upper) (Solver::set_bounds) get zero mass, which
// adds exactly zero force. Masses are scaled by msc (Fp32Scales).
//   FP32 {x, y, z, m} (positions rounded to FP32 once) for the plain method;
//   FP64 {x, y, z, m} for the mixed one: the kernel forms x_j - x_i in FP64 and
//   rounds the separation to FP32, so the pair force is FP32 but a close pair
//   does not lose ~|x|/r ulps to position rounding. The w slot carries the
//   FP32 mass in its low 32 bits, so the kernel reads it straight from the low
//   SGPR of the pair without a conversion.
__device__ __forceinline__ double pack_mass(float m) {
  return __longlong_as_double((long long)(unsigned long long)__float_as_uint(m));
}
__device__ __forceinline__ float unpack_mass(double w) {
  return __uint_as_float((unsigned)(unsigned long long)__double_as_longlong(w));
}

__device__ __forceinline__ float src_mass(const float4& q) { return q.w; }
__device__ __forceinline__ float src_mass(const double4& q) { return unpack_mass(q.w); }

template <bool SRC64>
struct SrcT;
template <>
struct SrcT<false> {
  using type = float4;
  static __device__ __forceinline__ float4 make(double x, double y, double z, float m) {
    return make_float4((float)x, (float)y, (float)z, m);
  }
};
template <>
struct SrcT<true> {
  using type = double4;
  static __device__ __forceinline__ double4 make(double x, double y, double z, float m) {
    return make_double4(x, y, z, pack_mass(m));
  }
};

// Source j: the body's record, its mass only inside [lower, upper); zeros past
// n. The mass scale is msc, or read from the device where dmsc is given.
struct SrcRange {
  int n, lower, upper;
  float msc;
  const double* dmsc;
  __device__ __forceinline__ float scale() const { return dmsc ? (float)dmsc[0] : msc; }
};
template <bool SRC64>
__device__ __forceinline__ typename SrcT<SRC64>::type load_src(const SrcRange& r, float msc, int j,
                                                               const double* __restrict__ x,
                                                               const double* __restrict__ m) {
  const int jj = min(j, r.n - 1);  // loads at a clamped index, so none waits for a branch
  const double px = x[jj], py = x[r.n + jj], pz = x[2 * r.n + jj];
  const float mj = (float)m[jj] * msc;
  const bool in = j >= r.lower && j < r.upper;
  return j < r.n ? SrcT<SRC64>::make(px, py, pz, in ? mj : 0.f) : SrcT<SRC64>::make(0.0, 0.0, 0.0, 0.f);
}

template <bool SRC64>
__global__ __launch_bounds__(256) void k_src(SrcRange r, int npad, const double* __restrict__ x,
                                             const double* __restrict__ m,
                                             typename SrcT<SRC64>::type* __restrict__ src) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < npad) src[i] = load_src<SRC64>(r, r.scale(), i, x, m);
}

// One target per lane.
template <bool MASK, bool SRC64>
struct PairSums {
  double px, py, pz;
  float fx, fy, fz;
  __device__ __forceinline__ void target(const double* __restrict__ x, int n, int i) {
    px = x[i];
    py = x[n + i];
    pz = x[2 * n + i];
    fx = (float)px;
    fy = (float)py;
    fz = (float)pz;
  }
  // Adds the pull of source q to t.
  __device__ __forceinline__ void pair(const typename SrcT<SRC64>::type& q, float eps2, float* t) const {
    float dx, dy, dz;
    if (SRC64) {
      dx = (float)(q.x - px);
      dy = (float)(q.y - py);
      dz = (float)(q.z - pz);
    } else {
      dx = q.x - fx;
      dy = q.y - fy;
      dz = q.z - fz;
    }
    float r2 = fmaf(dx, dx, eps2);
    r2 = fmaf(dy, dy, r2);
    r2 = fmaf(dz, dz, r2);
    float inv = __builtin_amdgcn_rsqf(r2);
    if (MASK) inv = (r2 > 0.f) ? inv : 0.f;
    const float inv2 = inv * inv;
    const float f = (src_mass(q) * inv) * inv2;
    t[0] = fmaf(f, dx, t[0]);
    t[1] = fmaf(f, dy, t[1]);
    t[2] = fmaf(f, dz, t[2]);
  }
};

// The FP32 sums of one tile of sources in LDS.
template <class P, class T>
__device__ __forceinline__ void tile_sums(const P& ps, const T* __restrict__ src, float eps2, float* t) {
  t[0] = t[1] = t[2] = 0.f;
  // The next kB sources are read before the sums over the present ones, and
  // kept there: left alone, the compiler reads each right before its use and
  // waits for LDS every time (leapfrog step at n = 1000, mixed: 9.1 -> 7.5 us).
  // kB = 4 needs twice the registers and loses where many waves share a SIMD
  // (n = 16384: 120 -> 135 us).
  constexpr int kB = 2;
  T q[kB], next[kB];
#pragma unroll
  for (int u = 0; u < kB; ++u) q[u] = src[u];
#pragma unroll 4
  for (int j = 0; j < kApTile; j += kB) {
#pragma unroll
    for (int u = 0; u < kB; ++u) next[u] = src[min(j + kB, kApTile - kB) + u];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kB; ++u) ps.pair(q[u], eps2, t);
#pragma unroll
    for (int u = 0; u < kB; ++u) {
      hold_pad(q[u]);
      q[u] = next[u];
    }
  }
}

// One target per lane (natural order), sources [s*slice_len, ...) of the
// padded source array; out: [S][3][n] doubles.
template <int ACC, bool MASK, bool SRC64>
__global__ __launch_bounds__(256) void k_allpairs_f32(const typename SrcT<SRC64>::type* __restrict__ src,
                                                      const double* __restrict__ x, int n, int npad, int slice_len,
                                                      float eps2, double* __restrict__ out) {
  const int i = blockIdx.x * kApBlock + threadIdx.x;
  const int jb = blockIdx.y * slice_len;
  const int je = min(jb + slice_len, npad);
  PairSums<MASK, SRC64> p;
  p.target(x, n, i < n ? i : n - 1);
  float s[3] = {0.f, 0.f, 0.f}, cmp[3] = {0.f, 0.f, 0.f};
  for (int t = jb; t < je; t += kApTile) {
    float ts[3] = {0.f, 0.f, 0.f};
#pragma unroll 16
    for (int k = 0; k < kApTile; ++k) p.pair(src[t + k], eps2, ACC == ACC_TILE_KAHAN ? ts : s);
    if (ACC == ACC_TILE_KAHAN)
#pragma unroll
      for (int c = 0; c < 3; ++c) kahan_add32(s[c], cmp[c], ts[c]);
  }
  if (i < n) {
    double* o = out + (size_t)blockIdx.y * 3 * n;
#pragma unroll
    for (int c = 0; c < 3; ++c) o[(size_t)c * n + i] = (double)s[c] - (double)cmp[c];
  }
}

// Small and middle-sized problems: sources in LDS, the tiles of a slice spread
// over the waves of a block. A block owns 64 / GR targets. Its W worker waves
// take GR 64-source tiles each per round: lane group g of 64 / GR lanes sums
// tile GR w + g for its targets. A wave stages its tiles through LDS by itself
// (the next round's sources are loaded during the sums) and leaves the tile
// sums there; one more wave takes them in tile order, Kahan-compensated within
// each slice, the slices in FP64: the bits of k_allpairs_f32 and k_combine with
// the same slices (plain method: the tile sums are added in FP64, where
// k_allpairs_f32 carries one FP32 sum through the slice).
// With GR = 4 even 1000 bodies occupy some hundred SIMDs, a block takes every
// source and the last wave applies the integrator's update too, so a step is
// one launch; the positions then go to a second buffer, since other blocks
// still read them. With f.part block row y takes slice y and writes its sums
// for k_combine. Bound: launch and one tile's latency at n = 1000 (7.5 us a
// step, mixed), VALU issue and LDS reads (32 bytes per source and wave) above.
struct TileSpan {
  int j0, tiles, slice_tiles;  // first source, number of tiles, tiles per slice
};
struct Finish {
  double* part;      // slice sums [S][3][n] (the rest unused), or null:
  const double* pn;  // FP64 post-Newtonian part, may be null
  double G;          // result scale, or read from the device where dG is given
  const double* dG;
  double* a;         // SoA planes, or AoS-d3 if aos
  int aos;
  StepPost post;
  double* x_out;
  double* v;
  uint32_t* flags;
};

template <int W, int GR, bool MASK, bool SRC64>
__global__ __launch_bounds__(64 * (W + 1)) void k_allpairs_tiles(SrcRange r, const double* __restrict__ x,
                                                                 const double* __restrict__ m, TileSpan sp,
                                                                 float eps2, Finish f) {
  constexpr int TG = 64 / GR;              // targets of the block, lanes of a group
  constexpr int R = GR * W;                // tiles per round
  constexpr int NC = (3 * TG + 63) / 64;   // sums per lane of the last wave
  constexpr int ACC = SRC64 ? ACC_TILE_KAHAN : ACC_PLAIN;
  // a tile's records end on another bank than they begin on, so the lane
  // groups read different banks
  __shared__ typename SrcT<SRC64>::type tiles[W][GR][kApTile + 1];
  __shared__ float sums[2][R][3][TG];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = r.n, i0 = blockIdx.x * TG;
  if (f.part) {  // this block's slice
    const int t0 = blockIdx.y * sp.slice_tiles;
    sp.j0 += t0 * kApTile;
    sp.tiles = min(sp.slice_tiles, sp.tiles - t0);
  }
  const int rounds = (sp.tiles + R - 1) / R;
  if (w < W) {
    const int ti = lane % TG, g = lane / TG;
    const float msc = r.scale();
    typename SrcT<SRC64>::type q[GR];
    auto fetch = [&](int rd) {
#pragma unroll
      for (int p = 0; p < GR; ++p)
        q[p] = load_src<SRC64>(r, msc, sp.j0 + (rd * R + GR * w + p) * kApTile + lane, x, m);
    };
    fetch(0);
    PairSums<MASK, SRC64> ps;
    ps.target(x, n, min(i0 + ti, n - 1));
    for (int rd = 0; rd < rounds; ++rd) {
      if (rd * R + GR * w < sp.tiles) {  // wave-uniform
        wave_sync();                     // the wave is done with its previous tiles
#pragma unroll
        for (int p = 0; p < GR; ++p) tiles[w][p][lane] = q[p];
        wave_sync();
        if (rd + 1 < rounds) fetch(rd + 1);
        float t[3];
        tile_sums(ps, tiles[w][g], eps2, t);
#pragma unroll
        for (int c = 0; c < 3; ++c) sums[rd & 1][GR * w + g][c][ti] = t[c];
      }
      __syncthreads();  // the sums of this round are there, those of the round before are taken
    }
    return;
  }
  double xs[NC], vs[NC], tot[NC];
  float s[NC], cmp[NC];
#pragma unroll
  for (int h = 0; h < NC; ++h) {
    const int ch = lane + 64 * h, c = ch / TG, i = min(i0 + ch % TG, n - 1);
    tot[h] = 0.0;
    s[h] = cmp[h] = 0.f;
    xs[h] = vs[h] = 0.0;
    if (f.post.kind != POST_NONE && c < 3) {
      xs[h] = x[(size_t)c * n + i];
      vs[h] = f.v[(size_t)c * n + i];
    }
  }
  int left = sp.slice_tiles;  // tiles to the end of the slice
  for (int rd = 0; rd < rounds; ++rd) {
    __syncthreads();
    const int cnt = min(R, sp.tiles - rd * R);
    for (int k = 0; k < cnt; ++k) {
      const bool end = --left == 0 || (rd + 1 == rounds && k + 1 == cnt);
#pragma unroll
      for (int h = 0; h < NC; ++h) {
        const int ch = min(lane + 64 * h, 3 * TG - 1);
        const float t = (&sums[rd & 1][k][0][0])[ch];
        if (ACC == ACC_TILE_KAHAN) {
          kahan_add32(s[h], cmp[h], t);
          if (end) {
            tot[h] += (double)s[h] - (double)cmp[h];
            s[h] = cmp[h] = 0.f;
          }
        } else {
          tot[h] += (double)t;
        }
      }
      if (end) left = sp.slice_tiles;
    }
  }
  const double G = f.dG ? f.dG[0] : f.G;
#pragma unroll
  for (int h = 0; h < NC; ++h) {
    const int ch = lane + 64 * h, c = ch / TG, i = i0 + ch % TG;
    if (c >= 3 || i >= n) continue;
    const size_t k = (size_t)c * n + i;
    if (f.part) {
      f.part[(size_t)blockIdx.y * 3 * n + k] = tot[h];
      continue;
    }
    double acc = G * tot[h];
    if (f.pn) acc += f.pn[k];
    f.a[f.aos ? 3 * (size_t)i + c : k] = acc;
    if (f.post.kind == POST_KICK) f.v[k] = kick_1(vs[h], acc, f.post.dt);
    if (f.post.kind == POST_KICK_DRIFT || f.post.kind == POST_SABA) {
      if (f.post.kind == POST_KICK_DRIFT) kick_drift_1(xs[h], vs[h], acc, f.post.dt_prev, f.post.dt);
      else saba_1(xs[h], vs[h], acc, f.post.d, f.post.cd, f.post.cd_next, f.post.dt);
      f.x_out[k] = xs[h];
      f.v[k] = vs[h];
      if (!(isfinite(xs[h]) && isfinite(vs[h]))) atomicOr(f.flags, (uint32_t)FLAG_NONFINITE);
    }
  }
}

// Sum S slice partials (and the optional FP64 1PN term) in slice order, then
// scale by G (times the mass scale's 2^k): a[c][i] = G * sum_s part[s][c][i]
// + pn[c][i]. POST then applies the integrator's next update of this body
// (StepPost) with the acceleration still in registers, the arithmetic of
// k_kick_drift, k_kick and k_saba_stage, and after a drift the body's source
// record of the next evaluation (src, may be null): between two evaluations
// of a step sequence one launch instead of three, of about 4.6 us each.
template <int POST, bool SRC64>
__global__ __launch_bounds__(256) void k_combine(int n, int npad, int S, const double* __restrict__ part,
                                                 const double* __restrict__ pn, double G, double* __restrict__ a,
                                                 StepPost post, double* __restrict__ x, double* __restrict__ v,
                                                 const double* __restrict__ m, SrcRange r,
                                                 typename SrcT<SRC64>::type* __restrict__ src,
                                                 uint32_t* __restrict__ flags) {
  constexpr bool kDrifts = POST == POST_KICK_DRIFT || POST == POST_SABA;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) {
    if (kDrifts && src && i < npad) src[i] = SrcT<SRC64>::make(0.0, 0.0, 0.0, 0.f);
    return;
  }
  double xs[3], vs[3];
  if (POST != POST_NONE)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if (kDrifts) xs[c] = x[(size_t)c * n + i];
      vs[c] = v[(size_t)c * n + i];
    }
  // 8 slices per round, their 24 loads issued before the first add (clamped
  // slice index); the adds stay in slice order
  double s[3] = {0.0, 0.0, 0.0};
  for (int k0 = 0; k0 < S; k0 += 8) {
    double w[8][3];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int k = min(k0 + u, S - 1);
#pragma unroll
      for (int c = 0; c < 3; ++c) w[u][c] = part[((size_t)k * 3 + c) * n + i];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (k0 + u < S)
#pragma unroll
        for (int c = 0; c < 3; ++c) s[c] += w[u][c];
  }
  bool finite = true;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const size_t k = (size_t)c * n + i;
    double acc = G * s[c];
    if (pn) acc += pn[k];
    a[k] = acc;
    if (POST == POST_KICK) v[k] = kick_1(vs[c], acc, post.dt);
    if (kDrifts) {
      if (POST == POST_KICK_DRIFT) kick_drift_1(xs[c], vs[c], acc, post.dt_prev, post.dt);
      else saba_1(xs[c], vs[c], acc, post.d, post.cd, post.cd_next, post.dt);
      x[k] = xs[c];
      v[k] = vs[c];
      finite = finite && isfinite(xs[c]) && isfinite(vs[c]);
    }
  }
  if (kDrifts) {
    if (!finite) atomicOr(flags, (uint32_t)FLAG_NONFINITE);
    if (src) {
      const bool in = i >= r.lower && i < r.upper;
      src[i] = SrcT<SRC64>::make(xs[0], xs[1], xs[2], in ? (float)m[i] * r.scale() : 0.f);
    }
  }
}

// ---------------------------------------------------------------- FP64 ----

// FP64 accelerations in the reference's arithmetic and order: for target i,
// sum over sources j in [lower, upper), j != i, in j order, of f/m_i with f =
// compute_gravitational (Parallelized::compute_forces,
// src/utils/builder_endpoint.cpp:729-757; tool_chain_impl.cpp:120-137), IEEE
// division and square root, no contraction. MODE 0: Newton (+ the
// post-Newtonian terms pnf selects if PN); MODE 1: only the post-Newtonian
// terms (added to an FP32 Newtonian result). x, v: SoA planes [3][n]; ic = 1/c.
//
// Every target's sum is one dependent chain over its sources; the pair
// contributions are independent. A block owns 16 targets and walks the sources
// in chunks of 64, one per lane: its 8 worker waves form the chunk's
// contributions f/m_i for two targets each (the targets' values are uniform,
// the next chunk's sources load during the arithmetic) and put them in LDS
// rows, one per target and coordinate; a ninth wave adds the chunk before, one
// row per lane, in j order. A contribution that does not count (the target's
// own, sources past upper) is written as 0: adding +0 changes no sum that
// began at +0, so every sum has the bits of a sequential loop.
// Bound: FP64 issue (45 FP64 instructions and a v_rsq_f64 per pair, 57 VALU in
// all, the adding wave's share included); few bodies: the adding wave's chain.
// Per evaluation, against 256 threads that formed a chunk with IEEE square
// root and division and then waited for 16 of them to add it (above 32768
// bodies: one target per lane): n = 1000 70 -> 16 us, 4096 264 -> 55 us, 16384
// 1.89 -> 0.64 ms, 65536 15.4 -> 9.2 ms; with the 1PN term 79 -> 31 us, 297 ->
// 114 us, 2.60 -> 1.78 ms, 31.6 -> 28.1 ms.
//
// The adding wave then applies the integrator's update (StepPost) to its
// targets; positions go to a second buffer, since other blocks still read them
// as sources. A launch less per step: 64 bodies
// 7.3 -> 4.8 us, 1000 20.0 -> 17.2, 4096 58.5 -> 56.0 (SABA4 235.8 -> 223.3),
// 16384 650 -> 639.
struct Update64 {
  StepPost post;
  double* x_out;
  double* v;
  uint32_t* flags;
};
constexpr int kF64Chunk = 64;

template <int W, int kPer, bool PN, int MODE>
__global__ __launch_bounds__(64 * (W + 1)) void k_allpairs_f64(int n, int lower, int upper,
                                                                        const double* __restrict__ x,
                                                                        const double* __restrict__ v,
                                                                        const double* __restrict__ m, double G,
                                                                        double ic, int pnf, double soft,
                                                                        double* __restrict__ a, Update64 up) {
#pragma clang fp contract(off)
  constexpr int kF64Targets = W * kPer;
  static_assert(3 * kF64Targets <= 64, "one row per lane of the adding wave");
  // rows start on different banks (16-byte reads of the adding wave)
  __shared__ double cf[2][3 * kF64Targets][kF64Chunk + 2];
  __shared__ int in_range[2][W];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = blockIdx.x * kF64Targets;
  const int chunks = (upper - lower + kF64Chunk - 1) / kF64Chunk;
  if (w < W) {
    double p1x[kPer], p1y[kPer], p1z[kPer], v1x[kPer], v1y[kPer], v1z[kPer];
    Divisor64 m1[kPer];
    bool range1 = law_in_range64(G, soft);
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
      const int i = min(i0 + w * kPer + q, n - 1);
      p1x[q] = x[i];
      p1y[q] = x[n + i];
      p1z[q] = x[2 * n + i];
      m1[q] = divisor64(m[i]);
      v1x[q] = PN ? v[i] : 0.0;
      v1y[q] = PN ? v[n + i] : 0.0;
      v1z[q] = PN ? v[2 * n + i] : 0.0;
      range1 = range1 && coord_in_range64(p1x[q]) && coord_in_range64(p1y[q]) && coord_in_range64(p1z[q]) &&
               mass_in_range64(m1[q].b);
    }
    // byte offsets of 32 bits from uniform plane addresses (n <= 2^28)
    auto at = [](const double* plane, uint32_t off) {
      return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(plane) + off);
    };
    const double *xp = x, *yp = x + n, *zp = x + 2 * (size_t)n;
    const uint32_t last = 8u * (uint32_t)(upper - 1);
    auto chunk_off = [&](int ch) { return min(8u * (uint32_t)(lower + ch * kF64Chunk + lane), last); };
    double sx, sy, sz, sm, svx = 0.0, svy = 0.0, svz = 0.0;
    auto fetch = [&](int ch) {
      const uint32_t o = chunk_off(ch);
      sx = at(xp, o);
      sy = at(yp, o);
      sz = at(zp, o);
      sm = at(m, o);
      if (PN) {
        svx = at(v, o);
        svy = at(v + n, o);
        svz = at(v + 2 * (size_t)n, o);
      }
    };
    // Each worker looks at the range of one chunk's sources of the next W and
    // leaves the verdict in LDS.
    double cx, cy, cz, cm;
    auto check_fetch = [&](int group) {
      const uint32_t o = chunk_off(min(group * W + w, chunks - 1));
      cx = at(xp, o);
      cy = at(yp, o);
      cz = at(zp, o);
      cm = at(m, o);
    };
    auto check_leave = [&](int group) {
      const bool ok = __all(coord_in_range64(cx) && coord_in_range64(cy) && coord_in_range64(cz) && mass_in_range64(cm));
      if (lane == 0) in_range[group & 1][w] = ok ? 1 : 0;
    };
    if (chunks > 0) {
      check_fetch(0);
      fetch(0);
      check_leave(0);
      check_fetch(1);
    }
    __syncthreads();
    for (int ch = 0; ch < chunks; ++ch) {
      const double p2x = sx, p2y = sy, p2z = sz, m2 = sm, v2x = svx, v2y = svy, v2z = svz;
      if (ch + 1 < chunks) fetch(ch + 1);
      const int jb = lower + ch * kF64Chunk;
      const int group = ch / W;
      const bool fast = range1 && __builtin_amdgcn_readfirstlane(in_range[group & 1][ch % W]) != 0;
      if (ch % W == 0) {  // the next group's verdicts, seen after this chunk's barrier
        check_leave(group + 1);
        check_fetch(group + 2);
      }
      // one straight stretch of code for the targets of a wave, so that their
      // chains overlap
      auto chunk = [&](auto fast_tag) {
        constexpr bool FAST = decltype(fast_tag)::value;
        double dx[kPer], dy[kPer], dz[kPer], r2[kPer], inv_r[kPer], f[kPer][3];
        bool odd = false, fdiv = FAST;
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
          dx[q] = p2x - p1x[q];
          dy[q] = p2y - p1y[q];
          dz[q] = p2z - p1z[q];
          r2[q] = dx[q] * dx[q] + dy[q] * dy[q] + dz[q] * dz[q] + soft;
        }
        if (FAST)
          odd = inv_sqrt64_fast<kPer>(r2, inv_r);
        else
#pragma unroll
          for (int q = 0; q < kPer; ++q) inv_r[q] = 1.0 / sqrt(r2[q]);
        if (FAST && __builtin_expect(__any(odd), 0)) {
#pragma unroll
          for (int q = 0; q < kPer; ++q) inv_r[q] = 1.0 / sqrt(r2[q]);
        }
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
          const double inv_r2 = inv_r[q] * inv_r[q];
          const double nx = dx[q] * inv_r[q], ny = dy[q] * inv_r[q], nz = dz[q] * inv_r[q];
          f[q][0] = f[q][1] = f[q][2] = 0.0;
          if (MODE == 0) {
            const double scal = G * m2 * m1[q].b * inv_r2;
            f[q][0] = nx * scal;
            f[q][1] = ny * scal;
            f[q][2] = nz * scal;
          }
          if (PN) {
            pn_add64(pnf, m1[q].b, m2, v1x[q], v1y[q], v1z[q], v2x, v2y, v2z, inv_r[q], -nx, -ny, -nz, G, ic, f[q][0], f[q][1],
                     f[q][2]);
            // the post-Newtonian terms have no bounds of their own
            fdiv = fdiv && zero_or_within64(f[q][0], 1023 - 800, 1023 + 800) &&
                   zero_or_within64(f[q][1], 1023 - 800, 1023 + 800) && zero_or_within64(f[q][2], 1023 - 800, 1023 + 800);
          }
        }
        if (FAST && (!PN || __all(fdiv))) {
#pragma unroll
          for (int q = 0; q < kPer; ++q) div64_fast<3>(f[q], m1[q]);
        } else {
#pragma unroll
          for (int q = 0; q < kPer; ++q) {
            f[q][0] = f[q][0] / m1[q].b;
            f[q][1] = f[q][1] / m1[q].b;
            f[q][2] = f[q][2] / m1[q].b;
          }
        }
#pragma unroll
        for (int q = 0; q < kPer; ++q) {
          const int t = w * kPer + q, i = i0 + t;
          if (jb + kF64Chunk > upper || (i >= jb && i < jb + kF64Chunk)) {  // wave-uniform
            const bool take = jb + lane < upper && jb + lane != i;
            f[q][0] = take ? f[q][0] : 0.0;
            f[q][1] = take ? f[q][1] : 0.0;
            f[q][2] = take ? f[q][2] : 0.0;
          }
          cf[ch & 1][t][lane] = f[q][0];
          cf[ch & 1][kF64Targets + t][lane] = f[q][1];
          cf[ch & 1][2 * kF64Targets + t][lane] = f[q][2];
        }
      };
      if (fast) chunk(std::true_type{});
      else chunk(std::false_type{});
      __syncthreads();  // this chunk's contributions are there, the chunk before is added
    }
    return;
  }
  const int row = min(lane, 3 * kF64Targets - 1);
  const int i = i0 + row % kF64Targets;
  const size_t k = (size_t)(row / kF64Targets) * n + min(i, n - 1);
  double acc = 0.0, xt = 0.0, vt = 0.0;
  if (!PN && up.post.kind != POST_NONE) {
    xt = x[k];
    vt = up.v[k];
  }
  __syncthreads();
  for (int ch = 0; ch < chunks; ++ch) {
    __syncthreads();
    const double2* __restrict__ c = reinterpret_cast<const double2*>(cf[ch & 1][row]);
    constexpr int kB = 8;  // values read ahead of the adds, and kept there
    double2 d[kB], next[kB];
#pragma unroll
    for (int u = 0; u < kB; ++u) d[u] = c[u];
#pragma unroll
    for (int s = 0; s < kF64Chunk / 2; s += kB) {
#pragma unroll
      for (int u = 0; u < kB; ++u) next[u] = c[min(s + kB, kF64Chunk / 2 - kB) + u];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        acc += d[u].x;
        acc += d[u].y;
        d[u] = next[u];
      }
    }
  }
  if (lane >= 3 * kF64Targets || i >= n) return;
  a[k] = acc;
  if (PN || up.post.kind == POST_NONE) return;
  if (up.post.kind == POST_KICK) {
    up.v[k] = kick_1(vt, acc, up.post.dt);
    return;
  }
  if (up.post.kind == POST_KICK_DRIFT) kick_drift_1(xt, vt, acc, up.post.dt_prev, up.post.dt);
  else saba_1(xt, vt, acc, up.post.d, up.post.cd, up.post.cd_next, up.post.dt);
  up.x_out[k] = xt;
  up.v[k] = vt;
  if (!(isfinite(xt) && isfinite(vt))) atomicOr(up.flags, (uint32_t)FLAG_NONFINITE);
}

// ----------------------------------------------------------------- EIH ----
//
// Einstein-Infeld-Hoffmann 1PN accelerations (harmonic gauge) in the form of
// Newhall, Standish & Williams (1983, A&A 125, 150, eq. 1) with beta = gamma
// = 1, mu = G m, r from the softened r^2 = d.d + softening:
//   a_i = sum_{j != i} mu_j d_ij / r^3 [1 - (4 phi_i + phi_j)/c^2
//           + (v_i^2 + 2 v_j^2 - 4 v_i.v_j)/c^2 - 3/2 (d_ij.v_j / r)^2/c^2
//           + d_ij.aN_j / (2 c^2)]
//       + sum_{j != i} mu_j / (c^2 r^3) [-d_ij.(4 v_i - 3 v_j)] (v_i - v_j)
//       + 7/(2 c^2) sum_{j != i} mu_j aN_j / r
// with d_ij = x_j - x_i, phi_i = sum_{k != i} mu_k / r_ik and aN the
// Newtonian accelerations. For two bodies it is the pairwise 1PN law.
// Pass 1 forms phi and aN, pass 2 the accelerations; one thread per body,
// sources in index order (the oracle's order, so the two agree bit for bit). One
// wavefront per SIMD at most below 65536 bodies: inv_sqrt64, whose range check
// ends the overlap of the unrolled pairs, was slower (leapfrog step of 2000 bodies,
// two evaluations, 3.01 -> 3.20 ms).
__global__ __launch_bounds__(256) void k_eih_pass1(int n, const double* __restrict__ x, const double* __restrict__ m,
                                                   double G, double soft, double* __restrict__ phi,
                                                   double* __restrict__ an) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double p1x = x[i], p1y = x[n + i], p1z = x[2 * n + i];
  double ph = 0.0, ax = 0.0, ay = 0.0, az = 0.0;
  for (int j = 0; j < n; ++j) {
    if (j == i) continue;
    const double dx = x[j] - p1x, dy = x[n + j] - p1y, dz = x[2 * n + j] - p1z;
    const double r2 = dx * dx + dy * dy + dz * dz + soft;
    const double inv_r = 1.0 / sqrt(r2);
    const double inv_r3 = inv_r * inv_r * inv_r;
    const double mu = G * m[j];
    ph += mu * inv_r;
    ax += mu * dx * inv_r3;
    ay += mu * dy * inv_r3;
    az += mu * dz * inv_r3;
  }
  phi[i] = ph;
  an[i] = ax;
  an[n + i] = ay;
  an[2 * n + i] = az;
}

__global__ __launch_bounds__(256) void k_eih_pass2(int n, const double* __restrict__ x, const double* __restrict__ v,
                                                   const double* __restrict__ m, double G, double ic, double soft,
                                                   const double* __restrict__ phi, const double* __restrict__ an,
                                                   double* __restrict__ a) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double ic2 = ic * ic;
  const double p1x = x[i], p1y = x[n + i], p1z = x[2 * n + i];
  const double v1x = v[i], v1y = v[n + i], v1z = v[2 * n + i];
  const double vi2 = v1x * v1x + v1y * v1y + v1z * v1z;
  const double phi_i = phi[i];
  double ax = 0.0, ay = 0.0, az = 0.0;
  for (int j = 0; j < n; ++j) {
    if (j == i) continue;
    const double dx = x[j] - p1x, dy = x[n + j] - p1y, dz = x[2 * n + j] - p1z;
    const double r2 = dx * dx + dy * dy + dz * dz + soft;
    const double inv_r = 1.0 / sqrt(r2);
    const double inv_r3 = inv_r * inv_r * inv_r;
    const double mu = G * m[j];
    const double v2x = v[j], v2y = v[n + j], v2z = v[2 * n + j];
    const double anx = an[j], any = an[n + j], anz = an[2 * n + j];
    const double vj2 = v2x * v2x + v2y * v2y + v2z * v2z;
    const double vij = v1x * v2x + v1y * v2y + v1z * v2z;
    const double rv = (dx * v2x + dy * v2y + dz * v2z) * inv_r;
    const double dan = dx * anx + dy * any + dz * anz;
    const double B = 1.0 - (4.0 * phi_i + phi[j]) * ic2 + (vi2 + 2.0 * vj2 - 4.0 * vij) * ic2 -
                     1.5 * (rv * rv) * ic2 + 0.5 * dan * ic2;
    const double s1 = mu * inv_r3 * B;
    const double w = -(dx * (4.0 * v1x - 3.0 * v2x) + dy * (4.0 * v1y - 3.0 * v2y) + dz * (4.0 * v1z - 3.0 * v2z));
    const double s2 = mu * inv_r3 * ic2 * w;
    const double s3 = 3.5 * mu * inv_r * ic2;
    ax += dx * s1;
    ax += (v1x - v2x) * s2;
    ax += anx * s3;
    ay += dy * s1;
    ay += (v1y - v2y) * s2;
    ay += any * s3;
    az += dz * s1;
    az += (v1z - v2z) * s2;
    az += anz * s3;
  }
  a[i] = ax;
  a[n + i] = ay;
  a[2 * n + i] = az;
}

// --------------------------------------------------------------- launch ----

template <int W, int PER>
static void launch_allpairs_f64_as(aster_ctx* c, bool pn, int mode, int n, int lower, int upper, double ic, int pnf,
                                   double* out, const Update64& up) {
  auto k = mode == 1 ? k_allpairs_f64<W, PER, true, 1>
                     : pn ? k_allpairs_f64<W, PER, true, 0> : k_allpairs_f64<W, PER, false, 0>;
  const int targets = W * PER;
  hipLaunchKernelGGL(k, dim3((n + targets - 1) / targets), dim3(64 * (W + 1)), 0, c->stream, n, lower, upper, c->x.p,
                     c->v.p, c->m.p, c->P.G, ic, pnf, c->P.softening, out, up);
}

// 16 targets a block fill the 256 CUs once at 4096 bodies and twice at 8192;
// seven workers and the adding wave load the four SIMDs evenly, which counts
// with many blocks: 8 and 7 workers ran 55 and 80 us at n = 4096, 165 and 205 at
// 8192, 797 and 672 at 16384, 10.9 and 9.9 ms at 65536 (with the 1PN term 28.5
// and 33.3 ms), both before the division took four steps instead of five.
static int launch_allpairs_f64(aster_ctx* c, bool pn, int mode, int n, int lower, int upper, double ic, int pnf,
                               double* out, const Update64& up = Update64{}) {
  if (pn || n <= 8192) launch_allpairs_f64_as<8, 2>(c, pn, mode, n, lower, upper, ic, pnf, out, up);
  else launch_allpairs_f64_as<7, 2>(c, pn, mode, n, lower, upper, ic, pnf, out, up);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

// Source slices for `target` waves of target-slice work over the 1024 SIMDs,
// each slice at least 1024 sources, at most 64 slices.
static int split_for_waves(int64_t npad, int64_t target) {
  const int64_t waves = npad / 64;
  int64_t S = (target + waves - 1) / waves;
  const int64_t max_by_len = npad / 1024;
  if (S > max_by_len) S = max_by_len;
  if (S < 1) S = 1;
  if (S > 64) S = 64;
  return (int)S;
}

// About 64 waves per SIMD. Measured against 8 per SIMD (the FP32 kernels,
// FP64 slice partials and their combine included): n = 65536 plain 1.41 ->
// 1.16 ms, mixed 1.99 -> 1.49 ms, adjoint backward kernel 3.73 -> 3.19 ms;
// n = 262144 plain 20.1 -> 17.5 ms, mixed 28.3 -> 22.4 ms. Shorter slices keep
// a wavefront's sources, read through the scalar cache, shared by more of
// the waves on a CU.
int default_split(int64_t npad) { return split_for_waves(npad, 64 * 1024); }

// The allocation-free entry point keeps about 8 waves per SIMD, which bounds
// its slice partials (S n) for a static scratch array of modest size.
static int noalloc_split(int64_t npad) { return split_for_waves(npad, 8 * 1024); }

// Slices of a span of sources (a multiple of kApTile) for the FP32 kernels:
// the requested count, at least 1024 sources each, rounded to whole tiles.
static void slice_span(int span, int requested, int* S, int* slice) {
  int s = requested;
  if ((int64_t)s * 1024 > span) s = std::max(1, span / 1024);
  const int64_t sl = round_up((span + s - 1) / s, kApTile);
  *slice = (int)sl;
  *S = (int)((span + sl - 1) / sl);
}

int choose_split(aster_ctx* c) {
  if (c->P.split > 0) return c->P.split;
  return default_split(c->npad);
}

int fp32_scales(aster_ctx* c, Fp32Scales* sc) {
  double M = 0.0, R = 0.0;
  int rc = total_mass(c, &M, &R);
  if (rc) return rc;
  const float e2 = (float)c->P.softening;
  sc->mask = !(e2 >= FLT_MIN);
  sc->eps2 = sc->mask ? 0.f : e2;
  const int k = fp32_mass_shift(M, R, sc->eps2, sc->mask);
  if (k > kMaxMassShift)
    return fail(c, ASTER_ERR_INVALID,
                "masses and softening are beyond the FP32 force range (use an FP64 method or a larger softening)");
  sc->msc = std::ldexp(1.0f, -k);
  sc->gsc = std::ldexp(c->P.G, k);
  return ASTER_OK;
}

// Which kernel takes n bodies. A leapfrog step in us, before (k_allpairs_f32,
// its sources, combine and update in launches of their own) / one launch, GR =
// 4 / k_allpairs_tiles by slices, GR = 1 / k_allpairs_f32, two launches. Mixed:
// n = 1000 156 / 7.5 / - / 152, 4096 159 / 15.2 / 19.2 / 156, 8192 158 / 47 / 37
// / 155, 16384 164 / 175 / 120 / 160, 20011 200 / 270 / 178 / 192, 32768 437 /
// 684 / 433 / 434, 65536 1453 / 2698 / 1712 / 1449. Plain: 1000 93 / 6.3 / - /
// 90, 4096 95 / 11.6 / 16.9 / 89, 8192 92 / 30 / 28 / 93, 16384 110 / 130 / 85 /
// 106, 20011 165 / 164 / 129 / 160, 32768 322 / 447 / 311 / 318, 65536 1135 /
// 1699 / 1211 / 1127. One launch fills the 256 CUs once up to 4096 bodies (16
// targets a block); above the line the scalar reads, which take no LDS bandwidth,
// hide their latency behind enough waves: k_allpairs_f32 against tiles by slices,
// mixed 24000 286 / 251, 26000 312 / 287, 28000 330 / 333, 30000 358 / 378, 31610
// 407 / 420; plain 28000 250 / 240, 32768 319 / 310.
static bool one_launch(int64_t n) { return n <= 4096; }
template <bool SRC64>
static bool in_tiles(int64_t n) {
  return n <= (SRC64 ? 26624 : 32768);
}

template <int W, int GR, bool SRC64>
static void launch_tiles_as(hipStream_t st, bool mask, const SrcRange& r, const double* x, const double* m,
                            const TileSpan& sp, int S, float eps2, const Finish& f) {
  auto k = mask ? k_allpairs_tiles<W, GR, true, SRC64> : k_allpairs_tiles<W, GR, false, SRC64>;
  const int tg = 64 / GR;
  hipLaunchKernelGGL(k, dim3((r.n + tg - 1) / tg, f.part ? S : 1), dim3(64 * (W + 1)), 0, st, r, x, m, sp, eps2, f);
}

// One launch: W = 4 waves hold 16 tiles (1024 sources) in one round.
template <bool SRC64>
static void launch_tiles(hipStream_t st, bool mask, const SrcRange& r, const double* x, const double* m,
                         const TileSpan& sp, int S, float eps2, const Finish& f) {
  if (f.part) launch_tiles_as<4, 1, SRC64>(st, mask, r, x, m, sp, S, eps2, f);
  else if (sp.tiles <= 16) launch_tiles_as<4, 4, SRC64>(st, mask, r, x, m, sp, S, eps2, f);
  else launch_tiles_as<8, 4, SRC64>(st, mask, r, x, m, sp, S, eps2, f);
}

template <bool SRC64>
static void launch_slices(hipStream_t st, bool mask, int n, int npad, int S, int span, int slice, float eps2,
                          const double* x, const typename SrcT<SRC64>::type* src, double* out) {
  constexpr int ACC = SRC64 ? ACC_TILE_KAHAN : ACC_PLAIN;
  auto k = mask ? k_allpairs_f32<ACC, true, SRC64> : k_allpairs_f32<ACC, false, SRC64>;
  hipLaunchKernelGGL(k, dim3(npad / kApBlock, S), dim3(kApBlock), 0, st, src, x, n, span, slice, eps2, out);
}

// One FP32 evaluation and the update that follows: the FP64 post-Newtonian
// part, then one launch; or sources (unless left by the update before), pair
// sums over slices and the combine with the update.
template <bool SRC64>
static int allpairs_f32(aster_ctx* c, DBuf<typename SrcT<SRC64>::type>& srcbuf, int lower, int upper, int pnf,
                        const StepPost& post) {
  const int n = (int)c->n, npad = (int)c->npad;
  Fp32Scales sc;
  int rc = fp32_scales(c, &sc);
  if (rc) return rc;
  const SrcRange r{n, lower, upper, sc.msc, nullptr};
  // Slices over the tiles that hold the source range (sources outside it and
  // the padding bodies have zero mass); an empty range behind the last body
  // takes the last tile.
  const int j0 = std::min(lower, npad - 1) / kApTile * kApTile;
  const int span = std::max<int>(j0 + kApTile, (int)round_up(upper, kApTile)) - j0;
  int S = 0, slice = 0;
  slice_span(span, choose_split(c), &S, &slice);
  const bool drifts = post.kind == POST_KICK_DRIFT || post.kind == POST_SABA;
  const double* pnp = nullptr;
  if (pnf) {
    ASTER_HIP(c, c->apn.reserve((size_t)3 * n));
    if ((rc = launch_allpairs_f64(c, true, 1, n, lower, upper, 1.0 / c->P.c, pnf, c->apn.p))) return rc;
    pnp = c->apn.p;
  }
  const TileSpan sp{j0, span / kApTile, slice / kApTile};
  if (one_launch(n)) {
    if (drifts) ASTER_HIP(c, c->x_next.reserve((size_t)3 * n));
    const Finish f{nullptr, pnp, sc.gsc, nullptr, c->a.p, 0, post, c->x_next.p, c->v.p, c->flags.p};
    phase_begin(c, ASTER_PHASE_ALLPAIRS);
    launch_tiles<SRC64>(c->stream, sc.mask, r, c->x.p, c->m.p, sp, S, sc.eps2, f);
    ASTER_HIP(c, hipGetLastError());
    phase_end(c, ASTER_PHASE_ALLPAIRS);
    if (drifts) std::swap(c->x, c->x_next);
    return ASTER_OK;
  }
  ASTER_HIP(c, c->apart.reserve((size_t)S * 3 * n));
  typename SrcT<SRC64>::type* src = nullptr;
  const SrcReady want{c->x.p, c->n, SRC64 ? 2 : 1, lower, upper, sc.msc};
  const bool have = c->src_ready == want;
  c->src_ready = SrcReady{};
  if (in_tiles<SRC64>(n)) {
    Finish f{};
    f.part = c->apart.p;
    phase_begin(c, ASTER_PHASE_ALLPAIRS);
    launch_tiles<SRC64>(c->stream, sc.mask, r, c->x.p, c->m.p, sp, S, sc.eps2, f);
  } else {
    ASTER_HIP(c, srcbuf.reserve((size_t)npad));
    src = srcbuf.p;
    if (!have) {
      phase_begin(c, ASTER_PHASE_TILES);
      hipLaunchKernelGGL(k_src<SRC64>, dim3(npad / 256), dim3(256), 0, c->stream, r, npad, c->x.p, c->m.p, src);
      ASTER_HIP(c, hipGetLastError());
      phase_end(c, ASTER_PHASE_TILES);
    }
    phase_begin(c, ASTER_PHASE_ALLPAIRS);
    launch_slices<SRC64>(c->stream, sc.mask, n, npad, S, span, slice, sc.eps2, c->x.p, src + j0, c->apart.p);
  }
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_ALLPAIRS);
  phase_begin(c, ASTER_PHASE_COMBINE);
  auto k = k_combine<POST_NONE, SRC64>;
  if (post.kind == POST_KICK_DRIFT) k = k_combine<POST_KICK_DRIFT, SRC64>;
  else if (post.kind == POST_KICK) k = k_combine<POST_KICK, SRC64>;
  else if (post.kind == POST_SABA) k = k_combine<POST_SABA, SRC64>;
  hipLaunchKernelGGL(k, dim3(npad / 256), dim3(256), 0, c->stream, n, npad, S, (const double*)c->apart.p, pnp, sc.gsc,
                     c->a.p, post, c->x.p, c->v.p, (const double*)c->m.p, r, src, c->flags.p);
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_COMBINE);
  if (drifts && src) c->src_ready = want;
  return ASTER_OK;
}

int launch_allpairs(aster_ctx* c, int method, const StepPost& post) {
  const int n = (int)c->n;
  const int lower = c->P.lower < 0 ? 0 : c->P.lower;
  const int upper = (c->P.upper < 0 || c->P.upper > n) ? n : c->P.upper;
  if (lower > upper) return fail(c, ASTER_ERR_INVALID, "source bounds: lower > upper");
  const int pnf = c->P.pn_flags & ASTER_PN_TERMS;
  const bool pn = pnf != 0;
  const double ic = 1.0 / c->P.c;
  if (pnf & ASTER_EIH) {
    if (method != ASTER_ALLPAIRS_FP64) return fail(c, ASTER_ERR_INVALID, "ASTER_EIH needs ASTER_ALLPAIRS_FP64");
    if (lower != 0 || upper != n) return fail(c, ASTER_ERR_INVALID, "ASTER_EIH covers the full source range only");
    ASTER_HIP(c, c->apn.reserve((size_t)4 * n));
    double* an = c->apn.p;
    double* phi = c->apn.p + 3 * (size_t)n;
    const dim3 grid((n + 255) / 256);
    phase_begin(c, ASTER_PHASE_ALLPAIRS);
    hipLaunchKernelGGL(k_eih_pass1, grid, dim3(256), 0, c->stream, n, c->x.p, c->m.p, c->P.G, c->P.softening, phi, an);
    hipLaunchKernelGGL(k_eih_pass2, grid, dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->m.p, c->P.G, ic,
                       c->P.softening, (const double*)phi, (const double*)an, c->a.p);
    ASTER_HIP(c, hipGetLastError());
    phase_end(c, ASTER_PHASE_ALLPAIRS);
    return launch_post(c, post, false);
  }
  if (method == ASTER_ALLPAIRS_FP64) {
    // Velocity-dependent terms read every body's velocity; above 16384 bodies a
    // launch is under 1% of the evaluation and not worth a second buffer.
    const bool fused = !pn && n <= 16384 && post.kind != POST_NONE;
    const bool drifts = fused && post.kind != POST_KICK;
    Update64 up{};
    if (drifts) ASTER_HIP(c, c->x_next.reserve((size_t)3 * n));
    if (fused) up = Update64{post, c->x_next.p, c->v.p, c->flags.p};
    phase_begin(c, ASTER_PHASE_ALLPAIRS);
    if (const int e = launch_allpairs_f64(c, pn, 0, n, lower, upper, ic, pnf, c->a.p, up)) return e;
    phase_end(c, ASTER_PHASE_ALLPAIRS);
    if (drifts) {
      std::swap(c->x, c->x_next);
      c->box_parts = 0;
      c->src_ready = SrcReady{};
    }
    return fused ? ASTER_OK : launch_post(c, post, false);
  }
  if (method != ASTER_ALLPAIRS_FP32 && method != ASTER_ALLPAIRS_FP32_KAHAN)
    return fail(c, ASTER_ERR_INVALID, "unknown all-pairs method");
  if (method == ASTER_ALLPAIRS_FP32) return allpairs_f32<false>(c, c->sh, lower, upper, pnf, post);
  return allpairs_f32<true>(c, c->src64, lower, upper, pnf, post);
}

}  // namespace aster

// ------------------------------------------------------ allocation-free ----
//
// aster_forces_noalloc: the ASTER_ALLPAIRS_FP32_KAHAN evaluation (same
// kernels and mass scale as aster_forces; the source split of about 8 waves
// per SIMD, which aster_forces uses with aster_params.split set to it) on
// caller-owned device arrays, with no device allocation. Its working memory is the file-scope
// array `scratch` below: each GPU the library runs on holds one copy until
// the process ends, and every call on that GPU uses it, so calls that
// overlap on one GPU race. Nothing in it needs clearing: every call writes
// each word it reads first.
namespace aster {

constexpr int64_t kNaMax = ASTER_NOALLOC_MAX_BODIES;
static_assert(kNaMax % kApBlock == 0, "the body limit must be a whole number of all-pairs blocks");
// Bound on S n of noalloc_split over n <= kNaMax (the largest is 587520, at
// n = 65280 with S = 9).
constexpr int64_t kNaPartMax = 589824;
// Layout in doubles: SoA positions | double4 sources | slice partials |
// mass-sum partials | the two scales.
constexpr size_t kNaX = 0;
constexpr size_t kNaSrc = kNaX + 3 * kNaMax;
constexpr size_t kNaPart = kNaSrc + 4 * kNaMax;
constexpr size_t kNaRed = kNaPart + 3 * kNaPartMax;
constexpr size_t kNaScale = kNaRed + (size_t)kComQ * (kComBlocks + 1);
constexpr size_t kNaTotal = kNaScale + 2;

static __device__ __align__(256) double scratch[kNaTotal];

// AoS-d3 positions -> SoA planes.
__global__ __launch_bounds__(256) void k_na_planes(int n, const double* __restrict__ pos, double* __restrict__ x) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int c = 0; c < 3; ++c) x[(size_t)c * n + i] = pos[3 * (size_t)i + c];
}

// The mass scale of fp32_scales, formed on the device from the mass sums:
// scale[0] = 2^-k, scale[1] = G 2^k. k beyond the FP32 range is clamped (the
// result is then not finite; aster_forces reports an error instead).
__global__ void k_na_scales(const double* __restrict__ sums, float eps2, int mask, double G,
                            double* __restrict__ scale) {
  if (threadIdx.x != 0) return;
  int k = fp32_mass_shift(sums[0], sums[4], eps2, mask != 0);
  if (k > kMaxMassShift) k = kMaxMassShift;
  scale[0] = (double)ldexpf(1.0f, -k);
  scale[1] = ldexp(G, k);
}

// k_combine (no post-Newtonian term) writing AoS-d3.
__global__ void k_na_combine(int n, int S, const double* __restrict__ part, const double* __restrict__ scale,
                             double* __restrict__ acc) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const double G = scale[1];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double s = 0.0;
    for (int k = 0; k < S; ++k) s += part[((size_t)k * 3 + c) * n + i];
    acc[3 * (size_t)i + c] = G * s;
  }
}

constexpr int kNaMaxDevices = 64;
static std::mutex g_na_lock;
static double* g_na_ptr[kNaMaxDevices] = {};

// The device address of `scratch` on device `dev` (current), looked up once
// per device. In host code the array's name is only a stand-in: kernels get
// this address.
static hipError_t na_scratch(int dev, double** out) {
  std::lock_guard<std::mutex> guard(g_na_lock);
  if (!g_na_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_na_ptr[dev] = static_cast<double*>(p);
  }
  *out = g_na_ptr[dev];
  return hipSuccess;
}

static int na_fail(int code, const std::string& msg) {
  set_global_error(msg);
  return code;
}

}  // namespace aster

extern "C" int aster_forces_noalloc(int64_t n, const double* d_pos, const double* d_mass, double G, double softening,
                                    double* d_acc, void* stream) {
  using namespace aster;
  if (n < 1 || !d_pos || !d_mass || !d_acc)
    return na_fail(ASTER_ERR_INVALID, "aster_forces_noalloc: need n >= 1 and device positions, masses, output");
  if (n > kNaMax)
    return na_fail(ASTER_ERR_CAPACITY, "aster_forces_noalloc: at most ASTER_NOALLOC_MAX_BODIES bodies");
  if (!(softening >= 0.0) || !std::isfinite(G)) return na_fail(ASTER_ERR_INVALID, "invalid G or softening");
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return na_fail(ASTER_ERR_HIP, std::string("hipGetDevice: ") + hipGetErrorString(e));
  if (dev < 0 || dev >= kNaMaxDevices) return na_fail(ASTER_ERR_CAPACITY, "device index beyond 63");
  double* base = nullptr;
  if ((e = na_scratch(dev, &base)) != hipSuccess)
    return na_fail(ASTER_ERR_HIP, std::string("hipGetSymbolAddress: ") + hipGetErrorString(e));
  const int ni = (int)n;
  const int npad = (int)round_up(n, kApBlock);
  // the slicing of launch_allpairs over the full source range
  const int span = (int)round_up(n, kApTile);
  int S = 0, slice = 0;
  slice_span(span, noalloc_split(npad), &S, &slice);
  if ((int64_t)S * n > kNaPartMax) return na_fail(ASTER_ERR_CAPACITY, "slice partials beyond the scratch layout");
  double* x = base + kNaX;
  double4* src = reinterpret_cast<double4*>(base + kNaSrc);
  double* part = base + kNaPart;
  double* red = base + kNaRed;
  double* sums = red + (size_t)kComQ * kComBlocks;
  double* scale = base + kNaScale;
  const float e2 = (float)softening;
  const bool mask = !(e2 >= FLT_MIN);
  const float eps2 = mask ? 0.f : e2;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 b256(256), gn((ni + 255) / 256);
  const int rblocks = (int)std::min<int64_t>((n + 255) / 256, kComBlocks);
  hipLaunchKernelGGL(k_na_planes, gn, b256, 0, st, ni, d_pos, x);
  hipLaunchKernelGGL(k_com_partial, dim3(rblocks), b256, 0, st, n, (const double*)x, d_mass, red);
  hipLaunchKernelGGL(k_com_final, dim3(1), dim3(64), 0, st, rblocks, (const double*)red, sums);
  hipLaunchKernelGGL(k_na_scales, dim3(1), dim3(64), 0, st, (const double*)sums, eps2, mask ? 1 : 0, G, scale);
  const SrcRange r{ni, 0, ni, 1.f, scale};
  const TileSpan sp{0, span / kApTile, slice / kApTile};
  if (one_launch(n)) {
    const Finish f{nullptr, nullptr, 0.0, scale + 1, d_acc, 1, StepPost{}, nullptr, nullptr, nullptr};
    launch_tiles<true>(st, mask, r, x, d_mass, sp, S, eps2, f);
  } else {
    if (in_tiles<true>(n)) {
      Finish f{};
      f.part = part;
      launch_tiles<true>(st, mask, r, x, d_mass, sp, S, eps2, f);
    } else {
      hipLaunchKernelGGL(k_src<true>, dim3(npad / 256), b256, 0, st, r, npad, (const double*)x, d_mass, src);
      launch_slices<true>(st, mask, ni, npad, S, span, slice, eps2, x, src, part);
    }
    hipLaunchKernelGGL(k_na_combine, gn, b256, 0, st, ni, S, (const double*)part, (const double*)scale, d_acc);
  }
  if ((e = hipGetLastError()) != hipSuccess)
    return na_fail(ASTER_ERR_HIP, std::string("aster_forces_noalloc launch: ") + hipGetErrorString(e));
  return ASTER_OK;
}
