// Batched ensembles: thousands of small independent systems (1..64 bodies)
// integrated by one persistent kernel per launch.
//
// Layout: every system lives in the lanes of one wavefront; with packing,
// several systems share a wavefront (systems are ordered by size, largest
// first, and filled next-fit into 64 lanes), so a 3-body system does not idle
// 61 lanes. Each lane keeps its body's FP64 position, velocity and
// acceleration in registers for the whole launch; the wavefront exchanges
// positions (and velocities for 1PN) through LDS once per force evaluation.
// Force per pair: all-pairs within the system, Newton (+ pairwise 1PN),
// optionally Plummer-softened.
//
// Two arithmetic modes:
//   fast  (precision != ASTER_FP64): FP64 with an rsqrt estimate refined by
//         one Newton step (1/r to 4.1e-15), terms grouped for fused
//         multiply-adds.
//   exact (precision == ASTER_FP64): compute_gravitational in the reference's
//         operation order and j order (src/physics/tool_chain_impl.cpp:120-137,
//         Parallelized::compute_forces, src/utils/builder_endpoint.cpp:729-757),
//         so each system's trajectory is bit-identical to the CPU path.
// Integrators as in aster_step: leapfrog (update_leapfrog,
// tool_chain_impl.cpp:169-185) or Yoshida-4, accelerations cached between
// steps and across launches.
//
// A step sequence is split into launches of steps_per_launch steps; the
// launches are captured once into a HIP graph and replayed.
#include <algorithm>
#include <cmath>
#include <numeric>
#include <type_traits>
#include <vector>

#include "common.hpp"
#include "device.hpp"

namespace aster {

constexpr int kBatchMaxWpb = 4;
constexpr int kBatchSimds = 1024;

struct BatchArgs {
  int nwaves;
  const int32_t* lane_body;
  const int32_t* lane_seg;  // (segment base lane << 8) | segment size
  const int32_t* wave_max;  // largest segment in the wavefront
  double* x;
  double* v;
  double* a;
  const double* m;
  int64_t nsteps;
  int nsub;
  double h[3];
  int init;
  double G, ic2, ic, soft;
  int pnf;  // post-Newtonian terms (exact mode; the fast mode has PN1 only)
};

// Exact mode: kU sources at a time, whose pair forces are formed step by step
// together (a wavefront often has a SIMD to itself, so its own chains have to
// overlap), then added in j order; a pair that does not count adds 0. Leapfrog
// step of 1000 / 8192 systems of 3-64 bodies, against IEEE square root and
// division: Newtonian 15.0 -> 11.5 / 46.5 -> 31.8 us, 1PN 61 -> 59 / 163 -> 156,
// EIH 75 -> 65.5 / 168 -> 146. (kU = 4: 11.3 / 33, 61 / 164, 65 / 152; the 1PN
// force's division by div64_fast, after a look at its size: 63 / 145.) An odd last
// source goes by itself: 16384 systems of 3 / 5 bodies with 1PN terms 4.2 -> 3.4 /
// 9.4 -> 8.0 us (3.5 / 8.5 with one source at a time and IEEE operations). Up to
// two bodies the look at the ranges costs more than it saves, and so does the
// overlap (16384 pairs of bodies 0.74 -> 0.68 us), as long as a wavefront has a
// SIMD to itself (32800 pairs 0.87 us against 1.09).
constexpr int kU = 2;

// The sources of a wavefront's systems, kU at a time and the odd one by itself;
// none where every system is a single body. !FAST: two one after the other, and
// with post-Newtonian terms no code for a single one (k_batch with both is over
// 64 KB as it is, and another 4000 lines cost 4% with many wavefronts).
template <bool PN, bool FAST, class F>
__device__ __forceinline__ void batch_each_source(int maxcnt, F sources) {
  if (maxcnt < 2) return;
  int j0 = 0;
  if (FAST || PN || maxcnt > 2)
    for (; j0 + (PN && !FAST ? 1 : kU) <= maxcnt; j0 += kU) sources(j0, std::integral_constant<int, kU>{});
  if constexpr (FAST || !PN)
    for (; j0 < maxcnt; ++j0) sources(j0, std::integral_constant<int, 1>{});
}

// Separations and 1 / r of sources first .. first + N - 1. FAST: every input
// within the ranges of inv_sqrt64_fast and div64_fast.
template <bool FAST, int N>
__device__ __forceinline__ void batch_separations(int first, const double* lx, const double* ly, const double* lz,
                                                  const double* X, double soft, double (*d)[3], double* inv) {
#pragma clang fp contract(off)
  double r2[N];
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int src = min(first + u, 63);
    d[u][0] = lx[src] - X[0];
    d[u][1] = ly[src] - X[1];
    d[u][2] = lz[src] - X[2];
    r2[u] = d[u][0] * d[u][0] + d[u][1] * d[u][1] + d[u][2] * d[u][2] + soft;
  }
  if (!FAST || __builtin_expect(__any(inv_sqrt64_fast<N>(r2, inv)), 0)) {
#pragma unroll
    for (int u = 0; u < N; ++u) inv[u] = 1.0 / sqrt(r2[u]);
  }
}

// The accelerations f of the lane's body by sources j0 .. j0 + N - 1 of its
// system; 0 for a pair that does not count.
template <bool PN, bool FAST, int N>
__device__ __forceinline__ void batch_exact_pairs(int lane, int base, int cnt, int j0, bool live, const double* lx,
                                                  const double* ly, const double* lz, const double* lm,
                                                  const double* lvx, const double* lvy, const double* lvz,
                                                  const double* X, const double* V, const Divisor64& mi, double G,
                                                  double ic, int pnf, double soft, double (*f)[3]) {
#pragma clang fp contract(off)
  double d[N][3], inv[N];
  batch_separations<FAST, N>(base + j0, lx, ly, lz, X, soft, d, inv);
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int src = min(base + j0 + u, 63);
    const double m2 = lm[src];
    const double scal = G * m2 * mi.b * (inv[u] * inv[u]);
    double n[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      n[c] = d[u][c] * inv[u];
      f[u][c] = n[c] * scal;
    }
    if (PN) {
      pn_add64(pnf, mi.b, m2, V[0], V[1], V[2], lvx[src], lvy[src], lvz[src], inv[u], -n[0], -n[1], -n[2], G, ic,
               f[u][0], f[u][1], f[u][2]);
    }
  }
  if (FAST && !PN) {  // the post-Newtonian terms have no bounds of their own
    div64_fast<3 * N>(&f[0][0], mi);
  } else {
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) f[u][c] = f[u][c] / mi.b;
  }
#pragma unroll
  for (int u = 0; u < N; ++u) {
    const int src = min(base + j0 + u, 63);
    const bool valid = live && j0 + u < cnt && src != lane;
#pragma unroll
    for (int c = 0; c < 3; ++c) f[u][c] = valid ? f[u][c] : 0.0;
  }
}

template <bool PN, bool FAST>
__device__ __forceinline__ void batch_exact(int lane, int base, int cnt, int maxcnt, bool live, const double* lx,
                                            const double* ly, const double* lz, const double* lm, const double* lvx,
                                            const double* lvy, const double* lvz, const double* X, const double* V,
                                            const Divisor64& mi, double G, double ic, int pnf, double soft,
                                            double* A) {
#pragma clang fp contract(off)
  double a[3] = {0.0, 0.0, 0.0};
  auto sources = [&](int j0, auto count) {
    constexpr int N = count();
    double f[N][3];
    batch_exact_pairs<PN, FAST, N>(lane, base, cnt, j0, live, lx, ly, lz, lm, lvx, lvy, lvz, X, V, mi, G, ic, pnf,
                                   soft, f);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int c = 0; c < 3; ++c) a[c] += f[u][c];
  };
  batch_each_source<PN, FAST>(maxcnt, sources);
#pragma unroll
  for (int c = 0; c < 3; ++c) A[c] = a[c];
}

// Fast mode. A body's record in LDS: {position, mass} and, with 1PN terms,
// {velocity, |v|^2}. Behind a wavefront's 64 bodies lies a record of mass 0 far
// away: a lane that has no more sources takes it, and both force terms vanish
// without any selects on values.
template <bool PN>
constexpr int kRecQuads = PN ? 2 : 1;
constexpr int kNoBody = 64;

template <bool PN>
__device__ __forceinline__ void put_no_body(double4* rec) {
  rec[kNoBody * kRecQuads<PN>] = make_double4(1e100, 0.0, 0.0, 0.0);
  if (PN) rec[kNoBody * kRecQuads<PN> + 1] = make_double4(0.0, 0.0, 0.0, 0.0);
}

// (61.5 -> 58.3 instructions per pair, of them 52 of FP64; with scalar loop counts
// and the priorities below a step of 8192 systems of 3-64 bodies 60.7 -> 53.6 us
// with 1PN, 15.6 -> 12.5 us without: the SIMDs issue in ~90% of their cycles.)
// Source j of a lane's body: its system's bodies in order, itself left out.
struct FastLane {
  int base, self, sources;  // first body's lane, the body's place, number of sources
};
__device__ __forceinline__ FastLane fast_lane(int lane, int base, int cnt, bool live) {
  return {base, lane - base, live ? cnt - 1 : 0};
}
__device__ __forceinline__ int fast_source(const FastLane& l, int j) {
  const int src = l.base + j + (j >= l.self ? 1 : 0);
  return j < l.sources ? src : kNoBody;
}

// The parts of a pair's acceleration, f d (d) and, with 1PN terms, g k (g):
// {f, d, k, g}.
template <bool PN>
constexpr int kFastVals = PN ? 8 : 4;

template <bool PN>
__device__ __forceinline__ void batch_fast_pair(const double4* rec, int src, const double* X, const double* V,
                                                double v11, double g5m1, double G, double ic2, double soft,
                                                double* q) {
  const double4 o = rec[src * kRecQuads<PN>];
  const double m2 = o.w;
  const double dx = o.x - X[0], dy = o.y - X[1], dz = o.z - X[2];
  const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, soft)));
  // one Newton step: 1/r to 4.1e-15 (two steps, 1.4e-16, cost 4 more
  // instructions per pair; the exact mode divides as the reference does)
  const double inv = rsqrt64_n<1>(r2);
  const double inv2 = inv * inv;
  const double gm2 = G * m2;
  q[0] = gm2 * (inv2 * inv);
  q[1] = dx;
  q[2] = dy;
  q[3] = dz;
  if constexpr (PN) {
    const double4 w = rec[src * kRecQuads<PN> + 1];
    // get_pn1 (tool_chain_impl.cpp:110-118) with n = (x1 - x2)/r, the same
    // terms grouped for fused multiply-adds:
    //   G m2/r^2 [n (-v1^2 - 2 v2^2 + 4 v1.v2 + 3/2 (n.v2)^2 + (5 G m1 + 4 G m2)/r)
    //             + (v1 - v2)(4 n.v1 - 3 n.v2)]
    const double nx = -dx * inv, ny = -dy * inv, nz = -dz * inv;
    const double nv1 = fma(nx, V[0], fma(ny, V[1], nz * V[2]));
    const double nv2 = fma(nx, w.x, fma(ny, w.y, nz * w.z));
    const double v12 = fma(V[0], w.x, fma(V[1], w.y, V[2] * w.z));
    double sc = fma(4.0, v12, -v11);
    sc = fma(-2.0, w.w, sc);
    sc = fma(1.5 * nv2, nv2, sc);
    sc = fma(fma(4.0 * G, m2, g5m1), inv, sc);
    const double t = fma(4.0, nv1, -3.0 * nv2);
    q[4] = gm2 * inv2 * ic2;
    q[5] = fma(nx, sc, (V[0] - w.x) * t);
    q[6] = fma(ny, sc, (V[1] - w.y) * t);
    q[7] = fma(nz, sc, (V[2] - w.z) * t);
  }
}

template <bool PN>
__device__ __forceinline__ void batch_fast_add(const double* q, double& ax, double& ay, double& az) {
  ax = fma(q[0], q[1], ax);
  ay = fma(q[0], q[2], ay);
  az = fma(q[0], q[3], az);
  if constexpr (PN) {
    ax = fma(q[5], q[4], ax);
    ay = fma(q[6], q[4], ay);
    az = fma(q[7], q[4], az);
  }
}

template <bool PN>
__device__ __forceinline__ void batch_fast(const FastLane& l, int sources, const double4* rec, const double* X,
                                           const double* V, double mi, double G, double ic2, double soft,
                                           double* A) {
  double ax = 0.0, ay = 0.0, az = 0.0;
  // 1PN: this body's |v1|^2 and 5 G m1 (get_pn1's per-body parts)
  const double v11 = V[0] * V[0] + V[1] * V[1] + V[2] * V[2];
  const double g5m1 = 5.0 * G * mi;
  // Four sources per iteration: independent pair forces, sums still taken
  // one by one in j order
#pragma unroll 4
  for (int j = 0; j < sources; ++j) {
    double q[kFastVals<PN>];
    batch_fast_pair<PN>(rec, fast_source(l, j), X, V, v11, g5m1, G, ic2, soft, q);
    batch_fast_add<PN>(q, ax, ay, az);
  }
  A[0] = ax;
  A[1] = ay;
  A[2] = az;
}

// Full N-body 1PN (EIH) accelerations of a lane's body within its system
// (exact mode): pass 1 forms each body's potential and Newtonian
// acceleration and publishes them in LDS; pass 2 is the EIH sum, in the
// order and arithmetic of the oracle's EIH (sources in system order), so a
// system's trajectory equals the oracle's bit for bit.
template <bool FAST>
__device__ __forceinline__ void batch_eih(int lane, int base, int cnt, int maxcnt, bool live, const double* lx,
                                          const double* ly, const double* lz, const double* lm, const double* lvx,
                                          const double* lvy, const double* lvz, const double* X, const double* V,
                                          double G, double ic, double soft, double* lphi, double* lanx, double* lany,
                                          double* lanz, double* A) {
#pragma clang fp contract(off)
  double ph = 0.0, nx = 0.0, ny = 0.0, nz = 0.0;
  batch_each_source<true, FAST>(maxcnt, [&](int j0, auto count) {
    constexpr int N = count();
    double d[N][3], inv[N];
    batch_separations<FAST, N>(base + j0, lx, ly, lz, X, soft, d, inv);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int j = j0 + u, src = min(base + j, 63);
      const bool valid = live && j < cnt && src != lane;
      const double dx = d[u][0], dy = d[u][1], dz = d[u][2];
      const double inv_r = inv[u];
      const double inv_r3 = inv_r * inv_r * inv_r;
      const double mu = G * lm[src];
      if (valid) {
        ph += mu * inv_r;
        nx += mu * dx * inv_r3;
        ny += mu * dy * inv_r3;
        nz += mu * dz * inv_r3;
      }
    }
  });
  lphi[lane] = ph;
  lanx[lane] = nx;
  lany[lane] = ny;
  lanz[lane] = nz;
  wave_sync();
  const double ic2 = ic * ic;
  const double vi2 = V[0] * V[0] + V[1] * V[1] + V[2] * V[2];
  double ax = 0.0, ay = 0.0, az = 0.0;
  batch_each_source<true, FAST>(maxcnt, [&](int j0, auto count) {
    constexpr int N = count();
    double d[N][3], inv[N];
    batch_separations<FAST, N>(base + j0, lx, ly, lz, X, soft, d, inv);
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const int j = j0 + u, src = min(base + j, 63);
      const bool valid = live && j < cnt && src != lane;
      const double dx = d[u][0], dy = d[u][1], dz = d[u][2];
      const double inv_r = inv[u];
      const double inv_r3 = inv_r * inv_r * inv_r;
      const double mu = G * lm[src];
      const double v2x = lvx[src], v2y = lvy[src], v2z = lvz[src];
      const double anx = lanx[src], any = lany[src], anz = lanz[src];
      const double vj2 = v2x * v2x + v2y * v2y + v2z * v2z;
      const double vij = V[0] * v2x + V[1] * v2y + V[2] * v2z;
      const double rv = (dx * v2x + dy * v2y + dz * v2z) * inv_r;
      const double dan = dx * anx + dy * any + dz * anz;
      const double B = 1.0 - (4.0 * ph + lphi[src]) * ic2 + (vi2 + 2.0 * vj2 - 4.0 * vij) * ic2 - 1.5 * (rv * rv) * ic2 +
                       0.5 * dan * ic2;
      const double s1 = mu * inv_r3 * B;
      const double w = -(dx * (4.0 * V[0] - 3.0 * v2x) + dy * (4.0 * V[1] - 3.0 * v2y) + dz * (4.0 * V[2] - 3.0 * v2z));
      const double s2 = mu * inv_r3 * ic2 * w;
      const double s3 = 3.5 * mu * inv_r * ic2;
      if (valid) {
        ax += dx * s1;
        ax += (V[0] - v2x) * s2;
        ax += anx * s3;
        ay += dy * s1;
        ay += (V[1] - v2y) * s2;
        ay += any * s3;
        az += dz * s1;
        az += (V[2] - v2z) * s2;
        az += anz * s3;
      }
    }
  });
  wave_sync();  // the next evaluation rewrites the LDS potentials
  A[0] = ax;
  A[1] = ay;
  A[2] = az;
}

template <int N = 3>
__device__ __forceinline__ void kick_drift_reg(double* X, double* V, const double* A, double dt_prev, double dt) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < N; ++c) {
    double vc = V[c];
    if (dt_prev != 0.0) vc = vc + 0.5 * A[c] * dt_prev;
    X[c] = X[c] + (vc * dt + 0.5 * A[c] * dt * dt);
    V[c] = vc + 0.5 * A[c] * dt;
  }
}

template <int N = 3>
__device__ __forceinline__ void kick_reg(double* V, const double* A, double dt) {
#pragma clang fp contract(off)
#pragma unroll
  for (int c = 0; c < N; ++c) V[c] = V[c] + 0.5 * A[c] * dt;
}

template <bool PN, bool EXACT>
__global__ __launch_bounds__(256) void k_batch(BatchArgs P) {
  // exact mode: positions, masses (and velocities) of each wavefront's bodies,
  // one plane per quantity in a single array, so a source's values sit at one
  // address plus constant plane offsets; fast mode: records
  constexpr int kX = EXACT ? kBatchMaxWpb : 1, kF = EXACT ? 1 : kBatchMaxWpb;
  __shared__ double planes[PN ? 7 : 4][kX][64];
  __shared__ double4 recs[kF][EXACT ? 1 : (kNoBody + 1) * kRecQuads<PN>];
  auto sx = planes[0];
  auto sy = planes[1];
  auto sz = planes[2];
  auto sm = planes[3];
  auto svx = planes[PN ? 4 : 0];
  auto svy = planes[PN ? 5 : 0];
  auto svz = planes[PN ? 6 : 0];
  constexpr int kE = (PN && EXACT) ? kBatchMaxWpb : 1;  // EIH potentials and Newtonian accelerations
  __shared__ double sphi[kE][64], sanx[kE][64], sany[kE][64], sanz[kE][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wl;
  if (wave >= P.nwaves) return;
  const int slot = wave * 64 + lane;
  const int b = P.lane_body[slot];
  const int seg = P.lane_seg[slot];
  const int base = seg >> 8, cnt = seg & 255;
  const int maxcnt = __builtin_amdgcn_readfirstlane(P.wave_max[wave]);
  // the longest loops first: a wavefront that is left alone issues at half the rate
  if (maxcnt > 48) __builtin_amdgcn_s_setprio(3);
  else if (maxcnt > 32) __builtin_amdgcn_s_setprio(2);
  else if (maxcnt > 16) __builtin_amdgcn_s_setprio(1);
  const bool live = b >= 0;
  double X[3] = {0.0, 0.0, 0.0}, V[3] = {0.0, 0.0, 0.0}, A[3] = {0.0, 0.0, 0.0};
  double mi = 0.0;
  if (live) {
    for (int c = 0; c < 3; ++c) {
      X[c] = P.x[3 * (size_t)b + c];
      V[c] = P.v[3 * (size_t)b + c];
      A[c] = P.a[3 * (size_t)b + c];
    }
    mi = P.m[b];
  }
  const int xl = EXACT ? wl : 0;
  double* lx = sx[xl];
  double* ly = sy[xl];
  double* lz = sz[xl];
  double* lvx = svx[xl];
  double* lvy = svy[xl];
  double* lvz = svz[xl];
  double* lm = sm[xl];
  double4* rec = recs[EXACT ? 0 : wl];
  const FastLane fl = fast_lane(lane, base, cnt, live);
  if (EXACT) lm[lane] = mi;
  else if (lane == 0) put_no_body<PN>(rec);
  const Divisor64 md = divisor64(live ? mi : 1.0);
  const bool ranges = EXACT && __all(!live || mass_in_range64(mi)) && law_in_range64(P.G, P.soft);
  auto publish = [&]() {
    if constexpr (EXACT) {
      lx[lane] = X[0];
      ly[lane] = X[1];
      lz[lane] = X[2];
      if (PN) {
        lvx[lane] = V[0];
        lvy[lane] = V[1];
        lvz[lane] = V[2];
      }
    } else {
      rec[lane * kRecQuads<PN>] = make_double4(X[0], X[1], X[2], mi);
      if (PN)
        rec[lane * kRecQuads<PN> + 1] =
            make_double4(V[0], V[1], V[2], fma(V[0], V[0], fma(V[1], V[1], V[2] * V[2])));
    }
    wave_sync();
  };
  const bool eih = PN && EXACT && (P.pnf & ASTER_EIH);
  auto in_ranges = [&]() {
    return EXACT && ranges && (maxcnt > 2 || P.nwaves > kBatchSimds) &&
           __all(!live || (coord_in_range64(X[0]) && coord_in_range64(X[1]) && coord_in_range64(X[2])));
  };
  auto accel = [&]() {
    if constexpr (!EXACT) {
      batch_fast<PN>(fl, maxcnt - 1, rec, X, V, mi, P.G, P.ic2, P.soft, A);
    } else if (eih) {
      const int e = PN ? wl : 0;
      if (in_ranges())
        batch_eih<true>(lane, base, cnt, maxcnt, live, lx, ly, lz, lm, lvx, lvy, lvz, X, V, P.G, P.ic, P.soft,
                        sphi[e], sanx[e], sany[e], sanz[e], A);
      else
        batch_eih<false>(lane, base, cnt, maxcnt, live, lx, ly, lz, lm, lvx, lvy, lvz, X, V, P.G, P.ic, P.soft,
                         sphi[e], sanx[e], sany[e], sanz[e], A);
    } else if (in_ranges()) {
      batch_exact<PN, true>(lane, base, cnt, maxcnt, live, lx, ly, lz, lm, lvx, lvy, lvz, X, V, md, P.G, P.ic, P.pnf,
                            P.soft, A);
    } else {
      batch_exact<PN, false>(lane, base, cnt, maxcnt, live, lx, ly, lz, lm, lvx, lvy, lvz, X, V, md, P.G, P.ic, P.pnf,
                             P.soft, A);
    }
  };
  if (P.init) {
    publish();
    accel();
    wave_sync();
  }
  double pending = 0.0;
  for (int64_t s = 0; s < P.nsteps; ++s) {
    for (int k = 0; k < P.nsub; ++k) {
      const double h = P.h[k];
      if (PN) {
        // Velocity-dependent forces: re-evaluate after the final kick, as
        // update_leapfrog's first compute_forces does.
        if (pending != 0.0) kick_reg(V, A, pending);
        pending = 0.0;
        publish();
        accel();
        wave_sync();
      }
      kick_drift_reg(X, V, A, pending, h);
      publish();
      accel();
      wave_sync();
      pending = h;
    }
  }
  if (P.nsteps > 0) kick_reg(V, A, pending);
  if (live) {
    for (int c = 0; c < 3; ++c) {
      P.x[3 * (size_t)b + c] = X[c];
      P.v[3 * (size_t)b + c] = V[c];
      P.a[3 * (size_t)b + c] = A[c];
    }
  }
}

// Few wavefronts of systems (team_size): W worker wavefronts form a wavefront's
// pair forces, kU sources each at a time, and pass them through LDS to three
// adding wavefronts, one per coordinate, which sum them in j order and advance
// the bodies; the workers are a chunk of W kU sources ahead. Same operations as
// k_batch's in the same order, so the same bits (the fast mode passes the
// factors of its last fused multiply-adds).
template <bool PN, bool EXACT, int W>
__global__ __launch_bounds__(64 * (W + 3)) void k_batch_team(BatchArgs P) {
#pragma clang fp contract(off)
  constexpr int kChunk = W * kU;
  constexpr int kVals = EXACT ? 3 : kFastVals<PN>;
  __shared__ double planes[PN ? 7 : 4][EXACT ? 64 : 1];
  __shared__ double4 rec[EXACT ? 1 : (kNoBody + 1) * kRecQuads<PN>];
  __shared__ double force[2][kChunk][kVals][64];
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const bool adder = w >= W;
  const int ax = __builtin_amdgcn_readfirstlane(adder ? w - W : 0);  // an adder's coordinate
  const int slot = blockIdx.x * 64 + lane;
  const int b = P.lane_body[slot];
  const int seg = P.lane_seg[slot];
  const int base = seg >> 8, cnt = seg & 255;
  const int maxcnt = __builtin_amdgcn_readfirstlane(P.wave_max[blockIdx.x]);
  const bool live = b >= 0;
  const double mi = live ? P.m[b] : 0.0;
  double x = 0.0, v = 0.0, a = 0.0;  // adder: its coordinate of the body
  const size_t at = 3 * (size_t)(live ? b : 0) + ax;
  if (live && adder) {
    x = P.x[at];
    v = P.v[at];
    a = P.a[at];
  }
  double X[3] = {0.0, 0.0, 0.0}, V[3] = {0.0, 0.0, 0.0};  // worker: the body
  const FastLane fl = fast_lane(lane, base, cnt, live);
  const int sources = EXACT ? maxcnt : maxcnt - 1;  // the exact mode passes 0 for the body itself
  if (EXACT && w == 0) planes[3][lane] = mi;
  if (!EXACT && w == 0) {
    rec[lane * kRecQuads<PN>].w = mi;
    if (lane == 0) put_no_body<PN>(rec);
  }
  const Divisor64 md = divisor64(EXACT && live ? mi : 1.0);
  const bool ranges = EXACT && __all(!live || mass_in_range64(mi)) && law_in_range64(P.G, P.soft);
  // past the sources: 0, so that a chunk always has the same length
  auto work = [&](int j0, bool fast, double (*out)[kVals][64]) {
    double f[kU][kVals] = {};
    const double* p = &planes[0][0];
    const double* vx = PN ? p + 4 * 64 : p;
    const double* vy = PN ? p + 5 * 64 : p;
    const double* vz = PN ? p + 6 * 64 : p;
    if constexpr (EXACT) {
      if (j0 < maxcnt && fast)
        batch_exact_pairs<PN, true, kU>(lane, base, cnt, j0, live, p, p + 64, p + 128, p + 192, vx, vy, vz, X, V, md, P.G,
                                    P.ic, P.pnf, P.soft, f);
      else if (j0 < maxcnt)
        batch_exact_pairs<PN, false, kU>(lane, base, cnt, j0, live, p, p + 64, p + 128, p + 192, vx, vy, vz, X, V, md, P.G,
                                     P.ic, P.pnf, P.soft, f);
    } else if (j0 < sources) {
      const double v11 = V[0] * V[0] + V[1] * V[1] + V[2] * V[2];
      const double g5m1 = 5.0 * P.G * mi;
#pragma unroll
      for (int u = 0; u < kU; ++u)
        batch_fast_pair<PN>(rec, fast_source(fl, j0 + u), X, V, v11, g5m1, P.G, P.ic2, P.soft, f[u]);
    }
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int c = 0; c < kVals; ++c) out[u][c][lane] = f[u][c];
  };
  // the adders' bodies to the workers, then the accelerations to the adders
  auto accel = [&]() {
    double* mine = reinterpret_cast<double*>(rec + lane * kRecQuads<PN>);  // fast mode: {x, y, z, m, v, |v|^2}
    if (adder) {
      (EXACT ? planes[ax][lane] : mine[ax]) = x;
      if (PN) (EXACT ? planes[4 + ax][lane] : mine[4 + ax]) = v;
    }
    __syncthreads();
    if (!adder) {
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        X[c] = EXACT ? planes[c][lane] : mine[c];
        if (PN) V[c] = EXACT ? planes[4 + c][lane] : mine[4 + c];
      }
    }
    if (PN && !EXACT) {
      if (w == 0) mine[7] = fma(V[0], V[0], fma(V[1], V[1], V[2] * V[2]));
      __syncthreads();
    }
    double sum = 0.0;
    auto add = [&](int j0) {
      const auto& f = force[(j0 / kChunk) & 1];
#pragma unroll
      for (int u = 0; u < kChunk; ++u) {
        if constexpr (EXACT) {
          sum += f[u][ax][lane];
        } else {
          sum = fma(f[u][0][lane], f[u][1 + ax][lane], sum);
          if constexpr (PN) sum = fma(f[u][5 + ax][lane], f[u][4][lane], sum);
        }
      }
    };
    const bool fast =
        ranges && __all(!live || (coord_in_range64(X[0]) && coord_in_range64(X[1]) && coord_in_range64(X[2])));
    int j0 = 0;
    for (; j0 < sources; j0 += kChunk) {
      if (!adder) work(j0 + w * kU, fast, &force[(j0 / kChunk) & 1][w * kU]);
      else if (j0 > 0) add(j0 - kChunk);
      __syncthreads();
    }
    if (adder) {
      if (j0 > 0) add(j0 - kChunk);
      a = sum;
    }
  };
  if (P.init) accel();
  double pending = 0.0;
  for (int64_t s = 0; s < P.nsteps; ++s) {
    for (int k = 0; k < P.nsub; ++k) {
      const double h = P.h[k];
      if (PN) {  // as k_batch
        if (adder && pending != 0.0) kick_reg<1>(&v, &a, pending);
        pending = 0.0;
        accel();
      }
      if (adder) kick_drift_reg<1>(&x, &v, &a, pending, h);
      accel();
      pending = h;
    }
  }
  if (!adder || !live) return;
  if (P.nsteps > 0) kick_reg<1>(&v, &a, pending);
  P.x[at] = x;
  P.v[at] = v;
  P.a[at] = a;
}

// Per-body energy terms: kinetic - 1/2 G m_i sum_j m_j / sqrt(r^2 + soft),
// and m x cross v; out [4][nbodies].
__global__ __launch_bounds__(256) void k_batch_energy(BatchArgs P, int nbodies, double* __restrict__ out) {
  __shared__ double sx[kBatchMaxWpb][64], sy[kBatchMaxWpb][64], sz[kBatchMaxWpb][64], sm[kBatchMaxWpb][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wl;
  if (wave >= P.nwaves) return;
  const int slot = wave * 64 + lane;
  const int b = P.lane_body[slot];
  const int seg = P.lane_seg[slot];
  const int base = seg >> 8, cnt = seg & 255;
  const int maxcnt = P.wave_max[wave];
  const bool live = b >= 0;
  double X[3] = {0.0, 0.0, 0.0}, V[3] = {0.0, 0.0, 0.0}, mi = 0.0;
  if (live) {
    for (int c = 0; c < 3; ++c) {
      X[c] = P.x[3 * (size_t)b + c];
      V[c] = P.v[3 * (size_t)b + c];
    }
    mi = P.m[b];
  }
  sx[wl][lane] = X[0];
  sy[wl][lane] = X[1];
  sz[wl][lane] = X[2];
  sm[wl][lane] = mi;
  wave_sync();
  double pot = 0.0;
  for (int j = 0; j < maxcnt; ++j) {
    const int src = min(base + j, 63);
    const bool valid = live && j < cnt && src != lane;
    const double dx = sx[wl][src] - X[0], dy = sy[wl][src] - X[1], dz = sz[wl][src] - X[2];
    const double r2 = dx * dx + dy * dy + dz * dz + P.soft;
    if (valid) pot += sm[wl][src] / sqrt(r2);
  }
  if (live) {
    out[b] = 0.5 * mi * (V[0] * V[0] + V[1] * V[1] + V[2] * V[2]) - 0.5 * P.G * mi * pot;
    out[(size_t)nbodies + b] = mi * (X[1] * V[2] - X[2] * V[1]);
    out[(size_t)2 * nbodies + b] = mi * (X[2] * V[0] - X[0] * V[2]);
    out[(size_t)3 * nbodies + b] = mi * (X[0] * V[1] - X[1] * V[0]);
  }
}

__global__ void k_batch_sum(int64_t nsys, const int64_t* __restrict__ off, int64_t nbodies,
                            const double* __restrict__ eb, double* __restrict__ es) {
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nsys) return;
  for (int q = 0; q < 4; ++q) {
    double acc = 0.0;
    for (int64_t k = off[s]; k < off[s + 1]; ++k) acc += eb[(size_t)q * nbodies + k];
    es[(size_t)q * nsys + s] = acc;
  }
}

// ----------------------------------------------------------------- host ----

// ---- Wisdom-Holman for central-mass systems ------------------------------
//
// Democratic-heliocentric Wisdom-Holman (Wisdom & Holman 1991; Duncan, Levison
// & Lee 1998). The reference's update_WH_planetary (tool_chain_impl.cpp:
// 235-274) drifts each body i >= 1 on a Kepler orbit about body 0 and then
// kicks with the full accelerations, which include body 0's pull again; this
// is the splitting that scheme is meant to be: H = H_Kepler(mu = G m_0) +
// H_interaction(planet pairs) + |sum m_i u_i|^2 / (2 m_0) in heliocentric
// positions Q_i = x_i - x_0 and barycentric velocities u_i. One step: half
// interaction kick, half jump Q_i += (sum m_j u_j / m_0) dt/2, Kepler drift,
// half jump, half kick. Body 0 of each system is the central mass. During a
// call the batch buffers hold the heliocentric state (planets: Q, u, and
// their interaction accelerations; body 0: the barycentre and its velocity),
// so launches can split the steps anywhere without changing a bit. Segment
// sums are taken by every lane of a system in body order, and pair forces are
// compute_gravitational (tool_chain_impl.cpp:120-137) in j order, Newtonian,
// so every system is bit-identical to the CPU restatement.
enum { WH_ENTER = 0, WH_STEPS = 1, WH_EXIT = 2 };

struct WhArgs {
  int nwaves;
  const int32_t* lane_body;
  const int32_t* lane_seg;
  const int32_t* wave_max;
  double* x;
  double* v;
  double* a;
  const double* m;
  int64_t nsteps;
  double dt, G, soft;
  int phase;
};

__global__ __launch_bounds__(256) void k_batch_wh(WhArgs P) {
#pragma clang fp contract(off)
  __shared__ double sx[kBatchMaxWpb][64], sy[kBatchMaxWpb][64], sz[kBatchMaxWpb][64], sm[kBatchMaxWpb][64];
  __shared__ double tx[kBatchMaxWpb][64], ty[kBatchMaxWpb][64], tz[kBatchMaxWpb][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wl;
  if (wave >= P.nwaves) return;
  const int slot = wave * 64 + lane;
  const int b = P.lane_body[slot];
  const int seg = P.lane_seg[slot];
  const int base = seg >> 8, cnt = seg & 255;
  const bool live = b >= 0;
  const bool head = live && lane == base;   // the system's central body
  const bool planet = live && lane != base;
  double* lx = sx[wl];
  double* ly = sy[wl];
  double* lz = sz[wl];
  double* lm = sm[wl];
  double* ux = tx[wl];
  double* uy = ty[wl];
  double* uz = tz[wl];
  double X[3] = {0.0, 0.0, 0.0}, V[3] = {0.0, 0.0, 0.0}, A[3] = {0.0, 0.0, 0.0};
  double mi = 0.0;
  if (live) {
    mi = P.m[b];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      X[c] = P.x[3 * (size_t)b + c];
      V[c] = P.v[3 * (size_t)b + c];
      A[c] = P.a[3 * (size_t)b + c];
    }
  }
  lm[lane] = mi;
  wave_sync();
  const double m0 = live ? lm[base] : 1.0;
  const double mu = P.G * m0;
  const int maxcnt = __builtin_amdgcn_readfirstlane(P.wave_max[wave]);
  const Divisor64 md = divisor64(live ? mi : 1.0);
  const bool ranges = __all(!live || mass_in_range64(mi)) && law_in_range64(P.G, P.soft);
  const double h = 0.5 * P.dt;

  // interaction accelerations of the planets at the positions in X (with the
  // sums below by every lane, two reads at a time: step of systems up to 64 bodies
  // 40 -> 33 us; the Kepler drift, up to ~50 iterations in some lane, is ~20 us of
  // it and all of it for a few bodies)
  auto interaction = [&]() {
    if (maxcnt < 3) {  // no pair of planets
      A[0] = A[1] = A[2] = 0.0;
      return;
    }
    lx[lane] = X[0];
    ly[lane] = X[1];
    lz[lane] = X[2];
    wave_sync();
    const bool fast =
        ranges && maxcnt > 3 &&
        __all(!live || (coord_in_range64(X[0]) && coord_in_range64(X[1]) && coord_in_range64(X[2])));
    if (fast)
      batch_exact<false, true>(lane, base + 1, cnt - 1, maxcnt - 1, planet, lx, ly, lz, lm, nullptr, nullptr, nullptr,
                               X, V, md, P.G, 0.0, 0, P.soft, A);
    else
      batch_exact<false, false>(lane, base + 1, cnt - 1, maxcnt - 1, planet, lx, ly, lz, lm, nullptr, nullptr, nullptr,
                                X, V, md, P.G, 0.0, 0, P.soft, A);
    wave_sync();
  };
  // sum over the system's planets of m_j w_j (j order), by every lane itself
  auto planet_sum = [&](const double* W, double* out) {
    ux[lane] = planet ? mi * W[0] : 0.0;
    uy[lane] = planet ? mi * W[1] : 0.0;
    uz[lane] = planet ? mi * W[2] : 0.0;
    wave_sync();
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int j0 = 1; j0 < cnt; j0 += 2) {  // past the system: 0
      double w[2][3];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int src = min(base + j0 + u, 63);
        w[u][0] = ux[src];
        w[u][1] = uy[src];
        w[u][2] = uz[src];
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool in = j0 + u < cnt;
        s0 += in ? w[u][0] : 0.0;
        s1 += in ? w[u][1] : 0.0;
        s2 += in ? w[u][2] : 0.0;
      }
    }
    out[0] = s0;
    out[1] = s1;
    out[2] = s2;
    wave_sync();
  };
  auto jump = [&]() {
    double S[3] = {0.0, 0.0, 0.0};
    planet_sum(V, S);
    if (planet)
#pragma unroll
      for (int c = 0; c < 3; ++c) X[c] = X[c] + S[c] / m0 * h;
  };

  if (P.phase == WH_ENTER) {
    // M, barycentre and its velocity over all bodies (j order), then
    // Q = x - x_0, u = v - V for the planets; body 0 keeps (X, V).
    lx[lane] = mi * X[0];
    ly[lane] = mi * X[1];
    lz[lane] = mi * X[2];
    ux[lane] = mi * V[0];
    uy[lane] = mi * V[1];
    uz[lane] = mi * V[2];
    wave_sync();
    double M = 0.0, Sx[3] = {0.0, 0.0, 0.0}, Sv[3] = {0.0, 0.0, 0.0};
    if (head)
      for (int j = 0; j < cnt; ++j) {
        M += lm[base + j];
        Sx[0] += lx[base + j];
        Sx[1] += ly[base + j];
        Sx[2] += lz[base + j];
        Sv[0] += ux[base + j];
        Sv[1] += uy[base + j];
        Sv[2] += uz[base + j];
      }
    wave_sync();
    if (head) {
      // publish x_0 (this lane's own position) and the barycentre velocity
      lx[lane] = X[0];
      ly[lane] = X[1];
      lz[lane] = X[2];
      ux[lane] = Sv[0] / M;
      uy[lane] = Sv[1] / M;
      uz[lane] = Sv[2] / M;
    }
    wave_sync();
    if (planet) {
      const double x0[3] = {lx[base], ly[base], lz[base]};
      const double vc[3] = {ux[base], uy[base], uz[base]};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        X[c] = X[c] - x0[c];
        V[c] = V[c] - vc[c];
      }
    }
    if (head)
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        X[c] = Sx[c] / M;
        V[c] = Sv[c] / M;
      }
    wave_sync();
    interaction();
  } else if (P.phase == WH_STEPS) {
    for (int64_t s = 0; s < P.nsteps; ++s) {
      if (planet)
#pragma unroll
        for (int c = 0; c < 3; ++c) V[c] = V[c] + A[c] * h;
      jump();
      if (planet) kepler_drift64(X, V, mu, P.dt);
      jump();
      interaction();
      if (planet)
#pragma unroll
        for (int c = 0; c < 3; ++c) V[c] = V[c] + A[c] * h;
      if (head)
#pragma unroll
        for (int c = 0; c < 3; ++c) X[c] = X[c] + V[c] * P.dt;
    }
  } else {
    // x_0 = X - sum m_j Q_j / M, x_i = Q_i + x_0, v_0 = V - sum m_j u_j / m_0,
    // v_i = u_i + V
    double SQ[3] = {0.0, 0.0, 0.0}, SU[3] = {0.0, 0.0, 0.0};
    planet_sum(X, SQ);
    planet_sum(V, SU);
    if (head) {
      double M = 0.0;
      for (int j = 0; j < cnt; ++j) M += lm[base + j];
#pragma unroll
      for (int c = 0; c < 3; ++c) X[c] = X[c] - SQ[c] / M;
      lx[lane] = X[0];
      ly[lane] = X[1];
      lz[lane] = X[2];
      ux[lane] = V[0];
      uy[lane] = V[1];
      uz[lane] = V[2];
    }
    wave_sync();
    if (planet) {
      const double x0[3] = {lx[base], ly[base], lz[base]};
      const double vb[3] = {ux[base], uy[base], uz[base]};
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        X[c] = X[c] + x0[c];
        V[c] = V[c] + vb[c];
      }
    }
    if (head)
#pragma unroll
      for (int c = 0; c < 3; ++c) V[c] = V[c] - SU[c] / m0;
#pragma unroll
    for (int c = 0; c < 3; ++c) A[c] = 0.0;
  }
  if (live) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      P.x[3 * (size_t)b + c] = X[c];
      P.v[3 * (size_t)b + c] = V[c];
      P.a[3 * (size_t)b + c] = A[c];
    }
  }
}

// Wavefront plan. pack = 0: one system per wavefront. pack = 1: first fit
// decreasing: each wavefront opens with the largest system left (its size is
// the wavefront's loop length) and fills its free lanes with the largest
// systems left that fit. Against next fit over the sorted sizes this fills the
// lanes beside a 33..63-body system instead of leaving them idle (lane use of
// 8192 systems of 3..64 bodies: 0.87 instead of 0.78).
static int upload_plan(aster_ctx* c) {
  BatchState& B = c->batch;
  const int64_t nsys = B.nsys;
  std::vector<std::vector<int64_t>> by_size(65);  // systems of each size, in index order
  for (int64_t s = 0; s < nsys; ++s) by_size[(size_t)(B.offsets[s + 1] - B.offsets[s])].push_back(s);
  std::vector<size_t> next(65, 0);  // first unplaced system of each size
  std::vector<int32_t> lb, ls, wm;
  auto place = [&](int64_t s, int used) {
    const int sz = (int)(B.offsets[s + 1] - B.offsets[s]);
    const size_t w = wm.size() - 1;
    for (int k = 0; k < sz; ++k) {
      lb[w * 64 + used + k] = (int32_t)(B.offsets[s] + k);
      ls[w * 64 + used + k] = (used << 8) | sz;
    }
    wm[w] = std::max(wm[w], sz);
    return used + sz;
  };
  for (int top = 64; top >= 1;) {
    if (next[top] == by_size[top].size()) {
      --top;
      continue;
    }
    lb.resize(lb.size() + 64, -1);
    ls.resize(ls.size() + 64, 0);
    wm.push_back(0);
    int used = place(by_size[top][next[top]++], 0);
    if (B.pack != 0)
      for (int sz = std::min(64 - used, top); sz >= 1; --sz)
        while (used + sz <= 64 && next[sz] < by_size[sz].size()) used = place(by_size[sz][next[sz]++], used);
  }
  B.nwaves = (int)wm.size();
  for (int r = 0; r < kTeamRounds; ++r)  // (the wavefronts are in descending order of their largest system)
    B.round_max[r] = (size_t)r * kTeamRound < wm.size() ? wm[(size_t)r * kTeamRound] : 0;
  B.lane_slots = 0;
  for (int32_t mx : wm) B.lane_slots += 64 * (int64_t)mx;
  ASTER_HIP(c, B.lane_body.reserve(lb.size()));
  ASTER_HIP(c, B.lane_seg.reserve(ls.size()));
  ASTER_HIP(c, B.wave_max.reserve(wm.size()));
  ASTER_HIP(c, hipMemcpyAsync(B.lane_body.p, lb.data(), lb.size() * 4, hipMemcpyHostToDevice, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(B.lane_seg.p, ls.data(), ls.size() * 4, hipMemcpyHostToDevice, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(B.wave_max.p, wm.data(), wm.size() * 4, hipMemcpyHostToDevice, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  return ASTER_OK;
}

static void drop_graph(BatchState& B) {
  if (B.exec) (void)hipGraphExecDestroy(B.exec);
  if (B.graph) (void)hipGraphDestroy(B.graph);
  B.exec = nullptr;
  B.graph = nullptr;
  B.g_steps = -1;
}

// New parameters (G, c, softening, force law, precision): the cached
// accelerations and the captured launches hold the old ones.
void batch_params_changed(aster_ctx* c) {
  if (c->batch.exec) (void)hipStreamSynchronize(c->stream);  // a replay may still run
  drop_graph(c->batch);
  c->batch.a_valid = false;
}

static BatchArgs make_args(aster_ctx* c, int64_t nsteps, int nsub, const double* h, int init) {
  BatchState& B = c->batch;
  BatchArgs P;
  P.nwaves = B.nwaves;
  P.lane_body = B.lane_body.p;
  P.lane_seg = B.lane_seg.p;
  P.wave_max = B.wave_max.p;
  P.x = B.x.p;
  P.v = B.v.p;
  P.a = B.a.p;
  P.m = B.m.p;
  P.nsteps = nsteps;
  P.nsub = nsub;
  for (int k = 0; k < 3; ++k) P.h[k] = h[k];
  P.init = init;
  P.G = c->P.G;
  P.ic2 = (1.0 / c->P.c) * (1.0 / c->P.c);
  P.ic = 1.0 / c->P.c;
  P.pnf = c->P.pn_flags & ASTER_PN_TERMS;
  P.soft = c->P.softening;
  return P;
}

// Workers per wavefront of systems (k_batch_team), 0 for k_batch: while the
// chip has more SIMDs than such wavefronts, their serial chains are what a step
// waits for. The 256 CUs take a workgroup each, the wavefronts with the largest
// systems first, so the time grows with every 256 wavefronts by what the largest
// system behind them needs: chunks of 8 sources per 4 workers. Step times of
// the teams over k_batch's, systems of one size, by the number of such rounds.
// Exact mode with post-Newtonian terms (the rounds add up): 3 bodies 0.88 / 1.75,
// 5 0.57 / 1.13, 6 0.49 / 0.97 / 1.45, 9 0.47 / 0.95 / 1.41, 16 0.28 / 0.57 / 0.85 /
// 1.11, 17 0.39 / 0.79 / 1.18, 33 0.31 / 0.63 / 0.95 / 1.25, 64 0.24 / 0.49 / 0.73 /
// 0.96. Exact Newtonian: 2 1.16, 3 0.90 / 1.15, 5 0.67 / 0.84 / 1.06, 8 0.48 / 0.62 /
// 0.77 / 1.08, 16 0.35 / 0.52 / 0.73 / 1.0, 25 0.39 / 0.57 / 0.85 / 1.17, 64 0.30 / 0.47 /
// 0.71 / 0.95; sizes 3..64 mixed 0.30 / 0.40 / 0.55 / 0.75. Fast Newtonian: 6 1.15, 7 0.95,
// 8 0.79 / 1.05, 10 1.11, 12 0.90 / 1.3, 16 0.72 / 1.05, 64 0.65 / 1.0; 3..64 mixed 0.66 / 0.8.
// Fast with 1PN: 7 1.07, 8 0.93 / 1.37, 10 1.19, 12 0.98 / 1.44, 16 0.79 / 1.18, 64 0.65 /
// 1.0; mixed 0.66 / 0.8.
static int team_size(int nwaves, const int* largest, int pnf, bool exact) {
  const bool pn = pnf != 0;
  const int n = largest[0], rounds = (nwaves + kTeamRound - 1) / kTeamRound;
  if (rounds > kTeamRounds) return 0;
  if (exact && pn) {
    int cost = 0;  // in hundredths of a source of k_batch
    for (int r = 0; r < rounds; ++r) {
      const int k = (largest[r] + 7) / 8;
      if (pnf == ASTER_PN1) cost += n > 8 ? std::max(310, 70 + 185 * k) : 290;
      else cost += n > 8 ? std::max(265, 60 + 180 * k) : 245;
    }
    return cost > 100 * n ? 0 : n > 8 ? 8 : 4;
  }
  const int last = 32 * largest[rounds - 1];  // of the round that would be added
  if (exact) {
    const bool team = rounds == 1   ? n >= 3
                      : rounds == 2 ? n >= 5
                      : rounds == 3 ? n >= 6
                                    : n >= 58 || (n >= 12 && last <= 24 * n);
    return !team ? 0 : n > 8 && rounds == 1 ? 8 : 4;
  }
  const bool team = rounds == 1 ? n >= (pn ? 8 : 7) && n != 10
                                : rounds == 2 && n >= 16 && last <= (n >= 32 ? 26 : 21) * n;
  return !team ? 0 : n > 9 && rounds == 1 && !pn ? 8 : 4;
}

static int launch_batch(aster_ctx* c, const BatchArgs& P) {
  if ((c->P.pn_flags & ASTER_EIH) && c->P.precision != ASTER_FP64)
    return fail(c, ASTER_ERR_INVALID, "ASTER_EIH in ensembles needs precision ASTER_FP64 (exact mode)");
  const int wpb = c->batch.waves_per_block;
  const dim3 grid((P.nwaves + wpb - 1) / wpb), block(64 * wpb);
  const bool pn = (c->P.pn_flags & ASTER_PN_TERMS) != 0;
  const bool exact = c->P.precision == ASTER_FP64;
  const int team = P.pnf & ASTER_EIH ? 0 : team_size(P.nwaves, c->batch.round_max, P.pnf, exact);
  if (team) {
    auto kern = exact ? (team == 8 ? (pn ? k_batch_team<true, true, 8> : k_batch_team<false, true, 8>)
                                   : (pn ? k_batch_team<true, true, 4> : k_batch_team<false, true, 4>))
                      : (pn ? k_batch_team<true, false, 4>
                            : team == 8 ? k_batch_team<false, false, 8> : k_batch_team<false, false, 4>);
    hipLaunchKernelGGL(kern, dim3(P.nwaves), dim3(64 * (team + 3)), 0, c->stream, P);
  } else if (pn && exact) hipLaunchKernelGGL((k_batch<true, true>), grid, block, 0, c->stream, P);
  else if (pn) hipLaunchKernelGGL((k_batch<true, false>), grid, block, 0, c->stream, P);
  else if (exact) hipLaunchKernelGGL((k_batch<false, true>), grid, block, 0, c->stream, P);
  else hipLaunchKernelGGL((k_batch<false, false>), grid, block, 0, c->stream, P);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

static int launch_wh(aster_ctx* c, int phase, double dt, int64_t nsteps) {
  BatchState& B = c->batch;
  WhArgs P;
  P.nwaves = B.nwaves;
  P.lane_body = B.lane_body.p;
  P.lane_seg = B.lane_seg.p;
  P.wave_max = B.wave_max.p;
  P.x = B.x.p;
  P.v = B.v.p;
  P.a = B.a.p;
  P.m = B.m.p;
  P.nsteps = nsteps;
  P.dt = dt;
  P.G = c->P.G;
  P.soft = c->P.softening;
  P.phase = phase;
  const int wpb = B.waves_per_block;
  hipLaunchKernelGGL(k_batch_wh, dim3((P.nwaves + wpb - 1) / wpb), dim3(64 * wpb), 0, c->stream, P);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

static int substeps(int integrator, double dt, double* h) {
  if (integrator == ASTER_LEAPFROG) {
    h[0] = dt;
    h[1] = h[2] = 0.0;
    return 1;
  }
  double w[3];
  aster_yoshida_weights(w);
  for (int k = 0; k < 3; ++k) h[k] = w[k] * dt;
  return 3;
}

int batch_step(aster_ctx* c, int integrator, double dt, int64_t nsteps, int spl, int use_graph) {
  BatchState& B = c->batch;
  if (B.nsys == 0) return fail(c, ASTER_ERR_STATE, "no batch loaded");
  const bool wh = integrator == ASTER_WH_PLANETARY;
  if (integrator != ASTER_LEAPFROG && integrator != ASTER_YOSHIDA4 && !wh)
    return fail(c, ASTER_ERR_INVALID, "integrator must be ASTER_LEAPFROG, ASTER_YOSHIDA4 or ASTER_WH_PLANETARY");
  if (!std::isfinite(dt) || nsteps < 0 || spl < 0) return fail(c, ASTER_ERR_INVALID, "invalid dt, nsteps or spl");
  const bool pn = (c->P.pn_flags & ASTER_PN_TERMS) != 0;
  if ((c->P.pn_flags & ASTER_EIH) && c->P.precision != ASTER_FP64)
    return fail(c, ASTER_ERR_INVALID, "ASTER_EIH in ensembles needs precision ASTER_FP64 (exact mode)");
  if (wh && pn) return fail(c, ASTER_ERR_INVALID, "ASTER_WH_PLANETARY is Newtonian: post-Newtonian terms are not supported");
  if ((c->P.pn_flags & (ASTER_PN2 | ASTER_PN25)) && c->P.precision != ASTER_FP64)
    return fail(c, ASTER_ERR_INVALID, "ASTER_PN2 / ASTER_PN25 in ensembles need precision ASTER_FP64 (exact mode)");
  double h[3] = {0.0, 0.0, 0.0};
  const int nsub = wh ? 1 : substeps(integrator, dt, h);
  const double h0[3] = {0.0, 0.0, 0.0};
  int rc;
  if (!wh && !B.a_valid) {
    if ((rc = launch_batch(c, make_args(c, 0, 1, h0, 1)))) return rc;
    B.a_valid = true;
  }
  if (nsteps == 0) return ASTER_OK;
  if (spl == 0) spl = B.steps_per_launch > 0 ? B.steps_per_launch : 256;
  const int64_t full = nsteps / spl, rem = nsteps % spl;
  const int exact = c->P.precision == ASTER_FP64;
  // every launch of this call; Wisdom-Holman converts to heliocentric
  // coordinates before and back after (the accelerations are then stale)
  auto enqueue = [&]() -> int {
    int e = ASTER_OK;
    if (wh && (e = launch_wh(c, WH_ENTER, dt, 0))) return e;
    for (int64_t l = 0; l < full && !e; ++l)
      e = wh ? launch_wh(c, WH_STEPS, dt, spl) : launch_batch(c, make_args(c, spl, nsub, h, 0));
    if (!e && rem) e = wh ? launch_wh(c, WH_STEPS, dt, rem) : launch_batch(c, make_args(c, rem, nsub, h, 0));
    if (!e && wh) e = launch_wh(c, WH_EXIT, dt, 0);
    return e;
  };
  if (wh) B.a_valid = false;
  if (!use_graph) return enqueue();
  const bool same = B.exec && B.g_steps == nsteps && B.g_integrator == integrator && B.g_spl == spl &&
                    B.g_dt == dt && B.g_pn == c->P.pn_flags && B.g_exact == exact && B.g_wpb == B.waves_per_block &&
                    B.g_pack == B.pack && B.g_G == c->P.G && B.g_c == c->P.c && B.g_soft == c->P.softening;
  if (!same) {
    if (B.exec) ASTER_HIP(c, hipStreamSynchronize(c->stream));  // a replay of the old graph may still run
    drop_graph(B);
    ASTER_HIP(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
    const int lrc = enqueue();
    hipGraph_t g = nullptr;
    hipError_t e = hipStreamEndCapture(c->stream, &g);
    if (lrc) {
      if (g) (void)hipGraphDestroy(g);
      return lrc;
    }
    if (e != hipSuccess) return hip_fail(c, e, "hipStreamEndCapture");
    B.graph = g;
    ASTER_HIP(c, hipGraphInstantiate(&B.exec, B.graph, nullptr, nullptr, 0));
    B.g_steps = nsteps;
    B.g_integrator = integrator;
    B.g_spl = spl;
    B.g_dt = dt;
    B.g_pn = c->P.pn_flags;  // the captured arguments carry every force-law flag
    B.g_exact = exact;
    B.g_wpb = B.waves_per_block;
    B.g_pack = B.pack;
    B.g_G = c->P.G;
    B.g_c = c->P.c;
    B.g_soft = c->P.softening;
  }
  ASTER_HIP(c, hipGraphLaunch(B.exec, c->stream));
  return ASTER_OK;
}

int batch_energy(aster_ctx* c, double* e, double* L) {
  BatchState& B = c->batch;
  if (B.nsys == 0) return fail(c, ASTER_ERR_STATE, "no batch loaded");
  ASTER_HIP(c, B.ebody.reserve((size_t)4 * B.nbodies));
  ASTER_HIP(c, B.esys.reserve((size_t)4 * B.nsys));
  const double h0[3] = {0.0, 0.0, 0.0};
  const BatchArgs P = make_args(c, 0, 1, h0, 0);
  const int wpb = B.waves_per_block;
  hipLaunchKernelGGL(k_batch_energy, dim3((P.nwaves + wpb - 1) / wpb), dim3(64 * wpb), 0, c->stream, P,
                     (int)B.nbodies, B.ebody.p);
  ASTER_HIP(c, hipGetLastError());
  hipLaunchKernelGGL(k_batch_sum, dim3((unsigned)((B.nsys + 255) / 256)), dim3(256), 0, c->stream, B.nsys, B.doff.p,
                     B.nbodies, B.ebody.p, B.esys.p);
  ASTER_HIP(c, hipGetLastError());
  std::vector<double> h((size_t)4 * B.nsys);
  ASTER_HIP(c, hipMemcpyAsync(h.data(), B.esys.p, h.size() * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  for (int64_t s = 0; s < B.nsys; ++s) {
    if (e) e[s] = h[s];
    if (L)
      for (int q = 0; q < 3; ++q) L[3 * s + q] = h[(size_t)(1 + q) * B.nsys + s];
  }
  return ASTER_OK;
}

// Times 16 steps of every (packing, wavefronts-per-block) candidate on the
// loaded batch, restoring the state after each trial, and keeps the fastest.
// Steps per launch are then chosen so that one launch lasts about 20 ms.
int batch_autotune(aster_ctx* c, int integrator, double dt, int32_t* spb, int32_t* spl) {
  BatchState& B = c->batch;
  if (B.nsys == 0) return fail(c, ASTER_ERR_STATE, "no batch loaded");
  const size_t nb3 = (size_t)3 * B.nbodies;
  DBuf<double> save;
  ASTER_HIP(c, save.reserve(3 * nb3));
  int rc;
  const double h0[3] = {0.0, 0.0, 0.0};
  if (!B.a_valid) {
    if ((rc = launch_batch(c, make_args(c, 0, 1, h0, 1)))) return rc;
    B.a_valid = true;
  }
  ASTER_HIP(c, hipMemcpyAsync(save.p, B.x.p, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(save.p + nb3, B.v.p, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(save.p + 2 * nb3, B.a.p, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
  const bool wh = integrator == ASTER_WH_PLANETARY;
  double h[3] = {0.0, 0.0, 0.0};
  const int nsub = wh ? 1 : substeps(integrator, dt, h);
  const int trial = 16;
  float best = 1e30f;
  int best_pack = B.pack, best_wpb = B.waves_per_block;
  for (int pack = 0; pack <= 1; ++pack) {
    B.pack = pack;
    if ((rc = upload_plan(c))) return rc;
    for (int wpb = 1; wpb <= kBatchMaxWpb; wpb *= 2) {
      B.waves_per_block = wpb;
      if (wh && (rc = launch_wh(c, WH_ENTER, dt, 0))) return rc;
      rc = wh ? launch_wh(c, WH_STEPS, dt, 2) : launch_batch(c, make_args(c, 2, nsub, h, 0));  // warm
      if (rc) return rc;
      ASTER_HIP(c, hipEventRecord(c->ev[14], c->stream));
      rc = wh ? launch_wh(c, WH_STEPS, dt, trial) : launch_batch(c, make_args(c, trial, nsub, h, 0));
      if (rc) return rc;
      ASTER_HIP(c, hipEventRecord(c->ev[15], c->stream));
      ASTER_HIP(c, hipEventSynchronize(c->ev[15]));
      float ms = 0.f;
      ASTER_HIP(c, hipEventElapsedTime(&ms, c->ev[14], c->ev[15]));
      if (ms < best) {
        best = ms;
        best_pack = pack;
        best_wpb = wpb;
      }
      ASTER_HIP(c, hipMemcpyAsync(B.x.p, save.p, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
      ASTER_HIP(c, hipMemcpyAsync(B.v.p, save.p + nb3, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
      ASTER_HIP(c, hipMemcpyAsync(B.a.p, save.p + 2 * nb3, nb3 * 8, hipMemcpyDeviceToDevice, c->stream));
    }
  }
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  save.release();
  B.pack = best_pack;
  B.waves_per_block = best_wpb;
  if ((rc = upload_plan(c))) return rc;
  const double ms_per_step = best / trial;
  int s = (int)std::max(1.0, std::floor(20.0 / std::max(ms_per_step, 1e-6)));
  B.steps_per_launch = std::min(s, 100000);
  drop_graph(B);
  if (spb) *spb = B.waves_per_block;
  if (spl) *spl = B.steps_per_launch;
  return ASTER_OK;
}

// ------------------------------------------------- ensemble trajectory adjoint
// Leapfrog with Newtonian FP64 forces (fast mode arithmetic); the positions of
// every step are stored (small systems: 4096 three-body systems x 513 steps is
// 150 MB), so the backward pass evaluates each vector-Jacobian product at the
// exact forward positions. Recursion as in adjoint.hip:
//   lvh = lv + dt lx ; w = c_s lvh (c_s = dt, c_0 = dt/2)
//   lx += J(x_s)^T w [+ dL/dx_s] ; lm += M(x_s)^T w ; lv = lvh
// with, per body k and partner j in its system (d = x_j - x_k, s^2 = |d|^2 + eps^2):
//   J^T w : G sum_j [u/s^3 - 3 d (d.u)/s^5],  u = m_k w_j - m_j w_k
//   M^T w : -G sum_j (w_j . d)/s^3

// Both kernels evaluate every pair once: in round r = 1 .. n/2 a lane takes the
// pair of its body with the body r places on (cyclically in its system; an even
// system's last round covers each pair twice, the first half keeps theirs) and
// passes the partner's part over LDS. A three-body system, one round, needs
// one pair per lane and step instead of three sources of which one is the body
// itself. Bound: latency (4096 three-body systems are some 200 wavefronts on
// 1024 SIMDs, a serial chain per step), so the backward pass loads positions
// kTrajAhead steps ahead and nothing in the loop waits for loads or stores.
// 200 steps of 4096 three-body systems, forward / backward: three sources per
// lane 112 / 222 us; pairs once 90 / 97; snapshot steps kept as scalars and the
// look-ahead kept through the loop 66 / 93; in quads of lanes 44 / 50.
constexpr int kTrajAhead = 4;

// A lane's partner and the lane it receives from in round r.
struct CyclicPair {
  int to, from;
  bool own;  // this lane evaluates the pair
};
__device__ __forceinline__ CyclicPair cyclic_pair(int lane, int base, int cnt, int r, bool live) {
  const int i = lane - base;
  CyclicPair p;
  const bool in = live && 2 * r <= cnt;
  p.own = in && (2 * r < cnt || i < r);
  p.to = in ? (i + r < cnt ? lane + r : lane + r - cnt) : lane;
  p.from = in ? (i >= r ? lane - r : lane - r + cnt) : lane;
  return p;
}

// Systems of three bodies in quads of lanes (TRIPLES): the exchanges with the
// next and the previous body are lane permutations within the quad instead of
// LDS round trips; a quad's last lane is idle.
__device__ __forceinline__ double quad_next(double x) {  // lanes 0, 1, 2 <- 1, 2, 0
  const int lo = __builtin_amdgcn_mov_dpp((int)lo32(x), 0xC9, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)hi32(x), 0xC9, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double quad_prev(double x) {  // lanes 0, 1, 2 <- 2, 0, 1
  const int lo = __builtin_amdgcn_mov_dpp((int)lo32(x), 0xD2, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)hi32(x), 0xD2, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// A lane's body, its system's first lane and size, and the wavefront's rounds.
struct TrajLane {
  int b, base, cnt, rounds;
};
template <bool TRIPLES>
__device__ __forceinline__ TrajLane traj_lane(const BatchArgs& P, int64_t nbodies, int wave, int lane) {
  if (TRIPLES) {
    const int64_t b = (int64_t)(wave * 16 + (lane >> 2)) * 3 + (lane & 3);
    return {(lane & 3) < 3 && b < nbodies ? (int)b : -1, lane & ~3, 3, 1};
  }
  const int slot = wave * 64 + lane, seg = P.lane_seg[slot];
  return {P.lane_body[slot], seg >> 8, seg & 255, __builtin_amdgcn_readfirstlane(P.wave_max[wave]) >> 1};
}

// 1 / sqrt(x) by one third-order step from the estimate.
__device__ __forceinline__ double rsqrt64_cubic(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-(x * y), y, 1.0);
  return fma(y * e, fma(0.375, e, 0.5), y);
}

// Snapshot step q as a scalar: kept as a loaded vector, every comparison would
// wait for all earlier stores or loads of the wavefront.
__device__ __forceinline__ int64_t snap_step(const int64_t* snaps, int q) {
  const int64_t s = snaps[q];
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)s);
  const int hi = __builtin_amdgcn_readfirstlane((int)(s >> 32));
  return (int64_t)(((uint64_t)(uint32_t)hi << 32) | lo);
}

struct TrajArgs {
  double* traj;          // positions of every step
  double* v0;            // initial velocities
  const int64_t* snaps;  // snapshot steps
  int nsnap;
  double* snap_pos;  // positions of the snapshots, forward; gradients, backward
  int64_t nbodies, nsteps;
  double dt;
  double* out;  // gradients: positions, velocities, masses
  int nwaves;
};

// Launch shape: quads of lanes where every system has three bodies, otherwise
// the batch's own packing.
struct TrajShape {
  bool triples;
  int nwaves, wpb;
};
static TrajShape traj_shape(const BatchState& B) {
  if (B.triples) return {true, (int)((B.nsys + 15) / 16), 1};
  return {false, B.nwaves, B.waves_per_block};
}

template <bool TRIPLES>
__global__ __launch_bounds__(256) void k_batch_traj_fwd(BatchArgs P, TrajArgs Q) {
  constexpr int kLds = TRIPLES ? 1 : kBatchMaxWpb;
  __shared__ double4 sbody[kLds][64];  // position, mass
  __shared__ double4 spart[kLds][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wl;
  if (wave >= Q.nwaves) return;
  const TrajLane me = traj_lane<TRIPLES>(P, Q.nbodies, wave, lane);
  const int b = me.b, base = me.base, cnt = me.cnt;
  const bool live = b >= 0;
  double X[3] = {0.0, 0.0, 0.0}, V[3] = {0.0, 0.0, 0.0}, a[3];
  double mi = 0.0;
  if (live) {
    for (int c = 0; c < 3; ++c) {
      X[c] = P.x[3 * (size_t)b + c];
      V[c] = P.v[3 * (size_t)b + c];
      Q.v0[3 * (size_t)b + c] = V[c];
    }
    mi = P.m[b];
  }
  const double mnext = quad_next(mi);
  const CyclicPair first = cyclic_pair(lane, base, cnt, 1, live);
  auto pair = [&](const CyclicPair& p) {
    const double4 q = TRIPLES ? make_double4(quad_next(X[0]), quad_next(X[1]), quad_next(X[2]), mnext)
                              : sbody[wl][p.to];
    const double d[3] = {q.x - X[0], q.y - X[1], q.z - X[2]};
    const double r2 = fma(d[0], d[0], fma(d[1], d[1], fma(d[2], d[2], P.soft)));
    const double inv = rsqrt64_cubic(r2);
    const double inv3 = p.own ? inv * inv * inv : 0.0;
    const double fk = q.w * inv3, fj = mi * inv3;
    if (TRIPLES) {
#pragma unroll
      for (int c = 0; c < 3; ++c) a[c] = fma(fk, d[c], -quad_prev(fj * d[c]));
      return;
    }
    spart[wl][lane] = make_double4(fj * d[0], fj * d[1], fj * d[2], 0.0);
#pragma unroll
    for (int c = 0; c < 3; ++c) a[c] = fma(fk, d[c], a[c]);
    wave_sync();
    const double4 o = spart[wl][p.from];
    a[0] -= o.x;
    a[1] -= o.y;
    a[2] -= o.z;
    wave_sync();
  };
  auto accel = [&]() {  // over G
    if (!TRIPLES) {
      sbody[wl][lane] = make_double4(X[0], X[1], X[2], mi);
      wave_sync();
    }
    a[0] = a[1] = a[2] = 0.0;
    pair(first);
    for (int r = 2; r <= me.rounds; ++r) pair(cyclic_pair(lane, base, cnt, r, live));
  };
  int q = 0;
  int64_t next = Q.nsnap > 0 ? snap_step(Q.snaps, 0) : -1;
  double* at = Q.traj + 3 * (size_t)(live ? b : 0);
  auto store = [&](int64_t s) {
    if (live)
      for (int c = 0; c < 3; ++c) at[c] = X[c];
    at += 3 * Q.nbodies;
    if (s == next) {
      if (live)
        for (int c = 0; c < 3; ++c) Q.snap_pos[((size_t)q * Q.nbodies + b) * 3 + c] = X[c];
      next = ++q < Q.nsnap ? snap_step(Q.snaps, q) : -1;
    }
  };
  accel();
  store(0);
  // kick_drift_reg and kick_reg, with a G / 2 dt formed once for the kick before
  // the drift, the drift and the kick behind it (one fused kick from drift to
  // drift doubles the error of the positions, which is 1e-17)
  const double dt = Q.dt, half = 0.5 * P.G;
  auto drift = [&](bool kick) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const double t = half * a[c] * dt;
      if (kick) V[c] = V[c] + t;
      X[c] = X[c] + (V[c] * dt + t * dt);
      V[c] = V[c] + t;
    }
    accel();
  };
  drift(false);
  store(1);
  for (int64_t s = 1; s < Q.nsteps; ++s) {
    drift(true);
    store(s + 1);
  }
  if (live)
    for (int c = 0; c < 3; ++c) {
      P.x[3 * (size_t)b + c] = X[c];
      P.v[3 * (size_t)b + c] = V[c] + half * a[c] * dt;
    }
}

// Also puts the initial state back.
template <bool TRIPLES>
__global__ __launch_bounds__(256) void k_batch_traj_bwd(BatchArgs P, TrajArgs Q) {
  constexpr int kLds = TRIPLES ? 1 : kBatchMaxWpb;
  __shared__ double4 sbody[kLds][64];  // position, mass
  __shared__ double4 sw[kLds][64];
  __shared__ double4 spart[kLds][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + wl;
  if (wave >= Q.nwaves) return;
  const TrajLane me = traj_lane<TRIPLES>(P, Q.nbodies, wave, lane);
  const int b = me.b, base = me.base, cnt = me.cnt;
  const bool live = b >= 0;
  const double mk = live ? P.m[b] : 0.0;
  double lx[3] = {0.0, 0.0, 0.0}, lv[3] = {0.0, 0.0, 0.0}, lm = 0.0;
  int q = Q.nsnap - 1;
  int64_t next = q >= 0 ? snap_step(Q.snaps, q) : -1;
  auto snapshot = [&](int64_t s) {  // dL/dx at step s
    if (s != next) return;
    if (live)
      for (int c = 0; c < 3; ++c) lx[c] += Q.snap_pos[((size_t)q * Q.nbodies + b) * 3 + c];
    next = --q >= 0 ? snap_step(Q.snaps, q) : -1;
  };
  const double mnext = quad_next(mk);
  const CyclicPair first = cyclic_pair(lane, base, cnt, 1, live);
  // J^T w and M^T w of the pair over G c_s (w = lv) for body k = this lane's,
  // with u and d; both change sign for the partner, whose M^T w has the other w
  double g[3], gm;
  auto pair = [&](const CyclicPair& p, const double* X) {
    const double4 o = TRIPLES ? make_double4(quad_next(X[0]), quad_next(X[1]), quad_next(X[2]), mnext)
                              : sbody[wl][p.to];
    const double4 wo = TRIPLES ? make_double4(quad_next(lv[0]), quad_next(lv[1]), quad_next(lv[2]), 0.0)
                               : sw[wl][p.to];
    const double d[3] = {o.x - X[0], o.y - X[1], o.z - X[2]};
    const double r2 = fma(d[0], d[0], fma(d[1], d[1], fma(d[2], d[2], P.soft)));
    const double inv = rsqrt64_cubic(r2);
    const double inv2 = p.own ? inv * inv : 0.0;
    const double inv3 = p.own ? inv2 * inv : 0.0;
    const double u[3] = {fma(mk, wo.x, -(o.w * lv[0])), fma(mk, wo.y, -(o.w * lv[1])), fma(mk, wo.z, -(o.w * lv[2]))};
    const double du = 3.0 * inv2 * fma(d[0], u[0], fma(d[1], u[1], d[2] * u[2]));
    double t[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      t[c] = inv3 * fma(-d[c], du, u[c]);
      g[c] += t[c];
    }
    const double tm = inv3 * fma(d[0], lv[0], fma(d[1], lv[1], d[2] * lv[2]));
    gm = fma(-inv3, fma(d[0], wo.x, fma(d[1], wo.y, d[2] * wo.z)), gm);
    if (TRIPLES) {
#pragma unroll
      for (int c = 0; c < 3; ++c) g[c] -= quad_prev(t[c]);
      gm += quad_prev(tm);
      return;
    }
    spart[wl][lane] = make_double4(t[0], t[1], t[2], tm);
    wave_sync();
    const double4 q = spart[wl][p.from];
    g[0] -= q.x;
    g[1] -= q.y;
    g[2] -= q.z;
    gm += q.w;
    wave_sync();
  };
  const double dt = Q.dt, gdt = P.G * dt;
  auto step = [&](int64_t s, const double* X) {
#pragma unroll
    for (int c = 0; c < 3; ++c) lv[c] = fma(dt, lx[c], lv[c]);
    if (!TRIPLES) {
      sbody[wl][lane] = make_double4(X[0], X[1], X[2], mk);
      sw[wl][lane] = make_double4(lv[0], lv[1], lv[2], 0.0);
      wave_sync();
    }
    g[0] = g[1] = g[2] = gm = 0.0;
    pair(first, X);
    for (int r = 2; r <= me.rounds; ++r) pair(cyclic_pair(lane, base, cnt, r, live), X);
    const double gc = s > 0 ? gdt : 0.5 * gdt;
#pragma unroll
    for (int c = 0; c < 3; ++c) lx[c] = fma(gc, g[c], lx[c]);
    lm = fma(gc, gm, lm);
    snapshot(s);
  };
  double ahead[kTrajAhead][3];
  auto load = [&](int64_t s, double* X) {
    const size_t at = ((size_t)(s > 0 ? s : 0) * Q.nbodies + (live ? b : 0)) * 3;
#pragma unroll
    for (int c = 0; c < 3; ++c) X[c] = Q.traj[at + c];
  };
#pragma unroll
  for (int k = 0; k < kTrajAhead; ++k) load(Q.nsteps - 1 - k, ahead[k]);
  snapshot(Q.nsteps);
  int64_t s = Q.nsteps - 1;
  for (; s >= kTrajAhead - 1; s -= kTrajAhead) {
#pragma unroll
    for (int k = 0; k < kTrajAhead; ++k) {
      step(s - k, ahead[k]);
      load(s - k - kTrajAhead, ahead[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < kTrajAhead - 1; ++k)
    if (s - k >= 0) step(s - k, ahead[k]);
  if (live) {
    for (int c = 0; c < 3; ++c) {
      const size_t i = 3 * (size_t)b + c;
      Q.out[i] = lx[c];
      Q.out[3 * (size_t)Q.nbodies + i] = lv[c];
      P.x[i] = Q.traj[i];
      P.v[i] = Q.v0[i];
    }
    Q.out[6 * (size_t)Q.nbodies + b] = lm;
  }
}

int batch_traj_forward(aster_ctx* c, double dt, int64_t nsteps, int32_t nsnap, const int64_t* snaps,
                       double* snap_pos) {
  BatchState& B = c->batch;
  B.traj_ready = false;
  if (B.nsys == 0) return fail(c, ASTER_ERR_STATE, "no batch loaded");
  if (!std::isfinite(dt) || nsteps < 1 || nsnap < 0 || (nsnap > 0 && !snaps))
    return fail(c, ASTER_ERR_INVALID, "need dt finite, nsteps >= 1 and snapshot steps");
  for (int q = 0; q < nsnap; ++q)
    if (snaps[q] < 1 || snaps[q] > nsteps || (q > 0 && snaps[q] <= snaps[q - 1]))
      return fail(c, ASTER_ERR_INVALID, "snapshot steps must be ascending within [1, nsteps]");
  if (c->P.pn_flags & ASTER_PN_TERMS) return fail(c, ASTER_ERR_INVALID, "the adjoint covers Newtonian forces");
  const size_t nb3 = (size_t)3 * B.nbodies;
  if ((double)(nsteps + 1) * nb3 * 8.0 > 64e9) return fail(c, ASTER_ERR_CAPACITY, "trajectory would exceed 64 GB");
  ASTER_HIP(c, B.traj.reserve((size_t)(nsteps + 1) * nb3));
  ASTER_HIP(c, B.v0.reserve(nb3));
  ASTER_HIP(c, B.tgrad.reserve(std::max<size_t>(1, nsnap * nb3)));
  ASTER_HIP(c, B.tsnap.reserve(std::max(1, nsnap)));
  if (nsnap > 0) ASTER_HIP(c, hipMemcpyAsync(B.tsnap.p, snaps, nsnap * 8, hipMemcpyHostToDevice, c->stream));
  const double h[3] = {dt, 0.0, 0.0};
  const BatchArgs P = make_args(c, nsteps, 1, h, 0);
  const TrajShape t = traj_shape(B);
  const TrajArgs Q{B.traj.p, B.v0.p, B.tsnap.p, nsnap, B.tgrad.p, B.nbodies, nsteps, dt, nullptr, t.nwaves};
  hipLaunchKernelGGL(t.triples ? k_batch_traj_fwd<true> : k_batch_traj_fwd<false>,
                     dim3((t.nwaves + t.wpb - 1) / t.wpb), dim3(64 * t.wpb), 0, c->stream, P, Q);
  ASTER_HIP(c, hipGetLastError());
  B.a_valid = false;  // this kernel's accelerations have not the bits of batch_step's
  if (snap_pos && nsnap > 0)
    ASTER_HIP(c, hipMemcpyAsync(snap_pos, B.tgrad.p, nsnap * nb3 * 8, hipMemcpyDeviceToHost, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  B.traj_snaps.assign(snaps, snaps + nsnap);
  B.traj_steps = nsteps;
  B.traj_dt = dt;
  B.traj_G = P.G;
  B.traj_soft = P.soft;
  B.traj_ready = true;
  return ASTER_OK;
}

int batch_traj_backward(aster_ctx* c, const double* gsnap, double* gx, double* gv, double* gm) {
  BatchState& B = c->batch;
  if (!B.traj_ready) return fail(c, ASTER_ERR_STATE, "call aster_batch_traj_forward first");
  const int nsnap = (int)B.traj_snaps.size();
  if (nsnap > 0 && !gsnap) return fail(c, ASTER_ERR_INVALID, "snapshot gradients required");
  const size_t nb3 = (size_t)3 * B.nbodies;
  ASTER_HIP(c, B.tout.reserve(7 * (size_t)B.nbodies));
  if (nsnap > 0)
    ASTER_HIP(c, hipMemcpyAsync(B.tgrad.p, gsnap, nsnap * nb3 * 8, hipMemcpyHostToDevice, c->stream));
  const double h0[3] = {0.0, 0.0, 0.0};
  BatchArgs P = make_args(c, 0, 1, h0, 0);
  P.G = B.traj_G;
  P.soft = B.traj_soft;
  const TrajShape t = traj_shape(B);
  const TrajArgs Q{B.traj.p, B.v0.p, B.tsnap.p, nsnap, B.tgrad.p, B.nbodies, B.traj_steps, B.traj_dt, B.tout.p,
                   t.nwaves};
  hipLaunchKernelGGL(t.triples ? k_batch_traj_bwd<true> : k_batch_traj_bwd<false>,
                     dim3((t.nwaves + t.wpb - 1) / t.wpb), dim3(64 * t.wpb), 0, c->stream, P, Q);
  ASTER_HIP(c, hipGetLastError());
  if (gx) ASTER_HIP(c, hipMemcpyAsync(gx, B.tout.p, nb3 * 8, hipMemcpyDeviceToHost, c->stream));
  if (gv) ASTER_HIP(c, hipMemcpyAsync(gv, B.tout.p + nb3, nb3 * 8, hipMemcpyDeviceToHost, c->stream));
  if (gm) ASTER_HIP(c, hipMemcpyAsync(gm, B.tout.p + 2 * nb3, B.nbodies * 8, hipMemcpyDeviceToHost, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  B.a_valid = false;
  B.traj_ready = false;
  return ASTER_OK;
}

}  // namespace aster

using namespace aster;

extern "C" {

int aster_batch_set(aster_ctx* c, int64_t nsys, const int64_t* offsets, const double* pos, const double* vel,
                    const double* mass) {
  if (!c) return ASTER_ERR_INVALID;
  if (nsys < 1 || !offsets || !pos || !mass) return fail(c, ASTER_ERR_INVALID, "need nsys >= 1, offsets, pos, mass");
  if (offsets[0] != 0) return fail(c, ASTER_ERR_INVALID, "offsets[0] must be 0");
  bool triples = true;
  for (int64_t s = 0; s < nsys; ++s) {
    const int64_t k = offsets[s + 1] - offsets[s];
    if (k < 1 || k > 64) return fail(c, ASTER_ERR_CAPACITY, "each system needs 1..64 bodies");
    triples = triples && k == 3;
  }
  const int64_t nb = offsets[nsys];
  if (nb > (int64_t(1) << 28)) return fail(c, ASTER_ERR_CAPACITY, "at most 2^28 bodies per batch");
  for (int64_t i = 0; i < nb; ++i) {
    if (!(mass[i] > 0.0) || !std::isfinite(mass[i])) return fail(c, ASTER_ERR_INVALID, "masses must be > 0");
    for (int q = 0; q < 3; ++q)
      if (!std::isfinite(pos[3 * i + q]) || (vel && !std::isfinite(vel[3 * i + q])))
        return fail(c, ASTER_ERR_NONFINITE, "non-finite position or velocity in input");
  }
  ASTER_HIP(c, hipSetDevice(c->device));
  BatchState& B = c->batch;
  drop_graph(B);
  B.traj_ready = false;  // a stored trajectory is that of the systems before
  B.nsys = nsys;
  B.nbodies = nb;
  B.offsets.assign(offsets, offsets + nsys + 1);
  B.triples = triples;
  ASTER_HIP(c, B.x.reserve(3 * nb));
  ASTER_HIP(c, B.v.reserve(3 * nb));
  ASTER_HIP(c, B.a.reserve(3 * nb));
  ASTER_HIP(c, B.m.reserve(nb));
  ASTER_HIP(c, B.doff.reserve(nsys + 1));
  ASTER_HIP(c, hipMemcpyAsync(B.x.p, pos, 3 * nb * 8, hipMemcpyHostToDevice, c->stream));
  if (vel)
    ASTER_HIP(c, hipMemcpyAsync(B.v.p, vel, 3 * nb * 8, hipMemcpyHostToDevice, c->stream));
  else
    ASTER_HIP(c, hipMemsetAsync(B.v.p, 0, 3 * nb * 8, c->stream));
  ASTER_HIP(c, hipMemsetAsync(B.a.p, 0, 3 * nb * 8, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(B.m.p, mass, nb * 8, hipMemcpyHostToDevice, c->stream));
  ASTER_HIP(c, hipMemcpyAsync(B.doff.p, offsets, (nsys + 1) * 8, hipMemcpyHostToDevice, c->stream));
  B.a_valid = false;
  return upload_plan(c);
}

int aster_batch_traj_forward(aster_ctx* c, double dt, int64_t nsteps, int32_t nsnap, const int64_t* snap_steps,
                             double* snap_pos) {
  if (!c) return ASTER_ERR_INVALID;
  ASTER_HIP(c, hipSetDevice(c->device));
  return batch_traj_forward(c, dt, nsteps, nsnap, snap_steps, snap_pos);
}

int aster_batch_traj_backward(aster_ctx* c, const double* grad_snap_pos, double* g_pos, double* g_vel,
                              double* g_mass) {
  if (!c) return ASTER_ERR_INVALID;
  ASTER_HIP(c, hipSetDevice(c->device));
  return batch_traj_backward(c, grad_snap_pos, g_pos, g_vel, g_mass);
}

int aster_batch_get(aster_ctx* c, double* pos, double* vel) {
  if (!c) return ASTER_ERR_INVALID;
  BatchState& B = c->batch;
  if (B.nsys == 0) return fail(c, ASTER_ERR_STATE, "no batch loaded");
  ASTER_HIP(c, hipSetDevice(c->device));
  if (pos) ASTER_HIP(c, hipMemcpyAsync(pos, B.x.p, 3 * B.nbodies * 8, hipMemcpyDeviceToHost, c->stream));
  if (vel) ASTER_HIP(c, hipMemcpyAsync(vel, B.v.p, 3 * B.nbodies * 8, hipMemcpyDeviceToHost, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  return ASTER_OK;
}

}  // extern "C"
