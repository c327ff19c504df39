// Kick/drift updates on the FP64 state, the FP32 shadow, energy and angular
// momentum reductions, the automatic Morton box and device error flags.
//
// The kick/drift arithmetic keeps the operation order of update_leapfrog
// (src/physics/tool_chain_impl.cpp:169-185):
//   x += v*dt + ((0.5*a)*dt)*dt ;  v += (0.5*a)*dt
// with contraction disabled, so given identical accelerations the device
// trajectory is bit-identical to the CPU path. The second half-kick of a step
// and the first half-kick of the next use the same accelerations, so they are
// applied in one pass (k_kick_drift with dt_prev != 0).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "device.hpp"

namespace aster {

// BOX: the block also writes the largest |coordinate| of its drifted bodies
// per axis to part[3 block + axis], the first stage of the automatic Morton
// box of the next force evaluation (k_box's partials for these positions).
template <bool BOX>
__global__ __launch_bounds__(256) void k_kick_drift(int n, double* __restrict__ x, double* __restrict__ v,
                                                    const double* __restrict__ a, double dt_prev, double dt,
                                                    uint32_t* __restrict__ flags, double* __restrict__ part) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (!BOX && i >= n) return;
  double mx[3] = {0.0, 0.0, 0.0};
  if (i < n) {
    bool finite = true;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const size_t k = (size_t)c * n + i;
      double xc = x[k], vc = v[k];
      kick_drift_1(xc, vc, a[k], dt_prev, dt);
      x[k] = xc;
      v[k] = vc;
      mx[c] = fabs(xc);
      finite = finite && isfinite(xc) && isfinite(vc);
    }
    if (!finite) atomicOr(flags, (uint32_t)FLAG_NONFINITE);
  }
  if (BOX) {
    __shared__ double wm[3][4];
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double r = mx[c];
      for (int off = 32; off > 0; off >>= 1) r = fmax(r, __shfl_xor(r, off, 64));
      if ((threadIdx.x & 63) == 0) wm[c][w] = r;
    }
    __syncthreads();
    if (threadIdx.x < 3) {
      const int c = threadIdx.x;
      part[3 * blockIdx.x + c] = fmax(fmax(wm[c][0], wm[c][1]), fmax(wm[c][2], wm[c][3]));
    }
  }
}

// One SABA stage after its force evaluation, as the per-body lambdas of
// update_SABAn (src/integrators/SABA.cpp:19-553): v += (a d) dt, then
// x += (v c) dt with the kicked v. kick = 0 is the sequence's opening drift.
// update_euler (tool_chain_impl.cpp:158-167) is d = c = 1, since (a 1) dt and
// (v 1) dt round exactly like a dt and v dt.
__global__ __launch_bounds__(256) void k_saba_stage(int n, double* __restrict__ x, double* __restrict__ v,
                                                    const double* __restrict__ a, int kick, double d, double cdrift,
                                                    double cd_next, double dt, uint32_t* __restrict__ flags) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  bool finite = true;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const size_t k = (size_t)c * n + i;
    double xc = x[k], vc = v[k];
    if (kick) {
      saba_1(xc, vc, a[k], d, cdrift, cd_next, dt);
      v[k] = vc;
    } else {
      xc = xc + vc * cdrift * dt;
    }
    x[k] = xc;
    finite = finite && isfinite(xc) && isfinite(vc);
  }
  if (!finite) atomicOr(flags, (uint32_t)FLAG_NONFINITE);
}

__global__ __launch_bounds__(256) void k_kick(int n, double* __restrict__ v, const double* __restrict__ a,
                                              double dt) {
#pragma clang fp contract(off)
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const size_t k = (size_t)c * n + i;
    v[k] = kick_1(v[k], a[k], dt);
  }
}

// Energy sums. Tile a of 64 bodies meets the tiles b >= a, so every pair counts
// once: block (a, y) of one wavefront takes the `strip` tiles from a + y strip
// on, one target per lane, the sources through LDS. It writes the wavefront's
// sums of G m_i m_j / (|r| + soft) and G m_i m_j / sqrt(r^2 + soft) to
// part[0/1][y ntiles + a], and for y = 0 those of the kinetic energy and of m x
// cross v to rows[0..3][a]. Every sum has a fixed order. Bound: FP64 issue at
// many bodies, latency at few. An aster_energy call (with a readback of about 25
// us), against one thread per body over all sources (every pair twice) and two
// readbacks: n = 1000 331 -> 44 us, 4096 1205 -> 59 us, 20011 5.83 -> 0.37 ms,
// 65536 20.6 -> 3.3 ms (1.7 ms unsoftened, where the two pair terms are one);
// with exact roots, a range check per term and IEEE fallbacks in line 4.4 (2.5) ms.
__device__ __forceinline__ double wave_sum64(double v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// N pair terms 1 / sqrt(r^2 + soft) and (SOFT) 1 / (|r| + soft): to about one
// unit in the last place by Newton and third-order steps from the estimates,
// with one look at the range for all of a wavefront's N (r^2 within 2^+-600;
// `plain` when the softening is beyond that).
__device__ __forceinline__ bool energy_range(double x) { return hi32(x) - 0x1a700000u < 0x65700000u - 0x1a700000u; }

template <int N, bool SOFT>
__device__ __forceinline__ void energy_terms(const double* r2, double soft, bool plain, double* pl, double* pr) {
  bool in = !plain;
#pragma unroll
  for (int u = 0; u < N; ++u) in = in && energy_range(r2[u]);
  if (__builtin_expect(__all(in), 1)) {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      const double x = r2[u] + soft;
      const double y = __builtin_amdgcn_rsq(x);
      const double e = fma(-(x * y), y, 1.0);
      pl[u] = fma(y * e, fma(0.375, e, 0.5), y);
      if (SOFT) {
        const double z = __builtin_amdgcn_rsq(r2[u]);
        double g = r2[u] * z, h = 0.5 * z;
        const double d = fma(-h, g, 0.5);
        g = fma(g, d, g);
        h = fma(h, d, h);
        const double q = fma(fma(-g, g, r2[u]), h, g) + soft;  // |r| + soft
        double w = __builtin_amdgcn_rcp(q);
        w = fma(fma(-q, w, 1.0), w, w);
        pr[u] = fma(fma(-q, w, 1.0), w, w);
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < N; ++u) {
      pl[u] = 1.0 / sqrt(r2[u] + soft);
      if (SOFT) pr[u] = 1.0 / (sqrt(r2[u]) + soft);
    }
  }
}

template <bool SOFT>
__global__ __launch_bounds__(64) void k_energy_pairs(int n, int ntiles, int strip, const double* __restrict__ x,
                                                     const double* __restrict__ v, const double* __restrict__ m,
                                                     double G, double soft, double* __restrict__ part,
                                                     double* __restrict__ rows) {
  __shared__ double4 tile[64];
  const int lane = threadIdx.x, a = blockIdx.x;
  const int i = a * 64 + lane, ii = min(i, n - 1);
  const double px = x[ii], py = x[n + ii], pz = x[2 * (size_t)n + ii];
  const double mi = i < n ? m[ii] : 0.0;
  const int b0 = a + (int)blockIdx.y * strip, b1 = min(b0 + strip, ntiles);
  auto fetch = [&](int b) {
    const int j = b * 64 + lane, jj = min(j, n - 1);
    return make_double4(x[jj], x[n + jj], x[2 * (size_t)n + jj], j < n ? m[jj] : 0.0);
  };
  const bool plain = soft != 0.0 && !energy_range(soft);
  double pref = 0.0, ppl = 0.0;
  double4 q = b0 < b1 ? fetch(b0) : make_double4(0.0, 0.0, 0.0, 0.0);
  for (int b = b0; b < b1; ++b) {
    wave_sync();
    tile[lane] = q;
    wave_sync();
    if (b + 1 < b1) q = fetch(b + 1);
    const int cnt = min(64, n - b * 64);
    const int from = b == a ? lane : -1;  // the pairs i < j of the tile with itself
    auto pairs = [&](int k, auto count) {
      constexpr int N = count();
      double r2[N], w[N], pl[N], pr[N];
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const double4 s = tile[k + u];
        const double dx = s.x - px, dy = s.y - py, dz = s.z - pz;
        r2[u] = fma(dx, dx, fma(dy, dy, dz * dz));
        w[u] = s.w;
      }
      energy_terms<N, SOFT>(r2, soft, plain, pl, pr);
#pragma unroll
      for (int u = 0; u < N; ++u) {
        const bool take = k + u > from;
        ppl += take ? w[u] * pl[u] : 0.0;
        if (SOFT) pref += take ? w[u] * pr[u] : 0.0;
      }
    };
    int k = 0;
    for (; k + 4 <= cnt; k += 4) pairs(k, std::integral_constant<int, 4>{});
    for (; k < cnt; ++k) pairs(k, std::integral_constant<int, 1>{});
  }
  const double gm = G * mi;
  const double sp = wave_sum64(i < n ? gm * ppl : 0.0);
  const double sr = SOFT ? wave_sum64(i < n ? gm * pref : 0.0) : sp;
  const size_t slot = (size_t)blockIdx.y * ntiles + a, slots = (size_t)gridDim.y * ntiles;
  if (lane == 0) {
    part[slot] = sr;
    part[slots + slot] = sp;
  }
  if (blockIdx.y == 0) {
    const double vx = v[ii], vy = v[n + ii], vz = v[2 * (size_t)n + ii];
    const double t[4] = {0.5 * mi * (vx * vx + vy * vy + vz * vz), mi * (py * vz - pz * vy), mi * (pz * vx - px * vz),
                         mi * (px * vy - py * vx)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const double w = wave_sum64(t[c]);
      if (lane == 0) rows[(size_t)c * ntiles + a] = w;
    }
  }
}

// out = {kinetic, 2 sum_{i<j} of the two pair terms, L}: one block, fixed order
// (strided per thread, wavefronts by a fixed tree, then their sums). The loads
// of a round are in flight together. (One sum after the other through LDS took
// 10.3 us at 4096 bodies, this 5.9 us.) out[6]: the error word, so that one readback
// serves both.
__global__ __launch_bounds__(1024) void k_energy_reduce(int slots, int ntiles, const double* __restrict__ part,
                                                        const double* __restrict__ rows,
                                                        const uint32_t* __restrict__ flags,
                                                        double* __restrict__ out) {
  __shared__ double sm[6][16];
  const int t = threadIdx.x;
  double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // two pair terms, four rows
  for (int i0 = t; i0 < slots; i0 += 4 * 1024) {
    double w[2][4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r) w[r][u] = part[(size_t)r * slots + min(i0 + u * 1024, slots - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int r = 0; r < 2; ++r) s[r] += i0 + u * 1024 < slots ? w[r][u] : 0.0;
  }
  for (int i = t; i < ntiles; i += 1024)
#pragma unroll
    for (int r = 0; r < 4; ++r) s[2 + r] += rows[(size_t)r * ntiles + i];
#pragma unroll
  for (int r = 0; r < 6; ++r) {
    const double w = wave_sum64(s[r]);
    if ((t & 63) == 0) sm[r][t >> 6] = w;
  }
  __syncthreads();
  if (t == 6) out[6] = (double)flags[0];
  if (t >= 6) return;
  double sum = 0.0;
#pragma unroll
  for (int w = 0; w < 16; ++w) sum += sm[t][w];
  out[t < 2 ? 1 + t : t == 2 ? 0 : t] = t < 2 ? 2.0 * sum : sum;
}

// Symmetric box: max |coordinate| per axis, in two stages (per-block maxima,
// then one block over those), so no two blocks contend for an address. fmax
// is exact and order-independent.
constexpr int kBoxBlocks = 1024;

__global__ __launch_bounds__(256) void k_box(int n, const double* __restrict__ x, double* __restrict__ part) {
  __shared__ double wm[3][4];
  double mx[3] = {0.0, 0.0, 0.0};
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
#pragma unroll
    for (int c = 0; c < 3; ++c) mx[c] = fmax(mx[c], fabs(x[(size_t)c * n + i]));
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    double r = mx[c];
    for (int off = 32; off > 0; off >>= 1) r = fmax(r, __shfl_xor(r, off, 64));
    if ((threadIdx.x & 63) == 0) wm[c][w] = r;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int c = threadIdx.x;
    part[3 * blockIdx.x + c] = fmax(fmax(wm[c][0], wm[c][1]), fmax(wm[c][2], wm[c][3]));
  }
}

// The final maximum in a launch of its own, for more partials than every
// workgroup of k_morton should read (kBoxSourceParts).
constexpr int kBoxFinishThreads = 1024;
__global__ __launch_bounds__(kBoxFinishThreads) void k_box_finish(BoxSource bs, double* __restrict__ box) {
  double b[3];
  box_final<kBoxFinishThreads>(bs, box, b, true);
}

__global__ void k_zero_u32(uint32_t* p, int k) {
  if ((int)threadIdx.x < k) p[threadIdx.x] = 0u;
}

// --------------------------------------------------------------- launch ----

int launch_reset_flags(aster_ctx* c) {
  hipLaunchKernelGGL(k_zero_u32, dim3(1), dim3(64), 0, c->stream, c->flags.p, 4);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

int launch_kick_drift(aster_ctx* c, double dt_prev, double dt, bool box) {
  const int n = (int)c->n;
  const int blocks = (n + 255) / 256;
  c->box_parts = 0;
  c->src_ready = SrcReady{};
  // (at least what launch_box reserves, so that it never reallocates the partials)
  if (box) ASTER_HIP(c, c->boxpart.reserve((size_t)3 * std::max(blocks, kBoxBlocks)));
  phase_begin(c, ASTER_PHASE_KICKDRIFT);
  if (box)
    hipLaunchKernelGGL(k_kick_drift<true>, dim3(blocks), dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->a.p, dt_prev,
                       dt, c->flags.p, c->boxpart.p);
  else
    hipLaunchKernelGGL(k_kick_drift<false>, dim3(blocks), dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->a.p, dt_prev,
                       dt, c->flags.p, nullptr);
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_KICKDRIFT);
  if (box) {
    c->box_parts = blocks;
    c->box_parts_x = c->x.p;
    c->box_parts_n = c->n;
  }
  return ASTER_OK;
}

int launch_saba_stage(aster_ctx* c, bool kick, double d, double cdrift, double dt, double cd_next) {
  const int n = (int)c->n;
  c->src_ready = SrcReady{};
  phase_begin(c, ASTER_PHASE_KICKDRIFT);
  hipLaunchKernelGGL(k_saba_stage, dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->a.p,
                     kick ? 1 : 0, d, cdrift, cd_next, dt, c->flags.p);
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_KICKDRIFT);
  return ASTER_OK;
}

int launch_kick(aster_ctx* c, double dt) {
  const int n = (int)c->n;
  hipLaunchKernelGGL(k_kick, dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->v.p, c->a.p, dt);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

int launch_post(aster_ctx* c, const StepPost& post, bool box) {
  switch (post.kind) {
    case POST_KICK_DRIFT: return launch_kick_drift(c, post.dt_prev, post.dt, box);
    case POST_KICK: return launch_kick(c, post.dt);
    case POST_SABA: return launch_saba_stage(c, true, post.d, post.cd, post.dt, post.cd_next);
    default: return ASTER_OK;
  }
}

int launch_energy(aster_ctx* c, double* out7) {
  const int n = (int)c->n;
  const int ntiles = (n + 63) / 64;
  // one tile per wavefront up to 128 tiles; above, strips that make about 32768
  // blocks, half of them past the last tile and at once done; from 32768 tiles on
  // one strip per tile, the longest first
  const int strip = ntiles <= 128 ? 1 : (int)(((int64_t)ntiles * ntiles + 32767) / 32768);
  const int ny = (ntiles + strip - 1) / strip;
  const size_t slots = (size_t)ny * ntiles;
  ASTER_HIP(c, c->ework.reserve(2 * slots + 4 * (size_t)ntiles));
  ASTER_HIP(c, c->eout.reserve(8));
  double* rows = c->ework.p + 2 * slots;
  auto k = c->P.softening != 0.0 ? k_energy_pairs<true> : k_energy_pairs<false>;
  hipLaunchKernelGGL(k, dim3(ntiles, ny), dim3(64), 0, c->stream, n, ntiles, strip, c->x.p, c->v.p, c->m.p, c->P.G,
                     c->P.softening, c->ework.p, rows);
  ASTER_HIP(c, hipGetLastError());
  hipLaunchKernelGGL(k_energy_reduce, dim3(1), dim3(1024), 0, c->stream, (int)slots, ntiles, (const double*)c->ework.p,
                     (const double*)rows, (const uint32_t*)c->flags.p, c->eout.p);
  ASTER_HIP(c, hipGetLastError());
  ASTER_HIP(c, hipMemcpyAsync(out7, c->eout.p, 7 * sizeof(double), hipMemcpyDeviceToHost, c->stream));
  ASTER_HIP(c, hipStreamSynchronize(c->stream));
  return ASTER_OK;
}

int launch_box(aster_ctx* c, bool user_box, BoxSource* bs) {
  const int n = (int)c->n;
  ASTER_HIP(c, c->boxpart.reserve(3 * kBoxBlocks));
  ASTER_HIP(c, c->boxd.reserve(8));
  // A user box was uploaded to boxd[4..6] by aster_set_params.
  const bool user = user_box && (c->P.box[0] != 0.0 || c->P.box[1] != 0.0 || c->P.box[2] != 0.0);
  int blocks = 0;
  // Partials of these very positions left by the drift just before (same
  // state buffer and body count): only their final maximum remains.
  const bool fused = c->box_parts > 0 && c->box_parts_x == c->x.p && c->box_parts_n == c->n;
  if (!user && fused) {
    blocks = c->box_parts;
  } else if (!user) {
    blocks = (n + 255) / 256;
    if (blocks > kBoxBlocks) blocks = kBoxBlocks;
    hipLaunchKernelGGL(k_box, dim3(blocks), dim3(256), 0, c->stream, n, c->x.p, c->boxpart.p);
    ASTER_HIP(c, hipGetLastError());
  }
  c->box_parts = 0;
  *bs = user ? BoxSource{c->boxd.p + 4, 0} : BoxSource{c->boxpart.p, blocks};
  if (blocks > kBoxSourceParts) {
    hipLaunchKernelGGL(k_box_finish, dim3(1), dim3(kBoxFinishThreads), 0, c->stream, *bs, c->boxd.p);
    ASTER_HIP(c, hipGetLastError());
    *bs = BoxSource{c->boxd.p, 0};
  }
  return ASTER_OK;
}

}  // namespace aster
