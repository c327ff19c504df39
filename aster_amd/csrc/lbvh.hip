// LBVH Barnes-Hut on CDNA4: Morton codes -> LDS radix sort -> Karras radix
// tree -> moments by subtrees, bottom-up -> escape links -> stackless or
// wavefront-cooperative traversal.
//
// Tree layout follows the reference's NodesArray indexing
// (src/solvers/barnes_hut.cpp:309-400): leaf k is the body at sorted position
// k, the internal node of split i is n + i, the root is n.
//
// Parity notes:
//  * Morton codes use the reference's FP64 normalisation and clamp
//    (src/solvers/bh_specialization.cpp:38-46): bit-identical.
//  * The sort is a stable LSD radix sort, i.e. the (code, index) order.
//  * The Karras split uses the reference's tie-break on sorted positions
//    (barnes_hut.cpp:340-342) and its search sequence: identical topology.
//  * Moments: M = m_R + m_L, COM = (c_R m_R + c_L m_L) / M in FP64 without
//    contraction (barnes_hut.cpp:145-150). Each node depends only on its two
//    children, so the bottom-up order cannot change the result: node masses
//    and centres of mass are bit-identical to the recursive unite().
//  * Traversal: the reference visits right children first (it pushes left,
//    then right, barnes_hut.cpp:241-256). Opening goes to the right child and
//    every accepted/skipped node continues at its escape link, which is the
//    next node of that same order, so the FP64 traversal accumulates in the
//    reference's order and is bit-identical to get_node_body (:202-261).
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "device.hpp"

namespace aster {

// Depth bound of the radix tree: an internal node's split bit strictly
// increases with depth over 30 code bits + 32 tie-break bits, so depth <= 63.
constexpr int kMaxLevels = 128;
// Leaves per unit of the moments above the groups. Step of the group method, us,
// with units of 2048 / 4096 / 8192 / 16384 leaves: 4000 bodies 95.5 / 93.1 / 93.2 /
// 93.6, 50000 155.7 / 155.9 / 149.4 / 154.1, 2^20 974 / 917 / 904 / 923, 2^21 1845 /
// 1769 / 1697 / 1695.
constexpr int kUnit = 8192;
// Leaves per unit of the nodes above those, where there are more (k_moments_above).
constexpr int kBigUnit = 1 << 21;
// Traversal groups (and the moment kernel's per-wavefront subtrees): subtrees
// of at most kGroup leaves whose parent has more.
constexpr int kGroup = 64;

// ------------------------------------------------------------ Morton -------

__device__ __forceinline__ uint32_t part1by2(uint32_t v) {
  v = (v | (v << 16)) & 0x030000FFu;
  v = (v | (v << 8)) & 0x0300F00Fu;
  v = (v | (v << 4)) & 0x030C30C3u;
  v = (v | (v << 2)) & 0x09249249u;
  return v;
}

__device__ __forceinline__ uint32_t cell_of(double p, double b, uint32_t* bad) {
#pragma clang fp contract(off)
  const double q = (p + b) / (2 * b);
  const double s = q * (1 << 10);
  // The reference converts without a lower clamp (undefined for q < 0): such
  // inputs are reported instead of guessed.
  if (!(q >= 0.0) || !(s < 4294967296.0)) *bad = 1u;
  const uint32_t c = (uint32_t)s;
  return c < 1023u ? c : 1023u;
}

// -------------------------------------------------------- radix sort ------

// LSD radix sort of (Morton code, body) pairs, 3 passes of 10 bits. A
// workgroup takes a tile of consecutive keys: it forms its digits' starts
// from the tiles' digit counts (the keys of smaller digits in all tiles, those
// of the same digit in earlier tiles), ranks its keys, reorders them in LDS and
// writes them out. Counts are two digits to a word, at most a tile's keys each:
// row b of a pass's table holds tile b's 512 words. The first pass's rows come
// with the codes (k_morton), the later ones from k_rs_hist. With many tiles the
// rows are first summed over groups of kRsGroup (k_rs_groups), so that a tile
// reads the groups' sums and at most kRsGroup rows; with many groups these are
// scanned (k_rs_group_scan) and a tile reads two of them. Bound: latency below ~2^19
// keys (a scatter is one chain of loads, ranks and stores), with launches as
// long as they can be short. Against 4 passes of 8 bits with counts and keys in
// separate arrays: sort 54 -> 31 us at 50000 keys, 84 -> 65 us at 2^20. (Adding
// each key to its next tile's counts while scattering, instead of k_rs_hist,
// was slower: 50000 bodies +25 us, many equal keys +200 us at 20000.)
constexpr int kDigBits = 10;
constexpr int kDigits = 1 << kDigBits;
constexpr int kRsWords = kDigits / 2;
constexpr int kRsPasses = 3;
constexpr int kRsThreads = 512;
constexpr int kRsGroup = 32;
constexpr int kRsSmall = 4096;  // keys that one workgroup sorts by itself
constexpr int kRsMaxRows = 64;    // more tiles: in groups
constexpr int kRsMaxGroups = 16;  // more groups: their sums scanned
constexpr int kRsAhead = 8;

__device__ __forceinline__ uint32_t rs_digit(uint32_t key, int pass) {
  return (key >> (pass * kDigBits)) & (uint32_t)(kDigits - 1);
}

template <int K>
__global__ __launch_bounds__(kRsThreads) void k_rs_hist(const uint2* __restrict__ kv, int n, int pass,
                                               uint32_t* __restrict__ rows) {
  constexpr int T = kRsThreads;
  __shared__ uint32_t cnt[kRsWords];
  const int t = threadIdx.x;
  const int base = blockIdx.x * (T * K);
  // every load of the thread is issued before the first is used (clamped
  // addresses, no branch around a load), so the tile costs one memory round
  // trip rather than K
  uint32_t key[K];
#pragma unroll
  for (int r = 0; r < K; ++r) key[r] = kv[min(base + r * T + t, n - 1)].x;
  for (int i = t; i < kRsWords; i += T) cnt[i] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const uint32_t d = rs_digit(key[r], pass);
    if (base + r * T + t < n) atomicAdd(&cnt[d >> 1], 1u << (16 * (d & 1)));
  }
  __syncthreads();
  for (int i = t; i < kRsWords; i += T) rows[(size_t)blockIdx.x * kRsWords + i] = cnt[i];
}

// Sums of kRsGroup rows: {even digit, odd digit} per word. A workgroup takes
// kRsWords / kRsShare words; kRsShare threads share a word and take a run of
// rows each, so that all loads of a thread are in flight at once (64 rows, one
// thread per word and 8 rounds of loads: the sort's kernels at 2^20 72.3 us; 64 rows
// and 4 threads 67.1, 32 rows and 4 threads 64.5, 16 rows 65.6).
constexpr int kRsShare = 4;
__global__ __launch_bounds__(kRsWords) void k_rs_groups(const uint32_t* __restrict__ rows, int ntiles,
                                                        uint2* __restrict__ groups) {
  constexpr int kWords = kRsWords / kRsShare, kRows = kRsGroup / kRsShare;
  __shared__ uint2 part[kRsWords];
  const int t = threadIdx.x, word = blockIdx.y * kWords + t % kWords;
  const int b0 = blockIdx.x * kRsGroup + t / kWords * kRows;
  uint32_t c[kRows];
#pragma unroll
  for (int u = 0; u < kRows; ++u) c[u] = rows[(size_t)min(b0 + u, ntiles - 1) * kRsWords + word];
  uint2 s = make_uint2(0u, 0u);
#pragma unroll
  for (int u = 0; u < kRows; ++u)
    if (b0 + u < ntiles) {
      s.x += c[u] & 0xffffu;
      s.y += c[u] >> 16;
    }
  part[t] = s;
  __syncthreads();
  if (t < kWords) {
#pragma unroll
    for (int q = 1; q < kRsShare; ++q) {
      s.x += part[t + q * kWords].x;
      s.y += part[t + q * kWords].y;
    }
    groups[(size_t)blockIdx.x * kRsWords + word] = s;
  }
}

// The groups' sums turned into what precedes each group, their totals behind
// them (row ng): what the tiles read would otherwise grow as the square of the
// keys. A workgroup takes kRsScanWords words; the threads of a word take a run
// of groups each. Bound: latency, 4.6 us at 2^24 keys, 7.1 us at 2^26. The sort with
// the tiles summing all groups / with this: 2^21 keys (16 groups) 95 / 98 us,
// 3 10^6 137 / 130, 2^22 174 / 155, 2^24 973 / 480 us, 2^26 11.6 / 1.8 ms.
constexpr int kRsScanThreads = 1024;
constexpr int kRsScanWords = 16;
__global__ __launch_bounds__(kRsScanThreads) void k_rs_group_scan(uint2* __restrict__ groups, int ng) {
  constexpr int kRuns = kRsScanThreads / kRsScanWords;
  __shared__ uint2 part[kRuns][kRsScanWords];
  const int t = threadIdx.x, wd = t % kRsScanWords, r = t / kRsScanWords;
  const int word = blockIdx.x * kRsScanWords + wd;
  const int len = (ng + kRuns - 1) / kRuns, g0 = min(r * len, ng), g1 = min(g0 + len, ng);
  uint2 s = make_uint2(0u, 0u);
  for (int g = g0; g < g1; ++g) {
    const uint2 c = groups[(size_t)g * kRsWords + word];
    s.x += c.x;
    s.y += c.y;
  }
  part[r][wd] = s;
  __syncthreads();
  for (int off = 1; off < kRuns; off <<= 1) {  // inclusive sums over the runs
    uint2 y = make_uint2(0u, 0u);
    if (r >= off) y = part[r - off][wd];
    __syncthreads();
    part[r][wd].x += y.x;
    part[r][wd].y += y.y;
    __syncthreads();
  }
  uint2 run = r > 0 ? part[r - 1][wd] : make_uint2(0u, 0u);
  for (int g = g0; g < g1; ++g) {
    const uint2 c = groups[(size_t)g * kRsWords + word];
    groups[(size_t)g * kRsWords + word] = run;
    run.x += c.x;
    run.y += c.y;
  }
  if (r == kRuns - 1) groups[(size_t)ng * kRsWords + word] = run;
}

// Inclusive sum over the lanes of a wavefront.
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, int lane) {
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(v, off, 64);
    if (lane >= off) v += y;
  }
  return v;
}

// Ranks of the keys of a tile. Each wavefront owns 64 K consecutive keys (K
// rounds of 64, the first `left` of them valid) and ranks them among equal
// digits with its own running counters in LDS: rank = the wavefront's earlier
// keys of the digit (mine) + earlier lanes of the round (ballot match mask).
// LDS operations of one wavefront execute in order, so the rounds need no
// workgroup barrier.
typedef uint16_t __attribute__((may_alias)) Count16;
constexpr uint32_t kRsNone = 0xFFFFFFFFu;

template <int K>
__device__ __forceinline__ void rs_rank(const uint2 (&kv)[K], int left, int pass, int lane, Count16* mine,
                                        uint32_t (&pos)[K]) {
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const bool valid = r * 64 + lane < left;
    const uint32_t d = rs_digit(kv[r].x, pass);
    uint64_t m = __ballot(valid);
#pragma unroll
    for (int b = 0; b < kDigBits; ++b) {
      const bool bit = (d >> b) & 1u;
      const uint64_t bal = __ballot(bit);
      m &= bit ? bal : ~bal;
    }
    const uint32_t rank = (uint32_t)__popcll(m & lt);
    const uint32_t prev = mine[d];
    wave_sync();  // every lane has read its digit's count before the leaders update it
    if (valid && rank == 0) mine[d] = (Count16)(prev + (uint32_t)__popcll(m));
    wave_sync();
    pos[r] = valid ? prev + rank : kRsNone;  // rank among this wavefront's keys of digit d
  }
}

// A word's two digits: their totals in the tile (packed), each wavefront's
// counts turned into its offsets inside them.
template <int W>
__device__ __forceinline__ uint32_t rs_totals(uint32_t (*wcnt)[kRsWords], int word) {
  uint32_t run = 0;
#pragma unroll
  for (int v = 0; v < W; ++v) {
    const uint32_t c = wcnt[v][word];
    wcnt[v][word] = run;
    run += c;
  }
  return run;
}

// The whole sort in one workgroup, for up to T K keys: three passes through LDS
// instead of five launches. Step of the group method: 4096 bodies 117 -> 111 us,
// 2000 132 -> 125 us; at 8192 the five launches are as fast (129 and 130 us).
template <int T, int K>
__global__ __launch_bounds__(T) void k_rs_small(uint32_t* __restrict__ codes, uint32_t* __restrict__ idx, int n) {
  constexpr int W = T / 64;
  static_assert(T >= kRsWords && T * K <= 0xffff, "a word per thread, 16 bits per count");
  __shared__ uint32_t wcnt[W][kRsWords];
  __shared__ uint32_t lpre[kDigits];
  __shared__ uint32_t lsum[W];
  __shared__ uint2 skv[T * K];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int base = w * (64 * K);
  uint2 kv[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int p = min(base + r * 64 + lane, n - 1);
    kv[r] = make_uint2(codes[p], (uint32_t)p);
  }
  Count16* mine = reinterpret_cast<Count16*>(wcnt[w]);
  for (int pass = 0; pass < kRsPasses; ++pass) {
    for (int i = lane; i < kRsWords; i += 64) wcnt[w][i] = 0;
    wave_sync();
    uint32_t pos[K];
    rs_rank<K>(kv, n - base, pass, lane, mine, pos);
    __syncthreads();
    const bool owner = t < kRsWords;
    const uint32_t run = owner ? rs_totals<W>(wcnt, t) : 0u;
    const uint32_t both = (run & 0xffffu) + (run >> 16);
    const uint32_t inc = wave_scan(both, lane);
    if (lane == 63) lsum[w] = inc;
    __syncthreads();
    if (owner) {
      uint32_t l = inc - both;
      for (int v = 0; v < w; ++v) l += lsum[v];
      lpre[2 * t] = l;
      lpre[2 * t + 1] = l + (run & 0xffffu);
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r) {
      if (pos[r] == kRsNone) continue;
      const uint32_t d = rs_digit(kv[r].x, pass);
      skv[lpre[d] + mine[d] + pos[r]] = kv[r];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < K; ++r) kv[r] = skv[min(base + r * 64 + lane, n - 1)];
    // (the next pass writes skv only behind further barriers)
  }
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int p = base + r * 64 + lane;
    if (p >= n) continue;
    codes[p] = kv[r].x;
    idx[p] = kv[r].y;
  }
}

// Stable scatter. The tile's digit totals give each digit's start in the tile
// (lpre) and each wavefront's offset inside it; the tile is reordered by digit
// in LDS and written out with consecutive lanes on consecutive addresses within
// each digit's run.
enum { RS_ROWS = 0, RS_GROUPS = 1, RS_SCANNED = 2 };  // what a tile sums: all rows, the groups, neither

template <int K, int SUMS>
__global__ __launch_bounds__(kRsThreads) void k_rs_scatter(const uint32_t* __restrict__ codes, const uint2* __restrict__ kin,
                                                  uint2* __restrict__ kout, uint32_t* __restrict__ codes_out,
                                                  uint32_t* __restrict__ idx_out, int n, int pass,
                                                  const uint32_t* __restrict__ rows,
                                                  const uint2* __restrict__ groups, int ntiles) {
  constexpr int T = kRsThreads;
  constexpr int W = T / 64;        // wavefronts per tile
  constexpr int TILE = T * K;
  constexpr int Q = T / (kRsWords / 4);  // threads that share 4 words of the rows
  static_assert(TILE <= 0xffff, "16 bits per count");
  __shared__ uint32_t wcnt[W][kRsWords];
  __shared__ uint32_t gbase[kDigits];
  __shared__ uint32_t lpre[kDigits];
  __shared__ uint32_t gsum[W], lsum[W];
  __shared__ uint2 skv[TILE];
  const int t = threadIdx.x;
  const int lane = t & 63, w = t >> 6;
  const int blk = (int)blockIdx.x;
  // This wavefront's keys, loaded first (clamped addresses, no branch around a
  // load) so that their latency overlaps the digit starts. The first pass
  // takes the codes in body order.
  const int base = blk * TILE + w * (64 * K);
  uint2 kv[K];
  if (pass == 0) {
#pragma unroll
    for (int r = 0; r < K; ++r) {
      const int p = min(base + r * 64 + lane, n - 1);
      kv[r] = make_uint2(codes[p], (uint32_t)p);
    }
  } else {
#pragma unroll
    for (int r = 0; r < K; ++r) kv[r] = kin[min(base + r * 64 + lane, n - 1)];
  }
  // Digit starts: totals over all rows and what precedes this tile. Q threads
  // share 4 words (16 bytes) of every row and take the rows in turns, kRsAhead
  // loads at a time; adjacent lanes, so they add up by shuffles, and the first
  // four keep a word each.
  const int wg = t / Q, q = t - wg * Q;
  uint32_t pre[8] = {}, tot[8] = {};
  constexpr bool GROUPS = SUMS != RS_ROWS;
  const int ng = (ntiles + kRsGroup - 1) / kRsGroup, g = blk / kRsGroup;
  const uint4* __restrict__ gs = reinterpret_cast<const uint4*>(groups) + 2 * wg;
  if (SUMS == RS_SCANNED) {
    static_assert(Q >= 2, "a thread for the sums before the group, another for the totals");
    if (q < 2) {
      const size_t row = (size_t)(q == 0 ? g : ng) * (kDigits / 4);
      const uint4 c0 = gs[row], c1 = gs[row + 1];
      const uint32_t e[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        pre[v] = q == 0 ? e[v] : 0u;
        tot[v] = q == 1 ? e[v] : 0u;
      }
    }
  }
  if (SUMS == RS_GROUPS) {
    for (int b = q; b < ng; b += 2 * Q) {
      uint4 c[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) c[u] = gs[(size_t)min(b + u / 2 * Q, ng - 1) * (kDigits / 4) + u % 2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool in = b + u * Q < ng, before = b + u * Q < g;
        const uint4 &c0 = c[2 * u], &c1 = c[2 * u + 1];
        const uint32_t e[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
#pragma unroll
        for (int v = 0; v < 8; ++v) {
          tot[v] += in ? e[v] : 0u;
          pre[v] += before ? e[v] : 0u;
        }
      }
    }
  }
  const int b0 = GROUPS ? blk / kRsGroup * kRsGroup : 0, b1 = GROUPS ? blk : ntiles;
  const uint4* __restrict__ rw = reinterpret_cast<const uint4*>(rows) + wg;
  for (int b = b0 + q; b < b1; b += kRsAhead * Q) {
    uint4 c[kRsAhead];
#pragma unroll
    for (int u = 0; u < kRsAhead; ++u) c[u] = rw[(size_t)min(b + u * Q, b1 - 1) * (kRsWords / 4)];
#pragma unroll
    for (int u = 0; u < kRsAhead; ++u) {
      const bool in = b + u * Q < b1, before = b + u * Q < blk;
      const uint32_t e[4] = {c[u].x, c[u].y, c[u].z, c[u].w};
#pragma unroll
      for (int v = 0; v < 8; ++v) {
        const uint32_t d = v & 1 ? e[v >> 1] >> 16 : e[v >> 1] & 0xffffu;
        if (!GROUPS) tot[v] += in ? d : 0u;
        pre[v] += before && in ? d : 0u;
      }
    }
  }
  for (int i = t; i < W * kRsWords; i += T) (&wcnt[0][0])[i] = 0;
#pragma unroll
  for (int off = 1; off < Q; off <<= 1)
#pragma unroll
    for (int v = 0; v < 8; ++v) {
      pre[v] += __shfl_xor(pre[v], off, 64);
      tot[v] += __shfl_xor(tot[v], off, 64);
    }
  const bool owner = q < 4;
  const int word = 4 * wg + (q & 3);
  uint32_t pre0 = 0, pre1 = 0, tot0 = 0, tot1 = 0;
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (q == v) {
      pre0 = pre[2 * v];
      pre1 = pre[2 * v + 1];
      tot0 = tot[2 * v];
      tot1 = tot[2 * v + 1];
    }
  __syncthreads();
  Count16* mine = reinterpret_cast<Count16*>(wcnt[w]);
  uint32_t pos[K];
  rs_rank<K>(kv, n - base, pass, lane, mine, pos);
  __syncthreads();
  // the exclusive sums over the digits, in the tile and over all keys
  const uint32_t run = owner ? rs_totals<W>(wcnt, word) : 0u;
  const uint32_t linc = wave_scan((run & 0xffffu) + (run >> 16), lane);
  const uint32_t ginc = wave_scan(tot0 + tot1, lane);
  if (lane == 63) {
    lsum[w] = linc;
    gsum[w] = ginc;
  }
  __syncthreads();
  if (owner) {
    uint32_t l = linc - (run & 0xffffu) - (run >> 16), g = ginc - tot0 - tot1;
    for (int v = 0; v < w; ++v) {
      l += lsum[v];
      g += gsum[v];
    }
    lpre[2 * word] = l;
    lpre[2 * word + 1] = l + (run & 0xffffu);
    gbase[2 * word] = g + pre0;
    gbase[2 * word + 1] = g + tot0 + pre1;
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < K; ++r) {
    if (pos[r] == kRsNone) continue;
    const uint32_t d = rs_digit(kv[r].x, pass);
    skv[lpre[d] + mine[d] + pos[r]] = kv[r];
  }
  __syncthreads();
  const int valid_here = min(TILE, n - blk * TILE);
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int j = r * T + t;
    if (j >= valid_here) continue;
    const uint2 e = skv[j];
    const uint32_t d = rs_digit(e.x, pass);
    const uint32_t g = gbase[d] + ((uint32_t)j - lpre[d]);
    if (pass + 1 == kRsPasses) {
      codes_out[g] = e.x;
      idx_out[g] = e.y;
    } else {
      kout[g] = e;
    }
  }
}

// Lengths of the lists that k_build writes.
enum { ABOVE_UNITS = 0, ABOVE_TOP = 1, ABOVE_BIG = 2, ABOVE_CROWN = 3, ABOVE_COUNT = 4 };

// Also packs {x, y, z, m} of each body into one 32-byte record, so the leaf
// initialisation gathers one record through the sort permutation instead of
// four scattered planes. A workgroup takes a tile of the sort: it counts its
// codes' first digits into the tile's row. Every workgroup also takes the box's
// last maximum from the drift's partials (at 50000 bodies 5.7 -> 7.0 us against a
// launch of 4.4 us before it).
template <int K>
__global__ __launch_bounds__(kRsThreads) void k_morton(int n, const double* __restrict__ x, const double* __restrict__ m,
                                              BoxSource bs, double* __restrict__ box, uint32_t* __restrict__ codes,
                                              double4* __restrict__ xm, uint32_t* __restrict__ above,
                                              uint32_t* __restrict__ rows, uint32_t* __restrict__ flags) {
  constexpr int T = kRsThreads;
  __shared__ uint32_t cnt[kRsWords];
  const int t = threadIdx.x, base = blockIdx.x * (T * K);
  if (blockIdx.x == 0 && t < ABOVE_COUNT) above[t] = 0u;  // lengths of the lists that k_build writes
  for (int i = t; i < kRsWords; i += T) cnt[i] = 0u;
  double4 p[K];
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int i = min(base + r * T + t, n - 1);
    p[r] = make_double4(x[i], x[n + i], x[2 * n + i], m[i]);
  }
  double b[3];
  box_final<T>(bs, box, b, blockIdx.x == 0);
  uint32_t bad = 0;
#pragma unroll
  for (int r = 0; r < K; ++r) {
    const int i = base + r * T + t;
    if (i >= n) continue;
    const uint32_t ix = cell_of(p[r].x, b[0], &bad);
    const uint32_t iy = cell_of(p[r].y, b[1], &bad);
    const uint32_t iz = cell_of(p[r].z, b[2], &bad);
    const uint32_t code = (part1by2(iz) << 2) | (part1by2(iy) << 1) | part1by2(ix);
    xm[i] = p[r];
    codes[i] = code;
    const uint32_t d = rs_digit(code, 0);
    atomicAdd(&cnt[d >> 1], 1u << (16 * (d & 1)));
  }
  if (bad) atomicOr(flags, (uint32_t)FLAG_OUT_OF_BOX);
  __syncthreads();
  for (int i = t; i < kRsWords; i += T) rows[(size_t)blockIdx.x * kRsWords + i] = cnt[i];
}

// Traversal groups from the start flags, a byte per sorted position (16 a
// thread): start[g] = first position of group g, start[count] = n, and scan[p]
// = g where a group starts at p. Up to kGsOne positions a workgroup counts the
// flags before its chunk itself (16 bytes a thread and chunk), so that this is
// one launch; above, it sums the chunks' counts (k_group_counts). No block
// waits on another. Bound: launch and load latency. Step of the group method, us,
// with an exclusive scan of 4-byte flags in two launches / one launch / two:
// 4000 bodies 93.7 / 89.9 / 90.0, 20000 120.0 / 114.8 / 116.8, 50000 152.0 / 145.9
// / 147.7, 100000 200 / 191.8 / 193.0, 262144 323.8 / 318.4 / 317.3, 2^20 903 /
// 909 / 900.
constexpr int kGsThreads = 1024;
constexpr int kGsChunk = 16 * kGsThreads;
constexpr int kGsOneChunks = 8;
constexpr int kGsOne = kGsOneChunks * kGsChunk;
constexpr uint32_t kGsBits = 0x01010101u;

__device__ __forceinline__ uint32_t flag_count(const uint4& f) {
  return (uint32_t)__popc((f.x & kGsBits) | (f.y & kGsBits) << 1 | (f.z & kGsBits) << 2 | (f.w & kGsBits) << 3);
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Full chunks only: the last one's count is never needed.
__global__ __launch_bounds__(kGsThreads) void k_group_counts(const uint4* __restrict__ flag,
                                                             uint32_t* __restrict__ part) {
  __shared__ uint32_t ws[kGsThreads / 64];
  const uint32_t c = wave_sum(flag_count(flag[(size_t)blockIdx.x * kGsThreads + threadIdx.x]));
  if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t sum = 0;
    for (int q = 0; q < kGsThreads / 64; ++q) sum += ws[q];
    part[blockIdx.x] = sum;
  }
}

__global__ __launch_bounds__(kGsThreads) void k_group_starts(const uint4* __restrict__ flag, int n,
                                                             const uint32_t* __restrict__ part,
                                                             uint32_t* __restrict__ scan, uint32_t* __restrict__ total,
                                                             int32_t* __restrict__ start) {
  __shared__ uint32_t wpre[kGsThreads / 64], wsum[kGsThreads / 64];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  const int chunk = blockIdx.x;
  const int base = chunk * kGsChunk + 16 * t;
  const uint4 own = flag[min(base, n - 1) / 16];
  uint32_t pre = 0;
  if (part) {
    for (int b = t; b < chunk; b += kGsThreads) pre += part[b];
  } else if (chunk > 0) {
    uint4 f[kGsOneChunks - 1];
#pragma unroll
    for (int q = 0; q < kGsOneChunks - 1; ++q) f[q] = flag[min(q, chunk - 1) * kGsThreads + t];
#pragma unroll
    for (int q = 0; q < kGsOneChunks - 1; ++q) pre += q < chunk ? flag_count(f[q]) : 0u;
  }
  const int left = min(max(n - base, 0), 16);  // this thread's positions
  uint32_t bits = 0;
  const uint32_t word[4] = {own.x, own.y, own.z, own.w};
#pragma unroll
  for (int r = 0; r < 16; ++r) bits |= (word[r >> 2] >> 8 * (r & 3) & 1u) << r;
  bits &= (1u << left) - 1u;
  const uint32_t s = (uint32_t)__popc(bits);
  const uint32_t inc = wave_scan(s, lane);
  pre = wave_sum(pre);
  if (lane == 63) {
    wpre[w] = pre;
    wsum[w] = inc;
  }
  __syncthreads();
  uint32_t run = inc - s;
#pragma unroll
  for (int q = 0; q < kGsThreads / 64; ++q) run += wpre[q] + (q < w ? wsum[q] : 0u);
  for (uint32_t m = bits; m; m &= m - 1) {
    const int p = base + __ffs(m) - 1;
    start[run] = p;
    scan[p] = run++;
  }
  if (left > 0 && base + left == n) {
    *total = run;
    start[run] = n;
  }
}

// ------------------------------------------------------- Karras build ------

__device__ __forceinline__ int kdelta(const uint32_t* __restrict__ codes, int n, int i, int j) {
  if (j < 0 || j >= n) return -1;
  const uint32_t a = codes[i], b = codes[j];
  if (a == b) return 32 + __clz((uint32_t)(i ^ j));
  return __clz(a ^ b);
}

// Thread k initialises leaf k (body perm[k]) and, for k < n-1, the internal
// node n+k with its sorted-position range; with leaf_records also the parent
// links and the leaves' records (the per-body traversals need them). VEL
// also gathers the velocities (only the 1PN traversal reads node velocities).
// A node of more than kGroup leaves splits between two traversal groups:
// gflag marks the position behind its split as a group's first (every
// boundary is one node's split). Nodes of more than kUnit leaves are listed in
// `top`, the largest nodes of at most kUnit leaves above the groups in
// `units`, those of more than kBigUnit leaves in `crown` too, the largest
// between both sizes in `big`, in any order (lengths in `above`;
// k_moments_above).
template <bool VEL>
__global__ __launch_bounds__(256) void k_build(int n, const uint32_t* __restrict__ codes,
                                               const uint32_t* __restrict__ perm, const double4* __restrict__ xm,
                                               const double* __restrict__ v,
                                               int32_t* __restrict__ left, int32_t* __restrict__ right,
                                               int32_t* __restrict__ parent, int2* __restrict__ grange,
                                               double4* __restrict__ nmc, double4* __restrict__ nvel,
                                               float4* __restrict__ nbox, float4* __restrict__ nrec,
                                               float4* __restrict__ gsh, int32_t* __restrict__ splitnode,
                                               uint8_t* __restrict__ gflag, uint32_t* __restrict__ above,
                                               int32_t* __restrict__ units, int32_t* __restrict__ top,
                                               int32_t* __restrict__ big, int32_t* __restrict__ crown,
                                               uint32_t* __restrict__ flags, int leaf_records) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  {
    const uint32_t b = perm[k];
    const double4 pm = xm[b];
    const double px = pm.x, py = pm.y, pz = pm.z, mb = pm.w;
    nmc[k] = pm;
    if (VEL) nvel[k] = make_double4(v[b], v[n + b], v[2 * n + b], 0.0);
    const float fx = (float)px, fy = (float)py, fz = (float)pz;
    const float4 r = make_float4(fx, fy, fz, (float)mb);
    if (leaf_records) {  // the moment passes form a leaf's box from nmc themselves
      const float4 p = make_float4(fx, fy, fz, 0.f);
      nbox[2 * k] = p;
      nbox[2 * k + 1] = p;
      nrec[k] = r;
    }
    gsh[k] = r;
  }
  if (k == 0) {
    if (leaf_records) parent[n] = -1;
    gflag[0] = 1;
    if (n > kGroup && n <= kUnit) units[atomicAdd(&above[ABOVE_UNITS], 1u)] = n;
  }
  if (k >= n - 1) return;
  const int i = k;
  const int d_left = (i == 0) ? -1 : kdelta(codes, n, i, i - 1);
  const int d_right = kdelta(codes, n, i, i + 1);
  const int d = (d_right > d_left) ? 1 : -1;
  const int d_min = (d == 1) ? d_left : d_right;
  int l_max = 2;
  while (kdelta(codes, n, i, i + l_max * d) > d_min) l_max *= 2;
  int l = 0;
  for (int t = l_max / 2; t >= 1; t /= 2)
    if (kdelta(codes, n, i, i + (l + t) * d) > d_min) l += t;
  const int j = i + l * d;
  const int d_node = kdelta(codes, n, i, j);
  int s = 0;
  for (int t = (l + 1) / 2; t >= 1; t = (t + 1) / 2) {
    if (kdelta(codes, n, i, i + (s + t) * d) > d_node) s += t;
    if (t == 1) break;
  }
  const int gamma = i + s * d + min(d, 0);
  const int lo = min(i, j), hi = max(i, j);
  const int L = (lo == gamma) ? gamma : n + gamma;
  const int R = (hi == gamma + 1) ? gamma + 1 : n + gamma + 1;
  if (gamma < 0 || gamma > n - 2 || R >= 2 * n - 1) {  // cannot happen for a sorted key array
    atomicOr(flags, (uint32_t)FLAG_TREE);
    return;
  }
  left[n + i] = L;
  right[n + i] = R;
  if (leaf_records) {
    parent[L] = n + i;
    parent[R] = n + i;
  }
  grange[i] = make_int2(lo, hi);
  splitnode[gamma] = n + i;  // every split position belongs to exactly one internal node
  gflag[gamma + 1] = l + 1 > kGroup ? 1 : 0;
  if (l + 1 > kUnit) {
    top[atomicAdd(&above[ABOVE_TOP], 1u)] = n + i;
    const int cl = gamma - lo + 1, cr = hi - gamma;
    if (cl > kGroup && cl <= kUnit) units[atomicAdd(&above[ABOVE_UNITS], 1u)] = L;
    if (cr > kGroup && cr <= kUnit) units[atomicAdd(&above[ABOVE_UNITS], 1u)] = R;
    if (l + 1 > kBigUnit) {
      crown[atomicAdd(&above[ABOVE_CROWN], 1u)] = n + i;
      if (cl > kUnit && cl <= kBigUnit) big[atomicAdd(&above[ABOVE_BIG], 1u)] = L;
      if (cr > kUnit && cr <= kBigUnit) big[atomicAdd(&above[ABOVE_BIG], 1u)] = R;
    }
  }
}

// A node's moments: FP64 centre of mass and mass (and centre-of-mass velocity),
// FP32 bounding box.
struct MomRec {
  double4 com, vel;
  float4 lo, hi;
};

// The group traversal reads, for each internal node, its two children's
// records, node ids and thresholds from slots kid_slot(node, 0/1): opening a
// node costs one load of 64 contiguous bytes. The node that forms its moments
// writes its children's slots; the root has the extra slot 2 (n - 1).
__host__ __device__ inline int kid_slot(int n, int parent, int side) { return 2 * (parent - n) + side; }

// Geometric opening threshold of a node from its FP32 box and record: accept
// when d^2 > crit2 = (l / theta + delta)^2, l = longest AABB side, delta =
// |COM - AABB centre| (a leaf's degenerate box gives 0).
__device__ __forceinline__ float geo_crit2(const float4& lo, const float4& hi, const float4& r, double theta) {
#pragma clang fp contract(off)
  const float l = fmaxf(hi.x - lo.x, fmaxf(hi.y - lo.y, hi.z - lo.z));
  const float cx = 0.5f * (hi.x + lo.x);
  const float cy = 0.5f * (hi.y + lo.y);
  const float cz = 0.5f * (hi.z + lo.z);
  const float ex = r.x - cx, ey = r.y - cy, ez = r.z - cz;
  const float delta = sqrtf(ex * ex + ey * ey + ez * ez);
  const float q = l / (float)theta + delta;
  return q * q;
}

__device__ __forceinline__ float4 node_rec(const double4& com) {
  return make_float4((float)com.x, (float)com.y, (float)com.z, (float)com.w);
}

// The group traversal's child slot (see k_links): record, node id, threshold.
__device__ __forceinline__ void put_kid(float4* __restrict__ kids, int slot, int node, const double4& com,
                                        const float4& lo, const float4& hi, double theta) {
  const float4 r = node_rec(com);
  kids[2 * slot] = r;
  kids[2 * slot + 1] = make_float4(__int_as_float(node), geo_crit2(lo, hi, r, theta), 0.f, 0.f);
}

// A leaf's box is its position rounded to FP32 (what k_build would store).
__device__ __forceinline__ float4 leaf_box(const double4& com) {
  return make_float4((float)com.x, (float)com.y, (float)com.z, 0.f);
}

template <bool VEL>
__device__ __forceinline__ MomRec load_moments(int n, int node, const double4* __restrict__ nmc,
                                               const double4* __restrict__ nvel, const float4* __restrict__ nbox) {
  MomRec r;
  r.com = nmc[node];
  r.vel = VEL ? nvel[node] : make_double4(0.0, 0.0, 0.0, 0.0);
  if (node < n) {
    r.lo = r.hi = leaf_box(r.com);
  } else {
    r.lo = nbox[2 * node];
    r.hi = nbox[2 * node + 1];
  }
  return r;
}

template <bool VEL>
__device__ __forceinline__ MomRec unite_moments(const MomRec& cl, const MomRec& cr) {
#pragma clang fp contract(off)
  const double mR = cr.com.w, mL = cl.com.w;
  const double total = mR + mL;
  MomRec me;
  me.com = make_double4(0.0, 0.0, 0.0, 0.0);
  me.vel = make_double4(0.0, 0.0, 0.0, 0.0);
  if (total > 0) {
    me.com.w = total;
    me.com.x = (cr.com.x * mR + cl.com.x * mL) / total;
    me.com.y = (cr.com.y * mR + cl.com.y * mL) / total;
    me.com.z = (cr.com.z * mR + cl.com.z * mL) / total;
    if (VEL) {
      me.vel.x = (cr.vel.x * mR + cl.vel.x * mL) / total;
      me.vel.y = (cr.vel.y * mR + cl.vel.y * mL) / total;
      me.vel.z = (cr.vel.z * mR + cl.vel.z * mL) / total;
    }
  }
  me.lo = make_float4(fminf(cl.lo.x, cr.lo.x), fminf(cl.lo.y, cr.lo.y), fminf(cl.lo.z, cr.lo.z), 0.f);
  me.hi = make_float4(fmaxf(cl.hi.x, cr.hi.x), fmaxf(cl.hi.y, cr.hi.y), fmaxf(cl.hi.z, cr.hi.z), 0.f);
  return me;
}

// Moments of every internal node inside a traversal group, one wavefront per
// group. Internal node n+i's range starts or ends at i (Karras), so the
// hi - lo internal nodes of a group with leaf range [lo, hi] are n+lo ..
// n+hi-1 when the group's root is n+lo, and n+lo+1 .. n+hi when it is n+hi.
// Lane t owns node n+base+t; the lanes sweep bottom-up, a node being ready
// once both children are (leaves always are). Finished records stay in LDS
// for the parents in the same wavefront; leaves come from k_build. Same
// arithmetic as unite_moments, so the results are the same bits.
template <bool VEL>
__global__ __launch_bounds__(256) void k_group_moments(int n, const int32_t* __restrict__ gstart,
                                                       const uint32_t* __restrict__ gcount,
                                                       const int2* __restrict__ grange,
                                                       const int32_t* __restrict__ left,
                                                       const int32_t* __restrict__ right, double4* __restrict__ nmc,
                                                       double4* __restrict__ nvel, float4* __restrict__ nbox,
                                                       float4* __restrict__ nrec, double theta,
                                                       float4* __restrict__ kids) {
#pragma clang fp contract(off)
  __shared__ double4 smc[4][64];
  __shared__ double4 svel[VEL ? 4 : 1][64];
  __shared__ float4 slo[4][64], shi[4][64];
  __shared__ int sdone[4][64];
  const int wl = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int ngroups = (int)*gcount;
  const int stride = (int)gridDim.x * 4;
  for (int g = blockIdx.x * 4 + wl; g < ngroups; g += stride) {
    const int lo = gstart[g], hi = gstart[g + 1] - 1;
    const int nint = hi - lo;  // internal nodes of the group
    if (nint == 0) continue;   // a single leaf (uniform across the wavefront)
    bool root_lo = lo <= n - 2;
    if (root_lo) {
      const int2 r = grange[lo];
      root_lo = r.x == lo && r.y == hi;
    }
    const int base = root_lo ? lo : lo + 1;
    const bool mine = lane < nint;
    const int node = n + base + lane;
    int L = 0, R = 0;
    // leaf children are loaded before the sweep (one round trip); internal
    // children come from LDS as their lanes finish
    double4 cL = make_double4(0.0, 0.0, 0.0, 0.0), cR = cL, vL = cL, vR = cL;
    float4 loL = make_float4(0.f, 0.f, 0.f, 0.f), hiL = loL, loR = loL, hiR = loL;
    if (mine) {
      L = left[node];
      R = right[node];
      if (L < n) {
        cL = nmc[L];
        if (VEL) vL = nvel[L];
        loL = hiL = leaf_box(cL);
      }
      if (R < n) {
        cR = nmc[R];
        if (VEL) vR = nvel[R];
        loR = hiR = leaf_box(cR);
      }
    }
    bool done = !mine;
    sdone[wl][lane] = done ? 1 : 0;
    wave_sync();
    double4 com = make_double4(0.0, 0.0, 0.0, 0.0), vel = com;
    float4 blo = loL, bhi = loL;
    for (int it = 0; it < 64; ++it) {
      bool ready = false;
      if (!done) {
        const bool rl = L < n || sdone[wl][L - n - base];
        const bool rr = R < n || sdone[wl][R - n - base];
        ready = rl && rr;
      }
      if (ready) {
        if (L >= n) {
          cL = smc[wl][L - n - base];
          if (VEL) vL = svel[wl][L - n - base];
          loL = slo[wl][L - n - base];
          hiL = shi[wl][L - n - base];
        }
        if (R >= n) {
          cR = smc[wl][R - n - base];
          if (VEL) vR = svel[wl][R - n - base];
          loR = slo[wl][R - n - base];
          hiR = shi[wl][R - n - base];
        }
        const double mR = cR.w, mL = cL.w;
        const double total = mR + mL;
        if (total > 0) {
          com.w = total;
          com.x = (cR.x * mR + cL.x * mL) / total;
          com.y = (cR.y * mR + cL.y * mL) / total;
          com.z = (cR.z * mR + cL.z * mL) / total;
          if (VEL) {
            vel.x = (vR.x * mR + vL.x * mL) / total;
            vel.y = (vR.y * mR + vL.y * mL) / total;
            vel.z = (vR.z * mR + vL.z * mL) / total;
          }
        }
        blo = make_float4(fminf(loL.x, loR.x), fminf(loL.y, loR.y), fminf(loL.z, loR.z), 0.f);
        bhi = make_float4(fmaxf(hiL.x, hiR.x), fmaxf(hiL.y, hiR.y), fmaxf(hiL.z, hiR.z), 0.f);
        smc[wl][lane] = com;
        if (VEL) svel[wl][lane] = vel;
        slo[wl][lane] = blo;
        shi[wl][lane] = bhi;
        done = true;
      }
      wave_sync();
      if (ready) sdone[wl][lane] = 1;
      wave_sync();
      if (__ballot(!done) == 0ull) break;
    }
    if (mine) {
      nmc[node] = com;
      if (VEL) nvel[node] = vel;
      // With child slots (the group traversal) nobody reads nrec, nor the
      // box of a node below its group's root.
      if (!kids || node == n + (root_lo ? lo : hi)) {
        nbox[2 * node] = blo;
        nbox[2 * node + 1] = bhi;
      }
      if (!kids) nrec[node] = node_rec(com);
      if (kids) {  // this node's child slots (and the root's own slot)
        put_kid(kids, kid_slot(n, node, 0), L, cL, loL, hiL, theta);
        put_kid(kids, kid_slot(n, node, 1), R, cR, loR, hiR, theta);
        if (node == n) put_kid(kids, 2 * (n - 1), n, com, blo, bhi, theta);
      }
    }
  }
}

// Moments of the nodes above the groups, a workgroup per unit: first the nodes
// of the subtrees of at most kUnit leaves (MOM_UNITS; their splits are the
// boundaries between the groups inside), then all larger nodes in one workgroup
// (MOM_TOP, from the list `top`). Above kBigUnit bodies, where these are more
// than the workgroup has threads, those of the subtrees of at most kBigUnit
// leaves come before (MOM_BIG, each workgroup picks its own out of `top`), and
// the last workgroup takes what is left (`crown`). A thread takes a node, loads
// the records of its children that are complete (group roots, leaves, units'
// roots) and polls the other children's flags, one barrier per sweep; records
// pass through LDS. A flag holds the sweep its node was formed in, and only
// earlier sweeps count, so a sweep needs no second barrier and the records'
// order never depends on timing. More nodes than threads (a unit of many small
// groups, a very uneven tree): the threads take turns and the records pass
// through global memory. Bound: latency, ~4 dependent loads and a sweep per
// level (at most 47 levels up to 2^17 bodies: 30 code bits, 17 of position).
// Neither the host nor a level census is needed to order the launches: against
// the census (four launches, a readback and a wait), bands of levels and a top
// pass, the tree's part of a step falls from 167 to 127 us at 50000 bodies
// (these two launches 16 + 9 us) and from 331 to 280 us at 2^20 (15 + 30 us).
// With the records stored after the sweeps 12 + 7 and 12 + 23 us (units of 4096
// leaves), with units of 8192 13 + 16 us at 2^20. All moments without / with the
// big units, us: 2.2 10^6 bodies 148 / 149, 3 10^6 235 / 192, 2^22 315 / 261, 2^24
// 1097 / 890, 2^26 4333 / 3491 (bands of levels 294, 984 and 3789 at the last three).
template <bool VEL, int CAP>
struct MomLds {
  double4 com[CAP];
  double4 vel[VEL ? CAP : 1];
  float4 lo[CAP], hi[CAP];
  int done[CAP];
  __device__ void put(int s, const MomRec& r) {
    com[s] = r.com;
    if (VEL) vel[s] = r.vel;
    lo[s] = r.lo;
    hi[s] = r.hi;
  }
  __device__ void get(int s, MomRec& r) const {
    r.com = com[s];
    if (VEL) r.vel = vel[s];
    r.lo = lo[s];
    r.hi = hi[s];
  }
};

constexpr int kUnitThreads = 512;
constexpr int kTopThreads = 512;

// What a launch forms: the units' nodes, the big units' nodes above units, or
// every node of more than `small` leaves (kUnit: all of `top`, kBigUnit: `crown`).
enum { MOM_UNITS = 0, MOM_BIG = 1, MOM_TOP = 2 };
struct MomLists {
  const int32_t* units;  // MOM_UNITS, MOM_BIG: the roots
  const uint32_t* nunits;
  const int32_t* top;  // MOM_BIG, MOM_TOP: the nodes
  const uint32_t* ntop;
  int small;  // children of at most so many leaves are complete
};

template <bool VEL, int KIND>
__global__ __launch_bounds__(KIND == MOM_TOP ? kTopThreads : kUnitThreads) void k_moments_above(
    int n, MomLists lists, const int32_t* __restrict__ gstart, const uint32_t* __restrict__ gcount,
    const uint32_t* __restrict__ gscan, const int32_t* __restrict__ splitnode, const int32_t* __restrict__ left,
    const int32_t* __restrict__ right, const int2* __restrict__ grange, double4* nmc, double4* nvel, float4* nbox,
    float4* __restrict__ nrec, double theta, float4* __restrict__ kids, int32_t* topslot,
    uint32_t* __restrict__ flags) {
  constexpr bool UNITS = KIND == MOM_UNITS, BIG = KIND == MOM_BIG;
  constexpr int T = KIND == MOM_TOP ? kTopThreads : kUnitThreads;
  constexpr int kNever = 0xFFFF;
  __shared__ MomLds<VEL, T> lds;
  __shared__ uint16_t uslot[UNITS ? kUnit : 1];  // unit: node - n - lo -> thread, or its sweep
  __shared__ int mine_of[BIG ? T : 1];           // big unit: its nodes, while they are at most T
  __shared__ int mine_count;
  __shared__ int rslot;
  const int t = threadIdx.x;
  const int nunits = KIND == MOM_TOP ? 1 : (int)*lists.nunits;
  const int ntop = UNITS ? 0 : (int)*lists.ntop;
  for (int u = blockIdx.x; u < nunits; u += gridDim.x) {
    int root = n, ulo = 0, uhi = 0, g0 = 0, m = ntop;
    if (KIND != MOM_TOP) {
      root = lists.units[u];
      const int2 r = grange[root - n];
      ulo = r.x;
      uhi = r.y;
    }
    if (UNITS) {
      g0 = (int)gscan[ulo];
      m = (uhi + 1 < n ? (int)gscan[uhi + 1] : (int)*gcount) - g0 - 1;
    }
    // Entry e of the big unit's list: a node of `top` inside it, or -1. (Node
    // n + i covers position i; a larger node may cover the unit's first or last.)
    auto in_big = [&](int e) -> int {
      const int node = lists.top[e], i = node - n;
      if (i < ulo || i > uhi) return -1;
      const int2 r = grange[i];
      return r.x >= ulo && r.y <= uhi ? node : -1;
    };
    if (BIG) {
      if (t == 0) mine_count = 0;
      __syncthreads();
      for (int e = t; e < ntop; e += T) {
        const int node = in_big(e);
        if (node < 0) continue;
        const int at = atomicAdd(&mine_count, 1);
        if (at < T) mine_of[at] = node;
      }
      __syncthreads();
      m = mine_count;
    }
    // a node's entry: a unit's in LDS, the others' in global memory
    auto state_put = [&](int node, int v) {
      if (!UNITS) topslot[node - n] = v;
      else uslot[node - n - ulo] = (uint16_t)v;
    };
    auto state_get = [&](int node) -> int { return !UNITS ? topslot[node - n] : (int)uslot[node - n - ulo]; };
    struct Kids {
      int L, R;
      bool inL, inR;  // formed here
    };
    auto kids_of = [&](int node) {
      Kids k;
      k.L = left[node];
      k.R = right[node];
      const int2 r = grange[node - n];  // children cover [r.x, gamma] and [gamma + 1, r.y]
      const int gamma = k.L < n ? k.L : k.L - n;
      k.inL = k.L >= n && gamma - r.x + 1 > lists.small;
      k.inR = k.R >= n && r.y - gamma > lists.small;
      return k;
    };
    auto store = [&](int node, const Kids& k, const MomRec& cl, const MomRec& cr, const MomRec& me) {
      nmc[node] = me.com;
      if (VEL) nvel[node] = me.vel;
      nbox[2 * node] = me.lo;
      nbox[2 * node + 1] = me.hi;
      if (!kids) nrec[node] = node_rec(me.com);
      if (kids) {  // this node's child slots (and the root's own slot)
        put_kid(kids, kid_slot(n, node, 0), k.L, cl.com, cl.lo, cl.hi, theta);
        put_kid(kids, kid_slot(n, node, 1), k.R, cr.com, cr.lo, cr.hi, theta);
        if (node == n) put_kid(kids, 2 * (n - 1), n, me.com, me.lo, me.hi, theta);
      }
    };
    if (m <= 0) continue;  // uniform; cannot happen for a valid tree
    if (m <= T) {
      const bool mine = t < m;
      int node = root;
      Kids k{};
      MomRec cl{}, cr{}, me{};
      if (mine) {
        node = BIG ? mine_of[t] : UNITS ? splitnode[gstart[g0 + t + 1] - 1] : lists.top[t];
        state_put(node, t);
        if (node == root) rslot = t;
        k = kids_of(node);
      }
      lds.done[t] = kNever;
      __syncthreads();
      int sl = -1, sr = -1;
      if (mine) {
        if (k.inL) sl = state_get(k.L);
        else cl = load_moments<VEL>(n, k.L, nmc, nvel, nbox);
        if (k.inR) sr = state_get(k.R);
        else cr = load_moments<VEL>(n, k.R, nmc, nvel, nbox);
      }
      bool wait = mine;
      for (int it = 1;; ++it) {
        if (wait && (sl < 0 || lds.done[sl] < it) && (sr < 0 || lds.done[sr] < it)) {
          if (sl >= 0) lds.get(sl, cl);
          if (sr >= 0) lds.get(sr, cr);
          me = unite_moments<VEL>(cl, cr);
          lds.put(t, me);
          lds.done[t] = it;
          wait = false;
        }
        __syncthreads();
        if (lds.done[rslot] <= it) break;
        if (it >= kMaxLevels) {  // cannot happen for a valid tree
          if (t == 0) atomicOr(flags, (uint32_t)FLAG_TREE);
          break;
        }
      }
      if (mine) store(node, k, cl, cr, me);  // not in the sweeps: a barrier waits for stores
    } else {
      const int entries = BIG ? ntop : m;  // (a big unit's list does not fit: all of `top` every time)
      auto node_at = [&](int e) { return BIG ? in_big(e) : UNITS ? splitnode[gstart[g0 + e + 1] - 1] : lists.top[e]; };
      for (int e = t; e < entries; e += T) {
        const int node = node_at(e);
        if (node >= 0) state_put(node, kNever);
      }
      __syncthreads();
      for (int it = 1;; ++it) {
        for (int e = t; e < entries; e += T) {
          const int node = node_at(e);
          if (node < 0 || state_get(node) != kNever) continue;
          const Kids k = kids_of(node);
          if ((k.inL && state_get(k.L) >= it) || (k.inR && state_get(k.R) >= it)) continue;
          const MomRec cl = load_moments<VEL>(n, k.L, nmc, nvel, nbox);
          const MomRec cr = load_moments<VEL>(n, k.R, nmc, nvel, nbox);
          store(node, k, cl, cr, unite_moments<VEL>(cl, cr));
          state_put(node, it);
        }
        __syncthreads();
        const int rs = state_get(root);
        if (rs <= it) break;
        if (it >= kMaxLevels) {
          if (t == 0) atomicOr(flags, (uint32_t)FLAG_TREE);
          break;
        }
      }
    }
    __syncthreads();  // the unit's entries are read before the next unit's are written
  }
}

// Per node: traversal record = right child (or -1), escape link, opening
// threshold crit2 (accept when d^2 > crit2) and, for leaves, the body.
// mac 0 (parity): crit2 = (s / theta)^2 with s = |box| 2^-depth; the depth in the
//                 body's place for internal nodes.
// mac 1 (geometric): crit2 = (l / theta + delta)^2, l = longest AABB side,
//                    delta = |COM - AABB centre|.
// The escape link is the next node of the right-first preorder after the node's
// subtree: the left sibling of the nearest ancestor (or the node itself) that is
// a right child, so the left child of the node whose split lies just before
// the subtree's first position. (Walked up for together with the depth, in a
// launch of its own, at 150001 bodies 12.7 + 4.6 us; now 11.9 us.) Bound:
// latency of the walk for the depth.
template <int MAC>
__global__ __launch_bounds__(256) void k_links(int n, const int32_t* __restrict__ left,
                                               const int32_t* __restrict__ right, const int32_t* __restrict__ parent,
                                               const int2* __restrict__ grange, const int32_t* __restrict__ splitnode,
                                               const float4* __restrict__ nbox, const float4* __restrict__ nrec,
                                               const double* __restrict__ boxd, double theta,
                                               int4* __restrict__ nlink, const uint32_t* __restrict__ perm,
                                               uint32_t* __restrict__ flags) {
  const int node = blockIdx.x * blockDim.x + threadIdx.x;
  const int nn = 2 * n - 1;
  if (node >= nn) return;
  const int first = node < n ? node : grange[node - n].x;
  const int esc = first > 0 ? left[splitnode[first - 1]] : -1;
  float crit2;
  int dep = -1;
  if (MAC == 0) {
    dep = 0;
    for (int p = parent[node]; p >= 0; p = parent[p])
      if (++dep >= kMaxLevels - 1) {  // cannot happen for a valid tree
        atomicOr(flags, (uint32_t)FLAG_TREE);
        break;
      }
    const double s = ldexp(boxd[3], -dep);
    const double q = s / theta;
    crit2 = (float)(q * q);
  } else {
    crit2 = geo_crit2(nbox[2 * node], nbox[2 * node + 1], nrec[node], theta);
  }
  nlink[node] = make_int4(node < n ? -1 : right[node], esc, __float_as_int(crit2), node < n ? (int)perm[node] : dep);
}

// --------------------------------------------------------- traversals ------

// FP32 per-body stackless traversal (lanes = consecutive sorted bodies).
// Post-Newtonian terms of the FP32 traversals: for every node a body takes,
// the pairwise 1PN / 2PN / 2.5PN terms of compute_gravitational
// (tool_chain_impl.cpp:126-136) in FP64, with the node's FP64 centre of mass,
// mass and mass-weighted velocity as get_node_body takes them
// (barnes_hut.cpp:202-261; nodes at distance 0 skipped, :235), times 1/m_i,
// added to the FP32 Newtonian sums.
struct NodePn {
  const double4* nmc;   // FP64 {centre of mass, mass} per node (leaf k: body perm[k])
  const double4* nvel;  // FP64 mass-weighted velocity per node
  double G, ic, soft;
  int pnf;
};

// The terms from a node (record nc, velocity nv) on the body of leaf record
// pme / velocity vme.
__device__ __forceinline__ void node_pn_rec(const NodePn& p, const double4& nc, const double4& nv,
                                            const double4& pme, const double4& vme, double inv_m, double& ax,
                                            double& ay, double& az) {
#pragma clang fp contract(off)
  const double dx = nc.x - pme.x, dy = nc.y - pme.y, dz = nc.z - pme.z;
  const double d2 = dx * dx + dy * dy + dz * dz;
  if (d2 == 0.0) return;
  if (p.pnf == ASTER_PN1) {
    // the pairwise 1PN term alone: get_pn1 (tool_chain_impl.cpp:110-118) as an
    // acceleration, n = (x_i - x_node)/r, grouped for fused multiply-adds:
    //   G m2/r^2 [n (-v1^2 - 2 v2^2 + 4 v1.v2 + 3/2 (n.v2)^2 + (5 G m1 + 4 G m2)/r)
    //             + (v1 - v2)(4 n.v1 - 3 n.v2)] / c^2
    const double inv = rsqrt64(d2 + p.soft);
    const double nx = -dx * inv, ny = -dy * inv, nz = -dz * inv;
    const double nv1 = fma(nx, vme.x, fma(ny, vme.y, nz * vme.z));
    const double nv2 = fma(nx, nv.x, fma(ny, nv.y, nz * nv.z));
    const double v11 = fma(vme.x, vme.x, fma(vme.y, vme.y, vme.z * vme.z));
    const double v12 = fma(vme.x, nv.x, fma(vme.y, nv.y, vme.z * nv.z));
    const double v22 = fma(nv.x, nv.x, fma(nv.y, nv.y, nv.z * nv.z));
    double sc = fma(4.0, v12, -v11);
    sc = fma(-2.0, v22, sc);
    sc = fma(1.5 * nv2, nv2, sc);
    sc = fma(fma(4.0 * p.G, nc.w, 5.0 * p.G * pme.w), inv, sc);
    const double t = fma(4.0, nv1, -3.0 * nv2);
    const double k = p.G * nc.w * (inv * inv) * (p.ic * p.ic);
    ax = fma(fma(nx, sc, (vme.x - nv.x) * t), k, ax);
    ay = fma(fma(ny, sc, (vme.y - nv.y) * t), k, ay);
    az = fma(fma(nz, sc, (vme.z - nv.z) * t), k, az);
    return;
  }
  const double inv_r = 1.0 / sqrt(d2 + p.soft);
  double fx = 0.0, fy = 0.0, fz = 0.0;
  pn_add64(p.pnf, pme.w, nc.w, vme.x, vme.y, vme.z, nv.x, nv.y, nv.z, inv_r, -(dx * inv_r), -(dy * inv_r),
           -(dz * inv_r), p.G, p.ic, fx, fy, fz);
  ax += fx * inv_m;
  ay += fy * inv_m;
  az += fz * inv_m;
}

__device__ __forceinline__ void node_pn(const NodePn& p, int node, const double4& pme, const double4& vme,
                                        double inv_m, double& ax, double& ay, double& az) {
  node_pn_rec(p, p.nmc[node], p.nvel[node], pme, vme, inv_m, ax, ay, az);
}

template <bool MASK, bool PN>
__global__ __launch_bounds__(256) void k_bh_f32(int n, const float4* __restrict__ gsh, const float4* __restrict__ nrec,
                                                const int4* __restrict__ nlink, float eps2, float msc, double G,
                                                double* __restrict__ a, unsigned long long* __restrict__ counters,
                                                uint32_t* __restrict__ flags, NodePn pnp) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = k < n;
  const float4 me = gsh[live ? k : n - 1];
  float ax = 0.f, ay = 0.f, az = 0.f;
  double4 pme = make_double4(0.0, 0.0, 0.0, 1.0), vme = make_double4(0.0, 0.0, 0.0, 0.0);
  double pax = 0.0, pay = 0.0, paz = 0.0, inv_m = 1.0;
  if (PN) {
    pme = pnp.nmc[live ? k : n - 1];
    vme = pnp.nvel[live ? k : n - 1];
    inv_m = 1.0 / pme.w;
  }
  uint32_t inter = 0, visits = 0;
  int node = live ? n : -1;
  const uint32_t limit = 4u * (uint32_t)n + 16u;
  while (node >= 0) {
    if (visits > limit) {
      atomicOr(flags, (uint32_t)FLAG_TREE);
      break;
    }
    const float4 r = nrec[node];
    const int4 L = nlink[node];
    ++visits;
    const float dx = r.x - me.x, dy = r.y - me.y, dz = r.z - me.z;
    const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
    if (d2 == 0.f) {
      node = L.y;
      continue;
    }
    if (node < n || d2 > __int_as_float(L.z)) {
      const float r2 = d2 + eps2;
      float inv = __builtin_amdgcn_rsqf(r2);
      if (MASK) inv = (r2 > 0.f) ? inv : 0.f;
      const float f = ((r.w * msc) * inv) * (inv * inv);
      ax = fmaf(f, dx, ax);
      ay = fmaf(f, dy, ay);
      az = fmaf(f, dz, az);
      if (PN) node_pn(pnp, node, pme, vme, inv_m, pax, pay, paz);
      ++inter;
      node = L.y;
    } else {
      node = L.x;
    }
  }
  if (live) {
    const int b = nlink[k].w;
    a[b] = G * (double)ax + pax;
    a[n + b] = G * (double)ay + pay;
    a[2 * n + b] = G * (double)az + paz;
  }
  unsigned long long ci = inter, cv = visits;
  for (int off = 32; off > 0; off >>= 1) {
    ci += __shfl_xor(ci, off, 64);
    cv += __shfl_xor(cv, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&counters[BHC_INTERACTIONS], ci);
    atomicAdd(&counters[BHC_VISITS], cv);
  }
}

// FP64 per-body traversal in the reference's order and arithmetic
// (get_node_body, barnes_hut.cpp:202-261).
template <bool PN>
__global__ __launch_bounds__(256) void k_bh_f64(int n, const double* __restrict__ x, const double* __restrict__ v,
                                                const double* __restrict__ m, const double4* __restrict__ nmc,
                                                const double4* __restrict__ nvel, const int4* __restrict__ nlink,
                                                const double* __restrict__ boxd, double theta, double G, double ic,
                                                int pnf,
                                                double soft, double* __restrict__ a,
                                                unsigned long long* __restrict__ counters,
                                                uint32_t* __restrict__ flags) {
#pragma clang fp contract(off)
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = k < n;
  const int b = nlink[live ? k : n - 1].w;
  const double pix = x[b], piy = x[n + b], piz = x[2 * n + b];
  double vix = 0.0, viy = 0.0, viz = 0.0;
  if (PN) {
    vix = v[b];
    viy = v[n + b];
    viz = v[2 * n + b];
  }
  const double mi = m[b];
  const double inv_m = 1.0 / mi;
  const double theta2 = theta * theta;
  const double bd = boxd[3];
  double ax = 0.0, ay = 0.0, az = 0.0;
  uint32_t inter = 0, visits = 0;
  int node = live ? n : -1;
  const uint32_t limit = 4u * (uint32_t)n + 16u;
  // The next node's record is loaded as soon as the step is decided, before the
  // force of the node just taken (150001 bodies 77 -> 73 us: the loads' latency
  // along the longest walk is what remains).
  int4 L;
  double4 nc, nv = make_double4(0.0, 0.0, 0.0, 0.0);
  auto fetch = [&]() {
    const int q = max(node, 0);
    L = nlink[q];
    nc = nmc[q];
    if (PN) nv = nvel[q];
  };
  fetch();
  while (node >= 0) {
    if (visits > limit) {
      atomicOr(flags, (uint32_t)FLAG_TREE);
      break;
    }
    ++visits;
    const double cx = nc.x, cy = nc.y, cz = nc.z, cm = nc.w;
    const double vnx = nv.x, vny = nv.y, vnz = nv.z;
    const double dx = pix - cx, dy = piy - cy, dz = piz - cz;
    const double d2 = dx * dx + dy * dy + dz * dz;
    const double s = ldexp(bd, -L.w);  // an internal node's depth
    const bool skip = d2 == 0.0;
    const bool take = !skip && ((s * s < d2 * theta2) || node < n);
    node = skip || take ? L.y : L.x;
    fetch();
    if (take) {
      double fx, fy, fz;
      grav64(mi, cm, vix, viy, viz, vnx, vny, vnz, pix, piy, piz, cx, cy, cz, G, ic, soft, PN ? pnf : 0, fx, fy, fz);
      ax += fx * inv_m;
      ay += fy * inv_m;
      az += fz * inv_m;
      ++inter;
    }
  }
  if (live) {
    a[b] = ax;
    a[n + b] = ay;
    a[2 * n + b] = az;
  }
  unsigned long long ci = inter, cv = visits;
  for (int off = 32; off > 0; off >>= 1) {
    ci += __shfl_xor(ci, off, 64);
    cv += __shfl_xor(cv, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    atomicAdd(&counters[BHC_INTERACTIONS], ci);
    atomicAdd(&counters[BHC_VISITS], cv);
  }
}

// ------------------------------------------------------------- groups ------
//
// The wavefront traversal works on groups of bodies that share one walk. A
// group is a subtree of the radix tree with at most kGroup leaves whose
// parent has more: its bodies are contiguous in Morton order and lie in one
// Morton cell (the subtree's common code prefix), so the group box is compact
// wherever the curve jumps. Groups partition the sorted bodies.

// Cooperative traversal, one group (at most 64 bodies) per workgroup of W
// wavefronts; W = 1 in what follows, more in bh_forces_all's rule: W times the
// candidates per iteration, the list, the stack and the lanes that share its
// evaluation, by workgroup barriers. The wavefront walks the tree once for the
// whole group with a shared LDS stack of opened nodes, testing up to 64
// candidate nodes per iteration: lane 2 i + s takes child s of the i-th popped
// node from that node's child slots (record, id and threshold of both
// children in 64 contiguous bytes), so a batch costs one load round trip.
// A node is accepted when the distance from its centre of
// mass to the group's bounding box exceeds its opening radius (the geometric
// test, so it holds for every body of the group); leaves are always accepted.
// Accepted nodes are appended to an LDS interaction list that the lanes then
// evaluate in pieces (below; 12 VALU + 1 rsq per entry and lane), FP32 sums
// per list flush, Kahan-compensated across flushes.
// Stack bound: an iteration pops up to 32 entries and pushes their opened
// children, at most one more each than it popped. It pops no more than leave
// kGrpDeep entries free, but at least one: single entries walk depth first,
// which adds at most one entry per level, and internal nodes have at most 61
// levels (their common prefix grows by a bit or more per level: 30 bits of
// code, then 31 of the position). So the stack suffices for every tree.
// Scheduling: the 8 XCDs take workgroups round-robin, so workgroup b works on
// the groups of chunk (b mod 8), consecutive in Morton order, and neighbouring
// groups (which open the same nodes) share an L2.
// List evaluation in pieces: the g bodies of a group would leave 64 - g lanes
// idle if each body took one lane through the whole list (groups average ~42
// bodies). Instead each body's list is cut into q pieces of equal length
// (lam = ceil(m / q), the list padded with zero-mass entries, which add exactly
// zero force), and the g q pieces are spread over P passes of the 64 lanes:
// slot j = 64 p + lane of pass p takes piece j mod q of body j / q (slots past
// g q repeat piece 0 of the last body and are discarded). Every lane of a pass
// runs the same lam iterations, so the loop stays uniform. After the passes
// the partial sums go to LDS and body b adds its pieces b q .. b q + q - 1 in
// that order (deterministic). (P, q) depends only on g and is chosen, for a
// list of ~96 entries, to minimise P (lam + 1) with P <= 3 and q <= 64; g = 64
// gives P = q = 1, g = 42 gives P = 2, q = 3 (98% of the lanes busy instead
// of 66%). Lane use over a 2^20-body tree, from the rsq count: 90.5% (73%
// with a power-of-two number of lanes per body of a group of <= 32).
// The list holds up to kGrpList entries (flushed once it has more than
// kGrpList - 64, since one round adds at most 64) plus the padding (< q <= 64
// entries); the same LDS holds the P 64 partial sums after the passes.
// 256-entry lists, a 4th pass and a smaller stack (more waves per CU) each
// measured within 1%: the kernel is VALU-issue bound.
constexpr int kGrpList = 128;
constexpr int kGrpListPad = 64;  // room for that padding
constexpr int kPieceMaxPasses = 3;
static_assert(kPieceMaxPasses * 64 <= kGrpList + kGrpListPad, "partial sums must fit the list LDS");

constexpr int kGrpStack = 384;
constexpr int kGrpDeep = 62;

struct PieceTable {
  uint8_t passes[65];
  uint8_t pieces[65];
};

constexpr PieceTable make_piece_table(int waves) {
  PieceTable t{};
  for (int g = 1; g <= 64; ++g) {
    int best = 1 << 30, bp = 1, bq = 1;
    for (int p = 1; p <= kPieceMaxPasses; ++p) {
      int q = (64 * waves * p) / g;
      if (q > 64) q = 64;
      const int cost = p * ((96 * waves + q - 1) / q + 1);
      if (cost < best) {
        best = cost;
        bp = p;
        bq = q;
      }
    }
    t.passes[g] = (uint8_t)bp;
    t.pieces[g] = (uint8_t)bq;
  }
  return t;
}

template <int W>
__constant__ PieceTable kPieces = make_piece_table(W);

// One piece: lam list entries from `p` against the body at `me`.
template <bool MASK>
__device__ __forceinline__ void group_piece_sum(const float4* __restrict__ p, int lam, const float4& me,
                                                float eps2, float& tx, float& ty, float& tz) {
#pragma unroll 4
  for (int e = 0; e < lam; ++e) {
    const float4 q = p[e];
    const float dx = q.x - me.x, dy = q.y - me.y, dz = q.z - me.z;
    float r2 = fmaf(dx, dx, eps2);
    r2 = fmaf(dy, dy, r2);
    r2 = fmaf(dz, dz, r2);
    float inv = __builtin_amdgcn_rsqf(r2);
    if (MASK) inv = (r2 > 0.f) ? inv : 0.f;
    const float f = (q.w * inv) * (inv * inv);
    tx = fmaf(f, dx, tx);
    ty = fmaf(f, dy, ty);
    tz = fmaf(f, dz, tz);
  }
}

// Post-Newtonian terms of the group traversal (PN): with every list flush the
// lanes also evaluate, in FP64, the terms of each list entry (NodePn), in the
// same pieces as the Newtonian sums. The list keeps its node ids in LDS; their
// FP64 records are loaded during the Newtonian passes (the next batch's during
// this one's terms) and put in LDS beside the group's bodies. Bound: FP64 issue
// (about 52 instructions and a v_rsq_f64 per pair, the SIMDs issue in 83% of
// their cycles). Traversal at theta 0.5 (Newtonian sums included), against one
// lane per body, which left a third of the lanes idle and waited for the
// gather, and 61 instructions: 1PN, 5000 bodies 352 -> 219 us, 100003 1219 ->
// 766 us, 2^20 9.8 -> 6.3 ms; 1PN + 2PN + 2.5PN 1023 -> 986 us, 4.62 -> 4.16 ms,
// 36.8 -> 30.3 ms (a wavefront per group; several: bh_forces_all).
constexpr int kPnBatch = 64;  // entries in LDS at a time, per wavefront
template <int W>
struct PnLds {                  // behind the list, the stack and the node ids
  double4 com[W * kPnBatch];    // entries: centre of mass, mass
  double4 vel[W * kPnBatch];    // velocity, -2 |v|^2
  double4 bpos[64];             // bodies: position, mass
  double4 bvel[64];             // velocity, -|v|^2
};
static_assert(kPieceMaxPasses * 64 * sizeof(double) <= (kGrpList + kGrpListPad) * sizeof(float4),
              "one coordinate of the pieces' sums takes the list's place");

// get_pn1 (tool_chain_impl.cpp:110-118) as an acceleration of the body at pb
// by the node at nc, over G / c^2, n = (x_i - x_node)/r, grouped for fused
// multiply-adds:
//   m2/r^2 [n (-v1^2 - 2 v2^2 + 4 v1.v2 + 3/2 (n.v2)^2 + (5 G m1 + 4 G m2)/r)
//           + (v1 - v2)(4 n.v1 - 3 n.v2)]
// N entries step by step together, so that their chains overlap. Every term
// carries n, so a node at distance 0 adds 0, as long as 1/r and the products
// with it (up to m G m / r^4) stay finite: r^2 is kept above 1e-100.
template <int N>
__device__ __forceinline__ void pn1_pairs(const double4* nc, const double4* nv, const double4& pb, const double4& vb,
                                          double g5m1, double g4, double soft, double* a) {
  double d[N][3], x[N], y[N], e[N], n1[N], n2[N], sc[N], k[N];
#define ASTER_EACH(...)                                          \
  _Pragma("unroll") for (int q = 0; q < N; ++q) { __VA_ARGS__; } \
  __builtin_amdgcn_sched_barrier(0);
  ASTER_EACH(d[q][0] = nc[q].x - pb.x; d[q][1] = nc[q].y - pb.y; d[q][2] = nc[q].z - pb.z)
  ASTER_EACH(x[q] = fma(d[q][0], d[q][0], fma(d[q][1], d[q][1], fma(d[q][2], d[q][2], soft))))
  ASTER_EACH(x[q] = fmax(x[q], 1e-100))
  ASTER_EACH(y[q] = __builtin_amdgcn_rsq(x[q]))
  // meanwhile what needs no 1 / r: d.v1, d.v2 and the velocity terms
  ASTER_EACH(n1[q] = fma(d[q][0], vb.x, fma(d[q][1], vb.y, d[q][2] * vb.z)))
  ASTER_EACH(n2[q] = fma(d[q][0], nv[q].x, fma(d[q][1], nv[q].y, d[q][2] * nv[q].z)))
  ASTER_EACH(sc[q] = fma(vb.x, nv[q].x, fma(vb.y, nv[q].y, vb.z * nv[q].z)))
  ASTER_EACH(sc[q] = fma(4.0, sc[q], vb.w) + nv[q].w)
  // 1 / r: one third-order step from the estimate (rsqrt64)
  ASTER_EACH(e[q] = x[q] * y[q])
  ASTER_EACH(e[q] = fma(-e[q], y[q], 1.0))
  ASTER_EACH(k[q] = fma(0.375, e[q], 0.5); e[q] = e[q] * y[q])
  ASTER_EACH(y[q] = fma(e[q], k[q], y[q]))
  // n = -d / r: n.v = -(d.v) / r
  ASTER_EACH(n2[q] = n2[q] * y[q]; n1[q] = n1[q] * y[q])
  ASTER_EACH(sc[q] = fma(1.5 * n2[q], n2[q], sc[q]); x[q] = fma(g4, nc[q].w, g5m1))
  ASTER_EACH(sc[q] = fma(x[q], y[q], sc[q]); k[q] = nc[q].w * (y[q] * y[q]); e[q] = fma(4.0, n1[q], -3.0 * n2[q]))
  ASTER_EACH(sc[q] = sc[q] * y[q]; e[q] = e[q] * k[q])
  ASTER_EACH(sc[q] = sc[q] * k[q])
  // a -= k (d sc / r + (v1 - v2) (4 d.v1 - 3 d.v2) / r)
  ASTER_EACH(a[0] = fma(-sc[q], d[q][0], a[0]); a[1] = fma(-sc[q], d[q][1], a[1]); a[2] = fma(-sc[q], d[q][2], a[2]))
  ASTER_EACH(a[0] = fma(-e[q], vb.x - nv[q].x, a[0]); a[1] = fma(-e[q], vb.y - nv[q].y, a[1]);
             a[2] = fma(-e[q], vb.z - nv[q].z, a[2]))
#undef ASTER_EACH
}

template <bool MASK, int PN, int W>  // PN: 0 none, 1 the 1PN term alone, 2 any terms; W: wavefronts per group
__global__ __launch_bounds__(64 * W, PN == 1 ? 3 : 1) void k_bh_group(int n, const int32_t* __restrict__ gstart,
                                                 const uint32_t* __restrict__ gcount, const float4* __restrict__ gsh,
                                                 const float4* __restrict__ kids, const uint32_t* __restrict__ perm,
                                                 float eps2, float msc, double G,
                                                 double* __restrict__ a, unsigned long long* __restrict__ counters,
                                                 uint32_t* __restrict__ flags, NodePn pnp) {
  extern __shared__ float4 grp_lds[];
  constexpr int kList = W * kGrpList, kPad = W * kGrpListPad, kStack = W * kGrpStack;
  float4* lst = grp_lds;                                   // kList + kPad entries
  int* stk = reinterpret_cast<int*>(grp_lds + kList + kPad);  // kStack entries
  int* lid = stk + kStack;  // PN: node id of each list entry (kList entries)
  PnLds<W>* pl = reinterpret_cast<PnLds<W>*>(grp_lds + kList + kPad + (kStack + kList) / 4);  // PN
  __shared__ int2 wsum[W];  // W > 1: each wavefront's accepted and opened candidates
  const int tid = threadIdx.x, lane = tid & 63, w = W > 1 ? tid >> 6 : 0;
  auto sync = [] {
    if (W > 1) __syncthreads();
    else wave_sync();
  };
  const int ngroups = (int)*gcount;
  const int per_xcd = (ngroups + 7) >> 3;
  const int xcd = blockIdx.x & 7;
  const int stride = (int)(gridDim.x >> 3);
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  unsigned long long tot_inter = 0, tot_visits = 0;
  for (int i = (int)(blockIdx.x >> 3); i < per_xcd; i += stride) {
    const int g = xcd * per_xcd + i;
    if (g >= ngroups) break;
    const int lo = gstart[g], hi = gstart[g + 1] - 1;
    const int gsz = __builtin_amdgcn_readfirstlane(hi - lo + 1);
    const int k = lo + lane;
    const bool live = k <= hi;
    const float4 me = gsh[live ? k : hi];
    double pacc[3] = {0.0, 0.0, 0.0};  // PN: the body's terms
    if (PN && w == 0) {  // the bodies' FP64 positions, masses and velocities (the leaves' records)
      double4 vme = pnp.nvel[live ? k : hi];
      vme.w = -fma(vme.x, vme.x, fma(vme.y, vme.y, vme.z * vme.z));
      pl->bpos[lane] = pnp.nmc[live ? k : hi];
      pl->bvel[lane] = vme;
    }
    // this lane's piece in each pass
    const int npass = __builtin_amdgcn_readfirstlane((int)kPieces<W>.passes[gsz]);
    const int npc = __builtin_amdgcn_readfirstlane((int)kPieces<W>.pieces[gsz]);
    float4 ppos[kPieceMaxPasses];
    int pidx[kPieceMaxPasses], pbody[kPieceMaxPasses];
#pragma unroll
    for (int p = 0; p < kPieceMaxPasses; ++p) {
      const int j = 64 * W * p + tid;
      int b = j / npc, pc = j - b * npc;
      if (b >= gsz) {
        b = gsz - 1;
        pc = 0;
      }
      ppos[p] = make_float4(__shfl(me.x, b, 64), __shfl(me.y, b, 64), __shfl(me.z, b, 64), 0.f);
      pidx[p] = pc;
      pbody[p] = b;
    }
    float blo[3] = {me.x, me.y, me.z}, bhi[3] = {me.x, me.y, me.z};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      for (int off = 32; off > 0; off >>= 1) {
        blo[c] = fminf(blo[c], __shfl_xor(blo[c], off, 64));
        bhi[c] = fmaxf(bhi[c], __shfl_xor(bhi[c], off, 64));
      }
      // every lane holds the same value; saying so keeps the list count and
      // the root test scalar
      blo[c] = uniform_f32(blo[c]);
      bhi[c] = uniform_f32(bhi[c]);
    }
    float sx = 0.f, sy = 0.f, sz = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    unsigned long long listed = 0, visits = 1;
    int sp = 0, cnt = 0;
    auto dmin2 = [&](const float4& r) {
      const float ex = fmaxf(fmaxf(blo[0] - r.x, r.x - bhi[0]), 0.f);
      const float ey = fmaxf(fmaxf(blo[1] - r.y, r.y - bhi[1]), 0.f);
      const float ez = fmaxf(fmaxf(blo[2] - r.z, r.z - bhi[2]), 0.f);
      return fmaf(ex, ex, fmaf(ey, ey, ez * ez));
    };
    auto flush = [&]() {
      const int m = __builtin_amdgcn_readfirstlane(cnt);
      const int lam = __builtin_amdgcn_readfirstlane((m + npc - 1) / npc);
      const int mp = npc * lam;  // m <= mp < m + npc <= m + 64
      if (tid < mp - m) lst[m + tid] = make_float4(0.f, 0.f, 0.f, 0.f);
      double4 ec, ev;
      auto gather = [&](int first) {
        const int node = lid[min(first + tid, m - 1)];
        ec = pnp.nmc[node];
        ev = pnp.nvel[node];
        if (first + tid >= m) ec.w = 0.0;  // padding: adds exactly zero
      };
      // whole pieces of at most kPnBatch entries
      const int batch = PN ? __builtin_amdgcn_readfirstlane(W * kPnBatch / npc * npc) : 0;
      if (PN) gather(0);  // in flight during the Newtonian passes
      sync();
      float px[kPieceMaxPasses], py[kPieceMaxPasses], pz[kPieceMaxPasses];
#pragma unroll
      for (int p = 0; p < kPieceMaxPasses; ++p) {
        px[p] = py[p] = pz[p] = 0.f;
        if (p < npass) group_piece_sum<MASK>(lst + pidx[p] * lam, lam, ppos[p], eps2, px[p], py[p], pz[p]);
      }
      sync();  // every lane is done with the list: its LDS takes the partial sums
#pragma unroll
      for (int p = 0; p < kPieceMaxPasses; ++p)
        if (p < npass) lst[64 * W * p + tid] = make_float4(px[p], py[p], pz[p], 0.f);
      sync();
      if (live && w == 0) {
        float tx = 0.f, ty = 0.f, tz = 0.f;
        const float4* __restrict__ mine = lst + lane * npc;
        for (int c = 0; c < npc; ++c) {
          const float4 v = mine[c];
          tx += v.x;
          ty += v.y;
          tz += v.z;
        }
        kahan_add32(sx, cx, tx);
        kahan_add32(sy, cy, ty);
        kahan_add32(sz, cz, tz);
      }
      if (PN) {
        double pa[kPieceMaxPasses][3];
#pragma unroll
        for (int p = 0; p < kPieceMaxPasses; ++p) pa[p][0] = pa[p][1] = pa[p][2] = 0.0;
        const double g4 = 4.0 * pnp.G;
        for (int first = 0; first < m; first += batch) {
          const int cntb = min(batch, m - first);
          const int lamb = __builtin_amdgcn_readfirstlane((cntb + npc - 1) / npc);
          pl->com[tid] = ec;
          ev.w = -2.0 * fma(ev.x, ev.x, fma(ev.y, ev.y, ev.z * ev.z));
          pl->vel[tid] = ev;
          sync();
          if (first + batch < m) gather(first + batch);
#pragma unroll
          for (int p = 0; p < kPieceMaxPasses; ++p) {
            if (p >= npass) continue;
            const double4 pb = pl->bpos[pbody[p]], vb = pl->bvel[pbody[p]];
            const int e0 = pidx[p] * lamb;
            if constexpr (PN == 1) {
              const double g5m1 = 5.0 * pnp.G * pb.w;
              int e = 0;
              for (; e + 2 <= lamb; e += 2) {
                const double4 nc[2] = {pl->com[e0 + e], pl->com[e0 + e + 1]};
                const double4 nv[2] = {pl->vel[e0 + e], pl->vel[e0 + e + 1]};
                pn1_pairs<2>(nc, nv, pb, vb, g5m1, g4, pnp.soft, pa[p]);
              }
              if (e < lamb) pn1_pairs<1>(&pl->com[e0 + e], &pl->vel[e0 + e], pb, vb, g5m1, g4, pnp.soft, pa[p]);
            } else {
              const double inv_m = 1.0 / pb.w;
              for (int e = 0; e < lamb; ++e)  // every term carries the node's mass: padding adds 0
                node_pn_rec(pnp, pl->com[e0 + e], pl->vel[e0 + e], pb, vb, inv_m, pa[p][0], pa[p][1], pa[p][2]);
            }
          }
          sync();  // every lane is done with these entries
        }
        // a body adds its pieces in order, one coordinate at a time through the
        // list's LDS
        double* ps = reinterpret_cast<double*>(lst);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
#pragma unroll
          for (int p = 0; p < kPieceMaxPasses; ++p)
            if (p < npass) ps[64 * W * p + tid] = pa[p][c];
          sync();
          if (live && w == 0) {
            double t = 0.0;
            for (int q = 0; q < npc; ++q) t += ps[lane * npc + q];
            pacc[c] += PN == 1 ? t * (pnp.G * (pnp.ic * pnp.ic)) : t;
          }
          sync();
        }
      }
      sync();  // the partial sums are read before the list is refilled
      listed += (unsigned long long)cnt;
      cnt = 0;
    };
    {
      const int root = n, rs = 2 * (n - 1);
      const float4 r = kids[2 * rs];
      if (dmin2(r) > kids[2 * rs + 1].y) {
        if (tid == 0) {
          lst[0] = make_float4(r.x, r.y, r.z, r.w * msc);
          if (PN) lid[0] = root;
        }
        cnt = 1;
      } else {
        if (tid == 0) stk[0] = root;
        sp = 1;
      }
    }
    sync();
    // The children of the next batch (the top of the stack) are
    // loaded before a pending flush evaluates the list, so the load's latency
    // overlaps that arithmetic. Lane 2 i + s takes child s of entry i: the two
    // children of a node are 64 contiguous bytes. Lanes past the batch load a
    // copy of its last entry and are masked off; every lane loads, so the
    // loop carries one definition of the record and needs no branches.
    int take = 0;
    float4 nr;
    float2 na;
    // With an empty stack (the walk is over) it loads the root's children.
    auto fetch = [&]() {
      take = min(min(sp, 32 * W), max(kStack - kGrpDeep - sp, 1));
      const int e = max(min(tid >> 1, take - 1), 0);
      const int opened = sp > 0 ? stk[sp - take + e] : n;
      const int slot = kid_slot(n, opened, tid & 1);
      nr = kids[2 * slot];
      na = *reinterpret_cast<const float2*>(kids + 2 * slot + 1);
    };
    fetch();
    bool overflow = false;
    while (sp > 0) {
      const float4 r = nr;
      const int node = __float_as_int(na.x);
      // both terms evaluated (no short circuit): the id and the threshold
      // arrive with the record in one round trip
      const bool take_it = (node < n) | (dmin2(r) > na.y);
      const bool mine = tid < 2 * take;
      const bool acc = mine & take_it, opn = mine & !take_it;
      sp -= take;
      visits += 2 * take;
      const uint64_t am = __ballot(acc), om = __ballot(opn);
      int nacc = (int)__popcll(am), nopen = (int)__popcll(om);  // of all wavefronts
      int e = cnt + (int)__popcll(am & lt), f = sp + (int)__popcll(om & lt);
      if (W > 1 && lane == 0) wsum[w] = make_int2(nacc, nopen);
      sync();  // also: every candidate's entry has been read off the stack
      if (W > 1) {
        nacc = nopen = 0;
#pragma unroll
        for (int v = 0; v < W; ++v) {
          const int2 c = wsum[v];
          e += v < w ? c.x : 0;
          f += v < w ? c.y : 0;
          nacc += c.x;
          nopen += c.y;
        }
        nacc = __builtin_amdgcn_readfirstlane(nacc);
        nopen = __builtin_amdgcn_readfirstlane(nopen);
      }
      // cannot happen for a valid tree (see bound above); the walk then ends
      // here (no early exit from the loop, which keeps its control flow simple)
      const bool over = sp + nopen > kStack;
      if (over) {
        if (tid == 0) atomicOr(flags, (uint32_t)FLAG_TREE);
        overflow = true;
      }
      // list entries carry the scaled mass (one multiply per entry, not per pair)
      if (acc) {
        lst[e] = make_float4(r.x, r.y, r.z, r.w * msc);
        if (PN) lid[e] = node;
      }
      if (opn && !over) stk[f] = node;
      cnt += nacc;
      sp = over ? 0 : sp + nopen;
      sync();
      fetch();
      if (cnt > kList - 64 * W) {
        flush();
        sync();
      }
    }
    if (cnt > 0) flush();
    sync();
    if (live && w == 0) {
      const int b = (int)perm[k];
      a[b] = G * ((double)sx - (double)cx) + pacc[0];
      a[n + b] = G * ((double)sy - (double)cy) + pacc[1];
      a[2 * n + b] = G * ((double)sz - (double)cz) + pacc[2];
    }
    // every body's own leaf is in its group's list (distance 0, no force)
    const unsigned long long nlive = (unsigned long long)(hi - lo + 1);
    tot_inter += listed * nlive - nlive;
    tot_visits += visits;
    if (overflow) break;
  }
  if (tid == 0 && (tot_inter | tot_visits)) {
    atomicAdd(&counters[BHC_INTERACTIONS], tot_inter);
    atomicAdd(&counters[BHC_VISITS], tot_visits);
  }
}

__global__ void k_zero_counters(unsigned long long* p) {
  if (threadIdx.x < BHC_COUNT) p[threadIdx.x] = 0ull;
}

// --------------------------------------------------------------- launch ----

// Tiles of the sort: kRsThreads times `keys` keys.
struct SortPlan {
  int keys, tiles;
  int sums;  // RS_ROWS, RS_GROUPS, RS_SCANNED
};

// Few keys per thread shorten the serial ranking of a tile, many tiles lengthen
// the sums of their rows. Leapfrog step of the group method, us, with 2 / 4 / 8
// keys: 20000 bodies 137 / 140 / 150, 50000 163 / 164 / 174, 262144 343 / 337 /
// 336. The sort's kernels, us: 524288 bodies 4 / 8 keys 54.2 / 57.6; 262144 rows
// summed in groups above 128 / 64 tiles 51.7 / 50.3 (above 32, step at 100000 191
// -> 199).
static SortPlan sort_plan(int64_t n) {
  SortPlan p{};
  p.keys = n <= (1 << 15) ? 2 : n <= (1 << 19) ? 4 : 8;
  p.tiles = (int)((n + p.keys * kRsThreads - 1) / (p.keys * kRsThreads));
  p.sums = p.tiles <= kRsMaxRows ? RS_ROWS : p.tiles <= kRsMaxGroups * kRsGroup ? RS_GROUPS : RS_SCANNED;
  return p;
}

static int reserve_sort(aster_ctx* c) {
  const size_t n = (size_t)c->n;
  const size_t tiles = (size_t)sort_plan(c->n).tiles;
  ASTER_HIP(c, c->codes.reserve(n));
  ASTER_HIP(c, c->idx.reserve(n));
  ASTER_HIP(c, c->kv.reserve(2 * n));
  ASTER_HIP(c, c->xm4.reserve(n));
  ASTER_HIP(c, c->above.reserve(ABOVE_COUNT));
  ASTER_HIP(c, c->rows.reserve(tiles * kRsWords));
  ASTER_HIP(c, c->rowsum.reserve((tiles / kRsGroup + 2) * kRsWords));
  return ASTER_OK;
}

// f with the plan's keys per thread as a compile-time constant.
template <class F>
static void with_keys(const SortPlan& p, F f) {
  if (p.keys == 2) f(std::integral_constant<int, 2>{});
  else if (p.keys == 4) f(std::integral_constant<int, 4>{});
  else f(std::integral_constant<int, 8>{});
}

// The groups from k_build's flags.
static int group_starts(aster_ctx* c, int n) {
  const int chunks = (n + kGsChunk - 1) / kGsChunk;
  const uint4* flag = reinterpret_cast<const uint4*>(c->gflag.p);
  uint32_t* part = n > kGsOne ? c->gpart.p : nullptr;
  if (part && chunks > 1) hipLaunchKernelGGL(k_group_counts, dim3(chunks - 1), dim3(kGsThreads), 0, c->stream, flag, part);
  hipLaunchKernelGGL(k_group_starts, dim3(chunks), dim3(kGsThreads), 0, c->stream, flag, n, part, c->gscan.p,
                     c->gcount.p, c->gstart.p);
  ASTER_HIP(c, hipGetLastError());
  return ASTER_OK;
}

static int reserve_tree(aster_ctx* c, bool full) {
  const size_t n = (size_t)c->n, nn = 2 * n - 1;
  int rc = reserve_sort(c);
  if (rc) return rc;
  ASTER_HIP(c, c->left.reserve(nn));
  ASTER_HIP(c, c->right.reserve(nn));
  ASTER_HIP(c, c->parent.reserve(nn));
  ASTER_HIP(c, c->splitnode.reserve(n));
  ASTER_HIP(c, c->units.reserve(n / kGroup + 1));
  ASTER_HIP(c, c->top.reserve(n));
  ASTER_HIP(c, c->big.reserve(n / kUnit + 1));
  ASTER_HIP(c, c->crown.reserve(kMaxLevels * (n / kBigUnit + 1)));  // disjoint at each level
  ASTER_HIP(c, c->topslot.reserve(n));
  ASTER_HIP(c, c->gflag.reserve((n + 15) / 16 * 16));  // read 16 at a time
  ASTER_HIP(c, c->gpart.reserve(n / kGsChunk + 1));
  ASTER_HIP(c, c->gscan.reserve(n));
  ASTER_HIP(c, c->gstart.reserve(n + 1));
  ASTER_HIP(c, c->gcount.reserve(1));
  ASTER_HIP(c, c->grange.reserve(n));
  ASTER_HIP(c, c->nmc.reserve(nn));
  ASTER_HIP(c, c->nbox.reserve(2 * nn));
  ASTER_HIP(c, c->nrec.reserve(nn));
  if (full) ASTER_HIP(c, c->nlink.reserve(nn));
  else ASTER_HIP(c, c->kids.reserve(2 * nn));  // 2 float4 per child slot; 2 (n - 1) + 1 slots
  ASTER_HIP(c, c->gsh.reserve(n));
  if (!c->bh_counters.p) {
    // Counters accumulate over evaluations until aster_bh_stats reads them.
    ASTER_HIP(c, c->bh_counters.reserve(BHC_COUNT));
    hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, c->stream, c->bh_counters.p);
    ASTER_HIP(c, hipGetLastError());
  }
  return ASTER_OK;
}

static int morton_codes(aster_ctx* c, bool user_box) {
  phase_begin(c, ASTER_PHASE_MORTON);
  BoxSource bs;
  int rc = launch_box(c, user_box, &bs);
  if (rc) return rc;
  const int n = (int)c->n;
  const SortPlan p = sort_plan(n);
  with_keys(p, [&](auto K) {
    hipLaunchKernelGGL(k_morton<K()>, dim3(p.tiles), dim3(kRsThreads), 0, c->stream, n, c->x.p, c->m.p, bs, c->boxd.p,
                       c->codes.p, c->xm4.p, c->above.p, c->rows.p, c->flags.p);
  });
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_MORTON);
  c->tree_valid = false;
  return ASTER_OK;
}

int bh_morton_only(aster_ctx* c) {
  int rc = reserve_sort(c);
  if (rc) return rc;
  return morton_codes(c, true);
}

// Morton codes of the current state, stably sorted: c->codes holds the sorted
// codes and c->idx the body at each sorted position. user_box = false always
// uses the symmetric box of the data.
int morton_sort(aster_ctx* c, bool user_box) {
  int rc = reserve_sort(c);
  if (rc) return rc;
  if ((rc = morton_codes(c, user_box))) return rc;
  const int n = (int)c->n;
  const SortPlan p = sort_plan(n);
  phase_begin(c, ASTER_PHASE_SORT);
  if (n <= kRsSmall) {
    hipLaunchKernelGGL((k_rs_small<1024, kRsSmall / 1024>), dim3(1), dim3(1024), 0, c->stream, c->codes.p, c->idx.p, n);
  }
  for (int pass = 0; pass < kRsPasses && n > kRsSmall; ++pass) {
    const uint2* kin = c->kv.p + (pass == 2 ? n : 0);  // pass 0: the codes -> kv, then -> kv + n -> codes, idx
    uint2* kout = c->kv.p + (pass == 1 ? n : 0);
    with_keys(p, [&](auto K) {
      const dim3 grid(p.tiles), block(kRsThreads);
      if (pass > 0)
        hipLaunchKernelGGL((k_rs_hist<K()>), grid, block, 0, c->stream, kin, n, pass, c->rows.p);
      const int ng = (p.tiles + kRsGroup - 1) / kRsGroup;
      if (p.sums != RS_ROWS)
        hipLaunchKernelGGL(k_rs_groups, dim3(ng, kRsShare), dim3(kRsWords), 0, c->stream, c->rows.p, p.tiles,
                           c->rowsum.p);
      if (p.sums == RS_SCANNED)
        hipLaunchKernelGGL(k_rs_group_scan, dim3(kRsWords / kRsScanWords), dim3(kRsScanThreads), 0, c->stream,
                           c->rowsum.p, ng);
      auto kern = p.sums == RS_ROWS     ? k_rs_scatter<K(), RS_ROWS>
                  : p.sums == RS_GROUPS ? k_rs_scatter<K(), RS_GROUPS>
                                        : k_rs_scatter<K(), RS_SCANNED>;
      hipLaunchKernelGGL(kern, grid, block, 0, c->stream, c->codes.p, kin, kout, c->codes.p, c->idx.p, n, pass,
                         c->rows.p, c->rowsum.p, p.tiles);
    });
  }
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_SORT);
  return ASTER_OK;
}

// full: also the links of every node (for the per-body traversals; the group
// traversal does not need them).
static int build_tree(aster_ctx* c, int mac, bool vel, bool full) {
  const int n = (int)c->n;
  int rc = reserve_tree(c, full);
  if (rc) return rc;
  float4* kids = full ? nullptr : c->kids.p;  // the group traversal's child slots
  if ((rc = morton_sort(c, true))) return rc;
  phase_begin(c, ASTER_PHASE_BUILD);
  if (vel) ASTER_HIP(c, c->nvel.reserve((size_t)2 * n - 1));
  auto build = vel ? k_build<true> : k_build<false>;
  hipLaunchKernelGGL(build, dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->codes.p, c->idx.p, c->xm4.p,
                     c->v.p, c->left.p, c->right.p, c->parent.p, c->grange.p, c->nmc.p, c->nvel.p, c->nbox.p,
                     c->nrec.p, c->gsh.p, c->splitnode.p, c->gflag.p, c->above.p, c->units.p, c->top.p, c->big.p,
                     c->crown.p, c->flags.p,
                     full ? 1 : 0);
  ASTER_HIP(c, hipGetLastError());
  // Groups of the wavefront traversal, also the subtrees of the first moment
  // pass: their first sorted positions in Morton order and the sentinel n; the
  // count stays on the device.
  if ((rc = group_starts(c, n))) return rc;
  phase_end(c, ASTER_PHASE_BUILD);
  const int nn = 2 * n - 1;
  phase_begin(c, ASTER_PHASE_MOMENTS);
  // the nodes inside the groups, then those above: units, then the top
  const int gblocks = ((n / 32 + 1) + 3) / 4;
  auto gmom = vel ? k_group_moments<true> : k_group_moments<false>;
  hipLaunchKernelGGL(gmom, dim3(gblocks), dim3(256), 0, c->stream, n, c->gstart.p, c->gcount.p, c->grange.p, c->left.p,
                     c->right.p, c->nmc.p, c->nvel.p, c->nbox.p, c->nrec.p, c->P.theta, kids);
  const uint32_t* len = c->above.p;
  auto above = [&](auto kern, int blocks, int threads, const MomLists& lists) {
    hipLaunchKernelGGL(kern, dim3(blocks), dim3(threads), 0, c->stream, n, lists, c->gstart.p, c->gcount.p, c->gscan.p,
                       c->splitnode.p, c->left.p, c->right.p, c->grange.p, c->nmc.p, c->nvel.p, c->nbox.p, c->nrec.p,
                       c->P.theta, kids, c->topslot.p, c->flags.p);
  };
  // (units hold ~5400 leaves each, big units ~1.4 million; the workgroups loop over more)
  if (n > kGroup)
    above(vel ? k_moments_above<true, MOM_UNITS> : k_moments_above<false, MOM_UNITS>, n / 1024 + 1, kUnitThreads,
          MomLists{c->units.p, len + ABOVE_UNITS, nullptr, nullptr, kGroup});
  if (n > kBigUnit)
    above(vel ? k_moments_above<true, MOM_BIG> : k_moments_above<false, MOM_BIG>, n / (kBigUnit / 4) + 1, kUnitThreads,
          MomLists{c->big.p, len + ABOVE_BIG, c->top.p, len + ABOVE_TOP, kUnit});
  if (n > kUnit)
    above(vel ? k_moments_above<true, MOM_TOP> : k_moments_above<false, MOM_TOP>, 1, kTopThreads,
          n > kBigUnit ? MomLists{nullptr, nullptr, c->crown.p, len + ABOVE_CROWN, kBigUnit}
                       : MomLists{nullptr, nullptr, c->top.p, len + ABOVE_TOP, kUnit});
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_MOMENTS);
  phase_begin(c, ASTER_PHASE_LINKS);
  if (full) {  // the group traversal's child slots were written with the moments
    hipLaunchKernelGGL(mac == 0 ? k_links<0> : k_links<1>, dim3((nn + 255) / 256), dim3(256), 0, c->stream, n,
                       c->left.p, c->right.p, c->parent.p, c->grange.p, c->splitnode.p, c->nbox.p, c->nrec.p,
                       c->boxd.p, c->P.theta, c->nlink.p, c->idx.p, c->flags.p);
    ASTER_HIP(c, hipGetLastError());
  }
  phase_end(c, ASTER_PHASE_LINKS);
  c->tree_valid = true;
  c->tree_mac = mac;
  return ASTER_OK;
}

// Barnes-Hut over every body of the context's state.
static int bh_forces_all(aster_ctx* c, int method) {
  const int n = (int)c->n;
  const int pnf = c->P.pn_flags & ASTER_PN_TERMS;
  const bool pn = pnf != 0;
  const bool f64 = method == ASTER_BH_PARITY && c->P.precision == ASTER_FP64;
  if (n == 1) {
    ASTER_HIP(c, hipMemsetAsync(c->a.p, 0, 3 * sizeof(double), c->stream));
    return ASTER_OK;
  }
  const int mac = (method == ASTER_BH_PARITY) ? 0 : 1;
  Fp32Scales sc{};
  int rc;
  if (!f64 && (rc = fp32_scales(c, &sc))) return rc;
  if ((rc = build_tree(c, mac, pn, method != ASTER_BH_GROUP))) return rc;
  phase_begin(c, ASTER_PHASE_TRAVERSE);
  const double ic = 1.0 / c->P.c;
  if (f64) {
    if (pn)
      hipLaunchKernelGGL((k_bh_f64<true>), dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->m.p,
                         c->nmc.p, c->nvel.p, c->nlink.p, c->boxd.p, c->P.theta, c->P.G, ic, pnf,
                         c->P.softening, c->a.p, c->bh_counters.p, c->flags.p);
    else
      hipLaunchKernelGGL((k_bh_f64<false>), dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->x.p, c->v.p, c->m.p,
                         c->nmc.p, c->nvel.p, c->nlink.p, c->boxd.p, c->P.theta, c->P.G, ic, pnf,
                         c->P.softening, c->a.p, c->bh_counters.p, c->flags.p);
  } else {
    const float eps2 = sc.eps2;
    const bool mask = sc.mask;
    if (method == ASTER_BH_GROUP) {
      // One workgroup per group while groups average more than 32 bodies
      // (the usual case); workgroups loop when there are more groups. The
      // count is a multiple of 8 for the XCD-interleaved group order.
      const int blocks = ((n / 32 + 1) + 7) & ~7;
      const NodePn gp{c->nmc.p, c->nvel.p, c->P.G, ic, c->P.softening, pnf};
      // Wavefronts per group. Below ~2^18 bodies the ~n/42 groups leave SIMDs
      // idle (there are 1024) and the longest walk decides. Evaluation at
      // theta 0.5 with 1 / 2 / 4 wavefronts, us: 2000 bodies 162 / 129 / 115,
      // 50000 222 / 180 / 164, 100000 273 / 239 / 235, 200000 374 / 349 / 365,
      // 400000 572 / 577 / 605, 2^20 1199 / 1285 / 1444. With the 1PN term: 5000
      // 298 / 209 / 204, 20000 417 / 322 / 341, 50000 580 / 479 / 485, 100000
      // 849 / 734 / 792, 2^20 6.5 / 6.4 ms; several wavefronts wait at barriers, so
      // registers are kept to three waves per SIMD there (785 / 868 without at
      // 100000). All terms: 5000 1073 / 667 / 390, 131072 5251 / 4285 / 3534, 2^20
      // 29.8 / 30.7 / 28.8 ms. The same line for all, so that the Newtonian sums
      // have the same bits with and without the terms.
      auto launch = [&](auto waves, auto terms) {
        constexpr int W = waves(), PN = terms();
        // PN: node ids, then (16-byte aligned) FP64 records and velocities of the list
        const size_t lds = W * ((kGrpList + kGrpListPad) * sizeof(float4) + kGrpStack * sizeof(int)) +
                           (PN ? W * kGrpList * sizeof(int) + sizeof(PnLds<W>) : 0);
        auto kern = mask ? k_bh_group<true, PN, W> : k_bh_group<false, PN, W>;
        hipLaunchKernelGGL(kern, dim3(blocks), dim3(64 * W), lds, c->stream, n, c->gstart.p, c->gcount.p, c->gsh.p,
                           c->kids.p, c->idx.p, eps2, sc.msc, sc.gsc, c->a.p, c->bh_counters.p, c->flags.p, gp);
      };
      auto waves = [&](auto terms) {
        if (n <= 1 << 16) launch(std::integral_constant<int, 4>{}, terms);
        else if (n <= 1 << 18) launch(std::integral_constant<int, 2>{}, terms);
        else launch(std::integral_constant<int, 1>{}, terms);
      };
      if (!pn) waves(std::integral_constant<int, 0>{});
      else if (pnf == ASTER_PN1) waves(std::integral_constant<int, 1>{});
      else waves(std::integral_constant<int, 2>{});
    } else {
      const NodePn gp{c->nmc.p, c->nvel.p, c->P.G, ic, c->P.softening, pnf};
      auto kern = pn ? (mask ? k_bh_f32<true, true> : k_bh_f32<false, true>)
                     : (mask ? k_bh_f32<true, false> : k_bh_f32<false, false>);
      hipLaunchKernelGGL(kern, dim3((n + 255) / 256), dim3(256), 0, c->stream, n, c->gsh.p, c->nrec.p, c->nlink.p,
                         eps2, sc.msc, sc.gsc, c->a.p, c->bh_counters.p, c->flags.p, gp);
    }
  }
  ASTER_HIP(c, hipGetLastError());
  phase_end(c, ASTER_PHASE_TRAVERSE);
  return ASTER_OK;
}

// Solver::set_bounds on Barnes-Hut (Barnes_Hut::make_tree and compute_forces,
// src/solvers/barnes_hut.cpp:309-322,414-417): the tree holds the bodies
// [lo, hi) only, and only those bodies get new accelerations; the others keep
// theirs. (The reference indexes the leaves from 0 instead of lower and takes
// the root at the full body count, so its own bounded tree is only right for
// the full range; this follows what the bounds mean.) The range is copied to
// contiguous sub-state planes, evaluated as a state of hi - lo bodies, and
// the accelerations copied back.
static int bh_forces_range(aster_ctx* c, int method, int lo, int hi) {
  const int64_t n = c->n, r = (int64_t)hi - lo;
  ASTER_HIP(c, c->sub_x.reserve((size_t)3 * r));
  ASTER_HIP(c, c->sub_v.reserve((size_t)3 * r));
  ASTER_HIP(c, c->sub_a.reserve((size_t)3 * r));
  ASTER_HIP(c, c->sub_m.reserve((size_t)r));
  for (int q = 0; q < 3; ++q) {
    ASTER_HIP(c, hipMemcpyAsync(c->sub_x.p + q * r, c->x.p + q * n + lo, r * sizeof(double), hipMemcpyDeviceToDevice,
                                c->stream));
    ASTER_HIP(c, hipMemcpyAsync(c->sub_v.p + q * r, c->v.p + q * n + lo, r * sizeof(double), hipMemcpyDeviceToDevice,
                                c->stream));
  }
  ASTER_HIP(c, hipMemcpyAsync(c->sub_m.p, c->m.p + lo, r * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
  // evaluate on the sub-state, then put the full state back whatever happened
  auto swap_state = [c]() {
    std::swap(c->x, c->sub_x);
    std::swap(c->v, c->sub_v);
    std::swap(c->a, c->sub_a);
    std::swap(c->m, c->sub_m);
  };
  const double mt = c->mass_total;
  const bool mt_valid = c->mass_total_valid;
  swap_state();
  c->n = r;
  c->npad = round_up(r, kApBlock);
  c->mass_total_valid = false;
  int rc = bh_forces_all(c, method);
  swap_state();
  c->n = n;
  c->npad = round_up(n, kApBlock);
  c->mass_total = mt;
  c->mass_total_valid = mt_valid;
  c->tree_valid = false;  // the tree holds the sub-state's bodies
  if (rc) return rc;
  for (int q = 0; q < 3; ++q)
    ASTER_HIP(c, hipMemcpyAsync(c->a.p + q * n + lo, c->sub_a.p + q * r, r * sizeof(double), hipMemcpyDeviceToDevice,
                                c->stream));
  return ASTER_OK;
}

int bh_forces(aster_ctx* c, int method) {
  const int n = (int)c->n;
  const int pnf = c->P.pn_flags & ASTER_PN_TERMS;
  const bool f64 = method == ASTER_BH_PARITY && c->P.precision == ASTER_FP64;
  if (pnf & ASTER_EIH) return fail(c, ASTER_ERR_INVALID, "ASTER_EIH needs ASTER_ALLPAIRS_FP64");
  if (!(c->P.theta >= 0.0)) return fail(c, ASTER_ERR_INVALID, "theta must be >= 0");
  const int lo = c->P.lower < 0 ? 0 : c->P.lower;
  const int hi = (c->P.upper < 0 || c->P.upper > n) ? n : c->P.upper;
  if (lo > hi) return fail(c, ASTER_ERR_INVALID, "body bounds: lower > upper");
  if (lo == 0 && hi == n) return bh_forces_all(c, method);
  if (lo == hi) return ASTER_OK;  // no bodies in range: nothing is evaluated (the reference warns and returns)
  return bh_forces_range(c, method, lo, hi);
}

}  // namespace aster
