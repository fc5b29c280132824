// Edge lists of a matrix for drivers that sweep it many times in one call
// (connected components, PageRank, shortest paths): the first pass over the
// tiles writes each nonzero as 4 bytes (row in a window of 64, column), and
// every sweep then streams those instead of finding the bits of every tile
// again.
//
// The unit of the first pass is an item: at most `per` consecutive tiles of one
// window of 64 rows (64 / bs block rows), one wavefront.  It writes its nonzeros
// in tile bit order from place first_tile * kRoom on, so that no places are
// handed out and a weight in tile bit order follows from an entry's number.  The
// few items that have more (hub rows) are only counted then, and listed
// elsewhere once the host has made room.  The pass is bound by the tiles' bytes
// (R-MAT 2^20 at bs 64, 5.2 GB: 1.12 ms).
//
// A sweep's unit is a part: at most kPart entries of an item, one wavefront,
// with the window's 64 results in LDS.  The partial results of a window of
// several parts are added in a fixed order; sums are in FP64 throughout.  What
// bounds a sweep is one gather of x per nonzero, 64 addresses an instruction.
#include <algorithm>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {
namespace {

constexpr int kWin = 64;       // rows of a window
constexpr int kColBits = 26;   // columns of an entry

// Entries an item has room for, per tile (an eighth of a tile at bs 64, R-MAT
// 2^20 has 3 a tile there and 1.3 at bs 8), and its tiles at most.  A matrix of
// more per tile on average is not listed.
template <int BS>
constexpr int kRoom = BS == 8 ? 3 : BS == 16 ? 6 : BS == 32 ? 8 : 16;
template <int BS>
constexpr int kItemTiles = BS <= 16 ? 1024 : 512;
constexpr int kPart = 4096;  // entries of a part at most

struct Item {
  int64_t t0, t1;
};
template <int BS>
__device__ __forceinline__ Item item_of(const ListView& l, int64_t it) {
  const int64_t w = l.win[it];
  const int64_t b0 = w * (kWin / BS), b1 = min(b0 + kWin / BS, (int64_t)l.nbr);
  const int64_t t0 = (int64_t)l.rowptr[b0] + (it - l.first[w]) * l.per;
  return {t0, min(t0 + l.per, (int64_t)l.rowptr[b1])};
}

template <int BS>
__global__ __launch_bounds__(256) void k_win_items(const ListView l, int32_t* __restrict__ cnt) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= l.nwin) return;
  const int64_t b0 = w * (kWin / BS), b1 = min(b0 + kWin / BS, (int64_t)l.nbr);
  cnt[w] = (int32_t)max(((int64_t)l.rowptr[b1] - l.rowptr[b0] + l.per - 1) / l.per, (int64_t)1);
}

__global__ __launch_bounds__(256) void k_item_wins(const ListView l, int32_t* __restrict__ win) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (w >= l.nwin) return;
  for (int64_t i = l.first[w]; i < l.first[w + 1]; ++i) win[i] = (int32_t)w;
}

// A tile's 64-bit words with their bits in row-major order from the top.
template <int BS>
__device__ __forceinline__ uint64_t row_major(uint64_t v) {
  if constexpr (BS == 8) return __builtin_bswap64(v);
  if constexpr (BS == 16) {
    v = (v << 32) | (v >> 32);
    return ((v & 0x0000FFFF0000FFFFull) << 16) | ((v >> 16) & 0x0000FFFF0000FFFFull);
  }
  if constexpr (BS == 32) return (v << 32) | (v >> 32);
  return v;
}

// Calls f(entry) for the set bits of tiles [t0, t1), step by step; before each
// step's bits go(words' bit counts of this lane) may end the walk.
template <int BS>
struct Walk {
  static constexpr int WPT = BS * BS / 64;  // 64-bit words of a tile
  static constexpr int TS = kWave / WPT;    // tiles of a step
  static constexpr int RPW = 64 / BS;       // rows of a word
  static constexpr int U = BS == 64 ? 8 : 4;  // steps loaded together

  int32_t rp[kWin / BS + 1];  // tiles at which the window's block rows begin

  __device__ __forceinline__ Walk(const ListView& l, int64_t w) {
#pragma unroll
    for (int j = 1; j < kWin / BS; ++j) rp[j] = l.rowptr[min(w * (kWin / BS) + j, (int64_t)l.nbr)];
  }
  // this lane's words of U steps from tile b on, and their entries with column 0
  __device__ __forceinline__ void load(const ListView& l, int64_t b, int64_t t1, uint64_t (&v)[U], uint32_t (&e)[U]) const {
    const int s = lane_id() / WPT, k = lane_id() % WPT;
    int32_t c[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = min(b + u * TS + s, t1 - 1);
      v[u] = __builtin_nontemporal_load((const uint64_t*)l.tiles + t * WPT + k);
      c[u] = l.colind[t];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t t = b + u * TS + s;
      v[u] = t < t1 ? row_major<BS>(v[u]) : 0;
      int local = 0;
#pragma unroll
      for (int j = 1; j < kWin / BS; ++j) local += t >= rp[j];
      e[u] = ((uint32_t)(local * BS + k * RPW) << kColBits) + (uint32_t)c[u] * BS;
    }
  }
  static __device__ __forceinline__ uint32_t entry(uint32_t e, int p) {
    return e + ((uint32_t)(p / BS) << kColBits) + (uint32_t)(p % BS);
  }
};

// Writes the entries of a step from place `at` on; returns how many.
template <int BS>
__device__ __forceinline__ int put_bits(uint32_t* __restrict__ out, int at, uint64_t v, uint32_t e) {
  using Wk = Walk<BS>;
  if (!__ballot((v & (v - 1)) != 0)) {  // a bit per lane at most
    const unsigned long long any = __ballot(v != 0);
    if (v) {
      const uint32_t k = __builtin_amdgcn_mbcnt_lo((uint32_t)any, 0);
      out[at + __builtin_amdgcn_mbcnt_hi((uint32_t)(any >> 32), k)] = Wk::entry(e, __builtin_clzll(v));
    }
    return __popcll(any);
  }
  const int own = __popcll(v), incl = wave_incl_scan(own);
  int to = at + incl - own;
  while (v) {
    const int p = __builtin_clzll(v);
    v &= ~(0x8000000000000000ull >> p);
    out[to++] = Wk::entry(e, p);
  }
  return __shfl(incl, kWave - 1);
}

// Bits in kSampleWaves * 64 words spread evenly over the tiles.
constexpr int kSampleWaves = 1024;
__global__ __launch_bounds__(256) void k_list_sample(const uint64_t* __restrict__ words, int64_t n,
                                                     ListInfo* __restrict__ info) {
  const int64_t k = wave_index(), at = (int64_t)((double)(n - kWave) * k / kSampleWaves);
  const int c = wave_incl_scan(__popcll(words[at + lane_id()]));
  if (lane_id() == kWave - 1 && c) atomicAdd(&info->sample[k % kListSlots], (unsigned long long)c);
}

template <int BS>
__global__ __launch_bounds__(256) void k_list(const ListView l, uint32_t* __restrict__ edges, int32_t* __restrict__ cnt) {
  using Wk = Walk<BS>;
  const int64_t it = wave_index();
  if (it >= l.first[l.nwin]) return;
  const Item I = item_of<BS>(l, it);
  const Wk walk(l, l.win[it]);
  const int room = (int)(I.t1 - I.t0) * kRoom<BS>;
  uint32_t* out = edges + I.t0 * kRoom<BS>;
  int n = 0;
  for (int64_t b = I.t0; b < I.t1; b += Wk::U * Wk::TS) {
    uint64_t v[Wk::U];
    uint32_t e[Wk::U];
    walk.load(l, b, I.t1, v, e);
    int own = 0;
#pragma unroll
    for (int u = 0; u < Wk::U; ++u) own += __popcll(v[u]);
    const int all = __shfl(wave_incl_scan(own), kWave - 1);
    if (n + all > room) {  // only counted from here on
      n += all;
      continue;
    }
#pragma unroll
    for (int u = 0; u < Wk::U; ++u) n += put_bits<BS>(out, n, v[u], e[u]);
  }
  if (lane_id() == 0) cnt[it] = n;
}

// An item's entries past its room (0: it is listed) and its parts; the items
// past their room, in any order.
template <int BS>
__global__ __launch_bounds__(256) void k_item_parts(const ListView l, const int32_t* __restrict__ cnt, int64_t cap,
                                                    int32_t* __restrict__ over, int32_t* __restrict__ parts,
                                                    int32_t* __restrict__ overs, ListInfo* __restrict__ info) {
  const int64_t it = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (it >= cap) return;
  int32_t o = 0, p = 0;
  if (it < l.first[l.nwin]) {
    const Item I = item_of<BS>(l, it);
    const int32_t n = cnt[it];
    if (n > (I.t1 - I.t0) * kRoom<BS>) {
      o = n;
      overs[atomicAdd(&info->overs, 1)] = (int32_t)it;  // one item in a hundred
    }
    p = max((n + kPart - 1) / kPart, 1);
  }
  over[it] = o;
  parts[it] = p;
}

template <int BS>
__global__ __launch_bounds__(256) void k_parts_fill(const ListView l, const int32_t* __restrict__ cnt,
                                                    const int64_t* __restrict__ opos, const int64_t* __restrict__ ppos,
                                                    const uint32_t* __restrict__ edges, const uint32_t* __restrict__ rest,
                                                    ListPart* __restrict__ parts) {
  const int64_t it = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (it >= l.first[l.nwin]) return;
  const Item I = item_of<BS>(l, it);
  const int32_t n = cnt[it], w = l.win[it];
  const uint32_t* base = opos[it + 1] > opos[it] ? rest + opos[it] : edges + I.t0 * kRoom<BS>;
  int32_t at = 0;
  for (int64_t k = ppos[it]; k < ppos[it + 1]; ++k, at += kPart)
    parts[k] = {base + at, min(kPart, n - at), w, (int32_t)I.t0, at};
}

// Windows of several parts, and the counts that the host needs.
__global__ __launch_bounds__(256) void k_win_parts(const ListView l, const int64_t* __restrict__ opos,
                                                   const int64_t* __restrict__ ppos, int64_t* __restrict__ wfirst,
                                                   int32_t* __restrict__ multi, ListInfo* __restrict__ info) {
  const int64_t w = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t p0 = 0, p1 = 0;
  if (w <= l.nwin) wfirst[w] = p0 = ppos[l.first[w]];
  if (w < l.nwin) p1 = ppos[l.first[w + 1]];
  const bool several = p1 - p0 > 1;
  const unsigned long long m = __ballot(several);
  int at = 0;
  if (lane_id() == 0 && m) at = atomicAdd(&info->multi, __popcll(m));
  at = __shfl(at, 0);
  if (several) multi[at + __popcll(m & ((1ull << lane_id()) - 1))] = (int32_t)w;
  if (w == 0) {
    info->items = l.first[l.nwin];
    info->parts = ppos[l.first[l.nwin]];
    info->over = opos[l.first[l.nwin]];
  }
}

// The items past their room, kOverSplit workgroups each: the waves of all of
// them take consecutive shares of the tiles and write one after another; a
// workgroup counts the shares up to its own.  (Workgroups for every item, most
// of which leave at once, took 212 us on R-MAT 2^20 at bs 64.)
constexpr int kOverThreads = 1024, kOverSplit = 4;
template <int BS>
__global__ __launch_bounds__(kOverThreads) void k_list_over(const ListView l, const int64_t* __restrict__ opos,
                                                            const int32_t* __restrict__ overs,
                                                            uint32_t* __restrict__ edges) {
  using Wk = Walk<BS>;
  constexpr int W = kOverThreads / kWave;
  __shared__ int sh[W * kOverSplit];
  const int wave = threadIdx.x / kWave, q = blockIdx.y;
  const int64_t it = overs[blockIdx.x];
  const Item I = item_of<BS>(l, it);
  const Wk walk(l, l.win[it]);
  const int64_t share = ((I.t1 - I.t0 + W * kOverSplit - 1) / (W * kOverSplit) + Wk::TS - 1) / Wk::TS * Wk::TS;
  for (int k = wave; k < (q + 1) * W; k += W) {
    const int64_t b0 = min(I.t0 + k * share, I.t1), b1 = min(b0 + share, I.t1);
    int own = 0;
    for (int64_t x = b0 * Wk::WPT + lane_id(); x < b1 * Wk::WPT; x += kWave) own += __popcll(((const uint64_t*)l.tiles)[x]);
    own = __shfl(wave_incl_scan(own), kWave - 1);
    if (lane_id() == 0) sh[k] = own;
  }
  __syncthreads();
  const int mine = q * W + wave;
  int at = 0;
  for (int k = 0; k < mine; ++k) at += sh[k];
  const int64_t b0 = min(I.t0 + mine * share, I.t1), b1 = min(b0 + share, I.t1);
  uint32_t* out = edges + opos[it];
  for (int64_t b = b0; b < b1; b += Wk::U * Wk::TS) {
    uint64_t v[Wk::U];
    uint32_t e[Wk::U];
    walk.load(l, b, b1, v, e);
#pragma unroll
    for (int u = 0; u < Wk::U; ++u) at += put_bits<BS>(out, at, v[u], e[u]);
  }
}

template <int OP>
struct Acc {
  using T = typename std::conditional<OP == OP_SUM, double, typename std::conditional<OP == OP_MIN, int32_t, uint32_t>::type>::type;
  static __device__ __forceinline__ T none() {
    if constexpr (OP == OP_SUM) return 0.0;
    else if constexpr (OP == OP_MIN) return INT32_MAX;
    else return kInfU32;
  }
  static __device__ __forceinline__ void add(T* p, T v) {
    if constexpr (OP == OP_SUM) unsafeAtomicAdd(p, v);
    else atomicMin(p, v);
  }
  static __device__ __forceinline__ T join(T a, T b) {
    if constexpr (OP == OP_SUM) return a + b;
    else return a < b ? a : b;
  }
  static __device__ __forceinline__ void out(const ListSweep& s, int64_t i, T v) {
    if constexpr (OP == OP_SUM) ((float*)s.out)[i] = (float)((double)s.scale * v + (double)s.bias);
    else ((T*)s.out)[i] = v;
  }
};

// Value of U entries (columns c), weight numbers wi where weighted.
template <int OP, int U>
__device__ __forceinline__ void values(const ListSweep& s, const uint32_t (&e)[U], const int64_t (&wi)[U],
                                       typename Acc<OP>::T (&v)[U]) {
  constexpr uint32_t kMask = (1u << kColBits) - 1;
  if constexpr (OP == OP_SUM) {
    float x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = ((const float*)s.x)[e[u] & kMask];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = (double)x[u];
  } else if constexpr (OP == OP_MIN) {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ((const int32_t*)s.x)[e[u] & kMask];
  } else {
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = ((const uint32_t*)s.x)[e[u] & kMask];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (v[u] == kInfU32) continue;
      const uint32_t w = s.w ? s.w[wi[u]] : 1u;
      v[u] = v[u] > kInfU32 - w ? kInfU32 : v[u] + w;
    }
  }
}

template <int OP>
__global__ __launch_bounds__(256) void k_list_sweep(const ListView l, const ListSweep s) {
  using A = Acc<OP>;
  using T = typename A::T;
  __shared__ T sh[4][kWin];
  T* acc = sh[threadIdx.x / kWave];
  const int lane = lane_id();
  const int64_t k = wave_index();
  if (k >= l.nparts || over(s.go)) return;
  const ListPart P = l.parts[k];
  acc[lane] = A::none();
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const int64_t w0 = OP == OP_MINPLUS && s.w && P.n > 0 ? s.woff[P.tile] + P.skip : 0;
  const uint32_t* __restrict__ edges = P.at;
  constexpr int U = 8;
  for (int p = lane; p - lane < P.n; p += U * kWave) {
    uint32_t e[U];
    int64_t wi[U];
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = min(p + u * kWave, P.n - 1);
      e[u] = edges[q];
      wi[u] = w0 + q;
    }
    values<OP, U>(s, e, wi, v);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p + u * kWave < P.n) A::add(&acc[e[u] >> kColBits], v[u]);
  }
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  const T v = acc[lane];
  const int64_t i = (int64_t)P.win * kWin + lane;
  if (l.first[P.win + 1] - l.first[P.win] > 1) ((T*)l.partial)[k * kWin + lane] = v;
  else if (i < l.n) A::out(s, i, v);
}

// Windows of several parts: their partial results, in order.
constexpr int kFoldThreads = 512;
template <int OP>
__global__ __launch_bounds__(kFoldThreads) void k_list_fold(const ListView l, const ListSweep s) {
  using A = Acc<OP>;
  using T = typename A::T;
  constexpr int G = kFoldThreads / kWin, U = 4;
  __shared__ T sh[G][kWin];
  if (over(s.go)) return;
  const int64_t w = l.multi[blockIdx.x];
  const int g = threadIdx.x / kWin, r = threadIdx.x % kWin;
  const int64_t i0 = l.first[w], i1 = l.first[w + 1];
  const T* __restrict__ part = (const T*)l.partial;
  T a = A::none();
  for (int64_t i = i0 + g; i < i1; i += U * G) {
    T v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = part[min(i + u * G, i1 - 1) * kWin + r];
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + u * G < i1) a = A::join(a, v[u]);
  }
  sh[g][r] = a;
  __syncthreads();
  if (g == 0) {
#pragma unroll
    for (int k = 1; k < G; ++k) a = A::join(a, sh[k][r]);
    const int64_t i = w * kWin + r;
    if (i < l.n) A::out(s, i, a);
  }
}

// ---- frontiers of KW words a vertex (multi-source BFS).  The entries of open
// rows and active block columns are listed in LDS, kMsStage looked at a time; KW
// lanes (4 for 3) then gather an entry's words.
constexpr int kMsStage = 4 * kWave;

template <int KW>
__global__ __launch_bounds__(256) void k_list_ms(const ListView l, const ListMs s) {
  constexpr int LPE = KW == 3 ? 4 : KW, EPI = kWave / LPE, U = 4, Q = kMsStage / kWave;
  __shared__ unsigned long long sacc[4][kWin * KW];
  __shared__ uint64_t sopen[4][kWin * KW];
  __shared__ uint32_t sstage[4][kMsStage];
  const int wave = threadIdx.x / kWave, lane = lane_id();
  unsigned long long* acc = sacc[wave];
  uint64_t* open = sopen[wave];
  uint32_t* stage = sstage[wave];
  const int64_t k = wave_index();
  if (k >= l.nparts || over(s.go)) return;
  const ListPart P = l.parts[k];
  const int64_t i = (int64_t)P.win * kWin + lane;
  uint64_t any = 0;
#pragma unroll
  for (int w = 0; w < KW; ++w) {
    const uint64_t o = i < l.n ? s.live[w] & ~s.V[i * KW + w] : 0;
    any |= o;
    open[lane * KW + w] = o;
    acc[lane * KW + w] = 0;
  }
  const uint64_t rows = __ballot(any != 0);
  constexpr uint32_t kMask = (1u << kColBits) - 1;
  const int lgbs = 31 - __builtin_clz(l.bs), wi = lane % LPE;
  const int n = rows ? P.n : 0;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  for (int p = 0; p < n; p += kMsStage) {
    uint32_t e[Q];
    uint64_t act[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) e[q] = P.at[min(p + q * kWave + lane, n - 1)];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const uint32_t J = (e[q] & kMask) >> lgbs;
      act[q] = s.active[J >> 6] >> (J & 63);
    }
    int m = 0;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const bool ok = p + q * kWave + lane < n && (act[q] & (rows >> (e[q] >> kColBits)) & 1);
      const unsigned long long b = __ballot(ok);
      if (ok) stage[m + __builtin_amdgcn_mbcnt_hi((uint32_t)(b >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)b, 0))] = e[q];
      m += __popcll(b);
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    for (int j = lane / LPE; j - lane / LPE < m; j += U * EPI) {
      uint32_t x[U];
      uint64_t f[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = stage[min(j + u * EPI, m - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) f[u] = s.F[(int64_t)(x[u] & kMask) * KW + (wi < KW ? wi : 0)];
#pragma unroll
      for (int u = 0; u < U; ++u) {  // the last entry again past the end: OR
        const int at = (int)(x[u] >> kColBits) * KW + wi;
        if (wi < KW && (f[u] & open[at])) atomicOr(&acc[at], (unsigned long long)f[u]);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  if (i >= l.n) return;
  const bool shared = l.first[P.win + 1] - l.first[P.win] > 1;
#pragma unroll
  for (int w = 0; w < KW; ++w) {
    const unsigned long long m = acc[lane * KW + w] & open[lane * KW + w];
    if (!shared) s.Fn[i * KW + w] = m;
    else if (m) atomicOr((unsigned long long*)&s.Fn[i * KW + w], m);
  }
}

unsigned grid_of(int64_t items, int per_block) {
  return (unsigned)std::max<int64_t>(1, (items + per_block - 1) / per_block);
}

// Rows from which on shortest paths at bs 8/16 over evenly spread columns (hardly
// a tile of two nonzeros) go by the tiles, which skip the inactive ones: the list
// gathers a word out of 8 MB and more for each nonzero on every sweep.  G(n, m),
// lists / tiles: 2^21 of 16 bs 8 11.0 / 9.25 ms, 2^22 of 8 bs 8 18.0 / 12.4 and bs
// 16 18.1 / 14.6, of 16 bs 16 33.5 / 25.6; lists / the sweeps over tiles of one look
// each: 1.2M of 8 bs 16 2.4 / 4.0, R-MAT 2^22 of 4 bs 8 2.8 / 3.8.
constexpr int32_t kSpreadRows = 3 << 19;

template <int BS>
int build_t(const gbo_bsr* A, ListUse use, Workspace& mem, ListView* out, hipStream_t st) {
  const char* who = "edge lists";
  ListView l{};
  l.bs = BS;
  l.n = A->nrows;
  l.nbr = A->nblockrows;
  l.nwin = (int32_t)(((int64_t)A->nrows + kWin - 1) / kWin);
  l.rowptr = A->rowptr;
  l.colind = A->colind;
  l.tiles = A->tiles;
  const int64_t T = A->nblocks;
  l.per = (int32_t)std::min<int64_t>(std::max<int64_t>(T / 4096 / 64 * 64, 64), kItemTiles<BS>);
  const int64_t cap = l.nwin + T / l.per;  // items at most
  const int64_t room = T * kRoom<BS>, words = T * (BS * BS / 64);
  int32_t *icnt = nullptr, *win = nullptr, *multi = nullptr, *cnt = nullptr, *over = nullptr, *np = nullptr;
  int64_t *first = nullptr, *opos = nullptr, *ppos = nullptr, *wfirst = nullptr;
  uint32_t* edges = nullptr;
  ListInfo* info = nullptr;
  ListInfo h{};
  int rc;
  if ((rc = mem.alloc(&info, sizeof(ListInfo), who))) return rc;
  GBO_HIP_CHECK(hipMemsetAsync(info, 0, sizeof(ListInfo), st));
  k_list_sample<<<kSampleWaves / 4, 256, 0, st>>>((const uint64_t*)A->tiles, words, info);
  GBO_LAUNCH_CHECK();
  if ((rc = read_back(&h, info, sizeof(ListInfo), st))) return rc;
  unsigned long long bits = 0;
  for (int i = 0; i < kListSlots; ++i) bits += h.sample[i];
  constexpr unsigned long long kSampleTiles = kSampleWaves * 64 / (BS * BS / 64);
  if (bits > kRoom<BS> * kSampleTiles) return GBO_OK;
  if (use == ListUse::kPaths && BS <= 16 && l.n > kSpreadRows && bits * 10 < kSampleTiles * 11) return GBO_OK;
  if ((rc = mem.alloc(&edges, sizeof(uint32_t) * (size_t)room, who)) ||
      (rc = mem.alloc(&icnt, sizeof(int32_t) * (size_t)l.nwin, who)) ||
      (rc = mem.alloc(&first, sizeof(int64_t) * ((size_t)l.nwin + 1), who)) ||
      (rc = mem.alloc(&wfirst, sizeof(int64_t) * ((size_t)l.nwin + 1), who)) ||
      (rc = mem.alloc(&multi, sizeof(int32_t) * (size_t)l.nwin, who)) ||
      (rc = mem.alloc(&win, sizeof(int32_t) * (size_t)cap * 5, who)) ||
      (rc = mem.alloc(&opos, sizeof(int64_t) * ((size_t)cap + 1), who)) ||
      (rc = mem.alloc(&ppos, sizeof(int64_t) * ((size_t)cap + 1), who)))
    return rc;
  cnt = win + cap;
  over = cnt + cap;
  np = over + cap;
  int32_t* overs = np + cap;
  l.first = first;
  l.win = win;
  k_win_items<BS><<<grid_of(l.nwin, 256), 256, 0, st>>>(l, icnt);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(icnt, first, l.nwin, st, mem))) return rc;
  k_item_wins<<<grid_of(l.nwin, 256), 256, 0, st>>>(l, win);
  k_list<BS><<<grid_of(cap, 4), 256, 0, st>>>(l, edges, cnt);
  k_item_parts<BS><<<grid_of(cap, 256), 256, 0, st>>>(l, cnt, cap, over, np, overs, info);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(over, opos, cap, st, mem)) ||
      (rc = scan_exclusive<int32_t, int64_t>(np, ppos, cap, st, mem)))
    return rc;
  k_win_parts<<<grid_of((int64_t)l.nwin + 1, 256), 256, 0, st>>>(l, opos, ppos, wfirst, multi, info);
  GBO_LAUNCH_CHECK();
  if ((rc = read_back(&h, info, sizeof(ListInfo), st))) return rc;
  if (h.over > room) return GBO_OK;  // denser than the sample
  ListPart* parts = nullptr;
  if ((rc = mem.alloc(&parts, sizeof(ListPart) * (size_t)h.parts, who))) return rc;
  if (h.multi && (rc = mem.alloc(&l.partial, sizeof(double) * (size_t)h.parts * kWin, who))) return rc;
  uint32_t* rest = nullptr;
  if (h.over && (rc = mem.alloc(&rest, sizeof(uint32_t) * (size_t)h.over, who))) return rc;
  k_parts_fill<BS><<<grid_of(h.items, 256), 256, 0, st>>>(l, cnt, opos, ppos, edges, rest, parts);
  if (h.over) k_list_over<BS><<<dim3((unsigned)h.overs, kOverSplit), kOverThreads, 0, st>>>(l, opos, overs, rest);
  GBO_LAUNCH_CHECK();
  l.first = wfirst;
  l.multi = multi;
  l.parts = parts;
  l.nparts = h.parts;
  l.nmulti = h.multi;
  l.on = true;
  *out = l;
  return GBO_OK;
}

template <int OP>
int sweep_t(const ListView& l, const ListSweep& s, hipStream_t st) {
  k_list_sweep<OP><<<grid_of(l.nparts, 4), 256, 0, st>>>(l, s);
  if (l.nmulti) k_list_fold<OP><<<(unsigned)l.nmulti, kFoldThreads, 0, st>>>(l, s);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

}  // namespace

// Building costs a pass over the tiles and about 0.1 ms of small launches; a
// sweep is bound by one gather per nonzero (R-MAT 2^20, 31M nonzeros: 80 us at
// bs 64 to 105 at bs 8).  Whole calls, tiles -> lists, by bytes of matrix:
//   15 to 20 sweeps (PageRank), bs 8: R-MAT 2^18, 62 MB, 1.01 -> 1.05 ms,
//   285 MB 3.18 -> 2.30; bs 16: 57 MB 0.79 -> 0.80, 143 MB 1.38 -> 1.02; bs 32,
//   63 MB 1.61 -> 0.73; bs 64, 41 MB 0.65 -> 0.56, 151 MB 1.04 -> 0.64, 5.2 GB
//   15.5 -> 3.1
//   weighted shortest paths, which skip the tiles of inactive block columns,
//   bs 8: 285 MB 1.94 -> 1.63, 1.26 GB 7.53 -> 7.72; bs 64 5.2 GB 8.4 -> 2.7
//   3 to 5 sweeps (components), bs 16: 700 MB 0.80 -> 0.82; bs 32: 207 MB
//   0.45 -> 0.49, 367 MB 0.62 -> 0.47, 1.9 GB 1.88 -> 1.13; bs 64: 350 MB
//   0.38 -> 0.39, 761 MB 0.99 -> 0.58, 5.2 GB 2.78 -> 1.77
//   256 sources, bs 8: 4 MB 0.36 -> 0.35 ms, 62 MB 1.42 -> 0.75; bs 64, 370 MB
//   2.24 -> 0.54, 890 MB 2.92 -> 1.07; 128 at bs 8, 19 MB 0.33 -> 0.31; 100 at
//   bs 16, 3 MB 0.16 -> 0.21
void lists_build(const gbo_bsr* A, ListUse use, Workspace& mem, ListView* out, hipStream_t st) {
  *out = ListView{};
  const int64_t bytes = A->nblocks * (A->bs * A->bs / 8 + 4), mb = 1 << 20;
  int64_t least = 0;
  switch (use) {
    case ListUse::kPaths:
      if (A->bs == 8 && bytes > 1024 * mb) return;
      [[fallthrough]];
    case ListUse::kMany: least = A->bs == 8 ? 192 * mb : A->bs == 16 ? 96 * mb : 48 * mb; break;
    case ListUse::kFew: least = A->bs <= 16 ? INT64_MAX : A->bs == 32 ? 256 * mb : 512 * mb; break;
    case ListUse::kFrontiers: least = 16 * mb; break;
  }
  if (bytes < least || A->nrows > (1 << kColBits) || A->ncols > (1 << kColBits) || ((uintptr_t)A->tiles & 7)) return;
  switch (A->bs) {
    case 8: (void)build_t<8>(A, use, mem, out, st); break;
    case 16: (void)build_t<16>(A, use, mem, out, st); break;
    case 32: (void)build_t<32>(A, use, mem, out, st); break;
    case 64: (void)build_t<64>(A, use, mem, out, st); break;
  }
}

int lists_sweep(int op, const ListView& l, const ListSweep& s, hipStream_t st) {
  switch (op) {
    case OP_SUM: return sweep_t<OP_SUM>(l, s, st);
    case OP_MIN: return sweep_t<OP_MIN>(l, s, st);
    case OP_MINPLUS: return sweep_t<OP_MINPLUS>(l, s, st);
  }
  return set_error(GBO_EUNSUPPORTED, "op %d not supported", op);
}

int lists_ms(int kw, const ListView& l, const ListMs& s, hipStream_t st) {
  const unsigned blocks = grid_of(l.nparts, 4);
  switch (kw) {
    case 1: k_list_ms<1><<<blocks, 256, 0, st>>>(l, s); break;
    case 2: k_list_ms<2><<<blocks, 256, 0, st>>>(l, s); break;
    case 3: k_list_ms<3><<<blocks, 256, 0, st>>>(l, s); break;
    case 4: k_list_ms<4><<<blocks, 256, 0, st>>>(l, s); break;
    default: return set_error(GBO_EUNSUPPORTED, "%d frontier words not supported", kw);
  }
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

}  // namespace gbo
