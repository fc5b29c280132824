// CSR -> bit-BSR on the device: the block rows of many nonzeros.  A block row's
// nonzeros are one contiguous run of the CSR, read by a workgroup with
// coalesced loads whatever its rows' lengths:
//   count    its block columns are marked in an LDS bitmap; the atomic OR that
//            finds its bit clear counts a tile.  An entry in the same block as
//            the one before it needs no mark, nor one whose bit a plain read
//            finds set: a hub's entries are neighbours, and atomics on one word
//            go one lane at a time.
//   columns  the same bitmap's bits in order are the block row's columns.
//   tiles    a window of consecutive tiles of one block row is built in LDS
//            and stored whole, 16 bytes a lane; an entry finds its tile by a
//            binary search in the window's columns.
// The two walks are bound by the latency of their loads in the few workgroups
// that have the hubs, hence 16 entries a thread in flight; the tiles by their
// stores (5.1 GB at bs 64 on R-MAT 2^20: 1.0 ms).  Merging these block rows'
// CSR rows takes one dependent step per tile: counting R-MAT 2^20 at bs 64 took
// 1.1 ms that way and filling it 2.1; now 0.29 and 0.29 + 1.0, a count and a
// fill together 4.9 -> 2.5 ms (bs 8 3.7 -> 1.2, 2^22 at bs 8 10.0 -> 5.1).
#include <algorithm>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {
namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
// Block columns of a bitmap: 32 KB, four workgroups a CU; wider matrices take
// several walks.
constexpr int32_t kColWindow = 1 << 18;

template <int BS>
constexpr int kShift = BS == 8 ? 3 : BS == 16 ? 4 : BS == 32 ? 5 : 6;

// Sum of v over the workgroup (every thread gets it).
__device__ __forceinline__ int64_t block_sum(int64_t v, int64_t* sh) {
  for (int off = 1; off < kWave; off <<= 1) v += __shfl_xor(v, off);
  __syncthreads();
  if (lane_id() == 0) sh[threadIdx.x / kWave] = v;
  __syncthreads();
  int64_t s = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) s += sh[w];
  return s;
}

// Sum of v over the threads before this one; *all: over the workgroup.
__device__ __forceinline__ int block_before(int v, int* sh, int* all) {
  const int incl = wave_incl_scan(v);
  __syncthreads();
  if (lane_id() == kWave - 1) sh[threadIdx.x / kWave] = incl;
  __syncthreads();
  int before = incl - v, sum = 0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    if (w < (int)threadIdx.x / kWave) before += sh[w];
    sum += sh[w];
  }
  *all = sum;
  return before;
}

struct ColArgs {
  const int32_t *rp, *ci;
  int32_t nrows, ncols;
  int32_t window;  // block columns of the bitmap
  const int32_t *list, *nlist;
  int32_t* cnt;        // count: tiles of each block row
  int* err;            // count: PACKERR flags
  const int64_t* off;  // columns: first tile of each block row
  int32_t* colind;
};

// Entries of a thread in flight; in runs long enough, kLong.
constexpr int kUnroll = 4;
constexpr int kLong = 16;

// A block row's tiles, and whether its rows are in range and ascending by
// block column: the descents between neighbours of the whole run have to be
// those at row starts.
template <int BS>
__global__ __launch_bounds__(kThreads) void k_block_count(const ColArgs a) {
  extern __shared__ uint32_t bm[];
  __shared__ int64_t sh[kWaves];
  constexpr int S = kShift<BS>;
  const int tid = threadIdx.x;
  const int64_t nlist = *a.nlist;
  if (blockIdx.x >= nlist) return;
  const int nwords = (a.window + 31) / 32;
  for (int w = tid; w < nwords; w += kThreads) bm[w] = 0;
  __syncthreads();
  const int32_t nbc = (int32_t)(((int64_t)a.ncols + BS - 1) >> S);
  for (int64_t li = blockIdx.x; li < nlist; li += gridDim.x) {
    const int64_t I = a.list[li];
    const int64_t row0 = I * BS, row1 = min(row0 + BS, (int64_t)a.nrows);
    const int32_t p0 = a.rp[row0];
    const uint32_t n = (uint32_t)(a.rp[row1] - p0);
    const int32_t* ci = a.ci + p0;
    int tiles = 0, falls = 0;
    if (tid < row1 - row0) {
      const int32_t s = a.rp[row0 + tid], e = a.rp[row0 + tid + 1];
      if (s > p0 && s < e && (a.ci[s - 1] >> S) > (a.ci[s] >> S)) --falls;
    }
    int32_t w0 = 0;
    do {  // once where the matrix has no columns: the entries are out of range
      auto turn = [&](auto unroll, uint32_t p) {
        constexpr int U = unroll;
        int32_t b[U], before[U];
        uint32_t was[U];
        bool in = true;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t q = min(p + u * kThreads, n - 1);
          const int32_t c = ci[q];
          in = in && c >= 0 && c < a.ncols;
          b[u] = c >> S;
          before[u] = ci[q - (q > 0)] >> S;
        }
        if (!in) atomicOr(a.err, PACKERR_COLRANGE);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const bool own = p + u * kThreads < n;
          if (w0 == 0) falls += own && before[u] > b[u];
          // marked by the entry before it, or outside the window
          const bool skip = !in || !own || (before[u] == b[u] && p + u * kThreads > 0) || b[u] < w0 ||
                            b[u] - w0 >= a.window;
          b[u] = skip ? -1 : b[u] - w0;
          was[u] = bm[max(b[u], 0) >> 5];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t bit = 1u << (b[u] & 31);
          if (b[u] >= 0 && !(was[u] & bit)) tiles += (atomicOr(&bm[b[u] >> 5], bit) & bit) == 0;
        }
      };
      uint32_t p = tid;
      for (; p - tid + kLong * kThreads <= n; p += kLong * kThreads) turn(std::integral_constant<int, kLong>(), p);
      for (; p < n; p += kUnroll * kThreads) turn(std::integral_constant<int, kUnroll>(), p);
      __syncthreads();
      if (nwords <= 2 * (int64_t)n) {
        for (int w = tid; w < nwords; w += kThreads) bm[w] = 0;
      } else {
        for (uint32_t q = tid; q < n; q += kThreads) {
          const int32_t c = ci[q], b = (c >> S) - w0;
          if (c >= 0 && c < a.ncols && b >= 0 && b < a.window) bm[b >> 5] = 0;
        }
      }
      __syncthreads();
      w0 += a.window;
    } while (w0 < nbc);
    const int64_t sum = block_sum(((int64_t)falls << 32) + tiles, sh);
    if (tid == 0) {
      a.cnt[I] = (int32_t)sum;
      if (sum >> 32) atomicOr(a.err, PACKERR_UNSORTED);
    }
  }
}

// A block row's columns, ascending.  A second bitmap marks the first one's
// words that have a bit, so that only those are looked at, one a thread.
template <int BS>
__global__ __launch_bounds__(kThreads) void k_block_cols(const ColArgs a) {
  extern __shared__ uint32_t bm[];
  __shared__ uint32_t used[kColWindow / 1024];
  __shared__ int sh[kWaves];
  constexpr int S = kShift<BS>;
  const int tid = threadIdx.x;
  const int64_t nlist = *a.nlist;
  if (blockIdx.x >= nlist) return;
  const int nwords = (a.window + 31) / 32;
  uint16_t* words = (uint16_t*)(bm + nwords);
  for (int w = tid; w < nwords; w += kThreads) bm[w] = 0;
  static_assert(kColWindow / 1024 <= kThreads, "a thread per word of the second bitmap");
  if (tid < kColWindow / 1024) used[tid] = 0;
  __syncthreads();
  const int32_t nbc = (int32_t)(((int64_t)a.ncols + BS - 1) >> S);
  for (int64_t li = blockIdx.x; li < nlist; li += gridDim.x) {
    const int64_t I = a.list[li];
    const int64_t row0 = I * BS, row1 = min(row0 + BS, (int64_t)a.nrows);
    const int32_t p0 = a.rp[row0];
    const uint32_t n = (uint32_t)(a.rp[row1] - p0);
    const int32_t* ci = a.ci + p0;
    int64_t base = a.off[I];
    for (int32_t w0 = 0; w0 < nbc; w0 += a.window) {
      auto turn = [&](auto unroll, uint32_t p) {
        constexpr int U = unroll;
        int32_t b[U], before[U];
        uint32_t was[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t q = min(p + u * kThreads, n - 1);
          b[u] = ci[q] >> S;
          before[u] = ci[q - (q > 0)] >> S;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          // marked by the entry before it, or outside the window
          const bool skip = (before[u] == b[u] && p + u * kThreads > 0) || b[u] < w0 || b[u] - w0 >= a.window;
          b[u] = skip ? -1 : b[u] - w0;
          was[u] = bm[max(b[u], 0) >> 5];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const uint32_t bit = 1u << (b[u] & 31);
          const int w = b[u] >> 5;
          if (b[u] >= 0 && !(was[u] & bit) && atomicOr(&bm[w], bit) == 0) atomicOr(&used[w >> 5], 1u << (w & 31));
        }
      };
      uint32_t p = tid;
      for (; p - tid + kLong * kThreads <= n; p += kLong * kThreads) turn(std::integral_constant<int, kLong>(), p);
      for (; p < n; p += kUnroll * kThreads) turn(std::integral_constant<int, kUnroll>(), p);
      __syncthreads();
      uint32_t m = tid < kColWindow / 1024 ? used[tid] : 0;
      int nused;
      int at = block_before(__popc(m), sh, &nused);
      if (m) used[tid] = 0;
      while (m) {
        words[at++] = (uint16_t)(tid * 32 + __builtin_ctz(m));
        m &= m - 1;
      }
      __syncthreads();
      for (int j0 = 0; j0 < nused; j0 += kThreads) {
        const int j = j0 + tid;
        const int w = j < nused ? words[j] : 0;
        uint32_t bits = 0;
        if (j < nused) {
          bits = bm[w];
          bm[w] = 0;
        }
        int all;
        int64_t to = base + block_before(__popc(bits), sh, &all);
        while (bits) {
          a.colind[to++] = w0 + w * 32 + __builtin_ctz(bits);
          bits &= bits - 1;
        }
        base += all;
      }
      __syncthreads();
    }
  }
}

// ---- tiles.  A window of kWin tiles is built at a time (32 KB at bs 32/64, 8
// and 16 KB at bs 8/16); an item is up to kItemWindows windows of a block row.
template <int BS>
constexpr int kWin = BS == 8 ? 1024 : BS == 16 ? 512 : BS == 32 ? 256 : 64;
// Windows of an item: as many as hold about kItemNnz entries, at most kItemWindows.
constexpr int kItemWindows = 8;
constexpr int64_t kItemNnz = 4096;

struct ItemArgs {
  const int32_t *rp, *list;
  int32_t nrows, n, bs, win;
  const int64_t* off;
};
__device__ __forceinline__ int64_t item_tiles(const ItemArgs& a, int64_t I, int64_t T) {
  const int64_t nnz = a.rp[min((I + 1) * a.bs, (int64_t)a.nrows)] - a.rp[I * a.bs];
  const int64_t w = kItemNnz * T / max(nnz * a.win, (int64_t)1);
  return a.win * min(max(w, (int64_t)1), (int64_t)kItemWindows);
}
__global__ __launch_bounds__(256) void k_items_count(const ItemArgs a, int32_t* __restrict__ cnt) {
  const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= a.n) return;
  const int64_t I = a.list[h], T = a.off[I + 1] - a.off[I], it = item_tiles(a, I, T);
  cnt[h] = (int32_t)((T + it - 1) / it);
}

// items: block row, first tile in it, tiles.
__global__ __launch_bounds__(256) void k_items_fill(const ItemArgs a, const int64_t* __restrict__ ioff,
                                                    int4* __restrict__ items) {
  const int64_t h = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= a.n) return;
  const int64_t I = a.list[h], T = a.off[I + 1] - a.off[I], it = item_tiles(a, I, T);
  int64_t k = ioff[h];
  for (int64_t t = 0; t < T; t += it) items[k++] = make_int4((int)I, (int)t, (int)min(it, T - t), 0);
}

// Block rows of more than `above` nonzeros, in any order.
__global__ __launch_bounds__(1024) void k_heavy(const int32_t* __restrict__ rp, int32_t nrows, int32_t nbr, int bs,
                                                int32_t above, int32_t* __restrict__ list, int32_t* __restrict__ n) {
  __shared__ int sh[1024 / kWave];
  const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int wave = threadIdx.x / kWave;
  const bool heavy = I < nbr && rp[min((I + 1) * bs, (int64_t)nrows)] - rp[I * bs] > above;
  const unsigned long long m = __ballot(heavy);
  if (lane_id() == 0) sh[wave] = __popcll(m);
  __syncthreads();
  if (threadIdx.x == 0) {  // one atomic a workgroup
    int sum = 0;
    for (int w = 0; w < 1024 / kWave; ++w) sum += sh[w];
    int at = sum ? atomicAdd(n, sum) : 0;
    for (int w = 0; w < 1024 / kWave; ++w) {
      const int c = sh[w];
      sh[w] = at;
      at += c;
    }
  }
  __syncthreads();
  if (heavy) list[sh[wave] + __popcll(m & ((1ull << lane_id()) - 1))] = (int32_t)I;
}

struct TileArgs {
  const int32_t *rp, *ci;
  int32_t nrows;
  const int64_t* off;     // first tile of each block row
  const int32_t* colind;
  const int64_t* nitems;
  const int4* items;
  void* tiles;
};

// DIR 0: word = tile row, bit bs-1-c; DIR 1: word = tile column, bit bs-1-r.
// VEC: bytes per store (the tiles' alignment).
template <int BS, int DIR, int VEC>
__global__ __launch_bounds__(kThreads) void k_fill_tiles(const TileArgs a) {
  constexpr int S = kShift<BS>, WIN = kWin<BS>, U = kUnroll;
  constexpr int TB = BS * BS / 8;  // bytes of a tile
  __shared__ __align__(16) uint32_t buf[WIN * TB / 4];
  __shared__ int32_t cols[WIN];
  __shared__ int32_t at[BS], end[BS];  // the rows' next entries and ends
  __shared__ int32_t rest[BS], live[BS];  // rows with entries of the window left
  __shared__ int nrest;
  const int tid = threadIdx.x;
  const int64_t nitems = *a.nitems;
  if (blockIdx.x >= nitems) return;
  for (int w = tid; w < WIN * TB / 4; w += kThreads) buf[w] = 0;
  for (int64_t it = blockIdx.x; it < nitems; it += gridDim.x) {
    const int4 item = a.items[it];
    const int64_t I = item.x;
    const int64_t ta = a.off[I] + item.y, tb = ta + item.z;
    const int64_t row = I * BS + tid;
    if (tid < BS) {
      int32_t p = 0, pe = 0;
      if (row < a.nrows) {
        p = a.rp[row];
        pe = a.rp[row + 1];
        if (item.y > 0) {  // from the item's first column on
          const int32_t first = a.colind[ta];
          int32_t hi = pe;
          while (p < hi) {
            const int32_t mid = p + (hi - p) / 2;
            if ((a.ci[mid] >> S) < first) p = mid + 1;
            else hi = mid;
          }
        }
      }
      at[tid] = p;
      end[tid] = pe;
    }
    for (int64_t t0 = ta; t0 < tb; t0 += WIN) {
      const int nt = (int)min((int64_t)WIN, tb - t0);
      for (int k = tid; k < nt; k += kThreads) cols[k] = a.colind[t0 + k];
      __syncthreads();
      const int32_t last = cols[nt - 1];
      int lg = 31 - __builtin_clz(kThreads / BS);  // log2 of the lanes per row
      for (int n = BS;;) {
        // each row's next entries, U a lane, up to block column `last`
        const int k = tid >> lg, s = tid & ((1 << lg) - 1);
        int used = 0, r = 0;
        int64_t p = 0, pe = 0;
        if (k < n) {
          r = n == BS ? k : rest[k];
          p = at[r];
          pe = end[r];
          int32_t c[U];
#pragma unroll
          for (int u = 0; u < U; ++u) c[u] = p < pe ? a.ci[min(p + s + (u << lg), pe - 1)] : 0;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int32_t b = c[u] >> S;
            if (p + s + (u << lg) >= pe || b > last) continue;
            int lo = 0, hi = nt - 1;  // the tile: cols holds b
            while (lo < hi) {
              const int mid = (lo + hi) >> 1;
              if (cols[mid] < b) lo = mid + 1;
              else hi = mid;
            }
            const int col = c[u] & (BS - 1);
            const int word = DIR == 0 ? r : col, bit = BS - 1 - (DIR == 0 ? col : r);
            const int x = (lo * BS + word) * BS + bit;  // bit of the window
            atomicOr(&buf[x >> 5], 1u << (x & 31));
            ++used;
          }
        }
        // a row's entries come in order, so it goes on after those used
        for (int off = 1; off < (1 << lg); off <<= 1) used += __shfl_xor(used, off);
        const bool more = k < n && used == (U << lg) && p + used < pe;
        __syncthreads();  // every lane has read at[]
        if (k < n && s == 0) {
          at[r] = (int32_t)(p + used);
          live[k] = more;
        }
        if (!__syncthreads_or(more)) break;
        // the rows that have more share the lanes in the next turn
        if (tid < kWave) {
          const bool m = tid < n && live[tid];
          const int32_t mine = m ? (n == BS ? tid : rest[tid]) : 0;
          const unsigned long long mask = __ballot(m);
          if (m) rest[__popcll(mask & ((1ull << tid) - 1))] = mine;
          if (tid == 0) nrest = __popcll(mask);
        }
        __syncthreads();
        n = nrest;
        lg = 0;
        while (lg < 6 && (n << (lg + 1)) <= kThreads) ++lg;
      }
      // the window goes out whole, cleared behind
      char* out = (char*)a.tiles + t0 * TB;
      if constexpr (VEC == 16) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        for (int k = tid; k < nt * (TB / 16); k += kThreads) {
          __builtin_nontemporal_store(((const u32x4*)buf)[k], (u32x4*)out + k);
          ((u32x4*)buf)[k] = (u32x4)(0u);
        }
      } else if constexpr (VEC == 8) {
        for (int k = tid; k < nt * (TB / 8); k += kThreads) {
          __builtin_nontemporal_store(((const uint64_t*)buf)[k], (uint64_t*)out + k);
          ((uint64_t*)buf)[k] = 0;
        }
      } else {
        for (int k = tid; k < nt * BS; k += kThreads) ((word_t<BS>*)out)[k] = ((const word_t<BS>*)buf)[k];
        __syncthreads();
        for (int k = tid; k < nt * (TB / 4); k += kThreads) buf[k] = 0;
      }
      __syncthreads();
    }
  }
}

template <int BS, bool FILL>
int launch_cols(ColArgs a, int32_t rows, hipStream_t st) {
  if (rows == 0) return GBO_OK;
  const int64_t nbc = ((int64_t)a.ncols + BS - 1) / BS;
  a.window = (int32_t)std::min<int64_t>(std::max<int64_t>(nbc, 1), kColWindow);
  const size_t nwords = (size_t)(a.window + 31) / 32, lds = nwords * (FILL ? 6 : 4);
  // several times the workgroups that fit: block rows differ
  const int64_t per_cu = std::min<int64_t>(8, ((int64_t)156 << 10) / (int64_t)(lds + 2048));
  const unsigned blocks = (unsigned)std::min<int64_t>(rows, 4 * 256 * per_cu);
  if constexpr (FILL) k_block_cols<BS><<<blocks, kThreads, lds, st>>>(a);
  else k_block_count<BS><<<blocks, kThreads, lds, st>>>(a);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

template <int BS, int DIR>
int launch_tiles(const TileArgs& a, int64_t cap, hipStream_t st) {
  const unsigned blocks = (unsigned)std::min<int64_t>(cap, 1 << 20);
  const uintptr_t al = (uintptr_t)a.tiles;
  if constexpr (BS > 8) {
    if (al % 16 == 0) k_fill_tiles<BS, DIR, 16><<<blocks, kThreads, 0, st>>>(a);
    else k_fill_tiles<BS, DIR, 0><<<blocks, kThreads, 0, st>>>(a);
  } else {
    if (al % 8 == 0) k_fill_tiles<BS, DIR, 8><<<blocks, kThreads, 0, st>>>(a);
    else k_fill_tiles<BS, DIR, 0><<<blocks, kThreads, 0, st>>>(a);
  }
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

template <int BS>
int fill_t(int dir, const PackCsr& A, const HeavyRows& h, int32_t nheavy, const int64_t* off, int64_t T,
           int32_t* colind, void* tiles, Workspace& mem, hipStream_t st) {
  ColArgs c{};
  c.rp = A.rp;
  c.ci = A.ci;
  c.nrows = A.nrows;
  c.ncols = A.ncols;
  c.list = h.list;
  c.nlist = h.n;
  c.off = off;
  c.colind = colind;
  int rc = launch_cols<BS, true>(c, nheavy, st);
  if (rc) return rc;
  const int64_t cap = (int64_t)nheavy + T / kWin<BS>;  // items at most
  int32_t* icnt = nullptr;
  int64_t* ioff = nullptr;
  int4* items = nullptr;
  const char* who = "gbo_csr2bsr_fill_dev";
  if ((rc = mem.alloc(&icnt, sizeof(int32_t) * (size_t)nheavy, who)) ||
      (rc = mem.alloc(&ioff, sizeof(int64_t) * ((size_t)nheavy + 1), who)) ||
      (rc = mem.alloc(&items, sizeof(int4) * (size_t)cap, who)))
    return rc;
  const unsigned blocks = (unsigned)((nheavy + 255) / 256);
  const ItemArgs ia{A.rp, h.list, A.nrows, nheavy, BS, kWin<BS>, off};
  k_items_count<<<blocks, 256, 0, st>>>(ia, icnt);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(icnt, ioff, nheavy, st, mem))) return rc;
  k_items_fill<<<blocks, 256, 0, st>>>(ia, ioff, items);
  GBO_LAUNCH_CHECK();
  TileArgs t{};
  t.rp = A.rp;
  t.ci = A.ci;
  t.nrows = A.nrows;
  t.off = off;
  t.colind = colind;
  t.nitems = ioff + nheavy;
  t.items = items;
  t.tiles = tiles;
  return dir == 0 ? launch_tiles<BS, 0>(t, cap, st) : launch_tiles<BS, 1>(t, cap, st);
}

int unsupported(int bs) { return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs); }

}  // namespace

int64_t heavy_walks(int bs, int32_t ncols) { return (((int64_t)ncols + bs - 1) / bs + kColWindow - 1) / kColWindow; }

int heavy_list(int bs, const PackCsr& A, Workspace& mem, HeavyRows* h, const char* who, hipStream_t st) {
  // A merge's steps are the block row's tiles, unknown yet but at most its
  // nonzeros.  King grid, 1M vertices, 8 nonzeros a row in few tiles, merged and
  // here: bs 64 182 and 350 us, bs 32 182 and 500, bs 8 185 and 990.  12 nonzeros a
  // row at random, 2^20 rows: bs 64 3480 and 1560.  Bounds of 64 to 512 are within
  // 20% of the best on R-MAT 2^20; 16 nonzeros a row at random at bs 8, block rows
  // of 128: 2^20 rows 1033 us at a bound of 128, 640 at 256.
  const int32_t least = std::max(256, 8 * bs);
  // Each walk of a wider matrix costs a block row some 7 us of a workgroup whatever
  // it holds (2^23 rows of 40 at random, bs 8: 29.4 ms at a bound of 128, 16.4 at 768),
  // but a merge of a thousand tiles is as long as the rest of the pass (R-MAT 2^23 of
  // 12: 11.8, 12.6 and 20.3 ms at 512, 768 and 1024).
  const int64_t walks = heavy_walks(bs, A.ncols);
  h->above = walks > 1 ? (int32_t)std::max<int64_t>(least, std::min<int64_t>(192 * walks, 768)) : least;
  int rc;
  if ((rc = mem.alloc(&h->list, sizeof(int32_t) * (size_t)std::max(A.nbr, 1), who)) ||
      (rc = mem.alloc(&h->n, sizeof(int32_t), who)))
    return rc;
  GBO_HIP_CHECK(hipMemsetAsync(h->n, 0, sizeof(int32_t), st));
  if (A.nbr == 0) return GBO_OK;
  k_heavy<<<(unsigned)(((int64_t)A.nbr + 1023) / 1024), 1024, 0, st>>>(A.rp, A.nrows, A.nbr, bs, h->above, h->list, h->n);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

int heavy_count(int bs, const PackCsr& A, const HeavyRows& h, int32_t* cnt, int* err, hipStream_t st) {
  ColArgs a{};
  a.rp = A.rp;
  a.ci = A.ci;
  a.nrows = A.nrows;
  a.ncols = A.ncols;
  a.list = h.list;
  a.nlist = h.n;
  a.cnt = cnt;
  a.err = err;
  switch (bs) {
    case 8: return launch_cols<8, false>(a, A.nbr, st);
    case 16: return launch_cols<16, false>(a, A.nbr, st);
    case 32: return launch_cols<32, false>(a, A.nbr, st);
    case 64: return launch_cols<64, false>(a, A.nbr, st);
  }
  return unsupported(bs);
}

int heavy_fill(int bs, int dir, const PackCsr& A, const HeavyRows& h, int32_t nheavy, const int64_t* off, int64_t T,
               int32_t* colind, void* tiles, Workspace& mem, hipStream_t st) {
  if (nheavy == 0) return GBO_OK;
  switch (bs) {
    case 8: return fill_t<8>(dir, A, h, nheavy, off, T, colind, tiles, mem, st);
    case 16: return fill_t<16>(dir, A, h, nheavy, off, T, colind, tiles, mem, st);
    case 32: return fill_t<32>(dir, A, h, nheavy, off, T, colind, tiles, mem, st);
    case 64: return fill_t<64>(dir, A, h, nheavy, off, T, colind, tiles, mem, st);
  }
  return unsupported(bs);
}

}  // namespace gbo
