// bsrbmm: bit-BSR x bit-BSR products reduced to a scalar.
//
// Triangle counting (bmm{N}_sparse_masked_v5, bsrbmm/bsrbmm.cu:969,1214):
//   count = sum_{i,k} A_ik (A B)_ik,  A = L packed by rows, B = L^T packed
//   by columns (word k of B tile (J,K) = column k of that tile).
// The reference walks, per mask tile (I,K), every tile (I,J) of block row I
// and binary-searches B's block row J for K -- O(deg^2 log) per block row.
// Here the block-column structure of B is transposed once (a stable radix
// sort of the tiles by block column on the device: csr2csc on blocks), and
// the count is, over the set bits (i, k) of A, |A_i and C_k|: row i of A
// against column k of B.  Sparse tiles are listed once as rows and columns of
// ids (k_tc_light, k_tc_heavy), dense ones are intersected word by word
// (k_tc_tiles).
//
// Plain product sum (bmm{N}_sparse, bsrbmm/bsrbmm.cu:296-555):
//   sum_{i,k} (A B)_ik = sum_j colsum_A(j) * rowsum_B(j),
// two linear passes over the tiles instead of the reference's tile-pair loop.
#include <algorithm>
#include <type_traits>

#include <rocprim/device/device_radix_sort.hpp>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {

// First index in [lo, hi) of sorted arr whose value is >= key.
__device__ __forceinline__ int64_t lower_bound_i32(const int32_t* __restrict__ arr, int64_t lo, int64_t hi, int32_t key) {
  while (lo < hi) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (arr[mid] < key) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

// colsum (rows=false): S[J*BS + c] += #rows of tile (I,J) with column c set.
// rowsum of a column-direction B (rows=true): word k of tile (J,K) holds
// column k with bit (BS-1-j) = row j, so S[J*BS + j] += #k with bit set --
// the same per-bit count over the words of the tile, indexed by the tile's
// block row instead of its block column.
template <int BS>
__global__ __launch_bounds__(256) void k_bitcount_by_col(const int32_t* __restrict__ rowptr,
                                                         const int32_t* __restrict__ colind,
                                                         const word_t<BS>* __restrict__ tiles, int64_t T,
                                                         int32_t nbr, bool by_block_row,
                                                         unsigned long long* __restrict__ S) {
  const int lane = lane_id();
  const int64_t t = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  if (t >= T) return;
  const uint64_t w = (lane < BS) ? (uint64_t)tiles[t * BS + lane] : 0ull;
  int32_t J;
  if (by_block_row) {
    // block row of tile t: upper_bound(rowptr, t) - 1
    int32_t lo = 0, hi = nbr;
    while (lo < hi) {
      const int32_t mid = lo + (hi - lo) / 2;
      if ((int64_t)rowptr[mid + 1] <= t) lo = mid + 1;
      else hi = mid;
    }
    J = lo;
  } else {
    J = colind[t];
  }
  int mycnt = 0;
  for (int cc = 0; cc < BS; ++cc) {
    const uint64_t b = __ballot((w >> (BS - 1 - cc)) & 1ull);
    if (lane == cc) mycnt = __popcll(b);
  }
  if (lane < BS && mycnt) atomicAdd(&S[(int64_t)J * BS + lane], (unsigned long long)mycnt);
}

__global__ __launch_bounds__(256) void k_dot_u64(const unsigned long long* __restrict__ x,
                                                 const unsigned long long* __restrict__ y, int64_t n,
                                                 unsigned long long* out) {
  uint64_t s = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    s += x[i] * y[i];
  for (int off = 1; off < kWave; off <<= 1) s += __shfl_xor(s, off);
  if (lane_id() == 0 && s) atomicAdd(out, (unsigned long long)s);
}

__global__ __launch_bounds__(256) void k_iota_i32(int32_t* __restrict__ v, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = (int32_t)i;
}

// ptr[c] = first position of sorted keys >= c, for c in [0, nbc].
__global__ __launch_bounds__(256) void k_col_bounds(const int32_t* __restrict__ keys, int64_t T, int32_t nbc,
                                                    int32_t* __restrict__ ptr) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c > nbc) return;
  ptr[c] = (int32_t)lower_bound_i32(keys, 0, T, (int32_t)c);
}

// row[i] = block row of tile tile[i]: the last J with rowptr[J] <= tile.
__global__ __launch_bounds__(256) void k_tile_block_row(const int32_t* __restrict__ rowptr, int32_t nbr,
                                                        const int32_t* __restrict__ tile, int64_t T,
                                                        int32_t* __restrict__ row) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T) return;
  const int32_t t = tile[i];
  int32_t lo = 0, hi = nbr;  // first J with rowptr[J + 1] > t
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if (rowptr[mid + 1] <= t) lo = mid + 1;
    else hi = mid;
  }
  row[i] = lo;
}

}  // namespace gbo

using namespace gbo;

// Block-CSC of a block structure on the device (csr2csc on blocks): a stable
// radix sort of the tile indices by block column.  The tiles are stored in
// block-row order, so every column's list comes out with ascending rows.
// The three outputs are owned by `mem` (the caller's allocations).
static int block_transpose(const gbo_bsr* B, Workspace& mem, int32_t** d_ptr, int32_t** d_row, int32_t** d_tile,
                           hipStream_t st) {
  const int32_t nbr = B->nblockrows, nbc = B->nblockcols;
  const int64_t T = B->nblocks;
  const size_t tb = sizeof(int32_t) * (size_t)std::max<int64_t>(T, 1);
  int rc;
  if ((rc = mem.alloc(d_ptr, sizeof(int32_t) * ((size_t)nbc + 1), "block_transpose")) ||
      (rc = mem.alloc(d_row, tb, "block_transpose")) || (rc = mem.alloc(d_tile, tb, "block_transpose")))
    return rc;
  int32_t *keys = nullptr, *idx = nullptr;
  void* tmp = nullptr;
  size_t tmp_bytes = 0;
  unsigned bits = 1;
  while (bits < 31 && (1ll << bits) <= nbc) ++bits;
  if ((rc = mem.alloc(&keys, tb, "block_transpose")) || (rc = mem.alloc(&idx, tb, "block_transpose"))) return rc;
  k_iota_i32<<<(unsigned)((T + 255) / 256), 256, 0, st>>>(idx, T);
  GBO_LAUNCH_CHECK();
  GBO_HIP_CHECK(rocprim::radix_sort_pairs(nullptr, tmp_bytes, B->colind, keys, idx, *d_tile, (size_t)T, 0, bits, st));
  if ((rc = mem.alloc(&tmp, std::max<size_t>(tmp_bytes, 1), "block_transpose"))) return rc;
  GBO_HIP_CHECK(rocprim::radix_sort_pairs(tmp, tmp_bytes, B->colind, keys, idx, *d_tile, (size_t)T, 0, bits, st));
  k_col_bounds<<<(unsigned)(((int64_t)nbc + 1 + 255) / 256), 256, 0, st>>>(keys, T, nbc, *d_ptr);
  GBO_LAUNCH_CHECK();
  k_tile_block_row<<<(unsigned)((T + 255) / 256), 256, 0, st>>>(B->rowptr, nbr, *d_tile, T, *d_row);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// ------------------------------------------ triangle counting on lists
// A_i goes into a set in LDS and the C_k are streamed past it: coalesced reads
// and one LDS probe per element.  (The form before worked on tiles: for a mask
// tile it looked the block columns of its row up in the rows of its column and
// gathered both tiles of every match, a chain of dependent loads for two or
// three bits: R-MAT 2^18 bs 32 13.0 ms against 2.0.)  Where C_k is much longer
// than A_i (a hub column under a short row) the elements of A_i are searched in
// C_k instead, so an edge costs about the shorter list.
//
// Rows of at most kTinyRow columns: eight to a wave.  Up to kLightRow: a wave
// each.  Their sets are hash tables of the wave's own, a quarter full at most.
// Longer rows: items of kHeavyKeys columns k, a workgroup takes one after
// another from a counter, the set a bitmap of up to 2^20 ids (more: window by
// window).  A bitmap probe is a load and a shift, a hash probe a loop, so the
// line is low: R-MAT 2^18 2.2 / 3.1 / 3.7 ms at 32 / 64 / 128 columns.
constexpr int kTinyRow = 8;
constexpr int kTinyRows = kWave / kTinyRow;  // tiny rows per wave
constexpr int kTinySlots = 32;
constexpr int kLightRow = 32;
constexpr int kLightSlots = 128;
constexpr int kHeavyKeys = 512;
constexpr int kHeavyThreads = 1024;
constexpr int64_t kWindow = (int64_t)1 << 20;  // ids of a bitmap: 128 KB of LDS

struct ListTcArgs {
  const int64_t* arp;   // A_i
  const int32_t* acol;
  const int64_t* crp;   // C_k
  const int32_t* ccol;
  int32_t nrows;        // rows of A
  int32_t nids;         // columns of A = rows of B: the ids in the sets
  int32_t nkeys;        // columns of B; a key past them (padding bits of A) has no list
  const int64_t* hoff;  // heavy items before row i (scan), [nrows + 1]
  const int2* items;    // heavy items: row, first key
  unsigned long long* next;  // heavy items taken
  unsigned long long* count;
};

// C_k is searched rather than streamed: a search is a chain of log2(dk)
// loads per 64 elements of A_i, a stream dk / 256 rounds.
__device__ __forceinline__ bool search_pays(int64_t dk, int64_t di) { return dk > 2048 * ((di + 63) / 64); }

// Elements of A_i (`di` from a) that are in c[0 .. dk), searched 64 at a time.
__device__ __forceinline__ int64_t count_searched(const int32_t* __restrict__ a, int64_t di,
                                                  const int32_t* __restrict__ c, int64_t dk) {
  int64_t hits = 0;
  for (int64_t e = lane_id(); e < di; e += kWave) {
    const int32_t v = a[e];
    int64_t lo = 0, hi = dk;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (c[mid] < v) lo = mid + 1;
      else hi = mid;
    }
    hits += lo < dk && c[lo] == v;
  }
  return hits;
}

// The keys of the wave's lanes (k, where `in`), each of the row of di columns
// from a0: the elements of their C_k that has(element, lane) holds, this
// lane's share.  Lists of 64 or more are streamed one after another by the
// whole wave; the shorter ones are laid end to end, 64 elements a round
// whatever lists they come from.
template <class Has>
__device__ __forceinline__ int64_t count_keys(const ListTcArgs& A, bool in, int32_t k, int64_t a0, int64_t di,
                                              bool searches, const Has& has) {
  const int lane = lane_id();
  in = in && k < A.nkeys;
  const int64_t c0 = in ? A.crp[k] : 0;
  const int64_t dk = in ? A.crp[k + 1] - c0 : 0;
  int64_t hits = 0;
  const bool far = search_pays(dk, di);
  for (uint64_t m = __ballot(far && searches); m; m &= m - 1) {
    const int j = __builtin_ctzll(m);
    hits += count_searched(A.acol + __shfl((long long)a0, j), __shfl((long long)di, j),
                           A.ccol + __shfl((long long)c0, j), __shfl((long long)dk, j));
  }
  for (uint64_t m = __ballot(!far && dk >= kWave); m; m &= m - 1) {
    const int j = __builtin_ctzll(m);
    const int32_t* __restrict__ c = A.ccol + __shfl((long long)c0, j);
    const int d = __shfl((int)dk, j);
    constexpr int U = 4;
    for (int e = lane; e < d; e += U * kWave) {
      int32_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = c[min(e + u * kWave, d - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) hits += e + u * kWave < d && has(v[u], j);
    }
  }
  const int w = dk < kWave ? (int)dk : 0;
  const int incl = wave_incl_scan(w);
  const int tot = __builtin_amdgcn_readlane(incl, kWave - 1);
  for (int p0 = 0; p0 < tot; p0 += kWave) {  // wave-uniform
    const int p = p0 + lane;
    int j = 0;  // the list of element p: how many lists end at or before p
#pragma unroll
    for (int step = kWave / 2; step >= 1; step >>= 1)
      if (__shfl(incl, j + step - 1) <= p) j += step;
    j = min(j, kWave - 1);
    const int e = p - (__shfl(incl, j) - __shfl(w, j));
    const int64_t b = __shfl((long long)c0, j);
    if (p < tot) hits += has(A.ccol[b + e], j);
  }
  return hits;
}

// One atomic per workgroup: thousands of waves queue on the address.
__device__ __forceinline__ void add_count(int64_t hits, unsigned long long* count) {
  __shared__ unsigned long long s_hits;
  if (threadIdx.x == 0) s_hits = 0;
  __syncthreads();
  for (int off = 1; off < kWave; off <<= 1) hits += __shfl_xor(hits, off);
  if (lane_id() == 0 && hits) atomicAdd(&s_hits, (unsigned long long)hits);
  __syncthreads();
  if (threadIdx.x == 0 && s_hits) atomicAdd(count, s_hits);
}

// Open addressing in N slots (a power of two), -1 = free; ids are not
// negative and at most a quarter of the slots are taken, so the loops end.
template <int N>
struct HashSet {
  static __device__ __forceinline__ uint32_t slot(int32_t v) {
    return (uint32_t)v * 2654435761u >> (32 - __builtin_ctz(N));
  }
  static __device__ __forceinline__ void insert(int32_t* t, int32_t v) {
    for (uint32_t s = slot(v);; s = (s + 1) % N) {
      const int32_t was = atomicCAS(&t[s], -1, v);
      if (was == -1 || was == v) return;
    }
  }
  static __device__ __forceinline__ int has(const int32_t* t, int32_t v) {
    for (uint32_t s = slot(v);; s = (s + 1) % N) {
      const int32_t x = t[s];
      if (x == v) return 1;
      if (x < 0) return 0;
    }
  }
};

// A wave takes kTinyRows rows at a time: lane l looks at row l / kTinyRow.
__global__ __launch_bounds__(256) void k_tc_light(const ListTcArgs A) {
  constexpr int kSlots = kTinyRows * kTinySlots;
  static_assert(kSlots >= kLightSlots, "the tiny rows' tables hold a light row's");
  __shared__ int32_t tables[256 / kWave][kSlots];
  int32_t* __restrict__ table = tables[threadIdx.x / kWave];
  const int lane = lane_id(), g = lane / kTinyRow, e = lane % kTinyRow;
  const int64_t nw = (int64_t)gridDim.x * (256 / kWave);
  const int64_t groups = ((int64_t)A.nrows + kTinyRows - 1) / kTinyRows;
  int64_t hits = 0;
  for (int64_t w = wave_index(); w < groups; w += nw) {  // wave-uniform
    const int64_t i = w * kTinyRows + g;
    const int64_t a0 = i < A.nrows ? A.arp[i] : 0;
    const int64_t d = i < A.nrows ? A.arp[i + 1] - a0 : 0;
    const bool tiny = d > 0 && d <= kTinyRow;
    if (__ballot(tiny)) {
      const bool in = tiny && e < d;
      const int32_t k = in ? A.acol[a0 + e] : -1;
      for (int s = lane; s < kSlots; s += kWave) table[s] = -1;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (in) HashSet<kTinySlots>::insert(table + g * kTinySlots, k);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      hits += count_keys(A, in, k, a0, d, true, [&](int32_t v, int j) {
        return HashSet<kTinySlots>::has(table + j / kTinyRow * kTinySlots, v);
      });
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    for (uint64_t m = __ballot(e == 0 && d > kTinyRow && d <= kLightRow); m; m &= m - 1) {
      const int j = __builtin_ctzll(m);
      const int64_t b0 = __shfl((long long)a0, j);
      const int db = __shfl((int)d, j);
      const int32_t k = lane < db ? A.acol[b0 + lane] : -1;
      for (int s = lane; s < kLightSlots; s += kWave) table[s] = -1;
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      if (lane < db) HashSet<kLightSlots>::insert(table, k);
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      hits += count_keys(A, lane < db, k, b0, db, true,
                         [&](int32_t v, int) { return HashSet<kLightSlots>::has(table, v); });
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
  }
  add_count(hits, A.count);
}

__global__ __launch_bounds__(256) void k_tc_items_count(const int64_t* __restrict__ arp, int32_t n,
                                                        int32_t* __restrict__ cnt) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t d = arp[i + 1] - arp[i];
  cnt[i] = d > kLightRow ? (int32_t)((d + kHeavyKeys - 1) / kHeavyKeys) : 0;
}

__global__ __launch_bounds__(256) void k_tc_items_fill(const int64_t* __restrict__ hoff, int32_t n,
                                                       int2* __restrict__ items) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  for (int64_t k = hoff[i]; k < hoff[i + 1]; ++k) items[k] = make_int2((int)i, (int)(k - hoff[i]) * kHeavyKeys);
}

// `bits`: LDS, a bit per id of a window.
__global__ __launch_bounds__(kHeavyThreads) void k_tc_heavy(const ListTcArgs A) {
  extern __shared__ uint32_t bits[];
  __shared__ unsigned long long s_item;
  const int tid = threadIdx.x, nt = blockDim.x;
  const int64_t total = A.hoff[A.nrows];
  const int window = (int)min(kWindow, (int64_t)A.nids);
  for (int s = tid; s < (window + 31) / 32; s += nt) bits[s] = 0;
  int64_t hits = 0;
  while (true) {
    __syncthreads();
    if (tid == 0) s_item = atomicAdd(A.next, 1ull);
    __syncthreads();
    const int64_t it = (int64_t)s_item;
    if (it >= total) break;  // each workgroup ends here: the counter only grows
    const int32_t i = A.items[it].x;
    const int64_t a0 = A.arp[i], d = A.arp[i + 1] - a0;
    const int32_t* __restrict__ ai = A.acol + a0;
    const int64_t k0 = A.items[it].y, k1 = min(k0 + kHeavyKeys, d);
    for (int64_t base = 0; base < A.nids; base += window) {
      for (int64_t e = tid; e < d; e += nt) {
        const uint32_t v = (uint32_t)((int64_t)ai[e] - base);
        if (v < (uint32_t)window) atomicOr(&bits[v >> 5], 1u << (v & 31));
      }
      __syncthreads();
      auto has = [&](int32_t id, int) -> int {
        const uint32_t v = (uint32_t)((int64_t)id - base);
        return v < (uint32_t)window ? (bits[v >> 5] >> (v & 31)) & 1u : 0;
      };
      // 16 keys per wave and turn, so that the waves of a workgroup share the
      // keys of a short item
      constexpr int KW = 16;
      for (int64_t k = k0 + (tid / kWave) * KW; k < k1; k += (nt / kWave) * KW) {
        const int64_t kk = k + lane_id();
        const bool in = lane_id() < KW && kk < k1;
        hits += count_keys(A, in, in ? ai[kk] : 0, a0, d, base == 0, has);
      }
      __syncthreads();
      for (int64_t e = tid; e < d; e += nt) {
        const uint32_t v = (uint32_t)((int64_t)ai[e] - base);
        if (v < (uint32_t)window) bits[v >> 5] = 0;
      }
      __syncthreads();
    }
  }
  add_count(hits, A.count);
}

// ------------------------------------------- triangle counting on tiles
// Dense tiles: row i of A as a vector of bs-bit words in LDS (word J = row i of
// tile (I,J)), against which the words of B's block column K are counted for
// every mask tile (I,K) that has bits in row i: lane r holds column k = r of
// the 64 / bs tiles of a step, one AND and popcount per bs ids.  At bs 8 the
// vector holds the whole tiles of block row I, and one 64-bit AND and popcount
// takes a column word against the rows of the mask's column.  A workgroup takes
// one row (block row) after another from a counter; a matrix wider than the
// vector window by window.
struct TileTcArgs {
  const int32_t *a_rowptr, *a_colind;
  const void* a_tiles;
  const int32_t *bt_ptr, *bt_row, *bt_tile;  // block columns of B: rows J, tiles
  const void* b_tiles;
  int32_t nrows, nblocks;  // rows (bs 8: block rows); block columns of A = block rows of B
  unsigned long long *next, *count;
};

template <int BS>
__global__ __launch_bounds__(kHeavyThreads) void k_tc_tiles(const TileTcArgs A) {
  using W = word_t<BS>;
  using X = typename std::conditional<BS == 8, uint64_t, W>::type;  // an element of the vector
  constexpr int G = kWave / BS;
  extern __shared__ uint64_t xs64[];
  X* __restrict__ xs = (X*)xs64;
  __shared__ unsigned long long s_row;
  const int tid = threadIdx.x, nt = blockDim.x, lane = lane_id(), g = lane / BS, r = lane % BS;
  const W* __restrict__ at = (const W*)A.a_tiles;
  const W* __restrict__ bt = (const W*)A.b_tiles;
  const int window = (int)min(kWindow / (8 * (int64_t)sizeof(X)), (int64_t)A.nblocks);
  for (int s = tid; s < window; s += nt) xs[s] = (X)0;
  int64_t hits = 0;
  while (true) {
    __syncthreads();
    if (tid == 0) s_row = atomicAdd(A.next, 1ull);
    __syncthreads();
    // the last rows first: those of a lower triangle are the longest
    const int64_t i = A.nrows - 1 - (int64_t)s_row;
    if (i < 0) break;  // each workgroup ends here: the counter only grows
    const int64_t I = BS == 8 ? i : i / BS;
    const int64_t t0 = A.a_rowptr[I], t1 = A.a_rowptr[I + 1];
    auto own = [&](int64_t t) -> X {  // row i of tile t; bs 8: the tile
      if constexpr (BS == 8) {
        uint64_t w;
        __builtin_memcpy(&w, at + t * 8, 8);
        return w;
      } else {
        return at[t * BS + i % BS];
      }
    };
    for (int64_t base = 0; base < A.nblocks; base += window) {
      for (int64_t t = t0 + tid; t < t1; t += nt) {
        const int64_t J = A.a_colind[t] - base;
        if (J >= 0 && J < window) xs[J] = own(t);
      }
      __syncthreads();
      for (int64_t t = t0 + tid / kWave; t < t1; t += nt / kWave) {  // wave-uniform
        uint64_t m = (uint64_t)own(t);
        if constexpr (BS == 8) {
          // the bytes of the rows that have column r
          m = ((m >> (7 - r)) & 0x0101010101010101ull) * 0xFFull;
        } else {
          if (m == 0) continue;
          m = (m >> (BS - 1 - r)) & 1ull;
        }
        const int32_t K = A.a_colind[t];
        const int64_t e1 = A.bt_ptr[K + 1];
        int acc = 0;
#pragma unroll 4
        for (int64_t e = A.bt_ptr[K] + g; e < e1; e += G) {
          const int64_t J = A.bt_row[e] - base;
          if (J >= 0 && J < window) {
            const W w = bt[(int64_t)A.bt_tile[e] * BS + r];
            if constexpr (BS == 8) acc += __popcll(xs[J] & (w * 0x0101010101010101ull) & m);
            else acc += popcw((W)(w & xs[J]));
          }
        }
        if (m) hits += acc;
      }
      __syncthreads();
      for (int64_t t = t0 + tid; t < t1; t += nt) {
        const int64_t J = A.a_colind[t] - base;
        if (J >= 0 && J < window) xs[J] = (X)0;
      }
      __syncthreads();
    }
  }
  add_count(hits, A.count);
}

// Workgroups and threads of a kernel whose workgroups hold `lds` bytes each:
// as many as fit a CU's 160 KB of LDS and 32 waves (`wide`: of 16 waves each).
static void lds_grid(size_t lds, bool wide, int* threads, int* blocks) {
  *threads = wide || lds > ((size_t)40 << 10) ? kHeavyThreads : 256;
  *blocks = 256 * std::max(1, (int)std::min<size_t>(2048 / *threads, ((size_t)158 << 10) / (lds + 1024)));
}

// A kernel's limit is every caller's: always the most that a call needs, so that
// none lowers it between another's limit and launch.
static hipError_t lds_limit(const void* kernel) {
  return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kWindow / 8));
}

// The list form: A's rows are in `a`, B's block lists by column in `cl`.
static int tc_lists(const gbo_bsr* A, const CsrList& a, const TileLists& cl, unsigned long long* count,
                    Workspace& mem, hipStream_t st) {
  const char* who = "gbo_bsrbmm_tc";
  const int32_t n = A->nrows;
  CsrList c;
  int rc = expand_lists(cl, mem, &c, st);
  if (rc) return rc;
  int32_t* cnt = nullptr;
  int64_t* hoff = nullptr;
  int2* items = nullptr;
  unsigned long long* next = nullptr;
  // an item has at least kLightRow + 1 nonzeros of a row or kHeavyKeys of one
  const int64_t cap = a.nnz / (kLightRow + 1) + a.nnz / kHeavyKeys + 1;
  if ((rc = mem.alloc(&cnt, sizeof(int32_t) * (size_t)n, who)) ||
      (rc = mem.alloc(&hoff, sizeof(int64_t) * ((size_t)n + 1), who)) ||
      (rc = mem.alloc(&items, sizeof(int2) * (size_t)cap, who)) || (rc = mem.alloc(&next, sizeof(*next), who)))
    return rc;
  const unsigned nb = (unsigned)(((int64_t)n + 255) / 256);
  k_tc_items_count<<<nb, 256, 0, st>>>(a.rowptr, n, cnt);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(cnt, hoff, n, st, mem))) return rc;
  k_tc_items_fill<<<nb, 256, 0, st>>>(hoff, n, items);
  GBO_HIP_CHECK(hipMemsetAsync(next, 0, sizeof(*next), st));
  ListTcArgs t{};
  t.arp = a.rowptr;
  t.acol = a.col;
  t.crp = c.rowptr;
  t.ccol = c.col;
  t.nrows = n;
  t.nids = A->ncols;
  t.nkeys = cl.n;
  t.hoff = hoff;
  t.items = items;
  t.next = next;
  t.count = count;
  const size_t lds = (size_t)(std::min<int64_t>(kWindow, A->ncols) + 31) / 32 * 4;
  int threads = 0, blocks = 0;
  lds_grid(lds, false, &threads, &blocks);
  GBO_HIP_CHECK(lds_limit((const void*)k_tc_heavy));
  k_tc_heavy<<<blocks, threads, lds, st>>>(t);
  GBO_LAUNCH_CHECK();
  k_tc_light<<<(unsigned)std::min<int64_t>(2048, ((int64_t)n + 4 * kTinyRows - 1) / (4 * kTinyRows)), 256, 0, st>>>(t);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

template <int BS>
static int tc_tiles(const TileTcArgs& t, hipStream_t st) {
  constexpr size_t X = BS == 8 ? 8 : BS / 8;  // bytes of an element of the vector
  const size_t lds = ((size_t)std::min<int64_t>(kWindow / 8 / (int64_t)X, t.nblocks) * X + 7) / 8 * 8;
  int threads = 0, blocks = 0;
  lds_grid(lds, t.nrows < 2048, &threads, &blocks);  // few rows: more waves on each
  GBO_HIP_CHECK(lds_limit((const void*)k_tc_tiles<BS>));
  k_tc_tiles<BS><<<blocks, threads, lds, st>>>(t);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// Whether the tiles are dense enough for the word form.  The lists' work falls
// with the third power of the density, the words' hardly: G(4096, p), lists /
// words: bs 8 p 0.1 (6 bits a tile) 496 / 648 us, 0.2 (13) 723 / 647; bs 16 0.2
// (51) 693 / 861, 0.3 (77) 1049 / 858; bs 32 0.1 (102) 480 / 528, 0.2 (203) 708
// / 551; bs 64 0.05 (202) 373 / 395, 0.1 (403) 514 / 427; p 1 6.1-7.2 ms / 0.8-
// 1.3 (the tile-pair form before 1.6-6.1).  King grids, 0.8 bits a tile row,
// belong to the lists.
static bool tc_dense(int bs, int64_t nnz, int64_t tiles) {
  const int64_t bits = bs == 8 ? 12 : bs == 16 ? 64 : bs == 32 ? 128 : 320;
  return nnz > bits * tiles;
}

extern "C" {

int gbo_bsrbmm_tc(const gbo_bsr* L, const gbo_bsr* LT, uint64_t* d_count, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  int rc = validate_bsr(L, 0, "gbo_bsrbmm_tc(A)");
  if (rc) return rc;
  rc = validate_bsr(LT, 1, "gbo_bsrbmm_tc(B)");
  if (rc) return rc;
  if (L->bs != LT->bs) return set_error(GBO_EINVAL, "gbo_bsrbmm_tc: block sizes differ");
  if (L->nrows != L->ncols) return set_error(GBO_EINVAL, "gbo_bsrbmm_tc: the mask A must be square");
  if (L->ncols != LT->nrows || L->nrows != LT->ncols)
    return set_error(GBO_EINVAL, "gbo_bsrbmm_tc: B must be %d x %d", L->ncols, L->nrows);
  if (!d_count) return set_error(GBO_EINVAL, "gbo_bsrbmm_tc: null count");
  hipStream_t st = stream;
  GBO_HIP_CHECK(hipMemsetAsync(d_count, 0, sizeof(uint64_t), st));
  if (L->nblocks == 0 || LT->nblocks == 0) return GBO_OK;
  Workspace mem(st);
  int32_t *bt_ptr = nullptr, *bt_row = nullptr, *bt_tile = nullptr;
  unsigned long long* count = (unsigned long long*)d_count;
  CsrList a;
  if ((rc = block_transpose(LT, mem, &bt_ptr, &bt_row, &bt_tile, st)) || (rc = expand_csr(L, mem, &a, st))) return rc;
  if (tc_dense(L->bs, a.nnz, L->nblocks)) {
    TileTcArgs t{};
    t.a_rowptr = L->rowptr;
    t.a_colind = L->colind;
    t.a_tiles = L->tiles;
    t.bt_ptr = bt_ptr;
    t.bt_row = bt_row;
    t.bt_tile = bt_tile;
    t.b_tiles = LT->tiles;
    t.nrows = L->bs == 8 ? L->nblockrows : L->nrows;
    t.nblocks = L->nblockcols;
    t.count = count;
    if ((rc = mem.alloc(&t.next, sizeof(*t.next), "gbo_bsrbmm_tc"))) return rc;
    GBO_HIP_CHECK(hipMemsetAsync(t.next, 0, sizeof(*t.next), st));
    switch (L->bs) {
      case 8: rc = tc_tiles<8>(t, st); break;
      case 16: rc = tc_tiles<16>(t, st); break;
      case 32: rc = tc_tiles<32>(t, st); break;
      case 64: rc = tc_tiles<64>(t, st); break;
    }
  } else {
    TileLists cl;
    cl.bs = LT->bs;
    cl.nbr = LT->nblockcols;
    cl.n = LT->ncols;
    cl.T = LT->nblocks;
    cl.ptr = bt_ptr;
    cl.ind = bt_row;
    cl.tiles = LT->tiles;
    cl.perm = bt_tile;
    rc = tc_lists(L, a, cl, count, mem, st);
  }
  return rc;  // the scratch waits for the stream
  GBO_TRY_END
}

int gbo_bsrbmm_sum(const gbo_bsr* A, const gbo_bsr* B, uint64_t* d_sum, gbo_stream_t stream) {
  int rc = validate_bsr(A, 0, "gbo_bsrbmm_sum(A)");
  if (rc) return rc;
  rc = validate_bsr(B, 1, "gbo_bsrbmm_sum(B)");
  if (rc) return rc;
  if (A->bs != B->bs) return set_error(GBO_EINVAL, "gbo_bsrbmm_sum: block sizes differ");
  if (A->ncols != B->nrows) return set_error(GBO_EINVAL, "gbo_bsrbmm_sum: inner dimensions differ");
  if (!d_sum) return set_error(GBO_EINVAL, "gbo_bsrbmm_sum: null output");
  hipStream_t st = stream;
  const int bs = A->bs;
  const int64_t n = (int64_t)A->nblockcols * bs;
  AsyncAllocs mem(st);
  unsigned long long* S = nullptr;
  if ((rc = mem.alloc(&S, sizeof(unsigned long long) * 2 * std::max<int64_t>(n, 1), "gbo_bsrbmm_sum"))) return rc;
  GBO_HIP_CHECK(hipMemsetAsync(S, 0, sizeof(unsigned long long) * 2 * std::max<int64_t>(n, 1), st));
  GBO_HIP_CHECK(hipMemsetAsync(d_sum, 0, sizeof(uint64_t), st));
  auto launch = [&](const gbo_bsr* M, bool by_row, unsigned long long* out) {
    if (M->nblocks == 0) return;
    const unsigned blocks = (unsigned)((M->nblocks + 3) / 4);
    switch (bs) {
      case 8: k_bitcount_by_col<8><<<blocks, 256, 0, st>>>(M->rowptr, M->colind, (const uint8_t*)M->tiles, M->nblocks, M->nblockrows, by_row, out); break;
      case 16: k_bitcount_by_col<16><<<blocks, 256, 0, st>>>(M->rowptr, M->colind, (const uint16_t*)M->tiles, M->nblocks, M->nblockrows, by_row, out); break;
      case 32: k_bitcount_by_col<32><<<blocks, 256, 0, st>>>(M->rowptr, M->colind, (const uint32_t*)M->tiles, M->nblocks, M->nblockrows, by_row, out); break;
      case 64: k_bitcount_by_col<64><<<blocks, 256, 0, st>>>(M->rowptr, M->colind, (const uint64_t*)M->tiles, M->nblocks, M->nblockrows, by_row, out); break;
    }
  };
  launch(A, false, S);
  launch(B, true, S + n);
  GBO_LAUNCH_CHECK();
  k_dot_u64<<<256, 256, 0, st>>>(S, S + n, n, (unsigned long long*)d_sum);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

}  // extern "C"
