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
// ids (k_tc_light, k_tc_heavy), dense ones are counted by pairs of tiles
// (k_tc_pairs).
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

// row[i] = block row of tile tile[i] (null: i): the last J with rowptr[J] <= tile.
__global__ __launch_bounds__(256) void k_tile_block_row(const int32_t* __restrict__ rowptr, int32_t nbr,
                                                        const int32_t* __restrict__ tile, int64_t T,
                                                        int32_t* __restrict__ row) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= T) return;
  const int32_t t = tile ? tile[i] : (int32_t)i;
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
  for (const void* p : {(const void*)keys, (const void*)idx, (const void*)tmp}) mem.drop(p);
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
// window, each list going on where the last window ended: taken whole in each, R-MAT
// 2^23 of 12 took 729 ms, 2^24 of 8 1724, now 202 and 320).  A bitmap probe is a load and a shift, a hash probe a loop, so the
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
// whatever lists they come from.  `cursor` (of this lane's key, in LDS; null: the
// lists are taken whole): only elements below `until` are, and the key's next call
// goes on after them.
template <class Has>
__device__ __forceinline__ int64_t count_keys(const ListTcArgs& A, bool in, int32_t k, int64_t a0, int64_t di,
                                              bool searches, const Has& has, int32_t* cursor = nullptr,
                                              int64_t until = 0) {
  const int lane = lane_id();
  in = in && k < A.nkeys;
  int64_t c0 = in ? A.crp[k] : 0;
  int64_t dk = in ? A.crp[k + 1] - c0 : 0;
  int64_t hits = 0;
  const bool far = search_pays(dk, di);
  for (uint64_t m = __ballot(far && searches); m; m &= m - 1) {
    const int j = __builtin_ctzll(m);
    hits += count_searched(A.acol + __shfl((long long)a0, j), __shfl((long long)di, j),
                           A.ccol + __shfl((long long)c0, j), __shfl((long long)dk, j));
  }
  if (cursor && in && !far) {  // lists are ascending
    const int64_t from = searches ? 0 : *cursor;
    int64_t lo = from, hi = dk;
    if (until >= A.nids) lo = hi;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if (A.ccol[c0 + mid] < until) lo = mid + 1;
      else hi = mid;
    }
    *cursor = (int32_t)lo;
    c0 += from;
    dk = lo - from;
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
  __shared__ int32_t s_cursor[kHeavyKeys];  // windows: where each key's list goes on
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
        hits += count_keys(A, in, in ? ai[kk] : 0, a0, d, base == 0, has,
                           window < A.nids ? s_cursor + (in ? kk - k0 : 0) : nullptr, base + window);
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
// Dense tiles: a wave takes a mask tile (I,K), looks the block columns J of the
// shorter one of A's block row I and B's block column K up in the other, 64 at a
// time, and counts each match word against word under the mask: lane k holds
// column k of B's tile and walks the rows of A's (bs 64, whose words are scalar
// loads; bs 32, two matches at a time), or a lane counts a match of its own, a
// 64-bit AND and popcount per four (bs 16) or eight rows.  Nothing in it is as
// wide as the matrix: communities of 256 on 2^20 vertices at bs 8 / 16 / 64 take 1.4,
// 0.95 and 0.30 ms (with a vector of each row in LDS 7.6, 16.7 and 14.5; the tile
// pairs taken bit by bit before 4.6, 4.4 and 0.8), G(4096, 1) 0.22 to 0.37 ms (0.8 to
// 1.3).
struct PairTcArgs {
  const int32_t *a_rowptr, *a_colind, *a_row;  // a_row: block row of each tile
  const void* a_tiles;
  const int32_t *bt_ptr, *bt_row, *bt_tile;  // block columns of B: rows J, tiles
  const void* b_tiles;
  int64_t T;
  unsigned long long* count;
};

// The tile's 32-bit words (bs 8: two, bs 16: eight), whatever its alignment.
template <int BS>
__device__ __forceinline__ void load_words(const word_t<BS>* tiles, int64_t t, uint32_t (&w)[BS * BS / 32]) {
  __builtin_memcpy(w, tiles + t * BS, BS * BS / 8);
}

// Mask bits up to which a lane takes a bit (row r, column k) of the mask and reads
// the one word of A's and of B's tile that it needs, match after match, instead of
// walking the rows: a turn of 64 bits is worth some 5 of 64 rows (communities of
// 4096 at bs 64, 80 / 197 bits a tile: 0.62 / 1.03 ms, by rows 3.3; at bs 32 50 bits
// 2.2, by rows 6.0).
template <int BS>
constexpr int kMaskBits = BS == 64 ? 768 : 320;

template <int BS>
__global__ __launch_bounds__(256) void k_tc_pairs(const PairTcArgs A) {
  using W = word_t<BS>;
  __shared__ uint16_t s_bits[256 / kWave][BS <= 16 ? 1 : kMaskBits<BS>];
  uint16_t* __restrict__ bits = s_bits[threadIdx.x / kWave];
  const int lane = lane_id();
  const W* __restrict__ at = (const W*)A.a_tiles;
  const W* __restrict__ bt = (const W*)A.b_tiles;
  const int64_t nw = (int64_t)gridDim.x * (256 / kWave);
  int64_t hits = 0;
  for (int64_t t = wave_index(); t < A.T; t += nw) {  // wave-uniform
    const int32_t I = ld_uniform(A.a_row, t), K = ld_uniform(A.a_colind, t);
    const int64_t a0 = ld_uniform(A.a_rowptr, I), a1 = ld_uniform(A.a_rowptr, I + 1);
    const int64_t b0 = ld_uniform(A.bt_ptr, K), b1 = ld_uniform(A.bt_ptr, K + 1);
    const bool a_short = a1 - a0 <= b1 - b0;
    const int32_t* __restrict__ from = a_short ? A.a_colind : A.bt_row;
    const int32_t* __restrict__ in = a_short ? A.bt_row : A.a_colind;
    const int64_t f0 = a_short ? a0 : b0, f1 = a_short ? a1 : b1, i0 = a_short ? b0 : a0, i1 = a_short ? b1 : a1;
    // the mask: at bs 8/16 its words (scalar), else the rows of this lane's column
    // (bit r)
    uint32_t ms[BS <= 16 ? BS * BS / 32 : 1] = {};
    uint64_t m[1] = {};
    int nbits = 0;  // of the mask, where they are listed; else past kMaskBits
    if constexpr (BS <= 16) {
      load_words<BS>(at, t, ms);
#pragma unroll
      for (auto& v : ms) v = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
    } else {
      const W own = at[t * BS + lane % BS];
      const int k = lane % BS;
      const int mine = lane < BS ? popcw(own) : 0, incl = wave_incl_scan(mine);
      nbits = __builtin_amdgcn_readlane(incl, kWave - 1);
      if (nbits <= kMaskBits<BS>) {
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        uint64_t w = lane < BS ? (uint64_t)own : 0;
        for (int to = incl - mine; w; ++to) {
          const int p = __builtin_ctzll(w);
          w &= w - 1;
          bits[to] = (uint16_t)(lane * BS + (BS - 1 - p));
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      }
#pragma unroll
      for (int r = 0; r < BS && nbits > kMaskBits<BS>; ++r) {
        uint64_t row = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)own, r);
        if constexpr (BS == 64) row |= (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)((uint64_t)own >> 32), r) << 32;
        m[0] |= ((row >> (BS - 1 - k)) & 1ull) << r;
      }
    }
    int acc = 0;
    for (int64_t f = f0; f < f1; f += kWave) {
      int32_t tA = -1, tB = -1;
      if (f + lane < f1) {
        const int32_t J = from[f + lane];
        const int64_t at_ = lower_bound_i32(in, i0, i1, J);
        if (at_ < i1 && in[at_] == J) {
          tA = (int32_t)(a_short ? f + lane : at_);
          tB = A.bt_tile[a_short ? at_ : f + lane];
        }
      }
      uint64_t found = __ballot(tA >= 0);
      if constexpr (BS <= 16) {
        constexpr int Q = BS * BS / 32, F = 32 / BS;  // words of a tile, rows of a word
        constexpr uint32_t kOnes = BS == 8 ? 0x01010101u : 0x00010001u;
        uint32_t a[Q] = {}, b[Q] = {};
        if (tA >= 0) {
          load_words<BS>(at, tA, a);
          load_words<BS>(bt, tB, b);
        }
        if (found) {
#pragma unroll
          for (int k = 0; k < BS; ++k) {
            // column k of B's tile once for each row of a word
            constexpr uint32_t kSel[4] = {0x00000000u, 0x01010101u, 0x02020202u, 0x03030303u};
            const uint32_t bw = b[k / F];
            const uint32_t col = BS == 8 ? __builtin_amdgcn_perm(bw, bw, kSel[k % F])
                                         : __builtin_amdgcn_perm(bw, bw, k % F ? 0x03020302u : 0x01000100u);
#pragma unroll
            for (int q = 0; q < Q; ++q)  // under the rows of word q that have column k
              acc += __popc(a[q] & col & (((ms[q] >> (BS - 1 - k)) & kOnes) * (uint32_t)low_mask<BS>()));
          }
        }
      } else {
        constexpr int G = kWave / BS;
        const int g = lane / BS, k = lane % BS;
        while (found && nbits <= kMaskBits<BS>) {  // wave-uniform
          constexpr int U = 4;
          int64_t sa[U], sb[U];
          int n = 0;
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (found) {
              const int l = __builtin_ctzll(found);
              found &= found - 1;
              sa[u] = __builtin_amdgcn_readlane(tA, l);
              sb[u] = __builtin_amdgcn_readlane(tB, l);
              ++n;
            } else {
              sa[u] = sa[0], sb[u] = sb[0];
            }
          }
          for (int p = lane; p - lane < nbits; p += kWave) {
            const int e = bits[min(p, nbits - 1)];
            W x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = at[sa[u] * BS + e / BS] & bt[sb[u] * BS + e % BS];
#pragma unroll
            for (int u = 0; u < U; ++u) acc += p < nbits && u < n ? popcw(x[u]) : 0;
          }
        }
        while (found) {
          int mine = -1;
          int64_t first = 0;  // bs 64: the match, wave-uniform
#pragma unroll
          for (int h = 0; h < G; ++h) {
            if (found) {
              const int l = __builtin_ctzll(found);
              found &= found - 1;
              if (g == h) mine = l;
              first = l;
            }
          }
          const int32_t sA = __shfl(tA, mine < 0 ? 0 : mine), sB = __shfl(tB, mine < 0 ? 0 : mine);
          const W w = mine < 0 ? (W)0 : bt[(int64_t)sB * BS + k];
          if constexpr (BS == 64) {
            const int64_t ta = __builtin_amdgcn_readlane(tA, (int)first);
#pragma unroll 16
            for (int r = 0; r < BS; ++r) {
              const uint64_t row = ld_uniform(at, ta * BS + r);
              const uint32_t on = (uint32_t)((int32_t)((uint32_t)(m[0] >> (r & 32)) << (31 - (r & 31))) >> 31);
              acc += __popc((uint32_t)w & (uint32_t)row & on) + __popc((uint32_t)(w >> 32) & (uint32_t)(row >> 32) & on);
            }
          } else {
            const W own = mine < 0 ? (W)0 : at[(int64_t)sA * BS + k];
#pragma unroll
            for (int r = 0; r < BS; ++r) {
              const uint32_t r0 = (uint32_t)__builtin_amdgcn_readlane((int)own, r);
              const uint32_t r1 = (uint32_t)__builtin_amdgcn_readlane((int)own, BS + r);
              const uint32_t on = (uint32_t)((int32_t)((uint32_t)m[0] << (31 - r)) >> 31);
              acc += __popc((uint32_t)w & (g ? r1 : r0) & on);
            }
          }
        }
      }
    }
    hits += acc;
  }
  add_count(hits, A.count);
}

// Workgroups and threads of k_tc_heavy, whose workgroups hold `lds` bytes each:
// as many as fit a CU's 160 KB of LDS and 32 waves.
static void lds_grid(size_t lds, int* threads, int* blocks) {
  *threads = lds > ((size_t)40 << 10) ? kHeavyThreads : 256;
  *blocks = 256 * std::max(1, (int)std::min<size_t>(2048 / *threads, ((size_t)158 << 10) / (lds + 3072)));
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
  lds_grid(lds, &threads, &blocks);
  // always the most that a call needs: none lowers it between another's limit and launch
  GBO_HIP_CHECK(hipFuncSetAttribute((const void*)k_tc_heavy, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kWindow / 8)));
  k_tc_heavy<<<blocks, threads, lds, st>>>(t);
  GBO_LAUNCH_CHECK();
  k_tc_light<<<(unsigned)std::min<int64_t>(2048, ((int64_t)n + 4 * kTinyRows - 1) / (4 * kTinyRows)), 256, 0, st>>>(t);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

template <int BS>
static int tc_pairs(const PairTcArgs& t, hipStream_t st) {
  k_tc_pairs<BS><<<(unsigned)std::min<int64_t>((t.T + 3) / 4, 4096), 256, 0, st>>>(t);  // one atomic each
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// Nonzeros up to which the lists are counted, by the bits per tile: the lists' work
// grows with the square of a row's length, the pairs' with its tiles.  ms, lists /
// pairs:
//   bs 8    communities of 512 on 2^18 vertices, 32 tiles a block row, 3.2 bits
//           0.65 / 0.80, 6.0 1.64 / 0.80; of 4096, 256 tiles, 6.0 9.2 / 19.0; G(4096),
//           6.3 0.49 / 0.38, 12.7 0.74 / 0.37: the search in long rows costs
//   bs 16   512, 12 bits 0.61 / 0.58, 24 1.65 / 0.56; 4096, 12 4.5 / 5.0, 24 9.0 / 5.0;
//           G(20000) 12.7 2.6 / 7.1
//   bs 32   512, 19 bits 0.34 / 0.24, 47 0.53 / 0.24; 4096, 20 2.7 / 2.1, 97 9.2 /
//           2.7; G(20000) 20 0.9 / 2.9, 51 2.6 / 3.0
//   bs 64   512, 72 bits 0.32 / 0.20; 4096, 80 2.65 / 0.62; G(20000) 81 0.87 / 0.94, 204
//           2.5 / 1.7
// King grids hold 6 to 55 bits a tile (0.34 / 0.27 to 0.30 / 0.20), R-MAT up to 8 (2^18 2.2 /
// 7.3 to 2.6 / 12.7).
static int64_t tc_listed(int bs, int64_t tiles, int32_t nbr) {
  const int64_t bits = bs == 8 ? (tiles <= 64 * (int64_t)nbr ? 5 : 8) : bs == 16 ? 16 : bs == 32 ? 32 : 48;
  return bits * tiles;
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
  if ((rc = block_transpose(LT, mem, &bt_ptr, &bt_row, &bt_tile, st)) || (rc = expand_csr(L, mem, &a, st, tc_listed(L->bs, L->nblocks, L->nblockrows))))
    return rc;
  if (!a.col) {
    PairTcArgs t{};
    int32_t* a_row = nullptr;
    if ((rc = mem.alloc(&a_row, sizeof(int32_t) * (size_t)L->nblocks, "gbo_bsrbmm_tc"))) return rc;
    k_tile_block_row<<<(unsigned)((L->nblocks + 255) / 256), 256, 0, st>>>(L->rowptr, L->nblockrows, nullptr,
                                                                           L->nblocks, a_row);
    GBO_LAUNCH_CHECK();
    t.a_rowptr = L->rowptr;
    t.a_colind = L->colind;
    t.a_row = a_row;
    t.a_tiles = L->tiles;
    t.bt_ptr = bt_ptr;
    t.bt_row = bt_row;
    t.bt_tile = bt_tile;
    t.b_tiles = LT->tiles;
    t.T = L->nblocks;
    t.count = count;
    switch (L->bs) {
      case 8: rc = tc_pairs<8>(t, st); break;
      case 16: rc = tc_pairs<16>(t, st); break;
      case 32: rc = tc_pairs<32>(t, st); break;
      case 64: rc = tc_pairs<64>(t, st); break;
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
