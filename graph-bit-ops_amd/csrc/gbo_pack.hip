// CSR -> bit-BSR packing on the GPU (replaces csr2bsr_batch_{N}, algorithm/
// csr2bsr_batch_bsrbmv.cu:180-947, and csr2bsr_batch_{N}_{row,col},
// bsrbmm/csr2bsr_batch.cu), vector packing (ToBit{N}Row) and the work
// decomposition ("plan") used by every bsrbmv/bsrbmm operation.
//
// The reference packs one block row per host-loop iteration through dense
// float tiles (cusparseScsr2bsr) and a ballot kernel.  Here one wavefront
// packs 64/bs block rows at once: lane r of a group follows CSR row r of its
// block row, the group takes the minimum pending block column (a k-way merge
// of the bs sorted rows), and every lane ORs its entries of that block
// column into its own row word -- which is directly word r of the tile in
// the reference layout (MSB = column 0).  Two passes: count tiles, scan, then
// fill colind/tiles.  No dense staging.  Block rows of many nonzeros are not
// merged (gbo_pack_fill.hip), or on very wide matrices merged in pieces.
#include <algorithm>
#include <cstring>
#include <vector>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {

// ------------------------------------------------------------------ scan
constexpr int kScanThreads = 256;
constexpr int kScanPer = 8;
constexpr int kScanTile = kScanThreads * kScanPer;

template <class TI>
__global__ __launch_bounds__(kScanThreads) void k_scan_reduce(const TI* __restrict__ in, int64_t n,
                                                              int64_t* __restrict__ bsum) {
  __shared__ int64_t sh[kScanThreads];
  const int64_t base = (int64_t)blockIdx.x * kScanTile;
  int64_t s = 0;
  for (int k = 0; k < kScanPer; ++k) {
    const int64_t i = base + threadIdx.x + (int64_t)k * kScanThreads;
    if (i < n) s += (int64_t)in[i];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = kScanThreads / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) bsum[blockIdx.x] = sh[0];
}

// Exclusive scan of one tile; thread t owns elements [base+t*P, base+t*P+P).
// In-place safe: each element is read and written by the same thread.
template <class TI, class TO>
__global__ __launch_bounds__(kScanThreads) void k_scan_apply(const TI* in, int64_t n,
                                                             const int64_t* __restrict__ boff,
                                                             TO* out) {
  __shared__ int64_t sh[kScanThreads];
  const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanPer;
  int64_t v[kScanPer];
  int64_t s = 0;
  for (int k = 0; k < kScanPer; ++k) {
    const int64_t i = base + k;
    v[k] = (i < n) ? (int64_t)in[i] : 0;
    s += v[k];
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < kScanThreads; off <<= 1) {
    const int64_t o = ((int)threadIdx.x >= off) ? sh[threadIdx.x - off] : 0;
    __syncthreads();
    sh[threadIdx.x] += o;
    __syncthreads();
  }
  int64_t run = sh[threadIdx.x] - s + (boff ? boff[blockIdx.x] : 0);
  for (int k = 0; k < kScanPer; ++k) {
    const int64_t i = base + k;
    if (i < n) out[i] = (TO)run;
    run += v[k];
    if (i == n - 1) out[n] = (TO)run;
  }
}

// The block sums' offsets of a scan of nb tiles (room for 2 nb + 1 int64 in
// bsum), then the scan itself; nested through itself where nb needs it.
template <class TI, class TO, class Alloc, class Drop>
static int scan_with(const TI* in, TO* out, int64_t n, hipStream_t st, Alloc alloc, Drop drop) {
  if (n <= 0) {
    GBO_HIP_CHECK(hipMemsetAsync(out, 0, sizeof(TO), st));
    return GBO_OK;
  }
  const int64_t nb = (n + kScanTile - 1) / kScanTile;
  if (nb == 1) {
    k_scan_apply<TI, TO><<<1, kScanThreads, 0, st>>>(in, n, nullptr, out);
    GBO_LAUNCH_CHECK();
    return GBO_OK;
  }
  int64_t* bsum = nullptr;
  int rc = alloc(&bsum, sizeof(int64_t) * (2 * nb + 1));
  if (rc) return rc;
  int64_t* boff = bsum + nb;
  k_scan_reduce<TI><<<(unsigned)nb, kScanThreads, 0, st>>>(in, n, bsum);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_with<int64_t, int64_t>(bsum, boff, nb, st, alloc, drop))) return rc;
  k_scan_apply<TI, TO><<<(unsigned)nb, kScanThreads, 0, st>>>(in, n, boff, out);
  GBO_LAUNCH_CHECK();
  drop(bsum);
  return GBO_OK;
}

// out[0..n] = exclusive prefix sums of in[0..n-1]; out[n] = total.
template <class TI, class TO>
int scan_exclusive(const TI* in, TO* out, int64_t n, hipStream_t st) {
  AsyncAllocs mem(st);
  return scan_with(in, out, n, st, [&](int64_t** p, size_t bytes) { return mem.alloc(p, bytes, "scan"); },
                   [](const void*) {});
}

template <class TI, class TO>
int scan_exclusive(const TI* in, TO* out, int64_t n, hipStream_t st, Workspace& mem) {
  return scan_with(in, out, n, st, [&](int64_t** p, size_t bytes) { return mem.alloc(p, bytes, "scan"); },
                   [&](const void* p) { mem.drop(p); });
}

template int scan_exclusive<int32_t, int32_t>(const int32_t*, int32_t*, int64_t, hipStream_t);
template int scan_exclusive<int32_t, int32_t>(const int32_t*, int32_t*, int64_t, hipStream_t, Workspace&);
template int scan_exclusive<int32_t, int64_t>(const int32_t*, int64_t*, int64_t, hipStream_t);
template int scan_exclusive<int32_t, int64_t>(const int32_t*, int64_t*, int64_t, hipStream_t, Workspace&);
template int scan_exclusive<int64_t, int64_t>(const int64_t*, int64_t*, int64_t, hipStream_t);
template int scan_exclusive<int64_t, int64_t>(const int64_t*, int64_t*, int64_t, hipStream_t, Workspace&);

// ---------------------------------------------------------------- packing
enum { PACK_COUNT = 0, PACK_ROW = 1, PACK_COL = 2, PACK_VALUES = 3 };

// Where values follow the tiles' bits, and on matrices of more than kMostWalks
// walks, a block row with more than kPieceNnz
// nonzeros is merged in pieces: ranges of block columns [lo, hi), one group
// each, cut at evenly spaced entries of the block row's longest CSR row.  A
// single group's merge over the hub block row of R-MAT s22 (129,447 tiles at
// bs 8, one dependent step per tile) had set the time of each whole pass
// (~75 ms).
constexpr int32_t kPieceNnz = 2048;

// The pieces: piece p is block row row[p] over block columns [lo[p], hi[p])
// (lo = INT_MIN: from the row's start, hi = INT_MAX: to its end).  Without a
// table (row == nullptr) piece p is block row p, whole.
struct PackPieces {
  const int32_t* row = nullptr;
  const int32_t* lo = nullptr;
  const int32_t* hi = nullptr;
  const int64_t* base = nullptr;  // fill: first tile of each piece
  int32_t* cnt = nullptr;         // count: tiles of each piece
  int32_t n = 0;
  int32_t above = INT_MAX;        // without a table: block rows of more nonzeros are left out
};

// Column indices a wave stages in LDS (4 KB): a merge step waits for LDS and
// not for memory (12 nonzeros a row, 2^20 rows at bs 8, count and fill:
// 690 -> 500 us).
constexpr int kStage = 1024;

// First index q in [q0, q1) with ci[q] / BS >= J (q1 if none).  On rows that
// are not sorted the result is still monotone in J, so the pieces of a row
// cover it exactly and the count pass sees every adjacent pair once.
template <int BS>
__device__ __forceinline__ int32_t first_blockcol_at_least(const int32_t* __restrict__ ci, int32_t q0, int32_t q1,
                                                           int32_t J) {
  while (q0 < q1) {
    const int32_t mid = q0 + (q1 - q0) / 2;
    if (ci[mid] / BS < J) q0 = mid + 1;
    else q1 = mid;
  }
  return q0;
}

// PIECES: by the table.  A kernel of its own, without the stage and the look at
// each block row's length, which cost the merge of pieces a tenth.
template <int BS, int MODE, bool PIECES>
__global__ __launch_bounds__(256) void k_pack(const int32_t* __restrict__ rp,
                                              const int32_t* __restrict__ ci, int32_t nrows,
                                              int32_t ncols, int32_t nbr,
                                              int32_t* __restrict__ bsr_rp,  // counts (COUNT) or rowptr
                                              int32_t* __restrict__ out_col,
                                              word_t<BS>* __restrict__ out_tiles,
                                              const uint32_t* __restrict__ val,
                                              const int64_t* __restrict__ woff,
                                              uint32_t* __restrict__ tval, int* __restrict__ err,
                                              const PackPieces pc) {
  using W = word_t<BS>;
  constexpr int G = kWave / BS;
  const int lane = lane_id();
  const int g = lane / BS, r = lane % BS;
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWave;
  const int64_t npc = PIECES ? (int64_t)pc.n : (int64_t)nbr;
  const int64_t pi = wave * G + g;  // piece of this group
  if (wave * G >= npc) return;      // wave-uniform
  bool blk_ok = pi < npc;
  const int64_t I = PIECES ? (blk_ok ? (int64_t)pc.row[pi] : 0) : pi;
  const int64_t row = I * BS + r;
  if (!PIECES && blk_ok && pc.above != INT_MAX) blk_ok = rp[min((I + 1) * BS, (int64_t)nrows)] - rp[I * BS] <= pc.above;
  int32_t p = 0, pe = 0;
  if (blk_ok && row < nrows) {
    const int32_t r0 = rp[row], r1 = rp[row + 1];
    p = r0;
    pe = r1;
    if constexpr (PIECES) {
      const int32_t lo = pc.lo[pi], hi = pc.hi[pi];
      if (lo != INT_MIN) p = first_blockcol_at_least<BS>(ci, r0, r1, lo);
      if (hi != INT_MAX) pe = first_blockcol_at_least<BS>(ci, r0, r1, hi);
      if (pe < p) pe = p;  // only on rows that are not sorted (flagged below)
      // the pair across the piece's start (pairs inside it are checked by the merge)
      if (MODE == PACK_COUNT && p > r0 && p < r1 && ci[p - 1] / BS > ci[p] / BS) atomicOr(err, PACKERR_UNSORTED);
    }
  }
  // the wave's rows are one run of the CSR: a short one is staged
  int32_t s0 = 0;
  bool staged = false;
  int32_t* sci = nullptr;
  if constexpr (!PIECES) {
    __shared__ int32_t stage[256 / kWave][kStage];
    sci = stage[threadIdx.x / kWave];
    const int64_t w0 = wave * G * BS;
    s0 = rp[w0];
    const int32_t s1 = rp[min(w0 + kWave, (int64_t)nrows)];
    staged = (int64_t)s1 - s0 <= kStage && __all(p == pe || (p >= s0 && pe <= s1));
    if (staged)
      for (int32_t q = lane; q < s1 - s0; q += kWave) sci[q] = ci[s0 + q];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  }
  int64_t base = 0;
  if (MODE != PACK_COUNT && blk_ok) base = pc.base ? pc.base[pi] : bsr_rp[I];
  int32_t k = 0;
  // one loop for staged entries, one for those in memory
  auto merge = [&](auto entry) {
    auto blockcol = [&](int32_t q) -> int32_t {
      const int32_t c = entry(q);
      if (MODE == PACK_COUNT && (c < 0 || c >= ncols)) {
        atomicOr(err, PACKERR_COLRANGE);
        return INT_MAX - 1;  // poison: still terminates
      }
      return c / BS;
    };
    int32_t cur = (p < pe) ? blockcol(p) : INT_MAX;
    while (true) {
      const int32_t m = group_min<BS>(cur);
      if (__all(m == INT_MAX)) break;
      uint64_t w = 0;
      int32_t p0 = p;
      if (m != INT_MAX) {
        while (cur == m) {
          w |= 1ull << (BS - 1 - (entry(p) % BS));
          ++p;
          const int32_t nxt = (p < pe) ? blockcol(p) : INT_MAX;
          if (MODE == PACK_COUNT && nxt < cur) atomicOr(err, PACKERR_UNSORTED);
          cur = nxt;
        }
      }
      if constexpr (MODE == PACK_ROW) {
        if (m != INT_MAX) {
          out_tiles[(base + k) * BS + r] = (W)w;
          if (r == 0) out_col[base + k] = m;
        }
      } else if constexpr (MODE == PACK_COL) {
        // Transpose the group's bs x bs bit tile with one ballot per column:
        // ballot bit (g*BS + r) = row r has column kk.
        uint64_t mine = 0;
        for (int kk = 0; kk < BS; ++kk) {
          const uint64_t b = __ballot((w >> (BS - 1 - kk)) & 1ull);
          const uint64_t grp = (b >> (g * BS)) & low_mask<BS>();
          if (kk == r) mine = brev_low<BS>(grp);
        }
        if (m != INT_MAX) {
          out_tiles[(base + k) * BS + r] = (W)mine;
          if (r == 0) out_col[base + k] = m;
        }
      } else if constexpr (MODE == PACK_VALUES) {
        // Rank of this row's first bit inside the tile = popcounts of the
        // rows above it (exclusive prefix over the group).
        int32_t cnt = (m != INT_MAX) ? popcw(w) : 0;
        int32_t incl = cnt;
        for (int off = 1; off < BS; off <<= 1) {
          const int32_t o = __shfl_up(incl, off, BS);
          if (r >= off) incl += o;
        }
        if (m != INT_MAX) {
          int64_t pos = woff[base + k] + (incl - cnt);
          for (int32_t q = p0; q < p; ++q) {
            if (q > p0 && ci[q] == ci[q - 1]) {
              tval[pos - 1] = min(tval[pos - 1], val[q]);
            } else {
              tval[pos++] = val[q];
            }
          }
        }
      }
      if (m != INT_MAX) ++k;
    }
  };
  if (!PIECES && staged) merge([&](int32_t q) -> int32_t { return sci[q - s0]; });
  else merge([&](int32_t q) -> int32_t { return ci[q]; });
  if constexpr (MODE == PACK_COUNT) {
    if (blk_ok && r == 0) {
      if constexpr (PIECES) pc.cnt[pi] = k;
      else bsr_rp[I] = k;
    }
  }
}

// Pieces per block row.
__global__ __launch_bounds__(256) void k_piece_n(const int32_t* __restrict__ rp, int32_t nrows, int32_t nbr, int bs,
                                                 int32_t* __restrict__ pn) {
  const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= nbr) return;
  const int64_t r0 = I * bs, r1 = min(r0 + bs, (int64_t)nrows);
  const int64_t nnz = (int64_t)rp[r1] - rp[r0];
  pn[I] = (int32_t)max((int64_t)1, (nnz + kPieceNnz - 1) / kPieceNnz);
}

// Piece table: block row I's pieces from poff[I], cut at evenly spaced
// entries of its longest CSR row.
__global__ __launch_bounds__(256) void k_piece_fill(const int32_t* __restrict__ rp, const int32_t* __restrict__ ci,
                                                    int32_t nrows, int32_t nbr, int bs,
                                                    const int32_t* __restrict__ poff, int32_t* __restrict__ prow,
                                                    int32_t* __restrict__ plo, int32_t* __restrict__ phi) {
  const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I >= nbr) return;
  const int32_t o = poff[I], P = poff[I + 1] - poff[I];
  int32_t best = 0, len = -1;
  const int64_t r0 = I * bs, r1 = min(r0 + bs, (int64_t)nrows);
  if (P > 1) {
    for (int64_t rr = r0; rr < r1; ++rr) {
      const int32_t l = rp[rr + 1] - rp[rr];
      if (l > len) {
        len = l;
        best = rp[rr];
      }
    }
  }
  for (int32_t j = 0; j < P; ++j) {
    prow[o + j] = (int32_t)I;
    plo[o + j] = j == 0 ? INT_MIN : ci[best + (int32_t)((int64_t)j * len / P)] / bs;
    phi[o + j] = j == P - 1 ? INT_MAX : ci[best + (int32_t)((int64_t)(j + 1) * len / P)] / bs;
  }
}

// off[I] = first tile of block row I's first piece (off[nbr] = total).
__global__ __launch_bounds__(256) void k_piece_off(const int32_t* __restrict__ poff, const int64_t* __restrict__ toff,
                                                   int32_t nbr, int64_t* __restrict__ off) {
  const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I <= nbr) off[I] = toff[poff[I]];
}

// rowptr[I] = first tile of block row I (rowptr[nbr] = total).
__global__ __launch_bounds__(256) void k_pack_rowptr(const int64_t* __restrict__ off, int32_t nbr,
                                                     int32_t* __restrict__ rowptr) {
  const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (I <= nbr) rowptr[I] = (int32_t)off[I];
}

struct PackSummary {
  int64_t total;
  int32_t err, heavy, given;
};
__global__ void k_pack_summary(const int64_t* __restrict__ total, const int* __restrict__ err,
                               const int32_t* __restrict__ heavy, const int32_t* __restrict__ given,
                               PackSummary* __restrict__ out) {
  out->total = *total;
  out->err = *err;
  out->heavy = *heavy;
  out->given = given ? *given : 0;
}

template <int BS>
__global__ __launch_bounds__(256) void k_tile_popc(const word_t<BS>* __restrict__ tiles, int64_t T,
                                                   int64_t* __restrict__ cnt) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= T) return;
  int64_t s = 0;
  for (int r = 0; r < BS; ++r) s += popcw(tiles[t * BS + r]);
  cnt[t] = s;
}

template <int BS>
__global__ __launch_bounds__(256) void k_pack_vec(const float* __restrict__ x, word_t<BS>* __restrict__ xb,
                                                  int32_t n, int32_t nw) {
  const int32_t j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= nw) return;
  uint64_t w = 0;
  for (int k = 0; k < BS; ++k) {
    const int64_t i = (int64_t)j * BS + k;
    if (i < n && x[i] > 0.0f) w |= 1ull << (BS - 1 - k);
  }
  xb[j] = (word_t<BS>)w;
}

// First block row of every chunk: the first row R with rowptr[R] >= b, or the
// row containing tile b when that row starts before b.  tail[c] = how many
// chunks after c hold tiles of a row that begins in c and is cut by its end
// (0: none is).  EVEN: chunks of `chunk` of the T tiles, `start` is not read.
// Clears the count slots: a call without a plan makes one in this one launch.
template <bool EVEN>
__global__ __launch_bounds__(256) void k_plan(const int32_t* __restrict__ rowptr, int32_t nbr,
                                              const int64_t* __restrict__ start, int32_t chunk, int64_t T,
                                              int32_t nchunks, int32_t* __restrict__ plan,
                                              int32_t* __restrict__ tail, unsigned long long* __restrict__ slots) {
  const int32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < kCountSlots) slots[c] = 0;
  if (c >= nchunks) return;
  auto at = [&](int32_t k) -> int64_t { return EVEN ? min((int64_t)k * chunk, T) : start[k]; };
  const int64_t b = at(c);
  int32_t lo = 0, hi = nbr;  // search in rowptr[0..nbr]
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if ((int64_t)rowptr[mid] < b) lo = mid + 1;
    else hi = mid;
  }
  int32_t R = lo;
  if (R > nbr || (int64_t)rowptr[R] > b) R -= 1;
  if (R >= nbr) R = nbr > 0 ? nbr - 1 : 0;
  if (R < 0) R = 0;
  plan[c] = R;
  if (c == nchunks - 1) tail[c] = 0;
  if (c == 0) return;
  const int64_t rs = rowptr[R], re = rowptr[R + 1];
  int32_t n = 0;
  if (rs < b && rs >= at(c - 1)) {
    int32_t l = c + 1, h = nchunks;  // first chunk that starts at or past the row's end
    if constexpr (EVEN) {
      l = (int32_t)min((re + chunk - 1) / chunk, (int64_t)nchunks);
    } else {
      while (l < h) {
        const int32_t mid = l + (h - l) / 2;
        if (start[mid] < re) l = mid + 1;
        else h = mid;
      }
    }
    n = l - c;
  }
  tail[c - 1] = n;
}

// start[c] = c * chunk, start[nchunks] = T.
__global__ __launch_bounds__(256) void k_even_starts(int64_t T, int32_t chunk, int32_t nchunks,
                                                     int64_t* __restrict__ start) {
  const int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (c <= nchunks) start[c] = min(c * chunk, T);
}

// ---- the library's own plan: chunks of about equal work.  Tiles are taken
// in units of kUnitTiles.  The work of a unit is kTileWork per tile and one per
// set bit past kFreeBits per tile (the value products gather one word per set
// bit, the first few of a tile with its own load; the count and the BFS step,
// whose tiles all cost the same, lose little to shorter chunks where tiles are
// dense, and the sparse rest keeps even chunks).  A unit starts a chunk where
// the prefix sum of the work passes a multiple of a chunk's work.  Cut
// evenly, a power-law matrix has chunks of ten to fifty times the mean number of
// bits, and one wave on the densest one sets the time of a sweep: R-MAT 2^18, 256 tiles a chunk, weighted min-plus bs 64
// 1.52 ms, sum bs 32 0.50 ms, against 0.15 and 0.08 ms of streaming.
template <int BS>
constexpr int kUnitTiles = BS == 64 ? 8 : 16;
template <int BS>
constexpr int kTileWork = BS >= 32 ? 16 : 8;
constexpr int kFreeBits = 4;

// What the host reads: the number of chunks (the last rank), of units of more than
// one and a half times the mean work, and all work.
enum { UNIT_CHUNKS, UNIT_DENSE, UNIT_TOTAL, UNIT_SUMS };

// Work of every unit.  Lanes take 16 bytes each: a unit is 8 lanes at bs 8,
// 32 at bs 16, a wave twice over at bs 32.  At bs 64 a wave reads a quarter of
// each tile, another quarter from tile to tile, and counts it four times: the
// bits are only a measure of work.
template <int BS>
__global__ __launch_bounds__(256) void k_unit_work(const uint4* __restrict__ tiles, int64_t T, int64_t nunits,
                                                   int32_t* __restrict__ work, unsigned long long* __restrict__ sums) {
  if (blockIdx.x == 0 && threadIdx.x == 0) sums[UNIT_DENSE] = 0;
  constexpr int UT = kUnitTiles<BS>, UL = BS == 8 ? 8 : BS == 16 ? 32 : 64;  // lanes per unit
  const int lane = lane_id();
  const int64_t u = (int64_t)wave_index() * (kWave / UL) + lane / UL;
  const int l = lane % UL;
  auto bits = [](uint4 v) { return __popc(v.x) + __popc(v.y) + __popc(v.z) + __popc(v.w); };
  int c = 0;
  if constexpr (BS == 8) {
    // lane l: tiles 2l, 2l + 1 of the unit; the last tile may be alone
    const int64_t t = u * UT + 2 * l;
    if (t + 1 < T) c = bits(tiles[t / 2]);
    else if (t < T) c = __popcll(((const uint64_t*)tiles)[t]);
  } else if constexpr (BS == 16) {
    const int64_t t = u * UT + l / 2;
    if (t < T) c = bits(tiles[t * 2 + l % 2]);
  } else if constexpr (BS == 32) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t t = u * UT + h * 8 + l / 8;
      if (t < T) c += bits(tiles[t * 8 + l % 8]);
    }
  } else {
    const int64_t t = u * UT + l / 8;
    if (t < T) c = 4 * bits(tiles[t * 32 + (t % 4) * 8 + l % 8]);
  }
  for (int off = 1; off < UL; off <<= 1) c += __shfl_xor(c, off);
  if (l == 0 && u < nunits) work[u] = UT * kTileWork<BS> + max(c - UT * kFreeBits, 0);
}

// Work of a chunk: that of `chunk` sparse tiles, and at bs 8/16 of as many mean
// ones where these are denser.  There a step of the count takes 256 and 64 tiles
// whatever they hold, and where all tiles are dense shorter chunks gain the value
// products nothing (G(16384, 1): bs 8 count 77 us at the 32 tiles that hold the work
// of 256 sparse ones, 24 at 256, min 1051 and 1007; bs 16 43 and 23, 1138 and 1011).
struct UnitCut {
  int32_t chunk, tile_work, unit;
  bool mean;
};
__device__ __forceinline__ int64_t cut_target(const int64_t* __restrict__ pre, int64_t nunits, const UnitCut& u) {
  const int64_t mean = u.mean ? pre[nunits] / (nunits * u.unit) : 0;
  return u.chunk * max((int64_t)u.tile_work, mean);
}
__device__ __forceinline__ bool unit_starts(const int64_t* __restrict__ pre, int64_t u, int64_t target) {
  return u == 0 || pre[u] / target != pre[u - 1] / target;
}

__global__ __launch_bounds__(256) void k_unit_heads(const int64_t* __restrict__ pre, int64_t nunits, const UnitCut cut,
                                                    int32_t* __restrict__ head,
                                                    unsigned long long* __restrict__ sums) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u < nunits) head[u] = unit_starts(pre, u, cut_target(pre, nunits, cut));
  const bool more = u < nunits && (pre[u + 1] - pre[u]) * 2 * nunits > pre[nunits] * 3;
  const int n = __syncthreads_count(more);
  if (threadIdx.x == 0 && n) atomicAdd(&sums[UNIT_DENSE], (unsigned long long)n);
  if (u == 0) sums[UNIT_TOTAL] = (unsigned long long)pre[nunits];
}

__global__ __launch_bounds__(256) void k_unit_chunks(const int64_t* __restrict__ pre,
                                                     const int64_t* __restrict__ rank, int64_t nunits,
                                                     const UnitCut cut, int64_t T, int64_t* __restrict__ start) {
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= nunits) return;
  if (unit_starts(pre, u, cut_target(pre, nunits, cut))) start[rank[u]] = u * cut.unit;
  if (u == 0) start[rank[nunits]] = T;
}

// Most tiles per chunk of the library's own plans: 256 on large matrices, and
// less where that leaves a sweep short of waves (8192 are resident), down to
// 16.  `uniform`: no tiles are denser than the rest, so that a chunk of as many
// tiles is as much work.
//   bs 8   a step of the count takes 256 tiles: G(n, m) with 1.6M tiles count /
//          min 15.3 / 19.1 us at 128 tiles, 14.6 / 17.6 at 256.  Where some tiles
//          are dense the sweep ends with them up to some 4M (R-MAT with 3.7M
//          count 37 / 42 us).
//   bs 16  256 tiles make few rounds of waves and an uneven last one (G(n, m)
//          with 8M min 95 / 103 us), with dense tiles up to 32M (R-MAT with 16.4M
//          count 172 / 197 us, with 23.7M min-plus 351 / 373; G(n, m) with 24M
//          488 / 479).
//   bs 32, 64  the starts of chunks of 128 tiles lie 16 and 64 KB apart, where
//          many waves read from the same memory channels at once: 96 / 128 tiles
//          on G(n, m) with 1.1M at bs 64 min 98 / 112 us, with 1.2M at bs 32
//          min-plus 37 / 43, R-MAT with 6.2M at bs 32 min-plus 309 / 337.  From
//          some 6M on a sum loses by the rows that more chunks cut (R-MAT with
//          7.7M at bs 64 799 / 771), from 12M on 256 are better still (G(n, m)
//          with 16.6M at bs 32 sum 512 / 487 at 128 / 256).  Uniform tiles of bs
//          32 that 8192 waves take in one round do so, in chunks of an odd
//          multiple of 16 tiles, from 208 on of 256: count of G(n, m) with 0.93M
//          28.0 / 25.3 us at 96 / 144, with 1.4M 36.7 / 35.4 at 96 / 176, with
//          1.6M 40.5 / 40.4 / 37.9 at 96 / 208 / 256; beyond one round 96 again
//          (with 2.3M min-plus 77 / 90 at 96 / 256).
// Small ones: G(n, m) with 0.5M tiles bs 8 12.6 / 8.3 / 8.1 us at 32 / 128 / 256;
// G(1024) bs 32 (1024 tiles) sum 9 / 18 / 59 us at 16 / 64 / 256.
int default_chunk(int bs, int64_t tiles, bool uniform) {
  const int64_t large = bs == 8 ? (uniform ? 1 : 4) : bs == 16 && !uniform ? 32 : 12;
  if (tiles >= large << 20) return 256;
  if (bs == 32 && uniform && tiles >= (512 << 10) && tiles <= (2ll << 20)) {
    const int once = 16 * (int)((tiles / 8192 + 15) / 16 | 1);
    return once > 192 ? 256 : once;
  }
  const int64_t most = bs >= 32 && tiles < (6ll << 20) ? 96 : 128;
  const int64_t c = (tiles / 4096 + 8) / 16 * 16;
  return (int)std::min(most, std::max<int64_t>(c, 16));
}

// Above this many tiles the densest chunk ends long before the sweep does,
// and even chunks of 256 are best (R-MAT 2^22 bs 8: count 465 us against 472
// with equal work, min 757 against 774).
constexpr int64_t kEvenTiles = 32ll << 20;

// The longest block row, in tiles, of a matrix whose chunks end at block rows:
// no product then has rows to zero or partial sums to add in a launch of its own
// (G(1024) of degree 20 at bs 32 count 7.7 -> 4.4 us, G(5003) of 16 at bs 8 sum 9.2
// -> 5.6, king grid of 62,500 at bs 64 min 10.0 -> 6.2).  Longer rows leave too
// few waves: min-plus at bs 32 with rows of 63 tiles 10.5 -> 13.2 us.  On larger
// matrices the rows have to be short against a chunk.
static int32_t whole_row(int bs, int64_t tiles, int32_t chunk) {
  const int32_t small = bs == 8 ? 256 : bs == 16 ? 128 : bs == 32 ? 32 : 16;
  return tiles <= (128 << 10) ? small : chunk / 8;
}

static bool bs_ok(int bs) { return bs == 8 || bs == 16 || bs == 32 || bs == 64; }

template <int BS, int MODE>
static int launch_pack(const int32_t* rp, const int32_t* ci, int32_t nrows, int32_t ncols, int32_t nbr,
                       int32_t* bsr_rp, int32_t* out_col, void* out_tiles, const uint32_t* val,
                       const int64_t* woff, uint32_t* tval, int* err, const PackPieces& pc, hipStream_t st) {
  constexpr int G = kWave / BS;
  const int64_t units = pc.row ? (int64_t)pc.n : (int64_t)nbr;
  const int64_t waves = (units + G - 1) / G;
  const int64_t blocks = (waves + 3) / 4;
  if (blocks == 0) return GBO_OK;
  auto* kernel = k_pack<BS, MODE, true>;
  if constexpr (MODE != PACK_VALUES) {  // values always come by the table
    if (!pc.row) kernel = k_pack<BS, MODE, false>;
  }
  kernel<<<(unsigned)blocks, 256, 0, st>>>(rp, ci, nrows, ncols, nbr, bsr_rp, out_col, (word_t<BS>*)out_tiles, val,
                                           woff, tval, err, pc);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

template <int MODE>
static int dispatch_pack(int bs, const int32_t* rp, const int32_t* ci, int32_t nrows, int32_t ncols,
                         int32_t nbr, int32_t* bsr_rp, int32_t* out_col, void* out_tiles,
                         const uint32_t* val, const int64_t* woff, uint32_t* tval, int* err,
                         const PackPieces& pc, hipStream_t st) {
  switch (bs) {
    case 8: return launch_pack<8, MODE>(rp, ci, nrows, ncols, nbr, bsr_rp, out_col, out_tiles, val, woff, tval, err, pc, st);
    case 16: return launch_pack<16, MODE>(rp, ci, nrows, ncols, nbr, bsr_rp, out_col, out_tiles, val, woff, tval, err, pc, st);
    case 32: return launch_pack<32, MODE>(rp, ci, nrows, ncols, nbr, bsr_rp, out_col, out_tiles, val, woff, tval, err, pc, st);
    case 64: return launch_pack<64, MODE>(rp, ci, nrows, ncols, nbr, bsr_rp, out_col, out_tiles, val, woff, tval, err, pc, st);
  }
  return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
}

static int check_err_flag(int h, const char* who) {
  if (h & PACKERR_COLRANGE) return set_error(GBO_EINVAL, "%s: column index out of range", who);
  if (h & PACKERR_UNSORTED) return set_error(GBO_EINVAL, "%s: CSR rows must be sorted ascending", who);
  return GBO_OK;
}

// The pieces of every block row, their tile counts (a count pass that also
// checks the rows: columns in range, block columns ascending) and the first
// tile of each (toff, npieces + 1 entries); *total = tiles.  Buffers are
// owned by `mem`.
struct PieceSet {
  PackPieces pc;
  const int32_t* poff = nullptr;  // each block row's first piece, nbr + 1
  int64_t total = 0;
};

static int make_pieces(int bs, const int32_t* d_rp, const int32_t* d_ci, int32_t nrows, int32_t ncols, int32_t nbr,
                       Workspace& mem, PieceSet* ps, const char* who, hipStream_t st) {
  int rc;
  int32_t *poff = nullptr, *prow = nullptr, *plo = nullptr, *phi = nullptr, *pcnt = nullptr;
  int64_t* toff = nullptr;
  int* d_err = nullptr;
  if ((rc = mem.alloc(&poff, sizeof(int32_t) * ((size_t)nbr + 1), who)) || (rc = mem.alloc(&d_err, sizeof(int), who)))
    return rc;
  GBO_HIP_CHECK(hipMemsetAsync(d_err, 0, sizeof(int), st));
  if (nbr > 0) {
    k_piece_n<<<(unsigned)(((int64_t)nbr + 255) / 256), 256, 0, st>>>(d_rp, nrows, nbr, bs, poff);
    GBO_LAUNCH_CHECK();
  }
  if ((rc = scan_exclusive<int32_t, int32_t>(poff, poff, nbr, st, mem))) return rc;
  int32_t np = 0;
  if ((rc = read_back(&np, poff + nbr, sizeof(int32_t), st))) return rc;
  if ((rc = mem.alloc(&prow, sizeof(int32_t) * std::max<int64_t>(np, 1), who)) ||
      (rc = mem.alloc(&plo, sizeof(int32_t) * std::max<int64_t>(np, 1), who)) ||
      (rc = mem.alloc(&phi, sizeof(int32_t) * std::max<int64_t>(np, 1), who)) ||
      (rc = mem.alloc(&pcnt, sizeof(int32_t) * std::max<int64_t>(np, 1), who)) ||
      (rc = mem.alloc(&toff, sizeof(int64_t) * ((size_t)np + 1), who)))
    return rc;
  if (nbr > 0) {
    k_piece_fill<<<(unsigned)(((int64_t)nbr + 255) / 256), 256, 0, st>>>(d_rp, d_ci, nrows, nbr, bs, poff, prow, plo,
                                                                         phi);
    GBO_LAUNCH_CHECK();
  }
  PackPieces pc;
  pc.row = prow;
  pc.lo = plo;
  pc.hi = phi;
  pc.cnt = pcnt;
  pc.n = np;
  if ((rc = dispatch_pack<PACK_COUNT>(bs, d_rp, d_ci, nrows, ncols, nbr, nullptr, nullptr, nullptr, nullptr,
                                      nullptr, nullptr, d_err, pc, st)))
    return rc;
  int err = 0;
  if ((rc = read_back(&err, d_err, sizeof(int), st)) || (rc = check_err_flag(err, who))) return rc;
  if ((rc = scan_exclusive<int32_t, int64_t>(pcnt, toff, np, st, mem))) return rc;
  if ((rc = read_back(&ps->total, toff + np, sizeof(int64_t), st))) return rc;
  if (ps->total >= ((int64_t)1 << 31))
    return set_error(GBO_ERANGE, "tile count %lld exceeds int32", (long long)ps->total);
  pc.cnt = nullptr;
  pc.base = toff;
  ps->pc = pc;
  ps->poff = poff;
  return GBO_OK;
}

// From how many walks on the bitmaps of the heavy block rows lose to merging
// them in pieces (bs 8, pieces / bitmaps: R-MAT 2^23 of 12, 4 walks, 15.2 / 12.5
// ms; 2^24 of 8, 8 walks, 19.9 / 22.3).
constexpr int64_t kMostWalks = 4;

// The tiles of every block row: off (nbr + 1 first tiles, owned by `mem`), the
// heavy block rows and one read of what the host needs.  Checks the rows.
struct PackCount {
  int64_t* off = nullptr;
  PackPieces pieces;  // with a table: all block rows, and none is heavy
  HeavyRows heavy;
  PackSummary sum{};
};

static int pack_count(int bs, const PackCsr& A, const int32_t* d_given, Workspace& mem, PackCount* pk, const char* who,
                      hipStream_t st) {
  int rc;
  if (heavy_walks(bs, A.ncols) > kMostWalks) {
    PieceSet ps;
    if ((rc = make_pieces(bs, A.rp, A.ci, A.nrows, A.ncols, A.nbr, mem, &ps, who, st)) ||
        (rc = mem.alloc(&pk->off, sizeof(int64_t) * ((size_t)A.nbr + 1), who)))
      return rc;
    k_piece_off<<<(unsigned)(((int64_t)A.nbr + 256) / 256), 256, 0, st>>>(ps.poff, ps.pc.base, A.nbr, pk->off);
    GBO_LAUNCH_CHECK();
    pk->pieces = ps.pc;
    pk->sum.total = ps.total;
    return d_given ? read_back(&pk->sum.given, d_given, sizeof(int32_t), st) : GBO_OK;
  }
  int32_t* cnt = nullptr;
  int* d_err = nullptr;
  PackSummary* d_sum = nullptr;
  if ((rc = mem.alloc(&cnt, sizeof(int32_t) * (size_t)std::max(A.nbr, 1), who)) ||
      (rc = mem.alloc(&pk->off, sizeof(int64_t) * ((size_t)A.nbr + 1), who)) ||
      (rc = mem.alloc(&d_err, sizeof(int), who)) || (rc = mem.alloc(&d_sum, sizeof(PackSummary), who)))
    return rc;
  GBO_HIP_CHECK(hipMemsetAsync(d_err, 0, sizeof(int), st));
  if ((rc = heavy_list(bs, A, mem, &pk->heavy, who, st))) return rc;
  PackPieces pc;
  pc.above = pk->heavy.above;
  if ((rc = dispatch_pack<PACK_COUNT>(bs, A.rp, A.ci, A.nrows, A.ncols, A.nbr, cnt, nullptr, nullptr, nullptr, nullptr,
                                      nullptr, d_err, pc, st)) ||
      (rc = heavy_count(bs, A, pk->heavy, cnt, d_err, st)) ||
      (rc = scan_exclusive<int32_t, int64_t>(cnt, pk->off, A.nbr, st, mem)))
    return rc;
  k_pack_summary<<<1, 1, 0, st>>>(pk->off + A.nbr, d_err, pk->heavy.n, d_given, d_sum);
  GBO_LAUNCH_CHECK();
  if ((rc = read_back(&pk->sum, d_sum, sizeof(PackSummary), st)) || (rc = check_err_flag(pk->sum.err, who))) return rc;
  if (pk->sum.total >= ((int64_t)1 << 31))
    return set_error(GBO_ERANGE, "tile count %lld exceeds int32", (long long)pk->sum.total);
  return GBO_OK;
}

static int pack_rowptr(const PackCount& pk, int32_t nbr, int32_t* d_rowptr, hipStream_t st) {
  k_pack_rowptr<<<(unsigned)(((int64_t)nbr + 1 + 255) / 256), 256, 0, st>>>(pk.off, nbr, d_rowptr);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// Block columns and tiles of counted rows.
static int pack_fill(int bs, int dir, const PackCsr& A, const PackCount& pk, int32_t* d_col, void* d_tiles,
                     Workspace& mem, hipStream_t st) {
  if (pk.sum.total == 0) return GBO_OK;
  PackPieces pc = pk.pieces;
  if (!pc.row) {
    pc.above = pk.heavy.above;
    pc.base = pk.off;
  }
  const int rc = dir == 0 ? dispatch_pack<PACK_ROW>(bs, A.rp, A.ci, A.nrows, A.ncols, A.nbr, nullptr, d_col, d_tiles,
                                                    nullptr, nullptr, nullptr, nullptr, pc, st)
                          : dispatch_pack<PACK_COL>(bs, A.rp, A.ci, A.nrows, A.ncols, A.nbr, nullptr, d_col, d_tiles,
                                                    nullptr, nullptr, nullptr, nullptr, pc, st);
  if (rc || pc.row) return rc;
  return heavy_fill(bs, dir, A, pk.heavy, pk.sum.heavy, pk.off, pk.sum.total, d_col, d_tiles, mem, st);
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

PlanLayout plan_layout(int bs, int64_t nchunks, int32_t nbr) {
  PlanLayout L;
  size_t off = align256(sizeof(int32_t) * (size_t)nchunks);
  L.start = off;
  off += align256(sizeof(int64_t) * ((size_t)nchunks + 1));
  L.tail = off;
  off += align256(sizeof(int32_t) * (size_t)nchunks);
  L.slots = off;
  off += align256(sizeof(unsigned long long) * kCountSlots);
  L.count = off;
  off += 256;
  L.partial = off;
  off += align256(sizeof(double) * 2 * (size_t)nchunks * bs);
  L.bfs_counts = off;
  off += align256(sizeof(int32_t) * (size_t)bs * ((size_t)nbr + 1));
  L.bytes = off;
  return L;
}

// Points the view's scratch pointers into a plan allocation made with scratch.
static void view_scratch(PlanView* pv, int bs, int32_t nbr, bool even) {
  const PlanLayout L = plan_layout(bs, pv->nchunks, nbr);
  char* base = (char*)const_cast<int32_t*>(pv->plan);
  if (!even) pv->start = (const int64_t*)(base + L.start);
  pv->tail = (const int32_t*)(base + L.tail);
  pv->slots = (unsigned long long*)(base + L.slots);
  pv->count = (int64_t*)(base + L.count);
  pv->partial = (double*)(base + L.partial);
  pv->bfs_counts = (int32_t*)(base + L.bfs_counts);
}

// *most = tiles of the longest block row (zero before).
__global__ __launch_bounds__(256) void k_row_most(const int32_t* __restrict__ rowptr, int32_t nbr,
                                                  int32_t* __restrict__ most) {
  const int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int t = R < nbr ? rowptr[R + 1] - rowptr[R] : 0;
  for (int off = 1; off < kWave; off <<= 1) t = max(t, __shfl_xor(t, off));
  if (lane_id() == 0 && t) atomicMax(most, t);
}

// Chunk starts moved back to the start of the block row they lie in.
__global__ __launch_bounds__(256) void k_whole_starts(const int32_t* __restrict__ rowptr, int32_t nbr, int32_t nchunks,
                                                      int64_t* __restrict__ start) {
  const int32_t c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= nchunks) return;
  const int64_t b = start[c];
  int32_t lo = 0, hi = nbr - 1;  // the first row that ends past b
  while (lo < hi) {
    const int32_t mid = lo + (hi - lo) / 2;
    if ((int64_t)rowptr[mid + 1] <= b) lo = mid + 1;
    else hi = mid;
  }
  start[c] = rowptr[lo];
}

static bool counts_evenly(const gbo_bsr* A) { return A->bs == 8 && A->nblocks >= kCountTiles; }

// Plan entries (of the chunks whose starts are in place, or of even chunks of
// `chunk` tiles) and zeroed count slots.
static int plan_fill(const gbo_bsr* A, int32_t chunk, bool even, bool whole, int64_t nch, int32_t* plan,
                     hipStream_t st) {
  const PlanLayout L = plan_layout(A->bs, nch, A->nblockrows);
  int64_t* start = (int64_t*)((char*)plan + L.start);
  const unsigned blocks = (unsigned)((nch + 255) / 256);
  if (whole) {
    if (even) k_even_starts<<<(unsigned)((nch + 256) / 256), 256, 0, st>>>(A->nblocks, chunk, (int32_t)nch, start);
    k_whole_starts<<<blocks, 256, 0, st>>>(A->rowptr, A->nblockrows, (int32_t)nch, start);
  }
  auto* kernel = even && !whole ? k_plan<true> : k_plan<false>;
  kernel<<<std::max<unsigned>(blocks, kCountSlots / 256), 256, 0, st>>>(
      A->rowptr, A->nblockrows, start, chunk, A->nblocks, (int32_t)nch, plan, (int32_t*)((char*)plan + L.tail),
      (unsigned long long*)((char*)plan + L.slots));
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// The chunks of about equal work: their number, and (owned by `mem`) the
// prefix sums and ranks k_unit_chunks writes their starts from.
struct WorkCut {
  int64_t *pre = nullptr, *rank = nullptr;
  int64_t nunits = 0, nch = 0, total = 0, dense = 0;
  UnitCut cut{};
};

template <int BS>
static int work_cut(const gbo_bsr* A, int32_t chunk, Workspace& mem, WorkCut* w, hipStream_t st) {
  constexpr int UT = kUnitTiles<BS>, G = BS == 8 ? 8 : BS == 16 ? 2 : 1;  // units per wave
  w->nunits = (A->nblocks + UT - 1) / UT;
  w->cut = {chunk, kTileWork<BS>, UT, BS <= 16};
  int32_t* work = nullptr;
  int rc;
  if ((rc = mem.alloc(&work, sizeof(int32_t) * (size_t)w->nunits, "gbo_bsr_plan")) ||
      (rc = mem.alloc(&w->pre, sizeof(int64_t) * ((size_t)w->nunits + 1), "gbo_bsr_plan")) ||
      (rc = mem.alloc(&w->rank, sizeof(int64_t) * ((size_t)w->nunits + UNIT_SUMS), "gbo_bsr_plan")))
    return rc;
  const unsigned blocks = (unsigned)((w->nunits + 255) / 256);
  auto* sums = (unsigned long long*)(w->rank + w->nunits);
  k_unit_work<BS><<<(unsigned)((w->nunits + 4 * G - 1) / (4 * G)), 256, 0, st>>>((const uint4*)A->tiles, A->nblocks,
                                                                                  w->nunits, work, sums);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(work, w->pre, w->nunits, st, mem))) return rc;
  k_unit_heads<<<blocks, 256, 0, st>>>(w->pre, w->nunits, w->cut, work, sums);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(work, w->rank, w->nunits, st, mem))) return rc;
  int64_t h[UNIT_SUMS];
  if ((rc = read_back(h, sums, sizeof(h), st))) return rc;
  w->nch = h[UNIT_CHUNKS];
  w->dense = h[UNIT_DENSE];
  w->total = h[UNIT_TOTAL];
  return GBO_OK;
}

// Plan for a matrix: uses A->plan (made by gbo_bsr_plan, with its scratch)
// when present, else builds a temporary one of even chunks with scratch
// (stream-ordered allocation, released by release_plan).
int acquire_plan(const gbo_bsr* A, PlanView* pv, hipStream_t st) {
  if (A->plan && A->plan_chunk > 0 && A->plan_nchunks > 0) {
    pv->plan = A->plan;
    pv->chunk = A->plan_chunk;
    pv->nchunks = A->plan_nchunks;
    pv->variant = A->plan_variant;
    pv->owned = false;
    pv->whole = A->plan_even == 2;
    pv->dense = A->plan_even == 3;
    view_scratch(pv, A->bs, A->nblockrows, A->plan_even == 1);
    if (A->plan_even == 0 && counts_evenly(A))
      pv->count_plan = (const int32_t*)((char*)A->plan + plan_layout(A->bs, A->plan_nchunks, A->nblockrows).bytes);
    return GBO_OK;
  }
  // bs 64: 128 tiles gain a sweep nothing that a plan of twice the chunks does not
  // cost (count of G(n, m) with 8.4M tiles 700 us at 256, 725 at 128)
  const int32_t chunk = A->bs == 64 && A->nblocks >= (6ll << 20) ? 256 : default_chunk(A->bs, A->nblocks, true);
  const int64_t nch = std::max<int64_t>(1, (A->nblocks + chunk - 1) / chunk);
  if (nch >= INT_MAX) return set_error(GBO_ERANGE, "too many chunks");
  const PlanLayout L = plan_layout(A->bs, nch, A->nblockrows);
  int32_t* plan = nullptr;
  GBO_HIP_CHECK(device_malloc_async((void**)&plan, L.bytes, st));
  pv->plan = plan;
  pv->chunk = chunk;
  pv->nchunks = (int32_t)nch;
  pv->variant = A->plan_variant;
  pv->owned = true;
  view_scratch(pv, A->bs, A->nblockrows, true);
  return plan_fill(A, chunk, true, false, nch, plan, st);
}

static int plan_create_with(gbo_bsr* A, int32_t chunk_tiles, int32_t variant, bool cut, hipStream_t st) {
  int32_t chunk = chunk_tiles > 0 ? chunk_tiles : default_chunk(A->bs, A->nblocks, false);
  // equal work needs the tiles' bits in 16-byte reads; the kernels that gain
  // from it need the same alignment
  bool even = !cut || chunk_tiles > 0 || A->nblocks == 0 || A->nblocks >= kEvenTiles || !A->tiles || ((uintptr_t)A->tiles & 15);
  int64_t nch = 0;
  Workspace mem(st);
  WorkCut w;
  if (!even) {
    int rc = GBO_OK;
    switch (A->bs) {
      case 8: rc = work_cut<8>(A, chunk, mem, &w, st); break;
      case 16: rc = work_cut<16>(A, chunk, mem, &w, st); break;
      case 32: rc = work_cut<32>(A, chunk, mem, &w, st); break;
      case 64: rc = work_cut<64>(A, chunk, mem, &w, st); break;
    }
    if (rc) return rc;
    // no unit has more than its tiles' work, or (bs 8/16) all have about as much
    // (G(16384, 0.2) bs 8 count 32 -> 26 us)
    even = w.total == w.nunits * w.cut.tile_work * w.cut.unit || (w.cut.mean && w.dense == 0);
    if (!even) nch = w.nch;
    else chunk = default_chunk(A->bs, A->nblocks, true);
  }
  if (even) nch = std::max<int64_t>(1, (A->nblocks + chunk - 1) / chunk);
  if (nch >= INT_MAX) return set_error(GBO_ERANGE, "gbo_bsr_plan: too many chunks");
  bool whole = false;
  const int32_t longest = whole_row(A->bs, A->nblocks, chunk);
  if (chunk_tiles <= 0 && A->nblocks > 0 && A->nblocks < kEvenTiles && A->nblocks <= (int64_t)A->nblockrows * longest) {
    int32_t most = 0, *d_most = nullptr;
    int rc = mem.alloc(&d_most, sizeof(int32_t), "gbo_bsr_plan");
    if (rc) return rc;
    GBO_HIP_CHECK(hipMemsetAsync(d_most, 0, sizeof(int32_t), st));
    k_row_most<<<(unsigned)(((int64_t)A->nblockrows + 255) / 256), 256, 0, st>>>(A->rowptr, A->nblockrows, d_most);
    GBO_LAUNCH_CHECK();
    if ((rc = read_back(&most, d_most, sizeof(int32_t), st))) return rc;
    whole = most <= longest;
  }
  gbo_bsr_plan_free(A);
  const PlanLayout L = plan_layout(A->bs, nch, A->nblockrows);
  const int64_t ncount = !even && !whole && counts_evenly(A) ? count_chunks(A->nblocks) : 0;
  if (device_malloc((void**)&A->plan, L.bytes + 2 * sizeof(int32_t) * ncount) != hipSuccess) {
    A->plan = nullptr;
    return set_error(GBO_ENOMEM, "gbo_bsr_plan: allocation of %zu bytes failed", L.bytes);
  }
  workspace_live(1);
  A->plan_chunk = chunk;
  A->plan_nchunks = (int32_t)nch;
  A->plan_variant = variant;
  // an eighth of the bits or more (blocks of 512 with 10 % of their bits at bs 32, weighted min-plus
  // 43 us, 49 where marked; of 2,048 with 20 % 278 and 156)
  const int64_t full = w.nunits * w.cut.unit * (w.cut.tile_work + A->bs * A->bs / 8 - kFreeBits);
  A->plan_even = whole ? 2 : even ? 1 : A->bs >= 32 && w.total >= full ? 3 : 0;
  if (!even) {
    k_unit_chunks<<<(unsigned)((w.nunits + 255) / 256), 256, 0, st>>>(w.pre, w.rank, w.nunits, w.cut, A->nblocks,
                                                                      (int64_t*)((char*)A->plan + L.start));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
      gbo_bsr_plan_free(A);
      return set_error(GBO_EDEVICE, "gbo_bsr_plan: %s", hipGetErrorString(e));
    }
  }
  if (ncount) {
    int32_t* count_plan = (int32_t*)((char*)A->plan + L.bytes);
    k_plan<true><<<(unsigned)((ncount + 255) / 256), 256, 0, st>>>(
        A->rowptr, A->nblockrows, nullptr, kCountChunk, A->nblocks, (int32_t)ncount, count_plan, count_plan + ncount,
        (unsigned long long*)((char*)A->plan + L.slots));
  }
  const int rc = plan_fill(A, chunk, even, whole, nch, A->plan, st);
  if (rc) gbo_bsr_plan_free(A);
  return rc;
}

int plan_create(gbo_bsr* A, int32_t chunk_tiles, int32_t variant, hipStream_t st) {
  int rc = plan_create_with(A, chunk_tiles, variant, true, st);
  // no room for the prefix sums (20 bytes a unit): even chunks need none
  if (rc == GBO_ENOMEM && chunk_tiles <= 0) rc = plan_create_with(A, chunk_tiles, variant, false, st);
  return rc;
}

int release_plan(PlanView* pv, hipStream_t st) {
  if (pv->owned && pv->plan) GBO_HIP_CHECK(hipFreeAsync(const_cast<int32_t*>(pv->plan), st));
  pv->plan = nullptr;
  pv->owned = false;
  return GBO_OK;
}

int validate_bsr(const gbo_bsr* A, int want_dir, const char* who) {
  if (!A) return set_error(GBO_EINVAL, "%s: null matrix", who);
  if (!bs_ok(A->bs)) return set_error(GBO_EUNSUPPORTED, "%s: block size %d not supported", who, A->bs);
  if (want_dir >= 0 && A->dir != want_dir)
    return set_error(GBO_EINVAL, "%s: matrix must have dir %d", who, want_dir);
  if (A->nrows < 0 || A->ncols < 0 || A->nblocks < 0)
    return set_error(GBO_EINVAL, "%s: negative size", who);
  if (A->nblockrows != (A->nrows + A->bs - 1) / A->bs || A->nblockcols != (A->ncols + A->bs - 1) / A->bs)
    return set_error(GBO_EINVAL, "%s: nblockrows/nblockcols inconsistent with nrows/ncols", who);
  if (A->nblocks >= ((int64_t)1 << 31)) return set_error(GBO_ERANGE, "%s: nblocks exceeds int32", who);
  if (!A->rowptr || (A->nblocks > 0 && (!A->colind || !A->tiles)))
    return set_error(GBO_EINVAL, "%s: null device array", who);
  return GBO_OK;
}

}  // namespace gbo

using namespace gbo;


extern "C" {

int gbo_csr2bsr_nnzb_dev(int bs, const int32_t* d_rp, const int32_t* d_ci, int32_t nrows, int32_t ncols,
                         int32_t* d_bsrRowPtr, int64_t* nblocks, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (nrows < 0 || ncols < 0 || !d_rp || !d_bsrRowPtr || !nblocks)
    return set_error(GBO_EINVAL, "gbo_csr2bsr_nnzb_dev: bad argument");
  hipStream_t st = stream;
  const int32_t nbr = (nrows + bs - 1) / bs;
  Workspace mem(st);
  PackCount pk;
  int rc = pack_count(bs, {d_rp, d_ci, nrows, ncols, nbr}, nullptr, mem, &pk, "gbo_csr2bsr_nnzb_dev", st);
  if (rc != GBO_OK || (rc = pack_rowptr(pk, nbr, d_bsrRowPtr, st))) return rc;
  GBO_HIP_CHECK(hipStreamSynchronize(st));
  *nblocks = pk.sum.total;
  return GBO_OK;
  GBO_TRY_END
}

int gbo_csr2bsr_fill_dev(int bs, int dir, const int32_t* d_rp, const int32_t* d_ci, int32_t nrows,
                         int32_t ncols, const int32_t* d_bsrRowPtr, int32_t* d_bsrColInd, void* d_tiles,
                         gbo_stream_t stream) {
  GBO_TRY_BEGIN
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (dir != 0 && dir != 1) return set_error(GBO_EINVAL, "dir must be 0 (row) or 1 (col)");
  if (nrows < 0 || ncols < 0 || !d_rp || !d_bsrRowPtr) return set_error(GBO_EINVAL, "gbo_csr2bsr_fill_dev: bad argument");
  hipStream_t st = stream;
  const int32_t nbr = (nrows + bs - 1) / bs;
  // the rows are counted and checked again: the tile offsets are that count's
  // (the same as d_bsrRowPtr at block-row starts)
  Workspace mem(st);
  const PackCsr A{d_rp, d_ci, nrows, ncols, nbr};
  PackCount pk;
  int rc = pack_count(bs, A, d_bsrRowPtr + nbr, mem, &pk, "gbo_csr2bsr_fill_dev", st);
  if (rc != GBO_OK) return rc;
  if (pk.sum.total > 0 && (!d_bsrColInd || !d_tiles)) return set_error(GBO_EINVAL, "gbo_csr2bsr_fill_dev: null output");
  if (pk.sum.given != pk.sum.total)  // the caller sized colind and tiles by rowptr[nbr]
    return set_error(GBO_EINVAL, "gbo_csr2bsr_fill_dev: rowptr[nblockrows] = %d, the CSR has %lld tiles", pk.sum.given,
                     (long long)pk.sum.total);
  rc = pack_fill(bs, dir, A, pk, d_bsrColInd, d_tiles, mem, st);
  return rc;
  GBO_TRY_END
}

int gbo_bsr_create_dev(int bs, int dir, const int32_t* d_rp, const int32_t* d_ci, int32_t nrows,
                       int32_t ncols, gbo_bsr* out, gbo_stream_t stream) {
  if (!out) return set_error(GBO_EINVAL, "gbo_bsr_create_dev: null output");
  std::memset(out, 0, sizeof(*out));
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (dir != 0 && dir != 1) return set_error(GBO_EINVAL, "dir must be 0 (row) or 1 (col)");
  if (nrows < 0 || ncols < 0 || !d_rp) return set_error(GBO_EINVAL, "gbo_bsr_create_dev: bad argument");
  const int32_t nbr = (nrows + bs - 1) / bs;
  gbo_bsr A{};
  A.bs = bs;
  A.dir = dir;
  A.nrows = nrows;
  A.ncols = ncols;
  A.nblockrows = nbr;
  A.nblockcols = (ncols + bs - 1) / bs;
  if (device_malloc((void**)&A.rowptr, sizeof(int32_t) * ((size_t)nbr + 1)) != hipSuccess)
    return set_error(GBO_ENOMEM, "gbo_bsr_create_dev: cannot allocate %d row pointers", nbr + 1);
  workspace_live(1);
  Workspace mem(stream);
  const PackCsr csr{d_rp, d_ci, nrows, ncols, nbr};
  PackCount pk;
  int rc = pack_count(bs, csr, nullptr, mem, &pk, "gbo_bsr_create_dev", stream);
  if (rc != GBO_OK || (rc = pack_rowptr(pk, nbr, A.rowptr, stream))) {
    gbo_bsr_free(&A);
    return rc;
  }
  A.nblocks = pk.sum.total;
  const size_t tile_bytes = (size_t)A.nblocks * bs * (bs / 8);
  hipError_t e1 = device_malloc((void**)&A.colind, sizeof(int32_t) * std::max<int64_t>(A.nblocks, 1));
  hipError_t e2 = device_malloc(&A.tiles, std::max<size_t>(tile_bytes, 8));
  if (e1 != hipSuccess || e2 != hipSuccess) {
    gbo_bsr_free(&A);
    return set_error(GBO_ENOMEM, "gbo_bsr_create: cannot allocate %zu tile bytes", tile_bytes);
  }
  rc = pack_fill(bs, dir, csr, pk, A.colind, A.tiles, mem, stream);
  if (rc != GBO_OK) {
    gbo_bsr_free(&A);
    return rc;
  }
  // variant 3: the fastest bs 8 count kernel on R-MAT s22 and, at bs 8/16,
  // the set-bit list min / min-plus (bs 16 count runs its variant 0)
  A.plan_variant = (bs <= 16) ? 3 : 0;
  *out = A;
  return GBO_OK;
}

// Uploads a host CSR, sorting a copy of any unsorted row first.
static int upload_csr(const int32_t* h_rp, const int32_t* h_ci, int32_t nrows, int32_t ncols,
                      int32_t** d_rp, int32_t** d_ci) {
  if (nrows < 0 || ncols < 0 || !h_rp) return set_error(GBO_EINVAL, "bad CSR");
  if (h_rp[0] != 0) return set_error(GBO_EINVAL, "rowptr[0] must be 0");
  for (int32_t r = 0; r < nrows; ++r)
    if (h_rp[r + 1] < h_rp[r]) return set_error(GBO_EINVAL, "rowptr not monotone at row %d", r);
  const int64_t nnz = h_rp[nrows];
  if (nnz > 0 && !h_ci) return set_error(GBO_EINVAL, "null colind");
  bool sorted = true;
  for (int32_t r = 0; r < nrows && sorted; ++r)
    for (int32_t k = h_rp[r] + 1; k < h_rp[r + 1]; ++k)
      if (h_ci[k] < h_ci[k - 1]) {
        sorted = false;
        break;
      }
  std::vector<int32_t> copy;
  const int32_t* src = h_ci;
  if (!sorted) {
    copy.assign(h_ci, h_ci + nnz);
    for (int32_t r = 0; r < nrows; ++r) std::sort(copy.begin() + h_rp[r], copy.begin() + h_rp[r + 1]);
    src = copy.data();
  }
  GBO_HIP_CHECK(device_malloc((void**)d_rp, sizeof(int32_t) * ((size_t)nrows + 1)));
  GBO_HIP_CHECK(device_malloc((void**)d_ci, sizeof(int32_t) * std::max<int64_t>(nnz, 1)));
  GBO_HIP_CHECK(hipMemcpy(*d_rp, h_rp, sizeof(int32_t) * ((size_t)nrows + 1), hipMemcpyHostToDevice));
  if (nnz) GBO_HIP_CHECK(hipMemcpy(*d_ci, src, sizeof(int32_t) * nnz, hipMemcpyHostToDevice));
  return GBO_OK;
}

int gbo_csr2bsr_nnzb(int bs, const int32_t* h_rp, const int32_t* h_ci, int32_t nrows, int32_t ncols,
                     int64_t* nblocks) {
  GBO_TRY_BEGIN
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (!nblocks) return set_error(GBO_EINVAL, "null nblocks");
  int32_t *d_rp = nullptr, *d_ci = nullptr, *d_brp = nullptr;
  int rc = upload_csr(h_rp, h_ci, nrows, ncols, &d_rp, &d_ci);
  const int32_t nbr = (nrows + bs - 1) / bs;
  if (rc == GBO_OK && device_malloc((void**)&d_brp, sizeof(int32_t) * ((size_t)nbr + 1)) != hipSuccess)
    rc = set_error(GBO_ENOMEM, "allocation failed");
  if (rc == GBO_OK) rc = gbo_csr2bsr_nnzb_dev(bs, d_rp, d_ci, nrows, ncols, d_brp, nblocks, nullptr);
  (void)hipFree(d_rp);
  (void)hipFree(d_ci);
  (void)hipFree(d_brp);
  return rc;
  GBO_TRY_END
}

int gbo_csr2bsr_batch(int bs, int dir, const int32_t* h_rp, const int32_t* h_ci, int32_t nrows,
                      int32_t ncols, int64_t nnz, int32_t* d_bsrRowPtr, int32_t* d_bsrColInd,
                      void* d_tiles, int32_t nblockrows, int64_t nblocks, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (!h_rp || h_rp[nrows] != nnz) return set_error(GBO_EINVAL, "gbo_csr2bsr_batch: nnz != rowptr[nrows]");
  if (nblockrows != (nrows + bs - 1) / bs) return set_error(GBO_EINVAL, "gbo_csr2bsr_batch: nblockrows != ceil(nrows/bs)");
  int32_t *d_rp = nullptr, *d_ci = nullptr;
  int rc = upload_csr(h_rp, h_ci, nrows, ncols, &d_rp, &d_ci);
  int64_t got = 0;
  if (rc == GBO_OK) rc = gbo_csr2bsr_nnzb_dev(bs, d_rp, d_ci, nrows, ncols, d_bsrRowPtr, &got, stream);
  if (rc == GBO_OK && got != nblocks)
    rc = set_error(GBO_EINVAL, "gbo_csr2bsr_batch: nblocks %lld does not match the %lld tiles of the matrix",
                   (long long)nblocks, (long long)got);
  if (rc == GBO_OK) rc = gbo_csr2bsr_fill_dev(bs, dir, d_rp, d_ci, nrows, ncols, d_bsrRowPtr, d_bsrColInd, d_tiles, stream);
  if (rc == GBO_OK) GBO_HIP_CHECK(hipStreamSynchronize(stream));
  (void)hipFree(d_rp);
  (void)hipFree(d_ci);
  return rc;
  GBO_TRY_END
}

int gbo_bsr_create(int bs, int dir, const int32_t* h_rp, const int32_t* h_ci, int32_t nrows, int32_t ncols,
                   gbo_bsr* out, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  int32_t *d_rp = nullptr, *d_ci = nullptr;
  int rc = upload_csr(h_rp, h_ci, nrows, ncols, &d_rp, &d_ci);
  if (rc == GBO_OK) rc = gbo_bsr_create_dev(bs, dir, d_rp, d_ci, nrows, ncols, out, stream);
  if (rc == GBO_OK) GBO_HIP_CHECK(hipStreamSynchronize(stream));
  (void)hipFree(d_rp);
  (void)hipFree(d_ci);
  return rc;
  GBO_TRY_END
}

void gbo_bsr_plan_free(gbo_bsr* A) {
  if (!A) return;
  if (A->plan) {
    (void)hipFree(A->plan);
    workspace_live(-1);
  }
  A->plan = nullptr;
  A->plan_chunk = 0;
  A->plan_nchunks = 0;
  A->plan_even = 0;
}

void gbo_bsr_free(gbo_bsr* A) {
  if (!A) return;
  gbo_bsr_plan_free(A);
  if (A->rowptr) {
    (void)hipFree(A->rowptr);
    workspace_live(-1);
  }
  if (A->colind) (void)hipFree(A->colind);
  if (A->tiles) (void)hipFree(A->tiles);
  A->rowptr = nullptr;
  A->colind = nullptr;
  A->tiles = nullptr;
  A->nblocks = 0;
}

int gbo_bsr_plan(gbo_bsr* A, int32_t chunk_tiles, gbo_stream_t stream) {
  return gbo_bsr_plan_ex(A, chunk_tiles, A ? A->plan_variant : 0, stream);
}

int gbo_bsr_plan_ex(gbo_bsr* A, int32_t chunk_tiles, int32_t variant, gbo_stream_t stream) {
  int rc = validate_bsr(A, -1, "gbo_bsr_plan");
  if (rc) return rc;
  if (chunk_tiles < 0) return set_error(GBO_EINVAL, "gbo_bsr_plan: negative chunk");
  if (variant < 0 || variant > 3) return set_error(GBO_EINVAL, "gbo_bsr_plan: variant must be 0, 1, 2 or 3");
  return plan_create(A, chunk_tiles, variant, stream);
}

int gbo_csr2bsr_values_u32(const gbo_bsr* A, const int32_t* d_rp, const int32_t* d_ci, const uint32_t* d_val,
                           uint32_t* d_tval, int64_t* d_woff, gbo_stream_t stream) {
  int rc = validate_bsr(A, 0, "gbo_csr2bsr_values_u32");
  if (rc) return rc;
  if (!d_rp || !d_val || !d_tval || !d_woff) return set_error(GBO_EINVAL, "gbo_csr2bsr_values_u32: null argument");
  hipStream_t st = stream;
  const int64_t T = A->nblocks;
  Workspace mem(st);
  int64_t* cnt = nullptr;
  if ((rc = mem.alloc(&cnt, sizeof(int64_t) * (size_t)std::max<int64_t>(T, 1), "gbo_csr2bsr_values_u32"))) return rc;
  if (T > 0) {
    const unsigned blocks = (unsigned)((T + 255) / 256);
    switch (A->bs) {
      case 8: k_tile_popc<8><<<blocks, 256, 0, st>>>((const uint8_t*)A->tiles, T, cnt); break;
      case 16: k_tile_popc<16><<<blocks, 256, 0, st>>>((const uint16_t*)A->tiles, T, cnt); break;
      case 32: k_tile_popc<32><<<blocks, 256, 0, st>>>((const uint32_t*)A->tiles, T, cnt); break;
      case 64: k_tile_popc<64><<<blocks, 256, 0, st>>>((const uint64_t*)A->tiles, T, cnt); break;
    }
    GBO_LAUNCH_CHECK();
  }
  if ((rc = scan_exclusive<int64_t, int64_t>(cnt, d_woff, T, st, mem))) return rc;
  PieceSet ps;
  if ((rc = make_pieces(A->bs, d_rp, d_ci, A->nrows, A->ncols, A->nblockrows, mem, &ps, "gbo_csr2bsr_values_u32", st)))
    return rc;
  if (ps.total != T) return set_error(GBO_EINVAL, "gbo_csr2bsr_values_u32: the CSR has %lld tiles, the matrix %lld",
                                      (long long)ps.total, (long long)T);
  return dispatch_pack<PACK_VALUES>(A->bs, d_rp, d_ci, A->nrows, A->ncols, A->nblockrows, A->rowptr, nullptr,
                                    nullptr, d_val, d_woff, d_tval, nullptr, ps.pc, st);
}

int gbo_pack_vec(int bs, const float* d_x, void* d_xbits, int32_t n, gbo_stream_t stream) {
  if (!bs_ok(bs)) return set_error(GBO_EUNSUPPORTED, "block size %d not supported (8, 16, 32, 64)", bs);
  if (n < 0 || (n > 0 && (!d_x || !d_xbits))) return set_error(GBO_EINVAL, "gbo_pack_vec: bad argument");
  const int32_t nw = (n + bs - 1) / bs;
  if (nw == 0) return GBO_OK;
  const unsigned blocks = (unsigned)((nw + 255) / 256);
  switch (bs) {
    case 8: k_pack_vec<8><<<blocks, 256, 0, stream>>>(d_x, (uint8_t*)d_xbits, n, nw); break;
    case 16: k_pack_vec<16><<<blocks, 256, 0, stream>>>(d_x, (uint16_t*)d_xbits, n, nw); break;
    case 32: k_pack_vec<32><<<blocks, 256, 0, stream>>>(d_x, (uint32_t*)d_xbits, n, nw); break;
    case 64: k_pack_vec<64><<<blocks, 256, 0, stream>>>(d_x, (uint64_t*)d_xbits, n, nw); break;
  }
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

}  // extern "C"
