// Bit-BSR -> CSR on the device, for solvers that run many products over one
// matrix inside one call: they list its nonzeros once and then stream 4
// bytes per nonzero instead of finding the bits of every tile again in each
// product.
//
// Two passes over the tiles.  The unit of work is an item: at most kItem
// consecutive tiles of one block row, one wavefront each, so a hub block row
// is spread over many wavefronts.  Lane l of a wave is tile row l % bs of
// tile slot l / bs (coalesced tile words).  Pass one counts each item's bits
// per tile row; the counts are laid out so that the items of one matrix row
// are adjacent and rows are in order, so one exclusive scan gives both the
// row pointer and every item's first position.  Pass two writes the columns
// of a row in ascending order (tiles in order, word from its top bit).
#include <algorithm>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {
namespace {

// Tiles per item: 512 at bs 8 to 64 at bs 64 (4 to 32 KB of tiles).
template <int BS>
constexpr int kItem = 4096 / BS;

__global__ __launch_bounds__(256) void k_item_count(const int32_t* __restrict__ rowptr, int32_t nbr, int32_t item,
                                                    int32_t* __restrict__ cnt) {
  const int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (R < nbr) cnt[R] = (int32_t)(((int64_t)rowptr[R + 1] - rowptr[R] + item - 1) / item);
}

__global__ __launch_bounds__(256) void k_item_rows(const int64_t* __restrict__ itemptr, int32_t nbr,
                                                   int32_t* __restrict__ itemrow) {
  const int64_t R = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (R >= nbr) return;
  for (int64_t k = itemptr[R]; k < itemptr[R + 1]; ++k) itemrow[k] = (int32_t)R;
}

struct ItemArgs {
  const int32_t* rowptr;
  const void* tiles;
  const int32_t* colind;
  const int32_t* perm;     // nullable: where tile t lies in `tiles`
  const int64_t* itemptr;  // [nbr + 1]
  const int32_t* itemrow;  // [items]
  int32_t nbr, n;
  int32_t* cnt;            // [items * bs], see item_slot
  const int64_t* pos;      // its exclusive scan
  int32_t* col;
};

// Where the count of tile row r of item k of block row R (m items) lies.
template <int BS>
__device__ __forceinline__ int64_t item_slot(int64_t first_item, int64_t m, int r, int64_t k) {
  return first_item * BS + r * m + k;
}

template <int BS>
__global__ __launch_bounds__(256) void k_item_bits(const ItemArgs a) {
  constexpr int G = kWave / BS;
  const int lane = lane_id(), g = lane / BS, r = lane % BS;
  const word_t<BS>* __restrict__ tiles = (const word_t<BS>*)a.tiles;
  const int64_t items = a.itemptr[a.nbr], nw = (int64_t)gridDim.x * (256 / kWave);
  for (int64_t it = wave_index(); it < items; it += nw) {
    const int32_t R = a.itemrow[it];
    const int64_t i0 = a.itemptr[R], m = a.itemptr[R + 1] - i0, k = it - i0;
    const int64_t t0 = (int64_t)a.rowptr[R] + k * kItem<BS>;
    const int64_t t1 = min(t0 + (int64_t)kItem<BS>, (int64_t)a.rowptr[R + 1]);
    int c = 0;
#pragma unroll 8
    for (int64_t t = t0 + g; t < t1; t += G) c += popcw(tiles[(a.perm ? (int64_t)a.perm[t] : t) * BS + r]);
    for (int off = BS; off < kWave; off <<= 1) c += __shfl_xor(c, off);
    if (g == 0) a.cnt[item_slot<BS>(i0, m, r, k)] = c;
  }
}

template <int BS>
__global__ __launch_bounds__(256) void k_item_rowptr(const ItemArgs a, int32_t n, int64_t* __restrict__ rowptr) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i > n) return;
  const int64_t R = i / BS;
  int64_t s = a.itemptr[a.nbr] * BS;  // past the last count: the total
  if (R < a.nbr) {
    const int64_t i0 = a.itemptr[R];
    s = item_slot<BS>(i0, a.itemptr[R + 1] - i0, (int)(i % BS), 0);
  }
  rowptr[i] = a.pos[s];
}

template <int BS>
__global__ __launch_bounds__(256) void k_item_fill(const ItemArgs a) {
  constexpr int G = kWave / BS;
  constexpr int U = 4;  // tiles per lane whose words are loaded together
  const int lane = lane_id(), g = lane / BS, r = lane % BS;
  const word_t<BS>* __restrict__ tiles = (const word_t<BS>*)a.tiles;
  const int64_t items = a.itemptr[a.nbr], nw = (int64_t)gridDim.x * (256 / kWave);
  for (int64_t it = wave_index(); it < items; it += nw) {
    const int32_t R = a.itemrow[it];
    const int64_t i0 = a.itemptr[R], m = a.itemptr[R + 1] - i0, k = it - i0;
    const int64_t t0 = (int64_t)a.rowptr[R] + k * kItem<BS>;
    const int64_t t1 = min(t0 + (int64_t)kItem<BS>, (int64_t)a.rowptr[R + 1]);
    int64_t pos = a.pos[item_slot<BS>(i0, m, r, k)];
    const bool own_row = (int64_t)R * BS + r < a.n;  // else past the total, with whatever bits the padding holds
    for (int64_t b = t0; b < t1; b += U * G) {  // wave-uniform
      uint64_t w[U];
      int32_t c[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t t = b + u * G + g;
        const int64_t tc = t < t1 ? t : t0;
        const uint64_t wv = (uint64_t)tiles[(a.perm ? (int64_t)a.perm[tc] : tc) * BS + r];
        c[u] = a.colind[tc];
        w[u] = t < t1 && own_row ? wv : 0ull;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        // bits of this row in the earlier tile slots of the step
        const int own = popcw(w[u]);
        int incl = own;
#pragma unroll
        for (int off = 1; off < G; off <<= 1) {
          const int o = __shfl_up(incl, off * BS);
          if (g >= off) incl += o;
        }
        int64_t p = pos + incl - own;
        uint64_t ww = w[u];
        while (ww) {
          const int bit = 63 - __builtin_clzll(ww);  // highest bit: lowest column
          ww &= ~(1ull << bit);
          a.col[p++] = c[u] * BS + (BS - 1 - bit);
        }
        pos += G > 1 ? __shfl(incl, kWave - BS + r) : incl;
      }
    }
  }
}

unsigned grid_of(int64_t items, int per_block) {
  return (unsigned)std::max<int64_t>(1, (items + per_block - 1) / per_block);
}
// A wave an item, past 2^24 of them several: a launch has less than 2^32
// threads, a matrix up to 2^28 block rows.
unsigned item_grid(int64_t cap) { return std::min(grid_of(cap, 4), 1u << 22); }

template <int BS>
int expand_t(const TileLists& A, Workspace& mem, CsrList* out, hipStream_t st, int64_t most) {
  const int32_t nbr = A.nbr, n = A.n;
  const int64_t cap = (int64_t)nbr + A.T / kItem<BS> + 1;  // items
  int32_t *icnt = nullptr, *itemrow = nullptr, *cnt = nullptr;
  int64_t *itemptr = nullptr, *pos = nullptr, *rowptr = nullptr;
  const char* who = "expand";
  int rc;
  if ((rc = mem.alloc(&icnt, sizeof(int32_t) * (size_t)std::max(nbr, 1), who)) ||
      (rc = mem.alloc(&itemptr, sizeof(int64_t) * ((size_t)nbr + 1), who)) ||
      (rc = mem.alloc(&itemrow, sizeof(int32_t) * (size_t)cap, who)) ||
      (rc = mem.alloc(&cnt, sizeof(int32_t) * (size_t)cap * BS, who)) ||
      (rc = mem.alloc(&pos, sizeof(int64_t) * ((size_t)cap * BS + 1), who)) ||
      (rc = mem.alloc(&rowptr, sizeof(int64_t) * ((size_t)n + 1), who)))
    return rc;
  k_item_count<<<grid_of(nbr, 256), 256, 0, st>>>(A.ptr, nbr, kItem<BS>, icnt);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int32_t, int64_t>(icnt, itemptr, nbr, st, mem))) return rc;
  k_item_rows<<<grid_of(nbr, 256), 256, 0, st>>>(itemptr, nbr, itemrow);
  ItemArgs a{};
  a.rowptr = A.ptr;
  a.tiles = A.tiles;
  a.colind = A.ind;
  a.perm = A.perm;
  a.itemptr = itemptr;
  a.itemrow = itemrow;
  a.nbr = nbr;
  a.n = n;
  a.cnt = cnt;
  a.pos = pos;
  k_item_bits<BS><<<item_grid(cap), 256, 0, st>>>(a);
  GBO_LAUNCH_CHECK();
  // counts past the last item are never written; what they hold only moves
  // positions past the total, which nothing reads
  if ((rc = scan_exclusive<int32_t, int64_t>(cnt, pos, cap * BS, st, mem))) return rc;
  k_item_rowptr<BS><<<grid_of((int64_t)n + 1, 256), 256, 0, st>>>(a, n, rowptr);
  GBO_LAUNCH_CHECK();
  int64_t nnz = 0;
  if ((rc = read_back(&nnz, rowptr + n, sizeof(int64_t), st))) return rc;
  out->rowptr = rowptr;
  out->col = nullptr;
  out->nnz = nnz;
  if (nnz > most) return GBO_OK;
  int32_t* col = nullptr;
  if ((rc = mem.alloc(&col, sizeof(int32_t) * (size_t)std::max<int64_t>(nnz, 1), who))) return rc;
  a.col = col;
  k_item_fill<BS><<<item_grid(cap), 256, 0, st>>>(a);
  GBO_LAUNCH_CHECK();
  out->col = col;
  for (const void* p : {(const void*)icnt, (const void*)itemptr, (const void*)itemrow, (const void*)cnt, (const void*)pos})
    mem.drop(p);
  return GBO_OK;
}

}  // namespace

int expand_lists(const TileLists& A, Workspace& mem, CsrList* out, hipStream_t st, int64_t most) {
  switch (A.bs) {
    case 8: return expand_t<8>(A, mem, out, st, most);
    case 16: return expand_t<16>(A, mem, out, st, most);
    case 32: return expand_t<32>(A, mem, out, st, most);
    case 64: return expand_t<64>(A, mem, out, st, most);
  }
  return set_error(GBO_EUNSUPPORTED, "block size %d not supported", A.bs);
}

int expand_csr(const gbo_bsr* A, Workspace& mem, CsrList* out, hipStream_t st, int64_t most) {
  TileLists l;
  l.bs = A->bs;
  l.nbr = A->nblockrows;
  l.n = A->nrows;
  l.T = A->nblocks;
  l.ptr = A->rowptr;
  l.ind = A->colind;
  l.tiles = A->tiles;
  return expand_lists(l, mem, out, st, most);
}

}  // namespace gbo
