// Graph algorithms on the bit-BSR engine: BFS (algorithm/bfs.cu), SSSP
// (algorithm/sssp.cu), PageRank (algorithm/pr.cu), connected components
// (algorithm/cc.cu, FastSV) and triangle counting (bsrbmm/tc.cu).
//
// The reference drivers launch five to nine kernels per iteration, fill
// vectors with single-thread <<<1,1>>> kernels inside the timed loop and
// copy a convergence scalar to the host each iteration.  Here an iteration is
// one product and one or two fused element-wise kernels (update of frontier/
// visited/levels, distances, scores or labels together with the convergence
// reduction), and the host looks at the flags of several iterations together.
#include <algorithm>
#include <cmath>
#include <mutex>
#include <type_traits>
#include <vector>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {

template <class T>
__global__ __launch_bounds__(256) void k_fill(T* __restrict__ p, int64_t n, T v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

template <class T>
static int fill(T* p, int64_t n, T v, hipStream_t st) {
  if (n <= 0) return GBO_OK;
  const int64_t blocks = std::min<int64_t>((n + 255) / 256, 65536);
  k_fill<T><<<(unsigned)blocks, 256, 0, st>>>(p, n, v);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// ------------------------------------------------------------------ BFS
template <int BS>
__global__ __launch_bounds__(256) void k_bfs_init(word_t<BS>* f, word_t<BS>* nx, word_t<BS>* vis, int32_t* level, int32_t nbr,
                                                  int32_t n, int32_t source) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < nbr) {
    const word_t<BS> w = (i == source / BS) ? (word_t<BS>)(1ull << (BS - 1 - (source % BS))) : (word_t<BS>)0;
    f[i] = w;
    nx[i] = 0;
    vis[i] = w;
  }
  if (i < n) level[i] = (i == source) ? 0 : -1;
}

// visited |= next; level[v] = lvl for each newly discovered v.
template <int BS>
__global__ __launch_bounds__(256) void k_bfs_update(const word_t<BS>* __restrict__ next, word_t<BS>* __restrict__ vis,
                                                    int32_t* __restrict__ level, int32_t nbr, int32_t n, int32_t lvl) {
  const int64_t J = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (J >= nbr) return;
  uint64_t w = (uint64_t)next[J];
  if (!w) return;
  vis[J] = (word_t<BS>)((uint64_t)vis[J] | w);
  while (w) {
    const int p = __builtin_ctzll(w);
    w &= w - 1;
    const int64_t v = J * BS + (BS - 1 - p);
    if (v < n) level[v] = lvl;
  }
}

// The same, counting the new vertices; the old frontier is cleared: the next
// step ORs the rows that chunk boundaries cut into its words.
template <int BS>
__global__ __launch_bounds__(256) void k_bfs_level(const word_t<BS>* __restrict__ next, word_t<BS>* __restrict__ f,
                                                   word_t<BS>* __restrict__ vis, int32_t* __restrict__ level,
                                                   int32_t nbr, int32_t n, int32_t lvl,
                                                   const unsigned long long* __restrict__ go,
                                                   unsigned long long* __restrict__ count) {
  __shared__ int sh[256 / kWave];
  if (over(go)) return;
  const int64_t J = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t w = 0;
  if (J < nbr) {
    w = (uint64_t)next[J];
    f[J] = (word_t<BS>)0;
  }
  int added = __popcll(w);
  if (w) {
    vis[J] = (word_t<BS>)((uint64_t)vis[J] | w);
    while (w) {
      const int p = __builtin_ctzll(w);
      w &= w - 1;
      const int64_t v = J * BS + (BS - 1 - p);
      if (v < n) level[v] = lvl;
    }
  }
  for (int off = 1; off < kWave; off <<= 1) added += __shfl_xor(added, off);
  if (lane_id() == 0) sh[threadIdx.x / kWave] = added;
  __syncthreads();
  if (threadIdx.x == 0) {
    const int all = sh[0] + sh[1] + sh[2] + sh[3];
    if (all) atomicAdd(count, (unsigned long long)all);
  }
}

// ---- push steps (direction-optimizing BFS) over A, the out-edge matrix.
// Frontier block rows are cut into segments of at most kPushSeg tiles so that
// a hub row is spread over many wavefronts.
constexpr int32_t kPushSeg = 4096;

template <int BS>
__global__ __launch_bounds__(256) void k_push_segs(const word_t<BS>* __restrict__ f, const int32_t* __restrict__ rowptr,
                                                   int32_t nbr, int32_t* __restrict__ segcnt) {
  const int64_t J = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (J > nbr) return;
  segcnt[J] = (J < nbr && f[J] != 0) ? (rowptr[J + 1] - rowptr[J] + kPushSeg - 1) / kPushSeg : 0;
}

// nx[J'] |= the unvisited out-neighbours of the frontier rows of every tile
// (J, J') of a frontier block row J; segments are taken grid-stride.
template <int BS>
__global__ __launch_bounds__(256) void k_push(const word_t<BS>* __restrict__ f, const word_t<BS>* __restrict__ vis,
                                              word_t<BS>* __restrict__ nx, const int32_t* __restrict__ rowptr,
                                              const int32_t* __restrict__ colind, const word_t<BS>* __restrict__ tiles,
                                              const int32_t* __restrict__ segoff, int32_t nbr) {
  const int lane = lane_id();
  const int64_t nw = (int64_t)gridDim.x * (blockDim.x / kWave);
  const int64_t S = segoff[nbr];
  for (int64_t sg = wave_index(); sg < S; sg += nw) {
    int32_t lo = 0, hi = nbr;  // block row: last J with segoff[J] <= sg
    while (lo < hi) {
      const int32_t mid = lo + (hi - lo + 1) / 2;
      if (segoff[mid] <= sg) lo = mid;
      else hi = mid - 1;
    }
    const int32_t J = lo;
    const int64_t t0 = (int64_t)rowptr[J] + (sg - segoff[J]) * kPushSeg;
    const int64_t t1 = min(t0 + kPushSeg, (int64_t)rowptr[J + 1]);
    const uint64_t fw = (uint64_t)f[J];
    for (int64_t t = t0 + lane; t < t1; t += kWave) {
      uint64_t nb = 0;  // out-neighbours of the frontier rows of this tile
      uint64_t rows = fw;
      while (rows) {
        const int p = __builtin_ctzll(rows);
        rows &= rows - 1;
        nb |= (uint64_t)tiles[t * BS + (BS - 1 - p)];
      }
      const int32_t J2 = colind[t];
      nb &= ~(uint64_t)vis[J2] & low_mask<BS>();
      if (nb) atomic_or_word<BS>(nx, J2, nb);
    }
  }
}

// ---- runs of levels with small frontiers in one launch.  One workgroup
// pushes level after level, its frontier (block, word, tile range) in LDS, for
// as long as the frontier stays below the limits: a level of the kernels above
// is ten launches and a host read (50 us, a mesh has hundreds of levels), one
// of these is bound by five dependent memory trips: a frontier block's tiles
// and columns, the visited words, the atomic that adds a next word, then that
// word and its visited word.  King grid 512 x 512 bs 8, 505 levels: 26 -> 3 ms.
constexpr int kRunThreads = 1024;
constexpr int kRunBlocks = 4096;   // most frontier blocks (LDS)
constexpr int kRunTiles = 12288;   // most tiles of a frontier (LDS; past it many workgroups are faster)
constexpr int kRunHeavy = 256;     // rows of more tiles are taken by the whole workgroup
constexpr int kRunLevels = 1024;   // most levels of a launch

enum { RUN_END = 0, RUN_STOP = 1, RUN_OVER = 2 };

// What a launch leaves.  RUN_END: the frontier emptied.  RUN_STOP: level
// `lvl` is complete and its frontier is in f (and, up to kRunBlocks, in
// `queue`).  RUN_OVER: nx holds the words of level lvl + 1, which is not
// entered into visited, level and f.
struct RunState {
  int32_t status, levels, lvl, qn;
  int64_t sizes[kRunLevels];  // vertices of levels lvl0 + 1, ...
};

template <int BS>
__global__ __launch_bounds__(256) void k_run_collect(const word_t<BS>* __restrict__ f, int32_t nbr,
                                                     int32_t* __restrict__ queue, RunState* __restrict__ st) {
  const int64_t J = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (J < nbr && f[J] != 0) {
    const int at = atomicAdd(&st->qn, 1);
    if (at < kRunBlocks) queue[at] = (int32_t)J;
  }
}

// What a frontier word selects in a tile: at bs 8 the bytes of its rows, so
// that a tile is one 8-byte load and a few operations; else the word.
template <int BS>
__device__ __forceinline__ uint64_t row_mask(uint64_t fw) {
  if constexpr (BS != 8) return fw;
  uint64_t m = 0;
#pragma unroll
  for (int r = 0; r < 8; ++r) m |= (fw >> (7 - r)) & 1ull ? 0xFFull << (8 * r) : 0ull;
  return m;
}

// OR of the rows of tile t that `sel` (row_mask) selects.
template <int BS>
__device__ __forceinline__ uint64_t tile_or(const word_t<BS>* __restrict__ tiles, int64_t t, uint64_t sel) {
  if constexpr (BS == 8) {
    uint64_t w = 0;
    if (((uintptr_t)tiles & 7) == 0) w = ((const uint64_t*)tiles)[t];
    else __builtin_memcpy(&w, tiles + t * 8, 8);
    w &= sel;
    uint32_t x = (uint32_t)w | (uint32_t)(w >> 32);
    x |= x >> 16;
    return (x | (x >> 8)) & 0xFFu;
  }
  uint64_t nb = 0;
  while (sel) {  // two rows' loads in flight
    const int p = __builtin_ctzll(sel);
    sel &= sel - 1;
    const int q = sel ? __builtin_ctzll(sel) : p;
    sel &= sel - 1;
    nb |= (uint64_t)tiles[t * BS + (BS - 1 - p)] | (uint64_t)tiles[t * BS + (BS - 1 - q)];
  }
  return nb;
}

// The words of `nx` and `vis` change during the launch, by this workgroup
// alone: they are read and OR-ed at workgroup scope, which stays in the L2 of
// the workgroup's die (agent scope goes to the memory side: 12.2 us a level).
template <class W>
__device__ __forceinline__ W ld_shared_word(const W* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <int BS>
__global__ __launch_bounds__(kRunThreads) void k_push_run(word_t<BS>* __restrict__ f, word_t<BS>* nx, word_t<BS>* vis,
                                                          int32_t* __restrict__ level, const int32_t* __restrict__ rowptr,
                                                          const int32_t* __restrict__ colind,
                                                          const word_t<BS>* __restrict__ tiles, int32_t n, int32_t lvl,
                                                          int64_t most_vertices, int32_t* __restrict__ queue,
                                                          RunState* __restrict__ st) {
  using W = word_t<BS>;
  using Sel = typename std::conditional<BS == 8, uint64_t, W>::type;
  constexpr int kHeavyMost = kRunTiles / kRunHeavy;
  __shared__ int32_t qj[kRunBlocks], next[kRunBlocks];  // frontier blocks; next frontier's blocks
  __shared__ W qw[kRunBlocks];                          // frontier words
  __shared__ Sel qm[BS == 8 ? kRunBlocks : 1];          // bs 8: their row masks
  __shared__ int32_t it_tile[kRunTiles];                // the frontier's tiles: tile, frontier entry
  __shared__ uint16_t it_entry[kRunTiles];
  __shared__ int32_t heavy[kHeavyMost][4];              // entry, first item, first tile, tiles
  __shared__ int32_t s_next, s_tiles, s_heavy;
  __shared__ unsigned long long s_new;
  const int tid = threadIdx.x, lane = lane_id();
  int qn = st->qn;  // at most kRunBlocks: the host sees to it
  if (tid == 0) s_next = s_tiles = s_heavy = 0, s_new = 0;
  __syncthreads();
  // Enters frontier entry e (block J, word w; `in`: the lane has one) and
  // lists its tiles.  Every lane of the wave takes part.
  auto enter = [&](bool in, int e, int32_t J, W w) {
    int32_t s = 0, d = 0;
    if (in) {
      s = rowptr[J];
      d = rowptr[J + 1] - s;
      qj[e] = J;
      qw[e] = w;
      if constexpr (BS == 8) qm[e] = row_mask<BS>(w);
    }
    const int dd = min(d, kRunTiles + 1);  // a wave's sum stays far below 2^31
    const int incl = wave_incl_scan(dd);
    int at = 0;
    if (lane == kWave - 1) at = atomicAdd(&s_tiles, min(incl, kRunTiles + 1));
    at = __builtin_amdgcn_readlane(at, kWave - 1) + incl - dd;
    if (at + dd > kRunTiles) return;  // the run ends before this frontier
    if (d <= kRunHeavy) {
      for (int k = 0; k < d; ++k) {
        it_tile[at + k] = s + k;
        it_entry[at + k] = (uint16_t)e;
      }
    } else {
      const int h = atomicAdd(&s_heavy, 1);  // below kHeavyMost: their tiles fit
      heavy[h][0] = e, heavy[h][1] = at, heavy[h][2] = s, heavy[h][3] = d;
    }
  };
  for (int e0 = 0; e0 < qn; e0 += kRunThreads) {
    const int e = e0 + tid;
    const bool in = e < qn;
    const int32_t J = in ? queue[e] : 0;
    const W w = in ? f[J] : (W)0;
    if (in) f[J] = (W)0;
    enter(in, e, J, w);
  }
  int status = RUN_STOP, done = 0;
  int64_t fsize = 0;  // not known at entry: the host has checked it
  while (true) {
    __syncthreads();
    const int ntiles = s_tiles, nheavy = s_heavy;
    if (ntiles > kRunTiles || fsize > most_vertices || done == kRunLevels) break;
    if (nheavy) {  // rows of many tiles: listed by all threads
      for (int h = 0; h < nheavy; ++h)
        for (int k = tid; k < heavy[h][3]; k += kRunThreads) {
          it_tile[heavy[h][1] + k] = heavy[h][2] + k;
          it_entry[heavy[h][1] + k] = (uint16_t)heavy[h][0];
        }
      __syncthreads();
    }
    // U tiles per thread at a time: their columns and words together, then
    // the visited words, then the atomics
    constexpr int U = 4;
    for (int i0 = tid; i0 < ntiles; i0 += U * kRunThreads) {
      int32_t J2[U];
      uint64_t nb[U];
      W v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + u * kRunThreads, ntiles - 1);
        const int32_t t = it_tile[i];
        const int e = it_entry[i];
        J2[u] = colind[t];
        uint64_t sel;
        if constexpr (BS == 8) sel = qm[e];
        else sel = qw[e];
        nb[u] = tile_or<BS>(tiles, t, i0 + u * kRunThreads < ntiles ? sel : 0ull);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = ld_shared_word(&vis[J2[u]]);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint64_t w = nb[u] & ~(uint64_t)v[u] & low_mask<BS>();
        if (w && atomic_or_word<BS, __HIP_MEMORY_SCOPE_WORKGROUP>(nx, J2[u], w) == 0) {
          const int at = atomicAdd(&s_next, 1);
          if (at < kRunBlocks) next[at] = J2[u];
        }
      }
    }
    __syncthreads();
    const int nn = s_next;
    if (nn > kRunBlocks) {
      status = RUN_OVER;
      break;
    }
    if (nn == 0) {
      status = RUN_END;
      qn = 0;
      break;
    }
    __syncthreads();
    if (tid == 0) s_next = s_tiles = s_heavy = 0, s_new = 0;
    __syncthreads();
    unsigned long long added = 0;
    for (int e0 = 0; e0 < nn; e0 += kRunThreads) {
      const int e = e0 + tid;
      const bool in = e < nn;
      const int32_t J = next[in ? e : 0];
      const W w = in ? ld_shared_word(&nx[J]) : (W)0;
      const W v = in ? ld_shared_word(&vis[J]) : (W)0;
      enter(in, e, J, w);
      if (!in) continue;
      nx[J] = (W)0;
      vis[J] = (W)(v | w);
      added += popcw(w);
      uint64_t m = (uint64_t)w;
      while (m) {
        const int p = __builtin_ctzll(m);
        m &= m - 1;
        const int64_t i = (int64_t)J * BS + (BS - 1 - p);
        if (i < n) level[i] = lvl + 1;
      }
    }
    // one LDS add per wave: 1024 threads adding to one word take turns
    for (int off = 1; off < kWave; off <<= 1) added += __shfl_xor(added, off);
    if (lane == 0 && added) atomicAdd(&s_new, added);
    __syncthreads();
    fsize = (int64_t)s_new;
    if (tid == 0) st->sizes[done] = fsize;
    qn = nn;
    ++lvl;
    ++done;
  }
  // the frontier goes back to memory (RUN_OVER: its next one is in nx)
  if (status == RUN_STOP) {
    for (int e = tid; e < qn; e += kRunThreads) {
      f[qj[e]] = qw[e];
      queue[e] = qj[e];
    }
  }
  if (tid == 0) {
    st->status = status;
    st->levels = done;
    st->lvl = lvl;
    st->qn = qn;
  }
}

// Set bits of the next-frontier words, summed per wave into the count slots
// (folded by count_fold): one counter for every wave took 85 us on a pushed
// level of 163K vertices (R-MAT s22), 8K waves queueing on one address.
template <int BS>
__global__ __launch_bounds__(256) void k_popc_words(const word_t<BS>* __restrict__ w, int32_t nbr,
                                                    unsigned long long* __restrict__ slots) {
  const int64_t J = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  uint64_t c = J < nbr ? (uint64_t)popcw(w[J]) : 0ull;
  for (int off = 1; off < kWave; off <<= 1) c += __shfl_xor(c, off);
  if (lane_id() == 0 && c) atomicAdd(&slots[(J / kWave) & (kCountSlots - 1)], (unsigned long long)c);
}

// Scratch of a BFS call supplied by the caller of bfs_t instead of being
// allocated: frontier / next / visited words (3 x nbr words), the levels' flags
// (kBfsFlagBytes) and (bs 8, where dense_bfs_step holds and they fit) the dense
// step's row counts (bs x (nbr + 1) int32, else null).
constexpr size_t kBfsFlagBytes = 8192;
struct BfsScratch {
  void* words;
  void* flags;
  int32_t* dense_counts;
};

static SpmvArgs bfs_args(const gbo_bsr* A, const PlanView& pv) {
  SpmvArgs a{};
  a.rowptr = A->rowptr;
  a.colind = A->colind;
  a.tiles = A->tiles;
  a.nrows = A->nrows;
  a.ncols = A->ncols;
  a.nbr = A->nblockrows;
  a.T = A->nblocks;
  a.plan = pv.plan;
  a.start = pv.start;
  a.tail = pv.tail;
  a.whole = pv.whole;
  a.dense = pv.dense;
  a.count_plan = pv.count_plan;
  a.chunk = pv.chunk;
  a.nchunks = pv.nchunks;
  a.variant = pv.variant;
  return a;
}

// From how many tiles on bs 8 takes the dense step: its kernels have no look at
// the flags, so its levels are not queued.  Queued, dense: 1.6M tiles (200,000
// vertices of 8) 216 and 269 us, 1.1M (R-MAT 2^16) 247 and 241, 5.2M (R-MAT
// 2^18) 490 and 447, 24M 1045 and 958.  At bs 16 to 64 k_bfs_scan leaves block
// rows early and is the better one at every size (R-MAT 2^22, dense where a
// quarter of the frontier words may have bits: bs 16 2.68 against 3.02 ms, bs 32
// 3.25 against 4.19).
constexpr int64_t kDenseTiles = 2 << 20;

// Pull BFS over AT, several levels between two looks at their sizes: one level
// of a king grid of 65,536 takes 11 us instead of 26 (bs 16 6.5 -> 2.7 ms).
// The dense step's row counts come from the plan's scratch; the frontier, next
// and visited words and the sizes are this call's -- or, with `ext`, all of them
// come from there.
template <int BS>
static int bfs_t(const gbo_bsr* A, int32_t source, int32_t* d_level, int64_t* sizes, int32_t max_levels,
                 int32_t* nlevels, hipStream_t st, const BfsScratch* ext = nullptr) {
  using W = word_t<BS>;
  const int32_t nbr = A->nblockrows, n = A->nrows;
  Workspace mem(st);
  W* f = nullptr;
  Rounds rounds;
  int rc;
  if (ext) {
    f = (W*)ext->words;
    rounds.place(ext->flags, kBfsFlagBytes);
  } else if ((rc = mem.alloc(&f, sizeof(W) * (size_t)std::max(nbr, 1) * 3 + 64, "gbo_bfs")) ||
             (rc = rounds.alloc(mem, "gbo_bfs"))) {
    return rc;
  }
  W* nx = f + std::max(nbr, 1);
  W* vis = nx + std::max(nbr, 1);
  PlanGuard g(st);
  if ((rc = acquire_plan(A, &g.pv, st))) return rc;
  const unsigned blocks_n = (unsigned)((std::max<int64_t>(n, nbr) + 255) / 256);
  k_bfs_init<BS><<<blocks_n, 256, 0, st>>>(f, nx, vis, d_level, nbr, n, source);
  GBO_LAUNCH_CHECK();
  SpmvArgs a = bfs_args(A, g.pv);
  a.prefilled = 1;
  // bs 8 variant 3, large matrices: levels while fewer than half the vertices
  // are visited take the dense step (count kernel + pack); later ones skip
  // visited rows
  int32_t* dense_counts = BS != 8 || !dense_bfs_step(BS, g.pv.variant) ? nullptr
                          : ext                                        ? ext->dense_counts
                                                                       : g.pv.bfs_counts;
  int64_t visited = 1;
  int32_t lvl = 0;
  if (sizes && max_levels > 0) sizes[0] = 1;
  for (bool more = true; more;) {
    int nb = 0;
    if ((rc = rounds.batch(lvl, &nb, st))) return rc;
    const bool dense = dense_counts && A->nblocks >= kDenseTiles && visited < (int64_t)n / 2;
    if (dense || (BS == 8 && g.pv.variant != 1 && g.pv.variant != 3)) nb = 1;
    for (int k = 0; k < nb; ++k) {
      a.xbits = f;
      a.visited = vis;
      a.out = nx;
      a.bfs_counts = dense ? dense_counts : nullptr;
      a.go = rounds.go(k);
      if ((rc = spmv_launch(BS, OP_BFS, a, st))) return rc;
      k_bfs_level<BS><<<(unsigned)((nbr + 255) / 256), 256, 0, st>>>(nx, f, vis, d_level, nbr, n, lvl + k + 1, a.go,
                                                                     rounds.again(k));
      GBO_LAUNCH_CHECK();
      std::swap(f, nx);
    }
    int ran = 0;
    if ((rc = rounds.look(nb, &ran, &more, st))) return rc;
    for (int k = 0; k < ran && rounds.h[k].again; ++k) {
      ++lvl;
      visited += (int64_t)rounds.h[k].again;
      if (sizes && lvl < max_levels) sizes[lvl] = (int64_t)rounds.h[k].again;
    }
  }
  if (nlevels) *nlevels = lvl + 1;
  return GBO_OK;
}

// Direction-optimizing BFS: levels whose frontier holds at most n/64 vertices
// are pushed over A (the out-edge matrix, AT itself for an undirected graph),
// the others pulled over AT.  The frontier-size slots and the dense step's row
// counts come from the plan's scratch.
template <int BS>
static int bfs_do_t(const gbo_bsr* A, const gbo_bsr* Aout, int32_t source, int32_t* d_level, int64_t* sizes,
                    int32_t max_levels, int32_t* nlevels, hipStream_t st) {
  using W = word_t<BS>;
  const int32_t nbr = A->nblockrows, n = A->nrows;
  Workspace mem(st);
  W* f = nullptr;
  int rc;
  if ((rc = mem.alloc(&f, sizeof(W) * (size_t)std::max(nbr, 1) * 3 + 64, "gbo_bfs_do"))) return rc;
  W* nx = f + std::max(nbr, 1);
  W* vis = nx + std::max(nbr, 1);
  int32_t *segoff = nullptr, *queue = nullptr;
  RunState* run = nullptr;
  if (((rc = mem.alloc(&segoff, sizeof(int32_t) * ((size_t)nbr + 1), "gbo_bfs_do")) ||
               (rc = mem.alloc(&queue, sizeof(int32_t) * kRunBlocks, "gbo_bfs_do")) ||
               (rc = mem.alloc(&run, sizeof(RunState), "gbo_bfs_do"))))
    return rc;
  PlanGuard g(st);
  if ((rc = acquire_plan(A, &g.pv, st))) return rc;
  const PlanView& pv = g.pv;
  int64_t* d_cnt = pv.count;
  const unsigned blocks_n = (unsigned)((std::max<int64_t>(n, nbr) + 255) / 256);
  k_bfs_init<BS><<<blocks_n, 256, 0, st>>>(f, nx, vis, d_level, nbr, n, source);
  GBO_LAUNCH_CHECK();
  SpmvArgs a = bfs_args(A, pv);
  a.count_slots = pv.slots;
  // bs 8 variant 3: levels while fewer than half the vertices are visited take
  // the dense step (count kernel + pack); later ones skip visited rows
  int32_t* dense_counts = BS == 8 && dense_bfs_step(BS, pv.variant) ? pv.bfs_counts : nullptr;
  int64_t visited = 1;
  int32_t lvl = 0;
  int64_t fsize = 1;  // vertices in the current frontier
  if (sizes && max_levels > 0) sizes[0] = 1;
  bool over = false;  // a run of levels left the next one in nx
  // Frontiers a run is tried on.  One that a run stopped at has too many tiles,
  // and so have the next ones as a rule: the run is tried again an eighth below
  // it.  (Tried at each of the wide levels, 200 on a king grid 1000 x 1000 from
  // its middle at bs 8: 22.3 ms, now 16.4; 2000 x 2000 55.7 and 47.)
  int64_t run_most = std::min<int64_t>(std::max<int64_t>(n / 64, 1), kRunBlocks);
  while (true) {
    if (fsize <= run_most) {
      // a run of small levels in one launch
      GBO_HIP_CHECK(hipMemsetAsync(nx, 0, sizeof(W) * (size_t)std::max(nbr, 1), st));
      GBO_HIP_CHECK(hipMemsetAsync(run, 0, offsetof(RunState, sizes), st));
      k_run_collect<BS><<<(unsigned)((nbr + 255) / 256), 256, 0, st>>>(f, nbr, queue, run);
      RunState h;
      do {
        k_push_run<BS><<<1, kRunThreads, 0, st>>>(f, nx, vis, d_level, Aout->rowptr, Aout->colind,
                                                  (const W*)Aout->tiles, n, lvl, std::max<int64_t>(n / 64, 1), queue, run);
        GBO_LAUNCH_CHECK();
        if ((rc = read_back(&h, run, sizeof(h), st))) return rc;
        for (int k = 0; k < h.levels; ++k) {
          ++lvl;
          fsize = h.sizes[k];
          visited += fsize;
          if (sizes && lvl < max_levels) sizes[lvl] = fsize;
        }
      } while (h.status == RUN_STOP && h.levels == kRunLevels);
      if (h.status == RUN_END) break;
      over = h.status == RUN_OVER;
      if (!over) run_most = std::min(run_most, fsize - fsize / 8 - 1);
    }
    // every step form ends with count_fold, which writes d_cnt
    if (over) {
      over = false;
      k_popc_words<BS><<<(unsigned)((nbr + 255) / 256), 256, 0, st>>>(nx, nbr, pv.slots);
      GBO_LAUNCH_CHECK();
      if ((rc = count_fold(pv.slots, d_cnt, st))) return rc;
    } else if (fsize <= std::max<int64_t>(n / 64, 1)) {
      // push: only the frontier rows' tiles of A are read
      GBO_HIP_CHECK(hipMemsetAsync(nx, 0, sizeof(W) * (size_t)std::max(nbr, 1), st));
      k_push_segs<BS><<<(unsigned)(((int64_t)nbr + 1 + 255) / 256), 256, 0, st>>>(f, Aout->rowptr, nbr, segoff);
      GBO_LAUNCH_CHECK();
      if ((rc = scan_exclusive<int32_t, int32_t>(segoff, segoff, (int64_t)nbr + 1, st, mem))) return rc;
      k_push<BS><<<2048, 256, 0, st>>>(f, vis, nx, Aout->rowptr, Aout->colind, (const W*)Aout->tiles, segoff, nbr);
      GBO_LAUNCH_CHECK();
      k_popc_words<BS><<<(unsigned)((nbr + 255) / 256), 256, 0, st>>>(nx, nbr, pv.slots);
      GBO_LAUNCH_CHECK();
      if ((rc = count_fold(pv.slots, d_cnt, st))) return rc;
    } else {
      a.xbits = f;
      a.visited = vis;
      a.out = nx;
      a.bfs_counts = (dense_counts && visited < (int64_t)n / 2) ? dense_counts : nullptr;
      if ((rc = spmv_launch(BS, OP_BFS, a, st))) return rc;
      if ((rc = count_fold(pv.slots, d_cnt, st))) return rc;
    }
    // the level update needs no count (an empty next frontier changes
    // nothing), so it is queued before the host waits for the count
    k_bfs_update<BS><<<(unsigned)((nbr + 255) / 256), 256, 0, st>>>(nx, vis, d_level, nbr, n, lvl + 1);
    GBO_LAUNCH_CHECK();
    int64_t cnt = 0;
    if ((rc = read_back(&cnt, d_cnt, sizeof(int64_t), st))) return rc;
    if (cnt == 0) break;
    ++lvl;
    fsize = cnt;
    visited += cnt;
    if (sizes && lvl < max_levels) sizes[lvl] = cnt;
    std::swap(f, nx);
  }
  if (nlevels) *nlevels = lvl + 1;
  return GBO_OK;
}

// ------------------------------------------------------------------ SSSP
// dist = min(dist, cand); the improved vertices form the next frontier: their
// distance goes to `fr` (INF elsewhere) and their block column is marked
// active so the next min-plus product only reads tiles of active columns.
constexpr int kSsspThreads = 512;  // vertices of whole bytes of `active` at every block size
__global__ __launch_bounds__(kSsspThreads) void k_sssp_update(uint32_t* __restrict__ cand,
                                                              uint32_t* __restrict__ dist, uint32_t* __restrict__ fr,
                                                              unsigned char* __restrict__ active, int32_t n, int bs,
                                                              const unsigned long long* __restrict__ go,
                                                              unsigned long long* __restrict__ changed) {
  __shared__ int sh[kSsspThreads / kWave];
  if (over(go)) return;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int improved = 0;
  if (i < n) {
    const uint32_t c = cand[i], d = dist[i];
    cand[i] = kInfU32;  // where the next product's split rows start from
    if (c < d) {
      dist[i] = c;
      fr[i] = c;
      improved = 1;
    } else {
      fr[i] = kInfU32;
    }
  }
  // block columns of the improved vertices: 64 / bs bits of each wave
  const int lane = lane_id(), per = kWave / bs;
  const unsigned long long m = __ballot(improved);
  if (lane == 0) {
    int bits = 0;
    for (int k = 0; k < per; ++k) bits |= (m >> (k * bs) & (~0ull >> (kWave - bs))) ? 1 << k : 0;
    sh[threadIdx.x / kWave] = bits;
  }
  __syncthreads();
  if ((int)threadIdx.x < per) {  // 512 / bs bits: `per` bytes
    int byte = 0;
    for (int k = 0; k < 8 / per; ++k) byte |= sh[threadIdx.x * (8 / per) + k] << (k * per);
    active[(int64_t)blockIdx.x * per + threadIdx.x] = (unsigned char)byte;
  }
  wave_flag(improved, changed);
}

__global__ void k_sssp_init(uint32_t* dist, uint32_t* fr, uint32_t* cand, unsigned long long* active, int32_t n, int bs, int32_t s) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    dist[i] = (i == s) ? 0u : kInfU32;
    fr[i] = (i == s) ? 0u : kInfU32;
    cand[i] = kInfU32;
  }
  if (i == 0) {
    const int64_t J = s / bs;
    active[J >> 6] = 1ull << (J & 63);
  }
}

// ------------------------------------------------------------------ PageRank
// x[j] = alpha * p[j] / outdeg[j] (0 for vertices without out-edges) -- the
// per-edge factor alpha*f1/nnz of bmv32_sparse_full (algorithm/bsrbmv.cu:
// 1276) computed once per vertex.
__global__ __launch_bounds__(256) void k_pr_scale(const float* __restrict__ p, const int32_t* __restrict__ outdeg,
                                                  float alpha, float* __restrict__ x, int32_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    const int32_t d = outdeg[i];
    x[i] = d > 0 ? alpha * p[i] / (float)d : 0.0f;
  }
}

// Per-block partial sums of |q-p| in double, and the next iteration's
// x[j] = alpha * q[j] / outdeg[j] (as k_pr_scale) from the same read of q.
// The partials are added in a fixed order by k_sum_partials, so the L1
// change is reproducible.  Up to kOneBlock vertices one block takes them all and
// writes the sum and the flag itself: a launch costs the host 5 us.
constexpr int kOneBlock = 1 << 14;
template <int THREADS>
__global__ __launch_bounds__(THREADS) void k_pr_tail(const float* __restrict__ q, const float* __restrict__ p,
                                                     const int32_t* __restrict__ outdeg, float alpha,
                                                     float* __restrict__ x, int32_t n, double tol,
                                                     double* __restrict__ part,
                                                     const unsigned long long* __restrict__ go,
                                                     unsigned long long* __restrict__ again) {
  __shared__ double sh[THREADS];
  if (over(go)) return;
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const float qi = q[i];
    s += fabs((double)qi - (double)p[i]);
    const int32_t d = outdeg[i];
    x[i] = d > 0 ? alpha * qi / (float)d : 0.0f;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = THREADS / 2; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    part[blockIdx.x] = sh[0];
    if (gridDim.x == 1) *again = sh[0] < tol ? 0 : 1;
  }
}

// *out = the sum of part[0..np) in a fixed order: thread t adds entries
// t, t+256, ... in turn, then a fixed tree over the threads (one block of
// 256 threads); *again = 0 where it is below tol.
__global__ __launch_bounds__(256) void k_sum_partials(const double* __restrict__ part, int np, double tol, double* out,
                                                      const unsigned long long* __restrict__ go,
                                                      unsigned long long* __restrict__ again) {
  __shared__ double sh[256];
  if (over(go)) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) s += part[i];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int off = 128; off > 0; off >>= 1) {
    if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *out = sh[0];
    *again = sh[0] < tol ? 0 : 1;
  }
}

// ------------------------------------------------------------------ CC
// FastSV hooking (Zhang, Azad, Hu; the GraphBLAST algorithm the reference
// follows, algorithm/cc.cu:1018-1083): stochastic hooking f[f[u]] = min(.,
// mngf[u]), aggressive hooking f[u] = min(f[u], mngf[u]) and shortcutting
// f[u] = min(f[u], gf[u]), all as min-accumulating atomics.  Labels only
// decrease, so an atomic whose candidate is not below a value read before it
// would change nothing and is not issued: millions of vertices share a few
// roots, and their atomics on the root's label serialised (0.26 ms a call
// at R-MAT s22).
__global__ __launch_bounds__(256) void k_cc_hook(int32_t* __restrict__ mngf, const int32_t* __restrict__ gf,
                                                 int32_t* __restrict__ f, int32_t n,
                                                 const unsigned long long* __restrict__ go) {
  if (over(go)) return;
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (u >= n) return;
  const int32_t m = mngf[u];
  mngf[u] = INT32_MAX;  // where the next product's split rows start from
  const int32_t fu = f[u];
  if (m < fu && m < f[fu]) atomicMin(&f[fu], m);
  const int32_t g = gf[u];
  const int32_t best = m < g ? m : g;
  if (best < fu) atomicMin(&f[u], best);
}

// gf[u] = f[f[u]]; *changed = 1 if any vertex's grandparent changed.
__global__ __launch_bounds__(256) void k_cc_grand(const int32_t* __restrict__ f, int32_t* __restrict__ gf, int32_t n,
                                                  const unsigned long long* __restrict__ go,
                                                  unsigned long long* __restrict__ changed) {
  if (over(go)) return;
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int ch = 0;
  if (u < n) {
    const int32_t g = f[f[u]];
    if (g != gf[u]) {
      gf[u] = g;
      ch = 1;
    }
  }
  wave_flag(ch, changed);
}

// f[u] = f[f[u]] until every vertex points at a root (final star shape).
__global__ __launch_bounds__(256) void k_cc_jump(int32_t* __restrict__ f, int32_t n, const unsigned long long* go,
                                                 unsigned long long* changed) {
  if (over(go)) return;
  const int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int ch = 0;
  if (u < n) {
    const int32_t p = f[u], gp = f[p];
    if (gp != p) {
      f[u] = gp;
      ch = 1;
    }
  }
  wave_flag(ch, changed);
}

__global__ void k_cc_init(int32_t* a, int32_t* b, int32_t* m, int32_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    a[i] = (int32_t)i;
    b[i] = (int32_t)i;
    m[i] = INT32_MAX;
  }
}

// One product of a driver, over the edge lists where it has them.
static int sweep(int bs, int op, const SpmvArgs& a, const ListView& lists, hipStream_t st) {
  if (!lists.on) return spmv_launch(bs, op, a, st);
  return lists_sweep(op, lists, {a.xval, a.out, a.w, a.woff, a.scale, a.bias, a.go}, st);
}

static int check_square(const gbo_bsr* A, const char* who) {
  int rc = validate_bsr(A, 0, who);
  if (rc) return rc;
  if (A->nrows != A->ncols) return set_error(GBO_EINVAL, "%s: matrix must be square", who);
  return GBO_OK;
}

// ------------------------------------------------- allocation-free BFS
// gbo_bfs_noalloc's scratch: one fixed array in device memory, held by
// every GPU the library runs on until the process ends.  Host code never
// passes `scratch` itself (in host code that name is only a stand-in); it
// uses the device address hipGetSymbolAddress returns, looked up once per
// device on the first call with that device current.
constexpr size_t kNoAllocScratchBytes = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

static std::mutex g_scratch_mu;
static void* g_scratch_ptr[64];  // device address of `scratch`, per device

static int noalloc_scratch(unsigned char** out) {
  int dev = 0;
  GBO_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) return set_error(GBO_EDEVICE, "gbo_bfs_noalloc: device %d out of range", dev);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return set_error(GBO_EDEVICE, "gbo_bfs_noalloc: hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *out = (unsigned char*)g_scratch_ptr[dev];
  return GBO_OK;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Carves the BFS scratch for AT out of the static array; GBO_ERANGE when it
// does not fit.
static int noalloc_layout(const gbo_bsr* AT, unsigned char* base, BfsScratch* s) {
  const size_t wbytes = (size_t)(AT->bs / 8) * (size_t)std::max(AT->nblockrows, 1) * 3 + 64;
  const size_t o_words = kBfsFlagBytes + 256;
  const size_t o_dense = o_words + align256(wbytes);
  // the dense step's row counts (4 bytes a vertex) when they fit as well;
  // without them every level takes the step that skips visited rows (same
  // levels)
  const size_t dbytes = sizeof(int32_t) * (size_t)AT->bs * ((size_t)AT->nblockrows + 1);
  const bool dense =
      AT->bs == 8 && dense_bfs_step(AT->bs, AT->plan_variant) && o_dense + align256(dbytes) <= kNoAllocScratchBytes;
  const size_t need = o_dense + (dense ? align256(dbytes) : 0);
  if (need > kNoAllocScratchBytes)
    return set_error(GBO_ERANGE,
                     "gbo_bfs_noalloc: %d vertices at bs %d need %zu bytes of scratch, the static array holds %zu",
                     AT->nrows, AT->bs, need, kNoAllocScratchBytes);
  s->flags = base;
  s->words = base + o_words;
  s->dense_counts = dense ? (int32_t*)(base + o_dense) : nullptr;
  return GBO_OK;
}

}  // namespace gbo

using namespace gbo;

extern "C" {

int gbo_bfs(const gbo_bsr* AT, int32_t source, int32_t* d_level, int64_t* h_level_sizes, int32_t max_levels,
            int32_t* h_nlevels, gbo_stream_t stream) {
  int rc = check_square(AT, "gbo_bfs");
  if (rc) return rc;
  if (source < 0 || source >= AT->nrows) return set_error(GBO_EINVAL, "gbo_bfs: source %d out of range", source);
  if (!d_level) return set_error(GBO_EINVAL, "gbo_bfs: null level");
  switch (AT->bs) {
    case 8: return bfs_t<8>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 16: return bfs_t<16>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 32: return bfs_t<32>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 64: return bfs_t<64>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
  }
  return set_error(GBO_EUNSUPPORTED, "gbo_bfs: block size");
}

int gbo_bfs_noalloc(const gbo_bsr* AT, int32_t source, int32_t* d_level, int64_t* h_level_sizes,
                    int32_t max_levels, int32_t* h_nlevels, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  int rc = check_square(AT, "gbo_bfs_noalloc");
  if (rc) return rc;
  if (source < 0 || source >= AT->nrows)
    return set_error(GBO_EINVAL, "gbo_bfs_noalloc: source %d out of range", source);
  if (!d_level) return set_error(GBO_EINVAL, "gbo_bfs_noalloc: null level");
  if (!AT->plan || AT->plan_chunk <= 0 || AT->plan_nchunks <= 0)
    return set_error(GBO_EINVAL, "gbo_bfs_noalloc: the matrix has no plan (make one with gbo_bsr_plan first)");
  unsigned char* base = nullptr;
  if ((rc = noalloc_scratch(&base))) return rc;
  BfsScratch s{};
  if ((rc = noalloc_layout(AT, base, &s))) return rc;
  switch (AT->bs) {
    case 8: return bfs_t<8>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream, &s);
    case 16: return bfs_t<16>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream, &s);
    case 32: return bfs_t<32>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream, &s);
    case 64: return bfs_t<64>(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream, &s);
  }
  return set_error(GBO_EUNSUPPORTED, "gbo_bfs_noalloc: block size");
  GBO_TRY_END
}

int gbo_bfs_do(const gbo_bsr* AT, const gbo_bsr* A, int32_t source, int32_t* d_level, int64_t* h_level_sizes,
               int32_t max_levels, int32_t* h_nlevels, gbo_stream_t stream) {
  int rc = check_square(AT, "gbo_bfs_do");
  if (rc) return rc;
  if (A) {
    rc = check_square(A, "gbo_bfs_do(A)");
    if (rc) return rc;
    if (A->bs != AT->bs || A->nrows != AT->nrows) return set_error(GBO_EINVAL, "gbo_bfs_do: A and AT differ in shape");
  }
  if (source < 0 || source >= AT->nrows) return set_error(GBO_EINVAL, "gbo_bfs_do: source %d out of range", source);
  if (!d_level) return set_error(GBO_EINVAL, "gbo_bfs_do: null level");
  if (!A) return gbo_bfs(AT, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
  switch (AT->bs) {
    case 8: return bfs_do_t<8>(AT, A, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 16: return bfs_do_t<16>(AT, A, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 32: return bfs_do_t<32>(AT, A, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
    case 64: return bfs_do_t<64>(AT, A, source, d_level, h_level_sizes, max_levels, h_nlevels, stream);
  }
  return set_error(GBO_EUNSUPPORTED, "gbo_bfs_do: block size");
}

int gbo_sssp(const gbo_bsr* AT, const uint32_t* d_w, const int64_t* d_woff, int32_t source, uint32_t* d_dist,
             int32_t* h_iters, gbo_stream_t stream) {
  int rc = check_square(AT, "gbo_sssp");
  if (rc) return rc;
  const int32_t n = AT->nrows;
  if (source < 0 || source >= n) return set_error(GBO_EINVAL, "gbo_sssp: source %d out of range", source);
  if (!d_dist) return set_error(GBO_EINVAL, "gbo_sssp: null dist");
  if ((d_w == nullptr) != (d_woff == nullptr)) return set_error(GBO_EINVAL, "gbo_sssp: weights need offsets");
  hipStream_t st = stream;
  const int bs = AT->bs;
  const int64_t nact = ((int64_t)AT->nblockcols + 63) / 64;
  Workspace mem(st);
  uint32_t* fr = nullptr;
  unsigned long long* active = nullptr;
  if ((rc = mem.alloc(&fr, sizeof(uint32_t) * (size_t)std::max(n, 1) * 2, "gbo_sssp"))) return rc;
  if ((rc = mem.alloc(&active, sizeof(unsigned long long) * (size_t)nact * 2, "gbo_sssp"))) return rc;
  Rounds rounds;
  if ((rc = rounds.alloc(mem, "gbo_sssp"))) return rc;
  uint32_t* cand = fr + std::max(n, 1);
  unsigned long long* active2 = active + nact;
  PlanGuard g(st);
  if ((rc = acquire_plan(AT, &g.pv, st))) return rc;
  const PlanView& pv = g.pv;
  GBO_HIP_CHECK(hipMemsetAsync(active, 0, sizeof(unsigned long long) * nact * 2, st));
  const unsigned blocks_n = (unsigned)((n + 255) / 256);
  k_sssp_init<<<blocks_n, 256, 0, st>>>(d_dist, fr, cand, active, n, bs, source);
  GBO_LAUNCH_CHECK();
  SpmvArgs a{};
  a.rowptr = AT->rowptr;
  a.colind = AT->colind;
  a.tiles = AT->tiles;
  a.nrows = n;
  a.ncols = AT->ncols;
  a.nbr = AT->nblockrows;
  a.T = AT->nblocks;
  a.plan = pv.plan;
  a.start = pv.start;
  a.tail = pv.tail;
  a.whole = pv.whole;
  a.dense = pv.dense;
  a.count_plan = pv.count_plan;
  a.chunk = pv.chunk;
  a.nchunks = pv.nchunks;
  a.variant = pv.variant;
  a.w = d_w;
  a.woff = d_woff;
  ListView lists;
  lists_build(AT, ListUse::kPaths, mem, &lists, st);
  int32_t it = 0;
  unsigned long long *act_cur = active, *act_next = active2;
  const unsigned blocks_u = (unsigned)(((int64_t)n + kSsspThreads - 1) / kSsspThreads);
  a.prefilled = 1;
  for (bool more = true; more;) {
    int nb = 0;
    if ((rc = rounds.batch(it, &nb, st))) return rc;
    for (int k = 0; k < nb; ++k) {
      a.xval = fr;
      a.out = cand;
      a.active = (const uint64_t*)act_cur;
      a.go = rounds.go(k);
      if ((rc = sweep(bs, OP_MINPLUS, a, lists, st))) return rc;
      k_sssp_update<<<blocks_u, kSsspThreads, 0, st>>>(cand, d_dist, fr, (unsigned char*)act_next, n, bs, a.go,
                                                       rounds.again(k));
      GBO_LAUNCH_CHECK();
      std::swap(act_cur, act_next);
    }
    int ran = 0;
    if ((rc = rounds.look(nb, &ran, &more, st))) return rc;
    it += ran;
    if (more && it > n + 1)  // distances only decrease: cannot happen
      return set_error(GBO_ENOCONV, "gbo_sssp: no convergence after %d iterations", it);
  }
  if (h_iters) *h_iters = it;
  return GBO_OK;
}

int gbo_pagerank(const gbo_bsr* AT, const int32_t* d_outdeg, float alpha, double tol, int32_t max_iter, float* d_p,
                 int32_t* h_iters, double* h_last_delta, gbo_stream_t stream) {
  int rc = check_square(AT, "gbo_pagerank");
  if (rc) return rc;
  const int32_t n = AT->nrows;
  if (!d_outdeg || !d_p) return set_error(GBO_EINVAL, "gbo_pagerank: null argument");
  if (!(alpha >= 0.0f && alpha < 1.0f) || max_iter < 1) return set_error(GBO_EINVAL, "gbo_pagerank: bad alpha/max_iter");
  if (n == 0) return GBO_OK;
  hipStream_t st = stream;
  const int nparts = 1024;
  Workspace mem(st);
  float* x = nullptr;
  double* dpart = nullptr;
  if ((rc = mem.alloc(&x, sizeof(float) * (size_t)n * 2, "gbo_pagerank"))) return rc;
  if ((rc = mem.alloc(&dpart, sizeof(double) * nparts, "gbo_pagerank"))) return rc;
  Rounds rounds;
  if ((rc = rounds.alloc(mem, "gbo_pagerank"))) return rc;
  float* y = x + n;
  PlanGuard g(st);
  if ((rc = acquire_plan(AT, &g.pv, st))) return rc;
  const PlanView& pv = g.pv;
  if ((rc = fill<float>(d_p, n, 1.0f / (float)n, st))) return rc;
  SpmvArgs a{};
  a.rowptr = AT->rowptr;
  a.colind = AT->colind;
  a.tiles = AT->tiles;
  a.nrows = n;
  a.ncols = AT->ncols;
  a.nbr = AT->nblockrows;
  a.T = AT->nblocks;
  a.plan = pv.plan;
  a.start = pv.start;
  a.tail = pv.tail;
  a.whole = pv.whole;
  a.dense = pv.dense;
  a.count_plan = pv.count_plan;
  a.chunk = pv.chunk;
  a.nchunks = pv.nchunks;
  a.variant = pv.variant;
  a.partial = pv.partial;  // split-row partials from the plan's scratch
  a.scale = 1.0f;
  a.bias = (1.0f - alpha) / (float)n;
  const unsigned blocks_n = (unsigned)((n + 255) / 256);
  const unsigned lblocks = (unsigned)std::min<int64_t>(nparts, (n + 255) / 256);
  ListView lists;
  lists_build(AT, ListUse::kMany, mem, &lists, st);
  int32_t it = 0;
  double delta = 0.0;
  k_pr_scale<<<blocks_n, 256, 0, st>>>(d_p, d_outdeg, alpha, x, n);
  GBO_LAUNCH_CHECK();
  for (bool more = true; more && it < max_iter;) {
    int nb = 0;
    if ((rc = rounds.batch(it, &nb, st))) return rc;
    nb = std::min(nb, max_iter - it);
    for (int k = 0; k < nb; ++k) {
      // iterate it + k is in d_p where that is even, else in y
      const float* from = (it + k) % 2 ? y : d_p;
      float* to = (it + k) % 2 ? d_p : y;
      a.xval = x;
      a.out = to;
      a.go = rounds.go(k);
      if ((rc = sweep(AT->bs, OP_SUM, a, lists, st))) return rc;
      // x for the next iteration, the change of this one
      if (n <= kOneBlock) {
        k_pr_tail<1024><<<1, 1024, 0, st>>>(to, from, d_outdeg, alpha, x, n, tol, rounds.value(k), a.go, rounds.again(k));
      } else {
        k_pr_tail<256><<<lblocks, 256, 0, st>>>(to, from, d_outdeg, alpha, x, n, tol, dpart, a.go, nullptr);
        k_sum_partials<<<1, 256, 0, st>>>(dpart, (int)lblocks, tol, rounds.value(k), a.go, rounds.again(k));
      }
      GBO_LAUNCH_CHECK();
    }
    int ran = 0;
    if ((rc = rounds.look(nb, &ran, &more, st))) return rc;
    it += ran;
    delta = rounds.h[ran - 1].value;
  }
  const float* p = it % 2 ? y : d_p;
  if (p != d_p) {
    GBO_HIP_CHECK(hipMemcpyAsync(d_p, p, sizeof(float) * n, hipMemcpyDeviceToDevice, st));
    GBO_HIP_CHECK(hipStreamSynchronize(st));
  }
  if (h_iters) *h_iters = it;
  if (h_last_delta) *h_last_delta = delta;
  if (!(delta < tol))
    return set_error(GBO_ENOCONV, "gbo_pagerank: not converged after %d iterations (delta %.3e)", it, delta);
  return GBO_OK;
}

int gbo_cc(const gbo_bsr* A, int32_t* d_label, int32_t* h_iters, gbo_stream_t stream) {
  int rc = check_square(A, "gbo_cc");
  if (rc) return rc;
  const int32_t n = A->nrows;
  if (!d_label) return set_error(GBO_EINVAL, "gbo_cc: null label");
  if (n == 0) return GBO_OK;
  hipStream_t st = stream;
  Workspace mem(st);
  int32_t* gf = nullptr;
  Rounds rounds;
  if ((rc = mem.alloc(&gf, sizeof(int32_t) * (size_t)n * 2, "gbo_cc"))) return rc;
  if ((rc = rounds.alloc(mem, "gbo_cc"))) return rc;
  int32_t* mngf = gf + n;
  int32_t* f = d_label;
  const unsigned blocks_n = (unsigned)((n + 255) / 256);
  k_cc_init<<<blocks_n, 256, 0, st>>>(f, gf, mngf, n);
  GBO_LAUNCH_CHECK();
  PlanGuard g(st);
  if ((rc = acquire_plan(A, &g.pv, st))) return rc;
  const PlanView& pv = g.pv;
  SpmvArgs a{};
  a.rowptr = A->rowptr;
  a.colind = A->colind;
  a.tiles = A->tiles;
  a.nrows = n;
  a.ncols = A->ncols;
  a.nbr = A->nblockrows;
  a.T = A->nblocks;
  a.plan = pv.plan;
  a.start = pv.start;
  a.tail = pv.tail;
  a.whole = pv.whole;
  a.dense = pv.dense;
  a.count_plan = pv.count_plan;
  a.chunk = pv.chunk;
  a.nchunks = pv.nchunks;
  a.variant = pv.variant;
  ListView lists;
  lists_build(A, ListUse::kFew, mem, &lists, st);
  int32_t it = 0;
  a.prefilled = 1;
  for (bool more = true; more;) {
    int nb = 0;
    if ((rc = rounds.batch(it, &nb, st))) return rc;
    for (int k = 0; k < nb; ++k) {
      a.xval = gf;
      a.out = mngf;
      a.go = rounds.go(k);
      if ((rc = sweep(A->bs, OP_MIN, a, lists, st))) return rc;
      k_cc_hook<<<blocks_n, 256, 0, st>>>(mngf, gf, f, n, a.go);
      k_cc_grand<<<blocks_n, 256, 0, st>>>(f, gf, n, a.go, rounds.again(k));
      GBO_LAUNCH_CHECK();
    }
    int ran = 0;
    if ((rc = rounds.look(nb, &ran, &more, st))) return rc;
    it += ran;
    if (more && it > n + 2) return set_error(GBO_ENOCONV, "gbo_cc: no convergence");
  }
  for (bool more = true; more;) {  // make every tree a star
    int nb = 0;
    if ((rc = rounds.batch(0, &nb, st))) return rc;
    for (int k = 0; k < nb; ++k) k_cc_jump<<<blocks_n, 256, 0, st>>>(f, n, rounds.go(k), rounds.again(k));
    GBO_LAUNCH_CHECK();
    int ran = 0;
    if ((rc = rounds.look(nb, &ran, &more, st))) return rc;
  }
  if (h_iters) *h_iters = it;
  return GBO_OK;
}

int gbo_tc(int bs, int32_t nrows, const int32_t* h_rp, const int32_t* h_ci, uint64_t* h_count, gbo_stream_t stream) {
  GBO_TRY_BEGIN
  if (!h_rp || !h_count || nrows < 0) return set_error(GBO_EINVAL, "gbo_tc: bad argument");
  int64_t lnnz = 0;
  int32_t *lp = nullptr, *li = nullptr, *tp = nullptr, *ti = nullptr;
  int rc = gbo_csr_tril(nrows, h_rp, h_ci, 1, &lnnz, &lp, &li);
  if (rc) return rc;
  rc = gbo_csr_transpose(nrows, nrows, lp, li, &tp, &ti);
  gbo_bsr L{}, LT{};
  if (rc == GBO_OK) rc = gbo_bsr_create(bs, 0, lp, li, nrows, nrows, &L, stream);
  if (rc == GBO_OK) rc = gbo_bsr_create(bs, 1, tp, ti, nrows, nrows, &LT, stream);
  gbo_free_host(lp);
  gbo_free_host(li);
  gbo_free_host(tp);
  gbo_free_host(ti);
  uint64_t* d = nullptr;
  if (rc == GBO_OK && device_malloc((void**)&d, sizeof(uint64_t)) != hipSuccess) rc = set_error(GBO_ENOMEM, "gbo_tc: alloc");
  if (rc == GBO_OK) rc = gbo_bsrbmm_tc(&L, &LT, d, stream);
  if (rc == GBO_OK && hipMemcpy(h_count, d, sizeof(uint64_t), hipMemcpyDeviceToHost) != hipSuccess)
    rc = set_error(GBO_EDEVICE, "gbo_tc: copy");
  (void)hipFree(d);
  gbo_bsr_free(&L);
  gbo_bsr_free(&LT);
  return rc;
  GBO_TRY_END
}

}  // extern "C"
