// Shared declarations between the packer, the bsrbmv/bsrbmm operations and
// the drivers (device-side translation units).
#pragma once
#include <algorithm>

#include <hip/hip_runtime.h>

#include "gbo_device.hpp"

namespace gbo {

// Work decomposition of a bit-BSR: the tiles [0, nblocks) are cut into
// nchunks chunks of consecutive tiles, chunk c being [start[c], start[c+1]);
// plan[c] is the first block row that chunk c touches (a row that begins
// before the chunk is "split" and its partial results are combined across
// chunks).  A chunk size given by the caller cuts evenly, chunk c starting at
// tile c * chunk; the library's own plan (plan_create) makes chunks of about
// equal work, at most `chunk` tiles, or moves their starts back to the start of a
// block row where these are short (at most `chunk` and the longest row's tiles).
//
// The scratch the operations need besides their inputs and outputs is kept
// in the plan's allocation, after the nchunks plan entries, so that a call
// on a planned matrix allocates nothing (each part 256-byte aligned):
//   start       nchunks+1 x i64     first tile of each chunk
//   tail        nchunks x i32       chunks after c that go on with a row begun in c
//   slots       kCountSlots x u64   BFS frontier-size slots (zero between calls)
//   count       1 x int64           the folded frontier size
//   partial     nchunks*2*bs x f64  split-row partials of the FP32 sum
//   bfs_counts  bs*(nbr+1) x int32  per-row counts of the dense BFS step
// Calls on one matrix therefore share that scratch: they must be ordered
// (one stream, or synchronised); separately created matrices do not share.
struct PlanLayout {
  size_t start = 0, tail = 0, slots = 0, count = 0, partial = 0, bfs_counts = 0, bytes = 0;
};
// The count at bs 8 takes even chunks of kCountChunk tiles, on plans of equal
// work from kCountTiles tiles on: their plan entries, then their tails, lie after
// the rest.
// All its tiles cost the same, and a look at the chunk's start before the first
// tile is asked for costs more than equal work gains: R-MAT 2^19 of 16 (11M tiles) 107
// -> 93 us, 2^20 of 12 143 -> 132, 2^21 of 8 208 -> 188 (2^18 of 28 67 -> 74); below,
// 2^18 of 16 (5M tiles) 63 and 71.
constexpr int64_t kCountTiles = 6 << 20;
constexpr int32_t kCountChunk = 256;
inline int64_t count_chunks(int64_t tiles) { return (tiles + kCountChunk - 1) / kCountChunk; }
PlanLayout plan_layout(int bs, int64_t nchunks, int32_t nbr);

struct PlanView {
  const int32_t* plan = nullptr;
  const int64_t* start = nullptr;  // null: even chunks of `chunk` tiles
  const int32_t* tail = nullptr;
  int32_t chunk = 0;
  int32_t nchunks = 0;
  int32_t variant = 0;
  bool owned = false;
  unsigned long long* slots = nullptr;
  int64_t* count = nullptr;
  double* partial = nullptr;
  int32_t* bfs_counts = nullptr;  // the dense BFS step's row counts
  const int32_t* count_plan = nullptr;  // even chunks of the count, where they are others; count_chunks tails behind
  bool whole = false;             // no block row is cut
  bool dense = false;             // an eighth of the tiles' bits are set, or more (equal work, bs 32/64)
};

// Most tiles per chunk of the library's own plans.
int default_chunk(int bs, int64_t tiles, bool uniform);
int acquire_plan(const gbo_bsr* A, PlanView* pv, hipStream_t st);
int release_plan(PlanView* pv, hipStream_t st);
// Allocates A->plan with its scratch (chunk tiles per chunk, 0 = the library's
// own plan, which reads the tiles once and synchronizes the stream).
int plan_create(gbo_bsr* A, int32_t chunk_tiles, int32_t variant, hipStream_t st);

// A plan acquired for the length of one call, released on every return path.
struct PlanGuard {
  PlanView pv;
  hipStream_t st;
  explicit PlanGuard(hipStream_t s) : st(s) {}
  ~PlanGuard() { (void)release_plan(&pv, st); }
  PlanGuard(const PlanGuard&) = delete;
  PlanGuard& operator=(const PlanGuard&) = delete;
};

// Scratch kept between calls at most, per device.
constexpr size_t kKeepBytes = (size_t)8 << 30;

// Device scratch of one call that waits for its stream before it returns:
// blocks kept between calls (gbo_workspace.hip), given back on every return
// path once the stream has been waited for.  What drop() is given is handed out
// again to the same call, in the order of its stream: a loop of any length
// holds the blocks of one turn.
class Workspace {
 public:
  explicit Workspace(hipStream_t st) : st_(st) {}
  ~Workspace();
  Workspace(const Workspace&) = delete;
  Workspace& operator=(const Workspace&) = delete;
  template <class T>
  int alloc(T** p, size_t bytes, const char* who) {
    void* q = nullptr;
    const int rc = take(&q, bytes, who);
    *p = (T*)q;
    return rc;
  }
  void drop(const void* p);

 private:
  int take(void** p, size_t bytes, const char* who);
  bool free_dropped();
  static constexpr int kMax = 64;
  hipStream_t st_;
  int dev_ = -1;
  void* ptrs_[kMax];
  size_t bytes_[kMax];
  bool spare_[kMax];  // dropped
  int n_ = 0;
};
// hipMalloc and hipMallocAsync that give the kept blocks back before they report
// that memory is out (every allocation of the library is one of them); gives all
// kept blocks of a device (-1: of each) back; counts the matrices and plans the
// library has allocated.
hipError_t device_malloc(void** p, size_t bytes);
hipError_t device_malloc_async(void** p, size_t bytes, hipStream_t st);
void workspace_release(int dev);
void workspace_live(int delta);
// Copies a few bytes to the host and waits for the stream.
int read_back(void* h, const void* d, size_t bytes, hipStream_t st);

// Stream-ordered device allocations of a call that does not wait for its
// stream, released with hipFreeAsync on every return path (success or error).
class AsyncAllocs {
 public:
  explicit AsyncAllocs(hipStream_t st) : st_(st) {}
  ~AsyncAllocs() {
    for (int i = 0; i < n_; ++i) (void)hipFreeAsync(ptrs_[i], st_);
  }
  AsyncAllocs(const AsyncAllocs&) = delete;
  AsyncAllocs& operator=(const AsyncAllocs&) = delete;
  template <class T>
  int alloc(T** p, size_t bytes, const char* who) {
    *p = nullptr;
    if (n_ == kMax) return set_error(GBO_EINVAL, "%s: too many scratch allocations", who);
    void* q = nullptr;
    const hipError_t e = device_malloc_async(&q, bytes ? bytes : 8, st_);
    if (e != hipSuccess) return set_error(GBO_ENOMEM, "%s: device allocation of %zu bytes failed: %s", who, bytes,
                                          hipGetErrorString(e));
    ptrs_[n_++] = q;
    *p = (T*)q;
    return GBO_OK;
  }

 private:
  static constexpr int kMax = 24;
  hipStream_t st_;
  void* ptrs_[kMax] = {};
  int n_ = 0;
};
int validate_bsr(const gbo_bsr* A, int want_dir, const char* who);

// The nonzeros of a row-direction bit-BSR as CSR (rows in order, columns
// ascending), in device memory owned by `mem`; one host read of the total.  More
// than `most` are counted only.
struct CsrList {
  const int64_t* rowptr = nullptr;  // [nrows + 1]
  const int32_t* col = nullptr;     // [nnz]; null past `most`
  int64_t nnz = 0;
};
int expand_csr(const gbo_bsr* A, Workspace& mem, CsrList* out, hipStream_t st, int64_t most = INT64_MAX);
// The same for any block lists: list R (of nbr) holds the blocks ind[t], t in
// [ptr[R], ptr[R+1]); word k of tile t (or perm[t]) holds list R * bs + k's
// bits in block ind[t], top bit first.
struct TileLists {
  int32_t bs = 0, nbr = 0, n = 0;  // n: lists of words (at most nbr * bs)
  int64_t T = 0;
  const int32_t *ptr = nullptr, *ind = nullptr;
  const void* tiles = nullptr;
  const int32_t* perm = nullptr;
};
int expand_lists(const TileLists& A, Workspace& mem, CsrList* out, hipStream_t st, int64_t most = INT64_MAX);

template <class TI, class TO>
int scan_exclusive(const TI* in, TO* out, int64_t n, hipStream_t st);
// The same with its block sums in a Workspace.
template <class TI, class TO>
int scan_exclusive(const TI* in, TO* out, int64_t n, hipStream_t st, Workspace& mem);

// Packing of the heavy block rows (gbo_pack_fill.hip), those of more than
// `above` nonzeros: heavy_list finds them, heavy_count writes their tile counts
// and raises PACKERR flags, heavy_fill writes their block columns and tiles
// (from off, the first tile of each block row), for rows that raised none.
// heavy_walks: how often each reads a block row, by the matrix's width.
enum { PACKERR_COLRANGE = 1, PACKERR_UNSORTED = 2 };
struct PackCsr {
  const int32_t *rp, *ci;
  int32_t nrows, ncols, nbr;
};
struct HeavyRows {
  int32_t* list = nullptr;
  int32_t* n = nullptr;  // device
  int32_t above = 0;
};
int64_t heavy_walks(int bs, int32_t ncols);
int heavy_list(int bs, const PackCsr& A, Workspace& mem, HeavyRows* h, const char* who, hipStream_t st);
int heavy_count(int bs, const PackCsr& A, const HeavyRows& h, int32_t* cnt, int* err, hipStream_t st);
int heavy_fill(int bs, int dir, const PackCsr& A, const HeavyRows& h, int32_t nheavy, const int64_t* off, int64_t T,
               int32_t* colind, void* tiles, Workspace& mem, hipStream_t st);

constexpr uint32_t kInfU32 = 0xFFFFFFFFu;

// The flags of the iterations queued between two looks at them: iteration k
// runs only if flag k - 1 of its batch is set, and sets flag k if another is to
// follow.  A look costs about 12 us with the stream's gap; an iteration past the
// end a few launches that do nothing, so that batches grow with the iterations
// there have been: by half of them.
struct Rounds {
  static constexpr int kMax = 32, kFlags = 1024;
  struct Flag {
    unsigned long long again;
    double value;
  };
  Flag* flags = nullptr;
  int cap = kFlags;
  int at = kFlags;  // first flag of the batch
  Flag h[kMax];

  int alloc(Workspace& mem, const char* who) { return mem.alloc(&flags, sizeof(Flag) * kFlags, who); }
  void place(void* p, size_t bytes) {
    flags = (Flag*)p;
    cap = at = (int)std::min<size_t>(bytes / sizeof(Flag), kFlags);
  }
  // iterations to queue after `done`; their flags are clear
  int batch(int done, int* n, hipStream_t st) {
    *n = done == 0 ? 3 : std::min(std::max(2, done / 2), kMax);
    if (at + *n > cap) {
      GBO_HIP_CHECK(hipMemsetAsync(flags, 0, sizeof(Flag) * cap, st));
      at = 0;
    }
    return GBO_OK;
  }
  const unsigned long long* go(int k) const { return k ? &flags[at + k - 1].again : nullptr; }
  unsigned long long* again(int k) const { return &flags[at + k].again; }
  double* value(int k) const { return &flags[at + k].value; }
  // iterations of the batch of n that ran; *more: the last of them asks for another
  int look(int n, int* ran, bool* more, hipStream_t st) {
    const int rc = read_back(h, flags + at, sizeof(Flag) * n, st);
    if (rc) return rc;
    at += n;
    *ran = 1;
    while (*ran < n && h[*ran - 1].again) ++*ran;
    *more = h[*ran - 1].again != 0;
    return GBO_OK;
  }
};

// Edge lists for drivers that sweep one matrix many times (gbo_lists.hip).
// lists_build leaves `on` false where sweeps over the tiles are to be used:
// few tiles, mostly dense ones, more than 2^26 rows, no memory.
struct ListPart {
  const uint32_t* at;  // entries
  int32_t n;
  int32_t win;   // window of 64 rows
  int32_t tile;  // first tile of its item
  int32_t skip;  // entries of the item before it
};
struct ListView {
  bool on = false;
  int bs;
  int32_t n, nbr, nwin, per, nmulti;
  int64_t nparts;
  const int32_t *rowptr, *colind;
  const void* tiles;
  const int64_t* first;   // building: items, then parts before each window
  const int32_t* win;     // window of each item
  const int32_t* multi;   // windows of several parts
  const ListPart* parts;
  double* partial;
};
constexpr int kListSlots = 64;
struct ListInfo {
  int64_t items, parts, over;
  unsigned long long sample[kListSlots];
  int32_t multi, overs;
};
struct ListSweep {
  const void* x;
  void* out;
  const uint32_t* w;
  const int64_t* woff;
  float scale, bias;  // sum: scale * (A x) + bias
  const unsigned long long* go;
};
struct ListMs {
  const uint64_t *F, *V;
  uint64_t* Fn;  // zero on entry
  const uint64_t *active, *live;
  const unsigned long long* go;
};
enum class ListUse { kMany, kPaths, kFew, kFrontiers };  // sweeps of a call: PageRank's, shortest paths', a few; multi-source BFS
void lists_build(const gbo_bsr* A, ListUse use, Workspace& mem, ListView* out, hipStream_t st);
// OP_SUM, OP_MIN, or OP_MINPLUS without the vertex's own value.
int lists_sweep(int op, const ListView& l, const ListSweep& s, hipStream_t st);
// Next frontiers: the unvisited (of the live sources) in-neighbours' words.
int lists_ms(int kw, const ListView& l, const ListMs& s, hipStream_t st);

constexpr int kCountSlots = 1024;

// bsrbmv operation codes.
enum SpmvOp { OP_COUNT = 0, OP_BFS = 1, OP_MINPLUS = 2, OP_SUM = 3, OP_MIN = 4 };

// Whether a BFS step at this block size and plan variant may take the dense
// form (count kernel into per-row counts, then a pack of the nonzero rows):
// bs 8/16 under variant 3, bs 32/64 under every variant.
inline bool dense_bfs_step(int bs, int variant) { return (bs <= 16 && variant == 3) || bs >= 32; }

struct SpmvArgs {
  const int32_t* rowptr;
  const int32_t* colind;
  const void* tiles;
  int32_t nrows, ncols, nbr;
  int64_t T;
  const int32_t* plan;
  const int64_t* start;  // first tile of each chunk, nchunks + 1 entries (null: even chunks of `chunk` tiles)
  const int32_t* tail;   // chunks that go on with a row begun in chunk c (0: no row is cut there)
  int32_t chunk, nchunks;
  int32_t variant;      // bs 8/16 COUNT/BFS kernel variant
  const void* xbits;    // COUNT: x bits; BFS: frontier bits
  const void* visited;  // BFS: visited bits (per block row)
  void* out;            // COUNT int32 y / BFS next bits / MINPLUS uint32 / SUM float / MIN int32
  const uint32_t* w;    // MINPLUS weights in tile bit order (nullable)
  const int64_t* woff;  // MINPLUS per-tile weight offsets
  const void* xval;     // MINPLUS dist / SUM x / MIN x
  unsigned long long* count_slots;  // BFS: newly set bits, summed per slot (kCountSlots, zero on entry; nullable)
  int32_t* bfs_counts;  // BFS where dense_bfs_step holds (nullable): int32 scratch of nbr*bs; when set the step runs
                        // the count kernel into it and packs the rows with a nonzero count (dense step)
  double* partial;      // SUM: split-row partials [nchunks][2][bs]
  const uint64_t* active;  // MINPLUS: optional per-block-column activity bits (nullable)
  int accumulate;       // COUNT: add into y
  float scale, bias;    // SUM: y = scale * (A x) + bias  (scale 1, bias 0 for the plain op)
  const unsigned long long* go;  // MINPLUS / SUM / MIN (kernels of their own: the look costs a plain product 0.2 us a
                                 // launch), BFS by columns (bs 16 to 64) and by a tile a lane (bs 8): nothing is
                                 // done where *go is 0 (nullable)
  int whole;            // no block row is cut by a chunk's end
  int dense;            // see PlanView
  const int32_t* count_plan;  // see PlanView (nullable)
  int prefilled;        // BFS / MINPLUS / MIN: `out` holds the identity where rows are split
};

// The iteration before this one was the last: a driver queues a few iterations
// between two looks at their flags, and those past the end do nothing.
__device__ __forceinline__ bool over(const unsigned long long* go) { return go && *go == 0; }

// First tile of chunk c, for c up to nchunks.  The even form is kept apart
// because it needs no load before the chunk's tiles can be asked for.
template <class Args>
__device__ __forceinline__ int64_t chunk_start(const Args& a, int64_t c) {
  return a.start ? a.start[c] : min(c * a.chunk, a.T);
}

int spmv_launch(int bs, int op, const SpmvArgs& a, hipStream_t st);

// BFS frontier-size counters.  Every wave adds its count of newly set bits
// to slot (chunk index mod kCountSlots) instead of one shared counter, so
// hundreds of thousands of waves do not serialise on a single address;
// count_fold() sums the slots into one int64 and clears them again.  The
// slots live in the plan's scratch (zeroed when the plan is made).
int count_fold(unsigned long long* slots, int64_t* d_count, hipStream_t st);

}  // namespace gbo
