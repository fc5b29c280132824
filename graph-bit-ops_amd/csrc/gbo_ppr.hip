// Personalized PageRank over K vectors with a hand-written adjoint.
// No reference counterpart: it generalises the PageRank of algorithm/pr.cu
// (p' = alpha * P^T p + (1-alpha)/n, P = D^-1 A) to K personalization
// vectors s_k and adds the reverse-mode solve.
//
//   forward:  p_k = alpha * P^T p_k + (1 - alpha) * s_k      (pull over A^T)
//   adjoint:  lambda_k = alpha * P lambda_k + w_k            (pull over A)
//   dL/ds_k = (1 - alpha) * lambda_k,
//   dL/dalpha = sum_k lambda_k . (P^T p_k - s_k)
// for L = sum_k w_k . p_k.  The adjoint needs only the converged p (no
// checkpointing of the forward iterates).
//
// Both solves run some tens of products over one matrix, so a call lists the
// nonzeros of its tiles once as CSR (expand_csr) and every product streams 4
// bytes per nonzero and gathers one row of X per nonzero.  Walking the tiles
// in each product instead (a wave per 1024 tiles, its set bits listed in LDS
// or taken one at a time) left most of the chip idle on matrices of a few
// million nonzeros and one wave at work on the densest tiles.
//
// The product (k_spmm): the rows are cut into segments of at most 64
// nonzeros (longer for hub rows), a unit of 16 lanes takes a segment.  X is
// kept with its rows padded to a multiple of four columns, so a lane gathers
// 16 bytes: at K > 32 the 16 lanes span a row of X and the unit takes one
// nonzero at a time, eight gathers in flight; at smaller K the unit takes 2
// to 16 nonzeros at a time.  Sums are FP64.  A segment that is its whole row
// finishes it in place: Y, the next product's scaled row, and its part of
// the convergence measure.  Rows of several segments leave FP64 partials
// that k_spmm_fix adds in a fixed order, so results are bitwise reproducible
// and independent of the block size and of the operands' alignment.
//
// The solves decide on convergence on the device (k_colsum): each kernel
// returns at once when the flag is up, and the host queues kBatch iterations
// between two looks at it.
#include <algorithm>
#include <cmath>
#include <vector>

#include "gbo_device.hpp"
#include "gbo_ops.hpp"

namespace gbo {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kUnit = 16;        // lanes per segment
constexpr int kBlk = 256;        // threads per workgroup
constexpr int kUnits = kBlk / kUnit;
constexpr int kMainBlocks = 2048;  // most workgroups of k_spmm (fixed, so that the order of the measure is too)
constexpr int kFixBlocks = 2048;   // and of k_spmm_fix
// Iterations queued between two host reads of the flag: a read costs about
// 30 us of idle GPU, an iteration after convergence three empty launches
// (about 9 us), and a solve takes 30 to 120 iterations.
constexpr int kBatch = 8;

// Nonzeros per segment of a row of `deg`: 64 keeps the units of a wave close
// to equal; hub rows take longer ones so that at most some hundred partials
// of a row are added one after another.
__host__ __device__ inline int64_t seg_len(int64_t deg) { return deg <= 4096 ? 64 : deg <= 65536 ? 256 : 1024; }

// A segment: row, start | length << 48 | (its row has several) << 63, and
// then the slot of its partial.
struct alignas(16) Seg {
  uint64_t sl;
  int32_t row;
  uint32_t slot;
};

__device__ __forceinline__ int64_t row_segs(int64_t deg) {
  const int64_t L = seg_len(deg);
  return deg <= L ? 1 : (deg + L - 1) / L;  // an empty row has one empty segment
}

// Per row: segments in the low half, partial slots (rows of several segments
// only) in the high half; and whether it has several.
__global__ __launch_bounds__(256) void k_seg_count(const int64_t* __restrict__ rowptr, int32_t n,
                                                   int64_t* __restrict__ cnt, int32_t* __restrict__ multi) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t s = row_segs(rowptr[i + 1] - rowptr[i]);
  cnt[i] = s | (s > 1 ? s << 32 : 0);
  multi[i] = s > 1;
}

__global__ __launch_bounds__(256) void k_seg_fill(const int64_t* __restrict__ rowptr, int32_t n,
                                                  const int64_t* __restrict__ off, const int64_t* __restrict__ moff,
                                                  Seg* __restrict__ segs, int32_t* __restrict__ mrow) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const int64_t r0 = rowptr[i], deg = rowptr[i + 1] - r0;
  const int64_t s = row_segs(deg), L = seg_len(deg);
  const int64_t at = off[i] & 0xFFFFFFFF;
  const uint32_t slot = (uint32_t)(off[i] >> 32);
  for (int64_t k = 0; k < s; ++k) {
    Seg g;
    g.sl = (uint64_t)(r0 + k * L) | ((uint64_t)min(L, deg - k * L) << 48) | (s > 1 ? 1ull << 63 : 0ull);
    g.row = (int32_t)i;
    g.slot = slot + (uint32_t)k;
    segs[at + k] = g;
  }
  if (s > 1) mrow[moff[i]] = (int32_t)i;
}

// Device-side state of a solve.
struct Ctl {
  unsigned long long done;  // 1: converged, later kernels return
  unsigned long long iters;
  unsigned long long ticket;
  double dmax;
  double val[64];   // the last column sums
  double norm[64];  // the columns' norms
};

struct SpmmArgs {
  const Seg* segs;
  int64_t nseg;
  const int32_t* mrow;   // rows of several segments
  int64_t nmulti;
  const int64_t* off;    // per row, as k_seg_count's scan
  const int32_t* col;
  int32_t K, ld;         // columns; row stride of the padded arrays (a multiple of 4)
  const float* X;        // [n][ld], already carrying any per-source scale
  const float* rowscale; // per output row factor (nullable -> 1)
  float a, b;            // Y = a * rowscale * (A X) + b * Z
  const float* Z;        // [n][K] (nullable)
  int zvec;              // Z rows are 16-byte aligned and K % 4 == 0
  float* Y;              // [n][ld] (nullable: measure only)
  const float* P;        // measure: [n][ld], against which Y is measured; may be Y itself
  const float* L;        // nullable: measure = sum |Y - P| per column; else sum L * (Y - Z'), Z' = P [n][K]
  float* Xs;             // nullable: next product's operand, Y * xscale
  const float* xscale;
  double* partial;       // [slots][ld]
  double* part;          // measure: [64][kMainBlocks + kFixBlocks]
  Ctl* ctl;
};

// Row i, columns 4 cl .. 4 cl + 3 from their sums; adds to the measure.
__device__ __forceinline__ void finish_row(const SpmmArgs& A, int64_t i, int cl, const double* acc, double* d) {
  const int k0 = cl * 4;
  float z[4] = {0.f, 0.f, 0.f, 0.f};
  if (A.Z) {
    if (A.zvec) {
      const f32x4 v = *(const f32x4*)(A.Z + i * A.K + k0);
      z[0] = v.x, z[1] = v.y, z[2] = v.z, z[3] = v.w;
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (k0 + q < A.K) z[q] = A.Z[i * A.K + k0 + q];
    }
  }
  const double rs = A.rowscale ? (double)A.rowscale[i] : 1.0;
  float y[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    double t = (double)A.a * rs * acc[q];
    if (A.Z) t += (double)A.b * (double)z[q];
    y[q] = k0 + q < A.K ? (float)t : 0.f;
  }
  if (A.L) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (k0 + q < A.K) d[q] += (double)A.L[i * A.ld + k0 + q] * ((double)y[q] - (double)A.P[i * A.K + k0 + q]);
    return;
  }
  const f32x4 p = *(const f32x4*)(A.P + i * A.ld + k0);
  d[0] += fabs((double)y[0] - (double)p.x);
  d[1] += fabs((double)y[1] - (double)p.y);
  d[2] += fabs((double)y[2] - (double)p.z);
  d[3] += fabs((double)y[3] - (double)p.w);
  *(f32x4*)(A.Y + i * A.ld + k0) = f32x4{y[0], y[1], y[2], y[3]};
  if (A.Xs) {
    const float s = A.xscale[i];
    *(f32x4*)(A.Xs + i * A.ld + k0) = f32x4{y[0] * s, y[1] * s, y[2] * s, y[3] * s};
  }
}

// The workgroup's measure: d of every unit's column lanes, added over the
// units in order, to column k's partial `slot`.
template <int LPR>
__device__ __forceinline__ void store_measure(const SpmmArgs& A, const double* d, int slot) {
  __shared__ double sh[kUnits][4 * LPR];
  const int unit = threadIdx.x / kUnit, l = threadIdx.x % kUnit;
  if (l < LPR) {
#pragma unroll
    for (int q = 0; q < 4; ++q) sh[unit][4 * l + q] = d[q];
  }
  __syncthreads();
  const int k = threadIdx.x;
  if (k < 4 * LPR && k < A.K) {
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kUnits; ++u) s += sh[u][k];
    A.part[(int64_t)k * (kMainBlocks + kFixBlocks) + slot] = s;
  }
}

// Lane n of the calling lane's row of 16 lanes (all 16 active): DPP
// row_newbcast, no LDS trip.
template <int N>
__device__ __forceinline__ int row_lane(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + N, 0xF, 0xF, false);
}

// Eight nonzeros of a segment, H .. H + 7 of the 16 whose columns the unit's
// lanes hold: eight gathers in flight, then the sums in order.
template <int H>
__device__ __forceinline__ void add8(const float* __restrict__ X, int64_t ld, int c, int nl, double* acc) {
  f32x4 x[8];
  const int v[8] = {row_lane<H>(c),     row_lane<H + 1>(c), row_lane<H + 2>(c), row_lane<H + 3>(c),
                    row_lane<H + 4>(c), row_lane<H + 5>(c), row_lane<H + 6>(c), row_lane<H + 7>(c)};
#pragma unroll
  for (int j = 0; j < 8; ++j) x[j] = *(const f32x4*)(X + v[j] * ld);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    if (H + j < nl) {
      acc[0] += (double)x[j].x;
      acc[1] += (double)x[j].y;
      acc[2] += (double)x[j].z;
      acc[3] += (double)x[j].w;
    }
  }
}

// LPR lanes span the (padded) columns of a row of X, kUnit / LPR nonzeros
// are taken at a time.
// Bound by the row gathers: R-MAT 2^17 vertices, 3.9M nonzeros, K = 64, a
// product of 1.0 GB of gathered rows and 0.13 GB of streamed ones takes 110
// us (10 TB/s out of L2 and the Infinity Cache), k_spmm_fix 11 us, k_colsum
// 7 us.  The kernels that walked the tiles took 556 us at bs 8 (chunks of
// 1024 tiles, the densest one set the time) and 1.7 ms at bs 16 already on
// 1007 vertices; forward and adjoint together 82.5 -> 21.7 ms, at 2^22
// vertices 980 -> 838 ms.
template <int LPR>
__global__ __launch_bounds__(kBlk) void k_spmm(const SpmmArgs A) {
  if (A.ctl->done) return;
  constexpr int EP = kUnit / LPR;
  const int unit = threadIdx.x / kUnit, l = threadIdx.x % kUnit;
  const int cl = l % LPR, el = l / LPR;
  const bool col_ok = cl * 4 < A.ld;
  const float* __restrict__ X = A.X + (col_ok ? cl * 4 : 0);
  const int64_t ld = A.ld;
  double d[4] = {0.0, 0.0, 0.0, 0.0};
  for (int64_t u = (int64_t)blockIdx.x * kUnits + unit; u < A.nseg; u += (int64_t)gridDim.x * kUnits) {
    const Seg s = A.segs[u];
    const int len = (int)(s.sl >> 48) & 0x7FFF;
    const int32_t* __restrict__ col = A.col + (s.sl & 0xFFFFFFFFFFFFull);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    if constexpr (LPR == kUnit) {
      for (int e = 0; e < len; e += kUnit) {
        // lanes past the end repeat the last column: their gathers hit the
        // line of the last nonzero and are not added
        const int c = col[min(e + l, len - 1)];
        add8<0>(X, ld, c, len - e, acc);
        if (e + 8 < len) add8<8>(X, ld, c, len - e, acc);
      }
    } else {
      constexpr int U = 4;
      for (int e = el; e < len; e += U * EP) {
        int c[U];
        f32x4 x[U];
#pragma unroll
        for (int j = 0; j < U; ++j) c[j] = col[min(e + j * EP, len - 1)];
#pragma unroll
        for (int j = 0; j < U; ++j) x[j] = *(const f32x4*)(X + c[j] * ld);
#pragma unroll
        for (int j = 0; j < U; ++j) {
          if (e + j * EP < len) {
            acc[0] += (double)x[j].x;
            acc[1] += (double)x[j].y;
            acc[2] += (double)x[j].z;
            acc[3] += (double)x[j].w;
          }
        }
      }
#pragma unroll
      for (int off = LPR; off < kUnit; off <<= 1) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] += __shfl_xor(acc[q], off);
      }
    }
    if (el == 0 && col_ok) {
      if (s.sl >> 63) {
        double* p = A.partial + (int64_t)s.slot * ld + cl * 4;
#pragma unroll
        for (int q = 0; q < 4; ++q) p[q] = acc[q];
      } else {
        finish_row(A, s.row, cl, acc, d);
      }
    }
  }
  store_measure<LPR>(A, d, blockIdx.x);
}

// Rows of several segments: a wave adds a row's partials, its four units (and
// the unit's spare lanes) each every (4 EP)-th of them in order, then the
// lanes' sums in a fixed tree.
template <int LPR>
__global__ __launch_bounds__(kBlk) void k_spmm_fix(const SpmmArgs A) {
  if (A.ctl->done) return;
  constexpr int EP = kUnit / LPR, W = (kWave / kUnit) * EP;
  const int lane = lane_id();
  const int cl = lane % LPR, el = lane / LPR;  // el in [0, W)
  const bool col_ok = cl * 4 < A.ld;
  double d[4] = {0.0, 0.0, 0.0, 0.0};
  const int64_t nw = (int64_t)gridDim.x * (kBlk / kWave);
  for (int64_t w = wave_index(); w < A.nmulti; w += nw) {  // wave-uniform
    const int32_t i = A.mrow[w];
    const int64_t s0 = A.off[i] >> 32, s1 = A.off[i + 1] >> 32;
    const double* __restrict__ P = A.partial + (col_ok ? cl * 4 : 0);
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    constexpr int U = 4;
    for (int64_t s = s0 + el; s < s1; s += U * W) {
      double v[U][4];
#pragma unroll
      for (int j = 0; j < U; ++j) {
        const double* p = P + min(s + j * W, s1 - 1) * A.ld;
#pragma unroll
        for (int q = 0; q < 4; ++q) v[j][q] = p[q];
      }
#pragma unroll
      for (int j = 0; j < U; ++j) {
        if (s + j * W < s1) {
#pragma unroll
          for (int q = 0; q < 4; ++q) acc[q] += v[j][q];
        }
      }
    }
#pragma unroll
    for (int off = LPR; off < kWave; off <<= 1) {
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] += __shfl_xor(acc[q], off);
    }
    if (el == 0 && col_ok) finish_row(A, i, cl, acc, d);
  }
  // one measure per wave: only its first unit's lanes hold any
  if (lane >= kUnit) d[0] = d[1] = d[2] = d[3] = 0.0;
  store_measure<LPR>(A, d, kMainBlocks + blockIdx.x);
}

// Column sums of |Y| ([n][K]) into the same partials, kMainBlocks of them.
__global__ __launch_bounds__(kBlk) void k_col_abs(const float* __restrict__ Y, int32_t n, int32_t K, double* part) {
  __shared__ double sh[kBlk];
  const int k = threadIdx.x & 63, sub = threadIdx.x >> 6;
  double s = 0.0;
  if (k < K) {
    for (int64_t i = (int64_t)blockIdx.x * 4 + sub; i < n; i += (int64_t)gridDim.x * 4)
      s += fabs((double)Y[i * K + k]);
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  if (sub == 0 && k < K)
    part[(int64_t)k * (kMainBlocks + kFixBlocks) + blockIdx.x] = sh[k] + sh[k + 64] + sh[k + 128] + sh[k + 192];
}

// Workgroup k adds column k's partials [0, n0) and [kMainBlocks, kMainBlocks
// + n1) in a fixed order.  NORM: they are the columns' norms.  Otherwise the
// last workgroup to finish compares them with tol: done where max_k val[k] /
// norm[k] (val[k] where norm[k] is 0) is below it.
template <bool NORM>
__global__ __launch_bounds__(kBlk) void k_colsum(const double* __restrict__ part, int n0, int n1, int K, double tol,
                                                 Ctl* ctl) {
  if (!NORM && ctl->done) return;
  __shared__ double sh[kBlk];
  const int k = blockIdx.x, t = threadIdx.x;
  const double* __restrict__ p = part + (int64_t)k * (kMainBlocks + kFixBlocks);
  double s = 0.0;
#pragma unroll 4
  for (int i = t; i < n0; i += kBlk) s += p[i];
  for (int i = t; i < n1; i += kBlk) s += p[kMainBlocks + i];
  sh[t] = s;
  __syncthreads();
  for (int off = kBlk / 2; off > 0; off >>= 1) {
    if (t < off) sh[t] += sh[t + off];
    __syncthreads();
  }
  __shared__ bool last;
  if (t == 0) {
    last = false;
    if (NORM) {
      ctl->norm[k] = sh[0];
    } else {
      __hip_atomic_store(&ctl->val[k], sh[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last = __hip_atomic_fetch_add(&ctl->ticket, 1ull, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) + 1 ==
             (unsigned long long)K;
    }
  }
  __syncthreads();
  if (!last || t >= kWave) return;
  double m = 0.0;
  if (t < K) {
    const double v = __hip_atomic_load(&ctl->val[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const double r = ctl->norm[t] > 0.0 ? v / ctl->norm[t] : v;
    m = m < r ? r : m;
  }
  for (int off = 1; off < kWave; off <<= 1) {
    const double o = __shfl_xor(m, off);
    m = m < o ? o : m;
  }
  if (t == 0) {
    ctl->ticket = 0;
    ctl->dmax = m;
    ctl->iters += 1;
    if (m < tol) ctl->done = 1;
  }
}

__global__ void k_invdeg(const int32_t* __restrict__ deg, float* __restrict__ inv, int32_t n) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) inv[i] = deg[i] > 0 ? 1.0f / (float)deg[i] : 0.0f;
}

__global__ void k_ctl_init(Ctl* ctl) {
  ctl->done = ctl->iters = ctl->ticket = 0;
  ctl->dmax = 0.0;
}

// dst = src ([n][K] -> [n][ld], zeros in the padding) and, with xs, xs =
// dst * scale (per row).  dst may be null.
__global__ __launch_bounds__(256) void k_pad(const float* __restrict__ src, int32_t n, int32_t K, int32_t ld,
                                             float* __restrict__ dst, const float* __restrict__ scale,
                                             float* __restrict__ xs) {
  const int64_t q4 = ld / 4, nt = (int64_t)gridDim.x * blockDim.x;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n * q4; idx += nt) {
    const int64_t i = idx / q4;
    const int k0 = (int)(idx % q4) * 4;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = k0 + q < K ? src[i * K + k0 + q] : 0.f;
    if (dst) *(f32x4*)(dst + i * ld + k0) = f32x4{v[0], v[1], v[2], v[3]};
    if (xs) {
      const float s = scale[i];
      *(f32x4*)(xs + i * ld + k0) = f32x4{v[0] * s, v[1] * s, v[2] * s, v[3] * s};
    }
  }
}

// dst [n][K] = a * src [n][ld].
__global__ __launch_bounds__(256) void k_unpad(const float* __restrict__ src, int32_t n, int32_t K, int32_t ld, float a,
                                               float* __restrict__ dst) {
  const int64_t nt = (int64_t)gridDim.x * blockDim.x;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < (int64_t)n * K; idx += nt) {
    const int64_t i = idx / K, k = idx % K;
    dst[idx] = a * src[i * ld + k];
  }
}

unsigned grid_of(int64_t items, int per_block) {
  return (unsigned)std::max<int64_t>(1, (items + per_block - 1) / per_block);
}

// For k_pad and k_unpad, which go on past it: a launch has less than 2^32
// threads, the arrays up to 2^31 rows of 64.
unsigned grid_most(int64_t items) { return std::min(grid_of(items, 256), 1u << 22); }

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The operand of a solve's products: the matrix as CSR segments.
struct Operand {
  CsrList csr;
  const Seg* segs = nullptr;
  const int64_t* off = nullptr;
  const int32_t* mrow = nullptr;
  int64_t nseg = 0, nslot = 0, nmulti = 0;
};

int make_operand(const gbo_bsr* M, Workspace& mem, Operand* o, hipStream_t st) {
  const char* who = "gbo_ppr";
  const int32_t n = M->nrows;
  int rc = expand_csr(M, mem, &o->csr, st);
  if (rc) return rc;
  int64_t *cnt = nullptr, *moff = nullptr, *off = nullptr;
  int32_t *multi = nullptr, *mrow = nullptr;
  if ((rc = mem.alloc(&cnt, sizeof(int64_t) * (size_t)std::max(n, 1), who)) ||
      (rc = mem.alloc(&multi, sizeof(int32_t) * (size_t)std::max(n, 1), who)) ||
      (rc = mem.alloc(&moff, sizeof(int64_t) * ((size_t)n + 1), who)) ||
      (rc = mem.alloc(&off, sizeof(int64_t) * ((size_t)n + 1), who)))
    return rc;
  k_seg_count<<<grid_of(n, 256), 256, 0, st>>>(o->csr.rowptr, n, cnt, multi);
  GBO_LAUNCH_CHECK();
  if ((rc = scan_exclusive<int64_t, int64_t>(cnt, off, n, st, mem))) return rc;
  if ((rc = scan_exclusive<int32_t, int64_t>(multi, moff, n, st, mem))) return rc;
  int64_t tot = 0;
  if ((rc = read_back(&tot, off + n, sizeof(int64_t), st)) || (rc = read_back(&o->nmulti, moff + n, sizeof(int64_t), st)))
    return rc;
  o->nseg = tot & 0xFFFFFFFF;
  o->nslot = tot >> 32;
  Seg* segs = nullptr;
  if ((rc = mem.alloc(&segs, sizeof(Seg) * (size_t)std::max<int64_t>(o->nseg, 1), who)) ||
      (rc = mem.alloc(&mrow, sizeof(int32_t) * (size_t)std::max<int64_t>(o->nmulti, 1), who)))
    return rc;
  k_seg_fill<<<grid_of(n, 256), 256, 0, st>>>(o->csr.rowptr, n, off, moff, segs, mrow);
  GBO_LAUNCH_CHECK();
  o->segs = segs;
  o->off = off;
  o->mrow = mrow;
  return GBO_OK;
}

int main_blocks(const Operand& o) { return (int)std::min<int64_t>(kMainBlocks, (o.nseg + kUnits - 1) / kUnits); }
int fix_blocks(const Operand& o) { return (int)std::min<int64_t>(kFixBlocks, (o.nmulti + kBlk / kWave - 1) / (kBlk / kWave)); }

template <int LPR>
int spmm_t(const Operand& o, const SpmmArgs& A, hipStream_t st) {
  const int nb = main_blocks(o), nf = fix_blocks(o);
  if (nb > 0) k_spmm<LPR><<<nb, kBlk, 0, st>>>(A);
  if (nf > 0) k_spmm_fix<LPR><<<nf, kBlk, 0, st>>>(A);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// One product with its measure, and the measure's verdict.
int spmm(const Operand& o, SpmmArgs A, double tol, hipStream_t st) {
  A.segs = o.segs;
  A.nseg = o.nseg;
  A.mrow = o.mrow;
  A.nmulti = o.nmulti;
  A.off = o.off;
  A.col = o.csr.col;
  A.zvec = A.K % 4 == 0 && al16(A.Z);
  int rc = A.ld > 32 ? spmm_t<16>(o, A, st)
           : A.ld > 16 ? spmm_t<8>(o, A, st)
           : A.ld > 8 ? spmm_t<4>(o, A, st)
           : A.ld > 4 ? spmm_t<2>(o, A, st)
                      : spmm_t<1>(o, A, st);
  if (rc) return rc;
  k_colsum<false><<<A.K, kBlk, 0, st>>>(A.part, main_blocks(o), fix_blocks(o), A.K, tol, A.ctl);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// Scratch of a solve: padded iterates, measure partials, state.
struct Scratch {
  float* inv = nullptr;
  double *part = nullptr, *partial = nullptr;
  Ctl* ctl = nullptr;
};

int make_scratch(const int32_t* d_outdeg, int32_t n, int32_t ld, int64_t nslot, Workspace& mem, Scratch* s,
                 hipStream_t st) {
  const char* who = "gbo_ppr";
  int rc;
  if ((rc = mem.alloc(&s->inv, sizeof(float) * (size_t)std::max(n, 1), who)) ||
      (rc = mem.alloc(&s->part, sizeof(double) * 64 * (kMainBlocks + kFixBlocks), who)) ||
      (rc = mem.alloc(&s->partial, sizeof(double) * (size_t)std::max<int64_t>(nslot * ld, 1), who)) ||
      (rc = mem.alloc(&s->ctl, sizeof(Ctl), who)))
    return rc;
  k_invdeg<<<grid_of(n, 256), 256, 0, st>>>(d_outdeg, s->inv, n);
  k_ctl_init<<<1, 1, 0, st>>>(s->ctl);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// The columns' norms of the driving vectors: the change is measured relative
// to them (1 for a distribution).
int col_norms(const float* Y, int32_t n, int32_t K, const Scratch& s, hipStream_t st) {
  const int nb = (int)std::min<int64_t>(kMainBlocks, grid_of(n, 16));
  k_col_abs<<<nb, kBlk, 0, st>>>(Y, n, K, s.part);
  k_colsum<true><<<K, kBlk, 0, st>>>(s.part, nb, 0, K, 0.0, s.ctl);
  GBO_LAUNCH_CHECK();
  return GBO_OK;
}

// Runs step(it) for it = 0, 1, ... until the device says done or max_iter.
template <class Step>
int iterate(int32_t max_iter, const Scratch& s, int32_t* iters, double* dmax, hipStream_t st, Step step) {
  int32_t it = 0;
  Ctl h{};
  while (it < max_iter && !h.done) {
    for (int b = 0; b < kBatch && it < max_iter; ++b, ++it) {
      const int rc = step(it);
      if (rc) return rc;
    }
    const int rc = read_back(&h, s.ctl, offsetof(Ctl, val), st);
    if (rc) return rc;
  }
  *iters = (int32_t)h.iters;
  *dmax = h.dmax;
  return GBO_OK;
}

}  // namespace
}  // namespace gbo

using namespace gbo;

extern "C" {

int gbo_ppr_forward(const gbo_bsr* AT, const int32_t* d_outdeg, int32_t K, float alpha, const float* d_s, float* d_p,
                    double tol, int32_t max_iter, int32_t* h_iters, double* h_delta, gbo_stream_t stream) {
  int rc = validate_bsr(AT, 0, "gbo_ppr_forward");
  if (rc) return rc;
  if (AT->nrows != AT->ncols) return set_error(GBO_EINVAL, "gbo_ppr_forward: matrix must be square");
  if (K < 1 || K > 64) return set_error(GBO_EINVAL, "gbo_ppr_forward: 1 <= K <= 64");
  if (!(alpha > 0.0f && alpha < 1.0f) || max_iter < 1) return set_error(GBO_EINVAL, "gbo_ppr_forward: bad alpha/max_iter");
  if (!d_outdeg || !d_s || !d_p) return set_error(GBO_EINVAL, "gbo_ppr_forward: null argument");
  if (AT->bs > 32) return set_error(GBO_EUNSUPPORTED, "gbo_ppr_forward: block sizes 8, 16, 32");
  if (AT->bs == 8 && AT->ncols > (1 << 29))
    return set_error(GBO_EUNSUPPORTED, "PPR at block size 8 supports up to 2^29 vertices");
  hipStream_t st = stream;
  const int32_t n = AT->nrows, ld = (K + 3) / 4 * 4;
  const size_t bytes = sizeof(float) * (size_t)std::max<int64_t>((int64_t)n * ld, 1);
  Workspace mem(st);
  Operand o;
  Scratch s;
  if ((rc = make_operand(AT, mem, &o, st)) || (rc = make_scratch(d_outdeg, n, ld, o.nslot, mem, &s, st))) return rc;
  // the iterate stays in the caller's buffer where its rows can be read 16
  // bytes at a time; the products read it scaled by 1 / outdeg, from two
  // buffers in turn
  float *p = d_p, *xs[2] = {nullptr, nullptr};
  const bool own = ld != K || !al16(d_p);
  if ((own && (rc = mem.alloc(&p, bytes, "gbo_ppr_forward"))) ||
      (rc = mem.alloc(&xs[0], bytes, "gbo_ppr_forward")) || (rc = mem.alloc(&xs[1], bytes, "gbo_ppr_forward")))
    return rc;
  k_pad<<<grid_most((int64_t)n * (ld / 4)), 256, 0, st>>>(d_s, n, K, ld, p, s.inv, xs[0]);  // p_0 = s
  GBO_LAUNCH_CHECK();
  if ((rc = col_norms(d_s, n, K, s, st))) return rc;
  SpmmArgs A{};
  A.K = K;
  A.ld = ld;
  A.a = alpha;
  A.b = 1.0f - alpha;
  A.Z = d_s;
  A.Y = p;
  A.P = p;
  A.xscale = s.inv;
  A.partial = s.partial;
  A.part = s.part;
  A.ctl = s.ctl;
  int32_t it = 0;
  double dmax = 0.0;
  rc = iterate(max_iter, s, &it, &dmax, st, [&](int32_t i) {
    A.X = xs[i & 1];
    A.Xs = xs[(i + 1) & 1];
    return spmm(o, A, tol, st);
  });
  if (rc) return rc;
  if (own) {
    k_unpad<<<grid_most((int64_t)n * K), 256, 0, st>>>(p, n, K, ld, 1.0f, d_p);
    GBO_LAUNCH_CHECK();
    GBO_HIP_CHECK(hipStreamSynchronize(st));
  }
  if (h_iters) *h_iters = it;
  if (h_delta) *h_delta = dmax;
  if (!(dmax < tol))
    return set_error(GBO_ENOCONV, "gbo_ppr_forward: not converged after %d iterations (%.3e)", it, dmax);
  return GBO_OK;
}

int gbo_ppr_adjoint(const gbo_bsr* A, const gbo_bsr* AT, const int32_t* d_outdeg, int32_t K, float alpha,
                    const float* d_s, const float* d_p, const float* d_w, float* d_grad_s, double* h_grad_alpha,
                    double tol, int32_t max_iter, int32_t* h_iters, gbo_stream_t stream) {
  int rc = validate_bsr(A, 0, "gbo_ppr_adjoint(A)");
  if (rc) return rc;
  rc = validate_bsr(AT, 0, "gbo_ppr_adjoint(AT)");
  if (rc) return rc;
  if (A->nrows != A->ncols || AT->nrows != A->nrows) return set_error(GBO_EINVAL, "gbo_ppr_adjoint: shapes");
  if (K < 1 || K > 64) return set_error(GBO_EINVAL, "gbo_ppr_adjoint: 1 <= K <= 64");
  if (!(alpha > 0.0f && alpha < 1.0f) || max_iter < 1) return set_error(GBO_EINVAL, "gbo_ppr_adjoint: bad alpha/max_iter");
  if (!d_outdeg || !d_s || !d_p || !d_w || !d_grad_s) return set_error(GBO_EINVAL, "gbo_ppr_adjoint: null argument");
  if (A->bs > 32 || AT->bs > 32) return set_error(GBO_EUNSUPPORTED, "gbo_ppr_adjoint: block sizes 8, 16, 32");
  if ((A->bs == 8 && A->ncols > (1 << 29)) || (AT->bs == 8 && AT->ncols > (1 << 29)))
    return set_error(GBO_EUNSUPPORTED, "PPR at block size 8 supports up to 2^29 vertices");
  hipStream_t st = stream;
  const int32_t n = A->nrows, ld = (K + 3) / 4 * 4;
  const size_t bytes = sizeof(float) * (size_t)std::max<int64_t>((int64_t)n * ld, 1);
  const bool same = A->rowptr == AT->rowptr && A->colind == AT->colind && A->tiles == AT->tiles && A->bs == AT->bs &&
                    A->nblocks == AT->nblocks;
  Workspace mem(st);
  Operand o, oT;
  Scratch s;
  if ((rc = make_operand(A, mem, &o, st))) return rc;
  if (same) oT = o;
  else if ((rc = make_operand(AT, mem, &oT, st))) return rc;
  if ((rc = make_scratch(d_outdeg, n, ld, std::max(o.nslot, oT.nslot), mem, &s, st))) return rc;
  float* lam[2] = {nullptr, nullptr};
  if ((rc = mem.alloc(&lam[0], bytes, "gbo_ppr_adjoint")) || (rc = mem.alloc(&lam[1], bytes, "gbo_ppr_adjoint")))
    return rc;
  const unsigned padg = grid_most((int64_t)n * (ld / 4));
  k_pad<<<padg, 256, 0, st>>>(d_w, n, K, ld, lam[0], nullptr, nullptr);
  GBO_LAUNCH_CHECK();
  if ((rc = col_norms(d_w, n, K, s, st))) return rc;
  // lambda' = alpha * D^-1 A lambda + w
  SpmmArgs S{};
  S.K = K;
  S.ld = ld;
  S.rowscale = s.inv;
  S.a = alpha;
  S.b = 1.0f;
  S.Z = d_w;
  S.partial = s.partial;
  S.part = s.part;
  S.ctl = s.ctl;
  int32_t it = 0;
  double dmax = 0.0;
  rc = iterate(max_iter, s, &it, &dmax, st, [&](int32_t i) {
    S.X = S.P = lam[i & 1];
    S.Y = lam[(i + 1) & 1];
    return spmm(o, S, tol, st);
  });
  if (rc) return rc;
  const float* cur = lam[it & 1];
  float* xs = lam[(it + 1) & 1];
  // grad_s = (1 - alpha) * lambda
  k_unpad<<<grid_most((int64_t)n * K), 256, 0, st>>>(cur, n, K, ld, 1.0f - alpha, d_grad_s);
  // dL/dalpha = sum_k lambda_k . (P^T p_k - s_k)
  k_pad<<<padg, 256, 0, st>>>(d_p, n, K, ld, nullptr, s.inv, xs);
  k_ctl_init<<<1, 1, 0, st>>>(s.ctl);
  GBO_LAUNCH_CHECK();
  SpmmArgs T{};
  T.K = K;
  T.ld = ld;
  T.X = xs;
  T.a = 1.0f;
  T.P = d_s;
  T.L = cur;
  T.partial = s.partial;
  T.part = s.part;
  T.ctl = s.ctl;
  if ((rc = spmm(oT, T, 0.0, st))) return rc;
  double ga[64];
  if ((rc = read_back(ga, s.ctl->val, sizeof(double) * K, st))) return rc;
  if (h_grad_alpha) {
    double g = 0.0;
    for (int32_t k = 0; k < K; ++k) g += ga[k];
    *h_grad_alpha = g;
  }
  if (h_iters) *h_iters = it;
  if (!(dmax < tol))
    return set_error(GBO_ENOCONV, "gbo_ppr_adjoint: not converged after %d iterations (%.3e)", it, dmax);
  return GBO_OK;
}

}  // extern "C"
