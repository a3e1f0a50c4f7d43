// tail.hip -- the V-cycle's smallest levels in one launch of one workgroup.
//
// A level of a few thousand rows keeps no more than a handful of CUs busy, and
// its V-cycle is a chain: 16 colour steps a sweep (ComputeSYMGS_ref.cpp:62-100
// by colours), the residual and restriction, the coarser levels, the
// prolongation and another sweep (ComputeMG_ref.cpp:39-63).  As launches each
// link costs 2.7 us (64 rows and less) to 4.6 us (4096 rows): the launch and,
// inside it, one memory latency each for the arguments, the tile's record, the
// matrix and x.  Here one workgroup of 16 wavefronts runs the levels' whole
// part of the V-cycle with x and the coarser residuals in LDS, so a step costs
// a barrier and one row's arithmetic.
//
// Wavefront w owns the tiles (64 rows of a colour) t with t % 16 == w, at most
// one of a colour.  The matrix of its next tile is on its way while the steps
// of other wavefronts' tiles run; where a level has at most 16 tiles it stays
// in registers for the whole sweep.
//
// With several right-hand sides each has a workgroup of its own: a one-level
// V-cycle of 16 of them, launches / here, 1000 rows 56 / 21 us, 4096 57 / 31,
// 5832 58 / 45.
//
// Every row meets the same terms in the same order as in the launches it
// replaces (kernels.hip's gs_row, mixed.hip's gs32_row and their transfers).
//
// Measured (MI355X): the four levels of 16^3 296 -> 128 us FP64, 233 -> 107 us
// FP32.  What bounds it: a step of a level whose matrix stays in registers is
// 0.6 us of dependent LDS reads, 27 subtractions, a division and the barrier;
// a step over 512 rows streamed from L2 1.8 us (27 loads of 512 bytes for each
// of 8 wavefronts); and 2 us of first loads a level and sweep.
#include <atomic>
#include <climits>

#include "internal.hpp"

namespace hpcgx {
namespace {

constexpr int kTailWaves = 16;
constexpr int kTailColors = 16;
// The largest level that runs so.  A one-level V-cycle, as launches / here (us,
// in a graph, about 10 of them the graph's own; FP64, FP32): 1000 rows 46.1 /
// 20.8, 38.2 / 19.7; 1728 rows 57.4 / 27.1, 44.3 / 23.5; 4096 rows 55.7 / 37.1,
// 42.9 / 27.6; 5832 rows 56.9 / 54.0, 44.5 / 39.9.  Beyond, one CU's loads of
// the matrix are what a step waits for, and many CUs' launches are faster.
constexpr int64_t kTailRows = 6000;
constexpr size_t kTailLds = 150 << 10;  // x and r of every level

template <class V, class T>
struct TailLevel {
  int n, ncolors, nc;
  int xo, ro;  // the level's x and r in LDS
  const int32_t *col;
  const V *val;
  const T *diag;
  const int32_t *f2c;
  const int32_t *trec;  // Level::trec, or null where the 32-bit ids are to be read
  int cptr[kTailColors + 1], ctile[kTailColors + 1];
};
template <class V, class T>
struct TailArgs {
  int nlev;
  int stride;  // right-hand sides of r and x, [n][stride]; workgroup k takes column k
  const T *r;
  T *x;
  double *rz;         // r.z partials of the last sweep, or null
  const double *r64;  // their r where T is float
  TailLevel<V, T> lev[kMaxLevels];
};

// Wait for the workgroup's LDS accesses only: the matrix loads in flight for
// the next step stay in flight.
__device__ inline void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// sum - v_0 x_0 - v_1 x_1 - ..  x(j) reads LDS kAhead slots ahead of the sum;
// the empty asm keeps the reads from all going first (128 registers).
template <class V, class T, class X>
__device__ inline T terms(T sum, const V (&v)[kSlots], X &&x) {
  constexpr int kAhead = sizeof(T) == 8 ? 14 : kSlots;
  T xs[kAhead];
#pragma unroll
  for (int j = 0; j < kAhead; ++j) xs[j] = x(j);
#pragma unroll
  for (int j = 0; j < kSlots; ++j) {
    sum -= (T)v[j] * xs[j % kAhead];
    if (j + kAhead < kSlots) {
      asm volatile("" : "+v"(sum) : : "memory");
      xs[j % kAhead] = x(j + kAhead);
    }
  }
  return sum;
}

// Element i of column j of an n-row array: one lane offset for all columns,
// the column's as the load's scalar offset (no address per column in
// registers).
typedef __amdgpu_buffer_rsrc_t BufView;
__device__ inline BufView column_view(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}
template <class V>
__device__ inline V column_at(BufView p, int j, int n, int i) {
  const int o = i * (int)sizeof(V), c = j * n * (int)sizeof(V);
  if constexpr (sizeof(V) == 8)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(p, o, c, 0));
  else if constexpr (sizeof(V) == 4)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(p, o, c, 0));
  else
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b16(p, o, c, 0));
}

typedef __attribute__((address_space(4))) int32_t ConstI32;  // read by scalar loads

// The first tile at or after tile0 that is wavefront w's.
__device__ inline int first_tile(int tile0, int w) {
  return tile0 + ((w - tile0) & (kTailWaves - 1));
}

template <class V, class T>
__global__ __launch_bounds__(64 * kTailWaves) void k_tail(const TailArgs<V, T> A) {
  constexpr bool F64 = sizeof(T) == 8;
  extern __shared__ double tail_lds[];
  T *const lds = reinterpret_cast<T *>(tail_lds);
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));

  __shared__ int32_t colours[kMaxLevels][2][kTailColors + 1];  // first rows, first tiles
  for (int k = threadIdx.x; k < A.nlev * (kTailColors + 1); k += 64 * kTailWaves) {
    const int l = k / (kTailColors + 1), c = k % (kTailColors + 1);
    colours[l][0][c] = A.lev[l].cptr[c];
    colours[l][1][c] = A.lev[l].ctile[c];
  }
  for (int l = 0; l < A.nlev; ++l)
    for (int i = threadIdx.x; i < A.lev[l].n; i += 64 * kTailWaves) lds[A.lev[l].xo + i] = (T)0;
  for (int i = threadIdx.x; i < A.lev[0].n; i += 64 * kTailWaves)
    lds[A.lev[0].ro + i] = A.r[(int64_t)i * A.stride + blockIdx.x];
  lds_barrier();

  // down the levels and up again
  for (int visit = 0; visit < 2 * A.nlev - 1; ++visit) {
    const bool up = visit >= A.nlev;
    const int l = up ? 2 * A.nlev - 2 - visit : visit;
    const TailLevel<V, T> &L = A.lev[l];
    T *const x = lds + L.xo;
    if (up) {  // prolongation
      const T *xc = lds + A.lev[l + 1].xo;
      for (int k = threadIdx.x; k < L.nc; k += 64 * kTailWaves) x[L.f2c[k]] += xc[k];
    }

    // the symmetric sweep: steps 0 .. 2 ncolors - 1
    const int nc = L.ncolors, steps = 2 * nc;
    const int32_t(&tab)[2][kTailColors + 1] = colours[l];
    // the colours of which this wavefront has a tile
    const int k = lane < nc ? lane : nc - 1;
    const uint32_t mine = (uint32_t)__ballot(lane < nc && first_tile(tab[1][k], w) < tab[1][k + 1]);
    // this wavefront's next step, its colour and tile, the colour's tiles
    int q = -1, c = -1, t = 0, tile0 = 0, tile1 = 0, have = -1;
    V v[kSlots] = {};
    int32_t cj[kSlots] = {};
    T d = (T)1, ri = (T)0;
    int i = 0;
    bool row = false, due = true;
    auto next = [&]() {
      uint32_t m = q < nc ? mine & (~0u << (c + 1)) : 0u;  // colours still to come, forward
      if (m) {
        c = q = __builtin_ctz(m);
      } else {
        m = q < nc ? mine : mine & ((1u << c) - 1u);  // backward
        c = m ? 31 - __builtin_clz(m) : 0;
        q = m ? steps - 1 - c : steps;
      }
      tile0 = __builtin_amdgcn_readfirstlane(tab[1][c]);
      tile1 = __builtin_amdgcn_readfirstlane(tab[1][c + 1]);
      t = first_tile(tile0, w);
    };
    auto load = [&]() {
      if (q >= steps || t == have) return;
      have = t;
      const int row0 = __builtin_amdgcn_readfirstlane(tab[0][c]);
      const int row1 = __builtin_amdgcn_readfirstlane(tab[0][c + 1]);
      const int tb = row0 + (t - tile0) * kTile;
      row = tb + lane < row1;
      i = min(tb + lane, row1 - 1);
      // (the slots' pointers formed here, not kept in registers over the loop)
      int ns = L.n;
      asm volatile("" : "+s"(ns));
      const BufView val = column_view(L.val, kSlots * ns * sizeof(V));
      const BufView col = column_view(L.col, kSlots * ns * 4);
#pragma unroll
      for (int j = 0; j < kSlots; ++j) v[j] = column_at<V>(val, j, ns, i);
      d = L.diag[i];
      ri = lds[L.ro + i];
      const ConstI32 *rec = (const ConstI32 *)(uintptr_t)(L.trec + t * kBaseStride);
      const uint32_t f = L.trec ? (uint32_t)rec[kRecFlags] : (uint32_t)kTile32;
      if ((f & 3u) == kTile8 && (f >> 8 & kAllAffine) == kAllAffine) {
#pragma unroll
        for (int j = 0; j < kSlots; ++j) cj[j] = rec[j] + (i - tb);
      } else {  // (the 32-bit ids: 8-bit ones would have to arrive here to be added to)
#pragma unroll
        for (int j = 0; j < kSlots; ++j) cj[j] = column_at<int32_t>(col, j, ns, i);
      }
    };
    const int rz_from = A.rz && visit == 2 * A.nlev - 2 ? nc : INT_MAX;  // steps with r.z
    next();
    for (int s = 0; s < steps; ++s) {
      if (s != nc) lds_barrier();  // the two steps of the turn are one colour's
      // a tile's loads go out a step after this wavefront's last one, when the
      // others no longer wait for its x
      if (due) load();
      due = false;
      if (q == s) {
        T sum = ri;
        const T xi = x[i];
        sum = terms<V, T>(sum, v, [&](int j) { return x[cj[j]]; });
        if (F64) sum += xi * d;
        T z = sum / d;
        if (row) x[i] = z;
        if (spoilt(sum)) {  // (after the store, which the next step waits for)
          sum = ri;
#pragma unroll 1
          for (int j = 0; j < kSlots; ++j) {
            const int32_t c = L.col[(int64_t)j * L.n + i];
            sum -= (T)L.val[(int64_t)j * L.n + i] * (c == i ? xi : x[c]);
          }
          if (F64) sum += xi * d;
          z = sum / d;
          if (row) x[i] = z;
        }
        if (s >= rz_from) {
          double p = 0.0;
          if (row) p = F64 ? (double)(ri * z) : A.r64[i] * (double)z;
#pragma unroll
          for (int off = 32; off > 0; off >>= 1) p += __shfl_down(p, off, 64);
          if (lane == 0) A.rz[tab[1][nc] - tile1 + (t - tile0)] = p;
        }
        next();
        due = true;
      }
    }
    lds_barrier();

    if (visit < A.nlev - 1) {  // residual at the rows that the next level takes
      T *const rc = lds + A.lev[l + 1].ro;
      for (int k = threadIdx.x; k < L.nc; k += 64 * kTailWaves) {
        const int f = L.f2c[k];
        T ax = (T)0;
        const BufView val = column_view(L.val, kSlots * L.n * sizeof(V));
        const BufView col = column_view(L.col, kSlots * L.n * 4);
        V a[kSlots];
        int32_t cs[kSlots];
#pragma unroll
        for (int j = 0; j < kSlots; ++j) cs[j] = column_at<int32_t>(col, j, L.n, f);
#pragma unroll
        for (int j = 0; j < kSlots; ++j) a[j] = column_at<V>(val, j, L.n, f);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
          if (j % 9 == 0) __builtin_amdgcn_sched_barrier(0);
          ax += (T)a[j] * x[cs[j]];
        }
        if (!F64) ax += L.diag[f] * x[f];
        rc[k] = lds[L.ro + f] - ax;
      }
      lds_barrier();
    }
  }
  for (int i = threadIdx.x; i < A.lev[0].n; i += 64 * kTailWaves)
    A.x[(int64_t)i * A.stride + blockIdx.x] = lds[A.lev[0].xo + i];
}

// Lets a kernel ask for kTailLds on the current device, once.  The limit belongs
// to the function, for every problem and thread: with each launch's own size,
// one thread could lower it between another's setting and launch.
template <class V, class T>
void allow_lds() {
  static std::atomic<uint64_t> done{0};  // devices
  int dev = 0;
  HPCGX_HIP(hipGetDevice(&dev));
  const uint64_t bit = dev < 64 ? (uint64_t)1 << dev : 0;
  if (done.load() & bit) return;
  HPCGX_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(k_tail<V, T>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kTailLds));
  done.fetch_or(bit);
}

template <class V, class T, class F>
bool tail(const Problem &P, int l0, int columns, const T *r, T *x, double *rz,
          const double *r64, hipStream_t s, F &&fields) {
  TailArgs<V, T> A = {};
  A.nlev = P.nlevels - l0;
  A.stride = columns;
  A.r = r;
  A.x = x;
  A.rz = rz;
  A.r64 = r64;
  int at = 0;
  for (int k = 0; k < A.nlev; ++k) {
    const Level &L = P.L[l0 + k];
    if (L.n > kTailRows || L.n < 1 || L.ncolors < 1 || L.ncolors > kTailColors ||
        (L.wave && P.use_wave))
      return false;
    TailLevel<V, T> &D = A.lev[k];
    D.n = (int)L.n;
    D.ncolors = L.ncolors;
    D.nc = k + 1 < A.nlev ? (int)L.nc : 0;
    D.col = L.col;
    D.f2c = L.f2c;
    D.trec = use_col16(P, L) ? L.trec : nullptr;
    fields(L, D);
    for (int c = 0; c <= L.ncolors; ++c) {
      if (c && L.color_ptr[c] - L.color_ptr[c - 1] > kTailWaves * kTile) return false;
      D.cptr[c] = (int)L.color_ptr[c];
      D.ctile[c] = L.color_tile[c];
    }
    D.xo = at;
    D.ro = at + D.n;
    at += 2 * D.n;
  }
  const size_t bytes = sizeof(T) * (size_t)at;
  if (bytes > kTailLds) return false;
  if (bytes > 32768) allow_lds<V, T>();  // (what any kernel may ask for)
  k_tail<V, T><<<(unsigned)columns, 64 * kTailWaves, bytes, s>>>(A);
  HPCGX_LAUNCHED();
  return true;
}
}  // namespace

bool launch_tail(const Problem &P, int l, const double *r, double *x, hipStream_t s, double *rz) {
  if (!P.use_tail || (P.L[l].finest && P.klog.on)) return false;
  return tail<double, double>(P, l, 1, r, x, rz, nullptr, s, [](const Level &L, auto &D) {
    D.val = L.val;
    D.diag = L.diag;
  });
}

bool launch_tail32(const Problem &P, int l, const float *r, float *x, hipStream_t s, double *rz,
                   const double *r64, int columns) {
  if (!P.use_tail) return false;
  return tail<_Float16, float>(P, l, columns, r, x, rz, r64, s, [](const Level &L, auto &D) {
    D.val = L.val16;
    D.diag = L.diag32;
  });
}

}  // namespace hpcgx
