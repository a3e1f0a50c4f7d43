// lex.hip -- the reference-order (lexicographic) Gauss-Seidel sweeps as two
// launches per symmetric sweep.
//
// The level schedule (rows of hyperplane s of the dependency DAG depend only
// on lower hyperplanes) run as one launch per hyperplane is bound by the
// launches and by memory latency: at 256^3 a V-cycle is 13400 launches of a
// few thousand rows each, whose entries lie scattered over the colour-ordered
// ELL (one 64-byte sector per 8-byte value): 438 ms.
//
// Here natural rows are cut into panels of consecutive rows (one grid plane,
// or as many rows as the matrix is wide), so that a row couples only to its
// own panel and the two next to it.  One workgroup owns one panel and walks
// its hyperplanes in order, with a workgroup barrier between them; it waits
// for the panel before it (after it in the backward sweep) only until that
// panel has finished the lower (higher) hyperplanes.  That wait goes one way,
// so the panels form a pipeline: the cross-workgroup latency is paid once per
// panel, not once per hyperplane.  In the forward sweep a row of hyperplane s
// reads updated x only from rows of lower hyperplanes, all of them finished,
// and old x only from rows of higher ones, which wait for it (the pattern is
// symmetric); the backward sweep mirrors this.  So every row meets exactly
// the values the sequential sweep gives it.
//
// The matrix is copied once into that order (LexPlan): rows by panel,
// hyperplane and natural row; entries of a chunk of at most 64 rows (one
// wavefront) stored slot by slot, the chunk's slots aligned by natural column
// offset, so that both the stored entries and the gathered x of a wavefront
// are consecutive.  x and r are permuted into the same order for the sweep.
//
// Measured (MI355X, one V-cycle in reference order): 256^3 439.2 -> 24.4 ms,
// 64x48x32 21.7 -> 2.54 ms (the first, which builds the copy, 155 and 5.1 ms).
// What bounds it now is the chain of hyperplanes:
// about 1.1 us a step (one wavefront a panel) to 1.5 us (two), for gathers
// behind the barrier, 27 dependent subtractions and a division, over
// (hyperplanes of a panel) + 7 (panels - 1) steps: each panel starts four
// hyperplanes, two steps of publishing and one of look-ahead after the last.
// Joining several planes into one panel (fewer hops, more wavefronts sharing a
// CU's L1) measured slower, 30 ms (two planes) and 33 ms (four) against 24.5
// at 256^3, as did matrix loads two or three steps ahead instead of one
// (24.5 against 23.8 ms; the 63 loads a wavefront may have in flight cap it).
#include <algorithm>
#include <climits>

#include "internal.hpp"

namespace hpcgx {
namespace {

constexpr int kLexWaves = 4;               // wavefronts per workgroup, at most
constexpr int kLexPad = 32;                // progress counters 128 bytes apart
constexpr int64_t kLexRows = 256;          // see build_lex
constexpr int64_t kLexWide = 6;            // see try_lex
constexpr int kLexAhead = 1;               // steps the matrix loads run ahead
constexpr int kLexIn = 4, kLexOut = 9;     // slots of the own and of a neighbour panel
static_assert(2 * kLexOut + 2 * kLexIn + 1 == kSlots, "slot groups");
constexpr int kLexStore = kSlots + 1;      // values stored per row
constexpr int kLexEdge = 64;               // rows of 0 before and after the copy of x
constexpr int kLexRing = 2048;             // fresh x values held in LDS
constexpr int kLexReach = kLexRing - 64 * kLexWaves - 64;  // furthest fresh row
// The wait that a sweep's progress rests on (k_lex_sweep): vector memory
// operations that may still be outstanding when a step ends.
constexpr int kLexLoads = kLexStore / 2 + 2 + (kSlots - kLexIn - 1) + 1;  // of one step
constexpr int kLexPinned = (kSlots - kLexIn - 1) + 2;  // those of x and of the neighbour's progress
constexpr int kLexWait = kLexLoads + 3;  // and a step's store, the progress, the last store
static_assert(kLexWait <= 2 * kLexPinned && kLexWait < 63, "covers the stores of two steps before");

inline unsigned grid_for(int64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }
__device__ inline int64_t gtid() { return (int64_t)blockIdx.x * blockDim.x + threadIdx.x; }

typedef double f64x2 __attribute__((ext_vector_type(2)));

template <bool STREAM, class T>
__device__ inline T mload(const T *p) {
  if (STREAM) return __builtin_nontemporal_load(p);
  return *p;
}
// x of another workgroup's rows: device-coherent, as in the wavefront sweep
// (kernels.hip): served past the per-XCD L2.
__device__ inline double xload(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void xstore(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline unsigned pload(const unsigned *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Panel p holds the natural rows [bound[p], bound[p + 1]).  FIND: the first and
// last hyperplane of each panel, span[2 p] and span[2 p + 1].  Else
// key[natural row] = first[panel] + hyperplane: the panel's own hyperplanes
// only, as a panel meets few of a long grid's.
template <bool FIND>
__global__ __launch_bounds__(kBlock) void k_lex_key(int64_t n, int nsched, int npanels,
                                                    const int64_t *__restrict__ bound,
                                                    const int64_t *__restrict__ level_ptr,
                                                    const int32_t *__restrict__ level_rows,
                                                    const int32_t *__restrict__ iperm,
                                                    int32_t *span,
                                                    const int32_t *__restrict__ first,
                                                    int32_t *__restrict__ key) {
  const int64_t k = gtid();
  if (k >= n) return;
  int lo = 0, hi = nsched - 1;  // last hyperplane with level_ptr <= k
  while (lo < hi) {
    const int mid = (lo + hi + 1) / 2;
    if (level_ptr[mid] <= k) lo = mid; else hi = mid - 1;
  }
  const int64_t g = iperm[level_rows[k]];
  int a = 0, b = npanels - 1;
  while (a < b) {
    const int mid = (a + b + 1) / 2;
    if (bound[mid] <= g) a = mid; else b = mid - 1;
  }
  if (FIND) {
    if (span[2 * a] > lo) atomicMin(&span[2 * a], lo);
    if (span[2 * a + 1] < lo) atomicMax(&span[2 * a + 1], lo);
  } else {
    key[g] = first[a] + lo;
  }
}

// row[k] = device row of position k, pos[device row] = k
__global__ __launch_bounds__(kBlock) void k_lex_rows(int64_t n, const int32_t *__restrict__ order,
                                                     const int32_t *__restrict__ perm,
                                                     int32_t *__restrict__ row,
                                                     int32_t *__restrict__ pos) {
  const int64_t k = gtid();
  if (k >= n) return;
  const int32_t i = perm[order[k]];
  row[k] = i;
  pos[i] = (int32_t)k;
}

__device__ inline int wave_min(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, __shfl_xor(v, o, 64));
  return v;
}

// Slot j of row q of a chunk of cnt rows from `start`: two slots side by side
// per row (16-byte loads), the diagonal again in slot kSlots.
__device__ inline int64_t lex_at(int32_t start, int cnt, int j, int q) {
  return (int64_t)start * kLexStore + ((int64_t)(j / 2) * cnt + q) * 2 + j % 2;
}

__device__ inline int wave_max(int v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
  return v;
}

// A chunk of a plan: rows [start, start + cnt) of a panel that holds [pb, pe);
// its and its neighbour panels' rows are [lo, hi).
struct LexChunk {
  int32_t start, cnt, pb, pe, lo, hi;
};
__device__ inline LexChunk lex_chunk(int64_t q, const LexRec *recs, const int32_t *panel_of,
                                     const int64_t *pstart, int npanels) {
  const int p = panel_of[q];
  const int32_t pb = (int32_t)pstart[p], pe = (int32_t)pstart[p + 1];
  return LexChunk{recs[q].start, recs[q].cnt, pb, pe, p > 0 ? (int32_t)pstart[p - 1] : pb,
                  p + 1 < npanels ? (int32_t)pstart[p + 2] : pe};
}

// Copies one chunk's rows (one wavefront).  Where it can, the chunk's slots
// are aligned by natural column offset (repeated wavefront minimum of each
// row's next offset, as k_tile_layout does) into five groups that keep the
// ascending order: kLexOut slots for the panel before, kLexIn for lower rows
// of its own panel, the diagonal, kLexIn for upper rows, kLexOut for the panel
// after; a slot's column must be one base plus the row's place in the chunk
// (rows of a hyperplane and their neighbours are consecutive in this order).  A
// row without the slot's offset gets the value 0 there.  Chunks that do not fit
// (offsets that do not ascend, stored zeros, more offsets or
// other couplings, rows further back than the ring of fresh x holds) keep the
// device slots and 32-bit columns (k_lex_cols).  Bit 0 of *found is set when a
// column lies further away than the next panel, bit 1 when a chunk does not fit;
// joint[p] when panels p - 1 and p couple.
__global__ __launch_bounds__(kBlock) void k_lex_fill(
    int64_t nrec, int64_t n, LexRec *recs, const int32_t *__restrict__ panel_of,
    const int64_t *__restrict__ pstart, int npanels, const int32_t *__restrict__ row,
    const int32_t *__restrict__ pos, const int32_t *__restrict__ iperm,
    const int32_t *__restrict__ col, const double *__restrict__ val,
    const double *__restrict__ diag, const uint8_t *__restrict__ dslot,
    const uint8_t *__restrict__ nnz_row, double *__restrict__ lval, int32_t *__restrict__ ldpos,
    int *found, int *joint) {
  const int64_t q = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (q >= nrec) return;  // whole wavefronts
  const LexChunk C = lex_chunk(q, recs, panel_of, pstart, npanels);
  const int cnt = C.cnt;
  const int lane = threadIdx.x & 63;
  const int32_t start = C.start, pb = C.pb, pe = C.pe;
  if (lane < kSlots) recs[q].base[lane] = (uint32_t)(start + kLexEdge) << 3;
  if (cnt == 0) return;
  const bool live = lane < cnt;
  const int32_t k = start + (live ? lane : 0);
  const int64_t i = row[k];
  const int32_t g = iperm[i];
  // the row's entries, in slot order: ascending offsets and no stored zeros?
  int m = 0, last = INT_MIN, ds = 0;
  bool plain = true, far = false, before = false, after = false;
  for (int j = 0; j < kSlots; ++j) {
    if (val[(int64_t)j * n + i] == 0.0) continue;
    const int32_t cd = col[(int64_t)j * n + i];
    const int o = iperm[cd] - g;
    const int32_t c = pos[cd];
    plain = plain && (m == 0 || o > last);
    far = far || c < C.lo || c >= C.hi;
    before = before || c < pb;
    after = after || c >= pe;
    last = o;
    ++m;
  }
  if (live && far) atomicOr(found, 1);
  if (__ballot(live && before) && lane == 0) joint[panel_of[q]] = 1;
  if (__ballot(live && after) && lane == 0) joint[panel_of[q] + 1] = 1;
  plain = plain && m == nnz_row[i];
  bool fits = __ballot(live && !plain) == 0ull;
  // two passes over the chunk's distinct offsets: count each group's, then
  // place them
  const int first[6] = {0, kLexOut, kLexOut + kLexIn, kLexOut + kLexIn + 1,
                        kLexOut + 2 * kLexIn + 1, kSlots};
  int used[5] = {0, 0, 0, 0, 0}, place[5];
  if (fits && live)
    for (int u = 0; u < kSlots; ++u) lval[lex_at(start, cnt, u, lane)] = 0.0;
  for (int pass = 0; pass < 2 && fits; ++pass) {
    int e = 0;
    for (;;) {
      while (e < kSlots && val[(int64_t)e * n + i] == 0.0) ++e;
      const int32_t cd = e < kSlots ? col[(int64_t)e * n + i] : 0;
      const int head = live && e < kSlots ? iperm[cd] - g : INT_MAX;
      const int mn = wave_min(head);
      if (mn == INT_MAX) break;
      const bool has = head == mn;
      const int32_t c = has ? pos[cd] : 0;
      const int grp = !has ? 0 : c < pb ? 0 : c >= pe ? 4 : c < k ? 1 : c > k ? 3 : 2;
      // one group and one base for all rows that have the offset; fresh x of
      // the own panel (groups 1 and 3) near enough for the ring
      const int g0 = wave_min(has ? grp : INT_MAX), g1 = wave_max(has ? grp : INT_MIN);
      const int b0 = wave_min(has ? c - lane : INT_MAX), b1 = wave_max(has ? c - lane : INT_MIN);
      const int away = wave_max(has && (grp == 1 || grp == 3) ? abs(c - k) : 0);
      fits = g0 == g1 && b0 == b1 && away <= kLexReach;
      if (!fits) break;
      if (pass == 0) {
        ++used[g0];
      } else {
        const int slot = place[g0]++;
        if (has) {
          lval[lex_at(start, cnt, slot, lane)] = val[(int64_t)e * n + i];
          if (grp == 2) ds = slot;
        }
        if (lane == 0) recs[q].base[slot] = (uint32_t)(b0 + kLexEdge) << 3;
      }
      if (has) ++e;
    }
    if (pass == 0 && fits) {
      for (int u = 0; u < 5; ++u) {
        place[u] = first[u];
        fits = fits && used[u] <= first[u + 1] - first[u];
      }
    }
  }
  if (!fits && live) {
    ds = dslot[i];  // (not by its value, which may be 0 until it is replaced)
    for (int u = 0; u < kSlots; ++u)
      lval[lex_at(start, cnt, u, lane)] = val[(int64_t)u * n + i];
  }
  if (live) {
    lval[lex_at(start, cnt, kSlots, lane)] = diag[i];
    ldpos[k] = ds;
  }
  if (lane == 0) {
    recs[q].general = fits ? 0u : 1u;
    if (!fits) atomicOr(found, 2);
  }
}

// No waiting where two panels do not couple (the last plane of one problem of a
// fleet and the first of the next).
__global__ __launch_bounds__(kBlock) void k_lex_apart(int64_t nrec, LexRec *recs,
                                                      const int32_t *__restrict__ panel_of,
                                                      const int *__restrict__ joint) {
  const int64_t q = gtid();
  if (q >= nrec) return;
  const int p = panel_of[q];
  if (!joint[p]) recs[q].need[0] = 0;
  if (!joint[p + 1]) recs[q].need[1] = 0;
}

// The 32-bit columns of the chunks that k_lex_fill marked general.
__global__ __launch_bounds__(kBlock) void k_lex_cols(
    int64_t nrec, int64_t n, const LexRec *recs, const int32_t *__restrict__ panel_of,
    const int64_t *__restrict__ pstart, int npanels, const int32_t *__restrict__ row,
    const int32_t *__restrict__ pos, const int32_t *__restrict__ col,
    const double *__restrict__ val, int32_t *__restrict__ lcol) {
  const int64_t q = (int64_t)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (q >= nrec) return;
  const LexChunk C = lex_chunk(q, recs, panel_of, pstart, npanels);
  const int lane = threadIdx.x & 63;
  if (!recs[q].general || lane >= C.cnt) return;
  const int32_t k = C.start + lane;
  const int64_t i = row[k];
  for (int u = 0; u < kSlots; ++u) {
    int32_t c = pos[col[(int64_t)u * n + i]];
    // an unused slot's column need not be near: the row's own x there
    if (val[(int64_t)u * n + i] == 0.0 && (c < C.lo || c >= C.hi)) c = k;
    lcol[(int64_t)C.start * kSlots + (int64_t)u * C.cnt + lane] = c;
  }
}

__global__ __launch_bounds__(kBlock) void k_lex_zero(int64_t n, double *x) {
  const int64_t i = gtid();
  if (i < n) x[i] = 0.0;
}

// x and r into the sweep's order; clears both sweeps' progress counters.  Where
// the level's diagonal has been replaced since the copy took its own (*taken is
// behind *gen, both counted on the device, so that a replacement replayed from
// a graph counts too), it goes into the copy first: slot ldpos of each row and
// the diagonal's own.
__global__ __launch_bounds__(kBlock) void k_lex_in(
    int64_t n, const int32_t *__restrict__ row, const double *__restrict__ r,
    const double *__restrict__ x, double *__restrict__ lr, double *__restrict__ lx,
    unsigned *prog, int64_t nprog, const unsigned *gen, const unsigned *taken, int64_t nrec,
    const LexRec *__restrict__ recs, const int32_t *__restrict__ ldpos,
    const double *__restrict__ diag, double *__restrict__ lval) {
  const int64_t k = gtid();
  if (*gen != *taken) {
    const int lane = threadIdx.x & 63;
    const int64_t waves = (int64_t)gridDim.x * (kBlock / 64);
    for (int64_t q = k / 64; q < nrec; q += waves) {
      const int cnt = recs[q].cnt;
      const int32_t start = recs[q].start;
      if (lane >= cnt) continue;
      const double v = diag[row[start + lane]];
      lval[lex_at(start, cnt, ldpos[start + lane], lane)] = v;
      lval[lex_at(start, cnt, kSlots, lane)] = v;
    }
  }
  if (k < nprog) prog[k] = 0u;
  if (k >= n) return;
  const int32_t i = row[k];
  lr[k] = r[i];
  lx[k] = x[i];
}

__global__ __launch_bounds__(kBlock) void k_lex_out(int64_t n, const int32_t *__restrict__ pos,
                                                    const double *__restrict__ lx,
                                                    double *__restrict__ x, const unsigned *gen,
                                                    unsigned *taken) {
  const int64_t i = gtid();
  if (i == 0) *taken = *gen;
  if (i < n) x[i] = lx[pos[i]];
}

// One sweep direction.  Workgroup order comes from a ticket, so a workgroup
// only ever waits for panels whose workgroups have already started; a wait
// that exceeds `polls` polls sets *err and gives up, as all later ones do,
// and the sweep ends with wrong values instead of hanging (check_status).
//
// A step's loads run ahead of it, so that between two barriers only the chain
// through the rows just finished remains: values, right-hand side, diagonal
// and old x kLexAhead steps ahead; x of the other panels and of rows not yet
// reached (neither changes before the step) one step ahead, after the wait
// for the neighbour panel; x of the own panel's fresh rows from a ring in LDS.
//
// Progress: counter p holds the steps of panel p whose x stores have
// completed.  Vector memory operations of a wavefront complete in order, and
// every wavefront ends every step, with rows in it or without, with a wait that
// leaves the last kLexWait of them outstanding.  Between a store of step k and
// the end of step k + 2 lie the loads that steps k + 1 and k + 2 issue
// unconditionally; the compiler moves none of those of x or of the neighbour's
// progress (kLexPinned a step) over the waits, which clobber memory.  They are
// more than kLexWait, so after the barrier that ends step k + 2 the stores of
// step k have been acknowledged for every wavefront, and step k is published.
// The wait costs the chain of steps nothing: what it waits for besides, the
// loads that step k + 1 issued, step k + 2 has used.
template <bool STREAM, int DIR>
__global__ __launch_bounds__(64 * kLexWaves) void k_lex_sweep(
    int npanels, int waves, const LexRec *__restrict__ recs, const int32_t *__restrict__ sptr,
    const int64_t *__restrict__ pstart, const double *__restrict__ lval,
    const int32_t *__restrict__ lcol, const double *__restrict__ r, double *x, unsigned *prog,
    unsigned polls, int *err) {
  __shared__ double ring[kLexRing];
  __shared__ int s_ticket;
  // rows without an entry in a fresh slot read the ring too (times 0)
  for (int k = threadIdx.x; k < kLexRing; k += blockDim.x) ring[k] = 0.0;
  if (threadIdx.x == 0) s_ticket = (int)atomicAdd(prog, 1u);
  __syncthreads();
  const int q = __builtin_amdgcn_readfirstlane(s_ticket);
  if (q >= npanels) return;
  const int p = DIR == 0 ? q : npanels - 1 - q;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t lane = threadIdx.x & 63, lane8 = lane * 8u;
  const int s0 = sptr[p], nsteps = sptr[p + 1] - s0;
  const uint32_t pb = ((uint32_t)pstart[p] + kLexEdge) << 3,
                 pe = ((uint32_t)pstart[p + 1] + kLexEdge) << 3;
  unsigned *mine = prog + (int64_t)(1 + p) * kLexPad;
  const unsigned *nbr = q > 0 ? (DIR == 0 ? mine - kLexPad : mine + kLexPad) : mine;
  unsigned seen = q > 0 ? 0u : ~0u;

  struct Mat { f64x2 v[kLexStore / 2]; double r, o; };  // values and diagonal; b, old x
  struct Gat { double x[kSlots]; uint32_t f[kLexIn], general; };  // x by slot; ring offsets
  constexpr int kFresh = DIR == 0 ? kLexOut : kLexOut + kLexIn + 1;  // first fresh slot
  constexpr int kDiag = kLexOut + kLexIn;
  constexpr int kOther = DIR == 0 ? 0 : kSlots - kLexOut;  // first slot of the neighbour panel
  // byte offsets of x count from kLexEdge rows before its first
  auto xat = [&](uint32_t off) {
    return reinterpret_cast<double *>(reinterpret_cast<char *>(x - kLexEdge) + off);
  };
  auto rec = [&](int k) -> const LexRec & {  // step k of the sweep, this wavefront's chunk
    const int kk = k < nsteps ? k : nsteps - 1;
    const int st = DIR == 0 ? s0 + kk : s0 + nsteps - 1 - kk;
    return recs[(int64_t)st * waves + w];
  };
  // rows of a step: first row and their number, read kLexAhead + 2 steps ahead
  // (with both ends of the record, so that all of it is in the scalar cache
  // when the gathers need it)
  struct Span { int start, cnt; uint32_t tail; };
  auto span = [&](int k) {
    const LexRec &C = rec(k);
    return Span{C.start, k < nsteps ? C.cnt : 0, C.base[kSlots - 1]};
  };
  // Loads are issued whether or not the wavefront has rows in the step (from
  // rows it may read): a load under a condition would make every later wait
  // count on its absence.
  auto lane_of = [&](const Span &S) { return min(lane, (uint32_t)max(S.cnt, 1) - 1u); };
  auto load = [&](Mat &M, const Span &S) {
    const uint32_t ln = lane_of(S);
    const f64x2 *vp = reinterpret_cast<const f64x2 *>(lval + (int64_t)S.start * kLexStore);
#pragma unroll
    for (int j = 0; j < kLexStore / 2; ++j) {
      M.v[j] = mload<STREAM>(vp + ln);
      vp += S.cnt;
    }
    M.r = (r + S.start)[ln];
    M.o = (x + S.start)[ln];
  };
  unsigned polled = 0;  // progress of the neighbour, asked for a step earlier
  // x of step k that is not fresh, after the wait for the neighbour panel
  auto gather = [&](Gat &G, const Span &S, int k) {
    const LexRec &C = rec(k);
    const unsigned need = (unsigned)C.need[DIR];
    if (seen < need) {
      seen = max(seen, (unsigned)__builtin_amdgcn_readfirstlane(polled));
      unsigned spins = 0;
      while (seen < need) {
        seen = __builtin_amdgcn_readfirstlane(pload(nbr));
        if (++spins > polls ||
            ((spins & 1023u) == 0u &&
             __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
          if (lane == 0) atomicOr(err, 1);
          seen = ~0u;
        }
      }
    }
    // x loads stay behind the poll (the compiler; the wavefront itself issues
    // in order and the poll's branch holds it)
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    polled = pload(nbr);
#pragma unroll
    for (int j = 0; j < kSlots; ++j) {
      const uint32_t off = (j == kSlots - 1 ? S.tail : C.base[j]) + lane8;
      if (j >= kFresh && j < kFresh + kLexIn)
        G.f[j - kFresh] = off & (kLexRing * 8u - 1u);
      else if (j != kDiag)  // the diagonal slot takes the old x
        G.x[j] = j >= kOther && j < kOther + kLexOut ? xload(xat(off)) : *xat(off);
    }
    G.general = C.general;
  };
  auto finish = [&](const Span &S, double sum, double o, double d) {
    sum += o * d;
    const double z = sum / d;
    if (lane < (uint32_t)S.cnt) {
      ring[(S.start + kLexEdge + lane) & (kLexRing - 1)] = z;
      xstore(x + S.start + lane, z);
    }
  };
  auto step = [&](Mat &M, Gat &G, const Span &S) {
    // a wavefront without rows in the step goes through it as well (and stores
    // nothing): its earlier stores are acknowledged as the others' are
    if (!G.general) {
      double fresh[kLexIn];
#pragma unroll
      for (int j = 0; j < kLexIn; ++j)
        fresh[j] = *reinterpret_cast<const double *>(reinterpret_cast<const char *>(ring) +
                                                     G.f[j]);
      auto xj = [&](int j) {
        return j >= kFresh && j < kFresh + kLexIn ? fresh[j - kFresh] : j == kDiag ? M.o : G.x[j];
      };
      double sum = M.r;
#pragma unroll
      for (int j = 0; j < kSlots; ++j) sum -= M.v[j / 2][j % 2] * xj(j);
      // without the slots that the row does not use (such rows store no zeros);
      // from registers: loads here would make every later step wait for them
      if (__builtin_expect(__ballot(__builtin_amdgcn_class(sum, kNotFinite)) != 0ull, 0)) {
        sum = M.r;
#pragma unroll
        for (int j = 0; j < kSlots; ++j) {
          const double v = M.v[j / 2][j % 2];
          sum -= v * (j != kDiag && v == 0.0 ? 0.0 : xj(j));
        }
      }
      finish(S, sum, M.o, M.v[kSlots / 2][1]);
    } else {
      const uint32_t ln = lane_of(S);
      const int32_t *cp = lcol + (int64_t)S.start * kSlots;
      double sum = (r + S.start)[ln];
      uint32_t c[kSlots];
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        c[j] = ((uint32_t)cp[ln] + kLexEdge) << 3;
        cp += S.cnt;
      }
#pragma unroll
      for (int j = 0; j < kSlots; ++j) {
        const bool other = DIR == 0 ? c[j] < pb : c[j] >= pe;
        const double xc = other ? xload(xat(c[j])) : *xat(c[j]);
        sum -= lval[lex_at(S.start, S.cnt, j, ln)] * xc;
      }
      finish(S, sum, (x + S.start)[ln], lval[lex_at(S.start, S.cnt, kSlots, ln)]);
      __builtin_amdgcn_s_waitcnt(0);
    }
  };

  Mat M[kLexAhead + 1];
  Gat G[2];
  Span S[kLexAhead + 2];  // of steps k .. k + kLexAhead + 1
#pragma unroll
  for (int a = 0; a < kLexAhead + 2; ++a) S[a] = span(a);
#pragma unroll
  for (int a = 0; a < kLexAhead; ++a) load(M[a], S[a]);
  gather(G[0], S[0], 0);
  constexpr int kUnroll = 2 * (kLexAhead + 1);
  for (int k = 0; k < nsteps; k += kUnroll) {
#pragma unroll
    for (int a = 0; a < kUnroll; ++a) {
      if (k + a >= nsteps) break;
      load(M[(a + kLexAhead) % (kLexAhead + 1)], S[kLexAhead]);
      gather(G[(a + 1) & 1], S[1], k + a + 1);
      const Span next = span(k + a + kLexAhead + 2);
      step(M[a % (kLexAhead + 1)], G[a & 1], S[0]);
      asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kLexWait) : "memory");
      __syncthreads();
      if (threadIdx.x == 0 && k + a >= 2)
        __hip_atomic_store(mine, (unsigned)(k + a - 1), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
      for (int b = 0; b < kLexAhead + 1; ++b) S[b] = S[b + 1];
      S[kLexAhead + 1] = next;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");  // this wavefront's x stores are complete
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(mine, (unsigned)nsteps, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct Buf {  // device buffer freed on scope exit
  void *p = nullptr;
  explicit Buf(size_t bytes) { HPCGX_HIP(hipMalloc(&p, bytes ? bytes : 1)); }
  ~Buf() { (void)hipFree(p); }
  template <class T> T *as() const { return static_cast<T *>(p); }
};

// What the copy takes: values, x, r and three row ids, a record for each
// wavefront and step, and 32-bit columns where a chunk needs them.
double lex_bytes(int64_t n, int64_t nrec, bool cols) {
  return (double)n * (8.0 * (kLexStore + 2) + 4.0 * (3 + (cols ? kSlots : 0))) +
         (double)nrec * sizeof(LexRec);
}

// The plan with panels of natural rows [bound[p], bound[p + 1]), in at most
// `room` bytes; false when some row couples further than to the next panel.
bool try_lex(Problem &P, Level &L, LexPlan &X, const std::vector<int64_t> &bound, double room,
             hipStream_t s) {
  const int64_t n = L.n;
  const int64_t np = (int64_t)bound.size() - 1;
  std::vector<int32_t> span(2 * np);   // first and last hyperplane of a panel
  std::vector<int32_t> first(np + 1);  // key of hyperplane 0 of a panel; last: all keys
  std::vector<int64_t> kp;             // positions of (panel, hyperplane) keys
  X.row = X.mem.alloc<int32_t>(n);
  X.pos = X.mem.alloc<int32_t>(n);
  {
    Buf key(sizeof(int32_t) * n), order(sizeof(int32_t) * n),
        lptr(sizeof(int64_t) * (L.nsched + 1)), bnd(sizeof(int64_t) * bound.size()),
        spn(sizeof(int32_t) * span.size()), fst(sizeof(int32_t) * first.size());
    for (int64_t p = 0; p < np; ++p) {
      span[2 * p] = L.nsched;
      span[2 * p + 1] = -1;
    }
    HPCGX_HIP(hipMemcpyAsync(spn.p, span.data(), sizeof(int32_t) * span.size(),
                             hipMemcpyHostToDevice, s));
    HPCGX_HIP(hipMemcpyAsync(bnd.p, bound.data(), sizeof(int64_t) * bound.size(),
                             hipMemcpyHostToDevice, s));
    HPCGX_HIP(hipMemcpyAsync(lptr.p, L.level_ptr.data(), sizeof(int64_t) * (L.nsched + 1),
                             hipMemcpyHostToDevice, s));
    auto keys = [&](auto kernel) {
      kernel<<<grid_for(n), kBlock, 0, s>>>(n, L.nsched, (int)np, bnd.as<int64_t>(),
                                            lptr.as<int64_t>(), L.level_rows, L.iperm,
                                            spn.as<int32_t>(), fst.as<int32_t>(),
                                            key.as<int32_t>());
      HPCGX_LAUNCHED();
    };
    keys(k_lex_key<true>);
    HPCGX_HIP(hipMemcpyAsync(span.data(), spn.p, sizeof(int32_t) * span.size(),
                             hipMemcpyDeviceToHost, s));
    HPCGX_HIP(hipStreamSynchronize(s));
    // a grid's planes meet at most 2 n hyperplanes together
    int64_t nkeys = 0;
    for (int64_t p = 0; p < np; ++p) {
      first[p] = (int32_t)(nkeys - span[2 * p]);
      nkeys += span[2 * p + 1] - span[2 * p] + 1;
      if (nkeys > 4 * n) return false;
    }
    first[np] = (int32_t)nkeys;
    HPCGX_HIP(hipMemcpyAsync(fst.p, first.data(), sizeof(int32_t) * first.size(),
                             hipMemcpyHostToDevice, s));
    keys(k_lex_key<false>);
    kp = sort_rows_by_key(n, key.as<int32_t>(), (int)nkeys, order.as<int32_t>(), s);
    k_lex_rows<<<grid_for(n), kBlock, 0, s>>>(n, order.as<int32_t>(), L.perm, X.row, X.pos);
    HPCGX_LAUNCHED();
    HPCGX_HIP(hipStreamSynchronize(s));
  }
  // steps: at most W chunks of one hyperplane of one panel
  int64_t widest = 0;
  for (size_t b = 0; b + 1 < kp.size(); ++b) widest = std::max(widest, kp[b + 1] - kp[b]);
  const int W = (int)std::min<int64_t>(kLexWaves, (widest + 63) / 64);
  std::vector<int32_t> sptr{0}, level, panel_of;
  std::vector<int64_t> pstart;
  std::vector<LexRec> recs;
  for (int64_t p = 0; p < np; ++p) {
    pstart.push_back(kp[first[p] + span[2 * p]]);
    for (int lv = span[2 * p]; lv <= span[2 * p + 1]; ++lv) {
      const int64_t e = kp[first[p] + lv + 1];
      for (int64_t b = kp[first[p] + lv]; b < e;) {
        level.push_back(lv);
        for (int w = 0; w < W; ++w) {
          LexRec r = {};
          r.start = (int32_t)std::min<int64_t>(b, n - 1);
          r.cnt = (int32_t)std::min<int64_t>(64, e - b);
          b += r.cnt;
          recs.push_back(r);
          panel_of.push_back((int32_t)p);
        }
      }
    }
    sptr.push_back((int32_t)level.size());
  }
  pstart.push_back(n);
  // steps of the panel before below a step's hyperplane, of the one after above it
  for (int64_t p = 0; p < np; ++p) {
    int64_t f = p > 0 ? sptr[p - 1] : 0, b = p + 1 < np ? sptr[p + 2] : 0;
    for (int64_t st = sptr[p]; st < sptr[p + 1]; ++st) {
      if (p > 0)
        while (f < sptr[p] && level[f] < level[st]) ++f;
      for (int w = 0; w < W; ++w) recs[st * W + w].need[0] = p > 0 ? (int32_t)(f - sptr[p - 1]) : 0;
    }
    for (int64_t st = (int64_t)sptr[p + 1] - 1; st >= sptr[p]; --st) {
      if (p + 1 < np)
        while (b > sptr[p + 1] && level[b - 1] > level[st]) --b;
      for (int w = 0; w < W; ++w)
        recs[st * W + w].need[1] = p + 1 < np ? (int32_t)(sptr[p + 2] - b) : 0;
    }
  }
  // A panel is one workgroup's, 256 rows a step at most, and rows whose fresh
  // neighbours lie beyond the ring of x (hyperplanes of over 570 rows a panel)
  // take about 4.9 us a step; a launch of a hyperplane of hundreds to thousands
  // of rows takes 27 to 34 us, spread over the chip.  So a panel of more than
  // six steps a hyperplane is slower, ms a sweep, panels / launches: one plane
  // of 2048^2 159 / 337, of 4096^2 (5.7 steps) 679 / 731, of 6000^2 (8.3) 1483 /
  // 1175, of 8192^2 (11) 2735 / 1573.
  int64_t longest = 0;
  for (int64_t p = 0; p < np; ++p) longest = std::max<int64_t>(longest, sptr[p + 1] - sptr[p]);
  if (longest > kLexWide * L.nsched) throw Error(HPCGX_EUNSUP, "hyperplanes too wide for panels");
  X.npanels = (int)np;
  X.waves = W;
  X.nrec = (int64_t)recs.size();
  if (lex_bytes(n, X.nrec, false) > room) return false;
  X.recs = X.mem.alloc<LexRec>(recs.size());
  X.sptr = X.mem.alloc<int32_t>(sptr.size());
  X.pstart = X.mem.alloc<int64_t>(pstart.size());
  X.val = X.mem.alloc<double>((size_t)kLexStore * n);
  X.dpos = X.mem.alloc<int32_t>(n);
  X.x = X.mem.alloc<double>(n + 2 * kLexEdge) + kLexEdge;
  k_lex_zero<<<grid_for(n + 2 * kLexEdge), kBlock, 0, s>>>(n + 2 * kLexEdge, X.x - kLexEdge);
  HPCGX_LAUNCHED();
  X.r = X.mem.alloc<double>(n);
  X.nprog = (int64_t)kLexPad * (np + 1);
  X.prog = X.mem.alloc<unsigned>(2 * X.nprog);
  HPCGX_HIP(hipMemcpyAsync(X.recs, recs.data(), sizeof(LexRec) * recs.size(),
                           hipMemcpyHostToDevice, s));
  HPCGX_HIP(hipMemcpyAsync(X.sptr, sptr.data(), sizeof(int32_t) * sptr.size(),
                           hipMemcpyHostToDevice, s));
  HPCGX_HIP(hipMemcpyAsync(X.pstart, pstart.data(), sizeof(int64_t) * pstart.size(),
                           hipMemcpyHostToDevice, s));
  X.taken = X.mem.alloc<unsigned>(1);
  HPCGX_HIP(hipMemcpyAsync(X.taken, L.diag_gen, sizeof(unsigned), hipMemcpyDeviceToDevice, s));
  // (flags: what k_lex_fill found, then its joint)
  Buf pof(sizeof(int32_t) * panel_of.size()), flags(sizeof(int) * (np + 2));
  HPCGX_HIP(hipMemcpyAsync(pof.p, panel_of.data(), sizeof(int32_t) * panel_of.size(),
                           hipMemcpyHostToDevice, s));
  HPCGX_HIP(hipMemsetAsync(flags.p, 0, sizeof(int) * (np + 2), s));
  const int64_t wpb = kBlock / 64;
  const unsigned g = (unsigned)((X.nrec + wpb - 1) / wpb);
  k_lex_fill<<<g, kBlock, 0, s>>>(X.nrec, n, X.recs, pof.as<int32_t>(), X.pstart, X.npanels,
                                  X.row, X.pos, L.iperm, L.col, L.val, L.diag, L.dslot, L.nnz_row,
                                  X.val, X.dpos, flags.as<int>(), flags.as<int>() + 1);
  HPCGX_LAUNCHED();
  k_lex_apart<<<grid_for(X.nrec), kBlock, 0, s>>>(X.nrec, X.recs, pof.as<int32_t>(),
                                                  flags.as<int>() + 1);
  HPCGX_LAUNCHED();
  int found = 0;
  HPCGX_HIP(hipMemcpyAsync(&found, flags.p, sizeof found, hipMemcpyDeviceToHost, s));
  HPCGX_HIP(hipStreamSynchronize(s));
  if (found & 1) return false;
  X.col = nullptr;
  if (found & 2) {
    if (lex_bytes(n, X.nrec, true) > room) return false;
    X.col = X.mem.alloc<int32_t>((size_t)kSlots * n);
    k_lex_cols<<<g, kBlock, 0, s>>>(X.nrec, n, X.recs, pof.as<int32_t>(), X.pstart, X.npanels,
                                    X.row, X.pos, L.col, L.val, X.col);
    HPCGX_LAUNCHED();
    HPCGX_HIP(hipStreamSynchronize(s));
  }
  return true;
}

// Panels: the planes of the grids the rows come from, where known.  Else one
// panel for the whole level where a hyperplane holds few rows on average
// (kLexRows: one workgroup keeps up, and no wait crosses workgroups), or as
// many rows as the matrix is wide.  Any choice is only used if every row is
// found to couple to its neighbour panels at most; levels without one keep
// one launch per hyperplane.
void build_lex(Problem &P, int l, hipStream_t s) {
  Level &L = P.L[l];
  LexPlan &X = L.lex;
  X.tried = true;
  const int64_t n = L.n;
  // at most half of what is free
  size_t avail = 0, total = 0;
  if (hipMemGetInfo(&avail, &total) != hipSuccess) {
    (void)hipGetLastError();
    return;
  }
  const double room = 0.5 * (double)avail;
  if (lex_bytes(n, 0, false) > room) return;
  std::vector<std::vector<int64_t>> tries;
  std::vector<int64_t> planes{0};
  for (const GridPart &g : grid_parts(P, l))
    for (int z = 1; z <= g.nz; ++z) planes.push_back(g.off + (int64_t)g.nx * g.ny * z);
  bool rising = planes.back() == n;
  for (size_t k = 1; k < planes.size(); ++k) rising = rising && planes[k] > planes[k - 1];
  if (rising) tries.push_back(planes);
  if (n / std::max(1, L.nsched) <= kLexRows) {
    tries.push_back({0, n});
  } else if (L.bandwidth > 0 && 2 * L.bandwidth <= n) {
    std::vector<int64_t> even;
    for (int64_t b = 0; b < n; b += L.bandwidth) even.push_back(b);
    even.push_back(n);
    tries.push_back(even);
  }
  for (const auto &bound : tries) {
    try {
      if (try_lex(P, L, X, bound, room, s)) {
        X.ready = true;
        return;
      }
      X.mem.clear();
    } catch (const std::exception &) {  // too wide, or no room: one launch per hyperplane
      (void)hipGetLastError();
      X.mem.clear();
      return;
    }
  }
}

// The copy's allocations, copies and waits would end a capture of other work
// under way on another stream (by any thread, in the global mode): this thread
// leaves that rule while it builds, and touches no captured stream.
struct BesideCaptures {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  BesideCaptures() { HPCGX_HIP(hipThreadExchangeStreamCaptureMode(&mode)); }
  ~BesideCaptures() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return st != hipStreamCaptureStatusNone;
}

}  // namespace

bool lex_drop(Problem &P) {
  bool any = false;
  for (int l = 0; l < P.nlevels; ++l) {
    LexPlan &X = P.L[l].lex;
    if (!X.ready) continue;
    // (captured iterations run inside calls that wait for them)
    if (X.done) HPCGX_HIP(hipEventSynchronize(X.done));
    X.mem.clear();
    X.ready = X.tried = false;
    any = true;
  }
  if (any) {
    P.graph.reset();
    P.fleet.graph.reset();
  }
  return any;
}

bool launch_symgs_lex(Problem &P, int l, const double *r, double *x, hipStream_t s) {
  Level &L = P.L[l];
  LexPlan &X = L.lex;
  // (two hyperplanes or fewer are no more launches than this path's four: 22 us
  // against 29)
  if (!P.use_lex || L.nsched < 3 || L.n >= ((int64_t)1 << 29) - 2 * kLexEdge)
    return false;
  // Under a caller's capture the copy cannot be built, and its scratch would
  // be used at replays this call cannot order; the problem's own captured
  // iterations run inside calls that own the problem's vectors anyway.
  const bool own = s && (s == P.graph.cap || s == P.fleet.graph.cap);
  if (!own && capturing(s)) return false;
  if (!X.tried && !own) {
    const BesideCaptures relaxed;
    build_lex(P, l, s);
  }
  if (!X.ready) return false;
  // one scratch per level: a sweep on another stream follows the last one
  if (!own) {
    if (!X.done)
      HPCGX_HIP(hipEventCreateWithFlags(&X.done, hipEventDisableTiming));
    else
      HPCGX_HIP(hipStreamWaitEvent(s, X.done, 0));
  }
  const int64_t n = L.n;
  k_lex_in<<<grid_for(std::max(n, 2 * X.nprog)), kBlock, 0, s>>>(n, X.row, r, x, X.r, X.x, X.prog,
                                                                 2 * X.nprog, L.diag_gen, X.taken,
                                                                 X.nrec, X.recs, X.dpos, L.diag,
                                                                 X.val);
  HPCGX_LAUNCHED();
  const dim3 g(X.npanels), b(64 * X.waves);
#define HPCGX_LEX(ST, DIR)                                                                       \
  k_lex_sweep<ST, DIR><<<g, b, 0, s>>>(X.npanels, X.waves, X.recs, X.sptr, X.pstart, X.val,      \
                                       X.col, X.r, X.x, X.prog + DIR * X.nprog, P.lex_polls,     \
                                       P.wave_err)
  if (L.stream) {
    HPCGX_LEX(true, 0);
    HPCGX_LEX(true, 1);
  } else {
    HPCGX_LEX(false, 0);
    HPCGX_LEX(false, 1);
  }
#undef HPCGX_LEX
  HPCGX_LAUNCHED();
  k_lex_out<<<grid_for(n), kBlock, 0, s>>>(n, X.pos, X.x, x, L.diag_gen, X.taken);
  HPCGX_LAUNCHED();
  if (!own) HPCGX_HIP(hipEventRecord(X.done, s));
  return true;
}

}  // namespace hpcgx
