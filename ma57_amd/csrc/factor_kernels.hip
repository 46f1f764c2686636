// factor_kernels.hip -- gfx950 kernels of the multifrontal numeric
// factorization: front reset, assembly (zero + value scatter + extend-add),
// small-front Bunch-Kaufman in LDS, and the large-front panel path (panel
// pivoting on the eligible rows, row-parallel multipliers for the remaining
// rows, FP64 MFMA symmetric rank-p trailing update).
//
// Pivot decision logic follows the reference's DenseLDLT::factor
// (include/symla/dense_kernel.hpp:585-792) and DenseLDLT::factorStatic
// (dense_kernel.hpp:962-1035); see the comments at each step.
#include <climits>

#include "device.hpp"
#include "kernels.hpp"

#include <cfloat>
#include <cmath>
#include <type_traits>
#include <utility>

namespace symla_hip {

namespace {

constexpr double kAlpha = 0.64038820320220756872767623199676;  // (1 + sqrt(17)) / 8, dense_kernel.hpp:400

__device__ inline double bitsToDouble(unsigned long long b) { return __longlong_as_double(static_cast<long long>(b)); }
__device__ inline unsigned long long doubleToBits(double d) {
  return static_cast<unsigned long long>(__double_as_longlong(d));
}
// max of non-negative doubles via the ordering of their bit patterns
__device__ inline void atomicMaxNonNeg(unsigned long long* addr, double v) {
  if (v > 0.0) atomicMax(addr, doubleToBits(v));
}

// Candidate combine for the lambda search: larger value wins; equal values
// keep the smaller row (the reference scans rows upward with a strict '>').
__device__ inline void argmaxCombine(double& v, int& i, double v2, int i2) {
  if (i2 < 0) return;
  if (i < 0 || v2 > v || (v2 == v && i2 < i)) {
    v = v2;
    i = i2;
  }
}

// Wavefront reductions of the device library (cross-lane DPP steps instead
// of LDS permutes).
extern "C" __device__ __attribute__((const)) double __ockl_wfred_max_f64(double);
extern "C" __device__ __attribute__((const)) int __ockl_wfred_min_i32(int);

// argmaxCombine over the 64 lanes of a wave (every lane active; a lane with
// no candidate holds v = 0, idx = -1): the largest value and, among lanes
// holding it, the smallest row.
__device__ inline void waveArgmax(double& v, int& idx) {
  const double wm = __ockl_wfred_max_f64(v);
  const int wi = __ockl_wfred_min_i32((idx >= 0 && v == wm) ? idx : INT_MAX);
  v = wm;
  idx = (wi == INT_MAX) ? -1 : wi;
}

template <int NT>
__device__ inline void blockArgmax(double& v, int& idx, double* sv, int* si) {
  waveArgmax(v, idx);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
    sv[w] = v;
    si[w] = idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double bv = sv[0];
    int bi = si[0];
    for (int t = 1; t < NT / 64; ++t) argmaxCombine(bv, bi, sv[t], si[t]);
    sv[NT / 64] = bv;
    si[NT / 64] = bi;
  }
  __syncthreads();
  v = sv[NT / 64];
  idx = si[NT / 64];
  __syncthreads();
}

template <int NT>
__device__ inline double blockMax(double v, double* sv) {
  v = __ockl_wfred_max_f64(v);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) sv[w] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double b = sv[0];
    for (int t = 1; t < NT / 64; ++t) b = fmax(b, sv[t]);
    sv[NT / 64] = b;
  }
  __syncthreads();
  v = sv[NT / 64];
  __syncthreads();
  return v;
}

__device__ inline void countInertia(double d, int& pos, int& neg, int& zero) {
  if (d > 0)
    ++pos;
  else if (d < 0)
    ++neg;
  else
    ++zero;
}

// Inertia of an accepted 2x2 block (dense_kernel.hpp:753-768).
__device__ inline void countInertia2(double d11, double d22, double det, int& pos, int& neg) {
  if (det < 0) {
    ++pos;
    ++neg;
  } else {
    const double tr = d11 + d22;
    if (tr > 0)
      pos += 2;
    else if (tr < 0)
      neg += 2;
    else {
      ++pos;
      ++neg;
    }
  }
}

// Static pivot (dense_kernel.hpp:982-1011): returns the pivot to use and the
// perturbation applied.
__device__ inline double staticPivot(double a_kk, int sign, double delta, double floorv, double& applied) {
  // (selects, no branches: it is on the panels' dependent chain)
  const double s = sign != 0 ? static_cast<double>(sign) : (a_kk >= 0.0 ? 1.0 : -1.0);
  const double towards = sign > 0 ? a_kk : (sign < 0 ? -a_kk : fabs(a_kk));
  const bool need = towards < floorv;  // false for NaN: such a pivot is taken as it is
  const double d = need ? a_kk + s * delta : a_kk;
  applied = need ? d - a_kk : 0.0;
  return d;
}

// Front owning flat block `b` of a batched launch: start[f] <= b < start[f+1].
__device__ inline int findSegment(const int* start, int count, int b) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= b)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

}  // namespace

// ---------------------------------------------------------------------------
// Reset per-front state for a factorization (no memset nodes: safe to record).
// ---------------------------------------------------------------------------
__global__ void k_reset_fronts(int numSN, DevFronts fd) {
  for (int s = blockIdx.x * blockDim.x + threadIdx.x; s < numSN; s += gridDim.x * blockDim.x) {
    fd.nF[s] = 0;
    fd.inertia[3 * s] = 0;
    fd.inertia[3 * s + 1] = 0;
    fd.inertia[3 * s + 2] = 0;
    fd.origMaxBits[s] = 0ull;
    fd.runMaxBits[s] = 0ull;
    fd.kcur[s] = 0;
    fd.pcount[s] = 0;
    fd.stopped[s] = 0;
    fd.cbDone[s] = 0;
    fd.pert[s] = 0.0;
    fd.npert[s] = 0;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0 && fd.schurFlops) *fd.schurFlops = 0ull;
}

__global__ void k_reset_perm(const int* list, int count, DevFronts fd) {
  if (static_cast<int>(blockIdx.x) >= count) return;
  const int s = list[blockIdx.x];
  const int m = fd.m[s];
  const int64_t io = fd.idxOff[s];
  for (int i = threadIdx.x; i < m; i += blockDim.x) fd.perm[io + i] = i;
}

// A front pointer read from the front table is generic; generic (flat)
// accesses count against the LDS wait counter too, so every LDS wait would
// also wait for them.  Front storage is global memory: this view makes the
// accesses global ones.
template <typename T>
using GlobalPtr = __attribute__((address_space(1))) T*;
template <typename T>
__device__ inline GlobalPtr<T> globalView(void* p) {
  return (GlobalPtr<T>)(p);
}

// ---------------------------------------------------------------------------
// Assembly of one tile of one front (multifrontal.hpp:498-535): A's own-column
// entries, then every child's contribution block in child order.  One wave
// owns each column of a tile, so every entry has exactly one writer and the
// summation order is fixed.  The tile's max |F| then goes into the front's
// orig_max (dense_kernel.hpp:413-415: the max over the assembled front is the
// max over its tiles).
//
// Bound by the chain of dependent loads per child (child -> its relabelling ->
// its entries) and, in large fronts, by memory traffic.  A tile is kAsmEntries
// entries in LDS (z - y columns from y, rows from w), so a front is written
// once and not read: summed in memory it is cleared, then read and written for
// each child, then read for the maximum.  The children's rows keep their order
// in the parent, so the rows and columns of a child that meet the tile are two
// runs, found by searches for 64 children at a time.  Wave v adds columns v, v + 4, ... of the
// tile: no barrier until the end.  Measured, all launches of a factorization,
// in memory -> here: 100 x 100 grid 715 -> 340 us; 53x57x59 27-point, FP32,
// 2.50 -> 1.38 ms; 192 systems at once 10.7 -> 8.5 ms; a KKT system whose top
// fronts have thousands of children 7.2 -> 4.8 ms (22 when every tile walked
// them one by one).
// ---------------------------------------------------------------------------
// First positions in [lo, hi) of the non-decreasing rel with values >= ca and
// >= cb (hi if none), for a child per lane: three probes of each search in
// flight at a time.  Called by whole waves; every lane's rel holds rel[last].
__device__ inline void lowerBounds(const int* rel, int lo, int hi, int last, int ca, int cb, int& pa, int& pb) {
  int la = lo, ha = hi, lb = lo, hb = hi;
  while (__any(la < ha || lb < hb)) {
    int qa[3], qb[3], ra[3], rb[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      qa[k] = la + (((ha - la) * (k + 1)) >> 2);
      qb[k] = lb + (((hb - lb) * (k + 1)) >> 2);
      ra[k] = rel[min(qa[k], last)];
      rb[k] = rel[min(qb[k], last)];
    }
#pragma unroll
    for (int k = 2; k >= 0; --k) {
      if (qa[k] < ha && ra[k] >= ca) ha = qa[k];
      if (qb[k] < hb && rb[k] >= cb) hb = qb[k];
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      if (qa[k] < ha && ra[k] < ca) la = max(la, qa[k] + 1);
      if (qb[k] < hb && rb[k] < cb) lb = max(lb, qb[k] + 1);
    }
  }
  pa = la;
  pb = lb;
}

// orders a wave's LDS accesses where its lanes read what others wrote
__device__ inline void waveLdsFence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The children's entries of a tile of R = 64 U rows, Q columns of a child at
// a time with every load in flight before any add; entries outside the tile
// go to the thread's own spare slot past the tile.
template <int U, int Q, typename T>
__device__ inline void assembleChildren(const DevFronts& fd, int s, int c0, int c1, int r0, int r1, T* tile) {
  constexpr int R = 64 * U;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int spare = kAsmEntries + threadIdx.x;
  const int ce = fd.childPtr[s + 1];
  for (int cg = fd.childPtr[s]; cg < ce; cg += 64) {
    // 64 children's metadata and runs at once, a child per lane: a front may
    // have thousands of small children, few of which meet the tile
    const int cl = fd.childList[min(cg + lane, ce - 1)];
    const int mcl = fd.m[cl];
    const int64_t iol = fd.idxOff[cl];
    const int* rl = fd.relmap + iol;
    int bl, al;
    lowerBounds(rl, fd.nF[cl], mcl, mcl - 1, c0, r0, bl, al);
    const bool meets = cg + lane < ce && bl < mcl && al < mcl && rl[min(bl, mcl - 1)] < c1 && rl[min(al, mcl - 1)] < r1;
    const uint64_t fl = reinterpret_cast<uint64_t>(fd.F[cl]);
    for (uint64_t cm = __ballot(meets); cm; cm &= cm - 1) {
      const int cb = __builtin_ctzll(cm);
      auto pick = [&](int x) { return __builtin_amdgcn_readlane(x, cb); };
      auto pick64 = [&](uint64_t x) {
        return static_cast<uint64_t>(static_cast<uint32_t>(pick(static_cast<int>(x)))) |
               static_cast<uint64_t>(static_cast<uint32_t>(pick(static_cast<int>(x >> 32)))) << 32;
      };
      const int mc = pick(mcl), bLo = pick(bl), aLo = pick(al);
      const GlobalPtr<T> Fc = globalView<T>(reinterpret_cast<void*>(pick64(fl)));
      const int* rel = fd.relmap + static_cast<int64_t>(pick64(static_cast<uint64_t>(iol)));
      const int rb = rel[min(bLo + lane, mc - 1)];
      int ac[U], rr[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        ac[u] = min(aLo + 64 * u + lane, mc - 1);
        rr[u] = rel[ac[u]];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (aLo + 64 * u + lane >= mc || rr[u] < r0 || rr[u] >= r1) rr[u] = -1;
      uint64_t mask = __ballot(bLo + lane < mc && rb >= c0 && rb < c1 && ((rb - c0) & 3) == wv);
      while (mask) {
        int b[Q], col[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int bit = mask ? __builtin_ctzll(mask) : 0;
          b[q] = bLo + bit;
          col[q] = mask ? __builtin_amdgcn_readlane(rb, bit) - c0 : -1;
          mask &= mask - 1;
        }
        T v[Q][U];
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int u = 0; u < U; ++u) v[q][u] = Fc[ac[u] + static_cast<size_t>(b[q]) * mc];
        int at[Q][U];
        T old[Q][U];
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int u = 0; u < U; ++u) {
            at[q][u] = (col[q] >= 0 && rr[u] >= 0 && ac[u] >= b[q]) ? col[q] * R + rr[u] - r0 : spare;
            old[q][u] = tile[at[q][u]];
          }
#pragma unroll
        for (int q = 0; q < Q; ++q)
#pragma unroll
          for (int u = 0; u < U; ++u) tile[at[q][u]] = old[q][u] + v[q][u];
      }
      waveLdsFence();
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_assemble(const int4* tasks, int ntasks, DevFronts fd,
                                                   const double* __restrict__ aVals) {
  __shared__ T tile[kAsmEntries + 256];
  __shared__ double wmax[4];
  const int task = blockIdx.x;
  if (task >= ntasks) return;
  const int4 tk = tasks[task];
  const int s = tk.x, c0 = tk.y, W = tk.z - tk.y, r0 = tk.w;
  const int m = fd.m[s];
  const int c1 = min(tk.z, m);
  const int R = kAsmEntries / W;  // 64, 128 or 256 rows
  const int r1 = min(r0 + R, m);
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;

  for (int j = wv; j < c1 - c0; j += 4)
    for (int i = lane; i < r1 - r0; i += 64) tile[j * R + i] = T(0);
  waveLdsFence();

  // A's entries of the own columns, a lane per column, eight at a time: rows
  // and values of a batch are loaded together, then added in entry order (a
  // caller's repeated entry lands on the same row and adds in turn)
  const int nc = fd.ncols[s];
  const int ja = 4 * lane + wv;
  if (ja < W && c0 + ja < min(c1, nc)) {
    const int gcol = fd.firstCol[s] + c0 + ja;
    const int64_t tb = fd.acolPtr[gcol], te = fd.acolPtr[gcol + 1];
    for (int64_t t0 = tb; t0 < te; t0 += 8) {
      int row[8];
      double av[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int64_t t = min(t0 + u, te - 1);
        row[u] = fd.aRow[t];
        av[u] = aVals[fd.aSrc[t]];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (t0 + u < te && row[u] >= r0 && row[u] < r1) tile[ja * R + row[u] - r0] += static_cast<T>(av[u]);
    }
  }
  waveLdsFence();

  if (R == 64)
    assembleChildren<1, 8>(fd, s, c0, c1, r0, r1, tile);
  else if (R == 128)
    assembleChildren<2, 8>(fd, s, c0, c1, r0, r1, tile);
  else
    assembleChildren<4, 4>(fd, s, c0, c1, r0, r1, tile);
  waveLdsFence();

  double v = 0.0;
  for (int j = c0 + wv; j < c1; j += 4)
    for (int i = r0 + lane; i < r1; i += 64)
      if (i >= j) {
        const T x = tile[(j - c0) * R + i - r0];
        F[i + static_cast<size_t>(j) * m] = x;
        v = fmax(v, fabs(static_cast<double>(x)));
      }
  v = __ockl_wfred_max_f64(v);
  if (lane == 0) wmax[wv] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) v = fmax(v, wmax[w]);
    // most tiles do not raise the maximum: look before the atomic
    if (doubleToBits(v) > __hip_atomic_load(fd.origMaxBits + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMaxNonNeg(fd.origMaxBits + s, v);
  }
}

// The same for a parent whose rows follow no order of its children's (the
// levels of a factorization whose pivots were delayed are laid out anew, one
// level at a time): columns [c0, c1) of a front straight in memory, every
// child's contribution block scanned whole.
template <typename T>
__global__ __launch_bounds__(256) void k_assemble_any(const int4* tasks, int ntasks, DevFronts fd,
                                                       const double* __restrict__ aVals) {
  const int task = blockIdx.x;
  if (task >= ntasks) return;
  const int s = tasks[task].x;
  const int c0 = tasks[task].y;
  const int m = fd.m[s];
  const int c1 = min(tasks[task].z, m);
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;

  for (int j = c0 + wv; j < c1; j += nw) {
    const GlobalPtr<T> col = F + static_cast<size_t>(j) * m;
    for (int i = j + lane; i < m; i += 64) col[i] = T(0);
  }
  __syncthreads();

  const int nc = fd.ncols[s];
  const int fc = fd.firstCol[s];
  // A's entries of the own columns, four at a time: the rows and values of a
  // batch are loaded together, then added in entry order (a caller's
  // repeated entry lands on the same row and adds in turn)
  for (int j = c0 + threadIdx.x; j < min(c1, nc); j += blockDim.x) {
    const int gcol = fc + j;
    const GlobalPtr<T> col = F + static_cast<size_t>(j) * m;
    const int64_t tb = fd.acolPtr[gcol], te = fd.acolPtr[gcol + 1];
    for (int64_t t0 = tb; t0 < te; t0 += 4) {
      int row[4];
      double av[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t t = min(t0 + u, te - 1);
        row[u] = fd.aRow[t];
        av[u] = aVals[fd.aSrc[t]];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (t0 + u < te) col[row[u]] += static_cast<T>(av[u]);
    }
  }
  __syncthreads();

  for (int ci = fd.childPtr[s]; ci < fd.childPtr[s + 1]; ++ci) {
    const int c = fd.childList[ci];
    const int mc = fd.m[c];
    const int nfc = fd.nF[c];
    const GlobalPtr<T> Fc = globalView<T>(fd.F[c]);
    const int* rel = fd.relmap + fd.idxOff[c];
    for (int b = nfc + wv; b < mc; b += nw) {
      const int lb = rel[b];
      if (lb < 0) continue;
      const GlobalPtr<T> ccol = Fc + static_cast<size_t>(b) * mc;
      // four rows per lane at a time, every load of a batch in flight before
      // any add (a skipped row reads the child's own entry (b, b) instead);
      // the relabelling is one to one, so no two rows meet in the parent
      for (int a0 = b + lane; a0 < mc; a0 += 256) {
        int la[4];
        T cv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int a = min(a0 + 64 * u, mc - 1);
          la[u] = rel[a];
          cv[u] = ccol[a];
        }
        size_t idx[4];
        bool ok[4];
        T old[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int tr = la[u] > lb ? la[u] : lb;
          const int tc = la[u] > lb ? lb : la[u];
          ok[u] = a0 + 64 * u < mc && la[u] >= 0 && tc >= c0 && tc < c1;
          idx[u] = tr + static_cast<size_t>(tc) * m;
          old[u] = ok[u] ? F[idx[u]] : T(0);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
          if (ok[u]) F[idx[u]] = old[u] + cv[u];
      }
    }
    __syncthreads();
  }

  __shared__ double wmax[4];
  double v = 0.0;
  for (int j = c0 + wv; j < c1; j += nw) {
    const GlobalPtr<T> col = F + static_cast<size_t>(j) * m;
    for (int i = j + lane; i < m; i += 64) v = fmax(v, fabs(static_cast<double>(col[i])));
  }
  v = __ockl_wfred_max_f64(v);
  if (lane == 0) wmax[wv] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < nw; ++w) v = fmax(v, wmax[w]);
    atomicMaxNonNeg(fd.origMaxBits + s, v);
  }
}

// ---------------------------------------------------------------------------
// Small fronts: the packed lower triangle lives in LDS; right-looking
// Bunch-Kaufman with the rank-1/rank-2 update applied eagerly after every
// pivot, which is the reference's panel_size = 1 schedule for fronts with
// fewer than 256 eligible columns (multifrontal.hpp:564-566).
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(kSmallThreads) void k_factor_small(const int* list, int count, DevFronts fd,
                                                                 FactorParams prm) {
  constexpr int NT = kSmallThreads;
  extern __shared__ double smem[];
  if (static_cast<int>(blockIdx.x) >= count) return;
  const int s = list[blockIdx.x];
  const int m = fd.m[s];
  const int nE = fd.nE[s];
  T* F = static_cast<T*>(fd.F[s]);
  const int64_t io = fd.idxOff[s];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nw = NT / 64;

  double* redV = smem;                                    // NT/64 + 1
  int* redI = reinterpret_cast<int*>(smem + 32);          // NT/64 + 1
  double* A = smem + 64;                                  // packed lower, m(m+1)/2
  const int npk = m * (m + 1) / 2;
  int* perm = reinterpret_cast<int*>(A + npk);            // m

  auto P = [m](int i, int j) { return j * m - (j * (j - 1)) / 2 + (i - j); };

  double om = 0.0;
  for (int j = wv; j < m; j += nw) {
    const T* col = F + static_cast<size_t>(j) * m;
    const int base = P(j, j) - j;
    for (int i = j + lane; i < m; i += 64) {
      const double v = col[i];
      A[base + i] = v;
      om = fmax(om, fabs(v));
    }
  }
  for (int i = tid; i < m; i += NT) perm[i] = i;
  __syncthreads();
  om = blockMax<NT>(om, redV);

  const bool stat = prm.staticMode != 0;
  double origMax = om;
  if (!stat && origMax < prm.zeroTol) origMax = 1.0;        // dense_kernel.hpp:414
  if (stat && origMax < prm.staticAbsFloor) origMax = 1.0;  // dense_kernel.hpp:935
  double tmax = origMax;  // thread-local contribution to running_max

  const double delta = prm.staticDelta > 0.0 ? prm.staticDelta : sqrt(DBL_EPSILON) * origMax;
  const double sfloor = fmax(prm.staticAbsFloor, prm.staticRelFloor * origMax);

  int npos = 0, nneg = 0, nzero = 0, npert = 0;
  double pert = 0.0;
  int k = 0;
  bool stopped = false;

  // symmetric interchange of positions a < b over the whole front
  auto swapSym = [&](int a, int b) {
    for (int t = tid; t < m; t += NT) {
      int x = -1, y = -1;
      if (t < a) {
        x = P(a, t);
        y = P(b, t);
      } else if (t == a) {
        x = P(a, a);
        y = P(b, b);
      } else if (t < b) {
        x = P(t, a);
        y = P(b, t);
      } else if (t > b) {
        x = P(t, a);
        y = P(t, b);
      }
      if (x >= 0) {
        const double tv = A[x];
        A[x] = A[y];
        A[y] = tv;
      }
    }
    if (tid == 0) {
      const int tp = perm[a];
      perm[a] = perm[b];
      perm[b] = tp;
    }
    __syncthreads();
  };

  // accept a 1x1 pivot at k: scale column, eager rank-1 update
  auto accept1 = [&](double d) {
    if (tid == 0) {
      fd.dDiag[io + k] = d;
      fd.dOff[io + k] = 0.0;
      fd.pkind[io + k] = 1;
    }
    countInertia(d, npos, nneg, nzero);
    tmax = fmax(tmax, fabs(d));
    const int ck = P(k, k) - k;
    for (int i = k + 1 + tid; i < m; i += NT) {
      const double c = A[ck + i];
      tmax = fmax(tmax, fabs(c));
      A[ck + i] = c / d;
    }
    __syncthreads();
    for (int j = k + 1 + wv; j < m; j += nw) {
      const double lj = A[ck + j];
      const int cj = P(j, j) - j;
      for (int i = j + lane; i < m; i += 64) {
        const double li = A[ck + i];
        const double v = fma(-(li * d), lj, A[cj + i]);
        A[cj + i] = v;
        tmax = fmax(tmax, fabs(v));
      }
    }
    __syncthreads();
    ++k;
  };

  if (stat) {
    const int* sg = prm.expectedSign;
    while (k < nE) {
      const double akk = A[P(k, k)];
      const int sign = sg ? sg[fd.frontIdx[io + k]] : 0;
      double applied;
      const double d = staticPivot(akk, sign, delta, sfloor, applied);
      if (applied != 0.0) {
        pert += fabs(applied);
        ++npert;
      }
      accept1(d);
    }
  } else {
    while (k < nE) {
      // lambda = max_{k<i<nE} |A(i,k)| at row r (dense_kernel.hpp:588-596)
      double lv = 0.0;
      int li = -1;
      {
        const int ck = P(k, k) - k;
        for (int i = k + 1 + tid; i < nE; i += NT) {
          const double v = fabs(A[ck + i]);
          if (v > 0.0) argmaxCombine(lv, li, v, i);
        }
      }
      blockArgmax<NT>(lv, li, redV, redI);
      const double akk = A[P(k, k)];
      int action;  // 0 stop, 1 1x1 at k, 2 1x1 after swap k<->r, 3 2x2 at (k, r)
      const int r = li;
      if (lv <= prm.zeroTol) {  // dense_kernel.hpp:601-616
        const double isolatedFloor = fmax(prm.zeroTol, prm.relFloor * origMax);
        action = (fabs(akk) <= isolatedFloor) ? 0 : 1;
      } else if (fabs(akk) >= kAlpha * lv) {  // :617
        action = 1;
      } else {
        double sg = 0.0;  // sigma over the eligible rows of column r, i != r (:628-633)
        for (int i = k + tid; i < nE; i += NT) {
          if (i == r) continue;
          const double v = fabs(i > r ? A[P(i, r)] : A[P(r, i)]);
          sg = fmax(sg, v);
        }
        sg = blockMax<NT>(sg, redV);
        if (fabs(akk) * sg >= kAlpha * lv * lv)  // :641-645
          action = 1;
        else if (fabs(A[P(r, r)]) >= kAlpha * sg)
          action = 2;
        else
          action = 3;
      }
      if (action == 0) {
        stopped = true;
        break;
      }
      if (action == 2) swapSym(k, r);
      if (action == 1 || action == 2) {
        accept1(A[P(k, k)]);
        continue;
      }
      // 2x2 pivot (dense_kernel.hpp:721-792)
      if (r != k + 1) swapSym(k + 1, r);
      const double d11 = A[P(k, k)];
      const double d21 = A[P(k + 1, k)];
      const double d22 = A[P(k + 1, k + 1)];
      const double det = d11 * d22 - d21 * d21;
      const double rmax = blockMax<NT>(tmax, redV);
      if (fabs(det) <= prm.zeroTol * fmax(1.0, rmax) * fmax(1.0, rmax)) {
        stopped = true;
        break;
      }
      tmax = fmax(tmax, fmax(fabs(d11), fmax(fabs(d21), fabs(d22))));
      if (tid == 0) {
        fd.dDiag[io + k] = d11;
        fd.dOff[io + k] = d21;
        fd.dDiag[io + k + 1] = d22;
        fd.dOff[io + k + 1] = 0.0;
        fd.pkind[io + k] = 2;
        fd.pkind[io + k + 1] = 0;
      }
      countInertia2(d11, d22, det, npos, nneg);
      const double inv11 = d22 / det, inv21 = -d21 / det, inv22 = d11 / det;
      const int c0 = P(k, k) - k, c1 = P(k + 1, k + 1) - (k + 1);
      for (int i = k + 2 + tid; i < m; i += NT) {
        const double a0 = A[c0 + i], a1 = A[c1 + i];
        tmax = fmax(tmax, fmax(fabs(a0), fabs(a1)));
        A[c0 + i] = a0 * inv11 + a1 * inv21;
        A[c1 + i] = a0 * inv21 + a1 * inv22;
      }
      __syncthreads();
      for (int j = k + 2 + wv; j < m; j += nw) {
        const double lj0 = A[c0 + j], lj1 = A[c1 + j];
        const int cj = P(j, j) - j;
        for (int i = j + lane; i < m; i += 64) {
          const double li0 = A[c0 + i], li1 = A[c1 + i];
          const double w0 = li0 * d11 + li1 * d21;
          const double w1 = li0 * d21 + li1 * d22;
          const double v = A[cj + i] - (w0 * lj0 + w1 * lj1);
          A[cj + i] = v;
          tmax = fmax(tmax, fabs(v));
        }
      }
      __syncthreads();
      k += 2;
    }
  }
  (void)stopped;

  // write back
  for (int j = wv; j < m; j += nw) {
    T* col = F + static_cast<size_t>(j) * m;
    const int base = P(j, j) - j;
    for (int i = j + lane; i < m; i += 64) col[i] = static_cast<T>(A[base + i]);
  }
  for (int i = tid; i < m; i += NT) fd.perm[io + i] = perm[i];
  const double rm = blockMax<NT>(tmax, redV);
  if (tid == 0) {
    fd.nF[s] = k;
    fd.inertia[3 * s] = npos;
    fd.inertia[3 * s + 1] = nneg;
    fd.inertia[3 * s + 2] = nzero;
    fd.origMaxBits[s] = doubleToBits(origMax);
    fd.runMaxBits[s] = doubleToBits(rm);
    fd.pert[s] = pert;
    fd.npert[s] = npert;
    fd.stopped[s] = (k < nE) ? 1 : 0;
    fd.kcur[s] = k;
  }
}

size_t smallFrontSmemBytes(int m) {
  return sizeof(double) * (64 + static_cast<size_t>(m) * (m + 1) / 2) + sizeof(int) * (m + 2);
}

// ---------------------------------------------------------------------------
// Building blocks of the panel kernels.
// ---------------------------------------------------------------------------
// Row values loaded in their storage type, every load issued before any is
// used: each load is unconditional (a skipped element reads the front's first
// entry, a valid address, and is zeroed afterwards), since a load under a
// branch completes before the branch joins.
template <int N, typename P, typename Off>
__device__ inline void loadWiden(double (&x)[N], P base, Off off) {
  decltype(+base[0]) raw[N];
  bool ok[N];
#pragma unroll
  for (int q = 0; q < N; ++q) {
    const int64_t o = off(q);
    ok[q] = o >= 0;
    raw[q] = base[ok[q] ? o : 0];
  }
#pragma unroll
  for (int q = 0; q < N; ++q) x[q] = ok[q] ? static_cast<double>(raw[q]) : 0.0;
}

// 1 / d for a pivot on a dependent chain: the hardware reciprocal refined by
// two Newton steps (within an ulp of the quotient), an IEEE division for
// zero, denormal and non-finite d.
__device__ inline double pivotRecip(double d) {
  const double a = fabs(d);
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  r = fma(fma(-d, r, 1.0), r, r);
  // (one branch for the wave, rarely taken)
  const bool special = !(a >= DBL_MIN && a <= DBL_MAX);
  if (__builtin_expect(__ballot(special) != 0, 0)) r = special ? 1.0 / d : r;
  return r;
}

// c / d rounded to the front's type, r the reciprocal of d: one residual step
// makes the quotient a correctly rounded one (c r alone is up to 1.5 ulp off,
// and what a column takes off the later ones is c, so the factors' backward
// error follows the multiplier's).  An FP32 multiplier hides it.  div_fixup
// gives the quotients of zero, infinite and NaN operands.
template <typename T>
__device__ inline T multiplier(double c, double d, double r) {
  double l = c * r;
  if constexpr (sizeof(T) == 8) l = __builtin_amdgcn_div_fixup(fma(fma(-l, d, c), r, l), d, c);
  return static_cast<T>(l);
}

// c / d with d on a dependent chain: one Newton step on the hardware
// reciprocal (24 bits) and the residual step; an IEEE division when d is zero
// or denormal or an operand is not finite.
__device__ inline double pivotQuot(double c, double d) {
  const double a = fabs(d);
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
  double l = c * r;
  l = fma(fma(-l, d, c), r, l);
  const bool special = !(a >= DBL_MIN && a <= DBL_MAX && fabs(c) <= DBL_MAX);
  if (__builtin_expect(__ballot(special) != 0, 0)) l = special ? c / d : l;
  return l;
}

// A double of lane `src` (the same for the whole wave) in every lane.
__device__ inline double readLane(double v, int src) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), src);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), src);
  return __hiloint2double(hi, lo);
}

template <int CTRL>
__device__ inline double dppMove(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
// Maximum over each group of 16 consecutive lanes, in all of them.
__device__ inline double max16(double v) {
  v = fmax(v, dppMove<0xB1>(v));   // lanes 1, 0, 3, 2 of a quad
  v = fmax(v, dppMove<0x4E>(v));   // lanes 2, 3, 0, 1
  v = fmax(v, dppMove<0x124>(v));  // 16-lane row rotated by 4
  v = fmax(v, dppMove<0x128>(v));  // and by 8
  return v;
}

// The panel kernels hold 16 rows x 16 panel columns as one FP64 MFMA result
// of the transposed block: lane j + 16 c, register s is row j, column
// 4 s + c.  That is also the layout of the instruction's second operand when
// its step s takes the columns 4 s .. 4 s + 3, so a solved group of four
// columns feeds the products with the later columns straight from the
// registers it was formed in.
typedef double v4d __attribute__((ext_vector_type(4)));
__device__ inline v4d mfma64(double a, double b, v4d c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// Waits for the matrix cores' results in x: 20 wait states cover an FP64
// 16x16x4 product.  The compiler keeps that distance for reads in
// straight-line code, but a register of a result that nothing reads may be
// given another value after only 11 (the late result then lands on top of
// it), and where a branch may be taken in between it can measure a read's
// distance along the longer way.  So every result of which only a part is
// used, or which is read after a branch, is settled whole.
__device__ inline void settle(v4d& x) { asm volatile("s_nop 15\n\ts_nop 3" : "+v"(x)); }
__device__ inline void settle(v4d (&x)[4]) {
  asm volatile("s_nop 15\n\ts_nop 3" : "+v"(x[0]), "+v"(x[1]), "+v"(x[2]), "+v"(x[3]));
}

// Workgroup barrier that orders LDS accesses only: stores to global memory
// stay in flight across it.
__device__ inline void ldsBarrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The four 16-lane rows of v, each in every lane's x[row].
__device__ inline void rows16(double v, double (&x)[4]) {
  uint32_t w[2] = {static_cast<uint32_t>(__double2loint(v)), static_cast<uint32_t>(__double2hiint(v))};
  uint32_t r[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const auto p = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);  // rows 0 0 2 2 and 1 1 3 3
    const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
    const auto o = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
    r[h][0] = e[0];
    r[h][1] = o[0];
    r[h][2] = e[1];
    r[h][3] = o[1];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) x[k] = __hiloint2double(static_cast<int>(r[1][k]), static_cast<int>(r[0][k]));
}

// One substitution step of a 16-column block held as above: the four columns
// of group s are solved one after the other, then the groups after it take
// x -= L x_s in one product.  `a` is the step's operand: -L(i, 4 s + k) in
// lane i + 16 k.  A column only ever reaches later ones, so an infinity or a
// NaN stays where a column-by-column substitution has it.
//
// (The inverse of the group's 4 x 4 unit block on the matrix cores in place
// of the six dependent products is as accurate only while the multipliers
// are bounded.  Static pivots on random dense fronts of 192 rows, emulated,
// componentwise backward error: 21 u, 292 u in the worst of six, against 1.8
// and 2.1 u; measured at 300 rows, with the block's rows rounded a second time
// as well: 46 and 1600 u against 1.4 and 2.0.)
template <int S>
__device__ inline void substStep(v4d& x, double a) {
  auto l = [&](int i, int k) { return readLane(a, 4 * S + i + 16 * k); };
  const int k = (threadIdx.x >> 4) & 3;
  double y[4];
  rows16(x[S], y);
  y[1] = fma(l(1, 0), y[0], y[1]);
  y[2] = fma(l(2, 1), y[1], fma(l(2, 0), y[0], y[2]));
  y[3] = fma(l(3, 2), y[2], fma(l(3, 1), y[1], fma(l(3, 0), y[0], y[3])));
  const double v = k < 2 ? (k == 0 ? y[0] : y[1]) : (k == 2 ? y[2] : y[3]);
  if constexpr (S < 3) {
    v4d d = mfma64(a, v, x);
    settle(d);
#pragma unroll
    for (int r = S + 1; r < 4; ++r) x[r] = d[r];
  }
  x[S] = v;
}

// The substitution of one 16-row tile by a 16-column block: x becomes the
// current values c_iq at each column's pivot.
__device__ inline void substTile(v4d& x, const double (&op)[4]) {
  substStep<0>(x, op[0]);
  substStep<1>(x, op[1]);
  substStep<2>(x, op[2]);
  substStep<3>(x, op[3]);
}

// 4 x 4 transpose of the 16-lane rows of four registers: row g of v[k] and
// row k of v[g] change places.
__device__ inline void transposeRows(double (&v)[4]) {
  uint32_t w[2][4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    w[0][k] = static_cast<uint32_t>(__double2loint(v[k]));
    w[1][k] = static_cast<uint32_t>(__double2hiint(v[k]));
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const auto a = __builtin_amdgcn_permlane16_swap(w[h][0], w[h][1], false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(w[h][2], w[h][3], false, false);
    const auto c = __builtin_amdgcn_permlane32_swap(a[0], b[0], false, false);
    const auto d = __builtin_amdgcn_permlane32_swap(a[1], b[1], false, false);
    w[h][0] = c[0];
    w[h][1] = d[0];
    w[h][2] = c[1];
    w[h][3] = d[1];
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = __hiloint2double(static_cast<int>(w[1][k]), static_cast<int>(w[0][k]));
}

// The same substitution of four tiles at once, with the same operations on
// every row: transposed, a lane holds the four columns of one row of one
// tile, so that the six dependent products serve four tiles and no lane
// repeats another's.
template <int S>
__device__ inline void substStep4(v4d* x, double a) {
  auto l = [&](int i, int k) { return readLane(a, 4 * S + i + 16 * k); };
  double y[4] = {x[0][S], x[1][S], x[2][S], x[3][S]};
  transposeRows(y);
  y[1] = fma(l(1, 0), y[0], y[1]);
  y[2] = fma(l(2, 1), y[1], fma(l(2, 0), y[0], y[2]));
  y[3] = fma(l(3, 2), y[2], fma(l(3, 1), y[1], fma(l(3, 0), y[0], y[3])));
  transposeRows(y);
  if constexpr (S < 3) {
    v4d d[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) d[t] = mfma64(a, y[t], x[t]);
    settle(d);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int r = S + 1; r < 4; ++r) x[t][r] = d[t][r];
  }
#pragma unroll
  for (int t = 0; t < 4; ++t) x[t][S] = y[t];
}
__device__ inline void substTiles4(v4d* x, const double (&op)[4]) {
  substStep4<0>(x, op[0]);
  substStep4<1>(x, op[1]);
  substStep4<2>(x, op[2]);
  substStep4<3>(x, op[3]);
}

// Lane J of each 16-lane group in every lane of the group.
template <int J>
__device__ inline double bcast16(double v) {
  return __longlong_as_double(__builtin_amdgcn_update_dpp(0ll, __double_as_longlong(v), 0x150 + J, 0xf, 0xf, true));
}
// a[j] += (lane j's v of each 16-lane group) * w for j = J .. J + N - 1, one
// instruction each.  A DPP operand must have been written two wait states
// before: they stand in the same asm statement as the reads, so no copy or
// reload of v by the compiler can come between.
template <int J, int N, int M>
__device__ inline void fmaBcast16(double (&a)[M], double v, double w) {
#define DPP_FMA(acc, src, mul, lane) "\n\tv_fmac_f64_dpp %" #acc ", %" #src ", %" #mul " row_newbcast:%" #lane " row_mask:0xf bank_mask:0xf"
  if constexpr (N >= 4) {
    asm("s_nop 1" DPP_FMA(0, 4, 5, 6) DPP_FMA(1, 4, 5, 7) DPP_FMA(2, 4, 5, 8) DPP_FMA(3, 4, 5, 9)
        : "+&v"(a[J]), "+&v"(a[J + 1]), "+&v"(a[J + 2]), "+&v"(a[J + 3])
        : "v"(v), "v"(w), "n"(J), "n"(J + 1), "n"(J + 2), "n"(J + 3));
    fmaBcast16<J + 4, N - 4>(a, v, w);
  } else if constexpr (N >= 2) {
    asm("s_nop 1" DPP_FMA(0, 2, 3, 4) DPP_FMA(1, 2, 3, 5)
        : "+&v"(a[J]), "+&v"(a[J + 1])
        : "v"(v), "v"(w), "n"(J), "n"(J + 1));
    fmaBcast16<J + 2, N - 2>(a, v, w);
  } else if constexpr (N == 1) {
    asm("s_nop 1" DPP_FMA(0, 1, 2, 3) : "+v"(a[J]) : "v"(v), "v"(w), "n"(J));
  }
#undef DPP_FMA
}
// a0 and a1 += (lane J's v of each 16-lane group) * b[J] for J = 0 .. 15, the
// even J into a0 and the odd ones into a1
__device__ inline void dotBcast16(double& a0, double& a1, double v, const double (&b)[16]) {
#define DPP_FMA(acc, src, mul, lane) "\n\tv_fmac_f64_dpp %" #acc ", %" #src ", %" #mul " row_newbcast:" #lane " row_mask:0xf bank_mask:0xf"
  asm("s_nop 1" DPP_FMA(0, 2, 3, 0) DPP_FMA(1, 2, 4, 1) DPP_FMA(0, 2, 5, 2) DPP_FMA(1, 2, 6, 3) DPP_FMA(0, 2, 7, 4)
      DPP_FMA(1, 2, 8, 5) DPP_FMA(0, 2, 9, 6) DPP_FMA(1, 2, 10, 7) DPP_FMA(0, 2, 11, 8) DPP_FMA(1, 2, 12, 9)
      DPP_FMA(0, 2, 13, 10) DPP_FMA(1, 2, 14, 11) DPP_FMA(0, 2, 15, 12) DPP_FMA(1, 2, 16, 13)
      DPP_FMA(0, 2, 17, 14) DPP_FMA(1, 2, 18, 15)
      : "+&v"(a0), "+&v"(a1)
      : "v"(v), "v"(b[0]), "v"(b[1]), "v"(b[2]), "v"(b[3]), "v"(b[4]), "v"(b[5]), "v"(b[6]), "v"(b[7]), "v"(b[8]),
        "v"(b[9]), "v"(b[10]), "v"(b[11]), "v"(b[12]), "v"(b[13]), "v"(b[14]), "v"(b[15]));
#undef DPP_FMA
}

template <int... I, typename Fn>
__device__ inline void unrolled(std::integer_sequence<int, I...>, Fn&& fn) {
  (fn(std::integral_constant<int, I>{}), ...);
}

// A 16 x 16 diagonal block's factorization and the operands of its
// substitution, in LDS for every wave of the workgroup.
struct Block16 {
  double op[4][64];  // step s, lane i + 16 k: -L(i, 4 s + k), zero on and above the diagonal
  double akk[16];    // current diagonal at each pivot
  double d[16], rd[16];  // the pivots (pivotOf) and their reciprocals
};

// LDL^T of a 16 x 16 block with 1x1 pivots in order, by one wave without
// barriers or branches: lane i (mod 16; the four groups work alike) holds
// row i of the lower triangle in a[], rows of a smaller block's padding those
// of the identity.  pivotOf(q, a_qq) is the pivot (for a lane's own column
// with q the lane).  Multipliers are rounded to the front's type T.  The
// chain per pivot is one quotient; a pivot row's multipliers reach the other
// rows as DPP operands of the updates, one instruction each (through lane
// reads into scalar registers, with a branch or two per pivot, a block took
// 8000 cycles).  The block's multipliers that the front keeps are these, not
// ones that the substitution forms again: all later products of the block's
// columns use these, and where static pivots make them large a second
// rounding of the same values is a backward error of its own (emulated as
// above: 17 u, 386 u at worst).
template <typename T, typename PivotOf>
__device__ inline void blockFactor16(double (&a)[16], Block16& B, PivotOf pivotOf) {
  const int lane = threadIdx.x & 63, i = lane & 15, k = lane >> 4;
  double akk = a[0];
  unrolled(std::make_integer_sequence<int, 16>{}, [&](auto qq) {
    constexpr int q = decltype(qq)::value;
    const double l = static_cast<double>(static_cast<T>(pivotQuot(a[q], pivotOf(q, bcast16<q>(a[q])))));
    const double c = -a[q];
    if (q > 0) akk = i == q ? a[q] : akk;
    fmaBcast16<q + 1, 15 - q>(a, l, c);
    a[q] = l;
  });
  const double d = pivotOf(i, akk);
  B.akk[i] = akk;  // (the four groups store the same values)
  B.d[i] = d;
  B.rd[i] = pivotRecip(d);
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const double l = k < 2 ? (k == 0 ? a[4 * s] : a[4 * s + 1]) : (k == 2 ? a[4 * s + 2] : a[4 * s + 3]);
    B.op[s][lane] = i > 4 * s + k ? -l : 0.0;
  }
}

// ---------------------------------------------------------------------------
// Large fronts.
// ---------------------------------------------------------------------------

// max|F| over the lower triangle (dense_kernel.hpp:413-415); `bpf` blocks
// per listed front.
template <typename T>
__global__ __launch_bounds__(256) void k_front_maxabs(const int* list, int count, int bpf, DevFronts fd) {
  const int f = blockIdx.x / bpf;
  if (f >= count) return;
  const int s = list[f];
  const int part = blockIdx.x % bpf;
  const int m = fd.m[s];
  const T* F = static_cast<const T*>(fd.F[s]);
  double v = 0.0;
  const int lane = threadIdx.x & 63;
  const int gw = part * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int nwTot = bpf * (blockDim.x >> 6);
  for (int j = gw; j < m; j += nwTot) {
    const T* col = F + static_cast<size_t>(j) * m;
    for (int i = j + lane; i < m; i += 64) v = fmax(v, fabs(static_cast<double>(col[i])));
  }
  for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
  if (lane == 0) atomicMaxNonNeg(fd.origMaxBits + s, v);
}

// Panel pivoting of one front: one workgroup takes the panel's (up to 64)
// pivots on the rows it holds, the eligible rows [k, nE), or every row
// [k, m) of a front that panelHoldsAllRows.  Columns not yet pivoted are
// never modified in place: the current value of a candidate column is its
// stored (pre-panel) value minus the correction of this panel's pivots, like
// the reference's setColumnRaw (dense_kernel.hpp:516-545).  Accepted pivots
// write their multipliers for the held rows; the remaining rows are solved
// by k_panel_rows.
//
// The next 16 columns from the current pivot are worked on at once.  Their
// current values are formed on the FP64 matrix cores (16 rows x 16 columns
// per tile, the panel's earlier pivots as the inner dimension), one wave
// factors the 16 x 16 diagonal block with 1x1 pivots in order, the rows
// below follow by MFMA substitution, and one reduction gives
// lambda = max |a_ik| of every column.  The pivots before the first column
// whose test |a_kk| >= alpha lambda fails are kept: the same decisions as
// pivot by pivot, up to the order of rounding.  The failing column takes the
// general step on column buffers, and the next block starts after it.
//
// What bounds it: the dependent chain (16 reciprocals per block, the
// barriers, memory round trips), then for many rows the one CU's FP64 rate:
// 64 columns of R rows take about 2048 R multiply-adds.  TPW 16-row tiles
// per wave stay in registers (128 TPW rows; the 2,048-row variant reloads some
// 64 values that do not change during the panel from scratch); TPW = 0 streams any number of
// rows eight tiles at a time, with the block's current values in the
// workspace between the test and the multipliers.  A panel of few rows
// (PanelShape::kInLds) lives in LDS from its first load to its write-back, so
// the earlier multipliers, the interchanges and the general step's columns
// cost no memory round trip.
//
// Where three blocks in turn of a panel with more than 256 rows keep few of
// their columns (kPoorBlock), columns are formed one by one on the general
// step's buffers until four in turn pass their test: a block costs the same
// whatever it keeps (75 us at 4,000 rows, 19 at 1,000).  After one poor block already, fronts with a failing column in every
// fifth lost more than they gained (192 systems, 1,024-row panels: 353 -> 422
// us; after three 365).  Random dense fronts (a failing column in every
// second), a panel of 4,000 rows: blocks throughout 3.7 ms, here 1.9 (sub-panels
// of four and eight columns before the blocks: 2.6); 2,000 rows 2.0 -> 1.1
// (1.9); 1,000 rows 1.26 -> 0.72 (1.33).
//
// Measured per panel of 64 columns (before: sub-panels of eight columns in LDS,
// each thread factoring the 8 x 8 block, rows loaded slot by slot): 30x30x30
// 27-point fronts, FP32, few failing columns, <= 128 rows 103 -> 23 us, <= 512
// rows 103 -> 54, <= 2048 rows 153 -> 107; 100x100 5-point fronts, FP64, a
// failing column in about every eight, 210 -> 98 us; dense FP64 panels that
// pass, 1,000 rows 165 -> 81, 2,000 273 -> 157, 4,000 (streamed) 620 -> 300 us.
// A block of the 5-point fronts takes about 15,000 cycles (6,000 of them the
// diagonal block), a general step 8,000.
constexpr int kPanelCols = 16;  // columns per block
constexpr int kAloneAfter = 3;  // poor blocks in turn before columns are taken one by one,
constexpr int kAloneRun = 4;    // until so many have passed in turn
template <int TPW, typename T>
struct PanelShape {
  static constexpr int kRows = 128 * TPW;
  static constexpr int kPoorBlock = TPW == 4 || TPW == 8 ? 2 : 4;  // columns kept
  // column stride in LDS: half the banks on from one column to the next, so
  // the four columns of an operand read do not collide
  static constexpr int kLd = kRows + 16;
  static constexpr bool kInLds = TPW > 0 && sizeof(T) * kRows <= 2048;
  static constexpr size_t lds() { return kInLds ? sizeof(T) * kPanel * kLd : 0; }
};
template <int TPW, typename T>
__global__ __launch_bounds__(kPanelThreads) void k_panel(const int* list, int count, DevFronts fd, FactorParams prm,
                                                          double* wsBase, const int64_t* wsOff) {
  using Shape = PanelShape<TPW, T>;
  constexpr bool kInLds = Shape::kInLds;
  constexpr int LD = Shape::kLd;
  constexpr int NT = kPanelThreads;
  constexpr int NW = NT / 64;
  constexpr int SW = kPanelCols;
  constexpr int CT = TPW > 0 ? TPW : 8;                  // tiles per wave of a chunk
  constexpr int GT = CT < 4 ? CT : (TPW >= 16 ? 2 : 4);  // tiles whose loads are in flight together
  constexpr int LR = TPW > 0 ? Shape::kRows : 1;         // rows of the column buffers kept in LDS
  constexpr bool kWide = TPW == 0 || TPW >= 4;           // columns one by one where the blocks keep few of theirs
  extern __shared__ double dynLds[];
  T* const Lp = reinterpret_cast<T*>(dynLds);  // panel column k0 + q, row k0 + i at [q * LD + i]
  __shared__ double bufK[LR], bufR[LR];        // current columns k and r of a general step, row k0 + i at [i]
  __shared__ double Wc[kInLds ? 1 : SW][kPanel + 3];  // weights of the panel's earlier pivots at the block's rows
  __shared__ double Ds[SW][SW + 1];            // diagonal block
  __shared__ Block16 blk;
  __shared__ double redM[NW][SW];              // per-wave column maxima
  __shared__ double redS[NW], redT[NW], redL[NW], redV[NW + 1];
  __shared__ int redI[NW];
  // pivot q of the panel, at [q + 1]: (D L^T)(q, row) = pdd l_q + pnx l_(q+1) + ppv l_(q-1)
  // (the neighbours: the other column of a 2x2 pivot)
  __shared__ double pdd[kPanel + 3], pnx[kPanel + 3], ppv[kPanel + 3];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  if (static_cast<int>(blockIdx.x) >= count) return;
  const int s = list[blockIdx.x];
  double* ws = wsBase + wsOff[s];
  if (fd.stopped[s]) {
    if (tid == 0) fd.pcount[s] = 0;
    return;
  }
  const int m = fd.m[s];
  const int nE = fd.nE[s];
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const int64_t io = fd.idxOff[s];
  // after a speculative step the panel started p0 pivots before kcur
  const int kc = fd.kcur[s];
  const bool sp = specFront(prm, nE);
  const int p0 = sp ? fd.pcount[s] : 0;
  const int k0 = kc - p0;
  if (kc >= nE) {
    if (tid == 0 && !sp) fd.pcount[s] = 0;
    return;
  }
  const int nbEnd = min(k0 + kPanel, nE);
  if (kc >= nbEnd) return;
  const bool allRows = panelHoldsAllRows(m, sp);
  const int rEnd = allRows ? m : nE;  // rows held: [k, rEnd)
  for (int q = tid; q < p0; q += NT) {  // the speculative step takes 1x1 pivots only
    pdd[q + 1] = fd.dDiag[io + k0 + q];
    pnx[q + 1] = 0.0;
    ppv[q + 1] = 0.0;
  }
  double* wsR = ws + nE;
  double* cbuf = ws + panelStreamOffset(m, nE, sp);  // streamed rows: current value of row i, block column j at [i + j nE]
  auto curK = [&](int i) -> double& {
    if constexpr (TPW > 0)
      return bufK[i - k0];
    else
      return ws[i];
  };
  auto curR = [&](int i) -> double& {
    if constexpr (TPW > 0)
      return bufR[i - k0];
    else
      return wsR[i];
  };
  auto at = [&](int i, int j) -> int64_t { return i + static_cast<int64_t>(j) * m; };
  // entry (i, j), i >= j: panel columns of held rows live in LDS when kInLds
  auto inLds = [&](int i, int j) { return kInLds && j >= k0 && j < k0 + kPanel && i < rEnd; };
  auto ldsAt = [&](int i, int j) { return (j - k0) * LD + (i - k0); };
  auto get = [&](int i, int j) -> T {
    if constexpr (kInLds)
      if (inLds(i, j)) return Lp[ldsAt(i, j)];
    return F[at(i, j)];
  };
  auto put = [&](int i, int j, T v) {
    if constexpr (kInLds)
      if (inLds(i, j)) {
        Lp[ldsAt(i, j)] = v;
        return;
      }
    F[at(i, j)] = v;
  };
  // panel column q at a held row
  auto panelEntry = [&](int i, int q) -> T {
    if constexpr (kInLds)
      return Lp[q * LD + (i - k0)];
    else
      return F[at(i, k0 + q)];
  };
  auto sync = [&]() {
    if constexpr (kInLds)
      ldsBarrier();
    else
      __syncthreads();
  };
  if constexpr (kInLds) {
    // load the panel, eight columns per wave, every load in flight at once
    const int pw = nbEnd - k0;
    constexpr int RB = Shape::kRows / 64;
    T v[RB][kPanel / NW];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int u = 0; u < kPanel / NW; ++u) {
        const int i = k0 + 64 * b + lane, q = wv + NW * u;
        v[b][u] = F[i < rEnd && q < pw ? at(i, k0 + q) : 0];
      }
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int u = 0; u < kPanel / NW; ++u) {
        const int i = k0 + 64 * b + lane, q = wv + NW * u;
        if (i < rEnd && q < pw) Lp[q * LD + (i - k0)] = v[b][u];
      }
  }
  sync();

  const bool stat = prm.staticMode != 0;
  double origMax = bitsToDouble(fd.origMaxBits[s]);
  if (!stat && origMax < prm.zeroTol) origMax = 1.0;
  if (stat && origMax < prm.staticAbsFloor) origMax = 1.0;
  const double isolatedFloor = fmax(prm.zeroTol, prm.relFloor * origMax);
  const double runMax0 = fmax(origMax, bitsToDouble(fd.runMaxBits[s]));
  double tmax = 0.0;
  const double delta = prm.staticDelta > 0.0 ? prm.staticDelta : sqrt(DBL_EPSILON) * origMax;
  const double sfloor = fmax(prm.staticAbsFloor, prm.staticRelFloor * origMax);

  // counts of thread 0 (general steps) and of wave 0's lanes (blocks), summed at the end
  int npos = 0, nneg = 0, nzero = 0, npert = 0;
  double pert = 0.0;
  int k = kc, p = p0;
  bool stop = false;
  bool has2 = false;       // the panel has a 2x2 pivot
  bool farStores = false;  // kInLds: an interchange has stored to global memory since the last full barrier

  // (D L^T)(q, row) for this panel's pivot q and a given row
  auto weight = [&](int q, int row) -> double {
    const double l = static_cast<double>(panelEntry(row, q));
    const double n = static_cast<double>(panelEntry(row, min(q + 1, p - 1)));
    const double v = static_cast<double>(panelEntry(row, max(q - 1, 0)));
    return pdd[q + 1] * l + (has2 ? pnx[q + 1] * n + ppv[q + 1] * v : 0.0);
  };
  // symmetric interchange of positions a < b in storage (all rows, incl. the
  // factored part and the not-fully-summed rows), the values of S turns of a
  // thread loaded before any is stored
  auto swapSym = [&](int a, int b) {
    constexpr int S = kInLds ? 1 : 4;
    for (int t0 = tid; t0 < m; t0 += S * NT) {
      T x[S], y[S];
      int i1[S], j1[S], i2[S], j2[S];
      bool ok[S];
#pragma unroll
      for (int u = 0; u < S; ++u) {
        // (a, t) and (b, t), each read from the lower triangle; (a, a) and (b, b) for t = a
        const int t = t0 + u * NT;
        ok[u] = t < m && t != b;
        i1[u] = ok[u] ? max(a, t) : 0;
        j1[u] = ok[u] ? min(a, t) : 0;
        i2[u] = ok[u] ? (t == a ? b : max(b, t)) : 0;
        j2[u] = ok[u] ? (t == a ? b : min(b, t)) : 0;
        if constexpr (kInLds) {
          const bool in1 = inLds(i1[u], j1[u]), in2 = inLds(i2[u], j2[u]);
          x[u] = Lp[in1 ? ldsAt(i1[u], j1[u]) : 0];
          y[u] = Lp[in2 ? ldsAt(i2[u], j2[u]) : 0];
          if (!in1 || !in2) {
            const T gx = F[in1 ? 0 : at(i1[u], j1[u])], gy = F[in2 ? 0 : at(i2[u], j2[u])];
            x[u] = in1 ? x[u] : gx;
            y[u] = in2 ? y[u] : gy;
          }
        } else {
          x[u] = F[at(i1[u], j1[u])];
          y[u] = F[at(i2[u], j2[u])];
        }
      }
#pragma unroll
      for (int u = 0; u < S; ++u)
        if (ok[u]) {
          put(i1[u], j1[u], y[u]);
          put(i2[u], j2[u], x[u]);
        }
    }
    if (tid == 0) {
      const int tp = fd.perm[io + a];
      fd.perm[io + a] = fd.perm[io + b];
      fd.perm[io + b] = tp;
    }
    farStores = true;
    sync();
  };
  auto setPivot = [&](int q, double d, int kind, double next, double prev) {
    fd.dDiag[io + k0 + q] = d;
    fd.dOff[io + k0 + q] = next;
    fd.pkind[io + k0 + q] = kind;
    pdd[q + 1] = d;
    pnx[q + 1] = next;
    ppv[q + 1] = prev;
  };
  // 1x1 pivot d at k with current column col(i)
  auto accept1 = [&](auto&& col, double d) {
    if (tid == 0) {
      setPivot(p, d, 1, 0.0, 0.0);
      put(k, k, static_cast<T>(d));
      countInertia(d, npos, nneg, nzero);
    }
    tmax = fmax(tmax, fabs(d));
    for (int i = k + 1 + tid; i < rEnd; i += NT) {
      const double c = col(i);
      tmax = fmax(tmax, fabs(c));
      put(i, k, static_cast<T>(c / d));
    }
    sync();
    ++k;
    ++p;
  };
  // out(i) = current column col of the held rows; returns the thread's max
  // over its eligible rows but col.  Lane q keeps the weight of pivot q; RG
  // groups of 64 rows per wave are in flight together (two where every panel
  // has rows for them).
  auto currentColumn = [&](int col, auto&& out) -> double {
    constexpr int RG = TPW == 0 || TPW >= 16 ? 2 : 1;
    const double wq = lane < p ? weight(lane, col) : 0.0;
    double v = 0.0;
    for (int i0 = k + 64 * wv; i0 < rEnd; i0 += RG * NT) {  // whole waves: the DPP operands come from every lane
      int i[RG];
      bool ok[RG];
      double raw[RG], a0[RG], a1[RG];
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        ok[g] = i0 + g * NT + lane < rEnd;
        i[g] = ok[g] ? i0 + g * NT + lane : rEnd - 1;
        raw[g] = static_cast<double>(get(max(i[g], col), min(i[g], col)));
        a0[g] = a1[g] = 0.0;
      }
#pragma unroll 1
      for (int q = 0; q < p; q += 16) {
        const double w16 = __shfl(wq, q + lr, 64);  // the weights past p are zero
        double lv[RG][16];
        if constexpr (kInLds) {
#pragma unroll
          for (int u = 0; u < 16; ++u) lv[0][u] = static_cast<double>(Lp[min(q + u, p - 1) * LD + (i[0] - k0)]);
        } else {
#pragma unroll
          for (int g = 0; g < RG; ++g)
            loadWiden<16>(lv[g], F, [&](int u) -> int64_t { return at(i[g], k0 + min(q + u, p - 1)); });
        }
#pragma unroll
        for (int g = 0; g < RG; ++g) dotBcast16(a0[g], a1[g], w16, lv[g]);
      }
#pragma unroll
      for (int g = 0; g < RG; ++g) {
        const double c = raw[g] - (a0[g] + a1[g]);
        if (ok[g]) out(i[g]) = c;
        if (ok[g] && i[g] < nE && i[g] != col) v = fmax(v, fabs(c));
      }
    }
    return v;
  };
  // one general step at pivot k (sigma test, swaps, 1x1 or 2x2, or a stop);
  // curK holds the current column k, lam = max |curK| over the eligible rows
  // below k (attained)
  auto generalStep = [&](double lam) {
    const double akk = curK(k);
    if (lam <= prm.zeroTol) {
      // dense_kernel.hpp:601-616: the block test failed on the isolated-pivot
      // floor, which NaN does not lie below
      if (fabs(akk) <= isolatedFloor)
        stop = true;
      else
        accept1([&](int i) { return curK(i); }, akk);
      return;
    }
    if (kInLds && farStores) {
      __syncthreads();  // column r may have been stored by another thread's interchange
      farStores = false;
    }
    // r: the first row that attains lambda (found by every wave for itself
    // where the column is in LDS)
    int li = INT_MAX;
    for (int i = k + 1 + (TPW > 0 ? lane : tid); i < nE; i += (TPW > 0 ? 64 : NT))
      if (fabs(curK(i)) == lam) {
        li = i;
        break;
      }
    int r = __ockl_wfred_min_i32(li);
    if constexpr (TPW == 0) {
      if (lane == 0) redI[wv] = r;
      __syncthreads();
      r = redI[0];
#pragma unroll
      for (int w = 1; w < NW; ++w) r = min(r, redI[w]);
    }
    r = __builtin_amdgcn_readfirstlane(r);
    if (r >= nE) {  // lambda is not a number: nothing to pivot on
      stop = true;
      return;
    }
    // sigma: the max of the current column r over the eligible rows but r (dense_kernel.hpp:628-633)
    double sg = currentColumn(r, curR);
    sg = __ockl_wfred_max_f64(sg);
    const double tm = __ockl_wfred_max_f64(tmax);
    if (lane == 0) {
      redS[wv] = sg;
      redT[wv] = tm;
    }
    sync();
    double rmax = runMax0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      sg = fmax(sg, redS[w]);
      rmax = fmax(rmax, redT[w]);
    }
    const double crk = curR(k), crr = curR(r);
    // the reference mirrors column r into row r, so column k's entry at row r
    // is column r's value at row k (dense_kernel.hpp:543)
    if (fabs(akk) * sg >= kAlpha * lam * lam) {
      accept1([&](int i) { return i == r ? crk : curK(i); }, akk);
      return;
    }
    if (fabs(crr) >= kAlpha * sg) {
      // 1x1 at r after the interchange with k
      swapSym(k, r);
      accept1([&](int i) { return i == r ? crk : curR(i); }, crr);
      return;
    }
    // 2x2 at (k, r): r comes to k + 1
    const double d11 = akk, d21 = crk, d22 = crr;
    const double det = d11 * d22 - d21 * d21;
    const double ck1 = curK(k + 1), cr1 = curR(k + 1);
    if (r != k + 1) swapSym(k + 1, r);
    if (fabs(det) <= prm.zeroTol * fmax(1.0, rmax) * fmax(1.0, rmax)) {
      stop = true;
      return;
    }
    tmax = fmax(tmax, fmax(fabs(d11), fmax(fabs(d21), fabs(d22))));
    if (tid == 0) {
      setPivot(p, d11, 2, d21, 0.0);
      setPivot(p + 1, d22, 0, 0.0, d21);
      put(k, k, static_cast<T>(d11));
      put(k + 1, k, static_cast<T>(d21));
      put(k + 1, k + 1, static_cast<T>(d22));
      countInertia2(d11, d22, det, npos, nneg);
    }
    const double inv11 = d22 / det, inv21 = -d21 / det, inv22 = d11 / det;
    for (int i = k + 2 + tid; i < rEnd; i += NT) {
      // row r holds what was row k + 1
      const double a0 = i == r ? ck1 : curK(i), a1 = i == r ? cr1 : curR(i);
      tmax = fmax(tmax, fmax(fabs(a0), fabs(a1)));
      put(i, k, static_cast<T>(a0 * inv11 + a1 * inv21));
      put(i, k + 1, static_cast<T>(a0 * inv21 + a1 * inv22));
    }
    sync();
    has2 = true;
    k += 2;
    p += 2;
  };

  // First row of tile t of this wave in chunk ch: tiles go to the waves in
  // turn, so all of them keep rows as the panel moves down.
  auto rowOf = [&](int ch, int t) { return k0 + 16 * ((ch * CT + t) * NW + wv); };
  // Current values of the block's columns c0 .. c0 + sw - 1 at NTL tiles (16
  // rows from row0(t)): stored values at and below the diagonal less the
  // correction of the panel's p pivots; zero above the diagonal and past rEnd.
  auto loadTiles = [&](auto& x, auto ntl, auto&& row0, int c0, int sw) {
    constexpr int NTL = decltype(ntl)::value;
    // panel column q, row `row` (any valid entry when !ok)
    auto entry = [&](int row, int q, bool ok) -> T {
      if constexpr (kInLds)
        return Lp[ok ? q * LD + (row - k0) : 0];
      else
        return F[ok ? at(row, k0 + q) : 0];
    };
    int lrL = lr;  // (see acceptChunk)
    if constexpr (TPW == 0 || TPW >= 8) asm volatile("" : "+v"(lrL));
    T raw[NTL][4];
#pragma unroll
    for (int t = 0; t < NTL; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = row0(t) + lrL, col = 4 * u + lk;
        raw[t][u] = entry(row, c0 - k0 + col, row < rEnd && col < sw && row >= c0 + col);
      }
#pragma unroll
    for (int t = 0; t < NTL; ++t)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int row = row0(t) + lrL, col = 4 * u + lk;
        x[t][u] = row < rEnd && col < sw && row >= c0 + col ? static_cast<double>(raw[t][u]) : 0.0;
      }
    // operands of 16 pivots
    T lv[NTL][4], ln[NTL][4];
    double w[4], wn[4];
    auto fetch = [&](int q0, T (&l)[NTL][4], double (&wt)[4]) {
#pragma unroll
      for (int t = 0; t < NTL; ++t)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int row = row0(t) + lrL, q = q0 + 4 * u + lk;
          l[t][u] = entry(row, q, row >= c0 && row < rEnd && q < p);
        }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = q0 + 4 * u + lk;
        if constexpr (kInLds) {
          // (columns past sw take weights that nothing uses)
          const int qc = min(q, p - 1), i = min(c0 + lr, rEnd - 1);
          wt[u] = -weight(qc, i);
        } else {
          wt[u] = -Wc[lr][q];
        }
      }
    };
    auto products = [&](int q0) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int t = 0; t < NTL; ++t) {
          const int row = row0(t) + lrL, q = q0 + 4 * u + lk;
          const double l = row >= c0 && row < rEnd && q < p ? static_cast<double>(lv[t][u]) : 0.0;
          x[t] = mfma64(w[u], l, x[t]);
        }
    };
    if constexpr (TPW == 1 || TPW == 2) {  // (with more tiles the registers are worth more)
      if (p > 0) fetch(0, ln, wn);
      for (int q0 = 0; q0 < p; q0 += 16) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          w[u] = wn[u];
#pragma unroll
          for (int t = 0; t < NTL; ++t) lv[t][u] = ln[t][u];
        }
        if (q0 + 16 < p) fetch(q0 + 16, ln, wn);
        products(q0);
      }
    } else {
      for (int q0 = 0; q0 < p; q0 += 16) {
        fetch(q0, lv, w);
        products(q0);
      }
    }
#pragma unroll
    for (int t = 0; t < NTL; ++t) settle(x[t]);
  };

  // columns that passed the first test since one failed; once two blocks in
  // turn kept few of theirs it starts at zero
  int passed = kAloneRun, poor = 0;
  while (k < nbEnd && !stop) {
    if (kWide && passed < kAloneRun) {
      double lam = __ockl_wfred_max_f64(currentColumn(k, curK));
      if (lane == 0) redL[wv] = lam;
      sync();
#pragma unroll
      for (int w = 0; w < NW; ++w) lam = fmax(lam, redL[w]);
      const double akk = curK(k);
      if (lam <= prm.zeroTol ? fabs(akk) > isolatedFloor : fabs(akk) >= kAlpha * lam) {
        accept1([&](int i) { return curK(i); }, akk);
        ++passed;
      } else {
        generalStep(lam);
        passed = 0;
      }
      continue;
    }
    const int c0 = k, sw = min(SW, nbEnd - k);
    if constexpr (!kInLds) {
      // weights of the earlier pivots at the block's rows
      for (int e = tid; e < SW * ((p + 15) & ~15); e += NT) {
        const int j = e & (SW - 1), q = e / SW;
        Wc[j][q] = (j < sw && q < p) ? weight(q, c0 + j) : 0.0;
      }
      sync();
    }
    v4d x[CT];
    // chunk ch of this wave's tiles; a group of tiles past the held rows or
    // above the block is skipped whole (zero)
    auto loadChunk = [&](int ch) {
#pragma unroll
      for (int t0 = 0; t0 < CT; t0 += GT) {
        if (rowOf(ch, t0) < rEnd && rowOf(ch, t0 + GT - 1) + 16 > c0) {
          v4d xt[GT];
          loadTiles(xt, std::integral_constant<int, GT>{}, [&](int t) { return rowOf(ch, t0 + t); }, c0, sw);
#pragma unroll
          for (int t = 0; t < GT; ++t) x[t0 + t] = xt[t];
        } else {
#pragma unroll
          for (int t = 0; t < GT; ++t) x[t0 + t] = v4d{0.0, 0.0, 0.0, 0.0};
        }
      }
    };
    if constexpr (TPW > 0) {
      loadChunk(0);
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const int i = rowOf(0, t) + lr - c0;
        if (i >= 0 && i < SW) {
#pragma unroll
          for (int u = 0; u < 4; ++u) Ds[i][4 * u + lk] = x[t][u];
        }
      }
    } else if (wv == 0) {
      v4d xd[1];
      loadTiles(xd, std::integral_constant<int, 1>{}, [&](int) { return c0; }, c0, sw);
#pragma unroll
      for (int u = 0; u < 4; ++u) Ds[lr][4 * u + lk] = xd[0][u];
    }
    sync();
    if (wv == 0) {
      double a[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) a[q] = Ds[lr][q];
#pragma unroll
      for (int q = 0; q < 16; ++q) a[q] = lr < sw ? (q <= lr ? a[q] : 0.0) : (q == lr ? 1.0 : 0.0);
      if (!stat) {
        blockFactor16<T>(a, blk, [](int, double v) { return v; });
      } else {
        const int sgn = prm.expectedSign && lr < sw ? prm.expectedSign[fd.frontIdx[io + c0 + lr]] : 0;
        blockFactor16<T>(a, blk, [&](int q, double v) {
          double applied;
          return staticPivot(v, __shfl(sgn, q, 64), delta, sfloor, applied);
        });
      }
    }
    sync();
    double op[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) op[u] = blk.op[u][lane];
    const double akk = blk.akk[lr];
    // substitution of the held rows and the maxima over the eligible rows below each pivot
    double vm[4] = {0.0, 0.0, 0.0, 0.0};
    auto solveChunk = [&](int ch) {
      constexpr int ST = CT >= 4 ? 4 : 1;  // tiles substituted together
#pragma unroll
      for (int t0 = 0; t0 < CT; t0 += ST) {
        if (rowOf(ch, t0) < rEnd && rowOf(ch, t0 + ST - 1) + 16 > c0) {
          if constexpr (ST == 4)
            substTiles4(&x[t0], op);
          else
            substTile(x[t0], op);
#pragma unroll
          for (int t = t0; t < t0 + ST; ++t) {
            const int row = rowOf(ch, t) + lr;
#pragma unroll
            for (int u = 0; u < 4; ++u)
              vm[u] = fmax(vm[u], row < nE && row > c0 + 4 * u + lk ? fabs(x[t][u]) : 0.0);
          }
        }
      }
    };
    const int nch = TPW > 0 ? 1 : (rEnd - k0 + 16 * NW * CT - 1) / (16 * NW * CT);
    if constexpr (TPW > 0) {
      solveChunk(0);
    } else {
      for (int ch = 0; ch < nch; ++ch) {
        loadChunk(ch);
        solveChunk(ch);
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          const int row = rowOf(ch, t) + lr;
          if (row >= c0 && row < rEnd) {
#pragma unroll
            for (int u = 0; u < 4; ++u) cbuf[row + static_cast<int64_t>(4 * u + lk) * nE] = x[t][u];
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double v = max16(vm[u]);
      if (lr == 0) redM[wv][4 * u + lk] = v;
    }
    sync();
    // first failing column (dense_kernel.hpp:601-618); static pivots are
    // always accepted (dense_kernel.hpp:982-1011)
    double lam = redM[0][lr];
#pragma unroll
    for (int w = 1; w < NW; ++w) lam = fmax(lam, redM[w][lr]);
    const bool pass = stat || ((lam <= prm.zeroTol) ? fabs(akk) > isolatedFloor : fabs(akk) >= kAlpha * lam);
    const unsigned long long bad = __ballot(lane < sw && !pass);
    const int qs = bad ? __ffsll(static_cast<long long>(bad)) - 1 : sw;
    // keep the columns before it: multipliers, pivots, counts
    double dc[4], rdc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      dc[u] = blk.d[4 * u + lk];
      rdc[u] = blk.rd[4 * u + lk];
    }
    // (rows from an index that the compiler cannot match with the loads': their
    // 4 CT addresses would stay in registers over the whole block)
    int lrA = lr;
    if constexpr (TPW == 0 || TPW >= 8) asm volatile("" : "+v"(lrA));
    auto acceptChunk = [&](int ch) {
#pragma unroll
      for (int t = 0; t < CT; ++t) {
        const int row0 = rowOf(ch, t), row = row0 + lrA;
        if (row0 >= rEnd || row0 + 16 <= c0) continue;
        T lt[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) lt[u] = multiplier<T>(x[t][u], dc[u], rdc[u]);
        if (row0 < c0 + sw && row0 + 16 > c0) {
          // the block's own rows keep the multipliers of its factorization
          const int i = row - c0, ic = min(max(i, 0), sw - 1);
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const T lb = static_cast<T>(-blk.op[u][ic + 16 * lk]);
            lt[u] = i == ic ? lb : lt[u];
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int q = 4 * u + lk;
          if (q < qs && row > c0 + q && row < rEnd) {
            tmax = fmax(tmax, fabs(x[t][u]));
            const T l = lt[u];
            if constexpr (kInLds)
              Lp[(c0 - k0 + q) * LD + (row - k0)] = l;
            else
              F[at(row, c0 + q)] = l;
          }
          // the failing column's current values for the general step
          if (q == qs && row >= c0 + q && row < rEnd) curK(row) = x[t][u];
        }
      }
    };
    if constexpr (TPW > 0) {
      acceptChunk(0);
    } else {
      for (int ch = 0; ch < nch; ++ch) {
#pragma unroll
        for (int t = 0; t < CT; ++t) {
          const int row = rowOf(ch, t) + lr;
#pragma unroll
          for (int u = 0; u < 4; ++u)
            x[t][u] = (row >= c0 && row < rEnd) ? cbuf[row + static_cast<int64_t>(4 * u + lk) * nE] : 0.0;
        }
        acceptChunk(ch);
      }
    }
    if (tid < qs) {
      const int q = tid;
      const double dpv = blk.d[q];
      setPivot(p + q, dpv, 1, 0.0, 0.0);
      put(k + q, k + q, static_cast<T>(dpv));
      countInertia(dpv, npos, nneg, nzero);
      tmax = fmax(tmax, fabs(dpv));
      if (stat && dpv != akk) {
        pert += fabs(dpv - akk);
        ++npert;
      }
    }
    if (kWide) {
      poor = qs < min(Shape::kPoorBlock, sw) ? poor + 1 : 0;
      if (poor == kAloneAfter) passed = poor = 0;
    }
    const double lamF = readLane(lam, min(qs, SW - 1));
    sync();
    k += qs;
    p += qs;
    if (qs < sw) generalStep(lamF);
  }

  if constexpr (kInLds) {
    ldsBarrier();
    // write the panel back: accepted columns, and the others as the interchanges left them
    const int pw = nbEnd - k0;
    for (int i0 = k0; i0 < rEnd; i0 += 64) {
      const int i = i0 + lane;
#pragma unroll
      for (int u = 0; u < kPanel / NW; ++u) {
        const int q = wv + NW * u;
        if (q < pw && i >= k0 + q && i < rEnd) F[at(i, k0 + q)] = Lp[q * LD + (i - k0)];
      }
    }
  }
  const double bm = blockMax<NT>(tmax, redV);
  if (tid < 64) {
    for (int off = 8; off > 0; off >>= 1) {  // lanes 0 .. 15 counted
      npos += __shfl_xor(npos, off, 64);
      nneg += __shfl_xor(nneg, off, 64);
      nzero += __shfl_xor(nzero, off, 64);
      npert += __shfl_xor(npert, off, 64);
      pert += __shfl_xor(pert, off, 64);
    }
  }
  if (tid == 0) {
    fd.kcur[s] = k;
    fd.nF[s] = k;
    fd.pcount[s] = p;
    fd.stopped[s] = stop ? 1 : 0;
    if (allRows) fd.cbDone[s] = 1;
    fd.inertia[3 * s] += npos;
    fd.inertia[3 * s + 1] += nneg;
    fd.inertia[3 * s + 2] += nzero;
    fd.pert[s] += pert;
    fd.npert[s] += npert;
    atomicMaxNonNeg(fd.runMaxBits + s, fmax(bm, origMax));
  }
}

// Device-coherent accesses for values exchanged between workgroups of one
// launch (no cache write-back or invalidation needed around them).
template <typename T>
__device__ inline void storeCoherent(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ inline T loadCoherent(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Cooperative panel of a front with more eligible rows than one workgroup
// holds (the same decisions as k_panel, dense_kernel.hpp:585-792).  The W
// workgroups of a front own kMwRows consecutive eligible rows each; the
// sub-panel (SW columns from the current pivot) of those rows lives in each
// workgroup's LDS.  Per pivot every workgroup posts its local max |a_ik|
// (workgroup 0 also a_kk and the pivot column's sub-panel rows) and reads
// everyone's, so all reach the same decision.  A decision other than "1x1
// at k" is carried out by workgroup 0 alone on the column buffers in global
// memory (the general path of k_panel) while the others wait; then all
// reload their sub-panel.  Waits are bounded (the error word is raised and
// the wait abandoned), so every workgroup runs to its end.
template <typename T>
__global__ __launch_bounds__(kPanelThreads) void k_panel_mw(const int* list, int count, const int* wgStart,
                                                             DevFronts fd, FactorParams prm, double* wsBase,
                                                             const int64_t* wsOff, MwSync* syncBase, int* err) {
  constexpr int NT = kPanelThreads;
  constexpr int SW = 8;
  constexpr int CSR = kMwRows;
  extern __shared__ double Cs[];  // [SW][CSR]
  __shared__ double Wsub[SW][kPanel + 2];
  __shared__ double wvec[kPanel + 2];
  __shared__ double pdd[kPanel + 2], pdo[kPanel + 2];
  __shared__ int pkd[kPanel + 2];
  __shared__ double redV[NT / 64 + 1];
  __shared__ int redI[NT / 64 + 1];
  __shared__ double bcast[16];
  __shared__ int bcastI[4];
  __shared__ double lastL[SW + 1];  // multipliers of the latest fast pivot at rows k + 1 .. k + SW
  __shared__ int abandon;

  const int tid = threadIdx.x;
  if (static_cast<int>(blockIdx.x) >= wgStart[count]) return;
  const int f = findSegment(wgStart, count, blockIdx.x);
  const int s = list[f];
  const int w = blockIdx.x - wgStart[f];
  const int W = wgStart[f + 1] - wgStart[f];
  MwSync* sy = syncBase + f;
  const unsigned long long base = static_cast<unsigned long long>(loadCoherent(&sy->epoch)) << 16;
  const bool lead = (w == 0);
  double* ws = wsBase + wsOff[s];
  const int m = fd.m[s];
  const int nE = fd.nE[s];
  T* F = static_cast<T*>(fd.F[s]);
  const int64_t io = fd.idxOff[s];
  // after a speculative step the panel started p0 pivots before kcur
  const int kc = fd.kcur[s];
  const bool sp = specFront(prm, nE);
  const int p0 = sp ? fd.pcount[s] : 0;
  const int k0 = kc - p0;
  const int nbEnd = min(k0 + kPanel, nE);
  const bool skip = fd.stopped[s] != 0 || kc >= nbEnd;
  if (skip || nE - k0 > W * kMwRows) {
    if (!skip && tid == 0) atomicExch(err, 2);  // the launch does not cover the rows (never planned so)
    if (lead && tid == 0 && !sp) fd.pcount[s] = 0;
    if (lead && tid == 0) storeCoherent(&sy->epoch, static_cast<unsigned>((base >> 16) + 1));
    return;
  }
  const int r0 = k0 + w * kMwRows;  // first row of this workgroup
  double* curK = ws;
  double* curR = ws + nE;
  auto Fat = [&](int i, int j) -> T& { return F[i + static_cast<size_t>(j) * m]; };

  const bool stat = prm.staticMode != 0;
  double origMax = bitsToDouble(fd.origMaxBits[s]);
  if (!stat && origMax < prm.zeroTol) origMax = 1.0;
  if (stat && origMax < prm.staticAbsFloor) origMax = 1.0;
  const double runMax0 = fmax(origMax, bitsToDouble(fd.runMaxBits[s]));
  double tmax = 0.0;
  const double delta = prm.staticDelta > 0.0 ? prm.staticDelta : sqrt(DBL_EPSILON) * origMax;
  const double sfloor = fmax(prm.staticAbsFloor, prm.staticRelFloor * origMax);
  int npos = 0, nneg = 0, nzero = 0, npert = 0;
  double pert = 0.0;
  int k = kc, p = p0;
  bool stop = false;
  unsigned step = 0;
  if (tid == 0) abandon = 0;
  for (int q = tid; q < p0; q += NT) {
    pdd[q] = fd.dDiag[io + k0 + q];
    pdo[q] = fd.dOff[io + k0 + q];
    pkd[q] = fd.pkind[io + k0 + q];
  }
  __syncthreads();

  // post this workgroup's step, then wait until every workgroup posted it
  auto post = [&](unsigned st) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (tid == 0) storeCoherent(&sy->flag[w], base | st);
  };
  auto waitFor = [&](int from, int to, unsigned st) {
    if (tid >= from && tid < to) {
      unsigned spins = 0;
      while (loadCoherent(&sy->flag[tid]) < (base | st)) {
        if (loadCoherent(err) != 0) {
          abandon = 1;
          break;
        }
        if (++spins > (1u << 22)) {
          atomicExch(err, 3);
          abandon = 1;
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __syncthreads();
  };

  // (D L^T)(q, row) of this panel's pivot q for a row
  auto weightCoherent = [&](int q, int row) -> double {
    auto L = [&](int c) { return static_cast<double>(loadCoherent(&Fat(row, k0 + c))); };
    const int kind = pkd[q];
    if (kind == 1) return pdd[q] * L(q);
    if (kind == 2) return pdd[q] * L(q) + pdo[q] * L(q + 1);
    return pdo[q - 1] * L(q - 1) + pdd[q] * L(q);
  };
  // lastFast: the pivot just taken (p - 1, at row c0 - 1) was a fast 1x1
  // whose multipliers workgroup 0 may still be storing, so its weights come
  // from lastL (the same values, formed from the broadcast pivot column);
  // every earlier pivot's multipliers were stored before workgroup 0 posted
  // the step that followed it.
  int c0 = k, sw = 0;
  auto loadSub = [&](bool lastFast) {
    c0 = k;
    sw = min(SW, nbEnd - k);
    for (int e = tid; e < sw * p; e += NT) {
      const int j = e % sw, q = e / sw;
      Wsub[j][q] = (lastFast && q == p - 1) ? pdd[q] * lastL[1 + j] : weightCoherent(q, c0 + j);
    }
    __syncthreads();
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      const int i = r0 + tid + jj * NT;
      if (i < k || i >= nE) continue;
      double acc[SW];
      loadWiden<SW>(acc, static_cast<const T*>(F), [&](int j) -> int64_t {
        const int col = c0 + j;
        if (j >= sw) return -1;
        return i >= col ? i + static_cast<int64_t>(col) * m : col + static_cast<int64_t>(i) * m;
      });
      // the panel's own rows were stored device-coherent: read them the same way
      const bool panelRow = i < k0 + kPanel + 2;
      constexpr int U = 8;
      int q = 0;
      for (; q + U <= p; q += U) {
        double lv[U];
        if (panelRow) {
          T raw[U];
#pragma unroll
          for (int u = 0; u < U; ++u) raw[u] = loadCoherent(&Fat(i, k0 + q + u));
#pragma unroll
          for (int u = 0; u < U; ++u) lv[u] = static_cast<double>(raw[u]);
        } else {
          loadWiden<U>(lv, static_cast<const T*>(F), [&](int u) -> int64_t { return i + static_cast<int64_t>(k0 + q + u) * m; });
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int j = 0; j < SW; ++j) acc[j] = fma(-lv[u], Wsub[j][q + u], acc[j]);
      }
      for (; q < p; ++q) {
        const double l = panelRow ? loadCoherent(&Fat(i, k0 + q)) : Fat(i, k0 + q);
#pragma unroll
        for (int j = 0; j < SW; ++j) acc[j] = fma(-l, Wsub[j][q], acc[j]);
      }
#pragma unroll
      for (int j = 0; j < SW; ++j)
        if (j < sw) Cs[j * CSR + (i - r0)] = acc[j];
    }
    __syncthreads();
  };

  // ---- general step (workgroup 0 alone; column buffers in global memory) ----
  auto computeW = [&](int row) {
    for (int q = tid; q < p; q += NT) {
      const int kind = pkd[q];
      double wq;
      if (kind == 1)
        wq = pdd[q] * static_cast<double>(Fat(row, k0 + q));
      else if (kind == 2)
        wq = pdd[q] * static_cast<double>(Fat(row, k0 + q)) + pdo[q] * static_cast<double>(Fat(row, k0 + q + 1));
      else
        wq = pdo[q - 1] * static_cast<double>(Fat(row, k0 + q - 1)) + pdd[q] * static_cast<double>(Fat(row, k0 + q));
      wvec[q] = wq;
    }
    __syncthreads();
  };
  auto currentColumn = [&](int col, double* out) {
    for (int i = k + tid; i < nE; i += NT) {
      const double raw = (i >= col) ? Fat(i, col) : Fat(col, i);
      double acc = 0.0;
      for (int q = 0; q < p; ++q) acc = fma(static_cast<double>(Fat(i, k0 + q)), wvec[q], acc);
      out[i] = raw - acc;
    }
    __syncthreads();
  };
  auto swapSym = [&](int a, int b) {
    for (int t = tid; t < m; t += NT) {
      if (t < a) {
        const T x = Fat(a, t);
        Fat(a, t) = Fat(b, t);
        Fat(b, t) = x;
      } else if (t == a) {
        const T x = Fat(a, a);
        Fat(a, a) = Fat(b, b);
        Fat(b, b) = x;
      } else if (t < b) {
        const T x = Fat(t, a);
        Fat(t, a) = Fat(b, t);
        Fat(b, t) = x;
      } else if (t > b) {
        const T x = Fat(t, a);
        Fat(t, a) = Fat(t, b);
        Fat(t, b) = x;
      }
    }
    if (tid == 0) {
      const int tp = fd.perm[io + a];
      fd.perm[io + a] = fd.perm[io + b];
      fd.perm[io + b] = tp;
      double x = curK[a];
      curK[a] = curK[b];
      curK[b] = x;
      x = curR[a];
      curR[a] = curR[b];
      curR[b] = x;
    }
    __syncthreads();
  };
  auto accept1 = [&](const double* col, double d) {
    if (tid == 0) {
      fd.dDiag[io + k] = d;
      fd.dOff[io + k] = 0.0;
      fd.pkind[io + k] = 1;
      pdd[p] = d;
      pdo[p] = 0.0;
      pkd[p] = 1;
      Fat(k, k) = static_cast<T>(d);
    }
    countInertia(d, npos, nneg, nzero);
    tmax = fmax(tmax, fabs(d));
    for (int i = k + 1 + tid; i < nE; i += NT) {
      const double c = col[i];
      tmax = fmax(tmax, fabs(c));
      Fat(i, k) = static_cast<T>(c / d);
    }
    __syncthreads();
    ++k;
    ++p;
  };
  // one general step at pivot k (sigma test, swaps, 1x1 or 2x2, or a stop);
  // curK holds the current column k for the rows [k, nE)
  auto generalStep = [&](double lv, int li, double akk) {
    const int r = li;
    computeW(r);
    currentColumn(r, curR);
    if (tid == 0) curK[r] = curR[k];  // dense_kernel.hpp:543
    __syncthreads();
    double sg = 0.0;
    for (int i = k + tid; i < nE; i += NT)
      if (i != r) sg = fmax(sg, fabs(curR[i]));
    sg = blockMax<NT>(sg, redV);
    int action;
    if (fabs(akk) * sg >= kAlpha * lv * lv)
      action = 1;
    else if (fabs(curR[r]) >= kAlpha * sg)
      action = 2;
    else
      action = 3;
    if (action == 1) {
      accept1(curK, curK[k]);
      return;
    }
    if (action == 2) {
      swapSym(k, r);
      accept1(curR, curR[k]);
      return;
    }
    if (r != k + 1) swapSym(k + 1, r);
    const double d11 = curK[k];
    const double d21 = curK[k + 1];
    const double d22 = curR[k + 1];
    const double det = d11 * d22 - d21 * d21;
    const double rmax = fmax(runMax0, blockMax<NT>(tmax, redV));
    if (fabs(det) <= prm.zeroTol * fmax(1.0, rmax) * fmax(1.0, rmax)) {
      stop = true;
      return;
    }
    tmax = fmax(tmax, fmax(fabs(d11), fmax(fabs(d21), fabs(d22))));
    if (tid == 0) {
      fd.dDiag[io + k] = d11;
      fd.dOff[io + k] = d21;
      fd.dDiag[io + k + 1] = d22;
      fd.dOff[io + k + 1] = 0.0;
      fd.pkind[io + k] = 2;
      fd.pkind[io + k + 1] = 0;
      pdd[p] = d11;
      pdo[p] = d21;
      pkd[p] = 2;
      pdd[p + 1] = d22;
      pdo[p + 1] = 0.0;
      pkd[p + 1] = 0;
      Fat(k, k) = static_cast<T>(d11);
      Fat(k + 1, k) = static_cast<T>(d21);
      Fat(k + 1, k + 1) = static_cast<T>(d22);
    }
    countInertia2(d11, d22, det, npos, nneg);
    const double inv11 = d22 / det, inv21 = -d21 / det, inv22 = d11 / det;
    for (int i = k + 2 + tid; i < nE; i += NT) {
      const double a0 = curK[i], a1 = curR[i];
      tmax = fmax(tmax, fmax(fabs(a0), fabs(a1)));
      Fat(i, k) = static_cast<T>(a0 * inv11 + a1 * inv21);
      Fat(i, k + 1) = static_cast<T>(a0 * inv21 + a1 * inv22);
    }
    __syncthreads();
    k += 2;
    p += 2;
  };

  loadSub(false);
  while (k < nbEnd && !abandon) {
    const int kk = k - c0;
    const double* col = Cs + kk * CSR;
    // local candidates of column k
    double lv = 0.0;
    int li = -1;
#pragma unroll
    for (int jj = 0; jj < 2; ++jj) {
      const int i = r0 + tid + jj * NT;
      if (i > k && i < nE) {
        const double v = fabs(col[i - r0]);
        if (v > 0.0) argmaxCombine(lv, li, v, i);
      }
    }
    blockArgmax<NT>(lv, li, redV, redI);
    const int par = step & 1;
    ++step;
    if (tid == 0) {
      storeCoherent(&sy->lv[par][w], lv);
      storeCoherent(&sy->li[par][w], li);
      if (lead) {
        // a_kk and the pivot column's next SW rows (rows k + t < nbEnd)
        storeCoherent(&sy->extra[par][0], col[k - r0]);
        for (int t = 1; t <= SW && k + t < nbEnd; ++t) storeCoherent(&sy->extra[par][t], col[k + t - r0]);
      }
    }
    post(step);
    waitFor(0, W, step);
    if (abandon) break;
    if (tid == 0) {
      double bv = 0.0;
      int bi = -1;
      for (int v = 0; v < W; ++v) argmaxCombine(bv, bi, loadCoherent(&sy->lv[par][v]), loadCoherent(&sy->li[par][v]));
      bcast[0] = bv;
      bcastI[0] = bi;
      bcast[1] = loadCoherent(&sy->extra[par][0]);
      for (int t = 1; t <= SW && k + t < nbEnd; ++t) bcast[1 + t] = loadCoherent(&sy->extra[par][t]);
    }
    __syncthreads();
    lv = bcast[0];
    li = bcastI[0];
    const double akk = bcast[1];

    // first Bunch-Kaufman tests (dense_kernel.hpp:601-618); static pivots
    // are always accepted at k (dense_kernel.hpp:982-1011)
    int action = -1;
    double dpiv = akk;
    if (stat) {
      const int sign = prm.expectedSign ? prm.expectedSign[fd.frontIdx[io + k]] : 0;
      double applied;
      dpiv = staticPivot(akk, sign, delta, sfloor, applied);
      if (applied != 0.0) {
        pert += fabs(applied);
        ++npert;
      }
      action = 1;
    } else if (lv <= prm.zeroTol) {
      const double isolatedFloor = fmax(prm.zeroTol, prm.relFloor * origMax);
      action = (fabs(akk) <= isolatedFloor) ? 0 : 1;
    } else if (fabs(akk) >= kAlpha * lv) {
      action = 1;
    }
    if (action == 0) {
      stop = true;
      break;
    }
    if (action == 1) {
      const double d = dpiv;
      double wj[SW];
#pragma unroll
      for (int j = 0; j < SW; ++j)
        wj[j] = (j > kk && j < sw) ? d * static_cast<double>(static_cast<T>(bcast[1 + j - kk] / d)) : 0.0;
      pdd[p] = d;
      pdo[p] = 0.0;
      pkd[p] = 1;
      if (tid >= 1 && tid <= SW && k + tid < nbEnd) lastL[tid] = static_cast<double>(static_cast<T>(bcast[1 + tid] / d));
      if (lead && tid == 0) {
        fd.dDiag[io + k] = d;
        fd.dOff[io + k] = 0.0;
        fd.pkind[io + k] = 1;
        Fat(k, k) = static_cast<T>(d);
      }
      if (lead) countInertia(d, npos, nneg, nzero);
      tmax = fmax(tmax, fabs(d));
#pragma unroll
      for (int jj = 0; jj < 2; ++jj) {
        const int i = r0 + tid + jj * NT;
        if (i > k && i < nE) {
          const double c = col[i - r0];
          tmax = fmax(tmax, fabs(c));
          const T lt = static_cast<T>(c / d);
          // rows of the panel are read by every workgroup (their weights)
          if (i < k0 + kPanel + 2)
            storeCoherent(&Fat(i, k), lt);
          else
            Fat(i, k) = lt;
          const double l = lt;
#pragma unroll
          for (int j = 0; j < SW; ++j)
            if (j > kk && j < sw) Cs[j * CSR + (i - r0)] = fma(-l, wj[j], Cs[j * CSR + (i - r0)]);
        }
      }
      __syncthreads();
      ++k;
      ++p;
      if (k - c0 >= sw && k < nbEnd) loadSub(true);
      continue;
    }
    // general step: everyone hands its rows of column k to curK, workgroup 0
    // decides and updates, then everyone reloads its sub-panel
    for (int jj = 0; jj < 2; ++jj) {
      const int i = r0 + tid + jj * NT;
      if (i >= k && i < nE) curK[i] = col[i - r0];
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
    ++step;
    post(step);
    if (lead) {
      waitFor(0, W, step);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      if (!abandon) generalStep(lv, li, akk);
      if (tid == 0) {
        storeCoherent(&sy->state[0], k);
        storeCoherent(&sy->state[1], p);
        storeCoherent(&sy->state[2], stop ? 1 : 0);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
      ++step;
      post(step);
    } else {
      ++step;
      waitFor(0, 1, step);
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      const int nk = loadCoherent(&sy->state[0]);
      const int np = loadCoherent(&sy->state[1]);
      stop = loadCoherent(&sy->state[2]) != 0;
      // the pivots workgroup 0 took in the general step
      for (int q = p + tid; q < np; q += NT) {
        pdd[q] = fd.dDiag[io + k0 + q];
        pdo[q] = fd.dOff[io + k0 + q];
        pkd[q] = fd.pkind[io + k0 + q];
      }
      k = nk;
      p = np;
      __syncthreads();
    }
    if (stop || abandon) break;
    if (k < nbEnd) loadSub(false);
  }
  __syncthreads();

  const double bm = blockMax<NT>(tmax, redV);
  if (tid == 0) atomicMaxNonNeg(fd.runMaxBits + s, fmax(bm, origMax));
  if (lead && tid == 0) {
    fd.kcur[s] = k;
    fd.nF[s] = k;
    fd.pcount[s] = p;
    fd.stopped[s] = stop ? 1 : 0;
    fd.inertia[3 * s] += npos;
    fd.inertia[3 * s + 1] += nneg;
    fd.inertia[3 * s + 2] += nzero;
    fd.pert[s] += pert;
    fd.npert[s] += npert;
    storeCoherent(&sy->epoch, static_cast<unsigned>((base >> 16) + 1));
  }
}

// ---------------------------------------------------------------------------
// Speculative panel step.  The threshold Bunch-Kaufman panel
// (dense_kernel.hpp:585-792) takes pivot k as a 1x1 without an interchange
// whenever |a_kk| >= alpha * lambda_k (lambda_k = max over the eligible rows
// below k of |a_ik|, current values), or lambda_k <= zero_tolerance and
// |a_kk| is above the isolated-pivot floor; static pivots are always taken
// at k (dense_kernel.hpp:982-1011).  When every pivot of a panel is taken
// that way, the panel is an unpivoted LDL^T of its diagonal block followed by
// the substitution of the rows below, and lambda_k is max |c_ik| over the
// values c_ik the substitution forms.  k_spec_block and k_spec_factor do
// both, writing the multipliers over the raw values they back up, and form
// the column maxima; k_spec_apply finds the first column whose test fails and
// restores the columns from there on, and the exact panel kernel continues.
// ---------------------------------------------------------------------------
struct SpecRec {
  unsigned long long* colmax;  // [2][kPanel]
  unsigned long long* emax;
  unsigned long long* nmax;
  double* cdiag;
  double* dval;
  double* bmax;
  double* rdiv;
  double* ops;
  double* wneg;
  int* k0;
  double* backup;
};
__device__ inline SpecRec specRec(double* ws, int nE) {
  double* r = ws + 2 * static_cast<int64_t>(nE);
  SpecRec x;
  x.colmax = reinterpret_cast<unsigned long long*>(r);
  x.emax = reinterpret_cast<unsigned long long*>(r + 2 * kPanel);
  x.nmax = reinterpret_cast<unsigned long long*>(r + 3 * kPanel);
  x.cdiag = r + 4 * kPanel;
  x.dval = r + 5 * kPanel;
  x.bmax = r + 6 * kPanel;
  x.rdiv = r + 7 * kPanel;
  x.ops = r + 8 * kPanel;
  x.wneg = x.ops + 4 * 4 * 64;
  x.k0 = reinterpret_cast<int*>(x.wneg + 6 * 4 * 64);
  x.backup = r + kSpecRec;
  return x;
}

// Smallest float at or above v (v >= 0): a bound that is never below the value.
__device__ inline double roundUpToFloat(double v) {
  float f = static_cast<float>(v);
  if (static_cast<double>(f) < v) f = nextafterf(f, INFINITY);
  return static_cast<double>(f);
}

// Pass 0: one workgroup per front factors the diagonal block (pw x pw,
// pw = min(kPanel, nE - k0)), 1x1 pivots in order, as four blocks of 16
// columns: wave w holds the block's rows 16 w .. 16 w + 15 as MFMA tiles, the
// wave of the diagonal tile factors it (blockFactor16), the waves below
// substitute their rows and update their later columns on the matrix cores.
// The raw values go to the record's backup and the multipliers into the
// front, where a failed test restores them; the record takes the pivots,
// their reciprocals, a_qq, the in-block column maxima and the row pass's
// operands.
//
// Bound by the dependent chain of 64 pivots: 4 x 6,000 cycles, 10 us of the
// 21 on the 80^3 27-point workload (a barrier per two pivots on registers and
// LDS took 37; 29 against 45 with static pivots).
template <typename T>
__global__ __launch_bounds__(256) void k_spec_block(const int* list, int count, DevFronts fd, FactorParams prm,
                                                    double* wsBase, const int64_t* wsOff) {
  constexpr int P = kPanel;
  __shared__ double Ds[16][17];
  __shared__ Block16 blk;
  __shared__ double Ls[4][64][4];  // multipliers of the current 16 columns: wave w's tile, lane-major
  __shared__ double redB[4][P];
  if (static_cast<int>(blockIdx.x) >= count) return;
  const int s = list[blockIdx.x];
  const int nE = fd.nE[s];
  if (!specFront(prm, nE)) return;
  const int m = fd.m[s];
  const int k0 = fd.kcur[s];
  const SpecRec rec = specRec(wsBase + wsOff[s], nE);
  const bool none = fd.stopped[s] || k0 >= nE;
  if (threadIdx.x == 0) *rec.k0 = none ? -1 : k0;
  if (none) return;
  const int pw = min(P, nE - k0);
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const int64_t io = fd.idxOff[s];
  T* const bk = reinterpret_cast<T*>(rec.backup);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const bool stat = prm.staticMode != 0;
  double origMax = bitsToDouble(fd.origMaxBits[s]);
  if (stat && origMax < prm.staticAbsFloor) origMax = 1.0;
  const double delta = prm.staticDelta > 0.0 ? prm.staticDelta : sqrt(DBL_EPSILON) * origMax;
  const double sfloor = fmax(prm.staticAbsFloor, prm.staticRelFloor * origMax);
  const int row = 16 * wv + lr;  // of the block
  const int sgn = stat && prm.expectedSign && row < pw ? prm.expectedSign[fd.frontIdx[io + k0 + row]] : 0;
  T raw[4][4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int col = 16 * b + 4 * u + lk;
      raw[b][u] = F[row < pw && col <= row ? (k0 + row) + static_cast<int64_t>(k0 + col) * m : 0];
    }
  v4d x[4];
#pragma unroll
  for (int b = 0; b < 4; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int col = 16 * b + 4 * u + lk;
      const bool in = row < pw && col <= row;
      if (in) bk[(k0 + row) + static_cast<int64_t>(col) * m] = raw[b][u];
      x[b][u] = in ? static_cast<double>(raw[b][u]) : (col == row ? 1.0 : 0.0);
    }
  unrolled(std::make_integer_sequence<int, 4>{}, [&](auto bb) {
    constexpr int b = decltype(bb)::value;
    if (16 * b >= pw) return;
    if (wv == b) {
#pragma unroll
      for (int u = 0; u < 4; ++u) Ds[lr][4 * u + lk] = x[b][u];
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      double a[16];
#pragma unroll
      for (int q = 0; q < 16; ++q) a[q] = Ds[lr][q];
#pragma unroll
      for (int q = 0; q < 16; ++q) a[q] = q <= lr ? a[q] : 0.0;
      if (!stat)
        blockFactor16<T>(a, blk, [](int, double v) { return v; });
      else
        blockFactor16<T>(a, blk, [&](int q, double v) {
          // (the identity padding is not a pivot)
          double applied;
          const double d = staticPivot(v, __shfl(sgn, q, 64), delta, sfloor, applied);
          return 16 * b + q < pw ? d : v;
        });
    }
    __syncthreads();
    if (wv == b) {
#pragma unroll
      for (int u = 0; u < 4; ++u) rec.ops[(4 * b + u) * 64 + lane] = blk.op[u][lane];
      if (lane < 16) {
        rec.cdiag[16 * b + lane] = blk.akk[lane];
        rec.dval[16 * b + lane] = blk.d[lane];
        rec.rdiv[16 * b + lane] = blk.rd[lane];
      }
    }
    double vm[4];
    if (wv >= b) {
      double op[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) op[u] = blk.op[u][lane];
      substTile(x[b], op);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = 4 * u + lk, col = 16 * b + q;
        // the block's own rows keep the multipliers of its factorization
        const T lt = wv == b ? static_cast<T>(-blk.op[u][lane]) : multiplier<T>(x[b][u], blk.d[q], blk.rd[q]);
        const double l = static_cast<double>(lt);
        if (row < pw && col < row) F[(k0 + row) + static_cast<int64_t>(k0 + col) * m] = lt;
        if (row < pw && col == row) F[(k0 + row) + static_cast<int64_t>(k0 + col) * m] = static_cast<T>(blk.d[q]);
        vm[u] = row < pw && col < row ? fabs(x[b][u]) : 0.0;
        if (wv > b) {
          Ls[wv][lane][u] = l;
          rec.wneg[((wv * (wv - 1) / 2 + b) * 4 + u) * 64 + lane] = row < pw ? -(blk.d[q] * l) : 0.0;
        }
      }
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) vm[u] = 0.0;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double v = max16(vm[u]);
      if (lr == 0) redB[wv][16 * b + 4 * u + lk] = v;
    }
    __syncthreads();
#pragma unroll
    for (int b2 = b + 1; b2 < 4; ++b2) {
      if (wv >= b2) {
#pragma unroll
        for (int u = 0; u < 4; ++u) x[b2] = mfma64(-Ls[b2][lane][u], x[b][u], x[b2]);
        settle(x[b2]);
      }
    }
  });
  __syncthreads();
  if (tid < pw) rec.bmax[tid] = fmax(fmax(redB[0][tid], redB[1][tid]), fmax(redB[2][tid], redB[3][tid]));
}

// Pass 1: every workgroup takes kSpecRows rows below the block of a front
// (eligible rows [k0 + pw, nE) and rows [nE, m) alike), 16 per wave as MFMA
// tiles: saves their raw panel values in the record's backup, substitutes
// them by the block's four 16-column blocks and stores the multipliers in the
// front.  What a block takes off the later columns is the stored multiplier
// times its pivot.  All operands come from the record in lane order, in
// flight together with the rows, so the pass is one memory round trip, 16
// substitution steps with 36 MFMAs between them and the stores.  The column maxima of
// the current values go to the record: over the eligible rows rounded up to
// float (colmax[parity], the threshold test) and exact (emax), over the rows
// [nE, m) exact (nmax).
//
// (One row per thread with the coefficients broadcast from LDS took 31 us a
// launch on the 80^3 27-point workload, this form 21.)
template <typename T>
__global__ __launch_bounds__(4 * kSpecRows) void k_spec_factor(const int* list, int count, const int* wgStart,
                                                               int parity, DevFronts fd, FactorParams prm,
                                                               double* wsBase, const int64_t* wsOff) {
  constexpr int P = kPanel;
  constexpr int NW = kSpecRows / 16;
  __shared__ double partE[NW][P], partN[NW][P];
  if (static_cast<int>(blockIdx.x) >= wgStart[count]) return;
  const int f = findSegment(wgStart, count, blockIdx.x);
  const int s = list[f];
  const int w = blockIdx.x - wgStart[f];
  const int nE = fd.nE[s];
  if (!specFront(prm, nE) || fd.stopped[s]) return;
  const int m = fd.m[s];
  const int k0 = fd.kcur[s];
  if (k0 >= nE) return;
  const int pw = min(P, nE - k0);
  const int rBeg = k0 + pw + w * kSpecRows;
  if (rBeg >= m) return;
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const SpecRec rec = specRec(wsBase + wsOff[s], nE);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int i0 = rBeg + 16 * wv, i = i0 + lr;
  const bool valid = i < m;
  // the panel's first nb blocks of 16 columns
  auto rows = [&](auto nb) {
    constexpr int NB = decltype(nb)::value;
    T raw[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = 16 * b + 4 * u + lk;
        raw[b][u] = F[valid && q < pw ? i + static_cast<int64_t>(k0 + q) * m : 0];
      }
    double op[NB][4], wn[NB > 1 ? NB * (NB - 1) / 2 : 1][4], dv[NB][4], rd[NB][4];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        op[b][u] = rec.ops[(4 * b + u) * 64 + lane];
        dv[b][u] = rec.dval[16 * b + 4 * u + lk];
        rd[b][u] = rec.rdiv[16 * b + 4 * u + lk];
      }
#pragma unroll
    for (int b = 0; b < NB * (NB - 1) / 2; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) wn[b][u] = rec.wneg[(4 * b + u) * 64 + lane];
    v4d x[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) x[b][u] = valid && 16 * b + 4 * u + lk < pw ? static_cast<double>(raw[b][u]) : 0.0;
    // the raw values saved for the exact kernel
    T* bk = reinterpret_cast<T*>(rec.backup);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = 16 * b + 4 * u + lk;
        if (valid && q < pw) bk[i + static_cast<int64_t>(q) * m] = raw[b][u];
      }
    // no branches among the products: see settle
    T l[NB][4];
    unrolled(std::make_integer_sequence<int, NB>{}, [&](auto bb) {
      constexpr int b = decltype(bb)::value;
      substTile(x[b], op[b]);
#pragma unroll
      for (int u = 0; u < 4; ++u) l[b][u] = multiplier<T>(x[b][u], dv[b][u], rd[b][u]);
#pragma unroll
      for (int b2 = b + 1; b2 < NB; ++b2) {
#pragma unroll
        for (int u = 0; u < 4; ++u)
          x[b2] = mfma64(wn[b2 * (b2 - 1) / 2 + b][u], static_cast<double>(l[b][u]), x[b2]);
      }
    });
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = 16 * b + 4 * u + lk;
        if (valid && q < pw) F[i + static_cast<int64_t>(k0 + q) * m] = l[b][u];
      }
    const bool anyE = i0 < nE, anyN = i0 + 16 > nE;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const double c = fabs(x[b][u]);
        const int q = 16 * b + 4 * u + lk;
        const double ve = anyE ? max16(i < nE ? c : 0.0) : 0.0;
        const double vn = anyN ? max16(i >= nE && valid ? c : 0.0) : 0.0;
        if (lr == 0) {
          partE[wv][q] = ve;
          partN[wv][q] = vn;
        }
      }
  };
  if (pw <= 16)
    rows(std::integral_constant<int, 1>{});
  else if (pw <= 32)
    rows(std::integral_constant<int, 2>{});
  else
    rows(std::integral_constant<int, 4>{});
  __syncthreads();
  if (tid < pw) {
    double ve = partE[0][tid], vn = partN[0][tid];
#pragma unroll
    for (int k = 1; k < NW; ++k) {
      ve = fmax(ve, partE[k][tid]);
      vn = fmax(vn, partN[k][tid]);
    }
    if (ve > 0.0) {
      atomicMaxNonNeg(rec.colmax + parity * P + tid, roundUpToFloat(ve));
      atomicMaxNonNeg(rec.emax + tid, ve);
    }
    if (vn > 0.0) atomicMaxNonNeg(rec.nmax + tid, vn);
  }
}

constexpr int kSpecApplyThreads = kSpecRows;
// Pass 2: every workgroup finds the first column q* whose test fails (all of
// them pass when static); when q* < pw it restores, for its rows, the raw
// values the exact kernel continues from (columns [q*, pw) of the eligible
// rows, the whole block of the rows [nE, m)).  Workgroup 0 commits the block's
// columns before q*, the pivots, inertia, perturbation counts and the running
// maximum, sets kcur = k0 + q*, pcount = q*, and clears the other colmax
// buffer and the exact maxima for the next panel.  Nothing orders workgroup 0
// against the others, so what they read is nothing that it writes: the panel's
// position is the record's k0, not kcur.
template <typename T>
__global__ __launch_bounds__(kSpecApplyThreads) void k_spec_apply(const int* list, int count, const int* wgStart, int parity,
                                                    DevFronts fd, FactorParams prm, double* wsBase,
                                                    const int64_t* wsOff) {
  constexpr int P = kPanel;
  __shared__ int qsh;
  if (static_cast<int>(blockIdx.x) >= wgStart[count]) return;
  const int f = findSegment(wgStart, count, blockIdx.x);
  const int s = list[f];
  const int w = blockIdx.x - wgStart[f];
  const int tid = threadIdx.x;
  const int m = fd.m[s];
  const int nE = fd.nE[s];
  if (!specFront(prm, nE)) return;  // this front's panels are all exact
  const SpecRec rec = specRec(wsBase + wsOff[s], nE);
  const int k0 = *rec.k0;
  if (k0 < 0) {
    if (w == 0 && tid == 0) {
      fd.pcount[s] = 0;
      fd.cbDone[s] = 0;
    }
    return;
  }
  const int pw = min(P, nE - k0);
  const int rBeg = k0 + pw + w * kSpecRows;
  if (w > 0 && rBeg >= m) return;
  T* F = static_cast<T*>(fd.F[s]);
  auto Fat = [&](int i, int j) -> T& { return F[i + static_cast<size_t>(j) * m]; };
  const int64_t io = fd.idxOff[s];
  const bool stat = prm.staticMode != 0;
  double origMax = bitsToDouble(fd.origMaxBits[s]);
  if (!stat && origMax < prm.zeroTol) origMax = 1.0;
  if (stat && origMax < prm.staticAbsFloor) origMax = 1.0;
  // first failing column: the first wave tests one column per lane
  if (tid < 64) {
    const int q = tid;
    bool fail = false;
    if (!stat && q < pw) {
      const double isolatedFloor = fmax(prm.zeroTol, prm.relFloor * origMax);
      const double lam = fmax(rec.bmax[q], bitsToDouble(rec.colmax[parity * P + q]));
      const double akk = rec.cdiag[q];
      fail = !((lam <= prm.zeroTol) ? fabs(akk) > isolatedFloor : fabs(akk) >= kAlpha * lam);
    }
    const unsigned long long bad = __ballot(fail);
    if (tid == 0) qsh = bad ? min(pw, __ffsll(static_cast<long long>(bad)) - 1) : pw;
  }
  __syncthreads();
  const int qs = qsh;
  if (qs < pw) {
    const T* bk = reinterpret_cast<const T*>(rec.backup);
    const int i = rBeg + tid;
    if (i < m) {
      for (int q = (i < nE) ? qs : 0; q < pw; ++q) Fat(i, k0 + q) = bk[i + static_cast<int64_t>(q) * m];
    }
    if (w == 0)  // the block's own rows
      for (int e = tid; e < pw * P; e += kSpecApplyThreads) {
        const int r = e & (P - 1), q = e / P;
        if (q >= qs && r >= q && r < pw) Fat(k0 + r, k0 + q) = bk[(k0 + r) + static_cast<int64_t>(q) * m];
      }
  }
  if (w != 0) return;
  double tmax = 0.0;
  if (tid < P) rec.colmax[(parity ^ 1) * P + tid] = 0ull;
  if (tid < 64) {
    // pivots, inertia, perturbation and the maxima of the kept columns: one column per lane
    const int q = tid;
    const double ev = bitsToDouble(rec.emax[q]), nv = bitsToDouble(rec.nmax[q]);
    rec.emax[q] = 0ull;
    rec.nmax[q] = 0ull;
    int npos = 0, nneg = 0, nzero = 0, npert = 0;
    double pert = 0.0;
    if (q < qs) {
      const double d = rec.dval[q];
      fd.dDiag[io + k0 + q] = d;
      fd.dOff[io + k0 + q] = 0.0;
      fd.pkind[io + k0 + q] = 1;
      tmax = fmax(fmax(fabs(d), rec.bmax[q]), ev);
      countInertia(d, npos, nneg, nzero);
      if (stat) {
        const double delta = prm.staticDelta > 0.0 ? prm.staticDelta : sqrt(DBL_EPSILON) * origMax;
        const double sfloor = fmax(prm.staticAbsFloor, prm.staticRelFloor * origMax);
        const int sign = prm.expectedSign ? prm.expectedSign[fd.frontIdx[io + k0 + q]] : 0;
        double applied;
        (void)staticPivot(rec.cdiag[q], sign, delta, sfloor, applied);
        if (applied != 0.0) {
          pert = fabs(applied);
          npert = 1;
        }
      }
    }
    if (qs == pw && q < pw) tmax = fmax(tmax, nv);
    for (int off = 32; off > 0; off >>= 1) {
      npos += __shfl_xor(npos, off, 64);
      nneg += __shfl_xor(nneg, off, 64);
      nzero += __shfl_xor(nzero, off, 64);
      npert += __shfl_xor(npert, off, 64);
      pert += __shfl_xor(pert, off, 64);
      tmax = fmax(tmax, __shfl_xor(tmax, off, 64));
    }
    if (tid == 0) {
      fd.inertia[3 * s] += npos;
      fd.inertia[3 * s + 1] += nneg;
      fd.inertia[3 * s + 2] += nzero;
      fd.pert[s] += pert;
      fd.npert[s] += npert;
      fd.kcur[s] = k0 + qs;
      fd.nF[s] = k0 + qs;
      fd.pcount[s] = qs;
      fd.cbDone[s] = (qs == pw) ? 1 : 0;
      atomicMaxNonNeg(fd.runMaxBits + s, fmax(tmax, origMax));
    }
  }
}

// Clears the colmax buffers and exact maxima of the speculative records of a
// level's fronts.
__global__ void k_spec_reset(const int* list, int count, DevFronts fd, double* wsBase, const int64_t* wsOff) {
  const int f = blockIdx.x;
  if (f >= count) return;
  const int s = list[f];
  const SpecRec rec = specRec(wsBase + wsOff[s], fd.nE[s]);
  for (int t = threadIdx.x; t < 4 * kPanel; t += blockDim.x) rec.colmax[t] = 0ull;
}

// Multipliers of the rows that are not fully summed ([nE, m)) for the last
// panel.  With U = D L^T of the panel, the multipliers of a row are
// f U^{-1} = (f L^{-T}) D^{-1} (dense_kernel.hpp:772-787 applied to the whole
// panel at once).  y = f L^{-T} is a substitution over the panel's columns in
// groups of four (substStep), -L of the panel's block in LDS: every wave takes
// 16 rows as 16 columns of the FP64 MFMA (layout above k_panel), group after
// group, the solved group feeding the products of the later columns from its
// own registers.  l = y D^{-1} follows for the 1x1 and 2x2 pivot blocks.  64
// rows per workgroup: a front's rows spread over as many CUs as they can; what
// is left is the latency of the panel block's loads and of 16 dependent steps.
template <typename T>
__global__ __launch_bounds__(256) void k_panel_rows(const int* list, int count, const int* blockStart,
                                                     DevFronts fd) {
  constexpr int P = kPanel + 1;  // a 2x2 pivot at the panel's last column makes it 65
  constexpr int G = (P + 3) / 4, PP = 4 * G;
  constexpr int NB = (PP + 15) / 16;
  __shared__ double Pm[16 * NB][PP + 1];  // -L of the panel's block, zero on and above its diagonal
  __shared__ double cSelf[PP], cNext[PP], cPrev[PP];  // l_q = y_q cSelf + y_{q+1} cNext + y_{q-1} cPrev
  __shared__ double cDiv[PP];  // 1x1 pivots (cSelf their reciprocals): l_q = y_q / cDiv
  __shared__ int pkd[PP];
  __shared__ int any2;
  if (static_cast<int>(blockIdx.x) >= blockStart[count]) return;
  const int f = findSegment(blockStart, count, blockIdx.x);
  const int s = list[f];
  const int p = fd.pcount[s];
  if (p == 0 || fd.cbDone[s]) return;  // the panel already wrote these rows
  const int m = fd.m[s];
  const int nE = fd.nE[s];
  const int k1 = fd.kcur[s];
  const int k0 = k1 - p;
  const GlobalPtr<T> F = globalView<T>(fd.F[s]);
  const int64_t io = fd.idxOff[s];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  auto at = [&](int i, int j) -> int64_t { return i + static_cast<int64_t>(j) * m; };
  // this wave's rows: column 16 b + 4 u + lk of the panel in register u of
  // block b, all loads in flight together with the panel block's below
  const int row = nE + (static_cast<int>(blockIdx.x) - blockStart[f]) * kPanelRowsWg + 16 * wv + lr;
  T raw[NB][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = 16 * b + 4 * u + lk;
      raw[b][u] = F[row < m && q < p ? at(row, k0 + q) : 0];
    }
  {
    // panel block: row `lane`, columns wv, wv + 4, ...; row 64 by the last loads
    T blk[kPanel / 4];
#pragma unroll
    for (int u = 0; u < kPanel / 4; ++u) {
      const int c = wv + 4 * u;
      blk[u] = F[lane < p && c < lane ? at(k0 + lane, k0 + c) : 0];
    }
    const T last = F[p > kPanel && tid < kPanel ? at(k0 + kPanel, k0 + tid) : 0];
    if (tid == 0) any2 = 0;
    for (int q = tid; q < PP; q += 256) pkd[q] = q < p ? fd.pkind[io + k0 + q] : 1;
    __syncthreads();
    for (int q = tid; q < PP; q += 256) {
      double cs = 1.0, cn = 0.0, cp = 0.0, cd = 1.0;
      if (q < p) {
        const double d = fd.dDiag[io + k0 + q];
        if (pkd[q] == 1) {
          cd = d;
          cs = 1.0 / d;
        } else {
          const int h = pkd[q] == 2 ? q : q - 1;  // first column of the 2x2 block
          const double d11 = fd.dDiag[io + k0 + h], d21 = fd.dOff[io + k0 + h], d22 = fd.dDiag[io + k0 + h + 1];
          const double det = d11 * d22 - d21 * d21;
          cs = (h == q ? d22 : d11) / det;
          (h == q ? cn : cp) = -d21 / det;
          any2 = 1;
        }
      }
      cSelf[q] = cs;
      cNext[q] = cn;
      cPrev[q] = cp;
      cDiv[q] = cd;
    }
    // (the (q+1, q) slot of a 2x2 block holds d21)
#pragma unroll
    for (int u = 0; u < kPanel / 4; ++u) {
      const int c = wv + 4 * u;
      Pm[lane][c] = (lane < p && c < lane && !(lane == c + 1 && pkd[c] == 2)) ? -static_cast<double>(blk[u]) : 0.0;
    }
    if (tid < kPanel) {
      Pm[kPanel][tid] = (p > kPanel && !(tid == kPanel - 1 && pkd[tid] == 2)) ? -static_cast<double>(last) : 0.0;
      for (int r = kPanel + 1; r < 16 * NB; ++r) Pm[r][tid] = 0.0;
    }
    if (tid < 16 * NB)
      for (int c = kPanel; c < PP; ++c) Pm[tid][c] = 0.0;
  }
  __syncthreads();
  v4d x[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u)
      x[b][u] = (row < m && 16 * b + 4 * u + lk < p) ? static_cast<double>(raw[b][u]) : 0.0;
  // group S of block B within the panel's first nb blocks
  auto group = [&](auto nb, auto bb, auto ss) {
    constexpr int N = decltype(nb)::value, B = decltype(bb)::value, S = decltype(ss)::value;
    if constexpr (B < N && 16 * B + 4 * S < PP) {
      substStep<S>(x[B], Pm[16 * B + lr][16 * B + 4 * S + lk]);
      const double y = x[B][S];
#pragma unroll
      for (int rb = B + 1; rb < N; ++rb) x[rb] = mfma64(Pm[16 * rb + lr][16 * B + 4 * S + lk], y, x[rb]);
    }
  };
  auto solve = [&](auto nb) __attribute__((always_inline)) {  // no branches: see settle
    auto block = [&](auto bb) {
      group(nb, bb, std::integral_constant<int, 0>{});
      group(nb, bb, std::integral_constant<int, 1>{});
      group(nb, bb, std::integral_constant<int, 2>{});
      group(nb, bb, std::integral_constant<int, 3>{});
    };
    block(std::integral_constant<int, 0>{});
    block(std::integral_constant<int, 1>{});
    block(std::integral_constant<int, 2>{});
    block(std::integral_constant<int, 3>{});
    block(std::integral_constant<int, 4>{});
#pragma unroll
    for (int b = 0; b < decltype(nb)::value; ++b) settle(x[b]);
  };
  if (p > kPanel)
    solve(std::integral_constant<int, 5>{});
  else if (p > 32)
    solve(std::integral_constant<int, 4>{});
  else if (p > 16)
    solve(std::integral_constant<int, 2>{});
  else
    solve(std::integral_constant<int, 1>{});
  double mx = 0.0;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = 16 * b + 4 * u + lk;
      if (q < p) mx = fmax(mx, fabs(x[b][u]));
    }
  double l[NB][4];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = min(16 * b + 4 * u + lk, PP - 1);
      const double own = x[b][u] * cSelf[q];
      l[b][u] = pkd[q] == 1 ? static_cast<double>(multiplier<T>(x[b][u], cDiv[q], cSelf[q])) : own;
    }
  if (any2) {
    // columns q + 1 and q - 1 of the same row: the neighbouring 16-lane
    // group, in the next or previous register where the group wraps
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int q = 16 * b + 4 * u + lk, qc = min(q, PP - 1);
        const int bn = u < 3 ? b : b + 1, un = (u + 1) & 3, bp = u > 0 ? b : b - 1, up = (u + 3) & 3;
        const double nOwn = __shfl(x[b][u], (lane + 16) & 63, 64);
        const double nWrap = bn < NB ? __shfl(x[bn < NB ? bn : b][un], (lane + 16) & 63, 64) : 0.0;
        const double pOwn = __shfl(x[b][u], (lane + 48) & 63, 64);
        const double pWrap = bp >= 0 ? __shfl(x[bp >= 0 ? bp : b][up], (lane + 48) & 63, 64) : 0.0;
        l[b][u] += (lk < 3 ? nOwn : nWrap) * cNext[qc] + (lk > 0 ? pOwn : pWrap) * cPrev[qc];
      }
  }
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int q = 16 * b + 4 * u + lk;
      if (q < p && row < m) F[at(row, k0 + q)] = static_cast<T>(l[b][u]);
    }
  mx = __ockl_wfred_max_f64(row < m ? mx : 0.0);
  if (lane == 0) atomicMaxNonNeg(fd.runMaxBits + s, mx);
}

// Trailing update T(k1:m, k1:m) -= (L D) L^T over the lower triangle, for
// the last panel's p pivots, on the matrix cores: v_mfma_f64_16x16x4f64 for
// FP64 fronts, v_mfma_f32_16x16x4f32 on FP32 operands for FP32 fronts (L D
// formed in FP64 from the FP64 pivots, then rounded).  Operand layout of the
// instructions on gfx950 (measured): A[i][k] from lane i + 16k, B[k][j] from
// lane j + 16k; the result D[i][j] is in lane j + 16*(i%4), register i/4
// (f64) or lane j + 16*(i/4), register i%4 (f32).
//
// 64x64 lower-triangle output tiles, four waves of 32x32.  The workgroups are
// persistent: each walks the tiles t = blockIdx.x, + gridDim.x, ...; while a
// tile's products and write-back run, the next tile's operand rows and C
// values are already being loaded into registers, and a front's pivots are
// read only when the walk enters a new front.  The product is formed
// transposed (L operand first), so a register holds 16 consecutive rows of a
// column: C is read and written in whole column segments.
//
// Bound by C's traffic (16 bytes per 128 flops in FP64) and by what a tile
// does between its products: L D is formed in registers while the operands
// are staged, behind one barrier and without branches (a neighbouring column
// of a 2x2 block is the thread's own), and every load is unconditional, so
// that the loads of a tile are in flight together.  Measured, all updates of
// a factorization, before (L D through LDS, a branch per column) -> here:
// 30^3 KKT, FP64, 56.1 -> 44.7 ms (17.6 -> 22 TFLOP/s); 64^3 27-point, FP64,
// 16.4 -> 12.9 ms; 53x57x59 27-point, FP32, 6.9 -> 6.0 ms.  FP64 tiles need
// 72 KiB of LDS, so two workgroups fit a CU and may use 256 registers a lane;
// FP32 ones spill below 168.
template <typename T>
struct SchurMfma;
template <>
struct SchurMfma<double> {
  typedef double v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mma(double a, double b, v4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // column (within the 16 x 16 block) of register r of this lane; the row is lane % 16
  static __device__ inline int col(int lane, int r) { return 4 * r + (lane >> 4); }
};
template <>
struct SchurMfma<float> {
  typedef float v4 __attribute__((ext_vector_type(4)));
  static __device__ inline v4 mma(float a, float b, v4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
  static __device__ inline int col(int lane, int r) { return 4 * (lane >> 4) + r; }
};

template <typename T>
__global__ __launch_bounds__(256, sizeof(T) == 8 ? 2 : 3) void k_schur(const int* list, int count, const int* tileStart, const int* tileTp,
                                               DevFronts fd) {
  using M = SchurMfma<T>;
  constexpr int TS = 64;
  constexpr int KP = kPanel + 4;  // padded K (a 2x2 at the panel end makes p = 65)
  constexpr int KU = KP / 4;      // staged columns per thread
  __shared__ T As[TS][KP + 1];    // L D rows of the tile's row block
  __shared__ T Bs[TS][KP + 1];    // L rows of the tile's column block
  // the panel's pivots: diagonal, coupling with the neighbour, its direction
  // (0: 1x1); zero past the panel's columns
  __shared__ double pdd[KP], pdn[KP];
  __shared__ int pdir[KP];
  const int total = tileStart[count];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int wr = (w >> 1) * 32, wc = (w & 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  // staging: row sr of both operand tiles, columns qb + u (a 2x2 block's
  // neighbouring column is then in the thread's own registers)
  const int sr = tid & 63, qb = (tid >> 6) * KU;

  // Geometry of tile t.  A front's tiles are numbered column block by
  // column block (tj, then ti = tj .. Tp-1 down the column), so the
  // workgroups running at the same time read and write consecutive pieces of
  // the same columns.  Tp is the planned tiles per side; the launch covers
  // the column blocks that start before the front's cut (all Tp of them, or
  // fewer when its contribution block is updated separately).  The front's
  // metadata is read again only when the walk enters another front.
  struct Tile {
    int f, s, p, m, k0, k1, Tp, cut, lo, hi, ti, tj;
    GlobalPtr<T> F;
  };
  auto tileOf = [&](int t, const Tile* prev) -> Tile {
    Tile x;
    if (prev && t >= prev->lo && t < prev->hi) {
      x = *prev;
    } else {
      x.f = findSegment(tileStart, count, t);
      x.lo = tileStart[x.f];
      x.hi = tileStart[x.f + 1];
      x.s = list[x.f];
      x.p = fd.pcount[x.s];
      x.m = fd.m[x.s];
      x.k1 = fd.kcur[x.s];
      x.k0 = x.k1 - x.p;
      x.F = globalView<T>(fd.F[x.s]);
      x.Tp = tileTp[x.f];
      x.cut = fd.schurCut[x.s];
    }
    // column block tj starts at S(tj) = tj Tp - tj (tj - 1) / 2
    const int lt = t - x.lo;
    const double b = x.Tp + 0.5;
    int tj = static_cast<int>(b - sqrt(fmax(b * b - 2.0 * lt, 0.0)));
    auto S = [&](int c) { return c * x.Tp - c * (c - 1) / 2; };
    while (tj > 0 && S(tj) > lt) --tj;
    while (tj + 1 < x.Tp && S(tj + 1) <= lt) ++tj;
    x.tj = tj;
    x.ti = tj + (lt - S(tj));
    return x;
  };
  // a tile does work when its front took pivots and the tile lies in the
  // trailing block, left of the cut
  auto live = [&](const Tile& x) { return x.p > 0 && x.k1 + x.ti * TS < x.m && x.k1 + x.tj * TS < x.cut; };
  T la[KU + 2], lb[KU], cv[2][2][4];  // la: columns qb - 1 .. qb + KU
  auto loadTile = [&](const Tile& x) {
    const int i0 = x.k1 + x.ti * TS, j0 = x.k1 + x.tj * TS;
    // every load is unconditional, at an address inside the front: rows past
    // its end only make results that are not stored, columns past the pivots
    // are zeroed when they are staged
    const int ri = min(i0 + sr, x.m - 1), rj = min(j0 + sr, x.m - 1);
#pragma unroll
    for (int u = 0; u < KU + 2; ++u)
      la[u] = x.F[ri + static_cast<size_t>(x.k0 + min(max(qb + u - 1, 0), x.p - 1)) * x.m];
#pragma unroll
    for (int u = 0; u < KU; ++u) lb[u] = x.F[rj + static_cast<size_t>(x.k0 + min(qb + u, x.p - 1)) * x.m];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int row = min(i0 + wr + bi * 16 + lr, x.m - 1);
          const int col = min(j0 + wc + bj * 16 + M::col(lane, rr), x.m - 1);
          cv[bi][bj][rr] = x.F[row + static_cast<size_t>(col) * x.m];
        }
  };

  // XCD-aware walk: workgroups go to the eight XCDs round-robin (blockIdx
  // modulo 8), so each XCD's workgroups take a contiguous eighth of the tiles
  // and neighbouring tiles, which share operand rows, meet in one L2.
  // (Any other placement only costs L2 hits.)
  constexpr int kXcd = 8;
  int t, stride, tEnd;
  if (static_cast<int>(gridDim.x) >= kXcd) {
    const int xcd = blockIdx.x % kXcd;
    const int chunk = (total + kXcd - 1) / kXcd;
    t = xcd * chunk + static_cast<int>(blockIdx.x) / kXcd;
    stride = (static_cast<int>(gridDim.x) - xcd + kXcd - 1) / kXcd;  // workgroups with this residue
    tEnd = min(total, (xcd + 1) * chunk);
  } else {
    t = blockIdx.x;
    stride = gridDim.x;
    tEnd = total;
  }
  if (t >= tEnd) return;
  Tile cur = tileOf(t, nullptr);
  int pivFront = -1;  // front whose pivots are in pdd / pdn / pdir
  bool any2 = false;  // some of them 2x2
  // running max |F| of the updated entries: per lane over the tiles of one
  // front, folded into the front's record when the walk leaves it
  int mxFront = -1;
  double lmx = 0.0;
  auto flushMax = [&]() {
    if (mxFront < 0) return;
    const double wmx = __ockl_wfred_max_f64(lmx);
    if (lane == 0) atomicMaxNonNeg(fd.runMaxBits + mxFront, wmx);
  };
  if (live(cur)) loadTile(cur);
  while (t < tEnd) {
    const int tn = t + stride;
    if (live(cur)) {
      if (cur.s != pivFront) {
        const int64_t io = fd.idxOff[cur.s] + cur.k0;
        bool two = false;
        if (tid < KP) {
          const bool in = tid < cur.p;
          const int kind = in ? fd.pkind[io + tid] : 1;
          pdd[tid] = in && (kind != 0 || tid > 0) ? fd.dDiag[io + tid] : 0.0;
          pdn[tid] = kind == 2 ? fd.dOff[io + tid] : kind == 0 && tid > 0 ? fd.dOff[io + tid - 1] : 0.0;
          pdir[tid] = kind == 2 ? 1 : kind == 0 ? -1 : 0;
          two = kind != 1;
        }
        any2 = __syncthreads_or(two);
        pivFront = cur.s;
      }
      if (cur.ti == 0 && cur.tj == 0 && tid == 0 && fd.schurFlops) {
        // p r (r + 1) over the trailing lower triangle, less the deferred contribution block
        const unsigned long long N = static_cast<unsigned long long>(cur.m - cur.k1);
        const unsigned long long C = static_cast<unsigned long long>(cur.m - max(cur.cut, cur.k1));
        atomicAdd(fd.schurFlops, static_cast<unsigned long long>(cur.p) * (N * (N + 1) - C * (C + 1)));
      }
      // stage the operands, L D formed on the way
      auto stage = [&](auto two) {
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const int q = qb + u;
          const double l = static_cast<double>(la[u + 1]);
          double a = l * pdd[q];
          if (decltype(two)::value) {
            const int d = pdir[q];
            const double n = static_cast<double>(d > 0 ? la[u + 2] : la[u]);
            a = d != 0 ? l * pdd[q] + n * pdn[q] : a;
          }
          As[sr][q] = q < cur.p ? static_cast<T>(a) : T(0);
          Bs[sr][q] = q < cur.p ? lb[u] : T(0);
        }
      };
      if (any2)
        stage(std::true_type());
      else
        stage(std::false_type());
      __syncthreads();
    }
    // the next tile's operands and C travel while this tile computes
    T cn[2][2][4];
#pragma unroll
    for (int bi = 0; bi < 2; ++bi)
#pragma unroll
      for (int bj = 0; bj < 2; ++bj)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) cn[bi][bj][rr] = cv[bi][bj][rr];
    Tile nxt;
    if (tn < tEnd) {
      nxt = tileOf(tn, &cur);
      if (live(nxt)) loadTile(nxt);
    }
    if (live(cur)) {
      const int pp = (cur.p + 3) & ~3;
      typename M::v4 acc[2][2];
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj) acc[bi][bj] = typename M::v4{0, 0, 0, 0};
      for (int kk = 0; kk < pp; kk += 4) {
        const T a0 = As[wr + lr][kk + lk];
        const T a1 = As[wr + 16 + lr][kk + lk];
        const T b0 = Bs[wc + lr][kk + lk];
        const T b1 = Bs[wc + 16 + lr][kk + lk];
        acc[0][0] = M::mma(b0, a0, acc[0][0]);
        acc[0][1] = M::mma(b1, a0, acc[0][1]);
        acc[1][0] = M::mma(b0, a1, acc[1][0]);
        acc[1][1] = M::mma(b1, a1, acc[1][1]);
      }
      const int i0 = cur.k1 + cur.ti * TS, j0 = cur.k1 + cur.tj * TS;
      if (cur.s != mxFront) {
        flushMax();
        mxFront = cur.s;
        lmx = 0.0;
      }
#pragma unroll
      for (int bi = 0; bi < 2; ++bi)
#pragma unroll
        for (int bj = 0; bj < 2; ++bj)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            const int row = i0 + wr + bi * 16 + lr;
            const int col = j0 + wc + bj * 16 + M::col(lane, rr);
            if (row < cur.m && col < cur.cut && (cur.ti != cur.tj || row >= col)) {
              const T v = static_cast<T>(cn[bi][bj][rr] - acc[bi][bj][rr]);
              cur.F[row + static_cast<size_t>(col) * cur.m] = v;
              lmx = fmax(lmx, fabs(static_cast<double>(v)));
            }
          }
      __syncthreads();  // the LDS tiles are restaged for the next tile
    }
    t = tn;
    if (t < tEnd) cur = nxt;
  }
  flushMax();
}

// Operand of the deferred contribution-block update of front s (a front
// whose panels' trailing updates stopped at column nE): for columns
// q0 .. q0 + kc - 1, W = L(nE:m, q) D, the 2x2 blocks coupling neighbouring
// columns as in the tile staging above; zero in the columns at or past the
// pivots the front took, so the rank-kc product CB -= W L(nE:m, q0:q0+kc)^T
// that follows adds nothing for them.  W is column-major with ld = m - nE.
constexpr int kFormCols = 16;
template <typename T>
__global__ __launch_bounds__(256) void k_form_w(DevFronts fd, int s, int q0, int kc, T* __restrict__ W) {
  __shared__ double pdd[kFormCols + 2], pdo[kFormCols + 2];
  __shared__ int pkd[kFormCols + 2];
  const int m = fd.m[s], nE = fd.nE[s], nF = fd.nF[s];
  const int N = m - nE;
  const int c0 = q0 + blockIdx.y * kFormCols;
  const int c1 = min(c0 + kFormCols, q0 + kc);
  const int64_t io = fd.idxOff[s];
  // slot t + 1 holds column c0 + t; slot 0 column c0 - 1
  for (int t = threadIdx.x; t < kFormCols + 2; t += blockDim.x) {
    const int q = c0 - 1 + t;
    const bool ok = q >= 0 && q < nF;
    pdd[t] = ok ? fd.dDiag[io + q] : 0.0;
    pdo[t] = ok ? fd.dOff[io + q] : 0.0;
    pkd[t] = ok ? fd.pkind[io + q] : -1;
  }
  __syncthreads();
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const T* F = static_cast<const T*>(fd.F[s]);
  const T* Lr = F + nE + i;  // row nE + i of the front, column q at Lr[q * m]
  for (int q = c0; q < c1; ++q) {
    const int t = q - c0 + 1;
    const int kind = pkd[t];
    double a = 0.0;
    if (kind == 1) {
      a = static_cast<double>(Lr[static_cast<size_t>(q) * m]) * pdd[t];
    } else if (kind == 2) {
      a = static_cast<double>(Lr[static_cast<size_t>(q) * m]) * pdd[t] +
          static_cast<double>(Lr[static_cast<size_t>(q + 1) * m]) * pdo[t];
    } else if (kind == 0) {
      a = static_cast<double>(Lr[static_cast<size_t>(q - 1) * m]) * pdo[t - 1] +
          static_cast<double>(Lr[static_cast<size_t>(q) * m]) * pdd[t];
    }
    W[i + static_cast<size_t>(q - q0) * N] = static_cast<T>(a);
  }
}

// rowIdx = frontIdx[perm[i]] for every position of the listed fronts.
__global__ void k_make_rowidx(const int* list, int count, DevFronts fd) {
  if (static_cast<int>(blockIdx.x) >= count) return;
  const int s = list[blockIdx.x];
  const int m = fd.m[s];
  const int64_t io = fd.idxOff[s];
  for (int i = threadIdx.x; i < m; i += blockDim.x) fd.rowIdx[io + i] = fd.frontIdx[io + fd.perm[io + i]];
}

// Sum of the per-front statistics (multifrontal.hpp:795-801): partial sums of
// up to kStatsParts workgroups, then their total, each in a fixed order, so
// the perturbation total does not depend on timing.  Bound by the loads'
// latency; one workgroup over all fronts took 34 us for a 100 x 100 grid and
// 1.6 ms for a batch of 192 systems.
constexpr int kStatsThreads = 256;
__device__ inline double waveSum(double v) {
#pragma unroll
  for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
__device__ inline long long waveSum(long long v) {
#pragma unroll
  for (int d = 32; d; d >>= 1) v += __shfl_xor(v, d, 64);
  return v;
}
// six sums over the workgroup, result in thread 0
__device__ inline void statsSum(long long (&r)[5], double& pert) {
  __shared__ long long sI[kStatsThreads / 64][5];
  __shared__ double sD[kStatsThreads / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < 5; ++q) r[q] = waveSum(r[q]);
  pert = waveSum(pert);
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < 5; ++q) sI[w][q] = r[q];
    sD[w] = pert;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int v = 1; v < kStatsThreads / 64; ++v) {
#pragma unroll
      for (int q = 0; q < 5; ++q) r[q] += sI[v][q];
      pert += sD[v];
    }
}
__global__ __launch_bounds__(kStatsThreads) void k_stats_part(int numSN, DevFronts fd, long long* outI, double* outD) {
  long long r[5] = {0, 0, 0, 0, 0};
  double pert = 0.0;
  for (int s = blockIdx.x * kStatsThreads + threadIdx.x; s < numSN; s += gridDim.x * kStatsThreads) {
    r[0] += fd.inertia[3 * s];
    r[1] += fd.inertia[3 * s + 1];
    r[2] += fd.inertia[3 * s + 2];
    r[3] += (fd.nF[s] < fd.nE[s]) ? 1 : 0;
    r[4] += fd.npert[s];
    pert += fd.pert[s];
  }
  statsSum(r, pert);
  if (threadIdx.x == 0) {
    for (int q = 0; q < 5; ++q) outI[kStatsOutI + 5 * blockIdx.x + q] = r[q];
    outD[kStatsOutD + blockIdx.x] = pert;
  }
}
__global__ __launch_bounds__(kStatsThreads) void k_stats_total(int parts, long long* outI, double* outD) {
  long long r[5] = {0, 0, 0, 0, 0};
  double pert = 0.0;
  const int t = threadIdx.x;
  if (t < parts) {
    for (int q = 0; q < 5; ++q) r[q] = outI[kStatsOutI + 5 * t + q];
    pert = outD[kStatsOutD + t];
  }
  statsSum(r, pert);
  if (t == 0) {
    for (int q = 0; q < 5; ++q) outI[q] = r[q];
    outD[0] = pert;
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
void launchResetFronts(int numSN, const DevFronts& fd, hipStream_t st) {
  if (numSN <= 0) return;
  const int blocks = (numSN + 255) / 256;
  k_reset_fronts<<<blocks, 256, 0, st>>>(numSN, fd);
  hipCheck(hipGetLastError(), "launchResetFronts");
}
void launchResetPerm(const int* list, int count, const DevFronts& fd, hipStream_t st) {
  if (count <= 0) return;
  k_reset_perm<<<count, 256, 0, st>>>(list, count, fd);
  hipCheck(hipGetLastError(), "launchResetPerm");
}
void launchAssemble(const int4* tasks, int ntasks, const DevFronts& fd, const double* aVals, int monotone,
                    hipStream_t st) {
  if (ntasks <= 0) return;
  if (monotone) {
    if (fd.fp32)
      k_assemble<float><<<ntasks, 256, 0, st>>>(tasks, ntasks, fd, aVals);
    else
      k_assemble<double><<<ntasks, 256, 0, st>>>(tasks, ntasks, fd, aVals);
  } else {
    if (fd.fp32)
      k_assemble_any<float><<<ntasks, 256, 0, st>>>(tasks, ntasks, fd, aVals);
    else
      k_assemble_any<double><<<ntasks, 256, 0, st>>>(tasks, ntasks, fd, aVals);
  }
  hipCheck(hipGetLastError(), "launchAssemble");
}
template <typename T>
static void factorSmallT(const int* list, int count, int maxM, const DevFronts& fd, const FactorParams& prm,
                         hipStream_t st) {
  const size_t smem = smallFrontSmemBytes(maxM);
  static bool attrSet = false;
  if (!attrSet) {
    hipCheck(hipFuncSetAttribute(reinterpret_cast<const void*>(k_factor_small<T>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize,
                                 static_cast<int>(smallFrontSmemBytes(kSmallFrontMax))),
             "k_factor_small LDS size");
    attrSet = true;
  }
  k_factor_small<T><<<count, kSmallThreads, smem, st>>>(list, count, fd, prm);
  hipCheck(hipGetLastError(), "factorSmallT");
}
void launchFactorSmall(const int* list, int count, int maxM, const DevFronts& fd, const FactorParams& prm,
                       hipStream_t st) {
  if (count <= 0) return;
  if (fd.fp32)
    factorSmallT<float>(list, count, maxM, fd, prm, st);
  else
    factorSmallT<double>(list, count, maxM, fd, prm, st);
  hipCheck(hipGetLastError(), "launchFactorSmall");
}
void launchFrontMaxAbs(const int* list, int count, int maxM, const DevFronts& fd, hipStream_t st) {
  if (count <= 0) return;
  int bpf = (maxM + 15) / 16;
  if (bpf > 64) bpf = 64;
  if (bpf < 1) bpf = 1;
  if (fd.fp32)
    k_front_maxabs<float><<<count * bpf, 256, 0, st>>>(list, count, bpf, fd);
  else
    k_front_maxabs<double><<<count * bpf, 256, 0, st>>>(list, count, bpf, fd);
  hipCheck(hipGetLastError(), "launchFrontMaxAbs");
}
template <int TPW, typename T>
static void panelLaunch(const int* list, int count, const DevFronts& fd, const FactorParams& prm, double* ws,
                        const int64_t* wsOff, hipStream_t st) {
  constexpr size_t lds = PanelShape<TPW, T>::lds();
  static const hipError_t attr =
      lds > 0 ? hipFuncSetAttribute(reinterpret_cast<const void*>(k_panel<TPW, T>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds))
              : hipSuccess;
  hipCheck(attr, "k_panel LDS size");
  k_panel<TPW, T><<<count, kPanelThreads, lds, st>>>(list, count, fd, prm, ws, wsOff);
  hipCheck(hipGetLastError(), "panelLaunch");
}
template <typename T>
static void panelT(const int* list, int count, int maxRows, const DevFronts& fd, const FactorParams& prm, double* ws,
                   const int64_t* wsOff, hipStream_t st) {
  // tiles per wave for the rows of the widest front
  if (maxRows <= kPanelRegRows / 16)
    panelLaunch<1, T>(list, count, fd, prm, ws, wsOff, st);
  else if (maxRows <= kPanelRegRows / 8)
    panelLaunch<2, T>(list, count, fd, prm, ws, wsOff, st);
  else if (maxRows <= kPanelRegRows / 4)
    panelLaunch<4, T>(list, count, fd, prm, ws, wsOff, st);
  else if (maxRows <= kPanelRegRows / 2)
    panelLaunch<8, T>(list, count, fd, prm, ws, wsOff, st);
  else if (maxRows <= kPanelRegRows)
    panelLaunch<16, T>(list, count, fd, prm, ws, wsOff, st);
  else
    panelLaunch<0, T>(list, count, fd, prm, ws, wsOff, st);
}
void launchPanel(const int* list, int count, int maxRows, const DevFronts& fd, const FactorParams& prm, double* ws,
                 const int64_t* wsOff, hipStream_t st) {
  if (count <= 0) return;
  if (fd.fp32)
    panelT<float>(list, count, maxRows, fd, prm, ws, wsOff, st);
  else
    panelT<double>(list, count, maxRows, fd, prm, ws, wsOff, st);
  hipCheck(hipGetLastError(), "launchPanel");
}
void launchPanelMw(const int* list, int count, const int* wgStart, int blocks, const DevFronts& fd,
                   const FactorParams& prm, double* ws, const int64_t* wsOff, MwSync* sync, int* err,
                   hipStream_t st) {
  if (count <= 0 || blocks <= 0) return;
  constexpr size_t lds = sizeof(double) * 8 * kMwRows;
  static bool attrSet[2] = {false, false};
  if (fd.fp32) {
    if (!attrSet[1]) {
      hipCheck(hipFuncSetAttribute(reinterpret_cast<const void*>(k_panel_mw<float>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
               "k_panel_mw LDS size");
      attrSet[1] = true;
    }
    k_panel_mw<float><<<blocks, kPanelThreads, lds, st>>>(list, count, wgStart, fd, prm, ws, wsOff, sync, err);
  } else {
    if (!attrSet[0]) {
      hipCheck(hipFuncSetAttribute(reinterpret_cast<const void*>(k_panel_mw<double>),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)),
               "k_panel_mw LDS size");
      attrSet[0] = true;
    }
    k_panel_mw<double><<<blocks, kPanelThreads, lds, st>>>(list, count, wgStart, fd, prm, ws, wsOff, sync, err);
  }
  hipCheck(hipGetLastError(), "launchPanelMw");
}
void launchSpecReset(const int* list, int count, const DevFronts& fd, double* ws, const int64_t* wsOff,
                     hipStream_t st) {
  if (count <= 0) return;
  k_spec_reset<<<count, 128, 0, st>>>(list, count, fd, ws, wsOff);
  hipCheck(hipGetLastError(), "launchSpecReset");
}
void launchSpecPanel(const int* list, int count, const int* wgStart, int blocks, int parity, const DevFronts& fd,
                     const FactorParams& prm, double* ws, const int64_t* wsOff, hipStream_t st) {
  if (count <= 0 || blocks <= 0) return;
  if (fd.fp32) {
    k_spec_block<float><<<count, 256, 0, st>>>(list, count, fd, prm, ws, wsOff);
    hipCheck(hipGetLastError(), "k_spec_block");
    k_spec_factor<float><<<blocks, 4 * kSpecRows, 0, st>>>(list, count, wgStart, parity, fd, prm, ws, wsOff);
    hipCheck(hipGetLastError(), "k_spec_factor");
    k_spec_apply<float><<<blocks, kSpecApplyThreads, 0, st>>>(list, count, wgStart, parity, fd, prm, ws, wsOff);
  } else {
    k_spec_block<double><<<count, 256, 0, st>>>(list, count, fd, prm, ws, wsOff);
    hipCheck(hipGetLastError(), "k_spec_block");
    k_spec_factor<double><<<blocks, 4 * kSpecRows, 0, st>>>(list, count, wgStart, parity, fd, prm, ws, wsOff);
    hipCheck(hipGetLastError(), "k_spec_factor");
    k_spec_apply<double><<<blocks, kSpecApplyThreads, 0, st>>>(list, count, wgStart, parity, fd, prm, ws, wsOff);
  }
  hipCheck(hipGetLastError(), "launchSpecPanel");
}
void launchPanelRows(const int* list, int count, const int* blockStart, int totalBlocks, const DevFronts& fd,
                     hipStream_t st) {
  if (count <= 0 || totalBlocks <= 0) return;
  if (fd.fp32)
    k_panel_rows<float><<<totalBlocks, 256, 0, st>>>(list, count, blockStart, fd);
  else
    k_panel_rows<double><<<totalBlocks, 256, 0, st>>>(list, count, blockStart, fd);
  hipCheck(hipGetLastError(), "launchPanelRows");
}
void launchSyrk(const int* list, int count, const int* tileStart, const int* tileTp, int totalTiles,
                const DevFronts& fd, hipStream_t st) {
  if (count <= 0 || totalTiles <= 0) return;
  // persistent workgroups: as many as are resident at once (LDS and
  // registers allow two per CU in FP64, three in FP32), so that none starts after the others have taken their
  // share of tiles
  static int resident[2] = {0, 0};
  int& res = resident[fd.fp32 ? 1 : 0];
  if (res == 0) {
    int dev = 0, cus = 0, per = 0;
    hipCheck(hipGetDevice(&dev), "hipGetDevice");
    hipCheck(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "CU count");
    hipCheck(hipOccupancyMaxActiveBlocksPerMultiprocessor(
                 &per, fd.fp32 ? reinterpret_cast<const void*>(k_schur<float>) : reinterpret_cast<const void*>(k_schur<double>),
                 256, 0),
             "k_schur occupancy");
    res = std::max(1, per) * std::max(1, cus);
  }
  const int blocks = std::min(totalTiles, res);
  if (fd.fp32)
    k_schur<float><<<blocks, 256, 0, st>>>(list, count, tileStart, tileTp, fd);
  else
    k_schur<double><<<blocks, 256, 0, st>>>(list, count, tileStart, tileTp, fd);
  hipCheck(hipGetLastError(), "launchSyrk");
}
void launchFormW(const DevFronts& fd, int s, int rows, int q0, int kc, void* W, hipStream_t st) {
  if (rows <= 0 || kc <= 0) return;
  const dim3 grid((rows + 255) / 256, (kc + kFormCols - 1) / kFormCols);
  if (fd.fp32)
    k_form_w<float><<<grid, 256, 0, st>>>(fd, s, q0, kc, static_cast<float*>(W));
  else
    k_form_w<double><<<grid, 256, 0, st>>>(fd, s, q0, kc, static_cast<double*>(W));
  hipCheck(hipGetLastError(), "launchFormW");
}
void launchMakeRowIdx(const int* list, int count, const DevFronts& fd, hipStream_t st) {
  if (count <= 0) return;
  k_make_rowidx<<<count, 256, 0, st>>>(list, count, fd);
  hipCheck(hipGetLastError(), "launchMakeRowIdx");
}
void launchReduceStats(int numSN, const DevFronts& fd, long long* outI, double* outD, hipStream_t st) {
  const int parts = std::max(1, std::min(kStatsParts, (numSN + kStatsThreads - 1) / kStatsThreads));
  k_stats_part<<<parts, kStatsThreads, 0, st>>>(numSN, fd, outI, outD);
  k_stats_total<<<1, kStatsThreads, 0, st>>>(parts, outI, outD);
  hipCheck(hipGetLastError(), "launchReduceStats");
}

}  // namespace symla_hip
