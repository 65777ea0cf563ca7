// runner.hip — the ADMM runner (runner.h): layout kernels and the loop kernel.
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include <algorithm>
#include <new>
#include <vector>

#include "panel.h"
#include "runner.h"

namespace osqp_hip {

namespace {

constexpr int kT = 1024;            // threads of a workgroup
constexpr int kW = kT / kWave;      // its wavefronts
constexpr int kSortMax = 16384;     // rows of a workgroup that the layout kernel sorts
constexpr uint16_t kNoRow = 0xFFFF;
constexpr size_t kRunLds = 159 * 1024;  // dynamic LDS of a launch
// Entries of A and P up to which one workgroup runs alone.  us per ADMM
// iteration (one CG iteration each) by one workgroup and by 32, FP64 / FP32:
// 3.4k entries 20.6 / 20.1 and 29.4 / 30.0, 17k 29.9 / 26.0 and 30.2 / 29.8,
// 26k 37.6 / 30.5 and 31.4 / 31.5, 44k 51.2 / 42.1 and 35.3 / 34.3.  The line
// is this high for problems with equality rows, which have only the one
// workgroup (the separate kernels take 104 and 103 at 44k); others past 20k
// entries would be faster on 32.
constexpr long long kRun1Work = 48000;
// Entries up to which the runner is taken, and built (20 bytes an entry in
// FP64, 12 in FP32): measured up to 60 M, where an iteration of 8000 x 150000
// takes 660 us and 884 on the separate kernels (FP32 467 and 531).
constexpr long long kRunMaxWork = 64000000;
constexpr int kRunChain = 24;  // entries that a lane adds up of a row, while a row has lanes left to take
constexpr int kRunPolls = 1 << 22;  // looks of a barrier's wait, some seconds

inline hipStream_t S() { return rt().stream; }

// ---- layout -----------------------------------------------------------------
// row ranges balanced by entries + 8 per row; sorted[0] = 0 if a column's rows
// are not ascending
__global__ void k_run_ranges(int m, int G, const int* rp, int* r0) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b > G) return;
  const long long total = (long long)rp[m] + 8LL * m, want = total * b / G;
  int lo = 0, hi = m;  // first r with rp[r] + 8 r >= want
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if ((long long)rp[mid] + 8LL * mid >= want) hi = mid;
    else lo = mid + 1;
  }
  r0[b] = b == G ? m : lo;
}
__global__ void k_run_sorted(int n, const int* trp, const int* tci, int* sorted) {
  for (int j = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave; j < n; j += gridDim.x * (blockDim.x / kWave))
    for (int k = trp[j] + (int)(threadIdx.x & (kWave - 1)); k + 1 < trp[j + 1]; k += kWave)
      if (tci[k] >= tci[k + 1]) *sorted = 0;
}
__global__ void k_run_cuts(int n, int G, const int* trp, const int* tci, const int* r0, int* cs) {
  for (long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x; t < (long long)(G + 1) * n;
       t += (long long)gridDim.x * blockDim.x) {
    const int b = (int)(t / n), j = (int)(t % n), r = r0[b];
    int lo = trp[j], hi = trp[j + 1];
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (tci[mid] >= r) hi = mid;
      else lo = mid + 1;
    }
    cs[t] = lo;
  }
}

// The three copies: A's rows of a range, the columns of those rows, and P's
// rows of a chunk of cw columns.
enum RunKind { kRowsA, kColsA, kRowsP };
struct RunSrc {
  int n, cw;
  const int *rp, *ci;   // CSR of A, CSC of A, or CSR of P
  const double* val;
  const int *r0, *cs;
};
template <RunKind K>
__device__ __forceinline__ int run_count(const RunSrc& s, int b) {
  if constexpr (K == kColsA) return s.n;
  else if constexpr (K == kRowsA) return s.r0[b + 1] - s.r0[b];
  else return (b + 1) * s.cw <= s.n ? s.cw : (b * s.cw < s.n ? s.n - b * s.cw : 0);
}
// first and one-past-last source entry of local row i
template <RunKind K>
__device__ __forceinline__ int run_begin(const RunSrc& s, int b, int i, int* end) {
  if constexpr (K == kColsA) {
    *end = s.cs[(long long)(b + 1) * s.n + i];
    return s.cs[(long long)b * s.n + i];
  } else {
    const int r = (K == kRowsA ? s.r0[b] : b * s.cw) + i;
    *end = s.rp[r + 1];
    return s.rp[r];
  }
}

// One workgroup a range: its rows sorted by steps (bitonic over key = length
// descending, then index), slice offsets, and its step count.
template <RunKind K>
__global__ __launch_bounds__(kT) void k_run_layout(RunSrc src, int lgT, int ns, int* soff, uint16_t* perm, int* steps) {
  extern __shared__ unsigned key[];  // a power of two >= rows
  const int b = blockIdx.x, rows = run_count<K>(src, b);
  int N = 1;
  while (N < rows) N <<= 1;
  for (int i = threadIdx.x; i < N; i += kT) {
    unsigned k = 0xFFFFFFFFu;
    if (i < rows) {
      int e;
      const int s = run_begin<K>(src, b, i, &e);
      const int st = (e - s + (1 << lgT) - 1) >> lgT;
      k = ((unsigned)(65535 - (st < 65535 ? st : 65535)) << 16) | (unsigned)i;
    }
    key[i] = k;
  }
  __syncthreads();
  for (int size = 2; size <= N; size <<= 1)
    for (int d = size >> 1; d > 0; d >>= 1) {
      for (int t = threadIdx.x; t < N / 2; t += kT) {
        const int i = 2 * d * (t / d) + (t % d), j = i + d;
        const unsigned a = key[i], c = key[j];
        const bool up = (i & size) == 0;
        if ((a > c) == up) {
          key[i] = c;
          key[j] = a;
        }
      }
      __syncthreads();
    }
  const int per = kWave >> lgT;  // rows of a slice
  for (int i = threadIdx.x; i < ns * per; i += kT)
    perm[(long long)b * ns * per + i] = i < rows ? (uint16_t)(key[i] & 0xFFFFu) : kNoRow;
  if (threadIdx.x == 0) {
    int at = 0;
    for (int s = 0; s < ns; ++s) {
      soff[(long long)b * (ns + 1) + s] = at;
      const int i = s * per;
      if (i < rows) at += 65535 - (int)(key[i] >> 16);
    }
    soff[(long long)b * (ns + 1) + ns] = at;
    steps[b] = at;
    steps[gridDim.x + b] = rows > 0 ? 65535 - (int)(key[0] >> 16) : 0;  // the longest row's
  }
}

// entries in slice order: columns (col != null) and values (val != null)
template <RunKind K, typename V>
__global__ __launch_bounds__(kT) void k_run_fill(RunSrc src, int lgT, int ns, const int* soff, const uint16_t* perm,
                                                 const long long* base, uint16_t* col, V* val) {
  const int b = blockIdx.x, lane = threadIdx.x & (kWave - 1), wv = threadIdx.x / kWave, T = 1 << lgT;
  const int per = kWave >> lgT, first = K == kColsA ? src.r0[b] : 0;
  const int zero = K == kColsA ? src.r0[b + 1] - first : src.n;  // padding reads the zero slot past the vector
  for (int s = wv; s < ns; s += kW) {
    const int s0 = soff[(long long)b * (ns + 1) + s], s1 = soff[(long long)b * (ns + 1) + s + 1];
    const int row = perm[((long long)b * ns + s) * per + (lane >> lgT)];
    int k = 0, e = 0;
    if (row != kNoRow) k = run_begin<K>(src, b, row, &e);
    k += lane & (T - 1);
    for (int i = s0; i < s1; ++i, k += T) {
      const long long at = (base[b] + i) * kWave + lane;
      if (col) col[at] = (uint16_t)(k < e ? src.ci[k] - first : zero);
      if (val) val[at] = k < e ? (V)src.val[k] : (V)0;
    }
  }
}

// One workgroup: entries in slice order, lanes per row by slice.  ci holds
// columns of the multiplied vector [x; w]; padding reads its zero slot.
template <typename V>
__global__ __launch_bounds__(kT) void k_run1_fill(int ns, const int* rp, const int* ci, const double* src,
                                                  const int2* sl, const uint16_t* perm, int zero, uint16_t* col, V* val) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int s = blockIdx.x * kW + threadIdx.x / kWave; s < ns; s += gridDim.x * kW) {
    const int s0 = sl[s].x, s1 = sl[s + 1].x, lgT = sl[s].y & 7, row = perm[(sl[s].y >> 3) + (lane >> lgT)];
    int k = 0, e = 0;
    if (row != kNoRow) {
      k = rp[row] + (lane & ((1 << lgT) - 1));
      e = rp[row + 1];
    }
    for (int i = s0; i < s1; ++i, k += 1 << lgT) {
      if (col) col[i * kWave + lane] = (uint16_t)(k < e ? ci[k] : zero);
      if (val) val[i * kWave + lane] = k < e ? (V)src[k] : (V)0;
    }
  }
}

// ---- the loop ------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T ldx(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void stx(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// one of the three copies, as a launch sees it
struct RunView {
  int lgT, ns, slots, res;  // slots: of one workgroup; res: entries of the largest one (LDS copy)
  const int* soff;
  const uint16_t* perm;
  const long long* base;
  const uint16_t* col;
  const void* val;
};
struct RunArgs {
  int n, m, G, cw, lgcw, rows_max;
  const int* r0;
  RunView A, At, P, A2;
  double *part, *xch;
  unsigned* bar;
  int polls;
  RunCall c;
};

// Grid barrier of workgroups that are all resident (cooperative launch), in
// two levels: 8 groups of workgroups (blockIdx mod 8, an XCD each in dispatch
// order), then the groups.  Words 64 apart.  Every wavefront's stores have
// completed (vmcnt) before its workgroup arrives.  The wait is bounded (polls):
// past it the workgroup sets the host's word and leaves the kernel, as the
// others do at their next barrier; the host then restores what the launch
// changed (runner_restore).
__device__ __forceinline__ bool grid_barrier(const RunArgs& a, unsigned epoch, int* flag) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned nb = gridDim.x, ng = nb < 8 ? nb : 8, g = blockIdx.x & 7, gs = (nb + 7 - g) / 8;
    unsigned* w = a.bar;
    int ok = 1;
    if (__hip_atomic_fetch_add(w + g * 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch * gs - 1) {
      if (__hip_atomic_fetch_add(w + 8 * 64, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch * ng - 1)
        for (unsigned k = 0; k < ng; ++k) stx(w + (9 + k) * 64, epoch);
    }
    for (int k = 0; ldx(w + (9 + g) * 64) < epoch; ++k) {
      if (k >= a.polls) {
        __hip_atomic_store(a.c.bad, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // with the host before this launch ends
        ok = 0;
        break;
      }
      __builtin_amdgcn_s_sleep(1);
    }
    *flag = ok;
  }
  __syncthreads();
  asm volatile("" ::: "memory");
  return *flag != 0;
}

// ---- reductions over the workgroup --------------------------------------------
// Within a wavefront by DPP moves (rows of 16 lanes, then row broadcasts; the
// total lands in lane 63), across wavefronts through LDS in wavefront order.
// Shuffles through LDS took about 0.4 us a reduction.  Two LDS buffers taken
// in turn, so one barrier a reduction is enough.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_d(double old, double v) {
  const long long o = __double_as_longlong(old), x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)x, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(x >> 32), CTRL, ROWS, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}
__device__ __forceinline__ double wave_sum63(double v) {
  v += dpp_d<0x111, 0xf>(0.0, v);  // row_shr:1, 2, 4, 8
  v += dpp_d<0x112, 0xf>(0.0, v);
  v += dpp_d<0x114, 0xf>(0.0, v);
  v += dpp_d<0x118, 0xf>(0.0, v);
  v += dpp_d<0x142, 0xa>(0.0, v);  // row_bcast:15 into rows 1, 3
  v += dpp_d<0x143, 0xc>(0.0, v);  // row_bcast:31 into rows 2, 3
  return v;
}
// of non-negative values
__device__ __forceinline__ double wave_max63(double v) {
  double o;
  o = dpp_d<0x111, 0xf>(0.0, v); v = o > v ? o : v;
  o = dpp_d<0x112, 0xf>(0.0, v); v = o > v ? o : v;
  o = dpp_d<0x114, 0xf>(0.0, v); v = o > v ? o : v;
  o = dpp_d<0x118, 0xf>(0.0, v); v = o > v ? o : v;
  o = dpp_d<0x142, 0xa>(0.0, v); v = o > v ? o : v;
  o = dpp_d<0x143, 0xc>(0.0, v); v = o > v ? o : v;
  return v;
}
struct BlkRed {
  double* lds;  // 2 x 2 kW
  int turn;
  __device__ __forceinline__ double* next() { return lds + 2 * kW * (turn++ & 1); }
  __device__ __forceinline__ double sum(double v) {
    double* w = next();
    v = wave_sum63(v);
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) w[threadIdx.x / kWave] = v;
    __syncthreads();
    double r = 0;
#pragma unroll
    for (int i = 0; i < kW; ++i) r += w[i];
    return r;
  }
  __device__ __forceinline__ double max(double v) {
    double* w = next();
    v = wave_max63(v);
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) w[threadIdx.x / kWave] = v;
    __syncthreads();
    double r = w[0];
#pragma unroll
    for (int i = 1; i < kW; ++i) r = w[i] > r ? w[i] : r;
    return r;
  }
  __device__ __forceinline__ void sum_max(double& s, double& m) {
    double* w = next();
    s = wave_sum63(s);
    m = wave_max63(m);
    if ((threadIdx.x & (kWave - 1)) == kWave - 1) {
      w[threadIdx.x / kWave] = s;
      w[kW + threadIdx.x / kWave] = m;
    }
    __syncthreads();
    double rs = 0, rm = w[kW];
#pragma unroll
    for (int i = 0; i < kW; ++i) rs += w[i];
#pragma unroll
    for (int i = 1; i < kW; ++i) rm = w[kW + i] > rm ? w[kW + i] : rm;
    s = rs;
    m = rm;
  }
};

// epi(row, sum) for the workgroup's rows of a sliced copy; x: LDS, with its
// zero slot.  soff and perm are LDS copies (a load from global memory per
// slice and wavefront cost more than the slice).  Slices go to wavefronts in
// turn, from `rot` on; kU steps' loads are in flight.
constexpr int kU = 8;
template <typename TX, typename VP, typename CP, typename X, typename Epi>
__device__ __forceinline__ void run_rows(const int lgT, const int ns, const int rot, const int* soff,
                                         const uint16_t* perm, VP val, CP col, X x, Epi epi) {
  const int lane = threadIdx.x & (kWave - 1);
  const int wv = (__builtin_amdgcn_readfirstlane(threadIdx.x / kWave) + kW - (rot % kW)) % kW;
  const int per = kWave >> lgT;
  for (int s = wv; s < ns; s += kW) {
    const int s0 = __builtin_amdgcn_readfirstlane(soff[s]), s1 = __builtin_amdgcn_readfirstlane(soff[s + 1]);
    const int row = perm[s * per + (lane >> lgT)];
    TX acc = 0;
    int i = s0;
    for (; i + kU <= s1; i += kU) {
      TX v[kU];
      int c[kU];
#pragma unroll
      for (int q = 0; q < kU; ++q) {
        v[q] = (TX)val[(i + q) * kWave + lane];
        c[q] = col[(i + q) * kWave + lane];
      }
#pragma unroll
      for (int q = 0; q < kU; ++q) acc += v[q] * x[c[q]];
    }
    if (i < s1) {
      TX v[kU];
      int c[kU];
#pragma unroll
      for (int q = 0; q < kU - 1; ++q)
        if (i + q < s1) {
          v[q] = (TX)val[(i + q) * kWave + lane];
          c[q] = col[(i + q) * kWave + lane];
        }
#pragma unroll
      for (int q = 0; q < kU - 1; ++q)
        if (i + q < s1) acc += v[q] * x[c[q]];
    }
    for (int o = 1; o < (1 << lgT); o <<= 1) acc += __shfl_xor(acc, o, kWave);
    if (row != kNoRow && (lane & ((1 << lgT) - 1)) == 0) epi(row, acc);
  }
}

// epi(c, sum) for the chunk's columns c0 + c: the G shares of a column added
// over fixed groups of workgroups, in FP64; red: kT doubles of LDS
template <typename TV, typename Epi>
__device__ __forceinline__ void chunk_sum(const TV* part, int n, int G, int c0, int nc, int lgcw, double* red, Epi epi) {
  const int cwp = 1 << lgcw, tid = threadIdx.x, c = tid & (cwp - 1), bi = tid >> lgcw, nbp = kT >> lgcw;
  for (int t0 = 0; t0 < nc; t0 += cwp) {
    double acc = 0.0;
    if (t0 + c < nc) {
      const TV* __restrict__ src = part + c0 + t0 + c;
      int b = bi;
      for (; b + 3 * nbp < G; b += 4 * nbp) {
        const TV v0 = ldx(src + (long long)b * n), v1 = ldx(src + (long long)(b + nbp) * n);
        const TV v2 = ldx(src + (long long)(b + 2 * nbp) * n), v3 = ldx(src + (long long)(b + 3 * nbp) * n);
        acc += (double)v0;
        acc += (double)v1;
        acc += (double)v2;
        acc += (double)v3;
      }
      for (; b < G; b += nbp) acc += (double)ldx(src + (long long)b * n);
    }
    for (int o = cwp; o < kWave; o <<= 1) acc += __shfl_xor(acc, o, kWave);
    if (cwp < kWave) {
      if ((tid & (kWave - 1)) < cwp) red[(tid / kWave) * cwp + c] = acc;
    } else {
      red[tid] = acc;
    }
    __syncthreads();
    if (tid < cwp && t0 + tid < nc) {
      const int k = cwp < kWave ? kW : nbp;
      double s = 0.0;
      for (int i = 0; i < k; ++i) s += red[i * cwp + tid];
      epi(t0 + tid, s);
    }
    __syncthreads();
  }
}

// LDS: X 8 (n + 1) | W 8 (rows + 1) | rho 8 rows | PP 8 cw | sums 8 kT | red |
// AP, U: CG precision, rows each | slice offsets and row lists | resident copies
__host__ __device__ inline size_t run_lds_list(int lgT, int ns) {
  return 4 * ((size_t)ns + 1) + 2 * (size_t)ns * (kWave >> lgT);
}
template <typename V>
__host__ __device__ inline size_t run_lds_vec(int n, int rows, int cw) {
  return 8 * ((size_t)n + 1) + 8 * ((size_t)rows + 1) + 8 * (size_t)rows + 8 * (size_t)cw + 8 * kT + 8 * 4 * kW +
         2 * sizeof(V) * (size_t)rows;
}

template <typename V, int NE, bool RES>
__global__ __launch_bounds__(kT) void k_admm_run(RunArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ int flag;
  const int tid = threadIdx.x, b = blockIdx.x, n = a.n, G = a.G;
  const RunCall& c = a.c;
  const int r0 = a.r0[b], nr = a.r0[b + 1] - r0;
  const int c0 = b * a.cw < n ? b * a.cw : n, nc = (n - c0) < a.cw ? (n - c0) : a.cw;
  double* X = (double*)lds;  // n + 1: p (CG precision), x64 or column sums
  V* p = (V*)lds;
  double* W = X + n + 1;     // rows + 1: w64, or w in the CG precision
  V* Wv = (V*)W;
  double* RH = W + a.rows_max + 1;
  double* PP = RH + a.rows_max;
  double* sums = PP + a.cw;
  BlkRed red{sums + kT, 0};
  V* AP = (V*)(sums + kT + 4 * kW);
  V* U = AP + a.rows_max;
  char* at = lds + ((run_lds_vec<V>(n, a.rows_max, a.cw) + 15) & ~(size_t)15);
  // the copies' slice offsets, row lists and (RES) entries
  struct Op {
    int lgT, ns;
    int* soff;
    uint16_t* perm;
    const V* gval;
    const uint16_t* gcol;
    V* lval;
    uint16_t* lcol;
  };
  auto open = [&](const RunView& v) {
    Op o;
    o.lgT = v.lgT;
    o.ns = v.ns;
    o.soff = (int*)at;
    o.perm = (uint16_t*)(o.soff + v.ns + 1);
    const int np = v.ns * (kWave >> v.lgT);
    for (int i = tid; i <= v.ns; i += kT) o.soff[i] = v.soff[(long long)b * (v.ns + 1) + i];
    for (int i = tid; i < np; i += kT) o.perm[i] = v.perm[(long long)b * np + i];
    at += (run_lds_list(v.lgT, v.ns) + 15) & ~(size_t)15;
    o.gval = (const V*)v.val + v.base[b] * kWave;
    o.gcol = v.col + v.base[b] * kWave;
    o.lval = nullptr;
    o.lcol = nullptr;
    if constexpr (RES) {
      const int ents = (int)(v.base[b + 1] - v.base[b]) * kWave;
      o.lval = (V*)at;
      o.lcol = (uint16_t*)(o.lval + v.res);
      for (int i = tid; i < ents; i += kT) {
        o.lval[i] = o.gval[i];
        o.lcol[i] = o.gcol[i];
      }
      at += (size_t)v.res * (sizeof(V) + 2);
    }
    return o;
  };
  const Op oA = open(a.A), oT = open(a.At), oP = open(a.P);
  auto rows = [&](const Op& o, int rot, auto zero, auto x, auto epi) {
    using TX = decltype(zero);
    if constexpr (RES) run_rows<TX>(o.lgT, o.ns, rot, o.soff, o.perm, o.lval, o.lcol, x, epi);
    else run_rows<TX>(o.lgT, o.ns, rot, o.soff, o.perm, o.gval, o.gcol, x, epi);
  };
  for (int i = tid; i < nr; i += kT) RH[i] = c.rho[r0 + i];
  unsigned epoch = 0;
  auto barrier = [&]() -> bool { return grid_barrier(a, ++epoch, &flag); };
  V* part_v = (V*)a.part;
  double* r64g = a.xch;
  V* kpg = (V*)(a.xch + n);

  // loop state, the same in every workgroup (read before the first barrier,
  // written back by workgroup 0 after the last)
  double eps_prev = *c.st.eps_prev, red_factor = *c.st.red_factor;
  int zero_iters = *c.st.zero_iters, cg_iter = *c.st.iter, solves = *c.st.solves, zc = c.z_count;
  long long total = 0;
  const double sg = c.sigma, al = c.alpha;

  // w64 = rho o (A x64 - b2), b2 = z - y / rho
  for (int i = tid; i < nr; i += kT) {
    const int r = r0 + i;
    const double b2 = (-1.0) * (c.rhoinv[r] * c.y[r]) + 1.0 * c.z[r];
    W[i] = RH[i] * (c.ax64[r] - b2);
    U[i] = 0;
  }
  if (tid == 0) W[nr] = 0.0;
  __syncthreads();

  for (int itn = 0; itn < c.iters; ++itn) {
    // this range's share of A' w64
    rows(oT, 0, 0.0, (const double*)W, [&](int j, double s) { X[j] = s; });
    __syncthreads();
    for (int j = tid; j < n; j += kT) stx(a.part + (long long)b * n + j, X[j]);
    if (!barrier()) return;
    // r64 = sigma x64 + [P A'] [x64; w64] - b1, b1 = sigma x - q
    for (int j = tid; j < n; j += kT) X[j] = ldx(c.x64 + j);
    if (tid == 0) X[n] = 0.0;
    __syncthreads();
    rows(oP, 0, 0.0, (const double*)X, [&](int i, double s) { PP[i] = s; });
    __syncthreads();
    chunk_sum(a.part, n, G, c0, nc, a.lgcw, sums, [&](int i, double s) {
      const int j = c0 + i;
      stx(r64g + j, (sg * X[j] + (PP[i] + s)) - (sg * c.x[j] + (-1.0) * c.q[j]));
    });
    if (!barrier()) return;
    double rr[NE];
    double mx = 0.0;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      rr[e] = 0.0;
      if (j < n) rr[e] = ldx(r64g + j);
      const double t = fabs(rr[e]);
      mx = t > mx ? t : mx;
    }
    const double rn0 = red.max(mx);
    const double scale = (rn0 > 0.0 && isfinite(rn0)) ? rn0 : 1.0, inv = 1.0 / scale;
    // tolerance (cuda_pcg_interface.cu:32-64, :266-268)
    if (solves > 0) zero_iters = cg_iter == 0 ? zero_iters + 1 : 0;
    if (zero_iters >= c.reduction_threshold) {
      red_factor /= 2;
      zero_iters = 0;
    }
    double eps = red_factor * sqrt(c.spr * c.sdr);
    eps = eps < eps_prev ? eps : eps_prev;
    eps = eps > 1e-7 ? eps : 1e-7;
    eps_prev = eps;
    solves++;
    const double eps_cmp = eps / scale;
    // CG on K d = -r64 / scale
    V r[NE], pv[NE], d[NE], di[NE];
    double rty = 0.0, rn = 0.0;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      di[e] = j < n ? ((const V*)c.dinv)[j] : (V)0;
      r[e] = (V)(rr[e] * inv);
      const V y = di[e] * r[e];
      pv[e] = -y;
      d[e] = 0;
      if (j < n) p[j] = pv[e];
      rty += (double)(y * r[e]);
      const double t = fabs((double)r[e]);
      rn = t > rn ? t : rn;
    }
    if (tid == 0) p[n] = 0;
    red.sum_max(rty, rn);
    int it = 0;
    bool go = rn > eps_cmp && it < c.max_iter;
    if (c.guard && !(rty > 0.0 && isfinite(rty))) go = false;
    while (go) {
      __syncthreads();
      rows(oA, 0, (V)0, (const V*)p, [&](int i, V s) {
        AP[i] = s;
        Wv[i] = (V)RH[i] * s;
      });
      if (tid == 0) Wv[nr] = 0;
      rows(oP, oA.ns, (V)0, (const V*)p, [&](int i, V s) { PP[i] = (double)((V)sg * p[c0 + i]) + (double)s; });
      __syncthreads();
      rows(oT, 0, (V)0, (const V*)Wv, [&](int j, V s) { p[j] = s; });
      __syncthreads();
      V kp[NE];
      for (int j = tid; j < n; j += kT) stx(part_v + (long long)b * n + j, p[j]);
      if (!barrier()) return;
      chunk_sum((const V*)part_v, n, G, c0, nc, a.lgcw, sums, [&](int i, double s) { stx(kpg + c0 + i, (V)(PP[i] + s)); });
      if (!barrier()) return;
      double pkp = 0.0;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int j = tid + e * kT;
        kp[e] = 0;
        if (j < n) kp[e] = ldx(kpg + j);
        pkp += (double)(pv[e] * kp[e]);
      }
      pkp = red.sum(pkp);
      if (c.guard && !(pkp > 0.0 && isfinite(pkp))) break;
      const V alpha = (V)(rty / pkp);
      double rty_n = 0.0;
      rn = 0.0;
      V yv[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        d[e] += alpha * pv[e];
        r[e] += alpha * kp[e];
        yv[e] = di[e] * r[e];
        rty_n += (double)(yv[e] * r[e]);
        const double t = fabs((double)r[e]);
        rn = t > rn ? t : rn;
      }
      for (int i = tid; i < nr; i += kT) U[i] += alpha * AP[i];
      red.sum_max(rty_n, rn);
      const V beta = (V)(rty_n / rty);
      it++;
      rty = rty_n;
      go = rn > eps_cmp && it < c.max_iter;
      if (c.guard && !(rty > 0.0 && isfinite(rty))) go = false;
      if (go) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
          const int j = tid + e * kT;
          pv[e] = beta * pv[e] - yv[e];
          if (j < n) p[j] = pv[e];
        }
        if (tid == 0) p[n] = 0;
      }
    }
    cg_iter = it;
    total += it;
    // x64 += scale d; x, delta x of this workgroup's chunk
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      if (j >= c0 && j < c0 + nc) {
        double xi = ldx(c.x64 + j);
        if (it > 0) xi += scale * (double)d[e];
        stx(c.x64 + j, xi);
        const double xp = c.x[j], v = al * xi + (1.0 - al) * xp;
        c.x[j] = v;
        c.dx[j] = v - xp;
      }
    }
    // A x64: from the CG's own products (U = A d), exactly every kRunRefresh-th time
    const bool exact = zc >= kRunRefresh - 1;
    zc = exact ? 0 : zc + 1;
    if (exact) {
      if (!barrier()) return;
      for (int j = tid; j < n; j += kT) X[j] = ldx(c.x64 + j);
      if (tid == 0) X[n] = 0.0;
      __syncthreads();
      rows(oA, 0, 0.0, (const double*)X, [&](int i, double s) { W[i] = s; });
      __syncthreads();
    } else {
      __syncthreads();
    }
    for (int i = tid; i < nr; i += kT) {
      const int k = r0 + i;
      double ax = c.ax64[k];
      if (exact) ax = W[i];
      else if (it > 0) ax += scale * (double)U[i];
      c.ax64[k] = ax;
      const double zp = c.z[k], yp = c.y[k], rho = RH[i], rhoinv = c.rhoinv[k];
      double v = rhoinv * yp;
      v += al * ax + (1.0 - al) * zp;
      v = v > c.l[k] ? v : c.l[k];
      v = v < c.u[k] ? v : c.u[k];
      double dy = al * ax + (1.0 - al) * zp + (-1.0) * v;
      dy = dy * rho;
      c.z[k] = v;
      c.dy[k] = dy;
      const double yn = yp + dy;
      c.y[k] = yn;
      // the next iteration's w64
      const double b2 = (-1.0) * (rhoinv * yn) + 1.0 * v;
      W[i] = rho * (ax - b2);
      U[i] = 0;
    }
    if (tid == 0) W[nr] = 0.0;
    __syncthreads();
  }
  if (b == 0 && tid == 0) {
    *c.st.eps_prev = eps_prev;
    *c.st.red_factor = red_factor;
    *c.st.zero_iters = zero_iters;
    *c.st.iter = cg_iter;
    *c.st.solves = solves;
    *c.st.total_iters += total;
    *c.st.active = 0;
    *c.st.done = 1;
  }
}

// ---- one workgroup ---------------------------------------------------------------
// The same loop for problems of one workgroup, over A's rows and the rows of
// K = [P A'] as the column-panel kernels take them where one panel holds all
// columns: each row on the lanes, in the order and with the epilogue of those
// kernels, and every dot product in the blocks of theirs, so the iterates are
// theirs to the bit, up to n + m of one panel's columns (their FP32
// rounding decides where a CG stops on problems with tight equality
// constraints, and the ADMM iterates part after that).  FP64 recomputes A x64
// in every iteration, as the separate kernels do.

// wave_sum's bits, the two wide steps by shuffle instead of lane swaps and
// selects, which took two MPC steps of horizon 10 in FP64 from 4.86 to 4.96 ms
// (horizon 50 in FP32: 5.17 to 5.25)
__device__ __forceinline__ double wave_sum_xor(double v) {
  v += __shfl_xor(v, 32, kWave);
  v += __shfl_xor(v, 16, kWave);
  v += dpp_d<0x128, 0xf>(0.0, v);  // row_ror:8, 4, 2, 1
  v += dpp_d<0x124, 0xf>(0.0, v);
  v += dpp_d<0x122, 0xf>(0.0, v);
  v += dpp_d<0x121, 0xf>(0.0, v);
  return v;
}
// Total of NB * 16 wavefronts' values w[]: blocks of four wavefronts added in
// order, then the blocks by a butterfly (the partials of 256-thread blocks,
// as the consumers of the separate kernels add them).
template <int NB>
__device__ __forceinline__ double blocks_total(const double* w) {
  double p[4 * NB];
#pragma unroll
  for (int k = 0; k < 4 * NB; ++k) p[k] = ((w[4 * k] + w[4 * k + 1]) + w[4 * k + 2]) + w[4 * k + 3];
#pragma unroll
  for (int o = 2 * NB; o > 0; o >>= 1)
#pragma unroll
    for (int k = 0; k < o; ++k) p[k] = p[k] + p[k + o];
  return p[0];
}

// FP32 products of one lane: compensated, as in the separate kernels
template <typename V>
struct LaneDot {
  double s = 0.0;
  __device__ __forceinline__ void add(double v) { s += v; }
  __device__ __forceinline__ double value() const { return s; }
};
template <>
struct LaneDot<float> {
  float s = 0.0f, c = 0.0f;
  __device__ __forceinline__ void add(float v) {
    const float y = v - c, t = s + y;
    c = (t - s) - y;
    s = t;
  }
  __device__ __forceinline__ double value() const { return (double)s - (double)c; }
};

constexpr int kU1 = 16;  // steps in flight: a row of the MPC's [P A'] in one round
// run_rows with the lanes per row of each slice beside its first step; a row's
// lanes are added in the panel kernel's order (its shuffle-down tree)
template <typename TX, typename VP, typename CP, typename X, typename Epi>
__device__ __forceinline__ void run1_rows(const int ns, const int2* sl, const uint16_t* perm, VP val, CP col, X x,
                                          Epi epi) {
  const int lane = threadIdx.x & (kWave - 1);
  for (int s = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); s < ns; s += kW) {
    const int s0 = __builtin_amdgcn_readfirstlane(sl[s].x), s1 = __builtin_amdgcn_readfirstlane(sl[s + 1].x);
    const int meta = __builtin_amdgcn_readfirstlane(sl[s].y), lgT = meta & 7, row0 = meta >> 3;
    const int row = perm[row0 + (lane >> lgT)];
    TX acc = 0;
    int i = s0;
    for (; i + kU1 <= s1; i += kU1) {
      TX v[kU1];
      int c[kU1];
#pragma unroll
      for (int q = 0; q < kU1; ++q) {
        v[q] = (TX)val[(i + q) * kWave + lane];
        c[q] = col[(i + q) * kWave + lane];
      }
#pragma unroll
      for (int q = 0; q < kU1; ++q) acc += v[q] * x[c[q]];
    }
    if (i < s1) {
      TX v[kU1];
      int c[kU1];
#pragma unroll
      for (int q = 0; q < kU1 - 1; ++q)
        if (i + q < s1) {
          v[q] = (TX)val[(i + q) * kWave + lane];
          c[q] = col[(i + q) * kWave + lane];
        }
#pragma unroll
      for (int q = 0; q < kU1 - 1; ++q)
        if (i + q < s1) acc += v[q] * x[c[q]];
    }
    for (int o = (1 << lgT) >> 1; o > 0; o >>= 1) acc += __shfl_xor(acc, o, kWave);
    if (row != kNoRow && (lane & ((1 << lgT) - 1)) == 0) epi(row, acc);
  }
}

// LDS: XW 8 (n + m + 1) | R 8 n | rho 8 m | sums | AP, U | lists | copies
template <typename V>
__host__ __device__ inline size_t run1_lds_vec(int n, int m) {
  return 8 * ((size_t)n + m + 1) + 8 * (size_t)n + 8 * (size_t)m + 8 * 2 * 4 * kW + 2 * sizeof(V) * (size_t)m;
}
__host__ __device__ inline size_t run1_lds_list(int ns, int slots) { return 8 * ((size_t)ns + 1) + 2 * (size_t)slots; }

// RES: 0 both copies read from memory, 1 A's in LDS, 2 both in LDS
template <typename V, int NE, int RES>
__global__ __launch_bounds__(kT) void k_admm_run1(RunArgs a) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int tid = threadIdx.x, n = a.n, m = a.m, lane = tid & (kWave - 1), wv = tid / kWave;
  const RunCall& c = a.c;
  double* XW = (double*)lds;  // [x64; w64], or [p; w] in the CG precision, and a zero slot
  V* pw = (V*)lds;
  double* R = XW + n + m + 1;  // r64, or K p in the CG precision
  V* KP = (V*)R;
  double* RH = R + n;
  double* red = RH + m;        // two turns of up to 4 kW values
  V* AP = (V*)(red + 2 * 4 * kW);
  V* U = AP + m;
  char* at = lds + ((run1_lds_vec<V>(n, m) + 15) & ~(size_t)15);
  struct Op {
    int ns;
    int2* sl;  // first step and lanes per row (log2) of each slice
    uint16_t* perm;
    const V* gval;
    const uint16_t* gcol;
    V* lval;
    uint16_t* lcol;
  };
  auto open = [&](const RunView& v, bool res) {
    Op o;
    o.ns = v.ns;
    o.sl = (int2*)at;
    o.perm = (uint16_t*)(o.sl + v.ns + 1);
    for (int i = tid; i <= v.ns; i += kT) o.sl[i] = ((const int2*)v.soff)[i];
    for (int i = tid; i < v.slots; i += kT) o.perm[i] = v.perm[i];
    at += (run1_lds_list(v.ns, v.slots) + 15) & ~(size_t)15;
    o.gval = (const V*)v.val;
    o.gcol = v.col;
    o.lval = nullptr;
    o.lcol = nullptr;
    if (res) {
      o.lval = (V*)at;
      o.lcol = (uint16_t*)(o.lval + v.res);
      for (int i = tid; i < v.res; i += kT) {
        o.lval[i] = o.gval[i];
        o.lcol[i] = o.gcol[i];
      }
      at += (size_t)v.res * (sizeof(V) + 2);
    }
    return o;
  };
  const Op oA = open(a.A, RES >= 1), oK = open(a.At, RES >= 2);
  auto rows_A = [&](auto zero, auto x, auto epi) {
    using TX = decltype(zero);
    if constexpr (RES >= 1) run1_rows<TX>(oA.ns, oA.sl, oA.perm, oA.lval, oA.lcol, x, epi);
    else run1_rows<TX>(oA.ns, oA.sl, oA.perm, oA.gval, oA.gcol, x, epi);
  };
  auto rows_K = [&](auto zero, auto x, auto epi) {
    using TX = decltype(zero);
    if constexpr (RES >= 2) run1_rows<TX>(oK.ns, oK.sl, oK.perm, oK.lval, oK.lcol, x, epi);
    else run1_rows<TX>(oK.ns, oK.sl, oK.perm, oK.gval, oK.gcol, x, epi);
  };
  // the FP64-vector products
  const Op oA2 = sizeof(V) == 4 ? open(a.A2, false) : oA, oK2 = sizeof(V) == 4 ? open(a.P, false) : oK;
  auto rows_A64 = [&](const double* x, auto epi) {
    if constexpr (sizeof(V) == 8) rows_A(0.0, x, epi);
    else run1_rows<double>(oA2.ns, oA2.sl, oA2.perm, oA2.gval, oA2.gcol, x, epi);
  };
  auto rows_K64 = [&](const double* x, auto epi) {
    if constexpr (sizeof(V) == 8) rows_K(0.0, x, epi);
    else run1_rows<double>(oK2.ns, oK2.sl, oK2.perm, oK2.gval, oK2.gcol, x, epi);
  };
  int turn = 0;
  auto next = [&]() -> double* { return red + 4 * kW * (turn++ & 1); };

  double eps_prev = *c.st.eps_prev, red_factor = *c.st.red_factor;
  int zero_iters = *c.st.zero_iters, cg_iter = *c.st.iter, solves = *c.st.solves, zc = c.z_count;
  long long total = 0;
  const double sg = c.sigma, al = c.alpha;
  // this thread's elements of x64 and of the loop's n-vectors
  double x64[NE], x[NE], q[NE], dx[NE];
  V di[NE];
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int j = tid + e * kT;
    x64[e] = x[e] = q[e] = dx[e] = 0.0;
    di[e] = 0;
    if (j < n) {
      x64[e] = c.x64[j];
      x[e] = c.x[j];
      q[e] = c.q[j];
      di[e] = ((const V*)c.dinv)[j];
      XW[j] = x64[e];
    }
  }
  for (int i = tid; i < m; i += kT) {
    const double rho = c.rho[i], b2 = (-1.0) * (c.rhoinv[i] * c.y[i]) + 1.0 * c.z[i];
    RH[i] = rho;
    XW[n + i] = rho * (c.ax64[i] - b2);
    U[i] = 0;
  }
  if (tid == 0) XW[n + m] = 0.0;
  __syncthreads();

  for (int itn = 0; itn < c.iters; ++itn) {
    // r64 = sigma x64 + [P A'] [x64; w64] - b1, b1 = sigma x - q
    rows_K64((const double*)XW, [&](int j, double s) { R[j] = sg * XW[j] + s; });
    __syncthreads();
    double rr[NE], mx = 0.0;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      rr[e] = j < n ? R[j] - (sg * x[e] + (-1.0) * q[e]) : 0.0;
      const double t = fabs(rr[e]);
      mx = t > mx ? t : mx;
    }
    double* w = next();
    mx = wave_max63(mx);
    if (lane == kWave - 1) w[wv] = mx;
    __syncthreads();
    double rn0 = w[0];
#pragma unroll
    for (int i = 1; i < kW; ++i) rn0 = w[i] > rn0 ? w[i] : rn0;
    const double scale = (rn0 > 0.0 && isfinite(rn0)) ? rn0 : 1.0, inv = 1.0 / scale;
    // tolerance (cuda_pcg_interface.cu:32-64, :266-268)
    if (solves > 0) zero_iters = cg_iter == 0 ? zero_iters + 1 : 0;
    if (zero_iters >= c.reduction_threshold) {
      red_factor /= 2;
      zero_iters = 0;
    }
    double eps = red_factor * sqrt(c.spr * c.sdr);
    eps = eps < eps_prev ? eps : eps_prev;
    eps = eps > 1e-7 ? eps : 1e-7;
    eps_prev = eps;
    solves++;
    const double eps_cmp = eps / scale;
    // r'y and max|r| of the lanes' elements
    double rty, rn;
    auto rty_rn = [&](const V (&rv)[NE], const V (&yv)[NE]) {
      double* t = next();
      double m1 = 0.0;
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const double v = wave_sum_xor((double)(yv[e] * rv[e]));
        if (lane == 0) t[e * kW + wv] = v;
        const double f = fabs((double)rv[e]);
        m1 = f > m1 ? f : m1;
      }
      m1 = wave_max63(m1);
      if (lane == kWave - 1) t[NE * kW + wv] = m1;
      __syncthreads();
      rty = blocks_total<NE>(t);
      rn = t[NE * kW];
#pragma unroll
      for (int i = 1; i < kW; ++i) rn = t[NE * kW + i] > rn ? t[NE * kW + i] : rn;
    };
    // CG on K d = -r64 / scale
    V r[NE], y[NE], pv[NE], d[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      r[e] = (V)(rr[e] * inv);
      y[e] = di[e] * r[e];
      pv[e] = -y[e];
      d[e] = 0;
      if (j < n) pw[j] = pv[e];
    }
    if (tid == 0) pw[n + m] = 0;
    rty_rn(r, y);
    int it = 0;
    bool go = rn > eps_cmp && it < c.max_iter;
    if (c.guard && !(rty > 0.0 && isfinite(rty))) go = false;
    while (go) {
      rows_A((V)0, (const V*)pw, [&](int i, V s) {
        AP[i] = s;
        pw[n + i] = (V)RH[i] * s;
      });
      __syncthreads();
      rows_K((V)0, (const V*)pw, [&](int j, V s) { KP[j] = (V)sg * pw[j] + s; });
      __syncthreads();
      // p'Kp: RB rows a lane where n divides, as the combine kernel takes them
      constexpr int RB = 16 / (int)sizeof(V);
      double* t = next();
      V kp[NE];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int j = tid + e * kT;
        kp[e] = j < n ? KP[j] : (V)0;
      }
      if (n % RB == 0) {
        LaneDot<V> dot;
        if (tid < n / RB)
#pragma unroll
          for (int k = 0; k < RB; ++k) dot.add(pw[RB * tid + k] * KP[RB * tid + k]);
        const double v = wave_sum_xor(dot.value());
        if (lane == 0) t[wv] = v;
      } else {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
          const double v = wave_sum_xor((double)(pv[e] * kp[e]));
          if (lane == 0) t[e * kW + wv] = v;
        }
      }
      __syncthreads();
      const double pkp = n % RB == 0 ? blocks_total<1>(t) : blocks_total<NE>(t);
      if (c.guard && !(pkp > 0.0 && isfinite(pkp))) break;
      const V alpha = (V)(rty / pkp);
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        d[e] += alpha * pv[e];
        r[e] += alpha * kp[e];
        y[e] = di[e] * r[e];
      }
      for (int i = tid; i < m; i += kT) U[i] += alpha * AP[i];
      const double rty_old = rty;
      rty_rn(r, y);
      const V beta = (V)(rty / rty_old);
      it++;
      go = rn > eps_cmp && it < c.max_iter;
      if (c.guard && !(rty > 0.0 && isfinite(rty))) go = false;
      if (go) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
          const int j = tid + e * kT;
          pv[e] = beta * pv[e] - y[e];
          if (j < n) pw[j] = pv[e];
        }
        __syncthreads();
      }
    }
    cg_iter = it;
    total += it;
    // every reader of [p; w] is past a barrier: the region takes x64 again
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const int j = tid + e * kT;
      if (it > 0) x64[e] += scale * (double)d[e];
      const double v = al * x64[e] + (1.0 - al) * x[e];
      dx[e] = v - x[e];
      x[e] = v;
      if (j < n) XW[j] = x64[e];
    }
    const bool exact = sizeof(V) == 8 || zc >= kRunRefresh - 1;
    zc = exact ? 0 : zc + 1;
    if (exact) {
      __syncthreads();
      rows_A64((const double*)XW, [&](int i, double s) { c.ax64[i] = s; });
      __syncthreads();
    }
    for (int i = tid; i < m; i += kT) {
      double ax = c.ax64[i];
      if (!exact) {
        if (it > 0) ax += scale * (double)U[i];
        c.ax64[i] = ax;
      }
      const double zp = c.z[i], yp = c.y[i], rho = RH[i], rhoinv = c.rhoinv[i];
      double v = rhoinv * yp;
      v += al * ax + (1.0 - al) * zp;
      v = v > c.l[i] ? v : c.l[i];
      v = v < c.u[i] ? v : c.u[i];
      double dy = al * ax + (1.0 - al) * zp + (-1.0) * v;
      dy = dy * rho;
      c.z[i] = v;
      c.dy[i] = dy;
      const double yn = yp + dy;
      c.y[i] = yn;
      const double b2 = (-1.0) * (rhoinv * yn) + 1.0 * v;
      XW[n + i] = rho * (ax - b2);
      U[i] = 0;
    }
    if (tid == 0) XW[n + m] = 0.0;
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const int j = tid + e * kT;
    if (j < n) {
      c.x64[j] = x64[e];
      c.x[j] = x[e];
      c.dx[j] = dx[e];
    }
  }
  if (tid == 0) {
    *c.st.eps_prev = eps_prev;
    *c.st.red_factor = red_factor;
    *c.st.zero_iters = zero_iters;
    *c.st.iter = cg_iter;
    *c.st.solves = solves;
    *c.st.total_iters += total;
    *c.st.active = 0;
    *c.st.done = 1;
  }
}

__global__ void k_zero_words(unsigned* p, int k) {
  for (int i = threadIdx.x; i < k; i += blockDim.x) p[i] = 0;
}

constexpr int kBarWords = 17 * 64;

// What a launch of several workgroups changes in place, copied before it (and
// back when it gave up): x, x64, z, y, A x64 and the PCG's state.  With
// delta x and delta y, which a later iteration writes whole, that is all.
size_t run_save_len(int n, int m, int state_len) { return 2 * (size_t)n + 3 * (size_t)m + (size_t)state_len; }
__global__ void k_run_save(int n, int m, int state_len, RunCall c, double* save, int back) {
  const long long total = 2LL * n + 3LL * m + state_len;
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long long)gridDim.x * blockDim.x) {
    long long k = i;
    double* p;
    if (k < n) p = c.x + k;
    else if ((k -= n) < n) p = c.x64 + k;
    else if ((k -= n) < m) p = c.z + k;
    else if ((k -= m) < m) p = c.y + k;
    else if ((k -= m) < m) p = c.ax64 + k;
    else p = c.state + (k - m);
    if (back) *p = save[i];
    else save[i] = *p;
  }
}

// copies in LDS: n up to 4 kT (runner_build)
template <typename V, int NE>
const void* run_kernel(bool res) {
  if constexpr (NE <= 4)
    if (res) return (const void*)k_admm_run<V, NE, true>;
  return (const void*)k_admm_run<V, NE, false>;
}
template <typename V>
const void* run_kernel_n(int n, bool res) {
  if (n <= 1 * kT) return run_kernel<V, 1>(res);
  if (n <= 2 * kT) return run_kernel<V, 2>(res);
  if (n <= 4 * kT) return run_kernel<V, 4>(res);
  if constexpr (sizeof(V) == 4)
    if (n > 8 * kT) return run_kernel<V, 12>(res);
  return run_kernel<V, 8>(res);  // all of FP64's
}
template <typename V, int NE>
const void* run1_kernel(int res) {
  return res == 2 ? (const void*)k_admm_run1<V, NE, 2> : res == 1 ? (const void*)k_admm_run1<V, NE, 1>
                                                                  : (const void*)k_admm_run1<V, NE, 0>;
}
template <typename V>
const void* run1_kernel_n(int n, int res) {
  return n <= kT ? run1_kernel<V, 1>(res) : run1_kernel<V, 2>(res);
}
const void* kernel_of(const Runner* r) {
  if (r->G > 1) return r->bits == 32 ? run_kernel_n<float>(r->n, r->resident) : run_kernel_n<double>(r->n, r->resident);
  return r->bits == 32 ? run1_kernel_n<float>(r->n, r->resident) : run1_kernel_n<double>(r->n, r->resident);
}
int run_n_max(int bits) { return bits == 32 ? 12 * kT : 8 * kT; }

void free_op(RunOp* o) {
  dev_free(o->soff);
  dev_free(o->perm);
  dev_free(o->base);
  dev_free(o->col);
  dev_free(o->val);
}

// lanes per row: enough to give every lane of the workgroup a row share, at
// most half an average row's entries; more where build_op finds a longer chain
int pick_lgT(long long rows, double len) {
  int lg = 0;
  while (lg < 6 && (rows << lg) < kT && (2 << lg) <= len / 2) ++lg;
  return lg;
}

template <RunKind K>
RunSrc run_src(const Runner* r, const OSQPMatrix* M) {
  return RunSrc{r->n, r->cw, K == kColsA ? M->trp : M->rp, K == kColsA ? M->tci : M->ci, K == kColsA ? M->tval : M->val,
                r->r0, r->cs};
}

// padding at most as much as the entries, and no workgroup far above its share
bool op_fits(const Runner* r, const RunOp& o, long long nnz) {
  return o.steps * kWave <= 2 * nnz + 4096LL * r->G && o.max_steps <= 64 + 4 * (nnz / kWave / r->G + 1);
}

// slices of one copy; 1 on an allocation failure, 2 when it does not fit.  Each lane adds up a chain of
// its row's entries, then the lanes are added by a tree.  In a panel task of
// rows of one length, up to 64 lanes' worth, a chain is at most 24 entries long
// in FP32; so that the error of a sum is no larger here, a copy takes more lanes
// a row than pick_lgT's until no row's chain is longer than that (a copy that
// does not fit on pick_lgT's lanes is not taken on more).
template <RunKind K>
int build_op(Runner* r, RunOp* o, const OSQPMatrix* M, int* d_steps, int* h_steps) {
  const int rows = K == kColsA ? r->n : K == kRowsA ? r->rows_max : r->cw, G = r->G;
  o->slots = 0;
  o->lgT = pick_lgT(rows, (double)M->nnz / ((double)G * (rows > 0 ? rows : 1)));
  int N = 1;
  while (N < rows) N <<= 1;
  const size_t kb = sizeof(unsigned) * (size_t)N;
  if (kb > 48 * 1024)
    HIPCHK(hipFuncSetAttribute((const void*)k_run_layout<K>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kb));
  o->base = (long long*)dev_try_alloc(sizeof(long long) * (G + 1));
  if (!o->base) return 1;
  for (;; ++o->lgT) {
    const int per = kWave >> o->lgT;
    o->ns = (rows + per - 1) / per;
    if (o->ns < 1) o->ns = 1;
    o->soff = (int*)dev_try_alloc(sizeof(int) * (size_t)G * (o->ns + 1));
    o->perm = (uint16_t*)dev_try_alloc(sizeof(uint16_t) * (size_t)G * o->ns * per);
    if (!o->soff || !o->perm) return 1;
    hipLaunchKernelGGL((k_run_layout<K>), dim3(G), dim3(kT), kb, S(), run_src<K>(r, M), o->lgT, o->ns, o->soff, o->perm,
                       d_steps);
    download(h_steps, d_steps, sizeof(int) * 2 * G);
    int chain = 0;
    o->steps = o->max_steps = 0;
    for (int b = 0; b < G; ++b) {
      chain = std::max(chain, h_steps[G + b]);
      o->steps += h_steps[b];
      o->max_steps = std::max(o->max_steps, h_steps[b]);
    }
    if (!op_fits(r, *o, M->nnz)) return 2;
    if (chain <= kRunChain || o->lgT == 6) {
      r->chain = std::max(r->chain, chain);
      break;
    }
    dev_free(o->soff);
    dev_free(o->perm);
    o->soff = nullptr;
    o->perm = nullptr;
  }
  std::vector<long long> base((size_t)G + 1, 0);
  for (int b = 0; b < G; ++b) base[(size_t)b + 1] = base[(size_t)b] + h_steps[b];
  upload(o->base, base.data(), sizeof(long long) * base.size());
  return 0;
}

int alloc_op(Runner* r, RunOp* o) {
  const size_t e = (size_t)(o->steps > 0 ? o->steps : 1) * kWave;
  o->col = (uint16_t*)dev_try_alloc(sizeof(uint16_t) * e);
  o->val = dev_try_alloc((size_t)(r->bits / 8) * e);
  return !o->col || !o->val;
}

template <RunKind K>
void fill_op(Runner* r, RunOp* o, const OSQPMatrix* M, bool cols) {
  uint16_t* col = cols ? o->col : nullptr;
  if (r->bits == 32)
    hipLaunchKernelGGL((k_run_fill<K, float>), dim3(r->G), dim3(kT), 0, S(), run_src<K>(r, M), o->lgT, o->ns,
                       (const int*)o->soff, (const uint16_t*)o->perm, (const long long*)o->base, col, (float*)o->val);
  else
    hipLaunchKernelGGL((k_run_fill<K, double>), dim3(r->G), dim3(kT), 0, S(), run_src<K>(r, M), o->lgT, o->ns,
                       (const int*)o->soff, (const uint16_t*)o->perm, (const long long*)o->base, col, (double*)o->val);
}
void fill_A(Runner* r, const OSQPMatrix* A, bool cols) {
  fill_op<kRowsA>(r, &r->A, A, cols);
  fill_op<kColsA>(r, &r->At, A, cols);
  r->ver_A = A->version;
}
void fill_P(Runner* r, const OSQPMatrix* P, bool cols) {
  fill_op<kRowsP>(r, &r->P, P, cols);
  r->ver_P = P->version;
}

RunView view(const RunOp& o) {
  return RunView{o.lgT, o.ns, o.slots, o.max_steps * kWave, o.soff, o.perm, o.base, o.col, o.val};
}

// ---- one workgroup -----------------------------------------------------------
// Slices of a CSR's rows (rp on the host): a row's lanes are those that the
// column-panel kernel gives it, from the row count of its task (panel_build's
// greedy ranges for one panel), and rows of equal lanes are sorted by length.
int build_op1(RunOp* o, const std::vector<int>& rp, int bits) {  // bits: of the panels
  const int rows = (int)rp.size() - 1, V = bits == 32 ? 4 : 2, cap = 64 * (bits == 32 ? 12 : 6) - (V - 1);
  std::vector<int> lg((size_t)rows), order((size_t)rows);
  auto task = [&](int a, int b) {
    const int nr = b - a;
    int l = 6;
    while (l > 0 && (nr << l) > kWave) --l;
    for (int i = a; i < b; ++i) lg[(size_t)i] = l;
  };
  int cur = 0;
  for (int i = 0; i < rows; ++i) {
    if (rp[i + 1] - rp[i] > cap) {
      if (i > cur) task(cur, i);
      task(i, i + 1);
      cur = i + 1;
    } else if (i > cur && (rp[i + 1] - rp[cur] > cap || i - cur >= kPanelRowCap)) {
      task(cur, i);
      cur = i;
    }
  }
  if (cur < rows) task(cur, rows);
  auto steps = [&](int i) { return (rp[i + 1] - rp[i] + (1 << lg[(size_t)i]) - 1) >> lg[(size_t)i]; };
  for (int i = 0; i < rows; ++i) order[(size_t)i] = i;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
    return lg[(size_t)a] != lg[(size_t)b] ? lg[(size_t)a] < lg[(size_t)b] : steps(a) > steps(b);
  });
  std::vector<int2> sl;
  std::vector<uint16_t> perm;
  int at = 0;
  for (int i = 0; i < rows;) {
    const int l = lg[(size_t)order[(size_t)i]], per = kWave >> l;
    sl.push_back(make_int2(at, (int)(perm.size() << 3) | l));
    at += steps(order[(size_t)i]);
    for (int k = 0; k < per; ++k) {
      const bool in = i < rows && lg[(size_t)order[(size_t)i]] == l;
      perm.push_back(in ? (uint16_t)order[(size_t)i] : kNoRow);
      if (in) ++i;
    }
  }
  o->ns = (int)sl.size();
  o->slots = (int)perm.size();
  sl.push_back(make_int2(at, 0));
  o->steps = o->max_steps = at;
  o->soff = (int*)dev_try_alloc(sizeof(int2) * sl.size());
  o->perm = (uint16_t*)dev_try_alloc(sizeof(uint16_t) * (perm.empty() ? 1 : perm.size()));
  if (!o->soff || !o->perm) return 1;
  upload(o->soff, sl.data(), sizeof(int2) * sl.size());
  upload(o->perm, perm.data(), sizeof(uint16_t) * perm.size());
  return 0;
}
void fill_op1(const Runner* r, const RunOp& o, const int* rp, const int* ci, const double* src, bool cols) {
  uint16_t* col = cols ? o.col : nullptr;
  const int g = (o.ns + kW - 1) / kW;
  if (r->bits == 32)
    hipLaunchKernelGGL(k_run1_fill<float>, dim3(g), dim3(kT), 0, S(), o.ns, rp, ci, src, (const int2*)o.soff,
                       (const uint16_t*)o.perm, r->n + r->m, col, (float*)o.val);
  else
    hipLaunchKernelGGL(k_run1_fill<double>, dim3(g), dim3(kT), 0, S(), o.ns, rp, ci, src, (const int2*)o.soff,
                       (const uint16_t*)o.perm, r->n + r->m, col, (double*)o.val);
}
void fill1(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, bool cols) {
  fill_op1(r, r->A, A->rp, A->ci, A->val, cols);
  fill_op1(r, r->At, k.rp, k.ci, k.val, cols);
  if (r->bits == 32) {
    fill_op1(r, r->A2, A->rp, A->ci, A->val, cols);
    fill_op1(r, r->P, k.rp, k.ci, k.val, cols);
  }
  r->ver_A = A->version;
  r->ver_P = P->version;
}
// 1 on an allocation failure; r->G = 0 when the problem does not fit
int build1(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k) {
  const int n = r->n, m = r->m;
  std::vector<int> arp((size_t)m + 1), krp((size_t)n + 1);
  download(arp.data(), A->rp, sizeof(int) * arp.size());
  download(krp.data(), k.rp, sizeof(int) * krp.size());
  if (build_op1(&r->A, arp, r->bits) || build_op1(&r->At, krp, r->bits)) return 1;
  if (r->bits == 32 && (build_op1(&r->A2, arp, 64) || build_op1(&r->P, krp, 64))) return 1;
  const size_t slot = (size_t)r->bits / 8 + 2, copyA = r->A.steps * kWave * slot, copyK = r->At.steps * kWave * slot;
  r->lds = r->bits == 32 ? run1_lds_vec<float>(n, m) : run1_lds_vec<double>(n, m);
  for (const RunOp* o : {&r->A, &r->At, &r->P, &r->A2}) r->lds += run1_lds_list(o->ns, o->slots) + 16;
  const bool pads = r->A.steps * kWave <= 2LL * A->nnz + 4096 && r->At.steps * kWave <= 2LL * krp[(size_t)n] + 4096;
  if (!pads || r->lds > kRunLds) {
    r->G = 0;
    return 0;
  }
  if (r->lds + copyA <= kRunLds) {
    r->resident = 1;
    r->lds += copyA;
    if (r->lds + copyK <= kRunLds) {
      r->resident = 2;
      r->lds += copyK;
    }
  }
  if (alloc_op(r, &r->A) || alloc_op(r, &r->At) || alloc_op(r, &r->A2) || alloc_op(r, &r->P)) return 1;
  fill1(r, A, P, k, true);
  return 0;
}

}  // namespace

void runner_free(Runner* r) {
  free_op(&r->A);
  free_op(&r->At);
  free_op(&r->P);
  free_op(&r->A2);
  dev_free(r->r0);
  dev_free(r->cs);
  dev_free(r->part);
  dev_free(r->xch);
  dev_free(r->bar);
  dev_free(r->save);
  memset(r, 0, sizeof(*r));
}

// several workgroups: 1 on an allocation failure; r->G = 0 when it does not fit
static int build_many(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P) {
  const int n = r->n, G = r->G;
  r->cw = (n + G - 1) / G;
  r->r0 = (int*)dev_try_alloc(sizeof(int) * (G + 2));
  r->cs = (int*)dev_try_alloc(sizeof(int) * (size_t)(G + 1) * n);
  struct Steps {
    int* p;
    ~Steps() { dev_free(p); }
  } d_steps{(int*)dev_try_alloc(sizeof(int) * 2 * G)};
  std::vector<int> h(2 * (size_t)G + 2);
  int rc = !r->r0 || !r->cs || !d_steps.p;
  bool fits = !rc;
  if (!rc) {
    const int one = 1;
    upload(r->r0 + G + 1, &one, sizeof(int));
    hipLaunchKernelGGL(k_run_ranges, dim3((G + kBlock) / kBlock), dim3(kBlock), 0, S(), r->m, G, (const int*)A->rp, r->r0);
    hipLaunchKernelGGL(k_run_sorted, dim3(grid_for((long long)n * kWave, kBlock, 4096)), dim3(kBlock), 0, S(), n,
                       (const int*)A->trp, (const int*)A->tci, r->r0 + G + 1);
    hipLaunchKernelGGL(k_run_cuts, dim3(grid_for((long long)(G + 1) * n, kBlock, 4096)), dim3(kBlock), 0, S(), n, G,
                       (const int*)A->trp, (const int*)A->tci, (const int*)r->r0, r->cs);
    download(h.data(), r->r0, sizeof(int) * ((size_t)G + 2));
    for (int b = 0; b < G; ++b) r->rows_max = std::max(r->rows_max, h[(size_t)b + 1] - h[(size_t)b]);
    r->lds = r->bits == 32 ? run_lds_vec<float>(n, r->rows_max, r->cw) : run_lds_vec<double>(n, r->rows_max, r->cw);
    fits = h[(size_t)G + 1] == 1 && r->rows_max < kSortMax && r->lds <= kRunLds;
  }
  if (fits) {
    rc = build_op<kRowsA>(r, &r->A, A, d_steps.p, h.data());
    if (!rc) rc = build_op<kColsA>(r, &r->At, A, d_steps.p, h.data());
    if (!rc) rc = build_op<kRowsP>(r, &r->P, P, d_steps.p, h.data());
    for (const RunOp* o : {&r->A, &r->At, &r->P}) r->lds = ((r->lds + 15) & ~(size_t)15) + run_lds_list(o->lgT, o->ns) + 16;
    fits = !rc && r->lds <= kRunLds;
    if (rc == 2) rc = 0;
  }
  if (rc || !fits) {
    r->G = 0;
    return rc;
  }
  r->part = (double*)dev_try_alloc(sizeof(double) * (size_t)G * n);
  r->xch = (double*)dev_try_alloc(sizeof(double) * 2 * (size_t)n);
  r->bar = (unsigned*)dev_try_alloc(sizeof(unsigned) * kBarWords);
  r->save = (double*)dev_try_alloc(sizeof(double) * run_save_len(n, r->m, r->state_len));
  if (alloc_op(r, &r->A) || alloc_op(r, &r->At) || alloc_op(r, &r->P) || !r->part || !r->xch || !r->bar || !r->save) return 1;
  fill_A(r, A, true);
  fill_P(r, P, true);
  const size_t copies = ((size_t)r->A.max_steps + r->At.max_steps + r->P.max_steps) * kWave * ((size_t)r->bits / 8 + 2);
  if (n <= 4 * kT && r->lds + copies <= kRunLds) {
    r->resident = 1;
    r->lds += copies;
  }
  return 0;
}

static int build_any(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, int bits, bool one, int state_len) {
  const int n = A->n, m = A->m;
  if (A->is_triu || n <= 0 || m <= 0 || A->nnz <= 0 || n > run_n_max(bits)) return 0;
  const long long work = (long long)A->nnz + P->nnz;
  if (work > kRunMaxWork) return 0;
  const int cus = rt().num_cu > 0 ? rt().num_cu : 256;
  int rc = 0;
  if (work <= kRun1Work && n <= 2 * kT && n + m < 65535) {
    r->n = n;
    r->m = m;
    r->bits = bits;
    r->G = 1;
    rc = build1(r, A, P, k);
    if (rc || r->G == 0) runner_free(r);
  }
  if (!rc && r->G == 0 && !one) {
    // Measured us per ADMM iteration with G = 32 / 64 / 128 / 256 workgroups:
    // 108k entries 33 / - / - / -, 180k 39 / 36 / 37 / 39, 624k 52 / 48 / 43 /
    // 46, 1.4M 62 / 50 / 46 / 48 (FP64): a workgroup's share against the
    // barrier and the G shares to add.  256 workgroups against the separate
    // kernels: 5 M entries 108 and 148, 16 M 250 and 276, 30 M (8000 columns)
    // 426 and 431, 60 M 660 and 884.
    int G = work <= 128000 ? 32 : work <= 400000 ? 64 : work <= 2000000 ? 128 : 256;
    while (G > cus) G /= 2;
    r->n = n;
    r->m = m;
    r->bits = bits;
    r->G = G;
    r->state_len = state_len;
    rc = build_many(r, A, P);
  }
  if (rc || r->G == 0) return 0;
  if (hipFuncSetAttribute(kernel_of(r), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kRunLds) != hipSuccess) {
    (void)hipGetLastError();
    return 0;
  }
  return LAUNCHCHK() == 0;
}

int runner_build(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, int bits, bool one, int state_len) {
  memset(r, 0, sizeof(*r));
  try {
    r->on = build_any(r, A, P, k, bits, one, state_len);
  } catch (const std::bad_alloc&) {
  }
  if (!r->on) runner_free(r);
  return r->on;
}

static void run_save(const Runner* r, const RunCall& c, int back) {
  const int g = grid_for((long long)run_save_len(r->n, r->m, r->state_len), kBlock, 1024);
  hipLaunchKernelGGL(k_run_save, dim3(g), dim3(kBlock), 0, S(), r->n, r->m, r->state_len, c, r->save, back);
}
void runner_restore(Runner* r, const RunCall& c) {
  run_save(r, c, 1);
}

int runner_run(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, const RunCall& c, int* z_count) {
  const bool many = r->G > 1;
  if (many) {
    if (r->ver_A != A->version) fill_A(r, A, false);
    if (r->ver_P != P->version) fill_P(r, P, false);
  } else if (r->ver_A != A->version || r->ver_P != P->version) {
    fill1(r, A, P, k, false);
  }
  RunArgs a;
  memset(&a, 0, sizeof(a));
  a.n = r->n;
  a.m = r->m;
  a.G = r->G;
  a.cw = r->cw;
  while ((1 << a.lgcw) < r->cw && (1 << a.lgcw) < kT) ++a.lgcw;
  a.rows_max = r->rows_max;
  a.r0 = r->r0;
  a.A = view(r->A);
  a.At = view(r->At);
  a.P = view(r->P);
  a.A2 = view(r->A2);
  a.part = r->part;
  a.xch = r->xch;
  a.bar = r->bar;
  a.polls = c.polls >= 0 ? c.polls : kRunPolls;
  a.c = c;
  void* args[] = {&a};
  hipError_t err;
  if (many) {
    run_save(r, c, 0);
    hipLaunchKernelGGL(k_zero_words, dim3(1), dim3(kBlock), 0, S(), r->bar, kBarWords);
    err = hipLaunchCooperativeKernel(kernel_of(r), dim3(r->G), dim3(kT), args, (unsigned)r->lds, S());
  } else {
    err = hipLaunchKernel(kernel_of(r), dim3(1), dim3(kT), args, r->lds, S());
  }
  if (err != hipSuccess) {
    (void)hipGetLastError();
    return 1;
  }
  *z_count = c.z_count;
  if (!many && r->bits == 64) return 0;  // A x64 is exact in every iteration
  for (int i = 0; i < c.iters; ++i) *z_count = *z_count >= kRunRefresh - 1 ? 0 : *z_count + 1;
  return 0;
}

}  // namespace osqp_hip
