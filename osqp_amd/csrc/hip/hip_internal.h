// hip_internal.h — shared definitions of the algebra/hip backend (gfx950).
//
// Storage model: every OSQP vector is an FP64 array in HBM; matrices keep
// CSR copies for the operator and its transpose (see matrix.hip).  All work
// is queued on one backend stream per process; calls returning host scalars
// synchronise that stream, nothing else does.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include "../../../include/osqp_amd_algebra.h"

namespace osqp_hip {

constexpr int kBlock = 256;          // threads per block for streaming kernels
constexpr int kMaxReduceBlocks = 2048;  // cap on per-block partials of a reduction
constexpr int kWave = 64;            // CDNA wavefront width

struct Runtime {
  int device = -1;
  int refcount = 0;
  hipStream_t stream = nullptr;
  double* h_scalars = nullptr;     // host-coherent slots for reduction results
  double* dh_scalars = nullptr;    // their device address
  double* d_partials = nullptr;    // per-block partials (4 * kMaxReduceBlocks doubles)
  unsigned* d_ticket = nullptr;    // finished-block counter of the running reduction
  double red_seq = 0.0;            // sequence number of the last reduction
  int last_error = 0;
  int num_cu = 0;
  char device_name[256] = {0};
};

Runtime& rt();

// Records (and prints once) a HIP failure; the public API keeps running and
// reports errors through return codes, never exit().
int check(hipError_t e, const char* what, const char* file, int line);
#define HIPCHK(x) ::osqp_hip::check((x), #x, __FILE__, __LINE__)
#define LAUNCHCHK() ::osqp_hip::check(hipGetLastError(), "kernel launch", __FILE__, __LINE__)

inline int grid_for(long long n, int per_block = kBlock, int cap = 65535 * 8) {
  long long g = (n + per_block - 1) / per_block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

inline int reduce_grid(long long n) {
  long long g = (n + kBlock * 4 - 1) / (kBlock * 4);
  if (g < 1) g = 1;
  if (g > kMaxReduceBlocks) g = kMaxReduceBlocks;
  return (int)g;
}

void* dev_alloc(size_t bytes);           // stream-ordered device allocation
void* dev_try_alloc(size_t bytes);       // the same; a failure is the caller's to handle and is not recorded
void dev_free(void* p);
void upload(void* dst, const void* src, size_t bytes);    // host or device src
void download(void* dst, const void* src, size_t bytes);  // host or device dst; syncs

// ---- block / wavefront reductions ----------------------------------------
// Sums and maxima over a wavefront whose lanes are all active, in the order of
// a butterfly of xor distances 32, 16, 8, 4, 2, 1: the two wide steps by
// v_permlane32_swap / v_permlane16_swap, the rest by DPP moves within rows of
// 16 lanes.  A sum takes row rotations there: the lanes that a rotation pairs
// hold the sums that the xor would pair.  A maximum takes the xor's own lanes:
// it keeps a lane's own NaN and passes over another lane's, so that with NaNs
// the lanes of a pair may hold different values.  Register moves only: a step
// through LDS (ds_bpermute) costs its latency, in a chain of six.  16 MPCs of
// horizon 180 on the batch engine's row groups: 35.3 to 33.7 ms in FP32, 55.4 to
// 51.5 in FP64.
template <typename T, typename F>
__device__ __forceinline__ T lane_words(T v, F f) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "4 or 8 bytes");
  if constexpr (sizeof(T) == 4) {
    return __builtin_bit_cast(T, f(__builtin_bit_cast(int, v)));
  } else {
    const long long x = __builtin_bit_cast(long long, v);
    const int lo = f((int)x), hi = f((int)(x >> 32));
    return __builtin_bit_cast(T, ((long long)hi << 32) | (long long)(unsigned)lo);
  }
}
// the value of lane l ^ 32 (WIDE = 32) or l ^ 16
template <int WIDE, typename T>
__device__ __forceinline__ T lane_xor_wide(T v) {
  const bool upper = (__lane_id() & WIDE) != 0;
  return lane_words(v, [&](int w) {
    if constexpr (WIDE == 32) {
      const auto r = __builtin_amdgcn_permlane32_swap(w, w, false, false);
      return (int)(upper ? r[0] : r[1]);
    } else {
      const auto r = __builtin_amdgcn_permlane16_swap(w, w, false, false);
      return (int)(upper ? r[0] : r[1]);
    }
  });
}
// row_ror:D within rows of 16 lanes
template <int D, typename T>
__device__ __forceinline__ T lane_ror(T v) {
  return lane_words(v, [](int w) { return __builtin_amdgcn_update_dpp(0, w, 0x120 + D, 0xf, 0xf, false); });
}

// the value of lane l ^ D, D = 8, 4, 2 or 1
template <int D, typename T>
__device__ __forceinline__ T lane_xor_row(T v) {
  return lane_words(v, [](int w) {
    if constexpr (D == 8) return __builtin_amdgcn_update_dpp(0, w, 0x128, 0xf, 0xf, false);  // row_ror:8
    else if constexpr (D == 2) return __builtin_amdgcn_update_dpp(0, w, 0x4E, 0xf, 0xf, false);  // quad_perm:[2,3,0,1]
    else if constexpr (D == 1) return __builtin_amdgcn_update_dpp(0, w, 0xB1, 0xf, 0xf, false);  // quad_perm:[1,0,3,2]
    else {
      static_assert(D == 4, "a distance within a row");
      const int lo = __builtin_amdgcn_update_dpp(0, w, 0x104, 0xf, 0x5, false);  // row_shl:4 into banks 0, 2
      return __builtin_amdgcn_update_dpp(lo, w, 0x114, 0xf, 0xa, false);         // row_shr:4 into banks 1, 3
    }
  });
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
  v += lane_xor_wide<32>(v);
  v += lane_xor_wide<16>(v);
  v += lane_ror<8>(v);
  v += lane_ror<4>(v);
  v += lane_ror<2>(v);
  v += lane_ror<1>(v);
  return v;
}

template <typename T>
__device__ __forceinline__ T wave_max(T v) {
  auto step = [&](T o) { v = o > v ? o : v; };
  step(lane_xor_wide<32>(v));
  step(lane_xor_wide<16>(v));
  step(lane_xor_row<8>(v));
  step(lane_xor_row<4>(v));
  step(lane_xor_row<2>(v));
  step(lane_xor_row<1>(v));
  return v;
}

// Block totals: every thread combines the wavefront totals itself, in
// wavefront order, so all threads get the same bits without a broadcast
// round; the final barrier lets the caller reuse lds at once.
template <typename T>
__device__ inline T block_sum(T v, T* lds) {
  v = wave_sum(v);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  if (lane == 0) lds[w] = v;
  __syncthreads();
  T r = 0;
  for (int i = 0; i < (int)(blockDim.x / kWave); ++i) r += lds[i];
  __syncthreads();
  return r;
}

template <typename T>
__device__ inline T block_max(T v, T* lds) {
  v = wave_max(v);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
  if (lane == 0) lds[w] = v;
  __syncthreads();
  T r = lds[0];
  for (int i = 1; i < (int)(blockDim.x / kWave); ++i) r = lds[i] > r ? lds[i] : r;
  __syncthreads();
  return r;
}

// block_sum(s) and block_max(m) in one round (lds holds 2 * blockDim.x / 64
// values); the same bits as the two calls.
__device__ inline void block_sum_max(double& s, double& m, double* lds) {
  s = wave_sum(s);
  m = wave_max(m);
  const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave, nw = (int)(blockDim.x / kWave);
  if (lane == 0) {
    lds[w] = s;
    lds[nw + w] = m;
  }
  __syncthreads();
  double rs = 0, rm = lds[nw];
  for (int i = 0; i < nw; ++i) rs += lds[i];
  for (int i = 1; i < nw; ++i) rm = lds[nw + i] > rm ? lds[nw + i] : rm;
  __syncthreads();
  s = rs;
  m = rm;
}

// Sum of a group of G consecutive lanes (G a power of two <= 64); every lane
// of the group receives the total.
template <int G, typename T>
__device__ inline T group_sum(T v) {
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, G);
  return v;
}

template <int G, typename T>
__device__ inline T group_max(T v) {
#pragma unroll
  for (int off = G / 2; off > 0; off >>= 1) {
    T o = __shfl_xor(v, off, G);
    v = o > v ? o : v;
  }
  return v;
}

// Unroll depth of the CSR row loops: each lane keeps kUnroll independent
// (index, value) loads in flight before it gathers.
constexpr int kUnroll = 4;

// Chooses lanes-per-row G for a CSR row kernel from the mean row length, so
// that one unrolled trip (G * kUnroll elements) covers a typical row.
inline int lanes_for_rows(long long nnz, long long rows) {
  double avg = rows > 0 ? (double)nnz / (double)rows : 0.0;
  double per_lane_trip = avg / kUnroll;
  if (per_lane_trip <= 4) return 4;
  if (per_lane_trip <= 8) return 8;
  if (per_lane_trip <= 16) return 16;
  if (per_lane_trip <= 32) return 32;
  return 64;
}

// Streaming loads of CSR index/value arrays: each element is read once per
// SpMV, so they bypass cache retention (keeping the gathered vector in L2).
template <typename T>
__device__ __forceinline__ T ld_stream(const T* p) {
  return __builtin_nontemporal_load(p);
}

// Partial dot product of one CSR row [beg, end) for one lane of a G-lane
// group: kUnroll predicated loads of (column, value) are issued before the
// gathers so that every lane has kUnroll memory requests in flight.  Lanes
// past the row end load nothing and gather element 0 with weight 0.
template <int G, typename TV, typename TX, typename Gather>
__device__ __forceinline__ TX csr_row_dot(const int* __restrict__ ci, const TV* __restrict__ val, int beg, int end,
                                         int lane, Gather gather) {
  TX acc = 0;
  for (int k = beg + lane; k < end; k += kUnroll * G) {
    int c[kUnroll];
    TV v[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) {
      const int idx = k + u * G;
      const bool ok = idx < end;
      c[u] = ok ? ld_stream(ci + idx) : 0;
      v[u] = ok ? ld_stream(val + idx) : (TV)0;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; ++u) acc += (TX)v[u] * gather(c[u]);
  }
  return acc;
}

// Grid of a G-lanes-per-row kernel: one group per row up to `cap` blocks,
// then the kernel strides over rows.
inline int rows_grid(long long rows, int G, int cap) {
  const int rpb = kBlock / G;
  long long g = (rows + rpb - 1) / rpb;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (int)g;
}

constexpr int kRowGridCap = 2048;  // 8192 wavefronts: every SIMD of 256 CUs 8-deep

struct PanelMatrix;

}  // namespace osqp_hip

// ---- concrete types behind the opaque handles -----------------------------
struct OSQPVectorf_ {
  double* d;
  OSQPInt length;
  int is_view;
};

struct OSQPVectori_ {
  OSQPInt* d;
  OSQPInt length;
};

// A sparse matrix of the backend.  For a general matrix A (m x n):
//   rp/ci/val   : CSR of A (m rows)            — operator A x
//   trp/tci/tval: CSR of A' (n rows) = the input CSC arrays  — operator A' y
// For the cost matrix P given by its upper triangle (is_triu):
//   rp/ci/val   : CSR of the full symmetric P (n rows), rows sorted by column
//   trp/tci/tval: unused (P' = P)
// csc2csr[k] / csc2mirror[k] map entry k of the input CSC onto its slot(s) in
// the CSR copy (mirror = transposed slot of an off-diagonal triu entry, -1 on
// the diagonal); csc2t[k] = k for A (the transpose *is* the CSC).
// val32/tval32 are FP32 shadows used by the FP32 PCG; they are regenerated
// from the FP64 values whenever `fp32_dirty` is set.
struct OSQPMatrix_ {
  OSQPInt m, n;
  int is_triu;
  OSQPInt nnz_in;    // nnz of the input CSC (triu part for P)
  OSQPInt nnz;       // nnz of the CSR copy (full for P)
  int *rp, *ci;
  double* val;
  int *trp, *tci;
  double* tval;
  int *csc2csr, *csc2mirror;
  int* diag_pos;     // P only: slot of (i,i) in the full CSR, -1 if absent
  float *val32, *tval32;
  int fp32_dirty;
  int lanes, tlanes; // lanes per row for A and A' kernels
  long long version; // bumped on every value change
  // row-block partitions (nonzero-balanced) of the CSR copy and of A'
  int rb_n, trb_n;
  int *rb_rows, *trb_rows;
  // FP64 column panels of A and of A' (general matrices; matrix_panels64)
  struct osqp_hip::PanelMatrix* pan64[2];
  int pan_state[2];   // 0: not tried, 1: built, -1: not used
  double* pan_part;   // per-(panel, row) partials of the panel products
  size_t pan_part_len;
};
