// runner.h — many ADMM iterations of one QP in one launch.
//
// A solve of a small or medium QP by separate kernels costs what its launches
// cost: about 12 + 6 k kernels an ADMM iteration (k CG iterations), each over
// in 2-4 us, and a host that has to see the CG stop before it queues more.
// The runner keeps the whole loop on the device between two points where the
// host takes part (termination check, rho update): one launch of G
// workgroups of 1024 threads runs up to check_termination ADMM iterations.
//
//   * A's rows are dealt to the G workgroups in contiguous, nonzero-balanced
//     ranges.  A workgroup keeps everything per row (z, y, rho, A x, the CG's
//     w and A p) to itself; it forms w = rho o (A p) of its rows and, from a
//     column-ordered copy of the same rows, its share of A' w at once, with
//     no exchange in between.
//   * The shares are added in column chunks (n / G columns a workgroup), and
//     the n-vectors of the CG are held by every workgroup (in registers, p
//     also in LDS): their updates and dot products are done by all of them
//     alike, in one fixed order, so a CG iteration needs two grid barriers
//     (shares written; K p written) and no reduction across workgroups.
//   * Data that crosses workgroups goes through relaxed agent-scope atomic
//     loads and stores (they are coherent across the XCDs' L2s by themselves),
//     so a barrier is a counter and not a write-back and invalidate of the
//     L2s, and the matrix stays cached.  Measured on 256 workgroups: 2.6 us a
//     barrier, 17.9 us with fences.
//   * With G = 1 the barriers are workgroup barriers.
//   * A barrier's wait is bounded; what a launch changes is copied before it
//     (3 us), so that a launch that gave up can be done again elsewhere.
//
// P's rows of a chunk belong to the chunk's workgroup.  The copies are sliced: 64 lanes hold 64 / T rows, T lanes a row, rows
// of a workgroup sorted by length (longest first) so that a slice's width is
// its first row's; entry i T + t of a row is step i of its lane t.  A row is
// summed lane by lane in step order and by a butterfly over its T lanes:
// results depend on the problem alone.
#pragma once

#include <stdint.h>

#include "hip_internal.h"

namespace osqp_hip {

// ADMM iterations between two exact recomputations of A x64 (one workgroup in
// FP64: every one).  Against 80-bit arithmetic the vector carried in between has
// 1.08 to 1.45 times a fresh product's relative error of 1.3e-16 to 3.5e-16
// (n = 300..5000); a product in every iteration took 5000 x 50000 in FP64 from
// 172 to 189 ms, with outputs that differ by 1e-15.
constexpr int kRunRefresh = 8;

struct RunOp {
  int lgT;            // log2 of the lanes per row
  int ns;             // slices per workgroup
  int slots;          // row slots of a workgroup (one workgroup only)
  int* soff;          // G * (ns + 1): first step of each slice, within the workgroup's steps
  uint16_t* perm;     // G * ns * (64 >> lgT): local row of each slot, 0xFFFF for none
  long long* base;    // G + 1: first step of each workgroup (a step is 64 entries)
  long long steps;    // base[G]
  int max_steps;      // of one workgroup
  uint16_t* col;      // steps * 64
  void* val;          // steps * 64, in the CG precision
};

struct Runner {
  int on;             // built and usable
  int n, m, G, bits;
  int state_len;      // doubles of the PCG's device state
  int cw;             // columns per chunk
  int rows_max;       // rows of the largest workgroup range
  int resident;       // the copies held in LDS
  int chain;          // entries that one lane adds up, at most (several workgroups)
  size_t lds;         // dynamic LDS of a launch
  int* r0;            // G + 1 row ranges
  int* cs;            // (G + 1) * n: first entry of column j at or below row r0[b] (CSC positions)
  // several workgroups: rows of A, columns of those rows, P's rows of the chunk;
  // one: rows of A and of [P A'] for the CG, and with an FP32 CG both again for
  // the FP64-vector products (P: [P A'], A2: A), on the lanes of those panels
  RunOp A, At, P, A2;
  double* part;       // G * n shares
  double* xch;        // 2 n: r64, K p
  unsigned* bar;      // barrier words
  double* save;       // what a launch changes, as it was before it (runner_restore)
  long long ver_A, ver_P;  // versions the values were copied from
};

// CSR of [P A'] (FP64 values)
struct RunK {
  const int *rp, *ci;
  const double* val;
};

// The device state of the PCG that a run continues and leaves (pcg.hip).
struct RunState {
  double *eps_prev, *red_factor;
  int *zero_iters, *iter, *solves, *active, *done;
  long long* total_iters;
};

struct RunCall {
  int iters, z_count, max_iter, reduction_threshold, guard;
  double alpha, sigma, spr, sdr;
  double *x, *dx, *z, *y, *dy;                      // in place
  const double *q, *l, *u, *rho, *rhoinv;
  double *x64, *ax64;
  const void* dinv;                                 // CG precision
  RunState st;
  double* state;                                    // the PCG's device state (Runner::state_len)
  int polls;          // looks after which a barrier's wait gives up (-1: the default)
  int* bad;           // host-coherent word, set where that happened
};

// Builds the runner for A (m x n, CSR and CSC on the device) when it pays, fits
// and its memory can be had; r->on stays 0 and r empty otherwise.  Returns
// r->on.  one: only the one-workgroup kernel will do.  state_len: doubles of
// the PCG's device state.
int runner_build(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, int bits, bool one, int state_len);
void runner_free(Runner* r);
// Queues c.iters ADMM iterations and leaves the new z_count; 1 when the launch
// was refused (nothing has changed then).
int runner_run(Runner* r, const OSQPMatrix* A, const OSQPMatrix* P, const RunK& k, const RunCall& c, int* z_count);
// Several workgroups: x, z, y, x64, A x64 and the PCG's state as they were
// before the last launch.
void runner_restore(Runner* r, const RunCall& c);

}  // namespace osqp_hip
