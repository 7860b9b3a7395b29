// nd_factor.h -- multifrontal Cholesky factor under a nested-dissection
// order (nd_factor.hip).
#pragma once

#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#include "nd_layout.h"

namespace shellgpu {

struct NdFactor {
  int nbatch = 0;          // designs factored
  long per_design = 0;     // doubles of M per design
  long q_len = 0, s_len[2] = {0, 0}, v_len = 0;
  int chunk = 1;           // designs factored together (workspace copies)
  long n = 0;              // dofs
  int rhs_cap = 0;         // vectors per design that V and W hold: 1 or 16
  std::vector<NdLevel> levels;  // deepest first
  NdDev *d_fronts = nullptr;
  int *d_lists = nullptr;
  double *M = nullptr, *Q = nullptr, *S[2] = {nullptr, nullptr}, *V = nullptr;
  double *W = nullptr;  // interleaved right-hand sides and solutions of several vectors
};

// leaves of the dissection: 24 nodes (144 dofs).  Fewer, larger leaves give
// fewer fronts but more fill (200 x 400 cylinder: 1.45 GB at 24 nodes, 1.33
// at 16 with a third more fronts, 1.79 at 48)
constexpr int kNdLeafNodes = 24;

// Buffers of a factor of nbatch designs with the fronts of L, for solves of
// nrhs vectors per design.  Returns an empty string or the error.
std::string nd_create(int nn, const NdLayout &L, int nbatch, int nrhs, NdFactor &F);
void nd_destroy(NdFactor &F);
// factor the designs' matrices (nnzb blocks of 36 values each, placed by
// blk_base, blk_ld and blk_flag: bits 6 + c for BC columns, bit 12 for a
// diagonal block); info[design] becomes 1 at a pivot that is not positive,
// else 0
hipError_t nd_compute(NdFactor &F, int nnzb, const double *vals, const long *blk_base, const int *blk_ld,
                      const int *blk_flag, int *info, hipStream_t stream);
// x = A^-1 b for nrhs vectors per design (vector r of design d at (r nbatch +
// d) n); act (nact designs): only these, one vector each
hipError_t nd_solve(const NdFactor &F, const double *b, double *x, long n, int nrhs, const int *act, int nact,
                    hipStream_t stream);
// hold the front vectors of nrhs vectors per design
hipError_t nd_reserve(NdFactor &F, int nrhs);

}  // namespace shellgpu
