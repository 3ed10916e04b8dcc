// bj_sweep.hpp -- the host form of a block-Jacobi block's triangular sweeps
// and the line-wavefront apply built from it (shared by precon.hip, which
// factorises the blocks, and bjlines.hip).
#pragma once

#include <vector>

#include "internal.hpp"

namespace parcel {

struct BlockSweep {
  // rows of the block in level order, with per-level boundaries
  std::vector<int> lev_start;   // offsets into order (size nlev+1)
  std::vector<int> order;       // local rows (0-based within the block)
  std::vector<int> ptr;         // entry ranges per local row (size nrow+1)
  std::vector<int> dep;         // local dependency rows
  std::vector<double> val;
  std::vector<double> diag;     // per local row
  // double-double factors: lo parts of val and diag (empty otherwise)
  std::vector<double> val_lo;
  std::vector<double> diag_lo;
};

// Barrier that orders LDS accesses only.  __syncthreads() also waits for
// every outstanding global load and store of the wave (CDNA counts both in
// vmcnt), which would drain the prefetch pipeline at every level.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Line-wavefront form of the block-Jacobi apply (bjlines.hip).  Sets P.M.line
// up from the block factors when they have its pattern (parts: 1 FP64, 2
// double-double) and returns whether it did.
bool line_setup(Plan& P, const std::vector<BlockSweep>& F, const std::vector<BlockSweep>& B,
                const std::vector<int>& blo, const std::vector<int>& bhi, int parts);
void line_apply(Plan& P, const double* r, double* s, const CGFuse* fuse, const int* skip);
void line_apply_dd(Plan& P, const double* rh, const double* rl, double* sh, double* sl, const int* skip);

}  // namespace parcel
