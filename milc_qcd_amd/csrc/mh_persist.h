// mh_persist.h -- whole Krylov loops in one cooperative kernel (small lattices).
#pragma once
#include "mh_common.h"

namespace mh {

constexpr int kPersistMaxBlocks = 256;
constexpr size_t kPersistFlagBytes = 256;

// Lanes per site, threads per workgroup and workgroups (one per CU, so that
// the grid is resident at once) for Vh sites of a parity; lps = 0: the lattice
// does not fit.
struct PersistShape {
  int lps, threads, blocks;
};
PersistShape persist_shape(int Vh);

// Sites per parity up to which a mixed-precision CG runs as the FP64 CG in one
// kernel (m = 0.02 to 1e-9, ms FP64 / FP32 sloppy / 16-bit sloppy: Vh = 2048
// 0.71 / 2.2 / 2.2; 20736 3.8 / 5.5 / 5.8; 49152 5.1 / 6.0 / 6.0; 65536
// 8.2 / 9.0 / 8.1; 98304 12.7 / 11.0 / 9.5).
constexpr int kPersistMixedSites = 49152;

// FP64 CG iterations from a restart (r the residual, |r|^2 in the context's
// CGScalars); x and the scalars are updated (iters = -1: a workgroup gave up
// waiting), the work fields are scratch.
int cg_persist(VecField& x, VecField& r, VecField (&work)[4], int pb, double msq_x4, int max_it);

}  // namespace mh
