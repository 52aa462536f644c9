// mh_persist.h -- whole Krylov loops in one cooperative kernel (small lattices).
#pragma once
#include "mh_common.h"

namespace mh {

constexpr int kPersistMaxBlocks = 256;

// Lanes per site, threads per workgroup and workgroups (one per CU, so that
// the grid is resident at once) for Vh sites of a parity; lps = 0: the lattice
// does not fit, or one-kernel solves are switched off.
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
// CGScalars); x and the scalars are updated, the work fields are scratch.
// Returns 1 when the device refuses the launch.  With `gone` set in the
// scalars a workgroup gave up waiting, and x holds a mixture of the guess and
// iterates: either way the solve has to go on launch by launch from the true
// residual.
int cg_persist(VecField& x, VecField& r, VecField (&work)[4], int pb, double msq_x4, int max_it);

// Multi-shift CG: most shifts of a solve, iterations of a window of deferred
// updates.
#define MS_MAX 32
#define MS_KW 8
// Sites per parity up to which the mixed multi-shift of `sources` sources runs
// in FP64 in one kernel, one source after another (ms of one source, 12 shifts
// to 1e-9, here / FP32 stage and refinement: Vh = 2048 1.3 / 7.6; 20736
// 5.4 / 16.8; 65536 10.5 / 24; 131072 22.6 / 36; three shifts at 131072
// 20.3 / 20.8).  Against the batched solve of up to four sources (all solves
// of one HISQ trajectory step pair, two sources): 20736 28 / 50, 65536
// 49 / 84, 131072 113 / 133, so that four sources break even near 16384.
constexpr int persist_mixed_shift_sites(int sources) {
  return sources <= 2 ? 131072 : (sources == 3 ? 65536 : (sources == 4 ? 16384 : (sources <= 6 ? 4096 : 0)));
}
// Sites per parity up to which the sources of a block call are solved one after
// another in one kernel each instead of as a batch (ms of one source here, of
// batches of 2 / 4 / 8 sources, CG to 1e-9 at m = 0.03: Vh = 2048 0.67, 4.5 /
// 4.2 / 4.4; 6000 0.93, 5.9 / 5.5 / 6.1; 13824 1.6, 7.7 / 6.9 / 8.6; 32768 3.5,
// 9.7 / 9.5 / 12.9; 65536 8.3, 18.1 / 20.4 / 27.5; two-shift multi-shifts alike).
constexpr int persist_block_sites(int sources) {
  return sources <= 2 ? 65536 : (sources <= 4 ? 16384 : (sources <= 6 ? 8192 : 0));
}

// What one FP64 multi-shift solve in one kernel takes and gives back (device memory).
struct MSPersist {
  double shifts[MS_MAX];  // the offsets, as given
  double stop[MS_MAX];    // |r_j|^2 below which shift j (not the smallest) is done; 0: never
  double source_norm, rsqstop, rsq;
  int n, j_low, max_iter, iters, converged;
  alignas(256) unsigned gone;  // as in CGScalars
};
// tab (device memory): psim_j in [0, n), pm_j in [MS_MAX, MS_MAX + n), the
// residuals of a window in [2 MS_MAX, 2 MS_MAX + MS_KW).  Returns 1 when the
// device refuses the launch; with `gone` set in io the solutions are void.
int ms_persist(const VecField& src, const VecField* tab, VecField (&work)[4], int pb, MSPersist* io);

}  // namespace mh
