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
// kernel, for either sloppy precision where the 16-bit one breaks even (m = 0.02
// to 1e-9, ms FP64 / FP32 sloppy / 16-bit sloppy: Vh = 2048 0.71 / 2.2 / 2.2;
// 20736 3.8 / 5.5 / 5.8; 49152 5.5 / 6.4 / 5.7; 57344 6.5 / 6.9 / 6.5; 65536
// 8.3 / 8.7 / 7.6; 98304 12.7 / 11.1 / 9.5).
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
// Sites per parity up to which the solves of `sources` sources with `shifts`
// shifts each (0: a CG) run in FP64 in one kernel, one source after another,
// instead of as a batch (the multi-shift of one source: instead of the FP32
// stage and grouped refinement).  ms here / there at the line and beyond it, to
// a true residual of 1e-6 and to one of 1e-9 (m = 0.03; beyond the line, the
// sources times the time of one).  The looser target needs less refinement and
// decides, except for two to four shifts of four sources, where the line is even
// between the two; tight ones alone would gain further out.
//   1 source, 1 shift    65536  5.1 / 6.0,   7.7 / 9.4    131072 11.7 / 9.5,  18.3 / 15.3
//             2          98304  9.1 / 9.7,  13.6 / 15.9   131072 12.5 / 10.9, 19.5 / 20.0
//             9, 12     131072 13.8 / 14.3, 21.6 / 34.2
//   2         CG         49152  8.5 / 8.6,  11.8 / 11.5    65536 11.5 / 10.1, 16.7 / 14.6
//             2          65536 11.4 / 11.8, 17.2 / 19.9    98304 18.3 / 14.3, 27.1 / 23.2
//             9          98304 20.0 / 19.1, 29.4 / 56.7   131072 27.7 / 21.8, 42.4 / 58.9
//   3         CG         16384  4.1 / 5.3,   5.6 / 7.5     24696  7.4 / 6.3,  10.4 / 8.7
//             2          16384  4.6 / 5.7,   6.7 / 9.4     24696  7.5 / 6.0,  11.0 / 10.1
//             9          65536 18.8 / 18.5, 27.8 / 49.7    98304 30.4 / 24.3, 44.1 / 68.9
//   4         CG, 1      16384  5.4 / 5.4,   7.4 / 7.6     24696  9.8 / 6.5,  13.9 / 8.9
//             2          16384  6.3 / 5.7,   8.9 / 9.3     24696 10.0 / 5.9,  14.6 / 10.0
//             5, 9       16384  6.9 / 7.6,   9.6 / 15.4    24696 11.8 / 9.9,  17.4 / 25.4
//   5         CG          8192  5.3 / 5.5,   7.1 / 7.9     13824  6.4 / 6.2,   8.5 / 8.1
//             2           8192  6.2 / 7.3,   8.6 / 11.8    13824  7.6 / 7.3,  10.6 / 11.3
//   6         CG          2048  3.4 / 3.0,   4.5 / 4.2
//             2           8192  7.4 / 7.3,  10.4 / 11.8    13824  9.1 / 7.3,  12.7 / 11.3
constexpr int persist_sites(int sources, int shifts) {
  switch (sources) {
    case 1: return shifts <= 1 ? 65536 : (shifts <= 4 ? 98304 : 131072);
    case 2: return shifts == 0 ? 49152 : (shifts < 9 ? 65536 : 98304);
    case 3: return shifts < 9 ? 16384 : 65536;
    case 4: return 16384;
    case 5: return 8192;
    case 6: return shifts == 0 ? 0 : 8192;
  }
  return 0;
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
