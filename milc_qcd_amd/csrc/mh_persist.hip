// mh_persist.hip -- Krylov loops of small lattices in one kernel.
//
// On a lattice whose links stay in the caches an iteration of the four- to
// six-kernel loops of mh_core.hip and mh_multicg.hip is launch latency: 30 us
// per FP64 CG iteration at 8^4, 69 us at 16^3x32, where the two stencils move
// their bytes in a few microseconds.  Here one cooperative launch runs the
// whole loop.  Every group of LPS lanes owns one site of the solved parity and
// the site of the same index of the other parity, and keeps r, x, p of the
// site and as many of its links as fit in registers and LDS over all
// iterations; only the two stencil sources (p, D p) and one record of partial
// sums per workgroup go through memory.  Bound by the latency of the exchanges
// on the smallest lattices (8^4: 1.5 MB out of the L2s in 7.7 us) and by the
// links that do not fit the CU on the largest (16^3x32: 263 MB per iteration,
// 25 of a site's 32 matrices, from the Infinity Cache at 6.2 TB/s).
//
// Exchange without barriers: a shared value is one 8-byte word, written and
// read with relaxed agent-scope accesses (they meet in the memory-side cache,
// nothing is flushed or invalidated), and a word that has not been written yet
// holds kEmpty, a signalling NaN that no arithmetic produces.  A reader polls
// the words it needs.  p and D p alternate between two buffers, the records
// between three; the owner empties a word again once the collected sums show
// that every workgroup has read it, and waits for those stores before it
// publishes its next sums, so a word is empty before anybody can poll it for a
// later iteration:
//   p_i, (D p)_i   read by all before the sums of iteration i are complete,
//                  emptied after them, polled again in iteration i + 2;
//   record i       read by all before the sums of iteration i + 1 are
//                  complete, emptied after those, polled again for i + 3.
#include <algorithm>

#include "mh_internal.h"
#include "mh_persist.h"

namespace mh {

namespace {

constexpr unsigned long long kEmpty = 0x7ff4dead5afe0001ull;

__device__ __forceinline__ double ld_word(const double* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_word(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_empty(double* p) {
  __hip_atomic_store((unsigned long long*)p, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ bool empty(double v) { return (unsigned long long)__double_as_longlong(v) == kEmpty; }

// Polls of one word before the kernel gives up: seconds, against the
// microseconds an exchange takes.  `gone` is the give-up word of the launch.
// The workgroups are resident at once when the launch has the card to itself;
// beside the kernels of another process they need not be, and the host then
// finishes the solve with launches that wait for nobody.
constexpr unsigned kMaxPolls = 4u << 20;

struct Waiter {
  unsigned* gone;
  bool dead;
  // a word that is set from the start ends every wait at its first poll
  __device__ __forceinline__ explicit Waiter(unsigned* g) : gone(g) { dead = anybody_gone(); }
  // another poll (true) or give up (false)
  __device__ __forceinline__ bool again(unsigned& polls) {
    if (dead) return false;
    if (++polls >= kMaxPolls || ((polls & 1023u) == 0 && anybody_gone())) {
      __hip_atomic_store(gone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dead = true;
      return false;
    }
    return true;
  }
  __device__ __forceinline__ bool anybody_gone() const {
    return __hip_atomic_load(gone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
  }
};

// N vectors, all requested before the first is looked at: one round trip when
// they are there.
template <int N>
__device__ __forceinline__ void poll_vecs(const VecField& f, const int (&cb)[N], Vec3<double> (&v)[N], Waiter& w) {
  const double* p = (const double*)f.data;
  const unsigned plane = (unsigned)f.stride;
  unsigned polls = 0;
  bool missing;
  do {
    missing = false;
#pragma unroll
    for (int q = 0; q < N; q++)
#pragma unroll
      for (int k = 0; k < 3; k++) {
        v[q].c[k].re = ld_word(p + 2u * k * plane + (unsigned)cb[q]);
        v[q].c[k].im = ld_word(p + (2u * k + 1u) * plane + (unsigned)cb[q]);
      }
#pragma unroll
    for (int q = 0; q < N; q++)
#pragma unroll
      for (int k = 0; k < 3; k++) missing = missing || empty(v[q].c[k].re) || empty(v[q].c[k].im);
  } while (missing && w.again(polls));
}

// A site's vector to memory (or the words emptied): lane `sub` of its LPS
// lanes stores components sub, sub + LPS, ...
template <int LPS>
__device__ __forceinline__ void put_vec(const VecField& f, int cb, int sub, const Vec3<double>& v) {
  double* p = (double*)f.data + cb;
#pragma unroll
  for (int e = 0; e < 6; e++)
    if (LPS == 1 || (e % LPS) == sub) st_word(p + (size_t)e * f.stride, (e & 1) ? v.c[e >> 1].im : v.c[e >> 1].re);
}
template <int LPS>
__device__ __forceinline__ void empty_vec(const VecField& f, int cb, int sub) {
  double* p = (double*)f.data + cb;
#pragma unroll
  for (int e = 0; e < 6; e++)
    if (LPS == 1 || (e % LPS) == sub) st_empty(p + (size_t)e * f.stride);
}

__global__ void k_empty_words(double* p, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
    ((unsigned long long*)p)[i] = kEmpty;
}

// N sums per workgroup to its record, after every earlier store of the
// workgroup (the emptied words among them) has been performed.
template <int N, int BS>
__device__ __forceinline__ void publish_sums(double (&v)[N], double* rec, double (*sm)[BS / 64]) {
#pragma unroll
  for (int k = 0; k < N; k++)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < N; k++) sm[k][wid] = v[k];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x < N) {
    double s = 0;
#pragma unroll
    for (int w = 0; w < BS / 64; w++) s += sm[threadIdx.x][w];
    st_word(rec + 4 * blockIdx.x + threadIdx.x, s);
  }
}
// The sums of all records, in the same association on every workgroup and in
// every run.  False when a workgroup gave up waiting.
template <int N, int BS>
__device__ __forceinline__ bool collect_sums(double (&v)[N], const double* rec, int nb, double (*sm)[BS / 64],
                                             int* lds_dead, Waiter& w) {
#pragma unroll
  for (int k = 0; k < N; k++) v[k] = 0;
  for (int i = threadIdx.x; i < nb; i += BS) {
    double t[N];
    unsigned polls = 0;
    bool missing;
    do {
      missing = false;
#pragma unroll
      for (int k = 0; k < N; k++) t[k] = ld_word(rec + 4 * i + k);
#pragma unroll
      for (int k = 0; k < N; k++) missing = missing || empty(t[k]);
    } while (missing && w.again(polls));
#pragma unroll
    for (int k = 0; k < N; k++) v[k] += t[k];
  }
#pragma unroll
  for (int k = 0; k < N; k++)
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_xor(v[k], off, 64);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // sm and lds_dead of the step before are read
  if (threadIdx.x == 0) *lds_dead = 0;
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < N; k++) sm[k][wid] = v[k];
  __syncthreads();
  if (w.dead) *lds_dead = 1;
#pragma unroll
  for (int k = 0; k < N; k++) {
    double s = 0;
#pragma unroll
    for (int q = 0; q < BS / 64; q++) s += sm[k][q];
    v[k] = s;
  }
  __syncthreads();
  return *lds_dead == 0;
}

// The stencil of one site pair over LPS lanes.  Lane `sub` takes the hops
// h = sub, sub + LPS ... of both parities, hop h = 4 mu + 2 (three-hop) +
// (back).
// `hops` of them are taken at a time: their links and vectors are all
// requested before the first is waited for.  Matrices that stay on the CU over
// the iterations: every one of the lane (2, 4 or 8) in registers with at least
// four lanes per site; with one lane, of the last pass, `lds` of the first
// parity in LDS and the next `regs` in registers, the others being read again
// in every application (a thread has 512 registers with 256 threads per CU,
// 256 with 512; a matrix takes 36, or 144 B of LDS).
template <int LPS, int BS> struct Resident;
template <> struct Resident<16, 256> { static constexpr int lds = 0, regs = 2, hops = 1; };
template <> struct Resident<8, 256> { static constexpr int lds = 0, regs = 4, hops = 2; };
template <> struct Resident<4, 256> { static constexpr int lds = 0, regs = 8, hops = 4; };
template <> struct Resident<1, 256> { static constexpr int lds = 4, regs = 3, hops = 4; };
template <> struct Resident<1, 512> { static constexpr int lds = 2, regs = 0, hops = 2; };

template <int LPS, int BS>
struct SiteStencil {
  static constexpr int HPL = 16 / LPS, LDSM = Resident<LPS, BS>::lds, REGS = Resident<LPS, BS>::regs;
  // hops of the last loop pass of apply: one direction, or the lane's one or two hops
  static constexpr int HPP = Resident<LPS, BS>::hops, PASSES = HPL / HPP;
  Mat3<double> m[REGS ? REGS : 1];

  // the lane's j-th hop (written so that what all lanes share is scalar)
  struct Hop {
    int mu;
    bool three, back;
  };
  __device__ __forceinline__ static Hop hop(int j, int sub) {
    Hop h;
    h.mu = LPS <= 4 ? (j * LPS) >> 2 : (j * LPS + sub) >> 2;
    h.three = LPS == 1 ? (j >> 1) & 1 : (sub >> 1) & 1;
    h.back = LPS == 1 ? j & 1 : sub & 1;
    return h;
  }
  __device__ __forceinline__ static int at(const Geom& g, const Coord& c, int cb, const Hop& h) {
    // scalar copies of the extents: an indexed g.X would move to memory
    const int X0 = __builtin_amdgcn_readfirstlane(g.X[0]), X1 = __builtin_amdgcn_readfirstlane(g.X[1]);
    const int X2 = __builtin_amdgcn_readfirstlane(g.X[2]), X3 = __builtin_amdgcn_readfirstlane(g.X[3]);
    const int x = h.mu == 0 ? c.x : (h.mu == 1 ? c.y : (h.mu == 2 ? c.z : c.t));
    const int L = h.mu == 0 ? X0 : (h.mu == 1 ? X1 : (h.mu == 2 ? X2 : X3));
    const int stride = h.mu == 1 ? g.sy : (h.mu == 2 ? g.sz : g.st);
    const int dist = h.three ? 3 : 1;
    int y = x + (h.back ? -dist : dist);
    y += y < 0 ? L : 0;
    y -= y >= L ? L : 0;
    return h.mu == 0 ? c.rowbase + (y >> 1) : cb + (y - x) * stride;
  }
  // the hop's matrix as it multiplies the neighbour: F, or -F^dag of the back link
  __device__ __forceinline__ static void link(const LinkField& fat, const LinkField& lng, int cb, int pb, const Hop& h,
                                              int n, Mat3<double>& out) {
    const bool back = h.back;
    const nat_d2* p = (const nat_d2*)(h.three ? lng.data : fat.data);
    const unsigned s = (unsigned)(((back ? pb ^ 1 : pb) * 4 + h.mu) * 9) * (unsigned)fat.stride +
                       (unsigned)(back ? n : cb);
    const unsigned di = (back ? 1u : 3u) * (unsigned)fat.stride, dj = (back ? 3u : 1u) * (unsigned)fat.stride;
    const double sr = back ? -1.0 : 1.0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        const nat_d2 a = p[s + i * di + j * dj];
        out.e[i][j].re = sr * a.x;
        out.e[i][j].im = a.y;
      }
  }

  // slot of hop k of the last pass: parity first (other = 0, 1), then the hop
  __device__ __forceinline__ void init(const Geom& g, const LinkField& fat, const LinkField& lng, int cb, int pb,
                                       int sub, nat_d2 (*lds)[9][BS]) {
#pragma unroll
    for (int q = 0; q < LDSM + REGS; q++) {
      const int p2 = q < HPP ? pb : pb ^ 1;
      const Hop h = hop(HPL - HPP + q % HPP, sub);
      const Coord c = site_coords(g, cb, p2);
      const int n = at(g, c, cb, h);
      if (q >= LDSM) {
        link(fat, lng, cb, p2, h, n, m[q >= LDSM ? q - LDSM : 0]);
      } else {
        Mat3<double> t;
        link(fat, lng, cb, p2, h, n, t);
#pragma unroll
        for (int e = 0; e < 9; e++) {
          nat_d2 a;
          a.x = t.e[e / 3][e % 3].re;
          a.y = t.e[e / 3][e % 3].im;
          lds[q][e][threadIdx.x] = a;
        }
      }
    }
  }

  // acc = D src at (cb, pb); OTHER = 1 on the second parity of init
  template <int OTHER>
  __device__ __forceinline__ void apply(const Geom& g, const LinkField& fat, const LinkField& lng,
                                        const VecField& src, int cb, int pb, int sub, const nat_d2 (*lds)[9][BS],
                                        Waiter& w, Vec3<double>& acc) const {
    zero(acc);
    // the addresses of the links that are read again are formed again, too:
    // kept over the iterations they would take the registers of the others
    if (PASSES > 1) asm volatile("" : "+v"(cb));
    const Coord c = site_coords(g, cb, pb);
#pragma unroll 1
    for (int d = 0; d < PASSES; d++) {
      const bool last = d == PASSES - 1;
      int n[HPP];
      Mat3<double> t[HPP];
      Vec3<double> v[HPP];
#pragma unroll
      for (int k = 0; k < HPP; k++) {
        const Hop h = hop(HPP * d + k, sub);
        n[k] = at(g, c, cb, h);
        if (!(last && OTHER * HPP + k < LDSM + REGS)) link(fat, lng, cb, pb, h, n[k], t[k]);
      }
      poll_vecs<HPP>(src, n, v, w);
#pragma unroll
      for (int k = 0; k < HPP; k++) {
        const int q = OTHER * HPP + k;
        const bool in_lds = q < LDSM, in_regs = !in_lds && q < LDSM + REGS;
        if (last && in_regs) {
          mv_acc(m[in_regs ? q - LDSM : 0], v[k], acc);
        } else {
          if (last && in_lds) {
#pragma unroll
            for (int e = 0; e < 9; e++) {
              const nat_d2 a = lds[in_lds ? q : 0][e][threadIdx.x];
              t[k].e[e / 3][e % 3].re = a.x;
              t[k].e[e / 3][e % 3].im = a.y;
            }
          }
          mv_acc(t[k], v[k], acc);
        }
      }
    }
#pragma unroll
    for (int off = 1; off < LPS; off <<= 1)
#pragma unroll
      for (int k = 0; k < 3; k++) {
        acc.c[k].re += __shfl_xor(acc.c[k].re, off, 64);
        acc.c[k].im += __shfl_xor(acc.c[k].im, off, 64);
      }
  }
};

// The exchanged words of a launch: p and D p in two buffers each (six planes of
// words, so that a wavefront's load is dense), the records of sums in three.
struct Exchange {
  VecField p[2], tmp[2];
  double* rec;       // 3 * nb records of 4 doubles
  unsigned* gone;
};

// FP64 CG from a restart (p = r, |r|^2 in the scalars) to the recurrence
// target or max_it iterations: ks_congrad_parity_cpu's normal iterations
// (d_congrad5_fn_milc.c:270-367, FEWSUMS) as enqueue_cg_iteration runs them.
template <int LPS, int BS>
__global__ void __launch_bounds__(BS, 1)
k_cg_persist(Geom g, LinkField fat, LinkField lng, VecField x, VecField r, Exchange ex, int pb, double msq_x4, int max_it,
             CGScalars* sc) {
  __shared__ double sm[4][BS / 64];
  __shared__ int lds_dead;
  constexpr int LDSM = Resident<LPS, BS>::lds;
  __shared__ nat_d2 lds[LDSM ? LDSM : 1][9][LDSM ? BS : 1];
  auto ldsp = (nat_d2(*)[9][BS])lds;
  const int nb = gridDim.x;
  const int t = xcd_block(blockIdx.x, nb) * BS + threadIdx.x;
  const int cb = t / LPS, sub = t % LPS;
  const bool on = cb < g.Vh;
  Vec3<double> xv, rv, pv, tv;
  SiteStencil<LPS, BS> st;
  Waiter w(ex.gone);
  zero(xv);
  zero(rv);
  if (on) {
    load_vec<P_F64>(x, cb, xv);
    load_vec<P_F64>(r, cb, rv);
    st.init(g, fat, lng, cb, pb ^ 1, sub, ldsp);
  }
  pv = rv;
  double rsq = sc->rsq, oldrsq = sc->actual_rsq, rr_here = 0.0, a = 0.0, b = 0.0, rsq_max = sc->rsq_max;
  double pkp = 0.0, c_tr = 0.0, c_tt = 0.0;
  const double stop = sc->rsq_stop;
  int it = 0, halt = 0;
  while (it < max_it && !halt) {
    const int e = it & 1;
    double s[4] = {0, 0, 0, rr_here};
    if (on) {
      put_vec<LPS>(ex.p[e], cb, sub, pv);
      st.template apply<0>(g, fat, lng, ex.p[e], cb, pb ^ 1, sub, ldsp, w, tv);
      put_vec<LPS>(ex.tmp[e], cb, sub, tv);
      st.template apply<1>(g, fat, lng, ex.tmp[e], cb, pb, sub, ldsp, w, tv);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        tv.c[k].re -= msq_x4 * pv.c[k].re;
        tv.c[k].im -= msq_x4 * pv.c[k].im;
        s[0] += pv.c[k].re * tv.c[k].re + pv.c[k].im * tv.c[k].im;
        s[1] += tv.c[k].re * rv.c[k].re + tv.c[k].im * rv.c[k].im;
        s[2] += tv.c[k].re * tv.c[k].re + tv.c[k].im * tv.c[k].im;
      }
      if (LPS > 1 && sub != 0) s[0] = s[1] = s[2] = 0.0;
    }
    double* rec = ex.rec + (size_t)(it % 3) * 4 * nb;
    publish_sums<4, BS>(s, rec, sm);
    if (!collect_sums<4, BS>(s, rec, nb, sm, &lds_dead, w)) break;
    if (on) {
      empty_vec<LPS>(ex.p[e], cb, sub);
      empty_vec<LPS>(ex.tmp[e], cb, sub);
    }
    if (it > 0 && threadIdx.x < 4) st_empty(ex.rec + (size_t)((it - 1) % 3) * 4 * nb + 4 * blockIdx.x + threadIdx.x);
    // the scalar step, by every thread from the same sums
    pkp = s[0];
    c_tr = s[1];
    c_tt = s[2];
    if (it > 0) oldrsq = s[3];
    a = -rsq / pkp;
    rsq = oldrsq + 2.0 * a * c_tr + a * a * c_tt;
    b = rsq / oldrsq;
    if (rsq > rsq_max) rsq_max = rsq;
    if (rsq < stop) halt = 1;
    it++;
    rr_here = 0.0;
    if (on) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        xv.c[k].re += a * pv.c[k].re;
        xv.c[k].im += a * pv.c[k].im;
        rv.c[k].re += a * tv.c[k].re;
        rv.c[k].im += a * tv.c[k].im;
        rr_here += rv.c[k].re * rv.c[k].re + rv.c[k].im * rv.c[k].im;
        pv.c[k].re = rv.c[k].re + b * pv.c[k].re;
        pv.c[k].im = rv.c[k].im + b * pv.c[k].im;
      }
      if (LPS > 1 && sub != 0) rr_here = 0.0;
    }
  }
  // A thread that gives up publishes the sums of what it did not get (NaN) only
  // after its give-up word: whoever collected those sums finds the word set, and
  // leaves x as it was.
  if (on && sub == 0 && !w.anybody_gone()) store_vec<P_F64>(x, cb, xv);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->rsq = rsq;
    sc->oldrsq = oldrsq;
    sc->actual_rsq = oldrsq;
    sc->pkp = pkp;
    sc->c_tr = c_tr;
    sc->c_tt = c_tt;
    sc->a = a;
    sc->b = b;
    sc->rsq_max = rsq_max;
    sc->iters = it;
    sc->halt = halt;
    sc->go = 0;
  }
}

// Multi-shift CG (ks_multicg_offset_field_cpu, ks_multicg_offset.c:291-460) in
// one kernel: the recurrences and deferred updates of mh_multicg.hip, the
// scalars of all shifts in LDS, computed alike by every workgroup (thread j has
// shift j).  tab: psim_j (MS_MAX), pm_j (MS_MAX), then the MS_KW residuals of
// the window, all touched by the lanes of their own site only; lane `sub` of a
// site brings shifts sub, sub + LPS ... up to date.  pm_j and psim_j start as
// the source and zero without being read.  A shift with a target of its own is
// left as it is once its residual zeta_j |r| is below it (zeta_j set to zero,
// as when it underflows).
template <int LPS, int BS>
__global__ void __launch_bounds__(BS, 1)
k_ms_persist(Geom g, LinkField fat, LinkField lng, VecField src, const VecField* __restrict__ tab, Exchange ex, int pb,
             MSPersist* io) {
  constexpr int LDSM = Resident<LPS, BS>::lds;
  __shared__ double sm[1][BS / 64];
  __shared__ int lds_dead;
  __shared__ nat_d2 lds[LDSM ? LDSM : 1][9][LDSM ? BS : 1];
  __shared__ double zi[MS_MAX], zm1[MS_MAX], zp1[MS_MAX], bi[MS_MAX], shf[MS_MAX], wa[MS_MAX], wx[MS_MAX];
  __shared__ double wc[MS_MAX][MS_KW], wb[MS_MAX][MS_KW];
  __shared__ int done[MS_MAX];  // nothing left to bring up to date in this window
  auto ldsp = (nat_d2(*)[9][BS])lds;
  const int nb = gridDim.x, tid = threadIdx.x;
  const int t = xcd_block(blockIdx.x, nb) * BS + tid;
  const int cb = t / LPS, sub = t % LPS;
  const bool on = cb < g.Vh;
  const int n = io->n, jl = io->j_low, max_iter = io->max_iter;
  const double rsqstop = io->rsqstop, shift0 = -io->shifts[jl];
  if (tid < n) {
    zi[tid] = zm1[tid] = 1.0;
    shf[tid] = tid == jl ? io->shifts[tid] : io->shifts[tid] - io->shifts[jl];
  }
  const double stop_shift = tid < n && tid != jl ? io->stop[tid] : 0.0;
  Vec3<double> rv, pv, tv;
  SiteStencil<LPS, BS> st;
  Waiter w(ex.gone);
  zero(rv);
  if (on) {
    load_vec<P_F64>(src, cb, rv);
    st.init(g, fat, lng, cb, pb ^ 1, sub, ldsp);
    empty_vec<LPS>(ex.p[1], cb, sub);
    empty_vec<LPS>(ex.tmp[1], cb, sub);
  }
  pv = rv;
  double rsq = io->source_norm, alpha_low = 0.0, beta_low_1 = -1.0;
  int it = 0, now = n, now_ws = n, m = 0, halt = 0, converged = 0;
  // `ok` only for iters: without it the loop is compiled to spill elsewhere, and
  // the kernel of four lanes per site is 6% slower (2.0 against 2.1 ms, two
  // shifts at Vh = 13824)
  bool first = true, ok = true;
  __syncthreads();
  while (!halt) {
    const int e = it & 1;
    if (m == 0) {
      now_ws = now;
      if (tid < n) {
        wa[tid] = 1.0;
        wx[tid] = 0.0;
        for (int l = 0; l < MS_KW; l++) wc[tid][l] = wb[tid][l] = 0.0;
        done[tid] = zi[tid] == 0.0;
      }
    }
    double s[1] = {0.0};
    if (on) {
      put_vec<LPS>(ex.p[e], cb, sub, pv);
      st.template apply<0>(g, fat, lng, ex.p[e], cb, pb ^ 1, sub, ldsp, w, tv);
      put_vec<LPS>(ex.tmp[e], cb, sub, tv);
      st.template apply<1>(g, fat, lng, ex.tmp[e], cb, pb, sub, ldsp, w, tv);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        tv.c[k].re += shift0 * pv.c[k].re;
        tv.c[k].im += shift0 * pv.c[k].im;
        s[0] += pv.c[k].re * tv.c[k].re + pv.c[k].im * tv.c[k].im;
      }
      if (LPS > 1 && sub != 0) s[0] = 0.0;
    }
    // records: <p, ttt> in buffers 0 and 1, |r|^2 in 2 and 3
    double* const rec_a = ex.rec + (size_t)e * 4 * nb;
    double* const rec_b = ex.rec + (size_t)(2 + e) * 4 * nb;
    publish_sums<1, BS>(s, rec_a, sm);
    if (!(ok = collect_sums<1, BS>(s, rec_a, nb, sm, &lds_dead, w))) break;
    if (on) {
      empty_vec<LPS>(ex.p[e], cb, sub);
      empty_vec<LPS>(ex.tmp[e], cb, sub);
    }
    if (it > 0 && tid == 0) st_empty(ex.rec + (size_t)(2 + (e ^ 1)) * 4 * nb + 4 * blockIdx.x);
    // beta and zeta (ks_multicg_offset.c:322-356)
    const double beta_low = -rsq / s[0];
    it++;
    m++;
    const int last = now - 1;
    const bool retire = last > jl && zi[last] == 0.0;
    if (tid < now) {
      if (tid == jl) {
        bi[tid] = beta_low;
        zp1[tid] = 1.0;
      } else {
        double z = zi[tid] * zm1[tid] * beta_low_1;
        const double c1 = beta_low * alpha_low * (zm1[tid] - zi[tid]);
        const double c2 = zm1[tid] * beta_low_1 * (1.0 + shf[tid] * beta_low);
        z = c1 + c2 != 0.0 ? z / (c1 + c2) : 0.0;
        if (zi[tid] != 0.0) {
          bi[tid] = beta_low * z / zi[tid];
        } else {
          z = 0.0;
          bi[tid] = 0.0;
        }
        zp1[tid] = z;
      }
    }
    if (retire) now--;
    if (tid < now) {
      const double b = bi[tid];
      wx[tid] += b * wa[tid];
      for (int l = 0; l < m - 1; l++) wb[tid][l] += b * wc[tid][l];
    }
    s[0] = 0.0;
    if (on) {
#pragma unroll
      for (int k = 0; k < 3; k++) {
        rv.c[k].re += beta_low * tv.c[k].re;
        rv.c[k].im += beta_low * tv.c[k].im;
        s[0] += rv.c[k].re * rv.c[k].re + rv.c[k].im * rv.c[k].im;
      }
      if (sub == 0) store_vec<P_F64>(tab[2 * MS_MAX + m - 1], cb, rv);
      if (LPS > 1 && sub != 0) s[0] = 0.0;
    }
    publish_sums<1, BS>(s, rec_b, sm);
    if (!(ok = collect_sums<1, BS>(s, rec_b, nb, sm, &lds_dead, w))) break;
    if (tid == 0) st_empty(rec_a + 4 * blockIdx.x);
    const double oldrsq = rsq;
    rsq = s[0];
    if (rsqstop > 0 && rsq <= rsqstop) {
      halt = converged = 1;
    } else {
      // alpha, the coefficients of the window, scroll (:358-463)
      alpha_low = rsq / oldrsq;
      if (tid < now) {
        double a = alpha_low;
        if (tid != jl)
          a = zi[tid] * beta_low != 0.0 ? alpha_low * zp1[tid] * bi[tid] / (zi[tid] * beta_low) : 0.0;
        wa[tid] *= a;
        for (int l = 0; l < m - 1; l++) wc[tid][l] *= a;
        wc[tid][m - 1] = zp1[tid];
        zm1[tid] = zi[tid];
        zi[tid] = zp1[tid] * zp1[tid] * rsq < stop_shift ? 0.0 : zp1[tid];
      }
      beta_low_1 = beta_low;
#pragma unroll
      for (int k = 0; k < 3; k++) {
        pv.c[k].re = rv.c[k].re + alpha_low * pv.c[k].re;
        pv.c[k].im = rv.c[k].im + alpha_low * pv.c[k].im;
      }
      if (1 + it >= max_iter) halt = 1;
    }
    if (m < MS_KW && !halt) continue;
    // psim_j and pm_j from the window's residuals
    __syncthreads();
    if (on) {
      Vec3<double> ring[MS_KW];
#pragma unroll
      for (int l = 0; l < MS_KW; l++) {
        if (l < m) load_vec<P_F64>(tab[2 * MS_MAX + l], cb, ring[l]);
        else zero(ring[l]);
      }
      for (int j = sub; j < now_ws; j += LPS) {
        Vec3<double> d, x;
        if (done[j]) continue;
        if (first) {
          load_vec<P_F64>(src, cb, d);
          zero(x);
        } else {
          load_vec<P_F64>(tab[MS_MAX + j], cb, d);
          load_vec<P_F64>(tab[j], cb, x);
        }
        const double cx = wx[j], ca = wa[j];
#pragma unroll
        for (int k = 0; k < 3; k++) {
          double xr = x.c[k].re + cx * d.c[k].re, xi = x.c[k].im + cx * d.c[k].im;
          double qr = ca * d.c[k].re, qi = ca * d.c[k].im;
#pragma unroll
          for (int l = 0; l < MS_KW; l++) {
            const double b = wb[j][l], cc = wc[j][l];
            xr += b * ring[l].c[k].re;
            xi += b * ring[l].c[k].im;
            qr += cc * ring[l].c[k].re;
            qi += cc * ring[l].c[k].im;
          }
          x.c[k].re = xr;
          x.c[k].im = xi;
          d.c[k].re = qr;
          d.c[k].im = qi;
        }
        store_vec<P_F64>(tab[j], cb, x);
        if (!halt) store_vec<P_F64>(tab[MS_MAX + j], cb, d);
      }
    }
    first = false;
    m = 0;
    __syncthreads();
  }
  if (blockIdx.x == 0 && tid == 0) {
    io->rsq = rsq;
    io->iters = ok ? it : -1;
    io->converged = converged;
  }
}

int cu_count() {
  static int n[64] = {0};
  const int dev = ctx().device;
  if (dev < 0 || dev >= 64) return 0;
  if (!n[dev]) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) v = 0;
    n[dev] = v;
  }
  return n[dev];
}

int empty_words(void* p, size_t bytes) {
  const size_t n = bytes / 8;
  hipLaunchKernelGGL(k_empty_words, dim3((unsigned)std::min<size_t>((n + 255) / 256, 1024)), dim3(256), 0, ctx().stream,
                     (double*)p, n);
  MH_CHECK(hipGetLastError());
  return 0;
}

}  // namespace

// As many lanes per site as one workgroup of 256 threads per CU leaves room
// for, except two: with two the matrices do not fit the registers any more and
// the lanes' two passes cost more than one lane's four (26.8 us per CG
// iteration against 24.6 at Vh = 20736, 30.1 against 27.8 at 32768).  512
// threads per CU only where 256 lanes are too few (20.9 us with one lane and
// 256 threads, 42 with 512, at Vh = 13824; 8 lanes and 512 threads 23.6).
// us per iteration here and with the launches of enqueue_cg_iteration: Vh = 128
// 6.3 / 22; 2048 8.1 / 30; 6000 8.1 / 38; 13824 12.8 / 52; 32768 27.8 / 60;
// 65536 42 / 69; 73728 55 / 89; 131072 95 / 113.
PersistShape persist_shape(int Vh) {
  if (!ctx().small_form) return PersistShape{0, 0, 0};
  const int cus = std::min(cu_count(), kPersistMaxBlocks);
  constexpr PersistShape shapes[] = {{16, 256, 0}, {8, 256, 0}, {4, 256, 0}, {1, 256, 0}, {1, 512, 0}};
  for (PersistShape s : shapes) {
    s.blocks = (int)(((long)Vh * s.lps + s.threads - 1) / s.threads);
    if (s.blocks <= cus) return s;
  }
  return PersistShape{0, 0, 0};
}

// The exchange of a launch, all words empty; gone: its give-up word.
static int start_exchange(const VecField (&work)[4], int nb, int records, unsigned* gone, Exchange& ex) {
  Context& c = ctx();
  int rc;
  for (int k = 0; k < 4; k++) {
    (k < 2 ? ex.p[k] : ex.tmp[k - 2]) = work[k];
    if ((rc = empty_words(work[k].data, vec_bytes(P_F64, work[k].stride)))) return rc;
  }
  ex.rec = c.ws.partials;
  ex.gone = gone;
  return empty_words(ex.rec, (size_t)records * 4 * nb * sizeof(double));
}

// 0: enqueued; 1: the device cannot hold the grid at once, or knows no such
// launches.
static int launch_persist(const void* kernel, const PersistShape& sh, void** args) {
  const hipError_t e =
      hipLaunchCooperativeKernel(kernel, dim3(sh.blocks), dim3(sh.threads), args, 0, ctx().stream);
  if (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorNotSupported) {
    (void)hipGetLastError();  // answered here
    return 1;
  }
  MH_CHECK(e);
  return 0;
}

// Kernel K<lanes, threads> of a shape.
#define PERSIST_KERNEL(K, sh)                                                            \
  ((sh).lps == 16  ? (const void*)K<16, 256>                                             \
   : (sh).lps == 8 ? (const void*)K<8, 256>                                              \
   : (sh).lps == 4 ? (const void*)K<4, 256>                                              \
                   : ((sh).threads == 256 ? (const void*)K<1, 256> : (const void*)K<1, 512>))

int cg_persist(VecField& x, VecField& r, VecField (&work)[4], int pb, double msq_x4, int max_it) {
  Context& c = ctx();
  const DevLinks& L = c.links[P_F64];
  const PersistShape sh = persist_shape(c.Vh);
  if (!L.valid || !sh.lps) return -3;
  Exchange ex;
  CGScalars* sc = c.ws.scal;
  int rc = start_exchange(work, sh.blocks, 3, &sc->gone, ex);
  if (rc) return rc;
  Geom g = c.geom;
  LinkField fat = L.fat, lng = L.lng;
  void* args[] = {&g, &fat, &lng, &x, &r, &ex, &pb, &msq_x4, &max_it, &sc};
  return launch_persist(PERSIST_KERNEL(k_cg_persist, sh), sh, args);
}

int ms_persist(const VecField& src, const VecField* tab, VecField (&work)[4], int pb, MSPersist* io) {
  Context& c = ctx();
  const DevLinks& L = c.links[P_F64];
  const PersistShape sh = persist_shape(c.Vh);
  if (!L.valid || !sh.lps) return -3;
  Exchange ex;
  int rc = start_exchange(work, sh.blocks, 4, &io->gone, ex);
  if (rc) return rc;
  Geom g = c.geom;
  LinkField fat = L.fat, lng = L.lng;
  VecField s = src;
  void* args[] = {&g, &fat, &lng, &s, &tab, &ex, &pb, &io};
  return launch_persist(PERSIST_KERNEL(k_ms_persist, sh), sh, args);
}

}  // namespace mh
