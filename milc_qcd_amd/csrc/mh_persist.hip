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
// sums per workgroup go through memory.
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
constexpr unsigned kMaxPolls = 4u << 20;

struct Waiter {
  unsigned* gone;
  bool dead;
  // another poll (true) or give up (false)
  __device__ __forceinline__ bool again(unsigned& polls) {
    if (dead) return false;
    if (++polls >= kMaxPolls ||
        ((polls & 1023u) == 0 && __hip_atomic_load(gone, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
      __hip_atomic_store(gone, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      dead = true;
      return false;
    }
    return true;
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
    const int dist = h.three ? 3 : 1;
    return neighbour(g, c, cb, h.mu, h.back ? -dist : dist);
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
  Waiter w{ex.gone, false};
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
  bool ok = true;
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
    if (!(ok = collect_sums<4, BS>(s, rec, nb, sm, &lds_dead, w))) break;
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
  if (on && sub == 0) store_vec<P_F64>(x, cb, xv);
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
    sc->iters = ok ? it : -1;
    sc->halt = halt;
    sc->go = 0;
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
  const int cus = std::min(cu_count(), kPersistMaxBlocks);
  constexpr PersistShape shapes[] = {{16, 256, 0}, {8, 256, 0}, {4, 256, 0}, {1, 256, 0}, {1, 512, 0}};
  for (PersistShape s : shapes) {
    s.blocks = (int)(((long)Vh * s.lps + s.threads - 1) / s.threads);
    if (s.blocks <= cus) return s;
  }
  return PersistShape{0, 0, 0};
}

int cg_persist(VecField& x, VecField& r, VecField (&work)[4], int pb, double msq_x4, int max_it) {
  Context& c = ctx();
  const DevLinks& L = c.links[P_F64];
  const PersistShape sh = persist_shape(c.Vh);
  if (!L.valid || !sh.lps) return -3;
  const int nb = sh.blocks;
  Exchange ex;
  int rc;
  for (int k = 0; k < 4; k++) {
    (k < 2 ? ex.p[k] : ex.tmp[k - 2]) = work[k];
    if ((rc = empty_words(work[k].data, vec_bytes(P_F64, work[k].stride)))) return rc;
  }
  ex.rec = c.ws.partials;
  ex.gone = c.ws.flags;
  if ((rc = empty_words(ex.rec, (size_t)3 * 4 * nb * sizeof(double)))) return rc;
  MH_CHECK(hipMemsetAsync(ex.gone, 0, kPersistFlagBytes, c.stream));
  Geom g = c.geom;
  LinkField fat = L.fat, lng = L.lng;
  CGScalars* sc = c.ws.scal;
  void* args[] = {&g, &fat, &lng, &x, &r, &ex, &pb, &msq_x4, &max_it, &sc};
  const void* k = nullptr;
#define SHAPE(l, b) if (sh.lps == l && sh.threads == b) k = (const void*)k_cg_persist<l, b>
  SHAPE(16, 256); SHAPE(8, 256); SHAPE(4, 256); SHAPE(1, 256); SHAPE(1, 512);
#undef SHAPE
  if (!k) return -3;
  MH_CHECK(hipLaunchCooperativeKernel(k, dim3(nb), dim3(sh.threads), args, 0, c.stream));
  return 0;
}

}  // namespace mh
