// lceq_kernels.hip -- gfx950 kernels of the lattice update and measurement
// path.  One thread owns one site of the parity being updated; a (parity, mu)
// link class or a Higgs parity is one launch, so the checkerboard replaces the
// reference's MPI halo exchanges and barriers.  All arithmetic is FP64.
#include <math.h>

#include <algorithm>

#include "lceq_internal.hpp"
#include "lceq_sites.hpp"

namespace lceq {

static constexpr int TB = 256;

int blocks_for(int n) { return (n + TB - 1) / TB; }

// ================================================================ links

// What a wave needs before it can issue its operand loads, as leading
// arguments: the compiler's kernel-argument preload (build.py) has them in
// scalar registers when the wave starts, 14 dwords, all there is room for.
// Loaded from the argument segment they put one memory round trip ahead of
// the gathers of every launch: 64^3 production sweep 172 -> 163.5 us,
// reference sweep 91.4 -> 86.1 us, one gauge-fixing iteration 20.4 -> 19.2 us;
// from 96^3 on 1%.  Pairs of 32-bit values share an argument.  (The same in
// four vector-typed arguments cost 1.5% on lattices beyond the Infinity Cache.)
#define HEAD_PARAMS                                                                           \
  double *hU, double *hA, uint64_t hn, uint64_t hb, uint64_t hh, uint64_t hw, uint64_t hr
#define HEAD_OF head_of(hU, hA, hn, hb, hh, hw, hr)
enum { HEAD_EO = 1, HEAD_XCD = 2, HEAD_STRIPS = 4, HEAD_WRAP = 8 };

struct Head {
  double *U, *A;
  Geom g;  // without the extents
  int nb, flags;
};
__device__ __forceinline__ Head head_of(double* U, double* A, uint64_t hn, uint64_t hb,
                                        uint64_t hh, uint64_t hw, uint64_t hr) {
  Geom g{0, 0, 0, half0(hh), half1(hh), half0(hn), half1(hn),
         __builtin_bit_cast(float, half0(hr)), __builtin_bit_cast(float, half1(hr)),
         half0(hw), half1(hw)};
  return Head{U, A, g, half0(hb), half1(hb)};
}

struct HeadArgs {
  double *U, *A;
  uint64_t n, b, h, w, r;
};
// r: the launch covers a range of the sites only; its head then carries the
// range's length and start in place of n and the number of blocks
static HeadArgs head_args(const lceq_lattice* L, double* U, double* A, int nb, int eo,
                          const SiteRange* r = nullptr) {
  const Geom& g = L->g;
  int flags = (eo ? HEAD_EO : 0) | (L->xcd ? HEAD_XCD : 0) | (strip_rows(L) ? HEAD_STRIPS : 0);
  if (r && (int64_t)r->p0 + r->len > g.n) flags |= HEAD_WRAP;
  return HeadArgs{U, A, halves(r ? r->len : g.n, g.npad), halves(r ? r->p0 : nb, flags),
                  halves(g.h1, g.h2),
                  halves(g.wy, g.wz), halves(__builtin_bit_cast(int, g.rh1),
                                             __builtin_bit_cast(int, g.rh2))};
}

// The rest of a link launch's arguments
struct LinkArgs {
  SiteOrder order;
  double beta, beta_a;
  const double* fed;
  Philox key;
  uint64_t pass;
  int measflag, renorm, reduce;
  int pstride;
  int n, nb;     // sites of the parity and blocks of the slot (RANGE)
  double* part;  // partial sums of this launch's slot: [LCEQ_NQ][pstride]
};

// Schedule of the update launches (link_update_site, higgs_update_site):
// the early issue and the fenced uniform phase measured faster from 48^3 to
// 128^3 (4-6% per sweep), where a launch has 512 waves or more (32768 sites
// per class) and the lattice's link and Higgs fields fit the 256 MB Infinity
// Cache; smaller and larger lattices keep the previous schedule
static bool early_schedule(const lceq_lattice* L) {
  return L->g.n >= 32768 && 30.0 * 8.0 * (double)L->g.npad <= 256.0 * 1024.0 * 1024.0;
}

// The strip rows of the launches: the caller's, or by the lattice's shape.  In
// index order a site's z neighbours are a plane away; from 8192 sites a plane
// and parity on (4 MB of fields, one XCD's L2) they have left the L2 when the
// next plane reads them, and strips keep them.  Production sweeps in ns per
// site, index order against strips: 128x128x100 0.672 0.645, 144x144x96 0.711
// 0.642, 160x160x80 0.784 0.636, 192x192x48 0.882 0.648, 256x256x32 0.897
// 0.636; 112^3 0.654 0.660 and 64^3 0.640 0.663 the other way.  Strips of 1024
// to 2047 sites a plane: 512 cost up to 15% (128x128x64 0.790 against 0.697).
// Where no power of two of rows gives that, strips of two rows, which pay from
// 12800 sites a plane on (200x200x40 0.890 0.677).
int strip_rows(const lceq_lattice* L) {
  const Geom& g = L->g;
  if (L->strip >= 0) return L->strip;
  if (g.h2 < 8192 || (int64_t)g.ly * g.lz >= (int64_t)1 << 22) return 0;
  int sy = 2;
  while ((int64_t)sy * g.h1 < 1024) sy *= 2;
  if (sy * g.h1 < 2048 && g.ly % sy == 0) return sy;
  return g.h2 >= 12800 ? 2 : 0;
}

// Block index in the launch's block order: XCD-aware (contiguous sites per
// XCD) or the launch order
__device__ __forceinline__ int shape_block(int nb, int xcd) {
  int b = xcd_block(nb);  // computed either way: no branch before the loads
  return xcd ? b : (int)blockIdx.x;
}

// Site and slot block of a launch over a range of the sites, which may run on
// past the last site to the first: s counts from the range's start
__device__ __forceinline__ unsigned range_site(const Head& h, unsigned s, int n) {
  s += (unsigned)h.nb;
  return h.flags & HEAD_WRAP && s >= (unsigned)n ? s - (unsigned)n : s;
}
template <int TBX>
__device__ __forceinline__ int range_block(const Head& h, int blk, int nb) {
  blk += h.nb / TBX;
  return blk >= nb ? blk - nb : blk;
}

// One site per thread, TBX sites per block
template <bool KP, bool FED, int TBX, int MU, bool EARLY, bool RANGE>
__global__ __launch_bounds__(TBX) void k_link(HEAD_PARAMS, LinkArgs a) {
  const Head h = HEAD_OF;
  int blk = shape_block(RANGE ? (h.g.n + TBX - 1) / TBX : h.nb, h.flags & HEAD_XCD);
  unsigned P = (unsigned)(blk * TBX + threadIdx.x);
  double red[3] = {0.0, 0.0, 0.0};
  if (P < (unsigned)h.g.n) {
    LinkSite p;
    p.g = h.g;
    p.U = h.U;
    p.A = h.A;
    p.eo = h.flags & HEAD_EO;
    p.mu = MU;
    p.beta = a.beta;
    p.beta_a = a.beta_a;
    p.fed = a.fed;
    p.key = a.key;
    p.pass = a.pass;
    p.measflag = a.measflag;
    p.renorm = a.renorm;
    unsigned s = h.flags & HEAD_STRIPS ? strip_site(p.g, a.order, P) : P;
    if (RANGE) s = range_site(h, s, a.n);
    link_update_site<KP, FED, EARLY>(p, s, red);
  }
  if (a.reduce)
    block_sum_store<3, TBX / 64>(red, a.part, a.pstride,
                                 RANGE ? range_block<TBX>(h, blk, a.nb) : blk);
}

int shape_blocks(const lceq_lattice* L) { return (L->g.n + L->tb - 1) / L->tb; }

template <bool KP, bool FED, int MU, bool EARLY, bool RANGE, int TBX>
static void link_launch(lceq_lattice* L, int eo, const LinkArgs& a, const SiteRange* r) {
  int nb = RANGE ? (r->len + TBX - 1) / TBX : shape_blocks(L);
  HeadArgs h = head_args(L, L->U, L->A, nb, eo, r);
  hipLaunchKernelGGL((k_link<KP, FED, TBX, MU, EARLY, RANGE>), dim3(nb), dim3(TBX), 0, L->stream,
                     h.U, h.A, h.n, h.b, h.h, h.w, h.r, a);
}

template <bool KP, bool FED, int MU, bool EARLY, bool RANGE>
static void link_dispatch_tb(lceq_lattice* L, int eo, const LinkArgs& a, const SiteRange* r) {
  switch (L->tb) {
    case 64: link_launch<KP, FED, MU, EARLY, RANGE, 64>(L, eo, a, r); break;
    case 128: link_launch<KP, FED, MU, EARLY, RANGE, 128>(L, eo, a, r); break;
    case 512: link_launch<KP, FED, MU, EARLY, RANGE, 512>(L, eo, a, r); break;
    default: link_launch<KP, FED, MU, EARLY, RANGE, 256>(L, eo, a, r); break;
  }
}

template <bool KP, bool FED, int MU>
static void link_dispatch_mu(lceq_lattice* L, int eo, const LinkArgs& a, const SiteRange* r) {
  if constexpr (!FED) {
    if (r) return link_dispatch_tb<KP, FED, MU, true, true>(L, eo, a, r);
  }
  if (early_schedule(L))
    link_dispatch_tb<KP, FED, MU, true, false>(L, eo, a, nullptr);
  else
    link_dispatch_tb<KP, FED, MU, false, false>(L, eo, a, nullptr);
}

// The direction is a template argument: the neighbour steps and link offsets
// of the staple are then fixed at compile time.
template <bool KP, bool FED>
static void link_dispatch(lceq_lattice* L, int eo, int mu, const LinkArgs& a,
                          const SiteRange* r) {
  switch (mu) {
    case 0: link_dispatch_mu<KP, FED, 0>(L, eo, a, r); break;
    case 1: link_dispatch_mu<KP, FED, 1>(L, eo, a, r); break;
    default: link_dispatch_mu<KP, FED, 2>(L, eo, a, r); break;
  }
}

void launch_link(lceq_lattice* L, int kp, int eo, int mu, int measflag, int renorm_on_write,
                 const double* fed, uint64_t pass, int reduce, const SiteRange* range) {
  LinkArgs a;
  a.n = L->g.n;
  a.nb = shape_blocks(L);
  a.order = site_order(range ? range->len / L->g.h2 : L->g.lz, strip_rows(L));
  a.beta = L->beta;
  a.beta_a = L->beta_a;
  a.fed = fed;
  a.key = Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)};
  a.pass = pass;
  a.measflag = measflag;
  a.renorm = renorm_on_write;
  a.reduce = reduce;
  a.pstride = L->pstride;
  a.part = L->partials + (size_t)(eo * 3 + mu) * LCEQ_NQ * L->pstride;
  int kc = kp ? KC_LINK_KP : KC_LINK_OR;
  prof_begin(L, kc);
  prof_count(L, kc);
  if (kp) {
    if (fed)
      link_dispatch<true, true>(L, eo, mu, a, range);
    else
      link_dispatch<true, false>(L, eo, mu, a, range);
  } else {
    if (fed)
      link_dispatch<false, true>(L, eo, mu, a, range);
    else
      link_dispatch<false, false>(L, eo, mu, a, range);
  }
  prof_end(L, kc);
}

// ============================================================ finalize

struct FinalizeArgs {
  const double* part;  // [LCEQ_NSLOT][LCEQ_NQ][pstride]
  int pstride, nb_link, nb_higgs;  // block partials per link / Higgs slot
  int link_kind, link_meas, higgs_kind, higgs_meas;
  double vol;
  double* obs;
  double* hist_row;
  double* host;  // pinned copy of the observables, or null
};

// One 1024-thread block sums every partial the closing routines wrote: six
// link slots x 3 quantities and two Higgs slots x 4 quantities.  Wave w owns
// quantities w and w+16; each lane sums its strided share of the block
// partials (the loads of both quantities in flight at once), a xor-butterfly
// finishes the wave sum (fixed order, so the result is reproducible), and
// thread 0 combines the slots in the reference's loop order: f/agauge.f:195-200
// (links), f/ahiggs1.f:107-123 and f/ahiggs2.f:138-143 (Higgs).  The
// observables are read by wave 0 alongside the partials, updated in LDS and
// written back (and to the history row) by 16 lanes at once.
constexpr int FIN_TB = 1024;
__global__ __launch_bounds__(1024) void k_finalize(FinalizeArgs p) {
  constexpr int NV = 6 * 3 + 2 * 4;
  __shared__ double tot[32];
  __shared__ double ob[LCEQ_OBS_N];
  int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double ov = threadIdx.x < LCEQ_OBS_N ? p.obs[threadIdx.x] : 0.0;
  const double* x[2];
  int nbq[2];
  bool on[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    int q = w + 16 * h;  // 0..17 link (slot*3 + quantity), 18..25 Higgs
    on[h] = q < NV && (q < 18 ? p.link_kind != 0 : p.higgs_kind != 0);
    size_t row = q < 18 ? (size_t)(q / 3) * LCEQ_NQ + q % 3
                        : (size_t)(6 + (q - 18) / 4) * LCEQ_NQ + (q - 18) % 4;
    x[h] = p.part + row * p.pstride;
    nbq[h] = on[h] ? (q < 18 ? p.nb_link : p.nb_higgs) : 0;
  }
  double t[2] = {0.0, 0.0};
  for (int i0 = lane; i0 < max(nbq[0], nbq[1]); i0 += 64 * 8) {
    double y[2][8];  // sixteen loads in flight before the adds
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 8; ++u) y[h][u] = i0 + 64 * u < nbq[h] ? x[h][i0 + 64 * u] : 0.0;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 8; ++u) t[h] += y[h][u];
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    t[h] = wave_sum(t[h]);
    if (lane == 0 && w + 16 * h < NV) tot[w + 16 * h] = t[h];
  }
  if (threadIdx.x < LCEQ_OBS_N) ob[threadIdx.x] = ov;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double* v = tot;
    double* obs = ob;
    if (p.link_kind) {
      double plaq = 0.0, nacch = 0.0, acc1 = 0.0;
      for (int slot = 0; slot < 6; ++slot) {
        plaq = plaq + v[slot * 3];
        nacch += v[slot * 3 + 1];
        acc1 += v[slot * 3 + 2];
      }
      obs[OBS_NACCH] = nacch;
      obs[OBS_NACC1] = acc1;
      if (p.link_meas == 1) obs[OBS_PLAQ0] = plaq / (12.0 * p.vol);
      double accept;
      if (p.link_kind == 1) {  // (nacch/3V)(acc1/12V) with measflag, else nacch
        accept = nacch;
        if (p.link_meas == 1) accept = (accept / (3.0 * p.vol)) * (acc1 / (12.0 * p.vol));
      } else {
        accept = acc1 / (3.0 * p.vol);
      }
      obs[OBS_ACC_LINK] = accept;
    }
    if (p.higgs_kind) {
      double acc = v[18] + v[22];
      double r2 = v[19] + v[23], r4 = v[20] + v[24], kin = v[21] + v[25];
      if (p.higgs_meas == 1) {
        obs[OBS_A02] = r2 / p.vol;
        obs[OBS_A04] = r4 / p.vol;
        obs[OBS_A0KIN] = kin / (6.0 * p.vol);
      }
      double accept = acc / p.vol;
      if (p.higgs_kind == 1) {
        obs[OBS_ACC_HIGGS] = accept;
        double d = obs[OBS_DELTA];
        if (fabs(accept - 0.5) > 0.1) d = (accept > 0.5) ? 1.1131241 * d : 0.8989669 * d;
        obs[OBS_DELTA] = d;
      } else if (p.higgs_meas == 1) {
        obs[OBS_ACC_HIGGS] = accept;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x < LCEQ_OBS_N) {
    double o = ob[threadIdx.x];
    p.obs[threadIdx.x] = o;
    if (p.hist_row) p.hist_row[threadIdx.x] = o;
    if (p.host) p.host[threadIdx.x] = o;
  }
}

__global__ __launch_bounds__(64) void k_set_obs(double* __restrict__ obs, int index, double value) {
  if (threadIdx.x == 0) obs[index] = value;
}

void launch_set_obs(lceq_lattice* L, int index, double value) {
  hipLaunchKernelGGL(k_set_obs, dim3(1), dim3(64), 0, L->stream, L->obs, index, value);
}

// Small results reach the host by stores to pinned memory: a copy command to
// pageable memory and its wait took 40 us (the seven averages of a lattice),
// this kernel and its wait 14
__global__ __launch_bounds__(TB) void k_export(const double* __restrict__ dev,
                                               double* __restrict__ host, unsigned n) {
  unsigned i = blockIdx.x * TB + threadIdx.x;
  if (i < n) host[i] = dev[i];
}

void launch_export(lceq_lattice* L, const double* dev, size_t n) {
  hipLaunchKernelGGL(k_export, dim3(blocks_for((int)n)), dim3(TB), 0, L->stream, dev,
                     L->pin + LCEQ_OBS_N, (unsigned)n);
}

void launch_finalize(lceq_lattice* L, int link_kind, int link_meas, int higgs_kind,
                     int higgs_meas, double* hist_row, bool to_host, int higgs_nb) {
  FinalizeArgs a;
  a.host = to_host ? L->pin : nullptr;
  a.part = L->partials;
  a.pstride = L->pstride;
  a.nb_link = shape_blocks(L);
  a.nb_higgs = higgs_nb > 0 ? higgs_nb : shape_blocks(L);
  a.link_kind = link_kind;
  a.link_meas = link_meas;
  a.higgs_kind = higgs_kind;
  a.higgs_meas = higgs_meas;
  a.vol = (double)L->vol;
  a.obs = L->obs;
  a.hist_row = hist_row;
  hipLaunchKernelGGL(k_finalize, dim3(1), dim3(FIN_TB), 0, L->stream, a);
}

// staple only, for the staples() entry point (f/staples.f:9)
__global__ __launch_bounds__(256) void k_staples(Geom g, const double* __restrict__ U,
                                                 double* __restrict__ Vst, int eo, int mu) {
  int s = blockIdx.x * TB + threadIdx.x;
  if (s >= g.n) return;
  Coord c = site_coord(g, eo, s);
  st_link(Vst, g, mu, eo, s, staple(U, g, eo, mu, s, c));
}

void launch_staples(lceq_lattice* L, int eo, int mu) {
  hipLaunchKernelGGL(k_staples, dim3(blocks_for(L->g.n)), dim3(TB), 0, L->stream, L->g, L->U,
                     L->Vst, eo, mu);
}

// ================================================================ Higgs

__global__ __launch_bounds__(256) void k_force(Geom g, const double* __restrict__ U,
                                               const double* __restrict__ A,
                                               double* __restrict__ F, int eo) {
  int s = blockIdx.x * TB + threadIdx.x;
  if (s >= g.n) return;
  st_higgs(F, g, 0, s, hop_force(U, A, g, eo, s, site_coord(g, eo, s)));
}

void launch_force(lceq_lattice* L, int eo) {
  hipLaunchKernelGGL(k_force, dim3(blocks_for(L->g.n)), dim3(TB), 0, L->stream, L->g, L->U, L->A,
                     L->F, eo);
}

struct HiggsArgs {
  SiteOrder order;
  int imode, measflag, reduce;
  double beta_a, beta_2, beta_4;
  const double* delta;
  const double* fed;
  Philox key;
  uint64_t pass;
  double* part;
  int pstride;
  int n, nb;  // as LinkArgs
};

// MODE: the whole lattice, a range of it, or the whole lattice with renorm first
enum { HIGGS_ALL, HIGGS_RANGE, HIGGS_RENORM };
template <int KIND, bool FED, int TBX, bool EARLY, int MODE>
__global__ __launch_bounds__(TBX) void k_higgs(HEAD_PARAMS, HiggsArgs a) {
  constexpr bool RANGE = MODE == HIGGS_RANGE;
  const Head h = HEAD_OF;
  int blk = shape_block(RANGE ? (h.g.n + TBX - 1) / TBX : h.nb, h.flags & HEAD_XCD);
  unsigned P = (unsigned)(blk * TBX + threadIdx.x);
  double red[4] = {0.0, 0.0, 0.0, 0.0};
  if (P < (unsigned)h.g.n) {
    HiggsSite p;
    p.g = h.g;
    p.U = h.U;
    p.A = h.A;
    p.eo = h.flags & HEAD_EO;
    p.imode = a.imode;
    p.beta_a = a.beta_a;
    p.beta_2 = a.beta_2;
    p.beta_4 = a.beta_4;
    p.delta = a.delta;
    p.fed = a.fed;
    p.key = a.key;
    p.pass = a.pass;
    p.measflag = a.measflag;
    unsigned s = h.flags & HEAD_STRIPS ? strip_site(p.g, a.order, P) : P;
    if (RANGE) s = range_site(h, s, a.n);
    higgs_update_site<KIND, FED, EARLY, MODE == HIGGS_RENORM>(p, s, red);
  }
  if (a.reduce)
    block_sum_store<4, TBX / 64>(red, a.part, a.pstride,
                                 RANGE ? range_block<TBX>(h, blk, a.nb) : blk);
}

template <int KIND, bool FED, bool EARLY, int MODE, int TBX>
static void higgs_launch(lceq_lattice* L, int eo, const HiggsArgs& a, const SiteRange* r) {
  int nb = MODE == HIGGS_RANGE ? (r->len + TBX - 1) / TBX : shape_blocks(L);
  HeadArgs h = head_args(L, L->U, L->A, nb, eo, r);
  hipLaunchKernelGGL((k_higgs<KIND, FED, TBX, EARLY, MODE>), dim3(nb), dim3(TBX), 0, L->stream,
                     h.U, h.A, h.n, h.b, h.h, h.w, h.r, a);
}

template <int KIND, bool FED, bool EARLY, int MODE>
static void higgs_dispatch_tb(lceq_lattice* L, int eo, const HiggsArgs& a, const SiteRange* r) {
  switch (L->tb) {
    case 64: higgs_launch<KIND, FED, EARLY, MODE, 64>(L, eo, a, r); break;
    case 128: higgs_launch<KIND, FED, EARLY, MODE, 128>(L, eo, a, r); break;
    case 512: higgs_launch<KIND, FED, EARLY, MODE, 512>(L, eo, a, r); break;
    default: higgs_launch<KIND, FED, EARLY, MODE, 256>(L, eo, a, r); break;
  }
}

// the early issue exists for ahiggs1 only (EARLY = KIND == 1 there), and so do
// launches over a range; renorm first exists for ahiggs2
template <int KIND, bool FED>
static void higgs_dispatch(lceq_lattice* L, int eo, const HiggsArgs& a, const SiteRange* r,
                           bool renorm) {
  if constexpr (KIND == 1 && !FED) {
    if (r) return higgs_dispatch_tb<KIND, FED, true, HIGGS_RANGE>(L, eo, a, r);
  }
  if constexpr (KIND == 2 && !FED) {
    if (renorm) return higgs_dispatch_tb<KIND, FED, false, HIGGS_RENORM>(L, eo, a, nullptr);
  }
  if (early_schedule(L))
    higgs_dispatch_tb<KIND, FED, KIND == 1, HIGGS_ALL>(L, eo, a, nullptr);
  else
    higgs_dispatch_tb<KIND, FED, false, HIGGS_ALL>(L, eo, a, nullptr);
}

void launch_higgs(lceq_lattice* L, int kind, int eo, int measflag, const double* fed,
                  uint64_t pass, int reduce, bool renorm, const SiteRange* range) {
  HiggsArgs a;
  a.reduce = reduce;
  a.n = L->g.n;
  a.nb = shape_blocks(L);
  a.order = site_order(range ? range->len / L->g.h2 : L->g.lz, strip_rows(L));
  a.imode = L->imode;
  a.measflag = measflag;
  a.beta_a = L->beta_a;
  a.beta_2 = L->beta_2;
  a.beta_4 = L->beta_4;
  a.delta = L->obs + OBS_DELTA;
  a.fed = fed;
  a.key = Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)};
  a.pass = pass;
  a.part = L->partials + (size_t)(6 + eo) * LCEQ_NQ * L->pstride;
  a.pstride = L->pstride;
  prof_begin(L, KC_HIGGS);
  prof_count(L, KC_HIGGS);
  if (kind == 1) {
    if (fed) higgs_dispatch<1, true>(L, eo, a, range, renorm); else higgs_dispatch<1, false>(L, eo, a, range, renorm);
  } else if (kind == 2) {
    if (fed) higgs_dispatch<2, true>(L, eo, a, range, renorm); else higgs_dispatch<2, false>(L, eo, a, range, renorm);
  } else {
    if (fed) higgs_dispatch<3, true>(L, eo, a, range, renorm); else higgs_dispatch<3, false>(L, eo, a, range, renorm);
  }
  prof_end(L, KC_HIGGS);
}

// =============================================================== renorm

// f/renorm.f:24-34 / f/u_f_renorm.f:93-103 over all 3V links
__global__ __launch_bounds__(256) void k_renorm(Geom g, double* __restrict__ U) {
  int s = blockIdx.x * TB + threadIdx.x;
  int cls = blockIdx.y;  // mu*2 + p
  if (s >= g.n) return;
  int mu = cls >> 1, p = cls & 1;
  st_link(U, g, mu, p, s, normalized(ld_link(U, g, mu, p, s)));
}

void launch_renorm(lceq_lattice* L, double* U) {
  hipLaunchKernelGGL(k_renorm, dim3(blocks_for(L->g.n), 6), dim3(TB), 0, L->stream, L->g, U);
}

// Field guard: per block of sites (both parities), the largest unitarity
// deviation | |alpha|^2 + |beta|^2 - 1 | of the finite links and the number
// of non-finite values among the links and the Higgs field:
// part[2 blk] = deviation, part[2 blk + 1] = count.
__global__ __launch_bounds__(256) void k_check_fields(Geom g, const double* __restrict__ U,
                                                      const double* __restrict__ A,
                                                      double* __restrict__ part) {
  __shared__ double wmax[4], wbad[4];
  int s = blockIdx.x * TB + threadIdx.x;
  double dev = 0.0, bad = 0.0;
  if (s < g.n) {
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
      for (int mu = 0; mu < 3; ++mu) {
        su2 u = ld_link(U, g, mu, p, s);
        double c[4] = {u.a.re, u.a.im, u.b.re, u.b.im};
#pragma unroll
        for (int k = 0; k < 4; ++k) bad += isfinite(c[k]) ? 0.0 : 1.0;
        double d = fabs(((c[0] * c[0] + c[1] * c[1]) + (c[2] * c[2] + c[3] * c[3])) - 1.0);
        if (isfinite(d)) dev = fmax(dev, d);
      }
      vec3 a = ld_higgs(A, g, p, s);
#pragma unroll
      for (int k = 0; k < 3; ++k) bad += isfinite(a.x[k]) ? 0.0 : 1.0;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    dev = fmax(dev, __shfl_xor(dev, off, 64));
    bad += __shfl_xor(bad, off, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    wmax[threadIdx.x >> 6] = dev;
    wbad[threadIdx.x >> 6] = bad;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[2 * blockIdx.x] = fmax(fmax(wmax[0], wmax[1]), fmax(wmax[2], wmax[3]));
    part[2 * blockIdx.x + 1] = ((wbad[0] + wbad[1]) + wbad[2]) + wbad[3];
  }
}

void launch_check_fields(lceq_lattice* L, double* part) {
  hipLaunchKernelGGL(k_check_fields, dim3(blocks_for(L->g.n)), dim3(TB), 0, L->stream, L->g,
                     L->U, L->A, part);
}

// ========================================================= gauge fixing

// odd site i (0..255) of a tile, in tile coordinates
struct TileSite {
  int x, y, z;
};
__device__ __forceinline__ TileSite tile_odd_site(int i) {
  int y = (i >> 3) & 7, z = i >> 6;
  return TileSite{2 * (i & 7) + ((y + z + 1) & 1), y, z};
}

struct GfArgs {
  int guarded;
  int lx, ly, lz, ntx, nty;  // extents and tiles (k_gfix<DA>)
  double lambda, alpha;
  double* obs;  // OBS_GF_DONE read when guarded; the convergence test writes
  double* part;            // da partials this launch writes, one per tile or block
  double* sites;           // or da itself, one per site (DA_SITES)
  const double* part_old;  // those of the iteration before (check)
  int ntiles, n;
  // convergence test of the previous iteration at the start of this launch
  // (landau_gauge iterations after the first of a batch): `iter` iterations
  // are complete, their last da is in `part_old`
  int check;
  double iter, limit_or, max_iter;
};

// da1 = (sum of the per-block partials of the eo = 1 half) / N
// (f/or_gauge_fixing1.f:156-157), summed in a fixed order that does not
// depend on the caller; every thread of a block of 256 or more must call it.
// The order is that of a block: thread t adds partials t, t + 256, ...; the
// waves' butterflies; the four waves in turn.  Up to 64 partials, one wave's,
// every wave does that by itself, so that a launch that tests the loop condition
// first has no block barriers ahead of its update (32^3: 0.4 us of an iteration;
// with more partials the waves' repeated loads cost more than the barriers: 64^3
// 18.9 us an iteration, 20.7 that way).
__device__ __forceinline__ double gfix_da(const double* __restrict__ part, int nb, double n) {
  if (nb <= 64) {
    const int lane = threadIdx.x & 63;
    return wave_sum(lane < nb ? part[lane] : 0.0) / n;
  }
  __shared__ double red[4];
  double v = 0.0;
  if (threadIdx.x < TB) {
    for (int i0 = threadIdx.x; i0 < nb; i0 += TB * 4) {
      double y[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) y[u] = i0 + TB * u < nb ? part[i0 + TB * u] : 0.0;
#pragma unroll
      for (int u = 0; u < 4; ++u) v += y[u];
    }
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  }
  __syncthreads();
  return (((red[0] + red[1]) + red[2]) + red[3]) / n;
}

// The loop condition of f/landau_gauge.f:54-59 after `iter` iterations
// whose last da is `da`, plus the iteration cap: returns whether to stop;
// one thread records da, the count and the flags.
__device__ __forceinline__ bool gfix_stop(double da, double iter, double limit_or,
                                          double max_iter, double* __restrict__ obs, bool writer) {
  bool conv = !(da > limit_or);
  bool stop = conv || iter >= max_iter;
  if (writer) {
    obs[OBS_DA] = da;
    obs[OBS_ITER] = iter;
    if (stop) obs[OBS_GF_DONE] = iter;
    if (stop && !conv) obs[OBS_GF_CAPPED] = 1.0;
  }
  return stop;
}

// The weighted sum of three links, f/or_gauge_fixing1.f:97-107, :116-142
__device__ __forceinline__ su2 gfix_sum(double alpha, const su2 (&u)[3]) {
  su2 s{c_add(u[0].a, u[1].a), c_add(u[0].b, u[1].b)};
  s.a = c_add(s.a, c_scale(alpha, u[2].a));
  s.b = c_add(s.b, c_scale(alpha, u[2].b));
  return s;
}
__device__ __forceinline__ su2 gfix_w(const su2& s1, const su2& s2) {  // :145-146
  return su2{c_add(s1.a, c_conj(s2.a)), c_sub(s1.b, s2.b)};
}
__device__ __forceinline__ double gfix_site_da(const su2& s1, const su2& s2, const su2& w) {
  double d = c_sub(s1.a, s2.a).im;  // :153-158
  return d * d + (w.b.re * w.b.re + w.b.im * w.b.im);
}
// the overrelaxed gauge transformation of w = s1 + s2^+, :169-242
__device__ __forceinline__ su2 gfix_rotation(const su2& w, double lambda) {
  double k = (w.a.re * w.a.re + w.a.im * w.a.im) + (w.b.re * w.b.re + w.b.im * w.b.im);
  double rk = rsqrt(k);  // w / sqrt(k), :169-183
  su2 o{c_scale(rk, w.a), c_scale(rk, w.b)};
  double ra = fmin(1.0, fmax(-1.0, o.a.re));
  double th = acos(ra);
  if (th != 0.0) {
    double tho = lambda * th, sn, cs;
    sincos(tho, &sn, &cs);
    // sin(th) for th = acos(ra) in (0, pi] is sqrt((1 - ra)(1 + ra)); the
    // factored form keeps full relative precision as th -> 0
    double f = sn * rsqrt((1.0 - ra) * (1.0 + ra));
    double t2 = f * o.a.im;
    o.a = c_mk(cs, -t2);
    o.b = c_mk(-(f * o.b.re), -(f * o.b.im));
  }
  return o;
}

// One parity half of f/or_gauge_fixing1.f:54-328.  Thread x reads and
// writes only U_mu(x) and U_mu(x-mu) for mu = 1..3 and a_f(x), so the half
// step has no cross-thread hazards.  With RENORM (eo = 1 of a
// landau_gauge iteration) every link of the lattice is written exactly once
// and f/u_f_renorm.f is applied on that write.  With check=1 every block
// first repeats the convergence test of the previous iteration (the same
// sum in the same order, so all blocks agree) and the launch returns when
// the loop has ended; the operand loads are issued before the test.
// DA (eo = 1): da's partial sums, one per block, the blocks being tiles or index
// ranges, or da per site (gfix_site_sums says which); the other half's blocks are
// index ranges.  DA and RENORM are template arguments: without a branch around
// each pair, the six normalisations' chains of dependent operations run side by
// side.
enum { DA_NONE, DA_TILES, DA_BLOCKS, DA_SITES };
template <int DA, bool RENORM>
__global__ __launch_bounds__(256) void k_gfix(HEAD_PARAMS, GfArgs p) {
  const Head h = HEAD_OF;
  const Geom& g = h.g;
  double *Uf = h.U, *Af = h.A;
  int blk = xcd_block(h.nb);
  int s = blk * TB + threadIdx.x;
  int eo = DA != DA_NONE ? 1 : h.flags & HEAD_EO, oe = eo ^ 1;
  bool act = s < g.n;
  if (DA == DA_TILES) {
    TileOrigin o = tile_origin<GT_X, GT_Y, GT_Z>(blk, p.ntx, p.nty);
    TileSite t = tile_odd_site(threadIdx.x);
    int x = o.x + t.x, y = o.y + t.y, z = o.z + t.z;
    act = x < p.lx && y < p.ly && z < p.lz;
    s = (x >> 1) + g.h1 * y + g.h2 * z;
  }
  su2 ux[3], uy[3];
  int sy[3];
  vec3 af;
  if (act) {
    Steps st = site_steps(g, site_coord(g, eo, s));
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {
      sy[mu] = s + st.m[mu];
      ux[mu] = ld_link(Uf, g, mu, eo, s);
      uy[mu] = ld_link(Uf, g, mu, oe, sy[mu]);
    }
    af = ld_higgs(Af, g, eo, s);
  }
  // uniform over the grid; tested after the operand loads are issued, so that
  // its round trip overlaps theirs
  if (p.guarded && gfix_ended(p.obs[OBS_GF_DONE], p.check ? p.iter : 0.0)) return;
  if (p.check) {
    double da = gfix_da(p.part_old, p.ntiles, (double)p.n);
    if (gfix_stop(da, p.iter, p.limit_or, p.max_iter, p.obs, blk == 0 && threadIdx.x == 0))
      return;  // block-uniform
  }
  double red[1] = {0.0};
  if (act) {
    su2 s1 = gfix_sum(p.alpha, ux), s2 = gfix_sum(p.alpha, uy), w = gfix_w(s1, s2);
    if (DA != DA_NONE) red[0] = gfix_site_da(s1, s2, w);
    if (DA == DA_SITES) p.sites[s] = red[0];
    su2 o = gfix_rotation(w, p.lambda);
    st_higgs(Af, g, eo, s, adj_rot<false>(o, af));  // g X(a_f) g^+, :243-252
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {  // :256-324
      su2 nx = m_nn(o, ux[mu]);
      su2 ny = m_nd(uy[mu], o);
      if (RENORM) {
        nx = normalized(nx);
        ny = normalized(ny);
      }
      st_link(Uf, g, mu, eo, s, nx);
      st_link(Uf, g, mu, oe, sy[mu], ny);
    }
  }
  if (DA == DA_TILES || DA == DA_BLOCKS) block_sum_store<1>(red, p.part, 0, blk);
}

// da of the odd sites, added by tiles as k_gfix<DA_TILES> and k_gfix_iter do
__global__ __launch_bounds__(256) void k_gfix_site_sums(const double* __restrict__ sites, Geom g,
                                                        int ntx, int nty,
                                                        double* __restrict__ part) {
  const int blk = blockIdx.x;
  const TileOrigin o = tile_origin<GT_X, GT_Y, GT_Z>(blk, ntx, nty);
  const TileSite t = tile_odd_site(threadIdx.x);
  const int x = o.x + t.x, y = o.y + t.y, z = o.z + t.z;
  double red[1] = {0.0};
  if (x < g.lx && y < g.ly && z < g.lz) red[0] = sites[(x >> 1) + g.h1 * y + g.h2 * z];
  block_sum_store<1>(red, part, 0, blk);
}

// Slot of the even site at tile coordinates (x, y, z), which is in the tile
// (0..255, in the order of tile_odd_site) or one step out of it along one axis:
// x = -1 16 slots from 256, x = 16 from 272, y = -1 32 from 288, y = 8 from 320,
// z = -1 64 from 352, z = 4 from 416
constexpr int GT_SLOTS = 480, GT_TB = 512;
__device__ __forceinline__ int tile_slot(int x, int y, int z) {
  if (x < 0) return 256 + 4 * z + (y >> 1);
  if (x >= GT_X) return 272 + 4 * z + (y >> 1);
  if (y < 0) return 288 + 8 * z + (x >> 1);
  if (y >= GT_Y) return 320 + 8 * z + (x >> 1);
  if (z < 0) return 352 + 8 * y + (x >> 1);
  if (z >= GT_Z) return 416 + 8 * y + (x >> 1);
  return 64 * z + 8 * y + (x >> 1);
}
// and the site of slot e
__device__ __forceinline__ TileSite tile_even_site(int e) {
  if (e < 256) {
    int y = (e >> 3) & 7, z = e >> 6;
    return TileSite{2 * (e & 7) + ((y + z) & 1), y, z};
  }
  if (e < 288) {  // x = -1 beside odd sites at x = 0: y + z odd; x = 16: even
    int f = (e - 256) & 15, far = e >= 272, z = f >> 2;
    return TileSite{far ? GT_X : -1, 2 * (f & 3) + ((z + 1 + far) & 1), z};
  }
  if (e < 352) {
    int f = (e - 288) & 31, far = e >= 320, z = f >> 3;
    return TileSite{2 * (f & 7) + ((z + 1 + far) & 1), far ? GT_Y : -1, z};
  }
  int f = (e - 352) & 63, far = e >= 416, y = f >> 3;
  return TileSite{2 * (f & 7) + ((y + 1 + far) & 1), y, far ? GT_Z : -1};
}

// One landau_gauge iteration, both half steps and u_f_renorm, from the links
// src to dst.  A block owns a tile's 256 odd sites, whose six links each are
// every link once.  The even half step's rotations that those links see, of the
// tile's even sites and the ones a step outside it, are formed first, one per
// thread, into LDS (480 for 256 sites; the ones outside are another block's
// too, and come out the same there, since src does not change).  Then each odd
// site applies them to its links, takes its own rotation, and writes its links
// normalised.  Both half steps as launches of their own read and write every
// link (432 bytes a site of the lattice and iteration with a_f), here once (240, and
// the faces), and one launch instead of two.  The arithmetic per site and link is
// k_gfix's.
// What bounds it on lattices the Infinity Cache holds is the chain of a block: two
// rounds of dependent gathers, the loop condition's flag and partials ahead of the
// first, a barrier in each, with half the waves idle after the second.  Counters at
// 64^3 (14.3 us): waves wait 43% of their cycles, the vector unit issues for 37% of
// the launch (763 instructions a wave, half of them FP64), and 71 MB pass the L2s,
// 5.0 TB/s (63 MB without the faces).  Beyond the cache HBM: 160^3 1.26 GB in 266 us,
// 4.7 TB/s.  Below 40^3 the launch.  An iteration in
// us, two launches and one: 8^3 8.6 6.4, 16^3 8.6 6.9, 32^3 9.4 7.4, 48^3 12.1
// 9.1, 64^3 18.5 14.1, 96^3 56 43, 160^3 361 276; 4^3 (16 odd sites) even.
// WT: links stored through the L2.  Beyond the Infinity Cache they are not: a
// tile's rows are 128-byte pieces, which end inside lines where lx is not a
// multiple of 16, and memory then takes the lines whole, not piece by piece: us
// an iteration, through and not, 140^3 254 223, 180x150x150 393 341, 160^3 288
// 276; in the cache 64^3 13.9 15.4.
template <bool WT>
__global__ __launch_bounds__(GT_TB) void k_gfix_iter(const double* __restrict__ src,
                                                     double* __restrict__ dst,
                                                     double* __restrict__ Af, uint64_t h1_ly,
                                                     uint64_t lz_npad, uint64_t tiles_ntx,
                                                     uint64_t nty_n, GfArgs p) {
  __shared__ double2 ga[GT_SLOTS], gb[GT_SLOTS];
  const int h1 = half0(h1_ly), ly = half1(h1_ly), lz = half0(lz_npad), lx = 2 * h1;
  Geom g{0, 0, 0, h1, h1 * ly, half1(nty_n), half1(lz_npad), 0.0f, 0.0f, (ly - 1) * h1,
         (lz - 1) * h1 * ly};
  const int blk = xcd_block(half0(tiles_ntx)), tid = threadIdx.x;
  const TileOrigin o = tile_origin<GT_X, GT_Y, GT_Z>(blk, half1(tiles_ntx), half0(nty_n));
  // the even sites
  const TileSite te = tile_even_site(min(tid, GT_SLOTS - 1));
  int ex = o.x + te.x, ey = o.y + te.y, ez = o.z + te.z;
  const bool eact = tid < GT_SLOTS && ex <= lx && ey <= ly && ez <= lz;
  const bool own = tid < 256 && ex < lx && ey < ly && ez < lz;
  ex = ex < 0 ? lx - 1 : ex >= lx ? ex - lx : ex;
  ey = ey < 0 ? ly - 1 : ey >= ly ? ey - ly : ey;
  ez = ez < 0 ? lz - 1 : ez >= lz ? ez - lz : ez;
  const unsigned es = (unsigned)((ex >> 1) + g.h1 * ey + g.h2 * ez);
  su2 ux[3], uy[3];
  vec3 ae;
  if (eact) {
    Steps st = site_steps(g, Coord{ex >> 1, ey * g.h1, ez * g.h2, (bool)(ex & 1)});
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {
      ux[mu] = ld_link(src, g, mu, 0, es);
      uy[mu] = ld_link(src, g, mu, 1, (unsigned)((int)es + st.m[mu]));
    }
    if (own) ae = ld_higgs(Af, g, 0, es);
  }
  // the loop condition, as in k_gfix
  if (gfix_ended(p.obs[OBS_GF_DONE], p.check ? p.iter : 0.0)) return;
  if (p.check) {
    double da = gfix_da(p.part_old, p.ntiles, (double)p.n);
    if (gfix_stop(da, p.iter, p.limit_or, p.max_iter, p.obs, blk == 0 && tid == 0)) return;
  }
  su2 w;
  if (eact) w = gfix_w(gfix_sum(p.alpha, ux), gfix_sum(p.alpha, uy));
  // the odd site's operands, on their way while the even rotation is formed
  const TileSite t = tile_odd_site(tid & 255);
  const int x = o.x + t.x, y = o.y + t.y, z = o.z + t.z;
  const bool act = tid < 256 && x < lx && y < ly && z < lz;
  const int s = (x >> 1) + g.h1 * y + g.h2 * z;
  int sy[3];
  vec3 ao;
  if (act) {
    Steps st = site_steps(g, Coord{x >> 1, y * g.h1, z * g.h2, (bool)(x & 1)});
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {
      sy[mu] = s + st.m[mu];
      ux[mu] = ld_link(src, g, mu, 1, (unsigned)s);
      uy[mu] = ld_link(src, g, mu, 0, (unsigned)sy[mu]);
    }
    ao = ld_higgs(Af, g, 1, (unsigned)s);
  }
  if (eact) {
    su2 r = gfix_rotation(w, p.lambda);
    ga[tid] = double2{r.a.re, r.a.im};
    gb[tid] = double2{r.b.re, r.b.im};
    if (own) st_higgs(Af, g, 0, es, adj_rot<false>(r, ae));
  }
  __syncthreads();
  double red[1] = {0.0};
  if (act) {
    auto rot = [&](int dx, int dy, int dz) {
      int e = tile_slot(t.x + dx, t.y + dy, t.z + dz);
      return su2{c_mk(ga[e].x, ga[e].y), c_mk(gb[e].x, gb[e].y)};
    };
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {
      ux[mu] = m_nd(ux[mu], rot(mu == 0, mu == 1, mu == 2));
      uy[mu] = m_nn(rot(-(mu == 0), -(mu == 1), -(mu == 2)), uy[mu]);
    }
    su2 s1 = gfix_sum(p.alpha, ux), s2 = gfix_sum(p.alpha, uy);
    w = gfix_w(s1, s2);
    red[0] = gfix_site_da(s1, s2, w);
    su2 r = gfix_rotation(w, p.lambda);
    st_higgs(Af, g, 1, (unsigned)s, adj_rot<false>(r, ao));
#pragma unroll
    for (int mu = 0; mu < 3; ++mu) {
      st_link<WT>(dst, g, mu, 1, (unsigned)s, normalized(m_nn(r, ux[mu])));
      st_link<WT>(dst, g, mu, 0, (unsigned)sy[mu], normalized(m_nd(uy[mu], r)));
    }
  }
  block_sum_store<1, GT_TB / 64>(red, p.part, 0, blk);
}

// da1 after one or_gauge_fixing call (guarded = 0), or the convergence test
// of a landau_gauge batch's last iteration (guarded = 1, `iter` iterations
// complete): the loop ends when da1 <= limit_or or at the iteration cap.  With
// `host` the loop's observables also go to pinned memory there.
__global__ __launch_bounds__(256) void k_gfix_finalize(const double* __restrict__ part, int nb,
                                                       double n, int guarded, double iter,
                                                       double limit_or, double max_iter,
                                                       double* __restrict__ obs,
                                                       double* __restrict__ host) {
  if (!guarded || obs[OBS_GF_DONE] == 0.0) {
    double da = gfix_da(part, nb, n);
    if (guarded)
      gfix_stop(da, iter, limit_or, max_iter, obs, threadIdx.x == 0);
    else if (threadIdx.x == 0)
      obs[OBS_DA] = da;
  }
  // thread 0 wrote what has changed, so it alone copies
  if (host && threadIdx.x == 0) {
    host[OBS_DA] = obs[OBS_DA];
    host[OBS_ITER] = obs[OBS_ITER];
    host[OBS_GF_DONE] = obs[OBS_GF_DONE];
    host[OBS_GF_CAPPED] = obs[OBS_GF_CAPPED];
  }
}

// Start of landau_gauge (f/landau_gauge.f:26-52): u -> u_f, a -> a_f, da1 =
// 10000, no iterations, not converged; one launch for two copies and two
// uploads (16-byte elements, the arrays are whole 64-site rows of them)
__global__ __launch_bounds__(TB) void k_gfix_begin(const double2* __restrict__ U,
                                                   const double2* __restrict__ A,
                                                   double2* __restrict__ Uf,
                                                   double2* __restrict__ Af, unsigned nu,
                                                   unsigned na, double* __restrict__ obs) {
  unsigned i = blockIdx.x * TB + threadIdx.x;
  if (i < nu)
    Uf[i] = U[i];
  else if (i - nu < na)
    Af[i - nu] = A[i - nu];
  if (i == 0) {
    obs[OBS_DA] = 10000.0;
    obs[OBS_ITER] = 0.0;
    obs[OBS_GF_DONE] = 0.0;
    obs[OBS_GF_CAPPED] = 0.0;
  }
}

void launch_gfix_begin(lceq_lattice* L, bool links) {
  unsigned nu = links ? 12 * (unsigned)L->g.npad : 0, na = 3 * (unsigned)L->g.npad;
  hipLaunchKernelGGL(k_gfix_begin, dim3((nu + na + TB - 1) / TB), dim3(TB), 0, L->stream,
                     (const double2*)L->U, (const double2*)L->A, (double2*)L->Uf,
                     (double2*)L->Af, nu, na, L->obs);
}

// da's partial sums: one per tile or per block of site indices
static int gfix_sums(const Geom& g) {
  return gfix_tile_order(g) ? lattice_tiles(g) : blocks_for(g.n);
}

static GfArgs gfix_args(lceq_lattice* L, int guarded, int check, int iter) {
  const Geom& g = L->g;
  GfArgs a;
  a.guarded = guarded;
  a.lx = g.lx;
  a.ly = g.ly;
  a.lz = g.lz;
  a.ntx = tiles_along(g.lx, GT_X);
  a.nty = tiles_along(g.ly, GT_Y);
  a.lambda = L->lambda;
  a.alpha = L->alpha;
  a.obs = L->obs;
  a.part = L->gf_part;
  a.part_old = L->gf_part;
  a.sites = L->gf_part + 2 * (size_t)lattice_tiles(g);
  a.ntiles = gfix_sums(g);
  a.n = g.n;
  a.check = check;
  a.iter = (double)iter;
  a.limit_or = L->limit_or;
  a.max_iter = (double)L->max_iter;
  return a;
}

void launch_gfix(lceq_lattice* L, int eo, int renorm, int guarded, int check, int iter) {
  GfArgs a = gfix_args(L, guarded, check, iter);
  prof_begin(L, KC_GFIX);
  prof_count(L, KC_GFIX);
  const Geom& g = L->g;
  const bool tiles = gfix_tile_order(g), sites = gfix_site_sums(g);
  int nb = eo && tiles && !sites ? a.ntiles : blocks_for(g.n);
  HeadArgs h = head_args(L, L->Uf, L->Af, nb, eo);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nb), dim3(TB), 0, L->stream, h.U, h.A, h.n, h.b, h.h, h.w, h.r,
                       a);
  };
  if (!eo)
    launch(k_gfix<DA_NONE, false>);
  else if (sites)
    renorm ? launch(k_gfix<DA_SITES, true>) : launch(k_gfix<DA_SITES, false>);
  else if (tiles)
    renorm ? launch(k_gfix<DA_TILES, true>) : launch(k_gfix<DA_TILES, false>);
  else
    renorm ? launch(k_gfix<DA_BLOCKS, true>) : launch(k_gfix<DA_BLOCKS, false>);
  prof_end(L, KC_GFIX);
  // after the loop's end the sites hold the last iteration's da, whose sums these
  // are again
  if (eo && sites)
    hipLaunchKernelGGL(k_gfix_site_sums, dim3(a.ntiles), dim3(TB), 0, L->stream, a.sites, g, a.ntx,
                       a.nty, a.part);
}

// The link array iteration `iter` (from 1) of the one-launch loop writes: u_f
// and the second array in turn
static double* gfix_out(const lceq_lattice* L, int iter) { return iter & 1 ? L->Uf : L->spare; }

void launch_gfix_iter(lceq_lattice* L, int iter, int check) {
  GfArgs a = gfix_args(L, 1, check, iter - 1);
  // the partials too: a block may write its own while another still tests
  a.part = L->gf_part + (size_t)(iter & 1) * a.ntiles;
  a.part_old = L->gf_part + (size_t)((iter - 1) & 1) * a.ntiles;
  const Geom& g = L->g;
  prof_begin(L, KC_GFIX);
  prof_count(L, KC_GFIX);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(a.ntiles), dim3(GT_TB), 0, L->stream,
                       iter == 1 ? L->U : gfix_out(L, iter - 1), gfix_out(L, iter), L->Af,
                       halves(g.h1, g.ly), halves(g.lz, g.npad), halves(a.ntiles, a.ntx),
                       halves(a.nty, g.n), a);
  };
  if (gfix_links_cached(g))
    launch(k_gfix_iter<true>);
  else
    launch(k_gfix_iter<false>);
  prof_end(L, KC_GFIX);
}

void launch_gfix_finalize(lceq_lattice* L, int guarded, int iter, bool to_host, bool one_launch) {
  int nt = gfix_sums(L->g);
  hipLaunchKernelGGL(k_gfix_finalize, dim3(1), dim3(TB), 0, L->stream,
                     L->gf_part + (one_launch ? (size_t)(iter & 1) * nt : 0), nt, (double)L->g.n,
                     guarded, (double)iter, L->limit_or, (double)L->max_iter, L->obs,
                     to_host ? L->pin : nullptr);
}

// ========================================================== correlators

// z-slice sums over both parities (f/correlator.f:53-79, f/scalarcorr.f:43-56,
// f/polyakov.f:47-58), each slice split over `split` blocks (about 512
// sites each, corr_split).  Quantities q (partial j at
// slices[(q*lz + z)*split + j]):
//   0-2 a_f(1..3); 3+3*mu: Im alpha_mu, 4+3*mu: Im beta_mu, 5+3*mu: -Re beta_mu
//   (the (Im a, -i b) projection of u_f); 12 rho(a); 13 cos(4|a|).
// A measurement sums only what it uses: MEAS 0 (correlator) 0-11 from u_f and
// a_f, 1 (scalarcorr) 12 and 2 (polyakov) 13 from a, 24 of 144 bytes a site.
template <int MEAS>
__global__ __launch_bounds__(256) void k_slices(Geom g, int split,
                                                const double* __restrict__ Uf,
                                                const double* __restrict__ Af,
                                                const double* __restrict__ A,
                                                double* __restrict__ slices) {
  constexpr int Q0 = MEAS == 0 ? 0 : 11 + MEAS, NQ = MEAS == 0 ? 12 : 1;
  __shared__ double red[4][NQ];
  int z = blockIdx.x, j = blockIdx.y;
  int nz = 2 * g.h2, chunk = (nz + split - 1) / split;
  int i0 = j * chunk, i1 = min(nz, i0 + chunk);
  double acc[NQ];
#pragma unroll
  for (int q = 0; q < NQ; ++q) acc[q] = 0.0;
  for (int i = i0 + threadIdx.x; i < i1; i += TB) {
    int p = i >= g.h2, s = z * g.h2 + (i - p * g.h2);
    if constexpr (MEAS == 0) {
      vec3 af = ld_higgs(Af, g, p, s);
#pragma unroll
      for (int k = 0; k < 3; ++k) acc[k] += af.x[k];
#pragma unroll
      for (int mu = 0; mu < 3; ++mu) {
        su2 u = ld_link(Uf, g, mu, p, s);
        acc[3 + 3 * mu] += u.a.im;
        acc[4 + 3 * mu] += u.b.im;
        acc[5 + 3 * mu] -= u.b.re;
      }
    } else {
      vec3 a = ld_higgs(A, g, p, s);
      double rho = a.x[0] * a.x[0] + a.x[1] * a.x[1] + a.x[2] * a.x[2];
      acc[0] += MEAS == 1 ? rho : cos(4.0 * sqrt(rho));
    }
  }
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    double t = wave_sum(acc[q]);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][q] = t;
  }
  __syncthreads();
  if (threadIdx.x < NQ) {
    int q = threadIdx.x;
    slices[((Q0 + q) * g.lz + z) * split + j] = ((red[0][q] + red[1][q]) + red[2][q]) + red[3][q];
  }
}

// Periodic z-correlators on the slice means (f/correlator.f:139-164,
// f/scalarcorr.f:96-104, f/polyakov.f:97-107).  corr layout: [0,lz) C_a,
// [lz,2lz) C_u, [2lz,3lz) C_3, [3lz,4lz) rho, [4lz,5lz) Polyakov, then
// mean(rho), mean(P)^2, a0f(1..3); a copy goes to pinned host memory where it
// fits (host), and a0f to the observables.
// A block sums the slice partials of its correlator's quantities in a fixed
// order into slice means, in LDS (dynamic, 6 lz doubles; LDS = false: read
// from `slices`, with split = 1, each time).  What bounds it is latency: a
// correlator is lz dependent additions in x0 order.  The three correlators of
// u_f and a_f take one block each per CORR_Z separations, whose threads form
// the products of CORR_X slices with their partners for one thread per
// separation to add; rho and Polyakov are one multiply-add a slice, a thread
// per separation.  At lz = 128, 19.5 us for correlator with a thread per
// separation that also forms the products, 7.0 us as here.
constexpr int CORR_TB = 256;
constexpr int CORR_MAX_SPLIT = 16;
constexpr int CORR_Z = 16, CORR_X = 128;

template <bool LDS>
__global__ __launch_bounds__(CORR_TB) void k_corr(Geom g, int split, int meas,
                                                  const double* __restrict__ slices,
                                                  double* __restrict__ corr,
                                                  double* __restrict__ host,
                                                  double* __restrict__ obs) {
  extern __shared__ double lds_slices[];
  __shared__ double prod[CORR_Z][CORR_X + 1];
  const int lz = g.lz, tid = threadIdx.x;
  const double area = (double)(g.lx * g.ly);
  const int kind = meas == 0 ? (int)blockIdx.y : 2 + meas;
  const int zper = meas == 0 ? CORR_Z : CORR_TB;
  const int z0 = (int)blockIdx.x * zper;
  const int q0 = kind < 2 ? 3 * kind : kind == 2 ? 9 : 9 + kind;  // first quantity
  const int nq = kind >= 3 ? 1 : kind == 1 ? 6 : 3;
  const double* part = slices + (size_t)q0 * lz * split;
  // all partials of an element are loaded before they are added (in order)
  if (LDS) {
    for (int i = tid; i < nq * lz; i += CORR_TB) {
      double y[CORR_MAX_SPLIT];
#pragma unroll
      for (int j = 0; j < CORR_MAX_SPLIT; ++j) y[j] = j < split ? part[i * split + j] : 0.0;
      double v = 0.0;
#pragma unroll
      for (int j = 0; j < CORR_MAX_SPLIT; ++j)
        if (j < split) v += y[j];
      lds_slices[i] = v / area;
    }
    __syncthreads();
  }
  auto mean = [&](int q, int x) {
    return LDS ? lds_slices[q * lz + x] : (0.0 + part[(size_t)q * lz + x]) / area;
  };
  auto put = [&](int i, double v) {
    corr[i] = v;
    if (host) host[i] = v;
  };
  auto product = [&](int x0, int x1) {
    if (kind == 0) {
      double d = 0.0;
#pragma unroll
      for (int k = 0; k < 3; ++k) d = d + mean(k, x0) * mean(k, x1);
      return d;
    }
    if (kind == 1) {  // Re[A1 A1' + A2 conj(A2')] for mu = 1,2, A1 real
      double t = 0.0;
#pragma unroll
      for (int mu = 0; mu < 2; ++mu) {
        double a1 = mean(3 * mu, x0), a1p = mean(3 * mu, x1);
        double br = mean(1 + 3 * mu, x0), bi = mean(2 + 3 * mu, x0);
        double brp = mean(1 + 3 * mu, x1), bip = mean(2 + 3 * mu, x1);
        t = t + a1 * a1p;
        t = t + (br * brp + bi * bip);
      }
      return t;
    }
    // mu = 3
    return mean(0, x0) * mean(0, x1) + (mean(1, x0) * mean(1, x1) + mean(2, x0) * mean(2, x1));
  };
  // the means, one quantity per thread, summed over z in order, by the last
  // wave of the first block while the first wave adds products
  auto means = [&]() {
    const int m = tid - (CORR_TB - 64);
    if (z0 != 0 || m < 0 || m >= (kind == 0 ? 3 : kind >= 3 ? 1 : 0)) return;
    double v = 0.0;
#pragma unroll 16
    for (int z = 0; z < lz; ++z) v += mean(m, z);
    v = v / lz;
    // mean(rho), mean(P)^2, a0f(1..3) = mean over sites = mean of slice means
    put(5 * lz + (kind == 0 ? 2 + m : kind - 3), kind == 4 ? v * v : v);
    if (kind == 0) obs[OBS_A0F + m] = v;
  };
  const int zt = z0 + tid;
  const bool adds = tid < zper && zt < lz;
  double c = 0.0;
  if (kind >= 3) {  // rho, Polyakov: one multiply-add per slice
    means();
    if (adds) {
#pragma unroll 16
      for (int x0 = 0; x0 < lz; ++x0) c = c + mean(0, x0) * mean(0, x0 + zt < lz ? x0 + zt : x0 + zt - lz);
    }
  } else {
    for (int xb = 0; xb < lz; xb += CORR_X) {
      const int nx = min(CORR_X, lz - xb);
      for (int i = tid; i < CORR_Z * CORR_X; i += CORR_TB) {
        int zi = i / CORR_X, xi = i % CORR_X, z = z0 + zi, x0 = xb + xi;
        if (xi < nx && z < lz) prod[zi][xi] = product(x0, x0 + z < lz ? x0 + z : x0 + z - lz);
      }
      __syncthreads();
      if (xb == 0) means();
      if (adds) {
#pragma unroll 16
        for (int xi = 0; xi < nx; ++xi) c = c + prod[tid][xi];
      }
      __syncthreads();
    }
  }
  if (adds) put(kind * lz + zt, kind == 1 ? c / (lz * 2) : c / lz);
}

// slice means in LDS up to this many bytes (64 KB per workgroup, of which the
// products take 16.1)
constexpr size_t CORR_LDS_MAX = 47 * 1024;
constexpr int CORR_LDS_Q = 6;  // most quantities of one correlator

int corr_split(const Geom& g) {
  if (CORR_LDS_Q * (size_t)g.lz * sizeof(double) > CORR_LDS_MAX) return 1;
  int nz = 2 * g.h2;
  // 512 sites per block, at most CORR_MAX_SPLIT blocks per slice.  One site
  // per thread (twice the blocks) was measured slower: 64^3 slice sums
  // 11.3 -> 13.4 us (twice the block reductions) and the correlator block
  // 12.5 -> 17.3 us (twice the partials per slice)
  return std::max(1, std::min(CORR_MAX_SPLIT, (nz + 2 * TB - 1) / (2 * TB)));
}

void launch_corr(lceq_lattice* L, int meas, double* host) {
  const Geom& g = L->g;
  int split = corr_split(g);
  dim3 grid(g.lz, split);
  if (meas == 0)
    hipLaunchKernelGGL(k_slices<0>, grid, dim3(TB), 0, L->stream, g, split, L->Uf, L->Af, L->A, L->slices);
  else if (meas == 1)
    hipLaunchKernelGGL(k_slices<1>, grid, dim3(TB), 0, L->stream, g, split, L->Uf, L->Af, L->A, L->slices);
  else
    hipLaunchKernelGGL(k_slices<2>, grid, dim3(TB), 0, L->stream, g, split, L->Uf, L->Af, L->A, L->slices);
  size_t lds = CORR_LDS_Q * (size_t)g.lz * sizeof(double);
  const int zper = meas == 0 ? CORR_Z : CORR_TB;
  dim3 kinds((g.lz + zper - 1) / zper, meas == 0 ? 3 : 1);
  if (lds <= CORR_LDS_MAX)
    hipLaunchKernelGGL(k_corr<true>, kinds, dim3(CORR_TB), lds, L->stream, g, split, meas,
                       L->slices, L->corr, host, L->obs);
  else
    hipLaunchKernelGGL(k_corr<false>, kinds, dim3(CORR_TB), 0, L->stream, g, split, meas,
                       L->slices, L->corr, host, L->obs);
}

// ============================================ array-level entry points

// f/heat_kpi.f:9-101 on n independent sites (b, a0_old in; W out as 4
// doubles per site in (alpha, beta) form); partial 0 of slot 0 counts accepts.
__global__ __launch_bounds__(256) void k_heat_kpi(int n, const double* __restrict__ b,
                                                  const double* __restrict__ a0_old,
                                                  double* __restrict__ v,
                                                  const double* __restrict__ fed, Philox key,
                                                  uint64_t pass, double* __restrict__ part,
                                                  int nb) {
  int s = blockIdx.x * TB + threadIdx.x;
  double red[1] = {0.0};
  if (s < n) {
    double r1, r2, r3, r4, r5, r6;
    if (fed) {
      r1 = fed[3 * s];
      r2 = fed[3 * s + 1];
      r3 = fed[3 * s + 2];
      r4 = fed[3 * n + s];
      r5 = fed[4 * n + s];
      r6 = fed[5 * n + s];
    } else {
      philox_pair(key, (uint32_t)s, 0, pass, 0, r1, r2);
      philox_pair(key, (uint32_t)s, 0, pass, 1, r3, r4);
      philox_pair(key, (uint32_t)s, 0, pass, 2, r5, r6);
    }
    if (r1 == 0.0) r1 = 0.0000033;
    if (r2 == 0.0) r2 = 0.0000066;
    double cc = cos(TPI * r3);
    double a0 = -(log(r1) + log(r2) * (cc * cc)) * b[s];
    bool lacc = r4 * r4 <= (1.0 - 0.5 * a0);
    red[0] = lacc ? 1.0 : 0.0;
    a0 = lacc ? 1.0 - a0 : a0_old[s];
    double a1 = 1.0 - a0 * a0;
    a1 = a1 >= 0.0 ? sqrt(a1) : 0.0;
    double a2 = 2.0 * (r5 - 0.5);
    double tt = 1.0 - a2 * a2;
    double a0b = tt >= 0.0 ? a1 * sqrt(tt) : 0.0;
    double ang = TPI * r6;
    v[4 * (size_t)s] = a0;
    v[4 * (size_t)s + 1] = a1 * a2;
    v[4 * (size_t)s + 2] = a0b * sin(ang);
    v[4 * (size_t)s + 3] = a0b * cos(ang);
  }
  block_sum_store<1>(red, part, nb, blockIdx.x);
}

void launch_heat_kpi(lceq_lattice* L, int n, const double* b, const double* a0_old, double* v,
                     const double* fed, uint64_t pass) {
  int nb = blocks_for(n);
  hipLaunchKernelGGL(k_heat_kpi, dim3(nb), dim3(TB), 0, L->stream, n, b, a0_old, v, fed,
                     Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)}, pass, L->partials, nb);
}

// f/gauss.f:10-31
__global__ __launch_bounds__(256) void k_gauss(int n, const double* __restrict__ r,
                                               double* __restrict__ x,
                                               const double* __restrict__ fed, Philox key,
                                               uint64_t pass) {
  int s = blockIdx.x * TB + threadIdx.x;
  if (s >= n) return;
  double w1, w2;
  if (fed) {
    w1 = fed[s];
    w2 = fed[n + s];
  } else {
    philox_pair(key, (uint32_t)s, 0, pass, 0, w1, w2);
  }
  double t = -1.0 * (1.0 / r[s]) * log(w1);
  x[s] = sqrt(t) * cos(TPI * w2);
}

void launch_gauss(lceq_lattice* L, int n, const double* r, double* x, const double* fed,
                  uint64_t pass) {
  hipLaunchKernelGGL(k_gauss, dim3(blocks_for(n)), dim3(TB), 0, L->stream, n, r, x, fed,
                     Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)}, pass);
}

// f/matmul.f MULTALL{NN,DN,ND,DD,AD,AN} on site vectors (kind 0..5); operands
// in (alpha, beta) quadruples, Higgs triples for AD/AN; s1/s2 may be null.
__global__ __launch_bounds__(256) void k_multall(int kind, const double* __restrict__ op1,
                                                 const double* __restrict__ op2,
                                                 double* __restrict__ out, int n,
                                                 const int* __restrict__ s1,
                                                 const int* __restrict__ s2) {
  int i = blockIdx.x * TB + threadIdx.x;
  if (i >= n) return;
  int i1 = s1 ? s1[i] : i, i2 = s2 ? s2[i] : i;
  const double* q2 = op2 + 4 * (size_t)i2;
  su2 q{c_mk(q2[0], q2[1]), c_mk(q2[2], q2[3])}, h;
  if (kind >= 4) {
    const double* a1 = op1 + 3 * (size_t)i1;
    vec3 a{{a1[0], a1[1], a1[2]}};
    h = kind == 4 ? m_ad(a, q) : m_an(a, q);
  } else {
    const double* q1 = op1 + 4 * (size_t)i1;
    su2 pp{c_mk(q1[0], q1[1]), c_mk(q1[2], q1[3])};
    h = kind == 0 ? m_nn(pp, q) : kind == 1 ? m_dn(pp, q) : kind == 2 ? m_nd(pp, q) : m_dd(pp, q);
  }
  double* o = out + 4 * (size_t)i;
  o[0] = h.a.re;
  o[1] = h.a.im;
  o[2] = h.b.re;
  o[3] = h.b.im;
}

void launch_multall(lceq_lattice* L, int kind, const double* op1, const double* op2, double* out,
                    int n, const int* s1, const int* s2) {
  hipLaunchKernelGGL(k_multall, dim3(blocks_for(n)), dim3(TB), 0, L->stream, kind, op1, op2, out,
                     n, s1, s2);
}

// ======================================================= start configs

// Haar links (four Box-Muller normals, stream 1) and N(0, sigma^2) Higgs
// components (stream 2); counter index = (mu*2+p)*n + s resp. p*n + s.
__global__ __launch_bounds__(256) void k_hotstart(Geom g, double* __restrict__ U,
                                                  double* __restrict__ A, Philox key,
                                                  double sigma) {
  int s = blockIdx.x * TB + threadIdx.x;
  int cls = blockIdx.y;  // 0..5 links, 6..7 Higgs
  if (s >= g.n) return;
  double u0, u1, u2, u3;
  if (cls < 6) {
    uint32_t idx = (uint32_t)(cls * g.n + s);
    philox_pair(key, idx, 1, 0, 0, u0, u1);
    philox_pair(key, idx, 1, 0, 1, u2, u3);
    double r0 = sqrt(-2.0 * log(u0)), r1 = sqrt(-2.0 * log(u2));
    double q0 = r0 * cos(TPI * u1), q1 = r0 * sin(TPI * u1);
    double q2 = r1 * cos(TPI * u3), q3 = r1 * sin(TPI * u3);
    double nrm = 1.0 / sqrt(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3);
    st_link(U, g, cls >> 1, cls & 1, s, su2{c_mk(q0 * nrm, q1 * nrm), c_mk(q2 * nrm, q3 * nrm)});
  } else {
    int p = cls - 6;
    uint32_t idx = (uint32_t)(p * g.n + s);
    philox_pair(key, idx, 2, 0, 0, u0, u1);
    philox_pair(key, idx, 2, 0, 1, u2, u3);
    double r0 = sqrt(-2.0 * log(u0)), r1 = sqrt(-2.0 * log(u2));
    st_higgs(A, g, p, s,
             vec3{{sigma * r0 * cos(TPI * u1), sigma * r0 * sin(TPI * u1),
                   sigma * r1 * cos(TPI * u3)}});
  }
}

void launch_hotstart(lceq_lattice* L, uint64_t seed, double sigma) {
  hipLaunchKernelGGL(k_hotstart, dim3(blocks_for(L->g.n), 8), dim3(TB), 0, L->stream, L->g, L->U,
                     L->A, Philox{(uint32_t)seed, (uint32_t)(seed >> 32)}, sigma);
}

// f/confget.f:295-307 (mode 0) and f/confget.f:528-575 on one rank (mode 1)
__global__ __launch_bounds__(256) void k_startconf(Geom g, double* __restrict__ U,
                                                   double* __restrict__ A, int mode) {
  int s = blockIdx.x * TB + threadIdx.x;
  int cls = blockIdx.y;
  if (s >= g.n) return;
  if (cls < 6) {
    int mu = cls >> 1;
    su2 u;
    if (mode == 0) {
      u = su2{c_mk(1.0, 0.0), c_mk(0.0, 0.0)};
    } else {
      double z = (double)(s / g.h2) * (mu + 1);
      u = su2{c_mk(0.0, z), c_mk(0.0, z)};
    }
    st_link(U, g, mu, cls & 1, s, u);
  } else {
    double c = 1.0 / sqrt(3.0);
    st_higgs(A, g, cls - 6, s, mode == 0 ? vec3{{0.0, 0.0, 1.0}} : vec3{{c, c, c}});
  }
}

void launch_unitconf(lceq_lattice* L) {
  hipLaunchKernelGGL(k_startconf, dim3(blocks_for(L->g.n), 8), dim3(TB), 0, L->stream, L->g, L->U,
                     L->A, 0);
}
void launch_testconf(lceq_lattice* L) {
  hipLaunchKernelGGL(k_startconf, dim3(blocks_for(L->g.n), 8), dim3(TB), 0, L->stream, L->g, L->U,
                     L->A, 1);
}

}  // namespace lceq
