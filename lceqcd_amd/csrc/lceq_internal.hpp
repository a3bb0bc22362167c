// lceq_internal.hpp -- the lattice context shared by the C-ABI layer
// (lceq_api.hip) and the kernel launchers (lceq_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/lceq.h"
#include "lceq_device.hpp"

// number of per-block partial quantities a reduction slot holds
#define LCEQ_NQ 4
// reduction slots per routine call (6 link sub-passes, 2 Higgs parities, ...)
#define LCEQ_NSLOT 8

// device observables (double obs[LCEQ_OBS_N])
enum {
  OBS_PLAQ0 = 0,   // plaq0 of the last link update (f/agauge.f:179-200)
  OBS_A0KIN = 1,   // a0kin of the last Higgs update (f/ahiggs2.f:126-147)
  OBS_A02 = 2,
  OBS_A04 = 3,
  OBS_A0F = 4,     // 4..6: a0f(1..3) (f/meas2a.f:39-48)
  OBS_ACC_LINK = 7,
  OBS_ACC_HIGGS = 8,
  OBS_DA = 9,
  OBS_ITER = 10,
  OBS_DELTA = 11,  // ahiggs1 Metropolis step (device-resident in sweeps)
  OBS_NACCH = 12,  // raw counts of the last link call
  OBS_NACC1 = 13,
  OBS_GF_DONE = 14,  // landau_gauge: iterations after which the loop ended, 0 before
  OBS_GF_CAPPED = 15,
  LCEQ_OBS_N = 16
};

// doubles of lceq_lattice::pin after the observables (64 KiB in all)
#define LCEQ_PIN_DOUBLES (8192 - LCEQ_OBS_N)

namespace lceq {
struct Pinned;
}

struct lceq_lattice {
  lceq::Geom g;
  int vol;
  int device;
  hipStream_t stream;
  // One allocation for the arrays of a small lattice (create_arrays), or null
  char* arena;
  size_t arena_bytes;
  // device fields
  double *U, *A, *Uf, *Af, *Vst, *F;
  // A second link array (spare_links): link sweeps and landau_gauge read one
  // array and write the other, which then change places.  Between calls it
  // holds nothing.  Lattices whose link sweeps use it have it from creation on,
  // so that a sweep allocates nothing, the others from their first landau_gauge.
  double* spare;
  // da partials of two iterations [2][lattice_tiles], then, where gfix_site_sums,
  // one da per odd site [n]
  double* gf_part;
  double *partials;  // [LCEQ_NSLOT][LCEQ_NQ][pstride]
  int pstride;       // >= number of 64-site blocks (the smallest launch shape)
  double *obs;       // [LCEQ_OBS_N]
  // pinned host memory that kernels write results to: the observables, then
  // PIN_DOUBLES values of any other small result
  double *pin;
  lceq::Pinned* pin_block;
  double *hist;      // [hist_cap][LCEQ_OBS_N] per-sweep records
  int hist_cap;
  int hist_rows;     // rows recorded since the last lceq_history
  double *slices;    // correlator slice partial sums [14][lz][corr_split]
  double *corr;      // correlator outputs [5][lz] + 4 scalars
  double *scratch;   // generic device scratch for host-array entry points
  size_t scratch_bytes;
  double *fed;       // fed uniforms
  int64_t fed_cap, fed_n, fed_pos;
  // parameters (reference COMMON /paramet/, f/INCLUDE/input_parameter.inc:66-69)
  double beta, beta_a, beta_2, beta_4, lambda, alpha, limit_or;
  int max_iter, imode;
  // RNG
  int rng_mode;  // 0 fed, 1 philox
  // launch shape of the link and Higgs updates: threads (= sites) per block
  // 64/128/256/512 and the XCD-aware block order (partials sized for 64)
  int tb, xcd;
  // site order of those launches: strips of `strip` y rows, 0 index order, -1 by
  // the lattice's shape (strip_rows)
  int strip;
  int tuning;  // an autotuner times these: sweeps take launches that they apply to
  uint64_t seed, pass;
  // timing of one kernel class (bench instrumentation): one event pair per
  // run of consecutive launches of that class, launches counted inside runs
  int prof_class;
  int prof_n, prof_cap, prof_depth, prof_launches;
  hipEvent_t *prof_ev;
};

namespace lceq {

// record a failure for lceq_last_error() and return `code`
int set_error(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

// Why an lx x ly x lz lattice cannot be created, or nullptr if it can.
// Besides even extents >= 2: 3 V links fit the 32-bit link counters, the
// index divisions need ly, lz < 2^22, and the device loads address a site
// of a class array as an unsigned 32-bit byte offset s * 16 (16-byte link
// halves) and the stores' raw buffer range is 2^32 - 1 bytes, so a parity
// holds fewer than 2^28 sites (s * 16 + 16 <= 2^32 - 16).  Checked before
// any device call.
inline const char* geom_reject(int lx, int ly, int lz) {
  if (lx < 2 || ly < 2 || lz < 2 || (lx & 1) || (ly & 1) || (lz & 1))
    return "extents must be even and >= 2";
  if ((int64_t)lx * ly * lz * 3 > INT32_MAX) return "lattice too large for 32-bit link counters";
  if (ly >= (1 << 22) || lz >= (1 << 22)) return "ly and lz must be below 2^22";
  if ((int64_t)lx * ly * lz / 2 >= ((int64_t)1 << 28))
    return "2^28 or more sites per parity (32-bit byte offsets of 16-byte link halves)";
  return nullptr;
}

enum KernelClass { KC_NONE = 0, KC_LINK_KP = 1, KC_LINK_OR = 2, KC_HIGGS = 3, KC_GFIX = 4 };

// Tiles of the gauge fixing kernels (256 sites of each parity)
constexpr int GT_X = 16, GT_Y = 8, GT_Z = 4;
inline int lattice_tiles(const Geom& g) {
  return tiles_along(g.lx, GT_X) * tiles_along(g.ly, GT_Y) * tiles_along(g.lz, GT_Z);
}
int blocks_for(int n);
// the strip rows of the update launches' site order (0: index order)
int strip_rows(const lceq_lattice* L);
// blocks of the link and Higgs update launches at the lattice's launch shape
int shape_blocks(const lceq_lattice* L);

// Event brackets around runs of launches of the profiled class.  Brackets
// nest (a sweep brackets its launches, each launcher brackets itself); only
// the outermost records events, so back-to-back launches of one class are
// timed without events between them and the average per launch matches the
// kernel's own duration up to the dispatch gaps inside the run.
inline void prof_begin(lceq_lattice* L, int kc) {
  if (L->prof_class != kc) return;
  if (L->prof_depth++ == 0 && L->prof_n + 2 <= L->prof_cap)
    (void)hipEventRecord(L->prof_ev[L->prof_n++], L->stream);
}
inline void prof_end(lceq_lattice* L, int kc) {
  if (L->prof_class != kc) return;
  if (--L->prof_depth == 0 && (L->prof_n & 1))
    (void)hipEventRecord(L->prof_ev[L->prof_n++], L->stream);
}
// one launch of class kc inside an open run
inline void prof_count(lceq_lattice* L, int kc) {
  if (L->prof_class == kc && (L->prof_n & 1)) ++L->prof_launches;
}

// Field transfers (lceq_transfer.hip): the nclass classes of a link (ncomp 4)
// or Higgs (ncomp 3) field of geometry g between `dev` and the caller's host
// array in the reference layout with leading dimension ld, ordered after the
// work queued on `stream`; complete on return.
int transfer_field(hipStream_t stream, int device, const Geom& g, double* dev, double* host,
                   int64_t ld, int ncomp, int nclass, bool get);
// a lattice or batch that transfers fields exists (+1) or is gone (-1)
void transfer_user(int change);
// Pinned host memory of a device, from and to a pool (lceq_transfer.hip); null
// without memory.  A block goes back when no kernel uses it any more.
enum { PINNED_RESULTS, PINNED_SMALL, PINNED_LARGE, PINNED_KINDS };
constexpr size_t PINNED_RESULTS_BYTES = (LCEQ_OBS_N + LCEQ_PIN_DOUBLES) * sizeof(double);
struct Pinned;
Pinned* pinned_take(int device, int kind);
void pinned_give(Pinned* block);
void* pinned_host(Pinned* block);

// launchers (lceq_kernels.hip); all enqueue on L->stream, no host sync.
// Link launches use reduction slots 0-5 ((eo, mu) order), Higgs launches
// slots 6-7 (eo); with reduce = 0 a launch writes no partial sums.
// range (Philox; Higgs: ahiggs1 only): the launch covers these sites alone,
// whole z planes; with partial sums its start is a multiple of the block size.
struct SiteRange {
  int p0, len;  // sites p0 .. p0 + len - 1, modulo the parity's n
};
void launch_link(lceq_lattice* L, int kp, int eo, int mu, int measflag, int renorm_on_write,
                 const double* fed, uint64_t pass, int reduce, const SiteRange* range = nullptr);
// A link sweep without partial sums (Philox), three directions of parity eo in
// one launch: passes pass .. pass + 2, from the links `src` (of parity eo) and
// `other` (of the other one) to `dst`, another array than `src`.  link3_tiles:
// its blocks on lattices where it is the faster way, otherwise 0.
// Half as many link updates again as the launches per direction have, in a third of
// the launches and with 168 bytes a site in place of 408.  Launches per direction
// cost a launch each, so that up to two blocks per CU (512) this one is the faster
// way whatever the tiles hold.  Then the sites count: it takes 0.72-0.74 ns a site
// and sweep from 64^3 to 80x80x64 alike, launches per direction 0.61 as long as the
// fields (31 MB at 64^3) are about the size of the L2s (32 MB), 0.71 at 39 MB
// (64x64x80) and 0.82 at 49 MB (80x80x64, 1600 whole tiles), from where it stays the
// faster way.  With tiles cut off, whose extra sites are more, it does not.  us per
// production sweep of n_or = 4 (one of the five link sweeps is a measured one),
// launches per direction and this one:
//   16^3 (16 tiles) 114-127 89, 32^3 (128) 114-128 91, 44^3 (363) 129 123,
//   64x64x32 (512) 132 118, 50^3 (676) 131 162, 64^3 (1024) 159 188,
//   64x64x80 (1280) 233 239, 80x80x64 (1600) 334 304, 96^3 (3456) 608 572,
//   112x112x96 (4704) 820 757; tiles cut off: 72x72x96 (2160) 371 386,
//   100^3 (4375) 684 758
// The second array counts against the Infinity Cache: 128x128x72 (0.25 GB of
// fields and second array) 786 755, 128x128x80 (0.28) 864 869, 128^3 (0.45)
// 1362 1643.
// A tile of two columns stores lone 16-byte pieces; where they are half the tiles
// or more, up to one block per CU: 18x34x50 (234) 136 102, 18x32x64 (256) 127 101,
// 18x34x66 (306) 137 138, 18x48x64 (384) 128 133, 18x64x64 (512) 122 131.
constexpr int L3_X = 16, L3_Y = 4, L3_Z = 4;
inline int link3_tiles(const Geom& g) {
  const int nt = tiles_along(g.lx, L3_X) * tiles_along(g.ly, L3_Y) * tiles_along(g.lz, L3_Z);
  const bool whole = g.lx % L3_X == 0 && g.ly % L3_Y == 0 && g.lz % L3_Z == 0;
  const bool cached = (240 + 192) * (int64_t)g.npad <= (int64_t)256 << 20;
  const bool narrow = g.lx % L3_X == 2 && g.lx < 2 * L3_X;
  return cached && (nt <= (narrow ? 256 : 512) || (nt >= 1600 && whole)) ? nt : 0;
}
// whether a link sweep without sums takes them: not while a kernel class is timed
// or a launch shape or site order is tuned, which are those of the launches per
// direction (measured and fed sweeps, agauge, link_or)
inline bool takes_link3(const lceq_lattice* L) {
  return L->rng_mode == LCEQ_RNG_PHILOX && L->prof_class == KC_NONE && !L->tuning && L->spare &&
         link3_tiles(L->g);
}
void launch_link3(lceq_lattice* L, int kp, int eo, int renorm_on_write, const double* src,
                  const double* other, double* dst, uint64_t pass);
// One-block reduction of the partial sums into the observables: link_kind
// 0 none, 1 KP (agauge), 2 overrelaxation; higgs_kind 0 none, 1-3 ahiggs1-3;
// with hist_row the observables are also copied into that history row.
// higgs_nb: block partials of the Higgs slots when their launch used another
// shape than the lattice's (0: the lattice's shape).  to_host: the
// observables also go to L->pin, for finish_obs
void launch_finalize(lceq_lattice* L, int link_kind, int link_meas, int higgs_kind,
                     int higgs_meas, double* hist_row, bool to_host, int higgs_nb = 0);
// obs[index] = value, and n doubles (at most LCEQ_PIN_DOUBLES) of device
// memory to L->pin + LCEQ_OBS_N
void launch_set_obs(lceq_lattice* L, int index, double value);
void launch_export(lceq_lattice* L, const double* dev, size_t n);
void launch_staples(lceq_lattice* L, int eo, int mu);
void launch_force(lceq_lattice* L, int eo);
// renorm (Philox ahiggs2 only): every link is normalised first, as by
// launch_renorm
void launch_higgs(lceq_lattice* L, int kind, int eo, int measflag, const double* fed,
                  uint64_t pass, int reduce, bool renorm = false,
                  const SiteRange* range = nullptr);
void launch_renorm(lceq_lattice* L, double* U);
// Whether a reference sweep's renorm goes into the next sweep's first launch;
// not while a kernel class is timed, whose launches are then its own alone
inline bool carries_renorm(const lceq_lattice* L) {
  return L->rng_mode == LCEQ_RNG_PHILOX && L->prof_class == KC_NONE;
}
// per-block (unitarity deviation, non-finite count) of U and A into part[2 nb]
void launch_check_fields(lceq_lattice* L, double* part);
// Whether the gauge-fixing loop ended ahead of a launch: `done` is OBS_GF_DONE,
// `testing` the iterations after which the launch itself tests the loop
// condition (0: it does not).  The launch that finds the loop ended writes the
// flag while other waves of it still read it; its own entry counts as none, so
// that all waves take the same way whichever value they see, on to the test,
// whose block sums need every wave of the block.
__host__ __device__ inline bool gfix_ended(double done, double testing) {
  return done != 0.0 && done != testing;
}
// One half-iteration of gauge fixing (eo = 1 forms da); check = 1 first tests
// the loop condition for the `iter` iterations already complete (see k_gfix).
void launch_gfix(lceq_lattice* L, int eo, int renorm, int guarded, int check = 0, int iter = 0);
// Iteration `iter` (from 1) in one launch, from u or the array the iteration
// before wrote into the other one of u_f and the second array
void launch_gfix_iter(lceq_lattice* L, int iter, int check);
// u_f and a_f are within the Infinity Cache
inline bool gfix_links_cached(const Geom& g) {
  return (192 + 48) * (int64_t)g.npad <= (int64_t)256 << 20;
}
// Whether a landau_gauge iteration is one launch over tiles between two link
// arrays, or two launches in place.  In place:
// - Where the tiles are mostly empty, whose blocks cost as much as full ones, up to
//   an eighth filled (us an iteration in place and in one launch: 2x16x16 7.1 9.4,
//   2x128x64 7.8 8.5, 4x4x2048 9.0 10.6; a quarter 4x64x64 7.8 6.8, 4x128x128 9.3
//   9.1), and up to half beyond two blocks per CU (4x128x256 12.4 15.8, 6x256x128
//   15.2 16.4, 6x256x256 27.0 30.2; half 8x256x256 33.9 31.9).
// - Where the Infinity Cache holds (nearly) one array and a_f but not two.  A row of
//   a tile is 128 bytes; where rows end inside lines (lx no multiple of 16) the
//   stores of neighbouring tiles meet there, and two arrays cost more well before
//   they fill the cache (MiB of two arrays): 102^3 (218) 76 63, 66x128x128 (222) 77
//   68, 104^3 (231, half lines) 78 56, 34x256x128 (229) 74 70-111, 18x256x256 (243)
//   77 73-125, 108^3 (259) 82 110, 110^3 (274) 92 122; whole rows 96x96x128 (243) 79
//   53-74, 128x128x80 (270) 84 82, 112^3 (289) 91 91, 128^3 (453) 140 168.
// - Beyond it, until one array is out of it as well: 132^3 (497) 171 195, 144x130x130
//   (501) 183 187, whole rows from there on: 128x142x142 (531) 180 180, 144^3 (615)
//   236 196, 160^3 361 276; others much later: 136^3 (518) 185 196, 140^3 (565) 197
//   222, 146^3 (641) 264 273, 148^3 (667) 277 271, 150^3 (695) 298 283, 170^3 (1012)
//   454 405; and where a lone site ends rows of few tiles, later still: 50x256x224
//   (590) 220 298, 50x512x512 (2700) 1178 1351, 34x512x400 (1434) 640 640.
inline bool gfix_one_launch(const Geom& g) {
  const int64_t tiles = lattice_tiles(g), room = 512 * tiles, sites = 2 * (int64_t)g.n;
  if (8 * sites <= room || (tiles > 512 && 2 * sites < room)) return false;
  const int64_t one_array = 240 * (int64_t)g.npad >> 20, two_arrays = 432 * (int64_t)g.npad >> 20;
  const int end = g.lx % GT_X;  // sites in the last tile of a row, 0: all
  if (two_arrays < (end == 0 ? 288 : end == 8 ? 232 : 224)) return true;
  if (one_array < 280) return false;
  return end == 0 || (two_arrays >= 650 && !(end == 2 && g.lx < 64));
}
// The order of da's sum, one for each lattice, so that landau_gauge and a host
// loop over or_gauge_fixing form the same da and stop after the same iteration: by
// tiles where landau_gauge's iterations are launches over tiles, otherwise by the
// half step's blocks of site indices
inline bool gfix_tile_order(const Geom& g) { return gfix_one_launch(g); }
// The odd half step of an order by tiles runs over tiles itself, or over site
// indices where cut-off tiles cost more (and beyond the Infinity Cache), with one
// da stored per site and added by tiles in a launch of its own.  us a call of
// or_gauge_fixing, by tiles and by indices (without that launch, 3 us): 34x64x64
// (384 tiles) 27.5 25.5, 50x64x64 (512) 31.4 28.0, 66x64x64 (640) 39.6 34.5, 100^3
// 88.4 76.1, 18x256x256 112.6 88.0; whole tiles 64^3 32.1 31.2.
inline bool gfix_site_sums(const Geom& g) {
  const bool whole = g.lx % GT_X == 0 && g.ly % GT_Y == 0 && g.lz % GT_Z == 0;
  return gfix_tile_order(g) && !(gfix_links_cached(g) && (whole || lattice_tiles(g) <= 512));
}
// one_launch: the iterations were launch_gfix_iter's
void launch_gfix_finalize(lceq_lattice* L, int guarded, int iter, bool to_host, bool one_launch);
// a_f = a, with `links` u_f = u, and the loop's observables as before its first
// iteration
void launch_gfix_begin(lceq_lattice* L, bool links);
// blocks per z slice of the slice sums (the slices buffer holds 14 lz split)
int corr_split(const Geom& g);
// the slice sums and correlators of measurement meas (0 correlator, which
// also sets a0f in the observables, 1 scalarcorr, 2 polyakov) into L->corr
// and, where host is not null, the pinned copy there
void launch_corr(lceq_lattice* L, int meas, double* host);
void launch_heat_kpi(lceq_lattice* L, int n, const double* b, const double* a0_old, double* v,
                     const double* fed, uint64_t pass);
void launch_gauss(lceq_lattice* L, int n, const double* r, double* x, const double* fed,
                  uint64_t pass);
void launch_multall(lceq_lattice* L, int kind, const double* op1, const double* op2,
                    double* out, int n, const int* s1, const int* s2);
void launch_hotstart(lceq_lattice* L, uint64_t seed, double sigma);
void launch_unitconf(lceq_lattice* L);
void launch_testconf(lceq_lattice* L);

}  // namespace lceq

// helpers of the C ABI layer (lceq_api.hip) shared with the other entry files
int check_launch();
uint64_t next_pass(lceq_lattice* L);
// n doubles of device memory to the host, after the work queued so far
int read_small(lceq_lattice* L, const double* dev, size_t n, double* host);
int read_obs(lceq_lattice* L, double* host);
// waits for a launch_finalize with to_host; its observables are in L->pin
int finish_obs(lceq_lattice* L);
// one full link sweep (six (eo, mu) launches) of the KP heatbath or the
// overrelaxation, partials in slots 0-5 when reduce is set
int link_sweep(lceq_lattice* L, int kp, int measflag, int renorm_on_write, int reduce);
