// lceq_link3.hip -- the three direction passes of one parity of a link sweep in
// one launch (no counterpart in the reference, whose f/agauge.f:53-57 runs them
// one after another; k_link is one of them).
//
// Pass mu of parity eo updates U_mu on the sites of that parity.  Of the links
// that the three passes change it reads U_nu at the site itself and at x + mu -
// nu, for nu != mu; every other operand, the links of the other parity and the
// Higgs field, stays as it is.  So, with x running over the sites of a tile T,
//   pass 2 needs the new U_0 and U_1 at x, U_0 at x + 2 - 0, U_1 at x + 2 - 1,
//   pass 1 needs the new U_0 at x and x + 1 - 0,
//   pass 0 nothing new,
// and a block that carries pass 0 out on T, T + 1 - 0, T + 2 - 0 and T + 2 - 1,
// pass 1 on T and T + 2 - 1, and pass 2 on T, has every value itself.  The
// extra sites (111 + 56 for 128 of a 16 x 4 x 4 tile) are other blocks' too and
// come out the same there: the old links are read from one array and the new
// ones written to another, and a draw depends on its site and pass only.
#include <math.h>

#include "lceq_internal.hpp"
#include "lceq_sites.hpp"

namespace lceq {
namespace {

constexpr int L3_TB = 256;
constexpr int L3_PASS2 = 128, L3_PASS1 = 184, L3_PASS0 = 239;  // sites of the passes

struct TileSite {
  int x, y, z;
};
// Site e, in tile coordinates, of parity eo: the tile; y = -1, z 1..4 (32) and
// z = 4, y 0..2 (24) for pass 1; y = 4 (32), x = -1 (15) and z = 4, y = 3 (8) for
// pass 0 alone.  Four of the 15 are sites that no pass needs.
__device__ __forceinline__ TileSite l3_site(int e, int eo) {
  if (e < L3_PASS2) {
    int y = (e >> 3) & 3, z = e >> 5;
    return TileSite{2 * (e & 7) + ((eo + y + z) & 1), y, z};
  }
  int f = e - L3_PASS2;
  if (f < 32) {
    int z = 1 + (f >> 3);
    return TileSite{2 * (f & 7) + ((eo + 1 + z) & 1), -1, z};
  }
  if (e < L3_PASS1) {
    f -= 32;
    int y = f >> 3;
    return TileSite{2 * (f & 7) + ((eo + y) & 1), y, L3_Z};
  }
  f = e - L3_PASS1;
  if (f < 32) {
    int z = f >> 3;
    return TileSite{2 * (f & 7) + ((eo + z) & 1), L3_Y, z};
  }
  f -= 32;
  if (f < 15) {
    int z = f / 3;
    return TileSite{-1, 2 * (f - 3 * z) + ((eo + 1 + z) & 1), z};
  }
  f -= 15;
  return TileSite{2 * f + ((eo + 7) & 1), 3, L3_Z};
}
// LDS place of a site of the box x -1..15, y -1..5, z 0..4 (x by pairs: the
// sites of one parity and row)
constexpr int L3_DY = 9, L3_DZ = 9 * 7, L3_BOX = L3_DZ * 5;
__device__ __forceinline__ int l3_place(int x, int y, int z) {
  return ((x + 1) >> 1) + L3_DY * (y + 1) + L3_DZ * z;
}

struct Link3Args {
  double beta, beta_a;
  Philox key;
  uint64_t pass;
  int n, nty, renorm;
};

// Below two blocks per CU what bounds it is one block's chain of three passes (5.8
// us a launch at 16^3 against three launches of 3.8).  Counters at 96^3, nine
// wave-passes a tile (six without the extra sites): the heatbath's launch (73.7 us)
// issues vector instructions for 65% of its time; the overrelaxation's (49.0 us) for
// 41%, and its waves, two per SIMD on average, wait for 40% of theirs; 200 MB pass the
// L2s, 4.1 TB/s, where three launches per direction move 361 in 55.9 us.  16 x 8 x 4
// tiles (8.3 extra wave-passes for 12) took 8.3 there and lost from 48^3 on;
// four waves per SIMD (the operands not loaded ahead of the draws) is 4% slower
// than three from 64^3 on.  The operands of a pass that the one before it does
// not change are loaded ahead of the barrier.
template <bool KP>
__global__ __launch_bounds__(L3_TB) void k_link3(const double* __restrict__ src,
                                                 const double* __restrict__ other,
                                                 double* __restrict__ dst,
                                                 const double* __restrict__ A, uint64_t h1_ly,
                                                 uint64_t lz_npad, uint64_t tiles_ntx_eo,
                                                 Link3Args p) {
  __shared__ double2 n0a[L3_BOX], n0b[L3_BOX], n1a[L3_BOX], n1b[L3_BOX];
  const int h1 = half0(h1_ly), ly = half1(h1_ly), lz = half0(lz_npad), lx = 2 * h1;
  const int eo = half1(tiles_ntx_eo) & 1, oe = eo ^ 1;
  const Geom g{0, 0, 0, h1, h1 * ly, p.n, half1(lz_npad), 0.0f, 0.0f, (ly - 1) * h1,
               (lz - 1) * h1 * ly};
  const int tid = threadIdx.x;
  const TileOrigin org = tile_origin<L3_X, L3_Y, L3_Z>(xcd_block(half0(tiles_ntx_eo)),
                                                       half1(tiles_ntx_eo) >> 1, p.nty);
  const TileSite t = l3_site(min(tid, L3_PASS0 - 1), eo);
  int x = org.x + t.x, y = org.y + t.y, z = org.z + t.z;
  // one step beyond the far faces (y, z) is the site they wrap to
  const bool in = x < lx && y <= ly && z <= lz;
  const bool act0 = in && tid < L3_PASS0, act1 = in && tid < L3_PASS1;
  const bool own = tid < L3_PASS2 && x < lx && y < ly && z < lz;
  x = x < 0 ? lx - 1 : x;
  y = y < 0 ? ly - 1 : y >= ly ? y - ly : y;
  z = z < 0 ? lz - 1 : z >= lz ? z - lz : z;
  const unsigned s = (unsigned)((x >> 1) + g.h1 * y + g.h2 * z);
  const Steps st = site_steps(g, Coord{x >> 1, y * g.h1, z * g.h2, (bool)(x & 1)});
  auto at_step = [&](int a) { return (unsigned)((int)s + a); };

  LinkSite q;
  q.g = g;
  q.eo = eo;
  q.beta = p.beta;
  q.beta_a = p.beta_a;
  q.key = p.key;
  q.measflag = 0;
  q.renorm = p.renorm;
  double red[3] = {0.0, 0.0, 0.0};  // not used
  bool taken;
  const vec3 ax = ld_higgs(A, g, eo, act0 ? s : 0);
  // operands of direction mu: the link and those that the passes before it do
  // not change (first, second: nu_x and nu_xpmumnu of that nu)
  auto load = [&](LinkOperands& o, int mu, bool first, bool second) {
    const unsigned sxm = at_step(st.p[mu]);
    o.u = ld_link(src, g, mu, eo, s);
    o.ax = ax;
    o.axp = ld_higgs(A, g, oe, sxm);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int nu = k == 0 ? (mu == 0 ? 1 : 0) : (mu == 2 ? 1 : 2);
      o.k.mu_xpnu[k] = ld_link(other, g, mu, oe, at_step(st.p[nu]));
      if (k == 0 ? first : second) o.k.nu_x[k] = ld_link(src, g, nu, eo, s);
      o.k.nu_xpmu[k] = ld_link(other, g, nu, oe, sxm);
      o.k.mu_xmnu[k] = ld_link(other, g, mu, oe, at_step(st.m[nu]));
      o.k.nu_xmnu[k] = ld_link(other, g, nu, oe, at_step(st.m[nu]));
      if (k == 0 ? first : second)
        o.k.nu_xpmumnu[k] = ld_link(src, g, nu, eo, at_step(st.p[mu] + st.m[nu]));
    }
  };
  // LDS places of the site and, less 1 along x, of its neighbours
  const int here = l3_place(t.x, t.y, t.z), left = here - (t.x & 1);
  auto from = [&](const double2* a, const double2* b, int i) {
    return su2{c_mk(a[i].x, a[i].y), c_mk(b[i].x, b[i].y)};
  };
  auto keep = [&](double2* a, double2* b, su2 u) {
    a[here] = double2{u.a.re, u.a.im};
    b[here] = double2{u.b.re, u.b.im};
  };
  auto draw = [&](LinkOperands& o, int mu) {
    q.mu = mu;
    q.pass = p.pass + (uint64_t)mu;
    __builtin_amdgcn_sched_barrier(0);
    link_prepare<KP, false>(q, s, o);
    __builtin_amdgcn_sched_barrier(0);
  };

  // pass 0
  if (act0) {
    LinkOperands o0;
    load(o0, 0, true, true);
    draw(o0, 0);
    su2 u = link_value<KP>(q, o0, taken, red);
    keep(n0a, n0b, u);
    if (own) st_link(dst, g, 0, eo, s, u);
  }
  LinkOperands o1;
  if (act1) {
    load(o1, 1, false, true);
    draw(o1, 1);
  }
  __syncthreads();
  if (act1) {
    o1.k.nu_x[0] = from(n0a, n0b, here);
    o1.k.nu_xpmumnu[0] = from(n0a, n0b, left + L3_DY);
    su2 u = link_value<KP>(q, o1, taken, red);
    keep(n1a, n1b, u);
    if (own) st_link(dst, g, 1, eo, s, u);
  }
  LinkOperands o2;
  if (own) {
    load(o2, 2, false, false);
    draw(o2, 2);
  }
  __syncthreads();
  if (own) {
    o2.k.nu_x[0] = from(n0a, n0b, here);
    o2.k.nu_xpmumnu[0] = from(n0a, n0b, left + L3_DZ);
    o2.k.nu_x[1] = from(n1a, n1b, here);
    o2.k.nu_xpmumnu[1] = from(n1a, n1b, here - L3_DY + L3_DZ);
    st_link(dst, g, 2, eo, s, link_value<KP>(q, o2, taken, red));
  }
}

}  // namespace

void launch_link3(lceq_lattice* L, int kp, int eo, int renorm_on_write, const double* src,
                  const double* other, double* dst, uint64_t pass) {
  const Geom& g = L->g;
  Link3Args a;
  a.beta = L->beta;
  a.beta_a = L->beta_a;
  a.key = Philox{(uint32_t)L->seed, (uint32_t)(L->seed >> 32)};
  a.pass = pass;
  a.n = g.n;
  a.nty = tiles_along(g.ly, L3_Y);
  a.renorm = renorm_on_write;
  const int nt = link3_tiles(g), ntx = tiles_along(g.lx, L3_X);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(nt), dim3(L3_TB), 0, L->stream, src, other, dst, L->A,
                       halves(g.h1, g.ly), halves(g.lz, g.npad), halves(nt, 2 * ntx + eo), a);
  };
  if (kp)
    launch(k_link3<true>);
  else
    launch(k_link3<false>);
}

}  // namespace lceq
