// h3dmg_kernels.hip -- gfx950 kernels of the pressure-Poisson multigrid.
//
// All kernels are HBM-streaming 7-point stencils over the colour-split level
// arrays described in h3dmg_internal.h.  A launch covers every (active) block
// at one level: workgroups read their (block, tile) from a tile table, so one
// launch serves a single 256^3 block and 48 uneven blocks alike.
//
// Arithmetic is written in the order of src_v70/mgsolver.for and the library
// is built with -ffp-contract=off, so the FP64 path is bitwise the reference.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "h3dmg_internal.h"

namespace h3dmg {

namespace {

__device__ __forceinline__ size_t cidx(int H, int nj, int i, int j, int k) {
  return ((size_t)k * (size_t)nj + (size_t)j) * (size_t)H + (size_t)(i >> 1);
}

// image of a 0-based coordinate that may lie one cell outside [0, n)
__device__ __forceinline__ int image(int x, int n, bool periodic) {
  if (x < 0) return periodic ? n - 1 : 0;
  if (x >= n) return periodic ? 0 : n - 1;
  return x;
}

template <class T>
struct Coef {
  T aw, ae, as, an, ab, at, ap;
};

// Face f (0 west, 1 east, 2 south, 3 north, 4 bottom, 5 top) of a level or
// finest-level descriptor is a wall when its axis is not periodic and no
// neighbour block lies across it.
template <class LD>
__device__ __forceinline__ bool wall_face(const LD &L, int f) {
  return !((L.per >> (f >> 1)) & 1) && L.nbr[f] < 0;
}

// coeff, mgsolver.for:185-210: 1/h^2 towards every face, 0 towards a
// physical (non-periodic, neighbourless) face, ap = -1*(sum) summed aw..at
// left to right.
template <class T>
__device__ __forceinline__ Coef<T> cell_coef(const LevelDev &L, int i, int j, int k) {
  const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
  Coef<T> c;
  c.aw = (i == 0 && wall_face(L, 0)) ? T(0) : cx;
  c.ae = (i == L.ni - 1 && wall_face(L, 1)) ? T(0) : cx;
  c.as = (j == 0 && wall_face(L, 2)) ? T(0) : cy;
  c.an = (j == L.nj - 1 && wall_face(L, 3)) ? T(0) : cy;
  c.ab = (k == 0 && wall_face(L, 4)) ? T(0) : cz;
  c.at = (k == L.nk - 1 && wall_face(L, 5)) ? T(0) : cz;
  c.ap = T(-1) * (c.aw + c.ae + c.as + c.an + c.ab + c.at);
  return c;
}

__device__ __forceinline__ Coef<double> fine_coef(const FineDev &F, int i, int j, int k) {
  Coef<double> c;
  c.aw = (i == 0 && wall_face(F, 0)) ? 0.0 : F.cx;
  c.ae = (i == F.ni - 1 && wall_face(F, 1)) ? 0.0 : F.cx;
  c.as = (j == 0 && wall_face(F, 2)) ? 0.0 : F.cy;
  c.an = (j == F.nj - 1 && wall_face(F, 3)) ? 0.0 : F.cy;
  c.ab = (k == 0 && wall_face(F, 4)) ? 0.0 : F.cz;
  c.at = (k == F.nk - 1 && wall_face(F, 5)) ? 0.0 : F.cz;
  c.ap = -1.0 * (c.aw + c.ae + c.as + c.an + c.ab + c.at);
  return c;
}

// The cell whose value a ghost holds after exchangepp (exchangepp.for:44-
// 1105, then mgbound and exchbc_mgpp, :2830-2832): (x, y, z) is a padded
// position in [-1, n] of descriptor d of `tab`; on return it is an interior
// position of the returned descriptor.  Walls mirror first, in the block
// itself (mgbound runs over whole faces after the face syncs); then along x,
// y and z in turn a coordinate outside the block moves into the neighbour
// across that face, or wraps around a periodic axis.  In a box of blocks
// this is the value the reference's sequence of whole-face copies, corner
// and edge messages and mirrors leaves in every face, edge and corner ghost.
template <class LD>
__device__ __forceinline__ int resolve_cell(const LD *__restrict__ tab, int d, int &x, int &y,
                                            int &z) {
  const LD *P = &tab[d];
  if (x < 0 && wall_face(*P, 0)) x = 0;
  if (x >= P->ni && wall_face(*P, 1)) x = P->ni - 1;
  if (y < 0 && wall_face(*P, 2)) y = 0;
  if (y >= P->nj && wall_face(*P, 3)) y = P->nj - 1;
  if (z < 0 && wall_face(*P, 4)) z = 0;
  if (z >= P->nk && wall_face(*P, 5)) z = P->nk - 1;
  int c[3] = {x, y, z};
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const int n = a == 0 ? P->ni : a == 1 ? P->nj : P->nk;
    if (c[a] < 0) {
      if (P->nbr[2 * a] >= 0) {
        d = P->nbr[2 * a];
        P = &tab[d];
        c[a] += a == 0 ? P->ni : a == 1 ? P->nj : P->nk;
      } else {
        c[a] = ((P->per >> a) & 1) ? c[a] + n : 0;
      }
    } else if (c[a] >= n) {
      if (P->nbr[2 * a + 1] >= 0) {
        d = P->nbr[2 * a + 1];
        P = &tab[d];
        c[a] -= n;
      } else {
        c[a] = ((P->per >> a) & 1) ? c[a] - n : n - 1;
      }
    }
  }
  // A position at most one cell outside the block is now inside block d.
  // Lanes that lie beyond their level (their results are discarded) may
  // pass positions further out; clamping keeps their reads inside block d.
  x = min(max(c[0], 0), P->ni - 1);
  y = min(max(c[1], 0), P->nj - 1);
  z = min(max(c[2], 0), P->nk - 1);
  return d;
}

// value of any cell at padded position (x,y,z) in [-1, n] of level
// descriptor d, buffer `buf`, ghosts resolved to the cell they hold
template <class T>
__device__ __forceinline__ T level_value(const LevelDev *__restrict__ levs, int d, int buf, int x,
                                         int y, int z) {
  d = resolve_cell(levs, d, x, y, z);
  const LevelDev &L = levs[d];
  const T *a = (const T *)L.phi[buf][(x + y + z) & 1];
  return a[cidx(L.H, L.nj, x, y, z)];
}

// the same for the finest-level FP64 pressure of block b
__device__ __forceinline__ double fine_value(const FineDev *__restrict__ fine, int b, int x, int y,
                                             int z) {
  b = resolve_cell(fine, b, x, y, z);
  const FineDev &F = fine[b];
  return F.p[(x + y + z) & 1][cidx(F.H, F.nj, x, y, z)];
}

// ---------------------------------------------------------------------------
// One colour half-sweep of the red-black smoother (mgsolver.for:553-605):
//   phi = (rhs - (aw*W + ae*E + as*S + an*N + ab*B + at*T)) / ap
// colour 0 = red, 1 = black.  A sweep reads buffer `src` and writes `1-src`:
//   red:   interior neighbours (black) from black[src]
//   black: interior neighbours (red)   from red[1-src] (just written)
//   ghost neighbours from buffer src, resolved to their image (the
//   pre-sweep state the reference's ghosts hold until exchangepp at the end
//   of the sweep, mgsolver.for:614-615).
// zero != 0: the level holds zeros in buffer src (the first sweep after
// mgrestr zeroed phi, mgsolver.for:655-662, or pp = 0 at the finest level).
//
// Two tile kinds share a half-sweep (one launch, k_rb_sweep): tiles whose
// cells have all y/z neighbours inside the block, and the others; blocks with
// neighbours and levels one cell wide in x go cell by cell (k_cell_sweep).
//
// Work layout of the march kernels.  A lane owns two adjacent entries m0,
// m0+1 of one row of the colour arrays; L.lpr lanes cover a row segment and a
// wavefront holds 64/L.lpr rows (coarse levels pack several short rows into
// one wavefront).  Each lane walks the planes [t.z0, t.z1).  For a cell
// i = 2m + s of colour c (s = (c+j+k)&1) entry m of the other colour in the
// same row is its east (s = 0) or west (s = 1) neighbour and entry m of planes
// k-1, k+1 its bottom and top neighbours: that "own column" pair streams once
// through a register window; the remaining x-neighbour is the lane's other
// entry or the adjacent lane's (DPP wavefront shift); y-neighbours are loaded.
template <class T>
struct Vec2;
template <>
struct Vec2<float> {
  typedef float __attribute__((ext_vector_type(2))) type;
};
template <>
struct Vec2<double> {
  typedef double __attribute__((ext_vector_type(2))) type;
};

// Workgroups are dispatched round-robin over the 8 XCDs (blockIdx % 8);
// give each XCD a contiguous range of tiles so that neighbouring rows and
// planes are read through the same L2.
__device__ __forceinline__ int xcd_remap(int b, int n) {
  const int per = n >> 3, rem = n & 7;
  const int x = b & 7, q = b >> 3;
  return x * per + min(x, rem) + q;
}

// Division by ap: the FP64 path divides, as the reference does (bitwise
// parity); the FP32 path multiplies by the reciprocal (one rounding more,
// within the FP32 V-cycle's own error).
__device__ __forceinline__ double div_ap(double num, double ap, double /*inv_ap*/) {
  return num / ap;
}
__device__ __forceinline__ float div_ap(float num, float /*ap*/, float inv_ap) {
  return num * inv_ap;
}

// n / d, correctly rounded, by a divisor used many times: y = RN(1/d) once,
// then q = RN(n*y) and two corrections q + RN(n - q*d)*y with fused
// multiply-adds.  After the first q is within one ulp of n/d (each of RN(1/d)
// and RN(n*y) is off by half an ulp at most, and the remainder of a q that
// close is exact), and the second then rounds n/d correctly (P. Markstein,
// IBM J. Res. Dev. 34(1), 1990: y correctly rounded, q faithful).  Six
// operations, bitwise the quotient as written.  The remainders are exact only away from the ends of the
// exponent range: a quotient whose numerator lies there is divided as
// written, as is every quotient when the divisor does (fast = false).
struct Divisor {
  double d, y;
  bool fast;
};
__device__ __forceinline__ bool divisor_fast(double d) {
  return fabs(d) > 0x1p-300 && fabs(d) < 0x1p300;
}
__device__ __forceinline__ double div_by(double n, const Divisor &D) {
  // biased exponent of n in [500, 1546]: |n| in [2^-523, 2^524), or n zero
  const unsigned e = ((unsigned)(__double_as_longlong(n) >> 52)) & 0x7ffu;
  if (__builtin_expect(!D.fast || (e - 500u > 1046u && n != 0.0), 0)) return n / D.d;
  double q = n * D.y;
  q = __builtin_fma(__builtin_fma(-q, D.d, n), D.y, q);
  q = __builtin_fma(__builtin_fma(-q, D.d, n), D.y, q);
  return __builtin_amdgcn_div_fixup(q, D.d, n);  // the sign of a zero quotient
}

// DPP wavefront shifts by one lane (GFX9 wave_shr:1 = 0x138, wave_shl:1 =
// 0x130): lane l receives lane l-1's (shr) or l+1's (shl) value; the end lane
// receives 0.  Every lane of the wavefront must be active at the call.
__device__ __forceinline__ int dpp_i32(int v, int ctrl_shr) {
  return ctrl_shr ? __builtin_amdgcn_update_dpp(0, v, 0x138, 0xf, 0xf, false)
                  : __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, false);
}
__device__ __forceinline__ float wave_shift(float v, int shr) {
  return __int_as_float(dpp_i32(__float_as_int(v), shr));
}
__device__ __forceinline__ double wave_shift(double v, int shr) {
  const long long b = __double_as_longlong(v);
  const int lo = dpp_i32((int)(b & 0xffffffffll), shr);
  const int hi = dpp_i32((int)(b >> 32), shr);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// Global-address-space views of the level arrays (the descriptor holds
// generic pointers; loads through these compile to global_load with a
// scalar base and a 32-bit lane offset).
template <class T>
using gmem = __attribute__((address_space(1))) T;

// March tile of KB planes with every load issued up front (one memory round
// trip per tile): the own-column window (KB+2 planes), rows j-1 and j+1, the
// rhs and one x-slot entry per plane, then the KB updates, then the stores.
//
// The tile also updates the cells on its block's faces.  A ghost neighbour
// takes the pre-sweep (buffer src) value of its image -- the cell on the
// opposite face across a periodic face, the cell itself across a wall (whose
// coefficient is 0) -- which is the exchange/boundary state the reference's
// ghosts hold during a sweep.  Every array of a level lies in one arena
// allocation, so each load is the level's base (scalar) plus a 32-bit lane
// offset that may select any of the arrays: the image rows and entries of
// face lanes cost no branch.
//   x faces: lane 0 of a row segment (entry m0 = 0) holds cell 0, the lane
//     with m0 = H-2 holds cell ni-1; their x-slot loads the x-ghost image.
//   y/z faces (BND tiles only): rows 0 and nj-1 read their image rows;
//     chunks at plane 0 or nk-1 read the image plane into the window.
// The arithmetic of every cell is cell_coef's and the sum of mgsolver.for's
// relaxation.
//
// UPD (level 1's last black half-sweep): also p = p + (pp - 0) (k_update) of
// the lane's entries of both colours.  The new black values and, in the
// window, the red ones are at hand: k_update would read both again (256^3,
// half-sweep and k_update: FP64 41 + 59 us, now 81; float 19 + 50, now 60).
template <class T, int KB, bool ZERO_INT, bool BND, bool UPD>
__device__ __forceinline__ void march_tile_fast(const Tile &t, const LevelDev &L, int colour,
                                                int src, int zero, bool on, const FineDev *F) {
  typedef typename Vec2<T>::type v2;
  constexpr unsigned SZ = sizeof(T);
  const int lpr = L.lpr;
  const int lane = (int)threadIdx.x;
  const int rl = lane & (lpr - 1);
  const int m0 = t.x0 + 2 * rl;
  const int j = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  const bool col_ok = on && m0 < H && j < nj;  // on: the block's flag gates the stores
  const int jc = min(j, nj - 1);
  const unsigned row = (unsigned)H * SZ, plane = row * (unsigned)nj;  // bytes
  // byte offsets of the level's arrays from its arena base (phi[0][0])
  const char *base = (const char *)L.phi[0][0];
  auto aoff = [&](const void *a) -> unsigned { return (unsigned)((const char *)a - base); };
  const unsigned aO = aoff(colour == 0 ? L.phi[src][1] : L.phi[1 - src][0]);
  const unsigned aOs = aoff(L.phi[src][1 - colour]);  // other colour, pre-sweep
  const unsigned aPs = aoff(L.phi[src][colour]);      // own colour, pre-sweep
  const unsigned aR = aoff(L.rhs[colour]);
  const unsigned aD = aoff(L.phi[1 - src][colour]);
  const gmem<char> *Bs = (const gmem<char> *)base;
  gmem<char> *Bd = (gmem<char> *)base;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  const bool zg = zero != 0;  // ghosts read the all-zero pre-sweep state
  // the image of a ghost across a periodic face of extent n has the other
  // colour when n is even; a wall's image (the cell itself) has its own
  const unsigned aGX = (px && !(ni & 1)) ? aOs : aPs;
  const unsigned aGY = (py && !(nj & 1)) ? aOs : aPs;
  const unsigned aGZ = (pz && !(nk & 1)) ? aOs : aPs;
  const unsigned jrow = (unsigned)jc * row;
  const unsigned cell = jrow + (unsigned)min(m0, H - 2) * SZ;
  const int me = (ni - 1) >> 1;  // entry of cell ni-1; its pair starts at H-2
  const bool tile_left = t.x0 > 0, tile_right = t.x0 + 2 * lpr < H;

  // x slots: entry m0-1 for lane 0 of a row segment (neighbouring tile or the
  // west ghost image), entry m0+2 for the last lane (neighbouring tile) or
  // the east ghost image for the lane of cell ni-1; one load serves both
  // unless a lane has both roles (one-lane rows, a last tile of one pair)
  const bool role_r = tile_right ? rl == lpr - 1 : m0 == H - 2;
  const unsigned off_l =
      tile_left ? aO + cell - SZ : aGX + jrow + (unsigned)(px ? me : 0) * SZ;
  const unsigned off_r =
      tile_right ? aO + cell + 2 * SZ : aGX + jrow + (unsigned)(px ? 0 : me) * SZ;
  const bool dual = lpr == 1 || (tile_left && t.x0 == H - 2);
  const unsigned off_x = rl == 0 ? off_l : (role_r ? off_r : aO + cell);
  const unsigned off_x2 = role_r ? off_r : aO + cell;
  const bool gx_l = rl == 0 && !tile_left, gx_r = role_r && !tile_right;
  const bool zx_1 = zg && (rl == 0 ? gx_l : gx_r), zx_2 = zg && gx_r;

  // y rows: image rows on the y faces of BND tiles
  unsigned off_s = aO + cell - row, off_n = aO + cell + row;
  bool zs = false, zn = false;
  T as = (T)L.cy, an = (T)L.cy;
  if (BND) {
    if (jc == 0) {
      off_s = py ? aGY + cell + (unsigned)(nj - 1) * row : aPs + cell;
      zs = zg;
      if (!py) as = T(0);
    }
    if (jc == nj - 1) {
      off_n = py ? aGY + cell - (unsigned)(nj - 1) * row : aPs + cell;
      zn = zg;
      if (!py) an = T(0);
    }
  }
  const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
  const T ap_in = T(-1) * (cx + cx + cy + cy + cz + cz);
  const T inv_in = T(1) / ap_in;
  const T ap_x1 = T(-1) * (cx + cy + cy + cz + cz);  // one x coefficient 0 (wall face)
  const T inv_x1 = T(1) / ap_x1;
  const v2 vz = {T(0), T(0)};

  auto ld2 = [&](unsigned off) -> v2 { return *(const gmem<v2> *)(Bs + off); };
  auto ld1 = [&](unsigned off) -> T { return *(const gmem<T> *)(Bs + off); };

  {
    const int k0 = t.z0;
    const unsigned p0 = (unsigned)k0 * plane;
    v2 own[KB + 2], S2[KB], N2[KB], R2[KB];
    T x1[KB], x2[KB];
    if (!ZERO_INT) {
#pragma unroll
      for (int p = 0; p < KB + 2; ++p) {
        const int k = k0 - 1 + p;
        if (!BND || (k >= 0 && k < nk))
          own[p] = ld2(aO + cell + (unsigned)k * plane);
        else if (zg)
          own[p] = vz;
        else if (k < 0)
          own[p] = ld2((pz ? aGZ + (unsigned)(nk - 1) * plane : aPs) + cell);
        else
          own[p] = ld2((pz ? aGZ : aPs + (unsigned)(nk - 1) * plane) + cell);
      }
#pragma unroll
      for (int p = 0; p < KB; ++p) {
        const unsigned pp = p0 + (unsigned)p * plane;
        S2[p] = ld2(off_s + pp);
        N2[p] = ld2(off_n + pp);
        // x slots: read by the lanes at a row segment's ends only
        x1[p] = (rl == 0 || role_r) ? ld1(off_x + pp) : T(0);
        x2[p] = dual ? ld1(off_x2 + pp) : T(0);
      }
#pragma unroll
      for (int p = 0; p < KB; ++p) {
        if (BND && zs) S2[p] = vz;
        if (BND && zn) N2[p] = vz;
        if (zx_1) x1[p] = T(0);
        if (zx_2) x2[p] = T(0);
      }
    } else {
#pragma unroll
      for (int p = 0; p < KB + 2; ++p) own[p] = vz;
#pragma unroll
      for (int p = 0; p < KB; ++p) {
        S2[p] = N2[p] = vz;
        x1[p] = x2[p] = T(0);
      }
    }
#pragma unroll
    for (int p = 0; p < KB; ++p) R2[p] = ld2(aR + cell + p0 + (unsigned)p * plane);
    typedef typename Vec2<double>::type d2;
    d2 pr[UPD ? KB : 1], pb[UPD ? KB : 1];
    auto p_at = [&](int c, int p) {
      return (gmem<d2> *)((gmem<char> *)F->p[c] +
                          (cell + p0 + (unsigned)p * plane) * (unsigned)(sizeof(double) / SZ));
    };
    if constexpr (UPD) {
#pragma unroll
      for (int p = 0; p < KB; ++p) {
        pr[p] = *p_at(0, p);
        pb[p] = *p_at(1, p);
      }
    }
#pragma unroll
    for (int p = 0; p < KB; ++p) {
      const int k = k0 + p;
      const v2 o_m = own[p], o_c = own[p + 1], o_p = own[p + 2];
      T lf = wave_shift(o_c.y, 1);  // entry m0-1: lane-1's second entry
      T rt = wave_shift(o_c.x, 0);  // entry m0+2: lane+1's first entry
      const T gr = dual && rl == 0 ? x2[p] : x1[p];
      if (rl == 0) lf = x1[p];
      if (role_r) rt = gr;
      const int s = (colour + j + k) & 1;
      const int i0 = 2 * m0 + s, i1 = i0 + 2;
      const bool fw0 = m0 == 0 && s == 0;  // cell 0
      const bool fe0 = i0 == ni - 1, fe1 = i1 == ni - 1;
      const T W0 = s ? o_c.x : lf;
      const T E0 = fe0 ? gr : (s ? o_c.y : o_c.x);
      const T W1 = s ? o_c.y : o_c.x;
      const T E1 = fe1 ? gr : (s ? rt : o_c.y);
      const T aw0 = (!px && fw0) ? T(0) : cx;
      const T ae0 = (!px && fe0) ? T(0) : cx;
      const T ae1 = (!px && fe1) ? T(0) : cx;
      T ab = cz, at = cz;
      if (BND) {
        if (!pz && k == 0) ab = T(0);
        if (!pz && k == nk - 1) at = T(0);
      }
      const T sum0 = aw0 * W0 + ae0 * E0 + as * S2[p].x + an * N2[p].x + ab * o_m.x + at * o_p.x;
      const T sum1 = cx * W1 + ae1 * E1 + as * S2[p].y + an * N2[p].y + ab * o_m.y + at * o_p.y;
      if (BND) {
        const T ap0 = T(-1) * (aw0 + ae0 + as + an + ab + at);
        const T ap1 = T(-1) * (cx + ae1 + as + an + ab + at);
        R2[p].x = div_ap(R2[p].x - sum0, ap0, T(1) / ap0);
        R2[p].y = div_ap(R2[p].y - sum1, ap1, T(1) / ap1);
      } else {
        const bool x0f = !px && (fw0 || fe0), x1f = !px && fe1;
        R2[p].x = div_ap(R2[p].x - sum0, x0f ? ap_x1 : ap_in, x0f ? inv_x1 : inv_in);
        R2[p].y = div_ap(R2[p].y - sum1, x1f ? ap_x1 : ap_in, x1f ? inv_x1 : inv_in);
      }
    }
#pragma unroll
    for (int p = 0; p < KB; ++p) {
      const int s = (colour + j + k0 + p) & 1;
      const int i0 = 2 * m0 + s, i1 = i0 + 2;
      const bool w0 = col_ok && i0 < ni, w1 = col_ok && i1 < ni;
      gmem<char> *dq = Bd + aD + cell + p0 + (unsigned)p * plane;
      if (w0 && w1) {
        *(gmem<v2> *)dq = R2[p];
      } else {
        if (w0) *(gmem<T> *)dq = R2[p].x;
        if (w1) *(gmem<T> *)(dq + SZ) = R2[p].y;
      }
      if constexpr (UPD) {  // (pad entries included: they are never read as cells)
        if (col_ok) {
          pr[p].x = pr[p].x + ((double)own[p + 1].x - 0.0);
          pr[p].y = pr[p].y + ((double)own[p + 1].y - 0.0);
          pb[p].x = pb[p].x + ((double)R2[p].x - 0.0);
          pb[p].y = pb[p].y + ((double)R2[p].y - 0.0);
          *p_at(0, p) = pr[p];
          *p_at(1, p) = pb[p];
        }
      }
    }
  }
}

// Cell-parallel kernels for blocks with neighbours, blocks one cell wide in
// x, and the variable-density operator.  The value across each face of the
// block lies in the block itself (a wall, a periodic wrap) or in the
// neighbour; which arrays and how they are laid out is the same for the whole
// workgroup (scalar registers), so a cell selects each neighbour's address
// instead of branching and its loads are all in flight together: a kernel
// with a branch per ghost read them one memory latency after the other.
template <class T>
struct FaceSrc {
  const gmem<T> *p[6][2];  // face f, by the colour of the cell at the face
  unsigned wH, wx, eH, ex;  // x neighbours: row pitch and the cell's entry
  unsigned sn, sy, nn, ny;  // y neighbours: rows per plane and the row
  unsigned bz, tz;          // z neighbours: the plane
};

template <class T>
__device__ __forceinline__ FaceSrc<T> face_src(const LevelDev *__restrict__ levs,
                                               const LevelDev &L, int src) {
  FaceSrc<T> S;
  const int nl[3] = {L.ni, L.nj, L.nk};
  int at[6];
  const LevelDev *P[6];
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const int a = f >> 1;
    P[f] = L.nbr[f] >= 0 ? &levs[L.nbr[f]] : &L;
    const int np = a == 0 ? P[f]->ni : a == 1 ? P[f]->nj : P[f]->nk;
    const bool wall = wall_face(L, f), low = (f & 1) == 0;
    // a wall mirrors the cell itself; else the far cell of the block across
    at[f] = wall ? (low ? 0 : nl[a] - 1) : low ? np - 1 : 0;
    const int flip = wall ? 0 : ((low ? np : nl[a]) - 1) & 1;
    S.p[f][0] = (const gmem<T> *)P[f]->phi[src][flip];
    S.p[f][1] = (const gmem<T> *)P[f]->phi[src][1 - flip];
  }
  S.wH = (unsigned)P[0]->H;
  S.wx = (unsigned)at[0] >> 1;
  S.eH = (unsigned)P[1]->H;
  S.ex = (unsigned)at[1] >> 1;
  S.sn = (unsigned)P[2]->nj;
  S.sy = (unsigned)at[2];
  S.nn = (unsigned)P[3]->nj;
  S.ny = (unsigned)at[3];
  S.bz = (unsigned)at[4];
  S.tz = (unsigned)at[5];
  return S;
}

// The six neighbours of cell (i, j, k) of colour c: O the other colour's
// array inside the block; zg: ghosts hold zero.  e: the cell's entry.
template <class T>
__device__ __forceinline__ void cell_neighbours(const FaceSrc<T> &S, const LevelDev &L,
                                                const gmem<T> *O, int c, int i, int j, int k,
                                                unsigned e, bool zg, T (&v)[6]) {
  const int s = i & 1;
  const unsigned H = (unsigned)L.H, nj = (unsigned)L.nj, plane = H * nj, m = (unsigned)i >> 1;
  const unsigned uj = (unsigned)j, uk = (unsigned)k;
  const bool g[6] = {i == 0, i >= L.ni - 1, j == 0, j == L.nj - 1, k == 0, k == L.nk - 1};
  const unsigned in[6] = {s ? e : e - 1, s ? e + 1 : e, e - H, e + H, e - plane, e + plane};
  const unsigned gh[6] = {(uk * nj + uj) * S.wH + S.wx,    (uk * nj + uj) * S.eH + S.ex,
                          (uk * S.sn + S.sy) * H + m,      (uk * S.nn + S.ny) * H + m,
                          (S.bz * nj + uj) * H + m,        (S.tz * nj + uj) * H + m};
#pragma unroll
  for (int f = 0; f < 6; ++f) {
    const gmem<T> *const b = g[f] ? (c ? S.p[f][1] : S.p[f][0]) : O;
    v[f] = b[g[f] ? gh[f] : in[f]];
  }
#pragma unroll
  for (int f = 0; f < 6; ++f)
    if (zg && g[f]) v[f] = T(0);
}

// the coefficients of entry e of colour c: aw, ae, as, an, ab, at, ap
template <class T, bool LSM>
__device__ __forceinline__ void cell_coefs(const LevelDev &L, int c, int i, int j, int k,
                                           unsigned e, T (&a)[7]) {
  if constexpr (LSM) {
#pragma unroll
    for (int q = 0; q < 7; ++q)
      a[q] = ((const gmem<double> *)L.lsm)[(size_t)(2 * q + c) * L.lsm_half + e];
  } else {
    const Coef<T> C = cell_coef<T>(L, i, j, k);
    a[0] = C.aw, a[1] = C.ae, a[2] = C.as, a[3] = C.an, a[4] = C.ab, a[5] = C.at, a[6] = C.ap;
  }
}

// One colour half-sweep (mgsolver.for:553-605; LSM: with per-cell
// coefficients) over natural tiles (TILE_X x TILE_Y cells of one plane): 128
// threads, one per cell of the colour.  The buffer rules are k_rb_sweep's.
// Bound by the launch and one round of loads.  Averages over four levels, us,
// with a branch per ghost | now: 64 joined blocks of 64x8x64, 18.3 | 5.9
// (restriction 74 | 11, prolongation 33 | 12); 96x64x80 with variable density
// 6.1 | 3.9 (restriction 70 | 6.3).
template <class T, bool LSM>
__global__ void __launch_bounds__(128)
    k_cell_sweep(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                 const int *__restrict__ active, int colour, int src, int zero, int ntiles) {
  const Tile t = tiles[xcd_remap((int)blockIdx.x, ntiles)];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const FaceSrc<T> S = face_src<T>(levs, L, src);
  const int q = (int)threadIdx.x + TILE_X * (int)threadIdx.y;
  const int jt = t.y0 + q / (TILE_X / 2), k = t.z0;
  const int mt = (t.x0 >> 1) + q % (TILE_X / 2);
  // lanes beyond the level read a valid cell and store nothing
  const int j = min(jt, L.nj - 1), m = min(mt, (L.ni - 1) >> 1);
  const int i = 2 * m + ((colour + j + k) & 1);
  const unsigned e = (unsigned)cidx(L.H, L.nj, i, j, k);
  T v[6], a[7];
  const T r = ((const gmem<T> *)L.rhs[colour])[e];
  cell_coefs<T, LSM>(L, colour, i, j, k, e, a);
  if (zero && colour == 0) {  // every neighbour is zero
#pragma unroll
    for (int f = 0; f < 6; ++f) v[f] = T(0);
  } else {
    cell_neighbours<T>(S, L,
                       (const gmem<T> *)(colour == 0 ? L.phi[src][1] : L.phi[1 - src][0]), colour,
                       i, j, k, e, zero != 0, v);
  }
  const T sum =
      a[0] * v[0] + a[1] * v[1] + a[2] * v[2] + a[3] * v[3] + a[4] * v[4] + a[5] * v[5];
  if (jt < L.nj && mt == m && i < L.ni)
    ((gmem<T> *)L.phi[1 - src][colour])[e] = div_ap(r - sum, a[6], T(1) / a[6]);
}

// Restriction (mgrestr, mgsolver.for:693-756) over natural tiles of the coarse
// level: grid.y is the tile's row; wavefront y of a workgroup forms, for 64
// coarse cells, the two fine residuals r = f - (aw*W + ae*E + as*S + an*N +
// ab*B + at*T + ap*P) of row y & 1, plane y >> 1 of the children, and
// wavefront 0 sums the eight i fastest, then j, then k, times 0.125.  (A
// thread per coarse cell walked its children one after the other, and a level
// had too few threads.)
template <class Tf, class Tc, bool LSM>
__global__ void __launch_bounds__(NTHREADS)
    k_cell_restrict(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                    const int *__restrict__ active, int src_f, int ntiles) {
  __shared__ Tf res[8][TILE_X];
  const Tile t = tiles[xcd_remap((int)blockIdx.x, ntiles)];
  const LevelDev &C = levs[t.lev];
  const int jc = t.y0 + (int)blockIdx.y, kc = t.z0;
  if (!active[C.blk] || jc >= C.nj) return;
  const LevelDev &F = levs[C.finer];
  const FaceSrc<Tf> S = face_src<Tf>(levs, F, src_f);
  const int lane = (int)threadIdx.x, ch = (int)threadIdx.y;
  const int lt = t.x0 + lane, l = min(lt, C.ni - 1);
  const int j = 2 * jc + (ch & 1), k = 2 * kc + (ch >> 1);
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    const int i = 2 * l + d, c = (i + j + k) & 1;
    const unsigned e = (unsigned)cidx(F.H, F.nj, i, j, k);
    Tf v[6], a[7];
    const Tf f = ((const gmem<Tf> *)F.rhs[c])[e];
    const Tf P = ((const gmem<Tf> *)F.phi[src_f][c])[e];
    cell_coefs<Tf, LSM>(F, c, i, j, k, e, a);
    cell_neighbours<Tf>(S, F, (const gmem<Tf> *)F.phi[src_f][1 - c], c, i, j, k, e, false, v);
    res[2 * ch + d][lane] = f - (a[0] * v[0] + a[1] * v[1] + a[2] * v[2] + a[3] * v[3] +
                                 a[4] * v[4] + a[5] * v[5] + a[6] * P);
  }
  __syncthreads();
  if (ch != 0 || lt >= C.ni) return;
  Tc acc = (Tc)res[0][lane];
#pragma unroll
  for (int q = 1; q < 8; ++q) acc = acc + (Tc)res[q][lane];
  ((gmem<Tc> *)C.rhs[(l + jc + kc) & 1])[cidx(C.H, C.nj, l, jc, kc)] = Tc(0.125) * acc;
}

// One launch per colour half-sweep over a level.  Every tile of the list is
// KB planes deep: kind 0 has every y/z neighbour inside the block, kind 3
// touches a y/z face; the tiles write disjoint cells.  One instantiation per depth keeps each one's register
// count to what its own tiles need.
template <class T, int KB, bool UPD>
__device__ __forceinline__ void rb_dispatch(const Tile &t, const LevelDev &L, int colour, int src,
                                            int zero, bool on, const FineDev *F);

// In the one-descriptor kernels, one empty asm statement takes the tile,
// the block's flag and every descriptor field the kernel reads: all of them
// are loaded before it, together (scalar loads complete out of order, so any
// earlier use would wait for every load issued before it).

// Kernel arguments are scalars only (no aggregate) and the grid size is
// passed in: every argument then arrives preloaded in SGPRs instead of being
// read from the argument buffer.
// ONE: every tile of the launch has descriptor one_lev of block one_blk.  The
// tile, the descriptor and the block's flag are then read together, and the
// flag masks the stores instead of ending inactive workgroups early, so that
// the data loads wait for none of them but the tile and the descriptor
// (small levels are bound by this chain of latencies).
template <class T, int KB, bool ONE, bool UPD>
__global__ void __launch_bounds__(NTHREADS)
    k_rb_sweep(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
               const int *__restrict__ active, int colour, int src, int zero, int one_lev,
               int one_blk, int ntiles, const FineDev *__restrict__ fine) {
  const Tile t = tiles[xcd_remap((int)blockIdx.x, ntiles)];
  if (ONE) {
    const LevelDev &L = levs[one_lev];
    const int on = active[one_blk];
    asm volatile("" ::"s"(t.x0), "s"(t.y0), "s"(t.z0), "s"(t.kind), "s"(on), "s"(L.ni), "s"(L.nj),
                 "s"(L.nk), "s"(L.H), "s"(L.per), "s"(L.lpr), "s"(L.cx), "s"(L.cy), "s"(L.cz),
                 "s"(L.phi[0][0]), "s"(L.phi[0][1]), "s"(L.phi[1][0]), "s"(L.phi[1][1]),
                 "s"(L.rhs[0]), "s"(L.rhs[1]));
    rb_dispatch<T, KB, UPD>(t, L, colour, src, zero, on != 0, UPD ? fine + one_blk : nullptr);
  } else {
    const LevelDev &L = levs[t.lev];
    if (!active[L.blk]) return;
    rb_dispatch<T, KB, UPD>(t, L, colour, src, zero, true, UPD ? fine + L.blk : nullptr);
  }
}

template <class T, int KB, bool UPD>
__device__ __forceinline__ void rb_dispatch(const Tile &t, const LevelDev &L, int colour, int src,
                                            int zero, bool on, const FineDev *F) {
  if constexpr (UPD) {
    if (t.kind == 0)
      march_tile_fast<T, KB, false, false, true>(t, L, 1, src, zero, on, F);
    else
      march_tile_fast<T, KB, false, true, true>(t, L, 1, src, zero, on, F);
    return;
  }
  // the interior neighbours are zeros in the red half of a zero-state sweep
  const bool zint = zero && colour == 0;
  if (t.kind == 0) {
    zint ? march_tile_fast<T, KB, true, false, false>(t, L, colour, src, zero, on, F)
         : march_tile_fast<T, KB, false, false, false>(t, L, colour, src, zero, on, F);
  } else {
    zint ? march_tile_fast<T, KB, true, true, false>(t, L, colour, src, zero, on, F)
         : march_tile_fast<T, KB, false, true, false>(t, L, colour, src, zero, on, F);
  }
}

// ---------------------------------------------------------------------------
// Two whole sweeps of a mid-size level of one block in one launch.  There a
// half-sweep is bound by its launch and one round of memory latency, not by
// its cells: a workgroup takes the 16^3 cells around a tile of 8^3
// into LDS and runs the four half-sweeps there, each on one layer of cells
// less, the cells around the tile being computed again by their own tiles.
// Bound by the latencies inside (a half-sweep, its barrier) and by instruction
// issue: 16 wavefronts of two entries a thread took 37 us a cycle for one level
// of 32^3 (FP64, V(2,2)), 8 wavefronts of four 39, half-sweep launches 49.
//
// Positions around the tile continue across a periodic face (an even number
// of cells: the colours continue, too).  A black cell reads across such a
// face the red value from before the sweep (`old`), as the ghosts hold it;
// across a wall the product of a zero coefficient and a zero, as the cells
// beyond are never set, where the other kernels multiply zero by the cell's own
// value before the sweep: NaN where that is not finite.  A tile that has loaded
// values beyond the middle of the exponent range (smaller ones stay finite over
// two sweeps) runs again that way: as the only way it took 9% of a 48^3 cycle
// (FP64), one path with a flag 4%, a second copy of the sweeps none (FP32, bound
// by its registers: 2% at 104x56x40).  The result goes to the other buffer, once:
// the launch is one step of the level's buffers.  zero != 0: the level holds
// zeros.
constexpr int RBT = 16, RBT_HALF = RBT * RBT * RBT / 2, RBT_THREADS = 1024;
template <class T>
__global__ void __launch_bounds__(RBT_THREADS, sizeof(T) == 4 ? 8 : 4)
    k_rb_tile(const LevelDev *__restrict__ levs, const int *__restrict__ active, int src, int zero,
              int one_lev, int one_blk, int tx, int ty, int ntiles,
              const FineDev *__restrict__ fine) {
  constexpr int HALO = 4, TS = RBT - 2 * HALO, U = RBT_HALF / RBT_THREADS;
  __shared__ T black[RBT_HALF], red[RBT_HALF], old[RBT_HALF];
  __shared__ int large;  // a thread has loaded such values
  const LevelDev &L = levs[one_lev];
  const int on = active[one_blk];
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  const int b = xcd_remap((int)blockIdx.x, ntiles);
  const int bz = b / (tx * ty), by = (b - bz * tx * ty) / tx, bx = b - (bz * ty + by) * tx;
  const int x0 = bx * TS - HALO, y0 = by * TS - HALO, z0 = bz * TS - HALO;
  // whether a periodic face cuts the positions
  const bool cross = (px && (x0 < 0 || x0 + RBT > ni)) || (py && (y0 < 0 || y0 + RBT > nj)) ||
                     (pz && (z0 < 0 || z0 + RBT > nk));
  const unsigned walls = (px ? 0u : 3u) | (py ? 0u : 12u) | (pz ? 0u : 48u);
  const gmem<T> *P[2] = {(const gmem<T> *)L.phi[src][0], (const gmem<T> *)L.phi[src][1]};
  const gmem<T> *R[2] = {(const gmem<T> *)L.rhs[0], (const gmem<T> *)L.rhs[1]};
  gmem<T> *D[2] = {(gmem<T> *)L.phi[1 - src][0], (gmem<T> *)L.phi[1 - src][1]};
  const int tid = (int)threadIdx.x, m = tid & 7, ry = (tid >> 3) & 15;
  auto wrap = [](int x, int n, bool per) { return !per ? x : x < 0 ? x + n : x >= n ? x - n : x; };
  const int y = y0 + ry, yw = wrap(y, nj, py);
  const bool oky = (unsigned)yw < (unsigned)nj;

  // a thread's entries: plane rz = tid/128 + 4u of both colours; bits 0..5 of
  // `face`: the cell lies on that face of the block, 6: it exists
  unsigned face[U][2], ent[U][2];
  T r[U][2], v1[U], v0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int rz = (tid >> 7) + RBT_THREADS / 128 * u, z = z0 + rz, zw = wrap(z, nk, pz);
    const bool okz = (unsigned)zw < (unsigned)nk;
    const unsigned fyz = (yw == 0 ? 4u : 0u) | (yw == nj - 1 ? 8u : 0u) | (zw == 0 ? 16u : 0u) |
                         (zw == nk - 1 ? 32u : 0u);
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int x = x0 + 2 * m + ((c + y + z) & 1), xw = wrap(x, ni, px);
      const bool ok = oky && okz && (unsigned)xw < (unsigned)ni;
      face[u][c] = fyz | (xw == 0 ? 1u : 0u) | (xw == ni - 1 ? 2u : 0u) | (ok ? 64u : 0u);
      // positions that do not exist read entry 0
      const unsigned e =
          ok ? ((unsigned)zw * (unsigned)nj + (unsigned)yw) * (unsigned)H + ((unsigned)xw >> 1)
             : 0u;
      ent[u][c] = e;
      r[u][c] = R[c][e];
    }
    v1[u] = zero ? T(0) : P[1][ent[u][1]];
    v0[u] = zero || !cross ? T(0) : P[0][ent[u][0]];
  }
  T most = T(0);
#pragma unroll
  for (int u = 0; u < U; ++u)
    most = most + fabs(r[u][0]) + fabs(r[u][1]) + fabs(v1[u]) + fabs(v0[u]);
  const bool big = !(most < (sizeof(T) == 4 ? T(0x1p64) : T(0x1p500)));
  auto fill = [&]() {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int q = tid + u * RBT_THREADS;
      black[q] = face[u][1] & 64u ? v1[u] : T(0);
      red[q] = face[u][0] & 64u ? v0[u] : T(0);
      if (cross) old[q] = T(0);
    }
    if (tid == 0) large = 0;
    __syncthreads();
  };
  fill();
  if (__builtin_expect(big, 0)) large = 1;
  const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
  // the update of entry q of colour c from the six values
  auto update = [&](unsigned f, T rhs, const T(&v)[6]) -> T {
    // FP32: the coefficients are formed each time, kept over the sweeps they
    // take the registers of a second workgroup on the CU (64^3: 107 | 102 us a
    // cycle); FP64 is bound by its arithmetic and keeps them (32^3: 79 | 81)
    if (sizeof(T) == 4) asm volatile("" : "+v"(f));
    const T aw = (!px && (f & 1u)) ? T(0) : cx, ae = (!px && (f & 2u)) ? T(0) : cx;
    const T as = (!py && (f & 4u)) ? T(0) : cy, an = (!py && (f & 8u)) ? T(0) : cy;
    const T ab = (!pz && (f & 16u)) ? T(0) : cz, at = (!pz && (f & 32u)) ? T(0) : cz;
    const T ap = T(-1) * (aw + ae + as + an + ab + at);
    const T sum = aw * v[0] + ae * v[1] + as * v[2] + an * v[3] + ab * v[4] + at * v[5];
    return div_ap(rhs - sum, ap, T(1) / ap);
  };
  auto at_walls = [&](unsigned f, T own, T(&v)[6]) {
#pragma unroll
    for (int q = 0; q < 6; ++q)
      if ((f & walls) >> q & 1u) v[q] = own;
  };
  // whether half-sweep h computes the entry: one layer less each
  auto in = [&](int c, int rz, int h) {
    const int rx = 2 * m + ((c + y0 + ry + z0 + rz) & 1), lo = h + 1, hi = RBT - 2 - h;
    return rx >= lo && rx <= hi && ry >= lo && ry <= hi && rz >= lo && rz <= hi;
  };
  auto sweeps = [&](auto own) __attribute__((always_inline)) {
    constexpr bool OWN = decltype(own)::value;
#pragma unroll 1
    for (int h = 0; h < HALO; h += 2) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = tid + u * RBT_THREADS, rz = (tid >> 7) + RBT_THREADS / 128 * u;
        if (!in(0, rz, h) || !(face[u][0] & 64u)) continue;
        const int s = (y0 + ry + z0 + rz) & 1;
        T v[6] = {black[q - 1 + s],       black[q + s],
                  black[q - RBT / 2],     black[q + RBT / 2],
                  black[q - RBT * RBT / 2], black[q + RBT * RBT / 2]};
        if constexpr (OWN) at_walls(face[u][0], red[q], v);
        const T x = update(face[u][0], r[u][0], v);
        if (cross) old[q] = red[q];
        red[q] = x;
      }
      __syncthreads();
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int q = tid + u * RBT_THREADS, rz = (tid >> 7) + RBT_THREADS / 128 * u;
        if (!in(1, rz, h + 1) || !(face[u][1] & 64u)) continue;
        const int s = (1 + y0 + ry + z0 + rz) & 1;
        const int at[6] = {q - 1 + s,   q + s, q - RBT / 2, q + RBT / 2, q - RBT * RBT / 2,
                           q + RBT * RBT / 2};
        T v[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) v[f] = red[at[f]];
        if (cross) {
#pragma unroll
          for (int f = 0; f < 6; ++f) {
            const T w = old[at[f]];
            if ((face[u][1] >> f) & 1u) v[f] = w;  // (at a wall its coefficient is 0)
          }
        }
        if constexpr (OWN) at_walls(face[u][1], black[q], v);
        black[q] = update(face[u][1], r[u][1], v);
      }
      __syncthreads();
    }
  };
  sweeps(std::false_type());
  if (__builtin_expect(large, 0)) {
    __syncthreads();  // every wavefront has read `large`
    for (int u = 0; u < U; ++u) {
      v1[u] = zero ? T(0) : P[1][ent[u][1]];
      v0[u] = zero ? T(0) : P[0][ent[u][0]];
    }
    fill();
    sweeps(std::true_type());
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int q = tid + u * RBT_THREADS, rz = (tid >> 7) + RBT_THREADS / 128 * u;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int x = x0 + 2 * m + ((c + y + z0 + rz) & 1);
      if (in(c, rz, HALO - 1) && x < ni && y < nj && z0 + rz < nk && on) {
        const T pp = c ? black[q] : red[q];
        D[c][ent[u][c]] = pp;
        if (fine) {  // level 1's last sweeps: also p = p + (pp - 0), as k_update
          gmem<double> *const p = (gmem<double> *)fine[one_blk].p[c] + ent[u][c];
          *p = *p + ((double)pp - 0.0);
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Fused red-black sweep for small levels: both colour halves of one sweep
// in one launch (the split sweep costs two launches, and small levels are
// bound by launch and memory latency, not by bandwidth).  A tile is FX x FY
// x FZ cells at (x0, y0, z0) in cell coordinates.
//   Phase 1: the new red value of every red cell of the block inside the
//   tile grown by one cell on each side (the tile's own red cells and the
//   halo its black cells need), into LDS; the tile's own red cells also go
//   to buffer 1-src.  A red cell reads black neighbours from buffer src and
//   ghosts as images in buffer src, as the split red half-sweep does.
//   Phase 2: the tile's black cells from the red values in LDS (neighbours
//   inside the block) and ghost images in buffer src (pre-sweep, as the
//   split black half-sweep reads them), into buffer 1-src.
// Halo red cells are also computed by the neighbouring tiles with the same
// arithmetic, so every red value a black cell uses is bitwise the one the
// split sweep stores.  zero != 0: the level holds zeros in buffer src.
constexpr int FX = FUSED_X, FY = FUSED_Y, FZ = FUSED_Z;
constexpr int FEX = FX + 2, FEY = FY + 2, FEZ = FZ + 2;
constexpr int F_RED = FEX / 2 * FEY * FEZ;   // red positions of the grown tile
constexpr int F_BLACK = FX / 2 * FY * FZ;    // black cells of the tile
constexpr int F_RED_PER = (F_RED + NTHREADS - 1) / NTHREADS;
constexpr int F_BLACK_PER = F_BLACK / NTHREADS;

template <class T>
__global__ void __launch_bounds__(NTHREADS)
    k_rb_fused(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
               const int *__restrict__ active, int src, int zero) {
  const Tile t = tiles[xcd_remap((int)blockIdx.x, (int)gridDim.x)];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  __shared__ T red[FEZ * FEY * FEX];
  const int tid = (int)(threadIdx.x + blockDim.x * threadIdx.y);
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  // Addresses are 32-bit byte offsets from the level's first array (all six
  // arrays of a level lie in one arena allocation), through a global-
  // address-space base: a generic pointer's loads would also count against
  // the LDS wait counter.
  constexpr unsigned SZ = sizeof(T);
  const char *base = (const char *)L.phi[0][0];
  auto aoff = [&](const void *a) -> unsigned { return (unsigned)((const char *)a - base); };
  const unsigned aP0 = aoff(L.phi[src][0]), dP = aoff(L.phi[src][1]) - aP0;  // pre-sweep
  const unsigned aR0 = aoff(L.rhs[0]), aR1 = aoff(L.rhs[1]);
  const unsigned aD0 = aoff(L.phi[1 - src][0]), aD1 = aoff(L.phi[1 - src][1]);
  const gmem<char> *Bs = (const gmem<char> *)base;
  gmem<char> *Bd = (gmem<char> *)base;
  const unsigned row = (unsigned)H * SZ, plane = row * (unsigned)nj;
  auto inside = [&](int x, int y, int z) {
    return (unsigned)x < (unsigned)ni && (unsigned)y < (unsigned)nj && (unsigned)z < (unsigned)nk;
  };
  // byte offset of cell (x, y, z) inside its colour array
  auto at = [&](int x, int y, int z) -> unsigned {
    return (unsigned)z * plane + (unsigned)y * row + (unsigned)(x >> 1) * SZ;
  };
  // pre-sweep value of the image of (x, y, z) (the cell itself inside the
  // block; positions up to two cells outside map into the block)
  auto pre = [&](int x, int y, int z) -> T {
    return *(const gmem<T> *)(Bs + aP0 + (unsigned)((x + y + z) & 1) * dP + at(x, y, z));
  };
  auto prex = [&](int x, int y, int z) { return pre(image(x, ni, px), y, z); };
  auto prey = [&](int x, int y, int z) { return pre(x, image(y, nj, py), z); };
  auto prez = [&](int x, int y, int z) { return pre(x, y, image(z, nk, pz)); };
  const bool zl = zero != 0;  // pre-sweep state all zero

  // Every global load first.  Black cells of the tile: rhs and the images
  // of their six neighbours (used where a neighbour is a ghost).
  int bi[F_BLACK_PER], bj[F_BLACK_PER], bk[F_BLACK_PER];
  T brhs[F_BLACK_PER], bg[F_BLACK_PER][6];
#pragma unroll
  for (int q = 0; q < F_BLACK_PER; ++q) {
    const int b = tid + q * NTHREADS;
    const int row = b / (FX / 2), m = b % (FX / 2);
    const int j = t.y0 + row % FY, k = t.z0 + row / FY;
    const int i = t.x0 + (((t.x0 + j + k) & 1) ^ 1) + 2 * m;
    bi[q] = i;
    bj[q] = j;
    bk[q] = k;
    // clamped into the block: cells of a clipped tile load a valid entry
    const int ic = min(i, ni - 1), jc = min(j, nj - 1), kc = min(k, nk - 1);
    brhs[q] = *(const gmem<T> *)(Bs + aR1 + at(ic, jc, kc));
    bg[q][0] = prex(ic - 1, jc, kc);
    bg[q][1] = prex(ic + 1, jc, kc);
    bg[q][2] = prey(ic, jc - 1, kc);
    bg[q][3] = prey(ic, jc + 1, kc);
    bg[q][4] = prez(ic, jc, kc - 1);
    bg[q][5] = prez(ic, jc, kc + 1);
  }
  // red cells of the grown tile: rhs and six (black) neighbours, all
  // pre-sweep images
  int ri[F_RED_PER], rj[F_RED_PER], rk[F_RED_PER], re[F_RED_PER];
  T rrhs[F_RED_PER], rn[F_RED_PER][6];
#pragma unroll
  for (int q = 0; q < F_RED_PER; ++q) {
    const int r = min(tid + q * NTHREADS, F_RED - 1);
    const int row = r / (FEX / 2), m = r % (FEX / 2);
    const int ey = row % FEY, ez = row / FEY;
    const int j = t.y0 - 1 + ey, k = t.z0 - 1 + ez;
    const int ex = ((t.x0 - 1 + j + k) & 1) + 2 * m;  // (i + j + k) even
    const int i = t.x0 - 1 + ex;
    ri[q] = i;
    rj[q] = j;
    rk[q] = k;
    re[q] = (ez * FEY + ey) * FEX + ex;
    // positions of the grown tile outside the block load their image (unused)
    const int ic = image(i, ni, px), jc = image(j, nj, py), kc = image(k, nk, pz);
    rrhs[q] = *(const gmem<T> *)(Bs + aR0 + at(ic, jc, kc));
    rn[q][0] = prex(ic - 1, jc, kc);
    rn[q][1] = prex(ic + 1, jc, kc);
    rn[q][2] = prey(ic, jc - 1, kc);
    rn[q][3] = prey(ic, jc + 1, kc);
    rn[q][4] = prez(ic, jc, kc - 1);
    rn[q][5] = prez(ic, jc, kc + 1);
  }

  // phase 1: red cells of the grown tile that lie in the block, into LDS
  // (the tile's own red cells go to global memory after phase 2, so that
  // the barrier waits for LDS only)
  T rval[F_RED_PER];
#pragma unroll
  for (int q = 0; q < F_RED_PER; ++q) {
    const int i = ri[q], j = rj[q], k = rk[q];
    rval[q] = T(0);
    if (tid + q * NTHREADS >= F_RED || !inside(i, j, k)) continue;
    const Coef<T> c = cell_coef<T>(L, i, j, k);
    T v[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) v[d] = zl ? T(0) : rn[q][d];
    const T sum = c.aw * v[0] + c.ae * v[1] + c.as * v[2] + c.an * v[3] + c.ab * v[4] +
                  c.at * v[5];
    rval[q] = div_ap(rrhs[q] - sum, c.ap, T(1) / c.ap);
    red[re[q]] = rval[q];
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes done
  __builtin_amdgcn_s_barrier();

  // phase 2: the tile's black cells; neighbours in the block from LDS, ghost
  // neighbours their pre-sweep images
#pragma unroll
  for (int q = 0; q < F_BLACK_PER; ++q) {
    const int i = bi[q], j = bj[q], k = bk[q];
    if (!inside(i, j, k)) continue;
    const int di[6] = {-1, 1, 0, 0, 0, 0}, dj[6] = {0, 0, -1, 1, 0, 0}, dk[6] = {0, 0, 0, 0, -1, 1};
    T v[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      const int x = i + di[d], y = j + dj[d], z = k + dk[d];
      v[d] = inside(x, y, z) ? red[((z - t.z0 + 1) * FEY + (y - t.y0 + 1)) * FEX + (x - t.x0 + 1)]
                             : (zl ? T(0) : bg[q][d]);
    }
    const Coef<T> c = cell_coef<T>(L, i, j, k);
    const T sum = c.aw * v[0] + c.ae * v[1] + c.as * v[2] + c.an * v[3] + c.ab * v[4] +
                  c.at * v[5];
    *(gmem<T> *)(Bd + aD1 + at(i, j, k)) = div_ap(brhs[q] - sum, c.ap, T(1) / c.ap);
  }
#pragma unroll
  for (int q = 0; q < F_RED_PER; ++q) {
    const int i = ri[q], j = rj[q], k = rk[q];
    if (tid + q * NTHREADS < F_RED && i >= t.x0 && i < t.x0 + FX && i < ni && j >= t.y0 &&
        j < t.y0 + FY && j < nj && k >= t.z0 && k < t.z0 + FZ && k < nk)
      *(gmem<T> *)(Bd + aD0 + at(i, j, k)) = rval[q];
  }
}

// ---------------------------------------------------------------------------
// mgrestr (mgsolver.for:693-756): fine residual
//   resf = rhs - (aw*W + ae*E + as*S + an*N + ab*B + at*T + ap*P)
// and coarse rhs = 0.125 * (sum of the 8 children, i fastest, then j, k).
// The coarse phi is not touched: the next relax of the coarse level runs with
// zero = 1, which is the zeroing of mgsolver.for:655-662.
//
// The first half-sweep of a relaxation from zero, for a red coarse cell: every
// neighbour is zero, so the sweep's sum is exactly zero and the cell becomes
// div_ap(rhs - 0, ap, 1/ap) with cell_coef's ap, which the restriction writes
// with the rhs (zbuf >= 0: into buffer zbuf), in the sweep's arithmetic.
template <class Tc>
__device__ __forceinline__ void zero_state_red(const LevelDev &C, int zbuf, int ic, int jc, int kc,
                                               unsigned q, Tc rhs) {
  if (zbuf < 0 || ((ic + jc + kc) & 1)) return;
  const Coef<Tc> c = cell_coef<Tc>(C, ic, jc, kc);
  ((gmem<Tc> *)C.phi[zbuf][0])[q] = div_ap(rhs - Tc(0), c.ap, Tc(1) / c.ap);
}

// Restriction tile of an FP64 fine level, KBC coarse planes (2*KBC fine
// planes): a rolling window
// of fine planes k-1, k, k+1 of rows 2jc and 2jc+1.  A lane holds two coarse
// cells l, l+1 of a coarse row: fine entries l, l+1 of both colours (cells
// 2l .. 2l+3), each array one vector load.  Neighbours are addressed by the
// coordinates of their image as 32-bit byte offsets from the fine level's
// arena base, so tiles touching a y/z face (BND) run the same code; their
// coefficients carry cell_coef's zeros towards walls.  Each coarse cell's
// eight residuals arrive in the reference's summation order (a, b of row
// 2jc, a, b of row 2jc+1; plane 2kc, then 2kc+1).  C.lpr1 lanes cover a
// coarse row segment; the tile's `lev` is the coarse descriptor.
template <class Tf, class Tc, int KBC, bool BND>
__device__ __forceinline__ void restrict_tile_two(const Tile &t, const LevelDev &C,
                                                  const LevelDev &F, int src_f, bool on,
                                                  int zbuf) {
  typedef typename Vec2<Tf>::type v2;
  constexpr unsigned SZ = sizeof(Tf);
  constexpr int NF = 2 * KBC;
  const int lpr = C.lpr1;
  const int lane = (int)threadIdx.x;
  const int rl = lane & (lpr - 1);
  const int l = t.x0 + 2 * rl;  // coarse cells l, l+1 = fine entries l, l+1
  const int jc = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = F.ni, nj = F.nj, nk = F.nk, H = F.H;
  // on: the block's flag gates the stores
  const bool ok0 = on && l < C.ni && jc < C.nj, ok1 = on && l + 1 < C.ni && jc < C.nj;
  const bool px = F.per & 1, py = F.per & 2, pz = F.per & 4;
  const unsigned row = (unsigned)H * SZ, plane = row * (unsigned)nj;  // bytes
  const int j0 = 2 * min(jc, C.nj - 1);  // even: a has colour (r + k) & 1 in row j0 + r
  // lanes past the row's last pair read that pair (nothing of theirs is stored)
  const unsigned ent = (unsigned)min(l, H - 2) * SZ;
  const char *base = (const char *)F.phi[0][0];
  auto aoff = [&](const void *a) -> unsigned { return (unsigned)((const char *)a - base); };
  const unsigned aP0 = aoff(F.phi[src_f][0]), dP = aoff(F.phi[src_f][1]) - aP0;
  const unsigned aR0 = aoff(F.rhs[0]), dR = aoff(F.rhs[1]) - aR0;
  const gmem<char> *Bs = (const gmem<char> *)base;
  auto ld = [&](unsigned off) -> Tf { return *(const gmem<Tf> *)(Bs + off); };
  auto ld2 = [&](unsigned off) -> v2 { return *(const gmem<v2> *)(Bs + off); };
  // colour array (parity & 1) of phi and of rhs, computed (not selected)
  auto pcol = [=](int par) -> unsigned { return aP0 + (unsigned)(par & 1) * dP; };
  auto rcol = [=](int par) -> unsigned { return aR0 + (unsigned)(par & 1) * dR; };
  const int x0 = 2 * l;  // fine cells x0 (a0), x0+1 (b0), x0+2 (a1), x0+3 (b1)
  // rows j0-1 and j0+2, ghosts resolved to their image row
  const int ys = BND ? image(j0 - 1, nj, py) : j0 - 1;
  const int yn = BND ? image(j0 + 2, nj, py) : j0 + 2;
  const unsigned o_r0 = (unsigned)j0 * row + ent, o_r1 = o_r0 + row;
  const unsigned o_s = (unsigned)ys * row + ent, o_n = (unsigned)yn * row + ent;
  // x neighbours no lane of the segment holds: fine cell x0-1 for the first
  // lane (the west ghost's image or the previous tile's last entry); for the
  // lane holding the last coarse cell (or lying past it) the east ghost's
  // image, for the segment's last lane otherwise the next tile's first entry
  const bool w_edge = rl == 0;
  const bool e_last = l + 1 >= C.ni - 1;
  const bool e_edge = e_last || rl == lpr - 1;
  const int xw = image(x0 - 1, ni, px);
  const int xe = e_last ? image(ni, ni, px) : x0 + 4;
  const unsigned w_ent = (unsigned)(xw >> 1) * SZ, e_ent = (unsigned)(xe >> 1) * SZ;
  const int w_par = xw & 1, e_par = xe & 1;
  const int x1_par = w_edge ? w_par : e_par;
  const unsigned x1_ent = w_edge ? w_ent : e_ent;
  const Tf cx = (Tf)F.cx, cy = (Tf)F.cy, cz = (Tf)F.cz;
  const Tf aw_a0 = (x0 == 0 && !px) ? Tf(0) : cx;
  const Tf ae_a0 = (x0 == ni - 1 && !px) ? Tf(0) : cx;
  const Tf ae_b0 = (x0 + 1 == ni - 1 && !px) ? Tf(0) : cx;
  const Tf ae_a1 = (x0 + 2 == ni - 1 && !px) ? Tf(0) : cx;
  const Tf ae_b1 = (x0 + 3 == ni - 1 && !px) ? Tf(0) : cx;
  const Tf as0 = (BND && !py && j0 == 0) ? Tf(0) : cy;       // row j0 towards j0-1
  const Tf an1 = (BND && !py && j0 + 1 == nj - 1) ? Tf(0) : cy;  // row j0+1 towards j0+2

  struct PlaneSet {
    v2 fa0, fb0, fa1, fb1;  // rhs of the a and b pairs in rows j0, j0+1
    v2 sa, sb, na, nb;      // rows j0-1 and j0+2
    v2 wa0, wb0, wa1, wb1;  // window plane k+1 of rows j0, j0+1
    Tf we0, we1, ee0, ee1;  // x-edge values of rows j0, j0+1
  };
  auto next_plane = [&](int k) -> int { return BND ? image(k + 1, nk, pz) : k + 1; };
  auto load_set = [&](int k) -> PlaneSet {
    PlaneSet q;
    const unsigned o = (unsigned)k * plane;
    const int c0 = k & 1;  // colour of a in row j0 (j0 even)
    q.fa0 = ld2(rcol(c0) + o + o_r0);
    q.fb0 = ld2(rcol(c0 + 1) + o + o_r0);
    q.fa1 = ld2(rcol(c0 + 1) + o + o_r1);
    q.fb1 = ld2(rcol(c0) + o + o_r1);
    q.sa = ld2(pcol(ys + k) + o + o_s);
    q.sb = ld2(pcol(ys + k + 1) + o + o_s);
    q.na = ld2(pcol(yn + k) + o + o_n);
    q.nb = ld2(pcol(yn + k + 1) + o + o_n);
    const int kp = next_plane(k);
    const unsigned op = (unsigned)kp * plane;
    q.wa0 = ld2(pcol(kp) + op + o_r0);
    q.wb0 = ld2(pcol(kp + 1) + op + o_r0);
    q.wa1 = ld2(pcol(kp + 1) + op + o_r1);
    q.wb1 = ld2(pcol(kp) + op + o_r1);
    // x-edge values: only the lanes at a row segment's ends load them
    const unsigned r0 = (unsigned)j0 * row;
    Tf x10 = Tf(0), x11 = Tf(0), x20 = Tf(0), x21 = Tf(0);
    if (w_edge || e_edge) {
      x10 = ld(pcol(x1_par + k) + o + r0 + x1_ent);
      x11 = ld(pcol(x1_par + k + 1) + o + r0 + row + x1_ent);
    }
    if (w_edge && e_edge) {
      x20 = ld(pcol(e_par + k) + o + r0 + e_ent);
      x21 = ld(pcol(e_par + k + 1) + o + r0 + row + e_ent);
    }
    q.we0 = x10;
    q.we1 = x11;
    q.ee0 = w_edge ? x20 : x10;
    q.ee1 = w_edge ? x21 : x11;
    return q;
  };
  const int k0 = 2 * t.z0;
  v2 ma0, mb0, ma1, mb1, ca0, cb0, ca1, cb1;  // window planes k-1 and k
  {
    const int km = BND ? image(k0 - 1, nk, pz) : k0 - 1;
    const unsigned om = (unsigned)km * plane, oc = (unsigned)k0 * plane;
    ma0 = ld2(pcol(km) + om + o_r0);
    mb0 = ld2(pcol(km + 1) + om + o_r0);
    ma1 = ld2(pcol(km + 1) + om + o_r1);
    mb1 = ld2(pcol(km) + om + o_r1);
    ca0 = ld2(pcol(k0) + oc + o_r0);
    cb0 = ld2(pcol(k0 + 1) + oc + o_r0);
    ca1 = ld2(pcol(k0 + 1) + oc + o_r1);
    cb1 = ld2(pcol(k0) + oc + o_r1);
  }
  // the four cells of one fine row: A/B its a and b pairs, S/N the pairs of
  // the rows below and above, M/W planes k-1 and k+1, F the rhs; adds the
  // residuals of cells a0, b0 to acc0 and a1, b1 to acc1
  auto row_cells = [&](const v2 &A, const v2 &B, const v2 &Sa, const v2 &Sb, const v2 &Na,
                       const v2 &Nb, const v2 &Ma, const v2 &Mb, const v2 &Wa, const v2 &Wb,
                       const v2 &Fa, const v2 &Fb, Tf we, Tf ee, Tf as, Tf an, Tf ab, Tf at,
                       bool first, Tc &acc0, Tc &acc1) {
    // cell x0-1 is lane-1's b1, cell x0+4 is lane+1's a0
    const Tf lf = wave_shift(B.y, 1), rt = wave_shift(A.x, 0);
    const Tf W_a0 = w_edge ? we : lf;
    const Tf E_b0 = l + 1 < C.ni ? A.y : ee;
    const Tf E_b1 = (l + 2 < C.ni && !e_edge) ? rt : ee;
    const Tf ap_a0 = Tf(-1) * (aw_a0 + ae_a0 + as + an + ab + at);
    const Tf ap_b0 = Tf(-1) * (cx + ae_b0 + as + an + ab + at);
    const Tf ap_a1 = Tf(-1) * (cx + ae_a1 + as + an + ab + at);
    const Tf ap_b1 = Tf(-1) * (cx + ae_b1 + as + an + ab + at);
    const Tf r_a0 = Fa.x - (aw_a0 * W_a0 + ae_a0 * B.x + as * Sa.x + an * Na.x + ab * Ma.x +
                            at * Wa.x + ap_a0 * A.x);
    const Tf r_b0 = Fb.x - (cx * A.x + ae_b0 * E_b0 + as * Sb.x + an * Nb.x + ab * Mb.x +
                            at * Wb.x + ap_b0 * B.x);
    const Tf r_a1 = Fa.y - (cx * B.x + ae_a1 * B.y + as * Sa.y + an * Na.y + ab * Ma.y +
                            at * Wa.y + ap_a1 * A.y);
    const Tf r_b1 = Fb.y - (cx * A.y + ae_b1 * E_b1 + as * Sb.y + an * Nb.y + ab * Mb.y +
                            at * Wb.y + ap_b1 * B.y);
    acc0 = first ? (Tc)r_a0 : acc0 + (Tc)r_a0;
    acc0 = acc0 + (Tc)r_b0;
    acc1 = first ? (Tc)r_a1 : acc1 + (Tc)r_a1;
    acc1 = acc1 + (Tc)r_b1;
  };
  Tc acc0 = Tc(0), acc1 = Tc(0);
#pragma unroll
  for (int p = 0; p < NF; ++p) {
    const int k = k0 + p;
    const PlaneSet cur = load_set(k);
    const Tf ab = (BND && !pz && k == 0) ? Tf(0) : cz;
    const Tf at = (BND && !pz && k == nk - 1) ? Tf(0) : cz;
    // row j0: S from row j0-1, N = row j0+1 of the window
    row_cells(ca0, cb0, cur.sa, cur.sb, ca1, cb1, ma0, mb0, cur.wa0, cur.wb0, cur.fa0, cur.fb0,
              cur.we0, cur.ee0, as0, cy, ab, at, !(p & 1), acc0, acc1);
    // row j0+1: S = row j0 of the window, N from row j0+2
    row_cells(ca1, cb1, ca0, cb0, cur.na, cur.nb, ma1, mb1, cur.wa1, cur.wb1, cur.fa1, cur.fb1,
              cur.we1, cur.ee1, cy, an1, ab, at, false, acc0, acc1);
    if (p & 1) {
      // coarse cells l, l+1 (l even): entry l/2 of the two colour arrays
      const int kc = k >> 1;
      const unsigned q =
          ((unsigned)kc * (unsigned)C.nj + (unsigned)jc) * (unsigned)C.H + (unsigned)(l >> 1);
      const int c0 = (l + jc + kc) & 1;
      const Tc v0 = Tc(0.125) * acc0, v1 = Tc(0.125) * acc1;
      if (ok0) {
        ((gmem<Tc> *)C.rhs[c0])[q] = v0;
        zero_state_red<Tc>(C, zbuf, l, jc, kc, q, v0);
      }
      if (ok1) {
        ((gmem<Tc> *)C.rhs[c0 ^ 1])[q] = v1;
        zero_state_red<Tc>(C, zbuf, l + 1, jc, kc, q, v1);
      }
    }
    ma0 = ca0;
    mb0 = cb0;
    ma1 = ca1;
    mb1 = cb1;
    ca0 = cur.wa0;
    cb0 = cur.wb0;
    ca1 = cur.wa1;
    cb1 = cur.wb1;
  }
}

// Restriction tile of an FP32 fine level (mixed precision), KBC coarse planes
// (2*KBC fine planes), software-
// pipelined over the fine planes: a rolling window of fine planes k-1, k, k+1
// of rows 2jc and 2jc+1, with the loads of plane k+1 (rhs of both rows, rows
// 2jc-1 and 2jc+2, x-edge values and window plane k+2) issued before plane k
// is computed.  Neighbours are addressed by the coordinates of their image
// as 32-bit byte offsets from the fine level's arena base, so tiles touching
// a y/z face (BND) run the same code; their coefficients carry cell_coef's
// zeros towards walls.  The eight residuals arrive in the reference's
// summation order (a, b of row 2jc, a, b of row 2jc+1; plane 2kc, then
// 2kc+1).  One coarse cell per lane (FP32 fine entries: four-byte loads; two
// cells per lane cost more occupancy than the loads they save here); C.lpr1
// lanes cover a coarse row; the tile's `lev` is the coarse descriptor.
template <class Tf, class Tc, int KBC, bool BND>
__device__ __forceinline__ void restrict_tile_one(const Tile &t, const LevelDev &C,
                                                  const LevelDev &F, int src_f, bool on,
                                                  int zbuf) {
  constexpr unsigned SZ = sizeof(Tf);
  constexpr int NF = 2 * KBC;
  const int lpr = C.lpr1;
  const int lane = (int)threadIdx.x;
  const int rl = lane & (lpr - 1);
  const int l = t.x0 + rl;
  const int jc = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = F.ni, nj = F.nj, nk = F.nk, H = F.H;
  const bool ok = on && l < C.ni && jc < C.nj;  // on: the block's flag gates the stores
  const bool px = F.per & 1, py = F.per & 2, pz = F.per & 4;
  const unsigned row = (unsigned)H * SZ, plane = row * (unsigned)nj;  // bytes
  const int j0 = 2 * min(jc, C.nj - 1);  // even: a has colour (r + k) & 1 in row j0 + r
  const unsigned ent = (unsigned)min(l, C.ni - 1) * SZ;
  const char *base = (const char *)F.phi[0][0];
  auto aoff = [&](const void *a) -> unsigned { return (unsigned)((const char *)a - base); };
  const unsigned aP0 = aoff(F.phi[src_f][0]), dP = aoff(F.phi[src_f][1]) - aP0;
  const unsigned aR0 = aoff(F.rhs[0]), dR = aoff(F.rhs[1]) - aR0;
  const gmem<char> *Bs = (const gmem<char> *)base;
  auto ld = [&](unsigned off) -> Tf { return *(const gmem<Tf> *)(Bs + off); };
  // colour array (parity & 1) of phi and of rhs, computed (not selected)
  auto pcol = [=](int par) -> unsigned { return aP0 + (unsigned)(par & 1) * dP; };
  auto rcol = [=](int par) -> unsigned { return aR0 + (unsigned)(par & 1) * dR; };
  const int ia = 2 * l, ib = ia + 1;
  // rows j0-1 and j0+2, ghosts resolved to their image row
  const int ys = BND ? image(j0 - 1, nj, py) : j0 - 1;
  const int yn = BND ? image(j0 + 2, nj, py) : j0 + 2;
  const unsigned o_r0 = (unsigned)j0 * row + ent, o_r1 = o_r0 + row;
  const unsigned o_s = (unsigned)ys * row + ent, o_n = (unsigned)yn * row + ent;
  // x neighbours not held by the adjacent lane: x-ghost image or the next
  // tile's entry
  const bool w_edge = ia == 0 || (rl == 0 && l > 0);
  const bool e_edge = ib + 1 >= ni || (rl == lpr - 1 && l + 1 < C.ni);
  const int xw = image(ia - 1, ni, px), xe = image(ib + 1, ni, px);
  const unsigned w_ent = w_edge ? (unsigned)(xw >> 1) * SZ : ent;
  const unsigned e_ent = e_edge ? (unsigned)(xe >> 1) * SZ : ent;
  const int w_par = w_edge ? (xw & 1) : 0, e_par = e_edge ? (xe & 1) : 0;
  const int x1_par = w_edge ? w_par : e_par;
  const unsigned x1_ent = w_edge ? w_ent : e_ent;
  const Tf cx = (Tf)F.cx, cy = (Tf)F.cy, cz = (Tf)F.cz;
  const Tf aw_a = (ia == 0 && !px) ? Tf(0) : cx;
  const Tf ae_a = (ia == ni - 1 && !px) ? Tf(0) : cx;
  const Tf ae_b = (ib == ni - 1 && !px) ? Tf(0) : cx;
  const Tf as0 = (BND && !py && j0 == 0) ? Tf(0) : cy;       // row j0 towards j0-1
  const Tf an1 = (BND && !py && j0 + 1 == nj - 1) ? Tf(0) : cy;  // row j0+1 towards j0+2

  struct PlaneSet {
    Tf fa0, fb0, fa1, fb1;  // rhs of a, b in rows j0, j0+1
    Tf sa, sb, na, nb;      // rows j0-1 and j0+2
    Tf wa0, wb0, wa1, wb1;  // window plane k+1 of rows j0, j0+1
    Tf we0, we1, ee0, ee1;  // x-edge values of rows j0, j0+1
  };
  auto next_plane = [&](int k) -> int { return BND ? image(k + 1, nk, pz) : k + 1; };
  auto load_set = [&](int k) -> PlaneSet {
    PlaneSet q;
    const unsigned o = (unsigned)k * plane;
    const int c0 = k & 1;  // colour of a in row j0 (j0 even)
    q.fa0 = ld(rcol(c0) + o + o_r0);
    q.fb0 = ld(rcol(c0 + 1) + o + o_r0);
    q.fa1 = ld(rcol(c0 + 1) + o + o_r1);
    q.fb1 = ld(rcol(c0) + o + o_r1);
    q.sa = ld(pcol(ys + k) + o + o_s);
    q.sb = ld(pcol(ys + k + 1) + o + o_s);
    q.na = ld(pcol(yn + k) + o + o_n);
    q.nb = ld(pcol(yn + k + 1) + o + o_n);
    const int kp = next_plane(k);
    const unsigned op = (unsigned)kp * plane;
    q.wa0 = ld(pcol(kp) + op + o_r0);
    q.wb0 = ld(pcol(kp + 1) + op + o_r0);
    q.wa1 = ld(pcol(kp + 1) + op + o_r1);
    q.wb1 = ld(pcol(kp) + op + o_r1);
    // x-edge values: only the lanes at a row segment's ends use them (the
    // others read no x-edge value at all)
    const unsigned r0 = (unsigned)j0 * row;
    Tf x10 = Tf(0), x11 = Tf(0), x20 = Tf(0), x21 = Tf(0);
    if (w_edge || e_edge) {
      x10 = ld(pcol(x1_par + k) + o + r0 + x1_ent);
      x11 = ld(pcol(x1_par + k + 1) + o + r0 + row + x1_ent);
    }
    if (w_edge && e_edge) {
      x20 = ld(pcol(e_par + k) + o + r0 + e_ent);
      x21 = ld(pcol(e_par + k + 1) + o + r0 + row + e_ent);
    }
    q.we0 = x10;
    q.we1 = x11;
    q.ee0 = w_edge ? x20 : x10;
    q.ee1 = w_edge ? x21 : x11;
    return q;
  };
  const int k0 = 2 * t.z0;
  Tf ma0, mb0, ma1, mb1, ca0, cb0, ca1, cb1;  // window planes k-1 and k
  {
    const int km = BND ? image(k0 - 1, nk, pz) : k0 - 1;
    const unsigned om = (unsigned)km * plane, oc = (unsigned)k0 * plane;
    ma0 = ld(pcol(km) + om + o_r0);
    mb0 = ld(pcol(km + 1) + om + o_r0);
    ma1 = ld(pcol(km + 1) + om + o_r1);
    mb1 = ld(pcol(km) + om + o_r1);
    ca0 = ld(pcol(k0) + oc + o_r0);
    cb0 = ld(pcol(k0 + 1) + oc + o_r0);
    ca1 = ld(pcol(k0 + 1) + oc + o_r1);
    cb1 = ld(pcol(k0) + oc + o_r1);
  }
  PlaneSet cur = load_set(k0);
  Tc acc = Tc(0);
#pragma unroll
  for (int p = 0; p < NF; ++p) {
    const int k = k0 + p;
    PlaneSet nxt;
    if (p + 1 < NF) nxt = load_set(k + 1);
    const Tf ab = (BND && !pz && k == 0) ? Tf(0) : cz;
    const Tf at = (BND && !pz && k == nk - 1) ? Tf(0) : cz;
    // row j0 (r = 0): S from row j0-1, N = row j0+1 of the window
    {
      const Tf Pa = ca0, Pb = cb0;
      // cell 2l-1 is lane l-1's b, cell 2l+2 is lane l+1's a
      const Tf lf = wave_shift(Pb, 1), rt = wave_shift(Pa, 0);
      const Tf Wa = w_edge ? cur.we0 : lf;
      const Tf Ea = ib < ni ? Pb : cur.ee0;
      const Tf Eb = e_edge ? cur.ee0 : rt;
      const Tf ap_a = Tf(-1) * (aw_a + ae_a + as0 + cy + ab + at);
      const Tf ap_b = Tf(-1) * (cx + ae_b + as0 + cy + ab + at);
      const Tf ra = cur.fa0 - (aw_a * Wa + ae_a * Ea + as0 * cur.sa + cy * ca1 + ab * ma0 +
                               at * cur.wa0 + ap_a * Pa);
      const Tf rb = cur.fb0 - (cx * Pa + ae_b * Eb + as0 * cur.sb + cy * cb1 + ab * mb0 +
                               at * cur.wb0 + ap_b * Pb);
      acc = (p & 1) ? acc + (Tc)ra : (Tc)ra;
      acc = acc + (Tc)rb;
    }
    // row j0+1 (r = 1): S = row j0 of the window, N from row j0+2
    {
      const Tf Pa = ca1, Pb = cb1;
      const Tf lf = wave_shift(Pb, 1), rt = wave_shift(Pa, 0);
      const Tf Wa = w_edge ? cur.we1 : lf;
      const Tf Ea = ib < ni ? Pb : cur.ee1;
      const Tf Eb = e_edge ? cur.ee1 : rt;
      const Tf ap_a = Tf(-1) * (aw_a + ae_a + cy + an1 + ab + at);
      const Tf ap_b = Tf(-1) * (cx + ae_b + cy + an1 + ab + at);
      const Tf ra = cur.fa1 - (aw_a * Wa + ae_a * Ea + cy * ca0 + an1 * cur.na + ab * ma1 +
                               at * cur.wa1 + ap_a * Pa);
      const Tf rb = cur.fb1 - (cx * Pa + ae_b * Eb + cy * cb0 + an1 * cur.nb + ab * mb1 +
                               at * cur.wb1 + ap_b * Pb);
      acc = acc + (Tc)ra;
      acc = acc + (Tc)rb;
    }
    if (p & 1) {
      const int kc = k >> 1;
      if (ok) {
        gmem<Tc> *D = (gmem<Tc> *)C.rhs[(l + jc + kc) & 1];
        const unsigned q =
            ((unsigned)kc * (unsigned)C.nj + (unsigned)jc) * (unsigned)C.H + (unsigned)(l >> 1);
        const Tc v = Tc(0.125) * acc;
        D[q] = v;
        zero_state_red<Tc>(C, zbuf, l, jc, kc, q, v);
      }
    }
    ma0 = ca0;
    mb0 = cb0;
    ma1 = ca1;
    mb1 = cb1;
    ca0 = cur.wa0;
    cb0 = cur.wb0;
    ca1 = cur.wa1;
    cb1 = cur.wb1;
    if (p + 1 < NF) cur = nxt;
  }
}

// The restriction tile of the fine level's storage type: two coarse cells per
// lane on an FP64 fine level (16-byte loads), one on an FP32 one; the tile
// geometry follows (restriction tiles span 2*lpr1 or lpr1 coarse cells).
template <class Tf, class Tc, int KBC, bool BND>
__device__ __forceinline__ void restrict_tile_fast(const Tile &t, const LevelDev &C,
                                                   const LevelDev &F, int src_f, bool on,
                                                   int zbuf) {
  if constexpr (sizeof(Tf) == 8)
    restrict_tile_two<Tf, Tc, KBC, BND>(t, C, F, src_f, on, zbuf);
  else
    restrict_tile_one<Tf, Tc, KBC, BND>(t, C, F, src_f, on, zbuf);
}

// One launch per coarse level: tiles of KBC coarse planes, kind 0 when every
// fine row and plane the tile reads is inside the block, kind 3 otherwise.
// ONE, scalar arguments: as k_rb_sweep (one_lev the coarse descriptor,
// one_lev2 its finer level).
template <class Tf, class Tc, int KBC, bool ONE>
__global__ void __launch_bounds__(NTHREADS)
    k_restrict(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
               const int *__restrict__ active, int src_f, int one_lev, int one_lev2, int one_blk,
               int ntiles, int zbuf) {
  const Tile t = tiles[xcd_remap((int)blockIdx.x, ntiles)];
  if (ONE) {
    const LevelDev &C = levs[one_lev], &F = levs[one_lev2];
    const int on = active[one_blk];
    asm volatile("" ::"s"(t.x0), "s"(t.y0), "s"(t.z0), "s"(t.kind), "s"(on), "s"(C.ni), "s"(C.nj),
                 "s"(C.H), "s"(C.lpr1), "s"(C.rhs[0]), "s"(C.rhs[1]), "s"(F.ni), "s"(F.nj),
                 "s"(F.nk), "s"(F.H), "s"(F.per), "s"(F.cx), "s"(F.cy), "s"(F.cz),
                 "s"(F.phi[0][0]), "s"(F.phi[0][1]), "s"(F.phi[1][0]), "s"(F.phi[1][1]),
                 "s"(F.rhs[0]), "s"(F.rhs[1]));
    if (t.kind == 0)
      restrict_tile_fast<Tf, Tc, KBC, false>(t, C, F, src_f, on != 0, zbuf);
    else
      restrict_tile_fast<Tf, Tc, KBC, true>(t, C, F, src_f, on != 0, zbuf);
    return;
  }
  const LevelDev &C = levs[t.lev];
  if (!active[C.blk]) return;
  const LevelDev &F = levs[C.finer];
  if (t.kind == 0)
    restrict_tile_fast<Tf, Tc, KBC, false>(t, C, F, src_f, true, zbuf);
  else
    restrict_tile_fast<Tf, Tc, KBC, true>(t, C, F, src_f, true, zbuf);
}

// ---------------------------------------------------------------------------
// mgcorr (mgsolver.for:828-896): fine += trilinear interpolation of coarse.
// Fine padded index ip = 2*icp + d with icp the coarse padded index; the
// weight of coarse corner (oi,oj,ok) is prod (3 if o==d else 1); terms are
// summed in the order c, c+j, c+k, c+k+j, c+i, c+i+j, c+i+k, c+i+j+k and the
// sum divided by 64.  Ghost corners are virtual (images of coarse interior).
//
// A thread owns fine entry l of both colours (cells 2l and 2l+1) in fine rows
// 2m-1, 2m and planes 2n-1, 2n (coarse row m and plane n in padded numbering):
// those eight fine cells share the twelve coarse corners x in {l-1, l, l+1},
// y in {m-1, m}, z in {n-1, n} (interior numbering), which are loaded once.
// Tile::x0 = first l, y0 = first m, z0 = n, kind = lanes per row: short rows
// share a wavefront (48 blocks of 32 to 128 cells per axis, a row a wavefront:
// 48 us on level 1, now 27).  The fine
// level is updated in place (each fine cell by exactly one thread).
// GEN: blocks with neighbours -- the coarse ghost corners (edges and corners
// included) may lie in another block.  All lanes of a row pair share its
// corner rows, and in x a corner is inside the row or across one of its two
// ends: the rows and their ends are resolved (resolve_cell) into LDS and every
// lane picks, instead of following the neighbour table for sixteen corners,
// one after the other.
// skip_red: a red half-sweep follows.  It replaces every red cell from black
// neighbours, and of the red values before it only those on open (periodic or
// shared) faces are read again, as ghosts of the black half-sweep: the other
// red cells are left as they are, unless a correction is not finite (a wall's
// term is zero times the cell's own value: NaN after an infinite correction).
// The kernel streams the fine level, so that takes up to half its traffic (four
// levels of 256^3, FP64: 18.0 us a launch, now 14.0; float 10.2 and 9.4).
// ONE, scalar arguments: as k_rb_sweep (one_lev the fine descriptor,
// one_lev2 its coarser level).
template <class Tf, class Tc, bool GEN, bool ONE>
__global__ void __launch_bounds__(NTHREADS)
    k_prolong(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
              const int *__restrict__ active, int src_f, int src_c, int one_lev, int one_lev2,
              int one_blk, int ntiles, int skip_red) {
  const Tile t = tiles[xcd_remap((int)blockIdx.x, ntiles)];
  const LevelDev &F = levs[ONE ? one_lev : t.lev];
  const int on = ONE ? active[one_blk] : 1;
  if (!ONE && !active[F.blk]) return;
  const LevelDev &C = levs[ONE ? one_lev2 : F.coarser];
  if (ONE)
    asm volatile("" ::"s"(t.x0), "s"(t.y0), "s"(t.z0), "s"(t.kind), "s"(on), "s"(F.ni), "s"(F.nj),
                 "s"(F.nk), "s"(F.H), "s"(F.phi[0][0]), "s"(F.phi[0][1]), "s"(F.phi[1][0]), "s"(F.phi[1][1]),
                 "s"(C.ni), "s"(C.nj), "s"(C.nk), "s"(C.H), "s"(C.per), "s"(C.phi[0][0]),
                 "s"(C.phi[0][1]), "s"(C.phi[1][0]), "s"(C.phi[1][1]));
  // a thread holds fine entries l, l+1 (l even): cells 2l .. 2l+3 of the
  // 2x2 rows and planes around coarse row pair m, plane pair n
  typedef typename Vec2<Tf>::type v2;
  const int lpr = t.kind;  // lanes per row, a power of two
  const int l = t.x0 + 2 * ((int)threadIdx.x & (lpr - 1));
  const int rw = ((int)threadIdx.y * 64 + (int)threadIdx.x) / lpr;  // row pair of the tile
  const int m = t.y0 + rw;
  const int n = t.z0;
  // GEN: the corner rows (y, z) of every row pair of the tile, inside the
  // block's x range, before it and after it: the row's arrays by the parity of
  // x, and the x of the end cell
  struct RowSrc {
    const gmem<Tc> *p[2];
    int x;
  };
  __shared__ RowSrc rows[GEN ? PROL_GEN_ROWS : 1][12];
  if (GEN) {
    const int nq = 12 * (NTHREADS / lpr);
    for (int q = (int)threadIdx.y * 64 + (int)threadIdx.x; q < nq; q += NTHREADS) {
      const int w = q / 12, e = q - 12 * w;
      int x = e % 3 == 0 ? 0 : e % 3 == 1 ? -1 : C.ni;
      int y = min(t.y0 + w, C.nj) - 1 + (e / 3) % 2, z = min(n, C.nk) - 1 + e / 6;
      const LevelDev &P = levs[resolve_cell(levs, F.coarser, x, y, z)];
      const size_t row = ((size_t)z * P.nj + y) * P.H;
      RowSrc &r = rows[w][e];
      r.p[0] = (const gmem<Tc> *)P.phi[src_c][(y + z) & 1] + row;
      r.p[1] = (const gmem<Tc> *)P.phi[src_c][(y + z + 1) & 1] + row;
      r.x = x;
    }
    __syncthreads();
  }
  if (2 * l >= F.ni || m > C.nj || n > C.nk) return;
  const bool two = 2 * l + 2 < F.ni;  // entry l+1 holds cells (F.ni is even)
  const bool px = C.per & 1, py = C.per & 2, pz = C.per & 4;
  const gmem<Tc> *C0 = (const gmem<Tc> *)C.phi[src_c][0];
  const gmem<Tc> *C1 = (const gmem<Tc> *)C.phi[src_c][1];
  // coarse corner coordinates x = l-1 .. l+2 (interior numbering, ghosts
  // resolved; the last is read only when entry l+1 holds cells)
  int xc[4], yc[2], zc[2];
  for (int a = 0; a < 4; ++a) xc[a] = image(min(l - 1 + a, two ? l + 2 : l + 1), C.ni, px);
  for (int a = 0; a < 2; ++a) {
    yc[a] = image(m - 1 + a, C.nj, py);
    zc[a] = image(n - 1 + a, C.nk, pz);
  }
  Tc cv[4][2][2];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        if (GEN) {
          const int x = min(l - 1 + a, two ? l + 2 : l + 1);
          const int at = x < 0 ? 1 : x >= C.ni ? 2 : 0;
          const RowSrc r = rows[rw][at + 3 * (b + 2 * c)];
          const int xx = at == 0 ? x : r.x;
          cv[a][b][c] = ((xx & 1) ? r.p[1] : r.p[0])[xx >> 1];
        } else {
          const unsigned off = ((unsigned)zc[c] * (unsigned)C.nj + (unsigned)yc[b]) *
                                   (unsigned)C.H + (unsigned)(xc[a] >> 1);
          cv[a][b][c] = ((xc[a] + yc[b] + zc[c]) & 1) ? C1[off] : C0[off];
        }
      }
  Tc all = cv[0][0][0];  // finite: every corner is
#pragma unroll
  for (int q = 1; q < 16; ++q) all = all + cv[q >> 2][(q >> 1) & 1][q & 1];
  const bool finite = isfinite(all);
  gmem<Tf> *F0 = (gmem<Tf> *)F.phi[src_f][0];
  gmem<Tf> *F1 = (gmem<Tf> *)F.phi[src_f][1];
  // lanes with a cell on an open x face (the fine and coarse level have the
  // same faces)
  const bool xw = GEN ? !wall_face(F, 0) : px, xe = GEN ? !wall_face(F, 1) : px;
  const bool x_open = (xw && l == 0) || (xe && 2 * l + 4 >= F.ni);
#pragma unroll
  for (int dk = 0; dk < 2; ++dk) {
    const int k = 2 * n - 1 + dk;
    if (k < 0 || k >= F.nk) continue;
#pragma unroll
    for (int dj = 0; dj < 2; ++dj) {
      const int j = 2 * m - 1 + dj;
      if (j < 0 || j >= F.nj) continue;
      const unsigned fq = ((unsigned)k * (unsigned)F.nj + (unsigned)j) * (unsigned)F.H + (unsigned)l;
      // the row's cells 2l+e with e = (j+k) & 1 are red
      bool red = !skip_red || x_open || !finite;
      if (GEN)
        red = red || (j == 0 && !wall_face(F, 2)) || (j == F.nj - 1 && !wall_face(F, 3)) ||
              (k == 0 && !wall_face(F, 4)) || (k == F.nk - 1 && !wall_face(F, 5));
      else
        red = red || (py && (j == 0 || j == F.nj - 1)) || (pz && (k == 0 || k == F.nk - 1));
      // the correction of cell 2(l+ee)+e: corners x = l+ee-1+e, l+ee+e with
      // di = 1-e, summed in the corner order c, c+j, c+k, c+k+j, c+i, ...
      Tc cr[2][2];  // [e][ee]
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int ee = 0; ee < 2; ++ee) {
          const int di = 1 - e;
          Tc s;
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            const int oi = q >> 2, oj = q & 1, ok = (q >> 1) & 1;
            const Tc w = (oi == di ? Tc(3) : Tc(1)) * (oj == dj ? Tc(3) : Tc(1)) *
                         (ok == dk ? Tc(3) : Tc(1));
            const Tc v = cv[ee + e + oi][oj][ok];
            s = (q == 0) ? w * v : s + w * v;
          }
          cr[e][ee] = s;
        }
      // cells 2l+e and 2l+2+e share a colour array: entries l, l+1
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const bool black = (e + j + k) & 1;
        if (!black && !red) continue;
        gmem<Tf> *fa = black ? F1 : F0;
        if (two) {
          v2 v = *(gmem<v2> *)(fa + fq);
          v.x = v.x + (Tf)(cr[e][0] / Tc(64));
          v.y = v.y + (Tf)(cr[e][1] / Tc(64));
          if (on) *(gmem<v2> *)(fa + fq) = v;
        } else {
          const Tf nv = fa[fq] + (Tf)(cr[e][0] / Tc(64));
          if (on) fa[fq] = nv;
        }
      }
    }
  }
}

template <class T>
__global__ void __launch_bounds__(NTHREADS)
    k_fill_zero(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                const int *__restrict__ active, int buf) {
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const int i = t.x0 + (int)threadIdx.x;
  const int j = t.y0 + (int)threadIdx.y;
  const int k = t.z0;
  if (i >= L.ni || j >= L.nj || k >= L.nk) return;
  ((T *)L.phi[buf][(i + j + k) & 1])[cidx(L.H, L.nj, i, j, k)] = T(0);
}

// 64-lane wavefront + LDS reduction in a fixed order (deterministic).
__device__ __forceinline__ void block_reduce(double &ss, double &am) {
  for (int off = 32; off > 0; off >>= 1) {
    ss += __shfl_xor(ss, off, 64);
    am = fmax(am, __shfl_xor(am, off, 64));
  }
  __shared__ double s_ss[NTHREADS / 64], s_am[NTHREADS / 64];
  const int tid = (int)(threadIdx.x + blockDim.x * threadIdx.y);
  const int w = tid >> 6;
  if ((tid & 63) == 0) {
    s_ss[w] = ss;
    s_am[w] = am;
  }
  __syncthreads();
  if (tid == 0) {
    double a = s_ss[0], b = s_am[0];
    for (int q = 1; q < NTHREADS / 64; ++q) {
      a += s_ss[q];
      b = fmax(b, s_am[q]);
    }
    ss = a;
    am = b;
  }
}

// ---------------------------------------------------------------------------
// Finest-level residual r = f - A p in FP64 (the rhs of the next V-cycle; in
// the reference it is su = div(u* - dt grad p)/dt, press.for:2-144), stored
// into the level-1 rhs in the level's precision, with per-tile partial sum of
// r^2 and max |r| for the REL_L2 and REF_RMAX criteria.
//
// A lane holds entry l of both colour arrays of one row: the two adjacent
// cells a = 2l (colour ca = (j+k)&1) and b = 2l+1.  Planes k-1..k+1 of both
// entries stream through a register window, x-neighbours come from the lane's
// other cell or the adjacent lanes (DPP shift), rows j-1, j+1 are loaded.
// A residual tile spans 2*F.lpr colour entries of a row (64/F.lpr rows per
// wavefront; the fast kernel gives each lane two entries); this path walks
// it as two halves of F.lpr entries, one entry per lane (x0: the half's
// first entry), over the planes [t.z0, t.z1).  Tile kind 0: every row/plane
// of the tile has its y/z neighbours inside the block; kind 1: the general
// path with ghost images.  use_p = 0 gives r = f (the norm of the
// right-hand side).
template <class T, bool INNER>
__device__ __forceinline__ void residual_half(const Tile &t, int x0, const FineDev *__restrict__ fine,
                                              const LevelDev &L, int use_p, double &ss,
                                              double &am) {
  const FineDev &F = fine[t.lev];
  const int lpr = F.lpr;
  const int lane = (int)threadIdx.x;
  const int rl = lane & (lpr - 1);
  const int l = x0 + rl;
  const int j = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = F.ni, nj = F.nj, nk = F.nk, H = F.H;
  const bool ok = 2 * l < ni && j < nj;
  const bool b_ok = 2 * l + 1 < ni && j < nj;
  const unsigned row = (unsigned)H, plane = (unsigned)H * (unsigned)nj;
  // jc: the lane's row clamped like cbase -- lanes beyond the last row load
  // in-bounds rows and resolve in-bounds ghosts (their results are not
  // stored); for every stored cell jc == j
  const int jc = min(j, nj - 1);
  const unsigned cbase = (unsigned)jc * row + (unsigned)min(l, H - 1);
  const gmem<double> *P0 = (const gmem<double> *)F.p[0], *P1 = (const gmem<double> *)F.p[1];
  const gmem<double> *F0 = (const gmem<double> *)F.f[0], *F1 = (const gmem<double> *)F.f[1];
  gmem<T> *R0 = (gmem<T> *)L.rhs[0], *R1 = (gmem<T> *)L.rhs[1];
  const bool tile_left = l > 0 && rl == 0;             // entry l-1 in another tile
  const bool tile_right = rl == lpr - 1 && l + 1 < H;  // entry l+1 in another tile
  const bool px = F.per & 1;
  const double cx = F.cx, cy = F.cy, cz = F.cz;
  auto ldp = [&](int c, unsigned off) -> double { return c ? P1[off] : P0[off]; };
  auto own = [&](int k, int c) -> double {
    if (!INNER && (unsigned)k >= (unsigned)nk) return 0.0;
    return ldp(c, (unsigned)k * plane + cbase);
  };

  const int k1 = t.z1;
  int k = t.z0;
  double w0m = 0, w1m = 0, w0c = 0, w1c = 0;
  if (use_p) {
    w0m = own(k - 1, 0);
    w1m = own(k - 1, 1);
    w0c = own(k, 0);
    w1c = own(k, 1);
  }
  for (; k < k1; ++k) {
    const unsigned q = (unsigned)k * plane + cbase;
    const int ca = (j + k) & 1, cb = ca ^ 1;
    double ra = ca ? F1[q] : F0[q];
    double rb = cb ? F1[q] : F0[q];
    double w0p = 0, w1p = 0;
    if (use_p) {
      w0p = own(k + 1, 0);
      w1p = own(k + 1, 1);
      const double Pa = ca ? w1c : w0c, Pb = ca ? w0c : w1c;
      // x-neighbours: cell 2l-1 is lane-1's b, cell 2l+2 is lane+1's a
      double lf = wave_shift(Pb, 1), rt = wave_shift(Pa, 0);
      if (tile_left) lf = ldp(cb, q - 1);
      if (tile_right) rt = ldp(ca, q + 1);
      const int ia = 2 * l, ib = ia + 1;
      const double Wa = ia == 0 ? fine_value(fine, t.lev, -1, jc, k) : lf;
      const double Ea = ib < ni ? Pb : fine_value(fine, t.lev, ni, jc, k);
      const double Wb = Pa;
      const double Eb = ib + 1 < ni ? rt : fine_value(fine, t.lev, ni, jc, k);
      // y- and z-neighbours of a (colour cb there) and b (colour ca)
      double Sa, Na, Sb, Nb;
      if (INNER || jc > 0) {
        Sa = ldp(cb, q - row);
        Sb = ldp(ca, q - row);
      } else {
        Sa = fine_value(fine, t.lev, ia, -1, k);
        Sb = fine_value(fine, t.lev, ib, -1, k);
      }
      if (INNER || jc + 1 < nj) {
        Na = ldp(cb, q + row);
        Nb = ldp(ca, q + row);
      } else {
        Na = fine_value(fine, t.lev, ia, nj, k);
        Nb = fine_value(fine, t.lev, ib, nj, k);
      }
      const double Ba = (INNER || k > 0) ? (cb ? w1m : w0m) : fine_value(fine, t.lev, ia, jc, -1);
      const double Bb = (INNER || k > 0) ? (ca ? w1m : w0m) : fine_value(fine, t.lev, ib, jc, -1);
      const double Ta = (INNER || k + 1 < nk) ? (cb ? w1p : w0p) : fine_value(fine, t.lev, ia, jc, nk);
      const double Tb = (INNER || k + 1 < nk) ? (ca ? w1p : w0p) : fine_value(fine, t.lev, ib, jc, nk);
      Coef<double> c_a, c_b;
      if (INNER) {
        c_a.as = c_a.an = c_b.as = c_b.an = cy;
        c_a.ab = c_a.at = c_b.ab = c_b.at = cz;
        c_a.aw = (ia == 0 && !px) ? 0.0 : cx;
        c_a.ae = (ia == ni - 1 && !px) ? 0.0 : cx;
        c_b.aw = cx;
        c_b.ae = (ib == ni - 1 && !px) ? 0.0 : cx;
        c_a.ap = -1.0 * (c_a.aw + c_a.ae + c_a.as + c_a.an + c_a.ab + c_a.at);
        c_b.ap = -1.0 * (c_b.aw + c_b.ae + c_b.as + c_b.an + c_b.ab + c_b.at);
      } else {
        c_a = fine_coef(F, ia, j, k);
        c_b = fine_coef(F, ib, j, k);
      }
      ra = ra - (c_a.aw * Wa + c_a.ae * Ea + c_a.as * Sa + c_a.an * Na + c_a.ab * Ba +
                 c_a.at * Ta + c_a.ap * Pa);
      rb = rb - (c_b.aw * Wb + c_b.ae * Eb + c_b.as * Sb + c_b.an * Nb + c_b.ab * Bb +
                 c_b.at * Tb + c_b.ap * Pb);
    }
    if (ok) {
      (ca ? R1 : R0)[q] = (T)ra;
      ss += ra * ra;
      am = fmax(am, fabs(ra));
    }
    if (b_ok) {
      (cb ? R1 : R0)[q] = (T)rb;
      ss += rb * rb;
      am = fmax(am, fabs(rb));
    }
    w0m = w0c;
    w1m = w1c;
    w0c = w0p;
    w1c = w1p;
  }
}

template <class T, bool INNER>
__device__ __forceinline__ void residual_tile(const Tile &t, const FineDev *__restrict__ fine,
                                              const LevelDev &L, int use_p, double &ss,
                                              double &am) {
  const int lpr = fine[t.lev].lpr;
  residual_half<T, INNER>(t, t.x0, fine, L, use_p, ss, am);
  residual_half<T, INNER>(t, t.x0 + lpr, fine, L, use_p, ss, am);
}

// Finest-level residual tile of KB planes, software-pipelined: a rolling
// window of planes k-1, k, k+1 of both colours, with the loads of plane k+1
// (its f, rows j-1/j+1, x-edge values and window plane k+2) issued before
// plane k is computed), two colour entries per lane.  Every neighbour is
// addressed by the coordinates of its image (a ghost row, plane or x position resolved once per lane or per
// plane), as a 32-bit byte offset from the block's first fine array, so
// boundary tiles (BND) run the same code as interior ones; only their
// coefficients differ (cell_coef's zeros towards walls).  The arithmetic of
// every cell is residual_tile's.
template <class T, int KB, bool BND>
__device__ __forceinline__ void residual_tile_fast(const Tile &t, const FineDev &F,
                                                   const LevelDev &L, double &ss, double &am,
                                                   int zbuf) {
  typedef typename Vec2<double>::type d2;
  typedef typename Vec2<T>::type t2;
  constexpr unsigned SZ = sizeof(double);
  // a lane holds entries l0, l0+1 of both colour arrays of its row: cells
  // x0 (a0), x0+1 (b0), x0+2 (a1), x0+3 (b1); a0/a1 share a colour array, as
  // do b0/b1, so each array is one 16-byte load
  const int lpr = F.lpr;
  const int lane = (int)threadIdx.x;
  const int rl = lane & (lpr - 1);
  const int l0 = t.x0 + 2 * rl;
  const int j = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = F.ni, nj = F.nj, nk = F.nk, H = F.H;
  const int x0 = 2 * l0;
  const bool row_ok = j < nj;
  const bool ok_a0 = row_ok && x0 < ni, ok_b0 = row_ok && x0 + 1 < ni;
  const bool ok_a1 = row_ok && x0 + 2 < ni, ok_b1 = row_ok && x0 + 3 < ni;
  const int jc = min(j, nj - 1);
  const bool px = F.per & 1, py = F.per & 2, pz = F.per & 4;
  const unsigned row = (unsigned)H * SZ, plane = row * (unsigned)nj;  // bytes
  const char *base = (const char *)F.p[0];
  const unsigned aP1 = (unsigned)((const char *)F.p[1] - base);
  const unsigned aF0 = (unsigned)((const char *)F.f[0] - base);
  const unsigned aF1 = (unsigned)((const char *)F.f[1] - base);
  const gmem<char> *Bs = (const gmem<char> *)base;
  gmem<T> *R[2] = {(gmem<T> *)L.rhs[0], (gmem<T> *)L.rhs[1]};
  auto ld = [&](unsigned off) -> double { return *(const gmem<double> *)(Bs + off); };
  auto ld2 = [&](unsigned off) -> d2 { return *(const gmem<d2> *)(Bs + off); };
  // p of the cells of parity `par` (x + y + k) in a row: colour array par & 1
  auto pcol = [&](int par) -> unsigned { return (par & 1) ? aP1 : 0u; };
  // lanes past the row's last pair read that pair (nothing of theirs is stored)
  const unsigned ent = (unsigned)min(l0, H - 2) * SZ;
  // rows of the y neighbours, ghosts resolved to their image row
  const int ys = BND ? image(jc - 1, nj, py) : jc - 1;
  const int yn = BND ? image(jc + 1, nj, py) : jc + 1;
  const unsigned o_c = (unsigned)jc * row + ent;
  const unsigned o_s = (unsigned)ys * row + ent, o_n = (unsigned)yn * row + ent;
  // x neighbours no lane of the row segment holds: cell x0-1 for the
  // segment's first lane (the west ghost's image, or the previous tile's last
  // entry); for the lane holding cell ni-1 (or lying past it) the east
  // ghost's image, for the segment's last lane otherwise the next tile's
  // first entry
  const bool w_edge = rl == 0;
  const bool e_last = x0 + 3 >= ni - 1;
  const bool e_edge = e_last || rl == lpr - 1;
  const int xw = image(x0 - 1, ni, px);
  const int xe = e_last ? image(ni, ni, px) : x0 + 4;
  const unsigned w_ent = (unsigned)jc * row + (unsigned)(xw >> 1) * SZ;
  const unsigned e_ent = (unsigned)jc * row + (unsigned)(xe >> 1) * SZ;
  const int w_par = xw & 1, e_par = xe & 1;
  const int x1_par = w_edge ? w_par : e_par;
  const unsigned x1_ent = w_edge ? w_ent : e_ent;
  const double cx = F.cx, cy = F.cy, cz = F.cz;
  const double aw_a0 = (x0 == 0 && !px) ? 0.0 : cx;
  const double ae_a0 = (x0 == ni - 1 && !px) ? 0.0 : cx;
  const double ae_b0 = (x0 + 1 == ni - 1 && !px) ? 0.0 : cx;
  const double ae_a1 = (x0 + 2 == ni - 1 && !px) ? 0.0 : cx;
  const double ae_b1 = (x0 + 3 == ni - 1 && !px) ? 0.0 : cx;
  const double as = (BND && !py && jc == 0) ? 0.0 : cy;
  const double an = (BND && !py && jc == nj - 1) ? 0.0 : cy;

  struct PlaneSet {
    d2 fa, fb, sa, sb, na, nb, ap1, bp1;  // ap1/bp1: window plane k+1
    double we, ee;
  };
  // the window plane after k: plane k+1 or its image
  auto next_plane = [&](int k) -> int { return BND ? image(k + 1, nk, pz) : k + 1; };
  auto load_set = [&](int k) -> PlaneSet {
    PlaneSet q;
    const unsigned o = (unsigned)k * plane;
    const int ca = (jc + k) & 1;
    q.fa = ld2((ca ? aF1 : aF0) + o + o_c);
    q.fb = ld2((ca ? aF0 : aF1) + o + o_c);
    q.sa = ld2(pcol(ys + k) + o + o_s);
    q.sb = ld2(pcol(ys + k + 1) + o + o_s);
    q.na = ld2(pcol(yn + k) + o + o_n);
    q.nb = ld2(pcol(yn + k + 1) + o + o_n);
    const int kp = next_plane(k);
    q.ap1 = ld2(pcol(jc + kp) + (unsigned)kp * plane + o_c);
    q.bp1 = ld2(pcol(jc + kp + 1) + (unsigned)kp * plane + o_c);
    // x-edge values: only the lanes at a row segment's ends load them
    double x1 = 0.0, x2 = 0.0;
    if (w_edge || e_edge) x1 = ld(pcol(x1_par + jc + k) + o + x1_ent);
    if (w_edge && e_edge) x2 = ld(pcol(e_par + jc + k) + o + e_ent);
    q.we = x1;
    q.ee = w_edge ? x2 : x1;
    return q;
  };
  const int k0 = t.z0;
  // window: the a and b pairs of planes k0-1 and k0
  d2 am1, bm1, A, B;
  {
    const int km = BND ? image(k0 - 1, nk, pz) : k0 - 1;
    am1 = ld2(pcol(jc + km) + (unsigned)km * plane + o_c);
    bm1 = ld2(pcol(jc + km + 1) + (unsigned)km * plane + o_c);
    A = ld2(pcol(jc + k0) + (unsigned)k0 * plane + o_c);
    B = ld2(pcol(jc + k0 + 1) + (unsigned)k0 * plane + o_c);
  }
#pragma unroll
  for (int p = 0; p < KB; ++p) {
    const int k = k0 + p;
    const PlaneSet cur = load_set(k);
    // cell x0-1 is lane-1's b1, cell x0+4 is lane+1's a0
    const double lf = wave_shift(B.y, 1), rt = wave_shift(A.x, 0);
    const double W_a0 = w_edge ? cur.we : lf;
    const double E_a0 = x0 + 1 < ni ? B.x : cur.ee;
    const double E_b0 = x0 + 2 < ni ? A.y : cur.ee;
    const double E_a1 = x0 + 3 < ni ? B.y : cur.ee;
    const double E_b1 = (x0 + 4 < ni && !e_edge) ? rt : cur.ee;
    const double ab = (BND && !pz && k == 0) ? 0.0 : cz;
    const double at = (BND && !pz && k == nk - 1) ? 0.0 : cz;
    const double ap_a0 = -1.0 * (aw_a0 + ae_a0 + as + an + ab + at);
    const double ap_b0 = -1.0 * (cx + ae_b0 + as + an + ab + at);
    const double ap_a1 = -1.0 * (cx + ae_a1 + as + an + ab + at);
    const double ap_b1 = -1.0 * (cx + ae_b1 + as + an + ab + at);
    const double r_a0 = cur.fa.x - (aw_a0 * W_a0 + ae_a0 * E_a0 + as * cur.sa.x + an * cur.na.x +
                                    ab * am1.x + at * cur.ap1.x + ap_a0 * A.x);
    const double r_b0 = cur.fb.x - (cx * A.x + ae_b0 * E_b0 + as * cur.sb.x + an * cur.nb.x +
                                    ab * bm1.x + at * cur.bp1.x + ap_b0 * B.x);
    const double r_a1 = cur.fa.y - (cx * B.x + ae_a1 * E_a1 + as * cur.sa.y + an * cur.na.y +
                                    ab * am1.y + at * cur.ap1.y + ap_a1 * A.y);
    const double r_b1 = cur.fb.y - (cx * A.y + ae_b1 * E_b1 + as * cur.sb.y + an * cur.nb.y +
                                    ab * bm1.y + at * cur.bp1.y + ap_b1 * B.y);
    const int ca = (jc + k) & 1, cb = ca ^ 1;
    const unsigned q = ((unsigned)k * plane + o_c) / SZ;  // even: a pair's first entry
    // (FP64 level 1 only: the host asks for it there, and the FP32 kernel
    // stays free of it)
    if (sizeof(T) == 8 && zbuf >= 0) {
      // the level-1 relaxation from zero starts with the red cells: rhs/ap
      // (zero_state_red's arithmetic) into buffer zbuf; the red pair is a0,
      // a1 or b0, b1
      const bool red_a = ca == 0;
      const T r0 = (T)(red_a ? r_a0 : r_b0), r1 = (T)(red_a ? r_a1 : r_b1);
      const int xr = x0 + (red_a ? 0 : 1);
      const bool w0 = red_a ? ok_a0 : ok_b0, w1 = red_a ? ok_a1 : ok_b1;
      const Coef<T> c0 = cell_coef<T>(L, xr, jc, k), c1 = cell_coef<T>(L, xr + 2, jc, k);
      t2 v;
      v.x = div_ap(r0 - T(0), c0.ap, T(1) / c0.ap);
      v.y = div_ap(r1 - T(0), c1.ap, T(1) / c1.ap);
      gmem<T> *P = (gmem<T> *)L.phi[zbuf][0];
      if (w1)
        *(gmem<t2> *)(P + q) = v;
      else if (w0)
        P[q] = v.x;
    }
    if (ok_a1) {
      t2 v;
      v.x = (T)r_a0;
      v.y = (T)r_a1;
      *(gmem<t2> *)(R[ca] + q) = v;
    } else if (ok_a0) {
      R[ca][q] = (T)r_a0;
    }
    if (ok_b1) {
      t2 v;
      v.x = (T)r_b0;
      v.y = (T)r_b1;
      *(gmem<t2> *)(R[cb] + q) = v;
    } else if (ok_b0) {
      R[cb][q] = (T)r_b0;
    }
    if (ok_a0) {
      ss += r_a0 * r_a0;
      am = fmax(am, fabs(r_a0));
    }
    if (ok_b0) {
      ss += r_b0 * r_b0;
      am = fmax(am, fabs(r_b0));
    }
    if (ok_a1) {
      ss += r_a1 * r_a1;
      am = fmax(am, fabs(r_a1));
    }
    if (ok_b1) {
      ss += r_b1 * r_b1;
      am = fmax(am, fabs(r_b1));
    }
    am1 = A;
    bm1 = B;
    A = cur.ap1;
    B = cur.bp1;
  }
}

// One launch over the finest level of every block.  k_residual: tiles of KB
// planes (kind 0 y/z interior, kind 3 touching a y/z face); k_residual_gen:
// the general path for r = f (use_p = 0) and for blocks one cell wide in x
// (kind 1 tiles), in a kernel of its own so that its registers do not cost
// the main kernel occupancy.
template <class T, int KB>
__global__ void __launch_bounds__(NTHREADS)
    k_residual(const Tile *__restrict__ tiles, const FineDev *__restrict__ fine,
               const LevelDev *__restrict__ levs, const int *__restrict__ active,
               RedPartial *__restrict__ partials, int zbuf) {
  // XCD-contiguous tile ranges: rows j-1, j+1 of a tile are in the same L2
  const int ti = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const Tile t = tiles[ti];
  const FineDev &F = fine[t.lev];
  const LevelDev &L = levs[t.lev];
  double ss = 0.0, am = 0.0;
  if (active[F.blk]) {
    if (t.kind == 0)
      residual_tile_fast<T, KB, false>(t, F, L, ss, am, zbuf);
    else
      residual_tile_fast<T, KB, true>(t, F, L, ss, am, zbuf);
  }
  block_reduce(ss, am);
  if (threadIdx.x == 0 && threadIdx.y == 0) partials[ti] = RedPartial{ss, am};
}

template <class T>
__global__ void __launch_bounds__(NTHREADS)
    k_residual_gen(const Tile *__restrict__ tiles, const FineDev *__restrict__ fine,
                   const LevelDev *__restrict__ levs, const int *__restrict__ active,
                   RedPartial *__restrict__ partials, int use_p) {
  const int ti = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const Tile t = tiles[ti];
  const FineDev &F = fine[t.lev];
  const LevelDev &L = levs[t.lev];
  double ss = 0.0, am = 0.0;
  if (active[F.blk]) {
    if (t.kind == 0)
      residual_tile<T, true>(t, fine, L, use_p, ss, am);
    else
      residual_tile<T, false>(t, fine, L, use_p, ss, am);
  }
  block_reduce(ss, am);
  if (threadIdx.x == 0 && threadIdx.y == 0) partials[ti] = RedPartial{ss, am};
}

// A block's right-hand side from a dense array: f, the level-1 rhs, and the
// partial sums of ||f||, tile by tile in k_residual_gen's layout and order.
// One pass over memory: a pack and a pass over every block's tiles took 59 +
// 54 us at 256^3 (float level 1), now 63; for each of 48 blocks 4 + 16, now
// 8.5.
template <class T, int KB>
__global__ void __launch_bounds__(NTHREADS)
    k_set_rhs(const Tile *__restrict__ tiles, const FineDev *__restrict__ fine,
              const LevelDev *__restrict__ levs, const double *__restrict__ src,
              RedPartial *__restrict__ partials) {
  const int ti = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const Tile t = tiles[ti];
  const FineDev &F = fine[t.lev];
  const LevelDev &L = levs[t.lev];
  const int lpr = F.lpr, lane = (int)threadIdx.x;
  const int j = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
  const int ni = F.ni, nj = F.nj;
  gmem<double> *const F0 = (gmem<double> *)F.f[0], *const F1 = (gmem<double> *)F.f[1];
  gmem<T> *const R0 = (gmem<T> *)L.rhs[0], *const R1 = (gmem<T> *)L.rhs[1];
  const gmem<double> *const A = (const gmem<double> *)src;
  double ss = 0.0, am = 0.0;
  // every load first: a small block has few workgroups (lanes and planes
  // outside the block read a cell of it and store nothing)
  const int jc = min(j, nj - 1);
  double fa[2][KB], fb[2][KB];
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int l = min(t.x0 + half * lpr + (lane & (lpr - 1)), (ni - 1) >> 1);
#pragma unroll
    for (int p = 0; p < KB; ++p) {
      const size_t row = (size_t)((unsigned)(t.z0 + p) * (unsigned)nj + (unsigned)jc) * ni;
      fa[half][p] = A[row + 2 * l];
      fb[half][p] = A[row + min(2 * l + 1, ni - 1)];
    }
  }
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int l = t.x0 + half * lpr + (lane & (lpr - 1));
    const bool ok = 2 * l < ni && j < nj, b_ok = 2 * l + 1 < ni && j < nj;
#pragma unroll
    for (int p = 0; p < KB; ++p) {
      const int k = t.z0 + p;
      const unsigned q = ((unsigned)k * (unsigned)nj + (unsigned)j) * (unsigned)F.H + (unsigned)l;
      const double a = fa[half][p], b = fb[half][p];
      const bool ca = (j + k) & 1;
      if (ok) {
        (ca ? F1 : F0)[q] = a;
        (ca ? R1 : R0)[q] = (T)a;
        ss += a * a;
        am = fmax(am, fabs(a));
      }
      if (b_ok) {
        (ca ? F0 : F1)[q] = b;
        (ca ? R0 : R1)[q] = (T)b;
        ss += b * b;
        am = fmax(am, fabs(b));
      }
    }
  }
  block_reduce(ss, am);
  if (threadIdx.x == 0 && threadIdx.y == 0) partials[ti] = RedPartial{ss, am};
}

// p = p + (pp - ppref) with ppref = 0 (newsolv_mg.for:39-49), streamed over
// the colour arrays of one block (pad entries included: they are never read
// as cells); pp is the level-1 correction in buffer `buf`.  Tile::x0 is the
// first entry, 4 entries per thread.
template <class T>
__global__ void __launch_bounds__(NTHREADS)
    k_update(const Tile *__restrict__ tiles, const FineDev *__restrict__ fine,
             const LevelDev *__restrict__ levs, const int *__restrict__ active, int buf) {
  typedef typename Vec2<T>::type v2t;
  typedef typename Vec2<double>::type v2d;
  const Tile t = tiles[blockIdx.x];
  const FineDev &F = fine[t.lev];
  const LevelDev &L = levs[t.lev];
  if (!active[F.blk]) return;
  const unsigned n = (unsigned)F.H * (unsigned)F.nj * (unsigned)F.nk;
  const int tid = (int)(threadIdx.x + blockDim.x * threadIdx.y);
  for (int c = 0; c < 2; ++c) {
    gmem<double> *P = (gmem<double> *)F.p[c];
    const gmem<T> *Q = (const gmem<T> *)L.phi[buf][c];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned e = (unsigned)t.x0 + 2u * (unsigned)(tid + h * NTHREADS);
      if (e >= n) continue;
      const v2t pp = *(const gmem<v2t> *)(Q + e);
      v2d p = *(gmem<v2d> *)(P + e);
      p.x = p.x + ((double)pp.x - 0.0);
      p.y = p.y + ((double)pp.y - 0.0);
      *(gmem<v2d> *)(P + e) = p;
    }
  }
}

// per-block reduction of the partials of k_residual, fixed order
constexpr int FIN_THREADS = 1024;
__device__ __forceinline__ void finalize_body(const int *__restrict__ tile_begin,
                                              const RedPartial *__restrict__ partials,
                                              RedPartial *__restrict__ out) {
  const int b = blockIdx.x;
  const int t0 = tile_begin[b], t1 = tile_begin[b + 1];
  double ss = 0.0, am = 0.0;
  for (int q = t0 + (int)threadIdx.x; q < t1; q += FIN_THREADS) {
    ss += partials[q].ss;
    am = fmax(am, partials[q].amax);
  }
  __shared__ double s_ss[FIN_THREADS], s_am[FIN_THREADS];
  s_ss[threadIdx.x] = ss;
  s_am[threadIdx.x] = am;
  __syncthreads();
  for (int w = FIN_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) {
      s_ss[threadIdx.x] += s_ss[threadIdx.x + w];
      s_am[threadIdx.x] = fmax(s_am[threadIdx.x], s_am[threadIdx.x + w]);
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) out[b] = RedPartial{s_ss[0], s_am[0]};
}

__global__ void __launch_bounds__(FIN_THREADS)
    k_finalize(const int *__restrict__ tile_begin, const RedPartial *__restrict__ partials,
               RedPartial *__restrict__ out) {
  finalize_body(tile_begin, partials, out);
}

// The solve loop's stopping rule after cycle ctl->it + 1, as h3dmg_solve's
// host loop applies it (newsolv_mg.for:57-59 for the reference criterion),
// in the same order and IEEE operations: per block ||r|| = sqrt(ss), rel =
// ||r|| / ||f|| (one global rel for blocks joined by faces), rmax = amax *
// rfac * vol; done when (REF) it >= max(min_cycles, 2) and the global rmax <
// tol, else it >= min_cycles and rel <= the block's tolerance.  One wavefront,
// a lane per block (one thread for all of them waits for memory block after
// block: 48 blocks took 54 us, now 7.6); sums are taken in block order
// like the host's, the maxima do not depend on it.
__device__ __forceinline__ void decide_body(const DecideBlock *__restrict__ blocks,
                                            DecideState *__restrict__ state,
                                            DecideCtl *__restrict__ ctl,
                                            const RedPartial *__restrict__ stats,
                                            int *__restrict__ active, char *__restrict__ ring,
                                            const DecideParams *__restrict__ prm_in) {
  const DecideParams prm = *prm_in;
  const int nb = prm.nb, lane = (int)threadIdx.x;
  const int it = ctl->it + 1;
  double grel = 0.0;
  if (prm.connected) {
    double ss = 0.0, ff = 0.0;
    for (int b0 = 0; b0 < nb; b0 += 64) {
      const int b = b0 + lane;
      const bool on = b < nb && blocks[b].enabled;
      const double s = on ? stats[b].ss : 0.0, f = on ? blocks[b].fnorm * blocks[b].fnorm : 0.0;
      for (int q = 0; q < min(64, nb - b0); ++q) {
        ss += __shfl(s, q);
        ff += __shfl(f, q);
      }
    }
    grel = ff > 0 ? sqrt(ss) / sqrt(ff) : sqrt(ss);
  }
  double worst = 0.0, gmax = 0.0;
  bool bad = false;
  for (int b = lane; b < nb; b += 64) {
    const DecideBlock B = blocks[b];
    const RedPartial r = stats[b];
    DecideState s = state[b];
    const int a = active[b];
    if (!B.enabled) continue;
    const double nrm = sqrt(r.ss);
    if (a) {
      s.rel = prm.connected ? grel : B.fnorm > 0 ? nrm / B.fnorm : nrm;
      s.rmax = r.amax * prm.rfac * B.vol;
      state[b] = s;
    }
    if (!isfinite(nrm)) bad = true;
    worst = worst < s.rel ? s.rel : worst;
    gmax = gmax < s.rmax ? s.rmax : gmax;
  }
  bad = __any(bad);
  // the maxima over the lanes that have a block (the others read neither)
  for (int w = nb > 32 ? 32 : nb > 1 ? 1 << (31 - __clz(nb - 1)) : 0; w > 0; w >>= 1) {
    const double x = __shfl_xor(worst, w), g = __shfl_xor(gmax, w);
    worst = worst < x ? x : worst;
    gmax = gmax < g ? g : gmax;
  }
  char *slot = ring + (size_t)(it & 1) * decide_slot_bytes(nb);
  DecideState *rs = (DecideState *)(slot + sizeof(DecideCtl));
  RedPartial *rp = (RedPartial *)(rs + nb);
  int *ra = (int *)(rp + nb);
  bool going = false;
  for (int b = lane; b < nb; b += 64) {
    const DecideBlock B = blocks[b];
    const RedPartial r = stats[b];
    const DecideState s = state[b];
    int a = active[b];
    bool done;
    if (!B.enabled)
      done = true;
    else if (prm.ref)
      done = it >= max(prm.min_cycles, 2) && gmax < prm.tol;
    else
      done = it >= prm.min_cycles && s.rel <= B.tol;
    // a non-finite norm ends the loop: a cycle queued behind this one does
    // nothing
    if (done || bad) active[b] = a = 0;
    if (a) going = true;
    rs[b] = s;
    rp[b] = r;
    ra[b] = a;
  }
  going = __any(going);
  if (lane == 0) {
    const DecideCtl c{it, going ? 0 : 1, bad ? 1 : 0, 0, prm.ref ? gmax : worst};
    *ctl = c;
    *(DecideCtl *)slot = c;
  }
}

// k_finalize followed by the stopping rule in one launch: each block's
// workgroup writes its statistics, and the last workgroup to finish (one
// counter, reset by that workgroup for the next launch) applies the rule to
// all of them.
__global__ void __launch_bounds__(FIN_THREADS)
    k_finalize_decide(const int *__restrict__ tile_begin, const RedPartial *__restrict__ partials,
                      RedPartial *__restrict__ out, const DecideBlock *__restrict__ blocks,
                      DecideState *__restrict__ state, DecideCtl *__restrict__ ctl,
                      int *__restrict__ active, char *__restrict__ ring,
                      const DecideParams *__restrict__ prm, unsigned *__restrict__ arrived) {
  finalize_body(tile_begin, partials, out);
  if (threadIdx.x >= 64) return;
  int last = 0;
  if (threadIdx.x == 0) {
    __threadfence();  // this block's statistics before the count
    last = atomicAdd(arrived, 1u) == gridDim.x - 1;
    if (last) *arrived = 0u;
  }
  if (!__builtin_amdgcn_readfirstlane(last)) return;
  __threadfence();  // every block's statistics after it
  decide_body(blocks, state, ctl, out, active, ring, prm);
}
// ---------------------------------------------------------------------------
// Exact FP64 solve of the coarsest level of one block (extension, no
// reference counterpart): A = Dx (+) Dy (+) Dz with Dx the 1-D Neumann or
// periodic second difference; with Q_a the orthonormal eigenvectors of D_a
// (columns) and l_a its eigenvalues, u = Q (Q^T f ./ (lx+ly+lz)) with the
// zero (constant) mode dropped -- the null-space projection.  The transforms
// run along x, y, z forwards and z, y, x back, every sum in index order, on
// one of three routes with the same arithmetic in the same order: inside the
// V-cycle tail (coarse_exact_lds), in three launches over the chip
// (k_exact_plane, k_exact_cols), or one launch per transform (k_exact_pass).
template <class T>
using lds = __attribute__((address_space(3))) T;

__device__ __forceinline__ int cidx32(int H, int nj, int i, int j, int k) {
  return (k * nj + j) * H + (i >> 1);
}

// q -> (i, j, k) of an n0 x n1 x . array, by float reciprocals with one exact
// correction (q < 2^24)
__device__ __forceinline__ void split3(int q, int n0, int n1, int &i, int &j, int &k) {
  int r = (int)((float)q * (1.0f / (float)n0));
  i = q - __mul24(r, n0);
  const int a = i < 0 ? -1 : i >= n0 ? 1 : 0;
  r += a;
  i -= a * n0;
  k = (int)((float)r * (1.0f / (float)n1));
  j = r - __mul24(k, n1);
  const int b = j < 0 ? -1 : j >= n1 ? 1 : 0;
  k += b;
  j -= b * n1;
}

// The six transforms, x y z forwards, then z y x back, one code for all (the
// tail runs them once per launch: instruction fetches count).  Along an axis
// of `len` points, for every row (the other two coordinates; points vs apart)
// and index a,
//   out(a) = sum over x, in order, of Q(x, a) * V(x),
// Q(x, a) = Q[x*len + a] forwards, Q[a*len + x] back.  A thread forms RI
// indexes x RR rows of outputs and reads RI + RR operands per term: one
// output per thread reads two operands per product, and LDS reads bound the
// transforms.  The sums run in the same order whatever RI and RR.
typedef lds<double> *ldsd;
template <int RI, int RR, class dp>
__device__ __forceinline__ void coarse_exact_passes(int n0, int n1, int n2, int H, dp Q0, dp Q1,
                                                    dp Q2, dp l0, dp l1, dp l2, dp A, dp Bs, dp P0,
                                                    dp P1) {
  const int plane = n0 * n1, n = plane * n2;
  const int tid = (int)threadIdx.x, nthr = (int)blockDim.x;
#pragma clang loop unroll(disable)
  for (int p = 0; p < 6; ++p) {
    const int ax = p < 3 ? p : 5 - p;
    const bool fwd = p < 3;
    const dp Q = ax == 0 ? Q0 : ax == 1 ? Q1 : Q2;
    const dp V = (p & 1) ? Bs : A, O = (p & 1) ? A : Bs;
    const int len = ax == 0 ? n0 : ax == 1 ? n1 : n2;
    const int vs = ax == 0 ? 1 : ax == 1 ? n0 : plane;
    const int qx = fwd ? len : 1, qa = fwd ? 1 : len;
    const int nrow = n / len, nib = (len + RI - 1) / RI, nrb = (nrow + RR - 1) / RR;
#pragma clang loop unroll(disable)
    for (int t = tid; t < nib * nrb; t += nthr) {
      int q, ib, dummy;
      split3(t, nrb, nib, q, ib, dummy);
      int at[RR], ix[RI];
#pragma unroll
      for (int r = 0; r < RR; ++r) {
        // rows: (j,k) pairs, (i,k) pairs, (i,j) pairs
        const int row = min(q + r * nrb, nrow - 1);
        int i, k, z;
        split3(row, n0, n2, i, k, z);
        at[r] = ax == 0 ? row * n0 : ax == 1 ? k * plane + i : row;
      }
#pragma unroll
      for (int a = 0; a < RI; ++a) ix[a] = min(ib * RI + a, len - 1) * qa;
      double s[RI][RR];
#pragma unroll
      for (int a = 0; a < RI; ++a)
#pragma unroll
        for (int r = 0; r < RR; ++r) s[a][r] = 0.0;
#pragma unroll 4
      for (int x = 0; x < len; ++x) {
        double qv[RI], vv[RR];
#pragma unroll
        for (int a = 0; a < RI; ++a) qv[a] = Q[x * qx + ix[a]];
#pragma unroll
        for (int r = 0; r < RR; ++r) vv[r] = V[at[r] + x * vs];
#pragma unroll
        for (int a = 0; a < RI; ++a)
#pragma unroll
          for (int r = 0; r < RR; ++r) s[a][r] += qv[a] * vv[r];
      }
#pragma unroll
      for (int a = 0; a < RI; ++a)
#pragma unroll
        for (int r = 0; r < RR; ++r) {
          const int ia = ib * RI + a, o = at[r] + ia * vs;
          if (ia < len && q + r * nrb < nrow) {
            if (p == 2 || p == 5) {
              int i, j, k;
              split3(o, n0, n1, i, j, k);
              if (p == 2) {
                // mode (0,0,0) is the constant (null-space) mode of every axis
                O[o] = o == 0 ? 0.0 : s[a][r] / (l0[i] + l1[j] + l2[k]);
              } else {
                (((i + j + k) & 1) ? P1 : P0)[cidx32(H, n1, i, j, k)] = s[a][r];
              }
            } else {
              O[o] = s[a][r];
            }
          }
        }
    }
    __syncthreads();
  }
}

// Every thread of the workgroup calls it; all arrays in LDS, rhs and phi
// colour split, A and Bs scratch of n0*n1*n2.
__device__ __forceinline__ void coarse_exact_lds(int n0, int n1, int n2, int H, ldsd R0, ldsd R1,
                                                 ldsd P0, ldsd P1, ldsd Q0, ldsd Q1, ldsd Q2,
                                                 ldsd l0, ldsd l1, ldsd l2, ldsd A, ldsd Bs) {
  const int n = n0 * n1 * n2;
  // gather rhs into natural layout A[i + n0*(j + n1*k)]
  for (int q = (int)threadIdx.x; q < n; q += (int)blockDim.x) {
    int i, j, k;
    split3(q, n0, n1, i, j, k);
    A[q] = (((i + j + k) & 1) ? R1 : R0)[cidx32(H, n1, i, j, k)];
  }
  __syncthreads();
  if (n <= (int)blockDim.x)
    coarse_exact_passes<1, 1, ldsd>(n0, n1, n2, H, Q0, Q1, Q2, l0, l1, l2, A, Bs, P0, P1);
  else
    coarse_exact_passes<2, 2, ldsd>(n0, n1, n2, H, Q0, Q1, Q2, l0, l1, l2, A, Bs, P0, P1);
}

// One axis of a transform in LDS: for every row r < nrow (points rs apart)
// and index a < len, out(r, a, sum over x, in order, of Q[x*qx + a*qa] *
// V[r*rs + x*vs]).
template <int RI, int RR, class F>
__device__ __forceinline__ void exact_axis(int len, int nrow, int rs, int vs, ldsd Q, int qx,
                                           int qa, ldsd V, F &&out) {
  const int nib = (len + RI - 1) / RI, nrb = (nrow + RR - 1) / RR;
#pragma clang loop unroll(disable)
  for (int t = (int)threadIdx.x; t < nib * nrb; t += (int)blockDim.x) {
    int q, ib, dummy;
    split3(t, nrb, nib, q, ib, dummy);
    int at[RR], ix[RI];
#pragma unroll
    for (int r = 0; r < RR; ++r) at[r] = min(q + r * nrb, nrow - 1) * rs;
#pragma unroll
    for (int a = 0; a < RI; ++a) ix[a] = min(ib * RI + a, len - 1) * qa;
    double s[RI][RR];
#pragma unroll
    for (int a = 0; a < RI; ++a)
#pragma unroll
      for (int r = 0; r < RR; ++r) s[a][r] = 0.0;
#pragma unroll 4
    for (int x = 0; x < len; ++x) {
      double qv[RI], vv[RR];
#pragma unroll
      for (int a = 0; a < RI; ++a) qv[a] = Q[x * qx + ix[a]];
#pragma unroll
      for (int r = 0; r < RR; ++r) vv[r] = V[at[r] + x * vs];
#pragma unroll
      for (int a = 0; a < RI; ++a)
#pragma unroll
        for (int r = 0; r < RR; ++r) s[a][r] += qv[a] * vv[r];
    }
#pragma unroll
    for (int a = 0; a < RI; ++a)
#pragma unroll
      for (int r = 0; r < RR; ++r)
        if (ib * RI + a < len && q + r * nrb < nrow) out(q + r * nrb, ib * RI + a, s[a][r]);
  }
}

// Odd row pitch: rows of doubles then start in different LDS banks.
__host__ __device__ inline int exact_pitch(int n) { return n | 1; }
constexpr int EXACT_COLS = 16;     // z-columns per workgroup of k_exact_cols
constexpr int EXACT_SMALL = 512;   // plane cells up to which a thread forms single outputs

// x and y transforms of plane blockIdx.y of block tiles[blockIdx.x]: rhs to
// scratch 0 (FWD), or back from scratch 1 to phi.  One workgroup per block is
// bound by its LDS reads (two per product): a two-level cycle of 52x28x20 took
// 215 us, of 64^3 2783; the planes and columns over the CUs 63 and 70,
// and 4 us a launch.  Output tiles (RI x RI) read RI operands per product
// less; below EXACT_SMALL cells there are not enough of them for the threads.
template <bool FWD>
__global__ void __launch_bounds__(256)
    k_exact_plane(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                  const int *__restrict__ active, const double *const *__restrict__ eig_q,
                  double *const *__restrict__ scratch, int buf) {
  extern __shared__ __align__(16) char smem[];
  const Tile t = tiles[blockIdx.x];  // lev = coarsest descriptor, x0 = block
  const int b = t.x0, k = (int)blockIdx.y;
  const LevelDev &L = levs[t.lev];
  const int n0 = L.ni, n1 = L.nj;
  if (!active[b] || k >= L.nk) return;
  const int p0 = exact_pitch(n0), p1 = exact_pitch(n1), plane = n0 * n1;
  const ldsd Q0 = (ldsd)smem, Q1 = Q0 + n0 * p0, V = Q1 + n1 * p1, W = V + p0 * n1;
  const int tid = (int)threadIdx.x;
  auto table = [&](ldsd Q, const double *g, int n, int p) {
    for (int e = tid; e < n * n; e += 256) {
      int i, j, z;
      split3(e, n, n, i, j, z);
      Q[j * p + i] = g[e];
    }
  };
  table(Q0, eig_q[3 * b], n0, p0);
  table(Q1, eig_q[3 * b + 1], n1, p1);
  const double *R[2] = {(const double *)L.rhs[0], (const double *)L.rhs[1]};
  double *P[2] = {(double *)L.phi[buf][0], (double *)L.phi[buf][1]};
  double *const A = scratch[2 * b] + (size_t)k * plane;
  const double *const B = scratch[2 * b + 1] + (size_t)k * plane;
  const size_t row0 = (size_t)k * n1;
  auto cell = [&](int i, int j) { return (row0 + j) * L.H + (i >> 1); };
  for (int e = tid; e < plane; e += 256) {
    int i, j, z;
    split3(e, n0, n1, i, j, z);
    V[j * p0 + i] = FWD ? (((i + j + k) & 1) ? R[1] : R[0])[cell(i, j)] : B[e];
  }
  __syncthreads();
  auto mid = [&](int r, int a, double s) { W[FWD ? r * p0 + a : a * p0 + r] = s; };
  auto end = [&](int r, int a, double s) {
    if (FWD)
      A[a * n0 + r] = s;
    else
      (((r + a + k) & 1) ? P[1] : P[0])[cell(a, r)] = s;
  };
  auto run = [&](auto ri) __attribute__((always_inline)) {
    constexpr int RI = decltype(ri)::value;
    if (FWD) {
      exact_axis<RI, RI>(n0, n1, p0, 1, Q0, p0, 1, V, mid);  // rows j
      __syncthreads();
      exact_axis<RI, RI>(n1, n0, 1, p0, Q1, p1, 1, W, end);  // rows i
    } else {
      exact_axis<RI, RI>(n1, n0, 1, p0, Q1, 1, p1, V, mid);
      __syncthreads();
      exact_axis<RI, RI>(n0, n1, p0, 1, Q0, 1, p0, W, end);
    }
  };
  if (plane <= EXACT_SMALL)
    run(std::integral_constant<int, 1>());
  else
    run(std::integral_constant<int, 2>());
}

// z transform, division by the eigenvalues and z transform back of
// EXACT_COLS columns: scratch 0 to scratch 1
__global__ void __launch_bounds__(256)
    k_exact_cols(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                 const int *__restrict__ active, const double *const *__restrict__ eig_q,
                 const double *const *__restrict__ eig_l, double *const *__restrict__ scratch) {
  extern __shared__ __align__(16) char smem[];
  const Tile t = tiles[blockIdx.x];
  const int b = t.x0;
  const LevelDev &L = levs[t.lev];
  const int n0 = L.ni, n2 = L.nk, plane = n0 * L.nj, c0 = (int)blockIdx.y * EXACT_COLS;
  if (!active[b] || c0 >= plane) return;
  const int p2 = exact_pitch(n2), nc = min(EXACT_COLS, plane - c0);
  const ldsd Q2 = (ldsd)smem, V = Q2 + n2 * p2, W = V + n2 * EXACT_COLS,
             lxy = W + n2 * EXACT_COLS, lz = lxy + EXACT_COLS;
  const int tid = (int)threadIdx.x;
  for (int e = tid; e < n2 * n2; e += 256) {
    int i, j, z;
    split3(e, n2, n2, i, j, z);
    Q2[j * p2 + i] = eig_q[3 * b + 2][e];
  }
  const double *const A = scratch[2 * b] + c0;
  for (int e = tid; e < n2 * EXACT_COLS; e += 256) {
    const int k = e / EXACT_COLS, c = e % EXACT_COLS;
    if (c < nc) V[e] = A[(size_t)k * plane + c];
  }
  if (tid < nc) {
    const int j = (c0 + tid) / n0, i = (c0 + tid) - j * n0;
    lxy[tid] = eig_l[3 * b][i] + eig_l[3 * b + 1][j];
  }
  for (int e = tid; e < n2; e += 256) lz[e] = eig_l[3 * b + 2][e];
  __syncthreads();
  exact_axis<1, 1>(n2, nc, 1, EXACT_COLS, Q2, p2, 1, V, [&](int r, int a, double s) {
    // mode (0,0,0) is the constant (null-space) mode of every axis
    W[a * EXACT_COLS + r] = (c0 + r == 0 && a == 0) ? 0.0 : s / (lxy[r] + lz[a]);
  });
  __syncthreads();
  double *const B = scratch[2 * b + 1] + c0;
  exact_axis<1, 1>(n2, nc, 1, EXACT_COLS, Q2, 1, p2, W,
                   [&](int r, int a, double s) { B[(size_t)a * plane + r] = s; });
}

// Any size: transform `pass` of the six, a thread per output.
__global__ void __launch_bounds__(256)
    k_exact_pass(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                 const int *__restrict__ active, const double *const *__restrict__ eig_q,
                 const double *const *__restrict__ eig_l, double *const *__restrict__ scratch,
                 int buf, int pass) {
  const Tile t = tiles[blockIdx.x];
  const int b = t.x0;
  if (!active[b]) return;
  const LevelDev &L = levs[t.lev];
  const int ax = pass < 3 ? pass : 5 - pass;
  const bool fwd = pass < 3;
  const int n0 = L.ni, n1 = L.nj, n2 = L.nk, len = ax == 0 ? n0 : ax == 1 ? n1 : n2;
  const size_t plane = (size_t)n0 * n1, n = plane * n2;
  const size_t vs = ax == 0 ? 1 : ax == 1 ? (size_t)n0 : plane;
  const double *const Q = eig_q[3 * b + ax];
  const double *const V = scratch[2 * b + (pass & 1)];
  double *const O = scratch[2 * b + 1 - (pass & 1)];
  for (size_t q = (size_t)blockIdx.y * 256 + threadIdx.x; q < n; q += (size_t)gridDim.y * 256) {
    const int i = (int)(q % n0), j = (int)((q / n0) % n1), k = (int)(q / plane);
    const int a = ax == 0 ? i : ax == 1 ? j : k;
    const size_t base = q - a * vs;
    double s = 0.0;
    if (pass == 0) {
      const size_t row = ((size_t)k * n1 + j) * L.H;
      for (int x = 0; x < len; ++x)
        s += Q[(size_t)x * len + a] * ((const double *)L.rhs[(x + j + k) & 1])[row + (x >> 1)];
    } else {
      const size_t qx = fwd ? len : 1, qa = fwd ? 1 : len;
      for (int x = 0; x < len; ++x) s += Q[x * qx + a * qa] * V[base + x * vs];
    }
    if (pass == 2)
      O[q] = q == 0 ? 0.0 : s / (eig_l[3 * b][i] + eig_l[3 * b + 1][j] + eig_l[3 * b + 2][k]);
    else if (pass == 5)
      ((double *)L.phi[buf][(i + j + k) & 1])[((size_t)k * n1 + j) * L.H + (i >> 1)] = s;
    else
      O[q] = s;
  }
}

// ---------------------------------------------------------------------------
// V-cycle tail: one workgroup per block runs every level from the tail level
// Lt down to the block's coarsest and back up (mgkcyc, mgsolver.for:272-352,
// restricted to levels >= Lt) entirely in LDS: pre-smoothing, restriction,
// the coarsest treatment, prolongation and post-smoothing, separated by
// workgroup barriers.  Small levels are latency-bound: one launch, LDS
// latency and on-chip barriers replace ~3 full-chip launches per level.
//
// Every cell's value is the expression of the per-level kernels, in the same
// order; a wall's term is the product with zero, where they multiply zero by
// the cell's own value before the sweep: NaN where that is not finite, so a
// run whose result is not finite is done again that way (tail_relax_walls).
// The tail's one CU is bound
// by instruction issue and, since it runs every piece of code a few times
// only, by instruction fetches: a thread sets up its entries once per visit
// of a level (TailCells) and the neighbours then lie constant steps away; no
// piece is unrolled over levels, sweeps or colours.
//
// LDS per level: four phi arrays [buffer][colour] and two rhs arrays in the
// global layout (colour split, pitch H), and between them a zero, the value
// behind every wall.  In: the top level's rhs (global).
// Out: the top level's phi in buffer (nu1+nu2)&1 (global), the buffer every
// level ends in on the host side.  The tile's `lev` is the block's level-Lt
// descriptor.  Levels are float in a mixed-precision handle except the
// coarsest (double).
constexpr int TAIL_U = TAIL_FAST_ENTRIES / TAIL_THREADS;  // entries a thread keeps per colour

// bytes of one array of a level in LDS
__host__ __device__ inline size_t tail_phi_bytes(size_t entries, size_t word) {
  return (entries * word + 15) & ~(size_t)15;
}

// a level's geometry and its arrays' byte offsets in dynamic LDS
struct TailLev {
  int ni, nj, nk, H, per, n;  // n: entries per colour array
  unsigned phi, ps, rhs, rs;  // first phi / rhs array and the step between arrays
  double cx, cy, cz;
};

// Level q (of nl) of the tail of a block whose top level is G, in scalar
// registers: cells halve from level to level, and 1/h^2 with h doubled is a
// quarter, exactly (a power of two).  The levels' arrays follow one another.
__device__ __forceinline__ double uniform(double v) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(b & 0xffffffffll));
  const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
template <bool MIXED>
__device__ __forceinline__ TailLev tail_level(const LevelDev &G, int q, int nl) {
  unsigned off = 0;
  TailLev L;
  for (int p = 0; p <= q; ++p) {
    const unsigned word = !MIXED || p == nl - 1 ? 8u : 4u;
    L.ni = G.ni >> p;
    L.nj = G.nj >> p;
    L.nk = G.nk >> p;
    L.H = (((L.ni + 1) / 2) + 1) & ~1;
    L.n = L.H * L.nj * L.nk;
    L.phi = off;
    L.ps = (unsigned)tail_phi_bytes((size_t)L.n, word);
    L.rhs = L.phi + 4 * L.ps + 16;  // (a zero slot after the phi arrays)
    L.rs = ((unsigned)L.n * word + 15u) & ~15u;
    off = L.rhs + 2 * L.rs;
  }
  const double s = 1.0 / (double)(1ull << (2 * q));
  L.per = G.per;
  L.cx = uniform(G.cx * s);
  L.cy = uniform(G.cy * s);
  L.cz = uniform(G.cz * s);
  return L;
}
// the first byte after a level's arrays
__device__ __forceinline__ unsigned tail_end(const TailLev &L) { return L.rhs + 2 * L.rs; }

// entry e -> (pair m, row j, plane k), by float reciprocals with one exact
// correction (n < 2^24)
struct TailSplit {
  int H, nj;
  float iH, iJ;
  __device__ explicit TailSplit(const TailLev &L)
      : H(L.H), nj(L.nj), iH(1.0f / (float)L.H), iJ(1.0f / (float)L.nj) {}
  __device__ __forceinline__ void operator()(int e, int &m, int &j, int &k) const {
    int r = (int)((float)e * iH);
    m = e - __mul24(r, H);
    const int a = m < 0 ? -1 : m >= H ? 1 : 0;
    r += a;
    m -= a * H;
    k = (int)((float)r * iJ);
    j = r - __mul24(k, nj);
    const int b = j < 0 ? -1 : j >= nj ? 1 : 0;
    k += b;
    j -= b * nj;
  }
};

template <class T>
__device__ __forceinline__ T tail_ld(unsigned off) {
  extern __shared__ __align__(16) char smem[];
  return *(const lds<T> *)((const lds<char> *)smem + off);
}
template <class T>
__device__ __forceinline__ void tail_st(unsigned off, T v) {
  extern __shared__ __align__(16) char smem[];
  *(lds<T> *)((lds<char> *)smem + off) = v;
}

// What a thread keeps of its entries tid + u*TAIL_THREADS of a level (from
// `first` on) while the level is swept: the entry's byte offset, the faces its
// cells touch, and each colour's ap and divisor.
template <class T>
struct TailDiv;
template <>
struct TailDiv<float> {  // FP32 multiplies by 1/ap (div_ap)
  float a, inv;
  __device__ __forceinline__ void set(float ap) {
    a = ap;
    inv = 1.0f / ap;
  }
  __device__ __forceinline__ float operator()(float num) const { return num * inv; }
};
template <>
struct TailDiv<double> {  // FP64 divides by ap, correctly rounded (div_by)
  double a, inv;
  __device__ __forceinline__ void set(double ap) {
    a = ap;
    inv = 1.0 / ap;
  }
  __device__ __forceinline__ double operator()(double num) const {
    return div_by(num, Divisor{a, inv, divisor_fast(a)});
  }
};

template <class T>
struct TailCells {
  // Byte offsets of the six neighbours while buffer 0 / 1 is being swept.
  // Inside the level they lie a constant step away in the other colour
  // (before the sweep for a red cell, after it for a black one); across a
  // periodic face their image does in the swept buffer, its colour fixed by
  // the axis' parity; across a wall it is the level's zero slot.
  unsigned a[TAIL_U][2][2][6];
  unsigned o[TAIL_U];  // entry * sizeof(T)
  bool in[TAIL_U];     // a valid entry
  bool wave, two;      // (uniform) the wave has entries; the second ones exist
  TailDiv<T> div[TAIL_U][2];

  __device__ __forceinline__ void set(const TailLev &L, int first) {
    constexpr unsigned SZ = sizeof(T);
    const TailSplit split(L);
    const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
    const unsigned row = (unsigned)L.H * SZ, plane = row * (unsigned)L.nj;
    const unsigned span = plane * (unsigned)(L.nk - 1), zero = L.phi + 4 * L.ps;
    const unsigned xl = (unsigned)((L.ni - 1) >> 1) * SZ;  // entry of cell ni-1 in its row
    const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
    const int w0 = __builtin_amdgcn_readfirstlane(first + (int)threadIdx.x);
    wave = w0 < L.n;
    two = w0 + TAIL_THREADS < L.n;
    static_assert(TAIL_U == 2, "two entries per thread");
#pragma unroll
    for (int u = 0; u < TAIL_U; ++u) {
      const int e0 = first + (int)threadIdx.x + u * TAIL_THREADS;
      in[u] = e0 < L.n;
      if (u ? !two : !wave) continue;
      const int q = min(e0, L.n - 1);  // lanes past the end read a valid entry
      int m, j, k;
      split(q, m, j, k);
      o[u] = (unsigned)q * SZ;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int sx = (c + j + k) & 1, i = 2 * m + sx;
        const bool fw = i == 0, fe = i == L.ni - 1, fs = j == 0, fn = j == L.nj - 1, fb = k == 0,
                   ft = k == L.nk - 1;
        const T aw = (!px && fw) ? T(0) : cx, ae = (!px && fe) ? T(0) : cx;
        const T as = (!py && fs) ? T(0) : cy, an = (!py && fn) ? T(0) : cy;
        const T ab = (!pz && fb) ? T(0) : cz, at = (!pz && ft) ? T(0) : cz;
        div[u][c].set(T(-1) * (aw + ae + as + an + ab + at));
        const unsigned gx = o[u] + L.phi + (unsigned)((c + L.ni - 1) & 1) * L.ps,
                       gy = o[u] + L.phi + (unsigned)((c + L.nj - 1) & 1) * L.ps,
                       gz = o[u] + L.phi + (unsigned)((c + L.nk - 1) & 1) * L.ps;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const unsigned g = (unsigned)(2 * b) * L.ps;
          const unsigned in0 =
              o[u] + L.phi + (unsigned)(2 * (c ? 1 - b : b) + (1 - c)) * L.ps;
          unsigned(&x)[6] = a[u][c][b];
          x[0] = fw ? (px ? gx + g + xl : zero) : in0 - (sx ? 0u : SZ);
          x[1] = fe ? (px ? gx + g - xl : zero) : in0 + (sx ? SZ : 0u);
          x[2] = fs ? (py ? gy + g + (plane - row) : zero) : in0 - row;
          x[3] = fn ? (py ? gy + g - (plane - row) : zero) : in0 + row;
          x[4] = fb ? (pz ? gz + g + span : zero) : in0 - plane;
          x[5] = ft ? (pz ? gz + g - span : zero) : in0 + plane;
        }
      }
    }
  }

  // One colour half-sweep from buffer SRC; skip: every neighbour is zero.
  template <int C, int SRC>
  __device__ __forceinline__ void half(const TailLev &L, bool skip) const {
    const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
    const unsigned rb = L.rhs + (unsigned)C * L.rs,
                   ob = L.phi + (unsigned)(2 * (1 - SRC) + C) * L.ps;
    auto one = [&](int u) __attribute__((always_inline)) {
      T v[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) v[f] = tail_ld<T>(a[u][C][SRC][f]);
      const T r = tail_ld<T>(rb + o[u]);
      const T q = cx * v[0] + cx * v[1] + cy * v[2] + cy * v[3] + cz * v[4] + cz * v[5];
      return div[u][C](r - (C == 0 && skip ? T(0) : q));
    };
    if (two) {
      const T x0 = one(0), x1 = one(1);
      tail_st<T>(ob + o[0], x0);
      if (in[1]) tail_st<T>(ob + o[1], x1);
    } else if (wave) {
      const T x0 = one(0);
      if (in[0]) tail_st<T>(ob + o[0], x0);
    }
    __syncthreads();
  }

  // the residual of both colours' cells from buffer `buf` into the other (a
  // black cell's interior neighbours in `buf` are those of a sweep from the
  // other buffer)
  __device__ __forceinline__ void residual(const TailLev &L, int buf) const {
    const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
    const unsigned border = L.phi + 2 * L.ps, zero = L.phi + 4 * L.ps;
#pragma unroll
    for (int u = 0; u < TAIL_U; ++u) {
      if (u ? !two : !wave) continue;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const unsigned p = L.phi + (unsigned)(2 * buf + c) * L.ps + o[u];
        T v[6];
#pragma unroll
        for (int f = 0; f < 6; ++f) {
          const unsigned x0 = a[u][c][0][f], x1 = a[u][c][1][f];
          v[f] = tail_ld<T>((x0 >= border) == (buf != 0) || x0 == zero ? x0 : x1);
        }
        const T P = tail_ld<T>(p), r = tail_ld<T>(L.rhs + (unsigned)c * L.rs + o[u]);
        const T res = r - (cx * v[0] + cx * v[1] + cy * v[2] + cy * v[3] + cz * v[4] +
                           cz * v[5] + div[u][c].a * P);
        if (in[u]) tail_st<T>(L.phi + (unsigned)(2 * (1 - buf) + c) * L.ps + o[u], res);
      }
    }
    __syncthreads();
  }

  __device__ __forceinline__ void half_any(const TailLev &L, int c, int src, bool skip) const {
    if (src == 0) {
      if (c == 0)
        half<0, 0>(L, skip);
      else
        half<1, 0>(L, false);
    } else {
      if (c == 0)
        half<0, 1>(L, skip);
      else
        half<1, 1>(L, false);
    }
  }
};

template <class T>
__device__ __forceinline__ void tail_fill_zero(const TailLev &L, int buf) {
  for (int e = (int)threadIdx.x; e < L.n; e += TAIL_THREADS)
    for (int c = 0; c < 2; ++c)
      tail_st<T>(L.phi + (unsigned)(2 * buf + c) * L.ps + (unsigned)e * (unsigned)sizeof(T), T(0));
  __syncthreads();
}

// tail_relax with every wall's term as the per-level kernels have it, cell by
// cell
template <class T>
__device__ __forceinline__ void tail_relax_walls(const TailLev &L, int nsweep, int &buf, bool zero,
                                                 bool resid) {
  if (zero) tail_fill_zero<T>(L, buf);
  const TailSplit split(L);
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  const T cx = (T)L.cx, cy = (T)L.cy, cz = (T)L.cz;
  auto at = [&](int b, int c, unsigned e) {
    return L.phi + (unsigned)(2 * b + c) * L.ps + e * (unsigned)sizeof(T);
  };
#pragma clang loop unroll(disable)
  for (int h = 0; h < 2 * nsweep + (resid ? 2 : 0); ++h) {
    const int c = h & 1;
    const bool res = h >= 2 * nsweep;
#pragma clang loop unroll(disable)
    for (int e = (int)threadIdx.x; e < L.n; e += TAIL_THREADS) {
      int m, j, k;
      split(e, m, j, k);
      const int i = 2 * m + ((c + j + k) & 1);
      if (i >= L.ni) continue;
      // a neighbour inside the level: the other colour, for a black cell after
      // the red half (a residual reads one buffer only); else its image
      auto val = [&](int x, int y, int z, bool ghost) -> T {
        x = image(x, L.ni, px);
        y = image(y, L.nj, py);
        z = image(z, L.nk, pz);
        const int b = !ghost && !res && c ? 1 - buf : buf;
        return tail_ld<T>(at(b, (x + y + z) & 1, (unsigned)cidx32(L.H, L.nj, x, y, z)));
      };
      const T W = val(i - 1, j, k, i == 0), E = val(i + 1, j, k, i == L.ni - 1);
      const T S = val(i, j - 1, k, j == 0), N = val(i, j + 1, k, j == L.nj - 1);
      const T B = val(i, j, k - 1, k == 0), U = val(i, j, k + 1, k == L.nk - 1);
      const T aw = (!px && i == 0) ? T(0) : cx, ae = (!px && i == L.ni - 1) ? T(0) : cx;
      const T as = (!py && j == 0) ? T(0) : cy, an = (!py && j == L.nj - 1) ? T(0) : cy;
      const T ab = (!pz && k == 0) ? T(0) : cz, au = (!pz && k == L.nk - 1) ? T(0) : cz;
      const T ap = T(-1) * (aw + ae + as + an + ab + au);
      const T r = tail_ld<T>(L.rhs + (unsigned)c * L.rs + (unsigned)e * (unsigned)sizeof(T));
      const T sum = aw * W + ae * E + as * S + an * N + ab * B + au * U;
      const T P = res ? tail_ld<T>(at(buf, c, (unsigned)e)) : T(0);
      tail_st<T>(at(1 - buf, c, (unsigned)e),
                 res ? r - (sum + ap * P) : div_ap(r - sum, ap, T(1) / ap));
    }
    __syncthreads();
    if (!res) buf ^= c;
  }
}

// nsweep sweeps of a level from buffer `buf` (zero: it starts from zeros,
// filled in here) and, with resid, the residual into the free buffer.  Levels
// of more than TAIL_U*TAIL_THREADS entries set their cells anew in every
// pass.
template <class T>
__device__ __forceinline__ void tail_relax(const TailLev &L, int nsweep, int &buf, bool zero,
                                           bool resid, bool walls) {
  if (__builtin_expect(walls, 0)) {
    tail_relax_walls<T>(L, nsweep, buf, zero, resid);
    return;
  }
  if (zero) {  // (the level's first visit: on the way up the zero slot is set)
    if (threadIdx.x == 0) tail_st<T>(L.phi + 4 * L.ps, T(0));
    tail_fill_zero<T>(L, buf);
  }
  TailCells<T> W;
  if (L.n <= TAIL_U * TAIL_THREADS) {
    W.set(L, 0);
#pragma clang loop unroll(disable)
    for (int h = 0; h < 2 * nsweep; ++h) {
      W.half_any(L, h & 1, buf, zero && h == 0);
      buf ^= h & 1;
    }
    if (resid) W.residual(L, buf);
    return;
  }
#pragma clang loop unroll(disable)
  for (int h = 0; h < 2 * nsweep + (resid ? 1 : 0); ++h) {
#pragma clang loop unroll(disable)
    for (int q = 0; q < L.n; q += TAIL_U * TAIL_THREADS) {
      W.set(L, q);
      if (h < 2 * nsweep)
        W.half_any(L, h & 1, buf, zero && h == 0);
      else
        W.residual(L, buf);
    }
    if (h < 2 * nsweep) buf ^= h & 1;
  }
}

// mgrestr: the 8-child sums (i fastest, then j, then k) of the residual in
// buffer 1-buf, times 0.125
template <class Tf, class Tc>
__device__ __forceinline__ void tail_sum8(const TailLev &F, const TailLev &C, int buf) {
  const TailSplit split(C);
  constexpr unsigned SZ = sizeof(Tf);
  const unsigned row = (unsigned)F.H * SZ, plane = row * (unsigned)F.nj;
  const unsigned base = F.phi + (unsigned)(2 * (1 - buf)) * F.ps;
  for (int q0 = (int)threadIdx.x; q0 < 2 * C.n; q0 += TAIL_THREADS) {
    const int c = q0 >= C.n, e = q0 - (c ? C.n : 0);
    int m, j, k;
    split(e, m, j, k);
    const int i = 2 * m + ((c + j + k) & 1);
    if (i >= C.ni) continue;
    // child (2i + q0, 2j + q1, 2k + q2): entry i of its row, colour the
    // parity of q0 + q1 + q2
    const unsigned o = base + __umul24(2 * k, plane) + __umul24(2 * j, row) + (unsigned)i * SZ;
    Tf r[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      r[q] = tail_ld<Tf>(o + ((q >> 1) & 1 ? row : 0u) + (q >> 2 ? plane : 0u) +
                         (((q & 1) + ((q >> 1) & 1) + (q >> 2)) & 1 ? F.ps : 0u));
    Tc acc = (Tc)r[0];
#pragma unroll
    for (int q = 1; q < 8; ++q) acc = acc + (Tc)r[q];
    tail_st<Tc>(C.rhs + (unsigned)c * C.rs + (unsigned)e * (unsigned)sizeof(Tc), Tc(0.125) * acc);
  }
  __syncthreads();
}

// mgcorr for the two cells 2m, 2m+1 of an entry (the arithmetic of
// k_prolong): they share the coarse corners x = m-1, m, m+1 of coarse row
// pair (j+1)>>1 and plane pair (k+1)>>1
template <class Tf, class Tc>
__device__ __forceinline__ void tail_prolong(const TailLev &F, const TailLev &C, int src_f,
                                             int src_c) {
  const TailSplit split(F);
  const bool px = C.per & 1, py = C.per & 2, pz = C.per & 4;
  for (int e = (int)threadIdx.x; e < F.n; e += TAIL_THREADS) {
    int m, j, k;
    split(e, m, j, k);
    if (2 * m >= F.ni) continue;
    const int mj = (j + 1) >> 1, dj = (j + 1) & 1, mk = (k + 1) >> 1, dk = (k + 1) & 1;
    int xc[3], yc[2], zc[2];
#pragma unroll
    for (int a = 0; a < 3; ++a) xc[a] = image(m - 1 + a, C.ni, px);
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      yc[a] = image(mj - 1 + a, C.nj, py);
      zc[a] = image(mk - 1 + a, C.nk, pz);
    }
    Tc cv[3][2][2];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int row = __mul24(__mul24(zc[c], C.nj) + yc[b], C.H);
#pragma unroll
        for (int a = 0; a < 3; ++a)
          cv[a][b][c] = tail_ld<Tc>(C.phi +
                                    (unsigned)(2 * src_c + ((xc[a] + yc[b] + zc[c]) & 1)) * C.ps +
                                    (unsigned)(row + (xc[a] >> 1)) * (unsigned)sizeof(Tc));
      }
#pragma unroll
    for (int d = 0; d < 2; ++d) {  // cell 2m+d; ni is even above the coarsest level
      const int di = 1 - d;
      Tc s = Tc(0);
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int oi = q >> 2, oj = q & 1, ok = (q >> 1) & 1;
        const Tc w = (oi == di ? Tc(3) : Tc(1)) * (oj == dj ? Tc(3) : Tc(1)) *
                     (ok == dk ? Tc(3) : Tc(1));
        const Tc v = cv[d + oi][oj][ok];
        s = (q == 0) ? w * v : s + w * v;
      }
      const unsigned o = F.phi + (unsigned)(2 * src_f + ((d + j + k) & 1)) * F.ps +
                         (unsigned)e * (unsigned)sizeof(Tf);
      tail_st<Tf>(o, tail_ld<Tf>(o) + (Tf)(s / Tc(64)));
    }
  }
  __syncthreads();
}

template <class D, class S>
__device__ __forceinline__ void tail_copy(D *dst, const S *src, int n) {
  for (int e = (int)threadIdx.x; e < n; e += TAIL_THREADS) dst[e] = src[e];
}

// the exact solve's tables as the block's region holds them: per axis of n
// points Q (n x n) and lambda (n), each 256-byte aligned
__host__ __device__ inline unsigned tail_eig_q(int n) {
  return ((unsigned)(n * n) * 8u + 255u) & ~255u;
}
__host__ __device__ inline unsigned tail_eig_axis(int n) {
  return tail_eig_q(n) + (((unsigned)n * 8u + 255u) & ~255u);
}
__host__ __device__ inline unsigned tail_eig_bytes(int ni, int nj, int nk) {
  return tail_eig_axis(ni) + tail_eig_axis(nj) + tail_eig_axis(nk);
}

// A barrier that waits for the wave's LDS
// accesses only (the loads and stores of global memory in flight stay so)
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// EX: mixed precision with the exact coarsest solve (its blocks have two
// levels or more): no FP64 sweeps in the kernel.  A second copy of the sweeps
// makes registers spill (51; none with one copy): us a cycle, 32^3 of 4 levels,
// 74.0 with both copies, now 69.9; FP64, whose coarsest level shares the copy
// of the others, 79.1 and 77.1.
template <bool MIXED, bool EX>
__global__ void __launch_bounds__(TAIL_THREADS)
    k_vtail(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
            const int *__restrict__ active, const double *const *__restrict__ eig_q,
            const double *const *__restrict__ eig_l, int nu1, int nu2, int exact) {
  extern __shared__ __align__(16) char smem[];
  __shared__ int bad;
  const Tile t = tiles[blockIdx.x];
  const int nl = t.z1;  // the block's levels from the tail level down
  const LevelDev &G = levs[t.lev];
  const int blk = G.blk;
  if (!active[blk]) return;
  typedef typename std::conditional<MIXED, float, double>::type T;  // above the coarsest level
  const int fin = (nu1 + nu2) & 1;
  const int last = nl - 1;
  const int tid = (int)threadIdx.x;
  const TailLev L0 = tail_level<MIXED>(G, 0, nl), Z = tail_level<MIXED>(G, last, nl);
  // as the host: not for a 1-level block
  const bool do_exact = MIXED ? EX : exact && (nl > 1 || G.finer >= 0);
  // the exact solve's tables (Q and lambda of each axis, one contiguous image
  // in the block's region, each part 256-byte aligned) and scratch follow the
  // levels
  unsigned eo = tail_end(Z);
  const gmem<char> *const eg = (const gmem<char> *)(do_exact ? eig_q[3 * blk] : nullptr);
  if (do_exact) {
    const unsigned bytes = tail_eig_bytes(Z.ni, Z.nj, Z.nk);
    for (unsigned e = (unsigned)tid * 8u; e < bytes; e += TAIL_THREADS * 8u)
      tail_st<double>(eo + e, *(const gmem<double> *)(eg + e));
  }
  if (tid == 0) bad = 0;
  // the top level's rhs into LDS; its phi starts from zero
  const bool top64 = !MIXED || nl == 1;
  for (int c = 0; c < 2; ++c) {
    if (top64)
      tail_copy((lds<double> *)(smem + L0.rhs + c * L0.rs), (const gmem<double> *)G.rhs[c], L0.n);
    else
      tail_copy((lds<float> *)(smem + L0.rhs + c * L0.rs), (const gmem<float> *)G.rhs[c], L0.n);
  }
  __syncthreads();
  // the top level's phi (buffer fin) back to global; `bad` when a cell of it
  // is not finite
  auto write_top = [&](auto zero) __attribute__((always_inline)) {
    typedef decltype(zero) S;
    for (int c = 0; c < 2; ++c) {
      const unsigned o = L0.phi + (unsigned)(2 * fin + c) * L0.ps;
      gmem<S> *const out = (gmem<S> *)G.phi[fin][c];
      for (int e = tid; e < L0.n; e += TAIL_THREADS) {
        const S v = tail_ld<S>(o + (unsigned)e * (unsigned)sizeof(S));
        out[e] = v;
        if (__builtin_expect(!isfinite(v), 0)) {
          int m, j, k;
          TailSplit{L0}(e, m, j, k);
          if (2 * m + ((c + j + k) & 1) < L0.ni) bad = 1;  // (not a pad entry)
        }
      }
    }
  };
  // the coarsest level's exact solve
  auto coarsest_exact = [&]() __attribute__((always_inline)) {
    const TailLev &L = Z;
    const unsigned q1 = eo + tail_eig_axis(L.ni), q2 = q1 + tail_eig_axis(L.nj),
                   sc = q2 + tail_eig_axis(L.nk), n3 = (unsigned)(L.ni * L.nj * L.nk) * 8u;
    auto at = [&](unsigned o) { return (ldsd)((lds<char> *)smem + o); };
    coarse_exact_lds(L.ni, L.nj, L.nk, L.H, at(L.rhs), at(L.rhs + L.rs),
                     at(L.phi + (unsigned)(2 * fin) * L.ps),
                     at(L.phi + (unsigned)(2 * fin + 1) * L.ps), at(eo), at(q1), at(q2),
                     at(eo + tail_eig_q(L.ni)), at(q1 + tail_eig_q(L.nj)),
                     at(q2 + tail_eig_q(L.nk)), at(sc), at(sc + n3));
  };
  bool walls = false;
  // One copy of every piece of code, run level by level: the kernel runs each
  // only a few times per launch, and its instruction fetches count (a cold
  // kilobyte of code costs ~0.8 us here).
#pragma clang loop unroll(disable)
  for (;;) {
#pragma clang loop unroll(disable)
    for (int q = 0, up = 0; q >= 0; up ? --q : ++q) {
      // one level on the way down (up = 0) or up; the coarsest (always FP64)
      // turns around
      const bool bottom = q == last;
      if (bottom && (do_exact || MIXED)) {
        int buf = 0;
        if (do_exact)
          coarsest_exact();
        else
          tail_relax<double>(Z, nu1 + nu2, buf, true, false, walls);
        up = 1;
        continue;
      }
      const TailLev L = tail_level<MIXED>(G, q, nl), C = tail_level<MIXED>(G, q + 1, nl);
      const bool c64 = !MIXED || q + 1 == last;
      int buf = up ? nu1 & 1 : 0;
      if (up) {
        if (c64)
          tail_prolong<T, double>(L, C, buf, fin);
        else
          tail_prolong<T, T>(L, C, buf, fin);
      }
      tail_relax<T>(L, bottom ? nu1 + nu2 : up ? nu2 : nu1, buf, !up, !up && !bottom, walls);
      if (!up && !bottom) {
        if (c64)
          tail_sum8<T, double>(L, C, buf);
        else
          tail_sum8<T, T>(L, C, buf);
      }
      if (bottom) up = 1;
    }
    if (top64)
      write_top(0.0);
    else
      write_top(0.0f);
    // An infinity or NaN stays in a level once a black cell has it, and goes
    // up with the corrections: a finite result has met none, and zero was
    // every wall's term.
    lds_barrier();
    if (__builtin_expect(walls || !bad, 1)) break;
    walls = true;
  }
}

// ---------------------------------------------------------------------------
// Variable-density operator (coeff under L_LSM, mgsolver.for:72-184).  The
// reference builds, per level, dens_mg (the density of the level's cells:
// the input at level 1, the 8-child average below) and from it per-cell
// coefficients in finite-volume form with the FINEST spacing at every level:
//   aw = dy*dz/dx/dens(i-1/2),  dens(i-1/2) = 0.5*(dens(i) + dens(i-1)), or
//   dens(i) on the block's first cell; likewise ae, as, an, ab, at; zero
//   towards a wall; ap = -(aw+ae+as+an+ab+at).
// Kernels here are per cell (one thread per cell or coarse cell) with the
// coefficients read from FP64 arrays laid out like phi.

__device__ __forceinline__ const double *lsm_coef(const LevelDev &L, int q, int colour) {
  return L.lsm + (size_t)(2 * q + colour) * L.lsm_half;
}

// dens_mg of a coarse level: 0.125 * (c(j0 i0 k0) + c(j1 i0 k0) + c(j0 i1 k0)
// + c(j1 i1 k0) + c(j0 i0 k1) + ... ), the reference's j-fastest packing
// order (mgsolver.for:99-118); arrays interior, i fastest
__global__ void k_lsm_dens_restrict(const double *__restrict__ fine, int fni, int fnj, int fnk,
                                    double *__restrict__ coarse) {
  const int cni = fni / 2, cnj = fnj / 2, cnk = fnk / 2;
  const size_t n = (size_t)cni * cnj * cnk;
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const int i = (int)(q % cni), j = (int)((q / cni) % cnj), k = (int)(q / ((size_t)cni * cnj));
  auto f = [&](int di, int dj, int dk) {
    return fine[((size_t)(2 * k + dk) * fnj + (2 * j + dj)) * fni + (2 * i + di)];
  };
  coarse[q] = 0.125 * (f(0, 0, 0) + f(0, 1, 0) + f(1, 0, 0) + f(1, 1, 0) + f(0, 0, 1) +
                       f(0, 1, 1) + f(1, 0, 1) + f(1, 1, 1));
}

// coefficients of every cell of one level of one block; walls: bit a*2 (+1)
// set = the low (high) face of axis a is a wall (coefficient 0)
__global__ void k_lsm_coef(const LevelDev *__restrict__ lev_dev, const double *__restrict__ dens,
                           int ni, int nj, int nk, double dx, double dy, double dz, int walls) {
  const size_t n = (size_t)ni * nj * nk;
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= n) return;
  const LevelDev &L = *lev_dev;
  const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
  const size_t si = 1, sj = (size_t)ni, sk = (size_t)ni * nj;
  const double d = dens[q];
  // face densities (mgsolver.for:130-164): the cell's own on the block's
  // first/last cell of an axis, else the mean with the neighbour (own first)
  const double dim = i == 0 ? d : 0.5 * (d + dens[q - si]);
  const double dip = i == ni - 1 ? d : 0.5 * (d + dens[q + si]);
  const double djm = j == 0 ? d : 0.5 * (d + dens[q - sj]);
  const double djp = j == nj - 1 ? d : 0.5 * (d + dens[q + sj]);
  const double dkm = k == 0 ? d : 0.5 * (d + dens[q - sk]);
  const double dkp = k == nk - 1 ? d : 0.5 * (d + dens[q + sk]);
  double c[7];
  c[0] = dy * dz / dx / dim;
  c[1] = dy * dz / dx / dip;
  c[2] = dx * dz / dy / djm;
  c[3] = dx * dz / dy / djp;
  c[4] = dx * dy / dz / dkm;
  c[5] = dx * dy / dz / dkp;
  // walls (mgsolver.for:194-205)
  if ((walls & 1) && i == 0) c[0] = 0.0;
  if ((walls & 2) && i == ni - 1) c[1] = 0.0;
  if ((walls & 4) && j == 0) c[2] = 0.0;
  if ((walls & 8) && j == nj - 1) c[3] = 0.0;
  if ((walls & 16) && k == 0) c[4] = 0.0;
  if ((walls & 32) && k == nk - 1) c[5] = 0.0;
  c[6] = -1.0 * (c[0] + c[1] + c[2] + c[3] + c[4] + c[5]);
  const int colour = (i + j + k) & 1;
  const size_t e = cidx(L.H, L.nj, i, j, k);
  for (int a = 0; a < 7; ++a) L.lsm[(size_t)(2 * a + colour) * L.lsm_half + e] = c[a];
}

// finest-level residual r = f - A p with per-cell coefficients into the
// level-1 rhs, with per-tile partial sum of r^2 and max |r| (the residual
// tiles' work layout: lane l holds cells 2l and 2l+1 of one row)
__global__ void __launch_bounds__(NTHREADS)
    k_lsm_residual(const Tile *__restrict__ tiles, const FineDev *__restrict__ fine,
                   const LevelDev *__restrict__ levs, const int *__restrict__ active,
                   RedPartial *__restrict__ partials) {
  const int ti = xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const Tile t = tiles[ti];
  const FineDev &F = fine[t.lev];
  const LevelDev &L = levs[t.lev];
  double ss = 0.0, am = 0.0;
  if (active[F.blk]) {
    const int lpr = F.lpr;
    const int lane = (int)threadIdx.x;
    const int j = t.y0 + (int)threadIdx.y * (64 / lpr) + lane / lpr;
    // the tile's two halves of lpr entries, one entry per lane
    for (int half = 0; half < 2; ++half)
    for (int k = t.z0; k < t.z1; ++k)
      for (int s = 0; s < 2; ++s) {
        const int l = t.x0 + half * lpr + (lane & (lpr - 1));
        const int i = 2 * l + s;
        if (i >= F.ni || j >= F.nj) continue;
        const int c = (i + j + k) & 1;
        const size_t e = cidx(F.H, F.nj, i, j, k);
        auto nb = [&](int x, int y, int z) -> double { return fine_value(fine, t.lev, x, y, z); };
        double cf[7];
        for (int a = 0; a < 7; ++a) cf[a] = lsm_coef(L, a, c)[e];
        const double P = F.p[c][e];
        const double r = F.f[c][e] - (cf[0] * nb(i - 1, j, k) + cf[1] * nb(i + 1, j, k) +
                                      cf[2] * nb(i, j - 1, k) + cf[3] * nb(i, j + 1, k) +
                                      cf[4] * nb(i, j, k - 1) + cf[5] * nb(i, j, k + 1) +
                                      cf[6] * P);
        ((double *)L.rhs[c])[e] = r;
        ss += r * r;
        am = fmax(am, fabs(r));
      }
  }
  block_reduce(ss, am);
  if (threadIdx.x == 0 && threadIdx.y == 0) partials[ti] = RedPartial{ss, am};
}

// ---------------------------------------------------------------------------
// Velocity projection of the outer loop (press.for:77-144 calvel and 2-75
// calmas, 2nd-order branch) on the device.  Face arrays are dense, i
// fastest: u (nk, nj, ni+1) with u[.., f] the face between cells f-1 and f,
// v (nk, nj+1, ni), w (nk+1, nj, ni); cell arrays (nk, nj, ni).
//
// calvel: face f of axis a between cells f-1 and f,
//     u = ustar - dt*alfapr*(p(f) - p(f-1))/h
// on the faces the reference updates (isu..ieu, localparameters.for:
// 106-192): the interior faces and, on a periodic axis, the wrap face (its
// second copy f = 0 is what exchange(1) gives it); wall-normal faces keep
// ustar.  Pressure ghosts are images, as after pbound/exchange(4).
__global__ void __launch_bounds__(256)
    k_calvel(const FineDev *__restrict__ fd, int axis, const double *__restrict__ us,
             double *__restrict__ u, double dt_alfa, double h) {
  const FineDev &F = *fd;
  const int n[3] = {F.ni, F.nj, F.nk};
  int dim[3] = {F.ni, F.nj, F.nk};
  dim[axis] += 1;  // faces along `axis`
  const size_t total = (size_t)dim[0] * dim[1] * dim[2];
  const bool per = (F.per >> axis) & 1;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total;
       q += (size_t)gridDim.x * blockDim.x) {
    int c[3];
    c[0] = (int)(q % dim[0]);
    c[1] = (int)((q / dim[0]) % dim[1]);
    c[2] = (int)(q / ((size_t)dim[0] * dim[1]));
    const int f = c[axis];
    const bool upd = (f > 0 && f < n[axis]) || per;
    double v = us[q];
    if (upd) {
      int hi[3] = {c[0], c[1], c[2]}, lo[3] = {c[0], c[1], c[2]};
      hi[axis] = f == n[axis] ? 0 : f;        // wrap: cell 0 (the ghost image)
      lo[axis] = f == 0 ? n[axis] - 1 : f - 1;
      const double ph = F.p[(hi[0] + hi[1] + hi[2]) & 1][cidx(F.H, F.nj, hi[0], hi[1], hi[2])];
      const double pl = F.p[(lo[0] + lo[1] + lo[2]) & 1][cidx(F.H, F.nj, lo[0], lo[1], lo[2])];
      if (F.dens) {
        // L_LSM: divided by the face density (press.for:93-96)
        const double dl = F.dens[((size_t)lo[2] * F.nj + lo[1]) * F.ni + lo[0]];
        const double dh = F.dens[((size_t)hi[2] * F.nj + hi[1]) * F.ni + hi[0]];
        v = v - dt_alfa * (ph - pl) / h / (0.5 * (dl + dh));
      } else {
        v = v - dt_alfa * (ph - pl) / h;
      }
    }
    u[q] = v;
  }
}

// calvel for blocks with neighbours (the same update): face f of `axis` is
// computed for 0 < f < n and, when a neighbour or a periodic wrap lies
// across the block's far face, for f = n (the reference's isu..ieu,
// localparameters.for:106-192); the near face f = 0 is not written here --
// it is the neighbour's far face, which exchange(1..3) copies
// (k_face_copy); wall-normal faces keep u*.  Pressure ghosts are read
// through resolve_cell (pbound/exchange(4)).
__global__ void __launch_bounds__(256)
    k_calvel_nb(const FineDev *__restrict__ fine, int b, int axis, const double *__restrict__ us,
                double *__restrict__ u, double dt_alfa, double h) {
  const FineDev &F = fine[b];
  const int n[3] = {F.ni, F.nj, F.nk};
  int dim[3] = {F.ni, F.nj, F.nk};
  dim[axis] += 1;
  const size_t total = (size_t)dim[0] * dim[1] * dim[2];
  const bool far_open = !wall_face(F, 2 * axis + 1), near_open = !wall_face(F, 2 * axis);
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total;
       q += (size_t)gridDim.x * blockDim.x) {
    int c[3];
    c[0] = (int)(q % dim[0]);
    c[1] = (int)((q / dim[0]) % dim[1]);
    c[2] = (int)(q / ((size_t)dim[0] * dim[1]));
    const int f = c[axis];
    if (f == 0 && near_open) continue;
    const bool upd = (f > 0 && f < n[axis]) || (f == n[axis] && far_open);
    double v = us[q];
    if (upd) {
      int lo[3] = {c[0], c[1], c[2]};
      lo[axis] = f - 1;
      const double ph = fine_value(fine, b, c[0], c[1], c[2]);
      const double pl = fine_value(fine, b, lo[0], lo[1], lo[2]);
      v = v - dt_alfa * (ph - pl) / h;
    }
    u[q] = v;
  }
}

// exchange(1..3) of one face: the near face (f = 0) of `axis` in dst takes
// the far face (f = n_src) of the block across it (a neighbour, or the block
// itself on a periodic axis); both blocks share the face's extent (nu, nv =
// the two other axes' cell counts, in dst's order).
__global__ void __launch_bounds__(256)
    k_face_copy(int axis, const double *__restrict__ src, int n_src, double *__restrict__ dst,
                int n_dst, int nu, int nv) {
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (size_t)nu * nv) return;
  const size_t a = q % nu, c = q / nu;  // u faster than v
  // face arrays are (nk, nj, ni) with the face axis extended by one
  size_t qs, qd;
  if (axis == 0) {  // (c = k, a = j): u[(k*nj + j)*(ni+1) + f]
    qs = (c * nu + a) * (size_t)(n_src + 1) + n_src;
    qd = (c * nu + a) * (size_t)(n_dst + 1);
  } else if (axis == 1) {  // (c = k, a = i): v[(k*(nj+1) + f)*ni + i]
    qs = (c * (size_t)(n_src + 1) + n_src) * nu + a;
    qd = (c * (size_t)(n_dst + 1)) * nu + a;
  } else {  // (c = j, a = i): w[(f*nj + j)*ni + i]
    qs = ((size_t)n_src * nv + c) * nu + a;
    qd = c * nu + a;
  }
  dst[qd] = src[qs];
}

// calmas: su = ((du/dx + dv/dy) + dw/dz)/dt per cell, and per workgroup the
// max of |fact*dx*dy*dz| (rmax before its MPI_ALLREDUCE, press.for:59-73).
// su goes to the dense array `su` (when not null) or, with to_fine, into the
// block's colour-split f arrays (the next V-cycle's right-hand side).
__global__ void __launch_bounds__(256)
    k_calmas(const FineDev *__restrict__ fd, const double *__restrict__ u,
             const double *__restrict__ v, const double *__restrict__ w, double *__restrict__ su,
             int to_fine, double dt, double dx, double dy, double dz,
             RedPartial *__restrict__ partials) {
  const FineDev &F = *fd;
  const int ni = F.ni, nj = F.nj, nk = F.nk;
  const size_t total = (size_t)ni * nj * nk;
  double am = 0.0, ss = 0.0;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total;
       q += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
    const size_t qu = ((size_t)k * nj + j) * (ni + 1) + i;
    const size_t qv = ((size_t)k * (nj + 1) + j) * ni + i;
    const size_t qw = ((size_t)k * nj + j) * ni + i;
    const double fact = (u[qu + 1] - u[qu]) / dx + (v[qv + ni] - v[qv]) / dy +
                        (w[qw + (size_t)ni * nj] - w[qw]) / dz;
    // L_LSM: sup = div(u) dx dy dz / dt (press.for:53-55)
    const double rhs = F.dens ? fact * dx * dy * dz / dt : fact / dt;
    if (to_fine)
      F.f[(i + j + k) & 1][cidx(F.H, F.nj, i, j, k)] = rhs;
    else if (su)
      su[q] = rhs;
    const double fact1 = fact * dx * dy * dz;
    am = fmax(am, fabs(fact1));
  }
  // fixed-order workgroup reduction (block_reduce needs 256 = NTHREADS threads)
  block_reduce(ss, am);
  if (threadIdx.x == 0) partials[blockIdx.x] = RedPartial{0.0, am};
}

// calvel and calmas of every block in one launch (grid.y: block, from b0).
// Each is a stream over the faces and cells; separate launches per axis and
// block read p three times and u, v, w twice, and cost a launch of 2-4 us
// each (a 64-block handle: 448 launches per step).  Here a lane owns cells
// 2l, 2l+1 of one row (one entry of both colour arrays of p) and walks kb
// planes: the west, south and bottom faces of its cells are its own to
// write, the east face comes from the next lane (DPP), the north face is
// computed again, the top face carries over as the next plane's bottom, and
// su and the rmax partial follow from the faces in registers.  Per cell that
// reads u*, v*, w*, p and writes u, v, w, su once: 64 B instead of 104.
// Every face and cell value is k_calvel's / k_calvel_nb's / k_calmas'
// expression.
//   connected: a near face across which a block lies takes that block's far
//     face -- its u* and this face's pressures, the value k_face_copy copies;
//   to_fine: su goes into the block's f arrays and, to_fine = 2, the level-1
//     rhs in the level's type T (the next V-cycle starts from it); 0: to V.su
//     if any;
//   calmas = 0: faces only (calmas' 4th-order branch follows on its own).
// Bound by memory: 192^3 takes 113 us (453 MB, 4.0 TB/s) where calvel x 3 +
// calmas took 174; 128x128x96 28 us where they took 47; the 64 blocks of a
// 64x8x64 layout 34 us where their 448 launches took ~1.4 ms.
// A workgroup strides over the tiles of its block (64-entry row segments or
// whole short rows x kb planes), so gridDim.x bounds the partials:
// partials[(block - b0) * gridDim.x + blockIdx.x].
typedef double __attribute__((ext_vector_type(2), aligned(8))) d2u;  // 8-byte aligned pair

// Every load of a plane is issued before its first use, with no branch that
// depends on a loaded value: ghosts are addresses (the array, row and plane
// that hold the image), selected per lane.  EVEN: ni even, so a lane's two
// cells are always a pair inside the row (16-byte accesses).
template <class T, bool LSM, bool EVEN>
__global__ void __launch_bounds__(NTHREADS)
    k_project(const FineDev *__restrict__ fine, const LevelDev *__restrict__ levs,
              const int *__restrict__ active, const VelDev *__restrict__ tab,
              const ProjDt *__restrict__ dtab, VelDev one, ProjDt dt_one, int b0, int kb,
              int connected, int to_fine, int calmas, RedPartial *__restrict__ partials) {
  typedef typename Vec2<double>::type d2;
  const int b = b0 + (int)blockIdx.y;
  const FineDev &F = fine[b];
  double am = 0.0, ss = 0.0;
  if (!active || active[b]) {
    const VelDev V = tab ? tab[b] : one;
    const ProjDt D = dtab ? *dtab : dt_one;
    const double dta = D.dta, dt = D.dt, dx = F.dx, dy = F.dy, dz = F.dz;
    const int ni = F.ni, nj = F.nj, nk = F.nk, H = F.H;
    const bool open_w = !wall_face(F, 0), open_e = !wall_face(F, 1), open_s = !wall_face(F, 2),
               open_n = !wall_face(F, 3), open_b = !wall_face(F, 4), open_t = !wall_face(F, 5);
    // the block across each face (itself on a periodic axis it spans)
    auto across = [&](int f) -> int { return F.nbr[f] >= 0 ? F.nbr[f] : b; };
    // lanes per row segment: the whole row's entries, or 64
    const int ne = (ni + 1) >> 1;
    const int lg = ne >= 64 ? 6 : ne <= 1 ? 0 : 32 - __clz(ne - 1);
    const int lp = 1 << lg, rows = NTHREADS >> lg;
    const int ntx = (ne + lp - 1) >> lg, nty = (nj + rows - 1) / rows, ntz = (nk + kb - 1) / kb;
    const int tid = (int)threadIdx.x, rl = tid & (lp - 1);
    typedef const gmem<double> *src;
    const src P0 = (src)F.p[0], P1 = (src)F.p[1];
    const src US = (src)V.us, VS = (src)V.vs, WS = (src)V.ws;
    gmem<double> *const U = (gmem<double> *)V.u, *const Vv = (gmem<double> *)V.v,
                 *const W = (gmem<double> *)V.w;
    gmem<double> *const F0 = (gmem<double> *)F.f[0], *const F1 = (gmem<double> *)F.f[1];
    gmem<T> *const R0 = (gmem<T> *)levs[b].rhs[0], *const R1 = (gmem<T> *)levs[b].rhs[1];
    const bool to_rhs = to_fine == 2;
    const size_t pu = (size_t)(ni + 1), plane = (size_t)ni * nj;
    // u = us - dta*(ph - pl)/h, over the face density of an L_LSM handle
    auto corr = [&](double us, double pl, double ph, double h, double dl, double dh) -> double {
      if (LSM) return us - dta * (ph - pl) / h / (0.5 * (dl + dh));
      return us - dta * (ph - pl) / h;
    };
    for (int t = (int)blockIdx.x; t < ntx * nty * ntz; t += (int)gridDim.x) {
      const int tx = t % ntx, tr = t / ntx, ty = tr % nty, tz = tr / nty;
      const int l = tx * lp + rl, j = ty * rows + (tid >> lg);
      const int k0 = tz * kb, k1 = min(k0 + kb, nk);
      const int a = 2 * l;  // cells a, a+1
      const bool ok = a < ni && j < nj, okb = a + 1 < ni && j < nj;
      // lanes outside the block read a valid entry and store nothing
      const int lc = min(l, ne - 1), jc = min(j, nj - 1), ac = 2 * lc;
      const int bo = EVEN ? 1 : min(1, ni - 1 - ac);  // cell a+1, or a again past an odd row's end
      // pressures of the lane's two cells in row y of an array pair (A0, A1)
      // with nr rows per plane: the even cell has colour (y + z) & 1
      auto pair = [&](src A0, src A1, int nr, int y, int z) -> d2 {
        const unsigned o = ((unsigned)z * (unsigned)nr + (unsigned)y) * (unsigned)H + (unsigned)lc;
        const double e0 = A0[o], e1 = A1[o];
        return ((y + z) & 1) ? d2{e1, e0} : d2{e0, e1};
      };
      auto ld = [&](src q, size_t o) -> d2 {
        if (EVEN) {
          const d2u v = *(const gmem<d2u> *)(q + o);
          return d2{v.x, v.y};
        }
        return d2{q[o], q[o + bo]};
      };
      auto st = [&](gmem<double> *q, size_t o, d2 v) {
        if (okb)
          *(gmem<d2u> *)(q + o) = d2u{v.x, v.y};
        else if (ok)
          q[o] = v.x;
      };
      // (L_LSM) the lane's two densities in row y, plane z
      auto dens2 = [&](int y, int z) -> d2 {
        if (!LSM) return d2{1.0, 1.0};
        return ld((src)F.dens, (size_t)z * plane + (size_t)y * ni + ac);
      };
      auto dens1 = [&](int x, int y, int z) -> double {
        return LSM ? ((src)F.dens)[(size_t)z * plane + (size_t)y * ni + x] : 1.0;
      };
      // rows and u* of the y faces: the image row across an open face
      const int qs = across(2), qn = across(3);
      const bool at_s = jc == 0, at_n = jc == nj - 1;
      const int njs = fine[qs].nj;
      const src S0 = at_s && open_s ? (src)fine[qs].p[0] : P0,
                S1 = at_s && open_s ? (src)fine[qs].p[1] : P1;
      const src N0 = at_n && open_n ? (src)fine[qn].p[0] : P0,
                N1 = at_n && open_n ? (src)fine[qn].p[1] : P1;
      const int ys = at_s ? (open_s ? njs - 1 : 0) : jc - 1, nrs = at_s && open_s ? njs : nj;
      const int yn = at_n ? (open_n ? 0 : jc) : jc + 1, nrn = at_n && open_n ? fine[qn].nj : nj;
      const bool nbr_s = connected && at_s && open_s;
      const src VSs = nbr_s ? (src)tab[qs].vs : VS;
      const int fs = nbr_s ? njs : jc, nfs = (nbr_s ? njs : nj) + 1;
      const bool up_s = !at_s || open_s, up_n = !at_n || open_n;
      // x edges: the first lane's west neighbour, the last lane's east one
      const bool edge_w = rl == 0, edge_e = rl == lp - 1 || ac + 2 >= ni;
      const bool at_w = ac == 0, at_e = ac + 2 >= ni;
      const int qw_ = across(0), qe = across(1);
      const int niw = fine[qw_].ni;
      const int xw = at_w ? (open_w ? niw - 1 : 0) : ac - 1;
      const int xe = at_e ? (open_e ? 0 : ni - 1) : ac + 2;
      const int Hw = at_w && open_w ? fine[qw_].H : H, He = at_e && open_e ? fine[qe].H : H;
      const bool img_w = at_w && open_w, img_e = at_e && open_e;
      const src W0 = img_w ? (src)fine[qw_].p[0] : P0, W1 = img_w ? (src)fine[qw_].p[1] : P1;
      const src E0 = img_e ? (src)fine[qe].p[0] : P0, E1 = img_e ? (src)fine[qe].p[1] : P1;
      const bool nbr_w = connected && img_w;
      const bool up_w = !at_w || open_w, up_e = !at_e || open_e;

      d2 pc = pair(P0, P1, nj, jc, k0), wb;
      d2 dc = dens2(jc, k0);
      {  // bottom faces of the first plane (k0, open_b: uniform)
        const size_t o = (size_t)jc * ni + ac;
        const int qb = across(4);
        wb = connected && k0 == 0 && open_b ? ld((src)tab[qb].ws, (size_t)fine[qb].nk * plane + o)
                                            : ld(WS, (size_t)k0 * plane + o);
        if (k0 > 0 || open_b) {
          const int zb = k0 > 0 ? k0 - 1 : fine[qb].nk - 1;
          const d2 pm = k0 > 0 ? pair(P0, P1, nj, jc, zb)
                               : pair((src)fine[qb].p[0], (src)fine[qb].p[1], nj, jc, zb);
          const d2 dm = dens2(jc, zb);
          wb.x = corr(wb.x, pm.x, pc.x, dz, dm.x, dc.x);
          wb.y = corr(wb.y, pm.y, pc.y, dz, dm.y, dc.y);
        }
      }
      for (int k = k0; k < k1; ++k) {
        const size_t qu = ((size_t)k * nj + jc) * pu + ac;
        const size_t qv = ((size_t)k * (nj + 1) + jc) * ni + ac;
        const size_t qw = (size_t)k * plane + (size_t)jc * ni + ac;
        // loads of the plane
        const d2u us = *(const gmem<d2u> *)(US + qu);  // faces a, a+1 (a+1 <= ni)
        d2 vs = ld(VSs, ((size_t)k * nfs + fs) * ni + ac), vn = ld(VS, qv + ni);
        d2 wt = ld(WS, qw + plane);
        const d2 ps = pair(S0, S1, nrs, ys, k), pn = pair(N0, N1, nrn, yn, k);
        const int qt = across(5);
        const bool top = k + 1 >= nk;
        const d2 pp = !top || !open_t
                          ? pair(P0, P1, nj, jc, min(k + 1, nk - 1))
                          : pair((src)fine[qt].p[0], (src)fine[qt].p[1], nj, jc, 0);
        double pw = 0.0, pe = 0.0, u0n = 0.0, u2 = 0.0;
        if (edge_w) {
          const unsigned o = ((unsigned)k * nj + jc) * (unsigned)Hw + (unsigned)(xw >> 1);
          pw = ((xw + jc + k) & 1) ? W1[o] : W0[o];
          if (nbr_w) u0n = ((src)tab[qw_].us)[((size_t)k * nj + jc) * (niw + 1) + niw];
        }
        if (edge_e) {
          const unsigned o = ((unsigned)k * nj + jc) * (unsigned)He + (unsigned)(xe >> 1);
          pe = ((xe + jc + k) & 1) ? E1[o] : E0[o];
          if (EVEN || ac + 2 <= ni) u2 = US[qu + 2];
        }
        d2 ds = d2{1.0, 1.0}, dn = ds, dp = ds;
        double dw = 1.0, de = 1.0;
        if (LSM) {
          ds = dens2(ys, k);
          dn = dens2(yn, k);
          dp = dens2(jc, top ? 0 : k + 1);
          dw = dens1(at_w ? ni - 1 : ac - 1, jc, k);
          de = dens1(at_e ? 0 : ac + 2, jc, k);
        }
        // x faces a, a+1, a+2
        const double lf = wave_shift(pc.y, 1);
        if (!edge_w) pw = lf;
        double u0 = nbr_w ? u0n : us.x, u1 = us.y;
        if (up_w) u0 = corr(u0, pw, pc.x, dx, dw, dc.x);
        if (EVEN || bo)
          u1 = corr(u1, pc.x, pc.y, dx, dc.x, dc.y);
        else if (open_e)  // an odd row's last cell
          u1 = corr(u1, pc.x, pe, dx, dc.x, de);
        const double rt = wave_shift(u0, 0);
        if (edge_e) {
          if (up_e) u2 = corr(u2, pc.y, pe, dx, dc.y, de);
        } else {
          u2 = rt;
        }
        st(U, qu, d2{u0, u1});
        if (!EVEN && ok && !okb) U[qu + 1] = u1;
        if (okb && a + 2 == ni) U[qu + 2] = u2;
        // y faces jc (south) and jc+1 (north)
        if (up_s) {
          vs.x = corr(vs.x, ps.x, pc.x, dy, ds.x, dc.x);
          vs.y = corr(vs.y, ps.y, pc.y, dy, ds.y, dc.y);
        }
        if (up_n) {
          vn.x = corr(vn.x, pc.x, pn.x, dy, dc.x, dn.x);
          vn.y = corr(vn.y, pc.y, pn.y, dy, dc.y, dn.y);
        }
        st(Vv, qv, vs);
        if (j == nj - 1) st(Vv, qv + ni, vn);
        // z faces k (bottom, carried) and k+1 (top)
        if (!top || open_t) {
          wt.x = corr(wt.x, pc.x, pp.x, dz, dc.x, dp.x);
          wt.y = corr(wt.y, pc.y, pp.y, dz, dc.y, dp.y);
        }
        st(W, qw, wb);
        if (top) st(W, qw + plane, wt);
        if (calmas) {
          const double fa = (u1 - u0) / dx + (vn.x - vs.x) / dy + (wt.x - wb.x) / dz;
          const double fb = (u2 - u1) / dx + (vn.y - vs.y) / dy + (wt.y - wb.y) / dz;
          // L_LSM: sup = div(u) dx dy dz / dt (press.for:53-55)
          const double ra = LSM ? fa * dx * dy * dz / dt : fa / dt;
          const double rb = LSM ? fb * dx * dy * dz / dt : fb / dt;
          if (to_fine) {
            const unsigned o = ((unsigned)k * nj + jc) * (unsigned)H + (unsigned)lc;
            const bool odd = (jc + k) & 1;
            if (ok) {
              (odd ? F1 : F0)[o] = ra;
              if (to_rhs) (odd ? R1 : R0)[o] = (T)ra;
            }
            if (okb) {
              (odd ? F0 : F1)[o] = rb;
              if (to_rhs) (odd ? R0 : R1)[o] = (T)rb;
            }
          } else if (V.su) {
            st((gmem<double> *)V.su, qw, d2{ra, rb});
          }
          if (ok) am = fmax(am, fabs(fa * dx * dy * dz));
          if (okb) am = fmax(am, fabs(fb * dx * dy * dz));
        }
        wb = wt;
        pc = pp;
        dc = dp;
      }
    }
  }
  if (!partials) return;
  block_reduce(ss, am);
  if (threadIdx.x == 0)
    partials[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = RedPartial{0.0, am};
}

// max of the `amax` fields of n partials into *out (one workgroup; a max is
// exact in any order)
__global__ void __launch_bounds__(256)
    k_partials_max(const RedPartial *__restrict__ parts, int n, double *__restrict__ out) {
  double ss = 0.0, am = 0.0;
  for (int q = (int)threadIdx.x; q < n; q += 256) am = fmax(am, parts[q].amax);
  block_reduce(ss, am);
  if (threadIdx.x == 0) *out = am;
}

// calmas, differencing = 2 (press.for:17-37): per axis
//   (((-u(i+1) + 27 u(i)) - 27 u(i-1)) + u(i-2)) / (24 dx)
// in the reference's order (u(i) the east face of cell i: dense faces
// c+2, c+1, c, c-1 of cell c), the three axes summed x + y, then + z;
// su = fact/dt, rmax from |fact*dx*dy*dz| as in k_calmas.  Faces -1 and
// n+1 come from Outer4.
__global__ void __launch_bounds__(256)
    k_calmas4(const FineDev *__restrict__ fd, const double *__restrict__ u,
              const double *__restrict__ v, const double *__restrict__ w, double *__restrict__ su,
              int to_fine, double dt, double dx, double dy, double dz,
              RedPartial *__restrict__ partials, Outer4 o) {
  const FineDev &F = *fd;
  const int ni = F.ni, nj = F.nj, nk = F.nk;
  const size_t total = (size_t)ni * nj * nk;
  // face f of axis 0 at (j, k): own array for 0..ni, else the outer source
  auto uface = [&](int f, int j, int k) -> double {
    if (f >= 0 && f <= ni) return u[((size_t)k * nj + j) * (ni + 1) + f];
    const int s = f < 0 ? 0 : 1, m = o.n[s];
    if (m == 0) return o.src[s][(size_t)k * nj + j];
    return o.src[s][((size_t)k * nj + j) * (m + 1) + (s ? 1 : m - 1)];
  };
  auto vface = [&](int f, int i, int k) -> double {
    if (f >= 0 && f <= nj) return v[((size_t)k * (nj + 1) + f) * ni + i];
    const int s = f < 0 ? 0 : 1, m = o.n[2 + s];
    if (m == 0) return o.src[2 + s][(size_t)k * ni + i];
    return o.src[2 + s][((size_t)k * (m + 1) + (s ? 1 : m - 1)) * ni + i];
  };
  auto wface = [&](int f, int i, int j) -> double {
    if (f >= 0 && f <= nk) return w[((size_t)f * nj + j) * ni + i];
    const int s = f < 0 ? 0 : 1, m = o.n[4 + s];
    if (m == 0) return o.src[4 + s][(size_t)j * ni + i];
    return o.src[4 + s][((size_t)(s ? 1 : m - 1) * nj + j) * ni + i];
  };
  double am = 0.0, ss = 0.0;
  for (size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x; q < total;
       q += (size_t)gridDim.x * blockDim.x) {
    const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
    const double dux = ((-uface(i + 2, j, k) + 27.0 * uface(i + 1, j, k)) - 27.0 * uface(i, j, k)) +
                       uface(i - 1, j, k);
    const double dvy = ((-vface(j + 2, i, k) + 27.0 * vface(j + 1, i, k)) - 27.0 * vface(j, i, k)) +
                       vface(j - 1, i, k);
    const double dwz = ((-wface(k + 2, i, j) + 27.0 * wface(k + 1, i, j)) - 27.0 * wface(k, i, j)) +
                       wface(k - 1, i, j);
    const double fact = (dux / (24.0 * dx) + dvy / (24.0 * dy)) + dwz / (24.0 * dz);
    const double rhs = fact / dt;
    if (to_fine)
      F.f[(i + j + k) & 1][cidx(F.H, F.nj, i, j, k)] = rhs;
    else if (su)
      su[q] = rhs;
    const double fact1 = fact * dx * dy * dz;
    am = fmax(am, fabs(fact1));
  }
  block_reduce(ss, am);
  if (threadIdx.x == 0) partials[blockIdx.x] = RedPartial{0.0, am};
}

// ---- layout conversion ---------------------------------------------------
// p (which 0) or f of a block to and from a dense array: a thread per entry of
// both colours in a row of lp lanes (a power of two), 32-bit row arithmetic.
// (A thread per cell divided 64-bit indexes: 59 in and 69 us out at 256^3, now
// 53 and 44.)
template <bool PACK>
__global__ void __launch_bounds__(256)
    k_copy_fine(const FineDev *__restrict__ fd, int which, double *__restrict__ dense, int lp,
                int xb) {
  const FineDev &F = *fd;
  const unsigned rb = blockIdx.x / (unsigned)xb, xt = blockIdx.x - rb * (unsigned)xb;
  const int tid = (int)threadIdx.x, rl = tid & (lp - 1);
  const unsigned row = rb * (unsigned)(256 / lp) + (unsigned)(tid / lp);
  const int l = (int)(xt * (unsigned)lp) + rl, ni = F.ni;
  if (row >= (unsigned)F.nj * (unsigned)F.nk || 2 * l >= ni) return;
  const unsigned k = row / (unsigned)F.nj, j = row - k * (unsigned)F.nj;
  double *const *const a = which == 0 ? F.p : F.f;
  gmem<double> *const a0 = (gmem<double> *)a[0], *const a1 = (gmem<double> *)a[1];
  const bool c = (j + k) & 1;
  gmem<double> *const pa = (c ? a1 : a0) + (row * (unsigned)F.H + (unsigned)l),
                *const pb = (c ? a0 : a1) + (row * (unsigned)F.H + (unsigned)l);
  gmem<double> *const d = (gmem<double> *)dense + ((size_t)row * ni + 2 * l);
  const bool two = 2 * l + 1 < ni;
  if (PACK) {
    const double va = d[0], vb = two ? d[1] : 0.0;
    *pa = va;
    if (two) *pb = vb;
  } else {
    const double va = *pa, vb = two ? *pb : 0.0;
    d[0] = va;
    if (two) d[1] = vb;
  }
}

// p of block b with its one-cell ghost layer, dense (nk+2, nj+2, ni+2), i
// fastest; ghosts are the cells resolve_cell names (pbound / exchange(4))
__global__ void k_unpack_fine_padded(const FineDev *__restrict__ fine, int b,
                                     double *__restrict__ dst) {
  const FineDev &F = fine[b];
  const int pi = F.ni + 2, pj = F.nj + 2, pk = F.nk + 2;
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= (size_t)pi * pj * pk) return;
  const int x = (int)(q % pi) - 1, y = (int)((q / pi) % pj) - 1, z = (int)(q / ((size_t)pi * pj)) - 1;
  dst[q] = fine_value(fine, b, x, y, z);
}

// which 0: phi (dense padded (n+2)^3 <-> buffer buf), 1: rhs (dense interior)
template <class T>
__global__ void k_pack_level(const LevelDev *__restrict__ ld, int which, int buf,
                             const double *__restrict__ src, int ni, int nj, int nk) {
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const size_t n = (size_t)ni * nj * nk;
  if (q >= n) return;
  const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
  const LevelDev &L = *ld;
  const size_t c = cidx(L.H, L.nj, i, j, k);
  const int col = (i + j + k) & 1;
  if (which == 0) {
    const size_t pi = (size_t)ni + 2, pj = (size_t)nj + 2;
    ((T *)L.phi[buf][col])[c] = (T)src[(size_t)(i + 1) + pi * ((size_t)(j + 1) + pj * (size_t)(k + 1))];
  } else {
    ((T *)L.rhs[col])[c] = (T)src[q];
  }
}

template <class T>
__global__ void k_unpack_level(const LevelDev *__restrict__ levs, int d, int which, int buf,
                               double *__restrict__ dst, int ni, int nj, int nk) {
  const size_t q = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  const LevelDev &L = levs[d];
  if (which == 0) {
    const int pi = ni + 2, pj = nj + 2, pk = nk + 2;
    const size_t n = (size_t)pi * pj * pk;
    if (q >= n) return;
    const int x = (int)(q % pi) - 1, y = (int)((q / pi) % pj) - 1, z = (int)(q / ((size_t)pi * pj)) - 1;
    dst[q] = (double)level_value<T>(levs, d, buf, x, y, z);
  } else {
    const size_t n = (size_t)ni * nj * nk;
    if (q >= n) return;
    const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
    dst[q] = (double)((const T *)L.rhs[(i + j + k) & 1])[cidx(L.H, L.nj, i, j, k)];
  }
}

// mean removal of p (FP64): one workgroup, fixed-order reduction
__global__ void __launch_bounds__(256)
    k_remove_mean(const FineDev *__restrict__ fd, int ni, int nj, int nk) {
  const FineDev &F = *fd;
  const size_t n = (size_t)ni * nj * nk;
  double s = 0.0;
  for (size_t q = threadIdx.x; q < n; q += 256) {
    const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
    s += F.p[(i + j + k) & 1][cidx(F.H, F.nj, i, j, k)];
  }
  __shared__ double sh[256];
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) sh[threadIdx.x] += sh[threadIdx.x + w];
    __syncthreads();
  }
  const double mean = sh[0] / (double)n;
  for (size_t q = threadIdx.x; q < n; q += 256) {
    const int i = (int)(q % ni), j = (int)((q / ni) % nj), k = (int)(q / ((size_t)ni * nj));
    double &v = F.p[(i + j + k) & 1][cidx(F.H, F.nj, i, j, k)];
    v = v - mean;
  }
}

inline dim3 tile_block() { return dim3(TILE_X, TILE_Y, 1); }


// ---------------------------------------------------------------------------
// Lexicographic Gauss-Seidel (mgsolver.for:407-432) and line TDMA
// (mgsolver.for:434-549), mg_itrsch = 1 and 2.
//
// The reference updates in place, in loop order.  A GS cell (loop k, j, i)
// reads its W, S and B neighbours after their update and E, N, T before it,
// so the cells of the hyperplane i+j+k = d depend on plane d-1 (updated) and
// plane d+1 (not yet) only: a hyperplane wavefront performs exactly the
// reference's arithmetic (k_gs_tile runs it over 8^3 tiles).  The TDMA
// passes are line-wise GS over the other two axes: j-lines (loop k, i) on
// diagonals i+k, i-lines (loop k, j) on j+k, k-lines (loop i, j) on i+j.  A
// sweep reads buffer src and writes 1-src:
//   GS and the j-line pass: values not yet updated from src, updated ones
//     from 1-src;
//   i-line and k-line passes: in place in 1-src;
//   ghosts, every pass: their images in src -- the pre-sweep state the
//     reference's ghosts keep until mgbound + exchangepp at the end of the
//     sweep (mgsolver.for:614-615).
// zero != 0: buffer src holds zeros.

// element e of a level array, read as global memory (no flat access)
__device__ __forceinline__ double gload(const void *base, size_t e) {
  return ((const gmem<double> *)base)[e];
}

// coefficients of one cell: the level's constant operator, or the
// variable-density arrays
__device__ __forceinline__ Coef<double> smoother_coef(const LevelDev &L, int i, int j, int k) {
  if (!L.lsm) return cell_coef<double>(L, i, j, k);
  const int colour = (i + j + k) & 1;
  const size_t e = cidx(L.H, L.nj, i, j, k);
  Coef<double> c;
  c.aw = gload(lsm_coef(L, 0, colour), e);
  c.ae = gload(lsm_coef(L, 1, colour), e);
  c.as = gload(lsm_coef(L, 2, colour), e);
  c.an = gload(lsm_coef(L, 3, colour), e);
  c.ab = gload(lsm_coef(L, 4, colour), e);
  c.at = gload(lsm_coef(L, 5, colour), e);
  c.ap = gload(lsm_coef(L, 6, colour), e);
  return c;
}

__device__ __forceinline__ double cell_at(const LevelDev &L, int buf, int i, int j, int k) {
  return gload(L.phi[buf][(i + j + k) & 1], cidx(L.H, L.nj, i, j, k));
}

// ghost or not-yet-updated value in buffer src (ghosts resolved to their
// image)
__device__ __forceinline__ double before_sweep(const LevelDev &L, int src, int zero, int x, int y,
                                               int z) {
  if (zero) return 0.0;
  x = image(x, L.ni, L.per & 1);
  y = image(y, L.nj, L.per & 2);
  z = image(z, L.nk, L.per & 4);
  return cell_at(L, src, x, y, z);
}

// One GS tile of GT^3 cells (Tile::x0, y0, z0): the tiles of one
// tile-diagonal I+J+K = D depend only on tiles of D-1 (updated) and D+1
// (not yet), as cells of a hyperplane do, so one launch per tile-diagonal
// repeats the reference's loop order, whatever the tile size.  The tile and
// its six face halos go to LDS -- the tile's cells and its east/north/top
// halo as before the sweep (src), its west/south/bottom halo as updated
// (dst, finished by earlier tile-diagonals), ghost positions as images of
// src -- and the wavefront walks the tile's own hyperplanes in place:
//   phi = (rhs - (aw*W + ae*E + as*S + an*N + ab*B + at*T)) / ap
// Thread (lx, ly) owns lz = h - lx - ly of plane h.  8^3 tiles (one
// wavefront, static LDS, variable-density coefficients staged too) and 16^3
// tiles (four wavefronts, constant coefficients, 79 KB of dynamic LDS:
// fewer tile-diagonals, so fewer launches per sweep).
template <int GT>
__device__ __forceinline__ void gs_tile_run(const Tile &t, const LevelDev &L, int src, int zero,
                                            double *v, double *rl, double *cl) {
  constexpr int GP = GT + 2;  // with the halo
  const int dst = 1 - src;
  const int tid = (int)threadIdx.x;
  const bool var = cl != nullptr && L.lsm != nullptr;
  // every load of the tile is issued before the first LDS store, with no
  // branch between them (clamped positions load an in-range cell whose
  // value is not stored or never read)
  constexpr int NT = GT * GT;
  constexpr int NR = GT * GT * GT / NT, NV = (GP * GP * GP + NT - 1) / NT;
  const int ni0 = L.ni, nj0 = L.nj, nk0 = L.nk, H0 = L.H;
  const bool px0 = L.per & 1, py0 = L.per & 2, pz0 = L.per & 4;
  // the level's phi arrays as byte offsets from src's colour 0
  const gmem<char> *const s0 = (const gmem<char> *)L.phi[src][0];
  const long long o_s1 = (const char *)L.phi[src][1] - (const char *)L.phi[src][0];
  const long long o_d0 = (const char *)L.phi[dst][0] - (const char *)L.phi[src][0];
  const long long o_d1 = (const char *)L.phi[dst][1] - (const char *)L.phi[src][0];
  double rr[NR], vv[NV];
#pragma unroll
  for (int it = 0; it < NR; ++it) {
    const int q = tid + it * NT;
    const int x = min(t.x0 + q % GT, ni0 - 1), y = min(t.y0 + (q / GT) % GT, nj0 - 1);
    const int z = min(t.z0 + q / (GT * GT), nk0 - 1);
    rr[it] = gload(L.rhs[(x + y + z) & 1], cidx(H0, nj0, x, y, z));
  }
#pragma unroll
  for (int it = 0; it < NV; ++it) {
    const int q = min(tid + it * NT, GP * GP * GP - 1);
    const int lz = q / (GP * GP) - 1, ly = (q / GP) % GP - 1, lx = q % GP - 1;
    int x = t.x0 + lx, y = t.y0 + ly, z = t.z0 + lz;
    const bool ghost = (unsigned)x >= (unsigned)ni0 || (unsigned)y >= (unsigned)nj0 ||
                       (unsigned)z >= (unsigned)nk0;
    // positions more than one cell outside the level (halo edges, corners
    // and the far side of a partial tile) are clamped; their values are
    // never read
    x = image(max(min(x, ni0), -1), ni0, px0);
    y = image(max(min(y, nj0), -1), nj0, py0);
    z = image(max(min(z, nk0), -1), nk0, pz0);
    // interior cells of the low-side halo: updated (dst); the tile, its
    // high-side halo and ghost images: before the sweep (src)
    const bool from_dst = !ghost && (lx < 0 || ly < 0 || lz < 0);
    const bool odd = (x + y + z) & 1;
    const long long o = from_dst ? (odd ? o_d1 : o_d0) : (odd ? o_s1 : 0);
    const double val =
        *(const gmem<double> *)(s0 + o + 8 * (((long long)z * nj0 + y) * H0 + (x >> 1)));
    vv[it] = (zero && !from_dst) ? 0.0 : val;
  }
#pragma unroll
  for (int it = 0; it < NR; ++it) rl[tid + it * NT] = rr[it];
#pragma unroll
  for (int it = 0; it < NV; ++it)
    if (tid + it * NT < GP * GP * GP) v[tid + it * NT] = vv[it];
  if (var)
    for (int q = tid; q < GT * GT * GT; q += NT) {
      const int x = t.x0 + q % GT, y = t.y0 + (q / GT) % GT, z = t.z0 + q / (GT * GT);
      if (x >= L.ni || y >= L.nj || z >= L.nk) continue;
      const size_t e = cidx(L.H, L.nj, x, y, z);
      for (int a = 0; a < 7; ++a) cl[a * GT * GT * GT + q] = gload(lsm_coef(L, a, (x + y + z) & 1), e);
    }
  __syncthreads();
  const int lx = tid % GT, ly = tid / GT;
  const int i = t.x0 + lx, j = t.y0 + ly;
  // the level's fields in registers: a barrier would make the compiler
  // reload them from memory on every plane
  const int ni = L.ni, nj = L.nj, nk = L.nk;
  const double cx = L.cx, cy = L.cy, cz = L.cz;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  // the planes touch LDS only: a barrier then waits for no global store
  for (int h = 0; h < 3 * GT - 2; ++h) {
    const int lz = h - lx - ly, k = t.z0 + lz;
    if (lz >= 0 && lz < GT && i < ni && j < nj && k < nk) {
      const int c0 = ((lz + 1) * GP + ly + 1) * GP + lx + 1;
      const int q = (lz * GT + ly) * GT + lx;
      Coef<double> c;
      if (var) {
        constexpr int S = GT * GT * GT;
        c.aw = cl[q], c.ae = cl[S + q], c.as = cl[2 * S + q], c.an = cl[3 * S + q];
        c.ab = cl[4 * S + q], c.at = cl[5 * S + q], c.ap = cl[6 * S + q];
      } else {  // cell_coef
        c.aw = (!px && i == 0) ? 0.0 : cx;
        c.ae = (!px && i == ni - 1) ? 0.0 : cx;
        c.as = (!py && j == 0) ? 0.0 : cy;
        c.an = (!py && j == nj - 1) ? 0.0 : cy;
        c.ab = (!pz && k == 0) ? 0.0 : cz;
        c.at = (!pz && k == nk - 1) ? 0.0 : cz;
        c.ap = -1.0 * (c.aw + c.ae + c.as + c.an + c.ab + c.at);
      }
      const double W = v[c0 - 1], E = v[c0 + 1];
      const double S = v[c0 - GP], N = v[c0 + GP];
      const double B = v[c0 - GP * GP], T = v[c0 + GP * GP];
      const double r = rl[q];
      const double sum = c.aw * W + c.ae * E + c.as * S + c.an * N + c.ab * B + c.at * T;
      v[c0] = (r - sum) / c.ap;
    }
    __syncthreads();
  }
  // the tile's column (lx, ly) to dst
  gmem<double> *const out0 = (gmem<double> *)L.phi[dst][0];
  gmem<double> *const out1 = (gmem<double> *)L.phi[dst][1];
  if (i < ni && j < nj)
    for (int lz = 0; lz < GT && t.z0 + lz < nk; ++lz) {
      const int k = t.z0 + lz;
      (((i + j + k) & 1) ? out1 : out0)[cidx(L.H, L.nj, i, j, k)] =
          v[((lz + 1) * GP + ly + 1) * GP + lx + 1];
    }
}

__global__ void __launch_bounds__(GS_TILE * GS_TILE)
    k_gs_tile(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
              const int *__restrict__ active, int src, int zero) {
  constexpr int GP = GS_TILE + 2;
  __shared__ double v[GP * GP * GP];                    // phi, tile + face halos
  __shared__ double rl[GS_TILE * GS_TILE * GS_TILE];      // rhs of the tile
  __shared__ double cl[7 * GS_TILE * GS_TILE * GS_TILE];  // variable-density coefficients
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  gs_tile_run<GS_TILE>(t, L, src, zero, v, rl, cl);
}

// 16^3 tiles, constant coefficients only (the host never launches it on a
// variable-density level): GS_BIG_LDS bytes of dynamic LDS
__global__ void __launch_bounds__(GS_BIG_TILE * GS_BIG_TILE)
    k_gs_tile_big(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                  const int *__restrict__ active, int src, int zero) {
  extern __shared__ double gs_lds[];
  constexpr int GP = GS_BIG_TILE + 2;
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk] || L.lsm) return;
  gs_tile_run<GS_BIG_TILE>(t, L, src, zero, gs_lds, gs_lds + GP * GP * GP, nullptr);
}

// positions of one line whose coefficients are loaded together
constexpr int TDMA_CHUNK = 8;

// cell (i, j, k) of position p on the line (u, v) of pass PASS
template <int PASS>
__device__ __forceinline__ void tdma_cell(int u, int v, int p, int &i, int &j, int &k) {
  if (PASS == 0) {
    i = u, j = p, k = v;
  } else if (PASS == 1) {
    i = p, j = u, k = v;
  } else {
    i = u, j = v, k = p;
  }
}

// Wall state of a cross coordinate c of a line (n cells on its axis): bit 0
// at the low wall, bit 1 at the high wall, 0 on a periodic axis.  Lines of
// one pass and state pair have the same coefficients along their length
// (cell_coef), so the same Thomas a(p) and 1/(ap - alo*a(p-1)).
__device__ __forceinline__ int wall_state(int c, int n, bool per) {
  return per ? 0 : (c == 0 ? 1 : 0) | (c == n - 1 ? 2 : 0);
}
// a coordinate of state s, or -1 when none has it
__device__ __forceinline__ int wall_rep(int s, int n, bool per) {
  if (per) return s == 0 ? 0 : -1;
  if (s == 0) return n >= 3 ? 1 : -1;
  if (s == 1 || s == 2) return n >= 2 ? (s == 1 ? 0 : n - 1) : -1;
  return n == 1 ? 0 : -1;
}

// geometry of the lines of pass PASS: lines (u, v), len cells each
template <int PASS>
struct TdmaGeom {
  int nu, nv, len;
  bool pu, pv;  // u / v axis periodic
  __device__ explicit TdmaGeom(const LevelDev &L) {
    nu = PASS == 1 ? L.nj : L.ni;
    nv = PASS == 2 ? L.nj : L.nk;
    len = PASS == 0 ? L.nj : PASS == 1 ? L.ni : L.nk;
    pu = PASS == 1 ? (L.per & 2) : (L.per & 1);
    pv = PASS == 2 ? (L.per & 2) : (L.per & 4);
  }
};

// (a(p), 1/(ap - alo*a(p-1))) of pass PASS, state pair `var`, position p
// of a constant-coefficient level: L.tdma + tdma_table_offset + 2*(var*len+p)
template <int PASS>
__device__ __forceinline__ size_t tdma_table_offset(const LevelDev &L) {
  return PASS == 0 ? 0 : PASS == 1 ? (size_t)32 * L.nj : (size_t)32 * (L.nj + L.ni);
}

template <int PASS>
__device__ __forceinline__ void tdma_table_fill(const LevelDev &L, int var) {
  const TdmaGeom<PASS> G(L);
  const int ru = wall_rep(var & 3, G.nu, G.pu), rv = wall_rep(var >> 2, G.nv, G.pv);
  if (ru < 0 || rv < 0) return;
  gmem<double> *tab = (gmem<double> *)(L.tdma + tdma_table_offset<PASS>(L) + (size_t)2 * var * G.len);
  double aprev = 0.0;
  for (int p = 0; p < G.len; ++p) {
    int i, j, k;
    tdma_cell<PASS>(ru, rv, p, i, j, k);
    const Coef<double> c = cell_coef<double>(L, i, j, k);
    const double alo = PASS == 0 ? c.as : PASS == 1 ? c.aw : c.ab;
    const double ahi = PASS == 0 ? c.an : PASS == 1 ? c.ae : c.at;
    const double apr = 1.0 / (c.ap - alo * aprev);
    aprev = ahi * apr;
    tab[2 * p] = aprev;
    tab[2 * p + 1] = apr;
  }
}

// a thread per (descriptor, pass, state pair)
__global__ void __launch_bounds__(256)
    k_tdma_tables(const LevelDev *__restrict__ levs, int ndesc) {
  const int q = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (q >= ndesc * 48) return;
  const LevelDev &L = levs[q / 48];
  if (!L.tdma) return;
  const int pass = (q / 16) % 3, var = q % 16;
  if (pass == 0)
    tdma_table_fill<0>(L, var);
  else if (pass == 1)
    tdma_table_fill<1>(L, var);
  else
    tdma_table_fill<2>(L, var);
}

// One diagonal d of one TDMA pass for the lines u0 .. u0+lw-1 (all threads
// of the workgroup call it; it holds one barrier), in two phases:
//  A (every thread, a cell at a time): the right-hand side of the Thomas
//    recurrence without its last term,
//      rs = rhs - x1*X1 - x2*X2 - x3*X3 - x4*X4,
//    with the cross terms in the reference's order -- j-lines ae*E, aw*W,
//    at*T, ab*B (mgsolver.for:459-466); i-lines an*N, as*S, at*T, ab*B
//    (:496-503); k-lines an*N, as*S, ae*E, aw*W (:533-540) -- into LDS at
//    xs[p*lwp + line].  The neighbours on the previous diagonal (W, B; S, B;
//    W, S) are updated ones.  On a constant-coefficient level the cell's
//    a(p) and 1/(ap - alo*a(p-1)) also go to LDS, from its line's table
//    (the same values the recurrence gives: a does not depend on the data).
//  B (a thread per line): the reference's recurrence (a(0) = 0, c(0) = the
//    ghost),
//      apr = 1/(ap - alo*a(p-1)),  a(p) = ahi*apr,
//      c(p) = (rs - alo*c(p-1))*apr,
//      phi(p) = c(p) - a(p)*phi(p+1),  phi(n) = the ghost,
//    (alo, ahi) = (as, an), (aw, ae), (ab, at); c overwrites rs in LDS.
//    Operands are read a chunk of positions ahead of the dependent chain.
// The subtraction of alo*c(p-1) is the last one of the reference's
// left-to-right sum, so splitting it off changes no rounding.  Lines of one
// diagonal never neighbour each other: phase A reads only lines of the
// diagonals before and after, which nothing writes meanwhile.
template <int PASS, int CPT, int NT = NTHREADS, bool PREV = false>
__device__ __forceinline__ void tdma_diagonal(const LevelDev &L, int u0, int lw, int lwp, int d,
                                              int src, int zero, double *xs, double *av,
                                              double *rv, int tid, double *prev = nullptr) {
  const TdmaGeom<PASS> G(L);
  const int nu = G.nu, nv = G.nv, len = G.len;
  const int ulo = max(u0, d - nv + 1), uhi = min(min(u0 + lw, nu), d + 1);
  const int dst = 1 - src;
  const bool tab = L.lsm == nullptr;
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  // the four phi arrays of the level as byte offsets from src's colour 0
  const gmem<char> *const s0 = (const gmem<char> *)L.phi[src][0];
  const long long o_s1 = (const char *)L.phi[src][1] - (const char *)L.phi[src][0];
  const long long o_d0 = (const char *)L.phi[dst][0] - (const char *)L.phi[src][0];
  const long long o_d1 = (const char *)L.phi[dst][1] - (const char *)L.phi[src][0];
  // value of a cross neighbour, with no branch: ghosts are images in src;
  // interior neighbours updated ones and (after the first pass) not-yet-
  // updated ones in dst, the first pass's others in src; src reads are 0
  // when src holds zeros
  auto cross = [=](int x, int y, int z, bool updated) -> double {
    const bool ghost = (unsigned)x >= (unsigned)ni || (unsigned)y >= (unsigned)nj ||
                       (unsigned)z >= (unsigned)nk;
    x = image(x, ni, px);
    y = image(y, nj, py);
    z = image(z, nk, pz);
    const bool from_dst = !ghost && (updated || PASS > 0);
    const bool odd = (x + y + z) & 1;
    const long long o = from_dst ? (odd ? o_d1 : o_d0) : (odd ? o_s1 : 0);
    const double val = *(const gmem<double> *)(s0 + o + 8 * (((long long)z * nj + y) * H + (x >> 1)));
    return (zero && !from_dst) ? 0.0 : val;
  };
  // the updated neighbours of line (u, v) lie on lines (u-1, v) and (u, v-1)
  // of diagonal d-1, at the same position: with `prev` (the previous
  // diagonal's solution in LDS, line u at prev[u*len + p]) they are read
  // from there -- the values the previous diagonal stored in dst -- instead
  // of from global memory
  auto upd = [=](int u, int v, int p, bool along_u, int x, int y, int z) -> double {
    if constexpr (PREV) {
      if (along_u ? u > 0 : v > 0) return prev[(along_u ? u - 1 : u) * len + p];
    }
    return cross(x, y, z, true);
  };
  // phase A: batches of CPT cells per thread, every load of a batch issued
  // before its first LDS store (positions past the end repeat the last cell
  // and are not stored)
  const int ncell = (uhi - ulo) * len;
  // q / len through a float reciprocal: exact while q < 2^12 * len
  const float inv_len = 1.0f / (float)len;
  for (int q0 = 0; q0 < ncell; q0 += CPT * NT) {
    double rsv[CPT], atv[CPT], rtv[CPT];
    int slot[CPT];
#pragma unroll
    for (int it = 0; it < CPT; ++it) {
      const int q = min(q0 + tid + it * NT, ncell - 1);
      const int lq = (int)(((float)q + 0.5f) * inv_len);
      const int l = ulo - u0 + lq, p = q - lq * len;
      const int u = u0 + l, v = d - u;
      int i, j, k;
      tdma_cell<PASS>(u, v, p, i, j, k);
      const Coef<double> c = smoother_coef(L, i, j, k);
      const double r = gload(L.rhs[(i + j + k) & 1], cidx(H, nj, i, j, k));
      double rs;
      if (PASS == 0)  // W on line (u-1, v), B on (u, v-1)
        rs = r - c.ae * cross(i + 1, j, k, false) - c.aw * upd(u, v, p, true, i - 1, j, k) -
             c.at * cross(i, j, k + 1, false) - c.ab * upd(u, v, p, false, i, j, k - 1);
      else if (PASS == 1)  // S on (u-1, v), B on (u, v-1)
        rs = r - c.an * cross(i, j + 1, k, false) - c.as * upd(u, v, p, true, i, j - 1, k) -
             c.at * cross(i, j, k + 1, false) - c.ab * upd(u, v, p, false, i, j, k - 1);
      else  // S on (u, v-1), W on (u-1, v)
        rs = r - c.an * cross(i, j + 1, k, false) - c.as * upd(u, v, p, false, i, j - 1, k) -
             c.ae * cross(i + 1, j, k, false) - c.aw * upd(u, v, p, true, i - 1, j, k);
      rsv[it] = rs;
      slot[it] = p * lwp + l;
      atv[it] = rtv[it] = 0.0;
      if (tab) {
        const int var = wall_state(u, nu, G.pu) | (wall_state(v, nv, G.pv) << 2);
        const size_t t = tdma_table_offset<PASS>(L) + (size_t)2 * (var * len + p);
        atv[it] = gload(L.tdma, t);
        rtv[it] = gload(L.tdma, t + 1);
      }
    }
#pragma unroll
    for (int it = 0; it < CPT; ++it)
      if (q0 + tid + it * NT < ncell) {
        xs[slot[it]] = rsv[it];
        if (tab) {
          av[slot[it]] = atv[it];
          rv[slot[it]] = rtv[it];
        }
      }
  }
  __syncthreads();
  const int l = tid, u = u0 + l, v = d - u;
  if (l >= lw || u < ulo || u >= uhi) return;
  int i, j, k;
  tdma_cell<PASS>(u, v, -1, i, j, k);
  double cprev = before_sweep(L, src, zero, i, j, k);
  if (tab) {
    // constant coefficients: alo is 1/h^2 of the line's axis, 0 at its
    // first cell next to a wall (cell_coef)
    const double cax = PASS == 0 ? L.cy : PASS == 1 ? L.cx : L.cz;
    const bool pax = PASS == 0 ? (L.per & 2) : PASS == 1 ? (L.per & 1) : (L.per & 4);
    for (int p0 = 0; p0 < len; p0 += TDMA_CHUNK) {
      // a chunk's operands, read with no branch in between (positions past
      // the line's end read its last cell and are not used)
      double rs[TDMA_CHUNK], apr[TDMA_CHUNK];
#pragma unroll
      for (int q = 0; q < TDMA_CHUNK; ++q) {
        const int p = min(p0 + q, len - 1);
        rs[q] = xs[p * lwp + l];
        apr[q] = rv[p * lwp + l];
      }
#pragma unroll
      for (int q = 0; q < TDMA_CHUNK; ++q) {
        const int p = p0 + q;
        if (p >= len) break;
        const double alo = (p == 0 && !pax) ? 0.0 : cax;
        cprev = (rs[q] - alo * cprev) * apr[q];
        xs[p * lwp + l] = cprev;
      }
    }
  } else {
    double aprev = 0.0;
    for (int p0 = 0; p0 < len; p0 += TDMA_CHUNK) {
      double rs[TDMA_CHUNK], ap[TDMA_CHUNK], alo[TDMA_CHUNK], ahi[TDMA_CHUNK];
#pragma unroll
      for (int q = 0; q < TDMA_CHUNK; ++q) {
        const int p = min(p0 + q, len - 1);
        tdma_cell<PASS>(u, v, p, i, j, k);
        const Coef<double> c = smoother_coef(L, i, j, k);
        rs[q] = xs[p * lwp + l];
        ap[q] = c.ap;
        alo[q] = PASS == 0 ? c.as : PASS == 1 ? c.aw : c.ab;
        ahi[q] = PASS == 0 ? c.an : PASS == 1 ? c.ae : c.at;
      }
#pragma unroll
      for (int q = 0; q < TDMA_CHUNK; ++q) {
        const int p = p0 + q;
        if (p >= len) break;
        const double a_r = 1.0 / (ap[q] - alo[q] * aprev);
        aprev = ahi[q] * a_r;
        cprev = (rs[q] - alo[q] * cprev) * a_r;
        xs[p * lwp + l] = cprev;
        av[p * lwp + l] = aprev;
      }
    }
  }
  tdma_cell<PASS>(u, v, len, i, j, k);
  double next = before_sweep(L, src, zero, i, j, k);
  // colour-split index of position p: base + p*step (j- and k-lines) or
  // base + p/2 (i-lines); colour (u+v+p) & 1.  The level's fields stay in
  // registers across the stores.
  gmem<double> *const out0 = (gmem<double> *)L.phi[dst][0];
  gmem<double> *const out1 = (gmem<double> *)L.phi[dst][1];
  const int base = PASS == 0 ? v * nj * H + (u >> 1) : PASS == 1 ? (v * nj + u) * H : v * H + (u >> 1);
  const int step = PASS == 0 ? H : PASS == 1 ? 0 : nj * H;
  for (int p1 = len - 1; p1 >= 0; p1 -= TDMA_CHUNK) {
    double cv[TDMA_CHUNK], aq[TDMA_CHUNK];
#pragma unroll
    for (int q = 0; q < TDMA_CHUNK; ++q) {
      const int p = max(p1 - q, 0);
      cv[q] = xs[p * lwp + l];
      aq[q] = av[p * lwp + l];
    }
#pragma unroll
    for (int q = 0; q < TDMA_CHUNK; ++q) {
      const int p = p1 - q;
      if (p < 0) break;
      next = cv[q] - aq[q] * next;
      const int e = PASS == 1 ? base + (p >> 1) : base + p * step;
      (((u + v + p) & 1) ? out1 : out0)[e] = next;
      if (PREV) prev[u * len + p] = next;
    }
  }
}

// one diagonal of one pass over groups of tdma_group_lines(len) lines
// (Tile::x0 = the group's first line)
template <int PASS>
__global__ void __launch_bounds__(NTHREADS)
    k_tdma_diag(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                const int *__restrict__ active, int d, int src, int zero) {
  __shared__ double xs[2 * TDMA_CELLS];  // rs, then c
  __shared__ double av[2 * TDMA_CELLS];  // a
  __shared__ double rv[2 * TDMA_CELLS];  // 1/(ap - alo*a(p-1)) (constant coefficients)
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const TdmaGeom<PASS> G(L);
  const int lw = tdma_group_lines(G.len), lwp = lw > 1 ? lw + 1 : 1;
  const int u0 = t.x0;
  if (max(u0, d - G.nv + 1) >= min(min(u0 + lw, G.nu), d + 1)) return;  // no line of d
  tdma_diagonal<PASS, TDMA_CELLS / NTHREADS>(L, u0, lw, lwp, d, src, zero, xs, av, rv,
                                            (int)threadIdx.x + TILE_X * (int)threadIdx.y);
}

// a whole TDMA sweep (three passes, every diagonal) of one small level in
// one workgroup per block: every line of a diagonal in dynamic LDS,
// 3 * (nu+1) * len doubles (tdma_sweep_lds_bytes)
template <int PASS>
__device__ __forceinline__ void tdma_pass_in_group(const LevelDev &L, int src, int zero, double *buf, int tid) {
  const TdmaGeom<PASS> G(L);
  const int lwp = G.nu + 1;
  const size_t n = (size_t)lwp * G.len;
  for (int d = 0; d < G.nu + G.nv - 1; ++d) {
    tdma_diagonal<PASS, TDMA_SWEEP_CPT, TDMA_SWEEP_THREADS, true>(
        L, 0, G.nu, lwp, d, src, zero, buf, buf + n, buf + 2 * n, tid, buf + 3 * n);
    __syncthreads();  // the diagonal's phi before the next one reads it
  }
}

// One TDMA pass of a constant-coefficient level in one workgroup, pipelined
// over the diagonals.  Diagonal d's right-hand sides need the solution of
// diagonal d-1 only through its two updated cross terms, so phase A splits:
//   A0 (everything that does not depend on diagonal d-1: the rhs, the two
//      not-updated cross terms, ghost images, the lines' end ghosts) runs
//      for diagonal d+1 on the waves that phase B does not use, while
//   B (the Thomas recurrence of diagonal d, one thread per line) runs on
//      the first waves;
//   A1 (the updated cross terms from the previous diagonal's solution in
//      LDS, and the last subtractions) runs for every cell between them.
// The reference's left-to-right sum r - x1*X1 - x2*X2 - x3*X3 - x4*X4 is
// kept: A0 forms t1 = r - x1*X1 and the product x3*X3, A1 finishes
// ((t1 - x2*X2) - x3*X3) - x4*X4.  X2 and X4 are the updated neighbours
// (pass 0: W on line (u-1, v) and B on (u, v-1); pass 1: S on (u-1, v), B
// on (u, v-1); pass 2: S on (u, v-1), W on (u-1, v)); a neighbour that is a
// ghost (its line coordinate 0) is an image before the sweep, taken by A0.
// The Thomas tables of the pass (a(p), 1/(ap - alo*a(p-1)) per wall state)
// sit in LDS for the whole pass.  LDS, doubles (tdma_sweep_lds_bytes):
// t1, x3*X3, rs/c: 3*(nu+1)*len; tables 32*len; previous diagonal nu*len;
// ghosts of the first line 2*len; line-end ghosts 2 x 2*nu.
template <int PASS>
__device__ __forceinline__ void tdma_pass_pipelined(const LevelDev &L, int src, int zero,
                                                    double *buf, int tid) {
  const TdmaGeom<PASS> G(L);
  const int nu = G.nu, nv = G.nv, len = G.len, lwp = nu + 1;
  const size_t n = (size_t)lwp * len;
  double *const t1 = buf, *const p3 = buf + n, *const xs = buf + 2 * n;
  double *const T = buf + 3 * n;
  double *const prev = T + (size_t)32 * len;
  double *const gA = prev + (size_t)nu * len;  // term 2's ghost values (line coordinate 0)
  double *const gB = gA + len;                 // term 4's ghost values
  double *const cg = gB + len;                 // [2][2*nu]: c(0) and phi(len) ghosts per line
  constexpr bool U2 = PASS != 2;               // term 2 lies along u (else along v)
  const int nb = 64 * ((nu + 63) / 64);        // phase-B threads (whole waves)
  const int na = TDMA_SWEEP_THREADS - nb;      // A0 threads
  const int dst = 1 - src;
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  const gmem<char> *const s0 = (const gmem<char> *)L.phi[src][0];
  const long long o_s1 = (const char *)L.phi[src][1] - (const char *)L.phi[src][0];
  const long long o_d0 = (const char *)L.phi[dst][0] - (const char *)L.phi[src][0];
  const long long o_d1 = (const char *)L.phi[dst][1] - (const char *)L.phi[src][0];
  // as tdma_diagonal's: ghosts are images in src; interior neighbours
  // updated ones and (after the first pass) not-yet-updated ones in dst
  auto cross = [=](int x, int y, int z, bool updated) -> double {
    const bool ghost = (unsigned)x >= (unsigned)ni || (unsigned)y >= (unsigned)nj ||
                       (unsigned)z >= (unsigned)nk;
    x = image(x, ni, px);
    y = image(y, nj, py);
    z = image(z, nk, pz);
    const bool from_dst = !ghost && (updated || PASS > 0);
    const bool odd = (x + y + z) & 1;
    const long long o = from_dst ? (odd ? o_d1 : o_d0) : (odd ? o_s1 : 0);
    const double val = *(const gmem<double> *)(s0 + o + 8 * (((long long)z * nj + y) * H + (x >> 1)));
    return (zero && !from_dst) ? 0.0 : val;
  };
  const float inv_len = 1.0f / (float)len;  // q / len, exact while q < 2^12 * len
  const int nd = nu + nv - 1;

  // A0 of diagonal d on threads [t0, t0 + cnt): CPT cells a batch, every
  // load of a batch issued before its first LDS store; then the "extra"
  // items: the ghost terms of the lines whose term-2 or term-4 coordinate is
  // 0 (one line each: items [0, 2*len)) and the lines' end ghosts c(0),
  // phi(len) (items [2*len, 2*len + 2*lines)).
  auto a0 = [=, &L](int d, int t0, int cnt) {
    constexpr int CPT = 5;
    const int ulo = max(0, d - nv + 1), uhi = min(nu, d + 1);
    const int ncell = (uhi - ulo) * len;
    // term 2's ghost line: u == 0 (passes 0, 1) or v == 0 (pass 2); term
    // 4's: v == 0 (passes 0, 1) or u == 0 (pass 2)
    const int ua = U2 ? 0 : d, ub = U2 ? d : 0;  // the line of each, if on d
    const bool has_a = ua >= ulo && ua < uhi, has_b = ub >= ulo && ub < uhi;
    const int nextra = 2 * len + 2 * (uhi - ulo);
    double *const cgd = cg + (d & 1) * 2 * nu;
    // item e: its value and its LDS index from buf (-1: nothing to store)
    struct Item {
      double v;
      int at;
    };
    auto extra = [=, &L](int e) -> Item {
      int i, j, k;
      if (e < 2 * len) {
        const bool second = e >= len;
        const int p = second ? e - len : e;
        if (second ? !has_b : !has_a) return Item{0.0, -1};
        const int u = second ? ub : ua, v = d - u;
        tdma_cell<PASS>(u, v, p, i, j, k);
        const int at = (int)(((second ? gB : gA) + p) - buf);
        if (PASS == 0)
          return Item{second ? cross(i, j, k - 1, true) : cross(i - 1, j, k, true), at};
        if (PASS == 1)
          return Item{second ? cross(i, j, k - 1, true) : cross(i, j - 1, k, true), at};
        return Item{second ? cross(i - 1, j, k, true) : cross(i, j - 1, k, true), at};
      }
      const int q = e - 2 * len, u = ulo + (q >> 1), v = d - u;
      tdma_cell<PASS>(u, v, (q & 1) ? len : -1, i, j, k);
      return Item{before_sweep(L, src, zero, i, j, k), (int)((cgd + 2 * u + (q & 1)) - buf)};
    };
    for (int q0 = 0; q0 < ncell; q0 += CPT * cnt) {
      double tv[CPT], pv[CPT];
      int slot[CPT];
#pragma unroll
      for (int it = 0; it < CPT; ++it) {
        const int q = min(q0 + t0 + it * cnt, ncell - 1);
        const int lq = (int)(((float)q + 0.5f) * inv_len);
        const int p = q - lq * len, u = ulo + lq, v = d - u;
        int i, j, k;
        tdma_cell<PASS>(u, v, p, i, j, k);
        const Coef<double> c = cell_coef<double>(L, i, j, k);
        const double r = gload(L.rhs[(i + j + k) & 1], cidx(H, nj, i, j, k));
        if (PASS == 0) {
          tv[it] = r - c.ae * cross(i + 1, j, k, false);
          pv[it] = c.at * cross(i, j, k + 1, false);
        } else if (PASS == 1) {
          tv[it] = r - c.an * cross(i, j + 1, k, false);
          pv[it] = c.at * cross(i, j, k + 1, false);
        } else {
          tv[it] = r - c.an * cross(i, j + 1, k, false);
          pv[it] = c.ae * cross(i + 1, j, k, false);
        }
        slot[it] = p * lwp + u;
      }
#pragma unroll
      for (int it = 0; it < CPT; ++it)
        if (q0 + t0 + it * cnt < ncell) {
          t1[slot[it]] = tv[it];
          p3[slot[it]] = pv[it];
        }
    }
    for (int e = t0; e < nextra; e += cnt) {
      const Item x = extra(e);
      if (x.at >= 0) buf[x.at] = x.v;
    }
  };

  // the pass's Thomas tables into LDS, and A0 of diagonal 0
  for (int q = tid; q < 16 * len; q += TDMA_SWEEP_THREADS) {
    const size_t t = tdma_table_offset<PASS>(L) + (size_t)2 * q;
    T[2 * q] = gload(L.tdma, t);
    T[2 * q + 1] = gload(L.tdma, t + 1);
  }
  a0(0, tid, TDMA_SWEEP_THREADS);
  __syncthreads();
  const double cax = PASS == 0 ? L.cy : PASS == 1 ? L.cx : L.cz;
  const bool pax = PASS == 0 ? (L.per & 2) : PASS == 1 ? (L.per & 1) : (L.per & 4);
  gmem<double> *const out0 = (gmem<double> *)L.phi[dst][0];
  gmem<double> *const out1 = (gmem<double> *)L.phi[dst][1];
  for (int d = 0; d < nd; ++d) {
    const int ulo = max(0, d - nv + 1), uhi = min(nu, d + 1);
    // A1: the updated cross terms and the last subtractions, every cell,
    // four a batch (every LDS read of a batch before its first store)
    const int ncell = (uhi - ulo) * len;
    for (int q0 = 0; q0 < ncell; q0 += 4 * TDMA_SWEEP_THREADS) {
      double rs[4];
      int sl[4];
#pragma unroll
      for (int it = 0; it < 4; ++it) {
        const int q = min(q0 + tid + it * TDMA_SWEEP_THREADS, ncell - 1);
        const int lq = (int)(((float)q + 0.5f) * inv_len);
        const int p = q - lq * len, u = ulo + lq, v = d - u;
        int i, j, k;
        tdma_cell<PASS>(u, v, p, i, j, k);
        const Coef<double> c = cell_coef<double>(L, i, j, k);
        const double x2 = PASS == 0 ? c.aw : c.as;
        const double x4 = PASS == 2 ? c.aw : c.ab;
        const bool in2 = U2 ? u > 0 : v > 0, in4 = U2 ? v > 0 : u > 0;
        const double X2 = in2 ? prev[(U2 ? u - 1 : u) * len + p] : gA[p];
        const double X4 = in4 ? prev[(U2 ? u : u - 1) * len + p] : gB[p];
        sl[it] = p * lwp + u;
        rs[it] = ((t1[sl[it]] - x2 * X2) - p3[sl[it]]) - x4 * X4;
      }
#pragma unroll
      for (int it = 0; it < 4; ++it)
        if (q0 + tid + it * TDMA_SWEEP_THREADS < ncell) xs[sl[it]] = rs[it];
    }
    __syncthreads();
    if (tid < nb) {
      // B: the reference's recurrence, one thread per line
      const int u = tid, v = d - u;
      if (u >= ulo && u < uhi) {
        const double *const cgd = cg + (d & 1) * 2 * nu;
        const int var = wall_state(u, nu, G.pu) | (wall_state(v, nv, G.pv) << 2);
        const double *const Tv = T + (size_t)2 * var * len;
        double cprev = cgd[2 * u];
        for (int p0 = 0; p0 < len; p0 += TDMA_CHUNK) {
          double rs[TDMA_CHUNK], apr[TDMA_CHUNK];
#pragma unroll
          for (int q = 0; q < TDMA_CHUNK; ++q) {
            const int p = min(p0 + q, len - 1);
            rs[q] = xs[p * lwp + u];
            apr[q] = Tv[2 * p + 1];
          }
#pragma unroll
          for (int q = 0; q < TDMA_CHUNK; ++q) {
            const int p = p0 + q;
            if (p >= len) break;
            const double alo = (p == 0 && !pax) ? 0.0 : cax;
            cprev = (rs[q] - alo * cprev) * apr[q];
            xs[p * lwp + u] = cprev;
          }
        }
        double next = cgd[2 * u + 1];
        const int base =
            PASS == 0 ? v * nj * H + (u >> 1) : PASS == 1 ? (v * nj + u) * H : v * H + (u >> 1);
        const int step = PASS == 0 ? H : PASS == 1 ? 0 : nj * H;
        for (int p1 = len - 1; p1 >= 0; p1 -= TDMA_CHUNK) {
          double cv[TDMA_CHUNK], aq[TDMA_CHUNK];
#pragma unroll
          for (int q = 0; q < TDMA_CHUNK; ++q) {
            const int p = max(p1 - q, 0);
            cv[q] = xs[p * lwp + u];
            aq[q] = Tv[2 * p];
          }
#pragma unroll
          for (int q = 0; q < TDMA_CHUNK; ++q) {
            const int p = p1 - q;
            if (p < 0) break;
            next = cv[q] - aq[q] * next;
            const int e = PASS == 1 ? base + (p >> 1) : base + p * step;
            (((u + v + p) & 1) ? out1 : out0)[e] = next;
            prev[u * len + p] = next;
          }
        }
      }
    } else if (d + 1 < nd) {
      a0(d + 1, tid - nb, na);
    }
    __syncthreads();  // prev and the next diagonal's A0 before A1 reads them
  }
}

// One TDMA pass of a constant-coefficient level whose lines and lanes have at
// most 64 cells, in two launches.
//
// A pass walks the diagonals u + v of its lines in order (line-wise GS); a
// line needs the solution of its two neighbours on the previous diagonal.
// The critical path is (lines' diagonals) x (forward + back substitution),
// and everything else is moved off it:
//   k_tdma_pre (the whole GPU, a thread per cell): everything known before
//     the pass -- the rhs, the two not-yet-updated cross terms, ghosts --
//     as t1 = r - x1*X1 and p3 = x3*X3 per cell, stored diagonal by
//     diagonal, so that the pass reads whole rows of 16-byte entries;
//   k_tdma_lines (one workgroup per block): wave 0 is the recurrence, a lane
//     per line, the line in registers between the two substitutions.  The
//     updated neighbours are the lane's own last solution and the next lower
//     lane's, which the back substitution leaves in LDS.  The other waves
//     load the next diagonal's entries while the forward substitution runs,
//     put them into LDS during the back substitution, and store the
//     solutions.
// Lanes are the axis of the second cross term, steps the axis of the fourth:
//   pass 0 (j-lines): lanes i, steps k;  ae*E, aw*W, at*T, ab*B
//   pass 1 (i-lines): lanes j, steps k;  an*N, as*S, at*T, ab*B
//   pass 2 (k-lines): lanes j, steps i;  an*N, as*S, ae*E, aw*W
// The reference's left-to-right sum is kept: ((t1 - x2*X2) - p3) - x4*X4.
// Where the second term's neighbour is a ghost (lane 0), the pass takes it
// with t1 (the product is the next subtraction anyway); the fourth term's
// ghost line (step 0) starts as the lane's "last solution".
//
// Bound by the dependent chain of FP64 operations, 3 per position forward
// and 2 back: ~120 cycles per position and diagonal of the ~100 that five
// dependent operations of 20 cycles take.  A 64^3 pass takes 415 us + 5 us of
// k_tdma_pre where the one-workgroup pipelined sweep took 1.1 ms, a 32^3 one
// 100 us where it took 350 us.
// waves of the workgroup: the recurrence's and the ones that load and store.
// Four leave each wave a SIMD's whole register file, which 64-cell lines need
constexpr int tl_waves(int len) { return len > 56 ? 4 : 5; }
constexpr int TL_ROW = 66;  // doubles per row of solutions in LDS

// a pass's axes: lane, step and line coordinates of cell (i, j, k)
struct TlAxes {
  int nl, ns, len;  // lanes, steps, cells per line
  int w;            // entries per diagonal: min(nl, ns)
};
__host__ __device__ inline TlAxes tl_axes(int pass, int ni, int nj, int nk) {
  TlAxes a;
  a.nl = pass == 0 ? ni : nj;
  a.ns = pass == 2 ? ni : nk;
  a.len = pass == 0 ? nj : pass == 1 ? ni : nk;
  a.w = a.nl < a.ns ? a.nl : a.ns;
  return a;
}
// workspace of one block (doubles): entries (t1, p3) at ((d*len + p)*w +
// lane - first lane of d), line-end ghosts (2 per line) at (step*nl + lane),
// ghost lines of step -1 at (p*nl + lane)
__host__ __device__ inline size_t tl_entries(const TlAxes &a) {
  return (size_t)2 * (a.nl + a.ns - 1) * a.len * a.w;
}
__host__ __device__ inline size_t tl_ends(const TlAxes &a) { return (size_t)2 * a.nl * a.ns; }

// Tile: natural tiles (TILE_X x TILE_Y cells of one plane)
template <int PASS>
__global__ void __launch_bounds__(NTHREADS)
    k_tdma_pre(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
               const int *__restrict__ active, int src, int zero) {
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const int i = t.x0 + (int)threadIdx.x, j = t.y0 + (int)threadIdx.y, k = t.z0;
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H;
  if (i >= ni || j >= nj) return;
  const TlAxes A = tl_axes(PASS, ni, nj, nk);
  const int u = PASS == 0 ? i : j, v = PASS == 2 ? i : k, p = PASS == 0 ? j : PASS == 1 ? i : k;
  const bool px = L.per & 1, py = L.per & 2, pz = L.per & 4;
  const int dst = 1 - src;
  const bool from_dst = PASS > 0;
  // a not-yet-updated cross neighbour (interior: dst after the first pass,
  // else src) or a ghost (its image in src); src reads are 0 when it holds
  // zeros
  auto val = [&](int x, int y, int z) -> double {
    const bool ghost = (unsigned)x >= (unsigned)ni || (unsigned)y >= (unsigned)nj ||
                       (unsigned)z >= (unsigned)nk;
    const bool d = from_dst && !ghost;
    x = image(x, ni, px);
    y = image(y, nj, py);
    z = image(z, nk, pz);
    const double q = gload(L.phi[d ? dst : src][(x + y + z) & 1], cidx(H, nj, x, y, z));
    return (zero && !d) ? 0.0 : q;
  };
  const Coef<double> c = cell_coef<double>(L, i, j, k);
  const double r = gload(L.rhs[(i + j + k) & 1], cidx(H, nj, i, j, k));
  double t1, p3;
  if (PASS == 0) {
    t1 = r - c.ae * val(i + 1, j, k);
    p3 = c.at * val(i, j, k + 1);
    if (u == 0) t1 = t1 - c.aw * val(-1, j, k);
  } else if (PASS == 1) {
    t1 = r - c.an * val(i, j + 1, k);
    p3 = c.at * val(i, j, k + 1);
    if (u == 0) t1 = t1 - c.as * val(i, -1, k);
  } else {
    t1 = r - c.an * val(i, j + 1, k);
    p3 = c.ae * val(i + 1, j, k);
    if (u == 0) t1 = t1 - c.as * val(i, -1, k);
  }
  gmem<double> *const ws = (gmem<double> *)L.tdma_ws;
  const int d = u + v, ulo = max(0, d - A.ns + 1);
  typedef double __attribute__((ext_vector_type(2))) d2;
  *(gmem<d2> *)(ws + 2 * (((size_t)d * A.len + p) * A.w + (u - ulo))) = d2{t1, p3};
  gmem<double> *const ends = ws + tl_entries(A), *const first = ends + tl_ends(A);
  if (p == 0)
    ends[2 * ((size_t)v * A.nl + u)] =
        PASS == 0 ? val(i, -1, k) : PASS == 1 ? val(-1, j, k) : val(i, j, -1);
  if (p == A.len - 1)
    ends[2 * ((size_t)v * A.nl + u) + 1] =
        PASS == 0 ? val(i, nj, k) : PASS == 1 ? val(ni, j, k) : val(i, j, nk);
  if (v == 0) first[(size_t)p * A.nl + u] = PASS == 2 ? val(-1, j, k) : val(i, j, -1);
}

// back substitution of k_tdma_lines: phi(p) = c(p) - a(p)*phi(p+1), the
// operands a chunk ahead of the chain.  SHORT: any chunk may lie past the
// line's end, not just part of the last one.
template <int LEN, bool SHORT>
__device__ __forceinline__ void tl_back(const double (&cv)[LEN], const lds<double> *a0,
                                        lds<double> *out, int len, double next) {
  constexpr int CH = 8;
  double aq[LEN];
#pragma unroll
  for (int q = 0; q < CH; ++q) aq[LEN - CH + q] = a0[LEN - CH + q];
#pragma unroll
  for (int p1 = LEN - CH; p1 >= 0; p1 -= CH) {
    if (p1 >= CH) {
#pragma unroll
      for (int q = 0; q < CH; ++q) aq[p1 - CH + q] = a0[p1 - CH + q];
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = CH - 1; q >= 0; --q) {
      const int p = p1 + q;
      const double x = cv[p] - aq[p] * next;
      next = (SHORT || p1 == LEN - CH) ? (p < len ? x : next) : x;
      out[p * TL_ROW] = next;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Tile::lev = the block's descriptor.  LEN: the longest line the kernel holds
// in registers (a multiple of the chunk of 8 positions a line's end is looked
// for at).  Dynamic LDS, doubles: entries 2*LEN*64, solutions LEN*TL_ROW (column 0 zeros,
// the neighbour below lane 0; lane u in column u+1; the last column takes
// what lanes whose line has not begun would write),
// tables a(p) and 1/(ap - alo*a(p-1)) 16*LEN each, line-end ghosts 2*64.
template <int LEN>
__global__ void __launch_bounds__(64 * tl_waves(LEN))
    k_tdma_lines(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                 const int *__restrict__ active, int pass, int src) {
  typedef double __attribute__((ext_vector_type(2))) d2;
  constexpr int CH = 8, AHEAD = 6, TL_WAVES = tl_waves(LEN);
  constexpr int ROWS = (LEN + TL_WAVES - 2) / (TL_WAVES - 1);
  static_assert(LEN % CH == 0 && LEN >= CH, "whole chunks");
  extern __shared__ __align__(16) double tl_lds[];
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const int ni = L.ni, nj = L.nj, nk = L.nk, H = L.H, per = L.per;
  const TlAxes A = tl_axes(pass, ni, nj, nk);
  const int nl = A.nl, ns = A.ns, len = A.len, w = A.w;
  const int lane = (int)threadIdx.x & 63,
            wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  lds<d2> *const tb = (lds<d2> *)tl_lds;                    // [LEN][64]
  lds<double> *const yb = (lds<double> *)(tl_lds + 2 * LEN * 64);  // [LEN][TL_ROW]
  lds<double> *const ta = yb + LEN * TL_ROW, *const tr = ta + 16 * LEN;
  lds<d2> *const eb = (lds<d2> *)(tr + 16 * LEN);        // [64]
  const gmem<double> *const ws = (const gmem<double> *)L.tdma_ws;
  const gmem<d2> *const en = (const gmem<d2> *)ws;
  const gmem<d2> *const ends = (const gmem<d2> *)(ws + tl_entries(A));
  const gmem<double> *const first = ws + tl_entries(A) + tl_ends(A);
  const int nd = nl + ns - 1;
  const bool pl = pass == 0 ? per & 1 : per & 2;           // lane axis periodic
  const bool ps = pass == 2 ? per & 1 : per & 4;           // step axis
  const bool pa = pass == 0 ? per & 2 : pass == 1 ? per & 1 : per & 4;  // line axis
  const double cl = pass == 0 ? L.cx : L.cy, cs = pass == 2 ? L.cx : L.cz;
  const double ca = pass == 0 ? L.cy : pass == 1 ? L.cx : L.cz;
  // the pass's tables (both line coordinates' wall states, position)
  const size_t toff = pass == 0 ? 0 : pass == 1 ? (size_t)32 * nj : (size_t)32 * (nj + ni);
  for (int q = (int)threadIdx.x; q < 16 * len; q += 64 * TL_WAVES) {
    const int var = q / len, p = q - var * len;
    ta[var * LEN + p] = gload(L.tdma, toff + 2 * (size_t)q);
    tr[var * LEN + p] = gload(L.tdma, toff + 2 * (size_t)q + 1);
  }
  // entries and line-end ghosts of a diagonal: rows of the helper waves
  const int hw = wave - 1;
  d2 hold[ROWS], hend = d2{0.0, 0.0};
  auto fetch = [&](int d) {
    const gmem<d2> *row = en + (size_t)d * len * w;
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      const int p = min(hw + q * (TL_WAVES - 1), len - 1);
      hold[q] = row[(size_t)p * w + min(lane, w - 1)];
    }
    if (hw == 0) {
      const int u = min(lane, nl - 1), v = min(max(d - u, 0), ns - 1);
      hend = ends[(size_t)v * nl + u];
    }
  };
  auto stage = [&]() {
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
      const int p = hw + q * (TL_WAVES - 1);
      if (p < len) tb[p * 64 + lane] = hold[q];
    }
    if (hw == 0) eb[lane] = hend;
  };
  // the solutions of diagonal d (in yb) to dst
  gmem<double> *const out0 = (gmem<double> *)L.phi[1 - src][0];
  gmem<double> *const out1 = (gmem<double> *)L.phi[1 - src][1];
  auto store = [&](int d) {
    const int u = lane, v = d - u;
    if (u < nl && v >= 0 && v < ns) {
      const int base = pass == 0 ? v * nj * H + (u >> 1) : pass == 1 ? (v * nj + u) * H
                                                                     : u * H + (v >> 1);
      const int step = pass == 0 ? H : pass == 1 ? 0 : nj * H;
#pragma unroll 4
      for (int q = 0; q < ROWS; ++q) {
        const int p = hw + q * (TL_WAVES - 1);
        if (p < len) {
          const int e = pass == 1 ? base + (p >> 1) : base + p * step;
          (((u + v + p) & 1) ? out1 : out0)[e] = yb[p * TL_ROW + 1 + lane];
        }
      }
    }
  };

  // the ghost lines before step 0, and the zeros below lane 0
  for (int q = (int)threadIdx.x; q < LEN * 64; q += 64 * TL_WAVES) {
    const int p = q >> 6, u = q & 63;
    yb[p * TL_ROW + 1 + u] = first[(size_t)min(p, len - 1) * nl + min(u, nl - 1)];
    if (u == 0) yb[p * TL_ROW] = 0.0;
  }
  // each role in its own loop: the registers of one are not held by the
  // other; both pass the same barriers
  if (wave != 0) {
    fetch(0);
    stage();
    lds_barrier();
    for (int d = 0; d < nd; ++d) {
      if (d + 1 < nd) fetch(d + 1);
      if (d > 0) store(d - 1);
      lds_barrier();  // the entries of d are read, the solutions of d-1 stored
      if (d + 1 < nd) stage();
      lds_barrier();  // the entries of d+1 and the solutions of d are in LDS
    }
    store(nd - 1);
    return;
  }
  __builtin_amdgcn_s_setprio(3);
  lds_barrier();
  for (int d = 0; d < nd; ++d) {
    const int u = lane, v = d - u;
    const int ulo = max(0, d - ns + 1);
    const int uc = min(u, nl - 1), vc = min(max(v, 0), ns - 1);
    const int wl = wall_state(uc, nl, pl), wst = wall_state(vc, ns, ps);
    // the tables' state pair is (i, k), (j, k) or (i, j)
    const int var = pass == 2 ? wst | (wl << 2) : wl | (wst << 2);
    const d2 end = eb[lane];
    double cv[LEN];
    // Forward substitution, software-pipelined by hand (the wave issues in
    // order): while the chain m = alo*c, t = rs - m, c = t/(..) of position p
    // waits for its operands, the right-hand sides of the next two positions
    // advance a stage each: x2*X2; t1 - x2*X2, x4*X4; - p3; - x4*X4.  Lanes
    // with no line on this diagonal work on values nobody reads.
    {
      const double x2 = u > 0 ? cl : 0.0, x4 = (v <= 0 && !ps) ? 0.0 : cs;
      const lds<d2> *const e0 = tb + min(max(u - ulo, 0), w - 1);
      const lds<double> *const r0 = tr + var * LEN;
      const lds<double> *const y0 = yb + lane;
      double c = end.x;
      d2 en_[LEN];
      double rr[LEN], X2[LEN], X4[LEN], rs[LEN];
#pragma unroll
      for (int p = 0; p < AHEAD; ++p) {
        en_[p] = e0[p * 64];
        rr[p] = r0[p];
        X2[p] = y0[p * TL_ROW];
        X4[p] = y0[p * TL_ROW + 1];
      }
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        X4[p] = x4 * X4[p];
        rs[p] = ((en_[p].x - x2 * X2[p]) - en_[p].y) - X4[p];
      }
#pragma unroll
      for (int p = 0; p < LEN; ++p) {
        const double m = ((p == 0 && !pa) ? 0.0 : ca) * c;
        if (p + AHEAD < LEN) {
          en_[p + AHEAD] = e0[(p + AHEAD) * 64];
          rr[p + AHEAD] = r0[p + AHEAD];
          X2[p + AHEAD] = y0[(p + AHEAD) * TL_ROW];
          X4[p + AHEAD] = y0[(p + AHEAD) * TL_ROW + 1];
        }
        if (p + 2 < LEN) X2[p + 2] = x2 * X2[p + 2];
        if (p + 1 < LEN && p > 0) rs[p + 1] = rs[p + 1] - en_[p + 1].y;
        __builtin_amdgcn_sched_barrier(0);
        const double t = rs[p] - m;
        if (p + 2 < LEN) X4[p + 2] = x4 * X4[p + 2];
        if (p + 1 < LEN && p > 0) rs[p + 1] = rs[p + 1] - X4[p + 1];
        __builtin_amdgcn_sched_barrier(0);
        c = t * rr[p];
        if (p + 2 < LEN) rs[p + 2] = en_[p + 2].x - X2[p + 2];
        cv[p] = c;
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lds_barrier();
    {
      const lds<double> *const a0 = ta + var * LEN;
      lds<double> *const out = yb + (v >= 0 ? 1 + lane : TL_ROW - 1);
      // positions past the line's end pass by: in the last chunk only, unless
      // the block's lines are shorter than the launch's longest by more
      if (len > LEN - CH)
        tl_back<LEN, false>(cv, a0, out, len, end.y);
      else
        tl_back<LEN, true>(cv, a0, out, len, end.y);
    }
    lds_barrier();
  }
}

__global__ void __launch_bounds__(TDMA_SWEEP_THREADS)
    k_tdma_sweep(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                 const int *__restrict__ active, int src, int zero) {
  extern __shared__ double line_lds[];
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk]) return;
  const int tid = (int)threadIdx.x + TILE_X * (int)threadIdx.y;
  tdma_pass_in_group<0>(L, src, zero, line_lds, tid);
  tdma_pass_in_group<1>(L, src, zero, line_lds, tid);
  tdma_pass_in_group<2>(L, src, zero, line_lds, tid);
}

// the same sweep on a constant-coefficient level, passes pipelined over the
// diagonals (a kernel of its own: its registers do not cost the other one)
__global__ void __launch_bounds__(TDMA_SWEEP_THREADS)
    k_tdma_sweep_pipe(const Tile *__restrict__ tiles, const LevelDev *__restrict__ levs,
                      const int *__restrict__ active, int src, int zero) {
  extern __shared__ double line_lds[];
  const Tile t = tiles[blockIdx.x];
  const LevelDev &L = levs[t.lev];
  if (!active[L.blk] || L.lsm != nullptr || L.tdma == nullptr) return;
  const int tid = (int)threadIdx.x + TILE_X * (int)threadIdx.y;
  tdma_pass_pipelined<0>(L, src, zero, line_lds, tid);
  tdma_pass_pipelined<1>(L, src, zero, line_lds, tid);
  tdma_pass_pipelined<2>(L, src, zero, line_lds, tid);
}

}  // namespace

// ---- launchers -----------------------------------------------------------
template <class T>
void launch_rb_sweep(hipStream_t s, const Tile *tiles, int ntiles, int depth, const LevelDev *levs,
                     const int *active, int colour, int src, int zero, OneDesc one,
                     const FineDev *upd) {
  if (ntiles <= 0) return;
  if (depth == 0) {  // natural tiles, cell by cell
    hipLaunchKernelGGL((k_cell_sweep<T, false>), dim3(ntiles), dim3(TILE_X, TILE_Y / 2), 0, s, tiles,
                       levs, active, colour, src, zero, ntiles);
    return;
  }
  auto pick = [&](auto u) {
    constexpr bool UPD = decltype(u)::value;
    return one.lev >= 0 ? (depth == 4   ? k_rb_sweep<T, 4, true, UPD>
                           : depth == 2 ? k_rb_sweep<T, 2, true, UPD>
                                        : k_rb_sweep<T, 1, true, UPD>)
                        : (depth == 4   ? k_rb_sweep<T, 4, false, UPD>
                           : depth == 2 ? k_rb_sweep<T, 2, false, UPD>
                                        : k_rb_sweep<T, 1, false, UPD>);
  };
  auto k = upd ? pick(std::true_type()) : pick(std::false_type());
  hipLaunchKernelGGL(k, dim3(ntiles), tile_block(), 0, s, tiles, levs, active, colour, src, zero,
                     one.lev, one.blk, ntiles, upd);
}

void launch_lsm_dens_restrict(hipStream_t s, const double *fine, int fni, int fnj, int fnk,
                              double *coarse) {
  const size_t n = (size_t)(fni / 2) * (fnj / 2) * (fnk / 2);
  if (!n) return;
  hipLaunchKernelGGL(k_lsm_dens_restrict, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, fine,
                     fni, fnj, fnk, coarse);
}

void launch_lsm_coef(hipStream_t s, const LevelDev *lev_dev, const double *dens, int ni, int nj,
                     int nk, double dx, double dy, double dz, int walls) {
  const size_t n = (size_t)ni * nj * nk;
  hipLaunchKernelGGL(k_lsm_coef, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, lev_dev, dens,
                     ni, nj, nk, dx, dy, dz, walls);
}

void launch_lsm_sweep(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                      const int *active, int colour, int src, int zero) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL((k_cell_sweep<double, true>), dim3(ntiles), dim3(TILE_X, TILE_Y / 2), 0, s,
                     tiles, levs, active, colour, src, zero, ntiles);
}

void launch_gs_tiles(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                     const int *active, int src, int zero, int tile) {
  if (ntiles <= 0) return;
  if (tile == GS_BIG_TILE)
    hipLaunchKernelGGL(k_gs_tile_big, dim3(ntiles), dim3(GS_BIG_TILE * GS_BIG_TILE), GS_BIG_LDS,
                       s, tiles, levs, active, src, zero);
  else
    hipLaunchKernelGGL(k_gs_tile, dim3(ntiles), dim3(GS_TILE * GS_TILE), 0, s, tiles, levs,
                       active, src, zero);
}

hipError_t gs_allow_lds() {
  return hipFuncSetAttribute((const void *)k_gs_tile_big,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)GS_BIG_LDS);
}

void launch_tdma_diag(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                      const int *active, int pass, int d, int src, int zero) {
  if (ntiles <= 0) return;
  auto k = pass == 0 ? k_tdma_diag<0> : pass == 1 ? k_tdma_diag<1> : k_tdma_diag<2>;
  hipLaunchKernelGGL(k, dim3(ntiles), tile_block(), 0, s, tiles, levs, active, d, src, zero);
}

void launch_tdma_sweep(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                       const int *active, int src, int zero, size_t lds_bytes, bool pipelined) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL(pipelined ? k_tdma_sweep_pipe : k_tdma_sweep, dim3(ntiles),
                     dim3(TILE_X, TDMA_SWEEP_THREADS / TILE_X), lds_bytes, s, tiles, levs, active,
                     src, zero);
}

hipError_t tdma_sweep_allow_lds(size_t lds_bytes) {
  hipError_t e = hipFuncSetAttribute((const void *)k_tdma_sweep,
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
  if (e != hipSuccess) return e;
  return hipFuncSetAttribute((const void *)k_tdma_sweep_pipe,
                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
}

size_t tdma_ws_doubles(const LevelDev &L) {
  size_t most = 0;
  for (int pass = 0; pass < 3; ++pass) {
    const TlAxes a = tl_axes(pass, L.ni, L.nj, L.nk);
    most = std::max(most, tl_entries(a) + tl_ends(a) + (size_t)a.len * a.nl);
  }
  return most;
}

bool tdma_lines_fit(const LevelDev &L) {
  return std::max(L.ni, std::max(L.nj, L.nk)) <= TDMA_LINES_MAX;
}

// LEN of the kernel for lines of at most `len` cells
static int tl_len(int len) { return (len + 7) & ~7; }

size_t tdma_lines_lds(int maxlen) {
  const size_t len = (size_t)tl_len(maxlen);
  return sizeof(double) * (2 * len * 64 + len * TL_ROW + 32 * len + 128);
}

// by tl_len / 8 - 1
static void (*const tl_kernels[8])(const Tile *, const LevelDev *, const int *, int, int) = {
    k_tdma_lines<8>,  k_tdma_lines<16>, k_tdma_lines<24>, k_tdma_lines<32>,
    k_tdma_lines<40>, k_tdma_lines<48>, k_tdma_lines<56>, k_tdma_lines<64>};

hipError_t tdma_lines_allow_lds() {
  const int most = (int)tdma_lines_lds(TDMA_LINES_MAX);
  for (auto k : tl_kernels) {
    hipError_t e = hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       most);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

void launch_tdma_pass(hipStream_t s, const Tile *nat, int nnat, const Tile *blocks, int nblocks,
                      const LevelDev *levs, const int *active, int pass, int maxlen, int src,
                      int zero) {
  if (nblocks <= 0) return;
  auto pre = pass == 0 ? k_tdma_pre<0> : pass == 1 ? k_tdma_pre<1> : k_tdma_pre<2>;
  hipLaunchKernelGGL(pre, dim3(nnat), tile_block(), 0, s, nat, levs, active, src, zero);
  hipLaunchKernelGGL(tl_kernels[tl_len(maxlen) / 8 - 1], dim3(nblocks), dim3(64 * tl_waves(tl_len(maxlen))), tdma_lines_lds(maxlen), s, blocks,
                     levs, active, pass, src);
}

void launch_tdma_tables(hipStream_t s, const LevelDev *levs, int ndesc) {
  if (ndesc <= 0) return;
  hipLaunchKernelGGL(k_tdma_tables, dim3((unsigned)((ndesc * 48 + 255) / 256)), dim3(256), 0, s,
                     levs, ndesc);
}

size_t tdma_sweep_lds_bytes(const LevelDev &L, bool pipelined) {
  // per pass (nu lines of len cells): rs/c, a and 1/(ap - alo*a) (or, for
  // the pipelined passes, t1, x3*X3 and rs/c) for (nu+1)*len positions, the
  // previous diagonal's solution, nu*len; pipelined passes also the tables
  // (32*len), the first lines' ghosts (2*len) and the line-end ghosts (4*nu)
  size_t most = 0;
  const int geo[3][2] = {{L.ni, L.nj}, {L.nj, L.ni}, {L.ni, L.nk}};  // (nu, len) per pass
  for (const auto &g : geo) {
    const size_t nu = (size_t)g[0], len = (size_t)g[1];
    size_t need = 3 * (nu + 1) * len + nu * len;
    if (pipelined) need += 32 * len + 2 * len + 4 * nu;
    most = std::max(most, need);
  }
  return most * sizeof(double);
}

void launch_lsm_residual(hipStream_t s, const Tile *tiles, int ntiles, const FineDev *fine,
                         const LevelDev *levs, const int *active, RedPartial *partials) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL(k_lsm_residual, dim3(ntiles), tile_block(), 0, s, tiles, fine, levs, active,
                     partials);
}

void launch_lsm_restrict(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                         const int *active, int src_f) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL((k_cell_restrict<double, double, true>), dim3(ntiles, TILE_Y), tile_block(), 0,
                     s, tiles, levs, active, src_f, ntiles);
}

template <class T>
void launch_rb_tile(hipStream_t s, const LevelDev *levs, const int *active, int src, int zero,
                    OneDesc one, int ni, int nj, int nk, const FineDev *upd) {
  auto n = [](int c) { return (c + 7) / 8; };
  const int ntiles = n(ni) * n(nj) * n(nk);
  hipLaunchKernelGGL(k_rb_tile<T>, dim3(ntiles), dim3(RBT_THREADS), 0, s, levs, active, src, zero,
                     one.lev, one.blk, n(ni), n(nj), ntiles, upd);
}

template <class T>
void launch_rb_fused(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                     const int *active, int src, int zero) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL(k_rb_fused<T>, dim3(ntiles), tile_block(), 0, s, tiles, levs, active, src,
                     zero);
}

template <class Tf, class Tc>
void launch_restrict(hipStream_t s, const Tile *tiles, int ntiles, int depth, const LevelDev *levs,
                     const int *active, int src_f, OneDesc one, int zbuf) {
  if (ntiles <= 0) return;
  if (depth == 0) {  // natural tiles of the coarse level, blocks with neighbours
    hipLaunchKernelGGL((k_cell_restrict<Tf, Tc, false>), dim3(ntiles, TILE_Y), tile_block(), 0, s,
                       tiles, levs, active, src_f, ntiles);
    return;
  }
  auto k = one.lev >= 0 ? (depth == 4   ? k_restrict<Tf, Tc, 4, true>
                           : depth == 2 ? k_restrict<Tf, Tc, 2, true>
                                        : k_restrict<Tf, Tc, 1, true>)
                        : (depth == 4   ? k_restrict<Tf, Tc, 4, false>
                           : depth == 2 ? k_restrict<Tf, Tc, 2, false>
                                        : k_restrict<Tf, Tc, 1, false>);
  hipLaunchKernelGGL(k, dim3(ntiles), tile_block(), 0, s, tiles, levs, active, src_f, one.lev,
                     one.lev2, one.blk, ntiles, zbuf);
}

template <class Tf, class Tc>
void launch_prolong(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                    const int *active, int src_f, int src_c, int gen, int skip_red, OneDesc one) {
  if (ntiles <= 0) return;
  if (gen)
    hipLaunchKernelGGL((k_prolong<Tf, Tc, true, false>), dim3(ntiles), tile_block(), 0, s, tiles,
                       levs, active, src_f, src_c, -1, -1, -1, ntiles,
                       skip_red);
  else if (one.lev >= 0)
    hipLaunchKernelGGL((k_prolong<Tf, Tc, false, true>), dim3(ntiles), tile_block(), 0, s, tiles,
                       levs, active, src_f, src_c, one.lev, one.lev2, one.blk, ntiles, skip_red);
  else
    hipLaunchKernelGGL((k_prolong<Tf, Tc, false, false>), dim3(ntiles), tile_block(), 0, s, tiles,
                       levs, active, src_f, src_c, -1, -1, -1, ntiles,
                       skip_red);
}

template <class T>
void launch_fill_zero(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                      const int *active, int buf) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL(k_fill_zero<T>, dim3(ntiles), tile_block(), 0, s, tiles, levs, active, buf);
}

template <class T>
void launch_residual(hipStream_t s, const Tile *tiles, int ntiles, int depth, const FineDev *fine,
                     const LevelDev *levs, const int *active, RedPartial *partials, int use_p,
                     int zbuf) {
  if (ntiles <= 0) return;
  if (!use_p || depth <= 0) {
    hipLaunchKernelGGL(k_residual_gen<T>, dim3(ntiles), tile_block(), 0, s, tiles, fine, levs,
                       active, partials, use_p);
    return;
  }
  auto k = depth == 8   ? k_residual<T, 8>
           : depth == 4 ? k_residual<T, 4>
           : depth == 2 ? k_residual<T, 2>
                        : k_residual<T, 1>;
  hipLaunchKernelGGL(k, dim3(ntiles), tile_block(), 0, s, tiles, fine, levs, active, partials,
                     zbuf);
}

template <class T>
void launch_set_rhs(hipStream_t s, const Tile *tiles, int ntiles, int planes, const FineDev *fine,
                    const LevelDev *levs, const double *src, RedPartial *partials) {
  if (ntiles <= 0) return;
  auto k = planes == 8   ? k_set_rhs<T, 8>
           : planes == 4 ? k_set_rhs<T, 4>
           : planes == 2 ? k_set_rhs<T, 2>
                         : k_set_rhs<T, 1>;
  hipLaunchKernelGGL(k, dim3(ntiles), tile_block(), 0, s, tiles, fine, levs, src,
                     partials);
}

template <class T>
void launch_update(hipStream_t s, const Tile *tiles, int ntiles, const FineDev *fine,
                   const LevelDev *levs, const int *active, int buf) {
  if (ntiles <= 0) return;
  hipLaunchKernelGGL(k_update<T>, dim3(ntiles), tile_block(), 0, s, tiles, fine, levs, active,
                     buf);
}

void launch_finalize_decide(hipStream_t s, const int *tile_begin, int nblocks,
                            const RedPartial *partials, RedPartial *out, const DecideBlock *blocks,
                            DecideState *state, DecideCtl *ctl, int *active, char *ring,
                            const DecideParams *prm, unsigned *arrived) {
  hipLaunchKernelGGL(k_finalize_decide, dim3(nblocks), dim3(FIN_THREADS), 0, s, tile_begin,
                     partials, out, blocks, state, ctl, active, ring, prm, arrived);
}

void launch_finalize(hipStream_t s, const int *tile_begin, int nblocks, const RedPartial *partials,
                     RedPartial *out) {
  hipLaunchKernelGGL(k_finalize, dim3(nblocks), dim3(FIN_THREADS), 0, s, tile_begin, partials, out);
}

void launch_coarse_exact(hipStream_t s, const Tile *tiles, int ntiles, const ExactGrid &grid,
                         const LevelDev *levs, const int *active, const double *const *eig_q,
                         const double *const *eig_l, double *const *scratch, int buf) {
  if (ntiles <= 0) return;
  if (grid.plane_lds) {
    const dim3 gp(ntiles, grid.planes), gc(ntiles, grid.chunks);
    hipLaunchKernelGGL(k_exact_plane<true>, gp, dim3(256), grid.plane_lds, s, tiles, levs, active,
                       eig_q, scratch, buf);
    hipLaunchKernelGGL(k_exact_cols, gc, dim3(256), grid.cols_lds, s, tiles, levs, active, eig_q,
                       eig_l, scratch);
    hipLaunchKernelGGL(k_exact_plane<false>, gp, dim3(256), grid.plane_lds, s, tiles, levs, active,
                       eig_q, scratch, buf);
    return;
  }
  for (int p = 0; p < 6; ++p)
    hipLaunchKernelGGL(k_exact_pass, dim3(ntiles, grid.blocks), dim3(256), 0, s, tiles, levs,
                       active, eig_q, eig_l, scratch, buf, p);
}

void exact_grid_add(ExactGrid &g, const LevelDev &L, size_t lds_budget) {
  const size_t p0 = exact_pitch(L.ni), p1 = exact_pitch(L.nj), p2 = exact_pitch(L.nk);
  const size_t plane = 8 * (L.ni * p0 + L.nj * p1 + 2 * p0 * L.nj);
  const size_t cols = 8 * (L.nk * p2 + (2 * (size_t)L.nk + 1) * EXACT_COLS + L.nk);
  const size_t n = (size_t)L.ni * L.nj * L.nk;
  g.split = g.split && plane <= lds_budget && cols <= lds_budget;
  g.plane_lds = g.split ? std::max(g.plane_lds, plane) : 0;
  g.cols_lds = g.split ? std::max(g.cols_lds, cols) : 0;
  g.planes = std::max(g.planes, L.nk);
  g.chunks = std::max(g.chunks, (L.ni * L.nj + EXACT_COLS - 1) / EXACT_COLS);
  g.blocks = std::max<unsigned>(g.blocks, (unsigned)std::min<size_t>((n + 255) / 256, 4096));
}

hipError_t exact_allow_lds(size_t lds_bytes) {
  for (const void *f : {(const void *)k_exact_plane<true>, (const void *)k_exact_plane<false>,
                        (const void *)k_exact_cols}) {
    const hipError_t e =
        hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

void launch_vtail(hipStream_t s, const Tile *tiles, int ntiles, const LevelDev *levs,
                  const int *active, const double *const *eig_q, const double *const *eig_l,
                  int nu1, int nu2, int exact, int mixed, size_t lds_bytes) {
  if (ntiles <= 0) return;
  auto k = !mixed ? k_vtail<false, false> : exact ? k_vtail<true, true> : k_vtail<true, false>;
  hipLaunchKernelGGL(k, dim3(ntiles), dim3(TAIL_THREADS), lds_bytes, s, tiles, levs, active, eig_q,
                     eig_l, nu1, nu2, exact);
}

hipError_t vtail_allow_lds(size_t lds_bytes) {
  for (const void *f : {(const void *)k_vtail<false, false>, (const void *)k_vtail<true, true>,
                        (const void *)k_vtail<true, false>}) {
    const hipError_t e =
        hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

size_t vtail_lds_bytes(const LevelDev *levs_host, int top, bool mixed, bool exact, bool padded) {
  size_t off = 0;
  int last = top, nl = 0;
  for (int d = top; d >= 0 && nl < TAIL_MAX_LEVELS; d = levs_host[d].coarser, ++nl) {
    const LevelDev &L = levs_host[d];
    const bool is64 = !mixed || L.coarser < 0;
    const size_t half = (size_t)L.H * L.nj * L.nk * (is64 ? 8 : 4);
    off += 6 * ((half + 15) & ~(size_t)15) + (padded ? 16 : 0);
    last = d;
  }
  const LevelDev &C = levs_host[last];
  if (exact && C.finer >= 0) {
    const int na[3] = {C.ni, C.nj, C.nk};
    for (int a = 0; a < 3; ++a)
      off += padded ? tail_eig_axis(na[a])
                    : (size_t)na[a] * na[a] * 8 + (((size_t)na[a] * 8 + 15) & ~(size_t)15);
    off += 2 * (size_t)C.ni * C.nj * C.nk * 8;
  }
  return off;
}

void launch_calvel(hipStream_t s, const FineDev *fd, int axis, const double *us, double *u,
                   double dt_alfa, double h, size_t faces) {
  const unsigned grid = (unsigned)std::min<size_t>((faces + 255) / 256, 4096);
  hipLaunchKernelGGL(k_calvel, dim3(grid), dim3(256), 0, s, fd, axis, us, u, dt_alfa, h);
}

void launch_calvel_nb(hipStream_t s, const FineDev *fine, int b, int axis, const double *us,
                      double *u, double dt_alfa, double h, size_t faces) {
  const unsigned grid = (unsigned)std::min<size_t>((faces + 255) / 256, 4096);
  hipLaunchKernelGGL(k_calvel_nb, dim3(grid), dim3(256), 0, s, fine, b, axis, us, u, dt_alfa, h);
}

void launch_face_copy(hipStream_t s, int axis, const double *src, int n_src, double *dst,
                      int n_dst, int nu, int nv) {
  const size_t n = (size_t)nu * nv;
  hipLaunchKernelGGL(k_face_copy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, axis, src,
                     n_src, dst, n_dst, nu, nv);
}

void launch_unpack_fine_padded(hipStream_t s, const FineDev *fine, int b, double *dst, int ni,
                               int nj, int nk) {
  const size_t n = (size_t)(ni + 2) * (nj + 2) * (nk + 2);
  hipLaunchKernelGGL(k_unpack_fine_padded, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                     fine, b, dst);
}

void launch_project(hipStream_t s, const ProjLaunch &a, const FineDev *fine, const LevelDev *levs,
                    const int *active, const VelDev *tab, const ProjDt *dtab, const VelDev &one,
                    const ProjDt &dt_one, int b0, int nblocks, RedPartial *partials) {
  auto k = a.even ? (a.lsm   ? k_project<double, true, true>
                     : a.f32 ? k_project<float, false, true>
                             : k_project<double, false, true>)
                  : (a.lsm   ? k_project<double, true, false>
                     : a.f32 ? k_project<float, false, false>
                             : k_project<double, false, false>);
  hipLaunchKernelGGL(k, dim3(a.groups, nblocks), dim3(NTHREADS), 0, s, fine, levs, active, tab,
                     dtab, one, dt_one, b0, a.kb, a.connected, a.to_fine, a.calmas, partials);
}

int launch_calmas(hipStream_t s, const FineDev *fd, const double *u, const double *v,
                  const double *w, double *su, int to_fine, double dt, double dx, double dy,
                  double dz, RedPartial *partials, size_t cells) {
  const int grid = calmas_groups(cells);
  hipLaunchKernelGGL(k_calmas, dim3(grid), dim3(256), 0, s, fd, u, v, w, su, to_fine, dt, dx, dy,
                     dz, partials);
  return grid;
}

void launch_partials_max(hipStream_t s, const RedPartial *parts, int n, double *out) {
  hipLaunchKernelGGL(k_partials_max, dim3(1), dim3(256), 0, s, parts, n, out);
}

int launch_calmas4(hipStream_t s, const FineDev *fd, const double *u, const double *v,
                   const double *w, double *su, int to_fine, double dt, double dx, double dy,
                   double dz, RedPartial *partials, size_t cells, const Outer4 &outer) {
  const int grid = calmas_groups(cells);
  hipLaunchKernelGGL(k_calmas4, dim3(grid), dim3(256), 0, s, fd, u, v, w, su, to_fine, dt, dx, dy,
                     dz, partials, outer);
  return grid;
}

static void copy_fine_grid(int ni, int nj, int nk, int &lp, int &xb, unsigned &grid) {
  const int half = (ni + 1) / 2;
  lp = 1;
  while (lp < 256 && lp < half) lp *= 2;
  xb = (half + lp - 1) / lp;
  grid = (unsigned)xb * (unsigned)(((size_t)nj * nk + 256 / lp - 1) / (256 / lp));
}

void launch_pack_fine(hipStream_t s, const FineDev *fd, int which, const double *src, int ni,
                      int nj, int nk) {
  int lp, xb;
  unsigned grid;
  copy_fine_grid(ni, nj, nk, lp, xb, grid);
  hipLaunchKernelGGL(k_copy_fine<true>, dim3(grid), dim3(256), 0, s, fd, which,
                     const_cast<double *>(src), lp, xb);
}

void launch_unpack_fine(hipStream_t s, const FineDev *fd, int which, double *dst, int ni, int nj,
                        int nk) {
  int lp, xb;
  unsigned grid;
  copy_fine_grid(ni, nj, nk, lp, xb, grid);
  hipLaunchKernelGGL(k_copy_fine<false>, dim3(grid), dim3(256), 0, s, fd, which, dst, lp, xb);
}

template <class T>
void launch_pack_level(hipStream_t s, const LevelDev *ld, int which, int buf, const double *src,
                       int ni, int nj, int nk) {
  const size_t n = (size_t)ni * nj * nk;
  hipLaunchKernelGGL(k_pack_level<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, ld,
                     which, buf, src, ni, nj, nk);
}

template <class T>
void launch_unpack_level(hipStream_t s, const LevelDev *levs, int d, int which, int buf, double *dst,
                         int ni, int nj, int nk) {
  const size_t n = (size_t)(ni + 2) * (nj + 2) * (nk + 2);
  hipLaunchKernelGGL(k_unpack_level<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, levs, d,
                     which, buf, dst, ni, nj, nk);
}

void launch_remove_mean(hipStream_t s, const FineDev *fd, int ni, int nj, int nk,
                        double * /*scratch*/) {
  hipLaunchKernelGGL(k_remove_mean, dim3(1), dim3(256), 0, s, fd, ni, nj, nk);
}

// explicit instantiations
template void launch_rb_fused<double>(hipStream_t, const Tile *, int, const LevelDev *,
                                      const int *, int, int);
template void launch_rb_fused<float>(hipStream_t, const Tile *, int, const LevelDev *, const int *,
                                     int, int);
template void launch_rb_sweep<double>(hipStream_t, const Tile *, int, int, const LevelDev *,
                                      const int *, int, int, int, OneDesc,
                                      const FineDev *);
template void launch_rb_sweep<float>(hipStream_t, const Tile *, int, int, const LevelDev *,
                                     const int *, int, int, int, OneDesc,
                                      const FineDev *);
template void launch_restrict<double, double>(hipStream_t, const Tile *, int, int, const LevelDev *,
                                              const int *, int, OneDesc, int);
template void launch_restrict<float, float>(hipStream_t, const Tile *, int, int, const LevelDev *,
                                            const int *, int, OneDesc, int);
template void launch_restrict<float, double>(hipStream_t, const Tile *, int, int, const LevelDev *,
                                             const int *, int, OneDesc, int);
template void launch_prolong<double, double>(hipStream_t, const Tile *, int, const LevelDev *,
                                             const int *, int, int, int, int, OneDesc);
template void launch_prolong<float, float>(hipStream_t, const Tile *, int, const LevelDev *,
                                           const int *, int, int, int, int, OneDesc);
template void launch_prolong<float, double>(hipStream_t, const Tile *, int, const LevelDev *,
                                            const int *, int, int, int, int, OneDesc);
template void launch_fill_zero<double>(hipStream_t, const Tile *, int, const LevelDev *,
                                       const int *, int);
template void launch_fill_zero<float>(hipStream_t, const Tile *, int, const LevelDev *,
                                      const int *, int);
template void launch_residual<double>(hipStream_t, const Tile *, int, int, const FineDev *,
                                      const LevelDev *, const int *, RedPartial *, int, int);
template void launch_residual<float>(hipStream_t, const Tile *, int, int, const FineDev *,
                                     const LevelDev *, const int *, RedPartial *, int, int);
template void launch_rb_tile<double>(hipStream_t, const LevelDev *, const int *, int, int, OneDesc,
                                     int, int, int, const FineDev *);
template void launch_rb_tile<float>(hipStream_t, const LevelDev *, const int *, int, int, OneDesc,
                                     int, int, int, const FineDev *);
template void launch_set_rhs<double>(hipStream_t, const Tile *, int, int, const FineDev *,
                                     const LevelDev *, const double *, RedPartial *);
template void launch_set_rhs<float>(hipStream_t, const Tile *, int, int, const FineDev *,
                                    const LevelDev *, const double *, RedPartial *);
template void launch_update<double>(hipStream_t, const Tile *, int, const FineDev *,
                                    const LevelDev *, const int *, int);
template void launch_update<float>(hipStream_t, const Tile *, int, const FineDev *,
                                   const LevelDev *, const int *, int);
template void launch_pack_level<double>(hipStream_t, const LevelDev *, int, int, const double *,
                                        int, int, int);
template void launch_pack_level<float>(hipStream_t, const LevelDev *, int, int, const double *,
                                       int, int, int);
template void launch_unpack_level<double>(hipStream_t, const LevelDev *, int, int, int, double *, int,
                                          int, int);
template void launch_unpack_level<float>(hipStream_t, const LevelDev *, int, int, int, double *, int,
                                         int, int);

}  // namespace h3dmg
