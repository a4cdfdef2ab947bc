// fx_march.hpp -- fused face-state + flux kernel: one workgroup per
// (block, TX x TY column tile), marching along z through the block.
//
// The kernel templates are instantiated in fx_march_inst.hip, one unit per
// (solver family, real type), behind the launchers of fx_march_launch.hpp.
//
// Per z-plane k the workgroup computes, each value once (the work of
// hy_getRiemannState.F90:356-1327 regrouped by quantity instead of by cell):
//   stage A  transverse fluxes sigma_x, sigma_y of plane k+1 into 3-plane LDS
//            rings (they feed the 3-D CTU terms of planes k and k+2) and,
//            from the same stencils, the limited characteristic slopes and
//            the flattening tildes along x and y of plane k+1 into 2-plane
//            rings; sigma_z of plane k; slopes along z (with the z
//            flattening tilde) of plane k+1 into 3-plane rings
//   stage B  x-, y- and z-face states of plane k: PPM with characteristic
//            tracing, 2-D CTU transverse corrections, 3-D full-CTU corner
//            terms, positivity fallback after either
//   stage C  x-, y- and z-face fluxes (HLLC, HLL or the hybrid switch, and
//            the aux internal-energy fluxes, hy_getFaceFlux.F90) to the
//            tile's flux arrays and the
//            face-averaged pressure of each interior cell to pavg.
// The conservative update then runs as k_update from those arrays; or, where
// the call keeps no fluxes (batch steps), stage C leaves the fluxes in LDS and
//   stage D  beside the next plane's stage B, updates the plane's cells.
// x/y states exist for interior planes only; z states for planes lo-1..hi+1.

#pragma once
#include "fx_common.hpp"

namespace fx {

// array sizes and stage-A item counts of a column tile of TX x TY columns
template <int TX, int TY> struct TileIdx {
  static constexpr int NRX = TX * (TY + 2), NRY = (TX + 2) * TY, NC = (TX + 2) * (TY + 2);
  static constexpr int NLX = (TX + 4) * TY, NLY = TX * (TY + 4);
  static constexpr int NFX = (TX + 1) * TY, NFY = TX * (TY + 1);
  // stage-A items along x: the cells of R_x and of the x slopes, rows
  // b = -1, [0,TY), TY; along y: the cells of R_y and of the y slopes,
  // rows b = -2, -1, [0,TY), TY, TY+1
  static constexpr int NUX = 2 * TX + (TX + 4) * TY, NUY = 4 * TX + (TX + 2) * TY;
};

// The extents of a column tile and the row arithmetic of its items.  Fixed:
// the template's.  Free: any extents that fit the TX x TY layout's arrays and
// thread roles (free_tile_fits), for blocks that no fixed tile divides; the
// component strides stay the layout's, only the rows' are the tile's own.
template <int TX, int TY> struct FixedShape {
  static constexpr bool kFree = false;
  static __device__ __forceinline__ int tx() { return TX; }
  static __device__ __forceinline__ int ty() { return TY; }
  // rows of tx, tx + 2 and tx + 4 items: a the place in the row, b the row
  static __device__ __forceinline__ void row(int w, int& a, int& b) { a = w % TX; b = w / TX; }
  static __device__ __forceinline__ void row2(int w, int& a, int& b) {
    a = w % (TX + 2);
    b = w / (TX + 2);
  }
  static __device__ __forceinline__ void row4(int w, int& a, int& b) {
    a = w % (TX + 4);
    b = w / (TX + 4);
  }
};
struct FreeShape {
  static constexpr bool kFree = true;
  int x, y;
  unsigned m0, m2, m4;  // reciprocals of x, x + 2 and x + 4
  __device__ __forceinline__ FreeShape(int x_, int y_)
      : x(x_), y(y_), m0(65536u / (unsigned)x_ + 1u), m2(65536u / (unsigned)(x_ + 2) + 1u),
        m4(65536u / (unsigned)(x_ + 4) + 1u) {}
  __device__ __forceinline__ int tx() const { return x; }
  __device__ __forceinline__ int ty() const { return y; }
  // w / d = (w m) >> 16: exact while w d < 65536 (w < 256, d <= 140 here)
  static __device__ __forceinline__ void part(int w, int d, unsigned m, int& a, int& b) {
    b = (int)(__umul24((unsigned)w, m) >> 16);
    a = w - b * d;
  }
  __device__ __forceinline__ void row(int w, int& a, int& b) const { part(w, x, m0, a, b); }
  __device__ __forceinline__ void row2(int w, int& a, int& b) const { part(w, x + 2, m2, a, b); }
  __device__ __forceinline__ void row4(int w, int& a, int& b) const { part(w, x + 4, m4, a, b); }
};
// LDS index helpers, tile-local coordinates a = i - ox, b = j - oy, and item
// counts of a tile of tx x ty columns:
//   R_x (rx)  a in [0, tx), b in [-1, ty]      sigma_x, y state cells
//   R_y (ry)  a in [-1, tx], b in [0, ty)      sigma_y, x state cells
//   C (cc)    a in [-1, tx], b in [-1, ty]     sigma_z
//   lx        a in [-2, tx + 1], b in [0, ty)  slopes along x
//   ly        a in [0, tx), b in [-2, ty + 1]  slopes along y
//   ux        a in [0, tx], b in [0, ty)       x faces
//   uy        a in [0, tx), b in [0, ty]       y faces
template <typename S> struct ShapeIdx {
  S s;
  __device__ __forceinline__ int rx(int a, int b) const { return (b + 1) * s.tx() + a; }
  __device__ __forceinline__ int ry(int a, int b) const { return b * (s.tx() + 2) + (a + 1); }
  __device__ __forceinline__ int cc(int a, int b) const { return (b + 1) * (s.tx() + 2) + (a + 1); }
  __device__ __forceinline__ int lx(int a, int b) const { return b * (s.tx() + 4) + (a + 2); }
  __device__ __forceinline__ int ly(int a, int b) const { return (b + 2) * s.tx() + a; }
  __device__ __forceinline__ int ux(int a, int b) const { return b * (s.tx() + 1) + a; }
  __device__ __forceinline__ int uy(int a, int b) const { return b * s.tx() + a; }
  __device__ __forceinline__ int nrx() const { return s.tx() * (s.ty() + 2); }
  __device__ __forceinline__ int nry() const { return (s.tx() + 2) * s.ty(); }
  __device__ __forceinline__ int nc() const { return (s.tx() + 2) * (s.ty() + 2); }
  __device__ __forceinline__ int ncol() const { return s.tx() * s.ty(); }
  __device__ __forceinline__ int nux() const { return 2 * s.tx() + (s.tx() + 4) * s.ty(); }
  __device__ __forceinline__ int nuy() const { return 4 * s.tx() + (s.tx() + 2) * s.ty(); }
};
// Whether a free tile of tx x ty columns fits the TX x TY layout: its LDS
// arrays, its wave-aligned stage-A segments and its one state cell per thread
template <int TX, int TY> constexpr bool free_tile_fits(int tx, int ty) {
  using I = TileIdx<TX, TY>;
  return tx >= 1 && ty >= 1 && tx * (ty + 2) <= I::NRX && (tx + 2) * ty <= I::NRY &&
         (tx + 2) * (ty + 2) <= I::NC && (tx + 4) * ty <= I::NLX && tx * (ty + 4) <= I::NLY &&
         (tx + 1) * ty <= I::NFX && tx * (ty + 1) <= I::NFY && tx * ty <= TX * TY &&
         2 * tx + (tx + 4) * ty <= (I::NUX + 63) / 64 * 64 &&
         4 * tx + (tx + 2) * ty <= (I::NUY + 63) / 64 * 64;
}

// LDS of one column tile (march_tile), as offsets into one array of R.
// FUSE: with the plane's face fluxes and face-averaged pressures.
constexpr int kUpdFluxes = 7;  // face fluxes the update takes: all but the pressure slot
// Where the update runs: in a kernel of its own, from flux arrays; in the
// march, into scratch that k_update_finish spreads over the blocks; in the
// march, into the blocks.
enum : int { kFuseNone = 0, kFuseScratch = 1, kFuseDirect = 2 };
template <int NDIM, int TX, int TY, int FUSE> struct MarchLds {
  using I = TileIdx<TX, TY>;
  static constexpr int NR = NDIM == 3 ? 3 : 1, NCOL = TX * TY, Z = NDIM == 3 ? 1 : 0;
  static constexpr int SX = 0;                                // sigma_x ring
  static constexpr int SY = SX + NR * 6 * I::NRX;             // sigma_y ring
  static constexpr int SZ = SY + NR * 6 * I::NRY;             // sigma_z of plane k
  static constexpr int NRL = NDIM == 3 ? 2 : 1;               // slope ring depth
  static constexpr int LX = SZ + (Z ? 6 * I::NC : 1);         // slopes along x, ring
  static constexpr int LY = LX + NRL * 6 * I::NLX;            // slopes along y, ring
  static constexpr int LZ = LY + NRL * 6 * I::NLY;            // slopes along z, ring
  static constexpr int FX = LZ + (Z ? 3 * 6 * NCOL : 1);      // flattening tilde along x, ring
  static constexpr int FY = FX + NRL * I::NLX;                // flattening tilde along y, ring
  static constexpr int FZ = FY + NRL * I::NLY;                // flattening tilde along z, ring
  static constexpr int WX = FZ + (Z ? 3 * NCOL : 1);          // x state cells' Wp
  static constexpr int WY = WX + 6 * I::NRY;                  // y state cells' Wp
  static constexpr int WZ = WY + 6 * I::NRX;                  // z state cells' Wp of the last plane done
  // (kept in registers where the fused FP64 8x8 tile would otherwise miss
  // half a CU's LDS)
  static constexpr bool WZ_LDS = Z && !(FUSE && TX == 8);
  static constexpr int PY = WZ + (WZ_LDS ? 6 * NCOL : 1);     // Wn + Wp pressures of the y state cells
  static constexpr int PZ = PY + I::NRX;                      // and of the z state cells
  static constexpr int CST = PZ + (Z ? NCOL : 1);             // the step's ratios, widths
  // x-face fluxes; in 2-D over sigmas and slopes that stage B has done with
  static constexpr int UX = Z ? CST + 12 : 0;
  static constexpr int UY = UX + (FUSE ? kUpdFluxes * I::NFX : 0);  // y-face fluxes
  static constexpr int UZ = UY + (FUSE ? kUpdFluxes * I::NFY : 0);  // z-face fluxes
  static constexpr int PA = UZ + (FUSE && Z ? kUpdFluxes * NCOL : 0);  // face-averaged pressures
  static constexpr int total = Z ? PA + (FUSE ? NCOL : 0) : CST + 12;
  static_assert(Z || PA + NCOL <= FX, "the 2-D fluxes fit over the sigmas and slopes");
};

// components stored for sigma and slopes: dens, vx, vy, vz, pres, eint
__device__ __forceinline__ int comp_slot(int q) { return q < 5 ? q : P_EINT; }

struct MarchLaunch {
  const fx_tile* tiles;
  int nTiles;
  int tilesX, tilesY;  // column tiles per block
  DevStatus* status;
  double dt;
  void* fstates;       // RS_STATES: per-face states for the separate Riemann stage, in R
  const double* dtp;   // device-resident dt (graph-captured steps), or null
  int fuse;            // where the update runs (kFuse*)
  double* upd;         // fused update: updated states, [tile][component][interior cell]
  int tx, ty;          // free tiles: columns of a tile (the last along an axis may have fewer)
  int tilesZ = 1;      // segments of a column tile along z, of nzSeg planes (the last may have
  int nzSeg = 1 << 20; // fewer): k_march and k_march_free, not kFuseDirect
  // RS_STATES with the learned seed (one tile shape): faces at or above the
  // gate join the list; null: none do
  SeedGate gate;
  unsigned* strongList;
  unsigned* strongCount;
  unsigned strongCap;
};
// components of a cell's fused-update scratch: density, velocities, eint (the
// sixth only in the FP32 march, on the way)
constexpr int kUpdComps = 6;
// rows below a column tile that its stages read (the guard layers of a block)
constexpr int kSeamRows = 4;

// Riemann-stage variant of the march: stage C stores each face's left and
// right states (dens, vx, vy, vz, pres, eint) instead of solving there.
constexpr int RS_STATES = 99;
constexpr bool is_states(int rs) { return rs == RS_STATES; }
constexpr int kFaceComps = 12;

// face-state scratch of one tile: [dir][comp 0..11][face], in the march's
// real type R (FP32 in the mixed mode); offsets below count elements
__device__ __forceinline__ long fstate_tile_stride(const DevParams& P) {
  return (long)kFaceComps * (P.nface[0] + P.nface[1] + P.nface[2]);
}
__device__ __forceinline__ long fstate_dir_offset(const DevParams& P, int d) {
  long o = 0;
  for (int e = 0; e < d; ++e) o += (long)kFaceComps * P.nface[e];
  return o;
}

template <int D, typename R>
__device__ __forceinline__ void write_face_states(const DevParams& P, R* base, long r,
                                                  const R VL[8], const R VR[8]) {
  const long nf = P.nface[D];
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    base[q * nf + r] = VL[comp_slot(q)];
    base[(6 + q) * nf + r] = VR[comp_slot(q)];
  }
}

// The learned seed's gate (seed_gate_pass, in FP64 from the stored values) on a
// face whose states are at hand: a strong one joins the list, one atomic per
// wavefront, ranks by ballot over the lanes that are here.
template <int D, typename R>
__device__ __forceinline__ void list_strong_face(const DevParams& P, const MarchLaunch& L, int t,
                                                 unsigned r, const R VL[8], const R VR[8]) {
  const double rl = VL[P_DENS], ul = VL[P_VELX + D], pl = VL[P_PRES];
  const double rr = VR[P_DENS], ur = VR[P_VELX + D], pr = VR[P_PRES];
  const bool strong = rl > 0. && rr > 0. && pl > 0. && pr > 0. &&
                      seed_gate_pass(L.gate, P.gamma, rl, ul, pl, rr, ur, pr);
  const unsigned long long mask = __ballot(strong);
  if (!mask) return;
  const int lane = (int)(threadIdx.x & 63), leader = __builtin_ctzll(mask);
  unsigned base = 0;
  if (lane == leader) base = atomicAdd(L.strongCount, (unsigned)__popcll(mask));
  base = __shfl(base, leader);
  const unsigned slot = base + (unsigned)__popcll(mask & ((1ULL << lane) - 1ULL));
  if (!strong || slot >= L.strongCap) return;
  const long before = D == 0 ? 0 : (D == 1 ? P.nface[0] : P.nface[0] + P.nface[1]);
  const long perTile = P.nface[0] + P.nface[1] + P.nface[2];
  L.strongList[slot] = (unsigned)(t * perTile + before + r);
}

template <typename R>
__device__ __forceinline__ void lds_put6(R* base, int n, int idx, const R v[8]) {
#pragma unroll
  for (int q = 0; q < 6; ++q) base[q * n + idx] = v[comp_slot(q)];
}
template <typename R>
__device__ __forceinline__ void lds_get6(const R* base, int n, int idx, R v[8]) {
#pragma unroll
  for (int q = 0; q < 6; ++q) v[comp_slot(q)] = base[q * n + idx];
  v[P_GAMC] = R(0.);
  v[P_GAME] = R(0.);
}

// First-order reset of one state cell's face states.  A state cell on a
// column-tile seam is computed by both tiles; only its owner (own = true)
// counts the reset, so the count is one per (state cell, direction), as the
// reference's (hy_dataReconstOneStep.F90:1124-1129).
template <typename R>
__device__ __forceinline__ void fallback_first_order(const R* Vc, R Wp[8], R Wn[8],
                                                     DevStatus* st, bool own) {
  if (own) atomicAdd(&st->fallbacks, 1ULL);
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    Wn[v] = Vc[v];
    Wp[v] = Vc[v];
  }
}

template <typename R>
__device__ __forceinline__ void sub_sigma(R Wp[8], R Wn[8], const R* sg, R hdt) {
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    Wn[v] = Wn[v] - hdt * sg[v];
    Wp[v] = Wp[v] - hdt * sg[v];
  }
}

template <typename R>
__device__ __forceinline__ void add_ctu(R Wp[8], R Wn[8], const R* tA, const R* tB, R fac) {
#pragma unroll
  for (int v = 0; v < 8; ++v) {
    Wp[v] = Wp[v] + (tA[v] + tB[v]) * fac;
    Wn[v] = Wn[v] + (tA[v] + tB[v]) * fac;
  }
}

template <typename R>
__device__ __forceinline__ bool nonpositive(const R* Wp, const R* Wn) {
  return Wp[P_DENS] <= R(0.) || Wn[P_DENS] <= R(0.) || Wp[P_PRES] <= R(0.) || Wn[P_PRES] <= R(0.);
}
template <typename R>
__device__ __forceinline__ bool negative(const R* Wp, const R* Wn) {
  return Wn[P_DENS] < R(0.) || Wp[P_DENS] < R(0.) || Wn[P_PRES] < R(0.) || Wp[P_PRES] < R(0.);
}

template <typename R>
__device__ __forceinline__ R flat_tilde_vals(R pm2, R pm1, R pp1, R pp2, R vm1, R vp1) {
  const R dp1 = (pp1 - pm1);
  const R dp2 = (pp2 - pm2);
  const R dv1 = vp1 - vm1;
  const R qp = quot(dp1, dp2);
  const R Sp = (fabs(dp2) > R(1.e-15)) ? qp - R(0.75) : R(0.);
  R ft = fmax(R(0.0), fmin(R(1.0), R(10.0) * Sp));
  if ((quot(fabs(dp1), fmin(pm1, pp1)) < R(1.) / R(3.)) || dv1 > R(0.)) ft = R(0.);
  return ft;
}

// Item counts rounded up to whole wavefronts: each stage lays its item kinds
// out in wave-aligned segments, so that no wavefront runs two kinds of item
// (two code paths) one after the other.
constexpr int wave_up(int n) { return (n + 63) / 64 * 64; }

// ---- a tile's cell data as the march reads it ----
// 32-bit byte offsets of cells (a tile holds far fewer than 2^29 cells),
// which serve every variable.  Outputs are stored through a uniform base
// address plus one vector offset (st_at).
typedef __attribute__((address_space(1))) char gchar;
template <typename T>
__device__ __forceinline__ void st_at(__attribute__((address_space(1))) T* base, unsigned boff,
                                      T v) {
  *reinterpret_cast<__attribute__((address_space(1))) T*>(reinterpret_cast<gchar*>(base) + boff) = v;
}

template <typename T>
__device__ __forceinline__ T ld_at(const __attribute__((address_space(1))) T* base, unsigned boff) {
  return *reinterpret_cast<const __attribute__((address_space(1))) T*>(
      reinterpret_cast<const gchar*>(base) + boff);
}

// The tile's primitives are read as one buffer (a scalar resource) with the
// variable's byte offset in a scalar operand and the cell's in a vector
// one, so no 64-bit address is formed per lane.  With 64-bit addresses several
// per stencil point stay live across the item loops: the FP32 march takes 161
// registers instead of 114, which leaves one workgroup on a CU for two (4096 x
// 16^3 mixed 5.83 against 4.05 ms a step), the FP64 one 5.97 against 5.80 ms.
struct TileView {
  __amdgpu_buffer_rsrc_t rs;  // the tile's guard-inclusive array
  unsigned ob[8];             // byte offsets of the primitive slots P_DENS .. P_EINT
  unsigned obShok;            // SHOK_VAR's (hybrid solver)
  unsigned obEner;            // ENER_VAR's (fused update)
};

// The workgroup's tile is uniform; saying so (readfirstlane) keeps the
// compiler from making each buffer load uniform on its own where the tile
// and its class come from a work list.
__device__ __forceinline__ unsigned fx_uniform(unsigned x) { return __builtin_amdgcn_readfirstlane(x); }

__device__ __forceinline__ TileView tile_view(const DevParams& P, const gdouble* U) {
  TileView tv;
  const unsigned long long u = reinterpret_cast<unsigned long long>(U);
  void* const base = reinterpret_cast<void*>(
      (static_cast<unsigned long long>(fx_uniform((unsigned)(u >> 32))) << 32) |
      fx_uniform((unsigned)u));
  // raw buffer: no stride, a byte range past any tile's array (offsets stay
  // below 2^31), and the resource word of untyped dword accesses
  tv.rs = __builtin_amdgcn_make_buffer_rsrc(base, (short)0, 0x7fffffff, 0x00020000);
  tv.ob[P_DENS] = fx_uniform((unsigned)P.voff[FX_DENS] * 8u);
  tv.ob[P_VELX] = fx_uniform((unsigned)P.voff[FX_VELX] * 8u);
  tv.ob[P_VELY] = fx_uniform((unsigned)P.voff[FX_VELY] * 8u);
  tv.ob[P_VELZ] = fx_uniform((unsigned)P.voff[FX_VELZ] * 8u);
  tv.ob[P_PRES] = fx_uniform((unsigned)P.voff[FX_PRES] * 8u);
  tv.ob[P_GAMC] = fx_uniform((unsigned)P.voff[FX_GAMC] * 8u);
  tv.ob[P_GAME] = fx_uniform((unsigned)P.voff[FX_GAME] * 8u);
  tv.ob[P_EINT] = fx_uniform((unsigned)P.voff[FX_EINT] * 8u);
  tv.obEner = fx_uniform((unsigned)P.voff[FX_ENER] * 8u);
  tv.obShok = fx_uniform(P.shokOff >= 0 ? (unsigned)P.shokOff * 8u : 0u);
  return tv;
}
// variable slot q (byte offset ob) of the cell at byte offset cb
__device__ __forceinline__ double tv_ld(const TileView& tv, unsigned ob, unsigned cb) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(tv.rs, (int)cb, (int)ob, 0));
}

__device__ __forceinline__ void tv_st(const TileView& tv, unsigned ob, unsigned cb, double v) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2u, v), tv.rs, (int)cb, (int)ob, 0);
}

// A stage's item number.  With OPAQUE it passes through an empty asm
// statement, which the compiler cannot see through: the index arithmetic of
// each stage's items (item kind, column, cell offsets) is then redone per
// plane instead of being hoisted out of the plane loop and kept live.  Hoisted,
// the FP64 16x8 march spills 106 registers instead of 10 (4096 x 16^3 7.70
// against 5.80 ms a step) and the FP32 one takes 167 instead of 114 (5.57
// against 4.05); the FP64 march over several classes spills 55 instead of none
// (29.4M zones 12.5 against 11.5 ms).
template <bool OPAQUE>
__device__ __forceinline__ int item_index(int w) {
  if constexpr (OPAQUE) asm volatile("" : "+v"(w));
  return w;
}

// byte offset of cell (i, j, k) in its tile
__device__ __forceinline__ unsigned cell_b(const DevParams& P, int i, int j, int k) {
  return (unsigned)((k * P.ny + j) * P.nx + i) * 8u;
}

// every variable of the updated cell at cb
__device__ __forceinline__ void tv_expand(const DevParams& P, const TileView& tv, unsigned cb,
                                          const UpdState& u) {
  double out[10];
  upd_expand(P, u, out);
#pragma unroll
  for (int v = 0; v < 10; ++v) tv_st(tv, fx_uniform((unsigned)P.voff[upd_var(v)] * 8u), cb, out[v]);
}

template <typename R>
__device__ __forceinline__ void tv_prim(const TileView& tv, unsigned cb, R V[8]) {
#pragma unroll
  for (int q = 0; q < 8; ++q) V[q] = R(tv_ld(tv, tv.ob[q], cb));
}

// sigma of the cell at cb along SD (the transverse-only PPM call; sb: the
// axis stride in bytes)
template <int SD, typename R>
__device__ __forceinline__ bool tv_sigma(const DevParams& P, const TileView& tv, unsigned cb,
                                         unsigned sb, R sig[8]) {
  R Vm[8], Vc[8], Vp[8];
  tv_prim(tv, cb - sb, Vm);
  tv_prim(tv, cb, Vc);
  tv_prim(tv, cb + sb, Vp);
  EigT<R> e;
  const bool ok = eig_make<SD>(Vc, e);
  trans_sigma<SD>(P, Vm, Vc, Vp, e, sig);
  return ok;
}

// Whether the face between the cells at cbl and cbr takes HLL (HLL, or the
// hybrid switch with a flagged cell on either side, hy_getFaceFlux.F90:353-367)
template <int RS>
__device__ __forceinline__ bool tv_use_hll(const DevParams& P, const TileView& tv, unsigned cbl,
                                           unsigned cbr) {
  if constexpr (RS == FX_HYBR) {
    if (P.riemann == FX_HLL) return true;
    if (P.riemann != FX_HYBR) return false;
    return tv_ld(tv, tv.obShok, cbl) + tv_ld(tv, tv.obShok, cbr) > 0.;
  } else {
    return false;
  }
}

// face flux densities F[0..7] to the tile's flux array of direction D at the
// face's byte offset rb (q-major, nface[D] faces per flux)
template <int D>
__device__ __forceinline__ void write_flux_b(const DevParams& P, gdouble* Fo, unsigned rb,
                                             const double F[8]) {
  const long nf = P.nface[D];
#pragma unroll
  for (int q = 0; q < FX_NFLUX; ++q) st_at(Fo + q * nf, rb, F[q]);
}

// The march's barrier: a workgroup's threads exchange data through LDS alone,
// so the LDS accesses are waited for and the global ones stay in flight.  The
// plain barrier also waits for every store to reach the cache, once per stage.
// What makes that safe where the update runs inside the march (stage D):
// - kFuseDirect stores a block's cells while other wavefronts load from it.
//   Beside stage B of plane k it stores plane k - 2 (in 2-D the one plane, after
//   the last stage), and no load still to come or in flight is below plane
//   k - 1: stage B and the z slopes of k + 1 reach down to k - 1, stage C(k) to
//   k - 1.  Contact steepening reads two planes down and takes kFuseScratch.
// - The neighbouring column tile's rows within a stencil's reach (kSeamRows) are
//   kept back until that tile is done (march_block).
// - Scratch that is read back during the march (FP32's carried cells) is read by
//   the thread that stored it; the seam rows, read by others, lie behind the full
//   barrier that ends a column tile.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One column tile (TX x TY columns at ox, oy, planes klo to khi) of tile t.  Every
// thread of the workgroup calls it with the same arguments; it ends on a
// barrier, so a workgroup may call it again for another column tile.  fsb:
// tile t's face-state scratch (RS_STATES).
//
// Two barriers per plane.  Between them run
//   stage B(k)          one state cell per thread (x, y and z state cells in
//                       wave-aligned roles): PPM, the 2-D and the 3-D CTU
//                       corrections.  The high-side state Wp goes to LDS for
//                       the next face up; the low-side state Wn stays in the
//                       thread's registers.
//   stage C(k), A(k+1)  the thread's own face (x, y or z) between its
//                       neighbour's Wp and its own Wn, then the stage-A items
//                       of the next plane.  C(k) reads only face states and
//                       A(k+1) writes only sigmas, slopes and tildes that
//                       B(k) has done with, so no barrier is needed between.
// Everything a state cell needs (its stencil, its eigen system, its two face
// states) is formed once in one thread; the waves that have no face start
// the next plane's stage A meanwhile.  The loads of a stage start right
// after its barrier, so fewer barriers are fewer times that all waves wait
// for the cache together.  Against the form with four barriers (face states,
// CTU and fluxes as stages of their own over LDS arrays of both states,
// tildes formed by the state cells) the step of 4096 x 16^3 went from 10.17
// to 8.89 ms (FP64 HLLC), of 2048 x 16^3 from 3.41 to 3.07 ms (mixed) and of
// 1024 x 16^3 from 3.52 to 3.15 ms (FP64 exact).
template <int NDIM, int TX, int TY, int NT, int RS, typename R, bool OPAQUE, int FUSE, typename SH>
__device__ __forceinline__ void march_tile(const DevParams& P, const MarchLaunch& L,
                                           const fx_tile& T, int t, int ox, int oy, R* fsb,
                                           ExactStats& es, R* smem, const SH shape, int klo,
                                           int khi) {
  using I = TileIdx<TX, TY>;
  using M = MarchLds<NDIM, TX, TY, FUSE>;
  constexpr int NR = NDIM == 3 ? 3 : 1;        // ring depth
  constexpr int NCOL = TX * TY;
  constexpr int Z = NDIM == 3 ? 1 : 0;
  R* const SX = smem + M::SX;
  R* const SY = smem + M::SY;
  R* const SZ = smem + M::SZ;
  R* const LX = smem + M::LX;
  R* const LY = smem + M::LY;
  R* const LZ = smem + M::LZ;
  R* const FX = smem + M::FX;
  R* const FY = smem + M::FY;
  R* const FZ = smem + M::FZ;
  R* const WX = smem + M::WX;
  R* const WY = smem + M::WY;
  R* const WZ = smem + M::WZ;
  R* const PY = smem + M::PY;
  R* const PZ = smem + M::PZ;
  R* const UX = smem + M::UX;
  R* const UY = smem + M::UY;
  R* const UZ = smem + M::UZ;
  R* const PA = smem + M::PA;

  const int tid = threadIdx.x;
  const ShapeIdx<SH> X{shape};
  const int tx = shape.tx(), ty = shape.ty();
  // A tile owns its high x (y) face row only at the block's high side;
  // otherwise the neighbouring tile computes that row (and the states
  // behind it) as its low row.  The fused update needs that row's fluxes in
  // either case, so there both tiles compute it.
  const bool ex = (ox + tx > P.hi[0]);
  const bool ey = (oy + ty > P.hi[1]);
  const TileView tv = tile_view(P, as_global(T.U));
  double dt = step_dt(L.dt, L.dtp);
  // (opaque: a workgroup that takes a block's tiles in turn would otherwise
  // keep the ratios below live through all of them)
  if constexpr (FUSE == kFuseDirect) asm volatile("" : "+v"(dt));
  const double dx = T.del[0], dy = T.del[1], dz = T.del[2];
  const unsigned sxb = 8u, syb = (unsigned)P.nx * 8u, szb = (unsigned)(P.nx * P.ny) * 8u;
  DevStatus* st = L.status;
  bool bad = false;  // eigen failure seen by this thread
  // The step's ratios of dt and the cell widths, and the widths, uniform over
  // the tile: read from LDS, written once per column tile by one thread (stage
  // B first reads them after a barrier, and the previous column tile ended on
  // one).  Held in registers they take 24 of the 168 an FP64 thread has (no
  // scalar FP64 arithmetic makes them scalar).
  const R rat[12] = {R(dt / dx), R(dt / dy), R(dt / dz),
                     R(0.5 * dt / dx), R(0.5 * dt / dy), R(0.5 * dt / dz),
                     R(dt * dt / (6. * dy * dz)), R(dt * dt / (6. * dz * dx)),
                     R(dt * dt / (6. * dx * dy)), R(dx), R(dy), R(dz)};
  R* const CST = smem + M::CST;
  if (tid == 0)
    for (int i = 0; i < 12; ++i) CST[i] = rat[i];
  auto ratio = [&](int i) -> R { return CST[i]; };

  auto ring = [](int k) { return NR == 3 ? (k % 3) : 0; };
  auto ringL = [](int k) { return M::NRL == 2 ? (k & 1) : 0; };

  // stage-A items: sigma_x (w < NRX) and sigma_y (w < NRY) of plane kk
  auto sig_x_item = [&](int w, int kk) {
    R sg[8];
    int a, b;
    shape.row(w, a, b);
    --b;
    bad |= !tv_sigma<0>(P, tv, cell_b(P, ox + a, oy + b, kk), sxb, sg);
    lds_put6(SX + ring(kk) * 6 * I::NRX, I::NRX, w, sg);
  };
  auto sig_y_item = [&](int w, int kk) {
    R sg[8];
    int a, b;
    shape.row2(w, a, b);
    --a;
    bad |= !tv_sigma<1>(P, tv, cell_b(P, ox + a, oy + b, kk), syb, sg);
    lds_put6(SY + ring(kk) * 6 * I::NRY, I::NRY, w, sg);
  };
  // stage-A items along x (w < NUX) and y (w < NUY) at plane p: one cell's
  // three-cell stencil and eigen system serve its sigma (sig: p is a plane
  // the sigma ring takes, and the cell lies in R_x / R_y), its limited slope
  // and its flattening tilde (sl: p is interior, and the cell lies in the
  // slope rows).  Each tilde is formed here once: formed by the state cells,
  // a state cell's coefficient took three (its own, and one of each
  // neighbour's in diverged branches) and five more loads.
  auto x_item = [&](int w, int p, bool sig, bool sl) {
    int a, b;
    if (w < tx) {
      a = w;
      b = -1;
    } else if (w < tx + (tx + 4) * ty) {
      shape.row4(w - tx, a, b);
      a -= 2;
    } else {
      a = w - tx - (tx + 4) * ty;
      b = ty;
    }
    const bool doS = sig && a >= 0 && a < tx;
    const bool doL = sl && b >= 0 && b < ty;
    if (!doS && !doL) return;
    const unsigned cb = cell_b(P, ox + a, oy + b, p);
    R Vm[8], Vc[8], Vp[8];
    tv_prim(tv, cb - sxb, Vm);
    tv_prim(tv, cb, Vc);
    tv_prim(tv, cb + sxb, Vp);
    EigT<R> e;
    bad |= !eig_make<0>(Vc, e);
    if (doS) {
      R sg[8];
      trans_sigma<0>(P, Vm, Vc, Vp, e, sg);
      lds_put6(SX + ring(p) * 6 * I::NRX, I::NRX, X.rx(a, b), sg);
    }
    if (doL) {
      R db[8];
      tvd_slope<0>(P, Vm, Vc, Vp, e, db);
      lds_put6(LX + ringL(p) * 6 * I::NLX, I::NLX, X.lx(a, b), db);
      if (P.flat)
        FX[ringL(p) * I::NLX + X.lx(a, b)] =
            flat_tilde_vals(R(tv_ld(tv, tv.ob[P_PRES], cb - 2 * sxb)), Vm[P_PRES], Vp[P_PRES],
                            R(tv_ld(tv, tv.ob[P_PRES], cb + 2 * sxb)), Vm[P_VELX], Vp[P_VELX]);
    }
  };
  auto y_item = [&](int w, int p, bool sig, bool sl) {
    int a, b;
    if (w < 2 * tx) {
      shape.row(w, a, b);
      b -= 2;
    } else if (w < 2 * tx + (tx + 2) * ty) {
      shape.row2(w - 2 * tx, a, b);
      --a;
    } else {
      shape.row(w - 2 * tx - (tx + 2) * ty, a, b);
      b += ty;
    }
    const bool doS = sig && b >= 0 && b < ty;
    const bool doL = sl && a >= 0 && a < tx;
    if (!doS && !doL) return;
    const unsigned cb = cell_b(P, ox + a, oy + b, p);
    R Vm[8], Vc[8], Vp[8];
    tv_prim(tv, cb - syb, Vm);
    tv_prim(tv, cb, Vc);
    tv_prim(tv, cb + syb, Vp);
    EigT<R> e;
    bad |= !eig_make<1>(Vc, e);
    if (doS) {
      R sg[8];
      trans_sigma<1>(P, Vm, Vc, Vp, e, sg);
      lds_put6(SY + ring(p) * 6 * I::NRY, I::NRY, X.ry(a, b), sg);
    }
    if (doL) {
      R db[8];
      tvd_slope<1>(P, Vm, Vc, Vp, e, db);
      lds_put6(LY + ringL(p) * 6 * I::NLY, I::NLY, X.ly(a, b), db);
      if (P.flat)
        FY[ringL(p) * I::NLY + X.ly(a, b)] =
            flat_tilde_vals(R(tv_ld(tv, tv.ob[P_PRES], cb - 2 * syb)), Vm[P_PRES], Vp[P_PRES],
                            R(tv_ld(tv, tv.ob[P_PRES], cb + 2 * syb)), Vm[P_VELY], Vp[P_VELY]);
    }
  };
  // stage-A item: z-slope and z flattening tilde of column w at plane m
  auto zslope_item = [&](int w, int m) {
    int a, b;
    shape.row(w, a, b);
    const unsigned cb = cell_b(P, ox + a, oy + b, m);
    R db[8], Vm[8], Vc[8], Vp[8];
    tv_prim(tv, cb - szb, Vm);
    tv_prim(tv, cb, Vc);
    tv_prim(tv, cb + szb, Vp);
    EigT<R> e;
    bad |= !eig_make<2>(Vc, e);
    tvd_slope<2>(P, Vm, Vc, Vp, e, db);
    lds_put6(LZ + ring(m) * 6 * NCOL, NCOL, w, db);
    if (P.flat)
      FZ[ring(m) * NCOL + w] =
          flat_tilde_vals(R(tv_ld(tv, tv.ob[P_PRES], cb - 2 * szb)), Vm[P_PRES], Vp[P_PRES],
                          R(tv_ld(tv, tv.ob[P_PRES], cb + 2 * szb)), Vm[P_VELZ], Vp[P_VELZ]);
  };
  // interior cell number within the tile's block
  auto cell_r = [&](int i, int j, int k) -> unsigned {
    return (unsigned)(((k - P.lo[2]) * P.nyb + (j - P.lo[1])) * P.nxb + (i - P.lo[0]));
  };
  // FlatCoeff of the cell whose pressures across are pm, pp, from its own
  // tilde and its neighbours' (hy_getRiemannState.F90:408-453)
  auto flat_of = [&](R pm, R pp, R fm, R f0, R fp) -> R {
    const R dp1 = pp - pm;
    return dp1 < R(0.0) ? fmax(f0, fp) : (dp1 == R(0.) ? f0 : fmax(f0, fm));
  };

  const int kBeg = Z ? klo - 1 : 0;
  const int kEnd = Z ? khi + 1 : 0;
  // ------------------------------ stage A ------------------------------
  // For plane k: sigma_x/y of plane k+1 (the ring's next plane), x/y slopes
  // and tildes of plane k+1 (the slope ring's next plane), sigma_z of plane
  // k, z slopes of plane k+1.  (2-D: plane 0's sigmas and slopes.)  Segments
  // in wave-aligned order (x items, y items, sigma_z, z slopes): one item
  // kind per wavefront.  Each work item is a lambda whose early exits are
  // returns, not loop continues: the compiler then allocates registers per
  // item kind.
  auto stageA = [&](int k) {
    const int pA = Z ? k + 1 : 0;
    const bool interiorA = !Z || (k >= klo && k <= khi);
    const bool wSig = !Z || k + 1 <= kEnd;
    const bool wL = !Z || (k + 1 >= klo && k + 1 <= khi);
    const bool uXY = wSig || wL;
    const int nSz = (Z && interiorA) ? X.nc() : 0;
    const int nZs = Z ? X.ncol() : 0;
    constexpr int PUX = wave_up(I::NUX), PUY = wave_up(I::NUY), PZ4 = wave_up(I::NC);
    const int s1 = uXY ? PUX + PUY : 0, s2 = s1 + (nSz ? PZ4 : 0), sEnd = s2 + nZs;
    auto itemA = [&](int v) {
      if (v < s1) {
        if (v < PUX) {
          if (v < X.nux()) x_item(v, pA, wSig, wL);
        } else if (v - PUX < X.nuy()) {
          y_item(v - PUX, pA, wSig, wL);
        }
        return;
      }
      if (v < s2) {
        const int r = v - s1;
        if (r >= X.nc()) return;
        R v8[8];
        int a, b;
        shape.row2(r, a, b);
        --a;
        --b;
        bad |= !tv_sigma<2>(P, tv, cell_b(P, ox + a, oy + b, k), szb, v8);
        lds_put6(SZ, I::NC, r, v8);
        return;
      }
      zslope_item(v - s2, k + 1);
    };
    // items past the first NT go to the wavefronts that had no face to solve
    // before (the 8x8 tile has seven wavefronts of items for six, five of them
    // with faces: 8192 x 8^3 FP64 3157 -> 2923 us, mixed 1807 -> 1650)
    constexpr int FACES = wave_up(I::NRY) + wave_up(I::NRX) + (Z ? NCOL : 0);
    constexpr int ROT = FACES < NT ? NT - FACES : 0;
    constexpr int MOST = Z ? PUX + PUY + PZ4 + NCOL : PUX + PUY;
    if constexpr (MOST <= NT || ROT == 0) {
      for (int v = tid; v < sEnd; v += NT) itemA(item_index<OPAQUE>(v));
    } else {
      for (int v = tid, next = NT + (tid + ROT) % NT; v < sEnd; v = next, next += NT)
        itemA(item_index<OPAQUE>(v));
    }
  };
  if (Z) {
    // prologue: sigma_x/y of plane kBeg, z slopes of kBeg-1 and kBeg
    constexpr int Q1 = wave_up(I::NRX), Q2 = Q1 + wave_up(I::NRY), Q3 = Q2 + wave_up(NCOL);
    for (int w = tid; w < Q3 + X.ncol(); w += NT) {
      if (w < Q1) { if (w < X.nrx()) sig_x_item(w, kBeg); }
      else if (w < Q2) { if (w - Q1 < X.nry()) sig_y_item(w - Q1, kBeg); }
      else if (w < Q3) { if (w - Q2 < X.ncol()) zslope_item(w - Q2, kBeg - 1); }
      else zslope_item(w - Q3, kBeg);
    }
  }
  stageA(kBeg);
  lds_barrier();

  // roles of stages B and C, one state cell and one face per thread: x state
  // cells (a in [-1, TX], with the face below each), y ones (b in [-1, TY]),
  // columns (z state cell and face).  The extents are fixed so that item
  // numbers split by compile-time divisors; the high row (a = TX) is skipped
  // unless the tile sits at the block's high side, where it owns that row.
  constexpr int NBX = (TX + 2) * TY, NBY = TX * (TY + 2);
  constexpr int B1 = wave_up(NBX), B2 = B1 + wave_up(NBY), B3 = B2 + (Z ? NCOL : 0);
  static_assert(B3 <= NT, "one state cell per thread");

  // Wn of the thread's state cell from stage B to C; in a column, Wp of the
  // plane below (the left state of the z face) as well, and the sum of the
  // state pressures for pavg in the x role
  R Wk[6], Wo[6], Wt[6], psum = R(0.);
#pragma unroll
  for (int q = 0; q < 6; ++q) Wk[q] = Wo[q] = Wt[q] = R(0.);

  // ------------------------------ stage D ------------------------------
  // The fused update: hy_unsplitUpdate, hy_energyFix and the EOS input of
  // one column's cells from the fluxes in LDS, as update_cell takes them.
  // Beside stage B of plane k it takes the x and y terms of the cell at plane
  // k-1 and the z term of the one at plane k-2, whose upper face's flux
  // stage C(k-1) left.  Where the block's cells are still to be read by other
  // column tiles, the new state (density, velocities, eint: the rest follows
  // from them) goes to scratch, to be spread later: every cell of
  // kFuseScratch (k_update_finish), the top kSeamRows rows of a kFuseDirect
  // tile with another above it (march_block).  The column's own planes are
  // done with: no stage reads below plane k-1 by then (contact steepening
  // does, and takes kFuseScratch).  The fluxes' way through memory (3.6 GB
  // written, read back by an update of its own) cost 1.8 ms of 8.0 on 4096 x
  // 16^3 in FP64; beside stage B, on wavefronts that have no state cell, the
  // update costs 0.1 ms, and 0.25 with the stores into the blocks.
  constexpr int D0 = (NT >= B3 + NCOL) ? B3 : 0;  // wavefronts without a role, if there are
  // carried from plane to plane: the cell after its x and y terms, its
  // face-averaged pressure, the flux through its lower z face.  The FP32
  // march carries the FP64 ones through the cell's scratch (kUpdComps
  // components, final values over them): in registers they would take it past
  // the 128 that two workgroups on a CU leave, and with one workgroup the
  // march of 2048 x 16^3 takes 2.50 ms; asking the compiler for 4 waves per
  // SIMD instead makes it load in small batches (2.76 ms).
  constexpr bool CARRY = sizeof(R) == 8;
  double cU[5] = {0., 0., 0., 0., 0.}, cI = 0.;
  R cP = R(0.), zlow[kUpdFluxes];
#pragma unroll
  for (int q = 0; q < kUpdFluxes; ++q) zlow[q] = R(0.);
  auto put_flux = [](R* U, int n, int idx, const double F[8]) {
#pragma unroll
    for (int q = 0; q < kUpdFluxes; ++q) U[q * n + idx] = R(F[q < 5 ? q : q + 1]);
  };
  auto get_flux = [](const R* U, int n, int idx, double F[8]) {
#pragma unroll
    for (int q = 0; q < kUpdFluxes; ++q) F[q < 5 ? q : q + 1] = double(U[q * n + idx]);
    F[5] = 0.;
  };
  auto stageD = [&](int k) {
    const int w = item_index<OPAQUE>(tid) - D0;
    if (w < 0 || w >= X.ncol()) return;
    int a, b;
    shape.row(w, a, b);
    double F0[8], F1[8];
    double S;  // the pressure source: zero (the whole pressure is in the flux)
    gdouble* const upd = as_global(L.upd + (long)t * (kUpdComps * P.icells));
    auto put_new = [&](int kk, double eintOld) {
      UpdPart part;
#pragma unroll
      for (int q = 0; q < 5; ++q) part.U0[q] = cU[q];
      part.IntEner = cI;
      part.S1 = part.S2 = 0.;
      const UpdState u = upd_state(P, dt, part, eintOld);
      if (FUSE == kFuseDirect && (b < ty - kSeamRows || ey)) {
        tv_expand(P, tv, cell_b(P, ox + a, oy + b, kk), u);
        return;
      }
      const unsigned r = cell_r(ox + a, oy + b, kk) * 8u;
      st_at(upd, r, u.dens);
      st_at(upd + P.icells, r, u.vx);
      st_at(upd + 2 * P.icells, r, u.vy);
      st_at(upd + 3 * P.icells, r, u.vz);
      st_at(upd + 4 * P.icells, r, u.eint);
    };
    if (Z && k - 2 >= klo) {  // z term and the rest of plane k-2
      if (!CARRY) {
        const unsigned r = cell_r(ox + a, oy + b, k - 2) * 8u;
#pragma unroll
        for (int q = 0; q < 5; ++q) cU[q] = ld_at(upd + q * P.icells, r);
        cI = ld_at(upd + 5 * P.icells, r);
      }
#pragma unroll
      for (int q = 0; q < kUpdFluxes; ++q) F0[q < 5 ? q : q + 1] = double(zlow[q]);
      F0[5] = 0.;
      get_flux(UZ, NCOL, w, F1);
      upd_dir(P, dt, dz, double(cP), F0, F1, cU, cI, S);
      put_new(k - 2, P.aux ? 0. : tv_ld(tv, tv.ob[P_EINT], cell_b(P, ox + a, oy + b, k - 2)));
    }
    const int kc = Z ? k - 1 : k;
    if (kc >= klo && kc <= khi) {
      const unsigned cb = cell_b(P, ox + a, oy + b, kc);
      if (P.aux) cP = PA[w];
      const UpdPart part = upd_init(P, tv_ld(tv, tv.ob[P_DENS], cb), tv_ld(tv, tv.ob[P_VELX], cb),
                                    tv_ld(tv, tv.ob[P_VELY], cb), tv_ld(tv, tv.ob[P_VELZ], cb),
                                    tv_ld(tv, tv.obEner, cb), tv_ld(tv, tv.ob[P_EINT], cb), 0.);
#pragma unroll
      for (int q = 0; q < 5; ++q) cU[q] = part.U0[q];
      cI = part.IntEner;
      get_flux(UX, I::NFX, X.ux(a, b), F0);
      get_flux(UX, I::NFX, X.ux(a + 1, b), F1);
      upd_dir(P, dt, dx, double(cP), F0, F1, cU, cI, S);
      get_flux(UY, I::NFY, X.uy(a, b), F0);
      get_flux(UY, I::NFY, X.uy(a, b + 1), F1);
      upd_dir(P, dt, dy, double(cP), F0, F1, cU, cI, S);
      if (Z && !CARRY) {
        const unsigned r = cell_r(ox + a, oy + b, kc) * 8u;
#pragma unroll
        for (int q = 0; q < 5; ++q) st_at(upd + q * P.icells, r, cU[q]);
        st_at(upd + 5 * P.icells, r, cI);
      }
      if (!Z) put_new(kc, tv_ld(tv, tv.ob[P_EINT], cb));
    }
    if (Z) {
#pragma unroll
      for (int q = 0; q < kUpdFluxes; ++q) zlow[q] = UZ[q * NCOL + w];
    }
  };

  for (int k = kBeg; k <= kEnd; ++k) {
    const bool interior = !Z || (k >= klo && k <= khi);
    const R* sxk = SX + ring(k) * 6 * I::NRX;
    const R* syk = SY + ring(k) * 6 * I::NRY;
    // ------------------------------ stage B ------------------------------
    {
      auto keep = [&](const R Wn[8]) {
#pragma unroll
        for (int q = 0; q < 6; ++q) Wk[q] = Wn[comp_slot(q)];
      };
      auto itemB = [&](int w) {
        R Wp[8], Wn[8], Vm[8], Vc[8], Vp[8], dbN[8], db0[8], dbP[8], sg[8];
        R sm[8], sc[8], sp[8], tA[8], tB[8];
        EigT<R> e0, e1, e2;
        if (w < B1) {
          if (!interior || w >= X.nry()) return;
          int a, b;
          shape.row2(w, a, b);
          --a;
          if (a == tx && !ex && !FUSE) return;
          // the tile owns this state cell (and counts its reset)
          const bool own = (a >= 0 || ox == P.lo[0]) && (a < tx || ex);
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
          tv_prim(tv, cb - sxb, Vm);
          tv_prim(tv, cb, Vc);
          tv_prim(tv, cb + sxb, Vp);
          const R* fx = FX + ringL(k) * I::NLX + X.lx(a, b);
          const R flat = P.flat ? flat_of(Vm[P_PRES], Vp[P_PRES], fx[-1], fx[0], fx[1]) : R(0.);
          const R* lxk = LX + ringL(k) * 6 * I::NLX;
          lds_get6(lxk, I::NLX, X.lx(a - 1, b), dbN);
          lds_get6(lxk, I::NLX, X.lx(a, b), db0);
          lds_get6(lxk, I::NLX, X.lx(a + 1, b), dbP);
          bad |= !eig_make<0>(Vc, e0);
          const R dmm = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb - 2 * sxb)) : R(0.);
          const R dpp = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb + 2 * sxb)) : R(0.);
          ppm_trace<0>(P, ratio(0), ratio(9), Vm, Vc, Vp, dmm, dpp, dbN, db0, dbP, flat, e0, Wp, Wn);
          lds_get6(syk, I::NRY, X.ry(a, b), sg);
          sub_sigma(Wp, Wn, sg, ratio(4));
          if (Z) {
            lds_get6(SZ, I::NC, X.cc(a, b), sc);
            sub_sigma(Wp, Wn, sc, ratio(5));
          }
          if (negative(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          if (Z && P.ctu3d) {
            // sigma_z over j with the y eigen system, sigma_y over k with z's
            e1 = e2 = e0;
            e1.un = Vc[P_VELY];
            e2.un = Vc[P_VELZ];
            lds_get6(SZ, I::NC, X.cc(a, b - 1), sm);
            lds_get6(SZ, I::NC, X.cc(a, b + 1), sp);
            trans_sigma<1>(P, sm, sc, sp, e1, tA);
            lds_get6(SY + ring(k - 1) * 6 * I::NRY, I::NRY, X.ry(a, b), sm);
            lds_get6(SY + ring(k + 1) * 6 * I::NRY, I::NRY, X.ry(a, b), sp);
            trans_sigma<2>(P, sm, sg, sp, e2, tB);
            add_ctu(Wp, Wn, tA, tB, ratio(6));
            if (nonpositive(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          }
          lds_put6(WX, I::NRY, X.ry(a, b), Wp);
          psum = Wn[P_PRES] + Wp[P_PRES];
          keep(Wn);
        } else if (w < B2) {
          const int w2 = w - B1;
          if (!interior || w2 >= X.nrx()) return;
          int a, b;
          shape.row(w2, a, b);
          --b;
          if (b == ty && !ey && !FUSE) return;
          const bool own = (b >= 0 || oy == P.lo[1]) && (b < ty || ey);
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
          tv_prim(tv, cb - syb, Vm);
          tv_prim(tv, cb, Vc);
          tv_prim(tv, cb + syb, Vp);
          const R* fy = FY + ringL(k) * I::NLY + X.ly(a, b);
          const R flat = P.flat ? flat_of(Vm[P_PRES], Vp[P_PRES], fy[-tx], fy[0], fy[tx]) : R(0.);
          const R* lyk = LY + ringL(k) * 6 * I::NLY;
          lds_get6(lyk, I::NLY, X.ly(a, b - 1), dbN);
          lds_get6(lyk, I::NLY, X.ly(a, b), db0);
          lds_get6(lyk, I::NLY, X.ly(a, b + 1), dbP);
          bad |= !eig_make<1>(Vc, e0);
          const R dmm = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb - 2 * syb)) : R(0.);
          const R dpp = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb + 2 * syb)) : R(0.);
          ppm_trace<1>(P, ratio(1), ratio(10), Vm, Vc, Vp, dmm, dpp, dbN, db0, dbP, flat, e0, Wp, Wn);
          lds_get6(sxk, I::NRX, X.rx(a, b), sg);
          sub_sigma(Wp, Wn, sg, ratio(3));
          if (Z) {
            lds_get6(SZ, I::NC, X.cc(a, b), sc);
            sub_sigma(Wp, Wn, sc, ratio(5));
          }
          if (negative(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          if (Z && P.ctu3d) {
            // sigma_x over k with z's eigen system, sigma_z over i with x's
            e1 = e2 = e0;
            e1.un = Vc[P_VELZ];
            e2.un = Vc[P_VELX];
            lds_get6(SX + ring(k - 1) * 6 * I::NRX, I::NRX, X.rx(a, b), sm);
            lds_get6(SX + ring(k + 1) * 6 * I::NRX, I::NRX, X.rx(a, b), sp);
            trans_sigma<2>(P, sm, sg, sp, e1, tA);
            lds_get6(SZ, I::NC, X.cc(a - 1, b), sm);
            lds_get6(SZ, I::NC, X.cc(a + 1, b), sp);
            trans_sigma<0>(P, sm, sc, sp, e2, tB);
            add_ctu(Wp, Wn, tA, tB, ratio(7));
            if (nonpositive(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          }
          lds_put6(WY, I::NRX, X.rx(a, b), Wp);
          PY[X.rx(a, b)] = Wn[P_PRES] + Wp[P_PRES];
          keep(Wn);
        } else if (Z && w < B3) {
          const int w2 = w - B2;
          if (SH::kFree && w2 >= X.ncol()) return;
          int a, b;
          shape.row(w2, a, b);
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
          tv_prim(tv, cb - szb, Vm);
          tv_prim(tv, cb, Vc);
          tv_prim(tv, cb + szb, Vp);
          const R flat = P.flat ? flat_of(Vm[P_PRES], Vp[P_PRES], FZ[ring(k - 1) * NCOL + w2],
                                          FZ[ring(k) * NCOL + w2], FZ[ring(k + 1) * NCOL + w2])
                                : R(0.);
          lds_get6(LZ + ring(k - 1) * 6 * NCOL, NCOL, w2, dbN);
          lds_get6(LZ + ring(k) * 6 * NCOL, NCOL, w2, db0);
          lds_get6(LZ + ring(k + 1) * 6 * NCOL, NCOL, w2, dbP);
          bad |= !eig_make<2>(Vc, e0);
          const R dmm = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb - 2 * szb)) : R(0.);
          const R dpp = P.steep ? R(tv_ld(tv, tv.ob[P_DENS], cb + 2 * szb)) : R(0.);
          ppm_trace<2>(P, ratio(2), ratio(11), Vm, Vc, Vp, dmm, dpp, dbN, db0, dbP, flat, e0, Wp, Wn);
          lds_get6(sxk, I::NRX, X.rx(a, b), sc);
          sub_sigma(Wp, Wn, sc, ratio(3));
          lds_get6(syk, I::NRY, X.ry(a, b), sg);
          sub_sigma(Wp, Wn, sg, ratio(4));
          const bool own = (k >= klo || klo == P.lo[2]) && (k <= khi || khi == P.hi[2]);
          if (negative(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          if (P.ctu3d) {
            // sigma_y over i with x's eigen system, sigma_x over j with y's
            e1 = e2 = e0;
            e1.un = Vc[P_VELX];
            e2.un = Vc[P_VELY];
            lds_get6(syk, I::NRY, X.ry(a - 1, b), sm);
            lds_get6(syk, I::NRY, X.ry(a + 1, b), sp);
            trans_sigma<0>(P, sm, sg, sp, e1, tA);
            lds_get6(sxk, I::NRX, X.rx(a, b - 1), sm);
            lds_get6(sxk, I::NRX, X.rx(a, b + 1), sp);
            trans_sigma<1>(P, sm, sc, sp, e2, tB);
            add_ctu(Wp, Wn, tA, tB, ratio(8));
            if (nonpositive(Wp, Wn)) fallback_first_order(Vc, Wp, Wn, st, own);
          }
          // the column's Wp stays with its thread: last plane's out, this one's in
#pragma unroll
          for (int q = 0; q < 6; ++q) {
            Wo[q] = M::WZ_LDS ? WZ[q * NCOL + w2] : Wt[q];
            if (!M::WZ_LDS) Wt[q] = Wp[comp_slot(q)];
          }
          if (M::WZ_LDS) lds_put6(WZ, NCOL, w2, Wp);
          PZ[w2] = Wn[P_PRES] + Wp[P_PRES];
          keep(Wn);
        }
      };
      // first, so that its stores are on their way during the state cell
      if (FUSE && Z) stageD(k);
      itemB(item_index<OPAQUE>(tid));
    }
    lds_barrier();

    // ------------------------------ stage C ------------------------------
    {
      auto right = [&](R VR[8]) {
#pragma unroll
        for (int q = 0; q < 6; ++q) VR[comp_slot(q)] = Wk[q];
      };
      auto gammas = [&](unsigned cl, unsigned cr, R VL[8], R VR[8]) {
        VL[P_GAMC] = R(tv_ld(tv, tv.ob[P_GAMC], cl));
        VL[P_GAME] = R(tv_ld(tv, tv.ob[P_GAME], cl));
        VR[P_GAMC] = R(tv_ld(tv, tv.ob[P_GAMC], cr));
        VR[P_GAME] = R(tv_ld(tv, tv.ob[P_GAME], cr));
      };
      auto itemC = [&](int w) {
        R VL[8], VR[8];
        double F[8];
        if (w < B1) {
          if (!interior || w >= X.nry()) return;
          int a, b;
          shape.row2(w, a, b);
          --a;
          if (a < 0 || (a == tx && !ex && !FUSE)) return;
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
          if (P.aux && a < tx) {
            // face-averaged pressure (hy_getFaceFlux.F90:507-561 and the
            // y, z analogues)
            R pres = R(0.5) * psum;
            pres = pres * R(0.5) + PY[X.rx(a, b)] * R(0.25);
            if (Z) pres = div_const<6>(pres * R(4.0) + PZ[X.uy(a, b)]);
            if constexpr (FUSE) PA[X.uy(a, b)] = pres;
            else st_at(as_global(T.pavg), cell_r(ox + a, oy + b, k) * 8u, double(pres));
          }
          lds_get6(WX, I::NRY, X.ry(a - 1, b), VL);
          right(VR);
          gammas(cb - sxb, cb, VL, VR);
          const unsigned fr = (unsigned)face_index(P, 0, ox + a, oy + b, k);
          if constexpr (is_states(RS)) {
            write_face_states<0>(P, fsb + fstate_dir_offset(P, 0), fr, VL, VR);
            if (L.strongList) list_strong_face<0>(P, L, t, fr, VL, VR);
          } else {
            if (face_flux<0, RS>(P, VL, VR, tv_use_hll<RS>(P, tv, cb - sxb, cb), F, es)) { report_error(st, 2, t, ox + a, oy + b, k, 0); return; }
            if constexpr (FUSE) put_flux(UX, I::NFX, X.ux(a, b), F);
            else write_flux_b<0>(P, as_global(T.flux[0]), fr * 8u, F);
          }
        } else if (w < B2) {
          const int w2 = w - B1;
          if (!interior || w2 >= X.nrx()) return;
          int a, b;
          shape.row(w2, a, b);
          --b;
          if (b < 0 || (b == ty && !ey && !FUSE)) return;
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
          lds_get6(WY, I::NRX, X.rx(a, b - 1), VL);
          right(VR);
          gammas(cb - syb, cb, VL, VR);
          const unsigned fr = (unsigned)face_index(P, 1, ox + a, oy + b, k);
          if constexpr (is_states(RS)) {
            write_face_states<1>(P, fsb + fstate_dir_offset(P, 1), fr, VL, VR);
            if (L.strongList) list_strong_face<1>(P, L, t, fr, VL, VR);
          } else {
            if (face_flux<1, RS>(P, VL, VR, tv_use_hll<RS>(P, tv, cb - syb, cb), F, es)) { report_error(st, 2, t, ox + a, oy + b, k, 1); return; }
            if constexpr (FUSE) put_flux(UY, I::NFY, X.uy(a, b), F);
            else write_flux_b<1>(P, as_global(T.flux[1]), fr * 8u, F);
          }
        } else if (Z && w < B3) {
          const int w2 = w - B2;
          // the face above a segment is the next one's, unless the update needs it here
          if (k < klo || (!FUSE && k > khi && khi < P.hi[2])) return;
          if (SH::kFree && w2 >= X.ncol()) return;
          int a, b;
          shape.row(w2, a, b);
          const unsigned cb = cell_b(P, ox + a, oy + b, k);
#pragma unroll
          for (int q = 0; q < 6; ++q) VL[comp_slot(q)] = Wo[q];
          right(VR);
          gammas(cb - szb, cb, VL, VR);
          const unsigned fr = (unsigned)face_index(P, 2, ox + a, oy + b, k);
          if constexpr (is_states(RS)) {
            write_face_states<2>(P, fsb + fstate_dir_offset(P, 2), fr, VL, VR);
            if (L.strongList) list_strong_face<2>(P, L, t, fr, VL, VR);
          } else {
            if (face_flux<2, RS>(P, VL, VR, tv_use_hll<RS>(P, tv, cb - szb, cb), F, es)) { report_error(st, 2, t, ox + a, oy + b, k, 2); return; }
            if constexpr (FUSE) put_flux(UZ, NCOL, w2, F);
            else write_flux_b<2>(P, as_global(T.flux[2]), fr * 8u, F);
          }
        }
      };
      itemC(item_index<OPAQUE>(tid));
    }
    if (k < kEnd) stageA(k + 1);
    lds_barrier();
  }
  if constexpr (FUSE != kFuseNone) {  // the last plane
    stageD(Z ? kEnd + 1 : kEnd);
    __syncthreads();  // (and the scratch rows reach the cache)
  }
  if (bad) report_error(st, 1, t, ox, oy, -1, -1);
}

// The column tiles of a block one column tile wide, in rising y, updated in
// place (kFuseDirect).  A tile reads the block from kSeamRows rows below its
// own up, so the top kSeamRows rows of each tile but the last wait in scratch
// until the next tile is done.
template <int NDIM, int TX, int TY, int NT, int RS, typename R>
__device__ __forceinline__ void march_block(const DevParams& P, const MarchLaunch& L, int t,
                                            ExactStats& es, R* smem) {
  // read before anything is stored: scalar loads
  const fx_tile T = L.tiles[t];
  for (int ty = 0; ty < L.tilesY; ++ty) {
    const int oy = P.lo[1] + ty * TY;
    march_tile<NDIM, TX, TY, NT, RS, R, true, kFuseDirect>(P, L, T, t, P.lo[0], oy, nullptr, es, smem,
                                                           FixedShape<TX, TY>{}, P.lo[2], P.hi[2]);
    if (ty == 0) continue;
    const TileView tv = tile_view(P, as_global(T.U));
    const gdouble* const upd = as_global(L.upd + (long)t * (kUpdComps * P.icells));
    const int j0 = oy - kSeamRows, items = P.nzb * kSeamRows * TX;
    for (int w = threadIdx.x; w < items; w += NT) {
      const int i = P.lo[0] + w % TX, j = j0 + (w / TX) % kSeamRows;
      const int k = P.lo[2] + w / (TX * kSeamRows);
      const unsigned r =
          (unsigned)(((k - P.lo[2]) * P.nyb + (j - P.lo[1])) * P.nxb + (i - P.lo[0])) * 8u;
      tv_expand(P, tv, cell_b(P, i, j, k),
                UpdState{ld_at(upd, r), ld_at(upd + P.icells, r), ld_at(upd + 2 * P.icells, r),
                         ld_at(upd + 3 * P.icells, r), ld_at(upd + 4 * P.icells, r)});
    }
  }
}

// the tile, column tile and first plane of a workgroup
struct MarchPlace {
  int t, tx, ty, klo;
};
__device__ __forceinline__ MarchPlace march_place(const DevParams& P, const MarchLaunch& L) {
  const int cols = L.tilesX * L.tilesY, per = cols * L.tilesZ;
  const int t = blockIdx.x / per, tr = blockIdx.x - t * per;
  const int tz = tr / cols, tc = tr - tz * cols;
  return MarchPlace{t, tc % L.tilesX, tc / L.tilesX, P.lo[2] + (L.tilesZ > 1 ? tz * L.nzSeg : 0)};
}

// One workgroup per column tile of a batch of equal-shape tiles, or per
// segment of one along z where column tiles alone leave the chip idle (a
// segment forms the states and sigmas of the planes next to it anew: three
// planes' work).  OCC > 0
// asks the compiler for OCC waves per SIMD (fewer registers, maybe spills);
// without the update the autotuner decides whether that pays in FP32.  The FP64
// 16x8 tile runs 768 threads: its LDS allows one workgroup per CU, stage A has
// 12 wavefronts of items, and 3 waves per SIMD leave 168 registers, of which
// the form with the update in place spills 10 (at 512 threads and 176 registers
// the step of 4096 x 16^3 takes 6.40 instead of 5.80 ms).
template <int NDIM, int TX, int TY, int NT, int RS, typename R, int OCC = 0, int FUSE = kFuseNone>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(OCC > 0 ? OCC : 1)))
k_march(DevParams P, MarchLaunch L) {
  if constexpr (FUSE == kFuseDirect) {  // one workgroup per block
    ExactStats es{0ULL, 0ULL};
    __shared__ R smem[MarchLds<NDIM, TX, TY, FUSE>::total];
    march_block<NDIM, TX, TY, NT, RS, R>(P, L, (int)blockIdx.x, es, smem);
    return;
  }
  const MarchPlace w = march_place(P, L);
  const int t = w.t, ox = P.lo[0] + w.tx * TX, oy = P.lo[1] + w.ty * TY, klo = w.klo;
  ExactStats es{0ULL, 0ULL};
  R* fsb = is_states(RS) ? static_cast<R*>(L.fstates) + t * fstate_tile_stride(P) : nullptr;
  __shared__ R smem[MarchLds<NDIM, TX, TY, FUSE>::total];
  march_tile<NDIM, TX, TY, NT, RS, R, true, FUSE>(P, L, L.tiles[t], t, ox, oy, fsb, es, smem, FixedShape<TX, TY>{},
                                                  klo, min(klo + L.nzSeg - 1, P.hi[2]));
  flush_exact(L.status, es);
}

// One workgroup per column tile of a batch of blocks that no fixed tile
// divides (extents not multiples of 8): tiles of L.tx x L.ty columns in the
// 16x8 layout, with the update (kFuseScratch, or kFuseDirect for blocks of one
// tile).  A row's length is then a value instead of a constant, which costs a
// reciprocal multiplication per item; its loads, arithmetic and bits are the
// fixed tile's.
// Bound by FP64 issue and latency as k_march, and by what of the 128 columns a
// tile leaves idle.  952 blocks of 12 x 10 x 14 664 us against 1460 by the three-
// kernel path (face states through memory, transverse fluxes formed anew by
// each state cell), 402 of 13 x 17 x 18 853 / 1399, 7407 of 6^3 1669 / 2026.
template <int NDIM, int NT, int RS, typename R, int OCC, int FUSE>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(OCC > 0 ? OCC : 1)))
k_march_free(DevParams P, MarchLaunch L) {
  const MarchPlace w = march_place(P, L);
  const int t = w.t, ox = P.lo[0] + w.tx * L.tx, oy = P.lo[1] + w.ty * L.ty, klo = w.klo;
  const FreeShape shape(min(L.tx, P.hi[0] + 1 - ox), min(L.ty, P.hi[1] + 1 - oy));
  ExactStats es{0ULL, 0ULL};
  __shared__ R smem[MarchLds<NDIM, 16, 8, FUSE>::total];
  const fx_tile T = L.tiles[t];
  march_tile<NDIM, 16, 8, NT, RS, R, true, FUSE>(P, L, T, t, ox, oy, nullptr, es, smem, shape, klo,
                                                  min(klo + L.nzSeg - 1, P.hi[2]));
}

// Tiles of several block classes in one persistent launch: workgroup b takes
// the column tiles b, b + G, b + 2G, ... of the item list (G = grid size).
// The host orders the items by falling column height, so the round-robin
// deals the long columns first and the short ones fill in behind them.
struct MarchItem {
  int t, cls, ox, oy;  // tile, its class, column-tile origin (guard-inclusive)
  int tx;              // column-tile width of the item (mixed-width launches)
};

template <int NDIM, int TX, int TY, int NT, int RS, typename R, int OCC = 0>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(OCC > 0 ? OCC : 1)))
k_march_multi(const DevParams* __restrict__ cls,
                                                    MarchLaunch L,
                                                    const MarchItem* __restrict__ items,
                                                    int nItems, const long* __restrict__ faceStart) {
  ExactStats es{0ULL, 0ULL};
  __shared__ R smem[MarchLds<NDIM, TX, TY, kFuseNone>::total];
  for (int it = blockIdx.x; it < nItems; it += gridDim.x) {
    const MarchItem w = items[it];
    const DevParams& P = cls[w.cls];
    const long faceBase = is_states(RS) ? faceStart[w.t] : 0;
    R* fsb = is_states(RS) ? static_cast<R*>(L.fstates) + kFaceComps * faceBase : nullptr;
    march_tile<NDIM, TX, TY, NT, RS, R, true, kFuseNone>(P, L, L.tiles[w.t], w.t, w.ox, w.oy, fsb, es, smem,
                                                         FixedShape<TX, TY>{}, P.lo[2], P.hi[2]);
  }
  flush_exact(L.status, es);
}

// The same with the column-tile width chosen per item: 16 columns across x
// for classes whose x extent allows it, 8 for the others.  One LDS array of
// the larger layout serves both; NT is the 16-wide tile's thread count.
template <int NDIM, int NT, int RS, typename R, int OCC = 0>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(OCC > 0 ? OCC : 1)))
k_march_mixw(const DevParams* __restrict__ cls, MarchLaunch L,
             const MarchItem* __restrict__ items, int nItems, const long* __restrict__ faceStart) {
  ExactStats es{0ULL, 0ULL};
  constexpr int n16 = MarchLds<NDIM, 16, 8, kFuseNone>::total,
                n8 = MarchLds<NDIM, 8, 8, kFuseNone>::total;
  __shared__ R smem[n16 > n8 ? n16 : n8];
  for (int it = blockIdx.x; it < nItems; it += gridDim.x) {
    const MarchItem w = items[it];
    const DevParams& P = cls[w.cls];
    const long faceBase = is_states(RS) ? faceStart[w.t] : 0;
    R* fsb = is_states(RS) ? static_cast<R*>(L.fstates) + kFaceComps * faceBase : nullptr;
    if (w.tx == 16) march_tile<NDIM, 16, 8, NT, RS, R, true, kFuseNone>(P, L, L.tiles[w.t], w.t, w.ox, w.oy, fsb, es, smem,
                                                                         FixedShape<16, 8>{}, P.lo[2], P.hi[2]);
    else march_tile<NDIM, 8, 8, NT, RS, R, true, kFuseNone>(P, L, L.tiles[w.t], w.t, w.ox, w.oy, fsb, es, smem,
                                                                 FixedShape<8, 8>{}, P.lo[2], P.hi[2]);
  }
  flush_exact(L.status, es);
}

}  // namespace fx
