/*
 * lb.hip -- fused D3Q19 pull-stream + bounce-back + moments + BGK/Guo collide.
 *
 * One pass per step replaces the reference's four full-grid passes
 * (fluid3d_collision_kernel LB_kernel.cu:1203-1304, fluid3d_stream_kernel
 * LB_kernel.cu:1312-1359, fluid3d_velocity_density_kernel LB_kernel.cu:1108-1199
 * and the wall kernels LB_kernel.cu:395-780): each cell pulls its 19
 * post-collision populations from the upstream neighbours of the previous step
 * (bounce-back where the upstream cell is a wall or a solid cell), takes its
 * moments with the current force, relaxes and writes its 19 new populations.
 * Each population is read once and written once: 152 B per cell update in
 * FP32 storage, 76 B in 16-bit storage.
 *
 * Storage holds deviations f_i - w_i (FP32), (f_i - w_i) * 2^s (FP16) or
 * f_i - w_i (BF16).  Arithmetic is FP32 in deviation form throughout
 * (rho - 1 = sum of deviations), so FP32 rounding acts on the deviations and
 * not on the O(1) weights; FP16 values stay in the scaled space and only the
 * four moments are unscaled.
 *
 * Layout (blocked SoA): the cells i = x + nx (y + ny z) of a lattice are cut
 * into blocks of 64 consecutive ones (one wavefront), across rows.  Block b
 * stores its 19 directions as 19 consecutive chunks of 64 values:
 *     element(d, i) = ((i / 64) * 19 + d) * 64 + i % 64.
 * A wavefront updates one block: its 19 stores fill one contiguous
 * 19*64-value segment, and each of its loads reads the 64 values of one
 * direction at a constant offset in i (one run in two neighbouring blocks),
 * so DRAM pages are reused across the directions instead of streaming 38
 * separate planes.  Only the last block of a lattice is partly empty: blocks
 * cut from each row, an earlier form, left a third of them empty in a batch
 * of lattices of 32 to 96 cells in x.
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <vector>

#include "pfg_internal.h"

namespace pfg {

/* ---------------- storage formats ---------------- */

/* Raw: a stored value in a register of its own (an array of 16-bit values that
 * is carried across branches is packed in pairs, each wait for the load of
 * one of a pair); value: a stored value as float (FP16 values stay scaled by
 * 2^s); pack: an already scaled value as it is stored. */
template <int S>
struct Store;

template <>
struct Store<PFG_STORE_F32> {
  using T = float;
  using Raw = float;
  static constexpr bool scaled = false;
  __device__ static inline float value(Raw v) { return v; }
  __device__ static inline T pack(float v) { return v; }
};

template <>
struct Store<PFG_STORE_F16> {
  using T = uint16_t;
  using Raw = uint32_t;
  static constexpr bool scaled = true;
  __device__ static inline float value(Raw v) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)v);
  }
  __device__ static inline T pack(float v) {
    return __builtin_bit_cast(uint16_t, (_Float16)v); /* round to nearest even */
  }
};

template <>
struct Store<PFG_STORE_BF16> {
  using T = uint16_t;
  using Raw = uint32_t;
  static constexpr bool scaled = false;
  __device__ static inline float value(Raw v) { return __builtin_bit_cast(float, v << 16); }
  __device__ static inline T pack(float v) {
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    u += 0x7FFFu + ((u >> 16) & 1u); /* round to nearest even */
    return (uint16_t)(u >> 16);
  }
};

/* Store value v; CACHED: through the caches, else streamed past them. */
template <int S, bool CACHED>
__device__ inline void put(typename Store<S>::T *p, float v) {
  if (CACHED) *p = Store<S>::pack(v);
  else __builtin_nontemporal_store(Store<S>::pack(v), p);
}

/* Element of direction d of cell i. */
__device__ __host__ inline int64_t felem(int d, int64_t i) {
  return ((i >> 6) * Q + d) * XBLOCK + (i & (XBLOCK - 1));
}

/* ---------------- the fused kernel ---------------- */

/* STEP: every block, with the IB force in flagged tiles.  FIELDS: rho and u
 * only.  BULK / REGION: the blocks whose stamp is not / is the current step
 * (blocks that this step's IB stencils touch), without / with the IB force. */
enum { LB_MODE_STEP = 0, LB_MODE_FIELDS = 1, LB_MODE_BULK = 2, LB_MODE_REGION = 3 };
/* Flag bit of MODE: the lattice has velocity faces on z (compiled only into
 * the variant that needs it, which keeps the scalar registers and the
 * occupancy of the default kernels). */
enum { LB_ZVEL = 4 };
/* Flag bit of MODE: the new populations are stored through the caches (they
 * fit the 256 MB cache in front of HBM together with the old ones, and the
 * next step reads them from there); otherwise they are streamed past them. */
enum { LB_CACHED = 8 };

/* Velocity face z = 0 (s = +1) or z = nz-1 (s = -1) on the pulled
 * deviations (fluid3d_in_out_flow_boundary_kernel,
 * LB_kernel_old_08102011.cu:586-1090): face velocity = wall velocity x the
 * duct profile 4 q (L - q) / L^2, q = i + 1/2, over each bounded transverse
 * axis; a cell next to a transverse wall takes feq(1, u); the others
 * Zou/He on the populations entering from outside,
 *   rho = (1 + sum_{cz=0} dev + 2 sum_{cz=-s} dev) / (1 - s uz),
 *   dev_{s z} = dev_{-s z} + s rho uz / 3,
 *   dev_{s z, t} = dev_{opp} + rho (s uz + c_t u_t) / 6 - c_t N_t,
 *   N_t = 1/2 sum_{cz=0} c_t dev - rho u_t / 3
 * (the weights cancel between opposite directions, so deviations take the
 * place of populations except in rho).  dev in storage units. */
template <class ST>
__device__ __forceinline__ void velocity_face(const LBArgs &a, int x, int y, int s,
                                              float dev[Q]) {
  const float *U = s > 0 ? a.zvel_u[0] : a.zvel_u[1];
  float shape = 1.0f;
  if (!a.periodic[0]) {
    const float q = (float)x + 0.5f;
    shape *= 4.0f * q * ((float)a.nx - q) / ((float)a.nx * (float)a.nx);
  }
  if (!a.periodic[1]) {
    const float q = (float)y + 0.5f;
    shape *= 4.0f * q * ((float)a.ny - q) / ((float)a.ny * (float)a.ny);
  }
  const float ux = U[0] * shape, uy = U[1] * shape, uz = U[2] * shape;
  const float sc = ST::scaled ? a.scale : 1.0f, isc = ST::scaled ? a.inv_scale : 1.0f;
  if ((!a.periodic[0] && (x == 0 || x == a.nx - 1)) ||
      (!a.periodic[1] && (y == 0 || y == a.ny - 1))) {
    const float usq = ux * ux + uy * uy + uz * uz;
#pragma unroll
    for (int d = 0; d < Q; ++d) {
      const float cu = 3.0f * (CX[d] * ux + CY[d] * uy + CZ[d] * uz);
      dev[d] = sc * weight(d) * (cu + 0.5f * cu * cu - 1.5f * usq);
    }
    return;
  }
  float S0 = 0.f, Sm = 0.f, Nx = 0.f, Ny = 0.f;
#pragma unroll
  for (int d = 0; d < Q; ++d) {
    if (CZ[d] == 0) {
      S0 += dev[d];
      Nx += CX[d] * dev[d];
      Ny += CY[d] * dev[d];
    } else if (CZ[d] == -s) {
      Sm += dev[d];
    }
  }
  const float rho = (1.0f + (S0 + 2.0f * Sm) * isc) / (1.0f - (float)s * uz);
  Nx = 0.5f * Nx * isc - rho * ux / 3.0f;
  Ny = 0.5f * Ny * isc - rho * uy / 3.0f;
#pragma unroll
  for (int d = 0; d < Q; ++d) {
    if (CZ[d] != s) continue;
    float t;
    if (CX[d] != 0) t = rho * ((float)s * uz + CX[d] * ux) / 6.0f - CX[d] * Nx;
    else if (CY[d] != 0) t = rho * ((float)s * uz + CY[d] * uy) / 6.0f - CY[d] * Ny;
    else t = (float)s * rho * uz / 3.0f;
    dev[d] = dev[BB[d]] + sc * t;
  }
}

/* The update of one cell from its pulled deviations: velocity face, moments,
 * collision, stores (own: the cell's element of direction 0 in the new
 * copy).  MODE as in lb_update. */
template <int S, int MODE>
__device__ __forceinline__ void lb_cell(const LBArgs &a, float (&dev)[Q], int x, int y, int z0,
                                        int z1, int64_t idx, bool flagged, float ax, float ay,
                                        float az, typename Store<S>::T *own, float *orho,
                                        float *oux, float *ouy, float *ouz) {
  constexpr int M = MODE & 3;
  constexpr bool ZV = (MODE & LB_ZVEL) != 0, CACHED = (MODE & LB_CACHED) != 0;
  using ST = Store<S>;
  const float isc = ST::scaled ? a.inv_scale : 1.0f;
  if (ZV && (z0 || z1)) velocity_face<ST>(a, x, y, z0 ? 1 : -1, dev);

  /* moments: rho - 1 and momentum from deviations (sum_i w_i c_i = 0),
   * over the nine pairs (d, opposite of d): the pair sum feeds the density,
   * the pair difference the momentum.  -0.0f starts are exact no-ops. */
  float drho = dev[0], jx = -0.0f, jy = -0.0f, jz = -0.0f;
#pragma unroll
  for (int d = 1; d < Q; ++d) {
    if (d < BB[d]) {
      const float s = dev[d] + dev[BB[d]], df = dev[d] - dev[BB[d]];
      drho += s;
      if (CX[d] > 0) jx += df; else if (CX[d] < 0) jx -= df;
      if (CY[d] > 0) jy += df; else if (CY[d] < 0) jy -= df;
      if (CZ[d] > 0) jz += df; else if (CZ[d] < 0) jz -= df;
    }
  }
  if (ST::scaled) {
    drho *= isc;
    jx *= isc;
    jy *= isc;
    jz *= isc;
  }
  const float rho = 1.0f + drho;
  float Fx = a.g[0], Fy = a.g[1], Fz = a.g[2];
  if (flagged) {
    Fx += ax;
    Fy += ay;
    Fz += az;
  }
  const float inv_rho = __builtin_amdgcn_rcpf(rho); /* hardware reciprocal, 1 ulp */
  const float ux = (jx + 0.5f * Fx) * inv_rho;
  const float uy = (jy + 0.5f * Fy) * inv_rho;
  const float uz = (jz + 0.5f * Fz) * inv_rho;

  if (M == LB_MODE_FIELDS) {
    if (orho) orho[idx] = rho;
    if (oux) oux[idx] = ux;
    if (ouy) ouy[idx] = uy;
    if (ouz) ouz[idx] = uz;
    return;
  }
  if (flagged) { /* velocity for the IB interpolation of this step */
    a.vel[idx] = make_float4(ux, uy, uz, 0.f);
  }

  /* BGK with Guo forcing, in deviation form and storage units:
   *   out_d = (1-omega) dev_d + omega (feq_d - w_d) + guo w_d (3 (c_d-u).F + 9 (c_d.u)(c_d.F))
   * split into the part even in c_d,
   *   E = w_d [K0 + cu (4.5 omega rho cu + 9 guo cF)],
   *   K0 = omega (drho - 1.5 rho u.u) - 3 guo u.F,
   * and the odd part O = w_d (3 omega rho cu + 3 guo cF); the pair
   * (d, opposite) takes E + O and E - O. */
  const float usq = ux * ux + uy * uy + uz * uz;
  const float uF = ux * Fx + uy * Fy + uz * Fz;
  const float K0 = fmaf(-a.guo3, uF, a.omega * fmaf(-1.5f * rho, usq, drho));
  const float Ab = a.om45 * rho, Cp = a.om3 * rho;
  put<S, CACHED>(own, fmaf(a.keep, dev[0], a.ws[0] * K0));
#pragma unroll
  for (int d = 1; d < Q; ++d) {
    if (d < BB[d]) {
      const int k = d < 7 ? 1 : 2;
      float cu = -0.0f, cF = -0.0f;
      if (CX[d] > 0) { cu += ux; cF += Fx; } else if (CX[d] < 0) { cu -= ux; cF -= Fx; }
      if (CY[d] > 0) { cu += uy; cF += Fy; } else if (CY[d] < 0) { cu -= uy; cF -= Fy; }
      if (CZ[d] > 0) { cu += uz; cF += Fz; } else if (CZ[d] < 0) { cu -= uz; cF -= Fz; }
      const float t = fmaf(a.gB[k], cF, (a.ws[k] * Ab) * cu);
      const float E = fmaf(cu, t, a.ws[k] * K0);
      const float O = fmaf(a.gD[k], cF, (a.ws[k] * Cp) * cu);
      put<S, CACHED>(own + d * XBLOCK, fmaf(a.keep, dev[d], E + O));
      put<S, CACHED>(own + BB[d] * XBLOCK, fmaf(a.keep, dev[BB[d]], E - O));
    }
  }
}

/* The populations that come in from a wall: directions whose component along
 * axis AX has sign SGN, each the opposite one that leaves the cell (bb). */
template <int AX, int SGN, typename RAW, typename T>
__device__ __forceinline__ void bounce_loads(RAW (&pop)[Q], const T *bb) {
#pragma unroll
  for (int d = 1; d < Q; ++d)
    if ((AX == 0 ? CX[d] : (AX == 1 ? CY[d] : CZ[d])) == SGN) pop[d] = bb[BB[d] * XBLOCK];
}

/* One wavefront per block of 64 cells; workgroup `blk` of the lattice
 * described by `a` (in memory that the whole workgroup reads), the
 * wavefront's place in it `wave` (default: its place in the launch's
 * workgroup); cells outside [lo, hi) are left alone (field windows).
 *
 * Bound by HBM.  What keeps it there: a lane decodes its own (x, y, z) from
 * the wavefront's first cell (64 cells meet few rows) and adds per-axis
 * offsets, periodic wraps included, to its cell index, about 100 integer
 * instructions that need no load; every load that does not depend on another
 * (the tile stamp, the 19 populations) is issued before the first is waited
 * for; the stamped tiles' force loads follow while the populations are in
 * flight.  Against a kernel whose wavefronts took 64-cell blocks of whole
 * rows from wavefront-uniform addresses (LB-only launches, us): 256 lattices
 * of 32 to 96 cells per axis FP32 2540 -> 1800, FP16 1970 -> 1010; 201x99x75
 * FP32 45 -> 30; 128^3 FP16 41 -> 26; 256x128x128 FP16 64 -> 55, FP32
 * 109 -> 108; 1024x512x512 FP16 3600 -> 3330, FP32 6780 -> 6720; a 512x256x256
 * tube with solid cells FP32 632 -> 587, FP16 342 -> 294. */
template <int S, int MODE>
__device__ __forceinline__ void lb_update(const LBArgs &a, uint32_t blk, float *orho,
                                          float *oux, float *ouy, float *ouz, int wave = -1,
                                          uint32_t lo = 0, uint32_t hi = ~0u) {
  constexpr int M = MODE & 3;
  using ST = Store<S>;
  using T = typename ST::T;
  constexpr uint32_t R = Q * XBLOCK; /* values per block */
  const T *__restrict__ fin = (const T *)a.fin;
  T *__restrict__ fout = (T *)a.fout;
  if (M != LB_MODE_FIELDS && a.halt != nullptr && *a.halt != 0) return;
  const uint32_t task =
      blk * 4u + __builtin_amdgcn_readfirstlane(wave < 0 ? (int)(threadIdx.x >> 6) : wave);
  const uint32_t i0 = task * XBLOCK;
  if (i0 >= a.ncell) return;
  /* IB force tiles and blocks are stamped with the step that touches them */
  const int32_t step32 = M == LB_MODE_FIELDS ? 0 : (int32_t)*a.step;
  if (M == LB_MODE_BULK || M == LB_MODE_REGION) {
    const bool touched = a.row_stamp[task] == step32;
    if (touched != (M == LB_MODE_REGION)) return;
  }
  const int kind = a.block_kind != nullptr ? a.block_kind[task] : BLOCK_FLUID;
  if (M != LB_MODE_FIELDS && kind == BLOCK_SOLID) return;
  const uint32_t lane = threadIdx.x & (XBLOCK - 1);
  const uint32_t i = i0 + lane;
  if (i < lo || i >= hi || i >= a.ncell) return;
  uint32_t mask = 0;
  if (kind != BLOCK_FLUID) {
    mask = a.bbmask[i];
    if (mask >> 31) { /* solid cell: its fields read 0 */
      if (M == LB_MODE_FIELDS) {
        if (orho) orho[i] = 0.f;
        if (oux) oux[i] = 0.f;
        if (ouy) ouy[i] = 0.f;
        if (ouz) ouz[i] = 0.f;
      }
      return;
    }
  }
  const bool wall_moves = a.wall_moves != 0;
  const uint32_t nx = (uint32_t)a.nx, ny = (uint32_t)a.ny, nxy = nx * ny;
  const uint32_t wz = i0 / nxy, wr = i0 - wz * nxy, wy = wr / nx, wx = wr - wy * nx;
  /* rows and planes passed since the wavefront's first cell: at most one of a
   * row longer than the wavefront; shorter ones by the reciprocal (v < 128,
   * and (v + 1/2) / n is at least 1/128 from an integer) */
  const uint32_t vx = wx + lane;
  const uint32_t qy = nx > XBLOCK ? (vx >= nx ? 1u : 0u)
                                  : (uint32_t)(((float)vx + 0.5f) * a.inv_nx);
  const uint32_t vy = wy + qy;
  const uint32_t qz = ny > XBLOCK ? (vy >= ny ? 1u : 0u)
                                  : (uint32_t)(((float)vy + 0.5f) * a.inv_ny);
  const int x = (int)(vx - qy * nx), y = (int)(vy - qz * ny), z = (int)(wz + qz);
  int32_t stamp = 0;
  if (M == LB_MODE_STEP || M == LB_MODE_REGION)
    stamp = a.tile_stamp[(x >> TILE_SHIFT_X) +
                         a.tnx * ((y >> TILE_SHIFT_Y) + a.tny * (z >> TILE_SHIFT_Z))];
  /* offset to the upstream neighbour along each axis, 0 outside a wall (what
   * that reads is replaced) */
  const bool xlo = x == 0, xhi = x == a.nx - 1, ylo = y == 0, yhi = y == a.ny - 1,
             zlo = z == 0, zhi = z == a.nz - 1;
  const bool oxm = xlo && !a.periodic[0], oxp = xhi && !a.periodic[0];
  const bool oym = ylo && !a.periodic[1], oyp = yhi && !a.periodic[1];
  const bool ozm = zlo && !a.periodic[2], ozp = zhi && !a.periodic[2];
  const int sx = a.nx, sy = (int)nxy, sz = (int)a.ncell;
  const int xm = xlo ? (oxm ? 0 : sx - 1) : -1, xp = xhi ? (oxp ? 0 : 1 - sx) : 1;
  const int ym = ylo ? (oym ? 0 : sy - sx) : -sx, yp = yhi ? (oyp ? 0 : sx - sy) : sx;
  const int zm = zlo ? (ozm ? 0 : sz - sy) : -sy, zp = zhi ? (ozp ? 0 : sy - sz) : sy;
  const uint64_t own = (uint64_t)task * R + lane;
  const bool edge = oxm || oxp || oym || oyp || ozm || ozp || mask != 0;
  auto upstream = [&](int d) { /* element of direction 0 */
    const int off = (CX[d] > 0 ? xm : (CX[d] < 0 ? xp : 0)) +
                    (CY[d] > 0 ? ym : (CY[d] < 0 ? yp : 0)) +
                    (CZ[d] > 0 ? zm : (CZ[d] < 0 ? zp : 0));
    const uint32_t src = i + (uint32_t)off;
    return (uint64_t)(src >> 6) * R + (src & (XBLOCK - 1));
  };
  /* Upstream cell outside a wall or solid: halfway bounce-back, the
   * population leaving this cell returns.  No lane waits for a load here: a
   * second load of the same population comes after the first, and values are
   * used when all are on their way (a pass that took both and added the wall's
   * term in one branch waited once for each of a wavefront's directions).
   * Streamed FP32, bound by HBM, selects the address instead and loads once.
   * LB-only launches with walls on all sides, us, one pass after the other /
   * now: FP16 192^3 119 / 87, 256^3 261 / 209, 100^3 19.8 / 13.7, 512x256x256
   * 463 / 419; FP32 192^3 196 / 181, 256^3 463 / 434, 100^3 24.6 / 20.3,
   * 512x256x256 893 / 869 (selecting in FP16: 256^3 284, its arithmetic being
   * the limit; loading twice in FP32: 256^3 445, 512x256x256 899).  A tube's
   * mixed blocks: 256^3 FP16 157 / 153, 201x99x75 FP16 16.3 / 14.5, FP32
   * 20.6 / 19.2.  64x32x32 without walls 4.0 / 4.4, with 5.9 / 4.5. */
  constexpr bool SELECT = S == PFG_STORE_F32 && !(MODE & LB_CACHED);
  typename ST::Raw pop[Q];
  if (!SELECT || __ballot(edge) == 0) {
#pragma unroll
    for (int d = 0; d < Q; ++d) pop[d] = fin[d * XBLOCK + upstream(d)];
  } else {
#pragma unroll
    for (int d = 0; d < Q; ++d) {
      const bool oz = CZ[d] > 0 ? ozm : (CZ[d] < 0 ? ozp : false);
      const bool oy = CY[d] > 0 ? oym : (CY[d] < 0 ? oyp : false);
      const bool ox = CX[d] > 0 ? oxm : (CX[d] < 0 ? oxp : false);
      const bool out = oz || oy || ox || ((mask >> d) & 1u); /* never for d = 0 */
      pop[d] = fin[out ? own + BB[d] * XBLOCK : d * XBLOCK + upstream(d)];
    }
  }
  if (!SELECT && edge) {
    const T *bb = fin + own;
    if (oxm) bounce_loads<0, 1>(pop, bb);
    if (oxp) bounce_loads<0, -1>(pop, bb);
    if (oym) bounce_loads<1, 1>(pop, bb);
    if (oyp) bounce_loads<1, -1>(pop, bb);
    if (ozm) bounce_loads<2, 1>(pop, bb);
    if (ozp) bounce_loads<2, -1>(pop, bb);
    if (mask != 0) {
#pragma unroll
      for (int d = 1; d < Q; ++d)
        if ((mask >> d) & 1u) pop[d] = bb[BB[d] * XBLOCK];
    }
  }
  /* the IB force of the tiles this step's stencils meet, read and consumed
   * (the next step's spreading adds into zeros) */
  bool flagged = false;
  float ax = 0.f, ay = 0.f, az = 0.f;
  if (M == LB_MODE_STEP || M == LB_MODE_REGION) {
    flagged = stamp == step32;
    if (flagged) {
      ax = a.aux[i];
      ay = a.aux[a.plane + i];
      az = a.aux[2 * a.plane + i];
    }
  }
  float dev[Q];
#pragma unroll
  for (int d = 0; d < Q; ++d) dev[d] = ST::value(pop[d]);
  /* the moving wall's momentum 6 w (c . u_wall), z wall over y wall over x */
  if (wall_moves && edge) {
    int k = 0; /* keeps the loads of the terms in here */
    asm volatile("" : "+s"(k));
#pragma unroll
    for (int d = 1; d < Q; ++d) {
      const bool oz = CZ[d] > 0 ? ozm : (CZ[d] < 0 ? ozp : false);
      const bool oy = CY[d] > 0 ? oym : (CY[d] < 0 ? oyp : false);
      const bool ox = CX[d] > 0 ? oxm : (CX[d] < 0 ? oxp : false);
      const int sx = CX[d] > 0 ? 0 : 1, sy = CY[d] > 0 ? 0 : 1, sz = CZ[d] > 0 ? 0 : 1;
      const float tx = CX[d] != 0 ? a.wall_term[0][sx][d + k] : 0.f;
      const float ty = CY[d] != 0 ? a.wall_term[1][sy][d + k] : 0.f;
      const float tz = CZ[d] != 0 ? a.wall_term[2][sz][d + k] : 0.f;
      dev[d] += oz ? tz : (oy ? ty : (ox ? tx : 0.f));
    }
  }
  lb_cell<S, MODE>(a, dev, x, y, zlo, zhi, i, flagged, ax, ay, az, fout + own, orho, oux, ouy,
                   ouz);
  /* zeros only where a marker added: many cells of a stamped tile hold none
   * (all of the tile's: 5161 against 5098 us per step with 2000 platelets in
   * 1024x512x512 FP16, 1026 against 1015 with 500 in a tube, 2100 against 2055
   * for 256 lattices) */
  if (M == LB_MODE_STEP || M == LB_MODE_REGION) {
    if ((__float_as_uint(ax) | __float_as_uint(ay) | __float_as_uint(az)) != 0u) {
      a.aux[i] = 0.f;
      a.aux[a.plane + i] = 0.f;
      a.aux[2 * a.plane + i] = 0.f;
    }
  }
}

/* Workgroups are dealt round-robin to the 8 XCDs.  With xcd_rows each XCD
 * takes a contiguous range of blocks instead, so that neighbouring blocks
 * (which read each other's populations) share its L2; the autotuner picks
 * the order. */
__device__ inline uint32_t launch_block(int xcd_rows) {
  uint32_t blk = blockIdx.x;
  if (xcd_rows) {
    const uint32_t q = gridDim.x / 8u;
    if (blk < 8u * q) blk = (blk % 8u) * q + blk / 8u;
  }
  return blk;
}

/* CPT: cells per lane, from blocks that follow each other.  WAVES: the
 * wavefronts a SIMD holds at most. */
template <int S, int CPT, int MODE, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void
lb_fused_kernel(LBArgs a) {
  const uint32_t blk = launch_block(a.xcd_rows) * CPT;
  for (uint32_t c = 0; c < CPT; ++c)
    lb_update<S, MODE>(a, blk + c, nullptr, nullptr, nullptr, nullptr);
}

/* A batch of lattices in one launch: workgroup task -> lattice through a
 * table of ntasks entries, each lattice's arguments read from device
 * memory. */
template <int S, int CPT, int MODE>
__global__ __launch_bounds__(256) void lb_batch_kernel(const LBArgs *args,
                                                       const int32_t *block_inst,
                                                       uint32_t ntasks, int xcd_rows) {
  const uint32_t blk = launch_block(xcd_rows) * CPT;
  for (uint32_t c = 0; c < CPT; ++c) {
    if (CPT > 1 && blk + c >= ntasks) return;
    const LBArgs &a = args[block_inst[blk + c]];
    lb_update<S, MODE>(a, (uint32_t)(blk + c - a.block0), nullptr, nullptr, nullptr, nullptr);
  }
}

/* A batch of lattices in one persistent launch: a grid of resident
 * workgroups whose wavefronts take the table's blocks (of any
 * lattice; row r is wavefront r % 4 of workgroup task r / 4) from a device
 * work queue until it is empty.  The rows are cut into LB_QUEUES contiguous
 * ranges, one per XCD (the hardware deals workgroup w to XCD w % 8), each
 * with its own counter, so neighbouring rows stay in one L2 and the counters
 * are not one hot spot; a grab takes LB_QUEUE_GRAB consecutive rows, and a
 * wavefront whose range is used up moves on to the next range.  Wavefronts
 * run on their own (no barrier).  queue[LB_QUEUES] counts the wavefronts
 * that are done; the last one resets every counter for the next launch (all
 * others have made their last grab by then), so a captured step needs no
 * clearing node. */
template <int S, int MODE>
__global__ __launch_bounds__(256) void lb_batch_queue_kernel(const LBArgs *args,
                                                             const int32_t *block_inst,
                                                             uint32_t ntasks, uint32_t *queue) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t nrows = ntasks * 4u;
  const uint32_t r0 = blockIdx.x % LB_QUEUES;
  for (uint32_t k = 0; k < LB_QUEUES; ++k) {
    const uint32_t r = (r0 + k) % LB_QUEUES;
    const uint32_t lo = (uint32_t)((uint64_t)nrows * r / LB_QUEUES);
    const uint32_t hi = (uint32_t)((uint64_t)nrows * (r + 1) / LB_QUEUES);
    for (;;) {
      uint32_t got = 0;
      if (lane == 0) got = atomicAdd(&queue[r], (uint32_t)LB_QUEUE_GRAB);
      got = __builtin_amdgcn_readfirstlane(__shfl(got, 0, 64));
      if (got >= hi - lo) break;
      const uint32_t t0 = lo + got;
      const uint32_t t1 = t0 + LB_QUEUE_GRAB < hi ? t0 + LB_QUEUE_GRAB : hi;
      for (uint32_t row = t0; row < t1; ++row) {
        const uint32_t blk = row >> 2;
        const LBArgs &a = args[block_inst[blk]];
        lb_update<S, MODE>(a, (uint32_t)(blk - a.block0), nullptr, nullptr, nullptr,
                                nullptr, (int)(row & 3u));
      }
    }
  }
  if (lane == 0) {
    __threadfence();
    if (atomicAdd(&queue[LB_QUEUES], 1u) == gridDim.x * 4u - 1u) {
      for (int r = 0; r <= LB_QUEUES; ++r) queue[r] = 0u;
      __threadfence();
    }
  }
}

/* ---------------- fields through a fixed device array ---------------- */

/* Staging of pfg_download_fields_noalloc: the fields of a window of whole
 * z-planes, [field][cell of the window].  One copy per device, held until the
 * process ends; calls on one device share it. */
static __device__ __align__(256) float scratch[FIELDS_SCRATCH_FLOATS];

/* The fields pass over the blocks [t0, t1) that hold the cells [lo, hi), one
 * wavefront per block; o* point lo cells before the window, so that each cell
 * lands at its offset in it. */
template <int S, int MODE>
__global__ __launch_bounds__(256) void lb_fields_window_kernel(LBArgs a, uint32_t blk0,
                                                               uint32_t t0, uint32_t t1,
                                                               uint32_t lo, uint32_t hi,
                                                               float *orho, float *oux,
                                                               float *ouy, float *ouz) {
  const uint32_t blk = blk0 + blockIdx.x;
  const uint32_t task = blk * 4u + (threadIdx.x >> 6);
  if (task < t0 || task >= t1) return;
  lb_update<S, MODE>(a, blk, orho, oux, ouy, ouz, -1, lo, hi);
}

/* Device address of `scratch` per device, looked up once with the device
 * current (the array's name in host code is a host-side stand-in). */
static std::mutex g_scratch_mu;
static float *g_scratch_ptr[FIELDS_SCRATCH_MAX_DEVICES];

hipError_t fields_scratch_setup(int device, float **out) {
  if (device < 0 || device >= FIELDS_SCRATCH_MAX_DEVICES) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = 0;
    hipError_t e = hipGetDevice(&cur);
    if (e != hipSuccess) return e;
    if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return e;
    void *ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (cur != device) hipSetDevice(cur);
    if (e != hipSuccess) return e;
    if (!ptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[device] = (float *)ptr;
  }
  if (out) *out = g_scratch_ptr[device];
  return hipSuccess;
}

template <int S>
static hipError_t fields_window_s(pfg_handle *h, const LBArgs &a, uint32_t lo, uint32_t hi,
                                  float *const win[4]) {
  const uint32_t t0 = lo / XBLOCK, t1 = (hi + XBLOCK - 1u) / XBLOCK;
  const uint32_t blk0 = t0 / 4u, blk1 = (t1 + 3u) / 4u;
  float *o[4];
  for (int c = 0; c < 4; ++c) o[c] = win[c] ? win[c] - (int64_t)lo : nullptr;
  if (a.zvel)
    hipLaunchKernelGGL((lb_fields_window_kernel<S, LB_MODE_FIELDS | LB_ZVEL>), dim3(blk1 - blk0),
                       dim3(256), 0, h->stream, a, blk0, t0, t1, lo, hi, o[0], o[1], o[2], o[3]);
  else
    hipLaunchKernelGGL((lb_fields_window_kernel<S, LB_MODE_FIELDS>), dim3(blk1 - blk0), dim3(256),
                       0, h->stream, a, blk0, t0, t1, lo, hi, o[0], o[1], o[2], o[3]);
  return hipGetLastError();
}

hipError_t launch_lb_fields_window(pfg_handle *h, int k, uint32_t lo, uint32_t hi,
                                   float *const win[4]) {
  LBArgs a;
  make_lb_args(h, k, h->cur, &a);
  switch (h->p.store) {
    case PFG_STORE_F16: return fields_window_s<PFG_STORE_F16>(h, a, lo, hi, win);
    case PFG_STORE_BF16: return fields_window_s<PFG_STORE_BF16>(h, a, lo, hi, win);
    default: return fields_window_s<PFG_STORE_F32>(h, a, lo, hi, win);
  }
}

hipError_t download_fields_noalloc(pfg_handle *h, float *const host[4]) {
  float *base = nullptr;
  hipError_t e = fields_scratch_setup(h->device, &base);
  if (e != hipSuccess) return e;
  int nf = 0;
  for (int c = 0; c < 4; ++c) nf += host[c] != nullptr;
  if (nf == 0) return hipSuccess;
  const int nz = h->p.nz;
  const int64_t plane = (int64_t)h->p.nx * h->p.ny;
  const int64_t zmax = FIELDS_SCRATCH_FLOATS / (plane * nf); /* planes per window */
  if (zmax < 1) return hipErrorInvalidValue;
  for (int z0 = 0; z0 < nz && e == hipSuccess; z0 += (int)zmax) {
    const int z1 = (int)std::min<int64_t>(nz, z0 + zmax);
    const int64_t n = plane * (z1 - z0);
    float *win[4] = {nullptr, nullptr, nullptr, nullptr};
    int slot = 0;
    for (int c = 0; c < 4; ++c)
      if (host[c]) win[c] = base + n * slot++;
    e = launch_lb_fields_window(h, 0, (uint32_t)(plane * z0), (uint32_t)(plane * z1), win);
    for (int c = 0; c < 4 && e == hipSuccess; ++c)
      if (host[c])
        e = hipMemcpyAsync(host[c] + (int64_t)z0 * plane, win[c], sizeof(float) * n,
                           hipMemcpyDeviceToHost, h->stream);
    /* the next window reuses the array */
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  }
  return e;
}

/* ---------------- auxiliary kernels ---------------- */

/* Per-cell bounce mask from the solid flags (built once per flag upload). */
__global__ void bbmask_kernel(LBArgs a, const uint8_t *solid, uint32_t *mask) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nxy = (int64_t)a.nx * a.ny;
  if (idx >= nxy * a.nz) return;
  if (solid[idx]) {
    mask[idx] = 1u << 31;
    return;
  }
  const int x = (int)(idx % a.nx), y = (int)((idx / a.nx) % a.ny), z = (int)(idx / nxy);
  uint32_t m = 0;
#pragma unroll
  for (int d = 1; d < Q; ++d) {
    int s[3] = {x - CX[d], y - CY[d], z - CZ[d]};
    const int n[3] = {a.nx, a.ny, a.nz};
    bool outside = false;
    for (int k = 0; k < 3; ++k) {
      if (s[k] < 0) {
        if (a.periodic[k]) s[k] += n[k]; else outside = true;
      } else if (s[k] >= n[k]) {
        if (a.periodic[k]) s[k] -= n[k]; else outside = true;
      }
    }
    if (!outside && solid[s[0] + (int64_t)a.nx * s[1] + nxy * s[2]]) m |= 1u << d;
  }
  mask[idx] = m;
}

/* Kind of each block, from its cells' masks: a wavefront per block.  The
 * update reads masks in mixed blocks only and leaves solid ones at once. */
__global__ __launch_bounds__(256) void block_kind_kernel(const uint32_t *mask, uint32_t ncell,
                                                         int32_t *kind) {
  const uint32_t task = blockIdx.x * 4u + (threadIdx.x >> 6);
  const uint32_t i = task * XBLOCK + (threadIdx.x & 63);
  if (task * XBLOCK >= ncell) return;
  const uint32_t m = i < ncell ? mask[i] : 0u;
  const uint64_t in = __ballot(i < ncell), any = __ballot(m != 0), solid = __ballot(m >> 31);
  if ((threadIdx.x & 63) == 0)
    kind[task] = solid == in ? BLOCK_SOLID : (any != 0 ? BLOCK_MIXED : BLOCK_FLUID);
}

/* per_z: the inputs hold one value per z-plane (a velocity that varies
 * along z only, like the reference's linear shear start) instead of one per
 * cell. */
template <int S>
__global__ void init_eq_kernel(LBArgs a, void *dst0, void *dst1, const float *rho_in,
                               const float *ux_in, const float *uy_in, const float *uz_in,
                               int64_t n, int per_z) {
  using ST = Store<S>;
  using T = typename ST::T;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  const int64_t src = per_z ? idx / ((int64_t)a.nx * a.ny) : idx;
  const float rho = rho_in ? rho_in[src] : 1.0f;
  const float ux = ux_in ? ux_in[src] : 0.f;
  const float uy = uy_in ? uy_in[src] : 0.f;
  const float uz = uz_in ? uz_in[src] : 0.f;
  const float usq15 = 1.5f * (ux * ux + uy * uy + uz * uz);
  const float drho = rho - 1.0f;
  const float sc = ST::scaled ? a.scale : 1.0f;
#pragma unroll
  for (int d = 0; d < Q; ++d) {
    const float w = weight(d);
    const float cu = CX[d] * ux + CY[d] * uy + CZ[d] * uz;
    const float dev = w * drho + w * rho * (3.0f * cu + 4.5f * cu * cu - usq15);
    const int64_t e = felem(d, idx);
    put<S, false>((T *)dst0 + e, dev * sc);
    put<S, false>((T *)dst1 + e, dev * sc);
  }
}

/* direction d: to_float -> buf[i] = w_d + dev; else stored <- buf[i] - w_d */
template <int S>
__global__ void convert_plane_kernel(LBArgs a, void *stored, float *buf, int d, int to_float,
                                     int64_t n) {
  using ST = Store<S>;
  using T = typename ST::T;
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= n) return;
  T *p = (T *)stored + felem(d, idx);
  const float w = weight(d);
  if (to_float) {
    buf[idx] = w + ST::value(*(p)) * (ST::scaled ? a.inv_scale : 1.0f);
  } else {
    put<S, false>(p, (buf[idx] - w) * (ST::scaled ? a.scale : 1.0f));
  }
}

/* FP64 totals of mass and momentum over fluid cells, one partial per block. */
template <int S>
__global__ __launch_bounds__(256) void conservation_kernel(LBArgs a, const void *stored,
                                                          double *partials, int64_t n) {
  using ST = Store<S>;
  using T = typename ST::T;
  const T *p = (const T *)stored;
  const double isc = ST::scaled ? (double)a.inv_scale : 1.0;
  double m = 0, jx = 0, jy = 0, jz = 0;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n;
       idx += (int64_t)gridDim.x * blockDim.x) {
    if (a.solid != nullptr && a.solid[idx]) continue;
    const int64_t e0 = felem(0, idx);
    double cm = 0, cx = 0, cy = 0, cz = 0;
#pragma unroll
    for (int d = 0; d < Q; ++d) {
      const double v = (double)ST::value(*(p + e0 + d * XBLOCK));
      cm += v;
      cx += CX[d] * v;
      cy += CY[d] * v;
      cz += CZ[d] * v;
    }
    m += 1.0 + cm * isc;
    jx += cx * isc;
    jy += cy * isc;
    jz += cz * isc;
  }
  __shared__ double sh[4][256];
  const int t = threadIdx.x;
  sh[0][t] = m;
  sh[1][t] = jx;
  sh[2][t] = jy;
  sh[3][t] = jz;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if (t < s) {
      for (int k = 0; k < 4; ++k) sh[k][t] += sh[k][t + s];
    }
    __syncthreads();
  }
  if (t == 0) {
    for (int k = 0; k < 4; ++k) partials[4 * blockIdx.x + k] = sh[k][0];
  }
}

/* ---------------- host launchers ---------------- */

/* Both copies of the populations, in bytes. */
static int64_t lb_bytes(const pfg_handle *h) {
  return 2 * (h->inst.back().fblk0 + h->inst.back().nfblk) * Q * XBLOCK * (int64_t)h->esize;
}

static bool lb_cached(const pfg_handle *h) { return lb_bytes(h) <= LB_CACHED_MAX_BYTES; }

int lb_default_xcd_rows(const pfg_handle *h) {
  return lb_bytes(h) <= LB_XCD_MAX_BYTES || (h->K == 1 && h->N >= LB_LARGE_CELLS) ? 1 : 0;
}

/* Arguments of lattice k of the handle, starting from copy `cur` of f. */
void make_lb_args(const pfg_handle *h, int k, int cur, LBArgs *a) {
  const Inst &L = h->inst[(size_t)k];
  const pfg_params &p = L.p;
  const size_t foff = (size_t)L.fblk0 * Q * XBLOCK * h->esize;
  a->fin = (const char *)h->f[cur] + foff;
  a->fout = (char *)h->f[1 - cur] + foff;
  a->aux = h->aux + L.cell0;
  a->plane = h->plane;
  a->vel = h->vel + L.cell0;
  a->tile_stamp = h->tile_stamp + L.tile0;
  a->solid = h->solid ? h->solid + L.cell0 : nullptr;
  a->bbmask = h->bbmask ? h->bbmask + L.cell0 : nullptr;
  a->halt = h->halt_on_detach ? h->m.counters + 1 : nullptr;
  a->row_stamp = h->row_stamp ? h->row_stamp + L.fblk0 : nullptr;
  a->step = h->m.d_step;
  a->nx = p.nx;
  a->ny = p.ny;
  a->nz = p.nz;
  a->block_kind = h->block_kind ? h->block_kind + L.fblk0 : nullptr;
  a->ncell = (uint32_t)L.N;
  a->inv_nx = 1.0f / (float)p.nx;
  a->inv_ny = 1.0f / (float)p.ny;
  a->block0 = L.lb_block0;
  a->tnx = L.tnx;
  a->tny = L.tny;
  for (int ax = 0; ax < 3; ++ax) a->periodic[ax] = p.wall[ax] == PFG_WALL_PERIODIC;
  a->omega = 1.0f / p.tau;
  a->guo = 1.0f - 0.5f / p.tau;
  for (int ax = 0; ax < 3; ++ax) a->g[ax] = p.body_force[ax];
  if (h->p.store == PFG_STORE_F16) {
    a->scale = ldexpf(1.0f, h->p.f16_scale_log2);
    a->inv_scale = ldexpf(1.0f, -h->p.f16_scale_log2);
  } else {
    a->scale = 1.0f;
    a->inv_scale = 1.0f;
  }
  a->keep = 1.0f - a->omega;
  a->om15 = 1.5f * a->omega;
  a->om45 = 4.5f * a->omega;
  a->om3 = 3.0f * a->omega;
  a->guo3 = 3.0f * a->guo;
  const int rep[3] = {0, 1, 7}; /* rest, axis, diagonal */
  for (int c = 0; c < 3; ++c) {
    a->ws[c] = weight(rep[c]) * a->scale;
    a->gB[c] = 9.0f * a->guo * a->ws[c];
    a->gD[c] = 3.0f * a->guo * a->ws[c];
  }
  /* halfway bounce-back with a moving wall (Ladd): the population entering
   * from the wall is f_bb(d) + 6 w_d rho_w (c_d . u_w), rho_w = 1; in the
   * storage units of the format */
  a->wall_moves = 0;
  for (int ax = 0; ax < 3; ++ax)
    for (int s = 0; s < 2; ++s)
      for (int d = 0; d < Q; ++d) {
        const float *u = s == 0 ? p.wall_u_lo[ax] : p.wall_u_hi[ax];
        const float cu = CX[d] * u[0] + CY[d] * u[1] + CZ[d] * u[2];
        a->wall_term[ax][s][d] = 6.0f * weight(d) * cu * a->scale;
        a->wall_moves |= a->wall_term[ax][s][d] != 0.0f;
      }
  a->zvel = p.wall[2] == PFG_WALL_VELOCITY ? 1 : 0;
  a->xcd_rows = h->lb_xcd_rows;
  for (int k = 0; k < 3; ++k) {
    a->zvel_u[0][k] = p.wall_u_lo[2][k];
    a->zvel_u[1][k] = p.wall_u_hi[2][k];
  }
}

template <int S, int CPT, int MODE, int WAVES>
static hipError_t launch_fused(const LBArgs &a, hipStream_t st) {
  constexpr int PER = 4 * XBLOCK * CPT; /* cells per workgroup */
  const dim3 grid((unsigned)(((int64_t)a.ncell + PER - 1) / PER));
  if (a.zvel)
    hipLaunchKernelGGL((lb_fused_kernel<S, CPT, MODE | LB_ZVEL, WAVES>), grid, dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((lb_fused_kernel<S, CPT, MODE, WAVES>), grid, dim3(256), 0, st, a);
  return hipGetLastError();
}

/* Which variant a step takes (LB-only launches, us, on one card):
 * - Both copies within LB_CACHED_MAX_BYTES: stores through the caches, the
 *   next step then reads from the 256 MB cache in front of HBM.  Streamed /
 *   cached: 201x99x75 FP32 (226 MB) 43 / 34, 128^3 FP16 (160 MB) 30.6 / 26,
 *   128^3 FP32 and 256x128x128 FP16 (319 MB) 56 / 52 and 55.7 / 54, but
 *   160x128x128 FP32 (398 MB) 70 / 72, 200^3 FP16 (608 MB) 102 / 107.
 * - XCD order (lb_default_xcd_rows) where they fit that cache, each XCD's
 *   range then mostly its own L2's: hardware / XCD order 201x99x75 FP32
 *   34 / 30, 150x75x67 19.3 / 17.2, but 256x128x128 108 / 114; and from
 *   LB_LARGE_CELLS up, where the order keeps the reads of neighbouring planes
 *   in one L2: 1024x512x512 FP32 7350 / 6720, FP16 3370 / 3330.
 * - Wavefronts per SIMD: fewer resident wavefronts walk fewer DRAM pages at
 *   once.  8 / 6 / 4: FP32 512x256x256 896 / 890 / 868, its tube 630 / 631 /
 *   587; 1024x512x512 FP32 7150 / 6700 / 6690, FP16 3510 / 3330 / 3560,
 *   FP16 512x256x256 427 / 415 / 431. */
template <int S>
static hipError_t launch_lb_s(const pfg_handle *h, const LBArgs &a, int mode, hipStream_t st) {
  switch (mode) {
    case LB_MODE_BULK: return launch_fused<S, 1, LB_MODE_BULK, 6>(a, st);
    case LB_MODE_REGION: return launch_fused<S, 1, LB_MODE_REGION, 6>(a, st);
  }
  if (h->lb_cpt == 2) return launch_fused<S, 2, LB_MODE_STEP, 6>(a, st);
  if (h->lb_cpt == 4) return launch_fused<S, 4, LB_MODE_STEP, 6>(a, st);
  if (lb_cached(h))
    return launch_fused<S, 1, LB_MODE_STEP | LB_CACHED, 6>(a, st);
  if constexpr (S == PFG_STORE_F32)
    if (a.ncell < LB_LARGE_CELLS)
      return launch_fused<S, 1, LB_MODE_STEP, 4>(a, st);
  return launch_fused<S, 1, LB_MODE_STEP, 6>(a, st);
}

static hipError_t dispatch_lb(pfg_handle *h, int mode, hipStream_t st) {
  LBArgs a;
  make_lb_args(h, 0, h->cur, &a);
  switch (h->p.store) {
    case PFG_STORE_F16: return launch_lb_s<PFG_STORE_F16>(h, a, mode, st);
    case PFG_STORE_BF16: return launch_lb_s<PFG_STORE_BF16>(h, a, mode, st);
    default: return launch_lb_s<PFG_STORE_F32>(h, a, mode, st);
  }
}

/* Resident workgroups of the persistent batched launch: what the CUs hold at
 * once (occupancy x CUs), at most the tasks there are. */
template <class KER>
static unsigned queue_grid(pfg_handle *h, KER kernel) {
  int per_cu = 0, cus = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, 256, 0) != hipSuccess ||
      per_cu <= 0)
    per_cu = 4;
  if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, h->device) !=
          hipSuccess ||
      cus <= 0)
    cus = 256;
  const int64_t g = std::min<int64_t>((int64_t)per_cu * cus, h->lb_blocks);
  return (unsigned)std::max<int64_t>(g, 1);
}

template <int S, int CPT, int MODE>
static void launch_batch(pfg_handle *h, hipStream_t st) {
  const uint32_t ntasks = (uint32_t)h->lb_blocks;
  const dim3 grid((ntasks + CPT - 1) / CPT), block(256);
  const LBArgs *args = h->d_lbargs[h->cur];
  const bool zvel = h->p.wall[2] == PFG_WALL_VELOCITY; /* the lattices of a batch share the walls */
  if (CPT == 1 && h->lb_persistent && MODE == LB_MODE_STEP && h->lb_queue) {
    if (zvel) {
      auto k = lb_batch_queue_kernel<S, MODE | LB_ZVEL>;
      hipLaunchKernelGGL(k, dim3(queue_grid(h, k)), block, 0, st, args, h->lb_block_inst, ntasks,
                         h->lb_queue);
    } else {
      auto k = lb_batch_queue_kernel<S, MODE>;
      hipLaunchKernelGGL(k, dim3(queue_grid(h, k)), block, 0, st, args, h->lb_block_inst, ntasks,
                         h->lb_queue);
    }
    return;
  }
  const int xcd = h->lb_xcd_rows;
  if (CPT == 1 && MODE == LB_MODE_STEP && !zvel && lb_cached(h))
    hipLaunchKernelGGL((lb_batch_kernel<S, 1, LB_MODE_STEP | LB_CACHED>), grid, block, 0, st, args,
                       h->lb_block_inst, ntasks, xcd);
  else if (zvel)
    hipLaunchKernelGGL((lb_batch_kernel<S, CPT, MODE | LB_ZVEL>), grid, block, 0, st, args,
                       h->lb_block_inst, ntasks, xcd);
  else
    hipLaunchKernelGGL((lb_batch_kernel<S, CPT, MODE>), grid, block, 0, st, args,
                       h->lb_block_inst, ntasks, xcd);
}

template <int S>
static hipError_t launch_lb_batch_s(pfg_handle *h, int mode, hipStream_t st) {
  switch (mode) {
    case LB_MODE_BULK: launch_batch<S, 1, LB_MODE_BULK>(h, st); break;
    case LB_MODE_REGION: launch_batch<S, 1, LB_MODE_REGION>(h, st); break;
    default: /* the persistent launch takes its blocks one at a time */
      switch (h->lb_persistent ? 1 : h->lb_cpt) {
        case 2: launch_batch<S, 2, LB_MODE_STEP>(h, st); break;
        case 4: launch_batch<S, 4, LB_MODE_STEP>(h, st); break;
        default: launch_batch<S, 1, LB_MODE_STEP>(h, st);
      }
  }
  return hipGetLastError();
}

/* All lattices of a batch in one launch. */
static hipError_t launch_lb_batch(pfg_handle *h, int mode, hipStream_t st) {
  switch (h->p.store) {
    case PFG_STORE_F16: return launch_lb_batch_s<PFG_STORE_F16>(h, mode, st);
    case PFG_STORE_BF16: return launch_lb_batch_s<PFG_STORE_BF16>(h, mode, st);
    default: return launch_lb_batch_s<PFG_STORE_F32>(h, mode, st);
  }
}

hipError_t launch_lb(pfg_handle *h) {
  hipError_t e = h->K > 1 ? launch_lb_batch(h, LB_MODE_STEP, h->stream)
                          : dispatch_lb(h, LB_MODE_STEP, h->stream);
  if (e == hipSuccess) h->cur = 1 - h->cur;
  return e;
}

hipError_t launch_lb_part(pfg_handle *h, int part, hipStream_t st) {
  if (!h->row_stamp) return hipErrorInvalidValue;
  const int mode = part == 1 ? LB_MODE_BULK : LB_MODE_REGION;
  hipError_t e = h->K > 1 ? launch_lb_batch(h, mode, st)
                          : dispatch_lb(h, mode, st);
  if (e == hipSuccess && part == 2) h->cur = 1 - h->cur;
  return e;
}

hipError_t launch_bbmask(pfg_handle *h, int k) {
  if (!h->solid || !h->bbmask) return hipSuccess;
  LBArgs a;
  make_lb_args(h, k, h->cur, &a);
  const Inst &L = h->inst[(size_t)k];
  hipLaunchKernelGGL(bbmask_kernel, dim3((unsigned)((L.N + 255) / 256)), dim3(256), 0,
                     h->stream, a, a.solid, h->bbmask + L.cell0);
  hipLaunchKernelGGL(block_kind_kernel, dim3((unsigned)((L.N + 255) / 256)), dim3(256), 0,
                     h->stream, h->bbmask + L.cell0, a.ncell, h->block_kind + L.fblk0);
  return hipGetLastError();
}

hipError_t launch_init_eq(pfg_handle *h, int k, const float *rho, const float *ux,
                          const float *uy, const float *uz, bool per_z) {
  LBArgs a;
  make_lb_args(h, k, 0, &a);
  const int64_t n = h->inst[(size_t)k].N;
  void *d0 = (void *)a.fin, *d1 = a.fout; /* both copies of lattice k */
  dim3 block(256), grid((unsigned)((n + 255) / 256));
  switch (h->p.store) {
    case PFG_STORE_F16:
      hipLaunchKernelGGL(init_eq_kernel<PFG_STORE_F16>, grid, block, 0, h->stream, a, d0, d1,
                         rho, ux, uy, uz, n, per_z ? 1 : 0);
      break;
    case PFG_STORE_BF16:
      hipLaunchKernelGGL(init_eq_kernel<PFG_STORE_BF16>, grid, block, 0, h->stream, a, d0, d1,
                         rho, ux, uy, uz, n, per_z ? 1 : 0);
      break;
    default:
      hipLaunchKernelGGL(init_eq_kernel<PFG_STORE_F32>, grid, block, 0, h->stream, a, d0, d1,
                         rho, ux, uy, uz, n, per_z ? 1 : 0);
  }
  return hipGetLastError();
}

/* [19][N] full f of a single-lattice handle to or from the current copy. */
hipError_t launch_convert_f(pfg_handle *h, float *f_out, const float *f_in) {
  LBArgs a;
  make_lb_args(h, 0, h->cur, &a);
  const int64_t n = h->N;
  float *buf = nullptr;
  hipError_t e = hipMalloc(&buf, sizeof(float) * (size_t)n);
  if (e != hipSuccess) return e;
  dim3 block(256), grid((unsigned)((n + 255) / 256));
  void *stored = h->f[h->cur];
  for (int d = 0; d < Q && e == hipSuccess; ++d) {
    const int to_float = f_out != nullptr;
    if (!to_float) {
      e = hipMemcpyAsync(buf, f_in + (int64_t)d * n, sizeof(float) * n, hipMemcpyHostToDevice,
                         h->stream);
      if (e != hipSuccess) break;
    }
    switch (h->p.store) {
      case PFG_STORE_F16:
        hipLaunchKernelGGL(convert_plane_kernel<PFG_STORE_F16>, grid, block, 0, h->stream, a,
                           stored, buf, d, to_float, n);
        break;
      case PFG_STORE_BF16:
        hipLaunchKernelGGL(convert_plane_kernel<PFG_STORE_BF16>, grid, block, 0, h->stream, a,
                           stored, buf, d, to_float, n);
        break;
      default:
        hipLaunchKernelGGL(convert_plane_kernel<PFG_STORE_F32>, grid, block, 0, h->stream, a,
                           stored, buf, d, to_float, n);
    }
    e = hipGetLastError();
    if (e != hipSuccess) break;
    if (to_float) {
      e = hipMemcpyAsync(f_out + (int64_t)d * n, buf, sizeof(float) * n, hipMemcpyDeviceToHost,
                         h->stream);
    }
    if (e == hipSuccess) e = hipStreamSynchronize(h->stream);
  }
  hipFree(buf);
  return e;
}

hipError_t launch_conservation(pfg_handle *h, int k, double out[4]) {
  LBArgs a;
  make_lb_args(h, k, h->cur, &a);
  const int64_t n = h->inst[(size_t)k].N;
  const int blocks = (int)std::min<int64_t>(h->red_blocks, (n + 255) / 256);
  switch (h->p.store) {
    case PFG_STORE_F16:
      hipLaunchKernelGGL(conservation_kernel<PFG_STORE_F16>, dim3(blocks), dim3(256), 0,
                         h->stream, a, a.fin, h->red, n);
      break;
    case PFG_STORE_BF16:
      hipLaunchKernelGGL(conservation_kernel<PFG_STORE_BF16>, dim3(blocks), dim3(256), 0,
                         h->stream, a, a.fin, h->red, n);
      break;
    default:
      hipLaunchKernelGGL(conservation_kernel<PFG_STORE_F32>, dim3(blocks), dim3(256), 0,
                         h->stream, a, a.fin, h->red, n);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  std::vector<double> part((size_t)blocks * 4);
  e = hipMemcpyAsync(part.data(), h->red, sizeof(double) * part.size(), hipMemcpyDeviceToHost,
                     h->stream);
  if (e != hipSuccess) return e;
  e = hipStreamSynchronize(h->stream);
  if (e != hipSuccess) return e;
  for (int c = 0; c < 4; ++c) out[c] = 0.0;
  for (int b = 0; b < blocks; ++b)
    for (int c = 0; c < 4; ++c) out[c] += part[4 * (size_t)b + c];
  return hipSuccess;
}

}  // namespace pfg
