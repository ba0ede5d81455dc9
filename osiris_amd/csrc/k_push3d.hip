// k_push3d.hip -- fused 3D push + deposit with compile-time tile shape.
//
// One workgroup of 4 waves (cubic splines) or 8 per (species, tile).  Compared with the
// generic 3D kernel in k_tiles.hip:
//  * TX/TY/TZ are template parameters, so the LDS pitches of the staged field and current
//    tiles are constants and every stencil offset is an immediate (the generic kernel
//    adds runtime row and plane pitches for each of the 4 x 4 lines of a cubic stencil,
//    about 400 VALU instructions per 64 particles in the gather alone);
//  * particle and mover arrays are addressed through global-address-space pointers with
//    scalar bases and 32-bit offsets;
//  * the particle loads of the next iteration are issued before the current particle is
//    processed;
//  * a particle that stays in its cell is deposited from registers; one that crosses a face
//    is queued in LDS, and the waves split and deposit 64 of them at a time (their third and
//    fourth virtual particles go back into the queue, so they run on full waves too).
//  * with cubic splines the lanes of a deposit are permuted first, so that the 64-bit adds of a
//    16-lane group mostly fall into different banks (spread_lanes).
// What bounds it: LDS.  Per 64 particles the cubic gather makes 192 paired 4-byte reads, whose
// lanes conflict through their half-cell shifts (9 cycles of a CU each, 5 without conflicts),
// and the deposit 161 64-bit adds (11 cycles each as the particles come, some 9 on permuted
// lanes, 7.4 without conflicts): about 90% of the cycles on 192^3, 8 per cell.  The permutation
// takes 11 crossbar operations and the splines once more, and 6.4 ms became 6.0; quadratic
// splines gain nothing from it (96^3, two beams of 4: 27.9 ms per 40 steps either way), linear
// ones lose (52x44x36: 2.70 -> 2.80 ms).  Linear and quadratic splines have room for
// 8 waves in 128 registers, 4 per SIMD instead of 2: 52x44x36 linear 34 -> 29.6 us, 96^3
// quadratic, two beams of 4, 464 -> 428 us; cubic spills there and gains nothing.
// The arithmetic (gather line/plane order, pusher, position advance, split, deposit) is
// the generic kernel's, operation for operation, so the results are bit-identical.
#include <type_traits>

#include "osr_device.hpp"
#include "osr_types.hpp"

namespace osr {

typedef __attribute__((address_space(3))) const float lcf32;

// LDS pointer to element `elem` of the LDS array `base`, made opaque to the compiler: the
// loads of one stencil line then share this one base register and carry their small
// constant offsets in the instruction (ds_read2_b32 offsets are 8 bits of dwords).  Left
// visible, the array's absolute LDS address is folded into every constant, which no
// longer fits, and a paired load costs one more address add.  The empty asm emits no
// instruction.
OSR_DEV lcf32* lds_line(const float* base, int elem) {
  unsigned a = (unsigned)(size_t)(lcf32*)base + 4u * (unsigned)elem;
  asm("" : "+v"(a));
  return (lcf32*)(size_t)a;
}

// A permutation of the lanes (the lane whose values each lane takes) that spreads the lanes
// with `on` over the 16-lane groups in which LDS makes 64-bit adds: lane 16 k + r takes the
// k-th one whose `res` (its base node mod 16, the pair of banks its adds fall into) is r, and
// what is over four of a kind fills the lanes left free.  Every lane is some lane's source.
OSR_DEV int spread_lanes(bool on, int res, int lane) {
  const unsigned long long m = __ballot(on);
  const unsigned long long b0 = __ballot(res & 1), b1 = __ballot(res & 2), b2 = __ballot(res & 4),
                           b3 = __ballot(res & 8);
  auto kind = [&](int v) {  // the lanes with `on` and residue v
    return m & (v & 1 ? b0 : ~b0) & (v & 2 ? b1 : ~b1) & (v & 4 ? b2 : ~b2) & (v & 8 ? b3 : ~b3);
  };
  const unsigned long long below = (1ull << lane) - 1ull;
  const int rank = __popcll(kind(res) & below);
  const bool placed = on && rank < 4;
  const bool taken = __popcll(kind(lane & 15)) > (lane >> 4);
  const unsigned long long mp = __ballot(placed), fr = ~__ballot(taken);
  // the lanes not placed, in order, those with `on` first
  const unsigned long long ov = m & ~mp, id = ~m;
  const int nov = __popcll(ov), rest = nov + __popcll(id);
  const int idx = on ? (placed ? rest + __popcll(mp & below) : __popcll(ov & below))
                     : nov + __popcll(id & below);
  const int order = __builtin_amdgcn_ds_permute(idx << 2, lane);
  // every lane not placed sends to a free lane, whose value is not used
  const int spare = fr ? __ffsll((long long)fr) - 1 : 0;
  const int from = __builtin_amdgcn_ds_permute((placed ? 16 * rank + res : spare) << 2, lane);
  const int fill = __builtin_amdgcn_ds_bpermute(__popcll(fr & below) << 2, order);
  return taken ? from : fill;
}

OSR_DEV float lane_from(float v, int src) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(v)));
}

template <int ORDER, int TX, int TY, int TZ>
struct Tile3 {
  using O = Ord<ORDER>;
  static constexpr int GX = TX + O::GLO + O::GHI, GY = TY + O::GLO + O::GHI,
                       GZ = TZ + O::GLO + O::GHI;
  static constexpr int JX = TX + O::JLO + O::JHI, JY = TY + O::JLO + O::JHI,
                       JZ = TZ + O::JLO + O::JHI;
  // LDS pitches of the staged fields: rows of RS floats, planes of GXY floats.  For 8x8
  // tiles 12 and 144 (padded for orders 1 and 2): the 4x4x2 cell block of a half wave
  // (cell_key) then starts its stencils in 32 distinct banks.
  static constexpr int RS = (TX == 8 && GX <= 12) ? 12 : GX;
  static constexpr int GYP = (TY == 8 && GY <= 12) ? 12 : GY;
  static constexpr int GXY = RS * GYP, GN = GXY * GZ;
  // planes of the current padded where LDS has room (13 x 13 nodes for cubic splines): 8%
  // fewer bank conflicts of the 64-bit adds in a model of the particle order
  static constexpr int JXY = JX * JY + (JX == 13 ? 5 : 0), JN = JXY * JZ;
  static constexpr bool SPREAD = ORDER == 3;
  static constexpr int NW = push3d_waves(ORDER), NT = 64 * NW, QC = 64;
};

template <int ORDER, int PUSHER, int TX, int TY, int TZ>
__global__ __launch_bounds__(64 * push3d_waves(ORDER), push3d_waves(ORDER) / 2) void push_deposit_3d_t(const SpecDesc* __restrict__ descs,
                                                            const int2* __restrict__ work) {
  using O = Ord<ORDER>;
  using T = Tile3<ORDER, TX, TY, TZ>;
  constexpr int NP = O::NP;
  constexpr int GX = T::GX, GY = T::GY, GZ = T::GZ, RS = T::RS, GXY = T::GXY, GN = T::GN;
  constexpr int JX = T::JX, JY = T::JY, JXY = T::JXY, JN = T::JN;
  constexpr int NT = T::NT, NW = T::NW, QC = T::QC;
  __shared__ float sF[6 * GN];
  __shared__ unsigned long long sJ[3 * JN];
  // queued particles: (x0, y0, z0, q), (x1, y1, z1, node and cell shifts)
  __shared__ f32x4 sQ[NW][2][QC];
  __shared__ int sQn[NW];
  static_assert((TX & (TX - 1)) == 0 && (TY & (TY - 1)) == 0 && (TZ & (TZ - 1)) == 0,
                "tile sides are powers of two");
  __shared__ double s_ene[NW];

  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (g.ctrl->halt != 0) return;
  const int tile = wk.y;
  const int ttx = tile % g.ntx, tty = (tile / g.ntx) % g.nty, ttz = tile / (g.ntx * g.nty);
  const int cx0 = ttx * TX, cy0 = tty * TY, cz0 = ttz * TZ;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const long long nc = g.ncell;

  {
    const gf32* __restrict__ E = (const gf32*)g.E;
    const gf32* __restrict__ B = (const gf32*)g.B;
    for (int i = threadIdx.x; i < GX * GY * GZ; i += NT) {
      const int lx = i % GX, ly = (i / GX) % GY, lz = i / (GX * GY);
      const int gx = wrapi(cx0 + lx - O::GLO, nx), gy = wrapi(cy0 + ly - O::GLO, ny),
                gz = wrapi(cz0 + lz - O::GLO, nz);
      const long long gi = gx + (long long)nx * (gy + (long long)ny * gz);
      const int li = lz * GXY + ly * RS + lx;
#pragma unroll
      for (int c = 0; c < 3; c++) {
        sF[c * GN + li] = E[c * nc + gi];
        sF[(3 + c) * GN + li] = B[c * nc + gi];
      }
    }
  }
  for (int i = threadIdx.x; i < 3 * JN; i += NT) sJ[i] = 0ull;
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int base = __builtin_amdgcn_readfirstlane(d.off[tile]);
  const int n = __builtin_amdgcn_readfirstlane(d.cnt[tile]);
  const int per_wave = ((n + NT - 1) / NT) * 64;
  const int w0 = wave * per_wave;
  const int w1 = min(w0 + per_wave, n);
  const float tem = d.tem;
  const float dtdx1 = g.dt_dx[0], dtdx2 = g.dt_dx[1], dtdx3 = g.dt_dx[2];
  const float jn1 = g.jnorm[0], jn2 = g.jnorm[1], jn3 = g.jnorm[2];
  const double jscale = g.jscale;
  const gu32* __restrict__ Pcell = (const gu32*)d.cell + base;
  const gf32* __restrict__ Px = (const gf32*)d.x + base;
  const gf32* __restrict__ Py = (const gf32*)d.y + base;
  const gf32* __restrict__ Pz = (const gf32*)d.z + base;
  const gf32* __restrict__ Pux = (const gf32*)d.ux + base;
  const gf32* __restrict__ Puy = (const gf32*)d.uy + base;
  const gf32* __restrict__ Puz = (const gf32*)d.uz + base;
  const gf32* __restrict__ Pq = (const gf32*)d.q + base;
  const gu32* __restrict__ Ppid = (const gu32*)d.pid + base;
  gu32* __restrict__ Wcell = (gu32*)d.cell + base;
  gf32* __restrict__ Wx = (gf32*)d.x + base;
  gf32* __restrict__ Wy = (gf32*)d.y + base;
  gf32* __restrict__ Wz = (gf32*)d.z + base;
  gf32* __restrict__ Wux = (gf32*)d.ux + base;
  gf32* __restrict__ Wuy = (gf32*)d.uy + base;
  gf32* __restrict__ Wuz = (gf32*)d.uz + base;
  gu32* __restrict__ Mcell = (gu32*)d.mcell + base;
  gf32* __restrict__ Mx = (gf32*)d.mx + base;
  gf32* __restrict__ My = (gf32*)d.my + base;
  gf32* __restrict__ Mz = (gf32*)d.mz + base;
  gf32* __restrict__ Mux = (gf32*)d.mux + base;
  gf32* __restrict__ Muy = (gf32*)d.muy + base;
  gf32* __restrict__ Muz = (gf32*)d.muz + base;
  gf32* __restrict__ Mq = (gf32*)d.mq + base;
  gu32* __restrict__ Mpid = (gu32*)d.mpid + base;
  gi32* __restrict__ Midx = (gi32*)d.midx + base;

  double ene = 0.0;
  int mcount = 0;
  bool bad = false;
  // cells of the tile inside the grid; a particle that leaves them changes tile, unless the
  // tile is the only one of a direction (it wraps into itself)
  const int tcx = min(TX, nx - cx0), tcy = min(TY, ny - cy0), tcz = min(TZ, nz - cz0);
  const bool lone = g.ntx == 1 || g.nty == 1 || g.ntz == 1;
  const uint32_t cell0 = pack3(cx0, cy0, cz0);
  constexpr uint32_t kIn = pack3(TX - 1, TY - 1, TZ - 1);

  // the wave's particles; RAW: how the deposit adds (fix_bits)
  auto push_all = [&](auto raw) {
    constexpr bool RAW = decltype(raw)::value;
    int qlen = 0;
    f32x4* const Q0 = sQ[wave][0];
    f32x4* const Q1 = sQ[wave][1];
    const unsigned long long below = (1ull << lane) - 1ull;
    // split and deposit of queued particles, one per lane (on: the lane holds one, (a, b));
    // virtual particles 2 and 3 are queued again, as particles that cross nothing
    auto deposit_queue = [&](bool on, const f32x4& a, const f32x4& b) {
      VP3 vp[4];
      int nvp = 0, nb0 = 0;
      if (on) {
        const int code = __float_as_int(b.w);
        nb0 = code >> 6;
        nvp = split3d(a.x, a.y, a.z, b.x, b.y, b.z, (code & 3) - 1, ((code >> 2) & 3) - 1,
                      ((code >> 4) & 3) - 1, a.w, vp);
      }
      const unsigned long long m2 = __ballot(nvp > 2), m3 = __ballot(nvp > 3);
      const int n2 = __popcll(m2), again = n2 + __popcll(m3);
      const bool requeue = again <= QC / 2;  // else deposited here, on partly idle waves
      const int nv = requeue ? 2 : 4;
#pragma unroll 1
      for (int v = 0; v < nv; v++) {
        if (v < nvp) {
          const VP3 V = pick(vp, v);
          float S0x[NP], S0y[NP], S0z[NP];
          spline<ORDER>(V.x0, S0x);
          spline<ORDER>(V.y0, S0y);
          spline<ORDER>(V.z0, S0z);
          dep_vp3<ORDER, RAW>(sJ, JN, S0x, S0y, S0z, V.x0, V.y0, V.z0, V.x1, V.y1, V.z1, V.q,
                              nb0 + V.dk * JXY + V.dj * JX + V.di, JX, JXY, jn1, jn2, jn3, jscale);
        }
      }
      qlen = 0;
      if (requeue && again > 0) {
        auto put = [&](int s, const VP3& V) {
          Q0[s] = f32x4{V.x0, V.y0, V.z0, V.q};
          Q1[s] = f32x4{V.x1, V.y1, V.z1,
                        __int_as_float((nb0 + V.dk * JXY + V.dj * JX + V.di) * 64 + 1 + 4 + 16)};
        };
        if (nvp > 2) put(__popcll(m2 & below), vp[2]);
        if (nvp > 3) put(n2 + __popcll(m3 & below), vp[3]);
        qlen = again;
      }
    };
    uint32_t f_cell = 0, f_pid = 0;
    float f_x = 0.f, f_y = 0.f, f_z = 0.f, f_u1 = 0.f, f_u2 = 0.f, f_u3 = 0.f, f_q = 0.f;
    // lanes past the end load the last particle again and are masked below
    auto prefetch = [&](int pf) {
      const unsigned upf = (unsigned)min(pf, w1 - 1);
      f_cell = *el(Pcell, upf);
      f_x = *el(Px, upf);
      f_y = *el(Py, upf);
      f_z = *el(Pz, upf);
      f_u1 = *el(Pux, upf);
      f_u2 = *el(Puy, upf);
      f_u3 = *el(Puz, upf);
      f_q = *el(Pq, upf);
      f_pid = *el(Ppid, upf);
    };
    if (w0 < w1) prefetch(w0 + lane);
    for (int p0 = w0; p0 < w1; p0 += 64) {
      const int p = p0 + lane;
      const unsigned up = (unsigned)p;
      const uint32_t cell = f_cell, pid = f_pid;
      const float x = f_x, y = f_y, z = f_z, q = f_q;
      float u1 = f_u1, u2 = f_u2, u3 = f_u3;
      if (p0 + 64 < w1) prefetch(p + 64);
      // cell within the tile: every field of the difference in range (a borrow shows too)
      const uint32_t dl = cell - cell0;
      const bool out = (dl & ~kIn) != 0u;
      const bool act = p < w1 && !out;
      bad |= p < w1 && out;
      int lx, ly, lz;
      unpack3(dl & kIn, lx, ly, lz);
      float wx[NP], wy[NP], wz[NP], wxh[NP], wyh[NP], wzh[NP];
      spline<ORDER>(x, wx);
      spline<ORDER>(y, wy);
      spline<ORDER>(z, wz);
      splineh<ORDER>(x, x < 0.f ? 1.f : 0.f, wxh);
      splineh<ORDER>(y, y < 0.f ? 1.f : 0.f, wyh);
      splineh<ORDER>(z, z < 0.f ? 1.f : 0.f, wzh);
      // stencil origins (full and half-shifted) as LDS element offsets
      const int g0 = (lz + O::GLO + O::LP) * GXY + (ly + O::GLO + O::LP) * RS + lx + O::GLO + O::LP;
      const int hx = x < 0.f ? 1 : 0, hy = y < 0.f ? RS : 0, hz = z < 0.f ? GXY : 0;
      const int oE1 = g0 - hx, oE2 = GN + g0 - hy, oE3 = 2 * GN + g0 - hz;
      const int oB1 = 3 * GN + g0 - hy - hz, oB2 = 4 * GN + g0 - hx - hz, oB3 = 5 * GN + g0 - hx - hy;
      // GET_EMF_3D line/plane order (os-emf-interpolate.f03:697-773): fma along k1, then k2,
      // then k3
      float e1 = 0.f, e2 = 0.f, e3 = 0.f;
#pragma unroll
      for (int k3 = 0; k3 < NP; k3++) {
        float p1 = 0.f, p2 = 0.f, p3 = 0.f;
        lcf32* L1 = lds_line(sF, oE1 + k3 * GXY);
        lcf32* L2 = lds_line(sF, oE2 + k3 * GXY);
        lcf32* L3 = lds_line(sF, oE3 + k3 * GXY);
#pragma unroll
        for (int k2 = 0; k2 < NP; k2++) {
          float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
          for (int k1 = 0; k1 < NP; k1++) {
            const int o = k2 * RS + k1;
            l1 = fma_(L1[o], wxh[k1], l1);
            l2 = fma_(L2[o], wx[k1], l2);
            l3 = fma_(L3[o], wx[k1], l3);
          }
          p1 = fma_(l1, wy[k2], p1);
          p2 = fma_(l2, wyh[k2], p2);
          p3 = fma_(l3, wy[k2], p3);
        }
        e1 = fma_(p1, wz[k3], e1);
        e2 = fma_(p2, wz[k3], e2);
        e3 = fma_(p3, wzh[k3], e3);
      }
      float b1 = 0.f, b2 = 0.f, b3 = 0.f;
#pragma unroll
      for (int k3 = 0; k3 < NP; k3++) {
        float p1 = 0.f, p2 = 0.f, p3 = 0.f;
        lcf32* L1 = lds_line(sF, oB1 + k3 * GXY);
        lcf32* L2 = lds_line(sF, oB2 + k3 * GXY);
        lcf32* L3 = lds_line(sF, oB3 + k3 * GXY);
#pragma unroll
        for (int k2 = 0; k2 < NP; k2++) {
          float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
          for (int k1 = 0; k1 < NP; k1++) {
            const int o = k2 * RS + k1;
            l1 = fma_(L1[o], wx[k1], l1);
            l2 = fma_(L2[o], wxh[k1], l2);
            l3 = fma_(L3[o], wxh[k1], l3);
          }
          p1 = fma_(l1, wyh[k2], p1);
          p2 = fma_(l2, wy[k2], p2);
          p3 = fma_(l3, wyh[k2], p3);
        }
        b1 = fma_(p1, wzh[k3], b1);
        b2 = fma_(p2, wzh[k3], b2);
        b3 = fma_(p3, wz[k3], b3);
      }
      const float ke = push<PUSHER>(tem, e1, e2, e3, b1, b2, b3, u1, u2, u3);
      ene = __builtin_fma((double)(act ? q : 0.f), (double)ke, ene);
      const float rg = rgamma(u1, u2, u3);
      const float x1 = fma_(u1 * rg, dtdx1, x), y1 = fma_(u2 * rg, dtdx2, y),
                  z1 = fma_(u3 * rg, dtdx3, z);
      const float tx = trim(x1), ty = trim(y1), tz = trim(z1);
      const int dix = (int)tx, diy = (int)ty, diz = (int)tz;
      const int nb0 =
          (lz + O::LP + O::JLO) * JXY + (ly + O::LP + O::JLO) * JX + lx + O::LP + O::JLO;
      const bool cross = act && (dix | diy | diz) != 0;
      const f32x4 qa = {x, y, z, q};
      const f32x4 qb = {x1, y1, z1,
                        __int_as_float(nb0 * 64 + (dix + 1) + 4 * (diy + 1) + 16 * (diz + 1))};
      // ---- store: stay in place, or leave through the mover buffer
      const int nlx = lx + dix, nly = ly + diy, nlz = lz + diz;
      bool stay = (unsigned)nlx < (unsigned)tcx && (unsigned)nly < (unsigned)tcy &&
                  (unsigned)nlz < (unsigned)tcz;
      uint32_t ncell = cell0 + pack3(0, nly, nlz) + (uint32_t)nlx;
      if (lone || !__all(stay || !act)) {
        const int nix = wrap1(nlx + cx0, nx), niy = wrap1(nly + cy0, ny),
                  niz = wrap1(nlz + cz0, nz);
        ncell = pack3(nix, niy, niz);
        stay = (nix / TX + g.ntx * (niy / TY + g.nty * (niz / TZ))) == tile;
      }
      const float xs = x1 - tx, ys = y1 - ty, zs = z1 - tz;
      if (act && stay) {
        *el(Wcell, up) = ncell;
        *el(Wx, up) = xs;
        *el(Wy, up) = ys;
        *el(Wz, up) = zs;
        *el(Wux, up) = u1;
        *el(Wuy, up) = u2;
        *el(Wuz, up) = u3;
      }
      const bool mv = act && !stay;
      const unsigned long long mm = __ballot(mv);
      if (mv) {
        const unsigned slot = (unsigned)(w0 + mcount + __popcll(mm & below));
        *el(Mcell, slot) = ncell;
        *el(Mx, slot) = xs;
        *el(My, slot) = ys;
        *el(Mz, slot) = zs;
        *el(Mux, slot) = u1;
        *el(Muy, slot) = u2;
        *el(Muz, slot) = u3;
        *el(Mq, slot) = q;
        *el(Mpid, slot) = pid;
        *el(Midx, slot) = p;
      }
      mcount += __popcll(mm);
      // ---- deposit of the particles that stay in their cell, with the gather's splines
      const bool in = act && !cross;
      if constexpr (T::SPREAD) {
        const int src = spread_lanes(in, nb0 & 15, lane);
        const float X = lane_from(x, src), Y = lane_from(y, src), Z = lane_from(z, src);
        const float X1 = lane_from(x1, src), Y1 = lane_from(y1, src), Z1 = lane_from(z1, src);
        const float Q = lane_from(q, src);
        const int nb = __builtin_amdgcn_ds_bpermute(src << 2, in ? nb0 : -1);
        if (nb >= 0) {
          float S0x[NP], S0y[NP], S0z[NP];
          spline<ORDER>(X, S0x);
          spline<ORDER>(Y, S0y);
          spline<ORDER>(Z, S0z);
          dep_vp3<ORDER, RAW>(sJ, JN, S0x, S0y, S0z, X, Y, Z, X1, Y1, Z1, Q, nb, JX, JXY, jn1,
                              jn2, jn3, jscale);
        }
      } else if (in) {
        dep_vp3<ORDER, RAW>(sJ, JN, wx, wy, wz, x, y, z, x1, y1, z1, q, nb0, JX, JXY, jn1, jn2,
                            jn3, jscale);
      }
      const unsigned long long mc = __ballot(cross);
      const int add = __popcll(mc);
      // twice at most: what a first call queues again crosses nothing
      while (qlen + add > QC) {
        wave_lds_sync();  // the entries of the other lanes
        const f32x4 a = Q0[lane], b = Q1[lane];
        wave_lds_sync();  // read before any is written again
        deposit_queue(lane < qlen, a, b);
      }
      if (cross) {
        const int s = qlen + __popcll(mc & below);
        Q0[s] = qa;
        Q1[s] = qb;
      }
      qlen += add;
    }
    // What is left in the queues, shared over the waves: a wave queues some 7 of 64 particles
    // and sees a few hundred, so its own queue ends a third full.  At most NW QC entries: one
    // batch per wave.  The second round takes what the first queued again.
    for (;;) {
      if (lane == 0) sQn[wave] = qlen;
      __syncthreads();
      int left = 64 * wave + lane, total = 0, w = 0;  // this lane's entry: `left` of queue w
#pragma unroll
      for (int k = 0; k < NW; k++) {
        const int c = sQn[k];
        total += c;
        if (w == k && left >= c) {
          left -= c;
          w = k + 1;
        }
      }
      const bool on = w < NW;
      const f32x4 a = sQ[on ? w : 0][0][on ? left : 0], b = sQ[on ? w : 0][1][on ? left : 0];
      __syncthreads();  // every wave has its entries before the queues are written again
      if (total == 0) break;
      deposit_queue(on, a, b);
    }
  };
  const bool raw = d.jraw != 0;
  if (raw)
    push_all(std::true_type());
  else
    push_all(std::false_type());

  if (bad) atomicOr(&g.ctrl->error, 1);
  if (lane == 0) d.mv_cnt[tile * NW + wave] = mcount;
  if (threadIdx.x == 0) d.mv_stride[tile] = per_wave;
  ene = wave_sum(ene);
  if (lane == 0) s_ene[wave] = ene;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < NW; w++) t += s_ene[w];
    d.epart[tile] = t;
  }
  gu64* __restrict__ GJ = (gu64*)g.J;
  for (int i = threadIdx.x; i < JX * JY * T::JZ; i += NT) {
    const int lx = i % JX, ly = (i / JX) % JY, lz = i / (JX * JY), li = lx + JX * ly + JXY * lz;
    const int gx = wrapi(cx0 + lx - O::JLO, nx), gy = wrapi(cy0 + ly - O::JLO, ny),
              gz = wrapi(cz0 + lz - O::JLO, nz);
    const long long gi = gx + (long long)nx * (gy + (long long)ny * gz);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const unsigned long long t = sJ[c * JN + li], v = raw ? fix_sum<true>(t) : t;
      if (v) __hip_atomic_fetch_add(&GJ[c * nc + gi], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

#define OSR_INST3(O, P, X, Y, Z) \
  template __global__ void push_deposit_3d_t<O, P, X, Y, Z>(const SpecDesc*, const int2*);
#define OSR_INST3T(X, Y, Z)                                                   \
  OSR_INST3(1, 0, X, Y, Z) OSR_INST3(2, 0, X, Y, Z) OSR_INST3(3, 0, X, Y, Z) \
  OSR_INST3(1, 1, X, Y, Z) OSR_INST3(2, 1, X, Y, Z) OSR_INST3(3, 1, X, Y, Z)
OSR_INST3T(8, 8, 4)
#undef OSR_INST3T
#undef OSR_INST3

}  // namespace osr
