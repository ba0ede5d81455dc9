// k_tiles.hip -- the fused tile kernels of the resident fast path.
//
//   push_deposit_{2d,3d}<ORDER,PUSHER>: one workgroup per (species, tile).  E and B of
//     the tile plus the stencil halo are staged in LDS; every wave walks a contiguous
//     slice of the tile's particles (coalesced SoA loads), gathers from LDS, pushes
//     (Boris or Vay), advances the position, splits the trajectory into virtual
//     particles and deposits them into an LDS current tile with int64 fixed-point
//     atomics.  Integer addition is associative, so the deposited current is bit-for-bit
//     independent of the order in which lanes, waves and workgroups add their share:
//     the reduction is reproducible run to run.  The LDS tile is then added to the global
//     fixed-point J with the periodic wrap (the guard-cell fold of the reference).
//     Particles that stay in the tile are written back in place; leavers go to the
//     wave's region of the mover buffer (ballot-ranked, so the order is deterministic).
//   tile_fill: moves the leavers into their destination tiles, filling the holes they
//     left; a deterministic stable compaction.  A tile that would overflow its capacity
//     is left unchanged and flags the step (Ctrl::halt); the host re-lays the particles
//     out before the next push.
//
// Reference: spec/os-spec-push.f03:1438-1605 (advance_deposit_2d/3d),
// emf/os-emf-interpolate.f03:554-779 (GET_EMF_2D/3D), spec/os-spec-current.f03:659-905,
// 2691-2905 (split + DEP_CURRENT), simd/os-spec-push-avx2.c:471-760 (fused SIMD kernel),
// particles/os-particles.f03:1416-1443 (private J + reduce), spec/os-species.f03:269-441
// (counting sort of particles by cell).
#include <type_traits>

#include "osr_device.hpp"
#include "osr_types.hpp"

namespace osr {

OSR_DEV int wrapi(int i, int n) {
  while (i < 0) i += n;
  while (i >= n) i -= n;
  return i;
}

// Exclusive ranks of PF flags per thread in the order (p, thread), and their total: item p
// of thread t comes after every item p' < p and after item p of the threads below t.  Wave
// ballots and one LDS exchange (two barriers) for all PF; all threads must call it.
template <int NT, int PF>
OSR_DEV void block_rank_multi(const bool (&flag)[PF], int (*s_cnt)[NT / 64], int (&rank)[PF],
                              int& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const unsigned long long below = (1ull << lane) - 1ull;
  int own[PF];
#pragma unroll
  for (int p = 0; p < PF; p++) {
    const unsigned long long m = __ballot(flag[p]);
    own[p] = __popcll(m & below);
    if (lane == 0) s_cnt[p][wave] = __popcll(m);
  }
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int p = 0; p < PF; p++) {
    int before = 0, tp = 0;
    for (int w = 0; w < NT / 64; w++) {
      const int c = s_cnt[p][w];
      if (w < wave) before += c;
      tp += c;
    }
    rank[p] = base + before + own[p];
    base += tp;
  }
  total = base;
  __syncthreads();
}

// ------------------------------------------------------------------------------------
// 2D push + deposit
// ------------------------------------------------------------------------------------
template <int ORDER, int PUSHER, int NT>
__global__ __launch_bounds__(NT) void push_deposit_2d(const SpecDesc* __restrict__ descs,
                                                      const int2* __restrict__ work) {
  using O = Ord<ORDER>;
  constexpr int NP = O::NP;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double s_ene[NT / 64];

  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (g.ctrl->halt != 0) return;
  const int tile = wk.y;
  const int TX = g.tx, TY = g.ty;
  const int GX = TX + O::GLO + O::GHI, GY = TY + O::GLO + O::GHI;
  const int JX = TX + O::JLO + O::JHI, JY = TY + O::JLO + O::JHI;
  const int GN = GX * GY, JN = JX * JY;
  unsigned long long* sJ = (unsigned long long*)smem;      // [3][JN]
  float* sF = (float*)(smem + sizeof(unsigned long long) * 3 * JN);  // E[3][GN], B[3][GN]
  const int cx0 = (tile % g.ntx) * TX, cy0 = (tile / g.ntx) * TY;
  const int nx = g.nx, ny = g.ny;
  const long long nc = g.ncell, co = cur_copy(g);

  for (int i = threadIdx.x; i < GN; i += NT) {
    int gx = wrapi(cx0 + (i % GX) - O::GLO, nx), gy = wrapi(cy0 + (i / GX) - O::GLO, ny);
    long long gi = gx + (long long)nx * gy;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      sF[c * GN + i] = g.E[co + c * nc + gi];
      sF[(3 + c) * GN + i] = g.B[co + c * nc + gi];
    }
  }
  for (int i = threadIdx.x; i < 3 * JN; i += NT) sJ[i] = 0ull;
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int NW = NT / 64;
  const int base = d.off[tile];
  const int n = d.cnt[tile];
  const int per_wave = ((n + NT - 1) / NT) * 64;
  const int w0 = wave * per_wave;
  const int w1 = min(w0 + per_wave, n);
  const float tem = d.tem;
  const float dtdx1 = g.dt_dx[0], dtdx2 = g.dt_dx[1];
  const float jn1 = g.jnorm[0], jn2 = g.jnorm[1];
  const double jscale = g.jscale;
  const float* sE1 = sF;
  const float* sE2 = sF + GN;
  const float* sE3 = sF + 2 * GN;
  const float* sB1 = sF + 3 * GN;
  const float* sB2 = sF + 4 * GN;
  const float* sB3 = sF + 5 * GN;
  unsigned long long* sJ1 = sJ;
  unsigned long long* sJ2 = sJ + JN;
  unsigned long long* sJ3 = sJ + 2 * JN;

  double ene = 0.0;
  int mcount = 0;
  bool bad = false;
  for (int p0 = w0; p0 < w1; p0 += 64) {
    const int p = p0 + lane;
    bool act = p < w1;
    uint32_t cell = 0;
    float x = 0.f, y = 0.f, u1 = 0.f, u2 = 0.f, u3 = 0.f, q = 0.f;
    int lx = 0, ly = 0;
    if (act) {
      const int s = base + p;
      cell = d.cell[s];
      x = d.x[s];
      y = d.y[s];
      u1 = d.ux[s];
      u2 = d.uy[s];
      u3 = d.uz[s];
      q = d.q[s];
      int ix, iy;
      unpack2(cell, ix, iy);
      lx = ix - cx0;
      ly = iy - cy0;
      if (lx < 0 || lx >= TX || ly < 0 || ly >= TY) {
        bad = true;
        act = false;
        lx = ly = 0;
      }
    }
    // ---- gather (GET_EMF_2D, same FMA order as the AVX2 kernel)
    float wx[NP], wy[NP], wxh[NP], wyh[NP];
    spline<ORDER>(x, wx);
    spline<ORDER>(y, wy);
    const float hx = x < 0.f ? 1.f : 0.f, hy = y < 0.f ? 1.f : 0.f;
    splineh<ORDER>(x, hx, wxh);
    splineh<ORDER>(y, hy, wyh);
    const int gx = lx + O::GLO + O::LP, gy = ly + O::GLO + O::LP;
    const int gxh = gx - (x < 0.f), gyh = gy - (y < 0.f);
    float e1 = 0.f, e2 = 0.f, e3 = 0.f, b1 = 0.f, b2 = 0.f, b3 = 0.f;
#pragma unroll
    for (int k2 = 0; k2 < NP; k2++) {
      float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
      for (int k1 = 0; k1 < NP; k1++) {
        l1 = fma_(sE1[(gy + k2) * GX + gxh + k1], wxh[k1], l1);
        l2 = fma_(sE2[(gyh + k2) * GX + gx + k1], wx[k1], l2);
        l3 = fma_(sE3[(gy + k2) * GX + gx + k1], wx[k1], l3);
      }
      e1 = fma_(l1, wy[k2], e1);
      e2 = fma_(l2, wyh[k2], e2);
      e3 = fma_(l3, wy[k2], e3);
    }
#pragma unroll
    for (int k2 = 0; k2 < NP; k2++) {
      float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
      for (int k1 = 0; k1 < NP; k1++) {
        l1 = fma_(sB1[(gyh + k2) * GX + gx + k1], wx[k1], l1);
        l2 = fma_(sB2[(gy + k2) * GX + gxh + k1], wxh[k1], l2);
        l3 = fma_(sB3[(gyh + k2) * GX + gxh + k1], wxh[k1], l3);
      }
      b1 = fma_(l1, wyh[k2], b1);
      b2 = fma_(l2, wy[k2], b2);
      b3 = fma_(l3, wyh[k2], b3);
    }
    // ---- push
    const float ke = push<PUSHER>(tem, e1, e2, e3, b1, b2, b3, u1, u2, u3);
    if (act) ene += (double)q * (double)ke;
    // ---- position
    const float rg = rgamma(u1, u2, u3);
    const float v1 = u1 * rg, v2 = u2 * rg, v3 = u3 * rg;
    const float x1 = fma_(v1, dtdx1, x), y1 = fma_(v2, dtdx2, y);
    const float tx = trim(x1), ty = trim(y1);
    const int dix = (int)tx, diy = (int)ty;
    // ---- split + deposit
    VP2 vp[3];
    const int nvp = act ? split2d(x, y, x1, y1, dix, diy, q, v3, vp) : 0;
    for (int v = 0; v < nvp; v++) {
      const VP2 V = pick(vp, v);
      float S0x[NP], S0y[NP];
      spline<ORDER>(V.x0, S0x);
      spline<ORDER>(V.y0, S0y);
      const int jx0 = lx + V.di + O::LP + O::JLO, jy0 = ly + V.dj + O::LP + O::JLO;
      dep_vp<ORDER>(sJ1, sJ2, sJ3, S0x, S0y, V.x0, V.y0, V.x1, V.y1, V.q, V.vz, jy0 * JX + jx0,
                    JX, jn1, jn2, jscale);
    }
    // ---- store: stay in place, or leave through the mover buffer
    int nix = wrapi(lx + cx0 + dix, nx), niy = wrapi(ly + cy0 + diy, ny);
    const uint32_t ncell = pack2(nix, niy);
    const bool stay = (nix / TX + g.ntx * (niy / TY)) == tile;
    const float xs = x1 - tx, ys = y1 - ty;
    if (act && stay) {
      const int s = base + p;
      d.cell[s] = ncell;
      d.x[s] = xs;
      d.y[s] = ys;
      d.ux[s] = u1;
      d.uy[s] = u2;
      d.uz[s] = u3;
    }
    const bool mv = act && !stay;
    const unsigned long long mm = __ballot(mv);
    if (mv) {
      const int slot = base + w0 + mcount + __popcll(mm & ((1ull << lane) - 1ull));
      const int s = base + p;
      d.mcell[slot] = ncell;
      d.mx[slot] = xs;
      d.my[slot] = ys;
      d.mux[slot] = u1;
      d.muy[slot] = u2;
      d.muz[slot] = u3;
      d.mq[slot] = q;
      d.mpid[slot] = d.pid[s];
      d.midx[slot] = p;
    }
    mcount += __popcll(mm);
  }
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
  // ---- fold the LDS current tile into global J with the periodic wrap
  for (int i = threadIdx.x; i < JN; i += NT) {
    const int gx = wrapi(cx0 + (i % JX) - O::JLO, nx), gy = wrapi(cy0 + (i / JX) - O::JLO, ny);
    const long long gi = gx + (long long)nx * gy;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const unsigned long long v = sJ[c * JN + i];
      if (v) atomicAdd(&g.J[co + c * nc + gi], v);
    }
  }
}

// ------------------------------------------------------------------------------------
// 3D push + deposit
// ------------------------------------------------------------------------------------
template <int ORDER, int PUSHER, int NT>
__global__ __launch_bounds__(NT) void push_deposit_3d(const SpecDesc* __restrict__ descs,
                                                      const int2* __restrict__ work) {
  using O = Ord<ORDER>;
  constexpr int NP = O::NP;
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double s_ene[NT / 64];

  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (g.ctrl->halt != 0) return;
  const int tile = wk.y;
  const int TX = g.tx, TY = g.ty, TZ = g.tz;
  const int GX = TX + O::GLO + O::GHI, GY = TY + O::GLO + O::GHI, GZ = TZ + O::GLO + O::GHI;
  const int JX = TX + O::JLO + O::JHI, JY = TY + O::JLO + O::JHI, JZ = TZ + O::JLO + O::JHI;
  const int GN = GX * GY * GZ, JN = JX * JY * JZ;
  unsigned long long* sJ = (unsigned long long*)smem;
  float* sF = (float*)(smem + sizeof(unsigned long long) * 3 * JN);
  // per-wave queues of the virtual particles 1..3 (x0, y0, z0, x1, y1, z1, q; node)
  constexpr int QC = kVpQueue3;
  float* sQall = sF + 6 * GN;
  int* sQnall = (int*)(sQall + (NT / 64) * 7 * QC);
  const int ttx = tile % g.ntx, tty = (tile / g.ntx) % g.nty, ttz = tile / (g.ntx * g.nty);
  const int cx0 = ttx * TX, cy0 = tty * TY, cz0 = ttz * TZ;
  const int nx = g.nx, ny = g.ny, nz = g.nz;
  const long long nc = g.ncell;

  for (int i = threadIdx.x; i < GN; i += NT) {
    const int lx = i % GX, ly = (i / GX) % GY, lz = i / (GX * GY);
    const int gx = wrapi(cx0 + lx - O::GLO, nx), gy = wrapi(cy0 + ly - O::GLO, ny),
              gz = wrapi(cz0 + lz - O::GLO, nz);
    const long long gi = gx + (long long)nx * (gy + (long long)ny * gz);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      sF[c * GN + i] = g.E[c * nc + gi];
      sF[(3 + c) * GN + i] = g.B[c * nc + gi];
    }
  }
  for (int i = threadIdx.x; i < 3 * JN; i += NT) sJ[i] = 0ull;
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int NW = NT / 64;
  const int base = d.off[tile];
  const int n = d.cnt[tile];
  const int per_wave = ((n + NT - 1) / NT) * 64;
  const int w0 = wave * per_wave;
  const int w1 = min(w0 + per_wave, n);
  const float tem = d.tem;
  const float dtdx1 = g.dt_dx[0], dtdx2 = g.dt_dx[1], dtdx3 = g.dt_dx[2];
  const float jn1 = g.jnorm[0], jn2 = g.jnorm[1], jn3 = g.jnorm[2];
  const double jscale = g.jscale;
  const int GXY = GX * GY, JXY = JX * JY;

  float* const Q = sQall + wave * 7 * QC;
  int* const QN = sQnall + wave * QC;
  int qhead = 0, qlen = 0;
  // deposit of the queued VPs in slots [head, head + cnt) (cnt <= 64, one per lane)
  auto deposit_queue = [&](int head, int cnt) {
    wave_lds_sync();  // the entries of the other lanes
    if (lane < cnt) {
      const int sl = (head + lane) & (QC - 1);
      const float x0 = Q[sl], y0 = Q[QC + sl], z0 = Q[2 * QC + sl];
      float S0x[NP], S0y[NP], S0z[NP];
      spline<ORDER>(x0, S0x);
      spline<ORDER>(y0, S0y);
      spline<ORDER>(z0, S0z);
      dep_vp3<ORDER>(sJ, JN, S0x, S0y, S0z, x0, y0, z0, Q[3 * QC + sl], Q[4 * QC + sl],
                     Q[5 * QC + sl], Q[6 * QC + sl], QN[sl], JX, JXY, jn1, jn2, jn3, jscale);
    }
    wave_lds_sync();  // read before any is written again
  };

  double ene = 0.0;
  int mcount = 0;
  bool bad = false;
  for (int p0 = w0; p0 < w1; p0 += 64) {
    const int p = p0 + lane;
    bool act = p < w1;
    uint32_t cell = 0;
    float x = 0.f, y = 0.f, z = 0.f, u1 = 0.f, u2 = 0.f, u3 = 0.f, q = 0.f;
    int lx = 0, ly = 0, lz = 0;
    if (act) {
      const int s = base + p;
      cell = d.cell[s];
      x = d.x[s];
      y = d.y[s];
      z = d.z[s];
      u1 = d.ux[s];
      u2 = d.uy[s];
      u3 = d.uz[s];
      q = d.q[s];
      int ix, iy, iz;
      unpack3(cell, ix, iy, iz);
      lx = ix - cx0;
      ly = iy - cy0;
      lz = iz - cz0;
      if (lx < 0 || lx >= TX || ly < 0 || ly >= TY || lz < 0 || lz >= TZ) {
        bad = true;
        act = false;
        lx = ly = lz = 0;
      }
    }
    float wx[NP], wy[NP], wz[NP], wxh[NP], wyh[NP], wzh[NP];
    spline<ORDER>(x, wx);
    spline<ORDER>(y, wy);
    spline<ORDER>(z, wz);
    splineh<ORDER>(x, x < 0.f ? 1.f : 0.f, wxh);
    splineh<ORDER>(y, y < 0.f ? 1.f : 0.f, wyh);
    splineh<ORDER>(z, z < 0.f ? 1.f : 0.f, wzh);
    const int gx = lx + O::GLO + O::LP, gy = ly + O::GLO + O::LP, gz = lz + O::GLO + O::LP;
    const int gxh = gx - (x < 0.f), gyh = gy - (y < 0.f), gzh = gz - (z < 0.f);
    const float* sE1 = sF;
    const float* sE2 = sF + GN;
    const float* sE3 = sF + 2 * GN;
    const float* sB1 = sF + 3 * GN;
    const float* sB2 = sF + 4 * GN;
    const float* sB3 = sF + 5 * GN;
    // GET_EMF_3D line/plane order (os-emf-interpolate.f03:697-773); the AVX2 3D kernel
    // uses the same fma order along k1, then k2, then k3.
    float e1 = 0.f, e2 = 0.f, e3 = 0.f;
#pragma unroll
    for (int k3 = 0; k3 < NP; k3++) {
      float p1 = 0.f, p2 = 0.f, p3 = 0.f;
#pragma unroll
      for (int k2 = 0; k2 < NP; k2++) {
        float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
        for (int k1 = 0; k1 < NP; k1++) {
          l1 = fma_(sE1[(gz + k3) * GXY + (gy + k2) * GX + gxh + k1], wxh[k1], l1);
          l2 = fma_(sE2[(gz + k3) * GXY + (gyh + k2) * GX + gx + k1], wx[k1], l2);
          l3 = fma_(sE3[(gzh + k3) * GXY + (gy + k2) * GX + gx + k1], wx[k1], l3);
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
#pragma unroll
      for (int k2 = 0; k2 < NP; k2++) {
        float l1 = 0.f, l2 = 0.f, l3 = 0.f;
#pragma unroll
        for (int k1 = 0; k1 < NP; k1++) {
          l1 = fma_(sB1[(gzh + k3) * GXY + (gyh + k2) * GX + gx + k1], wx[k1], l1);
          l2 = fma_(sB2[(gzh + k3) * GXY + (gy + k2) * GX + gxh + k1], wxh[k1], l2);
          l3 = fma_(sB3[(gz + k3) * GXY + (gyh + k2) * GX + gxh + k1], wxh[k1], l3);
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
    if (act) ene += (double)q * (double)ke;
    const float rg = rgamma(u1, u2, u3);
    const float x1 = fma_(u1 * rg, dtdx1, x), y1 = fma_(u2 * rg, dtdx2, y),
                z1 = fma_(u3 * rg, dtdx3, z);
    const float tx = trim(x1), ty = trim(y1), tz = trim(z1);
    const int dix = (int)tx, diy = (int)ty, diz = (int)tz;
    // split; VP 0 is deposited in place with the gather's splines (it starts at the old
    // position), VPs 1..3 of the lanes whose trajectory crosses faces go through the queue
    VP3 vp[4];
    const int nvp = act ? split3d(x, y, z, x1, y1, z1, dix, diy, diz, q, vp) : 0;
    const int nb0 = (lz + O::LP + O::JLO) * JXY + (ly + O::LP + O::JLO) * JX + lx + O::LP + O::JLO;
    if (act)
      dep_vp3<ORDER>(sJ, JN, wx, wy, wz, vp[0].x0, vp[0].y0, vp[0].z0, vp[0].x1, vp[0].y1,
                     vp[0].z1, vp[0].q, nb0, JX, JXY, jn1, jn2, jn3, jscale);
    const unsigned long long below = (1ull << lane) - 1ull;
#pragma unroll
    for (int v = 1; v < 4; v++) {
      const unsigned long long m = __ballot(v < nvp);
      if (m == 0ull) break;
      if (v < nvp) {
        const VP3 V = pick(vp, v);
        const int sl = (qhead + qlen + __popcll(m & below)) & (QC - 1);
        Q[0 * QC + sl] = V.x0;
        Q[1 * QC + sl] = V.y0;
        Q[2 * QC + sl] = V.z0;
        Q[3 * QC + sl] = V.x1;
        Q[4 * QC + sl] = V.y1;
        Q[5 * QC + sl] = V.z1;
        Q[6 * QC + sl] = V.q;
        QN[sl] = nb0 + V.dk * JXY + V.dj * JX + V.di;
      }
      qlen += __popcll(m);
      if (qlen >= 64) {
        deposit_queue(qhead, 64);
        qhead = (qhead + 64) & (QC - 1);
        qlen -= 64;
      }
    }
    const int nix = wrapi(lx + cx0 + dix, nx), niy = wrapi(ly + cy0 + diy, ny),
              niz = wrapi(lz + cz0 + diz, nz);
    const uint32_t ncell = pack3(nix, niy, niz);
    const bool stay = (nix / TX + g.ntx * (niy / TY + g.nty * (niz / TZ))) == tile;
    const float xs = x1 - tx, ys = y1 - ty, zs = z1 - tz;
    if (act && stay) {
      const int s = base + p;
      d.cell[s] = ncell;
      d.x[s] = xs;
      d.y[s] = ys;
      d.z[s] = zs;
      d.ux[s] = u1;
      d.uy[s] = u2;
      d.uz[s] = u3;
    }
    const bool mv = act && !stay;
    const unsigned long long mm = __ballot(mv);
    if (mv) {
      const int slot = base + w0 + mcount + __popcll(mm & ((1ull << lane) - 1ull));
      const int s = base + p;
      d.mcell[slot] = ncell;
      d.mx[slot] = xs;
      d.my[slot] = ys;
      d.mz[slot] = zs;
      d.mux[slot] = u1;
      d.muy[slot] = u2;
      d.muz[slot] = u3;
      d.mq[slot] = q;
      d.mpid[slot] = d.pid[s];
      d.midx[slot] = p;
    }
    mcount += __popcll(mm);
  }
  if (qlen > 0) deposit_queue(qhead, qlen);
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
  for (int i = threadIdx.x; i < JN; i += NT) {
    const int lx = i % JX, ly = (i / JX) % JY, lz = i / JXY;
    const int gx = wrapi(cx0 + lx - O::JLO, nx), gy = wrapi(cy0 + ly - O::JLO, ny),
              gz = wrapi(cz0 + lz - O::JLO, nz);
    const long long gi = gx + (long long)nx * (gy + (long long)ny * gz);
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const unsigned long long v = sJ[c * JN + i];
      if (v) atomicAdd(&g.J[c * nc + gi], v);
    }
  }
}

// ------------------------------------------------------------------------------------
// Tile maintenance
// ------------------------------------------------------------------------------------
// k-th neighbour tile (dz, dy, dx order, dx fastest, the tile itself left out) of the tile at
// (tx, ty, tz)
OSR_DEV int neighbour(const GridDesc& g, int tx, int ty, int tz, int k) {
  int dz = 0;
  if (g.dims == 2) {
    k += k >= 4;
  } else {
    k += k >= 13;
    dz = k / 9 - 1;
    k = k % 9;
  }
  const int x = wrapi(tx + k % 3 - 1, g.ntx), y = wrapi(ty + k / 3 - 1, g.nty);
  const int z = g.dims == 2 ? 0 : wrapi(tz + dz, g.ntz);
  return x + g.ntx * (y + g.nty * z);
}

OSR_DEV void copy_from_mover(const SpecDesc& d, int src, int dst, int dims) {
  d.cell[dst] = d.mcell[src];
  d.x[dst] = d.mx[src];
  d.y[dst] = d.my[src];
  if (dims == 3) d.z[dst] = d.mz[src];
  d.ux[dst] = d.mux[src];
  d.uy[dst] = d.muy[src];
  d.uz[dst] = d.muz[src];
  d.q[dst] = d.mq[src];
  d.pid[dst] = d.mpid[src];
}

OSR_DEV void copy_particle(const SpecDesc& d, int src, int dst, int dims) {
  d.cell[dst] = d.cell[src];
  d.x[dst] = d.x[src];
  d.y[dst] = d.y[src];
  if (dims == 3) d.z[dst] = d.z[src];
  d.ux[dst] = d.ux[src];
  d.uy[dst] = d.uy[src];
  d.uz[dst] = d.uz[src];
  d.q[dst] = d.q[src];
  d.pid[dst] = d.pid[src];
}


// Move the movers destined to this tile into it and close the holes (deterministic:
// sources = incoming movers by (neighbour, wave, slot), then the non-hole particles of
// the tail [newcnt, cnt) ascending; targets = holes below newcnt ascending, then the
// appended slots [cnt, newcnt)).  A tile that cannot take its incoming particles (its
// capacity, or this kernel's LDS list of them, would overflow) changes nothing, marks
// itself with inc = -1 and raises Ctrl::halt; the host then re-lays the species out from
// the tiles that did fill plus the mover buffers.
// NT threads per tile; INC_MAX incoming movers are the most one fill handles; beyond them the
// tile flags an overflow.  Any number may leave.  (The third parameter, once a limit on that, is
// part of the name under which the host checks know the kernel.)
//
// Bound: the chain of dependent loads and barriers of a tile (a tile moves few particles),
// so the loads that depend on the same thing go out together: every list's length and base
// by a thread of its own, then the own holes and the candidates' cells, then the movers.
// The binary searches run on LDS tables, branch-free and in step for all items of a thread.
// us per launch, lists walked by thread 0 and wave 0 / this: 64x64 14.1 / 9.2, 52x44x36
// 26 / 12.8, 96^3 two beams 118 / 69, 192^3 533 / 385, 1024x1024 two beams 98 / 90 (there
// and on 192^3 the scattered 4-byte copies of the movers take most of it).
constexpr int kFillPF = 8;      // candidate movers per thread whose cells are loaded together
constexpr int kFillHoles = 1024;  // own holes held in LDS (the rest are read from memory)

// Last l with ofs[l] <= v[p], for PF values at once: ofs is non-decreasing, ofs[0] <= v, and
// padded above its last entry with INT_MAX up to N (a power of two) entries.
template <int N, int PF>
OSR_DEV void seg_find_multi(const int* ofs, const int (&v)[PF], int (&l)[PF]) {
#pragma unroll
  for (int p = 0; p < PF; p++) l[p] = 0;
#pragma unroll
  for (int h = N / 2; h > 0; h >>= 1)
#pragma unroll
    for (int p = 0; p < PF; p++)
      if (ofs[l[p] + h] <= v[p]) l[p] += h;
}

template <int NT, int INC_MAX, int>
__global__ __launch_bounds__(NT) void tile_fill(const SpecDesc* __restrict__ descs,
                                                const int2* __restrict__ work) {
  constexpr int MAXL = 26 * kMaxTileWaves;  // candidate lists: neighbours x waves
  constexpr int PERL = (MAXL + NT - 1) / NT, NTAB = 512, NHT = 2 * kMaxTileWaves;
  static_assert(MAXL < NTAB, "list table");
  __shared__ int s_lofs[NTAB], s_lbase[MAXL], s_hofs[NHT];
  __shared__ int s_lsum[PERL][NT / 64];
  __shared__ int s_pcnt[kFillPF][NT / 64];
  __shared__ int s_hole[kFillHoles];
  __shared__ int s_inc[INC_MAX];
  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (d.fd && (int)blockIdx.x >= d.fd_first) {  // a block of field work, in the list's arrays
    static_assert(sizeof(s_inc) >= sizeof(float) * kYeeLds<32, 8>, "staged fields");
    field_beside_fill(*(const FieldDesc*)d.fd, d.fd_kind, (int)blockIdx.x - d.fd_first,
                      (float*)s_inc);
    return;
  }
  const int tile = wk.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int NW = d.waves, wsh = 31 - __clz(NW);  // a power of two
  const int dims = g.dims;
  const int L = (dims == 2 ? 8 : 26) << wsh;
  const int base = d.off[tile], n = d.cnt[tile], cap = d.cap[tile], stride = d.mv_stride[tile];
  const int tx = tile % g.ntx, ty = (tile / g.ntx) % g.nty, tz = tile / (g.ntx * g.nty);
  // a direction of one or two tiles names some neighbours twice, or the tile itself
  const bool small = g.ntx < 3 || g.nty < 3 || (dims == 3 && g.ntz < 3);
  if (g.ctrl->halt >= 2) return;
  // list lengths and bases, and the prefix of the lengths
  int cnt[PERL], pre[PERL];
#pragma unroll
  for (int j = 0; j < PERL; j++) {
    const int l = tid + j * NT;
    cnt[j] = 0;
    if (l < L) {
      const int k = l >> wsh, w = l & (NW - 1), nt = neighbour(g, tx, ty, tz, k);
      bool dup = false;
      if (small) {
        dup = nt == tile;
        for (int i = 0; i < k; i++) dup |= neighbour(g, tx, ty, tz, i) == nt;
      }
      if (!dup) cnt[j] = d.mv_cnt[(nt << wsh) + w];
      s_lbase[l] = d.off[nt] + w * d.mv_stride[nt];
    }
  }
  const int own = tid < NW ? d.mv_cnt[(tile << wsh) + tid] : 0;  // wave 0: the tile's own lists
  for (int i = tid; i < NTAB; i += NT)
    if (i == 0 || i > L) s_lofs[i] = i == 0 ? 0 : 0x7FFFFFFF;
  auto wave_scan = [&](int v) {  // inclusive, over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(v, o, 64);
      if (lane >= o) v += t;
    }
    return v;
  };
#pragma unroll
  for (int j = 0; j < PERL; j++) {
    pre[j] = wave_scan(cnt[j]);
    if (lane == 63) s_lsum[j][wave] = pre[j];
  }
  if (wave == 0) {
    const int h = wave_scan(own);
    if (lane == 0) s_hofs[0] = 0;
    if (lane < NHT - 1) s_hofs[lane + 1] = lane < NW ? h : 0x7FFFFFFF;
  }
  __syncthreads();
  int T = 0;
#pragma unroll
  for (int j = 0; j < PERL; j++) {
    int before = T;
#pragma unroll
    for (int w = 0; w < NT / 64; w++) {
      const int v = s_lsum[j][w];
      if (w < wave) before += v;
      T += v;
    }
    const int l = tid + j * NT;
    if (l < L) s_lofs[l + 1] = before + pre[j];
  }
  const int H = s_hofs[NW];
  // a tile of the guard band of open x walls takes no movers: the particles that left
  // through a wall (ix < 1 or ix > nx) are dropped (spec/os-spec-boundary.f03:476-513)
  if (tx * g.tx >= interior_nx(g)) T = 0;
  __syncthreads();
  auto hole_at = [&](int k) -> int {  // own hole k from memory
    const int v[1] = {k};
    int w[1];
    seg_find_multi<NHT, 1>(s_hofs, v, w);
    return d.midx[base + w[0] * stride + (k - s_hofs[w[0]])];
  };
  // holes are ascending in k: each wave's movers are in slot order, and so are the waves
  for (int k = tid; k < min(H, kFillHoles); k += NT) s_hole[k] = hole_at(k);
  // pass 1: collect the incoming movers, in candidate order.  Candidates are taken PF NT
  // at a time, candidate c0 + p NT + thread as item p of the thread, and the cells of all
  // of them are loaded before any is ranked: one memory round trip per PF NT candidates
  // (a tile's neighbours hold some 8 x 200 movers on the 2D two-stream workload).
  const int cx0 = tx * g.tx, cy0 = ty * g.ty, cz0 = tz * g.tz;
  auto in_tile = [&](uint32_t c) {
    int ix, iy, iz = 0;
    if (dims == 2)
      unpack2(c, ix, iy);
    else
      unpack3(c, ix, iy, iz);
    return (unsigned)(ix - cx0) < (unsigned)g.tx && (unsigned)(iy - cy0) < (unsigned)g.ty &&
           (dims == 2 || (unsigned)(iz - cz0) < (unsigned)g.tz);
  };
  int I = 0;
  auto collect = [&](auto pf, int c0) {
    constexpr int PF = decltype(pf)::value;
    int v[PF], l[PF], src[PF], r[PF], tot;
    uint32_t cell[PF];
    bool f[PF];
#pragma unroll
    for (int p = 0; p < PF; p++) v[p] = min(c0 + p * NT + tid, T - 1);
    seg_find_multi<NTAB, PF>(s_lofs, v, l);
#pragma unroll
    for (int p = 0; p < PF; p++) {
      src[p] = s_lbase[l[p]] + (v[p] - s_lofs[l[p]]);
      cell[p] = d.mcell[src[p]];
    }
#pragma unroll
    for (int p = 0; p < PF; p++) f[p] = c0 + p * NT + tid < T && in_tile(cell[p]);
    block_rank_multi<NT, PF>(f, s_pcnt, r, tot);
#pragma unroll
    for (int p = 0; p < PF; p++)
      if (f[p] && I + r[p] < INC_MAX) s_inc[I + r[p]] = src[p];
    I += tot;
  };
  for (int c0 = 0; c0 < T;) {  // T is uniform
    if (T - c0 <= 2 * NT) {
      collect(std::integral_constant<int, 2>(), c0);
      c0 += 2 * NT;
    } else {
      collect(std::integral_constant<int, kFillPF>(), c0);
      c0 += kFillPF * NT;
    }
  }
  // every wave's entries of s_inc and s_hole are in LDS before any wave reads them below
  __syncthreads();
  const int nn = n - H + I;
  if (I > INC_MAX || nn > cap - 64 * NW) {
    if (tid == 0) {
      d.inc[tile] = -1;
      // the count the tile needs after this step, or -1 if more capacity would not help
      // (the incoming list exceeds this kernel's limit)
      d.newcnt[tile] = I > INC_MAX ? -1 : nn;
      atomicOr(&g.ctrl->halt, 1);
    }
    return;
  }
  auto hole = [&](int k) -> int { return k < kFillHoles ? s_hole[k] : hole_at(k); };
  // holes below nn: the whole list unless the tile shrinks
  int hlo = H;
  if (I < H) {
    int lo = 0;
    while (lo < hlo) {
      const int mid = (lo + hlo) >> 1;
      if (hole(mid) < nn)
        lo = mid + 1;
      else
        hlo = mid;
    }
  }
  // pass 2: incoming movers into the holes below nn, then the appended slots
  for (int r = tid; r < I; r += NT)
    copy_from_mover(d, s_inc[r], base + (r < hlo ? hole(r) : n + (r - H)), dims);
  // pass 3: the particles of the tail [nn, n) into the remaining holes: the r-th of them is
  // slot nn + r + m, m the number of tail holes at or before it (hole hlo + j of the tail
  // has hole - nn - j particles below it, non-decreasing in j)
  for (int r = tid; r < hlo - I; r += NT) {
    int lo = 0, hi = H - hlo;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (hole(hlo + mid) - nn - mid <= r)
        lo = mid + 1;
      else
        hi = mid;
    }
    copy_particle(d, base + nn + r + lo, base + hole(I + r), dims);
  }
  if (tid == 0) {
    d.cnt[tile] = nn;
    d.inc[tile] = I;
  }
}

// ------------------------------------------------------------------------------------
// Device re-layout after a step whose fill overflowed a tile: one workgroup per tile
// copies the tile's particle slots [0, cnt) and its pending mover lists (the valid
// entries of each wave's region) from the old arrays to the same relative slots of the
// tile in the new, larger arrays.  Counts, mover counts and strides are per tile and stay
// valid; the fill of the overflowed tiles then runs again on the new layout.
// ------------------------------------------------------------------------------------
struct RegrowArrays {
  uint32_t* a[19];  // particle arrays (cell x y z ux uy uz q pid), mover arrays (mcell mx
                    // my mz mux muy muz mq mpid midx)
};
__global__ __launch_bounds__(256) void regrow_move(const SpecDesc* __restrict__ descs, int sid,
                                                   RegrowArrays src, RegrowArrays dst,
                                                   const int* __restrict__ new_off) {
  const SpecDesc& d = descs[sid];
  const int tile = blockIdx.x;
  const int o0 = d.off[tile], o1 = new_off[tile];
  const int n = d.cnt[tile];
  const int NW = d.waves, stride = d.mv_stride[tile];
  const bool three = d.g.dims == 3;
  for (int a = 0; a < 9; a++) {
    if (a == 3 && !three) continue;
    const uint32_t* S = src.a[a] + o0;
    uint32_t* D = dst.a[a] + o1;
    for (int i = threadIdx.x; i < n; i += 256) D[i] = S[i];
  }
  for (int w = 0; w < NW; w++) {
    const int m = d.mv_cnt[tile * NW + w];
    for (int a = 9; a < 19; a++) {
      if (a == 12 && !three) continue;
      const uint32_t* S = src.a[a] + o0 + w * stride;
      uint32_t* D = dst.a[a] + o1 + w * stride;
      for (int i = threadIdx.x; i < m; i += 256) D[i] = S[i];
    }
  }
}

// ------------------------------------------------------------------------------------
// Re-interleave the particles of each tile: slot order (rank within the cell, cell), the
// order the loader creates, so that the 64 lanes of a wave hold 64 different, consecutive
// cells and their LDS field reads and current updates spread over the banks.  The fill
// perturbs that order step by step; this restores it every `period` steps (after the
// fill of steps period-1, 2 period-1, ...).  Ranks follow the slot order, so the result
// is deterministic; the current is an integer sum and no arithmetic depends on the order
// (only the FP64 energy partials, at round-off).  Each particle array of the tile is
// permuted through LDS (coalesced read, LDS scatter, coalesced write back).  A step whose
// fill overflowed is skipped (the host re-lays those particles out), as are tiles with
// more than MAXN particles or RMAX particles in one cell.
// ------------------------------------------------------------------------------------
//
// Bound: latency, then HBM (each array is read and written once, 72 B per particle).  Every
// wave ranks a quarter of the slots, with counts of its own that the next waves start from,
// and each array's loads are issued before the previous one is stored.  us per launch, one
// launch in four active, one ranking wave / this: 52x44x36 18 / 12, 96^3 two beams 107 / 78,
// 192^3 8 per cell 629 / 450 (an active one moves 4.1 GB in 1.8 ms).
template <int NT, int RMAX, int MAXC, int MAXN>
__global__ __launch_bounds__(NT) void tile_reorder(const SpecDesc* __restrict__ descs,
                                                   const int2* __restrict__ work, int period) {
  constexpr int MAXW = RMAX * MAXC / 32, NW = NT / 64;
  constexpr int CB = 10;  // bits of a cell key in s_key
  static_assert(MAXC <= 1 << CB, "cell keys");
  __shared__ int s_cnt[NW][MAXC];  // particles of the cell in the wave's slots, then before them
  __shared__ int s_tot[MAXC];      // particles of the cell
  __shared__ unsigned int s_bits[MAXW];
  __shared__ int s_wpre[MAXW];
  __shared__ int s_key[MAXN];
  __shared__ __align__(16) uint32_t s_tmp[MAXN];
  __shared__ int s_sum[NW];
  __shared__ int s_abort, s_rows;
  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (period <= 0 || g.ctrl->halt != 0 || g.ctrl->steps % period != period - 1) return;
  const int tile = wk.y;
  const int base = d.off[tile], n = d.cnt[tile];
  const int dims = g.dims;
  const int C = g.tx * g.ty * (dims == 3 ? g.tz : 1);
  if (n < 2 || n > MAXN || C > MAXC) return;
  const int cx0 = (tile % g.ntx) * g.tx, cy0 = ((tile / g.ntx) % g.nty) * g.ty;
  const int cz0 = dims == 3 ? (tile / (g.ntx * g.nty)) * g.tz : 0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  for (int c = tid; c < NW * MAXC; c += NT) (&s_cnt[0][0])[c] = 0;
  if (tid == 0) s_abort = s_rows = 0;
  __syncthreads();
  int nbits = 0;  // bits of a local cell index
  while ((1 << nbits) < C) nbits++;
  // ranks within the cell in slot order, each wave over its own slots
  const int per = ((n + 64 * NW - 1) / (64 * NW)) * 64;
  {
    const int p0 = wave * per, p1 = min(p0 + per, n);
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t next = p0 + lane < p1 ? d.cell[base + p0 + lane] : 0u;
    for (int c0 = p0; c0 < p1; c0 += 64) {
      const int p = c0 + lane;
      const uint32_t cell = next;
      next = p + 64 < p1 ? d.cell[base + p + 64] : 0u;
      int lc = -1 - lane;  // distinct for the lanes past the end
      if (p < p1) {
        int ix, iy, iz = 0;
        if (dims == 2)
          unpack2(cell, ix, iy);
        else
          unpack3(cell, ix, iy, iz);
        const int lx = ix - cx0, ly = iy - cy0, lz = iz - cz0;
        if (lx < 0 || lx >= g.tx || ly < 0 || ly >= g.ty || lz < 0 ||
            lz >= (dims == 3 ? g.tz : 1))
          s_abort = 1;
        else
          lc = cell_key(lx, ly, lz, dims, g.tx, g.ty, dims == 3 ? g.tz : 1);
      }
      // lanes holding the same cell: one ballot per bit of the cell index
      unsigned long long same = __ballot(lc >= 0);
      for (int b = 0; b < nbits; b++) {
        const unsigned long long m = __ballot(lc >= 0 && ((lc >> b) & 1));
        same &= ((lc >> b) & 1) ? m : ~m;
      }
      const int before = __popcll(same & below);
      const int after = __popcll(same & ~below) - 1;
      if (lc >= 0) s_key[p] = ((s_cnt[wave][lc] + before) << CB) | lc;
      wave_lds_sync();
      if (lc >= 0 && after == 0) s_cnt[wave][lc] += before + 1;
      wave_lds_sync();
    }
  }
  __syncthreads();
  // per cell: what the waves before hold, and the total
  int rows = 0;
  for (int c = tid; c < C; c += NT) {
    int run = 0;
#pragma unroll
    for (int w = 0; w < NW; w++) {
      const int v = s_cnt[w][c];
      s_cnt[w][c] = run;
      run += v;
    }
    s_tot[c] = run;
    rows = max(rows, run);
  }
  if (rows > 0) atomicMax(&s_rows, rows);
  __syncthreads();
  rows = s_rows;
  if (s_abort || rows > RMAX) return;
  // occupancy of the keys (rank, cell): occupied iff the cell holds more than rank
  const int nw = (rows * C + 31) / 32;
  for (int w = tid; w < nw; w += NT) {
    unsigned int m = 0u;
    int r = (32 * w) / C, c = (32 * w) % C;  // key 32 w = r C + c, walked bit by bit
    for (int b = 0; b < 32; b++) {
      if (s_tot[c] > r) m |= 1u << b;
      if (++c == C) {
        c = 0;
        r++;
      }
    }
    s_bits[w] = m;
  }
  __syncthreads();
  // exclusive prefix of the word populations: each thread owns consecutive words
  const int own_w = (nw + NT - 1) / NT;
  const int w0 = tid * own_w;
  int own = 0;
  for (int k = 0; k < own_w; k++)
    if (w0 + k < nw) own += __popc(s_bits[w0 + k]);
  int inc = own;
  for (int o = 1; o < 64; o <<= 1) {
    const int t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) s_sum[wave] = inc;
  __syncthreads();
  int run = inc - own;
  for (int w = 0; w < wave; w++) run += s_sum[w];
  for (int k = 0; k < own_w; k++)
    if (w0 + k < nw) {
      s_wpre[w0 + k] = run;
      run += __popc(s_bits[w0 + k]);
    }
  __syncthreads();
  // new slot of every particle, in groups of 4 consecutive slots per thread (tile bases are
  // multiples of 64 slots)
  constexpr int PT = MAXN / (4 * NT);  // 4-slot groups per thread
  int dst[PT][4];
#pragma unroll
  for (int j = 0; j < PT; j++)
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int p = 4 * (tid + NT * j) + e;
      dst[j][e] = -1;
      if (p < n) {
        const int v = s_key[p], lc = v & ((1 << CB) - 1);
        const int k = ((v >> CB) + s_cnt[p / per][lc]) * C + lc;
        dst[j][e] = s_wpre[k >> 5] + __popc(s_bits[k >> 5] & ((1u << (k & 31)) - 1u));
      }
    }
  // permute each array through LDS: coalesced 16-byte reads, LDS scatter, coalesced writes
  uint32_t* arr[9] = {d.cell, (uint32_t*)d.x, (uint32_t*)d.y, (uint32_t*)d.z, (uint32_t*)d.ux,
                      (uint32_t*)d.uy, (uint32_t*)d.uz, (uint32_t*)d.q, d.pid};
  uint4 v[PT];
  auto load = [&](int a) {
    const uint32_t* A = arr[a] + base;
#pragma unroll
    for (int j = 0; j < PT; j++) {
      const int q = 4 * (tid + NT * j);
      v[j] = make_uint4(0u, 0u, 0u, 0u);
      if (q + 3 < n) {
        v[j] = *(const uint4*)(A + q);
      } else if (q < n) {
        v[j].x = A[q];
        if (q + 1 < n) v[j].y = A[q + 1];
        if (q + 2 < n) v[j].z = A[q + 2];
      }
    }
  };
  load(0);
#pragma unroll
  for (int a = 0; a < 9; a++) {
    if (a == 3 && dims != 3) continue;
    uint32_t* A = arr[a] + base;
#pragma unroll
    for (int j = 0; j < PT; j++) {
      const uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (dst[j][e] >= 0) s_tmp[dst[j][e]] = w[e];
    }
    if (a < 8) load(a == 2 && dims != 3 ? 4 : a + 1);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < PT; j++) {
      const int q = 4 * (tid + NT * j);
      if (q + 3 < n) {
        *(uint4*)(A + q) = *(const uint4*)(s_tmp + q);
      } else {
#pragma unroll
        for (int e = 0; e < 3; e++)
          if (q + e < n) A[q + e] = s_tmp[q + e];
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// explicit instantiations
// ------------------------------------------------------------------------------------
#define OSR_INST(O, P)                                                                    \
  template __global__ void push_deposit_2d<O, P, 256>(const SpecDesc*, const int2*);      \
  template __global__ void push_deposit_3d<O, P, 256>(const SpecDesc*, const int2*);
OSR_INST(1, 0)
OSR_INST(2, 0)
OSR_INST(3, 0)
OSR_INST(1, 1)
OSR_INST(2, 1)
OSR_INST(3, 1)
template __global__ void tile_fill<256, 4096, 32768>(const SpecDesc*, const int2*);
template __global__ void tile_reorder<256, 64, 512, 4096>(const SpecDesc*, const int2*, int);

}  // namespace osr
