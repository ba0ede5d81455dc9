// k_push2d.hip -- fused 2D push + deposit with compile-time tile shape.
//
// One workgroup of NW waves (4 or 8) per (species, tile); by default 8 for tiles of 512
// cells or more, whose LDS field and current tiles are then shared by twice as many
// waves.  Compared with the generic kernel in k_tiles.hip:
//  * TX/TY are template parameters, so every LDS stencil offset is an immediate;
//  * particle, mover and field arrays are accessed through global-address-space
//    pointers: uniform base + 32-bit offset, no per-array 64-bit address arithmetic, and
//    the loads do not share the LDS wait counter as flat accesses would;
//  * a particle that stays in its cell is one virtual particle (VP) and is deposited
//    straight from registers, with the start-point splines of the gather; one that crosses a
//    cell face (an eighth of them on the two-stream workload) is appended to a private LDS
//    queue of its wave, which splits and deposits 64 of them at a time, so that neither the
//    split nor the further VPs run on partly idle waves;
//  * the current of all waves is accumulated into one int64 fixed-point LDS tile; integer
//    adds are exact and order independent, so the deposit is bit-reproducible run to run
//    (FP32 LDS atomics were measured to be far slower here: a 40x longer LDS wait).
// What bounds it: LDS (bank conflicts of the 64-bit adds, whose lanes point at random nodes
// once the particles have moved: 12.7 cycles of a CU per add against 7.4 without conflicts)
// and VALU issue, together.  Two-stream 1024x1024, 64 per cell, quadratic, per 64 particles:
// 557 -> 443 VALU instructions (raw fixed-point bits, split and further VPs on full waves
// only), 36 -> 18 LDS reads; 1.270 -> 1.110 ms per step (3.63 TB/s of the 60 B a particle
// moves), VALU issue 83% of the cycles, bank conflicts 32%.  512x512, 16 per cell, cubic, Vay
// 170 -> 148 us, 515x267 quadratic 58 -> 54.5, 300x200 37 -> 31.6.
// The arithmetic of gather, push, position advance and split is the one of the generic
// kernel (the reference's AVX2 kernel, simd/os-spec-push-avx2.c:471-760).
#include <type_traits>

#include "osr_device.hpp"
#include "osr_types.hpp"

namespace osr {

typedef __attribute__((address_space(1))) float gf32;
typedef __attribute__((address_space(1))) uint32_t gu32;
typedef __attribute__((address_space(1))) int gi32;
typedef __attribute__((address_space(1))) unsigned long long gu64;
typedef __attribute__((address_space(1))) char gch;

// &b[i] through a 32-bit byte offset: base in scalar registers + one 32-bit VGPR, the
// form the saddr global loads and stores take directly (no 64-bit address arithmetic per
// array).  i * sizeof(*b) < 2^32 holds for every per-tile particle index.
template <class P>
OSR_DEV P el(P b, uint32_t i) {
  return (P)((gch*)b + i * (uint32_t)sizeof(*b));
}

// periodic wrap of a cell index at most one period outside [0, n)
OSR_DEV int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// LDS layout of the staged fields.  A ds_read_b128 takes about 10 cycles of a CU for 64
// lanes wherever they point (measured, also at random addresses), four 4-byte or two 8-byte
// reads 38 and 25 at random addresses (5 per 8 bytes without bank conflicts, which particles
// in the order a few steps leave them do not give).  So a 16-byte element per node holds what
// the node's x line needs next: the two components that share a stencil at the node and its
// right neighbour ((E1, B2) at half x, full y; (E2, B1) at full x, half y), and for E3 (full,
// full) and B3 (half, half) the node and the next three, or, with linear splines, whose line
// is two nodes, the node and the next one.
template <int ORDER>
struct Line2 {
  static constexpr int W = ORDER >= 2 ? 4 : 2;  // E3, B3 values per node
  typedef float V __attribute__((ext_vector_type(W)));
};
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

template <int ORDER, int PUSHER, int TX, int TY, int NW>
__global__ __launch_bounds__(64 * NW, 4) void push_deposit_2d_t(const SpecDesc* __restrict__ descs,
                                                                const int2* __restrict__ work) {
  using O = Ord<ORDER>;
  using LV = typename Line2<ORDER>::V;
  constexpr int NP = O::NP, LW = Line2<ORDER>::W;
  constexpr int NT = 64 * NW;
  // staged field tile GX x GY and current tile JX x JY
  constexpr int GX = TX + O::GLO + O::GHI, GY = TY + O::GLO + O::GHI, GN = GX * GY;
  constexpr int JX = TX + O::JLO + O::JHI, JY = TY + O::JLO + O::JHI, JN = JX * JY;
  constexpr int QC = 64;  // crossing particles queued per wave
  static_assert((TX & (TX - 1)) == 0 && (TY & (TY - 1)) == 0, "tile sides are powers of two");
  __shared__ f32x4 s12[GN], s21[GN];
  __shared__ LV s3[GN], s6[GN];
  __shared__ unsigned long long sJ[3 * JN];
  __shared__ f32x4 sQ[NW][2][QC];  // (x0, y0, x1, y1), (q, vz, node and cell shifts)
  __shared__ int sQn[NW];
  __shared__ double s_ene[NW];

  const int2 wk = work[blockIdx.x];
  const SpecDesc& d = descs[wk.x];
  const GridDesc& g = d.g;
  if (g.ctrl->halt != 0) return;
  const int tile = wk.y;
  const int cx0 = (tile % g.ntx) * TX, cy0 = (tile / g.ntx) * TY;
  const int nx = g.nx, ny = g.ny;
  const long long nc = g.ncell, co = cur_copy(g);

  {
    const gf32* __restrict__ E = (const gf32*)g.E + co;
    const gf32* __restrict__ B = (const gf32*)g.B + co;
    for (int i = threadIdx.x; i < GN; i += NT) {
      const int col = i % GX, row = i / GX;
      const int gx = wrapi(cx0 + col - O::GLO, nx), gy = wrapi(cy0 + row - O::GLO, ny);
      const long long gi = gx + (long long)nx * gy;
      const f32x2 p12 = {E[gi], B[nc + gi]}, p21 = {E[nc + gi], B[gi]};
      const float e3 = E[2 * nc + gi], b3 = B[2 * nc + gi];
      // this node's part of its own element and of those of the nodes on its left, as stores
      // of that part alone: other threads write the rest of each element
      ((f32x2*)s12)[2 * i] = p12;
      ((f32x2*)s21)[2 * i] = p21;
      if (col > 0) {
        ((f32x2*)s12)[2 * i - 1] = p12;
        ((f32x2*)s21)[2 * i - 1] = p21;
      }
#pragma unroll
      for (int k = 0; k < LW; k++)
        if (col >= k) {
          ((float*)s3)[LW * (i - k) + k] = e3;
          ((float*)s6)[LW * (i - k) + k] = b3;
        }
    }
  }
  for (int i = threadIdx.x; i < 3 * JN; i += NT) sJ[i] = 0ull;
  __syncthreads();

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // uniform per workgroup: keep them (and the array bases below) in scalar registers
  const int base = __builtin_amdgcn_readfirstlane(d.off[tile]);
  const int n = __builtin_amdgcn_readfirstlane(d.cnt[tile]);
  // this workgroup's waves among the split * NW of the tile (the work list names a tile
  // once per workgroup, back to back)
  const int split = d.split, part = (int)(blockIdx.x % (unsigned)split);
  const int tw = __builtin_amdgcn_readfirstlane(part * NW + wave);
  const int per_wave = ((n + NT * split - 1) / (NT * split)) * 64;
  const int w0 = tw * per_wave;
  const int w1 = min(w0 + per_wave, n);
  const float tem = d.tem;
  const float dtdx1 = g.dt_dx[0], dtdx2 = g.dt_dx[1];
  const float jn1 = g.jnorm[0], jn2 = g.jnorm[1];
  const double jscale = g.jscale;
  unsigned long long* const J1 = sJ;
  unsigned long long* const J2 = sJ + JN;
  unsigned long long* const J3 = sJ + 2 * JN;
  // particle and mover arrays of this tile, global address space
  const gu32* __restrict__ Pcell = (const gu32*)d.cell + base;
  const gf32* __restrict__ Px = (const gf32*)d.x + base;
  const gf32* __restrict__ Py = (const gf32*)d.y + base;
  const gf32* __restrict__ Pux = (const gf32*)d.ux + base;
  const gf32* __restrict__ Puy = (const gf32*)d.uy + base;
  const gf32* __restrict__ Puz = (const gf32*)d.uz + base;
  const gf32* __restrict__ Pq = (const gf32*)d.q + base;
  const gu32* __restrict__ Ppid = (const gu32*)d.pid + base;
  gu32* __restrict__ Wcell = (gu32*)d.cell + base;
  gf32* __restrict__ Wx = (gf32*)d.x + base;
  gf32* __restrict__ Wy = (gf32*)d.y + base;
  gf32* __restrict__ Wux = (gf32*)d.ux + base;
  gf32* __restrict__ Wuy = (gf32*)d.uy + base;
  gf32* __restrict__ Wuz = (gf32*)d.uz + base;
  gu32* __restrict__ Mcell = (gu32*)d.mcell + base;
  gf32* __restrict__ Mx = (gf32*)d.mx + base;
  gf32* __restrict__ My = (gf32*)d.my + base;
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
  const int tcx = min(TX, nx - cx0), tcy = min(TY, ny - cy0);
  const bool lone = g.ntx == 1 || g.nty == 1;
  const uint32_t cell0 = pack2(cx0, cy0);

  // the wave's particles; RAW: how the deposit adds (fix_bits)
  auto push_all = [&](auto raw) {
    constexpr bool RAW = decltype(raw)::value;
    int qlen = 0;
    f32x4* const Q0 = sQ[wave][0];
    f32x4* const Q1 = sQ[wave][1];
    const unsigned long long below = (1ull << lane) - 1ull;
    // split and deposit of queued particles, one per lane (on: the lane holds one, (a, b));
    // the third virtual particles of double crossings are queued again, as particles that
    // cross nothing
    auto deposit_queue = [&](bool on, const f32x4& a, const f32x4& b) {
      VP2 vp[3];
      int nvp = 0, nb0 = 0;
      if (on) {
        const int code = __float_as_int(b.z);
        nb0 = code >> 4;
        nvp = split2d_fast(a.x, a.y, a.z, a.w, (code & 3) - 1, ((code >> 2) & 3) - 1, b.x, b.y, vp);
      }
      const unsigned long long m2 = __ballot(nvp > 2);
      qlen = __popcll(m2);
      if (nvp > 2) {
        const int s = __popcll(m2 & below);
        Q0[s] = f32x4{vp[2].x0, vp[2].y0, vp[2].x1, vp[2].y1};
        Q1[s] = f32x4{vp[2].q, vp[2].vz,
                      __int_as_float((nb0 + vp[2].dj * JX + vp[2].di) * 16 + 1 + 4), 0.f};
      }
#pragma unroll
      for (int v = 0; v < 2; v++) {
        if (v < nvp) {
          float S0x[NP], S0y[NP];
          spline<ORDER>(vp[v].x0, S0x);
          spline<ORDER>(vp[v].y0, S0y);
          dep_vp<ORDER, RAW>(J1, J2, J3, S0x, S0y, vp[v].x0, vp[v].y0, vp[v].x1, vp[v].y1, vp[v].q,
                             vp[v].vz, nb0 + vp[v].dj * JX + vp[v].di, JX, jn1, jn2, jscale);
        }
      }
    };
    // The particle loads of the next iteration are issued before the current one is
    // processed (software pipelining): a wave otherwise waits a full memory latency per
    // iteration, and the bytes in flight per CU would cap the bandwidth well below peak.
    // Lanes past the end load the last particle again and are masked below.
    uint32_t f_cell = 0, f_pid = 0;
    float f_x = 0.f, f_y = 0.f, f_u1 = 0.f, f_u2 = 0.f, f_u3 = 0.f, f_q = 0.f;
    auto prefetch = [&](int pf) {
      const unsigned upf = (unsigned)min(pf, w1 - 1);
      f_cell = *el(Pcell, upf);
      f_x = *el(Px, upf);
      f_y = *el(Py, upf);
      f_u1 = *el(Pux, upf);
      f_u2 = *el(Puy, upf);
      f_u3 = *el(Puz, upf);
      f_q = *el(Pq, upf);
      f_pid = *el(Ppid, upf);
    };
    if (w0 < w1) prefetch(w0 + lane);
    for (int p0 = w0; p0 < w1; p0 += 64) {
      const int p = p0 + lane;
      const unsigned up = (unsigned)p;  // 32-bit unsigned offsets from the scalar bases
      const uint32_t cell = f_cell, pid = f_pid;
      const float x = f_x, y = f_y, q = f_q;
      float u1 = f_u1, u2 = f_u2, u3 = f_u3;
      if (p0 + 64 < w1) prefetch(p + 64);
      // cell within the tile: both halves of the difference in range (a borrow shows too)
      const uint32_t dl = cell - cell0;
      const bool out = (dl & ~((TX - 1u) | ((TY - 1u) << 16))) != 0u;
      const bool act = p < w1 && !out;
      bad |= p < w1 && out;
      const int lx = (int)(dl & (TX - 1u)), ly = (int)((dl >> 16) & (TY - 1u));
      // ---- gather
      float wx[NP], wy[NP], wxh[NP], wyh[NP];
      spline<ORDER>(x, wx);
      spline<ORDER>(y, wy);
      splineh<ORDER>(x, x < 0.f ? 1.f : 0.f, wxh);
      splineh<ORDER>(y, y < 0.f ? 1.f : 0.f, wyh);
      const int gb = (ly + O::GLO + O::LP) * GX + lx + O::GLO + O::LP;
      const int gbx = gb - (x < 0.f ? 1 : 0);
      const int gby = gb - (y < 0.f ? GX : 0);
      const int gbxy = gbx - (y < 0.f ? GX : 0);
      float e1 = 0.f, e2 = 0.f, e3 = 0.f, b1 = 0.f, b2 = 0.f, b3 = 0.f;
#pragma unroll
      for (int k2 = 0; k2 < NP; k2++) {
        // the row's line of each stencil
        float r12[2 * NP + 2], r21[2 * NP + 2], r3[NP + 1], r6[NP + 1];
        auto pairs = [&](const f32x4* L, float* r) {
#pragma unroll
          for (int k1 = 0; k1 < NP; k1 += 2) {
            f32x4 v = L[k1];
            if (k1 + 1 == NP) asm("" : "+v"(v));  // a full read: the low half alone is slower
            r[2 * k1] = v.x;
            r[2 * k1 + 1] = v.y;
            r[2 * k1 + 2] = v.z;
            r[2 * k1 + 3] = v.w;
          }
        };
        auto line = [&](const LV* L, float* r) {
#pragma unroll
          for (int k1 = 0; k1 < NP; k1 += LW) {
            const LV v = L[k1];
#pragma unroll
            for (int k = 0; k < LW; k++)
              if (k1 + k < NP) r[k1 + k] = v[k];
          }
        };
        pairs(s12 + gbx + k2 * GX, r12);
        pairs(s21 + gby + k2 * GX, r21);
        line(s3 + gb + k2 * GX, r3);
        line(s6 + gbxy + k2 * GX, r6);
        float le1 = 0.f, le2 = 0.f, le3 = 0.f, lb1 = 0.f, lb2 = 0.f, lb3 = 0.f;
#pragma unroll
        for (int k1 = 0; k1 < NP; k1++) {
          le1 = fma_(r12[2 * k1], wxh[k1], le1);
          le2 = fma_(r21[2 * k1], wx[k1], le2);
          le3 = fma_(r3[k1], wx[k1], le3);
          lb1 = fma_(r21[2 * k1 + 1], wx[k1], lb1);
          lb2 = fma_(r12[2 * k1 + 1], wxh[k1], lb2);
          lb3 = fma_(r6[k1], wxh[k1], lb3);
        }
        e1 = fma_(le1, wy[k2], e1);
        e2 = fma_(le2, wyh[k2], e2);
        e3 = fma_(le3, wy[k2], e3);
        b1 = fma_(lb1, wyh[k2], b1);
        b2 = fma_(lb2, wy[k2], b2);
        b3 = fma_(lb3, wyh[k2], b3);
      }
      // ---- push
      const float ke = push<PUSHER>(tem, e1, e2, e3, b1, b2, b3, u1, u2, u3);
      ene = __builtin_fma((double)(act ? q : 0.f), (double)ke, ene);
      // ---- position
      const float rg = rgamma(u1, u2, u3);
      const float v1 = u1 * rg, v2 = u2 * rg, v3 = u3 * rg;
      const float x1 = fma_(v1, dtdx1, x), y1 = fma_(v2, dtdx2, y);
      const float tx = trim(x1), ty = trim(y1);
      const int dix = (int)tx, diy = (int)ty;
      // ---- deposit of the particles that stay in their cell: one VP, with the gather's
      // splines; the others are queued for the split
      const int nb0 = (ly + O::LP + O::JLO) * JX + lx + O::LP + O::JLO;
      const bool cross = act && (dix | diy) != 0;
      const f32x4 qa = {x, y, x1, y1};
      const f32x4 qb = {q, v3, __int_as_float(nb0 * 16 + (dix + 1) + 4 * (diy + 1)), 0.f};
      if (act && !cross)
        dep_vp<ORDER, RAW>(J1, J2, J3, wx, wy, x, y, x1, y1, q, v3, nb0, JX, jn1, jn2, jscale);
      // ---- store: stay in place, or leave through the mover buffer
      const int nlx = lx + dix, nly = ly + diy;
      bool stay = (unsigned)nlx < (unsigned)tcx && (unsigned)nly < (unsigned)tcy;
      uint32_t ncell = cell0 + pack2(0, nly) + (uint32_t)nlx;
      if (lone || !__all(stay || !act)) {
        const int nix = wrap1(nlx + cx0, nx), niy = wrap1(nly + cy0, ny);
        ncell = pack2(nix, niy);
        stay = (nix / TX + g.ntx * (niy / TY)) == tile;
      }
      const float xs = x1 - tx, ys = y1 - ty;
      if (act && stay) {
        *el(Wcell, up) = ncell;
        *el(Wx, up) = xs;
        *el(Wy, up) = ys;
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
        *el(Mux, slot) = u1;
        *el(Muy, slot) = u2;
        *el(Muz, slot) = u3;
        *el(Mq, slot) = q;
        *el(Mpid, slot) = pid;
        *el(Midx, slot) = p;
      }
      mcount += __popcll(mm);
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
    // What is left in the queues, shared over the waves so that it runs on full ones: at most
    // NW QC entries, one batch per wave.  The second round takes what the first queued again.
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
  if (lane == 0) d.mv_cnt[tile * NW * split + tw] = mcount;
  if (threadIdx.x == 0 && part == 0) d.mv_stride[tile] = per_wave;
  ene = wave_sum(ene);
  if (lane == 0) s_ene[wave] = ene;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = s_ene[0];
#pragma unroll
    for (int w = 1; w < NW; w++) t += s_ene[w];
    d.epart[tile * split + part] = t;
  }
  // ---- fold the LDS current tile into the global fixed-point J (periodic wrap)
  gu64* __restrict__ GJ = (gu64*)g.J + co;
  for (int i = threadIdx.x; i < JN; i += NT) {
    const int gx = wrapi(cx0 + i % JX - O::JLO, nx), gy = wrapi(cy0 + i / JX - O::JLO, ny);
    const long long gi = gx + (long long)nx * gy;
#pragma unroll
    for (int c = 0; c < 3; c++) {
      const unsigned long long t = sJ[c * JN + i], v = raw ? fix_sum<true>(t) : t;
      if (v) __hip_atomic_fetch_add(&GJ[c * nc + gi], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

#define OSR_INST2(O, P, X, Y, W) \
  template __global__ void push_deposit_2d_t<O, P, X, Y, W>(const SpecDesc*, const int2*);
#define OSR_INST2T(X, Y, W)                                                            \
  OSR_INST2(1, 0, X, Y, W) OSR_INST2(2, 0, X, Y, W) OSR_INST2(3, 0, X, Y, W)           \
  OSR_INST2(1, 1, X, Y, W) OSR_INST2(2, 1, X, Y, W) OSR_INST2(3, 1, X, Y, W)
OSR_INST2T(8, 8, 4)
OSR_INST2T(16, 16, 4)
OSR_INST2T(16, 16, 8)
OSR_INST2T(32, 16, 4)
OSR_INST2T(32, 16, 8)

}  // namespace osr
