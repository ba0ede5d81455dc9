// k_smooth.hip -- current smoothing (digital filtering), vdf/os-vdf-smooth.f90.
//
// The filter is separable: one pass per direction with order n > 0, x before y before z
// (filter_2d :635-800, filter_3d :806-1100).  A pass replaces each value by
//   s(-n) o(i-n) + s(-n+1) o(i-n+1) + ... + s(n) o(i+n)
// summed left to right in FP32 with every product rounded (no contraction), o being the
// values before the pass -- the reference's single-precision arithmetic and order.
//
// Three forms:
//  * smooth2d: every direction of a 2D simulation in one launch;
//  * smooth_pass: one direction of a 3D simulation, planar interior arrays with periodic
//    index wraps (equal to the reference on the interior, whose guard cells hold the periodic
//    images after the current's boundary update, os-simulation.f03:650-657); the first
//    pass reads the folded fixed-point current and converts it as the E step would, later
//    passes read the previous output;
//  * smooth_vdf_pass: the stateless drop-in, a component-interleaved array with guard
//    cells, filtered exactly like smooth_vdf: cells closer than n to either end of a line
//    keep their values.
// The last two are memory-bound gathers along one direction: one thread per cell, consecutive
// threads on consecutive x, so every tap of a wave is a coalesced row segment.
#include "osr_device.hpp"
#include "osr_types.hpp"

namespace osr {

OSR_DEV int wrapn(int i, int n) {
  int w = i % n;
  return w < 0 ? w + n : w;
}

__global__ __launch_bounds__(256) void smooth_pass(const FieldDesc* __restrict__ fds,
                                                   const int2* __restrict__ work, int pass) {
  const int2 wk = work[blockIdx.x];
  const FieldDesc& fd = fds[wk.x];
  const GridDesc& g = fd.g;
  if (g.ctrl->halt >= 2 || pass >= fd.sm_np) return;
  const long long nc = g.ncell;
  const long long idx = (long long)wk.y * 256 + threadIdx.x;
  if (idx >= nc) return;
  const int nx = g.nx, ny = g.ny;
  const int dir = fd.sm_dir[pass], n = fd.sm_n[pass];
  const float* s = fd.sm_coef[pass] + 15;
  int ci, cj, ck;
  cell_xyz(g, idx, ci, cj, ck);
  int c, len;
  long long st;
  if (dir == 0) {
    c = ci;
    len = nx;
    st = 1;
  } else if (dir == 1) {
    c = cj;
    len = ny;
    st = nx;
  } else {
    c = ck;
    len = g.nz;
    st = (long long)nx * ny;
  }
  const long long row = idx - (long long)c * st;  // the line's first cell
  const unsigned long long* Jq = g.J;
  const float* P = fd.sm_buf[(pass + 1) & 1];  // previous pass's output
  float* dst = fd.sm_buf[pass & 1];
  const double jinv = g.jinv;
#pragma unroll
  for (int comp = 0; comp < 3; comp++) {
    const long long off = comp * nc + row;
    auto val = [&](int k) -> float {
      const long long id = off + (long long)wrapn(c + k, len) * st;
      return pass == 0 ? (float)((double)(long long)Jq[id] * jinv) : P[id];
    };
    float acc = val(-n) * s[-n];
    for (int k = -n + 1; k <= n; k++) acc = acc + val(k) * s[k];
    dst[comp * nc + idx] = acc;
  }
}

// Both passes of a 2D simulation.  A pass by smooth_pass is a launch whose threads wait for
// 2n+1 dependent loads of 8 bytes per component (10 us each at 300x200, 60000 cells, 2.9 MB);
// here a workgroup stages the cells of one component that its 32x16 tile needs (n more on each
// side; a wave loads a row, at most 62 cells, four rows in flight), filters the staged rows in
// x and the result in y from LDS: one launch and one read of the current, 7 us there.  A
// component per workgroup keeps three times the workgroups in flight on small grids.
constexpr int kSmX = 32, kSmY = 16, kSmN = 15;

__global__ __launch_bounds__(256) void smooth2d(const FieldDesc* __restrict__ fds) {
  constexpr int W = kSmX + 2 * kSmN, H = kSmY + 2 * kSmN;
  __shared__ float sa[H * W], sb[H * kSmX];
  const FieldDesc& fd = *fds;
  const GridDesc& g = fd.g;
  if (g.ctrl->halt >= 2) return;
  const int nx = g.nx, ny = g.ny;
  const long long nc = g.ncell;
  const int comp = (int)blockIdx.x % 3, tile = (int)blockIdx.x / 3;
  const int ntx = (nx + kSmX - 1) / kSmX;
  const int x0 = (tile % ntx) * kSmX, y0 = (tile / ntx) * kSmY;
  int n[2] = {0, 0};
  const float* s[2] = {nullptr, nullptr};
  for (int p = 0; p < fd.sm_np; p++) {
    if (fd.sm_dir[p] == 0) {
      n[0] = fd.sm_n[p];
      s[0] = fd.sm_coef[p] + 15;
    } else {
      n[1] = fd.sm_n[p];
      s[1] = fd.sm_coef[p] + 15;
    }
  }
  const int wd = kSmX + 2 * n[0], ht = kSmY + 2 * n[1];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int gx = wrap_any(x0 - n[0] + (lane < wd ? lane : wd - 1), nx);
  const long long base = comp * nc + gx;
  const unsigned long long* __restrict__ Jq = g.J + cur_copy(g);
  const float* __restrict__ Jp = (const float*)g.J;
  const double jinv = g.jinv;
  for (int r0 = wave; r0 < ht; r0 += 16) {
    float v[4];
    long long id[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int r = r0 + 4 * q;
      id[q] = base + (long long)nx * wrap_any(y0 - n[1] + (r < ht ? r : ht - 1), ny);
    }
    if (fd.sm_src == 0) {
      long long f[4];
#pragma unroll
      for (int q = 0; q < 4; q++) f[q] = (long long)Jq[id[q]];
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = (float)((double)f[q] * jinv);
    } else {
#pragma unroll
      for (int q = 0; q < 4; q++) v[q] = Jp[id[q]];
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
      if (r0 + 4 * q < ht && lane < wd) sa[(r0 + 4 * q) * W + lane] = v[q];
  }
  __syncthreads();
  const int col = threadIdx.x & (kSmX - 1), row = threadIdx.x / kSmX;  // 8 rows at a time
  for (int r0 = row; r0 < ht; r0 += 24) {
    const float* a[3];
    float acc[3];
#pragma unroll
    for (int q = 0; q < 3; q++) {
      a[q] = sa + (r0 + 8 * q < ht ? r0 + 8 * q : ht - 1) * W + col;
      acc[q] = a[q][0];
    }
    if (n[0] > 0) {
#pragma unroll
      for (int q = 0; q < 3; q++) acc[q] = acc[q] * s[0][-n[0]];
#pragma unroll 2
      for (int k = 1; k <= 2 * n[0]; k++)
#pragma unroll
        for (int q = 0; q < 3; q++) acc[q] = acc[q] + a[q][k] * s[0][k - n[0]];
    }
#pragma unroll
    for (int q = 0; q < 3; q++)
      if (r0 + 8 * q < ht) sb[(r0 + 8 * q) * kSmX + col] = acc[q];
  }
  __syncthreads();
  const float* b = sb + row * kSmX + col;
  float o[2] = {b[0], b[8 * kSmX]};
  if (n[1] > 0) {
    o[0] = o[0] * s[1][-n[1]];
    o[1] = o[1] * s[1][-n[1]];
#pragma unroll 2
    for (int k = 1; k <= 2 * n[1]; k++) {
      o[0] = o[0] + b[k * kSmX] * s[1][k - n[1]];
      o[1] = o[1] + b[(8 + k) * kSmX] * s[1][k - n[1]];
    }
  }
  float* __restrict__ dst = fd.Jf;
#pragma unroll
  for (int q = 0; q < 2; q++)
    if (x0 + col < nx && y0 + row + 8 * q < ny)
      dst[comp * nc + x0 + col + (long long)nx * (y0 + row + 8 * q)] = o[q];
}

struct SmoothCoef {
  float s[31];  // s(k) at [15 + k]
};

__global__ __launch_bounds__(256) void smooth_vdf_pass(const float* __restrict__ src,
                                                       float* __restrict__ dst, int fdim,
                                                       int ld0, int ld1, int ld2, int dir,
                                                       int n, SmoothCoef coef) {
  const long long total = (long long)fdim * ld0 * ld1 * ld2;
  const long long id = (long long)blockIdx.x * 256 + threadIdx.x;
  if (id >= total) return;
  const long long cell = id / fdim;
  int c, len;
  long long st;
  if (dir == 0) {
    c = (int)(cell % ld0);
    len = ld0;
    st = fdim;
  } else if (dir == 1) {
    c = (int)((cell / ld0) % ld1);
    len = ld1;
    st = (long long)fdim * ld0;
  } else {
    c = (int)(cell / ((long long)ld0 * ld1));
    len = ld2;
    st = (long long)fdim * ld0 * ld1;
  }
  if (c < n || c > len - 1 - n) {
    dst[id] = src[id];
    return;
  }
  const float* s = coef.s + 15;
  float acc = src[id - n * st] * s[-n];
  for (int k = -n + 1; k <= n; k++) acc = acc + src[id + k * st] * s[k];
  dst[id] = acc;
}

}  // namespace osr
