// k_readback.hip -- fields and particles laid out for the host on the device, so that a
// read-back is one pass over the device arrays and one copy per host array.
//
// Fields: the reference's interleaved, guarded arrays (every cell its periodic image).
// Particles: the reference's arrays in upload order.  The rank of a particle is its pid
// while none is missing; when absorbing walls removed some, a bitmap of the live pids and
// the prefix of its word populations give it.  Both are bound by memory (the particles by
// their scattered stores) and by the copy to the host.  Against the device arrays copied
// whole and rearranged by the host: 100 steps of 128x128 with a read-back of its 262144
// particles 28.8 -> 4.9 ms, fields of 192^3 (170 MB) about 65 ms less.
#include "osr_device.hpp"
#include "osr_types.hpp"

namespace osr {

// Rows [row0, row0 + rows) of the guarded arrays (row: y and z of the array), 256 cells of
// 3 components per workgroup; E, B planar and periodic with extents nx, ny, nz.
struct FieldsOut {
  int nx, ny, nz;
  long long ncell;
  int ld0, ld1;       // array extents along x and y
  int gcl[3];         // lower guard cells
  long long row0, rows;
};

__global__ __launch_bounds__(256) void fields_out(const float* __restrict__ F,
                                                  float* __restrict__ out, FieldsOut a) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= a.rows * a.ld0) return;
  const long long row = a.row0 + i / a.ld0;
  const int ai = (int)(i % a.ld0), aj = (int)(row % a.ld1), ak = (int)(row / a.ld1);
  auto wrap = [](int v, int n) {
    const int w = v % n;
    return w < 0 ? w + n : w;
  };
  const long long c = wrap(ai - a.gcl[0], a.nx) +
                      (long long)a.nx * (wrap(aj - a.gcl[1], a.ny) +
                                         (long long)a.ny * wrap(ak - a.gcl[2], a.nz));
#pragma unroll
  for (int m = 0; m < 3; m++) out[3 * i + m] = F[m * a.ncell + c];
}

__global__ __launch_bounds__(256) void pids_mark(const SpecDesc* __restrict__ descs, int sid,
                                                 unsigned* __restrict__ bits) {
  const SpecDesc& d = descs[sid];
  const int base = d.off[blockIdx.x], n = d.cnt[blockIdx.x];
  for (int p = threadIdx.x; p < n; p += 256) {
    const uint32_t id = d.pid[base + p];
    atomicOr(&bits[id >> 5], 1u << (id & 31));
  }
}

constexpr int kPidWords = 2048;  // bitmap words per workgroup of the prefix kernels

// population of each group of kPidWords words
__global__ __launch_bounds__(256) void pids_count(const unsigned* __restrict__ bits, long long nw,
                                                  unsigned* __restrict__ sums) {
  __shared__ unsigned s[4];
  unsigned v = 0;
  for (int k = threadIdx.x; k < kPidWords; k += 256) {
    const long long w = (long long)blockIdx.x * kPidWords + k;
    if (w < nw) v += __popc(bits[w]);
  }
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) sums[blockIdx.x] = s[0] + s[1] + s[2] + s[3];
}

// live pids before each word: the groups before (summed here: at most 65536 groups) and the
// words before in the group
__global__ __launch_bounds__(256) void pids_prefix(const unsigned* __restrict__ bits, long long nw,
                                                   const unsigned* __restrict__ sums,
                                                   unsigned* __restrict__ pre) {
  constexpr int PER = kPidWords / 256;
  __shared__ unsigned s_before[4], s_wave[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned v = 0;
  for (unsigned b = threadIdx.x; b < blockIdx.x; b += 256) v += sums[b];
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if (lane == 0) s_before[wave] = v;
  const long long w0 = (long long)blockIdx.x * kPidWords + threadIdx.x * PER;
  unsigned own = 0;
  for (int k = 0; k < PER; k++)
    if (w0 + k < nw) own += __popc(bits[w0 + k]);
  unsigned inc = own;
  for (int o = 1; o < 64; o <<= 1) {
    const unsigned t = __shfl_up(inc, o, 64);
    if (lane >= o) inc += t;
  }
  if (lane == 63) s_wave[wave] = inc;
  __syncthreads();
  unsigned run = inc - own;
  for (int k = 0; k < 4; k++) run += s_before[k] + (k < wave ? s_wave[k] : 0u);
  for (int k = 0; k < PER; k++)
    if (w0 + k < nw) {
      pre[w0 + k] = run;
      run += __popc(bits[w0 + k]);
    }
}

// the particles of ranks [r0, r0 + n), one workgroup per tile; pre: null when ranks are pids
struct ParticlesOut {
  int* ix;
  float* x;
  float* u;
  float* q;
  const unsigned* bits;
  const unsigned* pre;
  uint32_t r0, n;
};

__global__ __launch_bounds__(256) void particles_out(const SpecDesc* __restrict__ descs, int sid,
                                                     ParticlesOut a) {
  const SpecDesc& d = descs[sid];
  const int base = d.off[blockIdx.x], cnt = d.cnt[blockIdx.x];
  const int D = d.g.dims;
  for (int p = threadIdx.x; p < cnt; p += 256) {
    const int s = base + p;
    const uint32_t id = d.pid[s];
    uint32_t r = id;
    if (a.pre) r = a.pre[id >> 5] + __popc(a.bits[id >> 5] & ((1u << (id & 31)) - 1u));
    if (r < a.r0 || r - a.r0 >= a.n) continue;
    const size_t o = r - a.r0;
    int c[3] = {0, 0, 0};
    if (D == 2)
      unpack2(d.cell[s], c[0], c[1]);
    else
      unpack3(d.cell[s], c[0], c[1], c[2]);
    for (int k = 0; k < D; k++) a.ix[D * o + k] = c[k] + 1;
    a.x[D * o] = d.x[s];
    a.x[D * o + 1] = d.y[s];
    if (D == 3) a.x[D * o + 2] = d.z[s];
    a.u[3 * o] = d.ux[s];
    a.u[3 * o + 1] = d.uy[s];
    a.u[3 * o + 2] = d.uz[s];
    a.q[o] = d.q[s];
  }
}

}  // namespace osr
