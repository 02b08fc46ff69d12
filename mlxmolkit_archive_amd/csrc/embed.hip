// Start geometries on the device for gfx950: seeded restraint embedding, one workgroup per
// conformer, so a batch's start geometries are made where the minimizer reads them.
//
// Stands in for the reference pipeline's device DG -> 4D->3D -> ETK stages
// (mlxmolkit/conformer_pipeline_v2.py:176-290), which are out of scope; the method is the
// package's host embedder (csrc/embed.c) moved onto the GPU:
//   * coordinates start uniformly in a 4D box of half-width 1.5 N^(1/3) + 1 A, drawn from a
//     counter-based splitmix64 stream per conformer (draw k is the generator's k-th output,
//     so lanes draw independently and the draws equal the host embedder's);
//   * restraint energy: equality springs 100 (d - d0)^2 for 1-2, 1-3 and ring targets, and
//     lower-bound walls 10 (d_min - d)^2 for every other pair closer than d_min;
//   * three relaxations by gradient descent with a 0.3 A per-atom step cap and an adaptive
//     step (x1.2 on an accepted step, x0.5 on a rejected one): 250 steps in 4D, 150 steps
//     with the fourth coordinate penalised (weight 2), then 200 steps in 3D after dropping it;
//   * N(0, noise) is added to every coordinate (Box-Muller on the same stream).
// Arithmetic is FP64. Gradients are summed in 64-bit fixed point (2^-32) in LDS and energies
// are reduced in a fixed order, so a conformer's result does not depend on thread timing.
// Coordinates sit in LDS as two planes of coordinate pairs (one conflict-free 16-byte read for two
// coordinates of consecutive atoms) and gradient sums as four planes. Active restraints are
// queued and evaluated in full waves (restraint_eg). 4,087 ragged conformers of up to 131 atoms:
// 14.7 ms, against 49.6 ms with the test and the evaluation in one loop, 8-byte reads and the
// conformers in molecule order (25.7 ms before the caller ordered them longest first).
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <string>

#include "mmff_hip.h"
#include "wave_reduce.h"

// error state and LDS bytes of the current device's workgroups (0: no device), in mmff_hip.hip
__attribute__((visibility("hidden"))) int mmffhip_set_error(int code, const char* msg);
__attribute__((visibility("hidden"))) int mmffhip_lds_limit();

namespace {

constexpr double EFX_MAGIC = 1572864.0;  // 1.5 * 2^20: FP64 sums in [2^20, 2^21) step 2^-32
constexpr double EFX_CAP = 524000.0;     // |v| < 2^19
constexpr double EFX_UNIT = 2.3283064365386962890625e-10;  // 2^-32

// v rounded to the nearest multiple of 2^-32, as a two's-complement integer (exact negation)
__device__ __forceinline__ unsigned long long efx(double v) {
  const double c = (v == v) ? fmin(fmax(v, -EFX_CAP), EFX_CAP) : 0.0;
  return (unsigned long long)(__double_as_longlong(c + EFX_MAGIC) - __double_as_longlong(EFX_MAGIC));
}
__device__ __forceinline__ double efx_val(unsigned long long a) { return (double)(long long)a * EFX_UNIT; }

// k-th output (k = 0, 1, ...) of splitmix64 seeded with `seed`, as a double in [0, 1)
__device__ __forceinline__ double unif(uint64_t seed, uint64_t k) {
  uint64_t z = seed + (k + 1) * 0x9E3779B97F4A7C15ULL;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  z ^= z >> 31;
  return (double)(z >> 11) * (1.0 / 9007199254740992.0);
}

struct EmbedMol {
  int n_atoms, r_off, n_restr;
};

// One restraint's energy and gradient (into g) at x: coordinate c of atom a is x[c >> 1][a]'s
// component c & 1, and word c * ps + a of g.
template <int DIM>
__device__ __forceinline__ double restraint(uint32_t ij, float dd, const double2* x01, const double2* x23,
                                            unsigned long long* g, int ps) {
  const int i = (int)(ij & 0xffffu), j = (int)(ij >> 16);
  const bool wall = dd < 0.0f;
  const double d0 = fabs((double)dd);
  const double2 a01 = x01[i], b01 = x01[j], a23 = x23[i], b23 = x23[j];
  const double dv[4] = {a01.x - b01.x, a01.y - b01.y, a23.x - b23.x, a23.y - b23.y};
  double d2 = 0.0;
#pragma unroll
  for (int c = 0; c < DIM; c++) d2 += dv[c] * dv[c];
  const double d = sqrt(d2 + 1e-12);
  if (wall && d >= d0) return 0.0;
  const double diff = d - d0, k = wall ? 10.0 : 100.0;
  const double f = 2.0 * k * diff / d;
#pragma unroll
  for (int c = 0; c < DIM; c++) {
    const unsigned long long q = efx(f * dv[c]);
    atomicAdd(&g[c * ps + i], q);
    atomicSub(&g[c * ps + j], q);
  }
  return k * diff * diff;
}

// Restraint energy (this lane's part) and gradient (into g, zeroed by the caller).
//
// Nine in ten restraints are walls whose pair is too far apart to touch, and telling so takes
// four FP64 differences, while an active restraint takes a square root, a division and eight
// LDS atomics. Testing and evaluating in one loop made every wave run the long path for its one
// or two active lanes. So a wave tests 64 restraints at a time (the next ones' loads already in
// flight), appends the active ones to a queue of its own in LDS in lane order, and evaluates the
// queue in full waves; the order is fixed, so the energy is deterministic. QUEUE is off for
// molecules whose coordinates leave no LDS for the queues.
constexpr int QCAP = 128;  // at most 63 left over plus 64 new
template <int NT, int DIM, bool QUEUE>
__device__ double restraint_eg(const uint32_t* rij, const float* rd, const EmbedMol& m, const double2* x01,
                               const double2* x23, unsigned long long* g, uint2* queue, int ps, double w4) {
  double e = 0.0;
  const unsigned n = (unsigned)m.n_restr, last = n - 1;
  const int lane = threadIdx.x & 63;
  if (n > 0) {
    unsigned t = threadIdx.x;
    int cnt = 0;  // queued restraints of this wave
    uint32_t ij = rij[min(t, last)];
    float dd = rd[min(t, last)];
    for (unsigned base = threadIdx.x - lane; base < n; base += NT) {
      const uint32_t nij = rij[min(t + NT, last)];
      const float ndd = rd[min(t + NT, last)];
      const int i = (int)(ij & 0xffffu), j = (int)(ij >> 16);
      const double2 a01 = x01[i], b01 = x01[j], a23 = x23[i], b23 = x23[j];
      const double dv[4] = {a01.x - b01.x, a01.y - b01.y, a23.x - b23.x, a23.y - b23.y};
      double d2 = 0.0;
#pragma unroll
      for (int c = 0; c < DIM; c++) d2 += dv[c] * dv[c];
      const double d0 = (double)dd;
      // an inactive wall costs no square root
      const bool active = t < n && !(dd < 0.0f && d2 + 1e-12 >= d0 * d0);
      if constexpr (QUEUE) {
        const unsigned long long mask = __ballot(active);
        const int pos = cnt + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0u));
        if (active) queue[pos] = make_uint2(ij, __float_as_uint(dd));
        cnt += __popcll(mask);
        if (cnt >= 64) {
          cnt -= 64;
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
          const uint2 r = queue[cnt + lane];
          e += restraint<DIM>(r.x, __uint_as_float(r.y), x01, x23, g, ps);
          __builtin_amdgcn_wave_barrier();
          __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
      } else if (active) {
        e += restraint<DIM>(ij, dd, x01, x23, g, ps);
      }
      ij = nij;
      dd = ndd;
      t += NT;
    }
    if (QUEUE) {
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (lane < cnt) {
        const uint2 r = queue[lane];
        e += restraint<DIM>(r.x, __uint_as_float(r.y), x01, x23, g, ps);
      }
    }
  }
  if (DIM == 4 && w4 > 0.0) {
    for (int a = threadIdx.x; a < m.n_atoms; a += NT) {
      const double w = x23[a].y;
      e += w4 * w * w;
      atomicAdd(&g[3 * ps + a], efx(2.0 * w4 * w));
    }
  }
  return e;
}

constexpr int EMB_RED = 16;  // doubles of the reduction buffer (2 phases x 2 waves used)

// A geometry and its gradient sums in LDS
struct Geom {
  double2 *x01, *x23;
  unsigned long long* g;
};

// Gradient descent with a per-atom step cap and an adaptive step; the two geometries swap on an
// accepted step (every lane takes the same branch: the sums are identical on all lanes).
template <int NT, int DIM, bool QUEUE>
__device__ void relax(const uint32_t* rij, const float* rd, const EmbedMol& m, Geom& cur, Geom& tri,
                      mmff::Reducer<NT, 1>& R, uint2* queue, int ps, double w4, int steps) {
  double step = 0.002;
  for (int c = 0; c < DIM; c++)
    for (int a = threadIdx.x; a < m.n_atoms; a += NT) cur.g[c * ps + a] = 0ull;
  __syncthreads();
  double e = R.sum(restraint_eg<NT, DIM, QUEUE>(rij, rd, m, cur.x01, cur.x23, cur.g, queue, ps, w4));
  for (int s = 0; s < steps; s++) {
    for (int a = threadIdx.x; a < m.n_atoms; a += NT) {
      double gv[4] = {0.0, 0.0, 0.0, 0.0}, gn = 0.0;
#pragma unroll
      for (int c = 0; c < DIM; c++) {
        gv[c] = efx_val(cur.g[c * ps + a]);
        gn += gv[c] * gv[c];
        tri.g[c * ps + a] = 0ull;
      }
      gn = sqrt(gn);
      double sc = step;
      if (gn * sc > 0.3) sc = 0.3 / gn;
      const double2 p = cur.x01[a], q = cur.x23[a];
      tri.x01[a] = make_double2(p.x - sc * gv[0], p.y - sc * gv[1]);
      tri.x23[a] = make_double2(q.x - sc * gv[2], DIM == 4 ? q.y - sc * gv[3] : q.y);
    }
    __syncthreads();
    const double et = R.sum(restraint_eg<NT, DIM, QUEUE>(rij, rd, m, tri.x01, tri.x23, tri.g, queue, ps, w4));
    if (et <= e) {
      const Geom t = cur;
      cur = tri;
      tri = t;
      e = et;
      step *= 1.2;
    } else {
      step = fmax(step * 0.5, 1e-7);
    }
  }
}

template <int NT, bool QUEUE>
__global__ void __launch_bounds__(NT) k_embed(const int32_t* desc, const uint32_t* rij, const float* rd,
                                              const int32_t* conf_mol, const int32_t* conf_off,
                                              const uint64_t* seeds, int n_confs, int max_atoms, float noise,
                                              float* x_out) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int c = blockIdx.x;
  if (c >= n_confs) return;
  const int ps = max_atoms;  // plane stride
  double* red = (double*)smem;
  Geom cur, tri;
  cur.x01 = (double2*)(red + EMB_RED);
  cur.x23 = cur.x01 + ps;
  tri.x01 = cur.x23 + ps;
  tri.x23 = tri.x01 + ps;
  cur.g = (unsigned long long*)(tri.x23 + ps);
  tri.g = cur.g + 4 * ps;
  uint2* queue = (uint2*)(tri.g + 4 * ps) + (threadIdx.x >> 6) * QCAP;
  mmff::Reducer<NT, 1> R{red, 0};
  const int32_t* d = desc + 4 * conf_mol[c];
  EmbedMol m{d[0], d[1], d[2]};
  const uint32_t* r_ij = rij + m.r_off;
  const float* r_d = rd + m.r_off;
  const uint64_t seed = seeds[c];
  const int n = m.n_atoms;
  const double box = 1.5 * cbrt((double)n) + 1.0;
  // draw k = 4a + c is coordinate c of atom a (the host embedder's order)
  for (int i = threadIdx.x; i < 4 * n; i += NT) {
    double2* p = (i & 2) ? cur.x23 : cur.x01;
    ((double*)(p + (i >> 2)))[i & 1] = (unif(seed, (uint64_t)i) * 2.0 - 1.0) * box;
  }
  relax<NT, 4, QUEUE>(r_ij, r_d, m, cur, tri, R, queue, ps, 0.0, 250);
  relax<NT, 4, QUEUE>(r_ij, r_d, m, cur, tri, R, queue, ps, 2.0, 150);
  for (int a = threadIdx.x; a < n; a += NT) cur.x23[a].y = 0.0;  // drop the fourth coordinate
  relax<NT, 3, QUEUE>(r_ij, r_d, m, cur, tri, R, queue, ps, 0.0, 200);
  float* o = x_out + conf_off[c];
  const uint64_t base = 4 * (uint64_t)n;
  for (int q = threadIdx.x; q < 3 * n; q += NT) {
    double u1 = unif(seed, base + 2 * (uint64_t)q), u2 = unif(seed, base + 2 * (uint64_t)q + 1);
    if (u1 < 1e-300) u1 = 1e-300;
    const double z = sqrt(-2.0 * log(u1)) * cos(6.283185307179586 * u2);
    const int a = q / 3, k = q - 3 * a;
    const double v = k == 0 ? cur.x01[a].x : k == 1 ? cur.x01[a].y : cur.x23[a].x;
    o[q] = (float)(v + (double)noise * z);
  }
}

constexpr int EMB_NT = 128;
// reduction buffer, two geometries and their gradient sums, and the waves' queues
size_t embed_lds(int max_atoms, bool queue) {
  return 8 * EMB_RED + (size_t)4 * max_atoms * (8 + 8 + 8 + 8) + (queue ? (size_t)(EMB_NT / 64) * QCAP * 8 : 0);
}

}  // namespace

extern "C" {

int mmffhip_embed(const int32_t* mol_desc, const uint32_t* restr_ij, const float* restr_d, const int32_t* conf_mol,
                  const int32_t* conf_off, const uint64_t* seeds, int32_t n_confs, int32_t max_atoms, float noise,
                  float* x_out, void* stream) {
  if (n_confs < 0 || max_atoms < 0) return mmffhip_set_error(MMFFHIP_ERR_ARG, "negative batch size");
  if (n_confs == 0) return MMFFHIP_OK;
  if (!mol_desc || !restr_ij || !restr_d || !conf_mol || !conf_off || !seeds || !x_out)
    return mmffhip_set_error(MMFFHIP_ERR_ARG, "mmffhip_embed: a required pointer is NULL");
  if (max_atoms < 1 || max_atoms > 65535)
    return mmffhip_set_error(MMFFHIP_ERR_SIZE, "mmffhip_embed: max_atoms must be in [1, 65535]");
  const size_t limit = (size_t)mmffhip_lds_limit();
  if (limit == 0) return mmffhip_set_error(MMFFHIP_ERR_DEVICE, "mmffhip_embed: no HIP device");
  const bool queue = embed_lds(max_atoms, true) <= limit;
  const size_t lds = embed_lds(max_atoms, queue);
  if (lds > limit)
    return mmffhip_set_error(MMFFHIP_ERR_SIZE, "mmffhip_embed: molecule too large for one workgroup's LDS");
  const auto kernel = queue ? k_embed<EMB_NT, true> : k_embed<EMB_NT, false>;
  if (lds > 65536 &&
      hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return mmffhip_set_error(MMFFHIP_ERR_HIP, "mmffhip_embed: cannot raise the LDS limit");
  hipLaunchKernelGGL(kernel, dim3(n_confs), dim3(EMB_NT), lds, (hipStream_t)stream, mol_desc, restr_ij, restr_d,
                     conf_mol, conf_off, seeds, n_confs, max_atoms, noise, x_out);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return mmffhip_set_error(MMFFHIP_ERR_HIP, (std::string("mmffhip_embed: ") + hipGetErrorString(e)).c_str());
  return MMFFHIP_OK;
}

}  // extern "C"
