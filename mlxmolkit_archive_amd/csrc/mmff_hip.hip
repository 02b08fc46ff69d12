// Batched MMFF94 conformer minimization for gfx950 (MI355X): kernels + extern "C" ABI.
//
// Execution model (one conformer per workgroup, persistent grid with a work queue):
//   * positions, gradient accumulators and BFGS/L-BFGS vectors live in LDS;
//   * the dense inverse Hessian lives in a per-workgroup global slot as symmetric 4x4 blocks,
//     one per pair of row quads, each read once per iteration for both halves of H v (the
//     default), or in full storage read as coalesced 16-byte column quads, or in LDS as a
//     packed triangle with 16-byte aligned columns (n = 3N up to 264 at one workgroup per CU);
//   * term energies and gradients are FP32; each lane's energy is accumulated in FP64 and
//     reduced with wave shuffles + one LDS exchange, so the Armijo test and reported
//     energies are FP64 sums; gradients are summed exactly in 64-bit fixed point with LDS
//     atomics (order-independent, bit-reproducible).
// The control flow of each optimizer restates the reference kernel it replaces; the
// file:line citations are on each kernel.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <mutex>
#include <string>
#include <type_traits>

#include "bonded_windows.h"
#include "mmff_hip.h"
#include "mmff_terms.h"
#include "wave_reduce.h"

using namespace mmff;

namespace {

thread_local std::string g_last_error;

int fail(int code, const std::string& msg) {
  g_last_error = msg;
  return code;
}

#define HIP_TRY(expr)                                                                  \
  do {                                                                                 \
    hipError_t _e = (expr);                                                            \
    if (_e != hipSuccess)                                                              \
      return fail(MMFFHIP_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(_e)); \
  } while (0)

// ------------------------------------------------------------------------------------
// device-side view of the batch
struct KBatch {
  const int32_t* mol_desc;
  const uint32_t* bond_ij;
  const float2* bond_p;
  const uint2* ang_idx;
  const float2* ang_p;
  const uint2* sb_idx;
  const float4* sb_p;
  const float* sb_t0;
  const uint2* oop_idx;
  const float* oop_k;
  const uint2* tor_idx;
  const float4* tor_p;
  const uint32_t* pair_ij;
  const float4* pair_p;
  const int32_t* conf_mol;
  const int32_t* conf_off;
  int n_mols, n_confs, max_atoms;
};

KBatch to_kbatch(const mmffhip_batch* b) {
  KBatch k;
  k.mol_desc = b->mol_desc;
  k.bond_ij = b->bond_ij;
  k.bond_p = (const float2*)b->bond_p;
  k.ang_idx = (const uint2*)b->ang_idx;
  k.ang_p = (const float2*)b->ang_p;
  k.sb_idx = (const uint2*)b->sb_idx;
  k.sb_p = (const float4*)b->sb_p;
  k.sb_t0 = b->sb_t0;
  k.oop_idx = (const uint2*)b->oop_idx;
  k.oop_k = b->oop_k;
  k.tor_idx = (const uint2*)b->tor_idx;
  k.tor_p = (const float4*)b->tor_p;
  k.pair_ij = b->pair_ij;
  k.pair_p = (const float4*)b->pair_p;
  k.conf_mol = b->conf_mol;
  k.conf_off = b->conf_off;
  k.n_mols = b->n_mols;
  k.n_confs = b->n_confs;
  k.max_atoms = b->max_atoms;
  return k;
}

struct MolDesc {
  int n_atoms, bond_off, nb, ang_off, na, sb_off, nsb, oop_off, noop, tor_off, ntor, pair_off, npair;
};

__device__ __forceinline__ MolDesc load_desc(const int32_t* md) {
  MolDesc d;
  d.n_atoms = md[0];
  d.bond_off = md[1];
  d.nb = md[2];
  d.ang_off = md[3];
  d.na = md[4];
  d.sb_off = md[5];
  d.nsb = md[6];
  d.oop_off = md[7];
  d.noop = md[8];
  d.tor_off = md[9];
  d.ntor = md[10];
  d.pair_off = md[11];
  d.npair = md[12];
  return d;
}

// ------------------------------------------------------------------------------------
// 64-bit fixed-point gradient accumulation in LDS (scale 2^28). Each FP32 contribution is
// rounded once to a multiple of 2^-28, so the accumulated sum is the exact sum of the
// rounded contributions, independent of arrival order.
//
// Conversion: for |v| < 2^23 the double FX_MAGIC + v, FX_MAGIC = 1.5 * 2^24, lies in
// [2^24, 2^25), whose spacing is 2^-28, so the addition rounds v to the nearest multiple of
// 2^-28 (ties to even) and the low bits of the sum hold that multiple: bits(FX_MAGIC + v) -
// bits(FX_MAGIC) = round(v * 2^28) as a two's-complement integer. Round-to-nearest-even is
// symmetric, so to_fx(-v) == -to_fx(v) exactly. One conversion, one FP64 add and one 64-bit
// subtract, against the sign/split/recombine sequence of a truncating conversion.
constexpr double FX_MAGIC = 25165824.0;   // 1.5 * 2^24
constexpr float FX_CAP = 8388000.0f;      // |v| is capped just below 2^23
constexpr double FX_UNIT = 3.7252902984619140625e-09;  // 2^-28

__device__ __forceinline__ unsigned long long to_fx(float v) {
  // fmaxf / fminf return the non-NaN operand (one v_med3_f32), so a NaN contribution maps to
  // -FX_CAP: finite, and only ever met where the energy is NaN too
  const float c = fminf(fmaxf(v, -FX_CAP), FX_CAP);
  const double y = (double)c + FX_MAGIC;
  return (unsigned long long)(__double_as_longlong(y) - __double_as_longlong(FX_MAGIC));
}

__device__ __forceinline__ float from_fx(unsigned long long a) {
  return (float)((double)(long long)a * FX_UNIT);
}

// The accumulator of coordinate i = 3a + c is word i. Lanes updating consecutive atoms touch
// 8-byte words 24 bytes apart, and 3 is coprime to the 32 double banks, so they meet no bank
// twice; the three components are immediate offsets of one address (with three planes of N words
// each component took an address addition of its own, 6 of a pair's 95 vector instructions). The
// -g side of a pair term is an LDS subtract (ds_sub_u64) of the same integer, so it needs no
// negation.
template <bool G>
struct LdsAcc {
  unsigned long long* g;
  __device__ __forceinline__ void add(int a, float x, float y, float z) {
    if (G) {
      unsigned long long* p = g + 3 * a;
      atomicAdd(&p[0], to_fx(x));
      atomicAdd(&p[1], to_fx(y));
      atomicAdd(&p[2], to_fx(z));
    }
  }
  __device__ __forceinline__ static void sub(unsigned long long* p, unsigned long long v) {
    __hip_atomic_fetch_sub(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  // +g on atom a, -g on atom b: one conversion serves both
  __device__ __forceinline__ void add_pair(int a, int b, float x, float y, float z) {
    if (G) {
      const unsigned long long fx = to_fx(x), fy = to_fx(y), fz = to_fx(z);
      unsigned long long *p = g + 3 * a, *q = g + 3 * b;
      atomicAdd(&p[0], fx);
      atomicAdd(&p[1], fy);
      atomicAdd(&p[2], fz);
      sub(&q[0], fx);
      sub(&q[1], fy);
      sub(&q[2], fz);
    }
  }
};

// ------------------------------------------------------------------------------------
// energy (+ gradient) of one conformer whose positions are in LDS, spread over NT lanes.
// Term tables are read from global memory (L2-resident: shared by the molecule's
// conformers); each lane prefetches its next term's indices and parameters before it
// evaluates the current one, so table latency overlaps the term arithmetic.
// Returns this lane's FP64 energy partial.
struct TermData {
  uint32_t a, b;  // packed atom indices
  float4 p;       // parameters
  float q;        // fifth parameter (stretch-bend theta0)
};

// Pointers to one molecule's term tables (offsets folded in). Built either over the
// global batch tables or over a copy staged in LDS.
struct TView {
  const uint32_t* bond_ij;
  const float2* bond_p;
  const uint2* ang_idx;
  const float2* ang_p;
  const uint2* sb_idx;
  const float4* sb_p;
  const float* sb_t0;
  const uint2* oop_idx;
  const float* oop_k;
  const uint2* tor_idx;
  const float4* tor_p;
  const uint32_t* pair_ij;
  const float4* pair_p;
};

__device__ __forceinline__ TView global_view(const KBatch& B, const MolDesc& m) {
  TView v;
  v.bond_ij = B.bond_ij + m.bond_off;
  v.bond_p = B.bond_p + m.bond_off;
  v.ang_idx = B.ang_idx + m.ang_off;
  v.ang_p = B.ang_p + m.ang_off;
  v.sb_idx = B.sb_idx + m.sb_off;
  v.sb_p = B.sb_p + m.sb_off;
  v.sb_t0 = B.sb_t0 + m.sb_off;
  v.oop_idx = B.oop_idx + m.oop_off;
  v.oop_k = B.oop_k + m.oop_off;
  v.tor_idx = B.tor_idx + m.tor_off;
  v.tor_p = B.tor_p + m.tor_off;
  v.pair_ij = B.pair_ij + m.pair_off;
  v.pair_p = B.pair_p + m.pair_off;
  return v;
}

// bytes of one molecule's tables in the LDS staging layout
__host__ __device__ inline size_t table_lds_bytes(int nb, int na, int nsb, int noop, int ntor, int npair) {
  return 16 * (size_t)(ntor + nsb + npair) + 8 * (size_t)(2 * na + nsb + noop + ntor + nb) +
         4 * (size_t)(nb + nsb + noop + npair);
}

template <class T>
__device__ __forceinline__ void stage_copy(T* dst, const T* src, int count, int tid, int nt) {
  const int words = count * (int)(sizeof(T) / 4);
  uint32_t* d = (uint32_t*)dst;
  const uint32_t* s = (const uint32_t*)src;
  for (int i = tid; i < words; i += nt) d[i] = s[i];
}

// Copy a molecule's tables into LDS at `base` (16-byte aligned) and return a view of them.
// Without `pairs` only the bonded tables are copied and the view reads pairs from global
// memory (their loop streams them with loads one step ahead).
__device__ __forceinline__ TView stage_tables(const KBatch& B, const MolDesc& m, unsigned char* base, int tid,
                                              int nt, bool pairs) {
  TView v;
  const int npair = pairs ? m.npair : 0;
  unsigned char* p = base;
  auto take = [&](size_t bytes) {
    unsigned char* q = p;
    p += bytes;
    return q;
  };
  float4* tor_p = (float4*)take(16 * (size_t)m.ntor);
  float4* sb_p = (float4*)take(16 * (size_t)m.nsb);
  float4* pair_p = (float4*)take(16 * (size_t)npair);
  uint2* ang_idx = (uint2*)take(8 * (size_t)m.na);
  float2* ang_p = (float2*)take(8 * (size_t)m.na);
  uint2* sb_idx = (uint2*)take(8 * (size_t)m.nsb);
  uint2* oop_idx = (uint2*)take(8 * (size_t)m.noop);
  uint2* tor_idx = (uint2*)take(8 * (size_t)m.ntor);
  float2* bond_p = (float2*)take(8 * (size_t)m.nb);
  uint32_t* bond_ij = (uint32_t*)take(4 * (size_t)m.nb);
  float* sb_t0 = (float*)take(4 * (size_t)m.nsb);
  float* oop_k = (float*)take(4 * (size_t)m.noop);
  uint32_t* pair_ij = (uint32_t*)take(4 * (size_t)npair);
  stage_copy(tor_p, B.tor_p + m.tor_off, m.ntor, tid, nt);
  stage_copy(sb_p, B.sb_p + m.sb_off, m.nsb, tid, nt);
  stage_copy(pair_p, B.pair_p + m.pair_off, npair, tid, nt);
  stage_copy(ang_idx, B.ang_idx + m.ang_off, m.na, tid, nt);
  stage_copy(ang_p, B.ang_p + m.ang_off, m.na, tid, nt);
  stage_copy(sb_idx, B.sb_idx + m.sb_off, m.nsb, tid, nt);
  stage_copy(oop_idx, B.oop_idx + m.oop_off, m.noop, tid, nt);
  stage_copy(tor_idx, B.tor_idx + m.tor_off, m.ntor, tid, nt);
  stage_copy(bond_p, B.bond_p + m.bond_off, m.nb, tid, nt);
  stage_copy(bond_ij, B.bond_ij + m.bond_off, m.nb, tid, nt);
  stage_copy(sb_t0, B.sb_t0 + m.sb_off, m.nsb, tid, nt);
  stage_copy(oop_k, B.oop_k + m.oop_off, m.noop, tid, nt);
  stage_copy(pair_ij, B.pair_ij + m.pair_off, npair, tid, nt);
  v.bond_ij = bond_ij;
  v.bond_p = bond_p;
  v.ang_idx = ang_idx;
  v.ang_p = ang_p;
  v.sb_idx = sb_idx;
  v.sb_p = sb_p;
  v.sb_t0 = sb_t0;
  v.oop_idx = oop_idx;
  v.oop_k = oop_k;
  v.tor_idx = tor_idx;
  v.tor_p = tor_p;
  v.pair_ij = pairs ? pair_ij : B.pair_ij + m.pair_off;
  v.pair_p = pairs ? (const float4*)pair_p : B.pair_p + m.pair_off;
  return v;
}

__device__ __forceinline__ TermData load_term(const TView& V, int t, int c1, int c2, int c3, int c4, int c5) {
  TermData d;
  d.q = 0.f;
  if (t < c1) {
    d.a = V.bond_ij[t];
    d.b = 0;
    const float2 q = V.bond_p[t];
    d.p = make_float4(q.x, q.y, 0.f, 0.f);
  } else if (t < c2) {
    const int u = t - c1;
    const uint2 ix = V.ang_idx[u];
    d.a = ix.x;
    d.b = ix.y;
    const float2 q = V.ang_p[u];
    d.p = make_float4(q.x, q.y, 0.f, 0.f);
  } else if (t < c3) {
    const int u = t - c2;
    const uint2 ix = V.sb_idx[u];
    d.a = ix.x;
    d.b = ix.y;
    d.p = V.sb_p[u];
    d.q = V.sb_t0[u];
  } else if (t < c4) {
    const int u = t - c3;
    const uint2 ix = V.oop_idx[u];
    d.a = ix.x;
    d.b = ix.y;
    d.p = make_float4(V.oop_k[u], 0.f, 0.f, 0.f);
  } else if (t < c5) {
    const int u = t - c4;
    const uint2 ix = V.tor_idx[u];
    d.a = ix.x;
    d.b = ix.y;
    d.p = V.tor_p[u];
  } else {
    const int u = t - c5;
    d.a = V.pair_ij[u];
    d.b = 0;
    d.p = V.pair_p[u];
  }
  return d;
}

// One row of the pair table (its unused first parameter left out); 32-bit offsets from the
// (uniform) table bases
struct Pair {
  uint32_t ij;
  float eps, qq, ir;
};
__device__ __forceinline__ Pair load_pair(const TView& V, unsigned u) {
  const float* q = (const float*)((const char*)V.pair_p + 16u * u);
  return Pair{*(const uint32_t*)((const char*)V.pair_ij + 4u * u), q[1], q[2], q[3]};
}

// non-bonded pairs: two pairs per lane per step (independent dependency chains), the
// next two loaded while the current two are computed. The loads are unconditional (index
// clamped to the last pair; such duplicates are never used), so the wait before the
// current pairs' use leaves the next pairs' loads in flight. Every step but the last is full
// for all lanes, so the loop counts in scalar registers and masks nothing.
template <int FAM, bool G, int NT, bool EV>
__device__ __forceinline__ double eval_pairs(const TView& V, const MolDesc& m, const float* xs, LdsAcc<G>& acc,
                                             int diel) {
  if (m.npair <= 0) return 0.0;
  const unsigned np = (unsigned)m.npair, last = np - 1;
  double e = 0.0;
  // a pair's two parts are added in FP32 first (one rounding, as small as the parts' own), then
  // to the lane's FP64 sum
  auto term = [&](const Pair& p) {
    float ev = 0.f, ee = 0.f;
    t_pair<FAM, G, EV>(xs, acc, (int)(p.ij & 0xffff), (int)(p.ij >> 16), p.ir, p.eps, p.qq, diel, ev, ee);
    e += (double)(ev + ee);
  };
  unsigned u = threadIdx.x;
  Pair pa = load_pair(V, min(u, last)), pb = load_pair(V, min(u + NT, last));
  for (unsigned left = last / (2 * NT); left > 0; left--) {
    const Pair na = load_pair(V, min(u + 2 * NT, last)), nb = load_pair(V, min(u + 3 * NT, last));
    term(pa);
    term(pb);
    pa = na;
    pb = nb;
    u += 2 * NT;
  }
  if (u < np) term(pa);
  if (u + NT < np) term(pb);
  return e;
}

// PREF: load each bonded term's tables one step ahead (tables in global memory); with the
// tables in LDS the loads are short and the prefetch only holds registers.
// EV: the energies are used (otherwise only the gradient is).
template <int FAM, bool G, int NT, bool PREF, bool EV>
__device__ __forceinline__ double eval_terms(const TView& TV, const MolDesc& m, const float* xs,
                                             unsigned long long* gacc, int diel) {
  LdsAcc<G> acc{gacc};
  double e = 0.0;
  // bonded terms (one generic loop, next term prefetched when PREF)
  const int c1 = m.nb, c2 = c1 + m.na, c3 = c2 + m.nsb, c4 = c3 + m.noop, c5 = c4 + m.ntor;
  int t = threadIdx.x;
  TermData cur;
  if (PREF && t < c5) cur = load_term(TV, t, c1, c2, c3, c4, c5);
  while (t < c5) {
    const int tn = t + NT;
    TermData nxt;
    if (!PREF)
      cur = load_term(TV, t, c1, c2, c3, c4, c5);
    else if (tn < c5)
      nxt = load_term(TV, tn, c1, c2, c3, c4, c5);
    const int i0 = (int)(cur.a & 0xffff), i1 = (int)(cur.a >> 16);
    const int i2 = (int)(cur.b & 0xffff), i3 = (int)(cur.b >> 16);
    if (t < c1) {
      e += t_bond<FAM, G>(xs, acc, i0, i1, cur.p.x, cur.p.y);
    } else if (t < c2) {
      e += t_angle<FAM, G>(xs, acc, i0, i1, i2, cur.p.x, cur.p.y, i3 != 0);
    } else if (t < c3) {
      e += t_strbend<FAM, G>(xs, acc, i0, i1, (int)cur.b, cur.p.x, cur.p.y, cur.p.z, cur.p.w, cur.q);
    } else if (t < c4) {
      e += t_oop<FAM, G>(xs, acc, i0, i1, i2, i3, cur.p.x);
    } else {
      e += t_torsion<FAM, G>(xs, acc, i0, i1, i2, i3, cur.p.x, cur.p.y, cur.p.z);
    }
    if (PREF) cur = nxt;
    t = tn;
  }
  return e + eval_pairs<FAM, G, NT, EV>(TV, m, xs, acc, diel);
}

// The evaluation of the single points, the descent and the lock-step engine. Their workgroups have
// 256 threads, or 1,024 for batches of at most one conformer per CU, and a conformer's results do
// not depend on which: an energy is the sum over SUM_GROUPS groups of 256 lanes, each with a share
// of the terms of its own. A workgroup of 256 threads does one group after another and adds up a
// lane's four sums as it goes; one of 1,024 does the four at once and adds them in the same order
// in LDS (combine_groups). (Gradient sums are exact in any order.)
//
// Bonded terms go to the groups' 16 waves in tasks of 64 terms of one type, the heaviest types
// first and the waves taken back and forth, so no wave runs several types' code for parts of its
// lanes and the waves finish together. A task takes every T-th term of its type (T tasks), because
// neighbouring terms share atoms and their lanes' atomics would queue for the same LDS words. The
// minimizers that compare energies trial by trial use bonded_tasks below. A group's pairs are a
// quarter of the list, so one group after another is one walk over it.
// 12,139 ragged MEGA energies and gradients: generic loop 143 us, tasks of consecutive terms 123, of
// spread terms 103, without the sums of kinds 97.5; the Barzilai-Borwein descent of 1,000
// conformers: 6.08, 4.59, 4.00 ms, and again 4.00 with the sums by groups; the lock-step L-BFGS: 7.00,
// 6.28, 6.26 ms.
constexpr int SUM_LANES = 256, SUM_GROUPS = 4;

// A lane's energy sums: bonded terms, pairs, and each kind of term when PT
template <bool PT>
struct LaneSums {
  double b = 0.0, p = 0.0, kind[PT ? 7 : 1] = {};
};

// SEP: a pair's two parts go to FP64 sums of their own; otherwise they are added in FP32 first, as in
// eval_pairs
template <int FAM, bool G, bool SEP, bool PT, int NT>
__device__ __forceinline__ LaneSums<PT> eval_tasks(const TView& V, const MolDesc& m, const float* xs,
                                                   unsigned long long* gacc, int diel, uint32_t mask) {
  static_assert(NT == SUM_LANES || NT == SUM_LANES * SUM_GROUPS, "one group after another, or all at once");
  static_assert(SEP || !PT, "kinds are summed apart");
  constexpr bool ALL = NT == SUM_LANES;
  constexpr int GW = SUM_LANES / 64, NW = GW * SUM_GROUPS;
  LdsAcc<G> acc{gacc};
  LaneSums<PT> sum;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h0 = ALL ? 0 : w / GW, h1 = ALL ? SUM_GROUPS : h0 + 1, wg = w % GW;
  // first task of each type after the torsions
  const int t1 = (m.ntor + 63) >> 6, t2 = t1 + ((m.nsb + 63) >> 6), t3 = t2 + ((m.na + 63) >> 6),
            t4 = t3 + ((m.noop + 63) >> 6), t5 = t4 + ((m.nb + 63) >> 6);
  auto tor = [&](int u) {
    const uint2 ix = V.tor_idx[u];
    const float4 p = V.tor_p[u];
    return t_torsion<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff), (int)(ix.y >> 16),
                             p.x, p.y, p.z);
  };
  auto sb = [&](int u) {
    const uint2 ix = V.sb_idx[u];
    const float4 p = V.sb_p[u];
    return t_strbend<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)ix.y, p.x, p.y, p.z, p.w, V.sb_t0[u]);
  };
  auto ang = [&](int u) {
    const uint2 ix = V.ang_idx[u];
    const float2 p = V.ang_p[u];
    return t_angle<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff), p.x, p.y,
                           (ix.y >> 16) != 0);
  };
  auto oop = [&](int u) {
    const uint2 ix = V.oop_idx[u];
    return t_oop<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff), (int)(ix.y >> 16),
                         V.oop_k[u]);
  };
  auto bond = [&](int u) {
    const uint32_t ij = V.bond_ij[u];
    const float2 p = V.bond_p[u];
    return t_bond<FAM, G>(xs, acc, (int)(ij & 0xffff), (int)(ij >> 16), p.x, p.y);
  };
  // a wave's tasks of a group: every NW-th from its first
  auto first_task = [&](int h) { return GW * h + ((h & 1) ? GW - 1 - wg : wg); };
  int h = h0, t = first_task(h);
  double e = 0.0;
  // task t of kind c, whose tasks are first .. end - 1 and whose terms are n
  auto one = [&](int c, int first, int end, int n, auto term, double& k) {
    const int u = lane * (end - first) + (t - first);
    if ((mask >> c & 1u) && u < n) {
      const float v = term(u);
      e += v;
      if (PT) k += v;
    }
  };
  auto next_group = [&]() {
    sum.b += e;
    e = 0.0;
    if (++h < h1) t = first_task(h);
  };
  if constexpr (PT) {
#pragma unroll 1
    while (t < t5) {
      // a loop for each kind, so that one sum of kinds is in the making at a time
      auto all = [&](int c, int first, int end, int n, auto term) {
        double k = 0.0;
        for (; t < end; t += NW) one(c, first, end, n, term, k);
        sum.kind[c] += k;
      };
      all(4, 0, t1, m.ntor, tor);
      all(2, t1, t2, m.nsb, sb);
      all(1, t2, t3, m.na, ang);
      all(3, t3, t4, m.noop, oop);
      all(0, t4, t5, m.nb, bond);
      next_group();
    }
  } else {
    // one loop over the groups' tasks and one over their pairs below (a loop in a loop each: the
    // descent of 1,000 conformers 4.07 ms, so 4.05)
    double k;
    while (t < t5) {
      if (t < t1) one(4, 0, t1, m.ntor, tor, k);
      else if (t < t2) one(2, t1, t2, m.nsb, sb, k);
      else if (t < t3) one(1, t2, t3, m.na, ang, k);
      else if (t < t4) one(3, t3, t4, m.noop, oop, k);
      else one(0, t4, t5, m.nb, bond, k);
      t += NW;
      if (t >= t5) next_group();
    }
  }
  if (!(mask & 96u) || m.npair <= 0) return sum;
  // eval_pairs' walk, two pairs per lane and step
  constexpr unsigned STEP = 2 * SUM_LANES;
  const unsigned np = (unsigned)m.npair, last = np - 1;
  auto row = [&](unsigned u) { return load_pair(V, min(u, last)); };
  const float ke = (mask & 32u) ? 1.0f : 0.0f, kq = (mask & 64u) ? 1.0f : 0.0f;
  // group h has the steps h * per .. (h + 1) * per
  double sv = 0.0, se = 0.0;
  auto term = [&](const Pair& p) {
    float ev = 0.f, ee = 0.f;
    t_pair<FAM, G, true>(xs, acc, (int)(p.ij & 0xffff), (int)(p.ij >> 16), p.ir, ke * p.eps, kq * p.qq, diel, ev, ee);
    if (SEP) {
      sv += ev;
      se += ee;
    } else {
      sv += (double)(ev + ee);
    }
  };
  auto close = [&]() {  // a group's sums are complete
    sum.p += SEP ? sv + se : sv;
    if (PT) {
      sum.kind[5] += sv;
      sum.kind[6] += se;
    }
    sv = se = 0.0;
  };
  const unsigned steps = last / STEP + 1, per = (steps + SUM_GROUPS - 1) / SUM_GROUPS;
  unsigned s = min(h0 * per, steps);
  const unsigned end = min(h1 * per, steps), full = min(end, steps - 1);
  if (s < end) {
    unsigned u = s * STEP + (threadIdx.x & (SUM_LANES - 1)), left = per;  // steps left of this group
    Pair pa = row(u), pb = row(u + SUM_LANES);
    for (; s < full; s++) {
      const Pair na = row(u + STEP), nb = row(u + STEP + SUM_LANES);
      term(pa);
      term(pb);
      pa = na;
      pb = nb;
      u += STEP;
      if (ALL && --left == 0) {
        close();
        left = per;
      }
    }
    if (s < end) {  // the list's last step
      if (u < np) term(pa);
      if (u + SUM_LANES < np) term(pb);
    }
    close();
  }
  return sum;
}

// The groups' sums of K values, for the lanes of the first group (the others' are left as they
// are). buf: LDS for `room` >= 1 values of EX_WORDS doubles at a time; everybody is done with
// its earlier contents.
constexpr int EX_WORDS = SUM_LANES * (SUM_GROUPS - 1);
template <int NT, int K>
__device__ __forceinline__ void combine_groups(double (&v)[K], double* buf, int room) {
  if constexpr (NT > SUM_LANES) {
    const int t = (int)threadIdx.x;
    for (int k0 = 0; k0 < K; k0 += room) {
      if (k0 > 0) __syncthreads();
#pragma unroll
      for (int k = 0; k < K; k++)
        if (t >= SUM_LANES && k >= k0 && k < k0 + room) buf[(k - k0) * EX_WORDS + t - SUM_LANES] = v[k];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < K; k++)
        if (t < SUM_LANES && k >= k0 && k < k0 + room) {
          const double* b = buf + (k - k0) * EX_WORDS + t;
          v[k] = ((v[k] + b[0]) + b[SUM_LANES]) + b[2 * SUM_LANES];
        }
    }
  }
}
// The energy, on every lane; includes a barrier behind the evaluation
template <int NT, bool PT, class Red>
__device__ __forceinline__ double group_energy(const LaneSums<PT>& s, double* buf, int room, Red& R) {
  double v[2] = {s.b, s.p};
  combine_groups<NT>(v, buf, room);
  return R.sum(v[0] + v[1]);
}
// LDS bytes of an area of at least `bytes` that serves as combine_groups' buffer too: K values at
// once, or one if that does not fit beside `rest` other bytes
size_t ex_area(int nt, size_t bytes, int K, size_t rest, size_t limit) {
  if (nt == SUM_LANES) return bytes;
  const size_t one = EX_WORDS * sizeof(double);
  return std::max(bytes, rest + std::max(bytes, K * one) <= limit ? K * one : one);
}

// The bonded terms of eval_tasks for the minimizers that compare energies trial by trial, with
// the energy bits of eval_terms' generic loop over NT lanes: every task writes its terms' FP32
// energies to eb (eb_n >= BONDED_WINDOW_MIN floats of LDS) under eval_terms' numbering, and lane t < NT adds up
// numbers t, t + NT, ... in order. Gradient sums are exact in any order, so a task is free to take
// every T-th term of its type (T tasks): terms follow their central atoms in the tables, and 64
// consecutive ones send up to 27 lanes' atomics to one LDS word. With the generic loop the bonded
// terms took 49% of the n <= 96 launch of a 100,000-conformer ragged batch (pairs 14%), 39% for
// n <= 192, 29% for n <= 354 and 15% above; tasks of consecutive terms changed the batch from
// 1,095 to 1,084 ms, tasks of spread terms to 999 ms, and 8% of the n <= 96 launch (3% for
// n <= 354) is left to conflicts.
// Terms that eb cannot hold at once go in several windows of consecutive terms. The last window's
// sums are left to the caller, after a barrier of its own: ordered_sum with the returned bounds.
struct Window {
  int s, end;
};
template <int NT>
__device__ __forceinline__ void ordered_sum(double& e, const float* eb, Window w, int t) {
  if (t < NT)
    for (int k = w.s + ((t - w.s) % NT + NT) % NT; k < w.end; k += NT) e += eb[k - w.s];
}
template <int FAM, bool G, bool EV, int NT, int NR>
__device__ __forceinline__ Window bonded_tasks(const TView& V, const MolDesc& m, const float* xs, LdsAcc<G>& acc,
                                               float* eb, int eb_n, double& e) {
  constexpr int NW = NR / 64;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // eval_terms' numbering: bonds, angles, stretch-bends, out-of-planes, torsions
  const int c1 = m.nb, c2 = c1 + m.na, c3 = c2 + m.nsb, c4 = c3 + m.noop, c5 = c4 + m.ntor;
  const int t1 = (m.ntor + 63) >> 6, t2 = t1 + ((m.nsb + 63) >> 6), t3 = t2 + ((m.na + 63) >> 6),
            t4 = t3 + ((m.noop + 63) >> 6), t5 = t4 + ((m.nb + 63) >> 6);
  Window win{0, c5};
  const bool one = !EV || c5 <= eb_n;
  for (;;) {
    win.end = EV ? bonded_window_end({0, c1, c2, c3, c4, c5}, win.s, eb_n) : c5;
    for (int k = 0; k * NW < t5; k++) {
      const int t = (k & 1) ? (k + 1) * NW - 1 - w : k * NW + w;
      auto mine = [&](int first, int end, int base, int n, int& u) {
        if (one) {
          u = lane * (end - first) + (t - first);
          return u < n;
        }
        u = (t - first) * 64;
        const bool in = base + u >= win.s && base + u < win.end;
        u += lane;
        return in && u < n;
      };
      auto put = [&](int i, float v) {
        if (EV) eb[i - win.s] = v;
      };
      int u;
      if (t < t1) {
        if (mine(0, t1, c4, m.ntor, u)) {
          const uint2 ix = V.tor_idx[u];
          const float4 p = V.tor_p[u];
          put(c4 + u, t_torsion<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff),
                                        (int)(ix.y >> 16), p.x, p.y, p.z));
        }
      } else if (t < t2) {
        if (mine(t1, t2, c2, m.nsb, u)) {
          const uint2 ix = V.sb_idx[u];
          const float4 p = V.sb_p[u];
          put(c2 + u, t_strbend<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)ix.y, p.x, p.y, p.z,
                                        p.w, V.sb_t0[u]));
        }
      } else if (t < t3) {
        if (mine(t2, t3, c1, m.na, u)) {
          const uint2 ix = V.ang_idx[u];
          const float2 p = V.ang_p[u];
          put(c1 + u, t_angle<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff), p.x,
                                      p.y, (ix.y >> 16) != 0));
        }
      } else if (t < t4) {
        if (mine(t3, t4, c3, m.noop, u)) {
          const uint2 ix = V.oop_idx[u];
          put(c3 + u, t_oop<FAM, G>(xs, acc, (int)(ix.x & 0xffff), (int)(ix.x >> 16), (int)(ix.y & 0xffff),
                                    (int)(ix.y >> 16), V.oop_k[u]));
        }
      } else if (t < t5) {
        if (mine(t4, t5, 0, m.nb, u)) {
          const uint32_t ij = V.bond_ij[u];
          const float2 p = V.bond_p[u];
          put(u, t_bond<FAM, G>(xs, acc, (int)(ij & 0xffff), (int)(ij >> 16), p.x, p.y));
        }
      }
    }
    if (win.end >= c5) return win;
    __syncthreads();
    ordered_sum<NT>(e, eb, win, (int)threadIdx.x);
    __syncthreads();
    win.s = win.end;
  }
}

// eval_terms with the bonded terms as bonded_tasks: the same results
template <int FAM, bool G, bool EV, int NT>
__device__ __forceinline__ double eval_ordered(const TView& V, const MolDesc& m, const float* xs,
                                               unsigned long long* gacc, int diel, float* eb, int eb_n) {
  LdsAcc<G> acc{gacc};
  double e = 0.0;
  const Window win = bonded_tasks<FAM, G, EV, NT, NT>(V, m, xs, acc, eb, eb_n, e);
  const double pairs = eval_pairs<FAM, G, NT, EV>(V, m, xs, acc, diel);
  if (!EV) return 0.0;
  __syncthreads();
  ordered_sum<NT>(e, eb, win, (int)threadIdx.x);
  return e + pairs;
}

// eval_ordered with HELP times as many threads as the NT lanes whose energy sums it forms: every
// thread evaluates bonded terms and pairs (in steps of NT), and the pairs' FP32 energies go
// through LDS too, two rounds of them in ring. Returns the lane's energy partial; zero for the
// threads past NT.
constexpr int HELP_STEPS = 2;  // pairs per thread and round
template <int NT>
constexpr size_t help_ring_floats(int help) {
  return 2 * (size_t)HELP_STEPS * help * NT;
}
template <int FAM, bool G, bool EV, int NT, int HELP>
__device__ __forceinline__ double eval_help(const TView& V, const MolDesc& m, const float* xs,
                                            unsigned long long* gacc, int diel, float* eb, int eb_n, float* ring) {
  constexpr int NR = NT * HELP, K = HELP_STEPS * HELP;
  LdsAcc<G> acc{gacc};
  double e = 0.0;
  const Window win = bonded_tasks<FAM, G, EV, NT, NR>(V, m, xs, acc, eb, eb_n, e);
  // pairs: in round r thread (h, t) takes pairs (K r + HELP_STEPS h + j) NT + t
  const int np = m.npair, last = np - 1;
  const int t = threadIdx.x & (NT - 1), h = threadIdx.x / NT;
  const int rounds = np > 0 ? (np - 1) / (K * NT) + 1 : 0;
  double pairs = 0.0;
  uint32_t ij[HELP_STEPS];
  float4 pp[HELP_STEPS];
  const int u0 = HELP_STEPS * h * NT + t;
  if (rounds > 0) {
#pragma unroll
    for (int j = 0; j < HELP_STEPS; j++) {
      const unsigned u = (unsigned)min(u0 + j * NT, last);
      ij[j] = V.pair_ij[u];
      pp[j] = V.pair_p[u];
    }
  }
  if (EV && rounds == 0) __syncthreads();  // the bonded energies
  for (int r = 0; r < rounds; r++) {
    uint32_t nij[HELP_STEPS];
    float4 npp[HELP_STEPS];
    const int u1 = u0 + r * K * NT;
#pragma unroll
    for (int j = 0; j < HELP_STEPS; j++) {
      const unsigned u = (unsigned)min(u1 + (K + j) * NT, last);
      nij[j] = V.pair_ij[u];
      npp[j] = V.pair_p[u];
    }
    float* row = ring + (r & 1) * K * NT;
#pragma unroll
    for (int j = 0; j < HELP_STEPS; j++) {
      if (u1 + j * NT < np) {
        float ev = 0.f, ee = 0.f;
        t_pair<FAM, G, EV>(xs, acc, (int)(ij[j] & 0xffff), (int)(ij[j] >> 16), pp[j].w, pp[j].y, pp[j].z, diel, ev, ee);
        if (EV) row[(HELP_STEPS * h + j) * NT + t] = ev + ee;
      }
      ij[j] = nij[j];
      pp[j] = npp[j];
    }
    if (EV) {
      __syncthreads();  // this round's energies; the other half is free, its readers are past it
      if (h == 0) {
#pragma unroll
        for (int k = 0; k < K; k++)
          if ((r * K + k) * NT + t < np) pairs += (double)row[k * NT + t];
      }
    }
  }
  if (!EV) return 0.0;
  ordered_sum<NT>(e, eb, win, (int)threadIdx.x);
  return e + pairs;
}

// ------------------------------------------------------------------------------------
// four consecutive elements (t, j..j+3) of a symmetric matrix in padded packed storage
// (column c at pcol(c), cb = pcol(t), pj = pcol(j)), with the matching gradient entries
__device__ __forceinline__ void hrow_load4(const float* H, const float* gv, int t, int cb, int j, int pj,
                                           float (&h)[4], float (&w)[4]) {
  const int p1 = pj + ((j + 4) & ~3), p2 = p1 + ((j + 5) & ~3), p3 = p2 + ((j + 6) & ~3);
  h[0] = H[j <= t ? cb + j : pj + t];
  h[1] = H[j + 1 <= t ? cb + j + 1 : p1 + t];
  h[2] = H[j + 2 <= t ? cb + j + 2 : p2 + t];
  h[3] = H[j + 3 <= t ? cb + j + 3 : p3 + t];
  w[0] = gv[j];
  w[1] = gv[j + 1];
  w[2] = gv[j + 2];
  w[3] = gv[j + 3];
}

// one row of a column quad of the full Hessian gains a pending rank-2 update: column t's
// element gains ux[t] s + uy[t] h, with w = {s, h} of the row
__device__ __forceinline__ void hquad_upd(float4& h, float2 w, const float (&ux)[4], const float (&uy)[4]) {
  h.x = fmaf(uy[0], w.y, fmaf(ux[0], w.x, h.x));
  h.y = fmaf(uy[1], w.y, fmaf(ux[1], w.x, h.y));
  h.z = fmaf(uy[2], w.y, fmaf(ux[2], w.x, h.z));
  h.w = fmaf(uy[3], w.y, fmaf(ux[3], w.x, h.w));
}

// accumulate the row's gradient entry g into the quad's dot products
__device__ __forceinline__ void hquad_dot(const float4& h, float g, float (&a)[4]) {
  a[0] = fmaf(h.x, g, a[0]);
  a[1] = fmaf(h.y, g, a[1]);
  a[2] = fmaf(h.z, g, a[2]);
  a[3] = fmaf(h.w, g, a[3]);
}

// Rows [j, j1) of a column quad of the full Hessian (row r at base[r * nq]): accumulate
// H g into a, with H the stored rows plus the NU oldest pending rank-2 updates (update k:
// row vectors {s, h} in S[k], column coefficients cx[k], cy[k]). When all NPM slots are
// pending the updates are added to each element, oldest first, and the rows are written
// back. Otherwise the stored rows are only read, and the updates' part of H g is left as two
// dot products per update over these rows in lr (s.g, h.g), which the caller combines with
// the column coefficients after summing the quad's lanes. HQ rows are loaded together.
template <int HQ, int NU, int NPM>
__device__ __forceinline__ void hquad_rows(float4* base, int nq, int j, int j1, const float* gv,
                                           const float2* const (&S)[NPM], const float (&cx)[NPM][4],
                                           const float (&cy)[NPM][4], float (&a)[4], float (&lr)[2][NPM]) {
  constexpr bool FLUSH = NU == NPM;
  for (; j + HQ - 1 < j1; j += HQ) {
    float4 h[HQ];
#pragma unroll
    for (int u = 0; u < HQ; u++) h[u] = base[(size_t)(j + u) * nq];
#pragma unroll
    for (int u = 0; u < HQ; u++) {
      const float g = gv[j + u];
#pragma unroll
      for (int k = 0; k < NU; k++) {
        const float2 w = S[k][j + u];
        if (FLUSH) {
          hquad_upd(h[u], w, cx[k], cy[k]);
        } else {
          lr[0][k] = fmaf(w.x, g, lr[0][k]);
          lr[1][k] = fmaf(w.y, g, lr[1][k]);
        }
      }
      hquad_dot(h[u], g, a);
    }
    if (FLUSH) {
#pragma unroll
      for (int u = 0; u < HQ; u++) base[(size_t)(j + u) * nq] = h[u];
    }
  }
  for (; j < j1; j++) {
    float4 h = base[(size_t)j * nq];
    const float g = gv[j];
#pragma unroll
    for (int k = 0; k < NU; k++) {
      const float2 w = S[k][j];
      if (FLUSH) {
        hquad_upd(h, w, cx[k], cy[k]);
      } else {
        lr[0][k] = fmaf(w.x, g, lr[0][k]);
        lr[1][k] = fmaf(w.y, g, lr[1][k]);
      }
    }
    hquad_dot(h, g, a);
    if (FLUSH) base[(size_t)j * nq] = h;
  }
}

// hquad_rows for the run-time count of pending updates (0..NPM)
template <int HQ, int NPM, int NU = NPM>
__device__ __forceinline__ void hquad_dispatch(int npend, float4* base, int nq, int j, int j1, const float* gv,
                                               const float2* const (&S)[NPM], const float (&cx)[NPM][4],
                                               const float (&cy)[NPM][4], float (&a)[4], float (&lr)[2][NPM]) {
  if constexpr (NU == 0) {
    hquad_rows<HQ, 0, NPM>(base, nq, j, j1, gv, S, cx, cy, a, lr);
  } else {
    if (npend == NU)
      hquad_rows<HQ, NU, NPM>(base, nq, j, j1, gv, S, cx, cy, a, lr);
    else
      hquad_dispatch<HQ, NPM, NU - 1>(npend, base, nq, j, j1, gv, S, cx, cy, a, lr);
  }
}

// Row groups [ka, kb) (rows 4k..4k+3) of one column of the padded packed matrix gain
// alpha_i s + beta_i h (AB[i] = {alpha_i, beta_i}, u = {s, h} of the column); rows past the
// column's end are padding and never read as matrix elements.
__device__ __forceinline__ void hcol_update4(float* col, const float2* AB, float2 u, int ka, int kb) {
  float4* c4 = (float4*)col;
  const float4* ab4 = (const float4*)AB;
  for (int k = ka; k < kb; k++) {
    float4 h = c4[k];
    const float4 a01 = ab4[2 * k], a23 = ab4[2 * k + 1];
    h.x = fmaf(a01.y, u.y, fmaf(a01.x, u.x, h.x));
    h.y = fmaf(a01.w, u.y, fmaf(a01.z, u.x, h.y));
    h.z = fmaf(a23.y, u.y, fmaf(a23.x, u.x, h.z));
    h.w = fmaf(a23.w, u.y, fmaf(a23.z, u.x, h.w));
    c4[k] = h;
  }
}

constexpr int RED_WORDS = 2 * (SUM_LANES / 64) * 8;  // doubles of a Reducer<SUM_LANES>

// ------------------------------------------------------------------------------------
// Kernel: single-point energy / gradient / per-term energies, one workgroup per conformer.
// Replaces mmff_energy_grad_metal(_mega) (mmff_metal_kernel.py:713-775); the TG family is
// what the nk kernel evaluates (mmff_bfgs_header.metal).
// The groups' sums meet in LDS behind the positions (xs_bytes), room values at a time, or where the
// positions were when room is 0 (xs_bytes then hold one value at least)
// Registers let 8 (TG) and 6 (MEGA) waves onto a SIMD, 7 and 5 with kinds.
template <int FAM, bool PT, int NT>
__global__ void __launch_bounds__(NT) k_energy_grad(KBatch B, const float* __restrict__ x, double* e_out,
                                                    double* e_terms, float* g_out, uint32_t mask, int diel,
                                                    int xs_bytes, int room) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int c = blockIdx.x;
  if (c >= B.n_confs) return;
  double* red = (double*)smem;
  unsigned long long* gacc = (unsigned long long*)(red + RED_WORDS);
  const int mx = 3 * B.max_atoms;
  float* xs = (float*)(gacc + mx);
  const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
  const int n = 3 * m.n_atoms;
  const int off = B.conf_off[c];
  for (int i = threadIdx.x; i < n; i += NT) xs[i] = x[off + i];
  for (int i = threadIdx.x; i < n; i += NT) gacc[i] = 0ull;
  __syncthreads();
  Reducer<SUM_LANES, 8, (NT > SUM_LANES)> R{red, 0};
  LaneSums<PT> sum;
  if (g_out)
    sum = eval_tasks<FAM, true, true, PT, NT>(global_view(B, m), m, xs, gacc, diel, mask);
  else
    sum = eval_tasks<FAM, false, true, PT, NT>(global_view(B, m), m, xs, gacc, diel, mask);
  double* buf = (double*)((char*)xs + xs_bytes);
  if (NT > SUM_LANES && room == 0) {
    __syncthreads();  // the positions give way to the sums
    buf = (double*)xs;
    room = xs_bytes / (EX_WORDS * (int)sizeof(double));
  }
  const double e = group_energy<NT>(sum, buf, room, R);
  if constexpr (PT) {
    combine_groups<NT>(sum.kind, buf, room);
    double v4[4] = {sum.kind[0], sum.kind[1], sum.kind[2], sum.kind[3]};
    R.template run<4, 0>(v4);
    double v3[4] = {sum.kind[4], sum.kind[5], sum.kind[6], 0.0};
    R.template run<4, 0>(v3);
    if (threadIdx.x == 0) {
      for (int k = 0; k < 4; k++) e_terms[7 * c + k] = v4[k];
      for (int k = 0; k < 3; k++) e_terms[7 * c + 4 + k] = v3[k];
    }
  }
  if (threadIdx.x == 0) e_out[c] = e;
  if (g_out)
    for (int i = threadIdx.x; i < n; i += NT) g_out[off + i] = from_fx(gacc[i]);
}

// ------------------------------------------------------------------------------------
// nk minimizer (in-kernel BFGS / L-BFGS), TG formula family.
// Control flow: mlxmolkit/mmff_bfgs_source_tg.metal:1-372 (BFGS) and
// mlxmolkit/mmff_lbfgs_source_tg.metal:1-298 (L-BFGS); constants mmff_bfgs_header.metal:3-10.
constexpr double TOLX = 1.2e-6;
constexpr double FUNCTOL = 1e-4;
constexpr double MOVETOL = 1e-6;
constexpr double EPS_GUARD = 3e-7;
constexpr double MAX_STEP_FACTOR = 100.0;
constexpr int MAX_LS_ITERS = 1000;
constexpr float GRAD_SCALE_INIT = 0.1f;
constexpr double GRAD_CAP = 10.0;
constexpr int LBFGS_MAX_M = 16;
// pending rank-2 updates the global-Hessian BFGS pass applies on the fly before writing H back
constexpr int HPEND_MAX = 4;
// the same for the 512-thread kernel, which has the registers for more (one workgroup per CU,
// 233 VGPRs without spills at six): H is then written every sixth iteration. Ragged workload,
// n > 360 class: 1692.5 ms against 1726.2 ms with four and 1716.2 ms with eight
constexpr int HPEND_LARGE = 6;
__host__ __device__ constexpr int hpend_for(int nt) { return nt >= 512 ? HPEND_LARGE : HPEND_MAX; }

struct NkParams {
  const float* x_in;
  float* x_out;
  double* e_out;
  int32_t* status;
  int32_t* counters;
  const int32_t* order;
  int32_t* queue;     // work counters, zeroed before launch: one, or one per XCD
  float* hglob;       // per-workgroup global slots (H or L-BFGS history)
  size_t slot_floats;
  const float* precond;
  int max_iters;
  float grad_tol;
  int diel;
  int m;
  int max_n;          // 3 * max_atoms rounded up to a multiple of 4
  int ls_grad;
  int tbytes;         // LDS bytes reserved for staged term tables (TL kernels), else 0
  int eb_floats;      // LDS floats for bonded energies (HELP kernels)
  int xcd_on;         // order is split into 8 per-XCD queues at xcd_off
  int32_t xcd_off[9];
};

// Packed upper-triangle storage of a symmetric n x n matrix with every column padded to a
// multiple of 4 floats (16 bytes): column c holds rows 0..c from offset pcol(c) =
// sum_{k<c} round4(k + 1), so every column starts 16-byte aligned and can be walked in float4
// steps. packed_floats(n) = pcol(n) floats hold the matrix.
__host__ __device__ inline int pcol(int c) {
  const int m = c >> 2, r = c & 3;
  return 8 * m * (m + 1) + 4 * r * (m + 1);
}
__host__ __device__ inline size_t packed_floats(int n) { return (size_t)pcol(n); }

// Symmetric blocked storage in HBM: the matrix is cut into 4x4 blocks over the nq = n/4 row
// quads, and only one block per unordered quad pair {L, M} is kept. Block (s, L) holds rows
// 4L..4L+3 and columns 4M..4M+3 with M = (L + s) mod nq, for the cyclic distances
// s = 0 .. nq/2 (for even nq the pairs at distance nq/2 are kept once, by L < nq/2); its row r
// is float4 number (4 s + r) nq + L, so the lanes that walk consecutive L of one distance read
// consecutive 16-byte words. sym_slot_floats(max_n) floats hold the largest matrix.
__host__ __device__ inline int sym_dists(int nq) { return (nq >> 1) + 1; }
__host__ __device__ inline size_t sym_slot_floats(int max_n) {
  const int nq = max_n >> 2;
  return (size_t)16 * sym_dists(nq) * nq;
}
// LDS floats of one wave's private H v accumulators: up to 64/nq copies of the 4 nq entries
// when nq <= 64 (at most 256 floats), one copy otherwise
__host__ __device__ inline int sym_acc_floats(int max_n) { return max_n > 256 ? max_n : 256; }

// LDS footprint (bytes) of the nk kernel
// hm: Hessian placement (0 packed LDS, 1 full HBM, 2 packed HBM, 3 symmetric blocked HBM);
// only the full and symmetric HBM BFGS kernels keep the extra pending-update slots, and the
// symmetric one adds its per-wave accumulators
// help > 1: two rounds of pair energies and eb_floats of bonded energies
__host__ __device__ inline size_t nk_lds_bytes(int algo, int hm, int nt, int max_n, int m, size_t tbytes = 0,
                                               int help = 1, int eb_floats = 0) {
  const bool hlds = hm == 0;
  size_t nw = (size_t)nt / 64;
  size_t b = 16 * nw * sizeof(double) + 64 + 2 * (size_t)LBFGS_MAX_M * sizeof(double);
  b += (size_t)max_n * 8;  // gradient accumulators
  b += (size_t)max_n * 4 * 4;   // xs, d, xo, hd
  b += (size_t)max_n * 8;       // g, dg
  if (algo == MMFFHIP_BFGS)
    b += (size_t)max_n * 16;  // a pending update: s, h, alpha, beta
  else if (help == 1)
    b += (size_t)lbfgs_eb_floats(max_n) * 4;  // bonded energies
  if (algo == MMFFHIP_BFGS && (hm == 1 || hm == 3)) b += (size_t)(hpend_for(nt) - 1) * max_n * 16;  // more pending updates
  if (algo == MMFFHIP_BFGS && hm == 3) b += nw * (size_t)sym_acc_floats(max_n) * 4;
  if (algo == MMFFHIP_LBFGS) {
    if (hlds) b += 2 * (size_t)m * max_n * 4;
  } else if (hlds) {
    b += ((packed_floats(max_n) * 4) + 15) & ~(size_t)15;
  }
  b += (tbytes + 15) & ~(size_t)15;
  if (help > 1) b += 4 * (help_ring_floats<1>(help) * nt + (size_t)eb_floats);
  return b;
}

// initial inverse Hessian element: the identity, or the symmetric part of the learned
// per-atom 3x3 block times psc (blocks approximate (0.1 * Hessian block)^-1; psc = 0.1 /
// gradient scale rescales them to the scaled gradient the minimizer works with). BFGS keeps
// H symmetric, and every placement reads one orientation of each element, so the start is
// made symmetric rather than taken from one triangle of the block.
__device__ __forceinline__ float h_init(const float* pc, float psc, int i, int j) {
  if (pc) {
    if ((i / 3) != (j / 3)) return 0.0f;
    const float* b = pc + (j / 3) * 9;
    return psc * (0.5f * (b[(i % 3) * 3 + (j % 3)] + b[(j % 3) * 3 + (i % 3)]));
  }
  return i == j ? 1.0f : 0.0f;
}

// HM: where the dense inverse Hessian lives -- 0 packed in LDS, 1 full in HBM, 2 packed in HBM
// TL: term tables read from global memory (0), staged in LDS (1), or bonded tables staged and
// pairs read from global memory (2; 3: likewise, but a molecule whose bonded tables are larger than
// the reserve has them read from global memory too, by a second copy of the evaluation). Global-Hessian kernels of up to 256 threads are compiled
// for three waves per SIMD (at most 168 VGPRs), so three workgroups share a CU: their LDS
// use is small, and the extra resident conformers hide memory latency better than the
// registers the compiler would otherwise use (medium workload: 172.6 against 178.5 ms). One wave with
// everything in LDS is held to them too, where it would take 178-186: 18,000 conformers of 9-14 atoms
// 4.38 -> 3.67 ms (L-BFGS 6.66 -> 5.29), 8,000 of 26 atoms, which LDS limits first, 11.1 and 11.2.
// HELP: a conformer's workgroup has HELP * NT threads, of which the first NT do all that NT threads
// do and the others share the term evaluation (eval_help): same results, shorter iterations.
// For batches of at most one conformer per CU, whose time is the longest conformer's chain of
// iterations. Three times 256 threads keep three waves per SIMD and their 168 registers.
template <int ALGO, int HM, int TL, int NT, int HELP = 1>
__global__ void __launch_bounds__(
    NT * HELP, HELP == 1 && (((HM == 1 || HM == 3) && NT <= 256) || (TL == 1 && NT == 64)) ? 3 : 1)
    k_minimize_nk(KBatch B, NkParams P) {
  constexpr bool HLDS = HM == 0;    // LDS-resident (also selects the LDS L-BFGS history)
  constexpr bool PACKED = HM == 0 || HM == 2;  // packed upper triangle, select read + column-pair write-back
  constexpr bool SYM = HM == 3 && ALGO == MMFFHIP_BFGS;  // symmetric 4x4 blocks in HBM
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NW = NT / 64;
  // a helper's index lies past every loop's end
  const int tid = HELP == 1 || threadIdx.x < NT ? (int)threadIdx.x : 1 << 30;
  const int mn = P.max_n;
  double* red = (double*)smem;
  int* s_int = (int*)(red + 16 * NW);
  double* lb_sc = (double*)(s_int + 16);  // rho[16], alpha[16]
  unsigned long long* gacc = (unsigned long long*)(lb_sc + 2 * LBFGS_MAX_M);
  float* gv = (float*)(gacc + mn);  // scaled gradient g
  float* xs = gv + mn;
  float* d = xs + mn;   // direction (also y2 = H g scratch)
  float* xo = d + mn;   // previous x, then xi = x - x_old
  // A rank-2 update U(t, j) = alpha_t s_j + beta_t h_j (s = x - x_old, h = H dg) takes a slot of
  // 4 mn floats. Global-Hessian BFGS keeps up to NPM pending updates and writes H back once
  // every NPM iterations; the others apply theirs at once. The symmetric pass reads whole quads
  // of s, h, alpha and beta (and of g) in one instruction, so it keeps the four in planes:
  // one conflict-free 16-byte read per quad and plane, where {s, h} and {alpha, beta} pairs
  // (and {dg, g}) took two 16-byte reads at a 32-byte stride, each a 2-way bank conflict. With
  // pairs the LDS pipe was busy 63% of the n <= 360 launch of a 100,000-conformer ragged batch.
  // The other placements read an update row by row and keep the pairs.
  constexpr bool LAZY = (HM == 1 || HM == 3) && ALGO == MMFFHIP_BFGS;
  constexpr int NPM = LAZY ? hpend_for(NT) : 1;
  float* UP = xo + mn;
  auto up_plane = [&](int k, int c) { return UP + (size_t)(4 * k + c) * mn; };  // c: s, h, alpha, beta
  auto sh_slot = [&](int k) { return (float2*)up_plane(k, 0); };
  auto ab_slot = [&](int k) { return (float2*)up_plane(k, 2); };
  float* dgv = UP + (ALGO == MMFFHIP_BFGS ? NPM * 4 * mn : HELP == 1 ? lbfgs_eb_floats(mn) : 0);  // last change of g
  float* hd = dgv + mn;  // H dg (BFGS) / two-loop q (L-BFGS)
  float* big = hd + mn;
  float* H = HLDS ? big : P.hglob + (size_t)blockIdx.x * P.slot_floats;
  size_t big_floats = 0;
  if (HLDS) big_floats = ALGO == MMFFHIP_BFGS ? packed_floats(mn) : 2 * (size_t)P.m * mn;
  // symmetric storage: per-wave H v accumulators, cleared before each pass
  const int sacc_w = sym_acc_floats(mn);
  if (SYM) big_floats = (size_t)NW * sacc_w;
  // During an evaluation the bonded terms' energies lie in dgv, hd and the accumulators (at least
  // 12 floats per atom, which hold all but a cage molecule's at once, and never less than a task's
  // 64), none of which is live then; L-BFGS has that room where BFGS keeps its update.
  // The full-matrix kernels have no registers for the next term's tables: loading them ahead took
  // 112-132 bytes of scratch per lane at 64-256 threads, 20-44 without, and 8,000 ragged conformers of
  // 256 threads 103.6 -> 98.3 ms (128 threads, medium: 24.7 -> 24.2; 640, ragged: 31.1 -> 27.9).
  constexpr bool PREF = TL == 0 && HM != 1;
  constexpr bool ORDERED = HELP == 1 && (SYM || ALGO == MMFFHIP_LBFGS);
  float* ebuf = SYM ? dgv : UP;
  const int ebuf_n = SYM ? 2 * mn + NW * sacc_w : lbfgs_eb_floats(mn);
  unsigned char* tstage = (unsigned char*)(big + big_floats);
  float* ring = (float*)(tstage + P.tbytes);  // HELP: pair energies, then bonded energies
  float* eb = ring + help_ring_floats<NT>(HELP);
  const int M = P.m;
  float* S = H;
  float* Y = H + (size_t)M * mn;
  double* rho = lb_sc;
  double* alf = lb_sc + LBFGS_MAX_M;

  Reducer<NT, 8, (HELP > 1)> R{red, 0};

  for (;;) {
    if (tid == 0) {
      int kk;
      if (P.xcd_on) {
        // the queue of this workgroup's XCD first (workgroups are dispatched to the 8 XCDs
        // round-robin), then the others' until every queue is drained
        const int x0 = blockIdx.x & 7;
        kk = B.n_confs;
        for (int t = 0; t < 8; t++) {
          const int x = (x0 + t) & 7;
          const int cnt = P.xcd_off[x + 1] - P.xcd_off[x];
          if (cnt <= 0) continue;
          const int v = atomicAdd(P.queue + x, 1);
          if (v < cnt) {
            kk = P.xcd_off[x] + v;
            break;
          }
        }
      } else {
        kk = atomicAdd(P.queue, 1);
      }
      s_int[0] = kk;
    }
    __syncthreads();
    const int k = s_int[0];
    __syncthreads();
    if (k >= B.n_confs) break;
    const int c = P.order ? P.order[k] : k;
    const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
    const int n = 3 * m.n_atoms;
    const int off = B.conf_off[c];
    // packed-Hessian passes: 2^lsh lanes per row in the read pass, 2^lsh2 lanes per column
    // pair in the write-back (at most 8 lanes each)
    const int np = (n + 1) >> 1;
    int lsh = 0, lsh2 = 0;
    while (lsh < 3 && (n << (lsh + 1)) <= NT) lsh++;
    while (lsh2 < 3 && (np << (lsh2 + 1)) <= NT) lsh2++;
    const float* pc = P.precond ? P.precond + (size_t)(off / 3) * 9 : nullptr;
    TView TV;
    const bool fits = !TL || table_lds_bytes(m.nb, m.na, m.nsb, m.noop, m.ntor, TL == 1 ? m.npair : 0) <= (size_t)P.tbytes;
    if (TL) {
      if (TL != 3 && !fits) {
        // tables larger than the reserved LDS: report and skip (the planner never does this)
        for (int i = tid; i < n; i += NT) P.x_out[off + i] = P.x_in[off + i];
        if (tid == 0) {
          P.e_out[c] = __longlong_as_double(0x7ff8000000000000ll);
          P.status[c] = 2;
          if (P.counters) P.counters[3 * c] = P.counters[3 * c + 1] = P.counters[3 * c + 2] = 0;
        }
        continue;
      }
      TV = stage_tables(B, m, tstage, fits ? tid : 1 << 30, NT, TL == 1);
    } else {
      TV = global_view(B, m);
    }

    for (int i = tid; i < n; i += NT) xs[i] = P.x_in[off + i];
    for (int i = tid; i < n; i += NT) gacc[i] = 0ull;
    if (SYM) {
      // the padding rows of the last quad: zero gradient and update vectors, so that the
      // padding elements of H stay zero and add nothing to H v
      for (int i = n + tid; i < ((n + 3) & ~3); i += NT) {
        gv[i] = 0.f;
#pragma unroll
        for (int k = 0; k < 4 * NPM; k++) up_plane(0, k)[i] = 0.f;
      }
    }
    float psc = 1.0f;
    auto init_h = [&]() {
      if (ALGO != MMFFHIP_BFGS) return;
      if (PACKED) {
        for (int col = tid; col < n; col += NT) {
          float* cp = H + pcol(col);
          for (int i = 0; i < ((col + 4) & ~3); i++) cp[i] = i <= col ? h_init(pc, psc, i, col) : 0.0f;
        }
      } else if (SYM) {
        const int nq = (n + 3) >> 2;
        float4* H4 = (float4*)H;
        for (int f = tid; f < 4 * sym_dists(nq) * nq; f += NT) {
          const int sr = f / nq, L = f - sr * nq, r = sr & 3, s = sr >> 2;
          const int M = L + s < nq ? L + s : L + s - nq;
          const int jr = 4 * L + r;
          float v[4];
#pragma unroll
          for (int c = 0; c < 4; c++) {
            const int t = 4 * M + c;
            v[c] = (jr < n && t < n) ? h_init(pc, psc, jr, t) : 0.0f;
          }
          H4[f] = make_float4(v[0], v[1], v[2], v[3]);
        }
      } else {
        const int ldh = (n + 3) & ~3;  // rows padded to 16 bytes; padding columns stay zero
        for (int col = tid; col < ldh; col += NT)
          for (int j = 0; j < n; j++) H[(size_t)j * ldh + col] = col < n ? h_init(pc, psc, j, col) : 0.0f;
      }
    };
    __syncthreads();

    auto evaluate = [&](auto grad, auto energy) {
      constexpr bool G = decltype(grad)::value, EV = decltype(energy)::value;
      if constexpr (HELP > 1) {
        if (TL == 3 && !fits)
          return eval_help<FAM_TG, G, EV, NT, HELP>(global_view(B, m), m, xs, gacc, P.diel, eb, P.eb_floats, ring);
        return eval_help<FAM_TG, G, EV, NT, HELP>(TV, m, xs, gacc, P.diel, eb, P.eb_floats, ring);
      } else if constexpr (ORDERED)
        return eval_ordered<FAM_TG, G, EV, NT>(TV, m, xs, gacc, P.diel, ebuf, ebuf_n);
      else
        return eval_terms<FAM_TG, G, NT, PREF, EV>(TV, m, xs, gacc, P.diel);
    };
    const std::true_type yes;
    const std::false_type no;
    int n_grads = 1, n_evals = 0, iters = 0;
    // initial energy + gradient (mmff_bfgs_source_tg.metal:115-135)
    double E = R.sum(evaluate(yes, yes));
    float gscale = GRAD_SCALE_INIT;
    {
      double mxg = 0.0;
      for (int i = tid; i < n; i += NT) mxg = fmax(mxg, (double)fabsf(from_fx(gacc[i]) * gscale));
      mxg = R.max(mxg);
      while (mxg > GRAD_CAP) {
        gscale *= 0.5f;
        mxg *= 0.5;
      }
      for (int i = tid; i < n; i += NT) {
        dgv[i] = 0.f;
        gv[i] = from_fx(gacc[i]) * gscale;
      }
    }
    psc = GRAD_SCALE_INIT / gscale;
    init_h();  // H0 needs the gradient scale when it comes from the learned blocks
    __syncthreads();
    // initial direction: -g, or -H0 g with the learned preconditioner
    for (int i = tid; i < n; i += NT) {
      if (pc && ALGO == MMFFHIP_BFGS) {
        const int a = i / 3;
        float sacc = 0.f;
        for (int q = 0; q < 3; q++) sacc += h_init(pc, psc, i, 3 * a + q) * gv[3 * a + q];
        d[i] = -sacc;
      } else {
        d[i] = -gv[i];
      }
    }
    double ss = 0.0;
    for (int i = tid; i < n; i += NT) ss += (double)xs[i] * xs[i];
    ss = R.sum(ss);
    const double max_step = MAX_STEP_FACTOR * fmax(sqrt(ss), (double)n);  // :141-145
    int status = 1;
    int hist_count = 0, hist_idx = 0;
    bool fallback_used = (pc == nullptr);
    int npend = 0;  // rank-2 updates pending (applied lazily in later H passes)

    for (int it = 0; it < P.max_iters; it++) {
      iters = it + 1;
      const double E_old = E;
      double v3[3] = {0.0, 0.0, 0.0};
      for (int i = tid; i < n; i += NT) {
        xo[i] = xs[i];
        v3[0] += (double)d[i] * d[i];
        v3[1] += (double)d[i] * gv[i];
        v3[2] = fmax(v3[2], (double)(fabsf(d[i]) / fmaxf(fabsf(xs[i]), 1.0f)));
      }
      R.template run<2, 1>(v3);
      double slope = v3[1], test = v3[2];
      const double dn = sqrt(v3[0]);
      // a step longer than max_step is scaled down (:157-166); the scale goes into the
      // step length instead of into d, so that d stays -H g, which the next H pass uses
      double dsc = 1.0;
      if (dn > max_step) {
        dsc = (double)(float)(max_step / dn);
        slope *= dsc;
        test *= dsc;
      }
      if (slope >= 0.0) {  // ascent bail-out :170-174
        status = 0;
        break;
      }
      const double lam_min = MOVETOL / fmax(test, 1e-30);
      // backtracking line search :192-256
      double lam = 1.0, prev_lam = 1.0, prev_e = E_old;
      bool accepted = false, have_grad = false;
      for (int ls = 0; ls < MAX_LS_ITERS; ls++) {
        if (lam < lam_min) break;
        const float lf = (float)(lam * dsc);
        for (int i = tid; i < n; i += NT) {
          xs[i] = xo[i] + lf * d[i];
          if (P.ls_grad) gacc[i] = 0ull;
        }
        __syncthreads();
        double te;
        if (P.ls_grad)
          te = R.sum(evaluate(yes, yes));
        else
          te = R.sum(evaluate(no, yes));
        n_evals++;
        if (te - E_old <= FUNCTOL * lam * slope) {
          E = te;
          accepted = true;
          have_grad = P.ls_grad != 0;
          break;
        }
        double tmp;
        if (ls == 0) {
          tmp = -slope / (2.0 * (te - E_old - slope));
        } else {
          const double rhs1 = te - E_old - lam * slope;
          const double rhs2 = prev_e - E_old - prev_lam * slope;
          const double l2 = lam * lam, pl2 = prev_lam * prev_lam, dv = lam - prev_lam;
          if (fabs(dv) < 1e-30) {
            tmp = 0.5 * lam;
          } else {
            const double a = (rhs1 / l2 - rhs2 / pl2) / dv;
            const double b = (-prev_lam * rhs1 / l2 + lam * rhs2 / pl2) / dv;
            if (fabs(a) < 1e-30) {
              tmp = fabs(b) > 1e-30 ? -slope / (2.0 * b) : 0.5 * lam;
            } else {
              const double disc = b * b - 3.0 * a * slope;
              if (disc < 0.0)
                tmp = 0.5 * lam;
              else if (b <= 0.0)
                tmp = (-b + sqrt(disc)) / (3.0 * a);
              else
                tmp = -slope / (b + sqrt(disc));
            }
          }
        }
        tmp = fmin(tmp, 0.5 * lam);
        tmp = fmax(tmp, 0.1 * lam);
        prev_lam = lam;
        prev_e = te;
        lam = tmp;
      }
      if (!accepted) {
        for (int i = tid; i < n; i += NT) xs[i] = xo[i];
        if (!fallback_used) {
          // learned preconditioner fallback: restart as identity-scaled BFGS
          fallback_used = true;
          pc = nullptr;
          npend = 0;
          init_h();
          for (int i = tid; i < n; i += NT) d[i] = -gv[i];
          __syncthreads();
          continue;
        }
      }
      // xi = x - x_old and TOLX :258-279
      double tx = 0.0;
      for (int i = tid; i < n; i += NT) {
        const float xi = xs[i] - xo[i];
        xo[i] = xi;
        tx = fmax(tx, (double)(fabsf(xi) / fmaxf(fabsf(xs[i]), 1.0f)));
      }
      tx = R.max(tx);
      if (tx < TOLX) {
        status = 0;
        break;
      }
      // new gradient :285-298
      if (!have_grad) {
        for (int i = tid; i < n; i += NT) gacc[i] = 0ull;
        __syncthreads();
        evaluate(yes, no);
        __syncthreads();
      }
      n_grads++;
      double v2[2] = {0.0, 0.0};
      for (int i = tid; i < n; i += NT) {
        const float sg = fabsf(from_fx(gacc[i]) * gscale);
        v2[0] = fmax(v2[0], (double)sg);
        v2[1] = fmax(v2[1], (double)sg * fmax((double)fabsf(xs[i]), 1.0));
      }
      R.template run<0, 2>(v2);
      while (v2[0] > GRAD_CAP) {  // scale_grad_serial, mmff_bfgs_header.metal:435-454
        gscale *= 0.5f;
        v2[0] *= 0.5;
        v2[1] *= 0.5;
      }
      for (int i = tid; i < n; i += NT) {
        const float gn = from_fx(gacc[i]) * gscale;
        dgv[i] = gn - gv[i];
        gv[i] = gn;
      }
      if (SYM)
        for (int i = tid; i < NW * sacc_w; i += NT) big[i] = 0.f;
      if (v2[1] / fmax(E * (double)gscale, 1.0) < (double)P.grad_tol) {  // :300-316
        status = 0;
        break;
      }
      __syncthreads();  // V visible to every lane

      if (ALGO == MMFFHIP_BFGS) {
        // One pass over H computes hd = H_k dg and y2 = H_k g, where H_k = H_stored +
        // pending rank-2 update; the pending update is written back in the same pass.
        // The update U = fi s s^T - fei h h^T + fae a a^T (a = fi s - fei h) is kept in the
        // factored form U(t, j) = alpha_t s_j + beta_t h_j (2 FMAs per element).
        // Reference: H dg (:318-324), dots (:326-345), rank-2 update (:347-358), d = -H g (:360-366).
        if (PACKED) {
          // Packed upper triangle (column j holds rows 0..j), kept fully updated. 2^lsh
          // consecutive lanes share row t and split its n columns into equal segments;
          // element (t, j) is read from column t when j <= t and from column j otherwise, so
          // every lane reads the same number of elements and H is read-only here. The
          // partial sums of a row are combined with DPP in a fixed order. Loads of the next
          // four columns are issued before the current four are consumed.
            const int lpr = 1 << lsh, seg = (n + lpr - 1) >> lsh;
            for (int r = tid; r < (n << lsh); r += NT) {
              const int t = r >> lsh, q = r & (lpr - 1);
              const int j0 = q * seg, j1 = min(n, j0 + seg);
              const int cb = pcol(t);
              int pj = pcol(j0);
              float a2[4] = {0.f, 0.f, 0.f, 0.f};
              int j = j0;
              if (j + 3 < j1) {
                float h[4], w[4];
                hrow_load4(H, gv, t, cb, j, pj, h, w);
                while (j + 7 < j1) {
                  float hn[4], wn[4];
                  const int pn = pcol(j + 4);
                  hrow_load4(H, gv, t, cb, j + 4, pn, hn, wn);
  #pragma unroll
                  for (int u = 0; u < 4; u++) {
                    a2[u] += h[u] * w[u];
                    h[u] = hn[u];
                    w[u] = wn[u];
                  }
                  j += 4;
                  pj = pn;
                }
  #pragma unroll
                for (int u = 0; u < 4; u++) a2[u] += h[u] * w[u];
                j += 4;
                pj = pcol(j);
              }
              for (; j < j1; j++) {
                const float hv = H[j <= t ? cb + j : pj + t];
                a2[0] += hv * gv[j];
                pj += (j + 4) & ~3;
              }
              float s2 = (a2[0] + a2[1]) + (a2[2] + a2[3]);
              if (lsh >= 1) s2 += dpp_f<DPP_QUAD_XOR1>(s2);
              if (lsh >= 2) s2 += dpp_f<DPP_QUAD_XOR2>(s2);
              if (lsh >= 3) s2 += dpp_f<DPP_ROW_HALF_MIRROR>(s2);
              if (q == 0) {
                // H dg = H g_new - H g_old = H g_new + d_old
                hd[t] = s2 + d[t];
                d[t] = s2;
              }
            }
            __syncthreads();
        } else if (SYM) {
          // Symmetric blocked storage (sym_slot_floats): each kept 4x4 block B of the quad pair
          // (L, M) is read once and serves both halves of H v: rows 4L.. gain B v_M and, off
          // the diagonal, rows 4M.. gain B^T v_L. Wave w takes the distances s = w, w + NW, ...
          // and its lanes walk (distance, L) items: for nq <= 64, 64/nq groups of nq lanes take
          // one distance each; for nq >= 64 + NW the items run on consecutively, so that one
          // instruction spans at most two distances NW apart, whose rows 4M.. are disjoint;
          // in between, 64 lanes and then nq - 64 take each distance. The products go into the
          // wave's private LDS accumulators (one copy per lane group, a float4 per quad) by a
          // read, add and write of the quad: no two lanes of one instruction touch the same
          // quad and a wave's LDS operations complete in order, so each sum is formed in a
          // fixed order and results are deterministic. (LDS float atomics give the same sums
          // but ran the medium workload at 302.6 ms against 119.0 ms: waves waited on LDS for
          // 42% of their cycles.) When all NPM update slots are pending they are added to each
          // element as it is read, oldest first, and the block is written back; otherwise
          // the pending updates enter H v through their factored form, from dot products
          // taken after the pass.
          const int nq = (n + 3) >> 2, D = sym_dists(nq), n4 = nq << 2;
          const int lane = tid & 63, w = tid >> 6;
          const int Jw = w < D ? (D - 1 - w) / NW + 1 : 0;  // distances of this wave
          const int G = nq <= 64 ? 64 / nq : 1;             // lane groups (accumulator copies)
          float* acc = big + (size_t)w * sacc_w;
          int j, L, cp = 0;
          if (nq <= 64) {
            cp = lane / nq;
            L = lane - cp * nq;
            j = cp < G ? cp : Jw;  // lanes past the last group stay idle
          } else {
            j = 0;
            L = lane;
          }
          const int steps = nq <= 64 ? (Jw + G - 1) / G : nq < 64 + NW ? 2 * Jw : (Jw * nq + 63) >> 6;
          const bool flush = npend == NPM;
          const float4* gq = (const float4*)gv;
          float4* H4 = (float4*)H;
          // The next block's four rows are loaded while this one is used: a step is one load
          // latency long otherwise, with three waves per SIMD to cover it. 100,000 ragged
          // conformers 1,134 -> 1,095 ms. (Before the uniform reduction results and the shorter pair
          // loop its 16 registers spilled 76-244 bytes per lane and lost 5%; now they cost the kernels
          // of 128 and 256 threads with staged tables 20 and 28 bytes, the others none.)
          //
          // one block of a lane's walk: its quads, whether it is kept, and its first row
          struct Item {
            int L, M, s;
            bool on;
            float4* bp;
          };
          auto item = [&]() {
            Item it;
            it.L = L;
            it.s = w + j * NW;
            it.M = L + it.s < nq ? L + it.s : L + it.s - nq;
            it.on = j < Jw && L < nq && !((nq & 1) == 0 && it.s == D - 1 && it.s != 0 && L >= (nq >> 1));
            it.bp = H4 + (it.on ? 4 * it.s * nq + L : 0);
            if (nq <= 64) {
              j += G;
            } else if (nq < 64 + NW) {
              if (L < 64) {
                L += 64;
              } else {
                L -= 64;
                j++;
              }
            } else {
              L += 64;
              if (L >= nq) {
                L -= nq;
                j++;
              }
            }
            return it;
          };
          auto load = [&](const Item& it, float4 (&b)[4]) {
#pragma unroll
            for (int r = 0; r < 4; r++) b[r] = it.bp[r * nq];
          };
          // rows 4L.. gain B v_M; then, off the diagonal, rows 4M.. gain B^T v_L. Another lane of
          // this wave may touch quad M in the first update or quad L in the second, so the
          // compiler barriers keep each read behind the previous write (the hardware keeps a
          // wave's LDS operations in order).
          auto use = [&](const Item& it, float4 (&b)[4]) {
            if (it.on) {
              const int L = it.L, M = it.M;
              if (flush) {
#pragma unroll
                for (int k = 0; k < NPM; k++) {
                  const float4 sv = ((const float4*)up_plane(k, 0))[L], hv = ((const float4*)up_plane(k, 1))[L];
                  const float4 av = ((const float4*)up_plane(k, 2))[M], bv = ((const float4*)up_plane(k, 3))[M];
                  const float ux[4] = {av.x, av.y, av.z, av.w}, uy[4] = {bv.x, bv.y, bv.z, bv.w};
                  hquad_upd(b[0], make_float2(sv.x, hv.x), ux, uy);
                  hquad_upd(b[1], make_float2(sv.y, hv.y), ux, uy);
                  hquad_upd(b[2], make_float2(sv.z, hv.z), ux, uy);
                  hquad_upd(b[3], make_float2(sv.w, hv.w), ux, uy);
                }
#pragma unroll
                for (int r = 0; r < 4; r++) it.bp[r * nq] = b[r];
              }
              const float4 vm = gq[M];
              float4* a4 = (float4*)(acc + cp * n4);
              {
                float4 v = a4[L];
                v.x += fmaf(b[0].w, vm.w, fmaf(b[0].z, vm.z, fmaf(b[0].y, vm.y, b[0].x * vm.x)));
                v.y += fmaf(b[1].w, vm.w, fmaf(b[1].z, vm.z, fmaf(b[1].y, vm.y, b[1].x * vm.x)));
                v.z += fmaf(b[2].w, vm.w, fmaf(b[2].z, vm.z, fmaf(b[2].y, vm.y, b[2].x * vm.x)));
                v.w += fmaf(b[3].w, vm.w, fmaf(b[3].z, vm.z, fmaf(b[3].y, vm.y, b[3].x * vm.x)));
                a4[L] = v;
              }
              asm volatile("" ::: "memory");
              if (it.s != 0) {
                const float4 vl = gq[L];
                float4 v = a4[M];
                v.x += fmaf(b[3].x, vl.w, fmaf(b[2].x, vl.z, fmaf(b[1].x, vl.y, b[0].x * vl.x)));
                v.y += fmaf(b[3].y, vl.w, fmaf(b[2].y, vl.z, fmaf(b[1].y, vl.y, b[0].y * vl.x)));
                v.z += fmaf(b[3].z, vl.w, fmaf(b[2].z, vl.z, fmaf(b[1].z, vl.y, b[0].z * vl.x)));
                v.w += fmaf(b[3].w, vl.w, fmaf(b[2].w, vl.z, fmaf(b[1].w, vl.y, b[0].w * vl.x)));
                a4[M] = v;
              }
              asm volatile("" ::: "memory");
            }
          };
          Item ia = item();
          float4 ba[4], bb[4];
          load(ia, ba);
          for (int kk = 0; kk < steps; kk += 2) {
            const Item ib = item();
            load(ib, bb);
            use(ia, ba);
            ia = item();
            load(ia, ba);
            use(ib, bb);
          }
          // the pending updates' part of H g when they were not added element by element:
          // y_t += alpha_t (s.g) + beta_t (h.g), with the dot products reduced in FP64
          const bool fact = npend > 0 && npend < NPM;
          float fs[NPM], fh[NPM];
          if (fact) {
            double ds[NPM], dh[NPM];
#pragma unroll
            for (int k = 0; k < NPM; k++) ds[k] = dh[k] = 0.0;
            for (int i = tid; i < n; i += NT) {
              const double g = gv[i];
#pragma unroll
              for (int k = 0; k < NPM; k++) {
                if (k < npend) {
                  ds[k] += (double)up_plane(k, 0)[i] * g;
                  dh[k] += (double)up_plane(k, 1)[i] * g;
                }
              }
            }
            if constexpr (2 * NPM <= 8) {
              double v[2 * NPM];
#pragma unroll
              for (int k = 0; k < NPM; k++) {
                v[k] = ds[k];
                v[NPM + k] = dh[k];
              }
              R.template run<2 * NPM, 0>(v);
#pragma unroll
              for (int k = 0; k < NPM; k++) {
                ds[k] = v[k];
                dh[k] = v[NPM + k];
              }
            } else {
              R.template run<NPM, 0>(ds);
              R.template run<NPM, 0>(dh);
            }
#pragma unroll
            for (int k = 0; k < NPM; k++) {
              fs[k] = (float)ds[k];
              fh[k] = (float)dh[k];
            }
          } else {
            __syncthreads();  // every wave's accumulators are complete
          }
          // sum the waves' accumulators in a fixed order
          for (int t = tid; t < n4; t += NT) {
            const int idx = t;
            float y = 0.f;
            for (int ww = 0; ww < NW; ww++)
              for (int c = 0; c < G; c++) {
                y += big[(size_t)ww * sacc_w + c * n4 + idx];
              }
            if (t < n) {
              if (fact) {
#pragma unroll
                for (int k = 0; k < NPM; k++)
                  if (k < npend) {
                    y = fmaf(up_plane(k, 3)[t], fh[k], fmaf(up_plane(k, 2)[t], fs[k], y));
                  }
              }
              // H dg = H g_new - H g_old = H g_new + d_old
              hd[t] = y + d[t];
              d[t] = y;
            }
          }
          __syncthreads();
          if (npend == NPM) npend = 0;  // every pending update is in H now
        } else {
          // full storage in HBM with rows padded to ldh = round4(n) floats (16-byte aligned).
          // 2^lq consecutive lanes share the column quad 4tq..4tq+3 and split its rows into
          // equal segments; a row of a quad is one 16-byte load and consecutive quads are
          // consecutive addresses (coalesced). H is written once every NPM iterations: when all
          // NPM update slots are pending, they are added to each element as it is read, oldest
          // first (which rounds each stored element exactly as a write-back after every update
          // would), and the rows are written back by their only owner. In the other iterations
          // the stored rows are only read and the pending updates enter H v through their
          // factored form, alpha_t (s.v) + beta_t (h.v), from dot products the same pass takes.
          // HQ rows per lane are loaded together: four fits the three-waves-per-SIMD register
          // budget (with two waves per SIMD, four and eight rows measured 178.5 and 181.1 ms on
          // the medium workload).
          constexpr int HQ = 4;
          const int nq = (n + 3) >> 2;
          int lq = 0;
          while (lq < 3 && (nq << (lq + 1)) <= NT) lq++;
          const int lpr = 1 << lq, seg = (n + lpr - 1) >> lq;
          for (int r = tid; r < (nq << lq); r += NT) {
            const int tq = r >> lq, q = r & (lpr - 1);
            const int j0 = q * seg, j1 = min(n, j0 + seg);
            float cx[NPM][4], cy[NPM][4];
            const float2* S[NPM];
#pragma unroll
            for (int k = 0; k < NPM; k++) {
              S[k] = sh_slot(k);
              const float2* ab = ab_slot(k);
#pragma unroll
              for (int u = 0; u < 4; u++) {
                const int t = 4 * tq + u;
                const float2 c = (npend > k && t < n) ? ab[t] : make_float2(0.f, 0.f);
                cx[k][u] = c.x;
                cy[k][u] = c.y;
              }
            }
            float a2[4] = {0.f, 0.f, 0.f, 0.f};
            float4* base = (float4*)H + tq;  // row j of the quad at base[j * nq]
            float lr[2][NPM];
#pragma unroll
            for (int k = 0; k < NPM; k++) lr[0][k] = lr[1][k] = 0.f;
            hquad_dispatch<HQ, NPM>(npend, base, nq, j0, j1, gv, S, cx, cy, a2, lr);
            // the pending updates' part of H g when they were not added element by element:
            // sum the dot products over the quad's lanes, then y_t += alpha_t (s.g) + beta_t (h.g)
            if (npend > 0 && npend < NPM) {
#pragma unroll
              for (int k = 0; k < NPM; k++)
#pragma unroll
                for (int c = 0; c < 2; c++) {
                  float x = lr[c][k];
                  if (lq >= 1) x += dpp_f<DPP_QUAD_XOR1>(x);
                  if (lq >= 2) x += dpp_f<DPP_QUAD_XOR2>(x);
                  if (lq >= 3) x += dpp_f<DPP_ROW_HALF_MIRROR>(x);
                  lr[c][k] = x;
                }
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
              float s2 = a2[u];
              if (lq >= 1) s2 += dpp_f<DPP_QUAD_XOR1>(s2);
              if (lq >= 2) s2 += dpp_f<DPP_QUAD_XOR2>(s2);
              if (lq >= 3) s2 += dpp_f<DPP_ROW_HALF_MIRROR>(s2);
              if (npend > 0 && npend < NPM) {
#pragma unroll
                for (int k = 0; k < NPM; k++) s2 = fmaf(cy[k][u], lr[1][k], fmaf(cx[k][u], lr[0][k], s2));
              }
              const int t = 4 * tq + u;
              if (q == 0 && t < n) {
                // H dg = H g_new - H g_old = H g_new + d_old
                hd[t] = s2 + d[t];
                d[t] = s2;
              }
            }
          }
          __syncthreads();
          if (npend == NPM) npend = 0;  // every pending update is in H now
        }
        double v6[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
        for (int i = tid; i < n; i += NT) {
          const float g = gv[i], dg = dgv[i];
          const double xi = xo[i], h = hd[i];
          v6[0] += (double)dg * xi;
          v6[1] += (double)dg * h;
          v6[2] += (double)dg * dg;
          v6[3] += xi * xi;
          v6[4] += xi * g;
          v6[5] += h * g;
        }
        R.template run<6, 0>(v6);
        const double fac = v6[0], fae = v6[1];
        const bool upd = fac * fac > EPS_GUARD * v6[2] * v6[3] && fac > 0.0;  // :347
        if (upd) {
          // U = A s s^T + Bc (s h^T + h s^T) + Cc h h^T, the expansion of the a a^T term
          const double fi = 1.0 / fac, fei = 1.0 / fae;
          const double A = fi + fae * fi * fi, Bc = -fae * fi * fei, Cc = fae * fei * fei - fei;
          const double xig = v6[4], hdg = v6[5];
          // the new update goes behind the pending ones (slot 0 when H is kept updated)
          const int slot = LAZY ? npend : 0;
          for (int t = tid; t < n; t += NT) {
            const double xi = xo[t], h = hd[t];
            const double al = A * xi + Bc * h, be = Bc * xi + Cc * h;
            d[t] = -(float)((double)d[t] + al * xig + be * hdg);
            if (SYM) {
              up_plane(slot, 0)[t] = (float)xi;
              up_plane(slot, 1)[t] = (float)h;
              up_plane(slot, 2)[t] = (float)al;
              up_plane(slot, 3)[t] = (float)be;
            } else {
              sh_slot(slot)[t] = make_float2((float)xi, (float)h);
              ab_slot(slot)[t] = make_float2((float)al, (float)be);
            }
          }
          npend++;
        } else {
          for (int t = tid; t < n; t += NT) d[t] = -d[t];
        }
        __syncthreads();
        if (PACKED && npend) {
          // write the update into the packed triangle: column c gains alpha_i s_c + beta_i h_c
          // in rows i <= c. Columns c and n-1-c form a pair and 2^lsh2 consecutive lanes split
          // the pair's 4-row groups evenly; each lane walks its groups in float4 steps with
          // s_c, h_c in registers (columns are 16-byte aligned).
          const int lp = 1 << lsh2;
          for (int r = tid; r < (np << lsh2); r += NT) {
            const int g = r >> lsh2, q = r & (lp - 1);
            const int c1 = g, c2 = n - 1 - g;
            const bool two = c2 != c1;
            const int l1 = (c1 + 4) >> 2, lb = l1 + (two ? (c2 + 4) >> 2 : 0);  // 4-row groups
            const int sb = (lb + lp - 1) >> lsh2, f0 = q * sb, f1 = min(lb, f0 + sb);
            if (f0 < l1) hcol_update4(H + pcol(c1), ab_slot(0), sh_slot(0)[c1], f0, min(f1, l1));
            if (two && f1 > l1) hcol_update4(H + pcol(c2), ab_slot(0), sh_slot(0)[c2], max(f0, l1) - l1, f1 - l1);
          }
          npend = 0;
          __syncthreads();
        }
      } else {
        // L-BFGS history and two-loop recursion (mmff_lbfgs_source_tg.metal:249-292)
        double ys = 0.0;
        for (int i = tid; i < n; i += NT) ys += (double)dgv[i] * xo[i];
        ys = R.sum(ys);
        if (ys > 1e-10) {
          const int slot = hist_idx % M;
          for (int i = tid; i < n; i += NT) {
            S[(size_t)slot * mn + i] = xo[i];
            Y[(size_t)slot * mn + i] = dgv[i];
          }
          if (tid == 0) rho[slot] = 1.0 / ys;
          hist_idx++;
          if (hist_count < M) hist_count++;
        }
        for (int i = tid; i < n; i += NT) hd[i] = gv[i];
        __syncthreads();  // rho visible
        // The two-loop recursion with each axpy fused into the next dot product's pass (and
        // gamma's dots into the first pass, the gamma scaling into the last axpy of the first
        // loop): the same FP32 updates of q and the same FP64 dot products, element by
        // element and lane by lane, so results are bit-identical to running the passes one
        // by one, in 2m + 1 passes over the history instead of 4m + 3.
        const int h = hist_count;
        if (h == 0) {
          for (int i = tid; i < n; i += NT) d[i] = -hd[i];
        } else {
          int sl = (hist_idx - 1) % M;  // newest entry (j = h - 1)
          if (sl < 0) sl += M;
          double v3[3] = {0.0, 0.0, 0.0};  // s_{h-1}.q, and s.y, y.y of the newest pair for gamma
          for (int i = tid; i < n; i += NT) {
            const double s_ = S[(size_t)sl * mn + i], y_ = Y[(size_t)sl * mn + i];
            v3[0] += s_ * hd[i];
            v3[1] += s_ * y_;
            v3[2] += y_ * y_;
          }
          R.template run<3, 0>(v3);
          const float gam = (float)(v3[1] / fmax(v3[2], 1e-30));
          double aj = rho[sl] * v3[0];
          if (tid == 0) alf[h - 1] = aj;
          for (int j = h - 1; j >= 1; j--) {  // q -= alpha_j y_j, then s_{j-1}.q
            const int sn = sl == 0 ? M - 1 : sl - 1;
            const float af = (float)aj;
            double sq = 0.0;
            for (int i = tid; i < n; i += NT) {
              const float q = hd[i] - af * Y[(size_t)sl * mn + i];
              hd[i] = q;
              sq += (double)S[(size_t)sn * mn + i] * q;
            }
            sq = R.sum(sq);
            aj = rho[sn] * sq;
            if (tid == 0) alf[j - 1] = aj;
            sl = sn;
          }
          // q -= alpha_0 y_0, r = gamma q, then y_0.r (sl is entry 0's slot)
          double yq = 0.0;
          {
            const float af = (float)aj;
            for (int i = tid; i < n; i += NT) {
              const float y_ = Y[(size_t)sl * mn + i];
              float q = hd[i] - af * y_;
              q *= gam;
              hd[i] = q;
              yq += (double)y_ * q;
            }
          }
          yq = R.sum(yq);  // its barrier also makes alf visible
          for (int j = 0; j < h; j++) {  // r += (alpha_j - beta_j) s_j, then y_{j+1}.r
            const float cf = (float)(alf[j] - rho[sl] * yq);
            const int sn = sl + 1 == M ? 0 : sl + 1;
            if (j + 1 < h) {
              double y2 = 0.0;
              for (int i = tid; i < n; i += NT) {
                const float r = hd[i] + cf * S[(size_t)sl * mn + i];
                hd[i] = r;
                y2 += (double)Y[(size_t)sn * mn + i] * r;
              }
              yq = R.sum(y2);
            } else {
              for (int i = tid; i < n; i += NT) {
                const float r = hd[i] + cf * S[(size_t)sl * mn + i];
                hd[i] = r;
                d[i] = -r;
              }
            }
            sl = sn;
          }
        }
        __syncthreads();
      }
    }
    for (int i = tid; i < n; i += NT) P.x_out[off + i] = xs[i];
    if (tid == 0) {
      P.e_out[c] = E;
      P.status[c] = status;
      if (P.counters) {
        P.counters[3 * c] = iters;
        P.counters[3 * c + 1] = n_grads;
        P.counters[3 * c + 2] = n_evals;
      }
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------
// BB fused steepest descent, MEGA family: mmff_metal_kernel.py:845-1075.
// NR: threads of the workgroup. The first 256 do everything but the evaluation, which all share.
// ex_bytes: LDS where the groups' sums meet during an evaluation.
// The gradient is taken from its sums where it is used, and the pass that moves an atom clears them,
// so a step waits for the positions, the energy and the step's dot products only. 1,000 conformers: 4.11 ms
// with a gradient and a clearing pass of their own and three more barriers, 4.00 so.
template <int NR>
__global__ void __launch_bounds__(NR) k_bb_fused(KBatch B, const float* __restrict__ x_in, float* x_out,
                                                 double* e_out, int max_it, float max_step, float grad_lr,
                                                 int ex_bytes) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NT = SUM_LANES;
  const int c = blockIdx.x;
  if (c >= B.n_confs) return;
  const int tid = NR == NT || threadIdx.x < NT ? (int)threadIdx.x : 1 << 30;
  const int mx = 3 * B.max_atoms, room = ex_bytes / (EX_WORDS * (int)sizeof(double));
  double* red = (double*)smem;
  unsigned long long* gacc = (unsigned long long*)(red + RED_WORDS);
  double* buf = (double*)(gacc + mx);
  float* xs = (float*)((char*)buf + ex_bytes);
  float* pp = xs + mx;
  float* pg = pp + mx;
  const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
  const int n = 3 * m.n_atoms;
  const int off = B.conf_off[c];
  for (int i = tid; i < n; i += NT) {
    xs[i] = x_in[off + i];
    pp[i] = xs[i];
    pg[i] = 0.f;
    gacc[i] = 0ull;
  }
  Reducer<NT, 8, (NR > NT)> R{red, 0};
  float alpha = grad_lr;
  double E_prev = 1e30, E = 0.0;
  for (int it = 0; it < max_it; it++) {
    __syncthreads();
    E = group_energy<NR>(eval_tasks<FAM_MEGA, true, false, false, NR>(global_view(B, m), m, xs, gacc, 1, 0x7fu), buf, room, R);
    if (it > 0 && E > E_prev + 1.0) {  // energy guard :1031-1038
      for (int i = tid; i < n; i += NT) {
        xs[i] = pp[i];
        gacc[i] = 0ull;
      }
      alpha = fmaxf(alpha * 0.5f, 1e-7f);
      E = E_prev;
      continue;
    }
    if (it > 0) {  // BB step :1041-1052
      double v2[2] = {0.0, 0.0};
      for (int i = tid; i < n; i += NT) {
        const float si = xs[i] - pp[i], yi = from_fx(gacc[i]) - pg[i];
        v2[0] += (double)si * si;
        v2[1] += (double)si * yi;
      }
      R.template run<2, 0>(v2);
      if (v2[1] > 1e-20) alpha = fminf(fmaxf((float)(v2[0] / v2[1]), 1e-6f), 0.3f);
    }
    E_prev = E;
    for (int a = tid; a < m.n_atoms; a += NT) {  // per-atom capped step :1063-1071
      float *x = xs + 3 * a, *xp = pp + 3 * a, *gp = pg + 3 * a;
      unsigned long long* ga = gacc + 3 * a;
      const float gx = from_fx(ga[0]), gy = from_fx(ga[1]), gz = from_fx(ga[2]);
      const float gn = sqrtf(gx * gx + gy * gy + gz * gz + 1e-30f);
      const float s = fminf(max_step / gn, alpha);
      ga[0] = ga[1] = ga[2] = 0ull;
      xp[0] = x[0];
      xp[1] = x[1];
      xp[2] = x[2];
      gp[0] = gx;
      gp[1] = gy;
      gp[2] = gz;
      x[0] -= s * gx;
      x[1] -= s * gy;
      x[2] -= s * gz;
    }
  }
  __syncthreads();
  for (int i = tid; i < n; i += NT) x_out[off + i] = xs[i];
  if (tid == 0) e_out[c] = E;
}

// ------------------------------------------------------------------------------------
// multi_mol lock-step L-BFGS (MEGA family): mmff_optimize_metal_multi_mol
// (mmff_metal_optimizer.py:217-535). State per conformer in a global workspace; each
// launch runs `steps` iterations; launches that end at a sync point apply the best-x guard
// and convergence test and count unconverged conformers in a flag that the next launch
// reads to skip the rest (the reference's break), so no host round trip is needed.
struct MMState {
  float* x;       // [total]
  float* g;       // [total] scaled gradient
  float* bx;      // [total] best x
  float* S;       // [m][total]
  float* Y;       // [m][total]
  double* rho;    // [m][n_confs]
  double* best_e; // [n_confs]
  double* e_new;  // [n_confs]
  int32_t* ring;  // [2*n_confs] len, head
  int32_t* conv;  // [n_confs]
  int32_t* pci;   // [n_confs]
  int32_t* flags; // [n_flags]
  size_t total;
};

// the gradient sums come cleared; starts with a barrier, and ends with one
template <int NR, class Red>
__device__ void mm_eval(const KBatch& B, const MolDesc& m, float* xs, unsigned long long* gacc, Red& R, double& E,
                        double* buf = nullptr, int room = 0) {
  __syncthreads();
  E = group_energy<NR>(eval_tasks<FAM_MEGA, true, false, false, NR>(global_view(B, m), m, xs, gacc, 1, 0x7fu), buf, room, R);
}

// mode 0: initial (x = x_in), mode 1: polish restart (x = best_x); both compute E+G, scale g,
// reset history; mode 0 also initialises best_e/best_x/conv/pci.
template <int NT>
__global__ void __launch_bounds__(NT) k_mm_init(KBatch B, MMState S, const float* x_in, float gsc, int mode,
                                                int max_iters) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NW = NT / 64;
  const int c = blockIdx.x;
  if (c >= B.n_confs) return;
  const int mx = 3 * B.max_atoms;
  double* red = (double*)smem;
  unsigned long long* gacc = (unsigned long long*)(red + 16 * NW);
  float* xs = (float*)(gacc + mx);
  const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
  const int n = 3 * m.n_atoms, off = B.conf_off[c];
  for (int i = threadIdx.x; i < n; i += NT) {
    xs[i] = mode == 0 ? x_in[off + i] : S.bx[off + i];
    gacc[i] = 0ull;
  }
  Reducer<NT> R{red, 0};
  double E;
  mm_eval<NT>(B, m, xs, gacc, R, E);
  for (int i = threadIdx.x; i < n; i += NT) {
    S.x[off + i] = xs[i];
    S.g[off + i] = from_fx(gacc[i]) * gsc;
    if (mode == 0) S.bx[off + i] = xs[i];
  }
  if (threadIdx.x == 0) {
    S.ring[2 * c] = 0;
    S.ring[2 * c + 1] = 0;
    if (mode == 0) {
      S.best_e[c] = E;
      S.conv[c] = 0;
      S.pci[c] = max_iters;
    }
    S.e_new[c] = E;
  }
}

// K dot products over a conformer's n coordinates: f(i, p) adds coordinate i's products to p
template <int NT, int K, class Red, class F>
__device__ __forceinline__ void block_dots(Red& R, int tid, int n, double (&p)[K], F f) {
#pragma unroll
  for (int k = 0; k < K; k++) p[k] = 0.0;
  for (int i = tid; i < n; i += NT) f(i, p);
  R.template run<K, 0>(p);
}

// LDS of k_mm_chunk: reduction buffer, gradient accumulators, x, g, x_new and alpha, the (s, y, rho)
// history when hl, and q (q_bytes of it; the groups' sums meet there during an evaluation)
size_t mm_lds(int nr, int mx, int m, bool hl, size_t limit, int& q_bytes) {
  const size_t rest = RED_WORDS * 8 + (size_t)mx * (8 + 12) + 8 * (size_t)m + (hl ? 8 * (size_t)m * (mx + 1) : 0) + 32;
  q_bytes = (int)ex_area(nr, (size_t)mx * 4, 2, rest, limit);
  return rest + q_bytes;
}

// HL: the (s, y) history is worked on in LDS for the launch's iterations (and written through to
// the workspace, which the next launch reads); from memory, each of an iteration's 2 len + 1
// dependent passes waited for its loads. Each lane meets only its own coordinates of it (but for
// the step over atoms, which comes behind the reductions' barriers), so it needs no barrier of its
// own. 128 registers put four workgroups on a CU. 1,000 conformers of 69 atoms on
// average, 200 + 50 iterations: 6.26 ms, 10.7 ms with the history read from memory and one loop
// over all term types. Of that, measured before the reductions by readlane and the spread terms:
// 7.4 ms; 9.1 ms with three workgroups per CU, 10.5 ms with the history in memory. Dropped: the
// recursion in one wave while the others wait (the same sums without barriers: 7.6 against 7.4 ms,
// and 3.53 against 2.75 ms for 60 conformers), and one 64-thread workgroup per conformer (12.1 ms).
// What bounds it: the 2 len + 1 passes of an iteration, each a block reduction (a barrier and a
// wave's latency), then the evaluation's vector instructions.
// NR: threads of the workgroup. The first 256 do everything but the evaluation, which all share
// (1,024 for batches of at most one conformer per CU; 60 ragged conformers, 100 + 25 iterations:
// 2.59 -> 2.16 ms).
template <bool HL, int NR>
__global__ void __launch_bounds__(NR, NR > 256 ? 1 : 4) k_mm_chunk(KBatch B, MMState S, int steps, int it_end, int do_sync,
                                                     int phase, const int32_t* prev_flag, int32_t* my_flag, int M,
                                                     float max_step, float gsc, float tol, int q_bytes) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NT = SUM_LANES;
  const int c = blockIdx.x;
  if (c >= B.n_confs) return;
  if (prev_flag && *prev_flag == 0) return;  // every conformer converged at the last sync
  const int tid = NR == NT || threadIdx.x < NT ? (int)threadIdx.x : 1 << 30;
  const int mx = 3 * B.max_atoms;
  double* red = (double*)smem;
  double* alf = red + RED_WORDS;  // [M]
  double* lrho = alf + M;         // [M] when HL
  unsigned long long* gacc = (unsigned long long*)(HL ? lrho + M : lrho);
  float* q = (float*)(gacc + mx);
  float* xs = (float*)((char*)q + q_bytes);
  float* gs = xs + mx;
  float* xn = gs + mx;
  const int room = q_bytes / (EX_WORDS * (int)sizeof(double));
  const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
  const int n = 3 * m.n_atoms, off = B.conf_off[c];
  const size_t T = S.total, HT = HL ? (size_t)mx : T;
  float* gS = S.S + off;
  float* gY = S.Y + off;
  float* hS = HL ? xn + mx : gS;  // slot h's coordinate i at [h * HT + i]
  float* hY = HL ? hS + (size_t)M * mx : gY;
  int len = S.ring[2 * c], head = S.ring[2 * c + 1];
  for (int i = tid; i < n; i += NT) {
    xs[i] = S.x[off + i];
    gs[i] = S.g[off + i];
    gacc[i] = 0ull;
  }
  auto rho = [&](int k) { return HL ? lrho[k] : S.rho[(size_t)k * B.n_confs + c]; };
  if (HL) {
    // the ring fills slots 0 .. len - 1 first
    for (int k = tid; k < len; k += NT) lrho[k] = S.rho[(size_t)k * B.n_confs + c];
    for (int k = 0; k < len; k++)
      for (int i = tid; i < n; i += NT) {
        hS[k * HT + i] = gS[k * T + i];
        hY[k * HT + i] = gY[k * T + i];
      }
  }
  Reducer<NT, 8, (NR > NT)> R{red, 0};
  double E = S.e_new[c];
  __syncthreads();
  for (int st = 0; st < steps; st++) {
    // two-loop direction, mmff_metal_optimizer.py:47-74 (history oldest -> newest), with each
    // axpy fused into the next dot product's pass, gamma's dots into the first pass and the
    // gamma scaling into the first loop's last axpy: the same FP32 updates of q and FP64 dot
    // products as running the passes one by one (bit-identical), in 2 len + 1 passes with the step.
    int sl = head + len - 1;  // newest entry
    if (sl >= M) sl -= M;
    float cf = 0.f;
    if (len > 0) {
      double v3[3];
      block_dots<NT, 3>(R, tid, n, v3, [&](int i, double (&p)[3]) {
        const float qv = gs[i];
        q[i] = qv;
        const double s = hS[sl * HT + i], y = hY[sl * HT + i];
        p[0] += s * qv;
        p[1] += s * y;
        p[2] += y * y;
      });
      const float gf = (float)(v3[1] / (v3[2] + 1e-30));
      double a = rho(sl) * v3[0];
      if (tid == 0) alf[len - 1] = a;
      for (int h = len - 1; h >= 1; h--) {  // q -= alpha_h y_h, then s_{h-1}.q
        const int sn = sl == 0 ? M - 1 : sl - 1;
        const float af = (float)a;
        double sq[1];
        block_dots<NT, 1>(R, tid, n, sq, [&](int i, double (&p)[1]) {
          const float qv = q[i] - af * hY[sl * HT + i];
          q[i] = qv;
          p[0] += (double)hS[sn * HT + i] * qv;
        });
        a = rho(sn) * sq[0];
        if (tid == 0) alf[h - 1] = a;
        sl = sn;
      }
      double yr[1];  // q -= alpha_0 y_0, q *= gamma, then y_0.q
      {
        const float af = (float)a;
        block_dots<NT, 1>(R, tid, n, yr, [&](int i, double (&p)[1]) {
          const float y = hY[sl * HT + i];
          float qv = q[i] - af * y;
          qv *= gf;
          q[i] = qv;
          p[0] += (double)y * qv;
        });  // its barrier also makes alf visible
      }
      for (int h = 0;; h++) {  // q += (alpha_h - beta_h) s_h, then y_{h+1}.q
        cf = (float)(alf[h] - rho(sl) * yr[0]);
        if (h + 1 == len) break;  // the last axpy goes with the step
        const int sn = sl + 1 == M ? 0 : sl + 1;
        block_dots<NT, 1>(R, tid, n, yr, [&](int i, double (&p)[1]) {
          const float r = q[i] + cf * hS[sl * HT + i];
          q[i] = r;
          p[0] += (double)hY[sn * HT + i] * r;
        });
        sl = sn;
      }
    }
    // d = -q with the per-atom cap of max_step (:365-373); x_new = x + d
    auto dir = [&](int i) { return len > 0 ? -(q[i] + cf * hS[sl * HT + i]) : -gs[i]; };
    for (int a = tid; a < m.n_atoms; a += NT) {
      const float dx = dir(3 * a), dy = dir(3 * a + 1), dz = dir(3 * a + 2);
      const float disp = sqrtf(dx * dx + dy * dy + dz * dz + 1e-30f);
      const float f = fminf(max_step / disp, 1.0f);
      xn[3 * a] = xs[3 * a] + dx * f;
      xn[3 * a + 1] = xs[3 * a + 1] + dy * f;
      xn[3 * a + 2] = xs[3 * a + 2] + dz * f;
    }
    mm_eval<NR>(B, m, xn, gacc, R, E, (double*)q, room);
    // push (s, y, rho) into the ring (:385-399); rho = 0 on bad curvature
    if (len >= M) {
      sl = head;
      head = head + 1 == M ? 0 : head + 1;
    } else {
      sl = head + len >= M ? head + len - M : head + len;
      len++;
    }
    double sy[1];
    block_dots<NT, 1>(R, tid, n, sy, [&](int i, double (&p)[1]) {
      const float gn = from_fx(gacc[i]) * gsc;
      gacc[i] = 0ull;  // for the next evaluation
      const float s = xn[i] - xs[i], y = gn - gs[i];
      hS[sl * HT + i] = s;
      hY[sl * HT + i] = y;
      if (HL) {
        gS[sl * T + i] = s;
        gY[sl * T + i] = y;
      }
      p[0] += (double)s * y;
      xs[i] = xn[i];
      gs[i] = gn;
    });
    if (tid == 0) {
      const double r = sy[0] > 1e-10 ? 1.0 / (sy[0] + 1e-30) : 0.0;
      if (HL) lrho[sl] = r;
      S.rho[(size_t)sl * B.n_confs + c] = r;  // read behind the next step's first reduction
    }
  }
  if (do_sync) {
    // best-x guard (:408-412) and convergence (:354-359 main, :477-481 polish)
    const bool improved = E < S.best_e[c];
    double gmax = 0.0;
    for (int a = tid; a < m.n_atoms; a += NT) {
      const float gx = gs[3 * a], gy = gs[3 * a + 1], gz = gs[3 * a + 2];
      gmax = fmax(gmax, (double)sqrtf(gx * gx + gy * gy + gz * gz));
    }
    gmax = R.max(gmax);
    if (improved)
      for (int i = tid; i < n; i += NT) S.bx[off + i] = xs[i];
    if (tid == 0) {
      if (improved) S.best_e[c] = E;
      const bool under = gmax <= (double)tol;
      if (phase == 0) {
        if (!S.conv[c] && under) {
          S.conv[c] = 1;
          S.pci[c] = it_end;
        }
        if (!S.conv[c]) atomicAdd(my_flag, 1);
      } else if (!under) {
        atomicAdd(my_flag, 1);
      }
    }
  }
  for (int i = tid; i < n; i += NT) {
    S.x[off + i] = xs[i];
    S.g[off + i] = gs[i];
  }
  if (tid == 0) {
    S.ring[2 * c] = len;
    S.ring[2 * c + 1] = head;
    S.e_new[c] = E;
  }
}

// l2_norm: grad_norm = ||g_sc||_2 of the last iterate (mmff_optimize_metal_batch,
// mmff_metal_optimizer.py:186) instead of its largest per-atom norm (multi_mol, :504-525)
template <int NT>
__global__ void __launch_bounds__(NT) k_mm_final(KBatch B, MMState S, float* x_best, double* e_final,
                                                 float* grad_norm, int32_t* pci, int32_t* conv, int32_t* iters_used,
                                                 int n_main_flags, int eval_freq, int max_iters, int l2_norm) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int NW = NT / 64;
  const int c = blockIdx.x;
  if (c >= B.n_confs) return;
  const int mx = 3 * B.max_atoms;
  double* red = (double*)smem;
  unsigned long long* gacc = (unsigned long long*)(red + 16 * NW);
  float* xs = (float*)(gacc + mx);
  const MolDesc m = load_desc(B.mol_desc + 16 * B.conf_mol[c]);
  const int n = 3 * m.n_atoms, off = B.conf_off[c];
  for (int i = threadIdx.x; i < n; i += NT) xs[i] = S.bx[off + i];
  __syncthreads();
  Reducer<NT> R{red, 0};
  double E = group_energy<NT>(eval_tasks<FAM_MEGA, false, false, false, NT>(global_view(B, m), m, xs, gacc, 1, 0x7fu), nullptr,
                              0, R);
  double gmax = 0.0;
  if (l2_norm) {
    for (int i = threadIdx.x; i < n; i += NT) gmax += (double)S.g[off + i] * S.g[off + i];
    gmax = sqrt(R.sum(gmax));
  } else {
    for (int a = threadIdx.x; a < m.n_atoms; a += NT) {
      const float gx = S.g[off + 3 * a], gy = S.g[off + 3 * a + 1], gz = S.g[off + 3 * a + 2];
      gmax = fmax(gmax, (double)sqrtf(gx * gx + gy * gy + gz * gz));
    }
    gmax = R.max(gmax);
  }
  for (int i = threadIdx.x; i < n; i += NT) x_best[off + i] = xs[i];
  if (threadIdx.x == 0) {
    e_final[c] = E;
    grad_norm[c] = (float)gmax;
    pci[c] = S.pci[c];
    conv[c] = S.conv[c];
    if (c == 0) {
      int used = max_iters;
      for (int k = 0; k < n_main_flags; k++)
        if (S.flags[k] == 0) {
          used = (k + 1) * eval_freq;
          break;
        }
      *iters_used = used;
    }
  }
}

__global__ void k_fill_i32(int32_t* p, int n, int v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ------------------------------------------------------------------------------------
// host helpers
struct DevInfo {
  int n_cu = 0, lds = 0, ok = 0;
};

DevInfo dev_info() {
  constexpr int CACHED = 64;  // a node of eight GPUs in eight partitions each
  static thread_local DevInfo cache[CACHED];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return DevInfo{};
  DevInfo fresh;
  DevInfo& di = dev < CACHED ? cache[dev] : fresh;
  if (!di.ok) {
    hipDeviceProp_t p;
    if (hipGetDeviceProperties(&p, dev) == hipSuccess) {
      di.n_cu = p.multiProcessorCount;
      di.lds = (int)p.sharedMemPerBlock;
      di.ok = 1;
    }
  }
  return di;
}

// allow dynamic LDS above the 64 KB default for a kernel (gfx950 has 160 KB per workgroup)
void allow_lds(const void* kernel, size_t bytes) {
  if (bytes > 65536) hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}

int check_batch(const mmffhip_batch* b) {
  if (!b) return fail(MMFFHIP_ERR_ARG, "batch is NULL");
  if (b->n_confs < 0 || b->n_mols < 0) return fail(MMFFHIP_ERR_ARG, "negative batch size");
  if (b->n_confs > 0 && (!b->mol_desc || !b->conf_mol || !b->conf_off))
    return fail(MMFFHIP_ERR_ARG, "batch descriptor pointers are NULL");
  if (b->max_atoms <= 0 && b->n_confs > 0) return fail(MMFFHIP_ERR_ARG, "max_atoms must be positive");
  if (b->max_atoms > 65535) return fail(MMFFHIP_ERR_SIZE, "molecules above 65535 atoms are not supported");
  return MMFFHIP_OK;
}

// LDS of k_energy_grad and its last two arguments; always fits a wide workgroup where it fits a
// narrow one
size_t eg_lds(int nt, int max_atoms, bool terms, size_t limit, int& xs_bytes, int& room) {
  const size_t rest = RED_WORDS * 8 + (size_t)3 * max_atoms * 8 + 16, one = EX_WORDS * sizeof(double);
  xs_bytes = (3 * max_atoms * 4 + 7) & ~7;
  room = nt > SUM_LANES ? (terms ? 7 : 2) : 0;
  if (rest + xs_bytes + room * one > limit) {
    room = 0;
    xs_bytes = (int)ex_area(nt, (size_t)3 * max_atoms * 4, 1, rest, limit);
  }
  return rest + xs_bytes + room * one;
}

// At most one conformer per CU: sixteen waves per conformer, whose latency is the call's, from the
// size on where that gains more than four groups' meeting in LDS costs; four waves otherwise. TG
// energy and gradient of one conformer, us from launch to launch in a graph, four and sixteen waves: 9 atoms
// 3.1 and 3.6, 34 atoms 3.6 and 3.9, 42 atoms 4.2 and 3.9, 82 atoms 7.4 and 5.5, 253 atoms 38.0 and 19.7; with kinds
// 3.6 and 5.2, 4.3 and 5.7, 4.9 and 5.7, 8.0 and 7.2, 38.4 and 21.5 (63 atoms 6.0 and 6.1). (The Python entry point's host
// work takes 7.5 us a call.) A wide workgroup fills its CU, so with more conformers than CUs they
// queue: 300 conformers of 82 atoms 9.6 and 10.3 us, 768: 11.8 and 15.4.
template <int FAM, bool PT>
int launch_eg(const KBatch& kb, const float* x, double* e, double* et, float* g, uint32_t mask, int diel,
              hipStream_t s) {
  const DevInfo di = dev_info();
  int xs_bytes = 0, room = 0;
  size_t lds = eg_lds(256, kb.max_atoms, PT, di.lds, xs_bytes, room);
  if (lds > (size_t)di.lds) return fail(MMFFHIP_ERR_SIZE, "molecule too large for the LDS of one workgroup");
  int nt = 256;
  auto kernel = k_energy_grad<FAM, PT, 256>;
  if (kb.n_confs <= di.n_cu && kb.max_atoms > (PT ? 64 : 40)) {
    lds = eg_lds(1024, kb.max_atoms, PT, di.lds, xs_bytes, room);
    kernel = k_energy_grad<FAM, PT, 1024>;
    nt = 1024;
  }
  allow_lds((const void*)kernel, lds);
  hipLaunchKernelGGL(kernel, dim3(kb.n_confs), dim3(nt), lds, s, kb, x, e, et, g, mask, diel, xs_bytes, room);
  HIP_TRY(hipGetLastError());
  return MMFFHIP_OK;
}

// The launch of k_mm_chunk: wide workgroups when there is at most one conformer per CU and the
// molecules are not small, as in launch_eg (one conformer, 100 + 25 iterations, narrow and wide: 9 atoms 0.63
// and 0.74 ms, 34 atoms 1.19 and 1.37, 57 atoms 1.43 and 1.45, 63 atoms 1.47 and 1.46, 82 atoms 1.77 and 1.61, 253
// atoms 6.64 and 3.90; 300 conformers of 82 atoms 2.17 and 3.25 ms); the history in LDS when it fits
// there, or leaves three workgroups per CU.
struct MMChunk {
  void (*kernel)(KBatch, MMState, int, int, int, int, const int32_t*, int32_t*, int, float, float, float, int);
  int nr;
  size_t lds;
  int q_bytes;
};
MMChunk mm_chunk_plan(int n_confs, int mx, int m, const DevInfo& di) {
  const size_t limit = (size_t)di.lds;
  int q = 0;
  if (n_confs <= di.n_cu && mx > 3 * 60) {
    const size_t hl = mm_lds(1024, mx, m, true, limit, q);
    if (hl <= limit) return {k_mm_chunk<true, 1024>, 1024, hl, q};
    const size_t g = mm_lds(1024, mx, m, false, limit, q);
    if (g <= limit) return {k_mm_chunk<false, 1024>, 1024, g, q};
  }
  const size_t hl = mm_lds(256, mx, m, true, limit, q);
  if (hl <= limit / 3) return {k_mm_chunk<true, 256>, 256, hl, q};
  const size_t g = mm_lds(256, mx, m, false, limit, q);
  return {k_mm_chunk<false, 256>, 256, g, q};
}

int round4(int v) { return (v + 3) & ~3; }

struct NkPlan {
  int nt = 256;
  int hm = 0;  // Hessian placement of k_minimize_nk (0 packed LDS, 1 full HBM, 2 packed HBM, 3 symmetric HBM)
  int tl = 0;  // term tables: 0 global, 1 all staged in LDS, 2 bonded staged
  int tbytes = 0;
  int help = 1;       // threads per lane (k_minimize_nk's HELP)
  int eb_floats = 0;
  size_t lds = 0;
  int grid = 0;
  size_t slot_floats = 0;
  int max_n = 0;
};

template <int ALGO, int HM, int TL, int NT, int HELP = 1>
const void* nk_kernel_ptr() {
  return (const void*)&k_minimize_nk<ALGO, HM, TL, NT, HELP>;
}

// kernels with NK_HELP threads per lane of 256
constexpr int NK_HELP = 3;
#define NK_HELP_EACH(X) \
  X(0, 3, 2, 256) X(0, 3, 3, 256) X(0, 3, 0, 256)                                                       \
  X(1, 0, 2, 256) X(1, 0, 0, 256) X(1, 1, 2, 256) X(1, 1, 0, 256)

#define NK_FOR_EACH(X)                                                                                   \
  X(0, 0, 1, 64) X(0, 0, 1, 128) X(0, 0, 1, 192) X(0, 0, 1, 256) X(0, 0, 1, 384) X(0, 0, 1, 512)        \
  X(0, 0, 0, 64) X(0, 0, 0, 128) X(0, 0, 0, 192) X(0, 0, 0, 256) X(0, 0, 0, 320) X(0, 0, 0, 384)        \
  X(0, 0, 0, 512) X(0, 0, 0, 640) X(0, 0, 0, 768) X(0, 0, 0, 1024)                                     \
  X(0, 1, 0, 64) X(0, 1, 0, 128) X(0, 1, 0, 192) X(0, 1, 0, 256) X(0, 1, 0, 320) X(0, 1, 0, 512)        \
  X(0, 1, 0, 640) X(0, 1, 0, 768) X(0, 1, 0, 1024)                                                     \
  X(0, 1, 2, 64) X(0, 1, 2, 128) X(0, 1, 2, 192) X(0, 1, 2, 256) X(0, 1, 2, 320) X(0, 1, 2, 512)       \
  X(0, 2, 0, 256) X(0, 2, 0, 512) X(0, 2, 0, 640) X(0, 2, 0, 1024)                                     \
  X(0, 3, 0, 64) X(0, 3, 0, 128) X(0, 3, 0, 256) X(0, 3, 0, 512)                                        \
  X(0, 3, 2, 64) X(0, 3, 2, 128) X(0, 3, 2, 256) X(0, 3, 2, 512)                                        \
  X(1, 0, 1, 64) X(1, 0, 1, 128) X(1, 0, 1, 256)                                                       \
  X(1, 0, 0, 128) X(1, 0, 0, 256) X(1, 0, 0, 512)                                                      \
  X(1, 1, 0, 128) X(1, 1, 0, 192) X(1, 1, 0, 256) X(1, 1, 0, 512) X(1, 1, 2, 256)

const void* nk_kernel(int algo, int hm, int tl, int nt, int help = 1) {
#define NKSEL(A, H, TL, T) \
  if (algo == A && hm == H && tl == TL && nt == T && help == 1) return nk_kernel_ptr<A, H, TL, T>();
#define NKSELH(A, H, TL, T) \
  if (algo == A && hm == H && tl == TL && nt == T && help == NK_HELP) return nk_kernel_ptr<A, H, TL, T, NK_HELP>();
  NK_FOR_EACH(NKSEL)
  NK_HELP_EACH(NKSELH)
#undef NKSEL
#undef NKSELH
  return nullptr;
}

int make_nk_plan(const mmffhip_batch* b, const mmffhip_nk_opts* o, NkPlan& pl) {
  if (!o) return fail(MMFFHIP_ERR_ARG, "options are NULL");
  if (o->algo != MMFFHIP_BFGS && o->algo != MMFFHIP_LBFGS) return fail(MMFFHIP_ERR_ARG, "unknown algo");
  if (o->algo == MMFFHIP_LBFGS && (o->lbfgs_m < 1 || o->lbfgs_m > LBFGS_MAX_M))
    return fail(MMFFHIP_ERR_ARG, "lbfgs_m must be in [1, 16]");
  if (o->diel != 1 && o->diel != 2) return fail(MMFFHIP_ERR_ARG, "diel must be 1 or 2");
  if (o->max_iters < 0) return fail(MMFFHIP_ERR_ARG, "max_iters must be >= 0");
  DevInfo di = dev_info();
  if (!di.ok) return fail(MMFFHIP_ERR_DEVICE, "no HIP device");
  pl.nt = o->block > 0 ? o->block : (3 * b->max_atoms > 256 ? 512 : 256);
  if (pl.nt < 64 || pl.nt > 1024 || pl.nt % 64 != 0)
    return fail(MMFFHIP_ERR_ARG, "block must be a multiple of 64 in [64, 1024]");
  pl.max_n = round4(3 * std::max(b->max_atoms, 1));
  const int m = o->algo == MMFFHIP_LBFGS ? o->lbfgs_m : 0;
  const size_t lds_in = nk_lds_bytes(o->algo, 0, pl.nt, pl.max_n, m);
  if (o->hess_place == MMFFHIP_HESS_LDS) {
    pl.hm = 0;
  } else if (o->hess_place == MMFFHIP_HESS_GLOBAL) {
    pl.hm = 1;
  } else if (o->hess_place == MMFFHIP_HESS_GLOBAL_PACKED) {
    pl.hm = o->algo == MMFFHIP_BFGS ? 2 : 1;
  } else if (o->hess_place == MMFFHIP_HESS_GLOBAL_SYM) {
    pl.hm = o->algo == MMFFHIP_BFGS ? 3 : 1;
  } else if (o->hess_place == MMFFHIP_HESS_AUTO) {
    // dense BFGS: the symmetric blocks in HBM (they beat the LDS triangle even where it
    // fits); L-BFGS: the history in LDS when it fits, else in HBM
    pl.hm = o->algo == MMFFHIP_BFGS ? 3 : lds_in <= (size_t)di.lds ? 0 : 1;
  } else {
    return fail(MMFFHIP_ERR_ARG, "unknown hess_place");
  }
  pl.lds = nk_lds_bytes(o->algo, pl.hm, pl.nt, pl.max_n, m);
  if (pl.lds > (size_t)di.lds) return fail(MMFFHIP_ERR_SIZE, "plan exceeds the LDS of one workgroup");
  // Stage term tables in LDS when asked and when they fit: all of them next to an LDS
  // Hessian; only the bonded ones beside a global Hessian, and only when that keeps the
  // unstaged kernel's workgroups per CU (there, occupancy hides the pair loads).
  const int max_wg = std::max(1, 12 / (pl.nt / 64));  // workgroups per CU at most (below)
  bool help_stage = false;  // a launch without helpers could stage: as many workgroups per CU as launch without
  if (o->table_lds_bytes > 0) {
    const int tl = pl.hm == 0 ? 1 : 2;
    const size_t with = nk_lds_bytes(o->algo, pl.hm, pl.nt, pl.max_n, m, (size_t)o->table_lds_bytes);
    const void* kt = nk_kernel(o->algo, pl.hm, tl, pl.nt);
    bool take = with <= (size_t)di.lds && kt != nullptr;
    if (take && tl == 2) {
      const void* k0 = nk_kernel(o->algo, pl.hm, 0, pl.nt);
      int pc0 = 0, pc1 = 0;
      allow_lds(kt, with);
      if (k0) allow_lds(k0, pl.lds);
      take = k0 && hipOccupancyMaxActiveBlocksPerMultiprocessor(&pc0, k0, pl.nt, pl.lds) == hipSuccess &&
             hipOccupancyMaxActiveBlocksPerMultiprocessor(&pc1, kt, pl.nt, with) == hipSuccess;
      help_stage = take && pc1 >= std::min(pc0, max_wg);
      take = take && pc1 >= pc0;
    } else {
      help_stage = take;
    }
    if (take) {
      pl.tl = tl;
      pl.tbytes = ((o->table_lds_bytes + 15) / 16) * 16;
      pl.lds = with;
    }
  }
  // At most one conformer per CU: the time is the longest conformer's, so its workgroup gets
  // helper threads, and L-BFGS its history in LDS where that fits (both leave the results as
  // they are). The bonded tables are staged: ten conformers of 82 atoms 4.65 -> 4.48 ms (L-BFGS), 5.61 ->
  // 5.50 (BFGS). Where the rule above does not stage, a caller whose reserve is smaller than a molecule's
  // tables gets results all the same and must keep getting them: there BFGS takes the kernel that reads such
  // tables from memory (six ragged conformers 15.7 ms, 16.1 unstaged; its second copy of the evaluation
  // costs other batches up to 2%, so they keep the plain one), and L-BFGS, which staging gains nothing
  // there, none. The bonded
  // terms' energies take a word each; a bonded term has at least 12 table bytes, so
  // table_lds_bytes bounds their number (eval_help takes more in windows). Ten conformers of 48 atoms, BFGS,
  // host work included: 4.28 -> 3.99 ms; 221 chains of 199-329 atoms, L-BFGS: 180 -> 127 ms (151 with
  // the history in LDS alone); with the bonded tasks' spread terms 3.95 and 116 ms. A helped
  // workgroup takes its CU's twelve waves, so with more conformers than CUs they queue: 257
  // conformers of 82 atoms, without and with helpers, BFGS 4.28 and 5.70 ms, L-BFGS 4.05 and 5.89;
  // 600: 6.25 and 10.1, 4.92 and 8.76.
  if (b->n_confs <= di.n_cu && o->table_lds_bytes > 0) {
    const int eb = (o->table_lds_bytes / 12 + 64) & ~63, stage = help_stage ? 2 : 3;
    const struct {
      int hm, tl;
    } tries[] = {{0, stage}, {0, 0}, {pl.hm, stage}, {pl.hm, 0}};
    for (const auto& t : tries) {
      if (t.hm == 0 && o->algo != MMFFHIP_LBFGS) continue;
      const int tb = t.tl ? ((o->table_lds_bytes + 15) / 16) * 16 : 0;
      const size_t lds = nk_lds_bytes(o->algo, t.hm, pl.nt, pl.max_n, m, (size_t)tb, NK_HELP, eb);
      if (!nk_kernel(o->algo, t.hm, t.tl, pl.nt, NK_HELP) || lds > (size_t)di.lds) continue;
      pl.hm = t.hm;
      pl.tl = t.tl;
      pl.tbytes = tb;
      pl.help = NK_HELP;
      pl.eb_floats = eb;
      pl.lds = lds;
      break;
    }
  }
  const void* kp = nk_kernel(o->algo, pl.hm, pl.tl, pl.nt, pl.help);
  if (!kp) return fail(MMFFHIP_ERR_ARG, "no kernel instantiated for this (algo, placement, block) combination");
  allow_lds(kp, pl.lds);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kp, pl.nt * pl.help, pl.lds) != hipSuccess || per_cu < 1)
    per_cu = 1;
  // Twelve waves per CU at most, whatever registers a kernel leaves free: the resident Hessians
  // stay in the Infinity Cache, a fourth wave per SIMD gains 1% at best (100,000 ragged conformers
  // 1,084 -> 1,075 ms, 2,500 small ones 13.6 -> 15.0), and callers size their buckets by this grid.
  // (L-BFGS, which has no Hessian and 109 registers, would gain from sixteen: 8,000 medium conformers
  // 63.9 -> 54.5 ms, 2,000 chains the same.)
  per_cu = std::min(per_cu, std::max(1, max_wg / pl.help));
  pl.grid = std::max(1, std::min(b->n_confs, di.n_cu * per_cu));
  pl.slot_floats = 0;
  if (pl.hm != 0) {
    pl.slot_floats = o->algo == MMFFHIP_LBFGS ? (size_t)2 * m * pl.max_n
                     : pl.hm == 2             ? packed_floats(pl.max_n)
                     : pl.hm == 3             ? sym_slot_floats(pl.max_n)
                                              : (size_t)pl.max_n * pl.max_n;
    pl.slot_floats = (pl.slot_floats + 63) & ~(size_t)63;
  }
  return MMFFHIP_OK;
}

size_t nk_ws_bytes(const NkPlan& pl) { return 256 + (size_t)pl.grid * pl.slot_floats * 4; }

template <int ALGO, int HM, int TL, int NT, int HELP = 1>
void launch_nk_t(const KBatch& kb, const NkParams& P, const NkPlan& pl, hipStream_t s) {
  hipLaunchKernelGGL((k_minimize_nk<ALGO, HM, TL, NT, HELP>), dim3(pl.grid), dim3(NT * HELP), pl.lds, s, kb, P);
}

void launch_nk(int algo, const KBatch& kb, const NkParams& P, const NkPlan& pl, hipStream_t s) {
#define NKL(A, H, TL, T)                                          \
  if (algo == A && pl.hm == H && pl.tl == TL && pl.nt == T && pl.help == 1) { \
    launch_nk_t<A, H, TL, T>(kb, P, pl, s);                                   \
    return;                                                                   \
  }
#define NKLH(A, H, TL, T)                                                           \
  if (algo == A && pl.hm == H && pl.tl == TL && pl.nt == T && pl.help == NK_HELP) { \
    launch_nk_t<A, H, TL, T, NK_HELP>(kb, P, pl, s);                                \
    return;                                                                         \
  }
  NK_FOR_EACH(NKL)
  NK_HELP_EACH(NKLH)
#undef NKL
#undef NKLH
}

// Clear the work queue at the front of `workspace` with a fill kernel (graph-capture safe)
// and launch the plan's minimize kernel; the global slots follow the 256-byte queue header.
int run_nk(const mmffhip_batch* b, const mmffhip_nk_opts* o, const NkPlan& pl, const float* x_in, float* x_out,
           double* e_out, int32_t* status_out, int32_t* counters, const int32_t* order, void* workspace,
           hipStream_t s) {
  int32_t* queue = (int32_t*)workspace;
  hipLaunchKernelGGL(k_fill_i32, dim3(1), dim3(64), 0, s, queue, 8, 0);
  HIP_TRY(hipGetLastError());
  NkParams P;
  P.x_in = x_in;
  P.x_out = x_out;
  P.e_out = e_out;
  P.status = status_out;
  P.counters = counters;
  P.order = order;
  P.queue = queue;
  P.hglob = (float*)((char*)workspace + 256);
  P.slot_floats = pl.slot_floats;
  P.precond = o->precond;
  P.max_iters = o->max_iters;
  P.grad_tol = o->grad_tol;
  P.diel = o->diel;
  P.m = o->algo == MMFFHIP_LBFGS ? o->lbfgs_m : 1;
  P.max_n = pl.max_n;
  P.ls_grad = o->ls_grad;
  P.tbytes = pl.tl ? pl.tbytes : 0;
  P.eb_floats = pl.eb_floats;
  P.xcd_on = 0;
  for (int x = 0; x < 9; x++) P.xcd_off[x] = 0;
  if (o->xcd_offsets) {
    if (!order) return fail(MMFFHIP_ERR_ARG, "xcd_offsets need an order");
    int prev = 0;
    for (int x = 0; x < 9; x++) {
      const int v = o->xcd_offsets[x];
      if (v < prev || v > b->n_confs || (x == 0 && v != 0) || (x == 8 && v != b->n_confs))
        return fail(MMFFHIP_ERR_ARG, "xcd_offsets must rise from 0 to n_confs");
      P.xcd_off[x] = v;
      prev = v;
    }
    P.xcd_on = 1;
  }
  KBatch kb = to_kbatch(b);
  launch_nk(o->algo, kb, P, pl, s);
  HIP_TRY(hipGetLastError());
  return MMFFHIP_OK;
}

// Scratch of the allocation-free minimize entry point: the work-queue header and the
// per-workgroup global slots live in this file-scope device array (one copy per GPU, held
// until the process ends). Host code never passes `scratch` itself to a kernel: its address
// on each device comes from hipGetSymbolAddress, taken once per device on that device's
// first call.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)64 << 20;
__device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
void* g_scratch_ptr[MAX_DEVICES];
std::mutex g_scratch_mu;

int scratch_ptr(void** out) {
  int dev = 0;
  HIP_TRY(hipGetDevice(&dev));
  if (dev < 0 || dev >= MAX_DEVICES) return fail(MMFFHIP_ERR_DEVICE, "device ordinal out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    HIP_TRY(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) return fail(MMFFHIP_ERR_HIP, "hipGetSymbolAddress returned NULL for the scratch array");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return MMFFHIP_OK;
}

}  // namespace

// error reporting shared with the library's other translation units (not exported)
__attribute__((visibility("hidden"))) int mmffhip_set_error(int code, const char* msg) { return fail(code, msg); }
__attribute__((visibility("hidden"))) int mmffhip_lds_limit() { return dev_info().lds; }

// ====================================================================================
// extern "C" ABI
extern "C" {

int mmffhip_abi_version(void) { return MMFFHIP_ABI_VERSION; }

const char* mmffhip_last_error(void) { return g_last_error.c_str(); }

int mmffhip_device_info(int32_t* n_cu, int32_t* n_xcd, int32_t* lds_bytes) {
  DevInfo di = dev_info();
  if (!di.ok) return fail(MMFFHIP_ERR_DEVICE, "no HIP device");
  if (n_cu) *n_cu = di.n_cu;
  if (n_xcd) *n_xcd = 8;
  if (lds_bytes) *lds_bytes = di.lds;
  return MMFFHIP_OK;
}

int mmffhip_energy_grad(const mmffhip_batch* b, int family, int diel, const float* x, double* e_out,
                        double* e_terms, float* g_out, uint32_t term_mask, void* stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (b->n_confs == 0) return MMFFHIP_OK;
  if (!x || !e_out) return fail(MMFFHIP_ERR_ARG, "x and e_out are required");
  if (diel != 1 && diel != 2) return fail(MMFFHIP_ERR_ARG, "diel must be 1 or 2");
  if (family == MMFFHIP_FAMILY_MEGA && diel != 1)
    return fail(MMFFHIP_ERR_ARG, "the MEGA family has a constant dielectric only");
  KBatch kb = to_kbatch(b);
  hipStream_t s = (hipStream_t)stream;
  const bool tg = family == MMFFHIP_FAMILY_TG;
  if (!tg && family != MMFFHIP_FAMILY_MEGA) return fail(MMFFHIP_ERR_ARG, "unknown family");
  const auto launch = e_terms ? (tg ? launch_eg<FAM_TG, true> : launch_eg<FAM_MEGA, true>)
                              : (tg ? launch_eg<FAM_TG, false> : launch_eg<FAM_MEGA, false>);
  return launch(kb, x, e_out, e_terms, g_out, term_mask, tg ? diel : 1, s);
}

int mmffhip_minimize_nk_workspace(const mmffhip_batch* b, const mmffhip_nk_opts* o, size_t* bytes) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!bytes) return fail(MMFFHIP_ERR_ARG, "bytes is NULL");
  if (b->n_confs == 0) {
    *bytes = 256;
    return MMFFHIP_OK;
  }
  NkPlan pl;
  rc = make_nk_plan(b, o, pl);
  if (rc) return rc;
  *bytes = nk_ws_bytes(pl);
  return MMFFHIP_OK;
}

int mmffhip_minimize_nk_plan(const mmffhip_batch* b, const mmffhip_nk_opts* o, int32_t* grid, int32_t* block,
                             int32_t* lds_bytes, int32_t* hess_place) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!grid) return fail(MMFFHIP_ERR_ARG, "grid is NULL");
  NkPlan pl;
  rc = make_nk_plan(b, o, pl);
  if (rc) return rc;
  *grid = b->n_confs == 0 ? 0 : pl.grid;
  if (block) *block = pl.nt;
  if (lds_bytes) *lds_bytes = (int32_t)pl.lds;
  if (hess_place)
    *hess_place = pl.hm == 0   ? MMFFHIP_HESS_LDS
                  : pl.hm == 2 ? MMFFHIP_HESS_GLOBAL_PACKED
                  : pl.hm == 3 ? MMFFHIP_HESS_GLOBAL_SYM
                               : MMFFHIP_HESS_GLOBAL;
  return MMFFHIP_OK;
}

int mmffhip_minimize_nk(const mmffhip_batch* b, const mmffhip_nk_opts* o, const float* x_in, float* x_out,
                        double* e_out, int32_t* status_out, int32_t* counters, const int32_t* order,
                        void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (b->n_confs == 0) return MMFFHIP_OK;
  if (!x_in || !x_out || !e_out || !status_out || !workspace)
    return fail(MMFFHIP_ERR_ARG, "x_in, x_out, e_out, status_out and workspace are required");
  NkPlan pl;
  rc = make_nk_plan(b, o, pl);
  if (rc) return rc;
  if (workspace_bytes < nk_ws_bytes(pl)) return fail(MMFFHIP_ERR_SIZE, "workspace too small");
  if ((uintptr_t)workspace & 255) return fail(MMFFHIP_ERR_ARG, "workspace must be 256-byte aligned");
  return run_nk(b, o, pl, x_in, x_out, e_out, status_out, counters, order, workspace, (hipStream_t)stream);
}

int mmffhip_minimize_nk_noalloc(const mmffhip_batch* b, const mmffhip_nk_opts* o, const float* x_in, float* x_out,
                                double* e_out, int32_t* status_out, int32_t* counters, const int32_t* order,
                                void* stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (b->n_confs == 0) return MMFFHIP_OK;
  if (!x_in || !x_out || !e_out || !status_out)
    return fail(MMFFHIP_ERR_ARG, "x_in, x_out, e_out and status_out are required");
  NkPlan pl;
  rc = make_nk_plan(b, o, pl);
  if (rc) return rc;
  // The persistent grid is capped to the global slots that fit beside the queue header; a
  // plan needs at least one slot per compute unit (fewer would leave CUs idle), else the
  // batch's molecules are too large for the array and the call is refused.
  if (pl.slot_floats > 0) {
    const size_t slot_bytes = pl.slot_floats * 4;
    const size_t fit = (NOALLOC_SCRATCH_BYTES - 256) / slot_bytes;
    const size_t need = (size_t)std::min(pl.grid, dev_info().n_cu);
    if (fit < need)
      return fail(MMFFHIP_ERR_SIZE, "mmffhip_minimize_nk_noalloc: " + std::to_string(need) + " slots of " +
                                        std::to_string(slot_bytes) + " bytes (one per compute unit) exceed its 64 MiB "
                                        "scratch; use mmffhip_minimize_nk with a workspace, or a smaller largest molecule");
    pl.grid = (int)std::min<size_t>((size_t)pl.grid, fit);
  }
  void* ws = nullptr;
  rc = scratch_ptr(&ws);
  if (rc) return rc;
  return run_nk(b, o, pl, x_in, x_out, e_out, status_out, counters, order, ws, (hipStream_t)stream);
}

int mmffhip_bb_fused(const mmffhip_batch* b, const float* x_in, float* x_out, double* e_out, int32_t max_iters,
                     float max_step, float grad_lr, void* stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (b->n_confs == 0) return MMFFHIP_OK;
  if (!x_in || !x_out || !e_out) return fail(MMFFHIP_ERR_ARG, "x_in, x_out and e_out are required");
  if (max_iters < 0) return fail(MMFFHIP_ERR_ARG, "max_iters must be >= 0");
  const DevInfo di = dev_info();
  const size_t rest = RED_WORDS * 8 + (size_t)3 * b->max_atoms * (8 + 3 * 4) + 16;
  // the largest molecule is what it was when the LDS held the gradient too
  if (rest + (size_t)3 * b->max_atoms * 4 > (size_t)di.lds)
    return fail(MMFFHIP_ERR_SIZE, "molecule too large for the LDS of one workgroup");
  KBatch kb = to_kbatch(b);
  // at most one conformer per CU and molecules that are not small: sixteen waves each, as in
  // launch_eg. One conformer, 200 steps, four waves and sixteen: 9 atoms 0.43 and 0.55 ms, 33 atoms
  // 0.46 and 0.58 (one step of pairs), 36 atoms 0.57 and 0.59, 39 atoms 0.58 and 0.59 or 0.68 and 0.63 (a chain; three
  // rings), 48 atoms 0.69 and 0.66, 82 atoms 1.28 and 0.91, 253 atoms 7.35 and 3.98; 300 conformers of 82 atoms 1.68
  // and 1.84
  const size_t wide_ex = ex_area(1024, 0, 2, rest, di.lds);
  const bool wide = b->n_confs <= di.n_cu && b->max_atoms > 38 && rest + wide_ex <= (size_t)di.lds;
  const size_t ex = wide ? wide_ex : 0;
  const auto kernel = wide ? k_bb_fused<1024> : k_bb_fused<256>;
  allow_lds((const void*)kernel, rest + ex);
  hipLaunchKernelGGL(kernel, dim3(b->n_confs), dim3(wide ? 1024 : 256), rest + ex, (hipStream_t)stream, kb, x_in, x_out,
                     e_out, (int)max_iters, max_step, grad_lr, (int)ex);
  HIP_TRY(hipGetLastError());
  return MMFFHIP_OK;
}

int mmffhip_multimol_workspace(const mmffhip_batch* b, int32_t lbfgs_m, size_t* bytes) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (!bytes) return fail(MMFFHIP_ERR_ARG, "bytes is NULL");
  if (lbfgs_m < 1 || lbfgs_m > 64) return fail(MMFFHIP_ERR_ARG, "lbfgs_m must be in [1, 64]");
  // the total coordinate count is not known on the host without a device read; the
  // workspace is sized with n_confs * 3 * max_atoms as an upper bound
  const size_t T = (size_t)b->n_confs * 3 * b->max_atoms;
  const size_t C = (size_t)b->n_confs;
  auto r256 = [](size_t v) { return (v + 255) & ~(size_t)255; };
  size_t by = 0;
  by += 3 * r256(T * 4) + 2 * r256(T * 4 * (size_t)lbfgs_m);
  by += r256(C * 8 * (size_t)lbfgs_m) + 2 * r256(C * 8) + r256(C * 8) + 2 * r256(C * 4);
  by += r256(4096 * 4);
  *bytes = by + 1024;
  return MMFFHIP_OK;
}

int mmffhip_multimol_run(const mmffhip_batch* b, const float* x_in, float* x_best, double* e_final, float* grad_norm,
                         int32_t* per_conf_iters, int32_t* converged, int32_t* iters_used, int32_t max_iters,
                         int32_t eval_freq, float max_step_per_atom, int32_t lbfgs_m, float grad_scale,
                         float grad_tol, void* workspace, size_t workspace_bytes, void* stream) {
  return mmffhip_multimol_run_ex(b, x_in, x_best, e_final, grad_norm, per_conf_iters, converged, iters_used, max_iters,
                                 eval_freq, max_step_per_atom, lbfgs_m, grad_scale, grad_tol, 0, workspace,
                                 workspace_bytes, stream);
}

int mmffhip_multimol_run_ex(const mmffhip_batch* b, const float* x_in, float* x_best, double* e_final,
                            float* grad_norm, int32_t* per_conf_iters, int32_t* converged, int32_t* iters_used,
                            int32_t max_iters, int32_t eval_freq, float max_step_per_atom, int32_t lbfgs_m,
                            float grad_scale, float grad_tol, int32_t flags, void* workspace, size_t workspace_bytes,
                            void* stream) {
  int rc = check_batch(b);
  if (rc) return rc;
  if (b->n_confs == 0) return MMFFHIP_OK;
  if (!x_in || !x_best || !e_final || !grad_norm || !per_conf_iters || !converged || !iters_used || !workspace)
    return fail(MMFFHIP_ERR_ARG, "NULL output or workspace");
  if (max_iters < 0 || eval_freq < 1) return fail(MMFFHIP_ERR_ARG, "max_iters >= 0 and eval_freq >= 1 required");
  size_t need = 0;
  rc = mmffhip_multimol_workspace(b, lbfgs_m, &need);
  if (rc) return rc;
  if (workspace_bytes < need) return fail(MMFFHIP_ERR_SIZE, "workspace too small");
  if (flags & ~(int32_t)MMFFHIP_MM_BATCH) return fail(MMFFHIP_ERR_ARG, "unknown multimol flags");
  const bool batch = (flags & MMFFHIP_MM_BATCH) != 0;
  const int n_main = (max_iters + eval_freq - 1) / eval_freq;
  const int polish = batch ? 0 : max_iters / 4;
  const int n_pol = (polish + eval_freq - 1) / eval_freq;
  if (n_main + n_pol > 4096) return fail(MMFFHIP_ERR_ARG, "too many sync points (max_iters / eval_freq > 4096)");
  const size_t T = (size_t)b->n_confs * 3 * b->max_atoms;
  const size_t C = (size_t)b->n_confs;
  char* p = (char*)workspace;
  auto take = [&](size_t bytes) {
    char* q = p;
    p += (bytes + 255) & ~(size_t)255;
    return (void*)q;
  };
  MMState S;
  S.total = T;
  S.x = (float*)take(T * 4);
  S.g = (float*)take(T * 4);
  S.bx = (float*)take(T * 4);
  S.S = (float*)take(T * 4 * lbfgs_m);
  S.Y = (float*)take(T * 4 * lbfgs_m);
  S.rho = (double*)take(C * 8 * lbfgs_m);
  S.best_e = (double*)take(C * 8);
  S.e_new = (double*)take(C * 8);
  S.ring = (int32_t*)take(C * 8);
  S.conv = (int32_t*)take(C * 4);
  S.pci = (int32_t*)take(C * 4);
  S.flags = (int32_t*)take(4096 * 4);
  if ((size_t)(p - (char*)workspace) > workspace_bytes) return fail(MMFFHIP_ERR_SIZE, "workspace too small");
  hipStream_t s = (hipStream_t)stream;
  KBatch kb = to_kbatch(b);
  constexpr int NT = 256;
  const int mx = 3 * b->max_atoms;
  const size_t lds_init = 16 * (NT / 64) * 8 + (size_t)mx * (8 + 4) + 16;
  const DevInfo di = dev_info();
  const MMChunk ck = mm_chunk_plan(b->n_confs, mx, lbfgs_m, di);
  if (ck.lds > (size_t)di.lds) return fail(MMFFHIP_ERR_SIZE, "molecule too large for one workgroup");
  allow_lds((const void*)&k_mm_init<NT>, lds_init);
  allow_lds((const void*)ck.kernel, ck.lds);
  allow_lds((const void*)&k_mm_final<NT>, lds_init);
  hipLaunchKernelGGL(k_fill_i32, dim3((4096 + 255) / 256), dim3(256), 0, s, S.flags, 4096, 0);
  hipLaunchKernelGGL((k_mm_init<NT>), dim3(b->n_confs), dim3(NT), lds_init, s, kb, S, x_in, grad_scale, 0,
                     (int)max_iters);
  HIP_TRY(hipGetLastError());
  int it = 0, k = 0;
  while (it < max_iters) {
    int steps = std::min(eval_freq, max_iters - it);
    it += steps;
    const bool sync = (it % eval_freq) == 0;
    // the batch form has no convergence exit: no conformer ever passes the test (tolerance
    // -1) and no launch reads the previous sync point's count
    hipLaunchKernelGGL(ck.kernel, dim3(b->n_confs), dim3(ck.nr), ck.lds, s, kb, S, steps, it, sync ? 1 : 0,
                       0, (k > 0 && !batch) ? S.flags + (k - 1) : (const int32_t*)nullptr, S.flags + k,
                       (int)lbfgs_m, max_step_per_atom, grad_scale, batch ? -1.0f : grad_tol, ck.q_bytes);
    if (sync) k++;
  }
  HIP_TRY(hipGetLastError());
  if (!batch)
    hipLaunchKernelGGL((k_mm_init<NT>), dim3(b->n_confs), dim3(NT), lds_init, s, kb, S, x_in, grad_scale, 1,
                       (int)max_iters);
  it = 0;
  int kp = n_main;
  while (it < polish) {
    int steps = std::min(eval_freq, polish - it);
    it += steps;
    const bool sync = (it % eval_freq) == 0;
    hipLaunchKernelGGL(ck.kernel, dim3(b->n_confs), dim3(ck.nr), ck.lds, s, kb, S, steps, it, sync ? 1 : 0,
                       1, kp > n_main ? S.flags + (kp - 1) : (const int32_t*)nullptr, S.flags + kp, (int)lbfgs_m,
                       max_step_per_atom, grad_scale, grad_tol, ck.q_bytes);
    if (sync) kp++;
  }
  HIP_TRY(hipGetLastError());
  hipLaunchKernelGGL((k_mm_final<NT>), dim3(b->n_confs), dim3(NT), lds_init, s, kb, S, x_best, e_final, grad_norm,
                     per_conf_iters, converged, iters_used, batch ? 0 : (int)(max_iters / eval_freq),
                     (int)eval_freq, (int)max_iters, batch ? 1 : 0);
  HIP_TRY(hipGetLastError());
  return MMFFHIP_OK;
}

}  // extern "C"
