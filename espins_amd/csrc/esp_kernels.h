// esp_kernels.h -- sweep, measurement, exchange and energy kernels (gfx950, wave64).
//
// Device layout of one replica r (N sites, colour-major device order, stride Ns > N):
//   x[Ns], y[Ns], z[Ns]  spin components (structure of arrays: a gather of a partner spin
//                     is three 8-byte loads whose addresses are contiguous across a wave);
//                     index N holds a zero spin that padded bond slots point at
//   wpart[ncol][nw]   sum of the accepted dE of the sites of one wave of one colour phase
//                     since the last rebase, so the running energy ("by adding differences",
//                     mcarlo.F90:748) is e_base[r] + sum wpart, reproducibly (one writer per
//                     entry per phase, phases ordered by launches)
// Bonds: nbr[zmax][N] device partner indices (self-padded); coefficients per (basis, slot)
// in LDS when the lattice is periodic, else cJ/cB[zmax][N], cD[zmax][N][3].
#pragma once
#include <cstdint>
#include <vector>

#include "esp_device.h"
#include "esp_geo.h"
#include "esp_model.h"

namespace espk {
struct Clock {                   // device-side schedule counters (graph-replayable)
  unsigned long long sweep;      // Philox sweep counter of the next sweep
  unsigned long long step;       // exchange step counter
  int parity;                    // next exchange start (1 or 2)
  int pad;
};

namespace {  // internal linkage: each translation unit that launches these owns its copies
using namespace espd;

constexpr int kBlock = 256;      // reduce and measurement kernels (4 waves)
constexpr int kPhaseBlock = 256; // colour-phase kernels (64 and 512 measured the same, 1024 slower)
// Launches of a round that is captured into a graph at most.  The captured chain has a node per
// launch, and 528k of them ended in a segmentation fault of the host (within the runtime, whose graph
// calls most likely recurse along the chain).  A longer round is launched as it is; the host enqueues
// a launch in 3 us or less, the shortest phases take 4.
constexpr int64_t kCaptureMax = 4096;
constexpr int kLdsBlock = 512;   // LDS-resident kernel (8 waves per replica)
// Tuning constants (compile-time; the defaults are the measured best on MI355X).  Fewer
// gathers in flight per lane means fewer registers and more waves per SIMD, which hides the
// gather latency better than a wide chunk does: FCC 32^3 x 64, us per step with 2 / 3 / 4 in
// flight: 361 / 335 / 363; FCC 16^3 x 64 (two waves per SIMD) with 4 / 6 / 8: 139 / 133 / 150.
#ifndef ESP_CHUNK
#define ESP_CHUNK 3
#endif
#ifndef ESP_CHUNK_WIDE
#define ESP_CHUNK_WIDE 6
#endif
#ifndef ESP_PHASE_WAVES
#define ESP_PHASE_WAVES 0        // > 0: ask the compiler for this many waves per SIMD
#endif
#if ESP_PHASE_WAVES > 0
#define ESP_PHASE_ATTR __attribute__((amdgpu_waves_per_eu(ESP_PHASE_WAVES)))
#else
#define ESP_PHASE_ATTR
#endif
constexpr int kChunk = ESP_CHUNK;  // partner gathers issued together per lane
constexpr int kChunkWide = ESP_CHUNK_WIDE;  // ... for launches too small to fill the GPU with waves
constexpr int kChunkLds = 3;     // ... in the LDS-resident sweep
#ifndef ESP_CHUNK_LEARN
#define ESP_CHUNK_LEARN 8
#endif
constexpr int kChunkLearn = ESP_CHUNK_LEARN;  // ... in the learned sweep
// Rejections are counted per slot in kRejSub sub-counters, rej[kRejSub][R]: a wave adds to the
// sub-counter its global wave index selects.  Atomics on one 128-byte line queue at about 30
// cycles each, and a replica's waves run together on one XCD, so the sub-counters of a slot lie
// on different lines: with 16 of them side by side in one line the queue bounded the sweep of
// SC 64^3 x 32 (J + B + DM): 111 us per colour phase, 76 us so.  Readers sum the sub-counters.
constexpr int kRejSub = 32;
// Dynamic LDS of the LDS-resident kernel: [N+1 spins as double4][coefficient table]
// [kLdsRed doubles of reduction scratch]; every byte of LDS it uses is in that one region.
constexpr int kLdsRed = 4 * (512 / 64);

struct KArgs {
  double *sp;                    // [R][3][Ns]
  double *w;                     // [R][ncol][mpart_nw] per-wave accepted-dE sums
  const int *nbr;
  const double *cJ, *cB, *cD;
  const double *ctab;            // [nb][zmax][5]
  const double *mag;
  const uint8_t *basis;
  const int *dev2ref;
  const int *col_off;
  const double *si4, *h4;
  const double *beta_slot;
  const int *rep_slot;
  unsigned long long *rej;
  const Clock *clock;
  const double *prop, *unif;     // host-fed mode, reference order
  uint8_t *accepted;
  int N, Ns, nb, zmax, R, ncol;
  int c_begin, c_count, nblk;
  espg::FastDiv dnblk;           // by nblk
  int has_si, has_h;
  unsigned xcd_full;             // blocks of the replicas that keep to one XCD (espg::place_block)
  int sweep_off, tps;            // tps: lanes cooperating on one site (1, 2, 4, 8)
  double tilt;
  uint32_t key0, key1, stream_base;
  // per-wave sums of the spins after each colour phase, or null: mpart[R][ncol][mpart_nw][3];
  // phase `col` overwrites its waves' entries
  double *mpart;
  int col, mpart_nw;
  // implicit geometry (esp_geo.h): group records, bond lists and their coefficients (SegTables in
  // esp_model.h); ngc geometry groups make up the colour, cut into tseg tiles of spt sites each, taken in runs
  espg::Geo geo;
  const int *grp, *gcnt;             // [ngroups]
  const unsigned long long *gbond;   // [ngroups][zmax]
  const double *gcoef;               // [ngroups][zmax][1 + has_B + 3 has_D]
  int tseg, spt, run;
  espg::FastDiv drun, dngc;
  const espg::FastDiv *cngc;         // [ncol]: dngc of every colour (batched launches)
};

enum { M_RANDOM = 0, M_CONST = 1, M_HOSTFED = 2 };

// Global-memory access through address space 1.  A pointer that a kernel reads out of a
// struct in memory (the batched kernels' per-chain arguments) is a generic pointer to the
// compiler, which then emits flat instructions; a flat load also counts against the LDS wait
// counter, so every LDS read after it waits for all gathers in flight.  Accesses through these
// helpers are global loads, stores and atomics.
#define ESP_GLOBAL __attribute__((address_space(1)))
template <class T>
__device__ __forceinline__ T gldi(const T *p, size_t i) {
  return ((const ESP_GLOBAL T *)p)[i];
}
template <class T>
__device__ __forceinline__ void gsti(T *p, size_t i, T v) {
  ((ESP_GLOBAL T *)p)[i] = v;
}
template <class T>
__device__ __forceinline__ void gadd(T *p, T v) {     // no-return atomic add, device scope
  __hip_atomic_fetch_add((ESP_GLOBAL T *)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What blocks of one launch hand to each other: agent-scope atomic loads and stores act at the
// GPU's coherence point, past the L1s and the XCDs' L2s, and stores_done waits until a wave's own
// have been acknowledged there.  No cache needs writing back or invalidating, which agent-scope
// release and acquire fences do for whole caches.
template <class T>
__device__ __forceinline__ T ald(const T *p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
template <class T>
__device__ __forceinline__ void ast(T *p, T v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void stores_done() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// 32-bit byte offset from a wave-uniform base: lets the compiler use the SGPR-base
// addressing form (one VGPR offset per lane, no 64-bit address arithmetic).  The host keeps
// every table and replica below 4 GiB.
template <class T>
__device__ __forceinline__ T ld_off(const T *base, unsigned byte_off) {
  return *(const ESP_GLOBAL T *)((const ESP_GLOBAL char *)base + byte_off);
}

// Scalar load of a wave-uniform element that the launch does not write.
template <class T>
__device__ __forceinline__ T cldi(const T *p, size_t i) {
  return ((const __attribute__((address_space(4))) T *)p)[i];
}

struct GSpins {                  // one replica in global memory
  double *x, *y, *z;
  __device__ __forceinline__ V3 ld(unsigned j) const {
    const unsigned o = j * 8u;
    return {ld_off(x, o), ld_off(y, o), ld_off(z, o)};
  }
  __device__ __forceinline__ void st(unsigned j, const V3 &v) const {
    gsti(x, j, v.x); gsti(y, j, v.y); gsti(z, j, v.z);
  }
};
struct LSpins {                  // one replica in LDS (x, y, z, w)
  double4 *p;
  __device__ __forceinline__ V3 ld(unsigned j) const { const double4 t = p[j]; return {t.x, t.y, t.z}; }
};

struct Proposal {
  V3 so, sn;
  double u3;
};

// What the update of one site needs besides the spins: device index, reference index (the
// Philox counter and the host-fed arrays use it), basis atom and moment.
struct Site {
  int d, ir, a;
  double mag;
};

__device__ __forceinline__ Site site_info(const KArgs &a, int d) {
  return {d, gldi(a.dev2ref, d), gldi(a.basis, d), gldi(a.mag, d)};
}

// Proposal of one attempted update (identical on every lane of the site's group).
template <int MODE, class SP>
__device__ __forceinline__ Proposal propose(const KArgs &a, const SP &sp, const Site &st, int r,
                                            unsigned long long sweep) {
  Proposal p;
  p.so = sp.ld(st.d);
  const int ir = st.ir;
  if (MODE == M_HOSTFED) {
    const size_t q = 3 * ((size_t)r * a.N + ir);
    p.sn = {gldi(a.prop, q), gldi(a.prop, q + 1), gldi(a.prop, q + 2)};
    p.u3 = gldi(a.unif, (size_t)r * a.N + ir);
  } else {
    const uint4 rn = philox10(make_uint4((uint32_t)ir, (uint32_t)sweep, (uint32_t)(sweep >> 32),
                                         a.stream_base + (uint32_t)r),
                              a.key0, a.key1);
    p.sn = MODE == M_RANDOM ? propose_random(st.mag, u01(rn.x), u01(rn.y))
                            : propose_const(st.mag, p.so, a.tilt, u01(rn.x), u01(rn.y));
    p.u3 = u01(rn.z);
  }
  return p;
}

// How a wave finds its sites' bonds: per-bond coefficient tables and the partner table; the
// per-(basis, slot) coefficient table in LDS and the partner table; or, for a tile inside one
// geometry group, the group's bond list (scalar loads) and computed partners.
enum { LAY_BOND = 0, LAY_CMP = 1, LAY_IMP = 2 };

// One bond's contribution to the J, B, D sums of delta_energy_get (get_quant.F90:288-336).
// crow: the site's row of the coefficient table (LAY_CMP: in LDS; LAY_IMP: the group's list in
// global memory, wave-uniform; unused with per-bond tables).
template <int LAY, bool HB, bool HD>
__device__ __forceinline__ void bond_term(const KArgs &a, const double *crow, int l, int d,
                                          const V3 &ds, const V3 &si, const V3 &sj, double &eJ,
                                          double &eB, double &eD) {
  double cj, cb = 0.0, cx = 0.0, cy = 0.0, cz = 0.0;
  if (LAY == LAY_IMP) {
    constexpr int NC = 1 + (HB ? 1 : 0) + (HD ? 3 : 0), oD = HB ? 2 : 1;
    cj = cldi(crow, NC * l);
    if (HB) cb = cldi(crow, NC * l + 1);
    if (HD) { cx = cldi(crow, NC * l + oD); cy = cldi(crow, NC * l + oD + 1); cz = cldi(crow, NC * l + oD + 2); }
  } else if (LAY == LAY_CMP) {
    cj = crow[5 * l];
    if (HB) cb = crow[5 * l + 1];
    if (HD) { cx = crow[5 * l + 2]; cy = crow[5 * l + 3]; cz = crow[5 * l + 4]; }
  } else {
    cj = gldi(a.cJ, (size_t)l * a.N + d);
    if (HB) cb = gldi(a.cB, (size_t)l * a.N + d);
    if (HD) {
      const size_t q = 3 * ((size_t)l * a.N + d);
      cx = gldi(a.cD, q); cy = gldi(a.cD, q + 1); cz = gldi(a.cD, q + 2);
    }
  }
  const double dsj = dot(ds, sj);
  eJ = eJ - cj * dsj;
  if (HB) {
    const double sij = dot(si, sj);
    eB = eB + cb * (dsj * dsj + 2.0 * sij * dsj);
  }
  if (HD)  // D . (dS x S_j)  (utility_cross, utility.F90:212-234)
    eD = eD + (cx * (ds.y * sj.z - ds.z * sj.y) + cy * (ds.z * sj.x - ds.x * sj.z) +
               cz * (ds.x * sj.y - ds.y * sj.x));
}

// Partner indices of a site's first chunk (bond_sums).
template <int CH>
__device__ __forceinline__ void first_bonds(const KArgs &a, int d, int g, unsigned (&jn)[CH]) {
  const int tps = a.tps, nk = (a.zmax - g + tps - 1) / tps;
#pragma unroll
  for (int u = 0; u < CH; ++u) {
    const int l = u < nk ? g + tps * u : g;
    jn[u] = nk > 0 ? (unsigned)ld_off(a.nbr, ((unsigned)l * (unsigned)a.N + (unsigned)d) * 4u) : 0u;
  }
}
// Partial bond sums over the slots l = g, g+tps, ... of site st.  Inactive lanes return
// zeros.  Slots go in chunks of CH: the CH partner indices of the next chunk are loaded
// while the current chunk's CH partner gathers are in flight, so a
// wave waits for one gather round trip per chunk.  Full chunks need no masks; only the last
// partial chunk is masked (its spare lanes re-read slot g).  Padded slots point at the zero
// spin (index N), so they need no test; a self bond (SELF) reads the new spin.
template <int CH, bool CMP, bool HB, bool HD, bool SELF, class SP>
__device__ __forceinline__ void bond_sums(const KArgs &a, const SP &sp, const double *ctab, const Site &st,
                                          bool active, int g, const Proposal &p, unsigned (&jn)[CH], double &eJ,
                                          double &eB, double &eD) {
  constexpr int LAY = CMP ? LAY_CMP : LAY_BOND;
  eJ = 0.0; eB = 0.0; eD = 0.0;
  if (!active) return;
  const int d = st.d;
  const V3 ds = sub(p.sn, p.so);
  const V3 si = sub(p.sn, ds);  // old spin as the reference recovers it (get_quant.F90:306,320)
  const int tps = a.tps;
  const int nk = (a.zmax - g + tps - 1) / tps;
  const int nfull = nk - nk % CH;
  const double *crow = CMP ? ctab + (size_t)st.a * a.zmax * 5 : nullptr;
  const unsigned ud = (unsigned)d;
  // (jn: partner indices of the next chunk; the first was loaded by first_bonds)
  auto load_idx = [&](int k0) {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int l = k0 + u < nk ? g + tps * (k0 + u) : g;
      jn[u] = (unsigned)ld_off(a.nbr, ((unsigned)l * (unsigned)a.N + ud) * 4u);
    }
  };
  for (int k0 = 0; k0 < nfull; k0 += CH) {
    V3 sv[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const V3 t = sp.ld(jn[u]);
      sv[u] = (SELF && jn[u] == ud) ? p.sn : t;
    }
    if (k0 + CH < nk) load_idx(k0 + CH);
#pragma unroll
    for (int u = 0; u < CH; ++u) bond_term<LAY, HB, HD>(a, crow, g + tps * (k0 + u), d, ds, si, sv[u], eJ, eB, eD);
  }
  const int rem = nk - nfull;
  if (rem > 0) {
    V3 sv[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const V3 t = sp.ld(jn[u]);
      sv[u] = (SELF && jn[u] == ud) ? p.sn : t;
    }
#pragma unroll
    for (int u = 0; u < CH; ++u)
      if (u < rem) bond_term<LAY, HB, HD>(a, crow, g + tps * (nfull + u), d, ds, si, sv[u], eJ, eB, eD);
  }
}

// The bond sums of a site of geometry group sg.g over the group's bond list (one lane per site;
// the group is the same for the whole wave).  The list is sorted by the partners' sub-cell
// shift, so a lane wraps its sub-cell coordinates once per distinct shift (at most 8 for nearest
// and next-nearest shells on a colouring of period 2) and a bond adds the partner group's first
// index: about 1 + 13 x 8 / z vector instructions per partner index, against 25 when every lane
// unpacked each slot's shift from a table in LDS.  Coefficients come as scalar loads, not LDS
// reads.  Lists hold real bonds only, no padding.
template <int CH, bool HB, bool HD, bool SELF>
__device__ __forceinline__ void bond_sums_geo(const KArgs &a, const GSpins &sp, const espg::SiteGeo &sg, const Site &st,
                                              const Proposal &p, double &eJ, double &eB, double &eD) {
  eJ = 0.0; eB = 0.0; eD = 0.0;
  const V3 ds = sub(p.sn, p.so);
  const V3 si = sub(p.sn, ds);  // old spin as the reference recovers it (get_quant.F90:306,320)
  constexpr int NC = 1 + (HB ? 1 : 0) + (HD ? 3 : 0);
  const int n = cldi(a.gcnt, sg.g);
  const unsigned long long *bl = a.gbond + (size_t)sg.g * a.zmax;
  const double *crow = a.gcoef + (size_t)sg.g * a.zmax * NC;
  const unsigned ud = (unsigned)st.d;
  const int nfull = n - n % CH;
  unsigned jn[CH], off = 0;
  auto load_idx = [&](int k0) {
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const unsigned long long e = cldi(bl, min(k0 + u, n - 1));
      const unsigned q = (unsigned)(e >> 32);
      if (q >> 31) off = (unsigned)espg::geo_shift(a.geo, sg, q);   // a new shift
      jn[u] = off + (unsigned)e;
    }
  };
  if (n > 0) load_idx(0);
  for (int k0 = 0; k0 < nfull; k0 += CH) {
    V3 sv[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const V3 t = sp.ld(jn[u]);
      sv[u] = (SELF && jn[u] == ud) ? p.sn : t;
    }
    if (k0 + CH < n) load_idx(k0 + CH);
#pragma unroll
    for (int u = 0; u < CH; ++u) bond_term<LAY_IMP, HB, HD>(a, crow, k0 + u, 0, ds, si, sv[u], eJ, eB, eD);
  }
  if (n > nfull) {
    V3 sv[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const V3 t = sp.ld(jn[u]);
      sv[u] = (SELF && jn[u] == ud) ? p.sn : t;
    }
#pragma unroll
    for (int u = 0; u < CH; ++u)
      if (nfull + u < n) bond_term<LAY_IMP, HB, HD>(a, crow, nfull + u, 0, ds, si, sv[u], eJ, eB, eD);
  }
}

// Sum over the tps lanes of a site's group: xor butterfly, bitwise identical on every lane.
__device__ __forceinline__ double group_sum(double v, int tps) {
  for (int o = 1; o < tps; o <<= 1) v += __shfl_xor(v, o, 64);
  return v;
}

__device__ __forceinline__ void rej_add(unsigned long long *rej, int R, int slot, unsigned long long n) {
  // blocks of one replica are 8 apart (one XCD)
  const unsigned wv = ((blockIdx.x >> 3) * (blockDim.x >> 6) + (threadIdx.x >> 6)) & (kRejSub - 1);
  gadd(&rej[(size_t)wv * R + slot], n);
}

// Local terms and the accept test of metropolis (get_quant.F90:166-178): reject iff
// dE > 0 and exp(-beta dE) < u3.  Returns dE through *de.  UNI: the basis atom b is the same for
// the whole wave (scalar loads).
template <bool UNI = false>
__device__ __forceinline__ bool decide(const KArgs &a, int b, const Proposal &p, double eJ,
                                       double eB, double eD, double beta, double *de_out) {
  const V3 ds = sub(p.sn, p.so);
  const V3 si = sub(p.sn, ds);
  double de = eJ;
  auto ld4 = [&](const double *t, int k) { return UNI ? cldi(t, 4 * (size_t)b + k) : gldi(t, 4 * (size_t)b + k); };
  if (a.has_h) {
    const double h0 = ld4(a.h4, 0), h1 = ld4(a.h4, 1), h2 = ld4(a.h4, 2), h3 = ld4(a.h4, 3);
    de = de + h0 * (ds.x * h1 + ds.y * h2 + ds.z * h3);
  }
  if (a.has_si) {
    const double k0 = ld4(a.si4, 0), k1 = ld4(a.si4, 1), k2 = ld4(a.si4, 2), k3 = ld4(a.si4, 3);
    const double sa = si.x * k1 + si.y * k2 + si.z * k3;
    const double dsa = ds.x * k1 + ds.y * k2 + ds.z * k3;
    de = de + k0 * (dsa * dsa + 2.0 * sa * dsa);
  }
  de = de + eB;
  de = de + eD;
  *de_out = de;
  return (de > 0.0) && (exp(-beta * de) < p.u3);
}

// Lane moves of a double without LDS traffic: DPP within a row of 16 lanes, and the sum of a
// value with its neighbour row's / half wave's (v_permlane16_swap, v_permlane32_swap).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const int2 h = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_mov_dpp(h.x, CTRL, 0xf, 0xf, true),
                                              __builtin_amdgcn_mov_dpp(h.y, CTRL, 0xf, 0xf, true)));
}
__device__ __forceinline__ double add_rows(double v) {
  const int2 h = __builtin_bit_cast(int2, v);
  const auto x = __builtin_amdgcn_permlane16_swap(h.x, h.x, false, false);
  const auto y = __builtin_amdgcn_permlane16_swap(h.y, h.y, false, false);
  return __builtin_bit_cast(double, make_int2(x[0], y[0])) + __builtin_bit_cast(double, make_int2(x[1], y[1]));
}
__device__ __forceinline__ double add_halves(double v) {
  const int2 h = __builtin_bit_cast(int2, v);
  const auto x = __builtin_amdgcn_permlane32_swap(h.x, h.x, false, false);
  const auto y = __builtin_amdgcn_permlane32_swap(h.y, h.y, false, false);
  return __builtin_bit_cast(double, make_int2(x[0], y[0])) + __builtin_bit_cast(double, make_int2(x[1], y[1]));
}

// Sums of four values over the 64 lanes of a wave (every lane active): lane l returns the total
// of value {w, x, y, z}[l & 3].  The first two steps halve the number of values a lane carries
// (it keeps one half and hands the other to its neighbour), so the whole takes 7 additions
// instead of 24 -- with one butterfly per value the reduction was a seventh of a colour phase's
// vector instructions.  The order of the additions is fixed, so the result is reproducible.
__device__ __forceinline__ double wave_total4(double w, double x, double y, double z) {
  const bool odd = threadIdx.x & 1, hi = threadIdx.x & 2;
  const double p = (odd ? x : w) + dpp_f64<0xb1>(odd ? w : x);   // quad_perm [1,0,3,2]
  const double q = (odd ? z : y) + dpp_f64<0xb1>(odd ? y : z);
  double v = (hi ? q : p) + dpp_f64<0x4e>(hi ? p : q);           // quad_perm [2,3,0,1]
  v += dpp_f64<0x124>(v);                                        // row_ror:4
  v += dpp_f64<0x128>(v);                                        // row_ror:8
  return add_halves(add_rows(v));
}

// Per-wave sums of one colour phase: the accepted dE (added to the wave's accumulator, which
// the running energy sums) and the spins after the phase (stored; a site changes only in its
// own colour phase, so after a sweep these add up to the replica's magnetisation and the
// measurement reads them instead of every spin).  Fixed butterflies, one writer per entry: the
// wave loads its accumulator at its start (wave_old, latency hidden) and stores the sum.
// e: the wave's entry of its colour; a wave without an entry (past the colour's last lane) passes
// own = false.
__device__ __forceinline__ double wave_old(const KArgs &a, int r, int e, bool own) {
  return own ? gldi(a.w, ((size_t)r * a.ncol + a.col) * a.mpart_nw + e) : 0.0;
}
__device__ __forceinline__ void wave_sums(const KArgs &a, int r, int e, bool own, bool owner, bool rej, double de,
                                          const Proposal &p, double wold) {
  V3 sf = {0.0, 0.0, 0.0};
  if (owner) sf = rej ? p.so : p.sn;
  const double t = wave_total4(owner && !rej ? de : 0.0, sf.x, sf.y, sf.z);
  const int lane = threadIdx.x & 63;
  if (own && lane < 4) {
    const size_t i = ((size_t)r * a.ncol + a.col) * a.mpart_nw + e;
    if (lane == 0) {
      gsti(a.w, i, wold + t);
    } else if (a.mpart) {
      gsti(a.mpart, i * 3 + (lane - 1), t);
    }
  }
}

// Dynamic LDS of a colour-phase block: the coefficient table.
__host__ __device__ inline size_t phase_lds_bytes(int lay, int nb, int zmax) {
  return lay == LAY_CMP ? (size_t)nb * zmax * 5 * sizeof(double) : 0;
}

// Block b of colour phase (a.c_begin, a.c_count) of replica r (global-memory path, tables);
// a.tps lanes per site.  Shared by the single-context and the batched kernels.
template <int MODE, bool CMP, bool HB, bool HD, bool SELF, int CH>
__device__ __forceinline__ void phase_tab(const KArgs &a, int r, int b, double *s_ctab) {
  const int tps = a.tps;
  if (CMP) {
    const int n = a.nb * a.zmax * 5;
    for (int k = threadIdx.x; k < n; k += kPhaseBlock) s_ctab[k] = gldi(a.ctab, k);
    __syncthreads();
  }
  const int g = threadIdx.x & (tps - 1);
  const int k = (b * kPhaseBlock + threadIdx.x) / tps;
  const bool active = k < a.c_count;
  const int d = a.c_begin + (active ? k : 0);
  const int slot = gldi(a.rep_slot, r);
  const double beta = gldi(a.beta_slot, slot);
  const unsigned long long sweep = gldi(&a.clock->sweep, 0) + (unsigned long long)a.sweep_off;
  double *base = a.sp + (size_t)r * 3 * a.Ns;
  const GSpins sp{base, base + a.Ns, base + 2 * a.Ns};
  const Site st = site_info(a, d);
  const int wave = (b * kPhaseBlock + threadIdx.x) >> 6;
  const bool own = wave * 64 < a.c_count * tps;
  const double wold = wave_old(a, r, wave, own);
  Proposal p{};
  if (active) p = propose<MODE>(a, sp, st, r, sweep);
  double eJ, eB, eD;
  unsigned jn[CH];
  if (active) first_bonds(a, st.d, g, jn);
  bond_sums<CH, CMP, HB, HD, SELF>(a, sp, s_ctab, st, active, g, p, jn, eJ, eB, eD);
  eJ = group_sum(eJ, tps);
  if (HB) eB = group_sum(eB, tps);
  if (HD) eD = group_sum(eD, tps);
  bool rej = false;
  double de = 0.0;
  if (active) {
    rej = decide(a, st.a, p, eJ, eB, eD, beta, &de);
    if (g == 0) {
      if (MODE == M_HOSTFED) gsti(a.accepted, (size_t)r * a.N + st.ir, (uint8_t)(rej ? 0 : 1));
      if (!rej) sp.st(d, p.sn);
    }
  }
  const unsigned long long m = __ballot(rej && g == 0);
  if ((threadIdx.x & 63) == 0 && m) rej_add(a.rej, a.R, slot, (unsigned long long)__popcll(m));
  wave_sums(a, r, wave, own, active && g == 0, rej, de, p, wold);
}

// The same for a model with the implicit geometry, one lane per site: every wave takes one tile
// of at most 64 sites of one geometry group, so the group, its bond list, coefficients, basis
// atom, moment and local terms are wave-uniform (scalar loads) and nothing goes through LDS.
// The waves of a block take a run of up to `run` consecutive tiles of one group (their partners
// overlap in L1), consecutive runs the same place of the colour's next group, which is the same
// region of the lattice (its lines are in the XCD's L2).
// FCC 32^3 J1-J2 + B x 64 replicas (1 M updates per launch): 50 us with shifts and coefficients in
// LDS, 42 us so (25 G updates/s, 5.4 TB/s of minimal colour-phase traffic from the memory-side
// cache, which bounds it); SC 64^3 J + B + DM x 32 (4.2 M): 117 -> 76 us (55 G/s).
template <int MODE, bool HB, bool HD, bool SELF, int CH>
__device__ __forceinline__ void phase_geo(const KArgs &a, int r, int b) {
  const int t = __builtin_amdgcn_readfirstlane(b * (kPhaseBlock / 64) + (int)(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int mt = (int)a.geo.mt.d;
  const int q = (int)espg::fdiv((uint32_t)t, a.drun), cb = (int)espg::fdiv((uint32_t)q, a.dngc);
  const int gi = q - cb * (int)a.dngc.d;
  const int ch = cb * a.run + (t - q * a.run);              // tile of group gi of the colour
  if (ch >= a.tseg) return;                                 // a spare wave of a run
  const int first = a.c_begin + gi * mt;                    // the group's first site
  const int gg = (int)espg::fdiv((uint32_t)first, a.geo.mt);
  const int k = ch * a.spt + lane;                          // place inside the group
  const bool active = lane < a.spt && k < mt;
  const int slot = cldi(a.rep_slot, r);
  const double beta = cldi(a.beta_slot, slot);
  const unsigned long long sweep = cldi(&a.clock->sweep, 0) + (unsigned long long)a.sweep_off;
  double *base = a.sp + (size_t)r * 3 * a.Ns;
  const GSpins sp{base, base + a.Ns, base + 2 * a.Ns};
  const espg::SiteGeo sg = espg::geo_place(a.geo, cldi(a.grp, gg), gg, active ? k : ch * a.spt);
  const Site st{first + (active ? k : ch * a.spt), sg.ir, sg.a, cldi(a.mag, first)};
  const double wold = wave_old(a, r, gi * a.tseg + ch, true);
  Proposal p{};
  bool rej = false;
  double de = 0.0;
  if (active) {
    p = propose<MODE>(a, sp, st, r, sweep);
    double eJ, eB, eD;
    bond_sums_geo<CH, HB, HD, SELF>(a, sp, sg, st, p, eJ, eB, eD);
    rej = decide<true>(a, st.a, p, eJ, eB, eD, beta, &de);
    if (MODE == M_HOSTFED) gsti(a.accepted, (size_t)r * a.N + st.ir, (uint8_t)(rej ? 0 : 1));
    if (!rej) sp.st(st.d, p.sn);
  }
  const unsigned long long m = __ballot(rej);
  if (lane == 0 && m) rej_add(a.rej, a.R, slot, (unsigned long long)__popcll(m));
  wave_sums(a, r, gi * a.tseg + ch, true, active, rej, de, p, wold);
}

template <int MODE, int LAY, bool HB, bool HD, bool SELF, int CH = kChunk>
__device__ __forceinline__ void phase_body(const KArgs &a, int r, int b, double *s_ctab) {
  if (LAY == LAY_IMP) phase_geo<MODE, HB, HD, SELF, CH>(a, r, b);
  else phase_tab<MODE, LAY == LAY_CMP, HB, HD, SELF, CH>(a, r, b, s_ctab);
}

// One colour phase over every replica of one context.
template <int MODE, int LAY, bool HB, bool HD, bool SELF, int CH>
__global__ __launch_bounds__(kPhaseBlock) ESP_PHASE_ATTR void k_phase(KArgs a) {
  extern __shared__ double s_ctab[];
  int r, b;
  espg::place_block(blockIdx.x, a.xcd_full, a.dnblk, r, b);
  if (r >= a.R) return;  // uniform per block
  phase_body<MODE, LAY, HB, HD, SELF, CH>(a, r, b, s_ctab);
}

struct LdsMeas {
  double *acc;                   // [R][6] by slot
  double *e_run;                 // [R] by replica
  double *e_base;                // [R]: the launch's accepted dE is added at its end
  unsigned long long *nmeas;
  int measure_every;             // 0 = never
};

// Sums of v over the kLdsBlock threads, valid in wave 0; red: 4 values a wave.
__device__ __forceinline__ void block_total4(double (&v)[4], double *red) {
  constexpr int kW = kLdsBlock / 64;
  const int lane = threadIdx.x & 63;
  const double t = wave_total4(v[0], v[1], v[2], v[3]);
  if (lane < 4) red[4 * (threadIdx.x >> 6) + lane] = t;
  __syncthreads();
  if (threadIdx.x < 64) {
    double s = lane < 4 * kW ? red[lane] : 0.0;
#pragma unroll
    for (int off = 4; off < 4 * kW; off <<= 1) s += __shfl_xor(s, off);
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = __shfl(s, k);
  }
}

// All colours of nsweeps sweeps of one replica per block, spins resident in LDS,
// measurement (mcarlo.F90:536-543) fused every measure_every sweeps.
template <int MODE, bool CMP, bool HB, bool HD, bool SELF>
__device__ __forceinline__ void lds_body(const KArgs &a, int r, int nsweeps, const LdsMeas &m,
                                         double4 *s_sp) {
  double *ctab = reinterpret_cast<double *>(s_sp + a.N + 1);
  double *red = ctab + (CMP ? a.nb * a.zmax * 5 : 0);
  const double *gx = a.sp + (size_t)r * 3 * a.Ns;
  // w of a site in LDS: its accepted dE during this launch
  for (int d = threadIdx.x; d <= a.N; d += kLdsBlock)   // index N: the zero spin
    s_sp[d] = d < a.N ? make_double4(gldi(gx, d), gldi(gx, a.Ns + d), gldi(gx, 2 * (size_t)a.Ns + d), 0.0)
                      : make_double4(0.0, 0.0, 0.0, 0.0);
  if (CMP)
    for (int k = threadIdx.x; k < a.nb * a.zmax * 5; k += kLdsBlock) ctab[k] = gldi(a.ctab, k);
  // accepted dE the global-memory phases accumulated since the last rebase
  double wg[1] = {0.0};
  {
    const int ne = a.ncol * a.mpart_nw;
    const double *wr = a.w + (size_t)r * ne;
    for (int k = threadIdx.x; k < ne; k += kLdsBlock) wg[0] += gldi(wr, k);
  }
  block_sum<1>(wg, red);     // (its barriers also order the LDS fills above)
  const LSpins sp{s_sp};
  const int slot = gldi(a.rep_slot, r);
  const double beta = gldi(a.beta_slot, slot);
  const unsigned long long sweep0 = gldi(&a.clock->sweep, 0);
  const int tps = a.tps;
  const int g = threadIdx.x & (tps - 1);
  const int per = kLdsBlock / tps;
  // Colours of at most half a block: the two halves of the block (on the same SIMDs) take turns.
  // While one finishes a phase, the other draws its proposals of the next and loads its first
  // partner indices; a site's own spin changes only in its own phase.
  // (16 replicas of sc 8^3, 2 colours: 5.7 us a sweep without turns, 3.2 with; bcc 6^3, z = 14,
  // 12.2 and 7.4.  Three partner indices at a time: 6 gain 5 % for z = 6 and lose it for z = 14, 18.)
  constexpr int kHalf = kLdsBlock / 2;
  bool halves = a.ncol > 1;
  for (int c = 0; c < a.ncol; ++c) {
    const int n = gldi(a.col_off, c + 1) - gldi(a.col_off, c);
    halves &= n > 0 && n * tps <= kHalf;
  }
  const int half = __builtin_amdgcn_readfirstlane((int)threadIdx.x / kHalf);
  struct Turn {
    Site st;
    Proposal p;
    unsigned jn[kChunkLds];
    bool active;
  };
  auto begin = [&](int d0, int beg, int end, unsigned long long sweep) {
    Turn t;
    t.active = d0 < end;
    t.st = site_info(a, t.active ? d0 : beg);
    first_bonds(a, t.st.d, g, t.jn);
    t.p = Proposal{};
    if (t.active) t.p = propose<MODE>(a, sp, t.st, r, sweep);
    return t;
  };
  unsigned long long nrej = 0;   // 64-bit: one launch may run many sweeps at high rejection
  // The estimator sums of this replica's slot live in thread 0's registers during the
  // launch (same additions, same order as adding to memory each time) and are stored once
  // at the end: the sweep loop itself writes nothing but LDS.
  double A[6] = {0, 0, 0, 0, 0, 0};
  double e_last = 0.0;
  unsigned nmeas_local = 0;
  if (threadIdx.x == 0 && m.measure_every > 0)
    for (int k = 0; k < 6; ++k) A[k] = gldi(m.acc, 6 * slot + k);
  const double e_base = gldi(m.e_base, r);
  double w_launch = 0.0;      // thread 0: the launch's accepted dE at the last block sum
  auto finish = [&](Turn &t) {
    double eJ, eB, eD;
    bond_sums<kChunkLds, CMP, HB, HD, SELF>(a, sp, ctab, t.st, t.active, g, t.p, t.jn, eJ, eB, eD);
    eJ = group_sum(eJ, tps);
    if (HB) eB = group_sum(eB, tps);
    if (HD) eD = group_sum(eD, tps);
    if (!t.active) return;
    double de;
    const bool rej = decide(a, t.st.a, t.p, eJ, eB, eD, beta, &de);
    if (g != 0) return;
    if (rej) ++nrej;
    else {
      const double4 old = s_sp[t.st.d];
      s_sp[t.st.d] = make_double4(t.p.sn.x, t.p.sn.y, t.p.sn.z, old.w + de);
    }
  };
  Turn turn{};                 // (nobody's yet: inactive)
  int whose = 1;               // the half that finishes the phase (halves)
  for (int sw = 0; sw < nsweeps; ++sw) {
    // with halves, a phase -1 goes first, in which half 0 draws its proposals of phase 0
    for (int c = halves && sw == 0 ? -1 : 0; c < a.ncol; ++c) {
      const bool wrap = halves && c + 1 == a.ncol;
      const int cb = wrap ? 0 : halves ? c + 1 : c;            // the colour to begin
      const unsigned long long sweep = sweep0 + (unsigned long long)(sw + wrap);
      const int beg = gldi(a.col_off, cb), end = gldi(a.col_off, cb + 1);
      const int lane = halves ? (int)threadIdx.x & (kHalf - 1) : (int)threadIdx.x;
      for (int base = beg; base < end; base += per) {          // uniform trip count in the block
        if (!halves || half != whose) turn = begin(base + lane / tps, beg, end, sweep);
        if (!halves || half == whose) finish(turn);
      }
      whose ^= 1;
      __syncthreads();
    }
    const bool last = sw + 1 == nsweeps;
    const bool meas = m.measure_every > 0 && (sw + 1) % m.measure_every == 0;
    if (meas || last) {
      double v[4] = {0, 0, 0, 0};
      for (int d = threadIdx.x; d < a.N; d += kLdsBlock) {
        const double4 s = s_sp[d];
        v[0] += s.w; v[1] += s.x; v[2] += s.y; v[3] += s.z;
      }
      block_total4(v, red);
      if (threadIdx.x == 0) {
        const double e = e_base + wg[0] + v[0];
        w_launch = v[0];
        if (meas) {
          const double n = (double)a.N;
          const double mx = v[1] / n, my = v[2] / n, mz = v[3] / n;
          const double m2 = mx * mx + my * my + mz * mz;
          const double e2 = e * e;
          A[0] += e; A[1] += e2; A[2] += e2 * e2;
          A[3] += sqrt(m2); A[4] += m2; A[5] += m2 * m2;
          ++nmeas_local;
        }
        e_last = e;
      }
    }
  }
  if (threadIdx.x == 0) {
    if (nmeas_local) {
      for (int k = 0; k < 6; ++k) gsti(m.acc, 6 * slot + k, A[k]);
      if (r == 0) gsti(m.nmeas, 0, gldi(m.nmeas, 0) + nmeas_local);
    }
    if (nsweeps > 0) {
      gsti(m.e_run, r, e_last);
      gsti(m.e_base, r, e_base + w_launch);   // one block per replica: the only writer
    }
  }
  double *ox = a.sp + (size_t)r * 3 * a.Ns;
  for (int d = threadIdx.x; d < a.N; d += kLdsBlock) {
    const double4 s = s_sp[d];
    gsti(ox, d, s.x); gsti(ox, a.Ns + d, s.y); gsti(ox, 2 * (size_t)a.Ns + d, s.z);
  }
  unsigned long long v = nrej;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0 && v) rej_add(a.rej, a.R, slot, v);
}

template <int MODE, bool CMP, bool HB, bool HD, bool SELF>
__global__ __launch_bounds__(kLdsBlock) void k_lds(KArgs a, int nsweeps, LdsMeas m) {
  extern __shared__ double4 s_sp[];
  lds_body<MODE, CMP, HB, HD, SELF>(a, blockIdx.x, nsweeps, m, s_sp);
}

// Partial sums per (replica, block) for the running energy and m: the per-wave accepted-dE
// accumulators (ne entries per replica) and either the colour phases' per-wave spin sums
// (mpart, ne entries of 3) or, without them, the spins.  SHARED: read in the same launch (ald).
template <bool SHARED = false>
__device__ __forceinline__ void reduce_body(const double *sp, const double *wpart, int N, int Ns, int nblk,
                                            double *partial, const double *mpart, int ne, int r, int b) {
  __shared__ double red[4 * (kBlock / 64)];
  double v[4] = {0, 0, 0, 0};
  const int mc = (ne + nblk - 1) / nblk;
  const double *wr = wpart + (size_t)r * ne;
  for (int q = b * mc + threadIdx.x; q < min(ne, (b + 1) * mc); q += kBlock) v[0] += wr[q];
  if (mpart) {
    const double *mr = mpart + (size_t)r * ne * 3;
    for (int q = b * mc + threadIdx.x; q < min(ne, (b + 1) * mc); q += kBlock) {
      v[1] += mr[3 * q]; v[2] += mr[3 * q + 1]; v[3] += mr[3 * q + 2];
    }
  } else {
    const int chunk = (N + nblk - 1) / nblk;
    const int beg = b * chunk, end = min(N, beg + chunk);
    const double *x = sp + (size_t)r * 3 * Ns;
    for (int d = beg + threadIdx.x; d < end; d += kBlock) {
      v[1] += x[d]; v[2] += x[Ns + d]; v[3] += x[2 * Ns + d];
    }
  }
  block_sum<4>(v, red);
  if (threadIdx.x == 0)
    for (int k = 0; k < 4; ++k) {
      double *p = partial + ((size_t)r * nblk + b) * 4 + k;
      if (SHARED) ast(p, v[k]);
      else *p = v[k];
    }
}

__global__ __launch_bounds__(kBlock) void k_reduce(const double *sp, const double *wpart, int N, int Ns,
                                                   int nblk, double *partial, const double *mpart, int ne) {
  reduce_body(sp, wpart, N, Ns, nblk, partial, mpart, ne, blockIdx.y, blockIdx.x);
}

// e_base[r] += the sum of replica r's per-wave accumulators (fixed order); they are then zero.
// Used before the accumulators are re-laid out.
__global__ void k_fold_w(double *wpart, int ne, int R, double *e_base) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  double *w = wpart + (size_t)r * ne;
  double s = 0.0;
  for (int q = 0; q < ne; ++q) { s += w[q]; w[q] = 0.0; }
  e_base[r] += s;
}

struct FinArgs {
  const double *partial;         // [R][nblk][4] or null (e_run already fresh)
  int nblk, N, R;
  const double *e_base;
  double *e_run;
  double *acc;
  unsigned long long *nmeas;
  int *slot_rep, *rep_slot;
  const double *beta_slot;
  unsigned long long *nswap;     // [R][2]
  Clock *clock;
  int measure, exchange, advance_sweeps;
  uint32_t key0, key1, stream_base;
  double *trace;                 // [trace_cap][R][2] by slot: E, |m| per measurement, or null
  int trace_cap;
};

// Running energies / measurement, then the replica exchange (pt_swap, pt.F90:1235-1288)
// in label form.  One block per context; start parity and step come from the clock values
// the caller read.  SHARED: the partial sums were written in the same launch.
template <bool SHARED = false>
__device__ __forceinline__ void finalize_body(const FinArgs &f, int start, unsigned long long step) {
  if (f.partial)
    for (int r = threadIdx.x; r < f.R; r += blockDim.x) {
      double v[4] = {0, 0, 0, 0};
      const double *p = f.partial + (size_t)r * f.nblk * 4;
#pragma unroll 4
      for (int b = 0; b < f.nblk; ++b)
        for (int k = 0; k < 4; ++k) v[k] += SHARED ? ald(p + 4 * b + k) : p[4 * b + k];
      const double e = f.e_base[r] + v[0];
      f.e_run[r] = e;
      if (f.measure) {
        const double n = (double)f.N;
        const double mx = v[1] / n, my = v[2] / n, mz = v[3] / n;
        const double m2 = mx * mx + my * my + mz * mz;
        double *acc = f.acc + 6 * f.rep_slot[r];
        const double e2 = e * e;
        acc[0] += e; acc[1] += e2; acc[2] += e2 * e2;
        acc[3] += sqrt(m2); acc[4] += m2; acc[5] += m2 * m2;
        const unsigned long long k = f.nmeas[0];   // incremented after the barrier below
        if (f.trace && k < (unsigned long long)f.trace_cap) {
          double *t = f.trace + 2 * ((size_t)k * f.R + f.rep_slot[r]);
          t[0] = e;
          t[1] = sqrt(m2);
        }
      }
    }
  __syncthreads();
  if (f.exchange) {
    for (int t = start - 1 + 2 * threadIdx.x; t + 1 < f.R; t += 2 * blockDim.x) {
      const int ra = f.slot_rep[t], rb = f.slot_rep[t + 1];
      const double fac = (f.beta_slot[t] - f.beta_slot[t + 1]) * (f.e_run[ra] - f.e_run[rb]);
      bool sw = fac > 0.0;
      if (!sw) {
        const uint4 rn = philox10(make_uint4((uint32_t)t, (uint32_t)step, (uint32_t)(step >> 32),
                                             0xFFFFFFFFu - f.stream_base),
                                  f.key0 ^ 0x5bd1e995u, f.key1);
        sw = u01(rn.x) < exp(fac);
      }
      f.nswap[2 * t] += 1;
      f.nswap[2 * (t + 1)] += 1;
      if (sw) {
        f.slot_rep[t] = rb; f.slot_rep[t + 1] = ra;
        f.rep_slot[rb] = t; f.rep_slot[ra] = t + 1;
        f.nswap[2 * t + 1] += 1;
        f.nswap[2 * (t + 1) + 1] += 1;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0 && f.measure) f.nmeas[0] += 1;
}

__device__ __forceinline__ void advance_clock(Clock *c, bool exchange, int advance_sweeps) {
  if (exchange) {
    c->step += 1;
    c->parity = 3 - c->parity;
  }
  c->sweep += (unsigned long long)advance_sweeps;
}

__global__ __launch_bounds__(1024) void k_finalize(FinArgs f) {
  const int start = f.clock->parity;  // 1 or 2 (pt.F90:679,898)
  const unsigned long long step = f.clock->step;
  finalize_body(f, start, step);
  if (threadIdx.x == 0) advance_clock(f.clock, f.exchange, f.advance_sweeps);
}

// k_reduce followed by k_finalize in one launch: every block adds its partial sums
// (reduce_body); the last block to finish -- counted on a device-scope counter that it resets
// -- then runs finalize_body and advances the clock.  The partial sums move past the caches (ast,
// ald) and a block counts itself when its own are in place: with device fences, which write back
// the XCD's whole L2 with the spins that the sweep has just changed, it took 12.0 us for 64
// replicas of fcc 32^3 and 8.0 for 32 of fcc 16^3, without 10.8 and 6.9.
__global__ __launch_bounds__(kBlock) void k_reduce_fin(const double *sp, const double *wpart, int N, int Ns,
                                                       const double *mpart, int ne, double *partial, FinArgs f,
                                                       unsigned *done) {
  reduce_body<true>(sp, wpart, N, Ns, f.nblk, partial, mpart, ne, blockIdx.y, blockIdx.x);
  __shared__ int s_last;
  if (threadIdx.x == 0) {   // (the thread that stored the block's sums)
    stores_done();
    s_last = __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x * gridDim.y - 1;
  }
  __syncthreads();
  if (!s_last) return;   // uniform per block
  const int start = f.clock->parity;  // 1 or 2 (pt.F90:679,898)
  const unsigned long long step = f.clock->step;
  finalize_body<true>(f, start, step);
  if (threadIdx.x == 0) {
    advance_clock(f.clock, f.exchange, f.advance_sweeps);
    *done = 0u;
  }
}

// Direct energy (energy_get, get_quant.F90:186-261): per-site terms, block partials.
template <bool CMP, bool HB, bool HD>
__global__ __launch_bounds__(kBlock) void k_energy(KArgs a, int nblk, double *partial) {
  extern __shared__ double s_ctab[];   // [coefficient table][kBlock/64 scratch]
  double *red = s_ctab + (CMP ? a.nb * a.zmax * 5 : 0);
  const int r = blockIdx.y, bk = blockIdx.x;
  if (CMP) {
    for (int k = threadIdx.x; k < a.nb * a.zmax * 5; k += kBlock) s_ctab[k] = a.ctab[k];
    __syncthreads();
  }
  const int chunk = (a.N + nblk - 1) / nblk;
  const int beg = bk * chunk, end = min(a.N, beg + chunk);
  double *base = a.sp + (size_t)r * 3 * a.Ns;
  const GSpins sp{base, base + a.Ns, base + 2 * a.Ns};
  double v[1] = {0.0};
  for (int d = beg + threadIdx.x; d < end; d += kBlock) {
    const V3 s = sp.ld(d);
    const int b = a.basis[d];
    double e = 0.0;
    for (int l = 0; l < a.zmax; ++l) {
      const unsigned j = (unsigned)a.nbr[(size_t)l * a.N + d];
      const V3 t = sp.ld(j);
      const double dd = dot(s, t);
      double cj, cb = 0, cx = 0, cy = 0, cz = 0;
      if (CMP) {
        const double *c = s_ctab + ((size_t)b * a.zmax + l) * 5;
        cj = c[0]; cb = c[1]; cx = c[2]; cy = c[3]; cz = c[4];
      } else {
        cj = a.cJ[(size_t)l * a.N + d];
        if (HB) cb = a.cB[(size_t)l * a.N + d];
        if (HD) {
          const double *dv = a.cD + 3 * ((size_t)l * a.N + d);
          cx = dv[0]; cy = dv[1]; cz = dv[2];
        }
      }
      e = e - cj * dd;
      if (HB) e = e + cb * dd * dd;
      if (HD)
        e = e + (cx * (s.y * t.z - s.z * t.y) + cy * (s.z * t.x - s.x * t.z) +
                 cz * (s.x * t.y - s.y * t.x));
    }
    if (a.has_h) {
      const double *h = a.h4 + 4 * b;
      e = e + 2.0 * h[0] * (s.x * h[1] + s.y * h[2] + s.z * h[3]);
    }
    if (a.has_si) {
      const double *k = a.si4 + 4 * b;
      const double sa = s.x * k[1] + s.y * k[2] + s.z * k[3];
      e = e + 2.0 * k[0] * sa * sa;
    }
    v[0] += e;
  }
  block_sum<1>(v, red);
  if (threadIdx.x == 0) partial[(size_t)r * nblk + bk] = v[0];
}

__global__ void k_energy_fin(const double *partial, int nblk, int R, double *E) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= R) return;
  double s = 0.0;
  for (int b = 0; b < nblk; ++b) s += partial[(size_t)r * nblk + b];
  E[r] = s / 2.0;
}

// Spins in: reference order [R][N][3] -> device order SoA.
__global__ void k_put_spins(const double *in, const int *ref2dev, int N, int Ns, int R, double *sp) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= (size_t)N * R) return;
  const int r = (int)(t / N), i = (int)(t % N);
  const double *p = in + 3 * t;
  const int d = ref2dev[i];
  double *x = sp + (size_t)r * 3 * Ns;
  x[d] = p[0]; x[Ns + d] = p[1]; x[2 * Ns + d] = p[2];
}

// Spins out: sites t0 .. t0 + n - 1 of the [R][N] reference order.
__global__ void k_get_spins(const double *sp, const int *ref2dev, const int *src_rep, int N, int Ns,
                            size_t t0, size_t n, double *out) {
  const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  const size_t t = t0 + k;
  const int q = (int)(t / N), i = (int)(t % N);
  const int r = src_rep ? src_rep[q] : q;
  const double *x = sp + (size_t)r * 3 * Ns;
  const int d = ref2dev[i];
  double *p = out + 3 * k;
  p[0] = x[d]; p[1] = x[Ns + d]; p[2] = x[2 * Ns + d];
}

__global__ void k_set_clock(Clock *c, Clock v) { *c = v; }

// Statistics to zero: estimators, rejections, swaps, measurement count.
__global__ void k_zero_stats(double *acc, unsigned long long *rej, unsigned long long *nswap,
                             unsigned long long *nmeas, int R) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t < 6 * R) acc[t] = 0.0;
  if (t < kRejSub * R) rej[t] = 0;
  if (t < 2 * R) nswap[t] = 0;
  if (t == 0) *nmeas = 0;
}

// Plain streaming copy (grid-stride, 32 B per lane per iteration): calibrates the HBM
// traffic counters against a kernel whose bytes are known.
__global__ void k_copy(const double4 *src, double4 *dst, size_t n) {
  for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n; t += (size_t)gridDim.x * blockDim.x)
    dst[t] = src[t];
}

__global__ void k_fill(double *p, size_t n, double v) {
  const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) p[t] = v;
}

// Per-slot totals of the rejection sub-counters rej[kRejSub][R] (host side).
inline void sum_rej_sub(const std::vector<int64_t> &sub, int R, int64_t *out) {
  for (int s = 0; s < R; ++s) {
    int64_t t = 0;
    for (int k = 0; k < kRejSub; ++k) t += sub[(size_t)k * R + s];
    out[s] = t;
  }
}

// Geometry-group tiles of a colour (host).
inline bool geo_tiles(const esp::HostModel &m, int tps) {
  return m.implicit && m.compressed && tps == 1 && espg::tiles_serve((int)m.geo.mt.d);
}
inline int geo_tseg(const esp::HostModel &m) { return espg::tile_count((int)m.geo.mt.d); }
inline void geo_args(KArgs &a, const esp::HostModel &m) {
  constexpr int kW = kPhaseBlock / 64;
  a.tseg = geo_tseg(m);
  a.spt = ((int)m.geo.mt.d + a.tseg - 1) / a.tseg;
  const int runs = (a.tseg + kW - 1) / kW;
  a.run = (a.tseg + runs - 1) / runs;
  a.drun = espg::make_fastdiv((uint32_t)a.run);
}
inline espg::FastDiv geo_ngc(const esp::HostModel &m, int col) {   // groups of the colour
  return espg::make_fastdiv((uint32_t)((m.col_off[col + 1] - m.col_off[col]) / (int)m.geo.mt.d));
}
// Entries of the per-wave sums of one colour phase of one replica.
inline int colour_waves(const esp::HostModel &m, int col, int tps, bool geo) {
  const int n = m.col_off[col + 1] - m.col_off[col];
  return geo ? n / (int)m.geo.mt.d * geo_tseg(m) : (n * tps + 63) / 64;
}
// Its blocks.
inline int colour_blocks(const esp::HostModel &m, int col, int tps, bool geo) {
  constexpr int kW = kPhaseBlock / 64;
  int waves = colour_waves(m, col, tps, geo);
  if (geo) {
    KArgs a{};
    geo_args(a, m);
    waves = waves / a.tseg * ((a.tseg + a.run - 1) / a.run) * a.run;
  }
  return (waves + kW - 1) / kW;
}

}  // namespace
}  // namespace espk
