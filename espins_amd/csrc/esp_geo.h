// esp_geo.h -- implicit lattice geometry: partner indices, reference site indices and basis
// atoms computed from the device index instead of loaded from per-site tables.
//
// It applies to a periodic supercell L0 x L1 x L2 with nb basis atoms whose colouring has a
// period P (a site's colour depends only on its basis atom and its cell modulo P, P_k | L_k).
// The device order (esp_model.cpp) then consists of "groups": for every (basis atom a,
// residue r = cell mod P), in colour order, the M0 x M1 x M2 cells x = s * P + r (M = L / P),
// s in lexicographic order (s0 fastest).  Every group has Mt = M0 M1 M2 sites, so
//     device index d = g * Mt + (s2 * M1 + s1) * M0 + s0.
// The bond in slot l of a site of group g goes to the cell x + delta_l of the basis atom
// b_l, i.e. to group g'(g, l) at sub-cell (s + q(g, l)) mod M with q = floor((r + delta) / P).
// One table row per (group, slot) -- {first device index of g', q packed in bytes} -- gives
// every partner index with integer arithmetic: the per-site neighbour list (4 B per bond of
// HBM traffic) is not read at all.
//
// The same functions run on the host (to verify them against the explicit tables for every
// site and slot before a context uses them) and in the kernels.
#pragma once
#include <stdint.h>

#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define ESP_HD __host__ __device__ __forceinline__
#else
#define ESP_HD inline
#endif

namespace espg {

// Unsigned division by a run-time constant D >= 1 for 32-bit numerators: multiply-high,
// add, shift (Granlund & Montgomery 1994, the "round-up" method with a 33-bit multiplier
// split as 2^32 + m).
struct FastDiv {
  uint32_t m, s1, s2, d;
};

ESP_HD uint32_t umulhi32(uint32_t a, uint32_t b) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __umulhi(a, b);
#else
  return (uint32_t)(((uint64_t)a * b) >> 32);
#endif
}

inline FastDiv make_fastdiv(uint32_t D) {
  uint32_t l = 0;
  while (l < 32 && (1ull << l) < D) ++l;            // l = ceil(log2 D)
  FastDiv f;
  f.m = (uint32_t)(((1ull << 32) * ((1ull << l) - D)) / D + 1);
  f.s1 = l > 0 ? 1u : 0u;
  f.s2 = l > 0 ? l - 1 : 0u;
  f.d = D;
  return f;
}

ESP_HD uint32_t fdiv(uint32_t n, const FastDiv &f) {
  const uint32_t t = umulhi32(f.m, n);
  return (t + ((n - t) >> f.s1)) >> f.s2;
}

// Replica r and block b that block L of a launch of nblk blocks for each of R replicas takes
// (full = xcd_full(R, nblk), dnblk divides by nblk).  Blocks go round-robin over the 8 XCDs, each
// with an L2 of its own: eight replicas at a time are dealt one to an XCD, with all their blocks;
// the last R % 8 are spread.  A replica whose blocks run on every XCD is read into every L2: us per
// colour phase with all replicas spread / so: FCC 16^3 x 244, three shells 75.6 / 38.8, FCC 32^3 x 60
// 62.5 / 40.6, BCC 20^3 x 100 24.6 / 17.8, SC 64^3 x 30 75.1 / 66.5, FCC 18^3 x 41 learned 29.8 / 26.2.
ESP_HD void place_block(uint32_t L, uint32_t full, const FastDiv &dnblk, int &r, int &b) {
  const bool own = L < full;
  const uint32_t q = own ? L >> 3 : L, w = fdiv(q, dnblk);
  b = (int)(q - w * dnblk.d);
  r = (int)(own ? (L & 7u) + 8u * w : w);
}
inline uint32_t xcd_full(int R, int nblk) { return (uint32_t)(R / 8 * 8) * (uint32_t)nblk; }

// Geometry of one model (host-built, passed by value to the kernels).
struct Geo {
  FastDiv mt, m0, m1;            // Mt, M0, M1
  int M0, M1, M2, P0, P1, P2, L0, L1, nb;
  int ngroups, zmax, N;
};

// Tiles of a wave's 64 lanes that a group of mt sites is cut into, evenly.  They serve the colour
// phases where at least half of their lanes have a site, which is from 32 sites; else the phases read
// the tables.  us per colour phase, tiles / tables: 27 sites 21.3 / 14.2 (FCC 18^3 x 64) and 8.9 / 7.1
// (SC 6^3 x 1000), 64 sites 15.1 / 16.9 (FCC 24^3 x 32), 125 sites 24.5 / 31.2 (FCC 30^3 x 32).
ESP_HD int tile_count(int mt) { return (mt + 63) / 64; }
ESP_HD bool tiles_serve(int mt) { return 2 * mt >= 64 * tile_count(mt); }

// Per-group record: basis atom and residue, packed a | r0 << 8 | r1 << 16 | r2 << 24.
ESP_HD int grp_pack(int a, int r0, int r1, int r2) { return a | (r0 << 8) | (r1 << 16) | (r2 << 24); }

// Per-(group, slot) record: x = first device index of the partner group (-1: padding slot,
// which points at the zero spin N); y = the sub-cell shift reduced mod M, q_k in [0, M_k),
// packed as q0 | q1 << 8 | q2 << 16 (M_k <= 255).
ESP_HD int q_pack(int q0, int q1, int q2) { return q0 | (q1 << 8) | (q2 << 16); }

// 24-bit multiply-add (full-rate v_mad_u32_u24 on the device; operands < 2^24).
ESP_HD uint32_t umad24(uint32_t a, uint32_t b, uint32_t c) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __umul24(a, b) + c;
#else
  return a * b + c;
#endif
}

ESP_HD uint32_t umin32(uint32_t a, uint32_t b) { return a < b ? a : b; }

struct SiteGeo {
  int g;              // group
  int s0, s1, s2;     // sub-cell
  int a;              // basis atom
  int ir;             // reference site index (0-based): ((x2 L1 + x1) L0 + x0) nb + a
};

// Site k of group g, whose record is e.
ESP_HD SiteGeo geo_place(const Geo &G, int e, int g, int k) {
  SiteGeo s;
  const uint32_t uk = (uint32_t)k;
  const uint32_t t = fdiv(uk, G.m0);
  s.g = g;
  s.s0 = (int)(uk - t * (uint32_t)G.M0);
  const uint32_t u = fdiv(t, G.m1);
  s.s1 = (int)(t - u * (uint32_t)G.M1);
  s.s2 = (int)u;
  s.a = e & 0xff;
  const int x0 = s.s0 * G.P0 + ((e >> 8) & 0xff);
  const int x1 = s.s1 * G.P1 + ((e >> 16) & 0xff);
  const int x2 = s.s2 * G.P2 + ((e >> 24) & 0xff);
  s.ir = ((x2 * G.L1 + x1) * G.L0 + x0) * G.nb + s.a;
  return s;
}

ESP_HD SiteGeo geo_site(const Geo &G, const int *grp, int d) {
  const uint32_t g = fdiv((uint32_t)d, G.mt);
  return geo_place(G, grp[g], (int)g, (int)((uint32_t)d - g * (uint32_t)G.mt.d));
}

// (s + q) mod M for s, q in [0, M): t = s + q < 2M, and t - M wraps to a huge unsigned value
// when t < M, so the unsigned minimum is the reduced sum (three VALU instructions with the
// byte extraction folded into the add).
ESP_HD uint32_t wrap_add(uint32_t s, uint32_t q, uint32_t M) {
  const uint32_t t = s + q;
  return umin32(t, t - M);
}

// Place inside its group of the sub-cell of s shifted by the packed shift q.
ESP_HD int geo_shift(const Geo &G, const SiteGeo &s, uint32_t q) {
  const uint32_t v0 = wrap_add((uint32_t)s.s0, q & 0xffu, (uint32_t)G.M0);
  const uint32_t v1 = wrap_add((uint32_t)s.s1, (q >> 8) & 0xffu, (uint32_t)G.M1);
  const uint32_t v2 = wrap_add((uint32_t)s.s2, (q >> 16) & 0xffu, (uint32_t)G.M2);
  return (int)umad24(umad24(v2, (uint32_t)G.M1, v1), (uint32_t)G.M0, v0);
}

// Device index of the partner of site s through the (group, slot) record (pg, qp); padding
// slots (pg < 0) give the zero spin N.
ESP_HD int geo_partner(const Geo &G, const SiteGeo &s, int pg, int qp) {
  const int j = pg + geo_shift(G, s, (uint32_t)qp);
  return pg < 0 ? G.N : j;
}

}  // namespace espg
