// esp_cluster.hip -- sweeps of middle-sized replicas with every spin in LDS, each replica shared
// by a cluster of k blocks, one block per CU: whole runs -- sweeps, measurements and exchanges --
// in one launch.
//
// A replica too large for one CU's LDS (or one CU too slow for it) is cut into k parts of
// consecutive reference sites.  Block (r, j) keeps part j of replica r and the halo, the foreign
// sites its bonds reach, in LDS.  Phase by phase (one colour): it proposes for its sites (needs no
// neighbour), waits until the parts it borders have finished the phase before, refreshes the halo
// sites of that colour from global memory, updates its sites from LDS, stores the accepted spins
// to global memory (so the state there is always whole) and raises its flag.  A part can run at
// most one phase ahead of its neighbours, and a colour phase reads only other colours, so no value
// is overwritten while a neighbour may still read it.  At a measurement or exchange every block
// adds its partial sums and block 0 runs the estimators and the exchange for all replicas.
//
// Against one launch per colour (4 us of launch and drain each, partners from the memory-side
// cache, in as many round trips as a lane has gathers in a row) a phase costs about 1.5 us of flag
// and halo traffic beside its arithmetic.  Per step, launch-per-colour and so: FCC 16^3 x 64 (42
// bonds, k = 4) 133 -> 70 us; FCC 15^3 x 37, cone proposals, 10 colours (k = 6) 116 -> 65; SC 20^3 spin
// glass x 24 (k = 10) 27 -> 14; and against the one-block kernel SC 14^3 x 32, cone proposals (k = 8)
// 43 -> 23 us per sweep.
//
// Blocks wait for each other, so all of them must be resident.  The launch proves it before it
// changes anything: every block reports in, and if they have not all done so within 1 ms (another
// stream holds the CUs), all leave and the caller takes the other paths, for a while (cluster_skip,
// esp_hip.hip).  Once all are resident they stay so, and every wait ends; waits are bounded all the same.
// Contexts that run at the same time do not contend: while one's launch is on the device, the runs
// of others take the other paths.  One, two and four threads with a context of FCC 16^3 x 64 each
// (k = 4), ms a call of 20 steps: 0.85 / 1.3 / 2.9; on the other paths alone 1.55 / 2.08 / 3.27; all
// launching clusters, with 50 ms to wait for residency, 0.81 / 1.60 / 24.6.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "esp_ctx.h"

using namespace espd;
using namespace espk;

namespace {

constexpr int kCBlock = 512;
constexpr int kGroup = 6;                         // bonds whose partners are read together
constexpr int kCMaxGroups = 8;                    // bond groups of a site at most
constexpr int kCMaxCol = 64;
constexpr int kPhases = 1 << 18;                  // colour phases of one launch at most: a second or less
template <bool HB, bool HD>
constexpr int kTabCoef = 1 + (HB ? 1 : 0) + (HD ? 3 : 0);

// Tables of one part (offsets into the shared arrays) and the control words of a launch.
struct Part {
  int nown, nhalo, own0, hal0, col0, nb0, nnb, pitch;
  size_t tab0;                                    // first word of its partner table
};
struct Ctl {
  unsigned arrived, decided;                      // start: blocks that reported in; 1 go, 2 leave
  unsigned done[2], go;                           // partial sums added, by set; steps finalized
  unsigned failed, pad[2];
};
constexpr unsigned kGo = 1, kLeave = 2;
constexpr long long kTicksPerMs = 100000;         // wall_clock64 runs at 100 MHz
constexpr long long kResidentMs = 1;              // wait for the launch's blocks (they take microseconds)

struct CArgs {
  KArgs a;
  FinArgs f;
  const Part *part;
  const int *own_dev, *own_ref, *hal_dev, *col_off, *hal_off, *nbs;   // by part (Part offsets)
  const uint8_t *own_basis;
  const double *own_mag, *own_j;                  // moments; per-bond couplings [zmax][nown] of a part
  const unsigned *tab;                            // [pairs][pitch] local partner index pairs of a part
  Ctl *ctl;
  unsigned *flag;                                 // [R][k] phases finished
  double *partial;                                // [2][R][k][4]
  int *slots;                                     // [R] slots after an exchange
  int k, nl_max, ngroup, xcd;
  // steps of M sweeps; an exchange after every `round` steps, the first of them being step0 of a round
  int nsteps, M, measure, exchange, round, step0;
};

// What blocks exchange during a launch -- spins, partial sums, slots, flags -- moves by ald and ast
// only.  Before a block raises a flag every wave waits until its stores have been acknowledged
// (stores_done) and then for the block's other waves, so what a flag announces is in place when
// the flag is (with release and acquire fences a colour phase took 10 us, against 3).

// Waits until *p >= want; false after 60 s without it (only a lost block could cause that).
__device__ __forceinline__ bool wait_ge(const unsigned *p, unsigned want, const Ctl *ctl) {
  if (ald(p) >= want) return true;
  const long long t0 = wall_clock64();
  for (;;) {
    for (int i = 0; i < 64; ++i) {
      if (ald(p) >= want) return true;
      __builtin_amdgcn_s_sleep(1);
    }
    if (ald(&ctl->failed) || wall_clock64() - t0 > 60000 * kTicksPerMs) return false;
  }
}

// Block 0's working copy of the estimators during a launch, in LDS (finalize_body reads and
// writes it there; global memory costs it a chain of L2 round trips per step).
struct FinLds {
  double *e_base, *e_run, *beta, *acc, *part;     // [R], [R], [R], [R][6], [R][4]
  unsigned long long *nswap, *nmeas;              // [R][2], [1]
  int *slot_rep, *rep_slot;                       // [R]
};
__host__ __device__ inline size_t fin_lds_bytes(int R) {
  return (size_t)R * (13 * sizeof(double) + 2 * sizeof(unsigned long long) + 2 * sizeof(int)) + 8;
}
__device__ __forceinline__ FinLds fin_lds(double *p, int R) {
  FinLds f;
  f.e_base = p; f.e_run = p + R; f.beta = p + 2 * R; f.acc = p + 3 * R; f.part = p + 9 * R;
  f.nswap = reinterpret_cast<unsigned long long *>(p + 13 * R);
  f.nmeas = f.nswap + 2 * R;
  f.slot_rep = reinterpret_cast<int *>(f.nmeas + 1);
  f.rep_slot = f.slot_rep + R;
  return f;
}

// Sums of a replica's parts where they are more than 16 (of at most 15 replicas): 16 threads to a sum.
// One thread made 32 round trips for one replica on 256 CUs; a measured step of sc 32^3 took 28.3 us,
// 18.7 so.  Not inlined: the registers of the colour phases stay as they are without it (inlined, 60
// steps of fcc 15^3 x 37 took 3064 us, 3022 without, 3005 so).
__device__ __attribute__((noinline)) void sum_many(const double *part, int k, int R, double *out) {
  const int each = (k + 15) >> 4, b1 = (threadIdx.x & 15) * each, b2 = min(k, b1 + each);
  for (int q = threadIdx.x >> 4; q < R * 4; q += kCBlock / 16) {
    double x = 0.0;
    const double *p = part + (size_t)(q >> 2) * k * 4 + (q & 3);
    for (int b0 = b1; b0 < b2; b0 += 8) {
      double t[8];
#pragma unroll
      for (int b = 0; b < 8; ++b) t[b] = b0 + b < b2 ? ald(p + 4 * (b0 + b)) : 0.0;
#pragma unroll
      for (int b = 0; b < 8; ++b) x += t[b];
    }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) x += __shfl_xor(x, o);
    if (b1 == 0) out[q] = x;
  }
}

template <int MODE, bool CMP, bool HB, bool HD, bool SELF, int NG>
__global__ __launch_bounds__(kCBlock) void k_cluster(CArgs c) {
  constexpr int ZP = NG * kGroup / 2;            // partner pairs held in registers
  extern __shared__ double s_dyn[];
  __shared__ double s_red[4 * (kCBlock / 64)];
  __shared__ int s_ok, s_col[kCMaxCol + 1], s_hal[kCMaxCol + 1];
  __shared__ unsigned s_rej;
  const KArgs &a = c.a;
  int r, j;
  {
    const unsigned L = blockIdx.x;   // the parts of a replica on one XCD where the count allows
    const unsigned u = c.xcd ? (L & 7u) * (gridDim.x >> 3) + (L >> 3) : L;
    r = (int)(u / (unsigned)c.k);
    j = (int)(u - (unsigned)r * (unsigned)c.k);
  }
  const Part P = c.part[j];
  const int tid = threadIdx.x, nl = c.nl_max + 1, zs = NG * kGroup;
  double *lx = s_dyn, *ly = lx + nl, *lz = ly + nl, *ctab = lz + nl;
  const FinLds fl = fin_lds(ctab + (CMP ? a.nb * zs * kTabCoef<HB, HD> : 0), a.R);
  double *gx = a.sp + (size_t)r * 3 * a.Ns, *gy = gx + a.Ns, *gz = gy + a.Ns;
  const int *own_dev = c.own_dev + P.own0, *hal_dev = c.hal_dev + P.hal0;

  // every block reports in; all resident, or all leave before anything changed
  if (tid == 0) {
    s_rej = 0;
    const unsigned n = __hip_atomic_fetch_add(&c.ctl->arrived, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
    unsigned want = 0;
    if (n == gridDim.x)
      __hip_atomic_compare_exchange_strong(&c.ctl->decided, &want, kGo, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    const long long t0 = wall_clock64();
    unsigned d;
    while ((d = ald(&c.ctl->decided)) == 0) {
      __builtin_amdgcn_s_sleep(1);
      if (wall_clock64() - t0 > kResidentMs * kTicksPerMs) {
        want = 0;
        __hip_atomic_compare_exchange_strong(&c.ctl->decided, &want, kLeave, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    s_ok = d == kGo;
  }
  for (int i = tid; i < P.nown; i += kCBlock) {
    const int d = own_dev[i];
    lx[i] = gldi(gx, d); ly[i] = gldi(gy, d); lz[i] = gldi(gz, d);
  }
  for (int i = tid; i < P.nhalo; i += kCBlock) {
    const int d = hal_dev[i], q = P.nown + i;
    lx[q] = gldi(gx, d); ly[q] = gldi(gy, d); lz[q] = gldi(gz, d);
  }
  if (tid == 0) lx[c.nl_max] = ly[c.nl_max] = lz[c.nl_max] = 0.0;     // the zero spin
  if (CMP)                       // rows of zs slots (the spare ones zero), only the terms present
    for (int q = tid; q < a.nb * zs; q += kCBlock) {
      const int b = q / zs, l = q - b * zs;
      double *o = ctab + (size_t)q * kTabCoef<HB, HD>;
      auto co = [&](int t) { return l < a.zmax ? gldi(a.ctab, ((size_t)b * a.zmax + l) * 5 + t) : 0.0; };
      *o++ = co(0);
      if (HB) *o++ = co(1);
      if (HD) { *o++ = co(2); *o++ = co(3); *o++ = co(4); }
    }
  for (int q = tid; q <= a.ncol; q += kCBlock) {
    s_col[q] = c.col_off[P.col0 + q];
    s_hal[q] = c.hal_off[P.col0 + q];
  }
  if (blockIdx.x == 0) {
    for (int q = tid; q < a.R; q += kCBlock) {
      fl.e_base[q] = c.f.e_base[q]; fl.e_run[q] = 0.0; fl.beta[q] = c.f.beta_slot[q];
      fl.slot_rep[q] = c.f.slot_rep[q]; fl.rep_slot[q] = c.f.rep_slot[q];
      fl.nswap[2 * q] = c.f.nswap[2 * q]; fl.nswap[2 * q + 1] = c.f.nswap[2 * q + 1];
      for (int t = 0; t < 6; ++t) fl.acc[6 * q + t] = c.f.acc[6 * q + t];
    }
    if (tid == 0) *fl.nmeas = *c.f.nmeas;
  }
  __syncthreads();
  if (!s_ok) return;

  int slot = gldi(a.rep_slot, r);
  double beta = gldi(a.beta_slot, slot);
  const unsigned long long sweep0 = gldi(&a.clock->sweep, 0);
  unsigned long long xstep = gldi(&a.clock->step, 0);
  int parity = gldi(&a.clock->parity, 0);
  unsigned *myflag = c.flag + (size_t)r * c.k + j;
  double wsum = 0.0;              // accepted dE of this thread's sites since the launch began
  unsigned nrej = 0, phase = 0, fin = 0;
  int pc = 0;                     // colour of the phase before
  bool xwait = false;             // new slots are due from block 0
  // a site's data and partners: those of a phase's first pass are loaded while the stores of the
  // phase before drain
  Site s{};
  unsigned nb[ZP];
  double cj[CMP ? 1 : 2 * ZP];
  auto fetch = [&](int i, int end) {
    if (i >= end) return;
    s.d = gldi(own_dev, i);
    s.ir = gldi(c.own_ref, (size_t)P.own0 + i);
    s.a = gldi(c.own_basis, (size_t)P.own0 + i);
    s.mag = gldi(c.own_mag, (size_t)P.own0 + i);
    const unsigned *t = c.tab + P.tab0 + i;
#pragma unroll
    for (int g = 0; g < NG; ++g)
      if (g < c.ngroup) {
#pragma unroll
        for (int u = g * kGroup / 2; u < (g + 1) * kGroup / 2; ++u) nb[u] = gldi(t, (size_t)u * P.pitch);
      }
    if (!CMP) {
#pragma unroll
      for (int u = 0; u < 2 * ZP; ++u) cj[u] = u < a.zmax ? gldi(c.own_j, ((size_t)P.own0 * a.zmax + (size_t)u * P.nown) + i) : 0.0;
    }
  };
  fetch(s_col[0] + tid, s_col[1]);
  for (int st = 0; st < c.nsteps; ++st) {
    for (int m = 0; m < c.M; ++m) {
      const unsigned long long sweep = sweep0 + (unsigned long long)(st * c.M + m);
      for (int col = 0; col < a.ncol; ++col) {
        const int beg = s_col[col], end = s_col[col + 1];
        bool first = true;
        for (int i0 = beg; first || i0 < end; i0 += kCBlock, first = false) {
          const int i = i0 + tid;
          const bool on = i < end;
          if (!first) fetch(i, end);
          int hq = 0, hd = 0;      // this thread's first halo site to refresh
          if (first && phase > 0) {
            hq = s_hal[pc] + tid;
            if (hq < s_hal[pc + 1]) hd = gldi(hal_dev, hq);
          }
          Proposal p{};
          if (on) {
            p.so = {lx[i], ly[i], lz[i]};
            const uint4 rn = philox10(make_uint4((uint32_t)s.ir, (uint32_t)sweep, (uint32_t)(sweep >> 32),
                                                 a.stream_base + (uint32_t)r), a.key0, a.key1);
            p.sn = MODE == M_RANDOM ? propose_random(s.mag, u01(rn.x), u01(rn.y))
                                    : propose_const(s.mag, p.so, a.tilt, u01(rn.x), u01(rn.y));
            p.u3 = u01(rn.z);
          }
          if (first && phase > 0) {   // neighbours' phase before, then its colour's halo sites
            bool ok = true;
            if (tid < 64)
              for (int q = tid; q < P.nnb && ok; q += 64)
                ok = wait_ge(c.flag + (size_t)r * c.k + c.nbs[P.nb0 + q], phase, c.ctl);
            if (xwait && tid == 64) ok = wait_ge(&c.ctl->go, fin, c.ctl);
            if (!ok) ast(&c.ctl->failed, 1u);
            if (tid == 0) s_ok = 1;
            __syncthreads();
            if (!ok) s_ok = 0;
            if (xwait) {
              slot = ald(c.slots + r);
              xwait = false;
            }
            for (; hq < s_hal[pc + 1]; hq += kCBlock) {
              const double vx = ald(gx + hd), vy = ald(gy + hd), vz = ald(gz + hd);
              const int l = P.nown + hq;
              if (hq + kCBlock < s_hal[pc + 1]) hd = gldi(hal_dev, hq + kCBlock);
              lx[l] = vx; ly[l] = vy; lz[l] = vz;
            }
            beta = gldi(a.beta_slot, slot);
            __syncthreads();
            if (!s_ok) return;
          }
          if (on) {
            const V3 ds = sub(p.sn, p.so);
            const V3 si = sub(p.sn, ds);
            const double *crow = CMP ? ctab + (size_t)s.a * zs * kTabCoef<HB, HD> : nullptr;
            double eJ = 0.0, eB = 0.0, eD = 0.0;
#pragma unroll
            for (int g = 0; g < NG; ++g)
              if (g < c.ngroup) {      // whole groups: spare slots hold the zero spin
                V3 sv[kGroup];
#pragma unroll
                for (int u = 0; u < kGroup; ++u) {
                  const unsigned w = nb[(g * kGroup + u) / 2];
                  const unsigned q = u & 1 ? w >> 16 : w & 0xffffu;
                  sv[u] = {lx[q], ly[q], lz[q]};
                  if (SELF && (int)q == i) sv[u] = p.sn;
                }
#pragma unroll
                for (int u = 0; u < kGroup; ++u) {
                  const int l = g * kGroup + u;
                  const double *co = crow + l * kTabCoef<HB, HD>;
                  const V3 &sj = sv[u];
                  const double dsj = dot(ds, sj);
                  eJ = eJ - (CMP ? co[0] : cj[CMP ? 0 : l]) * dsj;
                  if (HB) {
                    const double sij = dot(si, sj);
                    eB = eB + co[1] * (dsj * dsj + 2.0 * sij * dsj);
                  }
                  if (HD) {
                    constexpr int o = HB ? 2 : 1;
                    eD = eD + (co[o] * (ds.y * sj.z - ds.z * sj.y) + co[o + 1] * (ds.z * sj.x - ds.x * sj.z) +
                               co[o + 2] * (ds.x * sj.y - ds.y * sj.x));
                  }
                }
              }
            double de;
            if (decide(a, s.a, p, eJ, eB, eD, beta, &de)) {
              ++nrej;
            } else {
              wsum += de;
              lx[i] = p.sn.x; ly[i] = p.sn.y; lz[i] = p.sn.z;
              ast(gx + s.d, p.sn.x); ast(gy + s.d, p.sn.y); ast(gz + s.d, p.sn.z);
            }
          }
        }
        const int nc = col + 1 < a.ncol ? col + 1 : 0;
        fetch(s_col[nc] + tid, s_col[nc + 1]);
        stores_done();
        __syncthreads();
        ++phase;
        if (tid == 0) ast(myflag, phase);
        pc = col;
      }
    }
    const bool last = st + 1 == c.nsteps;
    const bool xch = c.exchange && (c.step0 + st + 1) % c.round == 0;
    if (!c.measure && !xch && !last) continue;
    // Two sets of partial sums take turns, each with its own count: a block may start the next
    // step before a slower one has added to this one, but it reuses a set only when block 0 has
    // read it.
    if (fin >= 2 && tid == 0 && !wait_ge(&c.ctl->go, fin - 1, c.ctl)) ast(&c.ctl->failed, 1u);
    // partial sums: accepted dE since the launch began and the part's spins; rejections by slot
    double v[3] = {0.0, 0.0, 0.0};
    for (int i = tid; i < P.nown; i += kCBlock) { v[0] += lx[i]; v[1] += ly[i]; v[2] += lz[i]; }
    const double t4 = wave_total4(wsum, v[0], v[1], v[2]);
    if ((tid & 63) < 4) s_red[(tid & 63) * (kCBlock / 64) + (tid >> 6)] = t4;
    unsigned nr = nrej;     // (32 bits: a block of 6826 sites at most makes kPhases / 2 sweeps a launch at most)
    for (int o = 32; o > 0; o >>= 1) nr += __shfl_down(nr, o, 64);
    nrej = 0;
    if ((tid & 63) == 0 && nr) atomicAdd(&s_rej, nr);
    __syncthreads();
    double *part = c.partial + (size_t)(fin & 1) * gridDim.x * 4;
    unsigned *done = &c.ctl->done[fin & 1];
    const unsigned want = gridDim.x * ((fin >> 1) + 1);
    ++fin;
    if (tid < 4) {
      double x = 0.0;
#pragma unroll
      for (int w = 0; w < kCBlock / 64; ++w) x += s_red[tid * (kCBlock / 64) + w];
      ast(part + ((size_t)r * c.k + j) * 4 + tid, x);
    }
    if (tid < 64) {
      stores_done();
      if (tid == 0) {
        __hip_atomic_fetch_add(done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (s_rej) gadd(&a.rej[(size_t)(blockIdx.x % kRejSub) * a.R + slot], (unsigned long long)s_rej);
        s_rej = 0;
      }
    }
    if (blockIdx.x == 0) {
      if (tid == 0) s_ok = wait_ge(done, want, c.ctl);
      __syncthreads();
      if (!s_ok) { if (tid == 0) ast(&c.ctl->failed, 1u); return; }
      // block 0 sums the parts, runs the estimators and the exchange and publishes the slots
      if (c.k > 16) {
        sum_many(part, c.k, a.R, fl.part);
      } else {
        for (int q = tid; q < a.R * 4; q += kCBlock) {
          double x = 0.0;
          const double *p = part + (size_t)(q >> 2) * c.k * 4 + (q & 3);
          for (int b0 = 0; b0 < c.k; b0 += 8) {
            double t[8];
#pragma unroll
            for (int b = 0; b < 8; ++b) t[b] = b0 + b < c.k ? ald(p + 4 * (b0 + b)) : 0.0;
#pragma unroll
            for (int b = 0; b < 8; ++b) x += t[b];
          }
          fl.part[q] = x;
        }
      }
      __syncthreads();
      FinArgs f = c.f;
      f.partial = fl.part; f.nblk = 1; f.measure = c.measure; f.exchange = xch;
      f.e_base = fl.e_base; f.e_run = fl.e_run; f.acc = fl.acc; f.nmeas = fl.nmeas; f.nswap = fl.nswap;
      f.slot_rep = fl.slot_rep; f.rep_slot = fl.rep_slot; f.beta_slot = fl.beta;
      finalize_body(f, parity, xstep);
      __syncthreads();
      if (xch) for (int q = tid; q < a.R; q += kCBlock) ast(c.slots + q, fl.rep_slot[q]);
      if (last) {                  // the working copy back, the launch's dE into e_base, the clock
        for (int q = tid; q < a.R; q += kCBlock) {
          const_cast<double *>(c.f.e_base)[q] = fl.e_base[q] + fl.part[4 * q];
          c.f.e_run[q] = fl.e_run[q];
          c.f.slot_rep[q] = fl.slot_rep[q]; c.f.rep_slot[q] = fl.rep_slot[q];
          c.f.nswap[2 * q] = fl.nswap[2 * q]; c.f.nswap[2 * q + 1] = fl.nswap[2 * q + 1];
          for (int t = 0; t < 6; ++t) c.f.acc[6 * q + t] = fl.acc[6 * q + t];
        }
        if (tid == 0) {
          *c.f.nmeas = *fl.nmeas;
          Clock *k = c.f.clock;
          k->sweep = sweep0 + (unsigned long long)c.nsteps * c.M;
          k->step = xstep + (xch ? 1 : 0);
          k->parity = xch ? 3 - parity : parity;
        }
      }
      stores_done();
      __syncthreads();
      if (tid == 0) ast(&c.ctl->go, fin);
    }
    if (xch) {
      xstep += 1;
      parity = 3 - parity;
      xwait = true;
    }
  }
}

using ClusterFn = void (*)(CArgs);
template <int MODE, bool CMP, bool HB, bool HD, int NG>
ClusterFn cf3(bool self) { return self ? k_cluster<MODE, CMP, HB, HD, true, NG> : k_cluster<MODE, CMP, HB, HD, false, NG>; }
template <int MODE, int NG>
ClusterFn cf_cmp(bool hb, bool hd, bool self) {
  if (hb) return hd ? cf3<MODE, true, true, true, NG>(self) : cf3<MODE, true, true, false, NG>(self);
  return hd ? cf3<MODE, true, false, true, NG>(self) : cf3<MODE, true, false, false, NG>(self);
}
// Bond groups compiled in: 1, 3 or kCMaxGroups (the site's partners live in registers).
int groups_compiled(const esp::HostModel &m) {
  const int n = (m.zmax + kGroup - 1) / kGroup;
  return !m.compressed || n <= 1 ? 1 : n <= 3 ? 3 : kCMaxGroups;
}
template <int MODE>
ClusterFn cf_mode(const esp::HostModel &m) {
  if (!m.compressed) return cf3<MODE, false, false, false, 1>(m.has_self);
  const int n = groups_compiled(m);
  if (n == 1) return cf_cmp<MODE, 1>(m.has_B, m.has_D, m.has_self);
  return n == 3 ? cf_cmp<MODE, 3>(m.has_B, m.has_D, m.has_self) : cf_cmp<MODE, kCMaxGroups>(m.has_B, m.has_D, m.has_self);
}
ClusterFn cluster_fn(int mode, const esp::HostModel &m) {
  return mode == M_RANDOM ? cf_mode<M_RANDOM>(m) : cf_mode<M_CONST>(m);
}

size_t cluster_lds(const esp::HostModel &m, int nl_max, int R) {
  const int nc = 1 + (m.has_B ? 1 : 0) + (m.has_D ? 3 : 0);
  return (size_t)(nl_max + 1) * 3 * sizeof(double) +
         (m.compressed ? (size_t)m.nb * groups_compiled(m) * kGroup * nc * sizeof(double) : 0) + fin_lds_bytes(R);
}

// A block's LDS beside the kernel's static share.
bool cluster_fits(const esp::HostModel &m, int nl_max, int R, size_t lds_max) {
  return nl_max < 65535 && cluster_lds(m, nl_max, R) + 1024 <= lds_max;
}

// Parts to cut a replica into; 0 where clusters do not serve the model.
int cluster_parts(const esp::HostModel &m, int R, int num_cu) {
  if (m.ncol < 2 || m.ncol > kCMaxCol || m.zmax > kCMaxGroups * kGroup ||
      (!m.compressed && (m.zmax > kGroup || m.has_B || m.has_D)))
    return 0;
  return std::min(num_cu / R, m.N / m.ncol / 64);
}

struct Plan {
  std::vector<Part> part;
  std::vector<int> own_dev, own_ref, hal_dev, col_off, hal_off, nbs;
  std::vector<uint8_t> own_basis;
  std::vector<unsigned> tab;
  std::vector<double> own_mag, own_j;
  int nl_max = 0, ngroup = 0;
};

// Cuts the sites (reference order) into k parts and builds their tables; false, as soon as that is
// known, if a part does not fit.  (A replica whose k parts do not fit needs more CUs: fewer parts
// have more sites each and reach as many others.)
bool make_plan(const esp::HostModel &m, int k, int R, size_t lds_max, Plan &p) {
  const int N = m.N;
  p = Plan{};
  if (!cluster_fits(m, (N + k - 1) / k, R, lds_max)) return false;
  p.ngroup = (m.zmax + kGroup - 1) / kGroup;
  const int npair = p.ngroup * kGroup / 2;
  std::vector<int> part_of(N), local(N, -1), seen(N, -1);     // by device site
  for (int d = 0; d < N; ++d) part_of[d] = (int)((long long)m.dev2ref[d] * k / N);
  std::vector<std::vector<int>> own(k), hal(k);
  for (int d = 0; d < N; ++d) own[part_of[d]].push_back(d);   // device order: by colour
  std::vector<std::vector<char>> touch(k, std::vector<char>(k, 0));
  for (int j = 0; j < k; ++j) {
    for (int l = 0; l < m.zmax; ++l) {
      for (int d : own[j]) {
        const int q = m.nbr[(size_t)l * N + d];
        if (q == N || part_of[q] == j || seen[q] == j) continue;
        touch[j][part_of[q]] = touch[part_of[q]][j] = 1;      // reader and writer wait for each other
        seen[q] = j;
        hal[j].push_back(q);
      }
      if (!cluster_fits(m, (int)(own[j].size() + hal[j].size()), R, lds_max)) return false;
    }
    std::sort(hal[j].begin(), hal[j].end());                  // device order: by colour
    p.nl_max = std::max(p.nl_max, (int)(own[j].size() + hal[j].size()));
  }
  for (int j = 0; j < k; ++j) {
    Part t{};
    t.nown = (int)own[j].size();
    t.nhalo = (int)hal[j].size();
    t.own0 = (int)p.own_dev.size();
    t.hal0 = (int)p.hal_dev.size();
    t.col0 = (int)p.col_off.size();
    t.nb0 = (int)p.nbs.size();
    t.pitch = (t.nown + 63) / 64 * 64;
    t.tab0 = p.tab.size();
    for (int i = 0; i < t.nown; ++i) local[own[j][i]] = i;
    for (int i = 0; i < t.nhalo; ++i) local[hal[j][i]] = t.nown + i;
    for (int c = 0; c <= m.ncol; ++c) {
      auto cut = [&](const std::vector<int> &v) {
        return (int)(std::lower_bound(v.begin(), v.end(), m.col_off[c]) - v.begin());
      };
      p.col_off.push_back(cut(own[j]));
      p.hal_off.push_back(cut(hal[j]));
    }
    for (int q = 0; q < k; ++q)
      if (touch[j][q]) { p.nbs.push_back(q); ++t.nnb; }
    p.tab.resize(t.tab0 + (size_t)npair * t.pitch, 0u);
    for (int l = 0; l < 2 * npair; ++l) {
      unsigned *row = &p.tab[t.tab0 + (size_t)(l / 2) * t.pitch];
      const int *nbr = l < m.zmax ? &m.nbr[(size_t)l * N] : nullptr;
      for (int i = 0; i < t.nown; ++i) {
        const int q = nbr ? nbr[own[j][i]] : N;
        row[i] |= (q == N ? (unsigned)p.nl_max : (unsigned)local[q]) << (16 * (l & 1));
      }
    }
    for (int d : own[j]) {
      p.own_dev.push_back(d);
      p.own_ref.push_back(m.dev2ref[d]);
      p.own_basis.push_back(m.basis[d]);
      p.own_mag.push_back(m.mag[d]);
    }
    if (!m.compressed)
      for (int l = 0; l < m.zmax; ++l)
        for (int d : own[j]) p.own_j.push_back(m.coef[((size_t)l * N + d) * esp::kCoef]);
    for (int d : hal[j]) p.hal_dev.push_back(d);
    p.part.push_back(t);
  }
  return true;
}

}  // namespace

// Device tables of a context's clusters, one allocation.
struct esp_cluster {
  int k = 0, nl_max = 0, ngroup = 0;
  char *mem = nullptr;
  const Part *part = nullptr;
  const int *own_dev = nullptr, *own_ref = nullptr, *hal_dev = nullptr, *col_off = nullptr, *hal_off = nullptr,
            *nbs = nullptr;
  const uint8_t *own_basis = nullptr;
  const double *own_mag = nullptr, *own_j = nullptr;
  const unsigned *tab = nullptr;
  unsigned *ctl = nullptr;                   // Ctl, then the flags [R][k]
  double *partial = nullptr;
  int *slots = nullptr;
};

namespace esp {

void cluster_free(esp_ctx *c) {
  esp_cluster *q = c->cluster;
  c->cluster = nullptr;
  c->cluster_R = 0;
  if (!q) return;
  dfree(q->mem);
  delete q;
}

int cluster_built(const esp_ctx *c) { return c->cluster && c->cluster_R == c->R ? c->cluster->k : 0; }

// Decides whether clusters serve this context and builds their tables, once per (model, replica
// count).  c->cluster stays null if not.
int cluster_prepare(esp_ctx *c) {
  if (c->cluster_R == c->R) return ESP_OK;
  const HostModel &m = c->hm;
  const int k = cluster_parts(m, c->R, c->num_cu);
  // (the tables depend on the model and k, the LDS of a block also on the replica count)
  if (c->cluster && c->cluster->k == k && cluster_fits(m, c->cluster->nl_max, c->R, c->lds_max)) {
    c->cluster_R = c->R;
    return ESP_OK;
  }
  cluster_free(c);
  c->cluster_R = c->R;
  Plan p;
  if (k < 2 || !make_plan(m, k, c->R, c->lds_max, p)) return ESP_OK;
  esp_cluster *q = c->cluster = new esp_cluster();
  q->k = k; q->nl_max = p.nl_max; q->ngroup = p.ngroup;
  std::vector<char> img;
  std::vector<std::pair<const void **, size_t>> at;
  auto put = [&](auto *&ptr, const auto &v) {
    img.resize((img.size() + 255) / 256 * 256);
    at.push_back({(const void **)&ptr, img.size()});
    const char *b = reinterpret_cast<const char *>(v.data());
    img.insert(img.end(), b, b + v.size() * sizeof(v[0]));
  };
  put(q->part, p.part); put(q->own_dev, p.own_dev); put(q->own_ref, p.own_ref); put(q->hal_dev, p.hal_dev);
  put(q->col_off, p.col_off); put(q->hal_off, p.hal_off); put(q->nbs, p.nbs); put(q->own_basis, p.own_basis);
  put(q->own_mag, p.own_mag); put(q->own_j, p.own_j); put(q->tab, p.tab);
  // work areas for up to num_cu blocks (R k <= num_cu)
  put(q->partial, std::vector<double>((size_t)c->num_cu * 8));
  put(q->ctl, std::vector<unsigned>(sizeof(Ctl) / sizeof(unsigned) + (size_t)c->num_cu));
  put(q->slots, std::vector<int>((size_t)c->num_cu));
  int rc;
  if ((rc = dalloc(c, q->mem, img.size()))) {
    cluster_free(c);
    return rc;
  }
  for (const auto &[ptr, off] : at) *ptr = q->mem + off;
  HIPCHK(c, hipMemcpyAsync(q->mem, img.data(), img.size(), hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return ESP_OK;
}

// nsteps steps of M sweeps [+ measurement], an exchange after every `round` steps, from the device
// clock; launches end within steps where those are longer than kPhases.  *ran: sweeps finished; fewer
// than nsteps M where the blocks of a launch were not all resident (it changed nothing; *left), or
// another context's are on the device.
int cluster_run(esp_ctx *c, int mode, double tilt, uint64_t seed, int nsteps, int M, bool measure, bool exchange,
                int round, int64_t *ran, bool *left) {
  const HostModel &m = c->hm;
  esp_cluster *q = c->cluster;
  *ran = 0;
  *left = false;
  static std::mutex on_device[64];
  std::unique_lock<std::mutex> mine(on_device[c->device & 63], std::try_to_lock);
  if (!mine.owns_lock()) return ESP_OK;
  CArgs x{};
  x.a = base_args(c);
  x.a.tilt = tilt;
  x.a.key0 = (uint32_t)seed; x.a.key1 = (uint32_t)(seed >> 32);
  x.part = q->part;
  x.own_dev = q->own_dev; x.own_ref = q->own_ref; x.hal_dev = q->hal_dev; x.col_off = q->col_off; x.hal_off = q->hal_off;
  x.nbs = q->nbs; x.own_basis = q->own_basis; x.tab = q->tab;
  x.ctl = reinterpret_cast<Ctl *>(q->ctl);
  x.flag = q->ctl + sizeof(Ctl) / sizeof(unsigned);
  x.partial = q->partial; x.own_mag = q->own_mag; x.own_j = q->own_j; x.slots = q->slots;
  x.k = q->k; x.nl_max = q->nl_max; x.ngroup = q->ngroup;
  x.xcd = c->R % 8 == 0;
  x.round = round;
  x.f.N = m.N; x.f.R = c->R;
  x.f.e_base = c->d_ebase; x.f.e_run = c->d_erun; x.f.acc = c->d_acc; x.f.nmeas = c->d_nmeas;
  x.f.slot_rep = c->d_slot_rep; x.f.rep_slot = c->d_rep_slot; x.f.beta_slot = c->d_beta; x.f.nswap = c->d_nswap;
  x.f.clock = c->d_clock;
  x.f.key0 = (uint32_t)seed; x.f.key1 = (uint32_t)(seed >> 32); x.f.stream_base = c->stream_base;
  x.f.trace = c->d_trace; x.f.trace_cap = c->trace_cap;
  ClusterFn fn = cluster_fn(mode, m);
  const size_t shm = cluster_lds(m, q->nl_max, c->R);
  if (shm > 65536)
    HIPCHK(c, hipFuncSetAttribute((const void *)fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm));
  const int most = std::max(1, kPhases / m.ncol);           // sweeps of a launch
  const size_t nctl = sizeof(Ctl) + sizeof(unsigned) * (size_t)c->R * q->k;
  int done = 0, part = 0;                                   // steps done, sweeps of the next one done
  while (done < nsteps) {
    const bool whole = M - part <= most;                    // the launch ends a step
    x.nsteps = whole && part == 0 ? std::min(nsteps - done, most / M) : 1;
    x.M = whole ? M - part : most;
    x.measure = whole && measure;
    x.exchange = whole && exchange;
    x.step0 = done % round;
    HIPCHK(c, hipMemsetAsync(q->ctl, 0, nctl, c->stream));
    if (c->cluster_limit == 0)       // (decided before the first block asks)
      HIPCHK(c, hipMemsetD32Async((hipDeviceptr_t)&x.ctl->decided, (int)kLeave, 1, c->stream));
    else if (c->cluster_limit > 0)
      --c->cluster_limit;
    hipLaunchKernelGGL(fn, dim3(c->R * q->k), dim3(kCBlock), shm, c->stream, x);
    HIPCHK(c, hipGetLastError());
    Ctl h{};
    {
      std::lock_guard<std::mutex> lk(c->read_mu);
      espx::SmallRead rd(c->xfer, c->stream);
      rd.add(&h, q->ctl, sizeof h);
      HIPCHK(c, rd.finish());
    }
    if (h.failed) return fail(c, ESP_EHIP, "cluster sweep: a block stopped making progress");
    if (h.decided != kGo) {
      *left = true;
      return ESP_OK;
    }
    c->mpart_valid = false;
    ++c->cluster_launches;
    *ran += (int64_t)x.nsteps * x.M;
    done += whole ? x.nsteps : 0;
    part = whole ? 0 : part + x.M;
  }
  return ESP_OK;
}

}  // namespace esp

extern "C" {

int esp_plan_clusters(int N, int nb, const double *mag, int zJ, const int *j_cnt, const int *j_nbr,
                      const double *j_val, int zB, const int *b_cnt, const int *b_nbr, const double *b_val, int zD,
                      const int *d_cnt, const int *d_nbr, const double *d_vec, const int *L, int R, int num_cu,
                      int64_t lds_bytes, int64_t *out) {
  if (R < 1 || num_cu < 1 || lds_bytes < 1 || !out) return ESP_EINVAL;
  esp::HostModel hm;
  if (!esp::prepare_model(hm, N, nb, mag, zJ, j_cnt, j_nbr, j_val, zB, b_cnt, b_nbr, b_val, zD, d_cnt, d_nbr, d_vec, 0,
                          nullptr, nullptr, 0, nullptr, nullptr, L).empty())
    return ESP_EINVAL;
  const int k = cluster_parts(hm, R, num_cu);
  Plan p;
  const bool on = k >= 2 && make_plan(hm, k, R, (size_t)lds_bytes, p);
  out[0] = on ? k : 0;
  out[1] = on ? p.nl_max : 0;
  out[2] = on ? (int64_t)cluster_lds(hm, p.nl_max, R) : 0;
  return ESP_OK;
}

int esp_get_cluster_info(esp_ctx *c, int64_t *out) {
  if (!c || !out) return ESP_EINVAL;
  out[0] = esp::cluster_built(c);
  out[1] = c->cluster_sweeps;
  out[2] = c->cluster_launches;
  out[3] = c->cluster_skip;
  return ESP_OK;
}

int esp_set_cluster_limit(esp_ctx *c, int launches) {
  if (!c || launches < -1) return ESP_EINVAL;
  c->cluster_limit = launches;
  return ESP_OK;
}

}  // extern "C"
