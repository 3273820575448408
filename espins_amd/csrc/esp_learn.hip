// esp_learn.hip -- learned proposal for the Metropolis-Hastings sweep (gfx950).
//
// The energy of site i as a function of its own spin S (every other spin fixed) is
//     E_i(S) = -G.S + S^T Q S
// with G = sum_j J_ij S_j - sum_j S_j x D_ij - h a_h   (exchange, DM, Zeeman) and
//      Q = sum_j B_ij S_j S_j^T + Delta a a^T           (biquadratic, single ion),
// the same terms energy_get / delta_energy_get evaluate (get_quant.F90:186-337).  A small MLP
// maps five features of (G, Q, T) to a two-component von Mises-Fisher mixture q(S | env);
// moves are accepted with min(1, exp(-beta dE) q(S_old) / q(S_new)).  q depends only on the
// neighbours, which a colour phase never changes, so detailed balance holds for any weights:
// the network only decides how often moves are accepted.
//
// Network: 5 -> 32 -> 32 -> 32 -> 6, GELU (tanh form), BF16 weights for sampling (FP32 accumulate), FP32
// master weights for training with Adam.  Outputs per component k: log-scale s_k of the
// concentration kappa_k = beta|G| exp(s_k), weight logit, tilt t_k = (pi/2) tanh(.) of the
// mean direction from G-hat toward the nearer pole of the anisotropy axis.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "esp_ctx.h"

using namespace espd;
using namespace espk;

namespace {

constexpr int kIn = 5, kH = 32, kOut = 6;
constexpr int oW1 = 0, oB1 = oW1 + kH * kIn, oW2 = oB1 + kH, oB2 = oW2 + kH * kH, oW3 = oB2 + kH,
              oB3 = oW3 + kH * kH, oW4 = oB3 + kH, oB4 = oW4 + kOut * kH, kNP = oB4 + kOut;
static_assert(kNP == ESP_LEARN_NPARAMS, "parameter count");
constexpr int kRec = 16;   // record: x[5], kappa0, ghat[3], axis[3], s[3], pad
constexpr double kPi = 3.14159265358979323846;
// Weight of a fixed uniform-sphere component beside the two network components: the density
// of any direction stays >= kUniform / (4 pi), so a poorly fitted network slows the chain by
// at most a factor kUniform against uniform proposals instead of freezing it.
constexpr double kUniform = 1.0 / 32.0;

// Activation: GELU in its tanh form (Hendrycks & Gimpel 2016),
//   g(x) = x sigma(u),  u = c (x + 0.044715 x^3),  c = 2 sqrt(2 / pi),
// which equals 0.5 x (1 + tanh(u / 2)).  Evaluated as x / (1 + 2^(-u log2 e)) with the
// hardware exp2 and reciprocal: six VALU instructions, two of them transcendental, the same
// FP32 expression in training and in the sweep.  g'(x) = sigma + x sigma (1 - sigma) u'(x).
constexpr float kGeluC = 1.5957691216057308f;             // 2 sqrt(2 / pi)
constexpr float kGeluK = 2.3022081983067571f;             // 2 sqrt(2 / pi) log2(e)
__device__ __forceinline__ float gelu_sigma(float x) {
  const float a = x * fmaf(x * x, 0.044715f * kGeluK, kGeluK);
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-a));
}
__device__ __forceinline__ float act(float x) { return x * gelu_sigma(x); }
__device__ __forceinline__ float act_d(float x) {
  const float sg = gelu_sigma(x);
  return sg + x * sg * (1.0f - sg) * kGeluC * fmaf(x * x, 3.0f * 0.044715f, 1.0f);
}

// MLP forward (weights w in any address space).
__device__ __forceinline__ void mlp_forward(const float *w, const float x[kIn], float out[kOut]) {
  float h1[kH], h2[kH];
#pragma unroll 4
  for (int i = 0; i < kH; ++i) {
    float s = w[oB1 + i];
#pragma unroll
    for (int k = 0; k < kIn; ++k) s += w[oW1 + i * kIn + k] * x[k];
    h1[i] = act(s);
  }
#pragma unroll 2
  for (int i = 0; i < kH; ++i) {
    float s = w[oB2 + i];
#pragma unroll 8
    for (int k = 0; k < kH; ++k) s += w[oW2 + i * kH + k] * h1[k];
    h2[i] = act(s);
  }
#pragma unroll 2
  for (int i = 0; i < kH; ++i) {
    float s = w[oB3 + i];
#pragma unroll 8
    for (int k = 0; k < kH; ++k) s += w[oW3 + i * kH + k] * h2[k];
    h1[i] = act(s);  // h3
  }
#pragma unroll
  for (int i = 0; i < kOut; ++i) {
    float s = w[oB4 + i];
#pragma unroll 8
    for (int k = 0; k < kH; ++k) s += w[oW4 + i * kH + k] * h1[k];
    out[i] = s;
  }
}

// log(1 - kUniform), log(kUniform / (4 pi)), log(2 pi)
constexpr double kLog1mU = -0.0317486983145803;
constexpr double kLogUni = -5.996760149769017;
constexpr double kLog2Pi = 1.8378770664093453;

// The proposal density of one site:
//   q(x) = (1 - kUniform) sum_k w_k vMF(x; kappa_k, mu_k) + kUniform / (4 pi).
// The parameters (w, kappa, mu) are computed from the network outputs in FP32 -- any
// values work, provided sampling and density use the same ones -- and promoted to FP64;
// the density, its normaliser and the sampler are FP64.
// ---- the sweep's network: hidden layers on the matrix cores --------------------------------
// One wave evaluates the network for its 64 lanes' inputs.  Layer 1 (5 -> 32) and the output
// layer (32 -> 6) run per lane in FP32; the two 32 x 32 layers run as
//   Z^T = W H^T   (v_mfma_f32_32x32x16_bf16: A = W, B = H^T, D = Z^T)
// with BF16 weights and activations and FP32 accumulation, two 32-proposal column blocks per
// wave.  Operand layouts of the instruction (lane l, half h = l / 32):
//   A[32][16]: A[l % 32][8 h + e], e < 8        B[16][32]: B[8 h + e][l % 32]
//   D[32][32]: register v holds D[8 (v / 4) + 4 h + v % 4][l % 32]
// A lane's D registers cover hidden units {8 q + 4 h + r} of one proposal; the B fragment of
// the next layer needs units {16 ks + 8 h + e}: half of them are the partner lane's (l ^ 32),
// exchanged with one cross-half shuffle per register pair.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
// Two floats to BF16, round to nearest even, lo in bits 0-15: one v_cvt_pk_bf16_f32 on gfx950.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const floatx2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

__device__ __forceinline__ bf16x8 frag(uint32_t d0, uint32_t d1, uint32_t d2, uint32_t d3) {
  uint4 u = make_uint4(d0, d1, d2, d3);
  return __builtin_bit_cast(bf16x8, u);
}

// W2 / W3 A-fragments (BF16, from global memory): row l % 32, columns 16 ks + 8 h + 0..7.
struct NetA {
  bf16x8 a[2][2];   // [layer 2 / 3][ks]
};
__device__ __forceinline__ NetA load_net_a(const uint16_t *wbf16) {
  NetA n;
  const int l = threadIdx.x & 63, h = l >> 5, i = l & 31;
#pragma unroll
  for (int layer = 0; layer < 2; ++layer)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const uint4 u = *reinterpret_cast<const uint4 *>(wbf16 + (layer ? oW3 : oW2) + i * kH + 16 * ks + 8 * h);
      n.a[layer][ks] = __builtin_bit_cast(bf16x8, u);
    }
  return n;
}

// B fragments of one 32-proposal column block from D registers (after the activation):
// keep q in {h, 2 + h}, exchange q in {1 - h, 3 - h} with the partner lane.
__device__ __forceinline__ void d_to_b(const floatx16 &z, int h, bf16x8 b[2]) {
  uint32_t p[8];   // p[2 q + r / 2]: units 8 q + 4 h + r, r = 0..3, as BF16 pairs
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    p[2 * q] = pack_bf16(z[4 * q], z[4 * q + 1]);
    p[2 * q + 1] = pack_bf16(z[4 * q + 2], z[4 * q + 3]);
  }
  // send q = 1 - h and q = 3 - h; receive the partner's q = h' for the same slots
  const uint32_t s0 = h ? p[0] : p[2], s1 = h ? p[1] : p[3];
  const uint32_t s2 = h ? p[4] : p[6], s3 = h ? p[5] : p[7];
  const uint32_t r0 = __shfl_xor(s0, 32, 64), r1 = __shfl_xor(s1, 32, 64);
  const uint32_t r2 = __shfl_xor(s2, 32, 64), r3 = __shfl_xor(s3, 32, 64);
  // ks = 0: units 8 h + 0..7; ks = 1: units 16 + 8 h + 0..7
  //   h = 0: [own q = 2 ks | partner q = 2 ks];   h = 1: [partner q = 2 ks + 1 | own q = 2 ks + 1]
  b[0] = h ? frag(r0, r1, p[2], p[3]) : frag(p[0], p[1], r0, r1);
  b[1] = h ? frag(r2, r3, p[6], p[7]) : frag(p[4], p[5], r2, r3);
}

__device__ __forceinline__ floatx16 bias_d(const float *b, int h) {
  floatx16 z;
#pragma unroll
  for (int v = 0; v < 16; ++v) z[v] = b[8 * (v >> 2) + 4 * h + (v & 3)];
  return z;
}

// Network of the sweep for the calling lane's input x (every lane of the wave must call).
// wl: FP32 weights in LDS (layer 1, biases, layer 4 from the BF16 copy); na: W2/W3 fragments.
__device__ __forceinline__ void net_forward_mfma(const float *wl, const NetA &na, const float x[kIn],
                                                 float out[kOut]) {
  const int l = threadIdx.x & 63, h = l >> 5;
  // layer 1 per lane, then B fragments: own units 16 ks + 8 h + e for column block h, the
  // partner's same units for column block 1 - h
  uint32_t own[8], snd[8];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float z[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const int u = 16 * ks + 8 * (half ^ h) + e + t;   // half 0: own units, 1: the partner's
          float acc = wl[oB1 + u];
#pragma unroll
          for (int k = 0; k < kIn; ++k) acc += wl[oW1 + u * kIn + k] * x[k];
          z[t] = act(acc);
        }
        (half ? snd : own)[4 * ks + e / 2] = pack_bf16(z[0], z[1]);
      }
  uint32_t rcv[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) rcv[k] = __shfl_xor(snd[k], 32, 64);
  bf16x8 b[2][2];   // [column block][ks]
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const bf16x8 mine = frag(own[4 * ks], own[4 * ks + 1], own[4 * ks + 2], own[4 * ks + 3]);
    const bf16x8 theirs = frag(rcv[4 * ks], rcv[4 * ks + 1], rcv[4 * ks + 2], rcv[4 * ks + 3]);
    b[0][ks] = h ? theirs : mine;
    b[1][ks] = h ? mine : theirs;
  }
  // layers 2 and 3 on the matrix cores
  floatx16 z[2];
#pragma unroll
  for (int layer = 0; layer < 2; ++layer) {
    const float *bias = wl + (layer ? oB3 : oB2);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      z[cb] = bias_d(bias, h);
      z[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(na.a[layer][0], b[cb][0], z[cb], 0, 0, 0);
      z[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(na.a[layer][1], b[cb][1], z[cb], 0, 0, 0);
#pragma unroll
      for (int v = 0; v < 16; ++v) z[cb][v] = act(z[cb][v]);
    }
    if (layer == 0)
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) d_to_b(z[cb], h, b[cb]);
  }
  // output layer: partial sums over this lane's 16 units of each column block, completed
  // with the partner's; the lane's own proposal is column block h
#pragma unroll
  for (int q = 0; q < kOut; ++q) {
    float part[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      float acc = 0.0f;
#pragma unroll
      for (int v = 0; v < 16; ++v) acc += wl[oW4 + q * kH + 8 * (v >> 2) + 4 * h + (v & 3)] * z[cb][v];
      part[cb] = acc;
    }
    const float give = h ? part[0] : part[1];     // the partner's column block
    const float got = __shfl_xor(give, 32, 64);
    out[q] = wl[oB4 + q] + (h ? part[1] : part[0]) + got;
  }
}

__device__ __forceinline__ V3 vnorm(V3 v) {
  const double r = rsqrt(dot(v, v));
  return {v.x * r, v.y * r, v.z * r};
}

// Unit vector in the (ghat, axis) plane, normal to ghat, toward the pole of the axis nearer
// to ghat (any normal when ghat is along the axis).
__device__ __forceinline__ V3 tilt_frame(const V3 &ghat, const V3 &ax) {
  const double c = dot(ghat, ax);
  const double sgn = c < 0.0 ? -1.0 : 1.0;
  V3 e = {sgn * ax.x - sgn * c * ghat.x, sgn * ax.y - sgn * c * ghat.y, sgn * ax.z - sgn * c * ghat.z};
  if (dot(e, e) < 1e-24) e = fabs(ghat.x) < 0.9 ? V3{0.0, -ghat.z, ghat.y} : V3{-ghat.z, 0.0, ghat.x};
  return vnorm(e);
}

__device__ __forceinline__ float softplusf(float z) { return fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z))); }

// One component of the mixture in the log domain, from its outputs (o0: concentration, o1: weight
// logit, o2: tilt), the other component's weight logit p1 and the local frame (ghat, e).
struct Comp {
  double logw;      // log of (1 - kUniform) w_k
  double kappa;
  double lnorm;     // log of kappa / (2 pi (1 - e^{-2 kappa})): vMF density = exp(lnorm + kappa (mu.x - 1))
  double t;         // tilt angle of mu_k from ghat
  V3 mu;
};
__device__ __forceinline__ Comp make_comp(float o0, float o1, float o2, float p1, float kappa0, const V3 &ghat,
                                          const V3 &e) {
  Comp m;
  m.logw = (double)(-softplusf(p1 - o1)) + kLog1mU;   // log softmax of the two weight logits
  const float sc = fminf(fmaxf(o0, -8.0f), 8.0f);
  m.kappa = (double)(kappa0 * expf(sc)) + 1e-6;
  m.lnorm = log(m.kappa / -expm1(-2.0 * m.kappa)) - kLog2Pi;
  const float th = tanhf(o2);
  float sn, cs;
  sincospif(0.5f * th, &sn, &cs);
  m.t = 0.5 * kPi * (double)th;
  m.mu = vnorm(V3{cs * ghat.x + sn * e.x, cs * ghat.y + sn * e.y, cs * ghat.z + sn * e.z});
  return m;
}
// log of (1 - kUniform) w_k vMF_k(x), log vMF(x) = lnorm + kappa (mu . x - 1)
__device__ __forceinline__ double log_part(const Comp &m, const V3 &x) {
  return m.logw + (m.lnorm + m.kappa * (dot(m.mu, x) - 1.0));
}
// Log density of the mixture from its two components' parts.
__device__ __forceinline__ double log_mix(double l0, double l1) {
  const double mx = fmax(fmax(l0, l1), kLogUni);
  return mx + log(exp(l0 - mx) + exp(l1 - mx) + exp(kLogUni - mx));
}

// The mixture as the sweep uses it, without logarithms: selection weights ws_k = (1 - kUniform)
// w_k, concentrations, e^{-2 kappa_k} and density prefactors c_k = ws_k kappa_k / (2 pi (1 -
// e^{-2 kappa_k})), so that q(x) = sum_k c_k exp(kappa_k (mu_k . x - 1)) + kUniform / (4 pi).
// Sampling and density use the same ws_k, kappa_k and mu_k (the log-domain mixture of training
// differs from it only by rounding, which no sweep quantity depends on).
struct MixS {
  double ws0;       // selection weight of component 0 (component 1: 1 - kUniform - ws0)
  double kappa[2], e2k[2], c[2];
  V3 mu[2];
};
__device__ __forceinline__ MixS make_mix_sweep(const float o[kOut], float kappa0, const V3 &ghat, const V3 &ax) {
  MixS m;
  const V3 e = tilt_frame(ghat, ax);
  const double w0 = (double)__builtin_amdgcn_rcpf(1.0f + __expf(o[4] - o[1]));   // softmax of the logits
  const double ws[2] = {(1.0 - kUniform) * w0, (1.0 - kUniform) * (1.0 - w0)};
  m.ws0 = ws[0];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const float sc = fminf(fmaxf(o[3 * k], -8.0f), 8.0f);
    const double kap = (double)(kappa0 * expf(sc)) + 1e-6;
    m.kappa[k] = kap;
    // e^{-2 kappa} < 2^-54 for kappa > 19: expm1 would round to exactly -1 there
    const double em1 = kap > 19.0 ? -1.0 : expm1(-2.0 * kap);
    m.e2k[k] = 1.0 + em1;
    m.c[k] = ws[k] * kap / (2.0 * kPi * -em1);
    const float th = tanhf(o[3 * k + 2]);
    float sn, cs;
    sincospif(0.5f * th, &sn, &cs);
    m.mu[k] = vnorm(V3{cs * ghat.x + sn * e.x, cs * ghat.y + sn * e.y, cs * ghat.z + sn * e.z});
  }
  return m;
}

// Wood (1994) for S^2: w = 1 + log(v + (1 - v) e^{-2 kappa}) / kappa, azimuth 2 pi u; kappa = 0
// is the uniform density (w = 2 v - 1).
__device__ __forceinline__ V3 sample_vmf(double kappa, double e2k, const V3 &mu, double v, double u) {
  double w = kappa > 0.0 ? 1.0 + log(v + (1.0 - v) * e2k) / kappa : 2.0 * v - 1.0;
  w = fmin(1.0, fmax(-1.0, w));
  const double st = sqrt(fmax(0.0, 1.0 - w * w));
  const V3 e1 = vnorm(fabs(mu.x) < 0.9 ? V3{0.0, -mu.z, mu.y} : V3{-mu.z, 0.0, mu.x});
  const V3 e2 = {mu.y * e1.z - mu.z * e1.y, mu.z * e1.x - mu.x * e1.z, mu.x * e1.y - mu.y * e1.x};
  double sp, cp;
  sincospi(2.0 * u, &sp, &cp);
  return {w * mu.x + st * (cp * e1.x + sp * e2.x), w * mu.y + st * (cp * e1.y + sp * e2.y),
          w * mu.z + st * (cp * e1.z + sp * e2.z)};
}

// Local environment of device site d of one replica: G, Q_B (xx,yy,zz,xy,xz,yz).
template <bool CMP, bool HB, bool HD, class SP>
__device__ __forceinline__ void local_env(const KArgs &a, const SP &sp, const double *ctab, int d,
                                          V3 &G, double QB[6]) {
  G = {0, 0, 0};
  for (int k = 0; k < 6; ++k) QB[k] = 0.0;
  const double *crow = CMP ? ctab + (size_t)a.basis[d] * a.zmax * 5 : nullptr;
  const unsigned ud = (unsigned)d;
  for (int l0 = 0; l0 < a.zmax; l0 += kChunkLearn) {
    unsigned jj[kChunkLearn];
    V3 sv[kChunkLearn];
#pragma unroll
    for (int u = 0; u < kChunkLearn; ++u) {
      const int l = l0 + u < a.zmax ? l0 + u : 0;
      jj[u] = (unsigned)ld_off(a.nbr, ((unsigned)l * (unsigned)a.N + ud) * 4u);
    }
#pragma unroll
    for (int u = 0; u < kChunkLearn; ++u) sv[u] = sp.ld(jj[u]);
#pragma unroll
    for (int u = 0; u < kChunkLearn; ++u) {
      const int l = l0 + u;
      if (l >= a.zmax) continue;
      const V3 sj = sv[u];
      double cj, cb = 0, cx = 0, cy = 0, cz = 0;
      if (CMP) {
        cj = crow[5 * l];
        if (HB) cb = crow[5 * l + 1];
        if (HD) { cx = crow[5 * l + 2]; cy = crow[5 * l + 3]; cz = crow[5 * l + 4]; }
      } else {
        cj = a.cJ[(size_t)l * a.N + d];
        if (HB) cb = a.cB[(size_t)l * a.N + d];
        if (HD) {
          const double *dv = a.cD + 3 * ((size_t)l * a.N + d);
          cx = dv[0]; cy = dv[1]; cz = dv[2];
        }
      }
      G.x += cj * sj.x; G.y += cj * sj.y; G.z += cj * sj.z;
      if (HD) {  // -(S_j x D)
        G.x -= sj.y * cz - sj.z * cy;
        G.y -= sj.z * cx - sj.x * cz;
        G.z -= sj.x * cy - sj.y * cx;
      }
      if (HB) {
        QB[0] += cb * sj.x * sj.x; QB[1] += cb * sj.y * sj.y; QB[2] += cb * sj.z * sj.z;
        QB[3] += cb * sj.x * sj.y; QB[4] += cb * sj.x * sj.z; QB[5] += cb * sj.y * sj.z;
      }
    }
  }
  if (a.has_h) {
    const double *h = a.h4 + 4 * a.basis[d];
    G.x -= h[0] * h[1]; G.y -= h[0] * h[2]; G.z -= h[0] * h[3];
  }
}

__device__ __forceinline__ double quad(const double Q[6], const V3 &s) {
  return Q[0] * s.x * s.x + Q[1] * s.y * s.y + Q[2] * s.z * s.z +
         2.0 * (Q[3] * s.x * s.y + Q[4] * s.x * s.z + Q[5] * s.y * s.z);
}

// Features of the network from the environment of a spin of length mag: the site energy of
// direction x is beta E = -kappa0 (ghat.x) + beta mag^2 x^T Q x with kappa0 = beta mag |G|.
//   x0 = log(1 + kappa0)                    strength of the local field
//   x1 = |ghat . a|                         field direction against the anisotropy axis
//   x2 = log T
//   x3 = beta mag^2 (ghat^T Q_B ghat - tr Q_B / 3)   biquadratic projection on the field
//   x4 = beta mag^2 Delta                   single-ion anisotropy
__device__ __forceinline__ void features(const V3 &G, const double QB[6], const V3 &ax, double Delta,
                                         double beta, double mag, float x[kIn], float &kappa0, V3 &ghat) {
  const double g2 = dot(G, G);
  double g = 0.0;
  if (g2 > 1e-300) {
    g = sqrt(g2);
    const double r = 1.0 / g;
    ghat = {G.x * r, G.y * r, G.z * r};
  } else {
    ghat = ax;
  }
  kappa0 = (float)(beta * mag * g);
  const float bm2 = (float)(beta * mag * mag);
  const float trq = (float)(QB[0] + QB[1] + QB[2]);
  x[0] = log1pf(kappa0);
  x[1] = fabsf((float)dot(ghat, ax));
  x[2] = logf((float)(1.0 / beta));
  x[3] = bm2 * ((float)quad(QB, ghat) - trq * (1.0f / 3.0f));
  x[4] = bm2 * (float)Delta;
}

__device__ __forceinline__ void axis_of(const KArgs &a, int d, V3 &ax, double &Delta) {
  if (a.has_si) {
    const double *k = a.si4 + 4 * a.basis[d];
    Delta = k[0];
    ax = {k[1], k[2], k[3]};
  } else {
    Delta = 0.0;
    ax = {0.0, 0.0, 1.0};
  }
}

// One colour phase with learned proposals (global-memory path, one lane per site).
#ifndef ESP_LEARN_WAVES
#define ESP_LEARN_WAVES 4        // > 0: ask the compiler for this many waves per SIMD (4: no spills, no AGPRs)
#endif
#if ESP_LEARN_WAVES > 0
#define ESP_LEARN_ATTR __attribute__((amdgpu_waves_per_eu(ESP_LEARN_WAVES)))
#else
#define ESP_LEARN_ATTR
#endif

template <bool CMP, bool HB, bool HD>
__global__ __launch_bounds__(kBlock) ESP_LEARN_ATTR void k_phase_learned(KArgs a, const uint16_t *wbf16) {
  extern __shared__ double s_dyn[];  // [ctab][weights as float]
  int r, b;
  espg::place_block(blockIdx.x, a.xcd_full, a.dnblk, r, b);
  if (r >= a.R) return;
  const int nct = CMP ? a.nb * a.zmax * 5 : 0;
  double *ctab = s_dyn;
  float *w = reinterpret_cast<float *>(s_dyn + nct);
  for (int k = threadIdx.x; k < nct; k += kBlock) ctab[k] = a.ctab[k];
  for (int k = threadIdx.x; k < kNP; k += kBlock) w[k] = __uint_as_float((uint32_t)wbf16[k] << 16);
  __syncthreads();
  // every lane runs the network (matrix instructions need the whole wave); lanes past the
  // colour class evaluate a stand-in site and write nothing
  const int k = b * kBlock + threadIdx.x;
  const bool active = k < a.c_count;
  const int d = a.c_begin + (active ? k : 0);
  const int slot = a.rep_slot[r];
  const double beta = a.beta_slot[slot];
  const unsigned long long sweep = a.clock->sweep + (unsigned long long)a.sweep_off;
  double *base = a.sp + (size_t)r * 3 * a.Ns;
  const GSpins sp{base, base + a.Ns, base + 2 * a.Ns};
  const int wave = (b * kBlock + threadIdx.x) >> 6;
  const bool own = wave * 64 < a.c_count;
  const double wold = wave_old(a, r, wave, own);
  V3 G;
  double QB[6];
  local_env<CMP, HB, HD>(a, sp, ctab, d, G, QB);
  V3 ax;
  double Delta;
  axis_of(a, d, ax, Delta);
  double Q[6] = {QB[0] + Delta * ax.x * ax.x, QB[1] + Delta * ax.y * ax.y, QB[2] + Delta * ax.z * ax.z,
                 QB[3] + Delta * ax.x * ax.y, QB[4] + Delta * ax.x * ax.z, QB[5] + Delta * ax.y * ax.z};
  const double mag = a.mag[d];
  float x[kIn], o[kOut];
  float kappa0;
  V3 ghat;
  features(G, QB, ax, Delta, beta, mag, x, kappa0, ghat);
  net_forward_mfma(w, load_net_a(wbf16), x, o);
  const MixS mix = make_mix_sweep(o, kappa0, ghat, ax);
  const int ir = a.dev2ref[d];
  const uint4 rn = philox10(make_uint4((uint32_t)ir, (uint32_t)sweep, (uint32_t)(sweep >> 32),
                                       a.stream_base + (uint32_t)r),
                            a.key0, a.key1);
  // component: uniform with probability kUniform, else network component 0 or 1
  const double uc = u01(rn.x);
  const int comp = uc < kUniform ? 2 : (uc - kUniform < mix.ws0 ? 0 : 1);
  // select by value (a dynamic index into the register-resident mixture would spill it)
  const bool one = comp == 1;
  const V3 xn = sample_vmf(comp == 2 ? 0.0 : (one ? mix.kappa[1] : mix.kappa[0]),
                           comp == 2 ? 1.0 : (one ? mix.e2k[1] : mix.e2k[0]),
                           comp == 2 ? ghat : (one ? mix.mu[1] : mix.mu[0]), u01(rn.y), u01(rn.z));
  const V3 so = sp.ld((unsigned)d);
  const V3 sn = {mag * xn.x, mag * xn.y, mag * xn.z};
  const V3 xo = vnorm(so);
  const double dE = -(G.x * (sn.x - so.x) + G.y * (sn.y - so.y) + G.z * (sn.z - so.z)) + quad(Q, sn) - quad(Q, so);
  // Metropolis-Hastings ratio exp(-beta dE) q(xo) / q(xn) with q in the linear domain: the
  // uniform component keeps both densities >= kUniform / (4 pi) > 0
  const double c0 = mix.c[0], c1 = mix.c[1];
  const double cu = kUniform / (4.0 * kPi);
  const double qo = c0 * exp(mix.kappa[0] * (dot(mix.mu[0], xo) - 1.0)) +
                    c1 * exp(mix.kappa[1] * (dot(mix.mu[1], xo) - 1.0)) + cu;
  const double qn = c0 * exp(mix.kappa[0] * (dot(mix.mu[0], xn) - 1.0)) +
                    c1 * exp(mix.kappa[1] * (dot(mix.mu[1], xn) - 1.0)) + cu;
  const double ratio = exp(-beta * dE) * qo / qn;
  const bool acc = ratio >= 1.0 || u01(rn.w) < ratio;
  if (active && acc) {
    sp.x[d] = sn.x; sp.y[d] = sn.y; sp.z[d] = sn.z;
  }
  const unsigned long long m = __ballot(active && !acc);
  if ((threadIdx.x & 63) == 0 && m) rej_add(a.rej, a.R, slot, (unsigned long long)__popcll(m));
  Proposal pr;
  pr.so = so; pr.sn = sn; pr.u3 = 0.0;
  wave_sums(a, r, wave, own, active, !acc, dE, pr, wold);   // accepted dE into the wave's accumulator
}

// Records of local conditionals: n random (replica, site) pairs of the current state.
template <bool CMP, bool HB, bool HD>
__global__ __launch_bounds__(kBlock) void k_collect(KArgs a, int n, uint32_t s0, uint32_t s1, float *out) {
  extern __shared__ double s_dyn[];
  const int nct = CMP ? a.nb * a.zmax * 5 : 0;
  for (int k = threadIdx.x; k < nct; k += kBlock) s_dyn[k] = a.ctab[k];
  __syncthreads();
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= n) return;
  const uint4 rn = philox10(make_uint4((uint32_t)t, 0x636f6cu, 0u, 0u), s0, s1);
  const int r = (int)(rn.x % (uint32_t)a.R);
  const int d = (int)(rn.y % (uint32_t)a.N);
  double *base = a.sp + (size_t)r * 3 * a.Ns;
  const GSpins sp{base, base + a.Ns, base + 2 * a.Ns};
  V3 G;
  double QB[6];
  local_env<CMP, HB, HD>(a, sp, s_dyn, d, G, QB);
  V3 ax;
  double Delta;
  axis_of(a, d, ax, Delta);
  const double beta = a.beta_slot[a.rep_slot[r]];
  float x[kIn];
  float kappa0;
  V3 ghat;
  features(G, QB, ax, Delta, beta, a.mag[d], x, kappa0, ghat);
  const V3 s = vnorm(sp.ld((unsigned)d));
  float *rec = out + (size_t)t * kRec;
  for (int k = 0; k < kIn; ++k) rec[k] = x[k];
  rec[5] = kappa0;
  rec[6] = (float)ghat.x; rec[7] = (float)ghat.y; rec[8] = (float)ghat.z;
  rec[9] = (float)ax.x; rec[10] = (float)ax.y; rec[11] = (float)ax.z;
  rec[12] = (float)s.x; rec[13] = (float)s.y; rec[14] = (float)s.z;
  rec[15] = (float)((size_t)r * a.N + a.dev2ref[d]);  // replica * N + site (exact below 2^24)
}

// Unit vector stored at rec[o..o+2] (records hold FP32; renormalised in FP64).
__device__ __forceinline__ V3 rec_vec(const float *rec, int o) {
  return vnorm(V3{(double)rec[o], (double)rec[o + 1], (double)rec[o + 2]});
}

// ---- training: gradient of the mean negative log-likelihood ------------------------------------
// One block per 128 records, one wave per 16 of them from the first layer to the last delta: a
// layer is a 32 x 32 by 32 x 16 product on the FP32 matrix instructions (16 x 16 x 4, two unit
// tiles), which round like a chain of FMAs over the inputs in order.  Weights lie in LDS; a
// layer's values go through LDS rows [unit][record], where a wave reads only what it wrote (no
// block barrier between layers) and where the parameter gradients are summed from, up to
// five entries per thread, over the block's records in order.  Every sum has a fixed order -- inputs,
// records, blocks ascending -- and products enter the gradient sums rounded: Adam divides a
// gradient by its own size, so a changed rounding of an entry near zero changes its sign and the
// weight by a whole step (summing gradients on the matrix cores too moved epoch losses by 3e-7).
// A minibatch of 2048 records is 16 blocks, so the time is one block's chain of layers: 185 us
// with a record per thread and rows [record][unit] in LDS, 25 us on FMAs with scalar weights
// (whose loads it waited for), 18 us so -- the mixture's FP64 and the gradients' LDS reads.
constexpr int kTrainRec = 128;        // records of a block
constexpr int kTrainThreads = 512;    // 16 records a wave
constexpr int kTrow = kTrainRec + 4;  // LDS row of one unit's values over the block's records
constexpr int kWrow = kH + 4;         // LDS row of a weight matrix: 16 rows x 4 columns on 64 banks
struct TrainLds {
  float x[kIn][kTrow], g4[kOut][kTrow], one[kTrow];
  float a1[kH][kTrow], a2[kH][kTrow], a3[kH][kTrow], d1[kH][kTrow], d2[kH][kTrow], d3[kH][kTrow];
  float w1[kH][8], w2[kH][kWrow], w3[kH][kWrow], w4[16][kWrow];   // w1's columns and w4's rows padded with 0
  float b1[kH], b2[kH], b3[kH], b4[16];
  double loss[kTrainRec];
};
using F4 = float __attribute__((ext_vector_type(4)));
__device__ __forceinline__ F4 mfma4(float a, float b, F4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}
// LDS written by a wave's lanes, read by others of the same wave.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}
// z += W in for one wave's records; lane (h, c): record i of column c, units 16 t + 4 h + r in
// z[t][r].  TR: W transposed.
template <bool TR>
__device__ __forceinline__ void layer_mfma(const float (&w)[kH][kWrow], const float (&in)[kH][kTrow], int i, int h,
                                           int c, F4 (&z)[2]) {
#pragma unroll
  for (int s = 0; s < kH / 4; ++s) {
    const float b = in[4 * s + h][i];
#pragma unroll
    for (int t = 0; t < 2; ++t) z[t] = mfma4(TR ? w[4 * s + h][16 * t + c] : w[16 * t + c][4 * s + h], b, z[t]);
  }
}
__device__ __forceinline__ void bias4(const float (&b)[kH], int h, F4 (&z)[2]) {
#pragma unroll
  for (int t = 0; t < 2; ++t) z[t] = *reinterpret_cast<const F4 *>(&b[16 * t + 4 * h]);
}
// A gradient term: the product is rounded before it is added.
__device__ __forceinline__ float mad(float s, float d, float a) {
#pragma clang fp contract(off)
  const float p = d * a;
  return s + p;
}

__global__ __launch_bounds__(kTrainThreads) void k_train_block(const float *w, const float *recs, int n,
                                                               const int *perm, int off, float *part_grad,
                                                               double *part_loss) {
  extern __shared__ double s_tr[];
  TrainLds &t = *reinterpret_cast<TrainLds *>(s_tr);
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 4, c = lane & 15;
  const int i = 16 * (tid >> 6) + c, ir = blockIdx.x * kTrainRec + i;
  const bool on = ir < n;                         // rows of records past n hold zeros: they add nothing
  const float *rec = recs + (size_t)(perm ? perm[off + (on ? ir : 0)] : off + (on ? ir : 0)) * kRec;
  const float x0 = rec[h], x1 = h ? 0.f : rec[4];  // inputs h and 4 + h (kIn = 5)
  float rv[10];                                   // kappa_0, ghat, axis, spin
#pragma unroll
  for (int k = 0; k < 10; ++k) rv[k] = rec[5 + k];
  for (int e = tid; e < kH * 8; e += kTrainThreads) t.w1[e >> 3][e & 7] = (e & 7) < kIn ? w[oW1 + (e >> 3) * kIn + (e & 7)] : 0.f;
#pragma unroll
  for (int e = tid; e < kH * kH; e += kTrainThreads) {
    t.w2[e >> 5][e & 31] = w[oW2 + e];
    t.w3[e >> 5][e & 31] = w[oW3 + e];
  }
  if (tid < 16 * kH) t.w4[tid >> 5][tid & 31] = tid < kOut * kH ? w[oW4 + tid] : 0.f;
  if (tid < kH) { t.b1[tid] = w[oB1 + tid]; t.b2[tid] = w[oB2 + tid]; t.b3[tid] = w[oB3 + tid]; }
  if (tid < 16) t.b4[tid] = tid < kOut ? w[oB4 + tid] : 0.f;
  if (tid < kTrainRec) t.one[tid] = 1.f;
  t.x[h][i] = on ? x0 : 0.f;
  if (h == 0) t.x[4][i] = on ? x1 : 0.f;
  __syncthreads();

  F4 z[2], g1[2], g2[2], g3[2];                   // g: derivatives of the activations
  auto put = [&](float (&a)[kH][kTrow], F4 (&g)[2]) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        a[16 * m + 4 * h + r][i] = on ? act(z[m][r]) : 0.f;
        g[m][r] = act_d(z[m][r]);
      }
    wave_lds_sync();
  };
  bias4(t.b1, h, z);
#pragma unroll
  for (int m = 0; m < 2; ++m) z[m] = mfma4(t.w1[16 * m + c][4 + h], x1, mfma4(t.w1[16 * m + c][h], x0, z[m]));
  put(t.a1, g1);
  bias4(t.b2, h, z);
  layer_mfma<false>(t.w2, t.a1, i, h, c, z);
  put(t.a2, g2);
  bias4(t.b3, h, z);
  layer_mfma<false>(t.w3, t.a2, i, h, c, z);
  put(t.a3, g3);
  F4 zo = *reinterpret_cast<const F4 *>(&t.b4[4 * h]);
#pragma unroll
  for (int s = 0; s < kH / 4; ++s) zo = mfma4(t.w4[c][4 * s + h], t.a3[4 * s + h][i], zo);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * h + r < kOut) t.g4[4 * h + r][i] = zo[r];
  wave_lds_sync();
  {   // mixture, loss and d loss / d outputs in FP64: the lane's component k = h & 1, the other by a shuffle
    const int k = h & 1;
    const float o0 = t.g4[3 * k][i], o1 = t.g4[3 * k + 1][i], o2 = t.g4[3 * k + 2][i], p1 = t.g4[4 - 3 * k][i];
    wave_lds_sync();
    const V3 ghat = rec_vec(rv, 1), ax = rec_vec(rv, 4), sp = rec_vec(rv, 7);
    const V3 e = tilt_frame(ghat, ax);
    const Comp m = make_comp(o0, o1, o2, p1, rv[0], ghat, e);
    const double lv = log_part(m, sp), lse = log_mix(lv, __shfl_xor(lv, 16));
    if (h == 0) t.loss[i] = on ? -lse : 0.0;
    const double rk = exp(lv - lse);             // responsibility of the component
    const double rnet = rk + __shfl_xor(rk, 16); // ... of the network part
    const double dlk = 1.0 / m.kappa - 2.0 / expm1(2.0 * m.kappa) + (dot(m.mu, sp) - 1.0);  // d log f / d kappa
    const double sraw = (double)o0;
    const double dks = (sraw > -8.0 && sraw < 8.0) ? (m.kappa - 1e-6) : 0.0;                // d kappa / d o
    const double th = m.t / (0.5 * kPi);
    double sn, cs;
    sincos(m.t, &sn, &cs);
    const V3 dmu = {-sn * ghat.x + cs * e.x, -sn * ghat.y + cs * e.y, -sn * ghat.z + cs * e.z};
    if (h < 2) {
      t.g4[3 * k][i] = on ? (float)(-rk * dlk * dks) : 0.f;
      t.g4[3 * k + 1][i] = on ? (float)(exp(m.logw - kLog1mU) * rnet - rk) : 0.f;
      t.g4[3 * k + 2][i] = on ? (float)(-rk * m.kappa * dot(dmu, sp) * 0.5 * kPi * (1.0 - th * th)) : 0.f;
    }
    wave_lds_sync();
  }
  auto back = [&](float (&d)[kH][kTrow], const F4 (&g)[2]) {
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r) d[16 * m + 4 * h + r][i] = z[m][r] * g[m][r];
    wave_lds_sync();
  };
  const float q0 = t.g4[h][i], q1 = h < 2 ? t.g4[4 + (h & 1)][i] : 0.f;   // output deltas h and 4 + h
#pragma unroll
  for (int m = 0; m < 2; ++m)
    z[m] = mfma4(t.w4[4 + h][16 * m + c], q1, mfma4(t.w4[h][16 * m + c], q0, F4{0.f, 0.f, 0.f, 0.f}));
  back(t.d3, g3);
  z[0] = z[1] = F4{0.f, 0.f, 0.f, 0.f};
  layer_mfma<true>(t.w3, t.d3, i, h, c, z);
  back(t.d2, g2);
  z[0] = z[1] = F4{0.f, 0.f, 0.f, 0.f};
  layer_mfma<true>(t.w2, t.d2, i, h, c, z);
  back(t.d1, g1);
  __syncthreads();

  float *g = part_grad + (size_t)blockIdx.x * kNP;
  auto mad4 = [](float s, const float4 &d, const float4 &a) {
    return mad(mad(mad(mad(s, d.x, a.x), d.y, a.y), d.z, a.z), d.w, a.w);
  };
  auto ld4 = [](const float *p) { return *reinterpret_cast<const float4 *>(p); };
  {   // 2 x 2 entries of a square layer, the third by waves 0-3, the second by waves 4-7
    const bool third = tid < kTrainThreads / 2;
    const int e = tid & (kTrainThreads / 2 - 1), r = 2 * (e / (kH / 2)), k = 2 * (e % (kH / 2));
    const float *d = third ? t.d3[r] : t.d2[r], *a = third ? t.a2[k] : t.a1[k];
    float s[2][2] = {};
#pragma unroll 4
    for (int q = 0; q < kTrainRec; q += 4) {
      const float4 p[2] = {ld4(d + q), ld4(d + kTrow + q)}, v[2] = {ld4(a + q), ld4(a + kTrow + q)};
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int l = 0; l < 2; ++l) s[m][l] = mad4(s[m][l], p[m], v[l]);
    }
    float *go = g + (third ? oW3 : oW2) + r * kH + k;
#pragma unroll
    for (int m = 0; m < 2; ++m)
#pragma unroll
      for (int l = 0; l < 2; ++l) go[m * kH + l] = s[m][l];
  }
  // first and output layers, biases (delta times 1): one entry of a list per thread
  constexpr int nW1 = kH * kIn, nW4 = kOut * kH, nB = 3 * kH + kOut;
  static_assert(nW1 + nW4 + nB < kTrainThreads, "one entry per thread, the last thread sums the losses");
  if (tid < nW1 + nW4 + nB) {
    const float *d, *a = t.one;
    int p = tid, o;
    if (p < nW1) { d = t.d1[p / kIn]; a = t.x[p % kIn]; o = oW1 + p; }
    else if ((p -= nW1) < nW4) { d = t.g4[p / kH]; a = t.a3[p % kH]; o = oW4 + p; }
    else if ((p -= nW4) < kH) { d = t.d1[p]; o = oB1 + p; }
    else if ((p -= kH) < kH) { d = t.d2[p]; o = oB2 + p; }
    else if ((p -= kH) < kH) { d = t.d3[p]; o = oB3 + p; }
    else { p -= kH; d = t.g4[p]; o = oB4 + p; }
    float s = 0.f;
#pragma unroll 4
    for (int q = 0; q < kTrainRec; q += 4) s = mad4(s, ld4(d + q), ld4(a + q));
    g[o] = s;
  }
  if (tid == kTrainThreads - 1) {
    double l = 0.0;
#pragma unroll 16
    for (int q = 0; q < kTrainRec; ++q) l += t.loss[q];
    part_loss[blockIdx.x] = l;
  }
}

// Adam on the FP32 master weights; writes the BF16 copy used by the sweep.
struct AdamArgs {
  float *w, *mom, *vel;
  uint16_t *wbf16;
  float lr, b1, b2, eps;
  int t;                              // step, from 1; 0: gradient only
};

// Mean gradient and loss from the blocks' partial sums, block after block, then the Adam step in
// the same launch (one thread per parameter; the last thread sums the losses).
__global__ __launch_bounds__(64) void k_train_reduce(const float *part_grad, const double *part_loss, int nblk, int n,
                                                     float *grad, double *loss, AdamArgs ad) {
  const int p = blockIdx.x * 64 + threadIdx.x;
  if (p == kNP) {
    double l = 0.0;
#pragma unroll 8
    for (int b = 0; b < nblk; ++b) l += part_loss[b];
    *loss = l / (double)n;
  }
  if (p >= kNP) return;
  float g = 0.f;
#pragma unroll 16
  for (int b = 0; b < nblk; ++b) g += part_grad[(size_t)b * kNP + p];
  const float gp = g / (float)n;
  grad[p] = gp;
  if (ad.t == 0) return;
  const float m = ad.b1 * ad.mom[p] + (1.f - ad.b1) * gp;
  const float v = ad.b2 * ad.vel[p] + (1.f - ad.b2) * gp * gp;
  ad.mom[p] = m;
  ad.vel[p] = v;
  const float mh = m / (1.f - powf(ad.b1, (float)ad.t));
  const float vh = v / (1.f - powf(ad.b2, (float)ad.t));
  const float nw_ = ad.w[p] - ad.lr * mh / (sqrtf(vh) + ad.eps);
  ad.w[p] = nw_;
  // round to nearest even BF16
  const uint32_t u = __float_as_uint(nw_);
  const uint32_t rb = ((u >> 16) & 1u) + 0x7FFFu;
  ad.wbf16[p] = (uint16_t)((u + rb) >> 16);
}

__global__ void k_to_bf16(const float *w, uint16_t *wbf16) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kNP) return;
  const uint32_t u = __float_as_uint(w[p]);
  const uint32_t rb = ((u >> 16) & 1u) + 0x7FFFu;
  wbf16[p] = (uint16_t)((u + rb) >> 16);
}

// Evaluation: per record the six outputs, kappa_0, kappa_1, log q(s | env) and w_0, from the
// FP32 master network (sweep_net = 0) or from the network the sweep runs (BF16 weights and
// hidden activations on the matrix cores, sweep_net = 1).
constexpr int kEvalBlock = 128;
__global__ __launch_bounds__(kEvalBlock) void k_eval(const float *w, const uint16_t *wbf16, int sweep_net,
                                                     const float *recs, int n, double *out) {
  __shared__ float wl[kNP];
  const int i = blockIdx.x * kEvalBlock + threadIdx.x;
  const int ic = i < n ? i : n - 1;            // whole waves run the matrix-core network
  const float *rec = recs + (size_t)ic * kRec;
  float x[kIn], o[kOut];
  for (int k = 0; k < kIn; ++k) x[k] = rec[k];
  if (sweep_net) {
    for (int k = threadIdx.x; k < kNP; k += kEvalBlock) wl[k] = __uint_as_float((uint32_t)wbf16[k] << 16);
    const NetA na = load_net_a(wbf16);
    __syncthreads();
    net_forward_mfma(wl, na, x, o);
  } else {
    mlp_forward(w, x, o);
  }
  if (i >= n) return;
  const V3 ghat = rec_vec(rec, 6), ax = rec_vec(rec, 9), s = rec_vec(rec, 12);
  const V3 e = tilt_frame(ghat, ax);
  const Comp m0 = make_comp(o[0], o[1], o[2], o[4], rec[5], ghat, e);
  const Comp m1 = make_comp(o[3], o[4], o[5], o[1], rec[5], ghat, e);
  double *q = out + (size_t)i * 10;
  for (int k = 0; k < kOut; ++k) q[k] = o[k];
  q[6] = m0.kappa;
  q[7] = m1.kappa;
  q[8] = log_mix(log_part(m0, s), log_part(m1, s));
  q[9] = exp(m0.logw - kLog1mU);
}

using LearnFn = void (*)(KArgs, const uint16_t *);
using CollectFn = void (*)(KArgs, int, uint32_t, uint32_t, float *);
template <bool CMP, bool HB>
LearnFn lf2(bool hd) { return hd ? k_phase_learned<CMP, HB, true> : k_phase_learned<CMP, HB, false>; }
LearnFn learn_fn(const esp::HostModel &m) {
  if (m.compressed) return m.has_B ? lf2<true, true>(m.has_D) : lf2<true, false>(m.has_D);
  return m.has_B ? lf2<false, true>(m.has_D) : lf2<false, false>(m.has_D);
}
template <bool CMP, bool HB>
CollectFn cf2(bool hd) { return hd ? k_collect<CMP, HB, true> : k_collect<CMP, HB, false>; }
CollectFn collect_fn(const esp::HostModel &m) {
  if (m.compressed) return m.has_B ? cf2<true, true>(m.has_D) : cf2<true, false>(m.has_D);
  return m.has_B ? cf2<false, true>(m.has_D) : cf2<false, false>(m.has_D);
}

int learn_ready(esp_ctx *c, bool need_state) {
  if (!c) return ESP_EINVAL;
  if (hipSetDevice(c->device) != hipSuccess) return fail(c, ESP_EHIP, "hipSetDevice failed");
  if (need_state) {
    if (!c->have_model) return fail(c, ESP_ESTATE, "no model: call esp_set_model first");
    if (c->R <= 0) return fail(c, ESP_ESTATE, "no replicas: call esp_set_replicas first");
    if (c->hm.has_self)
      return fail(c, ESP_EINVAL, "learned proposals need a model without self bonds");
  }
  return ESP_OK;
}

int ensure_weights(esp_ctx *c) {
  if (c->d_lw) return ESP_OK;
  int rc;
  if ((rc = dalloc(c, c->d_lw, kNP)) || (rc = dalloc(c, c->d_lm, kNP)) || (rc = dalloc(c, c->d_lv, kNP)) ||
      (rc = dalloc(c, c->d_lbf, kNP)) || (rc = dalloc(c, c->d_grad, kNP)))
    return rc;
  return ESP_OK;
}

int ensure_records(esp_ctx *c, int need) {
  if (need <= c->rec_cap) return ESP_OK;
  int cap = std::max(need, 2 * c->rec_cap);
  float *nr = nullptr;
  int rc = dalloc(c, nr, (size_t)cap * kRec);
  if (rc) return rc;
  if (c->nrec > 0)
    HIPCHK(c, hipMemcpyAsync(nr, c->d_recs, sizeof(float) * kRec * c->nrec, hipMemcpyDeviceToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  dfree(c->d_recs);
  c->d_recs = nr;
  c->rec_cap = cap;
  return ESP_OK;
}

int train_blocks(int n) { return (n + kTrainRec - 1) / kTrainRec; }

// Gradient scratch for minibatches of up to n records and up to nsteps losses.
int ensure_grad_scratch(esp_ctx *c, int n, int nsteps) {
  const int nblk = train_blocks(n);
  int rc;
  if (nblk > c->pgrad_cap) {
    c->pgrad_cap = 0;
    if ((rc = dalloc(c, c->d_pgrad, (size_t)nblk * kNP)) || (rc = dalloc(c, c->d_ploss, nblk))) return rc;
    c->pgrad_cap = nblk;
  }
  if (nsteps > c->loss_cap) {
    c->loss_cap = 0;
    if ((rc = dalloc(c, c->d_loss, nsteps))) return rc;
    c->loss_cap = nsteps;
  }
  HIPCHK(c, hipFuncSetAttribute((const void *)k_train_block, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)sizeof(TrainLds)));
  return ESP_OK;
}

// Gradient of the mean loss over records (perm ? perm[off + i] : off + i), i < n; loss to d_loss[k];
// with ad.t > 0 also the Adam step.
int enqueue_grad(esp_ctx *c, const int *perm, int off, int n, int k, const AdamArgs &ad) {
  const int nblk = train_blocks(n);
  hipLaunchKernelGGL(k_train_block, dim3(nblk), dim3(kTrainThreads), sizeof(TrainLds), c->stream, (const float *)c->d_lw,
                     (const float *)c->d_recs, n, perm, off, c->d_pgrad, c->d_ploss);
  hipLaunchKernelGGL(k_train_reduce, dim3(kNP / 64 + 1), dim3(64), 0, c->stream, (const float *)c->d_pgrad,
                     (const double *)c->d_ploss, nblk, n, c->d_grad, c->d_loss + k, ad);
  HIPCHK(c, hipGetLastError());
  return ESP_OK;
}

}  // namespace

namespace esp {

// nsweeps sweeps of learned proposals from clock->sweep + off0 (global-memory path).
int learn_enqueue_sweeps(esp_ctx *c, uint64_t seed, int nsweeps, int off0, hipEvent_t *ev, int *nlaunch) {
  int rc = learn_ready(c, true);
  if (rc) return rc;
  if (!c->have_learn) return fail(c, ESP_ESTATE, "no proposal weights: call esp_learn_set_weights first");
  const esp::HostModel &m = c->hm;
  KArgs a = base_args(c);
  a.tps = 1;
  a.mpart = c->d_mpart_l;             // (null before the first call after the weights were set)
  a.key0 = (uint32_t)seed; a.key1 = (uint32_t)(seed >> 32);
  LearnFn fn = learn_fn(m);
  const size_t shm = (m.compressed ? c->ctab_bytes : 0) + kNP * sizeof(float);
  int k = 0;
  for (int s = 0; s < nsweeps; ++s)
    for (int col = 0; col < m.ncol; ++col) {
      a.col = col;
      a.c_begin = m.col_off[col];
      a.c_count = m.col_off[col + 1] - m.col_off[col];
      if (a.c_count == 0) continue;
      a.nblk = (a.c_count + kBlock - 1) / kBlock;
      a.dnblk = espg::make_fastdiv((uint32_t)a.nblk);
      a.xcd_full = espg::xcd_full(c->R, a.nblk);
      a.sweep_off = off0 + s;
      if (ev)
        hipExtLaunchKernelGGL(fn, dim3(a.nblk * c->R), dim3(kBlock), shm, c->stream, ev[2 * k], ev[2 * k + 1], 0,
                              a, (const uint16_t *)c->d_lbf);
      else
        hipLaunchKernelGGL(fn, dim3(a.nblk * c->R), dim3(kBlock), shm, c->stream, a, (const uint16_t *)c->d_lbf);
      ++k;
    }
  HIPCHK(c, hipGetLastError());
  if (nlaunch) *nlaunch = k;
  return ESP_OK;
}

void learn_free(esp_ctx *c) {
  dfree(c->d_lw); dfree(c->d_lm); dfree(c->d_lv); dfree(c->d_lbf); dfree(c->d_recs); dfree(c->d_pgrad);
  dfree(c->d_grad); dfree(c->d_ploss); dfree(c->d_loss); dfree(c->d_perm);
  c->have_learn = false;
  c->nrec = c->rec_cap = c->pgrad_cap = c->loss_cap = c->perm_cap = 0;
}

}  // namespace esp

extern "C" {

int esp_learn_set_weights(esp_ctx *c, const float *w, int nparams) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!w || nparams != kNP) return fail(c, ESP_EINVAL, "esp_learn_set_weights: need ESP_LEARN_NPARAMS weights");
  for (int p = 0; p < kNP; ++p)
    if (!std::isfinite(w[p])) return fail(c, ESP_EINVAL, "esp_learn_set_weights: non-finite weight");
  if ((rc = ensure_weights(c))) return rc;
  HIPCHK(c, hipMemcpyAsync(c->d_lw, w, sizeof(float) * kNP, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipMemsetAsync(c->d_lm, 0, sizeof(float) * kNP, c->stream));
  HIPCHK(c, hipMemsetAsync(c->d_lv, 0, sizeof(float) * kNP, c->stream));
  hipLaunchKernelGGL(k_to_bf16, dim3((kNP + 255) / 256), dim3(256), 0, c->stream, (const float *)c->d_lw, c->d_lbf);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->adam_t = 0;
  c->have_learn = true;
  drop_graph(c);
  return ESP_OK;
}

int esp_learn_get_weights(esp_ctx *c, float *w, int nparams) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!w || nparams != kNP) return fail(c, ESP_EINVAL, "esp_learn_get_weights: need ESP_LEARN_NPARAMS weights");
  if (!c->have_learn) return fail(c, ESP_ESTATE, "no proposal weights");
  HIPCHK(c, hipMemcpyAsync(w, c->d_lw, sizeof(float) * kNP, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return ESP_OK;
}

int esp_learn_collect(esp_ctx *c, int n, uint64_t seed) {
  int rc = learn_ready(c, true);
  if (rc) return rc;
  if (n < 0 || (int64_t)c->nrec + n > (int64_t)1 << 27)
    return fail(c, ESP_EINVAL, "esp_learn_collect: record count out of range (max 2^27)");
  if (n == 0) return ESP_OK;
  if ((rc = ensure_records(c, c->nrec + n))) return rc;
  KArgs a = base_args(c);
  const size_t shm = c->hm.compressed ? c->ctab_bytes : 0;
  hipLaunchKernelGGL(collect_fn(c->hm), dim3((n + kBlock - 1) / kBlock), dim3(kBlock), shm, c->stream, a, n,
                     (uint32_t)seed, (uint32_t)(seed >> 32), c->d_recs + (size_t)kRec * c->nrec);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->nrec += n;
  return ESP_OK;
}

int esp_learn_clear(esp_ctx *c) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  c->nrec = 0;
  return ESP_OK;
}

int esp_learn_num_records(esp_ctx *c, int *n) {
  if (!c || !n) return ESP_EINVAL;
  *n = c->nrec;
  return ESP_OK;
}

int esp_learn_get_records(esp_ctx *c, int first, int n, float *out) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!out || first < 0 || n < 0 || first + n > c->nrec) return fail(c, ESP_EINVAL, "record range");
  if (n == 0) return ESP_OK;
  HIPCHK(c, hipMemcpyAsync(out, c->d_recs + (size_t)kRec * first, sizeof(float) * kRec * n,
                           hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return ESP_OK;
}

int esp_learn_put_records(esp_ctx *c, const float *recs, int n) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if ((!recs && n > 0) || n < 0 || n > (1 << 27)) return fail(c, ESP_EINVAL, "esp_learn_put_records: bad size");
  c->nrec = 0;
  if (n == 0) return ESP_OK;
  if ((rc = ensure_records(c, n))) return rc;
  HIPCHK(c, hipMemcpyAsync(c->d_recs, recs, sizeof(float) * kRec * n, hipMemcpyHostToDevice, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->nrec = n;
  return ESP_OK;
}

int esp_learn_grad(esp_ctx *c, int first, int n, float *grad, double *loss) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!c->have_learn) return fail(c, ESP_ESTATE, "no proposal weights");
  if (!grad || !loss || first < 0 || n <= 0 || first + n > c->nrec) return fail(c, ESP_EINVAL, "record range");
  if ((rc = ensure_grad_scratch(c, n, 1))) return rc;
  if ((rc = enqueue_grad(c, nullptr, first, n, 0, AdamArgs{}))) return rc;
  HIPCHK(c, hipMemcpyAsync(grad, c->d_grad, sizeof(float) * kNP, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(loss, c->d_loss, sizeof(double), hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return ESP_OK;
}

int esp_learn_train(esp_ctx *c, int epochs, int batch, float lr, uint64_t seed, double *epoch_loss) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!c->have_learn) return fail(c, ESP_ESTATE, "no proposal weights");
  if (epochs < 0 || batch < 1 || batch > (1 << 20) || !(lr > 0.0f) || c->nrec < 1)
    return fail(c, ESP_EINVAL, "esp_learn_train: bad epochs / batch / lr, or no records");
  const int n = c->nrec;
  const int nb = (n + batch - 1) / batch;
  if ((rc = ensure_grad_scratch(c, std::min(batch, n), nb))) return rc;
  if (n > c->perm_cap) {
    if ((rc = dalloc(c, c->d_perm, n))) return rc;
    c->perm_cap = n;
  }
  std::vector<int> perm(n);
  std::vector<double> losses(nb);
  uint64_t st = seed ^ 0x9E3779B97F4A7C15ull;
  auto next = [&st]() {  // splitmix64
    uint64_t z = (st += 0x9E3779B97F4A7C15ull);
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
  };
  for (int e = 0; e < epochs; ++e) {
    for (int i = 0; i < n; ++i) perm[i] = i;
    for (int i = n - 1; i > 0; --i) std::swap(perm[i], perm[(int)(next() % (uint64_t)(i + 1))]);
    HIPCHK(c, hipMemcpyAsync(c->d_perm, perm.data(), sizeof(int) * n, hipMemcpyHostToDevice, c->stream));
    for (int b = 0; b < nb; ++b) {
      const int off = b * batch, cnt = std::min(batch, n - off);
      c->adam_t += 1;
      const AdamArgs ad{c->d_lw, c->d_lm, c->d_lv, c->d_lbf, lr, 0.9f, 0.999f, 1e-8f, c->adam_t};
      if ((rc = enqueue_grad(c, c->d_perm, off, cnt, b, ad))) return rc;
    }
    HIPCHK(c, hipGetLastError());
    HIPCHK(c, hipMemcpyAsync(losses.data(), c->d_loss, sizeof(double) * nb, hipMemcpyDeviceToHost, c->stream));
    HIPCHK(c, hipStreamSynchronize(c->stream));  // the host permutation buffer is reused
    if (epoch_loss) {
      double s = 0.0, wsum = 0.0;
      for (int b = 0; b < nb; ++b) {
        const double cnt = std::min(batch, n - b * batch);
        s += losses[b] * cnt;
        wsum += cnt;
      }
      epoch_loss[e] = s / wsum;
    }
  }
  drop_graph(c);
  return ESP_OK;
}

int esp_learn_eval(esp_ctx *c, int first, int n, int sweep_net, double *out) {
  int rc = learn_ready(c, false);
  if (rc) return rc;
  if (!c->have_learn) return fail(c, ESP_ESTATE, "no proposal weights");
  if (!out || first < 0 || n < 0 || first + n > c->nrec) return fail(c, ESP_EINVAL, "record range");
  if (n == 0) return ESP_OK;
  double *d_out = nullptr;
  if ((rc = dalloc(c, d_out, (size_t)n * 10))) return rc;
  hipLaunchKernelGGL(k_eval, dim3((n + kEvalBlock - 1) / kEvalBlock), dim3(kEvalBlock), 0, c->stream,
                     (const float *)c->d_lw, (const uint16_t *)c->d_lbf, sweep_net ? 1 : 0,
                     (const float *)c->d_recs + (size_t)kRec * first, n, d_out);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipMemcpyAsync(out, d_out, sizeof(double) * 10 * n, hipMemcpyDeviceToHost, c->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
  dfree(d_out);
  if (e != hipSuccess) return fail(c, ESP_EHIP, std::string("esp_learn_eval: ") + hipGetErrorString(e));
  return ESP_OK;
}

}  // extern "C"
