// Differentiable relaxation of the transmission step: expected infections per agent and day.
//
// The stochastic step draws, for every infectious source j and susceptible target i sharing an
// edge of layer l, an infection with probability x = beta * beta_l * rel_trans_j * viral_load *
// rel_sus_i (utils.py:88-123). The relaxation replaces the indicator states by probabilities:
//   s_i(t)   probability that i is still susceptible at the start of day t
//   D_i(t)   probability that i is infected on day t            (D_i(0) = seed fraction f)
//   tr_j(t)  expected infectiousness = rel_trans_j * sum_{d>=1} D_j(t-d) w_{bin(j)}(d), where w_b(d)
//            is the mean (viral load x infectious) factor d days after infection for age bin b
//   L_i(t)   = sum over layers l and neighbours j of i of log1p(-min(beta*beta_l*sigma_{bin(i)}*tr_j, XMAX))
//   D_i(t)   = s_i(t) * (1 - exp(L_i(t)))          s_i(t+1) = s_i(t) * exp(L_i(t))
//   E_t      = sum_i (transmission part of D_i(t))   (the expected new infections of day t)
// Parameters theta = (beta, beta_l for each layer, sigma_b for the 10 age bins of rel_sus).
//
// Contacts are undirected, so each layer is a neighbour CSR (both directions of every stored pair,
// self-loops dropped). The forward gathers over in-neighbours; the adjoint gathers over the same
// lists in the source role: every sum is a gather in a fixed order (deterministic, no float
// atomics). Reverse mode, day t from last to first (bars are adjoints, e_t = dJ/dE_t):
//   Dbar_i(t) = e_t + sum_{d>=1} Ibar_i(t+d) w_{bin(i)}(d)
//   Lbar_i(t) = s_i(t) e^{L_i} (sbar_i(t+1) - Dbar_i(t))      sbar_i(t) = Dbar_i (1 - e^{L_i}) + sbar_i(t+1) e^{L_i}
//   with g'(x) = -1/(1-x) below XMAX (0 above):
//   C_{a,l} = sum_{j in N_l(a)} g'(beta beta_l sigma_a tr_j) tr_j             (a as target)
//   Ibar_a(t) = rel_trans_a * sum_l beta beta_l sum_{j in N_l(a)} Lbar_j g'(beta beta_l sigma_j tr_a) sigma_j
//   dJ/dbeta += Lbar_a sigma_a sum_l beta_l C_{a,l};  dJ/dbeta_l += beta Lbar_a sigma_a C_{a,l};
//   dJ/dsigma_{bin(a)} += beta Lbar_a sum_l beta_l C_{a,l}
// With q_i = 1 - e^{L_i} and P_i = e^{L_i} taken over the list as running products (P <- P (1 - x), q <- q + x P,
// in double), no logarithm or exponential is needed, and small probabilities keep their relative precision.
// The forward keeps s at every checkpoint day and the backward re-runs each segment's forward, recording every day's
// escape, s, tr and d log P / d sigma, before walking it backwards; where the caller lets it hold the records of all
// days at once (segment_days), the forward records them and the backward re-runs nothing.
//
// A layer resampled every day enters in expectation (c_l = 2 E_l / N slots per agent, uniform sources,
// self-pairs left out): with x_{l,b} = beta beta_l sigma_b, g(y) = log1p(-min(y, XMAX)) and
// S_{l,b}(t) = sum_j g(x_{l,b} tr_j), its term of L_i is c_l / N (S_{l,bin(i)} - g(x_{l,bin(i)} tr_i)). Its
// adjoint needs, per day, Lambda_b = sum_{bin(i)=b} Lbar_i, G_{l,b} = sum_j g'(x_{l,b} tr_j) tr_j and
// H_{l,b} = sum_{bin(i)=b} Lbar_i g'(x_{l,b} tr_i) tr_i (block partials summed in a fixed order):
//   Ibar_a += rel_trans_a c_l / N sum_b x_{l,b} g'(x_{l,b} tr_a) (Lambda_b - [bin(a) = b] Lbar_a)
//   xbar_{l,b} = c_l / N (Lambda_b G_{l,b} - H_{l,b}), which feeds dJ/dbeta, dJ/dbeta_l and dJ/dsigma_b.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <memory>
#include <vector>

#include "cvk_host.h"
#include "cvk_kernels.h"
#include "cvk_scan.h"

namespace cvk {

constexpr int RELAX_BLOCK = 256;
constexpr int RELAX_BINS = 10;
constexpr double RELAX_XMAX = 0.999999;  // per-edge probabilities are capped below 1 (1 - x stays positive)
constexpr int RELAX_AB = 128;            // agents of a workgroup (64 for small populations)
constexpr int RELAX_UNROLL = 8;          // neighbour-list entries of a lane whose gathers are in flight together
constexpr int64_t RELAX_GROUP_SLOTS = (int64_t)1 << 31;  // most slots of a workgroup: its kernels count them in 32 bits
constexpr int RELAX_LAGS = 64;           // lags of the infectiousness table staged in LDS together
// packed slots: neighbour index, the held layer and the neighbour's age bin
constexpr uint32_t RELAX_IDX = (1u << 25) - 1u;
constexpr int RELAX_LAYER_SHIFT = 25, RELAX_BIN_SHIFT = 28;
static_assert(CVK_MAX_LAYERS <= 8 && RELAX_BINS <= 16, "layer and bin share a slot with the index");

template <class R>
struct RelaxTheta {
  R beta;
  R bl[CVK_MAX_LAYERS];
  R sig[RELAX_BINS];
};

template <class R>
struct RelaxDev {
  int64_t n;
  int32_t n_layers, n_days, kmax;        // kmax: longest lag with w != 0 that is kept (<= n_days)
  int32_t n_blocks;                      // workgroups of AB agents
  // The held layers' neighbour lists, laid out once per handle: workgroup w's slots are [wg_base[w], wg_base[w + 1]),
  // agent after agent (layer after layer within an agent), so a workgroup reads its lists with coalesced loads.
  int32_t n_held;
  int32_t held[CVK_MAX_LAYERS];          // their layer indices
  const int64_t* wg_base;                // [n_blocks + 1]
  const uint32_t* end;                   // [n] offset of the end of an agent's list in its workgroup
  const uint32_t* slots;                 // index | layer << 25 | bin << 28 (n up to 2^25), else the index
  const uint8_t* meta;                   // null, or above 2^25 agents the slot's layer | bin << 4
  const uint8_t* tgt;                    // the slot's agent, within its workgroup
  const uint8_t* bin;    // [n] age bin 0..9
  const float* rt;       // [n] rel_trans
  const R* w;            // [10][kmax + 1]
  R* delta;              // [n_days][n]
  R* s;                  // [n] running susceptible probability
  R* ibar;               // [n_days][n]
  R* sbar;               // [n]
  R* lbar;               // [2][n] of day t at t & 1
  R* ylb;                // [2][n] what the adjoint reads of a neighbour on day t (at t & 1): lbar * sig(bin)
  double* epart;         // [n_days][n_blocks] per-block sums of E_t
  double* gpart;         // [n_held + 10][n_blocks] per-block sums over days: tr_a src_{a,l}, then lbar_a Csig_a by age bin
  R seed_frac;
  // layers resampled every day (in expectation)
  int32_t n_dyn;
  int32_t dyn_layer[CVK_MAX_LAYERS];  // their layer indices
  double dyn_slots[CVK_MAX_LAYERS];   // c_l of dynamic layer k
  double* dyn_part;      // [(1 + 2 n_dyn) * 10][n_blocks] per-workgroup sums
  double* dyn_fsum;      // [n_dyn][10] the next day's S_{l,b} (forward)
  double* dyn_red;       // [n_days][(1 + 2 n_dyn) * 10]: Lambda_b, then G_{l,b}, then H_{l,b}
};

// log(1 - x): the series below 2^-6 (truncated at 1e-19 of the result), which nearly every contact is, else log1p.
__device__ inline double log1m(double x) {
  if (__builtin_fabs(x) < 0x1p-6) {
    double p = 1.0 / 10.0;
    p = __builtin_fma(p, x, 1.0 / 9.0);
    p = __builtin_fma(p, x, 1.0 / 8.0);
    p = __builtin_fma(p, x, 1.0 / 7.0);
    p = __builtin_fma(p, x, 1.0 / 6.0);
    p = __builtin_fma(p, x, 1.0 / 5.0);
    p = __builtin_fma(p, x, 1.0 / 4.0);
    p = __builtin_fma(p, x, 1.0 / 3.0);
    p = __builtin_fma(p, x, 1.0 / 2.0);
    p = __builtin_fma(p, x, 1.0);
    return -x * p;
  }
  return log1p(-x);
}

// 1 / d with d != 0: the hardware's reciprocal and one Newton step (float; the sums it feeds are double), or the
// division (double).
__device__ inline float relax_rcp(float d) {
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}
__device__ inline double relax_rcp(double d) { return 1.0 / d; }
// 1 / d of a normal double to its last bit or two: the hardware's reciprocal and two Newton steps.
__device__ inline double rcp_d(double d) {
  double r = __builtin_amdgcn_rcp(d);
  r = __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
  return __builtin_fma(__builtin_fma(-d, r, 1.0), r, r);
}

// g'(y) of g(y) = log1p(-min(y, XMAX)): 0 from XMAX up
template <class R>
__device__ inline R relax_gp(R y, R xmax) { return y < xmax ? relax_rcp(y - (R)1) : (R)0; }

// q = 1 - e^L and P = e^L in one value of type R: q up to a half (P = 1 - q), else 1 / P.
template <class R>
__device__ inline R escape_code(double q, double P) { return q <= 0.5 ? (R)q : (R)(1.0 / P); }
template <class R>
__device__ inline void escape_decode(R y, double& q, double& P) {
  if (y > (R)1) {
    P = 1.0 / (double)y;
    q = 1.0 - P;
  } else {
    q = (double)y;
    P = 1.0 - q;
  }
}

// expm1(x): the series below 2^-4 (truncated at 1e-17 of the result), else the library's.
__device__ inline double expm1_d(double x) {
  if (__builtin_fabs(x) < 0x1p-4) {
    double p = 1.0 / 3628800.0;
    p = __builtin_fma(p, x, 1.0 / 362880.0);
    p = __builtin_fma(p, x, 1.0 / 40320.0);
    p = __builtin_fma(p, x, 1.0 / 5040.0);
    p = __builtin_fma(p, x, 1.0 / 720.0);
    p = __builtin_fma(p, x, 1.0 / 120.0);
    p = __builtin_fma(p, x, 1.0 / 24.0);
    p = __builtin_fma(p, x, 1.0 / 6.0);
    p = __builtin_fma(p, x, 0.5);
    p = __builtin_fma(p, x, 1.0);
    return x * p;
  }
  return expm1(x);
}

__device__ inline double sum16(double v) {  // over the 16 lanes of a row group
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// A workgroup serves AB agents with 256 threads: RELAX_BLOCK / AB lanes share an agent (its lists, lags and sum rows).
template <int AB>
struct RelaxLanes {
  static constexpr int TPA = RELAX_BLOCK / AB;
  static_assert(TPA * AB == RELAX_BLOCK && TPA <= 16, "lanes per agent");
};

// out(r, the workgroup's sum over its agents of f(r)), r < nr <= NR, f evaluated on one lane per agent and
// row (16 lanes sum a row, fixed order). Block-wide; s_d: NR * AB doubles, free before and after.
template <int NR, int AB, class F, class O>
__device__ inline void rows_sum(const F& f, double* s_d, const O& out, int nr = NR) {
  constexpr int TPA = RelaxLanes<AB>::TPA;
  const int a = threadIdx.x / TPA, part = threadIdx.x % TPA;
  __syncthreads();
#pragma unroll 1
  for (int r0 = 0; r0 < NR; r0 += TPA)
    if (r0 + part < nr) s_d[(r0 + part) * AB + a] = f(r0 + part);
  __syncthreads();
  const int seg = threadIdx.x & 15;
  for (int r0 = 0; r0 < NR; r0 += RELAX_BLOCK / 16) {
    const int r = r0 + (threadIdx.x >> 4);
    double acc = 0.0;
    if (r < nr)
      for (int e = seg; e < AB; e += 16) acc += s_d[r * AB + e];
    acc = sum16(acc);
    if (r < nr && seg == 0) out(r, acc);
  }
  __syncthreads();
}

// The same by age bin: out(r, b, the sum of f(r) over the agents of bin b), r < nr. bin: 255 for no agent.
// s_d: nr * AB doubles.
template <int AB, class F, class O>
__device__ inline void bin_rows_sum(const F& f, int nr, uint32_t bin, double* s_d, uint8_t* s_bin, const O& out) {
  constexpr int TPA = RelaxLanes<AB>::TPA;
  const int a = threadIdx.x / TPA, part = threadIdx.x % TPA;
  __syncthreads();
  if (part == 0) s_bin[a] = (uint8_t)bin;
  for (int r = part; r < nr; r += TPA) s_d[r * AB + a] = f(r);
  __syncthreads();
  const int seg = threadIdx.x & 15, b = threadIdx.x >> 4;
  for (int r = 0; r < nr; ++r) {
    double acc = 0.0;
    for (int e = seg; e < AB; e += 16) acc += s_bin[e] == b ? s_d[r * AB + e] : 0.0;
    acc = sum16(acc);
    if (b < RELAX_BINS && seg == 0) out(r, b, acc);
  }
  __syncthreads();
}

// Lags [d0, d0 + m) of the infectiousness table into LDS.
template <class R>
__device__ inline void lag_table(const RelaxDev<R>& D, int32_t d0, int32_t m, R* s_w) {
  for (int32_t k = threadIdx.x; k < RELAX_BINS * RELAX_LAGS; k += RELAX_BLOCK)
    if (k % RELAX_LAGS < m) s_w[k] = D.w[(int64_t)(k / RELAX_LAGS) * (D.kmax + 1) + d0 + k % RELAX_LAGS];
}

// start + sum_{d=1}^{dmax} rows[(t0 + sgn * d) * n + i] w[bin][d], the lags dealt over the agent's lanes; the d = 1
// value is `first` when have_first. Block-wide (the caller staged the table's first RELAX_LAGS lags, the others follow
// RELAX_LAGS at a time); RELAX_UNROLL rows in flight per lane. Every lane of the agent returns the sum.
template <class R, int AB>
__device__ inline R lag_sum(const RelaxDev<R>& D, const R* rows, int64_t i, bool valid, uint32_t bin, int32_t t0,
                            int sgn, int32_t dmax, bool have_first, R first, R start, R* s_w) {
  constexpr int TPA = RelaxLanes<AB>::TPA;
  const int part = threadIdx.x % TPA;
  R acc = part == 0 ? start : (R)0;
  for (int32_t d0 = 1; d0 <= dmax; d0 += RELAX_LAGS) {
    const int32_t m = std::min(RELAX_LAGS, dmax - d0 + 1);
    if (d0 > 1) {
      __syncthreads();
      lag_table(D, d0, m, s_w);
    }
    __syncthreads();
    if (valid) {
      const R* wb = s_w + bin * RELAX_LAGS;
      for (int32_t k0 = part; k0 < m; k0 += RELAX_UNROLL * TPA) {
        R v[RELAX_UNROLL];
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) {
          const int32_t k = k0 + u * TPA;
          v[u] = (R)0;
          if (k < m) v[u] = d0 + k == 1 && have_first ? first : gmem(rows)[(int64_t)(t0 + sgn * (d0 + k)) * D.n + i];
        }
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u)
          if (k0 + u * TPA < m) acc += v[u] * wb[k0 + u * TPA];
      }
    }
  }
#pragma unroll
  for (int off = 1; off < TPA; off <<= 1) acc += __shfl_xor(acc, off, 64);
  return acc;
}

// Bytes of LDS a workgroup of AB agents stages one value per contact slot in; longer lists go through it in pieces.
constexpr int relax_stage(int ab) { return ab * 128; }
constexpr int RELAX_ROWS_ADJ = CVK_MAX_LAYERS + 2;  // Csig, Lambda and an H per resampled layer

// One day of the forward for AB agents. do_edge: day t's escape probabilities over the contact lists, infections and
// states; do_next: tr of day t + 1 (tr_next), which needs only the agents' own history, and the resampled layers'
// sums over it. rec_y / rec_s / rec_c (may be null): day t's record for the adjoint.
//
// Bound by the gathers of tr: 16.0M slots a day in the 1M workload, of 4 bytes each from a 4 MB table, which alone
// take 80 us from L2 (72 from a 2 MB table, 152 from one of 8 MB). A thread per agent walking its own list read the
// list uncoalesced and ran a float log1p (127 instructions) per slot; here the workgroup gathers all its slots with
// coalesced list reads into LDS, then each agent's lanes multiply its own up from there: with P the product of
// (1 - x) and P' its derivative with respect to sigma, four double FMAs a slot and no logarithm. P' / P is all that
// the adjoint needs of the target role, so it does not gather tr again. Measured, 1M agents, 60 days, an average day:
// 135 us against 202 (138 + 36 + 28, three launches); 30k agents in double, 36 slots each: 16 against 47.
template <class R, int AB>
__global__ __launch_bounds__(RELAX_BLOCK) void relax_day_kernel(RelaxDev<R> D, RelaxTheta<R> th, int32_t t, int do_edge,
                                                                int do_next, const R* tr, R* tr_next, R* rec_y,
                                                                R* rec_s, R* rec_c) {
  constexpr int TPA = RelaxLanes<AB>::TPA;
  constexpr int STAGE = relax_stage(AB);
  static_assert(STAGE >= (RELAX_BINS + 1) * AB * 8, "the row sums share the stage");
  __shared__ __attribute__((aligned(16))) unsigned char s_buf[STAGE];
  __shared__ R s_w[RELAX_BINS * RELAX_LAGS];
  __shared__ R s_rate[CVK_MAX_LAYERS];  // beta beta_l of the held layers
  __shared__ R s_sig[16];
  const int a = threadIdx.x / TPA, part = threadIdx.x % TPA;
  const int64_t i = (int64_t)blockIdx.x * AB + a;
  const bool valid = i < D.n;
  const uint32_t bin = valid ? D.bin[i] : 0u;
  const R rt = valid ? (R)D.rt[i] : (R)0;
  if (threadIdx.x < 16) s_sig[threadIdx.x] = threadIdx.x < RELAX_BINS ? th.sig[threadIdx.x] : (R)0;
  const R s0 = valid && do_edge ? D.s[i] : (R)0;
  const R sig = th.sig[bin];
  const R xmax = (R)RELAX_XMAX;
  R dnew = 0, inf = 0;
  if ((int)threadIdx.x < D.n_held) s_rate[threadIdx.x] = th.beta * th.bl[D.held[threadIdx.x]];
  if (do_next) lag_table(D, 1, std::min(RELAX_LAGS, D.kmax), s_w);
  if (do_edge) {  // uniform
    const uint32_t list0 = valid && a ? gmem(D.end)[i - 1] : 0u, list1 = valid ? gmem(D.end)[i] : 0u;
    __syncthreads();  // s_rate
    constexpr uint32_t CAP = STAGE / sizeof(R);
    R* stage = (R*)s_buf;
    const int64_t g0 = D.wg_base[blockIdx.x];
    const uint32_t total = (uint32_t)(D.wg_base[blockIdx.x + 1] - g0);
    double q = 0.0, P = 1.0, dP = 0.0;  // over this lane's slots; dP: derivative of P with respect to sigma
    for (uint32_t c0 = 0; c0 < total; c0 += CAP) {
      const uint32_t cn = std::min(CAP, total - c0);
      const CVK_GLOBAL uint32_t* src = gmem(D.slots) + g0 + c0;
      for (uint32_t u0 = threadIdx.x; u0 < cn; u0 += RELAX_BLOCK * RELAX_UNROLL) {
        uint32_t j[RELAX_UNROLL], h[RELAX_UNROLL];
        R v[RELAX_UNROLL];
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) {
          const uint32_t e = u0 + u * RELAX_BLOCK;
          j[u] = e < cn ? __builtin_nontemporal_load(src + e) : 0u;
          h[u] = j[u] >> RELAX_LAYER_SHIFT;
          if (D.meta) h[u] = e < cn ? gmem(D.meta)[g0 + c0 + e] : 0u;  // uniform
          else j[u] &= RELAX_IDX;
        }
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) v[u] = u0 + u * RELAX_BLOCK < cn ? gmem(tr)[j[u]] : (R)0;
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) {
          const uint32_t e = u0 + u * RELAX_BLOCK;
          if (e < cn) stage[e] = s_rate[h[u] & 7u] * v[u];
        }
      }
      __syncthreads();
      const uint32_t k1 = list1 > c0 ? std::min(list1 - c0, cn) : 0u;
      for (uint32_t k = (list0 > c0 ? list0 - c0 : 0u) + part; k < k1; k += TPA) {
        const R r = stage[k];
        const R x = sig * r;
        const bool below = x < xmax;
        const double xd = (double)(below ? x : xmax), rd = below ? (double)r : 0.0;
        q = __builtin_fma(xd, P, q);
        dP = __builtin_fma(-xd, dP, dP);
        dP = __builtin_fma(-rd, P, dP);
        P = __builtin_fma(-xd, P, P);
      }
      __syncthreads();
    }
    // d log P: below the normal doubles (rcp_d has no reciprocal there) the agent cannot escape, its lbar is at most
    // 2^-1022 and the sum that c goes into does not hold the product
    double c = P >= 0x1p-1022 ? dP * rcp_d(P) : 0.0;
#pragma unroll
    for (int off = 1; off < TPA; off <<= 1) {
      const int other = (int)lane_id() ^ off;
      const double q2 = shfl_d(q, other), P2 = shfl_d(P, other);
      q = __builtin_fma(P, q2, q);
      P *= P2;
      c += shfl_d(c, other);
    }
    if (valid && D.n_dyn) {  // c_l / N (S_{l,b} - g(x_{l,b} tr_i))
      double L = 0.0;
      const R tr_i = gmem(tr)[i];
      for (int k = 0; k < D.n_dyn; ++k) {
        R x = ((th.beta * th.bl[D.dyn_layer[k]]) * sig) * tr_i;
        x = x < xmax ? x : xmax;
        L += D.dyn_slots[k] / (double)D.n * (D.dyn_fsum[k * RELAX_BINS + bin] - log1m((double)x));
      }
      const double em = expm1_d(L);
      q = __builtin_fma(-em, P, q);
      P = __builtin_fma(em, P, P);
    }
    if (q <= 0.5) P = 1.0 - q;  // one rounding, where the product has one per slot
    if (valid) {
      inf = (R)((double)s0 * q);
      dnew = (t == 0 ? D.seed_frac : (R)0) + inf;
      if (part == 0) {
        D.s[i] = (R)((double)s0 * P);
        gmem(D.delta)[(int64_t)t * D.n + i] = dnew;
        if (rec_y) {
          gmem(rec_y)[i] = escape_code<R>(q, P);
          gmem(rec_s)[i] = s0;
          gmem(rec_c)[i] = (R)c;
        }
      }
    }
  }
  double* const e_out = D.epart + (int64_t)t * D.n_blocks + blockIdx.x;  // E_t, with do_edge
  if (!do_next) {
    rows_sum<1, AB>([&](int) { return (double)inf; }, (double*)s_buf, [&](int, double v) { *e_out = v; });
    return;
  }
  // tr_i(t + 1) = rel_trans_i * sum_{d=1}^{min(kmax, t + 1)} D_i(t + 1 - d) w_{bin(i)}(d)
  const R acc = lag_sum<R, AB>(D, D.delta, i, valid, bin, t + 1, -1, std::min(t + 1, D.kmax), do_edge != 0, dnew, (R)0, s_w);
  const R trn = valid ? rt * acc : (R)0;
  if (valid && part == 0) gmem(tr_next)[i] = trn;
  // S_{l,b} = sum_j g(x_{l,b} tr_j) of the resampled layers, E_t summed along with the first of them
  double* sink = D.dyn_part + blockIdx.x;
  for (int k = 0; k < std::max(D.n_dyn, 1); ++k) {
    const bool dyn = k < D.n_dyn;
    const R rate = dyn ? th.beta * th.bl[D.dyn_layer[k]] : (R)0;
    const bool with_e = k == 0 && do_edge;
    const auto f = [&](int b) {
      if (b == RELAX_BINS) return (double)inf;
      R x = (rate * s_sig[b]) * trn;
      x = x < xmax ? x : xmax;
      return valid ? log1m((double)x) : 0.0;
    };
    const auto o = [&](int b, double v) { *(b == RELAX_BINS ? e_out : sink + (int64_t)(k * RELAX_BINS + b) * D.n_blocks) = v; };
    if (dyn && with_e) rows_sum<RELAX_BINS + 1, AB>(f, (double*)s_buf, o);
    else if (dyn) rows_sum<RELAX_BINS, AB>(f, (double*)s_buf, o);
    else if (with_e) rows_sum<1, AB>([&](int) { return (double)inf; }, (double*)s_buf, [&](int, double v) { *e_out = v; });
  }
}

// One day of the adjoint for AB agents. do_edge: Ibar_a(t) (source role) over the contact lists and day t's parameter
// partials from the recorded C_{a,l}(t); do_agent: Dbar, Lbar, sbar of day t - 1, which need only the agents' own
// history, what the neighbours will read of them (ylb) and the resampled layers' sums.
// ebar, rec_y, rec_s, tr_prev: of day t - 1; tr, rec_c: of day t.
//
// Bound, as the forward, by one 4-byte gather per slot (lbar sig of the neighbour; its age bin travels in the slot
// word, so its sig does too). The 16-byte records (tr, lbar sig, sig) gathered before came from a 16 MB table
// (218 us for the gathers alone). The term of a slot is computed where it is gathered, a slot per lane, and only
// the sums run per agent. Measured as above: 165 us against 290 (217 + 39 + 23 + 6 + 5, five launches), and 19 us
// against 46; and with every day's record held, the forward's days are not run a second time.
template <class R, int AB>
__global__ __launch_bounds__(RELAX_BLOCK) void relax_adjoint_kernel(RelaxDev<R> D, RelaxTheta<R> th, int32_t t,
                                                                    int do_edge, int do_agent, R ebar, const R* tr,
                                                                    const R* tr_prev, const R* rec_y, const R* rec_s,
                                                                    const R* rec_c) {
  constexpr int TPA = RelaxLanes<AB>::TPA;
  constexpr int STAGE = relax_stage(AB);
  static_assert(STAGE >= RELAX_BINS * AB * 8 && STAGE >= RELAX_ROWS_ADJ * AB * 8, "the row sums share the stage");
  __shared__ __attribute__((aligned(16))) unsigned char s_buf[STAGE];
  __shared__ R s_w[RELAX_BINS * RELAX_LAGS];
  __shared__ R s_sig[16], s_tra[AB];
  extern __shared__ __attribute__((aligned(16))) unsigned char s_dyn[];
  R* s_g = (R*)s_dyn;  // [n_held][RELAX_BLOCK] this thread's slots' tr_a src by layer
  __shared__ R s_rate[CVK_MAX_LAYERS];  // beta beta_l of the held layers
  __shared__ uint8_t s_bin[AB];
  const int a = threadIdx.x / TPA, part = threadIdx.x % TPA;
  const int64_t i = (int64_t)blockIdx.x * AB + a;
  const bool valid = i < D.n;
  const uint32_t bin = valid ? D.bin[i] : 0u;
  const R sig = th.sig[bin];
  const R xmax = (R)RELAX_XMAX;
  const R rt = valid ? (R)D.rt[i] : (R)0;
  const R lbar_a = valid && do_edge ? gmem(D.lbar)[(int64_t)(t & 1) * D.n + i] : (R)0;
  const int64_t nb = D.n_blocks;
  const int n_c = do_edge ? 1 : 0;
  // lbar_a Csig_a by age bin, added to the sums over days
  const double c_val = valid && do_edge ? (double)lbar_a * (double)gmem(rec_c)[i] : 0.0;
  const auto c_out = [&](int b, double v) { D.gpart[(int64_t)(D.n_held + b) * nb + blockIdx.x] += v; };
  if (threadIdx.x < 16) s_sig[threadIdx.x] = threadIdx.x < RELAX_BINS ? th.sig[threadIdx.x] : (R)0;
  // the agent phase's inputs, on their way beside the edge phase
  R y_p = 0, s_p = 0, sb_next = 0, trp = 0;
  if (do_agent) {
    lag_table(D, 1, std::min(RELAX_LAGS, D.kmax), s_w);
    if (valid) {
      y_p = gmem(rec_y)[i];
      s_p = gmem(rec_s)[i];
      sb_next = D.sbar[i];
      trp = gmem(tr_prev)[i];
    }
  }
  R ib = 0;
  if (do_edge) {  // uniform
    constexpr uint32_t CAP = STAGE / sizeof(R);
    R* stage = (R*)s_buf;
    const R tr_a = valid ? gmem(tr)[i] : (R)0;
    if ((int)threadIdx.x < D.n_held) s_rate[threadIdx.x] = th.beta * th.bl[D.held[threadIdx.x]];
    if (part == 0) s_tra[a] = tr_a;
    const uint32_t list0 = valid && a ? gmem(D.end)[i - 1] : 0u, list1 = valid ? gmem(D.end)[i] : 0u;
    __syncthreads();
    const CVK_GLOBAL R* ylb = gmem((const R*)D.ylb) + (int64_t)(t & 1) * D.n;
    const int64_t g0 = D.wg_base[blockIdx.x];
    const uint32_t total = (uint32_t)(D.wg_base[blockIdx.x + 1] - g0);
    double ibar = 0.0;
    for (int h = 0; h < D.n_held; ++h) s_g[h * RELAX_BLOCK + threadIdx.x] = (R)0;
    for (uint32_t c0 = 0; c0 < total; c0 += CAP) {
      const uint32_t cn = std::min(CAP, total - c0);
      const CVK_GLOBAL uint32_t* src = gmem(D.slots) + g0 + c0;
      const CVK_GLOBAL uint8_t* tg = gmem(D.tgt) + g0 + c0;
      for (uint32_t u0 = threadIdx.x; u0 < cn; u0 += RELAX_BLOCK * RELAX_UNROLL) {
        uint32_t j[RELAX_UNROLL], aa[RELAX_UNROLL], m[RELAX_UNROLL];
        R y[RELAX_UNROLL];
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) {
          const uint32_t e = u0 + u * RELAX_BLOCK;
          j[u] = e < cn ? __builtin_nontemporal_load(src + e) : 0u;
          aa[u] = e < cn ? __builtin_nontemporal_load(tg + e) : 0u;
          m[u] = ((j[u] >> RELAX_LAYER_SHIFT) & 7u) | ((j[u] >> RELAX_BIN_SHIFT) << 4);
          if (D.meta) m[u] = e < cn ? gmem(D.meta)[g0 + c0 + e] : 0u;  // uniform
          else j[u] &= RELAX_IDX;
        }
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) y[u] = u0 + u * RELAX_BLOCK < cn ? ylb[j[u]] : (R)0;
#pragma unroll
        for (int u = 0; u < RELAX_UNROLL; ++u) {
          const uint32_t e = u0 + u * RELAX_BLOCK;
          if (e < cn) {
            const uint32_t h = m[u] & 7u;
            const R rate = s_rate[h], tra = s_tra[aa[u]];
            const R x = (rate * s_sig[m[u] >> 4]) * tra;  // a -> j
            const R term = x < xmax ? y[u] * relax_rcp(x - (R)1) : (R)0;  // (y: 0 * inf for an infinite sigma)
            stage[e] = rate * term;
            s_g[h * RELAX_BLOCK + threadIdx.x] += tra * term;
          }
        }
      }
      __syncthreads();
      const uint32_t k1 = list1 > c0 ? std::min(list1 - c0, cn) : 0u;
      for (uint32_t k = (list0 > c0 ? list0 - c0 : 0u) + part; k < k1; k += TPA) ibar += (double)stage[k];
      __syncthreads();
    }
    rows_sum<CVK_MAX_LAYERS, AB>(
        [&](int r) {
          double v = 0.0;
          for (int k = 0; k < TPA; ++k) v += (double)s_g[r * RELAX_BLOCK + a * TPA + k];
          return v;
        },
        (double*)s_buf, [&](int r, double v) { D.gpart[(int64_t)r * nb + blockIdx.x] += v; }, D.n_held);
#pragma unroll
    for (int off = 1; off < TPA; off <<= 1) ibar += shfl_d(ibar, (int)lane_id() ^ off);
    const double* red = D.dyn_red + (int64_t)t * RELAX_BINS * (1 + 2 * D.n_dyn);
    for (int k = 0; k < D.n_dyn; ++k) {  // the daily-resampled layers' source role, the bins dealt over the lanes
      const R rate = th.beta * th.bl[D.dyn_layer[k]];
      double acc = 0.0;
      for (int b = part; b < RELAX_BINS; b += TPA) {
        const R x = rate * s_sig[b];
        const double lam = red[b] - (b == (int)bin ? (double)lbar_a : 0.0);
        acc += (double)(x * relax_gp<R>(x * tr_a, xmax)) * lam;
      }
#pragma unroll
      for (int off = 1; off < TPA; off <<= 1) acc += shfl_d(acc, (int)lane_id() ^ off);
      ibar += D.dyn_slots[k] / (double)D.n * acc;
    }
    ib = (R)((double)rt * ibar);
    if (valid && part == 0) gmem(D.ibar)[(int64_t)t * D.n + i] = ib;
  }
  if (!do_agent) {
    bin_rows_sum<AB>([&](int) { return c_val; }, n_c, valid ? bin : 255u, (double*)s_buf, s_bin,
                     [&](int, int b, double v) { c_out(b, v); });
    return;
  }
  const int32_t tp = t - 1;
  // Dbar = e + sum_{d=1}^{min(kmax, T - 1 - tp)} Ibar(tp + d) w(d)
  const R dbar = lag_sum<R, AB>(D, D.ibar, i, valid, bin, tp, 1, std::min(D.kmax, D.n_days - 1 - tp), do_edge != 0, ib,
                                ebar, s_w);
  R lbar = 0;
  if (valid) {
    double q, P;
    escape_decode<R>(y_p, q, P);
    const double sd = (double)s_p, sb = (double)sb_next, db = (double)dbar;
    lbar = (R)((sd * P) * (sb - db));
    if (part == 0) {
      D.sbar[i] = (R)(db * q + sb * P);
      gmem(D.lbar)[(int64_t)(tp & 1) * D.n + i] = lbar;
      gmem(D.ylb)[(int64_t)(tp & 1) * D.n + i] = lbar * sig;
    }
  }
  // then Lambda_b, H_{l,b} = sum_{bin(i) = b} Lbar_i g'(x_{l,b} tr_i) tr_i, and G_{l,b} = sum_j g'(x_{l,b} tr_j) tr_j
  bin_rows_sum<AB>(
      [&](int r) {
        if (r < n_c) return c_val;
        r -= n_c;
        if (r == 0) return (double)lbar;
        const R x = (th.beta * th.bl[D.dyn_layer[r - 1]]) * sig;
        return (double)lbar * (double)(relax_gp<R>(x * trp, xmax) * trp);
      },
      n_c + (D.n_dyn ? 1 + D.n_dyn : 0), valid ? bin : 255u, (double*)s_buf, s_bin,
      [&](int r, int b, double v) {
        if (r < n_c) c_out(b, v);
        else D.dyn_part[(int64_t)((r - n_c) * RELAX_BINS + b) * nb + blockIdx.x] = v;
      });
  for (int k = 0; k < D.n_dyn; ++k) {
    const R rate = th.beta * th.bl[D.dyn_layer[k]];
    rows_sum<RELAX_BINS, AB>(
        [&](int b) {
          const R x = rate * s_sig[b];
          return valid ? (double)(relax_gp<R>(x * trp, xmax) * trp) : 0.0;
        },
        (double*)s_buf,
        [&](int b, double v) { D.dyn_part[(int64_t)(RELAX_BINS * (1 + D.n_dyn + k) + b) * nb + blockIdx.x] = v; });
  }
}

// Sums `rows` columns of per-block partials (row-major [rows][n_blocks]) into out[rows] (fixed order).
__global__ __launch_bounds__(256) void relax_reduce_kernel(const double* part, int64_t n_blocks, int32_t rows,
                                                           double* out) {
  __shared__ double s_w[4];
  for (int32_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const double* p = part + (int64_t)r * n_blocks;
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t b = threadIdx.x;
    for (; b + 768 < n_blocks; b += 1024) {  // four loads in flight
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] += p[b + 256 * u];
    }
    for (; b < n_blocks; b += 256) a[0] += p[b];
    const double acc = wave_sum_d((a[0] + a[1]) + (a[2] + a[3]));
    if (lane_id() == 0) s_w[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) out[r] = (s_w[0] + s_w[1]) + (s_w[2] + s_w[3]);
    __syncthreads();
  }
}

template <class R>
__global__ void relax_fill_kernel(R* p, int64_t n, R v) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) p[i] = v;
}

// ---------------------------------------------------------------------------
// Layout of the held layers' lists (once per handle)
// ---------------------------------------------------------------------------
struct RelaxLists {
  const int64_t* indptr[CVK_MAX_LAYERS];  // of the held layers
  const int32_t* nbr[CVK_MAX_LAYERS];
  int32_t n_held;
  int64_t n;
  int32_t ab;
};
struct RelaxGroupSlots {  // slots of workgroup w
  RelaxLists L;
  __device__ int64_t operator()(int64_t w) const {
    const int64_t i0 = w * L.ab, i1 = std::min<int64_t>(i0 + L.ab, L.n);
    int64_t tot = 0;
    for (int h = 0; h < L.n_held; ++h) tot += L.indptr[h][i1] - L.indptr[h][i0];
    return tot;
  }
};
struct RelaxWriteBase {
  int64_t* base;
  __device__ void operator()(int64_t w, int64_t prefix, int64_t) const { base[w] = prefix; }
};

template <int AB>
__global__ __launch_bounds__(RELAX_BLOCK) void relax_layout_kernel(RelaxLists L, const uint8_t* bin, const int64_t* wg_base,
                                                                   uint32_t* end, uint32_t* slots, uint8_t* meta,
                                                                   uint8_t* tgt) {
  __shared__ int64_t s_ptr[AB + 1];
  __shared__ uint32_t s_len[AB], s_pos[AB];  // an agent's slots in all, and where its next layer goes
  const int64_t i0 = (int64_t)blockIdx.x * AB;
  const int cnt = (int)std::min<int64_t>(AB, L.n - i0);
  const int64_t g0 = wg_base[blockIdx.x];
  const int me = threadIdx.x;
  if (me < cnt) {
    uint32_t len = 0;
    for (int h = 0; h < L.n_held; ++h) len += (uint32_t)(L.indptr[h][i0 + me + 1] - L.indptr[h][i0 + me]);
    s_len[me] = len;
  }
  __syncthreads();
  if (me < cnt) {
    uint32_t pos = 0;
    for (int k = 0; k < me; ++k) pos += s_len[k];
    s_pos[me] = pos;
    end[i0 + me] = pos + s_len[me];
  }
  for (int h = 0; h < L.n_held; ++h) {
    __syncthreads();
    for (int k = me; k <= cnt; k += RELAX_BLOCK) s_ptr[k] = L.indptr[h][i0 + k];
    __syncthreads();
    const int64_t p0 = s_ptr[0], m = s_ptr[cnt] - p0;
    for (int64_t k = me; k < m; k += RELAX_BLOCK) {
      int lo = 0, hi = cnt - 1;  // the last agent whose list starts at or before the slot
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_ptr[mid] <= p0 + k) lo = mid;
        else hi = mid - 1;
      }
      const uint32_t j = (uint32_t)L.nbr[h][p0 + k];
      const int64_t at = g0 + s_pos[lo] + (p0 + k - s_ptr[lo]);
      slots[at] = meta ? j : j | ((uint32_t)h << RELAX_LAYER_SHIFT) | ((uint32_t)bin[j] << RELAX_BIN_SHIFT);
      if (meta) meta[at] = (uint8_t)(h | (bin[j] << 4));
      tgt[at] = (uint8_t)lo;
    }
    __syncthreads();
    if (me < cnt) s_pos[me] += (uint32_t)(s_ptr[me + 1] - s_ptr[me]);
  }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct RelaxBase {
  virtual ~RelaxBase() {}
  virtual int forward(const double* theta, double* e_host, hipStream_t st) = 0;
  virtual int backward(const double* theta, const double* ebar_host, double* grad_host, hipStream_t st) = 0;
  int device = -1;
};

template <class R>
struct Relax : RelaxBase {
  RelaxDev<R> D;
  int32_t ab = RELAX_AB;       // agents per workgroup
  int32_t seg = 0;             // days whose records are held: all of them, or a segment's
  std::vector<R*> ck_s;        // s at days 0, seg, 2 seg, ... (segments only)
  R* rec_y = nullptr;          // [seg][n]
  R* rec_s = nullptr;          // [seg][n]
  R* rec_c = nullptr;          // [seg][n] Csig
  R* rec_tr = nullptr;         // [max(seg, 2)][n]
  R* w = nullptr;
  double* e_dev = nullptr;     // [n_days]
  double* g_dev = nullptr;     // [n_held + 10]
  std::vector<void*> owned;
  bool have_forward = false;
  std::vector<double> theta_fwd;

  ~Relax() override {
    for (void* p : owned)
      if (p) (void)hipFree(p);
  }

  template <class T>
  int alloc(T** p, int64_t count) {
    *p = nullptr;
    if (hipMalloc((void**)p, (size_t)std::max<int64_t>(count, 1) * sizeof(T)) != hipSuccess) {
      *p = nullptr;
      return fail(CVK_E_HIP, "cvk_relax: device allocation failed");
    }
    owned.push_back((void*)*p);
    return CVK_OK;
  }

  RelaxTheta<R> theta_of(const double* th) const {
    RelaxTheta<R> t;
    memset(&t, 0, sizeof(t));
    t.beta = (R)th[0];
    for (int l = 0; l < D.n_layers; ++l) t.bl[l] = (R)th[1 + l];
    for (int b = 0; b < RELAX_BINS; ++b) t.sig[b] = (R)th[1 + D.n_layers + b];
    return t;
  }

  template <class T>
  void fill(T* p, int64_t n, T v, hipStream_t st) {
    hipLaunchKernelGGL(relax_fill_kernel<T>, dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 1024))),
                       dim3(256), 0, st, p, n, v);
  }

  void reduce(const double* part, int32_t rows, double* out, hipStream_t st) {
    if (rows > 0)
      hipLaunchKernelGGL(relax_reduce_kernel, dim3(std::min(rows, 1024)), dim3(256), 0, st, part, (int64_t)D.n_blocks,
                         rows, out);
  }

  void day(const RelaxTheta<R>& th, int32_t t, bool edge, bool next, const R* tr, R* tr_next, R* y, R* s, R* c,
           hipStream_t st) {
    const auto fn = ab == 64 ? relax_day_kernel<R, 64> : relax_day_kernel<R, RELAX_AB>;
    hipLaunchKernelGGL(fn, dim3(D.n_blocks), dim3(RELAX_BLOCK), 0, st, D, th, t, (int)edge, (int)next, tr, tr_next, y, s, c);
    if (next) reduce(D.dyn_part, D.n_dyn * RELAX_BINS, D.dyn_fsum, st);
  }

  void adjoint(const RelaxTheta<R>& th, int32_t t, bool edge, bool agent, R ebar, const R* tr, const R* tr_prev,
               const R* y, const R* s, const R* c, hipStream_t st) {
    const auto fn = ab == 64 ? relax_adjoint_kernel<R, 64> : relax_adjoint_kernel<R, RELAX_AB>;
    hipLaunchKernelGGL(fn, dim3(D.n_blocks), dim3(RELAX_BLOCK), D.n_held * RELAX_BLOCK * sizeof(R), st, D, th, t, (int)edge,
                       (int)agent, ebar, tr, tr_prev,
                       y, s, c);
    if (agent && D.n_dyn) {
      const int32_t rows = RELAX_BINS * (1 + 2 * D.n_dyn);
      reduce(D.dyn_part, rows, D.dyn_red + (int64_t)(t - 1) * rows, st);
    }
  }

  R* row(R* rows, int64_t k) const { return rows + k * D.n; }

  // Runs days [t0, t1) from the current D.s, recording each (rows 0 .. t1 - t0 - 1), tr(t0) computed first.
  void recorded_days(const RelaxTheta<R>& th, int32_t t0, int32_t t1, hipStream_t st) {
    day(th, t0 - 1, false, true, nullptr, rec_tr, nullptr, nullptr, nullptr, st);
    for (int32_t t = t0; t < t1; ++t) {
      const int32_t k = t - t0;
      const bool next = t + 1 < t1;
      day(th, t, true, next, row(rec_tr, k), next ? row(rec_tr, k + 1) : nullptr, row(rec_y, k), row(rec_s, k),
          row(rec_c, k), st);
    }
  }

  int forward(const double* theta, double* e_host, hipStream_t st) override {
    const RelaxTheta<R> th = theta_of(theta);
    have_forward = false;
    fill(D.s, D.n, (R)1 - D.seed_frac, st);
    if (seg == D.n_days) {
      recorded_days(th, 0, D.n_days, st);
    } else {
      day(th, -1, false, true, nullptr, rec_tr, nullptr, nullptr, nullptr, st);
      for (int32_t t = 0; t < D.n_days; ++t) {
        if (t % seg == 0 && hipMemcpyAsync(ck_s[t / seg], D.s, (size_t)D.n * sizeof(R), hipMemcpyDeviceToDevice, st) != hipSuccess)
          return fail(CVK_E_HIP, "cvk_relax: checkpoint copy failed");
        day(th, t, true, t + 1 < D.n_days, row(rec_tr, t & 1), row(rec_tr, (t + 1) & 1), nullptr, nullptr, nullptr, st);
      }
    }
    reduce(D.epart, D.n_days, e_dev, st);
    const int rc = check_launch("cvk_relax forward");
    if (rc) return rc;
    if (hipMemcpyAsync(e_host, e_dev, (size_t)D.n_days * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
        hipStreamSynchronize(st) != hipSuccess)
      return fail(CVK_E_HIP, "cvk_relax: copy of E failed");
    have_forward = true;
    theta_fwd.assign(theta, theta + 1 + D.n_layers + RELAX_BINS);
    return CVK_OK;
  }

  int backward(const double* theta, const double* ebar_host, double* grad_host, hipStream_t st) override {
    const int np = 1 + D.n_layers + RELAX_BINS;
    if (!have_forward || !std::equal(theta_fwd.begin(), theta_fwd.end(), theta))
      return fail(CVK_E_INVALID, "cvk_relax_backward: needs a forward with the same parameters first");
    const RelaxTheta<R> th = theta_of(theta);
    fill(D.sbar, D.n, (R)0, st);
    fill(D.gpart, (int64_t)(D.n_held + RELAX_BINS) * D.n_blocks, 0.0, st);
    const int32_t n_seg = (D.n_days + seg - 1) / seg;
    for (int32_t k = n_seg - 1; k >= 0; --k) {
      const int32_t t0 = k * seg, t1 = std::min(D.n_days, t0 + seg);
      if (n_seg > 1) {  // re-run the segment, recording it
        if (hipMemcpyAsync(D.s, ck_s[k], (size_t)D.n * sizeof(R), hipMemcpyDeviceToDevice, st) != hipSuccess)
          return fail(CVK_E_HIP, "cvk_relax: checkpoint restore failed");
        recorded_days(th, t0, t1, st);
      }
      const int32_t last = t1 - 1 - t0;
      adjoint(th, t1, false, true, (R)ebar_host[t1 - 1], nullptr, row(rec_tr, last), row(rec_y, last), row(rec_s, last),
              nullptr, st);
      for (int32_t t = t1 - 1; t >= t0; --t) {
        const int32_t j = t - t0, jp = std::max(j - 1, 0);
        adjoint(th, t, true, j > 0, j > 0 ? (R)ebar_host[t - 1] : (R)0, row(rec_tr, j), row(rec_tr, jp), row(rec_y, jp),
                row(rec_s, jp), row(rec_c, j), st);
      }
    }
    reduce(D.gpart, D.n_held + RELAX_BINS, g_dev, st);
    const int rc = check_launch("cvk_relax backward");
    if (rc) return rc;
    const int rows = D.n_dyn ? RELAX_BINS * (1 + 2 * D.n_dyn) : 0;
    std::vector<double> A((size_t)D.n_held + RELAX_BINS, 0.0), red((size_t)D.n_days * rows, 0.0);
    if (hipMemcpyAsync(A.data(), g_dev, A.size() * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess ||
        (rows && hipMemcpyAsync(red.data(), D.dyn_red, red.size() * sizeof(double), hipMemcpyDeviceToHost, st) != hipSuccess) ||
        hipStreamSynchronize(st) != hipSuccess)
      return fail(CVK_E_HIP, "cvk_relax: copy of the gradient failed");
    for (int k = 0; k < np; ++k) grad_host[k] = 0.0;
    // Held layers. Over the pairs (target a, source j) of layer l, lbar_a sigma_a g' tr_j sums to the same by target
    // (lbar_a sigma_a C_{a,l}) and by source (tr_j src_{j,l}), so dJ/dbeta and dJ/dbeta_l come from the source sums;
    // dJ/dsigma_b from lbar_a Csig_a, Csig_a = d L_a / d sigma_a = sum_l beta beta_l C_{a,l}.
    for (int h = 0; h < D.n_held; ++h) {
      grad_host[0] += (double)th.bl[D.held[h]] * A[h];
      grad_host[1 + D.held[h]] += (double)th.beta * A[h];
    }
    for (int b = 0; b < RELAX_BINS; ++b) grad_host[1 + D.n_layers + b] += A[(size_t)D.n_held + b];
    // resampled layers: xbar_{l,b} = c_l / N (Lambda_b G_{l,b} - H_{l,b}) summed over days
    for (int k = 0; k < D.n_dyn; ++k)
      for (int b = 0; b < RELAX_BINS; ++b) {
        double xbar = 0.0;
        for (int32_t t = D.n_days - 1; t >= 0; --t) {
          const double* r = red.data() + (size_t)t * rows;
          xbar += D.dyn_slots[k] / (double)D.n * (r[b] * r[RELAX_BINS * (1 + D.n_dyn + k) + b] - r[RELAX_BINS * (1 + k) + b]);
        }
        const int l = D.dyn_layer[k];
        grad_host[0] += xbar * (double)th.bl[l] * (double)th.sig[b];
        grad_host[1 + l] += xbar * (double)th.beta * (double)th.sig[b];
        grad_host[1 + D.n_layers + b] += xbar * (double)th.beta * (double)th.bl[l];
      }
    return CVK_OK;
  }

  int layout(const cvk_relax_desc* d) {
    RelaxLists L;
    memset(&L, 0, sizeof(L));
    L.n = D.n;
    L.ab = ab;
    L.n_held = D.n_held;
    if (hipDeviceSynchronize() != hipSuccess)  // the lists may come from work on any stream
      return fail(CVK_E_HIP, "cvk_relax_create: device error");
    int64_t total = 0;
    for (int h = 0; h < D.n_held; ++h) {
      L.indptr[h] = d->indptr[D.held[h]];
      L.nbr[h] = d->nbr[D.held[h]];
      int64_t ends[2];
      if (hipMemcpy(&ends[0], L.indptr[h], sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess ||
          hipMemcpy(&ends[1], L.indptr[h] + D.n, sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess)
        return fail(CVK_E_HIP, "cvk_relax_create: cannot read the neighbour lists");
      total += std::max<int64_t>(0, ends[1] - ends[0]);
    }
    int64_t *base = nullptr, *tiles = nullptr;
    uint32_t *end = nullptr, *slots = nullptr;
    uint8_t *tgt = nullptr, *meta = nullptr;
    int rc = alloc(&base, (int64_t)D.n_blocks + 1);
    rc = rc ? rc : alloc(&tiles, scan_tiles(D.n_blocks) + 1);
    rc = rc ? rc : scan(RelaxGroupSlots{L}, RelaxWriteBase{base}, (int64_t)D.n_blocks, tiles, base + D.n_blocks,
                        (hipStream_t)nullptr);
    if (rc) return rc;
    if (total > RELAX_GROUP_SLOTS) {
      std::vector<int64_t> first((size_t)D.n_blocks + 1);
      if (hipMemcpy(first.data(), base, first.size() * sizeof(int64_t), hipMemcpyDeviceToHost) != hipSuccess)
        return fail(CVK_E_HIP, "cvk_relax_create: cannot read the workgroups' offsets");
      for (int32_t w = 0; w < D.n_blocks; ++w)
        if (first[w + 1] - first[w] > RELAX_GROUP_SLOTS)
          return failf(CVK_E_CAPACITY, "cvk_relax_create: agents %lld to %lld have more than 2^31 contact slots",
                       (long long)w * ab, std::min((long long)D.n, (long long)(w + 1) * ab) - 1);
    }
    rc = alloc(&end, D.n);
    rc = rc ? rc : alloc(&slots, total);
    rc = rc ? rc : alloc(&tgt, total);
    if (D.n > (int64_t)RELAX_IDX + 1) rc = rc ? rc : alloc(&meta, total);
    if (rc) return rc;
    D.wg_base = base;
    D.end = end;
    D.slots = slots;
    D.meta = meta;
    D.tgt = tgt;
    const auto fn = ab == 64 ? relax_layout_kernel<64> : relax_layout_kernel<RELAX_AB>;
    hipLaunchKernelGGL(fn, dim3(D.n_blocks), dim3(RELAX_BLOCK), 0, nullptr, L, D.bin, base, end, slots, meta, tgt);
    rc = check_launch("cvk_relax_create");
    if (!rc && hipDeviceSynchronize() != hipSuccess) rc = fail(CVK_E_HIP, "cvk_relax_create: layout failed");
    return rc;
  }
};

template <class R>
static int relax_create(const cvk_relax_desc* d, RelaxBase** out) {
  std::unique_ptr<Relax<R>> r(new Relax<R>());
  RelaxDev<R>& D = r->D;
  memset(&D, 0, sizeof(D));
  D.n = d->n_agents;
  D.n_layers = d->n_layers;
  D.n_days = d->n_days;
  D.kmax = std::min(d->kernel_len - 1, d->n_days);
  D.bin = d->age_bin;
  D.rt = d->rel_trans;
  D.seed_frac = (R)d->seed_frac;
  for (int l = 0; l < d->n_layers; ++l) {
    if (d->dyn_slots[l] > 0.0) {
      D.dyn_slots[D.n_dyn] = (double)(R)d->dyn_slots[l];
      D.dyn_layer[D.n_dyn++] = l;
    } else {
      D.held[D.n_held++] = l;
    }
  }
  int n_cu = 1;
  if (hipGetDevice(&r->device) != hipSuccess) return fail(CVK_E_HIP, "cvk_relax_create: no device");
  if (hipDeviceGetAttribute(&n_cu, hipDeviceAttributeMultiprocessorCount, r->device) != hipSuccess || n_cu < 1) n_cu = 1;
  // half as wide workgroups (four lanes an agent) while there are too few of them to fill the chip: at 30k agents 19 us
  // a day against 21; at 1M agents they take 27.6 ms a gradient against 21.6
  r->ab = D.n < (int64_t)128 * 4 * n_cu ? 64 : RELAX_AB;
  D.n_blocks = (int32_t)((D.n + r->ab - 1) / r->ab);
  int rc = r->layout(d);
  rc = rc ? rc : r->alloc(&r->w, (int64_t)RELAX_BINS * (D.kmax + 1));
  rc = rc ? rc : r->alloc(&D.delta, (int64_t)D.n_days * D.n);
  rc = rc ? rc : r->alloc(&D.s, D.n);
  rc = rc ? rc : r->alloc(&D.ibar, (int64_t)D.n_days * D.n);
  rc = rc ? rc : r->alloc(&D.sbar, D.n);
  rc = rc ? rc : r->alloc(&D.lbar, 2 * D.n);
  rc = rc ? rc : r->alloc(&D.ylb, 2 * D.n);
  rc = rc ? rc : r->alloc(&D.epart, (int64_t)D.n_days * D.n_blocks);
  rc = rc ? rc : r->alloc(&D.gpart, (int64_t)(D.n_held + RELAX_BINS) * D.n_blocks);
  rc = rc ? rc : r->alloc(&D.dyn_part, (int64_t)RELAX_BINS * (1 + 2 * D.n_dyn) * D.n_blocks);
  rc = rc ? rc : r->alloc(&D.dyn_fsum, (int64_t)RELAX_BINS * D.n_dyn);
  rc = rc ? rc : r->alloc(&D.dyn_red, (int64_t)D.n_days * RELAX_BINS * (1 + 2 * D.n_dyn));
  rc = rc ? rc : r->alloc(&r->e_dev, D.n_days);
  rc = rc ? rc : r->alloc(&r->g_dev, (int64_t)D.n_held + RELAX_BINS);
  if (rc) return rc;
  // Records of every day (y, s, tr and Csig, beside the 2 values of the histories) save the backward the second forward
  // (1M agents x 60 days: 19.0 ms a gradient and 1.56 GB in all, 26.9 ms and 0.79 GB with 10 days of them). They are
  // held at once where the caller asks for it, up to an eighth of the card (so that what a program holds does not
  // depend on its neighbours) and half of what is free (so that it fails no sooner than with segments).
  r->seg = std::min(d->checkpoint_every, d->n_days);
  if (d->segment_days == CVK_RELAX_ALL_DAYS) {
    size_t free_b = 0, total_b = 0;
    if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) free_b = total_b = 0;
    if (4 * D.n * (int64_t)sizeof(R) * D.n_days <= (int64_t)std::min(total_b / 8, free_b / 2)) r->seg = d->n_days;
  } else if (d->segment_days > 0 && d->segment_days <= d->n_days) {
    r->seg = d->segment_days;
  }
  rc = rc ? rc : r->alloc(&r->rec_y, (int64_t)r->seg * D.n);
  rc = rc ? rc : r->alloc(&r->rec_s, (int64_t)r->seg * D.n);
  rc = rc ? rc : r->alloc(&r->rec_c, (int64_t)r->seg * D.n);
  rc = rc ? rc : r->alloc(&r->rec_tr, (int64_t)std::max(r->seg, 2) * D.n);
  const int32_t n_seg = (D.n_days + r->seg - 1) / r->seg;
  for (int32_t k = 0; k < n_seg && n_seg > 1 && !rc; ++k) {
    R* p = nullptr;
    rc = r->alloc(&p, D.n);
    r->ck_s.push_back(p);
  }
  if (rc) return rc;
  // infectiousness table w[b][d], d = 0..kmax, converted to R
  std::vector<R> wh((size_t)RELAX_BINS * (D.kmax + 1));
  for (int b = 0; b < RELAX_BINS; ++b)
    for (int dd = 0; dd <= D.kmax; ++dd) wh[(size_t)b * (D.kmax + 1) + dd] = (R)d->w_host[(size_t)b * d->kernel_len + dd];
  if (hipMemcpy(r->w, wh.data(), wh.size() * sizeof(R), hipMemcpyHostToDevice) != hipSuccess)
    return fail(CVK_E_HIP, "cvk_relax_create: upload failed");
  D.w = r->w;
  *out = r.release();
  return CVK_OK;
}

}  // namespace cvk

using namespace cvk;

extern "C" int cvk_relax_create(const cvk_relax_desc* d, void** handle_out) {
  if (!handle_out) return fail(CVK_E_INVALID, "cvk_relax_create: null handle");
  *handle_out = nullptr;
  if (!d || d->n_agents <= 0 || d->n_agents >= (1ll << 31) || d->n_layers < 0 || d->n_layers > CVK_MAX_LAYERS ||
      d->n_days < 1 || d->kernel_len < 2 || d->checkpoint_every < 1 || !d->w_host || !d->age_bin || !d->rel_trans ||
      d->seed_frac < 0 || d->seed_frac > 1 || (d->precision != 32 && d->precision != 64))
    return fail(CVK_E_INVALID, "cvk_relax_create: invalid descriptor");
  for (int l = 0; l < d->n_layers; ++l) {
    if (!(d->dyn_slots[l] >= 0.0)) return fail(CVK_E_INVALID, "cvk_relax_create: dyn_slots must be >= 0");
    if (d->dyn_slots[l] == 0.0 && (!d->indptr[l] || !d->nbr[l]))
      return fail(CVK_E_INVALID, "cvk_relax_create: null neighbour list");
  }
  RelaxBase* r = nullptr;
  const int rc = d->precision == 64 ? relax_create<double>(d, &r) : relax_create<float>(d, &r);
  if (rc) return rc;
  *handle_out = (void*)r;
  return CVK_OK;
}

extern "C" int cvk_relax_destroy(void* handle) {
  if (!handle) return fail(CVK_E_INVALID, "cvk_relax_destroy: null handle");
  delete (RelaxBase*)handle;
  return CVK_OK;
}

extern "C" int cvk_relax_forward(void* handle, const double* theta_host, double* expected_host, void* stream) {
  if (!handle || !theta_host || !expected_host) return fail(CVK_E_INVALID, "cvk_relax_forward: null argument");
  return ((RelaxBase*)handle)->forward(theta_host, expected_host, (hipStream_t)stream);
}

extern "C" int cvk_relax_backward(void* handle, const double* theta_host, const double* grad_expected_host,
                                  double* grad_theta_host, void* stream) {
  if (!handle || !theta_host || !grad_expected_host || !grad_theta_host)
    return fail(CVK_E_INVALID, "cvk_relax_backward: null argument");
  return ((RelaxBase*)handle)->backward(theta_host, grad_expected_host, grad_theta_host, (hipStream_t)stream);
}
