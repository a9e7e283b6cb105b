// 1:1 mirrors of the reference's three numba kernels (covasim/utils.py:39-128),
// used as the parity boundary: same inputs, same float32 operation order, same
// output order. The production day loop (cvk_day.hip) fuses these steps.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>

#include "cvk_device.h"
#include "cvk_host.h"

namespace cvk {

// utils.py:39-79
__global__ void viral_load_kernel(int32_t t, const float* __restrict__ time_start,
                                  const float* __restrict__ time_recovered, const float* __restrict__ time_dead,
                                  int64_t n, float frac_time, float load_ratio, float high_cap,
                                  float* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float dead = time_dead[i];
  const float start = time_start[i];
  const float stop = isnan(dead) ? time_recovered[i] : dead;        // :61-63
  const float total = stop - start;                                   // :66
  const float trans_day = frac_time * total;                          // :67
  const float trans_point = trans_day > high_cap ? high_cap / total : frac_time;  // :68-73
  const bool early = ((float)t - start) / total < trans_point;        // :77
  const float one = 1.0f;
  const float num = load_ratio * (early ? 1.0f : 0.0f) + one * (early ? 0.0f : 1.0f);
  out[i] = num / (one + frac_time * (load_ratio - one));              // :78
}

// utils.py:82-90
__global__ void trans_sus_kernel(const float* __restrict__ rel_trans, const float* __restrict__ rel_sus,
                                 const uint8_t* __restrict__ inf, const uint8_t* __restrict__ sus, float beta_layer,
                                 const float* __restrict__ viral_load, const uint8_t* __restrict__ symp,
                                 const uint8_t* __restrict__ iso, const uint8_t* __restrict__ quar,
                                 float asymp_factor, float iso_factor, float quar_factor,
                                 const float* __restrict__ immunity_factors, int64_t n, float* __restrict__ rt_out,
                                 float* __restrict__ rs_out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float fsymp = symp[i] ? 1.0f : 0.0f;
  const float fiso = iso[i] ? 1.0f : 0.0f;
  const float fquar = quar[i] ? 1.0f : 0.0f;
  const float f_asymp = fsymp + (1.0f - fsymp) * asymp_factor;  // :85 (bool + bool*f32)
  const float f_iso = (1.0f - fiso) + fiso * iso_factor;          // :86
  const float f_quar = (1.0f - fquar) + fquar * quar_factor;      // :87
  float rt = rel_trans[i] * (inf[i] ? 1.0f : 0.0f);               // :88, strictly left to right
  rt = rt * f_quar;
  rt = rt * f_asymp;
  rt = rt * f_iso;
  rt = rt * beta_layer;
  rt = rt * viral_load[i];
  float rs = rel_sus[i] * (sus[i] ? 1.0f : 0.0f);                 // :89
  rs = rs * f_quar;
  rs = rs * (1.0f - immunity_factors[i]);
  rt_out[i] = rt;
  rs_out[i] = rs;
}

// ---------------------------------------------------------------------------
// compute_infections (utils.py:93-128): the transmitting pairs, direction by direction, edges ascending.
//
// Three launches. infections_bits: one bit per agent, rel_trans != 0. infections_scan: every wave takes a run of
// 512-edge chunks; an edge is a candidate if the source of either of its directions has its bit set, and a chunk's
// candidates, compacted in LDS, gather their factors and draw their uniform 64 at a time; one hit bit per
// (direction, edge) and the waves' counts are kept. infections_write: each wave, from the sum of the counts before
// its own, writes out its set bits. Reading the two endpoint columns once is what bounds the scan (80 MB and 20M
// bit lookups at 10M edges, the bitmap in LDS up to ~1.1M agents); before, both a counting and a writing pass
// gathered rel_trans at both ends of every edge and drew a Philox block per slot with a nonzero source, with one
// workgroup scanning the counts between them: 129 + 149 + 21 us at 1M agents and 10M edges, 5 % of them
// infectious, against 4 + 50 + 12 us. (The next chunk's columns loaded ahead of the candidates: 55 us.)
// cvk_infections_noalloc, whose scratch is fixed, keeps the waves' counts and a flag for each chunk: its writing pass
// finds the hits of the flagged chunks anew (213 us at the sizes above with 4050 pairs; 181 with a hit bit for
// every slot, which took 16 MiB of every process on every GPU; 302 without the flags).
// ---------------------------------------------------------------------------
struct InfArgs {
  float beta;
  const int32_t* p1;
  const int32_t* p2;
  const float* layer_betas;
  int64_t n_edges;
  const float* rel_trans;
  const float* rel_sus;
  const double* uniforms;
  uint64_t seed;
  int32_t t, variant, layer;
  int32_t dirs;        // 1 (legacy) or 2
  int64_t n_agents;
  // scratch
  uint64_t* bits;      // one bit per agent, 16-byte aligned and padded (null: rel_trans itself is gathered)
  int32_t lds_words;   // 32-bit words of it staged in LDS, or 0: read from memory
  int64_t chunks;
  uint32_t* hits;      // [2][chunks][16] hit bits (null: not kept, the writing pass finds them anew)
  uint8_t* flags;      // with hits null: [n_flags] whether chunk c has any; chunks from n_flags on are always searched
  int64_t n_flags;
  uint32_t* cnt;       // [2][waves] hits of each wave
  uint64_t* out;       // [2] the total, and nonzero if an endpoint is outside [0, n_agents)
};

constexpr int INF_BLOCK = 1024;
constexpr int INF_WAVES = INF_BLOCK / 64;
constexpr int INF_CHUNK = 512;                 // edges: 8 per lane
constexpr int INF_K = INF_CHUNK / 64;
constexpr int INF_CHUNK_WORDS = INF_CHUNK / 32;
constexpr int INF_WAVE_WORDS = INF_CHUNK / 2 + 2 * INF_CHUNK_WORDS;  // LDS: 16-bit queue of a chunk, its hit words
constexpr int INF_MAX_GRID = 256;
constexpr int64_t INF_CNT_WORDS = 2ll * INF_MAX_GRID * INF_WAVES;
constexpr int INF_LDS = 0, INF_L2 = 1, INF_DIRECT = 2;

__device__ inline uint32_t inf_lane() { return threadIdx.x & 63u; }
__device__ inline uint32_t inf_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}
__device__ inline void inf_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ inline uint32_t inf_wave_sum(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__global__ __launch_bounds__(256) void infections_bits_kernel(InfArgs a) {
  if (blockIdx.x == 0 && threadIdx.x < 2) a.out[threadIdx.x] = 0;
  if (!a.bits) return;
  const int64_t n_words = ((a.n_agents + 127) / 128) * 2;  // padded to 16 bytes
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n_words * 64; i += (int64_t)gridDim.x * 256) {
    const uint64_t m = __ballot(i < a.n_agents && !(a.rel_trans[i] == 0.0f));  // :116
    if (inf_lane() == 0) a.bits[i >> 6] = m;
  }
}

// This wave's chunks.
__device__ inline void inf_range(const InfArgs& a, int64_t& c0, int64_t& c1) {
  const int64_t w = (int64_t)blockIdx.x * INF_WAVES + (threadIdx.x >> 6), W = (int64_t)gridDim.x * INF_WAVES;
  c0 = a.chunks * w / W;
  c1 = a.chunks * (w + 1) / W;
}

// Hit bits of chunk c into s_hit (16 words a direction; wave-wide, the words and the queue are this wave's): whether
// this lane met an endpoint outside the population.
template <int MODE>
__device__ inline uint32_t inf_chunk_hits(const InfArgs& a, int64_t c, const uint32_t* map, uint16_t* queue, uint32_t* s_hit) {
  const uint32_t lane = inf_lane();
  // no index is above 2^31 - 1 (and a negative one is, taken as unsigned)
  const uint32_t n = a.n_agents < ((int64_t)1 << 31) ? (uint32_t)a.n_agents : 1u << 31, nm1 = n ? n - 1u : 0u;
  uint32_t bad = 0;
  const int64_t e0 = c * INF_CHUNK;
  uint32_t x[INF_K], y[INF_K];
#pragma unroll
  for (int k = 0; k < INF_K; ++k) {
    const int64_t e = e0 + k * 64 + lane;
    x[k] = e < a.n_edges ? (uint32_t)a.p1[e] : 0u;
    y[k] = e < a.n_edges ? (uint32_t)a.p2[e] : 0u;
  }
  uint32_t f1 = 0, f2 = 0;  // bit k: the direction's source can transmit
#pragma unroll
  for (int k = 0; k < INF_K; ++k) {
    const bool in = e0 + k * 64 + lane < a.n_edges;
    const bool ok = in && x[k] < n && y[k] < n;
    bad |= in && !ok ? 1u : 0u;
    const uint32_t xs = x[k] < nm1 ? x[k] : nm1, ys = y[k] < nm1 ? y[k] : nm1;
    bool s1 = false, s2 = false;
    if (ok) {
      if (MODE == INF_DIRECT) {
        s1 = !(a.rel_trans[xs] == 0.0f);
        s2 = !(a.rel_trans[ys] == 0.0f);
      } else {
        const uint32_t* words = MODE == INF_LDS ? map : (const uint32_t*)a.bits;
        s1 = (words[xs >> 5] >> (xs & 31u)) & 1u;
        s2 = (words[ys >> 5] >> (ys & 31u)) & 1u;
      }
    }
    f1 |= (uint32_t)s1 << k;
    f2 |= (uint32_t)(s2 && a.dirs == 2) << k;
  }
  uint32_t n_q = 0;
  inf_wave_sync();  // the previous chunk's words have been read
#pragma unroll
  for (int k = 0; k < INF_K; ++k) {
    const bool cand = ((f1 | f2) >> k) & 1u;
    const uint64_t m = __ballot(cand);
    if (cand) queue[n_q + inf_below(m)] = (uint16_t)((k * 64 + lane) | (((f1 >> k) & 1u) << 9) | (((f2 >> k) & 1u) << 10));
    n_q += (uint32_t)__popcll(m);
  }
  if (lane < 2 * INF_CHUNK_WORDS) s_hit[lane] = 0;
  inf_wave_sync();
  for (uint32_t r = 0; r < n_q; r += 64) {  // wave-uniform
    if (r + lane < n_q) {
      const uint32_t q = queue[r + lane], j = q & (INF_CHUNK - 1);
      const int64_t e = e0 + j;
      const int32_t xe = a.p1[e], ye = a.p2[e];
      const float bl = a.beta * a.layer_betas[e];
      float p[2] = {0.0f, 0.0f};
      if (q & (1u << 9)) p[0] = (bl * a.rel_trans[xe]) * a.rel_sus[ye];   // :117
      if (q & (1u << 10)) p[1] = (bl * a.rel_trans[ye]) * a.rel_sus[xe];
      if (p[0] != 0.0f || p[1] != 0.0f) {                                 // :118
        double u[2];
        if (a.uniforms) {
          u[0] = a.uniforms[e];
          u[1] = p[1] != 0.0f ? a.uniforms[a.n_edges + e] : 1.0;
        } else {
          const uint64_t ue = (uint64_t)e;
          const u32x4 w = philox_seeded(a.seed, (uint32_t)ue, (uint32_t)a.t,
                                        STREAM_TX | ((uint32_t)a.variant << 8) | (uint32_t)a.layer, (uint32_t)(ue >> 32));
          u[0] = u01(w.x, w.y);
          u[1] = u01(w.z, w.w);
        }
#pragma unroll
        for (int d = 0; d < 2; ++d)
          if (p[d] != 0.0f && u[d] < (double)p[d])                        // :123
            atomicOr(&s_hit[d * INF_CHUNK_WORDS + (j >> 5)], 1u << (j & 31u));
      }
    }
  }
  inf_wave_sync();
  return bad;
}

// This wave's part of the dynamic LDS after lds_words words of bitmap: the queue (edge of the chunk | dir 0 << 9 |
// dir 1 << 10) and the hit words.
__device__ inline void inf_wave_area(uint32_t* s_inf, int32_t lds_words, uint16_t** queue, uint32_t** s_hit) {
  uint32_t* area = s_inf + lds_words + (threadIdx.x >> 6) * INF_WAVE_WORDS;
  *queue = (uint16_t*)area;
  *s_hit = area + INF_CHUNK / 2;
}

template <int MODE>
__global__ __launch_bounds__(INF_BLOCK) void infections_scan_kernel(InfArgs a) {
  extern __shared__ __attribute__((aligned(16))) uint32_t s_inf[];
  if (MODE == INF_LDS) {
    const uint4* src = (const uint4*)a.bits;
    for (int j = threadIdx.x; j < (a.lds_words >> 2); j += INF_BLOCK) ((uint4*)s_inf)[j] = src[j];
    __syncthreads();
  }
  uint16_t* queue;
  uint32_t* s_hit;
  inf_wave_area(s_inf, MODE == INF_LDS ? a.lds_words : 0, &queue, &s_hit);
  const uint32_t lane = inf_lane();
  int64_t c0, c1;
  inf_range(a, c0, c1);
  uint32_t mine = 0, bad = 0;
  for (int64_t c = c0; c < c1; ++c) {  // wave-uniform
    bad |= inf_chunk_hits<MODE>(a, c, s_inf, queue, s_hit);
    const uint32_t h = lane < (uint32_t)(a.dirs * INF_CHUNK_WORDS) ? s_hit[lane] : 0u;
    mine += (uint32_t)__popc(h);
    if (!a.hits) {  // uniform
      const bool any = __ballot(h != 0) != 0;
      if (lane == 0 && c < a.n_flags) a.flags[c] = any ? 1 : 0;
    } else if (lane < (uint32_t)(a.dirs * INF_CHUNK_WORDS)) {
      a.hits[((int64_t)(lane / INF_CHUNK_WORDS) * a.chunks + c) * INF_CHUNK_WORDS + lane % INF_CHUNK_WORDS] = h;
    }
  }
  const uint32_t n0 = inf_wave_sum(lane < INF_CHUNK_WORDS ? mine : 0u), n1 = inf_wave_sum(lane < INF_CHUNK_WORDS ? 0u : mine);
  const int64_t w = (int64_t)blockIdx.x * INF_WAVES + (threadIdx.x >> 6);
  if (lane == 0) {
    a.cnt[w] = n0;
    a.cnt[(int64_t)gridDim.x * INF_WAVES + w] = n1;
  }
  if (__ballot(bad != 0) && lane == 0) a.out[1] = 1;
}

struct InfOut {
  int64_t capacity;
  int32_t *src, *tgt;
  float* prob;  // may be null
};

// Position of this wave's first pair of each direction, from the scan's counts (same grid); block 0 keeps the total.
// False, for the whole grid, where the call is refused: the outputs then stay as they were. Block-wide.
__device__ inline bool inf_positions(const InfArgs& a, const InfOut& o, uint64_t (&pos)[2]) {
  __shared__ unsigned long long s_sum[INF_WAVES][4];
  const uint32_t lane = inf_lane(), wave = threadIdx.x >> 6;
  const int W = (int)gridDim.x * INF_WAVES, first = (int)blockIdx.x * INF_WAVES;
  // hits in all and before this workgroup, by direction
  unsigned long long v[4] = {0, 0, 0, 0};
  for (int j = threadIdx.x; j < W; j += INF_BLOCK) {
    const uint32_t n0 = a.cnt[j], n1 = a.cnt[W + j];
    v[0] += n0;
    v[1] += n1;
    v[2] += j < first ? n0 : 0u;
    v[3] += j < first ? n1 : 0u;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[q] += __shfl_xor(v[q], off, 64);
    if (lane == 0) s_sum[wave][q] = v[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    v[q] = 0;
    for (int k = 0; k < INF_WAVES; ++k) v[q] += s_sum[k][q];
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) a.out[0] = v[0] + v[1];
  if ((int64_t)(v[0] + v[1]) > o.capacity || a.out[1]) return false;
  pos[0] = v[2];
  pos[1] = v[0] + v[3];
  for (int d = 0; d < a.dirs; ++d)
    for (uint32_t k = 0; k < wave; ++k) pos[d] += a.cnt[d * W + first + (int)k];
  return true;
}

// Writes the pairs of hit word h (edges e0 .. e0 + 31 in direction d) from position at on.
__device__ inline void inf_write_word(const InfArgs& a, const InfOut& o, uint32_t h, int64_t e0, int d, int64_t at) {
  while (h) {
    const int64_t e = e0 + (__ffs(h) - 1);
    h &= h - 1;
    const int32_t x = a.p1[e], y = a.p2[e];
    const int32_t src = d ? y : x, tgt = d ? x : y;
    if (at < o.capacity) {
      o.src[at] = src;
      o.tgt[at] = tgt;
      if (o.prob) o.prob[at] = ((a.beta * a.layer_betas[e]) * a.rel_trans[src]) * a.rel_sus[tgt];
    }
    ++at;
  }
}

// Same grid as the scan.
__global__ __launch_bounds__(INF_BLOCK) void infections_write_kernel(InfArgs a, InfOut o) {
  const uint32_t lane = inf_lane();
  uint64_t start[2];
  if (!inf_positions(a, o, start)) return;
  int64_t c0, c1;
  inf_range(a, c0, c1);
  for (int d = 0; d < a.dirs; ++d) {
    uint64_t pos = start[d];
    const uint32_t* hits = a.hits + (int64_t)d * a.chunks * INF_CHUNK_WORDS;
    for (int64_t w0 = c0 * INF_CHUNK_WORDS; w0 < c1 * INF_CHUNK_WORDS; w0 += 64) {  // wave-uniform
      const uint32_t h = w0 + lane < c1 * INF_CHUNK_WORDS ? hits[w0 + lane] : 0u;
      const uint32_t cnt = (uint32_t)__popc(h);
      uint32_t incl = cnt;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o2 = __shfl_up(incl, off, 64);
        if ((int)lane >= off) incl += o2;
      }
      inf_write_word(a, o, h, (w0 + lane) * 32, d, (int64_t)(pos + incl - cnt));
      pos += __shfl(incl, 63, 64);
    }
  }
}

// The same where the scan's hit bits were not kept (same grid): a flagged chunk's are found again, then written out.
__global__ __launch_bounds__(INF_BLOCK) void infections_rescan_kernel(InfArgs a, InfOut o) {
  extern __shared__ __attribute__((aligned(16))) uint32_t s_inf[];
  uint16_t* queue;
  uint32_t* s_hit;
  inf_wave_area(s_inf, 0, &queue, &s_hit);
  const uint32_t lane = inf_lane();
  uint64_t pos[2];
  if (!inf_positions(a, o, pos)) return;
  int64_t c0, c1;
  inf_range(a, c0, c1);
  const int d = lane / INF_CHUNK_WORDS;  // lanes 0 .. 15 hold direction 0's words, 16 .. 31 direction 1's
  static_assert(INF_CHUNK_WORDS == 16, "a direction's words are a group of 16 lanes");
  for (int64_t c = c0; c < c1; ++c) {  // wave-uniform
    if (c < a.n_flags && !a.flags[c]) continue;
    (void)inf_chunk_hits<INF_DIRECT>(a, c, s_inf, queue, s_hit);
    const uint32_t h = d < a.dirs ? s_hit[lane] : 0u;
    const uint32_t cnt = (uint32_t)__popc(h);
    uint32_t incl = cnt;
#pragma unroll
    for (int off = 1; off < INF_CHUNK_WORDS; off <<= 1) {
      const uint32_t o2 = __shfl_up(incl, off, INF_CHUNK_WORDS);
      if ((int)(lane % INF_CHUNK_WORDS) >= off) incl += o2;
    }
    inf_write_word(a, o, h, c * INF_CHUNK + (int64_t)(lane % INF_CHUNK_WORDS) * 32, d, (int64_t)((d ? pos[1] : pos[0]) + incl - cnt));
    pos[0] += __shfl(incl, INF_CHUNK_WORDS - 1, 64);
    pos[1] += __shfl(incl, 2 * INF_CHUNK_WORDS - 1, 64);
  }
}

static int64_t inf_chunks(int64_t n_edges) { return (n_edges + INF_CHUNK - 1) / INF_CHUNK; }
static int64_t inf_bits_bytes(int64_t n_agents) { return ((n_agents + 127) / 128) * 16; }
static int64_t inf_hits_bytes(int64_t n_edges) { return 2 * inf_chunks(n_edges) * INF_CHUNK_WORDS * 4; }

// Where the scan finds the bitmap (see infections_scan_kernel) and its dynamic LDS. The limits are the device's.
static int inf_lds_budget(int64_t* budget, int* n_cu) {
  static thread_local int configured = -1;
  static thread_local int64_t value = 0;
  static thread_local int cus = 1;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return fail(CVK_E_HIP, "cvk_infections: no current device");
  if (configured != dev) {
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipFuncSetAttribute((const void*)infections_scan_kernel<INF_LDS>, hipFuncAttributeMaxDynamicSharedMemorySize, lds) !=
            hipSuccess)
      return fail(CVK_E_HIP, "cvk_infections: cannot query the device");
    value = lds;
    configured = dev;
  }
  *budget = value;
  *n_cu = cus;
  return CVK_OK;
}

}  // namespace cvk

using namespace cvk;

extern "C" int cvk_viral_load(int32_t t, const float* time_start, const float* time_recovered,
                              const float* time_dead, int64_t n, float frac_time, float load_ratio, float high_cap,
                              float* out, void* stream) {
  if (n < 0 || (n > 0 && (!time_start || !time_recovered || !time_dead || !out)))
    return fail(CVK_E_INVALID, "cvk_viral_load: null pointer or negative n");
  if (n == 0) return CVK_OK;
  const int block = 256;
  const int64_t grid = (n + block - 1) / block;
  hipLaunchKernelGGL(viral_load_kernel, dim3((unsigned)grid), dim3(block), 0, (hipStream_t)stream, t, time_start,
                     time_recovered, time_dead, n, frac_time, load_ratio, high_cap, out);
  return check_launch("cvk_viral_load");
}

extern "C" int cvk_trans_sus(const float* rel_trans, const float* rel_sus, const uint8_t* inf, const uint8_t* sus,
                             float beta_layer, const float* viral_load, const uint8_t* symp, const uint8_t* iso,
                             const uint8_t* quar, float asymp_factor, float iso_factor, float quar_factor,
                             const float* immunity_factors, int64_t n, float* rel_trans_out, float* rel_sus_out,
                             void* stream) {
  if (n < 0 || (n > 0 && (!rel_trans || !rel_sus || !inf || !sus || !viral_load || !symp || !iso || !quar ||
                          !immunity_factors || !rel_trans_out || !rel_sus_out)))
    return fail(CVK_E_INVALID, "cvk_trans_sus: null pointer or negative n");
  if (n == 0) return CVK_OK;
  const int block = 256;
  const int64_t grid = (n + block - 1) / block;
  hipLaunchKernelGGL(trans_sus_kernel, dim3((unsigned)grid), dim3(block), 0, (hipStream_t)stream, rel_trans, rel_sus,
                     inf, sus, beta_layer, viral_load, symp, iso, quar, asymp_factor, iso_factor, quar_factor,
                     immunity_factors, n, rel_trans_out, rel_sus_out);
  return check_launch("cvk_trans_sus");
}

// Arguments of cvk_infections / cvk_infections_noalloc, validated; fills a. Returns CVK_OK, an
// error, or 1 when there is nothing to do (no edges).
static int infections_args(InfArgs& a, float beta, const int32_t* p1, const int32_t* p2, const float* layer_betas,
                           int64_t n_edges, const float* rel_trans, const float* rel_sus, int64_t n_agents,
                           const double* uniforms, uint64_t seed, int32_t t, int32_t variant, int32_t layer,
                           int32_t legacy, const int32_t* src_out, const int32_t* tgt_out, int64_t capacity,
                           int64_t* count_host, const char* name) {
  if (!count_host) return failf(CVK_E_INVALID, "%s: count_host is null", name);
  *count_host = 0;
  if (n_edges < 0 || n_agents < 0 || capacity < 0) return failf(CVK_E_INVALID, "%s: negative size", name);
  if (n_edges == 0) return 1;
  if (!p1 || !p2 || !layer_betas || !rel_trans || !rel_sus || (capacity > 0 && (!src_out || !tgt_out)))
    return failf(CVK_E_INVALID, "%s: null pointer", name);
  if (n_edges >= (1ll << 31)) return failf(CVK_E_INVALID, "%s: more than 2^31-1 edges", name);
  a.beta = beta;
  a.p1 = p1;
  a.p2 = p2;
  a.layer_betas = layer_betas;
  a.n_edges = n_edges;
  a.rel_trans = rel_trans;
  a.rel_sus = rel_sus;
  a.uniforms = uniforms;
  a.seed = seed;
  a.t = t;
  a.variant = variant;
  a.layer = layer;
  a.dirs = legacy ? 1 : 2;
  a.n_agents = n_agents;
  a.chunks = inf_chunks(n_edges);
  return CVK_OK;
}

// Runs the three launches; a's scratch pointers are set (a.bits and a.hits may both be null: rel_trans itself is
// gathered, and the hits are found twice). Reads the total back; *outside (if given) receives whether an endpoint lies
// outside [0, n_agents), an error otherwise.
static int infections_run(InfArgs a, int32_t* src_out, int32_t* tgt_out, float* prob_out, int64_t capacity,
                          int64_t* count_host, int32_t* outside, hipStream_t st, const char* name) {
  int64_t budget = 0;
  int n_cu = 1;
  int rc = inf_lds_budget(&budget, &n_cu);
  if (rc) return rc;
  const int64_t queues = (int64_t)INF_WAVES * INF_WAVE_WORDS * 4, bits = inf_bits_bytes(a.n_agents);
  const bool in_lds = a.bits && bits + queues <= budget;
  a.lds_words = in_lds ? (int32_t)(bits / 4) : 0;
  const int64_t bit_blocks = a.bits ? std::min<int64_t>((a.n_agents + 255) / 256, 2048) : 1;
  hipLaunchKernelGGL(infections_bits_kernel, dim3((unsigned)std::max<int64_t>(bit_blocks, 1)), dim3(256), 0, st, a);
  // a workgroup per CU (the bitmap takes most of its LDS), a chunk a wave at least
  const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(std::min(n_cu, INF_MAX_GRID), a.chunks));
  const auto scan = !a.bits ? infections_scan_kernel<INF_DIRECT> : in_lds ? infections_scan_kernel<INF_LDS> : infections_scan_kernel<INF_L2>;
  hipLaunchKernelGGL(scan, dim3(grid), dim3(INF_BLOCK), (size_t)((in_lds ? bits : 0) + queues), st, a);
  const InfOut o = {capacity, src_out, tgt_out, prob_out};
  if (a.hits) hipLaunchKernelGGL(infections_write_kernel, dim3(grid), dim3(INF_BLOCK), 0, st, a, o);
  else hipLaunchKernelGGL(infections_rescan_kernel, dim3(grid), dim3(INF_BLOCK), (size_t)queues, st, a, o);
  rc = check_launch(name);
  if (rc) return rc;
  uint64_t out[2] = {0, 0};
  if (hipMemcpyAsync(out, a.out, sizeof(out), hipMemcpyDeviceToHost, st) != hipSuccess ||
      hipStreamSynchronize(st) != hipSuccess)
    return failf(CVK_E_HIP, "%s: count readback failed", name);
  if (outside) *outside = out[1] ? 1 : 0;
  if (out[1]) return outside ? CVK_OK : failf(CVK_E_INVALID, "%s: contact indices outside [0, n_agents)", name);
  *count_host = (int64_t)out[0];
  if ((int64_t)out[0] > capacity) return failf(CVK_E_CAPACITY, "%s: output capacity too small", name);
  return CVK_OK;
}

// Scratch of one call, in a block of cvk_infections_work_bytes bytes (16-byte aligned).
static void infections_scratch(InfArgs& a, char* base) {
  a.out = (uint64_t*)base;
  a.cnt = (uint32_t*)(base + 16);
  a.bits = (uint64_t*)(base + 16 + INF_CNT_WORDS * 4);
  a.hits = (uint32_t*)(base + 16 + INF_CNT_WORDS * 4 + inf_bits_bytes(a.n_agents));
}

extern "C" int64_t cvk_infections_work_bytes(int64_t n_edges, int64_t n_agents) {
  if (n_edges < 0 || n_agents < 0) return 0;
  return 16 + INF_CNT_WORDS * 4 + inf_bits_bytes(n_agents) + inf_hits_bytes(n_edges);
}

extern "C" int cvk_infections_work(float beta, const int32_t* p1, const int32_t* p2, const float* layer_betas,
                                   int64_t n_edges, const float* rel_trans, const float* rel_sus, int64_t n_agents,
                                   const double* uniforms, uint64_t seed, int32_t t, int32_t variant, int32_t layer,
                                   int32_t legacy, int32_t* src_out, int32_t* tgt_out, float* prob_out,
                                   int64_t capacity, int64_t* count_host, int32_t* outside_host, void* work,
                                   int64_t work_bytes, void* stream) {
  InfArgs a = {};
  if (outside_host) *outside_host = 0;
  const int rc = infections_args(a, beta, p1, p2, layer_betas, n_edges, rel_trans, rel_sus, n_agents, uniforms, seed, t,
                                 variant, layer, legacy, src_out, tgt_out, capacity, count_host, "cvk_infections_work");
  if (rc != CVK_OK) return rc == 1 ? CVK_OK : rc;
  if (!work || ((uintptr_t)work & 15)) return fail(CVK_E_ALIGN, "cvk_infections_work: workspace must be 16-byte aligned");
  if (work_bytes < cvk_infections_work_bytes(n_edges, n_agents))
    return fail(CVK_E_CAPACITY, "cvk_infections_work: workspace too small");
  infections_scratch(a, (char*)work);
  return infections_run(a, src_out, tgt_out, prob_out, capacity, count_host, outside_host, (hipStream_t)stream,
                        "cvk_infections_work");
}

extern "C" int cvk_infections(float beta, const int32_t* p1, const int32_t* p2, const float* layer_betas,
                              int64_t n_edges, const float* rel_trans, const float* rel_sus, int64_t n_agents,
                              const double* uniforms, uint64_t seed, int32_t t, int32_t variant, int32_t layer,
                              int32_t legacy, int32_t* src_out, int32_t* tgt_out, float* prob_out, int64_t capacity,
                              int64_t* count_host, void* stream) {
  InfArgs a = {};
  int rc = infections_args(a, beta, p1, p2, layer_betas, n_edges, rel_trans, rel_sus, n_agents, uniforms, seed, t,
                           variant, layer, legacy, src_out, tgt_out, capacity, count_host, "cvk_infections");
  if (rc != CVK_OK) return rc == 1 ? CVK_OK : rc;
  char* work = nullptr;
  if (hipMalloc((void**)&work, (size_t)cvk_infections_work_bytes(n_edges, n_agents)) != hipSuccess)
    return fail(CVK_E_HIP, "cvk_infections: hipMalloc failed");
  infections_scratch(a, work);
  rc = infections_run(a, src_out, tgt_out, prob_out, capacity, count_host, nullptr, (hipStream_t)stream, "cvk_infections");
  (void)hipFree(work);
  return rc;
}

// ---- the same computation without allocation ----
// Scratch of cvk_infections_noalloc: the total, the waves' counts and, in the rest of 256 KiB, the chunks' flags (all
// but the last 32784 chunks of the largest legacy call). There is no room for a bit per agent of any population or per
// slot, so its scan gathers rel_trans itself and its writing pass finds the hits anew: nothing that one call leaves
// here is an index to another. Every GPU the library runs on holds its own copy until the process ends. In host code
// `scratch` only names the symbol; its device address comes from hipGetSymbolAddress, once per device, and only that
// address is passed to kernels.
constexpr int64_t SCRATCH_WORDS = 65536;  // the size the header gives
static __device__ __align__(256) uint32_t scratch[SCRATCH_WORDS];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
uint32_t* g_scratch_ptr[kMaxDevices] = {};
}  // namespace

// The current device's address of `scratch` (resolved on the first call on that device).
static int scratch_for_current_device(uint32_t** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices)
    return fail(CVK_E_HIP, "cvk_infections_noalloc: no current device");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return failf(CVK_E_HIP, "cvk_infections_noalloc: hipGetSymbolAddress failed (%s)", hipGetErrorString(e));
    g_scratch_ptr[dev] = (uint32_t*)p;
  }
  *out = g_scratch_ptr[dev];
  return CVK_OK;
}

extern "C" int cvk_infections_noalloc(float beta, const int32_t* p1, const int32_t* p2, const float* layer_betas,
                                      int64_t n_edges, const float* rel_trans, const float* rel_sus,
                                      int64_t n_agents, const double* uniforms, uint64_t seed, int32_t t,
                                      int32_t variant, int32_t layer, int32_t legacy, int32_t* src_out,
                                      int32_t* tgt_out, float* prob_out, int64_t capacity, int64_t* count_host,
                                      void* stream) {
  InfArgs a = {};
  int rc = infections_args(a, beta, p1, p2, layer_betas, n_edges, rel_trans, rel_sus, n_agents, uniforms, seed, t,
                           variant, layer, legacy, src_out, tgt_out, capacity, count_host, "cvk_infections_noalloc");
  if (rc != CVK_OK) return rc == 1 ? CVK_OK : rc;
  const int64_t n_slots = a.dirs * n_edges;
  if (n_slots > CVK_INFECTIONS_NOALLOC_MAX_SLOTS)
    return failf(CVK_E_CAPACITY, "cvk_infections_noalloc: %lld edge slots exceed the fixed scratch's limit of %lld "
                "(use cvk_infections)",
                (long long)n_slots, (long long)CVK_INFECTIONS_NOALLOC_MAX_SLOTS);
  uint32_t* base = nullptr;
  rc = scratch_for_current_device(&base);
  if (rc != CVK_OK) return rc;
  a.out = (uint64_t*)base;
  a.cnt = base + 4;
  a.flags = (uint8_t*)(base + 4 + INF_CNT_WORDS);
  a.n_flags = (SCRATCH_WORDS - 4 - INF_CNT_WORDS) * 4;
  return infections_run(a, src_out, tgt_out, prob_out, capacity, count_host, nullptr, (hipStream_t)stream,
                        "cvk_infections_noalloc");
}
