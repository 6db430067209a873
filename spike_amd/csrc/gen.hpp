// gen.hpp -- connectivity generated on the device: the Brunel fixed in-degree rule (below)
// and the fixed out-degree rule of large networks (further down).
//
// Fixed in-degree (Brunel 2000; the rule of Examples/UtilityFunctions.hpp:51-82, sources
// drawn with replacement): every neuron i receives ce synapses from the excitatory
// population [0, ne) and ci from the inhibitory population [ne, ne+ni).  Slot j of neuron
// i draws u = draw j of (i, stream 3) (output j mod 4 of Philox(seed, ctr = (j/4, i, 3))) and
// takes
//   pre = floor(u * ne / 2^32)            for j <  ce
//   pre = ne + floor(u * ni / 2^32)       for j >= ce
// The local targets are counting-sorted on the device by key (presynaptic unit, partition of
// the postsynaptic neuron), without a host copy: k_gen_count counts each tile's sources (a tile
// is a run of neurons of one partition), k_gen_rows scans a source's counts over the tiles --
// at the partitions' first tiles that is the persistent kernel's segment table, relative to the
// row --, k_gen_rowbase scans the rows and k_gen_seg adds the row starts, and k_gen_scatter
// draws again and writes every target at its tile's cursor.  Entries of one key land in any
// order; deliveries are exact fixed-point sums, so that order does not change any result.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"   // enc16
#include "philox.hpp"

namespace spk {

constexpr uint32_t kStreamConnect = 3;

struct BrunelGenArgs {
  uint64_t seed;
  int N, ne, ni, ce, ci, P;
  int tq, ts;               // tiles per partition, neurons per tile
  unsigned int* cnt;        // [P * tq][N] synapses of each source in a tile, then their row offsets
  unsigned int* rowbase;    // [N] synapses per row, then row starts
  uint32_t* seg;            // [N][P + 1]
  uint16_t* syn16;          // local targets
};

// First neuron of partition q (spk_prepare's split).
__host__ __device__ __forceinline__ int part_start(int N, int P, int q) { return (int)((int64_t)N * q / P); }

// The draws of a tile: f(local target, source) for every synapse.  One work item per (neuron,
// Philox block) uses all four outputs of its call.
template <typename F>
__device__ __forceinline__ void brunel_tile(const BrunelGenArgs& a, int tile, F f) {
  const int q = tile / a.tq;
  const int lo = part_start(a.N, a.P, q), hi = part_start(a.N, a.P, q + 1);
  const int i0 = lo + (tile - q * a.tq) * a.ts, i1 = min(hi, i0 + a.ts);
  const int C = a.ce + a.ci, nb = (C + 3) / 4;
  const int items = max(0, i1 - i0) * nb;
  for (int k = threadIdx.x; k < items; k += blockDim.x) {
    const int di = k / nb, b = k - di * nb;
    const u32x4 r = draw_block(a.seed, b, (uint32_t)(i0 + di), kStreamConnect);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int j = 4 * b + c;
      if (j >= C) break;
      const uint32_t u = pick(r, c);
      const int pre = j < a.ce ? (int)(((uint64_t)u * (uint64_t)a.ne) >> 32)
                               : a.ne + (int)(((uint64_t)u * (uint64_t)a.ni) >> 32);
      f(i0 + di - lo, pre);
    }
  }
}

constexpr int kGenBlock = 512;
// Sources up to which a tile's counters and cursors live in LDS (4 bytes each); networks with
// more count and scatter through global atomics, one tile per partition.
constexpr int kGenLdsSources = 32768;

// Workgroup per tile.  Bound by the scattered 2-byte stores of k_gen_scatter (130 of the 185 us
// of 10^4 neurons x 1000 synapses in 33 partitions; its draws and LDS atomics alone are
// k_gen_count's 20).  Networks of the sweep's sizes take 88 us on average; two kernels with a
// global atomic per synapse and 8-byte records took 402, and a copy of the counts to the host,
// a scan there and two copies back on top.
template <bool LDS>
__global__ __launch_bounds__(kGenBlock) void k_gen_count(BrunelGenArgs a) {
  extern __shared__ unsigned int sgen[];
  unsigned int* out = a.cnt + (size_t)blockIdx.x * a.N;
  unsigned int* c = LDS ? sgen : out;
  for (int u = threadIdx.x; u < a.N; u += blockDim.x) c[u] = 0u;
  if (!LDS) __threadfence();   // the zeros reach memory before the atomics
  __syncthreads();
  brunel_tile(a, blockIdx.x, [&](int, int pre) { atomicAdd(c + pre, 1u); });
  if (LDS) {
    __syncthreads();
    for (int u = threadIdx.x; u < a.N; u += blockDim.x) out[u] = sgen[u];
  }
}

// A workgroup scans kRowsWidth rows, each by kRowsParts threads over a share of the tiles (one
// thread per row waits for one load after another: 49 us for 512 tiles of 10^4 rows against 20).
constexpr int kRowsWidth = 64, kRowsParts = 8;
static __global__ __launch_bounds__(kRowsWidth * kRowsParts) void k_gen_rows(BrunelGenArgs a) {
  __shared__ unsigned int part[kRowsParts][kRowsWidth];
  const int r = (int)threadIdx.x % kRowsWidth, s = (int)threadIdx.x / kRowsWidth;
  const int u = blockIdx.x * kRowsWidth + r;
  const bool on = u < a.N;
  const int T = a.P * a.tq;
  const int t0 = (int)((int64_t)T * s / kRowsParts), t1 = (int)((int64_t)T * (s + 1) / kRowsParts);
  constexpr int kU = 8;   // counts read ahead
  unsigned int sum = 0;
  for (int t = t0; t < t1; t += kU) {
    unsigned int c[kU];
#pragma unroll
    for (int x = 0; x < kU; ++x) c[x] = on && t + x < t1 ? a.cnt[(size_t)(t + x) * a.N + u] : 0u;
#pragma unroll
    for (int x = 0; x < kU; ++x) sum += c[x];
  }
  part[s][r] = sum;
  __syncthreads();
  if (!on) return;
  unsigned int run = 0;
  for (int k = 0; k < s; ++k) run += part[k][r];
  uint32_t* seg = a.seg + (size_t)u * (a.P + 1);
  for (int t = t0; t < t1; t += kU) {
    unsigned int c[kU];
#pragma unroll
    for (int x = 0; x < kU; ++x) c[x] = t + x < t1 ? a.cnt[(size_t)(t + x) * a.N + u] : 0u;
#pragma unroll
    for (int x = 0; x < kU; ++x) {
      if (t + x < t1) {
        if ((t + x) % a.tq == 0) seg[(t + x) / a.tq] = run;
        a.cnt[(size_t)(t + x) * a.N + u] = run;
        run += c[x];
      }
    }
  }
  if (s == kRowsParts - 1) {
    seg[a.P] = run;
    a.rowbase[u] = run;
  }
}

// Exclusive scan of the row sizes (one workgroup; a run of rows per thread).
static __global__ __launch_bounds__(1024) void k_gen_rowbase(BrunelGenArgs a) {
  __shared__ unsigned int sh[1024 / kWave];
  const int per = (a.N + 1023) / 1024;
  const int u0 = min(a.N, (int)threadIdx.x * per), u1 = min(a.N, u0 + per);
  unsigned int sum = 0;
  for (int u = u0; u < u1; ++u) sum += a.rowbase[u];
  const int lane = (int)__lane_id(), w = (int)threadIdx.x / kWave;
  unsigned int incl = sum;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const unsigned int y = __shfl_up(incl, off);
    if (lane >= off) incl += y;
  }
  if (lane == kWave - 1) sh[w] = incl;
  __syncthreads();
  unsigned int run = incl - sum;
  for (int k = 0; k < w; ++k) run += sh[k];
  for (int u = u0; u < u1; ++u) {
    const unsigned int c = a.rowbase[u];
    a.rowbase[u] = run;
    run += c;
  }
}

static __global__ __launch_bounds__(256) void k_gen_seg(BrunelGenArgs a) {
  const int64_t n = (int64_t)a.N * (a.P + 1);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    a.seg[k] += a.rowbase[k / (a.P + 1)];
}

template <bool LDS>
__global__ __launch_bounds__(kGenBlock) void k_gen_scatter(BrunelGenArgs a) {
  extern __shared__ unsigned int sgen[];
  unsigned int* off = a.cnt + (size_t)blockIdx.x * a.N;
  if (LDS) {
    for (int u = threadIdx.x; u < a.N; u += blockDim.x) sgen[u] = off[u] + a.rowbase[u];
    __syncthreads();
  }
  brunel_tile(a, blockIdx.x, [&](int target, int pre) {
    const unsigned int pos = LDS ? atomicAdd(sgen + pre, 1u) : a.rowbase[pre] + atomicAdd(off + pre, 1u);
    a.syn16[pos] = (uint16_t)target;
  });
}

// Constants of a generated network's neurons and partitions and its cleared buffers, written
// where they are used (one launch instead of a copy or fill per array).
struct BrunelInitArgs {
  int N, P, ext_k;
  float v0, vreset, thr, c, rp;
  float *d_v0, *d_vreset, *d_thr, *d_c, *d_rp, *d_decay, *d_erev;
  int *nlo, *ilo;
  uint32_t* ext_cdf;
  unsigned long long* xlist;
  int64_t xwords;
  unsigned long long* stats;
  int* err;
  uint32_t cdf[kMaxExtTable];
};

static __global__ __launch_bounds__(256) void k_brunel_init(BrunelInitArgs a) {
  const int64_t k0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = k0; i < a.N; i += step) {
    a.d_v0[i] = a.v0;
    a.d_vreset[i] = a.vreset;
    a.d_thr[i] = a.thr;
    a.d_c[i] = a.c;
    a.d_rp[i] = a.rp;
  }
  for (int64_t i = k0; i <= a.P; i += step) {
    a.nlo[i] = part_start(a.N, a.P, (int)i);
    a.ilo[i] = 0;
  }
  for (int64_t i = k0; i < a.xwords; i += step) a.xlist[i] = 0ull;
  if (blockIdx.x == 0) {
    if ((int)threadIdx.x < a.ext_k) a.ext_cdf[threadIdx.x] = a.cdf[threadIdx.x];
    if (threadIdx.x < 4) a.stats[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) {
      *a.err = 0;
      *a.d_decay = 1.0f;
      *a.d_erev = 0.0f;
    }
  }
}

// ---------------------------------------------------------------------------------------
// Fixed out-degree connectivity generated on the device (the large-network builder).
//
// Units u in [0, N + Nin) are the neurons, then the Poisson inputs.  Unit u has K_u
// outgoing synapses (K for a neuron, Kin for an input), drawn with replacement.  Synapse j
// of unit u takes one Philox block r = philox(ctr = {j, 0, u, 5}, key = seed):
//   post   = floor(r.x * N / 2^32)
//   delay  = 1 + floor(r.y * dmax / 2^32)                  (steps)
//   weight = (r.z >> 8) * 2^-24 for excitatory sources (u < ne), U[0, 1) in float32;
//            w_inh for inhibitory neurons, w_in for inputs
//   scale  = scale_e / scale_i / scale_in by the same source classes
// and sits at CSR position rowptr[u] + j, rowptr[u] = u K (u <= N), N K + (u - N) Kin
// after.  The caller order of the synapses is that CSR order, so the row of a source
// needs no sort.  With `plastic`, every excitatory-to-excitatory synapse (u < ne,
// post < ne) belongs to one weight-dependent STDP rule, listed in CSR order.
//
// Two passes over the same draws: k_od_count gathers the delay range, the fixed-point
// bound of each neuron's per-step input and the rule's synapse counts per source and per
// target; after the host scans those counts, k_od_fill writes the synapse arrays and the
// rule's index tables (by source in CSR order; by target in atomic order -- the kernels
// that read that table update each synapse from one lane, so its order does not matter).
constexpr uint32_t kStreamOutDegree = 5;

struct OutDegreeArgs {
  uint64_t seed;
  int N, Nin, ne, K, Kin, dmax;
  float scale_e, scale_i, scale_in, w_inh, w_in;
  int plastic;          // E->E synapses carry the weight-dependent rule
  float cap_plastic;    // |w_max| of that rule (a bound of its weights)
  int wfmt;             // 16-bit weight words to write (0: none)
  // k_od_count
  double* bound;            // [N] sum over afferents of max|w| |scale|
  unsigned int* post_cnt;   // [N] rule synapses onto each neuron
  unsigned int* row_cnt;    // [U] rule synapses of each source
  int* drange;              // [2] min, max delay
  // k_od_fill
  const int64_t* pre_ptr;   // [U+1] exclusive scan of row_cnt
  const int64_t* post_ptr;  // [N+1] exclusive scan of post_cnt
  unsigned int* cursor;     // [N] zeroed
  int32_t* tgt;
  uint2* syn;               // {0, weight bits}
  uint16_t* delay;
  float* scale;
  uint32_t* wc;             // 16-bit weight words (compensation zero)
  int64_t* rpos;            // rule: CSR position, in CSR order
  int32_t* rpre;            //       its source unit
  uint32_t* epos;           // rule by target: CSR position
  int32_t* epre;            //                 source unit
};

struct OdSynapse {
  int post, delay;
  float w, scale;
  bool plastic;
};

__host__ __device__ __forceinline__ int64_t od_row(const OutDegreeArgs& a, int u) {
  return u <= a.N ? (int64_t)u * a.K : (int64_t)a.N * a.K + (int64_t)(u - a.N) * a.Kin;
}

__host__ __device__ __forceinline__ OdSynapse od_synapse(const OutDegreeArgs& a, int u, int j) {
  const u32x4 r = draw_block(a.seed, (int64_t)j, (uint32_t)u, kStreamOutDegree);
  OdSynapse s;
  s.post = (int)(((uint64_t)r.x * (uint64_t)a.N) >> 32);
  s.delay = 1 + (int)(((uint64_t)r.y * (uint64_t)a.dmax) >> 32);
  if (u < a.ne) {
    s.w = (float)(r.z >> 8) * 0x1p-24f;
    s.scale = a.scale_e;
  } else if (u < a.N) {
    s.w = a.w_inh;
    s.scale = a.scale_i;
  } else {
    s.w = a.w_in;
    s.scale = a.scale_in;
  }
  s.plastic = a.plastic && u < a.ne && s.post < a.ne;
  return s;
}

// one workgroup of 256 per source row (grid-stride over rows)
static __global__ __launch_bounds__(256) void k_od_count(OutDegreeArgs a) {
  __shared__ unsigned int swave[4];
  const int U = a.N + a.Nin;
  int lo = 1 << 30, hi = 0;
  for (int u = blockIdx.x; u < U; u += gridDim.x) {
    const int len = u < a.N ? a.K : a.Kin;
    unsigned int pc = 0;
    for (int j = threadIdx.x; j < len; j += blockDim.x) {
      const OdSynapse s = od_synapse(a, u, j);
      lo = min(lo, s.delay);
      hi = max(hi, s.delay);
      const float cap = s.plastic ? fmaxf(fabsf(s.w), a.cap_plastic) : fabsf(s.w);
      unsafeAtomicAdd(a.bound + s.post, (double)cap * fabs((double)s.scale));
      if (s.plastic) {
        ++pc;
        atomicAdd(a.post_cnt + s.post, 1u);
      }
    }
    for (int o = 32; o > 0; o >>= 1) pc += __shfl_xor(pc, o);
    if ((threadIdx.x & 63) == 0) swave[threadIdx.x >> 6] = pc;
    __syncthreads();
    if (threadIdx.x == 0) a.row_cnt[u] = swave[0] + swave[1] + swave[2] + swave[3];
    __syncthreads();
  }
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, __shfl_xor(lo, o));
    hi = max(hi, __shfl_xor(hi, o));
  }
  if ((threadIdx.x & 63) == 0 && hi > 0) {
    atomicMin(a.drange, lo);
    atomicMax(a.drange + 1, hi);
  }
}

static __global__ __launch_bounds__(256) void k_od_fill(OutDegreeArgs a) {
  __shared__ unsigned int swave[4];
  const int U = a.N + a.Nin;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int u = blockIdx.x; u < U; u += gridDim.x) {
    const int len = u < a.N ? a.K : a.Kin;
    const int64_t k0 = od_row(a, u);
    int64_t rbase = a.plastic ? a.pre_ptr[u] : 0;
    for (int j0 = 0; j0 < len; j0 += 256) {
      const int j = j0 + (int)threadIdx.x;
      OdSynapse s{};
      if (j < len) {
        s = od_synapse(a, u, j);
        const int64_t k = k0 + j;
        a.tgt[k] = s.post;
        a.syn[k] = make_uint2(0u, __float_as_uint(s.w));
        a.delay[k] = (uint16_t)s.delay;
        a.scale[k] = s.scale;
        if (a.wfmt) a.wc[k] = enc16(s.w, a.wfmt);
      }
      // rule index: the row's rule synapses before this one, in j order
      const uint64_t m = __ballot(s.plastic);
      const unsigned int before_w = (unsigned int)__popcll(m & ((1ull << lane) - 1ull));
      if (lane == 0) swave[wv] = (unsigned int)__popcll(m);
      __syncthreads();
      unsigned int before = before_w, tot = 0;
      for (int w = 0; w < 4; ++w) {
        if (w < wv) before += swave[w];
        tot += swave[w];
      }
      __syncthreads();
      if (s.plastic) {
        const int64_t k = k0 + j;
        const int64_t r = rbase + before;
        a.rpos[r] = k;
        a.rpre[r] = u;
        const int64_t e = a.post_ptr[s.post] + atomicAdd(a.cursor + s.post, 1u);
        a.epos[e] = (uint32_t)k;
        a.epre[e] = u;
      }
      rbase += tot;
    }
  }
}

}  // namespace spk
