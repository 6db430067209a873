// mlp.hip -- the sweep surrogate: a 5 -> 256 -> 256 -> 256 -> 256 -> 3 SiLU MLP trained and
// evaluated with hand-written gfx950 kernels.  Every matrix product runs on the BF16 MFMA
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation; the optimiser keeps FP32 master weights.
//
// One step of training = four launches on the surrogate's stream:
//   k_mlp_forward   rows in tiles of 128 or 64 per workgroup; the tile's activations stay in
//                   LDS from layer to layer, the weights come from L2; saves the activations
//                   and SiLU slopes the backward pass needs.
//   k_mlp_backward  the same tiles backwards: output gradient -> dZ4 -> ... -> dZ1, each a
//                   product with the transposed weights (kept as a BF16 copy).
//   k_mlp_wgrad     dW_l = dZ_l^T A_(l-1) and db_l, reduced over row chunks (split K);
//                   partial sums go to a [chunk][parameter] array.
//   k_mlp_adam      sums the chunks in a fixed order (deterministic), Adam on the masters,
//                   writes the BF16 copies (W, W^T, padded first and last layer).
// Every ensemble member is grid dimension y (z for the weight gradient), so one launch
// trains all members.
//
// MFMA 16x16x32 lane layout (64 lanes, l = lane): A operand 8 bf16 per lane with row
// l % 16 and reduction index 8 (l / 16) + j; B operand 8 bf16 with column l % 16 and
// reduction index 8 (l / 16) + j; result 4 floats with row 4 (l / 16) + r, column l % 16.
// A and B use the same reduction-index assignment, so a product does not depend on how
// the hardware orders the 32 reduction indices within one instruction.
//
// Tensors that a later kernel reads as MFMA operands are stored in "fragment order" FL:
// for a matrix X[m][c] (m = batch row, c = column; C columns in all)
//   FL(m, c) = ((m / 32) (C / 16) + c / 16) * 512 + ((c % 16) + 16 ((m % 32) / 8)) * 8 + m % 8
// so that one 16-byte load per lane fetches an operand fragment with the reduction running
// over rows -- what the weight gradient needs for both dZ and A.  The fragments of 32 rows lie
// in a row: with all rows of 16 columns together, the fragments that are read at one time were
// a power of two apart, on the same memory channels.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/spike_hip.h"
#include "../../include/spike_mlp.h"
#include "alloc.hpp"
#include "philox.hpp"

namespace spk {
void set_last_error(const std::string& msg);
}

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int H = SPK_MLP_HIDDEN;
constexpr int DIN = SPK_MLP_INPUTS;
constexpr int DOUT = SPK_MLP_OUTPUTS;
constexpr int K1 = 32;     // first-layer reduction: features hi (0..4), lo (5..9), zeros
constexpr int NO = 16;     // output layer padded to one 16-column block
constexpr int MT = SPK_MLP_ROW_TILE;  // rows per workgroup at most (a batch is a multiple of it)
constexpr int NT = 256;    // threads per workgroup (4 waves; wave w owns columns 64w..64w+63)
constexpr int NW = NT / 64;
constexpr int CW = H / NW, NB = CW / 16;   // columns of a wave, in blocks of 16
constexpr int LS = H + 8;  // LDS row stride in bf16 (16-byte pad: conflict-free operand reads)
constexpr int NLOSS = 64;  // rows per partial loss (those of the smaller tile)
constexpr size_t lds_bytes(int mt) { return (size_t)mt * LS * 2 + 4 * H * sizeof(float); }   // tile, biases
constexpr uint32_t kStreamBatch = 4;
constexpr int kMaxPieces = 8;   // pieces of a large inference (infer)

// FP32 master layout (per member)
constexpr int oW1 = 0, ob1 = oW1 + H * DIN;
constexpr int oW2 = ob1 + H, ob2 = oW2 + H * H;
constexpr int oW3 = ob2 + H, ob3 = oW3 + H * H;
constexpr int oW4 = ob3 + H, ob4 = oW4 + H * H;
constexpr int oW5 = ob4 + H, ob5 = oW5 + DOUT * H;
constexpr int P = ob5 + DOUT;
static_assert(P == SPK_MLP_PARAMS, "parameter count");

// BF16 working copies (per member), every matrix in operand order (wf_index): a wavefront's
// load of one fragment is 1 KB in a row.  From [row][column] matrices the same load touched
// half of 16 lines.
constexpr int bW1 = 0;               // [256][32]: W1 in columns 0..4 and again in 5..9
constexpr int bW = bW1 + H * K1;     // layers 2..4, [256][256] each, W[out][in]
constexpr int bWT = bW + 3 * H * H;  // layers 2..4 transposed, WT[in][out]
constexpr int bW5 = bWT + 3 * H * H; // [16][256]: rows 0..2 = W5
constexpr int bW5T = bW5 + NO * H;   // [256][32]: W5T[k][o] = W5[o][k], o < 3
constexpr int BF = bW5T + H * 32;

// Place of W[n][k] of a matrix of K columns in operand order: fragment (n / 16, k / 32), in it
// lane n % 16 + 16 (k % 32 / 8), element k % 8.
__host__ __device__ constexpr int wf_index(int n, int k, int K) {
  return ((n >> 4) * (K >> 5) + (k >> 5)) * 512 + ((n & 15) + 16 * ((k & 31) >> 3)) * 8 + (k & 7);
}

constexpr int oW[5] = {oW1, oW2, oW3, oW4, oW5};
constexpr int ob[5] = {ob1, ob2, ob3, ob4, ob5};

__device__ __forceinline__ uint16_t to_bf16(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest, ties to even
  return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// Four floats to four bf16 (round to nearest even; v_cvt_pk_bf16_f32 on gfx950).
__device__ __forceinline__ u16x4 pack4(float a, float b, float c, float d) {
  const uint32_t lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
  const uint32_t hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{c, d}, bf16x2));
  return u16x4{(unsigned short)lo, (unsigned short)(lo >> 16), (unsigned short)hi, (unsigned short)(hi >> 16)};
}

// logistic function with the hardware exp2 and reciprocal (about 1 ulp each)
__device__ __forceinline__ float sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * z));
}

__device__ __forceinline__ f32x4 mfma(u16x8 a, u16x8 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                 __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ size_t fl_index(int C, int m, int c) {
  return ((size_t)(m >> 5) * (size_t)(C >> 4) + (size_t)(c >> 4)) * 512 +
         (size_t)(((c & 15) + 16 * ((m & 31) >> 3)) * 8 + (m & 7));
}

// Columns [0, C) of the LDS tile (rows 0..TILE-1 = batch rows m0..) into fragment order.
template <int TILE>
__device__ __forceinline__ void store_fl(const uint16_t* lds, int C, uint16_t* dst, int m0, int w, int lane) {
  const int nmb = TILE / 32;
  const int nblk = (C / 16) * nmb;
  for (int b = w; b < nblk; b += NW) {
    const int mb = b / (C / 16), cb = b - mb * (C / 16);
    const int c = cb * 16 + (lane & 15), r = mb * 32 + (lane >> 4) * 8;
    u16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = lds[(r + j) * LS + c];
    *(u16x8*)(dst + fl_index(C, m0 + r, c)) = v;
  }
}

// Transposed tile product: acc[nb][mb] += W[CW w + 16 nb.., k] . lds[16 mb.., k] over KS steps
// of 32 (K = 32 KS), i.e. Z^T = W A^T.  Result element r of acc[nb][mb] belongs to batch
// row m = 16 mb + lane % 16 and output n = CW w + 16 nb + 4 (lane / 16) + r: every lane
// holds four consecutive outputs of one row, which it writes back as one 8-byte LDS store.
// `wf` holds the weight fragments of the first step (load_w, issued before the previous
// layer's epilogue); those of step ks + 1, and the activations of the next half step, are in
// flight while this one multiplies.
template <int KS>
__device__ __forceinline__ void load_w(const uint16_t* __restrict__ W, int w, int lane, int ks, u16x8 (&wf)[NB]) {
  const uint16_t* wp = W + ((size_t)(CW / 16 * w) * KS + ks) * 512 + lane * 8;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) wf[nb] = *(const u16x8*)(wp + (size_t)nb * KS * 512);
}

template <int KS, int MB>
__device__ __forceinline__ void mm_tile(const uint16_t* lds, const uint16_t* __restrict__ W, int w, int lane,
                                        u16x8 (&wf)[NB], f32x4 (&acc)[NB][MB]) {
  const uint16_t* ap = lds + (lane & 15) * LS + (lane >> 4) * 8;
  u16x8 wn[NB], af[2][MB / 2];
#pragma unroll
  for (int i = 0; i < MB / 2; ++i) af[0][i] = *(const u16x8*)(ap + 16 * i * LS);
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    if (ks + 1 < KS) load_w<KS>(W, w, lane, ks + 1, wn);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int mn = h == 0 ? MB / 2 : 0, kn = h == 0 ? ks : ks + 1;
      if (kn < KS) {
#pragma unroll
        for (int i = 0; i < MB / 2; ++i) af[h ^ 1][i] = *(const u16x8*)(ap + 16 * (mn + i) * LS + kn * 32);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < MB / 2; ++i)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[nb][h * (MB / 2) + i] = mfma(wf[nb], af[h][i], acc[nb][h * (MB / 2) + i]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) wf[nb] = wn[nb];
  }
}

template <int MB>
__device__ __forceinline__ size_t slope_index(int tile, int w, int nb, int mb, int lane) {
  return ((((size_t)tile * NW + w) * NB + nb) * MB + mb) * 256 + (size_t)lane * 4;
}

__device__ __forceinline__ uint16_t* lds_quad(uint16_t* lds, int w, int nb, int mb, int lane) {
  return lds + (16 * mb + (lane & 15)) * LS + CW * w + 16 * nb + 4 * (lane >> 4);
}

struct FwdArgs {
  const uint16_t* wb;    // [E][BF]
  const float* master;   // [E][P]
  const float* x;        // [n][5]
  int64_t n;             // rows of x
  int M;                 // rows per member
  int tiles, block0;     // row tiles per member; the launch's first (member, tile) in order
  int mode;              // 0: row r; 1: Philox-drawn rows
  uint64_t seed;
  const int* step;       // optimiser step (sampling counter)
  int* idx;              // [E][M] rows used (written in mode 1)
  float* y;              // [E][M][3]
  uint16_t* acts;        // [E][5][H*M] FL(A_l), l = 0..4; null in inference
  uint16_t* slopes;      // [E][4][H*M] SiLU slopes in result-fragment order
};

// Features of one row -> hi/lo bf16 pairs in columns 0..9, zeros up to 31.
__device__ __forceinline__ void feature_row(const float* x, uint16_t* row) {
#pragma unroll
  for (int j = 0; j < DIN; ++j) {
    const float f = x[j];
    const uint16_t hi = to_bf16(f);
    row[j] = hi;
    row[DIN + j] = to_bf16(f - from_bf16(hi));
  }
#pragma unroll
  for (int j = 2 * DIN; j < K1; ++j) row[j] = 0;
}

// Inference of few rows, bound by latency: tiles of 16 rows, 16 waves of 16 columns each.  A
// wave holds its weights of a whole layer in registers, loaded two layers ahead, so that a
// layer is eight products on the LDS rows and one epilogue of four values per lane; the rows
// alternate between two LDS tiles (one barrier per layer).  The products and their order are
// those of k_mlp_forward.
constexpr int NTS = 1024, TS = 16;
__global__ __launch_bounds__(NTS) void k_mlp_forward_small(FwdArgs a) {
  __shared__ __align__(16) uint16_t rows[2][TS * LS];
  const int tile = (int)blockIdx.x % a.tiles, e = (int)blockIdx.x / a.tiles;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63, r16 = lane & 15, kg = (lane >> 4) * 8;
  const int m0 = tile * TS, M = a.M;
  const uint16_t* wb = a.wb + (size_t)e * BF + lane * 8;
  const float* mst = a.master + (size_t)e * P;
  auto load = [&](const uint16_t* W, u16x8 (&f)[8]) {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) f[ks] = *(const u16x8*)(W + ks * 512);
  };
  const uint16_t* wl = wb + bW + w * 8 * 512;
  const u16x8 w1 = *(const u16x8*)(wb + bW1 + w * 512);
  f32x4 bv[4];
#pragma unroll
  for (int l = 0; l < 4; ++l) {
    const float* bq = mst + ob[l] + 16 * w + 4 * (lane >> 4);
    bv[l] = f32x4{bq[0], bq[1], bq[2], bq[3]};
  }
  u16x8 wa[8], wc[8];
  load(wl, wa);
  load(wl + H * H, wc);
  if (tid < TS) feature_row(a.x + (int64_t)min(m0 + tid, M - 1) * DIN, rows[0] + tid * LS);
  __syncthreads();
  auto epilogue = [&](f32x4 z, uint16_t* dst) {
    *(u16x4*)(dst + r16 * LS + 16 * w + 4 * (lane >> 4)) =
        pack4(z[0] * sigmoid(z[0]), z[1] * sigmoid(z[1]), z[2] * sigmoid(z[2]), z[3] * sigmoid(z[3]));
  };
  auto product = [&](const u16x8 (&f)[8], const uint16_t* src, f32x4 z) {
#pragma unroll
    for (int ks = 0; ks < 8; ++ks) z = mfma(f[ks], *(const u16x8*)(src + r16 * LS + ks * 32 + kg), z);
    return z;
  };
  epilogue(mfma(w1, *(const u16x8*)(rows[0] + r16 * LS + kg), bv[0]), rows[1]);
  __syncthreads();
  const f32x4 z2 = product(wa, rows[1], bv[1]);
  load(wl + 2 * H * H, wa);
  epilogue(z2, rows[0]);
  __syncthreads();
  const f32x4 z3 = product(wc, rows[0], bv[2]);
  if (w == 0) load(wb + bW5, wc);
  epilogue(z3, rows[1]);
  __syncthreads();
  epilogue(product(wa, rows[1], bv[3]), rows[0]);
  __syncthreads();
  if (w != 0) return;
  f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
  if (lane < 16) o = f32x4{mst[ob5], mst[ob5 + 1], mst[ob5 + 2], 0.0f};
  o = product(wc, rows[0], o);
  const int r = m0 + lane;
  if (lane < TS && r < M) {
    float* yp = a.y + ((size_t)e * M + r) * DOUT;
    yp[0] = o[0]; yp[1] = o[1]; yp[2] = o[2];
  }
}

// Bound by issue in inference: of a tile's layer, the matrix products take 4096 cycles of the
// matrix cores and half of that of the issue port, the SiLU of 128 values per lane about 4000
// (8 transcendental and 14 plain instructions per four values), and the two wavefronts of a
// SIMD (256 registers each) overlap the rest.  8 x 262147 rows: 1257 us with row-major weights
// (a fragment load touched half of 16 lines) and two activation fragments in flight, 920 us
// now = 906 TFLOP/s; more, smaller wavefronts (8 of 32 columns, 4 of a SIMD) 1010 us.  In
// training bound by memory: 8 x 4096 rows write 136 MB of activations and slopes in 41 us.
template <bool TRAIN, int TILE>
__global__ __launch_bounds__(NT, TILE == MT ? 2 : 3) void k_mlp_forward(FwdArgs a) {
  constexpr int MB = TILE / 16;
  extern __shared__ __align__(16) uint16_t lds[];
  float* lbias = (float*)(lds + TILE * LS);   // biases of layers 1..4
  const int tile = (a.block0 + (int)blockIdx.x) % a.tiles, e = (a.block0 + (int)blockIdx.x) / a.tiles;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int m0 = tile * TILE;
  const int M = a.M;
  const uint16_t* wb = a.wb + (size_t)e * BF;
  const float* mst = a.master + (size_t)e * P;

#pragma unroll
  for (int l = 0; l < 4; ++l) lbias[l * H + tid] = mst[ob[l] + tid];
  static_assert(NT == H, "a bias per thread and layer");
  if (tid < TILE) {
    const int r = m0 + tid;
    int64_t i;
    if (a.mode == 1) {
      const uint32_t u = spk::draw_u32(a.seed, (int64_t)(*a.step) * M + r, (uint32_t)e, kStreamBatch);
      i = (int64_t)(((uint64_t)u * (uint64_t)a.n) >> 32);
      if (r < M) a.idx[(size_t)e * M + r] = (int)i;
    } else {
      i = r < M ? r : M - 1;
    }
    feature_row(a.x + i * DIN, lds + tid * LS);
  }
  __syncthreads();
  if constexpr (TRAIN) store_fl<TILE>(lds, K1, a.acts + ((size_t)e * 5 + 0) * H * M, m0, w, lane);

  // a layer's first weights, loaded before the epilogue of the layer before
  u16x8 wf[NB];
  load_w<1>(wb + bW1, w, lane, 0, wf);
  for (int l = 1; l <= 4; ++l) {
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const f32x4 bv = *(const f32x4*)(lbias + (l - 1) * H + CW * w + 16 * nb + 4 * (lane >> 4));
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = bv;
    }
    if (l == 1)
      mm_tile<1, MB>(lds, wb + bW1, w, lane, wf, acc);
    else
      mm_tile<8, MB>(lds, wb + bW + (size_t)(l - 2) * H * H, w, lane, wf, acc);
    if (l < 4) load_w<8>(wb + bW + (size_t)(l - 1) * H * H, w, lane, 0, wf);
    __syncthreads();  // every wave has read the layer input
    uint16_t* sl = TRAIN ? a.slopes + ((size_t)e * 4 + (l - 1)) * H * M : nullptr;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const f32x4 z = acc[nb][mb];
        const f32x4 sg = {sigmoid(z[0]), sigmoid(z[1]), sigmoid(z[2]), sigmoid(z[3])};
        *(u16x4*)lds_quad(lds, w, nb, mb, lane) = pack4(z[0] * sg[0], z[1] * sg[1], z[2] * sg[2], z[3] * sg[3]);
        if constexpr (TRAIN)
          *(u16x4*)(sl + slope_index<MB>(tile, w, nb, mb, lane)) =
              pack4(sg[0] * (1.0f + z[0] * (1.0f - sg[0])), sg[1] * (1.0f + z[1] * (1.0f - sg[1])),
                    sg[2] * (1.0f + z[2] * (1.0f - sg[2])), sg[3] * (1.0f + z[3] * (1.0f - sg[3])));
      }
    __syncthreads();
    if constexpr (TRAIN) store_fl<TILE>(lds, H, a.acts + ((size_t)e * 5 + l) * H * M, m0, w, lane);
  }

  // output layer, transposed: Y^T = W5 A4^T; wave w takes row block w; lanes 0..15 hold
  // outputs 0..3 (3 used) of row 16 w + lane
  {
    const int r16 = lane & 15, kg = (lane >> 4) * 8;
    const uint16_t* wp = wb + bW5 + lane * 8;
#pragma unroll
    for (int rb = 0; rb < MB; rb += NW) {
      const int row = 16 * (rb + w);
      f32x4 o = {0.0f, 0.0f, 0.0f, 0.0f};
      if (lane < 16) o = f32x4{mst[ob5], mst[ob5 + 1], mst[ob5 + 2], 0.0f};
#pragma unroll
      for (int ks = 0; ks < 8; ++ks)
        o = mfma(*(const u16x8*)(wp + ks * 512), *(const u16x8*)(lds + (row + r16) * LS + ks * 32 + kg), o);
      const int r = m0 + row + lane;
      if (lane < 16 && r < M) {
        float* yp = a.y + ((size_t)e * M + r) * DOUT;
        yp[0] = o[0]; yp[1] = o[1]; yp[2] = o[2];
      }
    }
  }
}

// What all parameters of an Adam step share, computed by the thread that counts the step (per
// parameter: two powf and a cosf each).
constexpr float kBeta1 = 0.9f, kBeta2 = 0.999f;
__device__ __forceinline__ void adam_uniform(int t, float lr0, float lr_min, int total, float* uni) {
  const float u = (float)min(max(t - 1, 0), total) / (float)max(total, 1);
  uni[0] = lr_min + 0.5f * (lr0 - lr_min) * (1.0f + cosf(3.14159265358979f * u));
  uni[1] = 1.0f - powf(kBeta1, (float)t);
  uni[2] = 1.0f - powf(kBeta2, (float)t);
}

struct BwdArgs {
  const uint16_t* wb;
  const float* y;         // [E][M][3]
  const float* t;         // targets [n][3]
  const int* idx;         // [E][M] rows of t (null: row r)
  float w0, w1, w2;       // loss weights
  float scale;            // 2 / M
  const uint16_t* slopes; // [E][4][H*M]
  uint16_t* grads;        // [E][5][H*M]: FL(dZ_1..dZ_4) in slots 0..3, FL(dY) (16 columns) in 4
  float* loss_part;       // [E][M / NLOSS]
  int* step;              // incremented once when tick != 0, which also sets uni (adam_uniform)
  int tick;
  float lr0, lr_min;
  int total;
  float* uni;
  int M;
};

// Bound by memory: 8 x 4096 rows read 67 MB of slopes and write 67 MB of gradients in 32 us
// (42 us with row-major weights in 128-row tiles).
template <int TILE>
__global__ __launch_bounds__(NT, TILE == MT ? 2 : 3) void k_mlp_backward(BwdArgs a) {
  constexpr int MB = TILE / 16;
  extern __shared__ __align__(16) uint16_t lds[];
  const int tile = blockIdx.x, e = blockIdx.y;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int m0 = tile * TILE, M = a.M;
  const uint16_t* wb = a.wb + (size_t)e * BF;

  if (a.tick && tile == 0 && e == 0 && tid == 0) {
    *a.step += 1;
    adam_uniform(*a.step, a.lr0, a.lr_min, a.total, a.uni);
  }

  // output gradient dy = bf16(2 w_o (y - t) / M) in LDS columns 0..2, zeros up to 31
  float lsum = 0.0f;
  if (tid < TILE) {
    const int r = m0 + tid;
    const int64_t i = a.idx ? a.idx[(size_t)e * M + r] : r;
    const float wo[3] = {a.w0, a.w1, a.w2};
    uint16_t* row = lds + tid * LS;
#pragma unroll
    for (int o = 0; o < DOUT; ++o) {
      const float res = a.y[((size_t)e * M + r) * DOUT + o] - a.t[i * DOUT + o];
      lsum += wo[o] * res * res;
      row[o] = to_bf16(a.scale * wo[o] * res);
    }
#pragma unroll
    for (int j = DOUT; j < K1; ++j) row[j] = 0;
  }
  // loss of every NLOSS rows, summed in a fixed order
  static_assert(NLOSS == 64, "rows of a wavefront");
#pragma unroll
  for (int s = 32; s > 0; s >>= 1) lsum += __shfl_xor(lsum, s);
  if (lane == 0 && w < TILE / NLOSS) a.loss_part[(size_t)e * (M / NLOSS) + m0 / NLOSS + w] = lsum;
  __syncthreads();
  store_fl<TILE>(lds, NO, a.grads + ((size_t)e * 5 + 4) * H * M, m0, w, lane);

  u16x8 wf[NB];
  load_w<1>(wb + bW5T, w, lane, 0, wf);
  for (int l = 4; l >= 1; --l) {
    // dA_l^T = W_(l+1)^T dZ_(l+1)^T  (for l = 4: W5^T dY^T)
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    if (l == 4)
      mm_tile<1, MB>(lds, wb + bW5T, w, lane, wf, acc);
    else
      mm_tile<8, MB>(lds, wb + bWT + (size_t)(l - 1) * H * H, w, lane, wf, acc);
    if (l > 1) load_w<8>(wb + bWT + (size_t)(l - 2) * H * H, w, lane, 0, wf);
    __syncthreads();
    const uint16_t* sl = a.slopes + ((size_t)e * 4 + (l - 1)) * H * M;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const u16x4 sv = *(const u16x4*)(sl + slope_index<MB>(tile, w, nb, mb, lane));
        const f32x4 d = acc[nb][mb];
        *(u16x4*)lds_quad(lds, w, nb, mb, lane) =
            pack4(d[0] * from_bf16(sv[0]), d[1] * from_bf16(sv[1]), d[2] * from_bf16(sv[2]), d[3] * from_bf16(sv[3]));
      }
    __syncthreads();
    store_fl<TILE>(lds, H, a.grads + ((size_t)e * 5 + (l - 1)) * H * M, m0, w, lane);
  }
}

struct WgradArgs {
  const uint16_t* acts;   // [E][5][H*M]
  const uint16_t* grads;  // [E][5][H*M]
  float* part;            // [E][S][P]
  int M, chunk;           // rows, rows per split
  int S, models;
};

// Workgroups of layers 2..4 for `se` splits of members: four for each, in groups of 8 XCDs.
__host__ __device__ constexpr int wgrad_big_blocks(int se) { return (3 * se + 7) / 8 * 32; }

// 56 wave jobs per member and split: dW1 (4 row tiles of 64 x 32 columns), dW2..dW4
// (16 tiles of 64 x 64 each), dW5 (4 tiles of 16 rows x 64 columns); the first column
// tile of each layer also sums the bias gradient.  A workgroup takes the four tiles of one
// row of a layer, which share their dZ; the four workgroups of a layer share its A and follow
// each other at a distance of 8 in the grid, on one XCD, whose L2 then reads A once.  Layers 2
// to 4 of every member and split come first, then the two small layers.  Bound by memory: 8 x
// 4096 rows in 4 splits read 134 MB and write 26 MB in 40 us (55 us with A read by four XCDs,
// 32 rows at a time, and fragments a power of two apart).
__global__ __launch_bounds__(NT) void k_mlp_wgrad(WgradArgs a) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int S = a.S, M = a.M, SE = S * a.models, big = wgrad_big_blocks(SE);
  int layer, n0, k0, nrb, ncb, se;
  if ((int)blockIdx.x < big) {
    const int g = ((int)blockIdx.x / 32) * 8 + (int)blockIdx.x % 8;   // layer, split and member
    if (g >= 3 * SE) return;
    layer = 2 + g / SE; se = g % SE;
    n0 = 64 * (((int)blockIdx.x / 8) % 4); k0 = 64 * w; nrb = 4; ncb = 4;
  } else {
    const int q = (int)blockIdx.x - big;
    se = q % SE;
    if (q < SE) {
      layer = 1; n0 = 64 * w; k0 = 0; nrb = 4; ncb = 2;
    } else {
      layer = 5; n0 = 0; k0 = 64 * w; nrb = 1; ncb = 4;
    }
  }
  const int s = se % S, e = se / S;
  const uint16_t* dz = a.grads + ((size_t)e * 5 + (layer - 1)) * H * M;  // layer 5: dY
  const uint16_t* ac = a.acts + ((size_t)e * 5 + (layer - 1)) * H * M;
  const int dcb = layer == 5 ? 1 : H / 16, acb = layer == 1 ? K1 / 16 : H / 16;   // column blocks of dZ and A
  const int mb0 = (s * a.chunk) >> 5, mb1 = mb0 + (a.chunk >> 5);
  f32x4 acc[4][4];
  float rs[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const bool bias = k0 == 0;
  // fragments of the next 96 rows are in flight while 32 multiply
  u16x8 bv[4][4], av[4][4];
  auto load = [&](int mb, int k) {
#pragma unroll
    for (int cb = 0; cb < 4; ++cb)
      if (cb < ncb) bv[k][cb] = *(const u16x8*)(ac + ((size_t)mb * acb + (k0 >> 4) + cb) * 512 + lane * 8);
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
      if (rb < nrb) av[k][rb] = *(const u16x8*)(dz + ((size_t)mb * dcb + (n0 >> 4) + rb) * 512 + lane * 8);
  };
  auto mul = [&](int k) {
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      if (rb >= nrb) continue;
      if (bias) {
#pragma unroll
        for (int j = 0; j < 8; ++j) rs[rb] += from_bf16(av[k][rb][j]);
      }
#pragma unroll
      for (int cb = 0; cb < 4; ++cb)
        if (cb < ncb) acc[rb][cb] = mfma(av[k][rb], bv[k][cb], acc[rb][cb]);
    }
  };
#pragma unroll
  for (int k = 0; k < 3; ++k) load(mb0 + k, k);
  for (int mb = mb0; mb < mb1; mb += 4) {   // (chunks are multiples of 128 rows)
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      if (mb + k + 3 < mb1) load(mb + k + 3, (k + 3) & 3);
      __builtin_amdgcn_sched_barrier(0);
      mul(k);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  float* out = a.part + ((size_t)e * S + s) * P;
  const int r16 = lane & 15, rg = (lane >> 4) * 4;
  const int ndim = layer == 5 ? DOUT : H;
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    if (rb >= nrb) continue;
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) {
      if (cb >= ncb) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int n = n0 + 16 * rb + rg + r, k = k0 + 16 * cb + r16;
        float v = acc[rb][cb][r];
        if (layer == 1) {
          // W1 column k is used by the hi (k) and lo (k + 5) feature halves
          const float v5 = __shfl(v, (lane & 48) | ((r16 + DIN) & 15));
          if (cb == 0 && r16 < DIN && n < ndim) out[oW1 + n * DIN + r16] = v + v5;
        } else if (n < ndim) {
          out[oW[layer - 1] + n * H + k] = v;
        }
      }
    }
    if (bias) {
      float v = rs[rb];
      v += __shfl_xor(v, 16);
      v += __shfl_xor(v, 32);
      const int n = n0 + 16 * rb + lane;
      if (lane < 16 && n < ndim) out[ob[layer - 1] + n] = v;
    }
  }
}

struct AdamArgs {
  float* master; float* mom; float* vel;
  uint16_t* wb;
  const float* part; int S;   // partial gradients [E][S][P] (or)
  const float* gin;           // caller gradients [E][P]
  float* gout;                // gradients [E][P] (optional)
  const float* uni;           // learning rate and bias corrections of the step (adam_uniform)
  int apply;                  // 0: gradients only; 1: Adam step; 2: write the BF16 copies only
};

__device__ __forceinline__ void write_copies(uint16_t* wb, int p, float v) {
  const uint16_t h = to_bf16(v);
  if (p < ob1) {
    const int n = p / DIN, k = p - n * DIN;
    wb[bW1 + wf_index(n, k, K1)] = h;
    wb[bW1 + wf_index(n, DIN + k, K1)] = h;
  } else if (p >= oW2 && p < oW5) {
    int L = -1, q = 0;
    if (p < ob2) {
      L = 0; q = p - oW2;
    } else if (p >= oW3 && p < ob3) {
      L = 1; q = p - oW3;
    } else if (p >= oW4 && p < ob4) {
      L = 2; q = p - oW4;
    }
    if (L >= 0) {  // biases of layers 2..4 have no working copy
      const int n = q >> 8, k = q & 255;
      wb[bW + L * H * H + wf_index(n, k, H)] = h;
      wb[bWT + L * H * H + wf_index(k, n, H)] = h;
    }
  } else if (p >= oW5 && p < ob5) {
    const int o = (p - oW5) >> 8, k = (p - oW5) & 255;
    wb[bW5 + wf_index(o, k, H)] = h;
    wb[bW5T + wf_index(k, o, 32)] = h;
  }
}

// The parameter of a thread: tiles of 8 outputs x 32 inputs of the big matrices (a wavefront
// 8 x 8, whose working copies W and W^T are runs of 128 bytes each), then the other parameters
// in order; -1: none.  In plain order the copies W^T went out two bytes at a time into lines
// that eight XCDs shared.
constexpr int kAdamBig = 3 * H * H / 256, kAdamBlocks = kAdamBig + (P - 3 * H * H + 255) / 256;
__device__ __forceinline__ int adam_param(int block, int tid) {
  if (block < kAdamBig) {
    const int l = block / (H * H / 256), q = block % (H * H / 256);
    const int n = q / (H / 32) * 8 + (tid & 7), k = q % (H / 32) * 32 + (tid >> 3);
    return (l == 0 ? oW2 : l == 1 ? oW3 : oW4) + n * H + k;
  }
  const int r = (block - kAdamBig) * 256 + tid;   // W1, b1 | b2 | b3 | b4, W5, b5
  if (r < oW2) return r;
  if (r < oW2 + H) return ob2 + r - oW2;
  if (r < oW2 + 2 * H) return ob3 + r - oW2 - H;
  return r < P - 3 * H * H ? ob4 + r - oW2 - 2 * H : -1;
}

__global__ __launch_bounds__(256) void k_mlp_adam(AdamArgs a) {
  const int p = adam_param(blockIdx.x, threadIdx.x), e = blockIdx.y;
  if (p < 0) return;
  const size_t ep = (size_t)e * P + p;
  float* mst = a.master + ep;
  uint16_t* wb = a.wb + (size_t)e * BF;
  if (a.apply == 2) {
    write_copies(wb, p, *mst);
    return;
  }
  float g;
  if (a.gin) {
    g = a.gin[ep];
  } else {
    g = 0.0f;
    const float* pp = a.part + (size_t)e * a.S * P + p;
    for (int s = 0; s < a.S; ++s) g += pp[(size_t)s * P];
  }
  if (a.gout) a.gout[ep] = g;
  if (!a.apply) return;
  const float b1 = kBeta1, b2 = kBeta2, eps = 1e-8f;
  const float lr = a.uni[0], c1 = a.uni[1], c2 = a.uni[2];
  const float m = b1 * a.mom[ep] + (1.0f - b1) * g;
  const float v = b2 * a.vel[ep] + (1.0f - b2) * g * g;
  a.mom[ep] = m;
  a.vel[ep] = v;
  const float val = *mst - lr * (m / c1) / (sqrtf(v / c2) + eps);
  *mst = val;
  write_copies(wb, p, val);
}

// *bad = least index of a parameter that is not finite (from all ones).
__global__ __launch_bounds__(256) void k_mlp_check(const float* p, unsigned int n, unsigned int* bad) {
  for (unsigned int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256)
    if ((__float_as_uint(p[i]) & 0x7F800000u) == 0x7F800000u) atomicMin(bad, i);
}

__global__ void k_mlp_tick(int* step, float lr, float* uni) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    *step += 1;
    adam_uniform(*step, lr, lr, 1, uni);
  }
}

}  // namespace

// ------------------------------------------------------------------------------------------
// host side

struct spk_mlp {
  int E = 0, max_batch = 0;
  float *master = nullptr, *mom = nullptr, *vel = nullptr;
  uint16_t* wb = nullptr;
  float *x = nullptr, *t = nullptr;
  int64_t n = 0, cap = 0;
  int* idx = nullptr;
  float* y = nullptr;
  uint16_t *acts = nullptr, *slopes = nullptr, *grads = nullptr;
  float *part = nullptr, *loss_part = nullptr, *gbuf = nullptr, *gin = nullptr;
  int* step = nullptr;
  float* uni = nullptr;
  unsigned int* bad = nullptr;
  float *px = nullptr, *py = nullptr;
  int64_t pcap = 0;
  float* scratch = nullptr;  // this device's copy of the file-scope staging array
  float wout[3] = {1.0f, 1.0f, 1.0f};
  hipStream_t stream = nullptr, copy = nullptr;   // copy: results of a piece beside the next one
  hipEvent_t ev[6] = {};
  hipEvent_t piece[kMaxPieces] = {};
  hipGraphExec_t graph = nullptr;
  int graph_batch = 0, graph_mode = -1;
  uint64_t graph_seed = 0;
  float graph_lr0 = 0, graph_lrmin = 0;
  int graph_total = 0;
  spk_mlp_timing timing = {};
};

// Staging memory of spk_mlp_predict_noalloc: features then outputs, in a file-scope
// device array of kNoAllocBytes.  Every GPU the library runs on holds its own copy until
// the process ends.  The array's name is a host-side stand-in in host code: its device
// address (one per GPU) comes from hipGetSymbolAddress at spk_mlp_create.
constexpr size_t kNoAllocBytes = size_t(4) << 20;
constexpr size_t kNoAllocFloats = kNoAllocBytes / sizeof(float);
static __device__ __align__(256) float scratch[kNoAllocFloats];

namespace {

int mfail(int code, const std::string& msg);

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
float* g_scratch_addr[kMaxDevices] = {};

// Device address of `scratch` on the current device `dev`, looked up once per device.
int scratch_address(int dev, float** out) {
  if (dev < 0 || dev >= kMaxDevices) return mfail(SPK_ERR_ARG, "device ordinal out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_addr[dev]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return mfail(SPK_ERR_HIP, std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
    g_scratch_addr[dev] = (float*)p;
  }
  *out = g_scratch_addr[dev];
  return SPK_OK;
}

}  // namespace

namespace {

int mfail(int code, const std::string& msg) {
  spk::set_last_error(msg);
  return code;
}

#define MLP_HIP(expr)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      return mfail(SPK_ERR_HIP, std::string(#expr) + " failed: " + hipGetErrorString(e_)); \
  } while (0)

template <typename T>
int malloc_d(T** p, size_t n) {
  *p = nullptr;
  const hipError_t e = spk::device_malloc((void**)p, std::max<size_t>(n, 1) * sizeof(T));
  if (e != hipSuccess) return mfail(SPK_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  return SPK_OK;
}

template <typename T>
void free_d(T*& p) {
  if (p) (void)hipFree((void*)p);
  p = nullptr;
}

int lds_attributes() {
  static int done = 0;
  if (done) return SPK_OK;
  for (const void* fn : {(const void*)k_mlp_forward<false, MT>, (const void*)k_mlp_forward<true, MT>,
                         (const void*)k_mlp_backward<MT>})
    MLP_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes(MT)));
  done = 1;
  return SPK_OK;
}

// Inference: pieces have at least one round of the chip of 128-row tiles (8 members x 262147
// rows, 25 MB of results to pageable memory, one handle called in a loop: 2.51 ms in one piece,
// 2.05 in 2, 1.90 in 4, 1.78 in 8; the kernels alone 0.94 and 1.03 ms.  The copy's time hangs on
// the caller's pages: 1.75 to 1.9 ms in such loops, 2.5 to 2.6 where calls of several handles with
// other rows take turns); k_mlp_forward_small takes at most one 16-row tile per CU (8 members x
// 500 rows 10.3 us, in 64-row tiles 13.3; x 1000 rows, two rounds, 17.6 and 14.8; x 100 rows 10.8,
// 14.3).
constexpr int64_t kPieceTiles = 512, kSmallTiles = 256;

// Row tile of the passes over `rows` rows of `models` members: half tiles while whole ones give
// at most one workgroup for each of the 256 CUs of the MI355X.  A training step's two passes take,
// in whole and in half tiles, 71 and 55 us at 128 whole tiles, 85 and 80 at 256, 98 and 99 at 288,
// 115 and 112 at 320, 126 and 131 at 384, 144 and 174 at 512 (half tiles read the weights twice).
// Inference follows the same line: 26 and 22 us at 256 tiles; it would gain beyond it, too (35 and
// 27 at 288, 38 and 35 at 512, 53 and 48 at 768).
bool half_tiles(int64_t rows, int models) { return (rows + MT - 1) / MT * models <= 256; }

template <bool TRAIN>
void launch_forward(FwdArgs f, int models, hipStream_t st) {
  const int tile = half_tiles(f.M, models) ? MT / 2 : MT;
  f.tiles = (f.M + tile - 1) / tile;
  const dim3 grid((unsigned)(f.tiles * models));
  if (tile == MT) hipLaunchKernelGGL((k_mlp_forward<TRAIN, MT>), grid, dim3(NT), lds_bytes(MT), st, f);
  else hipLaunchKernelGGL((k_mlp_forward<TRAIN, MT / 2>), grid, dim3(NT), lds_bytes(MT / 2), st, f);
}

// Outputs of every member for n rows of features on the device, into `y` and from there to
// the host (`out`); ev[0], ev[1] around the kernels.  Few rows (at most one 16-row tile per CU)
// take the kernel made for latency.  Many rows are cut into pieces (`pieces`: not for callers
// that may not allocate, as the first such call makes a stream), and the copy of a piece runs
// on a second stream while the next one computes.
int infer(spk_mlp* m, const float* x, int64_t n, float* y, float* out, bool pieces_ok) {
  FwdArgs f{};
  f.wb = m->wb; f.master = m->master; f.x = x; f.n = n; f.M = (int)n; f.mode = 0; f.y = y;
  const size_t row = DOUT * sizeof(float);
  const int64_t small = (n + TS - 1) / TS * m->E, blocks = (n + MT - 1) / MT * m->E;
  MLP_HIP(hipEventRecord(m->ev[0], m->stream));
  if (pieces_ok && small > kSmallTiles && blocks >= 2 * kPieceTiles) {
    if (!m->copy) MLP_HIP(hipStreamCreateWithFlags(&m->copy, hipStreamNonBlocking));
    f.tiles = (int)((n + MT - 1) / MT);
    const int pieces = (int)std::min<int64_t>(kMaxPieces, blocks / kPieceTiles);
    auto first = [&](int k) { return blocks * k / pieces; };
    for (int k = 0; k < pieces; ++k) {
      f.block0 = (int)first(k);
      hipLaunchKernelGGL((k_mlp_forward<false, MT>), dim3((unsigned)(first(k + 1) - first(k))), dim3(NT), lds_bytes(MT),
                         m->stream, f);
      if (!m->piece[k]) MLP_HIP(hipEventCreateWithFlags(&m->piece[k], hipEventDisableTiming));
      MLP_HIP(hipEventRecord(m->piece[k], m->stream));
    }
    MLP_HIP(hipEventRecord(m->ev[1], m->stream));
    MLP_HIP(hipGetLastError());
    // the rows of the (member, tile) pairs before block b
    auto rows = [&](int64_t b) { return b / f.tiles * n + std::min<int64_t>(n, b % f.tiles * MT); };
    for (int k = 0; k < pieces; ++k) {
      const int64_t r0 = rows(first(k)), r1 = rows(first(k + 1));
      MLP_HIP(hipStreamWaitEvent(m->copy, m->piece[k], 0));
      MLP_HIP(hipMemcpyAsync((char*)out + r0 * row, (const char*)y + r0 * row, (r1 - r0) * row, hipMemcpyDeviceToHost,
                             m->copy));
    }
    MLP_HIP(hipStreamSynchronize(m->copy));
    MLP_HIP(hipStreamSynchronize(m->stream));
    return SPK_OK;
  }
  if (small <= kSmallTiles) {
    f.tiles = (int)((n + TS - 1) / TS);
    hipLaunchKernelGGL(k_mlp_forward_small, dim3((unsigned)small), dim3(NTS), 0, m->stream, f);
  } else {
    launch_forward<false>(f, m->E, m->stream);
  }
  MLP_HIP(hipEventRecord(m->ev[1], m->stream));
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipMemcpyAsync(out, y, (size_t)m->E * n * row, hipMemcpyDeviceToHost, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  return SPK_OK;
}

void launch_backward(const BwdArgs& b, int models, hipStream_t st) {
  if (half_tiles(b.M, models))
    hipLaunchKernelGGL(k_mlp_backward<MT / 2>, dim3(b.M / (MT / 2), models), dim3(NT), lds_bytes(MT / 2), st, b);
  else
    hipLaunchKernelGGL(k_mlp_backward<MT>, dim3(b.M / MT, models), dim3(NT), lds_bytes(MT), st, b);
}

// Row chunks of the weight gradient: chunks of about 1024 rows (8 tiles), at most
// kMaxSplits, dividing the batch evenly.  Every chunk writes a full parameter-sized partial
// sum, so fewer, longer chunks cost less traffic than many short ones.
constexpr int kMaxSplits = 16;
int splits(int batch) {
  const int q = batch / MT;
  for (int s = std::min(std::max(q / 8, 1), kMaxSplits); s > 1; --s)
    if (q % s == 0) return s;
  return 1;
}

// one training step (forward, backward, weight gradient, Adam) on the surrogate's stream
int enqueue_step(spk_mlp* m, int batch, int mode, uint64_t seed, int apply, float lr0, float lr_min, int total,
                 float* gout, float* loss_part, bool timed) {
  FwdArgs f{};
  f.wb = m->wb; f.master = m->master; f.x = m->x; f.n = m->n; f.M = batch; f.mode = mode; f.seed = seed;
  f.step = m->step; f.idx = m->idx; f.y = m->y; f.acts = m->acts; f.slopes = m->slopes;
  if (timed) MLP_HIP(hipEventRecord(m->ev[0], m->stream));
  launch_forward<true>(f, m->E, m->stream);
  if (timed) MLP_HIP(hipEventRecord(m->ev[1], m->stream));
  BwdArgs b{};
  b.wb = m->wb; b.y = m->y; b.t = m->t; b.idx = mode == 1 ? m->idx : nullptr;
  b.w0 = m->wout[0]; b.w1 = m->wout[1]; b.w2 = m->wout[2];
  b.scale = 2.0f / (float)batch;
  b.slopes = m->slopes; b.grads = m->grads; b.loss_part = loss_part; b.step = m->step; b.tick = apply == 1;
  b.lr0 = lr0; b.lr_min = lr_min; b.total = total; b.uni = m->uni;
  b.M = batch;
  launch_backward(b, m->E, m->stream);
  if (timed) MLP_HIP(hipEventRecord(m->ev[2], m->stream));
  const int S = splits(batch);
  const int chunk = batch / S;
  WgradArgs g{};
  g.acts = m->acts; g.grads = m->grads; g.part = m->part; g.M = batch; g.chunk = chunk; g.S = S; g.models = m->E;
  hipLaunchKernelGGL(k_mlp_wgrad, dim3(wgrad_big_blocks(S * m->E) + 2 * S * m->E), dim3(NT), 0, m->stream, g);
  if (timed) MLP_HIP(hipEventRecord(m->ev[3], m->stream));
  AdamArgs ad{};
  ad.master = m->master; ad.mom = m->mom; ad.vel = m->vel; ad.wb = m->wb; ad.part = m->part; ad.S = S;
  ad.gin = nullptr; ad.gout = gout; ad.uni = m->uni;
  ad.apply = apply;
  hipLaunchKernelGGL(k_mlp_adam, dim3(kAdamBlocks, m->E), dim3(256), 0, m->stream, ad);
  if (timed) MLP_HIP(hipEventRecord(m->ev[4], m->stream));
  MLP_HIP(hipGetLastError());
  return SPK_OK;
}

// The captured training step holds the data pointers, the row count and the loss weights
// as kernel arguments: any change to them drops it (it is captured again when needed).
void drop_graph(spk_mlp* m) {
  if (m->graph) (void)hipGraphExecDestroy(m->graph);
  m->graph = nullptr;
}

int check_batch(spk_mlp* m, int batch) {
  if (batch <= 0 || batch % MT || batch > m->max_batch)
    return mfail(SPK_ERR_ARG, "batch must be a positive multiple of " + std::to_string(MT) + " up to max_batch " +
                                  std::to_string(m->max_batch));
  return SPK_OK;
}

float elapsed(hipEvent_t a, hipEvent_t b) {
  float ms = 0.0f;
  (void)hipEventElapsedTime(&ms, a, b);
  return ms;
}

}  // namespace

extern "C" {

int spk_mlp_param_count(void) { return P; }

int spk_mlp_create(int models, int max_batch, spk_mlp** out) {
  if (!out) return mfail(SPK_ERR_ARG, "null output handle");
  *out = nullptr;
  if (models < 1 || models > 64) return mfail(SPK_ERR_ARG, "models must be 1..64");
  if (max_batch < 1 || max_batch > (1 << 20)) return mfail(SPK_ERR_ARG, "max_batch must be 1..2^20");
  int dev = 0, ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return mfail(SPK_ERR_NODEVICE, "no HIP device");
  MLP_HIP(hipGetDevice(&dev));
  int rc = lds_attributes();
  if (rc) return rc;
  float* scr = nullptr;
  if ((rc = scratch_address(dev, &scr))) return rc;
  spk_mlp* m = new spk_mlp();
  m->scratch = scr;
  m->E = models;
  m->max_batch = (max_batch + MT - 1) / MT * MT;
  const size_t E = models, Mx = m->max_batch;
  const size_t S = kMaxSplits;
  auto bail = [&](int r) { spk_mlp_destroy(m); return r; };
#define MLP_ALLOC(p, cnt) if ((rc = malloc_d(&(p), (cnt)))) return bail(rc)
  MLP_ALLOC(m->master, E * P);
  MLP_ALLOC(m->mom, E * P);
  MLP_ALLOC(m->vel, E * P);
  MLP_ALLOC(m->wb, E * BF);
  MLP_ALLOC(m->idx, E * Mx);
  MLP_ALLOC(m->y, E * Mx * DOUT);
  MLP_ALLOC(m->acts, E * 5 * H * Mx);
  MLP_ALLOC(m->slopes, E * 4 * H * Mx);
  MLP_ALLOC(m->grads, E * 5 * H * Mx);
  MLP_ALLOC(m->part, E * S * P);
  MLP_ALLOC(m->loss_part, E * (Mx / NLOSS));
  MLP_ALLOC(m->gbuf, E * P);
  MLP_ALLOC(m->step, 1);
  MLP_ALLOC(m->uni, 3);
  MLP_ALLOC(m->bad, 1);
#undef MLP_ALLOC
  hipError_t e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
  if (e != hipSuccess) return bail(mfail(SPK_ERR_HIP, "hipStreamCreate failed"));
  for (auto& ev : m->ev)
    if (hipEventCreate(&ev) != hipSuccess) return bail(mfail(SPK_ERR_HIP, "hipEventCreate failed"));
  if (hipMemset(m->master, 0, E * P * sizeof(float)) != hipSuccess ||
      hipMemset(m->wb, 0, E * BF * sizeof(uint16_t)) != hipSuccess)
    return bail(mfail(SPK_ERR_HIP, "hipMemset failed"));
  if ((rc = spk_mlp_reset_optimizer(m))) return bail(rc);
  *out = m;
  return SPK_OK;
}

int spk_mlp_destroy(spk_mlp* m) {
  if (!m) return SPK_OK;
  if (m->stream) (void)hipStreamSynchronize(m->stream);
  if (m->graph) (void)hipGraphExecDestroy(m->graph);
  free_d(m->master); free_d(m->mom); free_d(m->vel); free_d(m->wb);
  free_d(m->x); free_d(m->t); free_d(m->idx); free_d(m->y);
  free_d(m->acts); free_d(m->slopes); free_d(m->grads);
  free_d(m->part); free_d(m->loss_part); free_d(m->gbuf); free_d(m->gin); free_d(m->step); free_d(m->uni); free_d(m->bad);
  free_d(m->px); free_d(m->py);
  for (auto& ev : m->ev)
    if (ev) (void)hipEventDestroy(ev);
  for (auto& ev : m->piece)
    if (ev) (void)hipEventDestroy(ev);
  if (m->copy) (void)hipStreamDestroy(m->copy);
  if (m->stream) (void)hipStreamDestroy(m->stream);
  delete m;
  return SPK_OK;
}

int spk_mlp_reset_optimizer(spk_mlp* m) {
  if (!m) return mfail(SPK_ERR_ARG, "null handle");
  MLP_HIP(hipMemsetAsync(m->mom, 0, (size_t)m->E * P * sizeof(float), m->stream));
  MLP_HIP(hipMemsetAsync(m->vel, 0, (size_t)m->E * P * sizeof(float), m->stream));
  MLP_HIP(hipMemsetAsync(m->step, 0, sizeof(int), m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  return SPK_OK;
}

int spk_mlp_set_params(spk_mlp* m, const float* params) {
  if (!m || !params) return mfail(SPK_ERR_ARG, "null argument");
  // checked on the device before they take the place of the current ones (a pass over the
  // 1.6e6 parameters of 8 members takes 1 ms on the host, where they are checked without memory
  // for a copy)
  const size_t cnt = (size_t)m->E * P;
  size_t bad = cnt;
  if (m->gin || malloc_d(&m->gin, cnt) == SPK_OK) {
    MLP_HIP(hipMemcpyAsync(m->gin, params, cnt * sizeof(float), hipMemcpyHostToDevice, m->stream));
    MLP_HIP(hipMemsetAsync(m->bad, 0xFF, sizeof(unsigned int), m->stream));
    hipLaunchKernelGGL(k_mlp_check, dim3(512), dim3(256), 0, m->stream, m->gin, (unsigned int)cnt, m->bad);
    MLP_HIP(hipGetLastError());
    unsigned int first = 0;
    MLP_HIP(hipMemcpyAsync(&first, m->bad, sizeof(first), hipMemcpyDeviceToHost, m->stream));
    MLP_HIP(hipStreamSynchronize(m->stream));
    bad = std::min<size_t>(first, cnt);
  } else {
    for (size_t i = cnt; i-- > 0;)
      if (!std::isfinite(params[i])) bad = i;
  }
  if (bad < cnt) return mfail(SPK_ERR_ARG, "non-finite parameter at " + std::to_string(bad));
  if (m->gin) MLP_HIP(hipMemcpyAsync(m->master, m->gin, cnt * sizeof(float), hipMemcpyDeviceToDevice, m->stream));
  else MLP_HIP(hipMemcpyAsync(m->master, params, cnt * sizeof(float), hipMemcpyHostToDevice, m->stream));
  // padding entries of the working copies stay zero from creation; every used entry is rewritten
  AdamArgs ad{};
  ad.master = m->master; ad.wb = m->wb; ad.apply = 2;
  hipLaunchKernelGGL(k_mlp_adam, dim3(kAdamBlocks, m->E), dim3(256), 0, m->stream, ad);
  MLP_HIP(hipGetLastError());
  return spk_mlp_reset_optimizer(m);
}

int spk_mlp_get_params(spk_mlp* m, float* params) {
  if (!m || !params) return mfail(SPK_ERR_ARG, "null argument");
  MLP_HIP(hipMemcpyAsync(params, m->master, (size_t)m->E * P * sizeof(float), hipMemcpyDeviceToHost, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  return SPK_OK;
}

int spk_mlp_set_data(spk_mlp* m, const float* features, const float* targets, int64_t n) {
  if (!m || !features || !targets || n < 1 || n > ((int64_t)1 << 31) - 1)
    return mfail(SPK_ERR_ARG, "bad training set");
  MLP_HIP(hipStreamSynchronize(m->stream));
  drop_graph(m);
  if (n > m->cap) {
    MLP_HIP(hipStreamSynchronize(m->stream));
    free_d(m->x);
    free_d(m->t);
    m->cap = m->n = 0;   // no training set while there is no memory for one
    int rc;
    if ((rc = malloc_d(&m->x, (size_t)n * DIN)) || (rc = malloc_d(&m->t, (size_t)n * DOUT))) {
      free_d(m->x);
      return rc;
    }
    m->cap = n;
  }
  MLP_HIP(hipMemcpyAsync(m->x, features, (size_t)n * DIN * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLP_HIP(hipMemcpyAsync(m->t, targets, (size_t)n * DOUT * sizeof(float), hipMemcpyHostToDevice, m->stream));
  MLP_HIP(hipStreamSynchronize(m->stream));
  m->n = n;
  return SPK_OK;
}

int spk_mlp_set_loss_weights(spk_mlp* m, const float* w3) {
  if (!m || !w3) return mfail(SPK_ERR_ARG, "null argument");
  for (int i = 0; i < 3; ++i) {
    if (!(w3[i] >= 0.0f) || !std::isfinite(w3[i])) return mfail(SPK_ERR_ARG, "loss weights must be finite and >= 0");
  }
  MLP_HIP(hipStreamSynchronize(m->stream));
  drop_graph(m);
  for (int i = 0; i < 3; ++i) m->wout[i] = w3[i];
  return SPK_OK;
}

int spk_mlp_gradients(spk_mlp* m, int rows, float* grads, float* loss) {
  if (!m) return mfail(SPK_ERR_ARG, "null handle");
  int rc = check_batch(m, rows);
  if (rc) return rc;
  if (rows > m->n) return mfail(SPK_ERR_ARG, "rows exceed the training set");
  if ((rc = enqueue_step(m, rows, 0, 0, 0, 0.0f, 0.0f, 1, m->gbuf, m->loss_part, true))) return rc;
  MLP_HIP(hipStreamSynchronize(m->stream));
  if (grads) MLP_HIP(hipMemcpy(grads, m->gbuf, (size_t)m->E * P * sizeof(float), hipMemcpyDeviceToHost));
  if (loss) {
    const int tiles = rows / NLOSS;
    std::vector<float> lp((size_t)m->E * tiles);
    MLP_HIP(hipMemcpy(lp.data(), m->loss_part, lp.size() * sizeof(float), hipMemcpyDeviceToHost));
    for (int e = 0; e < m->E; ++e) {
      double s = 0.0;
      for (int k = 0; k < tiles; ++k) s += lp[(size_t)e * tiles + k];
      loss[e] = (float)(s / rows);
    }
  }
  m->timing = spk_mlp_timing{elapsed(m->ev[0], m->ev[4]), elapsed(m->ev[0], m->ev[1]), elapsed(m->ev[1], m->ev[2]),
                             elapsed(m->ev[2], m->ev[3]), elapsed(m->ev[3], m->ev[4]), 0, rows};
  return SPK_OK;
}

int spk_mlp_apply_gradients(spk_mlp* m, const float* grads, float lr) {
  if (!m || !grads) return mfail(SPK_ERR_ARG, "null argument");
  if (!(lr >= 0.0f) || !std::isfinite(lr)) return mfail(SPK_ERR_ARG, "bad learning rate");
  int rc;
  if (!m->gin && (rc = malloc_d(&m->gin, (size_t)m->E * P))) return rc;
  MLP_HIP(hipMemcpyAsync(m->gin, grads, (size_t)m->E * P * sizeof(float), hipMemcpyHostToDevice, m->stream));
  hipLaunchKernelGGL(k_mlp_tick, dim3(1), dim3(64), 0, m->stream, m->step, lr, m->uni);
  AdamArgs ad{};
  ad.master = m->master; ad.mom = m->mom; ad.vel = m->vel; ad.wb = m->wb; ad.gin = m->gin; ad.uni = m->uni; ad.apply = 1;
  hipLaunchKernelGGL(k_mlp_adam, dim3(kAdamBlocks, m->E), dim3(256), 0, m->stream, ad);
  MLP_HIP(hipGetLastError());
  MLP_HIP(hipStreamSynchronize(m->stream));
  return SPK_OK;
}

int spk_mlp_train(spk_mlp* m, int steps, int batch, int mode, uint64_t seed, float lr0, float lr_min,
                  int total_steps, int use_graph, float* loss_per_step) {
  if (!m) return mfail(SPK_ERR_ARG, "null handle");
  int rc = check_batch(m, batch);
  if (rc) return rc;
  if (steps < 0 || total_steps < 1) return mfail(SPK_ERR_ARG, "steps must be >= 0, total_steps >= 1");
  if (mode != SPK_MLP_BATCH_FIRST_ROWS && mode != SPK_MLP_BATCH_SAMPLED) return mfail(SPK_ERR_ARG, "bad mode");
  if (m->n < 1 || (mode == SPK_MLP_BATCH_FIRST_ROWS && batch > m->n))
    return mfail(SPK_ERR_STATE, "training set missing or smaller than the batch");
  if (!(lr0 >= 0.0f) || !(lr_min >= 0.0f) || !std::isfinite(lr0) || !std::isfinite(lr_min))
    return mfail(SPK_ERR_ARG, "bad learning rate");
  const int tiles = batch / NLOSS;
  float* lhist = nullptr;
  if (loss_per_step && steps > 0 && (rc = malloc_d(&lhist, (size_t)steps * m->E * tiles))) return rc;
  MLP_HIP(hipEventRecord(m->ev[5], m->stream));
  if (use_graph && !loss_per_step) {
    const bool same = m->graph && m->graph_batch == batch && m->graph_mode == mode && m->graph_seed == seed &&
                      m->graph_lr0 == lr0 && m->graph_lrmin == lr_min && m->graph_total == total_steps;
    if (!same) {
      if (m->graph) (void)hipGraphExecDestroy(m->graph);
      m->graph = nullptr;
      hipGraph_t g;
      MLP_HIP(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
      rc = enqueue_step(m, batch, mode, seed, 1, lr0, lr_min, total_steps, nullptr, m->loss_part, false);
      hipError_t ce = hipStreamEndCapture(m->stream, &g);
      if (rc) return rc;
      if (ce != hipSuccess) return mfail(SPK_ERR_HIP, "graph capture failed");
      hipError_t ie = hipGraphInstantiate(&m->graph, g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      if (ie != hipSuccess) return mfail(SPK_ERR_HIP, "graph instantiation failed");
      m->graph_batch = batch; m->graph_mode = mode; m->graph_seed = seed;
      m->graph_lr0 = lr0; m->graph_lrmin = lr_min; m->graph_total = total_steps;
    }
    for (int s = 0; s < steps; ++s) MLP_HIP(hipGraphLaunch(m->graph, m->stream));
  } else {
    for (int s = 0; s < steps; ++s) {
      float* lp = lhist ? lhist + (size_t)s * m->E * tiles : m->loss_part;
      if ((rc = enqueue_step(m, batch, mode, seed, 1, lr0, lr_min, total_steps, nullptr, lp, false))) {
        free_d(lhist);
        return rc;
      }
    }
  }
  MLP_HIP(hipEventRecord(m->ev[4], m->stream));
  hipError_t se = hipStreamSynchronize(m->stream);
  if (se != hipSuccess) {
    free_d(lhist);
    return mfail(SPK_ERR_HIP, std::string("training failed: ") + hipGetErrorString(se));
  }
  if (lhist) {
    std::vector<float> lp((size_t)steps * m->E * tiles);
    hipError_t ce = hipMemcpy(lp.data(), lhist, lp.size() * sizeof(float), hipMemcpyDeviceToHost);
    free_d(lhist);
    if (ce != hipSuccess) return mfail(SPK_ERR_HIP, "loss copy failed");
    for (int s = 0; s < steps; ++s)
      for (int e = 0; e < m->E; ++e) {
        double acc = 0.0;
        for (int k = 0; k < tiles; ++k) acc += lp[((size_t)s * m->E + e) * tiles + k];
        loss_per_step[(size_t)s * m->E + e] = (float)(acc / batch);
      }
  }
  m->timing = spk_mlp_timing{elapsed(m->ev[5], m->ev[4]), 0, 0, 0, 0, steps, batch};
  return SPK_OK;
}

int spk_mlp_predict(spk_mlp* m, const float* features, int64_t n, float* out) {
  if (!m || !features || !out || n < 1 || n > ((int64_t)1 << 28)) return mfail(SPK_ERR_ARG, "bad arguments");
  if (n > m->pcap) {
    MLP_HIP(hipStreamSynchronize(m->stream));
    free_d(m->px);
    free_d(m->py);
    m->pcap = 0;
    int rc;
    if ((rc = malloc_d(&m->px, (size_t)n * DIN)) || (rc = malloc_d(&m->py, (size_t)m->E * n * DOUT))) {
      free_d(m->px);
      return rc;
    }
    m->pcap = n;
  }
  MLP_HIP(hipMemcpyAsync(m->px, features, (size_t)n * DIN * sizeof(float), hipMemcpyHostToDevice, m->stream));
  if (int rc = infer(m, m->px, n, m->py, out, true)) return rc;
  const float ms = elapsed(m->ev[0], m->ev[1]);
  m->timing = spk_mlp_timing{ms, ms, 0, 0, 0, 0, n};
  return SPK_OK;
}

int spk_mlp_predict_noalloc(spk_mlp* m, const float* features, int64_t n, float* out) {
  if (!m || !features || !out || n < 1) return mfail(SPK_ERR_ARG, "bad arguments");
  // features at the start of the array, outputs from the next 256-byte boundary
  const int64_t xfl = (n * DIN + 63) / 64 * 64;
  const int64_t need = xfl + (int64_t)m->E * n * DOUT;
  if (n > (int64_t)kNoAllocFloats || need > (int64_t)kNoAllocFloats)
    return mfail(SPK_ERR_ARG, "spk_mlp_predict_noalloc: " + std::to_string(n) + " rows x " +
                                  std::to_string(m->E) + " members need " + std::to_string(need * 4) +
                                  " bytes of staging; the static limit is " + std::to_string(kNoAllocBytes));
  float* px = m->scratch;
  float* py = m->scratch + xfl;
  MLP_HIP(hipMemcpyAsync(px, features, (size_t)n * DIN * sizeof(float), hipMemcpyHostToDevice, m->stream));
  if (int rc = infer(m, px, n, py, out, false)) return rc;
  const float ms = elapsed(m->ev[0], m->ev[1]);
  m->timing = spk_mlp_timing{ms, ms, 0, 0, 0, 0, n};
  return SPK_OK;
}

int spk_mlp_last_timing(const spk_mlp* m, spk_mlp_timing* t) {
  if (!m || !t) return mfail(SPK_ERR_ARG, "null argument");
  *t = m->timing;
  return SPK_OK;
}

}  // extern "C"
