// Learned price surrogate: an MLP 8 -> 512 -> 512 -> 512 -> 512 -> 1 with
// SiLU, BF16 weights and activations, FP32 accumulation and FP32 master
// weights, trained with Adam by hand-written MFMA kernels (gfx950).
//
// Rows are independent through every layer, so one kernel takes a block of
// rows through the whole network with its activations in LDS: inference reads
// features and writes prices, a training step's first launch runs forward,
// loss and backward and leaves what the weight gradients need.  Then
//   dW_l = dZ_l^T A_{l-1}   (all layers in one launch, split along the batch)
//   Adam, which sums the splits and the row kernel's partial bias and head
//   gradients as it reads them.
//
// Matrix operands:
//   packed weights  fragment order of v_mfma_f32_16x16x32_bf16: a wave's 64
//                   output neurons, K step of 32, 4 blocks of 16, lane, 8
//                   elements -- a wave's K step is one contiguous 4 KB read.  W_l for the
//                   forward pass and its transpose for the backward pass are
//                   written by Adam as it updates the master weights.
//   T blocks        [row block of 64][neuron][64 rows]: activations and
//                   back-propagated gradients transposed for the weight-
//                   gradient GEMM, whose K stage of 64 rows is then contiguous;
//                   the rows of each 32 in the order t_row, in which a lane of
//                   the row kernel holds eight in a row.
// The input layer is zero-padded from 8 to 128 features in the parameter
// layout; products use the first 32.
#include "common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

typedef __bf16 bf16;
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(__bf16)))) __bf16 bf16x4;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

#define FDADI_RET(x)     \
  do {                   \
    int _st = (x);       \
    if (_st) return _st; \
  } while (0)

namespace fdadi {
namespace {

constexpr int kIn = 8;       // Heston features
constexpr int kMaxIn = 16;   // largest feature count of a network (fdadi_mlp_create_features)
constexpr int kInPad = 128;  // padded input width
constexpr int kH = 512;      // hidden width
constexpr int kLayers = 4;   // hidden layers (the 512 -> 1 head is separate)
constexpr int kTile = 128;
constexpr int kKStep = 64;   // K extent of one LDS stage of the GEMM, rows of a T block
constexpr int kMaxSplits = 8;  // split-K factor cap for the weight-gradient GEMMs
constexpr int kLdsPitch = kKStep + 8;  // bf16 elements per LDS row (16 B pad)
constexpr int kThreads = 512;          // work-groups of the GEMM and the row kernel: 8 waves
constexpr int kWN = 4;                 // GEMM: waves along N (2 along M)
constexpr int kBM = 4, kBN = 2;        // GEMM: 16 x 16 MFMA blocks per wave: 64 x 32

// Logistic sigmoid with the hardware reciprocal (about 1 ulp; every result
// that uses it is rounded to bf16).  silu(z) = z s(z), silu'(z) = s (1 + z (1 - s)).
__device__ __forceinline__ float sigmoid(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-z));
}

// ---- the network on a block of rows ----------------------------------------------
// A work-group of 8 waves holds 16 MB rows; wave w owns neurons 64 w .. +63 of
// every layer (4 blocks of 16).  The rows' activations live in LDS and are
// replaced in place, layer by layer, between two barriers.  A wave needs no
// one else's weights, so its weight operands go from L2 straight to registers:
// a ring of RING K steps in flight, running on from one layer into the next.
// MFMA operand layout (v_mfma_f32_16x16x32_bf16): lane l holds
//   A[i = l%16][k = 8*(l/16) .. +7],  B[k = 8*(l/16) .. +7][j = l%16],
//   D[i = 4*(l/16) + t][j = l%16] for t = 0..3.
// Training puts rows on i (a lane then holds four rows of a neuron: the T
// blocks' order), inference neurons on i (four neurons of a row: the next
// layer's order in LDS).
//
// What bounds it: at 32 rows the 1.6 MB of weights every work-group streams
// from L2, 64 bytes per clock and CU (12 us of a forward pass's 20, 23 us of a
// training pass's 47, the rest SiLU and the T blocks' 59 MB); from 64 rows on
// the matrix cores and the SiLU's exponentials (200,000 rows in 355 us: 0.9
// PFLOP/s).  A launch per layer and its activations through memory took 14 us
// per layer forward and 20 us back at 8,192 rows, 56 us for a prediction.
constexpr int kActPitch = kH + 8;  // bf16 elements per LDS row of activations
constexpr int kKSteps = kH / 32;   // K steps of a hidden layer
constexpr int kPart = 5 * kH + 4;  // floats of a work-group's partial sums
constexpr int kPackH = kH * kH, kPackIn = kH * 32;  // elements of a packed matrix

// Element (n, k) of a packed matrix with KS steps of K.
__device__ __forceinline__ int64_t packed_at(int n, int k, int KS) {
  return ((((int64_t)(n / 64) * KS + k / 32) * 4 + n / 16 % 4) * 64 + n % 16 + 16 * (k % 32 / 8)) *
             8 + k % 8;
}

struct RowArgs {
  const double *P, *T;  // features, targets
  const int *idx;       // training: rows of P and T (null: in order)
  int64_t rows;         // valid rows
  int nin;
  const double *lo, *hi;
  double tmean, tstd;
  const bf16 *Wp[2 * kLayers - 1];  // packed W_0 .. W_3, then W_3^T, W_2^T, W_1^T
  const float *bias[kLayers];
  const bf16 *w4;
  const float *b4;
  double *out;                        // inference: prices
  // training: T blocks (XT: of kInPad features), and per work-group kPart
  // floats: sums over its rows of dZ_0 .. dZ_3, of the head's weight gradient
  // and of its bias gradient and the loss
  bf16 *XT, *ActT[kLayers - 1], *dZT[kLayers];
  float *gpart;
};

// Place of row r of 32 in a T block: rows 16 a + 4 q + t (a lane's MFMA results,
// q its quarter) at 8 q + 4 a + t.
__device__ __forceinline__ int t_row(int r) { return r / 4 % 4 * 8 + r / 16 * 4 + r % 4; }

// x_f = 2 (p_f - lo_f) / (hi_f - lo_f) - 1 for the nin features of a row, 0
// for the padding.
__device__ __forceinline__ bf16 input_value(const RowArgs &a, int64_t r, int f) {
  float v = 0.f;
  if (r < a.rows && f < a.nin) {
    const int64_t src = a.idx ? a.idx[r] : r;
    v = (float)(2.0 * (a.P[src * a.nin + f] - a.lo[f]) / (a.hi[f] - a.lo[f]) - 1.0);
  }
  return static_cast<bf16>(v);
}

template <int MB, int RING, int WAVES, bool TRAIN>
__global__ void __launch_bounds__(kThreads, WAVES) mlp_rows_kernel(RowArgs a) {
  constexpr int M = 16 * MB;
  __shared__ __attribute__((aligned(16))) bf16 act[M * kActPitch];
  __shared__ float gs[M], es[M];
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int64_t row0 = (int64_t)blockIdx.x * M;
  const int lr = lane % 16, lq = lane / 16;  // lane's row / column and quarter of a block
  const int n0 = wave * 64;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);  // scalar: weights have scalar bases
  // this lane's place in a T block: neuron n0 + 16 b + lr, its eight rows
  const int64_t tblk =
      row0 / kKStep * (kH * kKStep) + (int64_t)(n0 + lr) * kKStep + row0 % kKStep + 8 * lq;
  float *const gpart = TRAIN ? a.gpart + (int64_t)blockIdx.x * kPart : nullptr;

  bf16x8 ring[RING][4];
  const uint32_t lane_off = lane * 16;
  auto load_w = [&](bf16x8 *w, const bf16 *Wp, int KS, int ks) {
    const char *base = reinterpret_cast<const char *>(Wp) + (wave_u * KS + ks) * 4096;
#pragma unroll
    for (int b = 0; b < 4; ++b)
      w[b] = *reinterpret_cast<const bf16x8 *>(base + 1024 * b + lane_off);
  };
  float bn[4][TRAIN ? 1 : 4];  // biases of this lane's neurons
  auto load_bias = [&](const float *bias) {
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if constexpr (TRAIN) {
        bn[b][0] = bias[n0 + 16 * b + lr];
      } else {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(bias + n0 + 16 * b + 4 * lq);
#pragma unroll
        for (int t = 0; t < 4; ++t) bn[b][t] = v[t];
      }
    }
  };
  bf16x8 w0[4];
  load_w(w0, a.Wp[0], 1, 0);
  load_bias(a.bias[0]);
#pragma unroll
  for (int j = 0; j < RING; ++j) load_w(ring[j], a.Wp[1], kKSteps, j);

  // the input rows, 32 columns
#pragma unroll
  for (int e = tid; e < M * 32; e += kThreads) {
    const int f = e / M, r = e % M;
    const bf16 v = input_value(a, row0 + r, f);
    act[r * kActPitch + f] = v;
    if (TRAIN && f < a.nin)
      a.XT[(row0 / kKStep * kInPad + f) * kKStep + row0 % kKStep + t_row(r)] = v;
  }
  __syncthreads();

  f32x4 acc[MB][4];
  auto zero_acc = [&]() {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b) acc[i][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto load_a = [&](bf16x8 *af, int ks) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
      af[i] = *reinterpret_cast<const bf16x8 *>(act + (16 * i + lr) * kActPitch + 32 * ks + 8 * lq);
  };
  auto k_step = [&](const bf16x8 *w, const bf16x8 *af) {
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int b = 0; b < 4; ++b)
        acc[i][b] = TRAIN ? __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i], w[b], acc[i][b], 0, 0, 0)
                          : __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[b], af[i], acc[i][b], 0, 0, 0);
  };
  // One 512 x 512 product, whose first K steps are in the ring; leaves those of
  // the product after it there.  The scheduler would sink each load to its use
  // (and did: 58 us instead of 47 for a training batch of 8,192): nothing moves across
  // the end of a K step.
  auto product = [&](const bf16 *Wp, const bf16 *next, const float *bias) {
    zero_acc();
    if (bias) load_bias(bias);  // ahead of the loads it would otherwise wait for
    bf16x8 af[2][MB];
    load_a(af[0], 0);
#pragma unroll 1
    for (int ks = 0; ks < kKSteps; ks += RING) {
      const bool here = ks + RING < kKSteps;
      const bf16 *src = here ? Wp : next;
      const int base = here ? ks + RING : 0;
#pragma unroll
      for (int j = 0; j < RING; ++j) {
        load_a(af[(j + 1) % 2], (ks + j + 1) % kKSteps);
        k_step(ring[j], af[j % 2]);
        load_w(ring[j], src, kKSteps, base + j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // silu' at the pre-activations, each thread its own elements (in LDS: 64
  // registers more would spill); the last layer's are used at once
  __shared__ bf16x4 dsilu[TRAIN ? kLayers - 1 : 1][TRAIN ? MB * 4 : 1][TRAIN ? kThreads : 1];
  bf16x4 dlast[TRAIN ? MB : 1][4], olast[TRAIN ? MB : 1][4];  // and the activations
  // bias + SiLU of layer l into LDS (every wave is done reading it)
  auto activate = [&](auto lc) {
    constexpr int l = decltype(lc)::value;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if constexpr (TRAIN) {
        bf16x8 o;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          bf16x4 d;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float z = acc[i][b][t] + bn[b][0], sg = sigmoid(z);
            o[4 * i + t] = static_cast<bf16>(z * sg);
            d[t] = static_cast<bf16>(sg * (1.0f + z * (1.0f - sg)));
            act[(16 * i + 4 * lq + t) * kActPitch + n0 + 16 * b + lr] = o[4 * i + t];
            if constexpr (l == kLayers - 1) olast[i][b][t] = o[4 * i + t];
          }
          if constexpr (l == kLayers - 1) dlast[i][b] = d;
          else dsilu[l][4 * i + b][tid] = d;
        }
        if constexpr (l < kLayers - 1)
          *reinterpret_cast<bf16x8 *>(a.ActT[l] + tblk + 16 * b * kKStep) = o;
      } else {
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          bf16x4 o;
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const float z = acc[i][b][t] + bn[b][t];
            o[t] = static_cast<bf16>(z * sigmoid(z));
          }
          *reinterpret_cast<bf16x4 *>(act + (16 * i + lr) * kActPitch + n0 + 16 * b + 4 * lq) = o;
        }
      }
    }
    __syncthreads();
  };
  zero_acc();
  bf16x8 a0[MB];
  load_a(a0, 0);
  k_step(w0, a0);
  activate(std::integral_constant<int, 0>{});
  product(a.Wp[1], a.Wp[2], a.bias[1]);
  activate(std::integral_constant<int, 1>{});
  product(a.Wp[2], a.Wp[3], a.bias[2]);
  activate(std::integral_constant<int, 2>{});
  product(a.Wp[3], a.Wp[TRAIN ? 4 : 3], a.bias[3]);
  activate(std::integral_constant<int, 3>{});

  if constexpr (!TRAIN) {
    // head: y = sum_n A[r, n] w[n] + b, one wave per row, fp32
#pragma unroll
    for (int rr = 0; rr < M / 8; ++rr) {
      const int r = wave * (M / 8) + rr;
      float y = 0.f;
#pragma unroll
      for (int q = 0; q < kH / 64; ++q)
        y += (float)act[r * kActPitch + lane + 64 * q] * (float)a.w4[lane + 64 * q];
      for (int d = 32; d > 0; d >>= 1) y += __shfl_down(y, d, 64);
      if (lane == 0 && row0 + r < a.rows) {
        const float v = y + a.b4[0];
        a.out[row0 + r] = (double)v * a.tstd + a.tmean;
      }
    }
  } else {
    // head and loss gradient: sixteen threads per row, 32 columns each, summed
    // in groups of four and then in order
    static_assert(M * 16 == kThreads && MB == 2, "sixteen threads per row, T blocks of 32");
    const int r = tid / 16, h = (tid % 16) * 32;
    float y = 0.f;
#pragma unroll
    for (int c = 0; c < 32; c += 8) {
      const bf16x8 av = *reinterpret_cast<const bf16x8 *>(act + r * kActPitch + h + c);
      const bf16x8 wv = *reinterpret_cast<const bf16x8 *>(a.w4 + h + c);
#pragma unroll
      for (int t = 0; t < 8; ++t) y += (float)av[t] * (float)wv[t];
    }
    y += __shfl_xor(y, 1, 64);
    y += __shfl_xor(y, 2, 64);
    float sum = a.b4[0];
#pragma unroll
    for (int j = 0; j < 4; ++j) sum += __shfl(y, (lane & ~15) + 4 * j, 64);
    if (tid % 16 == 0) {
      float g = 0.f, e2 = 0.f;
      if (row0 + r < a.rows) {
        const int64_t src = a.idx ? a.idx[row0 + r] : row0 + r;
        const float t = (float)((a.T[src] - a.tmean) / a.tstd);
        const float e = sum - t;
        g = 2.f * e / (float)a.rows;
        e2 = e * e / (float)a.rows;
      }
      gs[r] = g;
      es[r] = e2;
    }
    __syncthreads();
    if (lane == 0 && wave < 2) {
      const float *v = wave == 0 ? gs : es;
      float sum = 0.f;
      for (int k = 0; k < M; ++k) sum += v[k];
      gpart[5 * kH + wave] = sum;
    }
    // sum over the work-group's rows of neuron n0 + 16 b + lr
    auto put_sum = [&](int which, int b, float v) {
      v += __shfl_xor(v, 16, 64);
      v += __shfl_xor(v, 32, 64);
      if (lq == 0) gpart[which * kH + n0 + 16 * b + lr] = v;
    };
    // dZ of layer l into LDS, its T block and its sums
    auto put_dz = [&](int l, int b, bf16x8 v) {
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          act[(16 * i + 4 * lq + t) * kActPitch + n0 + 16 * b + lr] = v[4 * i + t];
          sum += (float)v[4 * i + t];
        }
      *reinterpret_cast<bf16x8 *>(a.dZT[l] + tblk + 16 * b * kKStep) = v;
      put_sum(l, b, sum);
    };
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float wn = (float)a.w4[n0 + 16 * b + lr];
      bf16x8 v;
      float gw = 0.f;
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const float g = gs[16 * i + 4 * lq + t];
          v[4 * i + t] = static_cast<bf16>(g * wn * (float)dlast[i][b][t]);
          gw += g * (float)olast[i][b][t];
        }
      put_sum(4, b, gw);
      put_dz(3, b, v);
    }
    // dZ_{l-1} = (dZ_l W_l) * silu'(Z_{l-1})
    auto back = [&](auto lc) {
      constexpr int l = decltype(lc)::value;
      __syncthreads();
      product(a.Wp[kLayers + 3 - l], a.Wp[l > 1 ? kLayers + 4 - l : kLayers + 3 - l], nullptr);
      __syncthreads();
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        bf16x8 v;
#pragma unroll
        for (int i = 0; i < MB; ++i) {
          const bf16x4 d = dsilu[l - 1][4 * i + b][tid];
#pragma unroll
          for (int t = 0; t < 4; ++t)
            v[4 * i + t] = static_cast<bf16>(acc[i][b][t] * (float)d[t]);
        }
        put_dz(l - 1, b, v);
      }
    };
    back(std::integral_constant<int, 3>{});
    back(std::integral_constant<int, 2>{});
    back(std::integral_constant<int, 1>{});
  }
}

// ---- GEMM ------------------------------------------------------------------------
// C[m,n] = sum_k A[m,k] B[n,k] (fp32) on MFMA 16x16x32 bf16.  512 threads = 8
// waves in a 2 x 4 grid, each wave owns a 64 x 32 sub-tile = 4 x 2 MFMA blocks;
// two waves per SIMD hide each other's LDS and barrier latency.  The K loop
// stages 128 x 64 tiles of A and B in LDS (two 32-deep MFMA steps per stage).
// An operand's rows are ld elements apart within a stage and its stages st
// apart: (K, 64) for a row-major matrix, (64, 64 x rows) for T blocks.
// The loads of a K stage must be in flight long before it: a ring of kDepth
// register stages keeps the next stage's global loads outstanding while the
// MFMAs of the current one run.  The K extent of a work-group is a multiple of
// kDepth stages, so the ring needs no remainder code.
constexpr int kDepth = 2;
constexpr int kKBlock = kKStep * kDepth;  // K granularity of the GEMM
constexpr int kChunks = kTile * kKStep / 8 / kThreads;  // 16-byte loads per operand per stage
constexpr int kLoopLds = 4 * kTile * kLdsPitch;  // two A and two B stages

// One GEMM of a launch: operands, sizes and its tile grid (gx x gy output
// tiles, gz splits of K; split z writes its partial product to slice z of C).
struct GemmArgs {
  const bf16 *A, *B;
  int64_t ldA, stA, ldB, stB;
  int M, N, K, gx, gy, gz;
  float *C;
};

// The work of work-group `Lin` (linear index within its GEMM's grid).
__device__ __forceinline__ void gemm_tile(bf16 *smem, const GemmArgs &g, int Lin) {
  const int M = g.M, N = g.N, K = g.K;
  // Two LDS stages: the MFMAs of stage s read buffer s % 2 while stage s + 1
  // is written to the other one, so one barrier per stage suffices.
  bf16 *const As[2] = {smem, smem + kTile * kLdsPitch};
  bf16 *const Bs[2] = {smem + 2 * kTile * kLdsPitch, smem + 3 * kTile * kLdsPitch};
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int wm = wave / kWN, wn = wave % kWN;
  // Work-groups are dealt to the 8 XCDs round-robin by linear id; renumber
  // them so that each XCD gets a contiguous run of tiles (x fastest): the
  // N tiles of one row block of A, and of one split, then share that XCD's L2.
  const int gx = g.gx, gy = g.gy, total = gx * gy * g.gz;
  int L = Lin;
  if (total % 8 == 0) L = (L % 8) * (total / 8) + L / 8;
  const int bx = L % gx, by = (L / gx) % gy, bz = L / (gx * gy);
  const int m0 = by * kTile, n0 = bx * kTile;
  // split-K: work-group z covers K columns [z*Ks, (z+1)*Ks) (gz = 1: all)
  const int Ks = K / g.gz, kbeg = bz * Ks, nsteps = Ks / kKStep;
  f32x4 acc[kBM][kBN];
#pragma unroll
  for (int a = 0; a < kBM; ++a)
#pragma unroll
    for (int b = 0; b < kBN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // Global -> registers -> LDS: chunk q = tid + kThreads * p of a 128 x 64
  // tile is row q / 8, elements 8 (q % 8) .. +7.
  const int lrow = tid / (kKStep / 8), lk = (tid % (kKStep / 8)) * 8;
  constexpr int kRowStep = kThreads / (kKStep / 8);  // rows between a thread's chunks
  const bf16 *Ag = g.A + (m0 + lrow) * g.ldA + kbeg / kKStep * g.stA + lk;
  const bf16 *Bg = g.B + (n0 + lrow) * g.ldB + kbeg / kKStep * g.stB + lk;
  bf16x8 ra[kDepth][kChunks], rb[kDepth][kChunks];
  auto fetch = [&](bf16x8 *xa, bf16x8 *xb, int step) {
#pragma unroll
    for (int p = 0; p < kChunks; ++p) {
      xa[p] = *reinterpret_cast<const bf16x8 *>(Ag + kRowStep * p * g.ldA + step * g.stA);
      xb[p] = *reinterpret_cast<const bf16x8 *>(Bg + kRowStep * p * g.ldB + step * g.stB);
    }
  };
  auto stage = [&](const bf16x8 *xa, const bf16x8 *xb, int buf) {
#pragma unroll
    for (int p = 0; p < kChunks; ++p) {
      const int r = lrow + kRowStep * p;
      *reinterpret_cast<bf16x8 *>(As[buf] + r * kLdsPitch + lk) = xa[p];
      *reinterpret_cast<bf16x8 *>(Bs[buf] + r * kLdsPitch + lk) = xb[p];
    }
  };
  auto compute = [&](int buf) {
#pragma unroll
    for (int kk = 0; kk < kKStep; kk += 32) {
      bf16x8 af[kBM], bfr[kBN];
      const int kseg = kk + (lane / 16) * 8;
#pragma unroll
      for (int a = 0; a < kBM; ++a) {
        const int row = wm * kBM * 16 + a * 16 + lane % 16;
        af[a] = *reinterpret_cast<const bf16x8 *>(As[buf] + row * kLdsPitch + kseg);
      }
#pragma unroll
      for (int b = 0; b < kBN; ++b) {
        const int col = wn * kBN * 16 + b * 16 + lane % 16;
        bfr[b] = *reinterpret_cast<const bf16x8 *>(Bs[buf] + col * kLdsPitch + kseg);
      }
#pragma unroll
      for (int a = 0; a < kBM; ++a)
#pragma unroll
        for (int b = 0; b < kBN; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[a], bfr[b], acc[a][b], 0, 0, 0);
    }
  };
#pragma unroll
  for (int j = 0; j < kDepth; ++j) fetch(ra[j], rb[j], j);
  stage(ra[0], rb[0], 0);
  __syncthreads();
  // Stage s computes from LDS buffer s % 2; its registers (ring slot s %
  // kDepth) were staged one stage earlier and now take stage s + kDepth.
  // The loop body is free of branches (past the end the loads repeat the
  // last stage and the store to LDS is never read), so the compiler's wait
  // counts keep the next stage's loads in flight.
  for (int s0 = 0; s0 < nsteps; s0 += kDepth) {
#pragma unroll
    for (int j = 0; j < kDepth; ++j) {
      const int st = s0 + j;
      fetch(ra[j], rb[j], min(st + kDepth, nsteps - 1));
      compute(j & 1);
      stage(ra[(j + 1) % kDepth], rb[(j + 1) % kDepth], (j + 1) & 1);
      __syncthreads();
    }
  }
  // Lane l of wave (wm, wn) holds, for MFMA block (a, b), rows
  // wm*64 + a*16 + 4*(l/16) + t (t = 0..3) of column wn*32 + b*16 + l%16.
  float *Cz = g.C + (size_t)bz * M * N;
#pragma unroll
  for (int a = 0; a < kBM; ++a)
#pragma unroll
    for (int b = 0; b < kBN; ++b) {
      const int n = n0 + wn * kBN * 16 + b * 16 + lane % 16;
      const int mb = m0 + wm * kBM * 16 + a * 16 + 4 * (lane / 16);
#pragma unroll
      for (int t = 0; t < 4; ++t) Cz[(size_t)(mb + t) * N + n] = acc[a][b][t];
    }
}

__global__ void __launch_bounds__(kThreads) gemm_nt_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) bf16 smem[kLoopLds];
  gemm_tile(smem, g, blockIdx.x + g.gx * (blockIdx.y + g.gy * blockIdx.z));
}

// The weight gradients of every layer in one launch, the last layer's first:
// work-groups [first[j], first[j + 1]) belong to GEMM j.  A layer alone is 16
// tiles, which took 16 splits to give each CU one work-group (20 us a layer, and
// a pass over 16 partial matrices); all layers fill the chip with 8 (24 us in
// all at 8,192 rows: 14 GFLOP at 0.58 PFLOP/s, half of what a large product
// reaches, with 416 work-groups on 256 CUs, 160 of which hold two, 218 MB of
// operands loaded and 27 MB of partials written).
struct WGradArgs {
  GemmArgs g[kLayers];
  int first[kLayers];
};
__global__ void __launch_bounds__(kThreads) wgrad_kernel(WGradArgs w) {
  __shared__ __attribute__((aligned(16))) bf16 smem[kLoopLds];
  const int k = blockIdx.x;
  const int j = k >= w.first[3] ? 3 : k >= w.first[2] ? 2 : k >= w.first[1] ? 1 : 0;
  gemm_tile(smem, w.g[j], k - w.first[j]);
}

// ---- parameters --------------------------------------------------------------------
// Layout of the flat arrays: W_0 [kH x kInPad], b_0 [kH], W_1, b_1, .., w_4
// [kH], b_4 [1]; every block but the last starts at a multiple of four.
static_assert(kInPad == (1 << 7) && kH == (1 << 9), "weights are indexed by shifts");
struct ParamMap {
  int64_t off[kLayers];  // start of W_0..W_3
  bf16 *Wp[kLayers], *WpT[kLayers], *w4b;
};

// What a parameter update does: complete the gradients, also take an Adam step
// and refresh the bf16 copies, or only refresh the copies.
enum UpdateMode { UPDATE_GRAD, UPDATE_ADAM, UPDATE_COPIES };

// Work-groups [0, kWeightBlocks): 8 rows x 128 columns of one W_l, four weights
// per thread; their gradient is the sum of the split-K partials part[split][..]
// in split order (one split: the GEMM wrote g itself).  The tile's bf16 copies
// go through LDS, so that both packed matrices are written 16 bytes at a time
// (the transposed one element by element: 18.8 us a step instead of 10.6).
// Then kSumBlocks work-groups for what the row kernel left as sums per
// work-group: 8 of 64 neurons for each bias and the head's weights, one for the
// head's bias and the loss.  Bound by the traffic of partials and moments.
struct UpdateArgs {
  float *p, *g, *m, *v;
  const float *part[kLayers];  // partial sums of W_l, the layer's size apart
  int splits;
  const float *gpart;
  int nsum;  // work-groups of the row kernel
  float *loss;
  int64_t off_sum[6];  // b_0 .. b_3, w_4, b_4
  float lr, b1, b2, eps, c1, c2;
  ParamMap pm;
};
constexpr int kWeightBlocks = kH / 8 + (kLayers - 1) * (kH / 8) * (kH / kTile);
constexpr int kSumBlocks = 5 * 8 + 1;

// New value of a parameter; m and v are updated.
__device__ __forceinline__ float adam(const UpdateArgs &a, float p, float g, float &m, float &v) {
  m = a.b1 * m + (1.f - a.b1) * g;
  v = a.b2 * v + (1.f - a.b2) * g * g;
  return p - a.lr * (m / a.c1) / (sqrtf(v / a.c2) + a.eps);
}

// Parameters i .. i + 3 (i a multiple of four) with gradient g.
template <int MODE>
__device__ __forceinline__ f32x4 update4(const UpdateArgs &a, int64_t i, f32x4 g, bool write_g) {
  f32x4 p = *reinterpret_cast<const f32x4 *>(a.p + i);
  if (MODE != UPDATE_COPIES && write_g) *reinterpret_cast<f32x4 *>(a.g + i) = g;
  if (MODE == UPDATE_ADAM) {
    f32x4 m = *reinterpret_cast<const f32x4 *>(a.m + i);
    f32x4 v = *reinterpret_cast<const f32x4 *>(a.v + i);
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      float mt = m[t], vt = v[t];
      p[t] = adam(a, p[t], g[t], mt, vt);
      m[t] = mt;
      v[t] = vt;
    }
    *reinterpret_cast<f32x4 *>(a.m + i) = m;
    *reinterpret_cast<f32x4 *>(a.v + i) = v;
    *reinterpret_cast<f32x4 *>(a.p + i) = p;
  }
  return p;
}

template <int MODE>
__global__ void __launch_bounds__(256) update_kernel(UpdateArgs a) {
  const int tid = threadIdx.x;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if ((int)blockIdx.x < kWeightBlocks) {
    __shared__ __attribute__((aligned(16))) bf16 tile[8][kTile + 8];
    const int h = (int)blockIdx.x - kH / 8;  // among the hidden layers' tiles
    const int per = (kH / 8) * (kH / kTile);
    const int l = h < 0 ? 0 : 1 + h / per, k = h < 0 ? (int)blockIdx.x : h % per;
    const int lg = l == 0 ? 7 : 9;
    const int o0 = (l == 0 ? k : k / (kH / kTile)) * 8, c0 = l == 0 ? 0 : k % (kH / kTile) * kTile;
    const int o = o0 + tid / 32, c = c0 + tid % 32 * 4;
    const int64_t e = ((int64_t)o << lg) + c, i = a.pm.off[l] + e, nw = (int64_t)kH << lg;
    if (MODE != UPDATE_COPIES) {
      if (a.splits > 1) {
        const float *part = a.part[l] + e;
#pragma unroll 8
        for (int z = 0; z < a.splits; ++z) acc += *reinterpret_cast<const f32x4 *>(part + z * nw);
      } else {
        acc = *reinterpret_cast<const f32x4 *>(a.g + i);
      }
    }
    const f32x4 p = update4<MODE>(a, i, acc, a.splits > 1);
    if (MODE == UPDATE_GRAD) return;
    bf16x4 b;
#pragma unroll
    for (int t = 0; t < 4; ++t) b[t] = static_cast<bf16>(p[t]);
    *reinterpret_cast<bf16x4 *>(&tile[tid / 32][tid % 32 * 4]) = b;
    __syncthreads();
    if (tid < 128) {  // 16 groups of 8 columns x 8 rows, rows fastest
      const int row = tid % 8, col = tid / 8 * 8;
      if (l > 0 || col < 32)  // layer 0: the columns beyond are padding
        *reinterpret_cast<bf16x8 *>(a.pm.Wp[l] +
                                    packed_at(o0 + row, c0 + col, l == 0 ? 1 : kKSteps)) =
            *reinterpret_cast<const bf16x8 *>(&tile[row][col]);
    } else if (l > 0) {  // a column's 8 rows
      bf16x8 w;
#pragma unroll
      for (int t = 0; t < 8; ++t) w[t] = tile[t][tid - 128];
      *reinterpret_cast<bf16x8 *>(a.pm.WpT[l] + packed_at(c0 + tid - 128, o0, kKSteps)) = w;
    }
    return;
  }
  const int blk = (int)blockIdx.x - kWeightBlocks, which = blk / 8;
  if (which < 5) {
    __shared__ f32x4 red[16][16];
    const int c = tid % 16, grp = tid / 16, col = blk % 8 * 64 + 4 * c;
    if (MODE != UPDATE_COPIES) {
      const float *src = a.gpart + which * kH + col;
#pragma unroll 16
      for (int q = grp; q < a.nsum; q += 16)
        acc += *reinterpret_cast<const f32x4 *>(src + (int64_t)q * kPart);
      red[grp][c] = acc;
      __syncthreads();
    }
    if (tid >= 16) return;
    if (MODE != UPDATE_COPIES)
      for (int k = 1; k < 16; ++k) acc += red[k][c];
    const f32x4 p = update4<MODE>(a, a.off_sum[which] + col, acc, true);
    if (MODE != UPDATE_GRAD && which == 4)
#pragma unroll
      for (int t = 0; t < 4; ++t) a.pm.w4b[col + t] = static_cast<bf16>(p[t]);
  } else if (MODE != UPDATE_COPIES) {
    __shared__ float red[2][256];
    float sg = 0.f, sl = 0.f;
    for (int q = tid; q < a.nsum; q += 256) {
      sg += a.gpart[(int64_t)q * kPart + 5 * kH];
      sl += a.gpart[(int64_t)q * kPart + 5 * kH + 1];
    }
    red[0][tid] = sg;
    red[1][tid] = sl;
    __syncthreads();
    for (int d = 128; d > 0; d >>= 1) {
      if (tid < d) {
        red[0][tid] += red[0][tid + d];
        red[1][tid] += red[1][tid + d];
      }
      __syncthreads();
    }
    if (tid > 0) return;
    a.loss[0] = red[1][0];
    const int64_t i = a.off_sum[5];
    a.g[i] = red[0][0];
    if (MODE == UPDATE_ADAM) a.p[i] = adam(a, a.p[i], red[0][0], a.m[i], a.v[i]);
  }
}

// Clears n floats (a kernel, so that it may be captured).
__global__ void zero_kernel(float *p, int64_t n) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.f;
}

__global__ void copy_kernel(const double *__restrict__ x, int64_t n, double *__restrict__ y) {
  const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (i < n) y[i] = x[i];
}

}  // namespace
}  // namespace fdadi

using namespace fdadi;

struct fdadi_mlp {
  int max_rows = 0;  // capacity of a training batch (multiple of 128)
  int64_t nparam = 0;
  int64_t off_W[kLayers] = {}, off_b[kLayers] = {}, off_w4 = 0, off_b4 = 0;
  float *p = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;  // master, grad, Adam moments
  bf16 *Wp[kLayers] = {}, *WpT[kLayers] = {}, *w4b = nullptr;    // packed copies
  bf16 *XT = nullptr, *ActT[kLayers - 1] = {}, *dZT[kLayers] = {};  // T blocks of a batch
  float *loss = nullptr, *gpart = nullptr;  // gpart: kPart sums per 32 rows
  float *wpart = nullptr;  // split-K partial weight gradients, layer by layer
  int n_in = kIn;          // features per input row
  double *lohi = nullptr;  // [lo(kMaxIn) | hi(kMaxIn)]
  double tmean = 0.0, tstd = 1.0;
  int64_t step = 0;
};

namespace fdadi {
namespace {

int in_dim(int l) { return l == 0 ? kInPad : kH; }

// Every device buffer of a model.
void free_buffers(fdadi_mlp *m) {
  void *ptrs[] = {m->p, m->g, m->m, m->v, m->w4b, m->XT, m->loss, m->gpart, m->wpart, m->lohi};
  for (void *q : ptrs) (void)hipFree(q);
  for (int l = 0; l < kLayers; ++l) {
    (void)hipFree(m->Wp[l]);
    (void)hipFree(m->WpT[l]);
    if (l < kLayers - 1) (void)hipFree(m->ActT[l]);
    (void)hipFree(m->dZT[l]);
  }
}

ParamMap param_map(const fdadi_mlp *m) {
  ParamMap pm;
  for (int l = 0; l < kLayers; ++l) {
    pm.off[l] = m->off_W[l];
    pm.Wp[l] = m->Wp[l];
    pm.WpT[l] = m->WpT[l];
  }
  pm.w4b = m->w4b;
  return pm;
}

UpdateArgs update_args(const fdadi_mlp *m) {
  UpdateArgs u{};
  u.p = m->p;
  u.g = m->g;
  u.m = m->m;
  u.v = m->v;
  u.gpart = m->gpart;
  u.loss = m->loss;
  for (int l = 0; l < kLayers; ++l) u.off_sum[l] = m->off_b[l];
  u.off_sum[4] = m->off_w4;
  u.off_sum[5] = m->off_b4;
  u.pm = param_map(m);
  return u;
}

template <int MODE>
int update(const UpdateArgs &u, hipStream_t s) {
  hipLaunchKernelGGL(update_kernel<MODE>, dim3(kWeightBlocks + kSumBlocks), dim3(256), 0, s, u);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

int refresh_bf16(fdadi_mlp *m, hipStream_t s) { return update<UPDATE_COPIES>(update_args(m), s); }

RowArgs row_args(const fdadi_mlp *m, const double *P, int64_t rows) {
  RowArgs a{};
  a.P = P;
  a.rows = rows;
  a.nin = m->n_in;
  a.lo = m->lohi;
  a.hi = m->lohi + kMaxIn;
  a.tmean = m->tmean;
  a.tstd = m->tstd;
  for (int l = 0; l < kLayers; ++l) {
    a.Wp[l] = m->Wp[l];
    if (l > 0) a.Wp[2 * kLayers - 1 - l] = m->WpT[l];
    a.bias[l] = m->p + m->off_b[l];
  }
  a.w4 = m->w4b;
  a.b4 = m->p + m->off_b4;
  return a;
}

// One launch for n rows.  One round of work-groups over
// the 256 CUs where that is enough: 32 rows each up to 8,192 (22.7 us; 28.0
// with 64), 64 up to 16,384 (31 us; 37 with 32, 39 with 48).  Beyond that two
// work-groups of 48 rows share a CU, one's SiLU beside the other's products:
// 99.8 us for 50,000 rows and 355 us for 200,000 (64 rows, one per CU: 110 and
// 368; 128 rows: 100 and 361).
int launch_rows(const fdadi_mlp *m, const double *d_P, int64_t n, double *d_out, hipStream_t s) {
  RowArgs a = row_args(m, d_P, n);
  a.out = d_out;
  if (n <= 256 * 32)
    hipLaunchKernelGGL((mlp_rows_kernel<2, 2, 4, false>), dim3(grid_for(n, 32)), dim3(kThreads), 0,
                       s, a);
  else if (n <= 256 * 64)
    hipLaunchKernelGGL((mlp_rows_kernel<4, 4, 2, false>), dim3(grid_for(n, 64)), dim3(kThreads), 0,
                       s, a);
  else
    hipLaunchKernelGGL((mlp_rows_kernel<3, 2, 4, false>), dim3(grid_for(n, 48)), dim3(kThreads), 0,
                       s, a);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

// Prices of n rows, no workspace -- unless they are to lie in the features' own
// memory: a work-group's prices would then overwrite rows that others have yet
// to read, so they go to the row kernel's sums first (1,282 prices' room per 32
// rows of the capacity: 5,128 at least), part by part.
int predict_rows(const fdadi_mlp *m, const double *d_P, int64_t n, double *d_out, hipStream_t s) {
  const uintptr_t p = reinterpret_cast<uintptr_t>(d_P), q = reinterpret_cast<uintptr_t>(d_out);
  const bool apart = q + n * sizeof(double) <= p || p + n * m->n_in * sizeof(double) <= q;
  if (apart) return launch_rows(m, d_P, n, d_out, s);
  double *const tmp = reinterpret_cast<double *>(m->gpart);
  const int64_t part = (int64_t)(m->max_rows / 32) * (kPart / 2);
  for (int64_t r = 0; r < n; r += part) {
    const int64_t rows = std::min(part, n - r);
    FDADI_RET(launch_rows(m, d_P + r * m->n_in, rows, tmp, s));
    hipLaunchKernelGGL(copy_kernel, dim3(grid_for(rows, 256)), dim3(256), 0, s, tmp, rows, d_out + r);
    FDADI_CHECK_LAUNCH();
  }
  return FDADI_OK;
}

// Most rows of a call without allocation: callers split their batches by it.
constexpr int kNoAllocRows = 4096;
static_assert(kNoAllocRows <= kTile / 32 * (kPart / 2), "one part at the smallest capacity");

}  // namespace
}  // namespace fdadi

extern "C" {

int fdadi_mlp_predict_noalloc(const fdadi_mlp *m, const double *d_P, int64_t n, double *d_out,
                              void *stream) {
  FDADI_REQUIRE(m && n >= 0 && (n == 0 || (d_P && d_out)), FDADI_ERR_ARG,
                "fdadi_mlp_predict_noalloc: bad arguments");
  FDADI_REQUIRE(n <= kNoAllocRows, FDADI_ERR_ARG,
                "fdadi_mlp_predict_noalloc: " + std::to_string(n) +
                    " rows exceed the maximum of " + std::to_string(kNoAllocRows) +
                    " per call (split the batch, or use fdadi_mlp_predict)");
  if (n == 0) return FDADI_OK;
  return predict_rows(m, d_P, n, d_out, as_stream(stream));
}

int fdadi_mlp_create(int32_t max_rows, const float *init_params, int64_t nparam,
                     const double *lo, const double *hi, double tmean, double tstd,
                     fdadi_mlp **out) {
  return fdadi_mlp_create_features(kIn, max_rows, init_params, nparam, lo, hi, tmean, tstd, out);
}

int fdadi_mlp_create_features(int32_t n_in, int32_t max_rows, const float *init_params,
                              int64_t nparam, const double *lo, const double *hi, double tmean,
                              double tstd, fdadi_mlp **out) {
  FDADI_REQUIRE(out && init_params && lo && hi, FDADI_ERR_ARG, "fdadi_mlp_create: null argument");
  FDADI_REQUIRE(n_in >= 1 && n_in <= kMaxIn, FDADI_ERR_ARG,
                "fdadi_mlp_create: 1 to 16 input features");
  FDADI_REQUIRE(max_rows > 0 && max_rows % kTile == 0, FDADI_ERR_ARG,
                "fdadi_mlp_create: max_rows must be a positive multiple of 128");
  fdadi_mlp *m = new fdadi_mlp();
  m->max_rows = max_rows;
  m->n_in = n_in;
  int64_t o = 0;
  for (int l = 0; l < kLayers; ++l) {
    m->off_W[l] = o;
    o += (int64_t)kH * in_dim(l);
    m->off_b[l] = o;
    o += kH;
  }
  m->off_w4 = o;
  o += kH;
  m->off_b4 = o;
  o += 1;
  m->nparam = o;
  if (nparam != o) {
    delete m;
    set_error("fdadi_mlp_create: expected " + std::to_string(o) + " parameters, got " +
              std::to_string(nparam));
    return FDADI_ERR_ARG;
  }
  m->tmean = tmean;
  m->tstd = tstd;
  hipError_t e = hipSuccess;
  auto al = [&](void **p, size_t bytes) {
    if (e == hipSuccess) e = hipMalloc(p, bytes);
  };
  const size_t R = (size_t)max_rows;
  al((void **)&m->p, sizeof(float) * o);
  al((void **)&m->g, sizeof(float) * o);
  al((void **)&m->m, sizeof(float) * o);
  al((void **)&m->v, sizeof(float) * o);
  size_t nw = 0;
  for (int l = 0; l < kLayers; ++l) {
    al((void **)&m->Wp[l], sizeof(bf16) * (l == 0 ? kPackIn : kPackH));
    if (l > 0) al((void **)&m->WpT[l], sizeof(bf16) * kPackH);
    if (l < kLayers - 1) al((void **)&m->ActT[l], sizeof(bf16) * R * kH);
    al((void **)&m->dZT[l], sizeof(bf16) * R * kH);
    nw += (size_t)kH * in_dim(l);
  }
  al((void **)&m->w4b, sizeof(bf16) * kH);
  al((void **)&m->XT, sizeof(bf16) * R * kInPad);
  al((void **)&m->gpart, sizeof(float) * (R / 32) * kPart);
  al((void **)&m->loss, sizeof(float));
  al((void **)&m->wpart, sizeof(float) * kMaxSplits * nw);
  al((void **)&m->lohi, sizeof(double) * 2 * kMaxIn);
  if (e == hipSuccess) e = hipMemcpy(m->p, init_params, sizeof(float) * o, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(m->lohi, lo, sizeof(double) * n_in, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(m->lohi + kMaxIn, hi, sizeof(double) * n_in, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    hipLaunchKernelGGL(zero_kernel, dim3(grid_for(o, 256)), dim3(256), 0, 0, m->m, o);
    hipLaunchKernelGGL(zero_kernel, dim3(grid_for(o, 256)), dim3(256), 0, 0, m->v, o);
    // the padding features' rows of the input's T blocks stay zero
    const int64_t nx = (int64_t)R * kInPad / 2;
    hipLaunchKernelGGL(zero_kernel, dim3(grid_for(nx, 256)), dim3(256), 0, 0, (float *)m->XT, nx);
    e = hipGetLastError();
  }
  if (e == hipSuccess && refresh_bf16(m, 0) != FDADI_OK) e = hipErrorUnknown;
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    set_error(std::string("fdadi_mlp_create: ") + hipGetErrorString(e));
    free_buffers(m);
    delete m;
    return FDADI_ERR_HIP;
  }
  *out = m;
  return FDADI_OK;
}

int fdadi_mlp_destroy(fdadi_mlp *m) {
  if (!m) return FDADI_OK;
  free_buffers(m);
  delete m;
  return FDADI_OK;
}

int fdadi_mlp_nparam(int64_t *n) {
  FDADI_REQUIRE(n, FDADI_ERR_ARG, "fdadi_mlp_nparam: null output");
  *n = (int64_t)kH * kInPad + kH + (kLayers - 1) * ((int64_t)kH * kH + kH) + kH + 1;
  return FDADI_OK;
}

int fdadi_mlp_get_params(const fdadi_mlp *m, float *params, float *grads) {
  FDADI_REQUIRE(m, FDADI_ERR_ARG, "fdadi_mlp_get_params: null model");
  FDADI_TRY_HIP(hipDeviceSynchronize());
  if (params) FDADI_TRY_HIP(hipMemcpy(params, m->p, sizeof(float) * m->nparam, hipMemcpyDeviceToHost));
  if (grads) FDADI_TRY_HIP(hipMemcpy(grads, m->g, sizeof(float) * m->nparam, hipMemcpyDeviceToHost));
  return FDADI_OK;
}

int fdadi_mlp_set_params(fdadi_mlp *m, const float *params, void *stream) {
  FDADI_REQUIRE(m && params, FDADI_ERR_ARG, "fdadi_mlp_set_params: null argument");
  FDADI_TRY_HIP(hipMemcpy(m->p, params, sizeof(float) * m->nparam, hipMemcpyHostToDevice));
  FDADI_RET(refresh_bf16(m, as_stream(stream)));
  return FDADI_OK;
}

// Gradient of the mean squared error (targets standardised with tmean/tstd)
// for rows idx[0..rows) of (P [n x nin], T [n]): the row kernel and the weight
// gradients; the update kernel (`up`) completes the sums over work-groups and
// splits.
static int grad_impl(fdadi_mlp *m, const double *d_P, const double *d_T, const int *d_idx,
                     int rows, UpdateArgs *up, hipStream_t s) {
  FDADI_REQUIRE(rows > 0 && rows <= m->max_rows, FDADI_ERR_ARG,
                "fdadi_mlp: batch rows exceed the model capacity");
  const int Mpad = (rows + kTile - 1) / kTile * kTile;
  RowArgs a = row_args(m, d_P, rows);
  a.T = d_T;
  a.idx = d_idx;
  a.XT = m->XT;
  for (int l = 0; l < kLayers; ++l) {
    if (l < kLayers - 1) a.ActT[l] = m->ActT[l];
    a.dZT[l] = m->dZT[l];
  }
  a.gpart = m->gpart;
  hipLaunchKernelGGL((mlp_rows_kernel<2, 4, 2, true>), dim3(Mpad / 32), dim3(kThreads), 0, s, a);
  FDADI_CHECK_LAUNCH();
  // dW_l = dZ_l^T A_{l-1}: the (kH x in_dim) output tiles are few, so the long
  // K = Mpad is split, and the partial products are summed in order
  int splits = 1;
  while (splits < kMaxSplits && Mpad % (kKBlock * splits * 2) == 0 && Mpad / (splits * 2) >= 512)
    splits *= 2;
  *up = update_args(m);
  up->splits = splits;
  up->nsum = Mpad / 32;
  WGradArgs w;
  float *part = m->wpart;
  for (int l = 0; l < kLayers; ++l) {
    up->part[l] = part;
    GemmArgs &g = w.g[kLayers - 1 - l];
    g.A = m->dZT[l];
    g.B = l == 0 ? m->XT : m->ActT[l - 1];
    g.ldA = g.ldB = kKStep;
    g.stA = (int64_t)kH * kKStep;
    g.stB = (int64_t)in_dim(l) * kKStep;
    g.M = kH;
    g.N = in_dim(l);
    g.K = Mpad;
    g.gx = g.N / kTile;
    g.gy = g.M / kTile;
    g.gz = splits;
    g.C = splits > 1 ? part : m->g + m->off_W[l];
    part += (size_t)kMaxSplits * kH * in_dim(l);
  }
  int total = 0;
  for (int j = 0; j < kLayers; ++j) {
    w.first[j] = total;
    total += w.g[j].gx * w.g[j].gy * w.g[j].gz;
  }
  hipLaunchKernelGGL(wgrad_kernel, dim3(total), dim3(kThreads), 0, s, w);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

int fdadi_mlp_grad(fdadi_mlp *m, const double *d_P, const double *d_T, const int *d_idx,
                   int32_t rows, float *loss, void *stream) {
  FDADI_REQUIRE(m && d_P && d_T, FDADI_ERR_ARG, "fdadi_mlp_grad: null argument");
  hipStream_t s = as_stream(stream);
  UpdateArgs up;
  FDADI_RET(grad_impl(m, d_P, d_T, d_idx, rows, &up, s));
  FDADI_RET(update<UPDATE_GRAD>(up, s));
  if (loss) {
    FDADI_TRY_HIP(hipMemcpyAsync(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost, s));
    FDADI_TRY_HIP(hipStreamSynchronize(s));
  }
  return FDADI_OK;
}

int fdadi_mlp_train_step(fdadi_mlp *m, const double *d_P, const double *d_T, const int *d_idx,
                         int32_t rows, float lr, void *stream) {
  FDADI_REQUIRE(m && d_P && d_T, FDADI_ERR_ARG, "fdadi_mlp_train_step: null argument");
  hipStream_t s = as_stream(stream);
  UpdateArgs up;
  FDADI_RET(grad_impl(m, d_P, d_T, d_idx, rows, &up, s));
  m->step += 1;
  up.lr = lr;
  up.b1 = 0.9f;
  up.b2 = 0.999f;
  up.eps = 1e-8f;
  up.c1 = 1.f - std::pow(up.b1, (float)m->step);
  up.c2 = 1.f - std::pow(up.b2, (float)m->step);
  return update<UPDATE_ADAM>(up, s);
}

int fdadi_mlp_loss(const fdadi_mlp *m, float *loss) {
  FDADI_REQUIRE(m && loss, FDADI_ERR_ARG, "fdadi_mlp_loss: null argument");
  FDADI_TRY_HIP(hipDeviceSynchronize());
  FDADI_TRY_HIP(hipMemcpy(loss, m->loss, sizeof(float), hipMemcpyDeviceToHost));
  return FDADI_OK;
}

int fdadi_mlp_predict(fdadi_mlp *m, const double *d_P, int64_t n, double *d_out, void *stream) {
  FDADI_REQUIRE(m && d_P && d_out && n >= 0, FDADI_ERR_ARG, "fdadi_mlp_predict: bad arguments");
  if (n == 0) return FDADI_OK;
  return predict_rows(m, d_P, n, d_out, as_stream(stream));
}

// Raw NT GEMM for tests: C (fp32, M x N) = A (bf16 bits, M x K) B^T (bf16 bits, N x K).
int fdadi_mlp_gemm_nt(const uint16_t *d_A, const uint16_t *d_B, int32_t M, int32_t N, int32_t K,
                      float *d_C, void *stream) {
  FDADI_REQUIRE(d_A && d_B && d_C, FDADI_ERR_ARG, "fdadi_mlp_gemm_nt: null argument");
  FDADI_REQUIRE(M % kTile == 0 && N % kTile == 0 && K % kKBlock == 0, FDADI_ERR_ARG,
                "mlp gemm: dimensions must be multiples of 128 x 128 x 128");
  GemmArgs g{reinterpret_cast<const bf16 *>(d_A), reinterpret_cast<const bf16 *>(d_B),
             K, kKStep, K, kKStep, M, N, K, N / kTile, M / kTile, 1, d_C};
  hipLaunchKernelGGL(gemm_nt_kernel, dim3(g.gx, g.gy, g.gz), dim3(kThreads), 0, as_stream(stream),
                     g);
  FDADI_CHECK_LAUNCH();
  return FDADI_OK;
}

}  // extern "C"
