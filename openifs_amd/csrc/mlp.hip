// BF16 MFMA multilayer perceptron for gfx950: forward, backward and Adam, all on the device.
//
// Network: x[n_in] -> (Linear, SiLU) x n_hidden_layers -> Linear -> y[n_out].  Weights W_l [n_out_l x n_in_l]
// are held in FP32 (master copy, Adam moments) and mirrored to BF16.  Activations are BF16, every product accumulates
// in FP32 on the matrix cores (v_mfma_f32_32x32x16_bf16), 16 contraction entries at a time in ascending order, so a
// result does not depend on the tile that computed it.
//
// All products have the one form C[M x N] = A[M x K] * B[N x K]^T:
//   forward        Z_l   = X_l  * W_l^T         (A = X_l,    B = W_l)
//   input grad     dX_l  = dZ_l * W_l           (A = dZ_l,   B = W_l^T)
//   weight grad    dW_l  = dZ_l^T * X_l         (A = dZ_l^T, B = X_l^T, contraction over the batch)
// Every matrix is stored once, row-major; an operand whose contraction index is its row index (W_l^T, dZ_l^T, X_l^T)
// is transposed on the way from LDS to the registers (ds_read_b64_tr_b16).
// Dimensions must be multiples of 128 (M, N) and 32 (K); callers pad features and outputs with zeros.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>
#include <cstring>
#include <type_traits>
#include <vector>

#include "../../include/cloudsc_surrogate.h"
#include "capi_util.h"
#include "mlp_internal.h"
#include "synth.h"

namespace mlp {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int BM = 128, BN = 128, BK = 32;  // granularity of every dimension
constexpr int MAX_SPLIT = 4;                // stretches of a split weight-gradient contraction

enum Epi : int {
  EPI_F32 = 0,      // C (fp32)
  EPI_HIDDEN = 1,   // z = acc + bias -> C (fp32, kept for the backward pass); a = silu(z) -> act (bf16)
  EPI_HIDDEN_INF = 2,  // inference: a = silu(acc + bias) -> act (bf16) only
  EPI_OUT = 3,      // y = acc + bias -> C (fp32)
  EPI_DHIDDEN = 4,  // g = acc * silu'(z) -> act (bf16): the gradient w.r.t. the previous pre-activation
  EPI_LOSS = 5,     // y as EPI_OUT, and the loss L = sum wgt[n] (y - t)^2 / M and its gradient -> act (bf16)
};

struct EpiArgs {
  const float* bias;
  float* c;        // fp32 [M x N], leading dimension ldc
  int ldc;
  bf16* act;       // bf16 [M x N], leading dimension ldc
  const float* z;  // fp32 [M x N] pre-activation (EPI_DHIDDEN) or target (EPI_LOSS), leading dimension ldc
  long zstride;    // split contraction (EPI_F32, grid z > 1): elements between the partial products of the splits
  const float* wgt;  // EPI_LOSS: weight per column
  float* loss;       // EPI_LOSS: accumulated here by atomics; EPI_HIDDEN: set to 0 if not NULL
  float batch;       // EPI_LOSS: rows of the batch
};

typedef float f32x4 __attribute__((ext_vector_type(4)));
// At pointers and leading dimensions of a caller, who need only align them to the element: the same instructions.
typedef f32x4 __attribute__((aligned(4))) f32x4_any;
typedef bf16x8 __attribute__((aligned(2))) bf16x8_any;

// 1 / (1 + exp(-z)).  For every float x from 1 to 2^126 one Newton step on v_rcp_f32 gives the correctly rounded 1 / x
// (all 1.06e9 checked against the division), in 3 instructions for the division's 10, which were two thirds of the hidden
// layers' epilogues (65,536 x 1,024 x 1,920 258 -> 247 us); beyond (z < -87), where 1 / x is denormal, the division.
__device__ __forceinline__ f32x4 sigmoid(f32x4 z) {
  f32x4 x, r;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    x[t] = 1.0f + __expf(-z[t]);
    const float r0 = __builtin_amdgcn_rcpf(x[t]);
    r[t] = __builtin_fmaf(__builtin_fmaf(-x[t], r0, 1.0f), r0, r0);
  }
  const float most = __builtin_fmaxf(__builtin_fmaxf(x[0], x[1]), __builtin_fmaxf(x[2], x[3]));
  if (__builtin_expect(most > 0x1p126f, 0)) {
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] = 1.0f / x[t];
  }
  return r;
}
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// Epilogue of a wave's FM x FN fragments of C^T = B A^T: register r of lane l holds C[m][n] with m = lane & 31 of the
// fragment's rows and n = 8 (r >> 2) + 4 (l >> 5) + (r & 3) of its columns.  Stored like that, an instruction touches 32
// rows with 16 or 32 bytes each; so each fragment goes through 4 KB of LDS (lds: this wave's own) into a layout of 8
// rows of 8 lanes x 4 consecutive columns, in which every load and store covers full runs of 64 (bf16) or 128 bytes.
// Row r's 16-byte chunk c is in slot c ^ ((r >> 1) & 7): 16 rows' equal chunks and two rows' chunks are both spread over
// all banks.  row, col: the wave's first row and column.  All loads come before the first store: loads and stores share
// one in-order wait counter.
template <int EPI, int NW, int FM, int FN>
__device__ __forceinline__ void epilogue(const EpiArgs& e, const f32x16 (&acc)[FM][FN], bf16* lds, int row, int col) {
  constexpr bool BIAS = EPI == EPI_HIDDEN || EPI == EPI_HIDDEN_INF || EPI == EPI_OUT || EPI == EPI_LOSS;
  constexpr bool READZ = EPI == EPI_DHIDDEN || EPI == EPI_LOSS;
  typedef f32x4 __attribute__((may_alias)) tile4;
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  float* wr = reinterpret_cast<float*>(lds) + 32 * r;                // this lane's row on the way in
  const float* rd = reinterpret_cast<float*>(lds) + 32 * (lane >> 3);  // and its first row on the way out
  row += lane >> 3;
  col += 4 * (lane & 7);
  f32x4 bias[FN], wgt[FN], z[FM][FN][4];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    if (BIAS) bias[j] = *reinterpret_cast<const f32x4*>(e.bias + col + j * 32);
    if (EPI == EPI_LOSS) wgt[j] = *reinterpret_cast<const f32x4_any*>(e.wgt + col + j * 32);
    if (READZ)
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          z[i][j][q] = *reinterpret_cast<const f32x4_any*>(e.z + (size_t)(row + i * 32 + 8 * q) * e.ldc + col + j * 32);
  }
  float l = 0.0f;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<tile4*>(wr + 4 * ((2 * q + h) ^ ((r >> 1) & 7))) =
            f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const size_t o = (size_t)(row + i * 32 + 8 * q) * e.ldc + col + j * 32;
        f32x4 v = *reinterpret_cast<const tile4*>(rd + 256 * q + 4 * ((lane & 7) ^ ((4 * q + (lane >> 4)) & 7)));
        if (BIAS) v = v + bias[j];
        if (EPI != EPI_HIDDEN_INF && EPI != EPI_DHIDDEN) *reinterpret_cast<f32x4_any*>(e.c + o) = v;
        if (EPI == EPI_F32 || EPI == EPI_OUT) continue;
        bf16x4 a;
        f32x4 sg;
        if (EPI == EPI_HIDDEN || EPI == EPI_HIDDEN_INF) sg = sigmoid(v);
        if (EPI == EPI_DHIDDEN) sg = sigmoid(z[i][j][q]);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          if (EPI == EPI_HIDDEN || EPI == EPI_HIDDEN_INF) {
            a[t] = (bf16)(v[t] * sg[t]);
          } else if (EPI == EPI_DHIDDEN) {
            const float zt = z[i][j][q][t], s = sg[t];
            a[t] = (bf16)(v[t] * (s * (1.0f + zt * (1.0f - s))));
          } else {
            const float d = v[t] - z[i][j][q][t];
            const float wd = wgt[j][t] * d;
            l += wd * d;
            a[t] = (bf16)(2.0f * wd / e.batch);
          }
        }
        *reinterpret_cast<bf16x4*>(e.act + o) = a;
      }
    }
  if constexpr (EPI == EPI_LOSS) {  // one atomic per group: they all go to one address and are served one by one
    __shared__ float part[NW];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_down(l, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int i = 1; i < NW; ++i) l += part[i];
      atomicAdd(e.loss, l / e.batch);
    }
  }
}

// One operand tile of TB rows x 64 contraction entries in LDS, filled by global_load_lds_dwordx4 (lane l of a load
// writes 16 bytes at 16 l).  Each lane fetches the global chunk that belongs in its LDS slot.  DIRECT = false: the same
// through registers, for matrices that start at an address that is no multiple of 16, which loads into LDS do not take.
//  T = false: the matrix is [rows][K].  LDS row r of 128 bytes, chunk c (16 B) in slot c ^ ((r >> 1) & 7): a fragment
//    read (16 lanes = 16 consecutive rows, one chunk) finds its rows in distinct slots of the banks.
//  T = true: the matrix is [K][rows].  LDS row k of TB entries, its 64-byte chunk c in slot c ^ f(k) such that the 4
//    rows k..k+3 which one transposing read touches lie in distinct quarters of the banks.
template <int TB, bool T, int NW, bool DIRECT = true>
struct Tile {
  static constexpr int W = T ? TB * 2 : 128;        // bytes per LDS row
  static constexpr int NLD = TB * 128 / 1024 / NW;  // loads per wave
  static __device__ __forceinline__ int swz(int k) { return TB == 128 ? (k & 3) : ((k >> 1) & 1); }
  // p: the matrix at (row0, k0 = 0).  CLAMP: only K entries may be read (the last step of a contraction that is no
  // multiple of 64 repeats its last entries, which are not multiplied).
  template <bool CLAMP>
  static __device__ __forceinline__ void load(bf16* lds, const bf16* p, int ld, int k0, int K, int w, int lane) {
    typedef bf16 __attribute__((address_space(3))) lbf16;
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
      const int g = NW * i + w;  // 1 KB group of the tile
      const bf16* src;
      if (T) {
        const int r = lane / (W / 16), s = lane % (W / 16), k = g * (1024 / W) + r;
        src = p + (size_t)(CLAMP ? min(k0 + k, K - 1) : k0 + k) * ld + 32 * ((s >> 2) ^ swz(k)) + 8 * (s & 3);
      } else {
        const int r = 8 * g + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
        src = p + (size_t)r * ld + (CLAMP ? min(k0 + 8 * c, K - 8) : k0 + 8 * c);
      }
      if constexpr (DIRECT)
        __builtin_amdgcn_global_load_lds((const void*)src, (lbf16*)(lds + g * 512), 16, 0, 0);
      else
        *reinterpret_cast<bf16x8*>(lds + g * 512 + 8 * lane) = *reinterpret_cast<const bf16x8_any*>(src);
    }
  }
  // MFMA 32x32x16 operand: lane l supplies row (l & 31) of the 32-row block rb and k = ks + 8 (l >> 5) .. +7.  A
  // transposing read gives lane i of 16 the column i of 4 rows, whose 16-byte quarters the lanes 4 j + q address.
  static __device__ __forceinline__ bf16x8 frag(const bf16* lds, int rb, int ks, int lane) {
    if (T) {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      typedef s16x4 __attribute__((address_space(3))) ls16x4;
      const int j = (lane >> 2) & 3, n = 16 * ((lane >> 4) & 1) + 4 * (lane & 3), k = ks + 8 * (lane >> 5) + j;
      const bf16* a = lds + k * TB + 32 * ((rb >> 5) ^ swz(k)) + n;
      const bf16* b = lds + (k + 4) * TB + 32 * ((rb >> 5) ^ swz(k + 4)) + n;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4*)a);
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((ls16x4*)b);
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(bf16x8, v);
    }
    const int r = rb + (lane & 31), c = (ks >> 3) + (lane >> 5);
    return *reinterpret_cast<const bf16x8*>(lds + r * 64 + 8 * (c ^ ((r >> 1) & 7)));
  }
};

// Waits until at most N of this wave's vector loads are in flight and its LDS reads are done, then for the group.
template <int N>
__device__ __forceinline__ void landed() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));  // vmcnt(N) lgkmcnt(0), no expcnt
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The kernel of the training products: a TBM x TBN tile by NW waves (2 x NW/2), contraction steps of 64 in a ring of 4
// LDS stages filled 3 steps ahead.  These products have about one tile per CU, so the loads ahead have to cover the
// latency: a step of 128 x 128 multiplies for ~0.2 us at the matrix cores' rate and its loads take
// several times that; it measures 0.5 us, which is the rate the tiles come from L2 (16 TB/s over the chip).  The stages
// are separate LDS objects and the step loop is unrolled over them, so that the compiler can tell a read of one stage
// from the loads in flight into the others.  4,096 x 1,024 x 1,024 with the hidden layer's epilogue (25 MB stored):
// 18 us, x 1,920: 26 us; the register-staged kernel with transposed copies of every activation and gradient that this
// one replaces took 39 us on average over the three, the weight gradient 25 -> 16 us and the input gradient 35 -> 20 us
// (1,024 x 1,024).
template <int EPI, int TBM, int TBN, int NW, bool TA, bool TB, bool DIRECT = true>
__global__ __launch_bounds__(64 * NW) void gemm_ring(const bf16* __restrict__ A, int lda, const bf16* __restrict__ B,
                                                 int ldb, int K, EpiArgs e) {
  constexpr int WN = NW / 2, WCOL = TBN / WN, FM = TBM / 64, FN = WCOL / 32;  // 2 x WN waves of FM x FN fragments
  typedef Tile<TBM, TA, NW, DIRECT> OpA;
  typedef Tile<TBN, TB, NW, DIRECT> OpB;
  constexpr int ELEMS = (TBM + TBN) * 64, NLD = OpA::NLD + OpB::NLD;
  __shared__ __attribute__((aligned(1024))) bf16 s0[ELEMS], s1[ELEMS], s2[ELEMS], s3[ELEMS];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  // XCD order: consecutive work-groups go to the 8 XCDs in turn; each XCD takes one contiguous eighth of the tiles
  // (N fastest, then M, then the stretch of a split contraction), so that its L2 holds what those tiles share.
  const uint32_t total = gridDim.x * gridDim.y * gridDim.z;
  const uint32_t id = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const uint32_t x = id & 7u, r8 = total & 7u;
  const uint32_t tile = x * (total >> 3) + (x < r8 ? x : r8) + (id >> 3);
  const int nt = tile % gridDim.x, mt = tile / gridDim.x % gridDim.y, zt = tile / (gridDim.x * gridDim.y);
  const int m0 = mt * TBM, n0 = nt * TBN;
  // split contraction: group zt multiplies the zt-th stretch of K entries into its own partial product
  const size_t kz = (size_t)zt * K;
  const bf16* ap = TA ? A + kz * lda + m0 : A + (size_t)m0 * lda + kz;
  const bf16* bp = TB ? B + kz * ldb + n0 : B + (size_t)n0 * ldb + kz;
  if (EPI == EPI_F32) e.c += (size_t)zt * e.zstride;
  if (EPI == EPI_HIDDEN && e.loss && tid == 0 && id == 0) *e.loss = 0.0f;
  auto load = [&](bf16* s, int t, auto clamp) {
    OpA::template load<decltype(clamp)::value>(s, ap, lda, 64 * t, K, w, lane);
    OpB::template load<decltype(clamp)::value>(s + TBM * 64, bp, ldb, 64 * t, K, w, lane);
  };
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  const int nk = (K + 63) / 64;
  auto sub = [&](const bf16* s, int ks) {  // 16 contraction entries
    bf16x8 a[FM], b[FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) a[i] = OpA::frag(s, wm * (TBM / 2) + i * 32, ks, lane);
#pragma unroll
    for (int j = 0; j < FN; ++j) b[j] = OpB::frag(s + TBM * 64, wn * WCOL + j * 32, ks, lane);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b[j], a[i], acc[i][j], 0, 0, 0);
  };
  // One step: this wave's loads of stage t have landed, then everyone's have (and everyone is done with stage t - 1,
  // whose buffer `next` takes step t + 3).  The loads of steps t + 1 and t + 2 stay in flight.
  auto step = [&](const bf16* cur, bf16* next, int t) {
    landed<2 * NLD>();
    load(next, t + 3, std::false_type());
#pragma unroll
    for (int ks = 0; ks < 64; ks += 16) sub(cur, ks);
  };
  // The last steps, and contractions of few steps.
  auto tail = [&](const bf16* cur, bf16* next, int t) {
    const int ahead = nk - 1 - t;  // later steps whose loads may still be in flight: 2 at most
    if (ahead >= 2)
      landed<2 * NLD>();
    else if (ahead == 1)
      landed<NLD>();
    else
      landed<0>();
    if (ahead >= 3) load(next, t + 3, std::true_type());
    sub(cur, 0);
    sub(cur, 16);
    if (K - 64 * t > 32) {
      sub(cur, 32);
      sub(cur, 48);
    }
  };
  load(s0, 0, std::true_type());  // contractions of fewer than 3 steps load entries of their last one again
  load(s1, 1, std::true_type());
  load(s2, 2, std::true_type());
  int t = 0;
  for (; t + 7 < nk; t += 4) {
    step(s0, s3, t);
    step(s1, s0, t + 1);
    step(s2, s1, t + 2);
    step(s3, s2, t + 3);
  }
  for (; t < nk; t += 4) {
    tail(s0, s3, t);
    if (t + 1 >= nk) break;
    tail(s1, s0, t + 1);
    if (t + 2 >= nk) break;
    tail(s2, s1, t + 2);
    if (t + 3 >= nk) break;
    tail(s3, s2, t + 3);
  }

  landed<0>();  // no load into LDS outlives the group, and its LDS is free
  epilogue<EPI, NW, FM, FN>(e, acc, s0 + w * 2048, m0 + wm * (TBM / 2), n0 + wn * WCOL);
}

// The large-product kernel: 256 x 256 block tile, 8 waves as 2 x 4, each computing 128 rows x 64 columns in 32x32
// fragments; contraction steps of 64, so that a load takes every row's full 128-byte line (half lines take as many L2
// requests), in an LDS ring of 3 stages for A, which comes from HBM, and 2 for B, which stays in L2 (160 KB in all).
// The fragments of a quarter step are read while the quarter before multiplies.  65,536 x 1,024 x 1,920 takes 247 us
// (1,040 TF/s; with the loads left out 218 us: the matrix cores' clock falls under this load), x 1,024 151 us, of which
// some 40 us are the epilogues, during which a CU's matrix cores idle; with two full LDS buffers of 64, waited for at
// each step, the sigmoid's division and stores of 8 bytes a row it was 278 and 166 us.  Two groups of 128 x 256 on a CU,
// so that one's epilogue would overlap the other's products, ask for 1.5 times the bytes: 361 and 174 us.
template <int EPI>
__global__ __launch_bounds__(512) void gemm_wide(const bf16* __restrict__ A, int lda, const bf16* __restrict__ B,
                                                 int ldb, int K, EpiArgs e) {
  constexpr int NW = 8, TBM = 256, TBN = 256, TBK = 64, WN = 4, WCOL = 64, FM = 4, FN = 2;
  typedef Tile<256, false, NW> Op;
  __shared__ __attribute__((aligned(1024))) bf16 a0[256 * TBK], a1[256 * TBK], a2[256 * TBK], b0[256 * TBK], b1[256 * TBK];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WN, wn = w % WN;
  // Tile mapping: the dispatcher hands consecutive workgroups to the 8 XCDs in turn, each with its own L2.  With the
  // M-tile count a multiple of 8, workgroup L goes to XCD L % 8 and takes, in that XCD's order, all N-tiles of one
  // M-tile before the next, so the A tile they share is fetched into one L2 only.
  int mt = blockIdx.y, nt = blockIdx.x;
  if ((gridDim.y & 7) == 0) {
    const int L = blockIdx.y * gridDim.x + blockIdx.x, slot = L >> 3;
    nt = slot % gridDim.x;
    mt = (slot / gridDim.x) * 8 + (L & 7);
  }
  const int m0 = mt * TBM, n0 = nt * TBN;
  const bf16* ap = A + (size_t)m0 * lda;
  const bf16* bp = B + (size_t)n0 * ldb;
  // past the last step: its entries again, which nobody reads
  auto load_a = [&](bf16* s, int t) { Op::template load<false>(s, ap, lda, min(TBK * t, K - TBK), K, w, lane); };
  auto load_b = [&](bf16* s, int t) { Op::template load<false>(s, bp, ldb, min(TBK * t, K - TBK), K, w, lane); };
  if (EPI == EPI_HIDDEN && e.loss && tid == 0 && blockIdx.x == 0 && blockIdx.y == 0) *e.loss = 0.0f;
  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

  struct Frags {
    bf16x8 a[FM], b[FN];
  };
  auto read = [&](const bf16* sa, const bf16* sb, int ks, Frags& f) {
#pragma unroll
    for (int j = 0; j < FN; ++j) f.b[j] = Op::frag(sb, wn * WCOL + j * 32, ks, lane);
#pragma unroll
    for (int i = 0; i < FM; ++i) f.a[i] = Op::frag(sa, wm * 128 + i * 32, ks, lane);
  };
  auto multiply = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[j], f.a[i], acc[i][j], 0, 0, 0);
  };
  auto interleave = [](auto loads, auto reads) {  // the order of a quarter step: a product, an LDS read, a load, ...
#pragma unroll
    for (int i = 0; i < FM * FN; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                             // matrix product
      if (decltype(reads)::value && i < FM + FN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      if (decltype(loads)::value && i < Op::NLD) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // load into LDS
    }
  };
  // Step t: this wave's loads of A(t) and B(t) have landed (those of A(t + 1) stay in flight), then everyone's have, and
  // everyone is done with step t - 1, whose buffers take B(t + 1) and A(t + 2).  The fragments of a quarter step are read
  // while the quarter before multiplies.
  auto step = [&](const bf16* ca, bf16* fa, const bf16* cb, bf16* fb, int t) {
    Frags f, g;
    landed<Op::NLD>();
    load_b(fb, t + 1);
    read(ca, cb, 0, f);
    __builtin_amdgcn_sched_group_barrier(0x100, FM + FN, 0);
    read(ca, cb, 16, g);
    multiply(f);
    interleave(std::true_type(), std::true_type());
    __builtin_amdgcn_sched_barrier(0);  // the wait counts on A's loads being the later ones
    load_a(fa, t + 2);
    read(ca, cb, 32, f);
    multiply(g);
    interleave(std::true_type(), std::true_type());
    read(ca, cb, 48, g);
    multiply(f);
    interleave(std::false_type(), std::true_type());
    multiply(g);
    interleave(std::false_type(), std::false_type());
  };
  const int nk = K / TBK;
  load_a(a0, 0);
  load_b(b0, 0);
  __builtin_amdgcn_sched_barrier(0);
  load_a(a1, 1);
  int t = 0;
  for (; t + 6 <= nk; t += 6) {
    step(a0, a2, b0, b1, t);
    step(a1, a0, b1, b0, t + 1);
    step(a2, a1, b0, b1, t + 2);
    step(a0, a2, b1, b0, t + 3);
    step(a1, a0, b0, b1, t + 4);
    step(a2, a1, b1, b0, t + 5);
  }
  if (t < nk) step(a0, a2, b0, b1, t);
  if (t + 1 < nk) step(a1, a0, b1, b0, t + 1);
  if (t + 2 < nk) step(a2, a1, b0, b1, t + 2);
  if (t + 3 < nk) step(a0, a2, b1, b0, t + 3);
  if (t + 4 < nk) step(a1, a0, b0, b1, t + 4);
  landed<0>();  // no load into LDS outlives the group, and its LDS is free
  epilogue<EPI, NW, FM, FN>(e, acc, a0 + w * 2048, m0 + wm * 128, n0 + wn * WCOL);
}

// Sum of the S partial products of a split contraction, in split order: out[i] = sum_z part[z * n + i].
__global__ void sum_splits(const float* __restrict__ part, size_t n, int S, float* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float v = part[i];
  for (int z = 1; z < S; ++z) v += part[(size_t)z * n + i];
  out[i] = v;
}

// Bias gradient: db[n] = sum_m G[m][n] (fp32 sum of the bf16 gradient the weight product also sees), NC = 8 columns per
// group of 256.  Partial sum i of a column holds the rows m = i, i + 256, ..., one per lane, and the 256 partials are
// added in a binary tree.  A group's rows are 16 bytes of a line: `group` deals 8 neighbouring groups to one XCD, whose
// L2 then fetches each line once (4,096 x 1,024: 32 columns per group took 12 us, on 32 CUs).  Returns the sum of column
// 8 * (its group) + threadIdx.x to the threads 0..7, with that column in *c.
constexpr int NC = 8;
__device__ __forceinline__ float column_sum(const bf16* __restrict__ g, int M, int ld, int id, int* c) {
  __shared__ float red[256][NC + 1];
  const int ngroups = ld / NC;  // a multiple of 16
  const int group = (id & 7) * (ngroups >> 3) + (id >> 3), t = threadIdx.x;
  const bf16* gp = g + (size_t)t * ld + group * NC;
  float s[NC] = {};
  auto add = [&](const bf16x8 v) {
#pragma unroll
    for (int i = 0; i < NC; ++i) s[i] += (float)v[i];
  };
  int m = 0;
  for (; m + 2048 <= M; m += 2048) {
    bf16x8 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = *reinterpret_cast<const bf16x8*>(gp + (size_t)(m + 256 * j) * ld);
#pragma unroll
    for (int j = 0; j < 8; ++j) add(v[j]);
  }
  for (; m + t < M; m += 256) add(*reinterpret_cast<const bf16x8*>(gp + (size_t)m * ld));
#pragma unroll
  for (int i = 0; i < NC; ++i) red[t][i] = s[i];
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    for (int i = t >> 3; i < h; i += 32) red[i][t & 7] += red[i + h][t & 7];
    __syncthreads();
  }
  *c = group * NC + (t & 7);
  return red[0][t & 7];
}

__global__ __launch_bounds__(256) void column_sums(const bf16* __restrict__ g, int M, int ld, float* __restrict__ db) {
  int c;
  const float v = column_sum(g, M, ld, blockIdx.x, &c);
  if (threadIdx.x < NC) db[c] = v;
}

// Adam on FP32 master weights (n entries, a multiple of 4) and biases (nb entries, a multiple of 64); refreshes the
// BF16 copy of the weights.  Weight gradient: gw, or with S > 1 the sum of the S partial products in part, in split
// order, which is stored to gw.  Bias gradient: gb, or with g the column sums of g [M x nb], which are stored to gb; the
// groups that form them come first and run while the others update the weights.
struct AdamArgs {
  float *w, *m1, *m2, *gw;
  const float* part;
  size_t n;
  bf16* wb;
  float *b, *mb1, *mb2, *gb;
  const bf16* g;
  int M, nb;
  float lr, beta1, beta2, eps, bc1, bc2;
};
__device__ __forceinline__ float adam1(const AdamArgs& a, float g, float& m1, float& m2, float w) {
  m1 = a.beta1 * m1 + (1.0f - a.beta1) * g;
  m2 = a.beta2 * m2 + (1.0f - a.beta2) * g * g;
  return w - a.lr * (m1 / a.bc1) / (sqrtf(m2 / a.bc2) + a.eps);
}
template <int S>
__global__ __launch_bounds__(256) void adam_update(AdamArgs a) {
  const int ngb = a.nb / NC;
  if ((int)blockIdx.x < ngb) {  // biases
    int i = blockIdx.x * NC + (threadIdx.x & 7);
    const float v = a.g ? column_sum(a.g, a.M, a.nb, blockIdx.x, &i) : a.gb[i];
    if (threadIdx.x < NC) {
      a.gb[i] = v;
      a.b[i] = adam1(a, v, a.mb1[i], a.mb2[i], a.b[i]);
    }
    return;
  }
  const size_t i = ((size_t)(blockIdx.x - ngb) * 256 + threadIdx.x) * 4;
  if (i >= a.n) return;
  auto at = [&](float* p) { return reinterpret_cast<f32x4*>(p + i); };
  f32x4 m1 = *at(a.m1), m2 = *at(a.m2), w = *at(a.w), g;
  if constexpr (S > 1) {
    f32x4 part[S];
#pragma unroll
    for (int z = 0; z < S; ++z) part[z] = *reinterpret_cast<const f32x4*>(a.part + (size_t)z * a.n + i);
    g = part[0];
#pragma unroll
    for (int z = 1; z < S; ++z) g = g + part[z];
    *at(a.gw) = g;
  } else {
    g = *at(a.gw);
  }
  bf16x4 h;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    float p = m1[t], q = m2[t];
    w[t] = adam1(a, g[t], p, q, w[t]);
    m1[t] = p;
    m2[t] = q;
    h[t] = (bf16)w[t];
  }
  *at(a.m1) = m1;
  *at(a.m2) = m2;
  *at(a.w) = w;
  *reinterpret_cast<bf16x4*>(a.wb + i) = h;
}

// FP32 -> BF16 copy of a weight matrix.
__global__ void to_bf16(const float* __restrict__ w, size_t n, bf16* __restrict__ wb) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) wb[i] = (bf16)w[i];
}

}  // namespace mlp

// ---------------------------------------------------------------------------------------------------------
// Model object and C-ABI
// ---------------------------------------------------------------------------------------------------------
using mlp::bf16;
using cloudsc_capi::fail;


namespace {

int dev_alloc(cloudsc_mlp* m, size_t bytes, void** p) {
  hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) return fail(CLOUDSC_ENOMEM, "cloudsc_mlp: hipMalloc", e);
  m->allocs.push_back(*p);
  return CLOUDSC_OK;
}

// Tile choice: 256 x 256 where that gives a tile for every CU (256), else 128 x 128 where that gives one for every
// other CU, else 64 x 64.  Training's other products take 128 x 128 at any batch, also where it would give 256 tiles of
// 256 x 256 (steps of 16,384 rows, 1,920 -> 3 x 1,024 -> 1,024: 1,367 us with those, register-staged, 819 with these; of
// 65,536 rows 5,154 and 3,278 us).  Operands of a caller (the input x, cloudsc_mlp_gemm_tn) that do not start at a
// multiple of 16 bytes: 64 x 64 through registers, the same bits.
template <int EPI, bool TA = false, bool TB = false>
hipError_t gemm(const bf16* A, int lda, const bf16* B, int ldb, int M, int N, int K, const mlp::EpiArgs& e,
                hipStream_t s, int splits = 1) {
  if constexpr (EPI == mlp::EPI_F32 || EPI == mlp::EPI_HIDDEN || EPI == mlp::EPI_HIDDEN_INF) {
    if (((uintptr_t)A | (uintptr_t)B) % 16 != 0) {
      hipLaunchKernelGGL((mlp::gemm_ring<EPI, 64, 64, 4, TA, TB, false>), dim3(N / 64, M / 64, splits), dim3(256), 0, s,
                         A, lda, B, ldb, K, e);
      return hipGetLastError();
    }
  }
  const long groups256 = (M % 256 == 0 && N % 256 == 0) ? (long)(M / 256) * (N / 256) : 0;
  if constexpr (!TA && !TB && EPI != mlp::EPI_LOSS) {  // (the loss epilogue does not fit that tile's registers)
    if (groups256 >= 256 && K % 64 == 0 && splits == 1) {
      hipLaunchKernelGGL((mlp::gemm_wide<EPI>), dim3(N / 256, M / 256), dim3(512), 0, s, A, lda, B, ldb, K, e);
      return hipGetLastError();
    }
  }
  if ((long)(M / 128) * (N / 128) * splits >= 128)
    hipLaunchKernelGGL((mlp::gemm_ring<EPI, 128, 128, 8, TA, TB>), dim3(N / 128, M / 128, splits), dim3(512), 0, s, A,
                       lda, B, ldb, K, e);
  else
    hipLaunchKernelGGL((mlp::gemm_ring<EPI, 64, 64, 4, TA, TB>), dim3(N / 64, M / 64, splits), dim3(256), 0, s, A, lda, B,
                       ldb, K, e);
  return hipGetLastError();
}

inline unsigned blocks(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

int check_batch(const cloudsc_mlp* m, int M) {
  if (M <= 0 || M > m->max_batch || M % mlp::BM)
    return fail(CLOUDSC_EDIMS, "cloudsc_mlp: batch must be a positive multiple of 128 and <= max_batch");
  return CLOUDSC_OK;
}

}  // namespace

namespace mlp {
// Forward pass; with loss, Z and the activations are kept for the backward pass, and the loss against target t with
// weights wgt and its gradient (into g0) are formed in the output layer's epilogue.
hipError_t forward(cloudsc_mlp* m, const bf16* x, int M, float* y, const float* t, const float* wgt, hipStream_t s) {
  const bool train = t != nullptr;
  hipError_t e = hipSuccess;
  const bf16* in = x;
  int ldin = m->din[0];
  for (int l = 0; l < m->nl && e == hipSuccess; ++l) {
    mlp::EpiArgs ea{};
    ea.bias = m->b[l];
    if (l < m->nl - 1) {
      ea.c = m->z[l];
      ea.ldc = m->dout[l];
      ea.act = m->a[l];
      if (train && l == 0) ea.loss = m->loss;  // cleared here
      e = train ? gemm<mlp::EPI_HIDDEN>(in, ldin, m->wb[l], m->din[l], M, m->dout[l], m->din[l], ea, s)
                : gemm<mlp::EPI_HIDDEN_INF>(in, ldin, m->wb[l], m->din[l], M, m->dout[l], m->din[l], ea, s);
      in = m->a[l];
      ldin = m->dout[l];
    } else {
      ea.c = y;
      ea.ldc = m->dout[l];
      ea.act = m->g0;
      ea.z = t;
      ea.wgt = wgt;
      ea.loss = m->loss;
      ea.batch = (float)M;
      e = train ? gemm<mlp::EPI_LOSS>(in, ldin, m->wb[l], m->din[l], M, m->dout[l], m->din[l], ea, s)
                : gemm<mlp::EPI_OUT>(in, ldin, m->wb[l], m->din[l], M, m->dout[l], m->din[l], ea, s);
    }
  }
  return e;
}
}  // namespace mlp

namespace {

struct AdamStep {
  float lr, beta1, beta2, eps, bc1, bc2;
};

AdamStep next_step(const cloudsc_mlp* m, float lr, float beta1, float beta2, float eps) {
  const float n = (float)(m->step + 1);
  return AdamStep{lr, beta1, beta2, eps, 1.0f - std::pow(beta1, n), 1.0f - std::pow(beta2, n)};
}

// Adam on layer l; S > 1: its weight gradient is still in S partial products in the workspace; g: its bias gradient is
// still to be summed over the M rows of g.
void adam_layer(cloudsc_mlp* m, int l, int S, const bf16* g, int M, const AdamStep& a, hipStream_t s) {
  const size_t nw = (size_t)m->din[l] * m->dout[l];
  const mlp::AdamArgs p{m->w[l],  m->mw[l], m->vw[l], m->gw[l],   m->ws, nw,      m->wb[l], m->b[l], m->mb[l],
                        m->vb[l], m->gb[l], g, M, m->dout[l], a.lr, a.beta1, a.beta2, a.eps, a.bc1, a.bc2};
  static_assert(mlp::MAX_SPLIT == 4, "splits are 1, 2 or 4");
  const dim3 grid(m->dout[l] / mlp::NC + blocks(nw / 4, 256));
  if (S == 4)
    hipLaunchKernelGGL(mlp::adam_update<4>, grid, dim3(256), 0, s, p);
  else if (S == 2)
    hipLaunchKernelGGL(mlp::adam_update<2>, grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL(mlp::adam_update<1>, grid, dim3(256), 0, s, p);
}

// dW = G^T X over the batch (C[dout x din], contraction over M rows).  With few output tiles (one 128x128 tile per CU or
// less) the contraction is split in S stretches over the grid's z dimension, each into its own partial product in the
// workspace; they are added in split order (deterministic) by sum_splits or by Adam.  Returns S in *splits.
hipError_t weight_gradient(cloudsc_mlp* m, const bf16* g, const bf16* x, int dout, int din, int M, float* gw,
                           int* splits, hipStream_t s) {
  const long tiles = (long)(dout / mlp::BM) * (din / mlp::BN);
  int S = 1;
  while (S < mlp::MAX_SPLIT && tiles * S < 256 && (M / (2 * S)) % mlp::BK == 0 && M / (2 * S) >= 512) S *= 2;
  if ((size_t)S * dout * din > m->ws_elems) S = 1;
  *splits = S;
  mlp::EpiArgs ep{};
  ep.c = S > 1 ? m->ws : gw;
  ep.ldc = din;
  ep.zstride = (long)dout * din;
  return gemm<mlp::EPI_F32, true, true>(g, dout, x, din, dout, din, M / S, ep, s, S);
}

// Backward pass from the output gradient in g0; fills gw, gb.  With adam, each layer is updated as soon as its weights
// have been read (its input gradient formed).
hipError_t backward(cloudsc_mlp* m, const bf16* x, int M, const AdamStep* adam, hipStream_t s) {
  hipError_t e = hipSuccess;
  bf16 *g = m->g0, *gn = m->g1;
  for (int l = m->nl - 1; l >= 0 && e == hipSuccess; --l) {
    const int dout = m->dout[l], din = m->din[l];
    int S = 1;
    e = weight_gradient(m, g, l == 0 ? x : m->a[l - 1], dout, din, M, m->gw[l], &S, s);
    if (e != hipSuccess) break;
    if (!adam) {
      hipLaunchKernelGGL(mlp::column_sums, dim3(dout / mlp::NC), dim3(256), 0, s, g, M, dout, m->gb[l]);
      const size_t n = (size_t)dout * din;
      if (S > 1) hipLaunchKernelGGL(mlp::sum_splits, dim3(blocks(n, 256)), dim3(256), 0, s, m->ws, n, S, m->gw[l]);
    }
    if (l > 0) {  // dX_l = G * W_l, then times silu'(Z_{l-1}) -> gradient of the previous layer
      mlp::EpiArgs ed{};
      ed.ldc = din;
      ed.act = gn;
      ed.z = m->z[l - 1];
      e = gemm<mlp::EPI_DHIDDEN, false, true>(g, dout, m->wb[l], din, M, din, dout, ed, s);
    }
    if (adam && e == hipSuccess) adam_layer(m, l, S, g, M, *adam, s);
    std::swap(g, gn);
  }
  if (e == hipSuccess) e = hipGetLastError();
  return e;
}

// Forward, loss and backward of one batch; with adam, the parameter update too.
int train_batch(cloudsc_mlp* m, const bf16* x, const float* t, const float* wgt, int M, const AdamStep* adam,
                hipStream_t s) {
  hipError_t e = mlp::forward(m, x, M, m->y, t, wgt, s);
  if (e == hipSuccess) e = backward(m, x, M, adam, s);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_mlp_gradients", e);
  return CLOUDSC_OK;
}

}  // namespace

namespace mlp {
int train_step(cloudsc_mlp* m, const bf16* x, const float* t, const float* wgt, int M, float lr, hipStream_t s) {
  const int rc = check_batch(m, M);
  if (rc) return rc;
  const AdamStep a = next_step(m, lr, 0.9f, 0.999f, 1e-8f);
  const int e = train_batch(m, x, t, wgt, M, &a, s);
  if (!e) m->step += 1;
  return e;
}
}  // namespace mlp

extern "C" {

int cloudsc_mlp_create(cloudsc_mlp_t** out, int n_in, int n_hidden, int n_hidden_layers, int n_out, int max_batch,
                       uint64_t seed) {
  if (!out) return fail(CLOUDSC_ENULL, "cloudsc_mlp_create: NULL output");
  *out = nullptr;
  if (n_in <= 0 || n_hidden <= 0 || n_out <= 0 || n_hidden_layers < 1 || max_batch <= 0 || n_in % 128 ||
      n_hidden % 128 || n_out % 128 || max_batch % 128)
    return fail(CLOUDSC_EDIMS, "cloudsc_mlp_create: widths and max_batch must be positive multiples of 128");
  int rc = cloudsc_capi::check_device();
  if (rc) return rc;
  cloudsc_mlp* m = new cloudsc_mlp();
  m->nl = n_hidden_layers + 1;
  m->max_batch = max_batch;
  for (int l = 0; l < m->nl; ++l) {
    m->din.push_back(l == 0 ? n_in : n_hidden);
    m->dout.push_back(l == m->nl - 1 ? n_out : n_hidden);
  }
  auto F = [&](size_t n, float** p) { return dev_alloc(m, n * sizeof(float), (void**)p); };
  auto H = [&](size_t n, bf16** p) { return dev_alloc(m, n * sizeof(bf16), (void**)p); };
  m->w.resize(m->nl); m->b.resize(m->nl); m->mw.resize(m->nl); m->vw.resize(m->nl); m->mb.resize(m->nl);
  m->vb.resize(m->nl); m->gw.resize(m->nl); m->gb.resize(m->nl); m->wb.resize(m->nl);
  for (int l = 0; l < m->nl && !rc; ++l) {
    const size_t nw = (size_t)m->din[l] * m->dout[l], nb = m->dout[l];
    rc = F(nw, &m->w[l]) || F(nb, &m->b[l]) || F(nw, &m->mw[l]) || F(nw, &m->vw[l]) || F(nb, &m->mb[l]) ||
         F(nb, &m->vb[l]) || F(nw, &m->gw[l]) || F(nb, &m->gb[l]) || H(nw, &m->wb[l]);
  }
  m->z.resize(m->nl - 1); m->a.resize(m->nl - 1);
  const size_t mh = (size_t)max_batch * n_hidden;
  for (int l = 0; l < m->nl - 1 && !rc; ++l) rc = F(mh, &m->z[l]) || H(mh, &m->a[l]);
  const size_t mg = (size_t)max_batch * std::max(n_hidden, n_out);
  if (!rc) rc = H(mg, &m->g0) || H(mg, &m->g1);
  if (!rc) rc = F((size_t)max_batch * n_out, &m->y) || F(1, &m->loss);
  size_t wmax = 0;
  for (int l = 0; l < m->nl; ++l) wmax = std::max(wmax, (size_t)m->din[l] * m->dout[l]);
  if (!rc) {
    m->ws_elems = (size_t)mlp::MAX_SPLIT * wmax;
    rc = F(m->ws_elems, &m->ws);
  }
  if (rc) {
    rc = CLOUDSC_ENOMEM;
    cloudsc_mlp_destroy(m);
    return rc;
  }
  // He-style initialisation: W ~ N(0, 1/n_in) from Philox (seed, layer, row, col); zero biases and moments.
  std::vector<float> hw;
  hipError_t e = hipSuccess;
  for (int l = 0; l < m->nl && e == hipSuccess; ++l) {
    const size_t nw = (size_t)m->din[l] * m->dout[l];
    hw.resize(nw);
    const double sd = std::sqrt(1.0 / m->din[l]);
    for (int r = 0; r < m->dout[l]; ++r)
      for (int c = 0; c < m->din[l]; ++c)
        hw[(size_t)r * m->din[l] + c] = (float)(sd * synth::draw(seed, 100u + (uint32_t)l, (uint32_t)c, (uint32_t)r).n);
    e = hipMemcpy(m->w[l], hw.data(), nw * sizeof(float), hipMemcpyHostToDevice);
    if (e != hipSuccess) break;
    e = hipMemset(m->b[l], 0, m->dout[l] * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->mw[l], 0, nw * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->vw[l], 0, nw * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->mb[l], 0, m->dout[l] * sizeof(float));
    if (e == hipSuccess) e = hipMemset(m->vb[l], 0, m->dout[l] * sizeof(float));
    if (e == hipSuccess) {
      hipLaunchKernelGGL(mlp::to_bf16, dim3(blocks(nw, 256)), dim3(256), 0, 0, m->w[l], nw, m->wb[l]);
      e = hipGetLastError();
    }
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e != hipSuccess) {
    cloudsc_mlp_destroy(m);
    return fail(CLOUDSC_EHIP, "cloudsc_mlp_create: initialisation", e);
  }
  *out = m;
  return CLOUDSC_OK;
}

int cloudsc_mlp_destroy(cloudsc_mlp_t* m) {
  if (!m) return CLOUDSC_OK;
  for (void* p : m->allocs) (void)hipFree(p);
  delete m;
  return CLOUDSC_OK;
}

int cloudsc_mlp_dims(const cloudsc_mlp_t* m, int* n_layers, int* din, int* dout) {
  if (!m || !n_layers) return fail(CLOUDSC_ENULL, "cloudsc_mlp_dims: NULL argument");
  *n_layers = m->nl;
  for (int l = 0; l < m->nl; ++l) {
    if (din) din[l] = m->din[l];
    if (dout) dout[l] = m->dout[l];
  }
  return CLOUDSC_OK;
}

int cloudsc_mlp_forward(cloudsc_mlp_t* m, const uint16_t* x, int M, float* y, void* stream) {
  if (!m || !x || !y) return fail(CLOUDSC_ENULL, "cloudsc_mlp_forward: NULL argument");
  int rc = check_batch(m, M);
  if (rc) return rc;
  hipError_t e = mlp::forward(m, (const bf16*)x, M, y, nullptr, nullptr, (hipStream_t)stream);
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_mlp_forward", e);
  return CLOUDSC_OK;
}

int cloudsc_mlp_gradients(cloudsc_mlp_t* m, const uint16_t* x, const uint16_t* xT, const float* t, const float* wgt,
                          int M, void* stream) {
  if (!m || !x || !xT || !t || !wgt) return fail(CLOUDSC_ENULL, "cloudsc_mlp_gradients: NULL argument");
  int rc = check_batch(m, M);
  if (rc) return rc;
  return train_batch(m, (const bf16*)x, t, wgt, M, nullptr, (hipStream_t)stream);
}

int cloudsc_mlp_adam(cloudsc_mlp_t* m, float lr, float beta1, float beta2, float eps, void* stream) {
  if (!m) return fail(CLOUDSC_ENULL, "cloudsc_mlp_adam: NULL model");
  hipStream_t s = (hipStream_t)stream;
  const AdamStep a = next_step(m, lr, beta1, beta2, eps);
  m->step += 1;
  for (int l = 0; l < m->nl; ++l) adam_layer(m, l, 1, nullptr, 0, a, s);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_mlp_adam", e);
  return CLOUDSC_OK;
}

int cloudsc_mlp_train_step(cloudsc_mlp_t* m, const uint16_t* x, const uint16_t* xT, const float* t, const float* wgt,
                           int M, float lr, void* stream) {
  if (!m || !x || !xT || !t || !wgt) return fail(CLOUDSC_ENULL, "cloudsc_mlp_gradients: NULL argument");
  return mlp::train_step(m, (const bf16*)x, t, wgt, M, lr, (hipStream_t)stream);
}

// Host copies of one layer's parameters (which: 0 = W [dout x din] fp32, 1 = b, 2 = dW, 3 = db, 4 = last output Y
// [M x n_out] of a training forward, 5 = loss scalar).  set: 0 = device -> host, 1 = host -> device (W, b only;
// refreshes the BF16 copies).
int cloudsc_mlp_param(cloudsc_mlp_t* m, int layer, int which, float* host, size_t n, int set) {
  if (!m || !host) return fail(CLOUDSC_ENULL, "cloudsc_mlp_param: NULL argument");
  if (layer < 0 || layer >= m->nl || which < 0 || which > 5)
    return fail(CLOUDSC_EDIMS, "cloudsc_mlp_param: layer or field out of range");
  const size_t nw = (size_t)m->din[layer] * m->dout[layer], nb = m->dout[layer];
  float* p = nullptr;
  size_t cap = 0;
  switch (which) {
    case 0: p = m->w[layer]; cap = nw; break;
    case 1: p = m->b[layer]; cap = nb; break;
    case 2: p = m->gw[layer]; cap = nw; break;
    case 3: p = m->gb[layer]; cap = nb; break;
    case 4: p = m->y; cap = (size_t)m->max_batch * m->dout[m->nl - 1]; break;
    default: p = m->loss; cap = 1; break;
  }
  if (n > cap) return fail(CLOUDSC_EDIMS, "cloudsc_mlp_param: count exceeds the field size");
  if (set && which > 1) return fail(CLOUDSC_EDIMS, "cloudsc_mlp_param: only W and b can be set");
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess)
    e = set ? hipMemcpy(p, host, n * sizeof(float), hipMemcpyHostToDevice)
            : hipMemcpy(host, p, n * sizeof(float), hipMemcpyDeviceToHost);
  if (e == hipSuccess && set && which == 0) {
    hipLaunchKernelGGL(mlp::to_bf16, dim3(blocks(nw, 256)), dim3(256), 0, 0, m->w[layer], nw, m->wb[layer]);
    e = hipDeviceSynchronize();
  }
  if (e != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_mlp_param", e);
  return CLOUDSC_OK;
}

// Plain product for tests: C[M x N] (fp32) = A[M x K] * B[N x K]^T, bf16 operands, device pointers.
int cloudsc_mlp_gemm_tn(const uint16_t* A, int lda, const uint16_t* B, int ldb, float* C, int ldc, int M, int N,
                        int K, void* stream) {
  if (!A || !B || !C) return fail(CLOUDSC_ENULL, "cloudsc_mlp_gemm_tn: NULL argument");
  if (M <= 0 || N <= 0 || K <= 0 || M % mlp::BM || N % mlp::BN || K % mlp::BK || lda < K || ldb < K || ldc < N ||
      lda % 8 || ldb % 8)
    return fail(CLOUDSC_EDIMS, "cloudsc_mlp_gemm_tn: need M, N multiples of 128, K of 32, lda/ldb >= K and of 8");
  int rc = cloudsc_capi::check_device();
  if (rc) return rc;
  mlp::EpiArgs e{};
  e.c = C;
  e.ldc = ldc;
  hipError_t err = gemm<mlp::EPI_F32>((const bf16*)A, lda, (const bf16*)B, ldb, M, N, K, e, (hipStream_t)stream);
  if (err != hipSuccess) return fail(CLOUDSC_EHIP, "cloudsc_mlp_gemm_tn", err);
  return CLOUDSC_OK;
}

}  // extern "C"
