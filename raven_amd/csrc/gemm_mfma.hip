// gemm_mfma.hip — products of float32, bfloat16 and float16 matrices of any size, stride and
// alignment, operands straight from memory into the matrix instruction.
//
// What bounds it: latency. These are the products that are too small or too ragged for the
// LDS-tiled kernels: a few tiles, so a few waves per compute unit at most, and a chain of loads
// and matrix instructions along K. A wave therefore owns one small result tile (16 x 16, or
// 32 x 32 where there are enough of those to fill the chip). Operands are not staged: a tile's rows
// are read by few waves and come out of L2, and staging would put a barrier into every step of the chain.
//
// float32 sums up to K = MAX_CHAIN are one chain of fused steps, in the order of the LDS-tiled kernels (of
// every eight k-values 0, 4, 1, 5, 2, 6, 3, 7): which kernel a product takes changes no bit of its
// result, and a select on its sign (max(x w, 0) and the mask of its gradient) falls the same way
// whatever the sizes. Past MAX_CHAIN, and for 16-bit elements, `kw` waves of a block share a tile's K: they walk
// their shares side by side and meet in LDS, added in wave order (the same bits on every call).
//
// A lane's fragment of a step is VE (four or eight) k-values of one row. An operand that is
// contiguous along K is read with one 16-byte load at whatever alignment the row has (global
// loads need the element's own); any other operand element by element, lanes side by side along
// the row index. Rows past the edge read the last row (those outputs are not stored); k-values
// past K are zeros in both operands.
//
// Before, these products ran as 128 x 128 blocks: [32,784] x [784,128] float32 was one block,
// 103 us, here 7.5.
#include <algorithm>
#include <mutex>

#include "gemm_args.hpp"
#include "gemm_tile.hpp"
#include "nxh_common.hpp"

namespace gemm_mfma {
using gemm_tile::bf16x8;
using gemm_tile::ElBF16;
using gemm_tile::ElF16;
using gemm_tile::ElF32;
using gemm_tile::f16x8;
using gemm_tile::f32x16;
using gemm_tile::f32x4;
using gemm_tile::V16;

// a register quad read at its elements' own alignment
typedef V16 V16a4 __attribute__((aligned(4)));
typedef V16 V16a2 __attribute__((aligned(2)));

constexpr int MAXW = 8;  // waves of a block at most
constexpr int64_t MAX_CHAIN = 2048;  // float32: a longer K is shared by the waves of a block

// Exchanges x of the wave's upper half with y of its lower half.
__device__ __forceinline__ void swap_halves(float &x, float &y) {
  const auto p = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
  const uint32_t u = p[0], v = p[1];
  x = __builtin_bit_cast(float, u);
  y = __builtin_bit_cast(float, v);
}

// The result tile of a wave. LPG lanes hold the rows of a fragment, 64 / LPG groups of lanes the
// k-values of a step, VE per lane: step width KS.
template <class EL, int T>
struct Tile {
  static constexpr int GROUPS = 64 / T, VE = EL::VE, KS = GROUPS * VE, NE = T * T / 64;
  using Acc = std::conditional_t<T == 32, f32x16, f32x4>;
  __device__ __forceinline__ static void mac(Acc &acc, const V16 &a, const V16 &b) {
    if constexpr (EL::F32 && T == 32) {
      const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
      for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[s], y[s], acc, 0, 0, 0);
    } else if constexpr (EL::F32) {
      mac_ordered(acc, ordered(a), ordered(b));
    } else if constexpr (EL::BF16) {
      const bf16x8 x = __builtin_bit_cast(bf16x8, a), y = __builtin_bit_cast(bf16x8, b);
      if constexpr (T == 32) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, acc, 0, 0, 0);
      else acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
    } else {
      const f16x8 x = __builtin_bit_cast(f16x8, a), y = __builtin_bit_cast(f16x8, b);
      if constexpr (T == 32) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, acc, 0, 0, 0);
      else acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, y, acc, 0, 0, 0);
    }
  }
  // float32, T = 16. The instruction takes a k-value from each quarter of the wave and adds in that order, where
  // two of the 32 x 32 form take k-values s, 4 + s, s + 1, 5 + s: the halves trade, and the bits are the same.
  __device__ __forceinline__ static f32x4 ordered(const V16 &a) {
    const f32x4 x = __builtin_bit_cast(f32x4, a);
    float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
    swap_halves(x0, x1), swap_halves(x2, x3);
    return f32x4{x0, x2, x1, x3};
  }
  __device__ __forceinline__ static void mac_ordered(f32x4 &acc, const f32x4 &x, const f32x4 &y) {
#pragma unroll
    for (int s = 0; s < 4; s++) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], y[s], acc, 0, 0, 0);
  }
  // accumulator element e of a lane
  __device__ __forceinline__ static int row(int e, int lane) {
    return T == 32 ? (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3) : 4 * (lane >> 4) + e;
  }
};

// VE k-values of one row, `p` at the first. KC: one after the other, else `ks` apart.
// TAIL: only the first `left` exist (left may be <= 0).
template <class EL, bool KC, bool TAIL>
__device__ __forceinline__ V16 fragment(const typename EL::S *p, int64_t ks, int left) {
  using S = typename EL::S;
  constexpr int VE = EL::VE;
  using V16u = std::conditional_t<EL::F32, V16a4, V16a2>;
  if constexpr (KC && !TAIL) {
    return *reinterpret_cast<const V16u *>(p);
  } else {
    union {
      S s[VE];
      V16 v;
    } u;
#pragma unroll
    for (int j = 0; j < VE; j++) {
      if constexpr (TAIL) u.s[j] = j < left ? p[KC ? j : j * ks] : (S)0;
      else u.s[j] = p[j * ks];
    }
    return u.v;
  }
}

// U: steps whose loads are in flight together. R = 2: a block of four waves with 2 x 2 tiles each (kw == 1).
template <class EL, bool A_KC, bool B_KC, int T, int U, int R>
__global__ __launch_bounds__(64 * MAXW) void kernel(GemmArgs a, uint32_t tiles_m, uint32_t tiles_n, uint32_t total,
                                                    int kw) {
  using S = typename EL::S;
  using TT = Tile<EL, T>;
  constexpr int VE = TT::VE, KS = TT::KS, NE = TT::NE;
  extern __shared__ __attribute__((aligned(16))) float fold[];  // [waves][NE][64]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int part = wave % kw;
  uint32_t t = blockIdx.x * (uint32_t)(waves / kw) + wave / kw;
  if constexpr (R > 1) {
    // (the tiles are those of a block of 2 x 2 waves; blocks with the same id modulo 8 share an L2 and get
    // a run of neighbours)
    t = blockIdx.x;
    if ((total & 7u) == 0) t = (t & 7u) * (total >> 3) + (t >> 3);
  }
  bool live = t < total;
  int64_t ao = 0, bo = 0, co = 0, m0 = 0, n0 = 0;
  if (live) {
    const uint32_t per = tiles_m * tiles_n, b = t / per, r = t - b * per;
    batch_decode(a.batch, b, ao, bo, co);
    m0 = (int64_t)(r / tiles_n) * (T * R);
    n0 = (int64_t)(r % tiles_n) * (T * R);
    if constexpr (R > 1) {
      m0 = 2 * m0 + (wave >> 1) * (T * R);
      n0 = 2 * n0 + (wave & 1) * (T * R);
      live = m0 < a.M && n0 < a.N;
    }
  }
  typename TT::Acc acc[R][R];
#pragma unroll
  for (int i = 0; i < R * R; i++)
#pragma unroll
    for (int e = 0; e < NE; e++) acc[i / R][i % R][e] = 0.0f;
  const int steps = (int)((a.K + KS - 1) / KS);
  const int per_wave = (steps + kw - 1) / kw;
  const int s0 = part * per_wave, s1 = s0 + per_wave < steps ? s0 + per_wave : steps;
  if (live && s0 < s1) {
    const int kg = lane / T * VE;
    const int64_t aks = A_KC ? 1 : a.acs, bks = B_KC ? 1 : a.brs;
    const int64_t stepA = (int64_t)KS * aks, stepB = (int64_t)KS * bks;
    const S *pA[R], *pB[R];
#pragma unroll
    for (int i = 0; i < R; i++) {
      const int64_t ra = m0 + i * T + lane % T, rb = n0 + i * T + lane % T;
      pA[i] = (const S *)a.A + ao + (ra < a.M ? ra : a.M - 1) * a.ars + ((int64_t)s0 * KS + kg) * aks;
      pB[i] = (const S *)a.B + bo + (rb < a.N ? rb : a.N - 1) * a.bcs + ((int64_t)s0 * KS + kg) * bks;
    }
    auto multiply = [&](const V16(&fa)[R], const V16(&fb)[R]) {
#pragma unroll
      for (int i = 0; i < R; i++)
#pragma unroll
        for (int j = 0; j < R; j++) TT::mac(acc[i][j], fa[i], fb[j]);
    };
    const int full = a.K / KS < s1 ? (int)(a.K / KS) : s1;  // steps before this one are whole
    for (int s = s0; s < full; s += U) {
      V16 fa[U][R], fb[U][R];
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s + u < full) {
#pragma unroll
          for (int i = 0; i < R; i++) {
            fa[u][i] = fragment<EL, A_KC, false>(pA[i] + u * stepA, aks, 0);
            fb[u][i] = fragment<EL, B_KC, false>(pB[i] + u * stepB, bks, 0);
          }
        }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (s + u < full) multiply(fa[u], fb[u]);
      const int64_t on = full - s < U ? full - s : U;
#pragma unroll
      for (int i = 0; i < R; i++) pA[i] += on * stepA, pB[i] += on * stepB;
    }
    if (full < s1) {  // the last step of K, not a whole one; the pointers stand at it
      const int left = (int)(a.K - (int64_t)full * KS) - kg;
      V16 fa[R], fb[R];
#pragma unroll
      for (int i = 0; i < R; i++) {
        fa[i] = fragment<EL, A_KC, true>(pA[i], aks, left);
        fb[i] = fragment<EL, B_KC, true>(pB[i], bks, left);
      }
      multiply(fa, fb);
    }
  }
  S *C = (S *)a.C + co;
  auto put = [&](int i, int j, int e, float x) {
    const int64_t row = m0 + i * T + TT::row(e, lane), col = n0 + j * T + lane % T;
    if (row >= a.M || col >= a.N) return;
    if constexpr (EL::F32) C[row * a.crs + col * a.ccs] = x;
    else C[row * a.crs + col * a.ccs] = EL::BF16 ? f32_to_bf16(x) : f32_to_f16(x);
  };
  if (kw == 1) {
    if (!live) return;
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int j = 0; j < R; j++)
#pragma unroll
        for (int e = 0; e < NE; e++) put(i, j, e, acc[i][j][e]);
    return;
  }
#pragma unroll
  for (int e = 0; e < NE; e++) fold[(wave * NE + e) * 64 + lane] = acc[0][0][e];
  __syncthreads();
  if (!live) return;
  const float *first = fold + (wave - part) * NE * 64 + lane;
  for (int e = part; e < NE; e += kw) {
    float sum = first[e * 64];
    for (int w = 1; w < kw; w++) sum += first[(w * NE + e) * 64];
    put(0, 0, e, sum);
  }
}

// A float32 tile of 16 x 16 whose K is one chain, where there are at most two tiles to a unit: the chain is
// one wave's (54 ns a step of 16 k-values), and what that wave can have in flight by itself does not feed it.
// All CW waves of the block fetch CS steps each into LDS, in the order in which the instruction takes
// them, while the stage before is summed ([38,1754] x [1754,86]: 12.8 us, a wave by itself 19.4; [32,784] x
// [784,128]: 7.5 and 10.1; K in eight sums, which is not the same result, 7.4 and 5.2).
constexpr int CW = 8;
template <bool A_KC, bool B_KC, int CS>
__global__ __launch_bounds__(64 * CW) void chain_kernel(GemmArgs a, uint32_t tiles_m, uint32_t tiles_n) {
  using TT = Tile<ElF32, 16>;
  constexpr int KS = TT::KS, PER_STAGE = CW * CS;
  extern __shared__ __attribute__((aligned(16))) f32x4 stage[];  // [2][PER_STAGE][A, B][64]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t per = tiles_m * tiles_n, b = blockIdx.x / per, r = blockIdx.x - b * per;
  int64_t ao, bo, co;
  batch_decode(a.batch, b, ao, bo, co);
  const int64_t m0 = (int64_t)(r / tiles_n) * 16, n0 = (int64_t)(r % tiles_n) * 16;
  const int kg = lane / 16 * TT::VE;
  const int64_t aks = A_KC ? 1 : a.acs, bks = B_KC ? 1 : a.brs;
  const int64_t ra = m0 + lane % 16, rb = n0 + lane % 16;
  const float *pA = (const float *)a.A + ao + (ra < a.M ? ra : a.M - 1) * a.ars + kg * aks;
  const float *pB = (const float *)a.B + bo + (rb < a.N ? rb : a.N - 1) * a.bcs + kg * bks;
  const int steps = (int)((a.K + KS - 1) / KS), full = (int)(a.K / KS);
  V16 fa[CS], fb[CS];
  auto fetch = [&](int first) {
#pragma unroll
    for (int u = 0; u < CS; u++) {
      const int s = first + wave * CS + u;
      const int64_t k = (int64_t)s * KS;
      if (s < full) {
        fa[u] = fragment<ElF32, A_KC, false>(pA + k * aks, aks, 0);
        fb[u] = fragment<ElF32, B_KC, false>(pB + k * bks, bks, 0);
      } else if (s < steps) {  // the last step of K, not a whole one
        fa[u] = fragment<ElF32, A_KC, true>(pA + k * aks, aks, (int)(a.K - k) - kg);
        fb[u] = fragment<ElF32, B_KC, true>(pB + k * bks, bks, (int)(a.K - k) - kg);
      }
    }
  };
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  fetch(0);
  for (int first = 0, at = 0; first < steps; first += PER_STAGE, at ^= PER_STAGE) {
    f32x4 *mine = stage + (at + wave * CS) * 128 + lane;
#pragma unroll
    for (int u = 0; u < CS; u++) {
      mine[u * 128] = TT::ordered(fa[u]);
      mine[u * 128 + 64] = TT::ordered(fb[u]);
    }
    fetch(first + PER_STAGE);
    // (also: wave 0 is through with the stage that is written next)
    __syncthreads();
    if (wave == 0) {
      const f32x4 *p = stage + at * 128 + lane;
      const int n = steps - first < PER_STAGE ? steps - first : PER_STAGE;
      // (four steps' operands are on their way while the four before are summed; past n: the stage's own memory)
      constexpr int AHEAD = CS > 2 ? 4 : 2;
      f32x4 x[2][AHEAD], y[2][AHEAD];
      auto take = [&](int set, int s) {
#pragma unroll
        for (int j = 0; j < AHEAD; j++) x[set][j] = p[(s + j) * 128], y[set][j] = p[(s + j) * 128 + 64];
      };
      take(0, 0);
      for (int s = 0; s < n; s += 2 * AHEAD) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          if (s + (h + 1) * AHEAD < PER_STAGE) take(h ^ 1, s + (h + 1) * AHEAD);
#pragma unroll
          for (int j = 0; j < AHEAD; j++)
            if (s + h * AHEAD + j < n) TT::mac_ordered(acc, x[h][j], y[h][j]);
        }
      }
    }
  }
  if (wave > 0) return;
  float *C = (float *)a.C + co;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int64_t row = m0 + TT::row(e, lane), col = n0 + lane % 16;
    if (row < a.M && col < a.N) C[row * a.crs + col * a.ccs] = acc[e];
  }
}
template <bool A_KC, bool B_KC, int CS>
static int launch_chain(nxh_context *ctx, const GemmArgs &a, uint32_t tiles_m, uint32_t tiles_n, uint32_t total) {
  constexpr int LDS = 2 * CW * CS * 2 * 64 * (int)sizeof(f32x4);
  auto kern = chain_kernel<A_KC, B_KC, CS>;
  static std::once_flag once;  // allow > 64 KiB of dynamic LDS
  static hipError_t attr_status = hipSuccess;
  std::call_once(once, [&] { attr_status = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, LDS); });
  NXH_HIP("matmul", attr_status);
  hipLaunchKernelGGL(kern, dim3(total), dim3(64 * CW), LDS, ctx->stream, a, tiles_m, tiles_n);
  NXH_HIP("matmul", hipGetLastError());
  return NXH_OK;
}
template <int CS>
static int launch_chain_oriented(nxh_context *ctx, const GemmArgs &a, uint32_t tiles_m, uint32_t tiles_n, uint32_t total) {
  if (a.acs == 1) return a.brs == 1 ? launch_chain<true, true, CS>(ctx, a, tiles_m, tiles_n, total) : launch_chain<true, false, CS>(ctx, a, tiles_m, tiles_n, total);
  return a.brs == 1 ? launch_chain<false, true, CS>(ctx, a, tiles_m, tiles_n, total) : launch_chain<false, false, CS>(ctx, a, tiles_m, tiles_n, total);
}

template <class EL, int T, int U, int R>
static void launch(nxh_context *ctx, const GemmArgs &a, uint32_t tiles_m, uint32_t tiles_n, uint32_t total, int kw) {
  const int waves = std::max(kw, 4), per_block = waves / kw;
  const size_t lds = kw > 1 ? sizeof(float) * (size_t)waves * T * T : 0;
  const dim3 grid(R > 1 ? total : (total + per_block - 1) / per_block), block(64 * waves);
  // two-byte elements read one by one take a register each: half the steps in flight
  constexpr int UE = EL::F32 || U <= 2 ? U : U / 2;
  if (a.acs == 1 && a.brs == 1) hipLaunchKernelGGL((kernel<EL, true, true, T, U, R>), grid, block, lds, ctx->stream, a, tiles_m, tiles_n, total, kw);
  else if (a.acs == 1) hipLaunchKernelGGL((kernel<EL, true, false, T, UE, R>), grid, block, lds, ctx->stream, a, tiles_m, tiles_n, total, kw);
  else if (a.brs == 1) hipLaunchKernelGGL((kernel<EL, false, true, T, UE, R>), grid, block, lds, ctx->stream, a, tiles_m, tiles_n, total, kw);
  else hipLaunchKernelGGL((kernel<EL, false, false, T, UE, R>), grid, block, lds, ctx->stream, a, tiles_m, tiles_n, total, kw);
}

template <class EL>
static int run(nxh_context *ctx, const GemmArgs &a, uint32_t nbatch) {
  const int64_t cus = ctx->compute_units > 0 ? ctx->compute_units : 256;
  auto count = [&](int64_t t) { return (double)((a.M + t - 1) / t) * (double)((a.N + t - 1) / t) * nbatch; };
  // Tiles: as large as leaves enough waves. 32 x 32 reads half of what 16 x 16 reads, and from half a
  // tile per unit on sharing K among eight waves fills the chip; a chain of float32 steps is four times as long in a 32 x 32
  // tile, which pays from two tiles per unit on ([1554,244] x [244,347]: 9.0 us against 10.6, [500,500]^2: 13.2
  // against 9.8). Blocks of 2 x 2 waves with 64 x 64 each only where their waves alone fill it ([2048,2048]^2 into
  // every second column, float32: 170 us against 283 on 32 x 32; [501,501]^2: 41 against 10).
  const bool chain = EL::F32 && a.K <= MAX_CHAIN;
  const bool wide = chain ? count(32) >= 2.0 * cus && a.M > 16 && a.N > 16 : count(32) >= 0.5 * cus;
  const int t = count(64) >= 4.0 * cus && a.M > 64 && a.N > 64 ? 128 : wide ? 32 : 16;
  if (count(t) > (double)0x7fffffff || a.K > (int64_t)0x7fffffff) return -1;
  const uint32_t tm = (uint32_t)((a.M + t - 1) / t), tn = (uint32_t)((a.N + t - 1) / t), total = tm * tn * nbatch;
  const int ks = (t == 16 ? 4 : 2) * EL::VE;
  const int64_t steps = (a.K + ks - 1) / ks;
  // waves that share a tile's K: as many as put two waves on every SIMD, and no fewer than two steps each
  int kw = 1;
  while (!chain && t < 128 && kw < MAXW && (int64_t)total * kw < 8 * cus && steps >= 4 * kw) kw *= 2;
  const bool deep = (steps + kw - 1) / kw > 4;  // steps a wave has to have in flight
  nxh_set_path("gemm_mfma");
  if constexpr (EL::F32) {
    if (chain && t == 16 && a.K > 128) {
      if (total <= cus) return launch_chain_oriented<4>(ctx, a, tm, tn, total);
      if (total <= 2 * cus) return launch_chain_oriented<2>(ctx, a, tm, tn, total);
    }
  }
  if (t == 128) launch<EL, 32, 4, 2>(ctx, a, tm, tn, total, 1);
  else if (t == 32 && deep) launch<EL, 32, 8, 1>(ctx, a, tm, tn, total, kw);
  else if (t == 32) launch<EL, 32, 4, 1>(ctx, a, tm, tn, total, kw);
  else if (deep) launch<EL, 16, 8, 1>(ctx, a, tm, tn, total, kw);
  else launch<EL, 16, 4, 1>(ctx, a, tm, tn, total, kw);
  NXH_HIP("matmul", hipGetLastError());
  return NXH_OK;
}

}  // namespace gemm_mfma

int nxh_gemm_mfma(nxh_context *ctx, int dtype, const GemmArgs &a, uint32_t nbatch) {
  if (dtype == NXH_F32) return gemm_mfma::run<gemm_mfma::ElF32>(ctx, a, nbatch);
  if (dtype == NXH_BF16) return gemm_mfma::run<gemm_mfma::ElBF16>(ctx, a, nbatch);
  return gemm_mfma::run<gemm_mfma::ElF16>(ctx, a, nbatch);
}
