// gemm_mfma.hip — products of float32, bfloat16 and float16 matrices of any size, stride and
// alignment, operands straight from memory into the matrix instruction.
//
// What bounds it: latency. These are the products that are too small or too ragged for the
// LDS-tiled kernels: a few tiles, so a few waves per compute unit at most, and a chain of loads
// and matrix instructions along K. A wave therefore owns one small result tile (16 x 16, or
// 32 x 32 where there are enough of those to fill the chip) and a share of K: the `kw` waves
// of a group walk their shares side by side and meet in LDS, added in wave order (the same bits
// on every call). Operands are not staged: a tile's rows are read by few waves and come out
// of L2, and staging would put a barrier into every step of the chain.
//
// A lane's fragment of a step is VE (four or eight) k-values of one row. An operand that is
// contiguous along K is read with one 16-byte load at whatever alignment the row has (global
// loads need the element's own); any other operand element by element, lanes side by side along
// the row index. Rows past the edge read the last row (those outputs are not stored); k-values
// past K are zeros in both operands.
//
// Before, these products ran as 128 x 128 blocks: [32,784] x [784,128] float32 was one block,
// 103 us; here it is 16 blocks of eight waves.
#include <algorithm>

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

// The result tile of a wave. LPG lanes hold the rows of a fragment, 64 / LPG groups of lanes the
// k-values of a step, VE per lane: step width KS.
template <class EL, int T>
struct Tile {
  static constexpr int GROUPS = 64 / T, VE = EL::VE, KS = GROUPS * VE, NE = T * T / 64;
  using Acc = std::conditional_t<T == 32, f32x16, f32x4>;
  __device__ __forceinline__ static void mac(Acc &acc, const V16 &a, const V16 &b) {
    if constexpr (EL::F32) {
      const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
      for (int s = 0; s < 4; s++) {
        if constexpr (T == 32) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(x[s], y[s], acc, 0, 0, 0);
        else acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], y[s], acc, 0, 0, 0);
      }
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
  // tile per unit on sharing K among eight waves fills the chip ([501,501]^2 float32: 7.9 us against
  // 8.7); blocks of 2 x 2 waves with 64 x 64 each only where their waves alone do ([2048,2048]^2 into
  // every second column: 170 us against 283 on 32 x 32; [501,501]^2: 41).
  const int t = count(64) >= 4.0 * cus && a.M > 64 && a.N > 64 ? 128 : count(32) >= 0.5 * cus ? 32 : 16;
  if (count(t) > (double)0x7fffffff || a.K > (int64_t)0x7fffffff) return -1;
  const uint32_t tm = (uint32_t)((a.M + t - 1) / t), tn = (uint32_t)((a.N + t - 1) / t), total = tm * tn * nbatch;
  const int ks = (t == 16 ? 4 : 2) * EL::VE;
  const int64_t steps = (a.K + ks - 1) / ks;
  // waves that share a tile's K: as many as put two waves on every SIMD, and no fewer than two steps each
  int kw = 1;
  while (t < 128 && kw < MAXW && (int64_t)total * kw < 8 * cus && steps >= 4 * kw) kw *= 2;
  const bool deep = (steps + kw - 1) / kw > 4;  // steps a wave has to have in flight
  nxh_set_path("gemm_mfma");
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
