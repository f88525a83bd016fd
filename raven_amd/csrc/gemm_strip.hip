// gemm_strip.hip — a few rows times a 16-bit matrix in memory order ([K][N], unit-stride rows), plain or
// with the fused linear's bias and residual: a network's layer over some tens to hundreds of tokens.
//
// What bounds it: latency, and what one compute unit can have in flight. There are too few result tiles
// to fill the chip, so a block is one tile, 16, 32 or 64 rows by 64 columns, and its eight waves cut K
// among them; they meet in LDS and are added in wave order (the same bits on every call, whatever the
// tile: K is cut alike for all). Nothing is staged: a step's operands go from memory into registers, four
// steps in flight a wave. A fragment of the matrix instruction holds eight k-values of one column, and
// rows of B run along the columns: a lane reads four neighbouring columns of eight rows (8 bytes each, a
// row of the tile is one 128-byte line) and turns them into the fragments of four column tiles, so a
// tile's columns are dealt out four to a lane and each lane stores four neighbours.
//
// [48,3072] x [3072,768] bfloat16: 29 us as 12 whole blocks of 128 x 64 and 9.5 as such blocks cut along K, here 7.8 (36 tiles, each cut among six
// blocks; one block a tile 11.2: a unit draws some 56 bytes a nanosecond and a tile reads 491 KB);
// [48,768] x [768,768]: 7.3 to 5.1 between launches of its own kind; [512,3072] x [3072,768]: 30 to 15.
#include <algorithm>

#include "gemm_args.hpp"
#include "gemm_strip.hpp"
#include "gemm_tile.hpp"
#include "nxh_common.hpp"

namespace gemm_strip {
using gemm_tile::bf16x8;
using gemm_tile::ElBF16;
using gemm_tile::ElF16;
using gemm_tile::f16x8;
using gemm_tile::f32x4;
using gemm_tile::V16;
typedef __attribute__((ext_vector_type(2))) uint32_t V8;
// read at their elements' own alignment
typedef V16 V16a2 __attribute__((aligned(2)));
typedef V8 V8a2 __attribute__((aligned(2)));

constexpr int KS = 32;   // k-values of a step
constexpr int BN = 64;   // columns of a tile
constexpr int MAXW = 8;  // waves that share a tile's K

template <class EL>
__device__ __forceinline__ void mac(f32x4 &acc, const V16 &a, const V16 &b) {
  if constexpr (EL::BF16)
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
  else
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
}

// Tile t of a launch: the operands' offsets of its batch and member, its first row, this lane's four columns.
template <bool EPI>
struct Where {
  int64_t ao = 0, bo = 0, co = 0, ro = 0, m0, col;
  const uint16_t *bias;
  __device__ __forceinline__ Where(const Args &a, uint32_t t, int rows, int lane) {
    uint32_t tn = t % a.tiles_n;
    t /= a.tiles_n;
    m0 = (int64_t)(t % a.tiles_m) * rows;
    uint32_t idx = t / a.tiles_m;
    bias = (const uint16_t *)a.bias;
    if constexpr (EPI) {
      if (a.ngroup > 1) {
        const uint32_t member = tn / a.gtn;
        tn -= member * a.gtn;
        if (member) {
          bo = member == 1 ? a.goff_b[0] : a.goff_b[1];
          co = member == 1 ? a.goff_c[0] : a.goff_c[1];
          if (bias) bias += member == 1 ? a.goff_bias[0] : a.goff_bias[1];
        }
      }
    }
#pragma unroll
    for (int i = 3; i >= 0; i--) {
      if (i < a.nbd) {
        const uint32_t q = idx / a.bshape[i], c = idx - q * a.bshape[i];
        idx = q;
        ao += (int64_t)c * a.ba[i];
        bo += (int64_t)c * a.bb[i];
        co += (int64_t)c * a.bc[i];
        if constexpr (EPI) ro += (int64_t)c * a.br[i];
      }
    }
    // past the edge the last four columns (computed twice, to the same bits)
    const int64_t want = (int64_t)tn * BN + (lane & 15) * 4;
    col = want + 4 <= a.N ? want : a.N - 4;
  }
};
// Piece p of a tile: this lane's four columns of row 4 (lane / 16) + p % 4 of row tile p / 4.
template <class EL, bool EPI>
__device__ __forceinline__ void put(const Args &a, const Where<EPI> &w, int p, int lane, const f32x4 &x) {
  const int64_t row = w.m0 + (p >> 2) * 16 + 4 * (lane >> 4) + (p & 3);
  if (row >= a.M) return;
  V8 v = {gemm_tile::epi_narrow2<EL>(x[0], x[1]), gemm_tile::epi_narrow2<EL>(x[2], x[3])};
  if constexpr (EPI) {
    if (w.bias) {
      const V8 y = *reinterpret_cast<const V8a2 *>(w.bias + w.col);
      v = V8{gemm_tile::epi_add2<EL>(v[0], y[0]), gemm_tile::epi_add2<EL>(v[1], y[1])};
    }
    if (a.gelu) v = V8{gemm_tile::epi_gelu2<EL>(v[0], a.gc[0], a.gc[1], a.gc[2], a.gc[3]), gemm_tile::epi_gelu2<EL>(v[1], a.gc[0], a.gc[1], a.gc[2], a.gc[3])};
    if (a.R) {
      const V8 y = *reinterpret_cast<const V8a2 *>((const uint16_t *)a.R + w.ro + row * a.ldr + w.col);
      v = V8{gemm_tile::epi_add2<EL>(v[0], y[0]), gemm_tile::epi_add2<EL>(v[1], y[1])};
    }
  }
  *reinterpret_cast<V8a2 *>((uint16_t *)a.C + w.co + row * a.ldc + w.col) = v;
}

// MT: row tiles of 16. U: steps in flight. kw: waves of the block. parts: waves that share a tile's K,
// kw of them in each of parts / kw blocks (blockIdx.y), whose sums go to `partial` if there are several.
template <class EL, int MT, int U, bool EPI>
__global__ __launch_bounds__(64 * MAXW) void kernel(Args a, int kw, int parts, uint32_t tiles, f32x4 *partial) {
  using S = uint16_t;
  extern __shared__ __attribute__((aligned(16))) float fold[];  // [waves][MT * 4][64][4]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Where<EPI> w(a, blockIdx.x, 16 * MT, lane);
  const int l16 = lane & 15, kg = (lane >> 4) * 8;

  f32x4 acc[MT][4];
#pragma unroll
  for (int t = 0; t < MT; t++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[t][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  const int steps = (int)(a.K / KS);
  const int part = (int)blockIdx.y * kw + wave, base = steps / parts, more = steps % parts;
  const int s0 = part * base + (part < more ? part : more), n = base + (part < more);
  // uniform addresses that move, 32-bit offsets of the lanes that don't
  const char *pA = (const char *)((const S *)a.A + w.ao + w.m0 * a.lda + (int64_t)s0 * KS);
  const char *pB = (const char *)((const S *)a.B + w.bo + (int64_t)s0 * KS * a.ldb);
  uint32_t oa[MT];
  const uint32_t ob = (uint32_t)((kg * a.ldb + w.col) * 2);
#pragma unroll
  for (int t = 0; t < MT; t++) {
    const int64_t row = w.m0 + t * 16 + l16;
    oa[t] = (uint32_t)((((row < a.M ? row : a.M - 1) - w.m0) * a.lda + kg) * 2);
  }
  const int64_t rowB = a.ldb * 2;
  V16 fa[U][MT];
  V8 fb[U][8];
  auto fetch = [&](int u) {
#pragma unroll
    for (int k = 0; k < 8; k++) fb[u][k] = *reinterpret_cast<const V8a2 *>(pB + k * rowB + ob);
#pragma unroll
    for (int t = 0; t < MT; t++) fa[u][t] = *reinterpret_cast<const V16a2 *>(pA + oa[t]);
    pB += KS * rowB;
    pA += KS * 2;
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      // column j of the four: its eight k-values, out of the eight rows read
      constexpr uint32_t LO = 0x05040100, HI = 0x07060302;
      V16 b;
#pragma unroll
      for (int d = 0; d < 4; d++)
        b[d] = __builtin_amdgcn_perm(fb[u][2 * d + 1][j >> 1], fb[u][2 * d][j >> 1], (j & 1) ? HI : LO);
#pragma unroll
      for (int t = 0; t < MT; t++) mac<EL>(acc[t][j], fa[u][t], b);
    }
  };
#pragma unroll
  for (int u = 0; u < U; u++)
    if (u < n) fetch(u);
  int s = 0;
  for (; s + 2 * U <= n; s += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      multiply(u);
      fetch(u);
    }
  }
  for (; s < n; s += U) {
#pragma unroll
    for (int u = 0; u < U; u++)
      if (s + u < n) {
        multiply(u);
        if (s + u + U < n) fetch(u);
      }
  }

  const int left = (int)(a.K % KS);
  if (left && part == parts - 1) {  // what K has past the last whole step: its own elements, zeros after them
    const S *qB = (const S *)pB;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      fb[0][k] = V8{0, 0};
      if (kg + k < left) fb[0][k] = *reinterpret_cast<const V8a2 *>((const char *)(qB + k * a.ldb) + ob);
    }
#pragma unroll
    for (int t = 0; t < MT; t++) {
      const S *qA = (const S *)(pA + oa[t]);
      union {
        S s[8];
        V16 v;
      } x;
#pragma unroll
      for (int k = 0; k < 8; k++) x.s[k] = kg + k < left ? qA[k] : (S)0;
      fa[0][t] = x.v;
    }
    multiply(0);
  }

  auto piece = [&](int p) { return f32x4{acc[p >> 2][0][p & 3], acc[p >> 2][1][p & 3], acc[p >> 2][2][p & 3], acc[p >> 2][3][p & 3]}; };
  if (!EPI && kw == 1) {  // (a linear's K is that of several waves)
#pragma unroll
    for (int p = 0; p < MT * 4; p++) put<EL, EPI>(a, w, p, lane, piece(p));
    return;
  }
  f32x4 *mine = reinterpret_cast<f32x4 *>(fold) + (wave * MT * 4) * 64 + lane;
#pragma unroll
  for (int p = 0; p < MT * 4; p++) mine[p * 64] = piece(p);
  __syncthreads();
  const f32x4 *first = reinterpret_cast<const f32x4 *>(fold) + lane;
  for (int p = wave; p < MT * 4; p += kw) {
    f32x4 sum = first[p * 64];
    for (int v = 1; v < kw; v++) sum += first[(v * MT * 4 + p) * 64];
    if (partial) partial[(((size_t)blockIdx.y * tiles + blockIdx.x) * (MT * 4) + p) * 64 + lane] = sum;
    else put<EL, EPI>(a, w, p, lane, sum);
  }
}
// The partial sums of `blocks` blocks a tile of 16 rows, added in order: a wave per piece.
template <class EL, bool EPI>
__global__ __launch_bounds__(256) void finish_kernel(Args a, int blocks, uint32_t tiles, const f32x4 *partial) {
  const int lane = threadIdx.x & 63, p = threadIdx.x >> 6;
  const Where<EPI> w(a, blockIdx.x, 16, lane);
  const f32x4 *q = partial + ((size_t)blockIdx.x * 4 + p) * 64 + lane;
  f32x4 sum = q[0];
  for (int b = 1; b < blocks; b++) sum += q[(size_t)b * tiles * 256];
  put<EL, EPI>(a, w, p, lane, sum);
}

template <class EL, int MT, bool EPI>
static int launch(nxh_context *ctx, Args &g, int kw, int blocks) {
  auto kern = kernel<EL, MT, 4, EPI>;
  const size_t lds = kw > 1 ? (size_t)kw * MT * 16 * 64 * sizeof(float) : 0;
  static std::once_flag once;  // allow > 64 KiB of dynamic LDS
  static hipError_t attr_status = hipSuccess;
  std::call_once(once, [&] {
    attr_status = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                      MAXW * MT * 16 * 64 * (int)sizeof(float));
  });
  NXH_HIP("matmul", attr_status);
  g.tiles_m = (uint32_t)((g.M + 16 * MT - 1) / (16 * MT));
  g.tiles_n = g.gtn = (uint32_t)((g.N + BN - 1) / BN);
  if (EPI) g.tiles_n *= g.ngroup;
  const uint32_t tiles = g.tiles_m * g.tiles_n * g.nbatch;
  void *partial = nullptr;
  if (blocks > 1)
    if (int rc = nxh_alloc_locked(ctx, (size_t)blocks * tiles * 16 * 64 * sizeof(float), &partial)) return rc;
  nxh_set_path(EPI ? "linear_strip" : "gemm_strip");
  hipLaunchKernelGGL(kern, dim3(tiles, blocks), dim3(64 * kw), lds, ctx->stream, g, kw, kw * blocks, tiles, (f32x4 *)partial);
  hipError_t e = hipGetLastError();
  if (blocks > 1) {
    if (e == hipSuccess) {
      hipLaunchKernelGGL((finish_kernel<EL, EPI>), dim3(tiles), dim3(256), 0, ctx->stream, g, blocks, tiles, (const f32x4 *)partial);
      e = hipGetLastError();
    }
    nxh_free_locked(ctx, partial);
  }
  NXH_HIP("matmul", e);
  return NXH_OK;
}
template <class EL, bool EPI>
static int run(nxh_context *ctx, Args &g) {
  const int64_t cus = ctx->compute_units > 0 ? ctx->compute_units : 256;
  // (how K is cut is decided without the group, so that a member has the bits of its own call)
  const int kw = (int)std::max<int64_t>(1, std::min<int64_t>(MAXW, g.K / KS));
  const int blocks = nxh_gemm_strip_blocks(ctx, g.M, g.N, g.K, g.nbatch);
  // the smallest tile whose blocks don't outnumber the units: a second block on a unit waits for the
  // same loads as the first ([512,3072] x [3072,768]: 384 tiles of 16 rows 20.6 us, 192 of 32 rows 15.4;
  // [256,768] x [768,3072]: 768 tiles 10.7, 384 11.3, 192 of 64 rows 8.7)
  auto tiles = [&](int64_t bm) { return ((g.M + bm - 1) / bm) * ((g.N + BN - 1) / BN) * (int64_t)g.nbatch * (EPI ? g.ngroup : 1); };
  if (tiles(16) > 0x7fffffffLL || (EPI && kw == 1)) return -1;
  if (blocks > 1 || g.M <= 16 || tiles(16) <= cus) return launch<EL, 1, EPI>(ctx, g, kw, blocks);
  if (g.M <= 32 || tiles(32) <= cus) return launch<EL, 2, EPI>(ctx, g, kw, 1);
  return launch<EL, 4, EPI>(ctx, g, kw, 1);
}
}  // namespace gemm_strip

// With one block a tile and less than half the units in use, a long K is cut among several blocks whose
// sums a second kernel adds: a block's share of B and A comes at about 56 bytes a nanosecond (2.9 ns per
// k-value of a tile of 16 rows), the second launch costs some 3.5 us and the sums a trip through memory.
// bfloat16 [48,3072] x [3072,768] 11.2 us whole and 7.8 cut, float16 [15,11109] x [11109,314] 16.4 (35 in
// the general kernel, 8 blocks of it).
int nxh_gemm_strip_blocks(const nxh_context *ctx, int64_t M, int64_t N, int64_t K, int64_t nbatch) {
  const int64_t cus = ctx->compute_units > 0 ? ctx->compute_units : 256;
  const int64_t tiles = ((M + 15) / 16) * ((N + gemm_strip::BN - 1) / gemm_strip::BN) * nbatch;
  // (two steps a wave at least)
  const int64_t blocks = std::min<int64_t>(cus / std::max<int64_t>(tiles, 1), K / (2 * gemm_strip::MAXW * gemm_strip::KS));
  if (blocks < 2) return 1;
  const double saved = (double)K * 2.9e-3 * (1.0 - 1.0 / (double)blocks);
  const double cost = 3.5 + (double)blocks * (double)tiles * 16.0 * 64.0 * 8.0 / 4e6;
  return saved > 1.2 * cost ? (int)blocks : 1;
}

int nxh_gemm_strip(nxh_context *ctx, int dtype, gemm_strip::Args &g) {
  using namespace gemm_strip;
  // what a lane's 32-bit offsets hold: 24 rows of B and a row's columns, 64 rows of A
  if (g.N < 4 || g.ldb < 0 || g.lda < 0 || g.K > 0x7fffffff || g.nbd > 4) return -1;
  if ((double)g.ldb * 48.0 + (double)g.N * 2.0 >= 4294967296.0 || (double)g.lda * 130.0 + 64.0 >= 4294967296.0) return -1;
  const bool epi = g.bias || g.R || g.gelu;
  if (dtype == NXH_BF16) return epi ? run<ElBF16, true>(ctx, g) : run<ElBF16, false>(ctx, g);
  return epi ? run<ElF16, true>(ctx, g) : run<ElF16, false>(ctx, g);
}
