// The products of gemm_strip.hip: few rows times a 16-bit matrix in memory order.
#pragma once
#include <cstdint>

struct nxh_context;

namespace gemm_strip {
struct Args {
  const void *A, *B;
  void *C;
  int64_t lda, ldb, ldc;  // A is contiguous along K, B and C along N
  int64_t M, N, K;
  const void *bias, *R;  // null: left out
  int64_t ldr;
  int gelu;  // no R: then the tanh GELU on the biased product (gemm_tile.hpp)
  float gc[4];
  uint32_t tiles_m, tiles_n, nbatch;
  int nbd;
  uint32_t bshape[4];
  int64_t ba[4], bb[4], bc[4], br[4];
  uint32_t ngroup, gtn;  // members of a group of linears (gemm_tile.hpp)
  int64_t goff_b[2], goff_c[2], goff_bias[2];
};
}  // namespace gemm_strip

// Blocks that share the K of a tile (a rule on the sizes: the same for a plain product and a linear).
int nxh_gemm_strip_blocks(const nxh_context *ctx, int64_t M, int64_t N, int64_t K, int64_t nbatch);
// bfloat16 / float16; any M, N >= 4, K and alignment. -1: left to the other kernels.
int nxh_gemm_strip(nxh_context *ctx, int dtype, gemm_strip::Args &g);
