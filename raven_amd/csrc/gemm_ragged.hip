// gemm_ragged.hip — the LDS-tiled products (gemm_tile.hpp) of operands as they come: any K, rows
// that start at any element, a result of any strides.
//
// What bounds it: the matrix pipe, as for the aligned form; the loads are 16 bytes at the element's
// alignment and only the last slab of K looks at what exists. Before, such products were run over
// zero-padded copies of both operands: two more launches, two allocations and a pass over memory
// ([32,64,784] x [32,784,288] float32: 18 of 38 us; [2047,2047]^2 bfloat16: 41 us against 25 for
// 2048).
#include <algorithm>
#include <cmath>

#include "gemm_args.hpp"
#include "gemm_tile.hpp"
#include "nxh_common.hpp"

namespace {
using namespace gemm_tile;

template <class EL, bool A_KC, bool B_KC, class SH>
int launch(nxh_context *ctx, Args &g) {
  auto kern = kernel<EL, A_KC, B_KC, SH, true, false, false, true>;
  constexpr size_t LDS = SH::template lds_bytes<EL>();
  static std::once_flag once;  // allow > 64 KiB of dynamic LDS
  static hipError_t attr_status = hipSuccess;
  std::call_once(once, [&] {
    attr_status = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)LDS);
  });
  NXH_HIP("matmul", attr_status);
  g.tiles_m = (uint32_t)((g.M + SH::BM - 1) / SH::BM);
  g.tiles_n = (uint32_t)((g.N + SH::BN - 1) / SH::BN);
  nxh_set_path("gemm_tile_padded");  // (K is padded in LDS)
  hipLaunchKernelGGL(kern, dim3(g.tiles_m * g.tiles_n * g.nbatch), dim3(SH::THREADS), LDS, ctx->stream, g);
  NXH_HIP("matmul", hipGetLastError());
  return NXH_OK;
}
template <class EL, class SH>
int launch_oriented(nxh_context *ctx, Args &g, bool a_kc, bool b_kc) {
  if (a_kc) return b_kc ? launch<EL, true, true, SH>(ctx, g) : launch<EL, true, false, SH>(ctx, g);
  return b_kc ? launch<EL, false, true, SH>(ctx, g) : launch<EL, false, false, SH>(ctx, g);
}

template <class EL>
int run(nxh_context *ctx, const GemmArgs &a, uint32_t nbatch, int kruns) {
  const bool a_kc = a.acs == 1, b_kc = a.brs == 1;
  if (a.batch.n > 4 || a.M < 32 || a.N < 32 || a.K < 32 || a.K > 0x7fffffff) return -1;
  Args g{};
  g.A = a.A;
  g.B = a.B;
  g.C = a.C;
  g.lda = a_kc ? a.ars : a.acs;
  g.ldb = b_kc ? a.bcs : a.brs;
  g.ldc = a.crs;
  g.ccs = a.ccs;
  // an operand contiguous along M / N is read past its rows' ends: into a neighbouring row
  if ((!a_kc && (a.ars != 1 || std::abs(g.lda) < a.M)) || (!b_kc && (a.bcs != 1 || std::abs(g.ldb) < a.N))) return -1;
  g.M = a.M;
  g.N = a.N;
  g.K = a.K;
  g.nbatch = nbatch;
  g.nbd = a.batch.n;
  for (int i = 0; i < a.batch.n; i++) {
    g.bshape[i] = a.batch.shape[i];
    g.ba[i] = a.batch.a[i];
    g.bb[i] = a.batch.b[i];
    g.bc[i] = a.batch.c[i];
  }
  if (kruns > 1) {  // (the caller has checked that there is no batch)
    g.kruns = kruns;
    g.nbatch = nbatch = (uint32_t)kruns;
    g.nbd = 1;
    g.bshape[0] = (uint32_t)kruns;
    g.bc[0] = a.M * a.N;
  }
  auto tiles = [&](int bm, int bn) { return ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn) * (int64_t)nbatch; };
  if (tiles(64, 64) > 0x7fffffffLL) return -1;
  const int64_t cus = ctx->compute_units > 0 ? ctx->compute_units : 256;
  // Rounds of blocks x area x cost per flop against the largest block, as for the aligned form.
  struct Cand {
    int bm, bn;
    double per, pen;
  };
  const Cand f32[] = {{256, 256, 1, 1.0}, {128, 128, 1, 1.12}, {64, 64, 1, 1.3}};
  const Cand f16[] = {{256, 256, 1, 1.0}, {128, 128, 2, 1.25}, {128, 64, 2, 1.5}};
  int pick = 0;
  double best = 0.0;
  for (int i = 0; i < 3; i++) {
    const Cand &c = EL::F32 ? f32[i] : f16[i];
    const double cost = std::ceil((double)tiles(c.bm, c.bn) / ((double)cus * c.per)) * c.per * c.bm * c.bn * c.pen;
    if (i == 0 || cost < best) best = cost, pick = i;
  }
  if (pick == 0) return launch_oriented<EL, Shape256x256>(ctx, g, a_kc, b_kc);
  if (pick == 1) return launch_oriented<EL, Shape128x128>(ctx, g, a_kc, b_kc);
  if constexpr (!EL::F32) {  // two groups of waves a block (gemm_tile.hpp), from eight slabs on
    if (kruns == 1 && a.K > 7 * Geo<EL>::BK && tiles(128, 64) <= cus) return launch_oriented<EL, Shape128x64Halves>(ctx, g, a_kc, b_kc);
  }
  return launch_oriented<EL, std::conditional_t<EL::F32, Shape64x64, Shape128x64>>(ctx, g, a_kc, b_kc);
}
}  // namespace

int nxh_gemm_ragged(nxh_context *ctx, int dtype, const GemmArgs &a, uint32_t nbatch, int kruns) {
  if (dtype == NXH_F32) return run<ElF32>(ctx, a, nbatch, kruns);
  if (dtype == NXH_BF16) return run<ElBF16>(ctx, a, nbatch, 1);
  return run<ElF16>(ctx, a, nbatch, 1);
}
