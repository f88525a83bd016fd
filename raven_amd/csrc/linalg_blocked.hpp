// linalg_blocked.hpp — cholesky and triangular_solve by blocks (included by linalg.hip,
// inside its namespace).
//
// Both are chains: column j of a factor, row i of a solution, waits for the one before
// it. A launch per column pays a launch (2 - 4 us) per link of the chain; here a link is
// some 200 cycles inside a workgroup, and everything that is no link (the updates of what
// comes later) is a product of 16 x 16 tiles on the f64 matrix instruction.
#pragma once

typedef __attribute__((ext_vector_type(4))) double la_f64x4;

// A batch of matrices in the storage type TS: element (r, c) of matrix b is p[b bs + r rs + c cs].
struct LaMat {
  void *p;
  int64_t rs, cs, bs;
};

// A numeric failure of a call (every one of a call has the same meaning): a kernel stores the call's number to `found`,
// in device memory, and kernels after it that see that number there write nothing. Nothing is cleared between calls.
// The call reads it from a report (nxh_report_word), which a kernel stores to `report` as soon as it is known.
struct LaFailure {
  int *found;
  uint64_t *report;  // null: this kernel does not report
  uint32_t seq;
  __device__ __forceinline__ void raise() const { __hip_atomic_store(found, (int)seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
  __device__ __forceinline__ bool raised() const { return *found == (int)seq; }
};

__device__ __forceinline__ double lane_value(double v, int lane) {  // `lane` uniform
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane), hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ c64 lane_value(c64 v, int lane) { return {lane_value(v.re, lane), lane_value(v.im, lane)}; }

__device__ __forceinline__ void to_storage(double v, float *p) { *p = (float)v; }
__device__ __forceinline__ void to_storage(double v, double *p) { *p = v; }
__device__ __forceinline__ void to_storage(c64 v, c64 *p) { *p = v; }

// What the lanes of a wave wrote to LDS before it is there for all of them after it.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A value that is there before what follows is chosen: keeps the compiler from turning a choice between two short
// computations, or the loading of one operand, into a branch of the wave and a wait behind it.
__device__ __forceinline__ double at_hand(double v) {
  asm("" : "+v"(v));
  return v;
}
__device__ __forceinline__ c64 at_hand(c64 v) { return v; }

// sqrt(d) and 1 / sqrt(d) of a positive d far from the ends of the exponents, each to the last bit or next to it: one
// hardware estimate and Newton steps. The chain of the factorisation runs through this once per column; the library's
// square root and division are four times as long, and scaling d first a good tenth of the chain (sixteen columns of
// [512,512] f32: 6 350 clocks scaled, 5 690 so; 28.3 us a launch -> 27.5).
__device__ __forceinline__ void plain_root_and_inverse(double d, double *root, double *inv) {
  double r = __builtin_amdgcn_rsq(d);
  const double err = fma(-(d * r), r, 1.0);
  r = fma(r * err, fma(0.375, err, 0.5), r);
  double l = d * r;
  l = fma(fma(-l, l, d), 0.5 * r, l);
  r = fma(fma(-l, r, 1.0), r, r);
  *root = l;
  *inv = r;
}
// The same of any positive d, scaled into [1/4, 1) by a power of four, which changes no digit.
__device__ __forceinline__ void root_and_inverse(double d, double *root, double *inv) {
  const int e = (__builtin_amdgcn_frexp_exp(d) + 1) >> 1;
  double l, r;
  plain_root_and_inverse(ldexp(d, -2 * e), &l, &r);
  *root = d < __builtin_inf() ? ldexp(l, e) : d;
  *inv = d < __builtin_inf() ? ldexp(r, -e) : 0.0;
}

// One 16 x 16 tile of accumulators: register v of lane l is row 4 v + l / 16, column l % 16
// (what v_mfma_f64_16x16x4 produces; the complex form uses the same places).
template <class T>
struct LaTile {
  T v[4];
};

// A B^H over K terms: A[row * lda + k], B[col * ldb + k] with the tile's first row and column in the
// pointers, as sums of four terms that meet pairwise; tile_sub takes it from acc. So there is one
// rounding at the size of acc per call and not one per term (one chain of fused steps from acc left a
// Gram matrix of 256 columns with four times the backward error, 0.30 against 0.07 eps).
// Up to eight products are under way before the first is added: left to itself, the compiler waits for each of them,
// some 140 clocks, and for its operands ([512,512] f32: the sums of a block column's last rows 470 clocks -> 260, those ahead
// of its diagonal tile, which the matrix units bound, 7 700 -> 7 350).
template <int K>
__device__ __forceinline__ la_f64x4 tile_sum(const double *A, int64_t lda, const double *B, int64_t ldb) {
  if constexpr (K > 32) {
    const la_f64x4 low = tile_sum<K / 2>(A, lda, B, ldb);
    return low + tile_sum<K / 2>(A + K / 2, lda, B + K / 2, ldb);
  } else {
    constexpr int N = K / 4;
    const int lane = threadIdx.x & 63, at = lane >> 4;
    double x[N], y[N];
    la_f64x4 p[N];
#pragma unroll
    for (int i = 0; i < N; i++) x[i] = A[(lane & 15) * lda + 4 * i + at], y[i] = B[(lane & 15) * ldb + 4 * i + at];
    if constexpr (N > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < N; i++) p[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[i], la_f64x4{0.0, 0.0, 0.0, 0.0}, 0, 0, 0);
    if constexpr (N > 4) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int d = 1; d < N; d *= 2)
#pragma unroll
      for (int i = 0; i + d < N; i += 2 * d) p[i] = p[i] + p[i + d];
    return p[0];
  }
}
template <int K>
__device__ __forceinline__ void tile_sub(LaTile<double> &acc, const double *A, int64_t lda, const double *B, int64_t ldb) {
  const la_f64x4 sum = tile_sum<K>(A, lda, B, ldb);
#pragma unroll
  for (int i = 0; i < 4; i++) acc.v[i] -= sum[i];
}
template <int K>
__device__ __forceinline__ LaTile<c64> tile_sum(const c64 *A, int64_t lda, const c64 *B, int64_t ldb) {  // (with its sign)
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  LaTile<c64> s;
  if constexpr (K > 4) {
    s = tile_sum<K / 2>(A, lda, B, ldb);
    const LaTile<c64> high = tile_sum<K / 2>(A + K / 2, lda, B + K / 2, ldb);
#pragma unroll
    for (int v = 0; v < 4; v++) s.v[v] = s.v[v] + high.v[v];
  } else {
#pragma unroll
    for (int v = 0; v < 4; v++) s.v[v] = Sc<c64>::make(0.0, 0.0);
#pragma unroll
    for (int k = 0; k < K; k++) {
      const c64 b = Sc<c64>::conj(B[r * ldb + k]);
#pragma unroll
      for (int v = 0; v < 4; v++) s.v[v] = Sc<c64>::sub_mul(s.v[v], A[(4 * v + q) * lda + k], b);
    }
  }
  return s;
}
template <int K>
__device__ __forceinline__ void tile_sub(LaTile<c64> &acc, const c64 *A, int64_t lda, const c64 *B, int64_t ldb) {
  LaTile<c64> sum;
#pragma unroll 1
  for (int k = 0; k < K; k += 16) {  // (sixteen terms of code)
    const LaTile<c64> s = tile_sum<16>(A + k, lda, B + k, ldb);
#pragma unroll
    for (int v = 0; v < 4; v++) sum.v[v] = k ? sum.v[v] + s.v[v] : s.v[v];
  }
#pragma unroll
  for (int v = 0; v < 4; v++) acc.v[v] = acc.v[v] + sum.v[v];
}

// Neither holds where x or dx is not finite.
__device__ __forceinline__ bool small_step(double x, double dx) { return dx == 0.0 || fabs(dx) < 0x1p-28 * fabs(x); }

// Substitution through a 16 x 16 triangle, four rows at a time on the matrix instruction, for
// sixteen right-hand sides: register v of lane (q, c) = 16 q + c holds row 4 v + q of side c, which is
// both where the instruction leaves a result and, for four rows, where it takes its second operand
// from: nothing moves between lanes. diag_inv[b] is the inverse of the b-th 4 x 4 triangle on
// the diagonal as a first operand (lane (q, r): element (r - 4 b, q), 0 in other rows), tri[b] columns
// 4 b .. 4 b + 3 (lane (q, r): element (r, 4 b + q), 0 above the diagonal). The product with the
// inverse is followed by one step on its remainder, which the instruction leaves in the same register.
// That stands for a substitution where the step is small: it divides the error of the product by as
// much as it is smaller than it, so below 2^-28 of every value what is left is less than a rounding.
// Where it is larger (a diagonal small against what is below it: the inverse grows, and the error of
// the product with it), or no number (the zeros of the operands meet every row of a group of four: a
// row that is not finite would make the rows before it NaN), nothing is changed and the answer is
// false: the caller substitutes row by row. 15 instructions of 64 cycles; row by row, with
// a right-hand side a lane, the chain through LDS took 4700 cycles.
__device__ __forceinline__ bool solve16(LaTile<double> &acc, const double (&diag_inv)[4], const double (&tri)[4]) {
  const la_f64x4 zero = {0.0, 0.0, 0.0, 0.0};
  la_f64x4 taken = zero;  // by the rows before, summed apart from acc: one rounding at its size
  LaTile<double> sol;
  bool small = true;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const double c = b > 0 ? acc.v[b] - taken[b] : acc.v[b];
    const double x = __builtin_amdgcn_mfma_f64_16x16x4f64(diag_inv[b], c, zero, 0, 0, 0)[b];
    const double rest = c - __builtin_amdgcn_mfma_f64_16x16x4f64(tri[b], x, zero, 0, 0, 0)[b];
    const double dx = __builtin_amdgcn_mfma_f64_16x16x4f64(diag_inv[b], rest, zero, 0, 0, 0)[b];
    sol.v[b] = x + dx;
    small = small && small_step(x, dx);
    if (b < 3) taken = __builtin_amdgcn_mfma_f64_16x16x4f64(tri[b], sol.v[b], taken, 0, 0, 0);
  }
  if (!__all(small)) return false;
  acc = sol;
  return true;
}

// Cholesky of a 16 x 16 tile in that layout (the tile is Hermitian: rows and columns may change
// places), four columns at a time: every lane factors the 4 x 4 block on the diagonal, element by
// element, the matrix instruction does the rest. The tile is acc - before; what its own columns take is
// summed beside `before`, so that an element of a diagonal block rounds once at its own size.
// Leaves the operands of solve16 in diag_inv and tri; tri is the factor itself. `blk`: 64 places of LDS.
// False where that is not the factor: a pivot that is not positive or near the ends of the exponents, or a step as in solve16.
__device__ __forceinline__ bool factor16(const LaTile<double> &acc, la_f64x4 before, double2 *blk, double (&diag_inv)[4], double (&tri)[4]) {
  const int lane = threadIdx.x & 63, c = lane & 15, q = lane >> 4;
  const la_f64x4 zero = {0.0, 0.0, 0.0, 0.0};
  la_f64x4 taken = zero;
  bool good = true;
#pragma unroll
  for (int b = 0; b < 4; b++) {
    const double off = b > 0 ? before[b] + taken[b] : before[b], t = acc.v[b] - off;
    blk[lane] = make_double2(acc.v[b], off);
    __builtin_amdgcn_wave_barrier();
    double a[4][4], sum[4][4];  // a[j][i]: element (4 b + i, 4 b + j); sum: what the columns before take from it
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = j; i < 4; i++) {
        const double2 v = blk[16 * j + 4 * b + i];
        a[j][i] = v.x, sum[j][i] = v.y;
      }
    __builtin_amdgcn_wave_barrier();
    double low[4][4], root[4];  // low[j][i]: the factor; root[j]: the inverse of its diagonal
    double own[4][4];           // what this block's columns take
#pragma unroll
    for (int j = 0; j < 4; j++) {
#pragma unroll
      for (int i = j; i < 4; i++) low[j][i] = a[j][i] - (j > 0 ? sum[j][i] + own[j][i] : sum[j][i]);
      good = good && low[j][j] > 0x1p-900 && low[j][j] < 0x1p900;
      plain_root_and_inverse(low[j][j], &low[j][j], &root[j]);
#pragma unroll
      for (int i = j + 1; i < 4; i++) low[j][i] *= root[j];
#pragma unroll
      for (int k = j + 1; k < 4; k++)
#pragma unroll
        for (int i = k; i < 4; i++) own[k][i] = j > 0 ? fma(low[j][i], low[j][k], own[k][i]) : low[j][i] * low[j][k];
    }
    double u[4][4];  // the unit triangle
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
      for (int i = j + 1; i < 4; i++) u[j][i] = low[j][i] * root[j];
    // rows of the inverse of the unit triangle, each times its root
    const double m10 = -u[0][1], m21 = -u[1][2], m32 = -u[2][3];
    const double m20 = fma(-m10, u[1][2], -u[0][2]), m31 = fma(-m21, u[2][3], -u[1][3]);
    const double m30 = fma(-m20, u[2][3], fma(-m10, u[1][3], -u[0][3]));
    const int i = c - 4 * b;
    double m = q == 0 ? m30 : q == 1 ? m31 : q == 2 ? m32 : 1.0;
    m = i == 2 ? (q == 0 ? m20 : q == 1 ? m21 : 1.0) : m;
    m = i == 1 ? (q == 0 ? m10 : 1.0) : m;
    m = i == 0 ? 1.0 : m;
    m *= i == 0 ? root[0] : i == 1 ? root[1] : i == 2 ? root[2] : root[3];
    diag_inv[b] = i >= q && i < 4 ? m : 0.0;
    // inside the block the factor itself, elsewhere (rows of the factor below it) the product
    double in = q == 0 ? low[0][3] : q == 1 ? low[1][3] : q == 2 ? low[2][3] : low[3][3];
    in = i == 2 ? (q == 0 ? low[0][2] : q == 1 ? low[1][2] : low[2][2]) : in;
    in = i == 1 ? (q == 0 ? low[0][1] : low[1][1]) : in;
    in = i == 0 ? low[0][0] : in;
    const double product = __builtin_amdgcn_mfma_f64_16x16x4f64(diag_inv[b], t, zero, 0, 0, 0)[b];
    const bool below = i >= 4;
    const double x = below ? product : i >= q ? in : 0.0;
    const double rest = t - __builtin_amdgcn_mfma_f64_16x16x4f64(x, x, zero, 0, 0, 0)[b];
    const double dx = __builtin_amdgcn_mfma_f64_16x16x4f64(diag_inv[b], rest, zero, 0, 0, 0)[b];
    tri[b] = below ? x + dx : x;
    good = good && (!below || small_step(x, dx));
    if (b < 3) taken = __builtin_amdgcn_mfma_f64_16x16x4f64(tri[b], tri[b], taken, 0, 0, 0);
  }
  return __all(good);
}

// The same column by column, in place on the lower triangle (the rest becomes 0), for what factor16
// refuses: pivots that are infinite or near it, or next to zero, tiles close to singular; a failure shows here. 1 / L_cc goes to
// the place that lane (q, c) of diag_inv[c / 4], q = c % 4, has in `inv`.
__device__ __forceinline__ bool factor16_columns(double *tile, int ld, double *inv) {
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  bool positive = true;
#pragma unroll 1
  for (int c = 0; c < 16; c++) {
    wave_sync();
    const double d = tile[c * ld + c], own = tile[r * ld + c];
    positive = positive && d > 0.0;
    double root, root_inv;
    root_and_inverse(d, &root, &root_inv);
    wave_sync();
    if (q == 0) tile[r * ld + c] = r == c ? root : r > c ? own * root_inv : 0.0;
    if (lane == 0) inv[(c >> 2) * 64 + (c & 3) * 16 + c] = root_inv;
    wave_sync();
    for (int k = c + 1 + q; k <= r; k += 4) tile[r * ld + k] = fma(-tile[r * ld + c], tile[k * ld + c], tile[r * ld + k]);
  }
  return positive;
}

// ── cholesky ────────────────────────────────────────────────────────────────
// NB x NB tiles, one launch per block column s, a workgroup per tile (i, j) with i >= j >= s.
// What block column s - 1 takes from tile (i, j) is first added to what the columns before it took.
// Column s then is finished: every workgroup of that column keeps the diagonal tile too, factors it (the same
// instructions on the same values everywhere), and solves its own tile against it, sixteen
// columns behind. Factoring the diagonal again in each workgroup costs nothing (it would
// be waited for) and saves a launch per block column. Sums and factor share one workspace: a tile of
// the factor goes where this workgroup's own sums were, those on the diagonal, whose sums the other
// workgroups of the column read too, to a place of their own. The matrix itself is only read; the result is
// written by cholesky_result_kernel, where there is one. The sums stay apart from
// the matrix until its column comes up, so that an element rounds a few times at its own size and not
// once a column: float64, g g^T + n I, relative error of the factor in eps (2-norm, against long double) for
// n = 64, 130, 400: 1.52, 2.03, 3.41 with the updates taken from the matrix one by one, 0.55, 0.50, 0.51 so
// (a column at a time with a wave per element: 1.44, 0.52, 0.52). float64 [512, 512] takes 226 us so, its
// result written by a launch of its own, against 213.
//
// The chain of a launch is the diagonal tile, sixteen columns at a time: factored by wave 0
// (factor16), then a wave per sixteen rows below solves against them (solve16), then wave 0
// updates and factors the next sixteen while the others update the rest and this workgroup's own
// tile follows, a wave per sixteen rows, one block of columns behind. Complex matrices, with no matrix
// instruction for them, are factored column by column, a row a lane.
// Matrices of ONE blocks of sixteen columns, 1 or 2, are a single tile: a wave per block, and the LDS of
// one tile, so that a compute unit holds several. (0: any size, eight waves and four tiles, one
// workgroup a unit: float64 factors of [16384,16,16] in 361 us against 68, of [1024,17,17] in 51 against 29; the
// form for one workgroup per matrix in a workspace took 281 and 52.)
template <class T, int ONE>
struct Chol {
  static constexpr int NB = ONE ? 16 * ONE : sizeof(T) == 8 ? 64 : 32, BLOCKS = NB / 16;
  static constexpr int THREADS = ONE ? 64 * ONE : 512, WAVES = THREADS / 64;
  static constexpr int LD = NB + 2;                        // 66 doubles: sixteen rows on different banks
  static constexpr int COLUMN = 80;                        // complex: 64 values of one column, and room for reads past them
  static constexpr int OPERANDS = 128 + 3 * BLOCKS * 256;  // double: factor16's scratch, the operands of solve16, diag_sum
  static constexpr size_t LDS = (ONE ? 1 : 4) * NB * LD * sizeof(T) + (sizeof(T) == 8 ? OPERANDS * sizeof(double) : COLUMN * sizeof(T) + NB * sizeof(double));
};

template <class T>
struct CholArgs {
  LaMat x, out;   // storage types
  T *A, *diag;    // n x n per matrix, row-major: what is taken from x, with its sign, then the factor below the
                  // diagonal tiles; those tiles, NB x NB each
  int n, s, upper;
  LaFailure failure;
};

template <class T, class TS, int ONE>
__global__ __launch_bounds__((Chol<T, ONE>::THREADS)) void cholesky_block_kernel(CholArgs<T> a) {
  using S = Sc<T>;
  using C = Chol<T, ONE>;
  constexpr int NB = C::NB, LD = C::LD, TILES = C::BLOCKS;
  extern __shared__ double lds_raw[];
  T *D = (T *)lds_raw;  // the diagonal tile
  T *column = D + NB * LD;
  double *inv = (double *)(column + C::COLUMN);
  double *blk = (double *)(D + NB * LD), *op_inv = blk + 128, *op_tri = op_inv + TILES * 256, *diag_sum = op_tri + TILES * 256;
  // ONE has neither of these: this workgroup's tile, block column s - 1 in the rows of tile (s, .) and of tile (i, .)
  T *own = (T *)((char *)lds_raw + C::LDS) - 3 * NB * LD, *ls = own + NB * LD, *li = ls + NB * LD;
  const int n = a.n, s = a.s, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int panels = (n + NB - 1) / NB - s;  // block rows from s down
  int i, j;
  if ((int)blockIdx.x < panels) {
    i = s + blockIdx.x, j = s;
  } else {  // the others, row by row of the triangle below
    int t = blockIdx.x - panels, row = 1;
    while (t >= row) t -= row, row++;
    i = s + row, j = s + 1 + t;
  }
  const TS *x = (const TS *)a.x.p + blockIdx.y * a.x.bs;
  T *A = a.A + (size_t)blockIdx.y * n * n;
  // Element (r, c) of the matrix (lower triangle), and what the launches before the last took from
  // it, with its sign. Rows and columns past n read the last one: what comes of them is not kept.
  auto element = [&](int r, int c) { return x[min(r, n - 1) * a.x.rs + min(c, n - 1) * a.x.cs]; };
  auto taken_before = [&](int r, int c) { return s > 1 ? A[(size_t)min(r, n - 1) * n + min(c, n - 1)] : S::make(0.0, 0.0); };
  // What a wave does in 16 x 16 sub-tiles before anything waits: a tile that is not finished in this launch,
  // or the lower half of the diagonal tile (the own tile of such a workgroup follows in the shadow of the
  // factorisation; complex: here).
  const bool panel = j == s, has_own = i > s;
  const int left = min(n - s * NB, NB), blocks = (left + 15) / 16;
  constexpr bool OWN_LATER = sizeof(T) == 8;
  constexpr int LOWER = TILES * (TILES + 1) / 2, ALL = TILES * TILES;
  auto job = [&](int t, int *diag, int *tr, int *tc) {  // job `t`, and whether there is anything to do
    *diag = panel && t < LOWER;
    if (*diag) {
      *tr = 0;
      for (int first = 0; first + *tr + 1 <= t; first += ++*tr) *tc = 0;
      *tc = t - *tr * (*tr + 1) / 2;
      return *tr < blocks;
    }
    t -= panel ? LOWER : 0;
    *tr = t / TILES, *tc = t % TILES;
    return t < ALL && (!panel || (has_own && !OWN_LATER)) && i * NB + *tr * 16 < n && j * NB + *tc * 16 < n && (i != j || *tc <= *tr);
  };
  constexpr int MOST = OWN_LATER ? ALL : ALL + LOWER, JOBS = (MOST + C::WAVES - 1) / C::WAVES;
  LaTile<T> acc[JOBS];
  LaTile<TS> raw[JOBS];  // (converted only once it is used: a conversion would wait for its load)
#pragma unroll
  for (int e = 0; e < JOBS; e++) {  // every load is on its way before the first is waited for
    int diag, tr, tc;
    if (!job(e * C::WAVES + wave, &diag, &tr, &tc)) continue;
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = (diag ? s : i) * NB + tr * 16 + 4 * v + q, c = j * NB + tc * 16 + r16;
      acc[e].v[v] = taken_before(r, c);
      if (panel) raw[e].v[v] = element(r, c);
    }
  }
  // Double: what is taken from the diagonal tile is summed apart from it, for a 16 x 16 tile below the
  // diagonal in the place of its mirror image, transposed; for one on the diagonal in diag_sum.
  auto taken_at = [&](int tr, int tc) { return (double *)(tr == tc ? diag_sum + tr * 256 + q * 16 + r16 : (double *)D + (tc * 16 + r16) * LD + tr * 16 + q); };
  auto taken_step = [](int tr, int tc) { return tr == tc ? 64 : 4; };
  constexpr int PER = NB * NB / C::THREADS;
  const int col_of = threadIdx.x % NB, row_of = threadIdx.x / NB;
  TS mine[PER];
  T mine_taken[PER];
  if (OWN_LATER && panel && has_own) {
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int r = i * NB + row_of + e * (C::THREADS / NB), c = s * NB + col_of;
      mine[e] = element(r, c);
      mine_taken[e] = taken_before(r, c);
    }
  }
  if (s > 0) {
    T vj[PER], vi[PER];
    const int c = col_of, r0 = row_of;
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int r = r0 + e * (C::THREADS / NB);
      vj[e] = A[(size_t)min(j * NB + r, n - 1) * n + (s - 1) * NB + c];
      vi[e] = A[(size_t)min(i * NB + r, n - 1) * n + (s - 1) * NB + c];
    }
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int r = r0 + e * (C::THREADS / NB);
      ls[r * LD + c] = vj[e];
      li[r * LD + c] = vi[e];
    }
    __syncthreads();
  }
#pragma unroll
  for (int e = 0; e < JOBS; e++) {
    int diag, tr, tc;
    if (!job(e * C::WAVES + wave, &diag, &tr, &tc)) continue;
    if (s > 0) tile_sub<NB>(acc[e], (diag ? ls : li) + tr * 16 * LD, LD, ls + tc * 16 * LD, LD);
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int r = tr * 16 + 4 * v + q, cc = tc * 16 + r16;
      const bool inside = r < left && cc < left;
      if (!panel) {
        if (i * NB + r < n && j * NB + cc < n) A[(size_t)(i * NB + r) * n + j * NB + cc] = acc[e].v[v];
      } else if (!diag) {
        own[r * LD + cc] = T(raw[e].v[v]) + acc[e].v[v];
      } else {  // past n the diagonal tile is the identity
        const T val = OWN_LATER ? T(raw[e].v[v]) : T(raw[e].v[v]) + acc[e].v[v];
        D[r * LD + cc] = inside ? val : S::make(r == cc ? 1.0 : 0.0, 0.0);
        if constexpr (OWN_LATER) taken_at(tr, tc)[v * taken_step(tr, tc)] = inside ? -acc[e].v[v] : 0.0;
      }
    }
  }
  if (OWN_LATER && panel && has_own) {
#pragma unroll
    for (int e = 0; e < PER; e++) own[(row_of + e * (C::THREADS / NB)) * LD + col_of] = T(mine[e]) + mine_taken[e];
  }
  if (!panel) return;
  __syncthreads();
  bool bad = false;
  if constexpr (sizeof(T) == 8) {
    // rows (sixteen, in LDS) against columns 16 jb .. of the diagonal tile; `before`: nothing has summed yet
    // what the columns before those take, of block column s - 1 (rows of li at `before`) and of this one
    auto solve_rows = [&](double *rows, int jb, const double *before) {
      LaTile<double> t;
#pragma unroll
      for (int v = 0; v < 4; v++) t.v[v] = rows[r16 * LD + jb * 16 + 4 * v + q];
      la_f64x4 taken = {0.0, 0.0, 0.0, 0.0};
      if (before) {
        if (s > 0) taken = tile_sum<NB>(ls + jb * 16 * LD, LD, before, LD);
#pragma unroll 1
        for (int k = 0; k < jb * 16; k += 16) taken += tile_sum<16>(D + jb * 16 * LD + k, LD, rows + k, LD);
      } else {
#pragma unroll
        for (int v = 0; v < 4; v++) taken[v] = D[(jb * 16 + 4 * v + q) * LD + wave * 16 + r16];
      }
      double di[4], tr[4];
#pragma unroll
      for (int v = 0; v < 4; v++) di[v] = op_inv[(jb * 4 + v) * 64 + lane], tr[v] = op_tri[(jb * 4 + v) * 64 + lane];
#pragma unroll
      for (int v = 0; v < 4; v++) t.v[v] -= taken[v];
      const bool solved = solve16(t, di, tr);
#pragma unroll
      for (int v = 0; v < 4; v++) rows[r16 * LD + jb * 16 + 4 * v + q] = t.v[v];
      if (solved) return;
      // column by column, four lanes a row
      double *row = rows + r16 * LD + jb * 16;
      const double *tri = D + jb * 16 * (LD + 1);
#pragma unroll 1
      for (int c = 0; c < 16; c++) {
        wave_sync();
        const double x = row[c] * op_inv[(jb * 4 + (c >> 2)) * 64 + (c & 3) * 16 + c];
        if (q == 0) row[c] = x;
        for (int k = c + 1 + q; k < 16; k += 4) row[k] = fma(-x, tri[k * LD + c], row[k]);
      }
    };
    auto solve_own = [&](int jb) {
      const int tr = wave == 1 ? 3 : wave - 5;  // (not wave 4: it shares a SIMD, and its matrix unit, with wave 0)
      if (has_own && tr >= 0 && i * NB + tr * 16 < n) solve_rows(own + tr * 16 * LD, jb, li + tr * 16 * LD);
    };
#pragma unroll 1
    for (int jb = 0; jb < blocks; jb++) {
      if (wave == 0) {
        double *tile = D + jb * 16 * (LD + 1);
        LaTile<double> t;
        la_f64x4 taken = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int v = 0; v < 4; v++) t.v[v] = tile[max(r16, 4 * v + q) * LD + min(r16, 4 * v + q)];  // (the lower triangle is what there is)
        if (jb > 0) taken = tile_sum<16>(tile - 16, LD, tile - 16, LD);
#pragma unroll
        for (int v = 0; v < 4; v++) taken[v] += taken_at(jb, jb)[64 * v];
        double di[4], tr[4];
        const bool stands = factor16(t, taken, (double2 *)blk, di, tr);
#pragma unroll
        for (int v = 0; v < 4; v++) tile[r16 * LD + 4 * v + q] = stands ? tr[v] : t.v[v] - taken[v];
#pragma unroll
        for (int v = 0; v < 4; v++) {  // (solve16 refuses operands that are no numbers)
          op_inv[(jb * 4 + v) * 64 + lane] = di[v];
          op_tri[(jb * 4 + v) * 64 + lane] = stands ? tr[v] : __builtin_nan("");
        }
        if (!stands) bad = !factor16_columns(tile, LD, op_inv + jb * 256) || bad;
      } else if (jb > 0 && (wave == 2 || wave == 3)) {
        for (int t = wave - 2; t < TILES * TILES; t += 2) {  // what block jb - 1 takes from the rest of the tile
          const int tr = t / TILES, tc = t % TILES;
          if (tc < jb || tc > tr || tr >= blocks || (tc == jb && tr == jb)) continue;
          la_f64x4 d = tile_sum<16>(D + tr * 16 * LD + (jb - 1) * 16, LD, D + tc * 16 * LD + (jb - 1) * 16, LD);
          double *to = taken_at(tr, tc);
          const int step = taken_step(tr, tc);
#pragma unroll
          for (int v = 0; v < 4; v++) to[v * step] += d[v];
        }
      } else if (jb > 0) {
        solve_own(jb - 1);
      }
      __syncthreads();
      if (wave > jb && wave < blocks) solve_rows(D + wave * 16 * LD, jb, nullptr);
      __syncthreads();
    }
    solve_own(blocks - 1);
  } else {
    // this workgroup's tile against the finished columns 16 jb .. of the diagonal one: a wave per
    // sixteen rows (waves 4 and up, beside wave 0's next columns)
    auto solve_own = [&](int jb) {
      const int tr = wave - 4;
      if (!has_own || tr < 0 || tr >= TILES || i * NB + tr * 16 >= n) return;
      T *rows = own + tr * 16 * LD;
      if (jb > 0) {
        LaTile<T> t;
#pragma unroll
        for (int v = 0; v < 4; v++) t.v[v] = rows[(4 * v + q) * LD + jb * 16 + r16];
#pragma unroll 1
        for (int k = 0; k < jb * 16; k += 16) tile_sub<16>(t, rows + k, LD, D + jb * 16 * LD + k, LD);
#pragma unroll
        for (int v = 0; v < 4; v++) rows[(4 * v + q) * LD + jb * 16 + r16] = t.v[v];
        __builtin_amdgcn_wave_barrier();
      }
      T xr[16];  // what the columns so far take from those after them
#pragma unroll
      for (int c = 0; c < 16; c++) xr[c] = S::make(0.0, 0.0);
      T *at = rows + r16 * LD + jb * 16;
      const T *col = D + jb * 16 * (LD + 1);  // (c, c) of the diagonal block; rows past it are read, their results dropped
#pragma unroll 1
      for (int c = 0; c < 16; c++, col += LD + 1) {
        const T v = S::scale(at[c] + xr[0], inv[jb * 16 + c]);
        if (q == 0) at[c] = v;
#pragma unroll
        for (int k = 1; k < 16; k++) xr[k - 1] = S::sub_mul(xr[k], v, S::conj(col[k * LD]));
      }
    };
#pragma unroll 1
    for (int jb = 0; jb < blocks; jb++) {
      if (wave == 0) {
        const int c0 = jb * 16, row = min(lane, NB - 1);
        // `head`: this lane's element of the column at hand, up to date; p: what the columns so far take
        // from those after it, still without `prev`, the column before it. That column's values come
        // back from LDS while the square root is under way; only the next column's head waits for a
        // value of this one, and takes it from its lane (a lane's value costs some 20 cycles a register)
        T p[16], prev = S::make(0.0, 0.0);
#pragma unroll
        for (int c = 0; c < 16; c++) p[c] = S::make(0.0, 0.0);
        T head = D[row * LD + c0];
        column[lane] = prev;
#pragma unroll 1
        for (int c = c0; c < c0 + 16; c++) {
          T before[16];
#pragma unroll
          for (int k = 1; k < 16; k++) before[k] = column[c + k];
          const T next = D[row * LD + min(c + 1, NB - 1)];
          const double d = S::re(lane_value(head, c));
          bad = bad || !(d > 0.0);
          double l, li1;
          root_and_inverse(d, &l, &li1);
#pragma unroll
          for (int k = 1; k < 16; k++) p[k - 1] = S::sub_mul(p[k], prev, S::conj(before[k]));
          const T col = lane == c ? S::make(l, 0.0) : S::scale(head, li1);
          column[lane] = col;
          if (lane == 0) inv[c] = li1;
          if (lane < NB && lane >= c0) D[lane * LD + c] = lane < c ? S::make(0.0, 0.0) : col;
          head = next + S::sub_mul(p[0], col, S::conj(lane_value(col, (c + 1) & 63)));
          prev = col;
        }
      } else if (jb > 0) {
        solve_own(jb - 1);
      }
      __syncthreads();
      // what the new columns take from the rest of the diagonal tile
      for (int t = wave; t < TILES * TILES; t += C::WAVES) {
        const int tr = t / TILES, tc = t % TILES;
        if (tc <= jb || tc > tr || tr >= blocks) continue;
        LaTile<T> d;
#pragma unroll
        for (int v = 0; v < 4; v++) d.v[v] = D[(tr * 16 + 4 * v + q) * LD + tc * 16 + r16];
        tile_sub<16>(d, D + tr * 16 * LD + jb * 16, LD, D + tc * 16 * LD + jb * 16, LD);
#pragma unroll
        for (int v = 0; v < 4; v++) D[(tr * 16 + 4 * v + q) * LD + tc * 16 + r16] = d.v[v];
      }
      __syncthreads();
    }
    solve_own(blocks - 1);
  }
  if (bad && wave == 0 && lane == 0) a.failure.raise();
  __syncthreads();
  const int rows = min(n - i * NB, NB);
  if (has_own) {
    for (int e = threadIdx.x; e < NB * NB; e += C::THREADS) {
      const int r = e / NB, c = e % NB;
      if (r < rows) A[(size_t)(i * NB + r) * n + s * NB + c] = own[r * LD + c];  // (a tile below the diagonal has all its columns)
    }
  } else {
    T *to = a.diag + ((size_t)blockIdx.y * (s + panels) + s) * NB * NB;
    for (int e = threadIdx.x; e < NB * NB; e += C::THREADS) {
      const int r = e / NB, c = e % NB;
      if (r < left && c <= r) to[e] = D[r * LD + c];
    }
  }
}

// The result with its zeros, a workgroup per tile (i, j), i >= j, and its mirror image. U = L^H. It is queued behind the
// factorisation and writes nothing where that failed; its first workgroup tells the host, which goes on meanwhile ([512,512]
// f32 and two solves: 413 us where each call waited for the stream and the result's launch for the host, 373 so; 300 of
// [40,40] f64 100 -> 66).
template <class T, class TS, int ONE>
__global__ __launch_bounds__(256) void cholesky_result_kernel(CholArgs<T> a) {
  using S = Sc<T>;
  constexpr int NB = Chol<T, ONE>::NB;
  __shared__ T tile[NB][NB + 1];
  const int n = a.n, cols = (n + NB - 1) / NB;
  int i = 0, j = blockIdx.x;
  while (j > i) j -= ++i;
  const T *A = a.A + (size_t)blockIdx.y * n * n + (size_t)i * NB * n + j * NB;
  const T *D = a.diag + ((size_t)blockIdx.y * cols + i) * NB * NB;
  TS *out = (TS *)a.out.p + blockIdx.y * a.out.bs;
  const int rows = min(n - i * NB, NB), width = min(n - j * NB, NB);
  const T zero = S::make(0.0, 0.0);
  constexpr int PER = NB * NB / 256;
  T v[PER];
  const bool failed = a.failure.raised();
  if (a.failure.report && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) nxh_report(a.failure.report, a.failure.seq, failed ? LA_NOT_PD : LA_OK);
  if (failed) return;
#pragma unroll
  for (int k = 0; k < PER; k++) {  // every load is on its way before the first is waited for: 10.4 -> 6.2 us at n = 512
    const int e = threadIdx.x + 256 * k, r = e / NB, c = e % NB;
    v[k] = zero;
    if (r < rows && c < width && (i > j || c <= r)) v[k] = i > j ? A[(size_t)r * n + c] : D[e];
  }
#pragma unroll
  for (int k = 0; k < PER; k++) tile[(threadIdx.x + 256 * k) / NB][threadIdx.x % NB] = v[k];
  __syncthreads();
  for (int e = threadIdx.x; e < NB * NB; e += 256) {
    const int r = e / NB, c = e % NB;
    if (r < rows && c < width) {  // a diagonal tile is its own mirror image
      const T val = !a.upper ? tile[r][c] : i > j ? zero : S::conj(tile[c][r]);
      to_storage(val, out + (int64_t)(i * NB + r) * a.out.rs + (int64_t)(j * NB + c) * a.out.cs);
    }
    if (i > j && r < width && c < rows)
      to_storage(a.upper ? S::conj(tile[c][r]) : zero, out + (int64_t)(j * NB + r) * a.out.rs + (int64_t)(i * NB + c) * a.out.cs);
  }
}

// ── triangular solve ────────────────────────────────────────────────────────
// M X = B with M lower triangular after reversing the order where the substitution runs
// backwards: coefficient (t, u), t > u, is m[t ts + u us] (conjugated for a conjugate
// transpose). A workgroup solves sixteen right-hand sides, which stay in LDS, sixteen rows a
// step: wave 0 brings the next sixteen rows up to date and substitutes through their
// triangle (solve16), while other waves take the step before from the rows further down (a
// wave per 16 x 16 tile) and one lays out what wave 0 needs of the matrix for the next step. What is read
// of the matrix is requested a step or two ahead: it depends on nothing. One barrier a step, no launch.
// Where solve16 refuses, and for complex matrices, the substitution goes row by row, a right-hand
// side a lane.
// Wave 0 is the chain: it neither reads memory nor works out an address. Wave 4 (of its SIMD) reads the triangle and
// the tile left of it, inverts the 4 x 4 triangles and puts all of it in LDS as the operands that wave 0 takes, without
// a matrix instruction; the other six bring up to TILES tiles each up to date per step, up to six at a time (float64 four: six are 22 registers
// too many, [1000,1000] with sixteen sides 245 us against 240), so that their products do not wait for each other. What a tile needs
// of the matrix is in registers two steps ahead, so that TILES decides how many workgroups a compute unit
// holds (11 tiles, 177 registers, float64 244: one; float32 with 5 tiles, 116, and 2 tiles, 90 and float64 120: two). A form
// serves systems of 2 + 6 TILES blocks and fewer, eleven tiles those of a pass, 64; systems of one block, TILES = 0, have a
// single wave, which places the triangle itself. Five tiles against eleven, float32, us: 1 000 systems of 300 rows 109 / 147,
// of 512 rows, which two workgroups' LDS just holds, 268 / 326, one system of 300 rows 30.8 / 32.3. (513 to 560 rows would fit
// twice without wave 0's operands in LDS: 1 000 of 530 rows 306 then, 344 so, one 91 and 68.)
// [512,512] float32, sixteen sides: 74 us while wave 0 took 3 400 clocks a step (0.6 the tile to the left in one chain, 0.7
// addresses and conversions, 2.0 solve16) and waited for the others, tile after tile, up to 6 400; 62 so, 3 000 a step but for the first ten, whose products keep the matrix units busy.
// (The 4 x 4 triangles row by row on the vector unit, four products in the chain for fifteen: 2.3 for solve16's 2.0.)
constexpr int TRSM_WAVES = 8, TRSM_LOADER = 4, TRSM_UPDATERS = 6, TRSM_TILES = 11, TRSM_SOME = 5, TRSM_FEW = 2;
template <int TILES>
constexpr int TRSM_THREADS = TILES > 0 ? 64 * TRSM_WAVES : 64;

template <class T>
struct TrsmArgs {
  const void *m;        // coefficient (0, 0) of this pass, storage type TS
  int64_t ts, us, mbs;  // strides along t, along u, and from matrix to matrix
  int conj, unit;
  LaMat b, x;           // rows from row 0 of the solution order on; b is read, x written (TS)
  int rows, nrhs;
  LaFailure failure;
  bool checked;  // trsm_check_kernel has looked through the batch: where it found a singular matrix, nothing is written
};

// A wave per matrix: whether an element of its diagonal is zero.
template <class T, class TS>
__global__ __launch_bounds__(256) void trsm_check_kernel(TrsmArgs<T> a, int64_t batch) {
  const int64_t b = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (b >= batch) return;
  const TS *m = (const TS *)a.m + b * a.mbs;
  bool zero = false;
  for (int t = threadIdx.x & 63; t < a.rows; t += 64) zero = zero || T(m[t * (a.ts + a.us)]) == Sc<T>::make(0.0, 0.0);
  if (zero) a.failure.raise();
}

template <class T, class TS>
__device__ __forceinline__ T trsm_coefficient(const TrsmArgs<T> &a, const TS *m, int t, int u) {
  const T v = T(m[t * a.ts + u * a.us]);
  return a.conj ? Sc<T>::conj(v) : v;
}

template <class T, class TS, int TILES>
__global__ __launch_bounds__(TRSM_THREADS<TILES>, TILES == TRSM_TILES ? 2 : 4) void trsm_block_kernel(TrsmArgs<T> a) {
  using S = Sc<T>;
  constexpr int AHEAD = TILES > 0 ? 2 : 1;  // triangles in LDS
  extern __shared__ double lds_raw[];
  T *X = (T *)lds_raw;  // rows rounded up to 16, times 16
  // by columns, each from its diagonal on: element r < 16 of column t is coefficient (t + r, t), element
  // 16 (double) the inverse of the diagonal (reads past a column's end meet the next one: their results are dropped)
  constexpr int TRI_LD = 18;
  __shared__ T tri[AHEAD][17][TRI_LD];
  constexpr int REAL = sizeof(T) == 8 ? AHEAD : 1;      // (complex has none of these)
  __shared__ double diag_inv[REAL][4][64], op_tri[REAL][4][64];  // operands of solve16, the first zero outside the 4 x 4 triangles
  __shared__ TS op_left[REAL][4][64];                   // the tile to the left of the triangle (float: two workgroups of 512 rows fit)
  __shared__ int singular;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int n = a.rows, nb = (n + 15) / 16, col0 = blockIdx.x * 16;
  const TS *m = (const TS *)a.m + blockIdx.y * a.mbs;
  const TS *b = (const TS *)a.b.p + blockIdx.y * a.b.bs;
  TS *x = (TS *)a.x.p + blockIdx.y * a.x.bs;
  for (int e = threadIdx.x; e < nb * 256; e += blockDim.x) {
    const int t = e >> 4, c = col0 + (e & 15);
    X[e] = t < n && c < a.nrhs ? T(b[t * a.b.rs + c * a.b.cs]) : S::make(0.0, 0.0);
  }
  if (threadIdx.x == 0) singular = 0;
  // the triangle of block `k` and the inverses of its diagonal (past n: the identity), by one wave
  auto fetch_triangle = [&](int k, TS(&raw)[4]) {
    const int last = min(15, n - 1 - k * 16);
    const TS *p = m + k * 16 * (a.ts + a.us) + min(r16, last) * a.us;
#pragma unroll
    for (int v = 0; v < 4; v++) raw[v] = p[min(4 * v + q, last) * a.ts];
  };
  auto place_triangle = [&](int k, const TS(&raw)[4]) {
    T own = S::make(1.0, 0.0);  // the diagonal element of a lane that has one
#pragma unroll
    for (int v = 0; v < 4; v++) {
      const int t = 4 * v + q;
      const bool diagonal = t == r16;
      T val = at_hand(a.conj ? S::conj(T(raw[v])) : T(raw[v]));
      const T edge = S::make(diagonal ? 1.0 : 0.0, 0.0);
      // (assigned, not chosen: of two complex values a choice is one of two addresses, and both go to scratch memory)
      if (k * 16 + max(t, r16) >= n || r16 > t || (a.unit && diagonal)) val = edge;
      if (r16 <= t) tri[k % AHEAD][r16][t - r16] = val;
      if (diagonal) own = val;
    }
    if (own == S::make(0.0, 0.0)) singular = 1;
    if constexpr (sizeof(T) == 8) {
      const double inverse = at_hand(1.0 / at_hand(own));
      if ((r16 & 3) == q) tri[k % AHEAD][r16][16] = inverse;
      // lane (b, i, j): element (i, j) of the inverse of the b-th 4 x 4 triangle on the diagonal
      wave_sync();
      const int bb = lane >> 4, i = (lane >> 2) & 3, j = lane & 3;
      const T(*t)[TRI_LD] = &tri[k % AHEAD][4 * bb];
      double column[4];  // of the operand of a product with the triangle
#pragma unroll
      for (int u = 0; u < 4; u++) column[u] = at_hand(tri[k % AHEAD][4 * u + q][max(r16 - 4 * u - q, 0)]);
      const double e0 = at_hand(t[0][16]), e1 = at_hand(t[1][16]), e2 = at_hand(t[2][16]), e3 = at_hand(t[3][16]);
      const double l10 = at_hand(t[0][1]), l20 = at_hand(t[0][2]), l30 = at_hand(t[0][3]), l21 = at_hand(t[1][1]), l31 = at_hand(t[1][2]), l32 = at_hand(t[2][1]);
      const double m10 = at_hand(-e1 * l10 * e0), m21 = at_hand(-e2 * l21 * e1), m32 = at_hand(-e3 * l32 * e2);
      const double m20 = at_hand(-e2 * fma(l21, m10, l20 * e0)), m31 = at_hand(-e3 * fma(l32, m21, l31 * e1));
      const double m30 = at_hand(-e3 * fma(l32, m20, fma(l31, m10, l30 * e0)));
      double v = j == 0 ? m30 : j == 1 ? m31 : j == 2 ? m32 : e3;
      v = i == 2 ? (j == 0 ? m20 : j == 1 ? m21 : e2) : v;
      v = i == 1 ? (j == 0 ? m10 : e1) : v;
      v = i == 0 ? e0 : v;
      diag_inv[k % AHEAD][bb][j * 16 + 4 * bb + i] = j <= i ? v : 0.0;
#pragma unroll
      for (int u = 0; u < 4; u++) op_tri[k % AHEAD][u][lane] = r16 >= 4 * u + q ? column[u] : 0.0;
    }
  };
  for (int e = threadIdx.x; e < REAL * 256; e += blockDim.x) (&diag_inv[0][0][0])[e] = 0.0;
  // One matrix (`report`): a wave that has nothing to do yet looks through its diagonal, and the host goes on.
  if (a.failure.report && blockIdx.x == 0 && blockIdx.y == 0 && wave == (TILES > 0 ? TRSM_WAVES - 1 : 0)) {
    bool zero = false;
    if (!a.unit) {
      constexpr int LOOK = 8;
      for (int t0 = lane; t0 < n; t0 += 64 * LOOK) {
        TS d[LOOK];
#pragma unroll
        for (int j = 0; j < LOOK; j++) d[j] = m[min(t0 + 64 * j, n - 1) * (a.ts + a.us)];
#pragma unroll
        for (int j = 0; j < LOOK; j++) zero = zero || T(d[j]) == S::make(0.0, 0.0);
      }
    }
    zero = __any(zero);
    if (lane == 0) nxh_report(a.failure.report, a.failure.seq, zero ? LA_SINGULAR : LA_OK);
  }
  __syncthreads();
  // coefficients of tile `t` against block `u` < `t`, as the matrix instruction takes them
  const TS *lane_full = m + r16 * a.ts + q * a.us, *lane_last = m + min(r16, n - 1 - (nb - 1) * 16) * a.ts + q * a.us;
  auto coefficients = [&](int t, int u, TS(&c)[4]) {
    if constexpr (sizeof(T) == 8) {
      const TS *p = (t == nb - 1 ? lane_last : lane_full) + (t * a.ts + u * a.us) * 16;
#pragma unroll
      for (int k = 0; k < 4; k++) c[k] = p[4 * k * a.us];
    }
  };
  auto load_rows = [&](int t) {
    LaTile<T> acc;
#pragma unroll
    for (int v = 0; v < 4; v++) acc.v[v] = X[(t * 16 + 4 * v + q) * 16 + r16];
    return acc;
  };
  auto store_rows = [&](int t, const LaTile<T> &acc) {
#pragma unroll
    for (int v = 0; v < 4; v++) X[(t * 16 + 4 * v + q) * 16 + r16] = acc.v[v];
  };
  // what block `u` takes from block `t` (complex)
  auto take = [&](LaTile<T> &acc, int t, int u) {
    if constexpr (sizeof(T) != 8) {
      for (int k = 0; k < 16; k++) {
        const T xv = X[(u * 16 + k) * 16 + r16];
#pragma unroll
        for (int v = 0; v < 4; v++)
          acc.v[v] = S::sub_mul(acc.v[v], trsm_coefficient<T, TS>(a, m, min(t * 16 + 4 * v + q, n - 1), u * 16 + k), xv);
      }
    }
  };
  // The tile to the left of block k's triangle (real only). Nothing the loader does depends on a branch: behind one,
  // a wait for loads is a wait for all of them, also those of the step just before.
  auto place_left = [&](int k, const TS(&c)[4]) {
    if constexpr (sizeof(T) == 8) {
#pragma unroll
      for (int v = 0; v < 4; v++) op_left[k % AHEAD][v][lane] = c[v];
    }
  };
  TS raw[2][4], left[2][4];
  if (TILES == 0 || wave == TRSM_LOADER) {
    fetch_triangle(0, raw[0]);
    if constexpr (TILES > 0) coefficients(1, 0, left[1]), fetch_triangle(1, raw[1]);
    place_triangle(0, raw[0]);
    if constexpr (TILES > 0) coefficients(min(2, nb - 1), min(2, nb - 1) - 1, left[0]), fetch_triangle(min(2, nb - 1), raw[0]);
  }
  __syncthreads();
  // Three loops with the same barriers: the registers of one role are not the others'. What is read of
  // the matrix is needed two steps later and has two sets of registers in turn (a copy from one
  // to the other would wait for it): the first pass over it comes from beyond the L2, some 3500
  // cycles away.
  if (TILES == 0 || wave == 0) {
    LaTile<T> before;    // the rows solved last,
    bool known = false;  // where they are
    auto step = [&](int k) {
      LaTile<T> acc = load_rows(k);
      if constexpr (sizeof(T) == 8) {
        double di[4], tr[4];
        if (k > 0) {  // what the tile to the left takes, in two chains and apart from acc
          double l[4], x[4];
#pragma unroll
          for (int v = 0; v < 4; v++) l[v] = (double)op_left[k % AHEAD][v][lane], x[v] = before.v[v];
          if (!known) {
#pragma unroll
            for (int v = 0; v < 4; v++) x[v] = X[((k - 1) * 16 + 4 * v + q) * 16 + r16];
          }
          const la_f64x4 zero = {0.0, 0.0, 0.0, 0.0};
          la_f64x4 even = __builtin_amdgcn_mfma_f64_16x16x4f64(l[0], x[0], zero, 0, 0, 0);
          la_f64x4 odd = __builtin_amdgcn_mfma_f64_16x16x4f64(l[1], x[1], zero, 0, 0, 0);
          even = __builtin_amdgcn_mfma_f64_16x16x4f64(l[2], x[2], even, 0, 0, 0);
          odd = __builtin_amdgcn_mfma_f64_16x16x4f64(l[3], x[3], odd, 0, 0, 0);
#pragma unroll
          for (int v = 0; v < 4; v++) di[v] = diag_inv[k % AHEAD][v][lane], tr[v] = op_tri[k % AHEAD][v][lane];
#pragma unroll
          for (int v = 0; v < 4; v++) acc.v[v] -= even[v] + odd[v];
        } else {
#pragma unroll
          for (int v = 0; v < 4; v++) di[v] = diag_inv[k % AHEAD][v][lane], tr[v] = op_tri[k % AHEAD][v][lane];
        }
        known = solve16(acc, di, tr);
        if (known) {
          store_rows(k, acc);
          before = acc;
          return;
        }
      } else {
        if (k > 0) take(acc, k, k - 1);
      }
      store_rows(k, acc);
      __builtin_amdgcn_wave_barrier();
      const T(*t16)[TRI_LD] = tri[k % AHEAD];
      T v[16];  // this lane's right-hand side from row t on; it moves up one place with every row
#pragma unroll
      for (int t = 0; t < 16; t++) v[t] = X[(k * 16 + t) * 16 + r16];
#pragma unroll 1
      for (int t = 0; t < 16; t++) {
        const T sol = v[0] / t16[t][0];
        if (q == 0) X[(k * 16 + t) * 16 + r16] = sol;
#pragma unroll
        for (int r = 1; r < 16; r++) v[r - 1] = S::sub_mul(v[r], t16[t][r], sol);
      }
    };
#pragma unroll 1
    for (int k = 0; k < nb; k++) {
      step(k);
      __syncthreads();
      if constexpr (sizeof(T) != 8) {  // two steps a turn: [512,512] complex64 852 -> 837 us
        if (++k == nb) break;
        step(k);
        __syncthreads();
      }
    }
  } else if (wave == TRSM_LOADER) {
    auto step = [&](int k, TS(&r)[4], TS(&l)[4]) {
      place_left(k + 1, l), place_triangle(k + 1, r);  // (past the last: the identity, for nobody)
      const int ahead = min(k + 3, nb - 1);
      coefficients(ahead, ahead - 1, l), fetch_triangle(ahead, r);
    };
#pragma unroll 1
    for (int k = 0; k < nb; k += 2) {
      step(k, raw[1], left[1]);
      __syncthreads();
      if (k + 1 < nb) {
        step(k + 1, raw[0], left[0]);
        __syncthreads();
      }
    }
  } else if constexpr (TILES > 0) {
    const int first = wave < TRSM_LOADER ? wave : wave - 1;  // 1 .. TRSM_UPDATERS
    TS c[2][TILES][4];
    auto request = [&](int k, TS(&to)[TILES][4]) {  // what step `k` takes
#pragma unroll
      for (int i = 0; i < TILES; i++) {
        const int t = k + first + i * TRSM_UPDATERS;
        if (t >= nb) break;
        coefficients(t, k - 1, to[i]);
      }
    };
    // G tiles from tile t on, every TRSM_UPDATERS: their rows less what the solved block x takes from them (coefficients: from)
    auto tiles = [&](auto g_c, int t, const double(&x)[4], const TS(*from)[4]) {
      constexpr int G = decltype(g_c)::value;
      if constexpr (sizeof(T) == 8) {
        la_f64x4 d[G];
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
          for (int v = 0; v < 4; v++) d[i][v] = X[((t + i * TRSM_UPDATERS) * 16 + 4 * v + q) * 16 + r16];
#pragma unroll
        for (int v = 0; v < 4; v++)
#pragma unroll
          for (int i = 0; i < G; i++) d[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(-(double)from[i][v], x[v], d[i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < G; i++)
#pragma unroll
          for (int v = 0; v < 4; v++) X[((t + i * TRSM_UPDATERS) * 16 + 4 * v + q) * 16 + r16] = d[i][v];
      }
    };
    auto step = [&](int k, TS(&from)[TILES][4]) {
      if constexpr (sizeof(T) == 8) {
        if (k > 0) {
          double x[4];
#pragma unroll
          for (int v = 0; v < 4; v++) x[v] = X[((k - 1) * 16 + 4 * v + q) * 16 + r16];
          constexpr int AT_ONCE = sizeof(TS) == 8 ? 4 : 6, MOST = TILES < AT_ONCE ? TILES : AT_ONCE;
#pragma unroll
          for (int i = 0; i < TILES; i += MOST) {
            const int t = k + first + i * TRSM_UPDATERS;
            if (t >= nb) break;
            const int more = min((nb - 1 - t) / TRSM_UPDATERS + 1, min(TILES - i, MOST));
            const auto some = [&](auto g_c) {
              constexpr int G = decltype(g_c)::value;
              if constexpr (G <= MOST)
                if (G <= TILES - i) tiles(g_c, t, x, &from[i]);
            };
            switch (more) {
              case 1: some(std::integral_constant<int, 1>{}); break;
              case 2: some(std::integral_constant<int, 2>{}); break;
              case 3: some(std::integral_constant<int, 3>{}); break;
              case 4: some(std::integral_constant<int, 4>{}); break;
              case 5: some(std::integral_constant<int, 5>{}); break;
              default: some(std::integral_constant<int, 6>{}); break;
            }
          }
        }
      } else if (k > 0) {
#pragma unroll
        for (int i = 0; i < TILES; i++) {
          const int t = k + first + i * TRSM_UPDATERS;
          if (t < nb) {
            LaTile<T> acc = load_rows(t);
            take(acc, t, k - 1);
            store_rows(t, acc);
          }
        }
      }
      if (k + 2 < nb) request(k + 2, from);
    };
    if (nb > 1) request(1, c[1]);
#pragma unroll 1
    for (int k = 0; k < nb; k += 2) {
      step(k, c[0]);
      __syncthreads();
      if (k + 1 < nb) {
        step(k + 1, c[1]);
        __syncthreads();
      }
    }
  }
  // (every workgroup of a matrix has seen its whole diagonal)
  if (singular || (a.checked && a.failure.raised())) {
    if (threadIdx.x == 0 && singular) a.failure.raise();
    return;
  }
  for (int e = threadIdx.x; e < n * 16; e += blockDim.x) {
    const int t = e >> 4, c = col0 + (e & 15);
    if (c < a.nrhs) to_storage(X[e], x + t * a.x.rs + c * a.x.cs);
  }
}

// Rows after a pass: X[t] -= sum_u M(t, u) X[u] over the pass's rows, for the next pass to solve
// (only systems longer than one pass holds come here). A wave per 16 x 16 tile; right-hand sides
// in the grid's x extent, which has room for any number of them.
template <class T, class TS>
__global__ __launch_bounds__(256) void trsm_rest_kernel(TrsmArgs<T> a, LaMat rest, int rest_rows) {
  using S = Sc<T>;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r16 = lane & 15, q = lane >> 4;
  const int t0 = (blockIdx.y * 4 + wave) * 16, c = blockIdx.x * 16 + r16;
  if (t0 >= rest_rows) return;
  const TS *m = (const TS *)a.m + blockIdx.z * a.mbs;
  const TS *x = (const TS *)a.x.p + blockIdx.z * a.x.bs;
  TS *y = (TS *)rest.p + blockIdx.z * rest.bs;
  const int cc = min(c, a.nrhs - 1);
  T acc[4];
#pragma unroll
  for (int v = 0; v < 4; v++) acc[v] = T(y[min(t0 + 4 * v + q, rest_rows - 1) * rest.rs + cc * rest.cs]);
  for (int u = 0; u < a.rows; u++) {
    const T xv = T(x[u * a.x.rs + cc * a.x.cs]);
#pragma unroll
    for (int v = 0; v < 4; v++)
      acc[v] = S::sub_mul(acc[v], trsm_coefficient<T, TS>(a, m, a.rows + min(t0 + 4 * v + q, rest_rows - 1), u), xv);
  }
  if (c >= a.nrhs) return;
#pragma unroll
  for (int v = 0; v < 4; v++)
    if (t0 + 4 * v + q < rest_rows) to_storage(acc[v], y + (t0 + 4 * v + q) * rest.rs + c * rest.cs);
}

// ── many small complex systems ──────────────────────────────────────────────
// The complex forms above are chains of one wave, with no matrix instruction to shorten them; a thousand of
// them queue up. Matrices of up to 64 rows then take a workgroup each whose lanes share every link: a
// column of the factor with a row a lane; a row of the solution, then its elimination from the others,
// with an element a lane. In place in a workspace of the compute type.
template <class T>
__global__ __launch_bounds__(LA_THREADS) void cholesky_small_kernel(T *all, int n, int upper, int *status) {
  using S = Sc<T>;
  T *A = all + (size_t)blockIdx.x * n * n;
  __shared__ int failed;
  if (threadIdx.x == 0) failed = 0;
  for (int j = 0; j < n; j++) {
    for (int i = j + threadIdx.x; i < n; i += blockDim.x) {
      T s = A[(size_t)i * n + j];
      const T *ri = A + (size_t)i * n, *rj = A + (size_t)j * n;
      for (int k = 0; k < j; k++) s = s - ri[k] * S::conj(rj[k]);
      A[(size_t)i * n + j] = s;
    }
    __syncthreads();
    const double d = S::re(A[(size_t)j * n + j]);
    if (threadIdx.x == 0 && !(d > 0.0)) failed = 1;
    __syncthreads();
    if (failed) {
      if (threadIdx.x == 0) raise(status, LA_NOT_PD);
      return;
    }
    const double l = sqrt(d);
    for (int i = j + threadIdx.x; i < n; i += blockDim.x)
      A[(size_t)i * n + j] = i == j ? S::make(l, 0.0) : S::scale(A[(size_t)i * n + j], 1.0 / l);
    __syncthreads();
  }
  // the other triangle: zero for L; for U the conjugate transpose moves there first
  for (int64_t e = threadIdx.x; e < (int64_t)n * n; e += blockDim.x) {
    const int i = (int)(e / n), k = (int)(e % n);
    if (i <= k) continue;
    if (upper) {
      A[(size_t)k * n + i] = S::conj(A[e]);
      A[e] = S::make(0.0, 0.0);
    } else {
      A[(size_t)k * n + i] = S::make(0.0, 0.0);
    }
  }
}

template <class T>
__global__ __launch_bounds__(LA_THREADS) void trsm_small_kernel(const T *a_all, T *x_all, int n, int nrhs, int upper,
                                                                int transpose, int unit, int *status) {
  using S = Sc<T>;
  const T *A = a_all + (size_t)blockIdx.x * n * n;
  T *X = x_all + (size_t)blockIdx.x * n * nrhs;
  const bool forward = (upper != 0) == (transpose != 0);
  for (int ii = 0; ii < n; ii++) {
    const int i = forward ? ii : n - 1 - ii;
    if (!unit) {
      T diag = A[(size_t)i * n + i];
      if (transpose) diag = S::conj(diag);
      if (diag == S::make(0.0, 0.0)) {  // uniform: every lane reads the same element
        if (threadIdx.x == 0) raise(status, LA_SINGULAR);
        return;
      }
      for (int j = threadIdx.x; j < nrhs; j += blockDim.x) X[(size_t)i * nrhs + j] = X[(size_t)i * nrhs + j] / diag;
      __syncthreads();
    }
    const int rest = n - 1 - ii;  // rows not yet solved
    for (int64_t e = threadIdx.x; e < (int64_t)rest * nrhs; e += blockDim.x) {
      const int rr = (int)(e / nrhs), j = (int)(e % nrhs);
      const int r = forward ? i + 1 + rr : i - 1 - rr;
      const T m = transpose ? S::conj(A[(size_t)i * n + r]) : A[(size_t)r * n + i];
      X[(size_t)r * nrhs + j] = X[(size_t)r * nrhs + j] - m * X[(size_t)i * nrhs + j];
    }
    __syncthreads();
  }
}
