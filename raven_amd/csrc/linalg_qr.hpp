// linalg_qr.hpp — Householder QR of float64 matrices by panels of sixteen columns (included by
// linalg.hip, inside its namespace).
//
// A column of a panel waits for the one before it: that chain is one workgroup per matrix, the panel
// in registers, one barrier a column. Everything else is two products per panel, V^T X and X - V W,
// on the f64 matrix instruction over the whole device (compact WY: H_0 .. H_15 = I - V T V^T).
// A launch per column and pass over the matrix, which this replaces, was bound by the launches, and a
// workgroup per small matrix by its walks over memory: [796,796] float64 11.3 -> 2.1 ms, [2048,2048] 55 -> 11.9, ten of
// [44,44] 411 -> 106 us, a hundred of [100,100] 1 130 -> 208. What bounds it now: the panels' chain (28 us for 512
// rows of sixteen columns, 20 of them the columns) and two applications of 10 us per panel. Root mean squares over
// some hundred normal matrices of 8 to 2048 rows: |Q R - A| 0.62 to 1.00 of what it was, |Q^T Q - I| 0.64 to 1.04.
#pragma once

constexpr int QR_NB = 16;
constexpr int QR_ROWS = 2048;  // the tallest panel held in registers

// Broadcasts lane J of every sixteen.
template <int J>
__device__ __forceinline__ double bcast16(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x150 + J, 0xf, 0xf, false);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x150 + J, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}

struct QrPanelArgs {
  double *at;  // [batch][n][m] column by column; on return R above and on the diagonal of the panel, zeros below
  double *v;   // [batch][k][m]: the panel's reflectors with their ones and zeros, rows from p0 on
  double *t;   // [batch][panels][16][16]: T, row by row
  int m, n, k, p0, panels;
};

// Lane (q, c) = 16 q + c of wave w holds rows 4 (e W + w) + q, e < E, of column c, counted from the
// panel's first row. The dot products of column j with every column (its own gives the norm, the
// later ones what the reflector takes from them) are then one
// fused step per element, two exchanges and one sum over the waves. The waves share four SIMDs, so a
// column is bound by the instructions per element: the reflectors are not scaled before the end (the
// scale goes into the coefficient of what a column takes), which leaves two fused steps and a
// broadcast in the register file.
template <int W, int E>
__global__ __launch_bounds__(64 * W) void qr_panel_kernel(QrPanelArgs a) {
  __shared__ double part[2][W][16], rowj[2][16], z[W][16][17], taus[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int rows = a.m - a.p0, w = min(QR_NB, a.k - a.p0);
  double *A = a.at + ((size_t)blockIdx.x * a.n + a.p0) * a.m + a.p0;
  auto row_of = [&](int e) { return 4 * (e * W + wave) + q; };
  constexpr int HEAD = W >= 4 ? 1 : 4 / W;  // elements that may lie in the first sixteen rows
  // Sixteen waves leave a lane 128 registers, which x fills by half: there the reflector is broadcast again for the
  // update instead of kept.
  constexpr bool KEEP = W < 16;
  double x[E], biggest = 0.0;
#pragma unroll
  for (int e = 0; e < E; e++) {
    x[e] = c < w && row_of(e) < rows ? A[(size_t)c * a.m + row_of(e)] : 0.0;
    biggest = fmax(biggest, fabs(x[e]));  // (passes over a NaN)
  }
  // The products below are of two columns as they come: a column whose square, or whose product with another, would
  // leave float64's range is worked on times a power of two and stored times its inverse. Columns between
  // 2^-400 and 2^480 are left alone; the others come to 2^0 and 2^400, the large ones so that their small
  // elements keep their bits.
  biggest = fmax(biggest, __shfl_xor(biggest, 16));
  biggest = fmax(biggest, __shfl_xor(biggest, 32));
  if constexpr (W > 1) {
    if (q == 0) part[1][wave][c] = biggest;  // (column 1 is the next to use it, a barrier later)
    __syncthreads();
#pragma unroll
    for (int i = 0; i < W; i++) biggest = fmax(biggest, part[1][i][c]);
  }
  int power = 0;
  if (biggest > 0.0 && biggest < __builtin_inf()) {
    const int ex = __builtin_amdgcn_frexp_exp(biggest);
    power = ex < -400 ? ex : ex > 480 ? ex - 400 : 0;
  }
  if (__any(power != 0)) {
#pragma unroll
    for (int e = 0; e < E; e++) x[e] = ldexp(x[e], -power);
  }
  // x / y, rounded, by the reciprocal of y: its own error is the same in every element
  auto divided = [](double x, double y, double inv) {
    const double d = x * inv;
    return fma(fma(-d, y, x), inv, d);
  };
  double my_scal = 1.0, my_rs = 1.0, my_beta = 0.0;  // of this lane's column, once it is done
  bool reflected = false;
  auto column = [&](auto jc) {
    constexpr int j = decltype(jc)::value, buf = j & 1;
    if (j >= w) return;
    constexpr int OWNER = W >= 4 ? j / 4 : 0, AT = W >= 4 ? 0 : j / 4;  // where row j is
    if (wave == OWNER && q == j % 4) rowj[buf][c] = x[AT];
    // the reflector's element of a lane's row, unscaled, and zero above the row below the diagonal
    auto reflector = [&](int e) {
      const double v = bcast16<j>(x[e]);
      return e < HEAD && row_of(e) <= j ? 0.0 : v;
    };
    double b[KEEP ? E : 1], p4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < E; e++) {
      const double v = reflector(e);
      if constexpr (KEEP) b[e] = v;
      // (rows that are done have no part in the sums: they may hold an infinity)
      p4[e & 3] = fma(v, e < HEAD && row_of(e) <= j ? 0.0 : x[e], p4[e & 3]);
    }
    double s = (p4[0] + p4[1]) + (p4[2] + p4[3]);
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if constexpr (W > 1) {
      if (q == 0) part[buf][wave][c] = s;
      __syncthreads();
      double p[W / 2];
#pragma unroll
      for (int i = 0; i < W / 2; i++) {
        p[i] = part[buf][i][c] + part[buf][i + W / 2][c];
        if (!KEEP && i % 2) __builtin_amdgcn_sched_barrier(0);  // (not all of them in registers at once)
      }
#pragma unroll
      for (int d = W / 4; d > 0; d /= 2)
#pragma unroll
        for (int i = 0; i < d; i++) p[i] += p[i + d];
      s = p[0];
    } else {
      wave_sync();
    }
    const double r = rowj[buf][c], alpha = bcast16<j>(r), norm2 = bcast16<j>(s);
    double tau = 0.0;
    if (norm2 != 0.0) {  // (uniform)
      // (the root to the last bit: the reflector is as orthogonal as its norm is exact)
      const double root = sqrt(fma(alpha, alpha, norm2));
      const double beta = alpha >= 0.0 ? -root : root, scal = alpha - beta, rs = 1.0 / scal;
      tau = (beta - alpha) / beta;
      const double wc = c > j ? tau * (divided(s, scal, rs) + r) : 0.0, wb = divided(wc, scal, rs);  // v . this lane's column, by tau
#pragma unroll
      for (int e = 0; e < E; e++) {
        double v;
        if constexpr (KEEP) {
          v = b[e];
        } else {
          asm volatile("" : "+v"(x[e]));  // (or the compiler keeps the first broadcast, in scratch memory)
          v = reflector(e);
        }
        x[e] = fma(-v, wb, x[e]);
        if (e < HEAD) x[e] = row_of(e) == j ? x[e] - wc : x[e];
        if constexpr (!KEEP) asm volatile("" : "+v"(x[e]));
        }
      if (c == j) my_scal = scal, my_rs = rs, my_beta = beta, reflected = true;
    }
    if (threadIdx.x == 0) taus[j] = tau;
  };
  column(std::integral_constant<int, 0>{});
  column(std::integral_constant<int, 1>{});
  column(std::integral_constant<int, 2>{});
  column(std::integral_constant<int, 3>{});
  column(std::integral_constant<int, 4>{});
  column(std::integral_constant<int, 5>{});
  column(std::integral_constant<int, 6>{});
  column(std::integral_constant<int, 7>{});
  column(std::integral_constant<int, 8>{});
  column(std::integral_constant<int, 9>{});
  column(std::integral_constant<int, 10>{});
  column(std::integral_constant<int, 11>{});
  column(std::integral_constant<int, 12>{});
  column(std::integral_constant<int, 13>{});
  column(std::integral_constant<int, 14>{});
  column(std::integral_constant<int, 15>{});
  // the reflectors, scaled, and V^T V of what is stored: a lane's element is where both operands want it
  la_f64x4 vtv = {0.0, 0.0, 0.0, 0.0};
  double *V = a.v + ((size_t)blockIdx.x * a.k + a.p0 + c) * a.m + a.p0;
#pragma unroll
  for (int e = 0; e < E; e++) {
    const int row = row_of(e);
    const bool in = c < w && row < rows;
    const double v = !in || row < c ? 0.0 : row == c ? 1.0 : divided(x[e], my_scal, my_rs);
    vtv = __builtin_amdgcn_mfma_f64_16x16x4f64(v, v, vtv, 0, 0, 0);
    if (in) {
      A[(size_t)c * a.m + row] = row > c ? 0.0 : ldexp(row == c && reflected ? my_beta : x[e], power);
      V[row] = v;
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) z[wave][4 * v + q][c] = vtv[v];
  if constexpr (W > 1) __syncthreads();
  else wave_sync();
  if (wave > 0) return;
  if constexpr (W > 1) {
#pragma unroll
    for (int v = 0; v < 4; v++) {
      double sum = z[0][4 * v + q][c];
#pragma unroll
      for (int i = 1; i < W; i++) sum += z[i][4 * v + q][c];
      z[0][4 * v + q][c] = sum;
    }
    wave_sync();
  }
  // T, a row a lane: T(i, j) = -tau_j sum over i <= k < j of T(i, k) z(k, j), tau_j on the diagonal
  if (lane < 16) {
    double *to = a.t + ((size_t)blockIdx.x * a.panels + a.p0 / QR_NB) * 256 + lane * 16;
    double row[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      double sum = 0.0;
#pragma unroll
      for (int k = 0; k < j; k++) sum = fma(row[k], k >= lane && j < w ? z[0][k][j] : 0.0, sum);
      const double tau = j < w ? taus[j] : 0.0;
      row[j] = j < lane ? 0.0 : j == lane ? tau : -tau * sum;
      to[j] = row[j];
    }
  }
}

struct QrApplyArgs {
  const double *v, *t;  // as the panels leave them
  double *x;            // [batch][cols][m]
  int m, k, p0, panels, cols, first, transpose;  // columns from `first` on; T^T (factoring) or T (forming Q)
};

// X <- (I - V T V^T) X, or with T^T, rows from p0 on: a workgroup per sixteen columns. Its eight
// waves share the rows of V^T X and meet in LDS, then each brings tiles of sixteen rows up to date.
// (X kept in registers between the two, in the instruction's own layout: 15 us against 10 at 512 rows, for
// its loads are eight bytes a lane.)
constexpr int QR_APPLY_WAVES = 8;
__global__ __launch_bounds__(64 * QR_APPLY_WAVES) void qr_apply_kernel(QrApplyArgs a) {
  typedef double f64x2 __attribute__((ext_vector_type(2)));
  typedef f64x2 f64x2_at8 __attribute__((aligned(8)));
  __shared__ double part[QR_APPLY_WAVES][4][64], wt[16][17], w2[16][17], tm[16][17];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int rows = a.m - a.p0, w = min(QR_NB, a.k - a.p0);
  const int col0 = a.first + (int)blockIdx.x * 16, cols = min(16, a.cols - col0);
  const double *V = a.v + ((size_t)blockIdx.y * a.k + a.p0) * a.m + a.p0;
  double *X = a.x + ((size_t)blockIdx.y * a.cols + col0) * a.m + a.p0;
  const double *T = a.t + ((size_t)blockIdx.y * a.panels + a.p0 / QR_NB) * 256;
  if (threadIdx.x < 256) tm[threadIdx.x >> 4][threadIdx.x & 15] = T[a.transpose ? (threadIdx.x & 15) * 16 + (threadIdx.x >> 4) : threadIdx.x];
  // (lanes past the last column read column 0 and drop it: zero in V, not stored in X)
  const double *vc = V + (size_t)(c < w ? c : 0) * a.m, *xc = X + (size_t)(c < cols ? c : 0) * a.m;
  // V^T X: eight rows a step, two of them a lane
  la_f64x4 acc = {0.0, 0.0, 0.0, 0.0};
  const int steps = (rows + 7) / 8;
  for (int s0 = wave; s0 < steps; s0 += 4 * QR_APPLY_WAVES) {
    f64x2 va[4], xb[4];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int r = (s0 + u * QR_APPLY_WAVES) * 8 + 2 * q;
      va[u] = xb[u] = f64x2{0.0, 0.0};
      if (r + 2 <= rows) {
        va[u] = *reinterpret_cast<const f64x2_at8 *>(vc + r);
        xb[u] = *reinterpret_cast<const f64x2_at8 *>(xc + r);
      } else if (r < rows) {
        va[u][0] = vc[r];
        xb[u][0] = xc[r];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; u++) {
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c < w ? va[u][0] : 0.0, xb[u][0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c < w ? va[u][1] : 0.0, xb[u][1], acc, 0, 0, 0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; v++) part[wave][v][lane] = acc[v];
  __syncthreads();
  if (threadIdx.x < 256) {  // element (4 v + q, c) of V^T X
    const int v = threadIdx.x >> 6;
    double sum = part[0][v][lane];
#pragma unroll
    for (int i = 1; i < QR_APPLY_WAVES; i++) sum += part[i][v][lane];
    wt[4 * v + q][c] = sum;
  }
  __syncthreads();
  if (threadIdx.x < 256) {
    const int i = threadIdx.x >> 4, j = threadIdx.x & 15;
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < 16; k++) sum = tm[i][k] != 0.0 ? fma(tm[i][k], wt[k][j], sum) : sum;  // (no part in it: X may hold an infinity)
    w2[i][j] = sum;
  }
  __syncthreads();
  // X^T -= W^T V^T, so that lanes next to each other hold rows next to each other: register v of lane (q, r)
  // is row r of column 4 v + q. The product is summed apart from X: one rounding at its size and not
  // sixteen (|Q^T Q - I| of [44,44]: 4.6e-15 so, 3.2e-15 with a reflector at a time).
  double wa[4];
#pragma unroll
  for (int s = 0; s < 4; s++) wa[s] = 4 * s + q < w ? w2[4 * s + q][c] : 0.0;
  for (int r0 = wave * 16; r0 < rows; r0 += 16 * QR_APPLY_WAVES) {
    const int r = r0 + c;
    const bool in = r < rows;
    double vb[4];
    la_f64x4 x, d = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int s = 0; s < 4; s++) vb[s] = in && 4 * s + q < w ? V[(size_t)(4 * s + q) * a.m + r] : 0.0;
#pragma unroll
    for (int v = 0; v < 4; v++) x[v] = in && 4 * v + q < cols ? X[(size_t)(4 * v + q) * a.m + r] : 0.0;
#pragma unroll
    for (int s = 0; s < 4; s++) d = __builtin_amdgcn_mfma_f64_16x16x4f64(wa[s], vb[s], d, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; v++)
      if (in && 4 * v + q < cols) X[(size_t)(4 * v + q) * a.m + r] = x[v] - d[v];
  }
}

// The same reflector by reflector, X and V in registers as in qr_panel_kernel: a column's chain per panel where
// the products with T take two passes, and as exact as a reflector at a time was for small matrices too.
// The products round at the panel's size: |Q^T Q - I| of [16,16] 2.39e-15, so 1.69e-15 (before panels 1.74e-15);
// [64,64] 5.6, 4.8 and 4.9; [96,96] 7.00, 6.82 and 6.91; from 100 columns on they are as exact ([100,100] 7.05 and
// 7.12) and |Q R - A| is smaller. Time: [44,44] 85 -> 106 us, [96,96] 163 -> 226 (before panels 396 and 803).
constexpr int QR_SINGLY = 96;         // columns up to which
constexpr int QR_SINGLY_ROWS = 1024;  // the tallest panel of which both fit (taller: |Q^T Q - I| 0.4 to 4 % larger than before panels)
template <class F, int... J>
__device__ __forceinline__ void qr_each(F &&f, std::integer_sequence<int, J...>) {
  (f(std::integral_constant<int, J>{}), ...);
}
template <int W, int E>
__global__ __launch_bounds__(64 * W) void qr_reflect_kernel(QrApplyArgs a) {
  __shared__ double part[2][W][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 15, q = lane >> 4;
  const int rows = a.m - a.p0, w = min(QR_NB, a.k - a.p0);
  const int col0 = a.first + (int)blockIdx.x * 16, cols = min(16, a.cols - col0);
  const double *V = a.v + ((size_t)blockIdx.y * a.k + a.p0 + c) * a.m + a.p0;
  double *X = a.x + ((size_t)blockIdx.y * a.cols + col0 + c) * a.m + a.p0;
  const double *T = a.t + ((size_t)blockIdx.y * a.panels + a.p0 / QR_NB) * 256;
  auto row_of = [&](int e) { return 4 * (e * W + wave) + q; };
  constexpr int HEAD = W >= 4 ? 1 : 4 / W;
  double x[E], v[E];
#pragma unroll
  for (int e = 0; e < E; e++) {
    x[e] = c < cols && row_of(e) < rows ? X[row_of(e)] : 0.0;
    v[e] = c < w && row_of(e) < rows ? V[row_of(e)] : 0.0;
  }
  const double taus = c < w ? T[c * 17] : 0.0;
  int buf = 0;
  auto reflect = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    const double tau = bcast16<j>(taus);
    if (j >= w || tau == 0.0) return;  // (uniform)
    double p4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < E; e++)  // (rows above the reflector have no part in it: they may hold an infinity)
      p4[e & 3] = fma(bcast16<j>(v[e]), e < HEAD && row_of(e) < j ? 0.0 : x[e], p4[e & 3]);
    double s = (p4[0] + p4[1]) + (p4[2] + p4[3]);
    s += __shfl_xor(s, 16);
    s += __shfl_xor(s, 32);
    if constexpr (W > 1) {
      if (q == 0) part[buf][wave][c] = s;
      __syncthreads();
      double p[W / 2];
#pragma unroll
      for (int i = 0; i < W / 2; i++) p[i] = part[buf][i][c] + part[buf][i + W / 2][c];
#pragma unroll
      for (int d = W / 4; d > 0; d /= 2)
#pragma unroll
        for (int i = 0; i < d; i++) p[i] += p[i + d];
      s = p[0];
      buf ^= 1;
    }
    const double wc = tau * s;
#pragma unroll
    for (int e = 0; e < E; e++) {
      asm volatile("" : "+v"(v[e]));  // (broadcast again: kept, they would take the registers of x or v)
      x[e] = fma(-bcast16<j>(v[e]), wc, x[e]);
      asm volatile("" : "+v"(x[e]));
    }
  };
  if (a.transpose) qr_each(reflect, std::make_integer_sequence<int, QR_NB>{});
  else qr_each([&](auto jc) { reflect(std::integral_constant<int, QR_NB - 1 - decltype(jc)::value>{}); }, std::make_integer_sequence<int, QR_NB>{});
#pragma unroll
  for (int e = 0; e < E; e++)
    if (c < cols && row_of(e) < rows) X[row_of(e)] = x[e];
}

// Q R of `batch` column-major matrices of at most QR_ROWS rows: R in At, Q's first nq columns in Qt.
static int run_qr_blocked(nxh_context *ctx, const char *op, int64_t batch, int m, int n, int nq, double *At, double *Qt) {
  const int k = std::min(m, n), panels = (k + QR_NB - 1) / QR_NB;
  void *v = nullptr, *t = nullptr;
  int rc = nxh_alloc_locked(ctx, sizeof(double) * (size_t)batch * k * m, &v);
  if (!rc) rc = nxh_alloc_locked(ctx, sizeof(double) * (size_t)batch * panels * 256, &t);
  if (!rc) {
    const int64_t qcount = batch * m * nq;
    if (qcount > 0) hipLaunchKernelGGL(qr_wide_identity<double>, dim3(la_blocks(qcount)), dim3(LA_THREADS), 0, ctx->stream, Qt, m, nq, qcount);
    for (int64_t b0 = 0; b0 < batch; b0 += LA_GRID_BATCH) {
      const unsigned nb = (unsigned)std::min(LA_GRID_BATCH, batch - b0);
      double *vb = (double *)v + b0 * k * m, *tb = (double *)t + b0 * panels * 256;
      auto apply = [&](int p0, double *x, int cols, int first, int transpose) {
        if (first >= cols) return;
        const QrApplyArgs a{vb, tb, x, m, k, p0, panels, cols, first, transpose};
        const dim3 grid((unsigned)((cols - first + 15) / 16), nb);
        const int rows = m - p0;
        if (k > QR_SINGLY || m > QR_SINGLY_ROWS) hipLaunchKernelGGL(qr_apply_kernel, grid, dim3(64 * QR_APPLY_WAVES), 0, ctx->stream, a);
        else if (rows <= 64) hipLaunchKernelGGL((qr_reflect_kernel<1, 16>), grid, dim3(64), 0, ctx->stream, a);
        else if (rows <= 256) hipLaunchKernelGGL((qr_reflect_kernel<4, 16>), grid, dim3(256), 0, ctx->stream, a);
        else if (rows <= 512) hipLaunchKernelGGL((qr_reflect_kernel<8, 16>), grid, dim3(512), 0, ctx->stream, a);
        else hipLaunchKernelGGL((qr_reflect_kernel<8, 32>), grid, dim3(512), 0, ctx->stream, a);
      };
      for (int p0 = 0; p0 < k; p0 += QR_NB) {
        QrPanelArgs a{At + b0 * n * m, vb, tb, m, n, k, p0, panels};
        const int rows = m - p0;
        // as few waves as hold the panel in 16 or 32 elements a lane: a column's chain is shorter with fewer to meet
        if (rows <= 64) hipLaunchKernelGGL((qr_panel_kernel<1, 16>), dim3(nb), dim3(64), 0, ctx->stream, a);
        else if (rows <= 256) hipLaunchKernelGGL((qr_panel_kernel<4, 16>), dim3(nb), dim3(256), 0, ctx->stream, a);
        else if (rows <= 512) hipLaunchKernelGGL((qr_panel_kernel<8, 16>), dim3(nb), dim3(512), 0, ctx->stream, a);
        else if (rows <= 1024) hipLaunchKernelGGL((qr_panel_kernel<8, 32>), dim3(nb), dim3(512), 0, ctx->stream, a);
        else hipLaunchKernelGGL((qr_panel_kernel<16, 32>), dim3(nb), dim3(1024), 0, ctx->stream, a);
        apply(p0, At + b0 * n * m, n, p0 + std::min(QR_NB, k - p0), 1);
      }
      for (int p0 = (panels - 1) * QR_NB; p0 >= 0; p0 -= QR_NB) apply(p0, Qt + b0 * nq * m, nq, p0, 0);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) rc = nxh_hip_fail(op, e);
  }
  if (t) nxh_free_locked(ctx, t);
  if (v) nxh_free_locked(ctx, v);
  return rc;
}
