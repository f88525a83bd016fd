// fft.hip — fft / ifft / rfft / irfft (packages/nx/lib/backend_c/nx_c_fft.c).
//
// Contract kept from the reference (nx_c_fft.c:30-32, 940-1144): transforms are
// UNNORMALISED (fft is the -sign DFT, ifft the +sign DFT without 1/n); all
// arithmetic is double precision, complex64 upcasts on load and rounds once on
// store; several axes are repeated 1-D passes in the order given, the first
// reading the input, the later ones transforming the output in place; rfft is
// the full transform of the real line keeping n/2+1 bins along the LAST listed
// axis, which is transformed first; irfft transforms the other axes first (in a
// complex128 temporary), then rebuilds the length-s spectrum of the last axis by
// conjugate symmetry (zero-padding or truncating the supplied half) and keeps
// the real part of its +sign transform.
//
// How it runs here: one axis pass = one launch in which a workgroup owns one
// line (or several short ones), loads it into registers as double2, transforms it
// by butterflies of up to sixteen elements per lane with exchanges through LDS in
// between, and stores it from registers, so a pass reads and writes the tensor
// exactly once. Real lines of an even length are transformed as complex lines of
// half the length (float64 ones where that is as exact). Lengths that are not a power of two go through Bluestein's
// identity inside the same kernel: chirp on load, a power-of-two convolution of
// length M >= 2n-1, chirp on store.
// Transforms longer than the LDS holds (power of two above 8192, other lengths
// above 4096) are staged through a complex128 workspace and done as a four-step
// (n = n1 x n2) pair of passes of the same kernel.
//
// Twiddles, chirps and chirp-filter spectra are built on the device with
// sincospi on exactly reduced arguments, once per (length, sign) and context,
// and kept until the context is destroyed (the reference's plan cache,
// nx_c_fft.c:34-44).

#include "nxh_common.hpp"

namespace {

constexpr int FFT_MAXD = 8;         // other dims of a tensor's lines after merging
constexpr int FFT_LOG_MAX = 13;
constexpr int FFT_LDS_MAX = 1 << FFT_LOG_MAX;  // longest transform held by one workgroup (68 KiB of LDS)
constexpr int64_t FFT_WORK_ELEMS = int64_t(1) << 25;  // workspace elements per chunk of lines (512 MiB)

enum Kind { K_C32 = 0, K_C64 = 1, K_F32 = 2, K_F64 = 3 };
enum LoadMode { LOAD_COMPLEX = 0, LOAD_REAL = 1, LOAD_HERMITIAN = 2 };
// Real lines of an even length 2n go as one complex line of length n whose element j is the pair
// (2j, 2j + 1), at half the arithmetic and LDS of the transform of the real line itself. Of float64
// lines only where that is no less exact than radix-2 stages over the whole line: spectra of 512 elements on
// (error in eps, stages / packed: 16 1.05 / 1.13, 256 1.71 / 1.76, 512 1.84 / 1.81, 5000 4.38 / 4.05), and no
// inverses (a whole transform drops half its error with the imaginary parts: 2048 1.72 / 1.99, 500 2.78 / 4.02).
// The rounding of float32 covers all of that.
enum Pack { PACK_NONE = 0, PACK_RFFT = 1, PACK_IRFFT = 2 };

static inline int kind_size(int k) { return k == K_C32 ? 8 : k == K_C64 ? 16 : k == K_F32 ? 4 : 8; }

// Every line of a tensor along one axis: line l is decoded over `dims`
// (row-major) into an element offset, element j of it is `estride` further each.
struct Lines {
  char *base;
  int kind, nd;
  int64_t dims[FFT_MAXD], strides[FFT_MAXD];
  int64_t estride;
};

struct FftArgs {
  Lines in, out;
  int64_t lines, line0;  // lines in total; first line of this launch (workspace passes address from line0)
  int n;                 // transform length
  int M, logM;           // LDS transform length: n, or the Bluestein convolution length
  int n_load, load_mode, herm_s;
  int n_store;           // (PACK_IRFFT: pairs; PACK_RFFT: bins before the last, which goes by itself)
  int sign;              // -1 forward, +1 inverse
  int pack;              // n is then half the real length
  int pair_aligned;      // the real side's float32 pairs lie side by side at addresses that are multiples of a pair
  int G;                 // lines per workgroup
  // The workgroup's G lines are neighbours in memory while a line's own elements are strided
  // (a transform down the columns of a row-major tensor): consecutive lanes then take the
  // same element of consecutive lines, so that a wave's accesses are contiguous runs of G
  // elements instead of 64 separate ones. Separately for the load and the store side.
  int in_lines_fast, out_lines_fast;
  int neighbours;  // lines next to each other in memory, whether a workgroup has several of them or one
  const double2 *tw;       // turns between the passes of length M (twiddle_kernel)
  const double2 *real_tw;  // packed lines: exp(-2 pi i k / 2n), k < n
  const double2 *chirp;  // Bluestein: exp(sign pi i j^2 / n), j < n
  const double2 *bf;     // Bluestein: forward transform (length M) of the wrapped conjugate chirp
  int64_t tw_total;      // four-step: multiply bin k of a line by exp(sign 2 pi i inner k / tw_total)
};

// Element i of a line lives at LDS index i + i / 16: one pad element per 16 turns
// the power-of-two strides of the exchanges into conflict-free ones.
__device__ __forceinline__ int pad(int i) { return i + (i >> 4); }

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(__builtin_fma(a.x, b.x, -(a.y * b.y)), __builtin_fma(a.x, b.y, a.y * b.x));
}

__device__ __forceinline__ double2 load_elem(const char *base, int kind, int64_t off) {
  switch (kind) {
    case K_C32: { const float2 v = *(const float2 *)(base + off * 8); return make_double2(v.x, v.y); }
    case K_C64: return *(const double2 *)(base + off * 16);
    case K_F32: return make_double2(*(const float *)(base + off * 4), 0.0);
    default: return make_double2(*(const double *)(base + off * 8), 0.0);
  }
}

__device__ __forceinline__ void store_elem(char *base, int kind, int64_t off, double2 v) {
  switch (kind) {
    case K_C32: *(float2 *)(base + off * 8) = make_float2((float)v.x, (float)v.y); break;
    case K_C64: *(double2 *)(base + off * 16) = v; break;
    case K_F32: *(float *)(base + off * 4) = (float)v.x; break;
    default: *(double *)(base + off * 8) = v.x; break;
  }
}

__device__ __forceinline__ int64_t line_offset(const Lines &v, int64_t l, int *inner) {
  int64_t off = 0;
  *inner = 0;
  for (int d = v.nd - 1; d >= 0; d--) {
    const int64_t next = d ? l / v.dims[d] : 0, c = l - next * (d ? v.dims[d] : 0);
    l = next;
    if (d == v.nd - 1) *inner = (int)c;
    off += c * v.strides[d];
  }
  return off;
}

// Element j (< n) of the sequence the transform sees, from the stored line.
__device__ __forceinline__ double2 fetch(const FftArgs &a, int64_t off, int j) {
  if (a.load_mode == LOAD_HERMITIAN) {  // nx_c_fft.c:1013-1023
    if (j < a.n_load) return load_elem(a.in.base, a.in.kind, off + j * a.in.estride);
    const int k = a.herm_s - j;
    if (k < a.n_load) {
      const double2 v = load_elem(a.in.base, a.in.kind, off + k * a.in.estride);
      return make_double2(v.x, -v.y);
    }
    return make_double2(0.0, 0.0);
  }
  if (j >= a.n_load) return make_double2(0.0, 0.0);
  return load_elem(a.in.base, a.in.kind, off + j * a.in.estride);
}

// ── the transform in registers ──────────────────────────────────────────────
// A line of M = 2^L elements belongs to T = M / E lanes that hold E elements each: slot e of
// lane t is element t + T e, before the transform, after it, and at the start of every pass (the
// self-sorting order: natural in, natural out). A pass does the butterflies of radix R <= E that
// a lane's own slots make up and then redistributes the line through LDS.
__host__ __device__ constexpr int log_elems(int L) { return L >= 8 ? 4 : L >= 6 ? 3 : L >= 4 ? 2 : L >= 1 ? 1 : 0; }

// v exp(-2 pi i k / 32), k < 32 known to the compiler
__device__ __forceinline__ double2 turn(double2 v, int k) {
  constexpr double c[9] = {1, 0.98078528040323043, 0.92387953251128674, 0.83146961230254524, 0.70710678118654757,
                           0.55557023301960218, 0.38268343236508978, 0.19509032201612825, 0};
  if (k & 16) v = make_double2(-v.x, -v.y);
  if (k & 8) v = make_double2(v.y, -v.x);
  k &= 7;
  return k ? cmul(v, make_double2(c[k], -c[8 - k])) : v;
}

// The forward DFT of length R over x[0], x[G], x[2 G], ... in natural order.
template <int R, int G, int N>
__device__ __forceinline__ void dft(double2 (&x)[N], int o) {
  if constexpr (R == 2) {
    const double2 u = x[o], v = x[o + G];
    x[o] = make_double2(u.x + v.x, u.y + v.y);
    x[o + G] = make_double2(u.x - v.x, u.y - v.y);
  } else if constexpr (R == 4) {
    const double2 a = x[o], b = x[o + G], c = x[o + 2 * G], d = x[o + 3 * G];
    const double2 s0 = make_double2(a.x + c.x, a.y + c.y), d0 = make_double2(a.x - c.x, a.y - c.y);
    const double2 s1 = make_double2(b.x + d.x, b.y + d.y), d1 = make_double2(b.x - d.x, b.y - d.y);
    x[o] = make_double2(s0.x + s1.x, s0.y + s1.y);
    x[o + 2 * G] = make_double2(s0.x - s1.x, s0.y - s1.y);
    x[o + G] = make_double2(d0.x + d1.y, d0.y - d1.x);
    x[o + 3 * G] = make_double2(d0.x - d1.y, d0.y + d1.x);
  } else {
    // R = P x 4: transforms of length 4 over every P-th element, twiddles, transforms of length P
    constexpr int P = R / 4;
    double2 y[R];
#pragma unroll
    for (int p = 0; p < P; p++) {
      double2 z[4];
#pragma unroll
      for (int b = 0; b < 4; b++) z[b] = x[o + (p + P * b) * G];
      dft<4, 1>(z, 0);
#pragma unroll
      for (int q = 0; q < 4; q++) {
        y[q * P + p] = turn(z[q], p * q * (32 / R));
      }
    }
#pragma unroll
    for (int q = 0; q < 4; q++) {
      double2 z[P];
#pragma unroll
      for (int p = 0; p < P; p++) z[p] = y[q * P + p];
      dft<P, 1>(z, 0);
#pragma unroll
      for (int p = 0; p < P; p++) x[o + (q + 4 * p) * G] = z[p];
    }
  }
}

// Slot e of every lane goes to place `to(e)` of its line, place t + T e comes back into slot e.
// Real and imaginary parts go one after the other through the same LDS: half the LDS per line,
// so twice the waves in flight (LDS is what limits them), for the same bytes moved.
template <int E, int T, class To>
__device__ __forceinline__ void exchange(double2 (&x)[E], double *line, const double *from, int t, To to) {
#pragma unroll
  for (int part = 0; part < 2; part++) {
    __syncthreads();  // what the LDS held before has been read
#pragma unroll
    for (int e = 0; e < E; e++) line[pad(to(e))] = part ? x[e].y : x[e].x;
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) (part ? x[e].y : x[e].x) = from[pad(t + T * e)];
  }
}

// The forward transform of the workgroup's lines, from sub-transforms of length 2^S on. `line` is
// the lane's own line in LDS. Element (jm, k) of a pass is turned by exp(-2 pi i k jm / 2^(S+r)), read
// from the table at (k << S) + jm: neighbouring lanes, neighbouring entries. (Products of the powers
// 1, 2, 4 and 8 are faster, complex64 [16, 512, 512] rows 20.8 us against 21.7, [4096, 4096] columns 119 against
// 126, rfft [8192, 2048] float32 43 against 44.5, but less exact, by 1 - 5 % in complex128; one table of roots for all powers, read at strides of
// k, kept the L1 busy for two thirds of the kernel's time.)
template <int L, int S>
__device__ __forceinline__ void fft_passes(double2 (&x)[1 << log_elems(L)], double *line, const double2 *tw, int t) {
  constexpr int E = 1 << log_elems(L), T = (1 << L) / E;
  constexpr int r = L - S < log_elems(L) ? L - S : log_elems(L), R = 1 << r, G = E / R;
  if constexpr (R > 1) {
    if constexpr (S > 0) {
      static_assert(G == 1 || S + r == L, "only the last pass has several butterflies a lane, T apart");
#pragma unroll
      for (int k = 1; k < R; k++)
#pragma unroll
        for (int g = 0; g < G; g++) x[g + k * G] = cmul(tw[(k << S) + ((t + g * T) & ((1 << S) - 1))], x[g + k * G]);
    }
#pragma unroll
    for (int g = 0; g < G; g++) dft<R, G>(x, g);
  }
  if constexpr (S + r < L) {
    exchange<E, T>(x, line, line, t, [&](int e) {
      const int j = t + (e % G) * T, k = e / G;
      return ((j >> S) << (S + r)) + (j & ((1 << S) - 1)) + (k << S);
    });
    fft_passes<L, S + r>(x, line, tw, t);
  }
}

// exp(-2 pi i k / 2n) for slot e of lane t (k = t + T e). Where n is the transform length itself
// the T e part is a constant.
template <int E, int T, bool BLUE>
__device__ __forceinline__ double2 real_twiddle(const FftArgs &a, int t, int e) {
  return BLUE ? a.real_tw[t + T * e < a.n ? t + T * e : 0] : turn(a.real_tw[t], e * (16 / E));
}

template <class V>
__device__ __forceinline__ double2 widen(V v) {
  if constexpr (std::is_same_v<V, float> || std::is_same_v<V, double>) return make_double2(v, 0.0);
  else return make_double2(v.x, v.y);
}

// The E elements t, t + T, ... of the line at `off`; what a line does not have reads as zero. All
// loads are issued, from addresses that every line has, before the first value is looked at: with
// the conversion to double beside each guarded load a wave waited for one load after the other
// (rfft [8192, 2048] float32: 76 us against 58).
template <int E, int T, bool BLUE>
__device__ __forceinline__ void load_line(const FftArgs &a, double2 (&x)[E], int64_t off, int t) {
  const int64_t es = a.in.estride;
  constexpr int USED = BLUE ? (E + 1) / 2 : E;  // the second half of a convolution's line is padding
#pragma unroll
  for (int e = 0; e < E; e++) x[e] = make_double2(0.0, 0.0);
  if (a.n_load < 1) return;
  // load(element number times `per`), for elements below `limit`
  const auto each = [&](int limit, int per, auto load) {
    decltype(load(off)) raw[USED];
    const int64_t at = off + (int64_t)t * per * es, step = (int64_t)T * per * es;
#pragma unroll
    for (int e = 0; e < USED; e++) raw[e] = load(t + T * e < limit ? at + e * step : off);
#pragma unroll
    for (int e = 0; e < USED; e++)
      if (t + T * e < limit) x[e] = widen(raw[e]);
  };
  const auto single = [&](auto p) { each(a.n_load < a.n ? a.n_load : a.n, 1, [=](int64_t at) { return p[at]; }); };
  if (a.pack == PACK_RFFT) {
    const float *pf = (const float *)a.in.base;
    const double *pd = (const double *)a.in.base;
    if (a.in.kind == K_F64) each(a.n, 2, [=](int64_t at) { return make_double2(pd[at], pd[at + es]); });
    else if (a.pair_aligned) each(a.n, 2, [=](int64_t at) { return *(const float2 *)(pf + at); });
    else each(a.n, 2, [=](int64_t at) { return make_float2(pf[at], pf[at + es]); });
  } else if (a.pack == PACK_IRFFT) {
    // The spectrum of the packed line, bins j and n - j at a time. The real part of the whole
    // transform never sees the imaginary parts of bins 0 and n (unless they are no numbers).
    const auto both = [&](auto p) {
      constexpr int HALF = (USED + 1) / 2;  // half at a time: twice the values are in registers here
#pragma unroll
      for (int e0 = 0; e0 < USED; e0 += HALF) {
        std::decay_t<decltype(p[0])> u[HALF], v[HALF];
#pragma unroll
        for (int e = e0; e < e0 + HALF && e < USED; e++) {
          const int j = t + T * e, k = a.n - j;
          u[e - e0] = p[off + (j < a.n_load ? j : 0) * es];
          v[e - e0] = p[off + (k >= 0 && k < a.n_load ? k : 0) * es];
        }
#pragma unroll
        for (int e = e0; e < e0 + HALF && e < USED; e++) {
          const int j = t + T * e, k = a.n - j;
          if (k <= 0) continue;
          double2 lo = j < a.n_load ? widen(u[e - e0]) : make_double2(0.0, 0.0);
          double2 hi = k < a.n_load ? widen(v[e - e0]) : make_double2(0.0, 0.0);
          if (j == 0) lo = make_double2(lo.x + 0.0 * lo.y, 0.0), hi = make_double2(hi.x + 0.0 * hi.y, 0.0);
          const double2 w = real_twiddle<E, T, BLUE>(a, t, e);
          const double2 odd = cmul(make_double2(lo.x - hi.x, lo.y + hi.y), make_double2(w.x, -w.y));
          x[e] = make_double2(lo.x + hi.x - odd.y, lo.y - hi.y + odd.x);
        }
      }
    };
    if (a.in.kind == K_C32) both((const float2 *)a.in.base);
    else both((const double2 *)a.in.base);
  } else if (a.load_mode == LOAD_HERMITIAN) {
#pragma unroll
    for (int e = 0; e < USED; e++)
      if (t + T * e < a.n) x[e] = fetch(a, off, t + T * e);
  } else {
    switch (a.in.kind) {
      case K_C32: single((const float2 *)a.in.base); break;
      case K_C64: single((const double2 *)a.in.base); break;
      case K_F32: single((const float *)a.in.base); break;
      default: single((const double *)a.in.base);
    }
  }
}

template <int E, int T, bool BLUE>
__device__ __forceinline__ void store_line(const FftArgs &a, const double2 (&x)[E], int64_t off, int t) {
  const int64_t es = a.out.estride;
  const auto each = [&](int per, auto store) {
    const int64_t at = off + (int64_t)t * per * es, step = (int64_t)T * per * es;
#pragma unroll
    for (int e = 0; e < E; e++)
      if ((!BLUE || e < (E + 1) / 2) && t + T * e < a.n_store) store(at + e * step, x[e]);
  };
  if (a.pack == PACK_IRFFT) {
    if (a.pair_aligned)
      each(2, [&](int64_t at, double2 v) { *(float2 *)(a.out.base + at * 4) = make_float2((float)v.x, (float)v.y); });
    else
      each(2, [&](int64_t at, double2 v) { float *p = (float *)a.out.base + at; p[0] = (float)v.x, p[es] = (float)v.y; });
    return;
  }
  switch (a.out.kind) {
    case K_C32: each(1, [&](int64_t at, double2 v) { store_elem(a.out.base, K_C32, at, v); }); break;
    case K_C64: each(1, [&](int64_t at, double2 v) { store_elem(a.out.base, K_C64, at, v); }); break;
    case K_F32: each(1, [&](int64_t at, double2 v) { store_elem(a.out.base, K_F32, at, v); }); break;
    default: each(1, [&](int64_t at, double2 v) { store_elem(a.out.base, K_F64, at, v); });
  }
}

// +sign transforms run as the forward one between two exchanges of real and imaginary parts.
__device__ __forceinline__ double2 flip(double2 v) { return make_double2(v.y, v.x); }

// One launch = one pass over the tensor: G lines a workgroup, read straight into registers,
// transformed, and stored from registers: besides the tensor's own traffic there are 32 bytes of
// LDS per element and exchange (two exchanges for M = 512 .. 4096). The form before went through
// LDS after the load, every four stages and before the store, and read a twiddle per butterfly.
// Measured: rfft [8192, 2048] float32 170 -> 52 us on new data, irfft back 158 -> 46 us
// (2.6 TB/s; three waves a SIMD by registers, and the waits of a wave's own chain bound it now).
// (The convolution of length 512 needs 170 registers when left alone, two more than three waves a SIMD have.)
template <int L, bool BLUE>
__global__ __launch_bounds__(512, BLUE && L == 9 ? 3 : 2) void fft_lines_kernel(FftArgs a) {
  extern __shared__ double lds[];
  constexpr int M = 1 << L, E = 1 << log_elems(L), T = M / E, PITCH = M + M / 16 + 1;
  // blocks that share an XCD (ids equal modulo 8) take neighbouring groups of lines: with
  // strided lines a 128-byte line of memory serves several workgroups, which then meet in one L2
  uint32_t bx = blockIdx.x;
  if (a.neighbours && (gridDim.x & 7u) == 0) bx = (bx & 7u) * (gridDim.x >> 3) + (bx >> 3);
  const int64_t first = (int64_t)bx * a.G;
  int g = threadIdx.x / T, t = threadIdx.x & (T - 1), unused;
  if (a.in_lines_fast) t = threadIdx.x / a.G, g = threadIdx.x - t * a.G;
  double2 x[E];
  // lanes beyond the last line work on it once more and store nothing
  const int64_t from_line = first + g < a.lines ? first + g : a.lines - 1;
  load_line<E, T, BLUE>(a, x, line_offset(a.in, a.line0 + from_line, &unused), t);
  if (BLUE) {
#pragma unroll
    for (int e = 0; e < (E + 1) / 2; e++) {
      const int j = t + T * e;
      if (j < a.n) x[e] = cmul(x[e], a.chirp[j]);
    }
  } else if (a.sign > 0) {
#pragma unroll
    for (int e = 0; e < E; e++) x[e] = flip(x[e]);
  }
  double *line = lds + g * PITCH;
  fft_passes<L, 0>(x, line, a.tw, t);
  if (BLUE) {
#pragma unroll
    for (int e = 0; e < E; e++) x[e] = flip(cmul(x[e], a.bf[t + T * e]));
    fft_passes<L, 0>(x, line, a.tw, t);
    const double inv_m = 1.0 / (double)M;
#pragma unroll
    for (int e = 0; e < (E + 1) / 2; e++) {
      const int j = t + T * e;
      x[e] = flip(x[e]);
      if (j < a.n) {
        const double2 c = a.chirp[j];
        x[e] = cmul(x[e], make_double2(c.x * inv_m, c.y * inv_m));
      }
    }
  } else if (a.sign > 0) {
#pragma unroll
    for (int e = 0; e < E; e++) x[e] = flip(x[e]);
  }
  if (a.pack == PACK_RFFT) {
    // bin k of the real line's transform from bins k and n - k of the packed one
    const double2 zero = x[0];
    double odd_im[E];
#pragma unroll
    for (int part = 0; part < 2; part++) {
      __syncthreads();
#pragma unroll
      for (int e = 0; e < E; e++) line[pad(t + T * e)] = part ? x[e].y : x[e].x;
      __syncthreads();
#pragma unroll
      for (int e = 0; e < E; e++) {
        const int k = t + T * e;
        const double m = line[pad(k && k < a.n ? a.n - k : 0)];
        if (part == 0) {
          odd_im[e] = 0.5 * (m - x[e].x);
          x[e].x = 0.5 * (x[e].x + m);
        } else if (k < a.n) {
          const double2 w = cmul(make_double2(0.5 * (x[e].y + m), odd_im[e]), real_twiddle<E, T, BLUE>(a, t, e));
          x[e] = make_double2(x[e].x + w.x, 0.5 * (x[e].y - m) + w.y);
        }
      }
    }
    if (t == 0 && first + g < a.lines) {  // bin n: the difference of the two halves' sums
      const int64_t off = line_offset(a.out, a.line0 + first + g, &unused);
      store_elem(a.out.base, a.out.kind, off + (int64_t)a.n * a.out.estride, make_double2(zero.x - zero.y, 0.0));
    }
  }
  if (a.in_lines_fast != a.out_lines_fast) {  // the store wants the other order of lanes
    const int from = t;
    g = threadIdx.x / T, t = threadIdx.x & (T - 1);
    if (a.out_lines_fast) t = threadIdx.x / a.G, g = threadIdx.x - t * a.G;
    exchange<E, T>(x, line, lds + g * PITCH, t, [&](int e) { return from + T * e; });
  }
  if (first + g >= a.lines) return;
  int inner;
  const int64_t off = line_offset(a.out, a.line0 + first + g, &inner);
  if (a.tw_total) {
#pragma unroll
    for (int e = 0; e < E; e++) {
      double sn, cs;
      sincospi(2.0 * (double)((int64_t)inner * (t + T * e)) / (double)a.tw_total, &sn, &cs);
      x[e] = cmul(x[e], make_double2(cs, a.sign > 0 ? sn : -sn));
    }
  }
  store_line<E, T, BLUE>(a, x, off, t);
}

// ── tables ──────────────────────────────────────────────────────────────────
// Of a transform of length 2^L: for each of its passes (sub-transforms of length 2^S become 2^(S+r) long),
// at (k << S) + j: exp(-2 pi i k j / 2^(S+r)), j < 2^S, 0 < k < 2^r. The first pass has none.
__global__ void twiddle_kernel(double2 *tw, int L) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= 1 << L) return;
  const int e = log_elems(L), S = e ? (31 - __clz(i | 1)) / e * e : 0, top = S + e < L ? S + e : L;
  const int turns = (i >> S) * (i & ((1 << S) - 1)) & ((1 << top) - 1);
  double sn, cs;
  sincospi(2.0 * (double)turns / (double)(1 << top), &sn, &cs);  // an exact argument
  tw[i] = make_double2(cs, -sn);
}

// exp(-2 pi i k / n), k < count
__global__ void real_twiddle_kernel(double2 *tw, int n, int count) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= count) return;
  double sn, cs;
  sincospi(2.0 * (double)k / (double)n, &sn, &cs);
  tw[k] = make_double2(cs, -sn);
}

// exp(sign pi i j^2 / n) with j^2 reduced mod 2n in integers (nx_c_fft.c:656-663).
__global__ void chirp_kernel(double2 *c, int64_t n, int sign) {
  const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n) return;
  const int64_t r = (j * j) % (2 * n);
  double sn, cs;
  sincospi((double)r / (double)n, &sn, &cs);
  c[j] = make_double2(cs, sign > 0 ? sn : -sn);
}

// The convolution filter conj(chirp[|d|]) wrapped to length M (nx_c_fft.c:665-710).
__global__ void chirp_filter_kernel(double2 *b, const double2 *chirp, int64_t n, int64_t M) {
  const int64_t d = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (d >= M) return;
  double2 v = make_double2(0.0, 0.0);
  if (d < n) v = chirp[d];
  else if (M - d < n) v = chirp[M - d];
  b[d] = make_double2(v.x, -v.y);
}

// ── workspace passes of the long transforms ─────────────────────────────────
struct StageArgs {
  Lines t;            // the tensor side
  double2 *w;         // workspace, [lines of this chunk][M]
  int64_t line0, lines;
  int64_t M, n, count;  // workspace line length; transform length; elements per line moved
  int n_load, load_mode, herm_s;
  const double2 *chirp;
  double scale;
};

__global__ __launch_bounds__(256) void stage_in_kernel(StageArgs s, FftArgs a) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= s.lines * s.M) return;
  const int64_t l = i / s.M, j = i - l * s.M;
  double2 v = make_double2(0.0, 0.0);
  if (j < s.n) {
    int unused;
    v = fetch(a, line_offset(s.t, s.line0 + l, &unused), (int)j);
    if (s.chirp) v = cmul(v, s.chirp[j]);
  }
  s.w[i] = v;
}

__global__ __launch_bounds__(256) void stage_out_kernel(StageArgs s) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= s.lines * s.count) return;
  const int64_t l = i / s.count, k = i - l * s.count;
  double2 v = s.w[l * s.M + k];
  if (s.chirp) {
    const double2 c = s.chirp[k];
    v = cmul(v, make_double2(c.x * s.scale, c.y * s.scale));
  }
  int unused;
  store_elem(s.t.base, s.t.kind, line_offset(s.t, s.line0 + l, &unused) + k * s.t.estride, v);
}

__global__ __launch_bounds__(256) void spectrum_mul_kernel(double2 *w, const double2 *bf, int64_t M, int64_t total) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  w[i] = cmul(w[i], bf[i % M]);
}

// ── host side ───────────────────────────────────────────────────────────────
static inline bool is_pow2(int64_t n) { return n > 0 && (n & (n - 1)) == 0; }
static inline int log2_of(int64_t n) {
  int l = 0;
  while ((int64_t(1) << l) < n) l++;
  return l;
}

// A transform too long for one workgroup is done as n1 x n2.
static inline int64_t four_step_n1(int64_t M) { return int64_t(1) << ((log2_of(M) + 1) / 2); }

enum TableKind : uint64_t { T_TWIDDLE = 1, T_CHIRP = 2, T_FILTER = 3, T_REAL = 4 };
static inline uint64_t table_key(TableKind k, int64_t n, int sign) {
  return ((uint64_t)k << 60) | ((uint64_t)(sign > 0) << 59) | (uint64_t)n;
}

static int table_lookup(nxh_context *ctx, uint64_t key, size_t bytes, double2 **out, bool *fresh) {
  auto it = ctx->device_tables.find(key);
  if (it != ctx->device_tables.end()) {
    *out = (double2 *)it->second;
    *fresh = false;
    return NXH_OK;
  }
  // A table is filled by a kernel on the context's stream. While that stream is being
  // recorded the fill would only be recorded too: the table would count as present with
  // nothing in it, for every eager transform until the first replay, and every replay
  // would rewrite a table that other work reads. So a length is never first used there.
  if (ctx->capture)
    return nxh_fail(NXH_FAILURE, "fft",
                    "first use of this transform length while a graph is being captured: run it once eagerly first");
  void *p = nullptr;
  if (hipMalloc(&p, bytes ? bytes : 16) != hipSuccess) {
    (void)hipGetLastError();
    return nxh_fail(NXH_FAILURE, "fft", NXH_ERR_ALLOC);
  }
  ctx->device_tables[key] = p;
  *out = (double2 *)p;
  *fresh = true;
  return NXH_OK;
}

// Takes a table whose fill could not be queued out of the registry again.
static void table_drop(nxh_context *ctx, uint64_t key) {
  auto it = ctx->device_tables.find(key);
  if (it == ctx->device_tables.end()) return;
  (void)hipStreamSynchronize(ctx->stream);  // a fill kernel already queued may still write it
  (void)hipFree(it->second);
  ctx->device_tables.erase(it);
}

// The table of transforms of length n: of their stages (T_TWIDDLE), or of packed real lines (T_REAL).
static int twiddles(nxh_context *ctx, TableKind kind, int n, const double2 **out) {
  double2 *t;
  bool fresh;
  const uint64_t key = table_key(kind, n, -1);
  const int count = kind == T_TWIDDLE ? n : n / 2;
  if (int rc = table_lookup(ctx, key, (size_t)count * sizeof(double2), &t, &fresh)) return rc;
  if (fresh) {
    const dim3 grid((count + 255) / 256), block(256);
    if (kind == T_TWIDDLE) hipLaunchKernelGGL(twiddle_kernel, grid, block, 0, ctx->stream, t, log2_of(n));
    else hipLaunchKernelGGL(real_twiddle_kernel, grid, block, 0, ctx->stream, t, n, count);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) {
      table_drop(ctx, key);
      return nxh_hip_fail("fft", e);
    }
  }
  *out = t;
  return NXH_OK;
}

static Lines workspace_lines(double2 *w, int64_t outer, int64_t outer_stride, int64_t innerdim, int64_t inner_stride,
                             int64_t estride) {
  Lines v{};
  v.base = (char *)w;
  v.kind = K_C64;
  v.nd = 2;
  v.dims[0] = outer;
  v.strides[0] = outer_stride;
  v.dims[1] = innerdim;
  v.strides[1] = inner_stride;
  v.estride = estride;
  return v;
}

using LinesKernel = void (*)(FftArgs);
template <bool BLUE, int... L>
static LinesKernel lines_kernel(int logM, std::integer_sequence<int, L...>) {
  static constexpr LinesKernel table[] = {fft_lines_kernel<L, BLUE>...};
  return table[logM];
}

static int launch_lines(nxh_context *ctx, FftArgs &a, bool blue) {
  // short lines share a wave; a longer line takes a workgroup of its own
  const int lanes = a.M >> log_elems(a.logM);
  a.G = lanes >= 64 ? 1 : 64 / lanes;
  // strided lines whose neighbours are adjacent in memory: as many lines per workgroup as make
  // runs of 128 bytes, or as the LDS holds
  auto neighbours = [](const Lines &v) { return v.estride != 1 && v.nd >= 1 && v.strides[v.nd - 1] == 1 && v.dims[v.nd - 1] > 1; };
  a.in_lines_fast = neighbours(a.in);
  a.out_lines_fast = neighbours(a.out);
  if (a.in_lines_fast || a.out_lines_fast) a.G = std::max(1, std::min(FFT_LDS_MAX / a.M, std::max(16, a.G)));
  if ((int64_t)a.G > a.lines) a.G = (int)a.lines;
  a.neighbours = a.in_lines_fast || a.out_lines_fast;
  if (a.G == 1) a.in_lines_fast = a.out_lines_fast = 0;
  const int64_t blocks = (a.lines + a.G - 1) / a.G;
  if (blocks > 0x7fffffffLL) return nxh_fail(NXH_FAILURE, "fft", "too many lines for one launch");
  const size_t lds = (size_t)a.G * (a.M + a.M / 16 + 1) * sizeof(double);
  constexpr auto lengths = std::make_integer_sequence<int, FFT_LOG_MAX + 1>{};
  const auto kern = blue ? lines_kernel<true>(a.logM, lengths) : lines_kernel<false>(a.logM, lengths);
  static std::once_flag once[2][FFT_LOG_MAX + 1];
  static hipError_t attr_status[2][FFT_LOG_MAX + 1];
  std::call_once(once[blue][a.logM], [&] {
    attr_status[blue][a.logM] = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                    (int)((FFT_LDS_MAX + FFT_LDS_MAX / 16) * sizeof(double) + 4096));
  });
  NXH_HIP("fft", attr_status[blue][a.logM]);
  hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(a.G * lanes), lds, ctx->stream, a);
  NXH_HIP("fft", hipGetLastError());
  return NXH_OK;
}

// Power-of-two transform of `lines` contiguous complex128 lines of length M in
// the workspace `src`; the result lands in `dst` (src is overwritten).
static int pow2_workspace(nxh_context *ctx, double2 *src, double2 *dst, int64_t lines, int64_t M, int sign) {
  FftArgs a{};
  a.sign = sign;
  a.load_mode = LOAD_COMPLEX;
  if (M <= FFT_LDS_MAX) {
    a.in = workspace_lines(src, lines, M, 1, 0, 1);
    a.out = workspace_lines(dst, lines, M, 1, 0, 1);
    a.lines = lines;
    a.n = a.M = a.n_load = a.n_store = (int)M;
    a.logM = log2_of(M);
    if (int rc = twiddles(ctx, T_TWIDDLE, a.M, &a.tw)) return rc;
    return launch_lines(ctx, a, false);
  }
  const int64_t n1 = four_step_n1(M), n2 = M / n1;
  if (n1 > FFT_LDS_MAX) return nxh_fail(NXH_FAILURE, "fft", "axis too long (the limit is 2^26 elements)");
  // x[j1 n2 + j2] -> X[k1 + n1 k2]: transforms of length n1 down the columns, a
  // twiddle exp(sign 2 pi i j2 k1 / M), transforms of length n2 along the rows
  a.in = a.out = workspace_lines(src, lines, M, n2, 1, n2);
  a.lines = lines * n2;
  a.n = a.M = a.n_load = a.n_store = (int)n1;
  a.logM = log2_of(n1);
  a.tw_total = M;
  if (int rc = twiddles(ctx, T_TWIDDLE, a.M, &a.tw)) return rc;
  if (int rc = launch_lines(ctx, a, false)) return rc;
  a.in = workspace_lines(src, lines, M, n1, n2, 1);
  a.out = workspace_lines(dst, lines, M, n1, 1, n1);
  a.lines = lines * n1;
  a.n = a.M = a.n_load = a.n_store = (int)n2;
  a.logM = log2_of(n2);
  a.tw_total = 0;
  if (int rc = twiddles(ctx, T_TWIDDLE, a.M, &a.tw)) return rc;
  return launch_lines(ctx, a, false);
}

struct Scratch {  // pool blocks released when the pass is done (stream-ordered reuse)
  nxh_context *ctx;
  void *p[2] = {nullptr, nullptr};
  ~Scratch() {
    for (void *q : p)
      if (q) nxh_free_locked(ctx, q);
  }
};

static int bluestein_tables(nxh_context *ctx, int64_t n, int64_t M, int sign, const double2 **chirp, const double2 **bf) {
  double2 *c, *f;
  bool fresh_c, fresh_f;
  if (int rc = table_lookup(ctx, table_key(T_CHIRP, n, sign), (size_t)n * sizeof(double2), &c, &fresh_c)) return rc;
  if (fresh_c) {
    hipLaunchKernelGGL(chirp_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream, c, n, sign);
    if (hipError_t e = hipGetLastError(); e != hipSuccess) {
      table_drop(ctx, table_key(T_CHIRP, n, sign));
      return nxh_hip_fail("fft", e);
    }
  }
  if (int rc = table_lookup(ctx, table_key(T_FILTER, n, sign), (size_t)M * sizeof(double2), &f, &fresh_f)) return rc;
  if (fresh_f) {
    // the filter counts as present only once every launch that fills it has been queued
    Scratch tmp{ctx};
    int rc = nxh_alloc_locked(ctx, (size_t)M * sizeof(double2), &tmp.p[0]);
    if (!rc) {
      hipLaunchKernelGGL(chirp_filter_kernel, dim3((unsigned)((M + 255) / 256)), dim3(256), 0, ctx->stream,
                         (double2 *)tmp.p[0], c, n, M);
      if (hipError_t e = hipGetLastError(); e != hipSuccess) rc = nxh_hip_fail("fft", e);
    }
    if (!rc) rc = pow2_workspace(ctx, (double2 *)tmp.p[0], f, 1, M, -1);
    if (rc) {
      table_drop(ctx, table_key(T_FILTER, n, sign));
      return rc;
    }
  }
  *chirp = c;
  *bf = f;
  return NXH_OK;
}

// Whether the tables of transforms of length n (convolved at length M) exist already.
static bool tables_present(nxh_context *ctx, int64_t n, int64_t M, int sign) {
  const auto have = [&](TableKind kind, int64_t len, int s) { return ctx->device_tables.count(table_key(kind, len, s)) != 0; };
  const bool stages = M <= FFT_LDS_MAX ? have(T_TWIDDLE, M, -1)
                                       : have(T_TWIDDLE, four_step_n1(M), -1) && have(T_TWIDDLE, M / four_step_n1(M), -1);
  return stages && (n == M || (have(T_CHIRP, n, sign) && have(T_FILTER, n, sign)));
}

static int line_tables(nxh_context *ctx, int64_t n, int64_t M, int sign) {
  if (tables_present(ctx, n, M, sign)) return NXH_OK;
  const double2 *unused, *unused2;
  const int64_t n1 = M <= FFT_LDS_MAX ? M : four_step_n1(M);
  if (n1 > FFT_LDS_MAX) return NXH_OK;  // a length that the general path refuses
  if (int rc = twiddles(ctx, T_TWIDDLE, (int)n1, &unused)) return rc;
  if (n1 < M)
    if (int rc = twiddles(ctx, T_TWIDDLE, (int)(M / n1), &unused)) return rc;
  return n == M ? NXH_OK : bluestein_tables(ctx, n, M, sign, &unused, &unused2);
}

// One axis pass: every line of `in` (n_load stored elements, read per
// `load_mode`) is transformed at length n and its first n_store bins are stored
// to `out` (their real parts when `out` is real). `in` and `out` may be the same tensor.
static int transform_lines(nxh_context *ctx, const Lines &in, const Lines &out, int64_t lines, int64_t n, int n_load,
                           int load_mode, int64_t n_store, int sign) {
  if (lines == 0 || n == 0 || n_store == 0) return NXH_OK;
  if (n > (int64_t(1) << 26)) return nxh_fail(NXH_FAILURE, "fft", "axis too long (the limit is 2^26 elements)");
  // real lines of an even length, one side real and the other the half spectrum, go packed (where exact enough)
  const int pack = n % 2 ? PACK_NONE
                   : load_mode == LOAD_REAL && (in.kind == K_F32 || n >= 512) && n_load == n && n_store == n / 2 + 1 ? PACK_RFFT
                   : load_mode == LOAD_HERMITIAN && out.kind == K_F32 && n_store == n && n_load <= n / 2 + 1 ? PACK_IRFFT
                                                                                                          : PACK_NONE;
  const auto conv_length = [](int64_t len) { return is_pow2(len) ? len : int64_t(1) << log2_of(2 * len - 1); };
  FftArgs a{};
  a.in = in;
  a.out = out;
  a.n_load = n_load;
  a.load_mode = load_mode;
  a.herm_s = (int)n;
  a.n_store = (int)n_store;
  a.sign = sign;
  const bool have_tables = !ctx->capture || (tables_present(ctx, n / 2, conv_length(n / 2), sign) &&
                                             ctx->device_tables.count(table_key(T_REAL, n, -1)));
  if (pack != PACK_NONE && conv_length(n / 2) <= FFT_LDS_MAX && have_tables) {
    a.pack = pack;
    // A length counts as used, for every transform that a graph may record later, once any of
    // its transforms has run: the tables of the line itself are made here too.
    if (!ctx->capture)
      if (int rc = line_tables(ctx, n, conv_length(n), sign)) return rc;
    if (int rc = twiddles(ctx, T_REAL, (int)n, &a.real_tw)) return rc;
    n /= 2;
    a.n_store = (int)n;
    const Lines &real = pack == PACK_RFFT ? in : out;
    a.pair_aligned = real.kind == K_F32 && real.estride == 1 && (uintptr_t)real.base % sizeof(float2) == 0;
    for (int d = 0; d < real.nd; d++) a.pair_aligned &= real.strides[d] % 2 == 0;
  }
  a.n = (int)n;
  const bool blue = !is_pow2(n);
  const int64_t M = conv_length(n);
  if (M > (int64_t(1) << 26)) return nxh_fail(NXH_FAILURE, "fft", "axis too long for a length that is not a power of two (the limit is 2^25 elements)");
  if (blue)
    if (int rc = bluestein_tables(ctx, n, M, sign, &a.chirp, &a.bf)) return rc;
  if (M <= FFT_LDS_MAX) {
    a.lines = lines;
    a.M = (int)M;
    a.logM = log2_of(M);
    if (int rc = twiddles(ctx, T_TWIDDLE, a.M, &a.tw)) return rc;
    return launch_lines(ctx, a, blue);
  }
  // long transform: chunks of lines through two workspaces
  const int64_t chunk = std::max<int64_t>(1, std::min(lines, FFT_WORK_ELEMS / M));
  Scratch ws{ctx};
  for (void *&p : ws.p)
    if (int rc = nxh_alloc_locked(ctx, (size_t)(chunk * M) * sizeof(double2), &p)) return rc;
  double2 *w0 = (double2 *)ws.p[0], *w1 = (double2 *)ws.p[1];
  for (int64_t l0 = 0; l0 < lines; l0 += chunk) {
    const int64_t nl = std::min(chunk, lines - l0);
    StageArgs s{};
    s.w = w0;
    s.line0 = l0;
    s.lines = nl;
    s.M = M;
    s.n = n;
    s.chirp = blue ? a.chirp : nullptr;
    s.t = in;
    const int64_t total = nl * M;
    if ((total + 255) / 256 > 0x7fffffffLL) return nxh_fail(NXH_FAILURE, "fft", "too many elements for one launch");
    hipLaunchKernelGGL(stage_in_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream, s, a);
    double2 *res = w1;
    if (int rc = pow2_workspace(ctx, w0, w1, nl, M, blue ? -1 : sign)) return rc;
    if (blue) {
      hipLaunchKernelGGL(spectrum_mul_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream, w1, a.bf, M, total);
      if (int rc = pow2_workspace(ctx, w1, w0, nl, M, +1)) return rc;
      res = w0;
    }
    s.w = res;
    s.t = out;
    s.count = n_store;
    s.scale = 1.0 / (double)M;
    const int64_t stores = nl * n_store;
    hipLaunchKernelGGL(stage_out_kernel, dim3((unsigned)((stores + 255) / 256)), dim3(256), 0, ctx->stream, s);
    NXH_HIP("fft", hipGetLastError());
  }
  return NXH_OK;
}

static int complex_kind(int dtype) { return dtype == NXH_C32 ? K_C32 : dtype == NXH_C64 ? K_C64 : -1; }
static int real_kind(int dtype) { return dtype == NXH_F32 ? K_F32 : dtype == NXH_F64 ? K_F64 : -1; }

// The lines of `src` and `dst` along `axis` (axis < 0: every element is a line
// of length one), with the other dims merged where both tensors allow it.
static int make_lines(const char *op, const nxh_tensor *src, int src_kind, const nxh_tensor *dst, int dst_kind, int axis,
                      Lines *in, Lines *out, int64_t *lines) {
  *in = Lines{};
  *out = Lines{};
  in->base = (char *)src->data + src->offset * kind_size(src_kind);
  out->base = (char *)dst->data + dst->offset * kind_size(dst_kind);
  in->kind = src_kind;
  out->kind = dst_kind;
  in->estride = axis >= 0 ? src->strides[axis] : 0;
  out->estride = axis >= 0 ? dst->strides[axis] : 0;
  int nd = 0;
  *lines = 1;
  for (int d = 0; d < dst->ndim; d++) {
    if (d == axis || dst->shape[d] == 1) continue;
    const int64_t e = dst->shape[d];
    *lines *= e;
    if (nd > 0 && in->strides[nd - 1] == src->strides[d] * e && out->strides[nd - 1] == dst->strides[d] * e) {
      in->dims[nd - 1] *= e;
      out->dims[nd - 1] *= e;
      in->strides[nd - 1] = src->strides[d];
      out->strides[nd - 1] = dst->strides[d];
      continue;
    }
    if (nd == FFT_MAXD) return nxh_fail(NXH_FAILURE, op, "too many non-mergeable dims beside the transformed axis (the limit is 8)");
    in->dims[nd] = out->dims[nd] = e;
    in->strides[nd] = src->strides[d];
    out->strides[nd] = dst->strides[d];
    nd++;
  }
  in->nd = out->nd = nd;
  return NXH_OK;
}

static int check_axes(const char *op, const int32_t *axes, int n_axes, int ndim) {
  if (n_axes < 0 || (n_axes > 0 && !axes)) return nxh_fail(NXH_INVALID_ARGUMENT, op, "null argument");
  for (int i = 0; i < n_axes; i++)
    if (axes[i] < 0 || axes[i] >= ndim) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_AXIS);
  return NXH_OK;
}

static int check_out(const char *op, const nxh_tensor *out) {
  for (int d = 0; d < out->ndim; d++)
    if (out->shape[d] > 1 && out->strides[d] == 0) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_OUT_ALIASED);
  return NXH_OK;
}

static inline int length_as_int(const char *op, int64_t n) {
  return n > (int64_t(1) << 26) ? nxh_fail(NXH_FAILURE, op, "axis too long (the limit is 2^26 elements)") : NXH_OK;
}

}  // namespace

// nx_c_fft.c:940-956
NXH_EXPORT int nxh_fft(nxh_context *ctx, const nxh_tensor *out, const nxh_tensor *x, const int32_t *axes, int n_axes,
                       int inverse) {
  NXH_DEFER_BARRIER(ctx, out);
  const char *op = inverse ? "ifft" : "fft";
  if (!ctx || !out || !x) return nxh_fail(NXH_INVALID_ARGUMENT, op, "null argument");
  int rc = nxh_check_tensor(op, out);
  if (!rc) rc = nxh_check_tensor(op, x);
  if (!rc) rc = check_axes(op, axes, n_axes, x->ndim);
  if (!rc) rc = check_out(op, out);
  if (rc) return rc;
  const int kind = complex_kind(out->dtype);
  if (kind < 0 || x->dtype != out->dtype) return nxh_fail(NXH_FAILURE, op, NXH_ERR_UNSUPPORTED);
  if (!nxh_same_shape(out, x)) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_SHAPE);
  std::lock_guard<std::mutex> guard(ctx->mu);
  NXH_HIP(op, hipSetDevice(ctx->device));
  nxh_set_path("fft_lines");
  const int passes = n_axes > 0 ? n_axes : 1;  // no axes: the transform over nothing, a copy
  for (int ai = 0; ai < passes; ai++) {
    const int axis = n_axes > 0 ? axes[ai] : -1;
    const nxh_tensor *src = ai == 0 ? x : out;
    const int64_t n = axis >= 0 ? out->shape[axis] : 1;
    if ((rc = length_as_int(op, n))) return rc;
    Lines in, o;
    int64_t lines;
    if ((rc = make_lines(op, src, kind, out, kind, axis, &in, &o, &lines))) return rc;
    if ((rc = transform_lines(ctx, in, o, lines, n, (int)n, LOAD_COMPLEX, n, inverse ? +1 : -1))) return rc;
  }
  return NXH_OK;
}

// nx_c_fft.c:958-982
NXH_EXPORT int nxh_rfft(nxh_context *ctx, const nxh_tensor *out, const nxh_tensor *x, const int32_t *axes, int n_axes) {
  NXH_DEFER_BARRIER(ctx, out);
  const char *op = "rfft";
  if (!ctx || !out || !x) return nxh_fail(NXH_INVALID_ARGUMENT, op, "null argument");
  int rc = nxh_check_tensor(op, out);
  if (!rc) rc = nxh_check_tensor(op, x);
  if (!rc) rc = check_axes(op, axes, n_axes, x->ndim);
  if (!rc) rc = check_out(op, out);
  if (rc) return rc;
  if (n_axes < 1) return nxh_fail(NXH_INVALID_ARGUMENT, op, "no axis to transform");
  const int ok = complex_kind(out->dtype), ik = real_kind(x->dtype);
  if (ok < 0 || ik < 0) return nxh_fail(NXH_FAILURE, op, NXH_ERR_UNSUPPORTED);
  const int last = axes[n_axes - 1];
  if (out->ndim != x->ndim) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_SHAPE);
  const int64_t n = x->shape[last], half = n / 2 + 1;
  for (int d = 0; d < x->ndim; d++)
    if (out->shape[d] != (d == last ? half : x->shape[d])) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_SHAPE);
  if ((rc = length_as_int(op, n))) return rc;
  std::lock_guard<std::mutex> guard(ctx->mu);
  NXH_HIP(op, hipSetDevice(ctx->device));
  nxh_set_path("fft_lines");
  Lines in, o;
  int64_t lines;
  if ((rc = make_lines(op, x, ik, out, ok, last, &in, &o, &lines))) return rc;
  if ((rc = transform_lines(ctx, in, o, lines, n, (int)n, LOAD_REAL, half, -1))) return rc;
  for (int ai = 0; ai < n_axes - 1; ai++) {
    const int axis = axes[ai];
    const int64_t m = out->shape[axis];
    if ((rc = length_as_int(op, m))) return rc;
    if ((rc = make_lines(op, out, ok, out, ok, axis, &in, &o, &lines))) return rc;
    if ((rc = transform_lines(ctx, in, o, lines, m, (int)m, LOAD_COMPLEX, m, -1))) return rc;
  }
  return NXH_OK;
}

// nx_c_fft.c:1029-1144
NXH_EXPORT int nxh_irfft(nxh_context *ctx, const nxh_tensor *out, const nxh_tensor *x, const int32_t *axes, int n_axes,
                         int64_t s_last) {
  NXH_DEFER_BARRIER(ctx, out);
  const char *op = "irfft";
  if (!ctx || !out || !x) return nxh_fail(NXH_INVALID_ARGUMENT, op, "null argument");
  int rc = nxh_check_tensor(op, out);
  if (!rc) rc = nxh_check_tensor(op, x);
  if (!rc) rc = check_axes(op, axes, n_axes, x->ndim);
  if (!rc) rc = check_out(op, out);
  if (rc) return rc;
  if (n_axes < 1) return nxh_fail(NXH_INVALID_ARGUMENT, op, "no axis to transform");
  const int ik = complex_kind(x->dtype), ok = real_kind(out->dtype);
  if (ok < 0 || ik < 0) return nxh_fail(NXH_FAILURE, op, NXH_ERR_UNSUPPORTED);
  const int last = axes[n_axes - 1];
  if (out->ndim != x->ndim) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_SHAPE);
  const int64_t in_half = x->shape[last];
  const int64_t s = s_last > 0 ? s_last : 2 * (in_half - 1);
  for (int d = 0; d < x->ndim; d++)
    if (out->shape[d] != (d == last ? s : x->shape[d])) return nxh_fail(NXH_INVALID_ARGUMENT, op, NXH_ERR_SHAPE);
  if ((rc = length_as_int(op, s))) return rc;
  const int64_t half = std::min(in_half, s / 2 + 1);
  std::lock_guard<std::mutex> guard(ctx->mu);
  NXH_HIP(op, hipSetDevice(ctx->device));
  nxh_set_path("fft_lines");
  // the other axes first, in a contiguous complex128 temporary of x's shape
  nxh_tensor tmp = *x;
  Scratch hold{ctx};
  const nxh_tensor *src = x;
  int src_kind = ik;
  if (n_axes > 1) {
    int64_t count = 1;
    for (int d = x->ndim - 1; d >= 0; d--) {
      tmp.strides[d] = count;
      count *= x->shape[d];
    }
    if (count == 0 || s == 0) return NXH_OK;
    if ((rc = nxh_alloc_locked(ctx, (size_t)count * sizeof(double2), &hold.p[0]))) return rc;
    tmp.data = hold.p[0];
    tmp.offset = 0;
    tmp.dtype = NXH_C64;
    for (int ai = 0; ai < n_axes - 1; ai++) {
      const int axis = axes[ai];
      const int64_t m = x->shape[axis];
      if ((rc = length_as_int(op, m))) return rc;
      Lines in, o;
      int64_t lines;
      if ((rc = make_lines(op, src, src_kind, &tmp, K_C64, axis, &in, &o, &lines))) return rc;
      if ((rc = transform_lines(ctx, in, o, lines, m, (int)m, LOAD_COMPLEX, m, +1))) return rc;
      src = &tmp;
      src_kind = K_C64;
    }
  }
  Lines in, o;
  int64_t lines;
  // lines are counted over the output's other dims, which equal the input's
  if ((rc = make_lines(op, src, src_kind, out, ok, last, &in, &o, &lines))) return rc;
  return transform_lines(ctx, in, o, lines, s, (int)half, LOAD_HERMITIAN, s, +1);
}
