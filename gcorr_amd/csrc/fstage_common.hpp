// Device helpers shared by the F-stage kernels: fstage16.hpp (16 points per
// thread, L = 64..1024), fstage_1k.hpp (a wave per FFT pair, 1024 real points),
// fstage_big.hpp (32 points per thread, L = 2048..32768) and fstage_mfma.hip
// (all passes on the matrix cores).
#pragma once

#include "gxc_internal.hpp"

namespace gxc {
namespace fs {

__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 mnegi(float2 a) { return make_float2(a.y, -a.x); }  // -i*a

// Compile-time cos/sin for twiddle constants (Taylor series in double,
// |x| <= 2 pi, 40 terms: accurate far below FP32 resolution).
constexpr double cx_sin(double x) {
  double term = x, sum = x;
  for (int n = 1; n < 40; n++) {
    term *= -x * x / ((2.0 * n) * (2.0 * n + 1.0));
    sum += term;
  }
  return sum;
}
constexpr double cx_cos(double x) {
  double term = 1.0, sum = 1.0;
  for (int n = 1; n < 40; n++) {
    term *= -x * x / ((2.0 * n - 1.0) * (2.0 * n));
    sum += term;
  }
  return sum;
}

// Multiply by the compile-time twiddle W_N^K = exp(-2 pi i K / N).  Multiples
// of pi/4 use exact forms; other angles use FP32-rounded constants.
template <int N, int K>
__device__ __forceinline__ float2 twc(float2 a) {
  constexpr int k = K % N;
  constexpr float c = 0.70710678118654752f;
  if constexpr (k == 0) {
    return a;
  } else if constexpr (4 * k == N) {
    return mnegi(a);
  } else if constexpr (2 * k == N) {
    return make_float2(-a.x, -a.y);
  } else if constexpr (4 * k == 3 * N) {
    return make_float2(-a.y, a.x);
  } else if constexpr (8 * k == N) {
    return make_float2((a.x + a.y) * c, (a.y - a.x) * c);
  } else if constexpr (8 * k == 3 * N) {
    return make_float2((a.y - a.x) * c, -(a.x + a.y) * c);
  } else if constexpr (8 * k == 5 * N) {
    return make_float2(-(a.x + a.y) * c, (a.x - a.y) * c);
  } else if constexpr (8 * k == 7 * N) {
    return make_float2((a.x - a.y) * c, (a.x + a.y) * c);
  } else {
    constexpr double ang = 2.0 * kPi * (double)k / (double)N;
    constexpr float wr = (float)cx_cos(ang), wi = (float)-cx_sin(ang);
    return make_float2(a.x * wr - a.y * wi, a.x * wi + a.y * wr);
  }
}

// plus = a + W_N^K b, minus = a - W_N^K b for a compile-time twiddle.
// Off the multiples of N/4 the twiddle is factored as W = c (1 + i t) with
// |t| <= 1 (|cos| >= |sin|) or W = s (t + i): b' = (1 + i t) b (or (t + i) b)
// takes 2 FMAs and a +- c b' 4 more, 6 instructions where a complex product
// and two complex additions take 8 (the fused multiply-add form of
// Linzer and Feig, 1993).
template <int N, int K>
__device__ __forceinline__ void bfly_tw(float2 a, float2 b, float2 &plus, float2 &minus) {
  constexpr int k = K % N;
  if constexpr (k == 0) {
    plus = cadd(a, b);
    minus = csub(a, b);
  } else if constexpr (4 * k == N || 2 * k == N || 4 * k == 3 * N) {
    const float2 w = twc<N, K>(b);
    plus = cadd(a, w);
    minus = csub(a, w);
  } else {
    constexpr double ang = 2.0 * kPi * (double)k / (double)N;
    constexpr double wr = cx_cos(ang), wi = -cx_sin(ang);
    constexpr bool cosform = (wr < 0 ? -wr : wr) >= (wi < 0 ? -wi : wi);
    constexpr float c = (float)(cosform ? wr : wi);
    constexpr float t = (float)(cosform ? wi / wr : wr / wi);
    const float2 bp = cosform ? make_float2(b.x - t * b.y, b.y + t * b.x)
                              : make_float2(t * b.x - b.y, t * b.y + b.x);
    plus = make_float2(a.x + c * bp.x, a.y + c * bp.y);
    minus = make_float2(a.x - c * bp.x, a.y - c * bp.y);
  }
}

__device__ __forceinline__ void dft4(float2 &a0, float2 &a1, float2 &a2, float2 &a3) {
  const float2 t0 = cadd(a0, a2), t1 = csub(a0, a2);
  const float2 t2 = cadd(a1, a3), t3 = mnegi(csub(a1, a3));
  a0 = cadd(t0, t2);
  a2 = csub(t0, t2);
  a1 = cadd(t1, t3);
  a3 = csub(t1, t3);
}

// v[q] = e[q] + W32^q o[q], v[q + 16] = e[q] - W32^q o[q] for q = Q .. 15
template <int Q>
__device__ __forceinline__ void bfly32(const float2 *e, const float2 *o, float2 *v) {
  if constexpr (Q < 16) {
    bfly_tw<32, Q>(e[Q], o[Q], v[Q], v[Q + 16]);
    bfly32<Q + 1>(e, o, v);
  }
}

// In-place forward DFT of R points v[0..R), natural order in and out.
template <int R>
__device__ __forceinline__ void dft(float2 *v) {
  if constexpr (R == 1) {
  } else if constexpr (R == 2) {
    const float2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    dft4(v[0], v[1], v[2], v[3]);
  } else if constexpr (R == 8) {
    // k = k1 + 2 k2: DFT4 over k2, twiddle W8^(k1 q2), DFT2 over k1.
    dft4(v[0], v[2], v[4], v[6]);
    dft4(v[1], v[3], v[5], v[7]);
    const float2 y00 = v[0], y01 = v[2], y02 = v[4], y03 = v[6];
    const float2 y10 = v[1], y11 = v[3], y12 = v[5], y13 = v[7];
    bfly_tw<8, 0>(y00, y10, v[0], v[4]);
    bfly_tw<8, 1>(y01, y11, v[1], v[5]);
    bfly_tw<8, 2>(y02, y12, v[2], v[6]);
    bfly_tw<8, 3>(y03, y13, v[3], v[7]);
  } else if constexpr (R == 16) {
    // k = k1 + 4 k2, q = 4 q1 + q2: DFT4 over k2, twiddle W16^(k1 q2), DFT4 over k1.
    dft4(v[0], v[4], v[8], v[12]);
    dft4(v[1], v[5], v[9], v[13]);
    dft4(v[2], v[6], v[10], v[14]);
    dft4(v[3], v[7], v[11], v[15]);
    // y[k1][q2] = W16^(k1 q2) v[k1 + 4 q2]; k1 = 2 enters its DFT4 as
    // y0 +- W16^(2 q2) v, one twiddled butterfly (bfly_tw)
    float2 y[4][4];
#pragma unroll
    for (int q2 = 0; q2 < 4; q2++) {
      y[0][q2] = v[4 * q2];
      y[2][q2] = v[2 + 4 * q2];
    }
    y[1][0] = v[1]; y[1][1] = twc<16, 1>(v[5]); y[1][2] = twc<16, 2>(v[9]);  y[1][3] = twc<16, 3>(v[13]);
    y[3][0] = v[3]; y[3][1] = twc<16, 3>(v[7]); y[3][2] = twc<16, 6>(v[11]); y[3][3] = twc<16, 9>(v[15]);
    float2 t0[4], t1[4];
    bfly_tw<16, 0>(y[0][0], y[2][0], t0[0], t1[0]);
    bfly_tw<16, 2>(y[0][1], y[2][1], t0[1], t1[1]);
    bfly_tw<16, 4>(y[0][2], y[2][2], t0[2], t1[2]);
    bfly_tw<16, 6>(y[0][3], y[2][3], t0[3], t1[3]);
#pragma unroll
    for (int q2 = 0; q2 < 4; q2++) {
      const float2 t2 = cadd(y[1][q2], y[3][q2]), t3 = mnegi(csub(y[1][q2], y[3][q2]));
      v[q2] = cadd(t0[q2], t2);
      v[8 + q2] = csub(t0[q2], t2);
      v[4 + q2] = cadd(t1[q2], t3);
      v[12 + q2] = csub(t1[q2], t3);
    }
  } else if constexpr (R == 32) {
    // Even/odd split: X[q] = E[q] + W32^q O[q], X[q+16] = E[q] - W32^q O[q].
    float2 e[16], o[16];
#pragma unroll
    for (int m = 0; m < 16; m++) {
      e[m] = v[2 * m];
      o[m] = v[2 * m + 1];
    }
    dft<16>(e);
    dft<16>(o);
    bfly32<0>(e, o, v);
  }
}

// Sizes of the per-item rotator tables for FFT length L (fxkernel.cpp:96-114):
// sub and step fringe-rotator factors, then sub and step fractional-sample
// factors.
template <int L, bool CPLX>
struct TabGeom {
  static constexpr int NCHAN = CPLX ? L : L / 2;
  static constexpr int S = 1 << (ilog2c(NCHAN) / 2);
  static constexpr int S2 = CPLX ? S : 2 * S;
  static constexpr int NSTEPS = L / S2;
  static constexpr int FRACSTEPS = NCHAN / S;
  static constexpr int NTAB = S2 + NSTEPS + S + FRACSTEPS;
};

// FP64 delay model and integer/fractional split for station st, FFT t:
// fxkernel.cpp:425-440 (getStationDelay) and 288-309, one rounding per
// operation (no contraction), so offsets and validity match the CPU exactly.
template <int L>
__device__ __forceinline__ bool split_offset(const FParams &p, int st, int t, int &offset,
                                             double &frac, double &a, double &b) {
#pragma clang fp contract(off)
  const double *dp = p.delays + 4 * st;
  const double c0 = dp[0], c1 = dp[1], c2 = dp[2], fileoffset = dp[3];
  const double t0 = (double)t, th = t + 0.5, t1 = t + 1.0;
  const double d0 = c0 * t0 * t0 + c1 * t0 + c2;
  const double d1 = c0 * th * th + c1 * th + c2;
  const double d2 = c0 * t1 * t1 + c1 * t1 + c2;
  a = d2 - d0;
  b = d0 + (d1 - (a * 0.5 + d0)) / 3.0;
  const double mean = a * 0.5 + b;
  const double ndf = (mean - fileoffset) / p.sampletime;
  if (!(fabs(ndf) < 1.0e9)) {
    offset = 0;
    frac = 0.0;
    return false;
  }
  const int nd = (int)(ndf + 0.5);  // truncation toward zero, fxkernel.cpp:290
  frac = -(ndf - nd) * p.sampletime;
  long long off = (long long)t * L - nd;
  if (off == -1) {
    ++off;
    frac += p.sampletime;
  }
  if (off == (long long)p.maxoffset + 1) {
    --off;
    frac -= p.sampletime;
  }
  offset = (int)off;
  if (off < 0 || off > p.maxoffset) return false;
  if (p.frame_ok) {
    // samples [off, off + L) lie in frames off/spf .. (off+L-1)/spf, all
    // below the station's slot count since off + L <= (numffts+1) L
    const uint8_t *ok = p.frame_ok[st];
    const long long spf = p.frame_samples[st];
    const long long f1 = (off + L - 1) / spf;
    for (long long f = off / spf; f <= f1; f++)
      if (!ok[f]) return false;
  }
  return true;
}

// Entries e = e0, e0+estep, ... of one item's rotator tables: sub, step
// (fringe rotation, fxkernel.cpp:498-567) and fsub, fstep (fractional-sample
// correction, fxkernel.cpp:595-634), the fsub entries multiplied by fscale (a
// power of two).  Phases in FP64 turns, reduced to half a turn, rounded to
// FP32 (at most 9e-8 rad), then sincospif.  (Phases rounded to FP32 in
// radians and the hardware sine and cosine, within ~5e-7, had been the largest
// part of the FP32 path's error: against FP64, 16 stations x 4096 channels,
// 6.2e-7 -> 3.8e-7 with 1 % more time in the F-stage.)
// Entry e of one item's tables.
template <int L, bool CPLX>
__device__ __forceinline__ float2 table_entry(const FParams &p, double frac, double a, double b, int e, float fscale) {
#pragma clang fp contract(off)
  using TG = TabGeom<L, CPLX>;
  constexpr int S = TG::S, S2 = TG::S2, NSTEPS = TG::NSTEPS;
  double ph;
  if (e < S2) {
    // subphase, fxkernel.cpp:107,508,514,519,525-530,535; whole seconds of
    // delay removed (fxkernel.cpp:503-505)
    const double intdelay = trunc(b);
    ph = ((double)e / (double)L) * a;
    ph = ph + (b - intdelay);
    ph = ph * p.lo;
    if (p.fraclo) ph = ph + p.lofrac * intdelay;
    ph = -ph;
  } else if (e < S2 + NSTEPS) {
    // stepphase, fxkernel.cpp:112,511,522,539
    const int i = e - S2;
    ph = ((double)(i * p.stepmul) / (double)L) * a;
    ph = -(ph * p.lo);
  } else {
    // channel c turns by c bw/nchan frac (fxkernel.cpp:600-611): in samples,
    // frac / (sampletime L) per channel
    const int i = e - S2 - NSTEPS;
    ph = (frac * p.samplerate) * (1.0 / (double)L) * (double)(i < S ? i : (i - S) * S);
  }
  float sn, cs;
  sincospif((float)(2.0 * (ph - rint(ph))), &sn, &cs);
  const float sc = e >= S2 + NSTEPS && e < S2 + NSTEPS + S ? fscale : 1.f;
  return make_float2(cs * sc, sn * sc);
}

template <int L, bool CPLX>
__device__ __forceinline__ void fill_tables(const FParams &p, double frac, double a, double b, float2 *tab,
                                            int e0, int estep, float fscale = 1.f) {
  for (int e = e0; e < TabGeom<L, CPLX>::NTAB; e += estep) tab[e] = table_entry<L, CPLX>(p, frac, a, b, e, fscale);
}

__device__ __forceinline__ uint32_t pack_f16(float re, float im) {
  const _Float16 a = (_Float16)re, b = (_Float16)im;
  return (uint32_t)__builtin_bit_cast(uint16_t, a) | ((uint32_t)__builtin_bit_cast(uint16_t, b) << 16);
}

__device__ __forceinline__ uint32_t bf16_bits(float x) {
  const uint32_t u = __builtin_bit_cast(uint32_t, x);
  return (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;  // round to nearest even
}

__device__ __forceinline__ uint32_t pack_bf16(float re, float im) {
  return bf16_bits(re) | (bf16_bits(im) << 16);
}

__device__ __forceinline__ uint16_t pack_fp8(float re, float im) {
  // e4m3 with saturation to the largest finite value before conversion.
  re = fminf(fmaxf(re, -448.f), 448.f);
  im = fminf(fmaxf(im, -448.f), 448.f);
  return (uint16_t)(__builtin_amdgcn_cvt_pk_fp8_f32(re, im, 0, false) & 0xffff);
}

// Scale of bin q of input srow (= 2*station+pol) for the reduced-precision
// forms; 1 for the others.
template <int OUT, int NCHAN>
__device__ __forceinline__ float bin_scale(const FParams &p, int srow, int q) {
  if constexpr (OUT == OUT_F32 || OUT == OUT_POWER) {
    return 1.f;
  } else {
    return *reinterpret_cast<const float *>(reinterpret_cast<const unsigned char *>(p.scales + (size_t)srow * NCHAN) +
                                            (unsigned)q * 4u);
  }
}

// Bytes of one stored bin, and where the launch's output starts.
constexpr unsigned out_bytes(int out) {
  return out == OUT_F32 ? 8 : out == OUT_FP8 ? 2 : 4;
}
template <int OUT>
__device__ __forceinline__ unsigned char *out_base(const FParams &p) {
  return static_cast<unsigned char *>(OUT == OUT_F32     ? static_cast<void *>(p.spectra)
                                      : OUT == OUT_POWER ? static_cast<void *>(p.power)
                                                         : p.out);
}

// Store one bin at d in the spectra format OUT, with its scale sc =
// bin_scale(...) already read.  (Callers form d as a uniform base plus a 32-bit
// byte offset: the store then takes the base from scalar registers.)
// The spectra are written once and read once, by the X-stage after the
// whole F-stage: streaming (nontemporal) stores of the 4- and 8-byte
// values, so that the X-stage no longer meets the write-back of dirty
// spectra lines (16 stations x 4096 channels on MI355X: FP16 X-stage 3.06
// -> 2.78 ms, FP32 F-stage -0.8 %).  The 2-byte FP8 values keep ordinary
// stores, which the caches combine (as streaming stores the 16-station FP8
// F-stage measured 2-5 % slower).
// NT false: ordinary stores, which L2 combines to lines, where a store's
// neighbouring lanes cover less than 64 bytes (8 stations, F-stage: 64 points,
// FP32 235 -> 88 us, complex 287 -> 70; 128 points, FP16 142 -> 75, complex 162 ->
// 52).  At 64 bytes (128 points, FP32) the F-stage takes 76 us either way, and the
// X-stage behind ordinary stores 54 instead of 49.
template <int OUT, bool NT = true>
__device__ __forceinline__ void store_val(unsigned char *d, float2 y, float sc) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  if constexpr (!NT && OUT == OUT_F32) {
    *reinterpret_cast<f32x2 *>(d) = f32x2{y.x, y.y};
  } else if constexpr (!NT && (OUT == OUT_F16 || OUT == OUT_BF16)) {
    *reinterpret_cast<uint32_t *>(d) = OUT == OUT_F16 ? pack_f16(y.x * sc, y.y * sc) : pack_bf16(y.x * sc, y.y * sc);
  } else if constexpr (OUT == OUT_F32) {
    const f32x2 v = {y.x, y.y};
    __builtin_nontemporal_store(v, reinterpret_cast<f32x2 *>(d));
  } else if constexpr (OUT == OUT_POWER) {
    // one row per sampled FFT; the scale kernel sums rows in a fixed order,
    // so the scales do not depend on scheduling
    *reinterpret_cast<float *>(d) = y.x * y.x + y.y * y.y;
  } else if constexpr (OUT == OUT_FP8) {
    *reinterpret_cast<uint16_t *>(d) = pack_fp8(y.x * sc, y.y * sc);
  } else if constexpr (OUT == OUT_F16) {
    __builtin_nontemporal_store(pack_f16(y.x * sc, y.y * sc), reinterpret_cast<uint32_t *>(d));
  } else {
    __builtin_nontemporal_store(pack_bf16(y.x * sc, y.y * sc), reinterpret_cast<uint32_t *>(d));
  }
}

// Store CON neighbouring bins at d (CON * the bin's bytes aligned) in one store
// (FP32: one per two bins).
template <int OUT, int CON>
__device__ __forceinline__ void store_row(unsigned char *d, const float2 (&y)[CON], const float (&sc)[CON]) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  if constexpr (CON == 1) {
    store_val<OUT>(d, y[0], sc[0]);
  } else if constexpr (OUT == OUT_F32) {
#pragma unroll
    for (int i = 0; i < CON; i += 2)
      __builtin_nontemporal_store((f32x4){y[i].x, y[i].y, y[i + 1].x, y[i + 1].y}, reinterpret_cast<f32x4 *>(d + 8 * i));
  } else if constexpr (OUT == OUT_POWER) {
    typedef float row __attribute__((ext_vector_type(CON)));
    row r;
#pragma unroll
    for (int i = 0; i < CON; i++) r[i] = y[i].x * y[i].x + y[i].y * y[i].y;
    *reinterpret_cast<row *>(d) = r;
  } else if constexpr (OUT == OUT_FP8) {
    typedef uint16_t row __attribute__((ext_vector_type(CON)));
    row r;
#pragma unroll
    for (int i = 0; i < CON; i++) r[i] = pack_fp8(y[i].x * sc[i], y[i].y * sc[i]);
    *reinterpret_cast<row *>(d) = r;
  } else {
    typedef uint32_t row __attribute__((ext_vector_type(CON)));
    row r;
#pragma unroll
    for (int i = 0; i < CON; i++)
      r[i] = OUT == OUT_F16 ? pack_f16(y[i].x * sc[i], y[i].y * sc[i]) : pack_bf16(y[i].x * sc[i], y[i].y * sc[i]);
    __builtin_nontemporal_store(r, reinterpret_cast<row *>(d));
  }
}

// Store bin q of output row `row` (= 2*station + pol within FFT row block).
template <int OUT, int NCHAN>
__device__ __forceinline__ void store_bin_sc(const FParams &p, size_t row, int q, float2 y, float sc) {
  store_val<OUT>(out_base<OUT>(p) + row * (NCHAN * out_bytes(OUT)) + (unsigned)q * out_bytes(OUT), y, sc);
}

// Store bin q of output row `row`; `srow` is the input index 2*station+pol.
template <int OUT, int NCHAN>
__device__ __forceinline__ void store_bin(const FParams &p, size_t row, int srow, int q, float2 y) {
  store_bin_sc<OUT, NCHAN>(p, row, q, y, bin_scale<OUT, NCHAN>(p, srow, q));
}

// Workgroups are dealt to the 8 XCDs round robin in dispatch order, each XCD
// with its own L2.  Renumbering unit v of `total` so that consecutive units
// run on one XCD one after another lets neighbouring units share lines in
// that L2 (the tail beyond a multiple of 8 keeps its number).
constexpr int kXcdCount = 8;
__device__ __forceinline__ long long xcd_order(long long v, long long total) {
  const long long per = total / kXcdCount;
  if (v >= per * kXcdCount) return v;
  return (v % kXcdCount) * per + v / kXcdCount;
}

// Segment of a launch over several subbands that holds unit u.
__device__ __forceinline__ int find_fseg(const FSeg *__restrict__ segs, int nseg, long long u) {
  int a = 0;
  for (int b = nseg; b - a > 1;) {
    const int m = (a + b) / 2;
    if (u >= segs[m].unit0)
      a = m;
    else
      b = m;
  }
  return __builtin_amdgcn_readfirstlane(a);
}

// Parameters of segment k.  The compiler takes a kernel argument's pointers as
// global memory, but those it loads from a table as generic ones (flat loads and
// stores, and 12 registers spilled at 2048 points): each goes by the global
// address space, from an integer, since a cast there and back is folded away.
template <typename T>
__device__ __forceinline__ T *as_global(T *p) {
  return (T *)(__attribute__((address_space(1))) T *)reinterpret_cast<uintptr_t>(p);
}
__device__ __forceinline__ FParams segment_params(const FSeg *__restrict__ segs, int k) {
  FParams p = segs[k].p;
  p.station = as_global(p.station);
  p.delays = as_global(p.delays);
  p.subchanfreq = as_global(p.subchanfreq);
  p.stepchanfreq = as_global(p.stepchanfreq);
  p.twiddle = as_global(p.twiddle);
  p.spectra = as_global(p.spectra);
  p.out = as_global(p.out);
  p.scales = as_global(p.scales);
  p.power = as_global(p.power);
  p.valid = as_global(p.valid);
  p.frame_ok = as_global(p.frame_ok);
  p.frame_samples = as_global(p.frame_samples);
  return p;
}

// Global-address-space view of the packed station buffers: the loads then
// use the global rather than the flat address path.
typedef const __attribute__((address_space(1))) uint8_t gbyte;

}  // namespace fs
}  // namespace gxc
